"""The matrix-core product behind sm_gemm_f32 and the fused training pass."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    from seismicmesh_amd import _lib
    _lib.require_gpu()


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


# edges of the 64 and 128 tiles and of the 16-deep slices, every layout, with
# and without a split; the last ones fall back to the vector kernel (rows too
# few, an unaligned stride, a stride below the run: overlapping rows)
@pytest.mark.parametrize("M,N,K,ta,tb,nsplit,off", [
    (64, 64, 16, False, False, 1, 0), (68, 60, 20, False, False, 1, 0),
    (128, 128, 16, True, False, 1, 0), (132, 124, 36, True, True, 1, 0),
    (256, 256, 4, False, True, 1, 0), (33, 256, 256, False, True, 1, 0),
    (256, 256, 5001, True, False, 7, 0), (256, 256, 17, True, False, 9, 0),
    (16500, 256, 256, False, True, 1, 0), (65535 * 64 + 33, 36, 4, False, True, 1, 0),
    (16384, 260, 64, False, False, 3, 0),
    (31, 256, 256, False, True, 1, 0), (256, 256, 30, False, True, 1, 0),
    (64, 64, 64, False, True, 1, 1)])
def test_gemm_matches_float64(M, N, K, ta, tb, nsplit, off):
    import torch
    from seismicmesh_amd import _lib
    rng = np.random.default_rng(M + N + K)
    A = rng.standard_normal((K, M) if ta else (M, K)).astype(np.float32)
    B = rng.standard_normal((N, K) if tb else (K, N)).astype(np.float32)
    C0 = rng.standard_normal((M, N)).astype(np.float32)
    dev = "cuda:0"
    Ad = torch.empty(A.size + off, dtype=torch.float32, device=dev)
    Ad[off:] = torch.from_numpy(A).to(dev).reshape(-1)
    Bd, Cd = torch.from_numpy(B).to(dev), torch.from_numpy(C0).to(dev)
    work = torch.empty(nsplit * M * N, dtype=torch.float32, device=dev)
    sam, sak = (1, M) if ta else (K, 1)
    sbk, sbn = (1, K) if tb else (N, 1)
    _lib.check(_lib.lib.sm_gemm_f32(M, N, K, 0.5, _p(Ad[off:]), sam, sak, _p(Bd), sbk, sbn, 2.0,
                                    _p(Cd), N, nsplit, _p(work), None), "sm_gemm_f32")
    torch.cuda.synchronize()
    Am, Bm = (A.T if ta else A).astype(np.float64), (B.T if tb else B).astype(np.float64)
    got = Cd.cpu().numpy()
    # each output: K roundings of its own partial sums at most, and four more
    bound = 2.0 ** -24 * (K + 4) * (0.5 * np.abs(Am) @ np.abs(Bm) + 2.0 * np.abs(C0))
    assert (np.abs(got - (0.5 * (Am @ Bm) + 2.0 * C0)) <= bound).all()


def _grad_tol(hidden, lam):
    """Of a gradient's largest entry.  A product of 256 terms, summed in FP32,
    is off by about sqrt(256) 2^-24 = 1e-6 of its terms' size, a layer has two
    of them and the sum over the rows one more: 3e-5 a layer leaves a factor of
    ten.  The eikonal term divides the difference of two outputs, each off by
    about 5e-7, by 2 x 5e-3: 7e-5 of a slope of 1, again with a margin."""
    return 3e-5 * (hidden + 1) + (5e-4 if lam > 0 else 0.0)


# row counts around the tile sizes and the switch between them (16384 rows),
# with and without the eikonal copies, no hidden layer at all, more layers
# than one launch of sums takes (15, 32, ...)
@pytest.mark.parametrize("n,dim,hidden,lam", [
    (1, 3, 1, 0.0), (63, 2, 2, 0.0), (65, 3, 3, 0.1), (300, 2, 0, 0.1), (2341, 3, 1, 0.1),
    (16383, 2, 1, 0.0), (16385, 3, 2, 0.0), (40, 2, 15, 0.0), (40, 2, 16, 0.1), (40, 3, 17, 0.0),
    (40, 2, 40, 0.0)])
def test_training_pass_matches_float64(n, dim, hidden, lam):
    import torch
    from oracle import mlp as omlp
    from seismicmesh_amd.neural import NeuralSDF
    net = NeuralSDF(dim, [-1.0, 1.0] * dim, hidden=hidden, seed=3)
    rng = np.random.default_rng(n)
    if hidden > 3:
        # the initial weights let a gradient (and the slope) die over many
        # layers, 1e-11 at the input of 16: wider ones, which keep them at 1
        flat = np.concatenate([rng.uniform(-b, b, k).astype(np.float32) for k, b in (
            (256 * dim, 3.0), (256, 1.0), (hidden * 65536, 2.6 / 16), (hidden * 256, 0.1),
            (256, 1 / 16), (1, 0.1))])
        net.set_params(flat)
    x = rng.uniform(-1, 1, (n, dim))
    t = (np.linalg.norm(x, axis=1) - 0.5).astype(np.float32)
    part = net.loss_and_grad(torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda(), eik=lam)
    g = net.grad.cpu().numpy().astype(np.float64)
    L, ref = omlp.loss_and_grad(net.numpy_params().astype(np.float64), dim, 256, hidden, x,
                                t.astype(np.float64), net.shift, net.scale, lam=lam, eik_h=5e-3)
    assert abs(float(part.cpu().numpy().astype(np.float64).sum()) - L) <= 1e-4 * abs(L)
    for name, (o, k) in net.layout.items():
        if k == 0:
            continue
        r = ref[o:o + k]
        assert np.abs(g[o:o + k] - r).max() <= _grad_tol(hidden, lam) * np.abs(r).max(), name


def test_training_pass_over_more_rows_than_a_grid_dimension():
    """More than 65535 tiles of 64 rows (26 GB of workspace): the gradient is
    the mean of those of two parts."""
    import torch
    from seismicmesh_amd.neural import NeuralSDF
    net = NeuralSDF(2, [-1.0, 1.0] * 2, hidden=1, seed=3)
    n, cut = 65535 * 64 + 77, 2000000
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.rand(n, 2, generator=g, device="cuda", dtype=torch.float64) * 2.0 - 1.0
    t = (x.norm(dim=1) - 0.5).to(torch.float32)
    whole, loss = None, []
    mean = 0.0
    for lo, hi in ((0, n), (0, cut), (cut, n)):
        part = net.loss_and_grad(x[lo:hi], t[lo:hi], eik=0.0)
        loss.append(float(part.double().sum()) * (hi - lo) / n)
        if whole is None:
            whole = net.grad.double()
        else:
            mean = mean + net.grad.double() * ((hi - lo) / n)
    net._bufs = {}
    assert abs(loss[0] - loss[1] - loss[2]) <= 1e-4 * loss[0]
    for name, (o, k) in net.layout.items():
        d = (whole - mean)[o:o + k].abs().max()
        assert float(d) <= _grad_tol(1, 0.0) * float(mean[o:o + k].abs().max()), name


@pytest.mark.parametrize("eik,eik_h", [(-0.1, 5e-3), (float("nan"), 5e-3), (0.0, -1.0)])
def test_an_eikonal_weight_not_above_zero_drops_the_term(eik, eik_h):
    import torch
    from seismicmesh_amd.neural import NeuralSDF
    net = NeuralSDF(2, [-1.0, 1.0] * 2, hidden=1, seed=3)
    x = torch.from_numpy(np.random.default_rng(0).uniform(-1, 1, (100, 2))).cuda()
    t = (x.norm(dim=1) - 0.5).to(torch.float32)
    part = net.loss_and_grad(x, t, eik=0.0).clone()
    grad = net.grad.clone()
    assert torch.equal(net.loss_and_grad(x, t, eik=eik, eik_h=eik_h), part)
    assert torch.equal(net.grad, grad)
    for bad in ((0.1, 0.0), (0.1, -1.0), (-0.1, 0.0), (float("nan"), 0.0)):
        with pytest.raises(RuntimeError, match="eik_h > 0"):
            net.loss_and_grad(x, t, eik=bad[0], eik_h=bad[1])


@pytest.mark.parametrize("hidden", [0, 1])
def test_activation_rounds_as_the_single_step(hidden):
    """One sample with gy = 1 and w_out = 0: the gradient of w_out is the last
    activation itself, bit for bit that of sm_mlp_bias_silu (the identity as
    hidden layer: the first one's activation once more)."""
    import torch
    from seismicmesh_amd import _lib
    from seismicmesh_amd.neural import NeuralSDF
    net = NeuralSDF(2, [-1.0, 1.0] * 2, hidden=hidden)
    x = torch.tensor([[1.0, 0.0]], dtype=torch.float64, device="cuda")
    t = torch.tensor([-0.5], dtype=torch.float32, device="cuda")
    rng = np.random.default_rng(7)
    o = {k: v[0] for k, v in net.layout.items()}
    for scale in (1e-3, 0.3, 3.0, 20.0, 100.0):
        z = (scale * rng.standard_normal(256)).astype(np.float32)
        flat = np.zeros(net.nparams, dtype=np.float32)
        flat[o["w_in"]:o["w_in"] + 512:2] = z
        if hidden:
            flat[o["w_hid"]:o["w_hid"] + 65536] = np.eye(256, dtype=np.float32).ravel()
        net.set_params(flat)
        net.loss_and_grad(x, t, eik=0.0)
        zero = torch.zeros(256, dtype=torch.float32, device="cuda")
        want = torch.from_numpy(z).cuda()
        for _ in range(hidden + 1):
            a = torch.empty_like(want)
            _lib.check(_lib.lib.sm_mlp_bias_silu(1, 256, _p(want), _p(zero), _p(a), None),
                       "sm_mlp_bias_silu")
            want = a
        assert torch.equal(net.grad[o["w_out"]:o["w_out"] + 256], want)


def _single_steps(net, x, t, lam, eik_h=5e-3):
    """The pass as a sequence of the single-step entry points on own buffers;
    returns the loss partials and the gradient."""
    import torch
    from seismicmesh_amd import _lib
    lib, dim, W, L = _lib.lib, net.dim, net.width, net.hidden
    dev, n = x.device, len(x)
    rows = n * (2 * dim + 1 if lam > 0 else 1)

    def buf(*shape):
        return torch.empty(shape, dtype=torch.float32, device=dev)

    def gemm(M, N, K, A, sam, sak, B, sbk, sbn, C):
        _lib.check(lib.sm_gemm_f32(M, N, K, 1.0, _p(A), sam, sak, _p(B), sbk, sbn, 0.0, _p(C), N,
                                   1, None, None), "sm_gemm_f32")

    o = {k: v[0] for k, v in net.layout.items()}
    w = {"in": net.params[o["w_in"]:], "out": net.params[o["w_out"]:]}
    hid = [net.params[o["w_hid"] + l * W * W:] for l in range(L)]
    bias = [net.params[o["b_in"]:]] + [net.params[o["b_hid"] + l * W:] for l in range(L)]
    X, Z, A = buf(rows, dim), [buf(rows, W) for _ in range(L + 1)], \
        [buf(rows, W) for _ in range(L + 1)]
    shift = np.r_[net.shift, 0.0][:3].copy()
    scale = np.r_[net.scale, 0.0][:3].copy()
    _lib.check(lib.sm_mlp_make_inputs(n, dim, _p(x), shift.ctypes.data, scale.ctypes.data,
                                      eik_h if lam > 0 else 0.0, _p(X), None), "make_inputs")
    for l in range(L + 1):
        if l == 0:
            gemm(rows, W, dim, X, dim, 1, w["in"], 1, dim, Z[0])
        else:
            gemm(rows, W, W, A[l - 1], W, 1, hid[l - 1], 1, W, Z[l])
        _lib.check(lib.sm_mlp_bias_silu(rows, W, _p(Z[l]), _p(bias[l]), _p(A[l]), None), "silu")
    y, gy, part = buf(rows), buf(rows), buf((n + 255) // 256)
    gemm(rows, 1, W, A[L], W, 1, w["out"], 1, 0, y)
    _lib.check(lib.sm_mlp_bias_silu(rows, 1, _p(y), _p(net.params[o["b_out"]:]), None, None), "b")
    _lib.check(lib.sm_mlp_sdf_loss(n, dim, _p(y), _p(t), eik_h, lam, 0.0, _p(gy), _p(part), None),
               "loss")
    grad = torch.zeros_like(net.params)
    ones = torch.ones(rows, dtype=torch.float32, device=dev)
    gemm(1, W, rows, gy, 0, 1, A[L], W, 1, grad[o["w_out"]:])
    gemm(1, 1, rows, gy, 0, 1, ones, 1, 0, grad[o["b_out"]:])
    dA, dZ = buf(rows, W), buf(rows, W)
    gemm(rows, W, 1, gy, 1, 0, w["out"], 0, 1, dA)
    for l in range(L, -1, -1):
        _lib.check(lib.sm_mlp_silu_backward(rows * W, _p(Z[l]), _p(dA), _p(dZ), None), "back")
        b = grad[o["b_in"]:] if l == 0 else grad[o["b_hid"] + (l - 1) * W:]
        gemm(1, W, rows, ones, 0, 1, dZ, W, 1, b)
        if l == 0:
            gemm(W, dim, rows, dZ, 1, W, X, dim, 1, grad[o["w_in"]:])
        else:
            gemm(W, W, rows, dZ, 1, W, A[l - 1], W, 1, grad[o["w_hid"] + (l - 1) * W * W:])
            gemm(rows, W, W, dZ, W, 1, hid[l - 1], W, 1, dA)
    torch.cuda.synchronize()
    return part, grad


@pytest.mark.parametrize("n,dim,hidden,lam", [(1, 2, 0, 0.0), (300, 3, 2, 0.1), (1000, 2, 3, 0.0)])
def test_the_single_steps_make_the_fused_pass(n, dim, hidden, lam):
    import torch
    from seismicmesh_amd.neural import NeuralSDF
    net = NeuralSDF(dim, [-1.0, 1.0] * dim, hidden=hidden, seed=4)
    x = torch.from_numpy(np.random.default_rng(n).uniform(-1, 1, (n, dim))).cuda()
    t = (x.norm(dim=1) - 0.5).to(torch.float32)
    part = net.loss_and_grad(x, t, eik=lam)
    part1, grad = _single_steps(net, x, t, lam)
    assert float((part - part1).abs().max()) <= 1e-4 * float(part.abs().max())
    for name, (o, k) in net.layout.items():
        if k:
            a, b = net.grad[o:o + k], grad[o:o + k]
            tol = 2 * _grad_tol(hidden, lam) * float(b.abs().max())
            assert float((a - b).abs().max()) <= tol, name
