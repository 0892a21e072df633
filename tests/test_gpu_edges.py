"""The sorted unique edges of pairs, triangles and tetrahedra at the edges of the builder's blocks
(512 tetrahedra, 1024 triangles or pairs), of its 256-vertex row blocks and of its bucket sorts
(16, 64 and 4096 ids), against numpy.  Whole numbers: equal."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from seismicmesh_amd import _lib  # noqa: E402

pytestmark = pytest.mark.gpu


def _oracle(items):
    k = items.shape[1]
    pairs = np.concatenate([items[:, [i, j]] for i in range(k) for j in range(i + 1, k)])
    return np.unique(np.sort(pairs, axis=1), axis=0)


def _device(items, nv):
    dev = torch.device("cuda")
    n, k = items.shape
    t = torch.tensor(items, dtype=torch.int32, device=dev).contiguous()
    npairs = n * {2: 1, 3: 3, 4: 6}[k]
    out = torch.full((npairs, 2), -7, dtype=torch.int32, device=dev)
    cnt = torch.zeros(1, dtype=torch.int64, device=dev)
    nbytes = (_lib.lib.sm_unique_edges_workspace(npairs, nv) if k == 2 else
              _lib.lib.sm_cell_edges_workspace(n, k - 1, nv))
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    p = [ctypes.c_void_p(x.data_ptr()) for x in (t, out, cnt, ws)]
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    if k == 2:
        rc = _lib.lib.sm_unique_edges(p[0], n, nv, p[1], p[2], p[3], nbytes, s)
    else:
        rc = _lib.lib.sm_cell_edges(p[0], n, k - 1, nv, p[1], p[2], p[3], nbytes, s)
    _lib.check(rc, "edges")
    c = int(cnt.item())
    out = out.cpu().numpy()
    assert (out[c:] == -7).all()  # the rest of the buffer stays as it was
    return out[:c]


@pytest.mark.parametrize("k", [2, 3, 4])
@pytest.mark.parametrize("n", [1, 511, 512, 513, 1023, 1024, 1025, 5000])
@pytest.mark.parametrize("kind", ["distinct", "local", "random", "hub"])
def test_unique_edges_block_edges(k, n, kind):
    rng = np.random.default_rng(n * 8 + k)
    if kind == "distinct":  # no vertex twice: every block's list is full
        items = rng.permutation(n * k).reshape(n, k)
    elif kind == "local":  # neighbours share nearly everything
        base = np.arange(n)[:, None] // 5
        items = base + np.stack([rng.permutation(8)[:k] for _ in range(n)])
    elif kind == "random":
        items = np.stack([rng.choice(max(n // 3, 8), k, replace=False) for _ in range(n)])
    else:  # every item holds vertex 0: one bucket of up to 5000 k ids
        items = np.concatenate([np.zeros((n, 1), int),
                                1 + np.arange(n * (k - 1)).reshape(n, k - 1)], 1)
    nv = int(items.max()) + 1 + (n % 3)
    np.testing.assert_array_equal(_device(items, nv), _oracle(items))


@pytest.mark.parametrize("nv", [255, 256, 257])
@pytest.mark.parametrize("length", [15, 16, 17, 63, 64, 65, 4096, 4097])
def test_unique_edges_bucket_lengths(nv, length):
    # buckets of one length with each id twice, from three vertices of a row block
    rng = np.random.default_rng(length)
    items = []
    for v in (0, 100, nv - 1):
        to = nv + rng.permutation(length * 2)[:(length + 1) // 2]
        items += [(v, int(b)) for b in np.concatenate([to, to])[:length]]
    items = rng.permutation(np.array(items))
    n = int(items.max()) + 1
    np.testing.assert_array_equal(_device(items, n), _oracle(items))


@pytest.mark.parametrize("n,nv", [(16384, 9000), (16385, 16385), (16385, 16384), (20000, 20001),
                                  (4000, 500), (4000, 501)])
@pytest.mark.parametrize("kind", ["random", "path", "equal"])
def test_unique_edges_few_pairs(n, nv, kind):
    # up to 16384 pairs, fewer than 8 to a vertex, or any number up to one to a
    # vertex are counted without the tables
    rng = np.random.default_rng(n + nv)
    if kind == "random":
        items = rng.integers(0, nv, (n, 2))
    elif kind == "path":
        i = rng.permutation(n) % (nv - 1)
        items = np.stack([i + 1, i], 1)
    else:
        items = np.tile([[nv - 1, 3]], (n, 1))
    np.testing.assert_array_equal(_device(items, nv), _oracle(items))


@pytest.mark.parametrize("nv", [31, 32, 33, 65, 1000, 32768, 32769])
def test_unique_edges_few_long_buckets(nv):
    # 8 pairs to a vertex and more: up to 32768 buckets are sorted 32 to a
    # workgroup; lengths around the per-thread, wave and workgroup sorts
    rng = np.random.default_rng(nv)
    first = np.repeat(np.arange(nv), rng.choice([0, 1, 16, 17, 20, 64, 65, 90], nv))
    first = np.concatenate([first, np.full(max(0, 8 * nv + 16385 - len(first)), nv - 1)])
    items = np.stack([first, rng.integers(0, nv, len(first))], 1)
    items = rng.permutation(items)
    np.testing.assert_array_equal(_device(items, nv), _oracle(items))
