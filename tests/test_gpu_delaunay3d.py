"""The device tetrahedralisation (csrc/stars3d.hip) against the host's:
the same cells in the same order, as integers, for every kind of point set
that takes another way through it (the tolerance is equality)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    from seismicmesh_amd import _lib
    _lib.require_gpu()


def _host(p):
    from seismicmesh_amd import _lib
    n = len(p)
    t = np.empty((40 * n + 64, 4), dtype=np.int32)
    ins = np.empty(n, dtype=np.uint8)
    m = _lib.lib.sm_host_delaunay3d(p.ctypes.data, n, t.ctypes.data, len(t), ins.ctypes.data)
    assert m >= 0
    return t[:m]


def _device(p, h):
    """Every cell of the handle's tetrahedralisation (a domain that holds
    them all), and whether the device built it."""
    from seismicmesh_amd import generation, geometry as geo
    lo, hi = p.min(0), p.max(0)
    dom = geo.Ball([float(v) for v in (lo + hi) / 2], 1e7 * float((hi - lo).max()))
    m = generation.Mesher([dom], generation._Sizing("const", value=h), h, 0.2, 0.1 * h, 1e-8 * h,
                          0, precision=32, dim=3)
    m.set_points(p)
    m.triangulate()
    s = m.stats()
    t = m.cells()
    m.close()
    assert s["host_rebuilds"] + s["device_builds"] == 1
    return t, s["device_builds"] == 1


def _box(rng, n, noise):
    # a jittered lattice whose outer layers lie in the six sides of a box,
    # exactly or up to rounding noise
    g = np.linspace(0.0, 1.0, n)
    p = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    side = (p == 0.0) | (p == 1.0)
    p = p + np.where(side, noise * rng.uniform(-1, 1, p.shape),
                     rng.uniform(-0.2, 0.2, p.shape) / n)
    return p


def _points(kind):
    rng = np.random.default_rng(11)
    if kind.startswith("random"):
        n = int(kind[6:])
        return rng.uniform(-1, 1, (n, 3)), 2.0 / n ** (1 / 3)
    if kind == "spacing_too_large":
        return rng.uniform(-1, 1, (2000, 3)), 1e3
    if kind == "spacing_too_small":
        return rng.uniform(-1, 1, (2000, 3)), 1e-7
    if kind == "clustered":
        return np.vstack([rng.normal(0, 0.02, (1500, 3)), rng.uniform(-1, 1, (1500, 3))]), 0.02
    if kind == "box_exact":
        return _box(rng, 13, 0.0), 1 / 12
    if kind == "box_noise":
        return _box(rng, 13, 1e-15), 1 / 12
    if kind.startswith("box_rows"):
        # rows of points exactly on the edges of the box, noise on its sides:
        # three of a row and a neighbour are coplanar, which the coordinates'
        # span keeps from the exact stage.  Evenly spaced, the rows' points
        # also lie on common spheres, which it cannot settle
        g = np.linspace(0.0, 1.0, 13)
        p = _box(rng, 13, 1e-14)
        q = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
        side = (q == 0.0) | (q == 1.0)
        edge = side.sum(1) >= 2
        p[edge] = q[edge]
        if kind == "box_rows":
            p += np.where(side | ~edge[:, None], 0.0, rng.uniform(-0.2, 0.2, p.shape) / 13)
        return p, 1 / 12
    if kind == "duplicates":
        p = rng.uniform(-1, 1, (1500, 3))
        return np.vstack([p, p[::7], p[::11]]), 0.15
    if kind == "hub":
        # one point amid many at nearly one distance: a star of hundreds
        # of cells, left to its neighbours
        d = rng.normal(size=(700, 3))
        d *= (1.0 + 1e-3 * rng.uniform(-1, 1, (700, 1))) / np.linalg.norm(d, axis=1)[:, None]
        return np.vstack([rng.normal(0, 1e-3, (3, 3)), d, 3.0 * rng.uniform(-1, 1, (900, 3))]), 0.3
    if kind == "long":
        return rng.uniform(0, 1, (3000, 3)) * np.array([400.0, 1.0, 1.0]), 0.5
    if kind == "far_from_origin":
        return rng.uniform(0, 1, (2000, 3)) + 1e6, 0.08
    if kind == "tiny":
        return rng.uniform(0, 1, (2000, 3)) * 1e-9, 0.08e-9
    if kind == "lattice":
        g = np.arange(12) * 0.1
        return np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3), 0.1
    assert kind == "plane"
    return np.column_stack([rng.uniform(0, 1, (200, 2)), np.zeros(200)]), 0.1


@pytest.mark.parametrize("kind", [
    "random511", "random512", "random513", "random2000", "random30000", "spacing_too_large",
    "spacing_too_small", "clustered", "box_exact", "box_noise", "box_rows", "box_rows_even",
    "duplicates", "hub", "long", "far_from_origin", "tiny", "lattice", "plane"])
def test_cells_equal_the_host_build(kind):
    p, h = _points(kind)
    p = np.ascontiguousarray(p)
    ref = _host(p)
    got, on_device = _device(p, h)
    assert np.array_equal(got, ref)
    if kind.startswith("random") or kind in ("box_exact", "box_noise", "box_rows", "hub", "long",
                                             "duplicates"):
        assert on_device == (len(p) >= 512)
    if kind == "plane":
        assert len(ref) == 0 and not on_device


def test_a_failed_build_is_followed_by_the_host_then_the_device_again():
    """One handle over point sets that the device build takes, leaves to the
    host, and takes again: each triangulation is that of its own points."""
    from seismicmesh_amd import generation, geometry as geo
    rng = np.random.default_rng(5)
    g = np.arange(11) * 0.1
    lat = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    m = generation.Mesher([geo.Ball([0.0, 0.0, 0.0], 1e7)],
                          generation._Sizing("const", value=0.1), 0.1, 0.2, 0.01, 1e-9, 0,
                          precision=32, dim=3)
    for p in [lat + rng.uniform(-0.02, 0.02, lat.shape), lat] + \
             [lat + rng.uniform(-0.02, 0.02, lat.shape) for _ in range(5)]:
        m.set_points(p)
        m.triangulate()
        assert np.array_equal(m.cells(), _host(np.ascontiguousarray(p)))
    assert m.stats()["device_builds"] >= 2
    m.close()


@pytest.mark.parametrize("side,share,by_device", [
    (8, 0.25, False), (8, 0.45, False), (10, 0.25, False), (13, 0.06, True), (13, 0.25, False),
    (16, 0.2, True), (16, 0.6, False), (40, 0.3, True), (41, 0.3, True), (41, 0.7, False)])
def test_lattice_share_left_to_the_host(side, share, by_device):
    # exact cubes in part of the box (their stars take the exact pass), a
    # jittered lattice in the rest: the device settles as many vertices
    # exactly as cost it what the host's one thread would take, a
    # thirty-second to a half.
    # Coordinates in [1, 2): one binary exponent, the exact stage's range
    rng = np.random.default_rng(side)
    g = 1.0 + np.arange(side) / 64.0
    p = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    moved = p[:, 0] > 1.0 + share * side / 64.0
    p[moved] += rng.uniform(0.0, 0.2 / 64.0, (int(moved.sum()), 3))
    p = np.ascontiguousarray(p)
    cells, dev = _device(p, 1 / 64)
    assert dev == by_device
    assert np.array_equal(cells, _host(p))


def test_a_build_without_room_for_its_scratch_goes_to_the_host():
    # 0.6 kB a point: 100 kB are too little for 2000, 10 MB are enough
    from seismicmesh_amd import generation, geometry as geo
    p, h = _points("random2000")
    m = generation.Mesher([geo.Ball([0.0, 0.0, 0.0], 1e7)], generation._Sizing("const", value=h),
                          h, 0.2, 0.1 * h, 1e-8 * h, 0, precision=32, dim=3)
    m.set_points(p)
    ref = _host(np.ascontiguousarray(p))
    for limit, built in ((100000, 0), (10000000, 1), (100000, 1), (0, 2)):
        m.set_scratch_limit(limit)
        m.triangulate()
        assert np.array_equal(m.cells(), ref)
        s = m.stats()
        assert s["device_builds"] == built and s["device_left"] == (8 if limit == 100000 else 0)
    m.close()


@pytest.mark.parametrize("share,radius,left", [(0.5, 0.02, 6), (0.5, 1e-4, 6), (0.5, 1e-9, 6),
                                               (0.05, 0.02, 0), (0.05, 1e-9, 2)])
def test_crowded_cells_are_left_to_the_host(share, radius, left):
    # `share` of 8000 points in a small ball, amid the rest: most of them
    # beyond the 24th of their cell of the search grid when the ball has few
    # cells; up to an eighth of all points may be (the last set's reason is
    # another: coordinates of 1e-9 next to ones of 1 span more bits than the
    # exact stage holds)
    rng = np.random.default_rng(3)
    k = int(8000 * share)
    d = rng.normal(size=(k, 3))
    d *= radius * rng.random((k, 1)) ** (1 / 3) / np.linalg.norm(d, axis=1)[:, None]
    p = np.vstack([d, rng.uniform(-1, 1, (8000 - k, 3))])
    from seismicmesh_amd import generation, geometry as geo
    m = generation.Mesher([geo.Ball([0.0, 0.0, 0.0], 1e7)],
                          generation._Sizing("const", value=0.1), 0.1, 0.2, 0.01, 1e-9, 0,
                          precision=32, dim=3)
    m.set_points(p)
    m.triangulate()
    assert np.array_equal(m.cells(), _host(np.ascontiguousarray(p)))
    s = m.stats()
    assert s["device_left"] == left and s["device_builds"] == (left == 0)
    m.close()


def _mixed_lattice(side, shift):
    # A staggered lattice around the origin whose coordinates are rounded
    # multiples of 0.1 (no common power of two), shifted by `shift`: zeros
    # become coordinates of 1e-30 next to ones of 1, beyond the exact stage
    g = (np.arange(side) - side // 2) * 0.1
    p = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    p[:, 0] += 0.05 * (np.arange(len(p)) // side % 2)
    return p + shift


@pytest.mark.parametrize("side", [16, 41])
def test_a_predicate_beyond_the_exact_stage(side):
    # 41^3 > 65536 points; enough of them moved that the build gets as far as
    # its exact stars
    p = _mixed_lattice(side, 1e-30)
    rng = np.random.default_rng(side)
    moved = rng.random(len(p)) < 0.7
    p[moved] += rng.uniform(-0.01, 0.01, (int(moved.sum()), 3))
    p = np.ascontiguousarray(p)
    from seismicmesh_amd import generation, geometry as geo
    m = generation.Mesher([geo.Ball([0.0, 0.0, 0.0], 1e7)],
                          generation._Sizing("const", value=0.1), 0.1, 0.2, 0.01, 1e-9, 0,
                          precision=32, dim=3)
    m.set_points(p)
    m.triangulate()
    s = m.stats()
    assert s["device_left"] == 2 and s["device_builds"] == 0
    assert np.array_equal(m.cells(), _host(p))
    m.close()


def test_new_points_are_tried_on_the_device_whatever_failed_before():
    from seismicmesh_amd import generation, geometry as geo
    m = generation.Mesher([geo.Ball([0.0, 0.0, 0.0], 1e7)],
                          generation._Sizing("const", value=0.1), 0.1, 0.2, 0.01, 1e-9, 0,
                          precision=32, dim=3)
    g = np.arange(13) / 16.0
    lattice = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    good = np.random.default_rng(1).uniform(-1, 1, (2000, 3))
    for p, built in ((lattice, 0), (good, 1), (good, 2), (lattice, 2), (good, 3)):
        m.set_points(p)
        m.triangulate()
        assert m.stats()["device_builds"] == built
        assert np.array_equal(m.cells(), _host(np.ascontiguousarray(p)))
    m.close()
