"""Skinning and the node graph against the oracle's scans: ids, edges and ties bit for bit, weights to FP32.

The grid of the skinning (up to 4096 nodes) may visit the nodes in any order, so equal distances go through the
same scan as the oracle's; the cases here have none, a few and only such surfels, positions outside the nodes' box,
one cell, flat boxes, non-finite positions, and node counts on both sides of every limit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    assert torch.cuda.is_available()
    torch.cuda.set_device(0)
    return torch


def _four(a):
    return np.ascontiguousarray(np.concatenate([a, np.ones((len(a), 1))], 1).astype(np.float32))


def _sphere(rng, n):
    v = rng.standard_normal((n, 3))
    return v / np.linalg.norm(v, axis=1, keepdims=True)


def _points(kind, S, N, rng):
    """(surfels, nodes, node radius squared)"""
    if kind == "sphere":
        return _sphere(rng, S), _sphere(rng, N), 16.0 / N
    if kind == "volume":
        return rng.uniform(-1, 1, (S, 3)), rng.uniform(-1, 1, (N, 3)), 0.02
    if kind == "plane":  # a box without a height
        p = lambda n: np.concatenate([rng.uniform(0, 2, (n, 2)), np.full((n, 1), 0.5)], 1)
        return p(S), p(N), 8.0 / N
    if kind == "line":
        p = lambda n: np.concatenate([rng.uniform(0, 2, (n, 1)), np.zeros((n, 2))], 1)
        return p(S), p(N), 0.01
    if kind == "lattice":  # equal distances everywhere
        side = int(np.ceil(N ** (1 / 3)))
        g = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)[:N] * 0.25
        return g[rng.integers(0, N, S)] + 0.125 * rng.integers(0, 2, (S, 3)), g[rng.permutation(N)], 0.1
    if kind == "some_ties":  # a few nodes twice, so that a few surfels of a wave meet equal distances
        n = _sphere(rng, N)
        n[rng.integers(0, N, max(1, N // 200))] = n[rng.integers(0, N, max(1, N // 200))]
        return _sphere(rng, S), n, 16.0 / N
    if kind == "outside":  # far from the box of the nodes, and its far corners
        s = np.concatenate([_sphere(rng, S // 2) * 30.0, rng.uniform(-3, 3, (S - S // 2, 3))])
        return s, _sphere(rng, N) * 0.7 + np.array([0.3, -0.2, 0.9]), 400.0
    if kind == "offset":  # coordinates far larger than the spacing
        return _sphere(rng, S) + 1000.0, _sphere(rng, N) + 1000.0, 16.0 / N
    if kind == "point":  # every node in one place
        return _sphere(rng, S) * 0.1, np.zeros((N, 3)), 0.01
    if kind == "clusters":  # most nodes in a few cells
        c = rng.uniform(-5, 5, (4, 3))
        return rng.uniform(-5, 5, (S, 3)), c[rng.integers(0, 4, N)] + 0.01 * rng.standard_normal((N, 3)), 4.0
    raise ValueError(kind)


KINDS = ["sphere", "volume", "plane", "line", "lattice", "some_ties", "outside", "offset", "point", "clusters"]


@pytest.mark.parametrize("K", [4, 8])
@pytest.mark.parametrize("kind", KINDS)
def test_skin_matches_scan(torch_dev, kind, K):
    import sho
    from starhub_amd import native
    torch = torch_dev
    for S, N in ((1, K), (63, 9), (1000, 65), (5001, 777), (4000, 4096)):
        rng = np.random.default_rng(S + 10 * K)
        s, n, r2 = _points(kind, S, N, rng)
        s, n = _four(s), _four(n)
        knn, w, c = native.skin_surfels(torch.from_numpy(s).cuda(), torch.from_numpy(n).cuda(), K, r2)
        rk, rw, rc = sho.skin(s, n, K, r2)
        print(kind, K, S, N, flush=True)
        assert np.array_equal(knn.cpu().numpy().view(np.uint16), rk), (kind, S, N)
        assert np.allclose(w.cpu().numpy(), rw, rtol=2e-5, atol=1e-7, equal_nan=True), (kind, S, N)
        assert np.array_equal(c.cpu().numpy(), rc)


@pytest.mark.parametrize("S,N", [(300007, 500), (2000, 4097), (1500, 6000)])
def test_skin_wide_and_long(torch_dev, S, N):
    """The persistent launch (more surfels than its work-groups take at once) and node sets past the grid's LDS."""
    import sho
    from starhub_amd import native
    torch = torch_dev
    rng = np.random.default_rng(N)
    s, n = _four(_sphere(rng, S)), _four(_sphere(rng, N))
    knn, w, _ = native.skin_surfels(torch.from_numpy(s).cuda(), torch.from_numpy(n).cuda(), 8, 16.0 / N)
    rk, rw, _ = sho.skin(s, n, 8, 16.0 / N)
    assert np.array_equal(knn.cpu().numpy().view(np.uint16), rk)
    assert np.allclose(w.cpu().numpy(), rw, rtol=2e-5, atol=1e-7)


@pytest.mark.parametrize("kind", ["sphere", "lattice", "some_ties"])
@pytest.mark.parametrize("S,N", [(900, 64), (900, 65), (900, 128), (900, 129), (5000, 300), (60001, 300), (300007, 300),
                                 (200, 2000)])
def test_skin_scan_rules(torch_dev, kind, S, N):
    """Both sides of the limits up to which the nodes are scanned without the grid, and surfels that the grid leaves to
    the scan: few of a work-group (a wave each), and more (a lane each)."""
    import sho
    from starhub_amd import native
    torch = torch_dev
    for K in (4, 8):
        rng = np.random.default_rng(S + N)
        s, n, r2 = _points(kind, S, N, rng)
        s, n = _four(s), _four(n)
        knn, w, _ = native.skin_surfels(torch.from_numpy(s).cuda(), torch.from_numpy(n).cuda(), K, r2)
        rk, rw, _ = sho.skin(s, n, K, r2)
        assert np.array_equal(knn.cpu().numpy().view(np.uint16), rk), K
        assert np.allclose(w.cpu().numpy(), rw, rtol=2e-5, atol=1e-7), K


def test_skin_non_finite_and_unaligned(torch_dev):
    """NaN and infinite positions take the scan's result, and outputs off a 16-byte boundary are stored as such."""
    import ctypes
    import sho
    from starhub_amd import native
    torch = torch_dev
    rng = np.random.default_rng(3)
    s, n = _four(_sphere(rng, 515)), _four(_sphere(rng, 130))
    s[7, 0], s[100, 2], s[300, 1] = np.nan, np.inf, -np.inf
    for bad in (None, np.nan, np.inf):
        m = n.copy()
        if bad is not None:
            m[[3, 77], [0, 2]] = bad
        ds, dn = torch.from_numpy(s).cuda(), torch.from_numpy(m).cuda()
        knn = torch.zeros(515 * 8 + 8, dtype=torch.int16, device="cuda")
        w = torch.zeros(515 * 8 + 8, device="cuda")
        c = torch.zeros(515 * 8 + 8, device="cuda")
        p = lambda t, off: ctypes.c_void_p(t.data_ptr() + off * t.element_size())
        native.check(native.lib().sh_skin_surfels(p(ds, 0), 515, p(dn, 0), 130, 8, ctypes.c_float(0.1), p(knn, 1),
                                                  p(w, 1), p(c, 3), ctypes.c_void_p()), "skin")
        rk, rw, rc = sho.skin(s, m, 8, 0.1)
        got = knn.cpu().numpy().view(np.uint16)
        assert np.array_equal(got[1:1 + 515 * 8].reshape(515, 8), rk)
        assert got[0] == 0 and not got[1 + 515 * 8:].any()
        assert np.allclose(w.cpu().numpy()[1:1 + 515 * 8].reshape(515, 8), rw, rtol=2e-5, atol=1e-7, equal_nan=True)
        assert np.array_equal(c.cpu().numpy()[3:3 + 515 * 8].reshape(515, 8), rc)


@pytest.mark.parametrize("K", [4, 8])
@pytest.mark.parametrize("kind", KINDS)
def test_node_graph_matches_scan(torch_dev, kind, K):
    import sho
    from starhub_amd import native
    torch = torch_dev
    for N in (K, 63, 64, 65, 200, 2048, 2051):
        rng = np.random.default_rng(N)
        _, n, r2 = _points(kind, 64, N, rng)
        n = _four(n)
        knn, w, edges, c = native.build_node_graph(torch.from_numpy(n).cuda(), K, r2)
        rk, rw, re, rc = sho.node_graph(n, K, r2)
        print(kind, K, N, flush=True)
        assert np.array_equal(knn.cpu().numpy().view(np.uint16), rk), (kind, N)
        assert np.array_equal(edges.cpu().numpy().view(np.uint16).reshape(re.shape), re), (kind, N)
        # the device rounds the last product-sum of a distance straight to 16 bits, the oracle through 32: they differ
        # where the 32-bit value lies midway between two 16-bit ones, by one unit, 2^-10 of the distance at most, and
        # exp(-d / (2 r2)) and the row's sum move by that of d / (2 r2)
        e = (n[:, None, :3] - n[rk.astype(np.int64), :3]).astype(np.float64)
        d = (e[..., 0] ** 2).astype(np.float32)
        for c3 in (1, 2):
            d = (e[..., c3] ** 2 + d).astype(np.float32)
        with np.errstate(invalid="ignore"):
            mid = np.where(d < 2.0 ** -14, (d * 2.0 ** 25) % 2 == 1, (d.view(np.uint32) & 0x1FFF) == 0x1000)
        rtol = 2e-5 + (np.where(mid, d, 0).max(1, keepdims=True) / (2 * r2) * 2.0 ** -9)
        print("rows with a midway distance", int(mid.any(1).sum()), "of", N, flush=True)
        assert np.isclose(w.cpu().numpy(), rw, rtol=rtol, atol=1e-7, equal_nan=True).all(), (kind, N)
        assert np.array_equal(c.cpu().numpy(), rc)
