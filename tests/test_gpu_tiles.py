"""The tile kernel against paths without tiles, for every tile size, FP32 and FP16 records and a last tile of a few
pixels: the matrix form with tiles of up to 32 distinct nodes (their weights whole) and of 33 to 64 (a group at a time),
the list form, which sums every tile of a small launch that holds one of more nodes or pairs, and a launch of both."""
from dataclasses import replace

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp16", [False, True])
@pytest.mark.parametrize("tile_pix", [64, 128, 256])
def test_tiles_by_node_count(tile_pix, fp16):
    """Tiles of 8 to 100 nodes and many pairs in one frame, so the list form and both ways its index is built."""
    import torch
    from starhub_amd import native, scene, workload
    assert torch.cuda.is_available()
    torch.cuda.set_device(0)
    flag = {64: native.SH_FLAG_TILE_PIX_64, 128: 0, 256: native.SH_FLAG_TILE_PIX_256}[tile_pix]
    base = scene.config_c2()
    cfg = replace(base, num_surfels=60000, num_nodes=700, width=331, height=203, fx=290.0, fy=290.0,
                  solver=replace(base.solver, gn_iterations=1, fp16=fp16))
    sc = scene.generate(cfg)
    _, prod = workload.device_frame(sc)
    K, N, idx = cfg.K, cfg.num_nodes, sc.index_map
    rng = np.random.default_rng(tile_pix)
    # bands of 64 columns whose surfels name nodes of one window each
    knn = prod["surfel_knn"].reshape(-1, K).copy()
    cover = 64 * np.arange(cfg.width // 64 + 1)
    for x0, size in zip(cover, (8, 30, 33, 48, 64, 100)):
        band = np.unique(idx[:, x0:x0 + 64])
        for s in band[band != 0xFFFFFFFF]:
            # eight different nodes: of a node named twice the tiles take the
            # last slot and the row segments each of them
            knn[s] = x0 + rng.choice(size, K, replace=False)
    prod = dict(prod, surfel_knn=knn.reshape(prod["surfel_knn"].shape))

    def solve(flags, prod=prod):
        s = native.WarpSolver(native.make_config(cfg.solver, cfg.width, cfg.height, N, K, flags=flags))
        f, _ = workload.device_frame(sc, producers=prod)
        s.process_frame(f)
        out = {n: s.debug(n, torch.float32).cpu().numpy() for n in ("blk", "rhs")}
        s.close()
        return out

    tiled, rows = solve(flag), solve(native.SH_FLAG_ROW_SEGMENTS)
    for name in ("blk", "rhs"):
        a, b = tiled[name], rows[name]
        print(tile_pix, fp16, name, "max diff", np.abs(a - b).max(), "max", np.abs(b).max(), flush=True)
        # the same products of the same records in FP32, in another order: 168
        # roundings of 2^-24 of the largest entry, all one way, reach 1e-5
        assert np.abs(a - b).max() <= 1e-5 * np.abs(b).max()

    # a weight that is not finite reaches the blocks and rows of its node's
    # pixels, and no others: the same entries as in the other path
    weights = prod["surfel_spatial"].reshape(-1, K).copy()
    row = idx[100][idx[100] != 0xFFFFFFFF]
    weights[row[::40], 2] = np.inf
    odd = dict(prod, surfel_spatial=weights.reshape(prod["surfel_spatial"].shape))
    split = native.SH_FLAG_NO_PERSISTENT_PCG  # its solve ends without exchanging what is not finite
    tiled, rows = solve(flag | split, odd), solve(native.SH_FLAG_ROW_SEGMENTS | split, odd)
    for name in ("blk", "rhs"):
        a, b = tiled[name], rows[name]
        fin = np.isfinite(b)
        print(tile_pix, fp16, name, "finite", fin.sum(), "of", fin.size, flush=True)
        assert 0 < fin.sum() < fin.size and np.array_equal(fin, np.isfinite(a))
        assert np.abs(a[fin] - b[fin]).max() <= 1e-5 * np.abs(b[fin]).max()


def _chains(tile_pix, size, fp16=False):
    """A frame whose full tiles name exactly `size` nodes each: the p-th pixel of the tile order names eight nodes in a
    row, the first of them p mod (size - 7), so any size - 7 pixels in a row name all of them, in at most 484 pairs of
    64 nodes.  Returns a solver of it by (flags, producers, scene), its scene and producers, and the pixel order."""
    import torch
    from starhub_amd import native, scene, workload
    torch.cuda.set_device(0)
    base = scene.config_c2()
    cfg = replace(base, num_surfels=60000, num_nodes=200, width=331, height=203, fx=290.0, fy=290.0, with_flow=False,
                  solver=replace(base.solver, gn_iterations=1, fp16=fp16))
    sc = scene.generate(cfg)
    there = sc.index_map != 0xFFFFFFFF
    index = sc.index_map.copy()
    index[there] = np.arange(there.sum())  # a surfel of its own for every pixel
    sc = replace(sc, index_map=index)
    _, prod = workload.device_frame(sc)

    def solve(flags, prod, scn=sc, names=("blk", "rhs")):
        s = native.WarpSolver(native.make_config(cfg.solver, cfg.width, cfg.height, cfg.num_nodes, cfg.K, flags=flags))
        s.process_frame(workload.device_frame(scn, producers=prod)[0])
        out = {n: s.debug(n, torch.int16 if n == "gpix" else torch.int32 if n == "tile_nodes" else torch.float32)
               .cpu().numpy() for n in names}
        s.close()
        return out

    flag = {64: native.SH_FLAG_TILE_PIX_64, 128: 0, 256: native.SH_FLAG_TILE_PIX_256}[tile_pix]
    pix = solve(flag, prod, names=("gpix",))["gpix"].view(np.uint16).reshape(-1, 4).astype(np.int64)
    knn = prod["surfel_knn"].reshape(-1, cfg.K).copy()
    knn[index[pix[:, 1], pix[:, 0]]] = (np.arange(len(pix)) % (size - 7))[:, None] + np.arange(cfg.K)
    return solve, sc, dict(prod, surfel_knn=knn.reshape(prod["surfel_knn"].shape)), pix, flag


@pytest.mark.parametrize("fp16", [False, True])
@pytest.mark.parametrize("size", [8, 32, 33, 63, 64, 65])
@pytest.mark.parametrize("tile_pix", [64, 128, 256])
def test_tiles_of_exact_node_counts(tile_pix, size, fp16):
    """The matrix form on both sides of its limits of 32 and 64 nodes (65: the list form), by the counts the index
    found."""
    from starhub_amd import native
    solve, _, prod, pix, flag = _chains(tile_pix, size, fp16)
    tiled = solve(flag, prod, names=("blk", "rhs", "tile_nodes"))
    nodes, full = tiled["tile_nodes"], len(pix) // tile_pix
    assert len(nodes) == -(-len(pix) // tile_pix) and (nodes[:full] == size).all() and (nodes <= size).all()
    rows = solve(native.SH_FLAG_ROW_SEGMENTS, prod)
    for name in ("blk", "rhs"):
        a, b = tiled[name], rows[name]
        print(tile_pix, size, fp16, name, "max diff", np.abs(a - b).max(), "max", np.abs(b).max(), flush=True)
        # a block's products of up to len(pix) / (size - 7) pixels in another order
        assert np.abs(a - b).max() <= 2.0 ** -24 * (len(pix) // (size - 7) + 8) * np.abs(b).max()


def test_both_tile_forms_in_a_launch():
    """Frames of 33-node tiles, enough pixels for a launch of their own, and one of 65-node tiles, which the list form
    sums: every solve has the bits it has alone."""
    import torch
    from starhub_amd import native, workload
    _, sc, prod, pix, _ = _chains(128, 33)
    _, sc2, prod2, _, _ = _chains(128, 65)
    n = 512 * 1024 // (len(pix) // 128 * 128) + 2
    frame, other = workload.device_frame(sc, producers=prod)[0], workload.device_frame(sc2, producers=prod2)[0]
    cfg, split = sc.cfg, native.SH_FLAG_NO_PERSISTENT_PCG
    conf = native.make_config(cfg.solver, cfg.width, cfg.height, cfg.num_nodes, cfg.K, flags=split)
    batch = native.BatchSolver(conf, n)
    for i in range(n):
        batch.set_inputs(i, other if i == 5 else frame)
    batch.solve(n)
    alone = []
    for f in (frame, other):
        s = native.WarpSolver(conf)
        s.process_frame(f)
        alone.append(s.node_se3())
        s.close()
    assert bool(torch.isfinite(alone[0]).all()) and not torch.equal(alone[0], alone[1])
    for i in range(n):
        assert torch.equal(batch.node_se3(i), alone[i == 5]), i
    batch.close()


@pytest.mark.parametrize("size", [8, 32, 33, 64, 65])
@pytest.mark.parametrize("tile_pix", [64, 128, 256])
def test_tiles_record_not_finite(tile_pix, size):
    """A measured normal that is NaN makes its pixel's record NaN, and so every block of two nodes that the pixel
    names, a node of weight zero too (0 x NaN), and no other block: the same entries as in the pair-major path."""
    from starhub_amd import native
    solve, sc, prod, pix, flag = _chains(tile_pix, size)
    normal = sc.measure_normal.copy()
    weights = prod["surfel_spatial"].reshape(-1, 8).copy()
    for p, slot in ((2 * len(pix) // 3, 2), (len(pix) - 3, 5)):  # one of them in the last, partial tile
        x, y, tx, ty = pix[p]
        normal[ty, tx, :3] = np.nan
        weights[sc.index_map[y, x], slot] = 0.0
    prod = dict(prod, surfel_spatial=weights.reshape(prod["surfel_spatial"].shape))
    odd = replace(sc, measure_normal=normal)
    split = native.SH_FLAG_NO_PERSISTENT_PCG  # its solve ends without exchanging what is not finite
    tiled, pairs = solve(flag | split, prod, odd), solve(native.SH_FLAG_PAIR_MAJOR | split, prod, odd)
    for name in ("blk", "rhs"):
        a, b = tiled[name], pairs[name]
        fin = np.isfinite(b)
        print(tile_pix, size, name, "finite", fin.sum(), "of", fin.size, "differ", (fin != np.isfinite(a)).sum(), flush=True)
        assert 0 < fin.sum() < fin.size and np.array_equal(fin, np.isfinite(a))
        # as in test_tiles_by_node_count, for the sums of more pixels: the
        # products of a block's up to P / (size - 7) pixels in another order
        assert np.abs(a[fin] - b[fin]).max() <= 2.0 ** -24 * (len(pix) // (size - 7) + 8) * np.abs(b[fin]).max()
