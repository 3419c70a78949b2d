"""The linear-solver plug-in (sh_block_pcg_*, sh_spmv_*: BlockPCG<6> over an
ApplySpMVBase<6> operator, BlockPCG.h:55-73, ApplySpMVBase.h:22-36) through
the C-ABI, on C1's first GN system, against the oracle's restatement of the
same solve (FP64, on the same FP32-rounded matrix, inverse diagonal and b).

Bars: 10 iterations from zero and from a non-zero x_init within 1e-3 of
max |x| (the plug-in keeps FP32 vectors, as the reference does, with FP64
dots, alpha and beta: the FP32 recurrences drift by a few 1e-4 over 10
iterations on this system); the same solve through a host callback operator, bit
for bit; the solver's own operator (sh_solver_spmv_ops) on its own FP32
system within 1e-3; the convergence-checked solve stopping where the
oracle's delta history crosses epsilon^2 delta_0."""
from dataclasses import replace

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def c1_system():
    import torch
    import sho
    from block_system import block_csr_of
    from starhub_amd import scene, workload
    assert torch.cuda.is_available()
    torch.cuda.set_device(0)
    cfg = scene.config_c1()
    sc = scene.generate(cfg)
    frame, prod = workload.device_frame(sc)
    params = replace(cfg.solver, gn_iterations=1)
    res = sho.solve(workload.host_inputs(sc, prod), params, 64, sho.max_threads())
    N = cfg.num_nodes
    rp, col, blk, dinv, b = block_csr_of(res, N)
    f32 = lambda a: a.astype(np.float32)
    return dict(sc=sc, frame=frame, prod=prod, params=params, N=N, rp=rp, col=col, blk=f32(blk), dinv=f32(dinv),
                b=f32(b), torch=torch)


def _dev(torch, a):
    a = np.ascontiguousarray(a)
    if a.dtype == np.uint32:
        return torch.from_numpy(a.view(np.int32)).cuda()
    return torch.from_numpy(a).cuda()


def _rel(x, ref):
    return float(np.abs(x - ref).max() / np.abs(ref).max())


def test_block_pcg_zero_and_nonzero_init(c1_system):
    import sho
    from starhub_amd import native
    s = c1_system
    torch, N = s["torch"], s["N"]
    A = native.BlockCsr(_dev(torch, s["rp"]), _dev(torch, s["col"]), _dev(torch, s["blk"]))
    assert A.check() == 0
    pcg = native.BlockPCG(6 * N)
    dinv, b = _dev(torch, s["dinv"]), _dev(torch, s["b"])
    x = torch.zeros(6 * N, device="cuda")
    assert pcg.set_input(dinv, A.ops(), b, x) == 0
    pcg.solve(10, zero_init=True)
    ref, hist = sho.block_pcg(s["rp"], s["col"], s["blk"], s["dinv"], s["b"], iters=10)
    err = _rel(x.cpu().numpy(), ref)
    print("block pcg zero init rel err", err, flush=True)
    assert err <= 1e-3
    dh = pcg.delta_history()
    assert dh.shape == (11,) and np.allclose(dh, hist, rtol=1e-3, atol=1e-6 * hist[0])
    rng = np.random.default_rng(6)
    x0 = (rng.standard_normal(6 * N) * np.abs(ref).max()).astype(np.float32)
    x.copy_(torch.from_numpy(x0))
    pcg.solve(10, zero_init=False)
    ref_n, _ = sho.block_pcg(s["rp"], s["col"], s["blk"], s["dinv"], s["b"], x0=x0, iters=10, zero_init=False)
    err = _rel(x.cpu().numpy(), ref_n)
    print("block pcg non-zero init rel err", err, flush=True)
    assert err <= 1e-3
    # from the converged solution it stays (r = b - A x ~ 0)
    x_star, _ = sho.block_pcg(s["rp"], s["col"], s["blk"], s["dinv"], s["b"], iters=6 * N)
    x.copy_(torch.from_numpy(x_star.astype(np.float32)))
    pcg.solve(3, zero_init=False)
    assert _rel(x.cpu().numpy(), x_star) <= 1e-3


def test_block_pcg_callback_operator_same_bits(c1_system):
    """A host callback operator (the ApplySpMVBase virtuals as function
    pointers, here forwarding to the block-CSR product) gives the bits of the
    built-in operator; without InitResidual the solver forms b - A x itself,
    to the same bits as the operator's own InitResidual."""
    from starhub_amd import native
    s = c1_system
    torch, N = s["torch"], s["N"]
    A = native.BlockCsr(_dev(torch, s["rp"]), _dev(torch, s["col"]), _dev(torch, s["blk"]))
    dinv, b = _dev(torch, s["dinv"]), _dev(torch, s["b"])
    calls = []

    @native.SPMV_APPLY_FN
    def apply(user, xp, yp, stream):
        calls.append(1)
        return A.apply(xp, yp)

    cb = native.SpmvOps(None, 6 * N, apply, native.SPMV_INIT_FN())
    rng = np.random.default_rng(8)
    x0 = rng.standard_normal(6 * N).astype(np.float32) * 1e-3
    outs = []
    for ops in (A.ops(), cb):
        for zero in (True, False):
            pcg = native.BlockPCG(6 * N)
            x = torch.from_numpy(x0.copy()).cuda()
            assert pcg.set_input(dinv, ops, b, x) == 0
            pcg.solve(10, zero_init=zero)
            outs.append(x.cpu().numpy())
            pcg.close()
    assert len(calls) == 10 + 11  # ApplySpMV per iteration, plus once for b - A x_init
    assert np.array_equal(outs[0], outs[2]) and np.array_equal(outs[1], outs[3])


def test_block_pcg_on_the_solvers_own_system(c1_system):
    """sh_solver_spmv_ops hands the solver's last-iteration system to the
    plug-in (materialised and matrix-free), with the solver's inverse diagonal
    rounded to FP32 and its right-hand side: within 1e-3 of the oracle's
    solve of the FP64 system (the GPU's system is its own FP32 assembly, whose
    blocks differ from the oracle's by up to 1e-5 relative)."""
    import sho
    from starhub_amd import native
    s = c1_system
    torch, N = s["torch"], s["N"]
    solver = native.WarpSolver(native.make_config(s["params"], s["sc"].cfg.width, s["sc"].cfg.height, N, 8))
    solver.process_frame(s["frame"])
    dinv = solver.debug("dinv", torch.float64).float()
    b = solver.debug("rhs", torch.float32)
    ref, _ = sho.block_pcg(s["rp"], s["col"], s["blk"].astype(np.float64), s["dinv"].astype(np.float64),
                           s["b"].astype(np.float64), iters=10)
    for mf in (False, True):
        pcg = native.BlockPCG(6 * N)
        x = torch.zeros(6 * N, device="cuda")
        assert pcg.set_input(dinv, native.solver_spmv_ops(solver, mf), b, x) == 0
        pcg.solve(10)
        err = _rel(x.cpu().numpy(), ref)
        print("solver operator", "matrix-free" if mf else "materialised", "rel err", err, flush=True)
        assert err <= 1e-3
        pcg.close()
    solver.close()


def test_block_pcg_converge_checked_and_errors(c1_system):
    import sho
    from starhub_amd import native
    s = c1_system
    torch, N = s["torch"], s["N"]
    A = native.BlockCsr(_dev(torch, s["rp"]), _dev(torch, s["col"]), _dev(torch, s["blk"]))
    dinv, b = _dev(torch, s["dinv"]), _dev(torch, s["b"])
    _, hist = sho.block_pcg(s["rp"], s["col"], s["blk"], s["dinv"], s["b"], iters=40)
    eps = 0.1
    want = int(np.argmax(np.abs(hist[1:]) < eps * eps * abs(hist[0]))) + 1
    assert abs(hist[want]) < eps * eps * abs(hist[0]) and want < 40
    pcg = native.BlockPCG(6 * N)
    x = torch.zeros(6 * N, device="cuda")
    assert pcg.set_input(dinv, A.ops(), b, x) == 0
    n = pcg.solve_converge_checked(40, True, eps)
    print("converge-checked iterations", n, "oracle", want, flush=True)
    assert abs(n - want) <= 1
    assert pcg.delta_history().shape == (n + 1,)
    small = native.BlockPCG(6 * (N - 1))
    assert small.set_input(dinv, A.ops(), b, x) == 2  # SH_E_CAPACITY
    bad_col = s["col"].copy()
    bad_col[5] = N
    Abad = native.BlockCsr(_dev(torch, s["rp"]), _dev(torch, bad_col), _dev(torch, s["blk"]))
    assert Abad.check() == 1  # SH_E_ARG: a column out of range, found before any product reads it


@pytest.mark.parametrize("rows,degree", [(1, 1), (2, 2), (7, 5), (11, 6), (41, 11), (40, 24), (300, 31), (8201, 4)])
def test_block_csr_sizes(rows, degree):
    """Rows that leave waves, work-groups and turns partly filled, rows of no
    block, of one trip and of several: the product is the exact sum rounded
    once (2^-24 of it, and an FP64 sum's own rounding), and the built-in
    operator's fused iteration gives the callback's bits."""
    import torch
    from starhub_amd import native
    torch.cuda.set_device(0)
    rng = np.random.default_rng(rows)
    cols = []
    for r in range(rows):
        near = rng.integers(0, rows, rng.integers(0, degree) if r % 5 else degree - 1)
        cols.append(np.unique(np.concatenate([near, [r]])))
    rp = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.uint32)
    col = np.concatenate(cols).astype(np.uint32)
    blk = (rng.standard_normal((len(col), 6, 6)) * 0.02).astype(np.float32)
    own = np.repeat(np.arange(rows), np.diff(rp)) == col
    blk[own] = (0.5 * (blk[own] + blk[own].transpose(0, 2, 1)) + np.eye(6) * 3).astype(np.float32)
    dinv = np.linalg.inv(blk[own].astype(np.float64)).astype(np.float32)
    b = rng.standard_normal(6 * rows).astype(np.float32)
    A = native.BlockCsr(_dev(torch, rp), _dev(torch, col), _dev(torch, blk.reshape(-1)))
    assert A.check() == 0
    v, y = _dev(torch, b), torch.full((6 * rows,), float("nan"), device="cuda")
    assert A.apply(v.data_ptr(), y.data_ptr()) == 0
    prod = blk.astype(np.float64) * b.reshape(-1, 6)[col][:, None, :]
    exact, size = (np.zeros((rows, 6)) for _ in range(2))
    np.add.at(exact, np.repeat(np.arange(rows), np.diff(rp)), prod.sum(2))
    np.add.at(size, np.repeat(np.arange(rows), np.diff(rp)), np.abs(prod).sum(2))
    torch.cuda.synchronize()
    err = np.abs(y.cpu().numpy().reshape(-1, 6) - exact)
    print("rows", rows, "blocks", len(col), "max err", err.max(), flush=True)
    assert (err <= 2.0 ** -24 * np.abs(exact) + 2.0 ** -44 * size).all()

    if rows > 1:  # the last row emptied
        end = int(rp[-2])
        rp2 = np.concatenate([rp[:-1], rp[-2:-1]])
        cut = native.BlockCsr(_dev(torch, rp2), _dev(torch, col[:end]), _dev(torch, blk[:end].reshape(-1)))
        y2 = torch.full_like(y, float("nan"))
        assert cut.apply(v.data_ptr(), y2.data_ptr()) == 0
        torch.cuda.synchronize()
        assert torch.equal(y2[:-6], y[:-6]) and (y2[-6:] == 0).all()

    @native.SPMV_APPLY_FN
    def apply(user, xp, yp, stream):
        return A.apply(xp, yp)

    outs = []
    for ops in (A.ops(), native.SpmvOps(None, 6 * rows, apply, native.SPMV_INIT_FN())):
        pcg = native.BlockPCG(6 * rows)
        x = torch.full((6 * rows,), 0.25, device="cuda")
        assert pcg.set_input(_dev(torch, dinv), ops, v, x) == 0
        pcg.solve(4, zero_init=False)
        outs.append((x.cpu().numpy(), pcg.delta_history()))
        pcg.close()
    assert np.isfinite(outs[0][0]).all() and outs[0][1].shape == (5,)
    assert np.array_equal(outs[0][0], outs[1][0]) and np.array_equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("rows,degree", [(8192, 40), (8193, 15), (8193, 17), (9001, 40), (41003, 6), (45001, 25)])
def test_block_csr_long_systems(rows, degree):
    """Both sides of 8192 rows and of 16 blocks a row, more rows than the row kernels' work-groups take in a turn, and
    enough blocks that the built-in product is a kernel of its own: the product is the exact sum rounded once, and the
    built-in operator's iterations are the callback's (where their sums of d.q group rows alike, bit for bit)."""
    import torch
    from starhub_amd import native
    torch.cuda.set_device(0)
    rng = np.random.default_rng(rows + degree)
    step = np.sort(rng.choice(np.arange(1, 3 * degree + 9), degree - 1, replace=False))
    col = np.sort((np.arange(rows)[:, None] + np.concatenate([[0], step])[None]) % rows, 1)
    own = torch.from_numpy(col == np.arange(rows)[:, None]).cuda()
    g = torch.Generator(device="cuda").manual_seed(rows)
    blk = torch.randn(rows, degree, 6, 6, generator=g, device="cuda") * 0.02
    blk[own] = 0.5 * (blk[own] + blk[own].transpose(1, 2)) + 3 * torch.eye(6, device="cuda")
    dinv = torch.linalg.inv(blk[own].double().cpu()).float().cuda().contiguous()
    b = torch.randn(6 * rows, generator=g, device="cuda")
    A = native.BlockCsr(_dev(torch, np.arange(rows + 1, dtype=np.uint32) * degree), _dev(torch, col.astype(np.uint32).reshape(-1)),
                        blk.reshape(-1))
    assert A.check() == 0
    y = torch.full_like(b, float("nan"))
    assert A.apply(b.data_ptr(), y.data_ptr()) == 0
    prod = blk.double() * b.double().view(-1, 6)[torch.from_numpy(col).cuda()][:, :, None, :]
    exact, size = prod.sum((1, 3)).reshape(-1), prod.abs().sum((1, 3)).reshape(-1)
    torch.cuda.synchronize()
    err = (y.double() - exact).abs()
    print("rows", rows, "degree", degree, "max err", err.max().item(), flush=True)
    assert bool((err <= 2.0 ** -24 * exact.abs() + 2.0 ** -44 * size).all())

    @native.SPMV_APPLY_FN
    def apply(user, xp, yp, stream):
        return A.apply(xp, yp)

    outs = []
    for ops in (A.ops(), native.SpmvOps(None, 6 * rows, apply, native.SPMV_INIT_FN())):
        pcg = native.BlockPCG(6 * rows)
        x = torch.full((6 * rows,), 0.25, device="cuda")
        assert pcg.set_input(dinv, ops, b, x) == 0
        pcg.solve(4, zero_init=False)
        outs.append((x.cpu().numpy(), pcg.delta_history()))
        n = pcg.solve_converge_checked(40, True, 1e-3)
        outs[-1] += (x.cpu().numpy(), n)
        pcg.close()
    assert np.isfinite(outs[0][0]).all() and outs[0][1].shape == (5,) and 0 < outs[0][3] < 40
    if rows <= 8192 or degree <= 16 or rows * degree >= 1 << 20:
        assert all(np.array_equal(u, v) for u, v in zip(*outs))
    else:  # sums of d.q in another order: 2^-53 of them, a rounding of 2^-24 in a few entries of a vector
        assert all(np.allclose(u, v, rtol=1e-5, atol=1e-6) for u, v in zip(*outs))
    # the residual the converge-checked solve stopped at
    assert A.apply(x.data_ptr(), y.data_ptr()) == 0
    r = (b - y).view(-1, 6, 1)
    torch.cuda.synchronize()
    assert float((r * (dinv.view(-1, 6, 6) @ r)).sum()) <= 1.01e-6 * float((b.view(-1, 6, 1) * (dinv.view(-1, 6, 6) @ b.view(-1, 6, 1))).sum())
