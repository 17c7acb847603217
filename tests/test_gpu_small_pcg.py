"""The PCG iterations of small systems in one cooperative launch
(csrc/pcg_small.hip) against the launches of one iteration after another."""
import numpy as np
import pytest

from libuipc_amd import abi, synth
from libuipc_amd.device import LinearSystem, rel_err

pytestmark = pytest.mark.gpu


def solve_both(ctx, ls, b, tol=1e-8, **kw):
    """one launch (the default; fits: does this system take it?), and use_graph = 0:
    plain launches"""
    out = []
    fits = kw.pop("fits", True)
    for use_graph in (1, 0):
        x = ctx.alloc(ls.n, np.float64)
        if "x_init" in kw:
            x.upload(kw["x0"])
        opts = {k: v for k, v in kw.items() if k != "x0"}
        st = ls.solve(b, x, tol=tol, use_graph=use_graph, true_residual=1, **opts)
        assert (ls.one_launch() > 0) == (fits and use_graph == 1)
        out.append((st, x.numpy()))
    return out


def check(ctx, ls, b, tol=1e-8, err=1e-6, criterion=abi.MI_CRIT_REL_RESIDUAL, **kw):
    (s1, x1), (s0, x0) = solve_both(ctx, ls, b, tol, criterion=criterion, **kw)
    assert s1["converged"] == s0["converged"] == 1
    # rounding moves a stiff system's count: at most 10% more, the bound of
    # test_mas_pcg (with float inverses it takes up to 20% fewer: the launches
    # restrict and add in float, this in double)
    assert s1["iters_exact"] <= max(s0["iters_exact"] + 2, 1.1 * s0["iters_exact"])
    # a float matrix leaves a residual of its rounding times the first residual,
    # which both have; CG's rounding spreads it by a small factor
    assert s1["rel_res_true"] < max(1e-7, 3.0 * s0["rel_res_true"])
    assert rel_err(x1, x0) < err


def dense_spd(B, per_row, seed):
    """a block-diagonally dominant system with about 2 per_row random blocks in a row"""
    rng = np.random.default_rng(seed)
    r = np.repeat(np.arange(B), per_row)
    c = rng.integers(0, B, r.size)
    lo, hi = np.minimum(r, c), np.maximum(r, c)
    off = lo != hi
    lo, hi = lo[off], hi[off]
    v = rng.standard_normal((lo.size, 9))
    rows = np.concatenate([np.arange(B), lo]).astype(np.int32)
    cols = np.concatenate([np.arange(B), hi]).astype(np.int32)
    diag = np.tile(np.eye(3).ravel() * 14.0 * per_row, (B, 1))
    return rows, cols, np.concatenate([diag, v])


@pytest.mark.parametrize("B,per_row,fits", [(1, 1, True), (63, 4, True), (64, 4, True), (65, 4, True), (700, 20, True),
                                            (2500, 30, True), (8192, 20, True), (2500, 60, False), (5000, 130, False),
                                            (16384, 6, True), (16385, 6, False)])
def test_small_pcg_rows(ctx, B, per_row, fits):
    """one row, workgroups one row short of and past 64 rows, blocks past the
    registers (3,072 per workgroup; 3,900 here), columns past LDS (2,048; 2,300),
    both, which it leaves to the launches, the most rows it takes and one more"""
    rows, cols, vals = dense_spd(B, per_row, seed=B)
    ls = LinearSystem(ctx, B)
    ls.assemble(ctx.to_device(rows), ctx.to_device(cols), ctx.to_device(vals))
    b = ctx.to_device(np.random.default_rng(1).standard_normal(3 * B))
    ls.add_preconditioner(abi.MI_PRECOND_DIAG3, 0, 3 * (B // 2))  # z = r on the other rows
    ls.assemble_preconditioners()
    check(ctx, ls, b, fits=fits)
    ls.close()


@pytest.mark.parametrize("precision,mas", [(abi.MI_FP64, abi.MI_FP64), (abi.MI_FP64, abi.MI_FP32),
                                           (abi.MI_FP32, abi.MI_FP32)])
@pytest.mark.parametrize("grid,contacts,levels", [(2, 0, 0), (5, 40, 0), (9, 900, 0), (9, 900, 1), (9, 900, 2),
                                                  (17, 2000, 0), (24, 0, 0), (25, 0, 0)])
def test_small_pcg_mas(ctx, grid, contacts, levels, precision, mas):
    """MAS over the whole vector in hierarchies of two (2^3) to five levels (17^3,
    24^3), with one and two of them applied, float and double storage; 24^3 has 13,824
    partition slots, 25^3 18,928, past the 16,384 of one launch"""
    s = synth.fem_system(grid, contacts, seed=grid + 1)
    ls = LinearSystem(ctx, s.block_rows, precision)
    ls.assemble(ctx.to_device(s.rows), ctx.to_device(s.cols), ctx.to_device(s.vals))
    ls.add_preconditioner(abi.MI_PRECOND_MAS, 0, s.n, part_ids=s.part_ids, tets=s.tets, mas_precision=mas,
                          active_levels=levels)
    ls.assemble_preconditioners()
    b = ctx.to_device(s.rhs)
    # contacts of four decades of stiffness: x to the residual times the condition
    check(ctx, ls, b, err=1e-3, fits=grid < 25)
    # from a given x0, and the rz criterion (r.z is about the residual's square)
    x0 = np.random.default_rng(3).standard_normal(s.n)
    check(ctx, ls, b, err=1e-3, x_init=1, x0=x0, fits=grid < 25)
    check(ctx, ls, b, err=1e-3, tol=1e-16, criterion=abi.MI_CRIT_RZ_RATIO, fits=grid < 25)
    ls.close()


def test_small_pcg_stops(ctx):
    """the iteration cap, the interval counts, and a NaN in b, which is found before
    the first iteration, as the launches"""
    s = synth.fem_system(9, 900, seed=2)
    ls = LinearSystem(ctx, s.block_rows)
    ls.assemble(ctx.to_device(s.rows), ctx.to_device(s.cols), ctx.to_device(s.vals))
    ls.add_preconditioner(abi.MI_PRECOND_DIAG3, 0, s.n)
    ls.assemble_preconditioners()
    b = ctx.to_device(s.rhs)
    for cap in (7.5, 530.5):  # within one launch and past its 512 iterations
        (s1, x1), (s0, x0) = solve_both(ctx, ls, b, criterion=abi.MI_CRIT_REL_RESIDUAL, tol=1e-12,
                                        max_iter_ratio=cap / s.n)
        assert [s1[k] for k in ("iters", "converged")] == [s0[k] for k in ("iters", "converged")] == [int(cap), 0]
        # up to 530 iterations of a stiff system, where rounding differences grow
        assert rel_err(x1, x0) < 1e-3
    # without contacts the counts do not depend on rounding
    free = synth.fem_system(9, 0, seed=2)
    lf = LinearSystem(ctx, free.block_rows)
    lf.assemble(ctx.to_device(free.rows), ctx.to_device(free.cols), ctx.to_device(free.vals))
    for ci in (1, 7):
        (s1, x1), (s0, x0) = solve_both(ctx, lf, ctx.to_device(free.rhs), tol=1e-6, check_interval=ci)
        assert [s1[k] for k in ("iters", "iters_exact")] == [s0[k] for k in ("iters", "iters_exact")]
        assert rel_err(x1, x0) < 1e-9
    lf.close()
    bad = s.rhs.copy()
    bad[5] = np.nan
    with pytest.raises(abi.MiError) as e:
        ls.solve(ctx.to_device(bad), ctx.alloc(s.n, np.float64))
    assert e.value.code == abi.MI_ERR_NONFINITE
    ls.close()


@pytest.mark.parametrize("precision", [abi.MI_FP64, abi.MI_FP32])
@pytest.mark.parametrize("pre", ["diag3", "mas"])
def test_small_pcg_goes_on_with_the_graph(ctx, precision, pre):
    """a solve whose launches end early (after 512 iterations here) goes on from
    the same x, r and p: an iteration count near the launches' own, and a true
    residual that agrees with the recurrence's"""
    s = synth.fem_system(9, 900, seed=2)
    ls = LinearSystem(ctx, s.block_rows, precision)
    ls.assemble(ctx.to_device(s.rows), ctx.to_device(s.cols), ctx.to_device(s.vals))
    if pre == "mas":
        ls.add_preconditioner(abi.MI_PRECOND_MAS, 0, s.n, part_ids=s.part_ids, tets=s.tets)
    else:
        ls.add_preconditioner(abi.MI_PRECOND_DIAG3, 0, s.n)
    ls.assemble_preconditioners()
    b, out = ctx.to_device(s.rhs), []
    for most in (0, 1, -1):
        ls.set_one_launch(most)
        x = ctx.alloc(s.n, np.float64)
        st = ls.solve(b, x, criterion=abi.MI_CRIT_REL_RESIDUAL, tol=1e-5, true_residual=1)
        assert st["converged"] == 1 and st["iters_exact"] > 512
        assert ls.one_launch() == (most if most >= 0 else -(-st["iters_exact"] // 512))
        out.append(st)
    graph = out[0]
    for st in out[1:]:
        # rounding moves a stiff system's count: 10%, the bound of test_mas_pcg
        assert abs(st["iters_exact"] - graph["iters_exact"]) <= 0.1 * graph["iters_exact"]
        # a float matrix leaves a residual of its rounding times the first one,
        # which the launches have too; CG's rounding spreads it by a small factor
        assert st["rel_res_true"] < max(1e-5 * 1.01, 3.0 * graph["rel_res_true"])
    ls.close()


@pytest.mark.parametrize("pre", ["diag3", "mas"])
@pytest.mark.parametrize("x_init", [0, 1])
def test_small_pcg_wait_runs_out(ctx, pre, x_init):
    """waits that end at their first look, so that the launch gives up: the solve
    starts again on the graph, from b and the given x0, and the system stays
    there until a setter is called"""
    s = synth.fem_system(9, 0, seed=2)
    ls = LinearSystem(ctx, s.block_rows)
    ls.assemble(ctx.to_device(s.rows), ctx.to_device(s.cols), ctx.to_device(s.vals))
    if pre == "mas":
        ls.add_preconditioner(abi.MI_PRECOND_MAS, 0, s.n, part_ids=s.part_ids, tets=s.tets)
    else:
        ls.add_preconditioner(abi.MI_PRECOND_DIAG3, 0, s.n)
    ls.assemble_preconditioners()
    b = ctx.to_device(s.rhs)
    x0 = np.random.default_rng(5).standard_normal(s.n)

    def solve():
        x = ctx.to_device(x0)
        st = ls.solve(b, x, criterion=abi.MI_CRIT_REL_RESIDUAL, tol=1e-8, x_init=x_init, true_residual=1)
        assert st["converged"] == 1 and st["rel_res_true"] < 1.01e-8
        return st, x.numpy()

    ls.set_one_launch(0)
    want, xw = solve()
    ls.set_one_launch(-1)
    ls.set_one_launch_wait(0)
    for _ in range(2):  # the one that gives up, and the next one
        st, x = solve()
        assert ls.one_launch() == 0
        # the same kernels on the same inputs; the MAS sums have no fixed order
        assert st["iters_exact"] == want["iters_exact"] and rel_err(x, xw) < 1e-9
    ls.set_one_launch_wait(-1)
    st, x = solve()
    assert ls.one_launch() == 1 and rel_err(x, xw) < 1e-6
    ls.close()


@pytest.mark.parametrize("pre", ["diag3", "mas"])
@pytest.mark.parametrize("hubs,reach,fits", [(1, 0, True), (1, 3900, True), (2, 1500, False), (8, 450, False),
                                             (60, 900, False)])
def test_small_pcg_dense_rows(ctx, pre, hubs, reach, fits):
    """`hubs` rows of one workgroup, each coupled to `reach` others: one long row
    stays on the one launch, several go to the launches (whose SpMV is split by
    blocks, not by rows), and so does the system's next solve; after an assembly
    without them it is on the one launch again"""
    s = synth.fem_system(16, 0, seed=2)
    rng = np.random.default_rng(hubs)
    rows, cols, vals = [s.rows], [s.cols], [s.vals]
    # rows that share a workgroup in the caller's order and in the partition's
    hub = np.arange(640, 704)[:hubs] if pre == "diag3" else np.argsort(s.part_ids, kind="stable")[640:640 + hubs]
    for h in hub.astype(np.int32):
        j = np.setdiff1d(rng.choice(s.block_rows, reach, replace=False), [h]).astype(np.int32)
        g = rng.standard_normal((j.size, 3))
        g /= np.linalg.norm(g, axis=1)[:, None]
        k = (g[:, :, None] * g[:, None, :]).reshape(-1, 9)
        at = np.full(j.size, h, np.int32)
        rows += [at, j, np.minimum(at, j)]
        cols += [at, j, np.maximum(at, j)]
        vals += [k, k, -k]
    ls = LinearSystem(ctx, s.block_rows)
    keep = [ctx.to_device(np.concatenate(v)) for v in (rows, cols, vals)]
    ls.assemble(*keep)
    if pre == "mas":
        ls.add_preconditioner(abi.MI_PRECOND_MAS, 0, s.n, part_ids=s.part_ids, tets=s.tets)
    else:
        ls.add_preconditioner(abi.MI_PRECOND_DIAG3, 0, s.n)
    ls.assemble_preconditioners()
    b = ctx.to_device(s.rhs)
    for _ in range(2):
        check(ctx, ls, b, fits=fits)
    free = [ctx.to_device(v) for v in (s.rows, s.cols, s.vals)]
    ls.assemble(*free)
    ls.assemble_preconditioners()
    ls.solve(b, ctx.alloc(s.n, np.float64), criterion=abi.MI_CRIT_REL_RESIDUAL, tol=1e-8)
    assert ls.one_launch() == 1
    ls.close()


@pytest.mark.parametrize("pre", ["diag3", "mas"])
def test_small_pcg_not_finite(ctx, pre):
    """a NaN in an off-diagonal block: r0.z0 is finite, the first iteration's r.z is
    not, and the launch ends there with the launches' error"""
    s = synth.fem_system(9, 900, seed=2)
    vals = s.vals.copy()
    # of two vertices in different parts: no preconditioner's cluster holds it
    at = np.flatnonzero((s.rows != s.cols) & (s.part_ids[s.rows] != s.part_ids[s.cols]))[7]
    vals[at, 4] = np.nan
    ls = LinearSystem(ctx, s.block_rows)
    ls.assemble(ctx.to_device(s.rows), ctx.to_device(s.cols), ctx.to_device(vals))
    if pre == "mas":
        ls.add_preconditioner(abi.MI_PRECOND_MAS, 0, s.n, part_ids=s.part_ids, tets=s.tets, active_levels=1)
    else:
        ls.add_preconditioner(abi.MI_PRECOND_DIAG3, 0, s.n)
    ls.assemble_preconditioners()
    b, text = ctx.to_device(s.rhs), []
    for use_graph in (1, 0):
        with pytest.raises(abi.MiError) as e:
            ls.solve(b, ctx.alloc(s.n, np.float64), tol=1e-8, use_graph=use_graph)
        assert e.value.code == abi.MI_ERR_NONFINITE and ls.one_launch() == use_graph
        text.append(str(e.value))
    assert "at iteration 1" in text[0] and "at iteration" in text[1]
    ls.close()


def test_small_pcg_survives_the_shape_tuner(ctx, monkeypatch):
    """a system whose solves run in one launch keeps the full BSR when its SpMV
    shapes are timed, also where the windows' products are faster (a timer that
    makes every shape faster than the one before); one without a solve is free"""
    from libuipc_amd import hip_events
    from libuipc_amd.tune import tune_spmv_shape

    class Timer:
        shapes = 0

        def __init__(self, stream):
            pass

        def start(self):
            Timer.shapes += 1

        def stop(self):
            return 1.0 / Timer.shapes

    monkeypatch.setattr(hip_events, "EventTimer", Timer)
    s = synth.fem_system(16, 0, seed=2)
    ls = LinearSystem(ctx, s.block_rows)
    ls.add_preconditioner(abi.MI_PRECOND_MAS, 0, s.n, part_ids=s.part_ids, tets=s.tets)
    ls.assemble(ctx.to_device(s.rows), ctx.to_device(s.cols), ctx.to_device(s.vals))
    ls.assemble_preconditioners()
    b, x = ctx.to_device(s.rhs), ctx.alloc(s.n, np.float64)
    assert tune_spmv_shape(ls, b, reps=2)["best"] >= 0
    ls.set_spmv_shape(abi.MI_SPMV_SHAPE_AUTO)
    ls.assemble_preconditioners()
    ls.solve(b, x, tol=1e-6)
    assert ls.one_launch() == 1
    Timer.shapes = 0
    t = tune_spmv_shape(ls, b, reps=2)
    assert t["best"] == abi.MI_SPMV_SHAPE_FULL and len(t["table"]) > 1
    ls.solve(b, x, tol=1e-6)
    assert ls.one_launch() == 1
    ls.close()
