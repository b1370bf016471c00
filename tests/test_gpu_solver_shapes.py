"""The Arnoldi kernels at the edges of their tiles: vector lengths off the
16-byte loads, bases on either side of the 8-vector tiles, cycles that end by
convergence, by their length or by an exhausted Krylov space."""
import numpy as np
import pytest

from oracle import orc
from tests import problems as pb
from tests.test_gpu_solver import _pressure_system  # noqa: F401
from tests.test_gpu_solver import ctx, nw  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu


def _system(nw, ctx, shape):
    nx, ny, nz = shape
    P = pb.Problem(nx, ny, nz, stretch=1.1, jitter=0.15, seed=nx + ny)
    P.upload(ctx)
    ctx.build_graph(1)
    o = nw.continuity_defaults()
    ctx.assemble_continuity(o)
    top = np.where(np.abs(P.coords[:, 2] - 1.0) < 1e-12)[0].astype(np.int32)
    ctx.field_upload(nw.F_DIFF_FLUX_COEFF, np.zeros(P.n))
    ctx.apply_dirichlet(top, nw.F_PRESSURE, nw.F_DIFF_FLUX_COEFF, 0, 1)
    A = P.oracle_continuity(pb.to_orc_continuity(o))
    A.apply_dirichlet(top, 0, 1, P.p, np.zeros(P.n))
    return P, A


# 45 (odd), 385 (one block and a rest), 1326 (= 2 mod 4), 9537 nodes
@pytest.mark.parametrize("shape", [(4, 2, 2), (10, 6, 4), (16, 12, 5), (32, 16, 16)])
@pytest.mark.parametrize("kspace", [1, 7, 8, 9, 17, 40])
def test_one_cycle_reaches_the_minimal_residual(nw, ctx, shape, kspace):
    """The residual norm after one whole cycle is the minimum over the Krylov
    space, a number that does not depend on how the basis was made: FP64
    rounding (a few 1e-15 per entry, grown by the basis' departure from
    orthogonality, of the same size under two Gram-Schmidt passes) leaves it
    to 1e-9 while it is above 1e-6 of the right-hand side."""
    P, A = _system(nw, ctx, shape)
    st = ctx.solve(nw.solver_cfg(kspace=kspace, max_iters=kspace, tol=1e-13,
                                 precond=nw.PREC_JACOBI), raise_on_noconv=False)
    r = A.rhs - A.spmv(ctx.solution())
    rel = np.linalg.norm(r) / np.linalg.norm(A.rhs)
    xo, so = A.gmres(A.rhs, kspace=kspace, max_iters=kspace, tol=1e-13, precond=1)
    ref = np.linalg.norm(A.rhs - A.spmv(xo)) / np.linalg.norm(A.rhs)
    assert st.iters <= kspace and st.final_rel == pytest.approx(rel, rel=1e-6, abs=1e-14)
    assert rel == pytest.approx(ref, rel=1e-9, abs=1e-12)


@pytest.mark.parametrize("mode,target", [(0, 1e-10), (1, 1e-8)])
@pytest.mark.parametrize("prec", [0, 1, 2, 3])
def test_cycles_end_where_the_residual_says(nw, ctx, mode, target, prec):
    """Cycles that stop inside (converged) after several whole ones: the
    step that ran ahead of the decision must leave no trace."""
    P, A = _system(nw, ctx, (12, 9, 8))
    cfg = nw.solver_cfg(kspace=9, max_iters=3000, tol=target, precond=prec, mode=mode,
                        inner_tol=1e-4, cheb_degree=3, cheb_ratio=20.0,
                        reuse_preconditioner=0)
    st = ctx.solve(cfg)
    x = ctx.solution()
    assert st.converged and st.iters > 0
    assert np.linalg.norm(A.rhs - A.spmv(x)) <= 1.0001 * target * np.linalg.norm(A.rhs)
    again = ctx.solve(cfg)
    np.testing.assert_array_equal(ctx.solution(), x)
    assert again.iters == st.iters


def test_exhausted_krylov_space(nw, ctx):
    """8 nodes, 4 of them Dirichlet: the space ends before the cycle does."""
    P, A = _system(nw, ctx, (1, 1, 1))
    st = ctx.solve(nw.solver_cfg(kspace=30, max_iters=60, tol=1e-12))
    xd = orc.dense_solve(A.dense(), A.rhs)
    assert st.converged and st.iters <= 8
    np.testing.assert_allclose(ctx.solution(), xd, rtol=0, atol=1e-9 * np.abs(xd).max())


@pytest.mark.parametrize("shape", [(4, 2, 2), (10, 9, 8), (11, 10, 9), (22, 21, 20)])
@pytest.mark.parametrize("mode", [0, 1])
def test_amg_levels(nw, ctx, shape, mode):
    """One level (solved directly), just below and above the direct solve's
    size, and several levels, the hierarchy reused for another matrix (its
    diagonal then is not the one the columns are scaled by)."""
    P, A = _system(nw, ctx, shape)
    tol = 1e-10 if mode == 0 else 1e-8
    cfg = nw.solver_cfg(kspace=30, max_iters=300, tol=tol, precond=nw.PREC_AMG, mode=mode,
                        inner_tol=1e-4, reuse_preconditioner=0)
    st = ctx.solve(cfg)
    levels = ctx.amg_levels()
    assert len(levels) == st.precond_levels
    if P.n <= 1000:
        assert st.precond_levels == 1 and st.iters <= (2 if mode == 0 else 6)
    r = A.rhs - A.spmv(ctx.solution())
    assert st.converged and np.linalg.norm(r) <= 1.0001 * tol * np.linalg.norm(A.rhs)
    # another time step, near enough for the smoothers' intervals
    o = nw.continuity_defaults(dt=0.95)
    ctx.assemble_continuity(o)
    top = np.where(np.abs(P.coords[:, 2] - 1.0) < 1e-12)[0].astype(np.int32)
    ctx.apply_dirichlet(top, nw.F_PRESSURE, nw.F_DIFF_FLUX_COEFF, 0, 1)
    cfg.reuse_preconditioner = 1
    s2 = ctx.solve(cfg)
    B = P.oracle_continuity(pb.to_orc_continuity(o))
    B.apply_dirichlet(top, 0, 1, P.p, np.zeros(P.n))
    r = B.rhs - B.spmv(ctx.solution())
    assert s2.converged and np.linalg.norm(r) <= 1.0001 * tol * np.linalg.norm(B.rhs)


@pytest.mark.parametrize("mode, shape", [(0, (97, 95, 101)), (1, (97, 95, 101)),
                                         (0, (104, 103, 102))])
def test_amg_levels_of_every_layout(nw, ctx, mode, shape):
    """Large enough for sliced ELL and wide CSR levels: two lanes per row; a
    wave per row (a restriction of more than 32 entries a row, two or more for
    each row of the finer level); a row count that the 8 dies do not share
    evenly, within one round of their stretches (8 x 131072 rows) and past it."""
    P, A = _system(nw, ctx, shape)
    tol = 1e-8
    st = ctx.solve(nw.solver_cfg(kspace=30, max_iters=300, tol=tol, precond=nw.PREC_AMG,
                                 mode=mode, inner_tol=1e-4))
    levels = [tuple(l)[:2] for l in ctx.amg_levels()]
    assert any(200000 <= n < 1000000 and 8 * n <= nnz <= 25 * n for n, nnz in levels[1:-1]), levels
    assert any(f > 16 * c for (f, _), (c, _) in zip(levels[1:], levels[2:])), levels
    r = A.rhs - A.spmv(ctx.solution())
    assert st.converged and np.linalg.norm(r) <= 1.0001 * tol * np.linalg.norm(A.rhs)


@pytest.mark.parametrize("mode,prec", [(0, 3), (1, 3), (0, 1), (1, 2)])
def test_last_slice_of_one_row(nw, ctx, mode, prec):
    """65^3 nodes: the fine matrix in offset form up to a last slice of a
    single row, whose 63 other lanes read the row's own columns."""
    P, A = _system(nw, ctx, (64, 64, 64))
    assert P.n % 64 == 1
    tol = 1e-8
    st = ctx.solve(nw.solver_cfg(kspace=50, max_iters=400, tol=tol, precond=prec, mode=mode,
                                 inner_tol=1e-4, cheb_degree=4, cheb_ratio=30.0),
                   raise_on_noconv=False)
    x = ctx.solution()
    rel = np.linalg.norm(A.rhs - A.spmv(x)) / np.linalg.norm(A.rhs)
    assert st.final_rel == pytest.approx(rel, rel=1e-3)
    assert rel <= 1.0001 * tol if prec == 3 else rel < 0.1


@pytest.mark.parametrize("mode", [0, 1])
def test_refused_matrix_leaves_no_hierarchy(nw, ctx, mode):
    """An AMG solve that a zero diagonal ends, then one on the good matrix
    with reuse on: its hierarchy must be of that matrix, whose columns it
    scales."""
    P, A = _system(nw, ctx, (12, 11, 10))
    cfg = nw.solver_cfg(kspace=30, max_iters=200, tol=1e-8, precond=nw.PREC_AMG, mode=mode,
                        inner_tol=1e-4, reuse_preconditioner=1)
    ctx.reset_rows([P.n // 2], 0, 1, diag=0.0)
    with pytest.raises(nw.NwError) as ei:
        ctx.solve(cfg)
    assert ei.value.code == nw.E_NONFINITE
    ctx.assemble_continuity(nw.continuity_defaults())  # the same graph
    top = np.where(np.abs(P.coords[:, 2] - 1.0) < 1e-12)[0].astype(np.int32)
    ctx.apply_dirichlet(top, nw.F_PRESSURE, nw.F_DIFF_FLUX_COEFF, 0, 1)
    st = ctx.solve(cfg)
    r = A.rhs - A.spmv(ctx.solution())
    assert st.converged and np.linalg.norm(r) <= 1.0001e-8 * np.linalg.norm(A.rhs)


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("shape,sliced", [((67, 66, 65), False), ((76, 75, 74), True)])
def test_amg_levels_about_the_sliced_ell_line(nw, ctx, mode, shape, sliced):
    """A level on either side of the 70 thousand rows from which levels are in
    sliced ELL form, two lanes per row."""
    P, A = _system(nw, ctx, shape)
    tol = 1e-8
    st = ctx.solve(nw.solver_cfg(kspace=30, max_iters=300, tol=tol, precond=nw.PREC_AMG,
                                 mode=mode, inner_tol=1e-4))
    n, nnz = tuple(ctx.amg_levels()[1])[:2]
    assert 8 * n <= nnz <= 25 * n and (n >= 70000) == sliced, (n, nnz)
    r = A.rhs - A.spmv(ctx.solution())
    assert st.converged and np.linalg.norm(r) <= 1.0001 * tol * np.linalg.norm(A.rhs)
