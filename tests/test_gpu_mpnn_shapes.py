"""The fused network layers at the edges of their tiles: fewer nodes than a
tile of 16, partial tiles, fewer tiles than the eight stretches of the grid,
rows of more than the eight slots a tile loads ahead (mixed meshes), both
widths and several depths."""
import ctypes

import numpy as np
import pytest

from oracle import orc
from tests import problems as pb
from tests.test_gpu_mpnn import _solved_pair
from tests.test_gpu_mpnn import ctx, nw  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu


def _system(nw, ctx, P):
    P.upload(ctx)
    ctx.build_graph(1)
    ctx.assemble_continuity(nw.continuity_defaults())
    top = np.where(P.coords[:, 2] > P.coords[:, 2].max() - 1e-12)[0].astype(np.int32)
    ctx.field_upload(nw.F_PRESSURE, np.zeros(P.n))
    ctx.field_upload(nw.F_DIFF_FLUX_COEFF, np.zeros(P.n))
    ctx.apply_dirichlet(top, nw.F_PRESSURE, nw.F_DIFF_FLUX_COEFF, 0, 1)
    rp, cols, vals, rhs = ctx.download()
    D = np.zeros((P.n, P.n))
    for r in range(P.n):
        D[r, cols[rp[r]:rp[r + 1]]] = vals[rp[r]:rp[r + 1]]
    return orc.CsrSystem.from_dense(D, rhs)


# 12, 18, 130, 150 nodes; a mixed box (rows of up to 20 slots)
@pytest.mark.parametrize("mesh", [(2, 1, 1), (2, 2, 1), (4, 12, 1), (4, 4, 5), "mixed"])
@pytest.mark.parametrize("H,L", [(32, 1), (32, 4), (64, 1), (64, 2)])
def test_layers_match_oracle(nw, ctx, mesh, H, L):
    if mesh == "mixed":
        P = pb.Problem(4, 4, 4, jitter=0.1, seed=3, mixed=(0.5, 0.3))
    else:
        nx, ny, nz = mesh
        P = pb.Problem(nx, ny, nz, stretch=1.1, jitter=0.1, seed=5)
    A = _system(nw, ctx, P)
    hist, xs = _solved_pair(nw, ctx, A, 21)
    net = nw.Mpnn(ctx, H, L, seed=3)
    rng = np.random.default_rng(H + L)
    p = rng.normal(size=net.nparams) * 0.3
    p = p.astype(np.float32).astype(np.float64)
    net.params = p
    net.record()
    loss, g = net.loss_grad(0)
    w = orc.mpnn_slot_weights(A)
    feat, sc = orc.mpnn_features(A, A.rhs, *hist)
    target = (xs - orc.mpnn_base_guess(*hist)) / sc[4]
    loss_o, g_o = orc.mpnn_loss_grad_residual(p, H, L, A, w, feat, target)
    # FP32 arithmetic against FP64, as for the large cases
    assert loss == pytest.approx(loss_o, rel=2e-5)
    assert np.linalg.norm(g - g_o) <= 2e-5 * np.linalg.norm(g_o)
    # predictions: the next step's guess behind the five of the history
    x0 = rng.normal(size=P.n)
    ctx.set_solution(x0)
    older = hist[:4]
    f2, s2 = orc.mpnn_features(A, A.rhs, x0, *older)
    inner = f2[:, 2] == 0
    xb = orc.mpnn_base_guess(x0, *older)
    x, so = net.predict()
    got = ((x - xb) / so)[inner]
    d_bf = orc.mpnn_forward_bf16(p, H, L, A, w, f2)[inner]
    assert np.linalg.norm(got - d_bf) < 3e-3 * np.linalg.norm(d_bf)
    net.precision = nw.MPNN_FP32
    x, so = net.predict()
    d = orc.mpnn_forward(p, H, L, A, w, f2)
    np.testing.assert_allclose((x[inner] - xb[inner]) / so, d[inner], rtol=0,
                               atol=2e-5 * np.abs(d).max() + 4e-16 * np.abs(xb).max() / so)


@pytest.mark.parametrize("precision,arrays", [("MPNN_BF16", 1.0), ("MPNN_FP32", 2.0)])
def test_prediction_holds_its_own_activations_only(nw, ctx, precision, arrays):
    """Device memory that a first prediction takes: two activation arrays of
    its precision (in units of one FP32 array [n][H]), the small per-node and
    per-slot arrays and the gradient partials; half an array more is within
    the allocator's granularity, a message array or the other precision's
    activations are not."""
    def free_memory():  # of the runtime that the library is linked to
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert nw.lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    P = pb.Problem(64, 64, 64, seed=2)
    P.upload(ctx)
    ctx.build_graph(1)
    ctx.assemble_continuity(nw.continuity_defaults())
    ctx.set_solution(np.random.default_rng(1).normal(size=P.n))
    ctx.solve(nw.solver_cfg(kspace=1, max_iters=0, x0=nw.X0_SOLUTION), raise_on_noconv=False)
    H, L = 64, 1
    net = nw.Mpnn(ctx, H, L, seed=3)
    net.params = 0.1 * np.random.default_rng(2).normal(size=net.nparams)
    net.precision = getattr(nw, precision)
    free = free_memory()
    net.predict()
    used = free - free_memory()
    row = 4 * P.n * H
    nnz = P.n + 2 * P.ne
    partials = 8 * 512 * (2 * H + 2 + L * H * (2 * H + 1) + 6 * H + 1)
    small = 4 * nnz + 4 * P.n * (5 + 5) + 8 * P.n * 3
    assert used < (arrays + 0.5) * row + partials + small
