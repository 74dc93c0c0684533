"""GPU: whole colour sweeps by independent blocks (one launch) against one
launch per colour (AFE_SWEEP_ROWS=0): levels of less than one block, of one
row more than a block, of many blocks; one, two and three sweeps a leg, the
symmetric and the stationary cycle, FP64 and FP32; hierarchies whose level 0 is
swept so, with and without the tail and the dense sub-cycle below; then after
new values.  The two forms sum a row's products in another grouping, so the
bounds are those of the matrix form (test_gpu_dense_cycle)."""
import numpy as np
import pytest

from tests.conftest import make_mesh
from tests.test_gpu_dense_cycle import compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n,lazy,smooth,dense,tail", [
    (1, 4, 1, 1, 0, 0), (1, 31, 0, 3, 0, 0), (1, 97, 1, 1, 200, 4096), (2, 16, 1, 2, 0, 0), (2, 60, 1, 1, 150, 0),
    (2, 60, 1, 3, 150, 4096), (3, 14, 1, 1, 60, 0), (1, 200, 1, 1, 2560, 4096)])
def test_block_sweeps_equal_the_colour_launches(ctx, monkeypatch, kind, n, lazy, smooth, dense, tail):
    import afepack_amd as afe
    print(f"case sweeps kind={kind} n={n} lazy={lazy} smooth={smooth} dense={dense} tail={tail}", flush=True)
    c, ev, vm = make_mesh(kind, n, 0.05, 21)
    sp = afe.Space(ctx, kind, c, ev, vm)
    A = afe.Matrix(sp)
    A.assemble(afe.OP_STIFF, 2)
    b = sp.rhs(2, afe.F_POISSON)
    A.apply_dirichlet(b)
    prm = afe.AmgParams(lazy=lazy, smooth=smooth, build_fp32=1)
    monkeypatch.setenv("AFE_DENSE_ROWS", str(dense))
    monkeypatch.setenv("AFE_SWEEP_ROWS", "0")
    g0 = afe.Amg(A, prm)
    monkeypatch.setenv("AFE_SWEEP_ROWS", "1000000")
    g1 = afe.Amg(A, prm)
    gs = [g0, g1]
    if lazy:
        gs.append(g1.clone(A))
    for g in gs:
        g.set_tail_rows(tail)
    rng = np.random.default_rng(n)
    for g in gs[1:]:
        compare(ctx, g0, g, sp.n_dof, rng)
    xs = []
    for g in gs:
        for prec in (afe.PREC_FP32, afe.PREC_FP64):
            x = afe.DeviceVector(ctx, sp.n_dof)
            assert g.pcg(x, b, rtol=1e-10, max_it=300, prec=prec).converged == 1
            xs.append(x.numpy())
    for x in xs[1:]:
        assert np.linalg.norm(x - xs[0]) <= 1e-9 * np.linalg.norm(xs[0])
    if lazy:
        assert np.array_equal(xs[2], xs[4]) and np.array_equal(xs[3], xs[5])  # the copy
        A.assemble(afe.OP_VARSTIFF, 2, afe.field_random(4, 3 if kind == 3 else 2, 0.5, 3))
        A.apply_dirichlet(b)
        for g in gs:
            g.lazy_reinit(A)
        compare(ctx, g0, g1, sp.n_dof, rng)
    for g in gs:
        g.set_smooth(2)
    compare(ctx, g0, g1, sp.n_dof, rng)
