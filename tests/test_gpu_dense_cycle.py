"""GPU: the small levels' sub-cycle applied as a matrix against the same levels
run step by step (AFE_DENSE_ROWS=0): the symmetric and the stationary cycle,
one and three sweeps, coarsest level solved by the inverse or smoothed, a
hierarchy whose every level below the first is in the matrix, one with tail
levels above it and one with the tail off; then after new values, after another
smoothing count and after the coarse solve changes.  Which cycles form the
matrix: solves, and the fourth single one on the same values and smoothing count.

The matrix is the FP64 cycle's: FP64 results differ by rounding in sums of at
most a few thousand terms (1e-12 relative bounds them, as in the other cycle
tests); the FP32 cycle's levels round every step to 6e-8 relative, and its few
hundred dependent steps differ by less than 1e-5.
"""
import numpy as np
import pytest

from tests.conftest import make_mesh

pytestmark = pytest.mark.gpu


def _pair(ctx, monkeypatch, A, prm, rows):
    import afepack_amd as afe
    monkeypatch.setenv("AFE_DENSE_ROWS", "0")
    a = afe.Amg(A, prm)
    monkeypatch.setenv("AFE_DENSE_ROWS", str(rows))
    return a, afe.Amg(A, prm)


def compare(ctx, g0, g1, n, rng, f32=True):
    import afepack_amd as afe
    r = afe.DeviceVector.from_numpy(ctx, rng.uniform(-1, 1, n))
    z = [afe.DeviceVector(ctx, n) for _ in range(2)]
    for prec, tol in ((afe.PREC_FP64, 1e-12), (afe.PREC_FP32, 1e-5)):
        for _ in range(4):  # the matrix is formed by the fourth cycle at the latest
            for g, v in zip((g0, g1), z):
                g.vcycle(v, r, prec)
            a, b = (v.numpy() for v in z)
            assert np.linalg.norm(a - b) <= tol * np.linalg.norm(a), prec
    for g, v in zip((g0, g1), z):
        v.zero()
        g.precondition(v, r, 3)  # four stationary cycles
    a, b = (v.numpy() for v in z)
    assert np.linalg.norm(a - b) <= 1e-12 * np.linalg.norm(a)


@pytest.mark.parametrize("kind,n,lazy,smooth,rows,tail", [
    (1, 24, 0, 3, 2560, 4096), (1, 24, 0, 1, 100, 4096), (2, 20, 1, 1, 64, 0), (2, 20, 1, 2, 400, 4096),
    (3, 9, 1, 1, 300, 4096), (3, 9, 1, 1, 2560, 0), (1, 60, 1, 1, 1100, 4096)])
def test_matrix_form_equals_the_steps(ctx, monkeypatch, kind, n, lazy, smooth, rows, tail):
    import afepack_amd as afe
    print(f"case dense kind={kind} n={n} lazy={lazy} smooth={smooth} rows={rows} tail={tail}", flush=True)
    c, ev, vm = make_mesh(kind, n, 0.05, 13)
    sp = afe.Space(ctx, kind, c, ev, vm)
    A = afe.Matrix(sp)
    A.assemble(afe.OP_STIFF, 2)
    b = sp.rhs(2, afe.F_POISSON)
    A.apply_dirichlet(b)
    g0, g1 = _pair(ctx, monkeypatch, A, afe.AmgParams(lazy=lazy, smooth=smooth, build_fp32=1), rows)
    assert g1.info()["n"][-1] <= rows
    for g in (g0, g1):
        g.set_tail_rows(tail)
    rng = np.random.default_rng(n)
    # the coarsest level alone: its matrix is the coarse solve's inverse
    lone = g1.dense_info()[0] == g1.info()["levels"] - 1

    def compare_formed():
        compare(ctx, g0, g1, sp.n_dof, rng)
        assert g0.dense_info() == (-1, (False, False))
        assert g1.dense_info()[0] > 0
        assert lone or g1.dense_info()[1] == (True, True)

    compare_formed()
    xs = []
    for g in (g0, g1):
        x = afe.DeviceVector(ctx, sp.n_dof)
        assert g.pcg(x, b, rtol=1e-10, max_it=300, prec=afe.PREC_FP32).converged == 1
        xs.append(x.numpy())
    assert np.linalg.norm(xs[0] - xs[1]) <= 1e-9 * np.linalg.norm(xs[0])
    if lazy:  # new values on the pattern
        A.assemble(afe.OP_VARSTIFF, 2, afe.field_random(4, 3 if kind == 3 else 2, 0.5, 3))
        A.apply_dirichlet(b)
        for g in (g0, g1):
            g.lazy_reinit(A)
        compare_formed()
    for g in (g0, g1):
        g.set_smooth(2)
    compare_formed()
    for g in (g0, g1):
        g.set_coarse_exact(False)
    compare_formed()


def test_which_cycles_form_the_matrix(ctx):
    import afepack_amd as afe
    print("case dense forming", flush=True)
    c, ev, vm = make_mesh(1, 40, 0.05, 13)
    sp = afe.Space(ctx, 1, c, ev, vm)
    A = afe.Matrix(sp)
    A.assemble(afe.OP_STIFF, 2)
    b = sp.rhs(2, afe.F_POISSON)
    A.apply_dirichlet(b)
    g = afe.Amg(A, afe.AmgParams(lazy=1, smooth=1, build_fp32=1))
    x = afe.DeviceVector(ctx, sp.n_dof)

    def formed():
        return g.dense_info()[1]

    for _ in range(3):  # new values, then three cycles each time
        for _ in range(3):
            g.vcycle(x, b, afe.PREC_FP32)
        x.zero()
        g.precondition(x, b, 2)
        assert formed() == (False, False)
        g.lazy_reinit(A)
    for k in range(4):  # either precision counts
        assert formed() == (False, False)
        g.vcycle(x, b, afe.PREC_FP64 if k % 2 else afe.PREC_FP32)
    assert formed() == (False, True)
    x.zero()
    g.precondition(x, b, 3)
    assert formed() == (True, True)
    g.set_smooth(2)  # another count: three cycles of it, then back to the matrix
    for _ in range(3):
        g.vcycle(x, b, afe.PREC_FP64)
    assert formed() == (False, False)
    g.set_smooth(1)
    assert formed() == (True, True)
    g.lazy_reinit(A)
    assert formed() == (False, False)
    x.zero()
    g.pcg(x, b, rtol=1e-8, max_it=100, prec=afe.PREC_FP32)
    assert formed() == (False, True)
    g.lazy_reinit(A)
    x.zero()
    g.pcg(x, b, rtol=1e-8, max_it=2**31 - 1, prec=afe.PREC_FP32)  # the largest bound
    assert formed() == (False, True)
    # the step form and the matrix agree along one call's cycles (captured both ways)
    ref = afe.DeviceVector(ctx, sp.n_dof)
    g.vcycle(ref, b, afe.PREC_FP64)
    for _ in range(2):
        g.lazy_reinit(A)
        for k in range(6):
            g.vcycle(x, b, afe.PREC_FP64)
            assert np.linalg.norm(x.numpy() - ref.numpy()) <= 1e-12 * np.linalg.norm(ref.numpy())


def test_what_a_solve_keeps(ctx):
    """A solve's first cycle keeps the matrix and workspace for 512 columns of
    three vectors on the levels down from it, not for all columns, beside the
    sweep tables of a level of 4225 rows (below 4 MB)."""
    import afepack_amd as afe
    print("case dense workspace", flush=True)
    c, ev, vm = make_mesh(1, 64, 0.05, 13)
    own = afe.Context(0)
    sp = afe.Space(own, 1, c, ev, vm)
    A = afe.Matrix(sp)
    A.assemble(afe.OP_STIFF, 4)
    b = sp.rhs(4, afe.F_POISSON)
    A.apply_dirichlet(b)
    g = afe.Amg(A, afe.AmgParams(lazy=0, smooth=3, build_fp32=0))
    x = afe.DeviceVector(own, sp.n_dof)
    held = own.device_bytes()
    g.solve(x, b)
    n = g.info()["n"]
    assert 512 < n[1] <= 2560
    assert own.device_bytes() - held <= 8 * n[1] ** 2 + 512 * 3 * 8 * sum(n[1:]) + (4 << 20)
