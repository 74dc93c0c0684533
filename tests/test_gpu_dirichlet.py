"""GPU: zero Dirichlet elimination through the space's entry lists, against a
dense restatement, bit for bit: no marked DOF, one, scattered interior marks
of several values, the whole boundary, and every DOF; on a space and on its
copy (afe_space_clone)."""
import numpy as np
import pytest

from tests.conftest import make_mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n", [(1, 1), (1, 19), (2, 9), (3, 5)])
@pytest.mark.parametrize("marks", ["none", "one", "scattered", "boundary", "all"])
def test_zero_elimination_is_the_dense_one(ctx, kind, n, marks):
    import afepack_amd as afe
    print(f"case dirichlet kind={kind} n={n} {marks}", flush=True)
    c, ev, vm = make_mesh(kind, n, 0.05, 5)
    rng = np.random.default_rng(n)
    if marks != "boundary":
        vm = np.zeros_like(vm)
    if marks == "one":
        vm[len(vm) // 2] = 3
    elif marks == "scattered":
        vm[:] = np.where(rng.uniform(size=len(vm)) < 0.3, rng.integers(-2, 4, len(vm)), 0)
    elif marks == "all":
        vm[:] = 1
    sides = None
    if kind == 2:  # side marks, so that edge DOFs follow the chosen marks
        t = ev.reshape(-1, 3)
        sv = np.unique(np.sort(np.concatenate([t[:, [0, 1]], t[:, [1, 2]], t[:, [2, 0]]]), axis=1), axis=0)
        sides = (sv, np.where(vm[sv[:, 0]] == vm[sv[:, 1]], vm[sv[:, 0]], 0))
    sp = afe.Space(ctx, kind, c, ev, vm, sides)
    rp, col = sp.pattern()
    mark = sp.dofs()[1] != 0
    rows = np.repeat(np.arange(sp.n_dof), np.diff(rp))
    out = (mark[rows] | mark[col]) & (rows != col)
    for space in (sp, sp.clone()):
        A = afe.Matrix(space)
        A.assemble(afe.OP_STIFF, 2)
        v = A.values()
        f = rng.uniform(-1, 1, sp.n_dof)
        d = afe.DeviceVector.from_numpy(ctx, f)
        A.apply_dirichlet(d)
        want = f.copy()
        want[mark] = v[rp[:-1]][mark] * 0.0
        assert np.array_equal(A.values(), np.where(out, 0.0, v))
        assert np.array_equal(d.numpy(), want)
