"""GPU: hierarchies without room for what their first cycle forms (the matrix of
the small levels' sub-cycle, the tables of the block sweeps): the cycle is the
one of a hierarchy that has these turned off, bit for bit, nothing of them stays
allocated, and after a refresh with room the cycle is the one of a hierarchy
that never ran short.  The shortage is AFE_DEVICE_BYTES, which bounds a
context's own buffers; the vector `ballast` makes the room afterwards.

And a context's kept workspace, which makes room for other allocations."""
import numpy as np
import pytest

from tests.conftest import make_mesh

pytestmark = pytest.mark.gpu


class Run:
    """a context with a matrix, its hierarchy and vectors, always allocated in the same order"""

    def __init__(self, monkeypatch, limit, dense, sweeps):
        import afepack_amd as afe
        monkeypatch.setenv("AFE_DENSE_ROWS", str(dense))
        monkeypatch.setenv("AFE_SWEEP_ROWS", str(sweeps))
        if limit:
            monkeypatch.setenv("AFE_DEVICE_BYTES", str(limit))
        else:
            monkeypatch.delenv("AFE_DEVICE_BYTES", raising=False)
        self.afe, self.ctx = afe, afe.Context(0)
        self.ballast = afe.DeviceVector(self.ctx, 1 << 23)
        c, ev, vm = make_mesh(1, 40, 0.05, 3)
        self.sp = afe.Space(self.ctx, 1, c, ev, vm)
        self.A = afe.Matrix(self.sp)
        self.A.assemble(afe.OP_STIFF, 2)
        self.b = self.sp.rhs(2, afe.F_POISSON)
        self.A.apply_dirichlet(self.b)
        self.g = afe.Amg(self.A, afe.AmgParams(lazy=1, smooth=1, build_fp32=1))
        self.g.set_tail_rows(0)
        self.r = afe.DeviceVector.from_numpy(self.ctx, np.random.default_rng(1).uniform(-1, 1, self.sp.n_dof))
        self.z = afe.DeviceVector(self.ctx, self.sp.n_dof)

    def cycles(self):
        out = []
        for prec in (self.afe.PREC_FP64, self.afe.PREC_FP32):
            for _ in range(6):  # the captured cycle too
                self.g.vcycle(self.z, self.r, prec)
            out.append(self.z.numpy())
        self.z.zero()
        self.g.precondition(self.z, self.r, 6)
        return out + [self.z.numpy()]


@pytest.mark.parametrize("dense,sweeps", [(2560, 0), (0, 131072)])
@pytest.mark.parametrize("some", [False, True])
def test_first_cycle_without_room(monkeypatch, dense, sweeps, some):
    print(f"case memory dense={dense} sweeps={sweeps} some={some}", flush=True)
    off, free = Run(monkeypatch, 0, 0, 0), Run(monkeypatch, 0, dense, sweeps)
    held = free.ctx.device_bytes()
    n = free.g.info()["n"][1]
    assert n <= 2560
    room = 1000
    if some:  # the matrix, but not what forms it; the first of the tables, but not all
        room = 8 * n * n + 100000 if dense else 60000
    want_off, want = off.cycles(), free.cycles()
    assert not np.array_equal(want_off[0], want[0])
    run = Run(monkeypatch, held + room, dense, sweeps)
    assert run.ctx.device_bytes() == held
    for a, b in zip(run.cycles(), want_off):
        assert np.array_equal(a, b)
    # the matrix is not held (the context's workspace may have grown), no table is
    assert run.ctx.device_bytes() < held + 8 * n * n if dense else run.ctx.device_bytes() <= held
    run.ballast.free()
    run.g.lazy_reinit(run.A)
    free.g.lazy_reinit(free.A)
    for a, b in zip(run.cycles(), free.cycles()):
        assert np.array_equal(a, b)


def test_kept_workspace_makes_room(monkeypatch):
    """A load keeps its element loads' buffer; the matrix assembled next finds
    room only without it, and a later load has none then."""
    import afepack_amd as afe
    print("case memory workspace", flush=True)
    c, ev, vm = make_mesh(1, 60, 0.05, 3)

    def parts(ctx):
        held = [ctx.device_bytes()]
        sp = afe.Space(ctx, 1, c, ev, vm)
        b = afe.DeviceVector(ctx, sp.n_dof)
        held.append(ctx.device_bytes())
        sp.rhs(2, afe.F_POISSON, out=b)
        held.append(ctx.device_bytes())
        A = afe.Matrix(sp)
        A.assemble(afe.OP_STIFF, 2)
        held.append(ctx.device_bytes())
        first = b.numpy()
        sp.rhs(2, afe.F_POISSON, out=b)
        assert np.array_equal(b.numpy(), first)
        return held, A.values()

    monkeypatch.delenv("AFE_DEVICE_BYTES", raising=False)
    (_, h1, h2, h3), want = parts(afe.Context(0))
    work = h2 - h1
    assert work >= 8 * 3 * 7200
    monkeypatch.setenv("AFE_DEVICE_BYTES", str(h3 - 1))
    ctx = afe.Context(0)
    with pytest.raises(afe.AfeError):  # the load that follows has no room
        parts(ctx)
    ctx = afe.Context(0)
    sp = afe.Space(ctx, 1, c, ev, vm)
    b = sp.rhs(2, afe.F_POISSON)
    A = afe.Matrix(sp)
    A.assemble(afe.OP_STIFF, 2)
    assert np.array_equal(A.values(), want)
    assert ctx.device_bytes() == h3 - work
