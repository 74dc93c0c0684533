"""GPU: whole colour sweeps by independent blocks (one launch) against one
launch per colour (AFE_SWEEP_ROWS=0): levels of one block, of one block that
took a fragment in, of two, of many blocks; one, two and three sweeps a leg, the
symmetric and the stationary cycle, FP64 and FP32; hierarchies whose level 0 is
swept so, with and without the tail and the dense sub-cycle below; then after
new values.  The two forms sum a row's products in another grouping, so the
bounds are those of the matrix form (test_gpu_dense_cycle).

The levels that have to run so are named with each case, with their number of
blocks where rows and block size fix it (blocks of 32 rows up to 8192 rows, a
rest of less than 8 rows joining another block), and every other level has to
have none: levels within the dense bound, the coarsest, and those whose rows have
more than 24 entries (Galerkin levels of tetrahedra, or of the full coarsening)."""
import numpy as np
import pytest

from tests.conftest import make_mesh
from tests.test_gpu_dense_cycle import compare
from tests.test_gpu_galerkin import _random_csr

pytestmark = pytest.mark.gpu


MANY = -1  # more than one block


@pytest.mark.parametrize("kind,n,lazy,smooth,dense,tail,blocks", [
    (1, 4, 1, 1, 0, 0, {0: 1}), (1, 5, 0, 1, 0, 0, {0: 1, 1: 1}), (1, 6, 1, 2, 0, 0, {0: 2, 1: 1}),
    (1, 31, 0, 3, 100, 0, {0: MANY}), (1, 97, 1, 1, 200, 4096, {0: MANY, 1: MANY, 2: MANY}),
    (2, 16, 1, 2, 200, 0, {0: MANY}), (2, 60, 1, 1, 1000, 0, {0: MANY, 1: MANY}),
    (2, 60, 1, 3, 1000, 4096, {0: MANY, 1: MANY}), (3, 14, 1, 1, 60, 0, {0: MANY}),
    (1, 200, 1, 1, 2560, 4096, {0: MANY, 1: MANY, 2: MANY})])
def test_block_sweeps_equal_the_colour_launches(ctx, monkeypatch, kind, n, lazy, smooth, dense, tail, blocks):
    import afepack_amd as afe
    print(f"case sweeps kind={kind} n={n} lazy={lazy} smooth={smooth} dense={dense} tail={tail}", flush=True)
    c, ev, vm = make_mesh(kind, n, 0.05, 21)
    sp = afe.Space(ctx, kind, c, ev, vm)
    A = afe.Matrix(sp)
    A.assemble(afe.OP_STIFF, 2)
    b = sp.rhs(2, afe.F_POISSON)
    A.apply_dirichlet(b)
    prm = afe.AmgParams(lazy=lazy, smooth=smooth, build_fp32=1, nmpo=8)
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
    for g in gs:
        for l, v in enumerate(g.sweep_info()):
            nn, nnz = g.info()["n"][l], g.info()["nnz"][l]
            may = l + 1 < g.info()["levels"] and nn > dense and nnz - nn <= 24 * nn
            if g is not g0 and may and l not in blocks and not lazy:
                continue  # the full coarsening's levels depend on the values
            want = blocks.get(l, 0) if g is not g0 else 0
            assert v["blocks"] == want if want != MANY else v["blocks"] > 1, (l, v)
            assert v["fused"] == (want != 0, want != 0), (l, v)
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


def test_hierarchies_without_own_cycles_form_no_tables(ctx, monkeypatch):
    """A hierarchy that only joins a batch, or is refreshed and copied, holds
    what one with the block sweeps turned off holds, and forms its tables with
    its first own cycle."""
    import afepack_amd as afe
    print("case sweeps first cycle", flush=True)
    c, ev, vm = make_mesh(2, 40, 0.05, 2)
    sp = afe.Space(ctx, 2, c, ev, vm)
    A = afe.Matrix(sp)
    A.assemble(afe.OP_STIFF, 2)
    b = sp.rhs(2, afe.F_POISSON)
    A.apply_dirichlet(b)
    monkeypatch.setenv("AFE_DENSE_ROWS", "0")
    prm = afe.AmgParams(lazy=1, smooth=1, build_fp32=1)
    held = []
    for rows in ("0", "131072"):
        monkeypatch.setenv("AFE_SWEEP_ROWS", rows)
        base = ctx.device_bytes()
        g = afe.Amg(A, prm)
        g.lazy_reinit(A)
        h = g.clone(A)
        held.append(ctx.device_bytes() - base)
        assert all(v["blocks"] == 0 for v in g.sweep_info() + h.sweep_info())
        bt = afe.Batch(ctx, smooth=1)
        x = afe.DeviceVector(ctx, sp.n_dof)
        bt.add(g, x, b, rtol=1e-8)
        bt.run()
        bt.close()
        assert all(v["blocks"] == 0 for v in g.sweep_info())
        g.vcycle(x, b, afe.PREC_FP32)
        assert (g.sweep_info()[0]["blocks"] > 1) == (rows != "0")
        assert g.sweep_info()[0]["fused"] == (False, rows != "0")
        g.close()
        h.close()
    assert held[0] == held[1]


def test_levels_with_large_closures_keep_the_colour_launches(ctx, monkeypatch):
    """Random couplings: the closure of a block of 32 rows is far beyond six
    times its size, so the level has no blocks and its cycle is the one of the
    colour launches, bit for bit."""
    import afepack_amd as afe
    print("case sweeps random couplings", flush=True)
    rng = np.random.default_rng(4)
    m = 3000
    rp, col = _random_csr(m, 3, rng)
    rows = np.repeat(np.arange(m), np.diff(rp))
    A = afe.Matrix(ctx=ctx, csr=(rp, col, np.where(rows == col, 1.0 + np.diff(rp)[rows], -1.0)))
    prm = afe.AmgParams(lazy=1, smooth=1, build_fp32=1)
    monkeypatch.setenv("AFE_DENSE_ROWS", "0")
    r = afe.DeviceVector.from_numpy(ctx, rng.uniform(-1, 1, m))
    out = []
    for bound in ("0", "1000000"):
        monkeypatch.setenv("AFE_SWEEP_ROWS", bound)
        g = afe.Amg(A, prm)
        z = afe.DeviceVector(ctx, m)
        g.vcycle(z, r, afe.PREC_FP64)
        assert g.sweep_info()[0]["blocks"] == 0
        out.append(z.numpy())
    assert np.array_equal(out[0], out[1])


def test_blocks_that_fit_in_lds_in_fp32_only(ctx, monkeypatch):
    """85184 rows of tetrahedra: a block's arrays take 98 KB in FP32 and 168 KB,
    more than a workgroup has, in FP64.  FP64 cycles keep the colour launches,
    bit for bit; FP32 ones take the blocks."""
    import afepack_amd as afe
    print("case sweeps fp32 only", flush=True)
    c, ev, vm = make_mesh(3, 43, 0.05, 21)
    sp = afe.Space(ctx, 3, c, ev, vm)
    A = afe.Matrix(sp)
    A.assemble(afe.OP_STIFF, 2)
    b = sp.rhs(2, afe.F_POISSON)
    A.apply_dirichlet(b)
    prm = afe.AmgParams(lazy=1, smooth=1, build_fp32=1)
    rng = np.random.default_rng(2)
    r = afe.DeviceVector.from_numpy(ctx, rng.uniform(-1, 1, sp.n_dof))
    out = []
    for rows in ("0", "131072"):
        monkeypatch.setenv("AFE_SWEEP_ROWS", rows)
        g = afe.Amg(A, prm)
        z = afe.DeviceVector(ctx, sp.n_dof)
        for prec in (afe.PREC_FP32, afe.PREC_FP64):
            g.vcycle(z, r, prec)
            out.append(z.numpy())
        v = g.sweep_info()[0]
        assert (v["blocks"] > 1, v["fused"]) == (rows != "0", (False, rows != "0"))
    assert np.array_equal(out[1], out[3])
    assert not np.array_equal(out[0], out[2])
    assert np.linalg.norm(out[0] - out[2]) <= 1e-5 * np.linalg.norm(out[0])
