"""GPU: the Fourier coefficient field and the manufactured functions against
extended precision, on meshes that reach outside the unit cube (negative and
large coordinates) and with wave numbers that are not integers.

With u = x_d on the nodes, u^T K u = sum_q Jxw a(x_q); the entries of the
manufactured load add up to sum_q Jxw f(x_q).  A mode's argument in half turns
is at most 2 k x D + 2 <= 77 here and takes D + 1 roundings of half an ulp
(7e-15), 3e-14 in all: 1e-13 in radians, so a = exp(g) is off by at most 1e-13
relative (amplitude 1), and its gradient by 2 pi k (at most 16) times that.
"""
import numpy as np
import pytest

from tests.conftest import make_mesh

pytestmark = pytest.mark.gpu

LD = np.longdouble
PI = LD("3.14159265358979323846264338327950288")


def _field_at(f, pts):
    k = f.k.reshape(f.n_modes, f.dim).astype(LD)
    arg = pts @ (2 * PI * k.T) + f.phi.astype(LD)
    g = LD(f.scale) * (np.sin(arg) @ f.w.astype(LD))
    dg = LD(f.scale) * ((np.cos(arg) * f.w.astype(LD)) @ (2 * PI * k))
    return g, dg


@pytest.mark.parametrize("kind,n", [(1, 9), (2, 5), (3, 4)])
def test_field_and_manufactured_load_outside_the_unit_cube(ctx, kind, n):
    import afepack_amd as afe
    print(f"case fields kind={kind} n={n}", flush=True)
    acc = 4
    c, ev, vm = make_mesh(kind, n, 0.05, 3)
    c = c * 8.0 - 3.0  # [-3, 5]
    dim = 3 if kind == 3 else 2
    rng = np.random.default_rng(kind)
    m = 7
    w = rng.uniform(-1, 1, m)
    f = afe.Field(rng.uniform(-2.5, 2.5, (m, dim)), rng.uniform(0, 2 * np.pi, m), w, 1.0 / np.abs(w).sum())
    sp = afe.Space(ctx, kind, c, ev, vm)
    pts, jxw = sp.qpoints(acc)
    pts, jxw = pts.reshape(-1, dim).astype(LD), jxw.reshape(-1).astype(LD)
    g, dg = _field_at(f, pts)
    a = np.exp(g)
    A = afe.Matrix(sp)
    A.assemble(afe.OP_VARSTIFF, acc, f)
    rp, col = sp.pattern()
    u = sp.dofs()[2].reshape(-1, dim)[:, 0].astype(LD)
    rows = np.repeat(np.arange(sp.n_dof), np.diff(rp))
    # the differences of u keep the row sums (zero in exact arithmetic) out
    got = -0.5 * np.sum(A.values().astype(LD) * (u[rows] - u[col]) ** 2)
    want = np.sum(jxw * a)
    assert abs(got - want) <= 1e-12 * abs(want)
    s, co = np.sin(PI * pts), PI * np.cos(PI * pts)
    du = np.stack([co[:, d] * np.prod(np.delete(s, d, 1), 1) for d in range(dim)], 1)
    fq = jxw * a * (dim * PI ** 2 * np.prod(s, 1) - np.sum(dg * du, 1))
    b = sp.rhs(acc, afe.F_VARCOEF, f).numpy().astype(LD)
    assert abs(b.sum() - fq.sum()) <= 4e-12 * np.abs(fq).sum()
    p = sp.rhs(acc, afe.F_POISSON).numpy().astype(LD)
    fp = jxw * dim * PI ** 2 * np.prod(s, 1)
    assert abs(p.sum() - fp.sum()) <= 1e-13 * np.abs(fp).sum()


@pytest.mark.parametrize("kind,n", [(1, 1), (2, 1), (3, 1), (1, 17), (2, 13), (3, 6)])
def test_loads_and_errors_match_plain_sums(ctx, kind, n):
    """Loads given at the DOFs and equal to one, and both error functionals,
    against sums over the quadrature points in extended precision: a load is
    a sum of at most nq * NL products of values of order one per element, so
    1e-14 of the largest entry; the errors' differences u - u_h are of order
    one (random DOF values), so 1e-13 relative."""
    import afepack_amd as afe
    print(f"case loads kind={kind} n={n}", flush=True)
    acc = 4
    c, ev, vm = make_mesh(kind, n, 0.05, 7)
    dim = 3 if kind == 3 else 2
    sp = afe.Space(ctx, kind, c, ev, vm)
    ed = sp.dofs()[0].reshape(sp.n_elem, -1)
    pts, jxw = (a.astype(LD) for a in sp.qpoints(acc))
    v = c.reshape(-1, dim).astype(LD)[ev.reshape(sp.n_elem, -1)]
    e = (v[:, 1:] - v[:, :1]).astype(np.float64)
    inv = np.linalg.inv(e).astype(LD)  # columns: gradients of barycentrics 1..D
    inv = inv @ (2 * np.eye(dim, dtype=LD) - e.astype(LD) @ inv)  # one Newton step to extended precision
    la = np.einsum("eqd,edk->eqk", pts - v[:, None, 0], inv)
    la = np.concatenate([1 - la.sum(-1, keepdims=True), la], -1)
    dl = np.concatenate([-inv.sum(-1, keepdims=True), inv], -1).transpose(0, 2, 1)
    if kind == 2:
        o, p = [1, 2, 0], [2, 0, 1]
        ph = np.concatenate([la * (2 * la - 1), 4 * la[..., o] * la[..., p]], -1)
        g = np.concatenate([(4 * la - 1)[..., None] * dl[:, None],
                            4 * (la[..., o, None] * dl[:, None, p] + la[..., p, None] * dl[:, None, o])], 2)
    else:
        ph, g = la, np.broadcast_to(dl[:, None], la.shape + (dim,))
    rng = np.random.default_rng(n)
    u = rng.uniform(-1, 1, sp.n_dof)
    for fkind, fq in ((afe.F_ONE, np.ones_like(jxw)), (afe.F_NODAL, np.einsum("eqj,ej->eq", ph, u[ed].astype(LD)))):
        want = np.zeros(sp.n_dof, dtype=LD)
        np.add.at(want, ed, np.einsum("eq,eqj->ej", jxw * fq, ph))
        got = sp.rhs(acc, fkind, nodal=u if fkind == afe.F_NODAL else None).numpy()
        assert np.abs(got - want).max() <= 1e-14 * np.abs(want).max()
    s, co = np.sin(PI * pts), PI * np.cos(PI * pts)
    du = np.stack([co[..., d] * np.prod(np.delete(s, d, -1), -1) for d in range(dim)], -1)
    uh = np.einsum("eqj,ej->eq", ph, u[ed].astype(LD))
    gh = np.einsum("eqjd,ej->eqd", g, u[ed].astype(LD))
    duh = afe.DeviceVector.from_numpy(ctx, u)
    l2 = np.sqrt(np.sum(jxw * (np.prod(s, -1) - uh) ** 2))
    h1 = np.sqrt(np.sum(jxw[..., None] * (du - gh) ** 2))
    assert abs(sp.error_l2(duh, acc) - l2) <= 1e-13 * l2
    assert abs(sp.error_h1(duh, acc) - h1) <= 1e-13 * h1
