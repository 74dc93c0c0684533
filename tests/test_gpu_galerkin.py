"""GPU: the device Galerkin products of a lazy refresh against a fresh host
build, bit for bit, where the lane groups can go wrong: coarse rows far longer
than a group owns in one pass, P^T rows longer than the four terms taken at a
time and than the term window, levels of one row, and enough coarse rows for
the 16-lane form (more than 24576)."""
import numpy as np
import pytest

from tests.conftest import make_mesh

pytestmark = pytest.mark.gpu


def _same(g, fresh):
    assert g.info()["levels"] == fresh.info()["levels"]
    for l in range(g.info()["levels"]):
        for a, b in zip(g.level_csr(l, 0), fresh.level_csr(l, 0)):
            assert np.array_equal(a, b), l


def _random_csr(m, extra, rng, hub=0):
    """symmetric pattern, diagonal first: a ring, `extra` random couplings per row and `hub` rows coupled to all"""
    i = np.concatenate([np.arange(m), rng.integers(0, m, extra * m), np.repeat(np.arange(hub), m)])
    j = np.concatenate([(np.arange(m) + 1) % m, rng.integers(0, m, extra * m), np.tile(np.arange(m), hub)])
    keep = i != j
    i, j = i[keep], j[keep]
    k = np.unique(np.concatenate([i * m + j, j * m + i]))
    r, c = np.concatenate([k // m, np.arange(m)]), np.concatenate([k % m, np.arange(m)])
    o = np.lexsort((np.where(r == c, -1, c), r))
    r, c = r[o], c[o]
    rp = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=m))]).astype(np.int64)
    return rp, c.astype(np.int64)


@pytest.mark.parametrize("m,extra,hub", [(3, 0, 0), (40, 1, 0), (700, 3, 0), (3000, 6, 0), (2500, 1, 3), (120, 30, 2)])
def test_refresh_of_random_patterns(ctx, m, extra, hub):
    import afepack_amd as afe
    print(f"case galerkin m={m} extra={extra} hub={hub}", flush=True)
    rng = np.random.default_rng(m)
    rp, col = _random_csr(m, extra, rng, hub)
    rows = np.repeat(np.arange(m), np.diff(rp))

    def values():
        v = rng.standard_normal(len(col))
        return np.where(rows == col, 4.0 * np.diff(rp)[rows], v)

    A = afe.Matrix(ctx=ctx, csr=(rp, col, values()))
    prm = afe.AmgParams(lazy=1, smooth=1, nmpo=8, nmpsd=0.0)
    g = afe.Amg(A, prm)
    A.set_values(values())
    g.lazy_reinit(A)
    _same(g, afe.Amg(A, prm))


@pytest.mark.parametrize("kind,n", [(1, 330), (3, 20)])
def test_refresh_of_mesh_hierarchies(ctx, kind, n):
    import afepack_amd as afe
    print(f"case galerkin kind={kind} n={n}", flush=True)
    c, ev, vm = make_mesh(kind, n, 0.05, 9)
    sp = afe.Space(ctx, kind, c, ev, vm)
    A = afe.Matrix(sp)
    A.assemble(afe.OP_STIFF, 2)
    prm = afe.AmgParams(lazy=1, smooth=1)
    g = afe.Amg(A, prm)
    if kind == 1:
        assert g.info()["n"][1] > 24576
    f = afe.field_random(4, 3 if kind == 3 else 2, 0.5, 2)
    A.assemble(afe.OP_VARSTIFF, 2, f)
    g.lazy_reinit(A)
    _same(g, afe.Amg(A, prm))
