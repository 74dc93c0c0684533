"""GPU: A x and A^T x of CSR matrices against the sequential sums, bit for bit
(products rounded, then added in stored order; the transposed product in
ascending row order): rows around the staged form's block of 256 rows and chunk
of 2048 products, rows far longer than the others, and blocks of rows long
enough for the one-thread form: beyond 8 chunks of entries, and beyond 8 times
the longest row, with rows shorter and longer than a chunk."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _matrix(m, lens, rng):
    lens = np.clip(np.broadcast_to(lens, m), 1, m)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    col = np.concatenate([np.concatenate([[i], np.sort(rng.permutation(np.delete(np.arange(m), i))[:n - 1])])
                          for i, n in enumerate(lens)])
    return rp, col.astype(np.int64), rng.standard_normal(rp[-1])


@pytest.mark.parametrize("m,lens", [(1, 1), (255, 3), (256, 8), (257, 8), (600, 64), (520, 65), (300, 300),
                                    (700, "one long"), (1000, "mixed"), (3000, "1 of 3000"), (3000, "5 of 3000"),
                                    (3000, "7 of 3000"), (3000, "8 of 3000"), (3000, "60 of 3000"),
                                    (3000, "30 of 500"), (3000, "40 of 500")])
def test_products_are_the_sequential_sums(ctx, monkeypatch, m, lens):
    import afepack_amd as afe
    print(f"case products m={m} lens={lens}", flush=True)
    rng = np.random.default_rng(m)
    if lens == "one long":
        lens = np.full(m, 5)
        lens[m // 2] = m
    elif lens != "mixed" and isinstance(lens, str):  # that many long rows together, across a block's end
        k, n = (int(v) for v in lens.split(" of "))
        lens = np.full(m, 5)
        lens[500:500 + k] = n
        lens[1100:1100 + k] = n
    elif isinstance(lens, str):
        lens = rng.integers(1, 60, m)
    rp, col, val = _matrix(m, lens, rng)
    A = afe.Matrix(ctx=ctx, csr=(rp, col, val))
    x = rng.standard_normal(m)
    y = np.zeros(m)
    for i in range(m):
        s = 0.0
        for p in val[rp[i]:rp[i + 1]] * x[col[rp[i]:rp[i + 1]]]:
            s += p
        y[i] = s
    yt = np.zeros(m)
    rows = np.repeat(np.arange(m), np.diff(rp))
    for j, p in zip(col, val * x[rows]):
        yt[j] += p
    dx, dy = afe.DeviceVector.from_numpy(ctx, x), afe.DeviceVector(ctx, m)
    A.vmult(dx, dy)
    assert np.array_equal(dy.numpy(), y)
    for _ in range(2):  # the map is built by the first call
        A.tvmult(dx, dy)
        assert np.array_equal(dy.numpy(), yt)
    # 64-bit positions, which matrices of 2^31 entries and more take
    monkeypatch.setenv("AFE_POS64", "1")
    B = afe.Matrix(ctx=ctx, csr=(rp, col, val))
    B.tvmult(dx, dy)
    assert np.array_equal(dy.numpy(), yt)
