"""Triangular solves on either side of the lines between 16 vectors per workgroup, a vector per thread (short or many ones)
and a tile per workgroup (batches of many tiles).  Residuals elementwise: |B - X op(A)| <= (n + 2) eps |X| |op(A)|, twice that
for the quotients' last bit."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,eps", [(np.float64, 2.2e-16), (np.float32, 1.2e-7)])
@pytest.mark.parametrize("order,count", [(1, 1), (8, 3), (8, 700), (9, 700), (12, 24575), (12, 24576), (32, 65535),
                                         (32, 65536), (33, 70000)])
def test_tile_solves(ctx, order, count, dtype, eps):
    """Right solves X op(A) = 2 B of `count` rows, all triangles and transposes, unit diagonals too (not read: NaN there)."""
    import hcorepp_amd as H
    rng = np.random.default_rng(order + count)
    b = rng.standard_normal((count, order)).astype(dtype)
    for uplo, trans, diag in (("L", "N", "N"), ("L", "T", "U"), ("U", "N", "U"), ("U", "T", "N")):
        full = rng.standard_normal((order, order)) / order + 3 * np.eye(order)
        tri = (np.tril(full) if uplo == "L" else np.triu(full)).astype(dtype)
        held, op = tri.copy(), tri.astype(float)
        if diag == "U":
            np.fill_diagonal(held, np.nan)
            np.fill_diagonal(op, 1.0)
        op = op.T if trans == "T" else op
        print(f"[case] {order} x {count} {uplo}{trans}{diag} {dtype.__name__}", flush=True)
        B = H.CompressedTile.from_cholesky_factors(np.zeros((count, order)), b, max_rank=order, dtype=dtype)
        H.HCore.trsm("R", uplo, trans, diag, 2.0, H.DenseTile(held, dtype=dtype), B, ctx)
        x = B.cholesky_factors()[1].astype(float)
        assert np.all(abs(x @ op - 2.0 * b) <= 2 * (order + 2) * eps * (abs(x) @ abs(op) + 2.0 * abs(b)))


@pytest.mark.parametrize("n,ranks,count", [(1, (1,), 2), (16, (2, 0, 5), 9), (32, (1, 40), 6), (33, (16,), 20), (33, (16,), 21),
                                           (40, (33,), 133), (40, (33,), 134), (64, (64, 3, 17), 160), (100, (300, 7), 60)])
def test_batched_solves(ctx, n, ranks, count):
    """V <- V L^{-T} of many tiles of several ranks."""
    import hcorepp_amd as H
    eps = np.finfo(np.float64).eps
    rng = np.random.default_rng(n + count)
    L = np.tril(rng.standard_normal((n, n)) / n + 3 * np.eye(n))
    vs = [rng.standard_normal((ranks[i % len(ranks)], n)) for i in range(count)]
    Bs = [H.CompressedTile(np.zeros((n, len(v))), v, max_rank=max(ranks) + 1) for v in vs]
    Ld = H.DenseTile(L + np.triu(np.full((n, n), np.nan), 1))  # the strict upper part is not read
    print(f"[case] {n} {ranks} x {count}", flush=True)
    H._check(H.lib().hcorepp_trsm_batch_d(ctx.h, count, C.byref(Ld.c()), (H._Tile * count)(*[b.c() for b in Bs])))
    ctx.sync()
    for v, b in zip(vs, Bs):
        x = b.factors()[1]
        assert np.all(abs(x @ L.T - v) <= 2 * (n + 2) * eps * (abs(x) @ abs(L).T + abs(v)))
