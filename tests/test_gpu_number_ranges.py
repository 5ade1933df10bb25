"""Branches taken for numbers out of the usual range: reflectors whose norms' squares leave it, Gram matrices that need
their scale, quotients whose reciprocal is no finite number, pivots beyond the range of a reciprocal square root or not
positive, factors that are no numbers in the mixed form."""
import ctypes as C

import numpy as np
import pytest

from helpers import rel_fro

pytestmark = pytest.mark.gpu


def _update(m, K, scale, dtype=np.float64):
    """Factors whose left sides carry `scale` and whose stacked rank is K, with a flat spectrum: nothing is truncated, and
    no column's square is smaller than the scale's by more than m."""
    rng = np.random.default_rng(K)
    ra = K // 2
    f = []
    for r, s in ((ra, scale), (ra + 1, 1.0), (K - ra, scale)):
        u, v = (np.linalg.qr(rng.standard_normal((m, r)))[0] for _ in range(2))
        f.append((u * s, np.linspace(1.0, 0.3, r)[:, None] * v.T))
    f[1] = (np.linalg.qr(np.hstack([f[0][1].T / np.linspace(1.0, 0.3, ra), rng.standard_normal((m, 1))]))[0], f[1][1])
    a, b, c = [tuple(x.astype(dtype).astype(float) for x in p) for p in f]
    return a, b, c, c[0] @ c[1] + (a[0] @ a[1]) @ (b[0] @ b[1])


@pytest.mark.parametrize("dtype,scale", [(np.float64, 1e-148), (np.float64, 1e-141), (np.float64, 1e141), (np.float64, 1e148),
                                         (np.float32, 1e-16), (np.float32, 1e16)])
@pytest.mark.parametrize("m,K", [(40, 19), (150, 130), (1100, 33)])
def test_plain_scales(ctx, m, K, dtype, scale):
    """The plain form's bound, a few K eps with a margin of about 30, holds at every scale."""
    import hcorepp_amd as H
    eps = np.finfo(dtype).eps
    a, b, c, full = _update(m, K, scale, dtype)
    print(f"[case] {m} {K} {scale} {dtype.__name__}", flush=True)
    tile = lambda f, **kw: H.CompressedTile(*(x.astype(dtype) for x in f), dtype=dtype, **kw)  # noqa: E731
    Ct = tile(c, max_rank=K)
    H.HCore.gemm(1.0, tile(a), tile(b), 1.0, Ct, ctx, H.CompressionParameters(scale * 1e-3 * eps))
    assert Ct.rank == K
    assert rel_fro(Ct.to_dense().astype(float) / scale, full / scale) < 100 * (K + 1) * eps
    u = Ct.factors()[0].astype(float)
    assert np.abs(u.T @ u - np.eye(K)).max() < 100 * (K + 1) * eps


@pytest.mark.parametrize("scale", [1e-148, 1e148])
@pytest.mark.parametrize("m,K", [(40, 19), (150, 130)])
def test_batched_scales(ctx, m, K, scale):
    """1e-9, the batched form's accuracy (its Jacobi stops at cosines of about 1e-10)."""
    import hcorepp_amd as H
    a, b, c, full = _update(m, K, scale)
    print(f"[case] {m} {K} {scale}", flush=True)
    Ct = H.CompressedTile(*c, max_rank=K)
    bt = H.Batch(ctx, [H.CompressedTile(*a)], [H.CompressedTile(*b)], [Ct], 1.0, 1.0, H.CompressionParameters(scale * 1e-13))
    bt.run()
    assert bt.status()[0] == 0 and bt.sync_ranks_to_tiles()[0] == K
    bt.close()
    assert rel_fro(Ct.to_dense() / scale, full / scale) < 1e-9


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_mixed_keeps_c_of_no_numbers(ctx, value):
    """A value that is no number in a factor of either side: that update reports NUMERIC and keeps C, the others complete."""
    import hcorepp_amd as H
    a, b, c, full = _update(70, 21, 1.0)
    for side in range(4):
        print(f"[case] {value} in factor {side}", flush=True)
        bad = [x.copy() for x in (*a, *b)]
        bad[side][min(3, bad[side].shape[0] - 1), 5] = value
        Cs = [H.CompressedTile(*c, max_rank=30) for _ in range(2)]
        bt = H.Batch(ctx, [H.CompressedTile(*bad[:2]), H.CompressedTile(*a)], [H.CompressedTile(*bad[2:]), H.CompressedTile(*b)],
                     Cs, 1.0, 1.0, H.CompressionParameters(1e-11), H.PREC_MIXED)
        bt.run()
        assert H.STATUS[bt.status()[0]] == "NUMERIC"
        bt.sync_ranks_to_tiles()
        bt.close()
        assert all(np.array_equal(x, y) for x, y in zip(Cs[0].factors(), c))
        assert rel_fro(Cs[1].to_dense(), full) < 1e-9


def _solve(ctx, form, L, b, dtype):
    """X with X L^T = B by one of the tile solves or of the batched ones."""
    import hcorepp_amd as H
    if form == "tile":
        B = H.CompressedTile.from_cholesky_factors(np.zeros(b.shape), b, max_rank=len(L), dtype=dtype)
        H.HCore.trsm("R", "L", "T", "N", 1.0, H.DenseTile(L, dtype=dtype), B, ctx)
        return B.cholesky_factors()[1]
    count = 200 if form == "batch of many" else 1
    Bs = [H.CompressedTile(np.zeros((len(L), len(b))), b, max_rank=len(b)) for _ in range(count)]
    d = H.DenseTile(L).c()
    H._check(H.lib().hcorepp_trsm_batch_d(ctx.h, count, C.byref(d), (H._Tile * count)(*[t.c() for t in Bs])))
    ctx.sync()
    xs = [t.factors()[1] for t in (Bs[0], Bs[-1])]
    assert np.array_equal(*xs, equal_nan=True)
    return xs[0]


@pytest.mark.parametrize("form,dtype", [("tile", np.float64), ("tile", np.float32), ("batch", np.float64),
                                        ("batch of many", np.float64)])
@pytest.mark.parametrize("n,j", [(8, 3), (40, 5), (40, 37), (70, 33)])
def test_solves_with_any_diagonal(ctx, n, j, form, dtype):
    """One diagonal element zero, infinite, subnormal or near the largest number.  Row j has no other one, so x_j is b_j / l_jj
    to a rounding; zero gives an infinity, from which the later ones are no numbers any more."""
    info = np.finfo(dtype)
    rng = np.random.default_rng(n + j)
    b = rng.uniform(0.5, 1.0, (20, n)).astype(dtype)
    L = np.tril(rng.uniform(0.1, 1.0, (n, n)) / n + 3 * np.eye(n)).astype(dtype)
    L[j, :j] = 0
    tiny, huge = dtype(3 * info.smallest_subnormal * 2 ** 8), dtype(0.9) * info.max
    for d in (dtype(0), dtype(np.inf), -dtype(np.inf), tiny, huge, -huge):
        Ld, bd = L.copy(), b.copy()
        Ld[j, j] = d
        if d == tiny:
            bd[:, j] = rng.integers(1, 99, 20) * info.smallest_subnormal * 16
        elif abs(d) == huge:
            bd[:, j] *= huge / 4
        print(f"[case] {form} {dtype.__name__} {n} {j} {d}", flush=True)
        x = _solve(ctx, form, Ld, bd, dtype)
        with np.errstate(divide="ignore"):
            xj = bd[:, j] / d
        if d == 0:
            assert np.all(x[:, j] == np.inf)
            assert not np.any(np.isfinite(x[:, j + 1:]))
            x, Ld, bd = x[:, :j], Ld[:j, :j], bd[:, :j]
        else:
            assert np.all(abs(x[:, j] - xj) <= 2 * info.eps * abs(xj))
            Ld[j, j], bd[:, j] = 1, xj
        x, Ld, bd = x.astype(float), Ld.astype(float), bd.astype(float)
        assert np.all(abs(x @ Ld.T - bd) <= 2 * (n + 2) * info.eps * (abs(x) @ abs(Ld).T + abs(bd)))


@pytest.mark.parametrize("dtype,order", [(np.float64, 395), (np.float64, 396), (np.float32, 982), (np.float32, 983)])
def test_longest_vectors_in_lds(ctx, order, dtype):
    """Solves at the longest vectors that stay in LDS and at one more element, forward and backward."""
    import hcorepp_amd as H
    eps = np.finfo(dtype).eps
    rng = np.random.default_rng(order)
    b = rng.standard_normal((18, order)).astype(dtype)
    full = rng.standard_normal((order, order)) / order + 3 * np.eye(order)
    for uplo, trans in (("L", "T"), ("L", "N"), ("U", "N"), ("U", "T")):
        tri = (np.tril(full) if uplo == "L" else np.triu(full)).astype(dtype)
        B = H.CompressedTile.from_cholesky_factors(np.zeros((18, order)), b, max_rank=order, dtype=dtype)
        H.HCore.trsm("R", uplo, trans, "N", 1.0, H.DenseTile(tri, dtype=dtype), B, ctx)
        x, op = B.cholesky_factors()[1].astype(float), tri.astype(float)
        op = op.T if trans == "T" else op
        assert np.all(abs(x @ op - b) <= 2 * (order + 2) * eps * (abs(x) @ abs(op) + abs(b)))


def _spd(n, dtype):
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n))
    return (a @ a.T / n + np.eye(n)).astype(dtype)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,j", [(5, 4), (70, 0), (70, 31), (70, 32), (70, 40), (70, 64), (70, 69)])
def test_potrf_pivots_not_positive(ctx, n, j, dtype):
    """A pivot that is negative, zero or no number is refused by its place, in any block; in the Cholesky form too."""
    import hcorepp_amd as H
    a = _spd(n, dtype)
    zero = np.eye(n, dtype=dtype)
    zero[j, j] = 0
    nan, neg = a.copy(), a.copy()
    nan[j, j], neg[j, j] = np.nan, -1
    for bad in (zero, nan, neg):
        for uplo in "LU":
            with pytest.raises(H.HCoreError, match=f"NUMERIC.*minor {j + 1} "):
                H.HCore.potrf(H.DenseTile(bad, dtype=dtype), uplo, ctx)
        if dtype == np.float64:
            d = H.DenseTile(bad).c()
            with pytest.raises(H.HCoreError, match=f"NUMERIC.*pivot {j + 1}\\)"):
                H._check(H.lib().hcorepp_potrf_d(ctx.h, C.byref(d)))


@pytest.mark.parametrize("dtype,scale", [(np.float64, 2.0 ** -940), (np.float64, 2.0 ** 940), (np.float32, 2.0 ** -106),
                                         (np.float32, 2.0 ** 106)])
@pytest.mark.parametrize("n", [20, 70])
def test_potrf_scales(ctx, n, dtype, scale):
    """Pivots beyond the range of the reciprocal square root: |A - L L^T| <= (n + 2) eps |L| |L|^T."""
    import hcorepp_amd as H
    a = _spd(n, dtype) * dtype(scale)
    t = H.DenseTile(a, dtype=dtype)
    H.HCore.potrf(t, "L", ctx)
    l = np.tril(t.to_numpy()).astype(float)
    diff = np.abs(np.tril(a.astype(float) - l @ l.T))
    assert np.all(diff <= (n + 2) * np.finfo(dtype).eps * (abs(l) @ abs(l).T))
