"""Plain form on blocks of more than 1024 rows, which have a register shape of their own: rows around its limits (a wave's
groups of 16 rows, the ends of a round of eight waves), either dimension the tall one, one panel and several.  Nothing is
truncated; the bound is that of two Householder QRs and a Jacobi, a few K eps, with a margin of about 30."""
import numpy as np
import pytest

from helpers import rel_fro

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,eps", [(np.float64, 2.2e-16), (np.float32, 1.2e-7)])
@pytest.mark.parametrize("ra,rc", [(1, 0), (2, 1), (16, 0), (20, 13)])
@pytest.mark.parametrize("m,n", [(1024, 1026), (1041, 1025), (1151, 40), (33, 1153), (1537, 1300), (2047, 50), (50, 2048)])
def test_tall_blocks(ctx, m, n, ra, rc, dtype, eps):
    import hcorepp_amd as H
    rng = np.random.default_rng(m + 3 * n + ra)

    def pair(p, q, r):
        return rng.standard_normal((p, r)) / np.sqrt(p), rng.standard_normal((r, q)) / np.sqrt(q)

    a, b, c = pair(m, 24, ra), pair(24, n, min(24, ra + 2)), pair(m, n, rc)
    full = c[0] @ c[1] + (a[0] @ a[1]) @ (b[0] @ b[1])
    print(f"[case] {m}x{n} ra={ra} rc={rc} {dtype.__name__}", flush=True)
    tile = lambda f, **kw: H.CompressedTile(*(x.astype(dtype) for x in f), dtype=dtype, **kw)  # noqa: E731
    C = tile(c, max_rank=ra + rc)
    H.HCore.gemm(1.0, tile(a), tile(b), 1.0, C, ctx, H.CompressionParameters(eps * 1e-3))
    assert rel_fro(C.to_dense(), full) < 100 * (ra + rc + 1) * eps
    u = C.factors()[0].astype(np.float64)
    assert np.abs(u.T @ u - np.eye(u.shape[1])).max() < 100 * (ra + rc + 1) * eps


@pytest.mark.parametrize("m,n", [(10, 2049), (2050, 10)])
def test_taller_blocks_are_refused(ctx, m, n):
    """More than 2048 rows of either QR, with the number and the limit in the message; C stays as it was."""
    import hcorepp_amd as H
    a, b, c = (np.ones((m, 1)), np.ones((1, 9))), (np.ones((9, 1)), np.ones((1, n))), (np.ones((m, 1)), np.ones((1, n)))
    C = H.CompressedTile(*c, max_rank=2)
    with pytest.raises(H.HCoreError, match=f"UNSUPPORTED.*{max(m, n)} rows.*2048"):
        H.HCore.gemm(1.0, H.CompressedTile(*a), H.CompressedTile(*b), 1.0, C, ctx, H.CompressionParameters(1e-8))
    assert C.rank == 1 and all(np.array_equal(x, y) for x, y in zip(C.factors(), c))
