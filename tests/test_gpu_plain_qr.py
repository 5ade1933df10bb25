"""Plain-form QR, reconstruction and rank rule at the edges of their blocks: rows around the 16-row groups
and around the limits between register shapes (128, 256, 512, 1024 rows), stacked ranks around the 16-column
panel, tiles with fewer rows or columns than stacked columns, FP64 and FP32.  Nothing is truncated, so the
result is the dense C + A B; the bound is that of two Householder QRs and a Jacobi, a few K eps, with a margin
of about 30."""
import numpy as np
import pytest

from helpers import rel_fro

pytestmark = pytest.mark.gpu

# rows, columns of C, rank of A, rank of C
SHAPES = [(1, 1, 1, 0), (3, 5, 1, 1), (15, 16, 3, 4), (16, 17, 8, 8), (17, 15, 8, 9), (20, 33, 15, 25), (33, 20, 16, 17),
          (127, 128, 15, 16), (128, 129, 16, 16), (129, 127, 17, 16), (255, 257, 31, 18), (512, 513, 20, 13),
          (513, 300, 40, 25), (1024, 200, 17, 16), (1025, 70, 16, 1), (64, 1100, 20, 30), (2048, 2047, 9, 8)]


def _pair(rng, m, n, r):
    return rng.standard_normal((m, r)) / np.sqrt(m), rng.standard_normal((r, n)) / np.sqrt(n)


@pytest.mark.parametrize("dtype,eps", [(np.float64, 2.2e-16), (np.float32, 1.2e-7)])
@pytest.mark.parametrize("m,n,ra,rc", SHAPES)
def test_block_edges(ctx, m, n, ra, rc, dtype, eps):
    import hcorepp_amd as H
    rng = np.random.default_rng(m * 7 + n)
    k = 24
    a, b = _pair(rng, m, k, ra), _pair(rng, k, n, min(k, ra + 2))
    c = _pair(rng, m, n, rc) if rc else (np.zeros((m, 0)), np.zeros((0, n)))
    full = c[0] @ c[1] + (a[0] @ a[1]) @ (b[0] @ b[1])
    print(f"[case] {m}x{n} ra={ra} rc={rc} {dtype.__name__}", flush=True)
    tile = lambda f, **kw: H.CompressedTile(*(x.astype(dtype) for x in f), dtype=dtype, **kw)  # noqa: E731
    C = tile(c, max_rank=max(ra + rc, 1))
    _, sig = H.HCore.gemm(1.0, tile(a), tile(b), 1.0, C, ctx, H.CompressionParameters(eps * 1e-3), want_sigma=True)
    assert rel_fro(C.to_dense(), full) < 100 * (ra + rc + 1) * eps
    want = np.linalg.svd(full, compute_uv=False)[: len(sig)]
    assert np.all(np.abs(sig - want) < 100 * (ra + rc + 1) * eps * want[0])
    u = C.factors()[0].astype(np.float64)
    good = sig[: u.shape[1]] > 1e3 * eps * sig[0]
    g = u[:, good].T @ u[:, good]
    assert np.abs(g - np.eye(len(g))).max() < 100 * (ra + rc + 1) * eps


@pytest.mark.parametrize("ra,rc", [(520, 520), (520, 521), (530, 530)])
def test_more_stacked_columns_than_one_launch_row(ctx, ra, rc):
    """Stacked ranks on either side of 1040, where the first trailing updates go from 4 columns per workgroup to 16; the
    result has full rank, so nothing is truncated.  Bound as above."""
    import hcorepp_amd as H
    rng = np.random.default_rng(ra + 3 * rc)
    m, n, k = 600, 560, 540
    a, b, c = _pair(rng, m, k, ra), _pair(rng, k, n, ra), _pair(rng, m, n, rc)
    full = c[0] @ c[1] + (a[0] @ a[1]) @ (b[0] @ b[1])
    C = H.CompressedTile(*c, max_rank=n)
    H.HCore.gemm(1.0, H.CompressedTile(*a), H.CompressedTile(*b), 1.0, C, ctx, H.CompressionParameters(1e-14))
    assert rel_fro(C.to_dense(), full) < 100 * (ra + rc + 1) * 2.2e-16
