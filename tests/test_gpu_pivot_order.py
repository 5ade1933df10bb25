"""Pivoting of the plain form's QR of Y: the trailing columns of largest norm come first, compared by the whole norm
and by position where norms are equal, for every length of the lists its lanes sort (64, 256 and 768 columns)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,step", [(np.float64, 2.0 ** -30), (np.float64, 2.0 ** -44), (np.float32, 2.0 ** -22)])
@pytest.mark.parametrize("K", [24, 64, 65, 200, 257])
def test_close_norms_in_order(ctx, K, dtype, step):
    """C + A B whose stacked right factor is diagonal, so the columns of Y are multiples of unit vectors whose norms differ
    by `step` or not at all: the first panel's permutation is the stable descending sort, and in FP64 with steps far
    above the rounding of a panel's update so is the whole one."""
    import hcorepp_amd as H
    n = 300
    rng = np.random.default_rng(K)
    val = (1.0 - step * (rng.permutation(K) // 2)).astype(dtype)  # pairs of equal ones
    e = np.eye(n)
    tile = lambda u, v, **kw: H.CompressedTile(u, v, dtype=dtype, **kw)  # noqa: E731
    Ct = tile(e[:, :K - 1], val[:K - 1, None] * e[:K - 1, :], max_rank=K)
    A, B = tile(e[:, K - 1:K], e[:1, :]), tile(e[:, :1], val[K - 1] * e[K - 1:K, :])
    H.HCore.gemm(1.0, A, B, 1.0, Ct, ctx, H.CompressionParameters(1e-3))
    info = np.zeros(16, dtype=np.int64)
    H.lib().hcorepp_debug_workspace(ctx.h, None, 0, info.ctypes.data_as(C.c_void_p))
    size, words = int(info[5]), int(info[6])
    ws = np.zeros(words * size, dtype=np.uint8)
    assert H.lib().hcorepp_debug_workspace(ctx.h, ws.ctypes.data_as(C.c_void_p), ws.nbytes,
                                           info.ctypes.data_as(C.c_void_p)) == ws.nbytes
    # the permutation lies before the region of info[15], rounded up to 32 elements
    at = (int(info[15]) - (-(-K * 4 // size) + 31) // 32 * 32) * size
    piv = ws[at:at + 4 * K].view(np.int32)
    assert np.array_equal(np.sort(piv), np.arange(K))
    want = np.argsort(-(val * val), kind="stable")
    sure = K if step > 2.0 ** -35 and dtype == np.float64 else 16
    got = piv[:sure]
    if sure == K:  # equal norms may swap once a panel's update has rounded them
        assert np.array_equal(got[:16], want[:16])
        assert np.array_equal(val[got], val[want])
    else:
        assert np.array_equal(got, want[:16])
