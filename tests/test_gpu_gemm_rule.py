"""Dense products on either side of the lines between the 32 x 32 and the 64 x 64 form: one to four rounds of 256 tiles and
the K where each changes, by transposes.  The bound is that of a K-term sum, K eps |A| |B|."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# the last of one round and the first of two, three and four, then 256 tiles of 64 x 64
SHAPES = [(512, 512), (544, 512), (33 * 32, 31), (704, 704), (736, 705), (832, 832), (896, 880), (960, 961), (1024, 1024)]


@pytest.mark.parametrize("k", [32, 33, 127, 128, 511, 512])
@pytest.mark.parametrize("m,n", SHAPES)
def test_products_around_the_rule(ctx, m, n, k):
    import hcorepp_amd as H
    eps = np.finfo(np.float64).eps
    rng = np.random.default_rng(m + n + k)
    a, b = rng.standard_normal((m, k)), rng.standard_normal((k, n))
    want, bound = a @ b, (k + 4) * eps * (np.abs(a) @ np.abs(b))
    for ta, tb in (("N", "N"), ("N", "T"), ("T", "N")):
        A, B = (H.DeviceBuffer.from_numpy(np.asfortranarray(x).reshape(-1, order="F"))
                for x in (a.T if ta == "T" else a, b.T if tb == "T" else b))
        C = H.DeviceBuffer(8 * m * n)
        H._check(H.lib().hcorepp_kernel_gemm_d(ctx.h, ta.encode(), tb.encode(), m, n, k, 1.0, A.ptr,
                                               k if ta == "T" else m, B.ptr, n if tb == "T" else k, 0.0, C.ptr, m))
        ctx.sync()
        assert np.all(np.abs(C.download(np.float64).reshape(m, n, order="F") - want) <= bound), (ta, tb)
