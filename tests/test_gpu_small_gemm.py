"""Dense products around the 32 x 32 tiles, the 16-deep chunks and the eight-way split of K of the small
form, and on either side of the size where the 64 x 64 form takes over, all transposes, FP64 and FP32;
the bound is that of a K-term sum, K eps |A| |B|."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (31, 33, 15), (32, 32, 16), (33, 31, 17), (64, 72, 127), (65, 63, 129), (40, 500, 512), (17, 90, 513),
          (200, 130, 640), (960, 1000, 20), (1024, 1025, 33), (5, 7, 0)]


@pytest.mark.parametrize("dtype,eps", [(np.float64, 2.2e-16), (np.float32, 1.2e-7)])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_dense_products(ctx, m, n, k, dtype, eps):
    import hcorepp_amd as H
    rng = np.random.default_rng(m + 3 * n + 7 * k)
    for ta, tb, beta in (("N", "N", 0.0), ("N", "T", 0.5), ("T", "N", -1.0), ("T", "T", 1.0)):
        a, b = rng.standard_normal((m, k)).astype(dtype), rng.standard_normal((k, n)).astype(dtype)
        c = rng.standard_normal((m, n)).astype(dtype)
        if dtype == np.float64:  # the raw kernel entry point takes any leading dimension and K = 0
            A, B, C = (H.DeviceBuffer.from_numpy(np.asfortranarray(x).reshape(-1, order="F"))
                       for x in (a.T if ta == "T" else a, b.T if tb == "T" else b, c))
            H._check(H.lib().hcorepp_kernel_gemm_d(ctx.h, ta.encode(), tb.encode(), m, n, k, 1.5, A.ptr,
                                                   max(k if ta == "T" else m, 1), B.ptr, max(n if tb == "T" else k, 1),
                                                   beta, C.ptr, m))
            ctx.sync()
            got = C.download(np.float64).reshape(m, n, order="F")
        else:
            if k == 0 or ta == "T" or tb == "T":
                continue
            Ct = H.DenseTile(c, dtype=dtype)
            H.HCore.gemm(1.5, H.DenseTile(a, dtype=dtype), H.DenseTile(b, dtype=dtype), beta, Ct, ctx)
            ctx.sync()
            got = Ct.to_numpy()
        a, b, c = (x.astype(np.float64) for x in (a, b, c))
        want = 1.5 * (a @ b) + beta * c
        bound = (k + 4) * eps * (1.5 * (np.abs(a) @ np.abs(b)) + np.abs(c))
        assert np.all(np.abs(got - want) <= bound + eps), (ta, tb, np.max(np.abs(got - want)))
