"""Core Jacobi at the edges of its tiles and paths: core widths around a block (8), a tile (16), the
LDS-resident and staged limits of the batched form (93 columns; 138, 276 and 554 rows), and the
one-workgroup / multi-workgroup limit of the plain form (112 columns), in FP64 (plain and batched) and
FP32.  The stacked factors have full rank and a flat spectrum, so the core keeps all its columns and
nothing is truncated: the result is the dense C + A B.

Tolerances (relative Frobenius error): plain FP64 and FP32, 100 K eps, the bound of the QRs and of the
Jacobi's backward error with a margin of about 30; batched FP64, whose Jacobi stops at cosines of about
1e-10, 1e-9."""
import numpy as np
import pytest

from helpers import rel_fro

pytestmark = pytest.mark.gpu

# stacked rank K, tile rows m (n = m)
SIZES = [(2, 16), (7, 40), (8, 33), (9, 64), (15, 64), (16, 50), (17, 64), (31, 80), (33, 65), (64, 128), (93, 128),
         (94, 128), (95, 131), (111, 150), (112, 150), (113, 113), (127, 256), (138, 140), (139, 256), (200, 256),
         (276, 300), (277, 300)]


def _factors(m, K, seed):
    rng = np.random.default_rng(seed)
    ra = max(K // 2, 1)
    rc = K - ra

    def orth(rows, r):
        return np.linalg.qr(rng.standard_normal((rows, r)))[0]

    def diag(r):
        return np.linspace(1.0, 0.3, r)[:, None]

    # B's left factor starts with A's right one, so that the product keeps A's rank and spectrum
    va = orth(m, ra)
    ub = np.linalg.qr(np.hstack([va, orth(m, 1)]))[0]
    a = (orth(m, ra), diag(ra) * va.T)
    b = (ub, diag(ra + 1) * orth(m, ra + 1).T)
    c = (orth(m, rc), diag(rc) * orth(m, rc).T)
    return a, b, c


@pytest.mark.parametrize("K,m", SIZES)
def test_core_widths(ctx, K, m):
    import hcorepp_amd as H
    a, b, c = _factors(m, K, 1000 + K)
    full = c[0] @ c[1] + (a[0] @ a[1]) @ (b[0] @ b[1])
    params = H.CompressionParameters(1e-13)
    print(f"[case] K={K} m={m} plain", flush=True)
    C = H.CompressedTile(*c, max_rank=K)
    H.HCore.gemm(1.0, H.CompressedTile(*a), H.CompressedTile(*b), 1.0, C, ctx, params)
    assert rel_fro(C.to_dense(), full) < 100 * K * 2.2e-16
    u = C.factors()[0]
    assert np.linalg.norm(u.T @ u - np.eye(u.shape[1])) < 1e-13 * np.sqrt(m)
    print(f"[case] K={K} m={m} batch", flush=True)
    Cb = [H.CompressedTile(*c, max_rank=K) for _ in range(3)]
    bt = H.Batch(ctx, [H.CompressedTile(*a)] * 3, [H.CompressedTile(*b)] * 3, Cb, 1.0, 1.0, params)
    bt.run()
    assert bt.status()[0] == 0
    bt.sync_ranks_to_tiles()
    for t in Cb:
        assert rel_fro(t.to_dense(), full) < 1e-9
    bt.close()
    print(f"[case] K={K} m={m} fp32", flush=True)
    f = lambda t: tuple(x.astype(np.float32) for x in t)  # noqa: E731
    C32 = H.CompressedTile(*f(c), max_rank=K, dtype=np.float32)
    H.HCore.gemm(1.0, H.CompressedTile(*f(a), dtype=np.float32), H.CompressedTile(*f(b), dtype=np.float32), 1.0, C32,
                 ctx, H.CompressionParameters(1e-6))
    assert rel_fro(C32.to_dense(), full) < 100 * K * 1.2e-7


def test_staged_limits_tall(ctx):
    """Cores on either side of the last staged height (554 rows; rotated in global memory above it)."""
    import hcorepp_amd as H
    for K in (553, 556):
        a, b, c = _factors(600, K, K)
        full = c[0] @ c[1] + (a[0] @ a[1]) @ (b[0] @ b[1])
        print(f"[case] staged K={K}", flush=True)
        Cb = H.CompressedTile(*c, max_rank=K)
        bt = H.Batch(ctx, [H.CompressedTile(*a)], [H.CompressedTile(*b)], [Cb], 1.0, 1.0, H.CompressionParameters(1e-13))
        bt.run()
        assert bt.status()[0] == 0
        bt.sync_ranks_to_tiles()
        assert rel_fro(Cb.to_dense(), full) < 1e-9
        bt.close()
