"""Core Jacobi of the batched form on either side of the limits between its forms, which go by rows | 1: LDS-resident (93
columns), 32 columns per super-block up to 137 rows, whose LDS is full at 136 and 137, 16 up to 277, 8 up to 555, rotated in
global memory beyond.  The stacked factors have full rank and a flat spectrum, so the core keeps all its columns and
nothing is truncated.  The form stops at cosines of about 1e-10: 1e-9 for the product and for U^T U - I."""
import numpy as np
import pytest

from helpers import rel_fro

pytestmark = pytest.mark.gpu


def _factors(m, K, seed):
    rng = np.random.default_rng(seed)
    ra = K // 2
    rc = K - ra

    def orth(rows, r):
        return np.linalg.qr(rng.standard_normal((rows, r)))[0]

    def diag(r):
        return np.linspace(1.0, 0.3, r)[:, None]

    va = orth(m, ra)
    ub = np.linalg.qr(np.hstack([va, orth(m, 1)]))[0]
    return (orth(m, ra), diag(ra) * va.T), (ub, diag(ra + 1) * orth(m, ra + 1).T), (orth(m, rc), diag(rc) * orth(m, rc).T)


@pytest.mark.parametrize("K", [93, 94, 136, 137, 138, 276, 277, 278, 555, 556])
def test_staged_limits(ctx, K):
    import hcorepp_amd as H
    a, b, c = _factors(K + 3, K, 3 * K)
    full = c[0] @ c[1] + (a[0] @ a[1]) @ (b[0] @ b[1])
    print(f"[case] staged K={K}", flush=True)
    C = H.CompressedTile(*c, max_rank=K)
    bt = H.Batch(ctx, [H.CompressedTile(*a)], [H.CompressedTile(*b)], [C], 1.0, 1.0, H.CompressionParameters(1e-13))
    bt.run()
    assert bt.status()[0] == 0
    bt.sync_ranks_to_tiles()
    assert bt.core_widths()[0] == K
    bt.close()
    assert rel_fro(C.to_dense(), full) < 1e-9
    u = C.factors()[0]
    assert np.linalg.norm(u.T @ u - np.eye(K)) < 1e-9


def test_batched_u_is_orthonormal(ctx):
    """||U^T U - I||_F of the benchmark's kind of updates (512 rows, ranks 8 to 192, decay 0.85): the form's 1e-10, of which
    the largest of 256 was 4.6e-11."""
    import hcorepp_amd as H
    from hcorepp_amd.workloads import batch_ccc
    ups = batch_ccc(96, 512, seed=1)
    Cs = [H.CompressedTile(u["cu"], u["cv"], max_rank=384) for u in ups]
    b = H.Batch(ctx, [H.CompressedTile(u["au"], u["av"]) for u in ups], [H.CompressedTile(u["bu"], u["bv"]) for u in ups], Cs,
                1.0, 1.0, H.CompressionParameters(1e-8))
    b.run()
    b.sync_ranks_to_tiles()
    assert b.status()[0] == 0
    b.close()
    off = []
    for t in Cs:
        u = t.factors()[0]
        off.append(np.linalg.norm(u.T @ u - np.eye(u.shape[1])))
    print(f"median {np.median(off):.1e}, largest {max(off):.1e}")
    assert max(off) < 1e-9 and np.median(off) < 1e-12
