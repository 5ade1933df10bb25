"""Mixed-precision factor products (64 x 64 tiles, 16-deep chunks of sliced operands) at the edges of their tiles."""
import numpy as np
import pytest

from helpers import rel_fro

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,ra,rb,rc", [(1, 1, 1, 1), (16, 16, 15, 3), (63, 17, 16, 1), (64, 1, 33, 20), (65, 40, 7, 9),
                                         (129, 65, 64, 30), (200, 31, 90, 66)])
def test_mixed_products_at_tile_edges(ctx, nb, ra, rb, rc):
    """C += A B in the mixed form against the dense sum.  A term of a factor product is within a few 2^-40 of
    its row's and column's largest magnitudes; products of up to 200 terms, with the factors scaled apart by powers of
    two, stay far below the form's 1e-8."""
    import hcorepp_amd as H
    from hcorepp_amd.workloads import lowrank_factors
    rng = np.random.default_rng(nb)
    (au, av), (bu, bv), (cu, cv) = (lowrank_factors(rng, nb, nb, r, 0.9) for r in (ra, rb, rc))
    av, bu = av * 2.0 ** -7, bu * 2.0 ** 9
    A, B = H.CompressedTile(au, av), H.CompressedTile(bu, bv)
    C = H.CompressedTile(cu, cv, max_rank=min(nb, min(ra, rb) + rc))
    b = H.Batch(ctx, [A], [B], [C], 1.0, 1.0, H.CompressionParameters(1e-12), H.PREC_MIXED)
    b.run()
    b.sync_ranks_to_tiles()
    assert b.status()[0] == 0
    b.close()
    want = (au @ av) @ (bu @ bv) + cu @ cv
    assert rel_fro(C.to_dense(), want) < 1e-8
