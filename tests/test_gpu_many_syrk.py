"""Batched syrk on either side of the lines between three launches of output tiles and a workgroup per tile."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ranks,count", [(32, (3, 0, 40), 300), (33, (3, 0, 40), 256), (33, (3, 0, 40), 257), (65, (64, 1), 300),
                                           (129, (5, 33), 384), (129, (5, 33), 385)])
def test_syrk_of_many_tiles(ctx, n, ranks, count):
    """C - U (V V^T) U^T of tiles of several ranks and of fewer rows than the largest; the bound is that of three products and a
    subtraction."""
    import hcorepp_amd as H
    eps = np.finfo(np.float64).eps
    rng = np.random.default_rng(n + count)
    us, vs, gs = [], [], []
    for i in range(count):
        m, r = n - (i % 3), ranks[i % len(ranks)]
        us.append(rng.standard_normal((m, r)))
        vs.append(rng.standard_normal((r, m)))
        gs.append(rng.standard_normal((m, m)))
    A = [H.CompressedTile(u, v, max_rank=max(ranks)) for u, v in zip(us, vs)]
    D = [H.DenseTile(g) for g in gs]
    print(f"[case] {n} {ranks} x {count}", flush=True)
    H._check(H.lib().hcorepp_syrk_batch_d(ctx.h, count, (H._Tile * count)(*[a.c() for a in A]),
                                          (H._Tile * count)(*[d.c() for d in D])))
    ctx.sync()
    for u, v, g, d in zip(us, vs, gs, D):
        out = d.to_numpy()
        assert np.array_equal(np.triu(out, 1), np.zeros_like(out))
        au, av, r = abs(u), abs(v), u.shape[1]
        bound = 2 * (len(g) + 2 * r + 3) * eps * (au @ (av @ av.T) @ au.T + abs(g))
        assert np.all(abs(np.tril(out - (g - u @ (v @ v.T) @ u.T))) <= bound)
