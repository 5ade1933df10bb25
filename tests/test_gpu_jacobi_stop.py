"""The end of the batched form's Jacobi: a sweep ends it when no pair it met had a cosine above 1e-5, compared in full
precision."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _updates(rng, cos, count):
    """C + A B of rank 2 whose core has two columns with exactly that cosine: the stacked left factor is (e0, e1), the
    stacked right one (a e0, b e0 + c e1) with c < a, so R = [[a, b], [0, c]] and the cosine b / hypot(a, b)."""
    import hcorepp_amd as H
    n = 8
    e = np.eye(n)
    As, Bs, Cs = [], [], []
    for _ in range(count):
        a = rng.uniform(1.0, 2.0)
        c = rng.uniform(0.1, 0.9) * a
        b = a * cos / np.sqrt(1.0 - cos * cos)
        As.append(H.CompressedTile(e[:, 1:2], e[:1, :]))
        Bs.append(H.CompressedTile(e[:, :1], b * e[:1, :] + c * e[1:2, :]))
        Cs.append(H.CompressedTile(e[:, :1], a * e[:1, :], max_rank=2))
    return As, Bs, Cs


def _sweeps(ctx, updates):
    import hcorepp_amd as H
    b = H.Batch(ctx, *updates, 1.0, 1.0, H.CompressionParameters(1e-12))
    b.run()
    st, sweeps = b.status()
    assert st == 0 and np.array_equal(b.ranks(), np.full(b.n, 2))
    b.close()
    return sweeps


def test_stop_bound_to_rounding(ctx):
    """Cosines a hundred-millionth above and below the bound (rounding of the core is 1e-10 of it at most): 64 pairs
    below it end after the sweep that meets them, each of 32 above it asks for another one."""
    rng = np.random.default_rng(11)
    assert _sweeps(ctx, _updates(rng, 1e-5 * (1 - 1e-8), 64)) == 0
    assert [_sweeps(ctx, _updates(rng, 1e-5 * (1 + 1e-8), 1)) for _ in range(32)] == [1] * 32
