"""Accuracy of the mixed form's factor products: the sums over a 16-deep chunk are exact, so all that is lost is the
slice pairs the form leaves out and what lies beyond a value's fourth slice."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(ctx, a, b, c, acc, max_rank):
    import hcorepp_amd as H
    C = H.CompressedTile(*c, max_rank=max_rank)
    bt = H.Batch(ctx, [H.CompressedTile(*a)], [H.CompressedTile(*b)], [C], 1.0, 1.0, H.CompressionParameters(acc),
                 H.PREC_MIXED)
    bt.run()
    bt.sync_ranks_to_tiles()
    assert bt.status()[0] == 0
    bt.close()
    return C.to_dense()


@pytest.mark.parametrize("seed", range(6))
def test_chunk_sums_are_exact(ctx, seed):
    """One dot product of 16 terms whose slices are known integers: the leading ones cancel, the next ones leave
    2^-7, and the pairs of weight 2^-40 add up to 1.25 x 2^24 of that unit, more than FP32 holds exactly in one sum.  The
    value is compared with the sum of the ten slice pairs in whole numbers.  The second product cuts it to 40 bits
    of its own scale (2^-47), and the rest is FP64: 4 x 2^-47 in all, 2^-45; one lost unit is 2^-40."""
    rng = np.random.default_rng(seed)
    n = 16
    sign = rng.permutation(np.repeat([1, -1], n // 2))
    xs = np.stack([np.full(n, 1023), rng.integers(505, 512, n), sign * rng.integers(505, 512, n)])
    ys = np.stack([1023 * sign, rng.integers(505, 512, n), rng.integers(505, 512, n)])
    # an odd sum of the pairs of weight 2^-40
    if (sum(int(xs[s] @ ys[2 - s]) for s in range(3)) % 2) == 0:
        ys[2, 0] += 1 if ys[2, 0] < 511 else -1
    assert sum(int(xs[s] @ ys[2 - s]) for s in range(3)) > 2 ** 24
    w = 2.0 ** (-10 * np.arange(1, 4))
    x, y = w @ xs, w @ ys
    want = sum(int(xs[s] @ ys[t]) * 2.0 ** (-10 * (s + t + 2)) for s in range(3) for t in range(3) if s + t < 4)
    e = np.eye(n)
    a, b = (e[:, :1], x[None, :]), (y[:, None], e[:1, :])
    c = (e[:, 1:2], e[1:2, :] * 2.0 ** -7)
    got = _run(ctx, a, b, c, 1e-14, 2)
    assert abs(got[0, 0] - want) < 2.0 ** -45, (got[0, 0] - want) * 2.0 ** 40


@pytest.mark.parametrize("nb,ra,rb,rc", [(16, 16, 15, 3), (65, 40, 7, 9), (129, 65, 64, 30), (200, 31, 90, 66)])
def test_rows_and_columns_scaled_apart(ctx, nb, ra, rb, rc):
    """Factors whose rows and columns differ by powers of two drawn one by one, against the dense sum, elementwise.  A term
    of a product loses at most 2^-40 of its row's and column's scales for the values' rests, as much for the pairs
    left out, and a scale is at most twice the largest magnitude: 8 x 2^-40 of those per term.  The products
    may be taken from either side, so the larger bound of the two orders holds; the recompression adds FP64
    rounding of the whole tile."""
    rng = np.random.default_rng(nb + 1)

    def spread(k):
        return 2.0 ** rng.integers(-6, 7, k)

    au, av = rng.standard_normal((nb, ra)) * spread(nb)[:, None], rng.standard_normal((ra, nb)) * spread(ra)[:, None]
    bu, bv = rng.standard_normal((nb, rb)) * spread(rb)[None, :], rng.standard_normal((rb, nb)) * spread(nb)[None, :]
    cu, cv = rng.standard_normal((nb, rc)), rng.standard_normal((rc, nb))
    got = _run(ctx, (au, av), (bu, bv), (cu, cv), 1e-13, min(nb, min(ra, rb) + rc))
    full = (au @ av) @ (bu @ bv) + cu @ cv

    def loss(p, q):
        return 8 * p.shape[1] * 2.0 ** -40 * np.outer(np.abs(p).max(1), np.abs(q).max(0))

    core, e = av @ bu, loss(av, bu)
    left = (loss(au, core) + np.abs(au) @ e) @ np.abs(bv)
    right = np.abs(au) @ (loss(core, bv) + e @ np.abs(bv))
    bound = np.maximum(left, right) + 1e-12 * np.linalg.norm(full)
    assert np.all(np.abs(got - full) <= bound), np.max(np.abs(got - full) / bound)
