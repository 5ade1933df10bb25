"""Products into a dense C with transposed operands of any shape, dense and compressed, and operands that do not fit C.
Bounds: a K-term sum, K eps |A| |B|, with the magnitudes of the factors where an operand is compressed."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(5, 7, 3), (3, 5, 7), (7, 3, 5), (40, 33, 50), (100, 30, 8), (30, 100, 8), (64, 65, 1)]


@pytest.mark.parametrize("dtype,eps", [(np.float64, 2.2e-16), (np.float32, 1.2e-7)])
@pytest.mark.parametrize("opA,opB", [("N", "N"), ("T", "N"), ("N", "T"), ("T", "T")])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_transposed_operands(ctx, m, n, k, opA, opB, dtype, eps):
    import hcorepp_amd as H
    rng = np.random.default_rng(m + 2 * n + 5 * k)
    r = min(m, n, k, 4)

    def operand(rows, cols, op, compressed):
        if op == "T":
            rows, cols = cols, rows
        if compressed:
            u, v = (rng.standard_normal(s).astype(dtype) for s in ((rows, r), (r, cols)))
            t, x, size = H.CompressedTile(u, v, max_rank=r + 1, dtype=dtype), u.astype(float) @ v, abs(u).astype(float) @ abs(v)
        else:
            x = rng.standard_normal((rows, cols)).astype(dtype)
            t, size = H.DenseTile(x, dtype=dtype), abs(x)
        return (t, x.T, size.T) if op == "T" else (t, x, size)

    for ca, cb in ((False, False), (True, False), (False, True), (True, True)):
        A, a, sa = operand(m, k, opA, ca)
        B, b, sb = operand(k, n, opB, cb)
        c = rng.standard_normal((m, n)).astype(dtype)
        C = H.DenseTile(c, dtype=dtype)
        print(f"[case] {m}x{n}x{k} {opA}{opB} {ca} {cb}", flush=True)
        H.HCore.gemm(1.5, A, B, -0.5, C, ctx, opA=opA, opB=opB)
        want = 1.5 * (a.astype(float) @ b.astype(float)) - 0.5 * c
        bound = (k + 2 * r + 6) * eps * (1.5 * (sa.astype(float) @ sb.astype(float)) + abs(c))
        assert np.all(abs(C.to_numpy() - want) <= bound), (ca, cb, np.max(abs(C.to_numpy() - want) / bound))


def test_operands_too_small_are_refused(ctx):
    """Operands that C would read past are an error on the host; C stays as it was."""
    import hcorepp_amd as H
    z = lambda *s: H.DenseTile(np.ones(s))  # noqa: E731
    for A, B, opA, opB in ((z(50, 40), z(40, 30), "N", "N"), (z(60, 40), z(40, 20), "N", "N"),
                           (z(40, 50), z(40, 30), "T", "N"), (z(60, 40), z(20, 40), "N", "T")):
        C = z(60, 30)
        with pytest.raises(H.HCoreError, match="INVALID"):
            H.HCore.gemm(1.0, A, B, 0.0, C, ctx, opA=opA, opB=opB)
        assert np.array_equal(C.to_numpy(), np.ones((60, 30)))
