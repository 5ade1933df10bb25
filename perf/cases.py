"""Performance cases of the TLR tile GEMM + recompression library.

Each case is one use of the public entry points on device-resident tiles: single tile updates
(``HCore.gemm`` with compressed and dense operands), the compression of a dense tile, the batched
form, the Cholesky-flow tile operations and a whole TLR Cholesky factorisation.

The factors of a truncated SVD are unique only up to signs (and rotations of near-equal singular
values), so a compressed result is returned as the tile it stands for, U * V formed on the device,
with its rank beside it.  Tiles live in torch tensors; a pass restores the tiles that the last
pass overwrote, as a program that reuses its buffers does, and then makes its calls.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import hcorepp_amd as H
from hcorepp_amd.cholesky import TLRCholesky
from hcorepp_amd.workloads import TLRMatrix, covariance_matrix, covariance_points, prefetch_tiles

_DTYPES = {"f64": (torch.float64, np.float64), "f32": (torch.float32, np.float32)}
_CONTEXT = []


def _ctx():
    """The one context a program keeps for all its calls."""
    if not _CONTEXT:
        _CONTEXT.append(H.RunContext(0))
    return _CONTEXT[0]


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------
def _gemm(name, combo, m, n, k, ra, rb, rc, cap, acc, decay, dtype="f64", fixed=0, op_b="N"):
    return {"name": name, "kind": "gemm", "combo": combo, "m": m, "n": n, "k": k, "ra": ra, "rb": rb, "rc": rc,
            "cap": cap, "acc": acc, "decay": decay, "dtype": dtype, "fixed": fixed, "op_b": op_b}


def _batch(name, count, nb, lo, hi, cap, ragged, form, acc=1e-8, decay=0.85):
    return {"name": name, "kind": "batch", "count": count, "nb": nb, "lo": lo, "hi": hi, "cap": cap,
            "ragged": ragged, "form": form, "acc": acc, "decay": decay}


def listed():
    return [
        # A small tile update on its own: 128 x 128 with ranks 12, 10 and 16, the size of a first
        # call; all latency and launches.
        _gemm("gemm_128", "CCC", 128, 128, 128, 12, 10, 16, 64, 1e-8, 0.8),
        # One update of the reference example's 4 x 4-tile GEMM: nb = 256, capacity nb / 3.
        _gemm("gemm_256", "CCC", 256, 256, 256, 62, 58, 70, 85, 1e-8, 0.8),
        # One update of the nb = 1024 covariance GEMM at accuracy 1e-10, capacity nb / 3: the
        # largest single tile.
        _gemm("gemm_1024", "CCC", 1024, 1024, 1024, 310, 290, 331, 341, 1e-10, 0.93),
        # A ragged edge tile with a dense left operand (a diagonal tile times a compressed one).
        _gemm("gemm_dcc_ragged", "DCC", 500, 437, 509, 0, 91, 102, 170, 1e-8, 0.85),
        # Single precision, ragged, truncated to a fixed rank (the fixed-rank drivers).
        _gemm("gemm_f32_fixed", "CCC", 384, 321, 300, 40, 44, 48, 64, 1e-4, 0.7, "f32", 32),
        # Accumulation of a compressed product into a dense (diagonal) tile: the cheapest call,
        # three small products.
        _gemm("dense_c_512", "CCD", 512, 512, 512, 64, 72, 0, 0, 1e-8, 0.85),
        # Building a TLR matrix: one off-diagonal covariance tile compressed from host memory.
        {"name": "compress_512", "kind": "compress", "m": 512, "n": 512, "cap": 170, "acc": 1e-8, "dtype": "f64"},
        # The trailing updates of a small factorisation step: a few dozen ragged updates, exact form.
        _batch("batch_48_ragged", 48, 256, 8, 96, 128, True, "exact"),
        # A step of a mid-size TLR GEMM: one update per compute unit, mixed-precision factor
        # products with the tolerance rule.
        _batch("batch_256_mixed", 256, 512, 8, 192, 192, False, "mixed_rule"),
        # The benchmark's batch: 4096 updates, nb = 512, ranks log-uniform in 8..192, tolerance
        # rule, replayed from a captured graph.
        _batch("batch_4096_rule", 4096, 512, 8, 192, 192, False, "rule_graph"),
        # One column step of a factorisation through the Cholesky-flow tile operations, tile by tile.
        {"name": "chol_step_512", "kind": "chol_step", "nb": 512, "rank": 96, "cap": 170, "tiles": 3, "acc": 1e-8,
         "dtype": "f64"},
        # A whole TLR Cholesky of a 3-D covariance matrix, batched driver.
        {"name": "cholesky_12x256", "kind": "cholesky", "tiles": 12, "nb": 256, "acc": 1e-6},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _unnamed(case):
    return {k: v for k, v in case.items() if k != "name"}


def draw(rng):
    pick = rng.random()
    if pick < 0.45:
        nb = _log_int(rng, 96, 1024)
        square = rng.random() < 0.5
        m, n, k = (nb, nb, nb) if square else (max(64, nb - rng.randrange(nb // 4)) for _ in range(3))
        cap = max(8, min(m, n) // 3)
        ra, rb, rc = (_log_int(rng, 6, min(cap, min(m, n, k) // 2)) for _ in range(3))
        form = rng.random()
        if form < 0.2:
            combo = rng.choice(["CCD", "CDD", "DDD"])
            op_b = rng.choice(["N", "T"]) if combo == "DDD" and square else "N"
            return _unnamed(_gemm("", combo, m, n, k, ra, rb, 0, 0, 1e-8, 0.85, rng.choice(["f64", "f32"]), 0, op_b))
        if form < 0.4:
            ra, rb, rc = (min(x, 48) for x in (ra, rb, rc))
            fixed = max(4, min(cap, ra + rc, 72) // 2)
            return _unnamed(_gemm("", "CCC", m, n, k, ra, rb, rc, cap, 1e-4, 0.7, "f32", fixed))
        combo = rng.choice(["CCC", "CCC", "DCC", "CDC"])
        return _unnamed(_gemm("", combo, m, n, k, ra, rb, rc, cap, 1e-8, rng.choice([0.8, 0.85, 0.9])))
    if pick < 0.55:
        m, n = _log_int(rng, 96, 600), _log_int(rng, 96, 600)
        return {"kind": "compress", "m": m, "n": n, "cap": max(min(m, n) // 3, 1), "acc": 1e-8, "dtype": "f64"}
    if pick < 0.85:
        nb = rng.choice([128, 192, 256, 384, 512])
        hi = min(192, (nb * 3) // 8)
        return _unnamed(_batch("", _log_int(rng, 8, 1500), nb, 8, hi, hi, rng.random() < 0.3,
                               rng.choice(["exact", "rule", "rule_graph", "mixed_rule"])))
    if pick < 0.95:
        nb = _log_int(rng, 96, 640)
        return {"kind": "chol_step", "nb": nb, "rank": _log_int(rng, 8, nb // 4), "cap": nb // 3,
                "tiles": rng.randrange(2, 5), "acc": 1e-8, "dtype": "f64"}
    return {"kind": "cholesky", "tiles": rng.randrange(4, 12), "nb": rng.choice([128, 160, 200, 256]), "acc": 1e-6}


# ---------------------------------------------------------------------------
# Tiles over torch memory
# ---------------------------------------------------------------------------
class _Dense(H.DenseTile):
    """A dense tile over device memory that a torch tensor holds (column-major, leading dimension ld)."""

    def __init__(self, rows, cols, buf, ld=None, dtype=np.float64):
        self.rows, self.cols, self.ld = rows, cols, max(ld or rows, 1)
        self.rank = self.max_rank = min(rows, cols)
        self.dtype, self.buf = dtype, buf


class _Compressed(H.CompressedTile):
    """A compressed tile [U rows x max_rank | V max_rank x cols] over a flat torch tensor."""

    def __init__(self, rows, cols, rank, max_rank, buf, dtype=np.float64):
        self.rows, self.cols, self.rank, self.max_rank, self.ld = rows, cols, rank, max_rank, rows
        self.dtype, self.buf = dtype, buf


def _copy(dst, src):
    H._check(H.lib().hcorepp_memcpy_async(_ctx().h, dst.data_ptr(), src.data_ptr(), dst.numel() * dst.element_size()))


def _product(tile, out, ld=None, v_cols=False):
    """out (a flat tensor) <- U * V of a compressed tile; v_cols: V is stored cols x rank."""
    m, n, r, off = tile.rows, tile.cols, tile.rank, tile.rows * tile.max_rank
    v = _Dense(n, r, tile.buf[off:], dtype=tile.dtype) if v_cols else _Dense(r, n, tile.buf[off:], dtype=tile.dtype)
    H.HCore.gemm(1.0, _Dense(m, r, tile.buf, dtype=tile.dtype), v, 0.0, _Dense(m, n, out, ld, tile.dtype), _ctx(),
                 opB="T" if v_cols else "N")


class _Bases:
    """Orthonormal factors: random column subsets of a few random orthogonal matrices per size."""

    POOL = 4

    def __init__(self, seed, device):
        self.rng, self.device, self.q = np.random.default_rng(seed), device, {}

    def __call__(self, rows, r):
        """r orthonormal columns of `rows` entries, as a rows x r tensor on the device."""
        if rows not in self.q:
            q = [np.linalg.qr(self.rng.standard_normal((rows, rows)))[0] for _ in range(self.POOL)]
            self.q[rows] = [torch.from_numpy(np.ascontiguousarray(x)).to(self.device) for x in q]
        cols = torch.from_numpy(self.rng.permutation(rows)[:r]).to(self.device)
        return self.q[rows][int(self.rng.integers(self.POOL))].index_select(1, cols)

    def factors(self, m, n, r, decay):
        """U (m x r, orthonormal) and V (r x n) carrying the singular values decay^i."""
        s = torch.from_numpy(decay ** np.arange(r, dtype=np.float64)).to(self.device)
        return self(m, r), (self(n, r) * s).T


def _put(flat, u, v, cap):
    """Factors into a flat tile buffer: U column-major, V (r x n) column-major with ld r."""
    m, r = u.shape
    n = v.shape[1]
    flat[: m * r].view(r, m).copy_(u.T)
    flat[m * cap: m * cap + n * r].view(n, r).copy_(v.T)


# ---------------------------------------------------------------------------
# Single updates
# ---------------------------------------------------------------------------
def _covariance(n, seed):
    """A smooth n-point covariance block, the dense (diagonal) tile of a TLR matrix."""
    return covariance_matrix(covariance_points(n, 3, seed), 0.3, 1e-2)


def _gemm_inputs(case, seed, device):
    """Operands of one update: (U, V) pairs of compressed tiles, matrices of dense ones, in the case's type."""
    td = _DTYPES[case["dtype"]][0]
    bases = _Bases(seed, device)
    m, n, k, combo = case["m"], case["n"], case["k"], case["combo"]

    def operand(form, rows, cols, r):
        if form == "D":
            p = max(rows, cols)
            a = torch.from_numpy(np.ascontiguousarray(_covariance(p, seed + rows)[:rows, :cols]) / math.sqrt(p))
            return a.to(device=device, dtype=td)
        u, v = bases.factors(rows, cols, max(r, 1), case["decay"])
        return u.to(td), v.to(td)

    a = operand(combo[0], m, k, case["ra"])
    b = operand(combo[1], *((n, k) if case["op_b"] == "T" else (k, n)), case["rb"])
    return a, b, operand(combo[2], m, n, case["rc"])


def _tile_of(x, cap, npd):
    """A device tile of an operand."""
    if isinstance(x, tuple):
        u, v = x
        cap = max(cap, u.shape[1])
        flat = torch.zeros((u.shape[0] + v.shape[1]) * cap, dtype=u.dtype, device="cuda")
        _put(flat, u, v, cap)
        return _Compressed(u.shape[0], v.shape[1], u.shape[1], cap, flat, npd)
    flat = x.T.contiguous().reshape(-1)
    return _Dense(x.shape[0], x.shape[1], flat, dtype=npd)


class _State:
    pass


def _prepare_gemm(case, seed):
    st, npd = _State(), _DTYPES[case["dtype"]][1]
    a, b, c = _gemm_inputs(case, seed, "cuda")
    st.kind, st.op_b = "gemm", case["op_b"]
    st.a, st.b, st.c = _tile_of(a, 0, npd), _tile_of(b, 0, npd), _tile_of(c, case["cap"], npd)
    st.c0, st.rank0 = st.c.buf.clone(), st.c.rank
    st.params = H.CompressionParameters(case["acc"], fixed_rank=case["fixed"])
    st.out = torch.empty(case["n"], case["m"], dtype=st.c0.dtype, device="cuda")
    return st


def _run_gemm(st):
    _copy(st.c.buf, st.c0)
    st.c.rank = st.rank0
    H.HCore.gemm(1.0, st.a, st.b, 1.0, st.c, _ctx(), st.params, opB=st.op_b)
    if st.c.type == H.DENSE:
        return {"c": st.c.buf}
    _product(st.c, st.out.view(-1))
    return {"c": st.out, "rank": st.c.rank}


def _truncate(us, vs, acc, cap, fixed=0):
    """(U, V) of the truncated SVD of us @ vs by the rank rule: the first singular value below acc (or the fixed rank)."""
    qu, ru = np.linalg.qr(us)
    qv, rv = np.linalg.qr(vs.T)
    w, s, zt = np.linalg.svd(ru @ rv.T)
    size = len(s)
    if fixed:
        r = min(fixed, size)
    else:
        below = np.nonzero(s[1:] < acc)[0]
        r = int(below[0]) + 1 if len(below) else size
    r = min(max(r, 1), cap)
    return qu @ w[:, :r], (s[:r, None] * zt[:r]) @ qv.T


def _host(x):
    return tuple(t.double().cpu().numpy() for t in x) if isinstance(x, tuple) else x.double().cpu().numpy()


def _exact_gemm(case, seed):
    a, b, c = (_host(x) for x in _gemm_inputs(case, seed, "cpu"))
    full = [x[0] @ x[1] if isinstance(x, tuple) else x for x in (a, b)]
    if case["op_b"] == "T":
        full[1] = full[1].T
    if not isinstance(c, tuple):
        return {"c": np.ascontiguousarray((c + full[0] @ full[1]).T).reshape(-1)}
    # the stacked factors of the sum, narrow where an operand is compressed
    if isinstance(a, tuple):
        left, right = a[0], a[1] @ full[1]
    else:
        left, right = full[0] @ b[0], b[1]
    u, v = _truncate(np.hstack([c[0], left]), np.vstack([c[1], right]), case["acc"], case["cap"], case["fixed"])
    return {"c": np.ascontiguousarray((u @ v).T), "rank": None}


def _recompress_flops(m, n, k_stack, r):
    """Two QRs of the stacked factors, the core product and its SVD, the new factors."""
    kk = min(k_stack, m, n)
    return (2.0 * (m + n) * k_stack * kk + 24.0 * kk ** 3 + 2.0 * (m + n) * kk * r)


def _new_rank(case, k_stack):
    if case.get("fixed"):
        return min(case["fixed"], k_stack)
    return min(case["cap"], k_stack, max(1, int(math.log(case["acc"]) / math.log(case["decay"]))))


def _work_gemm(case):
    m, n, k, (fa, fb, fc) = case["m"], case["n"], case["k"], case["combo"]
    size = 8 if case["dtype"] == "f64" else 4
    ra, rb, rc = case["ra"], case["rb"], case["rc"]
    elems = (m * k if fa == "D" else (m + k) * ra) + (k * n if fb == "D" else (k + n) * rb)
    if fa == "C" and fb == "C":
        prod, stacked = 2.0 * ra * k * rb + 2.0 * ra * rb * n, ra
    elif fa == "C":
        prod, stacked = 2.0 * ra * k * n, ra
    elif fb == "C":
        prod, stacked = 2.0 * m * k * rb, rb
    else:
        prod, stacked = 0.0, k
    if fc == "D":
        return {"bytes": size * (elems + 2 * m * n), "flops": prod + 2.0 * m * n * stacked}
    r = _new_rank(case, stacked + rc)
    flops = prod + _recompress_flops(m, n, stacked + rc, r) + 2.0 * m * n * r
    return {"bytes": size * (elems + (m + n) * (rc + r) + m * n), "flops": flops}


# ---------------------------------------------------------------------------
# Compression of a dense tile in host memory
# ---------------------------------------------------------------------------
def _compress_input(case, seed):
    m, n = case["m"], case["n"]
    # an off-diagonal block: the first m and the last n of 2 (m + n) points along the curve
    pts = covariance_points(2 * (m + n), 3, seed)
    return covariance_matrix(pts, 0.2, 0.0, slice(0, m), slice(2 * (m + n) - n, 2 * (m + n)))


def _prepare_compress(case, seed):
    st = _State()
    st.kind, st.a, st.cap = "compress", _compress_input(case, seed), case["cap"]
    st.params = H.CompressionParameters(case["acc"])
    st.out = torch.empty(case["n"], case["m"], dtype=torch.float64, device="cuda")
    return st


def _run_compress(st):
    t = H.CompressedTile.compress(_ctx(), st.a, st.params, max_rank=st.cap)
    u = _Dense(t.rows, t.rank, t.buf)
    v = _Dense(t.rank, t.cols, H.BufferView(t.buf, 8 * t.rows * t.max_rank, 8 * t.cols * t.max_rank))
    H.HCore.gemm(1.0, u, v, 0.0, _Dense(t.rows, t.cols, st.out), _ctx())
    return {"c": st.out, "rank": t.rank}


def _exact_compress(case, seed):
    a = _compress_input(case, seed)
    u, s, vt = np.linalg.svd(a, full_matrices=False)
    below = np.nonzero(s[1:] < case["acc"])[0]
    r = min(max(int(below[0]) + 1 if len(below) else len(s), 1), case["cap"])
    return {"c": np.ascontiguousarray(((u[:, :r] * s[:r]) @ vt[:r]).T), "rank": None}


def _work_compress(case):
    m, n = case["m"], case["n"]
    r, k = case["cap"], min(case["m"], case["n"])
    return {"bytes": 8 * (2 * m * n + (m + n) * r), "flops": 4.0 * m * n * k + 22.0 * k ** 3 + 4.0 * m * n * r}


# ---------------------------------------------------------------------------
# Batches
# ---------------------------------------------------------------------------
def _batch_shapes(case, seed):
    """(m, n, k, ra, rb, rc) of each update; ranks log-uniform in [lo, hi]."""
    rng = np.random.default_rng([seed, 1])
    nb, count = case["nb"], case["count"]
    sizes = np.full((count, 3), nb)
    if case["ragged"]:
        sizes = rng.choice([nb, nb - nb // 7, nb - nb // 3], size=(count, 3))
    ranks = np.rint(np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]), size=(count, 3)))).astype(np.int64)
    return np.hstack([sizes, ranks]).tolist()


def _batch_factors(case, seed, device):
    """Factors of every update, in turn: A, B and C as (U, V)."""
    bases = _Bases([seed, 2], device)
    for m, n, k, ra, rb, rc in _batch_shapes(case, seed):
        yield (bases.factors(m, k, ra, case["decay"]), bases.factors(k, n, rb, case["decay"]),
               bases.factors(m, n, rc, case["decay"]))


def _prepare_batch(case, seed):
    st = _State()
    shapes = _batch_shapes(case, seed)
    cap, count = case["cap"], case["count"]
    st.kind, st.mm, st.nn = "batch", max(s[0] for s in shapes), max(s[1] for s in shapes)
    # C tiles in one buffer, one after another, so that one copy restores them all; a tile of the
    # largest size has the whole stride
    stride = (st.mm + st.nn) * cap
    st.c = torch.zeros(count * stride, dtype=torch.float64, device="cuda")
    need = sum((m + k) * ra + (k + n) * rb for m, n, k, ra, rb, _ in shapes)
    st.ab = torch.zeros(need, dtype=torch.float64, device="cuda")
    at, As, Bs, Cs = 0, [], [], []
    for i, ((m, n, k, ra, rb, rc), (fa, fb, fc)) in enumerate(zip(shapes, _batch_factors(case, seed, "cuda"))):
        for (u, v), rows, cols, r, to in ((fa, m, k, ra, As), (fb, k, n, rb, Bs)):
            flat = st.ab[at: at + (rows + cols) * r]
            at += flat.numel()
            _put(flat, u, v, r)
            to.append(_Compressed(rows, cols, r, r, flat))
        flat = st.c[i * stride: (i + 1) * stride]
        _put(flat, *fc, cap)
        Cs.append(_Compressed(m, n, rc, cap, flat))
    st.c0, st.ranks0 = st.c.clone(), np.array([s[5] for s in shapes], dtype=np.int64)
    form = case["form"]
    st.graph = form == "rule_graph"
    precision = H.PREC_MIXED if form == "mixed_rule" else H.PREC_FP64
    torch.cuda.synchronize()
    st.batch = H.Batch(_ctx(), As, Bs, Cs, 1.0, 1.0, H.CompressionParameters(case["acc"]), precision)
    if form != "exact":
        st.batch.set_rank_model(None, tol=0.1, margin=0)
    if st.graph:
        st.batch.capture()
    # where each tile's factors start, for the dense result
    dev = lambda x: torch.tensor(x, dtype=torch.int64, device="cuda").view(-1, 1, 1)  # noqa: E731
    st.m, st.n = dev([s[0] for s in shapes]), dev([s[1] for s in shapes])
    st.base = dev([i * stride for i in range(count)])
    st.vbase = dev([i * stride + s[0] * cap for i, s in enumerate(shapes)])
    st.uniform = not case["ragged"]
    st.cap, st.stride, st.count = cap, stride, count
    st.out = torch.empty(count, st.nn, st.mm, dtype=torch.float64, device="cuda")
    return st


def _run_batch(st):
    _copy(st.c, st.c0)
    st.batch.set_ranks(st.ranks0)
    if st.graph:
        st.batch.launch_graph()
    else:
        st.batch.run()
    ranks = st.batch.ranks()
    # the dense tiles (column-major, in the corner of an nn x mm slot): V^T U^T over the largest rank
    r = int(ranks.max())
    rk = torch.from_numpy(ranks).cuda().view(-1, 1, 1)
    col = torch.arange(r, device="cuda").view(1, 1, -1)
    row = torch.arange(st.nn, device="cuda").view(1, -1, 1)
    keep = (col < rk) if st.uniform else (col < rk) & (row < st.n)
    v = st.c[torch.where(keep, row * rk + (col + st.vbase), 0)] * keep
    if st.uniform:
        u = st.c.view(st.count, st.stride)[:, : r * st.mm].view(st.count, r, st.mm)
    else:
        i = torch.arange(st.mm, device="cuda").view(1, 1, -1)
        col = col.view(1, -1, 1)
        keep = (col < rk) & (i < st.m)
        u = st.c[torch.where(keep, col * st.m + (i + st.base), 0)] * keep
    torch.bmm(v, u, out=st.out)
    return {"c": st.out, "ranks": ranks}


def _exact_batch(case, seed):
    if case["count"] * case["nb"] ** 2 > 256 * 512 ** 2:
        return None  # minutes of SVDs
    shapes = _batch_shapes(case, seed)
    mm, nn = max(s[0] for s in shapes), max(s[1] for s in shapes)
    out = np.zeros((len(shapes), nn, mm))

    def one(job):
        i, (fa, fb, fc) = job
        (au, av), (bu, bv), (cu, cv) = (_host(f) for f in (fa, fb, fc))
        u, v = _truncate(np.hstack([cu, au]), np.vstack([cv, (av @ bu) @ bv]), case["acc"], case["cap"])
        out[i, : v.shape[1], : u.shape[0]] = (u @ v).T

    for job in enumerate(_batch_factors(case, seed, "cpu")):
        one(job)
    return {"c": out, "ranks": None}


def _work_batch(case):
    # expectations over log-uniform ranks, with the mean rank in place of each
    nb, count = case["nb"] * (0.84 if case["ragged"] else 1.0), case["count"]
    mean = (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
    r = _new_rank(case, 2 * mean)
    flops = 4.0 * mean * mean * nb + _recompress_flops(nb, nb, 2 * mean, r) + 2.0 * nb * nb * r
    return {"bytes": count * 8 * (2 * nb * (3 * mean + r) + nb * nb), "flops": count * flops}


# ---------------------------------------------------------------------------
# Cholesky-flow tile operations: potrf of the diagonal tile, then per tile of its column a solve,
# the diagonal update and, for each pair, the compressed update (V stored cols x rank).
# ---------------------------------------------------------------------------
def _chol_step_inputs(case, seed):
    nb, r, t = case["nb"], case["rank"], case["tiles"]
    bases = _Bases([seed, 3], "cpu")
    diag = _covariance(nb, seed) + np.eye(nb)
    panel = [tuple(x.numpy() for x in bases.factors(nb, nb, r, 0.8)) for _ in range(t)]
    diags = [_covariance(nb, seed + 1 + i) + 2.0 * np.eye(nb) for i in range(t)]
    pairs = [(i, j) for i in range(t) for j in range(i)]
    trail = [tuple(x.numpy() for x in bases.factors(nb, nb, r, 0.8)) for _ in pairs]
    return diag, panel, diags, pairs, trail


def _prepare_chol_step(case, seed):
    st = _State()
    nb, cap = case["nb"], case["cap"]
    diag, panel, diags, st.pairs, trail = _chol_step_inputs(case, seed)
    st.kind, st.nb, st.rank = "chol_step", nb, case["rank"]

    def flat(u, v):
        t = np.zeros(2 * nb * cap)
        t[: u.size] = u.reshape(-1, order="F")
        t[nb * cap: nb * cap + v.size] = v.T.reshape(-1, order="F")  # V as cols x rank
        return t

    parts = [diag.reshape(-1)] + [d.reshape(-1) for d in diags] + [flat(*x) for x in panel] + [flat(*x) for x in trail]
    st.buf = torch.from_numpy(np.concatenate(parts)).cuda()
    st.buf0 = st.buf.clone()
    at = np.cumsum([0] + [len(x) for x in parts])
    views = [st.buf[a:b] for a, b in zip(at, at[1:])]
    t = case["tiles"]
    st.dense = [_Dense(nb, nb, v) for v in views[: t + 1]]
    st.panel = [_Compressed(nb, nb, st.rank, cap, v) for v in views[t + 1: 2 * t + 1]]
    st.trail = [_Compressed(nb, nb, st.rank, cap, v) for v in views[2 * t + 1:]]
    st.params = H.CompressionParameters(case["acc"])
    st.out = torch.empty(len(st.pairs), nb, nb, dtype=torch.float64, device="cuda")
    return st


def _run_chol_step(st):
    ctx = _ctx()
    _copy(st.buf, st.buf0)
    for t in st.trail:
        t.rank = st.rank
    H.HCore.potrf(st.dense[0], "L", ctx)
    for t in st.panel:
        H.HCore.trsm("L", "L", "N", "N", 1.0, st.dense[0], t, ctx)
    for t, d in zip(st.panel, st.dense[1:]):
        H.HCore.syrk(-1.0, t, "N", "L", 1.0, d, ctx)
    for (i, j), c, o in zip(st.pairs, st.trail, st.out):
        H.HCore.gemm(-1.0, st.panel[i], st.panel[j], 1.0, c, ctx, st.params, opB="T", cholesky=True)
        _product(c, o.view(-1), v_cols=True)
    nb = st.nb
    solved = [t.buf[nb * t.max_rank: nb * (t.max_rank + t.rank)] for t in st.panel]
    return {"dense": [d.buf for d in st.dense], "solved": solved, "trail": st.out,
            "ranks": np.array([t.rank for t in st.trail])}


def _exact_chol_step(case, seed):
    diag, panel, diags, pairs, trail = _chol_step_inputs(case, seed)
    low = np.linalg.cholesky(diag)
    # the factored tile keeps its other triangle
    dense = [np.tril(low) + np.triu(diag, 1)]
    solved = [np.linalg.solve(low, v.T) for _, v in panel]
    for (u, _), s, d in zip(panel, solved, diags):
        dense.append(np.tril(d - u @ (s.T @ s) @ u.T))
    out = []
    for (i, j), (cu, cv) in zip(pairs, trail):
        w = (solved[i].T @ solved[j]) @ panel[j][0].T
        u, v = _truncate(np.hstack([cu, -panel[i][0]]), np.vstack([cv, w]), case["acc"], case["cap"])
        out.append((u @ v).T)
    return {"dense": [np.ascontiguousarray(d.T).reshape(-1) for d in dense],
            "solved": [np.ascontiguousarray(s.T).reshape(-1) for s in solved],
            "trail": np.ascontiguousarray(np.stack(out)), "ranks": None}


def _work_chol_step(case):
    nb, r, t = case["nb"], case["rank"], case["tiles"]
    pairs = t * (t - 1) // 2
    new = min(case["cap"], 2 * r)
    flops = nb ** 3 / 3.0 + t * (nb * nb * r + 2.0 * nb * r * r + nb * nb * r)
    flops += pairs * (4.0 * nb * r * r + _recompress_flops(nb, nb, 2 * r, new) + 2.0 * nb * nb * new)
    words = 2 * nb * nb * (t + 1) + t * 3 * nb * r + pairs * (2 * nb * (r + new) + nb * nb)
    return {"bytes": 8 * words, "flops": flops}


# ---------------------------------------------------------------------------
# TLR Cholesky
# ---------------------------------------------------------------------------
def _matrix(case, seed):
    M = TLRMatrix(case["tiles"] * case["nb"], case["nb"], 3, 0.1, case["acc"], seed, nugget=1e-2)
    prefetch_tiles(M, [(i, j) for i in range(M.T) for j in range(i + 1)], 8)
    return M


def _prepare_cholesky(case, seed):
    st = _State()
    st.kind, st.nb = "cholesky", case["nb"]
    st.chol = TLRCholesky(_ctx(), _matrix(case, seed))
    st.saved = []
    for t in st.chol.D + list(st.chol.L.values()):
        words = t.ld * t.cols if t.type == H.DENSE else (t.rows + t.cols) * t.max_rank
        host = t.buf.download(np.float64, words)
        t.buf = torch.from_numpy(host).cuda()
        st.saved.append((t, t.buf.clone(), t.rank))
    st.params = H.CompressionParameters(case["acc"])
    n = case["tiles"] * case["nb"]
    st.out = torch.zeros(n, n, dtype=torch.float64, device="cuda")
    return st


def _run_cholesky(st):
    for t, saved, rank in st.saved:
        _copy(t.buf, saved)
        t.rank = rank
    st.chol.factor_batched(st.params)
    # the dense factor, column-major: column block j holds the tiles (i, j)
    nb, n = st.nb, st.out.shape[0]
    for k, d in enumerate(st.chol.D):
        st.out[k * nb: (k + 1) * nb, k * nb: (k + 1) * nb].copy_(d.buf.view(nb, nb))
    for (i, j), t in st.chol.L.items():
        _product(t, st.out.view(-1)[j * nb * n + i * nb:], ld=n)
    return {"factor": st.out, "ranks": np.array([t.rank for t in st.chol.L.values()])}


def _exact_cholesky(case, seed):
    M = _matrix(case, seed)
    T, nb, acc = M.T, M.nb, case["acc"]
    D = [M.tile(k, k)[1].copy() for k in range(T)]
    L = {(i, k): M.tile(i, k)[1:] for i in range(T) for k in range(i)}
    for k in range(T):
        D[k] = np.linalg.cholesky(D[k])
        for i in range(k + 1, T):
            u, v, cap = L[(i, k)]
            v = np.linalg.solve(D[k], v.T).T
            L[(i, k)] = (u, v, cap)
            D[i] = D[i] - u @ (v @ v.T) @ u.T
        for j in range(k + 1, T):
            for i in range(j + 1, T):
                (ui, vi, _), (uj, vj, _), (u, v, cap) = L[(i, k)], L[(j, k)], L[(i, j)]
                L[(i, j)] = (*_truncate(np.hstack([u, -ui]), np.vstack([v, (vi @ vj.T) @ uj.T]), acc, cap), cap)
    full = np.zeros((T * nb, T * nb))
    for k in range(T):
        full[k * nb: (k + 1) * nb, k * nb: (k + 1) * nb] = np.tril(D[k])
    for (i, j), (u, v, _) in L.items():
        full[i * nb: (i + 1) * nb, j * nb: (j + 1) * nb] = u @ v
    return {"factor": np.ascontiguousarray(full.T), "ranks": None}


def _work_cholesky(case):
    T, nb = case["tiles"], case["nb"]
    r = max(nb // 3, 1)
    pairs, updates = T * (T - 1) // 2, T * (T - 1) * (T - 2) // 6
    flops = T * nb ** 3 / 3.0 + pairs * (2.0 * nb * nb * r + 4.0 * nb * r * r + 2.0 * nb * nb * r)
    flops += updates * (4.0 * nb * r * r + _recompress_flops(nb, nb, 2 * r, r))
    words = 2 * T * nb * nb + 4 * pairs * nb * r + (T * nb) ** 2 // 2
    return {"bytes": 8 * words, "flops": flops}


_KINDS = {
    "gemm": (_prepare_gemm, _run_gemm, _exact_gemm, _work_gemm),
    "compress": (_prepare_compress, _run_compress, _exact_compress, _work_compress),
    "batch": (_prepare_batch, _run_batch, _exact_batch, _work_batch),
    "chol_step": (_prepare_chol_step, _run_chol_step, _exact_chol_step, _work_chol_step),
    "cholesky": (_prepare_cholesky, _run_cholesky, _exact_cholesky, _work_cholesky),
}


def prepare(case, seed):
    st = _KINDS[case["kind"]][0](case, seed)
    torch.cuda.synchronize()
    return st


def run(state):
    return _KINDS[state.kind][1](state)


def exact(case, seed):
    return _KINDS[case["kind"]][2](case, seed)


def work(case):
    return _KINDS[case["kind"]][3](case)
