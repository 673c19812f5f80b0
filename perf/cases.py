"""The work that a user has this library do, as cases to be timed.

listed() names twelve, draw() gives more of the same ranges, prepare() makes a
case's inputs on the GPU from a seed, run() is one pass through the public
entry points, exact() the same outputs in 64 bits from plain torch, and work()
the bytes and operations that no implementation can do without.

A case's "kind" says which entry point it calls:

  dense   sketch_general with a DenseSkOp, generated inside the product; as a
          left sketch B = op(S) op(A) or a right one B = op(A) op(S), over a
          submatrix of the operator where "ro" / "co" are not zero
  vector  sketch_vector with a DenseSkOp
  grad    autograd.left_sketch: B = S A and dA = S^T dB
  bf16    lskge3_bf16split with three terms
  fill    fill_dense
  saso    sketch_general with a SparseSkOp (short-axis vectors), sampled
          beforehand ("filled") or by the call itself
  sparse  rsksp3 on CSR data and the gradient of its values
  solve   sketch_solve and sketch_solve_adjoint
  sample  weights_to_cdf and sample_indices_iid

Sizes: S is d x m before op() for left sketches (A is m x n) and n x d for
right ones (A is m x n).
"""
import math

import torch

import randblas_amd as rb
from randblas_amd.autograd import left_sketch

DEV = "cuda"


def listed():
    return [
        # a small sketch: the call's latency and its launches
        {"name": "dense_small_f64", "kind": "dense", "side": "left", "dtype": "f64", "layout": "C", "opS": "N",
         "opA": "N", "d": 400, "n": 200, "m": 2000, "family": "G", "axis": "L", "ro": 0, "co": 0},
        # total least squares: [A b] with an odd number of rows and columns, d = 2 n
        {"name": "dense_tls_f64", "kind": "dense", "side": "left", "dtype": "f64", "layout": "C", "opS": "N",
         "opA": "N", "d": 1002, "n": 501, "m": 10001, "family": "G", "axis": "L", "ro": 0, "co": 0},
        # the range finder of a randomized SVD: A times a thin test matrix
        {"name": "dense_rangefinder_f32", "kind": "dense", "side": "right", "dtype": "f32", "layout": "C", "opS": "N",
         "opA": "N", "d": 110, "n": 2000, "m": 100000, "family": "G", "axis": "L", "ro": 0, "co": 0},
        # a large double-precision sketch
        {"name": "dense_large_f64", "kind": "dense", "side": "left", "dtype": "f64", "layout": "C", "opS": "N",
         "opA": "N", "d": 2048, "n": 1000, "m": 131072, "family": "G", "axis": "L", "ro": 0, "co": 0},
        # a sketching layer in training, forward and backward, torch's row-major layout, odd sizes
        {"name": "grad_ragged_f32", "kind": "grad", "dtype": "f32", "d": 777, "n": 301, "m": 50001, "family": "G",
         "axis": "L"},
        # the largest: the BF16-split sketch of an ill-conditioned tall matrix
        {"name": "bf16_headline", "kind": "bf16", "d": 4096, "n": 1024, "m": 262144},
        # an operator materialised for reuse
        {"name": "fill_dense_f32", "kind": "fill", "dtype": "f32", "rows": 4096, "cols": 65536, "family": "G",
         "axis": "L"},
        # a sparse operator, sampled once, on column-major data
        {"name": "saso_colmajor_f64", "kind": "saso", "side": "left", "dtype": "f64", "layout": "C", "opA": "N",
         "d": 2000, "n": 500, "m": 100000, "vec_nnz": 8, "filled": True},
        # the same use on row-major data of odd sizes
        {"name": "saso_rowmajor_f32", "kind": "saso", "side": "left", "dtype": "f32", "layout": "R", "opA": "N",
         "d": 1500, "n": 333, "m": 100003, "vec_nnz": 8, "filled": True},
        # sparse data with power-law columns: the sketch and the gradient of the stored values
        {"name": "sparse_powerlaw_f32", "kind": "sparse", "dtype": "f32", "m": 200000, "n": 50000, "d": 256,
         "per_row": 20},
        # differentiable sketch-and-solve least squares
        {"name": "solve_f64", "kind": "solve", "dtype": "f64", "d": 1024, "m": 65536, "n": 256},
        # weighted row sampling: weights to a distribution, then draws from it
        {"name": "sample_cdf_f64", "kind": "sample", "dtype": "f64", "n": 1000000, "k": 1 << 24},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: sizes spread over their logarithm, options as in use."""
    kind = rng.choices(["dense", "vector", "grad", "bf16", "fill", "saso", "sparse", "solve", "sample"],
                       [10, 2, 3, 2, 1, 4, 2, 1, 1])[0]
    dtype = rng.choice(["f32", "f64"])
    family, axis = rng.choice("GGGGU"), rng.choice("LLLLS")
    if kind == "dense":
        while True:
            d, n, m = _log(rng, 16, 4096), _log(rng, 2, 2048), _log(rng, 256, 300000)
            side = rng.choice(["left", "left", "right"])
            c = {"kind": kind, "side": side, "dtype": dtype, "layout": rng.choice("CR"), "opS": rng.choice("NNNT"),
                 "opA": rng.choice("NNNT"), "d": d, "n": n, "m": m, "family": family, "axis": axis,
                 "ro": rng.choice([0, 0, rng.randint(1, 64)]), "co": rng.choice([0, 0, rng.randint(1, 64)])}
            if side == "right":  # A is m x n, reduced to m x d
                c["n"], c["d"] = _log(rng, 64, 8192), min(d, 1024)
            if c["d"] <= (m if side == "left" else c["n"]) and 2.0 * c["d"] * c["n"] * m <= 2e11 and c["n"] * m <= 1 << 28:
                return c
    if kind == "vector":
        return {"kind": kind, "dtype": dtype, "opS": rng.choice("NNT"), "d": _log(rng, 16, 4096),
                "m": _log(rng, 1000, 300000), "family": family, "axis": axis}
    if kind == "grad":
        while True:
            c = {"kind": kind, "dtype": dtype, "d": _log(rng, 16, 2048), "n": _log(rng, 1, 1024),
                 "m": _log(rng, 1000, 300000), "family": family, "axis": axis}
            if c["d"] <= c["m"] and 4.0 * c["d"] * c["n"] * c["m"] <= 1e11:
                return c
    if kind == "bf16":
        while True:
            c = {"kind": kind, "d": _log(rng, 64, 4096), "n": _log(rng, 32, 1024), "m": _log(rng, 4096, 262144)}
            if c["d"] <= c["m"] and 2.0 * c["d"] * c["n"] * c["m"] <= 5e11:
                return c
    if kind == "fill":
        return {"kind": kind, "dtype": dtype, "rows": _log(rng, 16, 4096), "cols": _log(rng, 100, 65536),
                "family": family, "axis": axis}
    if kind == "saso":
        while True:
            side = rng.choice(["left", "left", "right"])
            c = {"kind": kind, "side": side, "dtype": dtype, "layout": rng.choice("CR"), "opA": rng.choice("NNT"),
                 "d": _log(rng, 50, 8000), "n": _log(rng, 4, 1000), "m": _log(rng, 1000, 300000),
                 "vec_nnz": rng.choice([1, 2, 4, 8, 8, 16]), "filled": rng.choice([True, True, False])}
            if side == "right":
                c["n"], c["m"] = c["m"], c["n"]
            big = max(c["m"], c["n"])
            if c["d"] <= big and c["m"] * c["n"] <= 1 << 27 and c["d"] * big <= 1 << 30:
                return c
    if kind == "sparse":
        return {"kind": kind, "dtype": dtype, "m": _log(rng, 2000, 200000), "n": _log(rng, 1000, 50000),
                "d": _log(rng, 16, 512), "per_row": rng.choice([4, 10, 20])}
    if kind == "solve":
        n = _log(rng, 10, 256)
        return {"kind": kind, "dtype": dtype, "d": 4 * n, "m": _log(rng, 8 * n, 65536), "n": n}
    return {"kind": kind, "dtype": "f64", "n": _log(rng, 1000, 1000000), "k": _log(rng, 1000, 1 << 24)}


# ------------------------------------------------------------------ inputs
def _dt(case):
    return torch.float32 if case.get("dtype", "f32") == "f32" else torch.float64


def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFF)


def _normal(seed, salt, count, dtype):
    return torch.randn(count, dtype=dtype, device=DEV, generator=_gen(seed, salt))


def _dims(case):
    """(rows, cols) of the operator that the case's sketch reads a window of,
    the window's (rows, cols), A's and B's stored (rows, cols)."""
    d, n, m = case["d"], case["n"], case["m"]
    win = (d, m) if case["side"] == "left" else (n, d)
    if case.get("opS", "N") == "T":
        win = win[::-1]
    full = (win[0] + case.get("ro", 0), win[1] + case.get("co", 0))
    a = (m, n) if case["opA"] == "N" else (n, m)
    b = (d, n) if case["side"] == "left" else (m, d)
    return full, win, a, b


def _dense_inputs(case, seed):
    _, _, a, _ = _dims(case)
    return _normal(seed, 1, a[0] * a[1], _dt(case))


def _dense_op(case, seed, rows, cols):
    dist = rb.DenseDist(rows, cols, rb.ScalarDist(case.get("family", "G")), rb.Axis(case.get("axis", "L")))
    return rb.DenseSkOp(dist, rb.RNGState(int(seed)), dtype=_dt(case))


def _csr(case, seed):
    """Power-law CSR data: Zipf columns, uniform rows, repeated pairs once."""
    m, n = case["m"], case["n"]
    k = m * case["per_row"]
    w = torch.arange(1, n + 1, dtype=torch.float64, device=DEV) ** (-1.0 / 1.1)
    cdf = torch.cumsum(w, 0)
    u = torch.rand(k, dtype=torch.float64, device=DEV, generator=_gen(seed, 1))
    col = torch.searchsorted(cdf, u * cdf[-1]).clamp_(max=n - 1)
    row = torch.randint(0, m, (k,), device=DEV, generator=_gen(seed, 2))
    pairs = torch.unique(row * n + col)
    row, col = pairs // n, pairs % n
    ptr = torch.zeros(m + 1, dtype=torch.int64, device=DEV)
    ptr[1:] = torch.cumsum(torch.bincount(row, minlength=m), 0)
    return row, col, ptr, _normal(seed, 3, pairs.numel(), _dt(case))


def _solve_inputs(case, seed):
    m, n, dt = case["m"], case["n"], _dt(case)
    A = _normal(seed, 1, m * n, dt)
    x = _normal(seed, 2, n, dt)
    b = torch.mv(A.view(n, m).t(), x) + 1e-3 * _normal(seed, 3, m, dt)
    return A, b, _normal(seed, 4, n, dt)


def _bf16_inputs(case, seed):
    """A column-major with column scales that fall to 1e-6 of the first."""
    m, n = case["m"], case["n"]
    A = _normal(seed, 1, m * n, torch.float32)
    A.view(n, m).mul_((10.0 ** (-6.0 * torch.arange(n, device=DEV, dtype=torch.float64) / max(n - 1, 1))).float()[:, None])
    return A


def prepare(case, seed):
    kind, dt = case["kind"], _dt(case)
    s = {"case": case}

    def empty(*shape, dtype=dt):
        return torch.empty(*shape, dtype=dtype, device=DEV)

    if kind == "dense":
        full, _, _, b = _dims(case)
        s.update(A=_dense_inputs(case, seed), S=_dense_op(case, seed, *full), B=empty(b[0] * b[1]))
    elif kind == "vector":
        d, m = case["d"], case["m"]
        inner, outer = (m, d) if case["opS"] == "N" else (d, m)
        s.update(x=_normal(seed, 1, inner, dt), S=_dense_op(case, seed, d, m), y=empty(outer))
    elif kind == "grad":
        d, n, m = case["d"], case["n"], case["m"]
        s.update(A=_normal(seed, 1, m * n, dt).view(m, n).requires_grad_(), G=_normal(seed, 2, d * n, dt).view(d, n),
                 S=_dense_op(case, seed, d, m))
    elif kind == "bf16":
        s.update(A=_bf16_inputs(case, seed), S=_dense_op(case, seed, case["d"], case["m"]),
                 B=empty(case["d"] * case["n"]))
    elif kind == "fill":
        dist = rb.DenseDist(case["rows"], case["cols"], rb.ScalarDist(case["family"]), rb.Axis(case["axis"]))
        s.update(D=dist, state=rb.RNGState(int(seed)), buff=empty(case["rows"] * case["cols"]))
    elif kind == "saso":
        full, _, _, b = _dims(case)
        S = rb.SparseSkOp(rb.SparseDist(*full, case["vec_nnz"], rb.Axis.Short), rb.RNGState(int(seed)), dtype=dt)
        if case["filled"]:
            rb.fill_sparse(S)
        s.update(A=_dense_inputs(case, seed), S=S, B=empty(b[0] * b[1]))
    elif kind == "sparse":
        m, n, d = case["m"], case["n"], case["d"]
        _, col, ptr, vals = _csr(case, seed)
        s.update(A=rb.CSRMatrix(m, n, vals, ptr, col), S=_dense_op(case, seed, n, d), B=empty(m * d),
                 G=_normal(seed, 4, m * d, dt), dvals=torch.zeros(m * case["per_row"], dtype=dt, device=DEV))
    elif kind == "solve":
        d, m, n = case["d"], case["m"], case["n"]
        A, b, xbar = _solve_inputs(case, seed)
        s.update(A=A, b=b, xbar=xbar, S=_dense_op(case, seed, d, m), x=empty(n), Abar=empty(m * n), bbar=empty(m))
    else:
        w = _normal(seed, 1, case["n"], dt).square_()
        s.update(w=w, cdf=empty(case["n"]), state=rb.RNGState(int(seed)), idx=empty(case["k"], dtype=torch.int64))
    return s


# ------------------------------------------------------------------ one pass
def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind in ("dense", "saso"):
        lay, opS, opA, d, n, m = c["layout"], c.get("opS", "N"), c["opA"], c["d"], c["n"], c["m"]
        _, _, a, b = _dims(c)
        lda, ldb = (a[0], b[0]) if lay == "C" else (a[1], b[1])
        ro, co = c.get("ro", 0), c.get("co", 0)
        if c["side"] == "left":
            rb.sketch_general(lay, opS, opA, d, n, m, 1.0, s["S"], ro, co, s["A"], lda, 0.0, s["B"], ldb)
        else:
            rb.sketch_general(lay, opA, opS, m, d, n, 1.0, s["A"], lda, s["S"], ro, co, 0.0, s["B"], ldb)
        return s["B"]
    if kind == "vector":
        rb.sketch_vector(c["opS"], 1.0, s["S"], s["x"], 1, 0.0, s["y"], 1)
        return s["y"]
    if kind == "grad":
        B = left_sketch(s["A"], s["S"])
        dA, = torch.autograd.grad(B, s["A"], s["G"])
        return {"B": B, "dA": dA}
    if kind == "bf16":
        d, n, m = c["d"], c["n"], c["m"]
        rb.lskge3_bf16split("C", "N", "N", d, n, m, 1.0, s["S"], 0, 0, s["A"], m, 0.0, s["B"], d)
        return s["B"]
    if kind == "fill":
        rb.fill_dense(s["D"], s["buff"], s["state"])
        return s["buff"]
    if kind == "sparse":
        m, n, d = c["m"], c["n"], c["d"]
        rb.rsksp3("R", "N", "N", m, d, n, 1.0, s["A"], 0, 0, s["S"], 0, 0, 0.0, s["B"], d)
        rb.rsksp3_adjoint("R", "N", m, d, n, 1.0, s["A"], s["S"], 0, 0, s["G"], d, s["dvals"])
        return {"B": s["B"], "dvals": s["dvals"]}
    if kind == "solve":
        d, m, n = c["d"], c["m"], c["n"]
        rb.sketch_solve("C", d, m, n, s["S"], 0, 0, s["A"], m, s["b"], s["x"])
        rb.sketch_solve_adjoint("C", d, m, n, s["S"], 0, 0, s["A"], m, s["b"], s["xbar"], s["Abar"], m, s["bbar"])
        return {"x": s["x"], "Abar": s["Abar"], "bbar": s["bbar"]}
    s["cdf"].copy_(s["w"])
    rb.weights_to_cdf(c["n"], s["cdf"])
    rb.sample_indices_iid(c["n"], s["cdf"], c["k"], s["idx"], s["state"])
    return {"cdf": s["cdf"], "idx": s["idx"]}


def work(case):
    kind = case["kind"]
    e = 4 if _dt(case) == torch.float32 else 8
    if kind in ("dense", "saso"):
        _, _, a, b = _dims(case)
        ab = e * (a[0] * a[1] + b[0] * b[1])
        if kind == "dense":
            return {"bytes": ab, "flops": 2.0 * case["d"] * case["n"] * case["m"]}
        big, small = (case["m"], case["n"]) if case["side"] == "left" else (case["n"], case["m"])
        long = max(big, case["d"])
        return {"bytes": ab, "flops": 2.0 * case["vec_nnz"] * long * small}
    if kind == "vector":
        return {"bytes": e * (case["d"] + case["m"]), "flops": 2.0 * case["d"] * case["m"]}
    if kind == "grad":
        d, n, m = case["d"], case["n"], case["m"]
        return {"bytes": e * 2 * n * (m + d), "flops": 4.0 * d * n * m}
    if kind == "bf16":
        d, n, m = case["d"], case["n"], case["m"]
        return {"bytes": 4 * n * (m + d), "flops": 2.0 * d * n * m}
    if kind == "fill":
        return {"bytes": e * case["rows"] * case["cols"], "flops": 0}
    if kind == "sparse":
        nnz = case["m"] * case["per_row"]
        return {"bytes": nnz * (2 * (8 + e) + e) + 16 * case["m"] + 2 * e * case["m"] * case["d"],
                "flops": 4.0 * nnz * case["d"]}
    if kind == "solve":  # the sketch of [A b] twice (once for each call) and the adjoint's product
        d, n, m = case["d"], case["n"], case["m"]
        return {"bytes": e * 3 * m * (n + 1), "flops": 6.0 * d * m * (n + 1)}
    return {"bytes": 2 * e * case["n"] + 8 * case["k"], "flops": 0}


# ------------------------------------------------------------------ in 64 bits
def _mulhilo(a, x):
    """High and low words of the 64-bit product of a constant and 32-bit words
    (int64 tensors; the wrapped product's bits are the unsigned product's)."""
    p = x * a
    return (p >> 32) & 0xFFFFFFFF, p & 0xFFFFFFFF


def _philox(lo, key):
    """Philox4x32-10 words of the 64-bit counters `lo` (high half zero)."""
    x = [lo & 0xFFFFFFFF, lo >> 32, torch.zeros_like(lo), torch.zeros_like(lo)]
    k0, k1 = int(key) & 0xFFFFFFFF, int(key) >> 32
    for _ in range(10):
        h0, l0 = _mulhilo(0xD2511F53, x[0])
        h1, l1 = _mulhilo(0xCD9E8D57, x[2])
        x = [h1 ^ x[1] ^ k0, l1, h0 ^ x[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return x


def _uneg11(w):
    signed = torch.where(w >= 1 << 31, w - (1 << 32), w)
    return signed.float() * 2.0 ** -31 + 2.0 ** -32


def _boxmuller(w0, w1):
    """The float32 pair whose factors are correctly rounded."""
    t = (_uneg11(w0) * torch.tensor(math.pi, dtype=torch.float32, device=DEV)).double()
    u = w1.float() * 2.0 ** -32 + 2.0 ** -33
    r = (-2.0 * torch.log(u.double()).float()).double().sqrt().float()
    return torch.sin(t).float() * r, torch.cos(t).float() * r


def _operator(case, seed, rows, cols):
    """The rows x cols dense operator in float64 (entries as the type holds them)."""
    lng = case.get("axis", "L") == "L"
    major = max(rows, cols) if lng else min(rows, cols)
    minor = rows + cols - major
    per = -(-major // 4)
    out = torch.empty(minor, major, dtype=torch.float64, device=DEV)
    step = max(1, (1 << 24) // per)
    for a in range(0, minor, step):
        b = min(minor, a + step)
        w = _philox(torch.arange(a * per, b * per, dtype=torch.int64, device=DEV), seed)
        if case.get("family", "G") == "G":
            e = [*_boxmuller(w[0], w[1]), *_boxmuller(w[2], w[3])]
        elif _dt(case) == torch.float32:
            e = [_uneg11(x) * torch.tensor(math.sqrt(3.0), dtype=torch.float32, device=DEV) for x in w]
        else:
            e = [_uneg11(x).double() * math.sqrt(3.0) for x in w]
        out[a:b] = torch.stack(e, -1).view(b - a, 4 * per)[:, :major]
    by_rows = (rows < cols) == lng  # the major axis runs along the rows of S
    return out if by_rows else out.t()


def _saso(case, seed, rows, cols):
    """The rows x cols short-axis operator as a dense float64 matrix: a partial
    Fisher-Yates shuffle and signs for each vector of the longer dimension."""
    short, long, k = min(rows, cols), max(rows, cols), case["vec_nnz"]
    S = torch.zeros(long, short, dtype=torch.float64, device=DEV)
    first = torch.arange(long, dtype=torch.int64, device=DEV) * k
    moved = []

    def at(x):
        v = x
        for pos, val in moved:
            v = torch.where(pos == x, val, v)
        return v

    for j in range(k):
        w = _philox(first + j, seed)
        ell = j + w[0] % (short - j)
        got, here = at(ell), at(torch.full_like(ell, j))
        moved.append((ell, here))
        S.scatter_(1, got[:, None], (1.0 - 2.0 * (w[1] % 2))[:, None].double())
    return S if rows > cols else S.t()


def _as_matrix(flat, rows, cols, layout):
    return flat.view(cols, rows).t() if layout == "C" else flat.view(rows, cols)


def _flat(M, layout):
    return (M.t() if layout == "C" else M).contiguous().view(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("dense", "saso"):
        full, win, a, _ = _dims(case)
        S = (_operator if kind == "dense" else _saso)(case, seed, *full)
        ro, co = case.get("ro", 0), case.get("co", 0)
        S = S[ro:ro + win[0], co:co + win[1]]
        S = S.t() if case.get("opS", "N") == "T" else S
        A = _as_matrix(_dense_inputs(case, seed).double(), *a, case["layout"])
        A = A.t() if case["opA"] == "T" else A
        return _flat(S @ A if case["side"] == "left" else A @ S, case["layout"])
    if kind == "vector":
        d, m = case["d"], case["m"]
        S = _operator(case, seed, d, m)
        x = _normal(seed, 1, m if case["opS"] == "N" else d, _dt(case)).double()
        return (S if case["opS"] == "N" else S.t()) @ x
    if kind == "grad":
        d, n, m = case["d"], case["n"], case["m"]
        S = _operator(case, seed, d, m)
        A = _normal(seed, 1, m * n, _dt(case)).double().view(m, n)
        return {"B": S @ A, "dA": S.t() @ _normal(seed, 2, d * n, _dt(case)).double().view(d, n)}
    if kind == "bf16":
        S = _operator(case, seed, case["d"], case["m"]).bfloat16().double()
        return _flat(S @ _as_matrix(_bf16_inputs(case, seed).double(), case["m"], case["n"], "C"), "C")
    if kind == "fill":
        rows, cols = case["rows"], case["cols"]
        S = _operator(case, seed, rows, cols)
        by_rows = (rows < cols) == (case["axis"] == "L")
        return _flat(S, "R" if by_rows else "C")
    if kind == "sparse":
        row, col, _, vals = _csr(case, seed)
        m, d = case["m"], case["d"]
        S, vals = _operator(case, seed, case["n"], d), vals.double()
        G = _normal(seed, 4, m * d, _dt(case)).double().view(m, d)
        B = torch.zeros(m, d, dtype=torch.float64, device=DEV)
        dvals = torch.zeros(m * case["per_row"], dtype=torch.float64, device=DEV)  # past the stored entries: zero
        for i in range(0, vals.numel(), 1 << 20):
            r, q = row[i:i + (1 << 20)], S[col[i:i + (1 << 20)]]
            B.index_add_(0, r, vals[i:i + (1 << 20), None] * q)
            dvals[i:i + r.numel()] = (G[r] * q).sum(1)
        return {"B": B.view(-1), "dvals": dvals}
    if kind == "solve":
        m, n = case["m"], case["n"]
        S = _operator(case, seed, case["d"], m)
        A, b, xbar = (t.double() for t in _solve_inputs(case, seed))
        M, c = S @ A.view(n, m).t(), S @ b
        Q, R = torch.linalg.qr(M)
        x = torch.linalg.solve_triangular(R, (Q.t() @ c)[:, None], upper=True)[:, 0]
        u = torch.linalg.solve_triangular(R.t(), xbar[:, None], upper=False)
        z, w = torch.linalg.solve_triangular(R, u, upper=True)[:, 0], (Q @ u)[:, 0]
        return {"x": x, "Abar": _flat(S.t() @ (torch.outer(c - M @ x, z) - torch.outer(w, x)), "C"), "bbar": S.t() @ w}
    w = _normal(seed, 1, case["n"], _dt(case)).square_().double()
    total = torch.cumsum(w, 0)
    return {"cdf": total / total[-1], "idx": None}
