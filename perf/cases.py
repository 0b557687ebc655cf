"""The GEMM calls this library's performance is measured on.

A case is one call of a front-end of `gemm_mmbo_amd` -- element type, transposes, sizes, batch, scalars, leading dimensions
-- with the automatic pick of the tile config, on operands that lie in device memory, as in bench.py and the report driver.
`listed()` holds the calls that stand for the library's range, `draw()` makes further ones of the same kinds.
"""
import math

import torch

import gemm_mmbo_amd as G

DTYPE = {"h": G.F16, "s": G.F32, "d": G.F64}
TORCH = {"h": torch.float16, "s": torch.float32, "d": torch.float64}
ESZ = {"h": 2, "s": 4, "d": 8}

# what one call may cost: the operations of the largest listed call of each type, and the bytes of the largest of all
MOST_FLOP = {"h": 2 * 8192 ** 3, "s": 2 * 4096 ** 3, "d": 2 * 44160 * 2048 * 384}
MOST_BYTES = 1.6e9


def _case(dtype, ta, tb, m, n, k, batch=1, alpha=1.0, beta=0.0, lda=0, ldb=0, ldc=0, workspace="own"):
    """Leading dimensions: 0 means packed.  workspace: "own" = gemm / gemm_strided_batched, "static" = the entry point that
    allocates nothing (tight loops, graph capture)."""
    return {"dtype": dtype, "ta": ta, "tb": tb, "m": m, "n": n, "k": k, "batch": batch, "alpha": alpha, "beta": beta,
            "lda": lda or (k if ta else m), "ldb": ldb or (n if tb else k), "ldc": ldc or m, "workspace": workspace}


def listed():
    return [
        # the headline product: large, square, fp16
        dict(_case("h", 0, 0, 8192, 8192, 8192), name="h_nn_8192"),
        # a large fp32 product with a transposed operand that updates C (alpha, beta both at work)
        dict(_case("s", 0, 1, 4096, 4096, 4096, alpha=1.5, beta=0.5), name="s_nt_4096_update"),
        # the small fp32 product of the first benchmark configuration
        dict(_case("s", 0, 0, 1024, 1024, 1024), name="s_nn_1024"),
        # one thin operand, long k: the irregular configuration
        dict(_case("h", 0, 0, 4096, 128, 4096), name="h_nn_4096x128x4096"),
        # odd in every direction: edge tiles, a partial last slice, rows off every alignment
        dict(_case("h", 0, 0, 1023, 777, 513), name="h_nn_1023x777x513"),
        # a batch of small products accumulated into C (per-head or per-element work)
        dict(_case("h", 1, 0, 512, 512, 512, batch=64, beta=1.0), name="h_tn_64x512_accumulate"),
        # the trailing update of an fp64 LU factorisation: its first step ...
        dict(_case("d", 0, 1, 44160, 2048, 384, alpha=-1.0, beta=1.0, ldc=44160), name="d_nt_44160_update"),
        # ... and one of its last (the same sweep goes down to 384 rows; C stays inside the large matrix)
        dict(_case("d", 0, 1, 1152, 2048, 384, alpha=-1.0, beta=1.0, ldc=44160), name="d_nt_1152_update"),
        # an ordinary fp16 product whose size is no power of two
        dict(_case("h", 0, 0, 3000, 3000, 3000), name="h_nn_3000"),
        # sixteen rows against a large matrix: a step of a serving loop, through the entry point that allocates nothing
        dict(_case("h", 0, 0, 16, 4096, 4096, workspace="static"), name="h_nn_16x4096x4096"),
        # a weight gradient: both operands summed over a long k, accumulated
        dict(_case("s", 1, 0, 640, 384, 10000, beta=1.0), name="s_tn_640x384x10000_accumulate"),
        # a handful of tiny products: the cost of a call
        dict(_case("s", 0, 0, 96, 72, 150, batch=5), name="s_nn_5x96x72x150"),
    ]


def _size(rng, low, high):
    """Spread over the logarithm; half of them as they fall, the others whole multiples of 8, 32 or 128."""
    v = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    if rng.random() < 0.5:
        step = rng.choice((8, 32, 128))
        v = max(1, round(v / step)) * step
    return min(max(v, low), high)


def draw(rng):
    kind = rng.choices(("square", "thin", "long_k", "batch", "update"), weights=(35, 20, 15, 15, 15))[0]
    dtype = rng.choices("hsd", weights=(50, 30, 20))[0]
    ta, tb, batch = rng.randint(0, 1), rng.randint(0, 1), 1
    alpha, beta = rng.choice(((1.0, 0.0), (1.0, 0.0), (1.0, 1.0), (1.5, 0.5), (-1.0, 1.0)))
    workspace = "static" if rng.random() < 0.15 else "own"
    ldc_rows = 0
    if kind == "square":            # all three dimensions of one order
        top = {"h": 8192, "s": 5120, "d": 3600}[dtype]
        s = math.exp(rng.uniform(math.log(48), math.log(top)))
        m, n, k = (_size(rng, max(16, int(s / 2)), max(17, min(top, int(s * 1.5)))) for _ in range(3))
    elif kind == "thin":            # few rows or few columns against a large matrix
        m, n, k = _size(rng, 1, 256), _size(rng, 512, 16384), _size(rng, 256, 16384)
        if rng.random() < 0.5:
            m, n = n, m
    elif kind == "long_k":          # small results of long sums
        m, n, k = _size(rng, 32, 1024), _size(rng, 32, 1024), _size(rng, 2048, 65536)
    elif kind == "batch":           # many small products in one call
        batch = _size(rng, 2, 256)
        m, n, k = (_size(rng, 16, 768) for _ in range(3))
    else:                           # a low-rank update of a large C
        m, n, k = _size(rng, 384, 44160), _size(rng, 256, 2048), _size(rng, 64, 512)
        ta, tb, alpha, beta = 0, 1, -1.0, 1.0
        ldc_rows = 44160 if rng.random() < 0.5 else 0
    # a call dearer than the largest listed one of its type: fewer rows (or problems), the largest dimension first
    while 2.0 * m * n * k * batch > MOST_FLOP[dtype] or (m * k + k * n + 2 * max(m, ldc_rows) * n) * batch * ESZ[dtype] > MOST_BYTES:
        if batch > 1:
            batch = batch // 2
        elif max(m, ldc_rows) >= max(n, k):
            m, ldc_rows = max(1, m // 2), 0
        elif n >= k:
            n = max(1, n // 2)
        else:
            k = max(1, k // 2)
    pad = rng.choice((0, 0, 0, 0, 1, 8, 64))          # operands inside larger matrices
    return _case(dtype, ta, tb, m, n, k, batch, alpha, beta, (k if ta else m) + pad, (n if tb else k) + pad,
                 max(ldc_rows, m + pad), workspace)


def _strides(c):
    return c["lda"] * (c["m"] if c["ta"] else c["k"]), c["ldb"] * (c["k"] if c["tb"] else c["n"]), c["ldc"] * c["n"]


def prepare(case, seed):
    """A, B and C of one call in device memory.  fp16: N(0, 1) * 0.1, C uniform [-1, 1]; fp32 and fp64: uniform [-1, 1]."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    d, batch, (sa, sb, sc) = case["dtype"], case["batch"], _strides(case)

    def uniform(count):
        t = torch.float32 if d == "h" else TORCH[d]
        return torch.rand(count, generator=g, device="cuda", dtype=t).mul_(2).sub_(1).to(TORCH[d])

    def operand(count):
        if d == "h":
            return torch.randn(count, generator=g, device="cuda", dtype=torch.float32).mul_(0.1).to(torch.float16)
        return uniform(count)

    A, B = operand(sa * batch), operand(sb * batch)
    C = uniform(sc * batch) if case["beta"] != 0.0 else torch.zeros(sc * batch, device="cuda", dtype=TORCH[d])
    return {"case": case, "A": A, "B": B, "C": C, "strides": (sa, sb, sc)}


def run(state):
    """One call; returns C (with the rows between m and ldc, which stay as they are)."""
    c, A, B, C = state["case"], state["A"], state["B"], state["C"]
    if c["batch"] == 1 and c["workspace"] == "own":
        G.gemm(DTYPE[c["dtype"]], c["ta"], c["tb"], c["m"], c["n"], c["k"], c["alpha"], A, c["lda"], B, c["ldb"], c["beta"], C,
               c["ldc"])
    else:
        sa, sb, sc = state["strides"]
        call = G.gemm_strided_batched if c["workspace"] == "own" else G.gemm_strided_batched_static_workspace
        call(DTYPE[c["dtype"]], c["ta"], c["tb"], c["m"], c["n"], c["k"], c["alpha"], A, c["lda"], sa, B, c["ldb"], sb, c["beta"],
             C, c["ldc"], sc, c["batch"])
    return C


def work(case):
    """Each operand once (C twice where it is updated), two operations per multiply-add."""
    m, n, k, batch = case["m"], case["n"], case["k"], case["batch"]
    return {"bytes": batch * (m * k + k * n + m * n * (2 if case["beta"] != 0.0 else 1)) * ESZ[case["dtype"]],
            "flops": 2 * batch * m * n * k}


def tolerance(case):
    """Sums of k products in another order: about four times what these calls and drawn ones showed against the same sums in
    64 bits.  fp16 results are fp32 sums rounded once to 11 bits (2.1e-4 in the 2-norm, half an ulp = 4.9e-4 at most); fp32
    showed 1.8e-8 * sqrt(k) and at most 1.6e-7 * sqrt(k), fp64 3.7e-17 * sqrt(k) and at most 1.2e-15 * sqrt(k)."""
    root = math.sqrt(case["k"])
    if case["dtype"] == "h":
        return {"rel": 8.5e-4, "max": 2e-3}
    if case["dtype"] == "s":
        return {"rel": 8e-8 * root + 1e-7, "max": 7e-7 * root + 1e-6}
    return {"rel": 1.5e-16 * root + 3e-16, "max": 5e-15 * root + 4e-15}
