"""The work that programs have this library do, as cases that can be timed through its public Python entry points.

A case is a dict of plain values.  Its ``kind`` names the entry point:

    srgemm   cuasr_amd.srgemm            one product, any semiring, element type, extents and layouts
    square   cuasr_amd.srgemm            one squaring of a distance matrix, D_out = min(D, D (x) D)
    splitk   cuasr_amd.srgemm_splitk     a small output over a long k range
    batched  cuasr_amd.srgemm_batched    many small products in one call
    apsp     cuasr_amd.apsp_blocked      all-pairs shortest paths with predecessors, from the edge matrix

Layouts are three letters for A, B and the output (c = column-major, r = row-major).  ``source`` says whether the
epilogue folds a C in (beta = the semiring's one) or not (beta = its zero).  Sums use true infinities as identities.
"""
import math

import torch

import cuasr_amd

PAIRS = {"minplus": ("minimum", "plus"), "maxplus": ("maximum", "plus"), "mintimes": ("minimum", "multiplies"),
         "maxtimes": ("maximum", "multiplies"), "minmax": ("minimum", "maximum"), "maxmin": ("maximum", "minimum"),
         "orand": ("logical_or", "logical_and"), "plustimes": ("plus", "multiplies"), "xorand": ("bit_xor", "bit_and")}
TORCH_OF = {"f32": torch.float32, "f64": torch.float64, "f16": torch.float16, "i32": torch.int32, "u32": torch.int32,
            "i8": torch.int32}
BYTES_OF = {"f32": 4, "f64": 8, "f16": 2, "i32": 4, "u32": 4, "i8": 4}     # of C, D and the accumulator


def _srgemm(name, pair, dtype, m, n, k, layouts, source, kernel="auto"):
    return {"name": name, "kind": "srgemm", "pair": pair, "dtype": dtype, "m": m, "n": n, "k": k, "layouts": layouts,
            "source": source, "kernel": kernel}


def listed():
    return [
        # the smallest size of the semiring x size benchmark matrix: what a call costs when the product is next to nothing
        _srgemm("minplus_f32_256", "minplus", "f32", 256, 256, 256, "ccc", True),
        # a step of all-pairs shortest paths on a graph whose vertex count nobody chose: odd, nothing aligned
        {"name": "square_f32_1533", "kind": "square", "dtype": "f32", "n": 1533, "density": 1.0},
        # the same step on a large sparse graph (10 % edges): the headline benchmark's first squaring
        {"name": "square_f32_4096", "kind": "square", "dtype": "f32", "n": 4096, "density": 0.1},
        # bottleneck paths in double precision, the largest product of the benchmark's configurations
        _srgemm("maxmin_f64_8192", "maxmin", "f64", 8192, 8192, 8192, "ccc", True),
        # critical paths (max-plus) in double precision on a few hundred events, rectangular
        _srgemm("maxplus_f64_600x500x700", "maxplus", "f64", 600, 500, 700, "rrr", True),
        # the ordinary ring, at the middle of the benchmark matrix
        _srgemm("plustimes_f32_1024", "plustimes", "f32", 1024, 1024, 1024, "ccc", False),
        # counting paths / integer inference: int8 operands, int32 sums, both operands k-contiguous
        _srgemm("plustimes_i8_4096", "plustimes", "i8", 4096, 4096, 4096, "rcr", False),
        # shortest paths where half precision is enough
        _srgemm("minplus_f16_2000", "minplus", "f16", 2000, 2000, 2000, "ccc", True),
        # GF(2) on bit-packed words, rectangular
        _srgemm("xorand_u32_3000x2500x2000", "xorand", "u32", 3000, 2500, 2000, "rrr", False),
        # a small output over a long reduction: partial tiles in a workspace, then the reduction kernel
        {"name": "splitk_f32_256x256x65536", "kind": "splitk", "pair": "minplus", "dtype": "f32", "m": 256, "n": 256, "k": 65536,
         "layouts": "rcr", "source": True, "slices": 32},
        # many small graphs at once
        {"name": "batched_f32_1024x64", "kind": "batched", "pair": "minplus", "dtype": "f32", "batch": 1024, "m": 64, "n": 64, "k": 64,
         "layouts": "rrr", "source": True},
        # a whole shortest-path job with predecessors on a graph of ordinary size
        {"name": "apsp_f32_2000", "kind": "apsp", "dtype": "f32", "n": 2000, "density": 0.1},
    ]


def _extent(rng, lo, hi):
    """Log-uniform in [lo, hi]; half of them whole multiples of 16 as padded data has, half anything."""
    x = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5:
        x = max(16, (x + 8) // 16 * 16)
    return min(max(x, lo), hi)


def draw(rng):
    kind = rng.choices(["srgemm", "square", "splitk", "batched", "apsp"], [6, 2, 1, 1, 2])[0]
    layouts = "".join(rng.choice("cr") for _ in range(3))
    source = rng.random() < 0.5
    if kind == "srgemm":
        dtype = rng.choices(["f32", "f64", "f16", "i8", "u32", "i32"], [6, 4, 2, 2, 1, 1])[0]
        kernel = "auto"
        if dtype == "u32":
            pair = "xorand"
        elif dtype == "i32":
            pair = rng.choice(["minplus", "maxplus"])
        elif dtype == "f16":
            # binary16 sums are accumulated in float, which the caller asks for by naming the matrix cores
            pair = rng.choice(["minplus", "maxplus", "maxmin", "plustimes"])
            kernel = "mfma" if pair == "plustimes" else "auto"
        elif dtype == "i8":
            pair = rng.choice(["plustimes", "plustimes", "minplus", "maxmin"])
        else:
            pair = rng.choice(["minplus", "maxplus", "mintimes", "maxtimes", "minmax", "maxmin", "orand", "plustimes", "plustimes"])
        m, n, k = (_extent(rng, 64, 4096) for _ in range(3))
        return {"kind": kind, "pair": pair, "dtype": dtype, "m": m, "n": n, "k": k, "layouts": layouts, "source": source,
                "kernel": kernel}
    if kind == "square":
        return {"kind": kind, "dtype": rng.choice(["f32", "f32", "f64"]), "n": _extent(rng, 200, 4096),
                "density": rng.choice([0.1, 1.0])}
    if kind == "splitk":
        return {"kind": kind, "pair": rng.choice(["minplus", "maxplus", "maxmin"]), "dtype": rng.choice(["f32", "f32", "f64"]),
                "m": _extent(rng, 64, 512), "n": _extent(rng, 64, 512), "k": _extent(rng, 4096, 65536), "layouts": layouts,
                "source": source, "slices": rng.choice([8, 16, 32, 64])}
    if kind == "batched":
        m, n, k = (_extent(rng, 32, 128) for _ in range(3))
        return {"kind": kind, "pair": rng.choice(["minplus", "maxplus", "maxmin", "plustimes"]), "dtype": rng.choice(["f32", "f32", "f64"]),
                "batch": int(round(math.exp(rng.uniform(math.log(64), math.log(2048))))), "m": m, "n": n, "k": k, "layouts": layouts,
                "source": source}
    return {"kind": kind, "dtype": rng.choice(["f32", "f32", "f64"]), "n": _extent(rng, 200, 4096), "density": rng.choice([0.02, 0.1, 0.5])}


# ---- inputs

def _values(gen, pair, dtype, k, *shape):
    """What the pair's operands hold in earnest."""
    dev = "cuda"
    if dtype == "u32":
        return torch.randint(-(1 << 31), 1 << 31, shape, generator=gen, device=dev, dtype=torch.int64).to(torch.int32)
    if dtype == "i32":
        return torch.randint(0, 1 << 20, shape, generator=gen, device=dev, dtype=torch.int32)
    if dtype == "i8":
        return torch.randint(-128, 128, shape, generator=gen, device=dev, dtype=torch.int32).to(torch.int8)
    real = torch.float64 if dtype == "f64" else torch.float32
    if pair == "plustimes":
        v = torch.randn(shape, generator=gen, device=dev, dtype=real)
    elif pair == "orand":     # adjacency: about half of the result's entries are reachable
        v = (torch.rand(shape, generator=gen, device=dev, dtype=real) < math.sqrt(0.7 / max(k, 1))).to(real)
    elif pair in ("mintimes", "maxtimes"):    # reliabilities
        v = torch.rand(shape, generator=gen, device=dev, dtype=real)
    else:                     # lengths, capacities
        v = 100.0 * torch.rand(shape, generator=gen, device=dev, dtype=real)
    return v.to(TORCH_OF[dtype])


def _matrix(gen, pair, dtype, k, rows, cols, layout, batch=()):
    shape = batch + ((cols, rows) if layout == "c" else (rows, cols))
    v = _values(gen, pair, dtype, k, *shape)
    return v.transpose(-1, -2) if layout == "c" else v


def _graph(gen, dtype, n, density):
    """Column-major n x n edge matrix: 0 on the diagonal, edges U[1, 100), +inf elsewhere."""
    real = TORCH_OF[dtype]
    w = 1.0 + 99.0 * torch.rand((n, n), generator=gen, device="cuda", dtype=real)
    if density < 1.0:
        w[torch.rand((n, n), generator=gen, device="cuda") >= density] = math.inf
    w.fill_diagonal_(0.0)
    return w.t()


def _constants(pair, dtype, source):
    add, mult = PAIRS[pair]
    ident = cuasr_amd.op_identity(add, dtype, True)
    one = cuasr_amd.op_identity(mult, dtype, True)
    return add, mult, one, (one if source else ident), ident, one


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind, dtype = case["kind"], case["dtype"]
    if kind == "apsp":
        n = case["n"]
        edges = _graph(gen, dtype, n, case["density"])
        dist = torch.empty((n, n), dtype=edges.dtype, device="cuda").t()
        parent = torch.empty((n, n), dtype=torch.int32, device="cuda").t()
        work = torch.empty(cuasr_amd.apsp_blocked_workspace_bytes(n, dtype), dtype=torch.uint8, device="cuda")
        return {"kind": kind, "edges": edges, "dist": dist, "parent": parent, "work": work}
    if kind == "square":
        n = case["n"]
        D = _graph(gen, dtype, n, case["density"])
        return {"kind": kind, "D": D, "out": torch.empty((n, n), dtype=D.dtype, device="cuda").t()}
    pair, m, n, k = case["pair"], case["m"], case["n"], case["k"]
    la, lb, lc = case["layouts"]
    batch = (case["batch"],) if kind == "batched" else ()
    A = _matrix(gen, pair, dtype, k, m, k, la, batch)
    B = _matrix(gen, pair, dtype, k, k, n, lb, batch)
    if dtype == "i8":
        C = torch.randint(-1000, 1000, (n, m) if lc == "c" else (m, n), generator=gen, device="cuda", dtype=torch.int32)
        C = C.t() if lc == "c" else C
    else:
        C = _matrix(gen, pair, dtype, k, m, n, lc, batch)
    D = torch.empty_like(C)           # (keeps the strides)
    state = {"kind": kind, "A": A, "B": B, "C": C, "D": D, "constants": _constants(pair, dtype, case["source"]), "dtype": dtype,
             "kernel": case.get("kernel", "auto")}
    if kind == "splitk":
        state["slices"] = case["slices"]
        state["work"] = torch.empty(cuasr_amd.splitk_workspace_bytes(m, n, case["slices"], dtype), dtype=torch.uint8, device="cuda")
    return state


def run(state):
    kind = state["kind"]
    if kind == "square":
        D = state["D"]
        return cuasr_amd.srgemm("minimum", "plus", D, D, D, state["out"], 0.0, 0.0, math.inf, 0.0)
    if kind == "apsp":
        state["dist"].copy_(state["edges"])
        state["parent"].fill_(-1)
        return cuasr_amd.apsp_blocked(state["dist"], state["parent"], state["work"])
    add, mult, alpha, beta, ident, one = state["constants"]
    A, B, C, D = state["A"], state["B"], state["C"], state["D"]
    if kind == "splitk":
        return cuasr_amd.srgemm_splitk(add, mult, A, B, C, D, state["slices"], state["work"], alpha, beta, ident, one,
                                       dtype=state["dtype"])
    if kind == "batched":
        return cuasr_amd.srgemm_batched(add, mult, A, B, C, D, alpha, beta, ident, one, dtype=state["dtype"])
    return cuasr_amd.srgemm(add, mult, A, B, C, D, alpha, beta, ident, one, dtype=state["dtype"], kernel=state["kernel"])


def work(case):
    """Each input read once, each output written once; two operations per term of the inner products."""
    es = BYTES_OF[case["dtype"]]
    if case["kind"] == "apsp":
        n = case["n"]
        return {"bytes": n * n * (2 * es + 4), "flops": 2 * n ** 3}
    if case["kind"] == "square":
        n = case["n"]
        return {"bytes": 2 * n * n * es, "flops": 2 * n ** 3}
    m, n, k, b = case["m"], case["n"], case["k"], case.get("batch", 1)
    os = 1 if case["dtype"] == "i8" else es
    return {"bytes": b * ((m * k + k * n) * os + m * n * es * (2 if case["source"] else 1)), "flops": 2 * b * m * n * k}


def tolerance(case):
    """Minima, maxima, bits and integers come out the same whatever the order of the terms; sums of rounded
    products do not.  Measured at k = 4096 against the same product in 64 bits (f32: 1.15e-6; f16 operands with
    float sums, one rounding at the end: 2.1e-4) and in extended precision (f64: 2.2e-15), times four."""
    if case.get("pair") == "plustimes" and case["dtype"] != "i8":
        return {"f32": {"rel": 5e-6}, "f64": {"rel": 1e-14}, "f16": {"rel": 8e-4}}[case["dtype"]]
    return "exact"
