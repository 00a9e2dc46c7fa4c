"""The work that a user of this library has it do, as cases that can be timed.

The library serves quantised linear layers.  A layer's weight is quantised
and laid out once, when a model is loaded; every call then quantises the
layer's bf16 activations and multiplies.  A case is one such pass:

* ``path`` "linear": ``layers`` layers of one shape, each with its own weight
  and activations [m, k] (``quant``: the pass starts from bf16 activations,
  otherwise from activations that the step before already quantised), for one
  of the operand formats in ``fmt``;
* ``path`` "group": one grouped launch over the projections of one decode step;
* ``path`` "weight": the quantisation and layout of one weight [n, k].

``graph``: the pass is a replay of a captured HIP graph, as a serving loop runs
its decode step (the capture and its warm-up belong to the preparation);
otherwise the entry points are called one by one, as a prefill does.

``fmt``: "bs" fp8 with fp32 1x128 / 128x128 scales and the K-panel weight,
"bypass" the same with the fragment-order weight, "e8m0" fp8 with E8M0 block
scales (``layout`` nt / nn / tt / tn), "mxfp8" and "mxfp4" one E8M0 scale per 32
K with row-major operands, "mxfp4_aiter" with the shuffled weight and scales.
"""
import importlib
import math

import torch

q = importlib.import_module("355_1_trans_amd")

DEV = "cuda"
FLOPS_MOST = 2.0 * 8192 ** 3
BYTES_MOST = 400e6

# (n, k) of one decode step's projections over the same tokens: the grouped launch.
GROUP = ((2112, 7168), (4096, 7168), (7168, 2048))


def _linear(name, fmt, m, n, k, *, layers=1, quant=True, graph=False, out="bf16", layout="nt"):
    return {"name": name, "path": "linear", "fmt": fmt, "m": m, "n": n, "k": k, "layers": layers, "quant": quant,
            "graph": graph, "out": out, "layout": layout}


def listed():
    return [
        # One token through one narrow projection, called eagerly: the smallest call, all latency and launches.
        _linear("token_bs_m1", "bs", 1, 2112, 7168),
        # The decode steps of a serving loop, replayed from a graph: a batch of 32 through narrow projections with
        # fp32 block scales, ...
        _linear("decode_bs_m32", "bs", 32, 1536, 7168, layers=4, graph=True),
        # ... the same batch through a wide long-K MXFP4 projection whose input is already quantised (bound by
        # reading the weight), ...
        _linear("decode_mxfp4_m32", "mxfp4", 32, 7168, 16384, layers=2, quant=False, graph=True),
        # ... a ragged batch through shuffled MXFP4 weights, ...
        _linear("decode_aiter_m57", "mxfp4_aiter", 57, 4096, 7168, layers=4, graph=True),
        # ... and all projections of the step in one grouped launch.
        {"name": "group_bypass_m16", "path": "group", "fmt": "bypass", "m": 16, "quant": True, "graph": True},
        # Chunked prefill: the few hundred tokens of a chunk, too few rows to fill the chip with large tiles, with a
        # ragged last chunk ...
        _linear("chunk_mxfp8_m500", "mxfp8", 500, 4096, 7168),
        # ... and a chunk through the LDS-bypass entry.
        _linear("chunk_bypass_m192", "bypass", 192, 7168, 2048),
        # Prefill of thousands of tokens: fp32 block scales with short K, ...
        _linear("prefill_bs_m4096", "bs", 4096, 7168, 2048),
        # ... E8M0 block scales, ...
        _linear("prefill_e8m0_m4096", "e8m0", 4096, 4096, 7168),
        # ... and a long MXFP4 prefill.
        _linear("prefill_aiter_m16384", "mxfp4_aiter", 16384, 7168, 2048),
        # The largest product: the benchmark's own MXFP8 shape, operands at hand.
        _linear("square_mxfp8_8192", "mxfp8", 8192, 8192, 8192, quant=False),
        # Loading a model: a bf16 weight is quantised to MXFP4 and shuffled for serving.
        {"name": "weight_aiter_7168", "path": "weight", "fmt": "mxfp4_aiter", "n": 7168, "k": 16384},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _aligned(rng, lo, hi, step):
    return max(step, _log_int(rng, lo, hi) // step * step)


def draw(rng):
    """One more case of the listed ranges: the path by how often it is listed, sizes over the logarithm of the range."""
    pick = rng.random()
    if pick < 0.1:
        return {"path": "group", "fmt": rng.choice(("bs", "bypass", "mxfp8", "mxfp4")), "m": _log_int(rng, 1, 64),
                "quant": True, "graph": True}
    while pick < 0.2:
        fmt = rng.choice(("bs", "bypass", "e8m0", "mxfp8", "mxfp4", "mxfp4_aiter"))
        case = {"path": "weight", "fmt": fmt, "n": _aligned(rng, 1536, 16384, 128), "k": _aligned(rng, 1536, 16384, 256)}
        if work(case)["bytes"] <= BYTES_MOST:
            return case
    while True:
        decode = rng.random() < 0.5
        fmt = rng.choice(("bs", "bypass", "mxfp8", "mxfp4", "mxfp4_aiter")) if decode else \
            rng.choice(("bs", "bypass", "e8m0", "mxfp8", "mxfp4", "mxfp4_aiter"))
        if decode:
            m = _log_int(rng, 1, 64)
        elif fmt == "e8m0":
            m = _aligned(rng, 512, 16384, 256)
        else:
            m = _log_int(rng, 65, 16384)
        n_step = 256 if fmt == "e8m0" else 16 if fmt == "mxfp4_aiter" else 1
        case = {"path": "linear", "fmt": fmt, "m": m, "n": _aligned(rng, 1536, 24576, n_step),
                "k": _aligned(rng, 1536, 16384, 256), "layers": rng.choice((1, 2, 4)) if decode else 1,
                "quant": rng.random() < 0.7, "graph": decode and rng.random() < 0.7,
                "out": rng.choice(("bf16", "bf16", "bf16", "fp32")),
                "layout": rng.choice(("nt", "nt", "nn", "tt", "tn")) if fmt == "e8m0" else "nt"}
        if case["layout"] in ("tt", "tn"):
            case["quant"] = False      # the quantisers write row-major activations
        w = work(case)
        if w["flops"] <= FLOPS_MOST and w["bytes"] <= BYTES_MOST:
            return case


# ------------------------------------------------------------------ inputs
def _normal(seed, stream, rows, cols):
    """bf16 N(0, 1) values with a few larger channels, as activations and weights have them."""
    g = torch.Generator(DEV).manual_seed(seed * 1000003 + stream)
    x = torch.randn((rows, cols), generator=g, device=DEV, dtype=torch.float32)
    x *= torch.exp(0.5 * torch.randn((1, cols), generator=g, device=DEV))
    return x.to(torch.bfloat16)


def _activations(case, seed, i, m, k):
    return _normal(seed, 2 * i, m, k)


def _weight(case, seed, i, n, k):
    return _normal(seed, 2 * i + 1, n, k) * 0.02


def _shapes(case):
    if case["path"] == "group":
        return [(case["m"], n, k) for n, k in GROUP]
    if case["path"] == "linear":
        return [(case["m"], case["n"], case["k"])] * case["layers"]
    return []


# ------------------------------------------------------- the library's side
def _quant_act(case, x):
    fmt = case["fmt"]
    if fmt in ("bs", "bypass"):
        return q.quant_fp8_blockscale(x)
    if fmt == "e8m0":
        return q.quant_fp8_e8m0_blockscale(x)
    if fmt == "mxfp8":
        return q.quant_mxfp8(x)
    return q.quant_mxfp4(x, shuffle=fmt == "mxfp4_aiter")


def _prepare_weight(case, w):
    """The weight as its GEMM takes it: (codes, scales)."""
    fmt = case["fmt"]
    if fmt in ("bs", "bypass"):
        codes, scale = q.quant_fp8_blockscale(w, block="128x128")
        return (q.shuffle_b_kpanel(codes) if fmt == "bs" else q.ldsbypass_pack_b(codes)), scale
    if fmt == "e8m0":
        codes, scale = q.quant_fp8_e8m0_blockscale(w, block="128x128")
        layout = case.get("layout", "nt")
        if layout == "nt":
            return q.shuffle_weight_16x16(codes), scale
        return (codes.view(torch.uint8).t().contiguous().view(codes.dtype) if layout[1] == "n" else codes), scale
    if fmt == "mxfp8":
        return q.quant_mxfp8(w)
    codes, scale = q.quant_mxfp4(w, shuffle=fmt == "mxfp4_aiter")
    return (q.shuffle_weight_16x16(codes) if fmt == "mxfp4_aiter" else codes), scale


def _gemm(case, act, weight, n):
    fmt, (a, sa), (b, sb) = case["fmt"], act, weight
    dtype = torch.float32 if case["out"] == "fp32" else torch.bfloat16
    if fmt == "bs":
        return q.gemm_a8w8_bpreshuffle(a, b, sa, sb, dtype=dtype)
    if fmt == "bypass":
        return q.gemm_a8w8_ldsbypass(a, b, sa, sb, n, dtype=dtype)
    if fmt == "e8m0":
        layout = case["layout"]
        if layout == "nt":
            return q.blockscale_bpreshuffle.gemm_a8w8_blockscale_bpreshuffle(a, b, sa, sb, dtype)
        y = torch.empty((sa.shape[0], n), dtype=dtype, device=DEV)
        return getattr(q, "opus_gemm_mxfp8_" + layout)(a, b, sa, sb, y)
    if fmt == "mxfp8":
        return q.gemm_a8w8_mxfp8(a, b, sa, sb, dtype=dtype)
    if fmt == "mxfp4":
        return q.gemm_a4w4_mxfp4(a, b, sa, sb, dtype=dtype)
    return q.gemm_a4w4(a, b, sa, sb, dtype=dtype)


def _pass(state):
    case = state["case"]
    if case["path"] == "weight":
        codes, scale = _prepare_weight(case, state["w"])
        return [codes.view(torch.uint8), scale]
    if case["path"] == "group":    # projections of one width read the same tokens
        acts = {k: _quant_act(case, x) for k, x in state["x"].items()}
        problems = [(acts[k][0], w[0], acts[k][1], w[1]) + ((n,) if case["fmt"] == "bypass" else ())
                    for w, (_, n, k) in zip(state["w"], _shapes(case))]
        return q.gemm_grouped({"bs": "bpreshuffle", "bypass": "ldsbypass"}.get(case["fmt"], case["fmt"]), problems)
    acts = [_quant_act(case, x) for x in state["x"]] if case["quant"] else state["x"]
    return [_gemm(case, a, w, case["n"]) for a, w in zip(acts, state["w"])]


_STREAM = []


def prepare(case, seed):
    state = {"case": case}
    if case["path"] == "weight":
        state["w"] = _weight(case, seed, 0, case["n"], case["k"])
        return state
    shapes = _shapes(case)
    state["w"] = [_prepare_weight(case, _weight(case, seed, i, n, k)) for i, (_, n, k) in enumerate(shapes)]
    acts = [_activations(case, seed, i, m, k) for i, (m, _, k) in enumerate(shapes)]
    state["x"] = {k: x for (_, _, k), x in zip(shapes, acts)} if case["path"] == "group" else acts
    if not case["quant"]:
        state["x"] = [_quant_act(case, x) for x in state["x"]]
        if case.get("layout", "nt")[0] == "t":
            state["x"] = [(a.view(torch.uint8).t().contiguous().view(a.dtype), s) for a, s in state["x"]]
    if case["graph"]:
        # Warm up and capture on one stream, the usual way: the warm-up brings the cached workspace.
        if not _STREAM:
            _STREAM.append(torch.cuda.Stream())
        side = _STREAM[0]
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            _pass(state)
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"], stream=side):
            state["y"] = _pass(state)
    return state


def run(state):
    if "graph" not in state:
        return _pass(state)
    state["graph"].replay()
    return state["y"]


# -------------------------------------------------------------------- work
def _operand_bytes(fmt, rows, k, weight=False):
    """Codes and scales of one quantised operand."""
    codes = rows * k / 2 if fmt.startswith("mxfp4") else rows * k
    if fmt.startswith("mx"):
        return codes + rows * k / 32
    scale = 1 if fmt == "e8m0" else 4
    return codes + scale * (math.ceil(rows / 128) if weight else rows) * (k / 128)


def work(case):
    if case["path"] == "weight":
        n, k = case["n"], case["k"]
        return {"bytes": 2.0 * n * k + _operand_bytes(case["fmt"], n, k, True), "flops": 0.0}
    total = {"bytes": 0.0, "flops": 0.0}
    read = set()
    for m, n, k in _shapes(case):
        out = 4 if case.get("out") == "fp32" else 2
        total["flops"] += 2.0 * m * n * k
        total["bytes"] += _operand_bytes(case["fmt"], n, k, True) + out * m * n
        if case["path"] == "linear" or k not in read:
            total["bytes"] += 2.0 * m * k if case["quant"] else _operand_bytes(case["fmt"], m, k)
        read.add(k)
    return total


def tolerance(case):
    if case["path"] == "weight":
        return "exact"
    # fp32 sums of products, rounded once to the output's type.  Measured against 64 bits: bf16 1.7e-3 / 3.9e-3 (its
    # own rounding), fp32 2.8e-5 / 4.2e-4 (the matrix instruction's sums of fp8 products; fp4 sums are exact).
    if case.get("out") == "fp32":
        return {"rel": 1e-4, "max": 1.6e-3}
    return {"rel": 7e-3, "max": 1.6e-2}


# ------------------------------------------------------------- the oracle
def _pow2_scale(amax, top):
    """2^ceil(log2(amax / top)), 1 for an all-zero group."""
    v = amax / torch.full_like(amax, top)      # a true division: by a number, torch multiplies by its reciprocal
    mant, exp = torch.frexp(v)
    return torch.where(amax > 0, torch.ldexp(torch.ones_like(v), exp - (mant == 0.5).to(exp.dtype)), torch.ones_like(v))


def _round(x, fp4):
    if not fp4:
        return x.clamp(-448, 448).to(torch.float8_e4m3fn).double()
    a = x.abs()
    step = torch.where(a < 2, 0.5, torch.where(a < 4, 1.0, 2.0))
    return (torch.sign(x) * torch.clamp(torch.round(a / step) * step, max=6.0)).double()


def _dequantised(case, x, weight=False):
    """The values that the codes and scales of x stand for, in 64 bits, by the formats' recipes."""
    fmt, (rows, k) = case["fmt"], x.shape
    fp4, x = fmt.startswith("mxfp4"), x.float()
    if fmt.startswith("mx"):
        t = x.reshape(rows, k // 32, 32)
        s = _pow2_scale(t.abs().amax(-1, keepdim=True), 6.0 if fp4 else 448.0)
    else:
        pad = -rows % 128 if weight else 0
        t = torch.nn.functional.pad(x, (0, 0, 0, pad))
        t = t.reshape(-1, 128 if weight else 1, k // 128, 128)
        amax = t.abs().amax((1, 3), keepdim=True)
        s = _pow2_scale(amax, 448.0) if fmt == "e8m0" else \
            torch.where(amax > 0, amax / torch.full_like(amax, 448.0), torch.ones_like(amax))
    return (_round(t / s, fp4) * s.double()).reshape(-1, k)[:rows]


def exact(case, seed):
    if case["path"] == "weight":
        return None
    got = []
    shapes = _shapes(case)
    stream = {k: i for i, (_, _, k) in enumerate(shapes)} if case["path"] == "group" else None
    for i, (m, n, k) in enumerate(shapes):
        a = _dequantised(case, _activations(case, seed, stream[k] if stream else i, m, k))
        b = _dequantised(case, _weight(case, seed, i, n, k), True)
        got.append(a @ b.t())
    return got
