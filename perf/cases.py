"""Performance cases of the vector-quantized GEMM framework: what users have it do, through its public entry points.

A case is a flat dict; its `kind` says which call a pass is made of:

  linear    a `VQLinear` layer called on activations [M, K] (`stages` > 1: additive codes, bias optional), one call
  e2e       the reference's call, `e2e_gemm(input, w, codebook)`, on K-axis codes
  native    the same call on the reference's own tensors: codes [K, Nc], codebook [Nc/4, 256, 2]
  mlp       a `VQGatedMLP` block (gate/up product with the gated epilogue, then the down projection), called once
  step      the gated MLP blocks of one decode step, captured in a HIP graph when the model is loaded and replayed
  gemm      the plain fp16 product `gemm(input, w)`, the other half of the reference's module
  codec     a weight onto its nearest codewords and back: `encode_b`, then `dequant_b` (the projection step of
            quantisation-aware training, and the check behind a checkpoint that was written)
  quantize  `kmeans_quantize` of a weight matrix: Lloyd iterations, once per layer when a model is quantised

M counts the rows of activations: 1 to 64 in decode (one per sequence), up to thousands in prefill.  Codes are uniform,
codebooks N(0, 0.02) and activations N(0, 1), the distributions of the repository's configurations.
"""
import math

import torch

from vq_gemm_amd import cabi, ops
from vq_gemm_amd.nn import VQGatedMLP, VQLinear
from vq_gemm_amd.quantize import kmeans_quantize

DEVICE = "cuda"

# (vector length, codebook entries, code bits) of the formats in use
FORMATS = ((8, 256, 8), (4, 256, 8), (4, 4096, 16))


def _linear(M, K, N, vec=8, entries=256, bits=8, books=1, stages=1, bias=False, **more):
    return dict(kind="linear", M=M, K=K, N=N, vec=vec, entries=entries, bits=bits, books=books, stages=stages, bias=bias, **more)


def listed():
    return [
        # one token through a 4096 x 4096 attention projection: the smallest call of a decode loop
        _linear(1, 4096, 4096, name="decode_proj_m1"),
        # sixteen sequences through a key or value projection, by the reference's own call
        dict(name="kv_proj_e2e_m16", kind="e2e", M=16, K=4096, N=1024, vec=4, entries=256, bits=8, books=1),
        # one token through the gated MLPs of eight layers, replayed as the one graph that a serving loop keeps
        dict(name="decode_step_mlp_m1", kind="step", M=1, K=4096, H=11008, layers=8),
        # sixteen sequences through an up-projection with 12-bit codes: the higher-quality format
        _linear(16, 4096, 11008, vec=4, entries=4096, bits=16, name="batch_up_proj_m16"),
        # five sequences through a layer quantised in two additive stages, with bias
        _linear(5, 4096, 4096, entries=256, bits=16, stages=2, bias=True, name="residual_bias_m5"),
        # a short prompt of odd length through a gated MLP whose width is no multiple of the tiles
        dict(name="prompt_mlp_ragged_m333", kind="mlp", M=333, K=2880, H=7680),
        # prefill of a 4096-token prompt through an attention projection, one codebook per 128 rows
        _linear(4096, 4096, 4096, books=32, name="prefill_proj_m4096"),
        # prefill through the up-projection of a large model, one codebook per 512 rows
        _linear(2048, 8192, 28672, books=56, name="prefill_large_m2048"),
        # the reference harness's shape on the reference's own tensors
        dict(name="native_m2048", kind="native", M=2048, K=4096, Nc=640),
        # the reference harness's control: the plain product
        dict(name="gemm_4096", kind="gemm", M=4096, K=4096, N=4096),
        # a projection's weight encoded with given codebooks and read back
        dict(name="codec_4096", kind="codec", N=4096, K=4096, vec=8, entries=256, bits=8, books=1),
        # a projection's weight quantised from scratch with the default ten iterations
        dict(name="quantize_4096", kind="quantize", N=4096, K=4096, vec=8, entries=256, bits=8, books=8, iters=10),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _rows(rng, lo, hi):
    return max(lo, min(hi, round(_log(rng, lo, hi))))


def _width(rng, lo, hi):
    """A layer width: mostly a multiple of 128, now and then only of 64."""
    step = rng.choice((128, 128, 64))
    return max(lo, step * round(_log(rng, lo, hi) / step))


def _outputs(rng, lo, hi):
    """A number of output features: a multiple of 128, of 16, or any."""
    step = rng.choice((128, 128, 16, 1))
    return max(lo, step * round(_log(rng, lo, hi) / step))


MOST_FLOPS = 2.0 * 2048 * 8192 * 28672


def _fit(M, per_row):
    """M, lowered where the product would cost more than the largest listed one."""
    return max(1, min(M, int(MOST_FLOPS // per_row)))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "linear", "e2e", "native", "mlp", "step", "gemm", "codec", "quantize"))
    if kind in ("linear", "e2e"):
        vec, entries, bits = rng.choice(FORMATS + FORMATS[:1])
        K, N = _width(rng, 512, 14336), _outputs(rng, 512, 28672)
        books = 1
        if rng.random() < 0.4 and N % 128 == 0:
            books = rng.choice([b for b in (1, 2, 3, 4, 8, 16, 32, 56, N // 512, N // 128) if b and (N // 128) % b == 0])
        M = _fit(_rows(rng, 1, 4096), 2.0 * K * N)
        if kind == "e2e" and (M < 4 or K * N < 1 << 22):
            kind = "linear"  # (products this small go through a layer)
        if kind == "e2e":
            return dict(kind="e2e", M=M, K=K, N=N, vec=vec, entries=entries, bits=bits, books=books)
        stages = 2 if rng.random() < 0.15 and entries == 256 else 1
        if stages == 2:
            return _linear(_fit(M, 4.0 * K * N), K, N, vec, entries, 16, books, 2, rng.random() < 0.5)
        return _linear(M, K, N, vec, entries, bits, books, 1, rng.random() < 0.3)
    if kind == "native":
        K, Nc = _width(rng, 512, 8192), 16 * round(_log(rng, 256, 4096) / 16)
        return dict(kind=kind, M=_fit(_rows(rng, 1, 4096), 4.0 * K * Nc), K=K, Nc=Nc)
    if kind in ("mlp", "step"):
        K, H = _width(rng, 1024, 8192), _width(rng, 2048, 28672)
        if kind == "step":
            return dict(kind=kind, M=_rows(rng, 1, 64), K=K, H=H, layers=rng.randint(2, 8))
        return dict(kind=kind, M=_fit(_rows(rng, 1, 4096), 6.0 * K * H), K=K, H=H)
    if kind == "gemm":
        K, N = _width(rng, 1024, 8192), _outputs(rng, 1024, 11008)
        return dict(kind=kind, M=_fit(_rows(rng, 16, 4096), 2.0 * K * N), K=K, N=N)
    vec, entries, bits = rng.choice(FORMATS if kind == "codec" else FORMATS[:2])
    K, N = _width(rng, 512, 4096), 16 * round(_log(rng, 512, 4096) / 16)
    books = rng.choice([b for b in (1, 2, 4, 8) if N % b == 0])
    if kind == "codec":
        return dict(kind=kind, N=N, K=K, vec=vec, entries=entries, bits=bits, books=books)
    return dict(kind=kind, N=N, K=K, vec=vec, entries=entries, bits=bits, books=books, iters=rng.randint(4, 10))


def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _half(gen, shape, std=1.0):
    return (torch.randn(shape, generator=gen, device=DEVICE) * std).half()


def _codes(gen, shape, entries, bits):
    c = torch.randint(0, entries, shape, generator=gen, device=DEVICE, dtype=torch.int32)
    return c.to(torch.uint8) if bits == 8 else c.to(torch.int16).view(torch.uint16)


def _codebook(gen, books, entries, vec):
    cb = _half(gen, (books, entries, vec), 0.02)
    return cb[0].contiguous() if books == 1 else cb


def _mlp(gen, K, H):
    gate_up = VQLinear(_codes(gen, (2 * H, K // 8), 256, 8), _codebook(gen, 1, 256, 8))
    down = VQLinear(_codes(gen, (K, H // 8), 256, 8), _codebook(gen, 1, 256, 8))
    return VQGatedMLP(gate_up, down, interleaved=True)


def prepare(case, seed):
    gen, kind = _gen(seed), case["kind"]
    if kind in ("linear", "e2e"):
        M, K, N, vec, entries, bits = (case[k] for k in ("M", "K", "N", "vec", "entries", "bits"))
        stages = case.get("stages", 1)
        x = _half(gen, (M, K))
        parts = [_codes(gen, (N, K // vec), entries, bits) for _ in range(stages)]
        codes = parts[0]
        if stages > 1:  # as residual_quantize lays them: side by side along K, each stage with its own rows of the codebook
            wide = [p.view(torch.int16).to(torch.int32) + s * entries for s, p in enumerate(parts)]
            codes = torch.cat(wide, dim=1).to(torch.int16).view(torch.uint16)
        codebook = _codebook(gen, case["books"], stages * entries, vec)
        if kind == "e2e":
            return {"kind": kind, "args": (x, codes, codebook)}
        bias = _half(gen, (N,)) if case["bias"] else None
        return {"kind": kind, "layer": VQLinear(codes, codebook, bias, k_repeat=stages), "x": x}
    if kind == "native":
        M, K, Nc = case["M"], case["K"], case["Nc"]
        return {"kind": "e2e", "args": (_half(gen, (M, K)), _codes(gen, (K, Nc), 256, 8), _half(gen, (Nc // 4, 256, 2), 0.02))}
    if kind == "mlp":
        return {"kind": "linear", "layer": _mlp(gen, case["K"], case["H"]), "x": _half(gen, (case["M"], case["K"]))}
    if kind == "step":
        blocks = [_mlp(gen, case["K"], case["H"]) for _ in range(case["layers"])]
        xs = [_half(gen, (case["M"], case["K"])) for _ in blocks]  # what the attention in front of each block hands it
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for block, x in zip(blocks, xs):
                block(x)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            ys = [block(x) for block, x in zip(blocks, xs)]
        return {"kind": kind, "graph": graph, "ys": ys, "keep": (blocks, xs)}
    if kind == "gemm":
        return {"kind": kind, "args": (_half(gen, (case["M"], case["K"])), _half(gen, (case["K"], case["N"]), 0.02))}
    w = _half(gen, (case["N"], case["K"]), 0.02)
    if kind == "codec":
        return {"kind": kind, "w": w, "codebook": _codebook(gen, case["books"], case["entries"], case["vec"])}
    return {"kind": kind, "w": w, "args": (case["vec"], case["entries"], case["books"], case["iters"])}


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["layer"](state["x"])
    if kind == "e2e":
        return ops.e2e_gemm(*state["args"])
    if kind == "step":
        state["graph"].replay()
        return state["ys"]
    if kind == "gemm":
        return ops.gemm(*state["args"])
    if kind == "codec":
        codes = cabi.encode_b(state["w"], state["codebook"])
        return codes, cabi.dequant_b(codes, state["codebook"])
    return kmeans_quantize(state["w"], *state["args"])


def work(case):
    """Inputs read once and outputs written once; the products' multiply-adds, a search's as the dot products it needs."""
    kind = case["kind"]
    if kind in ("linear", "e2e"):
        M, K, N, s = case["M"], case["K"], case["N"], case.get("stages", 1)
        codes = s * N * (K // case["vec"]) * (case["bits"] // 8)
        books = 2 * case["books"] * s * case["entries"] * case["vec"]
        return {"bytes": codes + books + 2 * M * (K + N) + (2 * N if case.get("bias") else 0), "flops": 2 * M * K * N}
    if kind == "native":
        M, K, Nc = case["M"], case["K"], case["Nc"]
        return {"bytes": K * Nc + Nc * 256 + 2 * M * (K + 2 * Nc), "flops": 4 * M * K * Nc}
    if kind in ("mlp", "step"):
        M, K, H, n = case["M"], case["K"], case["H"], case.get("layers", 1)
        return {"bytes": n * (3 * H * K // 8 + 2 * 4096 + 4 * M * K), "flops": n * 6 * M * K * H}
    if kind == "gemm":
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": 2 * (M * K + K * N + M * N), "flops": 2 * M * K * N}
    N, K, E = case["N"], case["K"], case["entries"]
    small = N * (K // case["vec"]) * (case["bits"] // 8) + 2 * case["books"] * E * case["vec"]
    if kind == "codec":
        return {"bytes": 4 * N * K + small, "flops": 2 * N * K * E}
    return {"bytes": 2 * N * K + small, "flops": 2 * N * K * E * (case["iters"] + 1)}


def tolerance(case):
    kind = case["kind"]
    if kind == "codec":
        return "exact"  # the encoder's rule fixes every bit, reading back is indexing
    if kind == "quantize":
        # the centroids are fp32 sums in no fixed order, rounded to fp16: an entry moves by a last place, and vectors
        # half way between two entries change sides
        return {"rel": 1e-2, "differ": 1e-2}
    # fp16 results of fp32 sums: half a last place each (rel 2^-12 to 2^-11), once more for the activations inside an MLP
    return {"rel": 2e-3 if kind in ("mlp", "step") else 1e-3}
