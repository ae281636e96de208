"""GPU parity tests: every kernel of libvqgemm.so, driven through the C ABI, against the CPU
oracle on identical seeded inputs.

Bars: dequantised weights bit-exact; GEMM outputs max |y-ref| / max(|ref|, tau) <= 2e-3 with
tau = 1e-2 * rms(ref), against an fp64-accumulated oracle (the fp32 oracle itself sits
within ~5e-4 of it; fp16 output rounding alone is <= 4.9e-4).
"""
import numpy as np
import pytest
import torch

from oracle import c_oracle
from oracle import vq_oracle as vo
from vq_gemm_amd import cabi
from vq_gemm_amd.problems import CONFIGS, GEOM_A, GEOM_B, ProblemSpec, make_problem

pytestmark = pytest.mark.gpu

TOL = 2e-3
DEV = "cuda:0"


def _say(*a):
    print(*a, flush=True)


def _np(t):
    return t.detach().cpu().numpy()


def _check_gemm(y_gpu, x, codes, cb, geometry=GEOM_B, what=""):
    if geometry == GEOM_B:
        ref = vo.vq_gemm_b(_np(x), _np(codes), _np(cb), acc=np.float64)
    else:
        ref = vo.vq_gemm_a(_np(x), _np(codes), _np(cb), acc=np.float64)
    e1, e2 = vo.rel_err(_np(y_gpu), ref)
    _say(f"  {what}: rel_err(floor)={e1:.3e} max/max={e2:.3e}")
    assert e1 <= TOL, (what, e1, e2)
    return e1


SMALL_B = [
    # name, M, K, N, vec, E, G, bits
    ("tiny_v8", 1, 512, 16, 8, 256, 1, 8),
    ("tiny_v4", 16, 1024, 64, 4, 256, 1, 8),
    ("m7_n_ragged", 7, 1024, 50, 8, 256, 1, 8),
    ("k_tail_v8", 3, 640, 32, 8, 256, 1, 8),          # K not a multiple of the 512 wave slice
    ("u16_v4", 16, 512, 48, 4, 4096, 1, 16),
    ("u16_v8", 5, 1024, 32, 8, 1000, 1, 16),
    ("u8_v2", 4, 256, 32, 2, 256, 1, 8),
    ("u16_v2", 2, 128, 16, 2, 300, 1, 16),
    ("multi_cb16", 9, 512, 64, 8, 256, 4, 8),          # 16 rows per codebook
    ("multi_cb128", 33, 512, 256, 8, 256, 2, 8),
    ("m17", 17, 512, 48, 8, 256, 1, 8),                  # decode kernel in 16-row slabs
    ("m64_slabs", 64, 1024, 80, 4, 4096, 1, 16),
    ("m65_prefill", 65, 256, 64, 8, 256, 1, 8),
    ("m300_ragged", 300, 384, 200, 8, 256, 1, 8),       # prefill kernel with ragged M, N and a K tail
    ("m64_v4", 64, 256, 96, 4, 256, 3, 8),
    ("deep_k", 2, 9216, 32, 8, 256, 1, 8),              # more K than one workgroup's waves cover at once
]


def _spec(row):
    name, M, K, N, v, E, G, bits = row
    return ProblemSpec(name, GEOM_B, M, K, N, v, E, G, bits, codebook_3d=(G > 1))


@pytest.mark.parametrize("row", SMALL_B, ids=[r[0] for r in SMALL_B])
def test_dequant_b_bit_exact(row):
    spec = _spec(row)
    _say("dequant_b", spec)
    _, codes, cb = make_problem(spec, seed=1, device=DEV)
    w = cabi.dequant_b(codes, cb)
    torch.cuda.synchronize()
    want = vo.dequant_b(_np(codes), _np(cb))
    assert np.array_equal(_np(w).view(np.uint16), want.view(np.uint16))
    assert np.array_equal(want.view(np.uint16), c_oracle.dequant_b(_np(codes), _np(cb)).view(np.uint16))


@pytest.mark.parametrize("N,K,v,E,G,bits", [(1030, 3080, 8, 8, 1, 8), (1026, 3100, 4, 16, 2, 16), (1551, 2050, 2, 31, 3, 8), (2000, 2056, 4, 250, 4, 8), (4100, 4096, 8, 256, 1, 8)])
def test_dequant_b_through_a_table_bit_exact(N, K, v, E, G, bits):
    """Enough weights for a codebook in the LDS: runs that are no multiple of a store or a pass, a result and codes off 16 bytes, codes
    past the last entry (which read that entry)."""
    g = torch.Generator().manual_seed(17)
    J = K // v
    wide = torch.randint(0, E + 3, (N * J + 1,), generator=g, dtype=torch.int32)
    codes = (wide.to(torch.uint8) if bits == 8 else wide.to(torch.int16).view(torch.uint16)).to(DEV)[1:].view(N, J)
    cb = torch.randn(G, E, v, generator=g).half().to(DEV)
    out = torch.full((N * K + 2 * v,), 7.0, dtype=torch.float16, device=DEV)
    _say("dequant_b table", N, K, v, E, G, bits)
    w = cabi.dequant_b(codes, cb, out=out[v:v + N * K].view(N, K))
    torch.cuda.synchronize()
    want = vo.dequant_b(np.minimum(_np(codes), E - 1), _np(cb))
    assert np.array_equal(_np(w).view(np.uint16), want.view(np.uint16))
    assert (out[:v] == 7.0).all() and (out[v + N * K:] == 7.0).all()


@pytest.mark.parametrize("K,Nc", [(1030, 1028), (4200, 256), (300, 4000)])
def test_dequant_a_through_a_table_bit_exact(K, Nc):
    g = torch.Generator().manual_seed(18)
    w = torch.randint(0, 256, (K, Nc), generator=g, dtype=torch.int32).to(torch.uint8).to(DEV)
    cb = torch.randn(Nc // 4, 256, 2, generator=g).half().to(DEV)
    _say("dequant_a table", K, Nc)
    got = cabi.dequant_a(w, cb)
    torch.cuda.synchronize()
    assert np.array_equal(_np(got).view(np.uint16), vo.dequant_a(_np(w), _np(cb)).view(np.uint16))


@pytest.mark.parametrize("row", SMALL_B, ids=[r[0] for r in SMALL_B])
def test_e2e_gemm_b_all_variants(row):
    spec = _spec(row)
    x, codes, cb = make_problem(spec, seed=2, device=DEV)
    auto = cabi.select_variant_b(spec.M, spec.K, spec.N, spec.vec, spec.entries, spec.n_codebooks, spec.code_bits)
    _say("e2e_gemm_b", spec, "auto ->", cabi.VARIANT_NAMES[auto])
    ran = []
    for variant in (cabi.VARIANT_AUTO, cabi.VARIANT_GENERIC, cabi.VARIANT_DECODE, cabi.VARIANT_PREFILL,
                    cabi.VARIANT_PREFILL_NARROW, cabi.VARIANT_PREFILL_SMALL, cabi.VARIANT_TWOPASS):
        _say("  variant", cabi.VARIANT_NAMES[variant])
        try:
            y = cabi.e2e_gemm_b(x, codes, cb, variant=variant)
        except cabi.VqGemmError as e:
            assert e.code == -4, e          # "variant cannot serve this shape" is the only accepted refusal
            assert variant in (cabi.VARIANT_DECODE, cabi.VARIANT_PREFILL, cabi.VARIANT_PREFILL_NARROW,
                               cabi.VARIANT_PREFILL_SMALL)
            continue
        torch.cuda.synchronize()
        _check_gemm(y, x, codes, cb, what=f"{spec.name}/{cabi.VARIANT_NAMES[variant]}")
        ran.append(variant)
    assert cabi.VARIANT_AUTO in ran and cabi.VARIANT_GENERIC in ran and cabi.VARIANT_TWOPASS in ran
    if spec.M <= 64 and spec.vec in (2, 4, 8):
        assert cabi.VARIANT_DECODE in ran


@pytest.mark.parametrize("variant", [cabi.VARIANT_DECODE, cabi.VARIANT_PREFILL, cabi.VARIANT_PREFILL_NARROW,
                                     cabi.VARIANT_PREFILL_SMALL, cabi.VARIANT_GENERIC])
@pytest.mark.parametrize("vec,bits,E", [(8, 8, 256), (4, 16, 4096), (4, 8, 256), (8, 16, 512)])
def test_one_hot_activations_return_weight_columns_bit_exactly(variant, vec, bits, E):
    """X = rows of the identity: Y[m,:] must equal W[:,m] exactly (1.0*w + zeros is exact), which
    checks the gather, the MFMA operand layout and the K permutation through the real kernels."""
    K, N, G = 1024, 96, 2
    spec = ProblemSpec("onehot", GEOM_B, 16, K, N, vec, E, G, bits, codebook_3d=True)
    _, codes, cb = make_problem(spec, seed=3, device=DEV)
    w = vo.dequant_b(_np(codes), _np(cb))
    for k0 in (0, 496, K - 16):
        _say("one-hot", cabi.VARIANT_NAMES[variant], vec, bits, "k0", k0)
        x = torch.zeros(16, K, dtype=torch.float16, device=DEV)
        x[torch.arange(16), k0 + torch.arange(16)] = 1.0
        try:
            y = cabi.e2e_gemm_b(x, codes, cb, variant=variant)
        except cabi.VqGemmError as e:
            assert variant == cabi.VARIANT_PREFILL_NARROW and e.code == -4 and E * vec * 2 >= 32768
            pytest.skip("codebooks too large for the narrow tile")
        torch.cuda.synchronize()
        assert np.array_equal(_np(y).view(np.uint16), w[:, k0:k0 + 16].T.copy().view(np.uint16))


# Shapes that give a workgroup of the batched decode kernel several tiles (full batches, short
# last batches, replicated and plain codebooks, every batch size), sized for a 256-CU device.
BATCHED_B = [
    # name, M, K, N, vec, E, bits
    ("u8v8_m1_7_tiles", 1, 4096, 28672, 8, 256, 8),
    ("u8v8_m16_9_tiles", 16, 4096, 36864, 8, 256, 8),
    ("u8v8_m5_k1024", 5, 1024, 40960, 8, 256, 8),
    ("u8v8_m3_e100", 3, 4096, 8192, 8, 100, 8),
    ("u16v8_m3_k2048", 3, 2048, 20480, 8, 300, 16),
    ("u8v4_m2", 2, 4096, 16384, 4, 256, 8),
    ("u8v2_m16_k512", 16, 512, 16384, 2, 256, 8),
    ("u16v4_m9_e4096", 9, 4096, 12288, 4, 4096, 16),
    # taller X: the 16-row slabs are a grid dimension of the same launch
    ("u8v8_m100_slabs", 100, 1024, 4096, 8, 256, 8),
    ("u16v4_m200_slabs", 200, 2048, 2048, 4, 4096, 16),
    ("u8v8_m300_slabs", 300, 4096, 4096, 8, 256, 8),
    # several codebooks: every workgroup works inside the rows of one
    ("u8v8_m130_32_codebooks", 130, 4096, 4096, 8, 256, 8, 32),
    ("u8v8_m2_7_codebooks", 2, 2048, 28672, 8, 256, 8, 7),
    ("u16v4_m40_4_codebooks", 40, 1024, 8192, 4, 1024, 16, 4),
    # K beyond 16 slices of 256: chunks of K, sums carried in the LDS (uneven chunks: 43 = 15+14+14 slices)
    ("u8v8_m1_k8192", 1, 8192, 8192, 8, 256, 8),
    ("u8v8_m16_k11008", 16, 11008, 4096, 8, 256, 8),
    ("u8v8_m40_k14336_4_codebooks", 40, 14336, 2048, 8, 256, 8, 4),
    ("u16v4_m3_k6144", 3, 6144, 12288, 4, 4096, 16),
    ("u8v8_m200_k8192", 200, 8192, 4096, 8, 256, 8),
    ("u8v8_m1_k28672", 1, 28672, 8192, 8, 256, 8),
]


@pytest.fixture
def batched_kernel_for_long_k():
    """The K-sliced path with its streaming kernel switched off: long K goes through the batched kernel's chunks."""
    before = {k: cabi.tuning()[k] for k in ("decode_stream_min_k", "decode_stream_min_k_few_rows")}
    cabi.set_tuning(decode_stream_min_k=1e8, decode_stream_min_k_few_rows=1e8)
    yield
    cabi.set_tuning(**before)


@pytest.mark.parametrize("row", BATCHED_B, ids=[r[0] for r in BATCHED_B])
def test_batched_decode_kernel_with_many_tiles_per_workgroup(row, batched_kernel_for_long_k):
    name, M, K, N, v, E, bits = row[:7]
    G = row[7] if len(row) > 7 else 1
    spec = ProblemSpec(name, GEOM_B, M, K, N, v, E, G, bits, codebook_3d=(G > 1))
    x, codes, cb = make_problem(spec, seed=21, device=DEV)
    _say("batched decode", spec)
    # (the automatic choice: this kernel, or the GEMV kernel for a short run with one row of X)
    assert cabi.select_variant_b(M, K, N, v, E, G, bits) in (cabi.VARIANT_DECODE, cabi.VARIANT_DECODE_GEMV)
    y = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE)
    torch.cuda.synchronize()
    w = vo.dequant_b(_np(codes), _np(cb))
    xf = _np(x).astype(np.float64)
    ref = np.concatenate([xf @ w[r:r + 4096].astype(np.float64).T for r in range(0, N, 4096)], axis=1)
    e1, e2 = vo.rel_err(_np(y), ref)
    _say(f"  {name}: rel_err(floor)={e1:.3e} max/max={e2:.3e}")
    assert e1 <= TOL
    # a permuted one-hot X reads W out bit for bit through the same kernel
    eye = torch.zeros(M, K, dtype=torch.float16, device=DEV)
    cols = [(37 * m + 11) % K for m in range(M)]
    for m, c in enumerate(cols):
        eye[m, c] = 1.0
    yw = cabi.e2e_gemm_b(eye, codes, cb, variant=cabi.VARIANT_DECODE)
    assert np.array_equal(_np(yw).view(np.uint16), w[:, cols].T.copy().view(np.uint16))
    assert torch.equal(cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE), y)
    # The same through the packed code matrix: the re-layout against the oracle's, the GEMM bit for
    # bit the plain layout's (same arithmetic in the same order), W read back through a one-hot X.
    assert cabi.decode_packed_supports(M, K, N, v, E, G, bits)
    packed = cabi.pack_codes_b(codes, v)
    assert np.array_equal(_np(packed), vo.pack_codes_b(_np(codes), v))
    assert torch.equal(cabi.pack_codes_b(packed, v, inverse=True), codes)
    yp = cabi.e2e_gemm_b(x, packed, cb, variant=cabi.VARIANT_DECODE_PACKED)
    assert torch.equal(yp, y)
    ywp = cabi.e2e_gemm_b(eye, packed, cb, variant=cabi.VARIANT_DECODE_PACKED)
    assert np.array_equal(_np(ywp).view(np.uint16), w[:, cols].T.copy().view(np.uint16))


# The streaming kernel of the K-sliced path (whole K per workgroup, K dealt to the waves in pieces of 128): one to seven
# tiles per group, ragged last groups, fewer groups than compute units and several per workgroup, codebooks that change
# between a workgroup's groups, tall X in slabs, K of fewer pieces than a workgroup has waves, short codebooks.
STREAM_B = [
    # name, M, K, N, E, G
    ("down_projection_m16", 16, 14336, 4096, 256, 1),
    ("down_projection_m4_k11008", 4, 11008, 4096, 256, 1),
    ("six_tiles_per_group", 16, 8192, 24576, 256, 1),
    ("seven_tiles_per_group", 12, 4096, 28672, 256, 1),
    ("three_tiles_ragged_last_group", 3, 4096, 11008, 256, 1),
    ("two_tiles_16_codebooks_slabs", 40, 8192, 8192, 256, 16),
    ("few_tiles_17_pieces", 1, 2176, 256, 256, 1),
    ("one_piece", 7, 128, 64, 77, 1),
    ("two_groups_per_workgroup_books_change", 9, 2048, 16 * 8 * 300, 200, 50),
    ("m64_four_slabs", 64, 5120, 2048, 256, 2),
    ("fourteen_pieces_per_wave", 5, 28672, 8192, 256, 1),
]


@pytest.mark.parametrize("row", STREAM_B, ids=[r[0] for r in STREAM_B])
def test_streaming_decode_kernel(row):
    name, M, K, N, E, G = row
    spec = ProblemSpec(name, GEOM_B, M, K, N, 8, E, G, 8, codebook_3d=(G > 1))
    x, codes, cb = make_problem(spec, seed=23, device=DEV)
    _say("streaming decode", spec)
    before = cabi.tuning()
    try:
        for gathers in (0.0, 1e8):   # the bank-replicated table, the plain table
            cabi.set_tuning(decode_stream_min_k=0.0, decode_stream_min_k_few_rows=0.0, decode_stream_min_m=0.0, decode_stream_max_m=1e8, decode_stream_max_groups_per_unit=1e8,
                            decode_stream_replicated_min_gathers=gathers)
            y = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE)
            torch.cuda.synchronize()
            w = vo.dequant_b(_np(codes), _np(cb))
            xf = _np(x).astype(np.float64)
            ref = np.concatenate([xf @ w[r:r + 4096].astype(np.float64).T for r in range(0, N, 4096)], axis=1)
            e1, e2 = vo.rel_err(_np(y), ref)
            _say(f"  {name}: rel_err(floor)={e1:.3e} max/max={e2:.3e}")
            assert e1 <= TOL
            # a permuted one-hot X reads W out bit for bit
            eye = torch.zeros(M, K, dtype=torch.float16, device=DEV)
            cols = [(37 * m + 11) % K for m in range(M)]
            for m, c in enumerate(cols):
                eye[m, c] = 1.0
            yw = cabi.e2e_gemm_b(eye, codes, cb, variant=cabi.VARIANT_DECODE)
            assert np.array_equal(_np(yw).view(np.uint16), w[:, cols].T.copy().view(np.uint16))
            for _ in range(5):
                assert torch.equal(cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE), y)
            bias = torch.randn(N, device=DEV).half()
            yb = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE, bias=bias)
            eb, _ = vo.rel_err(_np(yb), ref + _np(bias).astype(np.float64))
            assert eb <= TOL
        # the batched kernel on the same inputs: the same product within the bar
        cabi.set_tuning(decode_stream_min_k=1e8, decode_stream_min_k_few_rows=1e8)
        if K % 256 == 0:
            yd = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE)
            scale = yd.float().abs().max().item()
            assert ((y.float() - yd.float()).abs().max() / scale).item() <= TOL
    finally:
        cabi.set_tuning(**before)


@pytest.mark.parametrize("M,K,N,v,E,bits,G", [(16, 4096, 11008, 4, 4096, 16, 1), (16, 4096, 4096, 8, 256, 8, 1),
                                              (5, 8192, 2048, 8, 256, 8, 4), (40, 2048, 1536, 4, 256, 8, 2)])
def test_batched_decode_kernel_gives_the_same_bits_on_every_launch(M, K, N, v, E, bits, G):
    # The batched kernel keeps codes and gathered codewords in registers that the hardware is still writing while the
    # wave runs on, and waits for them by count: a count that does not match the order of issue, or a register the
    # compiler moved in that window, shows as a rare wrong element, not as a steady error.  C3 itself, one tile per
    # workgroup, chunked K with several codebooks, and two slabs of X: 40 launches each on fixed operands, back to back
    # and one at a time, every result equal to the first bit for bit; the first against the oracle.
    spec = ProblemSpec("steady", GEOM_B, M, K, N, v, E, G, bits, codebook_3d=(G > 1))
    x, codes, cb = make_problem(spec, seed=91, device=DEV)
    _say("batched decode, 40 launches", M, K, N, v, E, bits, G)
    first = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE).clone()
    torch.cuda.synchronize()
    _check_gemm(first, x, codes, cb, what="first launch")
    outs = [cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE) for _ in range(20)]
    torch.cuda.synchronize()
    for i, y in enumerate(outs):
        assert torch.equal(y, first), f"launch {i} differs"
    for i in range(20):
        y = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE)
        torch.cuda.synchronize()
        assert torch.equal(y, first), f"synchronised launch {i} differs"


def test_packed_codes_small_shapes_bias_and_rejections():
    for (M, K, N, v, E, G, bits) in [(1, 256, 16, 8, 256, 1, 8), (5, 512, 48, 4, 4096, 1, 16), (16, 256, 32, 2, 256, 2, 8),
                                     (33, 1024, 64, 8, 300, 4, 16), (3, 768, 32, 2, 1000, 1, 16), (16, 4096, 4096, 8, 256, 1, 8)]:
        spec = ProblemSpec("packed", GEOM_B, M, K, N, v, E, G, bits, codebook_3d=(G > 1))
        x, codes, cb = make_problem(spec, seed=5, device=DEV)
        _say("packed decode", spec)
        packed = cabi.pack_codes_b(codes, v)
        assert np.array_equal(_np(packed), vo.pack_codes_b(_np(codes), v))
        bias = torch.randn(N, device=DEV).half()
        y = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE, bias=bias)
        yp = cabi.e2e_gemm_b(x, packed, cb, variant=cabi.VARIANT_DECODE_PACKED, bias=bias)
        assert torch.equal(yp, y)
        # the unrounded product in float64 (the oracle's own GEMM returns it rounded to fp16)
        ref = _np(x).astype(np.float64) @ vo.dequant_b(_np(codes), _np(cb)).astype(np.float64).T + _np(bias).astype(np.float64)
        e1, _ = vo.rel_err(_np(yp), ref)
        assert e1 <= TOL
    # shapes outside the batched kernel: no packed layout, and the packed variant refuses them
    codes = torch.zeros(16, 40, dtype=torch.uint8, device=DEV)          # K = 320
    with pytest.raises(cabi.VqGemmError) as ei:
        cabi.pack_codes_b(codes, 8)
    assert ei.value.code == -4
    assert not cabi.decode_packed_supports(4, 320, 16, 8, 256, 1, 8)
    assert not cabi.decode_packed_supports(4, 512, 24, 8, 256, 1, 8)    # N not a multiple of 16
    x = torch.zeros(4, 320, dtype=torch.float16, device=DEV)
    cb = torch.zeros(256, 8, dtype=torch.float16, device=DEV)
    with pytest.raises(cabi.VqGemmError) as ei:
        cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE_PACKED)
    assert ei.value.code == -4
    with pytest.raises(cabi.VqGemmError):                                # not in place
        c2 = torch.zeros(16, 32, dtype=torch.uint8, device=DEV)
        cabi.pack_codes_b(c2, 8, out=c2)
    # the automatic choice never takes the packed variant
    assert cabi.select_variant_b(1, 4096, 4096, 8, 256, 1, 8) == cabi.VARIANT_DECODE_GEMV
    assert cabi.select_variant_b(16, 4096, 4096, 8, 256, 1, 8) == cabi.VARIANT_DECODE
    assert cabi.select_variant_b(2, 4096, 4096, 8, 256, 1, 8) == cabi.VARIANT_DECODE_GEMV
    assert cabi.select_variant_b(3, 4096, 4096, 8, 256, 1, 8) == cabi.VARIANT_DECODE
    assert cabi.select_variant_b(2, 4096, 28672, 8, 256, 1, 8) == cabi.VARIANT_DECODE_GEMV   # two rows of X: the wide form ...
    assert cabi.select_variant_b(2, 4096, 65536, 8, 256, 1, 8) == cabi.VARIANT_DECODE        # ... up to eleven rows per wave at K = 4096
    assert cabi.select_variant_b(2, 8192, 28672, 8, 256, 1, 8) == cabi.VARIANT_DECODE_GEMV   # ... nine at K = 8192
    assert cabi.select_variant_b(2, 8192, 49152, 8, 256, 1, 8) == cabi.VARIANT_DECODE
    assert cabi.select_variant_b(2, 8192, 8192, 8, 256, 1, 8) == cabi.VARIANT_DECODE_GEMV
    assert cabi.select_variant_b(2, 14336, 4096, 8, 256, 1, 8) == cabi.VARIANT_DECODE_GEMV
    assert cabi.select_variant_b(1, 4096, 32768, 8, 256, 1, 8) == cabi.VARIANT_DECODE_GEMV
    assert cabi.select_variant_b(1, 4096, 131072, 8, 256, 1, 8) == cabi.VARIANT_DECODE_GEMV
    assert cabi.select_variant_b(1, 4096, 32768, 8, 256, 2, 8) == cabi.VARIANT_DECODE_GEMV
    assert cabi.select_variant_b(1, 4096, 64 * 16 * 256 + 16, 8, 256, 1, 8) == cabi.VARIANT_DECODE   # more than 64 rows per wave
    assert cabi.select_variant_b(1, 4096, 32768, 4, 256, 1, 8) == cabi.VARIANT_DECODE               # other code formats
    assert cabi.pack_codes_b(torch.zeros(0, 64, dtype=torch.uint8, device=DEV), 8).shape == (0, 64)


GEMV_B = [
    # name, K, N, E, G, M
    ("one_run", 2048, 64, 256, 1, 1),
    ("c2", 4096, 4096, 256, 1, 1),
    ("few_entries_4_books", 4096, 4096, 100, 4, 1),
    ("three_runs_2_books", 6144, 1024, 256, 2, 1),
    ("four_runs", 8192, 2048, 256, 1, 1),
    ("16_row_books", 2048, 256, 256, 16, 1),
    ("many_tiles", 4096, 32768, 256, 1, 1),
    ("many_tiles_two_books", 4096, 32768, 256, 2, 1),
    # the wide form (one row of X from one row per wave on): rows that do not divide by anything, workgroups whose
    # rows reach into a second codebook (two tables), small codebooks, short codebooks
    ("wide_ragged_n", 4096, 5003, 256, 1, 1),
    ("wide_three_books_straddled", 2048, 12288, 256, 3, 1),
    ("wide_128_row_books_straddled", 4096, 6144, 256, 48, 1),
    ("wide_128_row_books_aligned", 2048, 8192, 200, 64, 1),
    ("wide_four_runs_two_books", 8192, 4096 + 32, 256, 2, 1),
    # the wide form on its plain table (a wave's rows are at most two runs of 2048 k): two tables, short codebooks, ragged rows
    ("wide_plain_table_books_straddled", 2048, 3 * 2000, 256, 3, 1),
    ("wide_plain_table_short_books", 4096, 4096, 77, 4, 1),
    ("wide_plain_table_ragged", 2048, 7001, 256, 1, 1),
    # no wave with more than one row: the single-group instance (codebooks that workgroups straddle, waves without a row,
    # the replicated table at three runs)
    ("wide_single_group_three_books_straddled", 4096, 3 * 1008, 200, 3, 1),
    ("wide_single_group_three_runs", 6144, 4096 - 7, 256, 1, 1),
    ("many_tiles_three_runs_ragged_walk", 6144, 16 * 1500, 256, 1, 1),
    ("many_tiles_one_run", 2048, 65536, 77, 1, 1),
    # the wide form's long rows (K beyond 8192, or no multiple of 2048), worked through in pieces of three or four runs:
    # a last piece that is partly or wholly padding, one to three rows per wave, several codebooks, the longest K
    ("long_k_11008_down_projection", 11008, 4096, 256, 1, 1),
    ("long_k_14336_down_projection", 14336, 4096, 256, 1, 1),
    ("long_k_28672_five_pieces", 28672, 2304, 256, 1, 1),
    ("long_k_16384_128_row_books", 16384, 4096, 200, 32, 1),
    ("long_k_2208_one_piece_ragged_n", 2208, 5003, 256, 1, 1),
    ("long_k_32768_longest", 32768, 2048 + 16, 77, 1, 1),
    ("long_k_10240_three_rows_per_wave_ragged", 10240, 9001, 256, 1, 1),
    ("long_k_12288_two_books", 12288, 8192, 256, 2, 1),
    ("two_rows_of_x", 4096, 4096, 256, 1, 2),
    # two rows of X in the wide form (K up to 4096): ragged N, codebooks that workgroups straddle, the single-group
    # instance with waves without a row, seven rows per wave in groups of two, one run
    ("wide_two_rows_of_x_ragged", 4096, 5003, 256, 1, 2),
    ("wide_two_rows_three_books_straddled", 2048, 12288, 256, 3, 2),
    ("wide_two_rows_single_group", 4096, 4096 - 7, 200, 1, 2),
    ("wide_two_rows_many_tiles", 4096, 28672, 256, 1, 2),
    ("wide_two_rows_one_run_two_books", 2048, 2 * 9008, 77, 2, 2),
    # ... and beyond K = 4096 in pieces of two runs: a last piece that is partly padding, several codebooks, the longest K
    ("wide_two_rows_long_k_8192_ragged", 8192, 5003, 200, 1, 2),
    ("wide_two_rows_long_k_14336_down_projection", 14336, 4096, 256, 1, 2),
    ("wide_two_rows_long_k_4128_padded_piece", 4128, 3000, 256, 1, 2),
    ("wide_two_rows_long_k_12288_two_books", 12288, 8192, 256, 2, 2),
    ("wide_two_rows_long_k_16384_longest", 16384, 2048 + 16, 77, 1, 2),
    ("two_rows_four_runs", 8192, 512, 256, 2, 2),
    ("three_rows", 2048, 1024, 256, 1, 3),
    ("four_rows_two_runs", 4096, 1024, 200, 4, 4),
]


@pytest.mark.parametrize("row", GEMV_B, ids=[r[0] for r in GEMV_B])
def test_gemv_kernel_few_rows_of_x(row):
    name, K, N, E, G, M = row
    spec = ProblemSpec(name, GEOM_B, M, K, N, 8, E, G, 8, codebook_3d=(G > 1))
    x, codes, cb = make_problem(spec, seed=31, device=DEV)
    _say("gemv", spec)
    y = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE_GEMV)
    torch.cuda.synchronize()
    _check_gemm(y, x, codes, cb, what=name)
    # one-hot x reads a column of W out bit for bit (fp16 subnormals included: nothing is flushed)
    w = vo.dequant_b(_np(codes), _np(cb))
    for col in (0, 7, K // 2 + 3, K - 1):
        eye = torch.zeros(M, K, dtype=torch.float16, device=DEV)
        cols = [(col + 41 * m) % K for m in range(M)]
        for m, c in enumerate(cols):
            eye[m, c] = 1.0
        yw = cabi.e2e_gemm_b(eye, codes, cb, variant=cabi.VARIANT_DECODE_GEMV)
        assert np.array_equal(_np(yw).view(np.uint16), w[:, cols].T.copy().view(np.uint16))
    bias = torch.randn(N, device=DEV).half()
    yb = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE_GEMV, bias=bias)
    ref = _np(x).astype(np.float64) @ w.astype(np.float64).T + _np(bias).astype(np.float64)
    e1, _ = vo.rel_err(_np(yb), ref)
    assert e1 <= TOL
    for _ in range(4):
        assert torch.equal(cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE_GEMV), y)
    # one or two rows of X go to the wide form at any N; the four-wave kernel takes the same launch when the wide form is
    # switched off: same product within the bar, a column of W bit for bit
    if M <= 2 and K % 2048 == 0 and K <= 8192 and N % 16 == 0 and N <= 4096:
        before = cabi.tuning()["gemv_wide_min_rows_per_wave"]
        cabi.set_tuning(gemv_wide_min_rows_per_wave=1e6)
        try:
            _check_gemm(cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE_GEMV), x, codes, cb, what=name + " (four-wave)")
            yw = cabi.e2e_gemm_b(eye, codes, cb, variant=cabi.VARIANT_DECODE_GEMV)
            assert np.array_equal(_np(yw).view(np.uint16), w[:, cols].T.copy().view(np.uint16))
        finally:
            cabi.set_tuning(gemv_wide_min_rows_per_wave=before)
    # the K-sliced MFMA kernel and the automatic choice on the same inputs: same product within the bar
    if K % 64 == 0:   # (the K-sliced kernels take K in whole matrix-core steps)
        _check_gemm(cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE), x, codes, cb, what=name + " (decode)")
    _check_gemm(cabi.e2e_gemm_b(x, codes, cb), x, codes, cb, what=name + " (auto)")


def test_gemv_wide_form_at_its_longest_64_rows_per_wave():
    """As many rows as the wide form takes: one result per lane, 63 or 64 rows per wave on a 256-CU device.  The oracle
    multiplies a sample of the rows (rows are independent): the first and last rows and a few thousand others."""
    K, N = 2048, 64 * 16 * 256 - 777
    spec = ProblemSpec("wide_longest", GEOM_B, 1, K, N, 8, 256, 1, 8)
    x, codes, cb = make_problem(spec, seed=33, device=DEV)
    _say("gemv wide, long", spec)
    y = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE_GEMV)
    torch.cuda.synchronize()
    rng = np.random.default_rng(5)
    rows = np.unique(np.concatenate([np.arange(0, 400), np.arange(N - 400, N), rng.integers(0, N, 4000)]))
    ref = vo.vq_gemm_b(_np(x), _np(codes)[rows], _np(cb), acc=np.float64)
    e1, e2 = vo.rel_err(_np(y)[:, rows], ref)
    _say(f"  sampled rows: rel_err(floor)={e1:.3e} max/max={e2:.3e}")
    assert e1 <= TOL
    # every row against the K-sliced MFMA kernel (pinned against the oracle elsewhere)
    yd = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE)
    scale = yd.float().abs().max().item()
    assert ((y.float() - yd.float()).abs().max() / scale).item() <= TOL
    assert torch.equal(cabi.e2e_gemm_b(x, codes, cb), y)   # the automatic choice is this kernel, and it is deterministic
    # one row more per wave than it takes, in a shape the four-wave kernel refuses as well (N not a multiple of 16)
    n_big = 64 * 16 * 256 + 8
    with pytest.raises(cabi.VqGemmError) as ei:
        cabi.e2e_gemm_b(x, torch.zeros(n_big, K // 8, dtype=torch.uint8, device=DEV), cb, variant=cabi.VARIANT_DECODE_GEMV)
    assert ei.value.code == -4


GEMV_FORMATS = [
    # name, M, K, N, vec, E, bits, G
    ("v4_u16_e4096_c3_weights", 1, 4096, 11008, 4, 4096, 16, 1),
    ("v4_u16_two_rows_two_books", 2, 2048, 256, 4, 1000, 16, 2),
    ("v4_u8", 1, 4096, 1024, 4, 256, 8, 1),
    ("v4_u8_three_runs_two_rows", 2, 6144, 512, 4, 100, 8, 4),
    ("v8_u16_e4096", 1, 4096, 512, 8, 4096, 16, 1),
    ("v8_u16_four_runs", 1, 8192, 256, 8, 333, 16, 1),
    ("v2_u8", 1, 2048, 1024, 2, 256, 8, 1),
    ("v2_u8_two_rows", 2, 4096, 256, 2, 200, 8, 2),
]


@pytest.mark.parametrize("row", GEMV_FORMATS, ids=[r[0] for r in GEMV_FORMATS])
def test_gemv_kernel_code_formats(row):
    name, M, K, N, v, E, bits, G = row
    spec = ProblemSpec(name, GEOM_B, M, K, N, v, E, G, bits, codebook_3d=(G > 1))
    x, codes, cb = make_problem(spec, seed=37, device=DEV)
    _say("gemv format", spec)
    y = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE_GEMV)
    torch.cuda.synchronize()
    _check_gemm(y, x, codes, cb, what=name)
    w = vo.dequant_b(_np(codes), _np(cb))
    for col in (0, 3, K // 2 + 5, K - 1):
        eye = torch.zeros(M, K, dtype=torch.float16, device=DEV)
        cols = [(col + 29 * m) % K for m in range(M)]
        for m, c in enumerate(cols):
            eye[m, c] = 1.0
        yw = cabi.e2e_gemm_b(eye, codes, cb, variant=cabi.VARIANT_DECODE_GEMV)
        assert np.array_equal(_np(yw).view(np.uint16), w[:, cols].T.copy().view(np.uint16))
    assert torch.equal(cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE_GEMV), y)
    _check_gemm(cabi.e2e_gemm_b(x, codes, cb), x, codes, cb, what=name + " (auto)")


def test_gemv_kernel_refuses_other_shapes():
    cb = torch.zeros(256, 8, dtype=torch.float16, device=DEV)
    for (M, K, N, v, bits) in [(5, 2048, 64, 8, 8), (4, 6144, 64, 8, 8), (1, 1024, 64, 8, 8), (1, 2056, 64, 8, 8), (1, 34816, 64, 8, 8), (3, 2048, 24, 8, 8), (2, 18432, 24, 8, 8),
                               (1, 2048, 64, 2, 16), (3, 2048, 64, 4, 8)]:
        x = torch.zeros(M, K, dtype=torch.float16, device=DEV)
        codes = torch.zeros(N, K // v, dtype=torch.uint8 if bits == 8 else torch.uint16, device=DEV)
        c = cb if v == 8 else torch.zeros(256, v, dtype=torch.float16, device=DEV)
        with pytest.raises(cabi.VqGemmError) as ei:
            cabi.e2e_gemm_b(x, codes, c, variant=cabi.VARIANT_DECODE_GEMV)
        assert ei.value.code == -4


def test_gemv_kernel_one_row_of_x_small_launches_in_the_long_form():
    """One row of X with a K or an N that the four-wave kernel does not take goes to the wide form at any size: K no whole
    number of runs, K beyond 8192, N no multiple of 16, on launches far smaller than the device."""
    for (K, N, E, G) in [(2080, 64, 256, 1), (10240, 64, 256, 1), (2048, 24, 100, 1), (6144, 8, 256, 1), (4096, 40, 256, 2)]:
        spec = ProblemSpec(f"small_k{K}_n{N}", GEOM_B, 1, K, N, 8, E, G, 8, codebook_3d=(G > 1))
        x, codes, cb = make_problem(spec, seed=77, device=DEV)
        _say("gemv small", spec)
        y = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE_GEMV)
        torch.cuda.synchronize()
        _check_gemm(y, x, codes, cb, what=spec.name)
        _check_gemm(cabi.e2e_gemm_b(x, codes, cb), x, codes, cb, what=spec.name + " (auto)")


# Shapes that walk the prefill kernel through each of its instantiations: both super-stage
# lengths (one or two 64-k stages per code tile), one or two 16-byte code chunks per row, a last
# stage of 32 k, four, three and two X buffers (large codebooks), several codebooks per 256-row
# tile (aligned and not), ragged M and N, fewer stages than the pipeline is deep.
PREFILL_B = [
    # name, M, K, N, vec, E, bits, G
    ("u8v8_one_super", 256, 128, 256, 8, 256, 8, 1),
    ("u8v8_odd_supers_2_books_per_tile", 256, 384, 256, 8, 256, 8, 2),
    ("u8v8_ragged_5_books", 1000, 1152, 1000, 8, 256, 8, 5),
    ("u8v8_n_not_mult_of_8", 513, 1024, 1001, 8, 256, 8, 1),
    ("u8v8_k11008_32_books", 600, 11008, 1024, 8, 256, 8, 32),
    ("u16v8_k_odd_stages", 512, 1088, 512, 8, 1024, 16, 2),
    ("u8v4", 512, 1088, 768, 4, 256, 8, 3),
    ("u16v4_e4096_three_buffers", 512, 1024, 512, 4, 4096, 16, 1),
    ("u16v4_e4096_tail32", 512, 1056, 512, 4, 4096, 16, 1),
    ("u16v4_e4096_two_books_two_buffers", 300, 1056, 96, 4, 4096, 16, 2),
    ("u8v2_tail32_ragged_n", 512, 1056, 520, 2, 256, 8, 1),
    ("u8v2_k32_only_a_tail", 260, 32, 264, 2, 256, 8, 1),
    ("u8v8_many_tiles", 2048, 2048, 4096, 8, 256, 8, 16),
    # more 256x256 tiles than a 256-CU device has units: whole rounds of them, the left-over columns in 256x128 tiles
    ("u8v8_rounds_and_a_narrow_tail", 2048, 256, 8704, 8, 256, 8, 17),
    # medium M: 128x128 tiles (the automatic choice here); ragged M and N, codebook changes inside a tile
    ("u8v8_medium_m", 640, 2048, 2048, 8, 256, 8, 1),
    ("u16v8_medium_m_ragged", 300, 1024, 1000, 8, 1000, 16, 5),
    ("u8v4_medium_m_24_row_books", 200, 512, 240, 4, 256, 8, 10),
    ("u8v2_medium_m", 129, 256, 136, 2, 256, 8, 1),
]


@pytest.mark.parametrize("variant", [cabi.VARIANT_PREFILL, cabi.VARIANT_PREFILL_NARROW, cabi.VARIANT_PREFILL_SMALL])
@pytest.mark.parametrize("row", PREFILL_B, ids=[r[0] for r in PREFILL_B])
def test_prefill_kernel_instantiations(row, variant):
    name, M, K, N, v, E, bits, G = row
    spec = ProblemSpec(name, GEOM_B, M, K, N, v, E, G, bits, codebook_3d=(G > 1))
    x, codes, cb = make_problem(spec, seed=33, device=DEV)
    _say("prefill", cabi.VARIANT_NAMES[variant], spec)
    try:
        y = cabi.e2e_gemm_b(x, codes, cb, variant=variant)
    except cabi.VqGemmError as e:
        assert e.code == -4
        if variant == cabi.VARIANT_PREFILL_SMALL:
            # the 128x128 tile wants K in whole code tiles (64 k, 128 k for 8-vectors with 8-bit codes)
            assert K % (128 if (v, bits) == (8, 8) else 64) != 0
            pytest.skip("K is not a whole number of code tiles")
        # the 256x128 tile keeps four X buffers and does not take the largest codebooks (or several large ones)
        assert variant == cabi.VARIANT_PREFILL_NARROW and E * v * 2 * min(G, 3) >= 32768
        pytest.skip("codebooks too large for the narrow tile")
    torch.cuda.synchronize()
    w = vo.dequant_b(_np(codes), _np(cb))
    ref = _np(x).astype(np.float64) @ w.astype(np.float64).T
    e1, e2 = vo.rel_err(_np(y), ref)
    _say(f"  {name}: rel_err(floor)={e1:.3e} max/max={e2:.3e}")
    assert e1 <= TOL
    # a permuted one-hot X reads W out bit for bit through the same kernel
    eye = torch.zeros(M, K, dtype=torch.float16, device=DEV)
    cols = [(37 * m + 11) % K for m in range(M)]
    eye[torch.arange(M), torch.tensor(cols)] = 1.0
    yw = cabi.e2e_gemm_b(eye, codes, cb, variant=variant)
    assert np.array_equal(_np(yw).view(np.uint16), w[:, cols].T.copy().view(np.uint16))
    assert torch.equal(cabi.e2e_gemm_b(x, codes, cb, variant=variant), y)


ENCODE_B = [
    # name, N, K, vec, E, G, bits
    ("u8v8_256", 64, 256, 8, 256, 1, 8),
    ("u16v4_4096_two_books", 96, 128, 4, 4096, 2, 16),
    ("u8v2_100_five_books", 50, 64, 2, 100, 5, 8),
    ("u16v8_5000_chunked_codebook", 40, 64, 8, 5000, 1, 16),
    ("u16v8_e300_ragged_block", 33, 136, 8, 300, 3, 16),
]


@pytest.mark.parametrize("row", ENCODE_B, ids=[r[0] for r in ENCODE_B])
def test_encoder_matches_the_c_oracle_bit_for_bit(row):
    name, N, K, v, E, G, bits = row
    _say("encode", row)
    g = torch.Generator(device="cpu").manual_seed(5)
    cb = torch.randn(G, E, v, generator=g).half()
    w = torch.randn(N, K, generator=g).half()
    # a third of the vectors sit on or next to codebook entries (exact zeros, near-ties)
    pick = torch.randint(0, E, (N, K // v), generator=g)
    near = cb[(torch.arange(N) // (N // G))[:, None], pick].reshape(N, K)
    mask = (torch.rand(N, K // v, generator=g) < 0.33).repeat_interleave(v, dim=1)
    w = torch.where(mask, near, w)
    codes = cabi.encode_b(w.to(DEV), cb.to(DEV), bits)
    torch.cuda.synchronize()
    want = c_oracle.encode_b(w.numpy(), cb.numpy(), bits)
    assert codes.dtype == (torch.uint8 if bits == 8 else torch.uint16)
    assert np.array_equal(_np(codes), want)
    # the codes dequantise (bit-exactly) to what the oracle's codes dequantise to
    assert np.array_equal(_np(cabi.dequant_b(codes, cb.to(DEV))), vo.dequant_b(want, cb.numpy()))


def test_encoder_inverts_the_dequantiser_on_the_gpu():
    spec = ProblemSpec("enc", GEOM_B, 1, 1024, 512, 8, 256, 4, 8, codebook_3d=True, codebook_std=1.0)
    _, codes, cb = make_problem(spec, seed=8, device=DEV)
    assert all(len({tuple(e) for e in _np(cb)[g].tolist()}) == 256 for g in range(4))
    w = cabi.dequant_b(codes, cb)
    assert torch.equal(cabi.encode_b(w, cb, 8), codes)


def test_kmeans_quantiser_feeds_the_gemm_path():
    from vq_gemm_amd.quantize import kmeans_quantize
    g = torch.Generator(device="cpu").manual_seed(9)
    N, K, v, E, G = 512, 1024, 8, 256, 2
    # weights drawn around 64 centres per block: a 256-entry codebook can represent them well
    centres = torch.randn(G, 64, v, generator=g) * 0.05
    which = torch.randint(0, 64, (N, K // v), generator=g)
    w = centres[(torch.arange(N) // (N // G))[:, None], which].reshape(N, K)
    w = (w + torch.randn(N, K, generator=g) * 0.002).half().to(DEV)
    codes, cb, hist = kmeans_quantize(w, v, E, n_codebooks=G, iters=6, seed=1)
    _say("k-means mse per element:", ["%.3e" % h for h in hist])
    assert codes.shape == (N, K // v) and codes.dtype == torch.uint8 and cb.shape == (G, E, v)
    assert hist[-1] <= hist[0] and hist[-1] < 0.2 * float((w.float() ** 2).mean())
    # the returned codes are the nearest entries of the returned codebook
    assert torch.equal(cabi.encode_b(w, cb, 8), codes)
    # and the pair drives the fused GEMM: same result as the oracle on the same codes
    x = torch.randn(32, K, generator=g).half().to(DEV)
    y = cabi.e2e_gemm_b(x, codes, cb)
    torch.cuda.synchronize()
    _check_gemm(y, x, codes, cb, what="quantised weights")


BIAS_B = [
    # name, M, K, N, vec, E, bits, G  -- every kernel with a bias input, ragged and aligned shapes
    ("decode_one_tile", 1, 1024, 64, 8, 256, 8, 1),
    ("decode_batched_many_tiles", 5, 4096, 8192, 8, 256, 8, 1),
    ("decode_batched_chunked_k_books", 40, 8192, 2048, 8, 256, 8, 4),
    ("decode_general_ragged_n", 7, 1024, 50, 8, 256, 8, 1),
    ("decode_slabs_u16v4", 200, 2048, 2048, 4, 4096, 16, 1),
    ("prefill_wide_ragged", 1000, 1152, 1000, 8, 256, 8, 5),
    ("prefill_n_not_mult_of_8", 513, 1024, 1001, 8, 256, 8, 1),
    ("prefill_narrow_choice", 1024, 1024, 1024, 8, 256, 8, 8),
    ("prefill_tail32_v2", 512, 1056, 520, 2, 256, 8, 1),
    ("generic_only_k_odd", 9, 72, 40, 8, 256, 8, 1),
]


@pytest.mark.parametrize("row", BIAS_B, ids=[r[0] for r in BIAS_B])
def test_bias_is_added_before_the_rounding_in_every_kernel(row):
    name, M, K, N, v, E, bits, G = row
    spec = ProblemSpec(name, GEOM_B, M, K, N, v, E, G, bits, codebook_3d=(G > 1))
    x, codes, cb = make_problem(spec, seed=44, device=DEV)
    g = torch.Generator(device="cpu").manual_seed(45)
    bias = torch.randn(N, generator=g).half().to(DEV)
    # the unrounded product in float64 (the oracle's own GEMM returns it rounded to fp16)
    w = vo.dequant_b(_np(codes), _np(cb)).astype(np.float64)
    ref = _np(x).astype(np.float64) @ w.T + _np(bias).astype(np.float64)
    ran = []
    for variant in (cabi.VARIANT_AUTO, cabi.VARIANT_GENERIC, cabi.VARIANT_DECODE, cabi.VARIANT_PREFILL,
                    cabi.VARIANT_PREFILL_NARROW, cabi.VARIANT_PREFILL_SMALL):
        _say("bias", name, cabi.VARIANT_NAMES[variant])
        try:
            y = cabi.e2e_gemm_b(x, codes, cb, variant=variant, bias=bias)
        except cabi.VqGemmError as e:
            assert e.code == -4 and variant not in (cabi.VARIANT_AUTO, cabi.VARIANT_GENERIC), e
            continue
        torch.cuda.synchronize()
        e1, e2 = vo.rel_err(_np(y), ref)
        _say(f"    rel_err(floor)={e1:.3e} max/max={e2:.3e}")
        assert e1 <= TOL, (name, variant, e1)
        # a zero bias changes nothing, bit for bit
        assert torch.equal(cabi.e2e_gemm_b(x, codes, cb, variant=variant, bias=torch.zeros_like(bias)),
                           cabi.e2e_gemm_b(x, codes, cb, variant=variant))
        ran.append(variant)
    assert cabi.VARIANT_AUTO in ran and cabi.VARIANT_GENERIC in ran
    assert len(ran) >= 3 or name.startswith("generic_only")
    # the two-pass route has no bias input and says so
    with pytest.raises(cabi.VqGemmError) as ei:
        cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_TWOPASS, bias=bias)
    assert ei.value.code == -4


def test_vqlinear_module_matches_a_dense_layer_on_its_dequantised_weight():
    from vq_gemm_amd.nn import VQLinear
    g = torch.Generator(device="cpu").manual_seed(12)
    N, K = 768, 512
    w = (torch.randn(N, K, generator=g) * 0.05).half().to(DEV)
    bias = torch.randn(N, generator=g).half().to(DEV)
    layer = VQLinear.from_float(w, vec=8, entries=256, n_codebooks=3, bias=bias, iters=3, seed=2)
    _say(layer)
    assert layer.in_features == K and layer.out_features == N
    for shape in ((5, K), (2, 7, K), (300, K)):
        x = torch.randn(*shape, generator=g).half().to(DEV)
        y = layer(x)
        torch.cuda.synchronize()
        assert y.shape == (*shape[:-1], N) and y.dtype == torch.float16
        wq = _np(layer.dequantized_weight()).astype(np.float64)
        ref = _np(x).astype(np.float64).reshape(-1, K) @ wq.T + _np(bias).astype(np.float64)
        e1, _ = vo.rel_err(_np(y).reshape(-1, N), ref)
        assert e1 <= TOL                 # the bias is added to the fp32 sums: still one rounding
    # the layer survives a state_dict round trip
    clone = VQLinear(torch.zeros_like(layer.codes), torch.zeros_like(layer.codebook), torch.zeros_like(bias))
    clone.load_state_dict(layer.state_dict())
    x = torch.randn(4, K, generator=g).half().to(DEV)
    assert torch.equal(clone(x), layer(x))
    # a second copy of the codes in the decode kernel's order: short inputs read it, same bits out
    packed = VQLinear(layer.codes, layer.codebook, bias).prepack_for_decode()
    assert packed.codes_packed is not None and "codes_packed" not in packed.state_dict()
    for shape in ((1, K), (2, 7, K), (300, K)):
        x = torch.randn(*shape, generator=g).half().to(DEV)
        assert torch.equal(packed(x), layer(x))
    with pytest.raises(ValueError):
        VQLinear(layer.codes[:, :40], layer.codebook).prepack_for_decode()    # K = 320


def test_residual_stages_accumulate_in_one_fused_gemm():
    """Additive quantisation: every stage lowers the error, the merged codes index the merged codebook
    stage by stage, and the layer's one GEMM over [X, X] equals X times the sum of the stage weights."""
    from vq_gemm_amd.nn import VQLinear
    from vq_gemm_amd.quantize import residual_quantize
    g = torch.Generator(device="cpu").manual_seed(21)
    N, K, v = 512, 1024, 8
    w = (torch.randn(N, K, generator=g) * 0.05).half().to(DEV)
    for entries, stages, G, dtype in ((128, 2, 2, torch.uint8), (256, 3, 1, torch.uint16)):
        _say("residual quantiser", entries, stages, G)
        codes, cb, hist = residual_quantize(w, v, entries, stages=stages, n_codebooks=G, iters=3, seed=3)
        _say("    mse per element after each stage:", ["%.3e" % h for h in hist])
        J = K // v
        assert codes.shape == (N, stages * J) and codes.dtype == dtype and cb.shape == (G, stages * entries, v)
        assert all(hist[s + 1] < 0.9 * hist[s] for s in range(stages - 1))
        c = _np(codes).astype(np.int64)
        for s in range(stages):
            blk = c[:, s * J:(s + 1) * J]
            assert blk.min() >= s * entries and blk.max() < (s + 1) * entries
        # the weight: sum over the stages of the oracle's dequantisation of each stage's block
        wd = vo.dequant_b(_np(codes), _np(cb)).astype(np.float64)          # [N, stages*K]
        w_sum = wd.reshape(N, stages, K).sum(axis=1)
        assert float(((w_sum - _np(w).astype(np.float64)) ** 2).mean()) == pytest.approx(hist[-1], rel=1e-3)
        layer = VQLinear(codes, cb, k_repeat=stages)
        assert layer.in_features == K and layer.out_features == N
        assert np.array_equal(_np(layer.dequantized_weight()), w_sum.astype(np.float32).astype(np.float16))
        for M in (1, 16, 300):
            x = torch.randn(M, K, generator=g).half().to(DEV)
            _say("residual layer", entries, stages, M)
            y = layer(x)
            torch.cuda.synchronize()
            e1, _ = vo.rel_err(_np(y), _np(x).astype(np.float64) @ w_sum.T)
            assert e1 <= TOL, (entries, stages, M, e1)
    layer = VQLinear.from_float(w, vec=v, entries=128, iters=2, residual_stages=2)
    assert layer.k_repeat == 2 and layer.codes.shape == (N, 2 * K // v)
    with pytest.raises(ValueError):
        VQLinear(layer.codes, layer.codebook, k_repeat=3)


def test_registered_op_traces_and_matches_eager():
    """torch.ops.vq_gemm_amd.vq_linear: the fake implementation agrees with the device one (opcheck)
    and a layer traced by torch.compile (no code generation: the aot_eager backend) gives the eager result."""
    from vq_gemm_amd.nn import VQLinear
    from vq_gemm_amd import torch_ops  # noqa: F401
    spec = ProblemSpec("op", GEOM_B, 24, 512, 384, 8, 256, 3, 8)
    x, codes, cb = make_problem(spec, seed=13, device=DEV)
    bias = torch.randn(spec.N, generator=torch.Generator().manual_seed(1)).half().to(DEV)
    _say("opcheck vq_linear")
    torch.library.opcheck(torch.ops.vq_gemm_amd.vq_linear.default, (x.view(2, 12, 512), codes, cb, bias),
                          test_utils=("test_schema", "test_faketensor"))
    layer = VQLinear(codes, cb, bias)
    want = layer(x)
    wq = _np(cabi.dequant_b(codes, cb)).astype(np.float64)
    e1, _ = vo.rel_err(_np(want), _np(x).astype(np.float64) @ wq.T + _np(bias).astype(np.float64))
    assert e1 <= TOL, e1
    _say("aot_eager trace")
    traced = torch.compile(layer, backend="aot_eager", fullgraph=True)
    got = traced(x)
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_layer_calls_are_seen_by_subclasses_and_function_modes(monkeypatch):
    """The layers' direct calls step aside for whatever overrides __torch_function__: a mode and a subclass see the registered
    operator, a subclass comes back as one.  A default device is no reason to leave them."""
    from torch.overrides import TorchFunctionMode
    from vq_gemm_amd.nn import VQGatedMLP, VQLinear

    class Sub(torch.Tensor):
        pass

    class Off(torch.Tensor):
        __torch_function__ = torch._C._disabled_torch_function_impl

    class Seen(TorchFunctionMode):
        def __init__(self):
            super().__init__()
            self.names = []

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.names.append(str(func))
            return func(*args, **(kwargs or {}))

    x, codes, cb = make_problem(ProblemSpec("s", GEOM_B, 5, 512, 768, 8, 256, 1, 8), seed=4, device=DEV)
    _, dcodes, _ = make_problem(ProblemSpec("s", GEOM_B, 5, 384, 512, 8, 256, 1, 8), seed=5, device=DEV)
    lin, mlp = VQLinear(codes, cb), VQGatedMLP(VQLinear(codes, cb), VQLinear(dcodes, cb), interleaved=True)
    packed = VQLinear(codes, cb).prepack_for_decode()
    for layer, op in ((lin, "vq_linear"), (packed, "vq_linear"), (mlp, "vq_gated_linear")):
        _say("watched layer calls", op)
        want = layer(x)
        assert type(want) is torch.Tensor and type(layer(x.as_subclass(Off))) is torch.Tensor
        y = layer(x.as_subclass(Sub))
        assert type(y) is Sub and torch.equal(y.as_subclass(torch.Tensor), want)
        with Seen() as mode:
            y = layer(x)
        assert type(y) is torch.Tensor and torch.equal(y, want) and any(op in n for n in mode.names), mode.names
    lin.codes = codes.as_subclass(Sub)
    assert type(lin(x)) is Sub
    lin.codes = codes
    def not_here(x):
        raise AssertionError("a default device sent the layer to the operator")
    monkeypatch.setattr(lin, "_forward_op", not_here)
    with torch.device(DEV):
        assert torch.equal(lin(x), packed(x))
    with Seen() as mode:
        decoded = cabi.dequant_b(codes, cb)
    assert mode.names and torch.equal(decoded, cabi.dequant_b(codes, cb))


def test_random_shapes_agree_across_kernels():
    """Seeded random shapes (ragged M and N, rows per codebook that are no multiple of anything, one
    to many K stages, with and without bias): the scalar kernel and the automatic choice against the
    oracle, and every kernel that accepts a shape against the scalar kernel."""
    import random
    rnd = random.Random(2024)
    done = 0
    for case in range(60):
        v = rnd.choice([2, 4, 8])
        bits = rnd.choice([8, 16])
        E = rnd.choice([16, 100, 256]) if bits == 8 else rnd.choice([300, 1024, 4096])
        kc = (16 // (bits // 8)) * v
        K = kc * rnd.choice([1, 2, 3, 5, 8, 9, 17])
        G = rnd.choice([1, 1, 2, 3, 8])
        N = G * rnd.choice([1, 5, 16, 37, 64, 128, 200, 512])
        M = rnd.choice([1, 3, 16, 17, 100, 255, 257, 600, 1500])
        if N * K > 20_000_000 or M * N > 2_000_000:
            continue
        spec = ProblemSpec("rnd", GEOM_B, M, K, N, v, E, G, bits, codebook_3d=(G > 1))
        x, codes, cb = make_problem(spec, seed=case, device=DEV)
        bias = torch.randn(N, generator=torch.Generator().manual_seed(case)).half().to(DEV) if case % 3 == 0 else None
        _say("random shape", case, spec, "bias" if bias is not None else "")
        y_scalar = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_GENERIC, bias=bias)
        ref = y_scalar.float()
        # the oracle on the same inputs (fp64 sums, the bias added before the one rounding)
        # (the unrounded product in float64: the oracle's own GEMM returns it rounded to fp16)
        want = _np(x).astype(np.float64) @ vo.dequant_b(_np(codes), _np(cb)).astype(np.float64).T
        if bias is not None:
            want = want + _np(bias).astype(np.float64)[None, :]
        e1, _ = vo.rel_err(_np(y_scalar), want)
        assert e1 <= TOL, (case, spec, "scalar kernel against the oracle", e1)
        y_auto = cabi.e2e_gemm_b(x, codes, cb, bias=bias)
        e1, _ = vo.rel_err(_np(y_auto), want)
        assert e1 <= TOL, (case, spec, "automatic choice against the oracle", e1)
        scale = max(ref.abs().max().item(), 1e-3)
        for variant in (cabi.VARIANT_AUTO, cabi.VARIANT_DECODE, cabi.VARIANT_PREFILL, cabi.VARIANT_PREFILL_NARROW,
                        cabi.VARIANT_PREFILL_SMALL):
            try:
                y = cabi.e2e_gemm_b(x, codes, cb, variant=variant, bias=bias)
            except cabi.VqGemmError as e:
                assert e.code == -4 and variant != cabi.VARIANT_AUTO, e
                continue
            torch.cuda.synchronize()
            err = ((y.float() - ref).abs().max() / scale).item()
            assert err <= TOL, (case, spec, cabi.VARIANT_NAMES[variant], err)
        done += 1
    assert done >= 40


def test_random_shapes_gemv_forms_against_the_scalar_kernel():
    """Seeded random launches of one and two rows of X through the GEMV kernels (K in whole runs, in long rows and in
    rows with a padded last piece; one to many codebooks, workgroups that straddle them, short codebooks; plain, with a
    bias and gated) against the scalar kernel of the same library, which the tests above pin to the oracle."""
    import random
    rnd = random.Random(77)
    ran = refused = 0
    for case in range(240):
        M = rnd.choice([1, 1, 2])
        K = rnd.choice([2048, 4096, 4096, 6144, 8192, 10240, 14336, 2208, 4128, 11008, 16384, 28672])
        G = rnd.choice([1, 1, 2, 3, 4, 7, 8, 16, 56])
        gated = rnd.random() < 0.35
        unit = 32 if gated else rnd.choice([1, 16, 16, 64])
        rows_per_cb = unit * rnd.randint(1, max(1, rnd.choice([3000, 9000, 30000]) // (unit * G)))
        N = G * rows_per_cb
        if N * K > 150_000_000:
            continue
        E = rnd.choice([256, 256, 200, 16])
        spec = ProblemSpec("rnd_gemv", GEOM_B, M, K, N, 8, E, G, 8, codebook_3d=(G > 1))
        x, codes, cb = make_problem(spec, seed=1000 + case, device=DEV)
        bias = (torch.randn(N, generator=torch.Generator().manual_seed(case)) * 0.5).half().to(DEV) if case % 2 else None
        _say("random gemv", case, spec, "gated" if gated else "", "bias" if bias is not None else "")
        call = cabi.e2e_gemm_b_gated if gated else cabi.e2e_gemm_b
        try:
            y = call(x, codes, cb, variant=cabi.VARIANT_DECODE_GEMV, bias=bias)
        except cabi.VqGemmError as e:
            assert e.code == -4, e
            refused += 1
            continue
        ref = call(x, codes, cb, variant=cabi.VARIANT_GENERIC, bias=bias).float()
        torch.cuda.synchronize()
        err = ((y.float() - ref).abs().max() / max(ref.abs().max().item(), 1e-3)).item()
        assert err <= TOL, (case, spec, gated, err)
        assert torch.equal(call(x, codes, cb, variant=cabi.VARIANT_DECODE_GEMV, bias=bias), y)
        ran += 1
    _say(f"  {ran} launches compared, {refused} shapes refused")
    assert ran >= 80


def test_every_m_from_1_to_16_on_the_decode_kernel():
    K, N = 1024, 80
    for M in range(1, 17):
        spec = ProblemSpec("m", GEOM_B, M, K, N, 8, 256, 1, 8)
        x, codes, cb = make_problem(spec, seed=10 + M, device=DEV)
        _say("decode M =", M)
        y = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE)
        torch.cuda.synchronize()
        _check_gemm(y, x, codes, cb, what=f"M={M}")


def test_properties_constant_codes_zero_codebook_scaling():
    spec = ProblemSpec("prop", GEOM_B, 16, 1024, 128, 8, 256, 1, 8)
    x, codes, cb = make_problem(spec, seed=4, device=DEV)
    for variant in (cabi.VARIANT_DECODE, cabi.VARIANT_PREFILL, cabi.VARIANT_PREFILL_NARROW, cabi.VARIANT_PREFILL_SMALL):
        _say("properties", cabi.VARIANT_NAMES[variant])
        const = torch.full_like(codes, 37)
        y = cabi.e2e_gemm_b(x, const, cb, variant=variant)
        assert torch.equal(y, y[:, :1].expand_as(y))            # all W rows identical
        z = cabi.e2e_gemm_b(x, codes, torch.zeros_like(cb), variant=variant)
        assert not z.any()
        y1 = cabi.e2e_gemm_b(x, codes, cb, variant=variant)
        y4 = cabi.e2e_gemm_b(x * 4, codes, cb, variant=variant)
        assert torch.equal(y4, (y1.float() * 4).half())          # power-of-two scaling is exact
        # G identical codebooks == one codebook: the same W exactly (a permuted one-hot X reads it
        # out bit for bit), the same product up to the order of the fp32 sums (the kernels for one
        # and for several codebooks split K differently)
        cb4 = cb.unsqueeze(0).repeat(4, 1, 1).contiguous()
        eye = torch.eye(16, 1024, dtype=torch.float16, device=DEV).roll(5, dims=1)
        assert torch.equal(cabi.e2e_gemm_b(eye, codes, cb4, variant=variant),
                           cabi.e2e_gemm_b(eye, codes, cb, variant=variant))
        y1g = cabi.e2e_gemm_b(x, codes, cb4, variant=variant)
        assert vo.rel_err(_np(y1g), _np(y1).astype(np.float64))[0] <= 2e-3
        # run-to-run determinism (the reference harness's own check, bench.py:118-132)
        for _ in range(4):
            assert torch.equal(cabi.e2e_gemm_b(x, codes, cb, variant=variant), y1)


def test_empty_problems_and_rejections_on_device():
    cb = torch.zeros(256, 8, dtype=torch.float16, device=DEV)
    x0 = torch.zeros(0, 64, dtype=torch.float16, device=DEV)
    codes = torch.zeros(16, 8, dtype=torch.uint8, device=DEV)
    assert cabi.e2e_gemm_b(x0, codes, cb).shape == (0, 16)
    x = torch.randn(2, 64, device=DEV).half()
    assert cabi.e2e_gemm_b(x, codes[:0], cb).shape == (2, 0)
    with pytest.raises(cabi.VqGemmError) as ei:   # prefill kernel explicitly requested with a misaligned x
        buf = torch.zeros(2 * 64 + 8, dtype=torch.float16, device=DEV)
        xm = buf[1:1 + 128].view(2, 64)
        cabi.e2e_gemm_b(xm, codes, cb, variant=cabi.VARIANT_PREFILL)
    assert ei.value.code == -5
    # ... while the automatic choice serves the same misaligned tensor with the generic kernel
    xm.copy_(x)
    y = cabi.e2e_gemm_b(xm, codes, cb)
    torch.cuda.synchronize()
    _check_gemm(y, xm, codes, cb, what="misaligned x")


# ------------------------------------------------------------------ geometry A (reference-native tensors)
# all but the second and the third are shapes the fused tiled kernel takes (K % 64 == 0, Nc % 16 == 0): a
# single row, ragged M and N, K of two stages only, a single 16-column piece of codes
@pytest.mark.parametrize("M,K,Nc", [(32, 256, 64), (5, 96, 8), (130, 512, 132), (300, 128, 80), (257, 64, 16),
                                    (1000, 1024, 400), (520, 2048, 640), (1, 64, 16), (16, 1024, 640)])
def test_geometry_a(M, K, Nc):
    spec = ProblemSpec("A", GEOM_A, M, K, 2 * Nc, 2, 256, Nc // 4, 8, codebook_std=1.0)
    x, w, cb = make_problem(spec, seed=5, device=DEV)
    _say("geometry A", M, K, Nc)
    dec = cabi.dequant_a(w, cb)
    torch.cuda.synchronize()
    want = vo.dequant_a(_np(w), _np(cb))
    assert np.array_equal(_np(dec).view(np.uint16), want.view(np.uint16))
    fused_ok = K % 64 == 0 and Nc % 16 == 0
    assert (cabi.select_variant_a(M, K, Nc) == cabi.VARIANT_PREFILL) == fused_ok
    for variant in (cabi.VARIANT_AUTO, cabi.VARIANT_GENERIC, cabi.VARIANT_TWOPASS, cabi.VARIANT_PREFILL):
        if variant == cabi.VARIANT_PREFILL and not fused_ok:
            with pytest.raises(cabi.VqGemmError) as ei:
                cabi.e2e_gemm_a(x, w, cb, variant=variant)
            assert ei.value.code == -4
            continue
        _say("geometry A", cabi.VARIANT_NAMES[variant])
        y = cabi.e2e_gemm_a(x, w, cb, variant=variant)
        torch.cuda.synchronize()
        _check_gemm(y, x, w, cb, geometry=GEOM_A, what=f"A/{cabi.VARIANT_NAMES[variant]}")
    if fused_ok:
        # one-hot rows of X read W_dec out through the fused kernel: exact
        idx = torch.randint(0, K, (M,), generator=torch.Generator().manual_seed(9)).to(DEV)
        xo = torch.zeros(M, K, dtype=torch.float16, device=DEV)
        xo[torch.arange(M, device=DEV), idx] = 1
        for kernel in ("fused", "wave_k"):
            _say("geometry A fused one-hot", M, K, Nc, kernel)
            call = lambda a: _with_geometry_a_kernel(kernel, lambda: cabi.e2e_gemm_a(a, w, cb, variant=cabi.VARIANT_PREFILL))
            y = call(xo)
            torch.cuda.synchronize()
            assert torch.equal(y, dec[idx]), kernel
            _check_gemm(call(x), x, w, cb, geometry=GEOM_A, what=f"A/{kernel}")


# ------------------------------------------------------------------ plain GEMM control and the hipBLASLt baseline
@pytest.mark.parametrize("M,K,N", [(128, 128, 128), (33, 72, 50), (257, 1024, 384), (1, 64, 8)])
def test_plain_gemm_and_hipblaslt_baseline(M, K, N):
    g = torch.Generator().manual_seed(6)
    x = torch.randn(M, K, generator=g).half().to(DEV)
    w = (torch.randn(K, N, generator=g) * 0.05).half().to(DEV)
    ref = vo.gemm(_np(x), _np(w), acc=np.float64)
    _say("plain gemm", M, K, N)
    y = cabi.gemm_f16(x, w)
    torch.cuda.synchronize()
    e1, _ = vo.rel_err(_np(y), ref)
    assert e1 <= TOL, e1
    _say("hipblaslt gemm", M, K, N)
    yb = cabi.ref_gemm_f16(x, w)
    ybt = cabi.ref_gemm_f16(x, w.t().contiguous(), w_is_nk=True)
    torch.cuda.synchronize()
    for t in (yb, ybt):
        e1, _ = vo.rel_err(_np(t), ref)
        assert e1 <= TOL, e1


@pytest.mark.parametrize("kernel", ["s1", "s2_128", "s3_wasp"])
def test_harness_with_the_reference_controls(kernel, tmp_path):
    """vq_gemm_amd.harness: the reference harness's three calls on its own tensor layout, with its checks
    made assertions; the full reference shape through the fused module, small shapes through the others."""
    from vq_gemm_amd import harness
    full = kernel == "s2_128"
    _say("harness", kernel, "vq gemm")
    r = harness.run(kernel, M=2048 if full else 300, K=4096 if full else 256, N=640 if full else 80, timing=False,
                    figures=None if full else str(tmp_path))
    assert r["deterministic"] and r["dequant_bit_exact"] and r["rel_err"] <= TOL
    if not full:   # the error picture (reference bench.py:105-116) is written where asked
        import os
        assert r["figure"] == os.path.join(str(tmp_path), "M=300_N=80_K=256_err.png") and os.path.getsize(r["figure"]) > 1000
    _say("harness", kernel, "plain gemm")
    r = harness.run(kernel, test_gemm=True, M=200, K=128, N=136, timing=False)
    assert r["deterministic"] and r["rel_err"] <= TOL
    _say("harness", kernel, "profiling launch")
    harness.run(kernel, profiling=True, M=128, K=64, N=32)


@pytest.mark.parametrize("M,N", [(1, 8), (16, 11008), (33, 50), (300, 1000), (2048, 4096)])
def test_silu_mul_kernel_against_the_oracle(M, N):
    g = torch.Generator().manual_seed(21)
    a = (torch.randn(M, 2 * N, generator=g) * 3).half().to(DEV)
    a[0, 0] = 0.0
    a[M - 1, N - 1] = 30.0
    a[M - 1, 0] = -30.0
    _say("silu_mul", M, N)
    out = cabi.silu_mul(a)
    torch.cuda.synchronize()
    want = vo.silu_mul(_np(a))
    # exp differs in the last fp32 bits between the device and the host: at most one fp16 step apart
    def ordered(h):   # fp16 bit patterns on one monotonic integer scale, -0 and +0 together
        b = h.view(np.uint16).astype(np.int32)
        return np.where(b & 0x8000, -(b & 0x7fff), b)
    steps = np.abs(ordered(_np(out)) - ordered(want))
    assert steps.max() <= 1, steps.max()
    assert (steps == 0).mean() > 0.99


def test_gated_mlp_module():
    from vq_gemm_amd.nn import VQGatedMLP, VQLinear
    K, H = 512, 768
    s_gu = ProblemSpec("gu", GEOM_B, 1, K, 2 * H, 8, 256, 2, 8, codebook_3d=True, codebook_std=0.05)
    s_d = ProblemSpec("d", GEOM_B, 1, H, K, 8, 256, 1, 8, codebook_std=0.05)
    _, c_gu, cb_gu = make_problem(s_gu, seed=31, device=DEV)
    _, c_d, cb_d = make_problem(s_d, seed=32, device=DEV)
    mlp = VQGatedMLP(VQLinear(c_gu, cb_gu), VQLinear(c_d, cb_d))
    w_gu = vo.dequant_b(_np(c_gu), _np(cb_gu)).astype(np.float64)
    w_d = vo.dequant_b(_np(c_d), _np(cb_d)).astype(np.float64)
    for M in (3, 200):
        x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).half().to(DEV)
        _say("gated mlp", M)
        y = mlp(x)
        torch.cuda.synchronize()
        # the same chain with the same rounding points: fp16 after the first product, after the gate, at the end
        h = (_np(x).astype(np.float64) @ w_gu.T).astype(np.float16)
        ref = vo.silu_mul(h).astype(np.float64) @ w_d.T
        # the device's intermediate results sit one fp16 step off the host's here and there (fp32 against
        # float64 sums at rounding boundaries), so the chain is held to the bound on the largest output
        e1, e2 = vo.rel_err(_np(y), ref)
        _say(f"  gated mlp M={M}: rel_err(floor)={e1:.3e} max/max={e2:.3e}")
        assert e2 <= TOL and e1 <= 0.1, (e1, e2)


@pytest.mark.parametrize("dims", [(1, 4096, 4096, 8, 256, 1, 8), (16, 4096, 4096, 8, 256, 1, 8), (16, 2048, 11008, 8, 16, 1, 8), (64, 4096, 2048, 4, 4096, 1, 16),
                                  (203, 2816, 7040, 8, 256, 1, 8), (954, 14080, 1920, 8, 256, 1, 8), (600, 1024, 2048, 8, 256, 1, 8)])
def test_the_automatic_choice_launches_what_the_report_names(dims):
    """Bit for bit (every kernel has its own order of sums), without a workspace and with the one asked for."""
    M, K, N, v, e, g, bits = dims
    x, codes, cb = make_problem(ProblemSpec("named", GEOM_B, *dims), seed=3, device=DEV)
    need = cabi.workspace_bytes_b(*dims)
    for ws_bytes in (0, max(need, 256)):
        name = cabi.auto_variant_name_b(*dims, ws_bytes)
        _say("named by the report", dims, ws_bytes, name)
        variant = {n: i for i, n in cabi.VARIANT_NAMES.items()}[name]
        ws = torch.empty(max(ws_bytes, cabi.workspace_bytes_b(*dims, variant)), dtype=torch.uint8, device=DEV)
        y = cabi.e2e_gemm_b_ws(x, codes, cb, workspace=ws) if ws_bytes else cabi.e2e_gemm_b(x, codes, cb)
        assert torch.equal(y, cabi.e2e_gemm_b_ws(x, codes, cb, variant=variant, workspace=ws)), name


def test_tune_reports_every_variant_and_the_automatic_choice():
    from vq_gemm_amd import tune
    _say("tune 300 512 520")
    r = tune.tune(300, 512, 520, 8, 256, 4, 8, verbose=False)
    assert {"prefill", "prefill_small", "twopass", "auto"} <= set(r["times_us"])
    assert "wave_k" in r["times_us"] and "wave_k" in tune.tune_cold(100, 512, 520, 8, 256, 4, 8, verbose=False)["times_us"]
    assert r["auto_picks"] in r["times_us"] and r["hipblaslt_us"] > 0
    # (how close the automatic choice comes to the fastest variant is a figure of the report, r["auto_over_fastest"]:
    # a timing, not a parity property, and not asserted here)
    assert r["auto_over_fastest"] > 0


def test_tune_fit_returns_the_table_and_the_library_takes_it():
    import math
    from vq_gemm_amd import tune
    before = cabi.tuning()
    fitted = tune.fit(verbose=False)
    assert set(fitted) == set(before)
    # (the fitted values are timings of the box at hand: printed, not asserted - only that they are numbers)
    _say("  fitted: " + ", ".join(f"{k}={v:.3g}" for k, v in sorted(fitted.items())))
    assert all(math.isfinite(v) for v in fitted.values())
    assert fitted["splitk_force_splits"] == before["splitk_force_splits"] == 0.0
    try:
        cabi.set_tuning(**fitted)
        assert cabi.tuning()["decode_tile_us"] == fitted["decode_tile_us"]
        # the library answers for the measured configurations under the refitted table (which kernel it names is
        # the fit's business; that it names one the shape can run is the library's)
        assert cabi.select_variant_b(4096, 4096, 4096, 8, 256, 32, 8) > 0
        assert cabi.select_variant_b(16, 4096, 11008, 4, 4096, 1, 16) > 0
    finally:
        cabi.set_tuning(**before)
    # with the compiled-in table the measured configurations keep their kernels
    assert cabi.select_variant_b(4096, 4096, 4096, 8, 256, 32, 8) == cabi.VARIANT_PREFILL
    assert cabi.select_variant_b(16, 4096, 11008, 4, 4096, 1, 16) == cabi.VARIANT_DECODE


def test_tune_search_tries_the_kernel_parameter_candidates_cold_and_the_library_takes_the_winners():
    import math
    from vq_gemm_amd import tune
    before = cabi.tuning()
    found = tune.search(verbose=False, quick=True)
    assert set(found) == set(before) and all(math.isfinite(v) for v in found.values())
    _say("  searched: " + ", ".join(f"{k}={found[k]:g}" for k in sorted(found) if found[k] != before[k]))
    _say("  report:", tune.search.last_report)
    # candidates stay inside what the kernels are built for
    assert found["gemv_wide_rows_per_group"] in (1.0, 2.0) and found["gemv_wide_groups_in_flight"] in (2.0, 3.0)
    assert found["gemv_wide_rows_per_group_long_k"] in (1.0, 2.0) and found["gemv_wide_groups_in_flight_long_k"] in (2.0, 3.0)
    assert found["decode_stream_min_k"] in (8192.0, 14336.0, 1e8) and found["decode_stream_min_k_few_rows"] in (8192.0, 14336.0, 1e8)
    assert found["gemv_wide_two_rows_max_runs"] in (before["gemv_wide_two_rows_max_runs"], 16.0, 22.0, 28.0)
    assert cabi.tuning() == before, "the search leaves the table as it found it"
    # every candidate of the wide form's loop gives the same bits as the default (same sums in the same order per row)
    spec = ProblemSpec("cand", GEOM_B, 1, 4096, 12288, 8, 256, 3, 8, codebook_3d=True)
    x, codes, cb = make_problem(spec, seed=81, device=DEV)
    want = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE_GEMV).clone()
    _check_gemm(want, x, codes, cb, what="wide GEMV, default loop")
    try:
        for g in (1, 2):
            for nbuf in (2, 3):
                for runs in (0, 1e6):
                    cabi.set_tuning(gemv_wide_rows_per_group=g, gemv_wide_groups_in_flight=nbuf, gemv_wide_plain_table_max_runs=runs)
                    assert torch.equal(cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE_GEMV), want), (g, nbuf, runs)
        # beyond K = 4096, plain and gated (one group of two rows, or the gate and the up row as two groups in turn)
        spec8 = ProblemSpec("cand8", GEOM_B, 1, 8192, 8192, 8, 256, 1, 8)
        x8, codes8, cb8 = make_problem(spec8, seed=82, device=DEV)
        want8 = vo.gated_gemm_b(_np(x8), _np(codes8), _np(cb8)).astype(np.float64)
        plain8 = None
        for g, nbuf in ((1, 2), (1, 3), (2, 2)):
            cabi.set_tuning(gemv_wide_rows_per_group_long_k=g, gemv_wide_groups_in_flight_long_k=nbuf)
            yp = cabi.e2e_gemm_b(x8, codes8, cb8, variant=cabi.VARIANT_DECODE_GEMV).clone()
            plain8 = yp if plain8 is None else plain8
            assert torch.equal(yp, plain8), (g, nbuf)
            e1, e2 = vo.rel_err(_np(cabi.e2e_gemm_b_gated(x8, codes8, cb8, variant=cabi.VARIANT_DECODE_GEMV)), want8)
            assert e2 <= TOL and e1 <= 2 * TOL, (g, nbuf, e1, e2)
        _check_gemm(plain8, x8, codes8, cb8, what="wide GEMV, K=8192")
        cabi.set_tuning(**found)
        assert cabi.tuning() == found
        y = cabi.e2e_gemm_b(x, codes, cb)
        _check_gemm(y, x, codes, cb, what="automatic choice under the searched table")
    finally:
        cabi.set_tuning(**before)


# shapes the tiled kernel takes (K a multiple of 64, N of 8): few tiles -> 128x128
# tiles (the first three and the fifth), about one 256x128 tile per compute unit -> those (the seventh and eighth),
# more -> 256x256 tiles (the fourth and the sixth); ragged M and N
TILED_GEMM = [(300, 128, 520), (512, 192, 1288), (1024, 256, 136), (1024, 128, 16384), (2048, 4096, 1280),
              (700, 64, 16392), (2000, 256, 4088), (1024, 192, 8192), (1, 64, 8), (16, 128, 520), (96, 256, 136)]


@pytest.mark.parametrize("M,K,N", TILED_GEMM)
def test_plain_gemm_tiled_kernel(M, K, N):
    g = torch.Generator().manual_seed(7)
    w = (torch.randn(K, N, generator=g) * 0.05).half().to(DEV)
    # one-hot rows of X read W out through the matrix cores: exact
    idx = torch.randint(0, K, (M,), generator=g).to(DEV)
    x = torch.zeros(M, K, dtype=torch.float16, device=DEV)
    x[torch.arange(M, device=DEV), idx] = 1
    _say("tiled gemm one-hot", M, K, N)
    y = cabi.gemm_f16(x, w)
    torch.cuda.synchronize()
    assert torch.equal(y, w[idx])
    x = torch.randn(M, K, generator=g).half().to(DEV)
    _say("tiled gemm random", M, K, N)
    y = cabi.gemm_f16(x, w)
    torch.cuda.synchronize()
    ref = (x.double() @ w.double()).cpu().numpy()
    e1, _ = vo.rel_err(_np(y), ref)
    assert e1 <= TOL, e1
    # and the [N,K] layout, through the two-pass route of the VQ entry point
    if K % 8 == 0 and M * K <= 1024 * 1024:
        spec = ProblemSpec("t", GEOM_B, M, K, N, 8, 256, 1, 8)
        x, codes, cb = make_problem(spec, seed=8, device=DEV)
        _say("tiled gemm two-pass", M, K, N)
        y = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_TWOPASS)
        torch.cuda.synchronize()
        wd = cabi.dequant_b(codes, cb)
        e1, _ = vo.rel_err(_np(y), (x.double() @ wd.double().T).cpu().numpy())
        assert e1 <= TOL, e1


def test_random_shapes_plain_gemm_and_reference_layout_against_the_library_gemm():
    """Seeded random shapes through the tiled plain GEMM ([K,N] and, by the two-pass route, [N,K]) and the
    fused kernel for the reference's layout, each against hipBLASLt on the same (dequantised) operands."""
    import random
    rnd = random.Random(77)

    def close(y, ref, what):
        scale = max(ref.float().abs().max().item(), 1e-3)
        err = ((y.float() - ref.float()).abs().max() / scale).item()
        assert err <= TOL, (what, err)

    for case in range(12):
        M = rnd.choice([97, 130, 256, 257, 300, 513, 777, 1024])
        K = 64 * rnd.randint(1, 24)
        N = 8 * rnd.randint(1, 300)
        g = torch.Generator().manual_seed(case)
        x = torch.randn(M, K, generator=g).half().to(DEV)
        w = (torch.randn(K, N, generator=g) * 0.05).half().to(DEV)
        _say("random plain gemm", M, K, N)
        yg = cabi.gemm_f16(x, w)
        close(yg, cabi.ref_gemm_f16(x, w), ("gemm", M, K, N))
        e1, _ = vo.rel_err(_np(yg), vo.gemm(_np(x), _np(w), acc=np.float64))
        assert e1 <= TOL, ("gemm against the oracle", M, K, N, e1)
    for case in range(10):
        M = rnd.choice([16, 97, 130, 256, 257, 300, 513, 777])
        K = 64 * rnd.randint(1, 24)
        Nc = 16 * rnd.randint(1, 60)
        spec = ProblemSpec("A", GEOM_A, M, K, 2 * Nc, 2, 256, Nc // 4, 8, codebook_std=0.05)
        x, w, cb = make_problem(spec, seed=case, device=DEV)
        _say("random reference layout", M, K, Nc)
        y = cabi.e2e_gemm_a(x, w, cb, variant=cabi.VARIANT_PREFILL)
        close(y, cabi.ref_gemm_f16(x, cabi.dequant_a(w, cb)), ("A", M, K, Nc))
        _check_gemm(y, x, w, cb, geometry=GEOM_A, what=f"random reference layout {M}x{K}x{Nc} against the oracle")
    for case in range(8):
        M = rnd.choice([97, 130, 256, 300, 513])
        K = 64 * rnd.randint(1, 24)
        N = rnd.randint(1, 1500)
        spec = ProblemSpec("B", GEOM_B, M, K, N, 8, 256, 1, 8)
        x, codes, cb = make_problem(spec, seed=case, device=DEV)
        _say("random two-pass", M, K, N)
        y = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_TWOPASS)
        close(y, cabi.ref_gemm_f16(x, cabi.dequant_b(codes, cb), w_is_nk=True), ("two-pass", M, K, N))
        _check_gemm(y, x, codes, cb, what=f"random two-pass {M}x{K}x{N} against the oracle")


# ------------------------------------------------------------------ the measured configurations at full size
def test_config_c1_full_against_golden_and_oracle():
    import json, os
    spec = CONFIGS["C1"]
    x, codes, cb = make_problem(spec, seed=42, device=DEV)
    _say("C1 full")
    y = cabi.e2e_gemm_b(x, codes, cb)
    w = cabi.dequant_b(codes, cb)
    torch.cuda.synchronize()
    _check_gemm(y, x, codes, cb, what="C1")
    g = os.path.join(os.path.dirname(__file__), "golden")
    data = np.load(os.path.join(g, "C1.npz"))
    e1, _ = vo.rel_err(_np(y)[data["sample_rows"]][:, data["sample_cols"]], data["y_samples_f64"])
    assert e1 <= TOL
    assert np.array_equal(_np(w)[data["w_rows"]][:, data["w_cols"]].view(np.uint16), data["w_samples"].view(np.uint16))


@pytest.mark.parametrize("name", ["C2", "C3"])
def test_decode_configs_full_size(name):
    spec = CONFIGS[name]
    x, codes, cb = make_problem(spec, seed=42, device=DEV)
    _say(name, "full", spec)
    y = cabi.e2e_gemm_b(x, codes, cb)
    w = cabi.dequant_b(codes, cb)
    torch.cuda.synchronize()
    want_w = vo.dequant_b(_np(codes), _np(cb))
    assert np.array_equal(_np(w).view(np.uint16), want_w.view(np.uint16))       # bit-exact dequant at full size
    ref = _np(x).astype(np.float64) @ want_w.astype(np.float64).T
    e1, e2 = vo.rel_err(_np(y), ref)
    _say(f"  {name}: rel_err={e1:.3e} {e2:.3e}")
    assert e1 <= TOL
    for _ in range(4):
        assert torch.equal(cabi.e2e_gemm_b(x, codes, cb), y)


@pytest.mark.parametrize("name", ["C4", "C5"])
def test_prefill_configs_full_size(name):
    """Full-size prefill: bit-exact dequant, fp64 oracle on a sample of output rows, one-hot rows,
    the two-pass route (dequant + plain GEMM) as a second on-device opinion, determinism."""
    spec = CONFIGS[name]
    x, codes, cb = make_problem(spec, seed=42, device=DEV)
    _say(name, "full", spec)
    # plant one-hot rows: those outputs must be bit-exact copies of weight columns
    hot_rows = [0, spec.M // 2 + 1, spec.M - 1]
    hot_k = [0, spec.K // 2 + 3, spec.K - 1]
    for r, k in zip(hot_rows, hot_k):
        x[r].zero_()
        x[r, k] = 1.0
    y = cabi.e2e_gemm_b(x, codes, cb)
    torch.cuda.synchronize()
    w = cabi.dequant_b(codes, cb)
    torch.cuda.synchronize()
    codes_np, cb_np = _np(codes), _np(cb)
    rows = np.random.default_rng(0).choice(spec.N, size=4096 if name == "C4" else 2048, replace=False)
    rows.sort()
    # bit-exact dequant on a sample of W rows
    g_of = rows // (spec.N // spec.n_codebooks)
    w_np = _np(w[torch.from_numpy(rows).to(DEV)])
    for g in np.unique(g_of):
        sel = g_of == g
        want = vo.dequant_b(codes_np[rows[sel]], cb_np[g])
        assert np.array_equal(w_np[sel].view(np.uint16), want.view(np.uint16))
    for r, k in zip(hot_rows, hot_k):
        assert torch.equal(y[r], w[:, k]), (r, k)
    # fp64 oracle on sampled X rows x sampled W rows
    m_idx = np.sort(np.random.default_rng(1).choice(spec.M, size=48, replace=False))
    ref = _np(x)[m_idx].astype(np.float64) @ w_np.astype(np.float64).T
    got = _np(y[torch.from_numpy(m_idx).to(DEV)][:, torch.from_numpy(rows).to(DEV)])
    e1, e2 = vo.rel_err(got, ref)
    _say(f"  {name}: sampled rel_err={e1:.3e} {e2:.3e}")
    assert e1 <= TOL
    # the whole output against fp32 torch on the device (a library matmul on the dequantised weights)
    ref_dev = (x.float() @ w.float().t())
    err = ((y.float() - ref_dev).abs() / ref_dev.abs().clamp_min(1e-2 * ref_dev.pow(2).mean().sqrt())).max().item()
    _say(f"  {name}: full-output rel_err vs device fp32 matmul={err:.3e}")
    assert err <= TOL
    del ref_dev
    assert torch.equal(cabi.e2e_gemm_b(x, codes, cb), y)


# ------------------------------------------------------------------ torch extension modules (the drop-in surface)
def test_torch_extension_modules_serve_both_geometries():
    from vq_gemm_amd import ops
    spec = CONFIGS["C1"]
    x, codes, cb = make_problem(spec, seed=42, device=DEV)
    ref = vo.vq_gemm_b(_np(x), _np(codes), _np(cb), acc=np.float64)
    for key in ("s1", "s2_128", "s2_512", "s3_naive", "s3_wasp"):
        _say("module", key)
        mod = ops.load_module(key)
        y = mod.e2e_gemm(x, codes, cb)
        torch.cuda.synchronize()
        assert y.dtype == torch.float16 and y.shape == (spec.M, spec.N) and y.device == x.device
        e1, _ = vo.rel_err(_np(y), ref)
        assert e1 <= TOL, (key, e1)
    # reference-native tensors, as bench.py:83-88 of the reference builds them
    sa = ProblemSpec("A", GEOM_A, 128, 256, 256, 2, 256, 32, 8, codebook_std=1.0)
    xa, wa, cba = make_problem(sa, seed=7, device=DEV)
    refa = vo.vq_gemm_a(_np(xa), _np(wa), _np(cba), acc=np.float64)
    for key in ("s1", "s2_128"):
        ya = ops.load_module(key).e2e_gemm(xa, wa, cba)
        torch.cuda.synchronize()
        assert ya.shape == (128, 256)
        e1, _ = vo.rel_err(_np(ya), refa)
        assert e1 <= TOL, (key, e1)
    # dequant + both gemm exports
    mod = ops.load_module("s2_128")
    assert np.array_equal(_np(mod.dequant(codes, cb)).view(np.uint16), vo.dequant_b(_np(codes), _np(cb)).view(np.uint16))
    wd = mod.dequant(wa, cba)
    assert np.array_equal(_np(wd).view(np.uint16), vo.dequant_a(_np(wa), _np(cba)).view(np.uint16))
    for key in ("s2_128", "cublas_gemm"):
        yg = ops.load_module(key).gemm(xa, wd)
        torch.cuda.synchronize()
        e1, _ = vo.rel_err(_np(yg), refa)
        assert e1 <= TOL, (key, e1)
    # non-contiguous / wrong-shape inputs
    yt = mod.e2e_gemm(x.t().contiguous().t(), codes, cb)
    assert torch.equal(yt, mod.e2e_gemm(x, codes, cb))
    with pytest.raises(RuntimeError):
        mod.e2e_gemm(x[:, :100], codes, cb)
    with pytest.raises(RuntimeError):
        mod.e2e_gemm(x.float(), codes, cb)


# ------------------------------------------------------------------ reference-native tensors through the modules: every route
# Shapes the fused kernel refuses (K % 64 != 0; Nc % 16 != 0) or does not prefer (more tiles than compute
# units: the two-pass route with the library's own tiled GEMM), as the reference's harness calls them
# (bench.py:83-88): module.e2e_gemm(input, w, codebook).
@pytest.mark.parametrize("M,K,Nc,route", [(130, 96, 64, "twopass_odd"), (257, 512, 132, "twopass_odd"), (4096, 4096, 2048, "twopass"),
                                          (2048, 1024, 2560, "twopass"), (2048, 4096, 640, "fused")])
def test_modules_serve_reference_native_shapes_on_every_route(M, K, Nc, route):
    from vq_gemm_amd import ops
    spec = ProblemSpec("A", GEOM_A, M, K, 2 * Nc, 2, 256, Nc // 4, 8, codebook_std=1.0)
    x, w, cb = make_problem(spec, seed=11, device=DEV)
    fused_ok = K % 64 == 0 and Nc % 16 == 0
    picked = cabi.select_variant_a(M, K, Nc, has_workspace=True)
    want_variant = {"twopass_odd": cabi.VARIANT_TWOPASS, "twopass": cabi.VARIANT_TWOPASS, "fused": cabi.VARIANT_PREFILL}[route]
    assert picked == want_variant and (route == "twopass_odd") == (not fused_ok), (picked, route)
    # the oracle on a sample of the rows of X (rows are independent): full height would be minutes of fp64 on the host
    rows = np.unique(np.concatenate([np.arange(0, M, max(1, M // 48)), [M - 1]]))
    ref = vo.vq_gemm_a(_np(x)[rows], _np(w), _np(cb), acc=np.float64)
    for key in ("s2_128", "s3_wasp", "s1"):
        _say("module", key, "reference-native", M, K, Nc, route)
        y = ops.load_module(key).e2e_gemm(x, w, cb)
        torch.cuda.synchronize()
        assert y.shape == (M, 2 * Nc) and y.dtype == torch.float16
        e1, e2 = vo.rel_err(_np(y)[rows], ref)
        _say(f"  {key}: rel_err(floor)={e1:.3e} max/max={e2:.3e}")
        assert e1 <= TOL, (key, e1, e2)
    # the fused modules' result is what the C ABI's automatic choice gives with scratch at hand
    ws = torch.empty(K, 2 * Nc, dtype=torch.float16, device=DEV)
    assert torch.equal(ops.load_module("s2_128").e2e_gemm(x, w, cb), cabi.e2e_gemm_a(x, w, cb, workspace=ws))


def _with_geometry_a_kernel(kernel, call):
    """`call` with geometry A's fused product by the one kernel or the other, whichever the cost models would take."""
    before = cabi.tuning()["wave_k_force"]
    try:
        cabi.set_tuning(wave_k_force={"wave_k": 1, "fused": 2}[kernel])
        return call()
    finally:
        cabi.set_tuning(wave_k_force=before)


@pytest.mark.parametrize("kernel", ["fused", "wave_k"])
@pytest.mark.parametrize("M,K,Nc", [(2048, 4096, 640), (512, 4096, 640), (2048, 2048, 2048)])
def test_fused_reference_layout_kernel_gives_the_same_bits_on_every_launch(M, K, Nc, kernel):
    # Both kernels wait for its hand-issued loads by count, and a count that does not match the order of the
    # loads shows as a rare wrong element on a fast launch, not as a steady error.  The reference's own shape
    # (128x128 tiles of the fused kernel, 160 of them), a shorter X on it and a shape of its 256x128 tiles: 50 launches each on fixed
    # operands, every result equal to the first bit for bit, the first within the bar of the oracle on sampled rows.
    spec = ProblemSpec("A", GEOM_A, M, K, 2 * Nc, 2, 256, Nc // 4, 8, codebook_std=1.0)
    x, w, cb = make_problem(spec, seed=71, device=DEV)
    _say("fused geometry A, 50 launches", M, K, Nc, kernel)
    launch = lambda: _with_geometry_a_kernel(kernel, lambda: cabi.e2e_gemm_a(x, w, cb, variant=cabi.VARIANT_PREFILL))
    first = launch().clone()
    torch.cuda.synchronize()
    rows = np.unique(np.concatenate([np.arange(0, M, max(1, M // 32)), [M - 1]]))
    e1, e2 = vo.rel_err(_np(first)[rows], vo.vq_gemm_a(_np(x)[rows], _np(w), _np(cb), acc=np.float64))
    _say(f"  rel_err(floor)={e1:.3e} max/max={e2:.3e}")
    assert e1 <= TOL, (e1, e2)
    # back to back (the next launch's prologue runs beside the previous one's tail), then one at a time
    outs = [launch() for _ in range(25)]
    torch.cuda.synchronize()
    for i, y in enumerate(outs):
        assert torch.equal(y, first), f"launch {i} differs"
    for i in range(25):
        y = launch()
        torch.cuda.synchronize()
        assert torch.equal(y, first), f"synchronised launch {i} differs"


def test_module_out_argument_receives_the_result():
    from vq_gemm_amd import ops
    spec = CONFIGS["C1"]
    x, codes, cb = make_problem(spec, seed=42, device=DEV)
    mod = ops.load_module("s2_128")
    want = mod.e2e_gemm(x, codes, cb)
    out = torch.full((spec.M, spec.N), 7.0, dtype=torch.float16, device=DEV)
    got = mod.e2e_gemm(x, codes, cb, out=out)
    torch.cuda.synchronize()
    assert got.data_ptr() == out.data_ptr() and torch.equal(out, want)
    assert torch.equal(ops.e2e_gemm(x, codes, cb, out=out), want)
    sa = ProblemSpec("A", GEOM_A, 128, 256, 256, 2, 256, 32, 8, codebook_std=1.0)
    xa, wa, cba = make_problem(sa, seed=7, device=DEV)
    outa = torch.empty(128, 256, dtype=torch.float16, device=DEV)
    assert torch.equal(mod.e2e_gemm(xa, wa, cba, out=outa), mod.e2e_gemm(xa, wa, cba))
    for bad in (torch.empty(spec.M, spec.N + 1, dtype=torch.float16, device=DEV),
                torch.empty(spec.M, spec.N, dtype=torch.float32, device=DEV),
                torch.empty(spec.N, spec.M, dtype=torch.float16, device=DEV).t(),
                torch.empty(spec.M, spec.N, dtype=torch.float16)):
        with pytest.raises(RuntimeError):
            mod.e2e_gemm(x, codes, cb, out=bad)


def test_code_range_check_and_defined_results_for_codes_past_a_short_table(monkeypatch):
    from vq_gemm_amd import ops
    # the largest code, over ragged counts and misaligned starts
    g = torch.Generator().manual_seed(3)
    for dtype, hi in ((torch.uint8, 256), (torch.uint16, 4096)):
        base = torch.randint(0, hi // 2, (40_001,), generator=g, dtype=torch.int32)
        for start, count, spike in ((0, 40_001, 123), (3, 1000, 0), (1, 17, 16), (5, 0, None), (7, 33_000, 32_999)):
            c = base.clone()
            if spike is not None:
                c[start + spike] = hi - 1 - start
            t = c.to(dtype).to(DEV)[start:start + count]
            want = int(c[start:start + count].max()) if count else 0
            assert cabi.max_code(t) == want, (dtype, start, count)
    # a table of 100 entries and codes up to 255: the GEMV kernel of 8-bit codes reads zeros past the table
    spec = ProblemSpec("short", GEOM_B, 1, 2048, 64, 8, 100, 1, 8)
    x, codes, cb = make_problem(spec, seed=4, device=DEV)
    wild = torch.randint(0, 256, codes.shape, generator=g, dtype=torch.int32).to(torch.uint8).to(DEV)
    cb_padded = torch.zeros(256, 8, dtype=torch.float16, device=DEV)
    cb_padded[:100] = cb
    y = cabi.e2e_gemm_b(x, wild, cb, variant=cabi.VARIANT_DECODE_GEMV)
    torch.cuda.synchronize()
    _check_gemm(y, x, wild, cb_padded, what="GEMV kernel, codes past a 100-entry table read zeros")
    # every other kernel stays inside its own memory on the same input (results differ by kernel: not compared)
    # (the scalar and dequant kernels clamp to the last entry; the tiled kernels gather whatever their LDS holds there)
    for variant in (cabi.VARIANT_GENERIC, cabi.VARIANT_TWOPASS):
        assert torch.isfinite(cabi.e2e_gemm_b(x, wild, cb, variant=variant).float()).all()
    xt = torch.randn(300, 2048, generator=g).half().to(DEV)
    cabi.e2e_gemm_b(x, wild, cb, variant=cabi.VARIANT_DECODE)
    for variant in (cabi.VARIANT_PREFILL, cabi.VARIANT_PREFILL_SMALL):
        cabi.e2e_gemm_b(xt, wild, cb, variant=variant)
    torch.cuda.synchronize()
    # the modules refuse such codes when asked to check
    mod = ops.load_module("s2_128")
    mod.e2e_gemm(x, wild, cb)   # unchecked by default, as in the reference
    monkeypatch.setenv("VQGEMM_CHECK_CODES", "1")
    with pytest.raises(RuntimeError, match="entries"):
        mod.e2e_gemm(x, wild, cb)
    with pytest.raises(RuntimeError, match="entries"):
        mod.dequant(wild, cb)
    assert torch.equal(mod.e2e_gemm(x, codes, cb), cabi.e2e_gemm_b(x, codes, cb))   # valid codes pass


def test_vqlinear_repacks_after_its_codes_change():
    from vq_gemm_amd.nn import VQLinear
    spec = ProblemSpec("lin", GEOM_B, 16, 4096, 8192, 8, 256, 1, 8)   # a shape the K-sliced decode kernel takes
    x, codes, cb = make_problem(spec, seed=1, device=DEV)
    _, codes2, _ = make_problem(spec, seed=2, device=DEV)
    layer = VQLinear(codes.clone(), cb).prepack_for_decode()
    dims = (16, spec.K, spec.N, 8, 256, 1, 8)
    assert cabi.select_variant_b(*dims) == cabi.VARIANT_DECODE and cabi.decode_packed_supports(*dims)
    assert torch.equal(layer(x), cabi.e2e_gemm_b(x, codes, cb))
    state = {k: v.clone() for k, v in layer.state_dict().items()}
    state["codes"] = codes2
    layer.load_state_dict(state)
    y = layer(x)
    torch.cuda.synchronize()
    assert torch.equal(y, cabi.e2e_gemm_b(x, codes2, cb)), "short inputs must see the new codes"
    layer.codes.copy_(codes)   # in-place update
    assert torch.equal(layer(x), cabi.e2e_gemm_b(x, codes, cb))


# K-sliced kernel, wave-K kernel, streaming kernel, GEMV kernel, prefill kernels; two additive stages
@pytest.mark.parametrize("M,K,N,v,entries,bits,stages", [(4, 4096, 8192, 8, 256, 8, 1), (64, 8192, 512, 4, 4096, 16, 1), (16, 14336, 512, 8, 256, 8, 1),
                                                         (1, 4096, 512, 8, 256, 8, 1), (300, 512, 256, 4, 256, 8, 1), (8, 1024, 512, 8, 256, 8, 2)])
def test_packed_layer_takes_the_native_call_and_gives_the_plain_layers_bits(M, K, N, v, entries, bits, stages, monkeypatch):
    from vq_gemm_amd.nn import VQLinear
    _say("packed layer", M, K, N, v, entries, bits, stages)
    spec = ProblemSpec("packed", GEOM_B, M, stages * K, N, v, entries, 1, bits, codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=19, device=DEV)
    x = x[:, :K].contiguous()
    bias = torch.randn(N + 1, generator=torch.Generator().manual_seed(2)).half().to(DEV)
    for b in (None, bias[:N], bias[1:]):   # (the last one begins off 8 bytes: no kernel but the scalar one takes it)
        plain = VQLinear(codes, cb, b, k_repeat=stages)
        packed = VQLinear(codes, cb, b, k_repeat=stages).prepack_for_decode()
        want = plain(x)
        with monkeypatch.context() as m:
            m.setattr(VQLinear, "_forward_op", lambda self, x: pytest.fail("a plain call went through the dispatcher"))
            y = packed(x)
        torch.cuda.synchronize()
        assert torch.equal(y, want)
        if b is None or b.data_ptr() % 8 == 0:
            assert torch.equal(packed._forward_op(x), want) or stages > 1


def test_ctypes_wrappers_check_dtypes_and_shapes_before_the_gpu_sees_them():
    spec = CONFIGS["C1"]
    x, codes, cb = make_problem(spec, seed=42, device=DEV)
    with pytest.raises(ValueError):
        cabi.e2e_gemm_b(x, codes.to(torch.int32), cb)
    with pytest.raises(ValueError):
        cabi.e2e_gemm_b(x.float(), codes, cb)
    with pytest.raises(ValueError):
        cabi.e2e_gemm_b(x, codes[:, :-1].contiguous(), cb)
    with pytest.raises(ValueError):
        cabi.e2e_gemm_b(x, codes, cb.float())
    with pytest.raises(ValueError):
        cabi.e2e_gemm_b(x, codes, cb, out=torch.empty(spec.M, spec.N - 1, dtype=torch.float16, device=DEV))
    with pytest.raises(ValueError):
        cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_TWOPASS, workspace=torch.empty(10, dtype=torch.float16, device=DEV))
    with pytest.raises(ValueError):
        cabi.dequant_b(codes.to(torch.int64), cb)
    with pytest.raises(ValueError):
        torch.ops.vq_gemm_amd.vq_linear(x, codes.to(torch.int32), cb)
    sa = ProblemSpec("A", GEOM_A, 16, 64, 32, 2, 256, 4, 8, codebook_std=1.0)
    xa, wa, cba = make_problem(sa, seed=7, device=DEV)
    with pytest.raises(ValueError):
        cabi.e2e_gemm_a(xa, wa, cba[:3].contiguous())
    with pytest.raises(ValueError):
        cabi.e2e_gemm_a(xa, wa[:32].contiguous(), cba)


# ------------------------------------------------------------------ the gated epilogue (gate/up pairs)
GATED_B = [
    # name, M, K, N (rows of the interleaved W), vec, E, bits, G
    ("wide_tile", 300, 512, 1024, 8, 256, 8, 1),              # 256x256 tiles, ragged M
    ("wide_tile_books_and_tail", 512, 1056, 768, 4, 4096, 16, 3),
    ("narrow_tile", 1024, 256, 1152, 8, 256, 8, 9),
    ("small_tile", 200, 256, 416, 8, 256, 8, 13),              # 128x128 tiles, 32-row codebooks, ragged N in tiles
    ("small_tile_v2", 129, 256, 160, 2, 256, 8, 1),
    ("gemv_wide", 1, 4096, 8192, 8, 256, 8, 1),                  # one row of X: one output per group of two code rows
    ("gemv_wide_ragged_two_books", 1, 2048, 8192 + 64, 8, 200, 8, 2),
    ("gemv_wide_many_books", 1, 4096, 16384, 8, 256, 8, 16),
    ("gemv_wide_k8192", 1, 8192, 16384, 8, 256, 8, 1),           # gate row and up row as two groups of one row in turn
    ("gemv_wide_k6144_books", 1, 6144, 3 * 2752, 8, 256, 8, 3),
    ("gemv_wide_two_rows_of_x", 2, 4096, 8192, 8, 256, 8, 1),     # two rows of X: two outputs per pair of code rows
    ("gemv_wide_two_rows_of_x_k2048_books", 2, 2048, 8192 + 64, 8, 200, 8, 2),
    ("decode_shape", 16, 1024, 2048, 4, 4096, 16, 1),           # batched K-sliced kernel: gate and up tiles summed in pairs
    ("decode_shape_m2", 2, 4096, 4096, 8, 256, 8, 1),
    ("decode_books_ragged_units", 16, 4096, 4 * 1056, 8, 256, 8, 4),   # 33 pairs per codebook: short last batches
    ("decode_chunked_k", 9, 8192, 1024, 8, 256, 8, 1),           # K in two chunks: gate and up sums carried in the LDS
    ("decode_two_slabs_u8v4", 40, 2048, 1536, 4, 256, 8, 2),
    ("decode_v2_u16_general", 16, 1024, 512, 2, 4096, 16, 1),    # batches of one tile in the batched kernel: the general kernel
    ("decode_general_k640_ragged", 7, 640, 224, 8, 256, 8, 1),    # K not a multiple of 256: the general K-sliced kernel
    ("decode_general_books_48_rows", 16, 1152, 480, 4, 4096, 16, 10),   # 48 rows per codebook: pairs that lie in two codebooks
    ("decode_general_k8320_chunks_m33", 33, 8192 + 128, 96, 8, 256, 8, 1),   # three slabs of X, K in chunks
    ("gemv4_c3_weights_m1", 1, 4096, 1376, 4, 4096, 16, 1),       # the four-wave GEMV kernel: 4-vectors, 16-bit codes, 4096 entries
    ("gemv4_c3_weights_m2", 2, 4096, 1376, 4, 4096, 16, 1),
    ("gemv4_v4_u8_m1", 1, 2048, 2048, 4, 256, 8, 4),
    ("gemv4_v4_u8_m2", 2, 4096, 1024, 4, 256, 8, 1),
    ("gemv4_v8_u8_few_rows_m2", 2, 4096, 2048, 8, 256, 8, 2),    # a quarter of a row per wave
    ("gemv4_v2_u8_m1", 1, 2048, 512, 2, 256, 8, 1),
    ("odd_k_scalar_only", 5, 72, 64, 8, 256, 8, 1),
]


@pytest.mark.parametrize("row", GATED_B, ids=[r[0] for r in GATED_B])
def test_gated_epilogue_against_the_oracle(row):
    name, M, K, N, v, E, bits, G = row
    spec = ProblemSpec(name, GEOM_B, M, K, N, v, E, G, bits, codebook_3d=(G > 1), codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=51, device=DEV)
    bias = (torch.randn(N, generator=torch.Generator().manual_seed(52)) * 0.5).half().to(DEV)
    ws = torch.empty(M, N, dtype=torch.float16, device=DEV)
    want = vo.gated_gemm_b(_np(x), _np(codes), _np(cb)).astype(np.float64)
    want_b = vo.gated_gemm_b(_np(x), _np(codes), _np(cb), _np(bias)).astype(np.float64)
    ran = []
    for variant in (cabi.VARIANT_AUTO, cabi.VARIANT_GENERIC, cabi.VARIANT_PREFILL, cabi.VARIANT_PREFILL_NARROW,
                    cabi.VARIANT_PREFILL_SMALL, cabi.VARIANT_DECODE_GEMV, cabi.VARIANT_TWOPASS, cabi.VARIANT_DECODE):
        for b, ref in ((None, want), (bias, want_b)):
            _say("gated", name, cabi.VARIANT_NAMES[variant], "bias" if b is not None else "")
            try:
                y = cabi.e2e_gemm_b_gated(x, codes, cb, variant=variant, bias=b, workspace=ws)
            except cabi.VqGemmError as e:
                assert e.code == -4 and variant not in (cabi.VARIANT_AUTO, cabi.VARIANT_GENERIC, cabi.VARIANT_TWOPASS), e
                continue
            torch.cuda.synchronize()
            assert y.shape == (M, N // 2)
            # Bar: the error over the largest output within 2e-3 as for the GEMM itself; element by element (with the
            # floor) twice that: an output is a product of two fp32 sums, each with the GEMM's own error, and where the
            # gate is near zero its slope turns the sum's absolute error into a relative one of the (small) product.
            # The two-pass route also rounds the product to fp16 before the gate.
            e1, e2 = vo.rel_err(_np(y), ref)
            _say(f"    rel_err(floor)={e1:.3e} max/max={e2:.3e}")
            assert e2 <= TOL and e1 <= 2 * TOL, (name, variant, e1, e2)
            ran.append(variant)
    assert cabi.VARIANT_AUTO in ran and cabi.VARIANT_GENERIC in ran
    if name.startswith("decode_"):
        assert cabi.VARIANT_DECODE in ran
    if name.startswith("gemv"):
        assert cabi.VARIANT_DECODE_GEMV in ran
    if name.startswith("gemv4") or name.startswith("decode_general"):
        # no gated call needs a workspace: the automatic choice without one is a decode kernel with its own epilogue
        g, e, vv = cabi._cb_dims(cb)
        assert cabi.select_variant_b(M, K, N, vv, e, g, bits) in (cabi.VARIANT_DECODE, cabi.VARIANT_DECODE_GEMV)
    if name.endswith("_tile") or "tile_" in name:
        assert cabi.VARIANT_PREFILL in ran
    # without a workspace the automatic choice answers the same way (no kernel needs one), and the same twice
    y0 = cabi.e2e_gemm_b_gated(x, codes, cb)
    e1, e2 = vo.rel_err(_np(y0), want)
    assert e2 <= TOL and e1 <= 2 * TOL and torch.equal(cabi.e2e_gemm_b_gated(x, codes, cb), y0)


def test_gated_epilogue_equals_the_plain_product_followed_by_the_gate():
    """The fused epilogue against this library's own plain product: gate and up sums are the same fp32 numbers, so
    silu(gate) * up computed from the unfused product (rounded to fp16 in between) sits within an fp16 step."""
    spec = ProblemSpec("pair", GEOM_B, 384, 1024, 2048, 8, 256, 4, 8, codebook_3d=True, codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=53, device=DEV)
    fused = cabi.e2e_gemm_b_gated(x, codes, cb)
    p = cabi.e2e_gemm_b(x, codes, cb).float().view(384, 2048 // 32, 2, 16)
    g, u = p[:, :, 0, :].reshape(384, 1024), p[:, :, 1, :].reshape(384, 1024)
    unfused = torch.nn.functional.silu(g) * u
    scale = unfused.abs().max().item()
    assert ((fused.float() - unfused).abs().max() / scale).item() <= TOL
    # rejections: rows of W that are no whole pairs; a null output
    with pytest.raises(ValueError):
        cabi.e2e_gemm_b_gated(x, codes[:2048 - 16].contiguous(), cb[:1].contiguous())


def test_gated_mlp_module_with_interleaved_rows():
    from vq_gemm_amd.nn import VQGatedMLP, VQLinear
    from vq_gemm_amd.quantize import interleave_gate_up
    K, H = 512, 768
    s_g = ProblemSpec("g", GEOM_B, 1, K, H, 8, 256, 1, 8, codebook_std=0.05)
    s_d = ProblemSpec("d", GEOM_B, 1, H, K, 8, 256, 1, 8, codebook_std=0.05)
    _, c_g, cb_gu = make_problem(s_g, seed=31, device=DEV)
    _, c_u, _ = make_problem(s_g, seed=33, device=DEV)
    _, c_d, cb_d = make_problem(s_d, seed=32, device=DEV)
    codes = interleave_gate_up(c_g, c_u)
    assert np.array_equal(_np(codes), vo.interleave_gate_up(_np(c_g), _np(c_u)))
    mlp = VQGatedMLP(VQLinear(codes, cb_gu), VQLinear(c_d, cb_d), interleaved=True)
    stacked = VQGatedMLP(VQLinear(torch.cat([c_g, c_u]), cb_gu), VQLinear(c_d, cb_d))
    w_d = vo.dequant_b(_np(c_d), _np(cb_d)).astype(np.float64)
    for M in (1, 3, 200):
        x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).half().to(DEV)
        _say("gated mlp, interleaved", M)
        y = mlp(x)
        torch.cuda.synchronize()
        h = vo.gated_gemm_b(_np(x), _np(codes), _np(cb_gu))
        ref = h.astype(np.float64) @ w_d.T
        e1, e2 = vo.rel_err(_np(y), ref)
        _say(f"  M={M}: rel_err(floor)={e1:.3e} max/max={e2:.3e}")
        # (a chain with an fp16 tensor in the middle: held to the bound on the largest output, as the stacked module's test)
        assert e2 <= TOL and e1 <= 0.25, (e1, e2)
        # the stacked layout with the element-wise kernel computes the same layer
        ys = stacked(x)
        assert ((y.float() - ys.float()).abs().max() / ys.float().abs().max()).item() <= 2 * TOL


# ------------------------------------------------------------------ split K over the 128x128 tiles
SPLITK_B = [
    # name, M, K, N, vec, E, bits, G
    ("mid_m_few_columns", 512, 4096, 4096, 8, 256, 8, 32),      # the shape the cost model was fitted on
    ("ragged_m_and_n", 300, 2048, 1000, 8, 256, 8, 1),          # Y rows not 16-byte aligned: the plain epilogue
    ("u16_v4_books", 200, 1024, 768, 4, 4096, 16, 3),
    ("v2", 129, 512, 256, 2, 256, 8, 1),
    ("one_tile", 64, 4096, 128, 8, 256, 8, 1),
    ("many_tiles", 1024, 1024, 2048, 8, 256, 8, 16),            # more workgroups than fit the device at once
]


@pytest.mark.parametrize("row", SPLITK_B, ids=[r[0] for r in SPLITK_B])
def test_split_k_against_the_oracle_and_from_run_to_run(row):
    name, M, K, N, v, E, bits, G = row
    spec = ProblemSpec(name, GEOM_B, M, K, N, v, E, G, bits, codebook_3d=(G > 1), codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=61, device=DEV)
    bias = (torch.randn(N, generator=torch.Generator().manual_seed(62)) * 0.5).half().to(DEV)
    # (the unrounded float64 product: the bias is added before the one rounding)
    want = _np(x).astype(np.float64) @ vo.dequant_b(_np(codes), _np(cb)).astype(np.float64).T
    need = cabi.workspace_bytes_b(M, K, N, v, E, G, bits, cabi.VARIANT_PREFILL_SPLITK)
    assert need > 0, "every shape of this list has a split"
    # the workspace's contents before the call do not matter: start from garbage
    ws = torch.empty(need, dtype=torch.uint8, device=DEV).random_()
    for b, ref in ((None, want), (bias, want + _np(bias).astype(np.float64)[None, :])):
        _say("split-k", name, "bias" if b is not None else "")
        y = cabi.e2e_gemm_b_ws(x, codes, cb, variant=cabi.VARIANT_PREFILL_SPLITK, workspace=ws, bias=b).clone()
        torch.cuda.synchronize()
        e1, e2 = vo.rel_err(_np(y), ref)
        _say(f"    rel_err(floor)={e1:.3e} max/max={e2:.3e}")
        assert e1 <= TOL, (name, e1, e2)
        # the partial sums are added in the order of the slices whoever finishes last: the same bits every time
        for _ in range(4):
            ws.random_()
            assert torch.equal(cabi.e2e_gemm_b_ws(x, codes, cb, variant=cabi.VARIANT_PREFILL_SPLITK, workspace=ws, bias=b), y)
    # and close to the unsplit kernel (the same fp32 products, summed in another order)
    y1 = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_PREFILL_SMALL)
    y2 = cabi.e2e_gemm_b_ws(x, codes, cb, variant=cabi.VARIANT_PREFILL_SPLITK, workspace=ws)
    assert vo.rel_err(_np(y2), _np(y1).astype(np.float64))[0] <= 2e-3
    # a workspace that is too small: an error for the explicit variant, no obstacle for the automatic choice
    small = torch.empty(256, dtype=torch.uint8, device=DEV)
    with pytest.raises(cabi.VqGemmError) as err:
        cabi.e2e_gemm_b_ws(x, codes, cb, variant=cabi.VARIANT_PREFILL_SPLITK, workspace=small)
    assert err.value.code == -6
    ya = cabi.e2e_gemm_b_ws(x, codes, cb, workspace=small)
    assert vo.rel_err(_np(ya), want)[0] <= TOL


# Whole rounds of large tiles over the first columns of W, the left-over columns in 128x128 tiles with K split: shapes
# whose large tiles are a few more than a round on a 256-unit device (K kept short: the oracle multiplies all of it).
TAIL_SPLIT_B = [
    # name, M, K, N, vec, E, bits, G
    ("wide_head_258_tiles", 1536, 512, 11008, 8, 256, 8, 1),
    ("narrow_head_258_tiles_86_books", 768, 1024, 11008, 8, 256, 8, 86),
    ("ragged_m_and_last_column", 1500, 512, 11008 + 72, 8, 256, 8, 1),
    ("u16_v4", 1536, 512, 11008, 4, 1024, 16, 2),
]


@pytest.mark.parametrize("row", TAIL_SPLIT_B, ids=[r[0] for r in TAIL_SPLIT_B])
def test_whole_rounds_of_large_tiles_then_the_left_over_columns_with_k_split(row):
    name, M, K, N, v, E, bits, G = row
    spec = ProblemSpec(name, GEOM_B, M, K, N, v, E, G, bits, codebook_3d=(G > 1), codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=71, device=DEV)
    bias = (torch.randn(N, generator=torch.Generator().manual_seed(72)) * 0.5).half().to(DEV)
    w = vo.dequant_b(_np(codes), _np(cb)).astype(np.float64)
    xf = _np(x).astype(np.float64)
    want = np.concatenate([xf @ w[r:r + 2048].T for r in range(0, N, 2048)], axis=1)
    before = cabi.tuning()
    try:
        cabi.set_tuning(tail_split_margin=0.0)
        y_single = cabi.e2e_gemm_b_ws(x, codes, cb).clone()           # the best single plan
        cabi.set_tuning(tail_split_margin=1e6, splitk_force_splits=2) # the two-launch plan wherever it exists, K in two slices
        need = cabi.workspace_bytes_b(M, K, N, v, E, G, bits)
        assert need > 0, "every shape of this list leaves columns over, and K can be split there"
        ws = torch.empty(need, dtype=torch.uint8, device=DEV).random_()
        for b, ref in ((None, want), (bias, want + _np(bias).astype(np.float64)[None, :])):
            _say("tail split", name, "bias" if b is not None else "")
            y = cabi.e2e_gemm_b_ws(x, codes, cb, workspace=ws, bias=b).clone()
            torch.cuda.synchronize()
            e1, e2 = vo.rel_err(_np(y), ref)
            _say(f"    rel_err(floor)={e1:.3e} max/max={e2:.3e}")
            assert e1 <= TOL, (name, e1, e2)
            for _ in range(3):   # the same bits whoever finishes last, whatever the workspace held
                ws.random_()
                assert torch.equal(cabi.e2e_gemm_b_ws(x, codes, cb, workspace=ws, bias=b), y)
        # the columns of the first launch are the single plan's bits where that plan used the same tiles; all of Y is close
        y2 = cabi.e2e_gemm_b_ws(x, codes, cb, workspace=ws)
        assert vo.rel_err(_np(y2), _np(y_single).astype(np.float64))[0] <= 2e-3
        # (it is this plan that ran: K split over every tile would need a slot per tile and slice)
        assert need < cabi.workspace_bytes_b(M, K, N, v, E, G, bits, cabi.VARIANT_PREFILL_SPLITK) // 4
        # a workspace that is too small is no obstacle: the automatic choice does without
        ya = cabi.e2e_gemm_b_ws(x, codes, cb, workspace=torch.empty(256, dtype=torch.uint8, device=DEV))
        assert vo.rel_err(_np(ya), want)[0] <= TOL
    finally:
        cabi.set_tuning(**before)


def test_split_k_gives_the_same_bits_whatever_the_workspace_held():
    # Every partial sum is written before the second launch reads it, and the slices are added in order.
    M, K, N = 512, 4096, 4096
    spec = ProblemSpec("splitk_bits", GEOM_B, M, K, N, 8, 256, 32, 8, codebook_3d=True, codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=67, device=DEV)
    need = cabi.workspace_bytes_b(M, K, N, 8, 256, 32, 8, cabi.VARIANT_PREFILL_SPLITK)
    ws = torch.empty(need, dtype=torch.uint8, device=DEV).random_()
    first = cabi.e2e_gemm_b_ws(x, codes, cb, variant=cabi.VARIANT_PREFILL_SPLITK, workspace=ws).clone()
    for _ in range(3):
        ws.random_()
        assert torch.equal(cabi.e2e_gemm_b_ws(x, codes, cb, variant=cabi.VARIANT_PREFILL_SPLITK, workspace=ws), first)


def test_split_k_is_what_the_automatic_choice_takes_for_medium_m_on_few_columns_and_only_with_a_workspace():
    M, K, N = 954, 14080, 1920
    spec = ProblemSpec("auto_split", GEOM_B, M, K, N, 8, 256, 15, 8, codebook_3d=True, codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=63, device=DEV)
    dims = (M, K, N, 8, 256, 15, 8)
    need = cabi.workspace_bytes_b(*dims)
    assert need > 0 and cabi.auto_variant_name_b(*dims, need) == "prefill_splitk" != cabi.auto_variant_name_b(*dims)
    want = vo.vq_gemm_b(_np(x), _np(codes), _np(cb), acc=np.float64)
    y_plain = cabi.e2e_gemm_b(x, codes, cb)                      # no workspace: the unsplit choice
    y_split = cabi.e2e_gemm_b_ws(x, codes, cb)                   # allocates what workspace_bytes_b says
    assert vo.rel_err(_np(y_plain), want)[0] <= TOL and vo.rel_err(_np(y_split), want)[0] <= TOL
    # where a split cannot pay the automatic choice wants no workspace: one row of X, a full device of large tiles
    assert cabi.workspace_bytes_b(1, 4096, 4096, 8, 256, 1, 8) == 0 and cabi.workspace_bytes_b(14, 512, 768, 8, 256, 3, 8) == 0
    assert cabi.workspace_bytes_b(4096, 4096, 4096, 8, 256, 32, 8) == 0
    # the kernels that were named are the ones that ran: the bits of the variants asked for
    ws = torch.empty(max(need, cabi.workspace_bytes_b(*dims, cabi.VARIANT_PREFILL_SPLITK)), dtype=torch.uint8, device=DEV)
    assert torch.equal(y_split, cabi.e2e_gemm_b_ws(x, codes, cb, variant=cabi.VARIANT_PREFILL_SPLITK, workspace=ws))
    assert torch.equal(y_plain, cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_WAVE_K))
    # captured into a graph and replayed (the counters are cleared by a kernel, not a memset node)
    out = torch.empty(M, N, dtype=torch.float16, device=DEV)
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        cabi.e2e_gemm_b_ws(x, codes, cb, workspace=ws, out=out)
        st.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=st):
            cabi.e2e_gemm_b_ws(x, codes, cb, workspace=ws, out=out)
        for _ in range(3):
            out.zero_()
            torch.cuda.synchronize()
            g.replay()
            st.synchronize()
            assert torch.equal(out, y_split)


def test_split_k_calls_on_two_streams_with_a_workspace_each_do_not_disturb_each_other():
    M, K, N = 384, 4096, 4096
    spec = ProblemSpec("two_streams", GEOM_B, M, K, N, 8, 256, 32, 8, codebook_3d=True, codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=71, device=DEV)
    x2 = (x * 0.5).contiguous()
    need = cabi.workspace_bytes_b(M, K, N, 8, 256, 32, 8, cabi.VARIANT_PREFILL_SPLITK)
    ws = [torch.empty(need, dtype=torch.uint8, device=DEV).random_() for _ in range(2)]
    want = [cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_GENERIC), cabi.e2e_gemm_b(x2, codes, cb, variant=cabi.VARIANT_GENERIC)]
    ref = [cabi.e2e_gemm_b_ws(xx, codes, cb, variant=cabi.VARIANT_PREFILL_SPLITK, workspace=ws[0]).clone() for xx in (x, x2)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]   # default priority
    outs = [torch.empty(M, N, dtype=torch.float16, device=DEV) for _ in range(2)]
    for _ in range(20):
        for i, (st, xx) in enumerate(zip(streams, (x, x2))):
            with torch.cuda.stream(st):
                cabi.e2e_gemm_b_ws(xx, codes, cb, variant=cabi.VARIANT_PREFILL_SPLITK, workspace=ws[i], out=outs[i])
    torch.cuda.synchronize()
    for i in range(2):
        assert torch.equal(outs[i], ref[i])
        assert vo.rel_err(_np(outs[i]), _np(want[i]).astype(np.float64))[0] <= 2 * TOL


def test_sized_workspace_entry_point_passes_the_other_variants_through():
    spec = ProblemSpec("ws_passthrough", GEOM_B, 48, 512, 256, 8, 256, 1, 8, codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=72, device=DEV)
    y0 = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE)
    assert torch.equal(cabi.e2e_gemm_b_ws(x, codes, cb, variant=cabi.VARIANT_DECODE), y0)
    # the two-pass route takes its scratch from the sized workspace, and says so when it is too small
    y2 = cabi.e2e_gemm_b_ws(x, codes, cb, variant=cabi.VARIANT_TWOPASS)
    assert vo.rel_err(_np(y2), _np(y0).astype(np.float64))[0] <= 2 * TOL
    with pytest.raises(cabi.VqGemmError) as err:
        cabi.e2e_gemm_b_ws(x, codes, cb, variant=cabi.VARIANT_TWOPASS, workspace=torch.empty(1024, dtype=torch.uint8, device=DEV))
    assert err.value.code == -6
    # split K is refused where no slice of K is long enough
    with pytest.raises(cabi.VqGemmError) as err:
        cabi.e2e_gemm_b_ws(x[:, :128].contiguous(), codes[:, :16].contiguous(), cb, variant=cabi.VARIANT_PREFILL_SPLITK,
                           workspace=torch.empty(1 << 20, dtype=torch.uint8, device=DEV))
    assert err.value.code == -4


RAGGED_B = [
    # name, M, K, N, vec, E, bits: K that ends inside a code tile or a K slice, N that ends inside a tile
    ("shortest", 16, 192, 16, 8, 256, 8),
    ("one_lane_load_over", 3, 320, 33, 8, 256, 8),
    ("three_lane_loads_over", 16, 2240, 47, 8, 200, 8),
    ("two_chunks_of_k", 5, 4160, 130, 8, 256, 8),
    ("slabs", 70, 1088, 1000, 8, 256, 8),
    ("many_tiles", 17, 576, 9001, 8, 256, 8),
    ("split_k", 130, 2880, 264, 8, 256, 8),
    ("prefill", 300, 1984, 520, 8, 256, 8),
    ("v8_u16", 9, 448, 50, 8, 700, 16),
    ("v4_u8", 12, 832, 61, 4, 256, 8),
    ("v4_u16", 16, 4288, 77, 4, 4096, 16),
]


@pytest.mark.parametrize("row", RAGGED_B, ids=[r[0] for r in RAGGED_B])
def test_widths_that_are_no_multiple_of_a_tile_or_a_slice(row):
    name, M, K, N, v, E, bits = row
    spec = ProblemSpec(name, GEOM_B, M, K, N, v, E, 1, bits, codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=81, device=DEV)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(3)).half().to(DEV)
    want = _np(x).astype(np.float64) @ vo.dequant_b(_np(codes), _np(cb)).astype(np.float64).T
    ran = []
    for variant in (cabi.VARIANT_AUTO, cabi.VARIANT_DECODE, cabi.VARIANT_PREFILL, cabi.VARIANT_PREFILL_NARROW, cabi.VARIANT_PREFILL_SMALL,
                    cabi.VARIANT_PREFILL_SPLITK):
        for b in (None, bias):
            _say(name, M, K, N, "variant", cabi.VARIANT_NAMES[variant], "bias", b is not None)
            try:
                y = cabi.e2e_gemm_b_ws(x, codes, cb, variant=variant, bias=b)
            except cabi.VqGemmError as e:
                assert e.code == -4
                continue
            torch.cuda.synchronize()
            e1, _ = vo.rel_err(_np(y), want if b is None else want + _np(b).astype(np.float64))
            assert e1 <= TOL, (name, variant, e1)
            ran.append(variant)
    assert {cabi.VARIANT_AUTO, cabi.VARIANT_DECODE, cabi.VARIANT_PREFILL} <= set(ran)
    assert cabi.VARIANT_PREFILL_SPLITK in ran or name != "split_k"
    if N >= 32:  # the gated epilogue on the same widths
        n = N // 32 * 32
        y = cabi.e2e_gemm_b_gated(x, codes[:n].contiguous(), cb)
        torch.cuda.synchronize()
        e1, e2 = vo.rel_err(_np(y), vo.gated_gemm_b(_np(x), _np(codes)[:n], _np(cb)).astype(np.float64))
        assert e2 <= TOL and e1 <= 2 * TOL, (name, "gated", e1, e2)


# K that ends inside a slice, a code tile or a unit, in every format; fewer than 16 columns and K % 64 = 32, which the general decode kernel takes
@pytest.mark.parametrize("M,K,N,v,entries,bits,G", [(5, 320, 48, 8, 256, 8, 1), (16, 2240, 33, 8, 100, 8, 1), (40, 4160, 80, 8, 256, 8, 1), (9, 448, 50, 8, 700, 16, 1),
                                                    (12, 832, 61, 4, 256, 8, 1), (16, 4288, 77, 4, 1024, 16, 1), (7, 576, 40, 2, 256, 8, 1), (3, 320, 32, 2, 300, 16, 1),
                                                    (5, 384, 8, 8, 256, 8, 1), (16, 1120, 48, 4, 300, 16, 3), (20, 4384, 33, 4, 300, 16, 1), (130, 1984, 160, 8, 256, 8, 1), (70, 416, 96, 4, 256, 8, 1)])
def test_infinite_codewords_reach_their_own_rows_only_and_as_infinities(M, K, N, v, entries, bits, G):
    """Entry 0 is infinite and selected nowhere, entry 1 by the first code of every third row: with positive X those rows are +inf, as
    the definition has them, and all others finite.  What a kernel multiplies beyond K must not bring either in."""
    spec = ProblemSpec("inf", GEOM_B, M, K, N, v, entries, G, bits, codebook_3d=(G > 1), codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=96, device=DEV)
    x = (x.float().abs() + 0.1).half()
    c = codes.to(torch.int32)
    c = torch.where(c < 2, torch.full_like(c, 2), c)
    c[::3, 0] = 1
    codes = c.to(codes.dtype)
    cb[..., :2, :] = float("inf")
    w = vo.dequant_b(_np(codes), _np(cb)).astype(np.float64)
    hit = np.zeros(N, bool)
    hit[::3] = True
    want = _np(x).astype(np.float64) @ w[~hit].T
    ran = []
    for variant in (cabi.VARIANT_AUTO, cabi.VARIANT_GENERIC, cabi.VARIANT_DECODE, cabi.VARIANT_PREFILL, cabi.VARIANT_PREFILL_NARROW,
                    cabi.VARIANT_PREFILL_SMALL, cabi.VARIANT_PREFILL_SPLITK, cabi.VARIANT_WAVE_K):
        _say("infinite codewords", M, K, N, v, entries, bits, G, cabi.VARIANT_NAMES[variant])
        try:
            y = _np(cabi.e2e_gemm_b_ws(x, codes, cb, variant=variant))
        except cabi.VqGemmError as e:
            assert e.code == -4
            continue
        assert np.isposinf(y[:, hit]).all(), (variant, int(np.isnan(y[:, hit]).sum()))
        assert vo.rel_err(y[:, ~hit], want)[0] <= TOL, variant
        ran.append(variant)
    assert cabi.VARIANT_GENERIC in ran and (M > 64 or cabi.VARIANT_DECODE in ran)


@pytest.mark.parametrize("K,N,v,E,G,gated", [(8192, 48, 4, 256, 1, False), (8192, 64, 4, 200, 2, True), (4096, 48, 4, 4096, 3, False), (6144, 32, 8, 300, 1, False),
                                             (8192, 32, 4, 1000, 1, True), (6144, 32, 4, 256, 1, False), (2048, 16, 8, 300, 1, False)])
def test_gemv_kernel_products_of_the_diagonal(K, N, v, E, G, gated):
    bits = 8 if E <= 256 else 16
    spec = ProblemSpec("diag4", GEOM_B, 1, K, N, v, E, G, bits, codebook_3d=(G > 1), codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=99, device=DEV)
    _say("gemv diagonal", K, N, v, E, G, gated)
    if gated:
        e1, e2 = vo.rel_err(_np(cabi.e2e_gemm_b_gated(x, codes, cb, variant=cabi.VARIANT_DECODE_GEMV)), vo.gated_gemm_b(_np(x), _np(codes), _np(cb)).astype(np.float64))
        assert e2 <= TOL and e1 <= 2 * TOL   # (a product of two sums, as in test_gated_epilogue_against_the_oracle)
        return
    w = vo.dequant_b(_np(codes), _np(cb))
    y = cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_DECODE_GEMV)
    assert vo.rel_err(_np(y), _np(x).astype(np.float64) @ w.astype(np.float64).T)[0] <= TOL
    for c in (0, K // 2 + 3, K - 1):
        eye = torch.zeros(1, K, dtype=torch.float16, device=DEV)
        eye[0, c] = 1.0
        yw = cabi.e2e_gemm_b(eye, codes, cb, variant=cabi.VARIANT_DECODE_GEMV)
        assert np.array_equal(_np(yw).view(np.uint16), w[:, [c]].T.copy().view(np.uint16)), c


# rows of X, K, N, codebooks, gated: products on the matrix cores or not, by rows per wave (4096 of them), pieces of a row and codebook boundaries
@pytest.mark.parametrize("M,K,N,G,gated", [(1, 2048, 8200, 1, False), (1, 2048, 12289, 1, False), (1, 4096, 4097, 1, False), (1, 4096, 16383, 3, False), (1, 8192, 8193, 1, False),
                                         (1, 4096, 96, 1, True), (1, 2048, 16416, 1, True), (1, 4096, 24608, 1, True), (1, 8192, 8224, 257, True), (1, 6144, 8192, 8, True),
                                         (1, 8224, 4096, 1, False), (1, 12288, 4097, 1, False), (1, 16384, 4096, 1, False), (1, 24576, 130, 1, False),
                                         (1, 26624, 130, 1, False), (1, 11008, 8192, 2, False), (1, 14336, 300, 1, False), (1, 11008, 5003, 1, False), (1, 8192, 10241, 1, False),
                                         (1, 4096, 1001, 1, False), (1, 6144, 33, 1, False), (1, 8192, 9248, 1, True), (2, 4096, 8193, 1, False), (2, 4096, 24608, 1, True), (2, 2048, 8224, 1, True),
                                           (2, 11008, 4100, 1, False), (2, 16384, 300, 1, False), (2, 4096, 8192, 2, False), (2, 4096, 28672, 1, False),
                                           # (ten runs a wave and hardly more; six with two rows of X)
                                           (1, 4096, 20480, 1, False), (1, 4096, 20481, 1, False), (1, 4096, 20544, 3, True), (1, 8192, 10248, 2, False),
                                           (1, 6144, 13672, 1, False), (1, 11008, 6840, 1, False), (2, 8192, 10241, 1, False), (2, 4096, 12289, 1, False)])
def test_gemv_wide_form_products_of_the_diagonal(M, K, N, G, gated):
    spec = ProblemSpec("diag", GEOM_B, M, K, N, 8, 256, G, 8, codebook_3d=(G > 1), codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=98, device=DEV)
    _say("gemv diagonal", M, K, N, G, gated)
    bias = torch.linspace(-1, 1, N, device=DEV).half()
    if gated:
        y = cabi.e2e_gemm_b_gated(x, codes, cb, bias=bias)
        e1, e2 = vo.rel_err(_np(y), vo.gated_gemm_b(_np(x), _np(codes), _np(cb), _np(bias)).astype(np.float64))
        assert e2 <= TOL and e1 <= 2 * TOL   # (a product of two sums, as in test_gated_epilogue_against_the_oracle)
        return
    assert cabi.select_variant_b(M, K, N, 8, 256, G, 8) == cabi.VARIANT_DECODE_GEMV
    y = cabi.e2e_gemm_b(x, codes, cb, bias=bias)
    w = vo.dequant_b(_np(codes), _np(cb))
    want = _np(x).astype(np.float64) @ w.astype(np.float64).T + _np(bias).astype(np.float64)
    assert vo.rel_err(_np(y), want)[0] <= TOL
    # a one-hot x reads W out bit for bit, subnormal halves too
    cb = cb.clone()
    cb[..., 3, :], cb[..., 5, :] = 6e-8, 3e-5
    w = vo.dequant_b(_np(codes), _np(cb))
    for c in (0, 5, K // 2 + 3, K - 1):
        eye = torch.zeros(M, K, dtype=torch.float16, device=DEV)
        cols = [c, (c + 9) % K][:M]
        eye[torch.arange(M), torch.tensor(cols)] = 1.0
        assert np.array_equal(_np(cabi.e2e_gemm_b(eye, codes, cb)).view(np.uint16), w[:, cols].T.copy().view(np.uint16)), c


@pytest.mark.parametrize("M,K,N,G", [(1, 2080, 48, 1), (2, 2080, 33, 1), (1, 8224, 64, 1), (2, 6176, 4096, 1), (1, 14336, 40, 1), (2, 14336, 2048, 1), (1, 4096, 32, 1)])
def test_a_row_that_ends_in_an_infinite_codeword_is_infinite_in_the_gemv_kernels(M, K, N, G):
    """The long form reads a row's last codes once more where K ends inside a piece of it."""
    spec = ProblemSpec("inf", GEOM_B, M, K, N, 8, 256, G, 8, codebook_3d=(G > 1), codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=97, device=DEV)
    x = (x.float().abs() + 0.1).half()
    c = codes.to(torch.int32)
    c = torch.where(c < 2, torch.full_like(c, 2), c)
    c[::3, -1] = 1
    c[1, 0], c[1, 1] = 0, 1                    # plus and minus infinity meet: NaN by the definition
    codes = c.to(codes.dtype)
    cb[..., 0, :], cb[..., 1, :] = -float("inf"), float("inf")
    w = vo.dequant_b(_np(codes), _np(cb)).astype(np.float64)
    hit, plain = np.zeros(N, bool), np.ones(N, bool)
    hit[::3] = True
    plain[::3] = plain[1] = False
    want = _np(x).astype(np.float64) @ w[plain].T
    bias = torch.ones(N, dtype=torch.float16, device=DEV)
    for variant in (cabi.VARIANT_DECODE_GEMV, cabi.VARIANT_AUTO, cabi.VARIANT_GENERIC):
        _say("infinite last codewords", M, K, N, G, cabi.VARIANT_NAMES[variant])
        y = _np(cabi.e2e_gemm_b(x, codes, cb, variant=variant, bias=bias))
        assert np.isposinf(y[:, hit]).all() and np.isnan(y[:, 1]).all(), (variant, int(np.isnan(y[:, hit]).sum()))
        assert vo.rel_err(y[:, plain], want + 1.0)[0] <= TOL, variant


LLOYD_B = [
    # N, K, vec, entries, G: codebooks in several workgroups, entries nothing is assigned to, a last tile of entries cut short
    (512, 1024, 8, 256, 2),
    (48, 264, 8, 33, 1),
    (96, 128, 4, 700, 3),
    (10, 64, 2, 5, 5),
    (8, 32, 8, 64, 1),      # fewer vectors than entries
]


@pytest.mark.parametrize("row", LLOYD_B, ids=["x".join(map(str, r)) for r in LLOYD_B])
def test_lloyd_iterations_on_the_device_against_the_definition(row):
    from vq_gemm_amd.quantize import _initial_vectors
    from vq_gemm_amd.torch_ops import native
    N, K, v, E, G = row
    _say("lloyd", row)
    g = torch.Generator(device="cpu").manual_seed(7)
    w = (torch.randn(N, K, generator=g) * 0.05).half().to(DEV)
    bits = 8 if E <= 256 else 16
    per_cb = N // G * (K // v)
    pick = _initial_vectors(per_cb, E, G, 3)
    vectors = _np(w).reshape(G, per_cb, v)
    book = np.stack([vectors[i][pick[i].numpy()] for i in range(G)])
    for iters in (0, 1, 2):
        codes, cb, errors = native.kmeans(w, pick, v, E, G, bits, iters)
        torch.cuda.synchronize()
        # the codes are the encoder's for the codebook returned, the last error is theirs
        assert torch.equal(codes, cabi.encode_b(w, cb, bits))
        c = _np(codes).astype(np.int64).reshape(G, per_cb)
        got = _np(cb)
        sq = sum(((got[i][c[i]].astype(np.float64) - vectors[i].astype(np.float64)) ** 2).sum() for i in range(G))
        assert errors.shape == (iters + 1,) and float(errors[-1]) == pytest.approx(sq, rel=1e-5, abs=1e-12)
        if iters == 0:
            assert np.array_equal(got, book)
        elif iters == 1:
            # the update of the first assignment: means in float64, an fp16 last place for the order of the fp32 sums
            c0 = c_oracle.encode_b(_np(w), book, bits).astype(np.int64).reshape(G, per_cb)
            for i in range(G):
                for e in range(E):
                    mine = vectors[i][c0[i] == e].astype(np.float64)
                    if len(mine) == 0:
                        assert np.array_equal(got[i, e], book[i, e])
                    else:
                        assert np.allclose(got[i, e].astype(np.float64), mine.mean(axis=0), rtol=1.1e-3, atol=1e-6)


@pytest.mark.parametrize("M,K,N,v,entries,stages,bits", [(5, 4096, 80, 8, 256, 2, 16), (16, 320, 50, 8, 100, 3, 16), (3, 4160, 33, 8, 128, 2, 8),
                                                         (20, 2048, 64, 4, 256, 4, 16), (1, 2048, 64, 8, 128, 2, 8), (130, 512, 72, 8, 128, 2, 8)])
def test_stages_multiply_the_same_x_without_a_copy_of_it(M, K, N, v, entries, stages, bits):
    from vq_gemm_amd.nn import VQLinear
    _say("stages", M, K, N, v, entries, stages)
    spec = ProblemSpec("stages", GEOM_B, M, stages * K, N, v, stages * entries, 1, bits, codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=17, device=DEV)
    x = x[:, :K].contiguous()
    bias = torch.randn(N, generator=torch.Generator().manual_seed(1)).half().to(DEV)
    for b in (None, bias):
        y = VQLinear(codes, cb, b, k_repeat=stages)(x)
        torch.cuda.synchronize()
        assert torch.equal(y, cabi.e2e_gemm_b_ws(x.repeat(1, stages), codes, cb, bias=b))


# shapes whose stages need no copy of x (decode kernel, wave-K kernel), and one that needs it (tall X); every operand begins off
# its alignment in turn, codes and codebook as slices of larger tensors like the bias
@pytest.mark.parametrize("M,K,N,v,entries,stages,bits", [(5, 4096, 80, 8, 128, 2, 8), (20, 2048, 64, 4, 256, 4, 16), (130, 512, 72, 8, 128, 2, 8)])
@pytest.mark.parametrize("which", ["bias", "codes", "codebook"])
def test_stages_take_operands_that_begin_anywhere(M, K, N, v, entries, stages, bits, which):
    from vq_gemm_amd.nn import VQLinear
    _say("stages, unaligned", which, M, K, N, v, entries, stages)
    spec = ProblemSpec("stages", GEOM_B, M, stages * K, N, v, stages * entries, 1, bits, codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=18, device=DEV)
    x = x[:, :K].contiguous()
    bias = torch.randn(N, generator=torch.Generator().manual_seed(1)).half().to(DEV)

    def shifted(t):
        big = torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)
        big[1:] = t.reshape(-1)
        return big[1:].view(t.shape)

    operands = {"codes": codes, "codebook": cb, "bias": bias}
    operands[which] = shifted(operands[which])
    layer = VQLinear(operands["codes"], operands["codebook"], operands["bias"], k_repeat=stages)
    assert getattr(layer, which).data_ptr() % 8 != 0
    y = layer(x)
    torch.cuda.synchronize()
    want = _np(x.repeat(1, stages)).astype(np.float64) @ vo.dequant_b(_np(codes), _np(cb)).astype(np.float64).T + _np(bias).astype(np.float64)
    assert vo.rel_err(_np(y), want)[0] <= TOL
    # the scalar kernel on a copy: the same sums in the same order
    assert torch.equal(y, cabi.e2e_gemm_b(x.repeat(1, stages), codes, cb, variant=cabi.VARIANT_GENERIC, bias=bias))


def _with_wave_tile(tile, call):
    before = cabi.tuning()
    try:
        cabi.set_tuning(wave_k_force=1, wave_k_force_tile=tile)
        return call()
    finally:
        cabi.set_tuning(**{k: before[k] for k in ("wave_k_force", "wave_k_force_tile")})


@pytest.mark.parametrize("row", [
    # M, K, N, v, E, bits, G: one row, a row more and less than a tile, K of one and two code tiles and a half one, ragged columns,
    # a short codebook, tiles that meet several codebooks
    (1, 128, 8, 8, 256, 8, 1),
    (129, 192, 129, 8, 256, 8, 1),
    (160, 1088, 131, 8, 100, 8, 1),
    (161, 320, 288, 8, 256, 8, 3),
    (225, 704, 192, 8, 200, 8, 6),
    (193, 64, 160, 4, 256, 8, 1),
    (223, 448, 257, 4, 30, 8, 1),
    (192, 576, 96, 4, 256, 8, 3),
    (131, 64, 33, 8, 512, 16, 1),
    (257, 832, 160, 8, 700, 16, 2),
    (159, 128, 130, 4, 4096, 16, 1),
    (224, 960, 256, 4, 1024, 16, 2),
], ids=lambda r: "x".join(map(str, r)))
def test_prefill_tiles_with_a_compute_unit_to_themselves(row):
    M, K, N, v, E, bits, G = row
    spec = ProblemSpec("mid", GEOM_B, M, K, N, v, E, G, bits, codebook_3d=(G > 1), codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=95, device=DEV)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(7)).half().to(DEV)
    want = _np(x).astype(np.float64) @ vo.dequant_b(_np(codes), _np(cb)).astype(np.float64).T
    before = cabi.tuning()
    calls = {"plain": lambda v: cabi.e2e_gemm_b(x, codes, cb, variant=v), "bias": lambda v: cabi.e2e_gemm_b(x, codes, cb, variant=v, bias=bias)}
    if N % 32 == 0:
        calls["gated"] = lambda v: cabi.e2e_gemm_b_gated(x, codes, cb, variant=v, bias=bias)
    for special in (False, True):
        if special:   # what is not finite goes where the sums of the other tiles take it
            flat = cb.view(-1, v)
            flat[E - 1, 0], flat[E // 2, v - 1], flat[0, 1] = float("inf"), float("nan"), float("-inf")
        for what, call in calls.items():
            other = call(cabi.VARIANT_PREFILL_SMALL)   # the 128x128 tiles: the same sums in the same order
            for rows in (128, 160, 192, 224):
                _say("mid", row, special, what, "rows", rows)
                try:
                    cabi.set_tuning(prefill_mid_force=rows)
                    y = call(cabi.VARIANT_PREFILL)
                finally:
                    cabi.set_tuning(prefill_mid_force=before["prefill_mid_force"])
                torch.cuda.synchronize()
                assert torch.equal(y.view(torch.int16), other.view(torch.int16)), (row, rows, what)
                if not special and what == "plain":
                    assert vo.rel_err(_np(y), want)[0] <= TOL, (row, rows)


WAVE_K_B = [
    # M, K, N, vec, E, bits, G: fewer units of K than waves, a last unit shorter than its load, edges of every tile, tiles over
    # several codebooks, a column more than a tile
    (1, 128, 16, 8, 256, 8, 1),
    (17, 192, 32, 8, 256, 8, 1),
    (65, 1088, 129, 8, 256, 8, 1),
    (130, 832, 160, 8, 100, 8, 5),
    (64, 2112, 128, 8, 300, 16, 4),
    (33, 1216, 65, 4, 256, 8, 1),
    (100, 704, 192, 4, 256, 8, 6),
    (48, 960, 96, 4, 1024, 16, 2),
    (70, 1024, 257, 4, 4096, 16, 1),
]


@pytest.mark.parametrize("row", WAVE_K_B, ids=["x".join(map(str, r)) for r in WAVE_K_B])
def test_k_dealt_out_to_waves_geometry_b(row):
    M, K, N, v, E, bits, G = row
    spec = ProblemSpec("wave_k", GEOM_B, M, K, N, v, E, G, bits, codebook_3d=(G > 1), codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=91, device=DEV)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(4)).half().to(DEV)
    want = _np(x).astype(np.float64) @ vo.dequant_b(_np(codes), _np(cb)).astype(np.float64).T
    for tile in (12, 14, 18, 22, 24, 44, 48):
        _say("wave_k", row, "tile", tile)
        for b in (None, bias):
            y = _with_wave_tile(tile, lambda: cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_WAVE_K, bias=b))
            torch.cuda.synchronize()
            assert vo.rel_err(_np(y), want if b is None else want + _np(b).astype(np.float64))[0] <= TOL, (row, tile)
        if N % 32 == 0:
            y = _with_wave_tile(tile, lambda: cabi.e2e_gemm_b_gated(x, codes, cb, variant=cabi.VARIANT_WAVE_K, bias=bias))
            p = want + _np(bias).astype(np.float64)
            p = p.reshape(M, N // 32, 2, 16)
            gated = (p[:, :, 0] / (1 + np.exp(-p[:, :, 0])) * p[:, :, 1]).reshape(M, N // 2)
            torch.cuda.synchronize()
            assert vo.rel_err(_np(y), gated)[1] <= TOL, (row, tile, "gated")


@pytest.mark.parametrize("row", WAVE_K_B + [(81, 192, 80, 8, 256, 8, 1), (97, 1088, 66, 4, 16, 8, 1), (31, 128, 130, 8, 300, 16, 1)],
                         ids=lambda r: "x".join(map(str, r)))
def test_k_dealt_out_to_waves_tall_and_wide_tiles(row):
    """32 x 128, 48, 80 and 96 x 64: an odd number of rows of pieces, one step a unit and two, edges on both sides."""
    M, K, N, v, E, bits, G = row
    spec = ProblemSpec("wave_k", GEOM_B, M, K, N, v, E, G, bits, codebook_3d=(G > 1), codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=93, device=DEV)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(6)).half().to(DEV)
    want = _np(x).astype(np.float64) @ vo.dequant_b(_np(codes), _np(cb)).astype(np.float64).T + _np(bias).astype(np.float64)
    ran = 0
    for tile in (28, 34, 54, 64):
        _say("wave_k", row, "tile", tile)
        try:
            y = _with_wave_tile(tile, lambda: cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_WAVE_K, bias=bias))
        except cabi.VqGemmError:
            continue   # no room for this tile's units beside the tables
        torch.cuda.synchronize()
        assert vo.rel_err(_np(y), want)[0] <= TOL, (row, tile)
        ran += 1
        if N % 32 == 0:
            y = _with_wave_tile(tile, lambda: cabi.e2e_gemm_b_gated(x, codes, cb, variant=cabi.VARIANT_WAVE_K, bias=bias))
            p = want.reshape(M, N // 32, 2, 16)
            gated = (p[:, :, 0] / (1 + np.exp(-p[:, :, 0])) * p[:, :, 1]).reshape(M, N // 2)
            torch.cuda.synchronize()
            assert vo.rel_err(_np(y), gated)[1] <= TOL, (row, tile, "gated")
    assert ran == (2 if v == 4 and bits == 16 else 4)   # (32 bytes of codes a row and unit: 80 and 96 x 64 only)


@pytest.mark.parametrize("row", WAVE_K_B + [(16, 128, 17, 8, 256, 8, 1), (15, 1152, 48, 4, 256, 8, 1), (9, 4224, 50, 8, 37, 8, 1), (32, 2048, 15, 8, 512, 16, 1)],
                         ids=lambda r: "x".join(map(str, r)))
def test_k_dealt_out_to_waves_an_odd_number_of_pieces_wide(row):
    """16 and 32 x 16 and x 48: sixteen waves and the table of copies where one codebook serves, eight waves elsewhere, more waves than units.
    A gated product needs pairs of pieces and refuses them."""
    M, K, N, v, E, bits, G = row
    spec = ProblemSpec("wave_k", GEOM_B, M, K, N, v, E, G, bits, codebook_3d=(G > 1), codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=95, device=DEV)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(8)).half().to(DEV)
    want = _np(x).astype(np.float64) @ vo.dequant_b(_np(codes), _np(cb)).astype(np.float64).T
    for tile in (11, 13, 21, 23):
        _say("wave_k", row, "tile", tile)
        for b in (None, bias):
            y = _with_wave_tile(tile, lambda: cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_WAVE_K, bias=b))
            torch.cuda.synchronize()
            assert vo.rel_err(_np(y), want if b is None else want + _np(b).astype(np.float64))[0] <= TOL, (row, tile)
        if N % 32 == 0:
            with pytest.raises(cabi.VqGemmError):
                _with_wave_tile(tile, lambda: cabi.e2e_gemm_b_gated(x, codes, cb, variant=cabi.VARIANT_WAVE_K, bias=bias))


@pytest.mark.parametrize("vec", [4, 8])
@pytest.mark.parametrize("M,K,N,E", [(1, 128, 6, 256), (16, 192, 258, 1 << 7), (33, 1088, 130, 254), (40, 4160, 34, 8), (32, 2048, 642, 256)])
def test_copies_of_the_codebook_change_no_bit(vec, M, K, N, E):
    """One codebook: a table of copies, where the tile has one.  The same codebook twice, each for half of the columns, such that
    tiles meet both: the plain table.  The same operands meet in the same order.  Infinite and NaN entries too."""
    spec = ProblemSpec("wave_k", GEOM_B, M, K, N, vec, E, 1, 8, codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=94, device=DEV)
    for special in (False, True):
        if special:
            cb[E - 1, 0], cb[E // 2, vec - 1], cb[0, 1] = float("inf"), float("nan"), float("-inf")
        twice = torch.stack([cb, cb]).contiguous()
        for tile in (12, 14, 18, 22, 24, 28):
            _say("copies", vec, M, K, N, E, special, "tile", tile)
            assert (N // 2) % (tile % 10 * 16) != 0
            one = _with_wave_tile(tile, lambda: cabi.e2e_gemm_b(x, codes, cb, variant=cabi.VARIANT_WAVE_K))
            two = _with_wave_tile(tile, lambda: cabi.e2e_gemm_b(x, codes, twice, variant=cabi.VARIANT_WAVE_K))
            torch.cuda.synchronize()
            assert torch.equal(one.view(torch.int16), two.view(torch.int16)), tile


@pytest.mark.parametrize("vec", [4, 8])
@pytest.mark.parametrize("M,K,N,E", [(1, 128, 6, 512), (16, 192, 258, 300), (33, 1088, 130, 512), (40, 4160, 34, 8), (5, 2048, 642, 512)])
def test_copies_of_a_codebook_with_16_bit_codes_change_no_bit(vec, M, K, N, E):
    """As above, up to 512 entries in rows of half the banks; 513 entries and more have no such table."""
    spec = ProblemSpec("wave_k", GEOM_B, M, K, N, vec, E, 1, 16, codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=95, device=DEV)
    cb[E - 1, 0], cb[E // 2, vec - 1] = float("inf"), float("nan")
    twice = torch.stack([cb, cb]).contiguous()
    more = torch.cat([cb, torch.ones(520 - E if E < 512 else 8, vec, dtype=torch.float16, device=DEV)]).contiguous()
    for tile in (12, 13, 14, 18, 23, 24, 28):
        if vec == 4 and tile == 28:
            continue
        _say("copies", vec, M, K, N, E, "tile", tile)
        one, two, plain = (_with_wave_tile(tile, lambda: cabi.e2e_gemm_b(x, codes, book, variant=cabi.VARIANT_WAVE_K)) for book in (cb, twice, more))
        torch.cuda.synchronize()
        assert torch.equal(one.view(torch.int16), two.view(torch.int16)) and torch.equal(one.view(torch.int16), plain.view(torch.int16)), tile


@pytest.mark.parametrize("M,K,N", [(1, 64, 8), (17, 96, 40), (33, 320, 65), (65, 1056, 2047), (130, 2048, 129), (16, 512, 64)])
@pytest.mark.parametrize("shift", [0, 1])   # elements by which w is off a 16-byte boundary
def test_k_dealt_out_to_waves_plain_gemm(M, K, N, shift):
    g = torch.Generator().manual_seed(5)
    x = torch.randn(M, K, generator=g).half().to(DEV)
    w = torch.randn(K * N + shift, generator=g).half().to(DEV)[shift:].view(K, N)
    want = _np(x).astype(np.float64) @ _np(w).astype(np.float64)
    for tile in (12, 22, 24, 42, 44):
        _say("wave_k gemm", M, K, N, "shift", shift, "tile", tile)
        y = _with_wave_tile(tile, lambda: cabi.gemm_f16(x, w))
        torch.cuda.synchronize()
        assert vo.rel_err(_np(y), want)[0] <= TOL, tile


@pytest.mark.parametrize("M,K,Nc", [(1, 64, 16), (17, 320, 48), (65, 1088, 112), (129, 512, 64)])
def test_k_dealt_out_to_waves_geometry_a(M, K, Nc):
    spec = ProblemSpec("A", GEOM_A, M, K, 2 * Nc, 2, 256, Nc // 4, 8, codebook_std=0.05)
    x, w, cb = make_problem(spec, seed=92, device=DEV)
    for tile in (12, 22, 24, 42, 44, 84, 86):
        _say("wave_k geometry A", M, K, Nc, "tile", tile)
        y = _with_wave_tile(tile, lambda: cabi.e2e_gemm_a(x, w, cb, variant=cabi.VARIANT_PREFILL))
        torch.cuda.synchronize()
        _check_gemm(y, x, w, cb, geometry=GEOM_A, what=f"tile {tile}")


@pytest.mark.parametrize("M,K,Nc", [(1, 64, 16), (130, 192, 48), (97, 320, 80), (65, 1088, 112), (129, 2112, 64), (257, 576, 96)])
def test_k_dealt_out_to_waves_geometry_a_table_of_copies(M, K, Nc):
    """The tiles of vq_wave_k_a.hip: waves with no step, one and an odd number of them, edges on both sides."""
    spec = ProblemSpec("A", GEOM_A, M, K, 2 * Nc, 2, 256, Nc // 4, 8, codebook_std=0.05)
    x, w, cb = make_problem(spec, seed=96, device=DEV)
    for tile in (144, 164, 166, 184, 186):
        _say("wave_k geometry A", M, K, Nc, "tile", tile)
        y = _with_wave_tile(tile, lambda: cabi.e2e_gemm_a(x, w, cb, variant=cabi.VARIANT_PREFILL))
        torch.cuda.synchronize()
        _check_gemm(y, x, w, cb, geometry=GEOM_A, what=f"tile {tile}")


@pytest.mark.parametrize("what", ["weights", "entries", "entry 0 is NaN", "both", "equal vectors and entries", "all zero"])
@pytest.mark.parametrize("N,K,v,E,G", [(64, 256, 8, 256, 2), (48, 520, 8, 100, 1), (40, 128, 4, 4096, 1), (50, 64, 2, 77, 1), (24, 64, 8, 5000, 1), (24, 64, 8, 3430, 1)])
def test_encoder_keeps_the_rule_where_nothing_is_finite_or_everything_is_equal(N, K, v, E, G, what):
    """A NaN distance never wins and entry 0 is taken as it is; among equals the lowest index is kept."""
    g = torch.Generator(device="cpu").manual_seed(17)
    cb, w = torch.randn(G, E, v, generator=g).half(), torch.randn(N, K, generator=g).half()
    odd = torch.tensor([float("inf"), float("-inf"), float("nan"), 65504.0, -65504.0, 0.0, -0.0]).half()
    some = lambda t, share: torch.where(torch.rand(t.shape, generator=g) < share, odd[torch.randint(0, 7, t.shape, generator=g)], t)
    if what in ("weights", "both"):
        w = some(w, 0.03)
    if what in ("entries", "both"):
        cb = some(cb, 0.01)
    if what == "entry 0 is NaN":
        cb[:, 0, v - 1] = float("nan")
    if what == "equal vectors and entries":
        cb[:, E // 2:] = cb[:, :E - E // 2].clone()
        w.view(N, K // v, v)[:, ::2] = cb[0, E // 3]
    if what == "all zero":
        cb[:], w[:] = 0.0, 0.0
    bits = 8 if E <= 256 else 16
    _say("encode", N, K, v, E, what)
    codes = cabi.encode_b(w.to(DEV), cb.to(DEV), bits)
    torch.cuda.synchronize()
    assert np.array_equal(_np(codes), c_oracle.encode_b(w.numpy(), cb.numpy(), bits))


@pytest.mark.parametrize("N,K,v", [(1024, 1032, 8), (1032, 1024, 8), (700, 768, 4)])   # the last and first sizes of a wave's 64 and 128 vectors
def test_encoder_on_both_sides_of_the_line_between_its_wave_sizes(N, K, v):
    g = torch.Generator(device="cpu").manual_seed(6)
    cb, w = torch.randn(1, 256, v, generator=g).half(), torch.randn(N, K, generator=g).half()
    _say("encode", N, K, v)
    codes = cabi.encode_b(w.to(DEV), cb.to(DEV))
    torch.cuda.synchronize()
    assert np.array_equal(_np(codes), c_oracle.encode_b(w.numpy(), cb.numpy(), 8))


@pytest.mark.parametrize("scale", [2e-7, 2e-5, 0.02, 40.0, 2e4, 65504.0])   # subnormal halves to norms that take more than one part
@pytest.mark.parametrize("N,K,v,E", [(96, 128, 4, 33), (96, 256, 4, 767), (64, 256, 4, 768), (40, 128, 4, 4096), (64, 256, 8, 513)])
def test_encoder_at_the_ends_of_the_range_of_halves(N, K, v, E, scale):
    """The half norms of 4-vectors as sums of halves: groups of eight and of sixteen, tiles left empty, entries of very different sizes."""
    g = torch.Generator(device="cpu").manual_seed(23)
    cb, w = torch.randn(1, E, v, generator=g), torch.randn(N, K, generator=g)
    cb[:, ::7] *= 2.0 ** -12
    w.view(N, K // v, v)[:, ::5] *= 2.0 ** -13
    cb, w = ((t * scale).clamp(-65504, 65504).half() for t in (cb, w))
    w.view(N, K // v, v)[:, ::3] = cb[0, torch.randint(0, E, (N, (K // v + 2) // 3), generator=g)]
    bits = 8 if E <= 256 else 16
    _say("encode", N, K, v, E, scale)
    codes = cabi.encode_b(w.to(DEV), cb.to(DEV), bits)
    torch.cuda.synchronize()
    assert np.array_equal(_np(codes), c_oracle.encode_b(w.numpy(), cb.numpy(), bits))


@pytest.mark.parametrize("N,K", [(4096, 1024), (4096, 1032)])
def test_encoder_in_workgroups_of_sixteen_waves(N, K):
    """Codebooks that leave no room for a second workgroup on the unit, every unit at work: rows picked from all over against the oracle."""
    v, E = 8, 5000
    g = torch.Generator(device="cpu").manual_seed(25)
    cb, w = torch.randn(1, E, v, generator=g).half(), torch.randn(N, K, generator=g).half()
    _say("encode", N, K, v, E)
    codes = cabi.encode_b(w.to(DEV), cb.to(DEV), 16)
    torch.cuda.synchronize()
    rows = list(range(0, N, 97)) + [N - 1]
    assert np.array_equal(_np(codes)[rows], c_oracle.encode_b(w[rows].contiguous().numpy(), cb.numpy(), 16))


@pytest.mark.parametrize("N,K,v,E,scale", [(1032, 1032, 8, 100, 2e-6), (1032, 1032, 8, 100, 0.02), (1032, 1032, 8, 100, 2e4),
                                           (4096, 1032, 8, 128, 0.02), (4104, 1024, 8, 900, 0.02), (2056, 1024, 4, 129, 2e-5), (4096, 1032, 8, 127, 0.02)])
def test_lloyd_assignments_make_the_codebook_of_the_encoders_codes(N, K, v, E, scale):
    """The first assignment of one iteration, whose kernel is another than the encoder's: half norms as parts of K, workgroups of sixteen
    waves (from 2**19 vectors and 128 entries on)."""
    from vq_gemm_amd.torch_ops import native
    g = torch.Generator(device="cpu").manual_seed(24)
    w = (torch.randn(N, K, generator=g) * scale).clamp(-65504, 65504).half().to(DEV)
    pick = torch.randperm(N * K // v, generator=g)[:E].to(torch.int32).view(1, E)
    _say("lloyd", N, K, v, E, scale)
    bits = 8 if E <= 256 else 16
    _, cb, errors = native.kmeans(w, pick, v, E, 1, bits, 1)
    vectors = w.view(-1, v)
    first = vectors[pick.view(-1).long().to(DEV)].contiguous()
    codes = cabi.encode_b(w, first, bits).view(-1)
    codes = (codes if bits == 8 else codes.view(torch.int16)).long()
    d = vectors.double() - first.double()[codes]
    assert abs(float(errors[0]) - float((d * d).sum())) <= 1e-4 * float((d * d).sum())   # fp32 sums of a wave's, 131 K of them
    sums = torch.zeros(E, v, dtype=torch.float64, device=DEV).index_add_(0, codes, vectors.double())
    mean = sums / torch.bincount(codes, minlength=E)[:, None].clamp(min=1)
    # a vector assigned to another entry moves a mean of a thousand vectors by a thousandth of them; the sums are fp32, the entries halves
    step = torch.maximum(mean.abs() * 2.0 ** -11, torch.full_like(mean, 2.0 ** -25))
    assert bool(((cb[0].double() - mean).abs() <= 1.01 * step + 1e-5 * scale).all())


@pytest.mark.parametrize("M,K,N", [(257, 192, 263), (130, 448, 129), (40, 256, 300)])
def test_rows_of_y_that_begin_anywhere(M, K, N):
    spec = ProblemSpec("odd_rows", GEOM_B, M, K, N, 8, 256, 1, 8, codebook_std=0.05)
    x, codes, cb = make_problem(spec, seed=93, device=DEV)
    want = _np(x).astype(np.float64) @ vo.dequant_b(_np(codes), _np(cb)).astype(np.float64).T
    for variant in (cabi.VARIANT_PREFILL, cabi.VARIANT_PREFILL_NARROW, cabi.VARIANT_PREFILL_SMALL):
        _say("rows of", N, "columns", cabi.VARIANT_NAMES[variant])
        guard = torch.full((M * N + 8,), 7.0, dtype=torch.float16, device=DEV)
        cabi.e2e_gemm_b(x, codes, cb, variant=variant, out=guard[:M * N].view(M, N))
        torch.cuda.synchronize()
        assert vo.rel_err(_np(guard[:M * N].view(M, N)), want)[0] <= TOL, variant
        assert bool((guard[M * N:] == 7.0).all())


@pytest.mark.parametrize("M,K,N", [(3914, 1024, 4616), (1800, 1024, 10240)])   # 16 x 19 and 8 x 40 large tiles: whole rounds and a few more
def test_plain_gemm_with_the_left_over_columns_in_a_second_launch(M, K, N):
    g = torch.Generator().manual_seed(7)
    x, w = torch.randn(M, K, generator=g).half().to(DEV), torch.randn(K, N, generator=g).half().to(DEV)
    _say("gemm", M, K, N)
    guard = torch.full((M * N + 8,), 7.0, dtype=torch.float16, device=DEV)
    y = cabi.gemm_f16(x, w, out=guard[:M * N].view(M, N))
    want = x.float() @ w.float()
    torch.cuda.synchronize()
    assert ((y.float() - want).norm() / want.norm()).item() <= TOL and bool((guard[M * N:] == 7.0).all())
    assert ((y.float() - want).abs().max() / want.abs().max()).item() <= TOL
