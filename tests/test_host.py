"""CPU-side checks of the boundary: the C-ABI libraries load and export what the headers
declare, argument validation rejects bad calls before anything touches a GPU, the torch
modules exist under the names the reference harness imports, and the workload table matches
the published byte/flop figures of the five configurations."""
import ctypes
import os

import pytest
import torch

from vq_gemm_amd import cabi, ops
from vq_gemm_amd.problems import CONFIGS, make_problem


def test_libvqgemm_exports_every_declared_symbol():
    lib = cabi.lib()
    names = cabi.declared_symbols("vq_gemm.h")
    assert {"vqgemm_e2e_gemm_b", "vqgemm_e2e_gemm_a", "vqgemm_dequant_b", "vqgemm_dequant_a", "vqgemm_gemm_f16",
            "vqgemm_select_variant_b", "vqgemm_error_string", "vqgemm_version"} <= set(names)
    for n in names:
        assert hasattr(lib, n), n
    assert lib.vqgemm_version() >= 100


def test_libvqgemm_ref_exports_every_declared_symbol():
    lib = cabi.ref_lib()
    names = cabi.declared_symbols("vq_gemm_ref.h")
    assert "vqref_gemm_f16" in names
    for n in names:
        assert hasattr(lib, n), n


def test_argument_validation_happens_before_any_gpu_call():
    lib = cabi.lib()
    one = ctypes.c_void_p(16)  # never dereferenced: every call below is rejected first
    call = lambda **kw: lib.vqgemm_e2e_gemm_b(one, one, one, one, kw.get("M", 1), kw.get("K", 64), kw.get("N", 16),
                                              kw.get("vec", 8), kw.get("E", 256), kw.get("G", 1), kw.get("bits", 8),
                                              kw.get("variant", 0), None, None)
    assert call(M=-1) == -2
    assert call(K=60) == -2                    # K % vec != 0
    assert call(N=10, G=4) == -2               # N % n_codebooks != 0
    assert call(bits=12) == -3
    assert call(E=257) == -3                   # 257 entries do not fit 8-bit codes
    assert call(variant=9) == -4
    assert call(M=0) == 0 and call(N=0) == 0   # empty problems succeed without a launch
    assert lib.vqgemm_e2e_gemm_b(None, one, one, one, 1, 64, 16, 8, 256, 1, 8, 0, None, None) == -1
    assert lib.vqgemm_e2e_gemm_b(ctypes.c_void_p(17), one, one, one, 1, 64, 16, 8, 256, 1, 8, 0, None, None) == -5
    assert lib.vqgemm_e2e_gemm_a(one, one, one, one, 1, 64, 6, 0, None, None) == -2   # Nc % 4 != 0
    assert lib.vqgemm_dequant_b(one, one, one, 16, 60, 8, 256, 1, 8, None) == -2
    assert lib.vqgemm_dequant_a(one, one, one, 16, 6, None) == -2
    assert lib.vqgemm_gemm_f16(one, one, one, -1, 1, 1, None) == -2
    for code in (0, -1, -2, -3, -4, -5):
        assert len(lib.vqgemm_error_string(code)) > 0


def test_variant_selection_for_the_measured_configurations():
    want = {"C1": cabi.VARIANT_DECODE, "C2": cabi.VARIANT_DECODE_GEMV, "C3": cabi.VARIANT_DECODE,
            "C4": cabi.VARIANT_PREFILL, "C5": cabi.VARIANT_PREFILL}
    for name, v in want.items():
        s = CONFIGS[name]
        assert cabi.select_variant_b(s.M, s.K, s.N, s.vec, s.entries, s.n_codebooks, s.code_bits) == v, name
    # shapes the tiled kernels cannot take fall back to the generic kernel
    assert cabi.select_variant_b(4, 36, 8, 3, 10, 1, 8) == cabi.VARIANT_GENERIC
    assert cabi.select_variant_b(4, 0, 8, 8, 256, 1, 8) == cabi.VARIANT_GENERIC
    assert cabi.select_variant_b(4, 60, 8, 8, 256, 1, 8) < 0


def test_workload_table_matches_published_figures():
    want = {"C1": (329_728, 33_554_432), "C2": (2_117_632, 33_554_432), "C3": (23_060_480, 1_442_840_576),
            "C4": (69_337_088, 137_438_953_472), "C5": (180_584_448, 962_072_674_304)}
    for name, (nbytes, flops) in want.items():
        assert CONFIGS[name].algorithmic_bytes == nbytes, name
        assert CONFIGS[name].flops == flops, name
    assert CONFIGS["REF"].codes_shape == (4096, 640) and CONFIGS["REF"].codebook_shape == (160, 256, 2)


def test_problem_generator_is_deterministic_and_in_range():
    s = CONFIGS["C1"]
    a = make_problem(s, seed=42)
    b = make_problem(s, seed=42)
    for t, u in zip(a, b):
        assert torch.equal(t, u)
    x, codes, cb = a
    assert x.dtype == torch.float16 and x.shape == (16, 1024)
    assert codes.dtype == torch.uint8 and codes.shape == (1024, 256)
    assert cb.shape == (256, 4) and abs(cb.float().std().item() - 0.02) < 2e-3
    x3, c3, cb3 = make_problem(CONFIGS["C3"].__class__("t", "B", 2, 64, 32, 4, 4096, 1, 16), seed=1)
    assert c3.dtype == torch.uint16 and int(c3.to(torch.int32).max()) < 4096


@pytest.mark.parametrize("key", ops.VARIANT_KEYS)
def test_torch_modules_exist_under_the_reference_names(key):
    mod = ops.load_module(key)
    assert mod.__name__ == f"vq_gemm_cuda_{key}"
    assert callable(mod.e2e_gemm) and callable(mod.gemm)


def test_torch_module_rejects_bad_tensors_with_runtime_error():
    mod = ops.load_module("s2_128")
    x = torch.zeros(2, 8, dtype=torch.float16)
    with pytest.raises(RuntimeError, match="GPU tensor"):
        mod.e2e_gemm(x, torch.zeros(4, 1, dtype=torch.uint8), torch.zeros(256, 8, dtype=torch.float16))
    with pytest.raises(RuntimeError):
        mod.gemm(x, torch.zeros(8, 4, dtype=torch.float16))
    with pytest.raises(KeyError):
        ops.load_module("s9")


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    monkeypatch.setattr(cabi, "_LIB_DIR", str(tmp_path))
    monkeypatch.setattr(cabi, "_lib", None)
    with pytest.raises(ImportError, match="no CPU fallback"):
        cabi.lib()
    monkeypatch.setattr(ops, "_LIB_DIR", str(tmp_path))
    monkeypatch.setattr(ops, "_modules", {})
    with pytest.raises(ImportError, match="no CPU fallback"):
        ops.load_module("s2_128")


def test_registered_op_propagates_shapes_and_has_no_cpu_implementation():
    import torch
    from vq_gemm_amd import torch_ops  # noqa: F401
    x = torch.empty(3, 5, 64, dtype=torch.float16, device="meta")
    codes = torch.empty(32, 8, dtype=torch.uint8, device="meta")
    cb = torch.empty(2, 256, 8, dtype=torch.float16, device="meta")
    y = torch.ops.vq_gemm_amd.vq_linear(x, codes, cb)
    assert y.shape == (3, 5, 32) and y.dtype == torch.float16
    with pytest.raises(ValueError):   # 64 features against 8 codes x 4
        torch.ops.vq_gemm_amd.vq_linear(x, codes, torch.empty(256, 4, dtype=torch.float16, device="meta"))
    with pytest.raises(NotImplementedError):
        torch.ops.vq_gemm_amd.vq_linear(torch.zeros(2, 64, dtype=torch.float16), torch.zeros(32, 8, dtype=torch.uint8),
                                        torch.zeros(256, 8, dtype=torch.float16))


def test_ctypes_wrappers_refuse_host_tensors():
    import torch
    from vq_gemm_amd import cabi
    x = torch.zeros(2, 64, dtype=torch.float16)
    codes = torch.zeros(32, 8, dtype=torch.uint8)
    cb = torch.zeros(256, 8, dtype=torch.float16)
    with pytest.raises(ValueError):
        cabi.e2e_gemm_b(x, codes, cb)
    with pytest.raises(ValueError):
        cabi.dequant_b(codes, cb)


def test_tuning_constants_can_be_read_set_and_loaded_from_a_file(tmp_path):
    import json
    from vq_gemm_amd import cabi
    before = cabi.tuning()
    assert {"prefill_stage_us_256x256", "decode_tile_us", "gemv_max_tiles_per_cu", "gemv_wide_min_rows_per_wave"} <= set(before)
    try:
        # the choice between the four-wave GEMV kernel and the K-sliced kernel follows the constant
        dims = (1, 4096, 16 * 256 * 2, 4, 256, 1, 8)   # one row of X, 4-vectors: two tiles per unit on a 256-CU device
        cabi.set_tuning(gemv_max_tiles_per_cu=4)
        assert cabi.select_variant_b(*dims) == cabi.VARIANT_DECODE_GEMV
        cabi.set_tuning(gemv_max_tiles_per_cu=1)
        assert cabi.select_variant_b(*dims) == cabi.VARIANT_DECODE
        path = tmp_path / "t.json"
        path.write_text(json.dumps({"device": "some name: 3", "gemv_max_tiles_per_cu": 8, "decode_tile_us": 0.5, "not_a_constant": 1}))
        assert cabi.lib().vqgemm_tuning_load(str(path).encode()) == 2
        assert cabi.tuning()["decode_tile_us"] == 0.5 and cabi.select_variant_b(*dims) == cabi.VARIANT_DECODE_GEMV
        assert cabi.lib().vqgemm_tuning_load(b"/nonexistent/file.json") == -1
        assert cabi.lib().vqgemm_tuning_set(b"no_such_constant", 1.0) == -4
        assert cabi.lib().vqgemm_tuning_set(b"decode_tile_us", -1.0) == -2
    finally:
        cabi.set_tuning(**before)
    assert cabi.tuning() == before


def test_vqlinear_codes_key_works_on_inference_tensors():
    # a module whose codes were made under torch.inference_mode(): such tensors keep no version counter
    from vq_gemm_amd.nn import VQLinear
    with torch.inference_mode():
        codes = torch.zeros(32, 32, dtype=torch.uint8)
        cb = torch.zeros(256, 8, dtype=torch.float16)
        layer = VQLinear(codes, cb)
        k1 = layer._codes_key()
    assert layer.codes.is_inference()
    assert layer._codes_key() == k1
    # an ordinary tensor: the key follows in-place updates
    layer2 = VQLinear(torch.zeros(32, 32, dtype=torch.uint8), cb.clone())
    k2 = layer2._codes_key()
    layer2.codes.add_(1)
    assert layer2._codes_key() != k2


@pytest.mark.parametrize("n,count,books,seed", [(1, 1, 3, 0), (2, 2, 2, 5), (256, 256, 4, 1), (700, 256, 3, 4294967295), (5000, 1, 2, 7), (262144, 256, 3, 0)])
def test_start_of_a_seeded_permutation_is_torch_randperm_s(n, count, books, seed):
    from vq_gemm_amd.quantize import _initial_vectors
    from vq_gemm_amd.torch_ops import native
    gen = torch.Generator().manual_seed(seed)
    want = torch.stack([torch.randperm(n, generator=gen)[:count] for _ in range(books)]).to(torch.int32)
    assert torch.equal(native.first_of_permutations(n, count, books, seed), want)
    assert torch.equal(_initial_vectors(n, count, books, seed), want)


def test_launches_of_the_wave_k_kernel_hold_what_the_copy_of_their_codebooks_writes(tmp_path):
    """The codebooks go into the LDS in wave loads of 1 KB: a launch asks for the LDS up to the end of the last one, whatever the
    tables' size.  Checked by the compiler (host pass, nothing is linked) for every tile and format, on the kernel's own
    configuration: tables of every size from one 16-byte chunk to just over four wave loads."""
    import subprocess
    from vq_gemm_amd import build
    src = tmp_path / "lds.hip"
    src.write_text("""
#include "vq_wave_k_b.hip"
namespace vq {
template <class C> constexpr bool holds_every_table()
{
    for (size_t chunks = 1; chunks <= 260; chunks++)   // 16-byte chunks; 64 lanes of 16 bytes a load
        if (C::lds_bytes(chunks * 16) < C::kRing + (chunks + 63) / 64 * 64 * 16) return false;
    return true;
}
template <class F, int MP, int NP> constexpr bool holds()
{
    typedef WaveKCfg<typename F::template Wave<MP, NP>, MP, NP> C;
    bool ok = true;
    if constexpr (C::kExists) ok = holds_every_table<C>();
    if constexpr (F::template kHasCopies<MP, NP>) {   // (one size of table: a row of the 64 banks for each of 256 entries)
        typedef WaveKCfg<typename F::template Copies<MP, NP>, MP, NP> D;
        static_assert(D::kExists);
        ok = ok && D::lds_bytes(16) >= D::kRing + 256 * 256 && D::lds_bytes(4096) <= 160 * 1024;
    }
    return ok;
}
template <class F> constexpr bool every_tile()
{
    bool ok = holds<F, 1, 1>() && holds<F, 1, 2>() && holds<F, 1, 3>() && holds<F, 1, 4>() && holds<F, 1, 8>() && holds<F, 2, 1>() && holds<F, 2, 2>() && holds<F, 2, 3>();
    ok = ok && holds<F, 2, 4>() && holds<F, 2, 8>() && holds<F, 3, 4>() && holds<F, 4, 4>() && holds<F, 4, 8>() && holds<F, 5, 4>() && holds<F, 6, 4>();
    return ok;
}
static_assert(every_tile<Format<8, uint8_t>>() && every_tile<Format<8, uint16_t>>(), "8-vectors");
static_assert(every_tile<Format<4, uint8_t>>() && every_tile<Format<4, uint16_t>>(), "4-vectors");
}
""")
    res = subprocess.run([build.HIPCC, "-x", "hip", "--offload-host-only", f"--offload-arch={build.ARCH}", "-std=c++17", "-fsyntax-only",
                          "-fconstexpr-steps=10000000", f"-I{build.CSRC}", str(src)], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout + res.stderr


def test_nothing_touches_the_registers_of_a_load_that_the_compiler_does_not_count(tmp_path):
    """The codebook entries of the wave-K kernel's table of copies come by inline assembly into registers that the compiler takes for
    written at once: no branch, at whose ends it may copy them, and no use may lie ahead of the wait.  On the assembly of
    two of its kernels, as the build looks at it for all of them."""
    import subprocess
    from vq_gemm_amd import build
    src, asm = tmp_path / "copies.hip", tmp_path / "copies.s"
    src.write_text("""
#include "vq_wave_k.h"
namespace vq {
namespace {
template __global__ void wave_k_kernel<WaveB<8, uint8_t, 2, true>, 1, 2>(const WaveKArgs);
template __global__ void wave_k_kernel<WaveB<4, uint8_t, 2, true>, 1, 1>(const WaveKArgs);
}
}
""")
    flags = [f for f in build.HIP_FLAGS if f not in ("-Wall", "-Wno-unused-function")]
    res = subprocess.run([build.HIPCC] + flags + ["-x", "hip", "--offload-device-only", "-S", f"-I{build.CSRC}", str(src), "-o", str(asm)], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout + res.stderr
    assert build.check_loads_in_flight(asm.read_text()) == 4   # (with as many units as are loaded ahead, and with fewer)
    load, wait = ";;#ASMSTART\nglobal_load_dwordx4 v[2:5], v[0:1], off\n;;#ASMEND\n", "s_waitcnt vmcnt(3)\n"
    assert build.check_loads_in_flight(load + "v_add_u32_e32 v6, 1, v7\n" + wait + "v_mov_b32_e32 v6, v2\n") == 1
    for between in ("v_mov_b32_e32 v6, v2\n", "ds_write_b128 v8, v[4:7]\n", "s_cbranch_scc1 .L1\n", ".L1:\n"):
        with pytest.raises(RuntimeError, match="being loaded"):
            build.check_loads_in_flight(load + between + wait)


@pytest.mark.skipif(torch.cuda.is_available(), reason="made-up addresses: only where no kernel can be launched")
def test_stages_need_no_more_scratch_than_they_ask_for_wherever_the_operands_begin():
    lib = cabi.lib()
    ptr = ctypes.c_void_p
    base = 1 << 20
    checked = 0
    for M, K, N, vec, entries, bits in ((5, 8192, 4096, 8, 256, 8), (20, 8192, 64, 4, 1024, 16), (3, 8320, 33, 8, 256, 8), (16, 960, 50, 8, 300, 16)):
        for stages in (2, 3):
            if K % stages or lib.vqgemm_stages_workspace_bytes_b(M, K, N, vec, entries, 1, bits, stages) != 0:
                continue
            for shift in ((0, 0, 0, 0, 0), (2, 0, 0, 0, 0), (0, 2, 0, 0, 0), (0, 0, 2, 0, 0), (0, 0, 0, 2, 0), (0, 0, 0, 0, 2)):
                x, codes, cb, bias, y = (ptr(base + s) for s in shift)
                rc = lib.vqgemm_e2e_gemm_b_stages(x, codes, cb, bias, y, M, K, N, vec, entries, 1, bits, stages, None, 0, None)
                assert rc > 0, (M, K, N, stages, shift, rc)   # as far as the launch, which finds no device
                checked += 1
    assert checked >= 18


def test_the_packed_layout_is_taken_where_the_automatic_choice_takes_its_kernel():
    # the K-sliced kernel's shapes; the wave-K kernel's (which serves the packed layout too, slower); the streaming kernel's; tall X
    assert cabi.packed_preferred_b(4, 4096, 8192, 8, 256, 1, 8)
    for dims in ((64, 8192, 14336, 4, 4096, 1, 16), (64, 4096, 4096, 8, 256, 1, 8), (16, 14336, 4096, 8, 256, 1, 8), (512, 4096, 4096, 8, 256, 1, 8)):
        assert cabi.decode_packed_supports(*dims) and not cabi.packed_preferred_b(*dims), dims
    assert not cabi.packed_preferred_b(4, 320, 8192, 8, 256, 1, 8)   # no packed layout for this K
    assert not cabi.packed_preferred_b(0, 4096, 8192, 8, 256, 1, 8)
    assert cabi.lib().vqgemm_packed_preferred_b(4, 60, 8, 8, 256, 1, 8) < 0


def test_native_calls_let_other_threads_run():
    """A long call of the compiled extension (the starts of twelve permutations of 2^24) works without the GIL."""
    import threading
    import time
    from vq_gemm_amd.torch_ops import native
    ran, stop = [], threading.Event()

    def beat():
        while not stop.is_set():
            ran.append(time.perf_counter())
            time.sleep(0.001)

    other = threading.Thread(target=beat)
    other.start()
    try:
        while not ran:
            time.sleep(0.001)
        t0 = time.perf_counter()
        native.first_of_permutations(1 << 24, 16, 12, 7)
        t1 = time.perf_counter()
    finally:
        stop.set()
        other.join()
    # (with the GIL held the other thread can run right at the edges of the call, not between)
    assert any(t0 + 0.25 * (t1 - t0) < t < t0 + 0.75 * (t1 - t0) for t in ran), (t1 - t0, len(ran))


def test_split_k_is_asked_for_where_it_was_measured_faster():
    """The workspace the automatic choice asks for: none where the wave-K kernel was measured at 0.75 to 0.85 of split K's time (657 x
    13376 x 1040: 28.1 us, split 34.3), slices of K where it was the other way round (3028 x 11264 x 640: 51.5 us, the wave-K kernel
    61.3; 954 x 14080 x 1920 59.9, 70.1; 118 x 11008 x 14080 55.0, 65.1)."""
    for M, K, N, v, e, bits in ((657, 13376, 1040, 8, 256, 8), (203, 2816, 7040, 8, 256, 8), (489, 3072, 3328, 8, 256, 8), (72, 2304, 8832, 4, 4096, 16), (438, 2944, 3072, 4, 4096, 16)):
        assert cabi.workspace_bytes_b(M, K, N, v, e, 1, bits) == 0, (M, K, N)
    for M, K, N, v, e, bits in ((3028, 11264, 640, 8, 256, 8), (954, 14080, 1920, 8, 256, 8), (118, 11008, 14080, 4, 4096, 16)):
        assert cabi.workspace_bytes_b(M, K, N, v, e, 1, bits) > 0, (M, K, N)


def test_a_workspace_is_asked_for_only_where_it_is_used():
    """Over random shapes: a call with the workspace that is asked for launches a plan that needs one."""
    import random
    rng = random.Random(5)
    asked = 0
    for _ in range(600):
        v, e, bits = rng.choice(((8, 256, 8), (4, 256, 8), (4, 4096, 16), (8, 512, 16)))
        dims = (int(17 * 170 ** rng.random()), 64 * int(8 * 28 ** rng.random()), 16 * int(32 * 50 ** rng.random()), v, e, 1, bits)
        need = cabi.workspace_bytes_b(*dims)
        assert need == 0 or cabi.auto_variant_name_b(*dims, need) in ("prefill_splitk", "prefill_tail_split"), (dims, need)
        asked += need > 0
    assert asked >= 20
    assert cabi.workspace_bytes_b(512, 4096, 4096, 8, 256, 32, 8) == 0 and cabi.auto_variant_name_b(512, 4096, 4096, 8, 256, 32, 8) == "wave_k"


def test_no_width_is_an_exception_in_the_choice_between_decode_and_wave_k():
    """One tile of the decode kernel to each of 256 compute units, and a tile less and more: 16 x 4096 x 4096 is 5.65 us by the wave-K
    kernel and 6.50 by the decode kernel, as it is 5.66 and 6.49 on 4080 columns."""
    name = cabi.auto_variant_name_b
    for M, K, v, e, bits in ((16, 4096, 8, 256, 8), (16, 2048, 8, 256, 8), (8, 8192, 8, 256, 8), (16, 4096, 4, 256, 8), (5, 8192, 4, 256, 8), (8, 8192, 8, 512, 16)):
        assert {name(M, K, N, v, e, 1, bits) for N in (4080, 4096, 4112)} == {"wave_k"}, (M, K, v, bits)
    assert {name(3, 1024, N, 8, 256, 1, 8) for N in (4080, 4096)} == {"decode"}


def test_many_codes_go_where_they_stream_faster():
    """Codes out of HBM, us by the wave-K and by the decode kernel: 60.5 and 45.8, 45.0 and 35.1, 30.2 and 24.0, 39.7 and 35.0; where every
    unit has a tile the other way round, 12.8 and 16.9, 15.8 and 21.2, 19.7 and 28.8."""
    name = cabi.auto_variant_name_b
    for dims, want in (((5, 11648, 27328, 4, 4096, 1, 16), "decode"), ((4, 8448, 26048, 4, 4096, 1, 16), "decode"), ((12, 5120, 24832, 4, 4096, 1, 16), "decode"),
                       ((8, 12288, 27968, 8, 512, 1, 16), "decode"), ((8, 8192, 8192, 4, 4096, 1, 16), "wave_k"), ((3, 12288, 8192, 4, 4096, 64, 16), "wave_k"),
                       ((3, 13440, 14848, 8, 512, 1, 16), "wave_k")):
        assert name(*dims) == want, dims


def test_geometry_a_takes_the_one_kernel_that_was_weighed_against_two_passes():
    """Beyond one round of tiles the fused kernels take two passes' place for the wave-K kernel's sake only: not where the tuning table
    rules that kernel out, and everywhere when the table asks for it."""
    before = cabi.tuning()
    wins, loses = (3262, 7488, 1376), (4096, 4096, 2048)
    pick = lambda: [cabi.select_variant_a(*dims, has_workspace=True) for dims in (wins, loses)]
    try:
        assert pick() == [cabi.VARIANT_PREFILL, cabi.VARIANT_TWOPASS]
        cabi.set_tuning(wave_k_force=2)
        assert pick() == [cabi.VARIANT_TWOPASS, cabi.VARIANT_TWOPASS]
        cabi.set_tuning(wave_k_force=1)
        assert pick() == [cabi.VARIANT_PREFILL, cabi.VARIANT_PREFILL]
    finally:
        cabi.set_tuning(wave_k_force=before["wave_k_force"])


def test_the_report_of_the_automatic_choice_names_what_it_launches():
    """Host only; that the kernels named are the ones launched is held bit for bit on the GPU."""
    name = cabi.auto_variant_name_b
    assert name(1, 4096, 4096, 8, 256, 1, 8) == "decode_gemv" and name(3, 4096, 4096, 8, 256, 1, 8) == "decode"
    assert name(64, 8192, 14336, 4, 4096, 1, 16) == "wave_k" and cabi.select_variant_b(64, 8192, 14336, 4, 4096, 1, 16) == cabi.VARIANT_DECODE
    assert name(4096, 4096, 4096, 8, 256, 32, 8) == "prefill" and name(4, 60, 20, 4, 256, 1, 8) == "generic"
    for dims, plan in (((954, 14080, 1920, 8, 256, 1, 8), "prefill_splitk"), ((1536, 4096, 11008, 8, 256, 43, 8), "prefill_tail_split")):
        need = cabi.workspace_bytes_b(*dims)
        assert need > 0 and name(*dims, need) == plan and name(*dims, need - 1) == name(*dims) != plan
    with pytest.raises(cabi.VqGemmError):
        name(4, 60, 8, 8, 256, 1, 8)
