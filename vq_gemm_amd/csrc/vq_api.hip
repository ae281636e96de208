// C ABI of libvqgemm.so: argument validation and kernel selection.  No torch types here;
// the torch extension and the tests both call these entry points.
#include "../../include/vq_gemm.h"
#include "vq_common.h"

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <limits.h>
#include <map>
#include <mutex>
#include <string>
#include <utility>

namespace vq {

namespace {

// the current device while a DeviceScope is alive on this thread, and how many are
thread_local int t_device = -1, t_scopes = 0;

int current_device()
{
    if (t_scopes > 0) return t_device;
    int dev = -1;
    return hipGetDevice(&dev) == hipSuccess ? dev : -1;
}

struct ResolvedKernel {
    const void *kernel = nullptr;
    int device = -1;
    hipFunction_t function = nullptr;
    size_t granted = 48 * 1024;  // dynamic LDS a launch may ask for; this much needs no leave
};

}  // namespace

DeviceScope::DeviceScope()
{
    if (t_scopes == 0) t_device = current_device();
    t_scopes++;
}

DeviceScope::~DeviceScope() { t_scopes--; }

int device_cu_count()
{
    constexpr int kMaxDev = 64;
    static std::atomic<int> cache[kMaxDev];
    const int dev = current_device();
    if (dev < 0 || dev >= kMaxDev) return 256;
    int v = cache[dev].load(std::memory_order_relaxed);
    if (v > 0) return v;
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
    cache[dev].store(cus, std::memory_order_relaxed);
    return cus;
}

hipError_t resolve_kernel(const void *kernel, size_t lds_bytes, hipFunction_t *function)
{
    // a small table per thread in front of the shared one: a serving thread launches few kernels, again and again
    constexpr int kSlots = 64;
    thread_local ResolvedKernel recent[kSlots];
    static std::mutex mu;
    static std::map<std::pair<int, const void *>, ResolvedKernel> known;
    const int dev = current_device();
    if (dev < 0) return hipErrorInvalidDevice;
    ResolvedKernel &slot = recent[((reinterpret_cast<uintptr_t>(kernel) >> 4) * 0x9e3779b97f4a7c15ull) >> 58];
    if (slot.kernel != kernel || slot.device != dev || lds_bytes > slot.granted) {
        std::lock_guard<std::mutex> lock(mu);
        ResolvedKernel &k = known[{dev, kernel}];
        if (!k.function) {
            const hipError_t e = hipGetFuncBySymbol(&k.function, kernel);
            if (e != hipSuccess) {
                k.function = nullptr;
                return e;
            }
            k.kernel = kernel;
            k.device = dev;
        }
        if (lds_bytes > k.granted) {
            const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
            if (e != hipSuccess) return e;
            k.granted = lds_bytes;
        }
        slot = k;
    }
    *function = slot.function;
    return hipSuccess;
}

namespace {

struct TuningEntry {
    const char *name;
    double Tuning::*field;
};
const TuningEntry kTuningEntries[] = {
    {"prefill_tile_fixed_us", &Tuning::prefill_tile_fixed_us},
    {"prefill_stage_us_256x256", &Tuning::prefill_stage_us_256x256},
    {"prefill_stage_us_256x128", &Tuning::prefill_stage_us_256x128},
    {"prefill_full_device_factor", &Tuning::prefill_full_device_factor},
    {"prefill_small_tile_fixed_us", &Tuning::prefill_small_tile_fixed_us},
    {"prefill_small_stage_us_idle", &Tuning::prefill_small_stage_us_idle},
    {"prefill_small_stage_us_busy", &Tuning::prefill_small_stage_us_busy},
    {"decode_prologue_us", &Tuning::decode_prologue_us},
    {"decode_prologue_shared_cu_us", &Tuning::decode_prologue_shared_cu_us},
    {"decode_tile_us", &Tuning::decode_tile_us},
    {"decode_tile_chunked_us", &Tuning::decode_tile_chunked_us},
    {"decode_pass_change_us", &Tuning::decode_pass_change_us},
    {"gemv_max_tiles_per_cu", &Tuning::gemv_max_tiles_per_cu},
    {"gemv_max_k", &Tuning::gemv_max_k},
    {"gemv_wide_min_rows_per_wave", &Tuning::gemv_wide_min_rows_per_wave},
    {"gemv_wide_max_m", &Tuning::gemv_wide_max_m},
    {"gemv_wide_two_rows_max_runs", &Tuning::gemv_wide_two_rows_max_runs},
    {"gemv_wide_two_rows_max_runs_long_k", &Tuning::gemv_wide_two_rows_max_runs_long_k},
    {"gemv_wide_plain_table_max_runs", &Tuning::gemv_wide_plain_table_max_runs},
    {"gemv_wide_single_rows_max", &Tuning::gemv_wide_single_rows_max},
    {"gemv_wide_rows_per_group", &Tuning::gemv_wide_rows_per_group},
    {"gemv_wide_groups_in_flight", &Tuning::gemv_wide_groups_in_flight},
    {"gemv_wide_rows_per_group_long_k", &Tuning::gemv_wide_rows_per_group_long_k},
    {"gemv_wide_groups_in_flight_long_k", &Tuning::gemv_wide_groups_in_flight_long_k},
    {"gemv_wide_rotate_priority", &Tuning::gemv_wide_rotate_priority},
    {"gemv_wide_min_units_share", &Tuning::gemv_wide_min_units_share},
    {"decode_replicated_table_min_tiles", &Tuning::decode_replicated_table_min_tiles},
    {"decode_stream_min_k", &Tuning::decode_stream_min_k},
    {"decode_stream_min_k_few_rows", &Tuning::decode_stream_min_k_few_rows},
    {"decode_stream_min_m", &Tuning::decode_stream_min_m},
    {"decode_stream_max_m", &Tuning::decode_stream_max_m},
    {"decode_stream_max_groups_per_unit", &Tuning::decode_stream_max_groups_per_unit},
    {"decode_stream_replicated_min_gathers", &Tuning::decode_stream_replicated_min_gathers},
    {"tail_split_margin", &Tuning::tail_split_margin},
    {"splitk_fixed_us", &Tuning::splitk_fixed_us},
    {"splitk_us_per_partial_mb", &Tuning::splitk_us_per_partial_mb},
    {"splitk_force_splits", &Tuning::splitk_force_splits},
    {"wave_k_force", &Tuning::wave_k_force},
    {"wave_k_force_tile", &Tuning::wave_k_force_tile},
    {"prefill_mid_force", &Tuning::prefill_mid_force},
};
constexpr int kTuningCount = (int)(sizeof(kTuningEntries) / sizeof(kTuningEntries[0]));

std::mutex g_tuning_mu;
Tuning g_tuning;             // written under the mutex; read without it (plain doubles, set before the launches that use them)
std::atomic<uint32_t> g_tuning_version{0};   // of the table: a plan made under another one is made again
std::atomic<bool> g_tuning_file_read{false};  // (acquire/release: a reader that sees true also sees what the file set)

const TuningEntry *find_tuning(const char *name)
{
    if (!name) return nullptr;
    for (const TuningEntry &e : kTuningEntries)
        if (std::strcmp(e.name, name) == 0) return &e;
    return nullptr;
}

// A flat JSON object of numbers, {"name": value, ...}: names this library does not know are skipped, and so
// is everything that is no number (a "device" string, for instance).  Returns how many constants were set.
int read_tuning_file(const char *path)
{
    FILE *f = std::fopen(path, "rb");
    if (!f) return -1;
    std::string text;
    char buf[4096];
    size_t n;
    while ((n = std::fread(buf, 1, sizeof(buf), f)) > 0) text.append(buf, n);
    std::fclose(f);
    int set = 0;
    size_t pos = 0;
    while ((pos = text.find('"', pos)) != std::string::npos) {
        const size_t end = text.find('"', pos + 1);
        if (end == std::string::npos) break;
        const std::string key = text.substr(pos + 1, end - pos - 1);
        size_t q = end + 1;
        while (q < text.size() && (text[q] == ' ' || text[q] == '\t' || text[q] == '\n' || text[q] == '\r')) q++;
        pos = end + 1;
        if (q >= text.size() || text[q] != ':') continue;   // a string value, not a key
        q++;
        while (q < text.size() && (text[q] == ' ' || text[q] == '\t' || text[q] == '\n' || text[q] == '\r')) q++;
        char *stop = nullptr;
        const double v = std::strtod(text.c_str() + q, &stop);
        if (stop == text.c_str() + q) { pos = q; continue; }  // no number behind the key
        pos = (size_t)(stop - text.c_str());
        const TuningEntry *e = find_tuning(key.c_str());
        if (e && v == v && v >= 0.0 && v < 1e9) {
            g_tuning.*(e->field) = v;
            g_tuning_version.fetch_add(1, std::memory_order_release);
            set++;
        }
    }
    return set;
}

bool aligned(const void *p, uintptr_t a) { return ((uintptr_t)p & (a - 1)) == 0; }

// Of the two fused geometry-A kernels (both take the same shapes), whether the wave-K kernel is expected to be the faster one.
bool wave_k_a_preferred(const ProblemA &p)
{
    const int force = (int)tuning().wave_k_force;
    return wave_k_a_supports(p) && force != 2 && (force == 1 || wave_k_a_cost_us(p) < fused_a_cost_us(p));
}

// Whether the automatic choice takes a fused geometry-A kernel: at every height (a short X
// leaves its 128-row tile mostly padding, and the kernel is still an order of magnitude ahead of the
// scalar one).  Its 4-byte gathers keep the LDS busier than the matrix cores, so once there is more
// than one round of tiles the two-pass route is faster - when the caller brings the scratch for it.
bool fused_a_preferred(const ProblemA &p, bool has_workspace)
{
    if (p.M < 1 || !fused_a_supports(p)) return false;
    if (!has_workspace) return true;
    const int64_t tiles = (int64_t)((p.M + 255) / 256) * ((2 * p.Nc + 127) / 128);
    if (tiles <= device_cu_count()) return true;
    // ... unless the wave-K kernel, which multiplies more than it gathers, is expected to be ahead of it: M = 3262, K = 7488, Nc = 1376
    // 198.7 -> 155.7 us.  (The first pass: 2 us and 1 us a million codes; 5 % off with the second, over 18 such shapes, and the choice
    // 0.3 % from the better one.)
    return wave_k_a_preferred(p) &&
           ((int)tuning().wave_k_force == 1 || wave_k_a_cost_us(p) < 2.0 + 1.0e-6 * p.K * p.Nc + gemm_tiled_cost_us(p.M, p.K, 2 * p.Nc));
}

int check_b(int64_t M, int64_t K, int64_t N, int32_t vec, int32_t entries, int32_t n_codebooks, int32_t code_bits)
{
    if (M < 0 || K < 0 || N < 0 || M > INT_MAX / 2 || K > INT_MAX / 2 || N > INT_MAX / 2) return VQGEMM_E_SHAPE;
    if (vec < 1 || vec > 4096 || entries < 1 || n_codebooks < 1) return VQGEMM_E_SHAPE;
    if (code_bits != 8 && code_bits != 16) return VQGEMM_E_CODEBITS;
    if ((int64_t)entries > ((int64_t)1 << code_bits)) return VQGEMM_E_CODEBITS;
    if (K % vec != 0) return VQGEMM_E_SHAPE;
    if (N % n_codebooks != 0) return VQGEMM_E_SHAPE;
    return VQGEMM_OK;
}

ProblemB make_b(const void *x, const void *codes, const void *codebook, void *y, int64_t M, int64_t K, int64_t N,
                int32_t vec, int32_t entries, int32_t n_codebooks, int32_t code_bits)
{
    ProblemB p;
    p.x = static_cast<const half_t *>(x);
    p.codes = codes;
    p.cb = static_cast<const half_t *>(codebook);
    p.y = static_cast<half_t *>(y);
    p.bias = nullptr;
    p.M = (int)M; p.K = (int)K; p.N = (int)N;
    p.k_x = (int)K;
    p.vec = vec; p.entries = entries; p.n_codebooks = n_codebooks; p.code_bits = code_bits;
    p.rows_per_cb = N > 0 ? (int)(N / n_codebooks) : 1;
    if (p.rows_per_cb < 1) p.rows_per_cb = 1;
    p.packed = false;
    p.gated = false;
    return p;
}

int select_b(const ProblemB &p, bool all_aligned16)
{
    if (p.K == 0 || !all_aligned16) return VQGEMM_VARIANT_GENERIC;
    if (decode_gemv_wide_preferred(p)) return VQGEMM_VARIANT_DECODE_GEMV;  // (also shapes the K-sliced kernels refuse)
    const bool prefill_ok = prefill_supports(p);
    if (decode_supports(p) && (!prefill_ok || decode_preferred(p)))
        return decode_gemv_preferred(p) ? VQGEMM_VARIANT_DECODE_GEMV : VQGEMM_VARIANT_DECODE;
    if (prefill_ok) return VQGEMM_VARIANT_PREFILL;
    return VQGEMM_VARIANT_GENERIC;
}

// select_b's kernel for an aligned operand set, or - above 64 rows of X, where the K-sliced path's model promises more than
// it keeps (65 rows, K = 1024, N = 11904, 4-vectors: 24 us, the prefill kernels 13) - the prefill kernels in that path's place
// wherever the wave-K kernel stands by for what they are slow at.
int plain_b(const ProblemB &p)
{
    const int v = select_b(p, true);
    return v == VQGEMM_VARIANT_DECODE && p.M > 64 && prefill_supports(p) && wave_k_b_supports(p) ? VQGEMM_VARIANT_PREFILL : v;
}

// Split K with the cost model's number of slices when that is expected to beat what the automatic choice would
// launch otherwise by a margin (and then at least two slices); 0: do not split.
int splitk_auto(const ProblemB &p, double *t_best, int *plain_variant)
{
    *t_best = 1e30;
    const int plain = plain_b(p);
    *plain_variant = plain;
    double t_plain;
    if (plain == VQGEMM_VARIANT_PREFILL) t_plain = prefill_cost_us(p);
    else if (plain == VQGEMM_VARIANT_DECODE) t_plain = decode_cost_us(p);
    else return 0;
    if (t_plain >= 1e29) return 0;  // (short X: the decode path is taken without a comparison, and stays)
    double t_split = 1e30;
    const int sp = prefill_splitk_choice(p, &t_split, 2);
    // (at even odds with the tiles that have a unit to themselves, whose model is as close as split K's: of 20 shapes above 200 rows
    // where the two were measured within 10 % of each other 9 were faster split, and they differ by 5 % on average)
    const bool take = sp >= 2 && t_split < (plain == VQGEMM_VARIANT_PREFILL && prefill_mid_plan(p).cost_us <= t_plain ? 1.005 : 0.95) * t_plain;
    *t_best = take ? t_split : t_plain;
    return take ? sp : 0;
}

// What the automatic choice does with a workspace: nothing, K split over every 128x128 tile (sp slices), or whole rounds
// of large tiles with the left-over columns in 128x128 tiles and K split there (tail) - whichever the cost models
// expect to be fastest by a margin.
struct WorkspaceChoice {
    bool wave;      // the wave-K kernel, which needs none
    int sp;
    TailSplitPlan tail;
    size_t bytes;
};
// Above 64 rows of X the wave-K kernel is taken below this share of what the other plan is expected to take, the models being 3 to 7 %
// off.  Over 150 shapes of M 65 to 2000 the choice takes 0.91 of the time that it took before the tiles with a compute unit to
// themselves, the wave-K kernel's last tile shapes and its faster reads of X (512 x 4096 x 4096: 27 us, split K 32).
constexpr double kWaveMargin = 0.95;

WorkspaceChoice workspace_auto(const ProblemB &p)
{
    WorkspaceChoice c = {false, 0, {false, 0, 0, 0, 1e30, 0}, 0};
    double t_best = 1e30;
    int plain = VQGEMM_VARIANT_GENERIC;
    c.sp = splitk_auto(p, &t_best, &plain);
    if (c.sp >= 2) c.bytes = prefill_splitk_workspace_bytes(p, c.sp);
    if (plain == VQGEMM_VARIANT_PREFILL && t_best < 1e29) {
        const TailSplitPlan tail = prefill_tail_split_plan(p);
        // (a margin of 1000 and more: wherever the plan exists - for measurements and tests)
        const double margin = tuning().tail_split_margin;
        if (tail.ok && (margin >= 1e3 || tail.cost_us < margin * t_best)) {
            c.sp = 0;
            c.tail = tail;
            c.bytes = tail.workspace_bytes;
        }
    }
    // (a split asked for by the tuning table is not weighed against anything)
    const bool asked = tuning().splitk_force_splits >= 2.0 || tuning().tail_split_margin >= 1e3;
    const double t_other = c.tail.ok ? c.tail.cost_us : c.sp >= 2 ? t_best : prefill_cost_us(p);
    if (!(asked && c.bytes > 0) && (plain == VQGEMM_VARIANT_DECODE || plain == VQGEMM_VARIANT_PREFILL) && wave_k_b_preferred(p, t_other, kWaveMargin))
        c = {true, 0, {false, 0, 0, 0, 1e30, 0}, 0};
    return c;
}

// What the automatic choice launches: without a workspace, and with one.  wave_tile: the wave-K kernel's tile where it is taken.
struct AutoPlan {
    int variant;
    WorkspaceChoice ws;
    int wave_tile;
};

// (The gated product takes what the plain one would run on: every tiled kernel carries the gated epilogue itself;
// the GEMV kernels and the K-sliced decode kernels want whole groups of 32 interleaved rows per codebook resp. per matrix,
// and where one of them refuses, the next in line takes the shape.)
AutoPlan make_plan(const ProblemB &p)
{
    AutoPlan plan = {VQGEMM_VARIANT_GENERIC, {false, 0, {false, 0, 0, 0, 1e30, 0}, 0}, 0};
    if (p.K == 0) return plan;
    ProblemB plain = p;
    plain.gated = false;
    const int v = p.gated && decode_gemv_wide_preferred(p) ? VQGEMM_VARIANT_DECODE_GEMV : plain_b(plain);
    const bool tiled = v == VQGEMM_VARIANT_DECODE || v == VQGEMM_VARIANT_PREFILL;
    const bool wave = tiled && wave_k_b_preferred(p, p.M > 64 ? prefill_cost_us(plain) : 0.0, kWaveMargin);
    if (wave) plan.variant = VQGEMM_VARIANT_WAVE_K;
    else if (!p.gated) plan.variant = v;
    else if (v == VQGEMM_VARIANT_DECODE_GEMV && decode_gemv_supports(p)) plan.variant = v;
    else if ((v == VQGEMM_VARIANT_DECODE || v == VQGEMM_VARIANT_DECODE_GEMV) && decode_gated_supports(p)) plan.variant = VQGEMM_VARIANT_DECODE;
    else if (prefill_supports(plain)) plan.variant = VQGEMM_VARIANT_PREFILL;
    if (!p.gated && tiled) plan.ws = p.M > 64 ? workspace_auto(p) : WorkspaceChoice{wave, 0, {false, 0, 0, 0, 1e30, 0}, 0};
    if (wave || plan.ws.wave) plan.wave_tile = wave_k_b_tile(p);
    return plan;
}

// The plan of a shape, kept per thread for the shapes it has met last: a serving thread multiplies by the same few weights
// again and again, and the cost models are a microsecond of arithmetic.
const AutoPlan &auto_plan(const ProblemB &p)
{
    struct Entry {
        uint64_t key[4];
        AutoPlan plan;
    };
    constexpr int kEntries = 64;
    thread_local Entry entries[kEntries];
    (void)tuning();   // (a file is read before its version is)
    const uint64_t key[4] = {(uint64_t)(uint32_t)p.M << 32 | (uint32_t)p.K, (uint64_t)(uint32_t)p.N << 32 | (uint32_t)p.entries,
                             (uint64_t)(uint32_t)p.n_codebooks << 32 | (uint32_t)(p.vec << 8 | p.code_bits << 1 | (p.gated ? 1 : 0)),
                             ((uint64_t)g_tuning_version.load(std::memory_order_acquire) << 32 | (uint32_t)current_device()) + 1};
    uint64_t h = key[0] * 0x9e3779b97f4a7c15ull ^ key[1] * 0xc2b2ae3d27d4eb4full ^ key[2] * 0x165667b19e3779f9ull;
    Entry &e = entries[(h ^ h >> 32) >> 8 & (kEntries - 1)];
    if (e.key[3] != key[3] || e.key[0] != key[0] || e.key[1] != key[1] || e.key[2] != key[2]) {
        e.plan = make_plan(p);
        for (int i = 0; i < 4; i++) e.key[i] = key[i];
    }
    return e.plan;
}

}  // namespace

const Tuning &tuning()
{
    // the file named by VQGEMM_TUNING_FILE is read once, at the first question
    if (!g_tuning_file_read.load(std::memory_order_acquire)) {
        std::lock_guard<std::mutex> lock(g_tuning_mu);
        if (!g_tuning_file_read.load(std::memory_order_relaxed)) {
            const char *path = std::getenv("VQGEMM_TUNING_FILE");
            if (path && path[0]) read_tuning_file(path);
            g_tuning_file_read.store(true, std::memory_order_release);
        }
    }
    return g_tuning;
}

}  // namespace vq

using namespace vq;

extern "C" {

int vqgemm_version(void) { return 200; }

int vqgemm_tuning_count(void) { return kTuningCount; }

const char *vqgemm_tuning_name(int index) { return index >= 0 && index < kTuningCount ? kTuningEntries[index].name : nullptr; }

int vqgemm_tuning_get(const char *name, double *value)
{
    const TuningEntry *e = find_tuning(name);
    if (!e) return VQGEMM_E_VARIANT;
    if (!value) return VQGEMM_E_NULL;
    *value = tuning().*(e->field);
    return VQGEMM_OK;
}

int vqgemm_tuning_set(const char *name, double value)
{
    const TuningEntry *e = find_tuning(name);
    if (!e) return VQGEMM_E_VARIANT;
    if (!(value >= 0.0) || value >= 1e9) return VQGEMM_E_SHAPE;
    (void)tuning();  // (a file is read before, not after, an explicit setting)
    std::lock_guard<std::mutex> lock(g_tuning_mu);
    g_tuning.*(e->field) = value;
    g_tuning_version.fetch_add(1, std::memory_order_release);
    return VQGEMM_OK;
}

int vqgemm_tuning_load(const char *path)
{
    if (!path) return VQGEMM_E_NULL;
    (void)tuning();
    std::lock_guard<std::mutex> lock(g_tuning_mu);
    const int n = read_tuning_file(path);
    return n < 0 ? VQGEMM_E_NULL : n;
}

const char *vqgemm_error_string(int code)
{
    switch (code) {
    case VQGEMM_OK: return "success";
    case VQGEMM_E_NULL: return "a required pointer is NULL";
    case VQGEMM_E_SHAPE: return "invalid shape (negative or too large size, K % vec != 0, N % n_codebooks != 0, ...)";
    case VQGEMM_E_CODEBITS: return "code_bits must be 8 or 16 and entries <= 2^code_bits";
    case VQGEMM_E_VARIANT: return "unknown kernel variant, or the variant cannot serve this shape";
    case VQGEMM_E_ALIGN: return "pointer not aligned as the selected kernel requires";
    case VQGEMM_E_SCRATCH: return "the problem needs more scratch than the library's fixed device array, or the workspace passed with its size, holds";
    default: break;
    }
    if (code > 0) return hipGetErrorString(static_cast<hipError_t>(code));
    return "unknown vqgemm error";
}

int vqgemm_select_variant_b(int64_t M, int64_t K, int64_t N, int32_t vec, int32_t entries, int32_t n_codebooks,
                            int32_t code_bits)
{
    const DeviceScope device;
    const int rc = check_b(M, K, N, vec, entries, n_codebooks, code_bits);
    if (rc != VQGEMM_OK) return rc;
    const ProblemB p = make_b(nullptr, nullptr, nullptr, nullptr, M, K, N, vec, entries, n_codebooks, code_bits);
    return select_b(p, true);
}

int vqgemm_e2e_gemm_b_bias(const void *x, const void *codes, const void *codebook, const void *bias, void *y,
                           int64_t M, int64_t K, int64_t N, int32_t vec, int32_t entries, int32_t n_codebooks,
                           int32_t code_bits, int32_t variant, void *workspace, void *stream)
{
    const DeviceScope device;
    int rc = check_b(M, K, N, vec, entries, n_codebooks, code_bits);
    if (rc != VQGEMM_OK) return rc;
    if (variant < VQGEMM_VARIANT_AUTO || variant > VQGEMM_VARIANT_WAVE_K || variant == VQGEMM_VARIANT_PREFILL_SPLITK) return VQGEMM_E_VARIANT;
    if (M == 0 || N == 0) return VQGEMM_OK;
    if (!y || !codebook || (K > 0 && (!x || !codes))) return VQGEMM_E_NULL;
    const uintptr_t code_align = code_bits / 8;
    if (!aligned(x, 2) || !aligned(y, 2) || !aligned(codebook, 2) || !aligned(codes, code_align)) return VQGEMM_E_ALIGN;
    if (!aligned(bias, 2)) return VQGEMM_E_ALIGN;
    // the tiled kernels read four bias values at a time
    const bool a16 = aligned(x, 16) && aligned(y, 16) && aligned(codebook, 16) && aligned(codes, 16) && aligned(bias, 8);
    ProblemB p = make_b(x, codes, codebook, y, M, K, N, vec, entries, n_codebooks, code_bits);
    p.bias = static_cast<const half_t *>(bias);
    hipStream_t s = static_cast<hipStream_t>(stream);
    int wave_tile = 0;
    if (variant == VQGEMM_VARIANT_AUTO) {
        const AutoPlan none = {VQGEMM_VARIANT_GENERIC, {}, 0};
        const AutoPlan &plan = a16 ? auto_plan(p) : none;
        variant = plan.variant;
        wave_tile = plan.wave_tile;
    }
    hipError_t e = hipSuccess;
    switch (variant) {
    case VQGEMM_VARIANT_GENERIC:
        e = launch_generic_b(p, s);
        break;
    case VQGEMM_VARIANT_DECODE:
        if (!a16) return VQGEMM_E_ALIGN;
        if (K == 0 || !decode_supports(p)) return VQGEMM_E_VARIANT;
        e = launch_decode_b(p, s);
        break;
    case VQGEMM_VARIANT_DECODE_GEMV:
        if (!a16) return VQGEMM_E_ALIGN;
        if (K == 0 || !decode_gemv_supports(p)) return VQGEMM_E_VARIANT;
        e = launch_decode_gemv(p, s);
        break;
    case VQGEMM_VARIANT_DECODE_PACKED:
        if (!a16) return VQGEMM_E_ALIGN;
        p.packed = true;
        if (K == 0 || !decode_packed_supports(p)) return VQGEMM_E_VARIANT;
        e = launch_decode_b(p, s);
        break;
    case VQGEMM_VARIANT_PREFILL:
        if (!a16) return VQGEMM_E_ALIGN;
        if (K == 0 || !prefill_supports(p)) return VQGEMM_E_VARIANT;
        e = launch_prefill_b(p, s);
        break;
    case VQGEMM_VARIANT_PREFILL_NARROW:
        if (!a16) return VQGEMM_E_ALIGN;
        if (K == 0 || !prefill_narrow_supports(p)) return VQGEMM_E_VARIANT;
        e = launch_prefill_b(p, s, 2);
        break;
    case VQGEMM_VARIANT_PREFILL_SMALL:
        if (!a16) return VQGEMM_E_ALIGN;
        if (K == 0 || !prefill_small_supports(p)) return VQGEMM_E_VARIANT;
        e = launch_prefill_small_b(p, s);
        break;
    case VQGEMM_VARIANT_WAVE_K:
        if (!a16) return VQGEMM_E_ALIGN;
        if (!wave_k_b_supports(p)) return VQGEMM_E_VARIANT;
        e = launch_wave_k_b(p, s, wave_tile);
        break;
    case VQGEMM_VARIANT_TWOPASS:
        if (bias) return VQGEMM_E_VARIANT;  // the plain GEMM of the two-pass route has no bias input
        if (!workspace) return VQGEMM_E_NULL;
        if (!aligned(workspace, 16)) return VQGEMM_E_ALIGN;
        e = launch_dequant_b(p, static_cast<half_t *>(workspace), s);
        if (e == hipSuccess)
            e = launch_gemm_nt(p.x, static_cast<const half_t *>(workspace), p.y, p.M, p.K, p.N, s);
        break;
    default:
        return VQGEMM_E_VARIANT;
    }
    return static_cast<int>(e);
}

int64_t vqgemm_workspace_bytes_b(int64_t M, int64_t K, int64_t N, int32_t vec, int32_t entries, int32_t n_codebooks,
                                 int32_t code_bits, int32_t variant)
{
    const DeviceScope device;
    const int rc = check_b(M, K, N, vec, entries, n_codebooks, code_bits);
    if (rc != VQGEMM_OK) return rc;
    if (M == 0 || N == 0 || K == 0) return 0;
    const ProblemB p = make_b(nullptr, nullptr, nullptr, nullptr, M, K, N, vec, entries, n_codebooks, code_bits);
    if (variant == VQGEMM_VARIANT_TWOPASS) return N * K * 2;
    if (variant == VQGEMM_VARIANT_AUTO) return (int64_t)auto_plan(p).ws.bytes;
    int sp = 0;
    if (variant == VQGEMM_VARIANT_PREFILL_SPLITK) sp = prefill_splitk_choice(p, nullptr, 2);
    return sp >= 2 ? (int64_t)prefill_splitk_workspace_bytes(p, sp) : 0;
}

int vqgemm_auto_variant_b(int64_t M, int64_t K, int64_t N, int32_t vec, int32_t entries, int32_t n_codebooks, int32_t code_bits,
                          int64_t workspace_bytes)
{
    const DeviceScope device;
    const int rc = check_b(M, K, N, vec, entries, n_codebooks, code_bits);
    if (rc != VQGEMM_OK) return rc;
    const ProblemB p = make_b(nullptr, nullptr, nullptr, nullptr, M, K, N, vec, entries, n_codebooks, code_bits);
    if (M == 0 || N == 0 || K == 0) return VQGEMM_VARIANT_GENERIC;
    const AutoPlan &plan = auto_plan(p);
    if (workspace_bytes <= 0) return plan.variant;
    if (plan.ws.wave) return VQGEMM_VARIANT_WAVE_K;
    if ((int64_t)plan.ws.bytes > workspace_bytes) return plan.variant;
    return plan.ws.tail.ok ? VQGEMM_PLAN_TAIL_SPLIT : plan.ws.sp >= 2 ? VQGEMM_VARIANT_PREFILL_SPLITK : plan.variant;
}

int vqgemm_e2e_gemm_b_ws(const void *x, const void *codes, const void *codebook, const void *bias, void *y, int64_t M,
                         int64_t K, int64_t N, int32_t vec, int32_t entries, int32_t n_codebooks, int32_t code_bits,
                         int32_t variant, void *workspace, int64_t workspace_bytes, void *stream)
{
    const DeviceScope device;
    if (workspace_bytes < 0 || (workspace_bytes > 0 && !workspace)) return VQGEMM_E_NULL;
    if (variant == VQGEMM_VARIANT_TWOPASS) {
        if (workspace_bytes < N * K * 2) return VQGEMM_E_SCRATCH;
        return vqgemm_e2e_gemm_b_bias(x, codes, codebook, bias, y, M, K, N, vec, entries, n_codebooks, code_bits, variant, workspace, stream);
    }
    if (variant != VQGEMM_VARIANT_AUTO && variant != VQGEMM_VARIANT_PREFILL_SPLITK)
        return vqgemm_e2e_gemm_b_bias(x, codes, codebook, bias, y, M, K, N, vec, entries, n_codebooks, code_bits, variant, nullptr, stream);
    int rc = check_b(M, K, N, vec, entries, n_codebooks, code_bits);
    if (rc != VQGEMM_OK) return rc;
    if (M == 0 || N == 0) return VQGEMM_OK;
    if (!y || !codebook || (K > 0 && (!x || !codes))) return VQGEMM_E_NULL;
    const bool a16 = aligned(x, 16) && aligned(y, 16) && aligned(codebook, 16) && aligned(codes, 16) && aligned(bias, 8) &&
                     aligned(workspace, 256);
    ProblemB p = make_b(x, codes, codebook, y, M, K, N, vec, entries, n_codebooks, code_bits);
    p.bias = static_cast<const half_t *>(bias);
    int sp;
    if (variant == VQGEMM_VARIANT_PREFILL_SPLITK) {
        if (!a16) return VQGEMM_E_ALIGN;
        sp = K > 0 ? prefill_splitk_choice(p, nullptr, 2) : 0;
        if (sp < 2) return VQGEMM_E_VARIANT;
        if ((int64_t)prefill_splitk_workspace_bytes(p, sp) > workspace_bytes) return VQGEMM_E_SCRATCH;
    } else {
        const AutoPlan none = {VQGEMM_VARIANT_GENERIC, {}, 0};
        const AutoPlan &plan = a16 && K > 0 ? auto_plan(p) : none;
        const WorkspaceChoice &c = plan.ws;
        if (c.wave) return static_cast<int>(launch_wave_k_b(p, static_cast<hipStream_t>(stream), plan.wave_tile));
        if (c.tail.ok && (int64_t)c.bytes <= workspace_bytes)
            return static_cast<int>(launch_prefill_tail_split(p, c.tail, static_cast<hipStream_t>(stream), workspace));
        // (a workspace that is too small is not an error for the automatic choice: it does without)
        sp = c.sp;
        if (sp < 2 || (int64_t)c.bytes > workspace_bytes)
            return vqgemm_e2e_gemm_b_bias(x, codes, codebook, bias, y, M, K, N, vec, entries, n_codebooks, code_bits, VQGEMM_VARIANT_AUTO,
                                          nullptr, stream);
    }
    return static_cast<int>(launch_prefill_small_b(p, static_cast<hipStream_t>(stream), sp, workspace));
}

namespace {

// Additive stages: the kernel that the automatic choice for the whole K takes on aligned operands, where that kernel reads an X
// that repeats along K as it is (VQGEMM_VARIANT_AUTO: it does not, X is repeated in memory).  A matter of the sizes only: the
// question for a workspace is asked before there are operands.
int stages_variant(ProblemB p, int stages)
{
    p.x = nullptr;
    ProblemB q = p;
    q.k_x = p.K / stages;
    const WorkspaceChoice &c = auto_plan(p).ws;
    if (c.wave) return wave_k_b_supports(q) ? VQGEMM_VARIANT_WAVE_K : VQGEMM_VARIANT_AUTO;
    return c.bytes == 0 && plain_b(p) == VQGEMM_VARIANT_DECODE && decode_stages_supports(q) ? VQGEMM_VARIANT_DECODE : VQGEMM_VARIANT_AUTO;
}
int64_t repeated_x_bytes(const ProblemB &p) { return ((int64_t)p.M * p.K * 2 + 255) & ~(int64_t)255; }

}  // namespace

int64_t vqgemm_stages_workspace_bytes_b(int64_t M, int64_t K, int64_t N, int32_t vec, int32_t entries, int32_t n_codebooks,
                                        int32_t code_bits, int32_t stages)
{
    const DeviceScope device;
    const int rc = check_b(M, K, N, vec, entries, n_codebooks, code_bits);
    if (rc != VQGEMM_OK) return rc;
    if (stages < 1 || K % stages != 0) return VQGEMM_E_SHAPE;
    if (M == 0 || N == 0 || K == 0) return 0;
    const ProblemB p = make_b(nullptr, nullptr, nullptr, nullptr, M, K, N, vec, entries, n_codebooks, code_bits);
    if (stages > 1 && stages_variant(p, stages) != VQGEMM_VARIANT_AUTO) return 0;
    return (stages > 1 ? repeated_x_bytes(p) : 0) + (int64_t)auto_plan(p).ws.bytes;
}

int vqgemm_e2e_gemm_b_stages(const void *x, const void *codes, const void *codebook, const void *bias, void *y, int64_t M, int64_t K,
                             int64_t N, int32_t vec, int32_t entries, int32_t n_codebooks, int32_t code_bits, int32_t stages,
                             void *workspace, int64_t workspace_bytes, void *stream)
{
    const DeviceScope device;
    int rc = check_b(M, K, N, vec, entries, n_codebooks, code_bits);
    if (rc != VQGEMM_OK) return rc;
    if (stages < 1 || K % stages != 0) return VQGEMM_E_SHAPE;
    if (workspace_bytes < 0 || (workspace_bytes > 0 && !workspace)) return VQGEMM_E_NULL;
    if (stages == 1 || M == 0 || N == 0 || K == 0)
        return vqgemm_e2e_gemm_b_ws(x, codes, codebook, bias, y, M, K, N, vec, entries, n_codebooks, code_bits, VQGEMM_VARIANT_AUTO,
                                    workspace, workspace_bytes, stream);
    if (!y || !codebook || !x || !codes) return VQGEMM_E_NULL;
    if (!aligned(x, 2) || !aligned(y, 2) || !aligned(codebook, 2) || !aligned(codes, code_bits / 8) || !aligned(bias, 2) ||
        !aligned(workspace, 256))
        return VQGEMM_E_ALIGN;
    ProblemB p = make_b(x, codes, codebook, y, M, K, N, vec, entries, n_codebooks, code_bits);
    p.bias = static_cast<const half_t *>(bias);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool a16 = aligned(x, 16) && aligned(y, 16) && aligned(codebook, 16) && aligned(codes, 16) && aligned(bias, 8);
    const int64_t repeated = repeated_x_bytes(p);
    const int variant = stages_variant(p, stages);
    // (operands that begin anywhere, and no room for a copy because for these sizes none is asked for: the scalar kernel, which
    // such operands go to in any case, reads X as it is too; whole vectors, since both kernels above want K / stages % 8 == 0)
    if (variant != VQGEMM_VARIANT_AUTO && (a16 || workspace_bytes < repeated)) {
        p.k_x = p.K / stages;
        if (!a16) return static_cast<int>(launch_generic_b(p, s));
        return static_cast<int>(variant == VQGEMM_VARIANT_WAVE_K ? launch_wave_k_b(p, s) : launch_decode_b(p, s));
    }
    if (workspace_bytes < repeated) return VQGEMM_E_SCRATCH;
    const hipError_t e = launch_repeat_columns(p.x, static_cast<half_t *>(workspace), M, K / stages, stages, s);
    if (e != hipSuccess) return static_cast<int>(e);
    const int64_t rest = workspace_bytes - repeated;
    return vqgemm_e2e_gemm_b_ws(workspace, codes, codebook, bias, y, M, K, N, vec, entries, n_codebooks, code_bits, VQGEMM_VARIANT_AUTO,
                                rest > 0 ? static_cast<uint8_t *>(workspace) + repeated : nullptr, rest, stream);
}

int vqgemm_e2e_gemm_b_gated(const void *x, const void *codes, const void *codebook, const void *bias, void *y, int64_t M,
                            int64_t K, int64_t N, int32_t vec, int32_t entries, int32_t n_codebooks, int32_t code_bits,
                            int32_t variant, void *workspace, void *stream)
{
    const DeviceScope device;
    int rc = check_b(M, K, N, vec, entries, n_codebooks, code_bits);
    if (rc != VQGEMM_OK) return rc;
    if (N % 32 != 0) return VQGEMM_E_SHAPE;  // whole pairs of 16 gate rows and 16 up rows
    if (M == 0 || N == 0) return VQGEMM_OK;
    if (!y || !codebook || (K > 0 && (!x || !codes))) return VQGEMM_E_NULL;
    const uintptr_t code_align = code_bits / 8;
    if (!aligned(x, 2) || !aligned(y, 2) || !aligned(codebook, 2) || !aligned(codes, code_align) || !aligned(bias, 2) ||
        !aligned(workspace, 2))
        return VQGEMM_E_ALIGN;
    const bool a16 = aligned(x, 16) && aligned(y, 16) && aligned(codebook, 16) && aligned(codes, 16) && aligned(bias, 8) &&
                     aligned(workspace, 16);
    ProblemB p = make_b(x, codes, codebook, y, M, K, N, vec, entries, n_codebooks, code_bits);
    p.bias = static_cast<const half_t *>(bias);
    p.gated = true;
    hipStream_t s = static_cast<hipStream_t>(stream);
    // the plain product of the same shape, for the kernels without a gated epilogue (into the workspace)
    ProblemB plain = p;
    plain.gated = false;
    plain.y = static_cast<half_t *>(workspace);
    int wave_tile = 0;
    if (variant == VQGEMM_VARIANT_AUTO) {
        variant = VQGEMM_VARIANT_GENERIC;
        if (a16 && K > 0) {
            const AutoPlan &plan = auto_plan(p);
            variant = plan.variant;
            wave_tile = plan.wave_tile;
        }
    }
    hipError_t e = hipSuccess;
    switch (variant) {
    case VQGEMM_VARIANT_GENERIC:
        e = launch_generic_b(p, s);
        break;
    case VQGEMM_VARIANT_DECODE_GEMV:
        if (!a16) return VQGEMM_E_ALIGN;
        if (K == 0 || !decode_gemv_supports(p)) return VQGEMM_E_VARIANT;
        e = launch_decode_gemv(p, s);
        break;
    case VQGEMM_VARIANT_DECODE:
        if (!a16) return VQGEMM_E_ALIGN;
        if (K == 0 || !decode_gated_supports(p)) return VQGEMM_E_VARIANT;
        e = launch_decode_b(p, s);
        break;
    case VQGEMM_VARIANT_PREFILL:
        if (!a16) return VQGEMM_E_ALIGN;
        if (K == 0 || !prefill_supports(plain)) return VQGEMM_E_VARIANT;
        e = launch_prefill_b(p, s);
        break;
    case VQGEMM_VARIANT_PREFILL_NARROW:
        if (!a16) return VQGEMM_E_ALIGN;
        if (K == 0 || !prefill_narrow_supports(plain)) return VQGEMM_E_VARIANT;
        e = launch_prefill_b(p, s, 2);
        break;
    case VQGEMM_VARIANT_PREFILL_SMALL:
        if (!a16) return VQGEMM_E_ALIGN;
        if (K == 0 || !prefill_small_supports(plain)) return VQGEMM_E_VARIANT;
        e = launch_prefill_small_b(p, s);
        break;
    case VQGEMM_VARIANT_WAVE_K:
        if (!a16) return VQGEMM_E_ALIGN;
        if (!wave_k_b_supports(p)) return VQGEMM_E_VARIANT;
        e = launch_wave_k_b(p, s, wave_tile);
        break;
    case VQGEMM_VARIANT_TWOPASS: {
        // (here: the fused product as the automatic choice runs it, then the element-wise pass)
        if (!workspace) return VQGEMM_E_NULL;
        rc = vqgemm_e2e_gemm_b_bias(x, codes, codebook, bias, workspace, M, K, N, vec, entries, n_codebooks, code_bits,
                                    VQGEMM_VARIANT_AUTO, nullptr, stream);
        if (rc != VQGEMM_OK) return rc;
        e = launch_silu_mul(static_cast<const half_t *>(workspace), p.y, M, N / 2, s, /*interleaved=*/true);
        break;
    }
    default:
        return VQGEMM_E_VARIANT;
    }
    return static_cast<int>(e);
}

int vqgemm_e2e_gemm_b(const void *x, const void *codes, const void *codebook, void *y, int64_t M, int64_t K,
                      int64_t N, int32_t vec, int32_t entries, int32_t n_codebooks, int32_t code_bits,
                      int32_t variant, void *workspace, void *stream)
{
    return vqgemm_e2e_gemm_b_bias(x, codes, codebook, nullptr, y, M, K, N, vec, entries, n_codebooks, code_bits, variant,
                                  workspace, stream);
}

int vqgemm_e2e_gemm_a(const void *x, const void *w, const void *codebook, void *out, int64_t M, int64_t K,
                      int64_t Nc, int32_t variant, void *workspace, void *stream)
{
    const DeviceScope device;
    if (M < 0 || K < 0 || Nc < 0 || M > INT_MAX / 2 || K > INT_MAX / 2 || Nc > INT_MAX / 4) return VQGEMM_E_SHAPE;
    if (Nc % 4 != 0) return VQGEMM_E_SHAPE;
    if (variant < VQGEMM_VARIANT_AUTO || variant > VQGEMM_VARIANT_TWOPASS) return VQGEMM_E_VARIANT;
    if (M == 0 || Nc == 0) return VQGEMM_OK;
    if (!out || !codebook || (K > 0 && (!x || !w))) return VQGEMM_E_NULL;
    if (!aligned(x, 2) || !aligned(out, 4) || !aligned(codebook, 4)) return VQGEMM_E_ALIGN;
    ProblemA p;
    p.x = static_cast<const half_t *>(x);
    p.w = static_cast<const uint8_t *>(w);
    p.cb = static_cast<const half_t *>(codebook);
    p.y = static_cast<half_t *>(out);
    p.M = (int)M; p.K = (int)K; p.Nc = (int)Nc;
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipError_t e = hipSuccess;
    // The fused tiled kernel where it applies and is expected to win; otherwise, with scratch, the
    // two-pass route (bit-exact dequant, then the MFMA GEMM), and without it the scalar kernel.
    if (variant == VQGEMM_VARIANT_AUTO) {
        if (fused_a_preferred(p, workspace != nullptr)) variant = VQGEMM_VARIANT_PREFILL;
        else variant = workspace ? VQGEMM_VARIANT_TWOPASS : VQGEMM_VARIANT_GENERIC;
    }
    switch (variant) {
    case VQGEMM_VARIANT_GENERIC:
        e = launch_generic_a(p, s);
        break;
    case VQGEMM_VARIANT_PREFILL:
        if (!fused_a_supports(p)) return aligned(x, 16) && aligned(w, 16) && aligned(codebook, 16) ? VQGEMM_E_VARIANT : VQGEMM_E_ALIGN;
        e = wave_k_a_preferred(p) ? launch_wave_k_a(p, s) : launch_fused_a(p, s);
        break;
    case VQGEMM_VARIANT_TWOPASS:
        if (!workspace) return VQGEMM_E_NULL;
        if (!aligned(workspace, 16)) return VQGEMM_E_ALIGN;
        e = launch_dequant_a(p, static_cast<half_t *>(workspace), s);
        if (e == hipSuccess)
            e = launch_gemm_nn(p.x, static_cast<const half_t *>(workspace), p.y, p.M, p.K, 2 * p.Nc, s);
        break;
    default:
        return VQGEMM_E_VARIANT;  // the decode tilings are geometry-B kernels
    }
    return static_cast<int>(e);
}

int vqgemm_select_variant_a(int64_t M, int64_t K, int64_t Nc, int32_t has_workspace)
{
    const DeviceScope device;
    if (M < 0 || K < 0 || Nc < 0 || M > INT_MAX / 2 || K > INT_MAX / 2 || Nc > INT_MAX / 4 || Nc % 4 != 0) return VQGEMM_E_SHAPE;
    ProblemA p = {};
    p.M = (int)M; p.K = (int)K; p.Nc = (int)Nc;
    if (fused_a_preferred(p, has_workspace != 0)) return VQGEMM_VARIANT_PREFILL;
    return has_workspace ? VQGEMM_VARIANT_TWOPASS : VQGEMM_VARIANT_GENERIC;
}

int vqgemm_dequant_b(const void *codes, const void *codebook, void *w_out, int64_t N, int64_t K, int32_t vec,
                     int32_t entries, int32_t n_codebooks, int32_t code_bits, void *stream)
{
    const DeviceScope device;
    const int rc = check_b(0, K, N, vec, entries, n_codebooks, code_bits);
    if (rc != VQGEMM_OK) return rc;
    if (N == 0 || K == 0) return VQGEMM_OK;
    if (!codes || !codebook || !w_out) return VQGEMM_E_NULL;
    if (!aligned(w_out, 2) || !aligned(codebook, 2) || !aligned(codes, code_bits / 8)) return VQGEMM_E_ALIGN;
    const ProblemB p = make_b(nullptr, codes, codebook, nullptr, 0, K, N, vec, entries, n_codebooks, code_bits);
    return static_cast<int>(launch_dequant_b(p, static_cast<half_t *>(w_out), static_cast<hipStream_t>(stream)));
}

int vqgemm_pack_codes_b(const void *codes, void *codes_out, int64_t N, int64_t K, int32_t vec, int32_t code_bits,
                        int32_t inverse, void *stream)
{
    const DeviceScope device;
    if (N < 0 || K < 0 || N > INT_MAX / 2 || K > INT_MAX / 2) return VQGEMM_E_SHAPE;
    if (code_bits != 8 && code_bits != 16) return VQGEMM_E_CODEBITS;
    if (vec < 1 || K % vec != 0) return VQGEMM_E_SHAPE;
    if (!pack_codes_supports(N, K, vec, code_bits)) return VQGEMM_E_VARIANT;
    if (N == 0 || K == 0) return VQGEMM_OK;
    if (!codes || !codes_out) return VQGEMM_E_NULL;
    if (codes == codes_out) return VQGEMM_E_NULL;  // not in place: a permutation of the whole matrix
    if (!aligned(codes, 16) || !aligned(codes_out, 16)) return VQGEMM_E_ALIGN;
    return static_cast<int>(launch_pack_codes(codes, codes_out, N, K, vec, code_bits, inverse != 0,
                                              static_cast<hipStream_t>(stream)));
}

int vqgemm_decode_packed_supports(int64_t M, int64_t K, int64_t N, int32_t vec, int32_t entries, int32_t n_codebooks,
                                  int32_t code_bits)
{
    const DeviceScope device;
    const int rc = check_b(M, K, N, vec, entries, n_codebooks, code_bits);
    if (rc != VQGEMM_OK) return rc;
    if (M == 0 || N == 0 || K == 0) return 0;
    ProblemB p = make_b(nullptr, nullptr, nullptr, nullptr, M, K, N, vec, entries, n_codebooks, code_bits);
    p.packed = true;
    return decode_packed_supports(p) ? 1 : 0;
}

int vqgemm_packed_preferred_b(int64_t M, int64_t K, int64_t N, int32_t vec, int32_t entries, int32_t n_codebooks,
                              int32_t code_bits)
{
    const DeviceScope device;
    const int rc = check_b(M, K, N, vec, entries, n_codebooks, code_bits);
    if (rc != VQGEMM_OK) return rc;
    if (M == 0 || N == 0 || K == 0) return 0;
    const ProblemB p = make_b(nullptr, nullptr, nullptr, nullptr, M, K, N, vec, entries, n_codebooks, code_bits);
    const AutoPlan &plan = auto_plan(p);
    return plan.variant == VQGEMM_VARIANT_DECODE && !plan.ws.wave && plan.ws.bytes == 0 && decode_packed_preferred(p) ? 1 : 0;
}

int vqgemm_encode_b(const void *w, const void *codebook, void *codes_out, int64_t N, int64_t K, int32_t vec,
                    int32_t entries, int32_t n_codebooks, int32_t code_bits, void *stream)
{
    const DeviceScope device;
    const int rc = check_b(0, K, N, vec, entries, n_codebooks, code_bits);
    if (rc != VQGEMM_OK) return rc;
    if (N == 0 || K == 0) return VQGEMM_OK;
    if (!w || !codebook || !codes_out) return VQGEMM_E_NULL;
    if (!aligned(w, 2) || !aligned(codebook, 2) || !aligned(codes_out, code_bits / 8)) return VQGEMM_E_ALIGN;
    const ProblemB p = make_b(nullptr, nullptr, codebook, nullptr, 0, K, N, vec, entries, n_codebooks, code_bits);
    if (!encode_supports(p)) return VQGEMM_E_VARIANT;
    return static_cast<int>(launch_encode_b(static_cast<const half_t *>(w), p, codes_out, static_cast<hipStream_t>(stream)));
}

int64_t vqgemm_kmeans_workspace_bytes_b(int64_t N, int64_t K, int32_t vec, int32_t entries, int32_t n_codebooks, int32_t code_bits)
{
    const DeviceScope device;
    const int rc = check_b(0, K, N, vec, entries, n_codebooks, code_bits);
    if (rc != VQGEMM_OK) return rc;
    if (N == 0 || K == 0) return VQGEMM_E_VARIANT;
    const ProblemB p = make_b(nullptr, nullptr, nullptr, nullptr, 0, K, N, vec, entries, n_codebooks, code_bits);
    if (!lloyd_supports(p) || (int64_t)p.rows_per_cb * (K / vec) > INT_MAX) return VQGEMM_E_VARIANT;
    return (int64_t)lloyd_workspace_bytes(p);
}

int vqgemm_kmeans_b(const void *w, const int32_t *pick, void *codes_out, void *codebook_out, double *errors_out, int64_t N, int64_t K,
                    int32_t vec, int32_t entries, int32_t n_codebooks, int32_t code_bits, int32_t iters, void *workspace,
                    int64_t workspace_bytes, void *stream)
{
    const DeviceScope device;
    const int64_t need = vqgemm_kmeans_workspace_bytes_b(N, K, vec, entries, n_codebooks, code_bits);
    if (need < 0) return (int)need;
    if (iters < 0) return VQGEMM_E_SHAPE;
    if (!w || !pick || !codes_out || !codebook_out || !errors_out || !workspace) return VQGEMM_E_NULL;
    if (!aligned(w, 8) || !aligned(pick, 4) || !aligned(codebook_out, 4) || !aligned(codes_out, code_bits / 8) || !aligned(errors_out, 8) ||
        !aligned(workspace, 256))
        return VQGEMM_E_ALIGN;
    if (workspace_bytes < need) return VQGEMM_E_SCRATCH;
    const ProblemB p = make_b(nullptr, nullptr, nullptr, nullptr, 0, K, N, vec, entries, n_codebooks, code_bits);
    return static_cast<int>(launch_lloyd(static_cast<const half_t *>(w), p, pick, iters, codes_out, static_cast<half_t *>(codebook_out),
                                         errors_out, workspace, static_cast<hipStream_t>(stream)));
}

int vqgemm_silu_mul(const void *gate_up, void *out, int64_t M, int64_t N, void *stream)
{
    const DeviceScope device;
    if (M < 0 || N < 0 || M > INT_MAX / 2 || N > INT_MAX / 4) return VQGEMM_E_SHAPE;
    if (M == 0 || N == 0) return VQGEMM_OK;
    if (!gate_up || !out) return VQGEMM_E_NULL;
    if (!aligned(gate_up, 2) || !aligned(out, 2)) return VQGEMM_E_ALIGN;
    return static_cast<int>(launch_silu_mul(static_cast<const half_t *>(gate_up), static_cast<half_t *>(out), M, N,
                                            static_cast<hipStream_t>(stream)));
}

int vqgemm_max_code(const void *codes, int64_t count, int32_t code_bits, void *max_out, void *stream)
{
    const DeviceScope device;
    if (count < 0) return VQGEMM_E_SHAPE;
    if (code_bits != 8 && code_bits != 16) return VQGEMM_E_CODEBITS;
    if (!max_out || (count > 0 && !codes)) return VQGEMM_E_NULL;
    if (!aligned(max_out, 4) || !aligned(codes, code_bits / 8)) return VQGEMM_E_ALIGN;
    return static_cast<int>(launch_max_code(codes, count, code_bits, static_cast<uint32_t *>(max_out),
                                            static_cast<hipStream_t>(stream)));
}

int vqgemm_dequant_a(const void *w, const void *codebook, void *w_out, int64_t K, int64_t Nc, void *stream)
{
    const DeviceScope device;
    if (K < 0 || Nc < 0 || K > INT_MAX / 2 || Nc > INT_MAX / 4 || Nc % 4 != 0) return VQGEMM_E_SHAPE;
    if (K == 0 || Nc == 0) return VQGEMM_OK;
    if (!w || !codebook || !w_out) return VQGEMM_E_NULL;
    if (!aligned(w_out, 4) || !aligned(codebook, 4)) return VQGEMM_E_ALIGN;
    ProblemA p;
    p.x = nullptr;
    p.w = static_cast<const uint8_t *>(w);
    p.cb = static_cast<const half_t *>(codebook);
    p.y = nullptr;
    p.M = 0; p.K = (int)K; p.Nc = (int)Nc;
    return static_cast<int>(launch_dequant_a(p, static_cast<half_t *>(w_out), static_cast<hipStream_t>(stream)));
}

int vqgemm_gemm_f16(const void *x, const void *w, void *y, int64_t M, int64_t K, int64_t N, void *stream)
{
    const DeviceScope device;
    if (M < 0 || K < 0 || N < 0 || M > INT_MAX / 2 || K > INT_MAX / 2 || N > INT_MAX / 2) return VQGEMM_E_SHAPE;
    if (M == 0 || N == 0) return VQGEMM_OK;
    if (!y || (K > 0 && (!x || !w))) return VQGEMM_E_NULL;
    if (!aligned(x, 2) || !aligned(w, 2) || !aligned(y, 2)) return VQGEMM_E_ALIGN;
    return static_cast<int>(launch_gemm_nn(static_cast<const half_t *>(x), static_cast<const half_t *>(w),
                                           static_cast<half_t *>(y), (int)M, (int)K, (int)N,
                                           static_cast<hipStream_t>(stream)));
}

}  // extern "C"
