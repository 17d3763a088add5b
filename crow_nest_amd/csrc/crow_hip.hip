// libcrow_hip.so: gfx950 code objects (built ahead of time from the headers below) and the C ABI
// declared in include/crow_hip.h.  One translation unit, so the device globals are shared.
#include <hip/hip_runtime.h>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../../include/crow_hip.h"
#include "../../include/crow_hip_bench.h"
#include "kernels.h"
#include "misc_kernels.h"
#include "gemm.h"

namespace {

struct FnEntry {
    const char* name;
    const void* stub;
    int nargs;
    unsigned lds_fixed;  // dynamic LDS of a launch (kernels outside the GEMV family)
    // GEMV family (gemv.h): tensors per block (0 = not of the family), and the dynamic LDS of a block: the zero area + one
    // staging area per wave
    int nr;
    int max_waves;  // per block (the kernel's launch bound)
    int lds_per_wave;
    int ns;  // adjacent 16-row strips per block (kernels for several activation rows: CROW_MULTI_STRIPS), else 1
    bool takes_ws;  // the launcher appends the scratch descriptor (every kernel of the GEMV family)
    // a twin of `stub` for strips of two to eight groups that one wave walks alone, started in its place when the launch
    // dimensions say so; its dynamic LDS is the zero area and one staging area of twelve rows per GROUP (per block, not per wave)
    const void* tile_stub;
    bool takes_geo;  // the launcher appends the model geometry (crow_hip_set_geo) by value, last
    const void* one_stub = nullptr;  // a twin of `stub` with one strip per block, started in its place when S = CROW_ONE_STRIP
    const void* two_stub = nullptr;  // ... and one with two runs of columns per wave, when S = CROW_TWO_RUNS
    const void* twin_stub = nullptr;  // a twin started when the launch's gz = CROW_TWIN: unquantised GEMVs, weights alone requested ahead; acc_combo, y stored
    bool ksplit = false;  // GEMM for few token rows: one of g_ksplit starts in its place when the launch's gz says which (CROW_KSPLIT)
    const void* rows_stub = nullptr;  // gemv_b: a twin with 4 x 4 rows per wave, when the launch's gz = CROW_ROWS | activation rows
    const void* whole_stub = nullptr;  // a twin for blocks of two waves and strips of up to CROW_WHOLE_GROUPS groups, one slice
};
// values of S in a launch's `gy` word (GEMV family, K up to 16384; a strip of at most 64 groups never has that many slices): one
// slice, and one strip per block where the kernel otherwise takes `ns` of them / two runs of columns per wave of the block
#define CROW_ONE_STRIP 0x81u
#define CROW_TWO_RUNS 0x82u
#define CROW_TWIN 2u  // (the grid of those kernels has no third dimension)
#define CROW_ROWS 0x80000000u
#define CROW_STORE 0x83u  // moe_down_combine: y is stored, not added to
// A K-split GEMM in gz: this bit, bits 0..7 the column slices, 8..11 the strips per block, 12..15 the 16-token blocks per block, 16..23
// the waves per block
#define CROW_KSPLIT 0x80000000u

// The launcher builds a kernel's argument array from the fields of its table entry: the caller's `nargs` values, then the
// geometry word (GEMV family), the scratch descriptor (takes_ws), the model geometry (takes_geo).  A kernel that gains a
// parameter its entry does not append would make HIP read an argument slot nobody wrote; the table is therefore checked
// against the kernels' own signatures when this file is compiled.
#define CROW_MAX_LAUNCH_ARGS 18
template <typename F>
struct arity;
template <typename... A>
struct arity<void (*)(A...)> {
    static constexpr int value = (int)sizeof...(A);
};
template <int NARGS, int APPENDED, typename F>
constexpr int checked_nargs(F) {
    static_assert(arity<F>::value == NARGS + APPENDED, "a kernel's parameter list and its table entry disagree");
    static_assert(NARGS + APPENDED <= CROW_MAX_LAUNCH_ARGS, "the launcher's argument array is too short for this kernel");
    return NARGS;
}
#define CROW_FN(name, nargs) {#name, (const void*)&name, checked_nargs<nargs, 0>(&name), 0u, 0, 16, 0, 1, false, nullptr, false}
// ... with a twin for several rows of both operands per wave, which is handed the activation row count
#define CROW_FN_KEEP_ROWS(name, nargs, twin, rows) \
    {#name, (const void*)&name, checked_nargs<nargs, 0>(&name) + 0 * checked_nargs<nargs, 0>(&twin) + 0 * checked_nargs<nargs, 1>(&rows), 0u, 0, 16, 0, 1, false, nullptr, false, nullptr, nullptr, (const void*)&twin, false, (const void*)&rows}
#define CROW_FN_KEEP(name, nargs, twin) \
    {#name, (const void*)&name, checked_nargs<nargs, 0>(&name) + 0 * checked_nargs<nargs, 0>(&twin), 0u, 0, 16, 0, 1, false, nullptr, false, nullptr, nullptr, (const void*)&twin}
#define CROW_FN_KSPLIT(name, nargs) \
    {#name, (const void*)&name, checked_nargs<nargs, 0>(&name), 0u, 0, 16, 0, 1, false, nullptr, false, nullptr, nullptr, nullptr, true}
#define CROW_FN_GEO_TWIN(name, nargs, twin) \
    {#name, (const void*)&name, checked_nargs<nargs, 1>(&name) + 0 * checked_nargs<nargs, 1>(&twin), 0u, 0, 16, 0, 1, false, nullptr, true, nullptr, nullptr, (const void*)&twin}
#define CROW_FN_GEO(name, nargs) {#name, (const void*)&name, checked_nargs<nargs, 1>(&name), 0u, 0, 16, 0, 1, false, nullptr, true}
// NR tensors per block, bodies for 1 .. MMAX activation rows, bf16 or f32 activations
// (the bodies for several rows need more registers than a block of sixteen waves leaves each: they run in blocks of eight)
#define CROW_GEMV(name, nargs, NR, MMAX, XBF16) \
    {#name, (const void*)&name, checked_nargs<nargs, 2>(&name), 0u, NR, MMAX > 1 ? 8 : 16, crow::crow_gemv_lds_per_wave(MMAX, XBF16), MMAX > 1 ? (XBF16 ? CROW_MULTI_STRIPS_BF16 : CROW_MULTI_STRIPS) : 1, true, nullptr, false}
// ... with a twin for one strip per block
#define CROW_GEMV_ONE(name, nargs, NR, MMAX) \
    {#name, (const void*)&name, checked_nargs<nargs, 2>(&name) + 0 * checked_nargs<nargs, 2>(&name##_one), 0u, NR, 8, crow::crow_gemv_lds_per_wave(MMAX, false), CROW_MULTI_STRIPS, true, nullptr, false, (const void*)&name##_one}
// ... for two runs per wave
#define CROW_GEMV_TWO(name, nargs, twin) \
    {#name, (const void*)&name, checked_nargs<nargs, 2>(&name) + 0 * checked_nargs<nargs, 2>(&twin), 0u, 1, 8, crow::crow_gemv_lds_per_wave(4, false), CROW_MULTI_STRIPS, true, nullptr, false, nullptr, (const void*)&twin}
#define CROW_GEMV_GEO(name, nargs, NR, MMAX, XBF16) \
    {#name, (const void*)&name, checked_nargs<nargs, 3>(&name), 0u, NR, 16, crow::crow_gemv_lds_per_wave(MMAX, XBF16), 1, true, nullptr, true}
const FnEntry g_table[] = {
    CROW_GEMV(gemv_nvfp4_w, 6, 1, 1, false),       CROW_GEMV(gemv_nvfp4_w_bf16, 6, 1, 1, true),  CROW_GEMV(gemv_nvfp4_w_argmax, 7, 1, 1, false),
    CROW_GEMV(gemv_nvfp4_gu, 8, 2, 1, false),      CROW_GEMV(gemv_nvfp4_gu_bf16, 8, 2, 1, true),
    CROW_GEMV_ONE(gemv_nvfp4_wm, 7, 1, 4),         CROW_GEMV_ONE(gemv_nvfp4_gum, 9, 2, 4),
    CROW_GEMV(gemv_nvfp4_wm_bf16, 7, 1, 4, true),  CROW_GEMV(gemv_nvfp4_gum_bf16, 9, 2, 4, true), CROW_GEMV(gemv_fp4, 6, 1, 1, false),
    CROW_GEMV_TWO(gemv_fp4_b, 7, gemv_fp4_b_two),  CROW_GEMV_TWO(gemv_fp4_b1k, 7, gemv_fp4_b_two), CROW_GEMV_TWO(gemv_fp4_bs, 8, gemv_fp4_bs_two),
    CROW_GEMV(gemv_fp4_ptrb, 8, 1, 1, false),      CROW_GEMV(moe_gate_up_silu, 8, 2, 1, false),  CROW_GEMV_GEO(moe_down_combine, 7, 1, 1, false),
    {"moe_route_gate_up_silu", (const void*)&moe_route_gate_up_silu, checked_nargs<11, 3>(&moe_route_gate_up_silu) + 0 * checked_nargs<11, 3>(&moe_route_gate_up_silu_whole), 0u, 2, 16,
     crow::crow_gemv_lds_per_wave(1, false), 1, true, nullptr, true, nullptr, nullptr, nullptr, false, nullptr, (const void*)&moe_route_gate_up_silu_whole},
    {"moe_gate_up_silu_grouped", (const void*)&moe_gate_up_silu_grouped, checked_nargs<11, 2>(&moe_gate_up_silu_grouped) + 0 * checked_nargs<11, 2>(&moe_gate_up_silu_grouped_tile), 0u, 2, 8, crow::crow_gemv_lds_per_wave(4, false), CROW_MULTI_STRIPS, true, (const void*)&moe_gate_up_silu_grouped_tile, false},
    {"moe_down_grouped", (const void*)&moe_down_grouped, checked_nargs<9, 2>(&moe_down_grouped) + 0 * checked_nargs<9, 2>(&moe_down_grouped_tile), 0u, 1, 8, crow::crow_gemv_lds_per_wave(4, false), CROW_MULTI_STRIPS, true, (const void*)&moe_down_grouped_tile, false},
    CROW_FN_GEO(moe_group, 6),
    CROW_FN_GEO(router_top10, 10), CROW_FN_GEO(silu_mul_combo, 3),  CROW_FN_GEO_TWIN(acc_combo, 3, acc_combo_store),
    CROW_FN(argmax_k, 3),          CROW_FN(dequant_fp4_flat, 4),    CROW_FN(repack_nvfp4, 4),
    CROW_FN(unpack_nvfp4, 4),      CROW_FN(dequant_nvfp4_tiled, 5),
    // shared-X GEMM blocks: two staged X tiles of MT rows x 528 bytes
    {"gemm_nvfp4_bf16", (const void*)&gemm_nvfp4_bf16, checked_nargs<7, 0>(&gemm_nvfp4_bf16), 2u * 128u * 528u, 0, 16, 0, 1, false},
    {"gemm_nvfp4_bf16_m64", (const void*)&gemm_nvfp4_bf16_m64, checked_nargs<7, 0>(&gemm_nvfp4_bf16_m64), 2u * 64u * 528u, 0, 16, 0, 1, false},
    {"gemm_nvfp4_bf16_m48", (const void*)&gemm_nvfp4_bf16_m48, checked_nargs<7, 0>(&gemm_nvfp4_bf16_m48), 2u * 48u * 528u, 0, 16, 0, 1, false},
    {"gemm_nvfp4_bf16_m96", (const void*)&gemm_nvfp4_bf16_m96, checked_nargs<7, 0>(&gemm_nvfp4_bf16_m96), 2u * 96u * 528u, 0, 16, 0, 1, false},
    {"gemm_nvfp4_bf16_w48", (const void*)&gemm_nvfp4_bf16_w48, checked_nargs<7, 0>(&gemm_nvfp4_bf16_w48), 2u * 48u * 528u, 0, 8, 0, 1, false},
    {"gemm_nvfp4_bf16_w64", (const void*)&gemm_nvfp4_bf16_w64, checked_nargs<7, 0>(&gemm_nvfp4_bf16_w64), 2u * 64u * 528u, 0, 8, 0, 1, false},
    {"gemm_nvfp4_bf16_w80", (const void*)&gemm_nvfp4_bf16_w80, checked_nargs<7, 0>(&gemm_nvfp4_bf16_w80), 2u * 80u * 528u, 0, 8, 0, 1, false},
    {"gemm_nvfp4_bf16_w96", (const void*)&gemm_nvfp4_bf16_w96, checked_nargs<7, 0>(&gemm_nvfp4_bf16_w96), 2u * 96u * 528u, 0, 8, 0, 1, false},
    {"gemm_nvfp4_bf16_t64", (const void*)&gemm_nvfp4_bf16_t64, checked_nargs<7, 0>(&gemm_nvfp4_bf16_t64), 2u * 64u * 528u, 0, 4, 0, 1, false},
    {"gemm_nvfp4_bf16_t96", (const void*)&gemm_nvfp4_bf16_t96, checked_nargs<7, 0>(&gemm_nvfp4_bf16_t96), 2u * 96u * 528u, 0, 4, 0, 1, false},
    {"gemm_nvfp4_bf16_t128", (const void*)&gemm_nvfp4_bf16_t128, checked_nargs<7, 0>(&gemm_nvfp4_bf16_t128), 2u * 128u * 528u, 0, 4, 0, 1, false},
    CROW_FN_KSPLIT(gemm_nvfp4_bf16_m32, 7), CROW_FN_KSPLIT(gemm_nvfp4_bf16_m16, 7), CROW_FN_KEEP(gemv_bf16_w, 5, gemv_bf16_ahead),
    CROW_FN_KEEP(gemv_bf16, 5, gemv_bf16_ahead), CROW_FN_KEEP(gemv_bf16_b, 5, gemv_bf16_ahead), CROW_FN_KEEP_ROWS(gemv_b, 5, gemv_b_ahead, gemv_b_rows),
    CROW_FN_KEEP(gemv_bf16_ws, 5, gemv_bf16_ws_ahead), CROW_FN_KEEP(gemv_bf16_bs, 6, gemv_bf16_bs_ahead),
    CROW_FN(gemv_nvfp4_w_valu1, 6), CROW_FN(gemv_nvfp4_w_valu2, 6), CROW_FN(gemv_nvfp4_w_valu4, 6),  // measurement only
};
const int g_table_n = (int)(sizeof(g_table) / sizeof(g_table[0]));

// The K-split GEMM kernels (gemm.h) by [16-token blocks - 1][strips - 1] of a block
struct KSplitEntry {
    const void* stub;
    int max_waves, lds_per_wave;
};
#define CROW_KSPLIT_ROW(TBK, NJ, MT, WAVES) \
    {(const void*)&gemm_ksplit_##MT##x##NJ, WAVES + 0 * checked_nargs<7, 2>(&gemm_ksplit_##MT##x##NJ), crow::KSplitTile<TBK, NJ>::AREA},
#define CROW_KSPLIT_NJ 5
const KSplitEntry g_ksplit[4 * CROW_KSPLIT_NJ] = {CROW_GEMM_KSPLIT_ALL(CROW_KSPLIT_ROW)};

const int STREAM_SLOTS = 4;
struct State {
    bool ready = false;
    int device = -1;
    int cus = 256;
    hipStream_t stream = nullptr;
    crow::Workspace ws{};  // the null stream's, and any stream's beyond the first STREAM_SLOTS others
    crow::Workspace ws_more[STREAM_SLOTS] = {};  // those streams': same roles and sizes, the one status word
    crow::Workspace ws_static{};  // the same roles inside `scratch`, through the device address crow_hip_init asked for
    unsigned* said = nullptr;  // pinned host words: the two status words as the layout calls last read them, eight pairs in turn
    int* scalars = nullptr;  // device words for the library's own launches: (rows, k_dim) of the layout calls, the encoder's maxima
    char name[256] = {0};
    crow::Geo model{0, 0, 0, 0};  // the routed geometry (crow_hip_set_geo): appended by value to the kernels that take it
    size_t lds_cap = 64u * 1024u;  // most LDS one workgroup may take on this device
} g;
std::atomic<hipStream_t> g_slot_of[STREAM_SLOTS];  // which stream ws_more[i] belongs to; kept until crow_hip_shutdown (a graph captured there may outlive the stream)
std::atomic<bool> g_other_streams{false};  // a launch has gone to a stream that is not the null stream (or been captured from one)

// Scratch memory of crow_hip_launch_noalloc: part of the code object, so it exists on a device from the moment the library
// is loaded there until the process ends, and no call ever allocates it.  Words [0, NOALLOC_PARTIAL_FLOATS) hold the partial
// sums of split launches, then NOALLOC_COUNTER_SLOTS arrival counters, the status word (alone on 32 words), and the fused
// head's keys (8 bytes per strip).
const unsigned HEAD_WORDS = 65536;  // the allocated workspace: heads of up to 1,048,576 rows
const unsigned NOALLOC_HEAD_WORDS = CROW_NOALLOC_MAX_HEAD_STRIPS;
const unsigned NOALLOC_PARTIAL_FLOATS = CROW_NOALLOC_MAX_PARTIAL_FLOATS;  // 4 MiB of split-K partial sums
const unsigned NOALLOC_COUNTER_SLOTS = CROW_NOALLOC_MAX_STRIPS;
const unsigned NOALLOC_TAIL_WORDS = 32 + 2 * NOALLOC_HEAD_WORDS;  // status line, then the head's 8-byte words
const unsigned NOALLOC_WORDS = NOALLOC_PARTIAL_FLOATS + NOALLOC_COUNTER_SLOTS + NOALLOC_TAIL_WORDS;
static __device__ __align__(256) unsigned scratch[NOALLOC_WORDS];
static_assert(sizeof(unsigned) * NOALLOC_WORDS == CROW_NOALLOC_SCRATCH_BYTES, "the header states the array's size");

const unsigned long long PARTIAL_FLOATS = 16ull << 20;  // 64 MiB of split-K partial sums
const unsigned COUNTER_SLOTS = 1u << 16;
// tile counters, then the status word
const unsigned COUNTER_WORDS = COUNTER_SLOTS + 1;

int hip_rc(hipError_t e) { return e == hipSuccess ? CROW_OK : (int)e; }

const FnEntry* find(const char* name) {
    if (!name) return nullptr;
    for (int i = 0; i < g_table_n; i++)
        if (strcmp(g_table[i].name, name) == 0) return &g_table[i];
    return nullptr;
}

// a handle is the address of a table entry, nothing else
const FnEntry* entry_of(crow_fn_t f) {
    const FnEntry* e = (const FnEntry*)(void*)f;
    if (e < g_table || e >= g_table + g_table_n) return nullptr;
    if (((const char*)e - (const char*)g_table) % (ptrdiff_t)sizeof(FnEntry) != 0) return nullptr;
    return e;
}


// The scratch memory of launches on stream s, and whether launches on other streams leave it alone
const crow::Workspace& workspace_of(hipStream_t s, bool& own) {
    own = true;
    if (s == nullptr || s == hipStreamLegacy) return g.ws;
    if (s != hipStreamPerThread)  // (one handle, a stream per thread)
        for (int i = 0; i < STREAM_SLOTS; i++) {
            hipStream_t at = g_slot_of[i].load();
            if (at == nullptr && g_slot_of[i].compare_exchange_strong(at, s)) return g.ws_more[i];
            if (at == s) return g.ws_more[i];
        }
    own = false;
    return g.ws;
}

// Groups per strip if the grouped expert kernels take their twin for K / 64 = pairs (strips of two to eight groups that one
// wave walks alone in the launch shapes chosen below: up to 7 groups for one tensor, 10 - here 8 - per tensor for two), else 0.
unsigned tile_groups(int nr, unsigned pairs) {
    const unsigned groups = (pairs + CROW_GROUP_PAIRS - 1) / CROW_GROUP_PAIRS;
    return groups >= 2 && groups <= (nr == 2 ? (unsigned)CROW_TILE_MAX_GROUPS : 7u) ? groups : 0u;
}

// The launch dimensions of the GEMV family carry the problem in `gy` (crow_hip_launch_dims writes it, callers pass it on
// unchanged): bits 0..19 = K / 64, bits 20..23 = activation rows of the last token group (0 = not given), bits 24..31 = S, the
// number of column slices per strip.  The real grid is (gx, S, gz); the low 24 bits reach the kernel by value.
// `ws`: the scratch memory the launch may use, handed by value to the kernels that take one; `own_ws`: no launch on another stream uses it.
int launch_entry(const FnEntry* e, dim3 grid, dim3 block, const uint64_t* vals, uint32_t n, hipStream_t s, const crow::Workspace& ws, bool own_ws) {
    if (!g.ready) return CROW_ERR_NOT_INITIALIZED;
    if (!e || !vals) return CROW_ERR_BAD_ARGUMENT;
    if ((int)n != e->nargs) return CROW_ERR_ARG_COUNT;
    // whole wavefronts only: every kernel derives its wave count (and its LDS layout) from block.x / 64
    if (grid.x == 0 || grid.y == 0 || grid.z == 0 || block.x == 0 || block.x > 64u * (unsigned)e->max_waves || block.x % 64 != 0) return CROW_ERR_BAD_ARGUMENT;
    void* args[CROW_MAX_LAUNCH_ARGS];
    for (uint32_t i = 0; i < n; i++) args[i] = (void*)&vals[i];
    uint32_t na = n;
    size_t lds = e->lds_fixed;
    int geo = 0;
    crow::Workspace ws_arg = ws;
    const void* stub = e->stub;
    if (e->nr != 0) {
        const unsigned word = grid.y;
        const int pairs = (int)(word & 0xFFFFFu);
        const int waves = (int)(block.x / 64), wpt = waves / e->nr;
        if (pairs == 0 || wpt == 0) return CROW_ERR_BAD_ARGUMENT;
        if (e->tile_stub != nullptr && tile_groups(e->nr, (unsigned)pairs) != 0 && block.x <= 512) {
            // the twin for strips that one wave walks alone: strips per wave ride where S sits (such a strip is never cut into
            // slices), and the kernel takes the whole word; one staging area per group and block
            if ((word >> 24) == 0) return CROW_ERR_BAD_ARGUMENT;
            stub = e->tile_stub;
            geo = (int)word;
            grid.y = 1;
            lds = (size_t)CROW_GEMV_ZERO_BYTES + (size_t)tile_groups(e->nr, (unsigned)pairs) * (size_t)(e->lds_per_wave / 2);
        } else {
            const bool one = e->one_stub != nullptr && (word >> 24) == CROW_ONE_STRIP && pairs <= 64 * CROW_GROUP_PAIRS;
            const bool two = e->two_stub != nullptr && (word >> 24) == CROW_TWO_RUNS && pairs <= 64 * CROW_GROUP_PAIRS;
            const bool store = e->stub == (const void*)&moe_down_combine && (word >> 24) == CROW_STORE;
            const int slices = one || two || store || (word >> 24) == 0 ? 1 : (int)(word >> 24);
            if (one) stub = e->one_stub;
            if (two) stub = e->two_stub;
            lds = (size_t)CROW_GEMV_ZERO_BYTES + (size_t)waves * (size_t)e->lds_per_wave;
            // a split launch must fit the scratch memory it is given (the kernels check again and report through the status word)
            if (slices > 1 && ((unsigned long long)grid.x * grid.z * (unsigned)slices * (unsigned)(e->nr * (one ? 1 : e->ns)) * 64ull > ws.partial_floats ||
                               (unsigned long long)grid.x * grid.z > ws.counter_slots))
                return CROW_ERR_WORKSPACE;
            geo = (int)(word & 0xFFFFFFu);
            if (store) geo = pairs | CROW_GEO_STORE;
            const int groups = (pairs + CROW_GROUP_PAIRS - 1) / CROW_GROUP_PAIRS;
            if (e->whole_stub != nullptr && waves == 2 && slices == 1 && groups <= CROW_WHOLE_GROUPS) {
                stub = e->whole_stub;
                lds = (size_t)crow::crow_gemv_lds_whole(groups);
            }
            grid.y = (unsigned)slices;
        }
        if (lds > g.lds_cap) return CROW_ERR_SHAPE;
        args[na++] = (void*)&geo;
    }
    bool with_ws = e->takes_ws;
    if (e->ksplit && (grid.z & CROW_KSPLIT) != 0) {
        const unsigned word = grid.z, nj = (word >> 8) & 0xFu, tbk = (word >> 12) & 0xFu, most = (word >> 16) & 0xFFu;
        if (nj < 1 || nj > CROW_KSPLIT_NJ || tbk < 1 || tbk > 4 || most == 0 || (word & 0xFFu) == 0) return CROW_ERR_BAD_ARGUMENT;
        const KSplitEntry& k = g_ksplit[(tbk - 1) * CROW_KSPLIT_NJ + nj - 1];
        if (block.x > 64u * (unsigned)k.max_waves) return CROW_ERR_BAD_ARGUMENT;
        stub = k.stub;
        // slices meet in scratch memory: a stream that has none of its own keeps the panels in one block (other bits, no slices)
        grid.z = own_ws ? word & 0xFFu : 1u;
        // (the kernel checks again and reports through the status word)
        if (grid.z > 1 && ((unsigned long long)grid.x * grid.y * nj * grid.z * 256ull * tbk > ws.partial_floats ||
                           (unsigned long long)grid.x * grid.y * nj > ws.counter_slots))
            return CROW_ERR_WORKSPACE;
        lds = (size_t)(block.x / 64) * (size_t)k.lds_per_wave;
        if (lds > g.lds_cap) return CROW_ERR_SHAPE;
        geo = (int)most;
        args[na++] = (void*)&geo;
        with_ws = true;
    }
    if (e->twin_stub != nullptr && grid.z == CROW_TWIN) {
        stub = e->twin_stub;
        grid.z = 1;
    }
    if (e->rows_stub != nullptr && (grid.z & CROW_ROWS) != 0) {
        geo = (int)(grid.z & ~CROW_ROWS);
        if (geo < 1) return CROW_ERR_BAD_ARGUMENT;
        stub = e->rows_stub;
        grid.z = 1;
        args[na++] = (void*)&geo;
    }
    if (with_ws) args[na++] = (void*)&ws_arg;
    crow::Geo model_arg = g.model;
    if (e->takes_geo) args[na++] = (void*)&model_arg;
    const bool head = e->stub == (const void*)&gemv_nvfp4_w_argmax;
    // the fused head keeps one key per strip (the kernel checks again and reports through the status word)
    if (head && grid.x > ws.head_words) return CROW_ERR_WORKSPACE;
    if (s != nullptr) g_other_streams.store(true);  // (before the launch: see layout_launch)
    hipError_t rc = hipLaunchKernel(stub, grid, block, args, lds, s);
    if (rc == hipSuccess && head) {  // ... and its finishing kernel right behind it: the token out of the strips' keys
        unsigned strips = grid.x;
        void* fargs[3] = {(void*)&vals[6], (void*)&strips, (void*)&ws_arg};
        rc = hipLaunchKernel((const void*)&argmax_finish, dim3(1), dim3(1024), fargs, 0, s);
    }
    if (rc != hipSuccess) (void)hipGetLastError();  // reported here: not left behind for an unrelated later call to find
    return hip_rc(rc);
}
int launch_on(const FnEntry* e, dim3 grid, dim3 block, const uint64_t* vals, uint32_t n, hipStream_t s) {
    if (!g.ready) return CROW_ERR_NOT_INITIALIZED;
    bool own;
    const crow::Workspace& ws = workspace_of(s, own);
    return launch_entry(e, grid, block, vals, n, s, ws, own);
}

}  // namespace

extern "C" {

int crow_hip_init(int device) {
    if (g.ready) return g.device == device ? CROW_OK : CROW_ERR_BAD_ARGUMENT;
    hipError_t e = hipSetDevice(device);
    if (e != hipSuccess) return (int)e;
    hipDeviceProp_t pr;
    if ((e = hipGetDeviceProperties(&pr, device)) != hipSuccess) return (int)e;
    snprintf(g.name, sizeof g.name, "%s (%s), %d CUs", pr.name, pr.gcnArchName, pr.multiProcessorCount);
    if (strncmp(pr.gcnArchName, "gfx950", 6) != 0) {
        fprintf(stderr, "crow_hip: this library holds gfx950 code objects only; device %d is %s\n", device, pr.gcnArchName);
        return CROW_ERR_BAD_ARGUMENT;
    }
    g.cus = pr.multiProcessorCount;
    g.lds_cap = pr.maxSharedMemoryPerMultiProcessor > 0 ? (size_t)pr.maxSharedMemoryPerMultiProcessor : (size_t)pr.sharedMemPerBlock;
    crow::Workspace ws{};
    ws.partial_floats = PARTIAL_FLOATS;
    ws.counter_slots = COUNTER_SLOTS;
    crow::Workspace more[STREAM_SLOTS] = {};
    int* scalars = nullptr;
    unsigned* said = nullptr;
    // one failure path: everything allocated so far is released again
    auto fail = [&](hipError_t why) {
        (void)hipFree(ws.partials);
        (void)hipFree(ws.counters);
        (void)hipFree(ws.head);
        for (crow::Workspace& m : more) (void)hipFree(m.partials), (void)hipFree(m.counters), (void)hipFree(m.head);
        (void)hipFree(scalars);
        (void)hipHostFree(said);
        return (int)why;
    };
    if ((e = hipMalloc((void**)&ws.partials, PARTIAL_FLOATS * sizeof(float))) != hipSuccess) return fail(e);
    if ((e = hipMalloc((void**)&ws.counters, COUNTER_WORDS * sizeof(unsigned))) != hipSuccess) return fail(e);
    if ((e = hipMalloc((void**)&ws.head, HEAD_WORDS * sizeof(unsigned long long))) != hipSuccess) return fail(e);
    if ((e = hipMemset(ws.head, 0, HEAD_WORDS * sizeof(unsigned long long))) != hipSuccess) return fail(e);
    ws.head_words = HEAD_WORDS;
    if ((e = hipMalloc((void**)&scalars, 32 * sizeof(int))) != hipSuccess) return fail(e);  // words 0..15: (rows, k_dim) of the layout calls, 16..23: the encoder's maxima, 24: the read probe's sink
    if ((e = hipHostMalloc((void**)&said, 16 * sizeof(unsigned), hipHostMallocDefault)) != hipSuccess) return fail(e);
    if ((e = hipMemset(ws.counters, 0, COUNTER_WORDS * sizeof(unsigned))) != hipSuccess) return fail(e);
    ws.status = ws.counters + COUNTER_SLOTS;
    for (crow::Workspace& m : more) {
        m = crow::Workspace{nullptr, nullptr, PARTIAL_FLOATS, COUNTER_SLOTS, ws.status, nullptr, HEAD_WORDS};
        if ((e = hipMalloc((void**)&m.partials, PARTIAL_FLOATS * sizeof(float))) != hipSuccess) return fail(e);
        if ((e = hipMalloc((void**)&m.counters, COUNTER_WORDS * sizeof(unsigned))) != hipSuccess) return fail(e);
        if ((e = hipMalloc((void**)&m.head, HEAD_WORDS * sizeof(unsigned long long))) != hipSuccess) return fail(e);
        if ((e = hipMemset(m.head, 0, HEAD_WORDS * sizeof(unsigned long long))) != hipSuccess) return fail(e);
        if ((e = hipMemset(m.counters, 0, COUNTER_WORDS * sizeof(unsigned))) != hipSuccess) return fail(e);
    }
    if ((e = hipMemcpyToSymbol(HIP_SYMBOL(crow::g_ws), &ws, sizeof ws)) != hipSuccess) return fail(e);
    // a GEMV block of 16 waves, and the GEMM's two staged X tiles, need more dynamic LDS than the default per-block limit
    for (int i = 0; i < g_table_n; i++) {
        size_t most = g_table[i].lds_fixed;
        if (g_table[i].nr != 0) {  // the GEMV family: the largest block the kernel takes, within the device's limit
            most = (size_t)CROW_GEMV_ZERO_BYTES + (size_t)g_table[i].max_waves * (size_t)g_table[i].lds_per_wave;
            if (most > g.lds_cap) most = g.lds_cap;
        }
        if (most > 48 * 1024 &&
            (e = hipFuncSetAttribute(g_table[i].stub, hipFuncAttributeMaxDynamicSharedMemorySize, (int)most)) != hipSuccess)
            return fail(e);
        for (const void* twin : {g_table[i].one_stub, g_table[i].two_stub})
            if (twin != nullptr && most > 48 * 1024 &&
                (e = hipFuncSetAttribute(twin, hipFuncAttributeMaxDynamicSharedMemorySize, (int)most)) != hipSuccess)
                return fail(e);
        // the twin for short strips stages up to eight groups of twelve rows per block
        const size_t tile_most = (size_t)CROW_GEMV_ZERO_BYTES + (size_t)CROW_TILE_MAX_GROUPS * (size_t)(g_table[i].lds_per_wave / 2);
        if (g_table[i].tile_stub != nullptr && tile_most > 48 * 1024 &&
            (e = hipFuncSetAttribute(g_table[i].tile_stub, hipFuncAttributeMaxDynamicSharedMemorySize, (int)tile_most)) != hipSuccess)
            return fail(e);
    }
    for (const KSplitEntry& k : g_ksplit) {
        const size_t most = (size_t)k.max_waves * (size_t)k.lds_per_wave;
        if (most > 48 * 1024 && (e = hipFuncSetAttribute(k.stub, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(most < g.lds_cap ? most : g.lds_cap))) != hipSuccess) return fail(e);
    }
    // `scratch` in host code is a stand-in, not a device address: ask for this device's copy once, and use only that
    unsigned* sp = nullptr;
    if ((e = hipGetSymbolAddress((void**)&sp, HIP_SYMBOL(scratch))) != hipSuccess || sp == nullptr) return fail(e != hipSuccess ? e : hipErrorInvalidSymbol);
    crow::Workspace st{};
    st.partials = (float*)sp;
    st.partial_floats = NOALLOC_PARTIAL_FLOATS;
    st.counters = sp + NOALLOC_PARTIAL_FLOATS;
    st.counter_slots = NOALLOC_COUNTER_SLOTS;
    st.status = st.counters + NOALLOC_COUNTER_SLOTS;
    st.head = (unsigned long long*)(st.status + 32);
    st.head_words = NOALLOC_HEAD_WORDS;
    // counters, status and key start at zero (a process that shut the library down and initialises it again included)
    if ((e = hipMemset(st.counters, 0, (NOALLOC_COUNTER_SLOTS + NOALLOC_TAIL_WORDS) * sizeof(unsigned))) != hipSuccess) return fail(e);
    if ((e = hipDeviceSynchronize()) != hipSuccess) return fail(e);
    g.scalars = scalars;
    g.said = said;
    g.ws = ws;
    for (int i = 0; i < STREAM_SLOTS; i++) g.ws_more[i] = more[i];
    g.ws_static = st;
    g.device = device;
    g.stream = nullptr;
    g.ready = true;
    return CROW_OK;
}

int crow_hip_shutdown(void) {
    if (!g.ready) return CROW_OK;
    (void)hipDeviceSynchronize();
    (void)hipFree(g.ws.partials);
    (void)hipFree(g.ws.counters);
    (void)hipFree(g.ws.head);
    for (int i = 0; i < STREAM_SLOTS; i++) {
        (void)hipFree(g.ws_more[i].partials), (void)hipFree(g.ws_more[i].counters), (void)hipFree(g.ws_more[i].head);
        g_slot_of[i].store(nullptr);
    }
    (void)hipFree(g.scalars);
    (void)hipHostFree(g.said);
    g = State{};
    return CROW_OK;
}

const char* crow_hip_error_string(int code) {
    switch (code) {
        case CROW_OK: return "ok";
        case CROW_ERR_NOT_INITIALIZED: return "crow_hip_init has not been called";
        case CROW_ERR_KERNEL_MISSING: return "kernel missing";
        case CROW_ERR_BAD_ARGUMENT: return "bad argument";
        case CROW_ERR_ARG_COUNT: return "wrong number of kernel arguments";
        case CROW_ERR_WORKSPACE: return "launch does not fit the split-K workspace";
        case CROW_ERR_SCALE_BYTE: return "scale byte 0xFF in an NVFP4 tensor (no encoder emits it; E4M3 cannot hold 480)";
        case CROW_ERR_SHAPE: return "shape not supported by this kernel";
        case CROW_ERR_GEO: return "geometry not set or out of range (crow_hip_set_geo)";
        default: return code > 0 ? hipGetErrorString((hipError_t)code) : "unknown crow_hip error";
    }
}

int crow_hip_device_name(char* out, size_t n) {
    if (!g.ready) return CROW_ERR_NOT_INITIALIZED;
    if (!out || n == 0) return CROW_ERR_BAD_ARGUMENT;
    snprintf(out, n, "%s", g.name);
    return CROW_OK;
}

// The module is the library itself: load/unload exist so that the reference's
// compile -> Module -> get -> unload sequence keeps its shape.
int crow_hip_module_load(crow_module_t* out) {
    if (!g.ready) return CROW_ERR_NOT_INITIALIZED;
    if (!out) return CROW_ERR_BAD_ARGUMENT;
    *out = (crow_module_t)(void*)g_table;
    return CROW_OK;
}
int crow_hip_module_unload(crow_module_t m) { return m == (crow_module_t)(void*)g_table ? CROW_OK : CROW_ERR_BAD_ARGUMENT; }
int crow_hip_module_get(crow_module_t m, const char* name, crow_fn_t* out) {
    if (m != (crow_module_t)(void*)g_table) return CROW_ERR_BAD_ARGUMENT;
    return crow_hip_get_function(name, out);
}
int crow_hip_get_function(const char* name, crow_fn_t* out) {
    if (!out || !name) return CROW_ERR_BAD_ARGUMENT;
    const FnEntry* e = find(name);
    if (!e) {
        *out = nullptr;
        return CROW_ERR_KERNEL_MISSING;
    }
    *out = (crow_fn_t)(void*)e;
    return CROW_OK;
}
int crow_hip_function_count(void) { return g_table_n; }
const char* crow_hip_function_name(int index) { return index >= 0 && index < g_table_n ? g_table[index].name : nullptr; }
int crow_hip_function_arg_count(crow_fn_t f) {
    const FnEntry* e = entry_of(f);
    return e ? e->nargs : CROW_ERR_BAD_ARGUMENT;
}

int crow_hip_set_geo(int experts, int topk, int hidden, int inter) {
    if (!g.ready) return CROW_ERR_NOT_INITIALIZED;
    if (experts < 0 || topk < 0 || hidden < 0 || inter < 0) return CROW_ERR_BAD_ARGUMENT;
    // what the routing kernels take: no routed experts at all, or a power of two of them in 64..1024 with 1..16 picks
    if (experts != 0 && (experts < 64 || experts > 1024 || (experts & (experts - 1)) != 0 || topk < 1 || topk > 16)) return CROW_ERR_GEO;
    // host state only: launches started from now on carry it by value (nothing is copied, nothing waits)
    g.model = crow::Geo{experts, topk, hidden, inter};
    return CROW_OK;
}

int crow_hip_launch(crow_fn_t f, uint32_t gx, uint32_t gy, uint32_t gz, uint32_t bx, const uint64_t* vals, uint32_t n_vals,
                    void* stream) {
    const FnEntry* e = entry_of(f);
    if (!e) return CROW_ERR_KERNEL_MISSING;
    return launch_on(e, dim3(gx, gy, gz), dim3(bx, 1, 1), vals, n_vals, stream ? (hipStream_t)stream : g.stream);
}

int crow_hip_launch_noalloc(crow_fn_t f, uint32_t gx, uint32_t gy, uint32_t gz, uint32_t bx, const uint64_t* vals,
                            uint32_t n_vals, void* stream) {
    const FnEntry* e = entry_of(f);
    if (!e) return CROW_ERR_KERNEL_MISSING;
    // only kernels that are handed their scratch memory as an argument can be pointed at the static array
    if (!e->takes_ws) return CROW_ERR_BAD_ARGUMENT;
    // launch_entry refuses (CROW_ERR_WORKSPACE) a split whose partial sums or counters do not fit what it is given
    return launch_entry(e, dim3(gx, gy, gz), dim3(bx, 1, 1), vals, n_vals, stream ? (hipStream_t)stream : g.stream, g.ws_static, false);
}

// Token rows, waves, strips and column slices of a K-split GEMM block (gemm.h: KSplitTile) for m token rows: what the following time is least
// for, of 1 to 5 strips, 4 / 8 / 12 waves, 1 to 8 slices and, beyond 64 rows, 48 or 64 rows a block.  `rounds` of blocks one behind the other, as many of them together on a
// compute unit as registers and LDS allow; panels per wave and per block; blocks per compute unit.
//   us = c0 + (slices > 1) (c1 + c2 slices) + rounds (c3 + panels per wave (c4 + c5 strips)) + rounds together panels (c6 strips + c7)
//        + blocks / compute units (panels (c8 strips + c9) + c10 strips) + c11 waves
// was fitted to the times of all of them on MI355X at 104 tensors (rows 512 .. 17408, K 512 .. 17408) x 5, 16, 17, 32, 48 and 64 rows, and at
// those for which gemm_choice names m32 x 96 .. 1999 rows; what it picks is 1 to 4 % behind the fastest on average.  Against the kernels
// that served these sizes before: 1.34 (64 rows) to 1.69 times as fast (17 rows), 1.40 (96 rows) to 1.20 (1999 rows) on average, up to 4.4;
// never behind by more than the noise of launches of 6 us.
struct KSplitPlan {
    double us;
    uint32_t tbk, nj, waves, slices;
};
static KSplitPlan ksplit_search(uint32_t strips, uint32_t panels, uint32_t m, uint32_t force_s, uint32_t force_w) {
    static const double coef[6][12] = {{2.452, 1.165, 0.201, 0.72, 0.099, 0.208, 0.028, 0.026, 0.056, 0.007, 0.0, 0.041},
                                       {2.398, 1.281, 0.276, 0.914, 0.291, 0.211, 0.052, 0.036, 0.04, 0.048, 0.024, 0.079},
                                       {2.745, 1.182, 0.383, 0.836, 0.164, 0.373, 0.028, 0.16, 0.049, 0.047, 0.07, 0.106},
                                       {2.671, 1.108, 0.402, 1.149, 0.307, 0.321, 0.058, 0.147, 0.031, 0.097, 0.098, 0.145},
                                       {2.341, 0.991, 0.478, 0.925, 0.0, 0.405, 0.029, 0.093, 0.046, 0.101, 0.014, 0.138},   // several token blocks of 48 rows
                                       {2.082, 0.79, 0.567, 1.506, 0.0, 0.423, 0.046, 0.09, 0.037, 0.155, 0.016, 0.175}};  // ... of 64
    static const unsigned char waves_per_simd[4][CROW_KSPLIT_NJ] = {{7, 5, 4, 4, 3}, {5, 4, 4, 3, 3}, {5, 4, 4, 3, 2}, {4, 3, 3, 2, 2}};  // (their registers)
    const uint32_t cus = g.cus > 0 ? (uint32_t)g.cus : 256u;
    KSplitPlan best{0.0, 0, 0, 0, 0};
    for (uint32_t tbk = m <= 64 ? (m + 15) / 16 : 3; tbk <= (m <= 64 ? (m + 15) / 16 : 4); tbk++) {
        for (uint32_t nj = 1; nj <= CROW_KSPLIT_NJ; nj++) {
            const double* c = coef[m <= 64 ? tbk - 1 : tbk + 1];
            const KSplitEntry& k = g_ksplit[(tbk - 1) * CROW_KSPLIT_NJ + nj - 1];
            const uint32_t token_blocks = (m + 16 * tbk - 1) / (16 * tbk);
            const unsigned long long all_tiles = (unsigned long long)((strips + nj - 1) / nj) * token_blocks;
            if (all_tiles > 0x0FFFFFFFull) continue;
            const uint32_t tiles = (uint32_t)all_tiles;
            for (uint32_t w = 4; w <= 12; w += 4) {
                if (w > (uint32_t)k.max_waves || w < nj || (force_w > 0 && w != force_w)) continue;
                uint32_t fit = 4u * waves_per_simd[tbk - 1][nj - 1] / w;
                const uint32_t by_lds = 163840u / (w * (uint32_t)k.lds_per_wave);
                if (fit > by_lds) fit = by_lds;
                if (fit < 1) fit = 1;
                for (uint32_t s = 1; s <= 8; s += s < 4 ? 1 : 2) {
                    if (force_s > 0 && s != force_s) continue;
                    if (s > 1 && ((s - 1) * w >= panels || (unsigned long long)tiles * nj * s * 256ull * tbk > PARTIAL_FLOATS || (unsigned long long)tiles * nj > COUNTER_SLOTS)) continue;
                    const uint32_t blocks = tiles * s, n = (blocks + cus - 1) / cus, rounds = (n + fit - 1) / fit, together = n < fit ? n : fit;
                    const double own = (double)((panels + w * s - 1) / (w * s)), all = (double)panels / s, f = (double)blocks / cus, r = rounds;
                    const double us = c[0] + (s > 1 ? c[1] + c[2] * s : 0.0) + r * (c[3] + own * (c[4] + c[5] * nj)) + r * together * all * (c[6] * nj + c[7]) +
                                      f * (all * (c[8] * nj + c[9]) + c[10] * nj) + c[11] * w;
                    if (best.nj == 0 || us < best.us) best = KSplitPlan{us, tbk, nj, w, s};
                }
            }
        }
    }
    return best;
}
// The search takes 0.5 to 1 us, a tenth of a small call: each thread keeps what it found for the last shapes (a program has a few dozen).
static KSplitPlan ksplit_plan(uint32_t strips, uint32_t panels, uint32_t m, uint32_t force_s, uint32_t force_w) {
    if (force_s != 0 || force_w != 0) return ksplit_search(strips, panels, m, force_s, force_w);
    struct Kept {
        uint32_t strips, panels, m;
        int cus;
        KSplitPlan plan;
    };
    static thread_local Kept kept[64] = {};
    Kept& k = kept[(strips * 0x9E3779B1u ^ panels * 0x85EBCA6Bu ^ m * 0xC2B2AE35u) >> 26];
    if (k.strips != strips || k.panels != panels || k.m != m || k.cus != g.cus) k = Kept{strips, panels, m, g.cus, ksplit_search(strips, panels, m, 0, 0)};
    return k.plan;
}

// Which GEMM entry point for m token rows on a [rows, k_dim] tensor.  Up to 64 rows: the K-split kernels.  Beyond that the
// launch lasts as long as the fullest compute unit, which takes `rounds` = ceil(blocks / compute units) blocks: one behind the other
// where a block fills the unit (eight waves, or four that keep most registers), some of them together for m32 / m48 / m64.  Short
// blocks that deal one 64-row tile's K over four waves (m32) win while there are few; large products go to the blocks whose
// decoded weights serve the most tokens (t64 .. t128, 320 rows each), unless the last round is nearly empty with them and full with
// others ([8192, 5120] x 1536: w96 has 256 blocks, one round, 114 us; t96 416, two, 140).
//   us = rounds (a + b K / 1024) + blocks / compute units (c + d K / 1024) + (alone + alone_k K / 1024, one block on a unit)
// was fitted to every entry point's time on MI355X at 1,122 sizes (rows 512 .. 17408, K 256 .. 17408, 17 .. 1999 tokens), the eight-wave ones' again
// at 770 after their body changed; what it names is 0.6 % behind the fastest of them on average, up to 10 % at K = 256 and 512.  m32's line is that of
// the body it had alone then; the K-split kernels that its dimensions start now are 1.2 to 1.4 times as fast where it is named, and would win at
// more sizes (by up to 1.27 times around 128 tokens, [17408, 5120] x 128 50 us against m48's 55), which stay with the kernels that add in one order.
// 96- and 128-token blocks of the shared-X body (m96, the general name) are never ahead and are left to callers by name.
// An entry point that would refuse the product is left out: those that address X with 32-bit element offsets from its start (m K up
// to 2^32 - 1) and count token blocks in the grid's second dimension; the tall tiles count from a block's first token row (K < 2^25).
// If none takes it, m32 is named, whose refusal the status reports.
static const char* gemm_choice(uint32_t rows, uint32_t m, uint32_t k_dim, bool k_known) {
    if (m <= 16) return "gemm_nvfp4_bf16_m16";
    if (m <= 64) return "gemm_nvfp4_bf16_m32";
    static const struct { const char* name; uint32_t mt, strips; double a, b, c, d, alone, alone_k; } cand[] = {
        {"gemm_nvfp4_bf16_m32", 32, 4, 2.31, 1.46, 0.0, 0.44, 2.43, 0.48},    {"gemm_nvfp4_bf16_m48", 48, 16, 2.03, 6.56, 0.84, 1.81, 1.58, 2.46},
        {"gemm_nvfp4_bf16_m64", 64, 16, 3.03, 5.5, 0.84, 4.96, 1.01, 4.51},   {"gemm_nvfp4_bf16_w48", 48, 32, 5.6, 11.58, 1.12, 1.3, 0.0, 0.0},
        {"gemm_nvfp4_bf16_w64", 64, 32, 6.56, 13.13, 2.63, 1.64, 0.0, 0.0},   {"gemm_nvfp4_bf16_w80", 80, 32, 7.48, 13.91, 3.55, 2.14, 0.0, 0.0},
        {"gemm_nvfp4_bf16_w96", 96, 32, 8.4, 14.89, 4.77, 2.49, 0.0, 0.0},    {"gemm_nvfp4_bf16_t64", 64, 20, 5.53, 10.69, 1.98, 0.0, 0.0, 0.0},
        {"gemm_nvfp4_bf16_t96", 96, 20, 4.69, 12.31, 5.31, 0.0, 0.0, 0.0},    {"gemm_nvfp4_bf16_t128", 128, 20, 9.56, 12.71, 1.44, 1.72, 0.0, 0.0}};
    const unsigned long long strips = (rows + CROW_STRIP_ROWS - 1) / CROW_STRIP_ROWS;
    const unsigned long long cus = g.cus > 0 ? (unsigned long long)g.cus : 256ull;
    const double k = (double)k_dim / 1024.0;
    const char* best = nullptr;
    double best_t = 0.0;
    for (const auto& c : cand) {
        const unsigned long long token_blocks = (m + c.mt - 1ull) / c.mt, blocks = ((strips + c.strips - 1) / c.strips) * token_blocks;
        const bool tall = c.name[16] == 't';
        if (tall ? k_dim >= 1u << 25 || blocks > 0x7FFFFFFFull : token_blocks > 65535 || (k_known && (unsigned long long)m * k_dim > 0xffffffffull)) continue;
        const unsigned long long rounds = (blocks + cus - 1) / cus;
        const double t = (double)rounds * (c.a + c.b * k) + (double)blocks / (double)cus * (c.c + c.d * k) + (rounds == 1 ? c.alone + c.alone_k * k : 0.0);
        if (best == nullptr || t < best_t) {
            best_t = t;
            best = c.name;
        }
    }
    return best != nullptr ? best : cand[0].name;
}
const char* crow_hip_gemm_kernel(uint32_t rows, uint32_t m) { return gemm_choice(rows, m, 5120, false); }
const char* crow_hip_gemm_kernel_for(uint32_t rows, uint32_t m, uint32_t k_dim) { return gemm_choice(rows, m, k_dim, true); }

// Split of a [rows, k_dim] product over the chip.  A block owns one 16-row strip; the strip's 256-column groups are dealt
// to W waves of the block (combined in LDS) and, only when a strip has more groups than one block's waves can hold, to S
// blocks (combined through the workspace).  The result depends on (rows, k_dim) only.
int crow_hip_launch_dims_split(const char* name, uint32_t rows, uint32_t k_dim, uint32_t z, uint32_t force_s, uint32_t force_w, crow_dims* out) {
    if (!out || !name || rows == 0) return CROW_ERR_BAD_ARGUMENT;
    const FnEntry* e = find(name);
    if (!e) return CROW_ERR_KERNEL_MISSING;
    // CROW_DIMS_COUNT_FROM_MEMORY (verify and token-row kernels only): the launch reads its row count from the word behind
    // m_p / t_p, as the reference's kernels do; the low bits are then the capacity the grid is sized for
    const bool from_memory = (z & CROW_DIMS_COUNT_FROM_MEMORY) != 0 || z == 0;
    z &= ~CROW_DIMS_COUNT_FROM_MEMORY;
    const bool combine = strcmp(name, "moe_down_combine") == 0 || strcmp(name, "acc_combo") == 0, store = combine && (z & CROW_DIMS_STORE) != 0;
    if (combine) z &= ~CROW_DIMS_STORE;
    {
        const bool takes_count = strcmp(name, "gemv_nvfp4_wm") == 0 || strcmp(name, "gemv_nvfp4_gum") == 0 || strcmp(name, "gemv_nvfp4_wm_bf16") == 0 ||
                                 strcmp(name, "gemv_nvfp4_gum_bf16") == 0 || strcmp(name, "gemv_fp4_b") == 0 || strcmp(name, "gemv_fp4_b1k") == 0 ||
                                 strcmp(name, "gemv_fp4_bs") == 0;
        if (from_memory && !takes_count) return CROW_ERR_BAD_ARGUMENT;
        if (z == 0) {
            if (strncmp(name, "gemv_nvfp4_", 11) != 0) return CROW_ERR_BAD_ARGUMENT;  // token rows: the capacity sizes the grid
            z = 4;                                                                   // the verify kernels' most
        }
    }
    const uint32_t strips = (rows + CROW_STRIP_ROWS - 1) / CROW_STRIP_ROWS;
    const uint32_t groups = (k_dim + CROW_GROUP_COLS - 1) / CROW_GROUP_COLS;
    const uint32_t rt = (rows + CROW_TILE_ROWS - 1) / CROW_TILE_ROWS, panels = groups;  // the GEMM's 64-row tiles
    if (strcmp(name, "gemv_bf16_w") == 0 || strcmp(name, "gemv_bf16") == 0 || strcmp(name, "gemv_bf16_b") == 0 || strcmp(name, "gemv_b") == 0 ||
        strcmp(name, "gemv_bf16_ws") == 0 || strcmp(name, "gemv_bf16_bs") == 0) {
        // z = T activation rows; whole 16-byte loads: 8 bf16 or 4 f32 weights
        if (k_dim == 0 || k_dim % (strcmp(name, "gemv_b") == 0 ? 4 : 8) != 0) return CROW_ERR_SHAPE;
        if (strcmp(name, "gemv_bf16") == 0 && z != 1) return CROW_ERR_SHAPE;  // the one-token form
        // short tensors: a block of four waves per (row, token); force_w = 4 / 1 asks for one shape or the other
        const bool f32 = strcmp(name, "gemv_b") == 0, block_per_row = force_w == 4 || (force_w == 0 && (unsigned long long)rows * z <= 2048);
        // Several rows against weights that the 256 MB memory-side cache cannot hold from one row to the next, and long bf16 rows in
        // more than three blocks per compute unit, are bound by memory: weights alone ahead (us, so / weights and activations together,
        // f32 [20000, 5120] x 4 231 / 258, [10240, 8192] x 2 103 / 109; bf16 [40000, 5120] x 2 141 / 150, [2048, 8192] x 1 8.5 / 9.0;
        // up to 256 MB together is ahead by up to 1.4 times: bf16 [10240, 8192] x 16 356 / 290)
        const bool ahead = (z > 1 && (unsigned long long)rows * k_dim * (f32 ? 4 : 2) > (256ull << 20)) ||
                           (!f32 && block_per_row && k_dim >= 4096 && (unsigned long long)rows * z > 768);
        // 4 x 4 rows per wave pay from about 8192 outputs on (us, a row each / 4 x 4: [256, 2048] x 24 5.0 / 5.7, x 32 5.9 / 5.7, x 64 9.6 / 6.0; [128, 2048] x 64
        // 5.9 / 5.7; [500, 2048] x 12 5.4 / 5.7, x 17 6.9 / 5.7; [256, 4096] x 64 16.7 / 8.2; [5000, 2048] x 3 18.7 / 9.0, x 500 2804 / 692)
        if (e->rows_stub != nullptr && force_w == 0 && !ahead && z >= 3 && z <= 0x7FFFFFFFu && (unsigned long long)rows * z >= 8192) {
            *out = crow_dims{(rows + 15) / 16, (z + 3) / 4, CROW_ROWS | z, 256};
            return CROW_OK;
        }
        *out = crow_dims{block_per_row ? rows : (rows + 3) / 4, z, ahead ? CROW_TWIN : 1u, 256};
        return CROW_OK;
    }
    if (e->nr != 0) {  // the NVFP4 GEMV family
        if (k_dim == 0 || k_dim % CROW_BLOCK_VALUES != 0 || k_dim / CROW_BLOCK_VALUES > 0xFFFFFu) return CROW_ERR_SHAPE;
        const uint32_t pairs = k_dim / CROW_BLOCK_VALUES;
        const bool down_combine = strcmp(name, "moe_down_combine") == 0;
        const bool routed = strcmp(name, "gemv_fp4_ptrb") == 0 || strncmp(name, "moe_", 4) == 0;
        const bool tokens = strcmp(name, "gemv_fp4_b") == 0 || strcmp(name, "gemv_fp4_b1k") == 0 || strcmp(name, "gemv_fp4_bs") == 0;
        const bool verify = strcmp(name, "gemv_nvfp4_wm") == 0 || strcmp(name, "gemv_nvfp4_gum") == 0 || strcmp(name, "gemv_nvfp4_wm_bf16") == 0 ||
                            strcmp(name, "gemv_nvfp4_gum_bf16") == 0;
        if (down_combine) {  // rows = hidden; one wave per picked expert, every wave all columns of its strip
            if (g.model.topk < 1 || g.model.topk > 16) return CROW_ERR_GEO;
            *out = crow_dims{strips, pairs | ((store ? CROW_STORE : 1u) << 24), z, 64u * (uint32_t)g.model.topk};
            return CROW_OK;
        }
        if (e->tile_stub != nullptr && tile_groups(e->nr, pairs) != 0) {
            // about sixteen records per wave; eight waves per block where the staged rows are large (two blocks per compute unit)
            // (force_s / force_w: strips per wave / waves per block, for measurements)
            uint32_t spw = 16u / ((uint32_t)e->nr * groups);
            if (spw < 1) spw = 1;
            if (force_s > 0) spw = force_s > 255 ? 255 : force_s;
            const uint32_t wb = force_w > 0 ? (force_w > 8 ? 8 : force_w) : (groups > 4 ? 8u : 4u), per_block = wb * spw;
            *out = crow_dims{(strips + per_block - 1) / per_block, pairs | (spw << 24), z, 64u * wb};
            return CROW_OK;
        }
        if (verify && z > 4) return CROW_ERR_SHAPE;
        // the fused head keeps one key per strip in the workspace
        if (strcmp(name, "gemv_nvfp4_w_argmax") == 0 && strips > HEAD_WORDS) return CROW_ERR_SHAPE;
        const uint32_t wmax = (uint32_t)e->max_waves / (uint32_t)e->nr;  // waves per tensor in a block
        // A wave walks its run of groups with four of them (9 KB) in flight; few long walks beat many short ones (every wave
        // pays its start, its staging set-up and the block's meeting in LDS once), as long as the launch still has a few
        // thousand waves.  Measured on MI355X: [17408, 5120] one tensor 3 waves per strip (7 groups each), two tensors 2 + 2
        // (10 groups each); [5120, 17408] (68 groups, only 320 strips) 5 slices of 4 waves, which meet through the workspace.
        // A strip stays inside one block up to 64 groups (K = 16384).
        uint32_t w, s;
        if (groups <= 64) {
            const uint32_t per_wave = e->nr == 2 ? 10 : 7;
            w = (groups + per_wave - 1) / per_wave;
            s = 1;
            // One tensor of up to 512 strips leaves the chip idle between such long walks: four waves there.  Measured with w = 1..8 at
            // 512 to 17408 rows, K = 1024..5120 and 1 to 64 rows of activations (us, one row unless said): [512, 2048] 3.7 -> 3.3,
            // [6151, 3008] 5.9 -> 4.8 (three rows 8.9 -> 7.0), [1024, 5120] 5.4 -> 5.0 (three rows 10.1 -> 8.6), 64 rows 52.5 -> 47.2 at
            // [4096, 5120].  Eight would win again up to four rows (4.3) and lose from sixteen on (60 against 47); at 1088 strips and 8
            // groups four waves lose (one row 8.1 against 7.1, five 13.6 against 12.3; see also CROW_TWO_RUNS below).  Up to seven groups a wave walks the strip
            // alone, here and in the grouped expert kernels.  The routed kernels keep the long walks: their launch is that many strips
            // per combo or tile, which fills the chip (gemv_fp4_ptrb [4096, 2048] x 512 combos 250 us, 332 with four waves, x 32 21 / 26;
            // moe_down_grouped [2048, 2560] x 64 tiles 52 / 61).
            // (The split depends on the tensor's shape only, never on the number of tokens or experts in the launch: a token's
            // bits are the same in every batch, and the grouped expert kernels reproduce the per-combo ones'.  Four waves per tensor at
            // batch 1 would take routed gate|up [1024, 2048] x 8 experts from 8.0 to 7.2 us and give that up.)
            // bf16 activations cost a wave less, so from 17 groups on three waves keep the chip as busy beyond 256 strips ([8192, 5376]
            // three rows 6.9 us, 7.3 with four waves, one row 6.2 / 6.4; [6144, 4608] three rows 6.2 / 6.4).
            const bool long_bf16 = strstr(name, "_bf16") != nullptr && groups > 16 && strips > 256;
            if (e->nr == 1 && !routed && !long_bf16 && strips <= 512 && groups > 7 && w < 4) w = 4;
        } else {
            w = 4;
            s = (groups + 13) / 14;
        }
        if (force_s > 0) s = force_s;
        if (force_w > 0) w = force_w;
        if (w > wmax) w = wmax;
        if (s > 255) s = 255;
        if (s * w > groups) {  // never more units than groups
            if (w > groups) w = groups;
            s = groups / w;
        }
        const uint32_t gz = routed ? z : (tokens ? (z + 3) / 4 : 1);
        const uint32_t hint = from_memory ? 0 : (verify ? z : (tokens ? (z - 1) % 4 + 1 : 0));
        // Two strips per block share the operand reads of several f32 rows; where that leaves compute units without a block, and
        // up to two blocks a unit where a strip is short, one strip per block is faster (three rows, us, two / one strips per block:
        // [2048, 5120] 8.6 / 7.4, [4096, 5120] 8.7 / 8.3, [8192, 2048] 6.0 / 5.5, [6144, 3072] 6.9 / 6.5, [8192, 3072] 7.2 / 6.5; one group more, [6144, 3328] 7.2 / 7.6; [5120, 5120] 8.8 / 10.1,
        // [12288, 3072] 9.2 / 9.6; gate|up [4096, 5120] 13.3 / 11.3, [5120, 2048] 10.8 / 11.1).  Same bits.
        // Four waves on a strip of up to 14 groups walk two to four groups each.  Many token groups fill the chip with such short walks:
        // there two waves take the four runs between them (blocks of more than three per compute unit; us, four waves / two waves with
        // two runs / two waves with a run each, which are other bits: [8192, 2560] x 257 208 / 169 / 170, [4096, 2048] x 257 75 / 66 / 66,
        // [4096, 3072] x 32 16.3 / 14.4 / 14.1; below the line, [2048, 3072] x 32, 9.6 / 13.7 / 13.3).
        const bool two = e->two_stub != nullptr && s == 1 && w == 4 && groups > 7 && groups <= 14 && force_w == 0 && force_s == 0 &&
                         (unsigned long long)((strips + 1) / 2) * gz > 768;
        if (two) w = 2;
        const bool one = e->one_stub != nullptr && s == 1 && (strips <= 256 || (e->nr == 1 && strips <= 512 && groups <= 12));
        const uint32_t ns = one ? 1u : (uint32_t)e->ns, gx = (strips + ns - 1) / ns;
        *out = crow_dims{gx, pairs | (hint << 20) | ((one ? CROW_ONE_STRIP : (two ? CROW_TWO_RUNS : s)) << 24), gz, 64u * w * (uint32_t)e->nr};
        if (s > 1 && ((unsigned long long)gx * gz * s * (unsigned)(e->nr * ns) * 64 > PARTIAL_FLOATS || (unsigned long long)gx * gz > COUNTER_SLOTS)) return CROW_ERR_WORKSPACE;
        return CROW_OK;
    }
    if (strncmp(name, "gemv_nvfp4_w_valu", 17) == 0) {  // a 16-lane group per RG rows, four groups per wave, four waves per block
        if (k_dim == 0 || k_dim % CROW_BLOCK_VALUES != 0) return CROW_ERR_SHAPE;
        const uint32_t per_block = 16u * (uint32_t)(name[17] - '0');
        *out = crow_dims{(rows + per_block - 1) / per_block, 1, 1, 256};
        return CROW_OK;
    }
    if (strncmp(name, "gemm_nvfp4_bf16", 15) == 0) {  // z = M token rows
        if (k_dim == 0 || k_dim % CROW_BLOCK_VALUES != 0) return CROW_ERR_SHAPE;
        const bool m16 = strcmp(name, "gemm_nvfp4_bf16_m16") == 0;
        if (m16 && z > 16) return CROW_ERR_SHAPE;
        if ((m16 || strcmp(name, "gemm_nvfp4_bf16_m32") == 0) && z >= 1 && z <= 48u * 65535u && k_dim < 1u << 25 && (unsigned long long)z * k_dim <= 0xffffffffull) {
            const KSplitPlan p = ksplit_plan(strips, panels, z, force_s, force_w);
            if (p.nj != 0) {
                *out = crow_dims{(strips + p.nj - 1) / p.nj, (z + 16 * p.tbk - 1) / (16 * p.tbk), CROW_KSPLIT | p.slices | (p.nj << 8) | (p.tbk << 12) | (p.waves << 16), 64u * p.waves};
                return CROW_OK;
            }
        }
        if (m16) {  // one panel per wave where the workspace allows it
            uint32_t s = (panels + 3) / 4;
            if (s > 16) s = 16;
            while (s > 1 && ((unsigned long long)rt * s * 16 * 64 > PARTIAL_FLOATS || rt > COUNTER_SLOTS)) s--;
            *out = crow_dims{rt, 1, s, 256};
            return CROW_OK;
        }
        if (name[15] == '_' && name[16] == 'w') {  // gemm_nvfp4_bf16_w<tokens per block>: eight row tiles per block
            const uint32_t mtw = (uint32_t)atoi(name + 17);
            *out = crow_dims{(rt + 7) / 8, (z + mtw - 1) / mtw, 1, 512};
            return CROW_OK;
        }
        if (name[15] == '_' && name[16] == 't') {  // gemm_nvfp4_bf16_t<tokens per block>: four waves of five strips
            const uint32_t mtt = (uint32_t)atoi(name + 17);
            const unsigned long long tiles = (unsigned long long)((strips + 19) / 20) * ((z + mtt - 1) / mtt);
            if (tiles > 0x7FFFFFFFull || k_dim >= 1u << 25) return CROW_ERR_SHAPE;
            *out = crow_dims{(uint32_t)tiles, 1, 1, 256};
            return CROW_OK;
        }
        const uint32_t mt = name[15] == '_' ? (uint32_t)atoi(name + 17) : 128;  // gemm_nvfp4_bf16_m<tokens per block>
        if (mt == 32) {
            *out = crow_dims{rt, (z + 31) / 32, 1, 256};
        } else {
            *out = crow_dims{(rt + 3) / 4, (z + mt - 1) / mt, 1, 256};
        }
        return CROW_OK;
    }
    if (strcmp(name, "repack_nvfp4") == 0 || strcmp(name, "dequant_nvfp4_tiled") == 0) {  // adjacent groups, one per wave
        const uint32_t waves = groups < CROW_LAYOUT_WAVES ? groups : CROW_LAYOUT_WAVES;
        *out = crow_dims{(groups + waves - 1) / waves, strips, 1, 64 * waves};
        return CROW_OK;
    }
    if (strcmp(name, "unpack_nvfp4") == 0) {
        *out = crow_dims{groups, strips, 1, 64};
        return CROW_OK;
    }
    if (strcmp(name, "router_top10") == 0) { *out = crow_dims{z, 1, 1, 64}; return CROW_OK; }
    if (strcmp(name, "moe_group") == 0) { *out = crow_dims{1, 1, 1, 1024}; return CROW_OK; }
    if (strcmp(name, "argmax_k") == 0) { *out = crow_dims{1, 1, 1, 1024}; return CROW_OK; }
    if (strcmp(name, "acc_combo") == 0) { *out = crow_dims{(rows + 255) / 256, z, store ? CROW_TWIN : 1u, 256}; return CROW_OK; }  // rows = hidden
    if (strcmp(name, "silu_mul_combo") == 0 || strcmp(name, "dequant_fp4_flat") == 0) {  // rows = element count
        *out = crow_dims{(rows + 255) / 256, 1, 1, 256};
        return CROW_OK;
    }
    return CROW_ERR_KERNEL_MISSING;
}

int crow_hip_launch_dims(const char* name, uint32_t rows, uint32_t k_dim, uint32_t z, crow_dims* out) {
    return crow_hip_launch_dims_split(name, rows, k_dim, z, 0, 0, out);
}

int crow_hip_status(void) {
    if (!g.ready) return CROW_ERR_NOT_INITIALIZED;
    // every stream idle: a launch on another stream (an explicit one, or a graph's) may be in the middle of a hand-over whose
    // arrival counters are cleared below, or may still be about to raise a status bit
    hipError_t e = hipDeviceSynchronize();
    if (e != hipSuccess) return (int)e;
    unsigned st = 0, st2 = 0;
    if ((e = hipMemcpy(&st, g.ws.status, sizeof st, hipMemcpyDeviceToHost)) != hipSuccess) return (int)e;
    if ((e = hipMemcpy(&st2, g.ws_static.status, sizeof st2, hipMemcpyDeviceToHost)) != hipSuccess) return (int)e;
    if (st == 0 && st2 == 0) return CROW_OK;
    if (st != 0) {
        (void)hipMemset(g.ws.status, 0, sizeof st);
        // a launch that bailed out may have left arrival counters behind
        (void)hipMemset(g.ws.counters, 0, COUNTER_WORDS * sizeof(unsigned));
        for (const crow::Workspace& m : g.ws_more) (void)hipMemset(m.counters, 0, COUNTER_WORDS * sizeof(unsigned));
    }
    if (st2 != 0) (void)hipMemset(g.ws_static.counters, 0, (NOALLOC_COUNTER_SLOTS + NOALLOC_TAIL_WORDS) * sizeof(unsigned));  // counters, status, key
    st |= st2;
    if (st & CROW_STATUS_BAD_SCALE_BYTE) return CROW_ERR_SCALE_BYTE;
    if (st & crow::STATUS_WORKSPACE_TOO_SMALL) return CROW_ERR_WORKSPACE;
    if (st & crow::STATUS_BAD_GEO) return CROW_ERR_GEO;
    return CROW_ERR_SHAPE;
}

int crow_hip_reset_workspace(void) {
    if (!g.ready) return CROW_ERR_NOT_INITIALIZED;
    hipError_t e = hipDeviceSynchronize();
    if (e != hipSuccess) return (int)e;
    // arrival counters and the status word of both scratch areas (the head's keys need no clearing: every launch overwrites
    // the words it reads)
    if ((e = hipMemset(g.ws_static.counters, 0, (NOALLOC_COUNTER_SLOTS + 32) * sizeof(unsigned))) != hipSuccess) return (int)e;
    for (const crow::Workspace& m : g.ws_more)
        if ((e = hipMemset(m.counters, 0, COUNTER_WORDS * sizeof(unsigned))) != hipSuccess) return (int)e;
    return hip_rc(hipMemset(g.ws.counters, 0, COUNTER_WORDS * sizeof(unsigned)));
}

void crow_hip_set_stream(void* stream) { g.stream = (hipStream_t)stream; }
void* crow_hip_cur_stream(void) { return (void*)g.stream; }
int crow_hip_sync(void) { return g.ready ? hip_rc(hipStreamSynchronize(g.stream)) : CROW_ERR_NOT_INITIALIZED; }

int crow_hip_alloc(size_t bytes, void** out) {
    if (!g.ready) return CROW_ERR_NOT_INITIALIZED;
    if (!out || bytes == 0) return CROW_ERR_BAD_ARGUMENT;
    hipError_t e = hipMalloc(out, bytes);
    if (e != hipSuccess) {
        *out = nullptr;
        return (int)e;
    }
    return hip_rc(hipMemset(*out, 0, bytes));
}
int crow_hip_free(void* p) { return p ? hip_rc(hipFree(p)) : CROW_OK; }
int crow_hip_upload(void* dst, const void* src, size_t bytes) {
    if (!g.ready) return CROW_ERR_NOT_INITIALIZED;
    if (!dst || !src) return CROW_ERR_BAD_ARGUMENT;
    hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, g.stream);
    if (e != hipSuccess) return (int)e;
    return g.stream == nullptr ? hip_rc(hipStreamSynchronize(nullptr)) : CROW_OK;
}
int crow_hip_download(void* dst, const void* src, size_t bytes) {
    if (!g.ready) return CROW_ERR_NOT_INITIALIZED;
    if (!dst || !src) return CROW_ERR_BAD_ARGUMENT;
    hipError_t e = hipStreamSynchronize(g.stream);
    if (e != hipSuccess) return (int)e;
    return hip_rc(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
}

int crow_hip_event_create(void** out) {
    if (!out) return CROW_ERR_BAD_ARGUMENT;
    hipEvent_t e;
    hipError_t rc = hipEventCreate(&e);
    *out = rc == hipSuccess ? (void*)e : nullptr;
    return hip_rc(rc);
}
int crow_hip_event_record(void* ev) { return ev ? hip_rc(hipEventRecord((hipEvent_t)ev, g.stream)) : CROW_ERR_BAD_ARGUMENT; }
int crow_hip_event_elapsed_ms(void* start, void* stop, float* ms) {
    if (!start || !stop || !ms) return CROW_ERR_BAD_ARGUMENT;
    hipError_t rc = hipEventSynchronize((hipEvent_t)stop);
    if (rc != hipSuccess) return (int)rc;
    return hip_rc(hipEventElapsedTime(ms, (hipEvent_t)start, (hipEvent_t)stop));
}
int crow_hip_event_destroy(void* ev) { return ev ? hip_rc(hipEventDestroy((hipEvent_t)ev)) : CROW_OK; }

int crow_hip_time_launches(crow_fn_t f, uint32_t gx, uint32_t gy, uint32_t gz, uint32_t bx, const uint64_t* vals, uint32_t n_vals,
                           uint32_t n_sets, uint32_t iters, float* us_per_launch) {
    if (!g.ready) return CROW_ERR_NOT_INITIALIZED;
    const FnEntry* e = entry_of(f);
    if (!e) return CROW_ERR_KERNEL_MISSING;
    if (!vals || !us_per_launch || n_sets == 0 || iters == 0) return CROW_ERR_BAD_ARGUMENT;
    hipEvent_t a, b;
    hipError_t rc;
    if ((rc = hipEventCreate(&a)) != hipSuccess) return (int)rc;
    if ((rc = hipEventCreate(&b)) != hipSuccess) return (int)rc;
    int out = hip_rc(hipEventRecord(a, g.stream));
    for (uint32_t i = 0; i < iters && out == CROW_OK; i++)
        out = launch_on(e, dim3(gx, gy, gz), dim3(bx), vals + (size_t)(i % n_sets) * n_vals, n_vals, g.stream);
    if (out == CROW_OK) out = hip_rc(hipEventRecord(b, g.stream));
    if (out == CROW_OK) out = hip_rc(hipEventSynchronize(b));
    float ms = 0.0f;
    if (out == CROW_OK) out = hip_rc(hipEventElapsedTime(&ms, a, b));
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    *us_per_launch = ms * 1000.0f / (float)iters;
    return out;
}

int crow_hip_time_sequence(uint32_t n_kernels, const crow_fn_t* fns, const crow_dims* dims, const uint32_t* n_vals,
                           const uint64_t* vals, uint32_t n_sets, uint32_t iters, float* us_per_iteration) {
    if (!g.ready) return CROW_ERR_NOT_INITIALIZED;
    if (!fns || !dims || !n_vals || !vals || !us_per_iteration || n_kernels == 0 || n_kernels > 16 || n_sets == 0 || iters == 0)
        return CROW_ERR_BAD_ARGUMENT;
    size_t per_set = 0;
    for (uint32_t k = 0; k < n_kernels; k++) {
        if (!entry_of(fns[k])) return CROW_ERR_KERNEL_MISSING;
        per_set += n_vals[k];
    }
    hipEvent_t a, b;
    hipError_t rc;
    if ((rc = hipEventCreate(&a)) != hipSuccess) return (int)rc;
    if ((rc = hipEventCreate(&b)) != hipSuccess) return (int)rc;
    int out = hip_rc(hipEventRecord(a, g.stream));
    for (uint32_t i = 0; i < iters && out == CROW_OK; i++) {
        const uint64_t* v = vals + (size_t)(i % n_sets) * per_set;
        for (uint32_t k = 0; k < n_kernels && out == CROW_OK; k++) {
            out = launch_on((const FnEntry*)(void*)fns[k], dim3(dims[k].gx, dims[k].gy, dims[k].gz), dim3(dims[k].bx), v, n_vals[k], g.stream);
            v += n_vals[k];
        }
    }
    if (out == CROW_OK) out = hip_rc(hipEventRecord(b, g.stream));
    if (out == CROW_OK) out = hip_rc(hipEventSynchronize(b));
    float ms = 0.0f;
    if (out == CROW_OK) out = hip_rc(hipEventElapsedTime(&ms, a, b));
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    *us_per_iteration = ms * 1000.0f / (float)iters;
    return out;
}

int crow_hip_time_pure_read(const uint64_t* bufs, uint32_t n_bufs, size_t bytes, uint32_t blocks, uint32_t threads, uint32_t pattern, uint32_t iters, float* us_per_launch) {
    if (!g.ready) return CROW_ERR_NOT_INITIALIZED;
    if (!bufs || !us_per_launch || n_bufs == 0 || iters == 0 || blocks == 0 || threads == 0 || threads % 64 != 0 || threads > 1024 || pattern > 2) return CROW_ERR_BAD_ARGUMENT;
    if (bytes == 0 || bytes % CROW_GROUP_BYTES != 0 || bytes / CROW_GROUP_BYTES > 0xFFFFFFFFull) return CROW_ERR_SHAPE;
    unsigned units = (unsigned)(bytes / CROW_GROUP_BYTES);
    unsigned* sink = (unsigned*)(g.scalars + 24);
    hipEvent_t a, b;
    hipError_t rc;
    if ((rc = hipEventCreate(&a)) != hipSuccess) return (int)rc;
    if ((rc = hipEventCreate(&b)) != hipSuccess) return (int)rc;
    int out = hip_rc(hipEventRecord(a, g.stream));
    for (uint32_t i = 0; i < iters && out == CROW_OK; i++) {
        const unsigned char* w = (const unsigned char*)(uintptr_t)bufs[i % n_bufs];
        if (pattern == 0) {
            void* args[3] = {(void*)&w, (void*)&units, (void*)&sink};
            out = hip_rc(hipLaunchKernel((const void*)&pure_read_groups, dim3(blocks), dim3(threads), args, 0, g.stream));
        } else {
            size_t n16 = bytes / 16;
            void* args[3] = {(void*)&w, (void*)&n16, (void*)&sink};
            out = hip_rc(hipLaunchKernel(pattern == 1 ? (const void*)&pure_read_flat_nt : (const void*)&pure_read_flat, dim3(blocks), dim3(threads), args, 0, g.stream));
        }
    }
    if (out == CROW_OK) out = hip_rc(hipEventRecord(b, g.stream));
    if (out == CROW_OK) out = hip_rc(hipEventSynchronize(b));
    float ms = 0.0f;
    if (out == CROW_OK) out = hip_rc(hipEventElapsedTime(&ms, a, b));
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    *us_per_launch = ms * 1000.0f / (float)iters;
    return out;
}

int crow_hip_stream_create(void** out) {
    if (!g.ready) return CROW_ERR_NOT_INITIALIZED;
    if (!out) return CROW_ERR_BAD_ARGUMENT;
    hipStream_t s = nullptr;
    const int rc = hip_rc(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    *out = (void*)s;
    return rc;
}
int crow_hip_stream_destroy(void* stream) {
    if (!stream) return CROW_OK;
    if (g.stream == (hipStream_t)stream) g.stream = nullptr;
    return hip_rc(hipStreamDestroy((hipStream_t)stream));
}
int crow_hip_begin_capture(void* stream) {
    if (!g.ready) return CROW_ERR_NOT_INITIALIZED;
    if (!stream) return CROW_ERR_BAD_ARGUMENT;  // the legacy default stream cannot be captured
    g.stream = (hipStream_t)stream;
    return hip_rc(hipStreamBeginCapture((hipStream_t)stream, hipStreamCaptureModeGlobal));
}
int crow_hip_end_capture_instantiate(void* stream, void** graph_exec_out) {
    if (!g.ready) return CROW_ERR_NOT_INITIALIZED;
    if (!stream || !graph_exec_out) return CROW_ERR_BAD_ARGUMENT;
    hipGraph_t graph = nullptr;
    hipError_t e = hipStreamEndCapture((hipStream_t)stream, &graph);
    if (e != hipSuccess) return (int)e;
    hipGraphExec_t exec = nullptr;
    e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);  // the executable graph is independent of its template
    if (e != hipSuccess) return (int)e;
    *graph_exec_out = (void*)exec;
    return CROW_OK;
}
int crow_hip_launch_graph(void* graph_exec, void* stream) {
    if (!g.ready) return CROW_ERR_NOT_INITIALIZED;
    if (!graph_exec) return CROW_ERR_BAD_ARGUMENT;
    return hip_rc(hipGraphLaunch((hipGraphExec_t)graph_exec, (hipStream_t)stream));
}
int crow_hip_graph_exec_destroy(void* graph_exec) {
    if (!graph_exec) return CROW_OK;
    return hip_rc(hipGraphExecDestroy((hipGraphExec_t)graph_exec));
}
int crow_hip_time_graph(void* graph_exec, void* stream, uint32_t iters, float* us_per_replay) {
    if (!g.ready) return CROW_ERR_NOT_INITIALIZED;
    if (!graph_exec || !us_per_replay || iters == 0) return CROW_ERR_BAD_ARGUMENT;
    hipEvent_t a, b;
    hipError_t rc;
    if ((rc = hipEventCreate(&a)) != hipSuccess) return (int)rc;
    if ((rc = hipEventCreate(&b)) != hipSuccess) return (int)rc;
    int out = hip_rc(hipEventRecord(a, (hipStream_t)stream));
    for (uint32_t i = 0; i < iters && out == CROW_OK; i++) out = hip_rc(hipGraphLaunch((hipGraphExec_t)graph_exec, (hipStream_t)stream));
    if (out == CROW_OK) out = hip_rc(hipEventRecord(b, (hipStream_t)stream));
    if (out == CROW_OK) out = hip_rc(hipEventSynchronize(b));
    float ms = 0.0f;
    if (out == CROW_OK) out = hip_rc(hipEventElapsedTime(&ms, a, b));
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    *us_per_replay = ms * 1000.0f / (float)iters;
    return out;
}

#ifdef CROW_TRACE  // measurement builds only: the per-block timestamps of gemv.h
int crow_hip_trace_read(unsigned long long* dst, size_t words, int clear) {
    hipError_t e = hipDeviceSynchronize();
    if (e != hipSuccess) return (int)e;
    if ((e = hipMemcpyFromSymbol(dst, HIP_SYMBOL(crow::crow_trace), words * 8)) != hipSuccess) return (int)e;
    if (clear) {
        void* p = nullptr;
        if ((e = hipGetSymbolAddress(&p, HIP_SYMBOL(crow::crow_trace))) != hipSuccess) return (int)e;
        return hip_rc(hipMemset(p, 0, sizeof(unsigned long long) * 16384 * 8));
    }
    return CROW_OK;
}
#endif

size_t crow_hip_container_bytes(uint32_t rows, uint32_t cols) { return crow_container_bytes(rows, cols); }
size_t crow_hip_tiled_bytes(uint32_t rows, uint32_t cols) { return crow_tiled_bytes(rows, cols); }
uint32_t crow_hip_tile_code_offset(uint32_t row, uint32_t wp) { return row < 16 && wp < 32 ? crow_group_code_offset(row, wp) : UINT32_MAX; }
uint32_t crow_hip_tile_scale_offset(uint32_t row, uint32_t sb) { return row < 16 && sb < 16 ? crow_group_scale_offset(row, sb) : UINT32_MAX; }

static int layout_launch(const char* name, const void* a, const void* b, const void* c, uint32_t rows, uint32_t cols) {
    if (!g.ready) return CROW_ERR_NOT_INITIALIZED;
    if (!a || !b || rows == 0 || cols == 0 || cols % CROW_BLOCK_VALUES != 0) return a && b ? CROW_ERR_SHAPE : CROW_ERR_BAD_ARGUMENT;
    // the two scalars ride in a small ring of device words so that back-to-back calls do not race; a kernel writes them (a copy
    // from the stack would have to be waited for)
    static std::atomic<unsigned> slot{0};
    const unsigned turn = slot.fetch_add(1) & 7u;
    int* sc = g.scalars + 2 * turn;
    int r = (int)rows, c2 = (int)cols;
    void* a0[3] = {(void*)&sc, (void*)&r, (void*)&c2};
    hipError_t e = hipLaunchKernel((const void*)&layout_words, dim3(1), dim3(1), a0, 0, g.stream);
    if (e != hipSuccess) return (int)e;
    crow_dims d;
    int rc = crow_hip_launch_dims(name, rows, cols, 1, &d);
    if (rc != CROW_OK) return rc;
    uint64_t vals[5];
    uint32_t n = 0;
    vals[n++] = (uint64_t)a;
    vals[n++] = (uint64_t)b;
    if (c) vals[n++] = (uint64_t)c;
    vals[n++] = (uint64_t)sc;
    vals[n++] = (uint64_t)(sc + 1);
    rc = launch_on(find(name), dim3(d.gx, d.gy, d.gz), dim3(d.bx), vals, n, g.stream);
    if (rc != CROW_OK) return rc;
    // A kernel puts both status words into pinned memory (two copies to pageable memory take longer); what they say when one is
    // raised is crow_hip_status's to report.  It must run when every stream is idle, as crow_hip_status reads them: behind a wait for the
    // device - but while all launches so far went to the null stream, it is behind all of them where it stands, and one wait does
    // (a small layout call 18 us, 27 with two waits).
    const bool elsewhere = g_other_streams.load();
    if (elsewhere && (e = hipDeviceSynchronize()) != hipSuccess) return (int)e;
    unsigned* said = g.said + 2 * turn;
    void* a1[3] = {(void*)&g.ws.status, (void*)&g.ws_static.status, (void*)&said};
    if ((e = hipLaunchKernel((const void*)&status_words, dim3(1), dim3(1), a1, 0, g.stream)) != hipSuccess) return (int)e;
    if ((e = elsewhere ? hipStreamSynchronize(g.stream) : hipDeviceSynchronize()) != hipSuccess) return (int)e;
    return (said[0] | said[1]) == 0 ? CROW_OK : crow_hip_status();
}

int crow_hip_quantize_nvfp4(const float* values_dev, size_t n_values, void* blocks_dev, float* global_scale_dev) {
    if (!g.ready) return CROW_ERR_NOT_INITIALIZED;
    if (!values_dev || !blocks_dev || !global_scale_dev) return CROW_ERR_BAD_ARGUMENT;
    if (n_values == 0 || n_values % CROW_BLOCK_VALUES != 0) return CROW_ERR_SHAPE;
    // the tensor's largest raw scale meets in one device word (one of the library's own, taken in turn so that calls in a
    // row do not share it)
    static std::atomic<unsigned> slot{0};
    unsigned* max_bits = (unsigned*)(g.scalars + 16 + (slot.fetch_add(1) & 7u));
    hipError_t e;
    void* a0[1] = {(void*)&max_bits};
    if ((e = hipLaunchKernel((const void*)&quantize_nvfp4_clear, dim3(1), dim3(1), a0, 0, g.stream)) != hipSuccess) return (int)e;
    unsigned long long n_sub = n_values / 16;
    const unsigned long long want = (n_sub + 255) / 256;
    const unsigned blocks1 = (unsigned)(want < 2048 ? want : 2048);
    const float* vals = values_dev;
    unsigned char* out = (unsigned char*)blocks_dev;
    const unsigned* max_ro = max_bits;
    void* a1[3] = {(void*)&vals, (void*)&n_sub, (void*)&max_bits};
    if ((e = hipLaunchKernel((const void*)&quantize_nvfp4_amax, dim3(blocks1), dim3(256), a1, 0, g.stream)) != hipSuccess) return (int)e;
    if (want > 0x7FFFFFFFull) return CROW_ERR_SHAPE;
    void* a2[5] = {(void*)&vals, (void*)&n_sub, (void*)&max_ro, (void*)&out, (void*)&global_scale_dev};
    return hip_rc(hipLaunchKernel((const void*)&quantize_nvfp4_encode, dim3((unsigned)want), dim3(256), a2, 0, g.stream));
}

int crow_hip_repack_nvfp4(const void* src_dev, uint32_t rows, uint32_t cols, void* dst_dev) {
    return layout_launch("repack_nvfp4", src_dev, dst_dev, nullptr, rows, cols);
}
int crow_hip_unpack_nvfp4(const void* src_dev, uint32_t rows, uint32_t cols, void* dst_dev) {
    return layout_launch("unpack_nvfp4", src_dev, dst_dev, nullptr, rows, cols);
}
int crow_hip_dequant_tiled(const void* w_dev, const float* gs_dev, uint32_t rows, uint32_t cols, float* out_dev) {
    return layout_launch("dequant_nvfp4_tiled", w_dev, gs_dev, out_dev, rows, cols);
}

}  // extern "C"
