// NVFP4 x bf16 batched GEMM on the gfx950 matrix cores: Y[M][N] = X[M][K] W[N][K]^T, M > 4 token rows.
//
// The reference's prefill projection (engine/src/gen.rs:3922-3924 -> gemm_fp4_dense, engine/src/kernels.rs:
// 533-751) quantises the activations to FP4 and runs Blackwell block-scaled MMA; its structural twin
// glm5_gemm_fp4_tc (engine/src/kernels_glm5_moe.cu:349-449) decodes the weights losslessly to 16-bit
// tiles and runs a plain tensor-core MMA with f32 accumulation and gs in the epilogue.  This kernel
// is the CDNA4 form of the latter: weights decode to EXACT bf16 (e2m1 * ue4m3 has at most 6
// significant bits), X is bf16, products are exact in f32, v_mfma_f32_16x16x32_bf16 accumulates.
//
// Data flow (of the shared-X bodies; the K-split, tall and eight-wave ones, which the launcher mostly starts, say below what they do otherwise).
// A wave owns a 64-row weight tile - four 16-row strips of the layout - per 256-column panel and MT = 16 * TBK token
// rows.  Per panel:
//   * the wave loads the panel's group of each of its four strips (4 x 2304 bytes) straight into registers; every code
//     dword is the B operand of one "unit" (16 weight rows x 32 columns, layout.h) as it stands;
//   * X[m0 .. m0 + MT][panel] is staged in LDS (row stride 528 B) and read back as A operands, 16 token rows x
//     32 columns per 16-byte-per-lane read, each used for the four row groups of the tile;
//   * per unit a lane turns its 8 codes into 8 bf16 values times the sub-block scale (cvt to f32, multiply,
//     keep the high 16 bits: exact) and feeds TBK matrix instructions.
// The weight rows ride on the N side and the tokens on the M side, so a lane's 4 results of an instruction are
// 4 tokens of one weight row and a store instruction writes four 64-byte runs of Y.
#pragma once
#include "gemv.h"

namespace crow {

#define CROW_GEMM_XS_STRIDE 264  // bf16 elements per staged X row (256 + 8 of padding)

// 8 codes (one word) times a sub-block scale -> 8 exact bf16 values, as an MFMA operand
__device__ __forceinline__ bf16x8 decode8_scaled(unsigned codes, float scale) {
    const f32x2 a = fp4x2_to_f32<0>(codes), b = fp4x2_to_f32<1>(codes), c = fp4x2_to_f32<2>(codes), d = fp4x2_to_f32<3>(codes);
    u32x4 r;
    // byte selector 0x07060302: high halves of (hi, lo) -> {lo[31:16], hi[31:16]}
    r.x = __builtin_amdgcn_perm(__float_as_uint(a.y * scale), __float_as_uint(a.x * scale), 0x07060302u);
    r.y = __builtin_amdgcn_perm(__float_as_uint(b.y * scale), __float_as_uint(b.x * scale), 0x07060302u);
    r.z = __builtin_amdgcn_perm(__float_as_uint(c.y * scale), __float_as_uint(c.x * scale), 0x07060302u);
    r.w = __builtin_amdgcn_perm(__float_as_uint(d.y * scale), __float_as_uint(d.x * scale), 0x07060302u);
    return __builtin_bit_cast(bf16x8, r);
}

#define CROW_TILE_ROWS 64    // four strips
#define CROW_PANEL_COLS 256  // one group per strip
// the registers of one panel of a 64-row tile: per strip J one scale dword and two code quadwords
struct PanelRegs {
    unsigned sc[4];
    uint4 cd[4][2];
};
// `w` = the tensor, `strips` / `groups` its strip and group counts; strips beyond the tensor re-read the last one (their rows
// are never stored)
__device__ __forceinline__ void load_panel(const unsigned char* w, int rt, int strips, int groups, int p, int lane, PanelRegs& r) {
#pragma unroll
    for (int J = 0; J < 4; J++) {
        const int strip = 4 * rt + J < strips ? 4 * rt + J : strips - 1;
        const unsigned char* g = w + ((size_t)strip * groups + p) * CROW_GROUP_BYTES;
        r.sc[J] = stream_load_u32((const unsigned*)g + lane);
        r.cd[J][0] = stream_load((const uint4*)(g + CROW_GROUP_SCALE_BYTES) + lane);
        r.cd[J][1] = stream_load((const uint4*)(g + CROW_GROUP_SCALE_BYTES + 1024) + lane);
    }
}

// The panel's scale bytes as the GEMM needs them.  A lane (g, n) holds, for each strip, the scales of segment g & 1 of every
// pair, sub-block half g >> 1 (layout.h); the other segment's are in the neighbouring 16-lane group.  After the exchange `even`
// holds the word of the even group of each 32-lane half in both groups, `odd` that of the odd one.
struct TileScales {
    unsigned even[4], odd[4];
    __device__ __forceinline__ void set(const unsigned (&sc)[4]) {
#pragma unroll
        for (int J = 0; J < 4; J++) {
            const u32x2 sw = __builtin_amdgcn_permlane16_swap(sc[J], sc[J], false, false);
            even[J] = sw.x;
            odd[J] = sw.y;
        }
    }
    // scale of this lane's operand of unit (strip J, segment S of the panel): pair S / 2, segment S % 2
    template <int S, int J>
    __device__ __forceinline__ float get() const {
        return e4m3_to_f32<(S >> 1)>((S & 1) ? odd[J] : even[J]);
    }
};

// one 32-column segment S of the panel: four units, TBK token blocks each
template <int TBK, int S>
__device__ __forceinline__ void gemm_segment(const PanelRegs& r, const TileScales& ts, const __bf16* xs_lane, f32x4 (&acc)[TBK][4]) {
    bf16x8 A[TBK];
#pragma unroll
    for (int tb = 0; tb < TBK; tb++) A[tb] = *(const bf16x8*)(xs_lane + tb * 16 * CROW_GEMM_XS_STRIDE + S * 32);
#define CROW_GEMM_UNIT(J)                                                                                      \
    {                                                                                                          \
        const bf16x8 B = decode8_scaled(u4_get(r.cd[J][S >> 2], S & 3), ts.get<S, J>());                       \
        _Pragma("unroll") for (int tb = 0; tb < TBK; tb++)                                                     \
            acc[tb][J] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[tb], B, acc[tb][J], 0, 0, 0);               \
    }
    CROW_GEMM_UNIT(0) CROW_GEMM_UNIT(1) CROW_GEMM_UNIT(2) CROW_GEMM_UNIT(3)
#undef CROW_GEMM_UNIT
}

template <int TBK>
__device__ __forceinline__ void gemm_panel(const PanelRegs& r, const __bf16* xs_lane, f32x4 (&acc)[TBK][4]) {
    TileScales ts;
    ts.set(r.sc);
    gemm_segment<TBK, 0>(r, ts, xs_lane, acc);
    gemm_segment<TBK, 1>(r, ts, xs_lane, acc);
    gemm_segment<TBK, 2>(r, ts, xs_lane, acc);
    gemm_segment<TBK, 3>(r, ts, xs_lane, acc);
    gemm_segment<TBK, 4>(r, ts, xs_lane, acc);
    gemm_segment<TBK, 5>(r, ts, xs_lane, acc);
    gemm_segment<TBK, 6>(r, ts, xs_lane, acc);
    gemm_segment<TBK, 7>(r, ts, xs_lane, acc);
}

// acc[tb][j][r] of lane (g, n): token m0 + 16 tb + 4 g + r, weight row 64 rt + 16 j + n
template <int TBK>
__device__ __forceinline__ void gemm_store(const f32x4 (&acc)[TBK][4], float gs, float* __restrict__ y, int rt, int m0, int rows, int m_total,
                                           int lane) {
    const int g = lane >> 4, n = lane & 15;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int col = rt * CROW_TILE_ROWS + 16 * j + n;
        if (col >= rows) continue;
#pragma unroll
        for (int tb = 0; tb < TBK; tb++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m0 + 16 * tb + 4 * g + r;
                if (m < m_total) y[(size_t)m * rows + col] = acc[tb][j][r] * gs;
            }
    }
}

// Token blocks of 16 TBK rows: a block is ONE row tile and one token block (blockIdx.y) whose panels are dealt to
// its W waves (wave w: panels w, w + W, ...; W = 4 as launched: 8 measured slower at M = 16), so that even a small M puts
// every SIMD to work.  Each wave stages
// its own X panel in its own LDS region and reads it back itself: no block barrier in the loop.  The
// four partial tiles are added in wave order through LDS at the end (deterministic).
template <int TBK>
__device__ __forceinline__ void gemm_small_body(const unsigned char* __restrict__ w, const unsigned short* __restrict__ x,
                                                const float* __restrict__ gs_ptr, float* __restrict__ y, int k_dim, int rows,
                                                int m_total, __bf16* xs_all) {
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int rt = (int)blockIdx.x, m0 = 32 * (int)blockIdx.y;
    const int panels = (k_dim + CROW_PANEL_COLS - 1) / CROW_PANEL_COLS;
    if (rt * CROW_TILE_ROWS >= rows || m0 >= m_total) return;  // a grid larger than the problem: the whole block leaves
    const int waves = block_threads() >> 6;  // 16 TBK staged rows per wave
    const int slice = (int)blockIdx.z, slices = (int)gridDim.z;  // the panels may also be dealt over blocks (workspace hand-over)
    __bf16* xs = xs_all + wave * (16 * TBK * CROW_GEMM_XS_STRIDE);
    const __bf16* xs_lane = xs + (lane & 15) * CROW_GEMM_XS_STRIDE + (lane >> 4) * 8;

    f32x4 acc[TBK][4];
#pragma unroll
    for (int tb = 0; tb < TBK; tb++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[tb][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int strips = (rows + CROW_STRIP_ROWS - 1) / CROW_STRIP_ROWS;
    // 16 TBK tokens x 256 columns = 512 TBK chunks of 16 bytes, 8 TBK per lane; wave-private.  Chunk i of this lane: token row
    // 2 i + lane / 32, 8 columns from 8 (lane % 32); its element offset in panel 0 is worked out once (32 bits: checked by
    // the entry points); rows beyond M read row M - 1, whose results are never stored.
    const int xq = (lane & 31) * 8;
    unsigned xoff[8 * TBK];
#pragma unroll
    for (int i = 0; i < 8 * TBK; i++) {
        const int m = m0 + 2 * i + (lane >> 5);
        xoff[i] = (unsigned)(m < m_total ? m : m_total - 1) * (unsigned)k_dim + (unsigned)xq;
    }
    for (int p = slice * waves + wave; p < panels; p += slices * waves) {
        // fetched before the weight loads are issued so that they do not queue behind them
        uint4 xv[8 * TBK];
        const int k0 = p * CROW_PANEL_COLS;
        if (k0 + CROW_PANEL_COLS <= k_dim) {  // uniform
#pragma unroll
            for (int i = 0; i < 8 * TBK; i++) xv[i] = *(const uint4*)(x + (size_t)(xoff[i] + (unsigned)k0));
        } else {  // the last, partial panel: columns beyond K are zeros
#pragma unroll
            for (int i = 0; i < 8 * TBK; i++) {
                xv[i] = make_uint4(0, 0, 0, 0);
                if (k0 + xq < k_dim) xv[i] = *(const uint4*)(x + (size_t)(xoff[i] + (unsigned)k0));
            }
        }
        PanelRegs pr;
        load_panel(w, rt, strips, panels, p, lane, pr);
#pragma unroll
        for (int i = 0; i < 8 * TBK; i++) {
            const int c = i * 64 + lane, r = c >> 5, q = c & 31;
            *(uint4*)(xs + r * CROW_GEMM_XS_STRIDE + q * 8) = xv[i];
        }
        __builtin_amdgcn_wave_barrier();
        gemm_panel<TBK>(pr, xs_lane, acc);
        __builtin_amdgcn_wave_barrier();  // the tile is read before the next stage overwrites it
    }
    // the other waves -> wave 0 through LDS (each wave's own region is free now), added in wave order
    float* red = (float*)xs;
    if (wave > 0) {
#pragma unroll
        for (int tb = 0; tb < TBK; tb++)
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) red[((tb * 4 + j) * 4 + r) * 64 + lane] = acc[tb][j][r];
    }
    __syncthreads();
    if (wave > 0) return;
    for (int ww = 1; ww < waves; ww++) {
        const float* q = (const float*)(xs_all + ww * (16 * TBK * CROW_GEMM_XS_STRIDE));
#pragma unroll
        for (int tb = 0; tb < TBK; tb++)
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[tb][j][r] += q[((tb * 4 + j) * 4 + r) * 64 + lane];
    }
    if (slices > 1) {  // slices of the row tile -> the block that arrives last, in slice order (the GEMV's protocol)
        float v[16 * TBK];
#pragma unroll
        for (int tb = 0; tb < TBK; tb++)
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) v[(tb * 4 + j) * 4 + r] = acc[tb][j][r];
        if (!slice_hand_over<16 * TBK>(v, (unsigned)blockIdx.y * gridDim.x + blockIdx.x, slice, slices, g_ws, lane)) return;
#pragma unroll
        for (int tb = 0; tb < TBK; tb++)
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[tb][j][r] = v[(tb * 4 + j) * 4 + r];
    }
    gemm_store<TBK>(acc, gs_ptr[0], y, rt, m0, rows, m_total, lane);
}

// Shared X: block = 4 waves; wave w owns row tile 4 * blockIdx.x + w and all of the block's MT = 16 * TBK token rows, staged
// once in LDS for the four row tiles.  The memory traffic of panel p + 1 is in flight while panel p is computed: the next
// weight tile waits in a second register set and the next X tile in registers, written to the OTHER LDS buffer after the
// compute, so one block barrier per panel (these kernels run one or two waves per SIMD: nothing else hides the latency).
template <int TBK>
__device__ __forceinline__ void gemm_pipe_body(const unsigned char* __restrict__ w, const unsigned short* __restrict__ x,
                                               const float* __restrict__ gs_ptr, float* __restrict__ y, int k_dim, int rows, int m_total,
                                               __bf16* xs2) {
    constexpr int MT = 16 * TBK;
    constexpr int XCH = MT * 32 / 256;  // 16-byte chunks of an X tile per thread
    constexpr int XBUF = MT * CROW_GEMM_XS_STRIDE;
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int row_tiles = (rows + CROW_TILE_ROWS - 1) / CROW_TILE_ROWS;
    const int rt = (int)blockIdx.x * 4 + wave;
    const bool has_rows = rt < row_tiles;  // wave-uniform; idle waves still stage X and join the barriers
    const int m0 = (int)blockIdx.y * MT;
    const int panels = (k_dim + CROW_PANEL_COLS - 1) / CROW_PANEL_COLS;

    f32x4 acc[TBK][4];
#pragma unroll
    for (int tb = 0; tb < TBK; tb++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[tb][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int strips = (rows + CROW_STRIP_ROWS - 1) / CROW_STRIP_ROWS;
    auto load_w = [&](int p, PanelRegs& r) { load_panel(w, has_rows ? rt : 0, strips, panels, p, lane, r); };
    // chunk c = i * 256 + thread: token row c / 32, 8 columns from 8 (c % 32).  The element offset of the chunk in panel 0 is
    // worked out once; rows beyond M read row M - 1 (their results are never stored), so whole panels load without masks.
    const int xq = ((int)threadIdx.x & 31) * 8;
    unsigned xoff[XCH];
#pragma unroll
    for (int i = 0; i < XCH; i++) {
        const int m = m0 + ((i * 256 + (int)threadIdx.x) >> 5);
        xoff[i] = (unsigned)(m < m_total ? m : m_total - 1) * (unsigned)k_dim + (unsigned)xq;
    }
    auto load_x = [&](int p, uint4 (&xv)[XCH]) {
        const int k0 = p * CROW_PANEL_COLS;
        if (k0 + CROW_PANEL_COLS <= k_dim) {  // uniform
#pragma unroll
            for (int i = 0; i < XCH; i++) xv[i] = *(const uint4*)(x + (size_t)(xoff[i] + (unsigned)k0));
        } else {  // the last, partial panel: columns beyond K are zeros (they meet zero weights, but must not be NaN)
#pragma unroll
            for (int i = 0; i < XCH; i++) {
                xv[i] = make_uint4(0, 0, 0, 0);
                if (k0 + xq < k_dim) xv[i] = *(const uint4*)(x + (size_t)(xoff[i] + (unsigned)k0));
            }
        }
    };
    auto store_x = [&](__bf16* xs, const uint4 (&xv)[XCH]) {
#pragma unroll
        for (int i = 0; i < XCH; i++) {
            const int c = i * 256 + (int)threadIdx.x, r = c >> 5, q = c & 31;
            *(uint4*)(xs + r * CROW_GEMM_XS_STRIDE + q * 8) = xv[i];
        }
    };
    const int lane_off = (lane & 15) * CROW_GEMM_XS_STRIDE + (lane >> 4) * 8;

    PanelRegs pr[2];
    uint4 xv[XCH];
    load_x(0, xv);
    load_w(0, pr[0]);
    store_x(xs2, xv);
    __syncthreads();
    // two panels per trip so that the register sets swap roles without copies
    for (int p = 0; p < panels; p += 2) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int pp = p + h;
            if (pp < panels) {
                const bool more = pp + 1 < panels;
                if (more) {
                    load_x(pp + 1, xv);
                    load_w(pp + 1, pr[h ^ 1]);
                }
                gemm_panel<TBK>(pr[h], xs2 + h * XBUF + lane_off, acc);
                if (more) store_x(xs2 + (h ^ 1) * XBUF, xv);
                __syncthreads();  // the other buffer is written, and this one read, by every wave
            }
        }
    }
    if (!has_rows) return;
    gemm_store<TBK>(acc, gs_ptr[0], y, rt, m0, rows, m_total, lane);
}

// Tall-tile body: a block is FOUR waves, one per SIMD, wave w owning NJ adjacent strips (16 NJ weight rows) and all of the
// block's MT = 16 TBK token rows, so that one decoded operand feeds TBK matrix instructions and the decode (17 vector
// instructions a unit) fits under them.  With one wave per SIMD nothing else hides a latency, so the wave's own stream does.
// It runs unit by unit - unit u = NJ S + J is segment S of strip J - and is written out in the order in which it is to be
// issued (sched_barrier keeps it so): a matrix instruction occupies the matrix pipe for as long as two to three vector
// instructions take to issue, and a wave that issues its matrix instructions back to back waits for each of them in turn.
//   * behind each matrix instruction of unit u stand two vector instructions of the decode of unit u + 1;
//   * the activation operands of segment S + 1 are read from LDS during segment S, across panels too;
//   * the codes of a half panel (segments 0..3 / 4..7) are requested again, for the next panel, as soon as that half has been
//     decoded: half a panel of matrix work covers the round trip with a single register set;
//   * the next X tile travels through registers, one 16-byte chunk requested per unit and one written per unit to the other LDS
//     buffer, and the panel's only barrier stands before segment 7, whose operands are in registers by then.
// Measured ([17408, 5120] x 512 tokens / [5120, 17408] x 1999, TBK = 8): 81 to 90 us / 281 to 308 us by the session against 107 to 111 /
// 342 to 354 for the eight-wave body at 80 tokens, 1.0 to 1.13 / 1.16 to 1.27 PFLOP/s; a library bf16 product of the first shape takes
// 100 us, and 8192^3 runs at 1.31 to 1.41.  A panel takes 8250 cycles at 1.9 to 2.0 GHz where its matrix instructions alone take 5280; without the decode 7000, without
// the matrix instructions 5000, with all activations zero the same cycles at 2.2 GHz: what remains is the two kinds of
// instruction that only partly overlap, and the power of the matrix cores.
// blockIdx.x counts tiles in an order that keeps the tiles of one compute die (blockIdx.x % 8) together: four row blocks by
// as many token blocks as fall to the die, so that its L2 serves both operands.
struct alignas(16) ZeroChunk {
    unsigned words[4];
};
static_assert(alignof(ZeroChunk) >= alignof(u32x4), "load_x reads it as one vector");
__device__ const ZeroChunk gemm_zeros = {{0u, 0u, 0u, 0u}};
typedef float f32x4_dword __attribute__((ext_vector_type(4), aligned(4)));  // rows of Y start at any dword
template <int TBK, int NJ>
struct TallTile {
    static constexpr int MT = 16 * TBK;
    static constexpr int XCH = MT * 32 / 256;  // 16-byte chunks of an X tile per thread
    static constexpr int XBUF = MT * CROW_GEMM_XS_STRIDE;
    static constexpr int UNITS = 8 * NJ, STORE0 = 7 * NJ - XCH;  // the first unit that writes a chunk of the next X tile
    static_assert(MT * 32 % 256 == 0 && STORE0 > XCH / 2, "whole chunks per thread, requested well before they are written");
    unsigned sc[NJ], even[NJ], odd[NJ];
    uint4 cd[2][NJ];
    uint4 xv[XCH];
    bf16x8 A[2][TBK];
    u32x4 B[2];
    f32x4 acc[TBK][NJ];
    const unsigned char* wp[NJ];
    unsigned xrow, xlast, kd;  // element offsets, from the block's first token row, of this thread's first row of X and of the last
                               // row; the row stride.  A block's rows fit 32 bits (K < 2^25), all of X need not.
    const unsigned short* x;   // the block's first token row
    const __bf16 *cur, *nxt;  // this lane's view of the X tile that is being multiplied / of the next one
    __bf16* put;              // this thread's first chunk of the next X tile
    f32x2 pair;               // the decode under way: two values, their scale, the first product
    float scale, low;
    const unsigned short* from;  // this lane's X, its column in the next panel and a mask for its row offsets
    unsigned at_k, inside;
    int lane;

    __device__ __forceinline__ void load_scale(int J, int p) { sc[J] = *((const unsigned*)(wp[J] + (size_t)p * CROW_GROUP_BYTES) + lane); }
    __device__ __forceinline__ void load_codes(int H, int J, int p) {
        cd[H][J] = *((const uint4*)(wp[J] + (size_t)p * CROW_GROUP_BYTES + CROW_GROUP_SCALE_BYTES + 1024 * H) + lane);
    }
    // both segments' scale words of every pair, as in TileScales
    __device__ __forceinline__ void set_scales() {
#pragma unroll
        for (int J = 0; J < NJ; J++) {
            const u32x2 sw = __builtin_amdgcn_permlane16_swap(sc[J], sc[J], false, false);
            even[J] = sw.x;
            odd[J] = sw.y;
        }
    }
    // columns beyond K (the last, partial panel) meet zero weights, but must not be NaN: their lanes read a word of zeros
    // (an address, not a branch: the panel stays one block of code, and the accumulators stay where they are)
    __device__ __forceinline__ void load_x(int i) { 
        const unsigned row = xrow + (unsigned)(8 * i) * kd;  // rows beyond M read row M - 1 (never stored)
        const u32x4 v = *(const __attribute__((address_space(1))) u32x4*)(from + (size_t)(((row < xlast ? row : xlast) & inside) + at_k));
        xv[i] = make_uint4(v.x, v.y, v.z, v.w);
    }
    __device__ __forceinline__ void store_x(int i) { *(uint4*)(put + i * 8 * CROW_GEMM_XS_STRIDE) = xv[i]; }
    // one of the eight steps of unit U's decode: a pair's conversion and first product / its second product and packing
    template <int U, int STEP>
    __device__ __forceinline__ void decode() {
        constexpr int S = U / NJ, J = U % NJ, Q = STEP / 2;
        const unsigned codes = u4_get(cd[S >> 2][J], S & 3);
        if constexpr (STEP == 0) scale = e4m3_to_f32<(S >> 1)>((S & 1) ? odd[J] : even[J]);
        if constexpr (STEP % 2 == 0) {
            pair = fp4x2_to_f32<Q>(codes);
            low = pair.x * scale;
        } else {
            B[U & 1][Q] = __builtin_amdgcn_perm(__float_as_uint(pair.y * scale), __float_as_uint(low), 0x07060302u);
        }
    }
    template <int U, int T>
    __device__ __forceinline__ void unit_steps() {
        if constexpr (T < TBK) {
            constexpr int J = U % NJ, S = U / NJ;
            acc[T][J] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, B[U & 1]), A[S & 1][T], acc[T][J], 0, 0, 0);
            constexpr int N = (U + 1) % UNITS;
            constexpr int D0 = T * 8 / TBK, D1 = (T + 1) * 8 / TBK;  // decode steps behind this matrix instruction
            if constexpr (D0 < D1) decode<N, D0>();
            if constexpr (D0 + 1 < D1) decode<N, D0 + 1>();
            static_assert(D1 - D0 <= 2, "at least four token blocks");
            __builtin_amdgcn_sched_barrier(0);
            unit_steps<U, T + 1>();
        }
    }
    template <int U>
    __device__ __forceinline__ void units(int pn) {
        if constexpr (U < UNITS) {
            constexpr int S = U / NJ, J = U % NJ;
            if constexpr (U == 7 * NJ) __syncthreads();  // the next X tile is written by every wave, this one's last operands are in registers
            // memory work of this unit: operands of segment S + 1, a chunk of the next X tile, the codes whose registers are free
#pragma unroll
            for (int tb = J * TBK / NJ; tb < (J + 1) * TBK / NJ; tb++)
                A[(S + 1) & 1][tb] = *(const bf16x8*)((S == 7 ? nxt : cur) + tb * 16 * CROW_GEMM_XS_STRIDE + ((S + 1) & 7) * 32);
            if constexpr (U < XCH) load_x(U);
            if constexpr (U >= STORE0 && U < 7 * NJ) store_x(U - STORE0);
            if constexpr (S == 4) load_scale(J, pn);
            if constexpr (S == 4) load_codes(0, J, pn);
            if constexpr (U == UNITS - 1) set_scales();
            __builtin_amdgcn_sched_barrier(0);
            unit_steps<U, 0>();
            units<U + 1>(pn);
        }
    }

    __device__ __forceinline__ void run(const unsigned char* __restrict__ w, const unsigned short* __restrict__ x_, const float* __restrict__ gs_ptr,
                                        float* __restrict__ y, int k_dim, int rows, int m_total, __bf16* xs2) {
        lane = lane_id();
        const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        const int strips = (rows + CROW_STRIP_ROWS - 1) / CROW_STRIP_ROWS;
        const int panels = (k_dim + CROW_PANEL_COLS - 1) / CROW_PANEL_COLS;
        const int row_blocks = (strips + 4 * NJ - 1) / (4 * NJ), token_blocks = (m_total + MT - 1) / MT;
        // tile of this block: runs of consecutive tile numbers per compute die, numbers counting four row blocks first
        const int blocks = (int)gridDim.x, die = (int)blockIdx.x & 7, at = (int)blockIdx.x >> 3;
        const int t = die * (blocks >> 3) + (die < (blocks & 7) ? die : (blocks & 7)) + at;
        if (t >= row_blocks * token_blocks) return;  // a grid larger than the problem: the whole block leaves
        const int band = t / (4 * token_blocks), in_band = t - band * 4 * token_blocks;
        const int band_rows = row_blocks - 4 * band < 4 ? row_blocks - 4 * band : 4;
        const int rb = 4 * band + in_band % band_rows, m0 = in_band / band_rows * MT;
        const int strip0 = (rb * 4 + wave) * NJ;  // strips beyond the tensor re-read the last one (their rows are never stored)
#pragma unroll
        for (int J = 0; J < NJ; J++) wp[J] = w + (size_t)(strip0 + J < strips ? strip0 + J : strips - 1) * panels * CROW_GROUP_BYTES;
#pragma unroll
        for (int tb = 0; tb < TBK; tb++)
#pragma unroll
            for (int j = 0; j < NJ; j++) acc[tb][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        // chunk c = i * 256 + thread: token row c / 32, 8 columns from 8 (c % 32)
        const int xq = ((int)threadIdx.x & 31) * 8;
        kd = (unsigned)k_dim;
        x = x_ + (size_t)m0 * k_dim;
        xlast = (unsigned)(m_total - m0 < MT ? m_total - m0 - 1 : MT - 1) * kd;
        xrow = (threadIdx.x >> 5) * kd;
        auto next_panel = [&](int p, int buf) {  // the X tile that load_x and store_x move
            const int k = p * CROW_PANEL_COLS + xq;
            from = k < k_dim ? x : (const unsigned short*)gemm_zeros.words;
            inside = k < k_dim ? ~0u : 0u;
            at_k = k < k_dim ? (unsigned)k : 0u;
            put = xs2 + buf * XBUF + ((int)threadIdx.x >> 5) * CROW_GEMM_XS_STRIDE + xq;
        };
        const int lane_off = (lane & 15) * CROW_GEMM_XS_STRIDE + (lane >> 4) * 8;
        next_panel(0, 0);
#pragma unroll
        for (int i = 0; i < XCH; i++) load_x(i);
#pragma unroll
        for (int J = 0; J < NJ; J++) {
            load_scale(J, 0);
            load_codes(0, J, 0);
        }
#pragma unroll
        for (int i = 0; i < XCH; i++) store_x(i);
        __syncthreads();
#pragma unroll
        for (int tb = 0; tb < TBK; tb++) A[0][tb] = *(const bf16x8*)(xs2 + lane_off + tb * 16 * CROW_GEMM_XS_STRIDE);
        set_scales();
        decode<0, 0>(), decode<0, 1>(), decode<0, 2>(), decode<0, 3>(), decode<0, 4>(), decode<0, 5>(), decode<0, 6>(), decode<0, 7>();
        int h = 0;
        for (int p = 0; p < panels; p++) {
            const int pn = p + 1 < panels ? p + 1 : p;  // behind the last panel: requested once more, never used
            cur = xs2 + h * XBUF + lane_off;
            h ^= 1;
            nxt = xs2 + h * XBUF + lane_off;
            next_panel(pn, h);
#pragma unroll
            for (int J = 0; J < NJ; J++) load_codes(1, J, p);
            units<0>(pn);
        }
        // acc[tb][j][r] of lane (g, n): weight row 16 (strip0 + j) + 4 g + r, token m0 + 16 tb + n (the weights ride on the M side, so
        // that a lane holds four neighbours of one row of Y: one store instruction instead of four)
        const float gs = gs_ptr[0];
        const int g = lane >> 4, n = lane & 15;
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int col = (strip0 + j) * CROW_STRIP_ROWS + 4 * g;
#pragma unroll
            for (int tb = 0; tb < TBK; tb++) {
                const int m = m0 + 16 * tb + n;
                const f32x4 v = acc[tb][j] * gs;
                if (m >= m_total) continue;
                float* to = y + (size_t)m * rows + col;
                if (col + 3 < rows) {
                    *(f32x4_dword*)to = v;
                } else {
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (col + r < rows) to[r] = v[r];
                }
            }
        }
    }
};


// Eight-wave body: the tall tile's stream of units with TWO waves per SIMD (256 registers each): wave w owns NJ = 4 adjacent strips (a 64-row
// tile; 512 rows a block) and all of the block's MT = 16 TBK token rows.  A lone wave issues a vector instruction every 8 cycles,
// two waves one every 4, so that a matrix instruction with two of them behind it takes 17 cycles, where the tall tile's takes 22; the price
// is a decode that serves fewer tokens and half the registers, and a block twice as large.  What differs from the tall tile:
//   * one set of activation operands: behind the last unit of a segment each one's register takes the next segment's as soon as it is
//     free (eight matrix instructions of two waves cover an LDS read);
//   * so the panel's barrier stands before its last unit.
// Measured (us, the compiler's own order of the same instructions before): w96 [8192, 5120] x 1536 122 -> 112, w80 [17408, 5120] x 512 107 -> 95,
// w64 [17408, 5120] x 512 180 -> 157, w48 [4096, 4096] x 1000 62 -> 56; with NJ = 3 and 128 tokens 98 / 300 where the tall tile takes 97 / 309
// ([17408, 5120] x 512 / [5120, 17408] x 1999): not kept.
template <int TBK>
struct EightWaveTile {
    static constexpr int NW = 8, NJ = 4;
    static constexpr int MT = 16 * TBK;
    static constexpr int XCH = MT * 32 / (64 * NW);  // 16-byte chunks of an X tile per thread, XROWS token rows apart
    static constexpr int XROWS = 2 * NW;
    static constexpr int XBUF = MT * CROW_GEMM_XS_STRIDE;
    static constexpr int UNITS = 8 * NJ, STORE0 = UNITS - 1 - XCH;  // the first unit that writes a chunk of the next X tile
    static_assert(MT * 32 % (64 * NW) == 0 && STORE0 > 2 * XCH, "whole chunks per thread, requested well before they are written");
    unsigned sc[NJ], even[NJ], odd[NJ];
    uint4 cd[2][NJ];
    uint4 xv[XCH];
    bf16x8 A[TBK];
    u32x4 B[2];
    f32x4 acc[TBK][NJ];
    const unsigned char* wp[NJ];
    unsigned xrow, xlast, kd;  // as in TallTile
    const unsigned short* x;
    const __bf16 *cur, *nxt;
    __bf16* put;
    f32x2 pair;
    float scale, low;
    const unsigned short* from;
    unsigned at_k, inside;
    int lane;

    __device__ __forceinline__ void load_scale(int J, int p) { sc[J] = *((const unsigned*)(wp[J] + (size_t)p * CROW_GROUP_BYTES) + lane); }
    __device__ __forceinline__ void load_codes(int H, int J, int p) {
        cd[H][J] = *((const uint4*)(wp[J] + (size_t)p * CROW_GROUP_BYTES + CROW_GROUP_SCALE_BYTES + 1024 * H) + lane);
    }
    __device__ __forceinline__ void set_scales() {
#pragma unroll
        for (int J = 0; J < NJ; J++) {
            const u32x2 sw = __builtin_amdgcn_permlane16_swap(sc[J], sc[J], false, false);
            even[J] = sw.x;
            odd[J] = sw.y;
        }
    }
    __device__ __forceinline__ void load_x(int i) {
        const unsigned row = xrow + (unsigned)(XROWS * i) * kd;  // rows beyond M read row M - 1 (never stored)
        const u32x4 v = *(const __attribute__((address_space(1))) u32x4*)(from + (size_t)(((row < xlast ? row : xlast) & inside) + at_k));
        xv[i] = make_uint4(v.x, v.y, v.z, v.w);
    }
    __device__ __forceinline__ void store_x(int i) { *(uint4*)(put + i * XROWS * CROW_GEMM_XS_STRIDE) = xv[i]; }
    template <int U, int D, int D1>
    __device__ __forceinline__ void decode() {  // steps D .. D1 - 1 of unit U's eight (TallTile::decode)
        if constexpr (D < D1) {
            constexpr int S = U / NJ, J = U % NJ, Q = D / 2;
            const unsigned codes = u4_get(cd[S >> 2][J], S & 3);
            if constexpr (D == 0) scale = e4m3_to_f32<(S >> 1)>((S & 1) ? odd[J] : even[J]);
            if constexpr (D % 2 == 0) {
                pair = fp4x2_to_f32<Q>(codes);
                low = pair.x * scale;
            } else {
                B[U & 1][Q] = __builtin_amdgcn_perm(__float_as_uint(pair.y * scale), __float_as_uint(low), 0x07060302u);
            }
            decode<U, D + 1, D1>();
        }
    }
    template <int U, int T>
    __device__ __forceinline__ void unit_steps() {
        if constexpr (T < TBK) {
            constexpr int J = U % NJ, S = U / NJ;
            acc[T][J] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, B[U & 1]), A[T], acc[T][J], 0, 0, 0);
            decode<(U + 1) % UNITS, T * 8 / TBK, (T + 1) * 8 / TBK>();
            if constexpr (J == NJ - 1) A[T] = *(const bf16x8*)((S == 7 ? nxt : cur) + T * 16 * CROW_GEMM_XS_STRIDE + ((S + 1) & 7) * 32);
            __builtin_amdgcn_sched_barrier(0);
            unit_steps<U, T + 1>();
        }
    }
    template <int U>
    __device__ __forceinline__ void units(int pn) {
        if constexpr (U < UNITS) {
            constexpr int S = U / NJ, J = U % NJ;
            if constexpr (U == UNITS - 1) __syncthreads();  // the next X tile is written by every wave; nobody reads this one's any more
            if constexpr (U < XCH) load_x(U);
            if constexpr (U >= STORE0 && U < UNITS - 1) store_x(U - STORE0);
            if constexpr (S == 4) load_scale(J, pn);
            if constexpr (S == 4) load_codes(0, J, pn);
            if constexpr (U == UNITS - 1) set_scales();
            __builtin_amdgcn_sched_barrier(0);
            unit_steps<U, 0>();
            units<U + 1>(pn);
        }
    }

    // grid (ceil(row tiles / 8), ceil(M / MT))
    __device__ __forceinline__ void run(const unsigned char* __restrict__ w, const unsigned short* __restrict__ x_, const float* __restrict__ gs_ptr,
                                        float* __restrict__ y, int k_dim, int rows, int m_total, __bf16* xs2) {
        lane = lane_id();
        const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        const int strips = (rows + CROW_STRIP_ROWS - 1) / CROW_STRIP_ROWS;
        const int panels = (k_dim + CROW_PANEL_COLS - 1) / CROW_PANEL_COLS;
        const int strip0 = ((int)blockIdx.x * NW + wave) * NJ, m0 = (int)blockIdx.y * MT;
        if ((int)blockIdx.x * NW * NJ >= strips || m0 >= m_total) return;  // a grid larger than the problem: the whole block leaves
#pragma unroll
        for (int J = 0; J < NJ; J++)  // strips beyond the tensor re-read the last one (their rows are never stored)
            wp[J] = w + (size_t)(strip0 + J < strips ? strip0 + J : strips - 1) * panels * CROW_GROUP_BYTES;
#pragma unroll
        for (int tb = 0; tb < TBK; tb++)
#pragma unroll
            for (int j = 0; j < NJ; j++) acc[tb][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        // chunk c = i * 512 + thread: token row c / 32, 8 columns from 8 (c % 32)
        const int xq = ((int)threadIdx.x & 31) * 8;
        kd = (unsigned)k_dim;
        x = x_ + (size_t)m0 * k_dim;
        xlast = (unsigned)(m_total - m0 < MT ? m_total - m0 - 1 : MT - 1) * kd;
        xrow = (threadIdx.x >> 5) * kd;
        auto next_panel = [&](int p, int buf) {  // the X tile that load_x and store_x move
            const int k = p * CROW_PANEL_COLS + xq;
            from = k < k_dim ? x : (const unsigned short*)gemm_zeros.words;
            inside = k < k_dim ? ~0u : 0u;
            at_k = k < k_dim ? (unsigned)k : 0u;
            put = xs2 + buf * XBUF + ((int)threadIdx.x >> 5) * CROW_GEMM_XS_STRIDE + xq;
        };
        const int lane_off = (lane & 15) * CROW_GEMM_XS_STRIDE + (lane >> 4) * 8;
        next_panel(0, 0);
#pragma unroll
        for (int i = 0; i < XCH; i++) load_x(i);
#pragma unroll
        for (int J = 0; J < NJ; J++) {
            load_scale(J, 0);
            load_codes(0, J, 0);
        }
#pragma unroll
        for (int i = 0; i < XCH; i++) store_x(i);
        __syncthreads();
#pragma unroll
        for (int tb = 0; tb < TBK; tb++) A[tb] = *(const bf16x8*)(xs2 + lane_off + tb * 16 * CROW_GEMM_XS_STRIDE);
        set_scales();
        decode<0, 0, 8>();
        int h = 0;
        for (int p = 0; p < panels; p++) {
            const int pn = p + 1 < panels ? p + 1 : p;  // behind the last panel: requested once more, never used
            cur = xs2 + h * XBUF + lane_off;
            h ^= 1;
            nxt = xs2 + h * XBUF + lane_off;
            next_panel(pn, h);
#pragma unroll
            for (int J = 0; J < NJ; J++) load_codes(1, J, p);
            units<0>(pn);
        }
        // acc[tb][j][r] of lane (g, n): weight row 16 (strip0 + j) + 4 g + r, token m0 + 16 tb + n (as in TallTile)
        const float gs = gs_ptr[0];
        const int g = lane >> 4, n = lane & 15;
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int col = (strip0 + j) * CROW_STRIP_ROWS + 4 * g;
#pragma unroll
            for (int tb = 0; tb < TBK; tb++) {
                const int m = m0 + 16 * tb + n;
                const f32x4 v = acc[tb][j] * gs;
                if (m >= m_total) continue;
                float* to = y + (size_t)m * rows + col;
                if (col + 3 < rows) {
                    *(f32x4_dword*)to = v;
                } else {
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (col + r < rows) to[r] = v[r];
                }
            }
        }
    }
};

// K-split body: up to 64 token rows, and as many as there are where a tensor of few strips leaves the larger tiles' blocks fewer than compute units.  A block is NJ adjacent strips and ONE token block
// of MT = 16 TBK rows; its W waves divide the 256-column panels among themselves (and, if a tensor has too few strips for the
// device, the S blocks of the grid's third dimension as well), each wave in runs of whole panels, and add their tiles through
// LDS (slices: in slice order through the workspace).  Nothing is shared before that, so there is no barrier in the loop.
//   * A decoded operand serves TBK matrix instructions only, and decoding it takes 17 vector instructions, so the instructions issued are a
//     bound beside the memory: 5.6 us of them for [17408, 5120] at 16 tokens if every SIMD always finds one.  A wave that has a SIMD to
//     itself issues a vector instruction every 8 cycles, two waves one every 4: eight to twelve waves per compute unit, in one round of blocks.
//   * The activations are read by every block: 160 KB at 16 tokens and K = 5120, as much as the block's weights with NJ = 4.  More strips per
//     block is less of that, and a chunk's operand reads from LDS serve all NJ strips.
//   * vmcnt counts in order: what a wave waits for includes all it requested before.  Per panel the activations of the next one are
//     requested first and its weights last, so that a wait for a chunk of activations never includes a load from memory that
//     was requested less than a panel ago.
// Measured ([17408, 5120], us; m16 / m32 before): 16 tokens 14.5 to 15.4 (18.5), 32 18.0 (24.7), 48 21.9 (35.0), 64 24.7 (36.8);
// [4096, 4096]: 16 tokens 6.3 (8.8), 64 10.8 (14.4); [1024, 8192] x 64 9.9 (22.8); [5120, 17408] x 128 38.6 (67.8), x 256 62.6 (103); [1024, 5120] x 256 11.6 (16.2).
template <int TBK, int NJ>
struct KSplitTile {
    static constexpr int MT = 16 * TBK;
    static constexpr int SEGS = TBK == 1 ? 8 : (TBK == 2 ? 4 : 2);  // 32-column segments per staged chunk of X: 32 registers of it at most
    static constexpr int XCH = TBK * SEGS;                         // 16-byte pieces of a chunk per lane
    static constexpr int PPR = SEGS * 4;                           // pieces per token row
    static constexpr int STRIDE = SEGS * 64 + 16;                  // bytes per staged row: eight rows 16 bytes apart modulo the bank cycle
    // LDS per wave: a chunk, and afterwards one token block's sums
    static constexpr int AREA = MT * STRIDE > NJ * 1024 ? MT * STRIDE : NJ * 1024;
    unsigned sc[NJ], even[NJ], odd[NJ];
    u32x4 cd[NJ][2];
    u32x4 xv[XCH];
    // One token block: a panel's sums start from zero and are added behind its last instruction (four additions per strip and panel),
    // which keeps the error of the long walks of few waves below that of one panel per wave over many slices ([17408, 5120] x 16
    // against 64 bits: 6.9e-8; 9.0e-8 with one running sum; m16 7.4e-8).  More token blocks: m32's four walks are longer than these.
    static constexpr bool BY_PANEL = TBK == 1;
    f32x4 acc[TBK][NJ], total[BY_PANEL ? NJ : 1];
    const unsigned char* wp[NJ];  // the wave's first group of each strip
    unsigned rowoff[XCH];         // element offsets of this lane's rows of X, from the block's first token row (K < 2^25: 32 bits do)
    const unsigned short* x;      // the block's first token row
    int k_dim, lane, xq, count;
    lds_p stage;

    // panel p of the wave's run; behind the last one every lane asks for the same word of the first, never used (an address and not a
    // branch, so that the loads in flight are the same on every path)
    __device__ __forceinline__ void load_w(int p) {
        const size_t at = p < count ? (size_t)p * CROW_GROUP_BYTES : 0;
        const int l = p < count ? lane : 0;
#pragma unroll
        for (int J = 0; J < NJ; J++) {
            const unsigned char* q = wp[J] + at;
            sc[J] = stream_load_u32((const unsigned*)q + l);
            cd[J][0] = stream_load_v((const uint4*)(q + CROW_GROUP_SCALE_BYTES) + l);
            cd[J][1] = stream_load_v((const uint4*)(q + CROW_GROUP_SCALE_BYTES + 1024) + l);
        }
    }
    // chunk c of panel p of the tensor; columns beyond K meet zero weights, but must not be NaN: their lanes read a word of zeros
    __device__ __forceinline__ void load_x(int p, int c) {
        const int col = p * CROW_PANEL_COLS + c * SEGS * 32 + xq;
        const bool in = col < k_dim;
        const unsigned short* from = in ? x : (const unsigned short*)gemm_zeros.words;
        const unsigned mask = in ? ~0u : 0u, at = in ? (unsigned)col : 0u;
#pragma unroll
        for (int i = 0; i < XCH; i++) xv[i] = *(const __attribute__((address_space(1))) u32x4*)(from + (size_t)((rowoff[i] & mask) + at));
    }
    __device__ __forceinline__ void store_x() {
#pragma unroll
        for (int i = 0; i < XCH; i++) {
            const int c = i * 64 + lane, r = c / PPR, q = c % PPR;
            *(__attribute__((address_space(3))) u32x4*)(stage + r * STRIDE + q * 16) = xv[i];
        }
        __builtin_amdgcn_wave_barrier();  // (the wave's LDS accesses execute in order: this only keeps the compiler from reordering them)
    }
    template <int S>
    __device__ __forceinline__ void segments(int p) {
        if constexpr (S < 8) {
            if constexpr (S % SEGS == 0) {
                store_x();
                if constexpr (S + SEGS < 8) load_x(p, S / SEGS + 1);
                else load_x(p + 1, 0);
            }
            typedef __attribute__((address_space(3))) const u32x4* lds_v4;
            const lds_p at = stage + (lane & 15) * STRIDE + (lane >> 4) * 16 + (S % SEGS) * 64;
            bf16x8 A[TBK];
#pragma unroll
            for (int tb = 0; tb < TBK; tb++) A[tb] = __builtin_bit_cast(bf16x8, *(lds_v4)(at + tb * 16 * STRIDE));
#pragma unroll
            for (int J = 0; J < NJ; J++) {
                const u32x4 q = cd[J][S >> 2];
                const unsigned codes = (S & 3) == 0 ? q.x : ((S & 3) == 1 ? q.y : ((S & 3) == 2 ? q.z : q.w));
                const bf16x8 B = decode8_scaled(codes, e4m3_to_f32<(S >> 1)>((S & 1) ? odd[J] : even[J]));
#pragma unroll
                for (int tb = 0; tb < TBK; tb++) acc[tb][J] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(B, A[tb], acc[tb][J], 0, 0, 0);
            }
            if constexpr (S % SEGS == SEGS - 1) __builtin_amdgcn_wave_barrier();  // the chunk is read before the next one overwrites it
            segments<S + 1>(p);
        }
    }

    __device__ __forceinline__ void run(const unsigned char* __restrict__ w, const unsigned short* __restrict__ x_, const float* __restrict__ gs_ptr,
                                        float* __restrict__ y, int k_dim_, int rows, int m_total, lds_p lds, const Workspace& ws) {
        lane = lane_id();
        k_dim = k_dim_;
        const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), waves = block_threads() >> 6;
        const int strips = (rows + CROW_STRIP_ROWS - 1) / CROW_STRIP_ROWS, panels = (k_dim + CROW_PANEL_COLS - 1) / CROW_PANEL_COLS;
        const int strip0 = (int)blockIdx.x * NJ, m0 = (int)blockIdx.y * MT;
        if (strip0 >= strips || m0 >= m_total) return;  // a grid larger than the problem: the whole block leaves
        // the panels in runs of floor(panels / units), the first ones one longer
        const int slice = (int)blockIdx.z, slices = (int)gridDim.z, units = slices * waves, unit = slice * waves + wave;
        const int base = panels / units, rem = panels - base * units, first = unit * base + (unit < rem ? unit : rem);
        count = base + (unit < rem ? 1 : 0);
        stage = lds + wave * AREA;
#pragma unroll
        for (int J = 0; J < NJ; J++)  // strips beyond the tensor re-read the last one (their rows are never stored)
            wp[J] = w + ((size_t)(strip0 + J < strips ? strip0 + J : strips - 1) * panels + first) * CROW_GROUP_BYTES;
        const int mlast = m_total - m0 - 1;  // rows beyond M read row M - 1 (never stored)
#pragma unroll
        for (int i = 0; i < XCH; i++) {
            const int r = (i * 64 + lane) / PPR;
            rowoff[i] = (unsigned)(r < mlast ? r : mlast) * (unsigned)k_dim;
        }
        xq = (lane % PPR) * 8;
        x = x_ + (size_t)m0 * k_dim;
#pragma unroll
        for (int tb = 0; tb < TBK; tb++)
#pragma unroll
            for (int j = 0; j < NJ; j++) acc[tb][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < (BY_PANEL ? NJ : 1); j++) total[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (count > 0) {  // wave-uniform
            load_x(first, 0);
            load_w(0);
            for (int p = 0; p < count; p++) {
#pragma unroll
                for (int J = 0; J < NJ; J++) {  // both segments' scale words of every pair, as in TileScales
                    const u32x2 sw = __builtin_amdgcn_permlane16_swap(sc[J], sc[J], false, false);
                    even[J] = sw.x;
                    odd[J] = sw.y;
                }
                segments<0>(first + p);
                __builtin_amdgcn_sched_barrier(0);
                load_w(p + 1);
                if constexpr (BY_PANEL) {
#pragma unroll
                    for (int j = 0; j < NJ; j++) {
                        total[j] += acc[0][j];
                        acc[0][j] = f32x4{0.f, 0.f, 0.f, 0.f};
                    }
                }
            }
        }
        if constexpr (BY_PANEL) {
#pragma unroll
            for (int j = 0; j < NJ; j++) acc[0][j] = total[j];
        }
        // the waves' tiles, one token block of 16 rows at a time: wave j < NJ adds strip j's, by fours (in pairs), the fours in order
        typedef __attribute__((address_space(3))) f32x4* lds_f4;
        f32x4 v[TBK];
#pragma unroll
        for (int tb = 0; tb < TBK; tb++) {
            if (tb > 0) __syncthreads();
#pragma unroll
            for (int j = 0; j < NJ; j++) *(lds_f4)(stage + j * 1024 + lane * 16) = acc[tb][j];
            __syncthreads();
            if (wave < NJ) {
                for (int w0 = 0; w0 < waves; w0 += 4) {
                    f32x4 t[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        t[i] = *(lds_f4)(lds + (w0 + i < waves ? w0 + i : 0) * AREA + wave * 1024 + lane * 16);
                        if (w0 + i >= waves) t[i] = f32x4{0.f, 0.f, 0.f, 0.f};
                    }
                    const f32x4 four = (t[0] + t[1]) + (t[2] + t[3]);
                    v[tb] = w0 == 0 ? four : v[tb] + four;
                }
            }
        }
        if (wave >= NJ) return;
        if (slices > 1) {
            float q[4 * TBK];
#pragma unroll
            for (int tb = 0; tb < TBK; tb++)
#pragma unroll
                for (int r = 0; r < 4; r++) q[4 * tb + r] = v[tb][r];
            if (!slice_hand_over<4 * TBK>(q, ((unsigned)blockIdx.y * gridDim.x + blockIdx.x) * NJ + wave, slice, slices, ws, lane)) return;
#pragma unroll
            for (int tb = 0; tb < TBK; tb++)
#pragma unroll
                for (int r = 0; r < 4; r++) v[tb][r] = q[4 * tb + r];
        }
        // v[tb][r] of lane (g, n): weight row 4 g + r of the strip, token m0 + 16 tb + n
        const float gs = gs_ptr[0];
        const int col = (strip0 + wave) * CROW_STRIP_ROWS + 4 * (lane >> 4);
#pragma unroll
        for (int tb = 0; tb < TBK; tb++) {
            const int m = m0 + 16 * tb + (lane & 15);
            if (m >= m_total) continue;
            const f32x4 o = v[tb] * gs;
            float* to = y + (size_t)m * rows + col;
            if (col + 3 < rows) {
                *(f32x4_dword*)to = o;
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (col + r < rows) to[r] = o[r];
            }
        }
    }
};

}  // namespace crow

// Y[M][rows] f32 = X[M][k_dim] bf16 times the tiled NVFP4 tensor, times gs.  The argument list is
// gemm_fp4_dense's (engine/src/kernels.rs:533-541) without the quantised-activation buffer: x is bf16.
// grid (ceil(row_tiles / 4), ceil(M / MT)), block 256, MT = 64 / 128 for the two general entry points.
// token blocks of 32: grid (row_tiles, ceil(M / 32)), block 256 (or fewer whole waves: the waves deal the panels)
extern "C" __global__ void __launch_bounds__(512) gemm_nvfp4_bf16_m32(const unsigned char* __restrict__ w, const unsigned short* __restrict__ x,
                                                                         const float* __restrict__ gs_ptr, float* __restrict__ y,
                                                                         const int* __restrict__ k_dim_p, const int* __restrict__ rows_p,
                                                                         const int* __restrict__ m_p) {
    __shared__ __attribute__((aligned(16))) __bf16 xs[4 * 32 * CROW_GEMM_XS_STRIDE];
    const int m = *m_p;
    // four waves stage and reduce in the static LDS below; X is addressed with 32-bit element offsets
    if (m < 1 || block_threads() > 256 || (unsigned long long)m * (unsigned long long)*k_dim_p > 0xffffffffull) {
        if (threadIdx.x == 0) atomicOr(crow::g_ws.status, crow::STATUS_BAD_SHAPE);
        return;
    }
    if (m <= 16) crow::gemm_small_body<1>(w, x, gs_ptr, y, *k_dim_p, *rows_p, m, xs);  // one 16-token block: half the matrix work and staging
    else crow::gemm_small_body<2>(w, x, gs_ptr, y, *k_dim_p, *rows_p, m, xs);
}
// M <= 16: one 16-token block, its panels dealt over grid.z blocks of 4 waves (one panel per wave at K = 5120): grid (row_tiles, 1, S)
extern "C" __global__ void __launch_bounds__(256) gemm_nvfp4_bf16_m16(const unsigned char* __restrict__ w, const unsigned short* __restrict__ x,
                                                                       const float* __restrict__ gs_ptr, float* __restrict__ y,
                                                                       const int* __restrict__ k_dim_p, const int* __restrict__ rows_p,
                                                                       const int* __restrict__ m_p) {
    __shared__ __attribute__((aligned(16))) __bf16 xs[4 * 16 * CROW_GEMM_XS_STRIDE];
    const int m = *m_p;
    if (m < 1 || m > 16 || block_threads() > 256 || (unsigned long long)m * (unsigned long long)*k_dim_p > 0xffffffffull) {  // uniform over the launch
        if (threadIdx.x == 0) atomicOr(crow::g_ws.status, crow::STATUS_BAD_SHAPE);
        return;
    }
    crow::gemm_small_body<1>(w, x, gs_ptr, y, *k_dim_p, *rows_p, m, xs);
}
// the shared-X body: grid (ceil(row_tiles / 4), ceil(M / MT)), block 256, MT = 16 TBK = 64 / 128 tokens; dynamic LDS = two X tiles
#define CROW_GEMM_PIPE_ENTRY(NAME, TBK, OCC)                                                                                   \
    extern "C" __global__ void __launch_bounds__(256, OCC) NAME(const unsigned char* __restrict__ w, const unsigned short* __restrict__ x, \
                                                           const float* __restrict__ gs_ptr, float* __restrict__ y,            \
                                                           const int* __restrict__ k_dim_p, const int* __restrict__ rows_p,    \
                                                           const int* __restrict__ m_p) {                                      \
        /* 256 threads; X is addressed with 32-bit element offsets */                                                         \
        if (block_threads() != 256 || *m_p < 1 || (unsigned long long)*m_p * (unsigned long long)*k_dim_p > 0xffffffffull) {   \
            if (threadIdx.x == 0) atomicOr(crow::g_ws.status, crow::STATUS_BAD_SHAPE);                                         \
            return;                                                                                                            \
        }                                                                                                                      \
        crow::gemm_pipe_body<TBK>(w, x, gs_ptr, y, *k_dim_p, *rows_p, *m_p, (__bf16*)crow_dyn_lds);                            \
    }
CROW_GEMM_PIPE_ENTRY(gemm_nvfp4_bf16_m48, 3, 2)
CROW_GEMM_PIPE_ENTRY(gemm_nvfp4_bf16_m64, 4, 2)
CROW_GEMM_PIPE_ENTRY(gemm_nvfp4_bf16_m96, 6, 1)
CROW_GEMM_PIPE_ENTRY(gemm_nvfp4_bf16, 8, 1)
// the eight-wave body: grid (ceil(row_tiles / 8), ceil(M / MT)), block 512, MT = 16 TBK tokens; dynamic LDS = two X tiles
#define CROW_GEMM_WIDE_ENTRY(NAME, TBK)                                                                                        \
    extern "C" __global__ void __launch_bounds__(512, 2) NAME(const unsigned char* __restrict__ w, const unsigned short* __restrict__ x, \
                                                         const float* __restrict__ gs_ptr, float* __restrict__ y,              \
                                                         const int* __restrict__ k_dim_p, const int* __restrict__ rows_p,      \
                                                         const int* __restrict__ m_p) {                                        \
        /* 512 threads; X is addressed with 32-bit element offsets */                                                         \
        if (block_threads() != 512 || *m_p < 1 || (unsigned long long)*m_p * (unsigned long long)*k_dim_p > 0xffffffffull) {   \
            if (threadIdx.x == 0) atomicOr(crow::g_ws.status, crow::STATUS_BAD_SHAPE);                                         \
            return;                                                                                                            \
        }                                                                                                                      \
        crow::EightWaveTile<TBK> t;                                                                                            \
        t.run(w, x, gs_ptr, y, *k_dim_p, *rows_p, *m_p, (__bf16*)crow_dyn_lds);                                                \
    }
CROW_GEMM_WIDE_ENTRY(gemm_nvfp4_bf16_w48, 3)
CROW_GEMM_WIDE_ENTRY(gemm_nvfp4_bf16_w64, 4)
CROW_GEMM_WIDE_ENTRY(gemm_nvfp4_bf16_w80, 5)
CROW_GEMM_WIDE_ENTRY(gemm_nvfp4_bf16_w96, 6)
// the tall-tile body: grid (ceil(strips / (4 NJ)) * ceil(M / MT)), block 256, MT = 16 TBK tokens; dynamic LDS = two X tiles
#define CROW_GEMM_TALL_ENTRY(NAME, TBK, NJ)                                                                                    \
    extern "C" __global__ void __launch_bounds__(256, 1) NAME(const unsigned char* __restrict__ w, const unsigned short* __restrict__ x, \
                                                         const float* __restrict__ gs_ptr, float* __restrict__ y,              \
                                                         const int* __restrict__ k_dim_p, const int* __restrict__ rows_p,      \
                                                         const int* __restrict__ m_p) {                                        \
        /* 256 threads; a block's rows of X are addressed with 32-bit element offsets */                                      \
        if (block_threads() != 256 || *m_p < 1 || (unsigned)*k_dim_p >= 1u << 25) {                                            \
            if (threadIdx.x == 0) atomicOr(crow::g_ws.status, crow::STATUS_BAD_SHAPE);                                         \
            return;                                                                                                            \
        }                                                                                                                      \
        crow::TallTile<TBK, NJ> t;                                                                                             \
        t.run(w, x, gs_ptr, y, *k_dim_p, *rows_p, *m_p, (__bf16*)crow_dyn_lds);                                                \
    }
CROW_GEMM_TALL_ENTRY(gemm_nvfp4_bf16_t64, 4, 5)
CROW_GEMM_TALL_ENTRY(gemm_nvfp4_bf16_t96, 6, 5)
CROW_GEMM_TALL_ENTRY(gemm_nvfp4_bf16_t128, 8, 5)
// The K-split body, which the launcher starts in the place of gemm_nvfp4_bf16_m16 / _m32 when the launch dimensions say so
// (crow_hip_launch_dims): grid (ceil(strips / NJ), ceil(M / MT), slices), block of W >= NJ waves, MT = 16 TBK tokens; dynamic LDS = AREA
// bytes per wave.  `waves` and the scratch memory come from the launcher.
#define CROW_GEMM_KSPLIT_ENTRY(TBK, NJ, MT, WAVES)                                                                             \
    extern "C" __global__ void __launch_bounds__(64 * WAVES) gemm_ksplit_##MT##x##NJ(                                           \
        const unsigned char* __restrict__ w, const unsigned short* __restrict__ x, const float* __restrict__ gs_ptr,           \
        float* __restrict__ y, const int* __restrict__ k_dim_p, const int* __restrict__ rows_p, const int* __restrict__ m_p, int waves, const Workspace ws) { \
        static_assert(MT == 16 * TBK, "the name says the token rows of a block");                                              \
        if (block_threads() != 64 * waves || waves < 2 || waves < NJ || *m_p < 1 || *m_p > MT * (int)gridDim.y || (unsigned)*k_dim_p >= 1u << 25) { \
            if (threadIdx.x == 0) atomicOr(ws.status, crow::STATUS_BAD_SHAPE);                                                 \
            return;                                                                                                            \
        }                                                                                                                      \
        crow::KSplitTile<TBK, NJ> t;                                                                                           \
        t.run(w, x, gs_ptr, y, *k_dim_p, *rows_p, *m_p, LDS, ws);                                                              \
    }
#define CROW_GEMM_KSPLIT_ALL(E)                                                                    \
    E(1, 1, 16, 12) E(1, 2, 16, 12) E(1, 3, 16, 12) E(1, 4, 16, 12) E(1, 5, 16, 12)                \
    E(2, 1, 32, 12) E(2, 2, 32, 12) E(2, 3, 32, 12) E(2, 4, 32, 12) E(2, 5, 32, 12)                \
    E(3, 1, 48, 12) E(3, 2, 48, 12) E(3, 3, 48, 8) E(3, 4, 48, 8) E(3, 5, 48, 8)                   \
    E(4, 1, 64, 12) E(4, 2, 64, 8) E(4, 3, 64, 8) E(4, 4, 64, 8) E(4, 5, 64, 8)
CROW_GEMM_KSPLIT_ALL(CROW_GEMM_KSPLIT_ENTRY)
