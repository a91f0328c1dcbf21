// Q8_0 x Q8_0 matrix-matrix product on the i8 matrix cores (prefill / batched
// token blocks).
//
// The reference has no prefill: every token runs the matvec of
// fortai_gguf_runtime.f90:424-465, i.e. per row and block the exact int32 dot
// of 32 int8 products, scaled by f32(w_scale) * a_scale and accumulated in
// fp32 (fortai_q8_dot.c:262-284 scalar, :287-331 AVX2).  Here the int32 block
// dot of 32 tokens x 32 rows is one v_mfma_i32_32x32x32_i8 (exact: integer
// arithmetic), and the scale-and-accumulate of every (token, row, block) runs
// on the vector ALUs: acc = fma(f32(w_scale) * x_scale, f32(dot), acc), the
// scalar reference's form.  The AVX2 reference splits each block dot into
// eight 4-product lane partials before the fp32 accumulation, so results
// agree with it to fp32 rounding (relative 1e-5 class), not bit for bit; the
// per-block int32 dots are bit-exact and exported for testing.
//
// Token activations ("X8") come in two layouts of the same size.  Block-major,
// written by q8_quantize_tokens_kernel and read by the entry points:
//   q[(b * ld + t) * 32 + k]   int8 value k of block b of token t
//   s[b * ld + t]              f32 scale (the fp16-rounded reference scale)
// Chunk-major, written and read inside the prompt prefill:
//   q[(c * ld + t) * 128 + l * 16 + j * 4 + k]  int8 value 4 l + k of block 4 c + j of token t
//   s[(c * ld + t) * 4 + j]                     its scale
// with ld = tokens rounded up to 128 and blocks padded to a multiple of 4.  The
// blocks past the width hold zeros.  Rows past the tokens are zeros too as
// q8_quantize_tokens_kernel writes them, and undefined inside the prefill: the
// products read them, but a token's outputs depend on its own row alone and those
// of rows past the tokens are not stored.  The int8 part precedes the scales in one buffer of
// q8_tokens_bytes() bytes.  Chunk-major, a token's chunk (four blocks) is 128
// contiguous bytes, lane part by lane part as the decode layouts have it: one
// 16-byte load gives a lane its part of four blocks, and the lines that a token
// tile's readers share at the same moment lie on different L2 channels
// (block-major they are 32 ld bytes apart: for up to 128 tokens always the
// same two).
//
// Weights stay in the decode layout (q8_kernels.hip): lanes 4h..4h+3 of a
// row's 16-byte pieces hold its bytes 16h..16h+15 of four consecutive blocks,
// so a lane that loads those four pieces holds the B operand of four MFMAs
// with no shuffling.  Both operands present their 16 bytes in natural order,
// so the products pair up whatever k order the instruction uses internally.
#include "fortai_hip_internal.h"
#include "fortai_hip_kernels.h"
#include "mmq_tiles.h"

#include <type_traits>


namespace fortai_hip {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kTokTile = 128;  // tokens per workgroup
constexpr int kRowTile = 128;  // rows per workgroup
constexpr int kRowTiles = 2;   // 32-row MFMA tiles per wave
constexpr int kMmqThreads = 512;

__device__ __forceinline__ v4i as_v4i(uint4 u) {
    v4i r;
    r.x = static_cast<int>(u.x); r.y = static_cast<int>(u.y);
    r.z = static_cast<int>(u.z); r.w = static_cast<int>(u.w);
    return r;
}

__device__ __forceinline__ uint32_t comp(const uint4 &u, int j) {
    return j == 0 ? u.x : (j == 1 ? u.y : (j == 2 ? u.z : u.w));
}

// LDS stage of one chunk (four blocks) of a 128-token x 128-row tile.
// Operand rows are 32 bytes; the two 16-byte halves of row n are stored
// swapped when bit 3 of n is set, so the 16-byte reads of 16 consecutive
// rows fall on distinct banks.
struct MmqStage {
    uint4 a[4][kTokTile][2];   // token bytes per block
    uint4 b[4][kRowTile][2];   // row bytes per block
    float as[4][kTokTile];     // token scales
    float bs[4][kRowTile];     // row scales (f32 of the fp16)
};

__device__ __forceinline__ int half_slot(int n, int h) { return h ^ ((n >> 3) & 1); }

// One workgroup: 128 tokens x 128 rows, eight waves; a wave covers 32 tokens x
// 64 rows (1 x 2 MFMA tiles of 32 x 32: a lane holds 16 tokens' scales, so one
// token tile costs half the LDS scale reads of two).  The scale-and-accumulate
// bounds it (48 vector instructions per MFMA), and 32 accumulators per lane
// leave room for four waves per SIMD.  Chunk c + 1 is loaded into registers
// while chunk c is consumed from LDS, then stored to the other stage (one
// barrier per chunk).  With the quantizer, against four waves of 64 x 64 (two
// per SIMD): 2560 x 9216 over 4096 tokens 486 -> 403 us, 9216 x 2560 over 4096
// 322 -> 307 us, over 1200 121 -> 105 us, 3584 x 1024 over 700 29 -> 21 us.
//   BLOCKS: X8 block-major, else chunk-major
//   EPI 0: out[t * ld_out + row] = acc;  EPI 1: out = acc + resid (same index)
//   DOTS: also write every int32 block dot to dots[(t * rows + row) * blocks + b]
template <int EPI, bool DOTS, bool BLOCKS>
__global__ __launch_bounds__(kMmqThreads, 4) void q8_mmq_kernel(Q8Matrix w, const int8_t *__restrict__ xq,
    const float *__restrict__ xs, int tokens, int ld, float *__restrict__ out, int ld_out,
    const float *__restrict__ resid, int32_t *__restrict__ dots) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    MmqStage *stage = reinterpret_cast<MmqStage *>(lds_raw);
    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & 63, wave = tid >> 6;
    const int i = lane & 31, h = lane >> 5;
    const int t0 = static_cast<int>(blockIdx.y) * kTokTile;
    const int r0 = static_cast<int>(blockIdx.x) * kRowTile;
    const int twl = (wave & 3) * 32;               // wave's first token within the tile
    const int rwl = (wave >> 2) * 32 * kRowTiles;  // wave's first row within the tile
    const int chunks = w.chunks;
    // global sources of this thread's share of a chunk:
    //  tokens: 128 tokens x 8 lane parts (BLOCKS: 4 blocks x 128 tokens x 2 halves) = 1024 pieces, 4 per thread
    //  rows:   16 row groups x 64 lanes          = 1024 pieces, 4 per thread
    //  token scales: 512 floats, 2 per thread;  row scales: 128 x uint2, threads < 128
    const int g_last = w.row_groups - 1;
    constexpr int kPieces = 1024 / kMmqThreads, kScales = 512 / kMmqThreads;
    u32x4_t ra[kPieces], rb[kPieces];  // plain vectors (arrays of the uint4 class stay in scratch)
    float rs[kScales];
    uint2 rws = make_uint2(0u, 0u);
    auto fetch = [&](int c) {
#pragma unroll
        for (int k = 0; k < kPieces; ++k) {
            const int p = tid + k * kMmqThreads;          // 0..1023
            if constexpr (BLOCKS)  // block p / 256, token p / 2 % 128, half p % 2
                ra[k] = *reinterpret_cast<const u32x4_t *>(xq + (static_cast<size_t>(4 * c + (p >> 8)) * ld + t0) * 32 + (p & 255) * 16);
            else
                ra[k] = *reinterpret_cast<const u32x4_t *>(xq + (static_cast<size_t>(c) * ld + t0) * 128 + p * 16);
            const int g = min((r0 >> 3) + (p >> 6), g_last);  // clamped; rows past the end are not stored
            // cached loads: every token tile of the launch re-reads these rows
            rb[k] = reinterpret_cast<const u32x4_t *>(w.quants)[(static_cast<size_t>(g) * chunks + c) * 64 + (p & 63)];
        }
#pragma unroll
        for (int k = 0; k < kScales; ++k) {
            const int p = tid + k * kMmqThreads;  // 0..511: token p / 4, block p % 4 (BLOCKS: block p / 128, token p % 128)
            rs[k] = BLOCKS ? xs[static_cast<size_t>(4 * c + (p >> 7)) * ld + t0 + (p & 127)]
                           : xs[(static_cast<size_t>(c) * ld + t0) * 4 + p];
        }
        if (tid < kRowTile) {
            const int g = min((r0 >> 3) + (tid >> 3), g_last);
            rws = w.scales[(static_cast<size_t>(g) * chunks + c) * 8 + (tid & 7)];
        }
    };
    auto stash = [&](MmqStage &st) {
        // piece p: token or row p / 8, bytes 4l..4l+3 (l = p % 8) of the four blocks
        uint32_t *da = reinterpret_cast<uint32_t *>(&st.a[0][0][0]), *db = reinterpret_cast<uint32_t *>(&st.b[0][0][0]);
#pragma unroll
        for (int k = 0; k < kPieces; ++k) {
            const int p = tid + k * kMmqThreads;
            const int n = p >> 3, l = p & 7;
            const int base = (n * 2 + half_slot(n, l >> 2)) * 4 + (l & 3);
            if constexpr (BLOCKS)
                *reinterpret_cast<u32x4_t *>(&st.a[p >> 8][(p >> 1) & 127][half_slot((p >> 1) & 127, p & 1)]) = ra[k];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if constexpr (!BLOCKS) da[base + j * kTokTile * 8] = ra[k][j];
                db[base + j * kRowTile * 8] = rb[k][j];
            }
        }
#pragma unroll
        for (int k = 0; k < kScales; ++k) {
            const int p = tid + k * kMmqThreads;
            if constexpr (BLOCKS) st.as[p >> 7][p & 127] = rs[k];
            else st.as[p & 3][p >> 2] = rs[k];
        }
        if (tid < kRowTile) {
            st.bs[0][tid] = half_bits_to_float(static_cast<uint16_t>(rws.x & 0xffffu));
            st.bs[1][tid] = half_bits_to_float(static_cast<uint16_t>(rws.x >> 16));
            st.bs[2][tid] = half_bits_to_float(static_cast<uint16_t>(rws.y & 0xffffu));
            st.bs[3][tid] = half_bits_to_float(static_cast<uint16_t>(rws.y >> 16));
        }
    };

    float acc[kRowTiles][16];
#pragma unroll
    for (int f = 0; f < kRowTiles; ++f)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[f][v] = 0.0f;

    fetch(0);
    stash(stage[0]);
    __syncthreads();
    for (int c = 0; c < chunks; ++c) {
        const MmqStage &st = stage[c & 1];
        if (c + 1 < chunks) fetch(c + 1);
        // one block at a time (unrolled, the compiler hoists all 16 MFMAs of
        // the chunk and spills)
#pragma unroll 1
        for (int j = 0; j < 4; ++j) {
            const int t = twl + i;
            const v4i af = as_v4i(st.a[j][t][half_slot(t, h)]);
            // this lane's 16 tokens: twl + 8 (v / 4) + 4 h + v % 4
            float tsc[16];
            const float4 *s4 = reinterpret_cast<const float4 *>(&st.as[j][twl + 4 * h]);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 s = s4[2 * q];
                tsc[4 * q] = s.x; tsc[4 * q + 1] = s.y; tsc[4 * q + 2] = s.z; tsc[4 * q + 3] = s.w;
            }
            v4i bf[kRowTiles];
            float wsc[kRowTiles];
#pragma unroll
            for (int f = 0; f < kRowTiles; ++f) {
                const int row = rwl + 32 * f + i;
                bf[f] = as_v4i(st.b[j][row][half_slot(row, h)]);
                wsc[f] = st.bs[j][row];
            }
#pragma unroll
            for (int f = 0; f < kRowTiles; ++f) {
                const v16i zero = {};
                const v16i d = __builtin_amdgcn_mfma_i32_32x32x32_i8(af, bf[f], zero, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    acc[f][v] = __builtin_fmaf(wsc[f] * tsc[v], static_cast<float>(d[v]), acc[f][v]);
                // keep one MFMA result live at a time (the other waves of the
                // SIMD cover the MFMA latency)
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (DOTS) {
                    const int row = r0 + rwl + 32 * f + i, blk = 4 * c + j;
                    if (row < w.rows && blk < w.blocks) {
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            const int tt = t0 + twl + 8 * (v >> 2) + 4 * h + (v & 3);
                            if (tt < tokens) dots[(static_cast<size_t>(tt) * w.rows + row) * w.blocks + blk] = d[v];
                        }
                    }
                }
            }
        }
        if (c + 1 < chunks) stash(stage[(c + 1) & 1]);
        __syncthreads();
    }
#pragma unroll
    for (int f = 0; f < kRowTiles; ++f) {
        const int row = r0 + rwl + 32 * f + i;
        if (row >= w.rows) continue;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int t = t0 + twl + 8 * (v >> 2) + 4 * h + (v & 3);
            if (t >= tokens) continue;
            const size_t o = static_cast<size_t>(t) * ld_out + row;
            if constexpr (EPI == 1) out[o] = acc[f][v] + resid[o];
            else out[o] = acc[f][v];
        }
    }
}

// The same product for few tokens or few rows, where 128 x 128 tiles leave most
// CUs idle: a wave takes 32 rows x 32 tokens, one MFMA per block, with no LDS
// but the token scales: the four 16-byte pieces that hold lane parts
// 4 h .. 4 h + 3 of row (or chunk-major token) i for four blocks are the
// operands of the chunk's four instructions as they are.  The four waves of a
// workgroup share the tokens.  Operands are loaded two chunks ahead.  With the
// quantizer, 128 x 128 tiles before: 9216 x 2560, 77 tokens 57 -> 21 us;
// 2560 x 9216, 301 tokens 192 -> 63 us; 32 x 2560, 2103 tokens 61 -> 24 us.
template <int EPI, bool BLOCKS>
__global__ __launch_bounds__(256, 2) void q8_mmq_kernel_few(Q8Matrix w, const int8_t *__restrict__ xq,
    const float *__restrict__ xs, int tokens, int ld, float *__restrict__ out, int ld_out,
    const float *__restrict__ resid, int token_tiles) {
    __shared__ __align__(16) float scales[4][4][kFewTokens];  // per wave: a chunk's token scales [block][token]
    const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, wave = tid >> 6;
    const int i = lane & 31, h = lane >> 5;
    // XCD-grouped as q8_mmq_exact_kernel_small's workgroups
    const int id = static_cast<int>(blockIdx.x);
    const bool grouped = w.rows > 7 * kFewRows;  // few_grouped
    const int row_tile = grouped ? id / 8 / token_tiles * 8 + id % 8 : id / token_tiles;
    const int t0 = (grouped ? id / 8 % token_tiles : id % token_tiles) * kFewTokens;
    const int row = row_tile * kFewRows + 32 * wave + i;
    if (row - i >= w.rows) return;  // no row of this wave (no barrier follows)
    const int chunks = w.chunks;
    const int g8 = min(row >> 3, w.row_groups - 1);  // clamped; rows past the end are not stored
    const u32x4_t *wq = reinterpret_cast<const u32x4_t *>(w.quants) + static_cast<size_t>(g8) * chunks * 64 + (row & 7) * 8 + 4 * h;
    const uint2 *ws = w.scales + static_cast<size_t>(g8) * chunks * 8 + (row & 7);
    const u32x4_t *aq = reinterpret_cast<const u32x4_t *>(xq) + (BLOCKS ? static_cast<size_t>(t0 + i) * 2 + h : static_cast<size_t>(t0 + i) * 8 + 4 * h);
    // scale word k of this lane: token lane / 4 + 16 k, block lane % 4 (BLOCKS: block h + 2 k, token i)
    const float *as = BLOCKS ? xs + static_cast<size_t>(h) * ld + t0 + i : xs + static_cast<size_t>(t0) * 4 + lane;
    float *sc = &scales[wave][0][0];
    const int slot = BLOCKS ? lane : (lane & 3) * kFewTokens + (lane >> 2);

    u32x4_t bq[2][4], av[2][4];
    uint2 bs[2];
    float at[2][2];
    auto fetch = [&](int c, int s) {
        const size_t cc = static_cast<size_t>(min(c, chunks - 1));
#pragma unroll
        for (int k = 0; k < 2; ++k) at[s][k] = as[cc * 4 * ld + (BLOCKS ? static_cast<size_t>(2 * k) * ld : 64 * k)];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            av[s][k] = BLOCKS ? aq[(cc * 4 + k) * ld * 2] : aq[cc * ld * 8 + k];
            bq[s][k] = wq[cc * 64 + k];
        }
        bs[s] = ws[cc * 8];
    };
    float acc[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
    auto operand = [](const u32x4_t (&p)[4], int j) {
        return v4i{static_cast<int>(p[0][j]), static_cast<int>(p[1][j]), static_cast<int>(p[2][j]), static_cast<int>(p[3][j])};
    };
    auto consume = [&](int s) {
#pragma unroll
        for (int k = 0; k < 2; ++k) sc[slot + (BLOCKS ? 64 : 16) * k] = at[s][k];
        wave_lds_fence();
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const v4i a = BLOCKS ? v4i{static_cast<int>(av[s][j].x), static_cast<int>(av[s][j].y), static_cast<int>(av[s][j].z),
                static_cast<int>(av[s][j].w)} : operand(av[s], j);
            const v16i zero = {};
            const v16i d = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, operand(bq[s], j), zero, 0, 0, 0);
            const uint32_t sh = j < 2 ? bs[s].x : bs[s].y;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 x = *reinterpret_cast<const float4 *>(sc + j * kFewTokens + 8 * q + 4 * h);
                const float xv[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const float p = j & 1 ? half_times<true>(sh, xv[u]) : half_times<false>(sh, xv[u]);
                    acc[4 * q + u] = __builtin_fmaf(p, static_cast<float>(d[4 * q + u]), acc[4 * q + u]);
                }
            }
        }
        wave_lds_fence();
    };
    fetch(0, 0);
    fetch(1, 1);
    int c = 0;
    for (; c + 2 <= chunks; c += 2) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            __builtin_amdgcn_sched_barrier(0);
            consume(k);
            __builtin_amdgcn_sched_barrier(0);
            fetch(c + k + 2, k);
        }
    }
    if (c < chunks) consume(0);
    if (row >= w.rows) return;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int t = t0 + 8 * (v >> 2) + 4 * h + (v & 3);
        if (t >= tokens) continue;
        const size_t o = static_cast<size_t>(t) * ld_out + row;
        if constexpr (EPI == 1) out[o] = acc[v] + resid[o];
        else out[o] = acc[v];
    }
}

// ------------------------------------------------------------- lane order
// The same product with the reference's AVX2 accumulation kept exactly
// (fortai_q8_dot.c:287-331): per (token, row) eight fp32 lane chains, lane L
// adding fma(f32(w_scale) * x_scale, f32(dot of bytes 4L..4L+3), acc_L) block
// by block, then the horizontal sum ((a0+a4)+(a2+a6))+((a1+a5)+(a3+a7)).  So
// every output is bit-identical to the decode matvec of that token.
//
// The 4-byte lane dots come from v_mfma_f32_16x16x4f16: four independent
// 16x16x4 products per instruction, one per lane part (lane l feeds block
// l / 16 with row or column l % 16; output register r of lane l is block
// r / 4, row 4 (l / 16) + r % 4, column l % 16), so two instructions give the
// eight lane dots of a 16 x 16 quadrant and block.  int8 values are exact in
// fp16, and the products and their 4-term sums (|sum| <= 4 * 128 * 127) are
// exact in the fp32 accumulator, so the dots arrive as exact floats and need
// no conversion.  Per lane dot the 16x16 shape costs the matrix cores what
// the 32x32x4 one does, with half the result registers, which leaves room
// for the next instruction's result while the vector ALUs run the fmas of
// the current one.  The int8 operands are widened to fp16 once, when a chunk
// (four blocks) is staged in LDS: the biased byte b + 128 under the fp16
// exponent of 1024 is 1024 + b + 128 exactly, and one packed fp16
// subtraction of 1152 leaves b.
//
// Staging: per block and token (or row) the eight 4-value lane parts in the
// order 0 4 1 5 2 6 3 7, so that the lane feeding block s reads parts s and
// s + 4 (one per instruction group) as 16 contiguous bytes.
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kXTile = 64;    // tokens and rows per workgroup (4 waves of 32 x 32)
constexpr int kXPitch = 36;   // halves per staged (block, token or row): 32 + 4 pad
constexpr int kXThreads = 256;

struct MmqExactStage {
    _Float16 a[4][kXTile][kXPitch];
    _Float16 b[4][kXTile][kXPitch];
    float as[4][kXTile];
    float bs[4][kXTile];
};

// the staged position of lane part L (order 0 4 1 5 2 6 3 7), in halves
__device__ __forceinline__ int part_slot(int L) { return ((L & 3) * 2 + (L >> 2)) * 4; }

// four signed bytes -> four fp16 values (exact)
__device__ __forceinline__ h4 i8x4_to_h4(uint32_t w) {
    const uint32_t u = w ^ 0x80808080u;  // b + 128
    const uint32_t lo = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u);
    const uint32_t hi = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);
    const h2 bias = {static_cast<_Float16>(1152.0f), static_cast<_Float16>(1152.0f)};
    const h2 a = __builtin_bit_cast(h2, lo) - bias;
    const h2 b = __builtin_bit_cast(h2, hi) - bias;
    return h4{a.x, a.y, b.x, b.y};
}

template <int EPI, bool BLOCKS>
__global__ __launch_bounds__(kXThreads, 2) void q8_mmq_exact_kernel(Q8Matrix w, const int8_t *__restrict__ xq,
    const float *__restrict__ xs, int tokens, int ld, float *__restrict__ out, int ld_out,
    const float *__restrict__ resid) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    MmqExactStage *stage = reinterpret_cast<MmqExactStage *>(lds_raw);
    const int tid = static_cast<int>(threadIdx.x);
    const int lane = tid & 63, wave = tid >> 6;
    const int i = lane & 15, s4 = lane >> 4;  // quadrant row / column, and lane part (block) s4
    const int t0 = static_cast<int>(blockIdx.y) * kXTile;
    const int r0 = static_cast<int>(blockIdx.x) * kXTile;
    const int twl = (wave & 1) * 32;   // wave's first token within the tile
    const int rwl = (wave >> 1) * 32;  // wave's first row within the tile
    const int chunks = w.chunks;
    const int g_last = w.row_groups - 1;

    // this thread's share of a chunk:
    //   tokens: 64 tokens x 8 lane parts        = 512 pieces of 16 bytes, 2 per thread
    //           (BLOCKS: a wave takes one block and half and 64 tokens, lane =
    //           token, so that its LDS stores, rows 18 dwords apart, meet no bank twice)
    //   rows:   8 row groups x 64 lanes         = 512 pieces of 16 bytes, 2 per thread
    //   token scales: 256 floats, 1 per thread; row scales: 64 x uint2, threads < 64
    u32x4_t ra[2], rb[2];
    float rs = 0.0f;
    uint2 rws = make_uint2(0u, 0u);
    auto fetch = [&](int c) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int p = tid + k * kXThreads;  // 0..511
            if constexpr (BLOCKS)
                ra[k] = *reinterpret_cast<const u32x4_t *>(xq + (static_cast<size_t>(4 * c + (p >> 7)) * ld + t0 + (p & 63)) * 32 +
                    ((p >> 6) & 1) * 16);
            else
                ra[k] = *reinterpret_cast<const u32x4_t *>(xq + (static_cast<size_t>(c) * ld + t0) * 128 + p * 16);
            const int g = min((r0 >> 3) + (p >> 6), g_last);  // clamped; rows past the end are not stored
            rb[k] = reinterpret_cast<const u32x4_t *>(w.quants)[(static_cast<size_t>(g) * chunks + c) * 64 + (p & 63)];
        }
        // token tid / 4, block tid % 4 (BLOCKS: block tid / 64, token tid % 64)
        rs = BLOCKS ? xs[static_cast<size_t>(4 * c + (tid >> 6)) * ld + t0 + (tid & 63)]
                    : xs[(static_cast<size_t>(c) * ld + t0) * 4 + tid];
        if (tid < kXTile) {
            const int g = min((r0 >> 3) + (tid >> 3), g_last);
            rws = w.scales[(static_cast<size_t>(g) * chunks + c) * 8 + (tid & 7)];
        }
    };
    auto stash = [&](MmqExactStage &st) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            // piece p: token (below: row) p / 8, lane part p % 8 of the four blocks
            const int p = tid + k * kXThreads;
            const int n = p >> 3, l = p & 7;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if constexpr (BLOCKS)
                    *reinterpret_cast<h4 *>(&st.a[p >> 7][p & 63][part_slot(4 * ((p >> 6) & 1) + j)]) = i8x4_to_h4(ra[k][j]);
                else
                    *reinterpret_cast<h4 *>(&st.a[j][n][part_slot(l)]) = i8x4_to_h4(ra[k][j]);
            }
        }
        // (a loop of its own: with the rows stored between the tokens every store
        // waits for all four loads, 9216 x 2560 x 4096 block-major 1,019 against 1,002 us)
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int p = tid + k * kXThreads;
            const int n = (p >> 6) * 8 + ((p & 63) >> 3), l = p & 7;
#pragma unroll
            for (int j = 0; j < 4; ++j) *reinterpret_cast<h4 *>(&st.b[j][n][part_slot(l)]) = i8x4_to_h4(rb[k][j]);
        }
        if constexpr (BLOCKS) st.as[tid >> 6][tid & 63] = rs;
        else st.as[tid & 3][tid >> 2] = rs;
        if (tid < kXTile) {
            st.bs[0][tid] = half_bits_to_float(static_cast<uint16_t>(rws.x & 0xffffu));
            st.bs[1][tid] = half_bits_to_float(static_cast<uint16_t>(rws.x >> 16));
            st.bs[2][tid] = half_bits_to_float(static_cast<uint16_t>(rws.y & 0xffffu));
            st.bs[3][tid] = half_bits_to_float(static_cast<uint16_t>(rws.y >> 16));
        }
    };

    float acc[8][16];
#pragma unroll
    for (int L = 0; L < 8; ++L)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[L][v] = 0.0f;

    fetch(0);
    stash(stage[0]);
    __syncthreads();
    for (int c = 0; c < chunks; ++c) {
        const MmqExactStage &st = stage[c & 1];
        if (c + 1 < chunks) fetch(c + 1);
#pragma unroll 1
        for (int j = 0; j < 4; ++j) {
            // parts s4 and s4 + 4 of tokens twl + 16 th + i and rows rwl + 16 rh + i
            h4 av[2][2], bv[2][2];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const h4 *ap = reinterpret_cast<const h4 *>(&st.a[j][twl + 16 * q + i][8 * s4]);
                const h4 *bp = reinterpret_cast<const h4 *>(&st.b[j][rwl + 16 * q + i][8 * s4]);
                av[q][0] = ap[0];
                av[q][1] = ap[1];
                bv[q][0] = bp[0];
                bv[q][1] = bp[1];
            }
            // scale products of this lane's outputs: tokens twl + 16 th + 4 s4 + u, rows rwl + 16 rh + i
            float sc[2][2][4];
#pragma unroll
            for (int rh = 0; rh < 2; ++rh) {
                const float wsc = st.bs[j][rwl + 16 * rh + i];
#pragma unroll
                for (int th = 0; th < 2; ++th) {
                    const float4 a4 = *reinterpret_cast<const float4 *>(&st.as[j][twl + 16 * th + 4 * s4]);
                    sc[th][rh][0] = wsc * a4.x;
                    sc[th][rh][1] = wsc * a4.y;
                    sc[th][rh][2] = wsc * a4.z;
                    sc[th][rh][3] = wsc * a4.w;
                }
            }
            // eight instructions (part group g, token half th, row half rh),
            // each issued before the fmas of the previous one
            const f32x16 zero = {};
            f32x16 d = __builtin_amdgcn_mfma_f32_16x16x4f16(av[0][0], bv[0][0], zero, 0, 0, 0);
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                const int g = m >> 2, th = (m >> 1) & 1, rh = m & 1;
                f32x16 dn = zero;
                if (m < 7) {
                    const int g1 = (m + 1) >> 2, th1 = ((m + 1) >> 1) & 1, rh1 = (m + 1) & 1;
                    dn = __builtin_amdgcn_mfma_f32_16x16x4f16(av[th1][g1], bv[rh1][g1], zero, 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    float &a_ = acc[4 * g + (r >> 2)][8 * th + 4 * rh + (r & 3)];
                    a_ = __builtin_fmaf(sc[th][rh][r & 3], d[r], a_);
                }
                __builtin_amdgcn_sched_barrier(0);
                d = dn;
            }
        }
        if (c + 1 < chunks) stash(stage[(c + 1) & 1]);
        __syncthreads();
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        // position v: token half v / 8, row half (v / 4) % 2, token 4 s4 + v % 4 of the half
        const int row = r0 + rwl + 16 * ((v >> 2) & 1) + i;
        const int t = t0 + twl + 16 * (v >> 3) + 4 * s4 + (v & 3);
        if (row >= w.rows || t >= tokens) continue;
        // the horizontal sum of fortai_q8_dot.c:323-330
        const float sum = ((acc[0][v] + acc[4][v]) + (acc[2][v] + acc[6][v])) +
            ((acc[1][v] + acc[5][v]) + (acc[3][v] + acc[7][v]));
        const size_t o = static_cast<size_t>(t) * ld_out + row;
        if constexpr (EPI == 1) out[o] = sum + resid[o];
        else out[o] = sum;
    }
}

// The same product for few tokens or few rows, where 64 x 64 tiles leave most
// CUs idle and a wave's 32 x 32 x 8 chains make each chunk a long serial
// stretch: a wave takes 16 rows, TT x 16 tokens and four of the eight lane
// parts (g = wave & 1: parts 4 g .. 4 g + 3), so a quadrant's chains are spread
// over two waves and a block costs a wave TT matrix instructions.  No LDS
// before the end: the decode layout already holds, for lane (row, part), the
// bytes of four blocks in 16 contiguous bytes, the B operand of four
// instructions, and a token's part is one dword of X8; both are widened in
// registers.  The waves of a workgroup meet once, when wave g = 1 hands its
// chains to wave g = 0 for the horizontal sum.  Operands are loaded
// kSmallAhead chunks ahead (the weights come from HBM).  With the quantizer's
// launch, same bits, 64 x 64 tiles before (chunk-major / block-major tokens):
// 2560 x 9216, 16 tokens 151 -> 29 / 48 us; 1024 x 3584, 77 tokens 63 -> 15 /
// 23 us; 32 x 2560, 4096 tokens 57 -> 22 / 23 us; 9216 x 2560, 33 tokens 46 -> 29 us
// (block-major: the 64 x 64 tiles).
constexpr int kSmallAhead = 4;   // chunks in flight (8: the same, with more registers)

template <int TT, int EPI, bool BLOCKS>
__global__ __launch_bounds__(256, 2) void q8_mmq_exact_kernel_small(Q8Matrix w, const int8_t *__restrict__ xq,
    const float *__restrict__ xs, int tokens, int ld, float *__restrict__ out, int ld_out,
    const float *__restrict__ resid, int token_tiles) {
    __shared__ float hand[2][TT * 16][64];
    __shared__ __align__(16) float scales[4][TT][64];  // per wave: a chunk's token scales [block][token]
    const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, wave = tid >> 6;
    const int g = wave & 1, pair = wave >> 1;
    const int i = lane & 15, s4 = lane >> 4;
    // workgroup b runs on XCD b % 8: with eight row tiles or more, the token
    // tiles of a row tile are consecutive there, so its L2 serves them the
    // weights; fewer row tiles would leave XCDs idle that way
    const int id = static_cast<int>(blockIdx.x);
    const bool grouped = w.rows > 7 * kSmallRows;  // few_grouped
    const int row_tile = grouped ? id / 8 / token_tiles * 8 + id % 8 : id / token_tiles;
    const int t0 = (grouped ? id / 8 % token_tiles : id % token_tiles) * (16 * TT);
    if (row_tile * kSmallRows >= w.rows) return;  // (the grid is padded to whole groups of eight)
    const int row = row_tile * kSmallRows + 16 * pair + i;
    const int chunks = w.chunks;
    const int g8 = min(row >> 3, w.row_groups - 1);  // clamped; rows past the end are not stored
    const u32x4_t *wq = reinterpret_cast<const u32x4_t *>(w.quants) + static_cast<size_t>(g8) * chunks * 64 + (row & 7) * 8 + s4 + 4 * g;
    const uint2 *ws = w.scales + static_cast<size_t>(g8) * chunks * 8 + (row & 7);
    // this lane's token and part; of the scales, token lane / 4 and block
    // lane % 4 (BLOCKS: block s4, token i)
    const uint32_t *aq = reinterpret_cast<const uint32_t *>(xq) + (static_cast<size_t>(t0 + i) * 8 + s4 + 4 * g) * (BLOCKS ? 1 : 4);
    const float *as = BLOCKS ? xs + static_cast<size_t>(s4) * ld + t0 + i : xs + static_cast<size_t>(t0) * 4 + lane;
    const int as_slot = BLOCKS ? lane : 16 * (lane & 3) + (lane >> 2);

    u32x4_t bq[kSmallAhead];
    uint2 bs[kSmallAhead];
    u32x4_t av[kSmallAhead][TT];
    float at[kSmallAhead][TT];
    auto fetch = [&](int c, int slot) {
        const int cc = min(c, chunks - 1);
        const size_t b = static_cast<size_t>(cc) * ld;
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) {
            if constexpr (BLOCKS) {
                at[slot][tt] = as[b * 4 + tt * 16];
#pragma unroll
                for (int j = 0; j < 4; ++j) av[slot][tt][j] = aq[b * 32 + static_cast<size_t>(j) * ld * 8 + tt * 128];
            } else {
                at[slot][tt] = as[b * 4 + tt * 64];
                av[slot][tt] = *reinterpret_cast<const u32x4_t *>(aq + b * 32 + tt * 512);
            }
        }
        bq[slot] = wq[static_cast<size_t>(cc) * 64];
        bs[slot] = ws[static_cast<size_t>(cc) * 8];
    };
    float acc[TT][16];
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[tt][r] = 0.0f;
    auto consume = [&](const u32x4_t &q4, const uint2 &sc, const u32x4_t (&a)[TT], const float (&asc)[TT]) {
        // the wave's own LDS, in order: no barrier
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) scales[wave][tt][as_slot] = asc[tt];
        wave_lds_fence();
        const f32x16 zero = {};
        f32x16 d = __builtin_amdgcn_mfma_f32_16x16x4f16(i8x4_to_h4(a[0][0]), i8x4_to_h4(q4[0]), zero, 0, 0, 0);
#pragma unroll
        for (int m = 0; m < 4 * TT; ++m) {  // block m / TT, token tile m % TT; each product issued before the last one's fmas
            const int j = m / TT, tt = m % TT;
            f32x16 dn = zero;
            if (m + 1 < 4 * TT) {
                const int j1 = (m + 1) / TT, tt1 = (m + 1) % TT;
                dn = __builtin_amdgcn_mfma_f32_16x16x4f16(i8x4_to_h4(a[tt1][j1]), i8x4_to_h4(q4[j1]), zero, 0, 0, 0);
            }
            const uint32_t sh = j < 2 ? sc.x : sc.y;
            const float4 x = *reinterpret_cast<const float4 *>(&scales[wave][tt][16 * j + 4 * s4]);
            // fl(f32(w_scale) * x_scale) of this lane's four tokens
            const float p[4] = {j & 1 ? half_times<true>(sh, x.x) : half_times<false>(sh, x.x),
                j & 1 ? half_times<true>(sh, x.y) : half_times<false>(sh, x.y),
                j & 1 ? half_times<true>(sh, x.z) : half_times<false>(sh, x.z),
                j & 1 ? half_times<true>(sh, x.w) : half_times<false>(sh, x.w)};
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[tt][r] = __builtin_fmaf(p[r & 3], d[r], acc[tt][r]);
            d = dn;
        }
        wave_lds_fence();
    };
#pragma unroll
    for (int k = 0; k < kSmallAhead; ++k) fetch(k, k);
    int c = 0;
    for (; c + kSmallAhead <= chunks; c += kSmallAhead) {
#pragma unroll
        for (int k = 0; k < kSmallAhead; ++k) {
            __builtin_amdgcn_sched_barrier(0);
            consume(bq[k], bs[k], av[k], at[k]);
            __builtin_amdgcn_sched_barrier(0);
            fetch(c + k + kSmallAhead, k);
        }
    }
#pragma unroll
    for (int k = 0; k < kSmallAhead - 1; ++k)
        if (c + k < chunks) consume(bq[k], bs[k], av[k], at[k]);  // uniform
    if (g == 1) {
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
#pragma unroll
            for (int r = 0; r < 16; ++r) hand[pair][tt * 16 + r][lane] = acc[tt][r];
    }
    __syncthreads();
    if (g == 1 || row >= w.rows) return;
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int t = t0 + 16 * tt + 4 * s4 + u;
            if (t >= tokens) continue;
            // chain L of token u: register 4 (L % 4) + u of wave g = L / 4; the
            // horizontal sum of fortai_q8_dot.c:323-330
            auto lo = [&](int L) { return acc[tt][4 * L + u]; };
            auto hi = [&](int L) { return hand[pair][tt * 16 + 4 * L + u][lane]; };
            const float sum = ((lo(0) + hi(0)) + (lo(2) + hi(2))) + ((lo(1) + hi(1)) + (lo(3) + hi(3)));
            const size_t o = static_cast<size_t>(t) * ld_out + row;
            if constexpr (EPI == 1) out[o] = sum + resid[o];
            else out[o] = sum;
        }
}

// fortai_q8_quantize (fortai_q8_dot.c:153-198) of every token into block-major X8: one
// thread per 4 values, 8 consecutive threads per block.
__global__ __launch_bounds__(256) void q8_quantize_tokens_kernel(const float *__restrict__ x, int tokens, int width,
    int ld_x, int ld, int blocks_pad, int8_t *__restrict__ xq, float *__restrict__ xs) {
    const size_t idx = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    const int groups_pad = blocks_pad * 8;
    const int t = static_cast<int>(idx / groups_pad), g = static_cast<int>(idx % groups_pad);
    if (t >= ld) return;  // whole 8-lane blocks exit together (groups_pad % 8 == 0)
    float4 y = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (t < tokens && g < width / 4) y = reinterpret_cast<const float4 *>(x + static_cast<size_t>(t) * ld_x)[g];
    float scale;
    uint16_t bits;
    const uint32_t packed = quantize_group(y, scale, bits);
    const int b = g >> 3, l = g & 7;
    reinterpret_cast<uint32_t *>(xq + (static_cast<size_t>(b) * ld + t) * 32)[l] = packed;
    if (l == 0) xs[static_cast<size_t>(b) * ld + t] = scale;
}

}  // namespace

int q8_tokens_ld(int tokens) { return (tokens + kTokTile - 1) / kTokTile * kTokTile; }

size_t q8_tokens_bytes(int tokens, int width) {
    const size_t blocks_pad = static_cast<size_t>((width / kQ8Block + 3) / 4) * 4;
    return static_cast<size_t>(q8_tokens_ld(tokens)) * blocks_pad * (32 + 4);
}

hipError_t launch_q8_quantize_tokens(const float *x, int tokens, int width, int ld_x, void *x8, hipStream_t stream) {
    if (tokens <= 0 || width <= 0 || width % kQ8Block || ld_x < width || ld_x % 4) return hipErrorInvalidValue;
    const int ld = q8_tokens_ld(tokens);
    const int blocks_pad = (width / kQ8Block + 3) / 4 * 4;
    int8_t *xq = static_cast<int8_t *>(x8);
    float *xs = reinterpret_cast<float *>(xq + static_cast<size_t>(ld) * blocks_pad * 32);
    const size_t threads = static_cast<size_t>(ld) * blocks_pad * 8;
    hipLaunchKernelGGL(q8_quantize_tokens_kernel, dim3(static_cast<unsigned>((threads + 255) / 256)), dim3(256), 0,
        stream, x, tokens, width, ld_x, ld, blocks_pad, xq, xs);
    return hipGetLastError();
}

hipError_t launch_q8_mmq_exact(const Q8Matrix &w, const void *x8, int tokens, float *out, int ld_out,
    const float *resid, X8Layout layout, hipStream_t stream) {
    if (tokens <= 0 || ld_out < w.rows || w.rows <= 0) return hipErrorInvalidValue;
    const int ld = q8_tokens_ld(tokens);  // a multiple of the 64-token tile
    const int8_t *xq = static_cast<const int8_t *>(x8);
    const float *xs = reinterpret_cast<const float *>(xq + static_cast<size_t>(ld) * w.chunks * 4 * 32);
    const dim3 grid((w.rows + kXTile - 1) / kXTile, (tokens + kXTile - 1) / kXTile);
    const bool blocks = layout == X8Layout::BLOCKS;
    const ExactTiles tiles = exact_tiles(w.rows, tokens, blocks);
    if (tiles != ExactTiles::LARGE) {
        auto small = [&](auto tt_c) {
            constexpr int TT = decltype(tt_c)::value;
            const int tt_n = static_cast<int>(tiles_of(tokens, 16 * TT));
            const dim3 sgrid(static_cast<unsigned>(few_grid(w.rows, tokens, kSmallRows, 16 * TT)));
            auto go = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, sgrid, dim3(256), 0, stream, w, xq, xs, tokens, ld, out, ld_out, resid, tt_n);
            };
            if (blocks) resid ? go(q8_mmq_exact_kernel_small<TT, 1, true>) : go(q8_mmq_exact_kernel_small<TT, 0, true>);
            else resid ? go(q8_mmq_exact_kernel_small<TT, 1, false>) : go(q8_mmq_exact_kernel_small<TT, 0, false>);
            note_launch("q8_mmq_exact_kernel_small<%d,%s> grid %d", TT, resid ? "add" : "store", sgrid.x);
        };
        if (tiles == ExactTiles::SMALL_16) small(std::integral_constant<int, 1>{});
        else small(std::integral_constant<int, 2>{});
        return hipGetLastError();
    }
    const size_t lds = 2 * sizeof(MmqExactStage);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(kXThreads), lds, stream, w, xq, xs, tokens, ld, out, ld_out, resid);
    };
    if (blocks) resid ? go(q8_mmq_exact_kernel<1, true>) : go(q8_mmq_exact_kernel<0, true>);
    else resid ? go(q8_mmq_exact_kernel<1, false>) : go(q8_mmq_exact_kernel<0, false>);
    note_launch("q8_mmq_exact_kernel<%s> grid %dx%d", resid ? "add" : "store", grid.x, grid.y);
    return hipGetLastError();
}

hipError_t launch_q8_mmq(const Q8Matrix &w, const void *x8, int tokens, float *out, int ld_out, const float *resid,
    int32_t *dots, X8Layout layout, hipStream_t stream) {
    if (tokens <= 0 || ld_out < w.rows || w.rows <= 0 || (dots && layout != X8Layout::BLOCKS)) return hipErrorInvalidValue;
    const int ld = q8_tokens_ld(tokens);
    const int8_t *xq = static_cast<const int8_t *>(x8);
    const float *xs = reinterpret_cast<const float *>(xq + static_cast<size_t>(ld) * w.chunks * 4 * 32);
    if (!dots && few_tiles(w.rows, tokens)) {
        const int tt_n = static_cast<int>(tiles_of(tokens, kFewTokens));
        const dim3 sgrid(static_cast<unsigned>(few_grid(w.rows, tokens, kFewRows, kFewTokens)));
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, sgrid, dim3(256), 0, stream, w, xq, xs, tokens, ld, out, ld_out, resid, tt_n);
        };
        if (layout == X8Layout::BLOCKS) resid ? go(q8_mmq_kernel_few<1, true>) : go(q8_mmq_kernel_few<0, true>);
        else resid ? go(q8_mmq_kernel_few<1, false>) : go(q8_mmq_kernel_few<0, false>);
        note_launch("q8_mmq_kernel_few<%s> grid %d", resid ? "add" : "store", sgrid.x);
        return hipGetLastError();
    }
    const dim3 grid((w.rows + kRowTile - 1) / kRowTile, ld / kTokTile);
    const size_t lds = 2 * sizeof(MmqStage);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(kMmqThreads), lds, stream, w, xq, xs, tokens, ld, out, ld_out, resid, dots);
    };
    if (dots) go(q8_mmq_kernel<0, true, true>);
    else if (layout == X8Layout::BLOCKS) resid ? go(q8_mmq_kernel<1, false, true>) : go(q8_mmq_kernel<0, false, true>);
    else resid ? go(q8_mmq_kernel<1, false, false>) : go(q8_mmq_kernel<0, false, false>);
    note_launch("q8_mmq_kernel<%s> grid %dx%d", resid ? "add" : "store", grid.x, grid.y);
    return hipGetLastError();
}

}  // namespace fortai_hip
