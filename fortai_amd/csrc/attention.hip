// Gated GQA decode attention for gfx950 (per-op path): per-head RMSNorm of q
// and k, RoPE, the fp16 KV append, and the reference's two-pass softmax with
// its summation orders kept (attention_exact.h), so the output is
// bit-identical to the CPU path (fortai_qwen35_cpu.f90:990-1033).
//
// Three kernels: scores (one workgroup per kv head x 64 positions; the one
// that holds the new position also appends it), softmax (e values and Z tables)
// and output (one workgroup per head x 8 value dims: the P.V chains and the
// sigmoid gate).  Beyond exact_max positions the first also sums its values
// (flash-decoding) and the last merges the blocks.
#include "attention_exact.h"
#include "fortai_hip_internal.h"
#include "fortai_hip_kernels.h"

namespace fortai_hip {

namespace {

namespace ea = exact_attention;

constexpr int kMaxGroup = 4;
constexpr int kMaxHead = 256;
constexpr int kLoads = ea::kPosBlock * (kMaxHead / 8) / ea::kThreads;
constexpr int kQLoads = kMaxGroup * kMaxHead / ea::kThreads;

typedef uint32_t v4u __attribute__((ext_vector_type(4)));

// The per-sequence workspace behind AttentionParams::partial, in floats:
//   scores [heads][max_context] | e values [heads][max_context] |
//   Z tables [heads][z_segments(max_context)][kZStride] |
//   block statistics [heads][score blocks][2] (the scores kernel's per
//   64-position block max m_b and sum of exp(s - m_b), for the softmax's
//   estimates of the running sums)
__host__ __device__ inline int score_blocks(int max_context) { return (max_context + ea::kPosBlock - 1) / ea::kPosBlock; }
__host__ __device__ inline size_t workspace_floats(int heads, int max_context) {
    return static_cast<size_t>(heads) * max_context * 2 +
        static_cast<size_t>(heads) * ea::z_segments(max_context) * ea::kZStride +
        static_cast<size_t>(heads) * score_blocks(max_context) * 2;
}
__device__ __forceinline__ float2 *block_stats_of(const AttentionParams &p) {
    return reinterpret_cast<float2 *>(p.partial + static_cast<size_t>(p.heads) * p.max_context * 2 +
        static_cast<size_t>(p.heads) * ea::z_segments(p.max_context) * ea::kZStride);
}
__device__ __forceinline__ float *evals_of(const AttentionParams &p) {
    return p.partial + static_cast<size_t>(p.heads) * p.max_context;
}
__device__ __forceinline__ float *ztab_of(const AttentionParams &p) {
    return p.partial + static_cast<size_t>(p.heads) * p.max_context * 2;
}

// Sequence s of a batch (blockIdx.y): every per-sequence buffer is laid out
// [batch][...] with the single-sequence size, and position[s] is its own.
__device__ __forceinline__ AttentionParams attention_seq(AttentionParams p, int s) {
    p.q += static_cast<size_t>(s) * p.heads * 2 * p.head;
    p.k += static_cast<size_t>(s) * p.kv_heads * p.head;
    p.v += static_cast<size_t>(s) * p.kv_heads * p.value;
    p.kcache += static_cast<size_t>(s) * p.max_context * p.kv_heads * p.head;
    p.vcache += static_cast<size_t>(s) * p.max_context * p.kv_heads * p.value;
    p.partial += static_cast<size_t>(s) * workspace_floats(p.heads, p.max_context);
    p.cache_flags += static_cast<size_t>(s) * p.kv_heads;
    p.out += static_cast<size_t>(s) * p.heads * p.value;
    if (p.out_q8l) p.out_q8l = static_cast<unsigned char *>(p.out_q8l) + static_cast<size_t>(s) * q8l_bytes(p.heads * p.value);
    p.position += s;
    if (p.split) p.split += static_cast<size_t>(s) * p.heads * score_blocks(p.max_context) * p.value;
    return p;
}

// Wave 0 of a workgroup holding 64 consecutive outputs (lane d: output
// h * value + d0 + d, 64-aligned): their Q8_0 quantization into p.out_q8l,
// the two blocks as the matvec's f32 prologue forms them (lane j of 16: the
// 4-value group j, fortai_q8_quantize's amax, scale and rounding).  lds: 64
// floats of the caller's LDS, free for this wave.
__device__ __forceinline__ void out_quantize64(const AttentionParams &p, int h, int d0, float val, float *lds) {
    const int lane = static_cast<int>(threadIdx.x) & 63;
    lds[lane] = val;
    wave_lds_fence();
    const float4 y = reinterpret_cast<const float4 *>(lds)[lane & 15];
    float scale;
    uint16_t bits;
    const uint32_t packed = quantize_group(y, scale, bits);
    if (lane < 16) {
        const int g = (h * p.value + d0) / 4 + lane, b = g >> 3, l = g & 7;
        unsigned char *base = static_cast<unsigned char *>(p.out_q8l);
        reinterpret_cast<uint32_t *>(base)[((b >> 2) * 8 + l) * 4 + (b & 3)] = packed;
        const int chunks = p.heads * p.value / 128;
        if (l == 0) reinterpret_cast<float *>(base + static_cast<size_t>(chunks) * 128)[b] = scale;
    }
}

struct ScoresLds {
    float qh[kMaxGroup * kMaxHead];  // normalized q of the group's heads; SPLIT: then e[head][position]
    float kn[kMaxHead];
    float2 rs[kMaxHead / 2];
    uint16_t ktile[ea::kPosBlock][kMaxHead + 8];  // SPLIT: then the position groups' value sums
    int overflow;
};

// Value pieces of a split block: thread t takes dims 8 (t % 32) .. + 7 of
// positions 8 (t / 32) .. + 7.
constexpr int kSplitSlices = kMaxHead / 8;
constexpr int kSplitGroups = ea::kThreads / kSplitSlices;
constexpr int kSplitPer = ea::kPosBlock / kSplitGroups;  // positions per thread
static_assert(kSplitPer % 4 == 0, "whole float4 reads of e");
static_assert(kMaxGroup * kSplitGroups * kMaxHead * sizeof(float) <= sizeof(ScoresLds::ktile), "the value sums fit the key tile");

template <bool FINITE>
__device__ __forceinline__ void split_values(const AttentionParams &p, const uint4 (&vv)[kSplitPer], int n, int group,
    ScoresLds &L, float *dst, size_t head_stride) {
    const int tid = static_cast<int>(threadIdx.x), slice = tid % kSplitSlices, pg = tid / kSplitSlices;
    float acc[kMaxGroup][8];
#pragma unroll
    for (int g = 0; g < kMaxGroup; ++g)
#pragma unroll
        for (int d = 0; d < 8; ++d) acc[g][d] = 0.0f;
#pragma unroll
    for (int i0 = 0; i0 < kSplitPer; i0 += 4) {
        float e[kMaxGroup][4];
#pragma unroll
        for (int g = 0; g < kMaxGroup; ++g) {
            const float4 e4 = *reinterpret_cast<const float4 *>(L.qh + g * ea::kPosBlock + pg * kSplitPer + i0);
            e[g][0] = e4.x; e[g][1] = e4.y; e[g][2] = e4.z; e[g][3] = e4.w;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (pg * kSplitPer + i0 + i >= n) continue;  // (a clamped copy of the last position)
            const uint32_t hw[4] = {vv[i0 + i].x, vv[i0 + i].y, vv[i0 + i].z, vv[i0 + i].w};
#pragma unroll
            for (int d = 0; d < 8; ++d) {
                const float v = ea::kv<FINITE>(static_cast<uint16_t>(hw[d >> 1] >> (16 * (d & 1))));
#pragma unroll
                for (int g = 0; g < kMaxGroup; ++g) acc[g][d] = __builtin_fmaf(e[g][i], v, acc[g][d]);
            }
        }
    }
    float *part = reinterpret_cast<float *>(&L.ktile[0][0]);  // [head][position group][dim]
#pragma unroll
    for (int g = 0; g < kMaxGroup; ++g) {
        float4 *o = reinterpret_cast<float4 *>(part + (g * kSplitGroups + pg) * kMaxHead + slice * 8);
        o[0] = make_float4(acc[g][0], acc[g][1], acc[g][2], acc[g][3]);
        o[1] = make_float4(acc[g][4], acc[g][5], acc[g][6], acc[g][7]);
    }
    __syncthreads();
    if (tid >= p.value) return;
    for (int g = 0; g < group; ++g) {
        float o = 0.0f;
#pragma unroll
        for (int k = 0; k < kSplitGroups; ++k) o += part[(g * kSplitGroups + k) * kMaxHead + tid];
        dst[g * head_stride + tid] = o;
    }
}

// One block of kPosBlock positions of one kv head, for its GQA group.
// SPLIT (beyond exact_max): instead of the scores, the block's max m_b (or, with
// exponent-31 halves about, a little more), sum Z_b of exp(s - m_b) and value sums o_b = sum exp(s - m_b) v, which merge_block
// combines (flash-decoding).  UNROLLED: the scores of 256-wide heads fully
// unrolled (more registers).
template <bool SPLIT, bool UNROLLED>
__device__ __forceinline__ void scores_block(const AttentionParams &p, int pos, ScoresLds &L) {
    float *qh = L.qh, *kn = L.kn;
    float2 *rs = L.rs;
    auto &ktile = L.ktile;
    int &overflow = L.overflow;
    const int tid = static_cast<int>(threadIdx.x), wave = tid >> 6, lane = tid & 63;
    const int positions = pos + 1;
    // block-major: the blocks that hold positions are dispatched first, the
    // ones past the current position (which only read it and exit) last
    const int b = div(static_cast<int>(blockIdx.x), p.div_kv_heads);
    const int kvh = static_cast<int>(blockIdx.x) - b * p.kv_heads;
    const int p0 = b * ea::kPosBlock;
    if (p0 >= positions) return;
    const int n = min(ea::kPosBlock, positions - p0);
    const bool owns_new = pos >= p0 && pos < p0 + n;
    const int group = static_cast<int>(p.div_group.d), HD = p.head, VD = p.value, NKV = p.kv_heads;
    const int half = p.rope_dim / 2;

    // q, k, the norm weights, v and the rope entry first (indices clamped in
    // bounds), then the key rows: the loads complete in order, so the q/k
    // norms and RoPE run while the key rows (the only HBM stream of this
    // kernel) are still arriving
    float qv[kQLoads];
#pragma unroll
    for (int i = 0; i < kQLoads; ++i) {
        const int e = min(tid + i * ea::kThreads, group * HD - 1);
        const int eh = div(e, p.div_head);
        qv[i] = p.q[static_cast<size_t>(kvh * group + eh) * 2 * HD + (e - eh * HD)];
    }
    const int th = min(tid, HD - 1), tv = min(tid, VD - 1);
    const float knv = p.k[static_cast<size_t>(kvh) * HD + th];
    // the q and k norm weights a lane applies (elements lane + 64 j of a head)
    constexpr int kNW = kMaxHead / 64;
    float qwr[kNW], kwr[kNW];
#pragma unroll
    for (int j = 0; j < kNW; ++j) {
        qwr[j] = p.q_norm[min(lane + 64 * j, HD - 1)];
        kwr[j] = p.k_norm[min(lane + 64 * j, HD - 1)];
    }
    const float vnv = p.v[static_cast<size_t>(kvh) * VD + tv];
    const float2 rsv = half > 0 ? p.rope[static_cast<size_t>(pos) * half + min(tid, half - 1)] : make_float2(0.0f, 0.0f);
    const int flag = p.cache_flags[kvh];
    v4u kr[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int li = tid + i * ea::kThreads;
        const int jj = div(li, p.div_segs), sg = li - jj * static_cast<int>(p.div_segs.d);
        const int j = min(jj, n - 1);  // rows past n re-read row n-1 (in bounds)
        kr[i] = reinterpret_cast<const v4u *>(p.kcache + (static_cast<size_t>(p0 + j) * NKV + kvh) * HD)[sg];
    }
#pragma unroll
    for (int i = 0; i < kQLoads; ++i)
        if (tid + i * ea::kThreads < group * HD) qh[tid + i * ea::kThreads] = qv[i];
    if (tid < HD) kn[tid] = knv;
    if (tid < half) rs[tid] = rsv;
    if (tid == 0) overflow = 0;
    FORTAI_ATT_MARK(17);
    __syncthreads();
    for (int sl = wave; sl < group + (owns_new ? 1 : 0); sl += ea::kThreads / 64) {
        if (sl < group) ea::norm_rope_regs(qh + sl * HD, HD, qwr, p.eps, rs, p.rope_dim, lane);
        else ea::norm_rope_regs(kn, HD, kwr, p.eps, rs, p.rope_dim, lane);
    }
    FORTAI_ATT_MARK(18);
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int li = tid + i * ea::kThreads;
        const int j = div(li, p.div_segs), sg = li - j * static_cast<int>(p.div_segs.d);
        if (j < n) *reinterpret_cast<v4u *>(&ktile[j][sg * 8]) = kr[i];
    }
    // the block's values, while the scores are formed (the keys' registers are free)
    const int vslice = tid % kSplitSlices, vpg = tid / kSplitSlices;
    const int vd0 = (vslice * 8 < VD ? vslice : 0) * 8;  // slices past VD repeat slice 0 and are not stored
    uint4 vv[SPLIT ? kSplitPer : 1];
    if constexpr (SPLIT) {
#pragma unroll
        for (int i = 0; i < kSplitPer; ++i)
            vv[i] = *reinterpret_cast<const uint4 *>(
                p.vcache + (static_cast<size_t>(p0 + min(vpg * kSplitPer + i, n - 1)) * NKV + kvh) * VD + vd0);
    }
    __syncthreads();
    FORTAI_ATT_MARK(19);
    if (owns_new) {
        // append at pos (fortai_qwen35_cpu.f90:1594-1601)
        if (tid < HD) {
            const uint16_t kb = float_to_half_kv(kn[tid]);
            p.kcache[(static_cast<size_t>(pos) * NKV + kvh) * HD + tid] = kb;
            ktile[pos - p0][tid] = kb;
            if ((kb & 0x7c00u) == 0x7c00u) overflow = 1;
        }
        if (tid < VD) {
            const uint16_t vb = float_to_half_kv(vnv);
            p.vcache[(static_cast<size_t>(pos) * NKV + kvh) * VD + tid] = vb;
            if ((vb & 0x7c00u) == 0x7c00u) overflow = 1;
        }
        __syncthreads();
        if (tid == 0 && overflow) p.cache_flags[kvh] = 1;
    }
    const bool finite = flag == 0 && overflow == 0;
    const float sqrt_head = sqrtf(static_cast<float>(HD));
    const int gi = tid >> 6, j = tid & 63;
    float ev = 0.0f;  // SPLIT: exp(s - m_b)
    if (gi < group) {  // wave gi: head kvh * group + gi, positions p0 + lane
        constexpr float kLowest = -3.402823466e38f;  // -huge(1.0_real32)
        float sc = kLowest;
        if (j < n) {
            const float *qg = qh + gi * HD;
            const uint16_t *kr = &ktile[j][0];
            if (finite) sc = UNROLLED && HD == 256 ? ea::score_n<true, 256>(qg, kr, sqrt_head) : ea::score<true>(qg, kr, HD, sqrt_head);
            else sc = ea::score<false>(qg, kr, HD, sqrt_head);
            if constexpr (!SPLIT) p.partial[static_cast<size_t>(kvh * group + gi) * p.max_context + p0 + j] = sc;
        }
        // (from the reference's first maximum -huge: a block whose every score is
        // -infinity then weighs 0 beside the others, not NaN)
        float mb = fmaxf(wave_max(sc), kLowest);
        // +-huge values (exponent-31 halves): with weights of up to 1 two of them
        // overflow the block's sum, however little the block weighs beside the
        // others.  Relative to m_b + 5 the 64 weights sum to 64 e^-5 < 1.
        if constexpr (SPLIT)
            if (!finite) mb += 5.0f;
        float2 *stats = block_stats_of(p) + static_cast<size_t>(kvh * group + gi) * score_blocks(p.max_context) + b;
        if constexpr (SPLIT) {
            ev = j < n ? expf_libm(sc - mb) : 0.0f;
            const float z = wave_sum(ev);
            if (j == 0) *stats = make_float2(mb, z);
        } else {
            // the block's max and sum of exp(s - max) (a fast exp, in double): the
            // softmax kernel's estimates start from these, not from every score
            double t = j < n ? static_cast<double>(__expf(sc - mb)) : 0.0;
            t = wave_sum(t);
            if (j == 0) *stats = make_float2(mb, static_cast<float>(t));
        }
    }
    FORTAI_ATT_MARK(20);
    if constexpr (SPLIT) {
        // the new position's values come from the projection, not from the cache
        if (owns_new) {
            // (loaded and rounded once: inside the loop's branch each position would wait for its own loads)
            const float *vn = p.v + static_cast<size_t>(kvh) * VD + vd0;
            uint32_t w[4];
#pragma unroll
            for (int d = 0; d < 4; ++d)
                w[d] = float_to_half_kv(vn[2 * d]) | static_cast<uint32_t>(float_to_half_kv(vn[2 * d + 1])) << 16;
            const uint4 row = make_uint4(w[0], w[1], w[2], w[3]);
#pragma unroll
            for (int i = 0; i < kSplitPer; ++i)
                if (p0 + vpg * kSplitPer + i >= pos) vv[i] = row;  // pos, and the clamped copies of it
        }
        __syncthreads();  // every wave is done with qh and the key tile
        qh[tid] = ev;     // [head][position]; 0 past n and past the group
        __syncthreads();
        const size_t head_stride = static_cast<size_t>(score_blocks(p.max_context)) * VD;
        float *dst = p.split + static_cast<size_t>(kvh * group) * head_stride + static_cast<size_t>(b) * VD;
        if (finite) split_values<true>(p, vv, n, group, L, dst, head_stride);
        else split_values<false>(p, vv, n, group, L, dst, head_stride);
    }
}

__global__ __launch_bounds__(ea::kThreads) void attention_scores_kernel(const AttentionParams p_batch) {
    FORTAI_TRACE_SCOPE(3);
    const AttentionParams p = attention_seq(p_batch, static_cast<int>(blockIdx.y));
    __shared__ __align__(16) ScoresLds L;
    FORTAI_ATT_MARK(16);
    const int pos = *p.position;
    if (pos < 0 || pos >= p.max_context) return;  // never index past the cache
    scores_block<false, true>(p, pos, L);
}

// The first kernel of contexts longer than exact_max: the scores up to it,
// scores and values in one pass beyond.  Bound by latency: position, q norm, key
// block, the 256 dependent adds of a score, values; four 40 KB workgroups share
// a CU and cover each other's waits (1024 of them, 32768 positions of two kv
// heads, are one round).  So its registers are held to four waves per SIMD, the
// values are loaded into the keys' registers, and the scores run in the rolled
// form (unrolled, at three waves per SIMD: 24 against 21-22 us).  A pass over
// the scores with the values, 256 positions per workgroup, and the merge were
// launches of their own before: 8 heads, whole call at 8300 positions 31.1 ->
// 20.4 us, 20000: 33.4 -> 24.2, 32768: 38.1 -> 29.0 (67 MB: 2.3 TB/s), 65536:
// 54.4 -> 43.6.  Exact positions, two launches fewer behind them: 1000: 25.6 ->
// 22.9, 4000: 32.8 -> 30.3, 8000: 43.4 -> 41.5.
__global__ __launch_bounds__(ea::kThreads, 4) void attention_split_kernel(const AttentionParams p_batch) {
    const AttentionParams p = attention_seq(p_batch, static_cast<int>(blockIdx.y));
    __shared__ __align__(16) ScoresLds L;
    const int pos = *p.position;
    if (pos < 0 || pos >= p.max_context) return;
    if (pos + 1 > p.exact_max) scores_block<true, false>(p, pos, L);
    else scores_block<false, false>(p, pos, L);
}

// Beyond exact_max, DIMS value dims of head h from the blocks' partials:
// M = max m_b, Z = sum Z_b e^(m_b - M), out = (sum o_b e^(m_b - M)) / Z *
// sigmoid(gate).  Blocks go to kMergeParts running sums per dim (block b to sum
// b % kMergeParts), whatever DIMS is, so that every output kernel gives the same
// bits.  lds: kMergeTile + kMergeParts * DIMS + 4 floats.
constexpr int kMaxSplitPositions = 1 << 20;
constexpr int kMergeTile = 1024;
constexpr int kMergeParts = 32;
template <int DIMS>
__device__ __forceinline__ void merge_block(const AttentionParams &p, int h, int d0, int positions, float *lds) {
    constexpr int kThreadsPerDim = ea::kThreads / DIMS, kSums = kMergeParts / kThreadsPerDim;
    static_assert(kSums * kThreadsPerDim == kMergeParts, "whole sums per thread");
    constexpr int kAhead = 16 / (kSums > 4 ? 4 : kSums);  // blocks in flight per sum
    float *f = lds, *part = lds + kMergeTile, *red = part + kMergeParts * DIMS;
    const int tid = static_cast<int>(threadIdx.x), wave = tid >> 6, lane = tid & 63;
    const int VD = p.value, nb = score_blocks(positions), nmax = score_blocks(p.max_context);
    const float2 *st = block_stats_of(p) + static_cast<size_t>(h) * nmax;
    const int dl = tid % DIMS, q = tid / DIMS, d = min(d0 + dl, VD - 1);
    const float *base = p.split + static_cast<size_t>(h) * nmax * VD + d;
    const float gate = p.q[static_cast<size_t>(h) * 2 * p.head + p.head + d];
    float mx = -__builtin_inff();
    for (int b = tid; b < nb; b += ea::kThreads) mx = fmaxf(mx, st[b].x);
    mx = wave_max(mx);
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    float zp = 0.0f, o[kSums];
#pragma unroll
    for (int k = 0; k < kSums; ++k) o[k] = 0.0f;
    for (int t0 = 0; t0 < nb; t0 += kMergeTile) {
        const int cnt = min(kMergeTile, nb - t0);
        for (int b = tid; b < cnt; b += ea::kThreads) {
            const float2 s2 = st[t0 + b];
            const float fb = expf_libm(s2.x - mx);
            f[b] = fb;
            zp = __builtin_fmaf(s2.y, fb, zp);
        }
        __syncthreads();
        for (int b0 = q * kSums; b0 < cnt; b0 += kAhead * kMergeParts) {
            float x[kAhead][kSums];
#pragma unroll
            for (int u = 0; u < kAhead; ++u)
#pragma unroll
                for (int k = 0; k < kSums; ++k)
                    x[u][k] = base[static_cast<size_t>(t0 + min(b0 + u * kMergeParts + k, cnt - 1)) * VD];
#pragma unroll
            for (int u = 0; u < kAhead; ++u)
#pragma unroll
                for (int k = 0; k < kSums; ++k)
                    if (b0 + u * kMergeParts + k < cnt) o[k] = __builtin_fmaf(x[u][k], f[b0 + u * kMergeParts + k], o[k]);
        }
        __syncthreads();
    }
    zp = wave_sum(zp);
    if (lane == 0) red[wave] = zp;
#pragma unroll
    for (int k = 0; k < kSums; ++k) part[(q * kSums + k) * DIMS + dl] = o[k];
    __syncthreads();
    if (tid >= DIMS || d0 + dl >= VD) return;
    const float z = (red[0] + red[1]) + (red[2] + red[3]);
    float sum = 0.0f;
#pragma unroll
    for (int k = 0; k < kMergeParts; ++k) sum += part[k * DIMS + dl];
    const float out = (sum / z) * sigmoid_ref(gate);
    p.out[static_cast<size_t>(h) * VD + d0 + dl] = out;
    if constexpr (DIMS == 64)
        if (p.out_q8l) out_quantize64(p, h, d0, out, f);
}

// e_p = expf(s_p - m) of kSeg-position segments of one head, stored for the
// output kernels, and each segment's Z candidate table (attention_exact.h,
// resolve_z): thread c runs the segment's left-to-right chain from candidate
// starting sum c.  grid (heads x G, batch): workgroup (k0, h) takes segments
// k0, k0 + G, ... of head h (G = z_segments(max_context) for one sequence, so
// one segment each; at most 8 for a batch, so that at a short position in a
// long cache few workgroups load the scores and exit idle), segments holding
// positions dispatched first.
__global__ __launch_bounds__(ea::kThreads) void attention_softmax_kernel(const AttentionParams p_batch) {
    FORTAI_TRACE_SCOPE(4);
    const AttentionParams p = attention_seq(p_batch, static_cast<int>(blockIdx.y));
    __shared__ __align__(16) float e_seg[ea::kSeg];
    __shared__ double dred[2 * ea::kWaves];
    __shared__ float fred[ea::kWaves];
    __shared__ MathTables mt;  // loaded after the scores are issued (the wait for it is theirs)
    static_assert(ea::kZCand == ea::kThreads && ea::kSeg == ea::kThreads, "one candidate and one position per thread");
    const int pos = *p.position;
    const int k0 = div(static_cast<int>(blockIdx.x), p.div_heads), h = static_cast<int>(blockIdx.x) - k0 * p.heads;
    const int G = div(static_cast<int>(gridDim.x), p.div_heads);
    const int tid = static_cast<int>(threadIdx.x), wave = tid >> 6, lane = tid & 63;
    const float *sc = p.partial + static_cast<size_t>(h) * p.max_context;
    FORTAI_ATT_MARK(21);
    // beyond exact_max there are no e values or Z tables (contexts that never
    // get there do not wait for the position here)
    if (p.max_context > p.exact_max && pos >= p.exact_max) return;
    // the statistics of every 64-position score block (max m_b, sum of
    // exp(s - m_b)) written by the scores kernel: one block per thread and
    // register up to kStatRegs * 256 blocks (clamped in bounds; those past the
    // position are masked), and the first segment's own scores
    constexpr int kStatRegs = 2;
    const int cap = p.max_context < p.exact_max ? p.max_context : p.exact_max;
    const int nb_cap = score_blocks(cap);
    const float2 *bst = block_stats_of(p) + static_cast<size_t>(h) * score_blocks(p.max_context);
    float2 st[kStatRegs];
#pragma unroll
    for (int i = 0; i < kStatRegs; ++i)
        if (i * ea::kThreads < nb_cap) st[i] = bst[min(tid + i * ea::kThreads, nb_cap - 1)];
    const float sv0 = sc[min(k0 * ea::kSeg + tid, cap - 1)];
    mt.load();  // visible after the barrier of the max below
    if (pos < 0 || pos >= p.max_context) return;
    const int n = pos + 1;
    if (k0 * ea::kSeg >= n) return;
    const int nb = score_blocks(n);
    // m = max over every score = max over the blocks' maxima (any order and
    // grouping gives the same value)
    constexpr float kLowest = -3.402823466e38f;  // -huge(1.0_real32)
    float m = kLowest;
#pragma unroll
    for (int i = 0; i < kStatRegs; ++i)
        if (tid + i * ea::kThreads < nb) m = fmaxf(m, st[i].x);
    for (int b = tid + kStatRegs * ea::kThreads; b < nb; b += ea::kThreads) m = fmaxf(m, bst[b].x);
    m = wave_max(m);
    if (lane == 0) fred[wave] = m;
    __syncthreads();
    m = fmaxf(fmaxf(fred[0], fred[1]), fmaxf(fred[2], fred[3]));
    // block b's share of the running sum, rescaled to m (a fast exp, in double)
    double tb[kStatRegs];
#pragma unroll
    for (int i = 0; i < kStatRegs; ++i) {
        const int b = tid + i * ea::kThreads;
        tb[i] = b < nb ? static_cast<double>(st[i].y) * static_cast<double>(__expf(st[i].x - m)) : 0.0;
    }
    FORTAI_ATT_MARK(22);
    for (int k = k0; k * ea::kSeg < n; k += G) {
    if (k != k0) __syncthreads();  // the previous segment's chains have read e_seg and dred
    const int p0 = k * ea::kSeg;
    const int cnt = min(ea::kSeg, n - p0);
    // the segment's own e values, exactly as the reference computes them
    const float sv = k == k0 ? sv0 : sc[min(p0 + tid, n - 1)];
    const float e = tid < cnt ? mt.expf(sv - m) : -0.0f;  // -0 leaves a sum unchanged
    e_seg[tid] = e;
    if (tid < cnt) evals_of(p)[static_cast<size_t>(h) * p.max_context + p0 + tid] = e;
    // the estimates of the running sums entering this segment and the next:
    // the blocks before it, and those before the next one (the next
    // segment's workgroup forms the same sum in the same order)
    const int b_in = p0 / ea::kPosBlock, b_next = (p0 + ea::kSeg) / ea::kPosBlock;
    double est = 0.0, est_next = 0.0;
#pragma unroll
    for (int i = 0; i < kStatRegs; ++i) {
        const int b = tid + i * ea::kThreads;
        if (b < b_in) est += tb[i];
        if (b < b_next) est_next += tb[i];
    }
    for (int b = tid + kStatRegs * ea::kThreads; b < nb && b < b_next; b += ea::kThreads) {
        const float2 sb = bst[b];
        const double t = static_cast<double>(sb.y) * static_cast<double>(__expf(sb.x - m));
        if (b < b_in) est += t;
        est_next += t;
    }
    est = wave_sum(est);
    est_next = wave_sum(est_next);
    if (lane == 0) {
        dred[wave] = est;
        dred[ea::kWaves + wave] = est_next;
    }
    __syncthreads();
    est = (dred[0] + dred[1]) + (dred[2] + dred[3]);
    est_next = (dred[4] + dred[5]) + (dred[6] + dred[7]);
    if (k == k0) FORTAI_ATT_MARK(23);
    const uint32_t skew = static_cast<uint32_t>(p.z_skew);
    const uint32_t centre = k == 0 ? 0u : __float_as_uint(static_cast<float>(est)) + skew;
    const uint32_t centre_next = __float_as_uint(static_cast<float>(est_next)) + skew;
    float acc = k == 0 ? 0.0f : __uint_as_float(centre + static_cast<uint32_t>(tid) - ea::kZCand / 2);
#pragma unroll 16
    for (int j = 0; j < ea::kSeg; j += 4) {
        const float4 v = *reinterpret_cast<const float4 *>(e_seg + j);
        acc = acc + v.x;
        acc = acc + v.y;
        acc = acc + v.z;
        acc = acc + v.w;
    }
    if (k == k0) FORTAI_ATT_MARK(24);
    const bool last = p0 + ea::kSeg >= n;
    float *tab = ztab_of(p) + (static_cast<size_t>(h) * ea::z_segments(p.max_context) + k) * ea::kZStride;
    tab[tid] = acc;
    tab[ea::kZNext + tid] = last ? acc : __int_as_float(ea::z_index(acc, centre_next));
    if (tid == 0) tab[ea::kZCentre] = __uint_as_float(centre);
    }
    FORTAI_ATT_MARK(25);
}

// Z of head h: the walk words of the candidate tables into LDS (up to
// kZLdsSegments segments; longer contexts walk in global memory), then
// resolve_z by one thread.  walk_lds: min(z_segments(n), kZLdsSegments) *
// kZCand words.  Returns Z in every thread.
constexpr int kZLdsSegments = 32;
__host__ __device__ inline int z_lds_segments(int positions) {
    return ea::z_segments(positions) < kZLdsSegments ? ea::z_segments(positions) : kZLdsSegments;
}
__device__ __forceinline__ const float *head_tab(const AttentionParams &p, int h) {
    return ztab_of(p) + static_cast<size_t>(h) * ea::z_segments(p.max_context) * ea::kZStride;
}
__device__ __forceinline__ float head_z(const AttentionParams &p, int h, int n, int32_t *walk_lds, float *slot) {
    const int tid = static_cast<int>(threadIdx.x);
    const int nseg = (n + ea::kSeg - 1) / ea::kSeg;
    const float *tab = head_tab(p, h);
    if (nseg <= kZLdsSegments) {
        for (int i = tid; i < nseg * ea::kZCand; i += ea::kThreads)
            walk_lds[i] = __float_as_int(tab[static_cast<size_t>(i / ea::kZCand) * ea::kZStride + ea::kZNext + i % ea::kZCand]);
    }
    __syncthreads();
    if (tid == 0) {
        const float *ev = evals_of(p) + static_cast<size_t>(h) * p.max_context;
        *slot = nseg <= kZLdsSegments
            ? ea::resolve_z(walk_lds, ea::kZCand, tab, ev, n)
            : ea::resolve_z(reinterpret_cast<const int32_t *>(tab + ea::kZNext), ea::kZStride, tab, ev, n);
    }
    __syncthreads();
    return *slot;
}

// The output of one head x kDims value dims.  Workgroups are numbered so
// that the ones reading the same 128-byte value lines (the 64 dims of a kv
// head that 8 slices x the GQA group share) are consecutive on one XCD
// (workgroup b runs on XCD b % 8).  Every load that does not depend on the
// position (the first value pieces, e values and the Z tables, all clamped to
// the cache) is issued together with the position's, in one round trip.
constexpr int kTabRegs = kZLdsSegments * ea::kZCand / ea::kThreads;  // walk words per thread
__global__ __launch_bounds__(ea::kThreads) void attention_output_kernel(const AttentionParams p_batch) {
    FORTAI_TRACE_SCOPE(5);
    const AttentionParams p = attention_seq(p_batch, static_cast<int>(blockIdx.y));
    extern __shared__ __align__(16) float lds[];
    // sigmoid of the gate: wave 1 forms it while thread 0 resolves Z
    __shared__ float gate_sig[ea::kDims];
    const int tid = static_cast<int>(threadIdx.x);
    FORTAI_ATT_MARK(0);
    const int pos = *p.position;
    const int group = static_cast<int>(p.div_group.d), HD = p.head, VD = p.value, NKV = p.kv_heads;
    const int slices = static_cast<int>(p.div_slices.d), nwg = p.heads * slices;
    const int b = static_cast<int>(blockIdx.x);
    int h, d0;
    if (nwg % 8 == 0 && VD % 64 == 0) {
        const int i = (b % 8) * (nwg / 8) + b / 8;  // logical index, consecutive on one XCD
        const int i8 = i / 8, sl = i % 8;
        const int t = div(i8, p.div_group), g = i8 - t * group;
        const int kvh = div(t, p.div_vd64), lg = t - kvh * static_cast<int>(p.div_vd64.d);
        h = kvh * group + g;
        d0 = (lg * 8 + sl) * ea::kDims;
    } else {
        h = div(b, p.div_slices);
        d0 = (b - h * slices) * ea::kDims;
    }
    const int kvh = div(h, p.div_group);
    const int cap = p.max_context < p.exact_max ? p.max_context : p.exact_max;  // positions this kernel serves
    const uint16_t *vbase = p.vcache + static_cast<size_t>(kvh) * VD + d0;
    const size_t vstride = static_cast<size_t>(NKV) * VD;
    const float *ev = evals_of(p) + static_cast<size_t>(h) * p.max_context;
    const float *tab = head_tab(p, h);
    const int rows = z_lds_segments(cap);
    if (p.max_context > p.exact_max && pos >= p.exact_max) {
        if (pos < p.max_context) merge_block<ea::kDims>(p, h, d0, pos + 1, lds);
        return;
    }
    ea::ValuePieces v;
    float e4[ea::kPieces];
    int32_t tr[kTabRegs];  // walk word tid of segment r
    ea::value_prefetch(vbase, vstride, p.max_context, v);
    ea::e_prefetch(ev, p.max_context, e4);
    static_assert(ea::kZCand == ea::kThreads, "one walk word per thread and segment");
    // unconditional loads (a branch around each would make the compiler wait
    // for it): rows past the cached ones re-read the last (row 0 always exists)
    const int last_row = max(rows, 1) - 1;
#pragma unroll
    for (int r = 0; r < kTabRegs; ++r)
        tr[r] = __float_as_int(tab[static_cast<size_t>(min(r, last_row)) * ea::kZStride + ea::kZNext + tid]);
    const float gate = p.q[static_cast<size_t>(h) * 2 * HD + HD + d0 + (tid & (ea::kDims - 1))];
    const int flag = p.cache_flags[kvh];
    FORTAI_ATT_MARK(3);
    if (pos < 0 || pos >= p.max_context) return;
    const int positions = pos + 1;
    float *work = lds;
    int32_t *walk_lds = reinterpret_cast<int32_t *>(lds + ea::work_floats());
    const int nseg = ea::z_segments(positions);
    if (nseg <= kZLdsSegments) {
#pragma unroll
        for (int r = 0; r < kTabRegs; ++r)
            if (r < nseg) walk_lds[r * ea::kZCand + tid] = tr[r];
    }
    __syncthreads();
    FORTAI_ATT_MARK(1);
    if (tid == 0)
        work[0] = nseg <= kZLdsSegments
            ? ea::resolve_z(walk_lds, ea::kZCand, tab, ev, positions)
            : ea::resolve_z(reinterpret_cast<const int32_t *>(tab + ea::kZNext), ea::kZStride, tab, ev, positions);
    // (glibc's algorithm with its table in constant memory: one lookup, off
    // the critical path; seen by wave 0 after the output step's barriers)
    if (tid >= 64 && tid < 64 + ea::kDims) gate_sig[tid - 64] = sigmoid_ref(gate);
    FORTAI_ATT_MARK(2);
    __syncthreads();
    const float z = work[0];
    FORTAI_ATT_MARK(5);
    const float acc = flag == 0 ? ea::attend_given_z<true>(ev, z, positions, vbase, vstride, work, v, e4)
                                : ea::attend_given_z<false>(ev, z, positions, vbase, vstride, work, v, e4);
    if (tid < ea::kDims) p.out[static_cast<size_t>(h) * VD + d0 + tid] = acc * gate_sig[tid];
    FORTAI_ATT_MARK(4);
}

static_assert(kMergeTile + kMergeParts * ea::kDims + 4 <= ea::work_floats(), "merge_block fits the output step's LDS");
size_t output_lds_bytes(int positions) {
    return (ea::work_floats() + static_cast<size_t>(z_lds_segments(positions)) * ea::kZCand) * sizeof(float);
}

// ------------------------------------------------------- exact, batches
// The same arithmetic as attention_output_kernel (the reference's two-pass
// softmax and P.V with its summation orders, fortai_qwen35_cpu.f90:1016-1031)
// with one workgroup per (head, 64 value dims, sequence) instead of one per
// (head, 8 value dims): Z from the candidate tables (head_z), then lane d of
// wave 0 runs the P.V chain of value dim d0 + d over the positions in order,
// out_d = fl(w_0 v_0,d) + fl(w_1 v_1,d) + ... with w_p = e_p / Z.  A batch has
// many (head, sequence) pairs, so this fills the chip with 1/8 as many
// workgroups, each chain step using all 64 lanes; a single sequence keeps the
// per-slice kernel, whose chains are shorter per workgroup.
//
// Values reach LDS in tiles of kWideTile positions, loaded by all four waves
// two tiles ahead of the chain: each thread loads 8 positions x 8 dims (eight
// 16-byte pieces), transposes them in registers and stores one 16-byte row
// of 8 positions per dim, so the tile is [dim][position] and a chain lane
// reads 8 positions of its dim with one 16-byte LDS read (and w_p of the tile,
// divided when the tile is stored, with two).  Row R (dim R) keeps its group g
// of 8 positions at column g + 2 (R / 16): with a row pitch of 49 16-byte bank
// groups (1 mod 16), the 16 lanes of a store pass (8 rows 8 apart, two column
// groups) and of a read pass (16 consecutive rows, one group) all fall on
// different banks.  The Z walk words use the tile's LDS before the first tile
// is stored; nothing is sized by the context.
constexpr int kWideTile = 256;                   // positions per value tile
constexpr int kWideDims = 64;                    // value dims per workgroup
constexpr int kWidePitchT = 392;                 // halves per LDS row: 32 + 6 column groups, 49 x 16 bytes
constexpr int kWideMaxPositions = 8192;
static_assert(kWideTile / 8 * (kWideDims / 8) == ea::kThreads, "one 8 x 8 block of (position, dim) per thread");
static_assert(kWidePitchT >= (kWideTile / 8 + 2 * (kWideDims / 16 - 1)) * 8 && kWidePitchT % 8 == 0 &&
    (kWidePitchT / 8) % 16 == 1, "every shifted column in the row; 16-byte rows one bank group apart");
static_assert(kWideDims * kWidePitchT * 2 >= kZLdsSegments * ea::kZCand * 4, "the Z walk words fit the tile's LDS");

// dynamic LDS of attention_output_wide_kernel: the transposed tile, then w of the tile
constexpr size_t kWideLdsBytes = static_cast<size_t>(kWideDims) * kWidePitchT * 2 + kWideTile * 4;
static_assert((kMergeTile + kMergeParts * kWideDims + 4) * sizeof(float) <= kWideLdsBytes, "merge_block fits");

// halves k of dwords a (low half of the result) and b (high half)
__device__ __forceinline__ uint32_t pick_halves(uint32_t a, uint32_t b, int hi) {
    return hi ? __builtin_amdgcn_perm(b, a, 0x07060302u) : __builtin_amdgcn_perm(b, a, 0x05040100u);
}

template <bool FINITE>
__device__ __forceinline__ void attend_wide(const AttentionParams &p, int h, int d0, int n, uint16_t *vt, float *wt,
    float *red) {
    const int tid = static_cast<int>(threadIdx.x), wave = tid >> 6, lane = tid & 63;
    const int group = p.heads / p.kv_heads, HD = p.head, VD = p.value, NKV = p.kv_heads;
    const int kvh = h / group;
    const uint16_t *vb = p.vcache + static_cast<size_t>(kvh) * VD + d0;
    const size_t vs = static_cast<size_t>(NKV) * VD;
    const int tiles = (n + kWideTile - 1) / kWideTile;
    const float *ev = evals_of(p) + static_cast<size_t>(h) * p.max_context;
    // this thread's block: positions pg * 8 .. + 7 of a tile, dims pc * 8 .. + 7
    const int pc = tid & 7, pg = tid >> 3;
    const int pcl = min(pc, (min(kWideDims, VD - d0) >> 3) - 1);  // dims past VD re-read the last piece
    FORTAI_ATTW_MARK(0);
    // tile t: eight 16-byte pieces and e of position t * kWideTile + tid (all clamped to the last position)
    auto fetch = [&](int t, uint4 (&regs)[8], float &e) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int pp = min(t * kWideTile + pg * 8 + i, n - 1);
            regs[i] = *reinterpret_cast<const uint4 *>(vb + static_cast<size_t>(pp) * vs + pcl * 8);
        }
        e = ev[min(t * kWideTile + tid, n - 1)];
    };
    // Z first: its table loads would otherwise return after the whole value
    // fetch (loads complete in order)
    const float z = head_z(p, h, n, reinterpret_cast<int32_t *>(vt), red + 4);  // ends with a barrier
    FORTAI_ATTW_MARK(3);
    uint4 ra[8], rb[8];
    float ea_ = 0.0f, eb_ = 0.0f;
    fetch(0, ra, ea_);
    if (tiles > 1) fetch(1, rb, eb_);
    FORTAI_ATTW_MARK(1);
    // the block transposed: row of dim pc * 8 + k holds positions pg * 8 .. + 7
    auto stash = [&](const uint4 (&r)[8], float e) {
        const uint32_t *w32 = reinterpret_cast<const uint32_t *>(r);  // w32[4 i + m]: dims 2m, 2m + 1 of position i
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int m = k >> 1, hi = k & 1;
            uint4 row;
            row.x = pick_halves(w32[0 * 4 + m], w32[1 * 4 + m], hi);
            row.y = pick_halves(w32[2 * 4 + m], w32[3 * 4 + m], hi);
            row.z = pick_halves(w32[4 * 4 + m], w32[5 * 4 + m], hi);
            row.w = pick_halves(w32[6 * 4 + m], w32[7 * 4 + m], hi);
            *reinterpret_cast<uint4 *>(vt + (pc * 8 + k) * kWidePitchT + (pg + 2 * (pc >> 1)) * 8) = row;
        }
        wt[tid] = e / z;
    };
    const int d = d0 + lane;
    // this lane's row from its shifted column 0 (lanes past VD read a row they do not write)
    const uint16_t *myrow = vt + lane * kWidePitchT + 2 * (lane >> 4) * 8;
    // the chain of one tile: groups of 8 positions from a ring of three
    // register sets, each group's LDS reads issued two groups before its adds
    struct Grp {
        uint4 v;
        float4 w0, w1;
    };
    // group g of the tile (a compile-time index: immediate LDS offsets)
    auto ld = [&](int g, Grp &r) {
        r.v = *reinterpret_cast<const uint4 *>(myrow + g * 8);
        r.w0 = *reinterpret_cast<const float4 *>(wt + g * 8);
        r.w1 = *reinterpret_cast<const float4 *>(wt + g * 8 + 4);
    };
    auto add8 = [&](const Grp &r, float acc) {
        if constexpr (FINITE) {
            // fl(w * f32(v)) in one instruction (exact widening, one rounding)
            acc = acc + half_times<false>(r.v.x, r.w0.x);
            acc = acc + half_times<true>(r.v.x, r.w0.y);
            acc = acc + half_times<false>(r.v.y, r.w0.z);
            acc = acc + half_times<true>(r.v.y, r.w0.w);
            acc = acc + half_times<false>(r.v.z, r.w1.x);
            acc = acc + half_times<true>(r.v.z, r.w1.y);
            acc = acc + half_times<false>(r.v.w, r.w1.z);
            acc = acc + half_times<true>(r.v.w, r.w1.w);
        } else {
            const uint32_t q[4] = {r.v.x, r.v.y, r.v.z, r.v.w};
            const float wv[8] = {r.w0.x, r.w0.y, r.w0.z, r.w0.w, r.w1.x, r.w1.y, r.w1.z, r.w1.w};
#pragma unroll
            for (int k = 0; k < 8; ++k)
                acc = acc + wv[k] * ea::kv<false>(static_cast<uint16_t>(q[k >> 1] >> (16 * (k & 1))));
        }
        return acc;
    };
    auto chain = [&](int t, float acc) {
        const int cnt = min(kWideTile, n - t * kWideTile);
        const int full = cnt >> 3;
        constexpr int kGroups = kWideTile / 8;
        Grp ring[3];
        ld(0, ring[0]);
        ld(1, ring[1]);
        // fully unrolled: every LDS offset is an immediate, and the scheduling
        // barriers keep each group's reads two groups ahead of its adds
#pragma unroll
        for (int g = 0; g < kGroups; ++g) {
            if (g < full) {  // uniform
                if (g + 2 < kGroups) ld(g + 2, ring[(g + 2) % 3]);
                __builtin_amdgcn_sched_barrier(0);
                acc = add8(ring[g % 3], acc);
            }
        }
        // the last cnt % 8 positions
        for (int k = 0; k < (cnt & 7); ++k) {
            const int pp = full * 8 + k;
            acc = acc + wt[pp] * ea::kv<FINITE>(myrow[pp]);
        }
        return acc;
    };
    float acc = 0.0f;
    for (int t = 0; t < tiles; t += 2) {
        stash(ra, ea_);
        __syncthreads();
        if (t + 2 < tiles) fetch(t + 2, ra, ea_);
        if (wave == 0) acc = chain(t, acc);
        __syncthreads();
        if (t + 1 >= tiles) break;
        stash(rb, eb_);
        __syncthreads();
        if (t + 3 < tiles) fetch(t + 3, rb, eb_);
        if (wave == 0) acc = chain(t + 1, acc);
        __syncthreads();
    }
    FORTAI_ATTW_MARK(5);
    if (wave == 0 && d < VD) {
        const float gate = p.q[static_cast<size_t>(h) * 2 * HD + HD + d];
        const float o = acc * sigmoid_ref(gate);
        p.out[static_cast<size_t>(h) * VD + d] = o;
        if (p.out_q8l) out_quantize64(p, h, d0, o, wt);  // (the tile is consumed: wt is free)
    }
}

// grid: (heads x ceil(value / 64), batch)
__global__ __launch_bounds__(ea::kThreads) void attention_output_wide_kernel(const AttentionParams p_batch) {
    FORTAI_TRACE_SCOPE(12);
    const AttentionParams p = attention_seq(p_batch, static_cast<int>(blockIdx.y));
    extern __shared__ __align__(16) float wide_lds[];
    __shared__ float red[8];
    const int pos = *p.position;
    if (pos < 0 || pos >= p.max_context) return;
    const int n = pos + 1;
    const int slices = (p.value + kWideDims - 1) / kWideDims;
    const int h = static_cast<int>(blockIdx.x) / slices, d0 = (static_cast<int>(blockIdx.x) % slices) * kWideDims;
    const int kvh = h / (p.heads / p.kv_heads);
    if (n > p.exact_max) {
        merge_block<kWideDims>(p, h, d0, n, wide_lds);
        return;
    }
    uint16_t *vt = reinterpret_cast<uint16_t *>(wide_lds);
    float *wt = wide_lds + kWideDims * kWidePitchT / 2;
    if (p.cache_flags[kvh] == 0)
        attend_wide<true>(p, h, d0, n, vt, wt, red);
    else
        attend_wide<false>(p, h, d0, n, vt, wt, red);
}

}  // namespace

size_t attention_scores_floats(int heads, int max_context) { return workspace_floats(heads, max_context); }

size_t attention_split_floats(int heads, int max_context, int value) {
    return static_cast<size_t>(heads) * score_blocks(max_context) * value;
}

// workgroups per head of attention_softmax_kernel: one per segment for a
// single sequence, at most 8 (each looping over segments) for a batch
int softmax_groups(int positions, int batch) {
    const int segs = ea::z_segments(positions);
    return batch > 1 && segs > 8 ? 8 : segs;
}

bool attention_quantizes_output(const AttentionParams &p, int batch) {
    const int exact_positions = p.max_context < p.exact_max ? p.max_context : p.exact_max;
    const bool wide = (batch > 1 || p.force_wide) && exact_positions <= kWideMaxPositions && p.value <= ea::kThreads;
    return wide && p.value % 64 == 0 && (p.heads * p.value) % 128 == 0;
}

hipError_t launch_attention(const AttentionParams &params, hipStream_t stream, int batch) {
    if (batch < 1) return hipErrorInvalidValue;
    if (params.out_q8l && !attention_quantizes_output(params, batch)) return hipErrorInvalidValue;
    const int group = params.kv_heads > 0 ? params.heads / params.kv_heads : 0;
    AttentionParams p = params;
    p.div_heads = fast_div(static_cast<uint32_t>(p.heads));
    p.div_kv_heads = fast_div(static_cast<uint32_t>(p.kv_heads));
    p.div_group = fast_div(static_cast<uint32_t>(group));
    p.div_head = fast_div(static_cast<uint32_t>(p.head));
    p.div_segs = fast_div(static_cast<uint32_t>(p.head / 8));
    p.div_slices = fast_div(static_cast<uint32_t>(p.value / ea::kDims));
    p.div_vd64 = fast_div(static_cast<uint32_t>(p.value / 64));
    const bool beyond = p.max_context > p.exact_max;  // (each kernel picks its regime from the device position)
    if (beyond && (!p.split || p.max_context > kMaxSplitPositions)) return hipErrorInvalidValue;
    if (group < 1 || group > kMaxGroup || p.heads % p.kv_heads || p.head > kMaxHead || p.head % 8 ||
        p.value % ea::kDims || p.value > p.head || p.rope_dim > p.head || p.rope_dim % 2 || !p.out || !p.partial)
        return hipErrorInvalidValue;
    const int exact_positions = p.max_context < p.exact_max ? p.max_context : p.exact_max;
    const int nblk_max = (p.max_context + ea::kPosBlock - 1) / ea::kPosBlock;
    const char *first = beyond ? "attention_split_kernel" : "attention_scores_kernel";
    hipLaunchKernelGGL(beyond ? attention_split_kernel : attention_scores_kernel, dim3(p.kv_heads * nblk_max, batch),
        dim3(ea::kThreads), 0, stream, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (exact_positions > 0) {
        hipLaunchKernelGGL(attention_softmax_kernel, dim3(p.heads * softmax_groups(exact_positions, batch), batch),
            dim3(ea::kThreads), 0, stream, p);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    const bool wide = (batch > 1 || p.force_wide) && exact_positions <= kWideMaxPositions && p.value <= ea::kThreads;
    if (wide) {
        const size_t wlds = kWideLdsBytes;
        const int wgrid = p.heads * ((p.value + kWideDims - 1) / kWideDims);
        hipLaunchKernelGGL(attention_output_wide_kernel, dim3(wgrid, batch), dim3(ea::kThreads), wlds, stream, p);
        e = hipGetLastError();
        note_launch("%s grid %dx%d + attention_softmax_kernel grid %dx%d + "
            "attention_output_wide_kernel grid %dx%d", first, p.kv_heads * nblk_max, batch,
            p.heads * softmax_groups(exact_positions, batch), batch, wgrid, batch);
    } else {
        hipLaunchKernelGGL(attention_output_kernel, dim3(p.heads * (p.value / ea::kDims), batch), dim3(ea::kThreads),
            output_lds_bytes(exact_positions), stream, p);
        e = hipGetLastError();
        note_launch("%s grid %dx%d + attention_softmax_kernel grid %dx%d + "
            "attention_output_kernel grid %dx%d", first, p.kv_heads * nblk_max, batch,
            p.heads * softmax_groups(exact_positions, batch), batch, p.heads * (p.value / ea::kDims), batch);
    }
    return e;
}

}  // namespace fortai_hip
