// Prompt prefill of a batch of sequences: T tokens per sequence in one pass.
//
// The reference has no prefill: it runs every prompt token through the decode
// step (fortai_qwen35_cpu.f90:591-711).  Here the projections of all
// batch x T tokens are token-block products on the matrix cores (mmq.hip), the
// causal conv1d (:856-879) and the norms and gates of every token run in
// parallel, and the delta rule (:880-906) runs over the tokens as a serial chain
// per 8 state rows of a value head.  Causal attention (:1006-1033) runs per
// query block.  The exact mode keeps every summation order of the per-token
// decode (in attention the two-pass softmax) and gives its bits; the fast mode
// (whole-block dots, fp16 matrix-core attention with an online softmax) agrees
// with it within rounding.  Rows are token-major: row n = s * T + t is token t of
// sequence s, at position t.
#include "attention_exact.h"
#include "fortai_hip_internal.h"
#include "fortai_hip_kernels.h"

#include <type_traits>

namespace fortai_hip {

namespace {

namespace ea = exact_attention;

constexpr int kRowThreads = 256;

// x [rows][width] (row pitch ld_x) -> optional RMSNorm (fortai_qwen35_cpu.f90:
// 1408-1432) -> fortai_q8_quantize of every row into X8.  One workgroup per row.
__global__ __launch_bounds__(kRowThreads) void rms_quantize_tokens_kernel(const float *__restrict__ x, int ld_x,
    int width, const float *__restrict__ norm, float eps, int ld, int blocks_pad, int8_t *__restrict__ xq,
    float *__restrict__ xs) {
    __shared__ double red[kRowThreads / 64];
    const int n = static_cast<int>(blockIdx.x), tid = static_cast<int>(threadIdx.x);
    const float *row = x + static_cast<size_t>(n) * ld_x;
    float inv = 1.0f;
    if (norm) {
        double ss = 0.0;
        for (int i = tid; i < width; i += kRowThreads) ss += static_cast<double>(row[i]) * static_cast<double>(row[i]);
        ss = wave_sum(ss);
        if ((tid & 63) == 0) red[tid >> 6] = ss;
        __syncthreads();
        double total = 0.0;
        for (int w = 0; w < kRowThreads / 64; ++w) total += red[w];
        inv = 1.0f / sqrtf(static_cast<float>(div_count(total, width)) + eps);
    }
    for (int g = tid; g < blocks_pad * 8; g += kRowThreads) {
        float4 y = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (g < width / 4) {
            y = reinterpret_cast<const float4 *>(row)[g];
            if (norm) {
                const float4 w4 = reinterpret_cast<const float4 *>(norm)[g];
                y.x = (y.x * inv) * w4.x; y.y = (y.y * inv) * w4.y; y.z = (y.z * inv) * w4.z; y.w = (y.w * inv) * w4.w;
            }
        }
        float scale;
        uint16_t bits;
        const uint32_t packed = quantize_group(y, scale, bits);
        const int b = g >> 3, l = g & 7;
        x8_store(xq, xs, ld, n, b, l, packed, scale);
    }
}

// GDN output o with the gate: per head ((o / rms(o)) * ssm_norm) * silu(z)
// (fortai_qwen35_cpu.f90:907-915), quantized into X8.  One workgroup per row;
// a head is head/4 consecutive threads (aligned power of two).
__global__ __launch_bounds__(kRowThreads) void gated_quantize_tokens_kernel(const float *__restrict__ o,
    const float *__restrict__ z, const float *__restrict__ norm, float eps, int width, int head, int ld,
    int blocks_pad, int8_t *__restrict__ xq, float *__restrict__ xs) {
    const int n = static_cast<int>(blockIdx.x), tid = static_cast<int>(threadIdx.x);
    const float *orow = o + static_cast<size_t>(n) * width;
    const float *zrow = z + static_cast<size_t>(n) * width;
    const int hl = head / 4;
    for (int g0 = 0; g0 < blocks_pad * 8; g0 += kRowThreads) {
        const int g = g0 + tid;
        const bool in = g < width / 4;
        float4 y = in ? reinterpret_cast<const float4 *>(orow)[g] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        double ss = static_cast<double>(y.x) * y.x + static_cast<double>(y.y) * y.y +
            static_cast<double>(y.z) * y.z + static_cast<double>(y.w) * y.w;
        ss = group_sum_up(ss, hl);
        if (in) {
            const float nf = sqrtf(static_cast<float>(div_count(ss, head)) + eps);
            const float4 w4 = reinterpret_cast<const float4 *>(norm)[g % hl];
            const float4 z4 = reinterpret_cast<const float4 *>(zrow)[g];
            y.x = ((y.x / nf) * w4.x) * silu_poly(z4.x);
            y.y = ((y.y / nf) * w4.y) * silu_poly(z4.y);
            y.z = ((y.z / nf) * w4.z) * silu_poly(z4.z);
            y.w = ((y.w / nf) * w4.w) * silu_poly(z4.w);
        }
        float scale;
        uint16_t bits;
        const uint32_t packed = quantize_group(y, scale, bits);
        if (g < blocks_pad * 8) {
            const int b = g >> 3, l = g & 7;
            x8_store(xq, xs, ld, n, b, l, packed, scale);
        }
    }
}

// FFN hidden silu(gate) * up (fortai_silu_product) quantized into X8.
__global__ __launch_bounds__(kRowThreads) void silu_product_quantize_kernel(const float *__restrict__ gate,
    const float *__restrict__ up, int width, int ld, int blocks_pad, int8_t *__restrict__ xq, float *__restrict__ xs) {
    const int n = static_cast<int>(blockIdx.x), tid = static_cast<int>(threadIdx.x);
    const float4 *g4 = reinterpret_cast<const float4 *>(gate + static_cast<size_t>(n) * width);
    const float4 *u4 = reinterpret_cast<const float4 *>(up + static_cast<size_t>(n) * width);
    for (int g = tid; g < blocks_pad * 8; g += kRowThreads) {
        float4 y = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (g < width / 4) {
            const float4 a = g4[g], b = u4[g];
            y = make_float4(silu_poly(a.x) * b.x, silu_poly(a.y) * b.y, silu_poly(a.z) * b.z, silu_poly(a.w) * b.w);
        }
        float scale;
        uint16_t bits;
        const uint32_t packed = quantize_group(y, scale, bits);
        const int b = g >> 3, l = g & 7;
        x8_store(xq, xs, ld, n, b, l, packed, scale);
    }
}

// Causal conv1d + SiLU over the prompt (fortai_qwen35_cpu.f90:856-879).  The
// conv has no recurrence: output t reads the inputs t-K+1..t, those before
// the prompt from conv_state [batch][K-1][C] (oldest first).  One thread per
// (sequence, channel, kConvTokens consecutive tokens) computes each output
// with the decode's conv_silu (same window, same order), reading the old
// state only; conv_state_advance_kernel then stores the last K-1 inputs.
// x: raw projections [batch*T][C].
constexpr int kConvTokens = 8;

__global__ __launch_bounds__(256) void conv_silu_tokens_kernel(const float *__restrict__ x,
    const float *__restrict__ conv_w, const float *__restrict__ conv_state, float *__restrict__ out, int T, int C,
    int K) {
    const int c = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
    const int t0 = static_cast<int>(blockIdx.y) * kConvTokens;
    const int s = static_cast<int>(blockIdx.z);
    if (c >= C) return;
    float taps[kConvMax];
#pragma unroll
    for (int i = 0; i < kConvMax; ++i) taps[i] = i < K ? conv_w[static_cast<size_t>(c) * K + i] : 0.0f;
    const float *cs = conv_state + static_cast<size_t>(s) * (K - 1) * C + c;
    const float *xs = x + static_cast<size_t>(s) * T * C + c;
    float *os = out + static_cast<size_t>(s) * T * C + c;
    // inputs t0-K+1 .. t0+kConvTokens-1 (kConvMax-1 window slots, then the tokens)
    float in[kConvMax - 1 + kConvTokens];
#pragma unroll
    for (int i = 0; i < kConvMax - 1 + kConvTokens; ++i) {
        const int u = t0 - (kConvMax - 1) + i;  // input index; < 0: from the state
        float v = 0.0f;
        if (u >= 0 && u < T) v = xs[static_cast<size_t>(u) * C];
        else if (u < 0 && u >= -(K - 1)) v = cs[static_cast<size_t>(K - 1 + u) * C];
        in[i] = v;
    }
#pragma unroll
    for (int j = 0; j < kConvTokens; ++j) {
        const int t = t0 + j;
        if (t >= T) break;
        float win[kConvMax - 1];
#pragma unroll
        for (int i = 0; i < kConvMax - 1; ++i) win[i] = i < K - 1 ? in[j + (kConvMax - K) + i] : 0.0f;
        os[static_cast<size_t>(t) * C] = conv_silu(win, taps, K, in[j + kConvMax - 1]);
    }
}

// conv_state <- the last K-1 inputs of the prompt (older state entries when
// the prompt is shorter than K-1); each thread reads its channel's old state
// before writing it.
__global__ __launch_bounds__(256) void conv_state_advance_kernel(const float *__restrict__ x, float *conv_state, int T,
    int C, int K) {
    const int c = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
    const int s = static_cast<int>(blockIdx.y);
    if (c >= C) return;
    float *cs = conv_state + static_cast<size_t>(s) * (K - 1) * C + c;
    const float *xs = x + static_cast<size_t>(s) * T * C + c;
    float nw[kConvMax - 1];
#pragma unroll
    for (int i = 0; i < kConvMax - 1; ++i) {
        if (i >= K - 1) break;
        const int u = T - (K - 1) + i;
        nw[i] = u >= 0 ? xs[static_cast<size_t>(u) * C] : cs[static_cast<size_t>(i + T) * C];
    }
#pragma unroll
    for (int i = 0; i < kConvMax - 1; ++i)
        if (i < K - 1) cs[static_cast<size_t>(i) * C] = nw[i];
}

// Per token: the L2 norms of every key head's q and k (1 / max(|x|, eps),
// fortai_qwen35_cpu.f90:1455-1471) and every value head's beta and decay
// (:890-894).  One workgroup per token; wave w takes key heads w, w + 4, ...
__global__ __launch_bounds__(256) void gdn_token_prep_kernel(const float *__restrict__ qkv, const float *__restrict__ alpha,
    const float *__restrict__ beta, const float *__restrict__ ssm_a, const float *__restrict__ ssm_dt, int C,
    int key_heads, int value_heads, int head, int state_size, float eps, float *__restrict__ qinv,
    float *__restrict__ kinv, float *__restrict__ beta_out, float *__restrict__ decay_out) {
    const int n = static_cast<int>(blockIdx.x), tid = static_cast<int>(threadIdx.x);
    const int lane = tid & 63, wave = tid >> 6;
    const float *row = qkv + static_cast<size_t>(n) * C;
    for (int kh = wave; kh < key_heads; kh += 4) {
        const float *q = row + kh * head, *k = row + state_size * key_heads + kh * head;
        double sq = 0.0, sk = 0.0;
        for (int i = lane; i < head; i += 64) {
            sq += static_cast<double>(q[i]) * q[i];
            sk += static_cast<double>(k[i]) * k[i];
        }
        sq = wave_sum(sq);
        sk = wave_sum(sk);
        if (lane == 0) {
            qinv[static_cast<size_t>(n) * key_heads + kh] = 1.0f / fmaxf(sqrtf(static_cast<float>(sq)), eps);
            kinv[static_cast<size_t>(n) * key_heads + kh] = 1.0f / fmaxf(sqrtf(static_cast<float>(sk)), eps);
        }
    }
    for (int h = tid; h < value_heads; h += 256) {
        const size_t i = static_cast<size_t>(n) * value_heads + h;
        beta_out[i] = sigmoid_ref(beta[i]);
        decay_out[i] = exp_rounded(ssm_a[h] * softplus_ref(alpha[i] + ssm_dt[h]));
    }
}

// The delta rule over time (fortai_q8_dot.c:356-398), the state in registers
// in the decode kernel's layout: S[row][8 i + l] at
// state[((h * HEAD + row) * 8 + l) * HEAD/8 + i].  A one-wave workgroup runs
// 8 rows of one value head of one sequence (blockIdx.y), lane l of a row its
// eighth.  The steps are a serial chain, so what counts is the latency
// of one: no barrier (the wave's own LDS operations are in order), nothing
// waited for inside a step, and two chains in flight -- the q dot of token t
// and the decay and k dot of token t + 1 run interleaved over the columns
// (each chain in its own order).  Tokens reach LDS kGdnChunk at a time from
// registers loaded one chunk ahead; a step's reads are issued before the
// horizontal sum that its column loop waits for.  A lane's 16 columns are
// contiguous with a 4-float pad per lane, so its 16-byte reads meet no bank
// twice.
// Measured (head 128, against 16 rows per two-wave workgroup with two barriers
// per 16 tokens and four-byte reads): 16 heads x 77 tokens 59 -> 24 us, 32
// heads x 3 x 701 538 -> 270 us, 32 heads x 8 x 512 490 -> 342 us.  Two rows per
// lane (each read of q and k shared) 414 us at the last.
constexpr int kGdnChunk = 4;

template <int HEAD>
__global__ __launch_bounds__(64) void gdn_prefill_kernel(const float *__restrict__ qkv,
    const float *__restrict__ qinv, const float *__restrict__ kinv, const float *__restrict__ beta,
    const float *__restrict__ decay, float *__restrict__ state, float *__restrict__ out, int T, int C, int key_heads,
    int value_heads, int state_size) {
    constexpr int kCols = HEAD / 8, kPitch = kCols + 4, kRows = 8;
    constexpr int kSlot = 2 * 8 * kPitch;
    // per token: q [8][kPitch], k [8][kPitch]; the 4-float pads of the 16 lane
    // rows hold 64 aux words: v of the rows, then beta, decay (and copies of it)
    __shared__ __align__(16) float ring[2 * kGdnChunk * kSlot];
    auto aux = [](int i) { return (i >> 2) * kPitch + kCols + (i & 3); };
    const int lane = static_cast<int>(threadIdx.x);
    const int s = static_cast<int>(blockIdx.y);
    constexpr int kBlocks = HEAD / kRows;
    const int h = static_cast<int>(blockIdx.x) / kBlocks, r0 = (static_cast<int>(blockIdx.x) % kBlocks) * kRows;
    const int kh = h / (value_heads / key_heads);
    const int r8 = lane >> 3, l = lane & 7;
    const int inner = value_heads * HEAD;
    float *sp = state + static_cast<size_t>(s) * value_heads * HEAD * HEAD +
        ((static_cast<size_t>(h) * HEAD + r0 + r8) * 8 + l) * kCols;
    float st[kCols];
#pragma unroll
    for (int i = 0; i < kCols; ++i) st[i] = sp[i];
    const float scale = 1.0f / sqrtf(static_cast<float>(HEAD));
    // this lane's share of a token: 4 values of q (lanes < HEAD/4) or k, the
    // head's inverse norm, and one aux word
    const bool has_qk = lane < HEAD / 2;
    const int ql = has_qk ? lane : 0, isk = ql >= HEAD / 4, c4 = (ql % (HEAD / 4)) * 4;
    const float *qk_src = qkv + (isk ? state_size * key_heads : 0) + kh * HEAD + c4;
    const float *inv_src = (isk ? kinv : qinv) + kh;
    const int al = min(lane, kRows + 1);
    const float *aux_src = al < kRows ? qkv + 2 * state_size * key_heads + h * HEAD + r0 + al
                                      : (al == kRows ? beta : decay) + h;
    const int aux_pitch = al < kRows ? C : value_heads;
    float4 fq[kGdnChunk];
    float fi[kGdnChunk], fa[kGdnChunk];
    auto fetch = [&](int chunk) {
#pragma unroll
        for (int j = 0; j < kGdnChunk; ++j) {
            const size_t n = static_cast<size_t>(s) * T + min(chunk * kGdnChunk + j, T - 1);
            fq[j] = *reinterpret_cast<const float4 *>(qk_src + n * C);
            fi[j] = inv_src[n * key_heads];
            fa[j] = aux_src[n * aux_pitch];
        }
    };
    auto stash = [&](int chunk) {
        float *base = ring + (chunk & 1) * (kGdnChunk * kSlot);
#pragma unroll
        for (int j = 0; j < kGdnChunk; ++j) {
            float *slot = base + j * kSlot;
            const float v[4] = {fq[j].x, fq[j].y, fq[j].z, fq[j].w};
            if (HEAD == 128 || has_qk) {
                float *dst = slot + isk * 8 * kPitch + c4 / 8;
#pragma unroll
                for (int u = 0; u < 4; ++u) dst[((c4 & 4) + u) * kPitch] = v[u] * fi[j];
            }
            slot[aux(lane)] = fa[j];
        }
        wave_lds_fence();
    };
    struct Token {  // k, v and beta of a token
        float k[kCols], v, b;
    };
    auto read_cols = [&](const float *src, float (&dst)[kCols]) {
#pragma unroll
        for (int i = 0; i < kCols / 4; ++i) {
            const float4 f = reinterpret_cast<const float4 *>(src + l * kPitch)[i];
            dst[4 * i] = f.x; dst[4 * i + 1] = f.y; dst[4 * i + 2] = f.z; dst[4 * i + 3] = f.w;
        }
    };
    auto read_token = [&](const float *slot, Token &t, float &d) {
        read_cols(slot + 8 * kPitch, t.k);
        t.v = slot[aux(r8)];
        t.b = slot[aux(kRows)];
        d = slot[aux(kRows + 1)];
    };
    fetch(0);
    stash(0);
    fetch(1);
    Token ta, tb;
    float kd = 0.0f;
    {
        float d0;
        read_token(ring, ta, d0);
#pragma unroll
        for (int i = 0; i < kCols; ++i) {
            const float d = st[i] * d0;
            st[i] = d;
            kd = __builtin_fmaf(d, ta.k[i], kd);
        }
    }
    float *orow = out + static_cast<size_t>(s) * T * inner + h * HEAD + r0 + r8;
    // token t (its slot) with token t + 1's decay and k dot
    auto step = [&](int t, const float *slot, const float *slot1, const Token &cur, Token &nxt) {
        float q[kCols], dn;
        read_token(slot1, nxt, dn);
        read_cols(slot, q);
        __builtin_amdgcn_sched_barrier(0);
        const float delta = (cur.v - row_hsum8(kd)) * cur.b;
        if (t + 1 >= T) dn = 1.0f;  // past the last token the state is kept: a factor of one
        float qd = 0.0f;
        kd = 0.0f;
#pragma unroll
        for (int i = 0; i < kCols; ++i) {
            const float u = __builtin_fmaf(delta, cur.k[i], st[i]);
            qd = __builtin_fmaf(u, q[i], qd);
            const float d = u * dn;
            st[i] = d;
            kd = __builtin_fmaf(d, nxt.k[i], kd);
        }
        // every lane of the row stores the same value: a branch here would
        // keep the compiler from interleaving the two chains
        orow[static_cast<size_t>(t) * inner] = row_hsum8(qd) * scale;
    };
    static_assert(kGdnChunk == 4, "the two tokens' registers swap an even number of times per chunk");
    int c = 0;
    for (; (c + 1) * kGdnChunk <= T; ++c) {
        const int t = c * kGdnChunk;
        const float *here = ring + (c & 1) * (kGdnChunk * kSlot), *other = ring + ((c & 1) ^ 1) * (kGdnChunk * kSlot);
        step(t, here, here + kSlot, ta, tb);
        step(t + 1, here + kSlot, here + 2 * kSlot, tb, ta);
        stash(c + 1);
        fetch(c + 2);
        step(t + 2, here + 2 * kSlot, here + 3 * kSlot, ta, tb);
        step(t + 3, here + 3 * kSlot, other, tb, ta);
    }
    // the last, partial chunk (its slot past the end is read but not used)
    const float *here = ring + (c & 1) * (kGdnChunk * kSlot);
    for (int t = c * kGdnChunk; t < T; ++t, here += kSlot) {
        step(t, here, here + kSlot, ta, tb);
        ta = tb;
    }
#pragma unroll
    for (int i = 0; i < kCols; ++i) sp[i] = st[i];
}

// Per token: q and k per-head RMSNorm + RoPE at the token's position
// (fortai_qwen35_cpu.f90:990-999, 1473-1497), q in place; k and v appended to
// the fp16 caches [batch][max_context][kv_heads][head] with the reference's
// float_to_half (:1594-1601); cache_flags [batch][kv_heads] set when an
// exponent-31 half is stored.  One workgroup per token, one wave per head.
__global__ __launch_bounds__(256) void qk_rope_append_kernel(float *__restrict__ q, const float *__restrict__ k,
    const float *__restrict__ v, const float *__restrict__ q_norm, const float *__restrict__ k_norm,
    const float2 *__restrict__ rope, uint16_t *__restrict__ kcache, uint16_t *__restrict__ vcache,
    int *__restrict__ flags, int T, int heads, int kv_heads, int head, int value, int rope_dim, int max_context,
    float eps) {
    __shared__ __align__(16) float buf[4][256];
    __shared__ __align__(16) float wq[256], wk[256];
    const int n = static_cast<int>(blockIdx.x), tid = static_cast<int>(threadIdx.x);
    const int lane = tid & 63, wave = tid >> 6;
    const int s = n / T, pos = n % T;
    for (int i = tid; i < head; i += 256) {
        wq[i] = q_norm[i];
        wk[i] = k_norm[i];
    }
    __syncthreads();
    const float2 *rp = rope + static_cast<size_t>(pos) * (rope_dim / 2);
    // q heads then k heads, one wave each
    for (int j = wave; j < heads + kv_heads; j += 4) {
        float *b = buf[wave];
        const bool isq = j < heads;
        const float *src = isq ? q + (static_cast<size_t>(n) * heads + j) * 2 * head
                               : k + (static_cast<size_t>(n) * kv_heads + (j - heads)) * head;
        for (int i = lane; i < head; i += 64) b[i] = src[i];
        wave_lds_fence();
        ea::norm_rope(b, head, isq ? wq : wk, eps, rp, rope_dim, lane);
        if (isq) {
            float *dst = q + (static_cast<size_t>(n) * heads + j) * 2 * head;
            for (int i = lane; i < head; i += 64) dst[i] = b[i];
        } else {
            const int kvh = j - heads;
            uint16_t *dst = kcache + ((static_cast<size_t>(s) * max_context + pos) * kv_heads + kvh) * head;
            int over = 0;
            for (int i = lane; i < head; i += 64) {
                const uint16_t hb = float_to_half_kv(b[i]);
                dst[i] = hb;
                over |= (hb & 0x7c00u) == 0x7c00u;
            }
            if (__any(over) && lane == 0) flags[static_cast<size_t>(s) * kv_heads + kvh] = 1;
        }
        wave_lds_fence();
    }
    for (int e = tid; e < kv_heads * value; e += 256) {
        const int kvh = e / value, i = e % value;
        const uint16_t hb = float_to_half_kv(v[(static_cast<size_t>(n) * kv_heads + kvh) * value + i]);
        vcache[((static_cast<size_t>(s) * max_context + pos) * kv_heads + kvh) * value + i] = hb;
        if ((hb & 0x7c00u) == 0x7c00u) flags[static_cast<size_t>(s) * kv_heads + kvh] = 1;
    }
}

// Causal attention of every prompt token with the reference's arithmetic
// and summation orders (fortai_qwen35_cpu.f90:1006-1031), so every output is
// bit-identical to the decode step's exact attention at that position:
//   s_j = (q . k_j, left to right, separately rounded) / sqrt(head)
//   m = max s_j;  e_j = expf(s_j - m);  Z = e_0 + e_1 + ... (left to right)
//   out_d = fl(e_0/Z v_0,d) + fl(e_1/Z v_1,d) + ... (left to right) * sigmoid(gate_d)
// One workgroup per (block of qb = 1 or 2 queries, head, sequence): this kernel
// serves the prompts past the tiled one below, where the scores of more than two
// queries do not fit in LDS.  Keys and values pass through LDS 64 positions at a
// time.  Wave w forms the scores and weights of query w.  A query's masked keys
// (past its position) get e = +0 and weight +0: adding +0 or -0 to a running
// sum leaves it unchanged, so every chain can run to the block's last key.
constexpr int kXKeys = 64;      // keys per staged tile
constexpr int kXFallbackQ = 2;  // queries per workgroup at most

template <int HEAD>
__global__ __launch_bounds__(256) void attention_prefill_exact_kernel(const float *__restrict__ q,
    const uint16_t *__restrict__ kcache, const uint16_t *__restrict__ vcache, float *__restrict__ out, int T,
    int heads, int kv_heads, int max_context, int qb, int kcap) {
    static_assert(HEAD % 64 == 0 && HEAD <= 256, "head 64, 128 or 256");
    extern __shared__ __align__(16) unsigned char lds_raw[];
    float *qs = reinterpret_cast<float *>(lds_raw);                  // [qb][HEAD] normalized q
    uint16_t *kv = reinterpret_cast<uint16_t *>(qs + qb * HEAD);    // K: [HEAD/8][kXKeys][8]; V: [kXKeys][HEAD]
    float *sc = reinterpret_cast<float *>(kv + kXKeys * HEAD);       // [qb][kcap] scores, then e, then weights
    const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, wave = tid >> 6;
    const int h = static_cast<int>(blockIdx.y), s = static_cast<int>(blockIdx.z);
    const int q0 = static_cast<int>(blockIdx.x) * qb;
    const int nq = min(qb, T - q0);
    const int keys = q0 + nq;  // keys 0..keys-1 cover the block
    const int kvh = h / (heads / kv_heads);
    const float sqrt_head = sqrtf(static_cast<float>(HEAD));
    for (int e = tid; e < qb * HEAD; e += 256) {
        const int qi = e / HEAD, d = e % HEAD;
        qs[e] = qi < nq ? q[((static_cast<size_t>(s) * T + q0 + qi) * heads + h) * 2 * HEAD + d] : 0.0f;
    }
    // ---- scores: lane = key, wave = query
    for (int j0 = 0; j0 < keys; j0 += kXKeys) {
        __syncthreads();
        for (int e = tid; e < kXKeys * (HEAD / 8); e += 256) {
            const int j = e / (HEAD / 8), piece = e % (HEAD / 8);
            const int p = min(j0 + j, keys - 1);
            const uint4 v8 = *reinterpret_cast<const uint4 *>(
                kcache + ((static_cast<size_t>(s) * max_context + p) * kv_heads + kvh) * HEAD + piece * 8);
            *reinterpret_cast<uint4 *>(kv + (piece * kXKeys + j) * 8) = v8;
        }
        __syncthreads();
        const int j = j0 + lane;
        if (wave >= qb) continue;
        float acc = 0.0f;
        for (int d = 0; d < HEAD; d += 8) {
            const uint4 k8 = *reinterpret_cast<const uint4 *>(kv + ((d / 8) * kXKeys + lane) * 8);
            const uint32_t kw[4] = {k8.x, k8.y, k8.z, k8.w};
            const float4 qa = *reinterpret_cast<const float4 *>(qs + wave * HEAD + d);
            const float4 qc = *reinterpret_cast<const float4 *>(qs + wave * HEAD + d + 4);
            const float qv[8] = {qa.x, qa.y, qa.z, qa.w, qc.x, qc.y, qc.z, qc.w};
#pragma unroll
            for (int u = 0; u < 8; ++u)
                acc = acc + qv[u] * gguf_half_to_real(static_cast<uint16_t>(u & 1 ? kw[u >> 1] >> 16 : kw[u >> 1] & 0xffffu));
        }
        if (j < keys) sc[wave * kcap + j] = acc / sqrt_head;
    }
    __syncthreads();
    // ---- softmax weights: wave = query, lanes over keys
    constexpr float kLowest = -3.402823466e38f;  // -huge(1.0_real32)
    float *row = sc + wave * kcap;
    if (wave < nq) {
        const int n = q0 + wave + 1;  // this query's keys
        float m = kLowest;
        for (int j = lane; j < n; j += 64) m = fmaxf(m, row[j]);
        m = wave_max(m);
        for (int j = lane; j < keys; j += 64) row[j] = j < n ? expf_libm(row[j] - m) : 0.0f;
    }
    __syncthreads();
    // Z of the query by one lane, left to right (masked keys add +0)
    if (lane == 0 && wave < nq) {
        float z = 0.0f;
        int j = 0;
        for (; j + 4 <= keys; j += 4) {
            const float4 e4 = *reinterpret_cast<const float4 *>(row + j);
            z = z + e4.x;
            z = z + e4.y;
            z = z + e4.z;
            z = z + e4.w;
        }
        for (; j < keys; ++j) z = z + row[j];
        qs[wave * HEAD] = z;  // q is no longer needed: slot 0 of the row holds Z
    }
    __syncthreads();
    if (wave < nq) {
        const float z = qs[wave * HEAD];
        for (int j = lane; j < keys; j += 64) row[j] = row[j] / z;
    }
    // ---- P.V: thread = (dim d, queries qd, qd + kQS)
    constexpr int kQS = 256 / HEAD;                                  // query phases per dim
    constexpr int kQPT = kXFallbackQ > kQS ? kXFallbackQ / kQS : 1;  // queries per thread
    const int d = tid % HEAD, qd = tid / HEAD;
    float acc[kQPT];
#pragma unroll
    for (int r = 0; r < kQPT; ++r) acc[r] = 0.0f;
    for (int j0 = 0; j0 < keys; j0 += kXKeys) {
        __syncthreads();
        for (int e = tid; e < kXKeys * (HEAD / 8); e += 256) {
            const int j = e / (HEAD / 8), piece = e % (HEAD / 8);
            const int p = min(j0 + j, keys - 1);
            *reinterpret_cast<uint4 *>(kv + j * HEAD + piece * 8) = *reinterpret_cast<const uint4 *>(
                vcache + ((static_cast<size_t>(s) * max_context + p) * kv_heads + kvh) * HEAD + piece * 8);
        }
        __syncthreads();
        const int jn = min(kXKeys, keys - j0);
        for (int jj = 0; jj < jn; jj += 4) {
            float vf[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) vf[u] = gguf_half_to_real(kv[min(jj + u, jn - 1) * HEAD + d]);
#pragma unroll
            for (int r = 0; r < kQPT; ++r) {
                const int qi = qd + kQS * r;
                if (qi >= nq) break;
                const float *w = sc + qi * kcap + j0 + jj;
                if (jj + 4 <= jn) {
                    const float4 w4 = *reinterpret_cast<const float4 *>(w);
                    float a = acc[r];
                    a = a + w4.x * vf[0];
                    a = a + w4.y * vf[1];
                    a = a + w4.z * vf[2];
                    a = a + w4.w * vf[3];
                    acc[r] = a;
                } else {
                    for (int u = 0; u < jn - jj; ++u) acc[r] = acc[r] + w[u] * vf[u];
                }
            }
        }
    }
#pragma unroll
    for (int r = 0; r < kQPT; ++r) {
        const int qi = qd + kQS * r;
        if (qi >= nq) break;
        const size_t row = (static_cast<size_t>(s) * T + q0 + qi) * heads + h;
        const float gate = q[row * 2 * HEAD + HEAD + d];
        out[row * HEAD + d] = acc[r] * sigmoid_ref(gate);
    }
}

// The same arithmetic and orders for prompts whose scores of QB queries fit in
// LDS.  One workgroup of eight waves per (block of QB queries, head,
// sequence).  The sums are chains of separately rounded products, so the
// kernel is bound by vector issue and by the LDS reads beside it, and needs
// many waves to cover the chains' dependent adds: QB is small, so that
// several workgroups share a CU, and each lane owns a few chains whose
// operands it shares in registers.
//   scores: a wave owns 32 keys; its lanes are KG key groups x QB queries
//     with KPL keys each.  No two waves share a key, so a key slice (32 keys x
//     32 dims) sits in a buffer of the wave's own and the waves meet no
//     barrier: a wave's LDS operations are in order.
//   softmax weights: one wave per query, lanes over keys; Z by one lane.
//   P.V: a thread owns DPL dims of one query; values pass through LDS 16
//     keys at a time, double buffered, one barrier per tile.
// Rows past the prompt are zero and never stored; keys are clamped into the
// cache and masked through zero weights.  FINITE (no exponent-31 half in this
// cache): each product fl(a * f32(h)) straight from the fp16 half by
// v_fma_mix_f32.
// Measured (one layer, heads of 256, against one workgroup of 16 queries per
// CU pair with a barrier per key tile up to 512 positions and the kernel
// above past them): 8 heads, 77 positions 57 -> 23 us, 511: 157 -> 67 us,
// 2000: 4,610 -> 589 us; 16 heads, 1024: 2,886 -> 338 us.  At 2000 positions
// its 256 M vector instructions are ~280 us of issue at eight waves per SIMD.
// 64-key wave tiles (more chains per lane, fewer waves busy) 629 us, 16
// queries per workgroup 717 us.
constexpr int kXWaves = 8;
constexpr size_t kXMaxLds = 160 * 1024;  // LDS of a CU
constexpr int kXTileKeys = 32;   // keys per wave tile (scores)
constexpr int kXValueKeys = 16;  // keys per staged value tile
constexpr int kXSliceDims = 32;  // dims of a staged key slice

template <bool FINITE>
__device__ __forceinline__ float times_half(uint32_t h2, bool hi, float a) {
    if constexpr (FINITE) return hi ? half_times<true>(h2, a) : half_times<false>(h2, a);
    return a * gguf_half_to_real(static_cast<uint16_t>(hi ? h2 >> 16 : h2 & 0xffffu));
}

// bytes of LDS before the scores: q and the waves' key slices, or the two value tiles
template <int HEAD, int QB>
constexpr int attention_exact_stage_bytes() {
    constexpr int qk = QB * HEAD * 4 + kXWaves * kXTileKeys * kXSliceDims * 2, v = 2 * kXValueKeys * HEAD * 2;
    return qk > v ? qk : v;
}

template <int HEAD, int QB, bool FINITE>
__device__ __forceinline__ void attention_exact_block(unsigned char *lds_raw, const float *__restrict__ q,
    const uint16_t *__restrict__ kbase, const uint16_t *__restrict__ vbase, float *__restrict__ out, int T, int heads,
    int kv_heads, int h, int s, int q0, int kcap) {
    static_assert(QB == 4 || QB == 8, "one query per wave in the softmax");
    constexpr int KG = 64 / QB, KPL = kXTileKeys / KG;
    constexpr int kSlices = HEAD / kXSliceDims;
    constexpr int kThreads = kXWaves * 64;
    float *qs = reinterpret_cast<float *>(lds_raw);  // [QB][HEAD] normalized q
    const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, wave = tid >> 6;
    uint4 *kb = reinterpret_cast<uint4 *>(lds_raw + QB * HEAD * 4) + wave * (kXTileKeys * kXSliceDims / 8);
    uint16_t *vt = reinterpret_cast<uint16_t *>(lds_raw);  // [2][16][HEAD], after the scores
    float *sc = reinterpret_cast<float *>(lds_raw + attention_exact_stage_bytes<HEAD, QB>());  // [QB][kcap]
    const int nq = min(QB, T - q0);
    const int keys = q0 + nq;  // keys 0..keys-1 cover the block
    const int tiles = (keys + kXTileKeys - 1) / kXTileKeys, kpad = tiles * kXTileKeys;
    const float sqrt_head = sqrtf(static_cast<float>(HEAD));
    const size_t kvstride = static_cast<size_t>(kv_heads) * HEAD;

    // ---- scores
    // key slice piece (lane, n): key lane / 4 + 16 n, dims 8 (lane % 4) .. of the slice; stored at
    // [piece][key ^ 2 piece], so neither the stores nor the reads of 8 consecutive keys meet a bank twice
    u32x4_t kr[2];
    const int pk = lane >> 2, pp = lane & 3;
    auto fetch_k = [&](int t, int sl) {
#pragma unroll
        for (int n = 0; n < 2; ++n)
            kr[n] = *reinterpret_cast<const u32x4_t *>(kbase +
                static_cast<size_t>(min(t * kXTileKeys + pk + 16 * n, keys - 1)) * kvstride + sl * kXSliceDims + pp * 8);
    };
    if (wave < tiles) fetch_k(wave, 0);
    for (int e = tid; e < QB * HEAD / 4; e += kThreads) {
        const int qi = e / (HEAD / 4), d = e % (HEAD / 4);
        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (qi < nq)
            v = reinterpret_cast<const float4 *>(q + ((static_cast<size_t>(s) * T + q0 + qi) * heads + h) * 2 * HEAD)[d];
        reinterpret_cast<float4 *>(qs)[e] = v;
    }
    __syncthreads();
    const int kg = lane % KG, qg = lane / KG;
    for (int t = wave; t < tiles; t += kXWaves) {
        float acc[KPL];
#pragma unroll
        for (int i = 0; i < KPL; ++i) acc[i] = 0.0f;
#pragma unroll 1
        for (int sl = 0; sl < kSlices; ++sl) {
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                const int key = pk + 16 * n;
                *reinterpret_cast<u32x4_t *>(&kb[pp * kXTileKeys + (key ^ (2 * pp))]) = kr[n];
            }
            wave_lds_fence();
            // the next slice (the last fetch of the wave is not used)
            const bool wrap = sl + 1 == kSlices;
            fetch_k(wrap ? min(t + kXWaves, tiles - 1) : t, wrap ? 0 : sl + 1);
#pragma unroll
            for (int pc = 0; pc < kXSliceDims / 8; ++pc) {
                uint32_t kw[KPL][4];
#pragma unroll
                for (int i = 0; i < KPL; ++i) {
                    const uint4 k8 = kb[pc * kXTileKeys + ((kg + KG * i) ^ (2 * pc))];
                    kw[i][0] = k8.x; kw[i][1] = k8.y; kw[i][2] = k8.z; kw[i][3] = k8.w;
                }
                const float4 *qp = reinterpret_cast<const float4 *>(qs + qg * HEAD + sl * kXSliceDims + pc * 8);
                const float4 qa = qp[0], qb = qp[1];
                const float qv[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
                // the lane's chains interleaved (each chain's order unchanged)
#pragma unroll
                for (int k = 0; k < 8; ++k)
#pragma unroll
                    for (int i = 0; i < KPL; ++i)
                        acc[i] = acc[i] + times_half<FINITE>(kw[i][k >> 1], (k & 1) != 0, qv[k]);
            }
            wave_lds_fence();
        }
#pragma unroll
        for (int i = 0; i < KPL; ++i) sc[qg * kcap + t * kXTileKeys + kg + KG * i] = acc[i] / sqrt_head;
    }
    // the first value tile, while the weights are formed
    constexpr int kVPieces = kXValueKeys * HEAD / 8;  // 16-byte pieces of a value tile
    constexpr int kVLoads = (kVPieces + kThreads - 1) / kThreads;
    u32x4_t vr[kVLoads];
    auto fetch_v = [&](int t) {
#pragma unroll
        for (int n = 0; n < kVLoads; ++n) {
            const int e = min(tid + kThreads * n, kVPieces - 1), j = e / (HEAD / 8), piece = e % (HEAD / 8);
            vr[n] = *reinterpret_cast<const u32x4_t *>(vbase +
                static_cast<size_t>(min(t * kXValueKeys + j, keys - 1)) * kvstride + piece * 8);
        }
    };
    fetch_v(0);
    __syncthreads();
    // ---- softmax weights of query `wave`: lanes over keys; e = +0 past the query's keys
    if (wave < QB) {
        constexpr float kLowest = -3.402823466e38f;  // -huge(1.0_real32)
        const int n = min(q0 + wave + 1, keys);
        float *row = sc + wave * kcap;
        float m = kLowest;
        for (int j = lane; j < n; j += 64) m = fmaxf(m, row[j]);
        m = wave_max(m);
        for (int j = lane; j < kpad; j += 64) row[j] = j < n ? expf_libm(row[j] - m) : 0.0f;
        wave_lds_fence();
        // Z left to right (the masked keys add +0), by one lane: the reads of
        // a whole wave would take the other waves' LDS bandwidth
        const float4 *row4 = reinterpret_cast<const float4 *>(row);
        float z = 0.0f;
        for (int j = 0; j < (lane == 0 ? kpad / 4 : 0); j += 8) {  // kpad % 32 == 0
            float4 e4[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) e4[u] = row4[j + u];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                z = z + e4[u].x;
                z = z + e4[u].y;
                z = z + e4[u].z;
                z = z + e4[u].w;
            }
        }
        wave_lds_fence();
        z = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(z)));
        for (int j = lane; j < kpad; j += 64) row[j] = row[j] / z;
    }

    // ---- P.V: thread = DPL dims of one query, keys left to right
    const int vtiles = kpad / kXValueKeys;
    constexpr int kCPT = QB * HEAD / kThreads;  // chains per thread
    constexpr int DPL = kCPT >= 4 ? 4 : (kCPT >= 2 ? 2 : 1);
    constexpr int LPQ = HEAD / DPL;  // threads per query
    const int d0 = (tid % LPQ) * DPL, qi = tid / LPQ;
    const float *wrow = sc + min(qi, QB - 1) * kcap;  // the narrowest blocks leave threads without a query
    float acc[DPL];
#pragma unroll
    for (int d = 0; d < DPL; ++d) acc[d] = 0.0f;
    for (int t = 0; t < vtiles; ++t) {
        uint16_t *tile = vt + (t & 1) * kXValueKeys * HEAD;
#pragma unroll
        for (int n = 0; n < kVLoads; ++n) {
            const int e = tid + kThreads * n;
            if (kVPieces % kThreads == 0 || e < kVPieces) *reinterpret_cast<u32x4_t *>(tile + e * 8) = vr[n];
        }
        // the tile is complete (and, the first time, the weights); the tile before last is consumed
        __syncthreads();
        if (t + 1 < vtiles) fetch_v(t + 1);
#pragma unroll 2
        for (int jj = 0; jj < kXValueKeys; jj += 4) {
            uint32_t vh[4][DPL == 4 ? 2 : 1];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const uint16_t *vp = tile + (jj + u) * HEAD + d0;
                if constexpr (DPL == 4) {
                    const uint2 v2 = *reinterpret_cast<const uint2 *>(vp);
                    vh[u][0] = v2.x; vh[u][1] = v2.y;
                } else if constexpr (DPL == 2) {
                    vh[u][0] = *reinterpret_cast<const uint32_t *>(vp);
                } else {
                    vh[u][0] = *vp;
                }
            }
            const float4 w = *reinterpret_cast<const float4 *>(wrow + t * kXValueKeys + jj);
            const float w4[4] = {w.x, w.y, w.z, w.w};
            // the thread's chains interleaved key by key (each chain's order unchanged)
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int d = 0; d < DPL; ++d)
                    acc[d] = acc[d] + times_half<FINITE>(vh[u][d >> 1], (d & 1) != 0, w4[u]);
        }
    }
    if (qi >= nq) return;
    const size_t row = (static_cast<size_t>(s) * T + q0 + qi) * heads + h;
#pragma unroll
    for (int d = 0; d < DPL; ++d) {
        const float gate = q[row * 2 * HEAD + HEAD + d0 + d];
        out[row * HEAD + d0 + d] = acc[d] * sigmoid_ref(gate);
    }
}

// blockIdx: x head, y sequence, z query block, the longest first (their keys
// take the most time, so the last workgroups to start are the short ones)
template <int HEAD, int QB>
__global__ __launch_bounds__(kXWaves * 64, 4) void attention_prefill_exact_tiled_kernel(const float *__restrict__ q,
    const uint16_t *__restrict__ kcache, const uint16_t *__restrict__ vcache, const int *__restrict__ flags,
    float *__restrict__ out, int T, int heads, int kv_heads, int max_context, int kcap) {
    static_assert(HEAD % 64 == 0 && HEAD <= 256, "head 64, 128 or 256");
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int h = static_cast<int>(blockIdx.x), s = static_cast<int>(blockIdx.y);
    const int q0 = static_cast<int>(gridDim.z - 1 - blockIdx.z) * QB;
    const int kvh = h / (heads / kv_heads);
    const size_t first = (static_cast<size_t>(s) * max_context * kv_heads + kvh) * HEAD;
    if (flags[static_cast<size_t>(s) * kv_heads + kvh] == 0)
        attention_exact_block<HEAD, QB, true>(lds_raw, q, kcache + first, vcache + first, out, T, heads, kv_heads, h, s, q0, kcap);
    else
        attention_exact_block<HEAD, QB, false>(lds_raw, q, kcache + first, vcache + first, out, T, heads, kv_heads, h, s, q0, kcap);
}

// Causal attention of every prompt token (fortai_qwen35_cpu.f90:1006-1033
// with an online softmax): one workgroup per (query block of 64, head,
// sequence); four threads per query, each with a quarter of the head dims;
// keys and values staged through LDS 32 positions at a time.  out =
// softmax(q k / sqrt(head)) v * sigmoid(gate).
constexpr int kQBlock = 64;
constexpr int kKTile = 32;

template <int HEAD>
__global__ __launch_bounds__(256) void attention_prefill_kernel(const float *__restrict__ q,
    const uint16_t *__restrict__ kcache, const uint16_t *__restrict__ vcache, const int *__restrict__ flags,
    int only_flagged, float *__restrict__ out, int T, int heads, int kv_heads, int max_context) {
    constexpr int kPart = HEAD / 4;
    constexpr int kPartPitch = kPart + 4;  // the four quarters of a row on different banks
    __shared__ __align__(16) float kt[kKTile][4 * kPartPitch];
    __shared__ __align__(16) float vt[kKTile][4 * kPartPitch];
    const int tid = static_cast<int>(threadIdx.x);
    const int qi = tid >> 2, part = tid & 3;
    const int h = static_cast<int>(blockIdx.y), s = static_cast<int>(blockIdx.z);
    const int q0 = static_cast<int>(blockIdx.x) * kQBlock;
    const int t = min(q0 + qi, T - 1);
    const int kvh = h / (heads / kv_heads);
    // after the matrix-core kernel: only the (sequence, kv head) pairs whose
    // cache holds exponent-31 halves, which that kernel leaves to this one
    if (only_flagged && flags[static_cast<size_t>(s) * kv_heads + kvh] == 0) return;
    const float *qrow = q + ((static_cast<size_t>(s) * T + t) * heads + h) * 2 * HEAD;
    float qv[kPart], o[kPart];
#pragma unroll
    for (int d = 0; d < kPart; ++d) {
        qv[d] = qrow[part * kPart + d];
        o[d] = 0.0f;
    }
    const float scale = 1.0f / sqrtf(static_cast<float>(HEAD));
    float m = -__builtin_inff(), z = 0.0f;
    const int last = min(q0 + kQBlock, T) - 1;  // keys 0..last cover the block
    for (int j0 = 0; j0 <= last; j0 += kKTile) {
        __syncthreads();
        for (int e = tid; e < kKTile * HEAD; e += 256) {
            const int j = e / HEAD, d = e % HEAD;
            const int p = min(j0 + j, last);
            const size_t off = ((static_cast<size_t>(s) * max_context + p) * kv_heads + kvh) * HEAD + d;
            const int dd = (d / kPart) * kPartPitch + d % kPart;
            kt[j][dd] = gguf_half_to_real(kcache[off]);
            vt[j][dd] = gguf_half_to_real(vcache[off]);
        }
        __syncthreads();
        const int jn = min(kKTile, t - j0 + 1);  // keys of this query in the tile
        for (int j = 0; j < kKTile; ++j) {
            float sc = 0.0f;
#pragma unroll
            for (int d = 0; d < kPart; ++d) sc = __builtin_fmaf(qv[d], kt[j][part * kPartPitch + d], sc);
            sc += __shfl_xor(sc, 1);
            sc += __shfl_xor(sc, 2);
            if (j >= jn) continue;  // masked (uniform per query: the 4 threads agree)
            sc *= scale;
            // online softmax; the running sums are rescaled only when the
            // maximum grows (within the fp32 tolerance of this path)
            if (sc > m) {
                const float corr = __expf(m - sc);
                z *= corr;
#pragma unroll
                for (int d = 0; d < kPart; ++d) o[d] *= corr;
                m = sc;
            }
            const float p = __expf(sc - m);
            z += p;
#pragma unroll
            for (int d = 0; d < kPart; ++d) o[d] = __builtin_fmaf(p, vt[j][part * kPartPitch + d], o[d]);
        }
    }
    if (q0 + qi >= T) return;
    const float *gate = qrow + HEAD;
    float *orow = out + ((static_cast<size_t>(s) * T + t) * heads + h) * HEAD;
#pragma unroll
    for (int d = 0; d < kPart; ++d) {
        const int dd = part * kPart + d;
        orow[dd] = (o[d] / z) * sigmoid_ref(gate[dd]);
    }
}

// The same causal attention on the fp16 matrix cores (the default prefill
// mode, within its tolerance): one workgroup per (32-query block, kv head,
// sequence), wave w taking q head kvh * group + w.  Per 32-key tile,
//   S^T = K Q^T  (v_mfma_f32_32x32x16_f16, keys x queries, q pre-scaled by
//                 1/sqrt(head) and rounded to fp16; K is the fp16 cache),
// an online softmax in fp32 (__expf; the running sums rescaled when a
// query's reference maximum moves, which it does only by jumps of more than
// 8), and
//   O^T += V^T P^T (the same instruction, dims x queries, P rounded to fp16).
// The accumulator of a 32x32 MFMA holds, in element i of lane l, row
// 8*(i/4) + 4*(l/32) + i%4 and column l%32: with keys and dims as rows and
// queries as columns, every value of a query stays in lanes l%32 == query,
// so the softmax rescale is a per-lane scalar, and the 16 probabilities of a
// lane are the B operand of the two P.V instructions of the tile as they are
// (A and B present the same keys in the same slots; which k the instruction
// assigns to a slot does not change the sum).  K reaches LDS key-major (the
// A operand of S^T: 16 bytes of one key per lane), V dim-major (the A operand
// of O^T: two 8-byte runs of keys per lane).  A (sequence, kv head) whose
// cache holds exponent-31 halves is left to attention_prefill_kernel.
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));
constexpr int kMfmaQ = 32;  // queries per workgroup (one MFMA column block)
constexpr int kMfmaK = 32;  // keys per tile

template <int HEAD>
__global__ __launch_bounds__(256) void attention_prefill_mfma_kernel(const float *__restrict__ q,
    const uint16_t *__restrict__ kcache, const uint16_t *__restrict__ vcache, const int *__restrict__ flags,
    float *__restrict__ out, int T, int heads, int kv_heads, int max_context) {
    static_assert(HEAD % 64 == 0, "whole 16-byte pieces per thread and tile");
    constexpr int kKPitch = HEAD + 8;             // halves per K row (key-major)
    constexpr int kVPitch = kMfmaK + 8;           // halves per V^T row (dim-major)
    constexpr int kSteps = HEAD / 16;             // k-steps of S^T
    constexpr int kDT = HEAD / 32;                // 32-dim tiles of O^T
    constexpr int kPieces = HEAD / 8;             // 16-byte pieces of a key row
    constexpr int kLoads = kMfmaK * kPieces / 256;  // pieces per thread and tile (K and V each)
    extern __shared__ __align__(16) _Float16 mfma_lds[];
    _Float16 *kt = mfma_lds;                                   // [kMfmaK][kKPitch]
    _Float16 *vt = kt + kMfmaK * kKPitch;                      // [HEAD][kVPitch]
    _Float16 *qs = vt + HEAD * kVPitch;                        // [4 waves][kMfmaQ][kKPitch]
    const int tid = static_cast<int>(threadIdx.x), wave = tid >> 6, lane = tid & 63;
    const int col = lane & 31, g = lane >> 5;
    const int kvh = static_cast<int>(blockIdx.y), s = static_cast<int>(blockIdx.z);
    const int q0 = static_cast<int>(blockIdx.x) * kMfmaQ;
    if (flags[static_cast<size_t>(s) * kv_heads + kvh] != 0) return;
    const int group = heads / kv_heads;
    const bool active = wave < group;
    const int h = kvh * group + (active ? wave : 0);
    const int qq = q0 + col;                       // this lane's query
    const int qt = min(qq, T - 1);
    const float *qrow = q + ((static_cast<size_t>(s) * T + qt) * heads + h) * 2 * HEAD;
    // the wave's 32 query rows, scaled by 1/sqrt(head), in fp16 (the B
    // operand of S^T, read from LDS each tile): lane l writes dims
    // 4 * (l % kPieces4) .. of rows l / kPieces4, l / kPieces4 + 64 / kPieces4, ...
    _Float16 *qw = qs + wave * kMfmaQ * kKPitch;
    {
        const float scale = 1.0f / sqrtf(static_cast<float>(HEAD));
        constexpr int kPieces4 = HEAD / 4;  // float4 pieces of a q row
        for (int e = lane; e < kMfmaQ * kPieces4; e += 64) {
            const int r = e / kPieces4, c4 = e % kPieces4;
            const int t = min(q0 + r, T - 1);
            const float4 a = *reinterpret_cast<const float4 *>(
                q + ((static_cast<size_t>(s) * T + t) * heads + h) * 2 * HEAD + c4 * 4);
            const half4_t v = {static_cast<_Float16>(a.x * scale), static_cast<_Float16>(a.y * scale),
                static_cast<_Float16>(a.z * scale), static_cast<_Float16>(a.w * scale)};
            *reinterpret_cast<half4_t *>(qw + r * kKPitch + c4 * 4) = v;
        }
    }
    const int last = min(q0 + kMfmaQ, T) - 1;      // keys 0..last cover the block
    const int ntiles = last / kMfmaK + 1;
    u32x4_t kr[kLoads], vr[kLoads];
    // K pieces key-major (consecutive lanes: consecutive 16 bytes of a key
    // row); V pieces key-minor (consecutive lanes: consecutive keys), so that
    // each transposed 2-byte LDS store of a wave covers 32 consecutive keys
    // of one dim row (no bank conflicts)
    auto fetch = [&](int j0) {
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const int li = tid + 256 * j;
            const int kkey = li / kPieces, kpc = li % kPieces;
            const int vkey = li % kMfmaK, vpc = li / kMfmaK;
            const size_t base = (static_cast<size_t>(s) * max_context) * kv_heads + kvh;
            kr[j] = *reinterpret_cast<const u32x4_t *>(
                kcache + (base + static_cast<size_t>(min(j0 + kkey, last)) * kv_heads) * HEAD + kpc * 8);
            vr[j] = *reinterpret_cast<const u32x4_t *>(
                vcache + (base + static_cast<size_t>(min(j0 + vkey, last)) * kv_heads) * HEAD + vpc * 8);
        }
    };
    auto stash = [&]() {
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const int li = tid + 256 * j;
            const int kkey = li / kPieces, kpc = li % kPieces;
            const int vkey = li % kMfmaK, vpc = li / kMfmaK;
            *reinterpret_cast<u32x4_t *>(kt + kkey * kKPitch + kpc * 8) = kr[j];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                vt[(vpc * 8 + 2 * e) * kVPitch + vkey] = __builtin_bit_cast(_Float16, static_cast<uint16_t>(vr[j][e] & 0xffffu));
                vt[(vpc * 8 + 2 * e + 1) * kVPitch + vkey] = __builtin_bit_cast(_Float16, static_cast<uint16_t>(vr[j][e] >> 16));
            }
        }
    };
    float16_t o[kDT];
#pragma unroll
    for (int dt = 0; dt < kDT; ++dt) o[dt] = float16_t{};
    float m = -__builtin_inff(), zl = 0.0f;
    fetch(0);
    for (int t = 0; t < ntiles; ++t) {
        const int j0 = t * kMfmaK;
        __syncthreads();  // every wave is done with the previous tile
        stash();
        __syncthreads();
        if (t + 1 < ntiles) fetch(j0 + kMfmaK);
        if (!active) continue;
        float16_t sc = float16_t{};
#pragma unroll
        for (int kk = 0; kk < kSteps; ++kk) {
            const half8_t a = *reinterpret_cast<const half8_t *>(kt + col * kKPitch + kk * 16 + g * 8);
            const half8_t b = *reinterpret_cast<const half8_t *>(qw + col * kKPitch + kk * 16 + g * 8);
            sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, sc, 0, 0, 0);
        }
        // element i: key j0 + 8 * (i / 4) + 4 * g + i % 4 of query qq
        float tmax = -__builtin_inff();
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int key = j0 + 8 * (i / 4) + 4 * g + (i % 4);
            if (key > qq || key >= T) sc[i] = -__builtin_inff();
            tmax = fmaxf(tmax, sc[i]);
        }
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
        // the reference maximum m of a query moves only when a score exceeds
        // it by more than 8 (probabilities stay <= e^8, well inside fp16), so
        // the sums are rescaled on few tiles: the first, and big jumps
        const bool grow = tmax > m + 8.0f;
        if (__any(grow)) {
            const float mnew = grow ? tmax : m;
            const float corr = __expf(m - mnew);  // 0 on the first tile (m = -inf), 1 where m stays
            m = mnew;
            zl *= corr;
#pragma unroll
            for (int dt = 0; dt < kDT; ++dt)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[dt][i] *= corr;
        }
        // the denominator sums the same fp16-rounded probabilities the P.V
        // products use, so numerator and denominator round alike
        float pl[16];
        float zt = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            pl[i] = sc[i] == -__builtin_inff() ? 0.0f : __expf(sc[i] - m);
            zt += static_cast<float>(static_cast<_Float16>(pl[i]));
        }
        zl += zt;
        const half8_t pb0 = {static_cast<_Float16>(pl[0]), static_cast<_Float16>(pl[1]), static_cast<_Float16>(pl[2]),
            static_cast<_Float16>(pl[3]), static_cast<_Float16>(pl[4]), static_cast<_Float16>(pl[5]),
            static_cast<_Float16>(pl[6]), static_cast<_Float16>(pl[7])};
        const half8_t pb1 = {static_cast<_Float16>(pl[8]), static_cast<_Float16>(pl[9]), static_cast<_Float16>(pl[10]),
            static_cast<_Float16>(pl[11]), static_cast<_Float16>(pl[12]), static_cast<_Float16>(pl[13]),
            static_cast<_Float16>(pl[14]), static_cast<_Float16>(pl[15])};
#pragma unroll
        for (int dt = 0; dt < kDT; ++dt) {
            const _Float16 *vrow = vt + (dt * 32 + col) * kVPitch + 4 * g;
            const half4_t v0 = *reinterpret_cast<const half4_t *>(vrow);
            const half4_t v1 = *reinterpret_cast<const half4_t *>(vrow + 8);
            const half4_t v2 = *reinterpret_cast<const half4_t *>(vrow + 16);
            const half4_t v3 = *reinterpret_cast<const half4_t *>(vrow + 24);
            const half8_t va0 = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
            const half8_t va1 = {v2[0], v2[1], v2[2], v2[3], v3[0], v3[1], v3[2], v3[3]};
            o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va0, pb0, o[dt], 0, 0, 0);
            o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va1, pb1, o[dt], 0, 0, 0);
        }
    }
    if (!active || qq >= T) return;
    // the gate: 1 / (1 + e^-g) with the hardware exp and reciprocal (this
    // mode's tolerance; the exact mode's kernel uses the reference sigmoid),
    // and one reciprocal of Z per query
    const float zi = __builtin_amdgcn_rcpf(zl + __shfl_xor(zl, 32));
    const float *gate = qrow + HEAD;
    float *orow = out + ((static_cast<size_t>(s) * T + qq) * heads + h) * HEAD;
    auto sig = [](float x) { return __builtin_amdgcn_rcpf(1.0f + __expf(-x)); };
#pragma unroll
    for (int dt = 0; dt < kDT; ++dt) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int d = dt * 32 + 8 * r + 4 * g;
            const float4 gt = *reinterpret_cast<const float4 *>(gate + d);
            float4 v;
            v.x = (o[dt][4 * r + 0] * zi) * sig(gt.x);
            v.y = (o[dt][4 * r + 1] * zi) * sig(gt.y);
            v.z = (o[dt][4 * r + 2] * zi) * sig(gt.z);
            v.w = (o[dt][4 * r + 3] * zi) * sig(gt.w);
            *reinterpret_cast<float4 *>(orow + d) = v;
        }
    }
}

// Rows [r0, r0 + count) of X8 -> the matvec's Q8L layout [count][q8l_bytes]
// (the same quantized values: used by the exact prefill mode).
__global__ __launch_bounds__(256) void x8_to_q8l_kernel(const int8_t *__restrict__ xq, const float *__restrict__ xs,
    int ld, int chunks, int r0, uint32_t *__restrict__ q8l) {
    const int rr = static_cast<int>(blockIdx.y), n = r0 + rr;
    uint32_t *dst = q8l + static_cast<size_t>(rr) * chunks * 36;
    for (int e = static_cast<int>(threadIdx.x); e < chunks * 36; e += 256) {
        if (e < chunks * 32) {
            dst[e] = reinterpret_cast<const uint32_t *>(xq + (static_cast<size_t>(e >> 5) * ld + n) * 128)[e & 31];
        } else {
            const int b = e - chunks * 32;
            reinterpret_cast<float *>(dst)[e] = xs[(static_cast<size_t>(b >> 2) * ld + n) * 4 + (b & 3)];
        }
    }
}

void x8_planes(void *x8, int tokens, int width, int8_t *&xq, float *&xs, int &ld, int &blocks_pad) {
    ld = q8_tokens_ld(tokens);
    blocks_pad = (width / kQ8Block + 3) / 4 * 4;
    xq = static_cast<int8_t *>(x8);
    xs = reinterpret_cast<float *>(xq + static_cast<size_t>(ld) * blocks_pad * 32);
}

}  // namespace

hipError_t launch_x8_to_q8l(const void *x8, int tokens, int width, int r0, int count, void *q8l, hipStream_t stream) {
    if (r0 < 0 || count < 1 || r0 + count > tokens || width % kQ8Block) return hipErrorInvalidValue;
    int8_t *xq; float *xs; int ld, bp;
    x8_planes(const_cast<void *>(x8), tokens, width, xq, xs, ld, bp);
    hipLaunchKernelGGL(x8_to_q8l_kernel, dim3(1, count), dim3(256), 0, stream, xq, xs, ld, bp / 4, r0,
        static_cast<uint32_t *>(q8l));
    note_launch("x8_to_q8l_kernel grid 1x%d", count);
    return hipGetLastError();
}

hipError_t launch_rms_quantize_tokens(const float *x, int rows, int width, const float *norm, float eps, void *x8,
    hipStream_t stream) {
    if (rows <= 0 || width <= 0 || width % kQ8Block) return hipErrorInvalidValue;
    int8_t *xq; float *xs; int ld, bp;
    x8_planes(x8, rows, width, xq, xs, ld, bp);
    hipLaunchKernelGGL(rms_quantize_tokens_kernel, dim3(rows), dim3(kRowThreads), 0, stream, x, width, width, norm, eps,
        ld, bp, xq, xs);
    note_launch("rms_quantize_tokens_kernel<%s> grid %d", norm ? "rmsnorm" : "f32", rows);
    return hipGetLastError();
}

hipError_t launch_gated_quantize_tokens(const float *o, const float *z, const float *norm, float eps, int rows,
    int width, int head, void *x8, hipStream_t stream) {
    const int hl = head / 4;
    if (rows <= 0 || width % kQ8Block || head % 4 || hl > 64 || (hl & (hl - 1)) || width % head) return hipErrorInvalidValue;
    int8_t *xq; float *xs; int ld, bp;
    x8_planes(x8, rows, width, xq, xs, ld, bp);
    hipLaunchKernelGGL(gated_quantize_tokens_kernel, dim3(rows), dim3(kRowThreads), 0, stream, o, z, norm, eps, width,
        head, ld, bp, xq, xs);
    note_launch("gated_quantize_tokens_kernel grid %d", rows);
    return hipGetLastError();
}

hipError_t launch_silu_product_quantize(const float *gate, const float *up, int rows, int width, void *x8,
    hipStream_t stream) {
    if (rows <= 0 || width % kQ8Block) return hipErrorInvalidValue;
    int8_t *xq; float *xs; int ld, bp;
    x8_planes(x8, rows, width, xq, xs, ld, bp);
    hipLaunchKernelGGL(silu_product_quantize_kernel, dim3(rows), dim3(kRowThreads), 0, stream, gate, up, width, ld, bp,
        xq, xs);
    note_launch("silu_product_quantize_kernel grid %d", rows);
    return hipGetLastError();
}

hipError_t launch_conv_silu_tokens(const float *x, const float *conv_w, float *conv_state, float *out, int batch, int T,
    int C, int K, hipStream_t stream) {
    if (batch < 1 || T < 1 || C < 1 || K < 2 || K > kConvMax) return hipErrorInvalidValue;
    const int cb = (C + 255) / 256, tb = (T + kConvTokens - 1) / kConvTokens;
    hipLaunchKernelGGL(conv_silu_tokens_kernel, dim3(cb, tb, batch), dim3(256), 0, stream, x, conv_w, conv_state, out,
        T, C, K);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(conv_state_advance_kernel, dim3(cb, batch), dim3(256), 0, stream, x, conv_state, T, C, K);
    note_launch("conv_silu_tokens_kernel grid %dx%dx%d + conv_state_advance_kernel grid %dx%d", cb, tb, batch, cb, batch);
    return hipGetLastError();
}

hipError_t launch_gdn_prefill(const GdnParams &p, int batch, int T, float *qinv, float *kinv, float *beta_t,
    float *decay_t, hipStream_t stream) {
    if (batch < 1 || T < 1 || p.key_heads <= 0 || p.value_heads % p.key_heads || p.state_size != p.head)
        return hipErrorInvalidValue;
    const int C = 2 * p.state_size * p.key_heads + p.value_heads * p.head;
    const int rows = batch * T;
    hipLaunchKernelGGL(gdn_token_prep_kernel, dim3(rows), dim3(256), 0, stream, p.qkv, p.alpha, p.beta, p.ssm_a,
        p.ssm_dt, C, p.key_heads, p.value_heads, p.head, p.state_size, p.eps, qinv, kinv, beta_t, decay_t);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const dim3 grid(p.value_heads * (p.head / 8), batch);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(64), 0, stream, p.qkv, qinv, kinv, beta_t, decay_t, p.state, p.out, T, C,
            p.key_heads, p.value_heads, p.state_size);
    };
    if (p.head == 64) go(gdn_prefill_kernel<64>);
    else if (p.head == 128) go(gdn_prefill_kernel<128>);
    else return hipErrorInvalidValue;
    note_launch("gdn_token_prep_kernel grid %d + gdn_prefill_kernel<%d> grid %dx%d", rows, p.head, grid.x, batch);
    return hipGetLastError();
}

hipError_t launch_attention_prefill(const AttentionParams &p, int batch, int T, float *out, hipStream_t stream,
    bool matrix_cores) {
    // every head width a kernel below is instantiated for; checked before
    // anything is enqueued, so an unsupported layer launches nothing
    if (batch < 1 || T < 1 || T > p.max_context || p.heads % p.kv_heads || p.head != p.value ||
        p.rope_dim > p.head || (p.head != 64 && p.head != 128 && p.head != 256))
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(qk_rope_append_kernel, dim3(batch * T), dim3(256), 0, stream, const_cast<float *>(p.q), p.k,
        p.v, p.q_norm, p.k_norm, p.rope, p.kcache, p.vcache, p.cache_flags, T, p.heads, p.kv_heads, p.head, p.value,
        p.rope_dim, p.max_context, p.eps);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    // the matrix-core kernel: head 64, 128 or 256, a GQA group of <= 4
    // (one wave per q head); it leaves the flagged (sequence, kv head) pairs
    // to the fp32 kernel below
    const bool mfma = matrix_cores && p.heads / p.kv_heads <= 4;
    if (mfma) {
        const dim3 mgrid((T + kMfmaQ - 1) / kMfmaQ, p.kv_heads, batch);
        // K tile, V^T tile and four waves' q rows, fp16
        const size_t mlds = static_cast<size_t>(kMfmaK * (p.head + 8) + p.head * (kMfmaK + 8) + 4 * kMfmaQ * (p.head + 8)) *
            sizeof(_Float16);
        switch (p.head) {
        case 64:
            hipLaunchKernelGGL(attention_prefill_mfma_kernel<64>, mgrid, dim3(256), mlds, stream, p.q, p.kcache, p.vcache,
                p.cache_flags, out, T, p.heads, p.kv_heads, p.max_context);
            break;
        case 128:
            hipLaunchKernelGGL(attention_prefill_mfma_kernel<128>, mgrid, dim3(256), mlds, stream, p.q, p.kcache,
                p.vcache, p.cache_flags, out, T, p.heads, p.kv_heads, p.max_context);
            break;
        case 256:
            hipLaunchKernelGGL(attention_prefill_mfma_kernel<256>, mgrid, dim3(256), mlds, stream, p.q, p.kcache,
                p.vcache, p.cache_flags, out, T, p.heads, p.kv_heads, p.max_context);
            break;
        }
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (!matrix_cores) {
        // Four queries per workgroup while two workgroups fit on a CU (head
        // 256: up to 3840 positions), eight while one fits (4352), four again
        // (8960), then the kernel with global tiles and one to two queries.
        // Head 256, 8 heads, QB 4 / 8: 511 positions 66 / 75 us, 2000: 586 /
        // 807 us, 4100: 3,949 / 3,157 us.
        const int kcap = (T + kXTileKeys - 1) / kXTileKeys * kXTileKeys;
        int tiled = 0;
        auto tiled_with = [&](auto qb_c, size_t lds_limit) {
            constexpr int QB = decltype(qb_c)::value;
            auto go = [&](auto head_c) {
                constexpr int H = decltype(head_c)::value;
                const size_t lds = static_cast<size_t>(attention_exact_stage_bytes<H, QB>()) + static_cast<size_t>(QB) * kcap * 4;
                if (lds > lds_limit) return;
                hipLaunchKernelGGL((attention_prefill_exact_tiled_kernel<H, QB>), dim3(p.heads, batch, (T + QB - 1) / QB),
                    dim3(kXWaves * 64), lds, stream, p.q, p.kcache, p.vcache, p.cache_flags, out, T, p.heads, p.kv_heads,
                    p.max_context, kcap);
                tiled = QB;
            };
            if (p.head == 64) go(std::integral_constant<int, 64>{});
            else if (p.head == 128) go(std::integral_constant<int, 128>{});
            else go(std::integral_constant<int, 256>{});
        };
        tiled_with(std::integral_constant<int, 4>{}, kXMaxLds / 2);
        if (!tiled) tiled_with(std::integral_constant<int, 8>{}, kXMaxLds);
        if (!tiled) tiled_with(std::integral_constant<int, 4>{}, kXMaxLds);
        if (tiled) {
            note_launch("qk_rope_append_kernel grid %d + attention_prefill_exact_tiled_kernel<%d, %d> grid %dx%dx%d",
                batch * T, p.head, tiled, p.heads, batch, (T + tiled - 1) / tiled);
            return hipGetLastError();
        }
        // longer prompts: queries per workgroup so that the block's scores fit in LDS
        const int kcap4 = (T + 3) / 4 * 4;
        int qb = kXFallbackQ;
        auto lds_of = [&](int b) {
            return static_cast<size_t>(b) * p.head * 4 + static_cast<size_t>(kXKeys) * p.head * 2 +
                static_cast<size_t>(b) * kcap4 * 4;
        };
        if (lds_of(qb) > 150 * 1024) qb = 1;
        if (lds_of(qb) > 150 * 1024) return hipErrorInvalidValue;
        const dim3 xgrid((T + qb - 1) / qb, p.heads, batch);
        switch (p.head) {
        case 64:
            hipLaunchKernelGGL(attention_prefill_exact_kernel<64>, xgrid, dim3(256), lds_of(qb), stream, p.q, p.kcache,
                p.vcache, out, T, p.heads, p.kv_heads, p.max_context, qb, kcap4);
            break;
        case 128:
            hipLaunchKernelGGL(attention_prefill_exact_kernel<128>, xgrid, dim3(256), lds_of(qb), stream, p.q, p.kcache,
                p.vcache, out, T, p.heads, p.kv_heads, p.max_context, qb, kcap4);
            break;
        case 256:
            hipLaunchKernelGGL(attention_prefill_exact_kernel<256>, xgrid, dim3(256), lds_of(qb), stream, p.q, p.kcache,
                p.vcache, out, T, p.heads, p.kv_heads, p.max_context, qb, kcap4);
            break;
        default: return hipErrorInvalidValue;
        }
        note_launch("qk_rope_append_kernel grid %d + attention_prefill_exact_kernel<%d> grid %dx%dx%d", batch * T, p.head,
            xgrid.x, xgrid.y, xgrid.z);
        return hipGetLastError();
    }
    const int only_flagged = mfma ? 1 : 0;
    const dim3 grid((T + kQBlock - 1) / kQBlock, p.heads, batch);
    switch (p.head) {
    case 64:
        hipLaunchKernelGGL(attention_prefill_kernel<64>, grid, dim3(256), 0, stream, p.q, p.kcache, p.vcache,
            p.cache_flags, only_flagged, out, T, p.heads, p.kv_heads, p.max_context);
        break;
    case 128:
        hipLaunchKernelGGL(attention_prefill_kernel<128>, grid, dim3(256), 0, stream, p.q, p.kcache, p.vcache,
            p.cache_flags, only_flagged, out, T, p.heads, p.kv_heads, p.max_context);
        break;
    case 256:
        hipLaunchKernelGGL(attention_prefill_kernel<256>, grid, dim3(256), 0, stream, p.q, p.kcache, p.vcache,
            p.cache_flags, only_flagged, out, T, p.heads, p.kv_heads, p.max_context);
        break;
    default: return hipErrorInvalidValue;
    }
    if (mfma)
        note_launch("qk_rope_append_kernel grid %d + attention_prefill_mfma_kernel<%d> grid %dx%dx%d + "
            "attention_prefill_kernel<%d> (exponent-31 caches only) grid %dx%dx%d", batch * T, p.head,
            (T + kMfmaQ - 1) / kMfmaQ, p.kv_heads, batch, p.head, grid.x, grid.y, grid.z);
    else
        note_launch("qk_rope_append_kernel grid %d + attention_prefill_kernel<%d> grid %dx%dx%d", batch * T, p.head,
            grid.x, grid.y, grid.z);
    return hipGetLastError();
}

}  // namespace fortai_hip
