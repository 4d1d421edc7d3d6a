// hai_deltanet_prefill.hip -- Gated DeltaNet over prompt chunks (the
// prefill's deltanet_grouped_conv_kernel + deltanet_recurrent_kernel,
// hip_kernels.hip:871-912, 985-1095, and the gated RMSNorm), tolerance mode.
//
// The recurrence per token (v-head h; normalised key k_t, scaled query q_t,
// decay a_t, beta_t; S [dk][dv] fp32):
//   S_t = a_t S_{t-1} + beta_t k_t (v_t - a_t S_{t-1}^T k_t)^T,  o_t = S_t^T q_t.
// Walked token by token it is a chain of dependent dot products (~0.8 us
// per token and layer at the 27B shape).  Here the tokens go in chunks of
// kChunk and the recurrence is restated per chunk -- the chunkwise form of
// the gated delta rule (Yang, Kautz and Hatamizadeh, "Gated Delta Networks",
// 2024): with g_t = sum_{u<=t} log a_u inside the chunk, S the state before
// it, L[t][s] = beta_t e^{g_t - g_s} k_t.k_s (s < t) and w_t the value token
// t writes (S_t = a_t S_{t-1} + k_t w_t^T),
//   (I + L) w = diag(beta) V - diag(beta e^g) K S,   so   w = U - W^ S  with
//   U = (I + L)^-1 diag(beta) V,   W^ = (I + L)^-1 diag(beta e^g) K;
//   o_t = e^{g_t} S^T q_t + sum_{s<=t} e^{g_t - g_s} (q_t.k_s) w_s;
//   S'  = e^{g_last} S + sum_s e^{g_last - g_s} k_s w_s^T.
// Everything but the last two lines is independent of S, so the work splits
// into three launches:
//   1. deltanet_chunk_prep_kernel, one block per (chunk, head, sequence), all
//      chunks at once: conv + SiLU of the chunk's inputs, gates, the Gram
//      matrices and with them the q / k norms (matrix cores), the 32 x 32
//      triangular inverse, U and W^ as products with it, and the scaled keys /
//      queries K~ = e^{g_last - g} K, Q~ = e^{g} Q and P[t][s] =
//      e^{g_t - g_s} q_t.k_s into a per-chunk record, W^ / K~ / Q~ / P already
//      split into bf16 pairs in the operand order of the next pass;
//   2. deltanet_chunk_state_kernel, one or two blocks per (head, sequence),
//      the chunks in order: W = U - W^ S, O = Q~ S + P W, S = e^{g_last} S +
//      K~^T W -- dense products on the matrix cores with the state held in
//      their accumulators, each record copied global -> LDS one chunk ahead by
//      waves of their own;
//   3. deltanet_gated_norm_ring_kernel: the gated RMSNorm per (token, head)
//      and the conv ring's last entries (two launches where the rows are not
//      16-byte aligned).
// The state is stored once, to slot (L + T) % nslots.  The sums are
// reassociated (and the gates use the hardware exp), so results equal the
// canonical recurrence to fp32 rounding, not bit for bit.
#include "hai_common.h"
#include "hai_device.h"
#include "hai_gemm_common.h"

#include <atomic>

namespace {

using namespace hai;

constexpr int kChunk = 32;   // tokens per chunk
constexpr int kMaxKc = 8;

struct PrefillArgs {
    float* o_ws;            // [B*T][nv*dv] unrounded outputs
    float* chunks;          // per (sequence, head, chunk): chunk_floats<DK, DV>() floats
    const uint16_t* proj;   // rows b*T + t: [qkv | z | a | b] at the offsets
    int64_t ld_proj, off_qkv, off_a, off_b;
    const uint16_t* conv_w;
    uint16_t* ring;
    int ring_n, nslots;
    float* state;
    const uint16_t *a_log, *dt_bias;
    const int32_t* lens;
    int pos_add;
    int B, T, nk, nv, Kc;
};

// Per-chunk record: U [C][DV], W^ [C][DK], K~ [C][DK], Q~ [C][DK], P [C][C],
// then e^{g_last} (padded to 16 floats).
template <int DK, int DV>
__host__ __device__ constexpr int64_t chunk_floats() {
    return static_cast<int64_t>(kChunk) * (DV + 3 * DK + kChunk) + 16;
}

// tolerance mode: the hardware exp and reciprocal
__device__ __forceinline__ float fast_silu(float x) { return x * __builtin_amdgcn_rcpf(1.0f + __expf(-x)); }

// ---- matrix-core operands (v_mfma_f32_32x32x16_bf16) ----
typedef __bf16 dn_bf16x8 __attribute__((ext_vector_type(8)));
typedef float dn_f32x16 __attribute__((ext_vector_type(16)));

// Position in a 16-k step of the operand slot q (0..7) of lane half lh: the
// k index 16s + op_slot(lh, q) of step s sits in k-slot 8 lh + q.  Elements
// 8s .. 8s + 7 of a lane's 32x32 result tile hold rows 16s + op_slot(lh, q),
// so a result tile is the B operand of the next product as it stands.
__host__ __device__ constexpr int op_slot(int lh, int q) { return 4 * lh + (q & 3) + 8 * (q >> 2); }

// Operand tables: per 16-k step (or tile block) blk, the 64 lanes' 8 bf16 of
// the high parts, then of the low parts (x = hi + lo, hi = bf16(x),
// lo = bf16(x - hi)).
__device__ __forceinline__ void dn_split8(const float (&x)[8], u32x4& hi, u32x4& lo) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint32_t hp = f2bf2(x[2 * q], x[2 * q + 1]);
        hi[q] = hp;
        lo[q] = f2bf2(x[2 * q] - lo_bf(hp), x[2 * q + 1] - hi_bf(hp));
    }
}
// x as three bf16 (largest first): the fp32 value whole
__device__ __forceinline__ void dn_split8x3(const float (&x)[8], u32x4 (&p)[3]) {
    float r[8];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        p[0][q] = f2bf2(x[2 * q], x[2 * q + 1]);
        r[2 * q] = x[2 * q] - lo_bf(p[0][q]);
        r[2 * q + 1] = x[2 * q + 1] - hi_bf(p[0][q]);
    }
    dn_split8(r, p[1], p[2]);
}
// elements off .. off + 7 of an accumulator tile, split the same way
__device__ __forceinline__ void dn_split8(const dn_f32x16& x, int off, u32x4& hi, u32x4& lo) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint32_t hp = f2bf2(x[off + 2 * q], x[off + 2 * q + 1]);
        hi[q] = hp;
        lo[q] = f2bf2(x[off + 2 * q] - lo_bf(hp), x[off + 2 * q + 1] - hi_bf(hp));
    }
}
__device__ __forceinline__ dn_f32x16 dn_mfma(u32x4 a, u32x4 b, dn_f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(dn_bf16x8, a), __builtin_bit_cast(dn_bf16x8, b),
                                                   c, 0, 0, 0);
}

// ---- pass 1: one block (4 waves) per (chunk c, head h, sequence b); KC: the
// conv taps (0: any count up to kMaxKc, read from the arguments) ----
// The conv outputs are bf16-exact, so q, k and v stay in LDS as bf16 and
// every scale (norms, decays, beta) is applied to a product's other side or
// its result: the Gram products K K^T, K Q^T and the diagonal of Q Q^T (which
// give the norms too) take one matrix instruction per step, and U and W^ come
// from the 32 x 32 inverse T = (I + L)^-1, found by forward substitution (one
// wave, lane = column), as
//   U = (T diag(beta)) V,   W^ = (T diag(beta e^g |k|^-1)) K
// with T's factor split into three bf16 (all 24 bits: K and V are bf16, so the
// products are those of fp32 factors; a pair leaves 2^-18 in U.  MI355X, the
// whole call, pair / three: 1000 tokens of 48 heads 117.1 / 117.4 us, 32 x 512
// 1067 / 1076).  Each product is oriented so that
// its result tile is the operand table the next pass wants: P from K Q^T and
// W^ from K^T T^T (lane = token, elements = tokens / keys in op_slot order).
// Columns of K and V come out of their rows through the transposing LDS reads.
// Bound by the records it writes (70 KB each) and a chain of four barrier-
// separated phases; MI355X, 1000 tokens of 48 heads: 57 -> 38 us (all scales
// applied to fp32 copies, U and W^ by 256 substitutions of 496 FMAs).
__device__ __forceinline__ uint2 dn_read_tr(const uint16_t* lds) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(
        uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)lds));
}
// Eight values of a lane's operand slots from an fp32 row: base + op_slot(lh, .)
__device__ __forceinline__ void dn_slots8(const float* base, int lh, float (&x)[8]) {
    const float4 a = *reinterpret_cast<const float4*>(base + 4 * lh);
    const float4 b = *reinterpret_cast<const float4*>(base + 4 * lh + 8);
    x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
    x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
}
// eight bf16 (two pairs of words) times eight factors, split and stored as
// block blk of an operand table
__device__ __forceinline__ void dn_store_split(uint32_t* tab, int blk, int lane, const float (&x)[8]) {
    u32x4 hi, lo;
    dn_split8(x, hi, lo);
    *reinterpret_cast<u32x4*>(tab + blk * 512 + lane * 4) = hi;
    *reinterpret_cast<u32x4*>(tab + blk * 512 + 256 + lane * 4) = lo;
}
__device__ __forceinline__ void dn_unpack8(uint2 a, uint2 b, float (&x)[8]) {
    x[0] = lo_bf(a.x); x[1] = hi_bf(a.x); x[2] = lo_bf(a.y); x[3] = hi_bf(a.y);
    x[4] = lo_bf(b.x); x[5] = hi_bf(b.x); x[6] = lo_bf(b.y); x[7] = hi_bf(b.y);
}

template <int DK, int DV, int KC>
__global__ __launch_bounds__(256) void deltanet_chunk_prep_kernel(PrefillArgs A) {
    constexpr int KM = KC > 0 ? KC : kMaxKc;  // tap registers
    constexpr int NT = 256;
    constexpr int NW = NT / 64;
    constexpr int QP = DK + 8, VP = DV + 8;  // padded LDS rows (16 bytes: row reads spread over banks)
    constexpr int NCH = 2 * DK + DV;
    __shared__ __align__(16) uint16_t qs[kChunk][QP];
    __shared__ __align__(16) uint16_t ks[kChunk][QP];
    __shared__ __align__(16) uint16_t vs[kChunk][VP];
    __shared__ __align__(16) float Lm[kChunk][kChunk + 4];  // rows read as float4
    __shared__ __align__(16) float Ti[kChunk][kChunk + 4];
    __shared__ __align__(16) float s_g[kChunk], s_beta[kChunk], s_q[kChunk], s_k[kChunk], s_ek[kChunk],
        s_eq[kChunk];

    const int c = blockIdx.x;
    const int h = blockIdx.y;
    const int b = blockIdx.z;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int nv = A.nv;
    const int gq = h / (nv / A.nk);
    const int64_t kw = static_cast<int64_t>(A.nk) * DK;
    const int64_t vw = static_cast<int64_t>(nv) * DV;
    const int64_t C = 2 * kw + vw;
    const int Kc = KC > 0 ? KC : A.Kc;
    const int hist = Kc - 1;
    const int T = A.T;
    const int t0 = c * kChunk;
    const int TS = min(kChunk, T - t0);
    const int64_t row0 = static_cast<int64_t>(b) * T;
    const int64_t p0 = static_cast<int64_t>(A.lens ? A.lens[b] : 0) + A.pos_add;

    // ---- gate inputs (last wave, lane = token), requested first ----
    float a_in = 0.0f, b_in = 0.0f, dt_b = 0.0f, a_lg = 0.0f;
    if (wave == NW - 1 && lane < TS) {
        a_in = bf2f(A.proj[(row0 + t0 + lane) * A.ld_proj + A.off_a + h]);
        b_in = bf2f(A.proj[(row0 + t0 + lane) * A.ld_proj + A.off_b + h]);
        dt_b = bf2f(A.dt_bias[h]);
        a_lg = bf2f(A.a_log[h]);
    }
    // ---- conv + SiLU: thread p < NCH / 2 takes the channel pair 2p, 2p + 1
    // (within one of q, k, v: their widths are even); input at prompt-chunk
    // row t0 + tt - hist + i, rows before the prompt chunk from the conv ring
    // (positions before 0: zero).  Every load is issued before the first use.
    constexpr int NP = NCH / 2;
    static_assert(NCH % 2 == 0 && NP <= NT - 64, "channel pairs leave the last wave to the gates");
    if (tid < NP) {
        const int ch = 2 * tid;
        int64_t chan;
        if (ch < DK) chan = static_cast<int64_t>(gq) * DK + ch;
        else if (ch < 2 * DK) chan = kw + static_cast<int64_t>(gq) * DK + (ch - DK);
        else chan = 2 * kw + static_cast<int64_t>(h) * DV + (ch - 2 * DK);
        float wc0[KM], wc1[KM];
#pragma unroll
        for (int i = 0; i < KM; ++i) {
            wc0[i] = i < Kc ? bf2f(A.conv_w[chan * Kc + i]) : 0.0f;
            wc1[i] = i < Kc ? bf2f(A.conv_w[(chan + 1) * Kc + i]) : 0.0f;
        }
        auto pair_at = [&](const uint16_t* p) { return *reinterpret_cast<const uint32_t*>(p); };
        uint32_t win[KM];  // the last Kc - 1 input pairs, oldest first
#pragma unroll
        for (int i = 0; i < KM; ++i) {
            uint32_t v = 0;
            if (i < hist) {
                const int r = t0 - hist + i;
                if (r >= 0) v = pair_at(A.proj + (row0 + r) * A.ld_proj + A.off_qkv + chan);
                else if (p0 + r >= 0)
                    v = pair_at(A.ring + (static_cast<int64_t>(b) * A.ring_n + (p0 + r) % A.ring_n) * C + chan);
            }
            win[i] = v;
        }
        uint32_t xr[kChunk];
#pragma unroll
        for (int tt = 0; tt < kChunk; ++tt)
            xr[tt] = tt < TS ? pair_at(A.proj + (row0 + t0 + tt) * A.ld_proj + A.off_qkv + chan) : 0u;
        uint16_t* col = ch < DK ? &qs[0][ch] : ch < 2 * DK ? &ks[0][ch - DK] : &vs[0][ch - 2 * DK];
        const int pitch = ch < 2 * DK ? QP : VP;
#pragma unroll
        for (int tt = 0; tt < kChunk; ++tt) {
            const uint32_t xin = xr[tt];
            float acc0 = lo_bf(hist > 0 ? win[0] : xin) * wc0[0];
            float acc1 = hi_bf(hist > 0 ? win[0] : xin) * wc1[0];
#pragma unroll
            for (int i = 1; i < KM; ++i) {
                if (i < hist) {
                    acc0 = fma_(lo_bf(win[i]), wc0[i], acc0);
                    acc1 = fma_(hi_bf(win[i]), wc1[i], acc1);
                } else if (i == hist) {
                    acc0 = fma_(lo_bf(xin), wc0[i], acc0);
                    acc1 = fma_(hi_bf(xin), wc1[i], acc1);
                }
            }
#pragma unroll
            for (int i = 0; i + 1 < KM; ++i)
                if (i + 1 < hist) win[i] = win[i + 1];
#pragma unroll
            for (int i = 0; i < KM; ++i)
                if (i == hist - 1) win[i] = xin;
            // rows past the chunk's tokens are zero: they take no part
            *reinterpret_cast<uint32_t*>(col + tt * pitch) = tt < TS ? f2bf2(fast_silu(acc0), fast_silu(acc1)) : 0u;
        }
    }
    // ---- gates: log of the decay exp(-exp(A_log) softplus(dt_bias + a)),
    // beta = sigmoid(b), the decay's running sum g (a scan over the lanes) ----
    if (wave == NW - 1) {
        float lg = 0.0f, be = 0.0f;
        if (lane < TS) {
            const float dtv = dt_b + a_in;
            const float sp = fmaxf(dtv, 0.0f) + log1pf(__expf(-fabsf(dtv)));
            lg = -(__expf(a_lg) * sp);
            be = __builtin_amdgcn_rcpf(1.0f + __expf(-b_in));
        }
        float g = lg;
#pragma unroll
        for (int o = 1; o < kChunk; o <<= 1) {
            const float v = __shfl_up(g, o);
            if (lane >= o) g += v;
        }
        const float glast = __shfl(g, kChunk - 1);
        if (lane < kChunk) {
            s_g[lane] = g;
            s_beta[lane] = be;
            s_ek[lane] = __expf(glast - g);
            s_eq[lane] = __expf(g);
        }
    }
    __syncthreads();

    const int lc = lane & 31, lh = lane >> 5, li = lane & 15;
    float* rec = A.chunks + ((static_cast<int64_t>(b) * nv + h) * ((T + kChunk - 1) / kChunk) + c) * chunk_floats<DK, DV>();
    float* rU = rec;
    uint32_t* rW = reinterpret_cast<uint32_t*>(rU + kChunk * DV);
    uint32_t* rK = rW + kChunk * DK;
    uint32_t* rQ = rK + kChunk * DK;
    uint32_t* rP = rQ + kChunk * DK;
    auto row_of = [&](int i) { return 8 * (i >> 2) + 4 * lh + (i & 3); };

    // ---- Gram products over d in 16-wide k steps (slot q of lane l: d = 16
    // step + 8 (l / 32) + q): wave 0 K K^T, wave 1 K Q^T, wave 2 Q Q^T; element
    // i of lane l: row 8 (i / 4) + 4 (l / 32) + i % 4, column l % 32 ----
    dn_f32x16 G;
#pragma unroll
    for (int i = 0; i < 16; ++i) G[i] = 0.0f;
    if (wave < 3) {
        const uint16_t* ar = (wave == 2 ? qs[lc] : ks[lc]) + 8 * lh;
        const uint16_t* br = (wave == 0 ? ks[lc] : qs[lc]) + 8 * lh;
#pragma unroll
        for (int kst = 0; kst < DK / 16; ++kst)
            G = dn_mfma(*reinterpret_cast<const u32x4*>(ar + 16 * kst), *reinterpret_cast<const u32x4*>(br + 16 * kst),
                        G);
        if (wave != 1) {  // the diagonal: squared norms
            float n2 = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; ++i)
                if (row_of(i) == lc) n2 = G[i];
            if (((lc >> 2) & 1) == lh) {
                const float inv = 1.0f / csqrt(n2 + 1.0e-6f);
                if (wave == 0) s_k[lc] = inv;
                else s_q[lc] = inv * (1.0f / csqrt(static_cast<float>(DK)));
            }
        }
    }
    __syncthreads();

    if (wave == 0) {
        // ---- L[t][s] = beta_t e^{g_t - g_s} k_t.k_s (s < t), then T = (I + L)^-1: lane = column ----
        const float gs = s_g[lc], ks_s = s_k[lc];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int t = row_of(i);
            Lm[t][lc] = lc < t && t < TS ? s_beta[t] * __expf(s_g[t] - gs) * (s_k[t] * ks_s * G[i]) : 0.0f;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        float x[kChunk];
#pragma unroll
        for (int t = 0; t < kChunk; ++t) {
            // four partial sums (s = u mod 4) shorten the dependent chain
            float part[4] = {t == lc ? 1.0f : 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s4 = 0; s4 < t; s4 += 4) {
                const float4 l4 = *reinterpret_cast<const float4*>(&Lm[t][s4]);
                const float lv[4] = {l4.x, l4.y, l4.z, l4.w};
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (s4 + u < t) part[u] = fma_(-lv[u], x[s4 + u], part[u]);
            }
            x[t] = (part[0] + part[1]) + (part[2] + part[3]);
        }
        if (lh == 0) {
#pragma unroll
            for (int t = 0; t < kChunk; ++t) Ti[t][lc] = x[t];
        }
    } else {
        if (wave == 1) {
            // ---- P[t][s] = e^{g_t - g_s} q_t.k_s (s <= t): lane = token t, elements = tokens s ----
            const float gt = s_g[lc], qt = s_q[lc];
            float x[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int s = row_of(i);
                x[i] = s <= lc && lc < TS ? __expf(gt - s_g[s]) * (qt * s_k[s] * G[i]) : 0.0f;
            }
            dn_store_split(rP, 0, lane, *reinterpret_cast<const float(*)[8]>(x));
            dn_store_split(rP, 1, lane, *reinterpret_cast<const float(*)[8]>(x + 8));
            if (lane == 0) rP[kChunk * kChunk] = __float_as_uint(s_eq[kChunk - 1]);
        }
        // ---- Q~ = e^{g} Q and K~ = e^{g_last - g} K, split, in operand order: a block per turn ----
        for (int task = wave - 1; task < DK / 8; task += NW - 1) {
            float x[8];
            if (task < DK / 16) {  // Q~ (A of Q~ S): token t, keys 16 blk + op_slot
                const uint16_t* row = &qs[lc][16 * task + 4 * lh];
                dn_unpack8(*reinterpret_cast<const uint2*>(row), *reinterpret_cast<const uint2*>(row + 8), x);
                const float f = s_eq[lc] * s_q[lc];
#pragma unroll
                for (int q = 0; q < 8; ++q) x[q] *= f;
                dn_store_split(rQ, task, lane, x);
            } else {  // K~ (A of K~^T w): key 32 m + lane % 32, tokens 16 st + op_slot
                const int blk = task - DK / 16, m = blk >> 1, st = blk & 1;
                const uint16_t* at = &ks[16 * st + 4 * lh + (li >> 2)][32 * m + (lane & 16) + 4 * (li & 3)];
                dn_unpack8(dn_read_tr(at), dn_read_tr(at + 8 * QP), x);
                float e[8], k[8];
                dn_slots8(s_ek + 16 * st, lh, e);
                dn_slots8(s_k + 16 * st, lh, k);
#pragma unroll
                for (int q = 0; q < 8; ++q) x[q] *= e[q] * k[q];
                dn_store_split(rK, blk, lane, x);
            }
        }
    }
    __syncthreads();

    // ---- U = (T beta) V and W^T = K^T (T beta e^g |k|^-1)^T, 32 columns / keys per turn ----
    for (int task = wave; task < (DV + DK) / 32; task += NW) {
        const bool isv = task < DV / 32;
        const int col0 = 32 * (isv ? task : task - DV / 32);
        dn_f32x16 R;
#pragma unroll
        for (int i = 0; i < 16; ++i) R[i] = 0.0f;
#pragma unroll
        for (int st = 0; st < 2; ++st) {  // tokens 16 st + op_slot
            float t8[8], f[8];
            dn_slots8(&Ti[lc][16 * st], lh, t8);
            dn_slots8(s_beta + 16 * st, lh, f);
            if (!isv) {
                float e[8], k[8];
                dn_slots8(s_eq + 16 * st, lh, e);
                dn_slots8(s_k + 16 * st, lh, k);
#pragma unroll
                for (int q = 0; q < 8; ++q) f[q] *= e[q] * k[q];
            }
#pragma unroll
            for (int q = 0; q < 8; ++q) t8[q] *= f[q];
            u32x4 t3[3];
            dn_split8x3(t8, t3);
            const int r = 16 * st + 4 * lh + (li >> 2), cc = col0 + (lane & 16) + 4 * (li & 3);
            const uint16_t* at = isv ? &vs[r][cc] : &ks[r][cc];
            const uint2 a = dn_read_tr(at), b2 = dn_read_tr(at + 8 * (isv ? VP : QP));
            const u32x4 xb = u32x4{a.x, a.y, b2.x, b2.y};
#pragma unroll
            for (int e = 2; e >= 0; --e) R = isv ? dn_mfma(t3[e], xb, R) : dn_mfma(xb, t3[e], R);
        }
        if (isv) {  // row = token, column = value column
#pragma unroll
            for (int i = 0; i < 16; ++i) rU[row_of(i) * DV + col0 + lc] = R[i];
        } else {  // row = key, column = token: W^ (A of W^ S) as it stands
            float x[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) x[i] = R[i];
            dn_store_split(rW, col0 / 16, lane, *reinterpret_cast<const float(*)[8]>(x));
            dn_store_split(rW, col0 / 16 + 1, lane, *reinterpret_cast<const float(*)[8]>(x + 8));
        }
    }
}

// ---- pass 2 on the matrix cores: one block per (head h, sequence b), one
// wave per 32 value columns, the chunks in order ----
// The state columns of a wave are DK/32 accumulator tiles of
// v_mfma_f32_32x32x16_bf16: tile m, lane l, element i holds
// S[32m + 8(i/4) + 4(l/32) + i%4][j0 + l%32], so elements 8s .. 8s + 7 of a
// tile are the B operand of the 16-k step over keys 32m + 16s + op_slot(.):
// W^ S and Q~ S take S straight from the accumulators, and w = U - W^ S comes
// out in the layout that makes it, in turn, the B operand of P w and K~^T w.
// The A operands (W^, Q~, K~, P) are written by pass 1 in exactly that order,
// split into bf16 pairs; every fp32 product is hi.hi + hi.lo + lo.hi (the
// small terms first), within ~2^-16 of it.
// A block holds NWB such waves (all DV / 32 of a head, or half of them when
// the heads leave CUs idle) and as many waves that only copy: records reach
// LDS by global -> LDS copies (no registers) a chunk ahead into the other of
// two buffers: the operand tables, the U columns of the block's waves, and
// e^{g_last}.  Requested by the computing waves themselves, the 30 copies a
// wave and chunk held up their matrix instructions for 0.4 us.  The copies
// are inline assembly, so that the compiler does not wait for them before
// unrelated LDS reads.
//
// Bound by the serial chain over the chunks: 78 MFMAs per wave and chunk
// (2500 cycles of its SIMD's matrix core), so the products are ordered as
// independent chains: W^ S and Q~ S by the parity of the 16-k step (four
// chains), then K~^T w per state tile with P w between them.  MI355X, 1000
// tokens of 48 heads: 112 -> 75 us (2.3 us a chunk; the 390 VALU
// instructions of the splits do not hide behind the products of the one wave
// a SIMD holds; forcing them between the products changed nothing).
template <int DK, int DV, int NWB>
struct StateShape {
    static constexpr int RW = 3 * kChunk * DK + kChunk * kChunk;  // operand words of a record
    static constexpr int OP_COPIES = RW * 4 / 1024;               // 1 KB copies of the operand tables
    static constexpr int U_COPIES = 4 * NWB;                      // 1 KB copies of the block's U columns
    static constexpr int BUF = RW * 4 + U_COPIES * 1024 + 256;    // bytes; the last part: e^{g_last}
    static constexpr size_t LDS_BYTES = 2 * static_cast<size_t>(BUF);
    static_assert(RW * 4 % (1024 * NWB) == 0, "whole copies per copying wave");
};

// One global -> LDS copy per lane of 16 (4) bytes at base + off, to lds + 16 (4) * lane;
// the M0 write needs one wait state before the copy.
__device__ __forceinline__ void dn_copy16(uint32_t off, const void* base, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(off), "s"(base), "s"(lds)
                 : "memory");
}
__device__ __forceinline__ void dn_copy4(uint32_t off, const void* base, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
                 :
                 : "v"(off), "s"(base), "s"(lds)
                 : "memory");
}

template <int DK, int DV, int NWB>
__global__ __launch_bounds__(128 * NWB, 2) void deltanet_chunk_state_kernel(PrefillArgs A) {
    using SH = StateShape<DK, DV, NWB>;
    constexpr int MT = DK / 32;  // state tiles per wave
    static_assert(DK % 32 == 0 && DV % (32 * NWB) == 0 && kChunk == 32, "state pass tiles");
    extern __shared__ __align__(16) unsigned char recs[];  // [2][BUF]

    const int h = blockIdx.x;
    const int b = blockIdx.z;
    const int lane = threadIdx.x & 63;
    const int w = wave_index() % NWB;
    const int jb = 32 * NWB * blockIdx.y;  // the block's first value column
    const int j0 = jb + 32 * w;
    const int lc = lane & 31;
    const int lh = lane >> 5;
    const int nv = A.nv;
    const int T = A.T;
    const int nchunks = (T + kChunk - 1) / kChunk;
    const int64_t vw = static_cast<int64_t>(nv) * DV;
    const int64_t row0 = static_cast<int64_t>(b) * T;
    const int64_t p0 = static_cast<int64_t>(A.lens ? A.lens[b] : 0) + A.pos_add;
    auto row_of = [&](int i) { return 8 * (i >> 2) + 4 * lh + (i & 3); };
    // column-tiled head: key i = q4*(DK/4) + 4m + e of column j at float ((m*DV + j)*4 + q4)*4 + e
    auto tiled = [&](int key, int col) {
        const int q4 = key / (DK / 4), m = (key % (DK / 4)) / 4, ee = key % 4;
        return ((static_cast<int64_t>(m) * DV + col) * 4 + q4) * 4 + ee;
    };
    const float* recs0 = A.chunks + (static_cast<int64_t>(b) * nv + h) * nchunks * chunk_floats<DK, DV>();
    const uint32_t lds0 = static_cast<uint32_t>(
        reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)recs));
    if (wave_index() >= NWB) {  // a copying wave
        constexpr int kOps = SH::OP_COPIES / NWB, kUs = SH::U_COPIES / NWB;
        constexpr int LPR = 8 * NWB;  // lanes per U row
        const uint32_t uoff = static_cast<uint32_t>((lane / LPR) * DV + (lane % LPR) * 4) * 4u;
        for (int c = 0; c < nchunks; ++c) {
            const float* rec = recs0 + static_cast<int64_t>(c) * chunk_floats<DK, DV>();
            const uint32_t dst = lds0 + (c & 1) * SH::BUF;
            // operand tables: KB i NWB + w; U: 8 / NWB rows of the block's columns per KB
            const char* op = reinterpret_cast<const char*>(rec + kChunk * DV) + w * 1024;
#pragma unroll
            for (int i = 0; i < kOps; ++i) dn_copy16(lane * 16, op + i * NWB * 1024, dst + (i * NWB + w) * 1024);
            const float* u = rec + static_cast<int64_t>(w) * (64 / LPR) * DV + jb;
#pragma unroll
            for (int i = 0; i < kUs; ++i)
                dn_copy16(uoff, u + static_cast<int64_t>(i) * NWB * (64 / LPR) * DV,
                          dst + SH::RW * 4 + (i * NWB + w) * 1024);
            if (w == 0)
                dn_copy4((lane & 15) * 4, rec + kChunk * DV + SH::RW, dst + SH::RW * 4 + SH::U_COPIES * 1024);
            wait_vmcnt<0>();
            lds_barrier();  // chunk c is staged; chunk c - 1's buffer, which chunk c + 1 takes, is free
        }
        return;
    }

    const float* hs = A.state + ((p0 % A.nslots) * A.B + b) * static_cast<int64_t>(nv) * DV * DK +
                      static_cast<int64_t>(h) * DV * DK;
    dn_f32x16 S[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < 16; ++i) S[m][i] = hs[tiled(32 * m + row_of(i), j0 + lc)];

    for (int c = 0; c < nchunks; ++c) {
        const int t0 = c * kChunk;
        const int TS = min(kChunk, T - t0);
        const int cur = c & 1;
        lds_barrier();  // this chunk is staged; the reads of the other buffer are done
        const unsigned char* rb = recs + cur * SH::BUF;
        const u32x4* opW = reinterpret_cast<const u32x4*>(rb) + lane;
        const u32x4* opK = opW + kChunk * DK / 4;
        const u32x4* opQ = opK + kChunk * DK / 4;
        const u32x4* opP = opQ + kChunk * DK / 4;
        const float* rU = reinterpret_cast<const float*>(rb + SH::RW * 4) + 32 * w + lc;
        // ---- W^ S and Q~ S (row t = lane % 32 of the A operands): state tile m is the two k steps 2m, 2m + 1,
        // a chain of its own for each step's parity and product; the next tile's operands are read ahead of this
        // tile's products ----
        dn_f32x16 Wa[2], Oa[2];
#pragma unroll
        for (int i = 0; i < 16; ++i) Wa[0][i] = Wa[1][i] = Oa[0][i] = Oa[1][i] = 0.0f;
        u32x4 ow[2][4], oq[2][4];  // [buffer][step hi, lo, next step hi, lo]
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            ow[0][e] = opW[e * 64];
            oq[0][e] = opQ[e * 64];
        }
        const float gl = *reinterpret_cast<const float*>(rb + SH::RW * 4 + SH::U_COPIES * 1024);
        float u[16];
        u32x4 kh[MT], kl[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            if (m + 1 < MT) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    ow[(m + 1) & 1][e] = opW[(4 * (m + 1) + e) * 64];
                    oq[(m + 1) & 1][e] = opQ[(4 * (m + 1) + e) * 64];
                }
            } else {
#pragma unroll
                for (int i = 0; i < 16; ++i) u[i] = rU[row_of(i) * 32 * NWB];
#pragma unroll
                for (int k = 0; k < MT; ++k) {
                    kh[k] = opK[(4 * k) * 64];
                    kl[k] = opK[(4 * k + 1) * 64];
                }
            }
            u32x4 sh[2], sl[2];
            dn_split8(S[m], 0, sh[0], sl[0]);
            dn_split8(S[m], 8, sh[1], sl[1]);
#pragma unroll
            for (int t = 0; t < 3; ++t)
#pragma unroll
                for (int e = 0; e < 2; ++e) {  // lo.hi, hi.lo, hi.hi of both steps and products
                    const u32x4 sb = t == 1 ? sl[e] : sh[e];
                    Wa[e] = dn_mfma(ow[m & 1][2 * e + (t == 0)], sb, Wa[e]);
                    Oa[e] = dn_mfma(oq[m & 1][2 * e + (t == 0)], sb, Oa[e]);
                }
#pragma unroll
            for (int i = 0; i < 16; ++i) S[m][i] *= gl;
        }
        // ---- w = U - W^ S ----
#pragma unroll
        for (int i = 0; i < 16; ++i) u[i] = u[i] - (Wa[0][i] + Wa[1][i]);
        u32x4 wh[2], wl[2];
        dn_split8(*reinterpret_cast<const float(*)[8]>(u), wh[0], wl[0]);
        dn_split8(*reinterpret_cast<const float(*)[8]>(u + 8), wh[1], wl[1]);
        // ---- S = e^{g_last} S + K~^T w (row = key 32m + lane % 32, k = tokens) and O = Q~ S + P w ----
#pragma unroll
        for (int st = 0; st < 2; ++st) {
            const u32x4 ph = opP[(2 * st) * 64], pl = opP[(2 * st + 1) * 64];
            if (st == 1) {
#pragma unroll
                for (int k = 0; k < MT; ++k) {
                    kh[k] = opK[(4 * k + 2) * 64];
                    kl[k] = opK[(4 * k + 3) * 64];
                }
            }
#pragma unroll
            for (int m = 0; m < MT; ++m) S[m] = dn_mfma(kl[m], wh[st], S[m]);
            Oa[st] = dn_mfma(pl, wh[st], Oa[st]);
#pragma unroll
            for (int m = 0; m < MT; ++m) S[m] = dn_mfma(kh[m], wl[st], S[m]);
            Oa[st] = dn_mfma(ph, wl[st], Oa[st]);
#pragma unroll
            for (int m = 0; m < MT; ++m) S[m] = dn_mfma(kh[m], wh[st], S[m]);
            Oa[st] = dn_mfma(ph, wh[st], Oa[st]);
        }
        float* orow = A.o_ws + (row0 + t0) * vw + static_cast<int64_t>(h) * DV + j0 + lc;
        if (TS == kChunk) {
#pragma unroll
            for (int i = 0; i < 16; ++i) orow[row_of(i) * vw] = Oa[0][i] + Oa[1][i];
        } else {
#pragma unroll
            for (int i = 0; i < 16; ++i)
                if (row_of(i) < TS) orow[row_of(i) * vw] = Oa[0][i] + Oa[1][i];
        }
    }
    float* hd = A.state + (((p0 + T) % A.nslots) * A.B + b) * static_cast<int64_t>(nv) * DV * DK +
                static_cast<int64_t>(h) * DV * DK;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < 16; ++i) hd[tiled(32 * m + row_of(i), j0 + lc)] = S[m][i];
}

// The conv ring's entries for the chunk's last Kc - 1 positions (the only
// ones a later step reads), after every block has read the entries before
// the chunk: a chunk of T = ring_n tokens maps its last positions onto the
// same entries.  grid (ceil(C / 256), Kc - 1, B).
__global__ __launch_bounds__(256) void deltanet_ring_update_kernel(uint16_t* __restrict__ ring, int ring_n,
                                                                   const uint16_t* __restrict__ proj,
                                                                   int64_t ld_proj, int64_t off_qkv, int64_t C,
                                                                   const int32_t* lens, int pos_add, int T, int hist) {
    const int64_t c = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int i = blockIdx.y;
    const int b = blockIdx.z;
    const int r = T - hist + i;
    if (c >= C || r < 0) return;  // a position before the chunk: the ring has it already
    const int64_t p = static_cast<int64_t>(lens ? lens[b] : 0) + pos_add + r;
    ring[(static_cast<int64_t>(b) * ring_n + p % ring_n) * C + c] = proj[(static_cast<int64_t>(b) * T + r) * ld_proj + off_qkv + c];
}

// Gated RMSNorm of the outputs: one wave per (row, head); rms of the
// unrounded output, then bf16(((bf16(o) * rms) * w) * silu(z)) (the verify
// kernel's epilogue, silu within 2^-21 of it).
template <int DV>
__global__ __launch_bounds__(256) void deltanet_gated_norm_kernel(uint16_t* __restrict__ out, int64_t ld_out,
                                                                  const float* __restrict__ o_ws,
                                                                  const uint16_t* __restrict__ proj, int64_t ld_proj,
                                                                  int64_t off_z, const uint16_t* __restrict__ norm_w,
                                                                  int64_t rows, int nv, float eps) {
    constexpr int PER = DV / 64;
    const int lane = threadIdx.x & 63;
    const int64_t task = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (task >= rows * nv) return;
    const int64_t row = task / nv;
    const int h = static_cast<int>(task % nv);
    const float* o = o_ws + (row * nv + h) * DV;
    const float ss = l64_sumsq_f32(o, DV, lane);
    const float rms = 1.0f / csqrt(ss / static_cast<float>(DV) + eps);
#pragma unroll
    for (int r = 0; r < PER; ++r) {
        const int jo = lane + 64 * r;
        const float z = bf2f(proj[row * ld_proj + off_z + static_cast<int64_t>(h) * DV + jo]);
        out[row * ld_out + static_cast<int64_t>(h) * DV + jo] = f2bf(((bfr(o[jo]) * rms) * bf2f(norm_w[jo])) * hw_silu(z));
    }
}

// Both of the above in one launch with 16-byte accesses: the first nblocks
// blocks take 256 / (DV / 8) head rows each (DV / 8 lanes a row), the rest the
// ring's entries as dword pairs.  Needs 16-byte aligned rows of out, proj's z
// columns and the norm weight; the same sums and gate as the two-byte form, bit
// for bit.  Bound by memory (o in fp32, z, out); MI355X, 1000 tokens of 48 heads:
// 20.4 + 4.6 -> 9.6 us (two bytes per lane, canonical exp and IEEE division in
// the gate, which here would take 4.5 us more).
template <int DV>
__global__ __launch_bounds__(256) void deltanet_gated_norm_ring_kernel(
    uint16_t* __restrict__ out, int64_t ld_out, const float* __restrict__ o_ws, const uint16_t* __restrict__ proj,
    int64_t ld_proj, int64_t off_z, const uint16_t* __restrict__ norm_w, int64_t rows, int nv, float eps, int nblocks,
    uint16_t* __restrict__ ring, int ring_n, int64_t off_qkv, int64_t C, const int32_t* lens, int pos_add, int T,
    int hist, int B) {
    constexpr int LPR = DV / 8;
    if (static_cast<int>(blockIdx.x) >= nblocks) {
        const int64_t e = (static_cast<int64_t>(blockIdx.x) - nblocks) * 256 + threadIdx.x;  // pair of channels
        const int64_t half = C / 2;
        const int64_t c = e % half * 2;
        const int i = static_cast<int>(e / half % hist);
        const int64_t b = e / half / hist;
        const int r = T - hist + i;
        if (b >= B || r < 0) return;  // (a position before the chunk: the ring has it already)
        const int64_t p = static_cast<int64_t>(lens ? lens[b] : 0) + pos_add + r;
        *reinterpret_cast<uint32_t*>(ring + (b * ring_n + p % ring_n) * C + c) =
            *reinterpret_cast<const uint32_t*>(proj + (b * T + r) * ld_proj + off_qkv + c);
        return;
    }
    const int64_t task = static_cast<int64_t>(blockIdx.x) * (256 / LPR) + threadIdx.x / LPR;
    if (task >= rows * nv) return;
    const int j0 = static_cast<int>(threadIdx.x % LPR) * 8;
    const int64_t row = task / nv;
    const int h = static_cast<int>(task % nv);
    const float4 o0 = *reinterpret_cast<const float4*>(o_ws + task * DV + j0);
    const float4 o1 = *reinterpret_cast<const float4*>(o_ws + task * DV + j0 + 4);
    const u32x4 z = *reinterpret_cast<const u32x4*>(proj + row * ld_proj + off_z + static_cast<int64_t>(h) * DV + j0);
    const u32x4 nw = *reinterpret_cast<const u32x4*>(norm_w + j0);
    const float o[8] = {o0.x, o0.y, o0.z, o0.w, o1.x, o1.y, o1.z, o1.w};
    float ss = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) ss = fma_(o[e], o[e], ss);
#pragma unroll
    for (int s = LPR / 2; s >= 1; s >>= 1) ss = ss + __shfl_xor(ss, s);
    const float rms = 1.0f / csqrt(ss / static_cast<float>(DV) + eps);
    uint32_t y[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
        y[q] = f2bf2(((bfr(o[2 * q]) * rms) * lo_bf(nw[q])) * hw_silu(lo_bf(z[q])),
                     ((bfr(o[2 * q + 1]) * rms) * hi_bf(nw[q])) * hw_silu(hi_bf(z[q])));
    *reinterpret_cast<u32x4*>(out + row * ld_out + static_cast<int64_t>(h) * DV + j0) = u32x4{y[0], y[1], y[2], y[3]};
}

// Compute units of the current device (one GPU model per process).
int64_t device_cus() {
    static std::atomic<int> cached{0};
    const int known = cached.load(std::memory_order_relaxed);
    if (known > 0) return known;
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && cus > 0) {
        cached.store(cus, std::memory_order_relaxed);
        return cus;
    }
    return 256;  // MI355X
}

// Whether the address ranges of `rows` rows of width elements at out (pitch ld_out) and of as many at proj (pitch
// ld_proj) meet.
bool rows_overlap(const uint16_t* out, int64_t ld_out, int64_t width, const uint16_t* proj, int64_t ld_proj,
                  int64_t rows) {
    const uintptr_t o0 = reinterpret_cast<uintptr_t>(out), p0 = reinterpret_cast<uintptr_t>(proj);
    const uintptr_t o1 = o0 + static_cast<uintptr_t>((rows - 1) * ld_out + width) * 2;
    const uintptr_t p1 = p0 + static_cast<uintptr_t>(rows * ld_proj) * 2;
    return o0 < p1 && p0 < o1;
}

template <int DK, int DV, int NWB>
int launch_state(const PrefillArgs& a, hipStream_t s) {
    constexpr size_t shmem = StateShape<DK, DV, NWB>::LDS_BYTES;
    static std::atomic<uint8_t> allowed[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return invalid("deltanet_prefill: device ordinal");
    if (!allowed[dev].load(std::memory_order_acquire)) {
        const int rc = check_hip(
            hipFuncSetAttribute(reinterpret_cast<const void*>(deltanet_chunk_state_kernel<DK, DV, NWB>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(shmem)),
            "hipFuncSetAttribute");
        if (rc != HAI_OK) return rc;
        allowed[dev].store(1, std::memory_order_release);
    }
    deltanet_chunk_state_kernel<DK, DV, NWB>
        <<<dim3(a.nv, DV / (32 * NWB), a.B), dim3(128 * NWB), shmem, s>>>(a);
    return launched("deltanet_chunk_state_kernel");
}

template <int DK, int DV>
int launch_prefill(const PrefillArgs& a, uint16_t* out, int64_t ld_out, int64_t off_z, const uint16_t* norm_w,
                   float eps, hipStream_t s) {
    const unsigned nchunks = static_cast<unsigned>((a.T + kChunk - 1) / kChunk);
    const dim3 pgrid(nchunks, a.nv, a.B);
    if (a.Kc == 4) deltanet_chunk_prep_kernel<DK, DV, 4><<<pgrid, dim3(256), 0, s>>>(a);
    else if (a.Kc == 3) deltanet_chunk_prep_kernel<DK, DV, 3><<<pgrid, dim3(256), 0, s>>>(a);
    else deltanet_chunk_prep_kernel<DK, DV, 0><<<pgrid, dim3(256), 0, s>>>(a);
    int rc = launched("deltanet_chunk_prep_kernel");
    if (rc != HAI_OK) return rc;
    // a head's value columns on two blocks while the CUs hold them all in one
    // round (MI355X, us for the whole call, one / two blocks per head: 1 x 1024
    // tokens of 48 heads 151 / 150, 2 x 1024 234 / 228; 4 x 512, 384 blocks of
    // two waves, 205 / 223)
    rc = DV > 64 && 2 * static_cast<int64_t>(a.B) * a.nv <= device_cus() ? launch_state<DK, DV, 2>(a, s)
                                                                         : launch_state<DK, DV, DV / 32>(a, s);
    if (rc != HAI_OK) return rc;
    const int hist = a.Kc - 1;
    const int64_t tasks = static_cast<int64_t>(a.B) * a.T * a.nv;
    // one launch for both, unless out lies among the projection rows: its blocks run in any order, and the ring's
    // take the last rows' inputs, which the norm's would then overwrite
    if (!rows_overlap(out, ld_out, static_cast<int64_t>(a.nv) * DV, a.proj, a.ld_proj, static_cast<int64_t>(a.B) * a.T) &&
        aligned16(out) && ld_out % 8 == 0 && aligned16(a.proj) && a.ld_proj % 8 == 0 && off_z % 8 == 0 &&
        aligned16(norm_w)) {
        const int64_t C = 2 * static_cast<int64_t>(a.nk) * DK + static_cast<int64_t>(a.nv) * DV;
        const int64_t per = 256 / (DV / 8);
        const int64_t nblocks = (tasks + per - 1) / per;
        const int64_t rblocks = (C / 2 * hist * a.B + 255) / 256;
        if (nblocks + rblocks <= INT32_MAX) {
            deltanet_gated_norm_ring_kernel<DV><<<dim3(static_cast<unsigned>(nblocks + rblocks)), dim3(256), 0, s>>>(
                out, ld_out, a.o_ws, a.proj, a.ld_proj, off_z, norm_w, static_cast<int64_t>(a.B) * a.T, a.nv, eps,
                static_cast<int>(nblocks), a.ring, a.ring_n, a.off_qkv, C, a.lens, a.pos_add, a.T, hist, a.B);
            return launched("deltanet_gated_norm_ring_kernel");
        }
    }
    if (hist > 0) {
        const int64_t C = 2 * static_cast<int64_t>(a.nk) * DK + static_cast<int64_t>(a.nv) * DV;
        deltanet_ring_update_kernel<<<dim3(static_cast<unsigned>((C + 255) / 256), hist, a.B), dim3(256), 0, s>>>(
            a.ring, a.ring_n, a.proj, a.ld_proj, a.off_qkv, C, a.lens, a.pos_add, a.T, hist);
        rc = launched("deltanet_ring_update_kernel");
        if (rc != HAI_OK) return rc;
    }
    deltanet_gated_norm_kernel<DV><<<dim3(static_cast<unsigned>((tasks + 3) / 4)), dim3(256), 0, s>>>(
        out, ld_out, a.o_ws, a.proj, a.ld_proj, off_z, norm_w, static_cast<int64_t>(a.B) * a.T, a.nv, eps);
    return launched("deltanet_gated_norm_kernel");
}

}  // namespace

// The unrounded outputs [B*T][nv*dv], then the per-chunk records (dk = dv).
static size_t chunk_record_bytes(int64_t B, int64_t T, int64_t nv, int64_t dv) {
    const int64_t per = dv == 64 ? chunk_floats<64, 64>() : chunk_floats<128, 128>();
    return static_cast<size_t>(B * nv * ((T + kChunk - 1) / kChunk) * per) * sizeof(float);
}
static size_t output_bytes(int64_t B, int64_t T, int64_t nv, int64_t dv) {
    return (static_cast<size_t>(B * T * nv * dv) * sizeof(float) + 255) / 256 * 256;
}

extern "C" size_t hai_deltanet_prefill_workspace_bytes(int64_t B, int64_t T, int64_t nv, int64_t dv) {
    if (B < 0 || T < 0 || nv < 0 || dv < 0) return 0;
    return output_bytes(B, T, nv, dv) + chunk_record_bytes(B, T, nv, dv);
}

extern "C" int hai_deltanet_prefill_bf16(void* out, int64_t ld_out, const void* proj, int64_t ld_proj,
                                         int64_t off_qkv, int64_t off_z, int64_t off_a, int64_t off_b,
                                         const void* conv_w, void* conv_ring, int64_t ring, float* state,
                                         int64_t nslots, const void* a_log, const void* dt_bias,
                                         const void* norm_w, const int32_t* lens, int32_t pos_add, int64_t B,
                                         int64_t T, int64_t nk, int64_t nv, int64_t dk, int64_t dv, int64_t Kc,
                                         float eps, void* workspace, int64_t workspace_bytes, void* stream) {
    if (out == nullptr || proj == nullptr || conv_w == nullptr || conv_ring == nullptr || state == nullptr ||
        a_log == nullptr || dt_bias == nullptr || norm_w == nullptr || workspace == nullptr)
        return invalid("deltanet_prefill: null pointer");
    if (B < 0 || T < 0 || nk <= 0 || nv <= 0 || nv % nk != 0 || Kc < 1 || Kc > kMaxKc || nslots < 1 || ring < Kc ||
        B > 65535 || nv > 65535 || T > INT32_MAX / 2 || static_cast<int64_t>(pos_add) + T > INT32_MAX)
        return invalid("deltanet_prefill: shape");
    if (lens == nullptr && pos_add < 0) return invalid("deltanet_prefill: negative position");
    if (!aligned16(state) || !aligned16(workspace)) return invalid("deltanet_prefill: alignment");
    // the conv reads channel pairs as one dword
    if ((reinterpret_cast<uintptr_t>(proj) & 3u) != 0 || (reinterpret_cast<uintptr_t>(conv_ring) & 3u) != 0 ||
        (ld_proj & 1) != 0 || (off_qkv & 1) != 0)
        return invalid("deltanet_prefill: proj and conv_ring must be 4-byte aligned, ld_proj and off_qkv even");
    if (workspace_bytes < 0 ||
        static_cast<size_t>(workspace_bytes) < hai_deltanet_prefill_workspace_bytes(B, T, nv, dv))
        return invalid("deltanet_prefill: workspace smaller than hai_deltanet_prefill_workspace_bytes");
    if (B == 0 || T == 0) return HAI_OK;
    PrefillArgs a{};
    a.o_ws = static_cast<float*>(workspace);
    a.chunks = reinterpret_cast<float*>(static_cast<char*>(workspace) + output_bytes(B, T, nv, dv));
    a.proj = static_cast<const uint16_t*>(proj);
    a.ld_proj = ld_proj;
    a.off_qkv = off_qkv;
    a.off_a = off_a;
    a.off_b = off_b;
    a.conv_w = static_cast<const uint16_t*>(conv_w);
    a.ring = static_cast<uint16_t*>(conv_ring);
    a.ring_n = int(ring);
    a.nslots = int(nslots);
    a.state = state;
    a.a_log = static_cast<const uint16_t*>(a_log);
    a.dt_bias = static_cast<const uint16_t*>(dt_bias);
    a.lens = lens;
    a.pos_add = pos_add;
    a.B = int(B);
    a.T = int(T);
    a.nk = int(nk);
    a.nv = int(nv);
    a.Kc = int(Kc);
    auto* o = static_cast<uint16_t*>(out);
    const auto* nw = static_cast<const uint16_t*>(norm_w);
    const auto s = as_stream(stream);
    if (dk == 128 && dv == 128) return launch_prefill<128, 128>(a, o, ld_out, off_z, nw, eps, s);
    if (dk == 64 && dv == 64) return launch_prefill<64, 64>(a, o, ld_out, off_z, nw, eps, s);
    return invalid("deltanet_prefill: (dk, dv) must be (128,128) or (64,64)");
}
