// hai_gemm_ring.hip -- batched-verify linear layer, ring-staged form (see
// hai_gemm_mfma.hip for the contract and the other forms).
#include <atomic>
#include <type_traits>

#include "hai_common.h"
#include "hai_device.h"
#include "hai_gemm_common.h"
#include "hai_gemm_ring.h"
#include "hai_mfma.h"

namespace {

using namespace hai;

// ---------------------------------------------------------------------------
// Ring-staged batched GEMM (bf16 and FP8 weights, up to 64 rows, K a multiple
// of 128).  A persistent block owns R weight rows (a multiple of 16, chosen so
// that the tiles fill the CUs, see ring_plan) and walks its items (tile, range
// of 128-k chunks) through two rings of LDS stages, weights [R] x 128 KC with
// their scales (FP8) and activations [32 MT] x 128 KC:
//   * two waves copy the weights and scales, SW - 1 stages ahead of the
//     products, across item boundaries too, and the computing waves copy the
//     activations (from L2) two stages ahead in their own in-order queue; each
//     waits for its oldest stage with a counted s_waitcnt.  The copies are
//     inline assembly, so that the compiler does not wait for them before its
//     LDS reads;
//   * NG x MT computing waves own 32 weight rows x 32 activation rows each:
//     codes decoded exactly to bf16 in the B operand, a chunk (one 128-k scale
//     block) summed by 8 MFMAs of 32 x 32 x 16, scaled in fp32;
//   * one barrier per step of KC chunks: the step's stages have landed and
//     those of the step before are free.
// Rows sit in LDS with their 16-byte pieces permuted (piece p of row r at p ^
// swizzle(r)) so that the rows of one operand read fall in distinct banks.
// Rows past N and M repeat the last row (never stored); columns past R of the
// last 32-row group read other LDS bytes (never stored either).
// Bound by the copies: weights and activations share a CU's 27-32 B per ns
// (about 64 KB in flight at the latency of HBM under load), so the activations,
// re-read once per R rows, weigh as much per byte as the weights.  MI355X,
// M = 64 FP8: gate|up 80 -> 50 us without a second pass, down 38 -> 30 us;
// M = 32 bf16: gate|up 71 -> 56, down 38 -> 32 us.
// ---------------------------------------------------------------------------
constexpr int kRingCopiers = 2;   // waves that copy weights
constexpr int kRingXStages = 3;   // activation stages
constexpr int kRingLds = 160 * 1024;
constexpr int kRingMaxStages = 12;

// Weight stages that fit beside the activations, with the copies of all but
// two of them in a wave's vmcnt range.
int ring_stages(int R, int mt, bool fp8, int kc) {
    const int ng = (R + 31) / 32;
    const int w = R * kc * kRingK * (fp8 ? 1 : 2);
    const int per = w / (1024 * kRingCopiers) + (fp8 ? (kc * ng + kRingCopiers - 1) / kRingCopiers : 0);
    int n = (kRingLds - kRingXStages * 32 * mt * kc * kRingK * 2) / (w + (fp8 ? kc * ng * 256 : 0));
    if (n > kRingMaxStages) n = kRingMaxStages;
    while (n > 2 && (n - 2) * per > 63) --n;
    return n;
}

// Chunks per step.  Two where one chunk is too little work between barriers:
// up to 32 rows (one computing wave per 32 weight rows) and short tiles.  The
// last step of an odd number of chunks holds its one chunk twice and takes the
// first copy (MI355X, one chunk per step / this, 8 rows FP8: 1024 x 1152 8.2 / 7.3
// us, 5568 x 4992 14.2 / 12.8, 5568 x 8320 18.1 / 15.9; 32 rows: 5568 x 4992 14.7 /
// 13.6, 14336 x 5248 22.7 / 23.8).
int ring_kc(int R, int M, int64_t K, bool fp8) { return M <= 32 && R <= (fp8 ? 96 : 64) && K >= 2 * kRingK ? 2 : 1; }

template <int MT, int NG, bool FP8, int KC>
struct RingShape {
    static constexpr int EB = FP8 ? 1 : 2;
    static constexpr int WROW = KC * kRingK * EB;         // bytes of a staged weight row
    static constexpr int XROW = KC * kRingK * 2;          // bytes of a staged activation row
    static constexpr int SB = FP8 ? KC * NG * 256 : 0;    // scale bytes of a weight stage
    static constexpr int XB = 32 * MT * XROW;             // bytes of an activation stage
    static constexpr int SX = kRingXStages;
    static constexpr int WAVES = NG * MT + kRingCopiers;
    static constexpr int SCALE_COPIES = FP8 ? (KC * NG + kRingCopiers - 1) / kRingCopiers : 0;  // per copying wave
    static constexpr int XCOPIES = (XB / 1024 + NG * MT - 1) / (NG * MT);                  // per computing wave
    __host__ __device__ static constexpr int w_stage(int R) { return R * WROW + SB; }
    // 16-byte piece positions within a row
    static __device__ __forceinline__ int w_swz(int r) { return WROW == 128 ? (r >> 1) & 7 : r & 15; }
    static __device__ __forceinline__ int x_swz(int r) { return r & 15; }
};

// s_waitcnt vmcnt(n) for a run-time (wave-uniform) n.
__device__ __forceinline__ void wait_vmcnt_n(int n) {
    switch (n) {
#define HAI_VM(v) case v: wait_vmcnt<v>(); break;
#define HAI_VM8(v) HAI_VM(v) HAI_VM(v + 1) HAI_VM(v + 2) HAI_VM(v + 3) HAI_VM(v + 4) HAI_VM(v + 5) HAI_VM(v + 6) HAI_VM(v + 7)
        HAI_VM8(0) HAI_VM8(8) HAI_VM8(16) HAI_VM8(24) HAI_VM8(32) HAI_VM8(40) HAI_VM8(48) HAI_VM8(56)
#undef HAI_VM8
#undef HAI_VM
        default: wait_vmcnt<0>(); break;
    }
}
// A wave-uniform pointer in scalar registers.
__device__ __forceinline__ const void* uniform_ptr(const void* p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
    return reinterpret_cast<const void*>((static_cast<uint64_t>(hi) << 32) | lo);
}
// One global -> LDS copy per lane of 16 (4) bytes at base + off, to lds + 16
// (4) * lane (the M0 write needs one wait state); nt: non-temporal.
__device__ __forceinline__ void ring_copy16(uint32_t off, const void* base, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(lds) : "memory");
}
__device__ __forceinline__ void ring_copy16_nt(uint32_t off, const void* base, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt" : : "v"(off), "s"(base), "s"(lds) : "memory");
}
__device__ __forceinline__ void ring_copy4(uint32_t off, const void* base, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" : : "v"(off), "s"(base), "s"(lds) : "memory");
}
__device__ __forceinline__ u32x4 ring_read16(uint32_t lds) {
    return *(const __attribute__((address_space(3))) u32x4*)(uintptr_t)lds;
}
template <int MT, int NG, bool FP8, bool CHECK, int KC, bool ODD>
__global__ __launch_bounds__(64 * (NG * MT + kRingCopiers)) void gemm_ring_mfma_kernel(RingArgs a, int SW) {
    using SH = RingShape<MT, NG, FP8, KC>;
    constexpr int SX = SH::SX;
    extern __shared__ __align__(1024) uint8_t ring_lds[];
    const int lane = threadIdx.x & 63;
    const int wave = wave_index();
    const int lc = lane & 31, lh = lane >> 5;
    const int R = a.R;
    const int wstage = SH::w_stage(R);
    const uint32_t lds0 = static_cast<uint32_t>(
        reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)ring_lds));
    const uint32_t ldsx = lds0 + SW * wstage;  // the activation stages
    // weights that the 256 MB cache behind the L2s cannot hold beside others are streamed past it (MI355X, gate|up
    // FP8, 178 MB, M = 32: 47.7 -> 42.1 us with the norm; 16384 x 5120, 84 MB: 24.2 -> 24.8)
    const bool nt = static_cast<int64_t>(a.N) * a.K * SH::EB > (int64_t{96} << 20);
    const int items = a.tiles * a.splits;
    // first step (of KC chunks) of a split: K is cut between pairs of chunks whatever KC is, so that a row's sums do
    // not depend on the form that the number of rows selects
    const int nck = a.K / kRingK;
    auto step_lo = [&](int split) {
        const int pair = static_cast<int>(static_cast<int64_t>(split) * ((nck + 1) / 2) / a.splits);
        return KC == 2 ? pair : min(2 * pair, nck);
    };
    // a step of one chunk, held twice (ODD: an odd number of chunks; an instance of its own, the tests cost the even
    // ones up to 10 %)
    auto half_step = [&](int step) { return KC == 2 && ODD && 2 * step + 1 == nck; };
    // total steps of this block
    int total = 0;
    for (int it = blockIdx.x; it < items; it += gridDim.x)
        total += step_lo(it / a.tiles + 1) - step_lo(it / a.tiles);

    if (wave >= NG * MT) {  // ---- a copying wave: weights and scales ----
        const int p = wave - NG * MT;
        const int per = R * SH::WROW / (1024 * kRingCopiers) + SH::SCALE_COPIES;  // copies per chunk
        constexpr int WL = 1024 / SH::WROW;  // weight rows per copy
        const int wr = lane / (64 / WL), wpos = lane % (64 / WL);
        // the chunk cursor: requests run ahead of the products
        int item = blockIdx.x, c = 0, cend = 0, slot = 0;
        uint32_t srow[SH::SCALE_COPIES > 0 ? SH::SCALE_COPIES : 1] = {};
        const char* wbase = nullptr;
        int last = 0;
        auto open_item = [&]() {  // (item < items)
            const int tile = item % a.tiles;
            const int split = item / a.tiles;
            c = step_lo(split);
            cend = step_lo(split + 1);
            const int64_t row0 = static_cast<int64_t>(tile) * R;
            last = static_cast<int>(min(static_cast<int64_t>(R), a.N - row0)) - 1;
            wbase = static_cast<const char*>(a.w) + row0 * a.K * SH::EB;
            if constexpr (FP8) {
                const int nkb = a.K / 128;
#pragma unroll
                for (int i = 0; i < SH::SCALE_COPIES; ++i) {
                    const int g = min(p + kRingCopiers * i, KC * NG - 1);  // (row group g / KC, chunk g % KC)
                    const int64_t n = min(row0 + 32 * (g / KC) + lc, static_cast<int64_t>(a.N) - 1);
                    const int64_t nsb = ((a.N >> 1) + 127) / 128;
                    const int64_t sr =
                        a.scale_rows ? a.scale_rows[n] : (a.paired ? (n & 1) * nsb + (n >> 1) / 128 : n / 128);
                    srow[i] = static_cast<uint32_t>((sr * nkb + g % KC) * 4);
                }
            }
        };
        // this wave's copies of a stage are i = p + 2 t; the piece permutation of a lane's row repeats every four,
        // so a whole tile needs four lane offsets and a scalar base per copy
        constexpr int PH = 4;
        const int ncopy = R / (WL * kRingCopiers);
        const uint32_t wpitch = static_cast<uint32_t>(a.K) * SH::EB;
        constexpr int HALF_ROW = SH::WROW / 2;  // the second chunk's bytes of a row (KC = 2)
        uint32_t woff[PH];
#pragma unroll
        for (int u = 0; u < PH; ++u)
            woff[u] = wr * wpitch + ((wpos ^ SH::w_swz((p + kRingCopiers * u) * WL + wr)) << 4);
        auto copy_w = [&](auto stream, const void* wb, uint32_t dst, bool half) {
            constexpr bool NT = decltype(stream)::value;
            uint32_t wo[PH];  // (half: the second chunk's pieces repeat the first's)
#pragma unroll
            for (int u = 0; u < PH; ++u)
                wo[u] = woff[u] - (half ? ((wpos ^ SH::w_swz((p + kRingCopiers * u) * WL + wr)) << 4) & HALF_ROW : 0);
            if (last == R - 1) {
                const char* base = static_cast<const char*>(wb) + static_cast<int64_t>(p * WL) * wpitch;
                const int64_t step = static_cast<int64_t>(kRingCopiers * WL) * wpitch;
                dst += p * 1024;
                for (int t = 0; t < ncopy; t += PH) {
#pragma unroll
                    for (int u = 0; u < PH; ++u) {
                        if (t + u >= ncopy) break;
                        if constexpr (NT) ring_copy16_nt(wo[u], base, dst);
                        else ring_copy16(wo[u], base, dst);
                        base += step;
                        dst += kRingCopiers * 1024;
                    }
                }
            } else {  // rows past N: the last one
                for (int t = 0; t < ncopy; ++t) {
                    const int i = p + kRingCopiers * t;
                    const int r = i * WL + wr;
                    const uint32_t piece = static_cast<uint32_t>(wpos ^ SH::w_swz(r)) << 4;
                    const uint32_t off =
                        static_cast<uint32_t>(min(r, last)) * wpitch + (half ? piece & ~static_cast<uint32_t>(HALF_ROW) : piece);
                    if constexpr (NT) ring_copy16_nt(off, wb, dst + i * 1024);
                    else ring_copy16(off, wb, dst + i * 1024);
                }
            }
        };
        auto request = [&]() {  // the cursor's chunk into the next slot
            const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + slot * wstage);
            const void* wb = uniform_ptr(wbase + static_cast<int64_t>(c) * SH::WROW);
            const bool half = half_step(c);
            if (nt) copy_w(std::true_type{}, wb, dst, half);
            else copy_w(std::false_type{}, wb, dst, half);
            if constexpr (FP8) {
#pragma unroll
                for (int i = 0; i < SH::SCALE_COPIES; ++i) {
                    const int g = min(p + kRingCopiers * i, KC * NG - 1);
                    ring_copy4(srow[i] + c * (4 * KC) - (half ? 4 * (g % KC) : 0), a.scales,
                               dst + R * SH::WROW + g * 256);
                }
            }
            slot = slot + 1 == SW ? 0 : slot + 1;
            if (++c == cend) {
                item += gridDim.x;
                if (item < items) open_item();
            }
        };
        open_item();
        int asked = 0;
        for (; asked < SW - 1 && asked < total; ++asked) request();
        for (int i = 0; i < total; ++i) {
            // chunk i has landed: at most the later chunks' requests are outstanding
            if (i + SW - 2 < total) wait_vmcnt_n((SW - 2) * per);
            else wait_vmcnt<0>();
            lds_barrier();
            if (asked < total) {
                request();
                ++asked;
            }
        }
        return;
    }

    // ---- a computing wave: weight rows 32 ng .. + 31, activation rows 32 mg .. + 31 ----
    const int ng = wave % NG, mg = wave / NG;
    const int wrow = 32 * ng + lc, xrow = 32 * mg + lc;
    const uint32_t w0 = lds0 + wrow * SH::WROW, x0 = ldsx + xrow * SH::XROW;
    const int wsw = SH::w_swz(wrow), xsw = SH::x_swz(xrow);
    // its share of the activation copies (the last ones of an uneven split repeat the last 1 KB)
    constexpr int XLANES = SH::XROW / 16;  // lanes per row
    uint32_t xoff[SH::XCOPIES], xdst[SH::XCOPIES];
#pragma unroll
    for (int j = 0; j < SH::XCOPIES; ++j) {
        const int i = min(wave + NG * MT * j, SH::XB / 1024 - 1);
        const int r = i * (64 / XLANES) + lane / XLANES;
        xoff[j] = static_cast<uint32_t>(min(r, a.M - 1)) * static_cast<uint32_t>(a.ldx * 2) +
                  (((lane % XLANES) ^ SH::x_swz(r)) << 4);
        xdst[j] = __builtin_amdgcn_readfirstlane(ldsx + i * 1024);
    }
    int xitem = blockIdx.x, xc = step_lo(xitem / a.tiles), xend = step_lo(xitem / a.tiles + 1), xslot = 0, xasked = 0;
    auto request_x = [&]() {
        const void* xb = uniform_ptr(reinterpret_cast<const char*>(a.x) + static_cast<int64_t>(xc) * SH::XROW);
        if (half_step(xc)) {  // the second chunk's pieces (the permutation leaves their bit alone) repeat the first's
#pragma unroll
            for (int j = 0; j < SH::XCOPIES; ++j)
                ring_copy16(xoff[j] - (((lane % XLANES) & (XLANES / 2)) << 4), xb,
                            __builtin_amdgcn_readfirstlane(xdst[j] + xslot * SH::XB));
        } else {
#pragma unroll
            for (int j = 0; j < SH::XCOPIES; ++j)
                ring_copy16(xoff[j], xb, __builtin_amdgcn_readfirstlane(xdst[j] + xslot * SH::XB));
        }
        xslot = xslot + 1 == SX ? 0 : xslot + 1;
        ++xasked;
        if (++xc == xend) {
            xitem += gridDim.x;
            if (xitem < items) {
                xc = step_lo(xitem / a.tiles);
                xend = step_lo(xitem / a.tiles + 1);
            }
        }
    };
    while (xasked < SX - 1 && xasked < total) request_x();
    int done = 0, slot = 0, xs = 0;
    for (int item = blockIdx.x; item < items; item += gridDim.x) {
        const int tile = item % a.tiles;
        const int split = item / a.tiles;
        const int cend = step_lo(split + 1);
        f32x16 tot;
#pragma unroll
        for (int i = 0; i < 16; ++i) tot[i] = 0.0f;
        for (int c = step_lo(split); c < cend; ++c) {
            // this wave's copies of the chunk have landed, then everyone's
            if (done + SX - 2 < total) wait_vmcnt<(SX - 2) * SH::XCOPIES>();
            else wait_vmcnt<0>();
            lds_barrier();
            if (xasked < total) request_x();
            ++done;
            const uint32_t so = slot * wstage, xo = xs * SH::XB;
            slot = slot + 1 == SW ? 0 : slot + 1;
            xs = xs + 1 == SX ? 0 : xs + 1;
            if constexpr (FP8) {
                // step 2 j + e of chunk q: k = 32 j + 16 lh + 8 e + [0, 8); the next pair's activations are read
                // while a pair's codes are decoded and multiplied
                auto x_at = [&](int q, int j) {
                    return ring_read16(x0 + xo + (((16 * q + 4 * (j >> 1) + 2 * lh + (j & 1)) ^ xsw) << 4));
                };
                u32x4 wq[KC][4], xa[2][KC][2];
                float sc[KC];
#pragma unroll
                for (int q = 0; q < KC; ++q) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        wq[q][j] = ring_read16(w0 + so + (((8 * q + 2 * j + lh) ^ wsw) << 4));
                    xa[0][q][0] = x_at(q, 0);
                    xa[0][q][1] = x_at(q, 1);
                    sc[q] = *(const __attribute__((address_space(3))) float*)(uintptr_t)(
                        lds0 + so + R * SH::WROW + (ng * KC + q) * 256 + lc * 4);
                }
                // (one chain of products per chunk in every form, so that a row's sums do not depend on how many
                // rows the call has)
                f32x16 acc[KC];
#pragma unroll
                for (int q = 0; q < KC; ++q)
#pragma unroll
                    for (int i = 0; i < 16; ++i) acc[q][i] = 0.0f;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    u32x4 d[KC][2];
#pragma unroll
                    for (int q = 0; q < KC; ++q) {
                        if (j < 3) {
                            xa[(j + 1) & 1][q][0] = x_at(q, 2 * j + 2);
                            xa[(j + 1) & 1][q][1] = x_at(q, 2 * j + 3);
                        }
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            uint32_t lo, hi;
                            if constexpr (CHECK) {
                                e4m3x4_to_bf16<true>(wq[q][j][e], lo, hi);
                            } else {
                                lo = e4m3x2_to_bf16(wq[q][j][e], false);
                                hi = e4m3x2_to_bf16(wq[q][j][e], true);
                            }
                            d[q][e >> 1][2 * (e & 1)] = lo;
                            d[q][e >> 1][2 * (e & 1) + 1] = hi;
                        }
                    }
#pragma unroll
                    for (int e = 0; e < 2; ++e)
#pragma unroll
                        for (int q = 0; q < KC; ++q) acc[q] = mfma32(xa[j & 1][q][e], d[q][e], acc[q]);
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int q = 0; q < KC; ++q) {
                    if (q > 0 && half_step(c)) break;
#pragma unroll
                    for (int i = 0; i < 16; ++i) tot[i] = fma_(sc[q], acc[q][i], tot[i]);
                }
            } else {
                u32x4 wb[8], xa[8];
#pragma unroll
                for (int q = 0; q < KC; ++q) {
                    if (q > 0 && half_step(c)) break;
#pragma unroll
                    for (int t = 0; t < 8; ++t) {
                        wb[t] = ring_read16(w0 + so + (((16 * q + 2 * t + lh) ^ wsw) << 4));
                        xa[t] = ring_read16(x0 + xo + (((16 * q + 2 * t + lh) ^ xsw) << 4));
                    }
#pragma unroll
                    for (int t = 0; t < 8; ++t) tot = mfma32(xa[t], wb[t], tot);
                }
            }
        }
        // result: lane = weight row (column n), element i = activation row 8 (i / 4) + 4 lh + i % 4
        const int64_t n = static_cast<int64_t>(tile) * R + wrow;
        const bool col = wrow < R && n < a.N;
        const int m0 = 32 * mg + 4 * lh;
        // the pitches are made opaque here, or the compiler forms the 16 row offsets before the item loop and spills them
        // (27B MLP, 64 rows FP8, two cards: 89 -> 79 us, 88 -> 85)
        int64_t ldy = a.ldy, ldres = a.ldres, pitch = a.N;
        asm volatile("" : "+s"(ldy), "+s"(ldres), "+s"(pitch));
        if (a.splits > 1) {
            if (col) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int m = m0 + 8 * (i >> 2) + (i & 3);
                    if (m < a.M) a.part[(static_cast<int64_t>(split) * a.M + m) * pitch + n] = tot[i];
                }
            }
        } else if (a.epi == HAI_EPI_SILU_MUL) {
            // lanes lc, lc ^ 1 hold a gate and its up column: the even one takes elements 0 .. 7, the odd one 8 .. 15
            const bool odd = (lc & 1) != 0;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float a0 = bfr(tot[i]), a1 = bfr(tot[i + 8]);
                const float b0 = quad_xor1(a0), b1 = quad_xor1(a1);
                const int m = m0 + 8 * (i >> 2) + (i & 3) + (odd ? 16 : 0);
                if (col && m < a.M)
                    a.y[static_cast<int64_t>(m) * ldy + n / 2] = f2bf(hw_silu(odd ? b1 : a0) * (odd ? a1 : b0));
            }
        } else if (col) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int m = m0 + 8 * (i >> 2) + (i & 3);
                if (m >= a.M) continue;
                float o = bfr(tot[i]);
                if (a.epi == HAI_EPI_RESIDUAL) o = bf2f(a.res[static_cast<int64_t>(m) * ldres + n]) + o;
                a.y[static_cast<int64_t>(m) * ldy + n] = f2bf(o);
            }
        }
    }
}

template <int MT, int NG, bool FP8, bool CHECK, int KC = 1, bool ODD = false>
int launch_ring_as(const RingArgs& r, int cus, hipStream_t s) {
    using SH = RingShape<MT, NG, FP8, KC>;
    static std::atomic<uint8_t> allowed[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return invalid("gemm_mfma: device");
    auto* kern = gemm_ring_mfma_kernel<MT, NG, FP8, CHECK, KC, ODD>;
    if (!allowed[dev].load(std::memory_order_acquire)) {
        const int rc = check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, kRingLds),
                                 "hipFuncSetAttribute");
        if (rc != HAI_OK) return rc;
        allowed[dev].store(1, std::memory_order_release);
    }
    const int sw = ring_stages(r.R, MT, FP8, KC);
    const size_t shmem = static_cast<size_t>(sw) * SH::w_stage(r.R) + SH::SX * SH::XB;
    const int64_t items = static_cast<int64_t>(r.tiles) * r.splits;
    const unsigned grid = static_cast<unsigned>(items < cus ? items : cus);
    kern<<<dim3(grid), dim3(64 * SH::WAVES), shmem, s>>>(r, sw);
    return launched("gemm_ring_mfma_kernel");
}
template <int MT, bool FP8, bool CHECK, bool ODD>  // two chunks per step
int launch_ring_pairs(const RingArgs& r, int cus, hipStream_t s) {
    if (r.R <= 32) return launch_ring_as<MT, 1, FP8, CHECK, 2, ODD>(r, cus, s);
    if constexpr (FP8)
        if (r.R > 64) return launch_ring_as<MT, 3, FP8, CHECK, 2, ODD>(r, cus, s);
    return launch_ring_as<MT, 2, FP8, CHECK, 2, ODD>(r, cus, s);
}
template <int MT, bool FP8, bool CHECK>
int launch_ring_ng(const RingArgs& r, int cus, hipStream_t s) {
    if constexpr (MT == 1) {
        if (ring_kc(r.R, r.M, r.K, FP8) == 2)
            return r.K / kRingK % 2 != 0 ? launch_ring_pairs<MT, FP8, CHECK, true>(r, cus, s)
                                         : launch_ring_pairs<MT, FP8, CHECK, false>(r, cus, s);
    }
    switch ((r.R + 31) / 32) {
        case 1: return launch_ring_as<MT, 1, FP8, CHECK>(r, cus, s);
        case 2: return launch_ring_as<MT, 2, FP8, CHECK>(r, cus, s);
        case 3: return launch_ring_as<MT, 3, FP8, CHECK>(r, cus, s);
        case 4: return launch_ring_as<MT, 4, FP8, CHECK>(r, cus, s);
        default: return launch_ring_as<MT, 5, FP8, CHECK>(r, cus, s);
    }
}

}  // namespace

namespace hai {

namespace {
// The tile height of N x K weights whose busiest CU copies the fewest bytes for
// M rows and `splits` splits, and those bytes: the copies are what bounds the
// kernel, weights (HBM) and activations (L2) alike, at 27-32 B per ns and CU
// however many stages are in flight (MI355X, M = 64 FP8: gate|up, 242 tiles of
// 144 rows, W alone 34 us, X alone 17, both 48).
int best_tile(int M, int64_t N, int64_t K, bool fp8, int splits, int cus, double& cost) {
    const int eb = fp8 ? 1 : 2;
    const int mt = M <= 32 ? 1 : 2;
    const int64_t nck = K / kRingK;
    int best = 0;
    for (int R = 32; R <= 160; R += 16) {
        if (ring_stages(R, mt, fp8, ring_kc(R, M, K, fp8)) < 3) break;
        const int64_t tiles = (N + R - 1) / R;
        const int64_t rounds = (tiles * splits + cus - 1) / cus;
        const double c = static_cast<double>(rounds) * static_cast<double>((nck + splits - 1) / splits) *
                         (R * kRingK * eb + mt * 32 * kRingK * 2);
        if (best == 0 || c < cost) {
            best = R;
            cost = c;
        }
    }
    return best;
}
}  // namespace

// The splits follow N, K and the weight format alone (priced for 64 rows), so
// that a row's sums are the same whatever the number of rows: a verify and a
// correction of the same row round alike.  FP8 tiles too tall for two chunks per
// step (more than 96 rows) are slower than their bytes.  Above 8192 columns they
// are not taken: MI355X, one / two splits at 8, 32 and 64 rows, 14336 x 5120 FP8
// 19.9 / 21.6, 23.0 / 23.2, 28.5 / 29.9 us, 16480 x 5120 21.1 / 23.6, 24.4 / 26.3, 32.5 /
// 33.6; where the tiles stay shorter two win, 12288 x 5120 20.3 / 17.7, 22.5 / 19.7,
// 26.4 / 26.9, for about 9 us of partial planes and second pass.  Up to 8192 the
// shorter walk over K outweighs the second pass wherever the splits shorten it,
// and tall tiles cost a step's worth: 1 / 2 / 3 / 4 splits at 8 and 64 rows FP8, 1024 x
// 2944 15.1 / 10.7 / 9.2 / 8.7 and 20.1 / 13.2 / 11.5 / 10.7 us, 5120 x 4096 18.5 / 13.7 /
// 12.5 / 12.1 and 24.4 / 16.6 / 15.8 / 16.2, 8192 x 4096 (tall from three on) 19.6 / 14.1 /
// 15.1 / 14.9 and 24.7 / 17.2 / 19.8 / 19.7.  (Over 81 shapes of 512-8192 x 1024-6144 the
// plan is 1-2 % behind the best split on average, 16 % at most; priced with 9 us
// for the second pass it was 13 % behind, 84 % at most.)
int ring_splits(int64_t N, int64_t K, bool fp8, int max_splits, int cus) {
    int best = 1;
    double cost = 0.0;
    for (int splits = 1; splits <= max_splits; ++splits) {
        double c = 0.0;
        const int R = best_tile(kRingMaxRows, N, K, fp8, splits, cus, c);
        if (splits > 1) {
            const bool tall = fp8 && ring_kc(R, 1, K, fp8) == 1;
            if (tall && N > 8192) continue;
            c += (N > 8192 ? 270e3 : tall ? 150e3 : 0.0) + 8.0 * splits * kRingMaxRows * static_cast<double>(N) / cus;
        }
        if (splits == 1 || c < cost) {
            best = splits;
            cost = c;
        }
    }
    return best;
}

void ring_plan(RingArgs& r, int splits, int cus) {
    double cost = 0.0;
    r.splits = splits;
    r.R = best_tile(r.M, r.N, r.K, r.scales != nullptr, splits, cus, cost);
    r.tiles = (r.N + r.R - 1) / r.R;
}

int launch_ring(const RingArgs& r, bool check, int cus, hipStream_t s) {
    if (r.M <= 32)
        return r.scales == nullptr ? launch_ring_ng<1, false, false>(r, cus, s)
               : check             ? launch_ring_ng<1, true, true>(r, cus, s)
                                   : launch_ring_ng<1, true, false>(r, cus, s);
    return r.scales == nullptr ? launch_ring_ng<2, false, false>(r, cus, s)
           : check             ? launch_ring_ng<2, true, true>(r, cus, s)
                               : launch_ring_ng<2, true, false>(r, cus, s);
}

}  // namespace hai
