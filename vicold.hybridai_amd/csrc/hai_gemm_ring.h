// hai_gemm_ring.h -- the ring-staged batched GEMM (hai_gemm_ring.hip) as the
// matrix-core dispatcher calls it.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hai {

struct RingArgs {
    uint16_t* y;
    int64_t ldy;
    const uint16_t* x;
    int64_t ldx;
    const void* w;             // bf16, or E4M3 codes when scales is set
    const float* scales;
    const int32_t* scale_rows;
    int paired;
    const uint16_t* res;
    int64_t ldres;
    int M, N, K;
    float* part;               // fp32 partial planes [splits][M][N]
    int epi;                   // HAI_EPI_*
    int R, tiles, splits;      // the plan
};

constexpr int kRingK = 128;        // k per chunk (one FP8 scale block)
constexpr int kRingMaxRows = 64;   // activation rows

// The K splits of N x K weights, at most max_splits (a plane of part each).
int ring_splits(int64_t N, int64_t K, bool fp8, int max_splits, int cus);
// Fills the plan for `splits` splits: the tile height R.
void ring_plan(RingArgs& r, int splits, int cus);
// Needs K % kRingK == 0, M <= kRingMaxRows, 16-byte aligned x and w rows.
// check: the codes may hold 0x7F / 0xFF.  With splits > 1 the partials are
// left in part.
int launch_ring(const RingArgs& r, bool check, int cus, hipStream_t s);

}  // namespace hai
