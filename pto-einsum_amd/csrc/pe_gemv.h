// Matrix-vector contractions: plan and launch (kernels in pe_gemv.hip).
#pragma once

#include "pe_common.h"

namespace pe {

// W is the operand with the free axis (extent N), x the other one.
struct GemvArgs {
    const void* w;
    const void* x;
    float* out;
    float* partial;           // [split][batch][N] when nsplit > 1
    int32_t N, K;
    uint32_t rows;            // batches * N
    uint32_t tiles;           // blocks per batch (all of them with one x per row)
    int32_t nsplit, k_per_split;
    int64_t w_ns, w_ks, x_ks, o_ns;
    FastDiv n_div;
    int32_t nbatch;
    FastDiv batch_div[PE_MAX_DIMS];
    int64_t w_bs[PE_MAX_DIMS], x_bs[PE_MAX_DIMS], o_bs[PE_MAX_DIMS];
};

struct GemvPlan {
    int kind;                 // 0 = not taken, 1 = rows (k contiguous), 2 = columns (n contiguous)
    bool a_vec;               // A is the vector (M = 1)
    bool xrow;                // rows of a tile have an x each
    int lpr;                  // lanes per row (kind 1) or column lanes (kind 2)
    int split, kps;           // K splits and k per split
    uint32_t tiles;
    int64_t N, blocks, ws_bytes;
};

// Up to this many splits a thread per output sums the partials, more a wave.
constexpr int kWaveReduceSplits = 16;

GemvPlan gemv_plan(const pe_gemm_desc& d, int64_t nb);
hipError_t launch_gemv(const pe_gemm_desc& d, const GemvPlan& p, int64_t nb, const void* a, const void* b, float* c,
                       void* ws, hipStream_t s);

}  // namespace pe
