// Dequant-GEMM for 17 rows to a few thousand: arguments, forms and the choice between them.
#pragma once

#include "sngguf_common.hpp"

namespace sngguf {

struct MidArgs {
    const bf16_t* x;
    bf16_t* y;
    int64_t M, N, K;
    const uint8_t* q[2];     // one matrix, or the gate and up matrices of a pair
    const bf16_t* bias;      // (one matrix, no partial sums)
    const bf16_t* residual;  // [M][N] added to the rounded output (one matrix, no partial sums)
    // K split over `ksplit` workgroups per tile: fp32 sums to partial[matrix][slice][M][N], to be added by a reduction; NULL:
    // ksplit = 1, outputs to y - for a pair silu(gate) * up, rounded as the decode kernels' gated pair rounds (N % 8 == 0).
    float* partial;
    int ksplit;
    bool pair;
    int64_t tile_rows, row_tiles, col_tiles;   // activation rows of a tile, tiles of the output
};

enum MidForm { kMidNarrow, kMidWide, kMidLong };   // see gemm_mid.hip

// One translation unit per block format.  `mt`: 16-row tiles the kernel instance holds, tile_rows <= 16 mt.
template <int QT>
int launch_mid_type(const MidArgs& a, int form, int mt, int numerics, hipStream_t stream);

struct MidPlan {
    int form, mt;            // form -1: no plan
    int64_t tile_rows, row_tiles;
    int slices;
    double us;               // what the model gives for it, the reduction included
};

// Whether the kernel takes a shape: a packed block format, 17 rows and more, whole super-blocks, 32-bit activation offsets.
bool mid_fits(int qtype, int64_t M, int64_t N, int64_t K);
// The fastest plan of a shape that fits by the model, with room for `max_slices` fp32 copies of the output (of both outputs of
// a pair); 0 or 1: no K split.
MidPlan mid_plan(int qtype, int64_t M, int64_t N, int64_t K, bool pair, int64_t max_slices);
// Output columns of a workgroup in a form.
int mid_columns(int form);
// Runs a plan; plan.slices > 1 needs `partial` (slices copies) and, for a pair, no bias or residual.
int launch_mid(const MidPlan& plan, const void* x, int64_t M, const void* q, const void* q_up, int qtype, int64_t N, int64_t K,
               const void* bias, const void* residual, void* y, float* partial, int numerics, hipStream_t stream);

}  // namespace sngguf
