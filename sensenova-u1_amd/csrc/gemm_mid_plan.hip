// Which form, tile and K split the mid-size dequant-GEMM takes (gemm_mid.hip), and its launch.
#include "gemm_mid.hpp"

#include "gemm_args.hpp"

namespace sngguf {

int launch_splitk_reduce(const GemmArgs& a, const uint8_t* indicator, int64_t n_text, hipStream_t stream);
int launch_splitk_reduce_gated(const float* gate, const float* up, int slices, int64_t M, int64_t N, bf16_t* h, hipStream_t stream);

#define SNGGUF_MID_TYPES(F) \
    F(SNGGUF_TYPE_Q4_0) F(SNGGUF_TYPE_Q4_1) F(SNGGUF_TYPE_Q5_0) F(SNGGUF_TYPE_Q5_1) F(SNGGUF_TYPE_Q8_0) \
    F(SNGGUF_TYPE_Q2_K) F(SNGGUF_TYPE_Q3_K) F(SNGGUF_TYPE_Q4_K) F(SNGGUF_TYPE_Q5_K) F(SNGGUF_TYPE_Q6_K)
#define SNGGUF_DECL(QT) template <> int launch_mid_type<QT>(const MidArgs&, int, int, int, hipStream_t);
SNGGUF_MID_TYPES(SNGGUF_DECL)
#undef SNGGUF_DECL

bool mid_fits(int qtype, int64_t M, int64_t N, int64_t K) {
#define SNGGUF_IS(QT) || qtype == QT
    return (false SNGGUF_MID_TYPES(SNGGUF_IS)) && M >= 17 && N >= 1 && K >= 256 && K % 256 == 0 && M * K < ((int64_t)1 << 31);
#undef SNGGUF_IS
}

namespace {

struct FormInfo {
    int cols;                  // output columns of a workgroup
    int kw;                    // K halves it works on at once
    int sizes[8];              // 16-row tiles an instance holds, ascending, 0-terminated
    double fixed, step, row;   // us of a workgroup: prologue and epilogue, a super-block, a super-block per 16 rows
};
// These pick the form, the tile and the split; one set for all formats.  Fitted (log least squares) to Q8_0, Q4_K and Q6_K at twelve
// shapes, 20 .. 1024 rows, with the kernel as it was when it issued a stage's requests in one go (it has become 4 % faster in the mean,
// unevenly, - 14 .. + 7 %; on ten shapes of 203 .. 1024 rows the pick is still the fastest of five to eight plans); measured then over all
// ten formats - eleven shapes of 512 .. 24576 columns and 2048 .. 12288 elements of K, 17 ..
// 1900 rows, every form and tile with 1 .. 16 K slices, 36090 timings - the pick is 0.6 % slower than the fastest of them in the
// mean (17 % at worst: 100 rows of 4096 x 4096 in Q4_0 and Q4_1).
constexpr FormInfo kForms[] = {
    {64, 2, {2, 3, 4, 0}, 1.16, 1.62, 0.16},
    {128, 2, {2, 3, 4, 6, 8, 10, 13, 0}, 3.26, 2.41, 0.35},
    {256, 1, {10, 13, 16, 0}, 3.49, 3.40, 0.19},
};

// Against other kernels it takes the time itself, which these constants miss by up to a quarter from format to format: us of a plan
// with the super-block's share scaled by format, the split's launch and sums, and the outputs, fitted to the same timings of what
// is picked (rms 5.8 %; one set for all 9 %, with Q6_K 19 % under).  They have not been fitted again since the kernel became faster, so a
// shape near the border still takes the other kernel where that was the faster one then.
double format_step(int qtype) {
    switch (qtype) {
    case SNGGUF_TYPE_Q4_0: return 0.776;
    case SNGGUF_TYPE_Q4_1: return 0.813;
    case SNGGUF_TYPE_Q5_0: return 0.977;
    case SNGGUF_TYPE_Q5_1: return 0.920;
    case SNGGUF_TYPE_Q8_0: return 0.911;
    case SNGGUF_TYPE_Q2_K: return 0.859;
    case SNGGUF_TYPE_Q3_K: return 0.981;
    case SNGGUF_TYPE_Q4_K: return 0.933;
    case SNGGUF_TYPE_Q5_K: return 1.034;
    default: return 1.185;   // Q6_K
    }
}

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

MidPlan best_plan(int qtype, int64_t M, int64_t N, int64_t K, bool pair, int64_t max_slices) {
    MidPlan best{-1, 0, 0, 0, 1, 1e30};
    const int64_t nsb = K >> 8, cols = pair ? 2 * N : N;
    const double scale = format_step(qtype), outputs = (double)(2 * M * N);
    double best_pick = 1e30;
    for (int form = 0; form < 3; form++) {
        const FormInfo& f = kForms[form];
        const int64_t col_tiles = ceil_div(cols, f.cols);
        // at least one super-block per K share of a workgroup, and no more slices than pay
        int64_t smax = nsb / f.kw < 16 ? nsb / f.kw : 16;
        if (smax > max_slices) smax = max_slices;
        if (smax < 1) smax = 1;
        int64_t last_tiles = 0;
        for (int i = 7; i >= 0; i--) {
            if (f.sizes[i] == 0) continue;
            // rows cut evenly into as many tiles as instances of this size need, each in the smallest instance that holds it
            const int64_t row_tiles = ceil_div(M, 16 * f.sizes[i]);
            if (row_tiles == last_tiles) continue;
            last_tiles = row_tiles;
            const int64_t tile_rows = 16 * ceil_div(ceil_div(M, row_tiles), 16);
            int at = 0;
            while (16 * f.sizes[at] < tile_rows) at++;
            const int mt = f.sizes[at];
            const double step = f.step + f.row * mt;
            for (int64_t s = 1; s <= smax; s++) {
                const int64_t wgs = col_tiles * row_tiles * s, per_cu = ceil_div(wgs, 256), steps = ceil_div(ceil_div(nsb, s), f.kw);
                // two workgroups of the narrow form run on a compute unit at once and hide some of each other's latency, but the
                // instructions of both have to be issued: two take as long as two
                const int64_t rounds = form == kMidNarrow ? ceil_div(per_cu, 2) : per_cu;
                const double fixed = 3.3 + (double)rounds * f.fixed, sums = (double)(s * M * cols) * 8.0, loop = (double)(per_cu * steps);
                const double pick = fixed + loop * step + (s > 1 ? 2.75 + sums / 6.7e6 : 0.0);
                if (pick >= best_pick) continue;
                best_pick = pick;
                best = MidPlan{form, mt, tile_rows, row_tiles, (int)s,
                               fixed + loop * (f.step * scale + f.row * mt) + (s > 1 ? 3.4 + sums / 5.4e6 : outputs * 0.32e-6)};
            }
        }
    }
    return best;
}

}  // namespace

int mid_columns(int form) { return kForms[form].cols; }

// A call asks for its plan two to four times (how much scratch, which kernel, the launch), 0.7 - 1.7 us each with a search over some
// hundred plans, and a layer's shapes come round with every layer: each thread keeps its last plans, a function of these
// numbers alone, one to a slot.
MidPlan mid_plan(int qtype, int64_t M, int64_t N, int64_t K, bool pair, int64_t max_slices) {
    struct Slot {
        int64_t M, N, K, max_slices;
        int qtype, pair;
        MidPlan plan;
    };
    constexpr int kSlots = 64;
    static thread_local Slot slots[kSlots] = {};   // (M = 0: empty)
    if (max_slices > 16) max_slices = 16;          // the most that a plan has
    if (M <= 0) return best_plan(qtype, M, N, K, pair, max_slices);
    const uint64_t h = ((uint64_t)M * 0x9E3779B97F4A7C15ull ^ (uint64_t)N * 0xC2B2AE3D27D4EB4Full ^ (uint64_t)K * 0x165667B19E3779F9ull) +
                       (uint64_t)(max_slices * 64 + qtype * 2 + pair) * 0xD6E8FEB86659FD93ull;
    Slot& slot = slots[h >> 58];
    if (slot.M != M || slot.N != N || slot.K != K || slot.max_slices != max_slices || slot.qtype != qtype || slot.pair != (int)pair)
        slot = Slot{M, N, K, max_slices, qtype, pair, best_plan(qtype, M, N, K, pair, max_slices)};
    return slot.plan;
}

int launch_mid(const MidPlan& plan, const void* x, int64_t M, const void* q, const void* q_up, int qtype, int64_t N, int64_t K,
               const void* bias, const void* residual, void* y, float* partial, int numerics, hipStream_t stream) {
    if (plan.form < 0 || plan.slices < 1 || (q_up && (N % 8 != 0 || bias || residual))) return SNGGUF_E_BADSHAPE;
    if (plan.slices > 1 && !partial) return SNGGUF_E_NULLPTR;
    MidArgs a{};
    a.x = static_cast<const bf16_t*>(x);
    a.y = static_cast<bf16_t*>(y);
    a.M = M; a.N = N; a.K = K;
    a.q[0] = static_cast<const uint8_t*>(q);
    a.q[1] = static_cast<const uint8_t*>(q_up);
    a.pair = q_up != nullptr;
    a.ksplit = plan.slices;
    a.partial = plan.slices > 1 ? partial : nullptr;
    a.bias = static_cast<const bf16_t*>(bias);
    a.residual = static_cast<const bf16_t*>(residual);
    a.tile_rows = plan.tile_rows;
    a.row_tiles = plan.row_tiles;
    a.col_tiles = ceil_div(a.pair ? 2 * N : N, kForms[plan.form].cols);
    if (a.col_tiles * a.row_tiles * a.ksplit >= ((int64_t)1 << 31)) return SNGGUF_E_BADSHAPE;
    int rc = SNGGUF_E_BADTYPE;
#define SNGGUF_GO(QT) if (qtype == QT) rc = launch_mid_type<QT>(a, plan.form, plan.mt, numerics, stream);
    SNGGUF_MID_TYPES(SNGGUF_GO)
#undef SNGGUF_GO
    if (rc != SNGGUF_OK || plan.slices == 1) return rc;
    if (a.pair)
        return launch_splitk_reduce_gated(partial, partial + (int64_t)plan.slices * M * N, plan.slices, M, N, a.y, stream);
    GemmArgs g{};
    g.y = a.y;
    g.M = M; g.N = N; g.K = K;
    g.bias[0] = a.bias;
    g.residual = a.residual;
    g.partial = partial;
    g.ksplit = plan.slices;
    return launch_splitk_reduce(g, nullptr, M, stream);
}

}  // namespace sngguf
