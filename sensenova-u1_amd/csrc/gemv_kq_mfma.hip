// Decode GEMV on the matrix cores (K % 256 == 0): the K-quants Q2_K .. Q6_K, one 256-element
// super-block per step, and the 32-element formats Q4_0, Q4_1, Q5_0, Q5_1, Q8_0, eight blocks per
// step.  Up to 16 activation rows are one matrix operand; 17 .. 64 rows, where gemm_mid.hip's kernel is estimated to be
// slower (decode_kernel_us), use MT = 2 .. 4 operands per decoded weight fragment, so the weights are still fetched and
// decoded once.  (Q8_0 with at most
// 16 rows has faster kernels of its own.)
//
// Same shape as the Q8_0 kernel: a workgroup owns R * 16 weight rows (for the SiLU-gated pair the
// same rows of the gate and of the up matrix, on separate wavefronts), its wavefronts split K by
// super-blocks and add their partial sums through LDS at the end.  Per wavefront and super-block
// (256 elements of each row):
//   * the packed bytes of the R * 16 rows are fetched with 16-byte loads, consecutive lanes walking
//     along a row, one super-block ahead, and dropped into the wavefront's private LDS slab.  Q4_K
//     and Q5_K super-blocks (144 / 176 bytes) are 16-byte aligned; Q6_K super-blocks (210 bytes) are only 2-byte
//     aligned and are fetched as 13 unaligned 16-byte pieces plus the 2-byte scale, which never
//     touches a byte outside the super-block and puts every field at an aligned LDS address; Q2_K
//     (84 bytes) and Q3_K (110 bytes) take their last piece from the last 16 bytes of the
//     super-block, so it overlaps the piece before it in memory but not in the slab;
//   * lane (r = lane % 16, g = lane / 16) decodes, for each 32-element sub-block j, elements
//     8 g .. 8 g + 7 of row r to bf16 (rounding chain by numerics mode) as the A operand of
//     v_mfma_f32_16x16x32_bf16; the B operand is x[m = lane % 16][256 s + 32 j + 8 g ..].  With R = 2
//     one activation fragment feeds two row groups, which halves the activation traffic per
//     packed byte at M = 16.
// Nothing dequantized is written to memory.

#include "kq_decode.hpp"
#include "sngguf_common.hpp"

#include <type_traits>

namespace sngguf {

namespace {

// XN (MT = 1 only): the B fragments come from LDS.  Each wavefront stages the K range it works on (all M rows)
// behind the slabs.  With `gamma` set, RMSNorm(x) with weight `gamma` is what gets contracted (see rmsnorm_piece):
// the workgroup adds up the sums of squares and every wavefront normalizes its own share in place.  Without it
// the rows are staged as they are, which takes the eight activation requests per step off the vector memory
// path (worth it for Q6_K, whose unaligned slab pieces already load that path most).
template <int QT, int NUM, int R, bool GATED, int WMAX, int MT, bool XN = false>
__global__ __launch_bounds__(64 * WMAX) void gemv_kq_mfma_kernel(const bf16_t* __restrict__ x, int M,
                                                                 const uint8_t* __restrict__ qa,
                                                                 const uint8_t* __restrict__ qb, int64_t N, int64_t K,
                                                                 const bf16_t* __restrict__ bias, const bf16_t* residual, bf16_t* __restrict__ y,
                                                                 const bf16_t* __restrict__ gamma, float eps, uint64_t* __restrict__ amax,
                                                                 const bf16_t* __restrict__ gate) {
    static_assert(!XN || MT == 1, "the fused norm is for at most 16 rows");
    typedef Slab<QT> S;
    constexpr int kRows = 16 * R;
    constexpr int kPieces = kRows * S::pieces;
    constexpr int kLoads = (kPieces + 63) / 64;
    constexpr int kSlab = kRows * S::stride;
    constexpr bool kQ6 = QT == SNGGUF_TYPE_Q6_K;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int waves = blockDim.x >> 6;
    const int W = GATED ? waves >> 1 : waves;  // wavefronts that share one row group's K
    const int kw = GATED ? (wave >= W ? wave - W : wave) : wave;
    const uint8_t* __restrict__ q = (GATED && wave >= W) ? qb : qa;
    const int r = lane & 15, g = lane >> 4;
    const half4_t ident = identity_row(lane);
    const int64_t nsb = K >> 8;
    const int64_t row_bytes = nsb * S::ts;
    const int64_t n0 = (int64_t)blockIdx.x * kRows;
    const int s0 = (int)((int64_t)kw * nsb / W), s1 = (int)((int64_t)(kw + 1) * nsb / W);

    // piece f = lane + 64 i: 16 bytes at 16 (f % pieces) of row f / pieces
    uint32_t off[kLoads], dst[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; i++) {
        const int f = lane + 64 * i;
        const bool ok = f < kPieces;
        const int fr = ok ? f / S::pieces : 0, fp = ok ? f % S::pieces : 0;
        int64_t n = n0 + fr;
        if (n >= N) n = N - 1;  // rows past the end are decoded from the last row and never stored
        off[i] = (uint32_t)((n - n0) * row_bytes + (fp == S::pieces - 1 ? S::last_src : 16 * fp));
        dst[i] = (uint32_t)(fr * S::stride + 16 * fp);
    }
    const bool tail_lane = lane + 64 * (kLoads - 1) < kPieces;
    // Q6_K: lane l < 16 R also fetches the fp16 scale (bytes 208, 209) of row l
    uint32_t doff = 0;
    if constexpr (kQ6) {
        int64_t n = n0 + (lane < kRows ? lane : 0);
        if (n >= N) n = N - 1;
        doff = (uint32_t)((n - n0) * row_bytes + 208);
    }
    const uint8_t* __restrict__ base = q + n0 * row_bytes;
    uint8_t* slab = lds + wave * kSlab;

    f32x4_t acc[R][MT];
#pragma unroll
    for (int rg = 0; rg < R; rg++)
#pragma unroll
        for (int t = 0; t < MT; t++) acc[rg][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    u32x4_t pre[kLoads];
    uint16_t pre_d = 0;
    auto fetch = [&](int s) {
        const uint8_t* p = base + (int64_t)s * S::ts;
#pragma unroll
        for (int i = 0; i < kLoads - 1; i++) pre[i] = ld_piece<S::align>(p + off[i]);
        if (tail_lane) pre[kLoads - 1] = ld_piece<S::align>(p + off[kLoads - 1]);
        if constexpr (kQ6) {
            if (lane < kRows) pre_d = ld_u16(p + doff);
        }
    };
    // Lane (r, g) supplies column r of B operand t, i.e. activation row 16 t + r.  Rows >= M are never
    // stored, so those lanes re-read the last activation row instead of being masked.
    const bf16_t* xrow[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) xrow[t] = x + (int64_t)(16 * t + r < M ? 16 * t + r : M - 1) * K + 8 * g;

    // Activations are buffered by half super-blocks (four fragments): `xa` holds the first half of
    // the current super-block on entry; the second half is requested into `xb` before the first is
    // used, and the first half of the next super-block into `xa` before the second is used, so each
    // request has half a step of decode work to cover its latency.
    // XN: this wavefront's normalized activations, [M][xrow_b bytes]; the fragment of super-block s, half, j of
    // row m sits at byte ((s - s0) * 8 + 4 * half + j) * 64 + 16 g of row m
    const int xrow_b = XN ? (int)((nsb + W - 1) / W) * 512 + 16 : 0;
    uint8_t* xw = lds + waves * kSlab + wave * (M * xrow_b);
    const uint8_t* xwrow = xw + (r < M ? r : M - 1) * xrow_b + 16 * g;
    auto load_x = [&](int s, int half, u32x4_t (&dstx)[MT][4]) {
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if constexpr (XN) dstx[t][j] = *reinterpret_cast<const u32x4_t*>(xwrow + ((s - s0) * 8 + 4 * half + j) * 64);
                else dstx[t][j] = *reinterpret_cast<const u32x4_t*>(xrow[t] + ((int64_t)s * 8 + 4 * half + j) * 32);
            }
    };
    u32x4_t xa[MT][4], xb[MT][4];
    auto step = [&](int s) {
#pragma unroll
        for (int i = 0; i < kLoads - 1; i++) *reinterpret_cast<u32x4_t*>(slab + dst[i]) = pre[i];
        if (tail_lane) *reinterpret_cast<u32x4_t*>(slab + dst[kLoads - 1]) = pre[kLoads - 1];
        if constexpr (kQ6) {
            if (lane < kRows) *reinterpret_cast<uint16_t*>(slab + lane * S::stride + 208) = pre_d;
        }
        load_x(s, 1, xb);
        if (s + 1 < s1) fetch(s + 1);
#pragma unroll
        for (int rg = 0; rg < R; rg++) {
            const uint8_t* row = slab + (16 * rg + r) * S::stride;
            auto emit = [&](int jj, const u32x4_t& a) {
#pragma unroll
                for (int t = 0; t < MT; t++)
                    acc[rg][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, xa[t][jj]), acc[rg][t], 0, 0, 0);
            };
            decode_half<QT, NUM, 0>(ident, row, g, emit);
        }
        if (s + 1 < s1) load_x(s + 1, 0, xa);
#pragma unroll
        for (int rg = 0; rg < R; rg++) {
            const uint8_t* row = slab + (16 * rg + r) * S::stride;
            auto emit = [&](int jj, const u32x4_t& a) {
#pragma unroll
                for (int t = 0; t < MT; t++)
                    acc[rg][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        __builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, xb[t][jj]), acc[rg][t], 0, 0, 0);
            };
            decode_half<QT, NUM, 1>(ident, row, g, emit);
        }
    };
    if constexpr (XN) {
        // the first slab is requested, then the activations are staged and normalized underneath it
        if (s0 < s1) fetch(s0);
        float* ssum = reinterpret_cast<float*>(lds + waves * kSlab + waves * (M * xrow_b));  // [M][waves]
        const int pieces = (s1 - s0) * 32;               // 16-byte pieces per row in this wavefront's K range
        const int64_t k0 = (int64_t)s0 * 256;
        if (!gamma) {
            // plain staging, four requests in flight per lane; a wavefront reads back only what it wrote itself
            for (int m = 0; m < M; m++)
                for (int c0 = lane; c0 < pieces; c0 += 256) {
                    u32x4_t v[4];
#pragma unroll
                    for (int u = 0; u < 4; u++)
                        if (c0 + 64 * u < pieces) v[u] = *reinterpret_cast<const u32x4_t*>(x + (int64_t)m * K + k0 + 8 * (c0 + 64 * u));
#pragma unroll
                    for (int u = 0; u < 4; u++)
                        if (c0 + 64 * u < pieces) *reinterpret_cast<u32x4_t*>(xw + m * xrow_b + 16 * (c0 + 64 * u)) = v[u];
                }
        }
        for (int m = 0; gamma && m < M; m++) {
            float ss = 0.f;
            for (int c = lane; c < pieces; c += 64) {
                const u32x4_t v = *reinterpret_cast<const u32x4_t*>(x + (int64_t)m * K + k0 + 8 * c);
                *reinterpret_cast<u32x4_t*>(xw + m * xrow_b + 16 * c) = v;
                ss += sumsq_piece(v);
            }
            ss = wave_sum(ss);
            if (lane == 0) ssum[m * waves + wave] = ss;
        }
        if (gamma) __syncthreads();   // (uniform over the workgroup)
        for (int m = 0; gamma && m < M; m++) {
            float tot = 0.f;
            for (int w = 0; w < W; w++) tot += ssum[m * waves + w];   // wavefronts [0, W) cover K once
            const float rstd = rms_rstd(tot, K, eps);
            for (int c = lane; c < pieces; c += 64) {
                u32x4_t* cell = reinterpret_cast<u32x4_t*>(xw + m * xrow_b + 16 * c);
                const u32x4_t gv = *reinterpret_cast<const u32x4_t*>(gamma + k0 + 8 * c);
                *cell = rmsnorm_piece(*cell, gv, rstd);
            }
        }
        if (s0 < s1) load_x(s0, 0, xa);
    } else if (s0 < s1) {
        load_x(s0, 0, xa);
        fetch(s0);
    }
    for (int s = s0; s < s1; s++) step(s);

    // ---- add the wavefronts' partial sums (the slabs are dead: reuse them) -------------------------
    __syncthreads();
    f32x4_t* red = reinterpret_cast<f32x4_t*>(lds);  // [waves][R][MT][64]
#pragma unroll
    for (int rg = 0; rg < R; rg++)
#pragma unroll
        for (int t = 0; t < MT; t++) red[((wave * R + rg) * MT + t) * 64 + lane] = acc[rg][t];
    __syncthreads();
    if constexpr (MT > 1) {
        // R * MT groups of sums: one wavefront each (one wavefront alone would walk through all of them, 8 R MT reads, while
        // the rest of the workgroup has left: with the gated epilogue below, 40 rows of an 8B layer in Q8_0 130 against
        // 142 us).  Layout of a group as below, sums added in the same order.
        for (int i = wave; i < R * MT; i += waves) {
            const int rg = i / MT, t = i - rg * MT, m = 16 * t + r;
            const int64_t n = n0 + 16 * rg + 4 * g, yi = (int64_t)m * N + n;
            if (m >= M || n >= N) continue;
            const bool whole = n + 3 < N && (N & 3) == 0;
            u32x2_t gv = {0u, 0u};
            if (gate) gv = *reinterpret_cast<const u32x2_t*>(gate + yi);   // requested ahead of the sums (N % 8 == 0: whole)
            f32x4_t sum = red[i * 64 + lane];
            for (int w = 1; w < W; w++) {
                const f32x4_t p = red[(w * R * MT + i) * 64 + lane];
                sum[0] += p[0]; sum[1] += p[1]; sum[2] += p[2]; sum[3] += p[3];
            }
            float o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int v = 0; v < 4; v++) {
                if (n + v >= N) continue;
                o[v] = add_residual(sum[v] + (bias ? bf16_to_f32(bias[n + v]) : 0.f), residual, yi + v);
                if (gate) {
                    // the up projection of a SiLU-gated pair: `gate` holds the gate projection's outputs, and the value is
                    // the rounded silu of those times the rounded output here, as the gated pair's own launch rounds
                    const float gt = (v & 1) ? bf16hi_to_f32(gv[v >> 1]) : bf16lo_to_f32(gv[v >> 1]);
                    o[v] = bf16_to_f32(f32_to_bf16(gt / (1.0f + expf(-gt)))) * bf16_to_f32(f32_to_bf16(o[v]));
                }
            }
            if (whole) {
                *reinterpret_cast<u32x2_t*>(y + yi) = u32x2_t{pack_bf16(o[0], o[1]), pack_bf16(o[2], o[3])};
            } else {
#pragma unroll
                for (int v = 0; v < 4; v++)
                    if (n + v < N) y[yi + v] = f32_to_bf16(o[v]);
            }
        }
        return;
    }
    if (wave != 0) return;
    // D[i][j]: j = lane % 16 is the activation row (of operand t), register v holds weight row 4 * (lane / 16) + v
#pragma unroll
    for (int t = 0; t < MT; t++) {
        const int m = 16 * t + r;
        if (m >= M) continue;
        uint64_t best = 0;   // arg-max form: best (value, column) of this workgroup's rows for activation row m
#pragma unroll
        for (int rg = 0; rg < R; rg++) {
            f32x4_t sum = red[(rg * MT + t) * 64 + lane];
            for (int w = 1; w < W; w++) {
                const f32x4_t p = red[((w * R + rg) * MT + t) * 64 + lane];
                sum[0] += p[0]; sum[1] += p[1]; sum[2] += p[2]; sum[3] += p[3];
            }
            const int64_t n = n0 + 16 * rg + 4 * g;
            float o[4];
            if constexpr (GATED) {
                f32x4_t up = red[((W * R + rg) * MT + t) * 64 + lane];
                for (int w = 1; w < W; w++) {
                    const f32x4_t p = red[(((W + w) * R + rg) * MT + t) * 64 + lane];
                    up[0] += p[0]; up[1] += p[1]; up[2] += p[2]; up[3] += p[3];
                }
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const float gt = bf16_to_f32(f32_to_bf16(sum[v]));
                    const float ut = bf16_to_f32(f32_to_bf16(up[v]));
                    const float sl = bf16_to_f32(f32_to_bf16(gt / (1.0f + expf(-gt))));
                    o[v] = sl * ut;
                }
            } else {
#pragma unroll
                for (int v = 0; v < 4; v++) o[v] = n + v < N ? add_residual(sum[v] + (bias ? bf16_to_f32(bias[n + v]) : 0.f), residual, (int64_t)m * N + n + v) : 0.f;
                if (amax) {
#pragma unroll
                    for (int v = 0; v < 4; v++)
                        if (n + v < N) best = u64_max(best, argmax_key(o[v], n + v));
                    continue;
                }
            }
            bf16_t* yr = y + (int64_t)m * N + n;
            if (n + 3 < N && (N & 3) == 0) {
                *reinterpret_cast<u32x2_t*>(yr) = u32x2_t{pack_bf16(o[0], o[1]), pack_bf16(o[2], o[3])};
            } else {
#pragma unroll
                for (int v = 0; v < 4; v++)
                    if (n + v < N) yr[v] = f32_to_bf16(o[v]);
            }
        }
        if constexpr (!GATED) {
            if (amax) argmax_store(best, g, amax, m, blockIdx.x, gridDim.x);
        }
    }
}

template <int QT, int NUM, int R>
int launch_r(const bf16_t* x, int M, const uint8_t* qa, const uint8_t* qb, int64_t N, int64_t K, const bf16_t* bias,
             const bf16_t* residual, bf16_t* y, bool gated, const bf16_t* gamma, float eps, hipStream_t stream, uint64_t* amax, const bf16_t* gate) {
    const int64_t groups = (N + 16 * R - 1) / (16 * R);
    const int nsb = (int)(K >> 8);
    const int mt = (M + 15) / 16;
    // wavefronts per row group: enough that the launch fills the chip (about 12 per compute unit),
    // at least one super-block each, at most 8 per workgroup; beyond 16 rows counted per 16 weight rows whatever R is
    const int64_t per_group = gated ? 2 : 1, counted = mt > 1 ? (N + 15) / 16 : groups;
    int64_t w = (256 * 12 + counted * per_group - 1) / (counted * per_group);
    if (w < 1) w = 1;
    // Q6_K from about 98300 columns on (fewer have two and more by the count above): two wavefronts with half of K each
    // (151936 x 4096, us against one wavefront: one row 132 / 148, two - each stages its half of them - 133 / 159, four
    // 141 / 145, sixteen 165 / 167; 100003 x 2048: one row 49 / 52, sixteen 60 / 63; four wavefronts gain less)
    if (QT == SNGGUF_TYPE_Q6_K && R == 2 && mt == 1 && w < 2) w = 2;
    if (w > nsb) w = nsb;
    // Beyond 16 rows at most four wavefronts per workgroup
    //  - with more workgroups than compute units: two operands and more leave room for eight wavefronts on a compute unit,
    //    so a workgroup of five to eight holds the next one back and a second round begins at 8193 columns (10240 x 4096,
    //    17 / 48 rows, us: Q8_0 21.3 / 32.2 against 27.7 / 37.0 with up to eight, Q5_0 20.4 / 30.2 against 31.3 / 37.5);
    //  - with exactly one workgroup each, rows of K of 8192 and more and enough activation rows: twice the run of K each
    //    (4096 x 12288, 40 rows: Q8_0 35.9 against 38.2 us, Q6_K 37.2 against 38.9).  With fewer rows the eight hide more of
    //    the decode (17 rows: Q4_K 20.3 against 21.6 us, Q5_0 21.3 against 24.0), longest in the formats with a fifth bit.
    constexpr int kFourFrom = QT == SNGGUF_TYPE_Q5_0 || QT == SNGGUF_TYPE_Q5_1 || QT == SNGGUF_TYPE_Q5_K ? 26 : 22;
    const bool four = mt > 1 && (groups > 256 || (groups == 256 && nsb >= 32 && M >= kFourFrom));
    const int64_t cap = gated || four ? 4 : 8;
    if (w > cap) w = cap;
    const int waves = (int)(gated ? 2 * w : w);
    const size_t slab = (size_t)waves * 16 * R * Slab<QT>::stride;
    const size_t red = (size_t)waves * R * mt * 64 * sizeof(f32x4_t);
    const dim3 grid((unsigned)groups), block((unsigned)(64 * waves));
    // Q6_K streams its activations from LDS too when one or two rows of them fit there and the matrix is large
    // (12288 x 4096 at M = 1: 13.6 against 15.3 us; the other formats and small matrices lose by it)
    const bool stage = QT == SNGGUF_TYPE_Q6_K && !gamma && M <= 2 && N * K >= ((int64_t)32 << 20) &&
                       (size_t)M * (2 * (size_t)K + 64) <= 36 * 1024;
    if (gamma || stage) {
        // slabs, then every wavefront's share of the activations ([M][xrow_b]), then [M][waves] sums of squares; the
        // caller keeps M (2 K + 64) within 36 KB
        if (mt > 1) return SNGGUF_E_BADSHAPE;
        const size_t xrow_b = (size_t)((nsb + w - 1) / w) * 512 + 16;
        const size_t staged = slab + (size_t)waves * M * xrow_b + (((size_t)4 * M * waves + 15) & ~(size_t)15);
        const size_t lds_norm = staged > red ? staged : red;
        if (lds_norm > 160 * 1024) return SNGGUF_E_BADSHAPE;
        // slabs of two row groups per wavefront plus the staged activations can pass the default dynamic-LDS limit:
        // raise it once per kernel instance
#define SNGGUF_LAUNCH_XN(G, WM)                                                                                        \
    do {                                                                                                               \
        static const hipError_t attr = hipFuncSetAttribute(                                                            \
            reinterpret_cast<const void*>(&gemv_kq_mfma_kernel<QT, NUM, R, G, WM, 1, true>),                            \
            hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);                                                    \
        if (attr != hipSuccess) return SNGGUF_E_LAUNCH;                                                                 \
        gemv_kq_mfma_kernel<QT, NUM, R, G, WM, 1, true><<<grid, block, lds_norm, stream>>>(x, M, qa, qb, N, K, bias,    \
                                                                                           residual, y, gamma, eps, amax, nullptr); \
    } while (0)
        if (gated) {
            if (waves <= 4) SNGGUF_LAUNCH_XN(true, 4);
            else SNGGUF_LAUNCH_XN(true, 8);
        } else {
            if (waves <= 4) SNGGUF_LAUNCH_XN(false, 4);
            else SNGGUF_LAUNCH_XN(false, 8);
        }
#undef SNGGUF_LAUNCH_XN
        return hipGetLastError() == hipSuccess ? SNGGUF_OK : SNGGUF_E_LAUNCH;
    }
    const size_t lds_bytes = slab > red ? slab : red;
#define SNGGUF_LAUNCH(G, WM, MT_) \
    gemv_kq_mfma_kernel<QT, NUM, R, G, WM, MT_><<<grid, block, lds_bytes, stream>>>(x, M, qa, qb, N, K, bias, residual, y, nullptr, 0.f, amax, gate)
    if (mt > 1) {
        // more than 16 activation rows: plain projections only.  The slabs of two row groups on eight wavefronts can pass
        // the default dynamic-LDS limit: raised once per kernel instance
        if (gated || mt > 4) return SNGGUF_E_BADSHAPE;
#define SNGGUF_LAUNCH_MT(MT_)                                                                                          \
    do {                                                                                                               \
        static const hipError_t attr = hipFuncSetAttribute(                                                            \
            reinterpret_cast<const void*>(&gemv_kq_mfma_kernel<QT, NUM, R, false, 8, MT_>),                            \
            hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);                                                    \
        if (attr != hipSuccess) return SNGGUF_E_LAUNCH;                                                                 \
        SNGGUF_LAUNCH(false, 8, MT_);                                                                                   \
    } while (0)
        if (mt == 2) SNGGUF_LAUNCH_MT(2);
        else if (mt == 3) SNGGUF_LAUNCH_MT(3);
        else SNGGUF_LAUNCH_MT(4);
#undef SNGGUF_LAUNCH_MT
    } else if (gated) {
        if (waves <= 4) SNGGUF_LAUNCH(true, 4, 1);
        else SNGGUF_LAUNCH(true, 8, 1);
    } else {
        if (waves <= 4) SNGGUF_LAUNCH(false, 4, 1);
        else SNGGUF_LAUNCH(false, 8, 1);
    }
#undef SNGGUF_LAUNCH
    return hipGetLastError() == hipSuccess ? SNGGUF_OK : SNGGUF_E_LAUNCH;
}

// Weight rows per workgroup (see launch_qt) as a function, so that the arg-max caller can size its slot array.
inline int rows_per_workgroup(int qtype, int64_t M, int64_t N) {
    if (M <= 16) return N >= 32768 ? 32 : 16;
    if (qtype == SNGGUF_TYPE_Q5_K && M > 48 && ((N > 8192 && N <= 12288) || (N > 16384 && N < 24576))) return 16;
    return N > 4096 ? 32 : 16;
}

template <int QT, int NUM>
int launch_qt(const bf16_t* x, int M, const uint8_t* qa, const uint8_t* qb, int64_t N, int64_t K, const bf16_t* bias,
              const bf16_t* residual, bf16_t* y, bool gated, const bf16_t* gamma, float eps, hipStream_t stream, uint64_t* amax, const bf16_t* gate) {
    // Up to 16 activation rows, two row groups per wavefront only when one per wavefront would already give far more
    // wavefronts than the chip holds (a vocabulary-sized projection): otherwise more, smaller workgroups spread more
    // evenly over the 256 compute units.  Beyond 16 rows what bounds the launch is the activation traffic - every
    // workgroup reads all of x, 16 rows a fragment - and two or more operands take so many registers that a compute unit
    // holds one workgroup of eight wavefronts: as soon as 16-row groups need a second round of workgroups (more than 256
    // of them), 32 rows per workgroup halve both.  40 rows, Q8_0 / Q4_K: 6144 x 4096 28.9 -> 20.3 / 26.7 -> 19.1 us,
    // 12288 x 4096 36.2 -> 31.9 / 34.2 -> 29.0 us; at 64 rows 39.8 -> 29.7 and 50.4 -> 47.3 us (Q8_0); where 16-row
    // groups fit one round it loses (4096 x 4096, 40 rows: 15.2 -> 18.9 us).  Measured for all ten formats at 1024 .. 151936
    // columns and 17 .. 64 rows: level to 1.9 times as fast, but for Q5_K beyond 48 rows, whose four operands and two row
    // groups do not fit the registers (45 of them go through memory): there one group stays where two leave compute units
    // waiting in their last round (49 rows, one / two groups, us: 10240 x 4096 40 / 45, 12288 x 4096 41 / 47, 20480 x 4096
    // 67 / 103, but 8192 x 4096 34 / 30, 14336 x 4096 53 / 49, 24576 x 4096 96 / 83).
    if (rows_per_workgroup(QT, M, N) == 32) return launch_r<QT, NUM, 2>(x, M, qa, qb, N, K, bias, residual, y, gated, gamma, eps, stream, amax, gate);
    return launch_r<QT, NUM, 1>(x, M, qa, qb, N, K, bias, residual, y, gated, gamma, eps, stream, amax, gate);
}

// ---- the SiLU-gated MLP of a decoder layer at decode sizes in ONE launch, K-quant weights ---------------------
// The organisation of mlp_q8_decode_kernel (gemv_q8_mfma.hip) with this file's decoders: 256 workgroups of twelve
// wavefronts, one per compute unit.  Phase A: workgroup b computes the gated activations of rows [48 b, +48) - three
// 16-row groups, each with four wavefronts as in the gated pair's own launch (gate / up x two K halves of eight
// super-blocks), the activations staged once per workgroup in LDS (normalized there if `gamma` is given) - and writes
// them as 8-byte words { two bf16, generation tag } with agent-scope stores, then the group's flag.  No barrier inside
// the phase: a wavefront leaves its partial sums in LDS and counts itself in for its row group; the group's storing
// wavefront waits for that count only.  Phase B: 16 rows of the down matrix, K = inter split over the twelve
// wavefronts, four super-blocks each; two of them are requested the moment the wavefront leaves phase A's loop, the
// other two when every wavefront of the workgroup has left it (a count in LDS; requested earlier, their traffic slows
// phase A's last wavefronts, which the whole device waits for), and all four wait as raw bytes in registers; the first is decoded into matrix-core operands
// while the activations are on their way.  Then the wavefront polls the flags of the 64 row groups its K range needs,
// reads the tagged words (every tag checked), contracts the decoded super-block, decodes and contracts the other three,
// and the twelve partial sums are added.  Bounded wait, status word, generation counter and workspace layout as in the
// Q8_0 kernel (MlpCtl).  Without `gamma` the gated activations are bit-identical to the gated pair's own launch (same
// fragments, same order of accumulation), and so is the output (the down projection's own launch splits K over eight
// wavefronts, not twelve: equal up to the order of twelve fp32 additions, which the tests allow for).
// The decode arithmetic, not memory, bounds these formats (phase A takes 15 us with its requests and 15 without them; 56.6
// MB are 10.5 us of memory): the launch is 0 - 5 % ahead of the two separate ones by device and down type (32.3 against 33.9
// us with a Q6_K down projection once the down projection's first requests are made behind phase A's epilogue instead of in
// front of it; 31.9 - 32.8 against 32.7 - 33.0 with Q4_K), where the Q8_0 kernel gains 10 %.  Since then, with the norm and
// Q6_K, one row, in a kernel trace of decode passes: 36.2 -> 33.7 us at best, 36.9 -> 35.0 in the mean; the staging without LDS round
// trips brings the first decoded super-block 2 us forward, the falling priorities the ends of both phases 1.5 us.  Two or four
// super-blocks requested ahead instead of one, both halves of a super-block decoded as one block, and Q4_K's quants taken as
// pairs with two instructions in eight fewer change nothing.
template <int QT>
struct SlabIo {
    typedef Slab<QT> S;
    static constexpr int kPieces = 16 * S::pieces;
    static constexpr int kLoads = (kPieces + 63) / 64;
    static constexpr int kSlab = 16 * S::stride;
    static constexpr bool kQ6 = QT == SNGGUF_TYPE_Q6_K;
    uint32_t off[kLoads], dst[kLoads];
    uint32_t doff;
    bool tail_lane;
    __device__ __forceinline__ void init(int lane, int64_t row_bytes) {
#pragma unroll
        for (int i = 0; i < kLoads; i++) {
            const int f = lane + 64 * i;
            const bool ok = f < kPieces;
            const int fr = ok ? f / S::pieces : 0, fp = ok ? f % S::pieces : 0;
            off[i] = (uint32_t)(fr * row_bytes + (fp == S::pieces - 1 ? S::last_src : 16 * fp));
            dst[i] = (uint32_t)(fr * S::stride + 16 * fp);
        }
        tail_lane = lane + 64 * (kLoads - 1) < kPieces;
        doff = (uint32_t)((lane < 16 ? lane : 0) * row_bytes + 208);
    }
    __device__ __forceinline__ void fetch(const uint8_t* __restrict__ base, int s, int lane, u32x4_t (&pre)[kLoads], uint16_t& pre_d) const {
        const uint8_t* p = base + (int64_t)s * S::ts;
#pragma unroll
        for (int i = 0; i < kLoads - 1; i++) pre[i] = ld_piece<S::align>(p + off[i]);
        // (lanes past the last piece request row 0's first again: a request that some lanes skip is one that the compiler
        // cannot count, and every wait behind it becomes a wait for all)
        pre[kLoads - 1] = ld_piece<S::align>(p + off[kLoads - 1]);
        if constexpr (kQ6) pre_d = ld_u16(p + doff);
    }
    __device__ __forceinline__ void store(uint8_t* slab, int lane, const u32x4_t (&pre)[kLoads], uint16_t pre_d) const {
#pragma unroll
        for (int i = 0; i < kLoads - 1; i++) *reinterpret_cast<u32x4_t*>(slab + dst[i]) = pre[i];
        if (tail_lane) *reinterpret_cast<u32x4_t*>(slab + dst[kLoads - 1]) = pre[kLoads - 1];
        if constexpr (kQ6) {
            if (lane < 16) *reinterpret_cast<uint16_t*>(slab + lane * S::stride + 208) = pre_d;
        }
    }
};

constexpr int kMlpKqWaves = 12;
// Super-blocks of the down matrix that a wavefront decodes into registers while it waits for the activations: one (32
// registers of operands beside a decoder's ~100 of temporaries is what 168 registers per lane hold; two spill).
#ifndef SNGGUF_MLPKQ_AHEAD
#define SNGGUF_MLPKQ_AHEAD 1
#endif
constexpr int kMlpKqSteps = 4;   // super-blocks of the down matrix per wavefront: inter = 12 x 4 x 256 (the launcher checks)
constexpr int kMlpKqHidden = 4096, kMlpKqRows = 2;   // the only hidden size and the most rows (mlp_kq_decode_fits)
static_assert(kMlpKqHidden / 8 <= 64 * kMlpKqWaves, "a thread stages at most 16 bytes of an activation row");

template <int QA, int QB>
struct MlpKqLds {
    // [12 slabs of phase A][x staged (M rows) + sums of squares][partial sums of phase A + counters][12 x (slab of phase B, two staged activation rows)]
    static constexpr int kSlabsA = kMlpKqWaves * SlabIo<QA>::kSlab;
    static constexpr int kWaveB = SlabIo<QB>::kSlab + 2 * kMlpKqSteps * 512;
    __host__ __device__ static size_t xs_bytes(int M, int64_t hidden, bool norm) {
        return (((size_t)M * (2 * (size_t)hidden + 64) + (norm ? (size_t)4 * M * kMlpKqWaves : 0)) + 255) & ~(size_t)255;
    }
    __host__ __device__ static size_t total(int M, int64_t hidden, bool norm) {
        return (size_t)kSlabsA + xs_bytes(M, hidden, norm) + (size_t)kMlpKqWaves * 64 * 16 + 64 + (size_t)kMlpKqWaves * kWaveB;
    }
};

template <int QA, int QB, int NUM>
__global__ __launch_bounds__(64 * kMlpKqWaves) void mlp_kq_decode_kernel(const bf16_t* __restrict__ x, int M, const uint8_t* __restrict__ q_gate,
                                                                         const uint8_t* __restrict__ q_up, const uint8_t* __restrict__ q_down,
                                                                         int64_t hidden, int64_t inter, const bf16_t* __restrict__ gamma, float eps,
                                                                         const bf16_t* residual, bf16_t* __restrict__ y, MlpCtl* ctl, uint64_t* ht,
                                                                         int spin_limit) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    typedef SlabIo<QA> IA;
    typedef SlabIo<QB> IB;
    typedef MlpKqLds<QA, QB> L;
    constexpr int kWaves = kMlpKqWaves, kSteps = kMlpKqSteps;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int bid = (int)blockIdx.x, nb = (int)gridDim.x;
    const int r = lane & 15, g = lane >> 4;
    const half4_t ident = identity_row(lane);
    // this launch's tag: nobody advances the generation before every workgroup, this one included, has finished
    const uint32_t tag = __hip_atomic_load(&ctl->gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u;

    uint8_t* const xs = lds + L::kSlabsA;
    const int64_t xs_stride = 2 * hidden + 64;
    f32x4_t* const red_a = reinterpret_cast<f32x4_t*>(xs + L::xs_bytes(M, hidden, gamma != nullptr));
    uint32_t* const cnt = reinterpret_cast<uint32_t*>(red_a + kWaves * 64);
    uint8_t* const slab_b = reinterpret_cast<uint8_t*>(cnt + 16) + wave * L::kWaveB;
    uint8_t* const xw = slab_b + IB::kSlab;   // [2][kSteps * 512] bytes

    // ---- phase A: row group 3 bid + grp, matrix mat (0 gate, 1 up), K half kh ----
    __builtin_amdgcn_s_setprio(2);
    const int grp = wave >> 2, lw = wave & 3, mat = lw >> 1, kh = lw & 1;
    const int nsb = (int)(hidden >> 8);
    const int sa0 = kh * (nsb >> 1), sa1 = sa0 + (nsb >> 1);
    const int64_t arow_bytes = (int64_t)nsb * IA::S::ts;
    const uint8_t* __restrict__ abase = (mat ? q_up : q_gate) + (int64_t)(3 * bid + grp) * 16 * arow_bytes;
    IA ia;
    ia.init(lane, arow_bytes);
    uint8_t* const slab_a = lds + wave * IA::kSlab;
    u32x4_t pre_a[IA::kLoads];
    uint16_t pre_ad = 0;
    if (tid < 16) cnt[tid] = 0;
    // the activations, staged once for the workgroup (normalized if gamma is given): a thread keeps its 16 bytes of each row
    // in registers across the sum of squares, and gamma's are on their way with them (one piece per thread and row: kMlpKqHidden,
    // kMlpKqRows)
    {
        const bool mine = tid < (int)(hidden >> 3);
        u32x4_t xv0 = {}, xv1 = {}, gv = {};
        if (mine) {
            xv0 = *reinterpret_cast<const u32x4_t*>(x + 8 * tid);
            if (M > 1) xv1 = *reinterpret_cast<const u32x4_t*>(x + hidden + 8 * tid);
            if (gamma != nullptr) gv = *reinterpret_cast<const u32x4_t*>(gamma + 8 * tid);
        }
        ia.fetch(abase, sa0, lane, pre_a, pre_ad);
        u32x4_t* const cell = reinterpret_cast<u32x4_t*>(xs + 16 * tid);
        u32x4_t* const cell1 = reinterpret_cast<u32x4_t*>(xs + xs_stride + 16 * tid);
        if (gamma != nullptr) {
            float* ssum = reinterpret_cast<float*>(xs + M * xs_stride);   // [M][waves]
            const float ss0 = wave_sum(mine ? sumsq_piece(xv0) : 0.f);
            if (lane == 0) ssum[wave] = ss0;
            if (M > 1) {
                const float ss1 = wave_sum(mine ? sumsq_piece(xv1) : 0.f);
                if (lane == 0) ssum[kWaves + wave] = ss1;
            }
            __syncthreads();
            float t0 = 0.f, t1 = 0.f;
            for (int w = 0; w < kWaves; w++) t0 += ssum[w];
            if (M > 1)
                for (int w = 0; w < kWaves; w++) t1 += ssum[kWaves + w];
            xv0 = rmsnorm_piece(xv0, gv, rms_rstd(t0, hidden, eps));
            if (M > 1) xv1 = rmsnorm_piece(xv1, gv, rms_rstd(t1, hidden, eps));
        }
        if (mine) {
            *cell = xv0;
            if (M > 1) *cell1 = xv1;
        }
        __syncthreads();
    }
    const bool has_x = r < M;
    const uint8_t* xsrow = xs + (has_x ? r : M - 1) * xs_stride + 16 * g;
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
    auto step_a = [&](int s, auto more) {
        ia.store(slab_a, lane, pre_a, pre_ad);
        if constexpr (decltype(more)::value) ia.fetch(abase, s + 1, lane, pre_a, pre_ad);
        const uint8_t* row = slab_a + r * IA::S::stride;
        auto emit0 = [&](int jj, const u32x4_t& a) {
            const u32x4_t xf = *reinterpret_cast<const u32x4_t*>(xsrow + (s * 8 + jj) * 64);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, xf), acc, 0, 0, 0);
        };
        decode_half<QA, NUM, 0>(ident, row, g, emit0);
        auto emit1 = [&](int jj, const u32x4_t& a) {
            const u32x4_t xf = *reinterpret_cast<const u32x4_t*>(xsrow + (s * 8 + 4 + jj) * 64);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, xf), acc, 0, 0, 0);
        };
        decode_half<QA, NUM, 1>(ident, row, g, emit1);
    };
    // A wavefront's priority falls as it gets on, a quarter of the loop at a time: the three wavefronts of a SIMD would
    // otherwise be served oldest first, and the last would run its second half alone, where its chains of dependent
    // instructions leave the SIMD idle (the wavefronts' ends lay 11 .. 19 us behind the start, now 13.5 .. 18).
    for (int s = sa0; s < sa1 - 1; s++) {
        switch ((s - sa0) * 4 / (sa1 - sa0)) {
            case 0: __builtin_amdgcn_s_setprio(3); break;
            case 1: __builtin_amdgcn_s_setprio(2); break;
            case 2: __builtin_amdgcn_s_setprio(1); break;
            default: __builtin_amdgcn_s_setprio(0); break;
        }
        step_a(s, std::true_type{});
    }
    step_a(sa1 - 1, std::false_type{});
    __builtin_amdgcn_s_setprio(3);

    // ---- phase B geometry: rows [16 bid, +16) of down, super-blocks [4 wave, +4) ----
    const int sb0 = wave * kSteps;
    const int64_t brow_bytes = (inter >> 8) * IB::S::ts;
    const uint8_t* __restrict__ bbase = q_down + (int64_t)bid * 16 * brow_bytes;
    IB ib;
    ib.init(lane, brow_bytes);
    u32x4_t raw[kSteps][IB::kLoads];
    uint16_t raw_d[kSteps] = {};
    // ---- phase A epilogue: partial sums, per-group count, the storing wavefront's SiLU and tagged stores; the down
    // projection's first requests come behind it, so that they do not queue in front of what other workgroups wait for ----
    red_a[wave * 64 + lane] = acc;
    if (lane == 0) __hip_atomic_fetch_add(cnt + grp, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (lw == 0) {
        while (__hip_atomic_load(cnt + grp, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) < 4u) __builtin_amdgcn_s_sleep(1);
        if (has_x) {
            // wavefronts 4 grp + {0, 1}: gate K halves, + {2, 3}: up K halves; D[i][j]: j = lane % 16 the activation row
            f32x4_t gs = red_a[(4 * grp) * 64 + lane], us = red_a[(4 * grp + 2) * 64 + lane];
            const f32x4_t g1 = red_a[(4 * grp + 1) * 64 + lane], u1 = red_a[(4 * grp + 3) * 64 + lane];
            float o[4];
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const float gt = bf16_to_f32(f32_to_bf16(gs[v] + g1[v]));
                const float ut = bf16_to_f32(f32_to_bf16(us[v] + u1[v]));
                const float sl = bf16_to_f32(f32_to_bf16(gt / (1.0f + expf(-gt))));
                o[v] = sl * ut;
            }
            const int64_t n = (int64_t)(3 * bid + grp) * 16 + 4 * g;
            uint64_t* yt = ht + (((int64_t)r * inter + n) >> 1);
            __hip_atomic_store(yt, (uint64_t)pack_bf16(o[0], o[1]) | ((uint64_t)tag << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(yt + 1, (uint64_t)pack_bf16(o[2], o[3]) | ((uint64_t)tag << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (lane == 0) __hip_atomic_store(&ctl->flags[3 * bid + grp], tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    ib.fetch(bbase, sb0, lane, raw[0], raw_d[0]);
    ib.fetch(bbase, sb0 + 1, lane, raw[1], raw_d[1]);
    // counted as having left the loop: the other two steps are requested when that count is full
    uint32_t* const left_a = cnt + 8;
    if (lane == 0) __hip_atomic_fetch_add(left_a, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);

    __builtin_amdgcn_s_setprio(0);

    // ---- phase B: decode the first kAhead super-blocks into matrix-core operands while the activations are on their
    // way (what the register file holds beside a decoder's temporaries); the others wait as raw bytes in registers ----
    constexpr int kAhead = SNGGUF_MLPKQ_AHEAD;
    u32x4_t afrag[kAhead > 0 ? kAhead * 8 : 1];
    const uint8_t* const brow = slab_b + r * IB::S::stride;
    auto decode = [&](int i) {
        ib.store(slab_b, lane, raw[i], raw_d[i]);
        auto e0 = [&](int jj, const u32x4_t& a) { afrag[i * 8 + jj] = a; };
        decode_half<QB, NUM, 0>(ident, brow, g, e0);
        auto e1 = [&](int jj, const u32x4_t& a) { afrag[i * 8 + 4 + jj] = a; };
        decode_half<QB, NUM, 1>(ident, brow, g, e1);
    };
    if constexpr (kAhead > 0) decode(0);
    if constexpr (kAhead > 1) decode(1);
    // every wavefront of the workgroup has left phase A's loop: now the other two steps' traffic
    while (__hip_atomic_load(left_a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < (uint32_t)kWaves) __builtin_amdgcn_s_sleep(1);
    ib.fetch(bbase, sb0 + 2, lane, raw[2], raw_d[2]);
    ib.fetch(bbase, sb0 + 3, lane, raw[3], raw_d[3]);
    if constexpr (kAhead > 2) decode(2);
    if constexpr (kAhead > 3) decode(3);

    // ---- wait for this wavefront's K range of the activations: flags of its 64 row groups, then the tagged words ----
    constexpr int xrow_b = kSteps * 512;
    {
        const int pairs = kSteps * 64;                    // 16-byte pairs of words per row in this wavefront's K range
        const int64_t w0 = (int64_t)sb0 * 128;            // first word of the range within a row
        const int64_t row_words = inter >> 1;
        const int g0 = sb0 * 16, ng = kSteps * 16;        // row groups of 16 outputs
        int polls = 0;
        bool gave_up = false;
        for (;;) {
            bool all = true;
            for (int j = lane; j < ng; j += 64) all = all && __hip_atomic_load(&ctl->flags[g0 + j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == tag;
            if (__builtin_amdgcn_ballot_w64(!all) == 0) break;
            if (++polls > spin_limit) { gave_up = true; break; }
            __builtin_amdgcn_s_sleep(2);
        }
        for (;;) {
            bool all = true;
            for (int m = 0; m < M; m++)
                for (int c = lane; c < pairs; c += 64) {
                    const uint64_t* src = ht + (int64_t)m * row_words + w0 + 2 * c;
                    const uint64_t a = __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    const uint64_t b = __hip_atomic_load(src + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    all = all && (uint32_t)(a >> 32) == tag && (uint32_t)(b >> 32) == tag;
                    *reinterpret_cast<uint64_t*>(xw + m * xrow_b + 8 * c) = (uint64_t)(uint32_t)a | (b << 32);
                }
            if (gave_up || __builtin_amdgcn_ballot_w64(!all) == 0) break;
            if (++polls > spin_limit) { gave_up = true; break; }
        }
        if (gave_up && lane == 0) __hip_atomic_store(&ctl->status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // ---- contract, add the twelve partial sums, residual, store ----
    __builtin_amdgcn_s_setprio(3);
    f32x4_t yacc = {0.f, 0.f, 0.f, 0.f};
    const uint8_t* xwrow = xw + (has_x ? r : M - 1) * xrow_b + 16 * g;
#pragma unroll
    for (int i = 0; i < kAhead * 8; i++) {
        const u32x4_t xf = *reinterpret_cast<const u32x4_t*>(xwrow + i * 64);
        yacc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, afrag[i]), __builtin_bit_cast(bf16x8_t, xf), yacc, 0, 0, 0);
    }
    auto decode_contract = [&](int i) {
        ib.store(slab_b, lane, raw[i], raw_d[i]);
        auto e0 = [&](int jj, const u32x4_t& a) {
            const u32x4_t xf = *reinterpret_cast<const u32x4_t*>(xwrow + (i * 8 + jj) * 64);
            yacc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, xf), yacc, 0, 0, 0);
        };
        decode_half<QB, NUM, 0>(ident, brow, g, e0);
        auto e1 = [&](int jj, const u32x4_t& a) {
            const u32x4_t xf = *reinterpret_cast<const u32x4_t*>(xwrow + (i * 8 + 4 + jj) * 64);
            yacc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, xf), yacc, 0, 0, 0);
        };
        decode_half<QB, NUM, 1>(ident, brow, g, e1);
    };
    if constexpr (kAhead <= 0) decode_contract(0);
    if constexpr (kAhead <= 1) decode_contract(1);
    __builtin_amdgcn_s_setprio(2);   // (as in phase A's loop)
    if constexpr (kAhead <= 2) decode_contract(2);
    __builtin_amdgcn_s_setprio(1);
    if constexpr (kAhead <= 3) decode_contract(3);
    __builtin_amdgcn_s_setprio(3);
    __syncthreads();   // every wavefront is past phase A's epilogue: its partial-sum area is free
    red_a[wave * 64 + lane] = yacc;
    __syncthreads();
    if (wave == 0 && has_x) {
        f32x4_t sum = red_a[lane];
        for (int w = 1; w < kWaves; w++) {
            const f32x4_t t = red_a[w * 64 + lane];
            sum[0] += t[0]; sum[1] += t[1]; sum[2] += t[2]; sum[3] += t[3];
        }
        const int64_t n = (int64_t)bid * 16 + 4 * g;
        float o[4];
#pragma unroll
        for (int v = 0; v < 4; v++) o[v] = add_residual(sum[v], residual, (int64_t)r * hidden + n + v);
        *reinterpret_cast<u32x2_t*>(y + (int64_t)r * hidden + n) = u32x2_t{pack_bf16(o[0], o[1]), pack_bf16(o[2], o[3])};
    }
    if (tid == 0) {
        const uint32_t old = __hip_atomic_fetch_add(&ctl->done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (old == (uint32_t)nb - 1u) {
            __hip_atomic_store(&ctl->done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&ctl->gen, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

template <int QA, int QB, int NUM>
int launch_mlp_kq(const void* x, int M, const void* gamma, float eps, const void* q_gate, const void* q_up, const void* q_down, int64_t hidden,
                  int64_t inter, const void* residual, void* y, void* workspace, int spin_limit, hipStream_t stream) {
    const size_t lds_bytes = MlpKqLds<QA, QB>::total(M, hidden, gamma != nullptr);
    if (lds_bytes > 160 * 1024) return SNGGUF_E_BADSHAPE;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&mlp_kq_decode_kernel<QA, QB, NUM>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (attr != hipSuccess) return SNGGUF_E_LAUNCH;
    MlpCtl* ctl = static_cast<MlpCtl*>(workspace);
    uint64_t* h = reinterpret_cast<uint64_t*>(static_cast<uint8_t*>(workspace) + kMlpCtlBytes);
    const int limit = spin_limit == 0 ? 1 << 20 : spin_limit < 0 ? 0 : spin_limit;
    mlp_kq_decode_kernel<QA, QB, NUM><<<dim3((unsigned)(inter / 48)), dim3(64 * kMlpKqWaves), lds_bytes, stream>>>(
        static_cast<const bf16_t*>(x), M, static_cast<const uint8_t*>(q_gate), static_cast<const uint8_t*>(q_up),
        static_cast<const uint8_t*>(q_down), hidden, inter, static_cast<const bf16_t*>(gamma), eps, static_cast<const bf16_t*>(residual),
        static_cast<bf16_t*>(y), ctl, h, limit);
    return hipGetLastError() == hipSuccess ? SNGGUF_OK : SNGGUF_E_LAUNCH;
}

}  // namespace

// The K-quant mixes the one-launch MLP takes: Q4_K gate / up with a Q6_K or Q4_K down projection (the "Q4_K_M" recipe),
// hidden 4096, inter 12288 (48 rows of gate / up and 16 rows of down per workgroup, 12 x 4 super-blocks per down row),
// one or two rows, one resident workgroup per compute unit.
bool mlp_kq_decode_fits(int qtype_gate_up, int qtype_down, int64_t M, int64_t hidden, int64_t inter) {
    if (qtype_gate_up != SNGGUF_TYPE_Q4_K || (qtype_down != SNGGUF_TYPE_Q6_K && qtype_down != SNGGUF_TYPE_Q4_K)) return false;
    if (M < 1 || M > kMlpKqRows || hidden != kMlpKqHidden || inter != kMlpKqWaves * kMlpKqSteps * 256) return false;
    static const int cus = [] {
        int dev = 0, n = 0, per_cu = 0;
        if (hipGetDevice(&dev) != hipSuccess) return 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
        const void* k = reinterpret_cast<const void*>(&mlp_kq_decode_kernel<SNGGUF_TYPE_Q4_K, SNGGUF_TYPE_Q6_K, 1>);
        if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) != hipSuccess) return 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, mlp_kq_decode_kernel<SNGGUF_TYPE_Q4_K, SNGGUF_TYPE_Q6_K, 1>, 64 * kMlpKqWaves,
                                                         160 * 1024) != hipSuccess)
            return 0;
        return per_cu >= 1 ? n : 0;
    }();
    return cus >= inter / 48;
}

int launch_mlp_kq_decode(const void* x, int64_t M, const void* gamma, float eps, const void* q_gate, const void* q_up, const void* q_down,
                         int qtype_down, int64_t hidden, int64_t inter, const void* residual, void* y, void* workspace, int numerics,
                         int spin_limit, hipStream_t stream) {
    if (!mlp_kq_decode_fits(SNGGUF_TYPE_Q4_K, qtype_down, M, hidden, inter)) return SNGGUF_E_BADSHAPE;
#define SNGGUF_GO(QB, NUMV) \
    return launch_mlp_kq<SNGGUF_TYPE_Q4_K, QB, NUMV>(x, (int)M, gamma, eps, q_gate, q_up, q_down, hidden, inter, residual, y, workspace, spin_limit, stream)
    if (qtype_down == SNGGUF_TYPE_Q6_K) {
        if (numerics == SNGGUF_NUM_GGML_FP32) SNGGUF_GO(SNGGUF_TYPE_Q6_K, 0);
        SNGGUF_GO(SNGGUF_TYPE_Q6_K, 1);
    }
    if (numerics == SNGGUF_NUM_GGML_FP32) SNGGUF_GO(SNGGUF_TYPE_Q4_K, 0);
    SNGGUF_GO(SNGGUF_TYPE_Q4_K, 1);
#undef SNGGUF_GO
}

// Workgroups of a plain decode launch = (value, column) slots per activation row that its arg-max form writes.
int64_t gemv_argmax_slots(int qtype, int64_t M, int64_t N) {
    const int64_t rows = qtype == SNGGUF_TYPE_Q8_0 ? 16 : rows_per_workgroup(qtype, M, N);   // (Q8_0 has kernels of its own)
    return (N + rows - 1) / rows;
}

// 1 <= M <= 64 (SiLU-gated pair: M <= 16), K % 256 == 0, 16-byte aligned x and q (checked by the caller).  `gamma`
// (K bf16, 16-byte aligned) switches the fused RMSNorm on; the caller keeps M (2 K + 64) <= 36 KB then.  `gate` ([M][N],
// 8-byte aligned, M > 16, N % 4 == 0, no bias or residual): y = silu(gate) * projection.
int launch_gemv_kq_mfma(const void* x, int64_t M, const void* qa, const void* qb, int qtype, int64_t N, int64_t K,
                        const void* bias, const void* residual, void* y, int numerics, bool gated, hipStream_t stream,
                        const void* gamma, float eps, uint64_t* amax, const void* gate) {
    if (gate && (gated || M <= 16 || N % 4 != 0 || bias || residual)) return SNGGUF_E_BADSHAPE;
    const bf16_t* gt = static_cast<const bf16_t*>(gate);
    if (amax && (gated || M > 16)) return SNGGUF_E_BADSHAPE;
    const bf16_t* gp = static_cast<const bf16_t*>(gamma);
    const bf16_t* xp = static_cast<const bf16_t*>(x);
    const uint8_t* a = static_cast<const uint8_t*>(qa);
    const uint8_t* b = static_cast<const uint8_t*>(qb);
    const bf16_t* bp = static_cast<const bf16_t*>(bias);
    const bf16_t* rp = static_cast<const bf16_t*>(residual);
    bf16_t* yp = static_cast<bf16_t*>(y);
#define SNGGUF_CASE(QT)                                                                                          \
    if (qtype == QT) {                                                                                           \
        if (numerics == SNGGUF_NUM_GGML_FP32)                                                                    \
            return launch_qt<QT, SNGGUF_NUM_GGML_FP32>(xp, (int)M, a, b, N, K, bp, rp, yp, gated, gp, eps, stream, amax, gt);          \
        if (numerics == SNGGUF_NUM_UPSTREAM_FP16)                                                                \
            return launch_qt<QT, SNGGUF_NUM_UPSTREAM_FP16>(xp, (int)M, a, b, N, K, bp, rp, yp, gated, gp, eps, stream, amax, gt);      \
        return SNGGUF_E_BADTYPE;                                                                                 \
    }
    SNGGUF_CASE(SNGGUF_TYPE_Q4_0)
    SNGGUF_CASE(SNGGUF_TYPE_Q4_1)
    SNGGUF_CASE(SNGGUF_TYPE_Q5_0)
    SNGGUF_CASE(SNGGUF_TYPE_Q5_1)
    SNGGUF_CASE(SNGGUF_TYPE_Q8_0)
    SNGGUF_CASE(SNGGUF_TYPE_Q2_K)
    SNGGUF_CASE(SNGGUF_TYPE_Q3_K)
    SNGGUF_CASE(SNGGUF_TYPE_Q4_K)
    SNGGUF_CASE(SNGGUF_TYPE_Q5_K)
    SNGGUF_CASE(SNGGUF_TYPE_Q6_K)
#undef SNGGUF_CASE
    return SNGGUF_E_BADTYPE;
}

}  // namespace sngguf
