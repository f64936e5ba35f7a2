// Standalone block dequantize: packed GGUF rows -> fp32 / fp16 / bf16 rows.
// One thread decodes eight consecutive elements, so a wavefront reads one contiguous run of
// packed bytes and writes one contiguous run of 512 outputs; the kernel is bound by the
// output stream (4 bytes out per ~1 byte in for fp32).  Q4_K and Q6_K to 16-bit outputs in the
// fp16 rounding chain go by whole quant bytes instead (HalfChain).
#include "sngguf_common.hpp"

namespace sngguf {

template <int OUT>
__device__ __forceinline__ void store8(void* __restrict__ out, int64_t idx, const float (&w)[8]) {
    if constexpr (OUT == SNGGUF_OUT_F32) {
        f32x4_t* o = reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(out) + idx);
        o[0] = f32x4_t{w[0], w[1], w[2], w[3]};
        o[1] = f32x4_t{w[4], w[5], w[6], w[7]};
    } else if constexpr (OUT == SNGGUF_OUT_F16) {
        u32x4_t v;
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = (uint32_t)f32_to_f16(w[2 * i]) | ((uint32_t)f32_to_f16(w[2 * i + 1]) << 16);
        *reinterpret_cast<u32x4_t*>(reinterpret_cast<uint16_t*>(out) + idx) = v;
    } else {
        u32x4_t v;
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = pack_bf16(w[2 * i], w[2 * i + 1]);
        *reinterpret_cast<u32x4_t*>(reinterpret_cast<uint16_t*>(out) + idx) = v;
    }
}

// Q4_K and Q6_K in the fp16 rounding chain, decoded as packed halves: the chain's last fp16 value IS the fp16 output
// (and what bf16 is rounded from), so nothing is widened to fp32 on the way.  Q4_K: R(R(D q) - DM) with D = R(d sc),
// DM = R(dmin m); Q6_K: R(D q) with D = R(d scale).
//
// One thread takes every element that eight consecutive quant bytes of a super-block hold: 2 x 8 for Q4_K (both nibbles),
// 4 x 8 for Q6_K (both nibbles of two byte runs that share their upper bits), each run of eight one 16-byte store.  Every
// quant byte is then requested once and a super-block's header once per 16 or 32 outputs, where one thread per eight
// consecutive elements asked for every byte twice (upper bits: four times) and for the header with each.  Four lanes fill
// 64 consecutive output bytes per store.  Bound by the output stream: three 12288 x 4096 Q4_K matrices to fp16 97.5 -> 78.8 us,
// 4.9 TB/s of the 5.4 that a large copy reaches; Q6_K 1.10 times as fast at that size, level below 1024 rows.
template <int QT>
struct HalfChain {
    static_assert(QT == SNGGUF_TYPE_Q4_K || QT == SNGGUF_TYPE_Q6_K, "packed decode exists for Q4_K and Q6_K");
    static constexpr int runs = QT == SNGGUF_TYPE_Q4_K ? 2 : 4;   // runs of eight elements, 32 elements apart
    static constexpr int items = 256 / (8 * runs);                // threads per super-block

    // Item `it` of super-block `blk`: runs -> v[run]; returns the first run's first element within the super-block.
    static __device__ __forceinline__ int decode(const uint8_t* __restrict__ blk, int it, u32x4_t (&v)[runs]) {
        typedef Num<SNGGUF_NUM_UPSTREAM_FP16> A;
        const int c = it >> 2, l0 = 8 * (it & 3);
        if constexpr (QT == SNGGUF_TYPE_Q4_K) {
            const u32x4_t head = *reinterpret_cast<const u32x4_t*>(blk);   // d, dmin, 12 scale bytes (144-byte blocks: aligned)
            const u32x2_t qs = *reinterpret_cast<const u32x2_t*>(blk + 16 + 32 * c + l0);
            const _Float16 d = A::scale((uint16_t)(head[0] & 0xFFFF)), dmin = A::scale((uint16_t)(head[0] >> 16));
            const half2_t k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
#pragma unroll
            for (int hi = 0; hi < 2; hi++) {
                uint32_t sc, mn;
                q4k_scale_min(head[1], head[2], head[3], 2 * c + hi, sc, mn);
                const _Float16 D = d * A::integer((int)sc), DM = dmin * A::integer((int)mn);
                const half2_t D2 = {D, D}, M2 = {DM, DM};
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const uint32_t n = (qs[i] >> (4 * hi)) & 0x0F0F0F0Fu;
                    // 0x6400 | n is the half 1024 + n
                    const half2_t q01 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, n, 0x04010400u)) - k1024;
                    const half2_t q23 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, n, 0x04030402u)) - k1024;
                    v[hi][2 * i] = __builtin_bit_cast(uint32_t, q01 * D2 - M2);       // two roundings each (no contraction)
                    v[hi][2 * i + 1] = __builtin_bit_cast(uint32_t, q23 * D2 - M2);
                }
            }
            return 64 * c + l0;
        } else {
            // (210-byte blocks: every field is 2-byte aligned only)
            uint32_t ql[2][2], qh[2], sc[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                ql[0][i] = ld_u32_a2(blk + 64 * c + l0 + 4 * i);
                ql[1][i] = ld_u32_a2(blk + 64 * c + 32 + l0 + 4 * i);
                qh[i] = ld_u32_a2(blk + 128 + 32 * c + l0 + 4 * i);
                sc[i] = ld_u32_a2(blk + 192 + 8 * c + 4 * i);
            }
            const _Float16 d = A::scale(ld_u16(blk + 208));
            const half2_t k1056 = {(_Float16)1056.0f, (_Float16)1056.0f};   // 1024 + the quant's offset of 32
#pragma unroll
            for (int quad = 0; quad < 4; quad++) {
                // sub-scale of element 32 quad + l0 of the half: byte 2 quad + l0 / 16 of its eight
                const int byte = 2 * (quad & 1) + (l0 >> 4);
                const _Float16 D = d * A::integer((int)(int8_t)((sc[quad >> 1] >> (8 * byte)) & 0xFFu));
                const half2_t D2 = {D, D};
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const uint32_t lo = (ql[quad & 1][i] >> (4 * (quad >> 1))) & 0x0F0F0F0Fu;
                    const uint32_t n = lo | (((qh[i] >> (2 * quad)) & 0x03030303u) << 4);   // 0 .. 63 per byte
                    const half2_t q01 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, n, 0x04010400u)) - k1056;
                    const half2_t q23 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, n, 0x04030402u)) - k1056;
                    v[quad][2 * i] = __builtin_bit_cast(uint32_t, q01 * D2);
                    v[quad][2 * i + 1] = __builtin_bit_cast(uint32_t, q23 * D2);
                }
            }
            return 128 * c + l0;
        }
    }
};

// `blocks` super-blocks in all, `per_row` of them in a row; rows go out as dequantize_kernel below spreads them.
template <int QT, int OUT>
__global__ __launch_bounds__(256) void dequantize_half_chain_kernel(const uint8_t* __restrict__ q, int64_t blocks, int64_t per_row,
                                                                    uint16_t* __restrict__ out, int spread, int64_t first) {
    typedef HalfChain<QT> H;
    const int64_t total = blocks * H::items;
    for (int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x; g < total; g += (int64_t)gridDim.x * 256) {
        const int64_t b = g / H::items;
        u32x4_t v[H::runs];
        const int e0 = H::decode(q + b * Fmt<QT>::ts, (int)(g & (H::items - 1)), v);
        int64_t shift = 0;   // super-blocks by which the row's output lies behind its place in the input
        if (spread < 63) {
            const int64_t r = b < ((int64_t)1 << 32) && per_row < ((int64_t)1 << 32) ? (int64_t)((uint32_t)b / (uint32_t)per_row) : b / per_row;
            shift = (((r >> spread) << spread) + first) * per_row;
        }
        uint16_t* o = out + (b + shift) * 256 + e0;
#pragma unroll
        for (int run = 0; run < H::runs; run++) {
            u32x4_t w = v[run];
            if constexpr (OUT == SNGGUF_OUT_BF16) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const uint32_t bits = w[i];   // (a bit cast applied to the element expression itself reads element 0)
                    const half2_t h = __builtin_bit_cast(half2_t, bits);
                    w[i] = pack_bf16((float)h[0], (float)h[1]);
                }
            }
            *reinterpret_cast<u32x4_t*>(o + 32 * run) = w;
        }
    }
}

// WIDE: the number of 8-element groups does not fit 32 bits (the index arithmetic then needs 64-bit divisions).
// Row r of the input is written to output row r + ((r >> spread) << spread) + first: with spread = 63 and first = 0
// that is row r; with spread = 7 the rows go out in blocks of 128 that leave 128 rows free behind each block (first = 0)
// or fill those (first = 128) - two matrices interleaved in blocks of 128 rows.
template <int QT, int NUM, int OUT, bool WIDE>
__global__ __launch_bounds__(256) void dequantize_kernel(const uint8_t* __restrict__ q, int64_t rows, int64_t cols,
                                                         int64_t row_bytes, void* __restrict__ out, int spread, int64_t first) {
    const int64_t groups_per_row = cols >> 3;
    const int64_t total = rows * groups_per_row;
    if constexpr (WIDE) {
        for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += (int64_t)gridDim.x * blockDim.x) {
            const int64_t r = g / groups_per_row;
            const int64_t e0 = (g - r * groups_per_row) << 3;
            float w[8];
            decode8<QT, NUM>(q + r * row_bytes, e0, w);
            store8<OUT>(out, (r + ((r >> spread) << spread) + first) * cols + e0, w);
        }
    } else {
        const uint32_t gpr = (uint32_t)groups_per_row, tot = (uint32_t)total, stride = gridDim.x * blockDim.x;
        for (uint32_t g = blockIdx.x * blockDim.x + threadIdx.x; g < tot; g += stride) {
            const uint32_t r = g / gpr;
            const int64_t e0 = (int64_t)(g - r * gpr) << 3;
            const int64_t ro = (int64_t)r + (((int64_t)r >> spread) << spread) + first;
            float w[8];
            decode8<QT, NUM>(q + (int64_t)r * row_bytes, e0, w);
            store8<OUT>(out, ro * cols + e0, w);
            if (g + stride < g) break;   // the next index would wrap
        }
    }
}

template <int QT, int NUM>
static int launch_out(const uint8_t* q, int64_t rows, int64_t cols, void* out, int out_dtype, hipStream_t stream,
                      int spread, int64_t first) {
    const int64_t row_bytes = cols / Fmt<QT>::bs * Fmt<QT>::ts;
    const int64_t total = rows * (cols >> 3);
    if (total == 0) return SNGGUF_OK;
    int64_t blocks = (total + 255) / 256;
    if (blocks > 256 * 64) blocks = 256 * 64;  // grid-stride beyond 64 blocks per CU
    dim3 grid((unsigned)blocks), block(256);
    if constexpr (NUM == SNGGUF_NUM_UPSTREAM_FP16 && (QT == SNGGUF_TYPE_Q4_K || QT == SNGGUF_TYPE_Q6_K)) {
        if (out_dtype == SNGGUF_OUT_F16 || out_dtype == SNGGUF_OUT_BF16) {
            const int64_t sblocks = rows * (cols >> 8);
            int64_t wgs = (sblocks * HalfChain<QT>::items + 255) / 256;
            if (wgs > 256 * 64) wgs = 256 * 64;
            uint16_t* o = static_cast<uint16_t*>(out);
            if (out_dtype == SNGGUF_OUT_F16)
                dequantize_half_chain_kernel<QT, SNGGUF_OUT_F16><<<dim3((unsigned)wgs), block, 0, stream>>>(q, sblocks, cols >> 8, o, spread, first);
            else
                dequantize_half_chain_kernel<QT, SNGGUF_OUT_BF16><<<dim3((unsigned)wgs), block, 0, stream>>>(q, sblocks, cols >> 8, o, spread, first);
            return hipGetLastError() == hipSuccess ? SNGGUF_OK : SNGGUF_E_LAUNCH;
        }
    }
    const bool wide = total >= ((int64_t)1 << 32);
#define SNGGUF_DEQ(OUT) \
    do { \
        if (wide) dequantize_kernel<QT, NUM, OUT, true><<<grid, block, 0, stream>>>(q, rows, cols, row_bytes, out, spread, first); \
        else dequantize_kernel<QT, NUM, OUT, false><<<grid, block, 0, stream>>>(q, rows, cols, row_bytes, out, spread, first); \
    } while (0)
    switch (out_dtype) {
    case SNGGUF_OUT_F32: SNGGUF_DEQ(SNGGUF_OUT_F32); break;
    case SNGGUF_OUT_F16: SNGGUF_DEQ(SNGGUF_OUT_F16); break;
    case SNGGUF_OUT_BF16: SNGGUF_DEQ(SNGGUF_OUT_BF16); break;
    default: return SNGGUF_E_BADTYPE;
    }
#undef SNGGUF_DEQ
    return hipGetLastError() == hipSuccess ? SNGGUF_OK : SNGGUF_E_LAUNCH;
}

template <int QT>
static int launch_num(const uint8_t* q, int64_t rows, int64_t cols, void* out, int out_dtype, int numerics, hipStream_t stream,
                      int spread, int64_t first) {
    if (numerics == SNGGUF_NUM_GGML_FP32) return launch_out<QT, SNGGUF_NUM_GGML_FP32>(q, rows, cols, out, out_dtype, stream, spread, first);
    if (numerics == SNGGUF_NUM_UPSTREAM_FP16) return launch_out<QT, SNGGUF_NUM_UPSTREAM_FP16>(q, rows, cols, out, out_dtype, stream, spread, first);
    return SNGGUF_E_BADTYPE;
}

int launch_dequantize(const void* q, int qtype, int64_t rows, int64_t cols, void* out, int out_dtype, int numerics,
                      hipStream_t stream) {
    const uint8_t* p = static_cast<const uint8_t*>(q);
#define SNGGUF_CALL(QT) launch_num<QT>(p, rows, cols, out, out_dtype, numerics, stream, 63, 0)
    SNGGUF_DISPATCH_TYPE(qtype, SNGGUF_CALL)
#undef SNGGUF_CALL
}

// The bf16 rows of one of two matrices that share an output in blocks of 128 rows: input row r goes to output row
// 256 (r / 128) + r % 128 (+ 128 for the second matrix).  What the gated dense GEMM reads: each of its 256-row weight
// tiles then holds 128 gate rows and the 128 up rows of the same output columns.
int launch_dequantize_interleaved(const void* q, int qtype, int64_t rows, int64_t cols, void* out, int second, int numerics,
                                  hipStream_t stream) {
    const uint8_t* p = static_cast<const uint8_t*>(q);
#define SNGGUF_CALL(QT) launch_num<QT>(p, rows, cols, out, SNGGUF_OUT_BF16, numerics, stream, 7, second ? 128 : 0)
    SNGGUF_DISPATCH_TYPE(qtype, SNGGUF_CALL)
#undef SNGGUF_CALL
}

}  // namespace sngguf
