// Decoders of the packed formats for the matrix-core kernels: 256 elements of a weight row in an LDS slab -> the A
// operands of v_mfma_f32_16x16x32_bf16.  Lane (r = lane % 16, g = lane / 16) gets, for each 32-element sub-block j,
// elements 8 g .. 8 g + 7 of its row as bf16, rounded as the numerics mode says.
#pragma once

#include "sngguf_common.hpp"

namespace sngguf {

namespace {

// Four small unsigned integers (one per byte of v, each < 256) -> (v - zero) * D - DM as two packed
// bf16 pairs.  NUM 1: every operation rounds to fp16 (0x6400 | b is the half 1024 + b, so the
// integer is formed without a convert); NUM 0: exact fp32 products, one rounding in the subtraction
// (the - 1024 - zero rides on the accumulator input of the widening instruction).  Must be called
// by all 64 lanes; `ident` is identity_row(lane).
// fp16 -> fp32 on the matrix cores (widen_f16x4): the vector ALU is the busier unit of the kernels that use these decoders.
// FUSED (formats with a minimum and zero = 0): the product and the operation next to it as one fused multiply-add
// where that gives the same bits.  NUM 0: D * q is exact in fp32 (at most 11 + 6 + 5 significant bits), so
// fma(D, q, -DM) rounds once exactly where D * q - DM does.  NUM 1: (1024 + q) * D - 1024 * D, exact inside the
// fused operation, rounds once to fp16(q * D); -1024 * D is exact in fp16 unless it overflows, so the caller takes
// this form only where every |D| of the wavefront is below 64 (a scale product that large has not been seen in a
// file; the plain form stays for it).
template <int NUM, bool HAS_MIN, bool FUSED>
__device__ __forceinline__ void kq_dword_bf16(half4_t ident, uint32_t v, float zero, typename Num<NUM>::T D,
                                              typename Num<NUM>::T DM, uint32_t& p01, uint32_t& p23) {
    const half2_t h01 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, v, 0x04010400u));
    const half2_t h23 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, v, 0x04030402u));
    if constexpr (NUM == SNGGUF_NUM_UPSTREAM_FP16) {
        const half2_t D2 = {D, D};
        half2_t a, b;
        if constexpr (FUSED) {
            const _Float16 c = (_Float16)(-1024.0f) * D;
            const half2_t C2 = {c, c};
            a = __builtin_elementwise_fma(h01, D2, C2);
            b = __builtin_elementwise_fma(h23, D2, C2);
        } else {
            const _Float16 off = (_Float16)(1024.0f + zero);
            const half2_t off2 = {off, off};
            a = (h01 - off2) * D2;
            b = (h23 - off2) * D2;
        }
        if constexpr (HAS_MIN) {
            const half2_t M2 = {DM, DM};
            a = a - M2;
            b = b - M2;
        }
        const f32x4_t w = widen_f16x4(ident, a, b, f32x4_t{0.f, 0.f, 0.f, 0.f});
        p01 = pack_bf16(w[0], w[1]);
        p23 = pack_bf16(w[2], w[3]);
    } else {
        const float c = -(1024.0f + zero);
        const f32x4_t qf = widen_f16x4(ident, h01, h23, f32x4_t{c, c, c, c});
        float w[4];
        if constexpr (FUSED && HAS_MIN) {
#pragma unroll
            for (int e = 0; e < 4; e++) w[e] = __builtin_fmaf(D, qf[e], -DM);
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) w[e] = D * qf[e];
            if constexpr (HAS_MIN) {
#pragma unroll
                for (int e = 0; e < 4; e++) w[e] = w[e] - DM;
            }
        }
        p01 = pack_bf16(w[0], w[1]);
        p23 = pack_bf16(w[2], w[3]);
    }
}

// Slab<QT>: how the `ts` bytes that hold 256 elements of one row travel to the wavefront's LDS slab.
// `pieces` 16-byte loads per row; piece p comes from byte 16 p of the run, except that the last one
// comes from byte `last_src` (formats whose run is not a multiple of 16 bytes end with a piece that
// overlaps its predecessor in memory); piece p lands at byte 16 p of the row's `stride`-byte slot.
// `align` is what the format guarantees for the address of a run when the matrix is 16-byte aligned.
// Strides are chosen so that 16 rows start in 16 different groups of four LDS banks.
template <int QT> struct Slab;
template <> struct Slab<SNGGUF_TYPE_Q4_0> {  // 8 blocks of 18 bytes
    static constexpr int ts = 144, pieces = 9, last_src = 128, stride = 144, align = 16;
};
template <> struct Slab<SNGGUF_TYPE_Q4_1> {  // 8 blocks of 20 bytes
    static constexpr int ts = 160, pieces = 10, last_src = 144, stride = 176, align = 16;
};
template <> struct Slab<SNGGUF_TYPE_Q5_0> {  // 8 blocks of 22 bytes
    static constexpr int ts = 176, pieces = 11, last_src = 160, stride = 176, align = 16;
};
template <> struct Slab<SNGGUF_TYPE_Q8_0> {  // 8 blocks of 34 bytes
    static constexpr int ts = 272, pieces = 17, last_src = 256, stride = 272, align = 16;
};
template <> struct Slab<SNGGUF_TYPE_Q5_1> {  // 8 blocks of 24 bytes
    static constexpr int ts = 192, pieces = 12, last_src = 176, stride = 208, align = 16;
};
// Q2_K: bytes 0..79 (scales, quants) as five pieces, bytes 68..83 as the sixth: d, dmin land at slab bytes 92, 94
template <> struct Slab<SNGGUF_TYPE_Q2_K> {
    static constexpr int ts = 84, pieces = 6, last_src = 68, stride = 112, align = 4;
};
// Q3_K: bytes 0..95 (mask, quants) as six pieces, bytes 94..109 as the seventh: the 12 scale bytes land at slab
// bytes 98..109, d at 110
template <> struct Slab<SNGGUF_TYPE_Q3_K> {
    static constexpr int ts = 110, pieces = 7, last_src = 94, stride = 112, align = 2;
};
template <> struct Slab<SNGGUF_TYPE_Q4_K> {
    static constexpr int ts = 144, pieces = 9, last_src = 128, stride = 144, align = 16;
};
template <> struct Slab<SNGGUF_TYPE_Q5_K> {
    static constexpr int ts = 176, pieces = 11, last_src = 160, stride = 176, align = 16;
};
// Q6_K: 13 pieces (208 bytes) + the fp16 scale at byte 208, fetched on its own
template <> struct Slab<SNGGUF_TYPE_Q6_K> {
    static constexpr int ts = 210, pieces = 13, last_src = 192, stride = 240, align = 2;
};

template <int ALIGN>
__device__ __forceinline__ u32x4_t ld_piece(const uint8_t* p) {
    if constexpr (ALIGN >= 16) return *reinterpret_cast<const u32x4_t*>(p);
    else if constexpr (ALIGN >= 4) return ld_u128_a4(p);
    else return ld_u128_a2(p);
}

// Eight bytes from slab address p, which is a multiple of 4 (ALIGNED) or 2 more than one.
template <bool ALIGNED>
__device__ __forceinline__ u32x2_t lds_u64(const uint8_t* p) {
    if constexpr (ALIGNED) {
        const uint32_t* w = reinterpret_cast<const uint32_t*>(p);
        return u32x2_t{w[0], w[1]};
    } else {
        const uint32_t* w = reinterpret_cast<const uint32_t*>(p - 2);
        const uint32_t w0 = w[0], w1 = w[1], w2 = w[2];
        return u32x2_t{__builtin_amdgcn_alignbit(w1, w0, 16), __builtin_amdgcn_alignbit(w2, w1, 16)};
    }
}
template <bool ALIGNED>
__device__ __forceinline__ uint32_t lds_u32(const uint8_t* p) {
    if constexpr (ALIGNED) {
        return *reinterpret_cast<const uint32_t*>(p);
    } else {
        const uint32_t* w = reinterpret_cast<const uint32_t*>(p - 2);
        return __builtin_amdgcn_alignbit(w[1], w[0], 16);
    }
}

// Q4_0 / Q4_1 / Q5_0 / Q5_1: sub-block jj of the half is block 4 HALF + jj of the eight in the slab
// row.  TS block bytes; HAS_MIN: f16 m after d, value d q + m, else d (q - 8 or 16); FIVE: 32-bit
// fifth-bit word before the quants.  Lane group g covers elements 8 g .. 8 g + 7: bytes
// 8 (g % 2) .. of qs, low nibbles for g < 2, high nibbles otherwise; fifth bits = byte g of qh.
template <int NUM, int B, int TS, bool HAS_MIN, bool FIVE>
__device__ __forceinline__ u32x4_t legacy_block(half4_t ident, const uint8_t* row, int g) {
    typedef Num<NUM> A;
    constexpr int kHdr = HAS_MIN ? 4 : 2;
    constexpr int kQs = kHdr + (FIVE ? 4 : 0);
    constexpr float kZero = HAS_MIN ? 0.f : (FIVE ? 16.f : 8.f);
    const uint8_t* blk = row + B * TS;
    const typename A::T d = A::scale(*reinterpret_cast<const uint16_t*>(blk));
    typename A::T DM = d;
    if constexpr (HAS_MIN) DM = -A::scale(*reinterpret_cast<const uint16_t*>(blk + 2));
    const int sh = 4 * (g >> 1);
    const u32x2_t qs = lds_u64<((B * TS + kQs) & 3) == 0>(blk + kQs + 8 * (g & 1));
    uint32_t v0 = (qs[0] >> sh) & 0x0F0F0F0Fu, v1 = (qs[1] >> sh) & 0x0F0F0F0Fu;
    if constexpr (FIVE) {
        const uint32_t bits = lds_u32<((B * TS + kHdr) & 3) == 0>(blk + kHdr) >> (8 * g);
        // bits 0..3 -> bit 4 of bytes 0..3
        v0 |= (((bits & 0xFu) * 0x00204081u) & 0x01010101u) << 4;
        v1 |= ((((bits >> 4) & 0xFu) * 0x00204081u) & 0x01010101u) << 4;
    }
    uint32_t a0, a1, a2, a3;
    kq_dword_bf16<NUM, HAS_MIN, false>(ident, v0, kZero, d, DM, a0, a1);
    kq_dword_bf16<NUM, HAS_MIN, false>(ident, v1, kZero, d, DM, a2, a3);
    return u32x4_t{a0, a1, a2, a3};
}
template <int NUM, int HALF, int TS, bool HAS_MIN, bool FIVE, typename Emit>
__device__ __forceinline__ void decode_legacy(half4_t ident, const uint8_t* row, int g, Emit&& emit) {
    emit(0, legacy_block<NUM, 4 * HALF + 0, TS, HAS_MIN, FIVE>(ident, row, g));
    emit(1, legacy_block<NUM, 4 * HALF + 1, TS, HAS_MIN, FIVE>(ident, row, g));
    emit(2, legacy_block<NUM, 4 * HALF + 2, TS, HAS_MIN, FIVE>(ident, row, g));
    emit(3, legacy_block<NUM, 4 * HALF + 3, TS, HAS_MIN, FIVE>(ident, row, g));
}

// Q8_0: block b at byte 34 b of the slab row: f16 d, then 32 int8 quants (2 bytes off a dword for even b)
template <int NUM, int B>
__device__ __forceinline__ u32x4_t q8_0_block(const uint8_t* row, int g) {
    const uint8_t* blk = row + B * 34;
    const uint16_t d = *reinterpret_cast<const uint16_t*>(blk);
    const u32x2_t qs = lds_u64<(B & 1) == 1>(blk + 2 + 8 * g);
    uint32_t a0, a1, a2, a3;
    q8_dword_bf16<NUM>(d, qs[0], a0, a1);
    q8_dword_bf16<NUM>(d, qs[1], a2, a3);
    return u32x4_t{a0, a1, a2, a3};
}
template <int NUM, int HALF, typename Emit>
__device__ __forceinline__ void decode_q8_0(const uint8_t* row, int g, Emit&& emit) {
    emit(0, q8_0_block<NUM, 4 * HALF + 0>(row, g));
    emit(1, q8_0_block<NUM, 4 * HALF + 1>(row, g));
    emit(2, q8_0_block<NUM, 4 * HALF + 2>(row, g));
    emit(3, q8_0_block<NUM, 4 * HALF + 3>(row, g));
}

// Q2_K: element 128 h + 32 j + l is bit pair j of qs[32 h + l]; its 16-element group
// 8 h + 2 j + l / 16 has scale (low nibble) and min (high nibble) in one byte.
template <int NUM, int HALF, typename Emit>
__device__ __forceinline__ void decode_q2_k(half4_t ident, const uint8_t* row, int g, Emit&& emit) {
    typedef Num<NUM> A;
    constexpr int h = HALF;
    const u32x2_t sm = *reinterpret_cast<const u32x2_t*>(row + 8 * h);  // groups 8 h .. 8 h + 7
    const uint32_t dd = *reinterpret_cast<const uint32_t*>(row + 92);
    const typename A::T d = A::scale((uint16_t)(dd & 0xFFFF)), dmin = A::scale((uint16_t)(dd >> 16));
    const u32x2_t qs = *reinterpret_cast<const u32x2_t*>(row + 16 + 32 * h + 8 * g);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t byte = (sm[j >> 1] >> (8 * (2 * (j & 1) + (g >> 1)))) & 0xFFu;
        const typename A::T D = d * A::integer((int)(byte & 15u)), DM = dmin * A::integer((int)(byte >> 4));
        uint32_t a0, a1, a2, a3;
        kq_dword_bf16<NUM, true, false>(ident, (qs[0] >> (2 * j)) & 0x03030303u, 0.f, D, DM, a0, a1);
        kq_dword_bf16<NUM, true, false>(ident, (qs[1] >> (2 * j)) & 0x03030303u, 0.f, D, DM, a2, a3);
        emit(j, u32x4_t{a0, a1, a2, a3});
    }
}

// Q3_K: stored quant (0..7) = bit pair as in Q2_K | mask bit (4 h + j of hmask[l]) << 2, value
// stored - 4; 6-bit group scales split over the 12 scale bytes, value stored - 32.
template <int NUM, int HALF, typename Emit>
__device__ __forceinline__ void decode_q3_k(half4_t ident, const uint8_t* row, int g, Emit&& emit) {
    typedef Num<NUM> A;
    constexpr int h = HALF;
    const u32x4_t t = *reinterpret_cast<const u32x4_t*>(row + 96);  // source bytes 94..109
    const uint32_t s0 = __builtin_amdgcn_alignbit(t[1], t[0], 16);  // scale bytes 0..3
    const uint32_t s1 = __builtin_amdgcn_alignbit(t[2], t[1], 16);  // 4..7
    const uint32_t s2 = __builtin_amdgcn_alignbit(t[3], t[2], 16);  // 8..11
    const typename A::T d = A::scale((uint16_t)(t[3] >> 16));
    const u32x2_t hm = *reinterpret_cast<const u32x2_t*>(row + 8 * g);
    const u32x2_t qs = *reinterpret_cast<const u32x2_t*>(row + 32 + 32 * h + 8 * g);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        // group 8 h + tt, tt = 2 j + g / 2: low nibble in byte tt (upper nibble for h = 1), high bits in
        // byte 8 + tt % 4 at bit 2 (2 h + tt / 4)
        const int t3 = (2 * (j & 1) + (g >> 1));  // tt % 4
        const uint32_t lo = (((j < 2 ? s0 : s1) >> (8 * t3)) >> (4 * h)) & 15u;
        const uint32_t hi = (((s2 >> (8 * t3)) & 0xFFu) >> (2 * (2 * h + (j >> 1)))) & 3u;
        const typename A::T D = d * A::integer((int)(lo | (hi << 4)) - 32);
        uint32_t a[4];
#pragma unroll
        for (int w = 0; w < 2; w++) {
            const uint32_t v = ((qs[w] >> (2 * j)) & 0x03030303u) | (((hm[w] >> (4 * h + j)) & 0x01010101u) << 2);
            kq_dword_bf16<NUM, false, false>(ident, v, 4.f, D, D, a[2 * w], a[2 * w + 1]);
        }
        emit(j, u32x4_t{a[0], a[1], a[2], a[3]});
    }
}


// (d * scale, dmin * min) of sub-blocks 4 HALF .. 4 HALF + 3 of the lane's row (Q4_K and Q5_K).  The four lanes
// (r, g = 0..3) that decode one row all need the same four pairs: lane (r, g) extracts and scales the pair of
// sub-block 4 HALF + g only, and the four exchange their results through the cross-lane network (ds_bpermute, which
// touches no LDS memory).  Same arithmetic on the same operands as computing every pair in every lane, so the
// values are bit-identical; it takes a quarter of the decode's vector instructions away.  Must be called by all
// 64 lanes.
template <int NUM, int HALF>
__device__ __forceinline__ bool q4k_pairs(const u32x4_t& head, int g, typename Num<NUM>::T (&D)[4], typename Num<NUM>::T (&DM)[4]) {
    typedef Num<NUM> A;
    uint32_t sc, mn;
    if constexpr (HALF == 0) {
        sc = (head[1] >> (8 * g)) & 63u;
        mn = (head[2] >> (8 * g)) & 63u;
    } else {
        const uint32_t b = (head[3] >> (8 * g)) & 0xFFu;
        sc = (b & 0x0Fu) | (((head[1] >> (8 * g + 6)) & 3u) << 4);
        mn = (b >> 4) | (((head[2] >> (8 * g + 6)) & 3u) << 4);
    }
    const typename A::T mine_d = A::scale((uint16_t)(head[0] & 0xFFFF)) * A::integer((int)sc);
    const typename A::T mine_m = A::scale((uint16_t)(head[0] >> 16)) * A::integer((int)mn);
    const int self = 4 * (int)(threadIdx.x & 15);  // byte address of lane (r, 0) for ds_bpermute
    if constexpr (NUM == SNGGUF_NUM_UPSTREAM_FP16) {
        const half2_t both = {mine_d, mine_m};
        const int bits = __builtin_bit_cast(int, both);
#pragma unroll
        for (int jj = 0; jj < 4; jj++) {
            const half2_t got = __builtin_bit_cast(half2_t, __builtin_amdgcn_ds_bpermute(self + 64 * jj, bits));
            D[jj] = got[0];
            DM[jj] = got[1];
        }
        // every |d * scale| of the wavefront below 64 (0x5400): the fused form of kq_dword_bf16 is exact
        return __builtin_amdgcn_ballot_w64(((uint32_t)bits & 0x7FFFu) >= 0x5400u) == 0;
    } else {
#pragma unroll
        for (int jj = 0; jj < 4; jj++) {
            D[jj] = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(self + 64 * jj, __builtin_bit_cast(int, mine_d)));
            DM[jj] = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(self + 64 * jj, __builtin_bit_cast(int, mine_m)));
        }
        return true;
    }
}

// The four A operands of half a super-block (sub-blocks 4 HALF .. 4 HALF + 3) of one row, fed to
// `emit(jj, a)` with jj = 0..3.  `row` points at the row's super-block in the slab; g = lane / 16.
template <int NUM, int HALF, bool FUSED, typename Emit>
__device__ __forceinline__ void decode_q4_k_body(half4_t ident, const uint8_t* row, int g, const typename Num<NUM>::T (&Ds)[4],
                                                 const typename Num<NUM>::T (&DMs)[4], Emit&& emit) {
#pragma unroll
    for (int cc = 0; cc < 2; cc++) {
        const int c = 2 * HALF + cc;
        const u32x2_t qs = *reinterpret_cast<const u32x2_t*>(row + 16 + 32 * c + 8 * g);
#pragma unroll
        for (int hi = 0; hi < 2; hi++) {
            const int j = 2 * c + hi;
            const typename Num<NUM>::T D = Ds[j - 4 * HALF], DM = DMs[j - 4 * HALF];
            const uint32_t v0 = (hi ? qs[0] >> 4 : qs[0]) & 0x0F0F0F0Fu, v1 = (hi ? qs[1] >> 4 : qs[1]) & 0x0F0F0F0Fu;
            uint32_t a0, a1, a2, a3;
            kq_dword_bf16<NUM, true, FUSED>(ident, v0, 0.f, D, DM, a0, a1);
            kq_dword_bf16<NUM, true, FUSED>(ident, v1, 0.f, D, DM, a2, a3);
            emit(j - 4 * HALF, u32x4_t{a0, a1, a2, a3});
        }
    }
}
template <int NUM, int HALF, typename Emit>
__device__ __forceinline__ void decode_q4_k(half4_t ident, const uint8_t* row, int g, Emit&& emit) {
    typedef Num<NUM> A;
    const u32x4_t head = *reinterpret_cast<const u32x4_t*>(row);  // d, dmin, 12 scale bytes
    typename A::T Ds[4], DMs[4];
    const bool fused = q4k_pairs<NUM, HALF>(head, g, Ds, DMs);
    if (fused) decode_q4_k_body<NUM, HALF, true>(ident, row, g, Ds, DMs, emit);
    else decode_q4_k_body<NUM, HALF, false>(ident, row, g, Ds, DMs, emit);
}

// Q5_K: as Q4_K, the fifth bit of element l of sub-block j is bit j of qh[l]
template <int NUM, int HALF, bool FUSED, typename Emit>
__device__ __forceinline__ void decode_q5_k_body(half4_t ident, const uint8_t* row, int g, const typename Num<NUM>::T (&Ds)[4],
                                                 const typename Num<NUM>::T (&DMs)[4], Emit&& emit) {
    const u32x2_t qh = *reinterpret_cast<const u32x2_t*>(row + 16 + 8 * g);
#pragma unroll
    for (int cc = 0; cc < 2; cc++) {
        const int c = 2 * HALF + cc;
        const u32x2_t qs = *reinterpret_cast<const u32x2_t*>(row + 48 + 32 * c + 8 * g);
#pragma unroll
        for (int hi = 0; hi < 2; hi++) {
            const int j = 2 * c + hi;
            const typename Num<NUM>::T D = Ds[j - 4 * HALF], DM = DMs[j - 4 * HALF];
            uint32_t a[4];
#pragma unroll
            for (int w = 0; w < 2; w++) {
                const uint32_t lo = (hi ? qs[w] >> 4 : qs[w]) & 0x0F0F0F0Fu;
                const uint32_t hb = ((qh[w] >> j) & 0x01010101u) << 4;
                kq_dword_bf16<NUM, true, FUSED>(ident, lo | hb, 0.f, D, DM, a[2 * w], a[2 * w + 1]);
            }
            emit(j - 4 * HALF, u32x4_t{a[0], a[1], a[2], a[3]});
        }
    }
}
template <int NUM, int HALF, typename Emit>
__device__ __forceinline__ void decode_q5_k(half4_t ident, const uint8_t* row, int g, Emit&& emit) {
    typedef Num<NUM> A;
    const u32x4_t head = *reinterpret_cast<const u32x4_t*>(row);  // d, dmin, 12 scale bytes
    typename A::T Ds[4], DMs[4];
    const bool fused = q4k_pairs<NUM, HALF>(head, g, Ds, DMs);
    if (fused) decode_q5_k_body<NUM, HALF, true>(ident, row, g, Ds, DMs, emit);
    else decode_q5_k_body<NUM, HALF, false>(ident, row, g, Ds, DMs, emit);
}

template <int NUM, int HALF, typename Emit>
__device__ __forceinline__ void decode_q6_k(half4_t ident, const uint8_t* row, int g, Emit&& emit) {
    typedef Num<NUM> A;
    constexpr int h = HALF;  // 128-element half of the super-block = sub-blocks 4 h .. 4 h + 3
    const u32x2_t scales = *reinterpret_cast<const u32x2_t*>(row + 192 + 8 * h);  // int8 sub-scales 8 h .. 8 h + 7
    const typename A::T d = A::scale(*reinterpret_cast<const uint16_t*>(row + 208));
    const u32x2_t qh = *reinterpret_cast<const u32x2_t*>(row + 128 + 32 * h + 8 * g);
#pragma unroll
    for (int half = 0; half < 2; half++) {  // ql bytes 64 h + 32 half + 8 g ..: low nibbles p = half, high nibbles p = half + 2
        const u32x2_t ql = *reinterpret_cast<const u32x2_t*>(row + 64 * h + 32 * half + 8 * g);
#pragma unroll
        for (int top = 0; top < 2; top++) {
            const int p = half + 2 * top;
            // sub-scale of elements 128 h + 32 p + 8 g ..: index 8 h + 2 p + g / 2
            const uint32_t sw = scales[p >> 1];
            const int sc = (int)(int8_t)((sw >> (8 * (2 * (p & 1) + (g >> 1)))) & 0xFF);
            const typename A::T D = d * A::integer(sc);
            uint32_t a[4];
#pragma unroll
            for (int w = 0; w < 2; w++) {
                const uint32_t lo = (top ? ql[w] >> 4 : ql[w]) & 0x0F0F0F0Fu;
                const uint32_t hb = ((qh[w] >> (2 * p)) & 0x03030303u) << 4;
                kq_dword_bf16<NUM, false, false>(ident, lo | hb, 32.f, D, D, a[2 * w], a[2 * w + 1]);
            }
            emit(p, u32x4_t{a[0], a[1], a[2], a[3]});
        }
    }
}

// One half (sub-blocks 4 HALF .. 4 HALF + 3) of a slab row -> four A operands through `emit(jj, a)`.
template <int QT, int NUM, int HALF, typename Emit>
__device__ __forceinline__ void decode_half(half4_t ident, const uint8_t* row, int g, Emit&& emit) {
    if constexpr (QT == SNGGUF_TYPE_Q4_0) decode_legacy<NUM, HALF, 18, false, false>(ident, row, g, emit);
    else if constexpr (QT == SNGGUF_TYPE_Q4_1) decode_legacy<NUM, HALF, 20, true, false>(ident, row, g, emit);
    else if constexpr (QT == SNGGUF_TYPE_Q5_0) decode_legacy<NUM, HALF, 22, false, true>(ident, row, g, emit);
    else if constexpr (QT == SNGGUF_TYPE_Q5_1) decode_legacy<NUM, HALF, 24, true, true>(ident, row, g, emit);
    else if constexpr (QT == SNGGUF_TYPE_Q8_0) decode_q8_0<NUM, HALF>(row, g, emit);
    else if constexpr (QT == SNGGUF_TYPE_Q2_K) decode_q2_k<NUM, HALF>(ident, row, g, emit);
    else if constexpr (QT == SNGGUF_TYPE_Q3_K) decode_q3_k<NUM, HALF>(ident, row, g, emit);
    else if constexpr (QT == SNGGUF_TYPE_Q4_K) decode_q4_k<NUM, HALF>(ident, row, g, emit);
    else if constexpr (QT == SNGGUF_TYPE_Q5_K) decode_q5_k<NUM, HALF>(ident, row, g, emit);
    else {
        static_assert(QT == SNGGUF_TYPE_Q6_K, "no matrix-core decoder for this quant type");
        decode_q6_k<NUM, HALF>(ident, row, g, emit);
    }
}

}  // namespace

}  // namespace sngguf
