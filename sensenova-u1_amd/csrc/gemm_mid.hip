// Dequant-GEMM for 17 rows to a few thousand (K % 256 == 0), all ten block formats: the packed rows go from memory to matrix-core
// operands in registers, each decoded once per tile of up to 256 activation rows; no weight pass, and no decoded weight in LDS.
//
// Eight wavefronts share one tile of activations; each owns 16 or 32 weight rows and (with KW = 2) one half of the
// workgroup's K range.  Three forms (mid_plan in gemm_mid_plan.hip picks):
//   narrow  16 rows per wavefront, two halves of K:  64 columns per workgroup, up to 64 rows, two workgroups per compute unit
//           (one with 64 rows in Q8_0 and Q6_K, whose slabs are the widest; up to three with 32 rows and one unit ahead)
//   wide    32 rows per wavefront, two halves of K: 128 columns, up to 208 rows
//   long    32 rows per wavefront, all of K:        256 columns, up to 256 rows
// (wide ends at 208 rows because its registers do: 206 - 252 of 256 are taken there, by format.  From 209 rows on two row tiles, or the
// long form, take 17 - 23 % longer than 208 rows.)
// What bounds it: up to about 64 rows the latency of a step (packed bytes -> slab -> decode -> matrix instructions, which two
// wavefronts a SIMD hide only partly), beyond that no one unit: a stage of 208 rows keeps the matrix cores busy for half of its
// cycles, the vector ALU for about as many, and the clock falls with the power drawn (1.85 - 1.95 GHz of 2.4), so that what
// counts is work left out rather than cycles.  Leaving out (203 rows, pair of 12288 x 4096 in Q4_K, 67 us in that copy) the activations'
// copies gives 54 us, the packed rows' requests 58, the decode 55, the matrix instructions 52.  So the loop is written out instruction group
// by instruction group: two matrix instructions, the activation fragment of four groups later, a part of the next sub-block's decode
// or one request, a scheduling fence.  Left to the compiler's scheduler the fragments are read one instruction ahead (100 us against 69).
// Measured and not taken: 32x32x16 instructions on groups of 32 rows (12 - 16 % fewer cycles, but up to 5 % more time from 500 rows on:
// twice the accumulator traffic per product, which the clock pays for), other cache hints on the copies (nontemporal + 10 %); from 160
// rows on, waiting for a unit's pieces at the head of the stage that stores them, where its own copies are not out yet (the compiler's
// wait in mid-stage takes these in): 54 timings 0.97 - 1.04, faster in Q4_K, slower in Q6_K.
//
// Per wavefront and unit of 128 elements of K: the packed bytes are requested a unit ahead into registers (16-byte pieces,
// consecutive lanes walking along a row) and put into a slab of the wavefront's own; the decode reads them from there.
// Activations: 64 (or, up to 64 rows, 128) columns of every row and half of K are copied global -> LDS directly one stage ahead,
// in rows of 128 bytes whose 16-byte chunk c sits at c ^ ((row / 2) % 8); one barrier a stage.  (FAR: two units ahead, the activations
// through registers.)
//
// Measured, launches back to back on weights from memory, reductions included (us; Q8_0 / Q4_K / Q6_K; pair: of 12288 x 4096).  First
// what ran before this kernel, then the kernel with a stage's requests in one go behind the barrier, bytes widened by permutes and
// an epilogue of single columns, then as it is:
//   40 rows    pair            66 / 57 / 67      38 / 36 / 44       35 / 33 / 43
//   203 rows   pair            84 / 83           71 / 64 / 73       65 / 60 / 69
//              4096 x 12288    51 / 50 / 75      46 / 41 / 44       42 / 38 / 42
//              6144 x 4096     37 / 37 / 49      32 / 30 / 32       29 / 28 / 31
//   509 rows   pair            150 / 142        122 / 121 / 129    115 / 115 / 128
//   1024 rows  pair            247 / 232           / 224              / 210
//              4096 x 12288                     123 / 121 / 130    118 / 119 / 129
//   90 rows    12288 x 4096                      30 / 29 / 34       30 / 27 / 35
//   24 rows    151936 x 4096                    163 / 143 / 202    162 / 140 / 197
// Over 290 such lines of all formats, 20 - 1024 rows, the last is 0.96 of the one before in the mean, 0.86 - 1.07; with 90 rows Q8_0, Q5_0
// and Q6_K are up to 4 % slower than it.
#include "gemm_mid.hpp"

#include "kq_decode.hpp"

#ifndef SNGGUF_MID_TYPE
#error "compiled once per block format: -DSNGGUF_MID_TYPE=<ggml type>"
#endif

// (a translation unit uses the traits of one format)
#pragma clang diagnostic ignored "-Wunused-const-variable"

namespace sngguf {

namespace {

constexpr int kWaves = 8;

template <int V> struct int_c { static constexpr int value = V; };
template <int N, int I = 0, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(int_c<I>{});
        static_for<N, I + 1>(f);
    }
}

// A pointer that is the same in all lanes, in scalar registers; only for requests written as instructions (through an
// integer it is no global pointer to the compiler any more, which would make a plain load of it a flat one: those count as
// LDS accesses too, and every wait for a fragment would wait for memory).
__device__ __forceinline__ const uint8_t* wave_ptr(const void* p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return reinterpret_cast<const uint8_t*>(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}

// Unit<QT>: how the bytes that hold 128 elements of one row (half a super-block, or four blocks) travel to the wavefront's
// slab: `pieces` 16-byte loads, piece p from byte src(h, p) of the super-block (or of the eight blocks) to byte 16 p of the
// row's `stride`-byte slot, an odd number of 16-byte groups, so that 16 rows start in 16 different groups of LDS banks.
// Formats whose unit is no multiple of 16 bytes end with a piece that overlaps its predecessor in memory.  `second`: how far every piece
// of the second unit lies behind the same piece of the first, so that one set of addresses serves both; 0 where that differs from piece
// to piece.
template <int TS, int PIECES, int STRIDE>
struct UnitBlocks {   // four blocks of TS bytes
    static constexpr int pieces = PIECES, stride = STRIDE, align = 4, last = 4 * TS - 16, second = 4 * TS;
    static __device__ __forceinline__ int src(int h, int p) { return 4 * TS * h + (p == PIECES - 1 ? last : 16 * p); }
};
template <int QT> struct Unit;
template <> struct Unit<SNGGUF_TYPE_Q4_0> : UnitBlocks<18, 5, 80> {};
template <> struct Unit<SNGGUF_TYPE_Q4_1> : UnitBlocks<20, 5, 80> {};
template <> struct Unit<SNGGUF_TYPE_Q5_0> : UnitBlocks<22, 6, 112> {};
template <> struct Unit<SNGGUF_TYPE_Q5_1> : UnitBlocks<24, 6, 112> {};
template <> struct Unit<SNGGUF_TYPE_Q8_0> : UnitBlocks<34, 9, 144> {};
template <> struct Unit<SNGGUF_TYPE_Q2_K> {   // scales, quants of the half, d and dmin in the last dword
    static constexpr int pieces = 4, stride = 80, align = 4, second = 0;
    static __device__ __forceinline__ int src(int h, int p) { return p == 0 ? 0 : p == 3 ? 68 : 32 * h + 16 * p; }
};
template <> struct Unit<SNGGUF_TYPE_Q3_K> {   // mask, quants of the half, scales and d
    static constexpr int pieces = 5, stride = 80, align = 2, second = 0;
    static __device__ __forceinline__ int src(int h, int p) { return p < 2 ? 16 * p : p == 4 ? 94 : 32 * h + 16 * p; }
};
template <> struct Unit<SNGGUF_TYPE_Q4_K> {   // head, quants of the half
    static constexpr int pieces = 5, stride = 80, align = 16, second = 0;
    static __device__ __forceinline__ int src(int h, int p) { return p == 0 ? 0 : 64 * h + 16 * p; }
};
template <> struct Unit<SNGGUF_TYPE_Q5_K> {   // head, fifth bits, quants of the half
    static constexpr int pieces = 7, stride = 112, align = 16, second = 0;
    static __device__ __forceinline__ int src(int h, int p) { return p < 3 ? 16 * p : 64 * h + 16 * p; }
};
template <> struct Unit<SNGGUF_TYPE_Q6_K> {   // low and high bits of the half, scales; d follows on its own at byte 112
    static constexpr int pieces = 7, stride = 144, align = 2, second = 0;
    static __device__ __forceinline__ int src(int h, int p) { return p < 4 ? 64 * h + 16 * p : p < 6 ? 64 + 32 * h + 16 * p : 192; }
};

// A field of MASK << P bits of every 16-bit half of v, as halves base + field with base = 2^(10 - P): under that exponent the field's
// lowest bit is worth one, so nothing is shifted down to bit 0.  Shifts and v_bitop3 issue in 2.3 - 2.5 cycles with two wavefronts on
// a SIMD; v_perm, v_and_or, the packed and the converting instructions in 4.2 - 4.4.
template <int P, uint32_t MASK>
__device__ __forceinline__ half2_t field(uint32_t v) {
    return __builtin_bit_cast(half2_t, (uint32_t)__builtin_amdgcn_bitop3_b32(v, MASK * 0x00010001u << P, (0x6400u - (P << 10)) * 0x00010001u, 0xEA));
}
// The same with TOP of w, shifted left by SHIFT (or right), at bit AT above it
template <int P, uint32_t MASK, uint32_t TOP, int AT, int SHIFT>
__device__ __forceinline__ half2_t field2(uint32_t v, uint32_t w) {
    const uint32_t ws = SHIFT > 0 ? w << (SHIFT > 0 ? SHIFT : 0) : w >> (SHIFT < 0 ? -SHIFT : 0);
    const uint32_t top = __builtin_amdgcn_bitop3_b32(ws, TOP * 0x00010001u << AT, (0x6400u - (P << 10)) * 0x00010001u, 0xEA);
    return __builtin_bit_cast(half2_t, (uint32_t)__builtin_amdgcn_bitop3_b32(v, MASK * 0x00010001u << P, top, 0xEA));
}

// Halves base + integer -> the same halves as weights in the rounding chain (fp16: three operations, or two without a minimum) ...
template <int NUM, bool HAS_MIN>
__device__ __forceinline__ void chain_pair(half2_t& h, float off, typename Num<NUM>::T D, typename Num<NUM>::T DM) {
    const _Float16 o = (_Float16)off;
    h = h - half2_t{o, o};   // whole numbers: exact
    if constexpr (NUM == SNGGUF_NUM_UPSTREAM_FP16) {
        h = h * half2_t{D, D};
        if constexpr (HAS_MIN) h = h - half2_t{DM, DM};
    }
}
// ... and elements 0 .. 3 of these as bf16
template <int NUM, bool HAS_MIN>
__device__ __forceinline__ void chain_bf16(half2_t a, half2_t b, typename Num<NUM>::T D, typename Num<NUM>::T DM, uint32_t& p01, uint32_t& p23) {
    float w[4] = {(float)a[0], (float)b[0], (float)a[1], (float)b[1]};
    if constexpr (NUM != SNGGUF_NUM_UPSTREAM_FP16) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            w[e] = D * w[e];
            if constexpr (HAS_MIN) w[e] = w[e] - DM;
        }
    }
    p01 = pack_bf16(w[0], w[1]);
    p23 = pack_bf16(w[2], w[3]);
}

// One 32-element sub-block of a slab row for lane group g, in three parts that the K loop places between matrix
// instructions: the LDS reads (`load`), the sub-block's scale and minimum (`scales`), and elements 4 W .. 4 W + 3 of the lane's eight
// (`pairs`: the halves (0, 2) and (1, 3), each base() + the stored unsigned integer).  J: sub-block 0 .. 7 of the 256 elements.
template <int QT, int NUM> struct Sub;

template <int NUM, int TS, bool HAS_MIN, bool FIVE>
struct SubLegacy {
    typedef typename Num<NUM>::T V;
    static constexpr bool kMin = HAS_MIN;
    static constexpr int kZero = HAS_MIN ? 0 : (FIVE ? 16 : 8);
    uint32_t hd, fifth;
    u32x2_t qs;
    template <int J> __device__ __forceinline__ void load(const uint8_t* row, int g) {
        constexpr int kHdr = HAS_MIN ? 4 : 2, kQs = kHdr + (FIVE ? 4 : 0), at = (J & 3) * TS;
        constexpr int shift = (4 * TS) % 16 != 0 && (J & 3) == 3 ? 8 : 0;   // the unit's last 8 bytes: in the overlapping piece
        if constexpr (HAS_MIN) hd = lds_u32<(at & 3) == 0>(row + at);
        else hd = *reinterpret_cast<const uint16_t*>(row + at);
        if constexpr (FIVE) fifth = lds_u32<((at + kHdr) & 3) == 0>(row + at + kHdr);
        qs = lds_u64<((at + kQs) & 3) == 0>(row + at + kQs + (8 + shift) * (g & 1));
    }
    template <int J> __device__ __forceinline__ void scales(int, V& D, V& DM) const {
        D = Num<NUM>::scale((uint16_t)(hd & 0xFFFF));
        DM = D;
        if constexpr (HAS_MIN) DM = -Num<NUM>::scale((uint16_t)(hd >> 16));
    }
    template <int J> static constexpr int base() { return 1024; }
    template <int J, int W> __device__ __forceinline__ void pairs(int g, half2_t& a, half2_t& b) const {
        const uint32_t v = qs[W] >> (4 * (g >> 1));
        if constexpr (FIVE) {
            // bits 0 .. 3 of this quarter to bit 4 of bytes 0 .. 3
            const uint32_t bits = (((fifth >> (8 * g + 4 * W)) & 0xFu) * 0x00204081u) & 0x01010101u;
            const uint32_t quants = (uint32_t)__builtin_amdgcn_bitop3_b32(v, 0x0F0F0F0Fu, bits << 4, 0xEA);
            a = field<0, 0x1F>(quants);
            b = field<0, 0x1F>(quants >> 8);
        } else {
            a = field<0, 0xF>(v);
            b = field<0, 0xF>(v >> 8);
        }
    }
};
template <int NUM> struct Sub<SNGGUF_TYPE_Q4_0, NUM> : SubLegacy<NUM, 18, false, false> {};
template <int NUM> struct Sub<SNGGUF_TYPE_Q4_1, NUM> : SubLegacy<NUM, 20, true, false> {};
template <int NUM> struct Sub<SNGGUF_TYPE_Q5_0, NUM> : SubLegacy<NUM, 22, false, true> {};
template <int NUM> struct Sub<SNGGUF_TYPE_Q5_1, NUM> : SubLegacy<NUM, 24, true, true> {};

template <int NUM> struct Sub<SNGGUF_TYPE_Q8_0, NUM> {
    typedef typename Num<NUM>::T V;
    static constexpr bool kMin = false;
    static constexpr int kZero = 128;
    uint32_t hd;
    u32x2_t qs;
    template <int J> __device__ __forceinline__ void load(const uint8_t* row, int g) {
        constexpr int jj = J & 3;
        hd = *reinterpret_cast<const uint16_t*>(row + 34 * jj);
        // (the unit's last 8 bytes lie in the overlapping piece)
        qs = lds_u64<(jj & 1) == 1>(row + 34 * jj + 2 + 8 * g + (jj == 3 && g == 3 ? 8 : 0));
    }
    template <int J> __device__ __forceinline__ void scales(int, V& D, V& DM) const { DM = D = Num<NUM>::scale((uint16_t)hd); }
    template <int J> static constexpr int base() { return 1024; }
    // (the sign bit of each byte is turned with the mask: stored + 128)
    template <int J, int W> __device__ __forceinline__ void pairs(int, half2_t& a, half2_t& b) const {
        a = __builtin_bit_cast(half2_t, (uint32_t)__builtin_amdgcn_bitop3_b32(qs[W], 0x00FF00FFu, 0x64806480u, 0x6A));
        b = __builtin_bit_cast(half2_t, (uint32_t)__builtin_amdgcn_bitop3_b32(qs[W] >> 8, 0x00FF00FFu, 0x64806480u, 0x6A));
    }
};

template <int NUM> struct Sub<SNGGUF_TYPE_Q2_K, NUM> {
    typedef typename Num<NUM>::T V;
    static constexpr bool kMin = true;
    static constexpr int kZero = 0;
    uint32_t sm, dd;
    u32x2_t qs;
    template <int J> __device__ __forceinline__ void load(const uint8_t* row, int g) {
        sm = *reinterpret_cast<const uint32_t*>(row + 8 * (J >> 2) + 4 * ((J & 3) >> 1));
        dd = *reinterpret_cast<const uint32_t*>(row + 60);
        qs = *reinterpret_cast<const u32x2_t*>(row + 16 + 8 * g);
    }
    template <int J> __device__ __forceinline__ void scales(int g, V& D, V& DM) const {
        const uint32_t byte = (sm >> (8 * (2 * (J & 1) + (g >> 1)))) & 0xFFu;
        D = Num<NUM>::scale((uint16_t)(dd & 0xFFFF)) * Num<NUM>::integer((int)(byte & 15u));
        DM = Num<NUM>::scale((uint16_t)(dd >> 16)) * Num<NUM>::integer((int)(byte >> 4));
    }
    template <int J> static constexpr int base() { return 1024 >> (2 * (J & 3)); }
    template <int J, int W> __device__ __forceinline__ void pairs(int, half2_t& a, half2_t& b) const {
        a = field<2 * (J & 3), 3>(qs[W]);
        b = field<2 * (J & 3), 3>(qs[W] >> 8);
    }
};

template <int NUM> struct Sub<SNGGUF_TYPE_Q3_K, NUM> {
    typedef typename Num<NUM>::T V;
    static constexpr bool kMin = false;
    static constexpr int kZero = 4;
    u32x4_t t;
    u32x2_t hm, qs;
    template <int J> __device__ __forceinline__ void load(const uint8_t* row, int g) {
        t = *reinterpret_cast<const u32x4_t*>(row + 64);   // source bytes 94 .. 109
        hm = *reinterpret_cast<const u32x2_t*>(row + 8 * g);
        qs = *reinterpret_cast<const u32x2_t*>(row + 32 + 8 * g);
    }
    template <int J> __device__ __forceinline__ void scales(int g, V& D, V& DM) const {
        constexpr int h = J >> 2, j = J & 3;
        const uint32_t s = j < 2 ? __builtin_amdgcn_alignbit(t[1], t[0], 16) : __builtin_amdgcn_alignbit(t[2], t[1], 16);
        const uint32_t s2 = __builtin_amdgcn_alignbit(t[3], t[2], 16);
        const int t3 = 2 * (j & 1) + (g >> 1);
        const uint32_t lo = ((s >> (8 * t3)) >> (4 * h)) & 15u;
        const uint32_t hi = ((s2 >> (8 * t3)) >> (2 * (2 * h + (j >> 1)))) & 3u;
        DM = D = Num<NUM>::scale((uint16_t)(t[3] >> 16)) * Num<NUM>::integer((int)(lo | (hi << 4)) - 32);
    }
    template <int J> static constexpr int base() { return 1024 >> (2 * (J & 3)); }
    template <int J, int W> __device__ __forceinline__ void pairs(int, half2_t& a, half2_t& b) const {
        constexpr int P = 2 * (J & 3);
        a = field2<P, 3, 1, P + 2, P + 2 - J>(qs[W], hm[W]);
        b = field2<P, 3, 1, P + 2, P + 2 - J - 8>(qs[W] >> 8, hm[W]);
    }
};

// Scale and minimum of sub-block J of a Q4_K or Q5_K head
template <int J, int NUM>
__device__ __forceinline__ void q45k_scales(const u32x4_t& head, typename Num<NUM>::T& D, typename Num<NUM>::T& DM) {
    constexpr int i = 8 * (J & 3);
    uint32_t sc, mn;
    if constexpr (J < 4) {
        sc = (head[1] >> i) & 63u;
        mn = (head[2] >> i) & 63u;
    } else {
        sc = ((head[3] >> i) & 15u) | (((head[1] >> (i + 6)) & 3u) << 4);
        mn = ((head[3] >> (i + 4)) & 15u) | (((head[2] >> (i + 6)) & 3u) << 4);
    }
    if constexpr (NUM == SNGGUF_NUM_UPSTREAM_FP16) {
        // both products in one packed multiplication; 0x6400 | n is the half 1024 + n
        const half2_t k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
        const half2_t both = (__builtin_bit_cast(half2_t, (mn << 16) | sc | 0x64006400u) - k1024) * __builtin_bit_cast(half2_t, head[0]);
        D = both[0];
        DM = both[1];
    } else {
        D = Num<NUM>::scale((uint16_t)(head[0] & 0xFFFF)) * Num<NUM>::integer((int)sc);
        DM = Num<NUM>::scale((uint16_t)(head[0] >> 16)) * Num<NUM>::integer((int)mn);
    }
}

template <int NUM, bool FIVE>
struct SubQ45K {
    typedef typename Num<NUM>::T V;
    static constexpr bool kMin = true;
    static constexpr int kZero = 0;
    u32x4_t head;
    u32x2_t qs, qh;
    template <int J> __device__ __forceinline__ void load(const uint8_t* row, int g) {
        head = *reinterpret_cast<const u32x4_t*>(row);
        if constexpr (FIVE) qh = *reinterpret_cast<const u32x2_t*>(row + 16 + 8 * g);
        qs = *reinterpret_cast<const u32x2_t*>(row + (FIVE ? 48 : 16) + 32 * ((J & 3) >> 1) + 8 * g);
    }
    template <int J> __device__ __forceinline__ void scales(int, V& D, V& DM) const { q45k_scales<J, NUM>(head, D, DM); }
    template <int J> static constexpr int base() { return 1024 >> (4 * (J & 1)); }
    template <int J, int W> __device__ __forceinline__ void pairs(int, half2_t& a, half2_t& b) const {
        constexpr int P = 4 * (J & 1);
        if constexpr (FIVE) {
            a = field2<P, 0xF, 1, P + 4, P + 4 - J>(qs[W], qh[W]);
            b = field2<P, 0xF, 1, P + 4, P + 4 - J - 8>(qs[W] >> 8, qh[W]);
        } else {
            a = field<P, 0xF>(qs[W]);
            b = field<P, 0xF>(qs[W] >> 8);
        }
    }
};
template <int NUM> struct Sub<SNGGUF_TYPE_Q4_K, NUM> : SubQ45K<NUM, false> {};
template <int NUM> struct Sub<SNGGUF_TYPE_Q5_K, NUM> : SubQ45K<NUM, true> {};

template <int NUM> struct Sub<SNGGUF_TYPE_Q6_K, NUM> {
    typedef typename Num<NUM>::T V;
    static constexpr bool kMin = false;
    static constexpr int kZero = 32;
    uint32_t sw, d;
    u32x2_t ql, qh;
    template <int J> __device__ __forceinline__ void load(const uint8_t* row, int g) {
        constexpr int h = J >> 2, p = J & 3;
        sw = *reinterpret_cast<const uint32_t*>(row + 96 + 8 * h + 4 * (p >> 1));
        d = *reinterpret_cast<const uint16_t*>(row + 112);
        qh = *reinterpret_cast<const u32x2_t*>(row + 64 + 8 * g);
        ql = *reinterpret_cast<const u32x2_t*>(row + 32 * (p & 1) + 8 * g);
    }
    template <int J> __device__ __forceinline__ void scales(int g, V& D, V& DM) const {
        const int sc = (int)(int8_t)((sw >> (8 * (2 * (J & 1) + (g >> 1)))) & 0xFF);
        DM = D = Num<NUM>::scale((uint16_t)d) * Num<NUM>::integer(sc);
    }
    template <int J> static constexpr int base() { return 1024 >> (4 * ((J & 3) >> 1)); }
    template <int J, int W> __device__ __forceinline__ void pairs(int, half2_t& a, half2_t& b) const {
        constexpr int p = J & 3, P = 4 * (p >> 1);
        a = field2<P, 0xF, 3, P + 4, P + 4 - 2 * p>(ql[W], qh[W]);
        b = field2<P, 0xF, 3, P + 4, P + 4 - 2 * p - 8>(ql[W] >> 8, qh[W]);
    }
};

// 64-wide tiles of the activations in a stage: two (half as many barriers) up to 64 rows.  (64 rows in the narrow form: 64 KB of
// activations and eight slabs, 82 KB in all for Q8_0 and Q6_K, which leaves room for one workgroup on a compute unit, 74 - 78 KB and
// two for the others; Q8_0 with one tile and two workgroups takes 27.0 against 24.7 us for 4096 x 12288.)
constexpr int mid_tiles(int mt) { return mt <= 4 ? 2 : 1; }

// Bytes of a row of 32 outputs, and of 32 sums, in LDS behind the loop: odd numbers of 16-byte groups, so that eight rows start in
// different banks
constexpr int kOutRow = 80, kTurnRow = 144;

template <int QT, int R, int MT, int KW>
constexpr int mid_lds_bytes() {
    constexpr int x = 2 * KW * mid_tiles(MT) * 16 * MT * 128, slab = kWaves * 16 * R * Unit<QT>::stride;
    constexpr int red = KW == 2 ? kWaves * MT * 1024 : kWaves * MT * 16 * kOutRow;
    return x + slab > red ? x + slab : red;
}

// R: 16-row groups per wavefront, MT: 16-row tiles of the activations, KW: wavefronts that share a K range (1 or 2), FAR: packed pieces
// two units ahead instead of one.
template <int QT, int NUM, int R, int MT, int KW, bool FAR>
__global__ __launch_bounds__(64 * kWaves, R == 1 ? 4 : 2) void gemm_mid_kernel(MidArgs a) {
    typedef Unit<QT> S;
    constexpr int T = mid_tiles(MT);
    constexpr int NW = kWaves / KW;
    constexpr int kRows = 16 * R;
    constexpr int kPieces = kRows * S::pieces;
    constexpr int kLoads = (kPieces + 63) / 64;
    constexpr bool kQ6 = QT == SNGGUF_TYPE_Q6_K;
    constexpr int kTs = Slab<QT>::ts;             // bytes of 256 elements
    constexpr int kTile = 16 * MT * 128;          // one 64-wide tile of the activations
    constexpr int kStage = KW * T * kTile;
    constexpr int kStages = 4 / T;                // per super-block
    constexpr int kBlocks = 2 * MT;               // blocks of 8 rows (one request of a wavefront) in a tile
    // a stage's copies: per tile; where only all of its tiles together divide by the wavefronts, block wave + 8 q of these in one row
    // (24 blocks a stage, 48 rows: three copies a wavefront, not four with a quarter of them masked)
    constexpr bool kEven = kBlocks % kWaves != 0 && KW * T * kBlocks % kWaves == 0;
    constexpr int kReq = (kBlocks + kWaves - 1) / kWaves;
    constexpr int kCopies = kEven ? KW * T * kBlocks / kWaves : KW * T * kReq;
    constexpr int kOffs = kEven ? kCopies : kReq;   // addresses that differ by more than the tile
    constexpr bool kEarly = MT <= 8;              // a sub-block's bytes are read one sub-block ahead of its decode
    // Copies and requests between the matrix instructions, not in one go; up to 64 rows a stage is short and waits for what it asked
    // for late (40 rows of 4096 x 12288 in Q8_0 22.5 us in one go, 24.9 spread; 509 of 6144 x 4096 51 and 48).
    constexpr bool kSpread = MT > 4;
    static_assert(!kSpread || T == 1, "two stages between a unit's requests and the next unit's");
    // One request a group from the stage's start on, not one every few groups, in the shortest stages that are spread (90 rows of 12288 x
    // 4096, every few groups / every group: Q6_K 36.0 / 35.3 us, Q8_0 30.5 / 29.9; pairs 54.5 / 53.5 and 47.4 / 45.6).
    constexpr bool kDense = MT == 6;
    // A part of the decode is pinned to its place between the matrix instructions; left to itself the compiler computes it where it is
    // used.  Not up to 64 rows, where the parts' chains hide each other's latency better unpinned, and not at 256 rows, whose registers do
    // not suffice for it (Q5_K in fp32 decode 46 of them spilled, 1024 rows of 4096 x 12288 164 us, unpinned 125; without spills level).
    constexpr bool kPinned = MT > 4 && MT < 16;
    // Two units ahead takes the activations through registers (see load_x), about 20 more of them than one.  Narrow form of 32 rows
    // (launch_form): us in Q4_0 / Q8_0 / Q4_K, one and two units, 12288 x 4096 at 32 rows 18.5, 23.6, 19.7 and 16.8, 19.8, 18.4.  With 48
    // rows level, with 64 5 % slower, and in the wide form level up to 256 workgroups and slower beyond, where a compute unit then holds
    // one instead of two (151936 x 4096 at 24 rows 127, 160, 133 and 136, 167, 148).
    constexpr bool kRegX = FAR;
    constexpr int kAhead = kRegX ? 2 : 1;
    // Activation fragments read ahead; one fewer keeps the wide form of 32 and 48 rows within the 128 registers of two workgroups on a
    // compute unit in most formats (65536 x 4096 at 32 rows in Q8_0, 130 and 124 registers: 73.8 and 69.7 us).
    constexpr int kRing = R == 2 && MT <= 3 ? 3 : 4;
    // The narrow form of 32 rows with one unit ahead is for launches that fill the device several times over, where other workgroups fill
    // the gaps: raised priorities would hold these back (24576 x 4096 pair at 24 rows in Q6_K 73 us with them, 64 without).
    constexpr bool kPrio = !(R == 1 && MT == 2 && !FAR);
    static_assert(!kRegX || kEven, "a wavefront's blocks lie in one row");
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kw = wave / NW, nw = wave % NW;
    const int r = lane & 15, g = lane >> 4;

    // ---- tile: row tiles of the same columns and K slice next to each other on one XCD (workgroup ids are dealt round-robin
    // over 8), so that they find the packed rows in its L2 ----
    const int64_t total = a.col_tiles * a.row_tiles * a.ksplit;
    const int64_t pid = blockIdx.x, per = total >> 3, rem = total & 7, xcd = pid & 7;
    int64_t idx = xcd * per + (xcd < rem ? xcd : rem) + (pid >> 3);
    const int64_t ty = idx % a.row_tiles;
    idx /= a.row_tiles;
    const int slice = (int)(idx % a.ksplit);
    const int64_t tn = idx / a.ksplit;

    const int64_t row_begin = ty * a.tile_rows;
    const int64_t row_end = row_begin + a.tile_rows < a.M ? row_begin + a.tile_rows : a.M;
    // a pair: the first half of the column wavefronts on the gate rows, the second half on the same rows of up
    const int second = a.pair && nw >= NW / 2;
    const int64_t n0 = a.pair ? tn * (NW * 8 * R) + (second ? nw - NW / 2 : nw) * kRows : tn * (NW * kRows) + nw * kRows;
    const uint8_t* __restrict__ q = second ? a.q[1] : a.q[0];
    const int nsb = (int)(a.K >> 8);
    const int sb0 = (int)((int64_t)slice * nsb / a.ksplit), sb1 = (int)((int64_t)(slice + 1) * nsb / a.ksplit);
    const int steps = (sb1 - sb0 + KW - 1) / KW;
    const int my0 = sb0 + kw * steps;
    const int mine = my0 + steps <= sb1 ? steps : (sb1 > my0 ? sb1 - my0 : 0);   // super-blocks of this wavefront's share
    const int64_t row_bytes = (int64_t)nsb * kTs;
    const int xlast = 2 * (int)a.K - 128 * T;

    // ---- packed rows: pieces of this wavefront's rows (rows past the end: the last row, never stored) ----
    uint32_t off[S::second ? 1 : 2][kLoads], dst[kLoads];
    const int64_t nbase = n0 < a.N ? n0 : a.N - 1;
#pragma unroll
    for (int i = 0; i < kLoads; i++) {
        int f = lane + 64 * i;
        if (f >= kPieces) f = kPieces - 1;      // (a count of requests that all lanes agree on: the waits below rely on it)
        const int fr = f / S::pieces, fp = f % S::pieces;
        int64_t n = nbase + fr;
        if (n >= a.N) n = a.N - 1;
        const uint32_t ro = (uint32_t)((n - nbase) * row_bytes);
        off[0][i] = ro + S::src(0, fp);
        if constexpr (S::second == 0) off[1][i] = ro + S::src(1, fp);
        dst[i] = (uint32_t)(fr * S::stride + 16 * fp);
    }
    uint32_t doff = 0;
    if constexpr (kQ6) {
        int64_t n = nbase + (lane & (kRows - 1));
        if (n >= a.N) n = a.N - 1;
        doff = (uint32_t)((n - nbase) * row_bytes + 208);
    }
    const uint8_t* __restrict__ base = q + nbase * row_bytes;
    uint8_t* slab = lds + 2 * kStage + wave * kRows * S::stride;
    u32x4_t pre[kAhead][kLoads];
    uint16_t pre_d[kAhead] = {};
    // request i of unit h of super-block s of the share (a share that ends early re-reads the slice's last super-block)
    constexpr int kFetch = kLoads + (kQ6 ? 1 : 0);
    auto fetch_req = [&](int s, auto H, int i) {
        constexpr int h = decltype(H)::value;
        const uint8_t* p = base + (int64_t)(my0 + s < sb1 ? my0 + s : sb1 - 1) * kTs;
        if (i < kLoads) pre[h % kAhead][i] = ld_piece<S::align>(p + h * S::second + off[S::second ? 0 : h][i]);
        else if constexpr (kQ6) pre_d[h % kAhead] = ld_u16(p + doff);
    };
    auto fetch = [&](int s, auto H) {
#pragma unroll
        for (int i = 0; i < kFetch; i++) fetch_req(s, H, i);
    };
    auto put = [&](auto H) {
        constexpr int set = decltype(H)::value % kAhead;
#pragma unroll
        for (int i = 0; i < kLoads; i++) *reinterpret_cast<u32x4_t*>(slab + dst[i]) = pre[set][i];
        if constexpr (kQ6) *reinterpret_cast<uint16_t*>(slab + (lane & (kRows - 1)) * S::stride + 112) = pre_d[set];
    };

    // ---- activations: rows past the end of the tile re-read its last row ----
    uint32_t xoff[kOffs];
#pragma unroll
    for (int i = 0; i < kOffs; i++) {
        const int row = 8 * (kEven ? (wave + kWaves * i) % kBlocks : wave + kWaves * i) + (lane >> 3);
        int64_t gr = row_begin + row;
        if (gr >= row_end) gr = row_end - 1;
        xoff[i] = (uint32_t)(2 * gr * a.K + 16 * ((lane & 7) ^ ((row >> 1) & 7)));
    }
    // (where the copies do not divide, the last of a tile is made with no lane enabled by the other wavefronts - a branch there would
    // cut the stage into basic blocks, and the decode that belongs between the matrix instructions of one stage would be moved to the
    // head of the next)
    const int last_req = __builtin_amdgcn_readfirstlane(wave < kBlocks - kWaves * (kReq - 1) ? -1 : 0);
    // request q of the tiles of stage st of super-block s of every K share
    auto load_x_req = [&](int s, int st, int q) {
        const int block = wave + kWaves * (kEven ? q : q % kReq), kt = kEven ? block / kBlocks : q / kReq;
        int col = (sb0 + kt / T * steps + s) * 512 + 128 * T * st;      // byte column
        if (KW > 1 && col > xlast) col = xlast;
        const uint8_t* xb = wave_ptr(reinterpret_cast<const uint8_t*>(a.x) + col + 128 * (kt % T));
        const uint32_t to = lds_addr(lds) + (uint32_t)((st & 1) * kStage + (kEven ? 0 : kt * kTile) + block * 1024);
        // (as the dense kernels' copies: M0 holds the destination, one wait state between its write and the request)
        if (!kEven && kBlocks % kWaves != 0 && q % kReq == kReq - 1)
            asm volatile("s_mov_b32 m0, %0\n\ts_mov_b32 exec_lo, %3\n\ts_mov_b32 exec_hi, %3\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1"
                         ::"s"(to), "v"(xoff[q % kOffs]), "s"(xb), "s"(last_req) : "memory", "m0");
        else
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(xoff[q % kOffs]), "s"(xb) : "memory", "m0");
    };
    // Through registers (kRegX), and to LDS at the stage's end (store_x): a copy straight to LDS is a request that the compiler does not
    // know of, and its waits for the packed pieces of one unit would then not let those of the next stay out.
    u32x4_t xreg[kRegX ? kCopies : 1];
    auto load_x = [&](int s, int st) {
#pragma unroll
        for (int q = 0; q < kCopies; q++) {
            if constexpr (kRegX) {
                const int kt = (wave + kWaves * q) / kBlocks;
                int col = (sb0 + kt / T * steps + s) * 512 + 128 * T * st;
                if (col > xlast) col = xlast;
                xreg[q] = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const uint8_t*>(a.x) + col + 128 * (kt % T) + xoff[q]);
            } else {
                load_x_req(s, st, q);
            }
        }
    };
    auto store_x = [&](int st) {
#pragma unroll
        for (int q = 0; q < (kRegX ? kCopies : 0); q++) *reinterpret_cast<u32x4_t*>(lds + (st & 1) * kStage + (wave + kWaves * q) * 1024 + 16 * lane) = xreg[q];
    };
    int foff[2];
#pragma unroll
    for (int j = 0; j < 2; j++) foff[j] = r * 128 + 16 * ((4 * j + g) ^ ((r >> 1) & 7));

    f32x4_t acc[R][MT];
#pragma unroll
    for (int rg = 0; rg < R; rg++)
#pragma unroll
        for (int t = 0; t < MT; t++) acc[rg][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // ---- decode of a sub-block into operands d: per row group its LDS reads, then five parts of at most a dozen instructions: scales, and
    // each dword of four weights in two halves ----
    Sub<QT, NUM> sub[kEarly ? 2 : 1][R];
    typename Num<NUM>::T D[R], DM[R];
    half2_t ha, hb;
    auto read_part = [&](auto J, int rg) {
        constexpr int j = decltype(J)::value & 7;
        sub[kEarly ? j & 1 : 0][rg].template load<j>(slab + (16 * rg + r) * S::stride, g);
    };
    auto decode_part = [&](auto J, auto C, u32x4_t (&d)[R]) {
        constexpr int j = decltype(J)::value & 7, rg = decltype(C)::value / 5, part = decltype(C)::value % 5, w = (part - 1) / 2;
        typedef Sub<QT, NUM> B;
        const B& b = sub[kEarly ? j & 1 : 0][rg];
        if constexpr (part == 0) {
            b.template scales<j>(g, D[rg], DM[rg]);
        } else if constexpr (part % 2 == 1) {
            constexpr float off = (float)(B::template base<j>() + B::kZero);
            b.template pairs<j, w>(g, ha, hb);
            chain_pair<NUM, B::kMin>(ha, off, D[rg], DM[rg]);
            chain_pair<NUM, B::kMin>(hb, off, D[rg], DM[rg]);
            if constexpr (kPinned) asm volatile("" : "+v"(ha), "+v"(hb));
        } else {
            uint32_t p01, p23;
            chain_bf16<NUM, B::kMin>(ha, hb, D[rg], DM[rg], p01, p23);
            if constexpr (kPinned) asm volatile("" : "+v"(p01), "+v"(p23));
            d[rg][2 * w] = p01; d[rg][2 * w + 1] = p23;
        }
    };
    u32x4_t af[2][R];
    // The sub-blocks of stage ST; under the matrix instructions of sub-block j the next one is decoded, and the bytes of the
    // one after it (kEarly) or of the next one are read - in front of a unit's first, the unit moves from registers to the slab
    // and the unit after it is requested.
    auto contract = [&](auto ST, auto LAST, int s) {
        constexpr int st = decltype(ST)::value;
        constexpr bool last = decltype(LAST)::value;
        constexpr int n = 2 * T * MT;           // activation fragments of the stage
        const uint8_t* xt = lds + (st & 1) * kStage + kw * (T * kTile);
        auto frag = [&](int i) { return *reinterpret_cast<const bf16x8_t*>(xt + (i / MT >> 1) * kTile + (i % MT) * 2048 + foff[i / MT & 1]); };
        bf16x8_t xf[kRing];
#pragma unroll
        for (int i = 0; i < kRing && i < n; i++) xf[i] = frag(i);
        __builtin_amdgcn_sched_barrier(0);
        static_for<n>([&](auto I) {
            constexpr int i = decltype(I)::value, u = i / MT, t = i % MT, j = 2 * T * st + u;
            constexpr int jr = kEarly ? j + 2 : j + 1;       // sub-block whose bytes are read under this one
            // A wavefront's priority falls as it gets through the stage: the two of a SIMD would otherwise be served oldest first, and
            // the younger would run its last third alone (203 rows: contracting took 2070 and 3180 cycles of a stage of 3340, now 2440
            // and 2950 of 3120).
            if constexpr (kPrio && i == 0) __builtin_amdgcn_s_setprio(3);
            else if constexpr (kPrio && i == n / 4) __builtin_amdgcn_s_setprio(2);
            else if constexpr (kPrio && i == n / 2) __builtin_amdgcn_s_setprio(1);
            else if constexpr (kPrio && i == 3 * n / 4) __builtin_amdgcn_s_setprio(0);
            if constexpr (t == 0 && (jr == 4 || (jr == 8 && !last))) {
                put(int_c<jr == 4>{});
                if constexpr (kRegX && !last) fetch(s + jr / 4, int_c<jr == 4>{});
                else if constexpr (!kSpread && !last) fetch(s + 1, int_c<jr / 4 - 1>{});
            }
#pragma unroll
            for (int rg = 0; rg < R; rg++)
                acc[rg][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, af[j & 1][rg]), xf[i % kRing], acc[rg][t], 0, 0, 0);
            if constexpr (i + kRing < n) xf[i % kRing] = frag(i + kRing);
            if constexpr (kSpread) {
                // the next stage's copies under the first half of this one, the packed pieces of the next unit but one under the
                // second half (kDense: behind the copies) of the stage in which the next unit went to the slab (the wait for the copies
                // counts on that order)
                static_assert(!kDense || kCopies + kFetch <= n, "a group for every request");
                if constexpr (!last || st + 1 < kStages)
#pragma unroll
                    for (int q = 0; q < kCopies; q++)
                        if ((kDense ? q : q * (n / 2) / kCopies) == i) load_x_req(s + (st + 1) / kStages, (st + 1) % kStages, q);
                if constexpr (!last && (st & 1) == 1)
#pragma unroll
                    for (int q = 0; q < kFetch; q++)
                        if ((kDense ? kCopies + q : n / 2 + q * (n / 2) / kFetch) == i) fetch_req(s + 1, int_c<st / 2>{}, q);
            }
            constexpr int first = (t * 6 * R + MT - 1) / MT, past = ((t + 1) * 6 * R + MT - 1) / MT;   // parts of this group
            static_for<past - first>([&](auto C) {
                constexpr int c = first + decltype(C)::value;
                if constexpr (c < R) { if constexpr (!last || jr < 8) read_part(int_c<jr>{}, c); }
                else if constexpr (!last || j < 7) decode_part(int_c<j + 1>{}, int_c<(c < R ? 0 : c - R)>{}, af[(j + 1) & 1]);
            });
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    // One super-block.  A stage's tiles must have arrived when it begins; they were requested at the start of the stage before
    // it, and requests return in order: the pieces requested under that stage (kLoads and, for Q6_K, one more; sub-blocks 2
    // or 3 and 6 or 7) may stay out.  WORK: this wavefront's share still has super-blocks, so it made those requests; LAST: the
    // workgroup's last super-block.  Every wavefront passes the same barriers.
    auto super_block = [&](auto WORK, auto LAST, int s) {
        constexpr bool work = decltype(WORK)::value, last = decltype(LAST)::value;
        static_for<kStages>([&](auto ST) {
            constexpr int st = decltype(ST)::value;
            constexpr int kYoung = work && !last && (T == 2 || (st & 1) == 0) ? kLoads : 0;
            if constexpr (kRegX) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kYoung) : "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if constexpr ((!work || !kSpread) && (!last || st + 1 < kStages)) load_x(s + (st + 1) / kStages, (st + 1) % kStages);
            if constexpr (work) contract(ST, LAST, s);
            if constexpr (kRegX && (!last || st + 1 < kStages)) store_x(st + 1);
        });
    };
    load_x(0, 0);
    fetch(0, int_c<0>{});
    if constexpr (kRegX) fetch(0, int_c<1>{});
    store_x(0);
    put(int_c<0>{});
    if constexpr (kRegX) fetch(1, int_c<0>{});
    else fetch(0, int_c<1>{});
#pragma unroll
    for (int c = 0; c < R; c++) {
        read_part(int_c<0>{}, c);
        if (kEarly) read_part(int_c<1>{}, c);
    }
    static_for<5 * R>([&](auto C) { decode_part(int_c<0>{}, C, af[0]); });
    int s = 0;
    for (const int whole = mine < steps ? mine : steps - 1; s < whole; s++) super_block(int_c<true>{}, int_c<false>{}, s);
    if (mine == steps) {
        super_block(int_c<true>{}, int_c<true>{}, s);
    } else {
        for (; s < steps - 1; s++) super_block(int_c<false>{}, int_c<false>{}, s);
        super_block(int_c<false>{}, int_c<true>{}, s);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __syncthreads();

    // ---- sums out: lane r holds activation row r of a row tile, its four values are four consecutive columns ----
    f32x4_t* red = reinterpret_cast<f32x4_t*>(lds);
    const bool vec = (a.N & 3) == 0;
    // columns n .. n + 3 of activation row m: outputs, or this slice's partial sums of matrix `sec`
    auto store = [&](int sec, int64_t m, int64_t n, const f32x4_t& v) {
        if (a.partial) {
            float* pp = a.partial + (((int64_t)sec * a.ksplit + slice) * a.M + m) * a.N + n;
            if (vec) {
                *reinterpret_cast<f32x4_t*>(pp) = v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (n + e < a.N) pp[e] = v[e];
            }
            return;
        }
        const int64_t yi = m * a.N + n;
        float o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (n + e < a.N) o[e] = add_residual(v[e] + (a.bias ? bf16_to_f32(a.bias[n + e]) : 0.f), a.residual, yi + e);
        if (vec) {
            *reinterpret_cast<u32x2_t*>(a.y + yi) = u32x2_t{pack_bf16(o[0], o[1]), pack_bf16(o[2], o[3])};
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n + e < a.N) a.y[yi + e] = f32_to_bf16(o[e]);
        }
    };
    auto gated_bf16 = [](float gv, float uv) { return bf16_to_f32(f32_to_bf16(silu_f32(gv))) * uv; };
    auto store_gated = [&](int64_t m, int64_t n, const f32x4_t& gt, const f32x4_t& ut) {
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = gated_bf16(bf16_to_f32(f32_to_bf16(gt[e])), bf16_to_f32(f32_to_bf16(ut[e])));
        *reinterpret_cast<u32x2_t*>(a.y + m * a.N + n) = u32x2_t{pack_bf16(o[0], o[1]), pack_bf16(o[2], o[3])};
    };
    if constexpr (R == 1) {
        // every (column wavefront, row tile) is added up and stored by one wavefront; a gated pair's with its up half's
#pragma unroll
        for (int t = 0; t < MT; t++) red[(wave * MT + t) * 64 + lane] = acc[0][t];
        __syncthreads();
        const bool gated = a.pair && !a.partial;
        auto sum = [&](int i) {
            f32x4_t v = red[i * 64 + lane];
            const f32x4_t p = red[(NW * MT + i) * 64 + lane];
            v[0] += p[0]; v[1] += p[1]; v[2] += p[2]; v[3] += p[3];
            return v;
        };
        for (int i = wave; i < (gated ? NW / 2 : NW) * MT; i += kWaves) {
            const int c = i / MT, t = i - c * MT, sec = a.pair && c >= NW / 2;
            const int64_t m = row_begin + 16 * t + r;
            const int64_t n = (a.pair ? tn * (NW * 8) + (sec ? c - NW / 2 : c) * 16 : tn * (NW * 16) + c * 16) + 4 * g;
            if (m >= row_end || n >= a.N) continue;
            if (gated) store_gated(m, n, sum(i), sum(i + NW / 2 * MT));
            else store(sec, m, n, sum(i));
        }
        return;
    }
    if constexpr (KW == 2) {
        // two halves of K: wavefront kw keeps tiles kw, kw + 2, .. and adds the other half's sums to them
        constexpr int kOdd = MT / 2, kEven = MT - kOdd;
        f32x4_t* give = red + (kw == 0 ? nw * kOdd : NW * kOdd + nw * kEven) * (R * 64) + lane;
        const f32x4_t* take = red + (kw == 0 ? NW * kOdd + nw * kEven : nw * kOdd) * (R * 64) + lane;
#pragma unroll
        for (int t = 0; t < MT; t++) {
            if ((t & 1) == kw) continue;
#pragma unroll
            for (int rg = 0; rg < R; rg++) give[(t / 2 * R + rg) * 64] = acc[rg][t];
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < MT; t++) {
            if ((t & 1) != kw) continue;
#pragma unroll
            for (int rg = 0; rg < R; rg++) {
                const f32x4_t p = take[(t / 2 * R + rg) * 64];
                acc[rg][t][0] += p[0]; acc[rg][t][1] += p[1]; acc[rg][t][2] += p[2]; acc[rg][t][3] += p[3];
            }
        }
        __syncthreads();
    }
    if (a.pair && !a.partial) {
        // both projections' outputs, rounded, as rows of 32 columns in LDS; gate wavefronts finish every other tile, up wavefronts
        // the rest, eight columns a lane
        constexpr int kOwn = (MT + KW - 1) / KW;
        uint8_t* out = lds + wave * (kOwn * 16 * kOutRow);
#pragma unroll
        for (int t = 0; t < MT; t++) {
            if (KW == 2 && (t & 1) != kw) continue;
#pragma unroll
            for (int rg = 0; rg < R; rg++)
                *reinterpret_cast<u32x2_t*>(out + (t / KW * 16 + r) * kOutRow + 32 * rg + 8 * g) =
                    u32x2_t{pack_bf16(acc[rg][t][0], acc[rg][t][1]), pack_bf16(acc[rg][t][2], acc[rg][t][3])};
        }
        __syncthreads();
        const uint8_t* gates = lds + (second ? wave - NW / 2 : wave) * (kOwn * 16 * kOutRow);
        const uint8_t* ups = gates + NW / 2 * (kOwn * 16 * kOutRow);
        const int row = lane >> 2;
        const int64_t n = n0 + 8 * (lane & 3);
        for (int o = second; o < kOwn; o += 2) {
            const int64_t m = row_begin + 16 * (KW == 2 ? 2 * o + kw : o) + row;
            if (m >= row_end || n >= a.N) continue;
            const u32x4_t gt = *reinterpret_cast<const u32x4_t*>(gates + (o * 16 + row) * kOutRow + 16 * (lane & 3));
            const u32x4_t ut = *reinterpret_cast<const u32x4_t*>(ups + (o * 16 + row) * kOutRow + 16 * (lane & 3));
            u32x4_t h;
#pragma unroll
            for (int e = 0; e < 4; e++)
                h[e] = pack_bf16(gated_bf16(bf16lo_to_f32(gt[e]), bf16lo_to_f32(ut[e])), gated_bf16(bf16hi_to_f32(gt[e]), bf16hi_to_f32(ut[e])));
            *reinterpret_cast<u32x4_t*>(a.y + m * a.N + n) = h;   // (a pair has whole groups of eight columns)
        }
        return;
    }
    // a tile at a time through LDS of the wavefront's own, so that a store writes whole rows of 32 columns (128 bytes of partial sums)
    uint8_t* turn = lds + wave * (16 * kTurnRow);
#pragma unroll
    for (int t = 0; t < MT; t++) {
        if (KW == 2 && (t & 1) != kw) continue;
#pragma unroll
        for (int rg = 0; rg < R; rg++) *reinterpret_cast<f32x4_t*>(turn + r * kTurnRow + 64 * rg + 16 * g) = acc[rg][t];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int row = 8 * i + (lane >> 3);
            const f32x4_t v = *reinterpret_cast<const f32x4_t*>(turn + row * kTurnRow + 16 * (lane & 7));
            const int64_t m = row_begin + 16 * t + row, n = n0 + 4 * (lane & 7);
            if (m < row_end && n < a.N) store(second, m, n, v);
        }
    }
}

template <int QT, int NUM, int R, int MT, int KW, bool FAR>
int launch(const MidArgs& a, hipStream_t stream) {
    constexpr int kLds = mid_lds_bytes<QT, R, MT, KW>();
    static_assert(kLds <= 160 * 1024, "LDS of a compute unit");
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_mid_kernel<QT, NUM, R, MT, KW, FAR>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (attr != hipSuccess) return SNGGUF_E_LAUNCH;
    gemm_mid_kernel<QT, NUM, R, MT, KW, FAR><<<dim3((unsigned)(a.col_tiles * a.row_tiles * a.ksplit)), dim3(64 * kWaves), kLds, stream>>>(a);
    return hipGetLastError() == hipSuccess ? SNGGUF_OK : SNGGUF_E_LAUNCH;
}

template <int NUM>
int launch_form(const MidArgs& a, int form, int mt, hipStream_t stream) {
    constexpr int QT = SNGGUF_MID_TYPE;
#define SNGGUF_CASE(FORM, R, MT, KW) if (form == FORM && mt == MT) return launch<QT, NUM, R, MT, KW, false>(a, stream)
    // Two units of packed rows ahead while every compute unit has at most the two workgroups that fit it so; beyond, one unit ahead (us in
    // Q4_0 / Q2_K / Q8_0 / Q6_K, two and one: pair of 20480 x 4096 at 32 rows, 640 workgroups, 41, 44.4, 51.6, 62.8 and 41, 40.6, 51.7, 61.6;
    // pair of 24576 x 4096 at 24 rows 49, 50.1, 56.4, 65.3 and 44.5, 43.7, 56.4, 64.0)
    if (form == kMidNarrow && mt == 2) {
        if (a.col_tiles * a.row_tiles * a.ksplit <= 512) return launch<QT, NUM, 1, 2, 2, true>(a, stream);
        return launch<QT, NUM, 1, 2, 2, false>(a, stream);
    }
    SNGGUF_CASE(kMidNarrow, 1, 3, 2);
    SNGGUF_CASE(kMidNarrow, 1, 4, 2);
    SNGGUF_CASE(kMidWide, 2, 2, 2);
    SNGGUF_CASE(kMidWide, 2, 3, 2);
    SNGGUF_CASE(kMidWide, 2, 4, 2);
    SNGGUF_CASE(kMidWide, 2, 6, 2);
    SNGGUF_CASE(kMidWide, 2, 8, 2);
    SNGGUF_CASE(kMidWide, 2, 10, 2);
    SNGGUF_CASE(kMidWide, 2, 13, 2);
    SNGGUF_CASE(kMidLong, 2, 10, 1);
    SNGGUF_CASE(kMidLong, 2, 13, 1);
    SNGGUF_CASE(kMidLong, 2, 16, 1);
#undef SNGGUF_CASE
    return SNGGUF_E_BADSHAPE;
}

}  // namespace

template <>
int launch_mid_type<SNGGUF_MID_TYPE>(const MidArgs& a, int form, int mt, int numerics, hipStream_t stream) {
    if (numerics == SNGGUF_NUM_GGML_FP32) return launch_form<SNGGUF_NUM_GGML_FP32>(a, form, mt, stream);
    if (numerics == SNGGUF_NUM_UPSTREAM_FP16) return launch_form<SNGGUF_NUM_UPSTREAM_FP16>(a, form, mt, stream);
    return SNGGUF_E_BADTYPE;
}

}  // namespace sngguf
