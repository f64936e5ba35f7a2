// Dequant-GEMM for 17 rows to a few thousand (K % 256 == 0), all ten block formats: the packed rows go from memory to matrix-core
// operands in registers, each decoded once per tile of up to 256 activation rows; no weight pass, and no decoded weight in LDS.
//
// Eight wavefronts share one tile of activations; each owns 16 or 32 weight rows and (with KW = 2) one half of the
// workgroup's K range.  Three forms (mid_plan in gemm_mid_plan.hip picks):
//   narrow  16 rows per wavefront, two halves of K:  64 columns per workgroup, up to 64 rows, two workgroups per compute unit
//           (one with 64 rows in Q8_0 and Q6_K, whose slabs are the widest)
//   wide    32 rows per wavefront, two halves of K: 128 columns, up to 208 rows
//   long    32 rows per wavefront, all of K:        256 columns, up to 256 rows
// (wide ends at 208 rows because its registers do: 224 - 256 of 256 are taken there, and Q8_0 already spills 7 of them, the only
// instance of any format that spills.  From 209 rows on two row tiles, or the long form, take 15 - 18 % longer than 208 rows.)
// What bounds it: up to about 64 rows the latency of a step (packed bytes -> slab -> decode -> matrix instructions, which two
// wavefronts a SIMD hide only partly), beyond that the issue slots of the SIMD, which matrix instructions and the decode's 3.5 - 4
// vector instructions per weight share (16x16x32 instructions alone take 3.3 us per super-block of 256 columns and 208 rows, the
// kernel 4.9 - 5.8).  So the loop is written out instruction group by instruction group: two matrix instructions, the
// activation fragment of four groups later, an eighth of the next sub-block's decode, a scheduling fence.  Left to the
// compiler's scheduler the fragments are read one instruction ahead (gate / up of 12288 x 4096 at 203 rows 100 us against 69).
//
// Per wavefront and unit of 128 elements of K: the packed bytes are requested a unit ahead into registers (16-byte pieces,
// consecutive lanes walking along a row) and put into a slab of the wavefront's own; the decode reads them from there.
// Activations: 64 (or, up to 64 rows, 128) columns of every row and half of K are copied global -> LDS directly one stage ahead,
// in rows of 128 bytes whose 16-byte chunk c sits at c ^ ((row / 2) % 8); one barrier a stage.
//
// Measured, one projection with its reduction / pair of 12288 x 4096 and what ran before it (us; graphs of launches on weights
// from memory, Q8_0 / Q4_K / Q6_K):
//   40 rows   pair 40 / 35 / 45 (decode kernels, two launches 66 / 57 / 67), 4096 x 12288 23 / 21 / 26 (36 / 33 / 36)
//   203 rows  pair 65 / 61 (split tiles 84 / 83), 4096 x 12288 41 / 39 / 44 (51 / 50 / 75), 6144 x 4096 31 / 30 / 32 (37 / 37 / 49)
//   509 rows  pair 114 / 109 (150 / 142), 4096 x 12288 70 / 70 (79 / 79)
//   1024 rows pair 220 / 220 (dense launch with two weight passes 247 / 232), 4096 x 4096 55 / 56 (68 / 68)
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
constexpr int kRing = 4;          // activation fragments read ahead

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
// Formats whose unit is no multiple of 16 bytes end with a piece that overlaps its predecessor in memory.
template <int TS, int PIECES, int STRIDE>
struct UnitBlocks {   // four blocks of TS bytes
    static constexpr int pieces = PIECES, stride = STRIDE, align = 4, last = 4 * TS - 16;
    static __device__ __forceinline__ int src(int h, int p) { return 4 * TS * h + (p == PIECES - 1 ? last : 16 * p); }
};
template <int QT> struct Unit;
template <> struct Unit<SNGGUF_TYPE_Q4_0> : UnitBlocks<18, 5, 80> {};
template <> struct Unit<SNGGUF_TYPE_Q4_1> : UnitBlocks<20, 5, 80> {};
template <> struct Unit<SNGGUF_TYPE_Q5_0> : UnitBlocks<22, 6, 112> {};
template <> struct Unit<SNGGUF_TYPE_Q5_1> : UnitBlocks<24, 6, 112> {};
template <> struct Unit<SNGGUF_TYPE_Q8_0> : UnitBlocks<34, 9, 144> {};
template <> struct Unit<SNGGUF_TYPE_Q2_K> {   // scales, quants of the half, d and dmin in the last dword
    static constexpr int pieces = 4, stride = 80, align = 4;
    static __device__ __forceinline__ int src(int h, int p) { return p == 0 ? 0 : p == 3 ? 68 : 32 * h + 16 * p; }
};
template <> struct Unit<SNGGUF_TYPE_Q3_K> {   // mask, quants of the half, scales and d
    static constexpr int pieces = 5, stride = 80, align = 2;
    static __device__ __forceinline__ int src(int h, int p) { return p < 2 ? 16 * p : p == 4 ? 94 : 32 * h + 16 * p; }
};
template <> struct Unit<SNGGUF_TYPE_Q4_K> {   // head, quants of the half
    static constexpr int pieces = 5, stride = 80, align = 16;
    static __device__ __forceinline__ int src(int h, int p) { return p == 0 ? 0 : 64 * h + 16 * p; }
};
template <> struct Unit<SNGGUF_TYPE_Q5_K> {   // head, fifth bits, quants of the half
    static constexpr int pieces = 7, stride = 112, align = 16;
    static __device__ __forceinline__ int src(int h, int p) { return p < 3 ? 16 * p : 64 * h + 16 * p; }
};
template <> struct Unit<SNGGUF_TYPE_Q6_K> {   // low and high bits of the half, scales; d follows on its own at byte 112
    static constexpr int pieces = 7, stride = 144, align = 2;
    static __device__ __forceinline__ int src(int h, int p) { return p < 4 ? 64 * h + 16 * p : p < 6 ? 64 + 32 * h + 16 * p : 192; }
};

// One 32-element sub-block of a slab row for lane group g, in three parts that the K loop places between matrix
// instructions: the LDS reads (`load`), the sub-block's scale and minimum (`scales`), and its eight quants as two dwords
// of four unsigned bytes (`quads`).  J: sub-block 0 .. 7 of the 256 elements.
template <int QT, int NUM> struct Sub;

template <int NUM, int TS, bool HAS_MIN, bool FIVE>
struct SubLegacy {
    typedef typename Num<NUM>::T V;
    static constexpr bool kMin = HAS_MIN;
    static constexpr float kZero = HAS_MIN ? 0.f : (FIVE ? 16.f : 8.f);
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
    template <int J, int W> __device__ __forceinline__ uint32_t quads(int g) const {
        uint32_t v = (qs[W] >> (4 * (g >> 1))) & 0x0F0F0F0Fu;
        if constexpr (FIVE) v |= ((((fifth >> (8 * g + 4 * W)) & 0xFu) * 0x00204081u) & 0x01010101u) << 4;
        return v;
    }
};
template <int NUM> struct Sub<SNGGUF_TYPE_Q4_0, NUM> : SubLegacy<NUM, 18, false, false> {};
template <int NUM> struct Sub<SNGGUF_TYPE_Q4_1, NUM> : SubLegacy<NUM, 20, true, false> {};
template <int NUM> struct Sub<SNGGUF_TYPE_Q5_0, NUM> : SubLegacy<NUM, 22, false, true> {};
template <int NUM> struct Sub<SNGGUF_TYPE_Q5_1, NUM> : SubLegacy<NUM, 24, true, true> {};

template <int NUM> struct Sub<SNGGUF_TYPE_Q8_0, NUM> {
    typedef typename Num<NUM>::T V;
    static constexpr bool kMin = false;
    static constexpr float kZero = 128.f;
    uint32_t hd;
    u32x2_t qs;
    template <int J> __device__ __forceinline__ void load(const uint8_t* row, int g) {
        constexpr int jj = J & 3;
        hd = *reinterpret_cast<const uint16_t*>(row + 34 * jj);
        // (the unit's last 8 bytes lie in the overlapping piece)
        qs = lds_u64<(jj & 1) == 1>(row + 34 * jj + 2 + 8 * g + (jj == 3 && g == 3 ? 8 : 0));
    }
    template <int J> __device__ __forceinline__ void scales(int, V& D, V& DM) const { DM = D = Num<NUM>::scale((uint16_t)hd); }
    template <int J, int W> __device__ __forceinline__ uint32_t quads(int) const { return qs[W] ^ 0x80808080u; }
};

template <int NUM> struct Sub<SNGGUF_TYPE_Q2_K, NUM> {
    typedef typename Num<NUM>::T V;
    static constexpr bool kMin = true;
    static constexpr float kZero = 0.f;
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
    template <int J, int W> __device__ __forceinline__ uint32_t quads(int) const { return (qs[W] >> (2 * (J & 3))) & 0x03030303u; }
};

template <int NUM> struct Sub<SNGGUF_TYPE_Q3_K, NUM> {
    typedef typename Num<NUM>::T V;
    static constexpr bool kMin = false;
    static constexpr float kZero = 4.f;
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
    template <int J, int W> __device__ __forceinline__ uint32_t quads(int) const {
        return ((qs[W] >> (2 * (J & 3))) & 0x03030303u) | (((hm[W] >> J) & 0x01010101u) << 2);
    }
};

template <int NUM, bool FIVE>
struct SubQ45K {
    typedef typename Num<NUM>::T V;
    static constexpr bool kMin = true;
    static constexpr float kZero = 0.f;
    u32x4_t head;
    u32x2_t qs, qh;
    template <int J> __device__ __forceinline__ void load(const uint8_t* row, int g) {
        head = *reinterpret_cast<const u32x4_t*>(row);
        if constexpr (FIVE) qh = *reinterpret_cast<const u32x2_t*>(row + 16 + 8 * g);
        qs = *reinterpret_cast<const u32x2_t*>(row + (FIVE ? 48 : 16) + 32 * ((J & 3) >> 1) + 8 * g);
    }
    template <int J> __device__ __forceinline__ void scales(int, V& D, V& DM) const {
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
    template <int J, int W> __device__ __forceinline__ uint32_t quads(int) const {
        uint32_t v = (qs[W] >> (4 * (J & 1))) & 0x0F0F0F0Fu;
        if constexpr (FIVE) v |= ((qh[W] >> J) & 0x01010101u) << 4;
        return v;
    }
};
template <int NUM> struct Sub<SNGGUF_TYPE_Q4_K, NUM> : SubQ45K<NUM, false> {};
template <int NUM> struct Sub<SNGGUF_TYPE_Q5_K, NUM> : SubQ45K<NUM, true> {};

template <int NUM> struct Sub<SNGGUF_TYPE_Q6_K, NUM> {
    typedef typename Num<NUM>::T V;
    static constexpr bool kMin = false;
    static constexpr float kZero = 32.f;
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
    template <int J, int W> __device__ __forceinline__ uint32_t quads(int) const {
        constexpr int p = J & 3;
        return ((ql[W] >> (4 * (p >> 1))) & 0x0F0F0F0Fu) | (((qh[W] >> (2 * p)) & 0x03030303u) << 4);
    }
};

// 64-wide tiles of the activations in a stage: two (half as many barriers) up to 64 rows.  (64 rows in the narrow form: 64 KB of
// activations and eight slabs, 82 KB in all for Q8_0 and Q6_K, which leaves room for one workgroup on a compute unit, 74 - 78 KB and
// two for the others; Q8_0 with one tile and two workgroups takes 27.0 against 24.7 us for 4096 x 12288.)
constexpr int mid_tiles(int mt) { return mt <= 4 ? 2 : 1; }

template <int QT, int R, int MT, int KW>
constexpr int mid_lds_bytes() {
    constexpr int x = 2 * KW * mid_tiles(MT) * 16 * MT * 128, slab = kWaves * 16 * R * Unit<QT>::stride;
    constexpr int red = KW == 2 ? kWaves * MT * 1024 : kWaves * R * ((MT + 1) / 2) * 1024;
    return x + slab > red ? x + slab : red;
}

// R: 16-row groups per wavefront, MT: 16-row tiles of the activations, KW: wavefronts that share a K range (1 or 2).
template <int QT, int NUM, int R, int MT, int KW>
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
    constexpr int kReq = (kBlocks + kWaves - 1) / kWaves;
    constexpr bool kEarly = MT <= 8;              // a sub-block's bytes are read one sub-block ahead of its decode
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kw = wave / NW, nw = wave % NW;
    const int r = lane & 15, g = lane >> 4;
    const half4_t ident = identity_row(lane);

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
    uint32_t off[2][kLoads], dst[kLoads];
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
        off[1][i] = ro + S::src(1, fp);
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
    u32x4_t pre[kLoads];
    uint16_t pre_d = 0;
    // unit h of super-block s of the share (a share that ends early re-reads the slice's last super-block)
    auto fetch = [&](int s, auto H) {
        constexpr int h = decltype(H)::value;
        const uint8_t* p = base + (int64_t)(my0 + s < sb1 ? my0 + s : sb1 - 1) * kTs;
#pragma unroll
        for (int i = 0; i < kLoads; i++) pre[i] = ld_piece<S::align>(p + off[h][i]);
        if constexpr (kQ6) pre_d = ld_u16(p + doff);
    };
    auto put = [&]() {
#pragma unroll
        for (int i = 0; i < kLoads; i++) *reinterpret_cast<u32x4_t*>(slab + dst[i]) = pre[i];
        if constexpr (kQ6) *reinterpret_cast<uint16_t*>(slab + (lane & (kRows - 1)) * S::stride + 112) = pre_d;
    };

    // ---- activations: rows past the end of the tile re-read its last row ----
    uint32_t xoff[kReq];
#pragma unroll
    for (int i = 0; i < kReq; i++) {
        const int row = 8 * (wave + kWaves * i) + (lane >> 3);
        int64_t gr = row_begin + row;
        if (gr >= row_end) gr = row_end - 1;
        xoff[i] = (uint32_t)(2 * gr * a.K + 16 * ((lane & 7) ^ ((row >> 1) & 7)));
    }
    // the tiles of stage st of super-block s of every K share (a shorter last share stays inside the row)
    auto load_x = [&](int s, int st) {
#pragma unroll
        for (int k = 0; k < KW; k++) {
            int col = (sb0 + k * steps + s) * 512 + 128 * T * st;      // byte column
            if (KW > 1 && col > xlast) col = xlast;
#pragma unroll
            for (int t = 0; t < T; t++) {
                const uint8_t* xb = wave_ptr(reinterpret_cast<const uint8_t*>(a.x) + col + 128 * t);
#pragma unroll
                for (int i = 0; i < kReq; i++) {
                    if (kBlocks % kWaves != 0 && i == kReq - 1 && wave >= kBlocks - kWaves * (kReq - 1)) break;
                    const uint32_t to = lds_addr(lds) + (uint32_t)((st & 1) * kStage + (k * T + t) * kTile + (wave + kWaves * i) * 1024);
                    // (as the dense kernels' copies: M0 holds the destination, one wait state between its write and the request)
                    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(xoff[i]), "s"(xb) : "memory", "m0");
                }
            }
        }
    };
    int foff[2];
#pragma unroll
    for (int j = 0; j < 2; j++) foff[j] = r * 128 + 16 * ((4 * j + g) ^ ((r >> 1) & 7));

    f32x4_t acc[R][MT];
#pragma unroll
    for (int rg = 0; rg < R; rg++)
#pragma unroll
        for (int t = 0; t < MT; t++) acc[rg][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // ---- decode of a sub-block into operands d: per row group its scales, then two dwords of quants ----
    Sub<QT, NUM> sub[kEarly ? 2 : 1][R];
    typename Num<NUM>::T D[R], DM[R];
    auto read_part = [&](auto J, int rg) {
        constexpr int j = decltype(J)::value & 7;
        sub[kEarly ? j & 1 : 0][rg].template load<j>(slab + (16 * rg + r) * S::stride, g);
    };
    auto decode_part = [&](auto J, int c, u32x4_t (&d)[R]) {
        constexpr int j = decltype(J)::value & 7;
        typedef Sub<QT, NUM> B;
        const int rg = c / 3, part = c % 3;
        const B& b = sub[kEarly ? j & 1 : 0][rg];
        uint32_t p01, p23;
        if (part == 0) {
            b.template scales<j>(g, D[rg], DM[rg]);
        } else if (part == 1) {
            kq_dword_bf16<NUM, B::kMin, false, false>(ident, b.template quads<j, 0>(g), B::kZero, D[rg], DM[rg], p01, p23);
            d[rg][0] = p01; d[rg][1] = p23;
        } else {
            kq_dword_bf16<NUM, B::kMin, false, false>(ident, b.template quads<j, 1>(g), B::kZero, D[rg], DM[rg], p01, p23);
            d[rg][2] = p01; d[rg][3] = p23;
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
        static_for<2 * T>([&](auto U) {
            constexpr int u = decltype(U)::value, j = 2 * T * st + u;
            constexpr int jr = kEarly ? j + 2 : j + 1;       // sub-block whose bytes are read under this one
            if constexpr (jr == 4) {
                put();
                if constexpr (!last) fetch(s + 1, int_c<0>{});
            } else if constexpr (jr == 8 && !last) {
                put();
                fetch(s + 1, int_c<1>{});
            }
#pragma unroll
            for (int t = 0; t < MT; t++) {
                const int i = u * MT + t;
#pragma unroll
                for (int rg = 0; rg < R; rg++)
                    acc[rg][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, af[j & 1][rg]), xf[i % kRing], acc[rg][t], 0, 0, 0);
                if (i + kRing < n) xf[i % kRing] = frag(i + kRing);
#pragma unroll
                for (int c = 0; c < 4 * R; c++) {
                    if (c * MT / (4 * R) != t) continue;
                    if (c < R) { if constexpr (!last || jr < 8) read_part(int_c<jr>{}, c); }
                    else { if constexpr (!last || j < 7) decode_part(int_c<j + 1>{}, c - R, af[(j + 1) & 1]); }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
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
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kYoung) : "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if constexpr (!last || st + 1 < kStages) load_x(s + (st + 1) / kStages, (st + 1) % kStages);
            if constexpr (work) contract(ST, LAST, s);
        });
    };
    load_x(0, 0);
    fetch(0, int_c<0>{});
    put();
    fetch(0, int_c<1>{});
#pragma unroll
    for (int c = 0; c < R; c++) {
        read_part(int_c<0>{}, c);
        if (kEarly) read_part(int_c<1>{}, c);
    }
#pragma unroll
    for (int c = 0; c < 3 * R; c++) decode_part(int_c<0>{}, c, af[0]);
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
    auto store_gated = [&](int64_t m, int64_t n, const f32x4_t& gt, const f32x4_t& ut) {
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float gv = bf16_to_f32(f32_to_bf16(gt[e])), uv = bf16_to_f32(f32_to_bf16(ut[e]));
            o[e] = bf16_to_f32(f32_to_bf16(gv / (1.0f + expf(-gv)))) * uv;
        }
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
    // two halves of K: wavefront kw keeps row group kw (in acc[0]) and adds the other half's sums to it
    constexpr int kOwn = KW == 2 ? 1 : R;
    const int64_t nown = n0 + (KW == 2 ? 16 * kw : 0) + 4 * g;
    if constexpr (KW == 2) {
#pragma unroll
        for (int t = 0; t < MT; t++) red[(wave * MT + t) * 64 + lane] = kw == 0 ? acc[R - 1][t] : acc[0][t];
        __syncthreads();
#pragma unroll
        for (int t = 0; t < MT; t++) {
            const f32x4_t p = red[((wave ^ NW) * MT + t) * 64 + lane];
            f32x4_t m = kw == 0 ? acc[0][t] : acc[R - 1][t];
            m[0] += p[0]; m[1] += p[1]; m[2] += p[2]; m[3] += p[3];
            acc[0][t] = m;
        }
        __syncthreads();
    }
    if (a.pair && !a.partial) {
        // gate wavefronts finish the even row tiles, up wavefronts the odd ones
        constexpr int kHalf = (MT + 1) / 2;
#pragma unroll
        for (int rg = 0; rg < kOwn; rg++)
#pragma unroll
            for (int t = 0; t < MT; t++)
                if ((t & 1) != second) red[((wave * kOwn + rg) * kHalf + t / 2) * 64 + lane] = acc[rg][t];
        __syncthreads();
        const int other = wave ^ (NW / 2);
#pragma unroll
        for (int rg = 0; rg < kOwn; rg++)
#pragma unroll
            for (int t = 0; t < MT; t++) {
                if ((t & 1) != second) continue;
                const int64_t m = row_begin + 16 * t + r, n = nown + 16 * rg;
                if (m >= row_end || n >= a.N) continue;
                const f32x4_t p = red[((other * kOwn + rg) * kHalf + t / 2) * 64 + lane];
                store_gated(m, n, second ? p : acc[rg][t], second ? acc[rg][t] : p);
            }
        return;
    }
#pragma unroll
    for (int t = 0; t < MT; t++) {
        const int64_t m = row_begin + 16 * t + r;
        if (m >= row_end) continue;
#pragma unroll
        for (int rg = 0; rg < kOwn; rg++) {
            const int64_t n = nown + 16 * rg;
            if (n < a.N) store(second, m, n, acc[rg][t]);
        }
    }
}

template <int QT, int NUM, int R, int MT, int KW>
int launch(const MidArgs& a, hipStream_t stream) {
    constexpr int kLds = mid_lds_bytes<QT, R, MT, KW>();
    static_assert(kLds <= 160 * 1024, "LDS of a compute unit");
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_mid_kernel<QT, NUM, R, MT, KW>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (attr != hipSuccess) return SNGGUF_E_LAUNCH;
    gemm_mid_kernel<QT, NUM, R, MT, KW><<<dim3((unsigned)(a.col_tiles * a.row_tiles * a.ksplit)), dim3(64 * kWaves), kLds, stream>>>(a);
    return hipGetLastError() == hipSuccess ? SNGGUF_OK : SNGGUF_E_LAUNCH;
}

template <int NUM>
int launch_form(const MidArgs& a, int form, int mt, hipStream_t stream) {
    constexpr int QT = SNGGUF_MID_TYPE;
#define SNGGUF_CASE(FORM, R, MT, KW) if (form == FORM && mt == MT) return launch<QT, NUM, R, MT, KW>(a, stream)
    SNGGUF_CASE(kMidNarrow, 1, 2, 2);
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
