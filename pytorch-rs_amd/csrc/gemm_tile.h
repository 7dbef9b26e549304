// gemm_tile.h -- the tile body of the fp32 matmul: fp32 products on the bf16
// matrix cores, three bf16 pieces per value.
//
// A float's 24 significant bits are the exact sum of three bf16 values:
// h = rn(x), m = rn(x - h), l = x - h - m (bf16 has 8 significant bits and
// float's exponent range, so nothing is scaled).  Of the nine products of
// two such sums the six of weight 2^-16 and above are computed, each exact in
// the matrix cores and added in fp32.  bf16 MFMA runs 16 times the rate of
// fp32 MFMA, so six products cost 3/8 of the fp32 instruction's time.
// Rounding to nearest matters: with truncated pieces every small product has
// the sign of the whole one, and the accumulator's alignment loses them in
// one direction (K = 4096 on positive data: 9.5e-6).
//
// Two sums are kept over all of K: `acc` of the leading products h h, and
// `low` of the five small ones, added to it once at the end.  `low` is 2^-8 of
// the result and its roundings do not count; `acc` adds products of 16 bits,
// rounded once per 8 k by the matrix core and mostly exactly.  An fp32 MFMA
// rounds a nonzero product each.  Adding `low` once per slot instead gives
// back a rounding a slot, which operands with many zeros (a relu's output
// under dropout, one-hot rows) show: with a 0.02 share of nonzeros it is
// behind fp32 MFMA (1.1 times its error), and with the small products added
// straight to `acc` in half the slots, which was faster (580-630 us at 4096^3),
// from a share of 0.35 down (1.6 times at 0.02).  The price is registers: a
// 256x256 tile has room for one sum only, so it is computed as two halves of
// 256x128, each splitting A again.
//
// Error against 64 bits (2-norm over 2-norm; the fp32 MFMA tiles this replaced
// on the same inputs in brackets), [1000, K] @ [K, 1000], normal values, left
// operand with the given share of nonzeros:
//   K       1                  0.25               0.05               0.005
//     64    5.0e-8 (1.4e-7)    3.4e-8 (7.6e-8)    2.7e-8 (4.0e-8)    2.6e-8 (2.8e-8)
//    512    7.7e-8 (2.1e-7)    5.9e-8 (1.1e-7)    5.0e-8 (6.6e-8)    3.9e-8 (4.1e-8)
//   6144    1.3e-7 (3.6e-7)    1.0e-7 (1.9e-7)    8.5e-8 (1.1e-7)    7.6e-8 (8.0e-8)
// and 4096^3 4.0e-7 (1.15e-6), 2.3e-7 (5.7e-7), 9.7e-8 (2.6e-7), 3.8e-8 (8.5e-8).
// The one case behind is an output, or a K slice's part of it, that is a single
// nonzero product: the three products left out, below 2^-24 of it together,
// take a diagonal operand from 2.52e-8 to 2.59e-8 (4% of such outputs are the
// neighbour of the correctly rounded product; K = 1 goes to fp32 MFMA) and
// [64, 512] @ [512, 200] in 8 slices with a 0.02 share of nonzeros from 5.52e-8
// to 5.58e-8.
//
// An output of a tile depends on its row of A and its column of B alone,
// wherever they stand in it.  The order of the products is not symmetric in A
// and B, so A @ A.mT is symmetric to rounding only; and a tile that falls back
// to fp32 MFMA (below) rounds all its outputs as that does.
//
// Where the split does not hold -- an infinity, a NaN, a sum that overflows on
// the way, or a value whose lowest bits fall below bf16's smallest subnormal
// (|x| < 2^-110 with low bits set) and can show in an output -- the part of the
// tile is computed again on fp32 MFMA (fp32_slots).  The first three leave a
// non-finite accumulator; the split notes lost bits as it goes, and harmed()
// bounds what they can do by the rows' largest values, which survey() reads.
// Lost bits in the first slots of rows that hold nothing larger go to fp32 MFMA
// at once (useless()).  4096^3, one value of 2^-119 in every 64 rows: 905-935 us
// (950 on the fp32 MFMA build; 1,630 where every such tile was computed
// again), all values that small: 1,110-1,140 (950; 1,590), a NaN in every 64 rows,
// whose tiles are all computed twice, 1,700 (950).
//
// What bounds it: the card's power.  At 4096^3 random values run 615-700 us by
// layout and card (1,180-1,340 TFLOP/s of bf16; 580-630 with one sum in a 256x256
// tile), where the MFMAs alone would take 466.  The fp32 MFMA kernel this
// replaced took 935-970 us.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace trs {

typedef float gt_f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float gt_f2 __attribute__((ext_vector_type(2)));
typedef float gt_f16 __attribute__((ext_vector_type(16)));
typedef uint32_t gt_u4 __attribute__((ext_vector_type(4)));
typedef const float __attribute__((address_space(1))) *gt_global;
typedef const char __attribute__((address_space(1))) *gt_global_bytes;
typedef char __attribute__((address_space(3))) *gt_lds;
typedef float __attribute__((address_space(3))) *gt_lds_floats;
typedef uint32_t __attribute__((address_space(3))) *gt_lds_words;
typedef __bf16 gt_bf2 __attribute__((ext_vector_type(2)));
typedef __bf16 gt_bf8 __attribute__((ext_vector_type(8)));

struct GemmArgs {
    const float *a;
    const float *b;
    float *c;
    int64_t M, N, K;
    int64_t lda;  // stride of A's non-unit dim (rows if k-contiguous, k if not)
    int64_t ldb;  // stride of B's non-unit dim (k if plain, columns if k-contiguous)
    int64_t ldc;
    int64_t bsa, bsb, bsc;  // batch strides (elements)
    int64_t batch;
    // Split K (batches are K slices of depth K): the full depth, so the last
    // slice stops at ktotal; 0 when every batch has depth K.
    int64_t ktotal;
    int32_t tiles_m, tiles_n;
    int32_t xcd_remap;
    // Stream-K: blocks, slices per tile, (tile, slice) units, the k per
    // slice, and the workspace of two partial tiles per block.
    int64_t sk_blocks, sk_q, sk_units;
    int32_t sk_depth;
    float *sk_ws;
};

// The kernel's arguments, read where they are used: from a copy of the pointer
// to them that the compiler cannot see through, so that a loop's fields are
// loaded again on each turn and not held in scalar registers over all of it.
typedef const GemmArgs __attribute__((address_space(4))) &GemmArgsRef;
__device__ __forceinline__ GemmArgsRef kernel_args() {
    auto p = (const GemmArgs __attribute__((address_space(4))) *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *p;
}

// Floats below this (2^-110) have bits below bf16's smallest subnormal, 2^-133;
// what the split loses of one is at most half of that.
constexpr uint32_t kTiny = (127u - 110u) << 23;

constexpr int kGroupM = 8;
constexpr int kXcds = 8;
constexpr int kSlot = 16;  // k per slot: the depth of one v_mfma_f32_32x32x16_bf16

// min by value: std::min of a kernel argument and a temporary returns a
// reference the compiler may have to keep in scratch memory.
__device__ __forceinline__ int64_t imin(int64_t a, int64_t b) { return a < b ? a : b; }

// A pointer that is the same in every lane, in scalar registers.
__device__ __forceinline__ const float *gt_uniform(const float *p) {
    const uint64_t u = (uint64_t)p;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)u);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(u >> 32));
    return (const float *)((uint64_t)hi << 32 | lo);
}

struct TileCoord {
    int64_t batch, m, n;
};

// Tile t of a launch (t over batch * tiles_m * tiles_n): tiles in groups of
// kGroupM tile rows, the group's tiles taken down its columns.  In 32 bits: a
// grid has below 2^31 tiles, and the 64-bit divisions are software loops of
// some 600 instructions before a block's first load.
__device__ __forceinline__ TileCoord decode_tile(GemmArgsRef args, uint32_t t) {
    const uint32_t tm = (uint32_t)args.tiles_m, tn = (uint32_t)args.tiles_n, tiles = tm * tn;
    TileCoord c;
    const uint32_t batch = t / tiles;
    t -= batch * tiles;
    const uint32_t group_span = (uint32_t)kGroupM * tn;
    const uint32_t group = t / group_span;
    const uint32_t first_m = group * kGroupM;
    const uint32_t gm = tm - first_m < (uint32_t)kGroupM ? tm - first_m : (uint32_t)kGroupM;
    const uint32_t within = t - group * group_span;
    // The divisions run on the vector units; back to scalar registers.
    c.batch = (uint32_t)__builtin_amdgcn_readfirstlane((int)batch);
    c.m = (uint32_t)__builtin_amdgcn_readfirstlane((int)(first_m + within % gm));
    c.n = (uint32_t)__builtin_amdgcn_readfirstlane((int)(within / gm));
    return c;
}

// Two floats as bf16 pairs h + m + l.  `lost` collects the bits of the last
// remainders: their low halves are zero exactly where l holds them whole.
__device__ __forceinline__ void split_pair(float a, float b, uint32_t &h, uint32_t &m, uint32_t &l, uint32_t &lost) {
    const auto pack = [](float x, float y) {
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((gt_f2){x, y}, gt_bf2));
    };
    const auto lo = [](uint32_t p) { return __uint_as_float(p << 16); };
    const auto hi = [](uint32_t p) { return __uint_as_float(p & 0xffff0000u); };
    h = pack(a, b);
    a -= lo(h);
    b -= hi(h);
    m = pack(a, b);
    a -= lo(m);
    b -= hi(m);
    l = pack(a, b);
    lost |= __float_as_uint(a) | __float_as_uint(b);
}

// One operand's share of a slot: ROWS rows (of M or N) by 16 k, dealt to the
// block's lanes in chunks of CH (8 or 4) consecutive k of one row.
//   KC (k contiguous in memory): a chunk is one or two 16-byte loads; they
//     need only dword alignment, so any row length will do.
//   otherwise (rows contiguous): a chunk is CH loads of one float, each a
//     whole 256 bytes across the wave (a wave's chunks are 64 rows of the
//     same k).
// Either way the lane holds consecutive k of one row, as an MFMA fragment
// takes them (8 a lane), so the pieces are packed in registers and stored as
// 8 or 16 bytes: no transpose, no alignment cases.  In LDS a plane (h, m or
// l) is kept in fragment order: 32 rows by 16 k are one KiB, (row, k) at
// 512*(k/8) + 16*row + 2*(k%8), which fragment reads walk in lane order, free
// of bank conflicts.
// Rows past the matrix's edge read its last row (never stored).
template <int ROWS, int NT, bool KC>
struct SlotOperand {
    static constexpr int CH = ROWS * 2 >= NT ? 8 : 4;
    static constexpr int NC = ROWS * kSlot / CH / NT;  // chunks per lane
    static_assert(NC >= 1 && NC * NT * CH == ROWS * kSlot && ROWS % 64 == 0, "whole chunks for every lane");
    static constexpr int kPlane = ROWS * 2 * kSlot;  // bytes
    static constexpr int kPitch = ROWS + 32;         // floats per k of the fp32 layout
    typedef float Regs[NC][CH];
    const float *ptr[NC];  // KC: the lane's chunk in the next slot to load; else the operand's first row of it
    uint32_t voff[NC];     // not KC: the lane's row, in bytes
    int row[NC], k[NC];    // the chunk's row and first k

    // base: element (row 0 of the tile, k 0); rows: rows of the matrix from the tile's first on.
    __device__ __forceinline__ void plan(const float *base, int64_t rows, int64_t ld, unsigned tid) {
#pragma unroll
        for (int q = 0; q < NC; q++) {
            const int c = (int)(tid + q * NT), l = c & 63;
            if constexpr (KC) {
                row[q] = c / (32 * kSlot / CH) * 32 + (l & 31);
                k[q] = ((c >> 6) * 2 + (l >> 5)) % (kSlot / CH) * CH;
            } else {
                row[q] = c % ROWS;
                k[q] = __builtin_amdgcn_readfirstlane(c / ROWS * CH);
            }
            const int64_t r = row[q] < rows ? row[q] : rows - 1;
            if constexpr (KC) {
                ptr[q] = base + r * ld + k[q];
            } else {
                ptr[q] = gt_uniform(base + k[q] * ld);
                voff[q] = (uint32_t)(r * 4);
            }
        }
    }
    __device__ __forceinline__ void advance(int64_t step) {
#pragma unroll
        for (int q = 0; q < NC; q++) ptr[q] += step;
    }
    // Rows contiguous: one scalar base per k and one 32-bit lane offset.  Both
    // go through an asm that the compiler cannot see past, since it otherwise
    // folds the two into a 64-bit lane address per k (16 registers, and
    // spills).
    __device__ __forceinline__ static gt_global column(gt_global &p, uint32_t off, int64_t ld) {
        asm("" : "+s"(p));
        const gt_global at = (gt_global)((gt_global_bytes)p + off);
        p += ld;
        return at;
    }
    __device__ __forceinline__ void load(Regs &v, int64_t ld) const {
#pragma unroll
        for (int q = 0; q < NC; q++) {
            if constexpr (KC) {
#pragma unroll
                for (int e = 0; e < CH; e += 4) {
                    const gt_f4u x = *(const gt_f4u *)(ptr[q] + e);
#pragma unroll
                    for (int i = 0; i < 4; i++) v[q][e + i] = x[i];
                }
            } else {
                gt_global p = (gt_global)ptr[q];
                uint32_t off = voff[q];
                asm("" : "+v"(off));
#pragma unroll
                for (int e = 0; e < CH; e++) v[q][e] = *column(p, off, ld);
            }
        }
    }
    // The first `tail` k of a slot, zero past them (no load is made there).
    __device__ __forceinline__ void load_tail(Regs &v, int64_t ld, int tail) const {
#pragma unroll
        for (int q = 0; q < NC; q++) {
            gt_global p = (gt_global)ptr[q];
#pragma unroll
            for (int e = 0; e < CH; e++) {
                v[q][e] = 0.f;
                if constexpr (KC) {
                    if (k[q] + e < tail) v[q][e] = p[e];
                } else {
                    const gt_global at = column(p, voff[q], ld);
                    if (k[q] + e < tail) v[q][e] = *at;
                }
            }
        }
    }
    __device__ __forceinline__ void store_split(const Regs &v, gt_lds lds, uint32_t &lost) const {
        typedef uint32_t Pack __attribute__((ext_vector_type(CH / 2)));
        typedef Pack __attribute__((address_space(3))) *PackLds;
#pragma unroll
        for (int q = 0; q < NC; q++) {
            Pack h, m, l;
#pragma unroll
            for (int e = 0; e < CH / 2; e++) {
                uint32_t x, y, z;
                split_pair(v[q][2 * e], v[q][2 * e + 1], x, y, z, lost);
                h[e] = x, m[e] = y, l[e] = z;
            }
            const gt_lds d = lds + (row[q] >> 5) * 1024 + (k[q] >> 3) * 512 + (row[q] & 31) * 16 + (k[q] & 7) * 2;
            *(PackLds)d = h;
            *(PackLds)(d + kPlane) = m;
            *(PackLds)(d + 2 * kPlane) = l;
        }
    }
    // For each chunk, as floats: the largest |value| so far, and 1 if a value was
    // one whose split may lose bits.
    __device__ __forceinline__ void note(const Regs &v, uint32_t (&most)[NC], uint32_t (&tiny)[NC]) const {
#pragma unroll
        for (int q = 0; q < NC; q++)
#pragma unroll
            for (int e = 0; e < CH; e++) {
                const uint32_t u = __float_as_uint(v[q][e]) & 0x7fffffffu;
                most[q] = most[q] > u ? most[q] : u;
                if (u - 1 < kTiny - 1) tiny[q] = 0x3f800000u;
            }
    }
    // As floats, [k][row]: the pitch puts k and k + 1 half the banks apart.
    __device__ __forceinline__ void store_fp32(const Regs &v, gt_lds_floats lds) const {
#pragma unroll
        for (int q = 0; q < NC; q++)
#pragma unroll
            for (int e = 0; e < CH; e++) lds[(k[q] + e) * kPitch + row[q]] = v[q][e];
    }
};

// A BM x BN tile of C on WGM x WGN waves, each (BM/WGM) x (BN/WGN) as 32x32
// MFMA tiles, and PARTS of them side by side, one after the other.  AHEAD slots
// are on their way from memory in registers (the depth is not what bounds it:
// 4096^3 by layout 667, 673 and 632 us with 1, 679, 660 and 663 with 2).  AKC,
// BKC: the operand is contiguous along k.
template <int BM, int BN, int WGM, int WGN, int AHEAD, bool AKC, bool BKC, int PARTS = 1>
struct GemmTile {
    static constexpr int NT = WGM * WGN * 64, WM = BM / WGM, WN = BN / WGN, TM = WM / 32, TN = WN / 32;
    using OA = SlotOperand<BM, NT, AKC>;
    using OB = SlotOperand<BN, NT, BKC>;
    static constexpr int kABytes = 3 * OA::kPlane, kBuf = kABytes + 3 * OB::kPlane;
    // Three slots in LDS, a word a wave for each of three notices, and survey()'s values.
    enum Notice { kFirstLost, kResult, kFails };
    static constexpr int NW = WGM * WGN, kNotices = 3 * kBuf;
    static constexpr int kSurvey = kNotices + 3 * NW * 4, kLds = kSurvey + 2 * (BM + BN) * 4;
    static constexpr int kFp32A = kSlot * OA::kPitch, kFp32Buf = kFp32A + kSlot * OB::kPitch;
    static_assert(2 * kFp32Buf * 4 <= 3 * kBuf, "the fp32 slots fit the split ones' LDS");
    static_assert(AHEAD == 1 || AHEAD == 2, "the slot loop is unrolled over two register sets");

    // The products of the leading pieces, and all the others'.
    gt_f16 acc[TM][TN], low[TM][TN];
    OA oa;
    OB ob;
    gt_lds lds;
    int64_t lda, ldb;
    int64_t astep, bstep;
    int lane, wave, wm0, wn0;

    __device__ __forceinline__ explicit GemmTile(gt_lds l) : lds(l) {}

    // What the waves of a block tell one another: each posts a word (the same in
    // all its lanes) ahead of a barrier, and reads the or of them behind it.  All
    // post every time, so nothing has to be cleared.
    __device__ __forceinline__ void post(Notice n, uint32_t word) const {
        ((gt_lds_words)(lds + kNotices))[n * NW + wave] = word;
    }
    __device__ __forceinline__ uint32_t posted(Notice n) const {
        uint32_t any = 0;
#pragma unroll
        for (int w = 0; w < NW; w++) any |= ((gt_lds_words)(lds + kNotices))[n * NW + w];
        return __builtin_amdgcn_readfirstlane(any);
    }
    // Whether a condition holds in a lane of this wave.
    __device__ __forceinline__ static bool in_wave(bool lane) { return __builtin_amdgcn_ballot_w64(lane) != 0; }

    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                acc[i][j] = low[i][j] = (gt_f16)(0.f);
                // Here, and not where they are first used.
                asm volatile("" : "+v"(acc[i][j]), "+v"(low[i][j]));
            }
    }
    struct Slot {  // a slot's floats on their way to LDS
        typename OA::Regs a;
        typename OB::Regs b;
    };
    __device__ __forceinline__ void load(Slot &r) const {
        oa.load(r.a, lda);
        ob.load(r.b, ldb);
    }

    // `whole` slots from the operands' current pointers on, after the `tail`
    // k (0: none) behind the last of them.  The partial slot goes first: its
    // checked loads then fall in the prologue, whose latency is exposed
    // anyway, and not behind the last whole slot.
    //
    // Slot t is computed from one of three LDS buffers while slot t + 2 is split from
    // registers into another and slot t + 2 + AHEAD is loaded into those
    // registers.  Slot t + 1's buffer was complete at the barrier before, so the
    // fragments a slot starts with are read before the barrier that ends the
    // slot ahead of it.  A wave walks its rows of MFMA tiles; the reads for
    // the next row, and the slot's splitting and loads, sit among the MFMAs
    // of the row before.  Loads past the last slot repeat it (a branch around
    // a load makes the compiler wait for every load at the join).
    __device__ __forceinline__ bool split_slots(int whole, int tail, unsigned tid, uint32_t &lost) {
        lost = 0;
        Slot in[AHEAD];
        const int T = whole + (tail ? 1 : 0);
        int left = whole;  // whole slots not yet loaded
        const auto move_on = [&]() {  // staying on the last slot
            left--;
            oa.advance(left > 0 ? astep : 0);
            ob.advance(left > 0 ? bstep : 0);
        };
        const auto put = [&](const Slot &r, int buf) {
            oa.store_split(r.a, lds + buf, lost);
            ob.store_split(r.b, lds + buf + kABytes, lost);
        };
        typedef const gt_bf8 __attribute__((address_space(3))) *Frag;
        const gt_lds fa = lds + wm0 * 32 + lane * 16, fb = lds + kABytes + wn0 * 32 + lane * 16;
        // The products (piece of A, piece of B): five for `low`, the sixth for `acc`.
        static constexpr int PA[6] = {2, 1, 1, 0, 0, 0}, PB[6] = {0, 0, 1, 1, 2, 0};
        int cur = 0, nxt = kBuf, wr = 2 * kBuf;  // this slot's buffer, the next one's, the one being written
        gt_bf8 A[2][3], B[TN][3];
        const auto read_a = [&](int buf, int i, gt_bf8 (&d)[3]) {
#pragma unroll
            for (int p = 0; p < 3; p++) d[p] = *(Frag)(fa + buf + p * OA::kPlane + i * 1024);
        };
        const auto read_b = [&](int buf, int j) {
#pragma unroll
            for (int p = 0; p < 3; p++) B[j][p] = *(Frag)(fb + buf + p * OB::kPlane + j * 1024);
        };
        // LEFT: the slots that follow this one, 2 for two or more.  D: the registers
        // holding slot t + 2.
        const auto slot = [&]<int LEFT, int D>() {
#pragma unroll
            for (int i = 0; i < TM; i++) {
                if (i + 1 < TM) read_a(cur, i + 1, A[(i + 1) & 1]);
                else if (LEFT > 0) read_a(nxt, 0, A[TM & 1]);
#pragma unroll
                for (int p = 0; p < 6; p++)
#pragma unroll
                    for (int j = 0; j < TN; j++) {
                        gt_f16 &d = p < 5 ? low[i][j] : acc[i][j];
                        d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[i & 1][PA[p]], B[j][PB[p]], d, 0, 0, 0);
                    }
                if constexpr (LEFT > 0) {
                    if (i == TM - 1) {
#pragma unroll
                        for (int j = 0; j < TN; j++) read_b(nxt, j);
                    }
                }
                if constexpr (LEFT > 1) {
                    if (i == 0) oa.store_split(in[D].a, lds + wr, lost);
                    if (i == (TM > 1 ? 1 : 0)) {
                        oa.load(in[D].a, lda);
                        ob.store_split(in[D].b, lds + wr + kABytes, lost);
                    }
                    if (i == (TM > 2 ? 2 : TM - 1)) {
                        ob.load(in[D].b, ldb);
                        move_on();
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (LEFT > 0 && TM % 2 == 1) {
#pragma unroll
                for (int p = 0; p < 3; p++) A[0][p] = A[1][p];
            }
            if constexpr (LEFT > 1) __syncthreads();
            const int c = cur;
            cur = nxt, nxt = wr, wr = c;
        };
        // The first slots are in LDS: the first fragments, and whether to give up.
        const auto first = [&](int slots, const Slot &s0, const Slot &s1) {
            post(kFirstLost, in_wave((lost & 0xffffu) != 0));
            __syncthreads();
            read_a(0, 0, A[0]);
#pragma unroll
            for (int j = 0; j < TN; j++) read_b(0, j);
            const uint32_t any = posted(kFirstLost);
            // All of these reads are out before the branch.
#pragma unroll
            for (int p = 0; p < 3; p++) {
                asm volatile("" : "+v"(A[0][p]));
#pragma unroll
                for (int j = 0; j < TN; j++) asm volatile("" : "+v"(B[j][p]));
            }
            if (__builtin_expect(!any, 1)) return false;
            Extremes x = {};
            note(s0, x);
            if (slots > 1) note(s1, x);
            merge(x, tid);
            return useless(tid);
        };
        // The first slots' loads all go out together.
        Slot s0, s1;
        if (tail) {
            // The partial slot lies `whole` slots on.
            OA ta = oa;
            OB tb = ob;
            ta.advance(whole * astep);
            tb.advance(whole * bstep);
            ta.load_tail(s0.a, lda, tail);
            tb.load_tail(s0.b, ldb, tail);
            if (!whole) {
                clear();
                put(s0, 0);
                if (__builtin_expect(first(1, s0, s0), 0)) return true;
                slot.template operator()<0, 0>();
                return false;
            }
        } else {
            load(s0);
            move_on();
        }
        load(s1);
        move_on();
#pragma unroll
        for (int d = 0; d < AHEAD; d++) {
            load(in[d]);
            move_on();
        }
        clear();  // under the loads
        put(s0, 0);
        put(s1, kBuf);
        if (__builtin_expect(first(2, s0, s1), 0)) return true;
        // Slot t takes registers t % AHEAD.  The last two slots of a short K split
        // and load nothing: a load past the end is waited for, a memory latency for
        // every tile (64^3 6.3 us with it, 5.6 without; batched 32 x 256x32x256 6.6
        // and 5.7).  The large tile, whose K is long or whose store is, does not
        // tell them apart: its loop comes out 5% slower with them (4096^3 645 us,
        // 683).
        constexpr int kEnd = PARTS == 1 ? 2 : 0;
        int t = 0;
#pragma unroll 1
        for (; t + 2 + kEnd <= T; t += 2) {
            slot.template operator()<2, 0>();
            slot.template operator()<2, 1 % AHEAD>();
        }
        if (t + 1 + kEnd == T) slot.template operator()<2, 0>();
        if constexpr (kEnd) {
            if (T > 1) slot.template operator()<1, 0>();
            slot.template operator()<0, 0>();
        }
        return false;
    }

    // What lost bits can do: every row of A's and column of B's largest |value|
    // and whether (1 or 0) it holds a tiny one, per lane and then into LDS.
    struct Extremes {
        uint32_t most_a[OA::NC], tiny_a[OA::NC], most_b[OB::NC], tiny_b[OB::NC];
    };
    __device__ __forceinline__ void note(const Slot &s, Extremes &x) const {
        oa.note(s.a, x.most_a, x.tiny_a);
        ob.note(s.b, x.most_b, x.tiny_b);
    }
    __device__ __forceinline__ void merge(const Extremes &x, unsigned tid) const {
        const gt_lds_words most = (gt_lds_words)(lds + kSurvey), tiny = most + BM + BN;
        for (int i = tid; i < 2 * (BM + BN); i += NT) most[i] = 0;
        __syncthreads();
        const auto raise = [](gt_lds_words p, uint32_t v) {
            __hip_atomic_fetch_max(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        };
#pragma unroll
        for (int q = 0; q < OA::NC; q++) raise(most + oa.row[q], x.most_a[q]), raise(tiny + oa.row[q], x.tiny_a[q]);
#pragma unroll
        for (int q = 0; q < OB::NC; q++)
            raise(most + BM + ob.row[q], x.most_b[q]), raise(tiny + BM + ob.row[q], x.tiny_b[q]);
        __syncthreads();
    }
    // Of all slots, four on their way at a time.
    __device__ __forceinline__ void survey(int whole, int tail, unsigned tid) {
        Extremes x = {};
        Slot in[4];
        const auto move_on = [&]() {
            oa.advance(astep);
            ob.advance(bstep);
        };
        int t = 0;
#pragma unroll 1
        for (; t + 4 <= whole; t += 4) {
#pragma unroll
            for (int d = 0; d < 4; d++) load(in[d]), move_on();
#pragma unroll
            for (int d = 0; d < 4; d++) note(in[d], x);
        }
#pragma unroll 1
        for (; t < whole; t++) load(in[0]), move_on(), note(in[0], x);
        if (tail) {
            oa.load_tail(in[0].a, lda, tail);
            ob.load_tail(in[0].b, ldb, tail);
            note(in[0], x);
        }
        merge(x, tid);
    }
    // After survey(): whether lost bits may show in one of this lane's outputs.
    // The split is off by at most 2^-134 in a tiny value, so an output by that
    // times the other operand's values.  Up to 2^-32 of the output it is 2^-8
    // of a rounding.
    static constexpr float kLeast = 0x1p-102f;
    __device__ __forceinline__ bool harmed(int whole, int tail) const {
        const gt_lds_floats most = (gt_lds_floats)(lds + kSurvey), tiny = most + BM + BN;
        const float scale = (float)(whole * kSlot + tail) * kLeast;
        float worst = 0.f;
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int col = BM + wn0 + j * 32 + (lane & 31);
            const float mb = scale * most[col], tb = scale * tiny[col];
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int row = wm0 + i * 32 + 8 * (r / 4) + 4 * (lane >> 5) + r % 4;
                    worst = __builtin_fminf(worst, __builtin_fabsf(acc[i][j][r]) - (tiny[row] * mb + most[row] * tb));
                }
        }
        return worst < 0.f;
    }
    // After merge() of the first slots: whether none of a row's (column's) outputs
    // is likely to pass that, its values so far being too small.
    __device__ __forceinline__ bool useless(unsigned tid) const {
        const gt_lds_floats most = (gt_lds_floats)(lds + kSurvey), tiny = most + BM + BN;
        bool none = false;
        for (int i = tid; i < BM + BN; i += NT) none |= tiny[i] != 0.f && most[i] < kLeast;
        post(kFails, in_wave(none));
        __syncthreads();
        return posted(kFails);
    }

    // The same slots on fp32 MFMA (v_mfma_f32_32x32x2_f32), double-buffered.
    __device__ __forceinline__ void fp32_slots(int whole, int tail) {
        Slot in;
        const gt_lds_floats f = (gt_lds_floats)lds;
        const int T = whole + (tail ? 1 : 0);
        const auto fetch = [&](int t) {
            if (t < whole) load(in);
            else oa.load_tail(in.a, lda, tail), ob.load_tail(in.b, ldb, tail);
            oa.advance(astep);
            ob.advance(bstep);
        };
        fetch(0);
        for (int t = 0; t < T; t++) {
            const gt_lds_floats buf = f + (t & 1) * kFp32Buf;
            oa.store_fp32(in.a, buf);
            ob.store_fp32(in.b, buf + kFp32A);
            if (t + 1 < T) fetch(t + 1);
            __syncthreads();
            const gt_lds_floats pa = buf + (lane >> 5) * OA::kPitch + wm0 + (lane & 31);
            const gt_lds_floats pb = buf + kFp32A + (lane >> 5) * OB::kPitch + wn0 + (lane & 31);
#pragma unroll 2
            for (int k = 0; k < kSlot; k += 2) {
                float x[TM], y[TN];
#pragma unroll
                for (int i = 0; i < TM; i++) x[i] = pa[k * OA::kPitch + i * 32];
#pragma unroll
                for (int j = 0; j < TN; j++) y[j] = pb[k * OB::kPitch + j * 32];
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[i], y[j], acc[i][j], 0, 0, 0);
            }
        }
        __syncthreads();
    }

    // The block's tile over its k in [k0, k1) (k1 past the last k: to the end;
    // k0 a multiple of 16): PARTS times BN columns, one after the other.
    // Stores it into C, or with `ws` set into ws[row * PARTS * BN + column].
    __device__ __forceinline__ void run(GemmArgsRef args, TileCoord tc, int64_t k0, int64_t k1, float *ws) {
        if constexpr (PARTS == 1) {
            run_part(args, tc.batch, tc.m * BM, tc.n * BN, k0, k1, ws, threadIdx.x);
        } else {
#pragma unroll 1
            for (int part = 0; part < PARTS; part++) {
                GemmArgsRef again = kernel_args();
                const int64_t n0 = (tc.n * PARTS + part) * BN;
                if (part && n0 >= again.N) break;
                // Nor is what a lane derives from its number kept over the parts.
                unsigned tid = threadIdx.x;
                asm volatile("" : "+v"(tid));
                run_part(again, tc.batch, tc.m * BM, n0, k0, k1, ws ? ws + part * BN : nullptr, tid);
            }
        }
    }

    __device__ __forceinline__ void run_part(GemmArgsRef args, int64_t batch, int64_t m0, int64_t n0, int64_t k0,
                                             int64_t k1, float *ws, unsigned tid) {
        lda = args.lda, ldb = args.ldb;
        lane = tid & 63;
        wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        wm0 = (wave / WGN) * WM;
        wn0 = (wave % WGN) * WN;
        const int64_t Kb = args.ktotal ? imin(args.K, args.ktotal - batch * args.K) : args.K;
        astep = AKC ? kSlot : kSlot * lda;
        bstep = BKC ? kSlot : kSlot * ldb;
        const int64_t kspan = imin(k1, Kb) - k0;
        // 64-bit compares run on the vector units; back to scalar registers.
        const int whole = __builtin_amdgcn_readfirstlane((int)(kspan >> 4));
        const int tail = __builtin_amdgcn_readfirstlane((int)(kspan & (kSlot - 1)));
        const auto to_first = [&](GemmArgsRef g) {
            const float *A = g.a + batch * g.bsa + (AKC ? m0 * lda + k0 : m0 + k0 * lda);
            const float *B = g.b + batch * g.bsb + (BKC ? n0 * ldb + k0 : n0 + k0 * ldb);
            oa.plan(A, g.M - m0, lda, tid);
            ob.plan(B, g.N - n0, ldb, tid);
        };
        to_first(args);
        // One k is one product per output, which the split does not always
        // round correctly (its time is that of the output's store either way).
        bool fp32 = kspan == 1;
        if (__builtin_expect(!fp32, 1)) {
            uint32_t lost;
            fp32 = split_slots(whole, tail, tid, lost);
            // What follows works its lane values out again, so that the slot loop
            // does not keep them live (nor the lane's number itself).
            lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
            asm volatile("" : "+v"(lane));
            tid = (unsigned)(wave * 64 + lane);
            if (__builtin_expect(!fp32, 1)) {
                // A non-finite accumulator leaves a non-finite sum of them.
                float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
#pragma unroll
                        for (int r = 0; r < 16; r++) {
                            acc[i][j][r] += low[i][j][r];
                            sum[r & 3] += acc[i][j][r];
                        }
                const float s = (sum[0] + sum[1]) + (sum[2] + sum[3]);
                const bool bad = !(__builtin_fabsf(s) < __builtin_inff());
                post(kResult, in_wave((lost & 0xffffu) != 0) | in_wave(bad) << 1);
                __syncthreads();
                const uint32_t result = posted(kResult);
                fp32 = result & 2;
                if (__builtin_expect(result == 1, 0)) {
                    to_first(kernel_args());
                    int slots = whole, rest = tail;  // nothing of this ahead of the slot loop
                    asm volatile("" : "+s"(slots), "+s"(rest));
                    survey(slots, rest, tid);
                    post(kFails, in_wave(harmed(slots, rest)));
                    __syncthreads();
                    fp32 = posted(kFails);
                }
            }
            if (__builtin_expect(fp32, 0)) to_first(kernel_args());
        }
        if (__builtin_expect(fp32, 0)) {
            clear();
            fp32_slots(whole, tail);
        }
        GemmArgsRef out = PARTS == 1 ? args : kernel_args();
        // Lane l, register r of a 32x32 tile: row 8*(r/4) + 4*(l/32) + r%4, column l%32.
        const int rl = 4 * (lane >> 5), cl = lane & 31;
        if (ws) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int r = 0; r < 16; r++)
                        ws[(wm0 + i * 32 + 8 * (r / 4) + rl + r % 4) * (PARTS * BN) + wn0 + j * 32 + cl] = acc[i][j][r];
            return;
        }
        float *C = out.c + batch * out.bsc;
        const int64_t mrow = m0 + wm0 + rl, ncol = n0 + wn0 + cl;
        float *cp = C + mrow * out.ldc + ncol;
        if (m0 + BM <= out.M && n0 + BN <= out.N) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    float *p = cp + (int64_t)(i * 32 + 8 * (r / 4) + r % 4) * out.ldc;
#pragma unroll
                    for (int j = 0; j < TN; j++) p[j * 32] = acc[i][j][r];
                }
            return;
        }
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int row = i * 32 + 8 * (r / 4) + r % 4;
                if (mrow + row >= out.M) continue;
                float *p = cp + (int64_t)row * out.ldc;
#pragma unroll
                for (int j = 0; j < TN; j++)
                    if (ncol + j * 32 < out.N) p[j * 32] = acc[i][j][r];
            }
    }
};

}  // namespace trs
