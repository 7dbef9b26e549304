// gemm.hip -- fp32 matmul.
//
// Replaces Tensor::matmul's three CPU paths (src/tensor.rs:2453-2533,
// 3872-3994).  The reference computes each C[i,j] as a sequential sum
// (+0.0, then k ascending, mul and add rounded separately); this kernel keeps
// fp32 inputs and fp32 accumulation ("highest" precision,
// python/torch_rs/__init__.py:81-85) but sums in MFMA order, so it is checked
// against the reference within |dC| <= 1e-5*sqrt(K)*(|A||B|).  The products
// run on the bf16 matrix cores, each float as three bf16 pieces (gemm_tile.h
// has the error, which is that of fp32 MFMA or less).
//
// Three tiles (GemmTile), each in the four operand layouts and at any M, N
// and K (rows past the edge repeat the last one and are not stored):
//   256x256  two 256x128 halves one after the other, 8 waves of 64x64, one
//            block per CU (111 KB of LDS)
//   128x128  4 waves of 64x64, two blocks per CU, or where blocks do not fill
//            the CUs twice 8 of 32x64, one per CU
//   64x128   4 waves of 32x64, two blocks per CU
// The 4-wave 128x128 tile reads a third less from LDS per product, which
// counts where the whole chip runs it and power sets the clock (batched
// 32x512^3 53.9 us against 58.3, 1000x2047x1500 48.7 against 58.0, on one
// card); the 8-wave one issues its slot in half the instructions per wave, which
// counts where one block has a CU to itself (700^3 16.8 us against 19.1,
// 2048x100x2048 11.8 against 12.2).
// Blocks are remapped so that consecutive tiles share an XCD (each XCD has
// its own L2), and tiles are walked in groups of kGroupM tile rows.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "gemm_skinny.h"
#include "gemm_tile.h"
#include "trs_internal.h"

namespace trs {

namespace {

template <bool AKC, bool BKC>
using LargeTile = GemmTile<256, 128, 4, 2, 1, AKC, BKC, 2>;
template <bool AKC, bool BKC>
using SmallTile = GemmTile<128, 128, 2, 2, 1, AKC, BKC>;
template <bool AKC, bool BKC>
using SmallTile8 = GemmTile<128, 128, 4, 2, 1, AKC, BKC>;
template <bool AKC, bool BKC>
using MediumTile = GemmTile<64, 128, 2, 2, 2, AKC, BKC>;
constexpr int64_t kLarge = 256;
constexpr int64_t kLargeTileFloats = kLarge * kLarge;

// The k that stream-K's units hold: two slots where A is contiguous along k and
// a long K is whole pairs of slots, else one.  The tile takes either alike
// (512x4096x4096, 3072^3 and 5120^3 within 0.3%); the plan reports it.
inline int slice_depth(const GemmArgs &g, bool a_plain) {
    return (a_plain && g.K % (2 * kSlot) == 0 && g.K >= 2048) ? 2 * kSlot : kSlot;
}

// One block per tile.
template <class T, int MINB>
__global__ void __launch_bounds__(T::NT, MINB) gemm_split_tile(GemmArgs) {
    GemmArgsRef args = kernel_args();
    __shared__ __attribute__((aligned(1024))) char lds[T::kLds];
    uint32_t bid = blockIdx.x;
    if (args.xcd_remap) {
        const uint32_t per_xcd = gridDim.x / kXcds;
        bid = (bid % kXcds) * per_xcd + bid / kXcds;
    }
    T tile((gt_lds)lds);
    tile.run(args, decode_tile(args, bid), 0, INT64_MAX, nullptr);
}

// Stream-K: one persistent block per CU, block b taking the (tile, slice)
// units [b*U/G, (b+1)*U/G) of the U = tiles * Q of the product (G blocks, Q
// slices per tile, tile-major).  A tile whose units fall to one block is
// stored into C; a block's first and last segments that cover only part of
// a tile's slices go to its two workspace slots (slot 0 the first segment,
// slot 1 the last), which gemm_streamk_fixup adds in k order.  No block waits
// for another.  Logical block b runs as blockIdx (b % (G/8)) * 8 + b / (G/8),
// so each XCD takes one contiguous eighth of the units.
template <class T>
__global__ void __launch_bounds__(T::NT, 1) gemm_split_tile_sk(GemmArgs) {
    GemmArgsRef first = kernel_args();
    __shared__ __attribute__((aligned(1024))) char lds[T::kLds];
    const int64_t G = first.sk_blocks, U = first.sk_units, Q = first.sk_q;
    const int64_t b = first.xcd_remap ? (blockIdx.x % kXcds) * (G / kXcds) + blockIdx.x / kXcds : blockIdx.x;
    const int64_t u0 = b * U / G, u1 = (b + 1) * U / G;
    // Segment: slices [qb, qe) of tile t; the next starts the next tile.
    int64_t t = u0 / Q, qb = u0 - t * Q;
    T tile((gt_lds)lds);
    for (int64_t u = u0; u < u1; t++, qb = 0) {
        GemmArgsRef args = kernel_args();
        const int64_t qe = imin(Q, qb + (u1 - u));
        float *ws = (qb == 0 && qe == Q) ? nullptr : args.sk_ws + (2 * b + (u == u0 ? 0 : 1)) * kLargeTileFloats;
        tile.run(args, decode_tile(args, (uint32_t)t), qb * args.sk_depth, qe * args.sk_depth, ws);
        u += qe - qb;
    }
}

// The pieces of the tiles stream-K split between blocks, added in k order
// (block order) into C.  Block (t, y) takes rows 16y..16y+15 of tile t; a
// tile that one block ran whole was stored by it and is skipped.
__global__ void __launch_bounds__(256) gemm_streamk_fixup(GemmArgs) {
    GemmArgsRef args = kernel_args();
    const int64_t G = args.sk_blocks, U = args.sk_units, Q = args.sk_q;
    const int64_t t = blockIdx.x;
    // The block whose units hold unit u: the largest b with b*U/G <= u.
    const auto block_of = [&](int64_t u) { return imin(G - 1, ((u + 1) * G - 1) / U); };
    const int64_t bf = block_of(t * Q), bl = block_of((t + 1) * Q - 1);
    if (bf == bl) return;
    const TileCoord tc = decode_tile(args, (uint32_t)t);
    float *Cp = args.c + tc.batch * args.bsc;
    const int r = (int)blockIdx.y * 16 + (int)(threadIdx.x >> 4);
    const int64_t m = tc.m * kLarge + r;
    if (m >= args.M) return;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int c = 4 * ((int)(threadIdx.x & 15) + 16 * i);
        float4 v = {0.f, 0.f, 0.f, 0.f};
        for (int64_t p = bf; p <= bl; p++) {
            // Slot 0 when the tile holds block p's first unit, else slot 1.
            const int64_t slot = p * U / G >= t * Q ? 0 : 1;
            const float4 x = *(const float4 *)(args.sk_ws + (2 * p + slot) * kLargeTileFloats + r * kLarge + c);
            if (p == bf) v = x;
            else v.x += x.x, v.y += x.y, v.z += x.z, v.w += x.w;
        }
        const int64_t n = tc.n * kLarge + c;
        float *o = Cp + m * args.ldc + n;
        if (n < args.N) o[0] = v.x;
        if (n + 1 < args.N) o[1] = v.y;
        if (n + 2 < args.N) o[2] = v.z;
        if (n + 3 < args.N) o[3] = v.w;
    }
}

// Split-K epilogue: c = ((p0 + p1) + p2) + ... over the S partial products,
// in slice order, four floats per lane.  NS is S when 2 <= S <= 16 (all S
// loads issued before the first add: one memory latency instead of one per
// slice, with no branch between the loads, where a copy at a branch join
// waits for every load issued before it), else 0 and S is read at run time.
template <int NS>
__global__ void __launch_bounds__(kHelperLanes) splitk_sum(const float4 *__restrict__ parts, float4 *__restrict__ c,
                                                  int64_t n4, int S) {
    const int64_t i = (int64_t)blockIdx.x * kHelperLanes + threadIdx.x;
    if (i >= n4) return;
    auto add = [](float4 &acc, const float4 &v) {
        acc.x += v.x;
        acc.y += v.y;
        acc.z += v.z;
        acc.w += v.w;
    };
    float4 acc;
    if constexpr (NS > 0) {
        float4 part[NS];
        const float4 *pq = parts + i;
#pragma unroll
        for (int q = 0; q < NS; q++) {
            part[q] = *pq;
            if (q + 1 < NS) pq += n4;
        }
        acc = part[0];
#pragma unroll
        for (int q = 1; q < NS; q++) add(acc, part[q]);
    } else {
        acc = parts[i];
        for (int q = 1; q < S; q++) add(acc, parts[(int64_t)q * n4 + i]);
    }
    c[i] = acc;
}

template <int NS = 2>
void launch_splitk_sum(int S, dim3 grid, hipStream_t s, const float4 *parts, float4 *c, int64_t n4) {
    if constexpr (NS > 16) hipLaunchKernelGGL(splitk_sum<0>, grid, dim3(kHelperLanes), 0, s, parts, c, n4, S);
    else if (S == NS) hipLaunchKernelGGL(splitk_sum<NS>, grid, dim3(kHelperLanes), 0, s, parts, c, n4, S);
    else launch_splitk_sum<NS + 1>(S, grid, s, parts, c, n4);
}

// Simple fallback for operands with no unit stride: one thread per output,
// sequential k (the reference's own order).
__global__ void __launch_bounds__(kHelperLanes) gemm_f32_strided(const float *a, const float *b, float *c, int64_t M,
                                                        int64_t N, int64_t K, int64_t sam, int64_t sak,
                                                        int64_t sbk, int64_t sbn, int64_t bsa, int64_t bsb,
                                                        int64_t batch) {
    const int64_t total = M * N * batch;
    const int64_t stride = (int64_t)gridDim.x * kHelperLanes;
    for (int64_t e = (int64_t)blockIdx.x * kHelperLanes + threadIdx.x; e < total; e += stride) {
        const int64_t t = e / (M * N), rem = e - t * M * N, i = rem / N, j = rem - i * N;
        const float *A = a + t * bsa, *B = b + t * bsb;
        float acc = 0.0f;
        for (int64_t k = 0; k < K; k++) {
            const float p = A[i * sam + k * sak] * B[k * sbk + j * sbn];
            acc = acc + p;
        }
        c[e] = acc;
    }
}

// Calls f<AKC, BKC>() for the operands' layouts.
template <class F>
int for_layout(bool a_plain, bool b_plain, F &&f) {
    if (a_plain && b_plain) return f.template operator()<true, false>();
    if (a_plain) return f.template operator()<true, true>();
    if (b_plain) return f.template operator()<false, false>();
    return f.template operator()<false, true>();
}

int64_t set_tiles(GemmArgs &g, int64_t bm, int64_t bn) {
    g.tiles_m = (int32_t)((g.M + bm - 1) / bm);
    g.tiles_n = (int32_t)((g.N + bn - 1) / bn);
    const int64_t tiles = (int64_t)g.tiles_m * g.tiles_n * g.batch;
    g.xcd_remap = tiles % kXcds == 0 ? 1 : 0;
    return tiles;
}

template <class T, int MINB>
int launch_tile(GemmArgs g, int64_t bm, int64_t bn, hipStream_t s) {
    const int64_t blocks = set_tiles(g, bm, bn);
    hipLaunchKernelGGL((gemm_split_tile<T, MINB>), dim3((unsigned)blocks), dim3(T::NT), 0, s, g);
    TRS_LAUNCH_CHECK("gemm kernel launch");
    return TRS_OK;
}

// Split K: an output with fewer tiles than CUs runs its K in S slices as S
// batches of its tile, into a workspace of S partial products that one more
// pass sums in slice order.  The workspace comes from the block cache and
// returns to it in stream order.  The last slice may be shorter (the kernel
// bounds each batch's k by the full depth).
//   - The large tile (the MLP's 8192x1024 and 4096x1024 GEMMs): S a power of
//     two up to 8, slices of at least kMinSplitDepth.
//   - The 128x128 and 64x128 tiles, when they give at most one block per CU
//     (1000^3 ran as 64 blocks, a 64x4096x4096 product as 32): S up to 16,
//     for about two blocks per CU, slices of at least 128 k, and at most
//     65,536 floats of partial products per CU.
constexpr int64_t kMaxSplitK = 8;
constexpr int64_t kMinSplitDepth = 1024;
constexpr int64_t kMaxTileSplit = 16;
constexpr int64_t kMinTileSplitDepth = 128;
constexpr int64_t kSplitFloatsPerCu = 65536;
// The least k per slice of a few 64x128 tiles (few_tiles in plan_gemm_tiles),
// and the least K that splits: a split costs its sum's launch, 2.3 us, and a
// 64x128 tile alone on a CU takes 0.032 us per k.
constexpr int64_t kMinFewDepth = 48, kMinFewK = 128;
// Time of a round of two 128x128 blocks per CU against one of a 256x256 block
// each: 0.50 to 0.57 for ragged single products and batches of K from 200 to
// 2200 (4095x300x4095 0.51, 700x600x700 x 24 0.55, 3318x2176x6109 0.53), 0.44
// at the least.  A ragged output takes the large tile when its rounds of
// blocks, so weighted, are no more: one round against two (5000x1000x3000 161 us,
// 177 on 128x128), not two against three (5348x192x4570 78, 67).
constexpr double kSmallPairOverLarge = 0.575;

// Which kernel a product runs.  Tile choice:
//   - the 256x256 tile when it divides M and N and gives every CU a block;
//     on ragged M or N (edge tiles bounds-checked, interior ones not) when
//     its rounds of blocks take no longer than the 128x128 tile's;
//   - a single matrix whose M or N exceeds such an output by at most 32 rows
//     or columns: the 256x256 tile on the rest, and the thin rims as skinny
//     products (4097^3 would otherwise run 17 x 17 large tiles, two rounds);
//   - else, for a single matrix with fewer large tiles than CUs, those
//     tiles at least 90% covered, and a long K, the 256x256 tile over S
//     K-slices, when S*tiles reaches half the CUs or at least the block
//     count of the tile it replaces;
//   - else 64x128 when 128x128 would give fewer than two blocks per CU and
//     64x128 divides the shape, whole pairs of slots in K (a CU with one block
//     then has two), else 128x128.  Other K would run as well on it: as it is
//     and on 64x128, us, 1024x1000x1024 29.0 and 26.8, 1024x500x2048 31.1 and
//     26.7, 1920x700x1280 33.9 and 35.6, but batches lose (448x700x896 x 9 39.7
//     and 46.8, 1024x300x1024 x 3 17.7 and 19.6);
//   - but 64x128 at any shape of 64 rows or more that leaves most CUs without
//     a block: half a 128x128 block's work on twice the CUs.  A single matrix
//     of at most a tile per four CUs (beyond, 128x128 in slices is as fast:
//     700^3 16.5 us, 16.1 on 64x128), split for at most one block per CU in
//     slices of at least kMinFewDepth; a K below kMinFewK and a batch, which do
//     not split, while their tiles have a CU each.  128x128 / 64x128, us:
//     64^3 6.5 / 5.9, 200x400x300 11.8 / 8.8, 300x784x500 13.4 / 12.0,
//     300x500x100 12.8 / 8.7, 96x6144x96 21.6 / 18.0, 1000x64x1000 7.5 / 6.8,
//     batches 32 of 100x128x100 9.5 / 8.2, 16 of 300^3 16.6 / 14.1, 8 of
//     200x200x700 12.8 / 11.1;
//   - a single matrix whose tile gives at most one block per CU splits K
//     over that tile (above);
//   - then stream-K on the 256x256 tile (below) replaces the plan where it
//     is estimated at least kStreamKGain faster.
enum class GemmKind { Strided, Large, SplitK, Medium, Small, StreamK };
struct GemmPlan {
    GemmKind kind = GemmKind::Strided;
    int bm = 0, bn = 0, bk = 0;
    int64_t splits = 1;
    int64_t blocks = 0;
    // SplitK only: the tile each slice runs on and the k per slice.
    // SplitK and StreamK: the plan run when no workspace can be allocated.
    GemmKind split_tile = GemmKind::Large;
    int64_t ks = 0;
    GemmKind fallback = GemmKind::Small;
    // Large with rims: the tile runs on rows [0, main_m) and columns
    // [0, main_n); the rest is peeled off as skinny products (0: nothing).
    int64_t main_m = 0, main_n = 0;
};

// One product (or K slice per batch) on a tile, without a split.
int launch_kind(GemmKind kind, const GemmArgs &g, bool a_plain, bool b_plain, int cu_count, hipStream_t s) {
    const bool alone = (g.M + 127) / 128 * ((g.N + 127) / 128) * g.batch <= cu_count;
    return for_layout(a_plain, b_plain, [&]<bool AKC, bool BKC>() -> int {
        switch (kind) {
        case GemmKind::Large: return launch_tile<LargeTile<AKC, BKC>, 1>(g, kLarge, kLarge, s);
        case GemmKind::Medium: return launch_tile<MediumTile<AKC, BKC>, 2>(g, 64, 128, s);
        default:
            if (alone) return launch_tile<SmallTile8<AKC, BKC>, 1>(g, 128, 128, s);
            return launch_tile<SmallTile<AKC, BKC>, 2>(g, 128, 128, s);
        }
    });
}

GemmPlan plan_gemm_tiles(const GemmArgs &g, bool a_plain, bool a_trans, bool b_plain, bool b_trans, int cu_count) {
    GemmPlan p;
    const int64_t M = g.M, N = g.N, K = g.K, batch = g.batch;
    if (!(a_plain || a_trans) || !(b_plain || b_trans)) {
        p.kind = GemmKind::Strided;
        p.blocks = std::min<int64_t>((M * N * batch + 255) / 256, (int64_t)cu_count * 16);
        return p;
    }
    constexpr int64_t L = kLarge;
    const auto ceil_div = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
    const int64_t large_tiles = ceil_div(M, L) * ceil_div(N, L) * batch;
    const int64_t small_tiles = ceil_div(M, 128) * ceil_div(N, 128) * batch;
    const bool large_div = M % L == 0 && N % L == 0;
    const auto use_large = [&](int64_t tiles) {
        p.kind = GemmKind::Large;
        p.bm = L, p.bn = L, p.bk = kSlot;
        p.blocks = tiles;
    };
    if (large_div && large_tiles >= cu_count) {
        use_large(large_tiles);
        return p;
    }
    // Thin rims peeled off a single matrix.
    if (batch == 1) {
        const int64_t mr = M % L, nr = N % L;
        const bool pm = M > L && mr >= 1 && mr <= kSkinnyMaxRows;
        const bool pn = N > L && nr >= 1 && nr <= kSkinnyMaxRows;
        const int64_t mm = pm ? M - mr : M, nn = pn ? N - nr : N;
        const int64_t tiles = ceil_div(mm, L) * ceil_div(nn, L);
        if ((pm || pn) && tiles >= cu_count) {
            use_large(tiles);
            p.main_m = mm;
            p.main_n = nn;
            return p;
        }
    }
    if (!large_div && large_tiles >= cu_count &&
        (double)ceil_div(large_tiles, cu_count) <= kSmallPairOverLarge * (double)ceil_div(small_tiles, 2 * cu_count)) {
        use_large(large_tiles);
        return p;
    }
    const int64_t medium_tiles = ceil_div(M, 64) * ceil_div(N, 128) * batch;
    const bool medium_div = M % 64 == 0 && N % 128 == 0 && K % 32 == 0 && small_tiles < 2 * (int64_t)cu_count;
    const bool splits = batch == 1 && K >= kMinFewK;
    const bool few_tiles = !medium_div && M >= 64 && medium_tiles <= (splits ? cu_count / 4 : cu_count);
    if (medium_div || few_tiles) {
        p.kind = GemmKind::Medium;
        p.bm = 64, p.bn = 128;
        p.blocks = medium_tiles;
    } else {
        p.kind = GemmKind::Small;
        p.bm = 128, p.bn = 128;
        p.blocks = small_tiles;
    }
    p.bk = kSlot;
    // The large split needs the 256x256 tiles nearly full (a 64-row output
    // would compute four times its rows): at least 90% of their area.
    const bool large_dense = (double)(M * N * batch) >= 0.9 * (double)(large_tiles * L * L);
    if (batch == 1 && large_dense && large_tiles > 0 && large_tiles < cu_count) {
        int64_t S = 1;
        while (S < kMaxSplitK && large_tiles * S * 2 <= cu_count && K / (S * 2) >= kMinSplitDepth) S *= 2;
        if (S > 1 && (2 * large_tiles * S >= cu_count || large_tiles * S >= p.blocks)) {
            const int64_t ks = ceil_div(ceil_div(K, S), 2 * kSlot) * (2 * kSlot);
            p.fallback = p.kind;
            p.kind = GemmKind::SplitK;
            p.split_tile = GemmKind::Large;
            p.bm = L, p.bn = L;
            p.splits = ceil_div(K, ks);
            p.ks = ks;
            p.blocks = large_tiles * p.splits;
            return p;
        }
    }
    if (batch == 1 && p.blocks <= cu_count && (splits || !few_tiles)) {
        int64_t S = std::min<int64_t>(kMaxTileSplit, (few_tiles ? 1 : 2) * (int64_t)cu_count / p.blocks);
        S = std::min<int64_t>(S, K / (few_tiles ? kMinFewDepth : kMinTileSplitDepth));
        S = std::min<int64_t>(S, kSplitFloatsPerCu * cu_count / (M * N));
        if (S >= 2) {
            const int64_t ks = ((K + S - 1) / S + p.bk - 1) / p.bk * p.bk;
            S = (K + ks - 1) / ks;
            if (S >= 2) {
                p.fallback = p.kind;
                p.split_tile = p.kind;
                p.kind = GemmKind::SplitK;
                p.splits = S;
                p.ks = ks;
                p.blocks *= S;
            }
        }
    }
    return p;
}

// Stream-K on the 256x256 tile: one block per CU, each taking
// an equal share of the product's (tile, slice) units, then one pass adding
// the pieces of the tiles split between blocks (gemm_split_tile_sk).  It
// removes the idle CUs of a last, partial round of tiles (6144^3: 576
// tiles, three rounds of 256 for 2.25 rounds of work) and of outputs with
// fewer tiles than CUs that no power-of-two K split fills (3072^3: 144).
//
// The choice compares estimated times in k steps of one 256x256 tile on one
// CU (0.16 us at 4096^3): the plan above by its rounds of
// blocks, and stream-K by its even share plus kStreamKCost for the pieces'
// extra traffic (two 256 KiB pieces per split tile written, read back and
// added, at most one split tile per block), the fix-up launch and a block's
// extra segment starts.  The 128x128 and 64x128 tiles cost 0.30 and 0.175
// of a large k step per k (their rates and areas; alone on a CU 2048^3 takes
// 0.048 us per k on 128x128, a 64x128 block 0.029).  Against every tile and up
// to 16 slices of 388 products of random shape, layout and batch the plan is
// the fastest for half, within 15% for nine in ten and 3.5% off in the mean;
// the worst split a short K that 128x128 tiles already give a round
// (5133x256x622 32.7 us in 2 slices, 17.3 whole; 5950x387x214 25.5 in 3, 16.0
// on 64x128 whole); of the large ones 512x4096x4096 115 us, 104 in 2 slices of
// 128x128, and 2048^3 114 on stream-K, 98.5 on 128x128 whole.  Stream-K needs
// tiles at least 85% covered, no K split of its own (ktotal), and at least
// kStreamKMinWork k steps per CU.
constexpr double kStreamKCost = 150.0;
constexpr double kStreamKMinWork = 192.0;
constexpr double kStreamKGain = 1.15;
constexpr double kSmallStep = 0.30, kMediumStep = 0.175;

double plan_k_steps(const GemmPlan &p, int64_t K, int cu_count) {
    const auto rounds = [&](int64_t blocks) { return (double)((blocks + cu_count - 1) / cu_count); };
    switch (p.kind) {
    case GemmKind::Large: return rounds(p.blocks) * (double)K;
    case GemmKind::SplitK: {
        const double step = p.split_tile == GemmKind::Large ? 1.0 : p.split_tile == GemmKind::Medium ? kMediumStep : kSmallStep;
        return rounds(p.blocks) * (double)p.ks * step + 50.0;
    }
    case GemmKind::Medium: return rounds(p.blocks) * (double)K * kMediumStep;
    case GemmKind::Small: return rounds(p.blocks) * (double)K * kSmallStep;
    default: return 0.0;
    }
}

GemmPlan plan_gemm(const GemmArgs &g, bool a_plain, bool a_trans, bool b_plain, bool b_trans, int cu_count) {
    GemmPlan p = plan_gemm_tiles(g, a_plain, a_trans, b_plain, b_trans, cu_count);
    if (p.kind == GemmKind::Strided || p.main_m || g.ktotal) return p;
    const int64_t tiles = ((g.M + 255) / 256) * ((g.N + 255) / 256) * g.batch;
    if ((double)(g.M * g.N * g.batch) < 0.85 * (double)(tiles * kLargeTileFloats)) return p;
    const double work = (double)tiles * (double)g.K / cu_count;
    if (work < kStreamKMinWork || plan_k_steps(p, g.K, cu_count) < kStreamKGain * (work + kStreamKCost)) return p;
    GemmPlan sk;
    sk.kind = GemmKind::StreamK;
    sk.bm = kLarge, sk.bn = kLarge, sk.bk = slice_depth(g, a_plain);
    sk.splits = 0;
    sk.blocks = cu_count;
    sk.fallback = p.kind == GemmKind::SplitK ? p.fallback : p.kind;
    return sk;
}

// Runs a stream-K plan; TRS_E_ALLOCATION_FAILED, with nothing launched, when
// the workspace (two partial tiles per block, 512 KiB per CU) cannot be had.
int launch_stream_k(const GemmPlan &p, GemmArgs g, bool a_plain, bool b_plain, int cu_count, hipStream_t s) {
    void *ws = nullptr;
    int rc = trs_alloc((size_t)(2 * (int64_t)cu_count * kLargeTileFloats) * sizeof(float), &ws);
    if (rc) return rc;
    g.sk_blocks = cu_count;
    g.sk_ws = (float *)ws;
    const int64_t tiles = set_tiles(g, kLarge, kLarge);
    g.sk_depth = p.bk;
    g.sk_q = (g.K + p.bk - 1) / p.bk;
    g.sk_units = tiles * g.sk_q;
    g.xcd_remap = cu_count % kXcds == 0 ? 1 : 0;
    rc = for_layout(a_plain, b_plain, [&]<bool AKC, bool BKC>() -> int {
        using T = LargeTile<AKC, BKC>;
        hipLaunchKernelGGL((gemm_split_tile_sk<T>), dim3((unsigned)cu_count), dim3(T::NT), 0, s, g);
        TRS_LAUNCH_CHECK("stream-k gemm launch");
        hipLaunchKernelGGL(gemm_streamk_fixup, dim3((unsigned)tiles, 16), dim3(256), 0, s, g);
        TRS_LAUNCH_CHECK("stream-k fix-up launch");
        return TRS_OK;
    });
    const int frc = trs_free(ws);
    return rc ? rc : frc;
}

// Runs a split plan; returns TRS_E_ALLOCATION_FAILED without launching
// anything when the workspace cannot be had (the caller then runs the
// unsplit tile).  `sak`/`sbk` are the operands' k strides.
int launch_split_k(const GemmPlan &p, GemmArgs g, bool a_plain, bool b_plain, int64_t sak, int64_t sbk,
                   int cu_count, hipStream_t s) {
    float *const C = g.c;
    const int64_t mn = g.M * g.N, S = p.splits, Ks = p.ks;
    void *ws = nullptr;
    int rc = trs_alloc((size_t)(S * mn) * sizeof(float), &ws);
    if (rc) return rc;
    g.c = (float *)ws;
    g.ktotal = g.K;
    g.K = Ks;
    g.bsa = Ks * sak;
    g.bsb = Ks * sbk;
    g.bsc = mn;
    g.batch = S;
    rc = launch_kind(p.split_tile, g, a_plain, b_plain, cu_count, s);
    if (rc == TRS_OK) {
        if (mn % 4 == 0 && (uintptr_t)C % 16 == 0) {
            const int64_t n4 = mn / 4;
            // A sum of at most two blocks per CU is load-latency bound: its
            // lanes issue every slice's load at once.  A larger one keeps one
            // load per lane in flight and leaves the latency to the many
            // resident waves (all at once measured 0.3 us slower at 1000^3
            // and 0.5% on the [8192,4096] -> 4096 -> 1024 MLP step).
            const dim3 grid((unsigned)((n4 + 255) / 256));
            if (n4 <= 2 * 256 * (int64_t)cu_count)
                launch_splitk_sum((int)S, grid, s, (const float4 *)ws, (float4 *)C, n4);
            else
                hipLaunchKernelGGL(splitk_sum<0>, grid, dim3(kHelperLanes), 0, s, (const float4 *)ws, (float4 *)C, n4, (int)S);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) rc = hip_fail(e, "split-k sum launch");
        } else {
            rc = launch_slice_sum((const float *)ws, C, mn, 1, S, s);
        }
    }
    const int frc = trs_free(ws);
    return rc ? rc : frc;
}

// Operand analysis shared by trs_matmul_f32 and trs_matmul_plan_f32: checks
// the layouts and fills the GEMM arguments.  *empty is set when nothing is
// to be computed (an empty output, or K = 0).
struct GemmSetup {
    GemmArgs g{};
    bool a_plain = false, a_trans = false, b_plain = false, b_trans = false;
    int64_t sam = 0, sak = 0, sbk = 0, sbn = 0;
    bool empty_output = false, zero_k = false;
};

int setup_gemm(const float *a, const trs_layout *la, const float *b, const trs_layout *lb, float *c,
               const trs_layout *lc, bool check_pointers, GemmSetup *st) {
    int rc = check_layout(la, "left");
    if (!rc) rc = check_layout(lb, "right");
    if (!rc) rc = check_layout(lc, "output");
    if (rc) return rc;
    if (la->rank != lb->rank || (la->rank != 2 && la->rank != 3))
        return set_error(TRS_E_MATMUL_REQUIRES_MATRICES,
                         "matmul currently requires two rank-2 tensors (or two rank-3 batches), got ranks %d and %d",
                         la->rank, lb->rank);
    const int r = la->rank;
    const int64_t batch = r == 3 ? la->shape[0] : 1;
    if (r == 3 && (lb->shape[0] != batch))
        return set_error(TRS_E_SHAPE_MISMATCH, "batch sizes differ (%lld and %lld)", (long long)batch,
                         (long long)lb->shape[0]);
    const int64_t M = la->shape[r - 2], K = la->shape[r - 1], K2 = lb->shape[r - 2], N = lb->shape[r - 1];
    if (K != K2)
        return set_error(TRS_E_MATMUL_INNER_MISMATCH, "mat1 and mat2 shapes cannot be multiplied (%lldx%lld and %lldx%lld)",
                         (long long)M, (long long)K, (long long)K2, (long long)N);
    if (lc->rank != r || lc->shape[r - 2] != M || lc->shape[r - 1] != N || (r == 3 && lc->shape[0] != batch))
        return set_error(TRS_E_SHAPE_MISMATCH, "matmul output layout has the wrong shape");
    if (!layout_is_contiguous(lc)) return set_error(TRS_E_INVALID_ARGUMENT, "matmul output must be contiguous");
    st->empty_output = M == 0 || N == 0 || batch == 0;
    st->zero_k = K == 0;
    if (st->empty_output) return TRS_OK;
    if (check_pointers) {
        // With K = 0 the operands are empty (no storage is needed) and C is +0.0.
        if (!c || (K > 0 && (!a || !b))) return set_error(TRS_E_INVALID_ARGUMENT, "null matmul operand");
        // C is written while A and B are still being read: no shared memory.
        const ByteRange out_bytes = byte_range(c, lc, 4);
        if (K > 0 && (ranges_overlap(out_bytes, byte_range(a, la, 4)) || ranges_overlap(out_bytes, byte_range(b, lb, 4))))
            return set_error(TRS_E_INVALID_ARGUMENT, "matmul output overlaps an operand");
    }
    st->sam = la->stride[r - 2], st->sak = la->stride[r - 1];
    st->sbk = lb->stride[r - 2], st->sbn = lb->stride[r - 1];
    const int64_t bsa = r == 3 ? la->stride[0] : 0, bsb = r == 3 ? lb->stride[0] : 0;
    // A unit-stride along k (plain) or along m (transposed view); same for B.
    st->a_plain = st->sak == 1 || K == 1;
    st->a_trans = !st->a_plain && (st->sam == 1 || M == 1);
    st->b_plain = st->sbn == 1 || N == 1;
    st->b_trans = !st->b_plain && (st->sbk == 1 || K == 1);
    GemmArgs &g = st->g;
    g.a = a ? a + la->offset : nullptr;
    g.b = b ? b + lb->offset : nullptr;
    g.c = c ? c + lc->offset : nullptr;
    g.M = M;
    g.N = N;
    g.K = K;
    g.lda = st->a_plain ? st->sam : st->sak;
    g.ldb = st->b_plain ? st->sbk : st->sbn;
    g.ldc = N;
    g.bsa = bsa;
    g.bsb = bsb;
    g.bsc = M * N;
    g.batch = batch;
    return TRS_OK;
}

// The skinny form of a product whose operands each have a unit stride and
// whose output has at most kSkinnyMaxRows rows or columns: the short side
// is X's rows (A's rows, or B's columns read as B^T) and the other operand
// is Y.  Returns false otherwise.
bool skinny_problem(const GemmSetup &st, SkinnyProblem *sp) {
    const GemmArgs &g = st.g;
    if (!(st.a_plain || st.a_trans) || !(st.b_plain || st.b_trans)) return false;
    const bool short_m = g.M <= g.N;
    if ((short_m ? g.M : g.N) > kSkinnyMaxRows) return false;
    SkinnyProblem p;
    p.K = g.K;
    p.batch = g.batch;
    p.out = g.c;
    if (short_m) {
        // X(i, k) = A(i, k); Y(k, j) = B(k, j); C(i, j) at i*N + j.
        p.x = g.a, p.y = g.b;
        p.R = g.M, p.L = g.N;
        p.xi = st.a_plain ? g.lda : 1;
        p.xk = st.a_plain ? 1 : g.lda;
        p.dot = !st.b_plain;
        p.yl = g.ldb;
        p.oi = g.N, p.oj = 1;
        p.bx = g.bsa, p.by = g.bsb;
    } else {
        // X(i, k) = B(k, i); Y(k, j) = A(j, k); C(j, i) at j*N + i.
        p.x = g.b, p.y = g.a;
        p.R = g.N, p.L = g.M;
        p.xi = st.b_plain ? 1 : g.ldb;
        p.xk = st.b_plain ? g.ldb : 1;
        p.dot = st.a_plain;
        p.yl = g.lda;
        p.oi = 1, p.oj = g.N;
        p.bx = g.bsb, p.by = g.bsa;
    }
    *sp = p;
    return true;
}

// A Large plan with rims: the tile on C[0:main_m, 0:main_n], then the rows
// below as one skinny product (X = those rows of A, Y = B, full width) and
// the columns to the right of the tile's rows as another (X = those columns
// of B read as B^T, Y = A's first main_m rows), each writing its part of C
// in place.
int run_peeled(const GemmPlan &p, const GemmSetup &st, int cu_count, hipStream_t s) {
    const GemmArgs &g = st.g;
    GemmArgs gm = g;
    gm.M = p.main_m;
    gm.N = p.main_n;
    TRS_CHECK(launch_kind(GemmKind::Large, gm, st.a_plain, st.b_plain, cu_count, s));
    if (p.main_m < g.M) {
        SkinnyProblem r;
        r.R = g.M - p.main_m, r.L = g.N, r.K = g.K, r.batch = 1;
        r.x = st.a_plain ? g.a + p.main_m * g.lda : g.a + p.main_m;
        r.xi = st.a_plain ? g.lda : 1;
        r.xk = st.a_plain ? 1 : g.lda;
        r.y = g.b, r.dot = !st.b_plain, r.yl = g.ldb;
        r.out = g.c + p.main_m * g.ldc, r.oi = g.ldc, r.oj = 1;
        SkinnyPlan rp;
        if (!plan_skinny(r, cu_count, &rp)) return set_error(TRS_E_INVALID_ARGUMENT, "gemm row rim has no plan");
        TRS_CHECK(run_skinny(r, rp, s));
    }
    if (p.main_n < g.N) {
        SkinnyProblem c;
        c.R = g.N - p.main_n, c.L = p.main_m, c.K = g.K, c.batch = 1;
        c.x = st.b_plain ? g.b + p.main_n : g.b + p.main_n * g.ldb;
        c.xi = st.b_plain ? 1 : g.ldb;
        c.xk = st.b_plain ? g.ldb : 1;
        c.y = g.a, c.dot = st.a_plain, c.yl = g.lda;
        c.out = g.c + p.main_n, c.oi = 1, c.oj = g.ldc;
        SkinnyPlan cp;
        if (!plan_skinny(c, cu_count, &cp)) return set_error(TRS_E_INVALID_ARGUMENT, "gemm column rim has no plan");
        TRS_CHECK(run_skinny(c, cp, s));
    }
    return TRS_OK;
}

}  // namespace

}  // namespace trs

using namespace trs;

extern "C" int trs_matmul_f32(const float *a, const trs_layout *la, const float *b, const trs_layout *lb,
                              float *c, const trs_layout *lc) {
    DeviceState *dev = device_state();
    if (!dev) return TRS_E_NO_DEVICE;
    GemmSetup st;
    int rc = setup_gemm(a, la, b, lb, c, lc, true, &st);
    if (rc || st.empty_output) return rc;
    const GemmArgs &g = st.g;
    if (st.zero_k) return trs_memset_zero(g.c, (size_t)(g.M * g.N * g.batch) * sizeof(float));
    SkinnyProblem sp;
    SkinnyPlan spl;
    if (skinny_problem(st, &sp) && plan_skinny(sp, dev->cu_count, &spl)) return run_skinny(sp, spl, dev->stream);
    const GemmPlan p = plan_gemm(g, st.a_plain, st.a_trans, st.b_plain, st.b_trans, dev->cu_count);
    if (p.main_m) return run_peeled(p, st, dev->cu_count, dev->stream);
    if (p.kind == GemmKind::Strided) {
        // An operand with no unit stride is gathered into a contiguous buffer
        // from the block cache (the library's copy kernel, bit for bit), and
        // the product runs on the MFMA tiles: 1024^3 over stride-2 views took
        // 0.589 ms in the one-lane-per-output kernel below, against 0.049 ms
        // for contiguous operands.  The buffers go back to the cache in stream
        // order.  Without memory for them, that kernel runs instead.
        const bool ga = !(st.a_plain || st.a_trans), gb = !(st.b_plain || st.b_trans);
        const trs_layout ca = contiguous_like(la), cb = contiguous_like(lb);
        void *ta = nullptr, *tb = nullptr;
        if (ga) rc = trs_alloc((size_t)layout_numel(la) * sizeof(float), &ta);
        if (!rc && gb) rc = trs_alloc((size_t)layout_numel(lb) * sizeof(float), &tb);
        if (!rc && ga) rc = trs_unary_f32(TRS_COPY, a, la, (float *)ta, &ca);
        if (!rc && gb) rc = trs_unary_f32(TRS_COPY, b, lb, (float *)tb, &cb);
        if (!rc)
            rc = trs_matmul_f32(ga ? (const float *)ta : a, ga ? &ca : la, gb ? (const float *)tb : b, gb ? &cb : lb,
                                c, lc);
        const bool no_memory = rc == TRS_E_ALLOCATION_FAILED;
        if (ta) trs_free(ta);
        if (tb) trs_free(tb);
        if (!no_memory) return rc;
        hipLaunchKernelGGL(gemm_f32_strided, dim3((unsigned)p.blocks), dim3(kHelperLanes), 0, dev->stream, g.a, g.b, g.c, g.M,
                           g.N, g.K, st.sam, st.sak, st.sbk, st.sbn, g.bsa, g.bsb, g.batch);
        TRS_LAUNCH_CHECK("strided gemm launch");
        return TRS_OK;
    }
    if (p.kind == GemmKind::StreamK) {
        rc = launch_stream_k(p, g, st.a_plain, st.b_plain, dev->cu_count, dev->stream);
        if (rc != TRS_E_ALLOCATION_FAILED) return rc;
        // No workspace: run the plan stream-K replaced, unsplit.
        return launch_kind(p.fallback, g, st.a_plain, st.b_plain, dev->cu_count, dev->stream);
    }
    if (p.kind == GemmKind::SplitK) {
        rc = launch_split_k(p, g, st.a_plain, st.b_plain, st.sak, st.sbk, dev->cu_count, dev->stream);
        if (rc != TRS_E_ALLOCATION_FAILED) return rc;
        // No workspace: the split is only an optimisation, so run the tile the
        // plan would otherwise have chosen (nothing was launched).
        return launch_kind(p.fallback, g, st.a_plain, st.b_plain, dev->cu_count, dev->stream);
    }
    return launch_kind(p.kind, g, st.a_plain, st.b_plain, dev->cu_count, dev->stream);
}

extern "C" int trs_matmul_plan_f32(const float *a, const trs_layout *la, const float *b, const trs_layout *lb,
                                   const float *c, const trs_layout *lc, int *tile_m, int *tile_n, int *tile_k,
                                   int64_t *splits, int64_t *blocks) {
    DeviceState *dev = device_state();
    if (!dev) return TRS_E_NO_DEVICE;
    GemmSetup st;
    int rc = setup_gemm(a, la, b, lb, const_cast<float *>(c), lc, false, &st);
    if (rc) return rc;
    GemmPlan p;
    const bool work = !st.empty_output && !st.zero_k;
    if (work) p = plan_gemm(st.g, st.a_plain, st.a_trans, st.b_plain, st.b_trans, dev->cu_count);
    GemmSetup sg;
    const GemmSetup *ran = &st;
    if (p.kind == GemmKind::Strided) {
        // What trs_matmul_f32 runs: the plan of the gathered, contiguous
        // operands (their buffers come from the block cache, 256-byte aligned).
        const bool ga = !(st.a_plain || st.a_trans), gb = !(st.b_plain || st.b_trans);
        const trs_layout ca = contiguous_like(la), cb = contiguous_like(lb);
        rc = setup_gemm(ga ? nullptr : a, ga ? &ca : la, gb ? nullptr : b, gb ? &cb : lb, const_cast<float *>(c), lc,
                        false, &sg);
        if (rc) return rc;
        p = plan_gemm(sg.g, sg.a_plain, sg.a_trans, sg.b_plain, sg.b_trans, dev->cu_count);
        ran = &sg;
    }
    SkinnyProblem sp;
    SkinnyPlan spl;
    if (work && skinny_problem(*ran, &sp) && plan_skinny(sp, dev->cu_count, &spl)) {
        // The short side's padded MFMA rows by the 64 columns of a block, or
        // for the matrix-vector kernel its 1, 2 or 4 rows by the 4 rows of
        // the long operand a block takes.
        const bool short_m = ran->g.M <= ran->g.N;
        const int rows = (spl.gemv || spl.axpy) ? spl.row_groups : 16 * spl.row_groups;
        const int cols = spl.gemv ? 4 : spl.axpy ? kAxpyCols : spl.lds ? kLdsSkinnyCols : kSkinnyCols;
        p.bm = short_m ? rows : cols;
        p.bn = short_m ? cols : rows;
        p.bk = (int)spl.kc;
        p.splits = spl.splits;
        p.blocks = spl.blocks;
    }
    if (tile_m) *tile_m = p.bm;
    if (tile_n) *tile_n = p.bn;
    if (tile_k) *tile_k = p.bk;
    if (splits) *splits = p.splits;
    if (blocks) *blocks = p.blocks;
    return TRS_OK;
}
