// bf16 products of more than 64 rows over the tiled copy of a weight (gemm_skinny.hip says how it is laid out): y = x W^T, the
// same with the activation of a joined [gate; up] matrix applied to the sums, and partial products over ranges of K for a norm
// that adds them up.  The reference leaves all of these to cuBLAS (base/src/engine.cu:652-671).
//
// Prompts, portions and steps of many decoding requests take them: some 65 to 3,000 rows of 1,000 to 30,000 outputs, sizes at
// which a tile's shape decides how full the 256 compute units are (one workgroup a unit: its stages take most of the LDS).  So
// there are ten shapes, and gt_plan below takes the one that it expects to be fastest.  The vendor library against these, us (in a graph, the rows
// just written by another kernel, weights from memory; activation included where the matrix is joined, and what the norm reads more of where
// the product is left in ranges):
//   2,048 outputs of 2,048 inputs: 128 rows 8.6 / 7.4, 512 11.4 / 9.8, 1,203 20.1 / 16.4, 2,048 21.6 / 19.8
//   16,384 joined of 2,048: 128 rows 24.7 / 21.4, 512 43 / 36, 1,203 88 / 78, 2,048 137 / 127, 4,096 240 / 236
//   2,048 of 8,192: 128 rows 21.2 / 16.1 (four ranges), 512 34.7 / 28.6 (four), 1,203 64.0 / 47.9 (two), 2,048 77 / 68 (two), 4,096 120 / 116
//   5,152 of 2,048: 512 rows 24.0 / 19.4, 2,048 50 / 49; 6,144 of 4,096: 128 rows 25.2 / 21.3, 1,024 54 / 51, 2,048 84 (the library's)
#include "tile_activations.h"
#include "tile_product.h"

#include <type_traits>

enum { GT_PLAIN = 0, GT_PARTS = 1, GT_GATED = 2 };

struct GtArgs {
    const bf16_t *x, *w;
    void *out;              // bf16 [M, N] ([M, N / 2] gated), or fp32 [splits, M, N]
    int M, N, K, splits, act;
};

template <class P, int FORM>
__global__ void __launch_bounds__(P::THREADS, P::WAVES / 4)
gemm_tiles_kernel(GtArgs a) {
    __shared__ __align__(16) typename P::Shared shared;
    const int lane = threadIdx.x % KVA_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KVA_WAVE), r = lane & 15, g = lane >> 4;
    const int halves = FORM == GT_GATED ? 2 : 1, outs = a.N / halves, half_tiles = (outs + 15) / 16, tiles = half_tiles * halves;
    const int row_tiles = (a.M + P::ROWS - 1) / P::ROWS, col_tiles = (tiles * 16 + P::OUTS - 1) / P::OUTS, per = row_tiles * col_tiles;
    // Neighbours of this list run on one die: up to eight row tiles of one column of tiles, then the next column's.  What they
    // share is in that die's L2 (eight x four tiles of a die at 2,048 rows; all row tiles first: 1-2 % slower).
    const int place = die_order(blockIdx.x, gridDim.x), split = place / per, id = place % per;
    constexpr int GROUP = 8;
    const int group = id / (GROUP * col_tiles), in = id % (GROUP * col_tiles), rows_in = min(GROUP, row_tiles - group * GROUP);
    const int m0 = (group * GROUP + in % rows_in) * P::ROWS, tile0 = in / rows_in * (P::OUTS / 16);
    P p;
    // (gate and up tiles of the same outputs alternate, so that a lane holds both)
    p.init(a.x, a.M, m0, a.w, tiles, a.K, [&](int j) {
        return FORM == GT_GATED ? (j & 1) * half_tiles + min(tile0 / 2 + j / 2, half_tiles - 1) : min(tile0 + j, tiles - 1);
    });
    const int k_per = (a.K / P::KS + a.splits - 1) / a.splits * P::KS, k_begin = split * k_per, k_end = min(a.K, k_begin + k_per);
    f32x4 acc[P::NT][P::RT];
    p.run(shared, k_begin, k_end, acc);
    const int wr = wave % P::WR, wn = wave / P::WR % P::WN;
    if constexpr (P::WK == 2) {
        // the second half of the wavefronts hands its sums over through LDS, lane by lane
        static_assert(sizeof(typename P::Shared) >= (size_t)P::WR * P::WN * P::NT * P::RT * 1024, "the sums fit where the operands were");
        f32x4 *box = reinterpret_cast<f32x4 *>(&shared) + (wave % (P::WR * P::WN)) * (P::NT * P::RT * KVA_WAVE) + lane;
        const bool hands_over = wave >= P::WR * P::WN;
        if (hands_over) {
#pragma unroll
            for (int i = 0; i < P::NT * P::RT; ++i) box[i * KVA_WAVE] = acc[i / P::RT][i % P::RT];
        }
        __syncthreads();
        if (hands_over) return;
#pragma unroll
        for (int i = 0; i < P::NT * P::RT; ++i) acc[i / P::RT][i % P::RT] += box[i * KVA_WAVE];
    }
    const bool whole4 = outs % 4 == 0;
    // (the activation is chosen in front: with the choice at every element the code of all of them, and not the sums, sets the time:
    // 16,384 joined outputs of 2,048 rows and inputs 126 us against 114.6)
    auto store = [&](auto silu) {
#pragma unroll
        for (int rt = 0; rt < P::RT; ++rt) {
            const int row = m0 + (wr * P::RT + rt) * 16 + r;
            if (row >= a.M) continue;
#pragma unroll
            for (int nt = 0; nt < P::NT; nt += FORM == GT_GATED ? 2 : 1) {
                const int n = (tile0 + wn * P::NT + nt) / halves * 16 + 4 * g;
                if (n >= outs) continue;
                f32x4 v = acc[nt][rt];
                if constexpr (FORM == GT_GATED) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) v[q] = (silu ? tile_silu(v[q]) : kva_activate(v[q], a.act)) * acc[nt + 1][rt][q];
                }
                if constexpr (FORM == GT_PARTS) {       // (N is a multiple of 4)
                    *reinterpret_cast<f32x4 *>(reinterpret_cast<float *>(a.out) + ((size_t)split * a.M + row) * a.N + n) = v;
                } else {
                    union {
                        b16x2 pair[2];
                        uint2 u;
                        uint16_t h[4];
                    } o;
                    o.pair[0] = pack_bf16(v[0], v[1]);
                    o.pair[1] = pack_bf16(v[2], v[3]);
                    uint16_t *to = reinterpret_cast<uint16_t *>(a.out) + (size_t)row * outs + n;
                    if (whole4) *reinterpret_cast<uint2 *>(to) = o.u;
                    else
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            if (n + q < outs) to[q] = o.h[q];
                }
            }
        }
    };
    if (FORM != GT_GATED || a.act == KVA_ACT_SILU) store(std::true_type{});
    else store(std::false_type{});
}

// The shapes: rows and outputs a workgroup, with what a launch of one turn of the units costs beside its stages (us), a stage of 64
// elements of K, a megabyte of operands, and a megabyte of partial products.  Fitted to 5,600 timings of 19 matrices of the 1B, 3B and 8B
// layer sizes and others at 65 to 8,190 rows, the same weights again from 1,000 rows on; 128 x 128's stage, 0.393 in that fit, is 0.41 because
// with weights from memory and the rows just written it takes 0.43.  In those conditions, 609 products of 18 matrices at 65 to
// 8,190 rows, what is chosen is 1.4 % behind the best of all shapes, ranges and the library on average, 4.5 % at the ninetieth of a hundred and 1.72 times
// at most (135 to 158 rows of 6,144 x 4,096, where the library's time jumps from 22 us to 38); the same from 0.40 to 0.42, with 0.393 0.05 % more, with all
// ten shapes fitted to these conditions 0.2 % more.  Five more shapes (64 x 128, 64 x 256, 96 x 256, 256 x 128, 128 x 256 by eight wavefronts) were tried
// and bring nothing on average.
struct GtShape {
    int rows, outs;
    float turn, stage, megabyte, part_megabyte;
};
#define GT_SHAPES(V)                                            \
    V(0, 8, 4, 2, 4, 1, 2, 2, 10.3f, 1.20f, 0.104f, 0.04f)      \
    V(1, 4, 8, 2, 2, 1, 2, 3, 6.53f, 0.665f, 0.075f, 0.08f)     \
    V(2, 4, 4, 2, 2, 2, 1, 4, 4.78f, 0.41f,  0.091f, 0.14f)     \
    V(3, 5, 4, 2, 4, 1, 2, 3, 7.90f, 0.80f, 0.047f, 0.07f)      \
    V(4, 5, 4, 2, 2, 2, 1, 4, 5.92f, 0.45f, 0.067f, 0.10f)      \
    V(5, 3, 4, 2, 2, 2, 1, 4, 4.25f, 0.337f, 0.118f, 0.145f)    \
    V(6, 6, 4, 2, 4, 1, 2, 2, 8.15f, 0.967f, 0.137f, 0.04f)     \
    V(7, 4, 6, 2, 2, 2, 1, 3, 6.02f, 0.511f, 0.095f, 0.09f)     \
    V(8, 2, 2, 2, 2, 2, 1, 8, 2.52f, 0.185f, 0.093f, 0.38f)     \
    V(9, 4, 2, 2, 2, 2, 1, 6, 3.37f, 0.277f, 0.085f, 0.25f)
#define GT_COUNT 10
static const GtShape gt_shapes[GT_COUNT] = {
#define GT_ROW(ID, RT, NT, WR, WN, WK, KSUB, ST, ...) {16 * RT * WR, 16 * NT * WN, __VA_ARGS__},
    GT_SHAPES(GT_ROW)
#undef GT_ROW
};
#define GT_UNITS 256
#define GT_STAGE 64
#define GT_MAX_SPLITS 4
#define GT_PARTS_BYTES (64ll << 20)     // partial products of one call

static long long gt_blocks(int shape, int M, int N, int splits) {
    const GtShape &s = gt_shapes[shape];
    return (long long)((M + s.rows - 1) / s.rows) * ((N + s.outs - 1) / s.outs) * splits;
}

static double gt_expected(int shape, int M, int N, int K, int splits) {
    const GtShape &s = gt_shapes[shape];
    const double turns = (double)((gt_blocks(shape, M, N, splits) + GT_UNITS - 1) / GT_UNITS);
    const double stages = (double)((K / GT_STAGE + splits - 1) / splits), operands = 2e-6 * K * ((double)N + M);
    // (the norm reads the ranges instead of a bf16 row: 5 TB/s)
    const double parts = splits > 1 ? 1e-6 * M * N * (4.0 * splits * s.part_megabyte + (4.0 * splits - 2.0) / 5.0) : 0.0;
    return turns * (s.turn + stages * s.stage) + operands * s.megabyte + parts;
}

// What the library is expected to take, from the same 19 matrices: 4.5 us and the operations at a rate that grows with the number
// of 256 x 256 tiles until they fill the units, falls back where a turn of them is partly empty, and is lower where the outputs are
// no multiple of 256; a few rows are a chain over K.  Its choices jump (192 rows of 3,072 x 8,192 58 us, 256 rows 33), so this is a
// middle.
static double gt_library(int M, int N, int K) {
    const double tiles = (double)M * N / 65536.0, turn = tiles / GT_UNITS;
    double rate = turn <= 1.0 ? 1550.0 * pow(turn, 0.3) : 1550.0 * pow(turn / ceil(turn), 0.55);
    if (N % 256) rate *= 0.87;
    return fmax(5.0 + 0.0024 * K, 4.5 + 2e-6 * M * N * K / rate);
}

static bool gt_sizes(int M, int N, int K, int form) {
    const int halves = form == GT_GATED ? 2 : 1;
    const long long padded = (long long)halves * ((N / halves + 15) / 16 * 16);
    return M > 0 && N > 0 && K >= GT_STAGE && K % GT_STAGE == 0 && N % halves == 0 && (form != GT_PARTS || N % 4 == 0) && padded * K * 2 <= 0x7fffffffll &&
           256ll * K * 2 <= 0x7fffffffll;
}

// Shape + 256 x ranges of K, or -1: the library is expected to be faster, or takes what these do not.
// Where the line lies, of the 19 matrices at 65 to 8,190 rows.  A layer's four products and two norms over all layers' weights in a graph, us by the
// library (with the activation's pass) / here, 96 / 517 / 1,203 / 2,048 / 4,096 rows: 1B sizes 77 / 130 / 216 / 272 / 451 -> 60 / 105 / 175 / 250 / 451, 3B 114 / 178 /
// 302 / 405 / 706 -> 84 / 149 / 273 / 388 / 694, 8B 180 / 348 / 563 / 781 / 1,324 -> 134 / 285 / 506 / 762 / 1,310.
// * the joined ones up to where rows x outputs x K make 3.3 million times 65,536: two passes over the sums are gone.  Of 170 of them with rows just
//   written and weights from memory five are slower than the library by 2 % and more: 421 to 512 and 766 rows of 28,672 x 4,096, 3 to 11 % (a turn of 224
//   workgroups); any line through the two estimates loses more elsewhere;
// * from 155 tiles of 256 x 256 on (2,048 rows x 5,120 outputs) the library's tiles of that size fill the units and run at 1.3 to 1.6
//   PFLOP/s against 1.2 to 1.4: 8,190 x 4,096 x 14,336 608 / 707 us; except where the outputs are no multiple of 256, 0.86 to 0.96 there;
// * below, where the expected time is at most 1.1 of the library's; up to 64 tiles 1.3 of it, because the library's
//   middle hides its slow choices: 0.53 to 0.98 in 111 of 129 cases.  Not where 64 x 64 tiles leave units idle over a long K (65 to 256 rows of 2,048 x
//   8,192 20-27 us by the library, 27-36 here) and not for a few outputs (16 of 2,048 rows and inputs: 5.1 / 6.9 us);
// * in ranges only where 1.15 of it is: 3,072 rows of 2,048 x 8,192 are 5 us slower in two ranges of 192 x 256 in a layer.
static int gt_plan(int M, int N, int K, int form) {
    if (!gt_sizes(M, N, K, form) || M <= 64) return -1;
    int best = -1, ranges = 1;
    double least = 0.0;
    for (int splits = 1; splits <= (form == GT_PARTS ? GT_MAX_SPLITS : 1); ++splits) {
        if (splits > 1 && (K < 512 * splits || 4ll * splits * M * N > GT_PARTS_BYTES)) break;
        const int stages = K / GT_STAGE, each = (stages + splits - 1) / splits;
        if ((splits - 1) * each >= stages) continue;
        for (int shape = 0; shape < GT_COUNT; ++shape) {
            const double t = gt_expected(shape, M, N, K, splits);
            if (gt_blocks(shape, M, N, splits) <= 0x7fffffffll && (best < 0 || t < least)) best = shape, ranges = splits, least = t;
        }
    }
    const double tiles = (double)M * N / 65536.0;
    const int chosen = best + 256 * ranges;
    if (form == GT_GATED) return tiles * K <= 3.3e6 ? chosen : -1;
    if (N < 256 || (tiles >= 155.0 && N % 256 == 0)) return -1;
    if (gt_shapes[best].rows == 64 && ranges == 1 && N < 2560 && K > 2560) return -1;
    return least * (ranges > 1 ? 1.15 : 1.0) <= gt_library(M, N, K) * (tiles < 64.0 ? 1.3 : 1.1) ? chosen : -1;
}

extern "C" int kva_gemm_tiles_plan(int M, int N, int K, int form) {
    return form < GT_PLAIN || form > GT_GATED ? -1 : gt_plan(M, N, K, form);
}

// x [M, K] bf16 and w in tiles (halves of their own for the gated form), both at addresses that are multiples of 16; out as in
// GtArgs, at a multiple of 16.  plan: shape + 256 x ranges (more than one range: partial products).
extern "C" int kva_gemm_tiles(void *out, const void *x, const void *w, int M, int N, int K, int form, int plan, int act,
                              hipStream_t stream) {
    const int shape = plan & 255, splits = plan >> 8;
    KVA_REQUIRE(form >= GT_PLAIN && form <= GT_GATED && gt_sizes(M, N, K, form), "gemm_tiles: no product of %d rows, %d outputs of %d inputs in form %d",
                M, N, K, form);
    KVA_REQUIRE(plan >= 0 && shape < GT_COUNT && splits >= 1 && splits <= GT_MAX_SPLITS && (form == GT_PARTS || splits == 1), "gemm_tiles: plan %d", plan);
    const int stages = K / GT_STAGE, each = (stages + splits - 1) / splits;
    KVA_REQUIRE((splits - 1) * each < stages, "gemm_tiles: %d ranges of %d stages of K", splits, stages);
    KVA_REQUIRE(out && x && w && (((uintptr_t)out | (uintptr_t)x | (uintptr_t)w) & 15) == 0, "gemm_tiles: operands must be at multiples of 16 bytes");
    KVA_REQUIRE(form != GT_GATED || kva_plain_activation(act), "gemm_tiles: activation %d", act);
    // (a joined matrix of N rows has tiles of 16 per half; a workgroup takes as many of either)
    const int halves = form == GT_GATED ? 2 : 1, padded = halves * ((N / halves + 15) / 16 * 16);
    const long long blocks = gt_blocks(shape, M, padded, splits);
    KVA_REQUIRE(blocks <= 0x7fffffffll, "gemm_tiles: too many workgroups");
    const GtArgs a{(const bf16_t *)x, (const bf16_t *)w, out, M, N, K, splits, act};
#define GT_LAUNCH(ID, RT, NT, WR, WN, WK, KSUB, ST, ...)                                                                                    \
    case ID: {                                                                                                                              \
        typedef TileProduct<RT, NT, WR, WN, WK, KSUB, ST> P;                                                                                \
        if (form == GT_PLAIN) hipLaunchKernelGGL((gemm_tiles_kernel<P, GT_PLAIN>), dim3(blocks), dim3(P::THREADS), 0, stream, a);           \
        else if (form == GT_PARTS) hipLaunchKernelGGL((gemm_tiles_kernel<P, GT_PARTS>), dim3(blocks), dim3(P::THREADS), 0, stream, a);      \
        else hipLaunchKernelGGL((gemm_tiles_kernel<P, GT_GATED>), dim3(blocks), dim3(P::THREADS), 0, stream, a);                            \
        break;                                                                                                                              \
    }
    switch (shape) { GT_SHAPES(GT_LAUNCH) }
#undef GT_LAUNCH
    KVA_CHECK_LAUNCH("gemm_tiles");
    return KVA_OK;
}
