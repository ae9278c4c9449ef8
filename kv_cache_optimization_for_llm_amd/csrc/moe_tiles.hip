// The experts' products of a prompt (moe.hip says what the list of slots is) over tiles of 64 x 64 to 256 x 256 (tile_product.h),
// for matrices in operand order whose K is a multiple of 64.
//
// The list has its slots in tiles of 16 by expert, and a workgroup takes up to G neighbouring tiles of one expert: where a block of
// G begins is worked out from the tiles' experts by every wavefront for itself, so one list serves both products in blocks of
// different heights.  (Lists in groups of G = 8, as moe.hip's kernel takes them, fix the height and pad every expert to it.)
//
// What bounds it: up to 2,000 tokens one or two turns of the units, a stage of 256 x 256 x 64 some 1.3 us of matrix products and loads,
// and around them the first operands' way from memory and the results' to it.  Before (moe.hip's 128 x 256, two workgroups a unit) and
// now, in the model, us: 2,048 tokens, 4 of 16 experts of 1,536 x 2,048 68 / 64 (805 TFLOP/s), of 2,048 x 768 58 / 48; 2,494 tokens, all of
// 4 of 1,536 x 2,048 66 / 64.  An activation that costs as much as the sums (erf-gelu, tanh) is better off in moe.hip's, where the other workgroup of
// the unit multiplies meanwhile, unless its turns divide badly (mt_first).
#include "tile_activations.h"
#include "tile_product.h"
#include <math.h>
#include <type_traits>

#define MT_TILE 16
#define MT_MAX_TILES 4096           // of a list: a lane keeps the blocks of 64 tiles in a mask

enum { MT_ACT_SILU = 0, MT_ACT_RELU = 1, MT_ACT_GELU_TANH = 2, MT_ACT_GELU = 3, MT_ACT_SWISH_CLAMPED = 4, MT_ACT_RELU2 = 5 };

struct MtArgs {
    const bf16_t *x, *w;
    void *out;
    const int *sorted_slot, *tile_expert;
    const float *slot_weight;       // first product: of the row that is read; second: of the row that is written; absent: 1
    int max_tiles, top, N, K, second, act;
    float limit;
};

template <int ACT>
__device__ __forceinline__ float mt_activate(float z) {
    if (ACT == MT_ACT_SILU) return tile_silu(z);
    if (ACT == MT_ACT_GELU) return tile_gelu(z);
    return kva_activate(z, ACT == MT_ACT_RELU ? KVA_ACT_RELU : ACT == MT_ACT_RELU2 ? KVA_ACT_RELU2 : KVA_ACT_GELU_TANH);
}

// The place of a workgroup: tile `first` and the tiles behind it that belong to its expert, G of them at most.  False: there is no
// work for this workgroup.
template <int G>
__device__ __forceinline__ bool mt_place(const int *__restrict__ tile_expert, int max_tiles, int n_blocks, int &first, int &tiles, int &column) {
    const int lane = threadIdx.x % KVA_WAVE;
    unsigned long long mine = 0;        // the tiles 64 lane .. 64 lane + 63 that begin a block
    int begin = 0;                      // of the run that reaches into the next 64
    for (int c0 = 0; c0 * KVA_WAVE < max_tiles; c0 += 8) {
        int e[8], before[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = (c0 + u) * KVA_WAVE + lane;
            e[u] = i < max_tiles ? tile_expert[i] : -1;
            before[u] = i > 0 && i < max_tiles ? tile_expert[i - 1] : -2;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int base = (c0 + u) * KVA_WAVE;
            const unsigned long long runs = __ballot(e[u] != before[u]), upto = runs & (~0ull >> (63 - lane));
            const int from = upto ? base + 63 - __clzll(upto) : begin;
            const unsigned long long blocks = __ballot(e[u] >= 0 && (base + lane - from) % G == 0);
            if (lane == c0 + u) mine = blocks;
            if (runs) begin = base + 63 - __clzll(runs);
        }
    }
    const int own = __popcll(mine);
    int upto = own;
#pragma unroll
    for (int off = 1; off < KVA_WAVE; off <<= 1) {
        const int v = __shfl_up(upto, off, KVA_WAVE);
        if (lane >= off) upto += v;
    }
    const int total = __shfl(upto, KVA_WAVE - 1, KVA_WAVE) * n_blocks;
    if ((int)blockIdx.x >= total) return false;
    // neighbours of the list of blocks run on one die, all columns of a block before the next one: a die reads few experts
    const int id = die_order(blockIdx.x, total), block = id / n_blocks;
    column = id % n_blocks;
    const int chunk = __popcll(__ballot(upto <= block));
    const unsigned long long mask = __shfl(mine, chunk, KVA_WAVE);
    const int nth = block - __shfl(upto - own, chunk, KVA_WAVE);
    const unsigned long long found = __ballot(((mask >> lane) & 1ull) && __popcll(mask & ((1ull << lane) - 1ull)) == nth);
    first = __builtin_amdgcn_readfirstlane(chunk * KVA_WAVE + __ffsll((long long)found) - 1);
    const int expert = tile_expert[first];
    tiles = __popcll(__ballot(lane < G && first + lane < max_tiles && tile_expert[min(first + lane, max_tiles - 1)] == expert));
    return true;
}

// (one variable in LDS: with several the compiler tells them apart, and waits for all loads on their way to one before it reads it)
template <class P>
struct MtShared {
    typename P::Shared operands;
    int slot_of[P::ROWS];
    float weight_of[P::ROWS];
};

template <class P, bool GATED>
__global__ void __launch_bounds__(P::THREADS, P::WAVES / 4)
moe_tiles_kernel(MtArgs a) {
    __shared__ __align__(16) MtShared<P> shared;
    const int lane = threadIdx.x % KVA_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KVA_WAVE), r = lane & 15, g = lane >> 4;
    int first, run, column;
    if (!mt_place<P::ROWS / MT_TILE>(a.tile_expert, a.max_tiles, (a.N + P::OUTS - 1) / P::OUTS, first, run, column)) return;
    const int rows = run * MT_TILE, place0 = first * MT_TILE, tile0 = column * (P::OUTS / 16), w_tiles = a.N / 16;
    for (int i = threadIdx.x; i < P::ROWS; i += P::THREADS) {
        const int slot = i < rows ? a.sorted_slot[place0 + i] : -1;
        shared.slot_of[i] = slot;
        shared.weight_of[i] = a.slot_weight && slot >= 0 ? a.slot_weight[slot] : 1.f;
    }
    P p;
    // (places without a slot, and rows past the expert's last tile: some row of the list, whose results go nowhere)
    p.init(buffer_at(a.x, 0xffffffffull), [&](int i) {
        const int place = place0 + min(i, rows - 1);
        return a.second ? place : max(a.sorted_slot[place], 0) / a.top;
    }, a.w + (size_t)__builtin_amdgcn_readfirstlane(a.tile_expert[first]) * a.N * a.K, w_tiles, a.K, [&](int j) { return min(tile0 + j, w_tiles - 1); });
    f32x4 acc[P::NT][P::RT];
    p.template run<GATED>(shared.operands, 0, a.K, acc);
    const int wr = wave % P::WR, wn = wave / P::WR % P::WN;
    if constexpr (P::WK == 2) {
        // the second half of the wavefronts hands its sums over through LDS, lane by lane
        static_assert(sizeof(typename P::Shared) >= (size_t)P::WR * P::WN * P::NT * P::RT * 1024, "the sums fit where the operands were");
        f32x4 *box = reinterpret_cast<f32x4 *>(&shared.operands) + (wave % (P::WR * P::WN)) * (P::NT * P::RT * KVA_WAVE) + lane;
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
    const int halves = GATED ? 2 : 1, outs = a.N / halves;      // a multiple of 8
    // (the activation is chosen in front of all elements)
    auto store = [&](auto act) {
        constexpr int ACT = decltype(act)::value;
#pragma unroll
        for (int rt = 0; rt < P::RT; ++rt) {
            const int row = (wr * P::RT + rt) * 16 + r, slot = shared.slot_of[row];
            if (slot < 0) continue;
            const float weight = shared.weight_of[row];
#pragma unroll
            for (int nt = 0; nt < P::NT; nt += halves) {
                const int n = (tile0 + wn * P::NT + nt) * (16 / halves) + 4 * g;
                if (n >= outs) continue;
                f32x4 v = acc[nt][rt] * weight;
                if constexpr (ACT < 0) {
                    *reinterpret_cast<f32x4 *>(reinterpret_cast<float *>(a.out) + (size_t)slot * outs + n) = v;
                } else {
                    if constexpr (GATED) {
                        const f32x4 o = acc[nt + 1][rt] * weight;
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const float gate = g < 2 ? v[q] : o[q], up = g < 2 ? o[q] : v[q];
                            v[q] = ACT == MT_ACT_SWISH_CLAMPED ? kva_gated_activate(gate, up, KVA_ACT_SWISH_CLAMPED, a.limit) : mt_activate<ACT>(gate) * up;
                        }
                    } else {
#pragma unroll
                        for (int q = 0; q < 4; ++q) v[q] = mt_activate<ACT>(v[q]);
                    }
                    union {
                        b16x2 pair[2];
                        uint2 u;
                    } o;
                    o.pair[0] = pack_bf16(v[0], v[1]);
                    o.pair[1] = pack_bf16(v[2], v[3]);
                    *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(a.out) + (size_t)(place0 + row) * outs + n) = o.u;
                }
            }
        }
    };
    if constexpr (!GATED) {
        if (a.second) {
            store(std::integral_constant<int, -1>{});
            return;
        }
    }
#define MT_STORE(ACT) case ACT: store(std::integral_constant<int, ACT>{}); break
    switch (a.act) {
        MT_STORE(MT_ACT_SILU);
        MT_STORE(MT_ACT_RELU);
        MT_STORE(MT_ACT_GELU_TANH);
        MT_STORE(MT_ACT_GELU);
        MT_STORE(MT_ACT_RELU2);
        default:
            if constexpr (GATED) store(std::integral_constant<int, MT_ACT_SWISH_CLAMPED>{});      // (a gated one)
    }
#undef MT_STORE
}

// The shapes: rows and outputs a workgroup, with what one turn of the units (one workgroup each) costs beside its stages (us), a stage of
// 64 elements of K, a megabyte of operands and one of results.  For the first product fitted, with moe_expert_rows' costs below, to the
// timings of all nine over 7,408 layers' experts, matrices from memory: 60 to 8,190 tokens, 1 to 6 of 4 to 64 experts chosen evenly, 1,024
// to 4,096 wide, 384 to 2,816 inside, six activations.  For the second to the nine over 45 sizes: 100 to 6,000 tokens, 4 to 64 experts, 512 to 4,096
// wide; the shape they choose there is 4 % behind the best of the nine on average.
struct MtShape {
    int rows, outs, threads;
    struct {
        float turn, stage, megabyte, results;
    } of[2];
};
#define MT_SHAPES(V)                                                                             \
    V(0, 8, 4, 2, 4, 1, 2, 2, 4.95f, 1.175f, 0.075f, 0.563f, 3.13f, 1.411f, 0.029f, 0.205f)      \
    V(1, 4, 8, 2, 2, 1, 2, 3, 5.08f, 0.643f, 0.080f, 0.470f, 2.58f, 0.842f, 0.063f, 0.208f)      \
    V(2, 4, 4, 2, 2, 2, 1, 4, 4.91f, 0.341f, 0.100f, 0.572f, 0.45f, 0.556f, 0.079f, 0.402f)      \
    V(3, 5, 4, 2, 4, 1, 2, 3, 5.94f, 0.735f, 0.072f, 0.632f, 0.98f, 1.025f, 0.031f, 0.251f)      \
    V(4, 5, 4, 2, 2, 2, 1, 4, 5.09f, 0.420f, 0.088f, 0.650f, 2.72f, 0.481f, 0.043f, 0.405f)      \
    V(5, 3, 4, 2, 2, 2, 1, 4, 4.22f, 0.314f, 0.097f, 0.671f, 0.00f, 0.606f, 0.031f, 0.410f)      \
    V(6, 6, 4, 2, 4, 1, 2, 2, 4.88f, 0.982f, 0.080f, 0.522f, 5.87f, 0.900f, 0.043f, 0.219f)      \
    V(7, 2, 2, 2, 2, 2, 1, 8, 5.02f, 0.191f, 0.065f, 0.188f, 0.00f, 0.262f, 0.115f, 1.008f)      \
    V(8, 4, 2, 2, 2, 2, 1, 6, 4.92f, 0.236f, 0.081f, 0.769f, 1.04f, 0.350f, 0.080f, 0.577f)
#define MT_COUNT 9
#define MT_BOTH(a, b, c, d, e, f, g, h) {a, b, c, d}, {e, f, g, h}
static const MtShape mt_shapes[MT_COUNT] = {
#define MT_ROW(ID, RT, NT, WR, WN, WK, KSUB, ST, ...) {16 * RT * WR, 16 * NT * WN, 64 * WR * WN, {MT_BOTH(__VA_ARGS__)}},
    MT_SHAPES(MT_ROW)
#undef MT_ROW
};
// an activation of each lane (MT_ACT_SILU ..), here a turn's and in moe_expert_rows
static const float mt_act_here[] = {0.0223f, 0.f, 0.0807f, 0.0591f, 0.0636f, 0.f}, mt_act_rows[] = {0.0483f, 0.f, 0.0853f, 0.0760f, 0.0581f, 0.f};
// moe_expert_rows' first product, two workgroups a unit: groups of 8 tiles against 256 outputs, against 128, groups of 4 against 128.  A stage of K in
// turns of 512 workgroups, a workgroup and a stage where turns even out, a workgroup and a stage in turns of 256, a megabyte of operands and of results.
struct MtRows {
    int rows, outs;
    float stage, even, even_stage, single, single_stage, megabyte, results;
};
static const MtRows mt_rows[] = {{128, 256, 0.2765f, 1.66f, 0.2623f, 0.72f, 0.4822f, 0.087f, 0.233f},
                                 {128, 128, 0.0765f, 3.37f, 0.f, 0.48f, 0.3150f, 0.112f, 0.403f},
                                 {64, 128, 0.0358f, 2.78f, 0.0492f, 0.f, 0.2069f, 0.134f, 0.f}};
#define MT_UNITS 256
#define MT_STAGE 64

static bool mt_sizes(long long tiles, int experts, int N, int K) {
    return tiles > 0 && tiles <= MT_MAX_TILES && experts > 0 && N > 0 && N % 16 == 0 && K >= MT_STAGE && K % MT_STAGE == 0 &&
           (long long)N * K * 2 <= 0x7fffffffll && tiles * MT_TILE * K * 2 <= 0x7fffffffll;
}

// (the second product: experts that all tokens take have as many rows each; else every expert's last block is half full on average)
static double mt_blocks(double slots, int experts, int top, int rows, int N, int outs) {
    return ceil(top == experts ? experts * ceil(slots / experts / rows) : slots / rows + 0.5 * experts) * ((N + outs - 1) / outs);
}

// Blocks of `rows` rows of one expert over all experts, on average, and their spread: an expert's rows are as many as all tokens', or spread as an even
// choice of `top` of `experts` spreads them.  Its blocks are those that surely fill and, of those around the mean, each by its likelihood.
struct MtSpread {
    double mean, spread;
};
static double mt_above(double z) { return 0.5 * erfc(z * 0.70710678118654752); }
static MtSpread mt_spread(double slots, int experts, int top, int rows) {
    const double n = slots / experts, sd = top < experts ? sqrt(n * (1.0 - (double)top / experts)) : 0.0;
    if (sd < 0.5) return {experts * ceil(n / rows), 0.0};
    const int sure = (int)fmax(0.0, (n - 4.0 * sd) / rows);
    double sum = 0.0, square = 0.0;
    for (int i = 0;; ++i) {
        const double p = mt_above(((double)rows * (sure + i) + 0.5 - n) / sd);
        if (p < 1e-4) break;
        sum += p, square += (2 * i + 1) * p;
    }
    return {experts * (sure + sum), sqrt(experts * fmax(0.0, square - sum * sum))};
}

// turns of `at_once` workgroups that these blocks against `columns` workgroups each take on average
static double mt_turns(MtSpread b, double columns, double at_once) {
    if (b.spread <= 0.05) return ceil(rint(b.mean) * columns / at_once);
    const int sure = (int)fmax(0.0, (b.mean - 4.0 * b.spread) * columns / at_once);
    double turns = sure;
    for (int i = sure;; ++i) {
        const double p = i == 0 ? 1.0 : mt_above((floor(at_once * i / columns) + 0.5 - b.mean) / b.spread);
        if (p < 1e-3) return turns;
        turns += p;
    }
}

// The first product: of the 7,408 (half of them not fitted to) the choice is 1.2 % behind the best on average, taken in 0.78 of them, 0.873 of
// moe_expert_rows' time over all, and slower by more than 3 % in 3 % (with a line at 1 instead of 0.97 4 %).  Without the activation, with turns from the
// mean number of workgroups and no estimate for moe_expert_rows: 4.7 %, 0.87, 0.903 and 14 %.  us, moe_expert_rows / here: 8,192 slots of
// 16 experts of 1,536 x 2,048, gated silu, 64.7 / 62.3, of 1,024 x 2,048, erf-gelu, 68.5 / 49.6, 1,024 slots of 4 16.8 / 12.2; but 8,192 slots of 4
// experts of 1,024 x 2,048 with erf-gelu 43.4 / 44.6 and with the tanh form 43.1 / 48.5, 4,812 of 32 of 1,024 x 1,024 27.3 / 33.3.
static int mt_first(int slots, int experts, int top, int N, int K, int act, int gated, int group, long long list) {
    const double halves = gated ? 2.0 : 1.0, operands = 2e-6 * K * ((double)N * experts + slots), results = 2e-6 * slots * N / halves, stages = K / MT_STAGE;
    int best = -1;
    double least = 0.0;
    for (int i = 0; i < MT_COUNT; ++i) {
        const MtShape &s = mt_shapes[i];
        const double turns = mt_turns(mt_spread(slots, experts, top, s.rows), (N + s.outs - 1) / s.outs, MT_UNITS);
        const double t = turns * (s.of[0].turn + stages * s.of[0].stage + mt_act_here[act] * s.rows * s.outs / halves / s.threads) +
                         operands * s.of[0].megabyte + results * s.of[0].results;
        if (best < 0 || t < least) best = i, least = t;
    }
    // (its kind: as ops/kernels.py:moe_wide has it, by the groups of the list)
    const MtRows &r = mt_rows[group != 8 ? 2 : ((N + 255) / 256) * (2 * (list / 8) - experts) > 576 ? 0 : 1];
    const MtSpread blocks = mt_spread(slots, experts, top, r.rows);
    const double columns = (N + r.outs - 1) / r.outs, even = fmax(1.0, blocks.mean * columns / (2 * MT_UNITS));
    const double rows = mt_turns(blocks, columns, 2 * MT_UNITS) * stages * r.stage +
                        even * (r.even + stages * r.even_stage + mt_act_rows[act] * r.rows * r.outs / halves / 256) +
                        mt_turns(blocks, columns, MT_UNITS) * (r.single + stages * r.single_stage) + operands * r.megabyte + results * r.results;
    return least <= 0.97 * rows ? best : -1;
}

// Which shape is expected to be fastest for `slots` of `experts`, of which a token takes `top`; -1: sizes the kernel does not take, or
// moe_expert_rows in groups of `group` tiles, two workgroups a unit, of which one writes or activates while the other multiplies, is expected to be faster.
// Second product: results in 32 bits are as long to write as a short K to multiply, and with one workgroup a unit nothing multiplies
// meanwhile.  8,192 slots of 4 experts of 2,048 x 1,024 38 / 40, 12,000 54 / 61; of 16 of 2,048 x 768 56 / 46, where moe_expert_rows' workgroups
// are just more than the units hold at once.  So only where a tenth less than there is expected, from the same sizes.
extern "C" int kva_moe_tiles_plan(int slots, int experts, int top, int N, int K, int second, int act, int gated, int group) {
    // (tiles: of a list in groups of eight, which the other product may need)
    const long long list = (slots + 127ll * experts + 127) / 128 * 8;
    if (slots <= 0 || experts <= 0 || top <= 0 || act < MT_ACT_SILU || act > MT_ACT_RELU2 || !mt_sizes(list, experts, N, K)) return -1;
    if (!second) return mt_first(slots, experts, top, N, K, act, gated, group, list);
    const double operands = 2e-6 * K * ((double)N * experts + slots), results = 4e-6 * slots * N, stages = K / MT_STAGE;
    int best = -1;
    double least = 0.0;
    for (int i = 0; i < MT_COUNT; ++i) {
        const auto &s = mt_shapes[i].of[1];
        const double turns = ceil(mt_blocks(slots, experts, top, mt_shapes[i].rows, N, mt_shapes[i].outs) / MT_UNITS);
        const double t = turns * (s.turn + stages * s.stage) + operands * s.megabyte + results * s.results;
        if (best < 0 || t < least) best = i, least = t;
    }
    if (slots < 160ll * experts) return K < 1280 ? -1 : best;
    // (moe_expert_rows' workgroups of the larger kind: past 288 of them they are taken, and below half as many outputs a workgroup)
    const double wide = mt_blocks(slots, experts, top, 128, N, 256);
    const double rows = wide > 288 ? ceil(wide / 512) * stages * 1.161 + operands * 0.175 + results * 0.193
                                   : ceil(mt_blocks(slots, experts, top, 128, N, 128) / 512) * (6.41 + stages * 0.207) + operands * 0.078 + results * 0.348;
    return least <= 0.9 * rows ? best : -1;
}

// x [tokens, K] (first product) or [places, K] (second), w [experts, N, K] in operand order; out bf16 [places, N] ([places, N / 2] gated) or
// (second) fp32 [slots, N]; all at multiples of 16 bytes, and the list in tiles of 16 without groups.
extern "C" int kva_moe_tiles(void *out, const void *x, const void *w, const int *sorted_slot, const int *tile_expert, const float *slot_weight,
                             int max_tiles, int experts, int top, int N, int K, int second, int act, int gated, float limit, int plan,
                             hipStream_t stream) {
    KVA_REQUIRE(mt_sizes(max_tiles, experts, N, K), "moe_tiles: no product of %d tiles of %d experts, %d outputs of %d inputs", max_tiles, experts, N, K);
    KVA_REQUIRE(plan >= 0 && plan < MT_COUNT && top > 0, "moe_tiles: plan %d, %d choices", plan, top);
    KVA_REQUIRE(act >= MT_ACT_SILU && act <= MT_ACT_RELU2 && (act != MT_ACT_SWISH_CLAMPED || gated) && !(gated && second),
                "moe_tiles: activation %d, gated %d, second product %d", act, gated, second);
    KVA_REQUIRE(out && x && w && sorted_slot && tile_expert, "moe_tiles: missing operand");
    KVA_REQUIRE((((uintptr_t)out | (uintptr_t)x | (uintptr_t)w) & 15) == 0, "moe_tiles: operands must be at multiples of 16 bytes");
    const int per = mt_shapes[plan].rows / MT_TILE;
    // (every expert's last block may hold less than `per` tiles)
    const long long blocks = (long long)((max_tiles + per - 1) / per + (experts < max_tiles ? experts : max_tiles)) *
                             ((N + mt_shapes[plan].outs - 1) / mt_shapes[plan].outs);
    KVA_REQUIRE(blocks <= 0x7fffffffll, "moe_tiles: too many workgroups");
    const MtArgs a{(const bf16_t *)x, (const bf16_t *)w, out, sorted_slot, tile_expert, slot_weight, max_tiles, top, N, K, second, act, limit};
#define MT_LAUNCH(ID, RT, NT, WR, WN, WK, KSUB, ST, ...)                                                                     \
    case ID: {                                                                                                               \
        typedef TileProduct<RT, NT, WR, WN, WK, KSUB, ST> P;                                                                 \
        if (gated) hipLaunchKernelGGL((moe_tiles_kernel<P, true>), dim3(blocks), dim3(P::THREADS), 0, stream, a);            \
        else hipLaunchKernelGGL((moe_tiles_kernel<P, false>), dim3(blocks), dim3(P::THREADS), 0, stream, a);                 \
        break;                                                                                                               \
    }
    switch (plan) { MT_SHAPES(MT_LAUNCH) }
#undef MT_LAUNCH
    KVA_CHECK_LAUNCH("moe_tiles");
    return KVA_OK;
}
