// The experts' products of a prompt (moe.hip says what the list of slots is) over tiles of 64 x 64 to 256 x 256 (tile_product.h),
// for matrices in operand order whose K is a multiple of 64.
//
// The list has its slots in tiles of 16 by expert, and a workgroup takes up to G neighbouring tiles of one expert: where a block of
// G begins is worked out from the tiles' experts by every wavefront for itself, so one list serves both products in blocks of
// different heights.  (Lists in groups of G = 8, as moe.hip's kernel takes them, fix the height and pad every expert to it.)
//
// What bounds it: up to 2,000 tokens one or two turns of the units, a stage of 256 x 256 x 64 some 1.3 us of matrix products and loads,
// and around them the first operands' way from memory and the results' to it.  Before (moe.hip's 128 x 256, two workgroups a unit) and
// now, in the model, us: 2,048 tokens, 4 of 16 experts of 1,536 x 2,048 68 / 62 (830 TFLOP/s), of 2,048 x 768 58 / 48; all of 4
// of 1,024 x 2,048 with erf-gelu 49.5 / 46; 2,494 tokens, all of 4 of 1,536 x 2,048 65 / 62.
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
// 64 elements of K, and a megabyte of operands, for the first product and, with a megabyte of results, for the second.  Fitted to the
// timings of nine shapes over 45 sizes of either product: 100 to 6,000 tokens, 4 to 64 experts, 512 to 4,096 wide; the shape they
// choose is 2 % (first) and 4 % (second) behind the best of the nine on average.
struct MtShape {
    int rows, outs;
    struct {
        float turn, stage, megabyte, results;
    } of[2];
};
#define MT_SHAPES(V)                                                                          \
    V(0, 8, 4, 2, 4, 1, 2, 2, 3.04f, 1.283f, 0.074f, 0.f, 3.13f, 1.411f, 0.029f, 0.205f)      \
    V(1, 4, 8, 2, 2, 1, 2, 3, 1.56f, 0.852f, 0.066f, 0.f, 2.58f, 0.842f, 0.063f, 0.208f)      \
    V(2, 4, 4, 2, 2, 2, 1, 4, 3.37f, 0.502f, 0.061f, 0.f, 0.45f, 0.556f, 0.079f, 0.402f)      \
    V(3, 5, 4, 2, 4, 1, 2, 3, 4.81f, 0.899f, 0.018f, 0.f, 0.98f, 1.025f, 0.031f, 0.251f)      \
    V(4, 5, 4, 2, 2, 2, 1, 4, 6.02f, 0.532f, 0.031f, 0.f, 2.72f, 0.481f, 0.043f, 0.405f)      \
    V(5, 3, 4, 2, 2, 2, 1, 4, 0.00f, 0.552f, 0.053f, 0.f, 0.00f, 0.606f, 0.031f, 0.410f)      \
    V(6, 6, 4, 2, 4, 1, 2, 2, 10.56f, 0.864f, 0.052f, 0.f, 5.87f, 0.900f, 0.043f, 0.219f)     \
    V(7, 2, 2, 2, 2, 2, 1, 8, 3.05f, 0.291f, 0.000f, 0.f, 0.00f, 0.262f, 0.115f, 1.008f)      \
    V(8, 4, 2, 2, 2, 2, 1, 6, 4.27f, 0.354f, 0.011f, 0.f, 1.04f, 0.350f, 0.080f, 0.577f)
#define MT_COUNT 9
#define MT_BOTH(a, b, c, d, e, f, g, h) {a, b, c, d}, {e, f, g, h}
static const MtShape mt_shapes[MT_COUNT] = {
#define MT_ROW(ID, RT, NT, WR, WN, WK, KSUB, ST, ...) {16 * RT * WR, 16 * NT * WN, {MT_BOTH(__VA_ARGS__)}},
    MT_SHAPES(MT_ROW)
#undef MT_ROW
};
#define MT_UNITS 256
#define MT_STAGE 64

static bool mt_sizes(long long tiles, int experts, int N, int K) {
    return tiles > 0 && tiles <= MT_MAX_TILES && experts > 0 && N > 0 && N % 16 == 0 && K >= MT_STAGE && K % MT_STAGE == 0 &&
           (long long)N * K * 2 <= 0x7fffffffll && tiles * MT_TILE * K * 2 <= 0x7fffffffll;
}

// (experts that all tokens take have as many rows each; else every expert's last block is half full on average)
static double mt_blocks(double slots, int experts, int top, int rows, int N, int outs) {
    return ceil(top == experts ? experts * ceil(slots / experts / rows) : slots / rows + 0.5 * experts) * ((N + outs - 1) / outs);
}

// Which shape is expected to be fastest for `slots` of `experts`, of which a token takes `top`; -1: sizes the kernel does not take, or
// moe_expert_rows is expected to be faster, two workgroups a unit, of which one writes while the other multiplies.
// First product (us, moe_expert_rows / here, matrices from memory): 8,192 slots of 16 experts of 1,536 x 2,048 68.6 / 60.6, of 4
// experts of 1,024 x 2,048 43.6 / 40.7, 1,024 slots of 4 24.1 / 15.8, 4,000 of 16 50.5 / 36.7; 0.84 on average.  Not where many turns even out
// what a turn costs: 12,288 slots of 64 experts of 2,816 x 2,048 212 / 241, 16,384 of 4 of 1,536 x 2,048 94 / 103 (but 8,000 of 8 of 7,168 x
// 4,096 726 / 482).
// Second: results in 32 bits are as long to write as a short K to multiply, and with one workgroup a unit nothing multiplies
// meanwhile.  8,192 slots of 4 experts of 2,048 x 1,024 38 / 40, 12,000 54 / 61; of 16 of 2,048 x 768 56 / 46, where moe_expert_rows' workgroups
// are just more than the units hold at once.  So only where a tenth less than there is expected, from the same sizes.
extern "C" int kva_moe_tiles_plan(int slots, int experts, int top, int N, int K, int second) {
    // (tiles: of a list in groups of eight, which the other product may need)
    if (slots <= 0 || experts <= 0 || top <= 0 || !mt_sizes((slots + 127ll * experts + 127) / 128 * 8, experts, N, K)) return -1;
    const double operands = 2e-6 * K * ((double)N * experts + slots), results = 4e-6 * slots * N, stages = K / MT_STAGE;
    int best = -1;
    double least = 0.0;
    for (int i = 0; i < MT_COUNT; ++i) {
        const auto &s = mt_shapes[i].of[second ? 1 : 0];
        const double turns = ceil(mt_blocks(slots, experts, top, mt_shapes[i].rows, N, mt_shapes[i].outs) / MT_UNITS);
        const double t = turns * (s.turn + stages * s.stage) + operands * s.megabyte + results * s.results;
        if (best < 0 || t < least) best = i, least = t;
    }
    const double wide = mt_blocks(slots, experts, top, 128, N, 256);        // moe_expert_rows' workgroups, the larger kind
    if (!second) return wide > 700 && K < 3072 ? -1 : best;
    if (slots < 160ll * experts) return K < 1280 ? -1 : best;
    // (past 288 of them they are taken, and below half as many outputs a workgroup)
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
