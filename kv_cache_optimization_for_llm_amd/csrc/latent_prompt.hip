// Attention over low-rank entries for prompts: keys and values expanded (bf16, gfx950).
//
// latent_attention_mfma.hip attends over the cached rows themselves - rank + rot elements a key, rank a value, for
// every head - which is what a decoded token wants: each row is read once for all heads.  A prompt's tokens see
// the same keys many times over, and per (token, key, head) that form costs 2 (rank + rot + rank) operations against
// 2 (dim + rot + vdim) over keys and values expanded per head: 2,176 against 640 at rank 512 and heads of
// 128 + 64 / 128.  Expanding a key costs 2 rank (dim + vdim) per head once, as much as 85 tokens looking at it save.
// Two kernels:
//   * latent_expand_kernel: the entries' whole contexts (cached rows, by page) times [U_k ; U_v], rounded to
//     bf16, written head by head in tiles of 16 keys or 32 keys' values in the order in which the products below read them; the rotated
//     key parts, which all heads share, are laid in such tiles in the same launch.  128 x 256 a workgroup, 128 x 128 where that is one
//     a compute unit or less (64 / 2,048 tokens of 16 heads 10.1 -> 7.7 / 16.3 -> 15.9 us; 4,096 tokens, 512 workgroups, 23.0 against 28.6).
//   * latent_prompt_kernel: a workgroup takes 64 tokens of an entry and one head (latent_prompt_form says how its wavefronts share them).
//     As in latent_attention_mfma.hip everything is transposed, S^T = K Q^T and O^T = V^T P^T.  Blocks of keys are copied to LDS as they
//     lie (buffer loads to LDS), the next one on its way; products and vector work of a block are a barrier apart.  The
//     queries' rotation happens as they are loaded, sink and output gate where the result is normalised.
// A SIMD issues matrix products (20 of 16 cycles a block of 32 keys and 16 tokens) or the softmax's vector work (about as much); with 1 to 3
// wavefronts a SIMD the chain of one block, reads, products, maximum, exponentials, products, is what is waited for.  The workgroups with
// the most keys are launched first; a head's workgroups are on one die where the heads are a multiple of eight, whose L2
// holds its keys and values.
//
// us a layer, one prompt of 2,048 tokens, 16 heads of 128 + 64 / 128, rank 512: over the cached rows 183, the products
// per head in front and behind 38 + 21; expanded 16 + 49 (16 + 58 through registers; 21.5 GFLOP in the second: 440 TFLOP/s).
#include "common.h"
#include "lds_product.h"
#include <math.h>
#include <type_traits>

#define LP_LOG2E 1.44269504088896340736f
#define LP_DIM 128                  // a head's plain query / key elements, rotated ones, values
#define LP_ROT 64
#define LP_VDIM 128
#define LP_ROWS 64                  // tokens a workgroup
#define LP_OUT (LP_VDIM + 4)        // floats of a row of results in LDS
static_assert(LP_DIM == LP_VDIM, "expanded keys and values lie in rows of one size");
struct LatentPrompt {
    bf16_t *out;                    // [T, heads * vdim]
    const bf16_t *q;                // token t, head h: LP_DIM plain elements, then LP_ROT to be rotated, at t q_row + h q_head
    const bf16_t *cache;            // [pages, page_size, rank + rot]
    const bf16_t *w;                // [heads (dim + vdim), rank] in operand order: all heads' U_k, then all heads' U_v
    bf16_t *kv, *rot;               // expanded: [entries, keys' heads then values' heads, context, 128] and [entries * context, rot]
    const int *block_table, *entry_seat, *entry_q_start, *entry_start_pos;
    const float *cos, *sin, *sinks; // tables [positions, rot / 2]; one number a head, or none
    const bf16_t *gates;            // or none: one a head at t gate_row + h, or one an element at t gate_row + h gate_head + i
    int q_row, q_head, gate_row, gate_head, gate_per_element;
    int max_blocks, page_size, heads, rank, context, interleaved;
    float scale;
};

// 8 keys of value element 16 dt + r as the second product's operand (see latent_attention_mfma.hip: lat_values)
typedef __attribute__((address_space(3))) s16x4 lp_lds_s16x4;
template <int STRIDE>
__device__ __forceinline__ Frag8 lp_values(const bf16_t *at, int dt) {
    union { s16x4 t[2]; Frag8 f; } u;
    u.t[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp_lds_s16x4 *)(at + 16 * dt));
    u.t[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp_lds_s16x4 *)(at + 16 * STRIDE + 16 * dt));
    return u.f;
}

template <int NT>
__global__ void __launch_bounds__(256, NT == 8 ? 2 : 3)
latent_expand_kernel(LatentPrompt a) {
    typedef LdsProduct<4, NT, 3> Product;
    constexpr int STRIDE = Product::OUTS + 8;
    __shared__ __align__(16) union {
        typename Product::Shared operands;
        bf16_t results[Product::ROWS * STRIDE];
    } shared;
    const int e = blockIdx.y, keys = a.entry_start_pos[e] + a.entry_q_start[e + 1] - a.entry_q_start[e];
    const int N = a.heads * (LP_DIM + LP_VDIM), n_blocks = N / Product::OUTS, total = (keys + Product::ROWS - 1) / Product::ROWS * n_blocks;
    if ((int)blockIdx.x >= total) return;
    const int id = die_order(blockIdx.x, total), m0 = id / n_blocks * Product::ROWS, n0 = id % n_blocks * Product::OUTS;
    const int *bt = a.block_table + (size_t)a.entry_seat[e] * a.max_blocks;
    const int KD = a.rank + LP_ROT;
    auto cached = [&](int p) {                              // (positions of an entry are all mapped)
        p = min(p, keys - 1);
        return a.cache + ((size_t)max(bt[p / a.page_size], 0) * a.page_size + p % a.page_size) * KD;
    };
    const size_t base = (size_t)e * a.context;
    if (n0 == 0)
        for (int x = threadIdx.x; x < Product::ROWS * LP_ROT / 8; x += 256) {
            const int p = m0 + x / (LP_ROT / 8), c = x % (LP_ROT / 8) * 8;
            if (p < keys)
                *reinterpret_cast<uint4 *>(a.rot + (base + p / 16 * 16) * LP_ROT + 16 * c + 8 * (p % 16)) = *reinterpret_cast<const uint4 *>(cached(p) + a.rank + c);
        }
    Product p;
#pragma unroll
    for (int i = 0; i < Product::XI; ++i) p.xp[i] = cached(m0 + p.row(i)) + p.element();
    p.tiled_w(a.w, N, a.rank, n0);
    f32x4 acc[NT][4];
    p.run(shared.operands, a.rank, acc);
    const int lane = threadIdx.x % KVA_WAVE, wave = threadIdx.x / KVA_WAVE, r = lane & 15, g = lane >> 4;
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            Frag4 f;
            const b16x2 lo = pack_bf16(acc[nt][rt][0], acc[nt][rt][1]), hi = pack_bf16(acc[nt][rt][2], acc[nt][rt][3]);
            f.u2 = make_uint2(__builtin_bit_cast(unsigned, lo), __builtin_bit_cast(unsigned, hi));
            *reinterpret_cast<uint2 *>(&shared.results[((wave & 1) * 64 + 16 * rt + r) * STRIDE + (wave >> 1) * (16 * NT) + 16 * nt + 4 * g]) = f.u2;
        }
    __syncthreads();
    // In the order in which the products read them: 16 keys [8 elements][key], 4 KiB; values of 32 keys [16 elements][lane][its 8 keys of
    // one element], 8 KiB.
#pragma unroll
    for (int half = 0; half < Product::OUTS / LP_DIM; ++half) {
        const int h = n0 / LP_DIM + half;
        bf16_t *to = a.kv + (((size_t)e * 2 * a.heads + h) * a.context + m0) * LP_DIM;
        const bf16_t *from = shared.results + half * LP_DIM;
        if (h < a.heads) {
#pragma unroll
            for (int x = 0; x < Product::ROWS / 16; ++x)
                if (m0 + 16 * x < keys)
                    *reinterpret_cast<uint4 *>(to + (256 * x + threadIdx.x) * 8) =
                        *reinterpret_cast<const uint4 *>(from + (16 * x + threadIdx.x % 16) * STRIDE + threadIdx.x / 16 * 8);
        } else {
#pragma unroll
            for (int x = 0; x < Product::ROWS / 16; ++x)
                if (m0 + x / 2 * 32 < keys)
                    *reinterpret_cast<uint4 *>(to + (256 * x + threadIdx.x) * 8) =
                        lp_values<STRIDE>(from + (x / 2 * 32 + 4 * g + (r >> 2)) * STRIDE + 4 * (r & 3), x % 2 * 4 + wave).u4;
        }
    }
}

// a query's rotated part: pairs of neighbours, or of elements 32 apart (which the same lane holds)
struct LpTurn {
    float c[8], n[8];
    __device__ __forceinline__ void load(const float *cos, const float *sin, int g, bool interleaved) {
        const int lo = interleaved ? 4 * g : 8 * g, hi = interleaved ? 16 + 4 * g : 8 * g + 4;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            c[i] = cos[i < 4 ? lo + i : hi + i - 4];
            n[i] = sin[i < 4 ? lo + i : hi + i - 4];
        }
    }
    __device__ __forceinline__ void apply(Frag8 &a, Frag8 &b, bool interleaved) const {
        Frag8 x, y;                     // first elements of the pairs, second ones
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float u = bf16_bits_to_float(interleaved ? (i < 4 ? a : b).h[i % 4 * 2] : a.h[i]);
            const float v = bf16_bits_to_float(interleaved ? (i < 4 ? a : b).h[i % 4 * 2 + 1] : b.h[i]);
            x.h[i] = float_to_bf16_bits(u * c[i] - v * n[i]);
            y.h[i] = float_to_bf16_bits(v * c[i] + u * n[i]);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            a.h[i] = interleaved ? (i % 2 ? y : x).h[i / 2] : x.h[i];
            b.h[i] = interleaved ? (i % 2 ? y : x).h[4 + i / 2] : y.h[i];
        }
    }
};

#define LP_SLOTS 2                  // blocks of keys that LDS holds

// A workgroup of GROUPS x PARTS wavefronts, each with 16 RT of its 64 tokens (wave % GROUPS) and 32 keys (wave / GROUPS) of every 32 PARTS that
// come through LDS; what the PARTS found is added up at the end.
template <int RT, int GROUPS, int PARTS>
__device__ __forceinline__ void latent_prompt_tile(const LatentPrompt &a, bf16_t *lds, const int e, const int head, const int tile) {
    constexpr int KD = LP_DIM + LP_ROT, KS = KD / 32, NDT = LP_VDIM / 16, WAVES = GROUPS * PARTS;
    static_assert(16 * RT * GROUPS == LP_ROWS, "64 tokens a workgroup");
    constexpr int ROWS = LP_ROWS, BLOCK = 32 * PARTS, TILES = 2 * PARTS, SLOTS = LP_SLOTS;
    constexpr int KTILE = 16 * KD, VTILE = 32 * LP_VDIM;        // elements in LDS of 16 keys, of 32 keys' values
    constexpr int SHARE = WAVES / TILES, VSHARE = WAVES / PARTS;        // wavefronts that fetch a tile together
    constexpr int LOADS = 6 / SHARE + 8 / VSHARE;               // a wavefront's of a block, 1 KiB each
    bf16_t *const ks = lds, *const vs = lds + SLOTS * TILES * KTILE;
    const int q0 = a.entry_q_start[e], n = a.entry_q_start[e + 1] - q0, start = a.entry_start_pos[e];
    if (tile * ROWS >= n) return;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / KVA_WAVE), lane = tid % KVA_WAVE, r = lane & 15, g = lane >> 4;
    const int rows = wave % GROUPS, keys = wave / GROUPS;
    const int first = tile * ROWS + 16 * RT * rows;             // the wavefront's first token
    int mine[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) mine[rt] = min(first + 16 * rt + r, n - 1);
    const int hi = first < n ? start + min(first + 16 * RT - 1, n - 1) : -1;    // newest key of the wavefront's tokens, and of the workgroup's
    const int end = start + min(tile * ROWS + ROWS, n);                 // (one past it)

    // A wavefront's part of a block's tiles, to the slot of its turn.  Tiles past the entry's last one are that one again: its
    // keys there are past every token's.
    const int last = start + n - 1;
    const bf16_t *k_from = a.kv + ((size_t)e * 2 * a.heads + head) * a.context * LP_DIM, *r_from = a.rot + (size_t)e * a.context * LP_ROT;
    const bf16_t *v_from = k_from + (size_t)a.heads * a.context * LP_DIM;
    auto pieces = [&](const bf16_t *from, auto kib, bf16_t *to, int part) {     // so many KiB, `part` of those that each fetch as many
        const Buffer buffer = buffer_at(from + part * decltype(kib)::value * 512, decltype(kib)::value * 1024);
#pragma unroll
        for (int i = 0; i < decltype(kib)::value; ++i) buffer_to_lds(buffer, 16 * lane, 1024 * i, to + 512 * (part * decltype(kib)::value + i));
    };
    auto fetch_keys = [&](int block) {
        const int its = wave / SHARE;
        const size_t t = min(TILES * block + its, last / 16);
        bf16_t *to = ks + (block % SLOTS * TILES + its) * KTILE;
        pieces(k_from + t * (16 * LP_DIM), std::integral_constant<int, 4 / SHARE>{}, to, wave % SHARE);
        pieces(r_from + t * (16 * LP_ROT), std::integral_constant<int, 2 / SHARE>{}, to + 16 * LP_DIM, wave % SHARE);
    };
    auto fetch_values = [&](int block) {
        const int its = wave / VSHARE;
        pieces(v_from + (size_t)min(PARTS * block + its, last / 32) * VTILE, std::integral_constant<int, 8 / VSHARE>{},
               vs + (block % SLOTS * PARTS + its) * VTILE, wave % VSHARE);
    };

    // (a scale below zero as turned queries: the largest score is then the largest product.  Zero: all probabilities alike)
    const float scale2 = fmaxf(fabsf(a.scale), 1e-30f) * LP_LOG2E, rebase = 8.f / scale2;
    const unsigned sign = a.scale < 0.f ? 0x80008000u : 0u;
    Frag8 qf[RT][KS];
    LpTurn turn[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const bf16_t *q = a.q + (size_t)(q0 + mine[rt]) * a.q_row + (size_t)head * a.q_head + 8 * g;
#pragma unroll
        for (int i = 0; i < KS; ++i) qf[rt][i].u4 = *reinterpret_cast<const uint4 *>(q + 32 * i);
        const size_t table = (size_t)(start + mine[rt]) * (LP_ROT / 2);
        turn[rt].load(a.cos + table, a.sin + table, g, a.interleaved != 0);
    }
    const int blocks = (end + BLOCK - 1) / BLOCK;               // uniform over the workgroup
    fetch_keys(0);
#pragma unroll
    for (int b = 1; b < SLOTS; ++b) {
        if (b < blocks) fetch_keys(b);
        if (b - 1 < blocks) fetch_values(b - 1);
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
        for (int i = 0; i < KS; ++i) qf[rt][i].u4 = make_uint4(qf[rt][i].u4.x ^ sign, qf[rt][i].u4.y ^ sign, qf[rt][i].u4.z ^ sign, qf[rt][i].u4.w ^ sign);
        turn[rt].apply(qf[rt][KS - 2], qf[rt][KS - 1], a.interleaved != 0);
    }
    f32x4 o[RT][NDT];
    float m[RT], l[RT];                                         // m of the products, l this lane's part
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        m[rt] = -INFINITY, l[rt] = 0.f;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) o[rt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // The products of a block: those of its scores, and a turn later those with its values.  Between them their vector work.
    auto key_of = [&](int block) { return block * BLOCK + 32 * keys; };
    auto cut_of = [&](int block) { return key_of(block) + 31 > start + first; };        // some of the tokens do not see some of the keys
    f32x4 s[RT][2];
    Frag8 pf[RT];
    b16x8 kf[2][KS], vf[NDT];
    auto read_keys = [&](int block, int t) {
        const bf16_t *kp = ks + (block % SLOTS * TILES + 2 * keys + t) * KTILE + 8 * lane;
#pragma unroll
        for (int i = 0; i < KS; ++i) kf[t][i] = *reinterpret_cast<const b16x8 *>(kp + 512 * i);
    };
    auto score = [&](int t) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) s[rt][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < KS; ++i)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) s[rt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[t][i], qf[rt][i].v, s[rt][t], 0, 0, 0);
    };
    // (operands are read well in front of their products: the wavefronts of a phase ask LDS for theirs at the same time)
    auto scores = [&](int block) {
        read_keys(block, 0);
        read_keys(block, 1);
        __builtin_amdgcn_sched_barrier(0);
        score(0);
        score(1);
    };
    auto weigh = [&](int block) {
        if (cut_of(block)) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) s[rt][t][i] = key_of(block) + 16 * t + 4 * g + i <= start + mine[rt] ? s[rt][t][i] : -INFINITY;
        }
        float mx[RT];
        bool moves = false;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            mx[rt] = -INFINITY;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) mx[rt] = fmaxf(mx[rt], s[rt][t][i]);
            moves = moves || mx[rt] > m[rt] + rebase;
        }
        // (the reference of the exponentials moves only when a maximum has grown by more than 2^8)
        if (__builtin_amdgcn_ballot_w64(moves) != 0) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const float m_new = fmaxf(m[rt], quad_rows_max(mx[rt]));
                const float corr = __builtin_amdgcn_exp2f((m[rt] - ((m_new == -INFINITY) ? 0.f : m_new)) * scale2);     // exp2(-inf) = 0
                l[rt] *= corr;
#pragma unroll
                for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                    for (int c = 0; c < 4; ++c) o[rt][dt][c] *= corr;
                m[rt] = m_new;
            }
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const float ref = m[rt] == -INFINITY ? 0.f : -m[rt] * scale2;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float p0 = __builtin_amdgcn_exp2f(fmaf(s[rt][j / 2][j % 2 * 2], scale2, ref));
                const float p1 = __builtin_amdgcn_exp2f(fmaf(s[rt][j / 2][j % 2 * 2 + 1], scale2, ref));
                l[rt] += p0 + p1;
                pf[rt].p2[j] = pack_bf16(p0, p1);
            }
        }
    };
    // A portion that starts up to 16 positions behind a multiple of 32 has one block of keys that the wavefront's last 16 tokens see and
    // the first 16 do not.  A probability of zero does not leave out a value that is not a number: they get zeros for it, and all of
    // them for keys past the workgroup's newest one, whose places may hold anything.
    auto read_values = [&](int block) {
        const bf16_t *get = vs + (block % SLOTS * PARTS + keys) * VTILE + 8 * lane;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) vf[dt] = *reinterpret_cast<const b16x8 *>(get + 512 * dt);
    };
    auto add = [&](auto cut_tag, int block) {
        constexpr bool CUT = decltype(cut_tag)::value;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
            Frag8 v;
            v.v = vf[dt];
            if (CUT) {
                v.u2[0] = keep_first_keys(v.u2[0], end - key_of(block) - 4 * g);
                v.u2[1] = keep_first_keys(v.u2[1], end - key_of(block) - 16 - 4 * g);
            }
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                Frag8 f = v;
                if (CUT && rt < RT - 1) {
                    const unsigned seen = key_of(block) <= start + first + 16 * rt + 15 ? ~0u : 0u;
                    f.u4 = make_uint4(v.u4.x & seen, v.u4.y & seen, v.u4.z & seen, v.u4.w & seen);
                }
                o[rt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.v, pf[rt].v, o[rt][dt], 0, 0, 0);
            }
        }
    };
    // Of eight wavefronts the second four, one beside each of the first on its SIMD, are a barrier behind: they have their vector work
    // while the first have their products.  (What a wavefront fetches its four read.)
    if (SLOTS <= blocks) wait_and_meet<(SLOTS - 1) * LOADS>();
    else wait_and_meet<0>();
    if (WAVES == 8 && wave >= 4) wait_and_meet<63>();
    if (key_of(0) <= hi) scores(0);
    for (int block = 0; block < blocks; ++block) {
        wait_and_meet<63>();                                    // the keys, and the values of the block before, are read
        if (block + SLOTS < blocks) fetch_keys(block + SLOTS);
        if (block + SLOTS - 1 < blocks) fetch_values(block + SLOTS - 1);
        if (key_of(block) <= hi) weigh(block);
        // its values and the next keys are there (near the end, where fewer are on their way: all that are)
        if (block + SLOTS < blocks) wait_and_meet<(SLOTS - 1) * LOADS>();
        else wait_and_meet<0>();
        const bool next = block + 1 < blocks && key_of(block + 1) <= hi;
        if (next && !cut_of(block)) {
            read_values(block);
            read_keys(block + 1, 0);
            __builtin_amdgcn_sched_barrier(0);
            add(std::false_type{}, block);
            read_keys(block + 1, 1);
            score(0);
            score(1);
        } else {
            if (key_of(block) <= hi) {
                read_values(block);
                add(std::true_type{}, block);
            }
            if (next) scores(block + 1);
        }
    }
    if (WAVES == 8 && wave < 4) wait_and_meet<0>();
    wait_and_meet<0>();                                         // nobody reads any more

    // Results, and in base 2 what they are relative to, through LDS: the parts of 8 elements of a token are added up by one thread.
    float *const at_o = reinterpret_cast<float *>(lds), *const at_m = at_o + PARTS * ROWS * LP_OUT, *const at_l = at_m + PARTS * ROWS;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int row = keys * ROWS + 16 * RT * rows + 16 * rt + r;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) *reinterpret_cast<f32x4 *>(at_o + row * LP_OUT + 16 * dt + 4 * g) = o[rt][dt];
        const float sum = quad_rows_sum(l[rt]);
        if (g == 0) at_m[row] = m[rt] * scale2, at_l[row] = sum;
    }
    __syncthreads();
#pragma unroll 1
    for (int x = tid; x < ROWS * (LP_VDIM / 8); x += 64 * WAVES) {
        const int row = x / (LP_VDIM / 8), c = x % (LP_VDIM / 8) * 8, t = q0 + tile * ROWS + row;
        if (tile * ROWS + row >= n) break;                      // (later ones are past it too)
        float both = at_m[row], scales[PARTS], sum = 0.f, v[8];
#pragma unroll
        for (int p = 1; p < PARTS; ++p) both = fmaxf(both, at_m[p * ROWS + row]);
        const float ref = both == -INFINITY ? 0.f : both;
#pragma unroll
        for (int p = 0; p < PARTS; ++p) {
            scales[p] = __builtin_amdgcn_exp2f(at_m[p * ROWS + row] - ref);
            sum += at_l[p * ROWS + row] * scales[p];
        }
        float mul = 1.f / sum;
        if (a.sinks) {                                          // one more term of the denominator, with no key and no value
            const float sk = a.sinks[head] * LP_LOG2E, m_new = fmaxf(both, sk), corr = __builtin_amdgcn_exp2f(both - m_new);
            mul = corr / (sum * corr + __builtin_amdgcn_exp2f(sk - m_new));
        }
        const bf16_t *gate = a.gates ? a.gates + (size_t)t * a.gate_row : nullptr;
        if (gate && !a.gate_per_element) mul *= 1.f / (1.f + expf(-to_float(gate[head])));
#pragma unroll
        for (int i = 0; i < 8; i += 4) {
            f32x4 y = *reinterpret_cast<const f32x4 *>(at_o + row * LP_OUT + c + i) * scales[0];
#pragma unroll
            for (int p = 1; p < PARTS; ++p) y += *reinterpret_cast<const f32x4 *>(at_o + (p * ROWS + row) * LP_OUT + c + i) * scales[p];
            v[i] = y[0] * mul, v[i + 1] = y[1] * mul, v[i + 2] = y[2] * mul, v[i + 3] = y[3] * mul;
        }
        if (gate && a.gate_per_element)
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] *= 1.f / (1.f + expf(-to_float(gate[(size_t)head * a.gate_head + c + i])));
        bf16_t *out = a.out + ((size_t)t * a.heads + head) * LP_VDIM + c;
#pragma unroll
        for (int i = 0; i < 8; i += 4) {
            const b16x2 lo = pack_bf16(v[i], v[i + 1]), hi2 = pack_bf16(v[i + 2], v[i + 3]);
            *reinterpret_cast<uint2 *>(out + i) = make_uint2(__builtin_bit_cast(unsigned, lo), __builtin_bit_cast(unsigned, hi2));
        }
    }
}

// (three workgroups of 16 tokens a wavefront fit a compute unit's registers, two of 32)
template <int RT, int GROUPS, int PARTS>
__global__ void __launch_bounds__(64 * GROUPS * PARTS, RT == 1 ? 3 : 2)
latent_prompt_kernel(LatentPrompt a, int tiles) {
    constexpr int RING = LP_SLOTS * PARTS * 32 * (LP_DIM + LP_ROT + LP_VDIM), RESULTS = PARTS * 16 * RT * GROUPS * (LP_OUT + 2) * 2;
    __shared__ __align__(16) bf16_t lds[RING > RESULTS ? RING : RESULTS];
    // (the longest first)
    latent_prompt_tile<RT, GROUPS, PARTS>(a, lds, blockIdx.y, blockIdx.x % a.heads, tiles - 1 - (int)(blockIdx.x / a.heads));
}

extern "C" int kva_latent_prompt_supported(int dim, int rot, int vdim, int rank) {
    return dim == LP_DIM && rot == LP_ROT && vdim == LP_VDIM && rank > 0 && rank % LDSP_K == 0;
}

// How a workgroup's wavefronts share its 64 tokens and the keys.  A block of keys is a chain of waits, products and vector work, 1.2 us for a
// wavefront with its SIMD to itself, 0.6 where three interleave.  With more workgroups than the chip takes at once, and with few blocks of
// keys, four wavefronts of 16 tokens (three workgroups a compute unit); with fewer, 32 tokens by two parts of the keys, which read LDS
// half as often; with one workgroup a compute unit or less, or up to two and long contexts, whose longest one all wait for, four parts.
// four of 16 tokens / two parts / four parts, us with the expansion, rank 512 (in brackets: through registers on the way to LDS, 16
// tokens a wavefront, or two parts up to 512 workgroups in contexts above 1,024):
//   one entry of 16 heads from position 0: 64 tokens 15/16/19 (16.5)  256 20/21/23 (22)  512 28/28/28 (30)  1,000 (256 workgroups)
//   40/37/36 (44)  1,400 (352) 53/50/48 (56)  2,048 (512) 69/65/64 (72)  3,000 (752) 101/91/107 (116)  4,096 (1,024) 141/136/155 (163)  8,000
//   424/421/465 (530);  of 8 heads 2,048 (256) 65/55/46 (68)  4,096 (512) 114/99/85 (114);  of 32 heads 1,000 (512) 47/46/52 (50)  2,048
//   (1,024) 94/97/114 (103);  of 64 heads 1,000 (1,024) 69/75/93 (74)  2,048 173/184/223 (196)
//   behind 1,024 positions, 16 heads:  64 44/40/37 (45)  512 54/49/43 (55)  four of 512 (512) 86/85/91 (95);  behind 4,000: 300 124/105/82
//   (126)  eight of 300 (640) 338/357/356 (380);  twenty of 200 57/67/92 (56)
enum LatentPromptForm { LP_TOKENS, LP_TWO_PARTS, LP_FOUR_PARTS };
static LatentPromptForm latent_prompt_form(long long workgroups, int context) {
    if (context <= 512 || workgroups > 768) return LP_TOKENS;
    return workgroups <= 256 || (workgroups <= 512 && context > 2048) ? LP_FOUR_PARTS : LP_TWO_PARTS;
}

// kv bf16 [entries, 2 heads, context, 128] and rot bf16 [entries * context, rot] are workspace; `context` is a multiple of 32 no
// smaller than any entry's first position + tokens, `longest` than its tokens.
extern "C" int kva_latent_prompt(void *out, const void *q, int q_row, int q_head, const void *cache, const void *w, void *kv,
                                 void *rot, const int *block_table, int max_blocks, const int *entry_seat,
                                 const int *entry_q_start, const int *entry_start_pos, int entries, const float *cos,
                                 const float *sin, int interleaved, const float *sinks, const void *gates, int gate_row,
                                 int gate_head, int gate_per_element, int page_size, int heads, int rank, int context,
                                 int longest, float scale, hipStream_t stream) {
    KVA_REQUIRE(out && q && cache && w && kv && rot && block_table && entry_seat && entry_q_start && entry_start_pos && cos && sin,
                "latent_prompt: missing operand");
    KVA_REQUIRE(kva_latent_prompt_supported(LP_DIM, LP_ROT, LP_VDIM, rank), "latent_prompt: rank %d is not a multiple of %d", rank, LDSP_K);
    KVA_REQUIRE(heads > 0 && heads <= 1024 && page_size > 0 && max_blocks > 0, "latent_prompt: bad sizes");
    KVA_REQUIRE(entries > 0 && entries <= 65535 && longest > 0 && longest <= context && context % 32 == 0, "latent_prompt: %d entries of up to %d tokens in contexts of %d",
                entries, longest, context);
    KVA_REQUIRE(q_row % 8 == 0 && q_head % 8 == 0 && ((uintptr_t)q | (uintptr_t)cache | (uintptr_t)w | (uintptr_t)kv | (uintptr_t)rot) % 16 == 0 &&
                    (uintptr_t)out % 8 == 0, "latent_prompt: rows must start at multiples of 16 bytes");
    const LatentPrompt a{(bf16_t *)out, (const bf16_t *)q, (const bf16_t *)cache, (const bf16_t *)w, (bf16_t *)kv, (bf16_t *)rot, block_table,
                         entry_seat, entry_q_start, entry_start_pos, cos, sin, sinks, (const bf16_t *)gates, q_row, q_head, gate_row,
                         gate_head, gate_per_element, max_blocks, page_size, heads, rank, context, interleaved, scale};
    const long long expand = (long long)((context + 127) / 128) * heads, tiles = (longest + LP_ROWS - 1) / LP_ROWS;
    KVA_REQUIRE(2 * expand <= 0x7fffffff && tiles * heads <= 0x7fffffff, "latent_prompt: too many workgroups");
    if (expand * entries <= 256) hipLaunchKernelGGL(latent_expand_kernel<4>, dim3((unsigned)(2 * expand), entries), dim3(256), 0, stream, a);
    else hipLaunchKernelGGL(latent_expand_kernel<8>, dim3((unsigned)expand, entries), dim3(256), 0, stream, a);
#define LP_LAUNCH(RT, GROUPS, PARTS)                                                                                              \
    hipLaunchKernelGGL((latent_prompt_kernel<RT, GROUPS, PARTS>), dim3((unsigned)(tiles * heads), entries), dim3(64 * GROUPS * PARTS), 0, \
                       stream, a, (int)tiles)
    switch (latent_prompt_form(tiles * heads * entries, context)) {
    case LP_TOKENS: LP_LAUNCH(1, 4, 1); break;
    case LP_TWO_PARTS: LP_LAUNCH(2, 2, 2); break;
    default: LP_LAUNCH(2, 2, 4); break;
    }
#undef LP_LAUNCH
    KVA_CHECK_LAUNCH("latent_prompt");
    return KVA_OK;
}
