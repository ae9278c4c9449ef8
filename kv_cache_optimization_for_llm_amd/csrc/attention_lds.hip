// Causal grouped-query attention for prompt portions, with the keys and values of a block shared
// by four wavefronts through LDS (bf16, gfx950, pages of 16 keys, head sizes 32/64/96/128).
//
// The one-wavefront kernel (attention_mfma.hip) loads every key and value block once per 32 query
// rows, straight from the page into operand registers; for long prompts that traffic through the
// vector memory path is what it waits for (halving it nearly halves its time).  Here a workgroup
// of four wavefronts takes 128 consecutive query rows of one request and kv head (row =
// token * G + head_in_group, as there), each wavefront 32 of them, and every 32-key block is
// copied from the pages to LDS once for all four, in the pages' own layout: two wavefronts a page of K each, two a page of
// V^T.  That layout is what operands are read in without a bank met twice: 16 keys' chunks of 8 elements of K next to each other
// are the 64 lanes' 16 bytes in order, 16 value dimensions of 16 keys their 8 bytes.  So the copies need no stop in registers
// (buffer loads to LDS); STAGES - 1 of them are on their way while one is computed, and the page of the one after those is
// looked up.  One barrier a block says that everybody's share of it has arrived and that the block before is read.
// One block ahead through registers, 8,190 tokens, 32 heads of 128 over 8: 762 us, 145 of
// them for that staging; 577 now (0.95 PFLOP/s of the visible half).  2,048 tokens 85 -> 77; 32 heads of 64, 8,190 tokens 398 -> 341.
// (Inside a model's prompt.  Calls of it alone, 8,192 tokens of 32 heads of 64 / 96 / 128: 335 / 588 / 589 -> 306 / 407 / 504.)
//
// The arithmetic per block is the other kernel's: S^T = K Q^T, online softmax in fp32 per query
// row with a lazily re-based reference, O^T += V^T P^T with P taken from the registers S^T came
// out in.  Usually every row's keys lie in one workgroup.  When a step has too few workgroups to
// fill the chip but each walks thousands of keys (a portion late in a long prompt), the keys are
// cut into `splits` ranges of `keys_per_split`, one workgroup each; a split writes un-normalised
// partials (o, m, l) as the one-wavefront kernel does and the same merge kernel combines them.
//
// Reference: the same recurrence as the tiled prefill kernel base/src/kernels.cu:361-466, which
// shares K/V tiles of 32 keys among the 8 query rows of a 256-thread block and cannot read keys
// from the cache.
#include "common.h"
#include "attention_frag.h"
#include "lds_product.h"
#include "kv_layout.h"
#include <math.h>
#include <type_traits>

#define LDS_PAGES 1024         // pages whose numbers stand in LDS at a time

// A workgroup of 4 GROUPS wavefronts; four of them (a group) walk blocks of KEYS keys, a stage holds a block of every group.
template <int D, int KEYS, int GROUPS>
struct LdsGeom {
    static constexpr int PAGE = 16 * D;                  // elements of a page of K or V^T (one kv head)
    static constexpr int BLOCK_TILES = KEYS / 16;        // pages, and tiles of 16 keys, of a block
    static constexpr int TILES = BLOCK_TILES * GROUPS;   // ... of a stage
    static constexpr int LOADS = TILES * 2 * D / (128 * GROUPS);                 // of 1 KiB a wavefront and stage
    static constexpr int STAGE = 2 * TILES * PAGE;       // K of all pages, then V^T of all
    static constexpr int STAGES = 6 * STAGE <= (GROUPS == 4 ? 120 : 75) * 1024 ? 3 : 2;
    static constexpr int STAGED = LDS_PAGES / TILES;     // stages whose pages stand in LDS
};
typedef __bf16 b16x4 __attribute__((ext_vector_type(4)));

template <int D, int KEYS, int GROUPS>
__device__ __forceinline__ void
attention_lds_item(bf16_t *lds, bf16_t *__restrict__ out, float *__restrict__ part_o, float *__restrict__ part_ml,
                   const bf16_t *__restrict__ q, int q_row_stride,
                   const bf16_t *__restrict__ k_cache, const bf16_t *__restrict__ v_cache,
                   const int *__restrict__ block_table, int max_blocks,
                   const int *__restrict__ item_meta, int num_q_heads, int num_kv_heads, float scale,
                   int window, int splits, int keys_per_split, const int item, const int kvh, const int split) {
    using Geo = LdsGeom<D, KEYS, GROUPS>;
    constexpr int RT = 2, NKS = D / 32, NDT = D / 16, TILES = Geo::BLOCK_TILES, STAGES = Geo::STAGES;
    const int tid = threadIdx.x, lane = tid & 63, wave = (tid >> 6) & 3, walk = __builtin_amdgcn_readfirstlane(tid >> 8);
    const int r = lane & 15, g = lane >> 4;
    const int G = num_q_heads / num_kv_heads;

    const int *meta = item_meta + (size_t)__builtin_amdgcn_readfirstlane(item) * 8;
    const int q_start = __builtin_amdgcn_readfirstlane(meta[0]);
    const int q_len = __builtin_amdgcn_readfirstlane(meta[1]);
    const int start_pos = __builtin_amdgcn_readfirstlane(meta[2]);
    const int seat = __builtin_amdgcn_readfirstlane(meta[3]);
    const int row0 = __builtin_amdgcn_readfirstlane(meta[4]);
    const int *bt = block_table + (size_t)seat * max_blocks;
    const int M = q_len * G;

    // ---- this wavefront's 32 rows
    const int wrow0 = row0 + 32 * wave;
    const bool wave_valid = wrow0 < M;
    bool row_valid[RT];
    int tq[RT], head[RT], my_pos[RT], my_lo[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int row = wrow0 + rt * 16 + r;
        row_valid[rt] = row < M;
        tq[rt] = row_valid[rt] ? row / G : 0;
        head[rt] = kvh * G + (row_valid[rt] ? row % G : 0);
        my_pos[rt] = start_pos + tq[rt];
        my_lo[rt] = kva_first_visible_signed(my_pos[rt], window);
    }
    const int w_last = (wrow0 + 31 < M - 1) ? wrow0 + 31 : M - 1;
    // (uniform over the wavefront: said explicitly, since the division by G is done in the vector
    // ALU and the compiler then takes every test on these for a per-lane one)
    const int w_hi = __builtin_amdgcn_readfirstlane(start_pos + w_last / G);      // last key the wave sees
    const int w_first_pos = __builtin_amdgcn_readfirstlane(start_pos + wrow0 / G);
    const int w_lo = kva_first_visible_signed(w_first_pos, window);
    const int w_hi_lo = kva_first_visible_signed(w_hi, window);      // where the window (or chunk) of the wave's last row starts
    const bool all_rows = wrow0 + 32 <= M;

    // ---- keys the workgroup visits
    const int g_last = (row0 + 127 < M - 1) ? row0 + 127 : M - 1;
    const int g_hi = __builtin_amdgcn_readfirstlane(start_pos + g_last / G);
    const int g_first_pos = __builtin_amdgcn_readfirstlane(start_pos + row0 / G);
    const int g_lo = kva_first_visible_signed(g_first_pos, window);
    int k_begin = g_lo & ~31;
    int k_end = g_hi + 1;
    if (splits > 1) {               // uniform over the workgroup; an empty range leaves m = -inf, l = 0
        const int s_lo = split * keys_per_split, s_hi = s_lo + keys_per_split;
        if (s_lo > k_begin) k_begin = s_lo;
        if (s_hi < k_end) k_end = s_hi;
    }
    const int lo_tile = g_lo & ~15, hi_tile = g_hi & ~15;

    // ---- Q^T operand: lane (r, g) holds Q[row r][ks * 32 + g * 8 ...]
    Frag8 qf[RT][NKS];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const bf16_t *qrow = q + (size_t)(q_start + tq[rt]) * q_row_stride + (size_t)head[rt] * D;
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
            qf[rt][ks].u4 = row_valid[rt] ? *reinterpret_cast<const uint4 *>(qrow + ks * 32 + g * 8)
                                          : make_uint4(0, 0, 0, 0);
    }

    // Running maximum m, accumulator O^T and denominator per query row.  The denominator is one more
    // tile of the second product: against a V^T tile of ones, O^T += V^T P^T adds up the row's P
    // (every element of the tile ends up as the row's sum) - on the matrix cores, which have time
    // to spare here, instead of 16 additions and a 4-lane reduction per block in the vector ALU,
    // which has none.  It also makes the denominator the sum of exactly the rounded P the numerator uses.
    float m[RT];
    f32x4 o[RT][NDT], ol[RT];
    Frag8 ones;
    ones.u4 = make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);      // 8 x bf16 1.0
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        m[rt] = -INFINITY;
        ol[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) o[rt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // ---- copies page -> LDS: of blocks of 32 keys a wavefront brings a page of a stage (the first half of the wavefronts one of K), of blocks of
    // 64 one of K and one of V^T.  A tile outside the keys the workgroup needs is redirected to the nearest needed one (its page is
    // certainly mapped); its scores are masked away.
    const int wave_s = __builtin_amdgcn_readfirstlane(tid >> 6);
    bf16_t *pages = lds + STAGES * Geo::STAGE;
    const int page_at = KEYS == 32 ? wave_s & (Geo::TILES - 1) : wave_s;
    auto page_of = [&](int stage) {         // (of those that stand in LDS; read as bf16 like the operands)
        union { b16x2 v; int i; } x;
        x.v = *reinterpret_cast<const b16x2 *>(pages + 2 * (Geo::TILES * min(stage, Geo::STAGED - 1) + page_at));
        return x.i;
    };
    // V^T: of every 16 value dimensions first their first 8 keys, then the others, 16 bytes each
    const int k_at = 16 * lane, v_at = (lane >> 5) * 512 + r * 32 + (g & 1) * 16;
    auto fetch_page = [&](const bf16_t *cache, int lane_at, int page, int to) {
        const Buffer from = buffer_at(cache + ((size_t)page * num_kv_heads + kvh) * Geo::PAGE, Geo::PAGE * sizeof(bf16_t));
#pragma unroll
        for (int i = 0; i < D / 32; ++i) buffer_to_lds(from, lane_at, i * 1024, lds + to + i * 512);
    };
    auto fetch = [&](int slot, int page_v) {
        const int page = __builtin_amdgcn_readfirstlane(page_v);
        if constexpr (KEYS == 32) {
            const bool keys = wave_s < Geo::TILES;
            fetch_page(keys ? k_cache : v_cache, keys ? k_at : v_at, page, slot * Geo::STAGE + wave_s * Geo::PAGE);
        } else {
            fetch_page(k_cache, k_at, page, slot * Geo::STAGE + wave_s * Geo::PAGE);
            fetch_page(v_cache, v_at, page, slot * Geo::STAGE + (Geo::TILES + wave_s) * Geo::PAGE);
        }
    };

    const float scale2 = scale * 1.44269504088896340736f;   // exp(x * scale) = exp2(x * scale * log2 e)
    constexpr float REBASE = 8.f;
    const float rebase_raw = REBASE / scale2;

    auto compute_as = [&](auto masked_tag, const bf16_t *buf, int kstart) {
        constexpr bool MASKED = decltype(masked_tag)::value;
        // operands from LDS: K: lane (r, g) holds K[key t*16 + r][ks*32 + g*8 ..]; V^T: lane (r, g)
        // holds V^T[dt*16 + r][keys t*16 + 4g .. +3] for both tiles of the block.  (Read as vectors of bf16: the compiler then knows
        // that no copy on its way writes what is read here, of which the barrier makes sure, and does not wait for all of them.)
        constexpr int HALVES = TILES / 2;          // 32 keys are one operand of the second product
        Frag8 vf[NDT][HALVES];
        auto values = [&](int dt) {
#pragma unroll
            for (int h = 0; h < HALVES; ++h) {
                union { b16x4 v; uint2 u2; } x[2];
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    x[t].v = *reinterpret_cast<const b16x4 *>(buf + (Geo::TILES + 2 * h + t) * Geo::PAGE + dt * 256 + (g >> 1) * 128 + r * 8 + (g & 1) * 4);
                // Behind the workgroup's last key a block holds whatever the page held before (or the nearest
                // needed tile, for a redirected one): P is zero there, and the values are made zero too, so
                // that nothing non-finite left in a page can reach this request.
                if (MASKED && kstart + KEYS - 1 > g_hi) {
                    const int n0 = g_hi + 1 - (kstart + 32 * h + 4 * g);
                    x[0].u2 = keep_first_keys(x[0].u2, n0);
                    x[1].u2 = keep_first_keys(x[1].u2, n0 - 16);
                }
                vf[dt][h].u2[0] = x[0].u2;
                vf[dt][h].u2[1] = x[1].u2;
            }
        };

        f32x4 s[RT][TILES];
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            Frag8 kf[NKS];
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) kf[ks].v = *reinterpret_cast<const b16x8 *>(buf + t * Geo::PAGE + ks * 512 + lane * 8);
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) s[rt][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) s[rt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[ks].v, qf[rt][ks].v, s[rt][t], 0, 0, 0);
        }
        float sv[RT][4 * TILES], mloc[RT];
        Frag8 pf[RT][HALVES];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            float mx = -INFINITY;
#pragma unroll
            for (int t = 0; t < TILES; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float x = s[rt][t][i];
                    if (MASKED) {
                        const int key = kstart + t * 16 + 4 * g + i;
                        const bool vis = row_valid[rt] && key <= my_pos[rt] && key >= my_lo[rt];
                        x = vis ? x : -INFINITY;
                    }
                    sv[rt][t * 4 + i] = x;
                    mx = fmaxf(mx, x);
                }
            mloc[rt] = mx;            // this lane's part of the row: the whole row's only when the reference moves
        }
        // the reference of the exponentials follows the running maximum lazily (see attention_mfma.hip)
        bool rebase = false;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) rebase = rebase || mloc[rt] > m[rt] + rebase_raw;
        if (__builtin_amdgcn_ballot_w64(rebase) != 0) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const float m_new = fmaxf(m[rt], quad_rows_max(mloc[rt]));
                const float c = __builtin_amdgcn_exp2f((m[rt] - ((m_new == -INFINITY) ? 0.f : m_new)) * scale2);
                ol[rt][0] *= c; ol[rt][1] *= c; ol[rt][2] *= c; ol[rt][3] *= c;
#pragma unroll
                for (int dt = 0; dt < NDT; ++dt) {
                    o[rt][dt][0] *= c; o[rt][dt][1] *= c; o[rt][dt][2] *= c; o[rt][dt][3] *= c;
                }
                m[rt] = m_new;
            }
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const float neg_ref = (MASKED && m[rt] == -INFINITY) ? 0.f : -m[rt] * scale2;
#pragma unroll
            for (int j = 0; j < 4 * TILES; j += 2) {
                const float p0 = __builtin_amdgcn_exp2f(fmaf(sv[rt][j], scale2, neg_ref));
                const float p1 = __builtin_amdgcn_exp2f(fmaf(sv[rt][j + 1], scale2, neg_ref));
                pf[rt][j / 8].p2[j % 8 / 2] = pack_bf16(p0, p1);
            }
        }
        // A SIMD issues either a matrix-core product or a vector instruction, from whichever wavefront: timed alone, 8 products
        // and 24 multiply-adds in one wavefront take 126 ns, the products without the multiply-adds 67 and the multiply-adds
        // without the products 56, and given to two wavefronts of one SIMD 109; so a key block costs its products plus its
        // softmax, however the two are interleaved.  (Nothing in a wavefront's priority during its products: 577 / 577 us.)
        // Values are read a tile ahead of their products and no further (head size 128, 8,190 tokens: two tiles ahead 605 us, one
        // 577; left to the compiler's order 613).
        values(0);
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
            if (dt + 1 < NDT) values(dt + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int h = 0; h < HALVES; ++h)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
                    o[rt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[dt][h].v, pf[rt][h].v, o[rt][dt], 0, 0, 0);
        }
#pragma unroll
        for (int h = 0; h < HALVES; ++h)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) ol[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones.v, pf[rt][h].v, ol[rt], 0, 0, 0);
    };

    // ---- the key loop.  Copies past the end are redirected inside page_of (never out of the mapped pages) and unused.
    auto compute = [&](const bf16_t *buf, int kstart) {
        if (wave_valid && kstart < k_end && kstart <= w_hi && kstart + KEYS - 1 >= w_lo) {
            const bool masked = kstart < w_hi_lo || kstart + KEYS - 1 > w_first_pos || !all_rows;
            if (masked) compute_as(std::true_type{}, buf, kstart);
            else compute_as(std::false_type{}, buf, kstart);
        }
    };
    constexpr int STEP = KEYS * GROUPS;
    for (int k0 = k_begin; k0 < k_end; k0 += STEP * Geo::STAGED) {             // uniform over the workgroup
        const int k1 = min(k_end, k0 + STEP * Geo::STAGED);
        for (int i = tid; i < min(LDS_PAGES, (k1 - k0 + 15) / 16 + Geo::TILES * (STAGES + 1)); i += 256 * GROUPS)
            reinterpret_cast<int *>(pages)[i] = bt[min(max(k0 + 16 * i, lo_tile), hi_tile) >> 4];
        __syncthreads();
#pragma unroll
        for (int b = 0; b < STAGES - 1; ++b) fetch(b, page_of(b));
        int slot = 0, stage = STAGES - 1, page = page_of(stage);
        for (int kstart = k0; kstart < k1; kstart += STEP) {
            wait_and_meet<(STAGES - 2) * Geo::LOADS>();
            // into the slot that was read in the turn before: every wavefront has passed the barrier since
            fetch(slot == 0 ? STAGES - 1 : slot - 1, page);
            page = page_of(++stage);
            compute(lds + slot * Geo::STAGE + walk * TILES * Geo::PAGE, kstart + walk * KEYS);
            slot = slot + 1 == STAGES ? 0 : slot + 1;
        }
        wait_and_meet<0>();                 // nothing is on its way any more, nobody reads
    }
    if constexpr (GROUPS > 1) {
        // The groups' sums of the same rows meet in LDS, a lane's own numbers in a place of their own, a row tile at a time: half of the
        // groups hands over to the other half until one is left.
        constexpr int EACH = NDT + 1;
        static_assert(2 * GROUPS * (EACH * 1024 + 256) <= STAGES * Geo::STAGE * 2, "half of the groups' sums fit where the blocks were");
#pragma unroll
        for (int left = GROUPS / 2; left > 0; left /= 2) {
            f32x4 *box = reinterpret_cast<f32x4 *>(lds) + (size_t)((walk % left) * 4 + wave) * EACH * KVA_WAVE + lane;
            float *refs = reinterpret_cast<float *>(lds) + (size_t)left * 4 * EACH * KVA_WAVE * 4 + ((walk % left) * 4 + wave) * KVA_WAVE + lane;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                if (walk >= left && walk < 2 * left) {
                    *refs = m[rt];
                    box[NDT * KVA_WAVE] = ol[rt];
#pragma unroll
                    for (int dt = 0; dt < NDT; ++dt) box[dt * KVA_WAVE] = o[rt][dt];
                }
                __syncthreads();
                if (walk < left) {
                    const float theirs = *refs, m_new = fmaxf(m[rt], theirs), ref = m_new == -INFINITY ? 0.f : m_new;
                    const float c = __builtin_amdgcn_exp2f((m[rt] - ref) * scale2), d = __builtin_amdgcn_exp2f((theirs - ref) * scale2);
                    ol[rt] = ol[rt] * c + box[NDT * KVA_WAVE] * d;
#pragma unroll
                    for (int dt = 0; dt < NDT; ++dt) o[rt][dt] = o[rt][dt] * c + box[dt * KVA_WAVE] * d;
                    m[rt] = m_new;
                }
                __syncthreads();                // (what goes there next: the other row tile, the next hand-over, the next item's pages)
            }
        }
        if (walk > 0) return;
    }

    // ---- lane (r, g) holds O[row r][dt * 16 + 4g + i]
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        if (!row_valid[rt]) continue;
        const size_t orow = (size_t)(q_start + tq[rt]) * num_q_heads + head[rt];
        if (splits > 1) {
            float *dst = part_o + (orow * splits + split) * D;
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
                *reinterpret_cast<float4 *>(dst + dt * 16 + 4 * g) =
                    make_float4(o[rt][dt][0], o[rt][dt][1], o[rt][dt][2], o[rt][dt][3]);
            if (g == 0) {
                part_ml[(orow * splits + split) * 2] = m[rt] * scale2;   // the merge works in the base-2 domain
                part_ml[(orow * splits + split) * 2 + 1] = ol[rt][0];
            }
            continue;
        }
        const float inv = 1.f / ol[rt][0];
        bf16_t *dst = out + orow * D;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
            union { b16x2 p2[2]; uint2 u2; } w;
            w.p2[0] = pack_bf16(o[rt][dt][0] * inv, o[rt][dt][1] * inv);
            w.p2[1] = pack_bf16(o[rt][dt][2] * inv, o[rt][dt][3] * inv);
            *reinterpret_cast<uint2 *>(dst + dt * 16 + 4 * g) = w.u2;
        }
    }
}

// One workgroup of four wavefronts per (item of 128 query rows or pair of items, kv head); the kv
// head varies fastest so that a die's L2 keeps meeting the same heads.  With `pair` a workgroup
// takes item w and then item n-1-w of the list, which the caller orders by keys visited.
template <int D, int KEYS, int GROUPS>
__device__ __forceinline__ void
attention_lds_body(bf16_t *__restrict__ out, float *__restrict__ part_o, float *__restrict__ part_ml,
                   const bf16_t *__restrict__ q, int q_row_stride,
                   const bf16_t *__restrict__ k_cache, const bf16_t *__restrict__ v_cache,
                   const int *__restrict__ block_table, int max_blocks,
                   const int *__restrict__ item_meta, int num_items, int pair, int num_q_heads,
                   int num_kv_heads, float scale, int window, int splits, int keys_per_split) {
    using Geo = LdsGeom<D, KEYS, GROUPS>;
    __shared__ __align__(16) bf16_t lds[Geo::STAGES * Geo::STAGE + 2 * LDS_PAGES];      // the ring, then pages
    const int kvh = blockIdx.x % num_kv_heads;
    const int w = blockIdx.x / num_kv_heads, split = blockIdx.z;
    attention_lds_item<D, KEYS, GROUPS>(lds, out, part_o, part_ml, q, q_row_stride, k_cache, v_cache, block_table, max_blocks,
                          item_meta, num_q_heads, num_kv_heads, scale, window, splits, keys_per_split, w, kvh, split);
    const int other = num_items - 1 - w;
    if (pair && other > w)      // the last barrier of the first item has passed: LDS is free again
        attention_lds_item<D, KEYS, GROUPS>(lds, out, part_o, part_ml, q, q_row_stride, k_cache, v_cache, block_table, max_blocks,
                              item_meta, num_q_heads, num_kv_heads, scale, window, splits, keys_per_split, other, kvh,
                              split);
}

#define LDS_KERNEL_PARAMS                                                                          \
    bf16_t *__restrict__ out, float *__restrict__ part_o, float *__restrict__ part_ml,             \
    const bf16_t *__restrict__ q, int q_row_stride,                                                \
    const bf16_t *__restrict__ k_cache, const bf16_t *__restrict__ v_cache,                        \
    const int *__restrict__ block_table, int max_blocks, const int *__restrict__ item_meta,        \
    int num_items, int pair, int num_q_heads, int num_kv_heads, float scale, int window,           \
    int splits, int keys_per_split
#define LDS_KERNEL_ARGS                                                                            \
    out, part_o, part_ml, q, q_row_stride, k_cache, v_cache, block_table, max_blocks, item_meta,   \
    num_items, pair, num_q_heads, num_kv_heads, scale, window, splits, keys_per_split

// Head sizes up to 64: four wavefronts a SIMD (up to 128 registers each, no spills).
template <int D>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
attention_lds_kernel_4(LDS_KERNEL_PARAMS) {
    attention_lds_body<D, 32, 1>(LDS_KERNEL_ARGS);
}

// Head sizes 96 and 128: left alone the compiler takes over 300 registers, which leaves one wavefront per SIMD and nothing to
// overlap matrix-core, vector and LDS work with.  Three (168 registers, 13 of them spilled at 128) against two without spills,
// 8,190 tokens of 32 heads of 128: 577 against 703 us.
template <int D>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
attention_lds_kernel_3(LDS_KERNEL_PARAMS) {
    attention_lds_body<D, 32, 1>(LDS_KERNEL_ARGS);
}

// Where few workgroups run at once a wavefront's chain through its blocks is the time (0.65 us a block of 32 keys with a SIMD or half of one to
// itself, 0.3 where four share it).  Blocks of 64 keys, two wavefronts a SIMD: 1.05 us a block.  us, blocks of 32 -> of 64: 32 heads of 64
// over 8, 3,072 / 4,096 / 6,000 tokens 66 -> 59, 96 -> 88, 193 -> 180; heads of 128, 24 over 8, 3,072 91 -> 84; 32 over 8, 3,072 100 -> 90.
// (Where either form is behind, and by how much: the lines in ops/attention.py.)
template <int D>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
attention_lds_kernel_64(LDS_KERNEL_PARAMS) {
    attention_lds_body<D, 64, 1>(LDS_KERNEL_ARGS);
}

// Fewer still: two groups of four wavefronts walk every other block and add up at the end.  Against the one-wavefront kernel with an item's
// keys shared by two (which was ahead there): 32 heads of 64 over 8, 2,048 / 2,304 tokens 39 -> 34, 46 -> 39; heads of 128, 24 over 8, 1,536 / 2,048 /
// 2,304 39 -> 35, 57 -> 43, 69 -> 51; 32 over 8, 1,536 / 2,048 47 -> 36, 62 -> 52 (blocks of 32, one group), 1,531 and 963 tokens together 68 -> 54.
// Four groups were no faster (2,048 tokens of 32 heads of 64 36).
template <int D>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(D <= 64 ? 4 : 2)))
attention_lds_kernel_pairs(LDS_KERNEL_PARAMS) {
    attention_lds_body<D, 32, 2>(LDS_KERNEL_ARGS);
}

extern "C" int kva_attention_lds_supported(int head_dim, int page_size) {
    return (page_size == 16 && (head_dim == 32 || head_dim == 64 || head_dim == 96 || head_dim == 128)) ? 1 : 0;
}

// item_meta: [num_items, 8] int32 = (q_start, q_len, start_pos, seat, row0, 0, 0, 0) per item of
// 128 query rows (row0 a multiple of 128).  q: bf16 rows `q_row_stride` elements apart; out
// [tokens, num_q_heads * head_dim] bf16.
// With splits > 1: part_o [tokens * num_q_heads, splits, head_dim] and part_ml [.., splits, 2] fp32
// take the partials, keys_per_split is a multiple of 32, and the merge runs after the kernel: over
// every row of out (`all_rows`: the items cover them all) or over the items' rows alone.  kind 1: blocks of 64 keys, 2: two groups
// of wavefronts (either with one range).
extern "C" int kva_attention_lds(void *out, float *part_o, float *part_ml, const void *q, int q_row_stride,
                                 const void *k_cache, const void *v_cache, const int *block_table, int max_blocks,
                                 const int *item_meta, int num_items, int pair, int num_q_heads,
                                 int num_kv_heads, int head_dim, int page_size, float scale, int window,
                                 int splits, int keys_per_split, int total_rows, int all_rows, int kind,
                                 hipStream_t stream) {
    KVA_REQUIRE(kind == 0 || ((kind == 1 || kind == 2) && splits == 1), "attention_lds: no kernel of kind %d for %d key ranges", kind, splits);
    KVA_REQUIRE(splits >= 1 && splits <= MERGE_MAX_SPLITS && num_kv_heads <= 65535,
                "attention_lds: 1..%d splits and at most 65535 kv heads", MERGE_MAX_SPLITS);
    KVA_REQUIRE(splits == 1 || (keys_per_split > 0 && keys_per_split % 32 == 0 && part_o && part_ml),
                "attention_lds: splits need a key count that is a multiple of 32 and a workspace");
    KVA_REQUIRE(num_items >= 0 && num_q_heads > 0 && num_kv_heads > 0 && max_blocks > 0, "attention_lds: bad sizes");
    KVA_REQUIRE(num_q_heads % num_kv_heads == 0, "attention_lds: %d query heads is not a multiple of %d kv heads",
                num_q_heads, num_kv_heads);
    KVA_REQUIRE(kva_attention_lds_supported(head_dim, page_size),
                "attention_lds: head_dim %d with pages of %d keys is not supported (32/64/96/128, 16)", head_dim, page_size);
    KVA_REQUIRE(q_row_stride % 8 == 0 && q_row_stride >= num_q_heads * head_dim, "attention_lds: q row stride %d", q_row_stride);
    KVA_REQUIRE(scale > 0.f, "attention_lds: the scale must be positive");     // (window < 0: chunks of -window positions)
    KVA_REQUIRE(item_meta != nullptr || num_items == 0, "attention_lds: item records are needed");
    if (num_items == 0) return KVA_OK;
    const int groups = pair ? (num_items + 1) / 2 : num_items;
    KVA_REQUIRE((long)groups * num_kv_heads < (1L << 31), "attention_lds: too many work items");
    dim3 grid(groups * num_kv_heads, 1, splits), block(kind == 2 ? 512 : 256);
#define LAUNCH(KERNEL, DD)                                                                          \
    hipLaunchKernelGGL((KERNEL<DD>), grid, block, 0, stream, (bf16_t *)out, part_o, part_ml,        \
                       (const bf16_t *)q, q_row_stride, (const bf16_t *)k_cache,                    \
                       (const bf16_t *)v_cache, block_table, max_blocks, item_meta, num_items, pair, \
                       num_q_heads, num_kv_heads, scale, window, splits, keys_per_split)
    if (kind == 1) {
        switch (head_dim) {
        case 32: LAUNCH(attention_lds_kernel_64, 32); break;
        case 64: LAUNCH(attention_lds_kernel_64, 64); break;
        case 96: LAUNCH(attention_lds_kernel_64, 96); break;
        default: LAUNCH(attention_lds_kernel_64, 128); break;
        }
    } else if (kind == 2) {
        switch (head_dim) {
        case 32: LAUNCH(attention_lds_kernel_pairs, 32); break;
        case 64: LAUNCH(attention_lds_kernel_pairs, 64); break;
        case 96: LAUNCH(attention_lds_kernel_pairs, 96); break;
        default: LAUNCH(attention_lds_kernel_pairs, 128); break;
        }
    } else
    switch (head_dim) {
    case 32: LAUNCH(attention_lds_kernel_4, 32); break;
    case 64: LAUNCH(attention_lds_kernel_4, 64); break;
    case 96: LAUNCH(attention_lds_kernel_3, 96); break;
    default: LAUNCH(attention_lds_kernel_3, 128); break;
    }
#undef LAUNCH
    KVA_CHECK_LAUNCH("attention_lds");
    if (splits > 1)
        return kva_attention_merge_launch(out, part_o, part_ml, head_dim, splits, item_meta, nullptr, nullptr, nullptr,
                                          num_items, 128, total_rows, num_q_heads, num_kv_heads, all_rows, stream);
    return KVA_OK;
}
