// Causal grouped-query attention over the paged cache: the plain kernel.
//
// One wavefront per token and query head, or several query heads of one key head.  The query at absolute position p of its request
// attends to keys lo..p of the same request (lo = 0, or p - window + 1 with a window, or the start of
// p's own chunk where positions see each other only inside chunks of a fixed size), all read
// from the cache through the request's block-table row - the step has already written this
// step's K and V there (the reference also scatters before it attends,
// base/src/engine.cu:726-737).  Same recurrence as the reference's decode kernel
// (paged_attention/src/kernels.cu:150-219): fp32 dot product, score scaled, running max m,
// denominator l and accumulator acc in fp32, out = acc / l.  GQA: kv_head = q_head / (nq / nkv).
//
// K pages are [kv_head, page_size, head_dim]; V pages are stored transposed,
// [kv_head, head_dim, page_size].
//
// Keys are taken in blocks of 64 aligned to absolute positions (0..63, 64..127, ...): lane i of
// the wavefront owns key 64*b + i.  Because the blocks do not depend on where a step starts
// or on what else is in the batch, the fp32 result for a (request, position) is bit-identical
// however the tokens were cut into steps.
//
// This kernel serves the fp32 path and every shape (head_dim any multiple of 4 up to 256);
// the bf16 path uses it where the MFMA kernels do not apply.
#include "common.h"
#include "kv_layout.h"
#include <math.h>
#include <type_traits>

#define ATTN_MAX_HEAD_DIM 256

template <typename T> struct Vec4;
template <> struct Vec4<float> {
    static __device__ inline void load(const float *p, float (&o)[4]) {
        const float4 v = *reinterpret_cast<const float4 *>(p);
        o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
    }
};
template <> struct Vec4<bf16_t> {
    static __device__ inline void load(const bf16_t *p, float (&o)[4]) {
        const uint2 v = *reinterpret_cast<const uint2 *>(p);
        o[0] = bf16_bits_to_float((uint16_t)(v.x & 0xffff));
        o[1] = bf16_bits_to_float((uint16_t)(v.x >> 16));
        o[2] = bf16_bits_to_float((uint16_t)(v.y & 0xffff));
        o[3] = bf16_bits_to_float((uint16_t)(v.y >> 16));
    }
};

// Multiply-adds are written out, and a product that is rounded by itself is kept apart from the addition behind it, in both kernels of this
// file: which of them the compiler folds into one is otherwise its own choice in every variant, and a token's bits are to be the same
// in all of them.
__device__ inline float attn_rounded(float x) {
    asm("" : "+v"(x));
    return x;
}

// H query heads of one key head go together: a key's and a value's elements are loaded once for all of them, and their
// sums, which are chains of dependent additions in a fixed order, run side by side.  With `fours` (pages of a multiple of
// 4 keys) a lane reads its value element of 4 keys at once, a row of the transposed page, and 32 keys' loads are under way
// together; a head's additions keep their order in every variant, so its bits do too.  One key's values a load, one head a
// wavefront -> this, fp32, us: 603 tokens of 32 heads of 64 over 8 key heads at up to 201 / 2,000 keys 253 / 731 -> 35 / 78,
// one token at 200 / 2,000 keys 34 / 307 -> 11 / 77 (bound by the chains: 64 dependent additions a block for the score,
// 64 for the values), heads of 128 at 2,000 keys 659 -> 185.  A head alone, which is what few rows get, has all of a block's
// loads under way together instead of a quarter and a half of them: 3 tokens at up to 200 keys 11.3 -> 10.6 (heads of 128 17.0 ->
// 15.5), one at 2,000 77 -> 66 (bf16 up to 32 keys 0.2 us more); several heads a wavefront have no registers for it and other
// wavefronts to hide behind, and heads that are not whole rounds of 64 elements would ask for the rest one load after the other (96
// elements at 200 keys 15.2 -> 17.0).
template <typename T, int H, bool ALL = false>
__global__ void __launch_bounds__(KVA_WAVE)
attention_rowwise_kernel(T *__restrict__ out, const T *__restrict__ q, int q_row_stride,
                         const T *__restrict__ k_cache, const T *__restrict__ v_cache,
                         const int *__restrict__ block_table, int max_blocks,
                         const int *__restrict__ tok_seat, const int *__restrict__ tok_pos,
                         int num_q_heads, int num_kv_heads, int head_dim, int value_dim, int page_size, int fours,
                         float scale, int window, int keep_first, int chunk, const float *__restrict__ sinks) {
    __shared__ __attribute__((aligned(16))) float q_s[H][ATTN_MAX_HEAD_DIM];
    __shared__ __attribute__((aligned(16))) float p_s[H][KVA_WAVE];
    __shared__ long long voff_s[KVA_WAVE];
    // ALL: 64 of a key's elements, and all values of a block, are asked for before the first is used
    constexpr int KEY_LOADS = ALL ? 16 : 4, FOURS = ALL ? 16 : 8;

    const int t = blockIdx.x;
    const int qh = blockIdx.y * H;
    const int lane = threadIdx.x;
    const int kvh = qh / (num_q_heads / num_kv_heads);
    const int pos = tok_pos[t];
    const int *bt = block_table + (size_t)tok_seat[t] * max_blocks;

    const T *qrow = q + (size_t)t * q_row_stride + (size_t)qh * head_dim;
#pragma unroll
    for (int h = 0; h < H; ++h)
        for (int j = lane; j < head_dim; j += KVA_WAVE) q_s[h][j] = to_float(qrow[h * head_dim + j]);
    __syncthreads();

    const int lo = kva_first_visible(pos, window, chunk);
    float m[H], l[H], corr[H];
    float acc[ATTN_MAX_HEAD_DIM / KVA_WAVE][H];
#pragma unroll
    for (int h = 0; h < H; ++h) {
        m[h] = -INFINITY;
        l[h] = 0.f;
#pragma unroll
        for (int c = 0; c < ATTN_MAX_HEAD_DIM / KVA_WAVE; ++c) acc[c][h] = 0.f;
    }

    for (int kb = keep_first > 0 ? 0 : lo / KVA_WAVE; kb <= pos / KVA_WAVE; ++kb) {
        // a block with no visible key: behind the window and past the kept first positions
        if (kb * KVA_WAVE + KVA_WAVE <= lo && kb * KVA_WAVE >= keep_first) continue;
        const int key = kb * KVA_WAVE + lane;
        const bool valid = key <= pos && (key >= lo || key < keep_first);
        const unsigned long long seen = __ballot(valid);
        float s[H];
#pragma unroll
        for (int h = 0; h < H; ++h) s[h] = -INFINITY;
        if (valid) {
            const int page = bt[key / page_size];
            const T *kpage = k_cache + ((long long)page * num_kv_heads + kvh) * page_size * (long long)head_dim;
            const int krow = key % page_size, kc = kva_k_chunk(head_dim);
            float dot[H];
#pragma unroll
            for (int h = 0; h < H; ++h) dot[h] = 0.f;
#pragma unroll KEY_LOADS
            for (int j = 0; j < head_dim; j += 4) {
                float kv[4];
                Vec4<T>::load(kpage + kva_k_at(krow, j, page_size, kc), kv);     // (4 elements never straddle a chunk)
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    const float4 qv = *reinterpret_cast<const float4 *>(&q_s[h][j]);
                    dot[h] = __builtin_fmaf(qv.x, kv[0], dot[h]);
                    dot[h] = __builtin_fmaf(qv.y, kv[1], dot[h]);
                    dot[h] = __builtin_fmaf(qv.z, kv[2], dot[h]);
                    dot[h] = __builtin_fmaf(qv.w, kv[3], dot[h]);
                }
            }
#pragma unroll
            for (int h = 0; h < H; ++h) s[h] = attn_rounded(dot[h] * scale);
        }
        __syncthreads();  // the previous block's p_s / voff_s have been consumed
#pragma unroll
        for (int h = 0; h < H; ++h) {
            const float m_new = fmaxf(m[h], wave_max(s[h]));
            corr[h] = (m[h] == -INFINITY) ? 0.f : expf(m[h] - m_new);
            const float p = valid ? expf(s[h] - m_new) : 0.f;
            l[h] = __builtin_fmaf(l[h], corr[h], wave_sum(p));
            m[h] = m_new;
            p_s[h][lane] = p;
        }
        // V is stored transposed inside a page: [page, kv_head, value_dim, page_size].  Four keys together are of one
        // page; where none of the four is visible, the first visible key's place is read in their stead and not used.
        const int first = __ffsll(seen) - 1;
        const int group = fours ? ((seen >> (lane & ~3)) & 15 ? lane : first & ~3) : (valid ? lane : first);
        const int vkey = kb * KVA_WAVE + group;
        voff_s[lane] = ((long long)bt[vkey / page_size] * num_kv_heads + kvh) * (long long)value_dim * page_size +
                       vkey % page_size;
        __syncthreads();
        const int last = (pos - kb * KVA_WAVE < KVA_WAVE - 1) ? pos - kb * KVA_WAVE : KVA_WAVE - 1;
#pragma unroll
        for (int c = 0; c < ATTN_MAX_HEAD_DIM / KVA_WAVE; ++c) {
            const int j = lane + c * KVA_WAVE;
            if (j < value_dim) {
                const T *vcol = v_cache + (long long)j * page_size;
                float a[H];
#pragma unroll
                for (int h = 0; h < H; ++h) a[h] = attn_rounded(acc[c][h] * corr[h]);
                if (fours) {
                    for (int i0 = 0; i0 <= last; i0 += 4 * FOURS) {
                        float v[FOURS][4];
#pragma unroll
                        for (int g = 0; g < FOURS; ++g) Vec4<T>::load(vcol + voff_s[i0 + 4 * g], v[g]);
                        const unsigned long long these = seen >> i0;
                        if (seen != ~0ull) {
#pragma unroll
                            for (int g = 0; g < FOURS; ++g)
#pragma unroll
                                for (int u = 0; u < 4; ++u) v[g][u] = (these >> (4 * g + u)) & 1 ? v[g][u] : 0.f;
                        }
#pragma unroll
                        for (int g = 0; g < FOURS; ++g) {
                            if (ALL && g == 8 && last < 32) break;      // (no keys in the block's second half)
#pragma unroll
                            for (int h = 0; h < H; ++h) {
                                const float4 p = *reinterpret_cast<const float4 *>(&p_s[h][i0 + 4 * g]);
                                a[h] = __builtin_fmaf(p.x, v[g][0], a[h]);
                                a[h] = __builtin_fmaf(p.y, v[g][1], a[h]);
                                a[h] = __builtin_fmaf(p.z, v[g][2], a[h]);
                                a[h] = __builtin_fmaf(p.w, v[g][3], a[h]);
                            }
                        }
                    }
                } else {
                    for (int i = 0; i <= last; ++i)
                        if ((seen >> i) & 1) {
                            const float v = to_float(vcol[voff_s[i]]);
#pragma unroll
                            for (int h = 0; h < H; ++h) a[h] = __builtin_fmaf(p_s[h][i], v, a[h]);
                        }
                }
#pragma unroll
                for (int h = 0; h < H; ++h) acc[c][h] = a[h];
            }
        }
    }
#pragma unroll
    for (int h = 0; h < H; ++h) {
        if (sinks) {
            // one more term of the denominator, exp(sink), with no key and no value
            const float s = sinks[qh + h], m_new = fmaxf(m[h], s);
            const float more = (m[h] == -INFINITY) ? 0.f : expf(m[h] - m_new);
            l[h] = __builtin_fmaf(l[h], more, expf(s - m_new));
#pragma unroll
            for (int c = 0; c < ATTN_MAX_HEAD_DIM / KVA_WAVE; ++c) acc[c][h] *= more;
        }
        T *orow = out + (size_t)t * num_q_heads * value_dim + (size_t)(qh + h) * value_dim;
#pragma unroll
        for (int c = 0; c < ATTN_MAX_HEAD_DIM / KVA_WAVE; ++c) {
            const int j = lane + c * KVA_WAVE;
            if (j < value_dim) orow[j] = from_float<T>(acc[c][h] / l[h]);
        }
    }
}

// The same for few rows: FEW_BLOCKS wavefronts a token and head, a block of 64 keys each at a time.  Everything of a block is asked for, and its
// scores and exponentials are made, beside the other blocks'; what stays one after the other are the sums over the values, whose
// additions keep their order, handed on through LDS from block to block.  So bits are those of the kernel above.
#define FEW_BLOCKS 4
#define FEW_MAX_DIM 128

// Whether a block has a key that is seen, which they are, and whose places its lanes read.  Pages that hold none of a token's keys may be given back (behind a
// window, past the kept first positions): their entries in the table name no page, and only a seen key's entry may be looked up.
__host__ __device__ inline bool few_block_seen(int kb, int pos, int lo, int keep_first) {
    return kb <= pos / KVA_WAVE && !(kb * KVA_WAVE + KVA_WAVE <= lo && kb * KVA_WAVE >= keep_first);
}
__host__ __device__ inline bool few_key_seen(int key, int pos, int lo, int keep_first) {
    return key <= pos && (key >= lo || key < keep_first);
}
// (`seen`: a bit a lane.)  A key not seen: the place of the first that is, its score goes unused.
__host__ __device__ inline int few_key_read(unsigned long long seen, int lane) {
    return (seen >> lane) & 1 ? lane : __builtin_ctzll(seen);
}
// Values are read four keys of a page together: where none of them is seen, those around the first seen one.
__host__ __device__ inline int few_value_read(unsigned long long seen, int lane) {
    return (seen >> (lane & ~3)) & 15 ? lane : __builtin_ctzll(seen) & ~3;
}

// VC: rounds of 64 value elements
template <typename T, int VC>
__global__ void __launch_bounds__(KVA_WAVE * FEW_BLOCKS)
attention_few_kernel(T *__restrict__ out, const T *__restrict__ q, int q_row_stride, const T *__restrict__ k_cache,
                     const T *__restrict__ v_cache, const int *__restrict__ block_table, int max_blocks, const int *__restrict__ tok_seat,
                     const int *__restrict__ tok_pos, int num_q_heads, int num_kv_heads, int head_dim, int value_dim, int page_size,
                     float scale, int window, int keep_first, int chunk, const float *__restrict__ sinks) {
    __shared__ __attribute__((aligned(16))) float q_s[FEW_MAX_DIM], p_s[FEW_BLOCKS][KVA_WAVE];
    __shared__ long long voff_s[FEW_BLOCKS][KVA_WAVE];
    __shared__ float max_s[FEW_BLOCKS], sum_s[FEW_BLOCKS], acc_s[VC * KVA_WAVE];

    const int t = blockIdx.x, qh = blockIdx.y, tid = threadIdx.x, lane = tid % KVA_WAVE;
    const int wave = __builtin_amdgcn_readfirstlane(tid / KVA_WAVE), kvh = qh / (num_q_heads / num_kv_heads);
    const int pos = tok_pos[t];
    const int *bt = block_table + (size_t)tok_seat[t] * max_blocks;
    const T *qrow = q + (size_t)t * q_row_stride + (size_t)qh * head_dim;
    if (tid < head_dim) q_s[tid] = to_float(qrow[tid]);
    if (tid < VC * KVA_WAVE) acc_s[tid] = 0.f;
    __syncthreads();

    const int lo = kva_first_visible(pos, window, chunk), end = pos / KVA_WAVE + 1;
    // a block with no visible key: behind the window and past the kept first positions, or past the token
    auto visible = [&](int kb) { return few_block_seen(kb, pos, lo, keep_first); };
    float m = -INFINITY, l = 0.f;
    for (int base = keep_first > 0 ? 0 : lo / KVA_WAVE; base < end; base += FEW_BLOCKS) {       // uniform over the workgroup
        if ((base + FEW_BLOCKS) * KVA_WAVE <= lo && base * KVA_WAVE >= keep_first) continue;
        const int kb = base + wave;
        const bool valid = few_key_seen(kb * KVA_WAVE + lane, pos, lo, keep_first);
        const unsigned long long seen = __ballot(valid);
        const bool on = seen != 0;
        float s = -INFINITY, v[VC][16][4];
        if (on) {
            const int kkey = kb * KVA_WAVE + few_key_read(seen, lane), vkey = kb * KVA_WAVE + few_value_read(seen, lane);
            const int page = bt[kkey / page_size];
            voff_s[wave][lane] = ((long long)bt[vkey / page_size] * num_kv_heads + kvh) * (long long)value_dim * page_size + vkey % page_size;
            const T *kpage = k_cache + ((long long)page * num_kv_heads + kvh) * page_size * (long long)head_dim;
            const int krow = kkey % page_size, kc = kva_k_chunk(head_dim);
            float kv[16][4];
            auto keys = [&](int j0) {
#pragma unroll
                for (int j = 0; j < 16; ++j) Vec4<T>::load(kpage + kva_k_at(krow, j0 + 4 * j, page_size, kc), kv[j]);
            };
            float dot = 0.f;
            auto score = [&](int j0) {
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    const float4 qv = *reinterpret_cast<const float4 *>(&q_s[j0 + 4 * j]);
                    dot = __builtin_fmaf(qv.x, kv[j][0], dot);
                    dot = __builtin_fmaf(qv.y, kv[j][1], dot);
                    dot = __builtin_fmaf(qv.z, kv[j][2], dot);
                    dot = __builtin_fmaf(qv.w, kv[j][3], dot);
                }
            };
            keys(0);
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int c = 0; c < VC; ++c) {
                const T *vcol = v_cache + (long long)min(lane + c * KVA_WAVE, value_dim - 1) * page_size;
#pragma unroll
                for (int g = 0; g < 16; ++g) Vec4<T>::load(vcol + voff_s[wave][4 * g], v[c][g]);
            }
            score(0);
            for (int j0 = 64; j0 < head_dim; j0 += 64) {
                keys(j0);
                score(j0);
            }
            if (valid) s = attn_rounded(dot * scale);
        }
        const float top = wave_max(s);
        if (lane == 0) max_s[wave] = top;
        __syncthreads();
        float corr[FEW_BLOCKS], mine = 0.f, my_corr = 1.f, m_new = m;
#pragma unroll
        for (int k = 0; k < FEW_BLOCKS; ++k) {
            corr[k] = 1.f;
            if (!visible(base + k)) continue;
            const float before = m_new;
            m_new = fmaxf(before, max_s[k]);
            corr[k] = (before == -INFINITY) ? 0.f : expf(before - m_new);
            mine = k == wave ? m_new : mine;
            my_corr = k == wave ? corr[k] : my_corr;
        }
        m = m_new;
        const float p = valid ? expf(s - mine) : 0.f, sum = wave_sum(p);
        p_s[wave][lane] = p;
        if (lane == 0) sum_s[wave] = sum;
        const bool half = pos - kb * KVA_WAVE < 32;             // no keys in the block's second half
        if (on && seen != ~0ull) {
#pragma unroll
            for (int c = 0; c < VC; ++c)
#pragma unroll
                for (int g = 0; g < 16; ++g)
#pragma unroll
                    for (int u = 0; u < 4; ++u) v[c][g][u] = (seen >> (4 * g + u)) & 1 ? v[c][g][u] : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < FEW_BLOCKS; ++k)
            if (visible(base + k)) l = __builtin_fmaf(l, corr[k], sum_s[k]);
#pragma unroll 1
        for (int k = 0; k < FEW_BLOCKS; ++k) {
            if (!visible(base + k)) continue;                   // (uniform over the workgroup)
            if (k == wave) {
                float a[VC];
#pragma unroll
                for (int c = 0; c < VC; ++c) a[c] = attn_rounded(acc_s[c * KVA_WAVE + lane] * my_corr);
                auto add = [&](auto first) {
#pragma unroll
                    for (int g = decltype(first)::value; g < decltype(first)::value + 8; ++g) {
                        const float4 w = *reinterpret_cast<const float4 *>(&p_s[wave][4 * g]);
#pragma unroll
                        for (int c = 0; c < VC; ++c) {
                            a[c] = __builtin_fmaf(w.x, v[c][g][0], a[c]);
                            a[c] = __builtin_fmaf(w.y, v[c][g][1], a[c]);
                            a[c] = __builtin_fmaf(w.z, v[c][g][2], a[c]);
                            a[c] = __builtin_fmaf(w.w, v[c][g][3], a[c]);
                        }
                    }
                };
                add(std::integral_constant<int, 0>{});
                if (!half) add(std::integral_constant<int, 8>{});
#pragma unroll
                for (int c = 0; c < VC; ++c) acc_s[c * KVA_WAVE + lane] = a[c];
            }
            __syncthreads();
        }
    }
    float more = 1.f;
    if (sinks) {
        // one more term of the denominator, exp(sink), with no key and no value
        const float s = sinks[qh], m_new = fmaxf(m, s);
        more = (m == -INFINITY) ? 0.f : expf(m - m_new);
        l = __builtin_fmaf(l, more, expf(s - m_new));
    }
    if (tid < value_dim) out[(size_t)t * num_q_heads * value_dim + (size_t)qh * value_dim + tid] = from_float<T>((sinks ? acc_s[tid] * more : acc_s[tid]) / l);
}

// What the few-rows kernel's wavefront over block `kb` reads for a token at `pos`: the keys whose places its 64 lanes look up, for
// keys and for values (-1: the block is passed by).  On the host; the rule is the kernel's own.
extern "C" int kva_attention_few_reads(int pos, int window, int keep_first, int chunk, int kb, int *keys, int *values) {
    const int lo = kva_first_visible(pos, window, chunk);
    unsigned long long seen = 0;
    for (int lane = 0; lane < KVA_WAVE; ++lane)
        if (few_key_seen(kb * KVA_WAVE + lane, pos, lo, keep_first)) seen |= 1ull << lane;
    KVA_REQUIRE((seen != 0) == few_block_seen(kb, pos, lo, keep_first), "attention: block %d of position %d: the rules for blocks and for keys differ", kb, pos);
    for (int lane = 0; lane < KVA_WAVE; ++lane) {
        keys[lane] = seen ? kb * KVA_WAVE + few_key_read(seen, lane) : -1;
        values[lane] = seen ? kb * KVA_WAVE + few_value_read(seen, lane) : -1;
    }
    return KVA_OK;
}

// `longest`: no token has a position past it (only the choice of kernel goes by it).
extern "C" int kva_attention_rowwise(void *out, const void *q, int q_row_stride, const void *k_cache,
                                     const void *v_cache, const int *block_table, int max_blocks,
                                     const int *tok_seat, const int *tok_pos, int tokens,
                                     int num_q_heads, int num_kv_heads, int head_dim, int value_dim, int page_size,
                                     float scale, int window, int keep_first, int chunk, const float *sinks, int longest,
                                     int dtype, hipStream_t stream) {
    KVA_REQUIRE(tokens >= 0 && num_q_heads > 0 && num_kv_heads > 0 && page_size > 0 && max_blocks > 0,
                "attention: bad sizes");
    KVA_REQUIRE(num_q_heads % num_kv_heads == 0, "attention: %d query heads is not a multiple of %d kv heads",
                num_q_heads, num_kv_heads);
    KVA_REQUIRE(head_dim % 4 == 0 && head_dim <= ATTN_MAX_HEAD_DIM,
                "attention: head_dim %d must be a multiple of 4 and at most %d", head_dim,
                ATTN_MAX_HEAD_DIM);
    KVA_REQUIRE(q_row_stride % 4 == 0, "attention: query row stride %d must be a multiple of 4", q_row_stride);
    KVA_REQUIRE(num_q_heads <= 65535, "attention: too many heads");
    KVA_REQUIRE(window >= 0 && keep_first >= 0 && chunk >= 0 && !(window > 0 && chunk > 0),
                "attention: negative window, kept first positions or chunk, or a window together with chunks");
    KVA_REQUIRE(value_dim > 0 && value_dim <= ATTN_MAX_HEAD_DIM, "attention: value size %d must be at most %d",
                value_dim, ATTN_MAX_HEAD_DIM);
    if (window == 0) keep_first = 0;
    if (tokens == 0) return KVA_OK;
    const size_t element = dtype == KVA_F32 ? 4 : 2;
    const int fours = page_size % 4 == 0 && (uintptr_t)v_cache % (4 * element) == 0;
    const int group = num_q_heads / num_kv_heads;
    // Heads together: wavefronts are few at first and then the heads' own chains of additions bound them (1 / 2 / 4 heads
    // of 64, fp32, us: 1 token at 200 keys 11 / 14 / 18, 32 at 500 25 / 27 / 35, 64 at 1,000 63 / 61 / 77), from some
    // 3,000 rows of a head on the reads do: 128 tokens of 32 heads 16 / 12 / 13, 201 26 / 21 / 22, 603 63 / 40 / 35;
    // three: 603 tokens of 24 heads of 128 over 8 key heads 93 -> 48.
    const long long rows = (long long)tokens * num_q_heads;
    const int together = rows >= 12288 && group % 4 == 0 ? 4
                         : rows >= 6144 && group % 3 == 0 ? 3
                         : rows >= 3072 && group % 2 == 0 ? 2 : 1;
    // Few rows with more than a block of keys: four blocks at a time, whose chains of additions are 6.5 us for two blocks and 2 more for each
    // one after the other.  One wavefront / four, fp32, us a call: 3 tokens of 32 heads of 64 at 66 / 130 / 201 / 1,000 keys 6.5 / 8.4 / 10.2 /
    // 42.5 -> 5.6 / 6.2 / 7.0 / 22.9, heads of 128 9.0 / 11.9 / 16.3 / 64.3 -> 7.7 / 8.7 / 10.5 / 36.2; 16 tokens (512 rows) at 201 keys 11.1 -> 8.6
    // (heads of 128 16.2 -> 13.5); but 32 tokens 13.7 -> 15.8, and at 40 keys, one block, 4.6 -> 5.2.
    const long long span = window > 0 ? (long long)window + keep_first : chunk > 0 ? chunk : longest;      // keys that a token sees, at most
    const bool few = fours && rows <= 512 && span > KVA_WAVE && longest > KVA_WAVE && head_dim % 64 == 0 && head_dim <= FEW_MAX_DIM &&
                     value_dim <= FEW_MAX_DIM;
    // (a head alone whose elements are whole rounds of 64 loads' worth; of others the last round would go one load at a time)
#define KVA_ROWWISE(T, H, ALL)                                                                                         \
    hipLaunchKernelGGL((attention_rowwise_kernel<T, H, ALL>), dim3(tokens, num_q_heads / H), dim3(KVA_WAVE), 0, stream, (T *)out, \
                       (const T *)q, q_row_stride, (const T *)k_cache, (const T *)v_cache, block_table, max_blocks,    \
                       tok_seat, tok_pos, num_q_heads, num_kv_heads, head_dim, value_dim, page_size, fours, scale,     \
                       window, keep_first, chunk, sinks)
#define KVA_FEW(T, VC)                                                                                                 \
    hipLaunchKernelGGL((attention_few_kernel<T, VC>), dim3(tokens, num_q_heads), dim3(KVA_WAVE * FEW_BLOCKS), 0, stream, (T *)out, \
                       (const T *)q, q_row_stride, (const T *)k_cache, (const T *)v_cache, block_table, max_blocks,    \
                       tok_seat, tok_pos, num_q_heads, num_kv_heads, head_dim, value_dim, page_size, scale, window,    \
                       keep_first, chunk, sinks)
#define KVA_ROWWISE_HEADS(T)                                                                                           \
    do {                                                                                                               \
        if (few && value_dim <= KVA_WAVE) KVA_FEW(T, 1);                                                               \
        else if (few) KVA_FEW(T, 2);                                                                                   \
        else                                                                                                           \
        if (together == 4) KVA_ROWWISE(T, 4, false);                                                                          \
        else if (together == 3) KVA_ROWWISE(T, 3, false);                                                                     \
        else if (together == 2) KVA_ROWWISE(T, 2, false);                                                                     \
        else if (head_dim % 64 == 0) KVA_ROWWISE(T, 1, true);                                                          \
        else KVA_ROWWISE(T, 1, false);                                                                                 \
    } while (0)
    if (dtype == KVA_F32) KVA_ROWWISE_HEADS(float);
    else if (dtype == KVA_BF16) KVA_ROWWISE_HEADS(bf16_t);
    else KVA_REQUIRE(false, "attention: unsupported dtype %d", dtype);
#undef KVA_ROWWISE_HEADS
#undef KVA_ROWWISE
#undef KVA_FEW
    KVA_CHECK_LAUNCH("attention_rowwise");
    return KVA_OK;
}

// ---- attention over low-rank entries: the plain kernel ----------------------------------------
//
// Every token keeps ONE row of `key_dim` = rank + rot elements for all heads: a latent vector of
// `rank` elements (the value, and - through the query-side product with the key expansion - the
// unrotated part of the key) followed by the rotated key part.  The query row of a head has the
// same layout, so score = q . row * scale over all key_dim elements, and the head's output is the
// probability-weighted sum of the first `rank` elements of the rows; the caller expands it to the
// head's values.  Rows lie in pages [page_size, key_dim].  Same walk over blocks of 64 keys at
// absolute positions, window / kept first positions and sink term as the kernel above.
#define LAT_MAX_KEY_DIM 1280
#define LAT_MAX_RANK 1024

template <typename T>
__global__ void __launch_bounds__(KVA_WAVE)
latent_attention_rowwise_kernel(T *__restrict__ out, const T *__restrict__ q, const T *__restrict__ cache,
                                const int *__restrict__ block_table, int max_blocks,
                                const int *__restrict__ tok_seat, const int *__restrict__ tok_pos, int heads,
                                int rank, int key_dim, int page_size, float scale, int window, int keep_first,
                                const float *__restrict__ sinks) {
    __shared__ float q_s[LAT_MAX_KEY_DIM];
    __shared__ float p_s[KVA_WAVE];
    __shared__ long long off_s[KVA_WAVE];
    const int t = blockIdx.x, qh = blockIdx.y, lane = threadIdx.x;
    const int pos = tok_pos[t];
    const int *bt = block_table + (size_t)tok_seat[t] * max_blocks;
    const T *qrow = q + ((size_t)t * heads + qh) * key_dim;
    for (int j = lane; j < key_dim; j += KVA_WAVE) q_s[j] = to_float(qrow[j]);
    __syncthreads();

    const int lo = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
    float m = -INFINITY, l = 0.f;
    float acc[LAT_MAX_RANK / KVA_WAVE];
#pragma unroll
    for (int c = 0; c < LAT_MAX_RANK / KVA_WAVE; ++c) acc[c] = 0.f;

    for (int kb = 0; kb <= pos / KVA_WAVE; ++kb) {
        if (kb * KVA_WAVE + KVA_WAVE <= lo && kb * KVA_WAVE >= keep_first) continue;
        const int key = kb * KVA_WAVE + lane;
        const bool valid = key <= pos && (key >= lo || key < keep_first);
        float s = -INFINITY;
        long long row_off = -1;
        if (valid) {
            row_off = ((long long)bt[key / page_size] * page_size + key % page_size) * key_dim;
            const T *krow = cache + row_off;
            float dot = 0.f;
            for (int j = 0; j < key_dim; ++j) dot += q_s[j] * to_float(krow[j]);
            s = dot * scale;
        }
        const float m_new = fmaxf(m, wave_max(s));
        const float corr = (m == -INFINITY) ? 0.f : expf(m - m_new);
        const float p = valid ? expf(s - m_new) : 0.f;
        l = l * corr + wave_sum(p);
        m = m_new;
        __syncthreads();
        p_s[lane] = p;
        off_s[lane] = row_off;
        __syncthreads();
        const int last = (pos - kb * KVA_WAVE < KVA_WAVE - 1) ? pos - kb * KVA_WAVE : KVA_WAVE - 1;
#pragma unroll
        for (int c = 0; c < LAT_MAX_RANK / KVA_WAVE; ++c) {
            const int j = lane + c * KVA_WAVE;
            if (j < rank) {
                float a = acc[c] * corr;
                for (int i = 0; i <= last; ++i)
                    if (off_s[i] >= 0) a += p_s[i] * to_float(cache[off_s[i] + j]);
                acc[c] = a;
            }
        }
    }
    if (sinks) {
        const float s = sinks[qh], m_new = fmaxf(m, s);
        const float corr = (m == -INFINITY) ? 0.f : expf(m - m_new);
        l = l * corr + expf(s - m_new);
#pragma unroll
        for (int c = 0; c < LAT_MAX_RANK / KVA_WAVE; ++c) acc[c] *= corr;
    }
    T *orow = out + ((size_t)t * heads + qh) * rank;
#pragma unroll
    for (int c = 0; c < LAT_MAX_RANK / KVA_WAVE; ++c) {
        const int j = lane + c * KVA_WAVE;
        if (j < rank) orow[j] = from_float<T>(acc[c] / l);
    }
}

extern "C" int kva_latent_attention_rowwise(void *out, const void *q, const void *cache, const int *block_table,
                                            int max_blocks, const int *tok_seat, const int *tok_pos, int tokens,
                                            int heads, int rank, int key_dim, int page_size, float scale,
                                            int window, int keep_first, const float *sinks, int dtype,
                                            hipStream_t stream) {
    KVA_REQUIRE(tokens >= 0 && heads > 0 && heads <= 65535 && page_size > 0 && max_blocks > 0,
                "latent attention: bad sizes");
    KVA_REQUIRE(rank > 0 && rank <= LAT_MAX_RANK && key_dim >= rank && key_dim <= LAT_MAX_KEY_DIM,
                "latent attention: rank %d (at most %d) and row size %d (at most %d) do not fit", rank,
                LAT_MAX_RANK, key_dim, LAT_MAX_KEY_DIM);
    KVA_REQUIRE(window >= 0 && keep_first >= 0, "latent attention: negative window or kept first positions");
    if (window == 0) keep_first = 0;
    if (tokens == 0) return KVA_OK;
    dim3 grid(tokens, heads), block(KVA_WAVE);
    if (dtype == KVA_F32)
        hipLaunchKernelGGL(latent_attention_rowwise_kernel<float>, grid, block, 0, stream, (float *)out,
                           (const float *)q, (const float *)cache, block_table, max_blocks, tok_seat, tok_pos,
                           heads, rank, key_dim, page_size, scale, window, keep_first, sinks);
    else if (dtype == KVA_BF16)
        hipLaunchKernelGGL(latent_attention_rowwise_kernel<bf16_t>, grid, block, 0, stream, (bf16_t *)out,
                           (const bf16_t *)q, (const bf16_t *)cache, block_table, max_blocks, tok_seat, tok_pos,
                           heads, rank, key_dim, page_size, scale, window, keep_first, sinks);
    else KVA_REQUIRE(false, "latent attention: unsupported dtype %d", dtype);
    KVA_CHECK_LAUNCH("latent_attention_rowwise");
    return KVA_OK;
}
