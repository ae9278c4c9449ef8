// Rotary position encoding of Q and K fused with the write of K and V into the paged cache.
//
// The reference does this in three launches per layer: ropePackedKernel on Q, on K
// (base/src/kernels.cu:289-319) and scatterKVPackedKernel
// (paged_attention/src/kernels.cu:335-363).  Pairing is rotate-half: inside a head, element j
// pairs with j + rot/2 and both use angle index j:
//     out[j]         = x[j] * cos - x[j + rot/2] * sin
//     out[j + rot/2] = x[j] * sin + x[j + rot/2] * cos
// cos and sin come from fp32 tables [max_positions, rot/2] built once on the host.
// K is rotated BEFORE it is cached, V is cached as it is.
//
// Cache layout: K is [num_pages, num_kv_heads, head_dim / 8, page_size, 8] (kv_layout.h: a key's
// elements in chunks of 8, the chunks of all keys of a page next to each other); V is stored transposed
// inside a page, [num_pages, num_kv_heads, head_dim, page_size], so that the attention kernels
// can load "several keys of one value dimension" as one vector (the matrix-core operand layout
// of P*V).  Slot s of the slot mapping is page s / page_size, row s % page_size.  A negative
// slot skips the write.
#include "common.h"
#include "kv_layout.h"
#include <algorithm>

template <typename T>
__global__ void rope_kv_write_kernel(T *__restrict__ qkv, T *__restrict__ k_cache,
                                     T *__restrict__ v_cache, const float *__restrict__ cos_table,
                                     const float *__restrict__ sin_table,
                                     const int *__restrict__ positions,
                                     const int *__restrict__ slot_mapping, int num_q_heads,
                                     int num_kv_heads, int head_dim, int rot_dim, int page_size,
                                     int write_cache) {
    const int t = blockIdx.x;
    const int row_width = (num_q_heads + 2 * num_kv_heads) * head_dim;
    T *row = qkv + (size_t)t * row_width;
    const int pos = positions[t];
    const int half = rot_dim / 2;
    const float *cs = cos_table ? cos_table + (size_t)pos * half : nullptr;
    const float *sn = sin_table ? sin_table + (size_t)pos * half : nullptr;

    int slot = -1;
    if (write_cache) slot = slot_mapping[t];
    const int page = slot >= 0 ? slot / page_size : 0;
    const int off = slot >= 0 ? slot % page_size : 0;

    // work item = (head among q and k heads, pair index in [0, head_dim/2)); pairs beyond the
    // rotated part (partial rotary) pass two plain elements through
    const int pairs_per_head = head_dim / 2;
    const int qk_heads = num_q_heads + num_kv_heads;
    for (int w = threadIdx.x; w < qk_heads * pairs_per_head; w += blockDim.x) {
        const int head = w / pairs_per_head;
        const int p = w % pairs_per_head;
        T *h = row + (size_t)head * head_dim;
        int i1, i2;
        float o1, o2;
        if (p < half) {
            i1 = p;
            i2 = p + half;
            const float x1 = to_float(h[i1]), x2 = to_float(h[i2]);
            if (cs) {
                const float c = cs[p], s = sn[p];
                o1 = x1 * c - x2 * s;
                o2 = x1 * s + x2 * c;
            } else {
                o1 = x1;
                o2 = x2;
            }
        } else {
            i1 = rot_dim + 2 * (p - half);
            i2 = i1 + 1;
            o1 = to_float(h[i1]);
            o2 = to_float(h[i2]);
        }
        const T r1 = from_float<T>(o1), r2 = from_float<T>(o2);
        if (head < num_q_heads) {
            h[i1] = r1;
            h[i2] = r2;
        } else if (slot >= 0) {
            const int kvh = head - num_q_heads;
            T *dst = k_cache + ((size_t)page * num_kv_heads + kvh) * page_size * head_dim;
            const int kc = kva_k_chunk(head_dim);
            dst[kva_k_at(off, i1, page_size, kc)] = r1;
            dst[kva_k_at(off, i2, page_size, kc)] = r2;
        }
    }
    if (slot >= 0) {
        const T *v = row + (size_t)(num_q_heads + num_kv_heads) * head_dim;
        for (int w = threadIdx.x; w < num_kv_heads * head_dim; w += blockDim.x) {
            const int kvh = w / head_dim, j = w % head_dim;
            v_cache[(((size_t)page * num_kv_heads + kvh) * head_dim + j) * page_size + off] = v[w];
        }
    }
}

// Full rotary (rot_dim == head_dim), head_dim a multiple of 16: a thread rotates as many pairs at a time as 16 bytes hold elements.
// Few tokens: a token's heads go to several workgroups (3 tokens of 32 + 2 x 8 heads of 64 / 128, fp32 2.6 / 2.6 us, pair by
// pair in one workgroup 4.5 / 7.2; bf16 3.0 / 3.1, in one workgroup 3.1 / 4.1).
template <typename T>
struct RopeVec {
    static constexpr int N = 16 / sizeof(T);
    __device__ static inline void load(const T *p, float (&f)[N]) {
        const uint4 v = *reinterpret_cast<const uint4 *>(p);
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < N; ++i)
            f[i] = __uint_as_float(N == 4 ? w[i % 4] : i % 2 ? w[i / 2] & 0xffff0000u : w[i / 2] << 16);
    }
    __device__ static inline void store(T *p, const float (&f)[N]) {
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            w[i] = N == 4 ? __float_as_uint(f[i % N])
                          : (uint32_t)float_to_bf16_bits(f[2 * i % N]) | ((uint32_t)float_to_bf16_bits(f[(2 * i + 1) % N]) << 16);
        *reinterpret_cast<uint4 *>(p) = make_uint4(w[0], w[1], w[2], w[3]);
    }
};

template <typename T>
__global__ void rope_kv_write_vec_kernel(T *__restrict__ qkv, T *__restrict__ k_cache, T *__restrict__ v_cache,
                                         const float *__restrict__ cos_table, const float *__restrict__ sin_table,
                                         const int *__restrict__ positions,
                                         const int *__restrict__ slot_mapping, int num_q_heads,
                                         int num_kv_heads, int head_dim, int page_size, int write_cache) {
    constexpr int N = RopeVec<T>::N;
    const int t = blockIdx.x, first = blockIdx.y * blockDim.x + threadIdx.x, step = gridDim.y * blockDim.x;
    const int row_width = (num_q_heads + 2 * num_kv_heads) * head_dim;
    T *row = qkv + (size_t)t * row_width;
    const int pos = positions[t];
    const int half = head_dim / 2;
    const float *cs = cos_table + (size_t)pos * half;
    const float *sn = sin_table + (size_t)pos * half;
    int slot = -1;
    if (write_cache) slot = slot_mapping[t];
    const int page = slot >= 0 ? slot / page_size : 0;
    const int off = slot >= 0 ? slot % page_size : 0;
    const int chunks = half / N;
    const int qk_heads = num_q_heads + num_kv_heads;
    for (int w = first; w < qk_heads * chunks; w += step) {
        const int head = w / chunks, p0 = (w % chunks) * N;
        if (head >= num_q_heads && slot < 0) continue;
        T *h = row + (size_t)head * head_dim;
        float x1[N], x2[N], c[N], s[N], o1[N], o2[N];
        RopeVec<T>::load(h + p0, x1);
        RopeVec<T>::load(h + half + p0, x2);
#pragma unroll
        for (int j = 0; j < N; j += 4) {
            const float4 cv = *reinterpret_cast<const float4 *>(cs + p0 + j), sv = *reinterpret_cast<const float4 *>(sn + p0 + j);
            c[j] = cv.x; c[j + 1] = cv.y; c[j + 2] = cv.z; c[j + 3] = cv.w;
            s[j] = sv.x; s[j + 1] = sv.y; s[j + 2] = sv.z; s[j + 3] = sv.w;
        }
#pragma unroll
        for (int j = 0; j < N; ++j) {
            o1[j] = x1[j] * c[j] - x2[j] * s[j];
            o2[j] = x1[j] * s[j] + x2[j] * c[j];
        }
        if (head >= num_q_heads) {
            // (head_dim is a multiple of 16 here: chunks of 8, of which p0 and half + p0 start one or its second half)
            T *dst = k_cache + ((size_t)page * num_kv_heads + (head - num_q_heads)) * page_size * head_dim;
            RopeVec<T>::store(dst + kva_k_at(off, p0, page_size, 8), o1);
            RopeVec<T>::store(dst + kva_k_at(off, half + p0, page_size, 8), o2);
        } else {
            RopeVec<T>::store(h + p0, o1);
            RopeVec<T>::store(h + half + p0, o2);
        }
    }
    if (slot >= 0) {
        const T *v = row + (size_t)(num_q_heads + num_kv_heads) * head_dim;
        for (int w = first; w < num_kv_heads * head_dim; w += step) {
            const int kvh = w / head_dim, j = w % head_dim;
            v_cache[(((size_t)page * num_kv_heads + kvh) * head_dim + j) * page_size + off] = v[w];
        }
    }
}

// Many tokens in bf16 with a cache: a workgroup takes 16 neighbouring tokens and some of the heads, q's, k's or v's (blockIdx.y).
// With a workgroup a token the cache bounds it: neighbouring tokens' keys and values share cache lines, an element of V goes a page's
// row further than the one before it, and eight dies write 16 and 2 bytes of a line each.  Here a line is one workgroup's, and eight
// keys that fill eight aligned places of a page go out as 16 bytes of V at a time, turned round in LDS.  A thread keeps its token's
// cosines and sines over all of its heads.  us, a workgroup a token and this: 1,203 tokens (portions that begin anywhere) / 2,048 of
// 32 + 2 x 8 heads of 64 8.5 / 12.1 and 7.6 / 8.1 (3 TB/s), 8,190 of 128 75 and 41 (4.9 TB/s).  (Runs of four and two keys as one store,
// too: 9.2 at 1,203 tokens, the search for them takes longer than the stores.)  Few tokens are too few workgroups with a long chain
// each: rope_tokens_wide.
#define ROPE_TOKENS 16
#define ROPE_HEADS 2                    // of q or k a thread takes at once
#define ROPE_V_COLS 256

struct RopeWide {
    bf16_t *qkv, *k_cache, *v_cache;
    const float *cos_table, *sin_table;
    const int *positions, *slot_mapping;
    int tokens, num_q_heads, num_kv_heads, head_dim, page_size;
    int lanes, q_blocks, k_blocks;              // threads that share a token's chunk; workgroups of 16 tokens' q and k heads
};

__global__ void __launch_bounds__(256)
rope_kv_write_wide_kernel(RopeWide a) {
    __shared__ __attribute__((aligned(16))) uint16_t turn[ROPE_TOKENS][ROPE_V_COLS + 8];
    const int t0 = blockIdx.x * ROPE_TOKENS, d = a.head_dim, half = d / 2, chunks = half / 8, tid = threadIdx.x;
    const size_t row_width = (size_t)(a.num_q_heads + 2 * a.num_kv_heads) * d;
    int block = blockIdx.y;
    if (block < a.q_blocks + a.k_blocks) {
        const bool keys = block >= a.q_blocks;
        if (keys) block -= a.q_blocks;
        // q: a token's chunks and heads by neighbouring threads, as they lie in the row; k: the tokens, as they lie in the cache
        const int per = chunks * a.lanes, token = keys ? tid % ROPE_TOKENS : tid / per, rest = keys ? tid / ROPE_TOKENS : tid % per, t = t0 + token;
        if (token >= ROPE_TOKENS || rest >= per || t >= a.tokens) return;
        const int chunk = rest % chunks, lane = rest / chunks, p0 = 8 * chunk, heads = keys ? a.num_kv_heads : a.num_q_heads;
        const int slot = keys ? a.slot_mapping[t] : 0;
        if (slot < 0) return;
        bf16_t *row = a.qkv + (size_t)t * row_width + (keys ? (size_t)a.num_q_heads * d : 0);
        const float *cs = a.cos_table + (size_t)a.positions[t] * half + p0, *sn = a.sin_table + (size_t)a.positions[t] * half + p0;
        float x1[ROPE_HEADS][8], x2[ROPE_HEADS][8], c[8], s[8];
        const int head0 = block * a.lanes * ROPE_HEADS + lane;
#pragma unroll
        for (int i = 0; i < ROPE_HEADS; ++i) {
            const bf16_t *h = row + (size_t)min(head0 + i * a.lanes, heads - 1) * d + p0;
            RopeVec<bf16_t>::load(h, x1[i]);
            RopeVec<bf16_t>::load(h + half, x2[i]);
        }
#pragma unroll
        for (int j = 0; j < 8; j += 4) {
            const float4 cv = *reinterpret_cast<const float4 *>(cs + j), sv = *reinterpret_cast<const float4 *>(sn + j);
            c[j] = cv.x; c[j + 1] = cv.y; c[j + 2] = cv.z; c[j + 3] = cv.w;
            s[j] = sv.x; s[j + 1] = sv.y; s[j + 2] = sv.z; s[j + 3] = sv.w;
        }
#pragma unroll
        for (int i = 0; i < ROPE_HEADS; ++i) {
            const int head = head0 + i * a.lanes;
            if (head >= heads) return;
            float o1[8], o2[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                o1[j] = fmaf(x1[i][j], c[j], -(x2[i][j] * s[j]));       // (as the compiler contracts it in the other kernels)
                o2[j] = fmaf(x2[i][j], c[j], x1[i][j] * s[j]);
            }
            bf16_t *to1 = row + (size_t)head * d + p0, *to2 = to1 + half;
            if (keys) {
                bf16_t *dst = a.k_cache + ((size_t)(slot / a.page_size) * a.num_kv_heads + head) * a.page_size * d;
                to1 = dst + kva_k_at(slot % a.page_size, p0, a.page_size, 8);
                to2 = dst + kva_k_at(slot % a.page_size, half + p0, a.page_size, 8);
            }
            RopeVec<bf16_t>::store(to1, o1);
            RopeVec<bf16_t>::store(to2, o2);
        }
        return;
    }
    const int col0 = (block - a.q_blocks - a.k_blocks) * ROPE_V_COLS, cols = min(ROPE_V_COLS, a.num_kv_heads * d - col0);
    const bf16_t *v = a.qkv + (size_t)(a.num_q_heads + a.num_kv_heads) * d + col0;
    int slot[ROPE_TOKENS];
#pragma unroll
    for (int i = 0; i < ROPE_TOKENS; ++i) {
        slot[i] = a.slot_mapping[min(t0 + i, a.tokens - 1)];
        if (t0 + i >= a.tokens) slot[i] = -1;
    }
#pragma unroll
    for (int i = 0; i < ROPE_TOKENS * ROPE_V_COLS / 8 / 256; ++i) {
        const int token = tid / (ROPE_V_COLS / 8) + i * (256 / (ROPE_V_COLS / 8)), col = 8 * (tid % (ROPE_V_COLS / 8));
        if (t0 + token < a.tokens && col < cols)            // (a whole number of 16 columns)
            *reinterpret_cast<uint4 *>(&turn[token][col]) = *reinterpret_cast<const uint4 *>(v + (size_t)(t0 + token) * row_width + col);
    }
    __syncthreads();
    if (tid >= cols) return;
    const int kvh = (col0 + tid) / d, j = (col0 + tid) % d;
    uint32_t pair[ROPE_TOKENS / 2];
#pragma unroll
    for (int i = 0; i < ROPE_TOKENS; i += 2) pair[i / 2] = (uint32_t)turn[i][tid] | ((uint32_t)turn[i + 1][tid] << 16);
    int next = 0;
#pragma unroll
    for (int i = 0; i < ROPE_TOKENS; ++i) {
        if (i < next || slot[i] < 0) continue;              // (the same in all threads)
        uint16_t *dst = reinterpret_cast<uint16_t *>(a.v_cache) +
                        (((size_t)(slot[i] / a.page_size) * a.num_kv_heads + kvh) * d + j) * a.page_size + slot[i] % a.page_size;
        bool run = i + 8 <= ROPE_TOKENS && slot[i] % 8 == 0;
#pragma unroll
        for (int k = 1; k < 8; ++k) run = run && slot[(i + k) % ROPE_TOKENS] == slot[i] + k;
        if (run) {
            uint32_t w[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int at = (i / 2 + k) % (ROPE_TOKENS / 2), then = (at + 1) % (ROPE_TOKENS / 2);
                w[k] = i % 2 ? (pair[at] >> 16) | (pair[then] << 16) : pair[at];
            }
            *reinterpret_cast<uint4 *>(dst) = make_uint4(w[0], w[1], w[2], w[3]);
            next = i + 8;
        } else {
            *dst = (uint16_t)(i % 2 ? pair[i / 2] >> 16 : pair[i / 2] & 0xffffu);
        }
    }
}

// From where on a step in bf16 goes to rope_kv_write_wide_kernel: 2^19 elements of V, or 1,536 tokens.  Below, a workgroup of 16 tokens
// does what 16 would at the same time: 65 / 256 tokens of a prompt of 32 + 2 x 8 heads of 64 3.5 / 4.0 us with a workgroup a token and
// 4.9 / 4.4, decoded tokens with a page each (single stores of V) 3.4 / 4.3 and 5.4 / 6.0.  Timed over steps of 65 to 7,168 tokens, 0 to
// 1,024 of them decoded, beside portions of 2 to 1,024, six geometries: the lines cross at 750 tokens with 512 elements of V a token,
// 380 with 1,024, 900 with 256, 1,050 with 128 (whole prompts alone earlier, 350, 150, 550, 550), and where the step's entries begin
// and how long they are moves them little.  All 1,842 steps: 0.86 of a workgroup a token, 0.91 with this kernel from 65 tokens on, 0.85
// with the faster one every time; what stays slower are steps of 500 and more decoded tokens without long portions (up to 1.16).  Without a cache nothing is
// turned round and this kernel has nothing to give: 1.39 at 65 tokens, 1.08 at 2,048, 0.94 to 1.10 at 4,096.
static bool rope_tokens_wide(int tokens, int num_kv_heads, int head_dim, int write_cache) {
    return write_cache && tokens > 64 && (tokens >= 1536 || (size_t)tokens * num_kv_heads * head_dim >= (size_t)1 << 19);
}

extern "C" int kva_rope_tokens_wide(int tokens, int num_kv_heads, int head_dim, int write_cache) {
    return rope_tokens_wide(tokens, num_kv_heads, head_dim, write_cache);
}

extern "C" int kva_rope_kv_write(void *qkv, void *k_cache, void *v_cache, const float *cos_table,
                                 const float *sin_table, const int *positions,
                                 const int *slot_mapping, int tokens, int num_q_heads,
                                 int num_kv_heads, int head_dim, int rot_dim, int page_size,
                                 int write_cache, int dtype, hipStream_t stream) {
    KVA_REQUIRE(tokens >= 0 && num_q_heads > 0 && num_kv_heads > 0, "rope_kv_write: bad sizes");
    KVA_REQUIRE(head_dim > 0 && head_dim % 2 == 0, "rope_kv_write: head_dim %d must be even", head_dim);
    KVA_REQUIRE(rot_dim >= 0 && rot_dim <= head_dim && rot_dim % 2 == 0,
                "rope_kv_write: rotary dim %d must be even and at most head_dim %d", rot_dim, head_dim);
    KVA_REQUIRE((cos_table == nullptr) == (sin_table == nullptr), "rope_kv_write: one table missing");
    KVA_REQUIRE(!write_cache || (k_cache && v_cache && slot_mapping && page_size > 0),
                "rope_kv_write: cache write asked for without cache, slots or page size");
    if (tokens == 0) return KVA_OK;
    dim3 grid(tokens), block(256);
    const uintptr_t all = (uintptr_t)qkv | (uintptr_t)k_cache | (uintptr_t)cos_table | (uintptr_t)sin_table;
    if (cos_table && rot_dim == head_dim && head_dim % 16 == 0 && (dtype == KVA_BF16 || (dtype == KVA_F32 && all % 16 == 0))) {
        if (dtype == KVA_BF16 && rope_tokens_wide(tokens, num_kv_heads, head_dim, write_cache) && head_dim <= 256 &&
            ((all | (uintptr_t)v_cache) & 15) == 0 && page_size % 8 == 0) {
            const int lanes = 256 / (ROPE_TOKENS * (head_dim / 16)), heads = lanes * ROPE_HEADS;
            const int q_blocks = (num_q_heads + heads - 1) / heads, k_blocks = (num_kv_heads + heads - 1) / heads;
            const int v_blocks = (num_kv_heads * head_dim + ROPE_V_COLS - 1) / ROPE_V_COLS;
            if (q_blocks + k_blocks + v_blocks <= 65535) {
                const RopeWide a{(bf16_t *)qkv, (bf16_t *)k_cache, (bf16_t *)v_cache, cos_table, sin_table, positions, slot_mapping, tokens, num_q_heads,
                                 num_kv_heads, head_dim, page_size, lanes, q_blocks, k_blocks};
                hipLaunchKernelGGL(rope_kv_write_wide_kernel, dim3((tokens + ROPE_TOKENS - 1) / ROPE_TOKENS, q_blocks + k_blocks + v_blocks), block, 0,
                                   stream, a);
                KVA_CHECK_LAUNCH("rope_kv_write");
                return KVA_OK;
            }
        }
        const int vectors = (num_q_heads + num_kv_heads) * head_dim / 2 / (dtype == KVA_BF16 ? 8 : 4);
        const dim3 vgrid(tokens, tokens <= 64 ? std::min(65535, (std::max(vectors, num_kv_heads * head_dim) + 255) / 256) : 1);
        if (dtype == KVA_BF16)
            hipLaunchKernelGGL(rope_kv_write_vec_kernel<bf16_t>, vgrid, block, 0, stream, (bf16_t *)qkv, (bf16_t *)k_cache, (bf16_t *)v_cache,
                               cos_table, sin_table, positions, slot_mapping, num_q_heads, num_kv_heads, head_dim, page_size, write_cache);
        else
            hipLaunchKernelGGL(rope_kv_write_vec_kernel<float>, vgrid, block, 0, stream, (float *)qkv, (float *)k_cache, (float *)v_cache,
                               cos_table, sin_table, positions, slot_mapping, num_q_heads, num_kv_heads, head_dim, page_size, write_cache);
        KVA_CHECK_LAUNCH("rope_kv_write");
        return KVA_OK;
    }
    if (dtype == KVA_F32)
        hipLaunchKernelGGL(rope_kv_write_kernel<float>, grid, block, 0, stream, (float *)qkv,
                           (float *)k_cache, (float *)v_cache, cos_table, sin_table, positions,
                           slot_mapping, num_q_heads, num_kv_heads, head_dim, rot_dim, page_size,
                           write_cache);
    else if (dtype == KVA_BF16)
        hipLaunchKernelGGL(rope_kv_write_kernel<bf16_t>, grid, block, 0, stream, (bf16_t *)qkv,
                           (bf16_t *)k_cache, (bf16_t *)v_cache, cos_table, sin_table, positions,
                           slot_mapping, num_q_heads, num_kv_heads, head_dim, rot_dim, page_size,
                           write_cache);
    else KVA_REQUIRE(false, "rope_kv_write: unsupported dtype %d", dtype);
    KVA_CHECK_LAUNCH("rope_kv_write");
    return KVA_OK;
}
