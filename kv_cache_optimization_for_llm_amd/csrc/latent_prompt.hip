// Attention over low-rank entries for prompts: keys and values expanded (bf16, gfx950).
//
// latent_attention_mfma.hip attends over the cached rows themselves - rank + rot elements a key, rank a value, for
// every head - which is what a decoded token wants: each row is read once for all heads.  A prompt's tokens see
// the same keys many times over, and per (token, key, head) that form costs 2 (rank + rot + rank) operations against
// 2 (dim + rot + vdim) over keys and values expanded per head: 2,176 against 640 at rank 512 and heads of
// 128 + 64 / 128.  Expanding a key costs 2 rank (dim + vdim) per head once, as much as 85 tokens looking at it save.
// Two kernels:
//   * latent_expand_kernel: the entries' whole contexts (cached rows, by page) times [U_k ; U_v], rounded to
//     bf16, keys' heads and then values' heads one after the other, a position a row of 128 elements; the rotated key parts,
//     which all heads share, are laid side by side in the same launch.
//   * latent_prompt_kernel: a workgroup takes 64 tokens of an entry and one head, a wavefront 16 of the tokens;
//     latent_prompt_wide_kernel: a wavefront 32 of the tokens and half of the keys (latent_prompt_wide says where).  As in
//     latent_attention_mfma.hip everything is transposed, S^T = K Q^T and O^T = V^T P^T; blocks of 32 or 64 keys go through LDS
//     for the four wavefronts (the next one's loads in flight), V^T is read there with the transposing load.  The
//     queries' rotation happens as they are loaded, sink and output gate where the result is normalised.
// A SIMD issues matrix products (20 of 16 cycles a block and wavefront; wide: 40) or the softmax's vector work (about as
// much), and LDS gives the four wavefronts 20 KiB each a block (640 cycles): without the wide form's second use of what is read, the
// three are about even.  The workgroups with the most keys are launched first (wide: the longest beside the shortest); a
// head's workgroups are on one die where the heads are a multiple of eight, whose L2 holds its keys and values.
//
// us a layer, one prompt of 2,048 tokens, 16 heads of 128 + 64 / 128, rank 512: over the cached rows 183, the products
// per head in front and behind 38 + 21; expanded 18 + 69 (21.5 GFLOP in the second: 312 TFLOP/s).
#include "common.h"
#include "lds_product.h"
#include <math.h>

#define LP_LOG2E 1.44269504088896340736f
#define LP_DIM 128                  // a head's plain query / key elements, rotated ones, values
#define LP_ROT 64
#define LP_VDIM 128
static_assert(LP_DIM == LP_VDIM, "expanded keys and values lie in rows of one size");
#define LP_BLOCK 32                 // keys a block
#define LP_WIDE_BLOCK 64            // ... of the wide kernel
#define LP_ROWS 64                  // tokens a workgroup

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

__global__ void __launch_bounds__(256, 2)
latent_expand_kernel(LatentPrompt a) {
    typedef LdsProduct<4, 8, 3> Product;
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
            if (p < keys) *reinterpret_cast<uint4 *>(a.rot + (base + p) * LP_ROT + c) = *reinterpret_cast<const uint4 *>(cached(p) + a.rank + c);
        }
    Product p;
#pragma unroll
    for (int i = 0; i < Product::XI; ++i) p.xp[i] = cached(m0 + p.row(i)) + p.element();
    p.tiled_w(a.w, N, a.rank, n0);
    f32x4 acc[8][4];
    p.run(shared.operands, a.rank, acc);
    const int lane = threadIdx.x % KVA_WAVE, wave = threadIdx.x / KVA_WAVE, r = lane & 15, g = lane >> 4;
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int nt = 0; nt < 8; ++nt) {
            Frag4 f;
            const b16x2 lo = pack_bf16(acc[nt][rt][0], acc[nt][rt][1]), hi = pack_bf16(acc[nt][rt][2], acc[nt][rt][3]);
            f.u2 = make_uint2(__builtin_bit_cast(unsigned, lo), __builtin_bit_cast(unsigned, hi));
            *reinterpret_cast<uint2 *>(&shared.results[((wave & 1) * 64 + 16 * rt + r) * STRIDE + (wave >> 1) * 128 + 16 * nt + 4 * g]) = f.u2;
        }
    __syncthreads();
    const int c = 8 * (threadIdx.x % 32);
    for (int row = threadIdx.x / 32; row < Product::ROWS && m0 + row < keys; row += 8)
        *reinterpret_cast<uint4 *>(a.kv + (((size_t)e * 2 * a.heads + (n0 + c) / LP_DIM) * a.context + m0 + row) * LP_DIM + c % LP_DIM) =
            *reinterpret_cast<const uint4 *>(&shared.results[row * STRIDE + c]);
}

// 8 keys of value element 16 dt + r as the second product's operand (see latent_attention_mfma.hip: lat_values)
typedef __attribute__((address_space(3))) s16x4 lp_lds_s16x4;
template <int STRIDE>
__device__ __forceinline__ Frag8 lp_values(const bf16_t *at, int dt) {
    union { s16x4 t[2]; Frag8 f; } u;
    u.t[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp_lds_s16x4 *)(at + 16 * dt));
    u.t[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp_lds_s16x4 *)(at + 16 * STRIDE + 16 * dt));
    return u.f;
}

// a query's rotated part: pairs of neighbours, or of elements 32 apart (which the same lane holds)
__device__ __forceinline__ void lp_rotate(Frag8 (&f)[2], const float *cos, const float *sin, int g, bool interleaved) {
    float x[2][8], y[2][8];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < 8; ++i) x[s][i] = bf16_bits_to_float(f[s].h[i]);
    if (interleaved) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int i = 0; i < 8; i += 2) {
                const float c = cos[16 * s + 4 * g + i / 2], n = sin[16 * s + 4 * g + i / 2];
                y[s][i] = x[s][i] * c - x[s][i + 1] * n;
                y[s][i + 1] = x[s][i + 1] * c + x[s][i] * n;
            }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float c = cos[8 * g + i], n = sin[8 * g + i];
            y[0][i] = x[0][i] * c - x[1][i] * n;
            y[1][i] = x[1][i] * c + x[0][i] * n;
        }
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < 8; ++i) f[s].h[i] = float_to_bf16_bits(y[s][i]);
}

// A wavefront takes 16 of the tokens and all keys; blocks of 32 keys go to one half of LDS while the other is read.
__global__ void __launch_bounds__(256, 2)
latent_prompt_kernel(LatentPrompt a, int tiles) {
    constexpr int KD = LP_DIM + LP_ROT, KS = KD / 32, NDT = LP_VDIM / 16;
    constexpr int KSTRIDE = KD + 8, VSTRIDE = LP_VDIM + 24;     // (rows of either kind of read on banks of their own)
    __shared__ __align__(16) bf16_t Ks[2][LP_BLOCK * KSTRIDE];
    __shared__ __align__(16) bf16_t Vs[2][LP_BLOCK * VSTRIDE];
    const int e = blockIdx.y, head = blockIdx.x % a.heads, tile = tiles - 1 - (int)(blockIdx.x / a.heads);
    const int q0 = a.entry_q_start[e], n = a.entry_q_start[e + 1] - q0, start = a.entry_start_pos[e];
    if (tile * LP_ROWS >= n) return;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / KVA_WAVE), lane = tid % KVA_WAVE, r = lane & 15, g = lane >> 4;
    const int first = tile * LP_ROWS + 16 * wave;               // the wavefront's first token
    const int mine = min(first + r, n - 1), pos = start + mine;
    const int hi = first < n ? start + min(first + 15, n - 1) : -1;     // newest key of the wavefront's tokens, and of the workgroup's
    const int end = start + min(tile * LP_ROWS + LP_ROWS, n);           // (one past it)
    const bf16_t *kv = a.kv + ((size_t)e * 2 * a.heads + head) * a.context * LP_DIM, *rot = a.rot + (size_t)e * a.context * LP_ROT;
    const size_t to_values = (size_t)a.heads * a.context * LP_DIM;

    Frag8 qf[KS];
    {
        const bf16_t *q = a.q + (size_t)(q0 + mine) * a.q_row + (size_t)head * a.q_head + 8 * g;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qf[ks].u4 = *reinterpret_cast<const uint4 *>(q + 32 * ks);
        Frag8 turned[2] = {qf[KS - 2], qf[KS - 1]};
        lp_rotate(turned, a.cos + (size_t)pos * (LP_ROT / 2), a.sin + (size_t)pos * (LP_ROT / 2), g, a.interleaved != 0);
        qf[KS - 2] = turned[0];
        qf[KS - 1] = turned[1];
    }
    // a block's pieces on their way: rows tid / 16 and 16 further of keys and values, row tid / 8 of the rotated parts
    uint4 k_lo, k_hi, v_lo, v_hi, turned_k;
    auto load = [&](int k0) {
        const bf16_t *lo = kv + (size_t)min(k0 + tid / 16, end - 1) * LP_DIM + 8 * (tid % 16);
        const bf16_t *up = kv + (size_t)min(k0 + tid / 16 + 16, end - 1) * LP_DIM + 8 * (tid % 16);
        k_lo = *reinterpret_cast<const uint4 *>(lo);
        v_lo = *reinterpret_cast<const uint4 *>(lo + to_values);
        k_hi = *reinterpret_cast<const uint4 *>(up);
        v_hi = *reinterpret_cast<const uint4 *>(up + to_values);
        turned_k = *reinterpret_cast<const uint4 *>(rot + (size_t)min(k0 + tid / 8, end - 1) * LP_ROT + 8 * (tid % 8));
    };
    f32x4 o[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;                               // m in the base-2 domain, l this lane's part
    const float scale2 = a.scale * LP_LOG2E;
    load(0);
    for (int k0 = 0, buf = 0; k0 < end; k0 += LP_BLOCK, buf ^= 1) {
        bf16_t *kp = &Ks[buf][tid / 16 * KSTRIDE + 8 * (tid % 16)], *vp = &Vs[buf][tid / 16 * VSTRIDE + 8 * (tid % 16)];
        *reinterpret_cast<uint4 *>(kp) = k_lo;
        *reinterpret_cast<uint4 *>(kp + 16 * KSTRIDE) = k_hi;
        *reinterpret_cast<uint4 *>(vp) = v_lo;
        *reinterpret_cast<uint4 *>(vp + 16 * VSTRIDE) = v_hi;
        *reinterpret_cast<uint4 *>(&Ks[buf][tid / 8 * KSTRIDE + LP_DIM + 8 * (tid % 8)]) = turned_k;
        __syncthreads();            // (a buffer was read last two turns ago: every wavefront has passed the barrier between)
        if (k0 + LP_BLOCK < end) load(k0 + LP_BLOCK);
        if (k0 > hi) continue;                                  // (the wavefront's tokens see none of these)
        f32x4 s[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                Frag8 k;
                k.u4 = *reinterpret_cast<const uint4 *>(&Ks[buf][(16 * t + r) * KSTRIDE + 32 * ks + 8 * g]);
                s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k.v, qf[ks].v, s[t], 0, 0, 0);
            }
        const bool whole = k0 + LP_BLOCK - 1 <= start + first;   // all of the wavefront's tokens see all of the keys
        float sv[8], mx = -INFINITY;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float x = s[t][i] * scale2;
                if (!whole) x = k0 + 16 * t + 4 * g + i <= pos ? x : -INFINITY;
                sv[4 * t + i] = x;
                mx = fmaxf(mx, x);
            }
        const float bm = quad_rows_max(mx);
        // (the reference of the exponentials moves only when a maximum has grown by more than 2^8)
        if (__builtin_amdgcn_ballot_w64(bm > m + 8.f) != 0) {
            const float m_new = fmaxf(m, bm), corr = __builtin_amdgcn_exp2f(m - ((m_new == -INFINITY) ? 0.f : m_new));     // exp2(-inf) = 0
            l *= corr;
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int c = 0; c < 4; ++c) o[dt][c] *= corr;
            m = m_new;
        }
        const float ref = m == -INFINITY ? 0.f : m;
        Frag8 pf;
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
            const float p0 = __builtin_amdgcn_exp2f(sv[j] - ref), p1 = __builtin_amdgcn_exp2f(sv[j + 1] - ref);
            l += p0 + p1;
            pf.p2[j / 2] = pack_bf16(p0, p1);
        }
        const bf16_t *get = &Vs[buf][(4 * g + (r >> 2)) * VSTRIDE + 4 * (r & 3)];
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lp_values<VSTRIDE>(get, dt).v, pf.v, o[dt], 0, 0, 0);
    }
    l = quad_rows_sum(l);
    if (first + r >= n) return;
    float mul = 1.f / l;
    if (a.sinks) {                                              // one more term of the denominator, with no key and no value
        const float sk = a.sinks[head] * LP_LOG2E, m_new = fmaxf(m, sk), corr = __builtin_amdgcn_exp2f(m - m_new);
        mul = corr / (l * corr + __builtin_amdgcn_exp2f(sk - m_new));
    }
    const bf16_t *gate = a.gates ? a.gates + (size_t)(q0 + mine) * a.gate_row : nullptr;
    if (gate && !a.gate_per_element) mul *= 1.f / (1.f + expf(-to_float(gate[head])));
    bf16_t *out = a.out + ((size_t)(q0 + mine) * a.heads + head) * LP_VDIM;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) {
        const int c = 16 * dt + 4 * g;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = o[dt][i] * mul;
            if (gate && a.gate_per_element) v[i] *= 1.f / (1.f + expf(-to_float(gate[(size_t)head * a.gate_head + c + i])));
        }
        const b16x2 lo = pack_bf16(v[0], v[1]), hi2 = pack_bf16(v[2], v[3]);
        *reinterpret_cast<uint2 *>(out + c) = make_uint2(__builtin_bit_cast(unsigned, lo), __builtin_bit_cast(unsigned, hi2));
    }
}

// 64 keys at a time through LDS; a wavefront takes 32 of the tokens (wave % 2) and 32 of the keys (wave / 2), and the two halves of
// the keys are added up at the end.  What bounds it is what the wavefronts read from LDS: 20 KiB of keys and values for 40 products
// of 16 cycles, twice as many as above.  Blocks of keys go through registers, the next ones on their way over the products.
__global__ void __launch_bounds__(256, 2)
latent_prompt_wide_kernel(LatentPrompt a, int tiles) {
    constexpr int KD = LP_DIM + LP_ROT, KS = KD / 32, NDT = LP_VDIM / 16;
    constexpr int KSTRIDE = KD + 8, VSTRIDE = LP_VDIM + 24;     // (rows of either kind of read on banks of their own)
    __shared__ __align__(16) union {
        struct {
            bf16_t k[LP_WIDE_BLOCK * KSTRIDE], v[LP_WIDE_BLOCK * VSTRIDE];
        } b;
        struct {
            float o[2][2][NDT][KVA_WAVE][4], m[2][2][KVA_WAVE], l[2][2][KVA_WAVE];
        } half;                                                 // of the wavefronts with the second half of the keys
    } lds;
    // (the chip takes all of them at once: the longest and the shortest on one compute unit)
    const int e = blockIdx.y, head = blockIdx.x % a.heads, at = blockIdx.x / a.heads, front = (tiles + 1) / 2;
    const int tile = at < front ? tiles - 1 - at : at - front;
    const int q0 = a.entry_q_start[e], n = a.entry_q_start[e + 1] - q0, start = a.entry_start_pos[e];
    if (tile * LP_ROWS >= n) return;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / KVA_WAVE), lane = tid % KVA_WAVE, r = lane & 15, g = lane >> 4;
    const int rows = wave & 1, keys = wave >> 1;
    const int first = tile * LP_ROWS + 32 * rows;               // the wavefront's first token
    int mine[2];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) mine[rt] = min(first + 16 * rt + r, n - 1);
    const int hi = first < n ? start + min(first + 31, n - 1) : -1;     // newest key of the wavefront's tokens, and of the workgroup's
    const int end = start + min(tile * LP_ROWS + LP_ROWS, n);           // (one past it)
    const bf16_t *kv = a.kv + ((size_t)e * 2 * a.heads + head) * a.context * LP_DIM, *rot = a.rot + (size_t)e * a.context * LP_ROT;

    Frag8 qf[2][KS];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
        const bf16_t *q = a.q + (size_t)(q0 + mine[rt]) * a.q_row + (size_t)head * a.q_head + 8 * g;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qf[rt][ks].u4 = *reinterpret_cast<const uint4 *>(q + 32 * ks);
        Frag8 turned[2] = {qf[rt][KS - 2], qf[rt][KS - 1]};
        const size_t table = (size_t)(start + mine[rt]) * (LP_ROT / 2);
        lp_rotate(turned, a.cos + table, a.sin + table, g, a.interleaved != 0);
        qf[rt][KS - 2] = turned[0];
        qf[rt][KS - 1] = turned[1];
    }
    // a block's pieces on their way: rows tid / 16 and 16, 32, 48 further of keys and values, tid / 8 and 32 further of the rotated parts
    kva_u32x4 kx[4], vx[4], tx[2];
    auto load = [&](int k0) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bf16_t *row = kv + (size_t)min(k0 + tid / 16 + 16 * j, end - 1) * LP_DIM + 8 * (tid % 16);
            kx[j] = *reinterpret_cast<const kva_u32x4 *>(row);
            vx[j] = *reinterpret_cast<const kva_u32x4 *>(row + (size_t)a.heads * a.context * LP_DIM);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j)
            tx[j] = *reinterpret_cast<const kva_u32x4 *>(rot + (size_t)min(k0 + tid / 8 + 32 * j, end - 1) * LP_ROT + 8 * (tid % 8));
    };
    f32x4 o[2][NDT];
    float m[2] = {-INFINITY, -INFINITY}, l[2] = {0.f, 0.f};     // m in the base-2 domain, l this lane's part
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) o[rt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const float scale2 = a.scale * LP_LOG2E;
    load(0);
    for (int k0 = 0; k0 < end; k0 += LP_WIDE_BLOCK) {
        __syncthreads();                                        // every wavefront is done with the block before
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            *reinterpret_cast<kva_u32x4 *>(&lds.b.k[(tid / 16 + 16 * j) * KSTRIDE + 8 * (tid % 16)]) = kx[j];
            *reinterpret_cast<kva_u32x4 *>(&lds.b.v[(tid / 16 + 16 * j) * VSTRIDE + 8 * (tid % 16)]) = vx[j];
        }
#pragma unroll
        for (int j = 0; j < 2; ++j)
            *reinterpret_cast<kva_u32x4 *>(&lds.b.k[(tid / 8 + 32 * j) * KSTRIDE + LP_DIM + 8 * (tid % 8)]) = tx[j];
        __syncthreads();
        if (k0 + LP_WIDE_BLOCK < end) load(k0 + LP_WIDE_BLOCK);
        const int kb = k0 + 32 * keys;
        if (kb > hi) continue;                                  // (the wavefront's tokens see none of these)
        const bf16_t *kp = &lds.b.k[(32 * keys + r) * KSTRIDE + 8 * g];
        f32x4 s[2][2];
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int t = 0; t < 2; ++t) s[rt][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                Frag8 k;
                k.u4 = *reinterpret_cast<const uint4 *>(kp + 16 * t * KSTRIDE + 32 * ks);
#pragma unroll
                for (int rt = 0; rt < 2; ++rt) s[rt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k.v, qf[rt][ks].v, s[rt][t], 0, 0, 0);
            }
        Frag8 pf[2];
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            const int pos = start + mine[rt];
            const bool whole = kb + 31 <= start + first + 16 * rt;      // all of the tile's tokens see all of the keys
            float sv[8], mx = -INFINITY;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float x = s[rt][t][i] * scale2;
                    if (!whole) x = kb + 16 * t + 4 * g + i <= pos ? x : -INFINITY;
                    sv[4 * t + i] = x;
                    mx = fmaxf(mx, x);
                }
            const float bm = quad_rows_max(mx);
            // (the reference of the exponentials moves only when a maximum has grown by more than 2^8)
            if (__builtin_amdgcn_ballot_w64(bm > m[rt] + 8.f) != 0) {
                const float m_new = fmaxf(m[rt], bm), corr = __builtin_amdgcn_exp2f(m[rt] - ((m_new == -INFINITY) ? 0.f : m_new));     // exp2(-inf) = 0
                l[rt] *= corr;
#pragma unroll
                for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                    for (int c = 0; c < 4; ++c) o[rt][dt][c] *= corr;
                m[rt] = m_new;
            }
            const float ref = m[rt] == -INFINITY ? 0.f : m[rt];
#pragma unroll
            for (int j = 0; j < 8; j += 2) {
                const float p0 = __builtin_amdgcn_exp2f(sv[j] - ref), p1 = __builtin_amdgcn_exp2f(sv[j + 1] - ref);
                l[rt] += p0 + p1;
                pf[rt].p2[j / 2] = pack_bf16(p0, p1);
            }
        }
        const bf16_t *get = &lds.b.v[(32 * keys + 4 * g + (r >> 2)) * VSTRIDE + 4 * (r & 3)];
        // A portion that starts up to 16 positions behind a multiple of 32 has one block of keys that the wavefront's last 16 tokens see
        // and the first 16 do not.  A probability of zero does not leave out a value that is not a number: they get zeros for it.
        const unsigned seen = kb <= start + first + 15 ? ~0u : 0u;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
            const Frag8 v = lp_values<VSTRIDE>(get, dt);
            Frag8 f = v;
            f.u4 = make_uint4(v.u4.x & seen, v.u4.y & seen, v.u4.z & seen, v.u4.w & seen);
            o[0][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.v, pf[0].v, o[0][dt], 0, 0, 0);
            o[1][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v.v, pf[1].v, o[1][dt], 0, 0, 0);
        }
    }
    __syncthreads();
    if (keys == 1) {
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            lds.half.m[rows][rt][lane] = m[rt];
            lds.half.l[rows][rt][lane] = l[rt];
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) *reinterpret_cast<f32x4 *>(lds.half.o[rows][rt][dt][lane]) = o[rt][dt];
        }
    }
    __syncthreads();
    if (keys == 1) return;
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
        const float other = lds.half.m[rows][rt][lane], both = fmaxf(m[rt], other), ref = both == -INFINITY ? 0.f : both;
        const float c0 = __builtin_amdgcn_exp2f(m[rt] - ref), c1 = __builtin_amdgcn_exp2f(other - ref);
        const float sum = quad_rows_sum(l[rt] * c0 + lds.half.l[rows][rt][lane] * c1);
        if (first + 16 * rt + r >= n) continue;
        float mul = 1.f / sum;
        if (a.sinks) {                                          // one more term of the denominator, with no key and no value
            const float sk = a.sinks[head] * LP_LOG2E, m_new = fmaxf(both, sk), corr = __builtin_amdgcn_exp2f(both - m_new);
            mul = corr / (sum * corr + __builtin_amdgcn_exp2f(sk - m_new));
        }
        const bf16_t *gate = a.gates ? a.gates + (size_t)(q0 + mine[rt]) * a.gate_row : nullptr;
        if (gate && !a.gate_per_element) mul *= 1.f / (1.f + expf(-to_float(gate[head])));
        bf16_t *out = a.out + ((size_t)(q0 + mine[rt]) * a.heads + head) * LP_VDIM;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
            const int c = 16 * dt + 4 * g;
            const f32x4 more = *reinterpret_cast<const f32x4 *>(lds.half.o[rows][rt][dt][lane]);
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[i] = (o[rt][dt][i] * c0 + more[i] * c1) * mul;
                if (gate && a.gate_per_element) v[i] *= 1.f / (1.f + expf(-to_float(gate[(size_t)head * a.gate_head + c + i])));
            }
            const b16x2 lo = pack_bf16(v[0], v[1]), hi2 = pack_bf16(v[2], v[3]);
            *reinterpret_cast<uint2 *>(out + c) = make_uint2(__builtin_bit_cast(unsigned, lo), __builtin_bit_cast(unsigned, hi2));
        }
    }
}

extern "C" int kva_latent_prompt_supported(int dim, int rot, int vdim, int rank) {
    return dim == LP_DIM && rot == LP_ROT && vdim == LP_VDIM && rank > 0 && rank % LDSP_K == 0;
}

// Whether a wavefront takes 32 tokens and half of the keys (or 16 and all of them).  That reads LDS half as often and ends with sums over the
// halves and two more barriers a block, which long contexts repay, as long as the chip takes all workgroups at once; past that, one more
// turn of them, four fewer wavefronts a compute unit weigh more.  16 tokens / 32, us with the expansion, rank 512:
//   one entry of 16 heads from position 0:  64 tokens 16.4/19.2  256 22.1/24.7  512 30.2/32.4  1,000 44.2/44.2  1,400 56.1/55.1  2,048 (512
//   workgroups) 75.5/68.8  4,096 (1,024) 157/169;  of 8 heads 2,048 70.4/68.4  4,096 (512) 127/112;  of 32 heads 1,000 50.3/50.2  1,400 (704)
//   69.2/69.2  2,048 (1,024) 98.9/109;  of 64 heads 1,000 (1,024) 73.9/79.6  2,048 202/209
//   behind 1,024 positions, 16 heads:  64 44.6/45.4  256 49.8/49.7  512 56.2/55.5  1,400 87.8/83.3  four of 512 90.0/89.3  four of 700 (704) 122/125
static bool latent_prompt_wide(long long workgroups, int longest, int context) { return workgroups <= 512 && context > 1024 && longest >= 256; }

// kv bf16 [entries, 2 heads, context, 128] and rot bf16 [entries * context, rot] are workspace; `context` is no
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
    KVA_REQUIRE(entries > 0 && entries <= 65535 && longest > 0 && longest <= context, "latent_prompt: %d entries of up to %d tokens in contexts of %d",
                entries, longest, context);
    KVA_REQUIRE(q_row % 8 == 0 && q_head % 8 == 0 && ((uintptr_t)q | (uintptr_t)cache | (uintptr_t)w | (uintptr_t)kv | (uintptr_t)rot) % 16 == 0 &&
                    (uintptr_t)out % 8 == 0, "latent_prompt: rows must start at multiples of 16 bytes");
    const LatentPrompt a{(bf16_t *)out, (const bf16_t *)q, (const bf16_t *)cache, (const bf16_t *)w, (bf16_t *)kv, (bf16_t *)rot, block_table,
                         entry_seat, entry_q_start, entry_start_pos, cos, sin, sinks, (const bf16_t *)gates, q_row, q_head, gate_row,
                         gate_head, gate_per_element, max_blocks, page_size, heads, rank, context, interleaved, scale};
    const long long expand = (long long)((context + 127) / 128) * heads, tiles = (longest + LP_ROWS - 1) / LP_ROWS;
    KVA_REQUIRE(expand <= 0x7fffffff && tiles * heads <= 0x7fffffff, "latent_prompt: too many workgroups");
    hipLaunchKernelGGL(latent_expand_kernel, dim3((unsigned)expand, entries), dim3(256), 0, stream, a);
    if (latent_prompt_wide(tiles * heads * entries, longest, context))
        hipLaunchKernelGGL(latent_prompt_wide_kernel, dim3((unsigned)(tiles * heads), entries), dim3(256), 0, stream, a, (int)tiles);
    else
        hipLaunchKernelGGL(latent_prompt_kernel, dim3((unsigned)(tiles * heads), entries), dim3(256), 0, stream, a, (int)tiles);
    KVA_CHECK_LAUNCH("latent_prompt");
    return KVA_OK;
}
