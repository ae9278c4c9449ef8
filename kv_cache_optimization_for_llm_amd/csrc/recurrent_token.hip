// One token of every request through a recurrent mixer, from the joined projection's columns to what the output
// projection reads, in one launch: the convolution (or the decays' low-rank product), the recurrence, the norm of the
// read-outs and the gate.  recurrent.hip and state_space.hip take the same way in three launches of 4 to 10 us, of which the work is
// a third: a decoded token's launches are as long as the trips to memory that follow each other in them, and one after
// the other.  Here everything a workgroup needs - its part of S first, 16 bytes a lane - is asked for at once.
//
// A workgroup takes what shares inputs: the heads of a key head (delta rule), a head (linear attention), the heads of
// a group (state-space): it alone reads and writes their part of the state, the convolution's last inputs among it.  Every sum is
// formed as the other kernels form it, in the same order: a token's numbers do not depend on which of them ran.
//
// us a call in a graph, three launches -> this, 1 / 8 / 64 / 256 requests of one token (bf16 rows):
//   delta rule, 8 heads of 128 x 128 over 4 key heads:      15.0 / 20.8 / 74.7 / 255 -> 12.2 / 14.1 / 18.2 / 66
//   linear attention, 16 heads of 64 x 128, decays of 16:   11.7 / 17.7 / 56.7 / 188 -> 5.7 / 7.2 / 18.7 / 61
//   state-space, 32 heads of 128 x 64 in 4 groups:          14.9 / 18.6 / 38.2 / 167 -> 11.0 / 13.6 / 28.5 / 135
// Few requests are bound by one unit's instructions and its 60 GB/s for S (128 and 256 KB a workgroup in the first and last line),
// many by S itself.
#include "recurrent.h"

#define TOKEN_THREADS 1024
#define TOKEN_MAX_DIM 128

// Loads of the projection's rows (T: bf16_t or float).  The type is known when the code is compiled: a load behind a branch is
// waited for in that branch, and a token's way is as long as its trips to memory.
template <typename T>
__device__ inline float token_ld(const void *p, size_t i) { return to_float(reinterpret_cast<const T *>(p)[i]); }
template <typename T>
__device__ inline void token_ld8(const void *p, size_t i, float (&f)[8]) { hng_ld8(p, sizeof(T) == 2 ? KVA_BF16 : KVA_F32, i, f); }

struct TokenIO {
    const void *y;                      // the projection's rows; the gate's and the result's are of the same type
    int y_stride;
    float *state;                       // seat rows; S at state_off, the convolution's inputs [channels, taps - 1] at conv_off
    size_t seat_stride;
    int state_off, conv_off, conv_col;  // (conv_col: the first channel's column)
    const float *conv_w, *conv_bias;    // [channels, taps]
    const int *entry_q_start, *entry_seat;
    void *out;
    int out_stride, out_off;
    const float *norm_w;                // absent: heads are not normed
    int norm_stride;
    float norm_eps, mul;
    HeadGate gate;
};

// A channel's convolution with silu for the token in row `row`: what it reads, and then its result; the state takes the
// token's input.
template <typename T, int TAPS>
struct TokenConv {
    float in[TAPS], w[TAPS], bias;
    __device__ inline void load(const TokenIO &io, const float *st, size_t row, int c) {
#pragma unroll
        for (int j = 0; j < TAPS - 1; ++j) in[j] = st[(size_t)c * (TAPS - 1) + j];
        in[TAPS - 1] = token_ld<T>(io.y, row * io.y_stride + io.conv_col + c);
#pragma unroll
        for (int j = 0; j < TAPS; ++j) w[j] = io.conv_w[(size_t)c * TAPS + j];
        bias = io.conv_bias ? io.conv_bias[c] : 0.f;
    }
    __device__ inline float finish(float *st, int c) const {
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < TAPS; ++j) acc = rec_fma(w[j], in[j], acc);
#pragma unroll
        for (int j = 0; j < TAPS - 1; ++j) st[(size_t)c * (TAPS - 1) + j] = in[j + 1];
        return rec_act(acc + bias, 1);
    }
};

template <int PERM>
__device__ inline float token_quad(float v) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(v), PERM, 0xf, 0xf, false));
}

// What comes from memory comes back in the order in which it was asked for: the little that the first steps need in front of S.
__device__ inline void token_keep_order() { __builtin_amdgcn_sched_barrier(0); }

// The sum over 2^lanes neighbouring lanes, added as by shuffles with the lane 2^(lanes - 1), .., 2, 1 further (a + b is b + a, and a
// rotation inside a row of 16 lanes meets the same lanes once the larger distances are added).
__device__ inline float token_lanes_sum(float v, int lanes) {
    if (lanes < 4) {
        for (int x = 1 << lanes >> 1; x > 0; x >>= 1) v += __shfl_xor(v, x, KVA_WAVE);
        return v;
    }
    if (lanes == 6) {
        const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = __uint_as_float(h[0]) + __uint_as_float(h[1]);
    }
    if (lanes >= 5) {
        const auto h = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = __uint_as_float(h[0]) + __uint_as_float(h[1]);
    }
    return row16_sum(v);
}

// Norm and gate of the read-outs o[units * width] (LDS), a unit by 2^lanes lanes with 8 elements each; the units are number
// unit0 .. of the row's.  What a thread needs of the gate and the weight is loaded before the recurrence.
template <typename T>
struct TokenNorm {
    float gt[8], wv[8];
    int unit, j;
    bool live;
    __device__ inline void load(const TokenIO &io, size_t row, int unit0, int units, int width, int lanes) {
        unit = threadIdx.x >> lanes;
        j = 8 * (threadIdx.x & ((1 << lanes) - 1));
        live = unit < units && j < width;
        const int at = (unit0 + min(unit, units - 1)) * width + min(j, width - 8);
#pragma unroll
        for (int i = 0; i < 8; ++i) gt[i] = wv[i] = 1.f;
        if (io.gate.p) token_ld8<T>(io.gate.p, row * io.gate.stride + io.gate.off + at, gt);
        if (io.norm_w) hng_ld8(io.norm_w, KVA_F32, (size_t)(unit0 + min(unit, units - 1)) * io.norm_stride + min(j, width - 8), wv);
    }
    __device__ inline void activate(const TokenIO &io) {           // (before the read-outs are there)
        if (!live || !io.gate.p) return;
#pragma unroll
        for (int i = 0; i < 8; ++i) gt[i] = io.gate.act == 1 ? rec_sigmoid(gt[i]) : rec_silu(gt[i]);
    }
    __device__ inline void finish(const TokenIO &io, const float *o, size_t row, int unit0, int units, int width, int lanes) {
        if (((threadIdx.x & ~(KVA_WAVE - 1)) >> lanes) >= units) return;        // (whole wavefronts: the sums go over lanes)
        float v[8], sq = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            v[i] = live ? o[unit * width + j + i] : 0.f;
            if (io.gate.first) v[i] *= gt[i];
            if (live) sq = rec_fma(v[i], v[i], sq);
        }
        float inv = 1.f;
        if (io.norm_w) {
            sq = token_lanes_sum(sq, lanes);
            inv = 1.0f / sqrtf(sq / (float)width + io.norm_eps);
        }
        if (!live) return;
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = v[i] * inv * wv[i] * (io.gate.first ? 1.f : gt[i]) * io.mul;
        const size_t at = row * io.out_stride + io.out_off + (size_t)(unit0 + unit) * width + j;
        if constexpr (sizeof(T) == 2) {
            uint32_t p[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                p[i] = (uint32_t)float_to_bf16_bits(v[2 * i]) | ((uint32_t)float_to_bf16_bits(v[2 * i + 1]) << 16);
            *reinterpret_cast<uint4 *>(reinterpret_cast<uint16_t *>(io.out) + at) = make_uint4(p[0], p[1], p[2], p[3]);
        } else {
            float4 *dst = reinterpret_cast<float4 *>(reinterpret_cast<float *>(io.out) + at);
            dst[0] = make_float4(v[0], v[1], v[2], v[3]);
            dst[1] = make_float4(v[4], v[5], v[6], v[7]);
        }
    }
};

// A thread holds 4 neighbouring value columns (of one head) and RP of the state's rows, 4 (16 (j / 4) + r) + j % 4 for lane r of 16.
template <int RP>
__device__ inline void token_load_state(const float *Sg, int dim, int vdim, int r, float4 (&S)[RP]) {
#pragma unroll
    for (int j = 0; j < RP; ++j) {
        const int i = 4 * (16 * (j / 4) + r) + j % 4;
        S[j] = *reinterpret_cast<const float4 *>(Sg + (size_t)min(i, dim - 1) * vdim);
    }
#pragma unroll
    for (int j = 0; j < RP; ++j) {
        const int i = 4 * (16 * (j / 4) + r) + j % 4;
        if (i >= dim) S[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
}
template <int RP>
__device__ inline void token_store_state(float *Sg, int dim, int vdim, int r, const float4 (&S)[RP]) {
#pragma unroll
    for (int j = 0; j < RP; ++j) {
        const int i = 4 * (16 * (j / 4) + r) + j % 4;
        if (i < dim) *reinterpret_cast<float4 *>(Sg + (size_t)i * vdim) = S[j];
    }
}

// ---- gated delta rule: grid (key heads, entries), 16 threads to 4 value columns of the key head's heads ---------------
struct DeltaToken {
    TokenIO io;
    int beta_off, decay_off;
    const float *a_log, *dt_bias, *channel_decay;
    int decay_stride;
    float unit_eps;
    int heads, kv_heads, dim, vdim, lanes;      // 2^lanes lanes a norm
};

// CD: a decay per key channel, handed in; the rows of S are then decayed one by one.
template <typename T, int RP, int TAPS, bool CD>
__global__ void __launch_bounds__(TOKEN_THREADS)
delta_token_kernel(DeltaToken a) {
    constexpr int DP = 16 * RP;
    __shared__ __attribute__((aligned(16))) float q[DP], k[DP], v[TOKEN_THREADS / 4], o[TOKEN_THREADS / 4];
    __shared__ float beta_s[TOKEN_THREADS / 4], keep_s[TOKEN_THREADS / 4], unit_s[2];
    const TokenIO &io = a.io;
    const int kvh = blockIdx.x, e = blockIdx.y, group = a.heads / a.kv_heads, d = a.dim, dv = a.vdim, cols = group * dv;
    const int q0 = io.entry_q_start[e];
    if (io.entry_q_start[e + 1] <= q0) return;
    const int tid = threadIdx.x, r = tid % 16, col = tid / 16 * 4;
    const bool on = col < cols;
    const int head = kvh * group + (on ? col / dv : 0), cc = on ? col % dv : 0;
    float *row_state = io.state + (size_t)io.entry_seat[e] * io.seat_stride;
    float *Sg = row_state + io.state_off + (size_t)head * d * dv + cc;
    // the convolution's channels: q and k of the key head, v of its heads
    float *st = row_state + io.conv_off;
    auto channel = [&](int c) {
        return c < 2 * DP ? (c % DP < d ? (c < DP ? 0 : a.kv_heads * d) + kvh * d + c % DP : -1) : 2 * a.kv_heads * d + kvh * cols + c - 2 * DP;
    };
    auto put = [&](int c, float x) { (c < DP ? q : c < 2 * DP ? k - DP : v - 2 * DP)[c] = x; };
    const int channels = 2 * DP + cols, mine = tid < channels ? channel(tid) : -1;
    TokenConv<T, TAPS> conv;
    if (mine >= 0) conv.load(io, st, q0, mine);
    float beta_in = 0.f, keep_in = 0.f, rate_log = 0.f;
    const bool counts = tid < group;
    if (counts) {
        const int h = kvh * group + tid;
        beta_in = token_ld<T>(io.y, (size_t)q0 * io.y_stride + a.beta_off + h);
        if constexpr (!CD) {
            keep_in = token_ld<T>(io.y, (size_t)q0 * io.y_stride + a.decay_off + h) + a.dt_bias[h];
            rate_log = a.a_log[h];
        }
    }
    TokenNorm<T> norm;
    norm.load(io, q0, kvh * group, group, dv, a.lanes);
    token_keep_order();
    if (tid < channels) put(tid, mine >= 0 ? conv.finish(st, mine) : 0.f);
    for (int c = tid + blockDim.x; c < channels; c += blockDim.x) {
        const int x = channel(c);
        if (x >= 0) conv.load(io, st, q0, x);
        put(c, x >= 0 ? conv.finish(st, x) : 0.f);
    }
    float4 S[RP], decays[RP / 4];
    token_load_state<RP>(Sg, d, dv, r, S);
    if constexpr (CD)
#pragma unroll
        for (int j = 0; j < RP / 4; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int x = 4 * (16 * j + r) + i;
                (&decays[j].x)[i] = x < d ? a.channel_decay[(size_t)q0 * a.decay_stride + head * d + x] : 0.f;
            }
    token_keep_order();
    norm.activate(io);
    if (counts) {
        beta_s[tid] = rec_sigmoid(beta_in);
        keep_s[tid] = CD ? 1.f : expf(-expf(rate_log) * rec_softplus(keep_in));
    }
    __syncthreads();
    if (tid < 4) {                      // what makes q and k unit vectors: four lanes, every fourth element each
        float sq = 0.f, sk = 0.f;
#pragma unroll
        for (int i = 0; i < DP; i += 4) {
            sq = rec_fma(q[i + tid], q[i + tid], sq);
            sk = rec_fma(k[i + tid], k[i + tid], sk);
        }
        sq += token_quad<0xB1>(sq); sq += token_quad<0x4E>(sq);         // lane ^ 1, lane ^ 2
        sk += token_quad<0xB1>(sk); sk += token_quad<0x4E>(sk);
        if (tid == 0) {
            unit_s[0] = 1.0f / sqrtf((float)d) / sqrtf(sq + a.unit_eps);
            unit_s[1] = 1.0f / sqrtf(sk + a.unit_eps);
        }
    }
    __syncthreads();
    const float mq = unit_s[0], mk = unit_s[1], g = keep_s[on ? col / dv : 0], beta = beta_s[on ? col / dv : 0];
    float u[4];
    float4 kk[RP / 4];
#pragma unroll
    for (int j = 0; j < RP / 4; ++j) {
        kk[j] = *reinterpret_cast<const float4 *>(k + 4 * (16 * j + r));
        kk[j].x *= mk; kk[j].y *= mk; kk[j].z *= mk; kk[j].w *= mk;
        if constexpr (CD)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float al = (&decays[j].x)[i];
                S[4 * j + i] = make_float4(al * S[4 * j + i].x, al * S[4 * j + i].y, al * S[4 * j + i].z, al * S[4 * j + i].w);
            }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        float p[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < RP; ++j) p[j % 4] = rec_fma((&S[j].x)[c], (&kk[j / 4].x)[j % 4], p[j % 4]);
        p[0] += p[1]; p[2] += p[3];
        u[c] = p[0] + p[2];
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const float s = row16_sum(u[c]);
        u[c] = beta * rec_fma(-g, s, v[on ? col + c : 0]);
    }
#pragma unroll
    for (int j = 0; j < RP; ++j)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float &s = (&S[j].x)[c];
            const float kj = (&kk[j / 4].x)[j % 4];
            s = rec_fma(kj, u[c], CD ? s : g * s);
        }
#pragma unroll
    for (int j = 0; j < RP / 4; ++j) kk[j] = *reinterpret_cast<const float4 *>(q + 4 * (16 * j + r));
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        float p[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < RP; ++j) p[j % 4] = rec_fma((&S[j].x)[c], (&kk[j / 4].x)[j % 4], p[j % 4]);
        p[0] += p[1]; p[2] += p[3];
        const float s = row16_sum(p[0] + p[2]);
        if (r == 0 && on) o[col + c] = s * mq;
    }
    __syncthreads();
    norm.finish(io, o, q0, kvh * group, group, dv, a.lanes);
    if (on) token_store_state<RP>(Sg, d, dv, r, S);
}

// ---- gated linear attention: grid (heads, entries) -----------------------------------------------------------------
// The decays alpha = sigmoid(a2 (a1 columns of y) + bias)^(1 / tau), a channel by a thread.
struct LinearToken {
    TokenIO io;
    int q_off, k_off, v_off, a_off, rank;
    const void *a2;                     // of the rows' type
    const float *a2_bias;
    float inv_tau, q_mul;
    int heads, dim, vdim, lanes;
};

template <typename T, int RP>
__global__ void __launch_bounds__(TOKEN_THREADS)
linear_token_kernel(LinearToken a) {
    constexpr int DP = 16 * RP;
    __shared__ __attribute__((aligned(16))) float q[DP], k[DP], al[DP], v[TOKEN_THREADS / 4], o[TOKEN_THREADS / 4];
    const TokenIO &io = a.io;
    const int head = blockIdx.x, e = blockIdx.y, d = a.dim, dv = a.vdim;
    const int q0 = io.entry_q_start[e];
    if (io.entry_q_start[e + 1] <= q0) return;
    const int tid = threadIdx.x, r = tid % 16, col = tid / 16 * 4;
    const bool on = col < dv;
    float *Sg = io.state + (size_t)io.entry_seat[e] * io.seat_stride + io.state_off + (size_t)head * d * dv + (on ? col : 0);
    const size_t yrow = (size_t)q0 * io.y_stride;
    // what number c of the chunk of LDS is made of: q, k, the decays, v
    auto make = [&](int c) {
        const int i = c % DP;
        if (c >= 3 * DP) { v[c - 3 * DP] = token_ld<T>(io.y, yrow + a.v_off + head * dv + c - 3 * DP); return; }
        float acc = 0.f;
        if (i < d && c < 2 * DP) {
            acc = token_ld<T>(io.y, yrow + (c < DP ? a.q_off : a.k_off) + head * d + i);
            if (c < DP) acc *= a.q_mul;
        } else if (i < d) {
            const size_t n = (size_t)head * d + i;
            for (int x = 0; x < a.rank; x += 8) {
                float f[8], z[8];
                token_ld8<T>(a.a2, n * a.rank + x, f);
#pragma unroll
                for (int y = 0; y < 8; ++y) z[y] = token_ld<T>(io.y, yrow + a.a_off + x + y);
#pragma unroll
                for (int y = 0; y < 8; ++y) acc = rec_fma(z[y], f[y], acc);
            }
            const float z = acc + a.a2_bias[n];
            acc = expf(-(fmaxf(-z, 0.f) + log1pf(expf(-fabsf(z)))) * a.inv_tau);
        }
        (c < DP ? q : c < 2 * DP ? k - DP : al - 2 * DP)[c] = acc;
    };
    TokenNorm<T> norm;
    norm.load(io, q0, head, 1, dv, a.lanes);
    if (tid < 3 * DP + dv) make(tid);
    token_keep_order();
    float4 S[RP];
    token_load_state<RP>(Sg, d, dv, r, S);
    token_keep_order();
    for (int c = tid + blockDim.x; c < 3 * DP + dv; c += blockDim.x) make(c);
    norm.activate(io);
    __syncthreads();
    float p[4][4] = {};
#pragma unroll
    for (int j = 0; j < RP / 4; ++j) {
        const float4 kk = *reinterpret_cast<const float4 *>(k + 4 * (16 * j + r)), qq = *reinterpret_cast<const float4 *>(q + 4 * (16 * j + r)),
                     aa = *reinterpret_cast<const float4 *>(al + 4 * (16 * j + r));
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                float &s = (&S[4 * j + i].x)[c];
                s = rec_fma((&kk.x)[i], v[on ? col + c : 0], (&aa.x)[i] * s);
                p[c][i] = rec_fma(s, (&qq.x)[i], p[c][i]);
            }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const float s = row16_sum((p[c][0] + p[c][1]) + (p[c][2] + p[c][3]));
        if (r == 0 && on) o[col + c] = s;
    }
    __syncthreads();
    norm.finish(io, o, q0, head, 1, dv, a.lanes);
    if (on) token_store_state<RP>(Sg, d, dv, r, S);
}

// ---- state-space: grid (groups, entries); 256 threads to 64 value columns of a head, PASSES times ------------------------------
struct SpaceToken {
    TokenIO io;
    int dt_off;
    const float *a_log, *dt_bias, *d_skip;
    int heads, groups, n, vdim, width, lanes;   // width: elements that are normed together
};
#define SPACE_COLS 512                          // value columns of a group's heads

template <typename T, int PASSES, int TAPS>
__global__ void __launch_bounds__(TOKEN_THREADS)
space_token_kernel(SpaceToken a) {
    __shared__ __attribute__((aligned(16))) float x[SPACE_COLS], o[SPACE_COLS], b[TOKEN_MAX_DIM], c[TOKEN_MAX_DIM];
    __shared__ float4 red[TOKEN_THREADS / KVA_WAVE * PASSES][16];
    __shared__ float dt_s[SPACE_COLS], keep_s[SPACE_COLS];
    const TokenIO &io = a.io;
    const int grp = blockIdx.x, e = blockIdx.y, hg = a.heads / a.groups, n = a.n, dv = a.vdim, cols = hg * dv;
    const int q0 = io.entry_q_start[e];
    if (io.entry_q_start[e + 1] <= q0) return;
    const int tid = threadIdx.x, cg = tid % 16, rg = tid / 16 % 16, lane = tid % KVA_WAVE, wave = tid / KVA_WAVE;
    const int slices = (dv + 63) / 64, units = hg * slices;
    float *row_state = io.state + (size_t)io.entry_seat[e] * io.seat_stride;
    const int parts = cols / a.width, channels = cols + 2 * n;
    // the convolution's channels: x of the group's heads, B and C; its outputs are kept in the projection's type
    float *st = row_state + io.conv_off;
    auto channel = [&](int i) { return i < cols ? grp * cols + i : a.heads * dv + (i < cols + n ? grp * n : (a.groups + grp) * n - n) + i - cols; };
    auto put = [&](int i, float f) {
        if (sizeof(T) == 2) f = bf16_bits_to_float(float_to_bf16_bits(f));
        (i < cols ? x : i < cols + n ? b - cols : c - cols - n)[i] = f;
    };
    TokenConv<T, TAPS> conv;
    if (tid < channels) conv.load(io, st, q0, channel(tid));
    float dt_in = 0.f, rate_log = 0.f;
    if (tid < hg) {
        dt_in = token_ld<T>(io.y, (size_t)q0 * io.y_stride + a.dt_off + grp * hg + tid) + a.dt_bias[grp * hg + tid];
        rate_log = a.a_log[grp * hg + tid];
    }
    TokenNorm<T> norm;
    norm.load(io, q0, grp * parts, parts, a.width, a.lanes);
    token_keep_order();
    float4 S[PASSES][8];
    float *Sg[PASSES];
    int head[PASSES], col[PASSES];              // in the group; in the head
    bool on[PASSES];
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
        const int unit = tid / 256 + p * (TOKEN_THREADS / 256);
        head[p] = min(unit, units - 1) / slices;
        col[p] = min(unit, units - 1) % slices * 64 + 4 * cg;
        on[p] = unit < units && col[p] < dv;
        Sg[p] = row_state + io.state_off + (size_t)(grp * hg + head[p]) * n * dv + (on[p] ? col[p] : 0);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int r = rg + 16 * k;
            S[p][k] = *reinterpret_cast<const float4 *>(Sg[p] + (size_t)min(r, n - 1) * dv);
        }
    }
    token_keep_order();
    if (tid < channels) put(tid, conv.finish(st, channel(tid)));
    for (int i = tid + blockDim.x; i < channels; i += blockDim.x) {
        conv.load(io, st, q0, channel(i));
        put(i, conv.finish(st, channel(i)));
    }
    norm.activate(io);
    if (tid < hg) {
        const float dt = rec_softplus(dt_in);
        dt_s[tid] = dt;
        keep_s[tid] = expf(-expf(rate_log) * dt);
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
        const float dt = dt_s[head[p]], keep = keep_s[head[p]];
        float xv[4], s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) xv[i] = on[p] ? x[head[p] * dv + col[p] + i] : 0.f;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int r = rg + 16 * k;
            const float br = r < n ? b[r < n ? r : 0] : 0.f, cr = r < n ? c[r < n ? r : 0] : 0.f, w = br * dt;
            float4 &t = S[p][k];
            if (!on[p] || r >= n) t = make_float4(0.f, 0.f, 0.f, 0.f);
            t.x = rec_fma(w, xv[0], keep * t.x);
            t.y = rec_fma(w, xv[1], keep * t.y);
            t.z = rec_fma(w, xv[2], keep * t.z);
            t.w = rec_fma(w, xv[3], keep * t.w);
            s[0] = rec_fma(t.x, cr, s[0]);
            s[1] = rec_fma(t.y, cr, s[1]);
            s[2] = rec_fma(t.z, cr, s[2]);
            s[3] = rec_fma(t.w, cr, s[3]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i] = quad_rows_sum(s[i]);
        if (lane < 16) red[wave + p * (TOKEN_THREADS / KVA_WAVE)][cg] = make_float4(s[0], s[1], s[2], s[3]);
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
        if (tid % 256 >= 16 || !on[p]) continue;
        const int w0 = wave + p * (TOKEN_THREADS / KVA_WAVE);
        float4 t = red[w0][cg];
#pragma unroll
        for (int w = 1; w < 4; ++w) {
            t.x += red[w0 + w][cg].x; t.y += red[w0 + w][cg].y; t.z += red[w0 + w][cg].z; t.w += red[w0 + w][cg].w;
        }
        const float skip = a.d_skip[grp * hg + head[p]];
        const int at = head[p] * dv + col[p];
        o[at] = rec_fma(skip, x[at], t.x);
        o[at + 1] = rec_fma(skip, x[at + 1], t.y);
        o[at + 2] = rec_fma(skip, x[at + 2], t.z);
        o[at + 3] = rec_fma(skip, x[at + 3], t.w);
    }
    __syncthreads();
    norm.finish(io, o, q0, grp * parts, parts, a.width, a.lanes);
#pragma unroll
    for (int p = 0; p < PASSES; ++p)
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (on[p] && rg + 16 * k < n) *reinterpret_cast<float4 *>(Sg[p] + (size_t)(rg + 16 * k) * dv) = S[p][k];
}

// ---- host ------------------------------------------------------------------------------------------------------------------
static int token_lanes(int width) {             // its logarithm
    int lanes = 0;
    while (1 << lanes < width / 8) ++lanes;
    return lanes;
}

static bool token_types(int y, int gate, int out) { return (y == KVA_BF16 || y == KVA_F32) && gate == y && out == y; }

// what the wide loads and stores of norm, gate and state ask of sizes and addresses
static bool token_aligned(const TokenIO &io, int width, int vdim) {
    return width % 8 == 0 && width <= 512 && vdim % 4 == 0 && io.out_stride % 8 == 0 && io.out_off % 8 == 0 && io.norm_stride % 8 == 0 &&
           (!io.gate.p || (io.gate.stride % 8 == 0 && io.gate.off % 8 == 0)) && io.seat_stride % 4 == 0 && io.state_off % 4 == 0 &&
           (((uintptr_t)io.out | (uintptr_t)io.gate.p | (uintptr_t)io.norm_w | (uintptr_t)io.state) & 15) == 0;
}

static int token_check(const char *what, const TokenIO &io, int entries) {
    KVA_REQUIRE(io.y && io.state && io.out && io.entry_q_start && io.entry_seat, "%s: missing operand", what);
    KVA_REQUIRE(io.gate.act == 0 || io.gate.act == 1, "%s: activation %d is neither silu (0) nor sigmoid (1)", what, io.gate.act);
    KVA_REQUIRE(entries >= 0 && entries <= 65535, "%s: %d entries", what, entries);
    return KVA_OK;
}

// Entries of one token each, or none.  `ask`: whether sizes and addresses fit is all that is asked (0 / 1, nothing is launched).
extern "C" int kva_delta_token(int ask, const void *y, int y_dtype, int y_stride, int conv_col, const float *conv_w, int taps, float *state,
                               long long seat_stride, int state_off, int conv_off, int beta_off, int decay_off, const float *a_log,
                               const float *dt_bias, const float *channel_decay, int decay_stride, float unit_eps, const float *norm_w,
                               float norm_eps, const void *gate, int gate_dtype, int gate_stride, int gate_off, int act, void *out,
                               int out_dtype, int out_stride, int out_off, float mul, const int *entry_q_start, const int *entry_seat,
                               int entries, int heads, int kv_heads, int dim, int vdim, hipStream_t stream) {
    const DeltaToken a{{y, y_stride, state, (size_t)seat_stride, state_off, conv_off, conv_col, conv_w, nullptr, entry_q_start, entry_seat,
                        out, out_stride, out_off, norm_w, 0, norm_eps, mul, {gate, gate_dtype, gate_stride, gate_off, act, 0}},
                       beta_off, decay_off, a_log, dt_bias, channel_decay, decay_stride, unit_eps, heads, kv_heads, dim, vdim, token_lanes(vdim)};
    const bool fits = heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && dim > 0 && dim <= TOKEN_MAX_DIM && taps >= 2 && taps <= 4 &&
                      heads / kv_heads * vdim * 4 <= TOKEN_THREADS && token_types(y_dtype, gate_dtype, out_dtype) && token_aligned(a.io, vdim, vdim);
    if (ask) return fits;
    if (int rc = token_check("delta_token", a.io, entries)) return rc;
    KVA_REQUIRE(fits && conv_w && ((a_log && dt_bias) || (channel_decay && decay_stride >= heads * dim)), "delta_token: sizes, addresses or operands do not fit");
    if (entries == 0) return KVA_OK;
    const int threads = max(256, (heads / kv_heads * vdim * 4 + 63) / 64 * 64);
    const dim3 grid(kv_heads, entries);
#define KVA_DELTA_TOKEN_OF(T, TAPS)                                                                                                \
    hipLaunchKernelGGL((dim <= 64 ? (channel_decay ? delta_token_kernel<T, 4, TAPS, true> : delta_token_kernel<T, 4, TAPS, false>)     \
                                  : (channel_decay ? delta_token_kernel<T, 8, TAPS, true> : delta_token_kernel<T, 8, TAPS, false>)),   \
                       grid, dim3(threads), 0, stream, a)
#define KVA_DELTA_TOKEN(TAPS)                                  \
    do {                                                       \
        if (y_dtype == KVA_BF16) KVA_DELTA_TOKEN_OF(bf16_t, TAPS); \
        else KVA_DELTA_TOKEN_OF(float, TAPS);                  \
    } while (0)
    if (taps == 2) KVA_DELTA_TOKEN(2);
    else if (taps == 3) KVA_DELTA_TOKEN(3);
    else KVA_DELTA_TOKEN(4);
#undef KVA_DELTA_TOKEN
#undef KVA_DELTA_TOKEN_OF
    KVA_CHECK_LAUNCH("delta_token");
    return KVA_OK;
}

extern "C" int kva_linear_token(int ask, const void *y, int y_dtype, int y_stride, int q_off, int k_off, int v_off, int a_off, int rank,
                                const void *a2, int a2_dtype, const float *a2_bias, float inv_tau, float q_mul, float *state,
                                long long seat_stride, int state_off, const float *norm_w, float norm_eps, const void *gate,
                                int gate_dtype, int gate_stride, int gate_off, int act, void *out, int out_dtype, int out_stride,
                                int out_off, float mul, const int *entry_q_start, const int *entry_seat, int entries, int heads,
                                int dim, int vdim, hipStream_t stream) {
    const LinearToken a{{y, y_stride, state, (size_t)seat_stride, state_off, 0, 0, nullptr, nullptr, entry_q_start, entry_seat, out,
                         out_stride, out_off, norm_w, 0, norm_eps, mul, {gate, gate_dtype, gate_stride, gate_off, act, 0}},
                        q_off, k_off, v_off, a_off, rank, a2, a2_bias, inv_tau, q_mul, heads, dim, vdim, token_lanes(vdim)};
    // (a longer low-rank product is worth its own launch, whose sums also go over a wavefront from 128 on)
    const bool fits = heads > 0 && dim > 0 && dim <= TOKEN_MAX_DIM && vdim > 0 && vdim * 4 <= TOKEN_THREADS && rank > 0 && rank % 8 == 0 && rank <= 64 &&
                      (uintptr_t)a2 % 32 == 0 && token_types(y_dtype, gate_dtype, out_dtype) && a2_dtype == y_dtype && token_aligned(a.io, vdim, vdim);
    if (ask) return fits;
    if (int rc = token_check("linear_token", a.io, entries)) return rc;
    KVA_REQUIRE(fits && a2 && a2_bias && inv_tau > 0.f, "linear_token: sizes, addresses or operands do not fit");
    if (entries == 0) return KVA_OK;
    const int threads = max(256, (vdim * 4 + 63) / 64 * 64);
    const dim3 grid(heads, entries);
    const auto kernel = y_dtype == KVA_BF16 ? (dim <= 64 ? linear_token_kernel<bf16_t, 4> : linear_token_kernel<bf16_t, 8>)
                                            : (dim <= 64 ? linear_token_kernel<float, 4> : linear_token_kernel<float, 8>);
    hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, stream, a);
    KVA_CHECK_LAUNCH("linear_token");
    return KVA_OK;
}

extern "C" int kva_space_token(int ask, const void *y, int y_dtype, int y_stride, int conv_col, const float *conv_w, const float *conv_bias,
                               int taps, float *state, long long seat_stride, int state_off, int conv_off, int dt_off, const float *a_log,
                               const float *dt_bias, const float *d_skip, const float *norm_w, float norm_eps, int gate_off, void *out,
                               int out_dtype, int out_stride, int out_off, float mul, const int *entry_q_start, const int *entry_seat,
                               int entries, int heads, int groups, int n, int vdim, int norm_groups, hipStream_t stream) {
    const int hg = groups > 0 ? heads / groups : 0, width = norm_groups > 0 ? heads * vdim / norm_groups : 0;
    const SpaceToken a{{y, y_stride, state, (size_t)seat_stride, state_off, conv_off, conv_col, conv_w, conv_bias, entry_q_start, entry_seat,
                        out, out_stride, out_off, norm_w, width, norm_eps, mul, {y, y_dtype, y_stride, gate_off, 0, 1}},
                       dt_off, a_log, dt_bias, d_skip, heads, groups, n, vdim, width, token_lanes(width)};
    const int units = hg * ((vdim + 63) / 64), per = TOKEN_THREADS / 256;
    const bool fits = heads > 0 && groups > 0 && norm_groups > 0 && heads % groups == 0 && (long long)heads * vdim % norm_groups == 0 && width > 0 &&
                      hg * vdim <= SPACE_COLS && hg * vdim % width == 0 && hg * vdim / width << token_lanes(width) <= TOKEN_THREADS &&
                      n > 0 && n <= TOKEN_MAX_DIM && taps >= 2 && taps <= 4 && units <= 2 * per && token_types(y_dtype, y_dtype, out_dtype) && token_aligned(a.io, width, vdim) &&
                      // (fp32 rows, a group's columns in two passes, more workgroups than the chip takes at once: three launches / one, us, 1,024 requests
                      // of 24 heads of 64 x 64 in 3 groups 188 / 223, 16 heads in 2 groups 125 / 141; 256 requests of 32 heads of 128 x 64 in 4 groups
                      // 103 / 108, of 24 in 3 50 / 51; 64 requests of the two 34 / 28 and 19 / 14)
                      (y_dtype != KVA_F32 || units <= per || (long long)groups * entries <= 768);
    if (ask) return fits;
    if (int rc = token_check("space_token", a.io, entries)) return rc;
    KVA_REQUIRE(fits && conv_w && a_log && dt_bias && d_skip, "space_token: sizes, addresses or operands do not fit");
    if (entries == 0) return KVA_OK;
    const dim3 grid(groups, entries);
    // (all 1,024 where 256 have work: 64 heads of 16 x 64 in groups of their own, 1 / 64 / 256 requests 6.8 / 70 / 280 us; 6.2 / 23 / 73 so, and
    // 11.7 / 32 / 94 in three launches)
    const int threads = 256 * min(units, per);
#define KVA_SPACE_TOKEN(TAPS)                                                                                                       \
    hipLaunchKernelGGL((y_dtype == KVA_BF16 ? (units <= per ? space_token_kernel<bf16_t, 1, TAPS> : space_token_kernel<bf16_t, 2, TAPS>)  \
                                            : (units <= per ? space_token_kernel<float, 1, TAPS> : space_token_kernel<float, 2, TAPS>)),  \
                       grid, dim3(threads), 0, stream, a)
    if (taps == 2) KVA_SPACE_TOKEN(2);
    else if (taps == 3) KVA_SPACE_TOKEN(3);
    else KVA_SPACE_TOKEN(4);
#undef KVA_SPACE_TOKEN
    KVA_CHECK_LAUNCH("space_token");
    return KVA_OK;
}
