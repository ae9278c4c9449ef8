// The gated delta rule and gated linear attention over prompts, 64 tokens at a time on the matrix cores.
//
// recurrent.hip walks a request's tokens one after the other, about 0.3 us a token whatever the chip could do beside
// it.  Written out over a chunk of tokens 1..C that starts from the state S, with D_ij the product of the decays
// (per key channel) of the tokens j + 1..i:
//
//   u_i = beta_i (v_i - S^T (D_i0 k_i) - sum_{j<i} (k_i . D_ij k_j) u_j)        (linear attention: u_i = v_i)
//   o_i = S^T (D_i0 q_i) + sum_{j<=i} (q_i . D_ij k_j) u_j
//   S  <- D_C0 S + sum_j (D_Cj k_j) u_j^T
//
// The u_i are the solution of a unit lower triangular system with right-hand sides beta v and beta D_0 k, so
//   U = Uv - W S,    O = Qd S + P U,    S <- diag(G) S + Kd^T U
// with Uv, W, Qd, P, Kd, G of a chunk known without S.  Three kernels: `prepare` makes those, all chunks side by side;
// `states` hands S on from chunk to chunk, a head's value columns 4, 8 or 16 to a workgroup, and leaves the S each chunk
// starts from and its U; `outputs` makes O, all chunks side by side again.
//
// Inputs, outputs and the state between steps are 32-bit as in the walk.  What the walk does not have is the sums over
// neighbouring tokens (A = beta k . D k and P = q . D k, their products with the u_i, U = Uv - W S): where keys share a
// direction the u_i alternate, and those sums are differences of numbers several times their size.  They are formed in
// 64 bits (v_mfma_f64_16x16x4_f64) from 32-bit operands, U and Uv are kept in 64, W, Qd, Kd, P and the S that chunks
// start from are rounded to 32; only linear attention, whose U is V, hands S on with 32-bit products.  Relative error
// against 64 bits, the walk -> all in 32 bits -> this: 3.9e-7 -> 8.8e-7 -> 0.8e-7 with keys that share half of their
// square, 2.2e-7 -> 7e-7 -> 1.1e-7 with nine tenths and decays from 0.9 up.  Decays only ever enter as products of decays
// between two tokens (at most 1, no logarithms, no quotients): a decay of zero or of anything else is as exact as in the walk.
// Where anything of an entry's inputs to a head is infinite or not a number, `prepare` says so and that (entry, head) is left
// to the walk behind these kernels: zeros above a diagonal would carry it to tokens in front of it.
// Order of sums: chunks are counted from the step's first token of the request, so here - unlike in the walk - the
// last bits of a token's result depend on how the request was cut into steps, and, with the delta rule, now and then on how many
// entries and heads the step has (how many value columns a workgroup takes orders the sums of 64-bit products).  The 32-bit
// path therefore walks.
//
// us a call, the walk -> these three kernels (in 32 bits alone), one prompt of 2,048 / 8,192 tokens:
//   delta rule, 8 heads of 128 x 128 over 4 key heads:  715 / 2,831 -> 119 / 447 (in 32 bits and 16 columns a workgroup 101 / 373)
//   linear attention, 16 heads of 64 x 128:             584 / 2,317 -> 89 / 377 (73 / 334)
// A 64-bit product takes two to three times the cycles of a 32-bit one.  `states` is a chain: 64 of them a wavefront and
// chunk and two trips through LDS (102 us of 154 with 16 columns a workgroup; with 4 on the smaller instruction 63: the same
// number of instructions, each a third as long); with operands row by row instead of in operand order and a head's workgroups
// spread over the dies it took twice as long.  `prepare` and `outputs` are short of workgroups (256) more than of anything else.
#include "recurrent.h"
#include <float.h>

#define CK REC_CHUNK_TOKENS         // tokens a chunk
#define CK_PAD 4                    // a row in LDS is that much longer: rows start in different banks

typedef float ck_f32x4 __attribute__((ext_vector_type(4)));
typedef double ck_f64x4 __attribute__((ext_vector_type(4)));

struct ChunkArgs {
    float *out;                     // [T, heads * vdim]
    float *state;                   // seat rows; S [heads, dim, vdim] at state_off
    size_t seat_stride;
    int state_off;
    const int *entry_q_start, *entry_seat;
    int heads, kv_heads, vdim;
    int entries, shortest, chunks;  // entries of fewer tokens than `shortest` are left to the walk, the others have so many chunks
    float *work;                    // per (chunk, head) a block of ck_block() floats
    int *odd;                       // per (chunk, head): whether an input is infinite or not a number
};

// A (chunk, head)'s block: W [CK][D], Qd [CK][D], Kd^T [D][CK], P [CK][CK], U^T [vdim][CK] (64-bit, linear attention uses half
// of it), S^T [vdim][D], each in operand order, and G [D].
__host__ __device__ inline size_t ck_block(int dim, int vdim) {
    return (size_t)3 * CK * dim + CK * CK + (size_t)vdim * (2 * CK + dim) + dim;
}

// Operand order: 16 rows x 16 columns at a time as the 64 lanes hold them, four columns a lane - so that a wavefront
// loads and stores 1 KiB of neighbouring bytes (row by row it is 64 bytes of each of 16 rows).  Lane (row r, group g)
// holds, as element c, column 4 g + c or column g + 4 c.  Which of the two does not matter to a product as long as both
// operands agree; a result has, in lane (r, g), the rows 4 g + c (32 bits) or g + 4 c (64 bits) of column r, the operand
// order of its transpose.  Tokens stand in the second order everywhere, key channels in that of the type S is summed in.
__device__ inline size_t ck_frag(int rowtile, int coltile, int coltiles, int lane) {
    return ((size_t)(rowtile * coltiles + coltile) * KVA_WAVE + lane) * 4;
}

template <int D>
struct ChunkBlock {
    float *w, *q, *kt, *p, *ut, *st, *g;
    __device__ inline ChunkBlock(const ChunkArgs &a, int number, int head) {
        w = a.work + ((size_t)number * a.heads + head) * ck_block(D, a.vdim);
        q = w + CK * D;
        kt = q + CK * D;
        p = kt + CK * D;
        ut = p + CK * CK;
        st = ut + (size_t)a.vdim * 2 * CK;
        g = st + (size_t)a.vdim * D;
    }
};

// Chunk `number`: the `chunk`th of entry `entry`, whose first one has the number `first`.  Asked by whole wavefronts;
// 64 entries a turn.
struct ChunkPlace {
    int entry, chunk, first;
};
__device__ inline ChunkPlace ck_find(const ChunkArgs &a, int number) {
    const int lane = threadIdx.x % KVA_WAVE;
    if (a.entries == 1) return {number < rec_chunks_of(a.entry_q_start, 0, a.shortest) ? 0 : -1, number, 0};
    for (int e0 = 0, before = 0; e0 < a.entries; e0 += KVA_WAVE) {
        const int mine = e0 + lane < a.entries ? rec_chunks_of(a.entry_q_start, e0 + lane, a.shortest) : 0;
        int upto = mine;
#pragma unroll
        for (int o = 1; o < KVA_WAVE; o <<= 1) {
            const int other = __shfl_up(upto, o, KVA_WAVE);
            if (lane >= o) upto += other;
        }
        const unsigned long long past = __ballot(number < before + upto);
        if (past) {
            const int owner = __builtin_amdgcn_readfirstlane(__ffsll(past) - 1);
            const int first = __builtin_amdgcn_readfirstlane(before + __shfl(upto - mine, owner, KVA_WAVE));
            return {e0 + owner, number - first, first};
        }
        before += __shfl(upto, KVA_WAVE - 1, KVA_WAVE);
    }
    return {-1, 0, 0};              // (more chunks asked for than the entries have)
}

template <bool DELTA> __device__ inline int ck_channel(int g, int c) { return DELTA ? g + 4 * c : 4 * g + c; }
__device__ inline int ck_token(int g, int c) { return g + 4 * c; }

__device__ inline ck_f32x4 ck_ld(const float *p) { return *reinterpret_cast<const ck_f32x4 *>(p); }
__device__ inline void ck_st(float *p, ck_f32x4 v) { *reinterpret_cast<ck_f32x4 *>(p) = v; }
__device__ inline ck_f32x4 ck_mul(ck_f32x4 a, ck_f32x4 b) {
    return ck_f32x4{a[0] * b[0], a[1] * b[1], a[2] * b[2], a[3] * b[3]};
}
__device__ inline ck_f64x4 ck_ld(const double *p) { return *reinterpret_cast<const ck_f64x4 *>(p); }
__device__ inline void ck_st(double *p, ck_f64x4 v) { *reinterpret_cast<ck_f64x4 *>(p) = v; }
__device__ inline ck_f64x4 ck_mul(ck_f64x4 a, ck_f64x4 b) { return a * b; }
__device__ inline ck_f64x4 ck_wide(ck_f32x4 a) { return __builtin_convertvector(a, ck_f64x4); }
__device__ inline ck_f64x4 ck_wide(ck_f64x4 a) { return a; }
__device__ inline ck_f32x4 ck_narrow(ck_f64x4 a) { return __builtin_convertvector(a, ck_f32x4); }
__device__ inline ck_f32x4 ck_narrow(ck_f32x4 a) { return a; }
// a 32-bit operand as the type of the sum it goes into
__device__ inline ck_f32x4 ck_as(ck_f32x4 a, ck_f32x4) { return a; }
__device__ inline ck_f64x4 ck_as(ck_f32x4 a, ck_f64x4) { return ck_wide(a); }
// 16 terms of the sums
__device__ inline ck_f32x4 ck_mfma(ck_f32x4 a, ck_f32x4 b, ck_f32x4 c) {
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c, 0, 0, 0);
    return c;
}
__device__ inline ck_f64x4 ck_mfma(ck_f64x4 a, ck_f64x4 b, ck_f64x4 c) {
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f64_16x16x4f64(a[e], b[e], c, 0, 0, 0);
    return c;
}
// sum over the four lanes of a row, all of them get it (quad_rows_sum in 64 bits)
__device__ inline double ck_row_sum(double v) {
    auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(v), false, false);
    auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(v), false, false);
    v = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
    lo = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v), false, false);
    hi = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v), false, false);
    return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}

// Where q, k, v and the decays come from.
struct ChunkInput {
    const float *qkv;               // delta rule: q, k, v after the convolution [T, qkv_stride]
    const void *y;                  // the projection [T, y_stride]: beta and decay columns; linear attention: q, k, v
    int qkv_stride, y_dtype, y_stride, q_off, k_off, v_off, beta_off, decay_off, act;
    const float *a_log, *dt_bias;   // one decay a head and token, from a column of y; or
    const float *channel_decay;     // one per head, token and key channel [T, decay_stride]; or
    const float *head_decay;        // one a head
    int decay_stride;
    float unit_eps;
    double q_mul;
};

__device__ inline bool ck_odd(float x) { return !(fabsf(x) <= FLT_MAX); }

// Where the four elements of a lane's share of 16 tokens lie next to each other: tokens g, g + 4, g + 8, g + 12 at 4 g.
__device__ inline int ck_place(int x) { return 4 * (x % 4) + x / 4; }

// One workgroup a (chunk, head), four wavefronts, wavefront b its tokens 16 b .. 16 b + 15.  CD: a decay per key channel.
// Without, decays are numbers that multiply products of q and k formed without them; with, a lane takes its share of
// D_ij k_j from token to token inside a block of 16 and blocks meet through their products of decays.
template <int D, bool DELTA, bool CD>
__global__ void __launch_bounds__(256)
chunk_prepare_kernel(ChunkArgs a, ChunkInput in) {
    constexpr int DS = D + CK_PAD, STEPS = D / 16;
    __shared__ __attribute__((aligned(32))) union {
        float q[CK][DS];                                            // q (CD: then D_i(block start) q)
        double t[DELTA ? CK : 1][CK + CK_PAD];                      // then (1 + A)^-1, columns in the order of ck_place
    } QT;
    __shared__ __attribute__((aligned(32))) float Kx[CK][DS];       // k (CD: then D_i(block start) k)
    __shared__ __attribute__((aligned(32))) float Al[CD ? CK : 1][DS];      // decays, then D_(block end)j k
    __shared__ __attribute__((aligned(32))) double Bt[CD ? 4 : 1][D];       // a block's product of decays
    __shared__ __attribute__((aligned(32))) double A[DELTA ? CK * CK : 4];  // beta k . D k, operand order
    __shared__ __attribute__((aligned(32))) double Ti[DELTA ? 4 : 1][16][16 + CK_PAD];  // (1 + A)^-1's diagonal blocks, as t
    __shared__ double gs[CK], nq[CK], nk[CK];
    __shared__ double Dd[CD ? 1 : 4][16][17];                       // decays between two tokens of a block
    __shared__ double from0[CK], to_end[CK], whole[4];              // D_i0; D_Cj; a block's own product
    __shared__ float beta[CK];
    auto &Q = QT.q;
    auto &T = QT.t;
    const int head = blockIdx.y;
    const ChunkPlace place = ck_find(a, blockIdx.x);
    const int e = place.entry, chunk = place.chunk;
    if (e < 0) return;
    const int q0 = a.entry_q_start[e], n = a.entry_q_start[e + 1] - q0;
    const int m = min(CK, n - chunk * CK), row0 = q0 + chunk * CK, kvh = head / (a.heads / a.kv_heads);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / KVA_WAVE), lane = tid % KVA_WAVE;
    const int r = lane % 16, g = lane / 16, b0 = wave * 16;
    ChunkBlock<D> out(a, blockIdx.x, head);
    bool odd = false;               // an input of this thread's is not a number, or infinite

    // ---- the chunk's tokens; rows behind the last one are zero (decay 1): they change nothing
    if (DELTA) {
        constexpr int PER = CK * D / 4 / 256;
        ck_f32x4 lq[PER], lk[PER];
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int x = tid + 256 * j, t = x / (D / 4), i = x % (D / 4) * 4;
            const float *row = in.qkv + (size_t)(row0 + min(t, m - 1)) * in.qkv_stride + kvh * D + i;
            lq[j] = ck_ld(row + in.q_off);
            lk[j] = ck_ld(row + in.k_off);
        }
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int x = tid + 256 * j, t = x / (D / 4), i = x % (D / 4) * 4;
#pragma unroll
            for (int c = 0; c < 4; ++c) odd |= ck_odd(lq[j][c]) || ck_odd(lk[j][c]);
            ck_st(&Q[t][i], t < m ? lq[j] : ck_f32x4{0.f, 0.f, 0.f, 0.f});
            ck_st(&Kx[t][i], t < m ? lk[j] : ck_f32x4{0.f, 0.f, 0.f, 0.f});
        }
    } else {
        constexpr int PER = CK * D / 256, AT = 16;
        for (int j0 = 0; j0 < PER; j0 += AT) {
            float lq[AT], lk[AT];
#pragma unroll
            for (int j = 0; j < AT; ++j) {
                const int x = tid + 256 * (j0 + j), t = x / D, i = x % D;
                const size_t row = (size_t)(row0 + min(t, m - 1)) * in.y_stride + head * D + i;
                lq[j] = rec_ld(in.y, in.y_dtype, row + in.q_off);
                lk[j] = rec_ld(in.y, in.y_dtype, row + in.k_off);
            }
#pragma unroll
            for (int j = 0; j < AT; ++j) {
                const int x = tid + 256 * (j0 + j), t = x / D, i = x % D;
                odd |= ck_odd(lq[j]) || ck_odd(lk[j]);
                Q[t][i] = t < m ? rec_act(lq[j], in.act) * (float)in.q_mul : 0.f;
                Kx[t][i] = t < m ? rec_act(lk[j], in.act) : 0.f;
            }
        }
    }
    if (CD) {
        constexpr int PER = CK * D / 256, AT = 16;
        for (int j0 = 0; j0 < PER; j0 += AT) {
            float la[AT];
#pragma unroll
            for (int j = 0; j < AT; ++j) {
                const int x = tid + 256 * (j0 + j), t = x / D, i = x % D;
                la[j] = in.channel_decay[(size_t)(row0 + min(t, m - 1)) * in.decay_stride + head * D + i];
            }
#pragma unroll
            for (int j = 0; j < AT; ++j) {
                const int x = tid + 256 * (j0 + j), t = x / D, i = x % D;
                odd |= ck_odd(la[j]);
                Al[CD ? t : 0][i] = t < m ? la[j] : 1.f;
            }
        }
    }
    if (tid < CK) {
        float b = 0.f, d = 1.f;
        if (tid < m) {
            const size_t yrow = (size_t)(row0 + tid) * in.y_stride;
            if (DELTA) b = rec_sigmoid(rec_ld(in.y, in.y_dtype, yrow + in.beta_off + head));
            if (in.head_decay) d = in.head_decay[head];
            else if (!CD)
                d = expf(-expf(in.a_log[head]) * rec_softplus(rec_ld(in.y, in.y_dtype, yrow + in.decay_off + head) + in.dt_bias[head]));
        }
        odd |= ck_odd(b) || ck_odd(d);
        beta[tid] = b;
        gs[tid] = d;
        nq[tid] = nk[tid] = 1.0;
    }
    __syncthreads();
    if (DELTA) {                    // what makes q and k unit vectors (q also times dim^-1/2): four lanes a token
        const int t = tid / 4, part = tid % 4;
        ck_f64x4 sq = {0.0, 0.0, 0.0, 0.0}, sk = sq;
#pragma unroll
        for (int i = 4 * part; i < D; i += 16) {
            const ck_f64x4 q = ck_wide(ck_ld(&Q[t][i])), k = ck_wide(ck_ld(&Kx[t][i]));
            sq += q * q;
            sk += k * k;
        }
        double uq = (sq[0] + sq[1]) + (sq[2] + sq[3]), uk = (sk[0] + sk[1]) + (sk[2] + sk[3]);
        uq += __shfl_xor(uq, 1, KVA_WAVE); uq += __shfl_xor(uq, 2, KVA_WAVE);
        uk += __shfl_xor(uk, 1, KVA_WAVE); uk += __shfl_xor(uk, 2, KVA_WAVE);
        uq = in.q_mul / sqrt(uq + in.unit_eps);
        uk = 1.0 / sqrt(uk + in.unit_eps);
        if (CD) {
#pragma unroll
            for (int i = 4 * part; i < D; i += 16) {
                ck_st(&Q[t][i], ck_narrow(ck_wide(ck_ld(&Q[t][i])) * uq));
                ck_st(&Kx[t][i], ck_narrow(ck_wide(ck_ld(&Kx[t][i])) * uk));
            }
        } else if (part == 0) {
            nq[t] = uq;
            nk[t] = uk;
        }
    }
    if (!CD && wave == 0) {         // lane (block g, j = r): the decays from token j on, then those before it
        double d = 0.0, pre = 1.0;
        for (int i = 0; i < 16; ++i) {
            const double x = gs[16 * g + i];
            d = r < i ? d * x : r == i ? 1.0 : 0.0;
            pre = i <= r ? pre * x : pre;
            Dd[CD ? 0 : g][i][r] = d;
        }
        const double b1 = __shfl(pre, 15, KVA_WAVE), b2 = __shfl(pre, 31, KVA_WAVE), b3 = __shfl(pre, 47, KVA_WAVE), b4 = __shfl(pre, 63, KVA_WAVE);
        const double lead = g == 0 ? 1.0 : g == 1 ? b1 : g == 2 ? b1 * b2 : b1 * b2 * b3;
        const double rest = g == 3 ? 1.0 : g == 2 ? b4 : g == 1 ? b3 * b4 : b2 * b3 * b4;
        from0[lane] = pre * lead;   // (token 16 g + r is `lane`)
        to_end[lane] = d * rest;
        if (r == 15) whole[g] = pre;
    }
    __syncthreads();

    // ---- P and A
    if (CD) {
        // inside a block: lane (j = r, g) takes its share of D_ij k_j from token to token; the sums over the channels that
        // token i needs with every j are formed side by side
        ck_f64x4 kd[STEPS], pre[STEPS];
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            kd[s] = ck_f64x4{0.0, 0.0, 0.0, 0.0};
            pre[s] = ck_f64x4{1.0, 1.0, 1.0, 1.0};
        }
        for (int i = 0; i < 16; ++i) {
            ck_f64x4 sp = {0.0, 0.0, 0.0, 0.0}, sa = sp;
#pragma unroll
            for (int s = 0; s < STEPS; ++s) {
                const ck_f64x4 al = ck_wide(ck_ld(&Al[CD ? b0 + i : 0][16 * s + 4 * g])), q = ck_wide(ck_ld(&Q[b0 + i][16 * s + 4 * g])),
                               k = ck_wide(ck_ld(&Kx[b0 + i][16 * s + 4 * g]));
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    pre[s][c] = i <= r ? pre[s][c] * al[c] : pre[s][c];
                    kd[s][c] = r < i ? kd[s][c] * al[c] : r == i ? k[c] : 0.0;
                }
                sp += q * kd[s];
                if (DELTA) sa += k * kd[s];
            }
            const double p = ck_row_sum((sp[0] + sp[1]) + (sp[2] + sp[3]));         // zero for r > i
            const size_t at = ck_frag(wave, wave, 4, i + 16 * (r % 4)) + r / 4;
            if (g == 0) out.p[at] = (float)p;
            if (DELTA) {
                const double x = ck_row_sum((sa[0] + sa[1]) + (sa[2] + sa[3]));
                if (g == 0) A[DELTA ? at : 0] = r < i ? beta[b0 + i] * x : 0.0;
            }
        }
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {           // (so far a wavefront has read only its own 16 rows)
            float *q = &Q[b0 + r][16 * s + 4 * g], *k = &Kx[b0 + r][16 * s + 4 * g];
            ck_st(q, ck_narrow(ck_wide(ck_ld(q)) * pre[s]));
            ck_st(k, ck_narrow(ck_wide(ck_ld(k)) * pre[s]));
            ck_st(&Al[CD ? b0 + r : 0][16 * s + 4 * g], ck_narrow(kd[s]));
            if (r == 15) ck_st(&Bt[CD ? wave : 0][16 * s + 4 * g], pre[s]);
        }
        __syncthreads();
    }
    // tiles (I, J): with CD the six with I > J, without it the diagonal ones too; P's first, then A's.  The result is
    // formed transposed, [j][i]: lane (i = r, j = g, g + 4 ..), operand order.
    constexpr int PAIRS = CD ? 6 : 10;
    for (int task = wave; task < (DELTA ? 2 : 1) * PAIRS; task += 4) {
        const int pair = task % PAIRS;
        const bool keys = task >= PAIRS;
        const int I = pair < 6 ? (pair == 0 ? 1 : pair <= 2 ? 2 : 3) : pair - 6, J = pair < 6 ? (pair == 0 ? 0 : pair <= 2 ? pair - 1 : pair - 3) : pair - 6;
        ck_f64x4 acc[2] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            const ck_f64x4 x = ck_wide(ck_ld(keys ? &Kx[16 * I + r][16 * s + 4 * g] : &Q[16 * I + r][16 * s + 4 * g]));
            ck_f64x4 k = ck_wide(ck_ld(CD ? &Al[CD ? 16 * J + r : 0][16 * s + 4 * g] : &Kx[16 * J + r][16 * s + 4 * g]));
            if (CD)
                for (int b = J + 1; b < I; ++b) k *= ck_ld(&Bt[CD ? b : 0][16 * s + 4 * g]);
            acc[s % 2] = ck_mfma(k, x, acc[s % 2]);
        }
        const int i = 16 * I + r;
        double mid = 1.0;                           // the product of the blocks between
        if (!CD)
            for (int b = J + 1; b < I; ++b) mid *= whole[b];
        ck_f64x4 v;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int jj = ck_token(g, c);
            v[c] = acc[0][c] + acc[1][c];
            if (!CD) {
                // D_ij: to the end of j's block, the blocks between, from the start of i's
                const double d = I == J ? Dd[CD ? 0 : I][r][jj] : Dd[CD ? 0 : J][15][jj] * mid * (Dd[CD ? 0 : I][r][0] * gs[16 * I]);
                v[c] *= d * nk[16 * J + jj] * (keys ? nk[i] : nq[i]);
            }
            if (keys) v[c] = I == J && jj >= r ? 0.0 : v[c] * beta[i];
        }
        if (keys) { if (DELTA) ck_st(&A[DELTA ? ck_frag(I, J, 4, lane) : 0], v); }
        else ck_st(out.p + ck_frag(I, J, 4, lane), ck_narrow(v));
    }
    __syncthreads();

    // ---- Qd, Kd^T, G
    for (int x = wave; x < 4 * STEPS; x += 4) {
        const int I = x / STEPS, s = x % STEPS;
        ck_f32x4 q;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int i = 16 * s + ck_channel<DELTA>(g, c);
            double mul = CD ? 1.0 : nq[16 * I + r] * from0[16 * I + r];
            if (CD) for (int b = 0; b < I; ++b) mul *= Bt[CD ? b : 0][i];
            q[c] = (float)(Q[16 * I + r][i] * mul);
        }
        ck_st(out.q + ck_frag(I, s, STEPS, lane), q);
    }
    for (int x = wave; x < 4 * STEPS; x += 4) {
        const int J = x % 4, c0 = x / 4 * 16;
        ck_f32x4 k;
        double rest = 1.0;
        if (CD) for (int b = J + 1; b < 4; ++b) rest *= Bt[CD ? b : 0][c0 + r];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int j = 16 * J + ck_token(g, c);
            k[c] = (float)(CD ? Al[CD ? j : 0][c0 + r] * rest : Kx[j][c0 + r] * (nk[j] * to_end[j]));
        }
        ck_st(out.kt + ck_frag(x / 4, J, 4, lane), k);
    }
    if (tid < D)            // (in the order in which a lane of `states` holds the channels)
        out.g[DELTA ? tid / 16 * 16 + ck_place(tid % 16) : tid] =
            (float)(CD ? Bt[0][tid] * Bt[CD ? 1 : 0][tid] * Bt[CD ? 2 : 0][tid] * Bt[CD ? 3 : 0][tid] : from0[CK - 1]);

    const size_t vrow = DELTA ? (size_t)in.qkv_stride : (size_t)in.y_stride;
    auto values = [&](int col, ck_f32x4(&v)[4]) {           // a lane's tokens of a value column
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int t = 16 * s + ck_token(g, c);
                const size_t at = (size_t)(row0 + min(t, m - 1)) * vrow + in.v_off + head * a.vdim + col;
                v[s][c] = DELTA ? in.qkv[at] : rec_ld(in.y, in.y_dtype, at);
            }
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                odd |= ck_odd(v[s][c]);
                if (!DELTA) v[s][c] = rec_act(v[s][c], in.act);
                if (16 * s + ck_token(g, c) >= m) v[s][c] = 0.f;
            }
    };
    auto note_odd = [&] {
        const int any = __syncthreads_or(odd ? 1 : 0);
        if (tid == 0) a.odd[(size_t)blockIdx.x * a.heads + head] = any;
    };
    if (!DELTA) {                   // U is V
        for (int tile = wave; tile < a.vdim / 16; tile += 4) {
            ck_f32x4 v[4];
            values(16 * tile + r, v);
#pragma unroll
            for (int s = 0; s < 4; ++s) ck_st(out.ut + ck_frag(tile, s, 4, lane), v[s]);
        }
        note_odd();
        return;
    }

    // ---- T = (1 + A)^-1: its diagonal blocks, column r by forward substitution ...
    if (g == 0) {
        double x[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            double s = i == r ? 1.0 : 0.0;
#pragma unroll
            for (int j = 0; j < i; ++j) s -= A[DELTA ? ck_frag(wave, wave, 4, i + 16 * (j % 4)) + j / 4 : 0] * x[j];
            x[i] = s;
            Ti[DELTA ? wave : 0][i][ck_place(r)] = s;
        }
    }
    __syncthreads();
    // ... then T_IJ = -T_II sum_{J<=K<I} A_IK T_KJ, wavefront J its block column, results being the next products' operands
    {
        const int J = wave;
        ck_f64x4 col[4];            // T_IJ for I = J .. 3: lane (column r, rows g, g + 4 ..)
#pragma unroll
        for (int I = 0; I < 4; ++I) {
            ck_f64x4 t = {0.0, 0.0, 0.0, 0.0};
            if (I == J) {
#pragma unroll
                for (int c = 0; c < 4; ++c) t[c] = Ti[DELTA ? J : 0][ck_token(g, c)][ck_place(r)];
            } else if (I > J) {
                ck_f64x4 sum = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int K = 0; K < I; ++K)
                    if (K >= J) sum = ck_mfma(ck_ld(&A[DELTA ? ck_frag(I, K, 4, lane) : 0]), col[K], sum);
                t = -ck_mfma(ck_ld(&Ti[DELTA ? I : 0][r][4 * g]), sum, t);
            }
            col[I] = t;
#pragma unroll
            for (int c = 0; c < 4; ++c) T[DELTA ? 16 * I + ck_token(g, c) : 0][16 * J + ck_place(r)] = t[c];
        }
    }
    __syncthreads();
    // ---- W = T (beta D_0 k), transposed: lane (i = r, channels g, g + 4 ..); Uv = T (beta v): lane (column r, tokens g, g + 4 ..)
    ck_f64x4 bj[4], wj[4];          // what token j's row is multiplied by
#pragma unroll
    for (int J = 0; J < 4; ++J)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int j = 16 * J + ck_token(g, c);
            bj[J][c] = beta[j];
            wj[J][c] = CD ? beta[j] : beta[j] * nk[j] * from0[j];
        }
    for (int tile = wave; tile < STEPS; tile += 4) {
        ck_f64x4 k[4];
        double lead = 1.0;
#pragma unroll
        for (int J = 0; J < 4; ++J) {
#pragma unroll
            for (int c = 0; c < 4; ++c) k[J][c] = Kx[16 * J + ck_token(g, c)][16 * tile + r] * lead * wj[J][c];
            if (CD) lead *= Bt[CD ? J : 0][16 * tile + r];
        }
#pragma unroll
        for (int I = 0; I < 4; ++I) {
            ck_f64x4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int J = 0; J <= I; ++J) acc = ck_mfma(k[J], ck_ld(&T[DELTA ? 16 * I + r : 0][16 * J + 4 * g]), acc);
            ck_st(out.w + ck_frag(I, tile, STEPS, lane), ck_narrow(acc));
        }
    }
    double *uv = reinterpret_cast<double *>(out.ut);
    for (int tile = wave; tile < a.vdim / 16; tile += 4) {
        ck_f32x4 x[4];
        values(16 * tile + r, x);
        ck_f64x4 v[4];
#pragma unroll
        for (int J = 0; J < 4; ++J) v[J] = ck_wide(x[J]) * bj[J];
#pragma unroll
        for (int I = 0; I < 4; ++I) {
            ck_f64x4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int J = 0; J <= I; ++J) acc = ck_mfma(ck_ld(&T[DELTA ? 16 * I + r : 0][16 * J + 4 * g]), v[J], acc);
            ck_st(uv + ck_frag(tile, I, 4, lane), acc);
        }
    }
    note_odd();
}

// One workgroup a (request, head, 16 value columns), chunk after chunk.  A wavefront keeps D / 64 tiles of 16 rows of
// S's columns in registers, all of S^T [16][D] stands in LDS for U = Uv - W S, of which a wavefront makes 16
// tokens; U^T goes through LDS to S <- G S + Kd^T U.  The next chunk's operands are on their way over a chunk.  A
// head's workgroups are `heads` apart in the launch: on one die where the heads are a multiple of eight, so that W
// and Kd come from memory once.
template <bool DELTA> struct CkSum { typedef float type; typedef ck_f32x4 type4; };
template <> struct CkSum<true> { typedef double type; typedef ck_f64x4 type4; };

template <int D, bool DELTA>
__global__ void __launch_bounds__(256)
chunk_states_kernel(ChunkArgs a) {
    constexpr int STEPS = D / 16, MT = D / 64;
    using R = typename CkSum<DELTA>::type;
    using R4 = typename CkSum<DELTA>::type4;
    __shared__ __attribute__((aligned(32))) R St[16 * D];           // operand order
    __shared__ __attribute__((aligned(32))) R Ut[16 * CK];
    const int e = blockIdx.y, head = blockIdx.x % a.heads, tile = blockIdx.x / a.heads;
    const int q0 = a.entry_q_start[e], n = a.entry_q_start[e + 1] - q0;
    if (n < a.shortest) return;
    const int first = __builtin_amdgcn_readfirstlane(rec_first_chunk(a.entry_q_start, e, a.shortest));
    if (first + (n + CK - 1) / CK > a.chunks || rec_odd_entry(a.odd, first, n, a.heads, head)) return;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / KVA_WAVE), lane = tid % KVA_WAVE;
    const int r = lane % 16, g = lane / 16, chunks = (n + CK - 1) / CK, col = 16 * tile + r;
    float *Sg = a.state + (size_t)a.entry_seat[e] * a.seat_stride + a.state_off + (size_t)head * D * a.vdim;
    R4 S[MT];                       // rows 16 (wave MT + t) + the lane's of the column
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int c = 0; c < 4; ++c) S[t][c] = Sg[(size_t)(16 * (wave * MT + t) + ck_channel<DELTA>(g, c)) * a.vdim + col];
    struct Operands {
        ck_f32x4 w[DELTA ? STEPS : 1], kt[MT][CK / 16], dec[MT];
        R4 uv;
    } o[2];
    auto fetch = [&](Operands &x, int chunk) {
        const ChunkBlock<D> b(a, first + min(chunk, chunks - 1), head);
        x.uv = ck_ld(reinterpret_cast<const R *>(b.ut) + ck_frag(tile, wave, 4, lane));
        if (DELTA)
#pragma unroll
            for (int s = 0; s < STEPS; ++s) x.w[DELTA ? s : 0] = ck_ld(b.w + ck_frag(wave, s, STEPS, lane));
#pragma unroll
        for (int t = 0; t < MT; ++t) {
#pragma unroll
            for (int s = 0; s < CK / 16; ++s) x.kt[t][s] = ck_ld(b.kt + ck_frag(wave * MT + t, s, 4, lane));
            x.dec[t] = ck_ld(b.g + 16 * (wave * MT + t) + 4 * g);
        }
    };
    auto step = [&](const Operands &x, Operands &next, int chunk) {
        const ChunkBlock<D> b(a, first + chunk, head);
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            if (DELTA) ck_st(&St[ck_frag(0, wave * MT + t, STEPS, lane)], S[t]);
            ck_st(b.st + ck_frag(tile, wave * MT + t, STEPS, lane), ck_narrow(S[t]));
        }
        __syncthreads();
        fetch(next, chunk + 1);
        R4 u = x.uv;
        if (DELTA) {
            // two chains of products: one alone waits for its own results
            R4 y[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
            for (int s = 0; s < STEPS; ++s)
                y[s % 2] = ck_mfma(ck_as(x.w[DELTA ? s : 0], R4{}), ck_ld(&St[ck_frag(0, s, STEPS, lane)]), y[s % 2]);
#pragma unroll
            for (int c = 0; c < 4; ++c) u[c] -= y[0][c] + y[1][c];
            ck_st(reinterpret_cast<R *>(b.ut) + ck_frag(tile, wave, 4, lane), u);
        }
        ck_st(&Ut[ck_frag(0, wave, 4, lane)], u);
        __syncthreads();
#pragma unroll
        for (int t = 0; t < MT; ++t) S[t] = ck_mul(S[t], ck_as(x.dec[t], R4{}));
#pragma unroll
        for (int s = 0; s < CK / 16; ++s) {
            const R4 y = ck_ld(&Ut[ck_frag(0, s, 4, lane)]);
#pragma unroll
            for (int t = 0; t < MT; ++t) S[t] = ck_mfma(ck_as(x.kt[t][s], R4{}), y, S[t]);
        }
    };
    fetch(o[0], 0);
    for (int chunk = 0; chunk < chunks; chunk += 2) {
        step(o[0], o[1], chunk);
        if (chunk + 1 < chunks) step(o[1], o[0], chunk + 1);
    }
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int c = 0; c < 4; ++c) Sg[(size_t)(16 * (wave * MT + t) + ck_channel<DELTA>(g, c)) * a.vdim + col] = (float)S[t][c];
}

// The delta rule's states with 4 NB value columns to a workgroup instead of 16, for launches that would leave units idle:
// v_mfma_f64_4x4x4_4b_f64 makes 16 rows of 4 columns (its four blocks are four groups of rows against the same columns), 9.6 ns an
// instruction where 16 x 16 take 30.4, so a quarter of the columns is a third of a chunk's products.  An operand's rows are held
// as by the 16 x 16 one; a result is one number a lane: lane (g, b, j) has row 4 b + g of column j.  S^T and U^T stand in
// LDS with the four rows g + 4 c of (16 rows, column) next to each other, as a lane (g, any b, j) takes them for the next product.
template <int D, int NB>
__global__ void __launch_bounds__(256)
chunk_states_narrow_kernel(ChunkArgs a) {
    constexpr int STEPS = D / 16, MT = D / 64;
    __shared__ __attribute__((aligned(32))) double St[NB][D * 4];
    __shared__ __attribute__((aligned(32))) double Ut[NB][CK * 4];
    const int e = blockIdx.y, head = blockIdx.x % a.heads, part = blockIdx.x / a.heads;
    const int q0 = a.entry_q_start[e], n = a.entry_q_start[e + 1] - q0;
    if (n < a.shortest) return;
    const int first = __builtin_amdgcn_readfirstlane(rec_first_chunk(a.entry_q_start, e, a.shortest));
    if (first + (n + CK - 1) / CK > a.chunks || rec_odd_entry(a.odd, first, n, a.heads, head)) return;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / KVA_WAVE), lane = tid % KVA_WAVE;
    const int g = lane / 16, b = lane / 4 % 4, j = lane % 4, chunks = (n + CK - 1) / CK;
    const int tile = 4 * NB * part / 16, sub = 4 * NB * part % 16 + j;          // of 16 columns; the lane's first one among them
    float *Sg = a.state + (size_t)a.entry_seat[e] * a.seat_stride + a.state_off + (size_t)head * D * a.vdim + 16 * tile + sub;
    double S[MT][NB];               // row 16 (wave MT + t) + 4 b + g of the columns
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int c = 0; c < NB; ++c) S[t][c] = Sg[(size_t)(16 * (wave * MT + t) + 4 * b + g) * a.vdim + 4 * c];
    struct Operands {
        ck_f32x4 w[STEPS], kt[MT][CK / 16];
        float dec[MT];
        double uv[NB];
    } o[2];
    // (in operand order the lane's element of 16 rows and its column)
    auto at = [&](int s, int steps, int c) { return ck_frag(tile, s, steps, sub + 4 * c + 16 * g) + b; };
    auto fetch = [&](Operands &x, int chunk) {
        const ChunkBlock<D> k(a, first + min(chunk, chunks - 1), head);
#pragma unroll
        for (int c = 0; c < NB; ++c) x.uv[c] = reinterpret_cast<const double *>(k.ut)[at(wave, 4, c)];
#pragma unroll
        for (int s = 0; s < STEPS; ++s) x.w[s] = ck_ld(k.w + ck_frag(wave, s, STEPS, lane));
#pragma unroll
        for (int t = 0; t < MT; ++t) {
#pragma unroll
            for (int s = 0; s < CK / 16; ++s) x.kt[t][s] = ck_ld(k.kt + ck_frag(wave * MT + t, s, 4, lane));
            x.dec[t] = k.g[16 * (wave * MT + t) + 4 * g + b];
        }
    };
    auto step = [&](const Operands &x, Operands &next, int chunk) {
        const ChunkBlock<D> k(a, first + chunk, head);
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int c = 0; c < NB; ++c) {
                St[c][((wave * MT + t) * 16 + 4 * g + j) * 4 + b] = S[t][c];
                k.st[at(wave * MT + t, STEPS, c)] = (float)S[t][c];
            }
        __syncthreads();
        fetch(next, chunk + 1);
        double y[NB][4];            // chains of products: one alone waits for its own results
#pragma unroll
        for (int c = 0; c < NB; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i) y[c][i] = 0.0;
#pragma unroll
        for (int s = 0; s < STEPS; ++s)
#pragma unroll
            for (int c = 0; c < NB; ++c) {
                const ck_f64x4 z = ck_ld(&St[c][(16 * s + 4 * g + j) * 4]);
#pragma unroll
                for (int i = 0; i < 4; ++i) y[c][i] = __builtin_amdgcn_mfma_f64_4x4x4f64((double)x.w[s][i], z[i], y[c][i], 0, 0, 0);
            }
#pragma unroll
        for (int c = 0; c < NB; ++c) {
            const double u = x.uv[c] - ((y[c][0] + y[c][1]) + (y[c][2] + y[c][3]));
            reinterpret_cast<double *>(k.ut)[at(wave, 4, c)] = u;
            Ut[c][(16 * wave + 4 * g + j) * 4 + b] = u;
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int c = 0; c < NB; ++c) {
                double lo = S[t][c] * x.dec[t], hi = 0.0;
#pragma unroll
                for (int s = 0; s < CK / 16; ++s) {
                    const ck_f64x4 z = ck_ld(&Ut[c][(16 * s + 4 * g + j) * 4]);
#pragma unroll
                    for (int i = 0; i < 4; i += 2) {
                        lo = __builtin_amdgcn_mfma_f64_4x4x4f64((double)x.kt[t][s][i], z[i], lo, 0, 0, 0);
                        hi = __builtin_amdgcn_mfma_f64_4x4x4f64((double)x.kt[t][s][i + 1], z[i + 1], hi, 0, 0, 0);
                    }
                }
                S[t][c] = lo + hi;
            }
    };
    fetch(o[0], 0);
    for (int chunk = 0; chunk < chunks; chunk += 2) {
        step(o[0], o[1], chunk);
        if (chunk + 1 < chunks) step(o[1], o[0], chunk + 1);
    }
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int c = 0; c < NB; ++c) Sg[(size_t)(16 * (wave * MT + t) + 4 * b + g) * a.vdim + 4 * c] = (float)S[t][c];
}

// One workgroup a (chunk, head), a wavefront every fourth 32 value columns, for all 64 tokens: O = Qd S + P U, every
// operand from where the other two kernels left it, in operand order.
template <int D, bool DELTA>
__global__ void __launch_bounds__(256)
chunk_outputs_kernel(ChunkArgs a) {
    constexpr int STEPS = D / 16;
    using R = typename CkSum<DELTA>::type;
    const int head = blockIdx.y;
    const ChunkPlace place = ck_find(a, blockIdx.x);
    const int e = place.entry, chunk = place.chunk;
    if (e < 0) return;
    const int q0 = a.entry_q_start[e], n = a.entry_q_start[e + 1] - q0;
    if (rec_odd_entry(a.odd, place.first, n, a.heads, head)) return;
    const int m = min(CK, n - chunk * CK), row0 = q0 + chunk * CK, tiles = a.vdim / 16;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KVA_WAVE), lane = threadIdx.x % KVA_WAVE, r = lane % 16, g = lane / 16;
    const ChunkBlock<D> b(a, blockIdx.x, head);
    for (int tile = 2 * wave; tile < tiles; tile += 8) {
        const int second = min(tile + 1, tiles - 1);        // (an odd last tile twice: the second result is dropped)
        ck_f64x4 acc[CK / 16][2];
#pragma unroll
        for (int t = 0; t < CK / 16; ++t) acc[t][0] = acc[t][1] = ck_f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
        for (int s = 0; s < STEPS; ++s) {
            const ck_f64x4 x = ck_wide(ck_ld(b.st + ck_frag(tile, s, STEPS, lane))), y = ck_wide(ck_ld(b.st + ck_frag(second, s, STEPS, lane)));
#pragma unroll
            for (int t = 0; t < CK / 16; ++t) {
                const ck_f64x4 q = ck_wide(ck_ld(b.q + ck_frag(t, s, STEPS, lane)));
                acc[t][0] = ck_mfma(q, x, acc[t][0]);
                acc[t][1] = ck_mfma(q, y, acc[t][1]);
            }
        }
        const R *ut = reinterpret_cast<const R *>(b.ut);
#pragma unroll
        for (int s = 0; s < CK / 16; ++s) {
            const ck_f64x4 x = ck_wide(ck_ld(ut + ck_frag(tile, s, 4, lane))), y = ck_wide(ck_ld(ut + ck_frag(second, s, 4, lane)));
#pragma unroll
            for (int t = s; t < CK / 16; ++t) {             // (P has no blocks above its diagonal)
                const ck_f64x4 p = ck_wide(ck_ld(b.p + ck_frag(t, s, 4, lane)));
                acc[t][0] = ck_mfma(p, x, acc[t][0]);
                acc[t][1] = ck_mfma(p, y, acc[t][1]);
            }
        }
#pragma unroll
        for (int t = 0; t < CK / 16; ++t)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int i = 16 * t + ck_token(g, c);
                float *o = a.out + (size_t)(row0 + i) * a.heads * a.vdim + head * a.vdim + r;
                if (i < m) {
                    o[16 * tile] = (float)acc[t][0][c];
                    if (tile + 1 < tiles) o[16 * (tile + 1)] = (float)acc[t][1][c];
                }
            }
    }
}

// Sizes these kernels are built for; other ones walk.
static bool ck_fits(int dim, int vdim) { return (dim == 64 || dim == 128) && vdim > 0 && vdim % 16 == 0; }

// floats of workspace for so many chunks of 64 tokens; 0: not for these sizes
extern "C" long long kva_recurrent_chunks_workspace(int chunks, int heads, int dim, int vdim) {
    if (!ck_fits(dim, vdim) || chunks < 0 || heads <= 0) return 0;
    return (long long)chunks * heads * (long long)ck_block(dim, vdim);
}

template <int D, bool DELTA>
static void ck_launch(const ChunkArgs &a, const ChunkInput &in, hipStream_t stream) {
    const dim3 grid(a.chunks, a.heads);
    if (in.channel_decay) hipLaunchKernelGGL((chunk_prepare_kernel<D, DELTA, true>), grid, dim3(256), 0, stream, a, in);
    else hipLaunchKernelGGL((chunk_prepare_kernel<D, DELTA, false>), grid, dim3(256), 0, stream, a, in);
    // A chain's length is its chunks whatever the workgroups hold, so the columns go to as many as a turn of the 256 units takes.
    // All three kernels at 4 / 8 / 16 columns a workgroup, heads of 128 x 128, us (a run of its own, 2 % above the figures at the top): 64 workgroups of 16 columns (8 heads, 2,048 tokens)
    // 121 / 139 / 160, 128 (16 heads) 194 / 182 / 199, 256 (32 heads) 400 / 383 / 333; of 64 x 64: 16 (4 heads, 2,048) 72 / 79 / 93,
    // 128 (32 heads, 1,024) 98 / 95 / 101.
    const int tiles = a.heads * (a.vdim / 16), entries = min(a.entries, a.chunks);
    if (DELTA && (long long)tiles * entries <= 64) hipLaunchKernelGGL((chunk_states_narrow_kernel<D, 1>), dim3(tiles * 4, a.entries), dim3(256), 0, stream, a);
    else if (DELTA && (long long)tiles * entries <= 128) hipLaunchKernelGGL((chunk_states_narrow_kernel<D, 2>), dim3(tiles * 2, a.entries), dim3(256), 0, stream, a);
    else hipLaunchKernelGGL((chunk_states_kernel<D, DELTA>), dim3(tiles, a.entries), dim3(256), 0, stream, a);
    hipLaunchKernelGGL((chunk_outputs_kernel<D, DELTA>), grid, dim3(256), 0, stream, a);
}

static int ck_check(const char *what, const ChunkArgs &a, int dim, long long work_floats) {
    KVA_REQUIRE(a.out && a.state && a.entry_q_start && a.entry_seat && a.work && a.odd, "%s: missing operand", what);
    KVA_REQUIRE(ck_fits(dim, a.vdim), "%s: chunks are built for key sizes 64 and 128 and value sizes that are multiples of 16, not %d x %d", what, dim, a.vdim);
    KVA_REQUIRE(a.heads > 0 && a.heads <= 65535 && a.kv_heads > 0 && a.heads % a.kv_heads == 0, "%s: %d heads over %d key heads", what, a.heads, a.kv_heads);
    KVA_REQUIRE(a.entries > 0 && a.entries <= 65535 && a.chunks > 0 && a.shortest >= 1, "%s: %d chunks in %d entries", what, a.chunks, a.entries);
    KVA_REQUIRE((uintptr_t)a.work % 32 == 0, "%s: the workspace must start at a multiple of 32 bytes", what);
    KVA_REQUIRE(a.heads * (long long)(a.vdim / 16) < (1LL << 31), "%s: %d heads of %d values", what, a.heads, a.vdim);
    KVA_REQUIRE(work_floats >= kva_recurrent_chunks_workspace(a.chunks, a.heads, dim, a.vdim), "%s: the workspace is too small", what);
    return KVA_OK;
}

// The same operands as kva_gated_delta_rule; entries of fewer than `shortest` tokens are left alone, the others have
// `chunks` chunks of 64 tokens (the last one of each may be shorter) between them.  `odd`: int32 [chunks, heads].
extern "C" int kva_gated_delta_rule_chunks(float *out, float *state, long long seat_stride, int state_off, const float *qkv,
                                           int conv_stride, const void *y, int y_dtype, int y_stride, int beta_off,
                                           int decay_off, const float *a_log, const float *dt_bias, float unit_eps,
                                           const float *channel_decay, int decay_stride, const int *entry_q_start,
                                           const int *entry_seat, int entries, int heads, int kv_heads, int dim, int vdim,
                                           int shortest, int chunks, float *work, long long work_floats,
                                           int *odd, hipStream_t stream) {
    const ChunkArgs a{out, state, (size_t)seat_stride, state_off, entry_q_start, entry_seat, heads, kv_heads, vdim, entries, shortest, chunks, work, odd};
    if (int rc = ck_check("gated_delta_rule", a, dim, work_floats)) return rc;
    KVA_REQUIRE(qkv && y && ((a_log && dt_bias) || (channel_decay && decay_stride >= heads * dim)), "gated_delta_rule: missing operand");
    KVA_REQUIRE((uintptr_t)qkv % 16 == 0 && conv_stride % 4 == 0, "gated_delta_rule: rows of q, k and v must start at multiples of 16 bytes");
    const ChunkInput in{qkv, y, conv_stride, y_dtype, y_stride, 0, kv_heads * dim, 2 * kv_heads * dim, beta_off, decay_off, 0,
                        a_log, dt_bias, channel_decay, nullptr, decay_stride, unit_eps, 1.0 / sqrt((double)dim)};
    if (dim == 64) ck_launch<64, true>(a, in, stream);
    else ck_launch<128, true>(a, in, stream);
    KVA_CHECK_LAUNCH("gated_delta_rule_chunks");
    return KVA_OK;
}

// The same operands as kva_gated_linear_attention.
extern "C" int kva_gated_linear_attention_chunks(float *out, float *state, long long seat_stride, int state_off,
                                                 const void *y, int y_dtype, int y_stride, int q_off, int k_off, int v_off,
                                                 const float *alpha, int alpha_stride, float q_mul, const float *head_decay,
                                                 int act, const int *entry_q_start, const int *entry_seat, int entries,
                                                 int heads, int dim, int vdim, int shortest, int chunks,
                                                 float *work, long long work_floats, int *odd, hipStream_t stream) {
    const ChunkArgs a{out, state, (size_t)seat_stride, state_off, entry_q_start, entry_seat, heads, heads, vdim, entries, shortest, chunks, work, odd};
    if (int rc = ck_check("gated_linear_attention", a, dim, work_floats)) return rc;
    KVA_REQUIRE(y && ((alpha && alpha_stride >= heads * dim) || (!alpha && head_decay)), "gated_linear_attention: missing operand");
    KVA_REQUIRE(act == 0 || act == 1, "gated_linear_attention: activation %d is neither none (0) nor silu (1)", act);
    const ChunkInput in{nullptr, y, 0, y_dtype, y_stride, q_off, k_off, v_off, 0, 0, act, nullptr, nullptr, alpha, head_decay,
                        alpha_stride, 0.f, q_mul};
    if (dim == 64) ck_launch<64, false>(a, in, stream);
    else ck_launch<128, false>(a, in, stream);
    KVA_CHECK_LAUNCH("gated_linear_attention_chunks");
    return KVA_OK;
}
