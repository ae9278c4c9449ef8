// True fp32 matrix product for the 32-bit path: C[M,N] = A[M,K] * W[N,K]^T, everything
// row-major fp32, on the matrix cores' 32-bit instruction (no reduced-precision mode).
//
// It stands where the reference calls cublasGemmEx with the OP_T/OP_N trick for a row-major
// [out,in] weight (base/src/engine.cu:652-671).  The order of an output's sum depends on K alone:
// K is cut into parts (gf_part), a part's products go 16 columns at a time through four
// v_mfma_f32_16x16x4_f32 into one accumulator (instruction j takes columns j, j + 4, j + 8, j + 12 of the 16:
// what the four lane groups hold at place j of the 16 bytes each of them loads), the parts of the front half are
// added in order, those of the back half are, and the two sums are added.  Both kernels below do just that, so a row
// of C does not depend on M, on the tile it falls in, on which kernel ran or on the other rows: the fp32 path is
// bit-identical under any batching.
//
// us a call, weights from memory, against one kernel of 64 x 64 tiles and plain FMAs for every M (before -> now;
// relative error against 64 bits at K = 2,048 / 8,192: 8e-7 / 1.6e-6 -> 2.1e-7 / 4.1e-7):
//   rows x outputs x K    3 x 128,256 x 2,048: 480 -> 231 -> 189 (5.6 TB/s)  3 x 16,384 x 2,048: 147 -> 35 -> 30 (4.5)
//                         3 x 2,048 x 8,192: 544 -> 20 -> 18 (3.8 TB/s)  3 x 2,048 x 2,048: 7.6 -> 6.7
//                         32 x 2,048 x 8,192: 545 -> 58                  64 x 2,048 x 8,192: 559 -> 59 (the tiles: 167)
// and of those with more rows, plain FMAs -> tiles through registers, K's halves on eight wavefronts -> the ring:
//                         64 x 128,256 x 2,048: 532 -> 369 -> 310        402 x 16,384 x 2,048: 449 -> 340 -> 250 (108 TFLOP/s)
//                         517 x 16,384 x 2,048: 424 -> 287 (121)         517 x 2,048 x 8,192: 308 -> 178 (97)
//                         517 x 3,072 x 2,048: 85 -> 66                  517 x 2,048 x 2,048: 85 -> 50
//                         100 x 2,048 x 8,192: 165 -> 85                 2,048 x 16,384 x 2,048: 1,748 -> 1,304 -> 1,009 (136)
// With K up to 128 a tile's result takes longer than its products: 2,000 x 16,384 x 128 130 -> 162 -> 105.
#include "common.h"
#include "lds_product.h"

typedef float gf_f32x4 __attribute__((ext_vector_type(4)));

#define GF_STEP 16                  // columns of K that one 16-byte load a lane covers
#define GF_MAX_PARTS 16
#define GF_ROWS_UP_TO 64            // rows up to which the few-rows kernel may run (gf_few_rows)
#define GF_BM 64                    // the tile kernel: rows a workgroup, columns of K a round, padding of a row in LDS
#define GF_BK 32
#define GF_PAD 4

// Columns of K a part takes: a sixteenth of K in whole rounds of the tile kernel - so at most 16 parts.
static inline int gf_part(int K) {
    const int rounds = (K + GF_BK - 1) / GF_BK;
    return (rounds + GF_MAX_PARTS - 1) / GF_MAX_PARTS * GF_BK;
}

// Parts of the front half: an output is (sum of the front parts, in order) + (sum of the others, in order).
__host__ __device__ inline int gf_half(int parts) { return (parts + 1) / 2; }

// four neighbouring elements of a row, zeros past the row's end or for a row that is not there
template <bool VEC>
__device__ inline gf_f32x4 gf_load(const float *__restrict__ p, int row, int rows, int k, int K, int ld) {
    gf_f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (row < rows) {
        const float *a = p + (size_t)row * ld + k;
        if (VEC) {
            if (k < K) v = *reinterpret_cast<const gf_f32x4 *>(a);      // (K is a multiple of 4)
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (k + e < K) v[e] = a[e];
        }
    }
    return v;
}

// Few rows: what bounds it is the stream of W.  A workgroup takes 16 outputs and 16 MT rows, a wavefront one part of
// K (all parts of a tile of W are on their way at once, `DEPTH` steps of each in registers before the first
// product); the parts are added in order through LDS.  PAIR: up to 8 rows and 8 outputs a workgroup, a wavefront
// takes two parts - operand rows 0-7 the first, 8-15 the second, on both sides, so that the products wanted are
// the two blocks on the diagonal.  That puts twice the workgroups on a narrow matrix (128 of them would leave
// half the chip without a share of the stream); from 8,192 outputs on there are enough, and twice the rows a workgroup are the
// faster way (3 rows, K = 2,048, pairs / not: 6,144 outputs 15.0 / 16.4 us, 8,192 18.3 / 18.4, 16,384 33.7 / 29.8, 128,256 216 /
// 189).  W goes through the caches: its loads take half a line of 128 bytes each, and with the non-temporal hint the line was
// asked for twice (128,256 outputs 231 -> 216 us, 2,048 x 8,192 20.1 -> 18.7).
template <int MT, int DEPTH, bool PAIR, bool VEC>
__global__ void __launch_bounds__(KVA_WAVE * GF_MAX_PARTS)
gemm_f32_rows_kernel(float *__restrict__ C, const float *__restrict__ A, const float *__restrict__ W, int M, int N,
                     int K, int lda, int ldw, int ldc, int part) {
    constexpr int OUT = PAIR ? 8 : 16;
    __shared__ float sums[GF_MAX_PARTS][MT][OUT][OUT + 1];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KVA_WAVE);     // (scalar: so are the branches around the products)
    const int lane = threadIdx.x % KVA_WAVE, r = lane % 16, g = lane / 16;
    const int n0 = blockIdx.x * OUT, m0 = blockIdx.y * 16 * MT;
    const int first = PAIR ? 2 * wave : wave;                       // the wavefront's (first) part
    const int steps = (min(K, (first + 1) * part) - first * part + GF_STEP - 1) / GF_STEP;
    const int mine = PAIR ? first + r / 8 : first, lo = mine * part, hi = min(K, lo + part);     // (lo may lie past K: zeros)
    const int wr = n0 + (PAIR ? r % 8 : r), ar = m0 + (PAIR ? r % 8 : r);
    gf_f32x4 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = gf_f32x4{0.f, 0.f, 0.f, 0.f};
    gf_f32x4 w[2][DEPTH], x[2][DEPTH][MT];
    auto fetch = [&](int buf, int s0) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            const int k = lo + (s0 + d) * GF_STEP + 4 * g;          // (past the part's end: zeros)
            w[buf][d] = gf_load<VEC>(W, wr, N, k, hi, ldw);
#pragma unroll
            for (int t = 0; t < MT; ++t) x[buf][d][t] = gf_load<VEC>(A, ar + 16 * t, M, k, hi, lda);
        }
    };
    auto products = [&](int buf, int s0) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d)
            if (s0 + d < steps)
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int t = 0; t < MT; ++t)
                        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[buf][d][j], x[buf][d][t][j], acc[t], 0, 0, 0);
    };
    fetch(0, 0);
    for (int s0 = 0; s0 < steps; s0 += 2 * DEPTH) {
        fetch(1, s0 + DEPTH);
        products(0, s0);
        fetch(0, s0 + 2 * DEPTH);
        products(1, s0 + DEPTH);
    }
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {                               // [row][output]
            if (!PAIR) sums[wave][t][r][4 * g + i] = acc[t][i];
            else if (r / 8 == g / 2) sums[mine][t][r % 8][(4 * g + i) % 8] = acc[t][i];
        }
    __syncthreads();
    const int parts = (K + part - 1) / part, half = gf_half(parts);
    for (int e = threadIdx.x; e < MT * OUT * OUT; e += blockDim.x) {
        const int t = e / (OUT * OUT), m = e % (OUT * OUT) / OUT, n = e % OUT;
        float front = 0.f, back = 0.f;
        for (int p = 0; p < half; ++p) front += sums[p][t][m][n];
        for (int p = half; p < parts; ++p) back += sums[p][t][m][n];
        if (m0 + 16 * t + m < M && n0 + n < N) C[(size_t)(m0 + 16 * t + m) * ldc + n0 + n] = front + back;
    }
}

// Many rows that start at any address, or more than 8 MiB apart: bound by the matrix cores, at odd addresses by loads of
// single elements.  A workgroup
// takes 64 rows x 32 NT outputs: four wavefronts (32 x 16 NT each) the front half of the parts, four the back half -
// two wavefronts a SIMD where the tiles are about as many as the compute units.  32 columns of both operands of
// each half go through LDS at a time (rows 36 elements apart: the 16 rows of an operand read start in different
// banks), the next ones' loads in flight over the products.  Workgroups of one stripe of outputs are neighbours on
// one die, whose L2 then holds that stripe of W for all of their rows.
template <int NT>
struct GfTile {
    float a[2][GF_BM][GF_BK + GF_PAD], w[2][32 * NT][GF_BK + GF_PAD];
};

template <int NT, bool VEC>
__global__ void __launch_bounds__(512)
gemm_f32_tile_kernel(float *__restrict__ C, const float *__restrict__ A, const float *__restrict__ W, int M, int N,
                     int K, int lda, int ldw, int ldc, int part, int mtiles, int tiles) {
    constexpr int BN = 32 * NT, AL = GF_BM * GF_BK / 4 / 256, WL = BN * GF_BK / 4 / 256;
    __shared__ GfTile<NT> lds[2];
    const int per = (tiles + 7) / 8, tile = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if (tile >= tiles) return;                                       // (the whole workgroup)
    const int m0 = tile % mtiles * GF_BM, n0 = tile / mtiles * BN;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KVA_WAVE), back = wave / 4;
    const int tid = threadIdx.x % 256, lane = tid % KVA_WAVE, r = lane % 16, g = lane / 16;
    const int wm = wave % 2 * 32, wn = wave / 2 % 2 * 16 * NT;
    const int split = min(K, gf_half((K + part - 1) / part) * part); // the back half's first column
    const int lo = back ? split : 0, hi = back ? K : split;
    GfTile<NT> &L = lds[back];
    gf_f32x4 acc[NT][2], tot[NT][2], la[2][AL], lw[2][WL];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = tot[i][j] = gf_f32x4{0.f, 0.f, 0.f, 0.f};
    const int lrow = tid / 8, lk = tid % 8 * 4;                      // 32 rows a pass, 8 lanes a row
    auto fetch = [&](int set, int k0) {                              // (past the half's end: zeros)
#pragma unroll
        for (int i = 0; i < AL; ++i) la[set][i] = gf_load<VEC>(A, m0 + lrow + 32 * i, M, k0 + lk, hi, lda);
#pragma unroll
        for (int i = 0; i < WL; ++i) lw[set][i] = gf_load<VEC>(W, n0 + lrow + 32 * i, N, k0 + lk, hi, ldw);
    };
    auto put = [&](int set) {
#pragma unroll
        for (int i = 0; i < AL; ++i) *reinterpret_cast<gf_f32x4 *>(&L.a[set][lrow + 32 * i][lk]) = la[set][i];
#pragma unroll
        for (int i = 0; i < WL; ++i) *reinterpret_cast<gf_f32x4 *>(&L.w[set][lrow + 32 * i][lk]) = lw[set][i];
    };
    int left = part;                                                 // columns of the current part still to come
    auto round = [&](int set) {
#pragma unroll
        for (int s = 0; s < GF_BK / GF_STEP; ++s) {
            gf_f32x4 a[2], w[NT];
#pragma unroll
            for (int j = 0; j < 2; ++j)
                a[j] = *reinterpret_cast<const gf_f32x4 *>(&L.a[set][wm + 16 * j + r][s * GF_STEP + 4 * g]);
#pragma unroll
            for (int i = 0; i < NT; ++i)
                w[i] = *reinterpret_cast<const gf_f32x4 *>(&L.w[set][wn + 16 * i + r][s * GF_STEP + 4 * g]);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < NT; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[i][e], a[j][e], acc[i][j], 0, 0, 0);
        }
        left -= GF_BK;
        if (left == 0) {
            left = part;
#pragma unroll
            for (int i = 0; i < NT; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
#pragma unroll
                    for (int c = 0; c < 4; ++c) tot[i][j][c] += acc[i][j][c];
                    acc[i][j] = gf_f32x4{0.f, 0.f, 0.f, 0.f};
                }
        }
    };
    // Two rounds at a time: while one is multiplied from its LDS buffer the next one waits in registers and the one
    // after that is asked for.  The front half is never the shorter one: its barriers are both halves'.
    fetch(0, lo);
    fetch(1, lo + GF_BK);
    for (int d = 0; d < split; d += 2 * GF_BK) {
        put(0);
        __syncthreads();
        fetch(0, lo + d + 2 * GF_BK);
        if (lo + d < hi) round(0);
        if (d + GF_BK >= split) break;                               // (of the front half, which no half is longer than)
        put(1);
        __syncthreads();
        fetch(1, lo + d + 3 * GF_BK);
        if (lo + d + GF_BK < hi) round(1);
    }
    __syncthreads();
    if (left != part)                                                // a last, shorter part
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int c = 0; c < 4; ++c) tot[i][j][c] += acc[i][j][c];
    // the back half's sums to the front half, through LDS (the operands there have been read)
    gf_f32x4 *over = reinterpret_cast<gf_f32x4 *>(&lds[0]);
    static_assert(sizeof(lds) >= sizeof(gf_f32x4) * 256 * NT * 2, "the back half's sums fit where the operands were");
    const bool halves = split < K;                                   // (else there is nothing in the back half)
    if (back && halves)
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) over[(i * 2 + j) * 256 + tid] = tot[i][j];
    __syncthreads();
    if (back) return;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int m = m0 + wm + 16 * j + r;
        if (m >= M) continue;
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            const int n = n0 + wn + 16 * i + 4 * g;
            float *c = C + (size_t)m * ldc + n;
            gf_f32x4 o = {0.f, 0.f, 0.f, 0.f};
            if (halves) o = over[(i * 2 + j) * 256 + tid];
            gf_f32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = tot[i][j][e] + o[e];
            if (VEC && n + 3 < N) *reinterpret_cast<gf_f32x4 *>(c) = v;
            else
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) c[e] = v[e];
        }
    }
}

// Many rows, every row of both operands at a multiple of 16 bytes: bound by the matrix cores (a 32-bit product takes 16 times the
// cycles of a 16-bit one; they give 142-152 TFLOP/s to one wavefront a SIMD, 156 to two), and by how evenly tiles divide among the
// compute units.  A workgroup of four wavefronts takes 16 MT rows
// x 64 outputs, a wavefront all of its rows x 16; MT is chosen so that the fullest compute unit has the least to do (gf_rows_a_tile).
// 32 columns of both operands are a stage; they go straight to LDS (buffer loads, 16 bytes a lane, the eight 16-byte pieces of
// a row in the order piece ^ row % 8, so that the rows of an operand read lie in different banks), STAGES - 1 stages on their
// way or waiting.  16 columns' operands are read into registers while the 16 before are multiplied, over the one barrier a stage
// too: a wavefront that has its SIMD to itself keeps it busy.  Workgroups of one stripe of outputs are neighbours on one die,
// whose L2 then holds that stripe of W for all of their rows.
template <int MT, int STAGES>
__global__ void __launch_bounds__(256, 2)
gemm_f32_ring_kernel(float *__restrict__ C, const float *__restrict__ A, const float *__restrict__ W, int M, int N,
                     int K, int lda, int ldw, int ldc, int part, int mtiles, int tiles) {
    constexpr int PIECES = 2 * MT + 8, LOADS = (PIECES + 3) / 4;     // of 1 KiB: 8 rows of 32; a wavefront's
    __shared__ __align__(16) float ring[STAGES][PIECES * 256];       // rows of A, then rows of W
    const int per = (tiles + 7) / 8, tile = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if (tile >= tiles) return;                                       // (the whole workgroup)
    const int m0 = tile % mtiles * 16 * MT, n0 = tile / mtiles * 64;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KVA_WAVE), lane = threadIdx.x % KVA_WAVE, r = lane % 16, g = lane / 16;
    const float *atile = A + (size_t)m0 * lda, *wtile = W + (size_t)n0 * ldw;
    const int arows = min(16 * MT, M - m0), wrows = min(64, N - n0);
    const Buffer abuf = buffer_at(atile, ((size_t)(arows - 1) * lda + K) * sizeof(float)),
                 wbuf = buffer_at(wtile, ((size_t)(wrows - 1) * ldw + K) * sizeof(float));
    int from[LOADS], to[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        // (one piece too few for all wavefronts: the last one again, so that all have as many loads on their way)
        const int piece = min(wave + 4 * i, PIECES - 1);
        from[i] = 4 * (piece < 2 * MT ? min(8 * piece + lane / 8, arows - 1) * lda : min(8 * (piece - 2 * MT) + lane / 8, wrows - 1) * ldw);
        to[i] = piece * 256;
    }
    const int column = 4 * ((lane % 8) ^ (lane / 8));
    auto load = [&](int i, int slot, int k0) {                       // (past the end: what is there is left out of the products)
        buffer_to_lds(to[i] < 2 * MT * 256 ? abuf : wbuf, from[i] + 4 * min(k0 + column, K - 4), 0, &ring[slot][to[i]]);
    };
    gf_f32x4 acc[MT], tot[MT], front[MT], a[2][MT], w[2];
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[j] = tot[j] = front[j] = gf_f32x4{0.f, 0.f, 0.f, 0.f};
    auto read = [&](int i, int set, int slot) {                      // half `set` of a stage: W's rows, then A's
        const float *base = &ring[slot][r * 32 + 4 * ((4 * set + g) ^ (r & 7))];
        if (i == 0) w[set] = *reinterpret_cast<const gf_f32x4 *>(base + (2 * MT + 2 * wave) * 256);
        else a[set][i - 1] = *reinterpret_cast<const gf_f32x4 *>(base + 2 * (i - 1) * 256);
    };
    const int rounds = (K + GF_BK - 1) / GF_BK, split = gf_half((K + part - 1) / part) * part;
    auto cut = [&](int set, int k0) {                                // columns past the end are left out
        if (k0 + 4 * g >= K) {
            w[set] = gf_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < MT; ++j) a[set][j] = gf_f32x4{0.f, 0.f, 0.f, 0.f};
        }
    };
    // 16 columns' products, and behind the i-th of them what `behind(i)` asks for: a wavefront waits where the next product is not
    // taken yet, so one load at a time is issued while a product runs
    auto products = [&](int set, auto behind) {
#pragma unroll
        for (int i = 0; i < 4 * MT; ++i) {
            acc[i % MT] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[set][i / MT], a[set][i % MT][i / MT], acc[i % MT], 0, 0, 0);
            behind(i);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    __builtin_amdgcn_s_waitcnt(0xc07f);     // (arguments' loads have arrived: the waits below are for operands alone, and counted)
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
#pragma unroll
        for (int i = 0; i < LOADS; ++i) load(i, s, s * GF_BK);
    wait_and_meet<(STAGES - 2) * LOADS>();
#pragma unroll
    for (int i = 0; i <= MT; ++i) read(i, 0, 0);
    int slot = 0, left = part;                                       // columns of the current part still to come
    auto round = [&](int t, bool ends) {                             // (`ends`: a constant where this is put in)
        const int k0 = t * GF_BK, next = slot + 1 == STAGES ? 0 : slot + 1, before = slot == 0 ? STAGES - 1 : slot - 1;
        if (ends) cut(0, k0);
        products(0, [&](int i) {
            if (i <= MT) read(i, 1, slot);
        });
        if (ends) cut(1, k0 + GF_STEP);
        products(1, [&](int i) {
            // the next stage is there; the slot of the stage before is free: every wavefront has multiplied with it
            if (i == 0) wait_and_meet<(STAGES - 3) * LOADS>();
            if (i <= MT) read(i, 0, next);
            else if (i <= MT + LOADS) load(i - MT - 1, before, k0 + (STAGES - 1) * GF_BK);
            if (i == 4 * MT - 1)                                     // (what had no product to be behind)
#pragma unroll
                for (int j = 4 * MT - MT - 1; j < LOADS; ++j) load(j, before, k0 + (STAGES - 1) * GF_BK);
        });
        slot = next;
        left -= GF_BK;
        if (left == 0 || t + 1 == rounds) {
            left = part;
#pragma unroll
            for (int j = 0; j < MT; ++j) {
#pragma unroll
                for (int c = 0; c < 4; ++c) tot[j][c] += acc[j][c];
                acc[j] = gf_f32x4{0.f, 0.f, 0.f, 0.f};
            }
            if (k0 + GF_BK == split)                                 // the front half is done
#pragma unroll
                for (int j = 0; j < MT; ++j) {
                    front[j] = tot[j];
                    tot[j] = gf_f32x4{0.f, 0.f, 0.f, 0.f};
                }
        }
    };
    for (int t = 0; t + 1 < rounds; ++t) round(t, false);
    round(rounds - 1, true);
    wait_and_meet<0>();                                              // nothing is on its way to LDS any more
    if (rounds * GF_BK < split)                                      // (one part, and a short one: it is the front half)
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            front[j] = tot[j];
            tot[j] = gf_f32x4{0.f, 0.f, 0.f, 0.f};
        }
    const int n = n0 + 16 * wave + 4 * g;
#pragma unroll
    for (int j = 0; j < MT; ++j) {
        const int m = m0 + 16 * j + r;
        if (m >= M) continue;
        float *c = C + (size_t)m * ldc + n;
        gf_f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = front[j][e] + tot[j][e];
        if (n + 3 < N) *reinterpret_cast<gf_f32x4 *>(c) = v;
        else
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (n + e < N) c[e] = v[e];
    }
}

// Rows a tile of the ring kernel takes (16 times the result): the compute unit with the most tiles is what a launch waits for.
// (us by rows a tile, 16 / 32 / 48 / 64 / 80 / 112 / 128: 517 x 16,384 x 2,048 350 300 292 301 292 287 322; 517 x 2,048 x 8,192
// 197 198 203 256 178 237 264; 250 x 16,384 x 2,048 182 153 167 137 169 176 133; 70 x 3,072 x 2,048 18 24 33 39 48 63 70.)
static int gf_rows_a_tile(int M, int N) {
    int best = 1;
    long long least = -1;
    for (int mt = 1; mt <= 8; ++mt) {
        const long long tiles = (long long)((M + 16 * mt - 1) / (16 * mt)) * ((N + 63) / 64), cost = (tiles + 255) / 256 * (2 * mt + 1);
        if (least < 0 || cost <= least) { least = cost; best = mt; }
    }
    return best;
}

// Whether few rows go to the kernel that streams W.  It makes 32 rows a pass over W, in a workgroup per 16 outputs and pass, and shares
// nothing between workgroups: its time goes up by half where a compute unit gets a second one, and with the rows of a pass.  The ring
// takes much the same from 17 to 64 rows, and longer than one such workgroup: a wavefront alone on its SIMD waits for W.  Weights from
// memory (sets of 800 MB and more), few-rows kernel / ring, us at K = 1,024, 2,048, 4,096, 8,192, 14,336:
//   one a unit:  17 rows, 2,048 outputs  9.0/14.0  14.1/24.9  25.0/45.2  45.1/88.0  77.9/156    32 rows, 4,096  10.9/14.2  18.6/25.9  31.9/46.3
//                64 rows, 2,048  10.0/13.8  16.5/24.8  29.5/44.6  55.0/87.4  95.5/154                           59.7/91.9  112/162
//   up to one and a half (two passes):  33 rows, 2,560  11.4/14.0  18.6/25.1  32.8/45.6  58.8/88.8  102/158     48 rows, 3,072  14.8/14.1
//                24.7/25.2  44.3/45.8  85.1/89.7  148/158    64 rows, 3,072  16.5/14.1  28.5/25.3  52.0/45.6  99.0/89.1  179/158
//   up to two:   17 rows, 8,192  16.3/15.4  27.5/27.4  51.0/51.9  93.2/100  166/181      20 rows, 4,608  15.7/14.5  26.6/25.9  48.2/47.1
//                90.7/92.9  162/163    24 rows, 4,608  95.7/92.5 at 8,192    40 rows, 4,096  15.7/14.5  27.0/25.5  47.5/46.1  90.0/90.9  160/161
//   more:        17 rows, 10,240  22.0/16.5  37.9/29.4  71.5/57.0  133/107  233/187      33 rows, 6,144  22.5/15.4  39.4/27.4  72.0/50.8
// Below K = 1,024 the ring is ahead from the second workgroup on (K = 512: 33 rows, 2,560 7.4 / 6.7).  Where the line is wrong it costs 5 % at most
// (48 rows of 3,072 outputs at K = 1,024; 17 rows of 7,168 at K = 4,096).  Without the ring the tiles are what many rows go to, and take a third
// longer: few-rows kernel / tiles, 17-32 rows, 8,192 outputs 28-33 / 46, 16,384 52-65 / 50; 33-64 rows, 4,096 28-33 / 45, 6,144 42-48 /
// 46, 8,192 51-62 / 46.
static bool gf_few_rows(int M, int N, int K, bool ring) {
    if (M <= 16) return true;
    if (M > GF_ROWS_UP_TO) return false;
    const int passes = (M + 31) / 32;
    const long long streamed = (long long)N * passes;              // 16 of them a workgroup, 4,096 one workgroup a compute unit
    if (!ring) return streamed <= 14336;
    return streamed <= 4096 || (streamed <= 6144 && passes == 2 && M <= 48 && K >= 1024) || (streamed <= 8192 && M <= 20 * passes && K >= 6144);
}

template <bool VEC>
static void gf_launch(float *C, const float *A, const float *W, int M, int N, int K, int lda, int ldw, int ldc,
                      bool ring, hipStream_t stream) {
    const int part = gf_part(K), parts = (K + part - 1) / part;
    if (gf_few_rows(M, N, K, ring)) {
        const int out = M <= 8 && N < 8192 ? 8 : 16;
        const dim3 grid((N + out - 1) / out, (M + 31) / 32), block(KVA_WAVE * (out == 8 ? (parts + 1) / 2 : M <= 16 ? parts : max(4, parts)));    // (four for the sums' last step)
        if (out == 8)
            hipLaunchKernelGGL((gemm_f32_rows_kernel<1, 2, true, VEC>), grid, block, 0, stream, C, A, W, M, N, K, lda, ldw, ldc, part);
        else if (M <= 16)
            hipLaunchKernelGGL((gemm_f32_rows_kernel<1, 2, false, VEC>), grid, block, 0, stream, C, A, W, M, N, K, lda, ldw, ldc, part);
        else
            hipLaunchKernelGGL((gemm_f32_rows_kernel<2, 2, false, VEC>), grid, block, 0, stream, C, A, W, M, N, K, lda, ldw, ldc, part);
        return;
    }
    if (ring) {
        const int mt = gf_rows_a_tile(M, N), mtiles = (M + 16 * mt - 1) / (16 * mt), tiles = mtiles * ((N + 63) / 64);
#define GF_RING(MT, STAGES)                                                                                              \
    hipLaunchKernelGGL((gemm_f32_ring_kernel<MT, STAGES>), dim3((tiles + 7) / 8 * 8), dim3(256), 0, stream, C, A, W, M, N, K, lda, ldw, \
                       ldc, part, mtiles, tiles)
        switch (mt) {
            case 1: GF_RING(1, 4); break;
            case 2: GF_RING(2, 4); break;
            case 3: GF_RING(3, 4); break;
            case 4: GF_RING(4, 4); break;
            case 5: GF_RING(5, 4); break;
            case 6: GF_RING(6, 3); break;
            case 7: GF_RING(7, 3); break;
            default: GF_RING(8, 3); break;
        }
#undef GF_RING
        return;
    }
    const int mtiles = (M + GF_BM - 1) / GF_BM, wide = mtiles * ((N + 127) / 128), narrow = mtiles * ((N + 63) / 64);
    if (wide >= 256)
        hipLaunchKernelGGL((gemm_f32_tile_kernel<4, VEC>), dim3((wide + 7) / 8 * 8), dim3(512), 0, stream, C, A, W, M, N, K, lda, ldw, ldc, part, mtiles, wide);
    else
        hipLaunchKernelGGL((gemm_f32_tile_kernel<2, VEC>), dim3((narrow + 7) / 8 * 8), dim3(512), 0, stream, C, A, W, M, N, K, lda, ldw, ldc, part, mtiles, narrow);
}

extern "C" int kva_gemm_nt_f32(float *C, const float *A, const float *W, int M, int N, int K,
                               int lda, int ldw, int ldc, hipStream_t stream) {
    KVA_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_f32: bad sizes M=%d N=%d K=%d", M, N, K);
    KVA_REQUIRE(lda >= K && ldw >= K && ldc >= N, "gemm_f32: leading dimensions too small");
    if (M == 0) return KVA_OK;
    KVA_REQUIRE((M + GF_BM - 1) / GF_BM <= 65535, "gemm_f32: M=%d is too large for one launch", M);
    // 16-byte loads and stores where every row of all three starts at a multiple of 16 bytes; the ring where a tile's rows lie
    // within 2 GiB too (its loads have 32-bit offsets)
    const bool vec = K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && ldc % 4 == 0 && ((uintptr_t)A | (uintptr_t)W | (uintptr_t)C) % 16 == 0;
    if (vec) gf_launch<true>(C, A, W, M, N, K, lda, ldw, ldc, lda <= 1 << 21 && ldw <= 1 << 21, stream);
    else gf_launch<false>(C, A, W, M, N, K, lda, ldw, ldc, false, stream);
    KVA_CHECK_LAUNCH("gemm_nt_f32");
    return KVA_OK;
}
