// Token sampling on the device: greedy argmax (lowest id wins ties) and temperature sampling by
// inverse CDF with a counter-based uniform, both over optionally penalised fp32 logits.
//
// What is computed is what the reference's sampling kernels compute (base/src/kernels.cu:489-835;
// numpy mirror python/sampling_reference.py:26-89): the token of a temperature row is the first i
// whose cumulative weight w_0 + ... + w_i, w_i = exp((l_i - max l) / T), exceeds u * sum(w) - the
// flat CDF's searchsorted(cdf, target, side="right") - with u = counter_uniform(seed, key, step);
// a greedy row takes the largest logit, the lowest id among equals; tokens marked in the request's
// mask row are penalised first (l > 0 ? l / p : l * p).
//
// How: two launches, and the logits are read once.
//   1. sample_scan_kernel, one workgroup per (chunk of a row, row): the tokens, up to 4,096 at a time, are loaded
//      into registers (16 bytes a lane where rows are aligned for it), the workgroup's best (value, id) is found,
//      then the sum of exp((l - maximum) / T); one record per chunk.
//   2. sample_pick_kernel, one workgroup per row: joins the chunk records (row maximum, argmax),
//      rescales the chunk sums to the row maximum, finds the chunk that holds the target by a
//      wavefront prefix scan and reads that one chunk again, 64 neighbouring tokens a load: the 64 that
//      hold the target are found by their sums, the token by a prefix scan over the lanes.  The chosen
//      token is also marked in the request's mask row when there is one.
//
// 64 rows of 128,256 logits (33 MB), half of them at a temperature: both kernels 14 us in a graph.  With 128 workgroups
// a row whose threads took four tokens each, one by one, and a single wavefront that walked its spans of the chunk: 30.
#include "common.h"
#include <math.h>

#define SAMPLE_THREADS 256
#define SCAN_TOKENS 4096         // tokens a workgroup holds in registers at a time
#define SAMPLE_MAX_CHUNKS 1024
#define KVA_NO_TOKEN (-1)       // what a row gets whose logits name no token

namespace {

struct Best {
    float value;
    int index;
};

// the larger value; the lower index among equal values
__device__ inline Best better(Best a, Best b) {
    return (b.value > a.value || (b.value == a.value && b.index < a.index)) ? b : a;
}

__device__ inline Best wave_best(Best x) {
#pragma unroll
    for (int off = KVA_WAVE / 2; off > 0; off >>= 1) {
        Best o;
        o.value = __shfl_xor(x.value, off, KVA_WAVE);
        o.index = __shfl_xor(x.index, off, KVA_WAVE);
        x = better(x, o);
    }
    return x;
}

// Inclusive prefix sum over the 64 lanes, lane order (six shift-and-add steps in the vector ALU).
__device__ inline float wave_prefix_sum(float v) {
    const int lane = threadIdx.x % KVA_WAVE;
#pragma unroll
    for (int off = 1; off < KVA_WAVE; off <<= 1) {
        const float below = __shfl_up(v, off, KVA_WAVE);
        if (lane >= off) v += below;
    }
    return v;
}

// Index of the lowest lane whose flag is set, or -1.
__device__ inline int first_lane(bool flag) {
    const unsigned long long votes = __ballot(flag);
    return votes == 0 ? -1 : __ffsll((long long)votes) - 1;
}

__device__ inline float penalised(float l, const unsigned char *mask, int token, float penalty) {
    if (mask != nullptr && mask[token] != 0) return l > 0.f ? l / penalty : l * penalty;
    return l;
}

__device__ inline const unsigned char *mask_row(const unsigned char *penalty_mask, const int *row_seat,
                                                int row, int vocab) {
    if (penalty_mask == nullptr || row_seat == nullptr) return nullptr;
    const int seat = row_seat[row];
    return seat < 0 ? nullptr : penalty_mask + (size_t)seat * vocab;
}

// exp((l - top) / T); a logit that is -inf or NaN weighs nothing
__device__ inline float token_weight(float l, float top, float inv_t) {
    return l > -INFINITY ? expf((l - top) * inv_t) : 0.f;
}

// Running softmax denominator: sum of exp((l - m) * inv_t) over what has been added, m their maximum.
struct Online {
    float m, s;
    __device__ inline void join(Online o, float inv_t) {
        if (o.m == -INFINITY) return;
        if (m == -INFINITY) {
            *this = o;
            return;
        }
        const float top = fmaxf(m, o.m);
        s = s * expf((m - top) * inv_t) + o.s * expf((o.m - top) * inv_t);
        m = top;
    }
};

} // namespace

__host__ __device__ inline float counter_uniform(unsigned int seed, unsigned int key, unsigned int step) {
    unsigned long long z = ((unsigned long long)key << 32) ^ (unsigned long long)step;
    z ^= (unsigned long long)seed * 0x9E3779B97F4A7C15ULL;
    z += 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    z = z ^ (z >> 31);
    return (float)(z >> 40) * (1.0f / 16777216.0f);
}

// One record per (row, chunk): the chunk's best (value, id), and for temperature rows the chunk's
// maximum and its sum of exp((l - maximum) / T).
struct ChunkRecord {
    float best_value;
    int best_index;
    float top;
    float sum;
};

// grid (chunks, rows).  VEC: rows and chunks start at multiples of 16 bytes.
template <bool VEC>
__global__ void __launch_bounds__(SAMPLE_THREADS)
sample_scan_kernel(const float *__restrict__ logits, int vocab, int chunk_tokens,
                   const unsigned char *__restrict__ penalty_mask, const int *__restrict__ row_seat,
                   float penalty, const float *__restrict__ inv_temperature,
                   ChunkRecord *__restrict__ records) {
    constexpr int WAVES = SAMPLE_THREADS / KVA_WAVE;
    __shared__ Best wave_b[2][WAVES];
    __shared__ float wave_s[2][WAVES];
    const int row = blockIdx.y, chunk = blockIdx.x, chunks = gridDim.x;
    const int lane = threadIdx.x % KVA_WAVE, wave = threadIdx.x / KVA_WAVE;
    const int begin = chunk * chunk_tokens;
    const int end = min(begin + chunk_tokens, vocab);
    const float *rl = logits + (size_t)row * vocab;
    const unsigned char *mk = mask_row(penalty_mask, row_seat, row, vocab);
    const float inv_t = inv_temperature != nullptr ? inv_temperature[row] : 0.f;
    const bool sampled = inv_t > 0.f;
    Best b{-INFINITY, vocab};
    Online o{-INFINITY, 0.f};
    for (int base = begin, turn = 0; base < end; base += SCAN_TOKENS, turn ^= 1) {
        // thread t's tokens: 4 t .. 4 t + 3 of every 1,024 (their loads side by side); past the end: -inf, no weight
        float l[SCAN_TOKENS / SAMPLE_THREADS];
#pragma unroll
        for (int j = 0; j < SCAN_TOKENS / SAMPLE_THREADS; j += 4) {
            const int t = base + j * SAMPLE_THREADS + 4 * threadIdx.x;
            if (VEC) {
                const float4 v = t < end ? *reinterpret_cast<const float4 *>(rl + t) : make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
                l[j] = v.x; l[j + 1] = v.y; l[j + 2] = v.z; l[j + 3] = v.w;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) l[j + i] = t + i < end ? rl[t + i] : -INFINITY;
            }
        }
        Best mine{-INFINITY, vocab};
#pragma unroll
        for (int j = 0; j < SCAN_TOKENS / SAMPLE_THREADS; ++j) {
            const int t = base + j / 4 * 4 * SAMPLE_THREADS + 4 * threadIdx.x + j % 4;
            if (mk != nullptr && t < end) l[j] = penalised(l[j], mk, t, penalty);
            if (l[j] > mine.value) mine = Best{l[j], t};        // (a thread's tokens come in ascending order: the first of equal ones)
        }
        mine = wave_best(mine);
        if (lane == 0) wave_b[turn][wave] = mine;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < WAVES; ++w) mine = better(mine, wave_b[turn][w]);
        b = better(b, mine);
        if (!sampled) continue;                                 // (the row's: the whole workgroup)
        float s = 0.f;
        if (mine.value > -INFINITY)
#pragma unroll
            for (int j = 0; j < SCAN_TOKENS / SAMPLE_THREADS; ++j) s += token_weight(l[j], mine.value, inv_t);
        s = wave_sum_valu(s);
        if (lane == 0) wave_s[turn][wave] = s;
        __syncthreads();
        s = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) s += wave_s[turn][w];
        o.join(Online{mine.value, s}, inv_t);
    }
    if (threadIdx.x == 0) records[(size_t)row * chunks + chunk] = ChunkRecord{b.value, b.index, o.m, o.s};
}

// grid (rows).  Every wavefront joins the records by itself (they agree); the chunk's tokens are shared out.
__global__ void __launch_bounds__(SAMPLE_THREADS)
sample_pick_kernel(const float *__restrict__ logits, int vocab, int chunk_tokens, int chunks,
                   const unsigned char *penalty_mask, const int *__restrict__ row_seat,
                   float penalty, const float *__restrict__ inv_temperature,
                   const ChunkRecord *__restrict__ records, unsigned int seed,
                   const unsigned int *__restrict__ rng_key, const unsigned int *__restrict__ rng_step,
                   unsigned char *mark_mask /* may be penalty_mask */, const int *__restrict__ mark_seat,
                   int *__restrict__ out_tokens, int *__restrict__ host_tokens) {
    constexpr int WAVES = SAMPLE_THREADS / KVA_WAVE, GROUPS = SCAN_TOKENS / SAMPLE_THREADS;
    __shared__ float wave_s[2][WAVES];
    __shared__ int found_by[2][WAVES];
    const int row = blockIdx.x, lane = threadIdx.x % KVA_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KVA_WAVE);
    const ChunkRecord *rec = records + (size_t)row * chunks;
    // this lane's chunks: a contiguous run, so that lane order is chunk order
    const int per_lane = (chunks + KVA_WAVE - 1) / KVA_WAVE;
    const int c0 = lane * per_lane, c1 = min(c0 + per_lane, chunks);
    Best b{-INFINITY, vocab};
    for (int c = c0; c < c1; ++c) b = better(b, Best{rec[c].best_value, rec[c].best_index});
    b = wave_best(b);
    int token = b.index;                    // the greedy choice; the row maximum is b.value
    bool bad_row = !(b.value > -INFINITY);  // NaN compares false too
    const float inv_t = inv_temperature != nullptr ? inv_temperature[row] : 0.f;
    if (inv_t > 0.f && !bad_row) {
        const float top = b.value;
        // chunk sums brought to the row maximum, summed per lane, scanned over the lanes
        auto weight = [&](int c) { return rec[c].sum > 0.f ? rec[c].sum * expf((rec[c].top - top) * inv_t) : 0.f; };
        float mine = 0.f;
        for (int c = c0; c < c1; ++c) mine += weight(c);
        const float upto = wave_prefix_sum(mine);
        const float total = __shfl(upto, KVA_WAVE - 1, KVA_WAVE);
        bad_row = !(total > 0.f) || total == INFINITY;
        const float target = counter_uniform(seed, rng_key[row], rng_step[row]) * total;
        // the first lane whose chunks reach past the target holds the chunk
        const int owner = first_lane(target < upto);
        int chunk = -1;
        float before = 0.f;
        if (lane == owner) {
            float run = upto - mine, last_before = run;
            int last_chunk = c0;
            for (int c = c0; c < c1 && chunk < 0; ++c) {
                const float w = weight(c);
                if (target < run + w) {
                    chunk = c;
                    before = run;
                } else {
                    last_before = run;
                    last_chunk = c;
                    run += w;
                }
            }
            if (chunk < 0) {                 // rounding between the lane's own sum and the scan's
                chunk = last_chunk;
                before = last_before;
            }
        }
        if (owner < 0) {
            // the target landed on the total through rounding: the last token of the last chunk
            // that weighs anything (before = -inf puts the target past every span below)
            int last = -1;
            for (int c = c0; c < c1; ++c)
                if (weight(c) > 0.f) last = c;
#pragma unroll
            for (int off = KVA_WAVE / 2; off > 0; off >>= 1) last = max(last, __shfl_xor(last, off, KVA_WAVE));
            chunk = last < 0 ? chunks - 1 : last;
            before = -INFINITY;
        } else {
            chunk = __shfl(chunk, owner, KVA_WAVE);
            before = __shfl(before, owner, KVA_WAVE);
        }
        // inside the chunk, 4,096 tokens at a time, a quarter a wavefront, lane = token: of 64 neighbouring tokens the
        // sum first, the place inside only where the target is
        const int begin = chunk * chunk_tokens, end = min(begin + chunk_tokens, vocab);
        const float *rl = logits + (size_t)row * vocab;
        const unsigned char *mk = mask_row(penalty_mask, row_seat, row, vocab);
        float inner = target - before;
        token = end - 1;                     // past every reach (rounding): the chunk's last token
        for (int base = begin, turn = 0; base < end; base += SCAN_TOKENS, turn ^= 1) {
            float w[GROUPS];
            const int first = base + wave * (SCAN_TOKENS / WAVES) + lane;
#pragma unroll
            for (int i = 0; i < GROUPS; ++i) w[i] = first + KVA_WAVE * i < end ? rl[first + KVA_WAVE * i] : -INFINITY;
            float all = 0.f;
#pragma unroll
            for (int i = 0; i < GROUPS; ++i) {
                if (mk != nullptr && first + KVA_WAVE * i < end) w[i] = penalised(w[i], mk, first + KVA_WAVE * i, penalty);
                w[i] = token_weight(w[i], top, inv_t);
            }
            float sums[GROUPS];
#pragma unroll
            for (int i = 0; i < GROUPS; ++i) {
                sums[i] = wave_sum_valu(w[i]);
                all += sums[i];
            }
            if (lane == 0) wave_s[turn][wave] = all;
            __syncthreads();
            float here = inner;
            for (int v = 0; v < wave; ++v) here -= wave_s[turn][v];
            int found = -1;
            if (here < all && (wave == 0 || here >= 0.f)) {       // (an earlier wavefront's share holds it: negative)
                float run = 0.f;
                bool done = false;
#pragma unroll
                for (int i = 0; i < GROUPS; ++i) {
                    if (!done && here < run + sums[i]) {
                        const float reach = run + wave_prefix_sum(w[i]);
                        const int at = first_lane(here < reach);
                        // (rounding between the sum and the scan: the last of the 64 that weighs anything)
                        const unsigned long long weighs = __ballot(w[i] > 0.f);
                        found = first - lane + KVA_WAVE * i + (at >= 0 ? at : weighs ? 63 - __clzll((long long)weighs) : 0);
                        done = true;
                    }
                    run += sums[i];
                }
            }
            if (lane == 0) found_by[turn][wave] = found;
            __syncthreads();
            int hit = -1;
#pragma unroll
            for (int v = WAVES - 1; v >= 0; --v) hit = found_by[turn][v] >= 0 ? found_by[turn][v] : hit;
            if (hit >= 0) {
                token = hit;
                break;
            }
#pragma unroll
            for (int v = 0; v < WAVES; ++v) inner -= wave_s[turn][v];
        }
    }
    if (wave != 0) return;
    // A row without a finite best logit (all NaN, all -inf) has no token to name, greedy or sampled,
    // and neither has a temperature row whose weights do not add up to a positive finite total.
    // Such a row gets KVA_NO_TOKEN (-1): the host sees it and ends the request with an error, and
    // the next step's lookup of this buffer on the device, which may already be queued, takes
    // token 0 for any negative value it finds (a row past the table's end would be a memory fault).
    if (bad_row || token < 0 || token >= vocab) token = KVA_NO_TOKEN;
    if (lane == 0) {
        out_tokens[row] = token;
        if (host_tokens != nullptr) host_tokens[row] = token;      // pinned host memory, mapped for the device
        if (mark_mask != nullptr && mark_seat != nullptr) {
            const int seat = mark_seat[row];
            if (seat >= 0 && token >= 0 && token < vocab) mark_mask[(size_t)seat * vocab + token] = 1;
        }
    }
}

// workspace: one record per (row, chunk)
extern "C" long long kva_sample_workspace_bytes(int rows, int chunks) {
    return (long long)rows * chunks * (long long)sizeof(ChunkRecord);
}

// out_tokens[row] = the sampled (inv_temperature[row] > 0) or the best token of logits[row, :].
// penalty_mask [seats, vocab] with row_seat[row] (-1: none) says which logits are penalised;
// mark_mask / mark_seat (may be the same mask, -1: none) get the chosen token marked afterwards.
// Whether a kernel may write to this host memory: pinned and mapped for the current device.
extern "C" int kva_host_memory_is_mapped(void *host) {
    void *dev = nullptr;
    if (host == nullptr || hipHostGetDevicePointer(&dev, host, 0) != hipSuccess) {
        (void)hipGetLastError();                                    // the query's failure is an answer, not an error to keep
        return 0;
    }
    return dev != nullptr ? 1 : 0;
}

// Queues a copy from pinned host memory.
extern "C" int kva_upload(void *device, const void *host, long long bytes, hipStream_t stream) {
    KVA_REQUIRE(device && host && bytes >= 0, "upload: missing operand");
    const hipError_t e = hipMemcpyAsync(device, host, (size_t)bytes, hipMemcpyHostToDevice, stream);
    KVA_REQUIRE(e == hipSuccess, "upload: %s", hipGetErrorString(e));
    return KVA_OK;
}

// host_tokens (optional): pinned host memory (hipHostMalloc, torch's pin_memory) with room for a token
// per row; the kernel that chooses the tokens writes them there as well, which saves the copy
// that would otherwise follow it on the stream.  Refused unless the runtime says the memory is
// mapped for the device.
extern "C" int kva_sample(int *out_tokens, const float *logits, int rows, int vocab, int chunks,
                          const unsigned char *penalty_mask, const int *row_seat, float penalty,
                          const float *inv_temperature, unsigned int seed,
                          const unsigned int *rng_key, const unsigned int *rng_step, int any_sampled,
                          void *workspace, unsigned char *mark_mask, const int *mark_seat,
                          int *host_tokens, hipStream_t stream) {
    int *host_mapped = nullptr;
    if (host_tokens != nullptr) {
        void *dev = nullptr;
        const hipError_t e = hipHostGetDevicePointer(&dev, host_tokens, 0);
        KVA_REQUIRE(e == hipSuccess && dev != nullptr, "sample: host_tokens is not pinned host memory mapped for the device (%s)",
                    hipGetErrorString(e));
        host_mapped = (int *)dev;
    }
    KVA_REQUIRE(rows >= 0 && vocab > 0, "sample: bad sizes rows=%d vocab=%d", rows, vocab);
    KVA_REQUIRE(chunks >= 1 && chunks <= SAMPLE_MAX_CHUNKS, "sample: chunk count %d is not in 1..%d", chunks,
                SAMPLE_MAX_CHUNKS);
    KVA_REQUIRE(rows <= 65535, "sample: at most 65535 rows per call");
    KVA_REQUIRE(penalty > 0.f, "sample: repetition penalty must be positive");
    KVA_REQUIRE(!any_sampled || (inv_temperature && rng_key && rng_step),
                "sample: temperature rows need inv_temperature, rng_key and rng_step");
    KVA_REQUIRE(workspace != nullptr || rows == 0, "sample: a workspace of kva_sample_workspace_bytes is needed");
    if (rows == 0) return KVA_OK;
    // chunks start at multiples of four tokens (the last ones may be empty)
    const int chunk_tokens = ((vocab + chunks - 1) / chunks + 3) / 4 * 4;
    const bool vec = vocab % 4 == 0 && (uintptr_t)logits % 16 == 0;
    ChunkRecord *records = (ChunkRecord *)workspace;
    const float *inv_t = any_sampled ? inv_temperature : nullptr;
    hipLaunchKernelGGL(vec ? sample_scan_kernel<true> : sample_scan_kernel<false>, dim3(chunks, rows), dim3(SAMPLE_THREADS), 0, stream, logits,
                       vocab, chunk_tokens, penalty_mask, row_seat, penalty, inv_t, records);
    hipLaunchKernelGGL(sample_pick_kernel, dim3(rows), dim3(SAMPLE_THREADS), 0, stream, logits, vocab,
                       chunk_tokens, chunks, penalty_mask, row_seat, penalty, inv_t, records, seed, rng_key,
                       rng_step, mark_mask, mark_seat, out_tokens, host_mapped);
    KVA_CHECK_LAUNCH("sample");
    return KVA_OK;
}

// mask[seat[i]][token[i]] = 1
__global__ void mark_tokens_kernel(unsigned char *__restrict__ mask, const int *__restrict__ seats,
                                   const int *__restrict__ tokens, int n, int vocab) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int seat = seats[i], tok = tokens[i];
    if (seat >= 0 && tok >= 0 && tok < vocab) mask[(size_t)seat * vocab + tok] = 1;
}

extern "C" int kva_mark_tokens(unsigned char *mask, const int *seats, const int *tokens, int n,
                               int vocab, hipStream_t stream) {
    KVA_REQUIRE(n >= 0 && vocab > 0, "mark_tokens: bad sizes");
    if (n == 0) return KVA_OK;
    hipLaunchKernelGGL(mark_tokens_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, mask, seats,
                       tokens, n, vocab);
    KVA_CHECK_LAUNCH("mark_tokens");
    return KVA_OK;
}
