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
//   1. sample_scan_kernel, one wavefront per (chunk of a row, row): the tokens, up to 1,280 at a time, are loaded
//      into registers, the best (value, id) is found, then the sum of exp((l - maximum) / T); one record per chunk.
//   2. sample_pick_kernel, one wavefront per row: joins the chunk records (row maximum, argmax),
//      rescales the chunk sums to the row maximum, finds the chunk that holds the target by a
//      wavefront prefix scan and reads that one chunk again, 64 neighbouring tokens a load: the 64 that
//      hold the target are found by their sums, the token by a prefix scan over the lanes.  The chosen
//      token is also marked in the request's mask row when there is one.
// The order of all sums follows from the vocabulary and the number of chunks alone: a row draws the same token alone
// and among others.
//
// Both kernels in a graph (rows' arguments in arrays), 128 chunks of a row of 128,256 logits, us, greedy / at a temperature: 1 row 5.5 / 10.9, 16 rows 6.5 /
// 12.4, 64 rows (33 MB) 8.6 / 17.3, 128 rows 14.8 / 24.0.  With 128 workgroups a row whose threads took four tokens each, one by
// one, and a single wavefront that walked its spans of the chunk: 64 rows 13.8 / 35.2.
#include "common.h"
#include <string.h>
#include <math.h>

#define SCAN_WAVES 4             // chunks a workgroup of the first kernel takes, a wavefront each, where there are enough
// Tokens a lane holds in registers at a time: chunks of up to 256 tokens (a small vocabulary's) and others, 1,280 a turn.
#define HELD_FEW 4
#define HELD_MANY 20
#define SAMPLE_MAX_CHUNKS 1024
#define SAMPLE_ROWS_BY_VALUE 128     // (2.6 KB of the 4 KB that a launch's arguments may take)
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

// The best of the 64 lanes, all of them get it: the largest value, then the lowest index among the lanes that have it (no
// lane's value is a NaN), each a chain of steps in the vector ALU where twelve shuffles would be as many trips through LDS.
__device__ inline Best wave_best(Best x) {
    float v = x.value;
    v = fmaxf(v, row16_rotated<8>(v));
    v = fmaxf(v, row16_rotated<4>(v));
    v = fmaxf(v, row16_rotated<2>(v));
    v = fmaxf(v, row16_rotated<1>(v));
    v = quad_rows_max(v);
    unsigned at = x.value == v ? (unsigned)x.index : 0x7fffffffu;
#define SAMPLE_ROTATED(n) __builtin_amdgcn_update_dpp(0u, at, 0x120 | n, 0xf, 0xf, false)
    at = min(at, SAMPLE_ROTATED(8));
    at = min(at, SAMPLE_ROTATED(4));
    at = min(at, SAMPLE_ROTATED(2));
    at = min(at, SAMPLE_ROTATED(1));
#undef SAMPLE_ROTATED
    auto a = __builtin_amdgcn_permlane16_swap(at, at, false, false);
    at = min(a[0], a[1]);
    auto b = __builtin_amdgcn_permlane32_swap(at, at, false, false);
    return Best{v, (int)min(b[0], b[1])};
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

// What a row is asked for: arrays on the device, or numbers in the launch itself (a few rows: no copy in front of the
// kernels, and a row's numbers are scalar loads of the launch's arguments).  A scan takes the first two of the arrays.
struct RowPointers {
    const float *inv_t;                 // absent: all rows are greedy
    const int *seat;                    // absent: no row is penalised
    const unsigned int *key, *step;
    const int *mark;                    // absent: nothing is marked
    __device__ inline float inverse_temperature(int row) const { return inv_t != nullptr ? inv_t[row] : 0.f; }
    __device__ inline int penalty_seat(int row) const { return seat != nullptr ? seat[row] : -1; }
    __device__ inline unsigned int rng_key(int row) const { return key[row]; }
    __device__ inline unsigned int rng_step(int row) const { return step[row]; }
    __device__ inline int mark_seat(int row) const { return mark != nullptr ? mark[row] : -1; }
};
template <int ARRAYS>
struct RowValues {
    bool sampled, penalised, marked;
    int v[ARRAYS][SAMPLE_ROWS_BY_VALUE];    // 1 / temperature, seat of the penalty, key, step, seat to mark
    __device__ inline float inverse_temperature(int row) const { return sampled ? __int_as_float(v[0][row]) : 0.f; }
    __device__ inline int penalty_seat(int row) const { return penalised ? v[1][row] : -1; }
    __device__ inline unsigned int rng_key(int row) const { return v[ARRAYS > 2 ? 2 : 0][row]; }
    __device__ inline unsigned int rng_step(int row) const { return v[ARRAYS > 2 ? 3 : 0][row]; }
    __device__ inline int mark_seat(int row) const { return marked ? v[ARRAYS > 2 ? 4 : 0][row] : -1; }
};

template <typename ROWS>
__device__ inline const unsigned char *mask_row(const unsigned char *penalty_mask, const ROWS &rows, int row, int vocab) {
    if (penalty_mask == nullptr) return nullptr;
    const int seat = rows.penalty_seat(row);
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

typedef float sample_f32x4 __attribute__((ext_vector_type(4), aligned(4)));     // (rows may start at any multiple of 4 bytes)

// grid (chunks / wavefronts of a workgroup, rows).  VEC: rows and chunks start at, and end before, multiples of 16 bytes.
template <int HELD, bool VEC, typename ROWS>
__global__ void __launch_bounds__(KVA_WAVE * SCAN_WAVES)
sample_scan_kernel(const float *__restrict__ logits, int vocab, int chunk_tokens, int chunks,
                   const unsigned char *__restrict__ penalty_mask, float penalty, ROWS rows, ChunkRecord *__restrict__ records) {
    const int row = blockIdx.y, lane = threadIdx.x % KVA_WAVE;
    const int chunk = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x / KVA_WAVE) + threadIdx.x / KVA_WAVE);
    if (chunk >= chunks) return;
    const int begin = chunk * chunk_tokens;
    const int end = min(begin + chunk_tokens, vocab);
    const float *rl = logits + (size_t)row * vocab;
    const unsigned char *mk = mask_row(penalty_mask, rows, row, vocab);
    const float inv_t = rows.inverse_temperature(row);
    const bool sampled = inv_t > 0.f;
    Best b{-INFINITY, vocab};
    Online o{-INFINITY, 0.f};
    for (int base = begin; base < end; base += HELD * KVA_WAVE) {
        // lane t's tokens: 4 t .. 4 t + 3 of every 256 (their loads side by side); past the end: -inf, no weight
        float l[HELD];
#pragma unroll
        for (int j = 0; j < HELD; j += 4) {
            const int t = base + j * KVA_WAVE + 4 * lane;
            if (VEC) {
                const float4 v = t < end ? *reinterpret_cast<const float4 *>(rl + t) : make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
                l[j] = v.x; l[j + 1] = v.y; l[j + 2] = v.z; l[j + 3] = v.w;
            } else if (t + 3 < end) {
                const sample_f32x4 v = *reinterpret_cast<const sample_f32x4 *>(rl + t);
                l[j] = v.x; l[j + 1] = v.y; l[j + 2] = v.z; l[j + 3] = v.w;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) l[j + i] = t + i < end ? rl[t + i] : -INFINITY;
            }
        }
        Best mine{-INFINITY, vocab};
#pragma unroll
        for (int j = 0; j < HELD; ++j) {
            const int t = base + j / 4 * 4 * KVA_WAVE + 4 * lane + j % 4;
            if (mk != nullptr && t < end) l[j] = penalised(l[j], mk, t, penalty);
            if (l[j] > mine.value) mine = Best{l[j], t};        // (a lane's tokens come in ascending order: the first of equal ones)
        }
        mine = wave_best(mine);
        b = better(b, mine);
        if (!sampled || !(mine.value > -INFINITY)) continue;    // (the row's; the same in all lanes)
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < HELD; ++j) s += token_weight(l[j], mine.value, inv_t);
        o.join(Online{mine.value, wave_sum_valu(s)}, inv_t);
    }
    if (lane == 0) records[(size_t)row * chunks + chunk] = ChunkRecord{b.value, b.index, o.m, o.s};
}

// grid (rows), one wavefront
template <int HELD, typename ROWS>
__global__ void __launch_bounds__(KVA_WAVE)
sample_pick_kernel(const float *__restrict__ logits, int vocab, int chunk_tokens, int chunks,
                   const unsigned char *penalty_mask, float penalty, ROWS rows,
                   const ChunkRecord *__restrict__ records, unsigned int seed, unsigned char *mark_mask /* may be penalty_mask */,
                   int *__restrict__ out_tokens, int *__restrict__ host_tokens) {
    const int row = blockIdx.x, lane = threadIdx.x;
    const ChunkRecord *rec = records + (size_t)row * chunks;
    // this lane's chunks: a contiguous run, so that lane order is chunk order
    const int per_lane = (chunks + KVA_WAVE - 1) / KVA_WAVE;
    const int c0 = lane * per_lane, c1 = min(c0 + per_lane, chunks);
    Best b{-INFINITY, vocab};
    for (int c = c0; c < c1; ++c) b = better(b, Best{rec[c].best_value, rec[c].best_index});
    b = wave_best(b);
    int token = b.index;                    // the greedy choice; the row maximum is b.value
    bool bad_row = !(b.value > -INFINITY);  // NaN compares false too
    const float inv_t = rows.inverse_temperature(row);
    if (inv_t > 0.f && !bad_row) {
        const float top = b.value;
        // chunk sums brought to the row maximum, summed per lane, scanned over the lanes
        auto weight = [&](int c) { return rec[c].sum > 0.f ? rec[c].sum * expf((rec[c].top - top) * inv_t) : 0.f; };
        float mine = 0.f;
        for (int c = c0; c < c1; ++c) mine += weight(c);
        const float upto = wave_prefix_sum(mine);
        const float total = __shfl(upto, KVA_WAVE - 1, KVA_WAVE);
        bad_row = !(total > 0.f) || total == INFINITY;
        const float target = counter_uniform(seed, rows.rng_key(row), rows.rng_step(row)) * total;
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
        // inside the chunk, 1,280 tokens at a time, lane = token: of 64 neighbouring tokens the sum first, the place
        // inside only where the target is
        const int begin = chunk * chunk_tokens, end = min(begin + chunk_tokens, vocab);
        const float *rl = logits + (size_t)row * vocab;
        const unsigned char *mk = mask_row(penalty_mask, rows, row, vocab);
        float inner = target - before;
        token = end - 1;                     // past every reach (rounding): the chunk's last token
        bool done = false;
        for (int base = begin; base < end && !done; base += HELD * KVA_WAVE) {
            float w[HELD], sums[HELD];
            const int first = base + lane;
#pragma unroll
            for (int i = 0; i < HELD; ++i) w[i] = first + KVA_WAVE * i < end ? rl[first + KVA_WAVE * i] : -INFINITY;
#pragma unroll
            for (int i = 0; i < HELD; ++i) {
                if (mk != nullptr && first + KVA_WAVE * i < end) w[i] = penalised(w[i], mk, first + KVA_WAVE * i, penalty);
                w[i] = token_weight(w[i], top, inv_t);
            }
#pragma unroll
            for (int i = 0; i < HELD; ++i) sums[i] = wave_sum_valu(w[i]);
            float run = 0.f;
#pragma unroll
            for (int i = 0; i < HELD; ++i) {
                if (!done && inner < run + sums[i]) {
                    const int at = first_lane(inner < run + wave_prefix_sum(w[i]));
                    // (rounding between the sum and the scan: the last of the 64 that weighs anything)
                    const unsigned long long weighs = __ballot(w[i] > 0.f);
                    token = base + KVA_WAVE * i + (at >= 0 ? at : weighs ? 63 - __clzll((long long)weighs) : 0);
                    done = true;
                }
                run += sums[i];
            }
            inner -= run;
        }
    }
    // A row without a finite best logit (all NaN, all -inf) has no token to name, greedy or sampled,
    // and neither has a temperature row whose weights do not add up to a positive finite total.
    // Such a row gets KVA_NO_TOKEN (-1): the host sees it and ends the request with an error, and
    // the next step's lookup of this buffer on the device, which may already be queued, takes
    // token 0 for any negative value it finds (a row past the table's end would be a memory fault).
    if (bad_row || token < 0 || token >= vocab) token = KVA_NO_TOKEN;
    if (lane == 0) {
        out_tokens[row] = token;
        if (host_tokens != nullptr) host_tokens[row] = token;      // pinned host memory, mapped for the device
        if (mark_mask != nullptr) {
            const int seat = rows.mark_seat(row);
            if (seat >= 0 && token >= 0 && token < vocab) mark_mask[(size_t)seat * vocab + token] = 1;
        }
    }
}

// An event of its own kind: what is recorded here costs a call into the runtime (1.5 us of host time where torch's event takes 4.5).
extern "C" int kva_event_create(void **event) {
    hipEvent_t e = nullptr;
    const hipError_t rc = hipEventCreateWithFlags(&e, hipEventDisableTiming);
    if (rc != hipSuccess) (void)hipGetLastError();
    KVA_REQUIRE(rc == hipSuccess, "event: not created: %s", hipGetErrorString(rc));
    *event = e;
    return KVA_OK;
}
extern "C" int kva_event_record(hipEvent_t event, hipStream_t stream) {
    const hipError_t rc = hipEventRecord(event, stream);
    if (rc != hipSuccess) (void)hipGetLastError();
    KVA_REQUIRE(rc == hipSuccess, "event: not recorded: %s", hipGetErrorString(rc));
    return KVA_OK;
}
// Waits for what was recorded last (nothing: returns at once).
extern "C" int kva_event_synchronize(hipEvent_t event) {
    const hipError_t rc = hipEventSynchronize(event);
    if (rc != hipSuccess) (void)hipGetLastError();
    KVA_REQUIRE(rc == hipSuccess, "event: waiting failed: %s", hipGetErrorString(rc));
    return KVA_OK;
}
extern "C" void kva_event_destroy(hipEvent_t event) { (void)hipEventDestroy(event); }

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

static int sample_check(int *host_tokens, int **host_mapped, int rows, int vocab, int chunks, float penalty, const void *workspace) {
    *host_mapped = nullptr;
    if (host_tokens != nullptr) {
        void *dev = nullptr;
        const hipError_t e = hipHostGetDevicePointer(&dev, host_tokens, 0);
        if (e != hipSuccess) (void)hipGetLastError();               // (told below, and to no later launch)
        KVA_REQUIRE(e == hipSuccess && dev != nullptr, "sample: host_tokens is not pinned host memory mapped for the device (%s)",
                    hipGetErrorString(e));
        *host_mapped = (int *)dev;
    }
    KVA_REQUIRE(rows >= 0 && vocab > 0, "sample: bad sizes rows=%d vocab=%d", rows, vocab);
    KVA_REQUIRE(chunks >= 1 && chunks <= SAMPLE_MAX_CHUNKS, "sample: chunk count %d is not in 1..%d", chunks,
                SAMPLE_MAX_CHUNKS);
    KVA_REQUIRE(rows <= 65535, "sample: at most 65535 rows per call");
    KVA_REQUIRE(penalty > 0.f, "sample: repetition penalty must be positive");
    KVA_REQUIRE(workspace != nullptr || rows == 0, "sample: a workspace of kva_sample_workspace_bytes is needed");
    return KVA_OK;
}

template <typename SCAN_ROWS, typename ROWS>
static int sample_launch(int *out_tokens, const float *logits, int rows, int vocab, int chunks, const unsigned char *penalty_mask,
                         float penalty, const SCAN_ROWS &first, const ROWS &second, unsigned int seed, void *workspace,
                         unsigned char *mark_mask, int *host_mapped, hipStream_t stream) {
    // chunks start at multiples of four tokens (the last ones may be empty)
    const int chunk_tokens = ((vocab + chunks - 1) / chunks + 3) / 4 * 4;
    ChunkRecord *records = (ChunkRecord *)workspace;
    const int waves = (long long)rows * chunks >= 2048 ? SCAN_WAVES : 1;      // (fewer: a compute unit each)
    const dim3 grid((chunks + waves - 1) / waves, rows), block(KVA_WAVE * waves);
    const bool few = chunk_tokens <= HELD_FEW * KVA_WAVE;
    const bool vec = vocab % 4 == 0 && (uintptr_t)logits % 16 == 0;
    const auto scan = few ? (vec ? sample_scan_kernel<HELD_FEW, true, SCAN_ROWS> : sample_scan_kernel<HELD_FEW, false, SCAN_ROWS>)
                          : (vec ? sample_scan_kernel<HELD_MANY, true, SCAN_ROWS> : sample_scan_kernel<HELD_MANY, false, SCAN_ROWS>);
    const auto pick = few ? sample_pick_kernel<HELD_FEW, ROWS> : sample_pick_kernel<HELD_MANY, ROWS>;
    hipLaunchKernelGGL(scan, grid, block, 0, stream, logits, vocab, chunk_tokens, chunks, penalty_mask, penalty, first, records);
    hipLaunchKernelGGL(pick, dim3(rows), dim3(KVA_WAVE), 0, stream, logits, vocab, chunk_tokens, chunks, penalty_mask, penalty, second,
                       records, seed, mark_mask, out_tokens, host_mapped);
    KVA_CHECK_LAUNCH("sample");
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
    if (int rc = sample_check(host_tokens, &host_mapped, rows, vocab, chunks, penalty, workspace)) return rc;
    KVA_REQUIRE(!any_sampled || (inv_temperature && rng_key && rng_step),
                "sample: temperature rows need inv_temperature, rng_key and rng_step");
    if (rows == 0) return KVA_OK;
    const RowPointers args{any_sampled ? inv_temperature : nullptr, row_seat, rng_key, rng_step, mark_seat};
    return sample_launch(out_tokens, logits, rows, vocab, chunks, penalty_mask, penalty, args, args, seed, workspace, mark_mask,
                         host_mapped, stream);
}

// The same for up to kva_sample_rows_by_value() rows whose arguments are on the host: `row_args` [5][stride] holds 1 / temperature
// (fp32), key, step, seat of the penalty and seat to mark, of which those are read that are used (any_sampled, penalty_mask,
// mark_mask).  They travel in the launches' arguments: read before this returns, and nothing to keep.  64 rows of
// 128,256, half of them at a temperature, us a call among others: 30 with a copy in front of the kernels (host 28), 18 here (host 17, kernels 15.5).
// `behind` (optional, of kva_event_create): recorded on the stream behind the kernels.
extern "C" int kva_sample_rows_by_value() { return SAMPLE_ROWS_BY_VALUE; }

extern "C" int kva_sample_by_value(int *out_tokens, const float *logits, int rows, int vocab, int chunks,
                                   const unsigned char *penalty_mask, float penalty, const int *row_args, int stride,
                                   unsigned int seed, int any_sampled, void *workspace, unsigned char *mark_mask, int *host_tokens,
                                   hipEvent_t behind, hipStream_t stream) {
    int *host_mapped = nullptr;
    if (int rc = sample_check(host_tokens, &host_mapped, rows, vocab, chunks, penalty, workspace)) return rc;
    KVA_REQUIRE(rows <= SAMPLE_ROWS_BY_VALUE && rows <= stride && (row_args || rows == 0),
                "sample: %d rows' arguments do not travel with the launch", rows);
    if (rows == 0) return KVA_OK;
    RowValues<2> first{any_sampled != 0, penalty_mask != nullptr, false, {}};
    RowValues<5> second{any_sampled != 0, penalty_mask != nullptr, mark_mask != nullptr, {}};
    const bool used[5] = {any_sampled != 0, penalty_mask != nullptr, any_sampled != 0, any_sampled != 0, mark_mask != nullptr};
    const int from[5] = {0, 3, 1, 2, 4};
    for (int i = 0; i < 5; ++i) {
        if (!used[i]) continue;
        memcpy(second.v[i], row_args + (size_t)from[i] * stride, sizeof(int) * rows);
        if (i < 2) memcpy(first.v[i], second.v[i], sizeof(int) * rows);
    }
    if (int rc = sample_launch(out_tokens, logits, rows, vocab, chunks, penalty_mask, penalty, first, second, seed, workspace, mark_mask,
                               host_mapped, stream))
        return rc;
    if (behind != nullptr) {
        const hipError_t e = hipEventRecord(behind, stream);
        if (e != hipSuccess) (void)hipGetLastError();
        KVA_REQUIRE(e == hipSuccess, "sample: the event behind the kernels was not recorded: %s", hipGetErrorString(e));
    }
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
