// A routed feed-forward (mixture of experts) whose work stays on the device from the router's
// logits to the weighted sum: no count of tokens per expert ever reaches the host, so the whole
// layer can be captured into a graph.
//
//  * kva_moe_route:  scores = softmax(logits) over all router outputs; the `top` largest of
//    scores + correction are chosen; their weights are the plain scores (optionally renormalised).
//    Or (`over_chosen`) the largest logits are chosen and the weights are the softmax over them alone.
//  * kva_moe_router: the router's product (bf16 operands), that choice and, for up to 16 tokens, the list below in one launch.
//  * kva_moe_align:  the (token, choice) slots of real experts sorted by expert into a list padded
//    so that every tile of 16 rows belongs to one expert (`sorted_slot`, -1 = padding), with the
//    expert of every tile (`tile_expert`, -1 = unused tile).  Without a router (`table`): the experts of a
//    token are the entries of its id's row in an integer table, all with one weight; the same launch looks
//    them up.
//  * kva_moe_expert_rows: one product per tile against its expert's matrix.  Mode 0 ("up"): rows of
//    x gathered by slot / top, activation applied (a gated expert: act(gate) * up, its gate and up rows
//    interleaved in one matrix), written at the sorted position.  Mode 1 ("down"):
//    rows at the sorted position, times the slot's routing weight, written at the slot (fp32).  The weight may
//    stand on the expert's input instead: it then multiplies the first product's rows, before the activation.
//    bf16 with K % 32 == 0 runs on the matrix cores (with many rows an expert through LDS, in groups of
//    tiles), everything else (fp32 too) on a plain tiled kernel that adds k ascending.
//  * kva_moe_combine: out[t] = sum over the token's choices of the slot's row, or, for a router
//    output past the real experts (an identity expert), weight * x[t].
//
// A row's result depends on that row and its expert's matrix only, never on which other rows
// share its tile: the same token gives the same numbers in any batch.
#include "common.h"
#include "attention_frag.h"
#include "lds_product.h"
#include <math.h>
#include <type_traits>

#define MOE_TILE 16
#define MOE_MAX_EXPERTS 1024
#define MOE_ROUTE_PER_LANE 8

__device__ inline float moe_activate(float z, int act) {
    if (act == 3) return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f));       // exact gelu
    if (act == 5) return kva_activate(z, KVA_ACT_RELU2);
    return kva_activate(z, act);
}

// ---- router ------------------------------------------------------------------------------
struct MoeRoute {
    const float *correction;
    int outputs, top, renormalise, over_chosen, sigmoid_scores, groups, keep_groups, group_top;
    float weight_scale, sum_eps;
};

// one token by one wavefront: `logits` [outputs] (memory or LDS) -> idx and wgt [top]; `choice` is the wavefront's own
// piece of LDS, KVA_WAVE * PL floats (16-byte aligned; with PL > 1 read with groups only).  A lane takes PL outputs.
// The choices are `top` different outputs whatever the scores hold (the few-token products rely on it): a score that is
// not a number counts as the largest, and of equal ones, -inf among them, the lowest index comes first.
template <int PL>
__device__ inline void moe_route_token(const MoeRoute &a, const float *logits, int *idx, float *wgt, float *choice) {
    const int lane = threadIdx.x % KVA_WAVE;
    float s[PL], ch[PL];
    float mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < PL; ++j) {
        const int e = lane + j * KVA_WAVE;
        s[j] = e < a.outputs ? logits[e] : -INFINITY;
        mx = fmaxf(mx, s[j]);
    }
    mx = wave_max(mx);
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < PL; ++j) {
        const int e = lane + j * KVA_WAVE;
        s[j] = e < a.outputs ? expf(s[j] - mx) : 0.f;
        sum += s[j];
    }
    sum = wave_sum(sum);
#pragma unroll
    for (int j = 0; j < PL; ++j) {
        const int e = lane + j * KVA_WAVE;
        if (a.over_chosen) {
            // the logits themselves are compared, and the weights are a softmax over the chosen ones
            // alone: exp(logit - max) here, divided by the chosen ones' sum below
            ch[j] = e < a.outputs ? logits[e] + (a.correction ? a.correction[e] : 0.f) : -INFINITY;
        } else {
            // scores: the softmax over all outputs, or every output's own sigmoid
            s[j] = a.sigmoid_scores ? (e < a.outputs ? 1.f / (1.f + expf(-logits[e])) : 0.f) : s[j] / sum;
            ch[j] = e < a.outputs ? s[j] + (a.correction ? a.correction[e] : 0.f) : -INFINITY;
        }
        if (ch[j] != ch[j]) ch[j] = INFINITY;
    }
    if (a.groups > 1) {
        // Outputs form `groups` equal runs of neighbours.  A group's score is the sum of its `group_top`
        // largest choice scores; only outputs of the `keep_groups` best groups (of equal ones the lowest
        // index) can be chosen: the others' choice scores become -inf.  Lane g takes group g.
        const int per = a.outputs / a.groups;
#pragma unroll
        for (int j = 0; j < PL; ++j)
            if (lane + j * KVA_WAVE < a.outputs) choice[lane + j * KVA_WAVE] = ch[j];
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
        float gs = -INFINITY;
        if (lane < a.groups) {
            gs = 0.f;
            unsigned long long taken = 0ull;            // (a group holds at most 64 outputs when it is scored this way; larger ones below)
            for (int k = 0; k < a.group_top && k < per; ++k) {
                float bv = -INFINITY;
                int bi = -1;
                for (int i = 0; i < per; ++i) {
                    const bool used = i < 64 ? ((taken >> i) & 1ull) != 0ull : false;
                    const float v = choice[lane * per + i];
                    if (!used && (bi < 0 || v > bv)) { bv = v; bi = i; }
                }
                if (bi >= 0 && bi < 64) taken |= 1ull << bi;
                gs += bv;
            }
        }
        unsigned long long allowed = 0ull;
        for (int k = 0; k < a.keep_groups; ++k) {
            float bv = gs;
            int bg = lane < a.groups && !((allowed >> lane) & 1ull) ? lane : 0x7fffffff;
            if (bg == 0x7fffffff) bv = -INFINITY;
#pragma unroll
            for (int off = KVA_WAVE / 2; off > 0; off >>= 1) {
                const float ov = __shfl_xor(bv, off, KVA_WAVE);
                const int og = __shfl_xor(bg, off, KVA_WAVE);
                if (og != 0x7fffffff && (bg == 0x7fffffff || ov > bv || (ov == bv && og < bg))) { bv = ov; bg = og; }
            }
            if (bg != 0x7fffffff) allowed |= 1ull << bg;
        }
#pragma unroll
        for (int j = 0; j < PL; ++j) {
            const int e = lane + j * KVA_WAVE;
            if (e < a.outputs && !((allowed >> (e / per)) & 1ull)) ch[j] = -INFINITY;
        }
    }
    if constexpr (PL == 1) {
        // every lane counts the outputs in front of its own (of equal ones the lowest index comes first)
        __builtin_amdgcn_wave_barrier();
        choice[lane] = ch[0];
        __threadfence_block();
        __builtin_amdgcn_wave_barrier();
        int rank = 0;
        for (int e = 0; e < a.outputs; e += 4) {
            const float4 c = *reinterpret_cast<const float4 *>(choice + e);
            rank += (c.x > ch[0] || (c.x == ch[0] && e < lane)) + (c.y > ch[0] || (c.y == ch[0] && e + 1 < lane)) +
                    (c.z > ch[0] || (c.z == ch[0] && e + 2 < lane)) + (c.w > ch[0] || (c.w == ch[0] && e + 3 < lane));
        }
        const bool chosen = lane < a.outputs && rank < a.top;
        if (chosen) idx[rank] = lane;
        if (!(a.renormalise || a.over_chosen)) {
            if (chosen) wgt[rank] = s[0] * a.weight_scale;
            return;
        }
        __builtin_amdgcn_wave_barrier();
        if (chosen) choice[rank] = s[0];
        __threadfence_block();
        __builtin_amdgcn_wave_barrier();
        float sum_chosen = 0.f;
        for (int k = 0; k < a.top; ++k) sum_chosen += choice[k];
        if (lane < a.top) wgt[lane] = choice[lane] / (sum_chosen + a.sum_eps) * a.weight_scale;
        return;
    }
    float total = 0.f;
    for (int k = 0; k < a.top; ++k) {
        // the largest remaining choice score; of equal ones the lowest index
        float bv = -INFINITY, bs = 0.f;
        int be = 0x7fffffff;
#pragma unroll
        for (int j = 0; j < PL; ++j) {
            const int e = lane + j * KVA_WAVE;
            if (e < a.outputs && (ch[j] > bv || (ch[j] == bv && e < be))) { bv = ch[j]; be = e; bs = s[j]; }
        }
#pragma unroll
        for (int off = KVA_WAVE / 2; off > 0; off >>= 1) {
            const float ov = __shfl_xor(bv, off, KVA_WAVE), os = __shfl_xor(bs, off, KVA_WAVE);
            const int oe = __shfl_xor(be, off, KVA_WAVE);
            if (ov > bv || (ov == bv && oe < be)) { bv = ov; be = oe; bs = os; }
        }
#pragma unroll
        for (int j = 0; j < PL; ++j)
            if (lane + j * KVA_WAVE == be) ch[j] = __builtin_nanf("");       // (taken: neither above nor equal to anything)
        total += bs;
        if (lane == 0) {
            idx[k] = be;
            wgt[k] = bs;
        }
    }
    if (lane == 0) {
        if (a.renormalise || a.over_chosen)
            for (int k = 0; k < a.top; ++k) wgt[k] = wgt[k] / (total + a.sum_eps) * a.weight_scale;
        else if (a.weight_scale != 1.f)
            for (int k = 0; k < a.top; ++k) wgt[k] *= a.weight_scale;
    }
}

template <int PL>
__global__ void __launch_bounds__(256)
moe_route_kernel(int *__restrict__ idx, float *__restrict__ wgt, const float *__restrict__ logits, MoeRoute a, int tokens,
                 int logits_stride) {
    __shared__ __attribute__((aligned(16))) float choice_s[4][KVA_WAVE * PL];
    const int t = blockIdx.x * (blockDim.x / KVA_WAVE) + threadIdx.x / KVA_WAVE;
    if (t >= tokens) return;
    moe_route_token<PL>(a, logits + (size_t)t * logits_stride, idx + (size_t)t * a.top, wgt + (size_t)t * a.top,
                    choice_s[threadIdx.x / KVA_WAVE]);
}

static int moe_route_check(const MoeRoute &a) {
    KVA_REQUIRE(a.groups >= 1 && a.groups <= KVA_WAVE && a.outputs % a.groups == 0 && a.keep_groups >= 1 &&
                    a.keep_groups <= a.groups && a.group_top >= 1,
                "moe_route: %d groups (at most %d, dividing the %d outputs) of which %d are kept", a.groups, KVA_WAVE, a.outputs,
                a.keep_groups);
    KVA_REQUIRE(a.groups == 1 || (a.outputs / a.groups <= 64 && a.top <= a.keep_groups * (a.outputs / a.groups)),
                "moe_route: groups of at most 64 outputs, and enough outputs in the kept groups for top %d", a.top);
    KVA_REQUIRE(!(a.sigmoid_scores && a.over_chosen), "moe_route: sigmoid scores exclude the softmax over the chosen logits");
    KVA_REQUIRE(a.outputs > 0 && a.outputs <= KVA_WAVE * MOE_ROUTE_PER_LANE, "moe_route: %d router outputs (at most %d)",
                a.outputs, KVA_WAVE * MOE_ROUTE_PER_LANE);
    KVA_REQUIRE(a.top > 0 && a.top <= a.outputs, "moe_route: top %d of %d", a.top, a.outputs);
    return KVA_OK;
}

extern "C" int kva_moe_route(int *idx, float *wgt, const float *logits, const float *correction, int tokens,
                             int outputs, int top, int renormalise, int over_chosen, int sigmoid_scores, int groups,
                             int keep_groups, int group_top, float weight_scale, float sum_eps, int logits_stride,
                             hipStream_t stream) {
    // logits_stride: elements between two tokens' rows of logits (the logits may be the first columns of a wider product)
    KVA_REQUIRE(logits_stride >= outputs, "moe_route: a row of logits holds at least the %d outputs", outputs);
    KVA_REQUIRE(idx && wgt && logits && tokens >= 0, "moe_route: missing operand");
    const MoeRoute a{correction, outputs, top, renormalise, over_chosen, sigmoid_scores, groups, keep_groups, group_top, weight_scale, sum_eps};
    if (int rc = moe_route_check(a)) return rc;
    if (tokens == 0) return KVA_OK;
    hipLaunchKernelGGL(outputs <= KVA_WAVE ? moe_route_kernel<1> : moe_route_kernel<MOE_ROUTE_PER_LANE>, dim3((tokens + 3) / 4), dim3(256), 0, stream, idx, wgt, logits, a, tokens, logits_stride);
    KVA_CHECK_LAUNCH("moe_route");
    return KVA_OK;
}

// ---- slots sorted by expert --------------------------------------------------------------
// experts by token id: idx[t, k] = table[id_t, k] and wgt[t, k] = weight.  A negative id -1 - r stands for
// feedback[r], as in the embedding gather.
struct MoeTable {
    const int *table, *ids, *feedback;
    int rows, top;
    float weight;
    float *wgt;
};

// `group` tiles form a group that belongs to one expert (its last tiles may be padding): what a kernel that
// takes several tiles at once walks over.  One workgroup; a thread keeps up to MOE_SLOTS_IN_REGISTERS slots
// and their places in their experts' runs in registers (all its loads in flight at once, ids and then the
// table's rows, one pass of counters); more slots than that are read and counted twice.  Where runs start is a
// sum over the wavefront, and only the places that no slot takes are filled with -1: nothing waits for a store.
// What bounds it is a chain of trips to memory and LDS on one compute unit.  A slot's two reads after the other, a
// thread for the runs' starts and the whole list filled first -> this, us (from a table of
// ids): 256 slots of 16 experts 4.7 -> 4.3 (4.9 -> 4.9), 8,192 8.9 -> 7.4 (11.3 -> 9.7), 9,976 of 4 experts 12.4 -> 8.9 (16.0 -> 11.7),
// 16,384 of 64 16.4 -> 12.4 (21.8 -> 16.2), of 256 29.8 -> 18.2 (34.9 -> 22.0).
#define MOE_SLOTS_IN_REGISTERS 16
__device__ inline int moe_slot_expert(int *idx, int s, const MoeTable &tab) {
    if (!tab.table) return idx[s];
    int id = tab.ids[s / tab.top];
    if (id < 0) id = tab.feedback[-1 - id];
    id = id < 0 ? 0 : (id >= tab.rows ? tab.rows - 1 : id);
    return tab.table[(size_t)id * tab.top + s % tab.top];
}

// A lane's sum over itself and the lanes in front of it: over a row of 16 lanes, then with the last lanes of the rows before.
__device__ inline int wave_sum_upto(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);         // row_shr:1, :2, :4, :8
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);         // row_bcast:15 to the second and fourth row
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);         // row_bcast:31 to the last two
    return v;
}

__device__ inline void moe_align_workgroup(int *sorted_slot, int *tile_expert, int *idx, int slots, int experts, int capacity,
                                           int max_tiles, int group, const MoeTable &tab, int *count, int *start) {
    const int threads = blockDim.x, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KVA_WAVE), lane = threadIdx.x % KVA_WAVE;
    const bool in_registers = slots <= threads * MOE_SLOTS_IN_REGISTERS;
    int ex[MOE_SLOTS_IN_REGISTERS], at[MOE_SLOTS_IN_REGISTERS];
#pragma unroll
    for (int j = 0; j < MOE_SLOTS_IN_REGISTERS; ++j) ex[j] = -1;
    if (in_registers && tab.table) {
        // slot threadIdx.x + j threads is choice `choice` of token `token`: stepped, not divided for.  (1,024 threads at most: the
        // half that is added is more than the reciprocal's error of 2^-22 makes of them, and less than the next quotient's distance.)
        const float per = __builtin_amdgcn_rcpf((float)tab.top);
        const int first_token = (int)((threadIdx.x + 0.5f) * per), first_choice = threadIdx.x - first_token * tab.top;
        const int tokens = (int)((threads + 0.5f) * per), choices = threads - tokens * tab.top;
        int token = first_token, choice = first_choice;
        auto next = [&]() {
            token += tokens;
            choice += choices;
            if (choice >= tab.top) choice -= tab.top, ++token;
        };
        bool feedback = false;
#pragma unroll
        for (int j = 0; j < MOE_SLOTS_IN_REGISTERS; ++j) {
            if (j * threads >= slots) break;
            at[j] = threadIdx.x + j * threads < slots ? tab.ids[token] : 0;
            next();
        }
#pragma unroll
        for (int j = 0; j < MOE_SLOTS_IN_REGISTERS; ++j)
            if (j * threads < slots) feedback |= at[j] < 0;
        if (feedback)
#pragma unroll
            for (int j = 0; j < MOE_SLOTS_IN_REGISTERS; ++j)
                if (j * threads < slots && at[j] < 0) at[j] = tab.feedback[-1 - at[j]];
        choice = first_choice;
#pragma unroll
        for (int j = 0; j < MOE_SLOTS_IN_REGISTERS; ++j) {
            if (j * threads >= slots) break;
            if (threadIdx.x + j * threads < slots) ex[j] = tab.table[(size_t)max(0, min(at[j], tab.rows - 1)) * tab.top + choice];
            next();
        }
    } else if (in_registers) {
#pragma unroll
        for (int j = 0; j < MOE_SLOTS_IN_REGISTERS; ++j) {
            const int s = threadIdx.x + j * threads;
            if (j * threads >= slots) break;
            ex[j] = s < slots ? idx[s] : -1;
        }
    }
    for (int e = threadIdx.x; e < experts; e += threads) count[e] = 0;
    __syncthreads();
    if (in_registers) {
#pragma unroll
        for (int j = 0; j < MOE_SLOTS_IN_REGISTERS; ++j)
            if (ex[j] >= 0 && ex[j] < experts) at[j] = atomicAdd(&count[ex[j]], 1);
    } else {
        for (int s = threadIdx.x; s < slots; s += threads) {
            const int e = moe_slot_expert(idx, s, tab);
            if (e >= 0 && e < experts) atomicAdd(&count[e], 1);
        }
    }
    __syncthreads();
    // every wavefront sums over all experts; the first one leaves the starts for the slots
    int taken = 0;                      // places in front of this turn's experts
    for (int e0 = 0; e0 < experts; e0 += KVA_WAVE) {
        const int e = e0 + lane, n = e < experts ? count[e] : 0;
        const int run = ((n + MOE_TILE - 1) / MOE_TILE + group - 1) / group * group * MOE_TILE;
        const int upto = wave_sum_upto(run);
        if (wave == 0 && e < experts) start[e] = taken + upto - run;
        for (int i = wave; i < min(KVA_WAVE, experts - e0); i += threads / KVA_WAVE) {      // (all lanes on expert e0 + i)
            const int length = __builtin_amdgcn_readlane(run, i), end = taken + __builtin_amdgcn_readlane(upto, i);
            const int used = __builtin_amdgcn_readlane(n, i), first = end - length;
            for (int p = first + used + lane; p < end; p += KVA_WAVE) sorted_slot[p] = -1;
            for (int t = lane; t < length / MOE_TILE; t += KVA_WAVE) tile_expert[first / MOE_TILE + t] = t * MOE_TILE < used ? e0 + i : -1;
        }
        taken += __builtin_amdgcn_readlane(upto, KVA_WAVE - 1);
    }
    for (int p = taken + threadIdx.x; p < capacity; p += threads) sorted_slot[p] = -1;
    for (int t = taken / MOE_TILE + threadIdx.x; t < max_tiles; t += threads) tile_expert[t] = -1;
    __syncthreads();
    if (in_registers) {
#pragma unroll
        for (int j = 0; j < MOE_SLOTS_IN_REGISTERS; ++j) {
            const int s = threadIdx.x + j * threads;
            if (s >= slots) continue;
            if (ex[j] >= 0 && ex[j] < experts) sorted_slot[start[ex[j]] + at[j]] = s;
            if (tab.table) {
                idx[s] = ex[j];
                tab.wgt[s] = tab.weight;
            }
        }
        return;
    }
    for (int s = threadIdx.x; s < slots; s += threads) {
        const int e = moe_slot_expert(idx, s, tab);
        if (e >= 0 && e < experts) sorted_slot[atomicAdd(&start[e], 1)] = s;
        if (tab.table) {
            idx[s] = e;
            tab.wgt[s] = tab.weight;
        }
    }
}

__global__ void __launch_bounds__(1024)
moe_align_kernel(int *__restrict__ sorted_slot, int *__restrict__ tile_expert, int *idx, int slots, int experts, int capacity,
                 int max_tiles, int group, MoeTable tab) {
    __shared__ int count[MOE_MAX_EXPERTS], start[MOE_MAX_EXPERTS];
    moe_align_workgroup(sorted_slot, tile_expert, idx, slots, experts, capacity, max_tiles, group, tab, count, start);
}

static int moe_align_check(const int *sorted_slot, const int *tile_expert, const int *idx, int slots, int experts, int capacity,
                           int max_tiles, int group) {
    KVA_REQUIRE(group >= 1 && max_tiles % group == 0, "moe_align: %d tiles do not come in groups of %d", max_tiles, group);
    KVA_REQUIRE(sorted_slot && tile_expert && idx, "moe_align: missing operand");
    KVA_REQUIRE(experts > 0 && experts <= MOE_MAX_EXPERTS, "moe_align: %d experts (at most %d)", experts, MOE_MAX_EXPERTS);
    KVA_REQUIRE(capacity == max_tiles * MOE_TILE && capacity >= slots + experts * (MOE_TILE * group - 1),
                "moe_align: a list of %d places cannot hold %d slots of %d experts in tiles of %d", capacity, slots,
                experts, MOE_TILE);
    return KVA_OK;
}

static int moe_align_launch(int *sorted_slot, int *tile_expert, int *idx, int slots, int experts, int capacity, int max_tiles,
                            int group, const MoeTable &tab, hipStream_t stream) {
    if (int rc = moe_align_check(sorted_slot, tile_expert, idx, slots, experts, capacity, max_tiles, group)) return rc;
    hipLaunchKernelGGL(moe_align_kernel, dim3(1), dim3(1024), 0, stream, sorted_slot, tile_expert, idx, slots, experts,
                       capacity, max_tiles, group, tab);
    KVA_CHECK_LAUNCH("moe_align");
    return KVA_OK;
}

extern "C" int kva_moe_align(int *sorted_slot, int *tile_expert, const int *idx, int slots, int experts, int capacity,
                             int max_tiles, int group, hipStream_t stream) {
    // (without a table the kernel only reads idx)
    return moe_align_launch(sorted_slot, tile_expert, const_cast<int *>(idx), slots, experts, capacity, max_tiles, group,
                            MoeTable{nullptr, nullptr, nullptr, 0, 1, 0.f, nullptr}, stream);
}

extern "C" int kva_moe_table_align(int *sorted_slot, int *tile_expert, int *idx, float *wgt, const int *table, int table_rows,
                                   const int *ids, const int *feedback, int tokens, int top, float weight, int experts,
                                   int capacity, int max_tiles, int group, hipStream_t stream) {
    KVA_REQUIRE(wgt && table && ids && table_rows > 0 && tokens >= 0 && top > 0, "moe_table_align: missing operand or bad sizes");
    return moe_align_launch(sorted_slot, tile_expert, idx, tokens * top, experts, capacity, max_tiles, group,
                            MoeTable{table, ids, feedback, table_rows, top, weight, wgt}, stream);
}

// ---- the router's product, the choice and (few tokens) the sorted list in one launch ---------------------------------
// A workgroup of 16 wavefronts takes 16 tokens: logits^T[n, t] = W[n, :] . x[t, :] + bias[n] on the matrix cores (bf16
// operands, whose products are exact, and fp32 sums), a tile of 16 outputs and a part of K a wavefront; the parts meet in
// LDS in a fixed order, and wavefront i then routes token i.  Outputs past the router's (an expert's gate, say) go to
// `rest` [tokens, N - outputs].  A single workgroup's slots are sorted by expert right behind it.  The order of every
// sum depends on the sizes alone.
#define MOE_ROUTER_MAX_N 512

struct MoeRouter {
    const bf16_t *x, *w;
    const float *bias;
    float *rest;
    int *idx;
    float *wgt;
    int tokens, N, K, x_stride;
};

// PARTS neighbouring parts of `each` steps of 32 from number part0 on, of `steps` in all: the loads of AHEAD steps of every part are on their
// way at once, and right behind the first ones what `behind()` asks for.  RAGGED: parts are no whole AHEADs of steps, or the last ones are
// shorter; what lies past a part's end is made zero on both sides.  (With a branch around every product instead the compiler moved its
// loads into the branch, and a part was a chain of two trips to memory, one part after the other.)
template <int PARTS, int AHEAD, bool RAGGED, class F>
__device__ __forceinline__ void moe_router_parts_as(const bf16_t *wrow, const bf16_t *xrow, int part0, int each, int steps, f32x4 (&acc)[PARTS], F behind) {
#pragma unroll
    for (int j = 0; j < PARTS; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int c = 0; c < each; c += AHEAD) {
        Frag8 xf[PARTS][AHEAD], wf[PARTS][AHEAD];
#pragma unroll
        for (int j = 0; j < PARTS; ++j)
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) {
                const int s = (part0 + j) * each + c + i, at = 32 * (RAGGED ? min(s, steps - 1) : s);
                xf[j][i].u4 = *reinterpret_cast<const uint4 *>(xrow + at);
                wf[j][i].u4 = *reinterpret_cast<const uint4 *>(wrow + at);
            }
        __builtin_amdgcn_sched_barrier(0);
        if (c == 0) behind();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < AHEAD; ++i)
#pragma unroll
            for (int j = 0; j < PARTS; ++j) {
                if (RAGGED) {
                    const uint32_t in = c + i < each && (part0 + j) * each + c + i < steps ? 0xffffffffu : 0u;
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        xf[j][i].u2[q].x &= in; xf[j][i].u2[q].y &= in;
                        wf[j][i].u2[q].x &= in; wf[j][i].u2[q].y &= in;
                    }
                }
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j][i].v, xf[j][i].v, acc[j], 0, 0, 0);
            }
    }
}
template <int PARTS, class F>
__device__ __forceinline__ void moe_router_parts(const bf16_t *wrow, const bf16_t *xrow, int part0, int each, int parts, int steps,
                                                 f32x4 (&acc)[PARTS], F behind) {
    // (parts of one to three steps ask for no more than they have.  With four asked for every time, the first product with the choice inside, one token of
    // four gated experts and a shared one, K of 512 / 1,024 / 1,536: 7.7 / 8.5 / 11.7 us, so 5.8 / 6.9 / 10.2)
    if (each <= 1) moe_router_parts_as<PARTS, 1, true>(wrow, xrow, part0, each, steps, acc, behind);
    else if (each <= 2) moe_router_parts_as<PARTS, 2, true>(wrow, xrow, part0, each, steps, acc, behind);
    else if (each <= 3) moe_router_parts_as<PARTS, 3, true>(wrow, xrow, part0, each, steps, acc, behind);
    else if (each % 4 == 0 && each * parts == steps) moe_router_parts_as<PARTS, 4, false>(wrow, xrow, part0, each, steps, acc, behind);
    else moe_router_parts_as<PARTS, 4, true>(wrow, xrow, part0, each, steps, acc, behind);
}

template <int PL>
__global__ void __launch_bounds__(1024)
moe_router_kernel(MoeRouter m, MoeRoute a, int *__restrict__ sorted_slot, int *__restrict__ tile_expert, int experts, int capacity,
                  int max_tiles, int group) {
    extern __shared__ __attribute__((aligned(16))) float moe_lds[];
    __shared__ int count[MOE_MAX_EXPERTS], start[MOE_MAX_EXPERTS];
    __shared__ float part[16][KVA_WAVE][4];
    const int lane = threadIdx.x % KVA_WAVE, wave = threadIdx.x / KVA_WAVE, r = lane & 15, g = lane >> 4;
    const int t0 = blockIdx.x * 16, tiles = (m.N + 15) / 16, parts = tiles < 16 ? 16 / tiles : 1;
    float *logits = moe_lds;                                     // [16 tokens][N]
    const int steps = m.K / 32, per = (steps + parts - 1) / parts;
    const bf16_t *xrow = m.x + (size_t)min(t0 + r, m.tokens - 1) * m.x_stride + 8 * g;
    for (int tile0 = 0; tile0 < tiles; tile0 += 16) {            // (more than 256 outputs: in turns)
        const int tile = tile0 + wave % min(tiles, 16), kp = wave / min(tiles, 16);
        const bool on = tile < tiles && kp < parts;
        f32x4 sums[1] = {f32x4{0.f, 0.f, 0.f, 0.f}};
        if (on) moe_router_parts(m.w + (size_t)min(16 * tile + r, m.N - 1) * m.K + 8 * g, xrow, kp, per, parts, steps, sums, []() {});
        const f32x4 acc = sums[0];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) part[wave][lane][i] = acc[i];
        __syncthreads();
        if (on && kp == 0) {                                     // lane (token r, group g): outputs 16 tile + 4 g .. + 3
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int n = 16 * tile + 4 * g + i;
                float v = acc[i];
                for (int p = 1; p < parts; ++p) v += part[wave + p * min(tiles, 16)][lane][i];
                if (n < m.N) logits[r * m.N + n] = v + (m.bias ? m.bias[n] : 0.f);
            }
        }
    }
    __syncthreads();
    const int t = t0 + wave;
    if (t < m.tokens) {
        moe_route_token<PL>(a, logits + wave * m.N, m.idx + (size_t)t * a.top, m.wgt + (size_t)t * a.top,
                            logits + 16 * m.N + (PL == 1 || a.groups > 1 ? wave * KVA_WAVE * PL : 0));
        for (int n = a.outputs + lane; n < m.N; n += KVA_WAVE) m.rest[(size_t)t * (m.N - a.outputs) + n - a.outputs] = logits[wave * m.N + n];
    }
    if (!sorted_slot) return;
    __threadfence_block();
    __syncthreads();
    moe_align_workgroup(sorted_slot, tile_expert, m.idx, m.tokens * a.top, experts, capacity, max_tiles, group,
                        MoeTable{nullptr, nullptr, nullptr, 0, 1, 0.f, nullptr}, count, start);
}

extern "C" int kva_moe_router_supported(int x_dtype, int w_dtype, int N, int K) {
    return x_dtype == KVA_BF16 && w_dtype == KVA_BF16 && K > 0 && K % 32 == 0 && N > 0 && N <= MOE_ROUTER_MAX_N;
}

// sorted_slot may be null: the list is then left to kva_moe_align (it must be for more than 16 tokens)
extern "C" int kva_moe_router(int *idx, float *wgt, float *rest, const void *x, int x_stride, const void *w, const float *bias,
                              const float *correction, int tokens, int N, int K, int outputs, int top, int renormalise,
                              int over_chosen, int sigmoid_scores, int groups, int keep_groups, int group_top,
                              float weight_scale, float sum_eps, int *sorted_slot, int *tile_expert, int experts,
                              int capacity, int max_tiles, int group, hipStream_t stream) {
    KVA_REQUIRE(idx && wgt && x && w && tokens >= 0 && outputs <= N && (outputs == N || rest), "moe_router: missing operand");
    KVA_REQUIRE(kva_moe_router_supported(KVA_BF16, KVA_BF16, N, K) && x_stride >= K && x_stride % 8 == 0 &&
                    ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15) == 0,
                "moe_router: no kernel for %d outputs of %d elements, or rows that do not start at multiples of 16 bytes", N, K);
    const MoeRoute a{correction, outputs, top, renormalise, over_chosen, sigmoid_scores, groups, keep_groups, group_top, weight_scale, sum_eps};
    if (int rc = moe_route_check(a)) return rc;
    if (sorted_slot) {
        KVA_REQUIRE(tokens <= 16, "moe_router: the list of more than 16 tokens is sorted by a launch of its own");
        if (int rc = moe_align_check(sorted_slot, tile_expert, idx, tokens * top, experts, capacity, max_tiles, group)) return rc;
    }
    if (tokens == 0) return KVA_OK;
    const int per_lane = outputs <= KVA_WAVE ? 1 : MOE_ROUTE_PER_LANE;
    const size_t lds = (size_t)(16 * N + (per_lane == 1 || groups > 1 ? 16 * KVA_WAVE * per_lane : 0)) * sizeof(float);
    auto kernel = per_lane == 1 ? moe_router_kernel<1> : moe_router_kernel<MOE_ROUTE_PER_LANE>;
    if (lds > 32 * 1024)
        hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(kernel, dim3((tokens + 15) / 16), dim3(1024), lds, stream,
                       MoeRouter{(const bf16_t *)x, (const bf16_t *)w, bias, rest, idx, wgt, tokens, N, K, x_stride}, a, sorted_slot,
                       tile_expert, experts, capacity, max_tiles, group);
    KVA_CHECK_LAUNCH("moe_router");
    return KVA_OK;
}

// ---- one product per tile ------------------------------------------------------------------
struct MoeRows {
    const int *sorted_slot, *tile_expert;
    const float *slot_weight;       // mode 1: of the row that is written; mode 0 (optional): of the row that is read
    int top, N, K, mode, act;
    int tiled;                      // the matrices lie in operand order: [N / 16][K / 32][lane][8] (lane = 16 (k % 32 / 8) + n % 16)
    int gated;                      // mode 0: rows 2 j and 2 j + 1 of the matrix are output j's gate and up rows
    float limit;                    // activation 4 (clamped swish): gate and up are cut off at this value
};

// mode 0 of a gated expert: outputs n (even) and n + 1 of the product are one output of the layer
// (a weight on the expert's input multiplies both of them in front of the activation: W (w x) = w (W x))
__device__ inline void moe_store_gated(const MoeRows &a, void *out, int out_dtype, int place, int slot, int n, float gate, float up) {
    if (a.slot_weight) {
        gate *= a.slot_weight[slot];
        up *= a.slot_weight[slot];
    }
    const float v = a.act == 4 ? kva_gated_activate(gate, up, KVA_ACT_SWISH_CLAMPED, a.limit) : moe_activate(gate, a.act) * up;
    const size_t at = (size_t)place * (a.N / 2) + n / 2;
    if (out_dtype == KVA_BF16) reinterpret_cast<uint16_t *>(out)[at] = float_to_bf16_bits(v);
    else reinterpret_cast<float *>(out)[at] = v;
}

__device__ inline void moe_store(const MoeRows &a, void *out, int out_dtype, int place, int slot, int n, float v) {
    if (a.mode == 0) {
        if (a.slot_weight) v *= a.slot_weight[slot];
        v = moe_activate(v, a.act);
        if (out_dtype == KVA_BF16) reinterpret_cast<uint16_t *>(out)[(size_t)place * a.N + n] = float_to_bf16_bits(v);
        else reinterpret_cast<float *>(out)[(size_t)place * a.N + n] = v;
    } else {
        reinterpret_cast<float *>(out)[(size_t)slot * a.N + n] = a.slot_weight ? v * a.slot_weight[slot] : v;
    }
}

// plain: a workgroup takes a tile of 16 rows and 64 outputs; thread (row, cx) 4 neighbouring outputs
template <typename T>
__global__ void __launch_bounds__(256)
moe_expert_rows_kernel(MoeRows a, void *__restrict__ out, int out_dtype, const T *__restrict__ x,
                       const T *__restrict__ w) {
    __shared__ float xs[MOE_TILE][33], ws[64][33];
    const int tile = blockIdx.y, e = a.tile_expert[tile];
    if (e < 0) return;
    const int n0 = blockIdx.x * 64, row = threadIdx.x / 16, cx = threadIdx.x % 16;
    const int place = tile * MOE_TILE + row, slot = a.sorted_slot[place];
    const T *wm = w + (size_t)e * a.N * a.K;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < a.K; k0 += 32) {
        __syncthreads();
        for (int i = threadIdx.x; i < MOE_TILE * 32; i += 256) {
            const int rr = i / 32, kk = k0 + i % 32;
            const int sl = a.sorted_slot[tile * MOE_TILE + rr];
            const size_t src = a.mode == 0 ? (size_t)(sl < 0 ? 0 : sl / a.top) : (size_t)(tile * MOE_TILE + rr);
            xs[rr][i % 32] = (kk < a.K && sl >= 0) ? to_float(x[src * a.K + kk]) : 0.f;
        }
        for (int i = threadIdx.x; i < 64 * 32; i += 256) {
            const int nn = n0 + i / 32, kk = k0 + i % 32;
            ws[i / 32][i % 32] = (nn < a.N && kk < a.K) ? to_float(wm[(size_t)nn * a.K + kk]) : 0.f;
        }
        __syncthreads();
        for (int kk = 0; kk < 32; ++kk) {
            const float xv = xs[row][kk];
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[j] += xv * ws[4 * cx + j][kk];
        }
    }
    if (slot < 0) return;
    if (a.gated) {
#pragma unroll
        for (int j = 0; j < 4; j += 2) {
            const int n = n0 + 4 * cx + j;
            if (n + 1 < a.N) moe_store_gated(a, out, out_dtype, place, slot, n, acc[j], acc[j + 1]);
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int n = n0 + 4 * cx + j;
        if (n < a.N) moe_store(a, out, out_dtype, place, slot, n, acc[j]);
    }
}

// matrix cores: a workgroup takes RT tiles of 16 rows and NT tiles of 16 outputs; out^T[n, t] =
// W[e][n, :] . x[t, :]; operands straight from memory, 16 bytes a lane and product.  Its four
// wavefronts take a quarter of K each (the same quarters whatever NT, RT and the batch are) and the
// first adds the four partial results up in a fixed order: with few tiles - decoded tokens - there are
// four times as many wavefronts streaming the experts' matrices.  Row tiles of one expert (the list is
// sorted by expert, so neighbours mostly are) share what is loaded of its matrix; a group of tiles
// that spans two experts is walked tile by tile.
template <int NT, int RT>
__device__ inline void moe_tiles_product(const MoeRows &a, void *__restrict__ out, int out_dtype,
                                         const bf16_t *__restrict__ x, const bf16_t *__restrict__ w, int first_tile,
                                         int e, int n_first, float (*red)[KVA_WAVE][4]) {
    const int lane = threadIdx.x % KVA_WAVE, wave = threadIdx.x / KVA_WAVE, r = lane & 15, g = lane >> 4;
    int place[RT], slot[RT];
    const bf16_t *xrow[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        place[rt] = (first_tile + rt) * MOE_TILE + r;
        slot[rt] = a.sorted_slot[place[rt]];
        const size_t src = a.mode == 0 ? (size_t)(slot[rt] < 0 ? 0 : slot[rt] / a.top) : (size_t)place[rt];
        xrow[rt] = x + src * a.K + 8 * g;
    }
    const bf16_t *wrow[NT];
    const int wstep = a.tiled ? 16 * 32 : 32;       // from one step of 32 to the next
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
        wrow[nt] = w + (a.tiled ? ((size_t)e * a.N + min(n_first + 16 * nt, a.N - 16)) * a.K + 8 * lane
                                : ((size_t)e * a.N + min(n_first + 16 * nt + r, a.N - 1)) * a.K + 8 * g);
    f32x4 acc[NT][RT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) acc[nt][rt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int steps = a.K / 32, per = (steps + 3) / 4;
    const int s0 = wave * per, s1 = min(steps, s0 + per);
    constexpr int AHEAD = NT * RT == 1 ? 8 : 2;         // a tile of its own: as many loads in flight as there are products
#pragma unroll AHEAD
    for (int s = s0; s < s1; ++s) {
        const int k0 = 32 * s;
        Frag8 xf[RT], wf[NT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) xf[rt].u4 = *reinterpret_cast<const uint4 *>(xrow[rt] + k0);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) wf[nt].u4 = *reinterpret_cast<const uint4 *>(wrow[nt] + (size_t)s * wstep);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
                acc[nt][rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[nt].v, xf[rt].v, acc[nt][rt], 0, 0, 0);
    }
    __syncthreads();                 // whoever still reads the partial results of the call before is done
    if (wave > 0)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int i = 0; i < 4; ++i) red[((wave - 1) * NT + nt) * RT + rt][lane][i] = acc[nt][rt][i];
    __syncthreads();
    if (wave > 0) return;
    // lane (row r, group g) holds outputs n0 + 4 g .. + 3 of its row
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        if (slot[rt] < 0) continue;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                v[i] = ((acc[nt][rt][i] + red[(0 * NT + nt) * RT + rt][lane][i]) + red[(1 * NT + nt) * RT + rt][lane][i])
                       + red[(2 * NT + nt) * RT + rt][lane][i];
            const int n = n_first + 16 * nt + 4 * g;
            if (a.gated) {
                if (n + 1 < a.N) moe_store_gated(a, out, out_dtype, place[rt], slot[rt], n, v[0], v[1]);
                if (n + 3 < a.N) moe_store_gated(a, out, out_dtype, place[rt], slot[rt], n + 2, v[2], v[3]);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (n + i < a.N) moe_store(a, out, out_dtype, place[rt], slot[rt], n + i, v[i]);
            }
        }
    }
}

template <int NT, int RT>
__global__ void __launch_bounds__(256)
moe_expert_rows_mfma_kernel(MoeRows a, void *__restrict__ out, int out_dtype, const bf16_t *__restrict__ x,
                            const bf16_t *__restrict__ w, int max_tiles) {
    __shared__ float red[3 * NT * RT][KVA_WAVE][4];
    const int first = blockIdx.y * RT, n_first = blockIdx.x * 16 * NT;
    const int e0 = a.tile_expert[first];
    bool same = e0 >= 0;
#pragma unroll
    for (int rt = 1; rt < RT; ++rt) same = same && first + rt < max_tiles && a.tile_expert[first + rt] == e0;
    if (same) {
        moe_tiles_product<NT, RT>(a, out, out_dtype, x, w, first, e0, n_first, red);
        return;
    }
    for (int rt = 0; rt < RT; ++rt) {
        const int e = first + rt < max_tiles ? a.tile_expert[first + rt] : -1;
        if (e >= 0) moe_tiles_product<NT, 1>(a, out, out_dtype, x, w, first + rt, e, n_first, red);
    }
}

// Eight neighbouring results of the first product, a place's from n on (n a multiple of 8), the slot's weight (or 1) at hand: as
// moe_store and moe_store_gated do one by one.  `aligned`: rows start at multiples of 16 bytes.
template <int ACT, bool GATED>
__device__ inline void moe_store8(const MoeRows &a, void *__restrict__ out, int place, float weight, int n, const float *v, bool aligned) {
    float f[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = v[i] * weight;
    if (GATED) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            f[i] = ACT == 4 ? kva_gated_activate(f[2 * i], f[2 * i + 1], KVA_ACT_SWISH_CLAMPED, a.limit) : moe_activate(f[2 * i], ACT) * f[2 * i + 1];
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] = moe_activate(f[i], ACT);
    }
    const int width = GATED ? a.N / 2 : a.N, at = GATED ? n / 2 : n, count = GATED ? 4 : 8;
    uint16_t *o = reinterpret_cast<uint16_t *>(out) + (size_t)place * width + at;
    if (aligned && n + 8 <= a.N) {
        const Frag8 h = {.p2 = {pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3]), pack_bf16(f[4], f[5]), pack_bf16(f[6], f[7])}};
        if (GATED) *reinterpret_cast<uint2 *>(o) = h.u2[0];
        else *reinterpret_cast<uint4 *>(o) = h.u4;
        return;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
        if (i < count && at + i < width) o[i] = float_to_bf16_bits(f[i]);
}

// four of the second one, to the slot's row (fp32)
__device__ inline void moe_store4(const MoeRows &a, void *__restrict__ out, int slot, float weight, int n, const float *v, bool aligned) {
    float *o = reinterpret_cast<float *>(out) + (size_t)slot * a.N + n;
    if (aligned && n + 4 <= a.N) {
        *reinterpret_cast<float4 *>(o) = make_float4(v[0] * weight, v[1] * weight, v[2] * weight, v[3] * weight);
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (n + i < a.N) o[i] = v[i] * weight;
}

// (one variable in LDS: with several the compiler tells them apart, and waits for all loads on their way to one before it reads it)
template <int RT, int NT, int STAGES>
struct MoeLds {
    static constexpr int STRIDE = 128 + 4, ROWS = RingProduct<RT, NT, STAGES>::ROWS;         // a row of results in LDS
    union {
        typename RingProduct<RT, NT, STAGES>::Shared operands;
        float results[ROWS * STRIDE];
    };
    int slot_of[ROWS];
    float weight_of[ROWS];
};

// matrix cores, many rows an expert: a workgroup takes a group of 2 RT tiles of one expert (32 RT rows) and 32 NT
// outputs, operands through LDS (lds_product.h).  The list was laid out for any split among the experts; the groups
// that hold something come first, and only they are dealt out, neighbours to one die: a die reads few experts.
template <int RT, int NT, int STAGES>
__global__ void __launch_bounds__(256, 2)
moe_expert_rows_lds_kernel(MoeRows a, void *__restrict__ out, int out_dtype, const bf16_t *__restrict__ x,
                           const bf16_t *__restrict__ w, int n_blocks, int groups) {
    typedef RingProduct<RT, NT, STAGES> Product;
    __shared__ __align__(16) MoeLds<RT, NT, STAGES> shared;
    const int lane = threadIdx.x % KVA_WAVE, wave = threadIdx.x / KVA_WAVE, r = lane & 15, g = lane >> 4;
    int used = 0;
    for (int g0 = 0; g0 < groups; g0 += KVA_WAVE)
        used += __popcll(__ballot(g0 + lane < groups && a.tile_expert[(size_t)min(g0 + lane, groups - 1) * 2 * RT] >= 0));
    const int total = used * n_blocks;
    if ((int)blockIdx.x >= total) return;
    const int id = die_order(blockIdx.x, total);
    const int first = (id / n_blocks) * 2 * RT, n0 = (id % n_blocks) * Product::OUTS;
    const int e = a.tile_expert[first];
    if (e < 0) return;
    const int wr = wave & 1, wn = wave >> 1;
    Product p;
    p.xbuf = buffer_at(x, 0xffffffffull);
#pragma unroll
    for (int i = 0; i < Product::XI; ++i) {
        const int place = first * MOE_TILE + p.row(i), slot = a.sorted_slot[place];
        p.xo[i] = 2 * ((a.mode == 0 ? (slot < 0 ? 0 : slot / a.top) : place) * a.K + p.element());
    }
    if (threadIdx.x < Product::ROWS) {
        const int slot = a.sorted_slot[first * MOE_TILE + threadIdx.x];
        shared.slot_of[threadIdx.x] = slot;
        shared.weight_of[threadIdx.x] = a.slot_weight && slot >= 0 ? a.slot_weight[slot] : 1.f;
    }
    const bf16_t *we = w + (size_t)e * a.N * a.K;
    if (a.tiled) p.tiled_w(we, a.N, a.K, n0);
    else p.plain_w(we, a.N, a.K, n0);
    f32x4 acc[NT][RT];
    p.run(shared.operands, a.K, acc);
    // The results go out by rows, through LDS in 32 bits (where the operands were): four tiles of either half of the
    // outputs at a time, then 8 neighbouring outputs a thread.  The activation is chosen once, in front: choosing it for every
    // element was most of the 25 us that 4,096 x 4,096 outputs cost beside their sums.
    const bool aligned = (a.gated ? a.N / 2 : a.N) % 8 == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
    auto store = [&](auto act, auto gated) {
#pragma unroll
        for (int part = 0; part < NT / 4; ++part) {
            if (part > 0) __syncthreads();
#pragma unroll
            for (int nt = 0; nt < 4; ++nt)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
                    *reinterpret_cast<f32x4 *>(&shared.results[((wr * RT + rt) * 16 + r) * MoeLds<RT, NT, STAGES>::STRIDE + wn * 64 + nt * 16 + 4 * g]) =
                        acc[4 * part + nt][rt];
            __syncthreads();
            // (second product: 4 outputs a thread, so that a store takes whole lines)
            constexpr int AT_ONCE = decltype(act)::value < 0 ? 4 : 8, ACROSS = 128 / AT_ONCE;
            const int c = AT_ONCE * (threadIdx.x % ACROSS), n = n0 + c / 64 * 16 * NT + part * 64 + c % 64;
            if (n < a.N)
                for (int row = threadIdx.x / ACROSS; row < Product::ROWS; row += 256 / ACROSS) {
                    const int slot = shared.slot_of[row];
                    const float *v = &shared.results[row * MoeLds<RT, NT, STAGES>::STRIDE + c];
                    if (slot < 0) continue;
                    if constexpr (AT_ONCE == 8)
                        moe_store8<decltype(act)::value, decltype(gated)::value>(a, out, first * MOE_TILE + row, shared.weight_of[row], n, v, aligned);
                    else moe_store4(a, out, slot, shared.weight_of[row], n, v, aligned);
                }
        }
    };
#define KVA_MOE_STORE(ACT)                                                                  \
    case ACT:                                                                               \
        if (a.gated) store(std::integral_constant<int, ACT>{}, std::true_type{});           \
        else store(std::integral_constant<int, ACT>{}, std::false_type{});                  \
        break
    if (a.mode == 1) {
        store(std::integral_constant<int, -1>{}, std::false_type{});
        return;
    }
    switch (a.act) {
        KVA_MOE_STORE(0);
        KVA_MOE_STORE(1);
        KVA_MOE_STORE(2);
        KVA_MOE_STORE(3);
        KVA_MOE_STORE(5);
        default: store(std::integral_constant<int, 4>{}, std::true_type{});         // (the clamped activation is a gated one)
    }
#undef KVA_MOE_STORE
}

// groups of so many tiles of 16 rows have a kernel of their own (for operands in bf16 whose K is a multiple of 32)
extern "C" int kva_moe_group_supported(int group, int K) { return (group == 4 || group == 8) && K > 0 && K % 32 == 0; }

extern "C" int kva_moe_expert_rows(void *out, int out_dtype, const void *x, const void *w, int dtype,
                                   const int *sorted_slot, const int *tile_expert, const float *slot_weight,
                                   int max_tiles, int top, int N, int K, int mode, int act, int gated, float limit,
                                   int group, int wide, int tiled, hipStream_t stream) {
    KVA_REQUIRE(!tiled || (dtype == KVA_BF16 && K % 32 == 0 && N % 16 == 0), "moe_expert_rows: no operand order for %d x %d", N, K);
    KVA_REQUIRE(group == 1 || (dtype == KVA_BF16 && kva_moe_group_supported(group, K) && max_tiles % group == 0),
                "moe_expert_rows: no kernel for groups of %d tiles, %d of them, with K = %d", group, max_tiles, K);
    KVA_REQUIRE(!wide || group == 8, "moe_expert_rows: 256 outputs a workgroup go with groups of 8 tiles, not %d", group);
    KVA_REQUIRE(act != 4 || gated, "moe_expert_rows: the clamped activation is a gated one");
    KVA_REQUIRE(!gated || (mode == 0 && N % 2 == 0), "moe_expert_rows: gate and up rows come in pairs, in the first product");
    KVA_REQUIRE(out && x && w && sorted_slot && tile_expert, "moe_expert_rows: missing operand");
    // slot_weight: in mode 1 of the row that is written, in mode 0 of the row that is read; absent: 1
    KVA_REQUIRE(mode == 0 || (mode == 1 && out_dtype == KVA_F32), "moe_expert_rows: mode 1 writes fp32 rows");
    KVA_REQUIRE(mode == 1 || out_dtype == dtype, "moe_expert_rows: mode 0 writes rows of the operands' type");
    KVA_REQUIRE(N > 0 && K > 0 && top > 0 && act >= 0 && act <= 5, "moe_expert_rows: bad sizes or activation");
    KVA_REQUIRE(max_tiles >= 0 && max_tiles <= 65535, "moe_expert_rows: %d tiles are too many for one launch", max_tiles);
    if (max_tiles == 0) return KVA_OK;
    MoeRows a{sorted_slot, tile_expert, slot_weight, top, N, K, mode, act, tiled, gated, limit};
    // (operands at other addresses than multiples of 16: loads that go straight to LDS do not take those, the kernels below do,
    // over a list in groups as over any other; and their rows lie within 2 GiB)
    if (group > 1 && (((uintptr_t)x | (uintptr_t)w) & 15) == 0 && (long long)max_tiles * MOE_TILE * K * 2 <= 0x7fffffffll) {
        const int groups = max_tiles / group, blocks = wide ? (N + 255) / 256 : (N + 127) / 128;
        KVA_REQUIRE((long long)blocks * groups <= 0x7fffffff, "moe_expert_rows: too many workgroups");
        if (wide)
            hipLaunchKernelGGL((moe_expert_rows_lds_kernel<4, 8, 3>), dim3(blocks * groups), dim3(256), 0, stream, a, out, out_dtype,
                               (const bf16_t *)x, (const bf16_t *)w, blocks, groups);
        else if (group == 8)
            hipLaunchKernelGGL((moe_expert_rows_lds_kernel<4, 4, 4>), dim3(blocks * groups), dim3(256), 0, stream, a, out, out_dtype,
                               (const bf16_t *)x, (const bf16_t *)w, blocks, groups);
        else
            hipLaunchKernelGGL((moe_expert_rows_lds_kernel<2, 4, 4>), dim3(blocks * groups), dim3(256), 0, stream, a, out, out_dtype,
                               (const bf16_t *)x, (const bf16_t *)w, blocks, groups);
    } else if (dtype == KVA_BF16 && K % 32 == 0) {
        // few tiles: 16 outputs a workgroup, so that enough of them stream the matrices; many: 64 outputs and
        // four row tiles, which share what they load
        if ((long long)max_tiles * ((N + 15) / 16) <= 8192)
            hipLaunchKernelGGL((moe_expert_rows_mfma_kernel<1, 1>), dim3((N + 15) / 16, max_tiles), dim3(256), 0, stream, a,
                               out, out_dtype, (const bf16_t *)x, (const bf16_t *)w, max_tiles);
        else
            hipLaunchKernelGGL((moe_expert_rows_mfma_kernel<4, 4>), dim3((N + 63) / 64, (max_tiles + 3) / 4), dim3(256), 0,
                               stream, a, out, out_dtype, (const bf16_t *)x, (const bf16_t *)w, max_tiles);
    } else if (dtype == KVA_BF16) {
        hipLaunchKernelGGL(moe_expert_rows_kernel<bf16_t>, dim3((N + 63) / 64, max_tiles), dim3(256), 0, stream, a, out,
                           out_dtype, (const bf16_t *)x, (const bf16_t *)w);
    } else if (dtype == KVA_F32) {
        hipLaunchKernelGGL(moe_expert_rows_kernel<float>, dim3((N + 63) / 64, max_tiles), dim3(256), 0, stream, a, out,
                           out_dtype, (const float *)x, (const float *)w);
    } else KVA_REQUIRE(false, "moe_expert_rows: unsupported dtype %d", dtype);
    KVA_CHECK_LAUNCH("moe_expert_rows");
    return KVA_OK;
}

// ---- few tokens ------------------------------------------------------------------------------
// Up to 16 tokens: a tile has a row for every one of them, so nothing is sorted.  A workgroup takes 16 outputs of one unit: an
// expert, or (fewer slots than experts) the expert of a slot, whose first slot's workgroups take it; one more unit is the expert
// that every token uses, in the same launch.  Which tokens chose the expert is read from idx by the lanes themselves, or (mode 0)
// looked up in a table by token id, in which case one workgroup leaves idx and the weights for whoever comes next.  A token's
// choices are distinct.  The four wavefronts take a quarter of K each, eight steps of 32 on their way at once: a workgroup is as long
// as its chain of trips to memory.  (Lists, rows and matrix one after another, a list's launch in front, and a tile of 16 places
// an expert: 8 tokens of 16 experts of 768 x 2,048, four each and a shared one, 19.6 + 7.6 and 16.4 + 4.8 us; now 20.7 and 10.3,
// 4.7 TB/s; one token of four experts of 1,024 x 2,048 11.9 and 8.2, now 6.5 and 5.6.  All 16 steps at once: 22.7 and 10.3.)
// Two tiles of outputs a workgroup share the rows where there are enough workgroups without: 16 tokens of 64 experts, 6,240 and
// 8,320 workgroups, 78 / 41 -> 67 / 37 us; 1,632 and 2,176 of them 20.8 / 10.3 -> 21.6 / 9.9.
//
// ROUTED (mode 0): the router's product and the choice are made here too, by every workgroup for itself, in the order of sums
// of the router's own launch: 16 parts of K.  A router of up to 16 outputs is 64 KB that all workgroups read from L2 while
// their matrix is on its way; where the workgroups and the tokens are few (the caller's rule) that saves 2 us of a launch's 6-8.  All of the
// router's loads, the matrix's first ones and what is added to the scores are on their way at once (228 registers: two
// workgroups a unit): one token of 4 experts of 1,024 x 2,048 11.5 -> 9.5 us in the model, of 1,536 x 2,048 and a shared one 13.8 -> 12.6.
//  mode 0: out[slot] = act(W[e] x[token]) (x's type),   mode 1: out[slot] = W[e] x[slot] * weight[slot] (fp32).
struct MoeFewRouter {
    const bf16_t *w;                // [N, K], N up to 16
    const float *bias;
    float *rest, *wgt;              // outputs past the router's [tokens, N - outputs]; weights [tokens, top]
    int N;
    MoeRoute rule;
};

struct MoeFew {
    const int *idx;
    MoeTable tab;
    int *idx_out;
    const float *slot_weight;
    int tokens, top, experts, units, by_slot, N, K, mode, act, gated;
    float limit;
    const bf16_t *shared_x, *shared_w;      // rows a token; a matrix in tiles of 16 rows (first product: gates' tiles, then ups')
    void *shared_out;
    int shared_N, shared_K, shared_act;
    float shared_limit;
};

__device__ inline float moe_gated(float gate, float up, int act, float limit) {
    return act == 4 ? kva_gated_activate(gate, up, KVA_ACT_SWISH_CLAMPED, limit) : moe_activate(gate, act) * up;
}

__device__ inline uint32_t moe_pack(float a, float b) { return __builtin_bit_cast(uint32_t, pack_bf16(a, b)); }

template <int AHEAD, int NT, bool ROUTED>
__global__ void __launch_bounds__(256)
moe_few_rows_kernel(MoeFew a, MoeFewRouter ro, void *__restrict__ out, const bf16_t *__restrict__ x, const bf16_t *__restrict__ w) {
    __shared__ float red[3][NT][KVA_WAVE][4];
    __shared__ __attribute__((aligned(16))) float part[ROUTED ? 16 : 1][KVA_WAVE][4], logits[ROUTED ? 16 : 1][16], choice[4][KVA_WAVE], wgt_s[ROUTED ? 256 : 1],
        correction_s[ROUTED ? 16 : 1];
    __shared__ int idx_s[ROUTED ? 256 : 1];
    const int lane = threadIdx.x % KVA_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KVA_WAVE), r = lane & 15, g = lane >> 4;
    const int unit = blockIdx.y, slots = a.tokens * a.top;
    const bool shared = unit == a.units;
    if (a.tab.table && unit == 0 && blockIdx.x == 0)
        for (int s = threadIdx.x; s < slots; s += 256) {
            a.idx_out[s] = moe_slot_expert(nullptr, s, a.tab);
            a.tab.wgt[s] = a.tab.weight;
        }
    const int N = shared ? a.shared_N : a.N, K = shared ? a.shared_K : a.K, first = 16 * NT * blockIdx.x;
    if (first >= N) return;
    int slot = -1, e = unit;            // this lane's token's slot with the expert
    const int steps = K / 32, per = (steps + 3) / 4, s0 = wave * per, s1 = min(steps, s0 + per);
    const bool pairs = shared && a.mode == 0;       // 8 gate rows and 8 up rows of two tiles
    const bf16_t *wrow[NT], *xrow;
    Frag8 wf[NT][AHEAD], xf[AHEAD];
    auto rows = [&]() {
        xrow = (shared ? a.shared_x : x) + (size_t)(shared || a.mode == 0 ? min(r, a.tokens - 1) : max(slot, 0)) * K + 8 * g;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int n0 = min(first + 16 * t, N - 16);
            wrow[t] = shared ? a.shared_w : w + (size_t)e * N * K;
            if (pairs) wrow[t] += (size_t)((r >> 3) * (N / 32) + n0 / 32) * 16 * K + 8 * (16 * g + n0 / 2 % 16 + (r & 7));
            else wrow[t] += (size_t)n0 * K + 8 * lane;
        }
    };
    auto load = [&](int s) {
#pragma unroll
        for (int i = 0; i < AHEAD; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t) wf[t][i].u4 = *reinterpret_cast<const uint4 *>(wrow[t] + (size_t)max(0, min(s + i, s1 - 1)) * 512);
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) xf[i].u4 = *reinterpret_cast<const uint4 *>(xrow + 32 * max(0, min(s + i, s1 - 1)));
    };
    if constexpr (ROUTED) {
        rows();                         // (the expert is the unit's number: its matrix comes while the choice is made)
        const bf16_t *rx = x + (size_t)min(r, a.tokens - 1) * a.K + 8 * g, *rw = ro.w + (size_t)min(r, ro.N - 1) * a.K + 8 * g;
        const int all = a.K / 32, each = (all + 15) / 16;
        // (what the choice adds to logits and scores: asked for first, or it is a trip to memory of its own behind the sums)
        const int own = 4 * (threadIdx.x / 64) + threadIdx.x % 4;
        const float bias = ro.bias ? ro.bias[min(own, ro.N - 1)] : 0.f;
        const float correction = ro.rule.correction ? ro.rule.correction[min((int)threadIdx.x, ro.rule.outputs - 1)] : 0.f;
        __builtin_amdgcn_sched_barrier(0);
        f32x4 sums[4];
        moe_router_parts(rw, rx, 4 * wave, each, 16, all, sums, [&]() { load(s0); });
#pragma unroll
        for (int j = 0; j < 4; ++j) *reinterpret_cast<f32x4 *>(part[4 * wave + j][lane]) = sums[j];
        __syncthreads();
        {                               // element i of lane l: token l % 16, output 4 (l / 16) + i
            const int l = threadIdx.x / 4, n = 4 * (l / 16) + threadIdx.x % 4;
            float v = part[0][l][threadIdx.x % 4];
#pragma unroll
            for (int p = 1; p < 16; ++p) v += part[p][l][threadIdx.x % 4];
            if (n < ro.N) logits[l % 16][n] = v + bias;
        }
        if (threadIdx.x < 16) correction_s[threadIdx.x] = correction;
        __syncthreads();
        MoeRoute rule = ro.rule;
        if (rule.correction) rule.correction = correction_s;
        for (int t = wave; t < a.tokens; t += 4)
            moe_route_token<1>(rule, logits[t], idx_s + t * a.top, wgt_s + t * a.top, choice[wave]);
        __syncthreads();
        if (unit == 0 && blockIdx.x == 0) {
            for (int s = threadIdx.x; s < slots; s += 256) {
                a.idx_out[s] = idx_s[s];
                ro.wgt[s] = wgt_s[s];
            }
            const int more = ro.N - ro.rule.outputs;
            for (int i = threadIdx.x; i < more * a.tokens; i += 256) ro.rest[i] = logits[i / more][ro.rule.outputs + i % more];
        }
    }
    if (shared) {
        slot = r < a.tokens ? r : -1;
    } else {
        int *idx = const_cast<int *>(a.idx);
        auto chosen = [&](int s) { return ROUTED ? idx_s[s] : moe_slot_expert(idx, s, a.tab); };
        if (a.by_slot) e = __builtin_amdgcn_readfirstlane(chosen(unit));
        if (r < a.tokens)
            for (int k = g; k < a.top; k += 4)
                if (chosen(r * a.top + k) == e) slot = r * a.top + k;
        slot = max(slot, __shfl_xor(slot, 16, KVA_WAVE));
        slot = max(slot, __shfl_xor(slot, 32, KVA_WAVE));
        const unsigned long long chose = __ballot(slot >= 0);
        if (e < 0 || e >= a.experts || !chose) return;
        if (a.by_slot && __shfl(slot, __ffsll(chose) - 1, KVA_WAVE) != unit) return;
    }
    if constexpr (!ROUTED) {
        rows();
        load(s0);
    }
    f32x4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s = s0; s < s1; s += AHEAD) {
        if (s > s0) load(s);
#pragma unroll
        for (int i = 0; i < AHEAD; ++i)
            if (s + i < s1)
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[t][i].v, xf[i].v, acc[t], 0, 0, 0);
    }
    if (wave > 0)
#pragma unroll
        for (int t = 0; t < NT; ++t) *reinterpret_cast<f32x4 *>(red[wave - 1][t][lane]) = acc[t];
    __syncthreads();
    if (wave > 0) return;
    const float weight = shared || slot < 0 ? 1.f : ROUTED && a.slot_weight ? wgt_s[slot] : a.slot_weight ? a.slot_weight[slot] : 1.f;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int n0 = first + 16 * t, n = n0 + 4 * g;
        if (n0 >= N) return;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = (((acc[t][i] + red[0][t][lane][i]) + red[1][t][lane][i]) + red[2][t][lane][i]) * weight;
        if (pairs) {                    // lanes of g and g + 2: outputs n0 / 2 + 4 g .. + 3, gates and ups
            float up[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) up[i] = __shfl_xor(v[i], 32, KVA_WAVE);
            if (g >= 2 || slot < 0) continue;
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = moe_gated(v[i], up[i], a.shared_act, a.shared_limit);
            *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(a.shared_out) + (size_t)slot * (N / 2) + n0 / 2 + 4 * g) =
                make_uint2(moe_pack(v[0], v[1]), moe_pack(v[2], v[3]));
        } else if (slot < 0) {
        } else if (a.mode == 1) {
            // (rounded as the product's bf16 rows are where it runs alone: what comes behind is the same for few tokens and many)
            if (shared)
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = bf16_bits_to_float(float_to_bf16_bits(v[i]));
            *reinterpret_cast<float4 *>((shared ? reinterpret_cast<float *>(a.shared_out) : reinterpret_cast<float *>(out)) + (size_t)slot * N + n) =
                make_float4(v[0], v[1], v[2], v[3]);
        } else if (a.gated) {
            *reinterpret_cast<uint32_t *>(reinterpret_cast<uint16_t *>(out) + (size_t)slot * (N / 2) + n / 2) =
                moe_pack(moe_gated(v[0], v[1], a.act, a.limit), moe_gated(v[2], v[3], a.act, a.limit));
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = moe_activate(v[i], a.act);
            *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(out) + (size_t)slot * N + n) =
                make_uint2(moe_pack(v[0], v[1]), moe_pack(v[2], v[3]));
        }
    }
}

extern "C" int kva_moe_few_max_tokens(void) { return 16; }

// whether the first product can make the choice itself (every expert its unit, one tile of router outputs, a place for every slot)
extern "C" int kva_moe_few_routes(int router_N, int slots, int experts) {
    return router_N > 0 && router_N <= 16 && slots >= experts && slots <= 256;
}

extern "C" int kva_moe_few_rows(void *out, const void *x, const void *w, const int *idx, const int *table, int table_rows, int table_top,
                                const int *ids, const int *feedback, float table_weight, int *idx_out, float *wgt_out,
                                int tokens, int top, int experts, int N, int K, int mode, int act, int gated, float limit,
                                const float *slot_weight, const void *shared_x, const void *shared_w, void *shared_out,
                                int shared_N, int shared_K, int shared_act, float shared_limit, const void *router_w, int router_N,
                                const float *router_bias, const float *correction, float *rest, int outputs, int renormalise,
                                int over_chosen, int sigmoid_scores, int groups, int keep_groups, int group_top, float weight_scale,
                                float sum_eps, hipStream_t stream) {
    // router_w: the router's product and the choice here (idx_out, wgt_out; slot_weight then means: weights stand on the inputs)
    const MoeFewRouter ro{(const bf16_t *)router_w, router_bias, rest, wgt_out, router_N,
                          MoeRoute{correction, outputs, top, renormalise, over_chosen, sigmoid_scores, groups, keep_groups, group_top, weight_scale, sum_eps}};
    if (router_w) {
        KVA_REQUIRE(mode == 0 && !table && idx_out && wgt_out && outputs <= router_N && (outputs == router_N || rest) &&
                        kva_moe_few_routes(router_N, tokens * top, experts) && ((uintptr_t)router_w & 15) == 0,
                    "moe_few_rows: no choice of %d outputs here", router_N);
        if (int rc = moe_route_check(ro.rule)) return rc;
    }
    KVA_REQUIRE(out && x && w && (idx || table || router_w) && tokens >= 0 && tokens <= 16 && top > 0 && experts > 0,
                "moe_few_rows: missing operand, or more than 16 tokens (%d)", tokens);
    KVA_REQUIRE(N > 0 && N % 16 == 0 && K > 0 && K % 32 == 0, "moe_few_rows: no operand order for %d x %d", N, K);
    KVA_REQUIRE(mode == 0 || mode == 1, "moe_few_rows: the first product (0) or the second (1)");
    KVA_REQUIRE(!table || (mode == 0 && ids && idx_out && wgt_out && table_rows > 0 && table_top == top),
                "moe_few_rows: a table goes with the first product, with ids and places for what it says");
    KVA_REQUIRE(act >= 0 && act <= 5 && (act != 4 || gated) && (!gated || mode == 0), "moe_few_rows: bad activation");
    KVA_REQUIRE(!shared_w || (shared_x && shared_out && shared_N > 0 && shared_N % (mode == 0 ? 32 : 16) == 0 && shared_K > 0 && shared_K % 32 == 0 &&
                              shared_act >= 0 && shared_act <= 5),
                "moe_few_rows: no operand order for %d x %d of the expert every token uses", shared_N, shared_K);
    KVA_REQUIRE((((uintptr_t)out | (uintptr_t)x | (uintptr_t)w | (uintptr_t)shared_x | (uintptr_t)shared_w | (uintptr_t)shared_out) & 15) == 0,
                "moe_few_rows: operands start at multiples of 16 bytes");
    if (tokens == 0) return KVA_OK;
    const int slots = tokens * top, by_slot = slots < experts, units = by_slot ? slots : experts;
    KVA_REQUIRE(units < 65535, "moe_few_rows: too many workgroups");
    const MoeFew a{idx, MoeTable{table, ids, feedback, table_rows, top, table_weight, wgt_out}, idx_out, slot_weight, tokens, top, experts,
                   units, by_slot, N, K, mode, act, gated, limit, (const bf16_t *)shared_x, (const bf16_t *)shared_w, shared_out, shared_N,
                   shared_K, shared_act, shared_limit};
    const int wide = shared_w && shared_N > N ? shared_N : N, deep = shared_w && shared_K > K ? shared_K : K, per = (deep / 32 + 3) / 4;
    const int tiles = (wide + 15) / 16, rows = units + (shared_w ? 1 : 0), nt = !router_w && tiles * rows > 4096 ? 2 : 1;
    const dim3 grid((tiles + nt - 1) / nt, rows);
#define KVA_MOE_FEW(AHEAD, NT, ROUTED) \
    hipLaunchKernelGGL((moe_few_rows_kernel<AHEAD, NT, ROUTED>), grid, dim3(256), 0, stream, a, ro, out, (const bf16_t *)x, (const bf16_t *)w)
    if (router_w) KVA_MOE_FEW(8, 1, true);
    else if (nt == 2) KVA_MOE_FEW(8, 2, false);
    else if (per > 4) KVA_MOE_FEW(8, 1, false);
    else KVA_MOE_FEW(4, 1, false);
#undef KVA_MOE_FEW
    KVA_CHECK_LAUNCH("moe_few_rows");
    return KVA_OK;
}

// ---- weighted sum --------------------------------------------------------------------------
__device__ inline float moe_ld(const void *p, int dtype, size_t i) {
    return dtype == KVA_BF16 ? bf16_bits_to_float(reinterpret_cast<const uint16_t *>(p)[i])
                             : reinterpret_cast<const float *>(p)[i];
}

__global__ void __launch_bounds__(256)
moe_combine_kernel(void *__restrict__ out, const void *__restrict__ x, int dtype, const float *__restrict__ rows,
                   const int *__restrict__ idx, const float *__restrict__ wgt, const void *__restrict__ extra, int extra_dtype,
                   const float *__restrict__ extra_gate, int extra_gate_stride, int width, int top, int experts) {
    const size_t t = blockIdx.x;
    // (optional) the addend enters times sigmoid(extra_gate[t * stride]), one number a token (a column of a wider array)
    const float eg = extra && extra_gate ? 1.f / (1.f + expf(-extra_gate[t * extra_gate_stride])) : 1.f;
    if (width % 4 == 0 && ((reinterpret_cast<uintptr_t>(rows) | reinterpret_cast<uintptr_t>(out)) & 15) == 0) {
        // four neighbouring columns a thread, 16 bytes of every row at a time; the additions per column are
        // in the order of the scalar loop below
        for (int j = threadIdx.x * 4; j < width; j += blockDim.x * 4) {
            float acc[4] = {0.f, 0.f, 0.f, 0.f};
            for (int k = 0; k < top; ++k) {
                const size_t s = t * top + k;
                if (idx[s] < experts) {
                    const float4 r = *reinterpret_cast<const float4 *>(rows + s * width + j);
                    acc[0] += r.x; acc[1] += r.y; acc[2] += r.z; acc[3] += r.w;
                } else {
                    const float g = wgt[s];
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[e] += g * moe_ld(x, dtype, t * width + j + e);
                }
            }
            if (extra) {
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] += eg * moe_ld(extra, extra_dtype, t * width + j + e);
            }
            if (dtype == KVA_BF16) {
                const uint2 o = make_uint2((uint32_t)float_to_bf16_bits(acc[0]) | ((uint32_t)float_to_bf16_bits(acc[1]) << 16),
                                           (uint32_t)float_to_bf16_bits(acc[2]) | ((uint32_t)float_to_bf16_bits(acc[3]) << 16));
                *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(out) + t * width + j) = o;
            } else {
                *reinterpret_cast<float4 *>(reinterpret_cast<float *>(out) + t * width + j) = make_float4(acc[0], acc[1], acc[2], acc[3]);
            }
        }
        return;
    }
    for (int j = threadIdx.x; j < width; j += blockDim.x) {
        float acc = 0.f;
        for (int k = 0; k < top; ++k) {
            const size_t s = t * top + k;
            if (idx[s] < experts) acc += rows[s * width + j];
            else acc += wgt[s] * (dtype == KVA_BF16 ? bf16_bits_to_float(reinterpret_cast<const uint16_t *>(x)[t * width + j])
                                                    : reinterpret_cast<const float *>(x)[t * width + j]);
        }
        // what an expert that every token uses returned, with weight 1
        if (extra) acc += eg * moe_ld(extra, extra_dtype, t * width + j);
        if (dtype == KVA_BF16) reinterpret_cast<uint16_t *>(out)[t * width + j] = float_to_bf16_bits(acc);
        else reinterpret_cast<float *>(out)[t * width + j] = acc;
    }
}

extern "C" int kva_moe_combine(void *out, const void *x, int dtype, const float *rows, const int *idx,
                               const float *wgt, const void *extra, int extra_dtype, const float *extra_gate, int extra_gate_stride,
                               int tokens, int width, int top, int experts, hipStream_t stream) {
    KVA_REQUIRE(out && x && rows && idx && wgt && width > 0 && top > 0, "moe_combine: missing operand");
    KVA_REQUIRE(dtype == KVA_BF16 || dtype == KVA_F32, "moe_combine: unsupported dtype %d", dtype);
    if (tokens <= 0) return KVA_OK;
    hipLaunchKernelGGL(moe_combine_kernel, dim3(tokens), dim3(256), 0, stream, out, x, dtype, rows, idx, wgt, extra, extra_dtype, extra_gate,
                       extra_gate_stride, width, top, experts);
    KVA_CHECK_LAUNCH("moe_combine");
    return KVA_OK;
}

// ---- small products with 32-bit results -------------------------------------------------------
// out[t, n] = sum_k x[t, k] * w[n, k] in fp32, for the small matrices whose results must not be rounded
// to 16 bits (a router's logits; the second half of a low-rank projection that makes decays, which
// may be finished here: bias, sigmoid, power).  x and
// w may be bf16 or fp32; every product and sum is fp32.  A workgroup takes a token: its row of x goes
// to LDS once; with a long K a wavefront takes an output and its lanes stride over K (sum by
// wavefront reduction), with a short K a thread takes an output.  The order of every sum depends on
// the sizes alone.
#define SMALL_PRODUCT_MAX_K 8192

// eight neighbouring elements from index i on (i a multiple of 8: 16 or 32 aligned bytes)
__device__ inline void moe_ld8(const void *p, int dtype, size_t i, float (&f)[8]) {
    if (dtype == KVA_BF16) {
        const uint4 v = *reinterpret_cast<const uint4 *>(reinterpret_cast<const uint16_t *>(p) + i);
        const unsigned u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            f[2 * j] = __uint_as_float(u[j] << 16);
            f[2 * j + 1] = __uint_as_float(u[j] & 0xffff0000u);
        }
    } else {
        const float4 a = *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(p) + i);
        const float4 b = *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(p) + i + 4);
        f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w; f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
    }
}

// the result as it is, plus a bias, or - with decay_inv_tau > 0 - turned into a decay:
// sigmoid(z)^(1 / tau) = exp(-softplus(-z) / tau) with z = the sum plus its bias
// or - with rate_log - into exp(-exp(rate_log[n / rate_group]) softplus(z)): a decay per output whose rate
// is shared by groups of neighbouring outputs (the key channels of a head)
__device__ inline float small_product_finish(float acc, const float *bias, int n, float decay_inv_tau,
                                             const float *rate_log, int rate_group) {
    const float z = acc + (bias ? bias[n] : 0.f);
    if (rate_log) return expf(-expf(rate_log[n / rate_group]) * (fmaxf(z, 0.f) + log1pf(expf(-fabsf(z)))));
    if (decay_inv_tau <= 0.f) return z;
    const float softplus = fmaxf(-z, 0.f) + log1pf(expf(-fabsf(z)));
    return expf(-softplus * decay_inv_tau);
}

__global__ void __launch_bounds__(256)
small_product_f32_kernel(float *__restrict__ out, const void *__restrict__ x, int x_dtype, int x_stride,
                         const void *__restrict__ w, int w_dtype, int N, int K, int per_block,
                         const float *__restrict__ bias, float decay_inv_tau, const float *__restrict__ rate_log,
                         int rate_group) {
    extern __shared__ float xs[];
    const size_t t = blockIdx.x;
    const int n_lo = blockIdx.y * per_block, n_hi = min(N, n_lo + per_block);
    for (int k = threadIdx.x; k < K; k += blockDim.x) xs[k] = moe_ld(x, x_dtype, t * x_stride + k);
    __syncthreads();
    const int K8 = (K % 8 == 0) ? K : 0;          // the part read eight elements at a time
    if (K >= 128) {
        const int lane = threadIdx.x % KVA_WAVE, wave = threadIdx.x / KVA_WAVE, waves = blockDim.x / KVA_WAVE;
        for (int n = n_lo + wave; n < n_hi; n += waves) {
            float acc = 0.f;
            for (int k = 8 * lane; k < K8; k += 8 * KVA_WAVE) {
                float f[8];
                moe_ld8(w, w_dtype, (size_t)n * K + k, f);
#pragma unroll
                for (int i = 0; i < 8; ++i) acc += xs[k + i] * f[i];
            }
            for (int k = K8 + lane; k < K; k += KVA_WAVE) acc += xs[k] * moe_ld(w, w_dtype, (size_t)n * K + k);
            acc = wave_sum(acc);
            if (lane == 0) out[t * N + n] = small_product_finish(acc, bias, n, decay_inv_tau, rate_log, rate_group);
        }
    } else {
        for (int n = n_lo + threadIdx.x; n < n_hi; n += blockDim.x) {
            float acc = 0.f;
            for (int k = 0; k < K8; k += 8) {
                float f[8];
                moe_ld8(w, w_dtype, (size_t)n * K + k, f);
#pragma unroll
                for (int i = 0; i < 8; ++i) acc = __builtin_fmaf(xs[k + i], f[i], acc);
            }
            for (int k = K8; k < K; ++k) acc = __builtin_fmaf(xs[k], moe_ld(w, w_dtype, (size_t)n * K + k), acc);
            out[t * N + n] = small_product_finish(acc, bias, n, decay_inv_tau, rate_log, rate_group);
        }
    }
}

extern "C" int kva_small_product_f32(float *out, const void *x, int x_dtype, int x_stride, const void *w, int w_dtype,
                                     int tokens, int N, int K, const float *bias, float decay_inv_tau,
                                     const float *rate_log, int rate_group, hipStream_t stream) {
    KVA_REQUIRE(!rate_log || (rate_group > 0 && N % rate_group == 0 && decay_inv_tau <= 0.f),
                "small_product_f32: rates are shared by whole groups of outputs, and exclude the other decay");
    KVA_REQUIRE(out && x && w && tokens >= 0 && N > 0, "small_product_f32: missing operand or bad sizes");
    KVA_REQUIRE(K > 0 && K <= SMALL_PRODUCT_MAX_K && x_stride >= K, "small_product_f32: K %d must lie in 1..%d", K, SMALL_PRODUCT_MAX_K);
    KVA_REQUIRE((x_dtype == KVA_BF16 || x_dtype == KVA_F32) && (w_dtype == KVA_BF16 || w_dtype == KVA_F32),
                "small_product_f32: unsupported dtype");
    if (tokens == 0) return KVA_OK;
    KVA_REQUIRE((reinterpret_cast<uintptr_t>(w) & 31) == 0, "small_product_f32: the matrix must be aligned to 32 bytes");
    const int per_block = K >= 128 ? 16 : 256;         // outputs a workgroup: four a wavefront, or one a thread
    const int blocks_y = (N + per_block - 1) / per_block;
    KVA_REQUIRE(tokens <= 0x7fffffff && blocks_y <= 65535, "small_product_f32: too many outputs");
    hipLaunchKernelGGL(small_product_f32_kernel, dim3(tokens, blocks_y), dim3(256), (size_t)K * sizeof(float), stream,
                       out, x, x_dtype, x_stride, w, w_dtype, N, K, per_block, bias, decay_inv_tau, rate_log,
                       rate_group > 0 ? rate_group : 1);
    KVA_CHECK_LAUNCH("small_product_f32");
    return KVA_OK;
}
