// A bf16 product of many rows on the matrix cores, operands through LDS: the middle of kernels that differ in
// where their operands' rows lie and in what they do with the result.  LdsProduct: products per head and expanded keys and
// values, whose rows lie anywhere; RingProduct, further down: experts' products, whose rows are reached from one base.
//
// A workgroup of four wavefronts takes 32 RT rows of x and 32 NT outputs (rows of w), a wavefront half of
// either.  32 elements of K of both operands are a stage; STAGES of them stand in LDS in a ring.  They get there
// without a stop in registers (global_load_lds, 16 bytes a lane), STAGES - 1 of them on their way while one is
// multiplied: a stage is 512 cycles of matrix products with RT = 4 and NT = 8, a trip to L2 two to four
// times that.  K (a multiple of 32) is added in ascending order into one accumulator an output.
//
// Before, operands went through registers, one stage of 64 elements ahead, 128 x 128 at a time, and results to memory
// one by one (LdsProduct, which the experts' products used then): of 8,192 slots of 16 experts, 1,536 x 2,048 / 2,048 x 768:
// 122 / 61 -> 78 / 60 us; of 4 experts, 1,024 x 2,048 / 2,048 x 1,024: 132 / 70 -> 56 / 43; 2,048 slots of 16: 67 / 29 -> 36 / 22.  The middle alone
// (4,096 x 4,096 x 2,048, w in operand order): 1.23 PFLOP/s; without its loads 1.61, without its reads 1.41.
//
// What bounds it: a wavefront reads (RT + NT) KiB of operands from LDS for RT NT products of 16 cycles; four of them
// at RT = 4, NT = 8 ask for 96 of the 128 bytes a cycle that LDS gives, at 4 x 4 for all 128.
#pragma once
#include "common.h"
#include "attention_frag.h"

#define LDSP_K 32

// 16 bytes a lane from memory to LDS, the wavefront's 1 KiB in the order of the lanes from `to` (the same in all) on
__device__ __forceinline__ void load_to_lds(const void *from, void *to) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) unsigned int *)from,
                                     (__attribute__((address_space(3))) unsigned int *)to, 16, 0, 0);
}
// The same from a buffer that starts at `base` (the same in all lanes): bytes `offset` (a lane's own) + `shared` from there on.  The
// compiler counts operand reads from LDS that are still on their way past these loads; past load_to_lds, which it takes for one
// that may read LDS itself, it waits for all of them.  Nothing is read past `bytes`.
typedef __amdgpu_buffer_rsrc_t Buffer;
__device__ __forceinline__ Buffer buffer_at(const void *base, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)(bytes < 0xffffffffull ? bytes : 0xffffffffull), 0x00027000);
}
__device__ __forceinline__ void buffer_to_lds(Buffer from, int offset, int shared, void *to) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(from, (__attribute__((address_space(3))) void *)to, 16, offset, shared, 0, 0);
}
// The wavefront's loads but the last N have arrived; then all wavefronts' have.  Nothing that reads or writes memory
// moves across.
template <int N>
__device__ __forceinline__ void wait_and_meet() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt((N & 15) | (N >> 4 << 14) | 0x70 | 0xf00);       // vmcnt(N), the other counters as they are
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
}

template <int RT, int NT, int STAGES>
struct LdsProduct {
    static constexpr int ROWS = 32 * RT, OUTS = 32 * NT;
    static constexpr int XI = ROWS * LDSP_K / 8 / 256, WI = OUTS * LDSP_K / 8 / 256;      // 16-byte pieces a thread loads
    // Blocks of 16 rows x 32 elements, 1 KiB each.  x (and w kept row by row): row by row, the four 16-byte pieces of
    // row r in the order piece ^ (r / 4 % 4), so that the 16 rows of an operand lie in different banks.  w kept in operand
    // order stands as it is kept.
    struct Shared {
        bf16_t x[STAGES][ROWS * LDSP_K], w[STAGES][OUTS * LDSP_K];
    };
    // Piece i of thread t: row row(i) of x, elements element() .. + 7: `xp` points at its first one of the row.
    const bf16_t *xp[XI], *wp[WI];
    int wmul;                       // elements of w's storage that go by per element of K
    bool w_swizzled;

    __device__ __forceinline__ static int row(int i) { return threadIdx.x / 4 + 64 * i; }
    __device__ __forceinline__ static int element() { return 8 * ((threadIdx.x % 4) ^ (threadIdx.x / 16 % 4)); }

    // w row by row, rows n0 .. n0 + OUTS - 1 (past the last one the last one again)
    __device__ __forceinline__ void plain_w(const bf16_t *w, int N, int K, int n0) {
        wmul = 1;
        w_swizzled = true;
#pragma unroll
        for (int i = 0; i < WI; ++i) wp[i] = w + (size_t)min(n0 + row(i), N - 1) * K + element();
    }
    // w in operand order [N / 16][K / 32][lane][8]: a wavefront's pieces are neighbouring bytes
    __device__ __forceinline__ void tiled_w(const bf16_t *w, int N, int K, int n0) {
        wmul = 16;
        w_swizzled = false;
#pragma unroll
        for (int i = 0; i < WI; ++i)
            wp[i] = w + (size_t)min(n0 + 16 * (int)(threadIdx.x / KVA_WAVE + 4 * i), N - 16) * K + 8 * (threadIdx.x % KVA_WAVE);
    }

    // acc[nt][rt]: lane (r = lane % 16, g = lane / 16) of wavefront (half of the rows wave % 2, of the outputs
    // wave / 2) gets outputs 16 NT (wave / 2) + 16 nt + 4 g .. + 3 of row (wave % 2) 16 RT + 16 rt + r
    __device__ __forceinline__ void run(Shared &s, int K, f32x4 (&acc)[NT][RT]) const {
        const int lane = threadIdx.x % KVA_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KVA_WAVE), r = lane & 15, g = lane >> 4;
        const int wr = wave & 1, wn = wave >> 1;
        const int swizzled = r * LDSP_K + 8 * (g ^ (r / 4)), xat = swizzled, wat = w_swizzled ? swizzled : 8 * lane;
        auto load = [&](int slot, int k0) {
#pragma unroll
            for (int i = 0; i < XI; ++i) load_to_lds(xp[i] + k0, &s.x[slot][(wave + 4 * i) * 512]);
#pragma unroll
            for (int i = 0; i < WI; ++i) load_to_lds(wp[i] + k0 * wmul, &s.w[slot][(wave + 4 * i) * 512]);
        };
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) acc[nt][rt] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int last = K - LDSP_K;        // (past the end the last stage again: as many loads are on their way in every turn)
#pragma unroll
        for (int i = 0; i < STAGES - 1; ++i) load(i, min(i * LDSP_K, last));
        int slot = 0;
        for (int k0 = 0; k0 < K; k0 += LDSP_K) {
            wait_and_meet<(STAGES - 2) * (XI + WI)>();
            const bf16_t *xr = &s.x[slot][wr * RT * 512 + xat], *wrow = &s.w[slot][wn * NT * 512 + wat];
            Frag8 xf[RT], wf[NT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) xf[rt].v = *reinterpret_cast<const b16x8 *>(xr + rt * 512);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) wf[nt].v = *reinterpret_cast<const b16x8 *>(wrow + nt * 512);
            // (read as vectors of bf16, in front of the next loads: the compiler then knows that no load on its way writes what
            // is read here - of which wait_and_meet makes sure - and does not wait for all of them)
            __builtin_amdgcn_sched_barrier(0);
            // the slot read in the turn before: every wavefront has passed the barrier since
            const int into = slot == 0 ? STAGES - 1 : slot - 1;
            load(into, min(k0 + (STAGES - 1) * LDSP_K, last));
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
                    acc[nt][rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[nt].v, xf[rt].v, acc[nt][rt], 0, 0, 0);
            slot = slot + 1 == STAGES ? 0 : slot + 1;
        }
        wait_and_meet<0>();                 // nothing is on its way any more, nobody reads: the caller may use the LDS
    }
};

// The same product with a stage's operands in registers while the ones before are multiplied: what a wavefront reads for the next
// 32 elements of K, and the loads that go to LDS, are issued one at a time behind products, over the one barrier a stage.
// Operands come from buffers (a base and byte offsets of 32 bits).  The experts' products use it, the two before and with it, the
// activation chosen once a workgroup (us): 64 experts of 1,536 x 2,048, 32,768 slots 302 -> 244; 16 experts, 8,192 slots 83 -> 71;
// 4 experts, 9,976 slots 73 -> 63; tiles of 64 x 128, 2,048 slots of 16 experts 47 -> 38.  One workgroup a compute unit would want more
// stages: two of them cover a load's way with their products (1.35 PFLOP/s from K = 2,048 on, either struct).
template <int RT, int NT, int STAGES>
struct RingProduct {
    static constexpr int ROWS = 32 * RT, OUTS = 32 * NT;
    static constexpr int XI = ROWS * LDSP_K / 8 / 256, WI = OUTS * LDSP_K / 8 / 256, LOADS = XI + WI;
    struct Shared {
        bf16_t x[STAGES][ROWS * LDSP_K], w[STAGES][OUTS * LDSP_K];
    };
    Buffer xbuf, wbuf;
    int xo[XI], wo[WI];             // bytes
    int wmul;                       // elements of w's storage that go by per element of K
    bool w_swizzled;

    __device__ __forceinline__ static int row(int i) { return threadIdx.x / 4 + 64 * i; }
    __device__ __forceinline__ static int element() { return 8 * ((threadIdx.x % 4) ^ (threadIdx.x / 16 % 4)); }
    __device__ __forceinline__ void plain_w(const bf16_t *w, int N, int K, int n0) {
        const int rows = min(OUTS, N - n0);
        wmul = 1;
        w_swizzled = true;
        wbuf = buffer_at(w + (size_t)n0 * K, (size_t)rows * K * 2);
#pragma unroll
        for (int i = 0; i < WI; ++i) wo[i] = 2 * (min(row(i), rows - 1) * K + element());
    }
    __device__ __forceinline__ void tiled_w(const bf16_t *w, int N, int K, int n0) {
        const int rows = min(OUTS, N - n0);
        wmul = 16;
        w_swizzled = false;
        wbuf = buffer_at(w + (size_t)n0 * K, (size_t)rows * K * 2);
#pragma unroll
        for (int i = 0; i < WI; ++i)
            wo[i] = 2 * (min(16 * (int)(threadIdx.x / KVA_WAVE + 4 * i), rows - 16) * K + 8 * (int)(threadIdx.x % KVA_WAVE));
    }

    __device__ __forceinline__ void run(Shared &s, int K, f32x4 (&acc)[NT][RT]) const {
        const int lane = threadIdx.x % KVA_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KVA_WAVE), r = lane & 15, g = lane >> 4;
        const int wr = wave & 1, wn = wave >> 1;
        const int swizzled = r * LDSP_K + 8 * (g ^ (r / 4)), xat = wr * RT * 512 + swizzled, wat = wn * NT * 512 + (w_swizzled ? swizzled : 8 * lane);
        const int last = K - LDSP_K;
        auto load = [&](int i, int slot, int k0) {
            const int k = min(k0, last);
            if (i < XI) buffer_to_lds(xbuf, xo[i], 2 * k, &s.x[slot][(wave + 4 * i) * 512]);
            else buffer_to_lds(wbuf, wo[i - XI], 2 * k * wmul, &s.w[slot][(wave + 4 * (i - XI)) * 512]);
        };
        b16x8 xf[2][RT], wf[2][NT];
        auto read = [&](int i, int set, int slot) {
            if (i < RT) xf[set][i] = *reinterpret_cast<const b16x8 *>(&s.x[slot][xat + i * 512]);
            else wf[set][i - RT] = *reinterpret_cast<const b16x8 *>(&s.w[slot][wat + (i - RT) * 512]);
        };
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) acc[nt][rt] = f32x4{0.f, 0.f, 0.f, 0.f};
        __builtin_amdgcn_s_waitcnt(0xc07f);
#pragma unroll
        for (int t = 0; t < STAGES; ++t)
#pragma unroll
            for (int i = 0; i < LOADS; ++i) load(i, t, t * LDSP_K);
        wait_and_meet<(STAGES - 1) * LOADS>();
#pragma unroll
        for (int i = 0; i < RT + NT; ++i) read(i, 0, 0);
        int slot = 0;
        // round t: the operands of stage t are in `set`; stage t + 1 is read, stage t + STAGES goes where stage t was
        auto round = [&](int set, int k0) {
            const int next = slot + 1 == STAGES ? 0 : slot + 1;
            // every wavefront has read stage t (into registers), stage t + 1 has arrived
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt((((STAGES - 2) * LOADS) & 15) | (((STAGES - 2) * LOADS) >> 4 << 14) | 0x70);
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("" ::: "memory");
#pragma unroll
            for (int i = 0; i < NT * RT; ++i) {
                acc[i / RT][i % RT] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[set][i / RT], xf[set][i % RT], acc[i / RT][i % RT], 0, 0, 0);
                // a read behind every second product (LDS takes longer for one than a product lasts), the loads between them
                constexpr int READS = RT + NT, EVERY = NT * RT >= 2 * READS + 2 ? 2 : 1;
                if (i % EVERY == 0 && i / EVERY < READS) read(i / EVERY, 1 - set, next);
                if (EVERY == 2 ? i % 2 == 1 && i / 2 < LOADS : i >= READS && i < READS + LOADS)
                    load(EVERY == 2 ? i / 2 : i - READS, slot, k0 + STAGES * LDSP_K);
                if (EVERY == 1 && i == NT * RT - 1)     // (what had no product to be behind)
#pragma unroll
                    for (int j = NT * RT - READS; j < LOADS; ++j) load(j, slot, k0 + STAGES * LDSP_K);
                __builtin_amdgcn_sched_barrier(0);
            }
            slot = next;
        };
        int k0 = 0;
        for (; k0 + LDSP_K < K; k0 += 2 * LDSP_K) {
            round(0, k0);
            round(1, k0 + LDSP_K);
        }
        if (k0 < K) round(0, k0);
        wait_and_meet<0>();
    }
};

// Workgroup id -> place in the work list such that neighbours of the list run on one of the 8 dies (the hardware
// deals workgroups out in turn): what they share is read into one L2.
__device__ __forceinline__ int die_order(int id, int total) {
    const int die = id % 8, q = total / 8, rem = total % 8;
    return die * q + min(die, rem) + id / 8;
}
