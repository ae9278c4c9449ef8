// A bf16 product of many rows on the matrix cores for weights kept in operand order, operands through LDS: the middle of the
// products in gemm_tiles.hip.
//
// WR x WN x WK wavefronts take 16 RT WR rows of x and 16 NT WN outputs.  WR and WN of them share rows and outputs, WK the elements
// of K: a stage is 32 WK KSUB of them, and wavefronts with other wk multiply other 32s of it (the caller adds their results up).
// STAGES stages stand in LDS in a ring; they get there without a stop in registers (16 bytes a lane), and a wavefront reads its
// next operands while it multiplies the ones before.  One barrier a stage.
//
// What bounds it: with 256 x 256 a workgroup the matrix cores and, of 1.4 PFLOP/s at 8,190 x 4,096 x 14,336, some 10 % the loads
// (without them 1.7; without the reads from LDS 1.55; with neither 2.2); smaller tiles the rate at which a compute unit takes
// operands in, 60 to 80 GB/s: 64 x 64 0.28 us a stage of 64 elements, 128 x 128 0.39, 256 x 256 1.1.  Stages of 64 elements, for
// which a row's piece is a whole cache line, against 32: 16,384 outputs of 2,048 rows and inputs 114 -> 112 us.  Tried: the
// 32 x 32 x 16 instruction (112 -> 121 us, 8,190 x 4,096 x 14,336 687 -> 737), four wavefronts of 128 x 128 (143: too few
// registers), every workgroup from a K of its own (112 -> 120: units that walk in step share what L2 holds).
#pragma once
#include "lds_product.h"

template <int RT_, int NT_, int WR_, int WN_, int WK_, int KSUB_, int STAGES_>
struct TileProduct {
    static constexpr int RT = RT_, NT = NT_, WR = WR_, WN = WN_, WK = WK_, KSUB = KSUB_, STAGES = STAGES_;
    static constexpr int WAVES = WR * WN * WK, THREADS = KVA_WAVE * WAVES, ROWS = 16 * RT * WR, OUTS = 16 * NT * WN;
    static constexpr int STEPS = WK * KSUB, KS = 32 * STEPS;                   // steps of 32 and elements of K a stage
    static_assert(STEPS == 2 && KSUB <= 2 && STAGES >= 2, "a row's piece of a stage is one cache line");
    // pieces of 1 KiB a stage, and how many of them a wavefront brings (where they do not come out even some bring the last one
    // again: the same bytes to the same place)
    static constexpr int XB = ROWS * KS / 512, WB = OUTS * KS / 512;
    static constexpr int XI = (XB + WAVES - 1) / WAVES, WI = (WB + WAVES - 1) / WAVES, LOADS = XI + WI;
    static_assert((STAGES - 1) * LOADS < 64, "loads on their way are counted in six bits");
    // x: pieces of 8 rows x 64 elements, row by row, the eight 16-byte parts of row r in the order part ^ (r % 8), so that the 16
    // rows of an operand lie in different banks.  w: a piece is 32 elements of a tile of 16 rows, in operand order.
    struct Shared {
        bf16_t x[STAGES][ROWS * KS], w[STAGES][OUTS * KS];
    };
    Buffer xbuf, wbuf;
    int xo[XI], wo[WI];             // bytes

    __device__ __forceinline__ static int x_piece(int wave, int i) { return XB % WAVES ? min(wave + WAVES * i, XB - 1) : wave + WAVES * i; }
    __device__ __forceinline__ static int w_piece(int wave, int i) { return WB % WAVES ? min(wave + WAVES * i, WB - 1) : wave + WAVES * i; }

    // rows m0 .. m0 + ROWS - 1 of x (past the last one the last one again); tile_of(j): which tile of w is the workgroup's j-th
    template <class F>
    __device__ __forceinline__ void init(const bf16_t *x, int M, int m0, const bf16_t *w, int tiles, int K, F tile_of) {
        const int rows = min(ROWS, M - m0);
        init(buffer_at(x + (size_t)m0 * K, (size_t)rows * K * 2), [&](int i) { return min(i, rows - 1); }, w, tiles, K, tile_of);
    }
    // row_of(i): which row of the buffer is the workgroup's i-th
    template <class R, class F>
    __device__ __forceinline__ void init(Buffer x, R row_of, const bf16_t *w, int tiles, int K, F tile_of) {
        const int lane = threadIdx.x % KVA_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KVA_WAVE);
        xbuf = x;
        wbuf = buffer_at(w, (size_t)tiles * 16 * K * 2);
#pragma unroll
        for (int i = 0; i < XI; ++i)
            xo[i] = 2 * (row_of(8 * x_piece(wave, i) + lane / 8) * K + 8 * ((lane % 8) ^ (lane / 8)));
#pragma unroll
        for (int i = 0; i < WI; ++i) {
            const int piece = w_piece(wave, i);
            wo[i] = 2 * (tile_of(piece / STEPS) * 16 * K + (piece % STEPS) * 512 + 8 * lane);
        }
    }

    // Elements k_begin .. k_end - 1 (both multiples of KS, at least one stage).  acc[nt][rt]: lane (r = lane % 16, g = lane / 16) gets
    // outputs 16 (NT wn + nt) + 4 g .. + 3 of row 16 (RT wr + rt) + r.
    // PAIRED: rows 2 j and 2 j + 1 of w are the gate and the up row of output j.  Two tiles hold 16 of them, and of each pair of tiles
    // (nt even) the lane gets the gate and the up rows of outputs 8 (NT wn + nt) + 4 g .. + 3: gates in acc[nt] and ups in acc[nt + 1]
    // where g < 2, the other way round where g >= 2 (so that the 16 rows read at once lie in different banks).
    template <bool PAIRED = false>
    __device__ __forceinline__ void run(Shared &s, int k_begin, int k_end, f32x4 (&acc)[NT][RT]) const {
        const int lane = threadIdx.x % KVA_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / KVA_WAVE), r = lane & 15, g = lane >> 4;
        const int wk = wave / (WR * WN), wr = wave % WR, wn = wave / WR % WN;
        const int last = k_end - KS;        // (past the end the last stage again: as many loads are on their way in every turn)
        int xat[KSUB];
#pragma unroll
        for (int j = 0; j < KSUB; ++j)
            xat[j] = (2 * wr * RT + r / 8) * 512 + (r % 8) * 64 + 8 * ((4 * (wk * KSUB + j) + g) ^ (r % 8));
        const int wat = (wn * NT * STEPS + wk * KSUB) * 512 + (PAIRED ? r / 8 * STEPS * 512 + 8 * (16 * g + 2 * (r % 8) + r / 8) : 8 * lane);
        const int odd = PAIRED ? 8 * (1 - 2 * (r / 8)) - STEPS * 512 : 0;       // elements from an even tile's place to the next one's
        auto load = [&](int i, int slot, int k0) {
            const int k = min(k0, last);
            if (i < XI) buffer_to_lds(xbuf, xo[i], 2 * k, &s.x[slot][x_piece(wave, i) * 512]);
            else buffer_to_lds(wbuf, wo[i - XI], 32 * k, &s.w[slot][w_piece(wave, i - XI) * 512]);
        };
        b16x8 xf[2][RT], wf[2][NT];
        auto read = [&](int i, int set, int slot, int j) {
            if (i < RT) xf[set][i] = *reinterpret_cast<const b16x8 *>(&s.x[slot][xat[j] + i * 1024]);
            else wf[set][i - RT] = *reinterpret_cast<const b16x8 *>(&s.w[slot][wat + ((i - RT) * STEPS + j) * 512 + ((i - RT) % 2 ? odd : 0)]);
        };
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) acc[nt][rt] = f32x4{0.f, 0.f, 0.f, 0.f};
        __builtin_amdgcn_s_waitcnt(0xc07f);
#pragma unroll
        for (int t = 0; t < STAGES; ++t)
#pragma unroll
            for (int i = 0; i < LOADS; ++i) load(i, t, k_begin + t * KS);
        wait_and_meet<(STAGES - 1) * LOADS>();
        constexpr int READS = RT + NT, PRODUCTS = NT * RT;
#pragma unroll
        for (int i = 0; i < READS; ++i) read(i, 0, 0, 0);
        int slot = 0;
        // The operands of a step are in `set`; behind its products the next step's are read.  With the last step of a stage goes
        // the stage that follows STAGES later: every wavefront has read this one (into registers) and the next has arrived.
        auto round = [&](int set, int j, int k0) {
            const bool edge = j + 1 == KSUB;
            const int after = slot + 1 == STAGES ? 0 : slot + 1, next = edge ? after : slot, nj = edge ? 0 : j + 1;
            if (edge) {
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_waitcnt((((STAGES - 2) * LOADS) & 15) | (((STAGES - 2) * LOADS) >> 4 << 14) | 0x70);
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
                asm volatile("" ::: "memory");
            }
            int reads = 0, loads = 0;
#pragma unroll
            for (int i = 0; i < PRODUCTS; ++i) {
                acc[i / RT][i % RT] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[set][i / RT], xf[set][i % RT], acc[i / RT][i % RT], 0, 0, 0);
                // (a read behind every second product where there are enough: LDS takes longer for one than a product lasts)
                const int upto = i == PRODUCTS - 1 ? READS : PRODUCTS >= 2 * READS ? (i + 2) / 2 : i + 1;
#pragma unroll
                for (; reads < READS && reads < upto; ++reads) read(reads, 1 - set, next, nj);
                if (edge) {
                    const int due = i == PRODUCTS - 1 ? LOADS : (i + 1) * LOADS / PRODUCTS;
#pragma unroll
                    for (; loads < due; ++loads) load(loads, slot, k0 + STAGES * KS);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (edge) slot = next;
        };
        int k0 = k_begin;
        if constexpr (KSUB == 2) {
            for (; k0 < k_end; k0 += KS) {
                round(0, 0, k0);
                round(1, 1, k0);
            }
        } else {
            for (; k0 + KS < k_end; k0 += 2 * KS) {
                round(0, 0, k0);
                round(1, 0, k0 + KS);
            }
            if (k0 < k_end) round(0, 0, k0);
        }
        wait_and_meet<0>();                 // nothing is on its way any more, nobody reads: the caller may use the LDS
    }
};
