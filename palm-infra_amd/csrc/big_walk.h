// The walk over K of a tile of a product X . W^T that a block of eight waves owns: 64 NT tokens (rows of X) x 256 rows of W,
// bfloat16, 32-bit sums, for the products of a prompt's rows and of many experts' rows.
//
// K goes by in stages of 64: rows of 128 bytes, a whole cache line, straight from memory into LDS (16 bytes a lane, an
// instruction fills 8 rows), two stages, features first, then tokens.  A row's eight 16-byte chunks are permuted by the row's
// number so that the lanes that LDS serves together hit different banks; the lane that fills a place fetches the chunk that
// belongs there.
// Waves: 2 (features) x 4 (tokens), a wave owns 128 x 16 NT.  A stage has two halves: the wave's tokens (both k-steps) and
// its first 64 features are read and multiplied, then its other 64 features.  So three quarters of a stage's rows (set P)
// are free again after the first half, the rest (set Q) after the second, and each is asked for again at once: a load has one
// and a half stages to arrive.
// The waves 0 .. 3 and 4 .. 7, one of each on a SIMD, work half a step apart: while one four read LDS and ask memory, the
// other four multiply, and a barrier swaps them.  All waits are counted by hand; the loads are not seen by the compiler.
#pragma once
#include "lds_stage.h"
#include "mfma.h"

constexpr int BIG_K = 64, BIG_ROW = BIG_K * 2, BIG_WAVES = 8, BIG_THREADS = BIG_WAVES * WAVE;
constexpr int BIG_FEAT = 256, BIG_DIES = 8;

__device__ __forceinline__ void big_load(const char* base, uint32_t offset, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(offset), "s"(base), "s"(lds) : "m0", "memory");
}
__device__ __forceinline__ void big_swap() {               // the barrier between the two fours of waves
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void big_lds_reads_done() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// A lane of a result tile holds four features of one token.  Row 4 g + v of a wave's f-th of four tiles is feature
// 16 g + 4 f + v of their 64, so that a lane's four tiles are 16 features side by side.
__device__ __forceinline__ int big_feature_row(int f, int r) { return 16 * (r / 4) + 4 * f + r % 4; }
__device__ __forceinline__ int big_w_swizzle(int row) { return ((row >> 1) & 1) | ((row >> 3) & 6); }      // rows big_feature_row(f, 0 .. 15)
__device__ __forceinline__ int big_x_swizzle(int row) { return (row >> 1) & 7; }                           // 16 rows side by side

// 16 features of one token's row of the result, from feature `at`
__device__ __forceinline__ void big_store(bf16_t* __restrict__ row, int at, int width, const float (&v)[16]) {
    if (at + 16 <= width) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            uint32_t w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = (uint32_t)f32_to_bf16(v[8 * h + 2 * i]).bits | ((uint32_t)f32_to_bf16(v[8 * h + 2 * i + 1]).bits << 16);
            *reinterpret_cast<uint4*>(row + at + 8 * h) = make_uint4(w[0], w[1], w[2], w[3]);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if (at + i < width) row[at + i] = f32_to_bf16(v[i]);
    }
}

__device__ __forceinline__ void big_store(float* __restrict__ row, int at, int width, const float (&v)[16]) {
    if (at + 16 <= width) {
#pragma unroll
        for (int h = 0; h < 4; ++h) *reinterpret_cast<float4*>(row + at + 4 * h) = make_float4(v[4 * h], v[4 * h + 1], v[4 * h + 2], v[4 * h + 3]);
    } else {
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if (at + i < width) row[at + i] = v[i];
    }
}

// x, w: the matrices' first rows and first column of the walk; x_row(i), w_row(i): the rows that are row i of the tile (of 64 NT
// and of 256); row_bytes from row to row in both.  acc[4 half + f][t][v], lane (r, g) of wave (wave_f, wave_t): token
// wave_t * 16 NT + 16 t + r, tile row 128 wave_f + 64 half + 16 g + 4 f + v.  TURNED: the walk begins at stage `turn` and wraps.
template <int NT, bool TURNED, class XRow, class WRow>
__device__ __forceinline__ void big_walk(char* lds, const void* x, const void* w, uint32_t row_bytes, int stages, int turn, XRow x_row, WRow w_row,
                                         f32x4 (&acc)[8][NT]) {
    constexpr int ROWS = BIG_FEAT + 64 * NT, STAGE = ROWS * BIG_ROW;
    constexpr int P = (64 * NT + 128) / 8 / BIG_WAVES, Q = 128 / 8 / BIG_WAVES;          // a wave's loads of each set
    static_assert(2 * STAGE <= 160 * 1024 && P * BIG_WAVES * 8 == 64 * NT + 128, "the stages fit LDS, the sets the waves");
    const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int wave_f = wave % 2, wave_t = wave / 2, r = lane % 16, g = lane / 16;
    const bool second = wave >= BIG_WAVES / 2;

    // ---- this wave's loads, 8 rows each: of set P the tokens and the first 64 features of each wave_f, of set Q the others
    uint32_t offset[P + Q], to[P + Q];
    const char* base[P + Q];
#pragma unroll
    for (int q = 0; q < P + Q; ++q) {
        const int id = q < P ? wave * P + q : wave * Q + q - P, w_id = q < P ? id - 8 * NT : id;
        const bool tokens = q < P && id < 8 * NT;
        const int R = tokens ? id * 8 : w_id / 8 * 128 + (q < P ? 0 : 64) + w_id % 8 * 8, row = R + lane / 8;
        const int chunk = (lane % 8) ^ (tokens ? big_x_swizzle(row) : big_w_swizzle(row));
        base[q] = reinterpret_cast<const char*>(tokens ? x : w);
        offset[q] = (uint32_t)(tokens ? x_row(row) : w_row(row)) * row_bytes + chunk * 16;
        to[q] = (uint32_t)((tokens ? BIG_FEAT : 0) + R) * BIG_ROW;
    }
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)lds);
    // (beyond the last stage the last one's rows again, for nobody: the waits count every wave's loads alike)
    auto stage_at = [&](int kt) __attribute__((always_inline)) {
        kt = min(kt, stages - 1);
        if (TURNED) kt = kt + turn < stages ? kt + turn : kt + turn - stages;
        return (size_t)kt * BIG_ROW;
    };
    auto bring_p = [&](int kt, int slot) __attribute__((always_inline)) {
        const size_t at = stage_at(kt);
#pragma unroll
        for (int q = 0; q < P; ++q) big_load(base[q] + at, offset[q], lds0 + slot * STAGE + to[q]);
    };
    auto bring_q = [&](int kt, int slot) __attribute__((always_inline)) {
        const size_t at = stage_at(kt);
#pragma unroll
        for (int q = P; q < P + Q; ++q) big_load(base[q] + at, offset[q], lds0 + slot * STAGE + to[q]);
    };

    // ---- the operands this lane reads: k-step i, chunk 4 i + g of its rows
    int wc[4][2], xc[2];
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int row = wave_f * 128 + big_feature_row(f, r);
            wc[f][i] = row * BIG_ROW + ((4 * i + g) ^ big_w_swizzle(row)) * 16;
        }
#pragma unroll
    for (int i = 0; i < 2; ++i) xc[i] = (BIG_FEAT + wave_t * 16 * NT + r) * BIG_ROW + ((4 * i + g) ^ big_x_swizzle(r)) * 16;
#pragma unroll
    for (int f = 0; f < 8; ++f)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[f][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    bf16x8 wf[2][4], xf[2][NT];
    auto read_tokens = [&](const char* stage) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t) xf[i][t] = *reinterpret_cast<const bf16x8*>(stage + xc[i] + t * 16 * BIG_ROW);
    };
    auto read_features = [&](const char* stage, int half) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int f = 0; f < 4; ++f) wf[i][f] = *reinterpret_cast<const bf16x8*>(stage + wc[f][i] + half * 64 * BIG_ROW);
    };
    auto multiply = [&](int half) __attribute__((always_inline)) {
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int f = 0; f < 4; ++f)
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[4 * half + f][t] = mfma_16x16x32(wf[i][f], xf[i][t], acc[4 * half + f][t]);
        __builtin_amdgcn_s_setprio(0);
    };

    // ---- the walk over K.  In steps of the first four waves (the others are one step later): 4 kt reads P of stage kt and asks
    // for Q of kt + 1 (whose place the others left at step 4 kt - 1), 4 kt + 1 multiplies, 4 kt + 2 reads Q of kt and asks for P
    // of kt + 2 (left at 4 kt + 1), 4 kt + 3 multiplies.  P of kt is read from step 4 kt on, Q from 4 kt + 2: each wave has waited
    // for its share, asked for six or four steps earlier with P + Q loads after it, before the barrier that ends the step before.
    bring_p(0, 0);
    bring_q(0, 0);
    bring_p(1, 1);
    all_but_the_youngest_have_arrived<P + Q>();
    big_swap();
    if (second) big_swap();
    for (int kt = 0; kt < stages; ++kt) {
        const int slot = kt & 1;
        const char* stage = lds + slot * STAGE;
        read_tokens(stage);
        read_features(stage, 0);
        bring_q(kt + 1, slot ^ 1);
        if (second) all_but_the_youngest_have_arrived<P + Q>();
        big_lds_reads_done();
        big_swap();
        multiply(0);
        if (!second) all_but_the_youngest_have_arrived<P + Q>();
        big_swap();
        read_features(stage, 1);
        bring_p(kt + 2, slot);
        if (second) all_but_the_youngest_have_arrived<P + Q>();
        big_lds_reads_done();
        big_swap();
        multiply(1);
        if (!second) all_but_the_youngest_have_arrived<P + Q>();
        big_swap();
    }
    if (!second) big_swap();
    all_but_the_youngest_have_arrived<0>();                  // nothing may land in LDS after the block's end
}
