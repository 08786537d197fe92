// The walk over K of tiles of a product X . W^T that a block of four waves owns: 64 NT tokens (rows of X) x 256 rows of W,
// bfloat16, 32-bit sums, for the products of a prompt's rows and of many experts' rows.
//
// What bounds it is power: the chip's clock falls as its matrix cores are kept busy (8,192 cubed: 1.6 to 1.7 GHz at 1.2 million
// cycles, 87 % of which the matrix cores work).  So a wave owns 128 x 32 NT of a tile, 128 x 128 of the largest (its sums are the 256
// accumulator registers), which reads a third less from LDS than eight waves of 128 x 64 would; and since each wave is alone on its SIMD,
// it keeps its own matrix cores busy: an instruction goes out every four clocks, a product takes sixteen, and reads of LDS and
// loads stand between the products one at a time.  (8,192 cubed, on one card: eight waves in two fours that read and multiply in
// turn 742 us, this walk 717; with four reads or loads in a row between four products and four 790.)
//
// K goes by in stages of 64: rows of 128 bytes, a whole cache line, straight from memory into LDS (16 bytes a lane, an
// instruction fills 8 rows): two stages of W and three of X for the high tiles (160 KB), one more of each for the low ones, whose
// stages are over sooner (16 experts of 1,024 x 2,048, 17 rows: 65 us with two and three, 55).  A row's eight 16-byte chunks are permuted by
// the row's number so that the lanes that LDS serves together hit different banks; the lane that fills a place fetches the chunk
// that belongs there.
// A stage is four quarters of 4 x 2 NT products: features' first half and second half in the first k-step of 32, both again in the
// second.  Its operands of the second k-step are read in the first two quarters, those of the next stage's first k-step in the last
// two, each into the registers of the k-step that is not being multiplied.  So one barrier a stage, between them, is enough: before
// it a wave has read all of this stage and waited for its share of the next; behind it the places of this stage's W are asked
// for again at once (quarters three and four), those of X, which has a stage more, in the next stage's first two.
//
// Tiles follow each other without a stop: the loads run two (three) stages ahead, into the next tile's where a tile ends, and are on
// their way while its sums are stored.
#pragma once
#include "lds_stage.h"
#include "mfma.h"

#include <type_traits>

constexpr int BIG_K = 64, BIG_ROW = BIG_K * 2, BIG_WAVES = 4, BIG_THREADS = BIG_WAVES * WAVE;
constexpr int BIG_FEAT = 256, BIG_DIES = 8;
// stages that the loads run ahead: W has as many places in LDS, X one more
constexpr int big_ahead(int nt) { return nt <= 2 ? 3 : 2; }
constexpr int big_lds_bytes(int nt) { return (big_ahead(nt) * BIG_FEAT + (big_ahead(nt) + 1) * 64 * nt) * BIG_ROW; }

__device__ __forceinline__ void big_swap() {               // the block's barrier; loads stay on their way
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void big_lds_reads_done() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

__device__ __forceinline__ void big_multiply(f32x4& acc, bf16x8 a, bf16x8 b) {
    asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
template <int N, int I = 0, class F> __device__ __forceinline__ void big_each(F f) {
    if constexpr (I < N) { f(std::integral_constant<int, I>{}); big_each<N, I + 1>(f); }
}
// A lane of a result tile holds four features of one token.  Row 4 g + v of a wave's f-th of four tiles is feature
// 16 g + 4 f + v of their 64, so that a lane's four tiles are 16 features side by side.
__device__ __forceinline__ int big_feature_row(int f, int r) { return 16 * (r / 4) + 4 * f + r % 4; }
__device__ __forceinline__ int big_w_swizzle(int row) { return ((row >> 1) & 1) | ((row >> 3) & 6); }      // rows big_feature_row(f, 0 .. 15)
__device__ __forceinline__ int big_x_swizzle(int row) { return (row >> 1) & 7; }                           // 16 rows side by side

// 16 features of one token's row of the result, from feature `at`; rows are a multiple of eight long
__device__ __forceinline__ void big_store(bf16_t* __restrict__ row, int at, int width, const float (&v)[16]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = (uint32_t)f32_to_bf16(v[8 * h + 2 * i]).bits | ((uint32_t)f32_to_bf16(v[8 * h + 2 * i + 1]).bits << 16);
        if (at + 8 * h < width) *reinterpret_cast<uint4*>(row + at + 8 * h) = make_uint4(w[0], w[1], w[2], w[3]);
    }
}
__device__ __forceinline__ void big_store(float* __restrict__ row, int at, int width, const float (&v)[16]) {
#pragma unroll
    for (int h = 0; h < 4; ++h)
        if (at + 4 * h < width) *reinterpret_cast<float4*>(row + at + 4 * h) = make_float4(v[4 * h], v[4 * h + 1], v[4 * h + 2], v[4 * h + 3]);
}

// The sums of token tile t, taken from their registers no sooner than here (a tile's all at once would not fit the others).
template <int TT> __device__ __forceinline__ void big_column(f32x4 (&acc)[8][TT], int t, f32x4 (&a)[8]) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int f = 0; f < 8; ++f) {
        asm volatile("" : "+a"(acc[f][t]));
        a[f] = acc[f][t];
    }
}

// silu(gate) * up by the hardware's own 2^x and reciprocal, 32-bit and within some units of the last place: a wave alone on its SIMD has
// nothing to hide the library's 25 instructions behind (13,331 x 24,576 x 4,096 gated: 1,906 us with them, 1,847 so, 1,830 with 2^x and
// the reciprocal alone).  The argument of 2^x is rounded: what is lost there (6e-7 of e^-gate at -10, 4e-6 at -87) comes back as a factor
// 1 + rest, where 2^x is neither 0 nor infinite.  And the reciprocal is of a quarter of 1 + e^-gate, whose least value is still a normal number.
// The 32-bit values are off by at most 2.4e-7 of themselves (library: 1.8e-7), the bfloat16 results by the same 0.00166 to six digits.
__device__ __forceinline__ float big_silu_gated(float gate, float up) {
    const float turns = gate * -1.4426950408889634f, power = __builtin_amdgcn_exp2f(turns);
    const float rest = fmaf(turns, 1.9046543e-9f, fmaf(turns, -0.69314718246459961f, -gate));        // -gate - turns ln 2, ln 2 in two parts
    const float e = fabsf(turns) < 128.f ? fmaf(power, rest, power) : power;
    return 0.25f * gate * __builtin_amdgcn_rcpf(fmaf(e, 0.25f, 0.25f)) * up;
}

// One tile's walk: where its rows begin (first column of the walk), its stages, and the stage it begins with (it wraps around).
struct BigItem {
    const char* x;
    const char* w;
    int stages, turn;
    int x_rows, w_rows;           // rows that there are (beyond them the last one again)
    int live = 0;                 // (RAGGED) column tiles that a wave multiplies, of its TT
};

// items: how many tiles the block owns; make(i): the i-th's BigItem, the same in every lane; x_row(item, i), w_row(item, i): where row i
// of the tile lies, in rows from item.x or item.w (for tiles with the same x_rows and w_rows the same); row_bytes from row to row
// in both.  finish(i, acc, live): acc[4 half + f][t][v], lane (r, g) of wave (wave_f, wave_t) = (wave % 2, wave / 2): token
// wave_t * 32 NT + 16 t + r, tile row 128 wave_f + 64 half + 16 g + 4 f + v.
// RAGGED (of the high tiles): a tile's last column tiles may be nobody's.  They are neither read from LDS nor multiplied, each number of
// them in a loop of its own, from half a tile on (below that the loads of a stage have no products left to stand between).  finish gets their
// number as a constant, `live`: sums from acc[..][live] on were never set and are not to be read.
template <int NT, bool TURNED, bool RAGGED = false, class Make, class XRow, class WRow, class Finish>
__device__ __forceinline__ void big_walk(char* lds, uint32_t row_bytes, int items, Make make, XRow x_row, WRow w_row, Finish finish) {
    constexpr int TT = 2 * NT, W_STAGE = BIG_FEAT * BIG_ROW, X_STAGE = 64 * NT * BIG_ROW, A = big_ahead(NT);
    constexpr int XL = 2 * NT, WL = 8;                       // a wave's loads of a stage, 8 rows each
    static_assert(A * W_STAGE + (A + 1) * X_STAGE == big_lds_bytes(NT) && big_lds_bytes(NT) <= 160 * 1024, "the stages fit LDS");
    const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int wave_f = wave % 2, wave_t = wave / 2, r = lane % 16, g = lane / 16;

    // ---- the loads: a cursor that runs A stages ahead of the products
    uint32_t w_off[WL], x_off[XL];
    auto offsets_of = [&](const BigItem& item) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < WL; ++q) {
            const int row = (q * BIG_WAVES + wave) * 8 + lane / 8;
            w_off[q] = (uint32_t)w_row(item, row) * row_bytes + ((lane % 8) ^ big_w_swizzle(row)) * 16;
        }
#pragma unroll
        for (int q = 0; q < XL; ++q) {
            const int row = (q * BIG_WAVES + wave) * 8 + lane / 8;
            x_off[q] = (uint32_t)x_row(item, row) * row_bytes + ((lane % 8) ^ big_x_swizzle(row)) * 16;
        }
    };
    BigItem ahead = make(0);
    int ahead_item = 0, ahead_left = ahead.stages, ahead_wrap = ahead.stages - ahead.turn;
    size_t ahead_at = (size_t)ahead.turn * BIG_ROW;
    offsets_of(ahead);
    auto advance = [&]() __attribute__((always_inline)) {
        ahead_at += BIG_ROW;
        if (TURNED && --ahead_wrap == 0) ahead_at = 0;
        if (--ahead_left == 0) {
            if (ahead_item + 1 < items) {
                const int x_rows = ahead.x_rows, w_rows = ahead.w_rows;
                ahead = make(++ahead_item);
                ahead_left = ahead.stages;
                ahead_wrap = ahead.stages - ahead.turn;
                ahead_at = (size_t)ahead.turn * BIG_ROW;
                if (ahead.x_rows != x_rows || ahead.w_rows != w_rows) offsets_of(ahead);
            } else {                                         // beyond the last: its first stage again, for nobody
                ahead_left = 1;
                ahead_wrap = 0;
                ahead_at = 0;
            }
        }
    };
    // A load in two parts, with a product between them: where in LDS (m0 stands for an instruction before it is used), and the load.
    const uint32_t lds_w = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)lds) + wave * 8 * BIG_ROW;
    const uint32_t lds_x = lds_w + A * W_STAGE;
    auto place = [&](uint32_t stage, auto q) __attribute__((always_inline)) {
        asm volatile("s_add_u32 m0, %0, %1" : : "s"(stage), "i"(decltype(q)::value * BIG_WAVES * 8 * BIG_ROW) : "m0", "scc", "memory");
    };
    auto fetch = [&](const char* from, uint32_t offset) __attribute__((always_inline)) {
        asm volatile("global_load_lds_dwordx4 %0, %1" : : "v"(offset), "s"(from) : "memory");
    };
    // loads FROM .. FROM + COUNT of a stage's, over the gaps of a quarter
    auto w_loads = [&](int n, auto from, auto count, uint32_t stage, auto live) __attribute__((always_inline)) {
        big_each<decltype(count)::value>([&](auto j) __attribute__((always_inline)) {
            constexpr int q = decltype(from)::value + decltype(j)::value, gap = decltype(j)::value * (4 * decltype(live)::value) / decltype(count)::value;
            if (n == gap) place(stage, std::integral_constant<int, q>{});
            if (n == gap + 1) fetch(ahead.w + ahead_at, w_off[q]);
        });
    };
    auto x_loads = [&](int n, auto from, auto count, uint32_t stage, auto live) __attribute__((always_inline)) {
        big_each<decltype(count)::value>([&](auto j) __attribute__((always_inline)) {
            constexpr int q = decltype(from)::value + decltype(j)::value, gap = decltype(j)::value * (4 * decltype(live)::value) / decltype(count)::value;
            if (n == gap) place(stage, std::integral_constant<int, q>{});
            if (n == gap + 1) fetch(ahead.x + ahead_at, x_off[q]);
        });
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
    for (int i = 0; i < 2; ++i) xc[i] = (A * BIG_FEAT + wave_t * 32 * NT + r) * BIG_ROW + ((4 * i + g) ^ big_x_swizzle(r)) * 16;
#define BIG_C(v) std::integral_constant<int, (v)>{}

#pragma unroll
    for (int s = 0; s < A; ++s) {
        big_each<XL>([&](auto q) __attribute__((always_inline)) { place(lds_x + s * X_STAGE, q); asm volatile("s_nop 0"); fetch(ahead.x + ahead_at, x_off[q]); });
        big_each<WL>([&](auto q) __attribute__((always_inline)) { place(lds_w + s * W_STAGE, q); asm volatile("s_nop 0"); fetch(ahead.w + ahead_at, w_off[q]); });
        advance();
    }
    all_but_the_youngest_have_arrived<(A - 1) * (XL + WL)>();
    big_swap();
    uint32_t xs_before = A * X_STAGE, xs = 0, xs_next = X_STAGE, ws = 0, ws_next = W_STAGE;
    // (the sums and what is multiplied live inside: with RAGGED nothing but the cursor and the offsets is carried from one tile's walk to another's)
    auto tile = [&](int item, auto live) __attribute__((always_inline)) {
        f32x4 acc[8][TT];
        bf16x8 wf[2][2][4], xf[2][TT];                       // [half][k-step][tile], [k-step][tile]
        constexpr int LIVE = decltype(live)::value;
        auto read_w = [&](const char* stage, int i, int f) __attribute__((always_inline)) {
            wf[f / 4][i][f % 4] = *reinterpret_cast<const bf16x8*>(stage + wc[f % 4][i] + f / 4 * 64 * BIG_ROW);
        };
        auto read_x = [&](const char* stage, int i, int t) __attribute__((always_inline)) {
            xf[i][t] = *reinterpret_cast<const bf16x8*>(stage + xc[i] + t * 16 * BIG_ROW);
        };
        // a stage's reads, not before the first product (where the last quarter's are waited for) and not in the last few gaps
        auto w_reads = [&](int n, const char* stage, int i) __attribute__((always_inline)) {
#pragma unroll
            for (int f = 0; f < 8; ++f)
                if (n == 1 + f * (4 * LIVE) * 3 / 32) read_w(stage, i, f);
        };
        auto x_reads = [&](int n, const char* stage, int i) __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < LIVE; ++t)
                if (n == 1 + t * 7 / 2) read_x(stage, i, t);
        };
        auto quarter = [&](int half, int i, auto between) __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < LIVE; ++t)
#pragma unroll
                for (int f = 0; f < 4; ++f) {
                    between(4 * t + f);
                    big_multiply(acc[4 * half + f][t], wf[half][i][f], xf[i][t]);
                    __builtin_amdgcn_sched_barrier(0);
                }
        };
#pragma unroll
        for (int f = 0; f < 8; ++f)
#pragma unroll
            for (int t = 0; t < LIVE; ++t) {
                acc[f][t] = f32x4{0.f, 0.f, 0.f, 0.f};
                asm volatile("" : "+a"(acc[f][t]));
            }
        asm volatile("s_nop 7" ::: "memory");                // (the products are written out: their distance to what writes or reads the sums is kept here)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < LIVE; ++t) read_x(lds + xs, 0, t); // (read again behind another tile's end, which has better use for the registers)
#pragma unroll
        for (int f = 0; f < 8; ++f) read_w(lds + ws, 0, f);
        const int stages = make(item).stages;
        for (int kt = 0; kt < stages; ++kt) {
            quarter(0, 0, [&](int n) __attribute__((always_inline)) {
                w_reads(n, lds + ws, 1);
                x_loads(n, BIG_C(0), BIG_C(XL / 2), lds_x + xs_before, live);
            });
            quarter(1, 0, [&](int n) __attribute__((always_inline)) {
                x_reads(n, lds + xs, 1);
                x_loads(n, BIG_C(XL / 2), BIG_C(XL - XL / 2), lds_x + xs_before, live);
            });
            all_but_the_youngest_have_arrived<(A - 1) * XL + (A - 2) * WL>();
            big_lds_reads_done();
            big_swap();
            quarter(0, 1, [&](int n) __attribute__((always_inline)) {
                x_reads(n, lds + xs_next, 0);
                w_loads(n, BIG_C(0), BIG_C(WL / 2), lds_w + ws, live);
            });
            quarter(1, 1, [&](int n) __attribute__((always_inline)) {
                w_reads(n, lds + ws_next, 0);
                w_loads(n, BIG_C(WL / 2), BIG_C(WL / 2), lds_w + ws, live);
            });
            advance();
            xs_before = xs; xs = xs_next; ws = ws_next;
            xs_next = xs_next == A * X_STAGE ? 0 : xs_next + X_STAGE;
            ws_next = ws_next == (A - 1) * W_STAGE ? 0 : ws_next + W_STAGE;
        }
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        finish(item, acc, live);
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int item = 0; item < items; ++item) {
        if constexpr (RAGGED) {
            static_assert(TT == 8, "tiles of 256 rows");
            const int live = make(item).live;
            if (live >= 8) tile(item, BIG_C(8));
            else if (live == 7) tile(item, BIG_C(7));
            else if (live == 6) tile(item, BIG_C(6));
            else if (live == 5) tile(item, BIG_C(5));
            else tile(item, BIG_C(4));
        } else {
            tile(item, BIG_C(TT));
        }
    }
#undef BIG_C
    all_but_the_youngest_have_arrived<0>();                  // nothing may land in LDS after the block's end
}
