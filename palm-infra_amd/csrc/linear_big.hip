// C[M, N] = X[M, K] . W[N, K]^T for a prompt's rows: bfloat16 operands on the matrix cores, 32-bit accumulation, a bfloat16
// result; or, with the gated epilogue (W = gate rows over up rows), C[M, N / 2] = silu(X G^T) * (X U^T).  The product is the
// reference's matmul (kernels/matmul_dense.cpp:939-953), which its GPU path hands to a library (engine/cuda_matmul.cu:245-260).
//
// What bounds it is power (big_walk.h); 32 x 32 x 16 instructions cost more of it than 16 x 16 x 32 (twice the accumulator traffic),
// operands in 64-byte pieces more than in whole cache lines (twice the L2 requests).  8,192 cubed 705 us (736 with eight waves a
// block), the library 684; 13,331 x 24,576 x 4,096 gated 1,805 (1,959), the library and the activation's pass 1,952.
//
// A block owns tiles of 64 NT tokens x 256 features (big_walk.h), one after the other.  They are numbered so that the 32 blocks that run on one
// die at a time (blocks go to the eight dies in turn) own neighbouring tiles, 4 tiles of tokens x 8 of features: a die's L2
// reads a fifth of what the blocks ask for.
//
// The last round.  256 compute units take 256 tiles at a time; the tiles beyond the last full round are cut along K into
// ranges where that fills the chip, whose float32 tiles a second kernel adds up in their order (4,309 x 4,096, K = 12,288:
// 272 tiles, 305 us, the library 620).
#include "big_walk.h"

#include <hip/hip_runtime.h>

constexpr int BIG_UNITS = 256;

struct BigShape {
    int M, N, K;              // N: rows of W
    int inter;                // gated: features of the result (N / 2), else 0
    int tiles_t, tiles_f;
    int whole;                // tiles that one block owns; the others are cut into `split` ranges of K
    int split;
};

struct BigPlace {             // which tile, and where its rows and features start
    int t0, f0;
    template <int NT>
    __device__ static BigPlace of(const BigShape& s, int tile) {
        constexpr int GROUP = NT == 2 ? 8 : NT == 3 ? 5 : 4;       // tiles of tokens in a group: about 1,024 tokens
        const int in_group = GROUP * s.tiles_f, first = tile / in_group * GROUP, rows = min(GROUP, s.tiles_t - first);
        const int rest = tile % in_group;
        return BigPlace{(first + rest % rows) * 64 * NT, rest / rows};
    }
};

// One token tile's column of a lane's sums (both halves' four tiles) into the result.
template <bool GATED>
__device__ __forceinline__ void big_finish(const BigShape& s, bf16_t* __restrict__ C, int f0, int token, int wave_f, int g, const f32x4 (&a)[8]) {
    if (token >= s.M) return;
    if (GATED) {
        float v[16];
#pragma unroll
        for (int f = 0; f < 4; ++f)
#pragma unroll
            for (int x = 0; x < 4; ++x) v[4 * f + x] = big_silu_gated(a[f][x], a[4 + f][x]);
        big_store(C + (size_t)token * s.inter, f0 * 128 + wave_f * 64 + 16 * g, s.inter, v);
    } else {
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            float v[16];
#pragma unroll
            for (int f = 0; f < 4; ++f)
#pragma unroll
                for (int x = 0; x < 4; ++x) v[4 * f + x] = a[4 * half + f][x];
            big_store(C + (size_t)token * s.N, f0 * 256 + wave_f * 128 + half * 64 + 16 * g, s.N, v);
        }
    }
}

// Blocks: one for each compute unit.  A block takes every 32nd of its die's whole tiles, and one range of a cut tile if there is one left
// for it.
template <int NT, bool GATED>
__global__ __launch_bounds__(BIG_THREADS) __attribute__((amdgpu_waves_per_eu(1, 1))) void linear_big_kernel(
    const bf16_t* __restrict__ X, const bf16_t* __restrict__ W, bf16_t* __restrict__ C, const BigShape s, f32x4* __restrict__ partial) {
    __shared__ __attribute__((aligned(1024))) char lds[big_lds_bytes(NT)];
    const int block = blockIdx.x, stride = max(1, (int)gridDim.x / BIG_DIES), stages = s.K / BIG_K;
    const int per_die = (s.whole + BIG_DIES - 1) / BIG_DIES, first = block % BIG_DIES * per_die + block / BIG_DIES;
    const int last = min(s.whole, (block % BIG_DIES + 1) * per_die), mine = first < last ? (last - first + stride - 1) / stride : 0;
    const bool cut = block < (s.tiles_t * s.tiles_f - s.whole) * s.split;
    const int items = mine + cut;
    if (items == 0) return;
    auto tile_of = [&](int item) __attribute__((always_inline)) { return item < mine ? first + item * stride : s.whole + block / s.split; };
    const uint32_t row_bytes = (uint32_t)(s.K * 2);
    const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int wave_f = wave % 2, wave_t = wave / 2, r = lane % 16, g = lane / 16;
    big_walk<NT, false>(lds, row_bytes, items,
        [&](int item) __attribute__((always_inline)) {
            const BigPlace place = BigPlace::of<NT>(s, tile_of(item));
            const int from = place.f0 * (GATED ? 128 : BIG_FEAT);
            BigItem it{reinterpret_cast<const char*>(X + (size_t)place.t0 * s.K), reinterpret_cast<const char*>(W + (size_t)from * s.K), stages, 0,
                       min(64 * NT, s.M - place.t0), min(GATED ? 128 : BIG_FEAT, (GATED ? s.inter : s.N) - from)};
            if (item >= mine) {
                const int per = (stages + s.split - 1) / s.split, stage0 = block % s.split * per;
                it.x += (size_t)stage0 * BIG_ROW;
                it.w += (size_t)stage0 * BIG_ROW;
                it.stages = min(per, stages - stage0);
            }
            return it;
        },
        [&](const BigItem& it, int row) __attribute__((always_inline)) { return min(row, it.x_rows - 1); },
        [&](const BigItem& it, int row) __attribute__((always_inline)) {
            return GATED ? (row & 64 ? s.inter : 0) + min(row / 128 * 64 + row % 64, it.w_rows - 1) : min(row, it.w_rows - 1);
        },
        [&](int item, f32x4 (&acc)[8][2 * NT], auto live) __attribute__((always_inline)) {
            static_assert(decltype(live)::value == 2 * NT, "every column's sums are there");
            f32x4 a[8];
            if (item < mine) {
                const BigPlace place = BigPlace::of<NT>(s, tile_of(item));
#pragma unroll
                for (int t = 0; t < 2 * NT; ++t) {
                    big_column(acc, t, a);
                    big_finish<GATED>(s, C, place.f0, place.t0 + wave_t * 32 * NT + t * 16 + r, wave_f, g, a);
                }
            } else {                                         // the sums as they lie in the lanes: [block][t][f][thread]
                uint32_t at = block * 2 * NT * 8 * BIG_THREADS + threadIdx.x;
#pragma unroll
                for (int t = 0; t < 2 * NT; ++t) {
                    asm volatile("" : "+v"(at));             // (or the addresses of all of them are kept over the walk)
                    big_column(acc, t, a);
#pragma unroll
                    for (int f = 0; f < 8; ++f) partial[at + (t * 8 + f) * BIG_THREADS] = a[f];
                }
            }
        });
}

// A block for each (tile that was cut, token tile of its waves): the ranges' sums in their order, then as above.
template <int NT, bool GATED>
__global__ __launch_bounds__(BIG_THREADS) void linear_big_sum_kernel(bf16_t* __restrict__ C, const BigShape s, const f32x4* __restrict__ partial) {
    const int j = blockIdx.x / (2 * NT), t = blockIdx.x % (2 * NT);
    const BigPlace place = BigPlace::of<NT>(s, s.whole + j);
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    f32x4 a[8];
#pragma unroll
    for (int f = 0; f < 8; ++f) a[f] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int p = 0; p < s.split; ++p) {
        const f32x4* from = partial + ((size_t)(j * s.split + p) * 2 * NT + t) * 8 * BIG_THREADS + threadIdx.x;
#pragma unroll
        for (int f = 0; f < 8; ++f) a[f] += from[f * BIG_THREADS];
    }
    big_finish<GATED>(s, C, place.f0, place.t0 + wave / 2 * 32 * NT + t * 16 + lane % 16, wave % 2, lane / 16, a);
}

// ---- launch -----------------------------------------------------------------------------------------
struct BigPlan { int nt; BigShape shape; double cost; };

// Tiles of 256, 192 or 128 tokens, and into how many ranges of K the tiles beyond the last full round are cut: what takes least by
// this count of microseconds.  With the chip full a stage of a tile of 256 tokens takes 1.37 us (64 stages 95 us, 256 stages 362, a
// second tile of 64 stages 89), of 192 1.11, of 128 0.83 and, in some sizes, 1.0; the beginning and end of a tile that are not hidden 2.6;
// a sum kernel 6, and the float32 tiles cross memory twice, at 4.1 TB/s.  (At 360 products of 330 to 13,331 rows the tiles so chosen are
// 1.1 % behind the best of the three in the mean.)
static BigPlan big_plan(int M, int N, int K, bool gated) {
    BigPlan best{};
    best.cost = 1e300;
    const int stages = K / BIG_K;
    for (int nt : {4, 3, 2}) {
        BigShape s{};
        s.M = M; s.N = N; s.K = K; s.inter = gated ? N / 2 : 0;
        s.tiles_t = (M + 64 * nt - 1) / (64 * nt);
        s.tiles_f = gated ? (s.inter + 127) / 128 : (N + BIG_FEAT - 1) / BIG_FEAT;
        const long long tiles = (long long)s.tiles_t * s.tiles_f;
        if (tiles > 1 << 24) continue;
        const int rounds = (int)(tiles / BIG_UNITS), rest = (int)(tiles % BIG_UNITS);
        const double stage_us = nt == 4 ? 1.37 : nt == 3 ? 1.11 : 0.97;
        for (int split = 1; split <= 8; ++split) {
            if (split > 1 && (rest == 0 || rest * split > BIG_UNITS || stages / split < 8)) break;
            if (split > 1 && (split - 1) * ((stages + split - 1) / split) >= stages) continue;      // a range without stages
            const double last = rest == 0 ? 0.0 : (double)((stages + split - 1) / split) * stage_us + 2.6;
            const double sums = split == 1 ? 0.0 : 6.0 + (double)rest * split * nt * 16 * BIG_THREADS * 16 * 2 / 4.1e6;
            const double cost = rounds * (stages * stage_us + 2.6) + last + sums;
            if (cost < best.cost) {
                s.split = split;
                s.whole = split == 1 ? (int)tiles : rounds * BIG_UNITS;
                best = BigPlan{nt, s, cost};
            }
        }
    }
    return best;
}

// Whether this kernel takes the product: whole stages, rows that start on 16 bytes, offsets of 32 bits.
static bool big_takes(int M, int N, int K, bool gated) {
    return M > 0 && N > 0 && K >= 2 * BIG_K && K % BIG_K == 0 && N % (gated ? 16 : 8) == 0 && (long long)M * K < (1ll << 31) - 8 * K &&
           (long long)N * K < (1ll << 31) - 8 * K;
}
PALM_API int palm_linear_big_takes(int M, int N, int K, int gated) { return big_takes(M, N, K, gated != 0); }
// 64-token pieces of a tile, times 16, and into how many ranges of K the last tiles are cut (1: not); 0 where it does not take the product
PALM_API int palm_linear_big_plan(int M, int N, int K, int gated) {
    if (!big_takes(M, N, K, gated != 0)) return 0;
    const BigPlan p = big_plan(M, N, K, gated != 0);
    return p.nt * 16 + p.shape.split;
}
// bytes of workspace for the tiles that are cut (0: none are)
PALM_API long long palm_linear_big_work(int M, int N, int K, int gated) {
    if (!big_takes(M, N, K, gated != 0)) return 0;
    const BigPlan p = big_plan(M, N, K, gated != 0);
    const long long tiles = (long long)p.shape.tiles_t * p.shape.tiles_f;
    return p.shape.split == 1 ? 0 : (tiles - p.shape.whole) * p.shape.split * p.nt * 16 * BIG_THREADS * 16;
}

template <int NT, bool GATED>
static int launch_big(hipStream_t stream, const void* x, const void* w, void* c, const BigShape& s, void* work) {
    const int tiles = s.tiles_t * s.tiles_f, cut = tiles - s.whole;
    const int blocks = min(BIG_UNITS, max((s.whole + BIG_DIES - 1) / BIG_DIES * BIG_DIES, cut * s.split));
    BigShape shape = s;
    linear_big_kernel<NT, GATED><<<blocks, BIG_THREADS, 0, stream>>>((const bf16_t*)x, (const bf16_t*)w, (bf16_t*)c, shape, (f32x4*)work);
    PALM_LAUNCHED();
    if (cut) {
        linear_big_sum_kernel<NT, GATED><<<cut * 2 * NT, BIG_THREADS, 0, stream>>>((bf16_t*)c, shape, (const f32x4*)work);
        PALM_LAUNCHED();
    }
    return 0;
}

// x [M, K], w [N, K], c [M, N] (gated: [M, N / 2]), all bfloat16; work: palm_linear_big_work bytes.
PALM_API int palm_linear_big(hipStream_t stream, const void* x, const void* w, void* c, int M, int N, int K, int gated, void* work, long long work_bytes) {
    PALM_CHECK(M >= 0 && N > 0 && K > 0, "linear_big: M=%d N=%d K=%d", M, N, K);
    if (M == 0) return 0;
    PALM_CHECK(big_takes(M, N, K, gated != 0), "linear_big: M=%d N=%d K=%d (gated %d) is not a product of whole stages and 16-byte rows", M, N, K, gated);
    PALM_CHECK(((uintptr_t)x | (uintptr_t)w | (uintptr_t)c | (uintptr_t)work) % 16 == 0, "linear_big: operands must be 16-byte aligned");
    const long long needed = palm_linear_big_work(M, N, K, gated);
    PALM_CHECK(needed == 0 || (work && work_bytes >= needed), "linear_big: %lld bytes of workspace where %lld are needed", work_bytes, needed);
    const BigPlan p = big_plan(M, N, K, gated != 0);
    if (p.nt == 3) return gated ? launch_big<3, true>(stream, x, w, c, p.shape, work) : launch_big<3, false>(stream, x, w, c, p.shape, work);
    if (p.nt == 4) return gated ? launch_big<4, true>(stream, x, w, c, p.shape, work) : launch_big<4, false>(stream, x, w, c, p.shape, work);
    return gated ? launch_big<2, true>(stream, x, w, c, p.shape, work) : launch_big<2, false>(stream, x, w, c, p.shape, work);
}
