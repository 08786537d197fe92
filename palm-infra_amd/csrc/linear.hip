// C[M, N] (+)= A[M, K] . W[N, K]^T with W in the checkpoint's [out, in] layout and 32-bit accumulation
// (kernels/matmul_dense.cpp:939-953 gives the semantics; the reference's GPU path calls a library
// with 32-bit compute, engine/cuda_matmul.cu:245-260).
//
// This is the exact path: no matrix-core mode of reduced precision.  Every output element adds its products in the same
// order of k whatever M and N are, so a row's result does not depend on how many rows are computed with it.  The sum goes
// in two levels, runs of SUM_RUN products and then the runs' sums: a 32-bit sum of K terms one after the other is off by
// about sqrt(K) roundings, which at K = 12288 and 36 layers adds up to more than 1e-4 on logits of order one; two levels
// leave sqrt(SUM_RUN) + sqrt(K / SUM_RUN).  Two kernels: linear_f32_kernel for float32 throughout, the float32 mode's
// products, on the matrix cores' 32-bit instruction; linear_tiled_kernel (plain FMA) for every mix of element types (a
// 32-bit matrix under bfloat16 activations) and for inner sizes that are not whole stages of it or beyond its offsets.
#include "lds_stage.h"

constexpr int TILE_M = 64, TILE_N = 64, TILE_K = 16;
constexpr int SUM_RUN = 256;          // products added one after the other before their sum joins the total
static_assert(SUM_RUN % TILE_K == 0, "a run is a whole number of tiles");

template <typename TA, typename TW, typename TC>
__global__ __launch_bounds__(256) void linear_tiled_kernel(const TA* __restrict__ A, const TW* __restrict__ W,
                                                          TC* __restrict__ C, int M, int N, int K, int accumulate) {
    // k-major tiles so that a thread's four rows (columns) are one 16-byte read
    __shared__ float As[TILE_K][TILE_M + 4];
    __shared__ float Ws[TILE_K][TILE_N + 4];
    const int tid = threadIdx.x;
    const int tx = tid % 16, ty = tid / 16;          // thread computes rows ty*4.., columns tx*4..
    const int m0 = blockIdx.y * TILE_M, n0 = blockIdx.x * TILE_N;
    const int lrow = tid / 4, lk = (tid % 4) * 4;    // what this thread loads: one row, four k
    float acc[4][4] = {}, total[4][4] = {};
    for (int k0 = 0; k0 < K; k0 += TILE_K) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = k0 + lk + j;
            const int m = m0 + lrow, n = n0 + lrow;
            As[lk + j][lrow] = (m < M && k < K) ? to_float(A[(size_t)m * K + k]) : 0.f;
            Ws[lk + j][lrow] = (n < N && k < K) ? to_float(W[(size_t)n * K + k]) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < TILE_K; ++k) {
            float a[4], w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) { a[i] = As[k][ty * 4 + i]; w[i] = Ws[k][tx * 4 + i]; }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], w[j], acc[i][j]);
        }
        if ((k0 + TILE_K) % SUM_RUN == 0 || k0 + TILE_K >= K) {      // the run is over: its sum joins the total
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) { total[i][j] += acc[i][j]; acc[i][j] = 0.f; }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + ty * 4 + i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + tx * 4 + j;
            if (n >= N) continue;
            float v = total[i][j];
            if (accumulate) v += to_float(C[(size_t)m * N + n]);
            C[(size_t)m * N + n] = from_float<TC>(v);
        }
    }
}

// ---- float32 throughout ---------------------------------------------------------------------------------------------
// v_mfma_f32_16x16x4: 32-bit operands, products and sums, at twice the rate of the vector units' FMA.  A wave's lane
// l = 16 g + r brings, of row r of each operand, the k-values 4 g .. 4 g + 3 of a run of 16 in one 16-byte read; instruction j
// of four takes element j of every lane.  The four waves of a block own the same 16 MT x 16 NT tile and a quarter of K each
// (stages of F32_STAGE values = a whole cache line a row, wave w the stages w, w + 4, ..), and no wave waits for another before
// the end, where LDS adds the four up in their order.  That split of K is the same for every M, N and tile: it is what keeps a
// row's result independent of its company.
// A stage goes from memory straight into a ring of the wave's own in LDS, whole lines (an instruction brings 8 rows x 128 bytes):
// read into registers the way the instruction wants it, 16 rows x 64 bytes, a compute unit gets 16 bytes a clock, which is what the
// products of 80 x 64 use up.  A row's eight 16-byte chunks are permuted by the row so that a read of 16 rows spreads over the banks;
// the next stage's operands are read from LDS while this one's products run.
// Bound: the matrix cores for many rows, the weight's bytes for few.  With operands read straight into registers and here:
// 157 x 24,576 x 4,096 311 and 245 us (129 TFLOP/s), 157 x 4,096 x 12,288 181 and 126, 91 x 24,576 x 4,096 227 and 156, one row of
// 151,936 x 4,096 494 and 430 (5.8 TB/s), of 24,576 x 4,096 90 and 75, of 4,096 x 12,288 38.5 and 37.3.  What is left of the 153
// TFLOP/s the library reaches: a compute unit gets some 45 GB/s from behind its die's L2, and tiles of 80 x 32 want 53.
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int F32_STAGE = 32, F32_WAVES = 4, F32_LINE = F32_STAGE * 4;
constexpr int F32_RUN = SUM_RUN / F32_STAGE;                         // a wave's own stages in a run

__device__ __forceinline__ int f32_swizzle(int row) { return (row >> 1) & 7; }

template <int MT, int NT, int DEPTH>
__global__ __launch_bounds__(F32_WAVES * WAVE) void linear_f32_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                                      float* __restrict__ C, int M, int N, int K, int accumulate) {
    constexpr int ROWS = 16 * (MT + NT), STAGE = ROWS * F32_LINE, LOADS = ROWS / 8;
    constexpr int RING = F32_WAVES * DEPTH * STAGE, PARTIAL = F32_WAVES * MT * NT * WAVE * 16;
    static_assert(RING <= 160 * 1024 && PARTIAL <= 160 * 1024 && (DEPTH - 1) * LOADS < 64, "the rings fit LDS, the waits the counter");
    __shared__ __attribute__((aligned(1024))) char lds[RING > PARTIAL ? RING : PARTIAL];
    const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), r = lane % 16, g = lane / 16;
    // blocks 8 apart run on one die: they are the row tiles of one tile of weights, which so passes through that die's L2 once
    const int tiles_m = (M + 16 * MT - 1) / (16 * MT);
    const int m0 = blockIdx.x / 8 % tiles_m * 16 * MT, n0 = (blockIdx.x / (8 * tiles_m) * 8 + blockIdx.x % 8) * 16 * NT;
    if (n0 >= N) return;                                             // (the launch is padded to whole groups of eight)
    const char* a_base = reinterpret_cast<const char*>(A + (size_t)m0 * K);
    const char* w_base = reinterpret_cast<const char*>(W + (size_t)n0 * K);
    uint32_t from[LOADS];                                            // bytes from the tile's first row (rows beyond the last: the last)
#pragma unroll
    for (int q = 0; q < LOADS; ++q) {
        const int row = q * 8 + lane / 8, chunk = (lane % 8) ^ f32_swizzle(row);
        from[q] = (uint32_t)(row < 16 * MT ? min(row, M - 1 - m0) : min(row - 16 * MT, N - 1 - n0)) * (uint32_t)(K * 4) + chunk * 16;
    }
    char* ring = lds + wave * DEPTH * STAGE;
    const uint32_t ring0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)ring);
    const int all_stages = K / F32_STAGE;
    const int stages = (all_stages - wave + F32_WAVES - 1) / F32_WAVES;             // of this wave
    // instructions [q0, q1) of stage s (beyond the last stage: values for nobody)
    auto bring = [&](int s, int q0, int q1) __attribute__((always_inline)) {
        const size_t at = (size_t)min(s * F32_WAVES + wave, all_stages - 1) * F32_LINE;
        const uint32_t to = ring0 + s % DEPTH * STAGE;
#pragma unroll
        for (int q = q0; q < q1; ++q) row_chunk_into_lds((q < 2 * MT ? a_base : w_base) + at, from[q], to + q * 1024);
    };
    f32x4 acc[MT][NT], total[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    struct Operands { f32x4 of[2][MT + NT]; };
    // pieces [p0, p1) of stage s: the first sixteen values of every row, then the others
    auto read = [&](int s, int p0, int p1, Operands& o) __attribute__((always_inline)) {
        const char* stage = ring + s % DEPTH * STAGE + r * F32_LINE;
#pragma unroll
        for (int p = p0; p < p1; ++p) {
            const int h = p / (MT + NT), row = p % (MT + NT);
            o.of[h][row] = *reinterpret_cast<const f32x4*>(stage + row * 16 * F32_LINE + ((4 * h + g) ^ f32_swizzle(r)) * 16);
        }
    };
    auto multiply = [&](const Operands& o, int h, int e) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.of[h][MT + j][e], o.of[h][i][e], acc[i][j], 0, 0, 0);
    };
    auto run_over = [&](int s) __attribute__((always_inline)) {
        if (s % F32_RUN != F32_RUN - 1) return;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) { total[i][j] += acc[i][j]; acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f}; }
    };
    // Step s, whose operands are in registers or on their way there: its products in eight groups, between which the wave asks memory for
    // stage s + DEPTH (its place in the ring is free once the operands are in registers) and LDS for the operands of stage s + 1 (which
    // has arrived when all but the DEPTH - 1 younger stages have).  Asked for in one go they keep the wave from issuing products.
    auto step = [&](int s, const Operands& now, Operands& next) __attribute__((always_inline)) {
#pragma unroll
        for (int group = 0; group < 8; ++group) {
            if (group == 1) lds_reads_done();
            if (group >= 1 && group <= 4) bring(s + DEPTH, LOADS * (group - 1) / 4, LOADS * group / 4);
            if (group == 5) { all_but_the_youngest_have_arrived<(DEPTH - 1) * LOADS>(); no_read_before_here(); }
            if (group >= 5) read(s + 1, LOADS * (group - 5) / 3, LOADS * (group - 4) / 3, next);
            multiply(now, group / 4, group % 4);
            __builtin_amdgcn_sched_barrier(0);
        }
        run_over(s);
    };
    Operands o[2];
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) bring(d, 0, LOADS);
    all_but_the_youngest_have_arrived<(DEPTH - 1) * LOADS>();
    no_read_before_here();
    read(0, 0, LOADS, o[0]);
    int s = 0;
    for (; s + 2 <= stages; s += 2) {
        step(s, o[0], o[1]);
        step(s + 1, o[1], o[0]);
    }
    if (s < stages) {
#pragma unroll
        for (int group = 0; group < 8; ++group) multiply(o[0], group / 4, group % 4);
        run_over(s);
    }
    all_but_the_youngest_have_arrived<0>();                  // nothing lands in LDS from here on
    __syncthreads();
    f32x4 (*partial)[MT * NT][WAVE] = reinterpret_cast<f32x4 (*)[MT * NT][WAVE]>(lds);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) partial[wave][i * NT + j][lane] = total[i][j] + acc[i][j];
    __syncthreads();
    // element v of a result tile: weight row 4 g + v of its sixteen, activation row r
    for (int t = wave; t < MT * NT; t += F32_WAVES) {
        const int m = m0 + 16 * (t / NT) + r, n = n0 + 16 * (t % NT) + 4 * g;
        const f32x4 sum = ((partial[0][t][lane] + partial[1][t][lane]) + partial[2][t][lane]) + partial[3][t][lane];
        if (m >= M) continue;
        float* c = C + (size_t)m * N + n;
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if (n + v < N) c[v] = accumulate ? sum[v] + c[v] : sum[v];
    }
}

template <int MT, int NT>
static void launch_f32(hipStream_t stream, const float* a, const float* w, float* c, int M, int N, int K, int accumulate) {
    // two blocks a compute unit where a block is small, else all of LDS for one (157 x 6,144: 66.7 us with half of it, 64.6 with all)
    constexpr int FIT = (MT == 1 || NT == 1 ? 80 : 160) * 1024 / (F32_WAVES * 16 * (MT + NT) * F32_LINE);
    constexpr int DEPTH = FIT > 4 ? 4 : FIT < 2 ? 2 : FIT;
    const int tiles_m = (M + 16 * MT - 1) / (16 * MT), tiles_n = (N + 16 * NT - 1) / (16 * NT);
    linear_f32_kernel<MT, NT, DEPTH><<<(tiles_n + 7) / 8 * 8 * tiles_m, F32_WAVES * WAVE, 0, stream>>>(a, w, c, M, N, K, accumulate);
}

constexpr int F32_MAX_TILES = 5;                     // 16-row tiles of a block: 80 rows
// A lane's row is an offset of 32 bits from its tile's first.  The limit is the highest tile's, whatever the tile of a call: a row's
// result does not depend on how many rows are computed with it.
constexpr int F32_MAX_K = (int)((1ll << 32) / (16 * F32_MAX_TILES * 4));

// The rows go in the fewest blocks of up to 80, of equal height (157 rows: two of 80).  How wide a block is: what takes the
// fewest rounds of 256 blocks times the work of one, its products and (0.7 of a product each) the operands it reads (157 x 6,144, K =
// 4,096: 64 us with 48 weight rows a block, 82 with 64).  Up to 16 rows the weight's bytes bound it: 16 weight rows a block, two blocks
// a compute unit (one row, 65,536 x 2,048: 88 us against 96 to 108 with more); 48 where there are blocks enough and the walk is long
// (16 rows, 24,576 x 4,096: 75 us against 86, one row 75 and 78).
static void dispatch_f32(hipStream_t stream, const float* a, const float* w, float* c, int M, int N, int K, int accumulate) {
    const int tiles = (M + 15) / 16, blocks_m = (tiles + F32_MAX_TILES - 1) / F32_MAX_TILES, mt = (tiles + blocks_m - 1) / blocks_m;
    int nt = N >= 256 * 48 && K >= 4096 ? 3 : 1;
    if (mt > 1) {
        double least = 1e300;
        for (int candidate : {4, 3, 2, 1}) {
            const long long blocks = (long long)((N + 16 * candidate - 1) / (16 * candidate)) * blocks_m;
            const double cost = (double)((blocks + 255) / 256) * (mt * candidate + 0.7 * (mt + candidate));
            if (cost < least) { least = cost; nt = candidate; }
        }
    }
#define PALM_F32_CASE(MT) case MT: \
        if (nt == 4) launch_f32<MT, 4>(stream, a, w, c, M, N, K, accumulate); \
        else if (nt == 3) launch_f32<MT, 3>(stream, a, w, c, M, N, K, accumulate); \
        else if (nt == 2) launch_f32<MT, 2>(stream, a, w, c, M, N, K, accumulate); \
        else launch_f32<MT, 1>(stream, a, w, c, M, N, K, accumulate); \
        break
    switch (mt) {
        case 1:
            if (nt == 3) launch_f32<1, 3>(stream, a, w, c, M, N, K, accumulate);
            else launch_f32<1, 1>(stream, a, w, c, M, N, K, accumulate);
            break;
        PALM_F32_CASE(2);
        PALM_F32_CASE(3);
        PALM_F32_CASE(4);
        PALM_F32_CASE(5);
    }
#undef PALM_F32_CASE
}

PALM_API int palm_linear(hipStream_t stream, const void* a, int a_dtype, const void* w, int w_dtype, void* c,
                         int c_dtype, int M, int N, int K, int accumulate) {
    PALM_CHECK(M >= 0 && N > 0 && K > 0, "linear: M=%d N=%d K=%d", M, N, K);
    if (M == 0) return 0;
    if (a_dtype == PALM_F32 && w_dtype == PALM_F32 && c_dtype == PALM_F32 && K % F32_STAGE == 0 && K <= F32_MAX_K &&
        ((uintptr_t)a | (uintptr_t)w) % 16 == 0 && M <= 65535 * 16) {
        dispatch_f32(stream, (const float*)a, (const float*)w, (float*)c, M, N, K, accumulate);
        PALM_LAUNCHED();
        return 0;
    }
    dim3 grid((N + TILE_N - 1) / TILE_N, (M + TILE_M - 1) / TILE_M);
    PALM_CHECK(grid.y <= 65535, "linear: M=%d is more than one launch takes (%d rows)", M, 65535 * TILE_M);
    PALM_DTYPE_SWITCH(a_dtype, TA, PALM_DTYPE_SWITCH(w_dtype, TW, PALM_DTYPE_SWITCH(c_dtype, TC,
        linear_tiled_kernel<TA, TW, TC><<<grid, 256, 0, stream>>>(
            (const TA*)a, (const TW*)w, (TC*)c, M, N, K, accumulate))));
    PALM_LAUNCHED();
    return 0;
}
