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
// 32-bit matrix under bfloat16 activations) and for inner sizes that are not whole stages of it.
#include "common.h"

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
// (stages of F32_STAGE values = a whole cache line a row, wave w the stages w, w + 4, ..), so operands go from memory straight
// into registers, DEPTH stages ahead, and no wave waits for another before the end, where LDS adds the four up in their order.
// That split of K is the same for every M, N and tile: it is what keeps a row's result independent of its company.
// Bound: the matrix cores for many rows, the weight's bytes for few.  With 157 rows:
// 24,576 x 4,096 in 312 us (101 TFLOP/s; 1,072 us with linear_tiled_kernel), 4,096 x 12,288 in 181 and 4,096 squared in 62
// (925, the mean of the two); one row of 4,096 x 12,288 in 40 us, 5.1 TB/s.
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int F32_STAGE = 32, F32_WAVES = 4;
constexpr int F32_RUN = SUM_RUN / F32_STAGE;                         // a wave's own stages in a run

template <int MT, int NT, int DEPTH>
__global__ __launch_bounds__(F32_WAVES * WAVE) void linear_f32_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                                      float* __restrict__ C, int M, int N, int K, int accumulate) {
    __shared__ f32x4 partial[F32_WAVES][MT * NT][WAVE];
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE, r = lane % 16, g = lane / 16;
    const int m0 = blockIdx.y * 16 * MT, n0 = blockIdx.x * 16 * NT;
    const float *a_row[MT], *w_row[NT];
#pragma unroll
    for (int i = 0; i < MT; ++i) a_row[i] = A + (size_t)min(m0 + 16 * i + r, M - 1) * K;
#pragma unroll
    for (int j = 0; j < NT; ++j) w_row[j] = W + (size_t)min(n0 + 16 * j + r, N - 1) * K;
    f32x4 acc[MT][NT], total[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int all_stages = (K + F32_STAGE - 1) / F32_STAGE;
    const int stages = (all_stages - wave + F32_WAVES - 1) / F32_WAVES;             // of this wave
    f32x4 a[DEPTH][MT][2], w[DEPTH][NT][2];
    auto bring = [&](int s, f32x4 (&av)[MT][2], f32x4 (&wv)[NT][2]) {               // (beyond the last stage: values for nobody)
        const int k = min((s * F32_WAVES + wave) * F32_STAGE, K - F32_STAGE) + 4 * g;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int i = 0; i < MT; ++i) av[i][h] = *reinterpret_cast<const f32x4*>(a_row[i] + k + 16 * h);
#pragma unroll
            for (int j = 0; j < NT; ++j) wv[j][h] = *reinterpret_cast<const f32x4*>(w_row[j] + k + 16 * h);
        }
    };
    auto multiply = [&](int s, const f32x4 (&av)[MT][2], const f32x4 (&wv)[NT][2]) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[j][h][e], av[i][h][e], acc[i][j], 0, 0, 0);
        if (s % F32_RUN == F32_RUN - 1) {                                           // the run is over: its sum joins the total
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) { total[i][j] += acc[i][j]; acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f}; }
        }
    };
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) bring(d, a[d], w[d]);
    int s0 = 0;
    for (; s0 + DEPTH <= stages; s0 += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            multiply(s0 + d, a[d], w[d]);
            bring(s0 + d + DEPTH, a[d], w[d]);
        }
    }
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d)
        if (s0 + d < stages) multiply(s0 + d, a[d], w[d]);
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
    constexpr int DEPTH = MT * NT <= 4 ? 4 : 2;      // few rows: the weight's reads in flight (8: no faster); many: the products hide two stages
    const dim3 grid((N + 16 * NT - 1) / (16 * NT), (M + 16 * MT - 1) / (16 * MT));
    linear_f32_kernel<MT, NT, DEPTH><<<grid, F32_WAVES * WAVE, 0, stream>>>(a, w, c, M, N, K, accumulate);
}

constexpr int F32_MAX_TILES = 5;                     // 16-row tiles of a block: 80 rows

// The rows go in the fewest blocks of up to 80, of equal height (157 rows: two of 80).  How wide a block is: what takes the
// fewest rounds of 256 blocks times the work of one, its products and (0.7 of a product each) the operands it reads.
// (157 rows x 6,144 columns, K = 4096: 192 blocks of 80 x 64 take 102 us, 768 of 80 x 16 136 us.)
static void dispatch_f32(hipStream_t stream, const float* a, const float* w, float* c, int M, int N, int K, int accumulate) {
    const int tiles = (M + 15) / 16, blocks_m = (tiles + F32_MAX_TILES - 1) / F32_MAX_TILES, mt = (tiles + blocks_m - 1) / blocks_m;
    int nt = 1;
    double least = 1e300;
    for (int candidate : {4, 2, 1}) {
        const long long blocks = (long long)((N + 16 * candidate - 1) / (16 * candidate)) * blocks_m;
        const double cost = (double)((blocks + 255) / 256) * (mt * candidate + 0.7 * (mt + candidate));
        if (cost < least) { least = cost; nt = candidate; }
    }
#define PALM_F32_CASE(MT) case MT: \
        if (nt == 4) launch_f32<MT, 4>(stream, a, w, c, M, N, K, accumulate); \
        else if (nt == 2) launch_f32<MT, 2>(stream, a, w, c, M, N, K, accumulate); \
        else launch_f32<MT, 1>(stream, a, w, c, M, N, K, accumulate); \
        break
    switch (mt) {
        PALM_F32_CASE(1);
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
    if (a_dtype == PALM_F32 && w_dtype == PALM_F32 && c_dtype == PALM_F32 && K % F32_STAGE == 0 && ((uintptr_t)a | (uintptr_t)w) % 16 == 0 && M <= 65535 * 16) {
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
