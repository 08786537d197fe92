// Products of 17 to 48 rows: the stream of linear_ring.h with two or three column tiles.  Every fragment of weights meets all rows,
// whose activations stay in registers (a tile takes 16 a super-step: three tiles hold four steps, two hold six).  They come through the
// ring: read into registers 16 rows x 64 bytes at a time the 390 KB of 48 rows took a compute unit ten microseconds.  (linear_mid.hip
// brings the rows through LDS beside the weights, for every 64 or 128 weight rows again.)
// Us, that kernel and this one, 17 / 32 / 48 rows: 24,576 x 4,096 gated 36 36 36 and 35 36 38, 34,816 x 5,120 gated (up to 32 rows) 81 84
// and 58 60, 6,144 x 4,096 13 14 14 and 11 12 13, 4,096 x 12,288 20 21 22 and 20 20 20; 4,096 x 4,096 with the norm after it 15 and 10 to 13 (before the
// weights' loads of both were marked as read once).
// (In a file of its own: a program loads a file's kernels when it first runs one of them, which takes milliseconds for these.)
#include "linear_ring.h"

PALM_API int palm_linear_ring_parts(int M, int N, int K, int epilogue, int planes_ok);
constexpr int RING_MANY_ROWS = 48;
static int ring_many_steps(int M) { return M <= 32 ? 6 : 4; }

// Into how many ranges of K the product is cut, each a whole number of steps for every wave that fits the registers: what gives the
// blocks the fewest steps, then the fewest ranges; only one where the result has to come whole.  0: not served.
PALM_API int palm_linear_ring_parts(int M, int N, int K, int epilogue, int planes_ok) {
    if (M <= 16 || M > RING_MANY_ROWS || N <= 0 || K <= 0 || K % (SUPER_K * RING_WAVES) != 0) return 0;
    if (epilogue == EPI_SWIGLU && N % 2 != 0) return 0;
    if ((double)RING_MANY_ROWS * K * 2 >= 2.0e9 || (double)RING_MANY_ROWS * N * 4 >= 2.0e9) return 0;          // (offsets of 32 bits)
    const int steps = K / (SUPER_K * RING_WAVES), strips = epilogue == EPI_SWIGLU ? (N / 2 + 7) / 8 : (N + 15) / 16;
    int best = 0, best_work = 1 << 30;
    for (int parts = 1; parts <= (planes_ok && epilogue == EPI_STORE ? 4 : 1); ++parts) {
        if (steps % parts != 0 || steps / parts > ring_many_steps(M)) continue;
        const int slots = RING_UNITS / parts, work = (strips + slots - 1) / slots * (steps / parts);
        if (work < best_work) { best = parts; best_work = work; }
    }
    return best;
}

template <int CT, bool ONCE, typename TC, int EPI>
static void dispatch_ring_many(hipStream_t stream, const void* a, const void* w, void* c, int M, int N, int K, int parts, int steps,
                               const RowNorm& norm) {
    if (steps == 1) launch_ring<3, 1, CT, ONCE, TC, EPI>(stream, a, w, c, M, N, K, parts, steps, norm);
    else if (steps == 2) launch_ring<3, 2, CT, ONCE, TC, EPI>(stream, a, w, c, M, N, K, parts, steps, norm);
    else if (steps == 3) launch_ring<3, 3, CT, ONCE, TC, EPI>(stream, a, w, c, M, N, K, parts, steps, norm);
    else if (steps == 4) launch_ring<3, 4, CT, ONCE, TC, EPI>(stream, a, w, c, M, N, K, parts, steps, norm);
    else if constexpr (CT == 2) {
        if (steps == 5) launch_ring<3, 5, CT, ONCE, TC, EPI>(stream, a, w, c, M, N, K, parts, steps, norm);
        else launch_ring<3, 6, CT, ONCE, TC, EPI>(stream, a, w, c, M, N, K, parts, steps, norm);
    }
}
template <bool ONCE, typename TC, int EPI>
static void dispatch_ring_tiles(hipStream_t stream, const void* a, const void* w, void* c, int M, int N, int K, int parts, const RowNorm& norm) {
    const int steps = K / (SUPER_K * RING_WAVES) / parts;
    if (M <= 32) dispatch_ring_many<2, ONCE, TC, EPI>(stream, a, w, c, M, N, K, parts, steps, norm);
    else dispatch_ring_many<3, ONCE, TC, EPI>(stream, a, w, c, M, N, K, parts, steps, norm);
}

// As palm_linear_thin, for 17 to 48 rows: parts as palm_linear_ring_parts says (1 with the gated epilogue or a norm that is folded into what follows).
PALM_API int palm_linear_ring(hipStream_t stream, const void* a, const void* w, void* c, int c_dtype, int M, int N, int K, int epilogue,
                              int parts, const float* ss_in, int pieces_in, float eps_in, float* resid, const float* w_out, float* ss_out) {
    RowNorm norm{ss_in, pieces_in, eps_in, K, resid, w_out, ss_out};
    const bool once = epilogue & EPI_ONCE;
    epilogue &= ~EPI_ONCE;
    PALM_CHECK(epilogue == EPI_STORE || epilogue == EPI_SWIGLU, "linear_ring: epilogue %d", epilogue);
    PALM_CHECK(parts >= 1 && parts == palm_linear_ring_parts(M, N, K, epilogue, parts > 1), "linear_ring: %d rows, %d x %d in %d ranges are not served", M, N, K, parts);
    PALM_CHECK(!ss_in || pieces_in > 0, "linear_ring: %d pieces of the rows' sums of squares", pieces_in);
    PALM_CHECK(!resid || (epilogue == EPI_STORE && parts == 1 && c_dtype == PALM_BF16 && w_out && ss_out),
               "linear_ring: adding to the residual stream needs a plain bfloat16 product in one plane, the next norm's weight and room for the "
               "sums of squares");
    PALM_CHECK(parts == 1 || c_dtype == PALM_F32, "linear_ring: planes of partial sums are float32");
    PALM_CHECK(((uintptr_t)a | (uintptr_t)w) % 16 == 0, "linear_ring: operands must be 16-byte aligned");
    if (epilogue == EPI_SWIGLU) {
        PALM_DTYPE_SWITCH(c_dtype, TC, (once ? dispatch_ring_tiles<true, TC, EPI_SWIGLU> : dispatch_ring_tiles<false, TC, EPI_SWIGLU>)(stream, a, w, c, M, N, K, parts, norm));
    } else {
        PALM_DTYPE_SWITCH(c_dtype, TC, (once ? dispatch_ring_tiles<true, TC, EPI_STORE> : dispatch_ring_tiles<false, TC, EPI_STORE>)(stream, a, w, c, M, N, K, parts, norm));
    }
    PALM_LAUNCHED();
    return 0;
}
