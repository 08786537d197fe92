// Products of up to 16 rows and a long K: which of the stream's kernels (linear_ring.h) serves.
// (Weights that pass once and weights that the caches keep have a file each: a program loads a file's kernels when it first runs one of them, which takes
// milliseconds for these, and a model has one kind.)
#pragma once
#include "linear_ring.h"

// Steps whose activations stay in registers: as many as a wave makes (a step beyond K takes a slot of the ring and a turn: K =
// 5,120 in six steps instead of its five, 16 rows: 7,168 features 19.0 us and 17.7, 5,120 17.4 and 16.2, gated 34,816 66.4 and
// 65.8).  Not 12 for K = 12,288: 48 pieces a lane to wait for before the first product, 23.4 us against 19.7 beside the weights.
template <bool ONCE, typename TC, int EPI>
static void dispatch_ring(hipStream_t stream, const void* a, const void* w, void* c, int M, int N, int K, int parts, int steps,
                          const RowNorm& norm) {
    if (steps <= 2) launch_ring<4, 2, 1, ONCE, TC, EPI>(stream, a, w, c, M, N, K, parts, steps, norm);
    else if (steps <= 3) launch_ring<4, 3, 1, ONCE, TC, EPI>(stream, a, w, c, M, N, K, parts, steps, norm);
    else if (steps <= 4) launch_ring<4, 4, 1, ONCE, TC, EPI>(stream, a, w, c, M, N, K, parts, steps, norm);
    else if (steps <= 5) launch_ring<4, 5, 1, ONCE, TC, EPI>(stream, a, w, c, M, N, K, parts, steps, norm);
    else if (steps <= 6) launch_ring<4, 6, 1, ONCE, TC, EPI>(stream, a, w, c, M, N, K, parts, steps, norm);
    else if (steps <= 7) launch_ring<4, 7, 1, ONCE, TC, EPI>(stream, a, w, c, M, N, K, parts, steps, norm);
    else if (steps <= 8) launch_ring<4, 8, 1, ONCE, TC, EPI>(stream, a, w, c, M, N, K, parts, steps, norm);
    else launch_ring<2, 0, 1, ONCE, TC, EPI>(stream, a, w, c, M, N, K, parts, steps, norm);
}

template <bool ONCE>
static void launch_linear_ring_of(hipStream_t stream, const void* a, const void* w, void* c, int c_dtype, int M, int N, int K,
                                  int epilogue, int parts, int steps, const RowNorm& norm) {
    if (epilogue == EPI_SWIGLU) {
        if (c_dtype == PALM_BF16) dispatch_ring<ONCE, bf16_t, EPI_SWIGLU>(stream, a, w, c, M, N, K, 1, steps, norm);
        else dispatch_ring<ONCE, float, EPI_SWIGLU>(stream, a, w, c, M, N, K, 1, steps, norm);
    } else {
        if (c_dtype == PALM_BF16) dispatch_ring<ONCE, bf16_t, EPI_STORE>(stream, a, w, c, M, N, K, parts, steps, norm);
        else dispatch_ring<ONCE, float, EPI_STORE>(stream, a, w, c, M, N, K, parts, steps, norm);
    }
}
