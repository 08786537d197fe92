// Products of up to 16 rows and a long K, weights that pass once (linear_ring_thin.h).
#include "linear_ring_thin.h"

void launch_linear_ring_once(hipStream_t stream, const void* a, const void* w, void* c, int c_dtype, int M, int N, int K,
                             int epilogue, int parts, int steps, const RowNorm& norm) {
    launch_linear_ring_of<true>(stream, a, w, c, c_dtype, M, N, K, epilogue, parts, steps, norm);
}
