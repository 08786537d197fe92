// Causal grouped-query attention over the paged cache, for prompts and for single tokens, any head
// size, all arithmetic in 32-bit with full-precision exp.  This is the exact path (the float32 mode)
// and the fallback for head sizes that the matrix-core kernels do not take.
//
// Semantics (models/qwen3.py:336-341; kernels/attention.cpp:937-962; engine/input_prep.cpp:8-15):
// head h reads kv head h / (nh / nkv); s_j = scale * q . k_j for the keys j <= p of the query's own
// sequence (and j > p - window if there is a window); softmax with the running maximum subtracted;
// o = sum_j p_j v_j.  The keys of the step's own tokens are already in the cache when this runs.
// K is [pages, nkv, 64, hd]; V is kept transposed, [pages, nkv, hd, 64].
//
// One block of four waves per (query, up to HEADS heads of a kv head).  A wave takes every fourth page of the key range; inside
// a page each lane scores one key for each of the heads, the wave keeps their running (max, sum, output) and the four partial
// results are merged at the end.  What is computed for a head, and in which order, does not depend on HEADS.
#include "common.h"

constexpr int ATT_WAVES = 4;
constexpr int ATT_MAX_HD = 512;
// (query, head) pairs, every sequence counted as the longest, from which a block takes four heads: below, the chip has room for a block
// each.  Us, one and four heads a block, 32 heads of 128 on eight: 544 pairs 6.0 and 9.2 (17 queries of a prompt), 1,024 448 and 57 (32 sequences
// of 900), 1,280 12.2 and 10.6, 5,024 64 and 30.  Groups of three heads (24 on eight), whose fourth is computed for nobody: 960 pairs 8.8 and 10.1, 1,536
// 17.8 and 11.7, 3,768 51 and 29; of five (40 on eight), two blocks: 1,280 13.3 and 10.2, 1,600 13.5 and 11.2, 6,280 77 and 44.  Ragged steps: a prompt of 20 beside
// seven sequences of 500 101 and 51, of 8 beside fifteen 315 and 176; where all is short a few microseconds either way (17, 1 and 1 tokens 6.1 and 9.4;
// 40, 7, 7, 7 and 7 16.1 and 10.7).
constexpr long long SIMPLE_SHARED_FROM = 1024;

// Four consecutive elements, widened.
__device__ inline float4 four_floats(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ inline float4 four_floats(const bf16_t* p) {
    const uint2 u = *reinterpret_cast<const uint2*>(p);
    return make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16), __uint_as_float(u.y & 0xffff0000u));
}

// A lane's value of `p`, the same lane's in every lane.
__device__ inline float of_lane(float p, int lane) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(p), lane)); }

// ACC: head elements that a lane holds, hd <= 64 ACC.  What bounds it is the reads of a page, a row a lane: each instruction
// meets 64 cache lines, so it should bring what it can of them, and what it brings should serve all heads of the group.  FOURS
// (hd a multiple of 4): K and V in pieces of four elements, the products in the same order.  (157 queries x 32 heads of 128 on
// eight kv heads, float32: 31 us, 66 with a block for each head, 201 an element at a time.)
template <typename T, int ACC, bool FOURS, int HEADS>
__global__ __launch_bounds__(ATT_WAVES * WAVE) void attention_simple_kernel(
    const T* __restrict__ q, const T* __restrict__ k_cache, const T* __restrict__ v_cache,
    const int* __restrict__ block_table, int max_pages, const int* __restrict__ seq_slot,
    const int* __restrict__ seq_start, const int* __restrict__ seq_new, const int* __restrict__ cu_new,
    int nh, int nkv, int hd, float scale, int window, T* __restrict__ out) {
    __shared__ __attribute__((aligned(16))) float q_s[HEADS][ACC * WAVE];
    __shared__ float m_s[HEADS][ATT_WAVES], l_s[HEADS][ATT_WAVES];
    __shared__ float acc_s[HEADS][ATT_WAVES][ACC * WAVE];

    const int qi = blockIdx.x, b = blockIdx.z;
    if (qi >= seq_new[b]) return;
    const int G = nh / nkv, per_group = (G + HEADS - 1) / HEADS;
    const int g = blockIdx.y / per_group, first = blockIdx.y % per_group * HEADS;
    const int h0 = g * G + first, heads = min(HEADS, G - first);      // (heads that there are not: the last one again, not kept)
    const int t = cu_new[b] + qi;
    const int pos = seq_start[b] + qi;
    const int lo = window > 0 ? max(0, pos - window + 1) : 0;
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    const int* pages = block_table + (size_t)seq_slot[b] * max_pages;

#pragma unroll
    for (int x = 0; x < HEADS; ++x) {
        const T* qp = q + ((size_t)t * nh + h0 + min(x, heads - 1)) * hd;
        for (int d = threadIdx.x; d < hd; d += blockDim.x) q_s[x][d] = to_float(qp[d]);
    }
    __syncthreads();

    float m[HEADS], l[HEADS], acc[HEADS][ACC];
#pragma unroll
    for (int x = 0; x < HEADS; ++x) {
        m[x] = -INFINITY;
        l[x] = 0.f;
#pragma unroll
        for (int i = 0; i < ACC; ++i) acc[x][i] = 0.f;
    }

    for (int pg = lo / PAGE_TOKENS + wave; pg <= pos / PAGE_TOKENS; pg += ATT_WAVES) {
        const int page = pages[pg];
        const T* kp = k_cache + ((size_t)page * nkv + g) * PAGE_TOKENS * hd;
        const T* vp = v_cache + ((size_t)page * nkv + g) * PAGE_TOKENS * hd;
        const int j = pg * PAGE_TOKENS + lane;
        const bool seen = j >= lo && j <= pos;
        float dot[HEADS], p[HEADS];
#pragma unroll
        for (int x = 0; x < HEADS; ++x) dot[x] = 0.f;
        if (seen) {
            const T* kr = kp + (size_t)lane * hd;
            if constexpr (FOURS) {
#pragma unroll 8
                for (int d = 0; d < hd; d += 4) {
                    const float4 kd = four_floats(kr + d);
#pragma unroll
                    for (int x = 0; x < HEADS; ++x) {
                        const float4 qd = *reinterpret_cast<const float4*>(&q_s[x][d]);
                        dot[x] = fmaf(qd.x, kd.x, dot[x]);
                        dot[x] = fmaf(qd.y, kd.y, dot[x]);
                        dot[x] = fmaf(qd.z, kd.z, dot[x]);
                        dot[x] = fmaf(qd.w, kd.w, dot[x]);
                    }
                }
            } else {
                for (int d = 0; d < hd; ++d) {
                    const float kd = to_float(kr[d]);
#pragma unroll
                    for (int x = 0; x < HEADS; ++x) dot[x] = fmaf(q_s[x][d], kd, dot[x]);
                }
            }
        }
#pragma unroll
        for (int x = 0; x < HEADS; ++x) {
            const float s = seen ? dot[x] * scale : -INFINITY;
            const float m_new = fmaxf(m[x], wave_max(s));
            const float alpha = expf(m[x] - m_new);     // m = -inf at the first page: exp(-inf) = 0
            p[x] = expf(s - m_new);                     // an invisible key: exp(-inf) = 0
            l[x] = l[x] * alpha + wave_sum(p[x]);
            m[x] = m_new;
#pragma unroll
            for (int i = 0; i < ACC; ++i) acc[x][i] *= alpha;
        }
        const int j_first = max(lo, pg * PAGE_TOKENS) - pg * PAGE_TOKENS;
        const int j_last = min(pos, pg * PAGE_TOKENS + PAGE_TOKENS - 1) - pg * PAGE_TOKENS;
        // keys that are not seen have weight 0, and what lies at their places is not read; jj is the same in every lane
        // (the weights come from all lanes, so before a lane leaves one out)
        auto one_key = [&](int jj) {
            float w[HEADS];
#pragma unroll
            for (int x = 0; x < HEADS; ++x) w[x] = of_lane(p[x], jj);
#pragma unroll
            for (int i = 0; i < ACC; ++i) {
                const int d = lane + i * WAVE;
                if (d >= hd) continue;
                const float vd = to_float(vp[(size_t)d * PAGE_TOKENS + jj]);
#pragma unroll
                for (int x = 0; x < HEADS; ++x) acc[x][i] = fmaf(w[x], vd, acc[x][i]);
            }
        };
        int jj = j_first;
        if constexpr (FOURS) {
            for (; jj <= j_last && jj % 4 != 0; ++jj) one_key(jj);
#pragma unroll 4
            for (; jj + 3 <= j_last; jj += 4) {
                float w[HEADS][4];
#pragma unroll
                for (int x = 0; x < HEADS; ++x)
#pragma unroll
                    for (int e = 0; e < 4; ++e) w[x][e] = of_lane(p[x], jj + e);
#pragma unroll
                for (int i = 0; i < ACC; ++i) {
                    const int d = min(lane + i * WAVE, hd - 1);
                    const float4 vd = four_floats(vp + (size_t)d * PAGE_TOKENS + jj);
#pragma unroll
                    for (int x = 0; x < HEADS; ++x) {
                        acc[x][i] = fmaf(w[x][0], vd.x, acc[x][i]);
                        acc[x][i] = fmaf(w[x][1], vd.y, acc[x][i]);
                        acc[x][i] = fmaf(w[x][2], vd.z, acc[x][i]);
                        acc[x][i] = fmaf(w[x][3], vd.w, acc[x][i]);
                    }
                }
            }
        }
        for (; jj <= j_last; ++jj) one_key(jj);
    }

#pragma unroll
    for (int x = 0; x < HEADS; ++x) {
        if (lane == 0) { m_s[x][wave] = m[x]; l_s[x][wave] = l[x]; }
#pragma unroll
        for (int i = 0; i < ACC; ++i) {
            const int d = lane + i * WAVE;
            if (d < hd) acc_s[x][wave][d] = acc[x][i];
        }
    }
    __syncthreads();
    for (int x = 0; x < heads; ++x) {
        float m_all = -INFINITY;
        for (int w = 0; w < ATT_WAVES; ++w) m_all = fmaxf(m_all, m_s[x][w]);
        float l_all = 0.f;
        for (int w = 0; w < ATT_WAVES; ++w) l_all += l_s[x][w] * expf(m_s[x][w] - m_all);
        T* op = out + ((size_t)t * nh + h0 + x) * hd;
        for (int d = threadIdx.x; d < hd; d += blockDim.x) {
            float o = 0.f;
            for (int w = 0; w < ATT_WAVES; ++w) o += acc_s[x][w][d] * expf(m_s[x][w] - m_all);
            op[d] = from_float<T>(o / l_all);
        }
    }
}

PALM_API int palm_attention_simple(hipStream_t stream, const void* q, int dtype, const void* k_cache,
                                   const void* v_cache, const int* block_table, int max_pages, const int* seq_slot,
                                   const int* seq_start, const int* seq_new, const int* cu_new, int n_seqs,
                                   int max_new, int nh, int nkv, int hd, float scale, int window, void* out) {
    PALM_CHECK(n_seqs >= 0 && max_new >= 0 && nh > 0 && nkv > 0 && hd > 0,
               "attention: seqs=%d max_new=%d heads=%d kv=%d hd=%d", n_seqs, max_new, nh, nkv, hd);
    PALM_CHECK(nh % nkv == 0, "attention: %d heads are not a multiple of %d kv heads", nh, nkv);
    PALM_CHECK(hd <= ATT_MAX_HD, "attention: head_dim %d exceeds %d", hd, ATT_MAX_HD);
    PALM_CHECK(window >= 0, "attention: window %d", window);
    PALM_CHECK(max_pages > 0, "attention: max_pages %d", max_pages);
    if (n_seqs == 0 || max_new == 0) return 0;
    PALM_CHECK(nh <= 65535 && n_seqs <= 65535, "attention: %d heads / %d sequences are more than one launch takes", nh, n_seqs);
    // Four heads of a kv head a block (two where it has no more) where the blocks still fill the chip several times over.
    const int G = nh / nkv;
    const bool shared = G > 1 && hd <= 2 * WAVE && (long long)max_new * nh * n_seqs >= SIMPLE_SHARED_FROM;
    const int heads = !shared ? 1 : G > 2 ? 4 : 2;
    dim3 grid(max_new, nkv * ((G + heads - 1) / heads), n_seqs);
#define PALM_SIMPLE(ACC, FOURS, HEADS) attention_simple_kernel<T, ACC, FOURS, HEADS><<<grid, ATT_WAVES * WAVE, 0, stream>>>( \
        (const T*)q, (const T*)k_cache, (const T*)v_cache, block_table, max_pages, seq_slot, seq_start, seq_new, \
        cu_new, nh, nkv, hd, scale, window, (T*)out)
    const bool fours = hd % 4 == 0 && ((uintptr_t)k_cache | (uintptr_t)v_cache) % 16 == 0;
    if (!fours) grid.y = nh;
    PALM_DTYPE_SWITCH(dtype, T,
        if (!fours) PALM_SIMPLE(ATT_MAX_HD / WAVE, false, 1);
        else if (hd <= WAVE) { if (heads == 4) PALM_SIMPLE(1, true, 4); else if (heads == 2) PALM_SIMPLE(1, true, 2); else PALM_SIMPLE(1, true, 1); }
        else if (hd <= 2 * WAVE) { if (heads == 4) PALM_SIMPLE(2, true, 4); else if (heads == 2) PALM_SIMPLE(2, true, 2); else PALM_SIMPLE(2, true, 1); }
        else if (hd <= 4 * WAVE) PALM_SIMPLE(4, true, 1);
        else PALM_SIMPLE(8, true, 1));
#undef PALM_SIMPLE
    PALM_LAUNCHED();
    return 0;
}
