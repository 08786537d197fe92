// Differential attention for prompts on the matrix cores, bfloat16, compiled for one padded key size and one padded
// value size (PALM_DIFF_KK: key size / 32 rounded up; PALM_DIFF_VT: value size / 16 rounded up).
//
// A block of four waves shares the pages of one key/value head: the waves take up to four of the query heads that read it, or runs of
// queries of one head; a wave owns 16 queries of one head and both of its score maps.  A page of 64 keys (the rows of both maps, and
// the transposed values) goes from memory straight into LDS, the next one on its way while this one is used where two fit; 16-byte
// chunks are permuted by the row so that an operand's reads spread over the banks (the lane that fills a place fetches the chunk that
// belongs there).  With a wave reading its pages for itself 64 KB came through the vector cache for 16 queries (16 heads, key size 128,
// values 256: 587 us for 2,048 tokens and 5,365 for 7,600); from LDS they come once for the block's 64 or 128 (101 and 691 us, 1,030
// TFLOP/s), and what bounds it is LDS, the matrix cores and the exponentials in turn.  (Two tiles of queries a wave: the outputs of two
// maps spill, 359 us for 2,048 tokens.)
//
// For every page a wave computes the transposed scores S^T = K Q^T (keys down, queries across), so that a lane's four results of
// a tile are four keys of ONE query: the softmax statistics of a query then live in the lanes of its column.  Which key is a
// tile's row is free: rows are dealt so that the eight weights a lane holds of 32 keys are neighbouring keys, and then the second
// product O^T += V^T P^T takes them as its B operand as they are, its A operand being one 16-byte read of a value row that serves both
// maps.  Scores leave the matrix cores as 32-bit sums; maximum, exponentials (base 2: the scores are scaled by scale * log2 e), sums,
// the combination a1 - lambda a2 and the unit norm are 32-bit; the weights are rounded to bfloat16 for the second product, whose sums
// are 32-bit again.  A query's weights are taken against a reference that follows its maximum only when that has risen by more than
// 2^REFERENCE_SLACK, so the outputs are seldom rescaled.
//
// Layouts as in attention_diff.hip: K [pages, 2 kv_heads, 64, dim], V [pages, kv_heads, vdim, 64].
#include "lds_stage.h"
#include "mfma.h"

#ifndef PALM_DIFF_KK
#error "compile with -DPALM_DIFF_KK=<ceil(key size / 32)> -DPALM_DIFF_VT=<ceil(value size / 16)>"
#endif

PALM_DEFINE_LAST_ERROR()

constexpr int KK = PALM_DIFF_KK;
constexpr int VT = PALM_DIFF_VT;
constexpr int K_CHUNKS = KK * 4;                               // 16-byte chunks of a key's row in LDS
constexpr int K_BYTES = 2 * PAGE_TOKENS * K_CHUNKS * 16, V_BYTES = VT * 16 * PAGE_TOKENS * 2, DM_STAGE = K_BYTES + V_BYTES;
constexpr int K_LOADS = K_BYTES / 1024, V_LOADS = V_BYTES / 1024;      // instructions that bring a page's keys and values (all waves)
constexpr int STAGES = 2 * DM_STAGE <= 160 * 1024 ? 2 : 1;
constexpr int COMPUTE_UNITS = 256;
constexpr float REFERENCE_SLACK = 8.f;                         // weights stay below 2^8, far within 32 bits and bfloat16's range

PALM_API int palm_attention_diff_mfma_sizes(int which) { return which == 0 ? KK * 32 : VT * 16; }

// By what a key row's chunks are permuted: of the eight rows that a read of an operand takes at once (rows 8 a + b, b < 4, for
// two neighbouring a), those that begin in the same bank get different places.
__device__ inline int key_swizzle(int row) {
    return KK % 2 == 0 ? (row & 3) | ((row >> 1) & 4) : ((row >> 1) & 1) | ((row >> 2) & 2);
}

__device__ inline bf16x8 load_row8(const bf16_t* row, int col, int dim) {
    // eight values of a row from column `col`; columns beyond `dim` are zero (dim is a multiple of eight).  The read
    // itself is unconditional (of the row's last eight values where the column lies beyond it): no branch around it
    const bf16x8 v = load_bf16x8(row + min(col, dim - 8));
    return col < dim ? v : zero_bf16x8();
}

template <int DM_WAVES>
__global__ __launch_bounds__(DM_WAVES * WAVE) void attention_diff_mfma_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
    const int* __restrict__ block_table, int max_pages, const int* __restrict__ seq_slot,
    const int* __restrict__ seq_start, const int* __restrict__ seq_new, const int* __restrict__ cu_new, int n_seqs, int tiles,
    int heads, int kv_heads, int heads_a_block, int dim, int vdim, float scale, float lambda, float gain, float eps, bf16_t* __restrict__ out) {
    __shared__ __attribute__((aligned(1024))) char lds[STAGES * DM_STAGE];
    // One after the other: the groups of heads of all sequences, then the next earlier tile of queries.  So blocks are handed out by
    // how far into its sequence a tile lies, which is how long it takes, the longest first; and with a few groups in all a die
    // meets the keys of some of them only.
    const int lists = heads / heads_a_block;
    const int which = blockIdx.x % (n_seqs * lists), tile = tiles - 1 - blockIdx.x / (n_seqs * lists);
    const int b = which / lists;
    const int n_new = seq_new[b];
    const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int runs = DM_WAVES / heads_a_block;                  // runs of queries in the block
    const int block_q0 = tile * runs * 16;
    if (block_q0 >= n_new) return;
    const int per_kv = heads / kv_heads, groups = per_kv / heads_a_block;
    const int kvh = which % lists / groups;
    const int h = kvh * per_kv + which % lists % groups * heads_a_block + wave / runs;
    const int q0 = block_q0 + wave % runs * 16;                 // the wave's first query (beyond the run: it only brings pages)
    const int r = lane % 16, g = lane / 16;
    const int start = seq_start[b];
    const int qi = min(q0 + r, n_new - 1);                      // a column beyond the run repeats the last query and stores nothing
    const int qpos = start + qi;
    const int seq_last = start + n_new - 1;
    const int first_pos = start + q0;
    const int last_page = q0 < n_new ? (start + min(q0 + 15, n_new - 1)) / PAGE_TOKENS : -1;
    const int block_last = __builtin_amdgcn_readfirstlane((start + min(block_q0 + runs * 16 - 1, n_new - 1)) / PAGE_TOKENS);
    const float scale2 = scale * 1.4426950408889634f;
    const int* pages = block_table + (size_t)seq_slot[b] * max_pages;

    // what this lane brings of every page: instruction i of the block fills 1 KB of the stage
    constexpr int K_MINE = K_LOADS / DM_WAVES;
    static_assert(K_LOADS % DM_WAVES == 0, "a page's keys are a whole number of instructions a wave");
    int k_off[K_MINE];
#pragma unroll
    for (int i = 0; i < K_MINE; ++i) {
        const int place = (i * DM_WAVES + wave) * WAVE + lane, row = place / K_CHUNKS;
        k_off[i] = row * dim + min(((place % K_CHUNKS) ^ key_swizzle(row)) * 8, dim - 8);     // (columns beyond the key meet zeros of the query)
    }
    constexpr int V_MINE = (V_LOADS + DM_WAVES - 1) / DM_WAVES;
    int v_off[V_MINE];
#pragma unroll
    for (int i = 0; i < V_MINE; ++i) {
        const int place = (i * DM_WAVES + wave) * WAVE + lane, row = place / 8;
        v_off[i] = min(row, vdim - 1) * PAGE_TOKENS + ((place % 8) ^ (row & 7)) * 8;
    }
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)lds);
    auto bring = [&](int pg, int stage) {
        const size_t head = (size_t)pages[pg] * kv_heads + kvh;
        const bf16_t* kp = k_cache + head * 2 * PAGE_TOKENS * dim;                            // the rows of both maps, one after the other
        const bf16_t* vp = v_cache + head * vdim * PAGE_TOKENS;
        const uint32_t to = __builtin_amdgcn_readfirstlane(lds0 + stage * DM_STAGE);
#pragma unroll
        for (int i = 0; i < K_MINE; ++i) row_chunk_into_lds(kp + k_off[i], to + (i * DM_WAVES + wave) * 1024);
#pragma unroll
        for (int i = 0; i < V_MINE; ++i)
            if (i * DM_WAVES + wave < V_LOADS) row_chunk_into_lds(vp + v_off[i], to + K_BYTES + (i * DM_WAVES + wave) * 1024);
    };

    // the queries, as the B operand: column r, eight values of group g for each step of 32 over the key size
    bf16x8 qf[2][KK];
    const bf16_t* qr = q + (((size_t)cu_new[b] + qi) * heads + h) * 2 * dim;
    f32x4 acc[2][VT];
    float ref[2], l[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) qf[m][kk] = load_row8(qr + m * dim, kk * 32 + g * 8, dim);
        ref[m] = -INFINITY; l[m] = 0.f;
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) acc[m][vt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    all_but_the_youngest_have_arrived<0>();                     // (the queries: nothing else of this wave is on its way from here on)
    if (STAGES == 2) bring(0, 0);
    for (int pg = 0; pg <= block_last; ++pg) {
        char* page = lds + (STAGES == 2 ? (pg & 1) * DM_STAGE : 0);
        if (STAGES == 1) {
            __syncthreads();                                    // everyone is done with the page before
            bring(pg, 0);
        }
        all_but_the_youngest_have_arrived<0>();
        __syncthreads();                                        // every wave's share of the page; and (two stages) everyone is done with the one before
        if (STAGES == 2 && pg < block_last) bring(pg + 1, (pg + 1) & 1);
        // on the page that holds the sequence's last key the values beyond it are made zero: their weights are zero, but pages are
        // handed out uncleared and zero times a stale NaN is NaN
        const int beyond = seq_last - pg * PAGE_TOKENS;
        if (beyond < PAGE_TOKENS - 1) {
            for (int i = threadIdx.x; i < VT * 16 * 8; i += DM_WAVES * WAVE) {
                const int row = i / 8, key0 = ((i % 8) ^ (row & 7)) * 8;
                bf16_t* at = reinterpret_cast<bf16_t*>(page + K_BYTES) + i * 8;
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (key0 + e > beyond) at[e].bits = 0;
            }
            __syncthreads();
        }
        if (pg > last_page) continue;                           // (the same in all lanes of the wave)
        const bool edge = pg * PAGE_TOKENS + PAGE_TOKENS - 1 > first_pos;      // the page reaches beyond some query of the wave
        bf16x8 pf[2][2];                                        // the weights as B operands: [map][32 keys]
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            f32x4 s[4];
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                const int row = m * PAGE_TOKENS + 32 * (n / 2) + 8 * (r / 4) + 4 * (n & 1) + (r & 3);
                const char* kr = page + row * (K_CHUNKS * 16);
                const int swizzle = key_swizzle(row);
                s[n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kk = 0; kk < KK; ++kk) {
                    const bf16x8 kf = *reinterpret_cast<const bf16x8*>(kr + ((4 * kk + g) ^ swizzle) * 16);
                    s[n] = mfma_16x16x32(kf, qf[m][kk], s[n]);
                }
            }
            // lane (r, g) holds the keys 32 (n / 2) + 8 g + 4 (n % 2) + i of query r; scores in units of log2: a weight is one exp2 away
            float top = -INFINITY;
            if (edge) {
#pragma unroll
                for (int n = 0; n < 4; ++n)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int j = pg * PAGE_TOKENS + 32 * (n / 2) + 8 * g + 4 * (n & 1) + i;
                        s[n][i] = j <= qpos ? s[n][i] * scale2 : -INFINITY;
                        top = fmaxf(top, s[n][i]);
                    }
            } else {
#pragma unroll
                for (int n = 0; n < 4; ++n)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        s[n][i] *= scale2;
                        top = fmaxf(top, s[n][i]);
                    }
            }
            if (__ballot(top > ref[m] + REFERENCE_SLACK)) {          // some query's maximum has risen far (or: the first page)
                top = fmaxf(top, __shfl_xor(top, 16, WAVE));
                top = fmaxf(top, __shfl_xor(top, 32, WAVE));
                const float now = top > ref[m] + REFERENCE_SLACK ? top : ref[m];      // finite from the first page on: key 0 is visible to all
                const float alpha = __builtin_amdgcn_exp2f(ref[m] - now);
                ref[m] = now;
                l[m] *= alpha;
#pragma unroll
                for (int vt = 0; vt < VT; ++vt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[m][vt][i] *= alpha;
            }
            float sum = 0.f;
#pragma unroll
            for (int n = 0; n < 4; ++n)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    s[n][i] = __builtin_amdgcn_exp2f(s[n][i] - ref[m]);
                    sum += s[n][i];
                }
            l[m] += sum;                                    // this lane's part; the groups are added at the end
#pragma unroll
            for (int half = 0; half < 2; ++half)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    pf[m][half][i] = (__bf16)s[2 * half][i];
                    pf[m][half][4 + i] = (__bf16)s[2 * half + 1][i];
                }
        }
        // O^T += V^T P^T: row r of a value tile, the same eight keys of group g as the weights hold
        const char* vr = page + K_BYTES + r * 128;
#pragma unroll
        for (int vt = 0; vt < VT; ++vt)
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const bf16x8 vf = *reinterpret_cast<const bf16x8*>(vr + vt * 2048 + ((4 * half + g) ^ (r & 7)) * 16);
                acc[0][vt] = mfma_16x16x32(vf, pf[0][half], acc[0][vt]);
                acc[1][vt] = mfma_16x16x32(vf, pf[1][half], acc[1][vt]);
            }
    }
    // lane (r, g) holds value dimensions 16 vt + 4 g + i of query r
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        l[m] += __shfl_xor(l[m], 16, WAVE);
        l[m] += __shfl_xor(l[m], 32, WAVE);
    }
    const float f0 = 1.0f / l[0], f1 = lambda / l[1];
    float ss = 0.f;
#pragma unroll
    for (int vt = 0; vt < VT; ++vt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float o = acc[0][vt][i] * f0 - acc[1][vt][i] * f1;
            acc[0][vt][i] = o;
            if (16 * vt + 4 * g + i < vdim) ss += o * o;
        }
    ss += __shfl_xor(ss, 16, WAVE);
    ss += __shfl_xor(ss, 32, WAVE);
    const float inv = gain / sqrtf(ss / (float)vdim + eps);
    if (q0 + r >= n_new) return;
    bf16_t* op = out + (((size_t)cu_new[b] + qi) * heads + h) * vdim;
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) {
        const int vd = 16 * vt + 4 * g;
        if (vd < vdim) {                                        // vdim is a multiple of four
            uint2 w;
            w.x = (uint32_t)f32_to_bf16(acc[0][vt][0] * inv).bits | ((uint32_t)f32_to_bf16(acc[0][vt][1] * inv).bits << 16);
            w.y = (uint32_t)f32_to_bf16(acc[0][vt][2] * inv).bits | ((uint32_t)f32_to_bf16(acc[0][vt][3] * inv).bits << 16);
            *reinterpret_cast<uint2*>(op + vd) = w;
        }
    }
}

struct DiffPlan {
    int heads_a_block, waves;
    long long lists;                          // groups of heads of all sequences
    int tiles;                                // of queries
};
// Eight waves a block bring a page for twice as many queries, and two waves a SIMD take turns; four leave more blocks.  Eight win where
// their blocks fill the compute units: in more than one round where a unit holds one block of either kind (128 and 256 elements, 16
// heads: 3,000 tokens 144 us against 224 with four, 7,600: 691 and 1,209, 8 prompts of 300: 30 and 40; 1,000 tokens 55 and 50), in
// two where it holds two of four waves (64 and 128: 4,096 tokens 131 us against 151, 3,000: 90 and 87, 300: 15 and 13).  Key sizes
// beyond 128 keep four: the registers of a lane.
static DiffPlan diff_plan(int n_seqs, int max_new, int heads, int kv_heads) {
    const int per_kv = heads / kv_heads, heads_a_block = per_kv % 4 == 0 ? 4 : per_kv % 2 == 0 ? 2 : 1;
    const long long lists = (long long)n_seqs * (heads / heads_a_block);
    auto tiles = [&](int waves) { const int run = waves / heads_a_block * 16; return (max_new + run - 1) / run; };
    const bool eight = KK <= 4 && lists * tiles(8) >= (2 * STAGES * DM_STAGE > 160 * 1024 ? COMPUTE_UNITS + 1 : 2 * COMPUTE_UNITS);
    const int waves = eight ? 8 : 4;
    return DiffPlan{heads_a_block, waves, lists, tiles(waves)};
}
PALM_API int palm_attention_diff_mfma_waves(int n_seqs, int max_new, int heads, int kv_heads) { return diff_plan(n_seqs, max_new, heads, kv_heads).waves; }

PALM_API int palm_attention_diff_mfma(hipStream_t stream, const void* q, const void* k_cache, const void* v_cache,
                                      const int* block_table, int max_pages, const int* seq_slot, const int* seq_start,
                                      const int* seq_new, const int* cu_new, int n_seqs, int max_new, int heads, int kv_heads,
                                      int dim, int vdim, float scale, float lambda, float gain, float eps, void* out) {
    PALM_CHECK(n_seqs >= 0 && max_new >= 0 && heads > 0 && kv_heads > 0 && dim > 0 && vdim > 0,
               "attention_diff_mfma: seqs=%d max_new=%d heads=%d kv=%d dim=%d vdim=%d", n_seqs, max_new, heads, kv_heads, dim, vdim);
    PALM_CHECK(heads % kv_heads == 0, "attention_diff_mfma: %d heads are not a multiple of %d kv heads", heads, kv_heads);
    PALM_CHECK(dim % 8 == 0 && dim <= KK * 32 && dim > (KK - 1) * 32, "attention_diff_mfma: built for key sizes %d..%d in steps of 8, not %d",
               (KK - 1) * 32 + 8, KK * 32, dim);
    PALM_CHECK(vdim % 4 == 0 && vdim <= VT * 16 && vdim > (VT - 1) * 16, "attention_diff_mfma: built for value sizes %d..%d in steps of 4, not %d",
               (VT - 1) * 16 + 4, VT * 16, vdim);
    PALM_CHECK(max_pages > 0, "attention_diff_mfma: max_pages %d", max_pages);
    if (n_seqs == 0 || max_new == 0) return 0;
    const DiffPlan p = diff_plan(n_seqs, max_new, heads, kv_heads);
    PALM_CHECK(p.lists * p.tiles < (1ll << 31), "attention_diff_mfma: %d heads / %d sequences of %d tokens are more than one launch takes", heads, n_seqs, max_new);
#define DIFF_LAUNCH(WAVES) attention_diff_mfma_kernel<WAVES><<<(unsigned)(p.lists * p.tiles), WAVES * WAVE, 0, stream>>>( \
        (const bf16_t*)q, (const bf16_t*)k_cache, (const bf16_t*)v_cache, block_table, max_pages, seq_slot, seq_start, seq_new, cu_new, \
        n_seqs, p.tiles, heads, kv_heads, p.heads_a_block, dim, vdim, scale, lambda, gain, eps, (bf16_t*)out)
    if constexpr (KK <= 4) {
        if (p.waves == 8) {
            DIFF_LAUNCH(8);
            PALM_LAUNCHED();
            return 0;
        }
    }
    DIFF_LAUNCH(4);
#undef DIFF_LAUNCH
    PALM_LAUNCHED();
    return 0;
}
