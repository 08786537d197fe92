// Routed experts for many rows (a prompt), planned on the device: the (token, choice) pairs are grouped by expert, and two
// grouped products on the matrix cores run all experts' rows in one launch each.
//
//   plan      count the pairs of every expert; pad every expert's run of pairs to whole tiles of rows and lay the
//             runs one after the other; place every pair in its run, in no particular order (a slot is a column of the
//             products by itself: no result depends on where in its run a pair lies); the slots that pad a run hold -1
//   grouped   for every tile (its expert comes from the plan): mid = silu(G_e x) * (U_e x) for the tile's rows x, then
//             y = D_e mid.  The weights are the first operand of the matrix instruction, so that a lane ends with
//             neighbouring features of one row.  Sizes in whole cache lines: blocks of 64 to 256 rows x 256 weight rows through
//             LDS (moe_big_kernel).  Otherwise a wave owns 32 features x 64 rows and reads its fragments from memory itself (a
//             weight fragment feeds four products, a row fragment two or four)
//   combine   out[t] = sum_c weight[t, c] * y[place of pair (t, c)], in the order of c, 32-bit, plus up to two rows that other
//             branches made and float32 planes of another (a shared expert's).  y is bfloat16, or float32 where the caller asks
//             for results that are rounded nowhere before the sum, as those of the kernels for few rows are
#include "big_walk.h"
#include "expert_form.h"

constexpr int GT_TOKENS = 64;                     // rows of a tile whose fragments come from memory
constexpr int GT_RUNS = GT_TOKENS / 16;           // runs of 16 rows: what one matrix instruction takes
constexpr int GT_WAVES = 4;
constexpr int GT_FEATURES = 32 * GT_WAVES;        // features of a block's tile
constexpr int PLAN_THREADS = 1024;
constexpr int PLAN_MAX_EXPERTS = 512;

__device__ inline bf16x8 grouped_row8(const bf16_t* row, int col, int dim) {
    // eight values of a row from column `col`; columns beyond `dim` are zero (dim is a multiple of eight); the read itself
    // is unconditional
    const bf16x8 v = load_bf16x8(row + min(col, dim - 8));
    return col < dim ? v : zero_bf16x8();
}

// What the plan says of a tile: its expert and how many of its slots are pairs, in one number; -1 beyond the last tile
constexpr int TILE_EXPERT_BITS = 10;
static_assert(PLAN_MAX_EXPERTS <= 1 << TILE_EXPERT_BITS, "an expert's number and a tile's rows in one int");
__device__ __forceinline__ int tile_expert_of(int t) { return t & ((1 << TILE_EXPERT_BITS) - 1); }
__device__ __forceinline__ int tile_rows_of(int t) { return t >> TILE_EXPERT_BITS; }
// Rows of each of an expert's tiles but the last.  Tiles of 256 rows that may stop early (moe_big_kernel) share up to 768 rows evenly, in whole
// steps of 32 (what a column tile of each of a tile's two waves of rows holds), so that no compute unit gets a full one and another little.  Filled one
// after the other, two tiles multiply up to 33 % more (257 rows: 384 and 288), three up to 18 % (513: 640 and 544), four would up to 12, five 9: not
// measured there.  Other tiles are filled one after the other.
__device__ __forceinline__ int rows_per_tile(int rows, int tile) {
    const int tiles = (rows + tile - 1) / tile;
    return tile == 256 && tiles >= 1 && tiles <= 3 ? ((rows + tiles - 1) / tiles + 31) / 32 * 32 : tile;
}

// One block.  starts[e] = first slot of expert e's run (runs padded to whole tiles); tile_expert[i]: see above; slot_pair[slot] = pair (-1 where a run is padded), pair_slot[pair] = slot.  The choices are rows [n, top], or with
// ids the rows of a table [vocab, top] that the tokens' ids pick.
__global__ __launch_bounds__(PLAN_THREADS) void moe_plan_kernel(const int* __restrict__ chosen, const int* __restrict__ ids, int vocab, int top,
                                                                int n_pairs, int experts, int max_tiles, int tile,
                                                                int* __restrict__ tile_expert, int* __restrict__ slot_pair,
                                                                int* __restrict__ pair_slot, int* __restrict__ used) {
    __shared__ int start_s[PLAN_MAX_EXPERTS + 1], cursor_s[PLAN_MAX_EXPERTS], per_s[PLAN_MAX_EXPERTS];
    const int lane = threadIdx.x % WAVE;
    auto choice = [&](int p) { return ids ? chosen[(size_t)min(max(ids[p / top], 0), vocab - 1) * top + p % top] : chosen[p]; };
    for (int e = threadIdx.x; e < experts; e += PLAN_THREADS) cursor_s[e] = 0;
    __syncthreads();
    for (int p = threadIdx.x; p < n_pairs; p += PLAN_THREADS) atomicAdd(&cursor_s[choice(p)], 1);
    __syncthreads();
    if (threadIdx.x < WAVE) {
        constexpr int PER = PLAN_MAX_EXPERTS / WAVE;
        int padded[PER], mine = 0;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = lane * PER + i;
            padded[i] = e < experts ? (cursor_s[e] + tile - 1) / tile * tile : 0;
            mine += padded[i];
        }
        int up_to = mine;                                             // the sum over the lanes up to this one
#pragma unroll
        for (int off = 1; off < WAVE; off <<= 1) {
            const int other = __shfl_up(up_to, off, WAVE);
            if (lane >= off) up_to += other;
        }
        int at = up_to - mine;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = lane * PER + i;
            if (e < experts) start_s[e] = at;
            at += padded[i];
        }
        if (lane == WAVE - 1) {
            start_s[experts] = up_to;
            *used = up_to / tile;
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < max_tiles; i += PLAN_THREADS) tile_expert[i] = -1;
    // the slots that pad each tile
    for (int e = threadIdx.x / WAVE; e < experts; e += PLAN_THREADS / WAVE) {
        const int rows = cursor_s[e], per = rows_per_tile(rows, tile);
        for (int s = lane; s < start_s[e + 1] - start_s[e]; s += WAVE)
            if (s % tile >= min(per, rows - s / tile * per)) slot_pair[start_s[e] + s] = -1;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < experts; e += PLAN_THREADS) {
        const int rows = cursor_s[e], per = rows_per_tile(rows, tile), tiles = (start_s[e + 1] - start_s[e]) / tile;
        for (int i = 0; i < tiles; ++i) tile_expert[start_s[e] / tile + i] = e | min(per, rows - i * per) << TILE_EXPERT_BITS;
        cursor_s[e] = 0;
        per_s[e] = per;
    }
    __syncthreads();
    for (int p = threadIdx.x; p < n_pairs; p += PLAN_THREADS) {
        const int e = choice(p), at = atomicAdd(&cursor_s[e], 1), per = per_s[e];
        const int slot = start_s[e] + at / per * tile + at % per;
        slot_pair[slot] = p;
        pair_slot[p] = slot;
    }
}

// grid (tiles, blocks of GT_FEATURES features).  a: the rows [*, k_dim]; row_of_slot: null (the rows lie in slot order) or
// slot -> pair, the pair's row being pair / top.  w: [experts, n_w_rows, k_dim]; FORM 1 (gated): n_w_rows = 2 n_features, an
// expert's gate rows first, and the result is silu(gate) * up; FORM 3: the same rows, capped gated; FORM 2: the product through
// the exact gelu; FORM 4: the product through the squared relu; FORM 0: the product as it is.  out: bfloat16 [slots, n_features].
template <int FORM>
__global__ __launch_bounds__(GT_WAVES * WAVE) void moe_grouped_kernel(const bf16_t* __restrict__ a, const int* __restrict__ slot_pair, int top,
                                                                      const bf16_t* __restrict__ w, const int* __restrict__ tile_expert,
                                                                      int n_features, int k_dim, ExpertCap cap, bf16_t* __restrict__ out) {
    constexpr bool GATED = FORM == 1 || FORM == 3;
    const int tile = blockIdx.x;
    const int planned = tile_expert[tile];
    if (planned < 0) return;
    const int e = tile_expert_of(planned);
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    const int r = lane % 16, g = lane / 16;
    const int f0 = blockIdx.y * GT_FEATURES + wave * 32;
    if (f0 >= n_features) return;
    const int slot0 = tile * GT_TOKENS;
    // the rows of the tile's runs of 16 slots, as the second operand: column r is a row of activations
    const bf16_t* ar[GT_RUNS];
#pragma unroll
    for (int tt = 0; tt < GT_RUNS; ++tt) {
        const int slot = slot0 + 16 * tt + r;
        const int pair = slot_pair ? slot_pair[slot] : slot;
        const int row = slot_pair ? max(pair, 0) / top : slot;          // a slot that pads the run reads row 0; nobody reads its result
        ar[tt] = a + (size_t)row * k_dim;
    }
    const size_t w_rows = GATED ? 2 * (size_t)n_features : (size_t)n_features;
    const bf16_t* wr[GATED ? 4 : 2];
#pragma unroll
    for (int ft = 0; ft < 2; ++ft) {
        const int f = min(f0 + 16 * ft + r, n_features - 1);
        wr[ft] = w + ((size_t)e * w_rows + f) * k_dim;
        if (GATED) wr[2 + ft] = w + ((size_t)e * w_rows + n_features + f) * k_dim;
    }
    f32x4 acc[GATED ? 4 : 2][GT_RUNS];
#pragma unroll
    for (int i = 0; i < (GATED ? 4 : 2); ++i)
#pragma unroll
        for (int tt = 0; tt < GT_RUNS; ++tt) acc[i][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < k_dim; k0 += 32) {
        const int col = k0 + 8 * g;
        bf16x8 af[GT_RUNS], wf[GATED ? 4 : 2];
#pragma unroll
        for (int tt = 0; tt < GT_RUNS; ++tt) af[tt] = grouped_row8(ar[tt], col, k_dim);
#pragma unroll
        for (int i = 0; i < (GATED ? 4 : 2); ++i) wf[i] = grouped_row8(wr[i], col, k_dim);
#pragma unroll
        for (int i = 0; i < (GATED ? 4 : 2); ++i)
#pragma unroll
            for (int tt = 0; tt < GT_RUNS; ++tt) acc[i][tt] = mfma_16x16x32(wf[i], af[tt], acc[i][tt]);
    }
    // lane (r, g) holds features f0 + 16 ft + 4 g + i of the row in slot slot0 + 16 tt + r
#pragma unroll
    for (int ft = 0; ft < 2; ++ft)
#pragma unroll
        for (int tt = 0; tt < GT_RUNS; ++tt) {
            const int f = f0 + 16 * ft + 4 * g;
            if (f >= n_features) continue;                              // n_features is a multiple of four
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (GATED) {
                    v[i] = FORM == 3 ? expert_capped(acc[ft][tt][i], acc[2 + ft][tt][i], cap) : expert_silu_gated(acc[ft][tt][i], acc[2 + ft][tt][i]);
                } else if (FORM == 2) {
                    v[i] = expert_gelu(acc[ft][tt][i]);
                } else if (FORM == 4) {
                    v[i] = expert_relu_squared(acc[ft][tt][i]);
                } else {
                    v[i] = acc[ft][tt][i];
                }
            }
            uint2 pk;
            pk.x = (uint32_t)f32_to_bf16(v[0]).bits | ((uint32_t)f32_to_bf16(v[1]).bits << 16);
            pk.y = (uint32_t)f32_to_bf16(v[2]).bits | ((uint32_t)f32_to_bf16(v[3]).bits << 16);
            *reinterpret_cast<uint2*>(out + (size_t)(slot0 + 16 * tt + r) * n_features + f) = pk;
        }
}

// The same products in tiles of 64 NT slots x 256 weight rows through the walk of a prompt's plain products (big_walk.h; gated
// forms: of every 128 weight rows the first 64 are gate rows and the others their up rows).  FORM as above.
//
// What bounds it up to some 200 rows an expert is the weights' way from memory (32 experts of 2,048 x 4,096, 352 rows of four
// choices: 1.07 GB in 212 us with the plan and the sum, 5 TB/s), from there on the number of stages.  So
//   - the tiles in use, not as many as there could be, are shared out evenly over the dies (each gets a run of neighbouring
//     tiles, features innermost: an expert's weights and a tile's rows are read into one L2); by the number there could be,
//     three of eight dies stood idle at 852 rows
//   - an expert's features begin their walk at stages of their own: rows lie 4 or 8 KB apart, and blocks that walk in step ask
//     all for the same few of memory's channels (352 rows: 288 us in step, 234 so, tiles of 128 rows)
//   - the tile is as high as an expert's rows need, as long as that spares another tile (see big_tile_of)
//   - a tile of 256 rows multiplies 128 to 256 of them, in steps of 32, and an expert's rows are shared out evenly over its tiles (experts of
//     362 rows: two tiles of 192 and 170, not of 256 and 106): both products of 32 experts of 2,048 x 4,096 with 188 / 362 / 425 / 588 rows each 300 462
//     462 696 -> 268 405 435 618.
// Us with plan and sum, squared relu, rows of four choices over 32 experts: 130 rows 484 -> 209 (fragments from memory before),
// 852: 372 -> 251, 2,048: 590 -> 388 (a ring of three stages of 32 x 32 x 16 instructions before; this walk with eight waves 262 and 440).
template <int NT, int FORM, typename TO>
__global__ __launch_bounds__(BIG_THREADS) __attribute__((amdgpu_waves_per_eu(1, 1))) void moe_big_kernel(
    const bf16_t* __restrict__ a, const int* __restrict__ slot_pair, int top, const bf16_t* __restrict__ w, const int* __restrict__ tile_expert,
    const int* __restrict__ used, int feature_tiles, int n_features, int k_dim, ExpertCap cap, TO* __restrict__ out) {
    constexpr bool GATED = FORM == 1 || FORM == 3;
    __shared__ __attribute__((aligned(1024))) char lds[big_lds_bytes(NT)];
    const int total = *used * feature_tiles, per_die = (total + BIG_DIES - 1) / BIG_DIES, stages = k_dim / BIG_K;
    const int first = (blockIdx.x % BIG_DIES) * per_die + blockIdx.x / BIG_DIES, stride = gridDim.x / BIG_DIES;
    const int last = min(total, (int)(blockIdx.x % BIG_DIES + 1) * per_die), items = first < last ? (last - first + stride - 1) / stride : 0;
    if (items == 0) return;
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE, wave_f = wave % 2, wave_t = wave / 2;
    // (RAGGED) A tile's rows, 32 at a time, are dealt to its two waves of rows: what a wave has lies in its first column tiles
    constexpr bool RAGGED = NT == 4;
    auto row_at = [&](int row) __attribute__((always_inline)) { return RAGGED ? row % (32 * NT) / 16 * 32 + row / (32 * NT) * 16 + row % 16 : row; };
    big_walk<NT, true, RAGGED>(lds, (uint32_t)(k_dim * 2), items,
        [&](int item) __attribute__((always_inline)) {
            const int pid = first + item * stride, tile = pid / feature_tiles, ft = pid % feature_tiles;
            const int planned = __builtin_amdgcn_readfirstlane(tile_expert[tile]), e = tile_expert_of(planned), from = ft * (GATED ? 128 : BIG_FEAT);
            // (x_rows names the tile of slots: the rows of another are others)
            return BigItem{reinterpret_cast<const char*>(a), reinterpret_cast<const char*>(w + ((size_t)e * (GATED ? 2 : 1) * n_features + from) * k_dim), stages,
                           (5 * e + 2 * ft) % stages, tile, min(GATED ? 128 : BIG_FEAT, n_features - from), (tile_rows_of(planned) + 31) / 32};
        },
        [&](const BigItem& it, int row) __attribute__((always_inline)) {
            const int slot = it.x_rows * 64 * NT + (RAGGED ? min(row_at(row), it.live * 32 - 1) : row);
            return FORM == 0 ? slot : max(slot_pair[slot], 0) / top;      // a slot that pads the run reads row 0; nobody reads its result
        },
        [&](const BigItem& it, int row) __attribute__((always_inline)) {
            return GATED ? (row & 64 ? n_features : 0) + min(row / 128 * 64 + row % 64, it.w_rows - 1) : min(row, it.w_rows - 1);
        },
        [&](int item, f32x4 (&acc)[8][2 * NT], auto live) __attribute__((always_inline)) {
            const int pid = first + item * stride, tile = pid / feature_tiles, ft = pid % feature_tiles;
            f32x4 z[8];
#pragma unroll
            for (int t = 0; t < decltype(live)::value; ++t) {
                big_column(acc, t, z);
                const int slot = tile * 64 * NT + row_at(wave_t * 32 * NT + 16 * t + lane % 16);
                if (sizeof(TO) == 4 && slot_pair[slot] < 0) continue;          // (few rows: most of a tile pads its run)
                TO* row = out + (size_t)slot * n_features;
#pragma unroll
                for (int half = 0; half < (GATED ? 1 : 2); ++half) {
                    float v[16];
#pragma unroll
                    for (int f = 0; f < 4; ++f)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const float x = z[4 * half + f][i];
                            v[4 * f + i] = FORM == 1 ? big_silu_gated(x, z[4 + f][i]) : FORM == 3 ? expert_capped(x, z[4 + f][i], cap)
                                           : FORM == 2 ? expert_gelu(x) : FORM == 4 ? expert_relu_squared(x) : x;
                        }
                    big_store(row, (GATED ? ft * 128 + wave_f * 64 : ft * 256 + wave_f * 128 + half * 64) + 16 * (lane / 16), n_features, v);
                }
            }
        });
}

__device__ inline void combine_load8(const bf16_t* p, float (&v)[8]) {
    const bf16x8 q = load_bf16x8(p);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = (float)q[i];
}
__device__ inline void combine_load8(const float* p, float (&v)[8]) {
    const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

// One block per token; eight neighbouring columns a thread (width is a multiple of eight).  weight: null, or [n, top] (null: 1 / top).
// planes: n_planes float32 [n, width] to be added.
template <typename TY>
__global__ void moe_combine_kernel(const TY* __restrict__ y, const int* __restrict__ pair_slot, const float* __restrict__ weight, int top,
                                   int width, const bf16_t* __restrict__ add0, const bf16_t* __restrict__ add1, const float* __restrict__ planes,
                                   int n_planes, float* __restrict__ out) {
    const size_t t = blockIdx.x;
    for (int d = threadIdx.x * 8; d < width; d += blockDim.x * 8) {
        float total[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) total[i] = 0.f;
        auto add = [&](const auto* row, float f) {
            float v[8];
            combine_load8(row + d, v);
#pragma unroll
            for (int i = 0; i < 8; ++i) total[i] = fmaf(f, v[i], total[i]);
        };
#pragma unroll 4
        for (int c = 0; c < top; ++c)
            add(y + (size_t)pair_slot[t * top + c] * width, weight ? weight[t * top + c] : 1.0f / (float)top);
        if (add0) add(add0 + t * width, 1.0f);
        if (add1) add(add1 + t * width, 1.0f);
        for (int p = 0; p < n_planes; ++p) add(planes + ((size_t)p * gridDim.x + t) * width, 1.0f);
        *reinterpret_cast<float4*>(out + t * width + d) = make_float4(total[0], total[1], total[2], total[3]);
        *reinterpret_cast<float4*>(out + t * width + d + 4) = make_float4(total[4], total[5], total[6], total[7]);
    }
}

struct MoeSizes {
    long long n_pairs;
    int experts, width, ff;
    bool gated, aligned;         // aligned: h, gate_up and down start on 16 bytes
};

// Rows of a tile for experts with n_pairs / experts rows each: what takes the fewest stages' time (0.75, 0.87, 1.13 and 1.42 us
// for 64 to 256 rows) for an expert with somewhat more rows than the mean, a second tile for a few experts costing
// almost a whole round.  Tiles that do not fill the chip run side by side, so few or small experts take low ones: 16 experts of 256 x
// 512 with 250 rows each 51 us in tiles of 192 rows, 30 in tiles of 64.  Measured with a full chip, us, 32 experts of 2,048 x 4,096, tiles of
// 64 / 128 / 192 / 256 rows (before tiles of 256 could stop early): mean 25: 210 / 222 / 242 / 271, 75: 291 / 230 / 247 / 268, 106: 345 / 294 / 251 / 279, 150: 390 / 314 / 257 / 281,
// 181: 439 / 323 / 345 / 288, 256: 571 / 438 / 388 / 450, 375: 752 / 549 / 519 / 472, 625: 1,125 / 794 / 724 / 709.  At 49 sizes (also before; 8 to 128 experts of 256
// to 2,048 x 512 to 4,096, means of 8 to 2,000 rows) it takes the best tile at 40 and is 1.0 % behind it in the mean, 10 % at worst (1,000 rows for each of
// 16 small experts); with the times that a fit over those sizes gives (0.65, 0.77, 1.04, 1.46) it chooses otherwise at three of them, no better.
static int big_tile_of(const MoeSizes& s) {
    const double mean = (double)s.n_pairs / s.experts, rows = mean + 2.25 * sqrt(mean), in_use = (double)min((long long)s.experts, s.n_pairs);
    const double stage_us[4] = {0.75, 0.87, 1.13, 1.42};
    int best = 64;
    double best_cost = 1e300;
    for (int nt = 1; nt <= 4; ++nt) {
        const double tiles = in_use * ceil(rows / (64 * nt));
        auto rounds = [&](int features, int of_tile) { return ceil(tiles * ((features + of_tile - 1) / of_tile) / 256.0); };
        const double cost = (rounds(s.ff, s.gated ? BIG_FEAT / 2 : BIG_FEAT) * s.width + rounds(s.width, BIG_FEAT) * s.ff) * stage_us[nt - 1];
        if (cost < best_cost) { best_cost = cost; best = 64 * nt; }
    }
    // Experts of many rows: tiles of 256 multiply no more than their rows need either, and read the weights less often.  But each takes longer, so only
    // where both products have enough that the compute units' last ones matter little: two rounds of them.  Us, tiles of 192 and of 256 rows: 32 experts of
    // 2,048 x 4,096, mean 500 611 and 596, 850 955 and 895, 1,000 1,115 and 1,028; 16 of them, mean 500 333 and 361, 700 382 and 395; 4, mean 500 117 and 137; 32
    // gated ones of 1,408 x 2,048, mean 600 434 and 373; 8, mean 700 125 and 143; 64 of 512 x 1,024, mean 500 166 and 182.  Over 364 sizes (4 to 128 experts, means of
    // 450 to 1,800) at which the stages' time alone chooses 192: 0.5 % behind the better tile in the geometric mean (256 at all of them 5.0, 192 1.2), and 256
    // taken where it is 3 % slower or more at 7 of them, 6 % at worst (at all of them: 194, 18 %).
    auto tiles_of_256 = [&](int features, int of_tile) { return in_use * ceil(mean / 256) * ((features + of_tile - 1) / of_tile); };
    if (best == 192 && mean >= 448 && fmin(tiles_of_256(s.ff, s.gated ? BIG_FEAT / 2 : BIG_FEAT), tiles_of_256(s.width, BIG_FEAT)) >= 512) best = 256;
    return best;
}
// Whether the tiles cross LDS: rows in whole stages that start on 16 bytes, offsets from a matrix's first row of 32 bits, and, for
// few rows an expert, first matrices that fill half a tile (512 experts of 64 x 512, four a row, 300 rows: 59 us through LDS, 50 by
// fragments).
static bool big_tiles(const MoeSizes& s) {
    const long long rows = s.n_pairs + 256ll * (s.experts + 1), inner = max(s.width, s.ff);
    return s.aligned && s.width % BIG_K == 0 && s.ff % BIG_K == 0 && rows * inner < (1ll << 31) && 2ll * s.ff * s.width < (1ll << 31) &&
           ((s.gated ? 2 : 1) * s.ff >= BIG_FEAT / 2 || s.n_pairs >= 40ll * s.experts);
}
static int tile_of(const MoeSizes& s) { return big_tiles(s) ? big_tile_of(s) : GT_TOKENS; }
PALM_API int palm_moe_tile_tokens(int n_pairs, int experts, int width, int ff, int gated, int aligned) {
    return tile_of(MoeSizes{n_pairs, experts, width, ff, gated != 0, aligned != 0});
}

// chosen, weight [n, top]; h bfloat16 [n, width]; gate_up bfloat16 [experts, 2 ff, width] (the plain forms: [experts, ff, width], up
// rows alone); add0, add1: null or bfloat16 rows [n, width]; down bfloat16 [experts, width, ff].
// With ids [n] chosen is a table [vocab, top] of which every token takes its id's row, and weight may be null (1 / top).
// Room, with tile = palm_moe_tile_tokens(n top, experts, width, ff, gated, aligned), max_tiles = ceil(n top / tile) + experts and
// slots = max_tiles * tile: plan: (max_tiles + slots + n top + 1) ints; mid: slots * ff bfloat16; y: slots * width, bfloat16 or with y32
// (for tiles that cross LDS) float32.  planes: n_planes float32 rows [n, width] to add.  out float32 [n, width].
PALM_API int palm_moe_grouped_in_tiles(int n_pairs, int experts, int width, int ff, int gated, int aligned) {
    return experts <= PLAN_MAX_EXPERTS && big_tiles(MoeSizes{n_pairs, experts, width, ff, gated != 0, aligned != 0});
}
PALM_API int palm_moe_grouped(hipStream_t stream, const void* h, const void* gate_up, const void* down, const int* chosen,
                              const float* weight, int n_tokens, int top, int experts, int width, int ff, int* plan, void* mid, void* y,
                              float* out, int form, float limit, float slope, float shift, const void* add0, const void* add1,
                              const int* ids, int vocab, int y32, const float* planes, int n_planes) {
    PALM_CHECK(ids ? vocab > 0 : weight != nullptr, "moe_grouped: choices come with weights, or from a table of %d ids", vocab);
    PALM_CHECK(experts <= PLAN_MAX_EXPERTS, "moe_grouped: %d experts exceed %d", experts, PLAN_MAX_EXPERTS);
    PALM_CHECK(form >= EXPERT_GATED_SILU && form <= EXPERT_RELU_SQUARED, "moe_grouped: form %d is neither gated silu (0) nor plain gelu (1) nor capped "
               "gated (2) nor squared relu (3)", form);
    PALM_CHECK(form != EXPERT_CAPPED || limit > 0.f, "moe_grouped: the cap %g must be positive", (double)limit);
    PALM_CHECK(n_tokens >= 0 && top > 0 && experts > 0 && width > 0 && ff > 0, "moe_grouped: n=%d top=%d experts=%d width=%d ff=%d", n_tokens,
               top, experts, width, ff);
    PALM_CHECK(width % 8 == 0 && ff % 8 == 0, "moe_grouped: width %d and inner size %d must be multiples of eight", width, ff);
    if (n_tokens == 0) return 0;
    const long long n_pairs = (long long)n_tokens * top;
    PALM_CHECK(n_pairs < (1ll << 30), "moe_grouped: %lld pairs are more than one launch takes", n_pairs);
    const MoeSizes sizes{n_pairs, experts, width, ff, expert_is_gated(form), ((uintptr_t)h | (uintptr_t)gate_up | (uintptr_t)down) % 16 == 0};
    const bool big = big_tiles(sizes);
    PALM_CHECK(big || !y32, "moe_grouped: 32-bit results come from tiles that cross LDS (sizes of whole stages, rows that start on 16 bytes)");
    PALM_CHECK(n_planes == 0 || (n_planes > 0 && planes && (uintptr_t)planes % 16 == 0), "moe_grouped: %d planes to add", n_planes);
    const int tile = tile_of(sizes);
    const int max_tiles = (int)((n_pairs + tile - 1) / tile) + experts;
    int* tile_expert = plan;
    int* slot_pair = tile_expert + max_tiles;
    int* pair_slot = slot_pair + (size_t)max_tiles * tile;
    int* used = pair_slot + n_pairs;
    moe_plan_kernel<<<1, PLAN_THREADS, 0, stream>>>(chosen, ids, vocab, top, (int)n_pairs, experts, max_tiles, tile, tile_expert, slot_pair, pair_slot, used);
    const int combine_threads = width >= 2048 ? 256 : 128;
#define MOE_COMBINE(TY) moe_combine_kernel<TY><<<n_tokens, combine_threads, 0, stream>>>((const TY*)y, pair_slot, weight, top, width, \
        (const bf16_t*)add0, (const bf16_t*)add1, planes, n_planes, out)
    const ExpertCap cap{limit, slope, shift};
    if (big) {
        auto blocks = [&](int feature_tiles) { return dim3(min(256, (max_tiles * feature_tiles + BIG_DIES - 1) / BIG_DIES * BIG_DIES)); };
        const int up_features = expert_is_gated(form) ? BIG_FEAT / 2 : BIG_FEAT;
        const int up_tiles = (ff + up_features - 1) / up_features, down_tiles = (width + BIG_FEAT - 1) / BIG_FEAT;
        PALM_CHECK((long long)max_tiles * max(up_tiles, down_tiles) < (1ll << 30), "moe_grouped: %d tiles of rows are more than one launch takes", max_tiles);
#define MOE_BIG_UP(NT, FORM) moe_big_kernel<NT, FORM, bf16_t><<<blocks(up_tiles), BIG_THREADS, 0, stream>>>((const bf16_t*)h, slot_pair, top, \
            (const bf16_t*)gate_up, tile_expert, used, up_tiles, ff, width, cap, (bf16_t*)mid)
#define MOE_BIG(NT) { \
        if (form == EXPERT_GATED_SILU) MOE_BIG_UP(NT, 1); \
        else if (form == EXPERT_GELU) MOE_BIG_UP(NT, 2); \
        else if (form == EXPERT_CAPPED) MOE_BIG_UP(NT, 3); \
        else MOE_BIG_UP(NT, 4); \
        if (y32) MOE_BIG_DOWN(NT, float); else MOE_BIG_DOWN(NT, bf16_t); }
#define MOE_BIG_DOWN(NT, TO) moe_big_kernel<NT, 0, TO><<<blocks(down_tiles), BIG_THREADS, 0, stream>>>((const bf16_t*)mid, slot_pair, top, \
            (const bf16_t*)down, tile_expert, used, down_tiles, width, ff, cap, (TO*)y)
        if (tile == 64) MOE_BIG(1)
        else if (tile == 128) MOE_BIG(2)
        else if (tile == 192) MOE_BIG(3)
        else MOE_BIG(4)
#undef MOE_BIG
#undef MOE_BIG_UP
#undef MOE_BIG_DOWN
        if (y32) MOE_COMBINE(float); else MOE_COMBINE(bf16_t);
        PALM_LAUNCHED();
        return 0;
    }
    const dim3 up_grid(max_tiles, (ff + GT_FEATURES - 1) / GT_FEATURES);
#define MOE_UP(FORM) moe_grouped_kernel<FORM><<<up_grid, GT_WAVES * WAVE, 0, stream>>>((const bf16_t*)h, slot_pair, top, (const bf16_t*)gate_up, \
        tile_expert, ff, width, cap, (bf16_t*)mid)
    if (form == EXPERT_GATED_SILU) MOE_UP(1);
    else if (form == EXPERT_GELU) MOE_UP(2);
    else if (form == EXPERT_CAPPED) MOE_UP(3);
    else MOE_UP(4);
#undef MOE_UP
    moe_grouped_kernel<0><<<dim3(max_tiles, (width + GT_FEATURES - 1) / GT_FEATURES), GT_WAVES * WAVE, 0, stream>>>(
        (const bf16_t*)mid, nullptr, top, (const bf16_t*)down, tile_expert, width, ff, cap, (bf16_t*)y);
    MOE_COMBINE(bf16_t);
#undef MOE_COMBINE
    PALM_LAUNCHED();
    return 0;
}
