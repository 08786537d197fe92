// Routed experts for up to 16 rows (a decode step's batch) in bfloat16: the matrices of the experts in use as one stream.
//
// What bounds it is memory: every expert that some row chose is read once.  The kernels of moe_few.hip give each (expert, run of
// rows) a block of its own, which looks for its rows before its first read, fills its reads once and ends; they reached 4.5 (up)
// and 5.1 TB/s (down).  Here, as in linear_ring.hip, a block of eight waves stays on its compute unit and walks over a list of
// work, each wave asking for 16 matrix rows x 128 values (4 KB) at a time as whole lines into a ring of its own in LDS, several
// ahead of its arithmetic and across the ends of experts.  All rows of the step are the columns of every matrix instruction, so
// no expert needs its rows gathered: a column whose row did not choose the expert is simply not kept.
//
//   up     strips of 16 matrix rows (gated: eight gate rows and their eight up rows) of the shared expert, then of the experts in
//          use, dealt to the blocks in turn; the rows' activations stay in registers, the waves take every eighth step of a strip
//   down   a block per (16 output features, plane): the steps of the shared expert and of the experts in use, dealt to the waves
//          in turn; the inner values come through LDS beside the weights; a step's sums go, weighted, into the wave's own
//          registers, and the waves' are added once, at the end, in their order
//
// The shared expert's steps come first, because they are known before it is known who chose what.
// 6 rows, 32 experts of 2,048 x 4,096 (17 in use) with a shared one of 4,096, both products: 127 -> 105 us, 5.7 TB/s; one row 78 -> 42;
// 16 rows (27 in use) 189 -> 166.  Where the matrices pass once (ONCE) their loads are marked so (nt, linear_ring.h): a decode step of six sequences through eight
// layers of 17 of 32 such experts 1,528 -> 1,447 us.
#include "mfma.h"
#include "expert_form.h"
#include "lds_stage.h"

constexpr int MR_ROWS = 16;                        // rows of a step at most: one tile of columns
constexpr int MR_WAVES = 8, MR_THREADS = MR_WAVES * WAVE;
constexpr int MR_K = 128;                          // values of a step
constexpr int MR_UNITS = 256;                      // blocks of a launch: one a compute unit
constexpr int MR_EXPERTS = 256, MR_TOP = 32;
constexpr int MR_STEPS = 8;                        // steps of a row of activations that a wave holds at most
constexpr int MR_UP_SLOTS = 4;
constexpr uint8_t MR_NOT_CHOSEN = 255;
static_assert(MR_ROWS * MR_TOP <= MR_THREADS && MR_EXPERTS <= MR_THREADS, "a thread for each choice, and for each expert");

__device__ __forceinline__ uint32_t mr_lds_address(const void* p) {
    return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p);
}
__device__ __forceinline__ void mr_barrier() {         // LDS traffic done, then the block's barrier; loads stay in flight
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
// all but the youngest `slots` slots of LOADS instructions each
template <int LOADS, int MAX> __device__ __forceinline__ void mr_wait_slots(int slots) {
    static_assert(MAX <= 3, "a ring of at most four slots");
    if (MAX >= 3 && slots >= 3) all_but_the_youngest_have_arrived<3 * LOADS>();
    else if (MAX >= 2 && slots == 2) all_but_the_youngest_have_arrived<2 * LOADS>();
    else if (MAX >= 1 && slots == 1) all_but_the_youngest_have_arrived<1 * LOADS>();
    else all_but_the_youngest_have_arrived<0>();
    no_read_before_here();
}

struct RingChoices {
    const int* rows;                 // [n, top], or with ids the table [vocab, top]
    const float* weight;             // [n, top]; null: 1 / top
    const int* ids;
    int vocab, top, n, experts;
};

// Who chose what, in LDS.  A row that names an expert twice counts once, with both weights; a choice outside the experts counts as
// none.  (The reads stand before the ring's first, the rest behind them: a wait for a read of the compiler's waits for the ring too.)
struct RingPlan {
    uint8_t slot[MR_EXPERTS * MR_ROWS];              // [expert][row]: which of the row's choices (the first that names it)
    int chosen[MR_ROWS * MR_TOP];
    float given[MR_ROWS * MR_TOP], weight[MR_ROWS * MR_TOP];
    uint32_t present[MR_EXPERTS / 32];
    uint16_t used[MR_EXPERTS];                       // the experts in use, in ascending order
    int n_used;
};
struct RingChoice { int expert; float weight; };
__device__ inline RingChoice mr_read_choice(const RingChoices& ch) {       // this thread's (row, choice)
    const int p = min((int)threadIdx.x, ch.n * ch.top - 1), t = p / ch.top;
    RingChoice c;
    c.weight = ch.weight ? ch.weight[p] : 1.0f / (float)ch.top;
    c.expert = ch.ids ? ch.rows[(size_t)min(max(ch.ids[t], 0), ch.vocab - 1) * ch.top + p % ch.top] : ch.rows[p];
    return c;
}
__device__ inline void mr_plan(RingPlan& plan, const RingChoices& ch, const RingChoice& mine) {
    const int p = threadIdx.x, pairs = ch.n * ch.top;
    for (int i = p; i < ch.experts * MR_ROWS / 16; i += MR_THREADS) reinterpret_cast<uint4*>(plan.slot)[i] = make_uint4(~0u, ~0u, ~0u, ~0u);
    if (p < MR_EXPERTS / 32) plan.present[p] = 0;
    if (p < pairs) { plan.chosen[p] = mine.expert; plan.given[p] = mine.weight; }
    mr_barrier();
    if (p < pairs && mine.expert >= 0 && mine.expert < ch.experts) {
        const int t = p / ch.top, c = p % ch.top;
        int first = MR_TOP;
        float sum = 0.f;
        for (int o = 0; o < ch.top; ++o) {
            const bool same = plan.chosen[t * ch.top + o] == mine.expert;
            first = same ? min(first, o) : first;
            sum += same ? plan.given[t * ch.top + o] : 0.f;
        }
        if (first == c) {
            plan.slot[mine.expert * MR_ROWS + t] = (uint8_t)c;
            plan.weight[p] = sum;
            atomicOr(&plan.present[mine.expert / 32], 1u << (mine.expert % 32));
        }
    }
    mr_barrier();
    int before = 0, all = 0;
#pragma unroll
    for (int i = 0; i < MR_EXPERTS / 32; ++i) {
        const int count = __popc(plan.present[i]);
        before += i < p / 32 ? count : 0;
        all += count;
    }
    if (p < ch.experts && (plan.present[p / 32] >> (p % 32) & 1)) plan.used[before + __popc(plan.present[p / 32] & ((1u << (p % 32)) - 1u))] = (uint16_t)p;
    if (p == 0) plan.n_used = all;
    mr_barrier();
}

// What a lane asks for in an instruction: 16 bytes of row (lane / 8) of eight, piece (lane % 8) ^ (lane / 8) of a line's eight; and
// where it finds its fragment of 32 values j: row r, pieces 4 (j % 2) + g of half j / 2 (linear_ring.h).
__device__ __forceinline__ uint32_t mr_fragment(int j, int r, int g) {
    return ((r / 8) + 2 * (j / 2)) * 1024 + (r % 8) * 128 + ((((j % 2) * 4 + g) ^ (r % 8)) * 16);
}

template <int TREG, bool GATED, bool ONCE>
__global__ __launch_bounds__(MR_THREADS) void moe_ring_up_kernel(const bf16_t* __restrict__ h, const bf16_t* __restrict__ up, RingChoices ch,
                                                                 int width, int ff, const bf16_t* __restrict__ shared_up, int shared_ff,
                                                                 int form, ExpertCap cap, bf16_t* __restrict__ mid) {
    constexpr int U = MR_UP_SLOTS, SLOT = 4096, LOADS = 4, FEATURES = GATED ? 8 : 16;
    __shared__ __attribute__((aligned(1024))) char ring[MR_WAVES * U * SLOT];
    __shared__ float part[2][MR_WAVES][16][17];
    __shared__ __attribute__((aligned(16))) RingPlan plan;
    const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int r = lane % 16, g = lane / 16, row8 = lane / 8, piece = (lane % 8) ^ row8;
    const int row_ff = ch.top * ff + shared_ff;
    const int shared_strips = shared_ff / FEATURES, per_expert = ff / FEATURES;
    const int T = max(0, (width / MR_K - wave + MR_WAVES - 1) / MR_WAVES);            // this wave's steps of a strip

    RingChoice mine = mr_read_choice(ch);                    // (waited for: what follows would only wait behind it)
    asm volatile("" : "+v"(mine.expert), "+v"(mine.weight));

    const uint32_t in_line = (uint32_t)row8 * (uint32_t)width * 2u + (uint32_t)piece * 16u;
    const uint32_t ring0 = mr_lds_address(ring) + wave * (U * SLOT);
    int total = 0, n_asked = 0, n_used = 0, ask_item = blockIdx.x, ask_t = 0;
    const char* base[2];
    auto bases_of = [&](int item) __attribute__((always_inline)) {
        const bf16_t* w;
        int strip = item, rows = shared_ff;
        if (item < shared_strips) {
            w = shared_up;
        } else {
            const int at = (item - shared_strips) / per_expert;
            strip = item - shared_strips - at * per_expert;
            w = up + (size_t)__builtin_amdgcn_readfirstlane((int)plan.used[at]) * (GATED ? 2 : 1) * ff * width;
            rows = ff;
        }
        base[0] = reinterpret_cast<const char*>(w + (size_t)strip * FEATURES * width);
        base[1] = base[0] + (size_t)(GATED ? rows : 8) * width * 2;
    };
    auto ask = [&]() __attribute__((always_inline)) {
        const uint32_t to = ring0 + (n_asked & (U - 1)) * SLOT;
        const uint32_t k0 = (uint32_t)(ask_t * MR_WAVES + wave) * (MR_K * 2);
        lds_reads_done();
#pragma unroll
        for (int i = 0; i < 4; ++i) row_chunk_into_lds<ONCE>(base[i % 2], in_line + k0 + (i / 2) * 128, to + i * 1024);
        ++n_asked;
        ++ask_t;
    };
    if (ask_item < shared_strips) {                          // what needs no plan is asked for before there is one
        bases_of(ask_item);
        for (int u = 0; u < U && u < T; ++u) ask();
    }
    bf16x8 xa[TREG][4];
    const bf16_t* xp = h + (size_t)min(r, ch.n - 1) * width + g * 8;
#pragma unroll
    for (int t = 0; t < TREG; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) xa[t][j] = load_bf16x8(xp + min((t * MR_WAVES + wave) * MR_K, width - MR_K) + j * 32);
    // The compiler's wait for these counts no load of the ring, so it waits for all that went out before: it stands here, where
    // that is the first filling and nothing more.
#pragma unroll
    for (int t = 0; t < TREG; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) asm volatile("" : "+v"(xa[t][j]));
    mr_plan(plan, ch, mine);
    const int items = shared_strips + __builtin_amdgcn_readfirstlane(plan.n_used) * per_expert;
    const int my_items = items > (int)blockIdx.x ? (items - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x : 0;
    total = my_items * T;
    auto ask_next = [&]() __attribute__((always_inline)) {
        if (ask_t == T) { ask_t = 0; ask_item += gridDim.x; }
        if (ask_t == 0) bases_of(ask_item);
        ask();
    };
    for (; n_asked < U && n_asked < total;) ask_next();

    int buf = 0;
    for (int item = blockIdx.x; item < items; item += gridDim.x) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < TREG; ++t) {
            if (t >= T) break;
            mr_wait_slots<LOADS, U - 1>(min(U - 1, n_asked - n_used - 1));
            const char* slot = ring + (wave * U + (n_used & (U - 1))) * SLOT;
#pragma unroll
            for (int j = 0; j < 4; ++j) acc = mfma_16x16x32(*reinterpret_cast<const bf16x8*>(slot + mr_fragment(j, r, g)), xa[t][j], acc);
            ++n_used;
            if (n_asked < total) ask_next();
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) part[buf][wave][4 * g + i][r] = acc[i];
        mr_barrier();                                        // (two buffers: one barrier a strip is enough)
        const bool is_shared = item < shared_strips;
        const int at = is_shared ? 0 : (item - shared_strips) / per_expert;
        const int strip = is_shared ? item : item - shared_strips - at * per_expert;
        if (threadIdx.x < 16 * FEATURES) {
            const int c = threadIdx.x % FEATURES, col = threadIdx.x / FEATURES;
            float first = 0.f, second = 0.f;
#pragma unroll
            for (int w = 0; w < MR_WAVES; ++w) {
                first += part[buf][w][c][col];
                if (GATED) second += part[buf][w][c + 8][col];
            }
            const int slot = is_shared ? ch.top : plan.slot[plan.used[at] * MR_ROWS + col];
            if (col < ch.n && slot != MR_NOT_CHOSEN) {
                float v;
                if constexpr (GATED) v = form == EXPERT_CAPPED ? expert_capped(first, second, cap) : expert_silu_gated(first, second);
                else v = expert_plain(form, first);
                mid[(size_t)col * row_ff + (size_t)slot * ff + strip * FEATURES + c] = f32_to_bf16(v);
            }
        }
        buf ^= 1;
    }
}

// HALVES: eight (1) or sixteen (2) rows of inner values beside a step's weights.
template <int HALVES, bool ONCE>
__global__ __launch_bounds__(MR_THREADS) void moe_ring_down_kernel(const bf16_t* __restrict__ mid, const bf16_t* __restrict__ down, RingChoices ch,
                                                                   int width, int ff, const bf16_t* __restrict__ shared_down, int shared_ff,
                                                                   const bf16_t* __restrict__ add0, const bf16_t* __restrict__ add1,
                                                                   float* __restrict__ out) {
    constexpr int U = HALVES == 1 ? 3 : 2, SLOT = 4096 + HALVES * 2048, LOADS = 4 + 2 * HALVES;
    __shared__ __attribute__((aligned(1024))) char ring[MR_WAVES * U * SLOT];
    __shared__ __attribute__((aligned(16))) RingPlan plan;
    const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int r = lane % 16, g = lane / 16, row8 = lane / 8, piece = (lane % 8) ^ row8;
    const int row_ff = ch.top * ff + shared_ff, j0 = blockIdx.x * 16, planes = gridDim.y;
    const int shared_steps = shared_ff / MR_K, per_expert = ff / MR_K;
    const int first_step = blockIdx.y * MR_WAVES + wave, stride = planes * MR_WAVES;

    RingChoice mine = mr_read_choice(ch);
    asm volatile("" : "+v"(mine.expert), "+v"(mine.weight));

    const uint32_t ring0 = mr_lds_address(ring) + wave * (U * SLOT);
    int steps = shared_steps, ask_step = first_step, ask_slot = 0, n_asked = 0, n_used = 0;
    auto ask = [&]() __attribute__((always_inline)) {
        const uint32_t to = ring0 + ask_slot * SLOT;
        const char* base;
        uint32_t row_bytes, x_off[HALVES];
        lds_reads_done();
        if (ask_step < shared_steps) {
            base = reinterpret_cast<const char*>(shared_down + (size_t)j0 * shared_ff + ask_step * MR_K);
            row_bytes = shared_ff * 2;
#pragma unroll
            for (int i = 0; i < HALVES; ++i) x_off[i] = (uint32_t)(min(8 * i + row8, ch.n - 1) * row_ff + ch.top * ff + ask_step * MR_K) * 2u;
        } else {
            const int at = (ask_step - shared_steps) / per_expert, k0 = (ask_step - shared_steps - at * per_expert) * MR_K;
            const int e = __builtin_amdgcn_readfirstlane((int)plan.used[at]);
            base = reinterpret_cast<const char*>(down + ((size_t)e * width + j0) * ff + k0);
            row_bytes = ff * 2;
#pragma unroll
            for (int i = 0; i < HALVES; ++i) {               // (a row that did not choose the expert: something finite or not, never kept)
                const int t = min(8 * i + row8, ch.n - 1), slot = plan.slot[e * MR_ROWS + t];
                x_off[i] = (uint32_t)(t * row_ff + (slot == MR_NOT_CHOSEN ? 0 : slot) * ff + k0) * 2u;
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            row_chunk_into_lds<ONCE>(base + (size_t)(i % 2) * 8 * row_bytes + (i / 2) * 128, row8 * row_bytes + piece * 16u, to + i * 1024);
#pragma unroll
        for (int i = 0; i < 2 * HALVES; ++i)
            row_chunk_into_lds(reinterpret_cast<const char*>(mid) + (i / HALVES) * 128, x_off[i % HALVES] + piece * 16u, to + 4096 + i * 1024);
        ++n_asked;
        ask_step += stride;
        ask_slot = ask_slot + 1 == U ? 0 : ask_slot + 1;
    };
    for (int u = 0; u < U && ask_step < shared_steps; ++u) ask();
    mr_plan(plan, ch, mine);
    steps += __builtin_amdgcn_readfirstlane(plan.n_used) * per_expert;
    while (n_asked < U && ask_step < steps) ask();

    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    int slot_at = 0;
    const int x_row = HALVES == 1 ? r % 8 : r;               // (columns beyond the rows are not kept)
    for (int s = first_step; s < steps; s += stride) {
        mr_wait_slots<LOADS, U - 1>(min(U - 1, n_asked - n_used - 1));
        const char* slot = ring + (wave * U + slot_at) * SLOT;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bf16x8 w = *reinterpret_cast<const bf16x8*>(slot + mr_fragment(j, r, g));
            const uint32_t x_at = 4096 + ((x_row / 8) + HALVES * (j / 2)) * 1024 + (x_row % 8) * 128 + ((((j % 2) * 4 + g) ^ (x_row % 8)) * 16);
            acc = mfma_16x16x32(w, *reinterpret_cast<const bf16x8*>(slot + x_at), acc);
        }
        float weight = 1.0f;
        bool kept = r < ch.n;
        if (s >= shared_steps) {
            const int e = plan.used[(s - shared_steps) / per_expert], choice = plan.slot[e * MR_ROWS + r];
            kept = kept && choice != MR_NOT_CHOSEN;
            weight = plan.weight[kept ? r * ch.top + choice : 0];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[i] = kept ? fmaf(weight, acc[i], sum[i]) : sum[i];
        ++n_used;
        slot_at = slot_at + 1 == U ? 0 : slot_at + 1;
        if (ask_step < steps) ask();
    }
    // the waves' sums, in the ring's place (a wave's own part of it: nothing is on its way any more)
    float* mine_s = reinterpret_cast<float*>(ring + wave * (U * SLOT));
    lds_reads_done();
#pragma unroll
    for (int i = 0; i < 4; ++i) mine_s[(4 * g + i) * 17 + r] = sum[i];
    mr_barrier();
    if (threadIdx.x < 256) {
        const int row = threadIdx.x % 16, t = threadIdx.x / 16, j = j0 + row;
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < MR_WAVES; ++w) v += reinterpret_cast<const float*>(ring + w * (U * SLOT))[row * 17 + t];
        if (t < ch.n) {
            if (blockIdx.y == 0 && add0) v += to_float(add0[(size_t)t * width + j]);
            if (blockIdx.y == 0 && add1) v += to_float(add1[(size_t)t * width + j]);
            out[((size_t)blockIdx.y * ch.n + t) * width + j] = v;
        }
    }
}

// How many planes of partial sums give every compute unit a block, for a reader that adds them (at most four).
PALM_API int palm_moe_ring_planes(int width) { return max(1, min(4, MR_UNITS / max(1, width / 16))); }

// h bfloat16 [n, width]; up, down, shared_up, shared_down, forms as in moe.hip, all bfloat16; chosen, weight [n, top], or with ids [n]
// the table [vocab, top] and no weight; add0, add1: null or bfloat16 rows [n, width]; mid: room for n * (top * ff + shared_ff) bfloat16;
// out float32 [planes, n, width].  once: the matrices pass once, more than the memory-side cache holds passes before they are read again (linear_ring.h).
PALM_API int palm_moe_ring(hipStream_t stream, const void* h, const void* up, const void* down, const int* chosen, const float* weight,
                           const int* ids, int vocab, int n_tokens, int top, int experts, int width, int ff, const void* shared_up,
                           const void* shared_down, int shared_ff, int form, float limit, float slope, float shift, const void* add0,
                           const void* add1, void* mid, int planes, float* out, int once) {
    PALM_CHECK(form >= EXPERT_GATED_SILU && form <= EXPERT_RELU_SQUARED, "moe_ring: form %d is neither gated silu (0) nor plain gelu (1) nor capped "
               "gated (2) nor squared relu (3)", form);
    PALM_CHECK(form != EXPERT_CAPPED || limit > 0.f, "moe_ring: the cap %g must be positive", (double)limit);
    PALM_CHECK(n_tokens >= 0 && n_tokens <= MR_ROWS && top > 0 && top <= min(experts, MR_TOP) && experts <= MR_EXPERTS,
               "moe_ring: n=%d (at most %d) top=%d (at most %d) experts=%d (at most %d)", n_tokens, MR_ROWS, top, MR_TOP, experts, MR_EXPERTS);
    PALM_CHECK(width > 0 && width % MR_K == 0 && width <= MR_STEPS * MR_WAVES * MR_K && ff > 0 && ff % MR_K == 0 && shared_ff >= 0 && shared_ff % MR_K == 0,
               "moe_ring: width %d (at most %d) and inner sizes %d, %d must be multiples of %d", width, MR_STEPS * MR_WAVES * MR_K, ff, shared_ff, MR_K);
    PALM_CHECK((long long)(top * (long long)ff + shared_ff) * MR_ROWS < (1ll << 30) && (long long)ff * 16 < (1ll << 30) && (long long)shared_ff * 16 < (1ll << 30),
               "moe_ring: inner sizes %d, %d are more than an offset of 32 bits takes", ff, shared_ff);
    PALM_CHECK(ids ? vocab > 0 : weight != nullptr, "moe_ring: choices come with weights, or from a table of %d ids", vocab);
    PALM_CHECK(shared_ff == 0 || (shared_up && shared_down), "moe_ring: a shared expert of inner size %d needs its matrices", shared_ff);
    PALM_CHECK(planes >= 1 && planes <= 4, "moe_ring: %d planes (at most four)", planes);
    if (n_tokens == 0) return 0;
    const RingChoices ch{chosen, weight, ids, vocab, top, n_tokens, experts};
    const ExpertCap cap{limit, slope, shift};
    const bool gated = expert_is_gated(form);
    const long long strips = ((long long)shared_ff + (long long)min(experts, n_tokens * top) * ff) / (gated ? 8 : 16);
    const int blocks = (int)min((long long)MR_UNITS, strips), steps = (width + MR_WAVES * MR_K - 1) / (MR_WAVES * MR_K);
#define MR_UP(TREG, GATED) (once ? moe_ring_up_kernel<TREG, GATED, true> : moe_ring_up_kernel<TREG, GATED, false>)<<<blocks, MR_THREADS, 0, stream>>>((const bf16_t*)h, (const bf16_t*)up, ch, width, ff, \
        (const bf16_t*)shared_up, shared_ff, form, cap, (bf16_t*)mid)
#define MR_UP_STEPS(TREG) if (gated) MR_UP(TREG, true); else MR_UP(TREG, false)
    if (steps <= 1) { MR_UP_STEPS(1); }
    else if (steps <= 2) { MR_UP_STEPS(2); }
    else if (steps <= 4) { MR_UP_STEPS(4); }
    else { MR_UP_STEPS(8); }
#undef MR_UP_STEPS
#undef MR_UP
    PALM_LAUNCHED();
#define MR_DOWN(HALVES) (once ? moe_ring_down_kernel<HALVES, true> : moe_ring_down_kernel<HALVES, false>)<<<dim3(width / 16, planes), MR_THREADS, 0, stream>>>((const bf16_t*)mid, (const bf16_t*)down, ch, \
        width, ff, (const bf16_t*)shared_down, shared_ff, (const bf16_t*)add0, (const bf16_t*)add1, out)
    if (n_tokens <= 8) MR_DOWN(1); else MR_DOWN(2);
#undef MR_DOWN
    PALM_LAUNCHED();
    return 0;
}
