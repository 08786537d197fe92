// Decode attention whose work is cut by pages, not by sequences: a part of attention_mfma.hip (which includes this file
// behind the pieces that all its decode kernels share), for the head sizes 64 and 128 and up to eight query heads a kv head.
//
// The pages of all sequences stand in one row, one sequence behind the other, and for each kv head the row is cut into equal runs, 256 blocks over all kv
// heads, and a block's run into equal runs of its eight waves.  So a step of sequences of 70 to 1,500 tokens keeps every compute unit reading to the end, where
// slices of every sequence alike leave the long ones' slices alone at the end, and the eight waves of a unit have 96 KB on their way.
// The cut follows from the step's lengths by arithmetic that every wave does for itself (a prefix sum over the sequences' pages).
//
// A block first makes the queries of its sequences from the projection's rows (a lane holds eight elements of a head, so a wave makes four
// heads of 128 at once; they go to the waves through LDS), and for a sequence whose last page it has, the new key and value too: into
// the cache, and as one more key for the wave that reads that last page.  A wave walks its pages as the slices' waves do
// (score_page, weigh_values), across the ends of sequences without a stop.  A sequence that lies in one wave is finished by it; the pieces of others
// meet in LDS at the block's end, and what blocks hold of one sequence meets in memory: a (sequence, head)'s pieces are written past the caches
// (an agent-scope store each), then counted; the wave that counts the last one adds them up in the order of the blocks.  No
// fence writes back or empties a die's cache for it, and no wave ever waits for another block.  The counters are zero between launches: the wave that
// finds the last piece sets its counter back.
// Where a sequence is cut, and so in which order its pieces are added, follows from the pages of all sequences of the step: a step made again gives the
// same bits, but a neighbour that is a page longer can change a sequence's last ones.  (Slices follow from the number of sequences and the
// longest one, rounded up.)
//
// What bounds it: the walk reads at 5.5 to 6.3 TB/s; before it lie 3 us (two round trips for the step's lengths and the page numbers, the queries through LDS;
// 96 KB a unit are on their way meanwhile), behind it 2 to 4 (pieces to memory, the count, the last one's reads).  Us, 32 heads of 8 (by slices of every
// sequence alike, and so): 45 sequences of 70 to 1,500 tokens 44.9 and 35.2 (4.0 TB/s with all of it), 64 of 2,048 106.8 and 100.4, 8 of 2,048 20.8 and 17.7, one of
// 777 8.9 and 12.0: ops.decode_pages_pays.  The pages pass once and are marked so (nt): without that 37.6 105.2 19.3 for the first three.  Pages through LDS in whole lines against fragments read as the matrix cores want them, 16 rows by 64 bytes: 45
// sequences 39.6 and 37.9, one of 100 15.8 and 10.8.  Tried: rings of 16 KB (no change).
constexpr bool PAGES_SERVE_HEAD = HD == 64 || HD == 128;
constexpr int DP_WAVES = 8, DP_THREADS = DP_WAVES * WAVE;
constexpr int DP_BLOCKS = 256;               // one a compute unit
constexpr int DP_HEADS = 8;                  // query heads of a kv head, at most
constexpr int DP_QUERIES = DP_WAVES;         // sequences whose queries a block holds at once: each wave makes one
constexpr int DP_SEQS = 2 * WAVE;            // sequences of a step, at most: two a lane

// A wave's ring of slots.  A slot is 16 key rows of a page, or as many bytes of its V^T; a page is four slots of keys, then four of values.
constexpr int DP_SLOT = 16 * HD * 2, DP_LOADS = DP_SLOT / 1024;           // bytes, and instructions that fill it
constexpr int DP_RING = 12 * 1024, DP_SLOTS = DP_RING / DP_SLOT;
constexpr int DP_PARTS = 8;                  // slots that make a page
constexpr int DP_V_TILES = DTILES / 4;       // tiles of 16 value rows in a slot

// LDS traffic of the block done, then its barrier; reads from memory stay on their way
__device__ __forceinline__ void pages_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ void wave_lds_done() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// A value that another compute unit is to read in this launch, or one that another unit wrote: past the vector cache and the die's L2.
// (N: one or two floats, as one access)
template <int N> __device__ __forceinline__ void store_across(float* p, const float (&v)[N]) {
    using Bits = std::conditional_t<N == 2, uint64_t, uint32_t>;
    __hip_atomic_store(reinterpret_cast<Bits*>(p), __builtin_bit_cast(Bits, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <int N> __device__ __forceinline__ void load_across(const float* p, float (&v)[N]) {
    using Bits = std::conditional_t<N == 2, uint64_t, uint32_t>;
    const Bits bits = __hip_atomic_load(reinterpret_cast<Bits*>(const_cast<float*>(p)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_memcpy(v, &bits, sizeof(v));
}

// n things cut into runs whose sizes differ by at most one, the longer ones first: `per` and for the first `extra` runs one more
__device__ __forceinline__ int quotient(int x, int d) {                     // x, d >= 0 and below 2^24 (the product with the reciprocal is off by one at most)
    int q = (int)((float)x * __builtin_amdgcn_rcpf((float)d));
    const int rest = x - q * d;
    q += rest >= d ? 1 : 0;
    q -= rest < 0 ? 1 : 0;
    return __builtin_amdgcn_readfirstlane(q);
}
struct EvenCut {
    int per, extra;
    __device__ EvenCut(int n, int runs) : per(quotient(n, runs)), extra(n - per * runs) {}
    __device__ int begin(int i) const { return i * per + min(i, extra); }
    __device__ int holder(int x) const {                                   // (per > 0 or x < extra)
        const int front = extra * (per + 1);
        return x < front ? quotient(x, per + 1) : extra + quotient(x - front, max(per, 1));
    }
};

// An index that no kernel writes while this one runs, at a place that is the same in every lane: through the scalar cache, beside the reads of pages
// (a vector read would have to wait for all of them).
__device__ __forceinline__ int read_index(const int* p) { return *(const __attribute__((address_space(4))) int*)p; }

// The keys of the cache that a new position sees, first .. last, as pages: lo and the n from there on.  With a key of its own making the step sees the
// cache up to the position before.  A sequence that sees none has one page, all of it hidden, so that it is somebody's.
struct SeenPages {
    int lo, n;
    __device__ SeenPages(int pos, int window, bool writes) {
        const int first = window > 0 ? max(0, pos - window + 1) : 0;
        lo = first / PAGE_TOKENS;
        n = max(writes ? pos - 1 : pos, first) / PAGE_TOKENS - lo + 1;
    }
};

// Sums over the lanes up to each one: within rows of 16 lanes, then the rows' ends handed on.
__device__ __forceinline__ int lanes_up_to(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);        // row_shr 1, 2, 4, 8
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);        // the last lane of a row to all of the next (rows 1 and 3), then of 1 to 2 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
    return v;
}

// Within groups of N = 8 or 16 neighbouring lanes: a lane's partner (i ^ N / 2), the sum of all and the largest, every lane's.
template <int CTRL> __device__ __forceinline__ float from_lane(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
template <int N> __device__ __forceinline__ float partner_half(float v) {
    static_assert(N == 8 || N == 16, "a row of 16 lanes, or half of one");
    if constexpr (N == 16) return from_lane<0x128>(v);                     // row_ror 8
    else return from_lane<0x1B>(from_lane<0x141>(v));                      // mirrored in eight lanes, then in four
}
template <int N> __device__ __forceinline__ float sum_of(float v) {
    v += from_lane<0xB1>(v);                                               // i ^ 1, i ^ 2, then the other four's and the other eight's sum
    v += from_lane<0x4E>(v);
    v += from_lane<0x141>(v);
    if constexpr (N == 16) v += from_lane<0x140>(v);
    return v;
}
__device__ __forceinline__ float max_of_8(float v) {
    v = fmaxf(v, from_lane<0xB1>(v));
    v = fmaxf(v, from_lane<0x4E>(v));
    return fmaxf(v, from_lane<0x141>(v));
}

// The step's sequences, two a lane (l and l + 64): new position, slot, and the pages of the sequences before.
struct StepPages {
    const int* __restrict__ block_table;
    int pos[2], slot[2], before[2], total, n_seqs, nkv, kvh, window, max_pages;
    bool writes;
    __device__ static int of(const int (&v)[2], int b) {                   // b the same in every lane
        const int low = __builtin_amdgcn_readlane(v[0], b % WAVE), high = __builtin_amdgcn_readlane(v[1], b % WAVE);
        return b < WAVE ? low : high;
    }
    __device__ int begin(int b) const { return b >= n_seqs ? total : of(before, b); }         // the total behind the last
    __device__ void read(const int* __restrict__ seq_start, const int* __restrict__ seq_slot, int lane) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            pos[i] = seq_start[min(lane + WAVE * i, n_seqs - 1)];
            slot[i] = seq_slot[min(lane + WAVE * i, n_seqs - 1)];
        }
        const int n0 = lane < n_seqs ? SeenPages(pos[0], window, writes).n : 0, sum0 = lanes_up_to(n0);
        before[0] = sum0 - n0;
        total = __builtin_amdgcn_readlane(sum0, WAVE - 1);
        before[1] = total;
        if (n_seqs > WAVE) {
            const int n1 = lane + WAVE < n_seqs ? SeenPages(pos[1], window, writes).n : 0, sum1 = lanes_up_to(n1);
            before[1] = total + sum1 - n1;
            total += __builtin_amdgcn_readlane(sum1, WAVE - 1);
        }
    }
    __device__ int sequence_of(int x, int lane) const {
        return __popcll(__ballot(lane < n_seqs && before[0] <= x)) + __popcll(__ballot(lane + WAVE < n_seqs && before[1] <= x)) - 1;
    }
    __device__ size_t page_bytes(int b, int page) const {                  // where a page of sequence b starts in K and in V^T; in scalar registers
        const uint32_t held = __builtin_amdgcn_readfirstlane(read_index(block_table + (size_t)of(slot, b) * max_pages + page));
        return ((size_t)held * nkv + kvh) * (PAGE_TOKENS * HD * 2);
    }
};

// A page of the row: its sequence, and which of the sequence's pages it is.
struct PagePlace {
    int b, p, n, lo, pos;
    __device__ PagePlace(const StepPages& s, int x, int lane) {
        b = s.sequence_of(x, lane);
        enter(s);
        p = x - s.begin(b);
    }
    __device__ void enter(const StepPages& s) {
        pos = StepPages::of(s.pos, b);
        const SeenPages seen(pos, s.window, s.writes);
        lo = seen.lo;
        n = seen.n;
    }
    __device__ void advance(const StepPages& s) {                          // (there is a next one)
        if (++p < n) return;
        p = 0;
        ++b;
        enter(s);
    }
    __device__ size_t bytes(const StepPages& s) const { return s.page_bytes(b, lo + p); }
};

// A number that the compiler takes for a new one: what is made of it is made where it is used, not kept from the kernel's start.
__device__ __forceinline__ int made_here(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// A pointer that is the same in every lane, in scalar registers whatever it was made from
__device__ __forceinline__ const char* in_scalars(const char* p) {
    const uint64_t bits = reinterpret_cast<uint64_t>(p);
    const uint32_t low = __builtin_amdgcn_readfirstlane((uint32_t)bits), high = __builtin_amdgcn_readfirstlane((uint32_t)(bits >> 32));
    return reinterpret_cast<const char*>((uint64_t)high << 32 | low);
}

// The places of a lane in a slot.  An instruction fills 1 KB in lane order, whole lines of memory: 64 / CHUNKS key rows, or eight value rows.  The 16-byte
// pieces of a row are permuted by its number, so that the lanes that LDS serves together find different banks.  Row r of key slot t is key tile_key(t, r).
struct RingPlaces {
    uint32_t ask_k[DP_LOADS], ask_v, key[KSTEPS], value[2];
    __device__ explicit RingPlaces(int lane) {
        const int r = lane % 16, g = lane / 16;
#pragma unroll
        for (int i = 0; i < DP_LOADS; ++i) {
            const int row = i * (WAVE / CHUNKS) + lane / CHUNKS;
            ask_k[i] = (row / 4 * 8 + row % 4) * (HD * 2) + ((lane % CHUNKS) ^ (row % CHUNKS)) * 16;
        }
        ask_v = lane / 8 * 128 + ((lane % 8) ^ (lane / 8)) * 16;
#pragma unroll
        for (int j = 0; j < KSTEPS; ++j) key[j] = r * (HD * 2) + ((j * 4 + g) ^ (r % CHUNKS)) * 16;
#pragma unroll
        for (int h = 0; h < 2; ++h) value[h] = r * 128 + ((h * 4 + g) ^ (r % 8)) * 16;
    }
    __device__ void ask(const char* keys, const char* values, int part, uint32_t lds) const {
        lds_reads_done();                                                  // the slot may be the one they read
#pragma unroll
        for (int i = 0; i < DP_LOADS; ++i) {
            if (part < 4) row_chunk_into_lds<true>(in_scalars(keys + (part / 2 * 32 + part % 2 * 4) * (HD * 2)), ask_k[i], lds + i * 1024);
            else row_chunk_into_lds<true>(in_scalars(values + (part - 4) * DP_SLOT + i * 1024), ask_v, lds + i * 1024);
        }
    }
};

template <int P> using Part = std::integral_constant<int, P>;

// score_page's softmax for scores that carry the scale and log2 e already; a page without hidden keys does without masks
__device__ __forceinline__ float weigh_scores(f32x4 (&s)[4], int lo, int hi, Columns& c, int lane, bf16x8 (&pv)[2]) {
    if (lo > 0 || hi < PAGE_TOKENS - 1) {
        const int g = made_here(lane) / 16;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = t / 2 * 32 + 8 * g + t % 2 * 4 + i;         // tile_key(t, 4 g + i)
                s[t][i] = key >= lo && key <= hi ? s[t][i] : -INFINITY;
            }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[t][i]);
    mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE));
    mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
    const float m_new = fmaxf(c.m, mx), m_sub = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = exp2_weight(c.m - m_sub);
    float sum = 0.f;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float p = exp2_weight(s[2 * h + e / 4][e % 4] - m_sub);
            sum += p;
            pv[h][e] = (__bf16)p;
        }
    c.l = c.l * alpha + sum;
    c.m = m_new;
    return alpha;
}
// Elements 0 .. last of a fragment, zeros behind (see blank_values_after)
__device__ __forceinline__ bf16x8 seen_values(bf16x8 v, int last) {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = e <= last ? v[e] : (__bf16)0.0f;
    return v;
}

template <typename TIN, int PLANES>
struct SequenceQueries {
    // What a wave makes of one sequence: the rows of G query heads, then the new key's and the new value's, CHUNKS lanes a row.
    static constexpr int HELD = PLANES > 0 ? PLANES : 1;
    static constexpr int LANES = PAGES_SERVE_HEAD ? CHUNKS : 16, ROWS = WAVE / LANES;           // lanes of a row, rows at once
    static constexpr int PASSES = (DP_HEADS + 2 + ROWS - 1) / ROWS;
    Raw8<TIN> raw[PASSES][HELD];
    Raw8<float> w[PASSES], cs, sn;
    const TIN* row[PASSES];

    __device__ void ask(const TIN* __restrict__ qkv, size_t plane_stride, const float* q_norm_w, const float* k_norm_w, const float* cos_t,
                        const float* sin_t, int b, int kvh, int G, int nh, int nkv, int lane) {
        const int sub = lane / CHUNKS, ch = lane % CHUNKS;
        const size_t turn = (size_t)b * (HD / 2) + ch % (CHUNKS / 2) * 8;
        cs.read(cos_t ? cos_t + turn : k_norm_w ? k_norm_w : (const float*)qkv);       // (something that is there, where nothing is asked for)
        sn.read(cos_t ? sin_t + turn : k_norm_w ? k_norm_w : (const float*)qkv);
#pragma unroll
        for (int i = 0; i < PASSES; ++i) {
            const int t = min(i * ROWS + sub, G + 1);
            const int head = t < G ? kvh * G + t : t == G ? nh + kvh : nh + nkv + kvh;
            row[i] = qkv + ((size_t)b * (nh + 2 * nkv) + head) * HD + ch * 8;
#pragma unroll
            for (int pl = 0; pl < HELD; ++pl) raw[i][pl].read(row[i] + pl * plane_stride);
            w[i].read(q_norm_w ? (t < G ? q_norm_w : k_norm_w) + ch * 8 : (const float*)qkv);
        }
    }

    // The rows' planes added in their order, RMS norm over a head, rotation of (i, i + HD/2), rounding.  q_lds: G rows whose chunks lie
    // permuted by the head's number; k_lds: the new key's row; v_new: the new value, rounded, as 32 bits; s_new: the new key's scores.
    __device__ void prepare(int planes, size_t plane_stride, bool normed, float eps, bool rotated, bool owner, int G, float scale_log2, int lane,
                            bf16x8* q_lds, bf16x8* k_lds, float* v_new, float* s_new, bf16_t* k_dst, bf16_t* v_dst) {
        const int sub = lane / CHUNKS, ch = lane % CHUNKS;
#pragma unroll
        for (int i = 0; i < PASSES; ++i) {
            if (i * ROWS >= (owner ? G + 2 : G)) break;
            const int t = i * ROWS + sub;
            float x[8];
            raw[i][0].widen(x);
#pragma unroll
            for (int pl = 1; pl < HELD; ++pl) {
                float y[8];
                raw[i][pl].widen(y);
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] += y[e];
            }
            if (PLANES == 0) {
                for (int pl = 1; pl < planes; ++pl) {
                    Raw8<TIN> more;
                    float y[8];
                    more.read(row[i] + pl * plane_stride);
                    more.widen(y);
#pragma unroll
                    for (int e = 0; e < 8; ++e) x[e] += y[e];
                }
            }
            if (normed) {
                float ss = 0.f, wt[8];
                w[i].widen(wt);
#pragma unroll
                for (int e = 0; e < 8; ++e) ss += x[e] * x[e];
                ss = sum_of<LANES>(ss);
                const float inv = 1.0f / sqrtf(ss / (float)HD + eps);
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = t <= G ? x[e] * inv * wt[e] : x[e];
            }
            if (rotated) {
                float c[8], s[8];
                cs.widen(c);
                sn.widen(s);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float other = partner_half<LANES>(x[e]);
                    const float turned = ch < CHUNKS / 2 ? x[e] * c[e] - other * s[e] : other * s[e] + x[e] * c[e];
                    x[e] = t <= G ? turned : x[e];
                }
            }
            bf16x8 rounded;
#pragma unroll
            for (int e = 0; e < 8; ++e) rounded[e] = (__bf16)x[e];
            if (t < G) q_lds[t * CHUNKS + (ch ^ (t & 7))] = rounded;
            if (owner && t == G) {
                k_lds[ch] = rounded;
                *reinterpret_cast<bf16x8*>(k_dst + ch * 8) = rounded;
            }
            if (owner && t == G + 1) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    v_new[ch * 8 + e] = (float)rounded[e];
                    v_dst[(size_t)(ch * 8 + e) * PAGE_TOKENS] = f32_to_bf16(x[e]);
                }
            }
        }
        if (!owner) return;
        wave_lds_done();
        // the new key's score with each query, both as the cache and the matrix cores hold them
        for (int t0 = 0; t0 < G; t0 += ROWS) {
            const int t = min(t0 + sub, G - 1);
            const bf16x8 q = q_lds[t * CHUNKS + (ch ^ (t & 7))], k = k_lds[ch];
            float s = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) s += (float)q[e] * (float)k[e];
            s = sum_of<LANES>(s);
            if (ch == 0 && t0 + sub < G) s_new[t] = s * scale_log2;
        }
        wave_lds_done();                                                   // (the next sequence's key takes k_lds again)
    }
};

template <typename TIN, int PLANES>
__global__ __launch_bounds__(DP_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void attention_decode_pages_kernel(
    const TIN* __restrict__ qkv, int planes, size_t plane_stride, const float* __restrict__ q_norm_w,
    const float* __restrict__ k_norm_w, float eps, const float* __restrict__ cos_t, const float* __restrict__ sin_t,
    int write_cache, bf16_t* __restrict__ k_cache, bf16_t* __restrict__ v_cache,
    const int* __restrict__ block_table, int max_pages, const int* __restrict__ seq_slot,
    const int* __restrict__ seq_start, int n_seqs, int nh, int nkv, float scale_log2, int window,
    float* work, int* arrivals, bf16_t* __restrict__ out) {
    if constexpr (PAGES_SERVE_HEAD) {
        __shared__ __attribute__((aligned(1024))) char ring[DP_WAVES][DP_RING];
        __shared__ bf16x8 queries[DP_QUERIES][DP_HEADS * CHUNKS];
        __shared__ bf16x8 new_key[DP_WAVES][CHUNKS];
        __shared__ __attribute__((aligned(16))) float new_value[DP_QUERIES][HD];
        __shared__ float new_score[DP_QUERIES][DP_HEADS];
        // What a wave holds of a sequence that it has not all of: of the one that its run ends in (in its ring's place, which is free by then), and
        // of the one that its run begins in, where that is another.
        __shared__ __attribute__((aligned(16))) float piece_begin[DP_WAVES][DP_HEADS][HD];
        __shared__ float2 piece_ml[DP_WAVES][2][DP_HEADS];                 // maximum and sum; 0: the sequence at the run's begin, 1: at its end
        static_assert(DP_HEADS * HD * 4 <= DP_RING, "a piece lies where the ring was");
        auto piece = [&](int w, int end) { return end ? reinterpret_cast<float*>(ring[w]) : &piece_begin[w][0][0]; };
        const int lane0 = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
        const int G = nh / nkv, kvh = blockIdx.y;
        if (wave == DP_WAVES - 1) __builtin_amdgcn_s_setprio(3);             // it makes queries, for which all wait

        StepPages step{block_table, {0, 0}, {0, 0}, {0, 0}, 0, n_seqs, nkv, kvh, window, max_pages, write_cache != 0};
        step.read(seq_start, seq_slot, lane0);
        const int runs = min((int)gridDim.x, step.total), run = blockIdx.x;
        if (run >= runs) return;
        const EvenCut over_blocks(step.total, runs);
        const int i0 = over_blocks.begin(run), i1 = over_blocks.begin(run + 1);

        for (int c0 = i0, c1; c0 < i1; c0 = c1) {
            // the block's run, or as much of it as DP_QUERIES sequences' queries serve (usually all of it)
            const int seq0 = step.sequence_of(c0, lane0);
            c1 = min(i1, step.begin(seq0 + DP_QUERIES));
            const int n_here = step.sequence_of(c1 - 1, lane0) - seq0 + 1;
            const EvenCut over_waves(c1 - c0, DP_WAVES);
            const int w0 = c0 + over_waves.begin(wave), w1 = c0 + over_waves.begin(wave + 1);

            // The queries, made by the waves from the last one on (whose runs are the shorter ones), which ask for their pages behind that: the wait for
            // the rows would be one for all loads before.
            const bool makes_queries = DP_WAVES - 1 - wave < n_here;
            if (makes_queries) {
                const int s = DP_WAVES - 1 - wave, b = seq0 + s, pos = StepPages::of(step.pos, b), lane = made_here(lane0);
                const bool owner = write_cache && step.begin(b + 1) <= c1;                    // this block has the sequence's last page
                SequenceQueries<TIN, PLANES> make;
                make.ask(qkv, plane_stride, q_norm_w, k_norm_w, cos_t, sin_t, b, kvh, G, nh, nkv, lane);
                const size_t new_page = owner ? step.page_bytes(b, pos / PAGE_TOKENS) / 2 : 0;
                make.prepare(planes, plane_stride, q_norm_w != nullptr, eps, cos_t != nullptr, owner, G, scale_log2, lane, queries[s],
                             new_key[wave], new_value[s], new_score[s], k_cache + new_page + (size_t)(pos % PAGE_TOKENS) * HD,
                             v_cache + new_page + pos % PAGE_TOKENS);
            }
            const RingPlaces places(made_here(lane0));
            const uint32_t ring0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)ring[wave]);
            int ask_at = 0, use_at = 0;                                    // slots, as bytes
            PagePlace at(step, min(w0, c1 - 1), lane0);
            const char* keys = reinterpret_cast<const char*>(k_cache);
            const char* values = reinterpret_cast<const char*>(v_cache);
            size_t base = at.bytes(step);
            auto ask = [&](size_t page, int part) __attribute__((always_inline)) {
                places.ask(keys + page, values + page, part, __builtin_amdgcn_readfirstlane(ring0 + ask_at));
                ask_at = ask_at + DP_SLOT == DP_RING ? 0 : ask_at + DP_SLOT;
            };
            auto ask_first = [&]() __attribute__((always_inline)) {
#pragma unroll
                for (int u = 0; u < DP_SLOTS; ++u) ask(base, u);
            };
            if (w0 < w1 && !makes_queries) ask_first();
            pages_barrier();
            if (w0 < w1 && makes_queries) ask_first();
            __builtin_amdgcn_s_setprio(0);

            // the wave's pages, across the ends of sequences
            Columns c;
            auto start_over = [&]() __attribute__((always_inline)) {
                c.m = -INFINITY;
                c.l = 0.f;
#pragma unroll
                for (int dt = 0; dt < DTILES; ++dt) c.o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
            };
            bf16x8 qv[KSTEPS];
            auto take_query = [&](int s) __attribute__((always_inline)) {
                const int l = made_here(lane0), col = l % 16, row = min(col, G - 1);
#pragma unroll
                for (int j = 0; j < KSTEPS; ++j) {
                    const bf16x8 v = queries[s][row * CHUNKS + ((j * 4 + l / 16) ^ (row & 7))];
                    qv[j] = col < G ? v : zero_bf16x8();
                }
            };
            start_over();
            int piece_from = w0;
            if (w0 < w1) take_query(at.b - seq0);
            // what the wave has of a sequence is finished, or left for those who add it up (x: its last page)
            auto leave_piece = [&](int x, bool ends, int end_of_run) __attribute__((always_inline)) {
                const int s = at.b - seq0;
                const int here = made_here(lane0), r = here % 16, g = here / 16;
                float l = c.l;
                l += __shfl_xor(l, 16, WAVE);
                l += __shfl_xor(l, 32, WAVE);
                if (ends && write_cache) {                                 // the new key, one more with its value
                    const float score = new_score[s][min(r, G - 1)];
                    const float m = fmaxf(c.m, score), m_sub = m == -INFINITY ? 0.f : m;
                    const float alpha_old = exp2_weight(c.m - m_sub), weight = exp2_weight(score - m_sub);
                    l = l * alpha_old + weight;
                    c.m = m;
#pragma unroll
                    for (int dt = 0; dt < DTILES; ++dt) {
                        const float4 v = *reinterpret_cast<const float4*>(&new_value[s][dt * 16 + 4 * g]);
                        c.o[dt] = c.o[dt] * alpha_old + f32x4{v.x, v.y, v.z, v.w} * weight;
                    }
                }
                if (r >= G) return;
                if (ends && x + 1 - at.n >= piece_from) {                  // all of the sequence: finished
                    const float inv = 1.0f / l;
                    bf16_t* o = out + ((size_t)at.b * nh + kvh * G + r) * HD;
#pragma unroll
                    for (int dt = 0; dt < DTILES; ++dt) {
                        uint2 four;
                        four.x = (uint32_t)f32_to_bf16(c.o[dt][0] * inv).bits | ((uint32_t)f32_to_bf16(c.o[dt][1] * inv).bits << 16);
                        four.y = (uint32_t)f32_to_bf16(c.o[dt][2] * inv).bits | ((uint32_t)f32_to_bf16(c.o[dt][3] * inv).bits << 16);
                        *reinterpret_cast<uint2*>(o + dt * 16 + 4 * g) = four;
                    }
                } else {
                    if (g == 0) piece_ml[wave][end_of_run][r] = make_float2(c.m, l);
                    float* o = piece(wave, end_of_run) + r * HD;
#pragma unroll
                    for (int dt = 0; dt < DTILES; ++dt)
                        *reinterpret_cast<float4*>(o + dt * 16 + 4 * g) = make_float4(c.o[dt][0], c.o[dt][1], c.o[dt][2], c.o[dt][3]);
                }
            };
            // One page, slot by slot: its fragments meet the queries (or the weights), then the slot asks for what comes DP_SLOTS slots later,
            // of this page or of the next one.  `more` (a constant): there is a next one.
            auto walk_page = [&](int x, auto more) __attribute__((always_inline)) {
                const bool ends = at.p + 1 == at.n;
                PagePlace next = at;
                size_t next_base = base;
                if constexpr (more.value) {
                    next.advance(step);
                    next_base = next.bytes(step);
                }
                auto slot_arrives = [&](auto part) __attribute__((always_inline)) {
                    constexpr int LEFT = DP_PARTS - 1 - part.value;
                    all_but_the_youngest_have_arrived<DP_LOADS * (more.value || LEFT > DP_SLOTS - 1 ? DP_SLOTS - 1 : LEFT)>();
                    no_read_before_here();
                    return ring[wave] + use_at;
                };
                auto slot_is_used = [&](auto part) __attribute__((always_inline)) {
                    use_at = use_at + DP_SLOT == DP_RING ? 0 : use_at + DP_SLOT;
                    constexpr int AHEAD = part.value + DP_SLOTS;
                    if constexpr (AHEAD < DP_PARTS) ask(base, AHEAD);
                    else if constexpr (more.value) ask(next_base, AHEAD - DP_PARTS);
                };
                const int key0 = (at.lo + at.p) * PAGE_TOKENS;
                const int lo = (window > 0 ? max(0, at.pos - window + 1) : 0) - key0, hi = (write_cache ? at.pos - 1 : at.pos) - key0;
                f32x4 s[4];
                auto score = [&](auto part) __attribute__((always_inline)) {
                    const char* slot = slot_arrives(part);
                    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int j = 0; j < KSTEPS; ++j) acc = mfma_16x16x32(*reinterpret_cast<const bf16x8*>(slot + places.key[j]), qv[j], acc);
                    s[part.value] = acc * scale_log2;
                    slot_is_used(part);
                };
                score(Part<0>{}), score(Part<1>{}), score(Part<2>{}), score(Part<3>{});
                bf16x8 pv[2];
                const float alpha = weigh_scores(s, lo, hi, c, lane0, pv);
                auto weigh = [&](auto part) __attribute__((always_inline)) {
                    const char* slot = slot_arrives(part);
#pragma unroll
                    for (int i = 0; i < DP_V_TILES; ++i) {
                        f32x4& o = c.o[(part.value - 4) * DP_V_TILES + i];
                        o *= alpha;
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            bf16x8 v = *reinterpret_cast<const bf16x8*>(slot + places.value[h] + i * 2048);
                            if (hi < PAGE_TOKENS - 1) v = seen_values(v, hi - h * 32 - made_here(lane0) / 16 * 8);           // the same in every lane
                            o = mfma_16x16x32(v, pv[h], o);
                        }
                    }
                    slot_is_used(part);
                };
                weigh(Part<4>{}), weigh(Part<5>{}), weigh(Part<6>{}), weigh(Part<7>{});
                if constexpr (more.value) {
                    if (ends) {
                        leave_piece(x, true, 0);
                        piece_from = x + 1;
                        start_over();
                        take_query(next.b - seq0);
                    }
                } else {
                    lds_reads_done();                                      // (the piece may lie where the last slot was)
                    leave_piece(x, ends, 1);
                }
                at = next;
                base = next_base;
            };
            if (w0 < w1) {
                for (int x = w0; x + 1 < w1; ++x) walk_page(x, std::true_type{});
                walk_page(w1 - 1, std::false_type{});
            }
            pages_barrier();

            // The pieces of a sequence's head that several waves hold: a wave takes one (sequence, head) after the other.  Of a sequence that other blocks hold
            // pieces of too the sum goes to memory; that can be the block's first and its last sequence, so a wave has two such heads at most.
            constexpr int PER = PAGES_SERVE_HEAD ? HD / WAVE : 1;          // output elements a lane
            // place 0 of a block's two for the sequence that began before it, 1 for the one that goes on
            auto record = [&](int blk, int from, int h) __attribute__((always_inline)) {
                return work + ((size_t)((kvh * gridDim.x + blk) * 2 + (over_blocks.begin(blk) <= from ? 1 : 0)) * G + h) * WORK_STRIDE;
            };
            int left[2] = {-1, -1};                                        // which head of the block's first and of its last sequence
            for (int i = wave; i < n_here * G; i += DP_WAVES) {
                const int lane = made_here(lane0), s = i / G, h = i % G, b = seq0 + s;
                const int from = step.begin(b), to = step.begin(b + 1);
                const int begins = c0 + over_waves.begin(lane % DP_WAVES);   // of the waves' runs, a wave a lane
                const int wa = __popcll(__ballot(lane < DP_WAVES && begins <= max(from, c0))) - 1;
                const int we = __popcll(__ballot(lane < DP_WAVES && begins < min(to, c1))) - 1;
                const bool whole = from >= c0 && to <= c1;
                if (whole && wa == we) continue;
                auto at_end = [&](int w) { return to >= c0 + over_waves.begin(w + 1) ? 1 : 0; };          // the wave's run ends in this sequence
                const int mine = min(wa + lane % 8, we);
                const bool holds = wa + lane % 8 <= we;
                const float2 ml = piece_ml[mine][at_end(mine)][h];
                float v[DP_WAVES][PER];
#pragma unroll
                for (int k = 0; k < DP_WAVES; ++k) {
                    const int w = min(wa + k, we);
#pragma unroll
                    for (int e = 0; e < PER; ++e) v[k][e] = piece(w, at_end(w))[h * HD + lane * PER + e];
                }
                const float m = max_of_8(holds ? ml.x : -INFINITY), m_sub = m == -INFINITY ? 0.f : m;
                const float wt = holds ? exp2_weight(ml.x - m_sub) : 0.f;
                const float l = sum_of<8>(holds ? ml.y * wt : 0.f);
                float o[PER] = {};
#pragma unroll
                for (int k = 0; k < DP_WAVES; ++k) {
                    const float wk = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wt), k));
#pragma unroll
                    for (int e = 0; e < PER; ++e) o[e] += wa + k <= we ? v[k][e] * wk : 0.f;
                }
                const size_t head = (size_t)b * nh + kvh * G + h;
                if (whole) {
#pragma unroll
                    for (int e = 0; e < PER; ++e) out[head * HD + lane * PER + e] = f32_to_bf16(o[e] / l);
                    continue;
                }
                float* rec = record(run, from, h);
                const float own_ml[2] = {m, l};
                if (lane == 0) store_across(rec, own_ml);
                store_across(rec + WORK_O + lane * PER, o);
                (s == 0 ? left[0] : left[1]) = h;
            }
            // Counted when the pieces are where other dies read them.  Whoever counts a head's last piece adds them all, in the order of the blocks.
            if (left[0] >= 0 || left[1] >= 0) {
                const int lane = made_here(lane0), last_seq = seq0 + n_here - 1;
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                int arrived = 0;
                if (lane == 0 && left[0] >= 0)
                    arrived = __hip_atomic_fetch_add(arrivals + (size_t)seq0 * nh + kvh * G + left[0], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (lane == 1 && left[1] >= 0)
                    arrived = __hip_atomic_fetch_add(arrivals + (size_t)last_seq * nh + kvh * G + left[1], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                for (int k = 0; k < 2; ++k) {
                    const int h = k == 0 ? left[0] : left[1], b = k == 0 ? seq0 : last_seq;
                    if (h < 0) continue;
                    const int from = step.begin(b), to = step.begin(b + 1), ba = over_blocks.holder(from), n_rec = over_blocks.holder(to - 1) - ba + 1;
                    if (__builtin_amdgcn_readlane(arrived, k) != n_rec - 1) continue;
                    asm volatile("" ::: "memory");
                    const size_t head = (size_t)b * nh + kvh * G + h;
                    if (lane == 0) __hip_atomic_store(arrivals + head, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    float big = -INFINITY, total = 0.f, sum[PER] = {};
                    for (int k0 = 0; k0 < n_rec; k0 += DP_WAVES) {
                        float rec_ml[DP_WAVES][2], rec_o[DP_WAVES][PER];
#pragma unroll
                        for (int q = 0; q < DP_WAVES; ++q) {
                            const float* p = record(ba + min(k0 + q, n_rec - 1), from, h);
                            load_across(p, rec_ml[q]);
                            load_across(p + WORK_O + lane * PER, rec_o[q]);
                        }
                        float top = big;
#pragma unroll
                        for (int q = 0; q < DP_WAVES; ++q) top = fmaxf(top, k0 + q < n_rec ? rec_ml[q][0] : -INFINITY);
                        const float top_sub = top == -INFINITY ? 0.f : top, before = exp2_weight(big - top_sub);
                        total *= before;
#pragma unroll
                        for (int e = 0; e < PER; ++e) sum[e] *= before;
#pragma unroll
                        for (int q = 0; q < DP_WAVES; ++q) {
                            const float wk = exp2_weight(rec_ml[q][0] - top_sub);
                            const bool there = k0 + q < n_rec;
                            total += there ? rec_ml[q][1] * wk : 0.f;
#pragma unroll
                            for (int e = 0; e < PER; ++e) sum[e] += there ? rec_o[q][e] * wk : 0.f;
                        }
                        big = top;
                    }
#pragma unroll
                    for (int e = 0; e < PER; ++e) out[head * HD + lane * PER + e] = f32_to_bf16(sum[e] / total);
                }
            }
            if (c1 < i1) pages_barrier();                                  // the next run takes the same places in LDS
        }
    }
}
