// The selective scan of a Mamba layer and the short causal convolution in front of it.
//
//   conv     u_t[c] = silu(bias[c] + sum_j w[c][j] x_(t - (taps-1) + j)[c]),  j = 0 .. taps-1 (the last column is the current
//            token's); inputs before the sequence's start are zero; the last taps-1 inputs are kept per sequence.
//   scan     dt_t[c] = softplus(dtl_t[c] + dt_bias[c]);   A[c][n] = -exp(A_log[c][n])
//            S_t[c][n] = exp(dt_t[c] A[c][n]) S_(t-1)[c][n] + dt_t[c] u_t[c] B_t[n]
//            y_t[c] = (sum_n S_t[c][n] C_t[n] + D[c] u_t[c]) * silu(z_t[c])
//
// S is 32-bit and kept per sequence; step sizes, decays, exponentials and the sums are 32-bit.  Both kernels walk
// over a sequence's new tokens whatever their number: a prompt leaves what its tokens one by one leave.
#include "conv_state.h"

__device__ inline float silu_f(float z) { return z / (1.0f + expf(-z)); }
__device__ inline float softplus_dt(float z) { return z > 20.f ? z : log1pf(expf(z)); }

// One thread per (token of a sequence, channel): grid (channel blocks, longest run of new tokens, sequences).
template <typename T>
__global__ void causal_conv_kernel(const T* __restrict__ x, int x_stride, const float* __restrict__ w,
                                   const float* __restrict__ bias, const float* __restrict__ conv_state,
                                   const int* __restrict__ seq_slot, const int* __restrict__ seq_new,
                                   const int* __restrict__ cu_new, int channels, int taps, T* __restrict__ out) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x, ti = blockIdx.y, b = blockIdx.z;
    if (c >= channels || ti >= seq_new[b]) return;
    const size_t row0 = (size_t)cu_new[b];
    const float* st = conv_state + (size_t)seq_slot[b] * (taps - 1) * channels;      // [taps-1, channels], oldest first
    float acc = bias ? bias[c] : 0.f;
    for (int j = 0; j < taps; ++j) {
        const int at = ti - (taps - 1) + j;                 // index among the step's tokens; negative: from the state
        const float v = at >= 0 ? to_float(x[(row0 + at) * x_stride + c]) : st[(size_t)(taps - 1 + at) * channels + c];
        acc = fmaf(w[(size_t)c * taps + j], v, acc);
    }
    out[(row0 + ti) * channels + c] = from_float<T>(silu_f(acc));
}

// The same for four neighbouring channels and a run of tokens a thread: the last inputs stay in registers, so that an input is read
// once and not once a tap, in eight or sixteen bytes a lane, four tokens' reads under way together.  What bounds it is memory (2,603
// rows of 8,192 channels out of 16,384, bfloat16: 85 MB; 33 us, 140 with a thread a token and channel).  The sum's order is the same.
constexpr int CONV_RUN = 16, CONV_AHEAD = 4;

__device__ inline void conv_load4(const float* p, float (&v)[4]) {
    const float4 t = *reinterpret_cast<const float4*>(p);
    v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
}
__device__ inline void conv_load4(const bf16_t* p, float (&v)[4]) {
    const uint2 t = *reinterpret_cast<const uint2*>(p);
    v[0] = __uint_as_float(t.x << 16); v[1] = __uint_as_float(t.x & 0xffff0000u);
    v[2] = __uint_as_float(t.y << 16); v[3] = __uint_as_float(t.y & 0xffff0000u);
}
__device__ inline void conv_store4(float* p, const float (&v)[4]) { *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]); }
__device__ inline void conv_store4(bf16_t* p, const float (&v)[4]) {
    *reinterpret_cast<uint2*>(p) = make_uint2((uint32_t)f32_to_bf16(v[0]).bits | ((uint32_t)f32_to_bf16(v[1]).bits << 16),
                                              (uint32_t)f32_to_bf16(v[2]).bits | ((uint32_t)f32_to_bf16(v[3]).bits << 16));
}

// grid (blocks of 4 blockDim channels, runs of CONV_RUN tokens, sequences); channels a multiple of four
template <typename T, int TAPS>
__global__ void causal_conv_run_kernel(const T* __restrict__ x, int x_stride, const float* __restrict__ w, const float* __restrict__ bias,
                                       const float* __restrict__ conv_state, const int* __restrict__ seq_slot, const int* __restrict__ seq_new,
                                       const int* __restrict__ cu_new, int channels, T* __restrict__ out) {
    const int c = (blockIdx.x * blockDim.x + threadIdx.x) * 4, t0 = blockIdx.y * CONV_RUN, b = blockIdx.z;
    const int n_new = seq_new[b];
    if (c >= channels || t0 >= n_new) return;
    const T* xs = x + (size_t)cu_new[b] * x_stride + c;
    const float* st = conv_state + (size_t)seq_slot[b] * (TAPS - 1) * channels + c;       // [taps-1, channels], oldest first
    float wv[4][TAPS], first[4], last[TAPS][4];             // last[j]: the input j - (taps-1) tokens back; the newest one goes to last[taps-1]
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        first[e] = bias ? bias[c + e] : 0.f;
#pragma unroll
        for (int j = 0; j < TAPS; ++j) wv[e][j] = w[(size_t)(c + e) * TAPS + j];
    }
#pragma unroll
    for (int j = 0; j < TAPS - 1; ++j) {
        const int at = t0 - (TAPS - 1) + j;                 // negative: from the state
        if (at >= 0) conv_load4(xs + (size_t)at * x_stride, last[j]);
        else {
#pragma unroll
            for (int e = 0; e < 4; ++e) last[j][e] = st[(size_t)(TAPS - 1 + at) * channels + e];
        }
    }
    T* to = out + ((size_t)cu_new[b] + t0) * channels + c;
    for (int i = 0; i < CONV_RUN && t0 + i < n_new; i += CONV_AHEAD) {
        float in[CONV_AHEAD][4];
#pragma unroll
        for (int a = 0; a < CONV_AHEAD; ++a) conv_load4(xs + (size_t)min(t0 + i + a, n_new - 1) * x_stride, in[a]);
#pragma unroll
        for (int a = 0; a < CONV_AHEAD; ++a) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                last[TAPS - 1][e] = in[a][e];
                float acc = first[e];
#pragma unroll
                for (int j = 0; j < TAPS; ++j) acc = fmaf(wv[e][j], last[j][e], acc);
                v[e] = silu_f(acc);
#pragma unroll
                for (int j = 0; j < TAPS - 1; ++j) last[j][e] = last[j + 1][e];
            }
            if (t0 + i + a < n_new) conv_store4(to + (size_t)(i + a) * channels, v);
        }
    }
}

// A run takes its 10 us whatever the work, a thread for every token and channel a launch's 6 and then what the work asks (us, one
// at a time and in runs, four taps, 2,048 channels: 300 tokens 8.6 and 10.5, 600 11 and 11, 2,600 29 and 17; 8,192 channels: 64 tokens
// 7.7 and 10.5, 200 13 and 11).  The blocks of short sequences beside a long one cost a little too (41 sequences, one of 2,000 tokens,
// 1,000 channels: 147 and 12).
constexpr long long CONV_RUN_WORK = 5ll << 18, CONV_RUN_GRID = 8ll << 20;       // elements of the step, and of its grid

PALM_API int palm_causal_conv(hipStream_t stream, const void* x, int dtype, int x_stride, const float* w, const float* bias,
                              float* conv_state, const int* seq_slot, const int* seq_new, const int* cu_new, int n_seqs,
                              int max_new, int n_tokens, int channels, int taps, void* out) {
    PALM_CHECK(n_seqs >= 0 && max_new >= 0 && channels > 0, "causal_conv: seqs=%d max_new=%d channels=%d", n_seqs, max_new, channels);
    PALM_CHECK(taps >= 1 && taps <= CONV_MAX_TAPS, "causal_conv: %d taps (1 to %d)", taps, CONV_MAX_TAPS);
    PALM_CHECK(n_seqs <= 65535 && max_new <= 65535, "causal_conv: %d sequences / %d tokens are more than one launch takes", n_seqs, max_new);
    if (n_seqs == 0 || max_new == 0) return 0;
    const int threads = 256, cb = (channels + threads - 1) / threads;
    // runs of tokens where there is work for them, for the tap counts that models use, rows that start on whole reads
    const size_t read = dtype == PALM_F32 ? 16 : 8;
    const bool much = (long long)n_tokens * channels >= CONV_RUN_WORK || (long long)max_new * n_seqs * channels >= CONV_RUN_GRID;
    const bool runs = much && max_new >= CONV_RUN && (taps == 3 || taps == 4) && channels % 4 == 0 && x_stride % 4 == 0 &&
                      ((uintptr_t)x | (uintptr_t)out) % read == 0;
    const dim3 run_grid((channels / 4 + threads - 1) / threads, (max_new + CONV_RUN - 1) / CONV_RUN, n_seqs);
    PALM_DTYPE_SWITCH(dtype, T, {
        if (runs && taps == 4)
            causal_conv_run_kernel<T, 4><<<run_grid, threads, 0, stream>>>(
                (const T*)x, x_stride, w, bias, conv_state, seq_slot, seq_new, cu_new, channels, (T*)out);
        else if (runs)
            causal_conv_run_kernel<T, 3><<<run_grid, threads, 0, stream>>>(
                (const T*)x, x_stride, w, bias, conv_state, seq_slot, seq_new, cu_new, channels, (T*)out);
        else
            causal_conv_kernel<T><<<dim3(cb, max_new, n_seqs), threads, 0, stream>>>(
                (const T*)x, x_stride, w, bias, conv_state, seq_slot, seq_new, cu_new, channels, taps, (T*)out);
        if (taps > 1)
            conv_state_kernel<T><<<dim3(cb, n_seqs), threads, 0, stream>>>((const T*)x, x_stride, conv_state, seq_slot, seq_new,
                                                                          cu_new, channels, taps);
    });
    PALM_LAUNCHED();
    return 0;
}

// ---- the scan ---------------------------------------------------------------------------------------
// A channel's row of S is spread over a group of G lanes (G a power of two, at most 64): lane j of the group holds the PER states
// from j PER on, of 128 states and more j, j + G, ..; a block of four waves serves 256 / G channels.  The block walks over a sequence's new tokens a tile at a time,
// in three phases with a barrier between them:
//   in     all threads bring the tile's inputs into LDS with reads that follow the memory's rows: B_t and C_t (the
//          same for all channels), and for the block's channels the step size softplus(dtl_t + bias) and its product
//          with u_t, computed once for each (token, channel)
//   scan   for every token a lane updates its states from LDS; nothing but the multiply-add on S waits for the token
//          before it.  A whole tile's sums over the groups are made together (group_sums), without a branch between tokens
//   out    all threads add the skip term, gate with silu(z_t) and store the tile's outputs row by row
// Up to 64 states the next tile's inputs are asked for before the scan and wait in registers (with more a thread has more of
// them to hold, and fewer blocks fit).  A part tile goes token by token: unrolled, it costs the registers of another wave a SIMD.
// What bounds it is the vector unit (11 instructions a token and state, beside those of a token) and, once the short sequences are
// done, the chain of tiles.  8,192 channels x 16 states, us, with sums and a branch a token, one state a lane and the library's softplus
// and silu, and now: 2,603 tokens 417 and 253, 717 + 572 + 1,314 330 and 218, 8 x 300 245 and 135, one token each of 64 sequences 38.6
// and 32.6; 2,048 channels x 64 states, 717 + 572 + 1,314, 437 and 203.  (A token's operands read from LDS four tokens ahead: a chain of
// 2,603 233 and 202, but 64 single tokens 32.6 and 37.5, 128 states 438 and 539; outputs stored a tile later, so that the wait for
// the next inputs is none for stores: 3 % slower.)
constexpr int SCAN_TILE = 16;

// Sum over groups of G consecutive lanes (G a power of two), every lane gets its group's sum.  Within a row of 16
// lanes the partners come through the data-parallel lane crossbar of the vector unit (one instruction a step: quads
// swap, halves of 8 and rows of 16 mirror: any pairing of disjoint partial sums does); only steps across rows go
// through the permute unit.
template <int CTRL> __device__ inline float dpp_move(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
template <int G> __device__ inline float group_sum(float y) {
    if constexpr (G >= 2) y += dpp_move<0xB1>(y);            // quad_perm [1, 0, 3, 2]
    if constexpr (G >= 4) y += dpp_move<0x4E>(y);            // quad_perm [2, 3, 0, 1]
    if constexpr (G >= 8) y += dpp_move<0x141>(y);           // row_half_mirror
    if constexpr (G >= 16) y += dpp_move<0x140>(y);          // row_mirror
    if constexpr (G >= 32) y += __shfl_xor(y, 16, WAVE);
    if constexpr (G >= 64) y += __shfl_xor(y, 32, WAVE);
    return y;
}
// The sums over a group's lanes of TG values at once, TG the group's size or 16 of it: lane j (j + 16, ..) gets the sum of y[j].  A step
// halves the values, each lane keeping those of its half and handing on the others': 15 additions and 30 selections for 16 values and
// lanes, where one after the other they take 64 additions and a write of one lane each, with a branch around it.  The
// widest step comes first, so that mirrored partners hold the same values.
template <int H> __device__ inline void fold_half(float* y, int j) {
    constexpr int CTRL = H == 8 ? 0x140 : H == 4 ? 0x141 : H == 2 ? 0x4E : 0xB1;
    const bool upper = j & H;
#pragma unroll
    for (int i = 0; i < H; ++i) {
        const float keep = upper ? y[i + H] : y[i], give = upper ? y[i] : y[i + H];
        y[i] = keep + dpp_move<CTRL>(give);
    }
}
template <int G> __device__ inline float group_sums(float* y, int j) {
    if constexpr (G >= 16) fold_half<8>(y, j);
    if constexpr (G >= 8) fold_half<4>(y, j);
    fold_half<2>(y, j);
    fold_half<1>(y, j);
    float sum = y[0];
    if constexpr (G >= 32) sum += __shfl_xor(sum, 16, WAVE);
    if constexpr (G >= 64) sum += __shfl_xor(sum, 32, WAVE);
    return sum;
}
// exp(dt A) for an A that stays: 2^(dt A log2 e) with the product's rounding and that of A log2 e made up for in first order, so that
// the error is the exponential unit's own and not that of a rounded argument.  Below 2^-150: 0, as any 32-bit exponential.
struct ScanDecay {
    float hi, lo;                                       // A log2 e and, times ln 2, what hi leaves of it
    float most;                                         // the step from which on nothing is left
    __device__ static ScanDecay of(float a) {
        constexpr float LOG2E = 1.44269504f, LOG2E_REST = 1.92596299e-8f, LN2 = 0.693147181f;
        if (a < -2e38f) a = -2e38f;                     // (hi stays finite; no number stays none)
        ScanDecay d;
        d.hi = a * LOG2E;
        d.lo = (fmaf(a, LOG2E, -d.hi) + a * LOG2E_REST) * LN2;
        d.most = a < 0.f ? -150.f / d.hi : __builtin_inff();
        return d;
    }
    __device__ float over(float dt) const {
        constexpr float LN2 = 0.693147181f;
        dt = fminf(dt, most);
        const float p = dt * hi, rest = fmaf(fmaf(dt, hi, -p), LN2, dt * lo), e = __builtin_amdgcn_exp2f(p);
        return fmaf(e, rest, e);
    }
};
// What a (token, channel) of the scan needs once, its softplus and its silu: 119 and 33 instructions of the library's, where a token's
// sixteen states take some 200 between them.  Arguments for which a step leaves the normal numbers, and what is no number, go to the
// library (behind a branch: the compiler would go both ways).
__device__ inline float scan_exp(float x) {             // |x| < 87: 2^f of the fraction, the whole powers exact
    constexpr float LOG2E = 1.44269504f, LOG2E_REST = 1.92596299e-8f;
    const float n = rintf(x * LOG2E);
    return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(fmaf(x, LOG2E_REST, fmaf(x, LOG2E, -n))), (int)n);
}
// log(1 + e^z) = max(z, 0) + log(1 + e), e = e^-|z|, and log(1 + e) = 2 artanh(s) with s = e / (2 + e), where 2 s = e - e s: what is
// rounded in s is small beside e.  s^2 <= 1/9: the series' terms from the ninth on are below 2^-29.
__device__ inline float scan_softplus(float z) {
    if (!(fabsf(z) < 87.f)) {
        asm volatile("" : "+v"(z));
        return softplus_dt(z);
    }
    const float e = scan_exp(-fabsf(z)), d = 2.f + e, d_rest = e - (d - 2.f), r = __builtin_amdgcn_rcpf(d), q = e * r;
    const float s = fmaf(fmaf(-d_rest, q, fmaf(-d, q, e)), r, q), t = s * s;
    float sum = 2.f / 17;
    sum = fmaf(sum, t, 2.f / 15);
    sum = fmaf(sum, t, 2.f / 13);
    sum = fmaf(sum, t, 2.f / 11);
    sum = fmaf(sum, t, 2.f / 9);
    sum = fmaf(sum, t, 2.f / 7);
    sum = fmaf(sum, t, 2.f / 5);
    sum = fmaf(sum, t, 2.f / 3);
    return fmaxf(z, 0.f) + fmaf(s, fmaf(t, sum, -e), e);
}
__device__ inline float scan_silu(float z) {
    if (!(fabsf(z) < 87.f)) {
        asm volatile("" : "+v"(z));
        return silu_f(z);
    }
    const float d = 1.f + scan_exp(-z), r = __builtin_amdgcn_rcpf(d), q = z * r;
    return fmaf(fmaf(-d, q, z), r, q);
}
constexpr int SCAN_WAVES = 4;
constexpr int SCAN_THREADS = SCAN_WAVES * WAVE;

template <typename T, int G, int PER>
__global__ __launch_bounds__(SCAN_THREADS) void selective_scan_kernel(
    const T* __restrict__ u, const T* __restrict__ z, int z_stride, const T* __restrict__ bc, int bc_stride, int b_off, int c_off,
    const float* __restrict__ dtl, const float* __restrict__ dt_bias, const float* __restrict__ a_log,
    const float* __restrict__ d_skip, float* __restrict__ state, const int* __restrict__ seq_slot,
    const int* __restrict__ seq_new, const int* __restrict__ cu_new, int channels, int n_state, T* __restrict__ out) {
    constexpr bool AHEAD = G * PER <= 64;
    constexpr int CH = SCAN_THREADS / G;               // channels of a block
    constexpr int NP = G * PER;                        // the state size, padded
    constexpr int NB = (SCAN_TILE * NP + SCAN_THREADS - 1) / SCAN_THREADS, NC = (SCAN_TILE * CH + SCAN_THREADS - 1) / SCAN_THREADS;
    // of B and C at a time: all, but where that costs blocks a compute unit (128 states, eight at a time: 88 registers and five waves a
    // SIMD; 2,048 channels, 717 + 572 + 1,314 tokens 694 us, in halves 617; one token each of 64 sequences 84 and 65).  (256 states:
    // LDS sets the number of blocks; in quarters 1,139 us, 981 all together.)  A tile of few tokens does not go through the rest: 64
    // sequences of one token, with it and without, 128 states 64 us and 59, 256 states, a token an element, 143 and 122.
    constexpr int HELD = NP == 128 ? 4 : NB;
    constexpr bool BY_TOKEN = NP == SCAN_THREADS;      // element first + i of every thread is of token first + i
    constexpr int TG = G < 16 ? G : 16;                // tokens whose sums are made at once
    __shared__ __attribute__((aligned(16))) float2 bc_s[SCAN_TILE][NP];        // B_t and C_t
    __shared__ float2 in_s[SCAN_TILE][CH];             // the step size, and times u_t
    __shared__ float y_s[SCAN_TILE][CH];
    const int j = threadIdx.x % G, ch = threadIdx.x / G;
    // The states of lane j.  Side by side, a token's B and C come in one read of LDS; but the lanes' reads of S and of a_log then lie PER numbers
    // apart, and with rows of 128 states and more those are most of a single token's time: side by side and G apart, us, one token each of 16
    // and 64 sequences, 2,048 channels x 128 states 19.0 14.4 and 60.0 49.7, 1,024 x 256 19.7 16.5 and 66.2 62.3; 200 of 200 states (2,048)
    // 422 442; prompts the same to 2 %.
    auto state_of = [&](int k) { return NP >= 128 ? j + k * G : j * PER + k; };
    const int c0 = blockIdx.x * CH, b = blockIdx.y;
    const int c = c0 + ch;
    const bool mine = c < channels;
    const int cc = mine ? c : channels - 1;
    const int n_new = seq_new[b];
    const size_t row0 = (size_t)cu_new[b];
    float* sp = state + ((size_t)seq_slot[b] * channels + cc) * n_state;
    float S[PER];
    ScanDecay A[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int n = state_of(k);
        S[k] = n < n_state ? sp[n] : 0.f;
        A[k] = ScanDecay::of(n < n_state ? -expf(a_log[(size_t)cc * n_state + n]) : 0.f);
    }
    // this thread's elements of a tile: idx = threadIdx + i SCAN_THREADS is token idx / NP (idx / CH), state (channel) the rest
    T b_r[HELD], c_r[HELD], u_r[NC], z_r[NC];          // (as they lie in memory: a conversion would wait for each)
    float dt_r[NC], skip[NC], bias[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        const int idx = threadIdx.x + i * SCAN_THREADS, ck = min(c0 + idx % CH, channels - 1);
        skip[i] = bias[i] = 0.f;
        if (idx / CH >= n_new) continue;
        skip[i] = d_skip[ck];
        bias[i] = dt_bias[ck];
    }
    auto ask_states = [&](int t0, int first) {         // (tokens beyond the sequence are not read and not used)
#pragma unroll
        for (int i = 0; i < HELD; ++i) {
            const int idx = threadIdx.x + (first + i) * SCAN_THREADS, n = idx % NP;
            if (BY_TOKEN && t0 + first + i >= n_new) break;
            b_r[i] = c_r[i] = T{};
            if (n >= n_state || t0 + idx / NP >= n_new) continue;
            const T* r = bc + (row0 + t0 + idx / NP) * bc_stride;
            b_r[i] = r[b_off + n];
            c_r[i] = r[c_off + n];
        }
    };
    auto keep_states = [&](int tt, int first) {
#pragma unroll
        for (int i = 0; i < HELD; ++i) {
            const int idx = threadIdx.x + (first + i) * SCAN_THREADS;
            if (BY_TOKEN && first + i >= tt) break;
            if (idx / NP < tt) bc_s[idx / NP][idx % NP] = make_float2(to_float(b_r[i]), to_float(c_r[i]));
        }
    };
    // (where a tile has fewer elements than the block threads, the threads beyond it read the next tiles': nearer when their turn
    // comes.  Leaving them out was 7 to 9 % slower for 64 and 128 states.)
    auto ask_channels = [&](int t0) {
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const int idx = threadIdx.x + i * SCAN_THREADS, ck = min(c0 + idx % CH, channels - 1);
            dt_r[i] = 0.f;
            u_r[i] = z_r[i] = T{};
            if (t0 + idx / CH >= n_new) continue;
            const size_t row = row0 + t0 + idx / CH;
            dt_r[i] = dtl[row * channels + ck];
            u_r[i] = u[row * channels + ck];
            z_r[i] = z[row * z_stride + ck];
        }
    };
    if (AHEAD) { ask_states(0, 0); ask_channels(0); }
    for (int t0 = 0; t0 < n_new; t0 += SCAN_TILE) {
        const int tt = min(SCAN_TILE, n_new - t0);
        if (!AHEAD) ask_channels(t0);
        float u_t[NC], z_t[NC];
#pragma unroll 1
        for (int first = 0; first < NB && (HELD == NB || first * SCAN_THREADS < tt * NP); first += HELD) {
            if (!AHEAD) ask_states(t0, first);
            keep_states(tt, first);
        }
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const int idx = threadIdx.x + i * SCAN_THREADS;
            if (idx / CH < tt) {
                const float dt = scan_softplus(dt_r[i] + bias[i]);
                in_s[idx / CH][idx % CH] = make_float2(dt, dt * to_float(u_r[i]));
            }
            u_t[i] = to_float(u_r[i]);
            z_t[i] = to_float(z_r[i]);
        }
        __syncthreads();
        if (AHEAD && t0 + SCAN_TILE < n_new) { ask_states(t0 + SCAN_TILE, 0); ask_channels(t0 + SCAN_TILE); }        // on their way while this tile is scanned
        auto token = [&](int ti) __attribute__((always_inline)) {
            const float2 in = in_s[ti][ch];
            float y = 0.f;
#pragma unroll
            for (int k = 0; k < PER; ++k) {
                const float2 v = bc_s[ti][state_of(k)];
                S[k] = fmaf(A[k].over(in.x), S[k], in.y * v.x);              // beyond the state size A, B and C are zero
                y = fmaf(S[k], v.y, y);
            }
            return y;
        };
        if (tt == SCAN_TILE) {                                  // a whole tile: no test between its tokens
#pragma unroll
            for (int t = 0; t < SCAN_TILE; t += TG) {
                float y[TG];
#pragma unroll
                for (int i = 0; i < TG; ++i) y[i] = token(t + i);
                const float sum = group_sums<G>(y, j);
                if (G == TG || j < TG) y_s[t + j % TG][ch] = sum;
            }
        } else {
#pragma unroll 1
            for (int ti = 0; ti < tt; ++ti) {
                const float y = group_sum<G>(token(ti));
                if (j == 0) y_s[ti][ch] = y;
            }
        }
        __syncthreads();
        // the next tile's elements may go to LDS while these are read: y_s is written behind the next barrier only
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const int idx = threadIdx.x + i * SCAN_THREADS, ti = idx / CH, k = idx % CH;
            if (ti < tt && c0 + k < channels) {
                const float y = fmaf(skip[i], u_t[i], y_s[ti][k]);
                out[(row0 + t0 + ti) * channels + c0 + k] = from_float<T>(y * scan_silu(z_t[i]));
            }
        }
    }
    if (mine && n_new > 0) {
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int n = state_of(k);
            if (n < n_state) sp[n] = S[k];
        }
    }
}

PALM_API int palm_selective_scan(hipStream_t stream, const void* u, const void* z, int z_stride, const void* bc, int bc_stride,
                                 int b_off, int c_off, int dtype, const float* dtl, const float* dt_bias, const float* a_log,
                                 const float* d_skip, float* state, const int* seq_slot, const int* seq_new, const int* cu_new,
                                 int n_seqs, int channels, int n_state, void* out) {
    PALM_CHECK(n_seqs >= 0 && channels > 0 && n_state > 0, "selective_scan: seqs=%d channels=%d state=%d", n_seqs, channels, n_state);
    PALM_CHECK(n_state <= 256, "selective_scan: a state of %d per channel exceeds 256", n_state);
    PALM_CHECK(n_seqs <= 65535, "selective_scan: %d sequences are more than one launch takes", n_seqs);
    if (n_seqs == 0) return 0;
#define SCAN_CASE(G, PER) { \
        const int per_block = SCAN_THREADS / G; \
        dim3 grid((channels + per_block - 1) / per_block, n_seqs); \
        selective_scan_kernel<T, G, PER><<<grid, SCAN_THREADS, 0, stream>>>((const T*)u, (const T*)z, z_stride, \
            (const T*)bc, bc_stride, b_off, c_off, dtl, dt_bias, a_log, d_skip, state, seq_slot, seq_new, cu_new, channels, n_state, (T*)out); }
    // States a lane: one, while that leaves each SIMD no more than four waves (a long sequence is a chain of its tokens, and a lane with
    // more states takes longer over each); else two or four, which share a token's reads and the sums over the group.  us with one,
    // two and four: 8,192 channels x 16 states, 2,603 tokens (2,048 waves) 253, 337, 548; 717 + 572 + 1,314 (6,144) 229, 218, 308;
    // 8 x 300 155, 135, 132; 2,048 channels x 64 states, 717 + 572 + 1,314 (6,144) 240, 203, 251; 8 x 300 (16,384) 179, 130, 113;
    // 128 states, two and four, 6,144 waves 438 and 456, 16,384 waves 302 and 243.  Up to eight states one is always the fastest.
    const long long lanes = n_state <= 8 ? 8 : n_state <= 16 ? 16 : n_state <= 32 ? 32 : 64, waves = lanes * n_seqs * channels / WAVE;
    const bool many = waves > 4096, more = waves > 8192;
    PALM_DTYPE_SWITCH(dtype, T, {
        if (n_state <= 4) SCAN_CASE(4, 1)
        else if (n_state <= 8) SCAN_CASE(8, 1)
        else if (n_state <= 16 && many) SCAN_CASE(8, 2)
        else if (n_state <= 16) SCAN_CASE(16, 1)
        else if (n_state <= 32 && many) SCAN_CASE(16, 2)
        else if (n_state <= 32) SCAN_CASE(32, 1)
        else if (n_state <= 64 && more) SCAN_CASE(16, 4)
        else if (n_state <= 64 && many) SCAN_CASE(32, 2)
        else if (n_state <= 64) SCAN_CASE(64, 1)
        else if (n_state <= 128 && more) SCAN_CASE(32, 4)
        else if (n_state <= 128) SCAN_CASE(64, 2)
        else SCAN_CASE(64, 4)
    });
#undef SCAN_CASE
    PALM_LAUNCHED();
    return 0;
}
