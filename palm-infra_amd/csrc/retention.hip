// Retention: linear attention with one fixed decay per head, no softmax and no denominator.
//
//   S_t = g_h S_(t-1) + k_t v_t^T        S: [dim, vdim] per sequence and head, 32-bit, kept between steps
//   o_t = S_t^T q_t
//   out_t = o_t / sqrt(mean_v(o_t^2) + eps) * silu(gate_t)         (the unit norm is per head)
//
// q and k are rotated first (pairs (i, i + rot/2) of the first `rot` dimensions, cos/sin rows of the tokens'
// positions) and k is multiplied by k_scale after the rotation; rotated values, state and sums are 32-bit.
//
// Two options make this the recurrence of other linear attentions as well: `act` puts q, k and v through silu first
// (q and k before the rotation), and `joined` leaves out the per-head unit norm and the gate: the heads' o_t are then
// written as they are, 32-bit, and a pass of its own norms a token's joined heads together, with a weight, and gates
// them (palm_joined_norm_gate).
//
// A first pass rotates q and k of all the step's tokens into 32-bit rows.  Runs of new tokens then go through the matrix cores
// in chunks (retention_local_kernel and what follows it); single tokens, short runs and other sizes walk over their tokens as
// linear_recurrence.h does.
#include "linear_recurrence.h"

// q and k of every token and head, rotated (k also scaled), 32-bit: qk[row][head][0 = q, 1 = k][pad], pad >= dim the
// key size that the main kernel is compiled for; the columns beyond dim are zero, so that the main kernel's loops
// over pad need no test (a zero k leaves its row of S zero, a zero q adds nothing).
template <typename T>
__global__ void retention_rotate_kernel(const T* __restrict__ qkvg, int row_stride, int q_off, int k_off,
                                        const float* __restrict__ cos_t, const float* __restrict__ sin_t, int rot, float k_scale,
                                        int act, int n_tokens, int heads, int dim, int pad, float* __restrict__ qk) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)n_tokens * heads * pad) return;
    const int d = (int)(idx % pad), h = (int)((idx / pad) % heads);
    const size_t row = (size_t)(idx / ((long long)pad * heads));
    float* o = qk + ((row * heads + h) * 2) * pad + d;
    if (d >= dim) { o[0] = 0.f; o[pad] = 0.f; return; }
    const int half = rot / 2;
    const T* qr = qkvg + row * row_stride + q_off + h * dim;
    const T* kr = qkvg + row * row_stride + k_off + h * dim;
    float qv = to_float(qr[d]), kv = to_float(kr[d]);
    if (act) { qv = rec_silu(qv); kv = rec_silu(kv); }
    if (d < rot) {
        const int i = d < half ? d : d - half;
        const float c = cos_t[row * half + i], sn = sin_t[row * half + i];
        const int partner = d < half ? d + half : d - half;
        float qp = to_float(qr[partner]), kp = to_float(kr[partner]);
        if (act) { qp = rec_silu(qp); kp = rec_silu(kp); }
        // the pair (u, w) becomes (u c - w s, w c + u s)
        qv = d < half ? qv * c - qp * sn : qv * c + qp * sn;
        kv = d < half ? kv * c - kp * sn : kv * c + kp * sn;
    }
    o[0] = qv;
    o[pad] = kv * k_scale;
}

// ---- a prompt's chunks on the matrix cores ----------------------------------------------------------------------------
// Token by token a chunk of C tokens is C dependent passes over S, and the linear recurrence's chunks walk twice: 2,600 tokens
// of 16 heads (key size 128, value size 256) took 940 us, a fifth of the vector units' rate, bound by the chain.  In matrix form
// a chunk that starts from S is
//   L = (K o w)^T V,  w_t = g^(n-1-t)                     what it adds to the state  (retention_local_kernel)
//   O = ((Q K^T) o D) V + (Q o u) S,  D_ts = g^(t-s) for s <= t, u_t = g^(t+1)      (retention_out_kernel)
// and the states between the chunks are the same elementwise walk as before, with the next chunk's sum read ahead.  All of it
// is 32-bit: v_mfma_f32_16x16x4 multiplies and adds 32-bit numbers, at twice the vector units' rate.
// Those 2,603 tokens (three sequences) now take 206 us with the pass that rotates q and k: 57 the sums, 35 the states, 90 the
// outputs; what bounds it is the reads of S and of the chunks' sums (64 tokens share 128 KB of S) and the matrix cores, half each.
//
// Operands: lane l = 16 g + r of a wave brings row r (A) or column r (B) and the k-value g of an instruction.  Which token, key
// or value dimension a row, column or k stands for is free, so every lane reads runs: 4 key dimensions of q and k (four
// instructions, element e of every lane each), VT neighbouring value dimensions of V and S (tile e is made of dimensions
// VT r + e).  A lane of a result then holds 4 VT neighbouring value dimensions of one token, or of one row of S.
// A block of four waves serves a (head, chunk, sequence), wave w the value dimensions 16 VT w .. : sizes of 64 VT.
// Chunk c of sequence b has place cu_new[b] / C + b + c: no two share one, a sequence's lie side by side, and they are at most
// n_tokens / C + n_seqs.  The starts have room for a window of RET_ROOM bytes of them, and the three kernels take one window of
// places after the other (16 heads of 128 x 256: 64 places, 4,096 tokens; a window is then 1,024 blocks, so the cuts cost nothing:
// 8,192 tokens 585 us with room for all, 566 in windows).
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int RET_CHUNK = 64;
constexpr long long RET_ROOM = 128ll << 20;

__device__ inline f32x4 ret_mfma(float a, float b, f32x4 acc) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0); }
template <int N> struct RetRun { float v[N]; };
template <int N> __device__ inline RetRun<N> ret_run(const float* p) {
    RetRun<N> o;
    if constexpr (N % 4 == 0) {
#pragma unroll
        for (int i = 0; i < N; i += 4) { const float4 q = *reinterpret_cast<const float4*>(p + i); o.v[i] = q.x; o.v[i + 1] = q.y; o.v[i + 2] = q.z; o.v[i + 3] = q.w; }
    } else {
        const float2 q = *reinterpret_cast<const float2*>(p);
        o.v[0] = q.x; o.v[1] = q.y;
    }
    return o;
}
template <int N> __device__ inline RetRun<N> ret_run(const bf16_t* p) {
    RetRun<N> o;
    uint32_t w[N / 2];
    if constexpr (N % 4 == 0) {
#pragma unroll
        for (int i = 0; i < N / 2; i += 2) { const uint2 q = *reinterpret_cast<const uint2*>(p + 2 * i); w[i] = q.x; w[i + 1] = q.y; }
    } else {
        w[0] = *reinterpret_cast<const uint32_t*>(p);
    }
#pragma unroll
    for (int i = 0; i < N / 2; ++i) { o.v[2 * i] = __uint_as_float(w[i] << 16); o.v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u); }
    return o;
}
__device__ inline void ret_store_run4(float* p, float a, float b, float c, float d) { *reinterpret_cast<float4*>(p) = make_float4(a, b, c, d); }
__device__ inline void ret_store_run4(bf16_t* p, float a, float b, float c, float d) {
    uint2 w;
    w.x = (uint32_t)f32_to_bf16(a).bits | ((uint32_t)f32_to_bf16(b).bits << 16);
    w.y = (uint32_t)f32_to_bf16(c).bits | ((uint32_t)f32_to_bf16(d).bits << 16);
    *reinterpret_cast<uint2*>(p) = w;
}

struct RetChunk {
    int row0, n;                 // the first row of a place's chunk and how many tokens it has (<= 0: none)
    __device__ RetChunk(const int* seq_new, const int* cu_new, int n_seqs, int place) {
        const int lane = threadIdx.x % WAVE;
        row0 = n = 0;            // of the last sequence whose first place is not beyond this one
        for (int s0 = 0; s0 < n_seqs; s0 += WAVE) {
            const int s = s0 + lane, first = cu_new[min(s, n_seqs - 1)], count = seq_new[min(s, n_seqs - 1)];
            const unsigned long long at_or_before = __ballot(s < n_seqs && first / RET_CHUNK + s <= place);
            if (!at_or_before) break;
            const int at = __popcll(at_or_before) - 1, done = (place - (s0 + at) - __shfl(first, at, WAVE) / RET_CHUNK) * RET_CHUNK;
            row0 = __shfl(first, at, WAVE) + done;
            n = min(RET_CHUNK, __shfl(count, at, WAVE) - done);
        }
    }
};

template <typename T, int DIM, int VT>
__global__ __launch_bounds__(256) void retention_local_kernel(const T* __restrict__ rows, int row_stride, int v_off, const float* __restrict__ qk,
                                                              const float* __restrict__ decay, const int* __restrict__ seq_new,
                                                              const int* __restrict__ cu_new, int n_seqs, int place0, int heads, int act,
                                                              float* __restrict__ starts) {
    constexpr int VDIM = 64 * VT, DQ = DIM / 64;
    __shared__ float power[RET_CHUNK];
    const int h = blockIdx.x;
    const RetChunk chunk(seq_new, cu_new, n_seqs, place0 + blockIdx.y);
    const int n = chunk.n;
    if (n <= 0) return;
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE, r = lane % 16, g = lane / 16, v0 = wave * 16 * VT;
    if (threadIdx.x < RET_CHUNK) power[threadIdx.x] = powf(decay[h], (float)threadIdx.x);
    __syncthreads();
    f32x4 acc[DQ][4][VT];                                // columns: key dimensions 64 q + 4 r + e; rows: value dimensions v0 + VT (4 g + x) + ve
#pragma unroll
    for (int q = 0; q < DQ; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int ve = 0; ve < VT; ++ve) acc[q][e][ve] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int s = 0; s < (n + 3) / 4; ++s) {
        const int t = 4 * s + g, row = chunk.row0 + min(t, n - 1);
        const float w = power[max(n - 1 - t, 0)];
        RetRun<VT> vv = ret_run<VT>(rows + (size_t)row * row_stride + v_off + h * VDIM + v0 + VT * r);
#pragma unroll
        for (int ve = 0; ve < VT; ++ve) {                // (a token beyond the chunk: zeros on both sides, as zero times infinity is none)
            if (act) vv.v[ve] = rec_silu(vv.v[ve]);
            vv.v[ve] = t < n ? vv.v[ve] : 0.f;
        }
        const float* kr = qk + ((size_t)row * heads + h) * 2 * DIM + DIM + 4 * r;
#pragma unroll
        for (int q = 0; q < DQ; ++q) {
            const RetRun<4> kv = ret_run<4>(kr + 64 * q);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int ve = 0; ve < VT; ++ve) acc[q][e][ve] = ret_mfma(vv.v[ve], t < n ? kv.v[e] * w : 0.f, acc[q][e][ve]);
        }
    }
    float* out = starts + ((size_t)blockIdx.y * heads + h) * DIM * VDIM + v0 + 4 * VT * g;
#pragma unroll
    for (int q = 0; q < DQ; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < VT; ++i) {               // four neighbours: places 4 i .. of (x, ve)
                auto at = [&](int j) { return acc[q][e][(4 * i + j) % VT][(4 * i + j) / VT]; };
                ret_store_run4(out + (size_t)(64 * q + 4 * r + e) * VDIM + 4 * i, at(0), at(1), at(2), at(3));
            }
}

// One thread for four elements of (sequence, head, dim, vdim): starts holds L_c of the window's places and leaves as S_c, the state is
// left as it is behind the window's last chunk; the next L is on its way.
__global__ void retention_starts_kernel(float* __restrict__ starts, float* __restrict__ state, const float* __restrict__ decay,
                                        const int* __restrict__ seq_slot, const int* __restrict__ seq_new, const int* __restrict__ cu_new,
                                        int place0, int places, int heads, int per_head) {
    const int e = (blockIdx.x * blockDim.x + threadIdx.x) * 4, b = blockIdx.y;
    if (e >= heads * per_head) return;
    const int first = cu_new[b] / RET_CHUNK + b;         // the sequence's first place
    const int before = max(place0 - first, 0);            // chunks of earlier windows
    const int n_new = seq_new[b] - before * RET_CHUNK, chunks = min((n_new + RET_CHUNK - 1) / RET_CHUNK, place0 + places - first - before);
    if (n_new <= 0 || chunks <= 0) return;
    const float g = decay[e / per_head], whole = powf(g, (float)RET_CHUNK);
    const size_t stride = (size_t)heads * per_head;
    float4* st = reinterpret_cast<float4*>(state + (size_t)seq_slot[b] * stride + e);
    float* at = starts + (first + before - place0) * stride + e;
    constexpr int AHEAD = 4;
    float4 s = *st, local[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) local[i] = *reinterpret_cast<const float4*>(at + min(i, chunks - 1) * stride);
    for (int c0 = 0; c0 < chunks; c0 += AHEAD) {
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            const int c = c0 + i;
            if (c >= chunks) break;
            const float4 l = local[i];
            local[i] = *reinterpret_cast<const float4*>(at + min(c + AHEAD, chunks - 1) * stride);
            *reinterpret_cast<float4*>(at + c * stride) = s;
            const int n = min(RET_CHUNK, n_new - c * RET_CHUNK);
            const float keep = n == RET_CHUNK ? whole : powf(g, (float)n);
            s = make_float4(fmaf(keep, s.x, l.x), fmaf(keep, s.y, l.y), fmaf(keep, s.z, l.z), fmaf(keep, s.w, l.w));
        }
    }
    *st = s;
}

template <typename T, int DIM, int VT>
__global__ __launch_bounds__(256) void retention_out_kernel(const T* __restrict__ rows, int row_stride, int v_off, int g_off,
                                                            const float* __restrict__ qk, const float* __restrict__ decay, float eps,
                                                            const int* __restrict__ seq_new, const int* __restrict__ cu_new, int n_seqs, int place0,
                                                            int heads, int act, const float* __restrict__ starts, T* __restrict__ out, int joined,
                                                            float* __restrict__ raw) {
    constexpr int VDIM = 64 * VT, TT = RET_CHUNK / 16;
    __shared__ float power[RET_CHUNK + 1];
    __shared__ __attribute__((aligned(16))) float P[RET_CHUNK][RET_CHUNK + 4];
    __shared__ float squares[4][RET_CHUNK];
    const int h = blockIdx.x;
    const RetChunk chunk(seq_new, cu_new, n_seqs, place0 + blockIdx.y);
    const int n = chunk.n;
    if (n <= 0) return;
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE, r = lane % 16, g = lane / 16, v0 = wave * 16 * VT;
    if (threadIdx.x <= RET_CHUNK) power[threadIdx.x] = powf(decay[h], (float)threadIdx.x);
    __syncthreads();
    auto q_row = [&](int t) { return qk + ((size_t)(chunk.row0 + min(t, n - 1)) * heads + h) * 2 * DIM; };

    // the ten 16 x 16 tiles of Q K^T on and below the diagonal, spread over the waves: rows s = 16 j + 4 g + x, columns t = 16 i + r
    for (int tile = wave; tile < TT * (TT + 1) / 2; tile += 4) {
        const int i = tile >= 6 ? 3 : tile >= 3 ? 2 : tile >= 1 ? 1 : 0, j = tile - i * (i + 1) / 2;
        if (16 * i >= n) break;
        const float *q = q_row(16 * i + r) + 4 * g, *k = q_row(16 * j + r) + DIM + 4 * g;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int d = 0; d < DIM; d += 16) {
            const RetRun<4> qv = ret_run<4>(q + d), kv = ret_run<4>(k + d);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = ret_mfma(kv.v[e], qv.v[e], acc);
        }
        const int t = 16 * i + r, s = 16 * j + 4 * g;
        float p[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) p[x] = s + x <= t ? acc[x] * power[max(t - s - x, 0)] : 0.f;
        ret_store_run4(&P[t][s], p[0], p[1], p[2], p[3]);
    }

    f32x4 o[TT][VT];                                     // columns: tokens 16 i + r; rows: value dimensions v0 + VT (4 g + x) + ve
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int ve = 0; ve < VT; ++ve) o[i][ve] = f32x4{0.f, 0.f, 0.f, 0.f};
    float from_start[TT];
#pragma unroll
    for (int i = 0; i < TT; ++i) from_start[i] = power[16 * i + r + 1];
    const float* start = starts + ((size_t)blockIdx.y * heads + h) * DIM * VDIM + v0 + VT * r;
#pragma unroll 2
    for (int d = 0; d < DIM; d += 16) {
        RetRun<4> qv[TT];
        RetRun<VT> sv[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) sv[e] = ret_run<VT>(start + (size_t)(d + 4 * g + e) * VDIM);
#pragma unroll
        for (int i = 0; i < TT; ++i) qv[i] = ret_run<4>(q_row(16 * i + r) + d + 4 * g);
#pragma unroll
        for (int i = 0; i < TT; ++i) {
            if (16 * i >= n) continue;                   // the same in every lane
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float q = qv[i].v[e] * from_start[i];
#pragma unroll
                for (int ve = 0; ve < VT; ++ve) o[i][ve] = ret_mfma(sv[e].v[ve], q, o[i][ve]);
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int sb = 0; sb < TT; ++sb) {
        if (16 * sb >= n) continue;
        RetRun<VT> vv[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            vv[e] = ret_run<VT>(rows + (size_t)(chunk.row0 + min(16 * sb + 4 * g + e, n - 1)) * row_stride + v_off + h * VDIM + v0 + VT * r);
            if (act) {
#pragma unroll
                for (int ve = 0; ve < VT; ++ve) vv[e].v[ve] = rec_silu(vv[e].v[ve]);
            }
        }
        float odd = 0.f;                                 // a number unless one of the values is none, or infinite
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int ve = 0; ve < VT; ++ve) odd = fmaf(vv[e].v[ve], 0.f, odd);
        const bool finite = __ballot(odd != odd) == 0;
#pragma unroll
        for (int i = sb; i < TT; ++i) {                  // the tokens before the block see none of it
            if (16 * i >= n) continue;
            const RetRun<4> p = ret_run<4>(&P[16 * i + r][16 * sb + 4 * g]);
            if (i == sb && !finite) {
                // within the block zeros stand for what a token does not see, and zero times infinity is no number: a token at a
                // time, and only the tokens that see it take it in
#pragma unroll 1
                for (int from = 0; from < 4; ++from)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int ve = 0; ve < VT; ++ve) {
                            const f32x4 one = ret_mfma(g == from ? vv[e].v[ve] : 0.f, g == from ? p.v[e] : 0.f, f32x4{0.f, 0.f, 0.f, 0.f});
                            if (r >= 4 * from + e) o[i][ve] += one;
                        }
                continue;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int ve = 0; ve < VT; ++ve) o[i][ve] = ret_mfma(vv[e].v[ve], p.v[e], o[i][ve]);
        }
    }

    auto at = [&](int i, int place) { return o[i][place % VT][place / VT]; };          // of the lane's 4 VT neighbours
    if (!joined) {
#pragma unroll
        for (int i = 0; i < TT; ++i) {
            float ss = 0.f;
#pragma unroll
            for (int p = 0; p < 4 * VT; ++p) ss += at(i, p) * at(i, p);
            ss += __shfl_xor(ss, 16, WAVE);
            ss += __shfl_xor(ss, 32, WAVE);
            if (g == 0) squares[wave][16 * i + r] = ss;
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < TT; ++i) {
        const int t = 16 * i + r;
        if (t >= n) continue;
        const size_t row = (size_t)(chunk.row0 + t);
        const int col = h * VDIM + v0 + 4 * VT * g;
        if (joined) {
#pragma unroll
            for (int p = 0; p < 4 * VT; p += 4) ret_store_run4(raw + row * ((size_t)heads * VDIM) + col + p, at(i, p), at(i, p + 1), at(i, p + 2), at(i, p + 3));
            continue;
        }
        const float total = ((squares[0][t] + squares[1][t]) + squares[2][t]) + squares[3][t];
        const float inv = 1.0f / sqrtf(total / (float)VDIM + eps);
#pragma unroll
        for (int p = 0; p < 4 * VT; p += 4) {
            const RetRun<4> gate = ret_run<4>(rows + row * row_stride + g_off + col + p);
            float y[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = at(i, p + e) * inv * rec_silu(gate.v[e]);
            ret_store_run4(out + row * ((size_t)heads * VDIM) + col + p, y[0], y[1], y[2], y[3]);
        }
    }
}

// The chunk with which a step's runs can go through the kernels above, or 0: sizes that fill the waves' tiles, and runs longer than
// one walk should take (16 heads of 128 x 256: 8 tokens 30 us and 25 walked, 16 tokens 32 and 45, 2,048 tokens 138 and 535).
PALM_API int palm_retention_matrix_chunk(int dim, int vdim, int max_new) {
    return (dim == 64 || dim == 128) && (vdim == 128 || vdim == 256) && max_new >= 16 ? RET_CHUNK : 0;
}

// Whether they should.  In chunks a sequence's state crosses memory six times, once a single token as well, in the walk twice; the
// walk is the longest run's chain, slower with more blocks a compute unit (as many as all tokens make in runs of that length).  In
// us, what chunks spare of that against what they cost.  16 heads of 128 x 256, walked and in chunks: 63 single tokens beside 16
// new ones 77 and 190, beside 512 1,280 and 312, 17 tokens of each of 64 sequences 152 and 271, 30 of 32 139 and 137.
// Drawn from 1,196 steps timed both ways (2 to 64 heads, 1 to 128 sequences; equal runs, one or some among single tokens, ragged); at
// 500 others 0.4 % from the better way in the mean, 8 % behind the walk at worst, 49 % behind chunks (92 of 16 tokens, four heads).
PALM_API int palm_retention_matrix_pays(int heads, int dim, int vdim, int n_seqs, int n_tokens, int max_new) {
    if (!palm_retention_matrix_chunk(dim, vdim, max_new)) return 0;
    const double a_unit = (double)heads * n_tokens / max_new / 256, mb = (double)n_seqs * heads * dim * vdim * sizeof(float) / (1 << 20);
    const double few = min(ceil(a_unit), 3.0), crowded = vdim == 128 ? max(0.72 * few, 0.22 * a_unit) : max(0.56 * few, 0.37 * a_unit);
    return (0.41 + 0.0105 * dim) * max_new * max(1.0, crowded) > 7.1 + 0.92 * mb + 0.44 * max(mb - 128.0, 0.0);
}

// Places of chunks that the starts have room for (as many as n_tokens tokens of n_seqs sequences need, up to RET_ROOM bytes).
PALM_API int palm_retention_places(int heads, int dim, int vdim, int n_tokens, int n_seqs) {
    const long long room = max(1ll, RET_ROOM / ((long long)heads * dim * vdim * (long long)sizeof(float)));
    return (int)min(min(room, 65535ll), (long long)n_tokens / RET_CHUNK + n_seqs);
}

template <typename T, int DIM, int VT>
static void launch_retention_chunks(hipStream_t stream, const T* rows, int row_stride, int v_off, int g_off, const float* qk, const float* decay,
                                    float eps, float* state, const int* seq_slot, const int* seq_new, const int* cu_new, int n_seqs, int n_tokens,
                                    int heads, float* starts, T* out, int act, int joined, float* raw) {
    const int per_head = DIM * 64 * VT, all = n_tokens / RET_CHUNK + n_seqs, window = palm_retention_places(heads, DIM, 64 * VT, n_tokens, n_seqs);
    for (int place0 = 0; place0 < all; place0 += window) {
        const int places = min(window, all - place0);
        const dim3 grid(heads, places);
        retention_local_kernel<T, DIM, VT><<<grid, 256, 0, stream>>>(rows, row_stride, v_off, qk, decay, seq_new, cu_new, n_seqs, place0, heads, act, starts);
        retention_starts_kernel<<<dim3((heads * per_head / 4 + 255) / 256, n_seqs), 256, 0, stream>>>(starts, state, decay, seq_slot, seq_new, cu_new,
                                                                                                       place0, places, heads, per_head);
        retention_out_kernel<T, DIM, VT><<<grid, 256, 0, stream>>>(rows, row_stride, v_off, g_off, qk, decay, eps, seq_new, cu_new, n_seqs, place0, heads,
                                                                   act, starts, out, joined, raw);
    }
}

// qk: room for n_tokens * heads * 2 * pad floats (the rotated q and k; pad = palm_retention_pad(dim)).  chunk == 0: every sequence's run in one block
// per head.  Else `starts` holds n_seqs * max_chunks * heads * dim * vdim floats, max_chunks = ceil(max_new / chunk); with
// matrix != 0 (chunk = palm_retention_matrix_chunk, rows and offsets of whole 16-byte pieces) palm_retention_places * heads * dim * vdim.
PALM_API int palm_retention_pad(int dim) { return dim <= 32 ? 32 : dim <= 64 ? 64 : dim <= 128 ? 128 : 256; }

PALM_API int palm_retention(hipStream_t stream, const void* qkvg, int dtype, int row_stride, int q_off, int k_off, int v_off,
                            int g_off, const float* cos_t, const float* sin_t, int rot, const float* decay, float k_scale,
                            float eps, float* state, const int* seq_slot, const int* seq_new, const int* cu_new, int n_seqs,
                            int heads, int dim, int vdim, void* out, int max_new, int chunk, float* starts, int n_tokens,
                            float* qk, int act, int joined, float* raw, int matrix) {
    PALM_CHECK(n_seqs >= 0 && heads > 0 && dim > 0 && vdim > 0, "retention: seqs=%d heads=%d dim=%d vdim=%d", n_seqs, heads, dim, vdim);
    PALM_CHECK(dim <= 256, "retention: a key size of %d exceeds 256", dim);
    PALM_CHECK(vdim <= 1024, "retention: a value size of %d exceeds 1024", vdim);
    PALM_CHECK(rot >= 0 && rot <= dim && rot % 2 == 0, "retention: %d rotated dimensions of %d", rot, dim);
    PALM_CHECK(rot == 0 || (cos_t && sin_t), "retention: a rotation needs its cos and sin rows");
    PALM_CHECK(chunk >= 0 && (chunk == 0 || (starts && max_new > 0)), "retention: chunks of %d tokens need their starting states", chunk);
    PALM_CHECK(n_tokens >= 0 && (n_tokens == 0 || qk), "retention: the rotated q and k need their room");
    PALM_CHECK(n_tokens == 0 || (joined ? raw != nullptr : out != nullptr), "retention: the outputs need their room (32-bit rows if the heads are normed together later)");
    if (n_seqs == 0 || n_tokens == 0) return 0;
    const int max_chunks = chunk > 0 ? (max_new + chunk - 1) / chunk : 1;
    PALM_CHECK(heads <= 65535 && (matrix ? n_seqs <= 65535 && max_chunks <= 65535 : (long long)n_seqs * max_chunks <= 65535), "retention: %d heads / %d sequences x %d chunks are more than one launch takes",
               heads, n_seqs, max_chunks);
    const int pad = palm_retention_pad(dim);
    const long long rot_threads = (long long)n_tokens * heads * pad;
#define RET_MATRIX(D, V) launch_retention_chunks<T, D, V / 64>(stream, (const T*)qkvg, row_stride, v_off, g_off, qk, decay, eps, state, seq_slot, seq_new, \
            cu_new, n_seqs, n_tokens, heads, starts, (T*)out, act, joined, raw)
#define RET_CASE(D) linear_recurrence_sized<T, D, false>(stream, n_seqs, max_new, chunk, starts, nullptr, (const T*)qkvg, row_stride, v_off, g_off, \
            PreparedRows<D, 2>{qk, heads}, \
            decay, nullptr, eps, state, seq_slot, seq_new, cu_new, heads, dim, vdim, (T*)out, act, joined, raw)
    PALM_DTYPE_SWITCH(dtype, T, {
        retention_rotate_kernel<T><<<(unsigned)((rot_threads + 255) / 256), 256, 0, stream>>>((const T*)qkvg, row_stride, q_off, k_off, cos_t,
                                                                                             sin_t, rot, k_scale, act, n_tokens, heads, dim, pad, qk);
        if (matrix) {
            PALM_CHECK(chunk == palm_retention_matrix_chunk(dim, vdim, max_new) && chunk > 0 && row_stride % 8 == 0 && v_off % 8 == 0 &&
                       g_off % 8 == 0 && ((uintptr_t)qkvg | (uintptr_t)out | (uintptr_t)raw | (uintptr_t)state | (uintptr_t)starts | (uintptr_t)qk) % 16 == 0,
                       "retention: key size %d, value size %d, rows of %d from %d and %d do not go through the matrix cores", dim, vdim, row_stride, v_off, g_off);
            if (dim == 64 && vdim == 128) RET_MATRIX(64, 128);
            else if (dim == 64) RET_MATRIX(64, 256);
            else if (vdim == 128) RET_MATRIX(128, 128);
            else RET_MATRIX(128, 256);
        }
        else if (pad == 32) RET_CASE(32);
        else if (pad == 64) RET_CASE(64);
        else if (pad == 128) RET_CASE(128);
        else RET_CASE(256);
    });
#undef RET_CASE
#undef RET_MATRIX
    PALM_LAUNCHED();
    return 0;
}

__device__ inline void ret_load4(const float* p, float (&o)[4]) {
    const float4 v = *reinterpret_cast<const float4*>(p);
    o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
}
__device__ inline void ret_load4(const bf16_t* p, float (&o)[4]) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    o[0] = __builtin_bit_cast(float, v.x << 16); o[1] = __builtin_bit_cast(float, v.x & 0xffff0000u);
    o[2] = __builtin_bit_cast(float, v.y << 16); o[3] = __builtin_bit_cast(float, v.y & 0xffff0000u);
}
__device__ inline void ret_store4(float* p, const float (&v)[4]) { *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]); }
__device__ inline void ret_store4(bf16_t* p, const float (&v)[4]) {
    uint2 w;
    w.x = (uint32_t)f32_to_bf16(v[0]).bits | ((uint32_t)f32_to_bf16(v[1]).bits << 16);
    w.y = (uint32_t)f32_to_bf16(v[2]).bits | ((uint32_t)f32_to_bf16(v[3]).bits << 16);
    *reinterpret_cast<uint2*>(p) = w;
}

// ---- the joined heads normed together and gated -------------------------------------------------------------
// out[t] = raw[t] / sqrt(mean(raw[t]^2) + eps) * weight * f(gate[t]) over a token's whole row of `width` values (all
// heads), f = sigmoid (gate_act 1) or silu (gate_act 0).  raw is 32-bit; the gate lies in rows `gate_stride` elements
// apart.  One block per token.
template <typename T>
__global__ __launch_bounds__(1024) void joined_norm_gate_kernel(const float* __restrict__ raw, const float* __restrict__ weight, float eps,
                                                               const T* __restrict__ gate, int gate_stride, int gate_act, int width,
                                                               T* __restrict__ out) {
    __shared__ float scratch[16];
    const size_t t = blockIdx.x;
    const float* r = raw + t * width;
    float ss = 0.f;
    // four values a read where the row and the gate's rows allow
    const bool by_four = width % 4 == 0 && gate_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(gate) % 16) == 0;
    if (by_four) {
        for (int c = threadIdx.x * 4; c < width; c += blockDim.x * 4) {
            const float4 v = *reinterpret_cast<const float4*>(r + c);
            ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
        }
    } else {
        for (int c = threadIdx.x; c < width; c += blockDim.x) { const float v = r[c]; ss += v * v; }
    }
    const float inv = 1.0f / sqrtf(block_sum(ss, scratch) / (float)width + eps);
    auto gated = [&](float o, float w, float g) {
        const float f = gate_act == 1 ? 1.0f / (1.0f + expf(-g)) : g / (1.0f + expf(-g));
        return o * inv * w * f;
    };
    if (by_four) {
        for (int c = threadIdx.x * 4; c < width; c += blockDim.x * 4) {
            const float4 v = *reinterpret_cast<const float4*>(r + c), w = *reinterpret_cast<const float4*>(weight + c);
            float g[4];
            ret_load4(gate + t * gate_stride + c, g);
            const float y[4] = {gated(v.x, w.x, g[0]), gated(v.y, w.y, g[1]), gated(v.z, w.z, g[2]), gated(v.w, w.w, g[3])};
            ret_store4(out + t * width + c, y);
        }
    } else {
        for (int c = threadIdx.x; c < width; c += blockDim.x)
            out[t * width + c] = from_float<T>(gated(r[c], weight[c], to_float(gate[t * gate_stride + c])));
    }
}

PALM_API int palm_joined_norm_gate(hipStream_t stream, const float* raw, const float* weight, float eps, const void* gate, int dtype,
                                   int gate_stride, int gate_act, int n_tokens, int width, void* out) {
    PALM_CHECK(n_tokens >= 0 && width > 0 && gate_stride >= width, "joined_norm_gate: tokens=%d width=%d gate rows %d apart", n_tokens, width, gate_stride);
    PALM_CHECK(gate_act == 0 || gate_act == 1, "joined_norm_gate: gate activation %d is neither silu (0) nor sigmoid (1)", gate_act);
    if (n_tokens == 0) return 0;
    PALM_DTYPE_SWITCH(dtype, T,
        joined_norm_gate_kernel<T><<<n_tokens, n_tokens >= 256 ? 256 : width >= 2048 ? 1024 : width >= 1024 ? 512 : 256, 0, stream>>>(raw, weight, eps, (const T*)gate, gate_stride, gate_act, width, (T*)out));
    PALM_LAUNCHED();
    return 0;
}

PALM_DEFINE_LAST_ERROR()
