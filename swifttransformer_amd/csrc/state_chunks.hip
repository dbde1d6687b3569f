// The additive recurrence with one decay a head and token, over prompts and portions in chunks of 64 rows:
//
//   S_t = b_t S_(t-1) + (a_t k_t) v_t^T,   o_t = S_t^T q_t + skip v_t          (S [key channels x value channels] a head)
//
// With F_i the sum of log b over a chunk's rows up to i (double; a decay of zero counts as e^-10000), a chunk of n rows that starts
// from the state S is
//
//   o_i = e^(F_i) S^T q_i + sum_(j<=i) e^(F_i - F_j) a_j (q_i . k_j) v_j + skip v_i
//   S'  = e^(F_n) S + sum_j e^(F_n - F_j) a_j k_j v_j^T
//
// with every exponent a difference that is never positive.  Three kernels as in gla_chunks.hip: the chunks' sums (all chunks side by
// side), the carry (a thread an element of the state), the outputs.  Operands are float, weights and sums double, on the matrix cores
// (v_mfma_f64_16x16x4_f64, half as fast as float): chains of 64 rows and channels in float were up to a tenth further from float64
// than the scan, which does as many roundings but of smaller sums.  Heads share queries
// and keys in groups.  Items of up to 16 rows are walked row by row in the third kernel, which is all that steps of single tokens
// launch.  The scan (state_scan.hip) keeps the delta rule and heads of more than 128 channels.
//
// Per chunk and head the products are 2 * 64 * (64 + 2 dv) * dk flops at 77 Tflop/s (double), the chunks' sums are written, walked and
// read once (4 dk dv bytes each): both take less than the launches' own time up to some 250 rows; from there the products bound it.
// Distance from float64, 32 heads of 64 x 64: outputs 6.2e-8 (scan) and 2.6e-8, states 5.5e-8 and 3.0e-8 of their norm at 2,048 rows,
// 8.6e-8 and 2.6e-8, 6.3e-8 and 3.5e-8 at 33; single rows 9.1e-8 and 7.6e-8 (sums in four chains).  With float products it was
// 6.3e-8, 6.2e-8, 9.0e-8, 6.6e-8.
// Times, 32 heads of 64 x 64, one prompt of 2,048 rows: scan 530 us, here 73 (with float products 57); three that make 2,048: 222 and 79;
// 512 rows and 24 single ones: 141 and 37; 130 rows: 44 and 25; 33 rows: 20 and 24; 48 single rows: 23 and 16, 8: 17 and 15.  32 heads of
// 128 x 128, 2,048 rows: 895 and 182, 256: 122 and 53, 96: 52 and 44, 64: 38 and 43; beside 24 single rows 200: 100 and 86, 104: 78 and
// 83; 24 single rows alone 27 and 31: heads of more than 64 key channels come here from a number of rows on that grows with the items,
// and never in steps of single tokens.
#include "api.h"
#include "common.h"
#include "chunk_tiles.h"
#include "fragment.h"


namespace st {

constexpr int kStateShort = 16;      // rows up to which an item is walked row by row

struct StateArgs {
    float* out;
    const float *q, *k, *v;
    int64_t q_stride, k_stride, v_stride;
    const float *gate_a, *gate_b;    // rows gate_stride apart (0: one row for all tokens)
    int64_t gate_stride;
    const float* skip;               // [heads] or null
    float* state;
    int64_t slot_stride;
    float *U, *fall;                 // [chunks][heads][dk * dv], [chunks][heads]
    const int *item_len, *item_tok_off, *item_slot;
    int num_items, heads, qk_heads, dk, dv, chunks;
};

// the first wave: F_i of a chunk's n rows; past them the last one's
__device__ inline double state_log_decays(const float* __restrict__ b, int64_t stride, int n) {
    const int lane = threadIdx.x & 63;
    const double x = log((double)b[(int64_t)min(lane, n - 1) * stride]);
    double F = lane < n ? (x < -10000.0 ? -10000.0 : x) : 0.0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const double up = __shfl_up(F, o, 64);
        if (lane >= o) F += up;
    }
    return F;
}

// U[idx, head] and fall[idx, head].  Grid (heads, chunks, blocks of 64 value channels).  LDS: w doubles [64] | k [64][4 KQ + 4] | v [64][68].
template <int KQ, bool VEC>
__global__ __launch_bounds__(256) void state_sums_kernel(StateArgs a) {
    extern __shared__ __attribute__((aligned(16))) float state_lds[];
    const int head = blockIdx.x, idx = blockIdx.y, vb = blockIdx.z * 64, tid = threadIdx.x;
    int item, chunk;
    if (!find_chunk(idx, a.item_len, a.item_slot, a.num_items, item, chunk, kChunkRows, kStateShort)) return;
    const int n = min(kChunkRows, a.item_len[item] - chunk * kChunkRows), dk = a.dk, dv = a.dv;
    const int64_t row0 = (int64_t)a.item_tok_off[item] + (int64_t)chunk * kChunkRows;
    const int group = head / (a.heads / a.qk_heads);
    constexpr int KS = 4 * KQ + 4, VS = 68;
    double* w = reinterpret_cast<double*>(state_lds);
    float* ks = state_lds + 128;
    float* vs = ks + 64 * KS;
    Tile<KQ> tk;
    Tile<16> tv;
    tk.template load<VEC>(a.k + row0 * a.k_stride + (int64_t)group * dk, a.k_stride, n, 0, dk);
    tv.template load<VEC>(a.v + row0 * a.v_stride + (int64_t)head * dv, a.v_stride, n, vb, dv);
    if (tid < 64) {
        const double F = state_log_decays(a.gate_b + row0 * a.gate_stride + head, a.gate_stride, n), last = __shfl(F, n - 1, 64);
        const float f = a.gate_a[(row0 + min(tid, n - 1)) * a.gate_stride + head];
        w[tid] = tid < n ? f * exp_le0_double(last - F) : 0.0;
        if (blockIdx.z == 0 && tid == 0) a.fall[(int64_t)idx * a.heads + head] = (float)exp_le0_double(last);
    }
    tv.store(vs, VS);
    tk.store(ks, KS);
    __syncthreads();
    const int lane = tid & 63, wave = tid >> 6, r16 = lane & 15, g = lane >> 4, p16 = double_row(r16);
    const int steps = (n + 15) >> 4, ktiles = (dk + 15) >> 4;
    float* u = a.U + ((int64_t)idx * a.heads + head) * dk * dv;
    for (int kt = wave; kt < ktiles; kt += 4) {
        doublex4 acc[4];
#pragma unroll
        for (int vt = 0; vt < 4; ++vt) acc[vt] = doublex4{0.0, 0.0, 0.0, 0.0};
        for (int s = 0; s < steps; ++s) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int j = 16 * s + 4 * g + r;
                const double x = ks[j * KS + 16 * kt + p16] * w[j];
#pragma unroll
                for (int vt = 0; vt < 4; ++vt)
                    acc[vt] = __builtin_amdgcn_mfma_f64_16x16x4f64(x, (double)vs[j * VS + 16 * vt + r16], acc[vt], 0, 0, 0);
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int kk = 16 * kt + 4 * g + r;
            if (kk >= dk) continue;
#pragma unroll
            for (int vt = 0; vt < 4; ++vt) {
                const int col = vb + 16 * vt + r16;
                if (col < dv) u[(int64_t)kk * dv + col] = (float)acc[vt][r];
            }
        }
    }
}

// A thread an element of a request's state: S walks the item's chunks, leaving at U's place the state each chunk starts from.
__global__ __launch_bounds__(256) void state_carry_kernel(StateArgs a) {
    const int head = blockIdx.x, item = blockIdx.y;
    const int e = blockIdx.z * 256 + threadIdx.x;
    const int slot = a.item_slot[item], len = a.item_len[item];
    if (slot < 0 || len <= kStateShort) return;
    const int base = chunks_before(item, a.item_len, a.item_slot, kChunkRows, kStateShort), chunks = (len + kChunkRows - 1) / kChunkRows;
    if (e >= a.dk * a.dv) return;
    const int64_t plane = (int64_t)a.dk * a.dv, first = (int64_t)base * a.heads + head;
    float* home = a.state + (int64_t)slot * a.slot_stride + (int64_t)head * plane + e;
    float* u = a.U + first * plane + e;
    const float* f = a.fall + first;
    *home = carry_states(u, (int64_t)a.heads * plane, f, a.heads, chunks, *home);
}

// 64 value channels (from vb) of an item of up to kStateShort rows from its slot's state, row by row.  Thread (wave, lane): KQ key
// channels from KQ * wave, value channel vb + lane; the waves' partial read-outs meet in LDS once a row.  (Value channels never meet:
// a wave with 128 of them holds twice the state and leaves a unit half as many workgroups: 49 against 31 us for 24 items of 32 heads of
// 128 x 128.)
// LONG: any number of rows, kStateShort of them in LDS at a time.
template <int KQ, bool LONG>
__device__ __forceinline__ void state_walk(float* lds, const StateArgs& a, int item, int rows, int head, int vb) {
    constexpr int C = 4 * KQ, V = 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, dk = a.dk, dv = a.dv;
    int64_t row0 = a.item_tok_off[item];
    const int group = head / (a.heads / a.qk_heads), col = vb + lane, colc = min(col, dv - 1);
    float* sq = lds;                       // [n][C], keys likewise, zeros past dk
    float* sk = sq + kStateShort * C;
    float* sv = sk + kStateShort * C;      // [n][V]
    float* sb = sv + kStateShort * V;      // [n], and the keys' factors [n]
    float* part = sb + 2 * kStateShort;    // [2][4][V]
    float* home = a.state + (int64_t)a.item_slot[item] * a.slot_stride + (int64_t)head * dk * dv;
    float S[KQ];
#pragma unroll
    for (int c = 0; c < KQ; ++c) {
        const int kk = wave * KQ + c;
        const float x = home[(int64_t)min(kk, dk - 1) * dv + colc];
        S[c] = kk < dk && col < dv ? x : 0.f;
    }
    const float skip = a.skip ? a.skip[head] : 0.f;
    do {
        const int n = LONG ? min(rows, kStateShort) : rows;
        for (int e = tid; e < n * C; e += 256) {
            const int j = e / C, c = e - j * C;
            const int64_t at = (int64_t)group * dk + min(c, dk - 1), row = row0 + j;
            const float x = a.q[row * a.q_stride + at], y = a.k[row * a.k_stride + at];
            sq[e] = c < dk ? x : 0.f;
            sk[e] = c < dk ? y : 0.f;
        }
        for (int j = wave; j < n; j += 4) {
            const float x = a.v[(row0 + j) * a.v_stride + (int64_t)head * dv + colc];
            sv[j * V + lane] = col < dv ? x : 0.f;
        }
        if (tid < n) {
            sb[tid] = a.gate_b[(row0 + tid) * a.gate_stride + head];
            sb[kStateShort + tid] = a.gate_a[(row0 + tid) * a.gate_stride + head];
        }
        __syncthreads();
        for (int j = 0; j < n; ++j) {
            float* p = part + (j & 1) * 4 * V;
            const float b = sb[j], vv = sv[j * V + lane], av = sb[kStateShort + j] * vv;
            float acc[4] = {0.f, 0.f, 0.f, 0.f};                   // (sums in short chains)
#pragma unroll
            for (int c = 0; c < KQ; c += 4) {
                const float4 q4 = *reinterpret_cast<const float4*>(sq + j * C + wave * KQ + c);
                const float4 k4 = *reinterpret_cast<const float4*>(sk + j * C + wave * KQ + c);
                S[c] = fmaf(b, S[c], k4.x * av);         acc[0] = fmaf(S[c], q4.x, acc[0]);
                S[c + 1] = fmaf(b, S[c + 1], k4.y * av); acc[1] = fmaf(S[c + 1], q4.y, acc[1]);
                S[c + 2] = fmaf(b, S[c + 2], k4.z * av); acc[2] = fmaf(S[c + 2], q4.z, acc[2]);
                S[c + 3] = fmaf(b, S[c + 3], k4.w * av); acc[3] = fmaf(S[c + 3], q4.w, acc[3]);
            }
            p[wave * V + lane] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
            __syncthreads();                   // (the other half of `part` was read before this row's sums were written)
            if (wave == 0 && col < dv)
                a.out[((row0 + j) * a.heads + head) * dv + col] = fmaf(skip, vv, (p[lane] + p[V + lane]) + (p[2 * V + lane] + p[3 * V + lane]));
        }
        if (LONG) __syncthreads();         // the rows have been read
        rows -= kStateShort;
        row0 += kStateShort;
    } while (LONG && rows > 0);
#pragma unroll
    for (int c = 0; c < KQ; ++c) {
        const int kk = wave * KQ + c;
        if (kk < dk && col < dv) home[(int64_t)kk * dv + col] = S[c];
    }
}

// One row, the same numbers as state_walk's: everything that is read is asked for before anything waits (state, query, key, value and gates
// one after the other were four trips to memory: 8 rows of 4 heads of 64 x 128 4.9 -> 3.4 us, 48 of 32 heads of 64 x 64 11.5 -> 8.1).
template <int KQ>
__device__ __forceinline__ void state_row(float* lds, const StateArgs& a, int64_t row, int slot, int head, int vb) {
    constexpr int C = 4 * KQ, V = 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, dk = a.dk, dv = a.dv;
    const int group = head / (a.heads / a.qk_heads), col = vb + lane, colc = min(col, dv - 1);
    float* sq = lds;                       // [C], and the keys
    float* part = sq + 2 * C;              // [4][V]
    float* home = a.state + (int64_t)slot * a.slot_stride + (int64_t)head * dk * dv;
    // a thread's channel of the query (the first C threads) or of the key
    const int c = tid < C ? tid : tid - C, in = tid < 2 * C && c < dk;
    const float* from = tid < C ? a.q + row * a.q_stride : a.k + row * a.k_stride;
    const float x = from[(int64_t)group * dk + (in ? c : 0)];
    const float v = a.v[row * a.v_stride + (int64_t)head * dv + colc];
    const float b = a.gate_b[row * a.gate_stride + head], ga = a.gate_a[row * a.gate_stride + head], skip = a.skip ? a.skip[head] : 0.f;
    float S[KQ];
#pragma unroll
    for (int i = 0; i < KQ; ++i) S[i] = home[(int64_t)min(wave * KQ + i, dk - 1) * dv + colc];
    if (tid < 2 * C) sq[tid] = in ? x : 0.f;
    __syncthreads();
    const float vv = col < dv ? v : 0.f, av = ga * vv;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < KQ; ++i) {
        const int kk = wave * KQ + i;
        S[i] = fmaf(b, kk < dk && col < dv ? S[i] : 0.f, sq[C + kk] * av);
        acc[i & 3] = fmaf(S[i], sq[kk], acc[i & 3]);
        if (kk < dk && col < dv) home[(int64_t)kk * dv + col] = S[i];
    }
    part[wave * V + lane] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
    __syncthreads();
    if (wave == 0 && col < dv)
        a.out[(row * a.heads + head) * dv + col] = fmaf(skip, vv, (part[lane] + part[V + lane]) + (part[2 * V + lane] + part[3 * V + lane]));
}

// Steps of single tokens: grid (heads, items, blocks of 64 value channels), a kernel of its own with few registers.  (The caller's word
// that there are no longer items is about speed: they are walked kStateShort rows at a time.)
template <int KQ>
__global__ __launch_bounds__(256) void state_walk_kernel(StateArgs a) {
    extern __shared__ __attribute__((aligned(16))) float state_lds[];
    const int item = blockIdx.y, len = a.item_len[item], slot = a.item_slot[item], row = a.item_tok_off[item];
    if (slot < 0 || len <= 0) return;
    if (len == 1) state_row<KQ>(state_lds, a, row, slot, blockIdx.x, blockIdx.z * 64);
    else if (len <= kStateShort) state_walk<KQ, false>(state_lds, a, item, len, blockIdx.x, blockIdx.z * 64);
    else state_walk<KQ, true>(state_lds, a, item, len, blockIdx.x, blockIdx.z * 64);
}

// Rows of a chunk, transposed as in gla_chunks.hip and the matrix memory's outputs.  LDS: F doubles [64] | a [64] | k [64][4 KQ + 4],
// later 64 key channels of the start state [64][16 NV + 4] | v [64][16 NV + 4].
template <int KQ, int NV>
struct StateOutLds {
    static constexpr int KS = 4 * KQ + 4, VS = 16 * NV + 4;
    static constexpr int first = KS > VS ? 64 * KS : 64 * VS;
    static constexpr size_t bytes = sizeof(double) * 64 + sizeof(float) * (size_t)(64 + first + 64 * VS);
    static constexpr size_t walk = sizeof(float) * (size_t)(kStateShort * (8 * KQ + 66) + 512);
    static constexpr size_t both = bytes > walk ? bytes : walk;
};

template <int KQ, int NV, bool VEC>
__global__ __launch_bounds__(256, KQ == 16 && NV == 4 ? 3 : 1) void state_out_kernel(StateArgs a) {
    extern __shared__ __attribute__((aligned(16))) float state_lds[];
    using L = StateOutLds<KQ, NV>;
    const int head = blockIdx.x, idx = blockIdx.y, tid = threadIdx.x;
    int item = idx - a.chunks, chunk;
    if (item >= 0) {
        if (a.item_slot[item] < 0 || a.item_len[item] <= 0 || a.item_len[item] > kStateShort) return;
        for (int vb = 0; vb < a.dv; vb += 64) {
            if (vb > 0) __syncthreads();                       // the rows before have been read
            state_walk<KQ, false>(state_lds, a, item, a.item_len[item], head, vb);
        }
        return;
    }
    if (!find_chunk(idx, a.item_len, a.item_slot, a.num_items, item, chunk, kChunkRows, kStateShort)) return;
    const int n = min(kChunkRows, a.item_len[item] - chunk * kChunkRows), dk = a.dk, dv = a.dv;
    const int64_t row0 = (int64_t)a.item_tok_off[item] + (int64_t)chunk * kChunkRows;
    const int group = head / (a.heads / a.qk_heads);
    double* sF = reinterpret_cast<double*>(state_lds);
    float* sa = reinterpret_cast<float*>(sF + 64);
    float* ks = sa + 64;
    float* vs = ks + L::first;
    const int lane = tid & 63, wave = tid >> 6, r16 = lane & 15, g = lane >> 4, p16 = double_row(r16);
    const int i = wave * 16 + r16;                             // this lane's row of the chunk
    const bool row_ok = i < n;
    {
        Tile<KQ> tk;
        Tile<4 * NV> tv;
        tk.template load<VEC>(a.k + row0 * a.k_stride + (int64_t)group * dk, a.k_stride, n, 0, dk);
        tv.template load<VEC>(a.v + row0 * a.v_stride + (int64_t)head * dv, a.v_stride, n, 0, dv);
        if (tid < 64) {
            sF[tid] = state_log_decays(a.gate_b + row0 * a.gate_stride + head, a.gate_stride, n);
            sa[tid] = tid < n ? a.gate_a[(row0 + tid) * a.gate_stride + head] : 0.f;
        }
        tk.store(ks, L::KS);
        tv.store(vs, L::VS);
    }
    float qf[KQ];                                              // key channels 16 s + 4 g .. + 3
    {
        const float* qr = a.q + (row0 + min(i, n - 1)) * a.q_stride + (int64_t)group * dk;
#pragma unroll
        for (int s = 0; s < KQ / 4; ++s) {
            const float4 x = load_piece<VEC>(qr, 16 * s + 4 * g, dk, row_ok);
            qf[4 * s] = x.x; qf[4 * s + 1] = x.y; qf[4 * s + 2] = x.z; qf[4 * s + 3] = x.w;
        }
    }
    // the start state's first 64 key channels, on their way during the scores
    const float* s0 = a.U + ((int64_t)idx * a.heads + head) * dk * dv;
    Tile<4 * NV> ts;
    ts.template load<VEC>(s0, dv, min(dk, 64), 0, dv);
    __syncthreads();
    const double Fi = sF[i];
    const double carried = exp_le0_double(Fi);
    doublex4 st[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        st[t] = doublex4{0.0, 0.0, 0.0, 0.0};
        if (t > wave || 16 * t >= n) continue;                 // uniform over the wave
#pragma unroll
        for (int s = 0; s < KQ / 4; ++s) {
            const float4 x = *reinterpret_cast<const float4*>(ks + (16 * t + p16) * L::KS + 16 * s + 4 * g);
            st[t] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)x.x, (double)qf[4 * s], st[t], 0, 0, 0);
            st[t] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)x.y, (double)qf[4 * s + 1], st[t], 0, 0, 0);
            st[t] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)x.z, (double)qf[4 * s + 2], st[t], 0, 0, 0);
            st[t] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)x.w, (double)qf[4 * s + 3], st[t], 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int j = 16 * t + 4 * g + r;
            st[t][r] = j <= i ? st[t][r] * (sa[j] * exp_le0_double(Fi - sF[j])) : 0.0;
        }
    }
    doublex4 o[NV];
#pragma unroll
    for (int vt = 0; vt < NV; ++vt) o[vt] = doublex4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int b = 0; b < (KQ + 15) / 16; ++b) {                 // S_0^T q, then times the row's factor
        if (64 * b >= dk) continue;
        __syncthreads();                                       // the keys (or the channels before) have been read
        ts.store(ks, L::VS);
        __syncthreads();
        if (64 * (b + 1) < dk) ts.template load<VEC>(s0 + (int64_t)64 * (b + 1) * dv, dv, min(dk - 64 * (b + 1), 64), 0, dv);
#pragma unroll
        for (int s = 0; s < (KQ < 16 ? KQ : 16); ++s) {
            const float* sr = ks + (16 * (s >> 2) + 4 * g + (s & 3)) * L::VS + p16;
#pragma unroll
            for (int vt = 0; vt < NV; ++vt)
                o[vt] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)sr[16 * vt], (double)qf[(16 * b + s) % KQ], o[vt], 0, 0, 0);
        }
    }
#pragma unroll
    for (int vt = 0; vt < NV; ++vt) o[vt] *= carried;
    // A row meets the later rows of its own block with a weight of zero, which an infinity or NaN among their values would turn into
    // NaN: such a block's rows are summed one by one instead, below.
    float zero = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int vt = 0; vt < NV; ++vt) zero = fmaf(vs[(16 * wave + 4 * g + r) * L::VS + 16 * vt + r16], 0.f, zero);
    const bool finite = !__any(!(zero == 0.f));
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        if (t > wave || 16 * t >= n || (t == wave && !finite)) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float* vr = vs + (16 * t + 4 * g + r) * L::VS + p16;
#pragma unroll
            for (int vt = 0; vt < NV; ++vt) o[vt] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)vr[16 * vt], st[t][r], o[vt], 0, 0, 0);
        }
    }
    if (!finite) {
        const doublex4 p = wave == 0 ? st[0] : wave == 1 ? st[1] : wave == 2 ? st[2] : st[3];
#pragma unroll 1
        for (int j4 = 0; j4 < 4; ++j4)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const double w = __shfl(p[e], r16 + 16 * j4, 64);
                if (4 * j4 + e > r16) continue;
#pragma unroll
                for (int vt = 0; vt < NV; ++vt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[vt][r] = fma(w, (double)vs[(16 * wave + 4 * j4 + e) * L::VS + 16 * vt + 4 * g + r], o[vt][r]);
            }
    }
    if (!row_ok) return;
    // o[vt][r]: value channel 16 vt + 4 g + r of row i
    const double skip = a.skip ? a.skip[head] : 0.f;
    float* dst = a.out + ((row0 + i) * a.heads + head) * dv;
#pragma unroll
    for (int vt = 0; vt < NV; ++vt) {
        const int v0 = 16 * vt + 4 * g;
        if (v0 >= dv) continue;
        const float* own = vs + i * L::VS + v0;
        const float4 y = make_float4((float)fma(skip, (double)own[0], o[vt][0]), (float)fma(skip, (double)own[1], o[vt][1]),
                                     (float)fma(skip, (double)own[2], o[vt][2]), (float)fma(skip, (double)own[3], o[vt][3]));
        if (VEC) *reinterpret_cast<float4*>(dst + v0) = y;
        else {
            const float z[4] = {y.x, y.y, y.z, y.w};
            for (int r = 0; r < 4 && v0 + r < dv; ++r) dst[v0 + r] = z[r];
        }
    }
}

template <int KQ, int NV, bool VEC>
static int launch_state_chunks(const StateArgs& a, bool single, hipStream_t stream) {
    using L = StateOutLds<KQ, NV>;
    if constexpr (KQ == 16) if (single) {
        state_walk_kernel<KQ><<<dim3(a.heads, a.num_items, (a.dv + 63) / 64), 256, L::walk, stream>>>(a);
        ST_LAUNCH_CHECK("state_chunks (single rows)");
        return 0;
    }
    constexpr int kSums = (int)sizeof(float) * (128 + 64 * (4 * KQ + 4) + 64 * 68), kOut = (int)L::both;
    ST_CHECK(hipFuncSetAttribute((const void*)state_sums_kernel<KQ, VEC>, hipFuncAttributeMaxDynamicSharedMemorySize, kSums) == hipSuccess &&
             hipFuncSetAttribute((const void*)state_out_kernel<KQ, NV, VEC>, hipFuncAttributeMaxDynamicSharedMemorySize, kOut) == hipSuccess,
             "state_chunks: cannot raise the LDS limit");
    if (a.chunks) {
        state_sums_kernel<KQ, VEC><<<dim3(a.heads, a.chunks, (a.dv + 63) / 64), 256, kSums, stream>>>(a);
        ST_LAUNCH_CHECK("state_chunks (sums)");
        state_carry_kernel<<<dim3(a.heads, a.num_items, (unsigned)((a.dk * a.dv + 255) / 256)), 256, 0, stream>>>(a);
        ST_LAUNCH_CHECK("state_chunks (carry)");
    }
    state_out_kernel<KQ, NV, VEC><<<dim3(a.heads, a.chunks + a.num_items), 256, kOut, stream>>>(a);
    ST_LAUNCH_CHECK("state_chunks (outputs)");
    return 0;
}

}  // namespace st

using namespace st;

extern "C" int st_state_chunks(float* out, const float* q, int64_t q_stride, const float* k, int64_t k_stride, const float* v,
                               int64_t v_stride, const float* gate_a, const float* gate_b, int64_t gate_stride, const float* skip,
                               float* state, int64_t slot_stride, const int* item_len, const int* item_tok_off, const int* item_slot,
                               int num_items, int num_rows, int heads, int qk_heads, int key_dim, int value_dim, float* scratch,
                               int64_t scratch_chunks, int single, hipStream_t stream) {
    ST_CHECK(num_items >= 0 && num_rows >= 0 && heads > 0 && qk_heads > 0 && heads % qk_heads == 0 && key_dim > 0 && value_dim > 0,
             "state_chunks: bad sizes");
    ST_CHECK(key_dim <= 128 && value_dim <= 128, "state_chunks: up to 128 key and 128 value channels a head, not %d and %d", key_dim, value_dim);
    ST_CHECK(!single || key_dim <= 64, "state_chunks: steps of single tokens take up to 64 key channels a head, not %d", key_dim);
    if (num_items == 0 || num_rows == 0) return 0;
    ST_CHECK(out && q && k && v && gate_a && gate_b && state && item_len && item_tok_off && item_slot, "state_chunks: null operand");
    const int64_t chunks = single ? 0 : most_chunks(num_rows, num_items, kStateShort);
    ST_CHECK(chunks == 0 || (scratch && scratch_chunks >= chunks), "state_chunks: scratch for %lld chunks, %lld needed", (long long)scratch_chunks, (long long)chunks);
    ST_CHECK(chunks + num_items <= 65535, "state_chunks: too many chunks or items");
    StateArgs a;
    a.out = out; a.q = q; a.k = k; a.v = v; a.q_stride = q_stride; a.k_stride = k_stride; a.v_stride = v_stride;
    a.gate_a = gate_a; a.gate_b = gate_b; a.gate_stride = gate_stride; a.skip = skip; a.state = state; a.slot_stride = slot_stride;
    a.U = scratch; a.fall = scratch + scratch_chunks * heads * key_dim * value_dim;
    a.item_len = item_len; a.item_tok_off = item_tok_off; a.item_slot = item_slot; a.num_items = num_items;
    a.heads = heads; a.qk_heads = qk_heads; a.dk = key_dim; a.dv = value_dim; a.chunks = (int)chunks;
    // four numbers at a time: rows and heads start on their size
    const bool vec = ((key_dim | value_dim) & 3) == 0 && ((q_stride | k_stride | v_stride) & 3) == 0 &&
                     (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out | (uintptr_t)scratch) & 15) == 0;
#define ST_STATE(KQ, NV) \
    (vec ? launch_state_chunks<KQ, NV, true>(a, single != 0, stream) : launch_state_chunks<KQ, NV, false>(a, single != 0, stream))
    if (key_dim <= 64) return value_dim <= 64 ? ST_STATE(16, 4) : ST_STATE(16, 8);
    return value_dim <= 64 ? ST_STATE(32, 4) : ST_STATE(32, 8);
#undef ST_STATE
}
