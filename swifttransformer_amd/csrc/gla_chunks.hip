// Gated linear attention over prompts and portions in chunks of 64 rows, with the head norm and the gate behind it:
//
//   S_t = diag(a_t) S_(t-1) + k_t v_t^T,   o_t = scale * S_t^T q_t,   y_t = o_t / rms(o_t) * gain * silu(gate_t)
//
// a_t = sigmoid(z_t)^(1 / tau) is a decay a key channel and token, between 0 and 1.  A chunk's outputs are products on the matrix cores
// once decays are folded into queries and keys.  Operands in memory and LDS are float; products of decays, sums and what meets them are
// double (v_mfma_f64_16x16x4_f64): chains of 64 rows and channels in float were up to a fifth further from float64 than the scan.  Nothing is divided by a product of decays (it may be
// zero): a chunk is four blocks of 16 rows, and only products over rows that lie between two points are formed, never above one:
//
//   q^_i = q_i * prod of a from its block's first row to i
//   k^_j = k_j * prod of a from row j + 1 to its block's last row,     B_J the product over all of block J
//   rows i, j of blocks I > J:  (q^_i * B_(J+1) .. B_(I-1)) . k^_j      (matrix cores)
//   the state at the chunk's start:  S_0^T (q^_i * B_0 .. B_(I-1))      (matrix cores)
//   rows of one block:  sum over the channels of q_i k_j times the product of a from j + 1 to i, on the vector units: a lane
//   keeps q_i and walks j downwards, one factor more a step, so that its last value is q^_i
//
// Three kernels: the chunks' sums U = sum_j k_j (product of a behind j) v_j^T with the chunks' decays A (no state needed, all
// chunks side by side), the carry S -> A S + U (a thread an element of the state; U's place then holds the chunk's start state),
// the outputs with norm and gate.  Chunks count from an item's first row of the step, so a portion may start anywhere; the state
// comes from and goes back to the request's slot.  Items of up to 16 rows are walked row by row in the third kernel, which is all
// that steps of single tokens launch.  The scan (csrc/recurrent.hip) keeps heads of more than 128 channels, whose tiles do not fit
// LDS.
//
// Measured beside decay gates, scan and norm kernel (which sums the scan's planes): one item of 2,011 rows, 32 heads of 64 x 64,
// 427 -> 97 us (the scan's 2,011 dependent steps; now the carry's 32, and the products at a few workgroups a unit; with everything in
// float 65); three items of 2,048 rows together 219 -> 104; 32 heads of 128 x 128 637 -> 297; 33 rows 35 -> 30; 512 rows beside 24 single
// tokens 123 -> 48; 8 single tokens 34 -> 14, 24 of 32 heads of 128 x 128 58 -> 29 us.  Relative distance from float64 behind norm and
// gate, in float: 2,011 rows outputs 1.5e-7 -> 9.3e-8, state 9.6e-8 -> 6.6e-8; 33 rows 1.4e-7 -> 7.7e-8 and 4.4e-8 -> 3.2e-8; 48 single
// tokens 1.4e-7 -> 1.2e-7 and 3.6e-8 -> 3.5e-8 (with everything in float 1.7e-7 and 9.9e-8, 1.3e-7 and 5.0e-8, 1.4e-7 and 3.9e-8).
#include "api.h"
#include "common.h"
#include "chunk_tiles.h"
#include "fragment.h"

#include <cfloat>

namespace st {

constexpr int kGlaShort = 16;        // rows up to which an item is walked row by row

// sigmoid(z)^inv_tau = e^(inv_tau (min(z, 0) - log(1 + e^-|z|))), rounded to float once; 1 for the largest float, which stands for
// rows that do not exist.  log(1 + u) = 2 artanh(s) = 2 s (1 + s^2 / 3 + ..), s = u / (2 + u) up to 1/3: the sum behind the one, up to s^16
// (the next term is below 2^-32), is at most 0.04 and float.  (With the exponential of -|z| and that sum in
// double too 2,011 rows of 32 heads of 64 take 102 us instead of 97, at the same distance from float64; the library's float functions,
// off by up to 2^-24 each, took 23 us more than the hardware's.)
__device__ inline float gla_decay(float z, float inv_tau) {
    const double u = exp_le0(-fabsf(z));
    const double r0 = __builtin_amdgcn_rcpf((float)(2.0 + u)), s = u * (r0 * fma(-(2.0 + u), r0, 2.0));
    const float s2 = (float)(s * s);
    float y = 1.f / 17.f;
    y = fmaf(y, s2, 1.f / 15.f);
    y = fmaf(y, s2, 1.f / 13.f);
    y = fmaf(y, s2, 1.f / 11.f);
    y = fmaf(y, s2, 1.f / 9.f);
    y = fmaf(y, s2, 1.f / 7.f);
    y = fmaf(y, s2, 1.f / 5.f);
    y = fmaf(y, s2, 1.f / 3.f);
    return (float)exp_le0_double(((z < 0.f ? (double)z : 0.0) - 2.0 * fma(s, (double)(y * s2), s)) * inv_tau);
}

// four neighbouring numbers of a row as floats, `fill` past its end or where the row does not exist (see load_piece)
template <typename T, bool VEC>
__device__ inline float4 gla_piece(const T* __restrict__ row, int c, int limit, bool ok, float fill) {
    float4 v;
    if (VEC) {
        const T* p = row + min(c, limit - 4);
        if constexpr (sizeof(T) == 4) {
            v = *reinterpret_cast<const float4*>(p);
        } else {
            const uint2 u = *reinterpret_cast<const uint2*>(p);
            v = make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                            __uint_as_float(u.y & 0xffff0000u));
        }
    } else {
        v = make_float4(Elem<T>::load(row + min(c, limit - 1)), Elem<T>::load(row + min(c + 1, limit - 1)),
                        Elem<T>::load(row + min(c + 2, limit - 1)), Elem<T>::load(row + min(c + 3, limit - 1)));
    }
    v.x = ok && c < limit ? v.x : fill;
    v.y = ok && c + 1 < limit ? v.y : fill;
    v.z = ok && c + 2 < limit ? v.z : fill;
    v.w = ok && c + 3 < limit ? v.w : fill;
    return v;
}

// a tile of 64 rows x 4 * P4 numbers by 256 threads, on its way to LDS
template <int P4>
struct GlaTile {
    float4 v[P4 / 4];
    template <typename T, bool VEC>
    __device__ inline void load(const T* __restrict__ base, int64_t stride, int rows, int first, int limit, float fill) {
#pragma unroll
        for (int i = 0; i < P4 / 4; ++i) {
            const int e = threadIdx.x + 256 * i, j = e / P4, c = 4 * (e % P4);
            v[i] = gla_piece<T, VEC>(base + (int64_t)min(j, rows - 1) * stride, first + c, limit, j < rows, fill);
        }
    }
    __device__ inline void store(float* lds, int lds_stride) const {
#pragma unroll
        for (int i = 0; i < P4 / 4; ++i) {
            const int e = threadIdx.x + 256 * i;
            *reinterpret_cast<float4*>(lds + (e / P4) * lds_stride + 4 * (e % P4)) = v[i];
        }
    }
    __device__ inline void store_decays(float* lds, int lds_stride, float inv_tau) const {
#pragma unroll
        for (int i = 0; i < P4 / 4; ++i) {
            const int e = threadIdx.x + 256 * i;
            *reinterpret_cast<float4*>(lds + (e / P4) * lds_stride + 4 * (e % P4)) =
                make_float4(gla_decay(v[i].x, inv_tau), gla_decay(v[i].y, inv_tau), gla_decay(v[i].z, inv_tau), gla_decay(v[i].w, inv_tau));
        }
    }
};

// U[idx, head] [dk, dv] and A[idx, head] [dk].  Grid (heads, chunks, blocks of 64 value channels); a wave takes rows of 16 x 16
// tiles.  KQ: dk <= 4 KQ.  LDS: k [64][4 KQ + 4] | a [64][4 KQ + 4] | v [64][68] | B doubles [4][4 KQ].
template <typename T, int KQ, bool VEC>
__global__ __launch_bounds__(256) void gla_sums_kernel(
    float* __restrict__ U, float* __restrict__ A, const T* __restrict__ k, int64_t k_stride, const T* __restrict__ v, int64_t v_stride,
    const float* __restrict__ z, float inv_tau, const int* __restrict__ item_len, const int* __restrict__ item_tok_off,
    const int* __restrict__ item_slot, int num_items, int heads, int dk, int dv) {
    extern __shared__ __attribute__((aligned(16))) float gla_lds[];
    const int head = blockIdx.x, idx = blockIdx.y, vb = blockIdx.z * 64, tid = threadIdx.x;
    int item, chunk;
    if (!find_chunk(idx, item_len, item_slot, num_items, item, chunk, kChunkRows, kGlaShort)) return;
    const int n = min(kChunkRows, item_len[item] - chunk * kChunkRows);
    const int64_t row0 = (int64_t)item_tok_off[item] + (int64_t)chunk * kChunkRows;
    constexpr int KS = 4 * KQ + 4, VS = 68;
    float* ks = gla_lds;
    float* as = ks + 64 * KS;
    float* vs = as + 64 * KS;
    double* bp = reinterpret_cast<double*>(vs + 64 * VS);
    const int lane = tid & 63, wave = tid >> 6, r16 = lane & 15, g = lane >> 4;
    {
        GlaTile<KQ> tk, ta;
        GlaTile<16> tv;
        tk.template load<T, VEC>(k + row0 * k_stride + (int64_t)head * dk, k_stride, n, 0, dk, 0.f);
        ta.template load<float, VEC>(z + (row0 * heads + head) * dk, (int64_t)heads * dk, n, 0, dk, FLT_MAX);
        tv.template load<T, VEC>(v + row0 * v_stride + (int64_t)head * dv, v_stride, n, vb, dv, 0.f);
        tk.store(ks, KS);
        ta.store_decays(as, KS, inv_tau);
        tv.store(vs, VS);
    }
    __syncthreads();
    // a wave's block of 16 rows: each key times the decays behind it in the block (those of the blocks behind meet it in the product)
    float* kw = ks + wave * 16 * KS;
    const float* aw = as + wave * 16 * KS;
    for (int c = lane; c < 4 * KQ; c += 64) {
        double run = 1.0;
#pragma unroll
        for (int j = 15; j >= 0; --j) {
            kw[j * KS + c] = (float)(kw[j * KS + c] * run);
            run *= aw[j * KS + c];
        }
        bp[wave * 4 * KQ + c] = run;
    }
    __syncthreads();
    const int p16 = double_row(r16);
    const int steps = (n + 15) >> 4, ktiles = (dk + 15) >> 4;    // steps of 16 keys
    float* u = U + ((int64_t)idx * heads + head) * dk * dv;
    for (int kt = wave; kt < ktiles; kt += 4) {
        double behind[4];
        behind[3] = 1.0;
#pragma unroll
        for (int s = 2; s >= 0; --s) behind[s] = behind[s + 1] * bp[(s + 1) * 4 * KQ + 16 * kt + p16];
        if (blockIdx.z == 0 && g == 0 && 16 * kt + p16 < dk)
            A[((int64_t)idx * heads + head) * dk + 16 * kt + p16] = (float)(behind[0] * bp[16 * kt + p16]);
        doublex4 acc[4];
#pragma unroll
        for (int vt = 0; vt < 4; ++vt) acc[vt] = doublex4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if (s >= steps) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int j = 16 * s + 4 * g + r;
                const double x = ks[j * KS + 16 * kt + p16] * behind[s];
#pragma unroll
                for (int vt = 0; vt < 4; ++vt)
                    acc[vt] = __builtin_amdgcn_mfma_f64_16x16x4f64(x, (double)vs[j * VS + 16 * vt + r16], acc[vt], 0, 0, 0);
            }
        }
        // acc[vt][r]: key channel 16 kt + 4 g + r, value channel 16 vt + r16
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

// A thread an element of a request's state: S walks the item's chunks, leaving at U's place the state each chunk starts from;
// the last S goes back to the slot.
__global__ __launch_bounds__(256) void gla_carry_kernel(
    float* __restrict__ U, const float* __restrict__ A, float* __restrict__ state, const int* __restrict__ item_len,
    const int* __restrict__ item_slot, int heads, int dk, int dv) {
    const int head = blockIdx.x, item = blockIdx.y;
    const int e = blockIdx.z * 256 + threadIdx.x;
    const int slot = item_slot[item], len = item_len[item];
    if (slot < 0 || len <= kGlaShort) return;
    const int base = chunks_before(item, item_len, item_slot, kChunkRows, kGlaShort);
    if (e >= dk * dv) return;
    const int chunks = (len + kChunkRows - 1) / kChunkRows;
    const int64_t plane = (int64_t)dk * dv, first = (int64_t)base * heads + head;
    float* home = state + ((int64_t)slot * heads + head) * plane + e;
    float* u = U + first * plane + e;
    const float* f = A + first * dk + e / dv;
    *home = carry_states(u, (int64_t)heads * plane, f, (int64_t)heads * dk, chunks, *home);
}

// Rows of a chunk, transposed as in the matrix memory's outputs: a wave has a block of 16 rows, lane (r16, g) row r16 of it with
// the key channels 16 s + 4 g .. + 3; S^T = K Q^T leaves a lane with keys 4 g + r of its row, which is the next product's operand
// as it lies (O^T += V^T P^T).  LDS: k [64][4 KQ + 4] | a [64][4 KQ + 4], later 64 key channels of the start state
// [64][16 NV + 4] | v [64][16 NV + 4] | B doubles [4][4 KQ].
//
// An item of up to kGlaShort rows is walked here from its slot's state instead, row by row, and leaves its state there: 16 x less
// traffic than a chunk for a single token.  Thread (wave, lane): KQ key channels from KQ * wave, value channels lane (and lane + 64);
// the waves' partial read-outs meet in LDS once a row.
// LONG: any number of rows, kGlaShort of them in LDS at a time.
template <typename T, int KQ, int NV, bool LONG>
__device__ __forceinline__ void gla_walk(float* lds, T* __restrict__ out, const T* __restrict__ q, int64_t q_stride, const T* __restrict__ k,
                                int64_t k_stride, const T* __restrict__ v, int64_t v_stride, const float* __restrict__ z, float inv_tau,
                                float* __restrict__ state, const T* __restrict__ gate, int64_t gate_stride, const float* __restrict__ gain,
                                int64_t row0, int rows, int heads, int head, int dk, int dv, float scale, float eps) {
    constexpr int C = 4 * KQ, V = 16 * NV, VL = NV / 4;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float* sq = lds;                       // [n][C], k and a likewise, zeros past dk
    float* sk = sq + kGlaShort * C;
    float* sa = sk + kGlaShort * C;
    float* sv = sa + kGlaShort * C;        // [n][V]
    float* so = sv + kGlaShort * V;        // [n][V] read-outs
    float* part = so + kGlaShort * V;      // [2][4][V]
    float S[KQ][VL];
#pragma unroll
    for (int c = 0; c < KQ; ++c)
#pragma unroll
        for (int u = 0; u < VL; ++u) {
            const int kk = wave * KQ + c, col = lane + 64 * u;
            const float x = state[(int64_t)min(kk, dk - 1) * dv + min(col, dv - 1)];
            S[c][u] = kk < dk && col < dv ? x : 0.f;
        }
    do {
        const int n = LONG ? min(rows, kGlaShort) : rows;
        for (int e = tid; e < n * C; e += 256) {
            const int j = e / C, c = e - j * C;
            const int64_t at = (int64_t)head * dk + min(c, dk - 1), row = row0 + j;
            const float x = Elem<T>::load(q + row * q_stride + at), y = Elem<T>::load(k + row * k_stride + at), f = gla_decay(z[row * heads * dk + at], inv_tau);
            sq[e] = c < dk ? x * scale : 0.f;
            sk[e] = c < dk ? y : 0.f;
            sa[e] = c < dk ? f : 0.f;
        }
        for (int e = tid; e < n * V; e += 256) {
            const int j = e / V, c = e - j * V;
            const float x = Elem<T>::load(v + (row0 + j) * v_stride + (int64_t)head * dv + min(c, dv - 1));
            sv[e] = c < dv ? x : 0.f;
        }
        __syncthreads();
        for (int j = 0; j < n; ++j) {
            float* p = part + (j & 1) * 4 * V;
            float vv[VL];
            float4 acc[VL];                    // (sums in short chains)
#pragma unroll
            for (int u = 0; u < VL; ++u) { vv[u] = sv[j * V + lane + 64 * u]; acc[u] = make_float4(0.f, 0.f, 0.f, 0.f); }
#pragma unroll
            for (int c = 0; c < KQ; c += 4) {
                const float4 q4 = *reinterpret_cast<const float4*>(sq + j * C + wave * KQ + c);
                const float4 k4 = *reinterpret_cast<const float4*>(sk + j * C + wave * KQ + c);
                const float4 a4 = *reinterpret_cast<const float4*>(sa + j * C + wave * KQ + c);
#pragma unroll
                for (int u = 0; u < VL; ++u) {
                    S[c][u] = fmaf(a4.x, S[c][u], k4.x * vv[u]);         acc[u].x = fmaf(S[c][u], q4.x, acc[u].x);
                    S[c + 1][u] = fmaf(a4.y, S[c + 1][u], k4.y * vv[u]); acc[u].y = fmaf(S[c + 1][u], q4.y, acc[u].y);
                    S[c + 2][u] = fmaf(a4.z, S[c + 2][u], k4.z * vv[u]); acc[u].z = fmaf(S[c + 2][u], q4.z, acc[u].z);
                    S[c + 3][u] = fmaf(a4.w, S[c + 3][u], k4.w * vv[u]); acc[u].w = fmaf(S[c + 3][u], q4.w, acc[u].w);
                }
            }
#pragma unroll
            for (int u = 0; u < VL; ++u) p[wave * V + lane + 64 * u] = (acc[u].x + acc[u].y) + (acc[u].z + acc[u].w);
            __syncthreads();                   // (the other half of `part` was read before this row's sums were written)
            if (tid < V) so[j * V + tid] = (p[tid] + p[V + tid]) + (p[2 * V + tid] + p[3 * V + tid]);
        }
        __syncthreads();
        for (int j = wave; j < n; j += 4) {
            float x[VL], ss = 0.f;
#pragma unroll
            for (int u = 0; u < VL; ++u) { x[u] = so[j * V + lane + 64 * u]; ss = fmaf(x[u], x[u], ss); }
            const float r = 1.f / sqrtf(wave_sum(ss) / (float)dv + eps);
#pragma unroll
            for (int u = 0; u < VL; ++u) {
                const int col = lane + 64 * u;
                if (col >= dv) continue;
                const float y = Elem<T>::load(gate + (row0 + j) * gate_stride + (int64_t)head * dv + col);
                Elem<T>::store(out + ((row0 + j) * heads + head) * dv + col, x[u] * r * gain[col] * (y / (1.f + expf(-y))));
            }
        }
        if (LONG) __syncthreads();             // the rows have been read
        rows -= kGlaShort;
        row0 += kGlaShort;
    } while (LONG && rows > 0);
#pragma unroll
    for (int c = 0; c < KQ; ++c)
#pragma unroll
        for (int u = 0; u < VL; ++u) {
            const int kk = wave * KQ + c, col = lane + 64 * u;
            if (kk < dk && col < dv) state[(int64_t)kk * dv + col] = S[c][u];
        }
}

// Steps of single tokens: grid (heads, items), a kernel of its own, whose few registers leave room for three workgroups a unit.  (That
// there are no longer items is about speed alone: the second walk takes them, at the price of registers in scratch.)
template <typename T, int KQ, int NV>
__global__ __launch_bounds__(256, KQ * NV <= 64 ? 6 : KQ * NV <= 128 ? 4 : 3) void gla_walk_kernel(
    T* __restrict__ out, const T* __restrict__ q, int64_t q_stride, const T* __restrict__ k, int64_t k_stride, const T* __restrict__ v,
    int64_t v_stride, const float* __restrict__ z, float inv_tau, float* __restrict__ state, const T* __restrict__ gate, int64_t gate_stride,
    const float* __restrict__ gain, const int* __restrict__ item_len, const int* __restrict__ item_tok_off,
    const int* __restrict__ item_slot, int heads, int dk, int dv, float scale, float eps) {
    extern __shared__ __attribute__((aligned(16))) float gla_lds[];
    const int head = blockIdx.x, item = blockIdx.y, slot = item_slot[item], len = item_len[item];
    if (slot < 0 || len <= 0) return;
    if (len <= kGlaShort)
        gla_walk<T, KQ, NV, false>(gla_lds, out, q, q_stride, k, k_stride, v, v_stride, z, inv_tau, state + ((int64_t)slot * heads + head) * dk * dv, gate,
                            gate_stride, gain, item_tok_off[item], len, heads, head, dk, dv, scale, eps);
    else
        gla_walk<T, KQ, NV, true>(gla_lds, out, q, q_stride, k, k_stride, v, v_stride, z, inv_tau, state + ((int64_t)slot * heads + head) * dk * dv, gate,
                            gate_stride, gain, item_tok_off[item], len, heads, head, dk, dv, scale, eps);
}

template <int KQ, int NV>
struct GlaOutLds {
    static constexpr int KS = 4 * KQ + 4, VS = 16 * NV + 4;
    static constexpr int second = KS > VS ? 64 * KS : 64 * VS;
    static constexpr size_t bytes = sizeof(float) * (size_t)(64 * KS + second + 64 * VS + 32 * KQ);
    static constexpr size_t walk = sizeof(float) * (size_t)(kGlaShort * (12 * KQ + 32 * NV) + 128 * NV);
    static_assert(walk <= bytes, "the short items' rows fit the chunks' LDS");
};

template <typename T, int KQ, int NV, bool VEC>
__global__ __launch_bounds__(256, KQ == 16 && NV == 4 ? 3 : 1) void gla_out_kernel(
    T* __restrict__ out, const T* __restrict__ q, int64_t q_stride, const T* __restrict__ k, int64_t k_stride, const T* __restrict__ v,
    int64_t v_stride, const float* __restrict__ z, float inv_tau, const float* __restrict__ S0, float* __restrict__ state, const T* __restrict__ gate, int64_t gate_stride,
    const float* __restrict__ gain, const int* __restrict__ item_len, const int* __restrict__ item_tok_off,
    const int* __restrict__ item_slot, int num_items, int chunks, int heads, int dk, int dv, float scale, float eps) {
    extern __shared__ __attribute__((aligned(16))) float gla_lds[];
    using L = GlaOutLds<KQ, NV>;
    const int head = blockIdx.x, idx = blockIdx.y, tid = threadIdx.x;
    int item = idx - chunks, chunk;
    if (item >= 0) {
        if (item_slot[item] < 0 || item_len[item] <= 0 || item_len[item] > kGlaShort) return;
        gla_walk<T, KQ, NV, false>(gla_lds, out, q, q_stride, k, k_stride, v, v_stride, z, inv_tau,
                            state + ((int64_t)item_slot[item] * heads + head) * dk * dv, gate, gate_stride, gain, item_tok_off[item],
                            item_len[item], heads, head, dk, dv, scale, eps);
        return;
    }
    if (!find_chunk(idx, item_len, item_slot, num_items, item, chunk, kChunkRows, kGlaShort)) return;
    const int n = min(kChunkRows, item_len[item] - chunk * kChunkRows);
    const int64_t row0 = (int64_t)item_tok_off[item] + (int64_t)chunk * kChunkRows;
    float* ks = gla_lds;
    float* as = ks + 64 * L::KS;
    float* vs = as + L::second;
    double* bp = reinterpret_cast<double*>(vs + 64 * L::VS);
    const int lane = tid & 63, wave = tid >> 6, r16 = lane & 15, g = lane >> 4, p16 = double_row(r16);
    const int i = wave * 16 + r16;                             // this lane's row of the chunk
    const bool row_ok = i < n;
    {
        GlaTile<KQ> tk, ta;
        GlaTile<4 * NV> tv;
        tk.template load<T, VEC>(k + row0 * k_stride + (int64_t)head * dk, k_stride, n, 0, dk, 0.f);
        ta.template load<float, VEC>(z + (row0 * heads + head) * dk, (int64_t)heads * dk, n, 0, dk, FLT_MAX);
        tv.template load<T, VEC>(v + row0 * v_stride + (int64_t)head * dv, v_stride, n, 0, dv, 0.f);
        tk.store(ks, L::KS);
        ta.store_decays(as, L::KS, inv_tau);
        tv.store(vs, L::VS);
    }
    double qd[KQ];
    {
        const T* qr = q + (row0 + min(i, n - 1)) * q_stride + (int64_t)head * dk;
#pragma unroll
        for (int s = 0; s < KQ / 4; ++s) {
            const float4 x = gla_piece<T, VEC>(qr, 16 * s + 4 * g, dk, row_ok, 0.f);
            qd[4 * s] = x.x * (double)scale; qd[4 * s + 1] = x.y * (double)scale; qd[4 * s + 2] = x.z * (double)scale; qd[4 * s + 3] = x.w * (double)scale;
        }
    }
    // the start state's first 64 key channels, on their way during the scores
    const float* s0 = S0 + ((int64_t)idx * heads + head) * dk * dv;
    GlaTile<4 * NV> ts;
    ts.template load<float, VEC>(s0, dv, min(dk, 64), 0, dv, 0.f);
    __syncthreads();
    doublex4 st[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) st[t] = doublex4{0.0, 0.0, 0.0, 0.0};
    doublex4 diag = doublex4{0.0, 0.0, 0.0, 0.0};
    float* kw = ks + wave * 16 * L::KS + 4 * g;
    const float* aw = as + wave * 16 * L::KS + 4 * g;
    if (wave * 16 < n) {                                       // (uniform over the wave)
#pragma unroll
        for (int j = 15; j >= 0; --j) {
            if (j < 15 && r16 > j) {
#pragma unroll
                for (int s = 0; s < KQ / 4; ++s) {
                    const float4 f = *reinterpret_cast<const float4*>(aw + (j + 1) * L::KS + 16 * s);
                    qd[4 * s] *= f.x; qd[4 * s + 1] *= f.y; qd[4 * s + 2] *= f.z; qd[4 * s + 3] *= f.w;
                }
            }
            double d[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int s = 0; s < KQ / 4; ++s) {
                const float4 x = *reinterpret_cast<const float4*>(kw + j * L::KS + 16 * s);
                d[0] = fma(qd[4 * s], (double)x.x, d[0]); d[1] = fma(qd[4 * s + 1], (double)x.y, d[1]);
                d[2] = fma(qd[4 * s + 2], (double)x.z, d[2]); d[3] = fma(qd[4 * s + 3], (double)x.w, d[3]);
            }
            double dot = (d[0] + d[1]) + (d[2] + d[3]);
            dot += __shfl_xor(dot, 16, 64);
            dot += __shfl_xor(dot, 32, 64);
            if (g == j >> 2) diag[j & 3] = r16 >= j ? dot : 0.0;
        }
#pragma unroll
        for (int s = 0; s < KQ / 4; ++s) {                     // the block's first row: qd is q^ now
            const float4 f = *reinterpret_cast<const float4*>(aw + 16 * s);
            qd[4 * s] *= f.x; qd[4 * s + 1] *= f.y; qd[4 * s + 2] *= f.z; qd[4 * s + 3] *= f.w;
        }
        // k^ in the place of k (this wave's own rows), and the block's decay
        for (int c = lane; c < 4 * KQ; c += 64) {
            double run = 1.0;
            float* kc = ks + wave * 16 * L::KS + c;
            const float* ac = as + wave * 16 * L::KS + c;
#pragma unroll
            for (int j = 15; j >= 0; --j) {
                kc[j * L::KS] = (float)(kc[j * L::KS] * run);
                run *= ac[j * L::KS];
            }
            bp[wave * 4 * KQ + c] = run;
        }
    }
    __syncthreads();
#pragma unroll
    for (int t = 2; t >= 0; --t) {
        if (t >= wave || 16 * wave >= n) continue;             // uniform over the wave
#pragma unroll
        for (int s = 0; s < KQ / 4; ++s) {
            const float4 x = *reinterpret_cast<const float4*>(ks + (16 * t + p16) * L::KS + 16 * s + 4 * g);
            st[t] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)x.x, qd[4 * s], st[t], 0, 0, 0);
            st[t] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)x.y, qd[4 * s + 1], st[t], 0, 0, 0);
            st[t] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)x.z, qd[4 * s + 2], st[t], 0, 0, 0);
            st[t] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)x.w, qd[4 * s + 3], st[t], 0, 0, 0);
        }
#pragma unroll
        for (int s = 0; s < KQ / 4; ++s) {
            const double* f = bp + t * 4 * KQ + 16 * s + 4 * g;
            qd[4 * s] *= f[0]; qd[4 * s + 1] *= f[1]; qd[4 * s + 2] *= f[2]; qd[4 * s + 3] *= f[3];
        }
    }
    doublex4 o[NV];
#pragma unroll
    for (int vt = 0; vt < NV; ++vt) o[vt] = doublex4{0.0, 0.0, 0.0, 0.0};
    // what the chunk's start state gives
#pragma unroll
    for (int b = 0; b < (KQ + 15) / 16; ++b) {
        if (64 * b >= dk) continue;
        if (b > 0) __syncthreads();                            // the channels before have been read (the decays: above)
        ts.store(as, L::VS);
        __syncthreads();
        if (64 * (b + 1) < dk)
            ts.template load<float, VEC>(s0 + (int64_t)64 * (b + 1) * dv, dv, min(dk - 64 * (b + 1), 64), 0, dv, 0.f);
#pragma unroll
        for (int s = 0; s < (KQ < 16 ? KQ : 16); ++s) {
            const float* sr = as + (16 * (s >> 2) + 4 * g + (s & 3)) * L::VS + p16;
#pragma unroll
            for (int vt = 0; vt < NV; ++vt)
                o[vt] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)sr[16 * vt], qd[(16 * b + s) % KQ], o[vt], 0, 0, 0);
        }
    }
    // A row meets the later rows of its block with a weight of zero, which an infinity or NaN among their values would turn into
    // NaN: such a block's rows are summed one by one instead, below.
    float zero = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int vt = 0; vt < NV; ++vt) zero = fmaf(vs[(16 * wave + 4 * g + r) * L::VS + 16 * vt + r16], 0.f, zero);
    const bool finite = !__any(!(zero == 0.f));
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        if (t > wave || 16 * wave >= n || (t == wave && !finite)) continue;
        const doublex4 p = t == wave ? diag : st[t];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float* vr = vs + (16 * t + 4 * g + r) * L::VS + p16;
#pragma unroll
            for (int vt = 0; vt < NV; ++vt) o[vt] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)vr[16 * vt], p[r], o[vt], 0, 0, 0);
        }
    }
    if (!finite) {
#pragma unroll 1
        for (int j4 = 0; j4 < 4; ++j4)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const double w = __shfl(diag[e], r16 + 16 * j4, 64);
                if (4 * j4 + e > r16) continue;
#pragma unroll
                for (int vt = 0; vt < NV; ++vt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[vt][r] = fma(w, (double)vs[(16 * wave + 4 * j4 + e) * L::VS + 16 * vt + 4 * g + r], o[vt][r]);
            }
    }
    // o[vt][r]: value channel 16 vt + 4 g + r of row i
    float ss = 0.f;
    floatx4 of[NV];
#pragma unroll
    for (int vt = 0; vt < NV; ++vt)
#pragma unroll
        for (int r = 0; r < 4; ++r) { of[vt][r] = (float)o[vt][r]; ss = fmaf(of[vt][r], of[vt][r], ss); }      // (channels past dv are zeros)
    ss = rows4_sum(ss);
    if (!row_ok) return;
    const float rms = 1.f / sqrtf(ss / (float)dv + eps);
    const T* gr = gate + (row0 + i) * gate_stride + (int64_t)head * dv;
    T* dst = out + (row0 + i) * ((int64_t)heads * dv) + (int64_t)head * dv;
#pragma unroll
    for (int vt = 0; vt < NV; ++vt) {
        const int v0 = 16 * vt + 4 * g;
        if (v0 >= dv) continue;
        const float4 x = gla_piece<T, VEC>(gr, v0, dv, true, 0.f), w = gla_piece<float, false>(gain, v0, dv, true, 0.f);
        const float y[4] = {of[vt][0] * rms * w.x * (x.x / (1.f + expf(-x.x))), of[vt][1] * rms * w.y * (x.y / (1.f + expf(-x.y))),
                            of[vt][2] * rms * w.z * (x.z / (1.f + expf(-x.z))), of[vt][3] * rms * w.w * (x.w / (1.f + expf(-x.w)))};
        if (VEC) Elem<T>::store4(dst + v0, y);
        else
            for (int r = 0; r < 4 && v0 + r < dv; ++r) Elem<T>::store(dst + v0 + r, y[r]);
    }
}

template <typename T, int KQ, bool VEC>
static int launch_gla_sums(float* U, float* A, const void* k, int64_t ks, const void* v, int64_t vs, const float* z, float inv_tau, const int* item_len,
                           const int* item_tok_off, const int* item_slot, int num_items, unsigned chunks, int heads, int dk, int dv,
                           hipStream_t stream) {
    constexpr int kLds = (int)sizeof(float) * (2 * 64 * (4 * KQ + 4) + 64 * 68 + 32 * KQ);
    ST_CHECK(hipFuncSetAttribute((const void*)gla_sums_kernel<T, KQ, VEC>, hipFuncAttributeMaxDynamicSharedMemorySize, kLds) == hipSuccess,
             "gla_chunks: cannot raise the LDS limit");
    gla_sums_kernel<T, KQ, VEC><<<dim3(heads, chunks, (dv + 63) / 64), 256, kLds, stream>>>(U, A, (const T*)k, ks, (const T*)v, vs, z, inv_tau, item_len,
        item_tok_off, item_slot, num_items, heads, dk, dv);
    ST_LAUNCH_CHECK("gla_chunks (sums)");
    return 0;
}

template <typename T, int KQ, int NV, bool VEC>
static int launch_gla_out(void* out, const void* q, int64_t qs, const void* k, int64_t ks, const void* v, int64_t vs, const float* z, float inv_tau,
                          const float* S0, float* state, const void* gate, int64_t gs, const float* gain, const int* item_len, const int* item_tok_off,
                          const int* item_slot, int num_items, unsigned chunks, int heads, int dk, int dv, float scale, float eps,
                          bool walk_only, hipStream_t stream) {
    constexpr int kLds = (int)GlaOutLds<KQ, NV>::bytes;
    if (walk_only) {
        gla_walk_kernel<T, KQ, NV><<<dim3(heads, num_items), 256, GlaOutLds<KQ, NV>::walk, stream>>>((T*)out, (const T*)q, qs, (const T*)k, ks,
            (const T*)v, vs, z, inv_tau, state, (const T*)gate, gs, gain, item_len, item_tok_off, item_slot, heads, dk, dv, scale, eps);
        ST_LAUNCH_CHECK("gla_chunks (single rows)");
        return 0;
    }
    ST_CHECK(hipFuncSetAttribute((const void*)gla_out_kernel<T, KQ, NV, VEC>, hipFuncAttributeMaxDynamicSharedMemorySize, kLds) == hipSuccess,
             "gla_chunks: cannot raise the LDS limit");
    gla_out_kernel<T, KQ, NV, VEC><<<dim3(heads, chunks + num_items), 256, kLds, stream>>>((T*)out, (const T*)q, qs, (const T*)k, ks,
        (const T*)v, vs, z, inv_tau, S0, state,
        (const T*)gate, gs, gain, item_len, item_tok_off, item_slot, num_items, (int)chunks, heads, dk, dv, scale, eps);
    ST_LAUNCH_CHECK("gla_chunks (outputs)");
    return 0;
}

}  // namespace st

using namespace st;

// scratch: float [chunks][heads][key_dim * value_dim] then [chunks][heads][key_dim], chunks = num_rows / 64 and one more for each of
// the items that may have more than 16 rows (num_items, or num_rows / 17 where that is less); may be null where that is none, and for
// steps of single tokens, `single`
extern "C" int st_gla_chunks(void* out, const void* q, int64_t q_stride, const void* k, int64_t k_stride, const void* v, int64_t v_stride,
                             const float* z, float inv_tau, const void* gate, int64_t gate_stride, const float* gain, float* state, const int* item_len,
                             const int* item_tok_off, const int* item_slot, int num_items, int num_rows, int heads, int key_dim,
                             int value_dim, float scale, float eps, float* scratch, int64_t scratch_chunks, int single, int dtype, hipStream_t stream) {
    ST_CHECK(num_items >= 0 && num_rows >= 0 && heads > 0 && key_dim > 0 && value_dim > 0, "gla_chunks: bad sizes");
    ST_CHECK(key_dim <= 128 && value_dim <= 128, "gla_chunks: up to 128 key and 128 value channels a head, not %d and %d", key_dim, value_dim);
    ST_CHECK(dtype == kF32 || dtype == kBF16, "gla_chunks: unknown dtype %d", dtype);
    ST_CHECK(eps > 0.f, "gla_chunks: eps must be positive");
    if (num_items == 0 || num_rows == 0) return 0;
    ST_CHECK(out && q && k && v && z && gate && gain && state && item_len && item_tok_off && item_slot, "gla_chunks: null operand");
    const int64_t chunks = single ? 0 : most_chunks(num_rows, num_items, kGlaShort);
    ST_CHECK(chunks == 0 || (scratch && scratch_chunks >= chunks), "gla_chunks: scratch for %lld chunks, %lld needed", (long long)scratch_chunks, (long long)chunks);
    ST_CHECK(chunks + num_items <= 65535, "gla_chunks: too many chunks or items");
    float* U = scratch;
    float* A = scratch + scratch_chunks * heads * key_dim * value_dim;
    // four numbers at a time: rows and heads start on their size, and the tables on 16 bytes
    const uintptr_t low = (uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)gate | (uintptr_t)out;
    const bool vec = ((key_dim | value_dim) & 3) == 0 && ((q_stride | k_stride | v_stride | gate_stride) & 3) == 0 &&
                     (low & (dtype == kF32 ? 15 : 7)) == 0 && (((uintptr_t)z | (uintptr_t)scratch) & 15) == 0;
    int rc = 0;
#define ST_GLA_SUMS(T, KQ, V)                                                                                                     \
    rc = launch_gla_sums<T, KQ, V>(U, A, k, k_stride, v, v_stride, z, inv_tau, item_len, item_tok_off, item_slot, num_items, (unsigned)chunks, \
                                   heads, key_dim, value_dim, stream)
#define ST_GLA_OUT(T, KQ, NV, V)                                                                                                  \
    rc = launch_gla_out<T, KQ, NV, V>(out, q, q_stride, k, k_stride, v, v_stride, z, inv_tau, U, state, gate, gate_stride, gain, item_len, \
                                      item_tok_off, item_slot, num_items, (unsigned)chunks, heads, key_dim, value_dim, scale, eps, single != 0, stream)
#define ST_GLA_T(what, ...)                                                        \
    do {                                                                           \
        if (dtype == kF32) { if (vec) what(float, __VA_ARGS__, true); else what(float, __VA_ARGS__, false); }      \
        else { if (vec) what(bf16_t, __VA_ARGS__, true); else what(bf16_t, __VA_ARGS__, false); }                  \
    } while (0)
    if (chunks) {
        if (key_dim <= 64) ST_GLA_T(ST_GLA_SUMS, 16);
        else ST_GLA_T(ST_GLA_SUMS, 32);
        if (rc) return rc;
        gla_carry_kernel<<<dim3(heads, num_items, (unsigned)((key_dim * value_dim + 255) / 256)), 256, 0, stream>>>(U, A, state, item_len,
                                                                                              item_slot, heads, key_dim, value_dim);
        ST_LAUNCH_CHECK("gla_chunks (carry)");
    }
    if (key_dim <= 64 && value_dim <= 64) ST_GLA_T(ST_GLA_OUT, 16, 4);
    else if (key_dim <= 64) ST_GLA_T(ST_GLA_OUT, 16, 8);
    else if (value_dim <= 64) ST_GLA_T(ST_GLA_OUT, 32, 4);
    else ST_GLA_T(ST_GLA_OUT, 32, 8);
#undef ST_GLA_T
#undef ST_GLA_OUT
#undef ST_GLA_SUMS
    return rc;
}
