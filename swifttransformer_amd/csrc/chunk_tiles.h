// Pieces of the recurrences that go by chunks of rows: which rows a chunk has, and tiles of rows on their way to LDS.
#pragma once

#include "common.h"

#include <type_traits>

namespace st {

constexpr int kChunkRows = 64;       // counted from an item's first row of the step

// an item's chunks: none for items of up to `least` rows, which the kernels that say so take without chunks
__device__ inline int chunks_of(int len, int slot, int rows, int least = 0) { return slot >= 0 && len > least ? (len + rows - 1) / rows : 0; }
// at most so many chunks has a step whose items have chunks from `least` + 1 rows on: every item's last one may be a short one
inline int64_t most_chunks(int64_t rows, int64_t items, int least) {
    return rows / kChunkRows + (items < rows / (least + 1) ? items : rows / (least + 1));
}

// The chunk of an item that a global chunk index means; false past the last one (`chunk` is then how far).  Whole waves: a lane an item, so that the items'
// lengths are one trip to memory and not one after the other (48 rows beside 24 single tokens through gla_chunks: 109 -> 91 us).
__device__ inline bool find_chunk(int idx, const int* __restrict__ item_len, const int* __restrict__ item_slot, int num_items, int& item,
                                  int& chunk, int rows = kChunkRows, int least = 0) {
    const int lane = threadIdx.x & 63;
    int base = 0;
    for (int b0 = 0; b0 < num_items; b0 += 64) {
        const int b = min(b0 + lane, num_items - 1), len = item_len[b], slot = item_slot[b];
        const int own = b0 + lane < num_items ? chunks_of(len, slot, rows, least) : 0;
        int upto = own;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int up = __shfl_up(upto, o, 64);
            if (lane >= o) upto += up;
        }
        const uint64_t past = __ballot(base + upto > idx);
        if (past) {
            const int at = __ffsll((unsigned long long)past) - 1;
            item = __builtin_amdgcn_readfirstlane(b0 + at);
            chunk = __builtin_amdgcn_readfirstlane(idx - base - __shfl(upto - own, at, 64));
            return true;
        }
        base += __shfl(upto, 63, 64);
    }
    chunk = __builtin_amdgcn_readfirstlane(idx - base);
    return false;
}

// the chunks of all items before `item`; whole waves
__device__ inline int chunks_before(int item, const int* __restrict__ item_len, const int* __restrict__ item_slot, int rows = kChunkRows,
                                    int least = 0) {
    const int lane = threadIdx.x & 63;
    int sum = 0;
    for (int b = lane; b < item; b += 64) sum += chunks_of(item_len[b], item_slot[b], rows, least);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
    return __builtin_amdgcn_readfirstlane(sum);
}

// S <- keep * S + add over an item's chunks: `u` holds an element of the chunks' sums (step floats apart) and receives the state that
// each chunk starts from, `f` their factors; returns the last S.
__device__ inline float carry_states(float* __restrict__ u, int64_t u_step, const float* __restrict__ f, int64_t f_step, int chunks, float S) {
    int c0 = 0;
    auto batch = [&](auto count) {                             // so many chunks' operands on their way at once
        constexpr int B = decltype(count)::value;
        for (; c0 + B <= chunks; c0 += B) {
            float add[B], keep[B];
#pragma unroll
            for (int b = 0; b < B; ++b) {
                add[b] = u[(c0 + b) * u_step];
                keep[b] = f[(c0 + b) * f_step];
            }
#pragma unroll
            for (int b = 0; b < B; ++b) {
                u[(c0 + b) * u_step] = S;
                S = fmaf(keep[b], S, add[b]);
            }
        }
    };
    batch(std::integral_constant<int, 16>());
    batch(std::integral_constant<int, 4>());
    batch(std::integral_constant<int, 1>());
    return S;
}

typedef double doublex4 __attribute__((ext_vector_type(4)));

// The matrix instruction for doubles (v_mfma_f64_16x16x4_f64) leaves rows g + 4 r of its result with a lane's group g, the one for floats
// rows 4 g + r; with the first operand's rows dealt like this a lane gets what it gets from the one for floats.
__device__ inline int double_row(int r16) { return 4 * (r16 & 3) + (r16 >> 2); }

// e^x for x <= 0 to 2^-31 of itself (the Taylor sum up to r^8 on |r| <= ln(2) / 2), so that a weight is rounded to float once, with
// all its factors; 0 below e^-200, which is none in float.  Doubles take as long as floats here, and a dozen of them no longer than
// the library's expf.
__device__ __forceinline__ double exp_le0_double(double x) {
    x = x < -200.0 ? -200.0 : x;
    const double n = rint(x * 1.4426950408889634), r = fma(n, -0.69314718055994531, x);
    double y = 1.0 / 40320.0;
    y = fma(y, r, 1.0 / 5040.0);
    y = fma(y, r, 1.0 / 720.0);
    y = fma(y, r, 1.0 / 120.0);
    y = fma(y, r, 1.0 / 24.0);
    y = fma(y, r, 1.0 / 6.0);
    y = fma(y, r, 0.5);
    y = fma(y, r, 1.0);
    y = fma(y, r, 1.0);
    return ldexp(y, (int)n);
}

// Four neighbouring floats of a row, zeros past its `limit` numbers or where the row does not exist.  VEC: the row starts
// on 16 bytes and the limit is a multiple of 4.  (Addresses are clamped and values cleared rather than loads behind a
// branch: the loads of a tile are then all on their way at once.)
template <bool VEC>
__device__ inline float4 load_piece(const float* __restrict__ row, int c, int limit, bool ok) {
    float4 v;
    if (VEC) {
        v = *reinterpret_cast<const float4*>(row + min(c, limit - 4));
    } else {
        v.x = row[min(c, limit - 1)];
        v.y = row[min(c + 1, limit - 1)];
        v.z = row[min(c + 2, limit - 1)];
        v.w = row[min(c + 3, limit - 1)];
    }
    v.x = ok && c < limit ? v.x : 0.f;
    v.y = ok && c + 1 < limit ? v.y : 0.f;
    v.z = ok && c + 2 < limit ? v.z : 0.f;
    v.w = ok && c + 3 < limit ? v.w : 0.f;
    return v;
}

// A tile of 64 rows x 4 * P4 floats (P4 a power of two) by 256 threads: piece i of a thread is row e / P4, floats 4 (e % P4)
// on, e = thread + 256 i; P4 / 4 pieces a thread.
template <int P4>
struct Tile {
    static constexpr int kPieces = P4 / 4;
    float4 v[kPieces];
    template <bool VEC>
    __device__ inline void load(const float* __restrict__ base, int64_t stride, int rows, int first, int limit) {
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const int e = threadIdx.x + 256 * i, j = e / P4, c = 4 * (e % P4);
            v[i] = load_piece<VEC>(base + (int64_t)min(j, rows - 1) * stride, first + c, limit, j < rows);
        }
    }
    __device__ inline void store(float* lds, int lds_stride) const {
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const int e = threadIdx.x + 256 * i;
            *reinterpret_cast<float4*>(lds + (e / P4) * lds_stride + 4 * (e % P4)) = v[i];
        }
    }
    __device__ inline void store_weighted(float* lds, int lds_stride, const float* w) const {
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const int e = threadIdx.x + 256 * i;
            const float f = w[e / P4];
            *reinterpret_cast<float4*>(lds + (e / P4) * lds_stride + 4 * (e % P4)) = make_float4(v[i].x * f, v[i].y * f, v[i].z * f, v[i].w * f);
        }
    }
};

}  // namespace st
