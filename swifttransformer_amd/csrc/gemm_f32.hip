// Float products of prompt-sized inputs on the bfloat16 matrix cores: y = x * W^T (+bias)(activation)(+residual),
// x[M,K], W[N,K] contiguous along K, float in and out.
//
// A float has 24 significant bits and a bfloat16 eight, so a float is the sum of three bfloat16 numbers, a = a0 + a1 + a2, exactly
// (each the rounded rest of the ones before it; a1 is at most 2^-9 of a, a2 2^-18).  Of the nine products of two such sums six are
// formed, a0 b0, a0 b1, a1 b0, a0 b2, a1 b1 and a2 b0, each exact in the matrix cores, whose sums are float; the three left out are
// together at most 2^-25.9 of |a b|, a quarter of a float product's own rounding.  a0 b0 has a sum of its own and the five small ones
// another, 2^-8 of it, which meet at the end: a product then takes one rounding of a running sum at full size, as with float products, and
// 16 products in depth share one where the float matrix instruction takes four or eight.  (One sum for all six: six roundings, and more
// error than float products where most of x is zero, 1.2 times at 10 % and 1.6 at 0.2 % of 701 x 6,144 x 2,048, at the same speed.)
// Error against float64 (x normal, W normal of 0.02), the library's float product and this: 701 x 6,144 x 2,048 8.1e-7 and 1.8e-7, with 1 % of x
// not zero 8.5e-8 and 3.9e-8, with 0.2 % 4.4e-8 and 3.0e-8; 701 x 2,048 x 8,192 1.6e-6 and 1.7e-7, 1.6e-7 and 5.7e-8, 7.7e-8 and 5.2e-8;
// 1,500 x 2,560 x 2,560 9.1e-7 and 2.1e-7, 9.4e-8 and 3.8e-8, 4.8e-8 and 2.8e-8.
//
// Where the parts do not do, a result is formed again by float products (a block of 64 x 64 at once; the others of the block keep theirs, so
// that no row's numbers change what another row gets):
// - Its row of either matrix holds a number that is more than its three parts.  bfloat16's least number is 2^-133, so numbers below 2^-109 may
//   be, whatever they are multiplied by.  The third part is the upper half of what the first two leave, and the row is marked if a lower half
//   is not zero (one instruction for two numbers; 701 x 6,144 x 2,048 takes 3 % longer for it).
// - Its sum is not finite: infinities, NaN and numbers that round past bfloat16's largest make a NaN of products that float would not
//   (infinity times a part that is zero).
// - Its sum is below 2^-90 and not zero: products of small parts may be below float's least number where the whole product is not.
//
// What bounds it: the chip's power, more than its matrix cores (six products a float product, 0.9 to 1.1 PFLOP/s of them where a large
// bfloat16 product reaches 1.6): with one sum for all six the same launch took 381 us on normal numbers and 320 on zeros, 290 without loads,
// 270 with products and LDS reads alone (2,048 x 8,192 x 2,048).  So every number is split once a workgroup, by all waves, between the
// products (a step's products and splitting one after the other, by waves in turn or all alike: 392 and 383 us), and what is multiplied next is
// read from LDS while there are products left that do not need the registers.
// us, the library's best of 32 and this: 701 rows of 6,144 x 2,048 139 and 120, of 2,048 x 8,192 177 and 155, 1,500 rows of 2,560 x 2,560
// 149 and 115, of 768 x 3,072 61 and 54 (more beside gemm_f32_split_pays).
//
// Reference: cuBLAS calls (src/csrc/util/cublas_wrapper.cc:29).
#include "common.h"
#include "api.h"
#include "gemm_extras.h"
#include "activation.h"

#include <type_traits>

namespace st {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kTile = 128;       // rows of W and rows of x of a workgroup's tile
constexpr int kStep = 32;        // in depth
constexpr int kParts = 3;        // bfloat16 numbers a float
constexpr int kBufs = 3;         // steps in LDS: the one after that which is multiplied is read, the next written

// the next part of two numbers, which keep what is left of them
__device__ inline uint32_t split_off(float& a, float& b) {
    const uint32_t p = pack_bf16x2(a, b);
    a -= __uint_as_float(p << 16);
    b -= __uint_as_float(p & 0xffff0000u);
    return p;
}

// four consecutive features n0 .. n0+3 (N % 4 == 0) of row m with their bias and residual (zeros without)
__device__ inline void store_result(float* out, const float4& v, const float4& bias, const float4& residual, int act, int m, int n0, int N,
                                    const StGemmExtras& ex) {
    float r[4] = {v.x, v.y, v.z, v.w};
    if (!ex.bias_unscaled) { r[0] += bias.x; r[1] += bias.y; r[2] += bias.z; r[3] += bias.w; }
    apply_activation4(act, r);
    if (ex.out_scale != 0.f) { r[0] *= ex.out_scale; r[1] *= ex.out_scale; r[2] *= ex.out_scale; r[3] *= ex.out_scale; }
    if (ex.bias_unscaled) { r[0] += bias.x; r[1] += bias.y; r[2] += bias.z; r[3] += bias.w; }
    const float4 y = make_float4(r[0] + residual.x, r[1] + residual.y, r[2] + residual.z, r[3] + residual.w);
    *reinterpret_cast<float4*>(out + (int64_t)m * N + n0) = y;
    if (ex.k_cache && n0 >= ex.q_size) {             // (q_size and head_dim are multiples of four: one head's)
        int which;
        const int64_t dst = kv_scatter_offset(ex, m, n0, &which);
        if (dst >= 0) *reinterpret_cast<float4*>((float*)(which ? ex.v_cache : ex.k_cache) + dst) = y;
    }
}

// the multiple of eight that neighbouring workgroups go round by (the dies), undone: workgroups of a die get neighbouring numbers
__device__ inline int by_die(int i, int n) { return n % 8 ? i : (i & 7) * (n >> 3) + (i >> 3); }

// Workgroups 0 .. whole-1 make a tile each; the others a `splits`-th of the depth of one of the tiles after those, into `part`
// ([tile - whole][split][128 rows of x][128 features]), which gemm_f32_sum_kernel sums.  Tile t: rows of x t % tiles_m, features
// t / tiles_m (so that tiles of the same weights are neighbours).  M, N, K >= 1, N % 4 == K % 4 == 0.
__global__ __launch_bounds__(512) void gemm_f32_split_kernel(
    float* __restrict__ out, const float* __restrict__ x, const float* __restrict__ w, const float* bias, const float* residual,
    float* __restrict__ part, int M, int N, int K, int act, int tiles_m, int tiles, int whole, int splits, const StGemmExtras ex) {
    __shared__ uint4 lds[kBufs][kParts][2 * kTile * 4];   // rows of W, then rows of x: four pieces of eight in depth each
    __shared__ int s_lost[2 * kTile];                     // of these rows: whether they hold a number that is more than its parts
    int tile, split = 0;
    if ((int)blockIdx.x < whole) {
        tile = by_die(blockIdx.x, whole);
    } else {
        const int rest = tiles - whole, i = by_die(blockIdx.x - whole, rest * splits);
        split = i / rest;
        tile = whole + (i - split * rest);
    }
    const bool parted = tile >= whole && splits > 1;
    const int m0 = tile % tiles_m * kTile, n0 = tile / tiles_m * kTile;
    const int steps = K / kStep, share = tile < whole ? steps : (steps + splits - 1) / splits;
    const int begin = split * share, end = min(steps, begin + share);          // (the host leaves no split without a step)
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // waves 0 to 3 multiply the first half of every step, 4 to 7 the second; the four of a half a block of 64 x 64 each
    const int half = wave >> 2, wn = wave & 1, wm = (wave >> 1) & 1, l32 = lane & 31, lh = lane >> 5;

    // A thread brings piece j of a row of W and of one of x: numbers 4 j .. +3 and 16 + 4 j .. +3 of a step, so that four lanes read
    // 64 bytes that lie together (which numbers of a step a piece holds is the same for W and x, and no sum depends on it).  Rows
    // past the matrices stand for their last row: their results are not stored.
    const int j = tid & 3, row = tid >> 2;
    const float* src[2] = {w + (int64_t)min(n0 + row, N - 1) * K + 4 * j, x + (int64_t)min(m0 + row, M - 1) * K + 4 * j};
    float4 raw[2][2][2];                             // of a step of either parity
    auto load = [&](auto parity, int s) {            // (past the last step that one again: how many loads are on their way is always known)
        constexpr int P = decltype(parity)::value;
        const int k = min(s, end - 1) * kStep;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) raw[P][i][h] = *reinterpret_cast<const float4*>(src[i] + k + 16 * h);
    };
    // Part `i` % 12 / 4 of numbers 2 (i % 4) and the next of row `i` / 12; a row's pieces go to LDS when they are whole, rotated by row / 4:
    // 16 neighbouring rows' like pieces lie in different banks.
    uint32_t piece[kParts][4], lost[2] = {0, 0};     // (lower halves: of what the parts leave of the row of W, of x)
    auto take = [&](auto parity, int i, int buf) {
        constexpr int P = decltype(parity)::value;
        float4& v = raw[P][i / 12][i % 4 / 2];
        if (i % 12 / 4 < kParts - 1) {
            piece[i % 12 / 4][i % 4] = i % 2 ? split_off(v.z, v.w) : split_off(v.x, v.y);
        } else {
            const uint32_t lo = __float_as_uint(i % 2 ? v.z : v.x), hi = __float_as_uint(i % 2 ? v.w : v.y);
            piece[i % 12 / 4][i % 4] = __builtin_amdgcn_perm(hi, lo, 0x07060302);      // the upper halves of both
            lost[i / 12] |= lo | hi;
        }
        if (i % 12 == 11)
#pragma unroll
            for (int q = 0; q < kParts; ++q)
                lds[buf][q][(kTile * (i / 12) + row) * 4 + (j ^ ((row >> 2) & 3))] = make_uint4(piece[q][0], piece[q][1], piece[q][2], piece[q][3]);
    };
    auto park = [&](auto parity, int buf) {
#pragma unroll
        for (int i = 0; i < 24; ++i) take(parity, i, buf);
    };
    floatx16 acc[2][2], low[2][2];                   // the sums of a0 b0; of the other products
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int u = 0; u < 16; ++u) acc[a][b][u] = low[a][b][u] = 0.f;
    bf16x8 a[2][kParts], b[2][kParts];               // a step's operands
    const int at = l32 * 4 + ((half * 2 + lh) ^ ((l32 >> 2) & 3));
    auto fetch = [&](bf16x8 (&to)[2][kParts], int p, int buf) {
#pragma unroll
        for (int q = 0; q < 2; ++q)
            to[q][p] = __builtin_bit_cast(bf16x8, lds[buf][p][((&to == &a ? wn * 64 : kTile + wm * 64) + q * 32) * 4 + at]);
    };
    // this wave's pieces are in LDS and its operands in registers; then everyone's are (loads from memory may be on their way)
    auto meet = [&] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    const std::integral_constant<int, 0> even;
    const std::integral_constant<int, 1> odd;
    if (begin < end) {
        load(even, begin);
        load(odd, begin + 1);
        park(even, 0);
        load(even, begin + 2);
        park(odd, 1);
        load(odd, begin + 3);
        meet();
#pragma unroll
        for (int p = 0; p < kParts; ++p) {
            fetch(a, p, 0);
            fetch(b, p, 0);
        }
    }
    // Each of a step's 24 products, which the matrix core takes 32 cycles for, goes with a piece of the splitting of the step after next.
    // An operand is read for the next step when it has had its last product of this one, four products or more ahead of its first there.
    int buf = 0;                                     // of step s
    auto step = [&](auto parity, int s) {
        constexpr int kA[6] = {1, 1, 2, 0, 0, 0}, kB[6] = {1, 0, 0, 1, 0, 2};
        const int next = buf == kBufs - 1 ? 0 : buf + 1, free = next == kBufs - 1 ? 0 : next + 1;
#pragma unroll
        for (int i = 0; i < 24; ++i) {
            const int t = i >> 2, q = (i >> 1) & 1, r = i & 1;
            floatx16& sum = kA[t] + kB[t] ? low[q][r] : acc[q][r];
            __builtin_amdgcn_sched_barrier(0);
            sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[q][kA[t]], b[r][kB[t]], sum, 0, 0, 0);
            take(parity, i, free);
            if (i == 7) fetch(a, 1, next);
            if (i == 11) fetch(a, 2, next);
            if (i == 15) fetch(b, 1, next);
            if (i == 19) fetch(b, 0, next);
            if (i == 23) {
                fetch(a, 0, next);
                fetch(b, 2, next);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        load(parity, s + 4);
        meet();
        buf = next;
    };
    for (int s = begin; s < end; s += 2) {
        step(even, s);
        if (s + 1 < end) step(odd, s + 1);
    }
    // a row's four threads mark it; the halves' sums meet in LDS
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        int bits = (int)(lost[i] & 0xffffu);
        bits |= __shfl_xor(bits, 1, 64);
        bits |= __shfl_xor(bits, 2, 64);
        if (j == 0) s_lost[kTile * i + row] = bits;
    }
    float4* other = reinterpret_cast<float4*>(lds) + (wave & 3) * 2048 + lane;       // [4 waves][16 fours of acc and of low][64 lanes]
    if (half)
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int u4 = 0; u4 < 4; ++u4) {
                    const floatx16 &h = acc[q][r], &l = low[q][r];
                    other[((q * 2 + r) * 4 + u4) * 128] = make_float4(h[4 * u4], h[4 * u4 + 1], h[4 * u4 + 2], h[4 * u4 + 3]);
                    other[((q * 2 + r) * 4 + u4) * 128 + 64] = make_float4(l[4 * u4], l[4 * u4 + 1], l[4 * u4 + 2], l[4 * u4 + 3]);
                }
    __syncthreads();
    if (half) return;
    uint32_t most = 0, least = 0xffffffffu;          // of the sums' sizes, as whole numbers; of those that are not zero, less one
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int u4 = 0; u4 < 4; ++u4) {
                const float4 h = other[((q * 2 + r) * 4 + u4) * 128], l = other[((q * 2 + r) * 4 + u4) * 128 + 64];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float sum = (acc[q][r][4 * u4 + i] + (&h.x)[i]) + (low[q][r][4 * u4 + i] + (&l.x)[i]);
                    const uint32_t size = __float_as_uint(sum) & 0x7fffffffu;
                    acc[q][r][4 * u4 + i] = sum;
                    most = max(most, size);
                    least = min(least, size - 1);
                }
            }
    // acc[q][r][u]: feature n0 + wn * 64 + q * 32 + 8 * (u / 4) + 4 * lh + u % 4 of row m0 + wm * 64 + r * 32 + l32.
    // Numbers k0 .. k1-1 of the depth as float products, straight from memory (a lane brings every other four of a row's numbers):
    // what is left of the depth behind whole steps, and everything again where the parts do not do.
    auto plain = [&](floatx16 (&to)[2][2], int k0, int k1) {
        const float *wr[2], *xr[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            wr[q] = w + (int64_t)min(n0 + wn * 64 + q * 32 + l32, N - 1) * K;
            xr[q] = x + (int64_t)min(m0 + wm * 64 + q * 32 + l32, M - 1) * K;
        }
        for (int k = k0 + 4 * lh; k - 4 * lh < k1; k += 8) {
            float4 wv[2], xv[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                wv[q] = k < k1 ? *reinterpret_cast<const float4*>(wr[q] + k) : make_float4(0.f, 0.f, 0.f, 0.f);
                xv[q] = k < k1 ? *reinterpret_cast<const float4*>(xr[q] + k) : make_float4(0.f, 0.f, 0.f, 0.f);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int r = 0; r < 2; ++r)
                        to[q][r] = __builtin_amdgcn_mfma_f32_32x32x2f32((&wv[q].x)[i], (&xv[r].x)[i], to[q][r], 0, 0, 0);
        }
    };
    constexpr uint32_t kInf = 0x7f800000u, kSmall = 0x12800000u;     // infinity, 2^-90
    if (__any(s_lost[wn * 64 + lane] | s_lost[kTile + wm * 64 + lane] || most >= kInf || least < kSmall - 1)) {
        floatx16 again[2][2];
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int u = 0; u < 16; ++u) again[q][r][u] = 0.f;
        plain(again, begin * kStep, end * kStep);
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int u = 0; u < 16; ++u) {
                    const uint32_t size = __float_as_uint(acc[q][r][u]) & 0x7fffffffu;
                    if (s_lost[kTile + wm * 64 + r * 32 + l32] | s_lost[wn * 64 + q * 32 + 8 * (u / 4) + 4 * lh + u % 4] || size >= kInf ||
                        size - 1 < kSmall - 1)
                        acc[q][r][u] = again[q][r][u];
                }
    }
    if (end == steps && steps * kStep < K) plain(acc, steps * kStep, K);
    // What is added to the results is asked for before the first is stored: one trip to memory a row of the block, not one a store.
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int mt = wm * 64 + r * 32 + l32, m = m0 + mt;
        if (m >= M) continue;
        float4 add[2][4], rest[2][4];
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int u4 = 0; u4 < 4; ++u4) {
                const int n = n0 + wn * 64 + q * 32 + 8 * u4 + 4 * lh;
                add[q][u4] = bias && !parted && n < N ? *reinterpret_cast<const float4*>(bias + n) : make_float4(0.f, 0.f, 0.f, 0.f);
                rest[q][u4] = residual && !parted && n < N ? *reinterpret_cast<const float4*>(residual + (int64_t)m * N + n)
                                                           : make_float4(0.f, 0.f, 0.f, 0.f);
            }
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int u4 = 0; u4 < 4; ++u4) {
                const int nt = wn * 64 + q * 32 + 8 * u4 + 4 * lh, n = n0 + nt;
                if (n >= N) continue;
                const float4 v = make_float4(acc[q][r][4 * u4], acc[q][r][4 * u4 + 1], acc[q][r][4 * u4 + 2], acc[q][r][4 * u4 + 3]);
                if (parted)
                    *reinterpret_cast<float4*>(part + ((int64_t)(tile - whole) * splits + split) * (kTile * kTile) + mt * kTile + nt) = v;
                else
                    store_result(out, v, add[q][u4], rest[q][u4], act, m, n, N, ex);
            }
    }
}

// the parted tiles' results: a thread four features; grid (parted tiles, 16)
__global__ __launch_bounds__(256) void gemm_f32_sum_kernel(
    float* __restrict__ out, const float* __restrict__ part, const float* bias, const float* residual, int M, int N, int act, int tiles_m,
    int whole, int splits, const StGemmExtras ex) {
    const int at = blockIdx.y * 1024 + threadIdx.x * 4, tile = whole + blockIdx.x;
    const int m = tile % tiles_m * kTile + at / kTile, n = tile / tiles_m * kTile + at % kTile;
    if (m >= M || n >= N) return;
    const float* from = part + (int64_t)blockIdx.x * splits * (kTile * kTile) + at;
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
    const float4 add = bias ? *reinterpret_cast<const float4*>(bias + n) : zero;
    const float4 rest = residual ? *reinterpret_cast<const float4*>(residual + (int64_t)m * N + n) : zero;
    float4 sum = zero;
#pragma unroll 4
    for (int s = 0; s < splits; ++s) {
        const float4 v = *reinterpret_cast<const float4*>(from + (int64_t)s * (kTile * kTile));
        sum.x += v.x; sum.y += v.y; sum.z += v.z; sum.w += v.w;
    }
    store_result(out, sum, add, rest, act, m, n, N, ex);
}

// How a product is dealt out: `whole` tiles by workgroups of their own (whole rounds of a workgroup a compute unit), the rest by
// `splits` workgroups each; the longest that a compute unit has to do are `steps` steps of a tile.
struct Deal { int tiles_m, tiles, whole, splits, steps; };

Deal deal(int M, int N, int K) {
    Deal d;
    const int units = device_compute_units();
    d.tiles_m = (M + kTile - 1) / kTile;
    d.tiles = d.tiles_m * ((N + kTile - 1) / kTile);
    d.whole = d.tiles / units * units;
    d.splits = 1;
    const int rest = d.tiles - d.whole, steps = K / kStep;
    // us: a step of a tile about 1, 64 KB of partial sums written and read again at about 4 TB/s and a kernel more
    double best = rest ? steps : 0;
    for (int s = 2; rest && s <= 8 && steps / s >= 8; ++s) {
        const int share = (steps + s - 1) / s;
        if ((s - 1) * share >= steps) continue;      // (every split has a step)
        const double cost = (double)((rest * s + units - 1) / units) * share + rest * s * 0.033 + 4;
        if (cost < best) { best = cost; d.splits = s; }
    }
    d.steps = d.tiles / units * steps + (rest * d.splits + units - 1) / units * ((steps + d.splits - 1) / d.splits);
    return d;
}

}  // namespace

// Whether a product of at least 2.5e9 multiply-adds goes here, from what it takes here and in the library (us).  Here: rounds of workgroups, each
// with its beginning and its results; the steps of the unit with the most to do, slower the more units are busy, as power bounds them; the
// partial sums.  The library: 72e6 multiply-adds a us on rows in tiles of 16, and the depth, which few tiles have to go through one after
// the other.  Both are fitted on 130 products with cold weights, 97 to 2,103 rows of 768 x 3,072 to 12,288 x 4,096, the library's best of 32, here
// to 11 % and there to 17 % of every one.  Up to 6 % more is taken for results that are closer to exact ones; with that no size of the
// 130 is taken that is over 7 % slower here (at 2.5e9 and above alone it was 8 to 27 % for 11 of them, where the rows fill a tile
// badly), and none left that is over 5 % faster.  Up to 96 rows the library has a tile of their size.  Rows x features x depth: library, here
// taken: 97 x 2,560 x 10,240 81, 62; 230 x 6,144 x 2,048 50.5, 54.0; 300 x 2,048 x 8,192 93, 80; 701 x 2,048 x 2,048 50.5, 53.5; 701 x 6,144 x
// 2,048 139, 120; 1,100 x 3,072 x 768 46.1, 41.7; 2,103 x 2,048 x 8,192 522, 388
// left: 96 x 2,560 x 10,240 59, 68; 140 x 10,240 x 2,560 73, 93; 290 x 7,680 x 2,560 95, 105; 300 x 6,144 x 2,048 64, 78; 2,048 x 3,072 x 768 72, 79
bool gemm_f32_split_pays(int M, int N, int K) {
    const double products = (double)M * N * K;
    if (M <= 96 || products < 2.5e9) return false;
    const Deal d = deal(M, N, K);
    const int units = device_compute_units(), parts = (d.tiles - d.whole) * d.splits, rounds = d.whole / units + (parts + units - 1) / units;
    const double here = 6.3 + 8.5 * rounds + 0.8 * d.steps + 0.49 * d.tiles * (K / kStep) / units + (d.splits > 1 ? 0.012 * parts : 0.0);
    const double library = 6.2 + 13.8e-9 * products / M * ((M + 15) / 16 * 16) + 0.00225 * K;
    return here < 1.06 * library;
}

// Floats of scratch with which gemm_f32_split deals its tiles out best (0: none).
int64_t gemm_f32_split_scratch(int M, int N, int K) {
    const Deal d = deal(M, N, K);
    return d.splits > 1 ? (int64_t)(d.tiles - d.whole) * d.splits * kTile * kTile : 0;
}

int gemm_f32_split(float* out, const float* x, const float* w, const float* bias, const float* residual, int M, int N, int K, int act,
                   const StGemmExtras& ex, hipStream_t stream) {
    Deal d = deal(M, N, K);
    if (d.splits > 1 && (!ex.scratch || ex.scratch_floats < gemm_f32_split_scratch(M, N, K))) d.splits = 1;
    const int rest = d.tiles - d.whole;
    gemm_f32_split_kernel<<<d.whole + rest * d.splits, 512, 0, stream>>>(out, x, w, bias, residual, ex.scratch, M, N, K, act, d.tiles_m,
                                                                         d.tiles, d.whole, d.splits, ex);
    ST_LAUNCH_CHECK("gemm_f32_split");
    if (d.splits > 1) {
        gemm_f32_sum_kernel<<<dim3(rest, kTile * kTile / 1024), 256, 0, stream>>>(out, ex.scratch, bias, residual, M, N, act, d.tiles_m, d.whole,
                                                                                  d.splits, ex);
        ST_LAUNCH_CHECK("gemm_f32_sum");
    }
    return 0;
}

}  // namespace st
