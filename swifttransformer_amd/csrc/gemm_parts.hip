// bfloat16 products of some hundred rows with deep matrices, y = x W^T: the depth dealt to several workgroups, whose float
// sums a second kernel adds to the bias and the residual.
//
// What bounds such a product is the way of its operands into a compute unit's LDS, some 40 bytes a nanosecond: a narrow result (the
// hidden size) has fewer tiles than the chip has units, and a unit that walks the whole depth of its tile alone takes four times as long as the
// weights' stream does.  So: tiles of 128 features by all rows (up to 256; a tile of 128, 192 or 256 rows) and as many parts of
// the depth as make a workgroup a unit.  A tile's operands go from memory into LDS directly (16 bytes a lane, rows' chunks rotated
// for the matrix instruction's reads), two steps of 64 in depth ahead of the one that is multiplied; four waves, each with 64 features and
// every other block of 32 rows (v_mfma_f32_32x32x16_bf16).  The parts of a depth are dealt to the dies in their order, so that an eighth of x
// passes through a die's L2 once; a workgroup begins its depth three steps after its neighbour, going round, since rows that lie a power of two
// apart meet in the same memory channels.  Partial sums are stored in the order of the lanes, whole lines an instruction.
// Feed-forward outputs of 150 rows, the library's best and both kernels here, cold weights: 2,048 x 8,192 25.4 -> 18.5 us, 2,560 x 10,240 32.8 ->
// 23.3, 4,096 x 16,384 68.2 -> 39.5 (the weights' stream 27.4); float sums in shares are closer to exact ones too (1.5e-7 for 9.2e-7 of a chain).
#include "common.h"
#include "api.h"
#include "gemm_extras.h"
#include "activation.h"

#include <type_traits>

namespace st {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kFeatures = 128;        // of a tile
constexpr int kStep = 64;             // of depth
constexpr int kMaxRowBlocks = 4;      // of 64 rows, of a tile
constexpr int kAhead = 2;             // steps on their way

#define ST_LDS_PTR(T, p) ((__attribute__((address_space(3))) T*)(p))
#define ST_GLOBAL_PTR(p) ((const __attribute__((address_space(1))) void*)(p))

// a row's chunk of 8 in depth lies at chunk ^ swizzle(row): 16 neighbouring rows' like chunks lie in different banks
__device__ inline int swizzle(int row) { return (row >> 1) & 7; }

template <int N> using Number = std::integral_constant<int, N>;

// NJ: blocks of 64 rows of a tile.  part [splits][tiles][2 NJ 4 of 4 waves][64 lanes][4]; grid: items rounded up to eights.
template <int NJ>
__global__ __launch_bounds__(256, 1) void gemm_parts_kernel(
    float* __restrict__ part, const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, int M, int N, int K, int tiles_n, int tiles, int splits) {
    constexpr int ROWS = 64 * NJ, BUF = (kFeatures + ROWS) * 8;                         // 16-byte pieces of a buffer: features, then rows
    constexpr int NW = kFeatures / 32, NL = NW + ROWS / 32;                             // direct loads a wave and step, eight rows each
    __shared__ uint4 lds[(kAhead + 1) * BUF];
    const int items = tiles * splits, share = (items + 7) / 8, item = (blockIdx.x & 7) * share + (blockIdx.x >> 3);
    if (item >= items) return;
    const int split = item / tiles, tile = item - split * tiles, tm = tile / tiles_n, tn = tile - tm * tiles_n;
    const int n0 = tn * kFeatures, m0 = tm * ROWS;
    const int all = K / kStep, first = (int)((int64_t)split * all / splits), steps = (int)((int64_t)(split + 1) * all / splits) - first;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave & 1, wm = wave >> 1, l32 = lane & 31, lh = lane >> 5;
    // Load t of a wave brings rows 8 (wave + 4 t) on, a lane 16 bytes of row + lane / 8: piece lane % 8 of the row's place in LDS, which is the
    // chunk that the row's swizzle puts there.  Rows past the matrix or past x stand for the last: their sums are not read.
    const int chunk = (lane & 7) ^ swizzle(8 * wave + (lane >> 3));
    const bf16_t* src[NL];
#pragma unroll
    for (int t = 0; t < NL; ++t) {
        const int row = 8 * (wave + 4 * t) + (lane >> 3);
        src[t] = (t < NW ? w + (int64_t)min(n0 + row, N - 1) * K : x + (int64_t)min(m0 + row - kFeatures, M - 1) * K) + first * kStep + chunk * 8;
    }
    const int begin = tn * 3 % steps;
    auto stage = [&](int s, int buf) {
        int k = s + begin;
        if (k >= steps) k -= steps;
        uint4* dst = lds + buf * BUF + wave * 64;
#pragma unroll
        for (int t = 0; t < NL; ++t)
            __builtin_amdgcn_global_load_lds(ST_GLOBAL_PTR(src[t] + k * kStep), ST_LDS_PTR(void, dst + t * 256), 16, 0, 0);
    };
    const uint4* own = lds + l32 * 8;
    const int swz = swizzle(l32);                    // (the rows before a lane's are a multiple of 32)
    floatx16 acc[2][NJ];
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int u = 0; u < 16; ++u) acc[q][j][u] = 0.f;
    bf16x8 a[2][2], b[2][NJ];
    auto walk = [&](auto blocks32) {                 // over the part of the depth; B of the wave's blocks of 32 rows
        constexpr int B = decltype(blocks32)::value;
        auto fetch = [&](int cur, int kk) {          // the operands of a product of depth 16
            const uint4* at = own + cur * BUF + ((kk * 2 + lh) ^ swz);
#pragma unroll
            for (int q = 0; q < 2; ++q) a[kk & 1][q] = __builtin_bit_cast(bf16x8, at[(wn * 64 + q * 32) * 8]);
#pragma unroll
            for (int j = 0; j < B; ++j) b[kk & 1][j] = __builtin_bit_cast(bf16x8, at[(kFeatures + (j * 2 + wm) * 32) * 8]);
        };
        auto multiply = [&](int kk) {
            __builtin_amdgcn_sched_barrier(0);       // (the next operands are on their way before these are multiplied)
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int j = 0; j < B; ++j)
                    acc[q][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[kk & 1][q], b[kk & 1][j], acc[q][j], 0, 0, 0);
        };
        // This wave's loads of step s have landed, those of the step after it may be on their way, and its reads of the step before are
        // done; then everyone's are, and that step's buffer may be filled again.
        auto meet = [&](int s) {
            if (s + kAhead > steps) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((kAhead - 1) * NL) : "memory");
        };
        stage(0, 0);
        if (steps > 1) stage(1, 1);
        meet(0);
        fetch(0, 0);
        if (kAhead < steps) stage(kAhead, kAhead);
        for (int s = 0, cur = 0; s < steps; ++s) {
            const int next = cur == kAhead ? 0 : cur + 1;
#pragma unroll
            for (int kk = 0; kk < 3; ++kk) {
                fetch(cur, kk + 1);
                multiply(kk);
            }
            // the waves meet before the step's last products, whose operands are in registers: those cover the way to the next step's first
            if (s + 1 < steps) {
                __builtin_amdgcn_sched_barrier(0);
                meet(s + 1);
                fetch(next, 0);
                if (s + 1 + kAhead < steps) stage(s + 1 + kAhead, cur);
            }
            multiply(3);
            cur = next;
        }
    };
    // (a tile has more than 64 (NJ - 1) rows, but where several make up the rows the last may have fewer: it multiplies what it need not)
    if (m0 + (2 * (NJ - 1) + wm) * 32 < M) walk(Number<NJ>());
    else walk(Number<NJ - 1>());
    float* dst = part + ((int64_t)split * tiles + tile) * (kFeatures * ROWS) + wave * (32 * NJ * 64) + lane * 4;
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int u4 = 0; u4 < 4; ++u4)
                *reinterpret_cast<float4*>(dst + ((q * NJ + j) * 4 + u4) * 256) =
                    make_float4(acc[q][j][4 * u4], acc[q][j][4 * u4 + 1], acc[q][j][4 * u4 + 2], acc[q][j][4 * u4 + 3]);
}

// The parts' sums: a thread four features of a row, the lanes as above; grid (tiles, 8 NJ: wave and its blocks), a block of 256 threads has a
// block of 32 x 32.  Eight parts are asked for at once; sums in their order.
template <bool OUT_F32>
__global__ __launch_bounds__(256) void gemm_parts_sum_kernel(
    void* __restrict__ out, const float* __restrict__ part, const float* bias, const float* residual, int M, int N, int act, float out_scale,
    int bias_unscaled, int nj, int tiles_n, int tiles, int splits) {
    const int tile = blockIdx.x, block = blockIdx.y, lane = threadIdx.x & 63, u4 = threadIdx.x >> 6;
    const int wave = block / (2 * nj), q = block / nj & 1, j = block % nj, wn = wave & 1, wm = wave >> 1;
    const int tm = tile / tiles_n, tn = tile - tm * tiles_n;
    const int mb = (tm * 2 * nj + 2 * j + wm) * 32, m = mb + (lane & 31), n = tn * kFeatures + wn * 64 + q * 32 + 8 * u4 + 4 * (lane >> 5);
    if (mb >= M) return;
    const int mc = min(m, M - 1), nc = min(n, N - 4);
    const int64_t plane = (int64_t)tiles * (kFeatures * 64 * nj);
    const float* from = part + (int64_t)tile * (kFeatures * 64 * nj) + (block * 4 + u4) * 256 + lane * 4;
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
    const floatx4 add = bias ? *reinterpret_cast<const floatx4*>(bias + nc) : zero;
    const floatx4 rest = residual ? *reinterpret_cast<const floatx4*>(residual + (int64_t)mc * N + nc) : zero;
    floatx4 sum = zero;
    for (int p0 = 0; p0 < splits; p0 += 8) {
        floatx4 v[8];
#pragma unroll
        for (int p = 0; p < 8; ++p) v[p] = *reinterpret_cast<const floatx4*>(from + min(p0 + p, splits - 1) * plane);
#pragma unroll
        for (int p = 0; p < 8; ++p) sum += p0 + p < splits ? v[p] : zero;
    }
    if (m >= M || n >= N) return;
    if (bias && !bias_unscaled) sum += add;
    if (act != kActNone)
        sum = floatx4{apply_activation(act, sum[0]), apply_activation(act, sum[1]), apply_activation(act, sum[2]), apply_activation(act, sum[3])};
    if (out_scale != 0.f) sum *= out_scale;
    if (bias && bias_unscaled) sum += add;
    if (residual) sum += rest;
    if constexpr (OUT_F32) {
        *reinterpret_cast<floatx4*>((float*)out + (int64_t)m * N + n) = sum;
    } else {
        const float s[4] = {sum[0], sum[1], sum[2], sum[3]};
        Elem<bf16_t>::store4((bf16_t*)out + (int64_t)m * N + n, s);
    }
}

// How a product is dealt out: tiles of 64 nj rows (nj of 2 to 4), the depth in `splits` parts, no more workgroups than compute units (a second one on some
// takes as long as on all), and what that takes (us, to some 10 % of 700 measured): launches, beginnings and ends, the steps of a
// workgroup or the weights' stream, the partial sums there and back.
struct Deal { int nj, tiles_n, tiles, splits; double us; };

Deal deal(int M, int N, int K) {
    Deal d{};
    const int units = device_compute_units(), blocks = (M + 63) / 64, tiles_m = (blocks + kMaxRowBlocks - 1) / kMaxRowBlocks, all = K / kStep;
    d.nj = blocks == 1 ? 2 : (blocks + tiles_m - 1) / tiles_m;       // (64 rows and fewer come by demand alone: half of a tile of 128)
    d.tiles_n = (N + kFeatures - 1) / kFeatures;
    d.tiles = d.tiles_n * ((M + 64 * d.nj - 1) / (64 * d.nj));
    const double step = (kFeatures + 64 * d.nj) * 128 / 56e3, stream = (double)N * K * 2 / 5.2e6, sums = (double)d.tiles * 64 * d.nj * kFeatures * 8 / 7e6;
    d.us = 1e30;
    for (int s = 2; s <= 32 && s <= all && (int64_t)d.tiles * s <= units; ++s) {
        const double walk = (all + s - 1) / s * step, us = 6.2 + (walk > stream ? walk : stream) + s * sums;
        if (us < d.us) { d.us = us; d.splits = s; }
    }
    return d;
}

}  // namespace

// What gemm_parts takes: up to 1,024 rows, whole steps of depth, features by fours, tiles that leave units for parts.
bool gemm_parts_can(int M, int N, int K) {
    return M >= 1 && M <= 64 * kMaxRowBlocks * 4 && K % kStep == 0 && K >= 2 * kStep && N % 4 == 0 && deal(M, N, K).splits > 1;
}

// Whether a product of 65 to 768 rows goes here: where what it takes is less than a part of the estimate for the library's best of 32, that of the
// weights' stream, of the products on rows in tiles of 16, of the depth that few tiles walk one after the other, and of rows times depth
// and features.  Both estimates are some tenths low, and by what depends on the sizes, so the part does too; it was set by 812 products timed
// beside the library's, 66 to 768 rows of 256 x 16,384 to 8,192 x 8,192 (cold weights; library and here, us).  394 go here, in 0.73 of the library's time; five of them
// in more, 256 x 256 x 16,384 in 1.14, the others in up to 1.05.
// Tiles of up to 192 rows: 0.95 up to 512 rows (100 x 2,048 x 8,192 19.2, 15.8; 150 25.4, 18.5; 150 x 4,096 x 4,096 21.2, 19.0; 100 x 4,096 x 16,384
// 49.2, 33.3; 150 x 2,560 x 10,240 32.8, 23.3; 100 x 16,384 x 4,096 40.2, 33.6; left: 150 x 2,048 x 2,048 11.9, 13.0; 150 x 6,144 x 2,048 15.0, 17.7;
// 100 x 768 x 3,072 6.9, 9.7) and all of it up to 576, where the library's time is a tenth above the estimate (of 105 products 0.78 of its time, at
// worst 1.04: 520 x 2,048 x 8,192 44.6, 33.8; 575 x 4,096 x 16,384 130.6, 117.0, of which a step of 575 rows keeps 4; 576 x 5,120 x 13,824 119.8, 119.4; 530 x 3,072 x 5,632 36.5, 37.9).
// Tiles of 256 rows take longer than estimated where there are two or three to a column: 0.84 (taken: 512 x 2,048 x 8,192 38.0, 33.7; 512 x 4,096 x 16,384
// 110.3, 90.2; left: 512 x 7,168 x 7,168 75.3, 86.7; 512 x 8,192 x 8,192 87.8, 103.4; 512 x 5,120 x 5,120 50.7, 53.6) and 0.82 (taken: 640 x 2,048 x
// 16,384 84.0, 62.8; left: 704 x 4,096 x 8,192 69.1, 84.6; 768 x 5,120 x 13,824 124.6, 138.2).
// Of narrow results the library deals out the depth too, which its estimate does not know: 0.82 below 1,024 features (taken: 192 x 768 x 12,288 28.5,
// 18.3; 704 x 768 x 8,192 34.9, 24.8; left: 150 x 768 x 8,192 14.6, 17.3; 192 x 640 x 8,192 14.7, 17.3), 0.7 up to 512 (taken: 320 x 512 x 12,288 28.1,
// 20.2; left: 256 x 512 x 8,192 13.1, 18.1; 480 17.4, 19.3).
// Left by their sizes: 64 rows and fewer, for which the library has tiles of their size (64 x 2,048 x 8,192 16.2, 13.0 alone, but 15.7, 16.4 in a step
// of 64 requests); more than 768 (900 x 2,048 x 8,192 47.2, 49.0); and more than 512 of a depth below 5,504, the least that was timed when that line was
// drawn (575 x 5,120 x 5,120 51.9, 55.4; 576 x 1,024 x 4,096 18.3, 21.9; but 560 x 2,048 x 5,120 31.7, 26.6; 575 x 2,560 x 5,312 40.0, 30.6).
bool gemm_parts_pays(int M, int N, int K) {
    if (M <= 64 || M > 768 || (M > 512 && K < 5504) || !gemm_parts_can(M, N, K)) return false;
    const Deal d = deal(M, N, K);
    const double rows = (M + 15) / 16 * 16;
    const double library = 3.3 + 0.78 * N * K * 2e-6 / 5 + 0.69 * 2e-9 * rows * N * K / 1.2 + 0.00058 * K + 0.305e-5 * rows * K +
                           0.31e-5 * (rows * N < 1e6 ? rows * N : 1e6);
    double part = d.nj < kMaxRowBlocks ? (M <= 512 ? 0.95 : 1.0) : M <= 256 ? 0.95 : M <= 512 ? 0.84 : 0.82;
    if (N < 1024 && part > 0.82) part = 0.82;
    if (N <= 512 && part > 0.7) part = 0.7;
    return d.us < part * library;
}

// Floats of scratch that it takes.
int64_t gemm_parts_scratch(int M, int N, int K) {
    const Deal d = deal(M, N, K);
    return (int64_t)d.tiles * d.splits * kFeatures * 64 * d.nj;
}

int gemm_parts(void* out, const bf16_t* x, const bf16_t* w, const float* bias, const float* residual, int M, int N, int K, int act, int out_f32,
               const StGemmExtras& ex, hipStream_t stream) {
    const Deal d = deal(M, N, K);
    ST_CHECK(gemm_parts_can(M, N, K) && ex.scratch && ex.scratch_floats >= gemm_parts_scratch(M, N, K),
             "gemm: the kernel of parted depths does not take M=%d N=%d K=%d", M, N, K);
    const unsigned grid = (unsigned)((d.tiles * d.splits + 7) / 8 * 8);
#define ST_PARTS(NJ) gemm_parts_kernel<NJ><<<grid, 256, 0, stream>>>(ex.scratch, x, w, M, N, K, d.tiles_n, d.tiles, d.splits)
    switch (d.nj) {
        case 2: ST_PARTS(2); break;
        case 3: ST_PARTS(3); break;
        default: ST_PARTS(4); break;
    }
#undef ST_PARTS
    ST_LAUNCH_CHECK("gemm_parts");
    const dim3 sums((unsigned)d.tiles, (unsigned)(8 * d.nj));
    if (out_f32) gemm_parts_sum_kernel<true><<<sums, 256, 0, stream>>>(out, ex.scratch, bias, residual, M, N, act, ex.out_scale, ex.bias_unscaled, d.nj,
                                                                       d.tiles_n, d.tiles, d.splits);
    else gemm_parts_sum_kernel<false><<<sums, 256, 0, stream>>>(out, ex.scratch, bias, residual, M, N, act, ex.out_scale, ex.bias_unscaled, d.nj,
                                                                d.tiles_n, d.tiles, d.splits);
    ST_LAUNCH_CHECK("gemm_parts_sum");
    return 0;
}

}  // namespace st
