// Routed experts: every token sends its vector, scaled by a routing weight, through `top` of
// `experts` small gated feed-forward layers.
//
// Everything stays on the device and has a fixed launch shape, so a step can be recorded:
//   route    per token the `top` best experts and their weights (five rules, see st_moe_route);
//   align    the (token, choice) pairs sorted by expert into tiles of 16, 64 or 128 places, a tile
//            holding pairs of one expert only, an expert's tiles neighbours (places left over are marked -1);
//   up       per tile and 64 inner features: both input products on the matrix cores, rows
//            gathered through the sorted list, then clamp, gate and product of the two halves (experts
//            without a gate: one product and the exact GELU);
//   down     per tile and 64 output features: the output product; with one expert a token the
//            result goes straight into the residual stream, otherwise to a row per pair that
//   combine  sums in the order of the token's choices.  Router outputs past the experts stand for identity
//            experts: a choice of one has no place in the tiles, and its result is the token's own vector.
// A wave computes 16 x 16 blocks of results with operands read straight from memory in the
// matrix instruction's own layout (16 bytes a lane and step): with 16 rows a tile the products
// are bound by the stream of expert weights, which every tile reads once.
#include "api.h"
#include "common.h"
#include "activation.h"
#include "fragment.h"

#include <algorithm>
#include <type_traits>

namespace st {

template <int N> using Steps = std::integral_constant<int, N>;
constexpr int kRows = 16;            // rows of one matrix-instruction block
constexpr int kMaxTop = 16;

struct RouteRule {
    const int* token_item;
    const float* correction;
    float scale;
    int experts, top, mode, groups, keep;
};

// the larger v of a lane and those O apart from it, and the lower index of equal ones
template <int O>
__device__ inline void better_across(float& v, int& i) {
    uint32_t va, vb, ia, ib;
    pair_across<O>(__float_as_uint(v), va, vb);
    pair_across<O>((uint32_t)i, ia, ib);
    const float a = __uint_as_float(va), b = __uint_as_float(vb);
    const bool second = b > a || (b == a && (int)ib < (int)ia);
    v = second ? b : a;
    i = second ? (int)ib : (int)ia;
}
// The largest v of G neighbouring lanes (16, 32 or 64, as across_lanes) and the lowest index that has it; every lane gets both.
// (By moves between the lanes: a choice is one after the other of these, and by way of LDS one of two words takes some 130 clocks.
// With what the rule needs asked for at the start and a wave's two pieces of a router 768 deep at once: router, choice and sorting of one
// token 6.0 -> 5.1 us, of eight 2,048 deep 9.7 -> 9.0, choice and sorting of 33 tokens 5.0 -> 4.2; a pass of fiterax-125m 7,706 -> 7,547.)
template <int G>
__device__ inline void group_best(float& v, int& i) {
    static_assert(G == 16 || G == 32 || G == 64, "whole rows of 16 lanes");
    if constexpr (G > 32) better_across<32>(v, i);
    if constexpr (G > 16) better_across<16>(v, i);
    better_across<8>(v, i);
    better_across<4>(v, i);
    better_across<2>(v, i);
    better_across<1>(v, i);
}

// What a lane needs beside its token's logit, asked for at the kernel's start: behind the choice, or behind the products that make the
// logits, each is a trip to memory of its own.
// (Where a rule has no such number, whatever lies at `any` is read and not used: a load behind a branch is waited for there.)
struct RouteLoads {
    float correction;
    int item;
    template <int G>
    __device__ inline void ask(const RouteRule& r, int token, const void* any) {
        const float* c = r.mode >= 3 ? r.correction + min((int)threadIdx.x & (G - 1), r.experts - 1) : reinterpret_cast<const float*>(any);
        const int* t = r.token_item ? r.token_item + token : reinterpret_cast<const int*>(any);
        correction = *c;
        item = *t;
    }
    __device__ inline bool none(const RouteRule& r) const { return r.token_item && item < 0; }
};

// A token's experts and weights by G lanes, a lane an expert (up to G of them): lane j < top returns choice j.  (A lane an expert
// instead of a thread a token: with the sorting 8
// tokens of 16 experts in groups 11.2 -> 5.8 us, 2,011 tokens 12.8 -> 7.7, 1,000 tokens of 64 experts 45 -> 9.6.)
template <int G>
__device__ inline void route_token(int& id, float& weight, float logit, const RouteLoads& own, const RouteRule& r) {
    constexpr int kNone = 1 << 20;
    const int lane = threadIdx.x & 63, e = lane & (G - 1), first = lane - e;
    const bool in = e < r.experts;
    const float z = in ? logit : -INFINITY;
    const float c = r.mode >= 3 && in ? own.correction : 0.f;
    // modes 2 and 4: shares of the softmax over all experts; mode 3 (and the weights of 0): the sigmoid
    float share = 0.f;
    if (r.mode == 2 || r.mode == 4) {
        const float m = across_lanes<G, true>(z);
        share = in ? expf(z - m) : 0.f;
        share *= 1.f / across_lanes<G, false>(share);
    } else if (r.mode != 1) {
        share = 1.f / (1.f + expf(-z));
    }
    float v = r.mode >= 3 ? share + c : z;             // what an expert is chosen by
    if (!(v == v)) v = -INFINITY;
    bool open = in;
    if (r.mode == 2 && r.keep < r.groups) {
        // a lane a group: its largest logit, then the best groups one after the other
        const int per = r.experts / r.groups;
        float gv = -INFINITY;
        for (int k = 0; k < per; ++k) gv = fmaxf(gv, __shfl(v, first + min(min(e, r.groups - 1) * per + k, r.experts - 1), 64));
        bool free_ = e < r.groups, kept = false;
        for (int k = 0; k < r.keep; ++k) {
            float bv = free_ ? gv : -INFINITY;
            int bi = free_ ? e : kNone;
            group_best<G>(bv, bi);
            if (bi == e) { free_ = false; kept = true; }
        }
        const uint64_t mask = __ballot(kept) >> first;
        open = in && ((mask >> min(e / per, G - 1)) & 1);
    }
    id = -1;
    for (int j = 0; j < r.top; ++j) {
        float bv = open ? v : -INFINITY;
        int bi = open ? e : kNone;
        group_best<G>(bv, bi);
        if (bi == e) open = false;
        if (e == j) id = bi;
    }
    const float s = __shfl(r.mode == 1 ? z : share, first + (id & (G - 1)), 64);
    weight = e < r.top ? s : 0.f;
    const float top_z = r.mode == 1 ? __shfl(s, first, 64) : 0.f;
    if (r.mode == 1 || r.mode == 3) {                  // over the chosen alone
        weight = e < r.top ? (r.mode == 1 ? expf(weight - top_z) : weight) : 0.f;
        const float sum = across_lanes<G, false>(weight);
        weight = r.mode == 1 ? weight / sum : weight / (sum + 1e-20f) * r.scale;
    }
}

template <int G>
__global__ __launch_bounds__(256) void moe_route_lanes_kernel(int* __restrict__ ids, float* __restrict__ weights,
                                                              const float* __restrict__ logits, int logit_stride, int num_tokens, RouteRule r) {
    const int t = (blockIdx.x * 256 + threadIdx.x) / G, e = threadIdx.x & (G - 1), tc = min(t, num_tokens - 1);
    RouteLoads own;
    own.ask<G>(r, tc, logits);
    int id;
    float w;
    route_token<G>(id, w, logits[(int64_t)tc * logit_stride + min(e, r.experts - 1)], own, r);
    if (t >= num_tokens || e >= r.top) return;
    const bool none = own.none(r);
    ids[(int64_t)t * r.top + e] = none ? -1 : id;
    weights[(int64_t)t * r.top + e] = none ? 0.f : w;
}

// Routers of more than 64 outputs: a thread a token.
__global__ __launch_bounds__(256) void moe_route_kernel(
    int* __restrict__ ids, float* __restrict__ weights, const float* __restrict__ logits,
    int logit_stride, const int* __restrict__ token_item, const float* __restrict__ correction, float scale, int num_tokens,
    int experts, int top, int mode, int groups, int keep, int stage) {
    // The rows of the workgroup's tokens go to LDS first, read side by side (a thread that walked its own row in
    // memory would wait for every logit by itself, several times over); rows are experts + 1 floats apart.
    extern __shared__ float s_z[];
    const int t0 = blockIdx.x * blockDim.x, t = t0 + threadIdx.x;
    if (stage) {
        const int n = min((int)blockDim.x, num_tokens - t0);
        const float* src = logits + (int64_t)t0 * logit_stride;
        for (int i = threadIdx.x; i < n * experts; i += blockDim.x) {
            const int r = i / experts;
            // (mode 3 chooses by the sigmoid of a logit plus the expert's correction: formed here, side by side)
            const float z = src[(int64_t)r * logit_stride + (i - r * experts)];
            s_z[r * (experts + 1) + (i - r * experts)] = mode == 3 ? 1.f / (1.f + expf(-z)) + correction[i - r * experts] : z;
        }
        __syncthreads();
    }
    if (t >= num_tokens) return;
    if (token_item && token_item[t] < 0) {
        for (int j = 0; j < top; ++j) { ids[(int64_t)t * top + j] = -1; weights[(int64_t)t * top + j] = 0.f; }
        return;
    }
    const float* z = stage ? s_z + threadIdx.x * (experts + 1) : logits + (int64_t)t * logit_stride;
    // mode 2: only the experts of the `keep` groups (of `groups` equal groups of neighbours) whose largest
    // logit is largest can be chosen; bit g of `open` says that group g is one of them
    uint64_t open = ~0ull;
    const int per = experts / groups;
    if (mode == 2 && keep < groups) {
        open = 0;
        for (int j = 0; j < keep; ++j) {
            int best = -1;
            float bv = 0.f;
            for (int g = 0; g < groups; ++g) {
                if ((open >> g) & 1) continue;
                float gv = z[g * per];
                for (int e = 1; e < per; ++e) gv = fmaxf(gv, z[g * per + e]);
                if (best < 0 || gv > bv) { best = g; bv = gv; }
            }
            open |= 1ull << best;
        }
    }
    // modes 2 and 4: the weights are the chosen experts' shares of the softmax over all experts, as they are
    float m_all = 0.f, inv_sum = 1.f;
    if (mode == 2 || mode == 4) {
        m_all = z[0];
        for (int e = 1; e < experts; ++e) m_all = fmaxf(m_all, z[e]);
        float sum = 0.f;
        for (int e = 0; e < experts; ++e) sum += expf(z[e] - m_all);
        inv_sum = 1.f / sum;
    }
    // mode 4: the share plus the expert's correction chooses; staged, it takes the logit's place in this thread's own row
    if (mode == 4 && stage) {
        float* own = s_z + threadIdx.x * (experts + 1);
        for (int e = 0; e < experts; ++e) own[e] = expf(own[e] - m_all) * inv_sum + correction[e];
    }
    // modes 3 and 4: what an expert is chosen by, where it was not staged
    auto choice = [&](int e) {
        if (stage || mode < 3) return z[e];
        return (mode == 3 ? 1.f / (1.f + expf(-z[e])) : expf(z[e] - m_all) * inv_sum) + correction[e];
    };
    auto weight_of = [&](float v) { return mode == 0 ? 1.f / (1.f + expf(-v)) : mode == 2 ? expf(v - m_all) * inv_sum : v; };
    int chosen[kMaxTop];
    for (int j = 0; j < top; ++j) {
        int best = -1;
        float bv = 0.f;
        for (int e = 0; e < experts; ++e) {
            bool taken = mode == 2 && !((open >> (e / per)) & 1);
            for (int u = 0; u < j; ++u) taken |= chosen[u] == e;
            const float v = choice(e);
            if (!taken && (best < 0 || v > bv)) { best = e; bv = v; }
        }
        chosen[j] = best;
        ids[(int64_t)t * top + j] = best;
        weights[(int64_t)t * top + j] = weight_of(bv);
    }
    if (mode == 1) {
        // softmax over the chosen logits alone; the first chosen is the largest
        float* w = weights + (int64_t)t * top;
        const float m = w[0];
        float sum = 0.f;
        for (int j = 0; j < top; ++j) { w[j] = expf(w[j] - m); sum += w[j]; }
        for (int j = 0; j < top; ++j) w[j] /= sum;
    } else if (mode == 3) {
        // the chosen experts' sigmoids, without the correction, over their sum
        float* w = weights + (int64_t)t * top;
        const float* raw = logits + (int64_t)t * logit_stride;
        float sum = 0.f;
        for (int j = 0; j < top; ++j) {
            w[j] = 1.f / (1.f + expf(-raw[ids[(int64_t)t * top + j]]));
            sum += w[j];
        }
        for (int j = 0; j < top; ++j) w[j] = w[j] / (sum + 1e-20f) * scale;
    } else if (mode == 4) {
        // the shares themselves, without the correction
        const float* raw = logits + (int64_t)t * logit_stride;
        for (int j = 0; j < top; ++j) weights[(int64_t)t * top + j] = expf(raw[ids[(int64_t)t * top + j]] - m_all) * inv_sum;
    }
}

// One workgroup: counts, padded offsets, then places.  Which place of its expert's tiles a pair
// gets depends on the order of the atomics; a pair's result does not depend on its place.
__device__ inline void moe_align(
    int* __restrict__ sorted, int* __restrict__ place_of_pair, int* __restrict__ tile_expert, const int* ids, int num_pairs, int experts,
    int capacity, int kTile, int* count, int* offset) {       // count [experts], offset [experts + 1] in LDS
    const int tid = threadIdx.x;
    for (int e = tid; e < experts; e += 1024) count[e] = 0;
    for (int i = tid; i < capacity; i += 1024) sorted[i] = -1;
    for (int i = tid; i < capacity / kTile; i += 1024) tile_expert[i] = -1;
    __syncthreads();
    for (int p = tid; p < num_pairs; p += 1024) {
        const int e = ids[p];                          // (an identity expert has no tiles)
        if (e >= 0 && e < experts) atomicAdd(&count[e], 1);
    }
    __syncthreads();
    if (tid < 64) {                                    // the first wave: sums of the experts' padded counts, 64 at a time
        int run = 0;
        for (int e0 = 0; e0 < experts; e0 += 64) {
            const int e = e0 + tid, own = e < experts ? (count[e] + kTile - 1) / kTile * kTile : 0;
            const int upto = wave_scan(own);
            if (e < experts) offset[e] = run + upto - own;
            run += __builtin_amdgcn_readlane(upto, 63);
        }
        if (tid == 0) offset[experts] = run;
    }
    __syncthreads();
    for (int e = tid; e < experts; e += 1024) {
        for (int i = offset[e] / kTile; i < offset[e + 1] / kTile; ++i) tile_expert[i] = e;
        count[e] = offset[e];          // from here on: the next free place of the expert
    }
    __syncthreads();
    for (int p = tid; p < num_pairs; p += 1024) {
        const int e = ids[p];
        int place = -1;
        if (e >= 0 && e < experts) {
            place = atomicAdd(&count[e], 1);
            sorted[place] = p;
        }
        place_of_pair[p] = place;
    }
}

__global__ __launch_bounds__(1024) void moe_align_kernel(
    int* __restrict__ sorted, int* __restrict__ place_of_pair, int* __restrict__ tile_expert,
    const int* __restrict__ ids, int num_pairs, int experts, int capacity, int tile) {
    extern __shared__ int lds[];
    moe_align(sorted, place_of_pair, tile_expert, ids, num_pairs, experts, capacity, tile, lds, lds + experts);
}

// Few tokens, all routed at once by one workgroup, which then sorts; the choices between them in LDS.  `experts` of r counts the
// router's outputs, `real` of them have weights.  (64 tokens of 16 experts 7.8 -> 4.5 us; with two turns, 200 tokens, 9.3 us, where
// the two kernels apart take 6 to 7.)
constexpr int kFusedPairs = 1024;
__host__ __device__ inline int route_lanes(int outputs) { return outputs <= 16 ? 16 : outputs <= 32 ? 32 : 64; }
template <int G>
__global__ __launch_bounds__(1024) void moe_route_align_kernel(
    int* __restrict__ ids, float* __restrict__ weights, int* __restrict__ sorted, int* __restrict__ place_of_pair,
    int* __restrict__ tile_expert, const float* __restrict__ logits, int logit_stride, int num_tokens, RouteRule r, int real, int capacity,
    int tile) {
    __shared__ int s_ids[kFusedPairs], s_count[64], s_offset[65];
    const int e = threadIdx.x & (G - 1);
    const int t = threadIdx.x / G, tc = min(t, num_tokens - 1);
    RouteLoads own;
    own.ask<G>(r, tc, logits);
    int id;
    float w;
    route_token<G>(id, w, logits[(int64_t)tc * logit_stride + min(e, r.experts - 1)], own, r);
    if (t < num_tokens && e < r.top) {
        const bool none = own.none(r);
        s_ids[t * r.top + e] = none ? -1 : id;
        ids[t * r.top + e] = none ? -1 : id;
        weights[t * r.top + e] = none ? 0.f : w;
    }
    moe_align(sorted, place_of_pair, tile_expert, s_ids, num_tokens * r.top, real, capacity, tile, s_count, s_offset);
}

// The same behind the router's own product, for the fewest rows: one workgroup forms the logits (each wave a share of the depth, its
// operands straight from memory in the matrix instruction's layout, all on their way at once; the shares meet in LDS), routes and sorts.
// What bounds it: trips to memory, the operands' and then the routing's own chain; a product kernel of its own adds another launch and a
// trip for its logits.  One row of 768, 16 outputs: with the product apart 2.7 and 4.5 us, so 6.2; a step of fiterax-125m 1.1 % shorter.
// RB x CB blocks of 16 rows and 16 outputs.
template <int RB, int CB, int G>
__global__ __launch_bounds__(1024) void moe_router_align_kernel(
    int* __restrict__ ids, float* __restrict__ weights, int* __restrict__ sorted, int* __restrict__ place_of_pair,
    int* __restrict__ tile_expert, const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, const float* __restrict__ bias, int num_tokens,
    int width, int w_rows, RouteRule r, int real, int capacity, int tile) {
    constexpr int D = Frag<bf16_t>::kDepth, WAVES = 16;
    __shared__ __attribute__((aligned(16))) float part[WAVES * RB * CB * 256];
    __shared__ float z[RB * 16 * CB * 16];
    __shared__ int s_ids[kFusedPairs], s_count[64], s_offset[65];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, r16 = lane & 15;
    const int e = tid & (G - 1), t = tid / G, tc = min(t, num_tokens - 1);
    RouteLoads own;
    own.ask<G>(r, tc, w);
    const float* shift_at = bias ? bias + min((tid >> 8) % CB * 16 + (tid & 15), r.experts - 1) : reinterpret_cast<const float*>(w);
    const float shift = *shift_at;
    const bf16_t *xr[RB], *wr[CB];
#pragma unroll
    for (int i = 0; i < RB; ++i) xr[i] = x + (int64_t)min(i * 16 + r16, num_tokens - 1) * width;
#pragma unroll
    for (int i = 0; i < CB; ++i) wr[i] = w + (int64_t)min(i * 16 + r16, w_rows - 1) * width;
    floatx4 acc[RB][CB];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int steps = (width + D - 1) / D, share = (steps + WAVES - 1) / WAVES;
    int k = wave * share * D;
    const int end = min(width, k + share * D);
    auto multiply = [&](const Frag<bf16_t>* a, const Frag<bf16_t>* b) {
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int j = 0; j < CB; ++j) acc[i][j] = Frag<bf16_t>::mma(a[i], b[j], acc[i][j]);
    };
    auto batches = [&](auto count) {
        constexpr int U = decltype(count)::value;
        for (; k + U * D <= end; k += U * D) {
            Frag<bf16_t> a[U][RB], b[U][CB];
#pragma unroll
            for (int u = 0; u < U; ++u) {
#pragma unroll
                for (int j = 0; j < CB; ++j) b[u][j].load_whole(wr[j] + k + u * D + 8 * g);
#pragma unroll
                for (int i = 0; i < RB; ++i) a[u][i].load_whole(xr[i] + k + u * D + 8 * g);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < U; ++u) multiply(a[u], b[u]);
        }
    };
    batches(Steps<4>());
    batches(Steps<2>());                             // (768 deep: two pieces a wave)
    for (; k < end; k += D) {
        Frag<bf16_t> a[RB], b[CB];
#pragma unroll
        for (int j = 0; j < CB; ++j) b[j].load(wr[j], k + 8 * g, width, true, true);
#pragma unroll
        for (int i = 0; i < RB; ++i) a[i].load(xr[i], k + 8 * g, width, true, true);
        multiply(a, b);
    }
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) *reinterpret_cast<floatx4*>(part + ((wave * RB + i) * CB + j) * 256 + lane * 4) = acc[i][j];
    __syncthreads();
    if (tid < RB * CB * 256) {
        const int block = tid >> 8, row = (tid >> 4) & 15, f = tid & 15, n = block % CB * 16 + f;
        const int from = block * 256 + ((row >> 2) * 16 + f) * 4 + (row & 3);
        float sum = 0.f;
#pragma unroll
        for (int q = 0; q < WAVES; ++q) sum += part[q * RB * CB * 256 + from];
        if (bias && n < r.experts) sum += shift;
        z[(block / CB * 16 + row) * (CB * 16) + n] = sum;
    }
    __syncthreads();
    int id;
    float weight;
    route_token<G>(id, weight, z[tc * (CB * 16) + min(e, CB * 16 - 1)], own, r);
    if (t < num_tokens && e < r.top) {
        const bool none = own.none(r);
        s_ids[t * r.top + e] = none ? -1 : id;
        ids[t * r.top + e] = none ? -1 : id;
        weights[t * r.top + e] = none ? 0.f : weight;
    }
    moe_align(sorted, place_of_pair, tile_expert, s_ids, num_tokens * r.top, real, capacity, tile, s_count, s_offset);
}

// ---- few rows an expert: tiles of 16 places, where only the weights' stream counts.  A workgroup takes 16 features; its
// four waves (of a choice) share the depth, so that a wave's part is one or a few batches of loads that are all on their way at once and
// that the waves' rows, which lie a whole row of weights apart, start at different offsets (equal offsets meet in the
// same memory channels); the waves' sums meet in LDS.  The addresses of rows and features that do not exist stand for
// row and feature 0: their results are not stored.
// Workgroups go through a tile's features before the next tile's: the list has a tile for every expert whether it was chosen or not, and
// the workgroups of those that were not, which leave at once, come last instead of between the others.  us, tile by tile within a block of
// features and so: gate and up of 2,048 x 2,048, one token of two experts 17.6 and 8.0, eight tokens of ten 34.7 and 30.9, output product
// 8.8 and 5.0, 17.1 and 16.4; 24 tokens, 4,096 x 4,096, thirteen experts 155 and 151, 77.8 and 74.2; one of 768 x 768 5.9 and 5.3, 4.0 and 3.5.
// (The output product with the rows of all 16 places read, pair or not: 12.3, 23.5, 101 and 4.8.)
// FIRST: pieces of depth a batch.
template <typename T, int MATS, int FIRST = MATS == 1 ? 16 : 8>
__device__ inline void moe_depth_share(floatx4* acc, const T* xr, const T* const* wr, int K, int vec) {
    constexpr int D = Frag<T>::kDepth, L = Frag<T>::kLane;
    const int lane = threadIdx.x & 63, wave = (threadIdx.x >> 6) & 3, g = lane >> 4;
    const int steps = (K + D - 1) / D, share = (steps + 3) / 4;
    int k0 = wave * share * D;
    const int end = min(K, k0 + share * D);
    auto batches = [&](auto count) {
        constexpr int U = decltype(count)::value;
        for (; k0 + U * D <= end; k0 += U * D) {
            Frag<T> a[U], b[MATS][U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int k = k0 + u * D + L * g;
#pragma unroll
                for (int m = 0; m < MATS; ++m) b[m][u].load_whole(wr[m] + k);
                a[u].load_whole(xr + k);
            }
            __builtin_amdgcn_sched_barrier(0);    // (left to itself the compiler keeps a few of the loads on their way)
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int m = 0; m < MATS; ++m) acc[m] = Frag<T>::mma(a[u], b[m][u], acc[m]);
        }
    };
    if (vec) {
        batches(Steps<FIRST>());
        batches(Steps<4>());
    }
    for (; k0 < end; k0 += D) {
        Frag<T> a, b;
        a.load(xr, k0 + L * g, K, true, vec);
#pragma unroll
        for (int m = 0; m < MATS; ++m) {
            b.load(wr[m], k0 + L * g, K, true, vec);
            acc[m] = Frag<T>::mma(a, b, acc[m]);
        }
    }
}

// the waves' blocks of 16 x 16 summed: thread t of the workgroup gets row t / 16, feature t % 16
template <int MATS>
__device__ inline void moe_sum_shares(float* sum, const floatx4* acc, float* lds) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int m = 0; m < MATS; ++m) *reinterpret_cast<floatx4*>(lds + ((wave * MATS + m) * 64 + lane) * 4) = acc[m];
    __syncthreads();
    const int row = threadIdx.x >> 4, from = ((row >> 2) * 16 + (threadIdx.x & 15)) * 4 + (row & 3);
#pragma unroll
    for (int m = 0; m < MATS; ++m) {
        sum[m] = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) sum[m] += lds[(w * MATS + m) * 256 + from];
    }
}

// `blocks` (features by 16) workgroups a tile
template <typename T, bool GATED>
__global__ __launch_bounds__(256) void moe_up_few_kernel(
    T* __restrict__ y, const T* __restrict__ x, const T* __restrict__ w_gate, const T* __restrict__ w_up,
    const int* __restrict__ sorted, const int* __restrict__ tile_expert, const float* __restrict__ weights,
    int blocks, int top, int width, int inner, float limit, int style, int vec) {
    constexpr int MATS = GATED ? 2 : 1;
    __shared__ __attribute__((aligned(16))) float lds[4 * MATS * 256];
    // (the tile's pairs are asked for beside its expert: one trip to memory before the weights', not two)
    const int tile = blockIdx.x / blocks, r16 = threadIdx.x & 15, f0 = (blockIdx.x - tile * blocks) * 16, base = tile * kRows;
    const int e = tile_expert[tile], pair = sorted[base + r16], p = sorted[base + (threadIdx.x >> 4)];
    if (e < 0) return;
    const int64_t feature = (int64_t)e * inner + min(f0 + r16, inner - 1);
    const T* wr[MATS];
    wr[0] = w_up + feature * width;
    if (GATED) wr[MATS - 1] = w_gate + feature * width;
    floatx4 acc[MATS];
#pragma unroll
    for (int m = 0; m < MATS; ++m) acc[m] = floatx4{0.f, 0.f, 0.f, 0.f};
    moe_depth_share<T, MATS>(acc, x + (int64_t)(pair >= 0 ? pair / top : 0) * width, wr, width, vec);
    float sum[MATS];
    moe_sum_shares<MATS>(sum, acc, lds);
    const int place = base + (threadIdx.x >> 4), f = f0 + r16;
    if (f >= inner) return;
    float out = 0.f;
    if (p >= 0 && !GATED) {
        out = apply_activation(kActGeluErf, sum[0]);
    } else if (p >= 0 && style == 1) {
        const float gv = sum[MATS - 1];
        out = gv / (1.f + expf(-gv)) * sum[0];
    } else if (p >= 0) {
        const float s = style == 0 ? weights[p] : 1.f;
        const float gv = fminf(s * sum[MATS - 1], limit);
        const float uv = fminf(fmaxf(s * sum[0], -limit), limit);
        out = gv / (1.f + expf(-1.702f * gv)) * (uv + 1.f);
    }
    Elem<T>::store(y + (int64_t)place * inner + f, out);
}

// `blocks` (features by 16) workgroups a tile
template <typename T>
__global__ __launch_bounds__(256) void moe_down_few_kernel(
    float* out, const float* residual, float* __restrict__ pair_out, const T* __restrict__ y, const T* __restrict__ w_down,
    const int* __restrict__ sorted, const int* __restrict__ tile_expert, int blocks, int top, int width, int inner, float out_scale,
    int vec) {
    __shared__ __attribute__((aligned(16))) float lds[4 * 256];
    const int tile = blockIdx.x / blocks, r16 = threadIdx.x & 15, n0 = (blockIdx.x - tile * blocks) * 16, base = tile * kRows;
    const int e = tile_expert[tile], p = sorted[base + (threadIdx.x >> 4)], pair = sorted[base + r16];
    if (e < 0) return;
    const T* wr[1] = {w_down + ((int64_t)e * width + min(n0 + r16, width - 1)) * inner};
    floatx4 acc[1] = {floatx4{0.f, 0.f, 0.f, 0.f}};
    // (places without a pair stand for the tile's first, which has one: a tile of few pairs reads few rows)
    moe_depth_share<T, 1>(acc, y + (int64_t)(base + (pair >= 0 ? r16 : 0)) * inner, wr, inner, vec);
    float sum[1];
    moe_sum_shares<1>(sum, acc, lds);
    const int place = base + (threadIdx.x >> 4), n = n0 + r16;
    if (n >= width || p < 0) return;
    if (pair_out) {
        pair_out[(int64_t)place * width + n] = sum[0];
    } else {                                           // one expert a token: p is the token
        const int64_t at = (int64_t)p * width + n;
        out[at] = fmaf(out_scale, sum[0], residual[at]);
    }
}

// The output product of one or two tokens with the sum over their choices: four waves a choice, whose sums meet in LDS in the order of the
// choices, so that neither the pairs' results nor a kernel that adds them stand between (the same numbers to the last bit).  Tokens do
// not share an expert's weights, so no more than two.  An instance a number of choices, so that the registers are those of its own threads
// (one of 1,024 threads for all spilled 27 of them: 2,048 x 2,048, 2 choices 23.6 us a call, 20.0 so); four choices, 128 registers a thread, ask
// for 8 pieces of depth at once instead of 16.  grid (ceil(width / 16), tokens), 256 threads a choice.
template <typename T, int TOP>
__global__ __launch_bounds__(256 * TOP) void moe_down_sum_kernel(
    float* out, const float* residual, const T* __restrict__ y, const T* __restrict__ w_down, const int* __restrict__ place_of_pair,
    const float* __restrict__ weights, const int* __restrict__ ids, const T* __restrict__ x, int experts, int width, int inner,
    float out_scale, int vec) {
    constexpr int top = TOP;
    __shared__ float lds[4 * TOP][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r16 = lane & 15, n0 = blockIdx.x * 16;
    const int64_t pair0 = (int64_t)blockIdx.y * top, at = (int64_t)blockIdx.y * width + min(n0 + r16, width - 1);
    const int place = place_of_pair[pair0 + (wave >> 2)], id = ids[pair0 + (wave >> 2)];
    // what the sum needs beside the products (by the lanes of the first wave that form it)
    const float base = residual && wave == 0 ? residual[at] : 0.f, own = x && wave == 0 ? Elem<T>::load(x + at) : 0.f;
    const float weight = weights && wave == 0 && lane < top ? weights[pair0 + lane] : 1.f;
    const int held = wave == 0 && lane < top ? place_of_pair[pair0 + lane] : -1, chosen = wave == 0 && lane < top ? ids[pair0 + lane] : -1;
    if (place >= 0) {
        const T* wr[1] = {w_down + ((int64_t)id * width + min(n0 + r16, width - 1)) * inner};
        floatx4 acc[1] = {floatx4{0.f, 0.f, 0.f, 0.f}};
        moe_depth_share<T, 1, TOP == 4 ? 8 : 16>(acc, y + (int64_t)place * inner, wr, inner, vec);
        if (lane < 16) lds[wave][lane] = acc[0][0];        // (all rows of the block are the pair's)
    }
    __syncthreads();
    if (wave != 0) return;
    float sum = 0.f;
    bool any = false;
    for (int j = 0; j < top; ++j) {
        const float w = __shfl(weight, j, 64);
        const bool here = __shfl(held, j, 64) >= 0, identity = x && __shfl(chosen, j, 64) >= experts;
        float r = 0.f;
        if (here)
#pragma unroll
            for (int q = 0; q < 4; ++q) r += lds[j * 4 + q][r16];
        if (here || identity) {
            sum = fmaf(w, identity ? own : r, sum);
            any = true;
        }
    }
    if (lane < 16 && n0 + lane < width) out[at] = any ? fmaf(out_scale, sum, base) : base;
}

// grid (tiles, ceil(inner / 64)); wave w of the workgroup takes inner features f0 + 16 w .. +15 of
// the tile's RT blocks of 16 rows: a step's weight operands are loaded once and meet RT blocks of
// rows (4 or 8, for prompts, where every tile reads its expert's weights again from the L2).
// Result layout of a block: lane (r16, g) holds rows 4g .. 4g+3 of feature r16.
// GATED false: one weight matrix (w_up) and the exact GELU of its product (style 2).
template <typename T, int RT, bool GATED>
__global__ __launch_bounds__(256) void moe_up_kernel(
    T* __restrict__ y, const T* __restrict__ x, const T* __restrict__ w_gate, const T* __restrict__ w_up,
    const int* __restrict__ sorted, const int* __restrict__ tile_expert, const float* __restrict__ weights,
    int top, int width, int inner, float limit, int style, int vec) {
    const int tile = blockIdx.x;
    const int e = tile_expert[tile];
    if (e < 0) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r16 = lane & 15, g = lane >> 4;
    const int f = blockIdx.y * 64 + wave * 16 + r16;           // this lane's feature as an operand row
    const bool f_ok = f < inner;
    const int base = tile * (kRows * RT);
    const T* xr[RT];
    bool p_ok[RT];
#pragma unroll
    for (int b = 0; b < RT; ++b) {
        const int pair = sorted[base + b * kRows + r16];       // this lane's token row as an operand row
        p_ok[b] = pair >= 0;
        xr[b] = x + (int64_t)(p_ok[b] ? pair / top : 0) * width;
    }
    const T* gr = (GATED ? w_gate : w_up) + ((int64_t)e * inner + (f_ok ? f : 0)) * width;
    const T* ur = w_up + ((int64_t)e * inner + (f_ok ? f : 0)) * width;
    floatx4 cg[RT], cu[RT];
#pragma unroll
    for (int b = 0; b < RT; ++b) { cg[b] = floatx4{0.f, 0.f, 0.f, 0.f}; cu[b] = floatx4{0.f, 0.f, 0.f, 0.f}; }
    constexpr int D = Frag<T>::kDepth, L = Frag<T>::kLane;

    // (the addresses of rows and features that do not exist stand for row and feature 0: their results are not stored)
    int k0 = 0;
    auto batches = [&](auto steps) {
        constexpr int U = decltype(steps)::value;
        for (; k0 + U * D <= width; k0 += U * D) {
            Frag<T> a[U][RT], bg[U], bu[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int k = k0 + u * D + L * g;
                if (GATED) bg[u].load_whole(gr + k);
                bu[u].load_whole(ur + k);
#pragma unroll
                for (int b = 0; b < RT; ++b) a[u][b].load_whole(xr[b] + k);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int b = 0; b < RT; ++b) {
                    if (GATED) cg[b] = Frag<T>::mma(a[u][b], bg[u], cg[b]);
                    cu[b] = Frag<T>::mma(a[u][b], bu[u], cu[b]);
                }
        }
    };
    if constexpr (RT == 4 && sizeof(T) == 4)           // (bfloat16 that allows it goes through LDS, below)
        if (vec) batches(Steps<2>());
    for (; k0 < width; k0 += D) {
        Frag<T> a[RT], bg, bu;
        const int k = k0 + L * g;
        if (GATED) bg.load(gr, k, width, f_ok, vec);
        bu.load(ur, k, width, f_ok, vec);
#pragma unroll
        for (int b = 0; b < RT; ++b) a[b].load(xr[b], k, width, p_ok[b], vec);
#pragma unroll
        for (int b = 0; b < RT; ++b) {
            if (GATED) cg[b] = Frag<T>::mma(a[b], bg, cg[b]);
            cu[b] = Frag<T>::mma(a[b], bu, cu[b]);
        }
    }
    if (!f_ok) return;
#pragma unroll
    for (int b = 0; b < RT; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int place = base + b * kRows + 4 * g + r;
            const int p = sorted[place];
            float out = 0.f;
            if (p >= 0 && !GATED) {
                out = apply_activation(kActGeluErf, cu[b][r]);
            } else if (p >= 0 && style == 1) {
                const float gv = cg[b][r];
                out = gv / (1.f + expf(-gv)) * cu[b][r];
            } else if (p >= 0) {
                const float s = style == 0 ? weights[p] : 1.f;
                const float gv = fminf(s * cg[b][r], limit);
                const float uv = fminf(fmaxf(s * cu[b][r], -limit), limit);
                out = gv / (1.f + expf(-1.702f * gv)) * (uv + 1.f);
            }
            Elem<T>::store(y + (int64_t)place * inner + f, out);
        }
}

// grid (tiles, ceil(width / 64)).
template <typename T, int RT>
__global__ __launch_bounds__(256) void moe_down_kernel(
    float* __restrict__ out, const float* __restrict__ residual, float* __restrict__ pair_out,
    const T* __restrict__ y, const T* __restrict__ w_down, const int* __restrict__ sorted,
    const int* __restrict__ tile_expert, int top, int width, int inner, float out_scale, int vec) {
    const int tile = blockIdx.x;
    const int e = tile_expert[tile];
    if (e < 0) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r16 = lane & 15, g = lane >> 4;
    const int n = blockIdx.y * 64 + wave * 16 + r16;
    const bool n_ok = n < width;
    const int base = tile * (kRows * RT);
    const T* yr = y + (int64_t)(base + r16) * inner;
    const T* wr = w_down + ((int64_t)e * width + (n_ok ? n : 0)) * inner;
    floatx4 c[RT];
#pragma unroll
    for (int b = 0; b < RT; ++b) c[b] = floatx4{0.f, 0.f, 0.f, 0.f};
    constexpr int D = Frag<T>::kDepth, L = Frag<T>::kLane;

    int k0 = 0;
    auto batches = [&](auto steps) {              // (as in moe_up_kernel)
        constexpr int U = decltype(steps)::value;
        for (; k0 + U * D <= inner; k0 += U * D) {
            Frag<T> a[U][RT], bw[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int k = k0 + u * D + L * g;
                bw[u].load_whole(wr + k);
#pragma unroll
                for (int b = 0; b < RT; ++b) a[u][b].load_whole(yr + (int64_t)b * kRows * inner + k);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int b = 0; b < RT; ++b) c[b] = Frag<T>::mma(a[u][b], bw[u], c[b]);
        }
    };
    if constexpr (RT == 4 && sizeof(T) == 4)           // (bfloat16 that allows it goes through LDS, below)
        if (vec) batches(Steps<2>());
    for (; k0 < inner; k0 += D) {
        Frag<T> a[RT], bw;
        const int k = k0 + L * g;
        bw.load(wr, k, inner, n_ok, vec);
#pragma unroll
        for (int b = 0; b < RT; ++b) a[b].load(yr + (int64_t)b * kRows * inner, k, inner, true, vec);
#pragma unroll
        for (int b = 0; b < RT; ++b) c[b] = Frag<T>::mma(a[b], bw, c[b]);
    }
    if (!n_ok) return;
#pragma unroll
    for (int b = 0; b < RT; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int place = base + b * kRows + 4 * g + r;
            const int p = sorted[place];
            if (p < 0) continue;
            if (pair_out) {
                pair_out[(int64_t)place * width + n] = c[b][r];
            } else {                                           // one expert a token: p is the token
                const int64_t at = (int64_t)p * width + n;
                out[at] = fmaf(out_scale, c[b][r], residual[at]);
            }
        }
}

// ---- prompts in bfloat16: tiles of 64 or 128 places, operands by direct loads into LDS -----------
// With some dozens of rows and more an expert a tile of 64 NJ places meets 64 WN rows of its expert's matrix, steps of 64 in depth.
// Both operand tiles go from memory into LDS without passing through registers (16 bytes a lane; a row's chunks are rotated by
// the lane's choice of address, so that the matrix instruction's reads spread over the banks), the AHEAD steps (1 or 2) after the one that is
// multiplied on their way into the other buffers: one barrier a step, before the last quarter of the step's products, whose operands are read
// by then; a wave waits there for its loads of the next step alone, and that step's first operands are read under the quarter that is left.  Each of 2 WN waves multiplies a 64 x 32 NJ part (v_mfma_f32_32x32x16_bf16), the operands of a product of depth 16 read ahead
// of the one before; the two waves that share weight rows take the tile's blocks of 32 places in turn, and a block without a pair
// (an expert's last tile) is not multiplied.
// UP: of every 64 weight rows 32 are inner features of the gate matrix and 32 the same features of the other one, so that a
// lane holds both halves of a result; rows of x are gathered through the sorted list.  GELU: the one input matrix of experts
// without a gate.  Otherwise: output features of the expert's output matrix over the rows of y.
//
// What bounds it: the weights' way from memory, all experts' matrices whatever the rows, and the operands' way from L2 into LDS, which
// a unit takes at some 25 bytes a clock.  So: tiles of 128 places meet 256 weight rows (a quarter fewer bytes for the same products than
// 128 rows, 48 KB a step, one workgroup a unit) unless that leaves units idle (the launch says where), tiles of 64 meet 128 (two workgroups a unit); and a workgroup begins its depth three
// steps after its neighbour does, going round, since rows that lie a power of two apart meet in the same memory channels while everyone
// reads at the same depth.  Workgroups go round the eight dies by their number; here each die takes
// an eighth of the work in the order (expert, weight rows, tile of that expert), so that an expert's matrix passes through one
// die's L2 once, its tiles next to each other, and a die gets the same number of tiles as any other, however the tokens chose.
// Measured on weights that no cache holds, up + down, beside the kernel before it (128 rows, the next step's loads alone on their way,
// all beginning at depth 0): 16 experts of 2,048 x 2,048, two a token, 2,011 tokens 220 -> 204 us, 1,024 tokens 145 -> 128, 753 tokens
// (tiles of 64) 138 -> 127, 128 tokens 106 -> 81; 14 experts of 4,096 x 4,096, 2,048 tokens 663 -> 613, 951 tokens 430 -> 390.  Tiles of
// 64 on 256 rows: 145 us at 753 tokens.  With the meeting before a step's last quarter instead of between two steps: 2,011 tokens
// 219 -> 205 us, 1,024 tokens 129 -> 123; 4,096 x 4,096, 2,048 tokens 656 -> 619, 951 tokens 395 -> 386; tiles of 64 within 2 %.
// (2,011 tokens before: 153 us with the loads taken out, 176 with the products taken out; 205 on matrices stored in the order of the tiles.)
// A workgroup of 256 rows is a unit's only one, so a die's last round may be nearly empty: what its whole rounds of a unit each leave over goes in
// halves (128 rows) where that is up to half of a round, in quarters (and 64 places) up to a quarter; 128 x 128 and 128 x 64 take two thirds and
// half of a whole one's time, the bytes of their operands.  Up and output product, us: 16 experts of 2,048 x 2,048, 2,011 tokens (8 to 16 of 32
// units in the last round) 127 + 80 -> 111 + 61, 1,024 tokens 88 + 44 -> 77 + 45; 8 of 2,048 x 3,072, 2,048 tokens 165 + 105 -> 151 + 81; 14 of
// 4,096 x 4,096 426 + 220 -> 403 + 205.
// Tried and no better: 256 places a tile (at 753 tokens 187 us; as the loop is now 195 to 199 at 2,011, 173 at 753, 413 at 951 of 4,096),
// 128 weight rows on 256 places (220 at 2,011), four waves with 128 weight rows each (206), two buffers for 256 rows (156),
// four and five for 128 rows, workgroups that stay and take the next item while the last one's results are stored (no gain), loads of
// one word a line that bring the weights into L2 two steps earlier (+ 25 %), streaming loads (twice as slow where tiles share weights).
typedef float floatx16 __attribute__((ext_vector_type(16)));
#define ST_LDS_PTR(T, p) ((__attribute__((address_space(3))) T*)(p))
#define ST_GLOBAL_PTR(p) ((const __attribute__((address_space(1))) void*)(p))
// a row's chunk of 8 in depth lies at chunk ^ swizzle(row): 16 neighbouring rows' like chunks lie in different banks
__device__ inline int swizzle(int row) { return (row >> 1) & 7; }

// the tile and the block of weight rows of a workgroup, and which of how many pieces of it; false where there is none left
struct MoeWork { int tile, block, expert, piece, pieces; };
__device__ inline bool moe_work_item(MoeWork& w, const int* __restrict__ tile_expert, int max_tiles, int blocks, int per_die) {
    const int lane = threadIdx.x & 63;
    int tiles = 0;
    for (int b = 0; b < max_tiles; b += 64)
        tiles += __popcll(__ballot(b + lane < max_tiles && tile_expert[min(b + lane, max_tiles - 1)] >= 0));
    const int items = tiles * blocks, share = (items + 7) / 8;       // (the host checks that the numbers fit)
    const int die = blockIdx.x & 7, j = blockIdx.x >> 3, mine = min(share, items - die * share);
    int at = j;
    w.piece = 0;
    w.pieces = 1;
    if (per_die > 0) {                                               // what whole rounds leave over goes in pieces, where those fill no more than a round
        const int whole = mine / per_die * per_die, rest = mine - whole;
        w.pieces = j < whole ? 1 : 4 * rest <= per_die ? 4 : 2 * rest <= per_die ? 2 : 1;
        at = j < whole ? j : whole + (j - whole) / w.pieces;
        w.piece = j < whole ? 0 : (j - whole) % w.pieces;
    }
    if (at >= mine) return false;
    const int i = die * share + at;
    w.expert = tile_expert[i / blocks];                              // (an expert's tiles are neighbours)
    int before = 0, own = 0;
    for (int b = 0; b < max_tiles; b += 64) {
        const int v = tile_expert[min(b + lane, max_tiles - 1)];
        const bool in = b + lane < max_tiles && v >= 0;
        before += __popcll(__ballot(in && v < w.expert));
        own += __popcll(__ballot(in && v == w.expert));
    }
    const int r = i - before * blocks;
    w.block = r / own;
    w.tile = before + (r - w.block * own);
    return true;
}

enum TiledKind : int { kTiledDown = 0, kTiledUp = 1, kTiledGelu = 2 };

struct MoeTiled {
    bf16_t* y_out; float* out; const float* residual; float* pair_out;
    const bf16_t *a_rows, *w0, *w1;
    const int* sorted; const float* weights;
    int top, N, K; float limit, out_scale; int style;
};

// PLACES places from `base` on by 64 RG weight rows from feature n0 on, of expert e, by RG x PG waves: each has 64 rows and NJ blocks of 32 places
// (waves past the places load with the others and multiply nothing).  AHEAD: steps on their way beside the one that is multiplied; DOUBLE:
// sums are carried in double every few steps.
template <int KIND, int RG, int PG, int NJ, int PLACES, int AHEAD, bool DOUBLE>
__device__ __forceinline__ void moe_tile_body(const MoeTiled& arg, uint4* lds, int buf_stride, int base, int n0, int turn, int e) {
    bf16_t* y_out = arg.y_out;
    float *out = arg.out, *pair_out = arg.pair_out;
    const float *residual = arg.residual, *weights = arg.weights;
    const bf16_t *a_rows = arg.a_rows, *w0 = arg.w0, *w1 = arg.w1;
    const int* sorted = arg.sorted;
    const int top = arg.top, N = arg.N, K = arg.K, style = arg.style;
    const float limit = arg.limit, out_scale = arg.out_scale;
    constexpr bool UP = KIND == kTiledUp, GATHER = KIND != kTiledDown;
    constexpr int WAVES = RG * PG, ROWS = 64 * RG;
    constexpr int NW = ROWS / (8 * WAVES), NP = PLACES / (8 * WAVES), NL = NW + NP;      // direct loads a wave and step, eight rows each
    static_assert(NW * 8 * WAVES == ROWS && NP * 8 * WAVES == PLACES, "whole loads");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave % RG, wm = wave / RG, l32 = lane & 31, lh = lane >> 5;
    const bool on = NJ * PG * 32 == PLACES || wm * 32 < PLACES;      // (where there are more waves than blocks, NJ is 1)
    int pair[NJ], full = 0;                        // the pairs of the lane's columns of results; how many of the wave's blocks hold one
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        pair[j] = sorted[base + (on ? (PG * j + wm) * 32 : 0) + l32];
        full += on && __ballot(pair[j] >= 0) != 0;       // (an expert's pairs come first in its tiles)
    }
    // Load t of a wave brings rows 8 (wave + WAVES t) on, a lane 16 bytes of row + lane / 8: piece lane % 8 of the row's place in
    // LDS, which is the chunk that the row's swizzle puts there, the same for all t.  Rows past the matrix stand for row 0 and places
    // without a pair for a row that is there: their results are not stored, or stored as zeros.
    const int chunk = (lane & 7) ^ swizzle(8 * wave + (lane >> 3));
    const bf16_t* src[NL];
#pragma unroll
    for (int t = 0; t < NL; ++t) {
        const int row = 8 * (wave + WAVES * t) + (lane >> 3);
        if (t < NW) {
            const int n = UP ? n0 + (row >> 6) * 32 + (row & 31) : n0 + row;
            const bf16_t* m = UP && ((row >> 5) & 1) ? w1 : w0;
            src[t] = m + ((int64_t)e * N + (n < N ? n : 0)) * K;
        } else {
            const int p = sorted[base + row - ROWS];
            src[t] = a_rows + (GATHER ? (int64_t)(p >= 0 ? p / top : 0) : (int64_t)base + (p >= 0 ? row - ROWS : 0)) * K;
        }
        src[t] += chunk * 8;
    }
    const int whole = K >> 6, steps = (K + 63) >> 6, begin = turn * 3 % steps;
    auto stage = [&](int s, int buf) {
        int k = s + begin;
        if (k >= steps) k -= steps;
        uint4* dst = lds + buf * buf_stride + wave * 64;
        if (k < whole) {
#pragma unroll
            for (int t = 0; t < NL; ++t)
                __builtin_amdgcn_global_load_lds(ST_GLOBAL_PTR(src[t] + k * 64), ST_LDS_PTR(void, dst + t * 64 * WAVES), 16, 0, 0);
        } else {                                   // the last, shorter step: zeros past the depth
            const bool in = k * 64 + chunk * 8 < K;
#pragma unroll
            for (int t = 0; t < NL; ++t) {
                const uint4 v = *reinterpret_cast<const uint4*>(src[t] + (in ? k * 64 : -chunk * 8));
                dst[t * 64 * WAVES + lane] = in ? v : make_uint4(0, 0, 0, 0);
            }
        }
    };
    // (the swizzle of a lane's rows is that of l32: the rows before it are a multiple of 32)
    const uint4* own = lds + l32 * 8;
    const int swz = swizzle(l32);
    floatx16 acc[2][NJ];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[a][j][q] = 0.f;
    double total[DOUBLE ? 2 : 1][DOUBLE ? NJ : 1][16];
    // (a chain's numbers are `per` steps long, so that it has no more roundings than the shares of the tiles of 16 places)
    const int per = max(1, min(4, K >> 9));
    int since = 0;
    if constexpr (DOUBLE)
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int q = 0; q < 16; ++q) total[a][j][q] = 0.0;
    bf16x8 a[2][2], b[2][NJ];
    auto walk = [&](auto blocks32) {                                // over the depth; the wave's blocks of 32 places that hold a pair
        constexpr int B = decltype(blocks32)::value;
        auto fetch = [&](int cur, int kk) {                         // the operands of a product of depth 16
            if constexpr (B > 0) {
                const uint4* at = own + cur * buf_stride + ((kk * 2 + lh) ^ swz);
#pragma unroll
                for (int q = 0; q < 2; ++q) a[kk & 1][q] = __builtin_bit_cast(bf16x8, at[(wn * 64 + q * 32) * 8]);
#pragma unroll
                for (int j = 0; j < B; ++j) b[kk & 1][j] = __builtin_bit_cast(bf16x8, at[(ROWS + (j * PG + wm) * 32) * 8]);
            }
        };
        auto multiply = [&](int kk) {
            __builtin_amdgcn_sched_barrier(0);     // (the next operands are on their way before these are multiplied)
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int j = 0; j < B; ++j)
                    acc[q][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[kk & 1][q], b[kk & 1][j], acc[q][j], 0, 0, 0);
        };
        // This wave's loads of step s have landed, those of the AHEAD - 1 steps after it may be on their way, and its reads of the step
        // before are done; then everyone's are, and that step's buffer may be filled again.
        auto meet = [&](int s) {
            if (s + AHEAD > steps) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((AHEAD - 1) * NL) : "memory");
        };
        stage(0, 0);
        if (AHEAD > 1 && steps > 1) stage(1, 1);
        meet(0);
        fetch(0, 0);
        if (AHEAD < steps) stage(AHEAD, AHEAD);
        for (int s = 0, cur = 0; s < steps; ++s) {
            const int next = cur == AHEAD ? 0 : cur + 1;
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
                if (s + 1 + AHEAD < steps) stage(s + 1 + AHEAD, cur);
            }
            multiply(3);
            cur = next;
            if constexpr (DOUBLE)
                if (++since == per || s + 1 == steps) {
                    since = 0;
#pragma unroll
                    for (int q = 0; q < 2; ++q)
#pragma unroll
                        for (int j = 0; j < NJ; ++j)
#pragma unroll
                            for (int u = 0; u < 16; ++u) {
                                total[q][j][u] += (double)acc[q][j][u];
                                acc[q][j][u] = s + 1 == steps ? (float)total[q][j][u] : 0.f;
                            }
                }
        }
    };
    if (full == NJ) walk(Steps<NJ>());
    else if (NJ > 1 && full > 0) walk(Steps<1>());
    else walk(Steps<0>());
    if (!on) return;
    // acc[q][j][u]: weight row wn * 64 + q * 32 + 8 * (u / 4) + 4 * lh + u % 4, place base + (PG * j + wm) * 32 + l32
    auto store_row = [&](int place, int f, const float* r) {
        bf16_t* dst = y_out + (int64_t)place * N + f;
        if (f + 3 < N && (N & 3) == 0) Elem<bf16_t>::store4(dst, r);
        else
            for (int u = 0; u < 4 && f + u < N; ++u) Elem<bf16_t>::store(dst + u, r[u]);
    };
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int place = base + (j * PG + wm) * 32 + l32;
        const int p = pair[j];
        if (UP) {
            const float scale = p >= 0 && style == 0 ? weights[p] : 1.f;
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                const int f = n0 + wn * 32 + 8 * q4 + 4 * lh;
                if (f >= N) continue;
                float r[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if (style == 1) {
                        const float gv = acc[0][j][4 * q4 + u];
                        r[u] = p >= 0 ? gv / (1.f + expf(-gv)) * acc[1][j][4 * q4 + u] : 0.f;
                        continue;
                    }
                    const float gv = fminf(scale * acc[0][j][4 * q4 + u], limit);
                    const float uv = fminf(fmaxf(scale * acc[1][j][4 * q4 + u], -limit), limit);
                    r[u] = p >= 0 ? gv / (1.f + expf(-1.702f * gv)) * (uv + 1.f) : 0.f;
                }
                store_row(place, f, r);
            }
        } else if (KIND == kTiledGelu) {
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4) {
                    const int f = n0 + wn * 64 + q * 32 + 8 * q4 + 4 * lh;
                    if (f >= N) continue;
                    float r[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) r[u] = p >= 0 ? apply_activation(kActGeluErf, acc[q][j][4 * q4 + u]) : 0.f;
                    store_row(place, f, r);
                }
        } else {
            if (p < 0) continue;
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4) {
                    const int n = n0 + wn * 64 + q * 32 + 8 * q4 + 4 * lh;
                    if (pair_out && (N & 3) == 0 && n + 3 < N) {
                        *reinterpret_cast<float4*>(pair_out + (int64_t)place * N + n) = make_float4(
                            acc[q][j][4 * q4], acc[q][j][4 * q4 + 1], acc[q][j][4 * q4 + 2], acc[q][j][4 * q4 + 3]);
                        continue;
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        if (n + u >= N) continue;
                        const float v = acc[q][j][4 * q4 + u];
                        if (pair_out) pair_out[(int64_t)place * N + n + u] = v;
                        else {
                            const int64_t at = (int64_t)p * N + n + u;       // one expert a token: p is the token
                            out[at] = fmaf(out_scale, v, residual[at]);
                        }
                    }
                }
        }
    }
}

// per_die: compute units of a die, where what whole rounds of them leave over goes in pieces (workgroups of 256 rows by 128 places), else 0
template <int KIND, int WN, int NJ, int AHEAD>
__global__ __launch_bounds__(128 * WN, WN == 2 && (NJ == 1 || AHEAD == 1) ? 2 : 1) void moe_tiled_kernel(
    const MoeTiled arg, const int* __restrict__ tile_expert, int max_tiles, int blocks, int per_die) {
    constexpr int ROWS = 64 * WN, PLACES = 64 * NJ, BUF = (ROWS + PLACES) * 8;           // 16-byte pieces a buffer: weight rows, then places
    __shared__ uint4 lds[(AHEAD + 1) * BUF];
    // Results that stay float, of tiles of 64 places: sums are carried in double every few steps.  With 7 to 31 pairs an expert the tiles of
    // 16 were used before, whose waves share the depth: their chains are an eighth as long (2,048 deep: 2.7e-7 off float64 in one chain,
    // 1.3e-7 in theirs).
    constexpr bool DOUBLE = KIND == kTiledDown && NJ == 1;
    constexpr int FEATURES = KIND == kTiledUp ? ROWS / 2 : ROWS;                         // of a block
    MoeWork w;
    if (!moe_work_item(w, tile_expert, max_tiles, blocks, per_die)) return;
    const int base = w.tile * PLACES, n0 = w.block * FEATURES;
    if constexpr (WN == 4 && NJ == 2) {
        if (w.pieces == 2) {
            moe_tile_body<KIND, 2, 4, 1, 128, AHEAD, DOUBLE>(arg, lds, BUF, base, n0 + w.piece * (FEATURES / 2), w.block, w.expert);
            return;
        }
        if (w.pieces == 4) {
            moe_tile_body<KIND, 2, 4, 1, 64, AHEAD, DOUBLE>(arg, lds, BUF, base + (w.piece >> 1) * 64, n0 + (w.piece & 1) * (FEATURES / 2), w.block, w.expert);
            return;
        }
    }
    moe_tile_body<KIND, WN, 2, NJ, PLACES, AHEAD, DOUBLE>(arg, lds, BUF, base, n0, w.block, w.expert);
}

template <int KIND>
static int launch_tiled(bf16_t* y, float* out, const float* residual, float* pair_out, const void* a_rows, const void* w0,
                        const void* w1, const int* sorted, const int* tile_expert, const float* weights, int capacity, int tile, int top,
                        int N, int K, float limit, float out_scale, int style, hipStream_t stream) {
    const int tiles = capacity / tile;
    const auto launch = [&](auto wn, auto nj, auto ahead) {
        constexpr int WN = decltype(wn)::value, NJ = decltype(nj)::value, AHEAD = decltype(ahead)::value;
        const int features = KIND == kTiledUp ? 32 * WN : 64 * WN, blocks = (N + features - 1) / features;
        ST_CHECK((int64_t)tiles * blocks < (1ll << 30), "moe: too many tiles");
        const int per_die = WN == 4 && NJ == 2 ? device_compute_units() / 8 : 0;
        const unsigned grid = (unsigned)((tiles * blocks + 7) / 8 + per_die) * 8;        // (pieces: up to a round more)
        const MoeTiled arg{y, out, residual, pair_out, (const bf16_t*)a_rows, (const bf16_t*)w0, (const bf16_t*)w1, sorted, weights, top, N, K,
                           limit, out_scale, style};
        moe_tiled_kernel<KIND, WN, NJ, AHEAD><<<grid, 128 * WN, 0, stream>>>(arg, tile_expert, tiles, blocks, per_die);
        return 0;
    };
    int rc;
    if (tile == 64) {
        rc = launch(Steps<2>(), Steps<1>(), Steps<2>());
    } else {
        // Tiles of 128 places meet 256 weight rows where that still fills the chip, else 128.  A list has fewer tiles than places for them
        // (an expert's last tile is counted whole, and one more for each expert): from two thirds on, with 112 pairs an expert and more.
        // Workgroups of 128 rows that are a compute unit's only one bring two steps ahead; where some units may get a second, one (two
        // buffers: two workgroups a unit have room).  Output products, us, with 256 rows, 128 and two steps, 128 and one step (workgroups
        // of 128 rows in the list): 16 experts of 768 x 768, 896 tokens (138) 19.3, 15.4, 16.1; 2,048 tokens (252) 20.1, 16.9, 17.1;
        // 8 of 3,072 x 768, 448 tokens (60) 56.0, 43.6, 50.3; 16 of 1,024 x 1,024, 1,600 tokens (264) 23.4, 34.5, 23.2; 16 of 1,536 x
        // 1,536, 2,048 tokens (444) 36.3, 50.6, 40.4; of 2,048 x 2,048, 896 tokens (384) 44.2, 61.5, 45.7.
        const int features = KIND == kTiledUp ? 64 : 128, units = device_compute_units();
        const int64_t narrow = (int64_t)tiles * ((N + features - 1) / features);
        rc = narrow <= units ? launch(Steps<2>(), Steps<2>(), Steps<2>())
             : 7 * narrow <= 10 * (int64_t)units ? launch(Steps<2>(), Steps<2>(), Steps<1>()) : launch(Steps<4>(), Steps<2>(), Steps<2>());
    }
    if (rc) return rc;
    ST_LAUNCH_CHECK("moe (tiled)");
    return 0;
}

// V columns a thread and turn (4: 16-byte accesses).  x (or null): the tokens' own vectors, the results of the identity
// experts, whose numbers are `experts` and above.
template <typename T, int V>
__global__ __launch_bounds__(1024) void moe_combine_kernel(
    float* out, const float* residual, const float* __restrict__ pair_out,
    const int* __restrict__ place_of_pair, const float* __restrict__ weights, const int* __restrict__ ids,
    const T* __restrict__ x, int experts, int top, int width, float out_scale) {
    const int t = blockIdx.x;
    for (int n = threadIdx.x * V; n < width; n += blockDim.x * V) {
        float sum[V], base[V], own[V];
        bool any = false;
        const int64_t at = (int64_t)t * width + n;
#pragma unroll
        for (int v = 0; v < V; ++v) { sum[v] = 0.f; base[v] = 0.f; own[v] = 0.f; }
        if (residual) {
            if (V == 4) {
                const float4 r = *reinterpret_cast<const float4*>(residual + at);
                base[0] = r.x; base[1 % V] = r.y; base[2 % V] = r.z; base[3 % V] = r.w;
            } else {
                base[0] = residual[at];
            }
        }
        if (x) {
#pragma unroll
            for (int v = 0; v < V; ++v) own[v] = Elem<T>::load(x + at + v);
        }
#pragma unroll 2
        for (int j = 0; j < top; ++j) {
            const int place = place_of_pair[(int64_t)t * top + j];
            const float w = weights ? weights[(int64_t)t * top + j] : 1.f;
            const bool identity = x && ids[(int64_t)t * top + j] >= experts;
            const float* src = pair_out + (int64_t)max(place, 0) * width + n;
            float r[V];
            if (V == 4) {
                const float4 q = *reinterpret_cast<const float4*>(src);
                r[0] = q.x; r[1 % V] = q.y; r[2 % V] = q.z; r[3 % V] = q.w;
            } else {
                r[0] = src[0];
            }
            if (place >= 0 || identity) {
#pragma unroll
                for (int v = 0; v < V; ++v) sum[v] = fmaf(w, identity ? own[v] : r[v], sum[v]);
                any = true;
            }
        }
        if (residual && !any && out == residual) continue;
#pragma unroll
        for (int v = 0; v < V; ++v) sum[v] = any ? fmaf(out_scale, sum[v], base[v]) : base[v];
        if (V == 4) *reinterpret_cast<float4*>(out + at) = make_float4(sum[0], sum[1 % V], sum[2 % V], sum[3 % V]);
        else out[at] = sum[0];
    }
}

}  // namespace st

using namespace st;

static int check_route(const float* correction, int num_tokens, int experts, int top, int mode, int groups, int keep) {
    ST_CHECK(mode >= 0 && mode <= 4, "moe_route: mode 0 (sigmoid of each), 1 (softmax over the chosen), 2 (softmax "
             "over all, the choice within the best groups), 3 (sigmoids over their sum, a corrected choice) or 4 (softmax over "
             "all, a corrected choice)");
    ST_CHECK(mode < 3 || correction, "moe_route: modes 3 and 4 choose by corrected scores");
    ST_CHECK(num_tokens >= 0 && experts > 0, "moe_route: bad sizes");
    ST_CHECK(groups >= 1 && groups <= 64 && experts % groups == 0 && keep >= 1 && keep <= groups,
             "moe_route: %d experts in %d groups of which %d are kept (up to 64 equal groups)", experts, groups, keep);
    ST_CHECK(top <= keep * (experts / groups), "moe_route: %d experts a token do not fit %d groups of %d", top, keep,
             experts / groups);
    ST_CHECK(top >= 1 && top <= kMaxTop && top <= experts, "moe_route: 1 to %d experts a token (of %d), not %d",
             kMaxTop, experts, top);
    return 0;
}

static int check_places(int num_pairs, int experts, int capacity, int tile) {
    ST_CHECK(tile == 16 || tile == 64 || tile == 128, "moe_align: tiles of 16, 64 or 128 places, not %d", tile);
    ST_CHECK(capacity % tile == 0 && capacity >= (num_pairs + tile - 1) / tile * tile + tile * experts,
             "moe_align: %d places do not hold %d pairs of %d experts in tiles of %d", capacity, num_pairs, experts, tile);
    return 0;
}

extern "C" int st_moe_route(int* ids, float* weights, const float* logits, int logit_stride, const int* token_item,
                            const float* correction, float scale, int num_tokens, int experts, int top, int mode, int groups, int keep,
                            hipStream_t stream) {
    if (mode != 2) groups = keep = 1;
    if (const int rc = check_route(correction, num_tokens, experts, top, mode, groups, keep)) return rc;
    ST_CHECK(logits && logit_stride >= experts, "moe_route: null operand or short rows");
    ST_CHECK(ids && weights, "moe_route: null operand");
    if (num_tokens == 0) return 0;
    if (experts <= 64) {
        const RouteRule r{token_item, correction, scale, experts, top, mode, groups, keep};
        const auto launch = [&](auto lanes) {
            constexpr int G = decltype(lanes)::value;
            const int64_t threads = (int64_t)num_tokens * G;
            moe_route_lanes_kernel<G><<<(unsigned)((threads + 255) / 256), 256, 0, stream>>>(ids, weights, logits, logit_stride, num_tokens, r);
        };
        if (experts <= 16) launch(Steps<16>());
        else if (experts <= 32) launch(Steps<32>());
        else launch(Steps<64>());
        ST_LAUNCH_CHECK("moe_route");
        return 0;
    }
    // workgroups of as many tokens as have their rows side by side in 48 KB of LDS (256, 64, or none staged)
    const size_t row = (size_t)(experts + 1) * sizeof(float);
    const int threads = 256 * row <= 48 * 1024 ? 256 : 64;
    const int stage = threads * row <= 48 * 1024;
    moe_route_kernel<<<(num_tokens + threads - 1) / threads, threads, stage ? threads * row : 0, stream>>>(
        ids, weights, logits, logit_stride, token_item, correction, scale, num_tokens, experts, top, mode, groups, keep, stage);
    ST_LAUNCH_CHECK("moe_route");
    return 0;
}

extern "C" int st_moe_route_align(int* ids, float* weights, int* sorted, int* place_of_pair, int* tile_expert, const float* logits,
                                  int logit_stride, const int* token_item, const float* correction, float scale, int num_tokens, int outputs,
                                  int experts, int top, int mode, int groups, int keep, int capacity, int tile, hipStream_t stream) {
    if (mode != 2) groups = keep = 1;
    if (const int rc = check_route(correction, num_tokens, outputs, top, mode, groups, keep)) return rc;
    ST_CHECK(logits && logit_stride >= outputs, "moe_route: null operand or short rows");
    ST_CHECK(outputs <= 64 && experts >= 1 && experts <= outputs, "moe_route_align: up to 64 router outputs, not %d", outputs);
    ST_CHECK((int64_t)num_tokens * route_lanes(outputs) <= 1024, "moe_route_align: up to %d tokens of %d experts", 1024 / route_lanes(outputs), outputs);
    static_assert(kFusedPairs >= 1024 / 16 * kMaxTop, "the choices of all tokens fit LDS");
    if (num_tokens == 0) return st_moe_align(sorted, place_of_pair, tile_expert, ids, 0, experts, capacity, tile, stream);
    if (const int rc = check_places(num_tokens * top, experts, capacity, tile)) return rc;
    ST_CHECK(ids && weights && sorted && place_of_pair && tile_expert, "moe_route_align: null operand");
    const RouteRule r{token_item, correction, scale, outputs, top, mode, groups, keep};
    const auto launch = [&](auto lanes) {
        constexpr int G = decltype(lanes)::value;
        moe_route_align_kernel<G><<<1, 1024, 0, stream>>>(ids, weights, sorted, place_of_pair, tile_expert, logits, logit_stride, num_tokens, r,
                                                          experts, capacity, tile);
    };
    if (outputs <= 16) launch(Steps<16>());
    else if (outputs <= 32) launch(Steps<32>());
    else launch(Steps<64>());
    ST_LAUNCH_CHECK("moe_route_align");
    return 0;
}

// Whether st_moe_router_align takes the product too: up to 32 rows of 16 outputs or 16 of 32, and operands that one workgroup brings in
// little more than a trip to memory (8 rows of 2,048 and 16 outputs, 96 KB: 11.8 us apart, 10.0 so; beyond, product and routing by kernels of
// their own are as fast or faster).
constexpr int64_t kRouterAlignBytes = 128 * 1024;
extern "C" int st_moe_router_align_offered(int num_tokens, int w_rows, int outputs, int width, int dtype) {
    return dtype == kBF16 && num_tokens >= 1 && outputs >= 1 && w_rows >= outputs && width >= 8 && width % 8 == 0 &&
           ((num_tokens <= 32 && outputs <= 16) || (num_tokens <= 16 && outputs <= 32)) &&
           ((int64_t)num_tokens + w_rows) * width * 2 <= kRouterAlignBytes ? 1 : 0;
}

// st_moe_route_align of the logits x [num_tokens, width] . w [w_rows, width]^T (+ bias), in bfloat16.
extern "C" int st_moe_router_align(int* ids, float* weights, int* sorted, int* place_of_pair, int* tile_expert, const void* x, const void* w,
                                   const float* bias, int width, int w_rows, const int* token_item, const float* correction, float scale,
                                   int num_tokens, int outputs, int experts, int top, int mode, int groups, int keep, int capacity, int tile,
                                   hipStream_t stream) {
    if (mode != 2) groups = keep = 1;
    if (const int rc = check_route(correction, num_tokens, outputs, top, mode, groups, keep)) return rc;
    ST_CHECK(st_moe_router_align_offered(num_tokens, w_rows, outputs, width, kBF16), "moe_router_align: not for %d rows of %d and %d outputs",
             num_tokens, width, outputs);
    ST_CHECK(experts >= 1 && experts <= outputs, "moe_router_align: %d experts of %d outputs", experts, outputs);
    if (const int rc = check_places(num_tokens * top, experts, capacity, tile)) return rc;
    ST_CHECK(ids && weights && sorted && place_of_pair && tile_expert && x && w, "moe_router_align: null operand");
    ST_CHECK((((uintptr_t)x | (uintptr_t)w) & 15) == 0, "moe_router_align: rows are 16-byte aligned");
    const RouteRule r{token_item, correction, scale, outputs, top, mode, groups, keep};
#define ST_RA(RB, CB, G)                                                                                              \
    moe_router_align_kernel<RB, CB, G><<<1, 1024, 0, stream>>>(ids, weights, sorted, place_of_pair, tile_expert, (const bf16_t*)x,   \
        (const bf16_t*)w, bias, num_tokens, width, w_rows, r, experts, capacity, tile)
    if (outputs > 16) ST_RA(1, 2, 32);
    else if (num_tokens > 16) ST_RA(2, 1, 16);
    else ST_RA(1, 1, 16);
#undef ST_RA
    ST_LAUNCH_CHECK("moe_router_align");
    return 0;
}

extern "C" int st_moe_align(int* sorted, int* place_of_pair, int* tile_expert, const int* ids, int num_pairs,
                            int experts, int capacity, int tile, hipStream_t stream) {
    ST_CHECK(num_pairs >= 0 && experts > 0 && experts <= 4096, "moe_align: bad sizes (up to 4096 experts)");
    if (const int rc = check_places(num_pairs, experts, capacity, tile)) return rc;
    ST_CHECK(sorted && place_of_pair && tile_expert && ids, "moe_align: null operand");
    moe_align_kernel<<<1, 1024, (2 * experts + 1) * sizeof(int), stream>>>(sorted, place_of_pair, tile_expert, ids,
                                                                          num_pairs, experts, capacity, tile);
    ST_LAUNCH_CHECK("moe_align");
    return 0;
}

static bool rows_vectorised(const void* a, const void* b, const void* c, int depth, int dtype) {
    const int per = dtype == kF32 ? 4 : 8;
    return depth % per == 0 && ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) |
                                 reinterpret_cast<uintptr_t>(c)) & 15) == 0;
}

extern "C" int st_moe_up(void* y, const void* x, const void* w_gate, const void* w_up, const int* sorted,
                         const int* tile_expert, const float* weights, int capacity, int tile, int top, int width,
                         int inner, float limit, int style, int dtype, hipStream_t stream) {
    const int kTile = tile;
    ST_CHECK(style >= 0 && style <= 3, "moe_up: style 0 (weighted, clamped inputs), 1 (plain gated unit), 2 (no gate, GELU) or 3 "
             "(clamped inputs, no weight)");
    if (style == 2) w_gate = w_up;
    ST_CHECK(tile == 16 || tile == 64 || tile == 128, "moe_up: tiles of 16, 64 or 128 places, not %d", tile);
    ST_CHECK(capacity > 0 && capacity % kTile == 0 && top >= 1 && width > 0 && inner > 0, "moe_up: bad sizes");
    ST_CHECK(y && x && w_gate && w_up && sorted && tile_expert && weights, "moe_up: null operand");
    const dim3 grid(capacity / kTile, (inner + 63) / 64);
    ST_CHECK(grid.y <= 65535, "moe_up: too many inner features");
    const int vec = rows_vectorised(x, w_gate, w_up, width, dtype);
    if (dtype == kBF16 && tile >= 64 && vec) {
        if (style == 2)
            return launch_tiled<kTiledGelu>((bf16_t*)y, nullptr, nullptr, nullptr, x, w_up, nullptr, sorted, tile_expert, weights,
                                            capacity, tile, top, inner, width, limit, 1.f, style, stream);
        return launch_tiled<kTiledUp>((bf16_t*)y, nullptr, nullptr, nullptr, x, w_gate, w_up, sorted, tile_expert, weights,
                                      capacity, tile, top, inner, width, limit, 1.f, style, stream);
    }
#define ST_UP_G(T, RT, G)                                                                                    \
    moe_up_kernel<T, RT, G><<<grid, 256, 0, stream>>>((T*)y, (const T*)x, (const T*)w_gate, (const T*)w_up, sorted, \
                                                      tile_expert, weights, top, width, inner, limit, style, vec)
    if (tile == 16) {
        const int blocks = (inner + 15) / 16;
        ST_CHECK((int64_t)(capacity / 16) * blocks < (1ll << 31), "moe_up: too many tiles");
        const unsigned few = (unsigned)(capacity / 16) * blocks;
#define ST_UP_FEW(T, G)                                                                                      \
    moe_up_few_kernel<T, G><<<few, 256, 0, stream>>>((T*)y, (const T*)x, (const T*)w_gate, (const T*)w_up, sorted, tile_expert, \
                                                     weights, blocks, top, width, inner, limit, style, vec)
        if (dtype == kF32) { if (style == 2) ST_UP_FEW(float, false); else ST_UP_FEW(float, true); }
        else if (dtype == kBF16) { if (style == 2) ST_UP_FEW(bf16_t, false); else ST_UP_FEW(bf16_t, true); }
        else ST_CHECK(false, "moe_up: unknown dtype %d", dtype);
#undef ST_UP_FEW
        ST_LAUNCH_CHECK("moe_up (few rows)");
        return 0;
    }
#define ST_UP(T, RT) do { if (style == 2) ST_UP_G(T, RT, false); else ST_UP_G(T, RT, true); } while (0)
    if (dtype == kF32) { if (tile == 64) ST_UP(float, 4); else ST_UP(float, 8); }
    else if (dtype == kBF16) { if (tile == 64) ST_UP(bf16_t, 4); else ST_UP(bf16_t, 8); }
    else ST_CHECK(false, "moe_up: unknown dtype %d", dtype);
#undef ST_UP
#undef ST_UP_G
    ST_LAUNCH_CHECK("moe_up");
    return 0;
}

extern "C" int st_moe_down(float* out, const float* residual, float* pair_out, const void* y, const void* w_down,
                           const int* sorted, const int* tile_expert, int capacity, int tile, int top, int width,
                           int inner, float out_scale, int dtype, hipStream_t stream) {
    const int kTile = tile;
    ST_CHECK(tile == 16 || tile == 64 || tile == 128, "moe_down: tiles of 16, 64 or 128 places, not %d", tile);
    ST_CHECK(capacity > 0 && capacity % kTile == 0 && top >= 1 && width > 0 && inner > 0, "moe_down: bad sizes");
    ST_CHECK(y && w_down && sorted && tile_expert, "moe_down: null operand");
    ST_CHECK(pair_out ? true : (top == 1 && out && residual),
             "moe_down: without a row per pair the result goes to the stream, for one expert a token only");
    const dim3 grid(capacity / kTile, (width + 63) / 64);
    ST_CHECK(grid.y <= 65535, "moe_down: too wide");
    const int vec = rows_vectorised(y, w_down, w_down, inner, dtype);
    if (dtype == kBF16 && tile >= 64 && vec)
        return launch_tiled<kTiledDown>(nullptr, out, residual, pair_out, y, w_down, nullptr, sorted, tile_expert, nullptr, capacity,
                                        tile, top, width, inner, 0.f, out_scale, 0, stream);
    if (tile == 16) {
        const int blocks = (width + 15) / 16;
        ST_CHECK((int64_t)(capacity / 16) * blocks < (1ll << 31), "moe_down: too many tiles");
        const unsigned few = (unsigned)(capacity / 16) * blocks;
#define ST_DOWN_FEW(T)                                                                                       \
    moe_down_few_kernel<T><<<few, 256, 0, stream>>>(out, residual, pair_out, (const T*)y, (const T*)w_down, sorted, tile_expert, \
                                                    blocks, top, width, inner, out_scale, vec)
        if (dtype == kF32) ST_DOWN_FEW(float);
        else if (dtype == kBF16) ST_DOWN_FEW(bf16_t);
        else ST_CHECK(false, "moe_down: unknown dtype %d", dtype);
#undef ST_DOWN_FEW
        ST_LAUNCH_CHECK("moe_down (few rows)");
        return 0;
    }
#define ST_DOWN(T, RT)                                                                                        \
    moe_down_kernel<T, RT><<<grid, 256, 0, stream>>>(out, residual, pair_out, (const T*)y, (const T*)w_down,      \
                                                     sorted, tile_expert, top, width, inner, out_scale, vec)
    if (dtype == kF32) { if (tile == 64) ST_DOWN(float, 4); else ST_DOWN(float, 8); }
    else if (dtype == kBF16) { if (tile == 64) ST_DOWN(bf16_t, 4); else ST_DOWN(bf16_t, 8); }
    else ST_CHECK(false, "moe_down: unknown dtype %d", dtype);
#undef ST_DOWN
    ST_LAUNCH_CHECK("moe_down");
    return 0;
}

// Whether st_moe_down_sum is no slower than st_moe_down and st_moe_combine.  It saves a kernel, 1.5 to 2.5 us, but a workgroup reads all of a
// token's choices where the other has one for each: where `width` has few blocks of 16 features, few compute units then read long rows.
// So the bytes a workgroup reads of each feature are bounded, the more workgroups there are the less.  us a call, two kernels and one:
// one token, bfloat16, 768 x 768 of 2, 3, 4 choices (3, 4.6, 6.1 KB) 14.5 and 13.4, 15.4 and 14.7, 16.5 and 16.1; width 768, inner 2,048 of
// 2, 3, 4 (8, 12, 16 KB) 16.2 and 16.3, 18.2 and 20.3, 20.0 and 23.7; 2,048 x 2,048 of 2, 3, 4 20.7 and 20.0, 28.3 and 27.1, 29.4 and 30.8;
// 1,024, inner 4,096 of 1, 2, 4 (8, 16, 32 KB) 19.0 and 17.4, 22.5 and 24.6, 31.9 and 39.9, in float 28.0 and 25.1, 34.5 and 39.5, 51.4 and 73.6;
// 4,096 x 4,096 of 2 45.7 and 44.3.  Two tokens that share an expert read it twice, which large matrices do not forgive: 2,048 x 2,048 of 2
// 28.6 and 26.2, in float (16 MB) 46.4 and 42.2, 4,096 x 4,096 of 2 46.7 and 54.5.
extern "C" int st_moe_down_sum_offered(int num_tokens, int top, int width, int inner, int dtype) {
    if (num_tokens > 2 || top < 1 || top > 4) return 0;
    const int64_t elem = dtype == kF32 ? 4 : 2, units = device_compute_units();
    const int64_t groups = std::min<int64_t>((int64_t)(width + 15) / 16 * num_tokens, units);
    return (top == 1 || top * inner * elem <= 6144 + 12288 * groups / units) && (num_tokens < 2 || elem * width * inner <= 16 << 20);
}

// st_moe_down (into the pairs' results) and st_moe_combine at once, for the tokens of tiles of 16 places.
extern "C" int st_moe_down_sum(float* out, const float* residual, const void* y, const void* w_down, const int* place_of_pair,
                               const float* weights, const int* ids, const void* x, int experts, int num_tokens, int top, int width, int inner,
                               float out_scale, int dtype, hipStream_t stream) {
    ST_CHECK(num_tokens >= 0 && width > 0 && inner > 0, "moe_down_sum: bad sizes");
    ST_CHECK(num_tokens <= 2 && top >= 1 && top <= 4, "moe_down_sum: one or two tokens of up to four choices, not %d of %d", num_tokens, top);
    ST_CHECK(out && y && w_down && place_of_pair && ids, "moe_down_sum: null operand");
    ST_CHECK(dtype == kF32 || dtype == kBF16, "moe_down_sum: unknown dtype %d", dtype);
    if (num_tokens == 0) return 0;
    const int vec = rows_vectorised(y, w_down, nullptr, inner, dtype);
    const dim3 grid((width + 15) / 16, num_tokens);
#define ST_MDS(T, TOP)                                                                                                    \
    moe_down_sum_kernel<T, TOP><<<grid, 256 * TOP, 0, stream>>>(out, residual, (const T*)y, (const T*)w_down, place_of_pair, weights, ids, \
                                                                (const T*)x, experts, width, inner, out_scale, vec)
#define ST_MDS_T(T) do { if (top == 1) ST_MDS(T, 1); else if (top == 2) ST_MDS(T, 2); else if (top == 3) ST_MDS(T, 3); else ST_MDS(T, 4); } while (0)
    if (dtype == kF32) ST_MDS_T(float); else ST_MDS_T(bf16_t);
#undef ST_MDS_T
#undef ST_MDS
    ST_LAUNCH_CHECK("moe_down_sum");
    return 0;
}

// ids and x (both or neither): a choice of `experts` or above is an identity expert, whose result is the token's row of x
// [tokens, width] in the storage type.
extern "C" int st_moe_combine(float* out, const float* residual, const float* pair_out, const int* place_of_pair,
                              const float* weights, const int* ids, const void* x, int experts, int num_tokens, int top,
                              int width, float out_scale, int dtype, hipStream_t stream) {
    ST_CHECK(num_tokens >= 0 && top >= 1 && width > 0, "moe_combine: bad sizes");
    ST_CHECK(out && pair_out && place_of_pair && (!x || ids), "moe_combine: null operand");
    ST_CHECK(dtype == kF32 || dtype == kBF16, "moe_combine: unknown dtype %d", dtype);
    if (num_tokens == 0) return 0;
    const bool vec = width % 4 == 0 && (((uintptr_t)out | (uintptr_t)residual | (uintptr_t)pair_out) & 15) == 0;
    // a turn is two trips to memory (a choice's place, then its result): few rows have a thread for every piece, up to 1,024 (us, 256 threads
    // and so, alone: 8 rows of 2,048 2.7 and 2.15, 24 of 4,096 4.0 and 2.5, 256 of 2,048 3.0 and 2.5; a call in a step, behind the product that
    // writes the results: 24 of 4,096 10.8 and 7.4, 8 of 2,048 5.0 either way)
    int threads = 256;
    while (num_tokens <= device_compute_units() && threads < 1024 && threads * (vec ? 4 : 1) < width) threads <<= 1;
#define ST_MC(T, V)                                                                                                    \
    moe_combine_kernel<T, V><<<num_tokens, threads, 0, stream>>>(out, residual, pair_out, place_of_pair, weights, ids, (const T*)x, \
                                                             experts, top, width, out_scale)
    if (dtype == kF32) { if (vec) ST_MC(float, 4); else ST_MC(float, 1); }
    else { if (vec) ST_MC(bf16_t, 4); else ST_MC(bf16_t, 1); }
#undef ST_MC
    ST_LAUNCH_CHECK("moe_combine");
    return 0;
}
