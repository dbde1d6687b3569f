// The attention of sink_attention.hip (a window that may keep the first tokens, a sink, heads mixed before the softmax, keys and
// values of their own sizes) for prompts and portions in bfloat16, on the matrix cores: tiles of 16 query rows of one item, keys in
// blocks of 32.
//
// A wave has the tile's rows with HW heads that share a key head.  S^T = K Q^T (v_mfma_f32_16x16x32_bf16) leaves a lane with keys
// 16 t + 4 g + e of one row; keys come straight from the pages in the instruction's layout, values through the wave's own LDS, read
// back transposed (ds_read_b64_tr_b16) as the operand of O^T += V^T P^T.  Everything between the two products stays float, as in
// the row kernel: scores, mix, maxima, sums; a weight meets the values as the sum of three bfloat16 numbers, which hold its 24 bits,
// in three products.
//
// A product of whole blocks meets the values of keys that a row does not see with a weight of zero, which an infinity or NaN among
// them would turn into NaN.  A tile whose results are not finite is therefore walked once more, the keys that a row sees one by one
// on the vector units: the row kernel's answer, for such inputs alone.
//
// MIX: the workgroup holds all heads.  Their products with a block lie in LDS as [head][key][row]; a wave takes some of the
// block's keys and mixes them over the heads in place (M is one operand, in registers for the whole walk, a key's products of all
// heads and rows the other: v_mfma_f32_16x16x4_f32), then every wave takes its own heads back.  Two barriers a block.
//
// What bounds it: vector instructions around the products (exponentials, roundings, masks) and, with the mix, its float products
// (heads^2 multiply-adds a row and key) with two barriers a block and one workgroup a unit.  Rows whose tiles leave units idle have
// their keys split over workgroups; the row kernel's merge adds them up.
// Measured beside the row kernel, 32 heads of 64 on 8 key heads, window 1,024: mixed, one prompt of 2,048 rows 736 -> 164 us, 64 single
// tokens of 900 keys beside 448 rows 314 -> 111; not mixed 628 -> 95 and 268 -> 75; 32 heads of 128 x 128, 1,024 rows,
// 510 -> 241 (mixed), 454 -> 190.  The sums' distance from float64 before they are rounded to bfloat16: 512 rows behind 600 keys, mixed
// 3.8e-7 -> 3.3e-7, not mixed 3.0e-7 -> 1.8e-7; with weights of two bfloat16 numbers, some 7 % faster, 1.7e-6 and 2.0e-6.
#include "api.h"
#include "common.h"
#include "chunk_tiles.h"
#include "fragment.h"

#include <type_traits>

namespace st {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef short short4v __attribute__((ext_vector_type(4)));
#define ST_LDS_PTR(T, p) ((__attribute__((address_space(3))) T*)(p))

constexpr int kSinkRows = 16, kSinkKeys = 32;
constexpr int kSinkKeyStride = 20;                                   // floats between a head's keys, and between heads: the four
constexpr int kSinkHeadStride = kSinkKeys * kSinkKeyStride + 16;     // lane groups of an access meet different banks
constexpr int kSinkMaxPages = 2048;

struct SinkTileArgs {
    bf16_t* out;               // [T, heads * value_dim]
    float* part_o;             // [T, splits, heads * value_dim] and
    float* part_ml;            // [T, splits, heads, 2] when splits > 1
    const bf16_t* q; int64_t q_stride;
    const bf16_t* k_cache; int64_t k_page_stride;
    const bf16_t* v_cache; int64_t v_page_stride;
    const float* mix;
    const int* token_item; const int* positions; const int* block_table;
    const int* item_len; const int* item_tok_off; const int* item_slot;
    int num_items, num_tokens, max_pages, page_size, heads, kv_heads, key_dim, value_dim, window, keep_first, sink, splits, table, page_shift;
    float scale;
};

template <int DS, int NV, int HW, int MT>
__global__ __launch_bounds__(MT ? 512 : 256, MT || HW * NV >= 32 ? 1 : 2) void sink_tiles_kernel(SinkTileArgs a) {
    extern __shared__ __attribute__((aligned(16))) char sink_lds[];
    constexpr bool MIX = MT > 0;                                     // heads in tiles of 16, up to 16 MT of them
    constexpr int ROWB = 32 * NV + 16;                               // bytes between a block's values in LDS
    // eight waves have 256 registers a lane: the largest heads' queries and next values are not kept there
    constexpr bool KEEP_Q = !(MIX && HW * DS >= 16), AHEAD_V = !(HW * NV >= 32 && (MIX || DS >= 4));
    const int W = blockDim.x >> 6, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int r16 = lane & 15, g = lane >> 4;
    const int H = a.heads, dk = a.key_dim, dv = a.value_dim, width = H * dv, per = H / a.kv_heads;
    int item, chunk;
    if (!find_chunk(blockIdx.x, a.item_len, a.item_slot, a.num_items, item, chunk, kSinkRows)) {
        // the workgroups past the last tile (one at least) share the rows of no item: zeros, or nothing for the merge to add
        const int spare = gridDim.x - (blockIdx.x - chunk);
        for (int t = blockIdx.z == 0 ? chunk : a.num_tokens; t < a.num_tokens; t += spare) {
            if (a.token_item[t] >= 0) continue;
            if (a.splits == 1)
                for (int e = threadIdx.x; e < width; e += blockDim.x) Elem<bf16_t>::store(a.out + (int64_t)t * width + e, 0.f);
            else
                for (int h = threadIdx.x; h < H; h += blockDim.x) {
                    float* ml = a.part_ml + (((int64_t)t * a.splits + blockIdx.y) * H + h) * 2;
                    ml[0] = -INFINITY;
                    ml[1] = 0.f;
                }
        }
        return;
    }
    const int n = min(kSinkRows, a.item_len[item] - chunk * kSinkRows);
    const int row0 = a.item_tok_off[item] + chunk * kSinkRows, p0 = a.positions[row0];
    const int split = blockIdx.y, h0 = (MIX ? wave : (int)blockIdx.z * W + wave) * HW;
    const bool own = h0 < H;                                         // (a wave past the last head has nothing to do)
    const int kvh = own ? h0 / per : 0;

    // the pages of the tile's keys: those of the first tokens that stay visible, then the window's
    const int lo = a.window > 0 ? max(0, p0 - a.window + 1) : 0, last = p0 + n - 1, ps = a.page_size;
    const int kept = min(a.keep_first, lo), kept_pages = (kept + ps - 1) / ps, first_page = lo / ps;
    int* pages = reinterpret_cast<int*>(sink_lds);
    const int* bt = a.block_table + (int64_t)item * a.max_pages;
    for (int i = threadIdx.x; i < kept_pages + last / ps - first_page + 1; i += blockDim.x)
        pages[i] = max(bt[i < kept_pages ? i : first_page + i - kept_pages], 0);
    float* rs = reinterpret_cast<float*>(sink_lds + a.table);        // [16 MT heads][32][16] products
    char* vs = sink_lds + a.table + MT * 16 * kSinkHeadStride * 4 + wave * (kSinkKeys * ROWB);
    if (MIX)                                                         // heads that do not exist are zeros
        for (int i = H * kSinkHeadStride + threadIdx.x; i < MT * 16 * kSinkHeadStride; i += blockDim.x) rs[i] = 0.f;

    const int kept_blocks = (kept + kSinkKeys - 1) / kSinkKeys, blocks = kept_blocks + (last - lo) / kSinkKeys + 1;
    const int share = (blocks + a.splits - 1) / a.splits, b0 = split * share, b1 = min(blocks, b0 + share);

    // operands that stay: this wave's queries (row r16, channels 32 s + 8 g on), the mix (rows of a tile in the order g + 4 r, so
    // that a result's four lane groups are neighbouring heads)
    bf16x8 qf[KEEP_Q ? HW : 1][DS];
    const bf16_t* qrow = a.q + (int64_t)(row0 + min(r16, n - 1)) * a.q_stride;
    auto load_q = [&](int h, bf16x8* to) {
#pragma unroll
        for (int s = 0; s < DS; ++s) {
            const int d = 32 * s + 8 * g;
            const u32x4 x = *reinterpret_cast<const u32x4*>(qrow + (own ? h0 + h : 0) * dk + min(d, dk - 8));
            to[s] = __builtin_bit_cast(bf16x8, own && d < dk ? x : u32x4{0, 0, 0, 0});
        }
    };
    if (KEEP_Q)
#pragma unroll
        for (int h = 0; h < HW; ++h) load_q(h, qf[KEEP_Q ? h : 0]);
    float mf[MIX ? MT : 1][MIX ? 4 * MT : 1];
    if constexpr (MIX) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int s = 0; s < 4 * MT; ++s) {
                const int to = 16 * t + (r16 >> 2) + 4 * (r16 & 3), from = 4 * s + g;
                const float x = a.mix[min(to, H - 1) * H + min(from, H - 1)];
                mf[t][s] = to < H && from < H ? x : 0.f;
            }
    }
    floatx4 o[HW][NV];
    float m[HW], l[HW];
    const int pos = p0 + r16;
    __syncthreads();                                                 // the pages

    // block b: positions from j0, how many
    auto block_of = [&](int b, int& j0, int& nk) {
        j0 = b < kept_blocks ? b * kSinkKeys : lo + (b - kept_blocks) * kSinkKeys;
        nk = min(kSinkKeys, (b < kept_blocks ? kept : last + 1) - j0);
    };
    auto place = [&](int b, int j, int& page) {
        const int pi = j >> a.page_shift;
        page = pages[b < kept_blocks ? pi : kept_pages + pi - first_page];
        return j & (ps - 1);
    };
    u32x4 kr[2][DS], vr[NV];
    auto load_k = [&](int b) {                                       // (keys past the block's stand for its last one)
        int j0, nk, page;
        block_of(b, j0, nk);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int at = place(b, j0 + min(16 * t + r16, nk - 1), page);
            const bf16_t* p = a.k_cache + (int64_t)page * a.k_page_stride + ((int64_t)kvh * ps + at) * dk;
#pragma unroll
            for (int s = 0; s < DS; ++s) kr[t][s] = *reinterpret_cast<const u32x4*>(p + min(32 * s + 8 * g, dk - 8));
        }
    };
    auto load_v = [&](int b) {
        int j0, nk, page;
        block_of(b, j0, nk);
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int e = lane + 64 * i, key = e / (2 * NV), c = e % (2 * NV);
            const int at = place(b, j0 + min(key, nk - 1), page);
            vr[i] = *reinterpret_cast<const u32x4*>(a.v_cache + (int64_t)page * a.v_page_stride + ((int64_t)kvh * ps + at) * dv + min(8 * c, dv - 8));
        }
    };
    auto store_v = [&]() {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int e = lane + 64 * i, key = e / (2 * NV), c = e % (2 * NV);
            *reinterpret_cast<u32x4*>(vs + key * ROWB + 16 * c) = vr[i];
        }
    };
    auto walk = [&](auto one_by_one) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < HW; ++h) {
            m[h] = a.sink && split == 0 ? 0.f : -INFINITY;
            l[h] = a.sink && split == 0 && g == 0 ? 1.f : 0.f;           // (a lane's own keys; summed over the groups at the end)
#pragma unroll
            for (int v = 0; v < NV; ++v) o[h][v] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
        if (b0 < b1) {
            load_k(b0);
            if (AHEAD_V) load_v(b0);
        }
        for (int b = b0; b < b1; ++b) {
            int j0, nk;
            block_of(b, j0, nk);
            if (AHEAD_V) store_v();
            // a head's products with the block; kept (or, mixed, put into LDS) one head after the other, so that few are in registers
            floatx4 sc[MIX ? 1 : HW][2];
#pragma unroll
            for (int h = 0; h < HW; ++h) {
                if (!KEEP_Q) load_q(h, qf[0]);
                floatx4* x = sc[MIX ? 0 : h];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    x[t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int s = 0; s < DS; ++s) {
                        const u32x4 k = 32 * s + 8 * g < dk ? kr[t][s] : u32x4{0, 0, 0, 0};
                        x[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, k), qf[KEEP_Q ? h : 0][s], x[t], 0, 0, 0);
                    }
                    x[t] *= a.scale;
                    if (MIX && own)
#pragma unroll
                        for (int e = 0; e < 4; ++e) rs[(h0 + h) * kSinkHeadStride + (16 * t + 4 * g + e) * kSinkKeyStride + r16] = x[t][e];
                }
            }
            if (!AHEAD_V) load_v(b);
            if (b + 1 < b1) {
                load_k(b + 1);
                if (AHEAD_V) load_v(b + 1);
            }
            if constexpr (MIX) {
                __syncthreads();
                for (int key = wave; key < kSinkKeys; key += 2 * W) {    // two keys at a time: chains of products side by side
                    const bool second = key + W < kSinkKeys;
                    float* col = rs + key * kSinkKeyStride + r16;
                    float* col2 = rs + (second ? key + W : key) * kSinkKeyStride + r16;
                    float x[4 * MT], y[4 * MT];
#pragma unroll
                    for (int s = 0; s < 4 * MT; ++s) { x[s] = col[(4 * s + g) * kSinkHeadStride]; y[s] = col2[(4 * s + g) * kSinkHeadStride]; }
                    floatx4 acc[MT][2];
#pragma unroll
                    for (int t = 0; t < MT; ++t) acc[t][0] = acc[t][1] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int s = 0; s < 4 * MT; ++s)
#pragma unroll
                        for (int t = 0; t < MT; ++t) {
                            acc[t][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(mf[t][s], x[s], acc[t][0], 0, 0, 0);
                            acc[t][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(mf[t][s], y[s], acc[t][1], 0, 0, 0);
                        }
#pragma unroll
                    for (int t = 0; t < MT; ++t)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            if (H < 16 * MT && 16 * t + g + 4 * r >= H) continue;        // (these stay zeros)
                            col[(16 * t + g + 4 * r) * kSinkHeadStride] = acc[t][0][r];
                            if (second) col2[(16 * t + g + 4 * r) * kSinkHeadStride] = acc[t][1][r];
                        }
                }
                __syncthreads();
            }
            if (!AHEAD_V) store_v();
            // bit 4 t + e: key 16 t + 4 g + e is visible to this row (most blocks: every key to every row)
            uint32_t seen = 0xff;
            const bool whole = nk == kSinkKeys && j0 + nk - 1 <= p0 && (a.window <= 0 || last - j0 < a.window);
            if (!whole) seen = 0;
#pragma unroll
            for (int t = 0; t < 2 && !whole; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int kk = 16 * t + 4 * g + e, j = j0 + kk;
                    if (kk < nk && j <= pos && (a.window <= 0 || pos - j < a.window || j < a.keep_first)) seen |= 1u << (4 * t + e);
                }
            // (the wave's own values: stored above, read here by other lanes of the same wave, whose LDS accesses keep their order)
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
            for (int h = 0; h < HW; ++h) {
                float p[8];
                float top = -INFINITY;
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    p[u] = MIX ? rs[(own ? h0 + h : 0) * kSinkHeadStride + (16 * (u >> 2) + 4 * g + (u & 3)) * kSinkKeyStride + r16]
                               : sc[MIX ? 0 : h][u >> 2][u & 3];
                    if (!whole) p[u] = seen >> u & 1 ? p[u] : -INFINITY;
                    top = fmaxf(top, p[u]);
                }
                top = fmaxf(m[h], rows4_max(top));
                // (rows of which nothing was seen yet: any finite maximum makes their weights zeros)
                const float base = top == -INFINITY ? 0.f : top;
                const bool moved = __any(top != m[h]);
                const float alpha = moved ? exp_le0(m[h] - base) : 1.f;
                m[h] = top;
                uint32_t hb[4], mb[4], lb[4];
                float sum = 0.f;
#pragma unroll
                for (int u = 0; u < 8; u += 2) {
                    const float x = exp_le0(p[u] - base), y = exp_le0(p[u + 1] - base);        // (unseen: e^-inf)
                    sum += x + y;
                    if (one_by_one) { p[u] = x; p[u + 1] = y; }
                    const uint32_t both = pack_bf16x2(x, y);
                    hb[u >> 1] = both;
                    const float dx = x - __uint_as_float(both << 16), dy = y - __uint_as_float(both & 0xffff0000u);
                    const uint32_t rest = pack_bf16x2(dx, dy);
                    mb[u >> 1] = rest;
                    lb[u >> 1] = pack_bf16x2(dx - __uint_as_float(rest << 16), dy - __uint_as_float(rest & 0xffff0000u));
                }
                l[h] = fmaf(l[h], alpha, sum);
                const bf16x8 hi = __builtin_bit_cast(bf16x8, u32x4{hb[0], hb[1], hb[2], hb[3]});
                const bf16x8 mid = __builtin_bit_cast(bf16x8, u32x4{mb[0], mb[1], mb[2], mb[3]});
                const bf16x8 low = __builtin_bit_cast(bf16x8, u32x4{lb[0], lb[1], lb[2], lb[3]});
                if (moved)
#pragma unroll
                    for (int v = 0; v < NV; ++v) o[h][v] *= alpha;
                if constexpr (one_by_one) {
#pragma unroll 1
                    for (int gg = 0; gg < 4; ++gg) {
                        const uint32_t visible = __shfl(seen, r16 + 16 * gg, 64);
#pragma unroll
                        for (int u = 0; u < 8; ++u) {
                            const float w = __shfl(p[u], r16 + 16 * gg, 64);
                            const char* at = vs + (16 * (u >> 2) + 4 * gg + (u & 3)) * ROWB + 8 * g;
                            if (visible >> u & 1)
#pragma unroll
                                for (int v = 0; v < NV; ++v) {
                                    const uint2 x = *reinterpret_cast<const uint2*>(at + 32 * v);
                                    o[h][v][0] = fmaf(w, __uint_as_float(x.x << 16), o[h][v][0]);
                                    o[h][v][1] = fmaf(w, __uint_as_float(x.x & 0xffff0000u), o[h][v][1]);
                                    o[h][v][2] = fmaf(w, __uint_as_float(x.y << 16), o[h][v][2]);
                                    o[h][v][3] = fmaf(w, __uint_as_float(x.y & 0xffff0000u), o[h][v][3]);
                                }
                            __builtin_amdgcn_sched_barrier(0);           // (one key's values in registers at a time)
                        }
                    }
                    continue;
                }
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    if (16 * v >= dv) continue;                          // uniform
                    const char* at = vs + (4 * g + (r16 >> 2)) * ROWB + 32 * v + 8 * (r16 & 3);
                    const uint2 x = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(ST_LDS_PTR(short4v, at)));
                    const uint2 y = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(ST_LDS_PTR(short4v, at + 16 * ROWB)));
                    const bf16x8 v8 = __builtin_bit_cast(bf16x8, u32x4{x.x, x.y, y.x, y.y});
                    o[h][v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v8, low, o[h][v], 0, 0, 0);
                    o[h][v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v8, mid, o[h][v], 0, 0, 0);
                    o[h][v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v8, hi, o[h][v], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0x100);                   // (one head's weights in registers at a time; LDS reads may go ahead)
            }
            __builtin_amdgcn_wave_barrier();
        }
    };
    walk(std::false_type());
    float finite = 0.f;
#pragma unroll
    for (int h = 0; h < HW; ++h)
#pragma unroll
        for (int v = 0; v < NV; ++v)
#pragma unroll
            for (int r = 0; r < 4; ++r) finite = fmaf(o[h][v][r], 0.f, finite);
    // (mixed: every wave walks, or none)
    if (MIX ? __syncthreads_or(!(finite == 0.f)) : __any(!(finite == 0.f))) walk(std::true_type());
    // o[h][v][r]: value channel 16 v + 4 g + r of row r16
    const bool row_ok = r16 < n && own;
    const int64_t row = row0 + r16;
#pragma unroll
    for (int h = 0; h < HW; ++h) {
        const float sum = rows4_sum(l[h]);
        if (!row_ok) continue;
        const float f = a.splits > 1 ? 1.f : sum > 0.f ? 1.f / sum : 0.f;
        const int64_t first = (int64_t)(h0 + h) * dv + 4 * g;
        float* po = a.part_o + (row * a.splits + split) * width + first;
        bf16_t* dst = a.out + row * width + first;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            if (16 * v >= dv) continue;
            const float y[4] = {o[h][v][0] * f, o[h][v][1] * f, o[h][v][2] * f, o[h][v][3] * f};
            if (a.splits > 1) *reinterpret_cast<float4*>(po + 16 * v) = make_float4(y[0], y[1], y[2], y[3]);
            else Elem<bf16_t>::store4(dst + 16 * v, y);
        }
        if (a.splits > 1 && g == 0) {
            float* ml = a.part_ml + ((row * a.splits + split) * H + h0 + h) * 2;
            ml[0] = m[h];
            ml[1] = sum;
        }
    }
}

template <int DS, int NV, int HW, int MT>
static int launch_sink_tiles(const SinkTileArgs& a, int tiles, hipStream_t stream) {
    const int groups = a.heads / HW, waves = MT ? groups : groups < 4 ? groups : 4;
    const int lds = a.table + MT * 16 * kSinkHeadStride * 4 + waves * kSinkKeys * (32 * NV + 16);
    ST_CHECK(hipFuncSetAttribute((const void*)sink_tiles_kernel<DS, NV, HW, MT>, hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess,
             "sink_tiles: cannot raise the LDS limit to %d", lds);
    sink_tiles_kernel<DS, NV, HW, MT><<<dim3(tiles, a.splits, MT ? 1 : (groups + waves - 1) / waves), 64 * waves, lds, stream>>>(a);
    ST_LAUNCH_CHECK("sink_tiles");
    return 0;
}

// heads a wave takes, 0 where these sizes stay with the row kernel
static int sink_tiles_heads(int heads, int kv_heads, int key_dim, int value_dim, int mixed) {
    if (heads <= 0 || kv_heads <= 0 || heads % kv_heads || key_dim % 8 || value_dim % 16 || key_dim > 128 || value_dim > 128) return 0;
    const int hw = heads / kv_heads % 4 == 0 ? 4 : 1;
    if (mixed && (heads > 32 || heads / hw > 8)) return 0;
    return hw;
}

}  // namespace st

using namespace st;

extern "C" int st_sink_tiles_fit(int heads, int kv_heads, int key_dim, int value_dim, int mixed, int window, int keep_first, int max_pages,
                                 int page_size) {
    if (!sink_tiles_heads(heads, kv_heads, key_dim, value_dim, mixed) || page_size <= 0 || (page_size & (page_size - 1))) return 0;
    const int64_t pages = window > 0 ? ((int64_t)window + kSinkRows + page_size - 1) / page_size + 2 + ((int64_t)keep_first + page_size - 1) / page_size
                                     : max_pages;
    return pages <= kSinkMaxPages;
}

extern "C" int st_sink_tiles(void* out, float* part_o, float* part_ml, const void* q, int64_t q_stride, const void* k_cache,
                             int64_t k_page_stride, const void* v_cache, int64_t v_page_stride, const float* mix, const int* token_item,
                             const int* positions, const int* block_table, int max_pages, int page_size, const int* item_len,
                             const int* item_tok_off, const int* item_slot, int num_items, int num_tokens, int heads, int kv_heads,
                             int key_dim, int value_dim, float scale, int window, int keep_first, int sink, int splits, hipStream_t stream) {
    ST_CHECK(num_tokens >= 0 && num_items >= 0 && window >= 0 && keep_first >= 0 && max_pages > 0 && splits >= 1 && splits <= 16,
             "sink_tiles: bad sizes");
    ST_CHECK(st_sink_tiles_fit(heads, kv_heads, key_dim, value_dim, mix != nullptr, window, keep_first, max_pages, page_size),
             "sink_tiles: %d heads of %d / %d on %d key heads stay with the row kernel", heads, key_dim, value_dim, kv_heads);
    if (num_tokens == 0) return 0;
    ST_CHECK(out && q && k_cache && v_cache && token_item && positions && block_table && item_len && item_tok_off && item_slot,
             "sink_tiles: null operand");
    ST_CHECK(splits == 1 || (part_o && part_ml), "sink_tiles: split keys need room for the partial results");
    ST_CHECK(((q_stride | k_page_stride | v_page_stride) & 7) == 0 && (((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)out |
             (uintptr_t)part_o) & 15) == 0, "sink_tiles: rows and pages start on 16 bytes");
    const int64_t pages = window > 0 ? ((int64_t)window + kSinkRows + page_size - 1) / page_size + 2 + ((int64_t)keep_first + page_size - 1) / page_size
                                     : max_pages;
    SinkTileArgs a;
    a.out = (bf16_t*)out; a.part_o = part_o; a.part_ml = part_ml; a.q = (const bf16_t*)q; a.q_stride = q_stride;
    a.k_cache = (const bf16_t*)k_cache; a.k_page_stride = k_page_stride; a.v_cache = (const bf16_t*)v_cache; a.v_page_stride = v_page_stride;
    a.mix = mix; a.token_item = token_item; a.positions = positions; a.block_table = block_table; a.item_len = item_len;
    a.item_tok_off = item_tok_off; a.item_slot = item_slot; a.num_items = num_items; a.num_tokens = num_tokens; a.max_pages = max_pages;
    a.page_size = page_size; a.heads = heads; a.kv_heads = kv_heads; a.key_dim = key_dim; a.value_dim = value_dim; a.window = window;
    a.keep_first = window > 0 ? keep_first : 0; a.sink = sink; a.splits = splits; a.table = (int)((pages * 4 + 15) / 16 * 16); a.scale = scale;
    a.page_shift = __builtin_ctz((unsigned)page_size);
    const int64_t tiles = num_tokens / kSinkRows + num_items + 1;      // (every item's last tile may be a short one; one without a tile)
    ST_CHECK(tiles <= 0x7fffffff, "sink_tiles: too many rows");
    int rc = 0;
#define ST_SINK(DS, NV, HW)                                                                                                    \
    rc = !mix ? launch_sink_tiles<DS, NV, HW, 0>(a, (int)tiles, stream)                                                        \
       : heads > 16 ? launch_sink_tiles<DS, NV, HW, 2>(a, (int)tiles, stream)                                                  \
                    : launch_sink_tiles<DS, NV, HW, 1>(a, (int)tiles, stream)
#define ST_SINK_SIZES(HW)                                                                                                      \
    do {                                                                                                                       \
        if (key_dim <= 64 && value_dim <= 64) ST_SINK(2, 4, HW);                                                               \
        else if (key_dim <= 64) ST_SINK(2, 8, HW);                                                                             \
        else if (value_dim <= 64) ST_SINK(4, 4, HW);                                                                           \
        else ST_SINK(4, 8, HW);                                                                                                \
    } while (0)
    if (sink_tiles_heads(heads, kv_heads, key_dim, value_dim, mix != nullptr) == 4) ST_SINK_SIZES(4);
    else ST_SINK_SIZES(1);
#undef ST_SINK_SIZES
#undef ST_SINK
    if (rc || splits == 1) return rc;
    return st_sink_attention_merge(out, part_o, part_ml, num_tokens, heads, value_dim, splits, kBF16, stream);
}
