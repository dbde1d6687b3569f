// A short causal convolution over time with one filter a channel, for batches of portions of
// sequences: what lies before a portion's first row comes from the request's state slot, which
// holds the inputs at the last taps - 1 positions.
//
//   y[t, c] = act((x[t, c] if add_input) + bias[c] + sum_{j < taps} w[c, j] * x(position p_t - (taps - 1) + j, c))
//
// The input rows are float or in the storage type, with any row stride (a slice of a product's
// output); the state is float with any stride between slots (a part of a larger state of the
// request).  A row depends on earlier rows of the same launch only through x, which the kernel
// does not write; the state is moved on by a second kernel after all rows have read it.  Sums are float.
#include "api.h"
#include "common.h"
#include "activation.h"

namespace st {

constexpr int kMaxTaps = 8;

template <typename TI, typename TO>
__global__ __launch_bounds__(256) void token_conv_kernel(
    TO* __restrict__ out, const TI* __restrict__ x, int64_t x_stride, const float* __restrict__ w,
    const float* __restrict__ bias, const float* __restrict__ state, int64_t slot_stride,
    const int* __restrict__ token_item, const int* __restrict__ item_tok_off, const int* __restrict__ item_slot,
    int channels, int taps, int add_input, int activation) {
    const int t = blockIdx.x;
    const int c = blockIdx.y * 256 + threadIdx.x;
    if (c >= channels) return;
    const int item = token_item[t];
    const int slot = item >= 0 ? item_slot[item] : -1;
    if (slot < 0) {                                  // a padding row of a batch of fixed size
        Elem<TO>::store(out + (int64_t)t * channels + c, 0.f);
        return;
    }
    const int r = t - item_tok_off[item];            // row within the item's portion
    const int hist = taps - 1;
    const float* st_c = state + (int64_t)slot * slot_stride + c;
    const TI* x_c = x + (int64_t)t * x_stride + c;
    float acc = add_input ? Elem<TI>::load(x_c) : 0.f;
    if (bias) acc += bias[c];
    for (int j = 0; j < taps; ++j) {
        const int back = hist - j;                   // rows back from this one
        const float v = (r - back >= 0) ? Elem<TI>::load(x_c - (int64_t)back * x_stride)
                                        : st_c[(int64_t)(hist + r - back) * channels];
        acc = fmaf(w[(int64_t)c * taps + j], v, acc);
    }
    Elem<TO>::store(out + (int64_t)t * channels + c, apply_activation(activation, acc));
}

// Four channels and ROWS rows a thread, TAPS known: the input rows that the thread's rows share are read once, in whole 8- or 16-byte pieces, and the
// filters once for all rows.  What bounds it: reading the rows and writing the results.  2,011 rows of 2,048 channels, 4 taps, float to
// bfloat16: 24.1 us by element and row, 11.9 so; bfloat16 to float, 2,560 channels with SiLU 37.8 and 13.6.  Sums in the same order as above.
template <typename T> __device__ inline void load4(const T* p, float* v);
template <> __device__ inline void load4<float>(const float* p, float* v) { Elem<float>::load_vec(p, v); }
template <> __device__ inline void load4<bf16_t>(const bf16_t* p, float* v) {
    const uint2 q = *reinterpret_cast<const uint2*>(p);
    v[0] = __uint_as_float(q.x << 16); v[1] = __uint_as_float(q.x & 0xffff0000u);
    v[2] = __uint_as_float(q.y << 16); v[3] = __uint_as_float(q.y & 0xffff0000u);
}

template <typename TI, typename TO, int TAPS, int ROWS>
__global__ __launch_bounds__(256) void token_conv_rows_kernel(
    TO* __restrict__ out, const TI* __restrict__ x, int64_t x_stride, const float* __restrict__ w,
    const float* __restrict__ bias, const float* __restrict__ state, int64_t slot_stride,
    const int* __restrict__ token_item, const int* __restrict__ item_tok_off, const int* __restrict__ item_slot,
    int num_tokens, int channels, int add_input, int activation) {
    constexpr int HIST = TAPS - 1;
    const int t0 = blockIdx.x * ROWS, c = (blockIdx.y * 256 + threadIdx.x) * 4;
    if (c >= channels) return;
    float rows[ROWS + HIST][4], f[4 * TAPS], b[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < ROWS + HIST; ++k)            // rows t0 - HIST on (some of another item: not used)
        load4<TI>(x + (int64_t)min(max(t0 - HIST + k, 0), num_tokens - 1) * x_stride + c, rows[k]);
#pragma unroll
    for (int j = 0; j < TAPS; ++j) Elem<float>::load_vec(w + (int64_t)c * TAPS + 4 * j, f + 4 * j);
    if (bias) Elem<float>::load_vec(bias + c, b);
    int item[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) item[r] = token_item[min(t0 + r, num_tokens - 1)];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        const int t = t0 + r;
        if (t >= num_tokens) return;
        float acc[4] = {0.f, 0.f, 0.f, 0.f};
        const int slot = item[r] >= 0 ? item_slot[item[r]] : -1;
        if (slot >= 0) {                             // (else a padding row of a batch of fixed size: zeros)
            const int own = t - item_tok_off[item[r]];       // row within the item's portion
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (add_input) acc[u] = rows[HIST + r][u];
                if (bias) acc[u] += b[u];
            }
#pragma unroll
            for (int j = 0; j < TAPS; ++j) {
                float v[4];
                if (own - (HIST - j) >= 0) {
#pragma unroll
                    for (int u = 0; u < 4; ++u) v[u] = rows[r + j][u];
                } else {
                    Elem<float>::load_vec(state + (int64_t)slot * slot_stride + (int64_t)(own + j) * channels + c, v);
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) acc[u] = fmaf(f[u * TAPS + j], v[u], acc[u]);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) acc[u] = apply_activation(activation, acc[u]);
        }
        Elem<TO>::store4(out + (int64_t)t * channels + c, acc);
    }
}

// One thread per (item, channel): the new state is the last taps - 1 of (old state, the item's rows).
template <typename TI>
__global__ __launch_bounds__(256) void token_conv_state_kernel(
    float* __restrict__ state, int64_t slot_stride, const TI* __restrict__ x, int64_t x_stride,
    const int* __restrict__ item_len, const int* __restrict__ item_tok_off, const int* __restrict__ item_slot,
    int channels, int taps) {
    const int item = blockIdx.x;
    const int c = blockIdx.y * 256 + threadIdx.x;
    if (c >= channels) return;
    const int slot = item_slot[item], n = item_len[item];
    if (slot < 0 || n <= 0) return;
    const int hist = taps - 1;
    float* st_c = state + (int64_t)slot * slot_stride + c;
    const TI* x_c = x + (int64_t)item_tok_off[item] * x_stride + c;
    float keep[kMaxTaps];
#pragma unroll
    for (int i = 0; i < kMaxTaps; ++i) {
        if (i >= hist) break;
        const int p = n - hist + i;                  // row of the portion, negative: still in the old state
        keep[i] = p >= 0 ? Elem<TI>::load(x_c + (int64_t)p * x_stride) : st_c[(int64_t)(hist + p) * channels];
    }
#pragma unroll
    for (int i = 0; i < kMaxTaps; ++i) {
        if (i >= hist) break;
        st_c[(int64_t)i * channels] = keep[i];
    }
}

}  // namespace st

using namespace st;

extern "C" int st_token_conv(void* out, const void* x, int64_t x_stride, int in_dtype, const float* w,
                             const float* bias, const float* state, int64_t slot_stride, const int* token_item,
                             const int* item_tok_off, const int* item_slot, int num_tokens, int channels, int taps,
                             int add_input, int activation, int out_dtype, hipStream_t stream) {
    ST_CHECK(num_tokens >= 0 && channels > 0, "token_conv: bad sizes T=%d C=%d", num_tokens, channels);
    ST_CHECK(taps >= 1 && taps <= kMaxTaps, "token_conv: 1 to %d taps, not %d", kMaxTaps, taps);
    ST_CHECK(out && x && w && token_item && item_tok_off && item_slot && (state || taps == 1), "token_conv: null operand");
    ST_CHECK(out != x, "token_conv: the result cannot take its input's place");
    ST_CHECK(activation_known(activation), "token_conv: activation %d has no kernel", activation);
    ST_CHECK((in_dtype == kF32 || in_dtype == kBF16) && (out_dtype == kF32 || out_dtype == kBF16),
             "token_conv: unknown dtype %d -> %d", in_dtype, out_dtype);
    if (num_tokens == 0) return 0;
    // Four channels a thread where every row of x, of the state and of the filters starts on a whole piece; filters of 2 to 4 taps, which
    // all mixers and streams here have.  Four rows a thread where that still gives every compute unit a workgroup: with fewer, threads are
    // what is missing (100 rows of 2,048 channels, 4 taps, by element 5.5 us, four rows a thread 6.4, one row 5.0; 505 rows of 768 6.1, 6.8 and
    // 5.1).  One row or two go by element (one of 2,048, 2 taps, 4.2 and 4.5; eight 4.2 and 4.3, 4 taps 4.8 and 4.7).
    const int in_bytes = in_dtype == kF32 ? 16 : 8, out_bytes = out_dtype == kF32 ? 16 : 8;
    const bool four = channels % 4 == 0 && x_stride % 4 == 0 && slot_stride % 4 == 0 && (uintptr_t)x % in_bytes == 0 &&
                      (uintptr_t)out % out_bytes == 0 && (((uintptr_t)w | (uintptr_t)bias | (uintptr_t)state) & 15) == 0;
#define ST_CONV4(TI, TO, TAPS, ROWS)                                                                            \
    token_conv_rows_kernel<TI, TO, TAPS, ROWS><<<dim3((num_tokens + ROWS - 1) / ROWS, (channels / 4 + 255) / 256), 256, 0, stream>>>( \
        (TO*)out, (const TI*)x, x_stride, w, bias, state, slot_stride, token_item, item_tok_off, item_slot, num_tokens, channels,  \
        add_input, activation)
#define ST_CONV_TAPS(TI, TO, ROWS)                                                                              \
    do { if (taps == 2) ST_CONV4(TI, TO, 2, ROWS); else if (taps == 3) ST_CONV4(TI, TO, 3, ROWS); else ST_CONV4(TI, TO, 4, ROWS); } while (0)
#define ST_CONV_ROWS(TI, TO) do { if (four_rows) ST_CONV_TAPS(TI, TO, 4); else ST_CONV_TAPS(TI, TO, 1); } while (0)
    const bool four_rows = ((int64_t)num_tokens + 3) / 4 * ((channels + 1023) / 1024) >= device_compute_units();
    if (four && num_tokens > 2 && taps >= 2 && taps <= 4) {
        if (in_dtype == kF32 && out_dtype == kF32) ST_CONV_ROWS(float, float);
        else if (in_dtype == kF32) ST_CONV_ROWS(float, bf16_t);
        else if (out_dtype == kF32) ST_CONV_ROWS(bf16_t, float);
        else ST_CONV_ROWS(bf16_t, bf16_t);
        ST_LAUNCH_CHECK("token_conv");
        return 0;
    }
#undef ST_CONV4
#undef ST_CONV_TAPS
#undef ST_CONV_ROWS
    const dim3 grid(num_tokens, (channels + 255) / 256);
#define ST_CONV(TI, TO)                                                                                      \
    token_conv_kernel<TI, TO><<<grid, 256, 0, stream>>>((TO*)out, (const TI*)x, x_stride, w, bias, state,   \
        slot_stride, token_item, item_tok_off, item_slot, channels, taps, add_input, activation)
    if (in_dtype == kF32 && out_dtype == kF32) ST_CONV(float, float);
    else if (in_dtype == kF32) ST_CONV(float, bf16_t);
    else if (out_dtype == kF32) ST_CONV(bf16_t, float);
    else ST_CONV(bf16_t, bf16_t);
#undef ST_CONV
    ST_LAUNCH_CHECK("token_conv");
    return 0;
}

extern "C" int st_token_conv_state(float* state, int64_t slot_stride, const void* x, int64_t x_stride, int in_dtype,
                                   const int* item_len, const int* item_tok_off, const int* item_slot, int num_items,
                                   int channels, int taps, hipStream_t stream) {
    ST_CHECK(num_items >= 0 && channels > 0, "token_conv_state: bad sizes");
    ST_CHECK(taps >= 1 && taps <= kMaxTaps, "token_conv_state: 1 to %d taps, not %d", kMaxTaps, taps);
    ST_CHECK(in_dtype == kF32 || in_dtype == kBF16, "token_conv_state: unknown dtype %d", in_dtype);
    if (num_items == 0 || taps == 1) return 0;
    ST_CHECK(state && x && item_len && item_tok_off && item_slot, "token_conv_state: null operand");
    const dim3 grid(num_items, (channels + 255) / 256);
    if (in_dtype == kF32)
        token_conv_state_kernel<float><<<grid, 256, 0, stream>>>(state, slot_stride, (const float*)x, x_stride,
                                                                 item_len, item_tok_off, item_slot, channels, taps);
    else
        token_conv_state_kernel<bf16_t><<<grid, 256, 0, stream>>>(state, slot_stride, (const bf16_t*)x, x_stride,
                                                                  item_len, item_tok_off, item_slot, channels, taps);
    ST_LAUNCH_CHECK("token_conv_state");
    return 0;
}
