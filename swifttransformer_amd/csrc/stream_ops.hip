// Small float operations on the residual stream that are no product's epilogue:
//
//   dynamic tanh   y = tanh(alpha x) * w + b   per element (no mean, no variance), alpha one number on
//                  the device; optionally of picked rows, optionally added to a second stream
//                  (out32 = base + y: a branch's result normalised on its way into the stream), and
//                  optionally followed by a second dynamic tanh of that sum in the storage type (what
//                  the next sublayer reads), so that norm-after, residual sum and norm-before are one pass;
//   unit add       x += y / sqrt(mean(y^2) + eps) * w   per row (a branch that enters the stream at
//                  unit root mean square);
//   row add        out = x (+ first) + vec   (a pass over a group of layers that starts from the stream
//                  plus the step's embedding plus that pass's vector).
//   token side     x += unit(P (gelu_tanh(G x) * e[token])) * w   per row: a narrow embedding row gates a
//                  projection of the stream, which re-enters it at unit root mean square; lookup, the two
//                  small products, the activation, the norm and the sum in one kernel.
//
// Everything is float except the optional copy of the dynamic tanh in the storage type and the token side
// input's matrices and table, which are of the storage type.
#include "activation.h"
#include "api.h"
#include "common.h"

#include <type_traits>

namespace st {

// V columns a thread (4: 16-byte accesses); a workgroup takes 256 V columns of one row.  1,024 rows of 2,048 into the storage type, by
// element and by four: 8.8 and 6.0 us.
template <typename T, int V>
__global__ __launch_bounds__(256) void dynamic_tanh_kernel(
    T* __restrict__ out_t, float* __restrict__ out32, const float* __restrict__ x, const int* __restrict__ rows,
    const float* __restrict__ w, const float* __restrict__ b, const float* __restrict__ alpha,
    const float* __restrict__ base, const float* __restrict__ w2, const float* __restrict__ b2,
    const float* __restrict__ alpha2, int width) {
    const int64_t r = blockIdx.x;
    int64_t src = r;
    if (rows) {
        src = rows[r];
        if (src < 0) return;                              // a padding entry
    }
    auto load = [](const float* p, float* v) {
        if (V == 4) Elem<float>::load_vec(p, v);
        else v[0] = p[0];
    };
    for (int64_t c = ((int64_t)blockIdx.y * 256 + threadIdx.x) * V; c < width; c += (int64_t)gridDim.y * 256 * V) {
        const int64_t idx = r * width + c;
        float y[V], g[V], s[V], g2[V], s2[V], on[V];
        load(x + src * width + c, y);
        load(w + c, g);
        if (b) load(b + c, s);
        if (base) load(base + idx, on);
        if (w2) load(w2 + c, g2);
        if (b2) load(b2 + c, s2);
        const float a = alpha[0], a2 = w2 ? alpha2[0] : 0.f;
#pragma unroll
        for (int u = 0; u < V; ++u) {
            y[u] = tanhf(a * y[u]) * g[u] + (b ? s[u] : 0.f);
            if (base) y[u] += on[u];
        }
        if (out32) {
            if (V == 4) Elem<float>::store_vec(out32 + idx, y);
            else out32[idx] = y[0];
        }
        if (w2) {                                             // the next norm, of the sum just made
#pragma unroll
            for (int u = 0; u < V; ++u) y[u] = tanhf(a2 * y[u]) * g2[u] + (b2 ? s2[u] : 0.f);
        }
        if (out_t) {
            if (V == 4) Elem<T>::store4(out_t + idx, y);
            else Elem<T>::store(out_t + idx, y[0]);
        }
    }
}

// logits through a factor and a smooth limit: cap * tanh(x * scale / cap)
__global__ __launch_bounds__(256) void scale_softcap_kernel(float* __restrict__ x, int64_t n, float scale, float cap) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float v = x[i] * scale;
    x[i] = cap > 0.f ? cap * tanhf(v / cap) : v;
}

// a workgroup a row
__global__ __launch_bounds__(256) void unit_add_kernel(float* __restrict__ x, const float* __restrict__ y,
                                                       const float* __restrict__ w, int width, float eps) {
    __shared__ float red[16];
    const int64_t row = blockIdx.x;
    const float* yr = y + row * width;
    float ss = 0.f;
    for (int c = threadIdx.x; c < width; c += 256) ss = fmaf(yr[c], yr[c], ss);
    ss = block_sum(ss, red);
    const float r = 1.f / sqrtf(ss / (float)width + eps);
    float* xr = x + row * width;
    for (int c = threadIdx.x; c < width; c += 256) xr[c] += yr[c] * r * w[c];
}

__global__ __launch_bounds__(256) void row_add_kernel(float* __restrict__ out, const float* __restrict__ x,
                                                      const float* __restrict__ first, const float* __restrict__ vec,
                                                      int width, int64_t total) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= total) return;
    float v = x[idx];
    if (first) v += first[idx];
    out[idx] = v + vec[idx % width];
}

// A workgroup a row: 16 waves where rows are few (a decode step: every gate feature's row of G in flight
// at once, the kernel's time a handful of dependent trips to memory), 4 otherwise.  LDS: the float row,
// later the projection's result; the gated vector.  Only the matrices and the table are of the storage
// type: the row, the gate's sums and the gated vector stay float (a unit norm follows, and a gated vector
// of a few entries near zero would turn a rounding into a direction).
// g_j = gelu(G_j . x) * e_j, y = P g, x += y / sqrt(mean(y^2) + eps) * w.
// VEC: rows of G and P allow 16-byte loads.
template <typename T, bool VEC>
__global__ __launch_bounds__(1024) void token_side_kernel(
    float* __restrict__ x, const int* __restrict__ token_ids, const int* __restrict__ token_item,
    const T* __restrict__ table, int64_t table_stride, int vocab, const T* __restrict__ w_gate,
    const T* __restrict__ w_proj, const float* __restrict__ gain, int dim, int width, float eps) {
    extern __shared__ __attribute__((aligned(16))) float side_lds[];
    __shared__ float red[16];
    float* xs = side_lds;                 // [width]
    float* gs = side_lds + width;         // [dim]
    const int64_t row = blockIdx.x;
    if (token_item && token_item[row] < 0) return;        // a padding row (uniform over the workgroup)
    constexpr int V = Elem<T>::kVec;
    const int threads = blockDim.x, waves = threads >> 6;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float* xr = x + row * width;
    const int tok = token_ids[row];
    const bool known = tok >= 0 && tok < vocab;
    const T* er = table + (int64_t)(known ? tok : 0) * table_stride;
    // the first feature's table entry is asked for before the row arrives
    float e = (known && wave < dim) ? Elem<T>::load(er + wave) : 0.f;
    for (int c = threadIdx.x; c < width; c += threads) xs[c] = xr[c];
    __syncthreads();
    for (int j = wave; j < dim; j += waves) {
        const T* gr = w_gate + (int64_t)j * width;
        float acc = 0.f;
        if (VEC) {
            for (int c = lane * V; c < width; c += 64 * V) {
                float w[V];
                Elem<T>::load_vec(gr + c, w);
#pragma unroll
                for (int u = 0; u < V; ++u) acc = fmaf(w[u], xs[c + u], acc);
            }
        } else {
            for (int c = lane; c < width; c += 64) acc = fmaf(Elem<T>::load(gr + c), xs[c], acc);
        }
        acc = wave_sum(acc);
        if (lane == 0) gs[j] = apply_activation(kActGeluTanh, acc) * e;
        if (j + waves < dim) e = known ? Elem<T>::load(er + j + waves) : 0.f;
    }
    __syncthreads();                      // every wave has read xs; gs is complete
    float ss = 0.f;
    for (int c = threadIdx.x; c < width; c += threads) {
        const T* pr = w_proj + (int64_t)c * dim;
        float y = 0.f;
        if (VEC) {
            for (int j = 0; j < dim; j += V) {
                float w[V];
                Elem<T>::load_vec(pr + j, w);
#pragma unroll
                for (int u = 0; u < V; ++u) y = fmaf(w[u], gs[j + u], y);
            }
        } else {
            for (int j = 0; j < dim; ++j) y = fmaf(Elem<T>::load(pr + j), gs[j], y);
        }
        xs[c] = y;                        // this thread's own entries from here on
        ss = fmaf(y, y, ss);
    }
    ss = block_sum(ss, red);
    const float r = 1.f / sqrtf(ss / (float)width + eps);
    for (int c = threadIdx.x; c < width; c += threads) xr[c] += xs[c] * r * gain[c];
}

// The same for more bfloat16 rows than there are compute units: a workgroup two rows, so that G and P pass from the L2 to a compute unit
// once for both (a row a workgroup: 128 KB a row at 2,048 columns, 134 MB for 1,024 rows).  Everything that is read, the rows, G (a wave a
// feature), P, the table's entries and the gains, is asked for before anything waits: one trip to memory.  What bounds it then is the LDS, from
// which every wave reads the rows.  us, a row a workgroup of 256 threads and this, columns of 2,048: 300 rows 11.0 and 6.8, 512 11.4 and 7.3, 768
// 12.5 and 10.9, 1,024 13.5 and 11.5, 2,048 23.1 and 21.2.  Four rows a workgroup: 12.2 at 512, 14.1 at 1,024.  NC: columns a thread.
template <int NC>
__global__ __launch_bounds__(1024) void token_side_rows_kernel(
    float* __restrict__ x, const int* __restrict__ token_ids, const int* __restrict__ token_item, const bf16_t* __restrict__ table,
    int64_t table_stride, int vocab, const bf16_t* __restrict__ w_gate, const bf16_t* __restrict__ w_proj, const float* __restrict__ gain,
    int num_rows, int dim, int width, float eps) {
    constexpr int R = 2;
    constexpr int DIM = 16, V = Elem<bf16_t>::kVec, NV = 2 * NC;         // NV: pieces of eight columns of G a lane
    extern __shared__ __attribute__((aligned(16))) float side_rows_lds[];
    __shared__ __attribute__((aligned(16))) float gs[R][DIM], red[16][R];
    float* xs = side_rows_lds;                                           // [R][width]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, row0 = blockIdx.x * R, quads = width >> 2;
    // a row's quads of numbers in LDS: the even ones, then the odd ones (a lane reads two neighbouring ones)
    const auto place = [&](int r, int q) { return r * quads + (q & 1) * (quads >> 1) + (q >> 1); };
    // (rows past the last stand for it)
    constexpr int XV = (NC + 1) / 2;                                     // quads a thread: half of the workgroup a row
    const int half = tid >> 9, first = tid & 511;
    const float* xr = x + (int64_t)min(row0 + half, num_rows - 1) * width;
    float4 xv[XV];
#pragma unroll
    for (int i = 0; i < XV; ++i) xv[i] = *reinterpret_cast<const float4*>(xr + 4 * min(first + 512 * i, quads - 1));
    uint4 g[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int c = (lane + 64 * v) * V;
        g[v] = *reinterpret_cast<const uint4*>(w_gate + (int64_t)min(wave, dim - 1) * width + (c < width ? c : 0));
    }
    float e = 0.f;                                                       // lane r: row r's entry of the wave's feature
    if (lane < R && row0 + lane < num_rows && wave < dim) {
        const int tok = token_ids[row0 + lane];
        if (tok >= 0 && tok < vocab) e = Elem<bf16_t>::load(table + (int64_t)tok * table_stride + wave);
    }
    uint4 p[NC][DIM / V];
    float gn[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        const int c = min(tid + 1024 * i, width - 1);
#pragma unroll
        for (int h = 0; h < DIM / V; ++h)
            p[i][h] = h * V < dim ? *reinterpret_cast<const uint4*>(w_proj + (int64_t)c * dim + h * V) : make_uint4(0, 0, 0, 0);
        gn[i] = gain[c];
    }
#pragma unroll
    for (int i = 0; i < XV; ++i) {
        if (first + 512 * i < quads) reinterpret_cast<float4*>(xs)[place(half, first + 512 * i)] = xv[i];
    }
    __syncthreads();
    float sum[R];
#pragma unroll
    for (int r = 0; r < R; ++r) sum[r] = 0.f;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int c = (lane + 64 * v) * V;
        if (c >= width) continue;
        float w[V];
        Elem<bf16_t>::unpack(g[v], w);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float4 lo = reinterpret_cast<const float4*>(xs)[place(r, c >> 2)], hi = reinterpret_cast<const float4*>(xs)[place(r, (c >> 2) + 1)];
            sum[r] = fmaf(w[0], lo.x, sum[r]); sum[r] = fmaf(w[1], lo.y, sum[r]); sum[r] = fmaf(w[2], lo.z, sum[r]); sum[r] = fmaf(w[3], lo.w, sum[r]);
            sum[r] = fmaf(w[4], hi.x, sum[r]); sum[r] = fmaf(w[5], hi.y, sum[r]); sum[r] = fmaf(w[6], hi.z, sum[r]); sum[r] = fmaf(w[7], hi.w, sum[r]);
        }
    }
    float own = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        sum[r] = wave_sum(sum[r]);
        if (lane == r) own = sum[r];
    }
    if (lane < R) gs[lane][wave] = wave < dim ? apply_activation(kActGeluTanh, own) * e : 0.f;
    __syncthreads();
    float y[R][NC], ss[R];
#pragma unroll
    for (int r = 0; r < R; ++r) ss[r] = 0.f;
    float w[NC][DIM];
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
        for (int h = 0; h < DIM / V; ++h) Elem<bf16_t>::unpack(p[i][h], w[i] + h * V);
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int i = 0; i < NC; ++i) y[r][i] = 0.f;
#pragma unroll
        for (int j = 0; j < DIM; j += 4) {
            const float4 v = *reinterpret_cast<const float4*>(&gs[r][j]);
#pragma unroll
            for (int i = 0; i < NC; ++i) {
                y[r][i] = fmaf(w[i][j], v.x, y[r][i]); y[r][i] = fmaf(w[i][j + 1], v.y, y[r][i]);
                y[r][i] = fmaf(w[i][j + 2], v.z, y[r][i]); y[r][i] = fmaf(w[i][j + 3], v.w, y[r][i]);
            }
        }
#pragma unroll
        for (int i = 0; i < NC; ++i)
            if (tid + 1024 * i < width) ss[r] = fmaf(y[r][i], y[r][i], ss[r]);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        ss[r] = wave_sum(ss[r]);
        if (lane == 0) red[wave][r] = ss[r];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (row0 + r >= num_rows || (token_item && token_item[row0 + r] < 0)) continue;      // past the last row, or a padding row
        float total = 0.f;
#pragma unroll
        for (int w = 0; w < 16; ++w) total += red[w][r];
        const float scale = 1.f / sqrtf(total / (float)width + eps);
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const int c = tid + 1024 * i;
            if (c < width) x[(int64_t)(row0 + r) * width + c] = xs[place(r, c >> 2) * 4 + (c & 3)] + y[r][i] * scale * gn[i];
        }
    }
}

}  // namespace st

using namespace st;

extern "C" int st_dynamic_tanh(void* out_t, float* out32, const float* x, const int* rows, const float* w,
                               const float* b, const float* alpha, const float* base, const float* w2,
                               const float* b2, const float* alpha2, int num_rows, int width, int dtype,
                               hipStream_t stream) {
    ST_CHECK(num_rows >= 0 && width > 0, "dynamic_tanh: bad sizes");
    if (num_rows == 0) return 0;
    ST_CHECK(x && w && alpha && (out_t || out32), "dynamic_tanh: null operand");
    ST_CHECK(!w2 || (alpha2 && out_t), "dynamic_tanh: a second norm needs its alpha and the storage-type output");
    ST_CHECK(dtype == kF32 || dtype == kBF16, "dynamic_tanh: unknown dtype %d", dtype);
    const uintptr_t align = (uintptr_t)out32 | (uintptr_t)x | (uintptr_t)w | (uintptr_t)b | (uintptr_t)base | (uintptr_t)w2 | (uintptr_t)b2;
    // (by fours where that gives every compute unit more than a workgroup: with base and second norm 8 rows of 2,048 by element 2.65 us, by
    // fours 3.02, 64 rows of 4,096 3.2 and 3.3, 500 rows of 2,048 5.2 and 4.2)
    const bool four = width % 4 == 0 && (align & 15) == 0 && (uintptr_t)out_t % (dtype == kF32 ? 16 : 8) == 0 &&
                      (int64_t)num_rows * (((int64_t)width + 1023) / 1024) > device_compute_units();
    const int span = four ? 1024 : 256;
    const int64_t blocks = ((int64_t)width + span - 1) / span;
    const dim3 grid((unsigned)num_rows, (unsigned)(blocks < 65535 ? blocks : 65535));
#define ST_DT(T, V)                                                                                             \
    dynamic_tanh_kernel<T, V><<<grid, 256, 0, stream>>>((T*)out_t, out32, x, rows, w, b, alpha, base, w2, b2, alpha2, width)
    if (dtype == kF32) { if (four) ST_DT(float, 4); else ST_DT(float, 1); }
    else { if (four) ST_DT(bf16_t, 4); else ST_DT(bf16_t, 1); }
#undef ST_DT
    ST_LAUNCH_CHECK("dynamic_tanh");
    return 0;
}

extern "C" int st_scale_softcap(float* x, int64_t n, float scale, float cap, hipStream_t stream) {
    ST_CHECK(n >= 0 && scale == scale && cap == cap, "scale_softcap: bad operands");
    if (n == 0) return 0;
    ST_CHECK(x, "scale_softcap: null operand");
    scale_softcap_kernel<<<(unsigned)((n + 255) / 256), 256, 0, stream>>>(x, n, scale, cap);
    ST_LAUNCH_CHECK("scale_softcap");
    return 0;
}

extern "C" int st_unit_add(float* x, const float* y, const float* w, int num_rows, int width, float eps,
                           hipStream_t stream) {
    ST_CHECK(num_rows >= 0 && width > 0 && eps > 0.f, "unit_add: bad sizes");
    if (num_rows == 0) return 0;
    ST_CHECK(x && y && w, "unit_add: null operand");
    unit_add_kernel<<<(unsigned)num_rows, 256, 0, stream>>>(x, y, w, width, eps);
    ST_LAUNCH_CHECK("unit_add");
    return 0;
}

extern "C" int st_row_add(float* out, const float* x, const float* first, const float* vec, int num_rows, int width,
                          hipStream_t stream) {
    ST_CHECK(num_rows >= 0 && width > 0, "row_add: bad sizes");
    if (num_rows == 0) return 0;
    ST_CHECK(out && x && vec, "row_add: null operand");
    const int64_t total = (int64_t)num_rows * width;
    row_add_kernel<<<(unsigned)((total + 255) / 256), 256, 0, stream>>>(out, x, first, vec, width, total);
    ST_LAUNCH_CHECK("row_add");
    return 0;
}

extern "C" int st_token_side(float* x, const int* token_ids, const int* token_item, const void* table,
                             int64_t table_stride, int vocab, const void* w_gate, const void* w_proj,
                             const float* gain, int num_rows, int dim, int width, float eps, int dtype,
                             hipStream_t stream) {
    ST_CHECK(num_rows >= 0 && width > 0 && dim > 0 && vocab > 0 && eps > 0.f && table_stride >= dim,
             "token_side: bad sizes");
    ST_CHECK(dtype == kF32 || dtype == kBF16, "token_side: unknown dtype %d", dtype);
    const size_t lds = sizeof(float) * ((size_t)width + dim);
    ST_CHECK(lds <= 60 * 1024, "token_side: a row of %d and a gated vector of %d do not fit the LDS", width, dim);
    if (num_rows == 0) return 0;
    ST_CHECK(x && token_ids && table && w_gate && w_proj && gain, "token_side: null operand");
    const int threads = num_rows <= 256 ? 1024 : 256;
    const int vec = dtype == kF32 ? 4 : 8;
    const bool aligned = width % vec == 0 && dim % vec == 0 && (uintptr_t)w_gate % 16 == 0 && (uintptr_t)w_proj % 16 == 0;
    // Two rows a workgroup up to two rounds of rows a unit, and beyond that where the rows are neither so short that their weights are not what
    // counts nor so long that few of their workgroups run at once (us, a row a workgroup and two: 600 rows of 768 7.3 and 7.6, 1,024 8.2 and
    // 8.3; 600 of 2,560 13.6 and 18.7, 1,024 of 4,096 22.6 and 24.3; but 300 of 4,096 18.4 and 12.1, of 768 7.0 and 5.4).
    const int units = device_compute_units();
    if (dtype == kBF16 && aligned && dim <= 16 && width <= 4096 && (uintptr_t)x % 16 == 0 && num_rows > 256 &&
        (num_rows <= 2 * units || (width > 1024 && width <= 2048))) {
        const auto launch = [&](auto columns) {
            token_side_rows_kernel<decltype(columns)::value><<<(unsigned)((num_rows + 1) / 2), 1024, sizeof(float) * 2 * width, stream>>>(
                x, token_ids, token_item, (const bf16_t*)table, table_stride, vocab, (const bf16_t*)w_gate, (const bf16_t*)w_proj, gain, num_rows,
                dim, width, eps);
        };
        if (width <= 1024) launch(std::integral_constant<int, 1>());
        else if (width <= 2048) launch(std::integral_constant<int, 2>());
        else launch(std::integral_constant<int, 4>());
        ST_LAUNCH_CHECK("token_side");
        return 0;
    }
#define ST_SIDE(T, VEC)                                                                                          \
    token_side_kernel<T, VEC><<<(unsigned)num_rows, threads, lds, stream>>>(                                         \
        x, token_ids, token_item, (const T*)table, table_stride, vocab, (const T*)w_gate, (const T*)w_proj, gain, dim, \
        width, eps)
    if (dtype == kF32) {
        if (aligned) ST_SIDE(float, true); else ST_SIDE(float, false);
    } else {
        if (aligned) ST_SIDE(bf16_t, true); else ST_SIDE(bf16_t, false);
    }
#undef ST_SIDE
    ST_LAUNCH_CHECK("token_side");
    return 0;
}
