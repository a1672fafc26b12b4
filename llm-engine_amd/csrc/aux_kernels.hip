// Small kernels around the products:
//   naive_kernel    GpuKernel::naive, one thread per element of C
//                   (reference sgemm_naive, cuda_matmul.cu:34-47)
//   reduce_slices   fixed-order split-K sum, scale and residual add
//                   (reference sum_slices, cuda_matmul.cu:245-254)
//   rmsnorm_rows    the separate norm pass for kernels that don't fuse it
//                   (reference rmsnorm_rows, cuda_matmul.cu:256-266)
//   fill_zero       k == 0 output (cuda_matmul.cu:419-422), as a kernel so a
//                   captured graph holds no memset node
//   quantize_q8     quant.cpp:6-28 on the GPU, bit-exact: column absmax in
//                   slices + an order-free max, then scale = absmax / 127 and
//                   inv = 1 / scale with IEEE division (in a launch of their
//                   own for large matrices), then
//                   q = clamp(round-half-away(B * inv), -127, 127)
//   dequantize_q8   quant.cpp:30-36
//   stream_read     a read-only pass over a buffer (probes.hip's read kernel
//                   in its fastest shape): the HBM ceiling that the GEMV is
//                   compared with (no counterpart in the reference, whose
//                   bench times a device-to-device copy instead,
//                   bench_cuda.cpp:79-88)
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "internal.hpp"

namespace em {
namespace {

template <class BT>
__device__ __forceinline__ float load_b(const BT* B, int idx, const float* scale, int col) {
    if constexpr (std::is_same<BT, float>::value) {
        return B[idx];
    } else {
        return static_cast<float>(B[idx]) * scale[col];
    }
}

template <class BT>
__global__ __launch_bounds__(kThreads) void naive_kernel(int m, int n, int k, const float* A,
                                                         const BT* B, const float* scale,
                                                         float* C, int accumulate) {
    const int col = blockIdx.x * 64 + threadIdx.x % 64;
    const int row = blockIdx.y * 4 + threadIdx.x / 64;
    if (row >= m || col >= n) return;
    float acc = 0.0f;
    for (int p = 0; p < k; ++p) acc = fmaf(A[row * k + p], load_b(B, p * n + col, scale, col), acc);
    float* c = C + static_cast<size_t>(row) * n + col;
    *c = accumulate ? *c + acc : acc;
}

// One output per thread. C and the scale are loaded with the first
// partials, so no round trip waits on them alone. With ssq,
// each wave (outputs 64w .. 64w + 63, one row of C when n is a multiple of
// 64) also writes the sum of their squares, by a fixed butterfly.
// 256-thread workgroups: 64-thread ones measured 0.5 us slower per call.
static_assert(kSsqChunk == kWave, "one sum of squares per wave");

__global__ __launch_bounds__(kThreads) void reduce_slices_kernel(
    int mn, int n, int slices, const float* __restrict__ partial, const float* __restrict__ scale,
    float* __restrict__ C, int accumulate, float* __restrict__ ssq) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    const bool in = i < mn;
    const int ii = in ? i : mn - 1;
    const float prior = accumulate ? C[ii] : 0.0f;
    const float sc = scale ? scale[ii % n] : 1.0f;
    float total = ordered_sum(partial, static_cast<uint32_t>(ii), static_cast<uint32_t>(mn), slices);
    if (scale) total *= sc;
    const float out = accumulate ? prior + total : total;
    if (in) C[i] = out;
    if (ssq) {
        const float sq = wave_sum(in ? out * out : 0.0f);
        if (in && threadIdx.x % kWave == 0) ssq[i / kSsqChunk] = sq;
    }
}

// One workgroup a row, R columns of each thread in flight; a row of one round
// is not read again, and the sum's order is the same for any R. A load at a
// time, a row of 4096 waited for 16 trips to memory in each pass: 300 rows 12.1
// us, 6.2 with R = 16; 128 of 11008 13.2 -> 6.8; 2048 of 4096 16.3 -> 12.1.
// Rows to 1024 take R = 4 (64 rows of 288: 2.8 us, 3.3 with 16 clamped loads).
template <int R>
__global__ __launch_bounds__(kThreads) void rmsnorm_rows_kernel(int k, const float* A,
                                                                const float* w, float* out) {
    __shared__ float part[4];
    const float* in = A + static_cast<size_t>(blockIdx.x) * k;
    float* o = out + static_cast<size_t>(blockIdx.x) * k;
    // Columns j0, j0 + kThreads, ...: past the row its last column.
    auto load = [&](const float* src, int j0, float (&v)[R]) {
#pragma unroll
        for (int u = 0; u < R; ++u) v[u] = src[min(j0 + u * kThreads, k - 1)];
    };
    const int tid = threadIdx.x;
    float x[R], y[R], ss = 0.0f;
    load(in, tid, x);
    load(w, tid, y);
    auto add = [&](int j0) {
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const float v = j0 + u * kThreads < k ? x[u] : 0.0f;
            ss = fmaf(v, v, ss);
        }
    };
    add(tid);
    for (int j0 = tid + R * kThreads; j0 < k; j0 += R * kThreads) {
        load(in, j0, x);
        add(j0);
    }
    const float s = 1.0f / sqrtf(block_sum(ss, part) / static_cast<float>(k) + kRmsEps);
    for (int j0 = tid; j0 < k; j0 += R * kThreads) {
        if (k > R * kThreads) {
            load(in, j0, x);
            load(w, j0, y);
        }
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const int j = j0 + u * kThreads;
            if (j < k) o[j] = x[u] * s * y[u];
        }
    }
}

__global__ __launch_bounds__(kThreads) void fill_zero_kernel(float* p, size_t count) {
    for (size_t i = static_cast<size_t>(blockIdx.x) * kThreads + threadIdx.x; i < count;
         i += static_cast<size_t>(gridDim.x) * kThreads)
        p[i] = 0.0f;
}

// --- quantize_q8 -----------------------------------------------------------

// A thread of both kernels owns four adjacent columns, 4 idx .. + 3, and reads
// them as one 16-byte load (4-byte aligned: a row of any width starts on a
// float), all rows of a round in flight before any is used. The last group
// of a width that is not whole groups is shifted back to end at the last
// column: its columns are then also another thread's, with the same result.
struct __attribute__((packed, aligned(4))) Floats4 {
    float v[4];
};

__device__ __forceinline__ int column_group(int idx, int cols) { return min(4 * idx, cols - 4); }

constexpr int kQuantRound = 16;  // rows in flight per thread

// Column maxima of |B| over one slice of rows: partial[slice][4 idx + e] of
// column column_group(idx) + e, `stride` floats to a slice. Bound by the read
// of B (4096 x 11008: 180 MB). With W = 1, fewer than four columns, a thread
// owns one: partial[slice][idx] of column idx.
template <int W>
__global__ __launch_bounds__(kThreads) void colmax_kernel(int rows, int cols, int span, int stride,
                                                          const float* B, float* partial) {
    const int idx = blockIdx.x * kThreads + threadIdx.x;
    if (W * idx >= stride) return;
    const float* col = B + (W == 4 ? column_group(idx, cols) : idx);
    const int r0 = blockIdx.y * span, r1 = min(rows, r0 + span);
    // fmaxf keeps the running value when |B| is NaN, as std::max(scale, v)
    // does in quant.cpp:14; on ordered values max is exact in any order, so
    // the last round may read its last row again.
    float mx[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int r = r0; r < r1; r += kQuantRound) {
        Floats4 x[kQuantRound];
#pragma unroll
        for (int u = 0; u < kQuantRound; ++u) {
            const float* at = col + static_cast<size_t>(min(r + u, r1 - 1)) * cols;
            if constexpr (W == 4)
                x[u] = *reinterpret_cast<const Floats4*>(at);
            else
                x[u].v[0] = *at;
        }
#pragma unroll
        for (int u = 0; u < kQuantRound; ++u)
#pragma unroll
            for (int e = 0; e < W; ++e) mx[e] = fmaxf(mx[e], fabsf(x[u].v[e]));
    }
    float* out = partial + static_cast<size_t>(blockIdx.y) * stride + W * idx;
    if constexpr (W == 4)
        *reinterpret_cast<floatx4*>(out) = floatx4{mx[0], mx[1], mx[2], mx[3]};
    else
        *out = mx[0];
}

// lround for the range that matters, half away from zero: x + 0.5 less one
// ulp of it, with x's sign, truncated. The sum reaches the next integer from
// a fraction of one half up (a tie that rounds to even, or nearer) and from
// nothing below. The product is rounded to fp32 before anything else reads
// it (no contraction into the sum), as quant.cpp:23 computes B * inv first.
__device__ __forceinline__ int quantize_one(float b, float inv) {
#pragma clang fp contract(off)
    const float x = b * inv;
    const float r = x + copysignf(0x1.fffffep-2f, x);
    return static_cast<int>(fminf(fmaxf(r, -127.0f), 127.0f));
}

// One slab of rows: scale = absmax / 127 and inv = 1 / scale (0 for a zero
// column) of the thread's columns, both correctly rounded (the library is
// built with IEEE fp32 division), from the slices' maxima; then the rows.
// The first slab writes the scales. Forming them here costs each workgroup
// `slices` L2 reads a thread and saves a launch.
__global__ __launch_bounds__(kThreads) void quantize_kernel(int rows, int cols, int span, int stride,
                                                            int slices, const float* B,
                                                            const float* partial, float* scale,
                                                            int8_t* q) {
    const int idx = blockIdx.x * kThreads + threadIdx.x;
    if (4 * idx >= stride) return;
    const int c = column_group(idx, cols);
    float inv[4];
    {
        floatx4 mx{0.f, 0.f, 0.f, 0.f};
        for (int s = 0; s < slices; s += 16) {
            floatx4 v[16];
#pragma unroll
            for (int i = 0; i < 16; ++i)
                v[i] = *reinterpret_cast<const floatx4*>(
                    partial + static_cast<size_t>(min(s + i, slices - 1)) * stride + 4 * idx);
#pragma unroll
            for (int i = 0; i < 16; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) mx[e] = fmaxf(mx[e], v[i][e]);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float sc = mx[e] / 127.0f;
            inv[e] = sc > 0.0f ? 1.0f / sc : 0.0f;
            if (blockIdx.y == 0) scale[c + e] = sc;
        }
    }
    const int r0 = blockIdx.y * span, r1 = min(rows, r0 + span);
    for (int r = r0; r < r1; r += kQuantRound) {
        Floats4 x[kQuantRound];
#pragma unroll
        for (int u = 0; u < kQuantRound; ++u)
            x[u] = *reinterpret_cast<const Floats4*>(B + static_cast<size_t>(min(r + u, r1 - 1)) * cols + c);
#pragma unroll
        for (int u = 0; u < kQuantRound; ++u) {
            if (r + u >= r1) break;
            uint32_t w = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                w |= (static_cast<uint32_t>(quantize_one(x[u].v[e], inv[e])) & 0xffu) << (8 * e);
            __builtin_memcpy(q + static_cast<size_t>(r + u) * cols + c, &w, 4);
        }
    }
}

// scale and inv of every column from the slices' maxima, a wave per 16
// columns: lane 16 p + e takes every fourth slice from p of column e.
__global__ __launch_bounds__(kThreads) void scale_kernel(int cols, int stride, int slices,
                                                         const float* partial, float* scale,
                                                         float* inv) {
    const int lane = threadIdx.x % kWave, part = lane / 16;
    const int i = (blockIdx.x * (kThreads / kWave) + threadIdx.x / kWave) * 16 + lane % 16;
    const int at = min(i, stride - 1);
    float mx = 0.0f;
    for (int s = part; s < slices; s += 64) {
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u)
            v[u] = partial[static_cast<size_t>(min(s + 4 * u, slices - 1)) * stride + at];
#pragma unroll
        for (int u = 0; u < 16; ++u) mx = fmaxf(mx, v[u]);
    }
    mx = max32(max16(mx));
    if (part != 0 || i >= stride) return;
    const int c = cols < 4 ? i : column_group(i / 4, cols) + i % 4;
    const float sc = mx / 127.0f;
    scale[c] = sc;
    inv[c] = sc > 0.0f ? 1.0f / sc : 0.0f;
}

// The rows of a large matrix, read in address order by the whole grid: four
// consecutive elements of one row per thread and step (V4: cols % 4 == 0, B
// 16-byte and q 4-byte aligned), else one.
template <bool V4>
__global__ __launch_bounds__(kThreads) void quantize_flat_kernel(int total, int cols, const float* B,
                                                                 const float* inv, int8_t* q) {
    if constexpr (V4) {
        const int quads = total / 4;
        for (int i = blockIdx.x * kThreads + threadIdx.x; i < quads; i += gridDim.x * kThreads) {
            const int c = (4 * i) % cols;
            const float4 b = reinterpret_cast<const float4*>(B)[i];
            const float4 s = *reinterpret_cast<const float4*>(inv + c);
            reinterpret_cast<uint32_t*>(q)[i] =
                (static_cast<uint32_t>(quantize_one(b.x, s.x)) & 0xffu) |
                (static_cast<uint32_t>(quantize_one(b.y, s.y)) & 0xffu) << 8 |
                (static_cast<uint32_t>(quantize_one(b.z, s.z)) & 0xffu) << 16 |
                (static_cast<uint32_t>(quantize_one(b.w, s.w)) & 0xffu) << 24;
        }
    } else {
        for (int i = blockIdx.x * kThreads + threadIdx.x; i < total; i += gridDim.x * kThreads)
            q[i] = static_cast<int8_t>(quantize_one(B[i], inv[i % cols]));
    }
}

// Fewer than four columns of a few rows: one thread per column does it all.
__global__ __launch_bounds__(kThreads) void quantize_narrow_kernel(int rows, int cols, const float* B,
                                                                   int8_t* q, float* scale) {
    const int c = threadIdx.x;
    if (c >= cols) return;
    float mx = 0.0f;
    for (int r = 0; r < rows; ++r) mx = fmaxf(mx, fabsf(B[static_cast<size_t>(r) * cols + c]));
    const float sc = mx / 127.0f, inv = sc > 0.0f ? 1.0f / sc : 0.0f;
    scale[c] = sc;
    for (int r = 0; r < rows; ++r)
        q[static_cast<size_t>(r) * cols + c] =
            static_cast<int8_t>(quantize_one(B[static_cast<size_t>(r) * cols + c], inv));
}

__global__ __launch_bounds__(kThreads) void dequantize_kernel(int total, int cols,
                                                              const int8_t* q, const float* scale,
                                                              float* out) {
    for (int i = blockIdx.x * kThreads + threadIdx.x; i < total; i += gridDim.x * kThreads)
        out[i] = static_cast<float>(q[i]) * scale[i % cols];
}

int grid_for(size_t count) {
    const size_t blocks = (count + kThreads - 1) / kThreads;
    const size_t cap = static_cast<size_t>(cu_count()) * 16;
    return static_cast<int>(blocks < cap ? (blocks ? blocks : 1) : cap);
}

}  // namespace

template <class BT>
void run_naive(const MatmulArgs& a) {
    const dim3 grid(ceil_div(a.n, 64), ceil_div(a.m, 4));
    hipLaunchKernelGGL((naive_kernel<BT>), grid, dim3(kThreads), 0, a.stream, a.m, a.n, a.k, a.A,
                       static_cast<const BT*>(a.B), a.scale, a.C, a.accumulate ? 1 : 0);
}

template void run_naive<float>(const MatmulArgs&);
template void run_naive<int8_t>(const MatmulArgs&);

void run_reduce_slices(int m, int n, int slices, const float* partial, const float* scale,
                       float* C, bool accumulate, hipStream_t stream, float* ssq) {
    const int mn = m * n;
    hipLaunchKernelGGL(reduce_slices_kernel, dim3(ceil_div(mn, kThreads)), dim3(kThreads), 0,
                       stream, mn, n, slices, partial, scale, C, accumulate ? 1 : 0,
                       n % kSsqChunk == 0 ? ssq : nullptr);
}

// The read ceiling: 1024 workgroups, 16 loads in flight per thread, each
// workgroup on one contiguous chunk -- the fastest shape of the floor
// study's sweep over a 600 MiB buffer (6.95-6.98 TB/s against 5.1-5.4 for
// a 2048-workgroup grid stride with 8 loads in flight).
void run_stream_read(const void* buf, std::size_t bytes, uint32_t* sink, hipStream_t stream) {
    const std::size_t per = static_cast<std::size_t>(kThreads) * 16 * 16;
    const int blocks = static_cast<int>(std::max<std::size_t>(
        1, std::min<std::size_t>(1024, (bytes + per - 1) / per)));
    run_probe_read(buf, bytes, blocks, 16, true, sink, stream);
}

void run_rmsnorm_rows(int m, int k, const float* A, const float* w, float* out,
                      hipStream_t stream) {
    hipLaunchKernelGGL(k <= 4 * kThreads ? rmsnorm_rows_kernel<4> : rmsnorm_rows_kernel<16>, dim3(m),
                       dim3(kThreads), 0, stream, k, A, w, out);
}

void run_fill_zero(float* p, size_t count, hipStream_t stream) {
    hipLaunchKernelGGL(fill_zero_kernel, dim3(grid_for(count)), dim3(kThreads), 0, stream, p,
                       count);
}

// Past kQuantSmall values (kQuantLarge where the columns' maxima come in few
// slices) the scales get a launch of their own and the rows are read in
// address order; up to it the quantising workgroups form them. us, two
// launches / three: 1000 x 1001 9.5 / 11.2, 300 x 11000 (19 slices) 10.4 /
// 11.5, 11008 x 257 (256 slices) 19.5 / 15.7, 4096 x 11008 81 / 75.6 (79
// before). Tall matrices go the same way once a slice of a workgroup per CU is
// deeper than kQuantDeep rows, which few of its threads then walk (two launches
// / three, with the calls' host work: 12000 x 32 17 / 19, 16000 x 64 18.7 /
// 18.8, 32768 x 64 25 / 19, 131072 x 16 59 / 18, 500000 x 4 187 / 30). So do
// fewer than four columns past kQuantNarrow rows (a thread a column / three;
// on the card alone 16 x 3 3.2 / 5.2, 64 x 3 8 / 5.4; 300 x 1 57 / 16, 20000 x 3
// 3500 / 22).
constexpr size_t kQuantSmall = size_t{1} << 21, kQuantLarge = size_t{1} << 23;
constexpr int kQuantFewSlices = 32, kQuantDeep = 4 * kQuantRound, kQuantNarrow = 32;

void run_quantize_q8(int rows, int cols, const float* B, int8_t* q, float* scale,
                     hipStream_t stream) {
    if (rows == 0) {
        run_fill_zero(scale, cols, stream);
        return;
    }
    if (cols < 4 && rows <= kQuantNarrow) {
        hipLaunchKernelGGL(quantize_narrow_kernel, dim3(1), dim3(kThreads), 0, stream, rows, cols, B,
                           q, scale);
        return;
    }
    const int stride = cols < 4 ? cols : ceil_div(cols, 4) * 4;
    const int tiles = ceil_div(stride, 4 * kThreads);
    // Workgroups towards `per_cu` a CU, each with at least one round of rows.
    auto slabs = [&](int per_cu, int* span) {
        const int want = ceil_div(static_cast<long long>(per_cu) * cu_count(), tiles);
        const int n = std::max(1, std::min(want, ceil_div(rows, kQuantRound)));
        *span = ceil_div(rows, n);
        return ceil_div(rows, *span);
    };
    const size_t total = static_cast<size_t>(rows) * cols;
    int span_max = 0, span = 0;
    int slices = slabs(1, &span_max);
    const bool large = total > kQuantLarge || (total > kQuantSmall && slices > kQuantFewSlices) ||
                       span_max > kQuantDeep || cols < 4;
    if (large) slices = slabs(4, &span_max);
    const int parts = slabs(2, &span);
    float* partial = scratch(kQuant, static_cast<size_t>(slices) * stride + stride);
    hipLaunchKernelGGL(cols < 4 ? colmax_kernel<1> : colmax_kernel<4>, dim3(tiles, slices),
                       dim3(kThreads), 0, stream, rows, cols, span_max, stride, B, partial);
    if (!large) {
        hipLaunchKernelGGL(quantize_kernel, dim3(tiles, parts), dim3(kThreads), 0, stream, rows,
                           cols, span, stride, slices, B, partial, scale, q);
        return;
    }
    float* inv = partial + static_cast<size_t>(slices) * stride;
    hipLaunchKernelGGL(scale_kernel, dim3(ceil_div(stride, 64)), dim3(kThreads), 0, stream, cols,
                       stride, slices, partial, scale, inv);
    const bool v4 = cols % 4 == 0 && reinterpret_cast<uintptr_t>(B) % 16 == 0 &&
                    reinterpret_cast<uintptr_t>(q) % 4 == 0;
    if (v4) {
        hipLaunchKernelGGL(quantize_flat_kernel<true>, dim3(grid_for(total / 4)), dim3(kThreads), 0,
                           stream, static_cast<int>(total), cols, B, inv, q);
    } else {
        hipLaunchKernelGGL(quantize_flat_kernel<false>, dim3(grid_for(total)), dim3(kThreads), 0,
                           stream, static_cast<int>(total), cols, B, inv, q);
    }
}

void run_dequantize_q8(int rows, int cols, const int8_t* q, const float* scale, float* out,
                       hipStream_t stream) {
    const size_t total = static_cast<size_t>(rows) * cols;
    if (total)
        hipLaunchKernelGGL(dequantize_kernel, dim3(grid_for(total)), dim3(kThreads), 0, stream,
                           static_cast<int>(total), cols, q, scale, out);
}

}  // namespace em
