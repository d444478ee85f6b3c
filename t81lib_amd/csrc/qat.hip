// t81lib_amd/csrc/qat.hip -- the weight side of quantization-aware training
// (t81/nn/linear.py:72-99, t81/qat.py:12-46): scale, ternarized weight, surrogate gradient.
//
// HBM-bound passes over the weight.  As separate tensor operations these were ~25 passes
// (4096 x 4096 float32, forward + backward ~450 us); here one read for the scale, one read
// and write for the weight (with its packed trits and a bitmap for the backward), one read
// and write for its gradient.  Every operation keeps the rounding of the tensor expression it
// replaces: values are float, rounded to the weight's type T after each operation.
#include "pack_common.hpp"
#include "t81_device.hpp"
#include "t81_kernels.hpp"

#pragma clang fp contract(off)

namespace t81hip {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename T>
__device__ __forceinline__ float round_to(float v) {
    if constexpr (sizeof(T) == 4) return v;
    else if constexpr (__is_same(T, _Float16)) return static_cast<float>(static_cast<_Float16>(v));
    else return bf16_bits_to_float(bf16_bits_rne(v));
}

template <typename T>
__device__ __forceinline__ void store_as(T *p, float v) {
    if constexpr (sizeof(T) == 4) *p = v;
    else if constexpr (__is_same(T, _Float16)) *p = static_cast<_Float16>(v);
    else *p = bf16_bits_rne(v);
}

// 12 consecutive values (zeros past `limit`); whole runs of aligned rows as wide loads.
template <typename T, bool kVec>
__device__ __forceinline__ void load12(const T *src, int64_t c0, int64_t limit, float (&v)[12]) {
    if (kVec && c0 + 12 <= limit) {
        if constexpr (sizeof(T) == 4) {
            const f32x4 *p = reinterpret_cast<const f32x4 *>(src + c0);
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const f32x4 x = p[i];
#pragma unroll
                for (int j = 0; j < 4; ++j) v[4 * i + j] = x[j];
            }
        } else {
            const uint2 *p = reinterpret_cast<const uint2 *>(src + c0);
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const uint2 x = p[i];
                v[4 * i] = from_bits16<T>(x.x & 0xFFFFu);
                v[4 * i + 1] = from_bits16<T>(x.x >> 16);
                v[4 * i + 2] = from_bits16<T>(x.y & 0xFFFFu);
                v[4 * i + 3] = from_bits16<T>(x.y >> 16);
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < 12; ++i) v[i] = c0 + i < limit ? load_as_float<T>(src + c0 + i) : 0.0f;
    }
}

template <typename T, bool kVec>
__device__ __forceinline__ void store12(T *dst, int64_t c0, int64_t limit, const float (&v)[12]) {
    if (kVec && c0 + 12 <= limit) {
        if constexpr (sizeof(T) == 4) {
            f32x4 *p = reinterpret_cast<f32x4 *>(dst + c0);
#pragma unroll
            for (int i = 0; i < 3; ++i)
                p[i] = f32x4{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
        } else {
            T t[12];
#pragma unroll
            for (int i = 0; i < 12; ++i) store_as<T>(t + i, v[i]);
            uint2 *p = reinterpret_cast<uint2 *>(dst + c0);
#pragma unroll
            for (int i = 0; i < 3; ++i) __builtin_memcpy(p + i, t + 4 * i, 8);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 12; ++i)
            if (c0 + i < limit) store_as<T>(dst + c0 + i, v[i]);
    }
}

// max |w| as the bits of a non-negative float, whose order is the integers'; any NaN is
// larger than every number, so it is the result.
constexpr int kMaxBlocks = 1024;

__device__ __forceinline__ uint32_t block_max(uint32_t m) {
    __shared__ uint32_t part[4];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const uint32_t o = __shfl_xor(m, off, 64);
        m = o > m ? o : m;
    }
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) m = part[i] > m ? part[i] : m;
    return m;
}

template <typename T, bool kVec>
__global__ __launch_bounds__(256) void abs_max_kernel(const T *__restrict__ w, int64_t count,
                                                      uint32_t *__restrict__ part) {
    constexpr int V = kVec ? 16 / sizeof(T) : 1;
    const int64_t step = static_cast<int64_t>(gridDim.x) * 256 * V;
    uint32_t m = 0;
    int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * V;
    if constexpr (kVec) {
        auto fold = [&](const uint4 &x) {
            const uint32_t d[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if constexpr (sizeof(T) == 4) {
                    const uint32_t b = d[j] & 0x7FFFFFFFu;
                    m = b > m ? b : m;
                } else {
                    const uint32_t a = __float_as_uint(fabsf(from_bits16<T>(d[j] & 0xFFFFu)));
                    const uint32_t b = __float_as_uint(fabsf(from_bits16<T>(d[j] >> 16)));
                    m = a > m ? a : m;
                    m = b > m ? b : m;
                }
            }
        };
        // four loads in flight per lane
        for (; i + 3 * step + V <= count; i += 4 * step) {
            uint4 x[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) x[j] = *reinterpret_cast<const uint4 *>(w + i + j * step);
#pragma unroll
            for (int j = 0; j < 4; ++j) fold(x[j]);
        }
        for (; i + V <= count; i += step) fold(*reinterpret_cast<const uint4 *>(w + i));
    }
    for (; i < count; i += step)
        for (int64_t j = i; j < count && j < i + V; ++j) {
            const uint32_t b = __float_as_uint(fabsf(load_as_float<T>(w + j)));
            m = b > m ? b : m;
        }
    m = block_max(m);
    if (threadIdx.x == 0) part[blockIdx.x] = m;
}

// s = max(max |w|, 1e-6), moved 1 % of the way from `previous` when that is given.
template <typename T>
__global__ __launch_bounds__(256) void scale_kernel(const uint32_t *__restrict__ part, int blocks,
                                                    const float *__restrict__ previous,
                                                    float *__restrict__ scale) {
    uint32_t m = 0;
    for (int i = threadIdx.x; i < blocks; i += 256) m = part[i] > m ? part[i] : m;
    m = block_max(m);
    if (threadIdx.x != 0) return;
    const float a = __uint_as_float(m);
    float s = round_to<T>(a < 1e-6f ? 1e-6f : a);  // (a NaN stays)
    if (previous != nullptr) {
        const float old = *previous * 0.99f;
        const float now = s * 0.01f;
        s = old + now;
        s = s < 1e-6f ? 1e-6f : s;
    }
    *scale = s;
}

// One thread per 12 weights of a row (a packed dword): u = w / s, its trit q (sign of u where
// |u| >= thr after a clamp to [-1, 1], NaN 0), wq = q * s, the packed trits, and bit i of
// inner where the surrogate's slope is not zero: neither u >= 0.5 nor u <= -0.5.
template <typename T, bool kVec>
__global__ __launch_bounds__(256) void qat_quantize_kernel(
    const T *__restrict__ w, const float *__restrict__ scale, float thr, T *__restrict__ wq,
    uint32_t *__restrict__ packed, uint16_t *__restrict__ inner, int64_t rows, int64_t cols,
    int64_t per_row) {
    const int64_t d = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (d >= rows * per_row) return;
    const int64_t r = d / per_row;
    const int64_t c0 = (d - r * per_row) * 12;
    const float s = round_to<T>(*scale);
    thr = round_to<T>(thr);  // (the comparison's scalar takes the tensor's type)
    float v[12];
    load12<T, kVec>(w + r * cols, c0, cols, v);
    uint32_t word = 0, bits = 0;
    int t[12];
#pragma unroll
    for (int i = 0; i < 12; ++i) {
        const float u = round_to<T>(v[i] / s);
        const float c = u < -1.0f ? -1.0f : (u > 1.0f ? 1.0f : u);
        const int q = fabsf(c) >= thr ? (c > 0.0f) - (c < 0.0f) : 0;
        if (c0 + i < cols && !(u >= 0.5f) && !(u <= -0.5f)) bits |= 1u << i;
        t[i] = c0 + i < cols ? q : 0;
        v[i] = round_to<T>(static_cast<float>(q) * s);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
        word |= static_cast<uint32_t>(13 + t[3 * j] + 3 * t[3 * j + 1] + 9 * t[3 * j + 2]) << (8 * j);
    store12<T, kVec>(wq + r * cols, c0, cols, v);
    packed[d] = word;
    inner[d] = static_cast<uint16_t>(bits);
}

// out = inner ? ((g * s) * 2) / s : 0 / s, each operation rounded to T.
template <typename T, bool kVec>
__global__ __launch_bounds__(256) void qat_weight_grad_kernel(
    const T *__restrict__ g, const float *__restrict__ scale, const uint16_t *__restrict__ inner,
    T *__restrict__ out, int64_t rows, int64_t cols, int64_t per_row) {
    const int64_t d = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (d >= rows * per_row) return;
    const int64_t r = d / per_row;
    const int64_t c0 = (d - r * per_row) * 12;
    const float s = round_to<T>(*scale);
    const uint32_t bits = inner[d];
    float v[12];
    load12<T, kVec>(g + r * cols, c0, cols, v);
#pragma unroll
    for (int i = 0; i < 12; ++i) {
        float y = round_to<T>(v[i] * s);
        y = (bits >> i) & 1u ? y : 0.0f;
        y = round_to<T>(y * 2.0f);
        v[i] = round_to<T>(y / s);
    }
    store12<T, kVec>(out + r * cols, c0, cols, v);
}

// Column sums of a row-major float32 matrix.  A block of four waves takes 256 columns (64: V =
// 1) of a run of rows, wave w rows w, w + 4, ... with four loads in flight, and adds its waves'
// sums; the runs' sums are added in order by a second kernel.  (1024 x 14336: tensor sum 53
// us, the two kernels 17.)
template <int V>
__global__ __launch_bounds__(256) void column_sum_kernel(const float *__restrict__ g,
                                                         float *__restrict__ out, int64_t rows,
                                                         int64_t cols, int64_t run) {
    __shared__ float part[4][64 * V];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int64_t c = (static_cast<int64_t>(blockIdx.x) * 64 + lane) * V;
    const int64_t r0 = static_cast<int64_t>(blockIdx.y) * run;
    const int64_t r1 = r0 + run < rows ? r0 + run : rows;
    float acc[4][V] = {};
    auto load = [&](int64_t r, float (&v)[V]) {
        if constexpr (V == 4) {
            const f32x4 x = *reinterpret_cast<const f32x4 *>(g + r * cols + c);
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = x[u];
        } else {
            v[0] = g[r * cols + c];
        }
    };
    if (c < cols) {
        int64_t r = r0 + wave;
        for (; r + 12 < r1; r += 16) {
            float v[4][V];
#pragma unroll
            for (int i = 0; i < 4; ++i) load(r + 4 * i, v[i]);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int u = 0; u < V; ++u) acc[i][u] += v[i][u];
        }
        for (; r < r1; r += 4) {
            float v[V];
            load(r, v);
#pragma unroll
            for (int u = 0; u < V; ++u) acc[0][u] += v[u];
        }
    }
#pragma unroll
    for (int u = 0; u < V; ++u)
        part[wave][lane * V + u] = (acc[0][u] + acc[1][u]) + (acc[2][u] + acc[3][u]);
    __syncthreads();
    for (int i = threadIdx.x; i < 64 * V; i += 256) {
        const int64_t col = static_cast<int64_t>(blockIdx.x) * 64 * V + i;
        if (col < cols)
            out[blockIdx.y * cols + col] = (part[0][i] + part[1][i]) + (part[2][i] + part[3][i]);
    }
}

__global__ __launch_bounds__(256) void column_sum_runs_kernel(const float *__restrict__ part,
                                                              float *__restrict__ out,
                                                              int64_t cols, int runs) {
    const int64_t c = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (c >= cols) return;
    float a = 0.0f;
    for (int r = 0; r < runs; r += 8) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = r + i < runs ? part[(r + i) * cols + c] : 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) a += v[i];
    }
    out[c] = a;
}

int64_t blocks_for(int64_t n) { return (n + 255) / 256; }

template <typename T>
hipError_t qat_scale_t(const void *w, int64_t count, const float *previous, float *scale,
                       uint32_t *scratch, hipStream_t s) {
    constexpr int V = 16 / sizeof(T);
    const bool vec = reinterpret_cast<uintptr_t>(w) % 16 == 0;
    int64_t blocks = blocks_for((count + V - 1) / V);
    if (blocks > kMaxBlocks) blocks = kMaxBlocks;
    auto kernel = vec ? abs_max_kernel<T, true> : abs_max_kernel<T, false>;
    kernel<<<dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s>>>(static_cast<const T *>(w),
                                                                     count, scratch);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    scale_kernel<T><<<dim3(1), dim3(256), 0, s>>>(scratch, static_cast<int>(blocks), previous,
                                                  scale);
    return hipGetLastError();
}

template <typename T>
hipError_t qat_quantize_t(const void *w, const float *scale, float thr, void *wq, uint8_t *packed,
                          uint16_t *inner, int64_t rows, int64_t cols, hipStream_t s) {
    const int64_t per_row = (cols + kTrits - 1) / kTrits * 4;
    const bool vec = cols % 4 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(wq) % 16 == 0;
    auto kernel = vec ? qat_quantize_kernel<T, true> : qat_quantize_kernel<T, false>;
    kernel<<<dim3(static_cast<unsigned>(blocks_for(rows * per_row))), dim3(256), 0, s>>>(
        static_cast<const T *>(w), scale, thr, static_cast<T *>(wq),
        reinterpret_cast<uint32_t *>(packed), inner, rows, cols, per_row);
    return hipGetLastError();
}

template <typename T>
hipError_t qat_weight_grad_t(const void *g, const float *scale, const uint16_t *inner, void *out,
                             int64_t rows, int64_t cols, hipStream_t s) {
    const int64_t per_row = (cols + kTrits - 1) / kTrits * 4;
    const bool vec = cols % 4 == 0 && reinterpret_cast<uintptr_t>(g) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(out) % 16 == 0;
    auto kernel = vec ? qat_weight_grad_kernel<T, true> : qat_weight_grad_kernel<T, false>;
    kernel<<<dim3(static_cast<unsigned>(blocks_for(rows * per_row))), dim3(256), 0, s>>>(
        static_cast<const T *>(g), scale, inner, static_cast<T *>(out), rows, cols, per_row);
    return hipGetLastError();
}

}  // namespace

// Rows per run: 64, more once there would be over 64 runs.
static int64_t column_sum_run(int64_t rows) {
    const int64_t run = (rows + 63) / 64;
    return run < 64 ? 64 : (run + 15) / 16 * 16;
}

int64_t column_sum_scratch_bytes(int64_t rows, int64_t cols) {
    const int64_t runs = (rows + column_sum_run(rows) - 1) / column_sum_run(rows);
    return runs > 1 ? runs * cols * 4 : 0;
}

hipError_t launch_column_sum(const float *g, float *out, int64_t rows, int64_t cols,
                             float *scratch, hipStream_t s) {
    if (cols == 0) return hipSuccess;
    const int64_t run = column_sum_run(rows);
    const int64_t runs = rows > 0 ? (rows + run - 1) / run : 1;
    float *part = runs > 1 ? scratch : out;
    const bool vec = cols % 4 == 0 && reinterpret_cast<uintptr_t>(g) % 16 == 0;
    const int64_t wide = vec ? 256 : 64;
    const dim3 grid(static_cast<unsigned>((cols + wide - 1) / wide), static_cast<unsigned>(runs));
    auto kernel = vec ? column_sum_kernel<4> : column_sum_kernel<1>;
    kernel<<<grid, dim3(256), 0, s>>>(g, part, rows, cols, run);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || runs == 1) return e;
    column_sum_runs_kernel<<<dim3(static_cast<unsigned>(blocks_for(cols))), dim3(256), 0, s>>>(
        part, out, cols, static_cast<int>(runs));
    return hipGetLastError();
}

hipError_t launch_qat_scale(const void *w, int dtype, int64_t count, const float *previous,
                            float *scale, uint32_t *scratch, hipStream_t s) {
    switch (dtype) {
        case kDtypeF32: return qat_scale_t<float>(w, count, previous, scale, scratch, s);
        case kDtypeBF16: return qat_scale_t<uint16_t>(w, count, previous, scale, scratch, s);
        default: return qat_scale_t<_Float16>(w, count, previous, scale, scratch, s);
    }
}

hipError_t launch_qat_quantize(const void *w, int dtype, const float *scale, float thr, void *wq,
                               uint8_t *packed, uint16_t *inner, int64_t rows, int64_t cols,
                               hipStream_t s) {
    if (rows == 0 || cols == 0) return hipSuccess;
    switch (dtype) {
        case kDtypeF32: return qat_quantize_t<float>(w, scale, thr, wq, packed, inner, rows, cols, s);
        case kDtypeBF16:
            return qat_quantize_t<uint16_t>(w, scale, thr, wq, packed, inner, rows, cols, s);
        default: return qat_quantize_t<_Float16>(w, scale, thr, wq, packed, inner, rows, cols, s);
    }
}

hipError_t launch_qat_weight_grad(const void *g, int dtype, const float *scale,
                                  const uint16_t *inner, void *out, int64_t rows, int64_t cols,
                                  hipStream_t s) {
    if (rows == 0 || cols == 0) return hipSuccess;
    switch (dtype) {
        case kDtypeF32: return qat_weight_grad_t<float>(g, scale, inner, out, rows, cols, s);
        case kDtypeBF16: return qat_weight_grad_t<uint16_t>(g, scale, inner, out, rows, cols, s);
        default: return qat_weight_grad_t<_Float16>(g, scale, inner, out, rows, cols, s);
    }
}

}  // namespace t81hip
