// t81lib_amd/csrc/tq.hip -- GGUF ternary block codecs: TQ1_0 and TQ2_0 (llama.cpp's
// ggml block_tq1_0 / block_tq2_0, 256 weights per block), as the reference writes and
// reads them in t81/gguf.py:518-663 and 1020-1069.
//
// One wavefront per block.  Quantize: d = max |v| over the block (NaN if any value is
// NaN), inv_d = 0 if d == 0 else 1 / d, trit of v * inv_d (threshold form
// |v| >= thr -> sign, else round half away from zero clipped to [-1, 1]), digit
// q = trit + 1; the scale is stored as IEEE half (round to nearest even).
//  TQ2_0 (66 B): byte a*32 + c holds the digits of elements a*128 + s*32 + c at
//   bits 2s (a < 2, s < 4, c < 32); then the half scale.
//  TQ1_0 (54 B): bytes 0..31 hold base-3 numbers of 5 digits (first weighted 81)
//   over elements i*32 + c, bytes 32..47 over 160 + i*16 + c, bytes 48..51 four
//   digits weighted 81, 27, 9, 3 over 240 + i*4 + c; a number v < 243 is stored as
//   (v * 256 + 242) / 243, so digit n reads back as ((uint8)(byte * 3^n) * 3) >> 8.
// All float arithmetic is float32 with separate roundings (no contraction), as numpy
// evaluates it.  Rows are zero-padded to whole blocks.  Dequantize writes with the
// non-temporal hint (every output byte is written once); rows of whole float4s into an
// aligned output as one float4 per lane.
#include <hip/hip_fp16.h>

#include <type_traits>

#include "t81_device.hpp"
#include "t81_kernels.hpp"

#pragma clang fp contract(off)

namespace t81hip {

namespace {

constexpr int kQK = 256;
constexpr int kTq1 = 34;
constexpr int kTq2 = 35;

__host__ __device__ constexpr int tq_bytes(int quant) { return quant == kTq1 ? 54 : 66; }

__device__ __forceinline__ int tq_trit(float v, int use_thr, float thr) {
    if (use_thr) {
        if (!(fabsf(v) >= thr)) return 0;
        return v > 0.0f ? 1 : (v < 0.0f ? -1 : 0);
    }
    if (v != v) return 0;
    float r = v >= 0.0f ? floorf(v + 0.5f) : ceilf(v - 0.5f);
    r = r > 1.0f ? 1.0f : (r < -1.0f ? -1.0f : r);
    return static_cast<int>(r);
}

// Between a wavefront's LDS writes and its reads of what other lanes wrote.  Its LDS operations
// complete in order; the fences keep the compiler from moving them (the barrier alone orders
// no memory).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Row of block b with nb blocks per row (a 64-bit division is a long sequence: 1.7 us of the
// dequantize's 17 at 8192 x 3072).
__device__ __forceinline__ int64_t block_row(int64_t b, int64_t nb) {
    if (((b | nb) >> 32) == 0)
        return static_cast<uint32_t>(b) / static_cast<uint32_t>(nb);
    return b / nb;
}

// Max over the wavefront (lane values >= 0 or NaN-free by construction).
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
    return v;
}

// Max of max(v, the value `ctrl` brings from another lane), without LDS.
template <int ctrl, int rows = 0xF>
__device__ __forceinline__ float dpp_max(float v) {
    const int o = __builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), ctrl, rows, 0xF,
                                              false);
    return fmaxf(v, __int_as_float(o));
}
__device__ __forceinline__ float wave_max_dpp(float v) {
    v = dpp_max<0xB1>(v);         // quad_perm 1 0 3 2
    v = dpp_max<0x4E>(v);         // quad_perm 2 3 0 1
    v = dpp_max<0x141>(v);        // row_half_mirror
    v = dpp_max<0x140>(v);        // row_mirror: every lane holds its row's max
    v = dpp_max<0x142, 0xA>(v);   // row_bcast 15 into rows 1 and 3
    v = dpp_max<0x143, 0xC>(v);   // row_bcast 31 into rows 2 and 3: lane 63 holds all
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// B = 4 consecutive blocks per wavefront (2 below 8192 blocks, where few wavefronts are in
// flight).  HBM-bound (4 bytes read per weight): B 16-byte loads are in flight per lane, and
// the rest is kept off their way.  Lane l holds weights
// 4 l .. 4 l + 3 of each block and writes their digits (trit + 1) as one dword to the
// wavefront's LDS slot; since a base-3 number of five digits stays below 243 and two-bit
// fields do not meet, an output dword (four bytes) is then formed from 4 or 5 such dwords
// with no carry between its bytes: 13 lanes (TQ1_0) or 16 (TQ2_0) per block, all the blocks
// at once.  Their payload bytes are contiguous and go out as dwords through
// LDS.  kVec: rows are 16-byte aligned runs of whole float4s, else element loads; columns past
// the row are zeros.  The slots are private to the wavefront (wave_lds_sync, no barrier).
// 8192 x 3072: TQ1_0 29.2 -> 25.0 us, TQ2_0 25.3 -> 21.3 against one block per wavefront with
// byte gathers; 8192 x 3008 (partial blocks) TQ1_0 63.7 -> 21.8, 8191 x 3071 64.6 -> 28.2
// against strided loads read twice (calls over eight tensors in turn; from a graph 8192 x 3072
// takes 21.7 and 21.2).
template <int Q, bool kVec, int B>
__global__ __launch_bounds__(256) void tq_quantize_vec_kernel(const float *__restrict__ src,
                                                              uint8_t *__restrict__ dst,
                                                              int64_t blocks, int64_t cols,
                                                              int64_t nb, float thr,
                                                              int use_thr) {
    static_assert(B % 2 == 0, "a wavefront's payload is whole dwords");
    constexpr int kDw = Q == kTq1 ? 13 : 16;           // digit dwords per block
    constexpr int kHalves = tq_bytes(Q) / 2;           // 16-bit words per block
    __shared__ uint32_t slots[4][B * 64];
    __shared__ __attribute__((aligned(4))) uint16_t outs[4][B * kHalves];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t blk0 = (static_cast<int64_t>(blockIdx.x) * 4 + wave) * B;
    if (blk0 >= blocks) return;  // whole wavefront
    const int n = blocks - blk0 < B ? static_cast<int>(blocks - blk0) : B;
    floatx4 x[B];
    int64_t r = block_row(blk0, nb), cb = blk0 - r * nb;
#pragma unroll
    for (int u = 0; u < B; ++u) {
        x[u] = floatx4{0.f, 0.f, 0.f, 0.f};
        const int64_t col = cb * kQK + 4 * lane;
        const float *p = src + r * cols + col;
        if (u < n) {
            if constexpr (kVec) {
                if (col < cols) x[u] = __builtin_nontemporal_load(reinterpret_cast<const floatx4 *>(p));
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (col + j < cols) x[u][j] = p[j];
            }
        }
        if (++cb == nb) cb = 0, ++r;
    }
    uint16_t *out = outs[wave];
#pragma unroll
    for (int u = 0; u < B; ++u) {
        float mx = 0.0f;
        bool nan = false;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float a = fabsf(x[u][j]);
            nan |= a != a;
            mx = fmaxf(mx, a);
        }
        mx = wave_max_dpp(mx);
        const float d = __builtin_amdgcn_ballot_w64(nan) != 0 ? __builtin_nanf("") : mx;
        const float inv_d = d == 0.0f ? 0.0f : 1.0f / d;
        uint32_t dig = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            dig |= static_cast<uint32_t>(tq_trit(x[u][j] * inv_d, use_thr, thr) + 1) << (8 * j);
        slots[wave][64 * u + lane] = dig;
        if (lane == u) out[kHalves * (u + 1) - 1] = __half_as_ushort(__float2half_rn(d));
    }
    wave_lds_sync();
    if (lane < B * kDw) {
        const int u = lane / kDw, o = lane - u * kDw;
        const uint32_t *sd = slots[wave] + 64 * u;
        uint32_t b = 0;
        if constexpr (Q == kTq2) {
#pragma unroll
            for (int s = 0; s < 4; ++s) b |= sd[32 * (o >> 3) + 8 * s + (o & 7)] << (2 * s);
        } else {
            // dwords 0-7: five digits 32 weights apart; 8-11: 16 apart from 160; 12: four
            // digits 4 apart from 240, weighted 81, 27, 9, 3
            const int first = o < 8 ? o : (o < 12 ? 40 + (o - 8) : 60);
            const int step = o < 8 ? 8 : (o < 12 ? 4 : 1);
            uint32_t v = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) v = v * 3u + sd[first + i * step];
            v = v * 3u + (o < 12 ? sd[first + 4 * step] : 0u);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                b |= ((((v >> (8 * j)) & 0xFFu) * 256u + 242u) / 243u) << (8 * j);
        }
        out[kHalves * u + 2 * o] = static_cast<uint16_t>(b);
        out[kHalves * u + 2 * o + 1] = static_cast<uint16_t>(b >> 16);
    }
    wave_lds_sync();
    // blk0 is a multiple of B and two blocks are whole dwords: dst + blk0 tq_bytes is 4-byte
    // aligned where dst is
    uint32_t *g = reinterpret_cast<uint32_t *>(dst + blk0 * tq_bytes(Q));
    const int halves = n * kHalves;
    for (int i = lane; i < halves / 2; i += 64)
        g[i] = out[2 * i] | static_cast<uint32_t>(out[2 * i + 1]) << 16;
    if (halves % 2 != 0 && lane == 0)
        reinterpret_cast<uint16_t *>(g)[halves - 1] = out[halves - 1];
}

template <int Q>
__global__ __launch_bounds__(256) void tq_quantize_kernel(const float *__restrict__ src,
                                                          uint8_t *__restrict__ dst,
                                                          int64_t rows, int64_t cols,
                                                          int64_t nb, float thr, int use_thr) {
    const int lane = threadIdx.x & 63;
    const int64_t blk =
        static_cast<int64_t>(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (blk >= rows * nb) return;  // whole wavefront
    const int64_t r = blk / nb;
    const int64_t col0 = (blk - r * nb) * kQK;
    const float *row = src + r * cols;
    auto at = [&](int j) -> float {
        const int64_t col = col0 + j;
        return col < cols ? row[col] : 0.0f;
    };

    float mx = 0.0f;
    bool nan = false;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const float a = fabsf(at(lane + 64 * u));
        nan |= a != a;
        mx = fmaxf(mx, a);
    }
    mx = wave_max(mx);
    const float d = __builtin_amdgcn_ballot_w64(nan) != 0 ? __builtin_nanf("") : mx;
    const float inv_d = d == 0.0f ? 0.0f : 1.0f / d;

    uint8_t *out = dst + blk * tq_bytes(Q);
    if constexpr (Q == kTq2) {
        const int a = lane >> 5;
        const int c = lane & 31;
        uint32_t b = 0;
#pragma unroll
        for (int s = 0; s < 4; ++s)
            b |= static_cast<uint32_t>(tq_trit(at(a * 128 + s * 32 + c) * inv_d, use_thr, thr) + 1)
                 << (2 * s);
        out[lane] = static_cast<uint8_t>(b);
    } else {
        if (lane < 52) {
            int first, stride, ndig;
            if (lane < 32) {
                first = lane, stride = 32, ndig = 5;
            } else if (lane < 48) {
                first = 160 + (lane - 32), stride = 16, ndig = 5;
            } else {
                first = 240 + (lane - 48), stride = 4, ndig = 4;
            }
            uint32_t v = 0;
#pragma unroll
            for (int i = 0; i < 5; ++i)
                if (i < ndig)
                    v = v * 3 + static_cast<uint32_t>(
                                    tq_trit(at(first + i * stride) * inv_d, use_thr, thr) + 1);
            if (ndig == 4) v *= 3;  // four digits weighted 81, 27, 9, 3
            out[lane] = static_cast<uint8_t>((v * 256u + 242u) / 243u);
        }
    }
    if (lane == 0) {
        const uint16_t h = __half_as_ushort(__float2half_rn(d));
        out[tq_bytes(Q) - 2] = static_cast<uint8_t>(h & 0xFFu);
        out[tq_bytes(Q) - 1] = static_cast<uint8_t>(h >> 8);
    }
}

// One wavefront per block.  Rows of whole float4s (cols a multiple of 4) into a 16-byte aligned
// output (kVec): lane l writes weights 4 l .. 4 l + 3 of its block with one non-temporal
// float4, past the row none (8192 x 3008 TQ1_0 28.4 -> 18.0 us against element stores).
// Else the block turns through LDS so that each store is 64 consecutive floats (8191 x 3071
// TQ1_0 64.5 -> 36.8).  Those four share a digit position: TQ2_0 bits 2s of four
// consecutive bytes; TQ1_0 digit n of four consecutive bytes (n = e / 32 below 160,
// (e - 160) / 16 below 240, (e - 240) / 4 after, e = 4 l).
template <int Q, bool kVec>
__global__ __launch_bounds__(256) void tq_dequantize_kernel(const uint8_t *__restrict__ src,
                                                                float *__restrict__ dst,
                                                                int64_t blocks, int64_t cols,
                                                                int64_t nb) {
    const int lane = threadIdx.x & 63;
    const int64_t blk =
        static_cast<int64_t>(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (blk >= blocks) return;
    const uint8_t *in = src + blk * tq_bytes(Q);
    const uint16_t h = static_cast<uint16_t>(in[tq_bytes(Q) - 2] | (in[tq_bytes(Q) - 1] << 8));
    const float d = __half2float(__ushort_as_half(h));
    const int e = 4 * lane;
    int digit[4];
    if constexpr (Q == kTq2) {
        const int base = (e >> 7) * 32 + (e & 31);
        const int sh = 2 * ((e >> 5) & 3);
#pragma unroll
        for (int j = 0; j < 4; ++j) digit[j] = (in[base + j] >> sh) & 3;
    } else {
        int base, n;
        if (e < 160) {
            base = e & 31, n = e >> 5;
        } else if (e < 240) {
            base = 32 + ((e - 160) & 15), n = (e - 160) >> 4;
        } else {
            base = 48, n = (e - 240) >> 2;
        }
        uint32_t p = 1;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (i < n) p *= 3;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t q = (static_cast<uint32_t>(in[base + j]) * p) & 0xFFu;
            digit[j] = static_cast<int>((q * 3u) >> 8);
        }
    }
    floatx4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = d * static_cast<float>(digit[j] - 1);
    if (kVec && cols == nb * kQK) {  // whole blocks: no row to find
        __builtin_nontemporal_store(o, reinterpret_cast<floatx4 *>(dst + blk * kQK + e));
        return;
    }
    const int64_t r = block_row(blk, nb);
    const int64_t col0 = (blk - r * nb) * kQK;
    float *row = dst + r * cols;
    if constexpr (kVec) {
        if (col0 + e < cols)
            __builtin_nontemporal_store(o, reinterpret_cast<floatx4 *>(row + col0 + e));
    } else {
        __shared__ __attribute__((aligned(16))) float turn[4][kQK];
        float *t = turn[threadIdx.x >> 6];
        *reinterpret_cast<floatx4 *>(t + e) = o;
        wave_lds_sync();
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t col = col0 + 64 * j + lane;
            if (col < cols) row[col] = t[64 * j + lane];
        }
    }
}

}  // namespace

hipError_t launch_tq_quantize(const float *src, uint8_t *dst, int64_t rows, int64_t cols,
                              float thr, int use_thr, int quant, hipStream_t s) {
    const int64_t nb = (cols + kQK - 1) / kQK;
    const int64_t blocks = rows * nb;
    if (blocks == 0) return hipSuccess;
    if (reinterpret_cast<uintptr_t>(dst) % 4 != 0) {  // dword stores of the payload
        const dim3 grid(static_cast<unsigned>((blocks + 3) / 4));
        auto kernel = quant == kTq2 ? tq_quantize_kernel<kTq2> : tq_quantize_kernel<kTq1>;
        kernel<<<grid, 256, 0, s>>>(src, dst, rows, cols, nb, thr, use_thr);
        return hipGetLastError();
    }
    const bool vec = cols % 4 == 0 && (reinterpret_cast<uintptr_t>(src) & 15u) == 0;
    const bool few = blocks < 8192;
    const int64_t per = few ? 8 : 16;
    const dim3 grid(static_cast<unsigned>((blocks + per - 1) / per));
    auto pick = [&](auto q) {
        constexpr int Q = decltype(q)::value;
        if (few) return vec ? tq_quantize_vec_kernel<Q, true, 2> : tq_quantize_vec_kernel<Q, false, 2>;
        return vec ? tq_quantize_vec_kernel<Q, true, 4> : tq_quantize_vec_kernel<Q, false, 4>;
    };
    auto kernel = quant == kTq2 ? pick(std::integral_constant<int, kTq2>())
                                : pick(std::integral_constant<int, kTq1>());
    kernel<<<grid, 256, 0, s>>>(src, dst, blocks, cols, nb, thr, use_thr);
    return hipGetLastError();
}

hipError_t launch_tq_dequantize(const uint8_t *src, float *dst, int64_t rows, int64_t cols,
                                int quant, hipStream_t s) {
    const int64_t nb = (cols + kQK - 1) / kQK;
    const int64_t blocks = rows * nb;
    if (blocks == 0) return hipSuccess;
    const dim3 grid(static_cast<unsigned>((blocks + 3) / 4));
    const bool vec = cols % 4 == 0 && (reinterpret_cast<uintptr_t>(dst) & 15u) == 0;
    auto kernel = quant == kTq2 ? (vec ? tq_dequantize_kernel<kTq2, true> : tq_dequantize_kernel<kTq2, false>)
                                : (vec ? tq_dequantize_kernel<kTq1, true> : tq_dequantize_kernel<kTq1, false>);
    kernel<<<grid, 256, 0, s>>>(src, dst, blocks, cols, nb);
    return hipGetLastError();
}

}  // namespace t81hip
