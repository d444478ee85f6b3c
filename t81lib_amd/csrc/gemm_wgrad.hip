// t81lib_amd/csrc/gemm_wgrad.hip -- the weight gradient's product of a training step:
//
//   C[n, k] = sum_m G[m, n] * X[m, k]        (float32, G: M x N, X: M x K, row-major)
//
// on the bf16 matrix cores.  Both operands are split into three bf16 planes that hold them
// exactly (x = hi + mid + lo, round to nearest), and six of the nine plane products are
// summed: hi hi, hi mid, mid hi, mid mid, hi lo, lo hi.  Of the three left out, mid lo and lo mid
// reach 2^-25 of a product each.  What bounds it is the matrix pipe: 12 M N K flops at the bf16
// rate, against 2 M N K at a float32 rate a tenth of it (2048 x 4096 x 4096: the float32 library
// product 479-550 us, this kernel 298 = 1.38 PFLOP/s, with the images 340; 7.1e-7 from 64 bits
// against 8.1e-7).
//
// Plane images, written by a first kernel per operand: pieces of 8 consecutive rows m of one
// column (16 bytes),
//   [32-column block][plane][m / 8][column of the block] x 16 bytes
// with rows up to a multiple of 16 and columns up to a multiple of 32 as zeros.  A fragment of
// v_mfma_f32_32x32x16_bf16 (32 columns x 16 rows m) is then 1 KB of consecutive bytes, in
// global memory as in LDS.
//
// The operands are multiplied by 2^16 first (and the sums by 2^-32 last): float32 values are
// multiples of 2^-149 and bf16 ones of 2^-133, so the planes then hold the smallest exactly too.
//
// Plane products overflow where float32 ones need not, with the signs of the residuals, and an
// infinity times a zero plane is NaN.  So the image kernels note whether they saw a value of
// 2^37 or more, an infinity or a NaN; below that no sum of fewer than 2^19 products reaches
// 2^126.  Operands with such a value are multiplied in float32 by a kernel of its own, launched
// last: of the two products the one that the note does not mean ends at once.
#include <type_traits>

#include "t81_device.hpp"
#include "t81_kernels.hpp"

namespace t81hip {

namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kGTile = 256;          // columns of X and of G per workgroup
constexpr int kGFrags = 48;          // 1 KB fragments per step: 2 x 8 blocks x 3 planes
constexpr int kGStageStride = 68;
constexpr uint32_t kGOob = 0x80000000u;
constexpr float kGScale = 65536.0f;
constexpr float kGUnscale = 1.0f / (kGScale * kGScale);
constexpr uint32_t kGLarge = 0x52000000u;  // bits of 2^37
constexpr int64_t kGMostM8 = 65535;        // rows / 8 (M < 2^19)

__global__ void wgrad_clear_kernel(uint32_t *flag) { *flag = 0u; }

// A thread takes one column's 8 rows: lanes read consecutive columns of each row and write
// 512-byte runs.
__global__ __launch_bounds__(256) void wgrad_image_kernel(const float *__restrict__ x,
                                                          uint8_t *__restrict__ out,
                                                          uint32_t *__restrict__ flag, int M,
                                                          int C, int M8) {
    const int c = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
    const int m8 = static_cast<int>(blockIdx.y);
    if (c >= (C + 31) / 32 * 32) return;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int m = 8 * m8 + i;
        v[i] = m < M && c < C ? x[static_cast<int64_t>(m) * C + c] : 0.0f;
    }
    bf16x8 pl[3];
    bool large = false;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        large |= (__float_as_uint(v[i]) & 0x7FFFFFFFu) >= kGLarge;
        const float y = v[i] * kGScale;
        pl[0][i] = static_cast<__bf16>(y);
        const float r = y - static_cast<float>(pl[0][i]);
        pl[1][i] = static_cast<__bf16>(r);
        pl[2][i] = static_cast<__bf16>(r - static_cast<float>(pl[1][i]));
    }
    if (large) *flag = 1u;  // (every writer writes the same)
    uint8_t *dst = out + (static_cast<int64_t>(c >> 5) * 3 * M8 + m8) * 512 + (c & 31) * 16;
#pragma unroll
    for (int p = 0; p < 3; ++p)
        *reinterpret_cast<u32x4 *>(dst + static_cast<int64_t>(p) * M8 * 512) =
            __builtin_bit_cast(u32x4, pl[p]);
}

// Four waves, one per SIMD, compute 256 columns k of X x 256 columns n of G: wave (wr, wc) owns
// 128 x 128, 4 x 4 blocks (A = X, B = G, so that a lane's four accumulators are consecutive k
// of one row n of C).  A step is 16 rows m: 48 KB of fragments, straight copies into one of two
// LDS buffers, and 24 chunks of four MFMAs (column block cb = g / 6 of G, plane pair g % 6).
// A fragments are read once per step, B fragments once per column block, ahead of their use;
// the barrier follows chunk 17, past which nothing reads this step's buffer: the last six
// chunks load the step after next into it and read the next step's first fragments.
__global__ __launch_bounds__(256) void gemm_wgrad_kernel(
    const uint8_t *__restrict__ xa, int64_t xa_bytes, const uint8_t *__restrict__ gb,
    int64_t gb_bytes, const uint32_t *__restrict__ flag, float *__restrict__ c, int N, int K,
    int M8, int sps, int nsplit, float *__restrict__ part) {
    __shared__ __attribute__((aligned(1024))) uint8_t xs0[kGFrags * 1024];
    __shared__ __attribute__((aligned(1024))) uint8_t xs1[kGFrags * 1024];
    static_assert(4 * 32 * kGStageStride * 4 <= kGFrags * 1024, "the staging fits a tile buffer");
    static_assert(2 * kGFrags * 1024 + 2048 <= kLdsDmaLimit, "LDS-load targets past 128 KiB");
    if (*flag != 0u) return;
    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, 1>;
    auto tile = [&](auto bufc) -> uint8_t * {
        if constexpr (decltype(bufc)::value == 0) return xs0;
        else return xs1;
    };
    constexpr int kWaitAll = waitcnt_vm<0>();
    constexpr int kWaitTile = waitcnt_vm<12>();  // all but the newest tile's loads

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave & 1, wc = wave >> 1;
    const int tiles_k = (K + kGTile - 1) / kGTile;
    const int tiles_n = (N + kGTile - 1) / kGTile;
    const int tiles = tiles_k * tiles_n;
    const int total = tiles * nsplit;
    const int steps = M8 / 2;
    const int grid = static_cast<int>(gridDim.x);
    const int b = static_cast<int>(blockIdx.x);
    // each XCD (workgroup index mod 8) takes a contiguous run of a round's items
    const int pos = grid % 8 == 0 ? (b & 7) * (grid >> 3) + (b >> 3) : b;

    for (int q = pos; q < total; q += grid) {
        const int item = __builtin_amdgcn_readfirstlane(q);
        const int sp = item / tiles;
        const int tt = item - sp * tiles;
        const int k0 = (tt % tiles_k) * kGTile;
        const int n0 = (tt / tiles_k) * kGTile;
        const int s_begin = sp * sps;
        const int s_end = s_begin + sps < steps ? s_begin + sps : steps;
        __syncthreads();  // every wave is past the previous item's staging

        int lane = tid & 63;
        asm volatile("" : "+v"(lane));
        const int r = lane & 31;
        const int h = lane >> 5;
        const uint32_t lane16 = static_cast<uint32_t>(lane) * 16u;
        const __amdgpu_buffer_rsrc_t asrc = uniform_rsrc(xa, xa_bytes);
        const __amdgpu_buffer_rsrc_t bsrc = uniform_rsrc(gb, gb_bytes);
        // load i of a wave: fragment f = 4 i + wave; f < 24 of X, block f / 3, plane f % 3
        uint32_t fbase[12];
#pragma unroll
        for (int i = 0; i < 12; ++i) {
            const int f = (4 * i + wave) % 24;
            const int blk = (i < 6 ? k0 : n0) / 32 + f / 3;
            const int lim = ((i < 6 ? K : N) + 31) / 32;
            fbase[i] = blk < lim ? static_cast<uint32_t>(blk * 3 + f % 3) *
                                       (static_cast<uint32_t>(M8) * 512u)
                                 : kGOob;
        }
        auto load_part = [&](int s, auto bufc, int i) {
            load_lds16(i < 6 ? asrc : bsrc, &tile(bufc)[1024 * (4 * i + wave)],
                       lane16 + (fbase[i] + static_cast<uint32_t>(s) * 1024u));
        };
        auto read_a = [&](auto bufc, int f) -> u32x4 {  // f = rb * 3 + plane
            return *reinterpret_cast<const u32x4 *>(&tile(bufc)[(12 * wr + f) * 1024 + lane16]);
        };
        auto read_b = [&](auto bufc, int cb, int p) -> u32x4 {
            return *reinterpret_cast<const u32x4 *>(
                &tile(bufc)[(24 + 12 * wc + 3 * cb + p) * 1024 + lane16]);
        };

        floatx16 acc[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

        u32x4 a0[12], a1[12], bq[2][3];
#pragma unroll
        for (int i = 0; i < 12; ++i) load_part(s_begin, B0(), i);
        if (s_begin + 1 < s_end) {
#pragma unroll
            for (int i = 0; i < 12; ++i) load_part(s_begin + 1, B1(), i);
            __builtin_amdgcn_s_waitcnt(kWaitTile);
        } else {
            __builtin_amdgcn_s_waitcnt(kWaitAll);
        }
        __syncthreads();
#pragma unroll
        for (int f = 0; f < 12; ++f) a0[f] = read_a(B0(), f);
#pragma unroll
        for (int p = 0; p < 3; ++p) bq[0][p] = read_b(B0(), 0, p);

        auto step_body = [&](int s, auto bufc, auto otherc, const u32x4 (&a)[12],
                             u32x4 (&an)[12]) {
            const bool more = s + 2 < s_end;
#pragma unroll
            for (int g = 0; g < 24; ++g) {
                const int cb = g / 6, pr = g % 6;
                // plane pairs: (0,0) (0,1) (1,0) (1,1) (0,2) (2,0)
                const int pa = pr == 2 || pr == 3 ? 1 : (pr == 5 ? 2 : 0);
                const int pb = pr == 1 || pr == 3 ? 1 : (pr == 4 ? 2 : 0);
                if (cb < 3 && pr < 3) bq[(cb + 1) % 2][pr] = read_b(bufc, cb + 1, pr);
                if (g >= 18) {
                    an[2 * (g - 18)] = read_a(otherc, 2 * (g - 18));
                    an[2 * (g - 18) + 1] = read_a(otherc, 2 * (g - 18) + 1);
                    if (pr < 3) bq[0][pr] = read_b(otherc, 0, pr);
                    if (more) {
                        load_part(s + 2, bufc, 2 * (g - 18));
                        load_part(s + 2, bufc, 2 * (g - 18) + 1);
                    }
                }
                const bf16x8 bb = __builtin_bit_cast(bf16x8, bq[cb % 2][pb]);
#pragma unroll
                for (int rb = 0; rb < 4; ++rb)
                    acc[rb][cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        __builtin_bit_cast(bf16x8, a[3 * rb + pa]), bb, acc[rb][cb], 0, 0, 0);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // MFMA
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // LDS read
                    __builtin_amdgcn_sched_group_barrier(0x006, 2, 0);   // VALU, SALU
                    __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);   // buffer load
                }
                __builtin_amdgcn_sched_barrier(0);
                if (g == 17) {
                    __builtin_amdgcn_s_waitcnt(kWaitAll);  // the next tile has landed
                    __syncthreads();
                }
            }
        };
        int s = s_begin;
        for (; s + 1 < s_end; s += 2) {
            step_body(s, B0(), B1(), a0, a1);
            step_body(s + 1, B1(), B0(), a1, a0);
        }
        if (s < s_end) step_body(s, B0(), B1(), a0, a1);
        // (the last steps' reads of the other buffer fetch unused bytes; no load is pending)
        __syncthreads();  // the staging below overwrites a tile that other waves read from

        const float al = nsplit > 1 ? 1.0f : kGUnscale;
        float *dst = nsplit > 1 ? part + static_cast<int64_t>(sp) * N * K : c;
        const bool vec4 = K % 4 == 0 && (reinterpret_cast<uintptr_t>(dst) & 15u) == 0;
        float *st = reinterpret_cast<float *>(xs0) + wave * (32 * kGStageStride);
        const int tq = lane >> 4;
        const int tc = 4 * (lane & 15);
#pragma unroll
        for (int ps = 0; ps < 8; ++ps) {
            const int cb = ps >> 1, rp = ps & 1;
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int a4 = 0; a4 < 4; ++a4)
                    *reinterpret_cast<float4 *>(&st[r * kGStageStride + 32 * j + 8 * a4 + 4 * h]) =
                        make_float4(acc[2 * rp + j][cb][4 * a4], acc[2 * rp + j][cb][4 * a4 + 1],
                                    acc[2 * rp + j][cb][4 * a4 + 2],
                                    acc[2 * rp + j][cb][4 * a4 + 3]);
            const int kc = k0 + 128 * wr + 64 * rp + tc;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int row = 4 * i + tq;
                const f32x4 t = *reinterpret_cast<const f32x4 *>(&st[row * kGStageStride + tc]);
                const f32x4 v = {al * t[0], al * t[1], al * t[2], al * t[3]};
                const int n = n0 + 128 * wc + 32 * cb + row;
                if (n >= N) continue;
                float *cr = dst + static_cast<int64_t>(n) * K;
                if (vec4 && kc + 3 < K) {
                    __builtin_nontemporal_store(v, reinterpret_cast<f32x4 *>(cr + kc));
                } else {
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (kc + u < K) cr[kc + u] = v[u];
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// The same sums in float32, straight from the operands: 128 x 128 tiles, a wave 64 columns k of
// X x 64 columns n of G as 2 x 2 blocks of v_mfma_f32_32x32x2_f32 (whose sums run as chains of
// fused multiply-adds, so that finite terms leave an infinity as it is), 16 rows m a step,
// double-buffered through registers.  Rows of LDS are 160 floats apart: the two halves of a
// wave read different banks.  Only for operands of large values: the float32 rate is a tenth
// of the bf16 one's (2048 x 4096 x 4096 728 us in all, 1623 x 3520 x 1015 214).
constexpr int kFTile = 128;
constexpr int kFStep = 16;
constexpr int kFStride = 160;

__global__ __launch_bounds__(256) void gemm_wgrad_f32_kernel(const float *__restrict__ x,
                                                             const float *__restrict__ g,
                                                             const uint32_t *__restrict__ flag,
                                                             float *__restrict__ c, int M, int N,
                                                             int K) {
    __shared__ float xs[2][kFStep][kFStride];
    __shared__ float gs[2][kFStep][kFStride];
    if (*flag == 0u) return;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wr = wave & 1, wc = wave >> 1;
    const int r = lane & 31;
    const int h = lane >> 5;
    const int col = tid & 127;  // of the tile, the column that this thread loads
    const int row = tid >> 7;   // ... and its rows row, row + 2, ...
    const int tiles_k = (K + kFTile - 1) / kFTile;
    const int total = tiles_k * ((N + kFTile - 1) / kFTile);
    const int steps = (M + kFStep - 1) / kFStep;
    for (int item = blockIdx.x; item < total; item += gridDim.x) {
        const int k0 = (item % tiles_k) * kFTile;
        const int n0 = (item / tiles_k) * kFTile;
        float rx[kFStep / 2], rg[kFStep / 2];
        auto load = [&](int s) {
#pragma unroll
            for (int i = 0; i < kFStep / 2; ++i) {
                const int m = kFStep * s + row + 2 * i;
                rx[i] = m < M && k0 + col < K ? x[static_cast<int64_t>(m) * K + k0 + col] : 0.0f;
                rg[i] = m < M && n0 + col < N ? g[static_cast<int64_t>(m) * N + n0 + col] : 0.0f;
            }
        };
        auto store = [&](int buf) {
#pragma unroll
            for (int i = 0; i < kFStep / 2; ++i) {
                xs[buf][row + 2 * i][col] = rx[i];
                gs[buf][row + 2 * i][col] = rg[i];
            }
        };
        floatx16 acc[2][2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
        // (the barrier that ends a step lets the buffer before it be refilled; the last one
        // covers the next item's first)
        load(0);
        store(0);
        __syncthreads();
        for (int s = 0; s < steps; ++s) {
            const int buf = s & 1;
            if (s + 1 < steps) load(s + 1);
#pragma unroll
            for (int m = 0; m < kFStep; m += 2) {
                float a[2], b[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    a[i] = xs[buf][m + h][64 * wr + 32 * i + r];
                    b[i] = gs[buf][m + h][64 * wc + 32 * i + r];
                }
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        acc[i][j] =
                            __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
            }
            if (s + 1 < steps) store(buf ^ 1);
            __syncthreads();
        }
        const bool vec4 = K % 4 == 0 && (reinterpret_cast<uintptr_t>(c) & 15u) == 0;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = n0 + 64 * wc + 32 * j + r;
            if (n >= N) continue;
            float *cr = c + static_cast<int64_t>(n) * K;
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int a4 = 0; a4 < 4; ++a4) {
                    const int k = k0 + 64 * wr + 32 * i + 8 * a4 + 4 * h;
                    if (vec4 && k + 3 < K) {
                        *reinterpret_cast<f32x4 *>(cr + k) =
                            f32x4{acc[i][j][4 * a4], acc[i][j][4 * a4 + 1], acc[i][j][4 * a4 + 2],
                                  acc[i][j][4 * a4 + 3]};
                    } else {
#pragma unroll
                        for (int u = 0; u < 4; ++u)
                            if (k + u < K) cr[k + u] = acc[i][j][4 * a4 + u];
                    }
                }
        }
    }
}

constexpr int64_t kWgradWsBytes = int64_t{1} << 30;

struct WgradPlan {
    int64_t m8 = 0, x_bytes = 0, g_bytes = 0;
    int64_t nsplit = 1, sps = 0;
    int64_t bytes = 0;  // 0: not taken
};

// Splits of M so that few tiles still fill the CUs, at least eight steps each.
WgradPlan wgrad_plan(int64_t m, int64_t n, int64_t k) {
    WgradPlan p;
    constexpr int64_t kMost = int64_t{1} << 24;
    if (m <= 0 || n <= 0 || k <= 0 || m > kMost || n > kMost || k > kMost) return p;
    p.m8 = (m + 15) / 16 * 2;
    p.x_bytes = (k + 31) / 32 * 3 * p.m8 * 512;
    p.g_bytes = (n + 31) / 32 * 3 * p.m8 * 512;
    const int64_t tiles = ((n + kGTile - 1) / kGTile) * ((k + kGTile - 1) / kGTile);
    const int64_t steps = p.m8 / 2;
    // (a grid's second dimension and 32-bit buffer offsets)
    if (p.m8 > kGMostM8 || p.x_bytes >= 0x40000000 || p.g_bytes >= 0x40000000 || tiles > (int64_t{1} << 24)) return p;
    int64_t ns = cu_count() / tiles;
    if (ns > steps / 8) ns = steps / 8;
    if (ns < 1) ns = 1;
    p.sps = (steps + ns - 1) / ns;
    p.nsplit = (steps + p.sps - 1) / p.sps;
    const int64_t bytes = 256 + p.x_bytes + p.g_bytes + (p.nsplit > 1 ? p.nsplit * n * k * 4 : 0);
    if (bytes <= kWgradWsBytes) p.bytes = bytes;
    return p;
}

}  // namespace

int64_t gemm_wgrad_workspace_bytes(int64_t m, int64_t n, int64_t k) {
    return wgrad_plan(m, n, k).bytes;
}

hipError_t launch_gemm_wgrad(const float *g, const float *x, float *c, int64_t m, int64_t n,
                             int64_t k, hipStream_t s, void *ws) {
    const WgradPlan p = wgrad_plan(m, n, k);
    uint32_t *flag = static_cast<uint32_t *>(ws);
    uint8_t *xa = static_cast<uint8_t *>(ws) + 256;
    uint8_t *gb = xa + p.x_bytes;
    float *part = reinterpret_cast<float *>(gb + p.g_bytes);
    wgrad_clear_kernel<<<dim3(1), dim3(1), 0, s>>>(flag);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    auto image = [&](const float *src, uint8_t *dst, int64_t cols) {
        const dim3 grid(static_cast<unsigned>(((cols + 31) / 32 * 32 + 255) / 256),
                        static_cast<unsigned>(p.m8));
        wgrad_image_kernel<<<grid, dim3(256), 0, s>>>(src, dst, flag, static_cast<int>(m),
                                                      static_cast<int>(cols),
                                                      static_cast<int>(p.m8));
        return hipGetLastError();
    };
    if ((e = image(x, xa, k)) != hipSuccess) return e;
    if ((e = image(g, gb, n)) != hipSuccess) return e;
    const int64_t items =
        ((n + kGTile - 1) / kGTile) * ((k + kGTile - 1) / kGTile) * p.nsplit;
    const int64_t cus = cu_count();
    const dim3 grid(static_cast<unsigned>(items < cus ? items : cus));
    gemm_wgrad_kernel<<<grid, dim3(256), 0, s>>>(
        xa, p.x_bytes, gb, p.g_bytes, flag, c, static_cast<int>(n), static_cast<int>(k),
        static_cast<int>(p.m8), static_cast<int>(p.sps), static_cast<int>(p.nsplit), part);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (p.nsplit > 1) {
        e = launch_planes_sum(part, c, n, k, static_cast<int>(p.nsplit), kGUnscale, s);
        if (e != hipSuccess) return e;
    }
    // (past a split's sum, which then has added nothing that counts)
    const int64_t f32_tiles = ((n + kFTile - 1) / kFTile) * ((k + kFTile - 1) / kFTile);
    gemm_wgrad_f32_kernel<<<dim3(static_cast<unsigned>(f32_tiles < 2 * cus ? f32_tiles : 2 * cus)),
                            dim3(256), 0, s>>>(x, g, flag, c, static_cast<int>(m),
                                               static_cast<int>(n), static_cast<int>(k));
    return hipGetLastError();
}

}  // namespace t81hip
