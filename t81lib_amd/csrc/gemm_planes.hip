// t81lib_amd/csrc/gemm_planes.hip -- K3 through an image of the activations' bf16 planes.
//
//   C[m, n] = alpha * sum_k X[m, k] * T[n, k] + beta * C[m, n] + bias[n]
//
// x is cut into P bf16 planes (P = 2: float32 as hi + lo, |x - hi - lo| <= 2^-17 |x|; P = 3:
// float32 exactly, but for digits below 2^-140; P = 1: bf16 as it is) by a first small kernel,
// and the product kernel accumulates every plane's products into the same accumulators (P = 3:
// hi's apart from the others'): each decoded weight fragment meets P planes before it is dropped,
// so the trit decode and the weight loads per MFMA are 1 / P of the bf16 kernel's.  What bounds
// it is the matrix pipe (2 P M N K flops).
//
// Plane image.  The planes are stored piece by piece (8 values of one token, 16 bytes), so a
// tile load is a straight copy into LDS and a B read is 64 consecutive pieces:
//   [32-token block][plane][k / 8][token of the block] x 16 bytes
// (the last block holds the tokens there are).  Values past K in the last piece are zeros,
// pieces past K and tokens past M are out-of-range loads, which read zeros: any K and any
// alignment of x.
#include <type_traits>

#include "t81_device.hpp"
#include "t81_kernels.hpp"

namespace t81hip {

namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kPRows = 512;          // weight rows per tile: four waves of 128
constexpr uint32_t kPOob = 0x80000000u;
constexpr int kPStageStride = 68;    // floats per staged output row: 64 columns + 4 pad

// Training's product applies a scale to each output that the tensor expression applies to the
// weights; with trits of one its sums would be 1 / scale larger and overflow where the
// expression's do not.  Its trits are therefore a power of two (2^-32 .. 1) that keeps every sum
// within half the expression's size (the other half: hi planes round up), and the rest of the
// scale (2..4, or a scale of 2 and more as it is) remains for the output.
__device__ __forceinline__ float scale_of_trits(const float *scale) {
    if (scale == nullptr) return 1.0f;
    const int e = static_cast<int>(__float_as_uint(*scale) >> 23 & 0xFFu) - 128;
    return __uint_as_float(static_cast<uint32_t>(127 + (e < -32 ? -32 : (e < 0 ? e : 0))) << 23);
}
// Turns the trits of ones that lut_fill wrote into that power of two (each thread the words it
// wrote itself).
__device__ __forceinline__ void lut_scale(uint8_t *lds, int tid, int nthreads, float size) {
    const uint32_t one = __float_as_uint(size) >> 16;
    uint32_t *words = reinterpret_cast<uint32_t *>(lds);
    for (int i = tid; i < kLutBytes / 4; i += nthreads) {
        const uint32_t w = words[i];
        words[i] = (w & 0x80008000u) | (w & 0x7FFFu ? one : 0u) | (w & 0x7FFF0000u ? one << 16 : 0u);
    }
}
__device__ __forceinline__ float scale_of_output(const float *scale) {
    return scale == nullptr ? 1.0f : *scale / scale_of_trits(scale);
}

// Training's mid and lo planes, whose sums are apart from hi's to the end, are stored times 2^7:
// digits then go down to 2^-140 (bf16's smallest value is 2^-133), and the largest value's mid
// plane, below 2^120, stays in range.
constexpr float kSmallPlanes = 128.0f;

// ---- the plane image ----
// A wave takes 8 tokens x 8 consecutive pieces: it reads 256 contiguous bytes of each token
// row (K values of ldx) and writes 128 contiguous bytes per piece and plane.
template <int P, bool kVec>
__global__ __launch_bounds__(256) void planes_kernel(
    const std::conditional_t<P == 1, __bf16, float> *__restrict__ x, uint8_t *__restrict__ out,
    int M, int64_t ldx, int K, int K8, int groups) {
    const int lane = threadIdx.x & 63;
    const int64_t wv = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    const int64_t tg = wv / groups;  // group of eight tokens
    const int64_t tok = 8 * tg + (lane & 7);
    const int c8 = 8 * static_cast<int>(wv - tg * groups) + (lane >> 3);
    if (tok >= M || c8 >= K8) return;
    const int k0 = 8 * c8;
    const auto *p = x + tok * ldx + k0;
    bf16x8 pl[P];
    float v[8];
    if constexpr (P == 1) {
        if (kVec && k0 + 8 <= K) {
            pl[0] = *reinterpret_cast<const bf16x8 *>(p);
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) pl[0][i] = k0 + i < K ? p[i] : static_cast<__bf16>(0.0f);
        }
    } else if (kVec && k0 + 8 <= K) {
        const float4 a = reinterpret_cast<const float4 *>(p)[0];
        const float4 b = reinterpret_cast<const float4 *>(p)[1];
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
        v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = k0 + i < K ? p[i] : 0.0f;
    }
    const int64_t blk = tok >> 5;
    const int nt = M - 32 * blk < 32 ? static_cast<int>(M - 32 * blk) : 32;
    uint8_t *dst = out + blk * (static_cast<int64_t>(P) * 512 * K8) +
                   static_cast<int64_t>(c8) * nt * 16 + (tok & 31) * 16;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        if constexpr (P == 2) {
            pl[0][i] = static_cast<__bf16>(v[i]);
            pl[1][i] = static_cast<__bf16>(v[i] - static_cast<float>(pl[0][i]));
        } else if constexpr (P == 3) {
            // x = hi + mid + lo (8 bits each, round to nearest; of |x| < 2^-117 the digits below
            // 2^-140 are rounded off); |x| past bf16's largest value rounds to it, not to
            // infinity, and an infinity or NaN is hi alone
            const uint32_t u = __float_as_uint(v[i]);
            const uint32_t mag = u & 0x7FFFFFFFu;
            const bool top = mag >= 0x7F7F8000u;
            uint32_t hb = mag >= 0x7F800000u ? u >> 16 : (u >> 16 & 0x8000u) | 0x7F7Fu;
            if (mag > 0x7F800000u) hb |= 0x40u;
            const uint16_t h16 = static_cast<uint16_t>(hb);
            pl[0][i] = top ? __builtin_bit_cast(__bf16, h16) : static_cast<__bf16>(v[i]);
            const float r = mag >= 0x7F800000u
                                ? 0.0f
                                : (v[i] - static_cast<float>(pl[0][i])) * kSmallPlanes;
            pl[1][i] = static_cast<__bf16>(r);
            pl[2][i] = static_cast<__bf16>(r - static_cast<float>(pl[1][i]));
        }
    }
#pragma unroll
    for (int q = 0; q < P; ++q)
        *reinterpret_cast<u32x4 *>(dst + q * (static_cast<int64_t>(K8) * nt * 16)) =
            __builtin_bit_cast(u32x4, pl[q]);
}

// ---- the product ----
// A workgroup of four waves (one per SIMD) computes 512 weight rows x 32 CB tokens of C^T,
// wave w rows 128 w .. of all the tokens: 4 x CB blocks of v_mfma_f32_32x32x16_bf16.  A half
// step is 3 P CB chunks of four MFMAs (one B fragment each, read three chunks ahead); the
// chunks carry the table reads and merges of the next half step's A fragments and the tile
// loads (global -> LDS, no registers).  Steps alternate between two tile buffers, which are
// separate LDS objects so that loads into one provably do not alias reads of the other.
// Items: (split, token tile, row tile), row tile fastest; a round of items is dealt so that
// each XCD (workgroup index mod 8) takes a contiguous run of them and its L2 sees few token
// tiles.  nsplit > 1: split sp runs limb pairs [sp sps, (sp + 1) sps) and writes raw sums to
// part + sp M N, which planes_sum_kernel adds in split order.
template <int P, int CB, bool kBeta>
__global__ __launch_bounds__(256) void gemm_planes_kernel(
    const uint8_t *__restrict__ xp, int64_t xp_bytes, const uint8_t *__restrict__ w,
    float *__restrict__ c, int M, int N, int pitch, int L, int K8, float alpha, float beta,
    const float *__restrict__ bias, int sps, int nsplit, float *__restrict__ part,
    const float *__restrict__ scale) {
    constexpr int RB = 4;
    constexpr int NCH = 3 * P * CB;             // chunks per half step
    constexpr int kFrags = 3 * P * CB;          // 1 KB fragments per tile
    constexpr int LPW = (kFrags + 3) / 4;       // tile loads per wave
    constexpr int kTileBytes = 4 * LPW * 1024;  // (spare loads land inside it)
    constexpr int kTok = 32 * CB;
    constexpr int NF = NCH >= 10 ? 8 : 4;       // chunks that read the table
    constexpr int FPC = 8 / NF;                 // weight dwords looked up per such chunk
    constexpr int kWaitW = waitcnt_vm<RB>();         // all but the newest fetch_w
    constexpr int kWaitTwo = waitcnt_vm<RB + LPW>(); // and all but the newest tile
    constexpr int kWaitAll = waitcnt_vm<0>();
    __shared__ __attribute__((aligned(1024))) uint8_t lut[kLutBytes];
    __shared__ __attribute__((aligned(1024))) uint8_t xs0[kTileBytes];
    __shared__ __attribute__((aligned(1024))) uint8_t xs1[kTileBytes];
    __shared__ __attribute__((aligned(16))) float stg[4 * 32 * kPStageStride];
    static_assert((2 * NCH) % 4 == 0, "two half steps turn the fragment ring whole rounds");
    static_assert(2048 + 2 * kTileBytes + 4 * 32 * kPStageStride * 4 + 1024 <= kLdsDmaLimit,
                  "LDS-load targets past 128 KiB");
    auto tile = [&](auto bufc) -> uint8_t * {
        if constexpr (decltype(bufc)::value == 0) return xs0;
        else return xs1;
    };
    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, 1>;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tiles_n = (N + kPRows - 1) / kPRows;
    const int tiles_m = (M + kTok - 1) / kTok;
    const int tiles = tiles_n * tiles_m;
    const int total = tiles * nsplit;
    const int all_pairs = (L + 1) / 2;
    const int grid = static_cast<int>(gridDim.x);
    const int b = static_cast<int>(blockIdx.x);
    const int pos = grid % 8 == 0 ? (b & 7) * (grid >> 3) + (b >> 3) : b;
    alpha *= scale_of_output(scale);
    lut_fill(lut, tid, 256);  // published by the first item's barrier
    if (scale != nullptr) lut_scale(lut, tid, 256, scale_of_trits(scale));

    for (int q = pos; q < total; q += grid) {
        const int item = __builtin_amdgcn_readfirstlane(q);
        const int sp = item / tiles;
        const int tt = item - sp * tiles;
        const int tm = tt / tiles_n;
        const int nwg = (tt - tm * tiles_n) * kPRows;
        const int m0 = tm * kTok;
        const int t_begin = sp * sps;
        const int t_end = t_begin + sps < all_pairs ? t_begin + sps : all_pairs;
        __syncthreads();  // every wave is past the previous item's tile reads

        // the lane index passes through an empty asm once per item, so that what derives
        // from it is not kept live across the epilogue
        int lane = tid & 63;
        asm volatile("" : "+v"(lane));
        const int r = lane & 31;
        const int h = lane >> 5;

        // Weights: L limbs of rows `pitch` limbs apart; rows past N read zeros; a limb past L
        // (odd L) reads the next row's first limb or zeros, finite trits that meet zero
        // activations.
        const __amdgpu_buffer_rsrc_t wsrc =
            uniform_rsrc(w + static_cast<int64_t>(nwg) * pitch * kTrytes,
                       (static_cast<int64_t>(N - 1 - nwg) * pitch + L) * kTrytes);
        uint32_t woff[RB];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
            woff[rb] = (static_cast<uint32_t>(128 * wave + 32 * rb + r) * static_cast<uint32_t>(pitch) +
                        static_cast<uint32_t>(h)) * kTrytes;
        auto fetch_w = [&](int t, u32x4 (&dst)[RB]) {
            const uint32_t koff = static_cast<uint32_t>(t) * (2 * kTrytes);
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
                dst[rb] = __builtin_bit_cast(
                    u32x4, __builtin_amdgcn_raw_buffer_load_b128(wsrc, woff[rb] + koff, 0, 0));
        };

        // Tile load i of a wave: fragment f = 4 i + wave of the tile, token block f / 3P, plane
        // and j from f % 3P: lane (h, r) takes piece 12 t + 3 half + 6 h + j of token r.
        // Blocks and tokens past M, pieces past K and spare loads are out of range.
        const __amdgpu_buffer_rsrc_t xsrc = uniform_rsrc(xp, xp_bytes);
        const uint32_t lane16 = static_cast<uint32_t>(lane) * 16u;
        uint32_t loff[LPW];
        int piece[LPW];  // bytes between pieces
#pragma unroll
        for (int i = 0; i < LPW; ++i) {
            const int f = 4 * i + wave;
            const int cb = f / (3 * P), fr = f - cb * 3 * P;
            const int left = f < kFrags ? M - m0 - 32 * cb : 0;
            const int nt = left < 32 ? left : 32;
            piece[i] = 16 * nt;
            loff[i] = r < nt ? static_cast<uint32_t>(m0 / 32 + cb) * (P * 512u * K8) +
                                   static_cast<uint32_t>((fr / 3) * K8 + 6 * h + fr % 3) * piece[i] +
                                   16u * r
                             : kPOob;
        }
        auto load_tile_part = [&](int v, auto bufc, int i) {
            const int f = 4 * i + wave;
            const int k8 = 6 * v - 3 * (v & 1);  // 12 t + 3 half
            const uint32_t off = 6 * h < K8 - k8 - f % 3
                                     ? loff[i] + static_cast<uint32_t>(k8 * piece[i])
                                     : kPOob;
            load_lds16(xsrc, &tile(bufc)[1024 * (4 * i + wave)], off);
        };
        auto load_tile = [&](int v, auto bufc) {
#pragma unroll
            for (int i = 0; i < LPW; ++i) load_tile_part(v, bufc, i);
        };

        // P = 3: the hi plane's sums and the other two's are kept apart to the end, so the
        // small terms are not rounded at the size of the large ones
        constexpr int AC = P == 3 ? 2 * CB : CB;
        static_assert(AC <= 4, "256 accumulator registers");
        floatx16 acc[RB][AC];
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int j = 0; j < AC; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

        // B fragment g of a half step: plane and j from g / CB, token block g % CB.
        auto read_b = [&](auto bufc, int g) -> u32x4 {
            return *reinterpret_cast<const u32x4 *>(
                &tile(bufc)[((g % CB) * 3 * P + g / CB) * 1024 + lane16]);
        };
        auto table_fetch = [&](uint32_t wd, uint2 (&e)[4]) {
            const uint32_t w8 = wd << 3;
            e[0] = *reinterpret_cast<const uint2 *>(lut + kLutE + (w8 & 0xFFu));
            e[1] = *reinterpret_cast<const uint2 *>(lut + kLutF + ((w8 >> 8) & 0xFFu));
            e[2] = *reinterpret_cast<const uint2 *>(lut + kLutE + ((w8 >> 16) & 0xFFu));
            e[3] = *reinterpret_cast<const uint2 *>(lut + kLutF + (w8 >> 24));
        };
        auto table_merge = [&](const uint2 (&e)[4], uint32_t *out) {
            out[0] = e[0].x;
            out[1] = e[0].y | e[1].x;
            out[2] = e[1].y;
            out[3] = e[2].x;
            out[4] = e[2].y | e[3].x;
            out[5] = e[3].y;
        };

        u32x4 wcur[RB], wnxt[RB], wnn[RB];
        bf16x8 a0[RB][3], a1[RB][3];
        fetch_w(t_begin, wcur);
        load_tile(2 * t_begin, B0());
        if constexpr (CB == 2) {
            // a half-width step is too short to cover its tile loads: the second half
            // step's tile too (every step then loads the tile of the step after next)
            load_tile(2 * t_begin + 1, B1());
            fetch_w(t_begin + 1, wnxt);
            __builtin_amdgcn_s_waitcnt(kWaitTwo);
        } else {
            fetch_w(t_begin + 1, wnxt);
            __builtin_amdgcn_s_waitcnt(kWaitW);
        }
        __syncthreads();
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            uint32_t pairs[12];
            decode_dword(lut, wcur[rb][0], pairs);
            decode_dword(lut, wcur[rb][1], pairs + 6);
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const u32x4 raw = {pairs[4 * j], pairs[4 * j + 1], pairs[4 * j + 2],
                                   pairs[4 * j + 3]};
                a0[rb][j] = __builtin_bit_cast(bf16x8, raw);
            }
        }
        u32x4 bq[4];
        bq[0] = read_b(B0(), 0);
        bq[1] = read_b(B0(), 1);
        bq[2] = read_b(B0(), 2);

        // Half step v = 2 t + p from buffer bufc with the A fragments a; decodes the next
        // half step's into an (p = 0: the other half of wcur, p = 1: the first half of wnxt).
        // The barrier follows the last read of bufc (chunk NCH - 4): past it the next tile is
        // complete, and bufc may be refilled.
        auto step_body = [&](int v, auto pc, auto bufc, auto otherc, const bf16x8 (&a)[RB][3],
                             bf16x8 (&an)[RB][3]) {
            constexpr int p = decltype(pc)::value;
            uint2 e[3][FPC][4];
            uint32_t pairs[RB][12];
#pragma unroll
            for (int g = 0; g < NCH; ++g) {
                // (the fragment ring carries on across half steps: NCH may be 2 mod 4)
                constexpr int o = NCH * p;
                if (g + 3 < NCH) bq[(g + 3 + o) % 4] = read_b(bufc, g + 3);
                else bq[(g + 3 + o) % 4] = read_b(otherc, g + 3 - NCH);
                // eight weight dwords to decode, FPC a chunk, merged two chunks later
                if (g < NF) {
#pragma unroll
                    for (int f = FPC * g; f < FPC * g + FPC; ++f)
                        table_fetch(p == 0 ? wcur[f / 2][2 + f % 2] : wnxt[f / 2][f % 2],
                                    e[g % 3][f % FPC]);
                }
                if (g >= 2 && g < NF + 2) {
#pragma unroll
                    for (int f = FPC * (g - 2); f < FPC * (g - 2) + FPC; ++f)
                        table_merge(e[(g - 2) % 3][f % FPC], &pairs[f / 2][6 * (f % 2)]);
                }
                if constexpr (CB == 4) {
                    if (g < LPW) load_tile_part(v + 1, otherc, g);
                    if (p == 0 && g == LPW) fetch_w(v / 2 + 2, wnn);
                } else {
                    if (p == 0 && g == 0) fetch_w(v / 2 + 2, wnn);
                    if (g >= NCH - 3 && v + 2 < 2 * t_end) {
#pragma unroll
                        for (int i = 0; i < LPW; ++i)
                            if (i % 3 == g - (NCH - 3)) load_tile_part(v + 2, bufc, i);
                    }
                }
                const bf16x8 bb = __builtin_bit_cast(bf16x8, bq[(g + o) % 4]);
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) {
                    const int ai = g % CB + (P == 3 && g >= 3 * CB ? CB : 0);
                    acc[rb][ai] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        a[rb][(g / CB) % 3], bb, acc[rb][ai], 0, 0, 0);
                }
                if (g == NCH - 1) {
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                        for (int j = 0; j < 3; ++j) {
                            const u32x4 raw = {pairs[rb][4 * j], pairs[rb][4 * j + 1],
                                               pairs[rb][4 * j + 2], pairs[rb][4 * j + 3]};
                            an[rb][j] = __builtin_bit_cast(bf16x8, raw);
                        }
                }
                // each MFMA followed by a few of the chunk's other instructions: with one
                // wave per SIMD, issue is in order
#pragma unroll
                for (int k = 0; k < RB; ++k) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // MFMA
                    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);   // LDS read
                    __builtin_amdgcn_sched_group_barrier(0x006, 3, 0);   // VALU, SALU
                    __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);   // buffer load
                }
                __builtin_amdgcn_sched_barrier(0);
                if (g == NCH - 4) {
                    // the next tile's loads are older than a p = 0 step's weight loads; in a
                    // p = 1 step they are the newest
                    if constexpr (p == 0) __builtin_amdgcn_s_waitcnt(kWaitW);
                    else __builtin_amdgcn_s_waitcnt(kWaitAll);
                    __syncthreads();
                }
            }
        };
        for (int t = t_begin; t < t_end; ++t) {
            step_body(2 * t, B0(), B0(), B1(), a0, a1);
            step_body(2 * t + 1, B1(), B1(), B0(), a1, a0);
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                wcur[rb] = wnxt[rb];
                wnxt[rb] = wnn[rb];
            }
        }

        if constexpr (P == 3) {
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int j = 0; j < CB; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v)
                        acc[i][j][v] += acc[i][j + CB][v] * (1.0f / kSmallPlanes);
        }

        // ---- epilogue: through the wave's LDS region, 32 tokens x 64 rows at a time, so a
        // store covers four 256-byte runs of C ----
        float *cdst = nsplit > 1 ? part + static_cast<int64_t>(sp) * M * N : c;
        const bool raw = nsplit > 1;
        const float al = raw ? 1.0f : alpha;
        const float *bi = raw ? nullptr : bias;
        const bool vec4 = N % 4 == 0 && (reinterpret_cast<uintptr_t>(cdst) & 15u) == 0 &&
                          (reinterpret_cast<uintptr_t>(bi) & 15u) == 0;
        float *st = stg + wave * (32 * kPStageStride);
        const int tq = lane >> 4;
        const int tc = 4 * (lane & 15);
        auto c_pass = [&](int ps, f32x4 (&cv)[8]) {
            const int nb = nwg + 128 * wave + 64 * (ps & 1) + tc;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int m = m0 + 32 * (ps >> 1) + 4 * i + tq;
                cv[i] = f32x4{0.f, 0.f, 0.f, 0.f};
                if (vec4 && m < M && nb + 3 < N)
                    cv[i] = __builtin_nontemporal_load(
                        reinterpret_cast<const f32x4 *>(cdst + static_cast<int64_t>(m) * N + nb));
            }
        };
        f32x4 cva[8], cvb[8];
        if constexpr (kBeta) c_pass(0, cva);
#pragma unroll
        for (int ps = 0; ps < 2 * CB; ++ps) {
            const int cb = ps >> 1, rp = ps & 1;
            f32x4 (&cvc)[8] = ps % 2 == 0 ? cva : cvb;
            f32x4 (&cvn)[8] = ps % 2 == 0 ? cvb : cva;
            if constexpr (kBeta)
                if (ps + 1 < 2 * CB) c_pass(ps + 1, cvn);
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int a4 = 0; a4 < 4; ++a4)
                    *reinterpret_cast<float4 *>(&st[r * kPStageStride + 32 * j + 8 * a4 + 4 * h]) =
                        make_float4(acc[2 * rp + j][cb][4 * a4], acc[2 * rp + j][cb][4 * a4 + 1],
                                    acc[2 * rp + j][cb][4 * a4 + 2],
                                    acc[2 * rp + j][cb][4 * a4 + 3]);
            const int nb = nwg + 128 * wave + 64 * rp + tc;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int tok = 4 * i + tq;
                const float4 v = *reinterpret_cast<const float4 *>(&st[tok * kPStageStride + tc]);
                const int m = m0 + 32 * cb + tok;
                if (m >= M) continue;
                float *cr = cdst + static_cast<int64_t>(m) * N;
                f32x4 y = {al * v.x, al * v.y, al * v.z, al * v.w};
                if (vec4 && nb + 3 < N) {
                    if constexpr (kBeta) {
#pragma unroll
                        for (int u = 0; u < 4; ++u) y[u] += beta * cvc[i][u];
                    }
                    if (bi != nullptr) {
                        const f32x4 bv = *reinterpret_cast<const f32x4 *>(bi + nb);
#pragma unroll
                        for (int u = 0; u < 4; ++u) y[u] += bv[u];
                    }
                    __builtin_nontemporal_store(y, reinterpret_cast<f32x4 *>(cr + nb));
                } else {
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const int n = nb + u;
                        if (n < N) {
                            float t = y[u];
                            if constexpr (kBeta) t = t + beta * cr[n];
                            if (bi != nullptr) t = t + bi[n];
                            cr[n] = t;
                        }
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// C from the splits, added in split order, then alpha, beta and bias as above.
template <bool kVec>
__global__ __launch_bounds__(256) void planes_sum_kernel(const float *__restrict__ part,
                                                         float *__restrict__ c, int64_t M,
                                                         int64_t N, int nsplit, float alpha,
                                                         float beta,
                                                         const float *__restrict__ bias,
                                                         const float *__restrict__ scale) {
    alpha *= scale_of_output(scale);
    constexpr int V = kVec ? 4 : 1;
    const int64_t total = M * N;
    for (int64_t g = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * V; g < total;
         g += static_cast<int64_t>(gridDim.x) * 256 * V) {
        // eight splits in flight: few threads with many splits wait out each load otherwise
        using VT = std::conditional_t<kVec, f32x4, float>;
        VT a = {};
        for (int s0 = 0; s0 < nsplit; s0 += 8) {
            VT t[8];
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (s0 + i < nsplit)
                    t[i] = __builtin_nontemporal_load(
                        reinterpret_cast<const VT *>(part + (s0 + i) * total + g));
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (s0 + i < nsplit) a = s0 + i == 0 ? t[i] : a + t[i];
        }
        float acc[V];
        if constexpr (kVec) {
#pragma unroll
            for (int u = 0; u < V; ++u) acc[u] = a[u];
        } else {
            acc[0] = a;
        }
        const int64_t n = g % N;
        float y[V];
#pragma unroll
        for (int u = 0; u < V; ++u) {
            y[u] = alpha * acc[u];
            if (beta != 0.0f) y[u] = y[u] + beta * c[g + u];
            if (bias != nullptr) y[u] = y[u] + bias[n + u];
        }
        if constexpr (kVec) {
            const f32x4 yv = {y[0], y[1], y[2], y[3]};
            *reinterpret_cast<f32x4 *>(c + g) = yv;
        } else {
            c[g] = y[0];
        }
    }
}


// ---- the plan ----
// The plane image and the split partials fit kPlanesWsBytes (so every shape stays within the
// no-allocation entry's static scratch): tokens run in chunks, or K in parts, each part's
// product added to C.
constexpr int64_t kPlanesWsBytes = int64_t{64} << 20;
// three planes serve training, whose workspace comes from the caller's allocator
constexpr int64_t planes_ws_limit(int P) { return P == 3 ? int64_t{512} << 20 : kPlanesWsBytes; }

struct PlanesPlan {
    int cb = 0;                   // 32-token blocks per tile (4 or 2); 0: not taken
    int64_t rows = 0, count = 0;  // tokens per chunk (the last may hold fewer), chunks
    int64_t pairs = 0, parts = 1; // limb pairs per part of K, parts
    int64_t nsplit = 1, sps = 0;  // splits of a part, limb pairs per split
    int64_t bytes = 0;            // workspace of a chunk
};

int64_t planes_image_bytes(int P, int64_t rows, int64_t k) { return 2 * P * rows * ((k + 7) / 8 * 8); }
int64_t planes_part_offset(int P, int64_t rows, int64_t k) {
    return (planes_image_bytes(P, rows, k) + 255) / 256 * 256;
}

// Estimated microseconds of a chunk's product and split sum: rounds of items over the CUs,
// each its half steps plus an epilogue; a split's partials are written by the epilogues and
// read once (5.5 TB/s).  A half step of 128 tokens took 2.05 us and of 64 tokens 1.09 us at
// P = 2 (14336 -> 4096, M = 2048: 256 items of 150 half steps 314 us, of 300 narrow ones
// 334 us), 1.0 / 0.72 at P = 1, 1.6 (64 tokens) at P = 3.
float planes_cost(int P, int cb, int64_t tiles, int64_t ns, int64_t sps, int64_t rows, int64_t n) {
    const float step = cb == 4 ? (P == 1 ? 1.0f : 2.05f) : (P == 1 ? 0.72f : (P == 2 ? 1.09f : 1.6f));
    const int64_t cus = cu_count();
    const float rounds = static_cast<float>((tiles * ns + cus - 1) / cus);
    float t = 4.0f + rounds * (2.0f * sps * step + (cb == 4 ? 6.0f : 4.0f));
    if (ns > 1) t += 4.0f + static_cast<float>((ns + 1) * rows * n) * (4.0f / 5.5e6f);
    return t;
}

// The cheapest of: 128- or 64-token tiles, K whole or split so that the items fill one to
// three rounds of the CUs, and, where the image is too large, chunks of tokens or parts of K
// (14336 -> 4096 at M = 2048: two chunks 488 us, two parts 394).
PlanesPlan planes_plan(int P, int64_t m, int64_t n, int64_t k) {
    PlanesPlan best;
    const int64_t limit = planes_ws_limit(P);
    const int64_t L = (k + kTrits - 1) / kTrits;
    const int64_t all_pairs = (L + 1) / 2;
    if (m <= 0 || n <= 0 || k <= 0 || 32 * planes_image_bytes(P, 1, k) > limit ||
        n >= (int64_t{1} << 30) || m >= (int64_t{1} << 30) ||
        int64_t{kPRows} * L * kTrytes >= 0x7FFFFFFF)
        return best;
    const int64_t tiles_n = (n + kPRows - 1) / kPRows;
    const int64_t cus = cu_count();
    float best_t = 0.0f;
    const int64_t max_parts = planes_image_bytes(P, m, k) > limit ? 4 : 1;
    for (int64_t np = 1; np <= max_parts; ++np) {
        const int64_t pairs = (all_pairs + np - 1) / np;
        const int64_t parts = (all_pairs + pairs - 1) / pairs;
        const int64_t kp = parts == 1 ? k : 2 * kTrits * pairs;
        const int64_t per_tok = planes_image_bytes(P, 1, kp);
        for (int cb = P == 3 ? 2 : 4; cb >= 2; cb -= 2) {
            for (int fill = 0; fill <= 3; ++fill) {
                int64_t count = (m * per_tok + limit - 1) / limit;
                for (int tries = 0; tries < 4; ++tries, ++count) {
                    const int64_t rows = (m + count - 1) / count;
                    const int64_t tiles = tiles_n * ((rows + 32 * cb - 1) / (32 * cb));
                    int64_t ns = 1;
                    if (fill > 0) {
                        ns = fill * cus / tiles;
                        if (ns > pairs / 2) ns = pairs / 2;
                        if (ns < 2) break;
                    }
                    const int64_t sps = (pairs + ns - 1) / ns;
                    ns = (pairs + sps - 1) / sps;
                    if (tiles * ns >= (int64_t{1} << 30)) break;
                    const int64_t bytes = ns > 1
                                              ? planes_part_offset(P, rows, kp) + ns * rows * n * 4
                                              : planes_image_bytes(P, rows, kp);
                    if (bytes > limit) continue;
                    float t = planes_cost(P, cb, tiles, ns, sps, rows, n) * (count * parts);
                    // C read and written again by every part after the first
                    t += static_cast<float>((parts - 1) * m * n) * (8.0f / 4e6f);
                    if (best.cb == 0 || t < best_t) {
                        best_t = t;
                        best.cb = cb;
                        best.rows = rows;
                        best.count = count;
                        best.pairs = pairs;
                        best.parts = parts;
                        best.nsplit = ns;
                        best.sps = sps;
                        best.bytes = bytes;
                    }
                    break;
                }
            }
        }
    }
    return best;
}

template <int P>
hipError_t launch_planes(const void *x, const uint8_t *w, float *c, int64_t m, int64_t n,
                         int64_t k, float alpha, float beta, const float *bias, hipStream_t s,
                         void *ws, const float *scale = nullptr) {
    using XT = std::conditional_t<P == 1, __bf16, float>;
    const PlanesPlan plan = planes_plan(P, m, n, k);
    const int64_t L = (k + kTrits - 1) / kTrits;
    const int64_t kp = plan.parts == 1 ? k : 2 * kTrits * plan.pairs;  // of all parts but the last
    const bool vec = k % 8 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0;
    uint8_t *image = static_cast<uint8_t *>(ws);
    float *part = reinterpret_cast<float *>(image + planes_part_offset(P, plan.rows, kp));
    for (int64_t t0 = 0; t0 < m; t0 += plan.rows) {
        const int64_t rows = m - t0 < plan.rows ? m - t0 : plan.rows;
        float *cc = c + t0 * n;
        for (int64_t pt = 0; pt < plan.parts; ++pt) {
            const int64_t k0 = pt * kp;
            const int64_t kn = k - k0 < kp ? k - k0 : kp;
            const int64_t l0 = 2 * plan.pairs * pt;
            const int64_t ln = L - l0 < 2 * plan.pairs ? L - l0 : 2 * plan.pairs;
            const int K8 = static_cast<int>((kn + 7) / 8);
            const int groups = (K8 + 7) / 8;
            const float be = pt == 0 ? beta : 1.0f;
            const float *bi = pt == 0 ? bias : nullptr;
            const XT *xc = static_cast<const XT *>(x) + t0 * k + k0;
            const int64_t waves = (rows + 7) / 8 * groups;
            const dim3 pgrid(static_cast<unsigned>((waves + 3) / 4));
            auto prep = vec ? planes_kernel<P, true> : planes_kernel<P, false>;
            prep<<<pgrid, dim3(256), 0, s>>>(xc, image, static_cast<int>(rows), k,
                                             static_cast<int>(kn), K8, groups);
            hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
            const int64_t tiles =
                (n + kPRows - 1) / kPRows * ((rows + 32 * plan.cb - 1) / (32 * plan.cb));
            const int64_t part_pairs = (ln + 1) / 2;
            const int64_t ns = (part_pairs + plan.sps - 1) / plan.sps;
            const int64_t items = tiles * ns;
            const int64_t cus = cu_count();
            const dim3 grid(static_cast<unsigned>(items < cus ? items : cus));
            const bool add = be != 0.0f && ns == 1;  // (a split's sum applies beta)
            auto kernel = add ? gemm_planes_kernel<P, 2, true> : gemm_planes_kernel<P, 2, false>;
            if constexpr (P != 3) {
                if (plan.cb == 4)
                    kernel = add ? gemm_planes_kernel<P, 4, true> : gemm_planes_kernel<P, 4, false>;
            }
            kernel<<<grid, dim3(256), 0, s>>>(
                image, planes_image_bytes(P, rows, kn), w + l0 * kTrytes, cc,
                static_cast<int>(rows), static_cast<int>(n), static_cast<int>(L),
                static_cast<int>(ln), K8, alpha, be, bi, static_cast<int>(plan.sps),
                static_cast<int>(ns), part, scale);
            e = hipGetLastError();
            if (e != hipSuccess) return e;
            if (ns == 1) continue;
            const bool v4 = n % 4 == 0 && reinterpret_cast<uintptr_t>(cc) % 16 == 0;
            const int64_t threads = rows * n / (v4 ? 4 : 1);
            const int64_t blocks = (threads + 255) / 256 < 8192 ? (threads + 255) / 256 : 8192;
            auto sum = v4 ? planes_sum_kernel<true> : planes_sum_kernel<false>;
            sum<<<dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s>>>(
                part, cc, rows, n, static_cast<int>(ns), alpha, be, bi, scale);
            e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
    }
    return hipSuccess;
}

}  // namespace

// Where the planes are taken, against the eight-wave kernel (14336 -> 4096 at M = 1024 828 ->
// 223 us, 4096 -> 14336 at M = 100 / 512 103 -> 39 / 230 -> 99, at M = 33 / 64 33 -> 26 /
// 42 -> 32): past 32 tokens, of 33..64 only over 4 Mi weights or a K the vector loads do not
// take -- three launches cost 14-18 us whatever the size (1000 -> 1000 at 64 tokens 17.6 ->
// 18.5, at 65 24.6 -> 18.8; 3072 -> 3072 at 64 20.5 -> 18.6), and at 17..32 tokens the
// eight-wave kernel's 32-token tiles take 13-26 us (4096 -> 14336 at 32 25.4 -> 26.1, 4096 ->
// 4096 14.2 -> 18.5).  The size is never less than the two planes, 4 bytes a value, of the fewest
// equal token chunks, within the bound that the plan itself keeps (ceil(m / count) tokens pass
// it by up to one where that many just fit).
int64_t gemm_planes_workspace_bytes(int64_t m, int64_t n, int64_t k) {
    if (m <= 32) return 0;
    if (m <= 64 && k % 8 == 0 && (n >= (int64_t{1} << 30) || n * k < (int64_t{1} << 22))) return 0;
    const PlanesPlan plan = planes_plan(2, m, n, k);
    if (plan.cb == 0) return 0;
    const int64_t per_tok = planes_image_bytes(2, 1, k);
    const int64_t count = (m * per_tok + kPlanesWsBytes - 1) / kPlanesWsBytes;
    int64_t chunk = (m + count - 1) / count * per_tok;
    if (chunk > kPlanesWsBytes) chunk = kPlanesWsBytes;
    return plan.bytes > chunk ? plan.bytes : chunk;
}

hipError_t launch_gemm_planes(const float *x, const uint8_t *w, float *c, int64_t m, int64_t n,
                              int64_t k, float alpha, float beta, const float *bias,
                              hipStream_t s, void *ws) {
    return launch_planes<2>(x, w, c, m, n, k, alpha, beta, bias, s, ws);
}

int64_t gemm_plane_workspace_bytes(int64_t m, int64_t n, int64_t k) {
    return planes_plan(1, m, n, k).bytes;
}

hipError_t launch_gemm_plane(const void *x, const uint8_t *w, float *c, int64_t m, int64_t n,
                             int64_t k, float alpha, float beta, const float *bias,
                             hipStream_t s, void *ws) {
    return launch_planes<1>(x, w, c, m, n, k, alpha, beta, bias, s, ws);
}

// Training's product: three planes and a scale in device memory,
//   C[m, n] = *scale * sum_k X[m, k] * T[n, k] + bias[n].
int64_t gemm_exact_workspace_bytes(int64_t m, int64_t n, int64_t k) {
    return planes_plan(3, m, n, k).bytes;
}

hipError_t launch_gemm_exact(const float *x, const uint8_t *w, float *c, int64_t m, int64_t n,
                             int64_t k, const float *scale, const float *bias, hipStream_t s,
                             void *ws) {
    return launch_planes<3>(x, w, c, m, n, k, 1.0f, 0.0f, bias, s, ws, scale);
}

hipError_t launch_planes_sum(const float *part, float *c, int64_t rows, int64_t cols, int nsplit,
                             float alpha, hipStream_t s) {
    const bool v4 = cols % 4 == 0 && reinterpret_cast<uintptr_t>(c) % 16 == 0 &&
                    reinterpret_cast<uintptr_t>(part) % 16 == 0;
    const int64_t threads = rows * cols / (v4 ? 4 : 1);
    const int64_t blocks = (threads + 255) / 256 < 8192 ? (threads + 255) / 256 : 8192;
    auto sum = v4 ? planes_sum_kernel<true> : planes_sum_kernel<false>;
    sum<<<dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s>>>(part, c, rows, cols, nsplit, alpha,
                                                                  0.0f, nullptr, nullptr);
    return hipGetLastError();
}

}  // namespace t81hip
