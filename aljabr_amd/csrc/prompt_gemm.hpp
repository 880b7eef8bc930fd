// prompt_gemm.hpp - the prompt GEMM: Y[M,N] = X[M,K] . W[N,K]^T for more
// tokens than one pass of the small-M kernels holds, over every block format
// of the library, on v_mfma_f32_32x32x16_f16.
//
// The small-M kernels (matmul_mfma.hip, matmul_kquant.hip) read and decode
// the whole weight matrix once per 8 to 64 tokens, so a prompt paid for the
// weights M/64 (NF4), M/32 (K-quants) or M/8 (Q4_0, Q8_0) times. Here
//   1. prompt_pack_kernel writes the activations as fp16 A fragments,
//   2. prompt_weights_kernel the weights' codes in B-fragment order (a lane's
//      codes of a 64-element chunk in one 16-byte piece): read as stored, 32
//      rows a lane apart, every load of the GEMM fetched whole lines for a
//      few bytes of each (Q8_0 FFN, 2048 tokens: 2.07 -> 1.65 ms with it),
//   3. prompt_gemm_kernel multiplies: four waves side by side along N share
//      MT tiles of 32 tokens, a wave owns two tiles of 32 rows and decodes
//      them once for all its tokens. Both images arrive by LDS-DMA in
//      lane-contiguous pieces, two chunks ahead.
//
// What bounds it: the matrix cores (32 cycles per product of a 32x32x16
// step, one to three products per weight) and, beside them on one wave per
// SIMD, the vector ALU (16 FMAs per tile and scale group, the decode). Of a
// wave's time the matrix cores are busy 59 % (NF4, Q6_K) or 39 % (Q4_K in one
// part), the vector ALU issues 45 to 50 %; no LDS conflicts. NF4 MLP
// 4096 x 14336: 512 tokens 742 -> 424 us; Q8_0 Q/K/V 3840 x 2560, 197 tokens
// 727 -> 31 us; Q4_K_M FFN 4096 x 14336, 2048 tokens 5.35 -> 1.43 ms.
//
// Arithmetic, as in the small-M kernels: weights are exact fp16 integers (or
// NF4's exact H + R level pair, or Q6_K's two exact parts), the block scales
// stay fp32 on the accumulators, and the activations are one fp16 part (XP =
// 1, the rounding those kernels apply to the same shape) or an fp16 hi and lo
// part (XP = 2: an element to 2^-22, or 2^-25 in absolute terms if that is
// more; rows scaled by a power of two to a largest magnitude of 2^8 to 2^9
// where fp32 is replaced, so 2^-33 of the row's largest).
//   NF4   xh.H + xh.R (+ xl.H), acc += absmax * (per 64 elements)
//   Q4_0  B = q - 8, Q8_0 B = q: xh.B + xl.B, acc += d * (per 32 elements)
//   Q4_K  B = q * sc: xh.B (+ xl.B), acc += d * (...); per super-block the
//         min term acc -= dmin * (split sub-block sums of x) . (min codes)
//   Q6_K  B = (q - 32) * sc in two exact parts: xh.lo + xh.hi + xl.sum
//
// Operand layout: lane l = 32h + i supplies A[i][8h + e] and B[8h + e][i];
// accumulator r is C[8*(r/4) + 4h + r%4][i]. Step j of a 64-element chunk
// covers elements 16j + 8h + e, for NF4 32h + 8j + e (so that a lane's 32
// codes of a chunk are one 16-byte load); the activation image uses the same
// order.
#pragma once

#include <atomic>

#include "device.hpp"
#include "internal.hpp"
#include "kernels.hpp"
#include "kquant.hpp"

namespace aljabr {

enum : int { kPgNF4 = 0, kPgQ40 = 1, kPgQ80 = 2, kPgQ4K = 3, kPgQ6K = 4 };

constexpr int kPgWaves = 4;
constexpr int kPgThreads = kPgWaves * 64;
constexpr int kPgChunk = 64;                     // elements of K staged at a time

struct PgArgs {
    float *y[3];
    const uint8_t *w[3];
    const float *absmax[3];
    int end[3];                                  // stacked row ends (a 32-row tile lies in one segment)
    int nseg;
    const uint8_t *codes;                        // weight image [row tile][chunk][part][lane] x 16 bytes
    const uint32_t *aux;                         // [row tile][chunk][row] x PgFmt::AUX words
    int tile0, ntiles;                           // row tiles of this panel
    const uint8_t *xh, *xl;                      // activation image [chunk][token tile][step][lane] x 16 bytes
    const uint8_t *sums;                         // Q4_K: [super-block][token tile][lane] x 16 bytes
    const float *scale;                          // [tokens of the image] powers of two its rows were divided by, or null
    const float *x;                              // [M][K], for the row scales
    int scale_rows;                              // rows whose scale the weight image's launch writes
    float *part;                                 // [slice][M][N] with several K slices, else null
    int M, N, K;
    int chunks;                                  // ceil(K / 64)
    int per;                                     // chunks per K slice (a multiple of 4 for the K-quants)
    int slices, tiles, mt_groups, n_groups;      // token tiles of the image, workgroup grid
};

namespace pg {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x2v __attribute__((ext_vector_type(2)));
typedef half8 __attribute__((address_space(3))) lds_half8;
typedef u32x2v __attribute__((address_space(3))) lds_u32x2v;
typedef u32x4 __attribute__((address_space(3))) lds_u32x4;
typedef uint32_t __attribute__((address_space(3))) lds_u32;
typedef uint16_t u16u __attribute__((aligned(1)));
typedef uint32_t u32u __attribute__((aligned(1)));

template <class T>
__device__ __forceinline__ T *at(uint32_t offset) {
    return reinterpret_cast<T *>(static_cast<uintptr_t>(offset));
}

template <class T>
__device__ __forceinline__ T gread(const uint8_t *p) {
    return *reinterpret_cast<const __attribute__((address_space(1))) T *>(reinterpret_cast<uintptr_t>(p));
}

__device__ __forceinline__ uint32_t pack_half2(float lo, float hi) {
    const _Float16 a = static_cast<_Float16>(lo), b = static_cast<_Float16>(hi);
    return static_cast<uint32_t>(__builtin_bit_cast(uint16_t, a)) |
           (static_cast<uint32_t>(__builtin_bit_cast(uint16_t, b)) << 16);
}

__device__ __forceinline__ uint32_t h2fma(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(half2v, a),
                                                                  __builtin_bit_cast(half2v, b),
                                                                  __builtin_bit_cast(half2v, c)));
}

// Halves 0x64bb (1024 + byte, exact) of bytes 2I and 2I+1 of w.
template <int I>
__device__ __forceinline__ uint32_t magic(uint32_t w) {
    constexpr uint32_t b0 = 2 * I, b1 = 2 * I + 1;
    return __builtin_amdgcn_perm(0x64646464u, w, 0x04000400u | (b1 << 16) | b0);
}

__device__ __forceinline__ half8 fma_frag(uint32_t w0, uint32_t w1, uint32_t mul2, uint32_t add2) {
    return __builtin_bit_cast(half8, u32x4{h2fma(magic<0>(w0), mul2, add2), h2fma(magic<1>(w0), mul2, add2),
                                           h2fma(magic<0>(w1), mul2, add2), h2fma(magic<1>(w1), mul2, add2)});
}

__device__ __forceinline__ uint32_t dup_half(float v) {
    const uint32_t b = __builtin_bit_cast(uint16_t, static_cast<_Float16>(v));
    return b | (b << 16);
}

// The weight image. A lane's codes of a 64-element chunk of its row are CP
// 16-byte parts; AUX words per row and chunk hold the scales. read() takes
// them from the weights as stored (the packing kernel), load() from the image
// (the GEMM); frags() makes the B fragments of step J, scale(b) is the fp32
// factor of the products of 32-element half b.
//   NF4   codes; absmax                Q4_0  codes of both blocks; d0 | d1 << 16
//   Q8_0  codes; d0 | d1 << 16         Q4_K  codes; d | sc0 << 16 | sc1 << 24
//   Q6_K  6-bit codes, one per byte; four int8 scales, d
template <int F> struct Raw;

template <int CP, int AUX> struct RawBase {
    static constexpr int kParts = CP, kAux = AUX;
    u32x4 q[CP];
    uint32_t x[AUX];
    // From this wave's slot in LDS: code parts of 1 KiB, word p of row i of
    // both tiles at 256p + 4 * (32 * tile + i).
    __device__ __forceinline__ void load(uint32_t codes, uint32_t aux) {
#pragma unroll
        for (int p = 0; p < CP; ++p) q[p] = *at<lds_u32x4>(codes + 1024 * p);
#pragma unroll
        for (int p = 0; p < AUX; ++p) x[p] = *at<lds_u32>(aux + 256 * p);
    }
};

template <> struct Raw<kPgNF4> : RawBase<1, 1> {
    __device__ __forceinline__ void read(const uint8_t *row, const float *scale, int kb, int, int h) {
        q[0] = gread<u32x4>(row + 32 * static_cast<size_t>(kb) + 16 * h);
        x[0] = gread<uint32_t>(reinterpret_cast<const uint8_t *>(scale + kb));
    }
    __device__ __forceinline__ float scale(int) const { return __uint_as_float(x[0]); }
    // Table entry of byte e: the fp16 H pair of its two levels at e * E + 4r
    // and the R pair E / 2 on, in E / 8 replicas r (E = 256, or 128 where the
    // activations' two parts need the LDS); `ch` = 4r * 256 / E. Every read
    // lands in its fragment register; the relaxed atomic keeps the pairs'
    // reads apart (paired they would need moves, and a wait right here).
    template <uint32_t E>
    __device__ __forceinline__ void frags(half8 (&f)[2], int J, uint32_t ch) const {
        const uint32_t w = q[0][J];
        constexpr int sh = E == 256 ? 0 : 1;
        const uint32_t a[4] = {__builtin_amdgcn_perm(w, ch, 0x0C0C0400u) >> sh, __builtin_amdgcn_perm(w, ch, 0x0C0C0500u) >> sh,
                               __builtin_amdgcn_perm(w, ch, 0x0C0C0600u) >> sh, __builtin_amdgcn_perm(w, ch, 0x0C0C0700u) >> sh};
        u32x4 hi, rest;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            hi[i] = *at<lds_u32>(a[i]);
            rest[i] = __hip_atomic_load(at<lds_u32>(a[i] + E / 2), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        f[0] = __builtin_bit_cast(half8, hi);
        f[1] = __builtin_bit_cast(half8, rest);
    }
};

// Blocks past the row's end (K % 64 == 32) re-read the last one and take a
// zero scale.
template <> struct Raw<kPgQ40> : RawBase<1, 1> {
    __device__ __forceinline__ void read(const uint8_t *row, const float *, int kb, int K, int h) {
        const int last = (K >> 5) - 1;
        const uint8_t *b0 = row + 18 * static_cast<size_t>(2 * kb);
        const uint8_t *b1 = row + 18 * static_cast<size_t>(min(2 * kb + 1, last));
        const u32x2u c0 = gread<u32x2u>(b0 + 2 + 8 * h), c1 = gread<u32x2u>(b1 + 2 + 8 * h);
        q[0] = u32x4{c0.x, c0.y, c1.x, c1.y};
        x[0] = gread<u16u>(b0) | (2 * kb + 1 <= last ? static_cast<uint32_t>(gread<u16u>(b1)) << 16 : 0u);
    }
    __device__ __forceinline__ float scale(int b) const { return f16_bits_to_f32((x[0] >> (16 * b)) & 0xffffu); }
    template <uint32_t>
    __device__ __forceinline__ void frags(half8 (&f)[1], int J, uint32_t) const {
        const uint32_t w0 = q[0][2 * (J >> 1)], w1 = q[0][2 * (J >> 1) + 1];
        f[0] = J & 1 ? fma_frag(w0 & 0xf0f0f0f0u, w1 & 0xf0f0f0f0u, dup_half(0.0625f), dup_half(-72.0f))
                     : fma_frag(w0 & 0x0f0f0f0fu, w1 & 0x0f0f0f0fu, dup_half(1.0f), dup_half(-1032.0f));
    }
};

template <> struct Raw<kPgQ80> : RawBase<2, 1> {
    __device__ __forceinline__ void read(const uint8_t *row, const float *, int kb, int K, int h) {
        const int last = (K >> 5) - 1;
        uint32_t d[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const uint8_t *blk = row + 34 * static_cast<size_t>(min(2 * kb + b, last));
            const u32x2u c0 = gread<u32x2u>(blk + 2 + 8 * h), c1 = gread<u32x2u>(blk + 18 + 8 * h);
            // Biased to unsigned codes.
            q[b] = u32x4{c0.x, c0.y, c1.x, c1.y} ^ 0x80808080u;
            d[b] = 2 * kb + b <= last ? gread<u16u>(blk) : 0;
        }
        x[0] = d[0] | (d[1] << 16);
    }
    __device__ __forceinline__ float scale(int b) const { return f16_bits_to_f32((x[0] >> (16 * b)) & 0xffffu); }
    template <uint32_t>
    __device__ __forceinline__ void frags(half8 (&f)[1], int J, uint32_t) const {
        f[0] = fma_frag(q[J >> 1][2 * (J & 1)], q[J >> 1][2 * (J & 1) + 1], dup_half(1.0f), dup_half(-1152.0f));
    }
};

// The min codes and dmin of a row's super-blocks: three words (eight codes,
// one a byte; dmin as fp16) beside the chunk words of its last chunk.
template <> struct Raw<kPgQ4K> : RawBase<1, 1> {
    __device__ __forceinline__ void read(const uint8_t *row, const float *, int kb, int, int h) {
        const uint8_t *blk = row + kQ4KBytes * static_cast<size_t>(kb >> 2);
        const int c = kb & 3;
        const u32x2 c0 = gread<u32x2>(blk + 16 + 32 * c + 8 * h), c1 = gread<u32x2>(blk + 32 + 32 * c + 8 * h);
        q[0] = u32x4{c0.x, c0.y, c1.x, c1.y};
        const u32x4 hdr = gread<u32x4>(blk);
        const uint32_t sa = c >= 2 ? (hdr.w & 0x0f0f0f0fu) | ((hdr.y >> 2) & 0x30303030u) : hdr.y & 0x3f3f3f3fu;
        x[0] = (hdr.x & 0xffffu) | ((sa >> (16 * (c & 1))) << 16);
    }
    // A block whose min codes are all zero has no min term, whatever dmin
    // holds.
    static __device__ __forceinline__ void read_mins(const uint8_t *row, int sb, uint32_t (&m)[3]) {
        const u32x4 hdr = gread<u32x4>(row + kQ4KBytes * static_cast<size_t>(sb));
        m[0] = hdr.z & 0x3f3f3f3fu;
        m[1] = ((hdr.w >> 4) & 0x0f0f0f0fu) | ((hdr.z >> 2) & 0x30303030u);
        m[2] = (m[0] | m[1]) == 0 ? 0u : hdr.x >> 16;
    }
    __device__ __forceinline__ float scale(int) const { return f16_bits_to_f32(x[0] & 0xffffu); }
    // Steps 0, 1: low nibbles (the chunk's first sub-block); 2, 3: high ones.
    template <uint32_t>
    __device__ __forceinline__ void frags(half8 (&f)[1], int J, uint32_t) const {
        const float sc = J >> 1 ? ubyte_f<3>(x[0]) : ubyte_f<2>(x[0]);
        const uint32_t w0 = q[0][2 * (J & 1)], w1 = q[0][2 * (J & 1) + 1];
        f[0] = J >> 1 ? fma_frag(w0 & 0xf0f0f0f0u, w1 & 0xf0f0f0f0u, dup_half(sc * 0.0625f), dup_half(sc * -64.0f))
                      : fma_frag(w0 & 0x0f0f0f0fu, w1 & 0x0f0f0f0fu, dup_half(sc), dup_half(sc * -1024.0f));
    }
};

template <> struct Raw<kPgQ6K> : RawBase<2, 2> {
    __device__ __forceinline__ void read(const uint8_t *row, const float *, int kb, int, int h) {
        const uint8_t *blk = row + kQ6KBytes * static_cast<size_t>(kb >> 2);
        const int half = (kb >> 1) & 1, par = kb & 1;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const u32x2u ql = gread<u32x2u>(blk + 64 * half + 16 * j + 8 * h);
            const u32x2u qh = gread<u32x2u>(blk + 128 + 32 * half + 16 * (j & 1) + 8 * h);
            const uint32_t s4 = 4 * par, s2 = 2 * (2 * par + (j >> 1));
#pragma unroll
            for (int i = 0; i < 2; ++i)
                q[j >> 1][2 * (j & 1) + i] = ((ql[i] >> s4) & 0x0f0f0f0fu) | (((qh[i] >> s2) & 0x03030303u) << 4);
        }
        x[0] = gread<u32u>(blk + 192 + 4 * (kb & 3));
        x[1] = gread<u16u>(blk + 208);
    }
    __device__ __forceinline__ float scale(int) const { return f16_bits_to_f32(x[1]); }
    // (q - 32) * sl, (q - 32) * (sc - sl) with sl = sc & 15 (both exact) and
    // their fp16 sum, which meets the lo activations only.
    template <uint32_t>
    __device__ __forceinline__ void frags(half8 (&f)[3], int J, uint32_t) const {
        const int sv = static_cast<int8_t>((x[0] >> (8 * J)) & 0xffu);
        const int sl = sv & 15;
        const half2v ml = __builtin_bit_cast(half2v, dup_half(static_cast<float>(sl)));
        const half2v mh = __builtin_bit_cast(half2v, dup_half(static_cast<float>(sv - sl)));
        const uint32_t w0 = q[J >> 1][2 * (J & 1)], w1 = q[J >> 1][2 * (J & 1) + 1];
        const uint32_t p[4] = {magic<0>(w0), magic<1>(w0), magic<0>(w1), magic<1>(w1)};
        u32x4 lo, hi, sum;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const half2v v = __builtin_bit_cast(half2v, p[i]) + __builtin_bit_cast(half2v, 0xE420E420u);   // -1056
            const half2v a = v * ml, b = v * mh;
            lo[i] = __builtin_bit_cast(uint32_t, a);
            hi[i] = __builtin_bit_cast(uint32_t, b);
            sum[i] = __builtin_bit_cast(uint32_t, a + b);
        }
        f[0] = __builtin_bit_cast(half8, lo);
        f[1] = __builtin_bit_cast(half8, hi);
        f[2] = __builtin_bit_cast(half8, sum);
    }
};

// Words per (row tile, chunk) of `aux`, and of the Q4_K mins per (row tile,
// super-block), which follow the panel's chunk words.
template <int F> constexpr int kAuxWords = 32 * Raw<F>::kAux;
constexpr int kMinWords = 32 * 4;

// LDS-DMA from a uniform base plus a per-lane byte offset (dma16 and dma4 with
// a scalar address: the pieces of the images cost no address registers).
__device__ __forceinline__ void dma16_at(const void *base, uint32_t offset, uint32_t lds_base) {
    uint32_t save;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3\n\t"
                 "s_mov_b32 m0, %0"
                 : "=&s"(save)
                 : "s"(lds_base), "v"(offset), "s"(base)
                 : "memory");
}
__device__ __forceinline__ void dma4_at(const void *base, uint32_t offset, uint32_t lds_base) {
    uint32_t save;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %2, %3\n\t"
                 "s_mov_b32 m0, %0"
                 : "=&s"(save)
                 : "s"(lds_base), "v"(offset), "s"(base)
                 : "memory");
}

// The power of two that brings a token row's largest finite magnitude into
// [2^8, 2^9): with it any fp32 row fits the fp16 parts.
__device__ __forceinline__ void row_scale(const float *x, int K, float *scale) {
    __shared__ float best[4];
    const float4 *row = reinterpret_cast<const float4 *>(x);
    const int quads = K >> 2;                            // K % 32 == 0
    float top = 0.0f;
    for (int k0 = threadIdx.x; k0 < quads; k0 += 8 * 256) {
        float4 v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = row[min(k0 + 256 * i, quads - 1)];   // past the end: the last again
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float e[4] = {fabsf(v[i].x), fabsf(v[i].y), fabsf(v[i].z), fabsf(v[i].w)};
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (e[j] <= 3.4028235e38f) top = fmaxf(top, e[j]);
        }
    }
    top = wave_max(top);
    if ((threadIdx.x & 63) == 0) best[threadIdx.x >> 6] = top;
    __syncthreads();
    if (threadIdx.x) return;
    top = fmaxf(fmaxf(best[0], best[1]), fmaxf(best[2], best[3]));
    int e = 9;
    if (top > 0.0f) (void)frexpf(top, &e);               // top in [2^(e-1), 2^e)
    *scale = ldexpf(1.0f, (e < -100 ? -100 : e) - 9);
}

// Weights -> image: one workgroup per row tile and four chunks, a wave each
// (the lines of a row are read by one workgroup at a time). The first
// `scale_rows` workgroups write a token row's scale each: it is needed after
// this launch, and a launch of its own took 4 to 8 us more.
template <int F>
__global__ __launch_bounds__(256) void prompt_weights_kernel(PgArgs a, uint8_t *codes, uint32_t *aux, float *scale) {
    using R = Raw<F>;
    if (static_cast<int>(blockIdx.x) < a.scale_rows) {
        row_scale(a.x + static_cast<size_t>(blockIdx.x) * a.K, a.K, scale + blockIdx.x);
        return;
    }
    const int item = blockIdx.x - a.scale_rows;
    const int lane = threadIdx.x & 63, h = lane >> 5, i = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int quads = (a.chunks + 3) >> 2;
    const int tile = item / quads, quad = item % quads;
    const int kb = 4 * quad + wave;
    if (kb >= a.chunks) return;
    const int r = (a.tile0 + tile) * 32;
    int s = (r >= a.end[0]) + (r >= a.end[1]);
    if (s > a.nseg - 1) s = a.nseg - 1;
    const int start = s == 0 ? 0 : s == 1 ? a.end[0] : a.end[1];
    const int rows = (s == 0 ? a.end[0] : s == 1 ? a.end[1] : a.end[2]) - start;
    const int local = min(r - start + i, rows - 1);   // rows past the end re-read the last
    const uint8_t *w = s == 0 ? a.w[0] : s == 1 ? a.w[1] : a.w[2];
    const float *am = s == 0 ? a.absmax[0] : s == 1 ? a.absmax[1] : a.absmax[2];
    const size_t row_bytes = F == kPgNF4   ? static_cast<size_t>(a.K >> 1)
                             : F == kPgQ40 ? static_cast<size_t>(a.K >> 5) * 18
                             : F == kPgQ80 ? static_cast<size_t>(a.K >> 5) * 34
                             : F == kPgQ4K ? static_cast<size_t>(a.K >> 8) * kQ4KBytes
                                           : static_cast<size_t>(a.K >> 8) * kQ6KBytes;
    const uint8_t *row = w + local * row_bytes;
    R raw;
    raw.read(row, am + static_cast<size_t>(local) * (a.K >> 6), kb, a.K, h);
    const size_t piece = static_cast<size_t>(tile) * a.chunks + kb;
#pragma unroll
    for (int p = 0; p < R::kParts; ++p)
        *reinterpret_cast<u32x4 *>(codes + ((piece * R::kParts + p) * 64 + lane) * 16) = raw.q[p];
    if (h == 0) {
#pragma unroll
        for (int p = 0; p < R::kAux; ++p) aux[(piece * 32 + i) * R::kAux + p] = raw.x[p];
        if constexpr (F == kPgQ4K) {
            if (wave == 3) {
                uint32_t m[3];
                R::read_mins(row, quad, m);
                uint32_t *dst = aux + static_cast<size_t>(a.ntiles) * a.chunks * kAuxWords<F> +
                                ((static_cast<size_t>(tile) * quads + quad) * 32 + i) * 4;
                *reinterpret_cast<u32x4 *>(dst) = u32x4{m[0], m[1], m[2], 0u};
            }
        }
    }
}

template <int F> constexpr int kWeightParts = F == kPgNF4 ? 2 : F == kPgQ6K ? 3 : 1;

// LDS: the NF4 pair table, then rings of three chunks: the workgroup's
// activation pieces, each wave's weight pieces (codes, aux words, Q4_K mins)
// and Q4_K's sub-block sums.
template <int F, int XP, int MT, int NT> struct PgLds {
    static constexpr uint32_t kEntry = XP == 1 ? 256 : 128;             // NF4 pair-table entry
    static constexpr uint32_t kTable = F == kPgNF4 ? 256 * kEntry : 0;
    static constexpr uint32_t kPlane = MT * 4096;
    static constexpr uint32_t kBuf = XP * kPlane;
    static constexpr uint32_t kCodes = Raw<F>::kParts * 1024;
    static constexpr uint32_t kAux = NT * kCodes;                       // within a wave's slot
    static constexpr uint32_t kMins = kAux + Raw<F>::kAux * 256;
    static constexpr uint32_t kSlot = kMins + (F == kPgQ4K ? 1024 : 0);
    static constexpr uint32_t kWaves = kTable + 3 * kBuf;
    static constexpr uint32_t kSums = kWaves + kPgWaves * 3 * kSlot;
    static constexpr uint32_t kBytes = kSums + (F == kPgQ4K ? 3 * MT * 1024 : 0);
    static_assert(kBytes <= 160 * 1024, "LDS budget of a CU");
    static constexpr int kSimdWaves = 2 * kBytes <= 160 * 1024 ? 2 : 1;   // workgroups that fit a CU
    // LDS-DMA instructions of a wave per chunk.
    static constexpr int kLoads = XP * MT + NT * Raw<F>::kParts + Raw<F>::kAux + (F == kPgQ4K ? 2 : 0);
};

__device__ __forceinline__ f32x16 mfma(half8 a, half8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// The products of one step on one tile.
template <int F, int XP>
__device__ __forceinline__ f32x16 products(const half8 (&x)[XP], const half8 (&w)[kWeightParts<F>], f32x16 t) {
    t = mfma(x[0], w[0], t);
    if constexpr (F == kPgNF4 || F == kPgQ6K) t = mfma(x[0], w[1], t);
    if constexpr (XP == 2) t = mfma(x[1], F == kPgQ6K ? w[kWeightParts<F> - 1] : w[0], t);
    return t;
}

// Scheduling of a tile: its Q products with V vector operations and R LDS
// reads between them. Plain tiles issue two products first: the previous
// tile's accumulators are ready only after the first.
template <int Q, int V, int R>
__device__ __forceinline__ void pace() {
    if constexpr (R == 0) __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
    constexpr int G = R == 0 ? Q - 1 : Q;
#pragma unroll
    for (int q = 0; q < G; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);                             // MFMA
        __builtin_amdgcn_sched_group_barrier(0x2, (V + G - 1) / G, 0);               // VALU
        if constexpr (R > 0) __builtin_amdgcn_sched_group_barrier(0x100, (R + G - 1) / G, 0);   // LDS reads
    }
}

// One wave per SIMD where the LDS takes one workgroup a CU (four token tiles;
// two for NF4, Q6_K): the wave overlaps its own work in 256 VGPRs, and what
// does not fit or rests (tot) is in AGPRs. Its tiles run one after the other, each tile's products (US steps into one
// fresh accumulator tile) issued while the vector ALU scales the previous
// tile's products into acc and decodes fragments of the next US steps;
// weights and activations arrive two chunks ahead by LDS-DMA, every wait for
// them an explicit vmcnt, so nothing else is in flight through registers.
template <int F, int XP, int MT, int NT, int US>
__global__ __launch_bounds__(kPgThreads, (PgLds<F, XP, MT, NT>::kSimdWaves)) void prompt_gemm_kernel(PgArgs a) {
    using L = PgLds<F, XP, MT, NT>;
    using R = Raw<F>;
    constexpr int WP = kWeightParts<F>;
    constexpr int U = 4 / US;                    // units of US steps per chunk
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, i = lane & 31;
    // XCD-aware order: workgroup b runs on XCD b % 8, which takes a contiguous
    // run of (row group, slice, token group) items, token groups innermost, so
    // the workgroups that share weights share an L2.
    const int total = a.n_groups * a.slices * a.mt_groups;
    const int per_xcd = (total + 7) / 8;
    const int item = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (item >= total) return;
    const int mg = item % a.mt_groups, ns = item / a.mt_groups;
    const int slice = ns % a.slices, ng = ns / a.slices;
    const int kb0 = slice * a.per, kb1 = min(kb0 + a.per, a.chunks);

    uint32_t ch = 0;
    if constexpr (F == kPgNF4) {
        // Thread t fills replica t % (E / 8) of every low nibble's entries.
        constexpr uint32_t REP = L::kEntry / 8;
        const uint32_t rep = tid % REP;
#pragma unroll
        for (uint32_t c = tid / REP; c < 16; c += kPgThreads / REP) {
            const float lo = nf4_level_sel(c);
            const float lo_r = lo - static_cast<float>(static_cast<_Float16>(lo));
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const float hi = nf4_level_sel(k);
                const float hi_r = hi - static_cast<float>(static_cast<_Float16>(hi));
                const uint32_t e = (16 * k + c) * L::kEntry + 4 * rep;
                *at<lds_u32>(e) = pack_half2(hi, lo);
                *at<lds_u32>(e + L::kEntry / 2) = pack_half2(hi_r, lo_r);
            }
        }
        ch = 4 * (lane % REP) * (256 / L::kEntry);
        __syncthreads();
    }

    // This wave's row tiles in the weight image (tiles past the panel re-read
    // its last one).
    const int rt0 = (ng * kPgWaves + wave) * NT;
    const int t0 = min(rt0, a.ntiles - 1), t1 = min(rt0 + 1, a.ntiles - 1);
    const uint8_t *codes[NT] = {a.codes + static_cast<size_t>(t0) * a.chunks * L::kCodes,
                                a.codes + static_cast<size_t>(t1) * a.chunks * L::kCodes};
    // Lane halves fetch the words of the two tiles, from tile t0's base.
    const uint32_t *aux = a.aux + static_cast<size_t>(t0) * a.chunks * kAuxWords<F>;
    const uint32_t *mins = a.aux + static_cast<size_t>(a.ntiles) * a.chunks * kAuxWords<F> +
                           static_cast<size_t>(t0) * (a.chunks >> 2) * kMinWords;
    const uint32_t lane16 = lane * 16;
    const uint32_t aux_at = 4 * (h * (t1 - t0) * a.chunks * kAuxWords<F> + i * R::kAux);
    const uint32_t mins_at = 4 * (h * (t1 - t0) * (a.chunks >> 2) * kMinWords + i * 4);
    static_assert(NT == 2, "the aux words of a wave's two tiles fill one LDS-DMA instruction");
    const uint32_t slots = L::kWaves + wave * (3 * L::kSlot);

    // LDS-DMA p of chunk kb into ring slot r: MT * 4 activation pieces of 1 KiB
    // per plane (wave w the pieces w + 4q), then this wave's weights.
    const auto stage_piece = [&](int kb, int r, int p) {
        constexpr int XN = XP * MT, WN = NT * R::kParts;
        const uint32_t slot = slots + r * L::kSlot;
        if (p < XN) {
            const int q = p % MT, plane = p / MT;
            dma16_at((plane ? a.xl : a.xh) + (static_cast<size_t>(kb) * a.tiles + mg * MT + q) * 4096 + wave * 1024,
                     lane16, L::kTable + r * L::kBuf + plane * L::kPlane + q * 4096 + wave * 1024);
        } else if (p < XN + WN) {
            const int n = (p - XN) / R::kParts, part = (p - XN) % R::kParts;
            dma16_at(codes[n] + static_cast<size_t>(kb) * L::kCodes + 1024 * part, lane16,
                     slot + n * L::kCodes + 1024 * part);
        } else if (p < XN + WN + R::kAux) {
            const int word = p - XN - WN;
            dma4_at(aux + static_cast<size_t>(kb) * kAuxWords<F> + word, aux_at, slot + L::kAux + 256 * word);
        } else if (p == XN + WN + R::kAux) {
            dma16_at(mins + static_cast<size_t>(kb >> 2) * kMinWords, mins_at, slot + L::kMins);
        } else {
            const int t = wave & (MT - 1);
            dma16_at(a.sums + (static_cast<size_t>(kb >> 2) * a.tiles + mg * MT + t) * 1024, lane16,
                     L::kSums + (r * MT + t) * 1024);
        }
    };
    const auto stage = [&](int kb, int r) {
#pragma unroll
        for (int p = 0; p < L::kLoads; ++p) stage_piece(kb, r, p);
    };

    f32x16 acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[m][n] = f32x16{};
    f32x16 t[2] = {f32x16{}, f32x16{}};
    half8 w[NT][US][WP];
    float sc[NT];
    float s_prev = 0.0f;

    // The words of tile column n in ring slot r; the fragments and scale of
    // column n for the unit starting at step j0.
    R raw[NT];
    const auto read_raw = [&](int n, int r) {
        raw[n].load(slots + r * L::kSlot + n * L::kCodes + lane16, slots + r * L::kSlot + L::kAux + (32 * n + i) * 4);
    };
    const auto decode = [&](int n, int j0) {
#pragma unroll
        for (int j = 0; j < US; ++j) raw[n].template frags<L::kEntry>(w[n][j], j0 + j, ch);
        sc[n] = raw[n].scale(j0 >> 1);
    };
    // Activation fragments, double-buffered where the registers allow it (one
    // part); else each step's are replaced as the row's last tile has used
    // them.
    constexpr int XB = XP == 1 ? 2 : 1;
    half8 x[XB][US][XP];
    const auto read_x = [&](half8 (&v)[XP], int r, int u, int m, int j) {
        const uint32_t xb = L::kTable + r * L::kBuf + lane16;
#pragma unroll
        for (int p = 0; p < XP; ++p) v[p] = *at<lds_half8>(xb + p * L::kPlane + m * 4096 + (u * US + j) * 1024);
    };

    stage(kb0, 0);
    stage(min(kb0 + 1, kb1 - 1), 1);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L::kLoads) : "memory");
    lds_barrier();
    read_raw(0, 0);
    decode(0, 0);
    read_raw(1, 0);
#pragma unroll
    for (int j = 0; j < US; ++j) read_x(x[0][j], 0, 0, 0, j);

    // Two parts: the sums of earlier chunks. acc itself runs over kFold chunks
    // only (half of that in short slices): one fp32 chain over all of K rounds
    // more than the waves and slices of the passes do. Error against float64 of
    // the passes, one chain, this: Q8_0 4096 x 14336, 512 tokens 1.18e-7,
    // 2.08e-7, 1.10e-7; K = 1024 0.98, 1.25, 0.94. The passes of NF4 and Q6_K
    // round more (1.9e-7 to 2.1e-7): half as many folds. They cost 2 to 8 % of
    // the time at four token tiles. One part is rounded to 2e-4 anyway: none.
    constexpr int kFold = F == kPgNF4 || F == kPgQ6K ? 16 : 8;
    const int step = XP == 1 ? a.chunks : kb1 - kb0 <= 2 * kFold ? kFold / 2 : kFold;
    f32x16 tot[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) tot[m][n] = f32x16{};

    // One chunk in ring slot r (the next in r1, the one after into r2). Column
    // 0's fragments are decoded during the previous unit's last tile (of
    // column 1), column 1's during the unit's first tile, each from words
    // read one tile earlier.
    const auto chunk = [&](int kb, int r, int r1, int r2) {
        const int ahead = min(kb + 2, kb1 - 1);
        if constexpr (F == kPgQ4K) {
            if ((kb & 3) == 3) {                 // the super-block's min term
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    const u32x4 mn = *at<lds_u32x4>(slots + r * L::kSlot + L::kMins + (32 * n + i) * 16);
                    const half8 bm = fma_frag(mn.x, mn.y, dup_half(1.0f), dup_half(-1024.0f));
                    const float dm = -f16_bits_to_f32(mn.z);
#pragma unroll
                    for (int m = 0; m < MT; ++m) {
                        const half8 xs = *at<lds_half8>(L::kSums + (r * MT + m) * 1024 + lane16);
                        const f32x16 v = mfma(xs, bm, f32x16{});
#pragma unroll
                        for (int q = 0; q < 16; ++q) acc[m][n][q] = fmaf(dm, v[q], acc[m][n][q]);
                        __builtin_amdgcn_sched_barrier(0);   // one tile's registers at a time
                    }
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const int xi = XB == 2 ? (u * MT + m) & 1 : 0;
                // The next token tile's unit (0 of the next chunk after the last).
                const int nu = m + 1 < MT ? u : (u + 1) % U, nm = m + 1 < MT ? m + 1 : 0;
                const int nr = m + 1 == MT && u + 1 == U ? r1 : r;
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    const int g = (u * MT + m) * NT + n;
                    const bool first = m == 0 && n == 0, last = m == MT - 1 && n == NT - 1;
                    constexpr int TT = U * MT * NT;
#pragma unroll
                    for (int p = 0; p < L::kLoads; ++p)
                        if (p * (TT - 2) / L::kLoads == g) stage_piece(ahead, r2, p);
                    if (g == TT - 2) {
                        // The next chunk is in, in every wave (its other readers of
                        // slot r are done with it too: what is left of this chunk is
                        // in registers).
                        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L::kLoads) : "memory");
                        lds_barrier();
                    }
                    if (m == MT - 1) read_raw(n, u == U - 1 ? r1 : r);
                    if (XB == 2 && n == 0) {
#pragma unroll
                        for (int j = 0; j < US; ++j) read_x(x[XB - 1 - xi][j], nr, nu, nm, j);
                    }
                    const float sp = s_prev;         // the previous tile's scale
                    if (first) decode(1, u * US);
                    if (last) decode(0, (u + 1) % U * US);
                    f32x16 v = f32x16{};
#pragma unroll
                    for (int j = 0; j < US; ++j) {
                        v = products<F, XP>(x[xi][j], w[n][j], v);
                        if (XB == 1 && n == NT - 1) read_x(x[0][j], nr, nu, nm, j);
                    }
                    t[g & 1] = v;
                    const int pm = n ? m : (m + MT - 1) % MT, pn = n ? n - 1 : NT - 1;   // the previous tile
#pragma unroll
                    for (int q = 0; q < 16; ++q) acc[pm][pn][q] = fmaf(sp, t[(g & 1) ^ 1][q], acc[pm][pn][q]);
                    s_prev = sc[n];
                    constexpr int Q = US * (F == kPgQ6K ? 3 : F == kPgNF4 ? 1 + XP : XP);
                    constexpr int D = US * (F == kPgNF4 ? 4 : F == kPgQ6K ? 30 : 14);   // a column's decode
                    if (first || last) pace<Q, 16 + D, F == kPgNF4 ? 8 * US : 1>();
                    else pace<Q, 16, 0>();
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    };

    int r = 0;
    for (int kb = kb0; kb < kb1;) {
        const int fold = min(kb + step, kb1);
        for (; kb < fold; ++kb) {
            const int r1 = r == 2 ? 0 : r + 1, r2 = r1 == 2 ? 0 : r1 + 1;
            chunk(kb, r, r1, r2);
            r = r1;
        }
        if constexpr (XP == 1) continue;
        // acc goes on with what the addition to tot rounded off.
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    float sum = tot[m][n][q] + acc[m][n][q];
                    // (A bound no such rest reaches: infinite sums have none, inf - inf.)
                    acc[m][n][q] = __builtin_amdgcn_fmed3f(acc[m][n][q] - (sum - tot[m][n][q]), -1e32f, 1e32f);
                    if constexpr (MT == 4) asm volatile("" : "+a"(sum));
                    tot[m][n][q] = sum;
                }
    }
    if constexpr (XP == 1) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n) tot[m][n] = acc[m][n];
    }
    // The last tile's products; nothing may still be landing in LDS at the end.
#pragma unroll
    for (int q = 0; q < 16; ++q) tot[MT - 1][NT - 1][q] = fmaf(s_prev, t[1][q], tot[MT - 1][NT - 1][q]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    // Column i of each tile: one stacked row.
    float *dst[NT];
    size_t ld[NT];
    bool mine[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int row = (a.tile0 + rt0 + n) * 32;
        mine[n] = rt0 + n < a.ntiles && row + i < a.N;
        int s = (row >= a.end[0]) + (row >= a.end[1]);
        if (s > a.nseg - 1) s = a.nseg - 1;
        const int start = s == 0 ? 0 : s == 1 ? a.end[0] : a.end[1];
        const int rows = (s == 0 ? a.end[0] : s == 1 ? a.end[1] : a.end[2]) - start;
        dst[n] = a.part ? a.part + static_cast<size_t>(slice) * a.M * a.N + row + i
                        : (s == 0 ? a.y[0] : s == 1 ? a.y[1] : a.y[2]) + (row - start + i);
        ld[n] = a.part ? a.N : rows;
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int tok0 = (mg * MT + m) * 32 + 4 * h;
        if (a.scale) {                           // four of a tile's tokens at a time, not a load before every store
            float4 f[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) f[q] = *reinterpret_cast<const float4 *>(a.scale + tok0 + 8 * q);
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int q = 0; q < 16; ++q)
                    tot[m][n][q] *= (q & 3) == 0 ? f[q >> 2].x : (q & 3) == 1 ? f[q >> 2].y : (q & 3) == 2 ? f[q >> 2].z : f[q >> 2].w;
        }
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            if (!mine[n]) continue;
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int tok = tok0 + 8 * (q >> 2) + (q & 3);
                if (tok < a.M) dst[n][static_cast<size_t>(tok) * ld[n]] = tot[m][n][q];
            }
        }
    }
}

template <int F>
void pack_weights(const PgArgs &a, hipStream_t s) {
    const int quads = (a.chunks + 3) / 4;
    hipLaunchKernelGGL((prompt_weights_kernel<F>), dim3(static_cast<unsigned>(a.ntiles * quads + a.scale_rows)), dim3(256), 0,
                       s, a, const_cast<uint8_t *>(a.codes), const_cast<uint32_t *>(a.aux), const_cast<float *>(a.scale));
}

// Launch of one instantiation (the LDS attribute is per kernel, per process).
template <int F, int XP, int MT, int NT, int US>
void launch(const PgArgs &a, hipStream_t s) {
    const auto fn = prompt_gemm_kernel<F, XP, MT, NT, US>;
    constexpr uint32_t lds = PgLds<F, XP, MT, NT>::kBytes;
    static std::atomic<bool> set{false};
    if (!set.load(std::memory_order_acquire)) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(fn), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  static_cast<int>(lds));
        set.store(true, std::memory_order_release);
    }
    const int total = a.n_groups * a.slices * a.mt_groups;
    hipLaunchKernelGGL(fn, dim3(static_cast<unsigned>(8 * ((total + 7) / 8))), dim3(kPgThreads), lds, s, a);
}

}  // namespace pg

// Per format file: the weight image of a panel, and the GEMM with mt (2 or 4)
// x 2 tiles per wave and xp activation parts.
template <int F> void prompt_pack(const PgArgs &a, hipStream_t s);
template <int F> void prompt_multiply(const PgArgs &a, int xp, int mt, hipStream_t s);

}  // namespace aljabr
