// attention_chunk.hip - attention of several query rows per sequence (a chunk
// of a prompt, a draft being verified) over a contiguous fp16 cache, on the
// matrix cores.
//
// The split kernel (attention.hip) runs one workgroup per (KV head, query
// row): every query row read the whole cache again. Here the G query heads of
// a KV head and the query positions are stacked into rows r = qi * G + g, a
// wave takes 32 of them, and a workgroup's 128 rows walk the keys in tiles of
// 32 that arrive in LDS once for all of them.
//   1. chunk_pack_kernel writes K (rows) and V (transposed) as tile images
//      that are copied to LDS as they are (keys past Sk are zeros);
//   2. chunk_attention_kernel computes S^T = K Q^T and O^T += V^T P^T with
//      v_mfma_f32_32x32x16_f16 and an online softmax per row;
//   3. with several key splits, the split kernel's merge combines them.
//
// Precision: K and V are exact fp16 operands. A query row is scaled by a power
// of two to a largest magnitude in [2^14, 2^15) and split into two fp16 parts
// (2^-24 of each element), a weight, scaled by 2^11 (largest in [2^11, 2^13]),
// likewise; all sums are fp32.
//
// What bounds it: the matrix cores and the softmax's vector work of a wave's
// own tile in turn (32 products of 32 cycles a tile at D = 128), then the
// split partials (16 KB a row block and split). 32 / 8 heads, D = 128: 256
// rows at 2048 keys 283 -> 52 us, error against float64 2.6e-7 -> 2.0e-7.
//
// Infinities and NaN: zero weights and parts times an infinity would make a
// NaN that the exact sum does not have, and a masked key's V must not reach a
// row that cannot see it. A row whose sums are not finite is therefore done
// again over its own keys in plain fp32. With an infinite V element that every
// row sees, 256 rows at 2048 keys take 0.70 ms (the split kernel 0.30 ms
// whatever the values; 5.3 ms a row and key at a time).
#include <cmath>

#include "device.hpp"
#include "internal.hpp"
#include "kernels.hpp"

namespace aljabr {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kRows = 32 * kWaves;           // stacked query rows per workgroup
constexpr int kKeys = 32;                    // keys per tile
constexpr int kVtStride = kKeys + 4;         // halves: 72-byte rows, conflict-free 8-byte reads
constexpr int kRedo = 8;                     // rows that a wave does again together
constexpr float kLog2eC = 1.4426950408889634f;
constexpr float kWeightScale = 2048.0f;      // weights are split, and summed over V, times this

struct ChunkParams {
    const float *q;
    const _Float16 *k, *v;
    float *out;                  // [B][Hq][Sq][D], as q
    float *part_o, *part_ml;     // [row][split][D] and [row][split](m, l), or null with one split
    int B, Hq, Hkv, G, Sq, Sk;
    float scale;
    int causal;
    int ntiles, splits, tiles_per_split, row_blocks;
};

// Halves of a tile's image: K as [kKeys][D + 8], V^T as [D][kVtStride], padded
// to whole rounds of the workgroup's 16-byte copies.
template <int D>
constexpr int tile_halves() {
    constexpr int used = kKeys * (D + 8) + D * kVtStride, round = kThreads * 8;
    return (used + round - 1) / round * round;
}

// Keys visible to query position qi (causal: bottom-right aligned, Sq <= Sk).
__device__ __forceinline__ int visible(const ChunkParams &p, int qi) {
    return p.causal ? p.Sk - p.Sq + qi + 1 : p.Sk;
}

template <int D>
__global__ __launch_bounds__(256) void chunk_pack_kernel(ChunkParams p, _Float16 *__restrict__ pk) {
    constexpr int KS = D + 8;
    const int tile = blockIdx.x % p.ntiles, k0 = tile * kKeys;
    const size_t head = static_cast<size_t>(blockIdx.x / p.ntiles) * p.Sk * D;   // b * Hkv + kvh
    const _Float16 *kbase = p.k + head, *vbase = p.v + head;
    _Float16 *dst = pk + static_cast<size_t>(blockIdx.x) * tile_halves<D>();
    for (int i = threadIdx.x; i < kKeys * (D / 8); i += 256) {
        const int key = i / (D / 8), d = 8 * (i % (D / 8));
        half8 x = {};
        if (k0 + key < p.Sk) x = *reinterpret_cast<const half8 *>(kbase + static_cast<size_t>(k0 + key) * D + d);
        *reinterpret_cast<half8 *>(dst + key * KS + d) = x;
    }
    for (int i = threadIdx.x; i < (kKeys / 4) * (D / 4); i += 256) {
        const int kg = 4 * (i / (D / 4)), d = 4 * (i % (D / 4));
        half4 r[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            r[c] = half4{};
            if (k0 + kg + c < p.Sk)
                r[c] = *reinterpret_cast<const half4 *>(vbase + static_cast<size_t>(k0 + kg + c) * D + d);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            *reinterpret_cast<half4 *>(dst + kKeys * KS + (d + e) * kVtStride + kg) =
                half4{r[0][e], r[1][e], r[2][e], r[3][e]};
    }
}

__device__ __forceinline__ void split_half(float v, _Float16 &hi, _Float16 &lo) {
    hi = static_cast<_Float16>(v);
    lo = static_cast<_Float16>(v - static_cast<float>(hi));
}

template <int D>
__global__ __launch_bounds__(kThreads, 2) void chunk_attention_kernel(ChunkParams p, const _Float16 *__restrict__ pk) {
    constexpr int KS = D + 8;                // K row stride (halves): conflict-free 16-byte reads
    constexpr int STEPS = D / 16, DT = D / 32;
    constexpr int BUF = tile_halves<D>();
    constexpr int CH = BUF / 8 / kThreads;   // 16-byte copies per lane per tile
    __shared__ __attribute__((aligned(16))) _Float16 lds[2 * BUF];

    const int tid = threadIdx.x;
    const int lane = tid & 63, h = lane >> 5, nl = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // The KV head varies fastest: with 8 heads, each XCD keeps one in its L2.
    int idx = blockIdx.x;
    const int kvh = idx % p.Hkv;
    idx /= p.Hkv;
    const int rb = idx % p.row_blocks;
    idx /= p.row_blocks;
    const int split = idx % p.splits;
    const int b = idx / p.splits;

    const int total = p.Sq * p.G;            // stacked rows of a (sequence, KV head)
    const int w0 = rb * kRows + wave * 32;
    const int row = min(w0 + nl, total - 1); // rows past the end repeat the last and are not stored
    const int hi_t = visible(p, row / p.G);
    const int w_hi = visible(p, min(w0 + 31, total - 1) / p.G);
    const int full_hi = visible(p, min(w0, total - 1) / p.G);
    const int g_hi = visible(p, (min(rb * kRows + kRows, total) - 1) / p.G);
    const size_t qrow = (static_cast<size_t>(b) * p.Hq + kvh * p.G + row % p.G) * p.Sq + row / p.G;

    // The row times scale * log2(e) as B fragments: step s holds d = 16s + 8h .. + 8.
    half8 qh[STEPS], ql[STEPS];
    float unscale;
    {
        const float *qr = p.q + qrow * D + 8 * h;
        const float qs = p.scale * kLog2eC;
        float top = 0.0f;
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            const float4 a = *reinterpret_cast<const float4 *>(qr + 16 * s);
            const float4 c = *reinterpret_cast<const float4 *>(qr + 16 * s + 4);
            top = fmaxf(top, fmaxf(fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))),
                                   fmaxf(fmaxf(fabsf(c.x), fabsf(c.y)), fmaxf(fabsf(c.z), fabsf(c.w)))));
        }
        top = fmaxf(top, __shfl_xor(top, 32)) * qs;
        int e = 0;
        if (top > 0.0f && top <= 3.4028235e38f) (void)frexpf(top, &e);   // top in [2^(e-1), 2^e)
        e = e < -100 ? -100 : e;
        const float up = ldexpf(1.0f, 15 - e);
        unscale = ldexpf(1.0f, e - 15);
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            const float4 a = *reinterpret_cast<const float4 *>(qr + 16 * s);
            const float4 c = *reinterpret_cast<const float4 *>(qr + 16 * s + 4);
            const float x[8] = {a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                _Float16 hi, lo;
                split_half(x[i] * qs * up, hi, lo);
                qh[s][i] = hi;
                ql[s][i] = lo;
            }
        }
    }

    const _Float16 *tiles = pk + static_cast<size_t>(b * p.Hkv + kvh) * p.ntiles * BUF;
    auto load_tile = [&](int kt, _Float16 *dst) {
        const _Float16 *src = tiles + static_cast<size_t>(kt) * BUF;
#pragma unroll
        for (int j = 0; j < CH; ++j) {
            const int base = 8 * (kThreads * j + 64 * wave);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(src + base + 8 * lane),
                                             (__attribute__((address_space(3))) void *)(dst + base), 16, 0, 0);
        }
    };

    f32x16 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt] = f32x16{};
    // Weights are 2^(s - m). The reference m is raised only when a score
    // exceeds it by more than 2 (the rounding of the exponent grows with the
    // distance, so the scale is not part of it either).
    float m = -INFINITY, l = 0.0f;
    const int kt0 = split * p.tiles_per_split;
    const int kt1 = min(min(kt0 + p.tiles_per_split, p.ntiles), (g_hi + kKeys - 1) / kKeys);
    if (kt0 < kt1) load_tile(kt0, lds);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    for (int kt = kt0; kt < kt1; ++kt) {
        const int cur = (kt - kt0) & 1;
        // The other buffer's readers finished before the barrier that ended the last trip.
        if (kt + 1 < kt1) load_tile(kt + 1, lds + (cur ^ 1) * BUF);
        const _Float16 *kl = lds + cur * BUF, *vl = kl + kKeys * KS;
        const int k0 = kt * kKeys;
        if (k0 < w_hi) {
            // S^T (in two chains, of half the roundings each): accumulator r is key k0 + 8(r/4) + 4h + r%4 of this lane's row.
            f32x16 s = {}, s1 = {}, t = {};
#pragma unroll
            for (int st = 0; st < STEPS; ++st) {
                const half8 a = *reinterpret_cast<const half8 *>(kl + nl * KS + 16 * st + 8 * h);
                if (st < STEPS / 2) s = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qh[st], s, 0, 0, 0);
                else s1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qh[st], s1, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, ql[st], t, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = (s[r] + (s1[r] + t[r])) * unscale;
            if (k0 + kKeys > full_hi) {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (k0 + 8 * (r >> 2) + 4 * h + (r & 3) >= hi_t) s[r] = -INFINITY;
            }
            float mx = s[0];
#pragma unroll
            for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            if (__any(mx > m + 2.0f)) {
                if (mx > m + 2.0f) {
                    const float alpha = __builtin_amdgcn_exp2f(m - mx);      // 0 while m is -inf
                    l *= alpha;
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) o[dt] *= alpha;
                    m = mx;
                }
            }
            const float ref = m == -INFINITY ? 0.0f : m;                     // no key so far: weights 0
            half8 ph[2], pl[2];
            float sum[4] = {};                       // the tile's weights before the running sum: fewer roundings of l
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float w = __builtin_amdgcn_exp2f(s[r] - ref);
                sum[r & 3] += w;
                _Float16 hi, lo;
                split_half(w * kWeightScale, hi, lo);
                ph[r >> 3][r & 7] = hi;
                pl[r >> 3][r & 7] = lo;
            }
            l += (sum[0] + sum[1]) + (sum[2] + sum[3]);
            // Lane half h supplies contraction entries 0..3 -> key 16j + 4h + e
            // and 4..7 -> key 16j + 8 + 4h + e - 4: its accumulators 8j .. 8j + 7.
            // Small terms first, into a fresh tile: o is rounded once per tile of keys.
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                half8 a[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const _Float16 *at = vl + (32 * dt + nl) * kVtStride + 16 * j + 4 * h;
                    const half4 a0 = *reinterpret_cast<const half4 *>(at), a1 = *reinterpret_cast<const half4 *>(at + 8);
                    a[j] = half8{a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
                }
                f32x16 v = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0], pl[0], f32x16{}, 0, 0, 0);
                v = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[1], pl[1], v, 0, 0, 0);
                v = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0], ph[0], v, 0, 0, 0);
                v = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[1], ph[1], v, 0, 0, 0);
                o[dt] += v;
            }
        }
        __builtin_amdgcn_s_waitcnt(0);               // this wave's copies of the next tile have landed
        __syncthreads();
    }

    l += __shfl_xor(l, 32);                          // the lane halves share one reference
    const bool mine = w0 + nl < total;
    float probe = l * 0.0f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) probe = fmaf(o[dt][r], 0.0f, probe);
    probe += __shfl_xor(probe, 32);
    const bool bad = !(probe == 0.0f);
    if (mine && !bad) {
        float *dst = p.part_o ? p.part_o + (qrow * p.splits + split) * D : p.out + qrow * D;
        const float f = (p.part_o ? 1.0f : l > 0.0f ? 1.0f / l : 0.0f) * (1.0f / kWeightScale);
        // Accumulator r of tile dt is d = 32dt + 8(r/4) + 4h + r%4.
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                *reinterpret_cast<float4 *>(dst + 32 * dt + 8 * j + 4 * h) = make_float4(
                    o[dt][4 * j] * f, o[dt][4 * j + 1] * f, o[dt][4 * j + 2] * f, o[dt][4 * j + 3] * f);
        if (p.part_o && h == 0) {
            p.part_ml[(qrow * p.splits + split) * 2] = m;
            p.part_ml[(qrow * p.splits + split) * 2 + 1] = l;
        }
    }
    // Rows that are not finite: the wave does them again, kRedo at a time, over
    // the keys of this split that each sees: a lane per key for the scores (the
    // rows in LDS, which the tiles have left), a lane per element for the
    // weights over V.
    uint32_t todo = static_cast<uint32_t>(__ballot(mine && bad));
    float *qs = reinterpret_cast<float *>(lds) + wave * (kRedo * D);
    const size_t head = static_cast<size_t>(b * p.Hkv + kvh) * p.Sk * D;
    while (todo) {
        size_t qr[kRedo];
        int end[kRedo], rows = 0, last = 0;
#pragma unroll
        for (int i = 0; i < kRedo; ++i) {            // past the last row: it again, over no keys
            const int rr = w0 + (todo ? __builtin_ctz(todo) : 0);
            qr[i] = (static_cast<size_t>(b) * p.Hq + kvh * p.G + rr % p.G) * p.Sq + rr / p.G;
            end[i] = todo ? min(visible(p, rr / p.G), (kt0 + p.tiles_per_split) * kKeys) : 0;
            rows += todo != 0;
            last = max(last, end[i]);
            todo &= todo - 1;
        }
#pragma unroll
        for (int i = 0; i < kRedo; ++i)
#pragma unroll
            for (int j = 0; j < D / 64; ++j) qs[i * D + 64 * j + lane] = p.q[qr[i] * D + 64 * j + lane] * (p.scale * kLog2eC);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // this wave's own writes
        float mr[kRedo], lr[kRedo], acc[kRedo][D / 64];
#pragma unroll
        for (int i = 0; i < kRedo; ++i) {
            mr[i] = -INFINITY;
            lr[i] = 0.0f;
#pragma unroll
            for (int j = 0; j < D / 64; ++j) acc[i][j] = 0.0f;
        }
        for (int k0 = kt0 * kKeys; k0 < last; k0 += 64) {
            const int key = k0 + lane;
            const _Float16 *kr = p.k + head + static_cast<size_t>(min(key, p.Sk - 1)) * D;
            float w[kRedo], dot[kRedo][4] = {};      // four chains: of D / 4 roundings each
#pragma unroll 1
            for (int d0 = 0; d0 < D; d0 += 32) {
                half8 x[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) x[c] = *reinterpret_cast<const half8 *>(kr + d0 + 8 * c);
#pragma unroll
                for (int c = 0; c < 4; ++c) {
#pragma unroll
                    for (int i = 0; i < kRedo; ++i)
#pragma unroll
                        for (int e = 0; e < 8; ++e)
                            dot[i][e & 3] = fmaf(qs[i * D + d0 + 8 * c + e], static_cast<float>(x[c][e]), dot[i][e & 3]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            uint64_t live[kRedo], any = 0, all = ~0ull;   // keys with a weight; the others' V is not touched
#pragma unroll
            for (int i = 0; i < kRedo; ++i) {
                w[i] = (dot[i][0] + dot[i][1]) + (dot[i][2] + dot[i][3]);
                const bool on = key < end[i] && !(w[i] == -INFINITY);
                const float mn = fmaxf(mr[i], wave_max(on ? w[i] : -INFINITY));
                const float alpha = mr[i] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mr[i] - mn);
                w[i] = on ? __builtin_amdgcn_exp2f(w[i] - mn) : 0.0f;
                live[i] = __ballot(on);
                any |= live[i];
                all &= live[i];
                lr[i] = fmaf(lr[i], alpha, wave_sum(w[i]));
#pragma unroll
                for (int j = 0; j < D / 64; ++j) acc[i][j] *= alpha;
                mr[i] = mn;
            }
#pragma unroll 1
            for (int c0 = 0; c0 < 64 && any >> c0; c0 += 8) {
                float v[8][D / 64];
#pragma unroll
                for (int c = 0; c < 8; ++c)
#pragma unroll
                    for (int j = 0; j < D / 64; ++j)
                        v[c][j] = static_cast<float>(
                            p.v[head + static_cast<size_t>(min(k0 + c0 + c, p.Sk - 1)) * D + 64 * j + lane]);
                const bool whole = (all >> c0 & 0xff) == 0xff;
#pragma unroll
                for (int c = 0; c < 8; ++c)
#pragma unroll
                    for (int i = 0; i < kRedo; ++i) {
                        const float wc = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w[i]), c0 + c));
                        if (whole || (live[i] >> (c0 + c) & 1))
#pragma unroll
                            for (int j = 0; j < D / 64; ++j) acc[i][j] = fmaf(wc, v[c][j], acc[i][j]);
                    }
            }
        }
#pragma unroll
        for (int i = 0; i < kRedo; ++i) {
            if (i >= rows) continue;
            // A NaN score alone leaves no reference: any finite one carries it.
            if (mr[i] == -INFINITY && lr[i] != lr[i]) mr[i] = 0.0f;
            float *dst = p.part_o ? p.part_o + (qr[i] * p.splits + split) * D : p.out + qr[i] * D;
#pragma unroll
            for (int j = 0; j < D / 64; ++j)
                dst[64 * j + lane] = p.part_o ? acc[i][j] : lr[i] == 0.0f ? 0.0f : acc[i][j] / lr[i];
            if (p.part_o && lane == 0) {
                p.part_ml[(qr[i] * p.splits + split) * 2] = mr[i];
                p.part_ml[(qr[i] * p.splits + split) * 2 + 1] = lr[i];
            }
        }
    }
}

template <int D>
void launch(const ChunkParams &p, _Float16 *pk, hipStream_t s) {
    hipLaunchKernelGGL(chunk_pack_kernel<D>, dim3(static_cast<unsigned>(p.B * p.Hkv * p.ntiles)), dim3(256), 0, s, p, pk);
    hipLaunchKernelGGL(chunk_attention_kernel<D>, dim3(static_cast<unsigned>(p.row_blocks * p.Hkv * p.splits * p.B)),
                       dim3(kThreads), 0, s, p, pk);
}

// Where the tiles beat the split kernel, in us at one sequence, split kernel
// against this one (Hq / Hkv / D):
//   32/8/128  1024 keys: 16 rows of Q 17.9/19.1, 32: 24.7/22.6, 64: 41.7/26.6
//             4096 keys: 4: 17.2/22.5, 8: 26.3/23.1, 64: 150/35
//             128 keys, 64: 10.3/14.2
//   8/8/64    1024 keys, 64: 11.6/14.1;  4096 keys, 32: 19.0/18.2, 64: 34/20
//   32/4/128  4096 keys: 4: 19.8/20.0, 8: 29/22
// and at the line (2^27) with several:
//   32/8/128  8 x 16 rows of Q, 256 keys 26.2/27.1; 4 x 16, 512: 24.5/25.0;
//             2 x 16, 1024: 24.1/24.4;  64/8/64 (one wave of four with rows)
//             16 x 4, 512: 26.7/27.4; 16 x 4, 8192: 294/284
// The line is the split kernel's work (it runs ~7e6 of these products per us,
// the launches here take ~10 us more), and at least the rows that pay for
// writing the tile images, a second and third pass over the cache.
constexpr long long kMinRows = 32;               // G * Sq
constexpr long long kMinWork = 1LL << 27;        // B * Hq * Sq * Sk * D
constexpr size_t kMaxScratch = size_t{1} << 30;      // bounds what the stream's scratch grows to

}  // namespace

int enqueue_attention_chunk(const AttnParams &a) {
    const int G = a.Hkv > 0 ? a.Hq / a.Hkv : 0;
    if ((a.D != 64 && a.D != 128) || !a.kv_f16 || a.Sq < 2 || G < 1 || static_cast<long long>(a.Sq) * G < kMinRows ||
        a.mask || a.kv_len || a.block_table || a.q_sq || a.xpack || a.soft_cap != 0.0f || a.norm_eps != 0.0f ||
        a.scratch_only || a.cap != a.Sk || (a.causal && a.Sq > a.Sk) || !aligned(a.q, 16) || !aligned(a.out, 16) ||
        !aligned(a.k, 16) || !aligned(a.v, 16) || !mfma_enabled())
        return ALJABR_ROCM_ERR_UNSUPPORTED;
    const long long rows = static_cast<long long>(a.Sq) * G;
    if (static_cast<double>(a.B) * a.Hkv * rows * a.Sk * a.D < static_cast<double>(kMinWork)) return ALJABR_ROCM_ERR_UNSUPPORTED;
    const long long ntiles = (static_cast<long long>(a.Sk) + kKeys - 1) / kKeys;
    const long long blocks = (rows + kRows - 1) / kRows * a.Hkv * a.B;
    const long long packs = ntiles * a.Hkv * a.B;
    if (rows > 0x3fffffff || blocks > 0xffffff || packs > 0x7fffffffLL) return ALJABR_ROCM_ERR_UNSUPPORTED;
    ChunkParams p{};
    p.q = a.q;
    p.k = static_cast<const _Float16 *>(a.k);
    p.v = static_cast<const _Float16 *>(a.v);
    p.out = a.out;
    p.B = a.B;
    p.Hq = a.Hq;
    p.Hkv = a.Hkv;
    p.G = G;
    p.Sq = a.Sq;
    p.Sk = a.Sk;
    p.scale = a.scale;
    p.causal = a.causal;
    p.ntiles = static_cast<int>(ntiles);
    p.row_blocks = static_cast<int>((rows + kRows - 1) / kRows);
    // Key splits: one workgroup per CU, of at least four tiles each.
    const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
    long long splits = (cus + blocks - 1) / blocks;
    if (splits > ntiles / 4) splits = ntiles / 4;
    if (splits < 1) splits = 1;
    p.tiles_per_split = static_cast<int>((ntiles + splits - 1) / splits);
    p.splits = static_cast<int>((ntiles + p.tiles_per_split - 1) / p.tiles_per_split);
    const size_t image = static_cast<size_t>(packs) * (a.D == 64 ? tile_halves<64>() : tile_halves<128>()) * 2;
    const size_t all = static_cast<size_t>(a.B) * a.Hq * a.Sq;
    const size_t part = p.splits > 1 ? all * p.splits * (a.D + 2) * sizeof(float) : 0;
    if (image + part > kMaxScratch) return ALJABR_ROCM_ERR_UNSUPPORTED;
    uint8_t *buf = static_cast<uint8_t *>(stream_scratch_try(image + part, kScratchPartials));
    if (!buf) return ALJABR_ROCM_ERR_UNSUPPORTED;
    if (part) {
        p.part_o = reinterpret_cast<float *>(buf + image);
        p.part_ml = p.part_o + all * p.splits * a.D;
    }
    hipStream_t s = current_stream();
    if (a.D == 64) launch<64>(p, reinterpret_cast<_Float16 *>(buf), s);
    else launch<128>(p, reinterpret_cast<_Float16 *>(buf), s);
    if (part) enqueue_attention_merge(a, p.part_o, p.part_ml, p.splits);
    return ALJABR_ROCM_OK;
}

}  // namespace aljabr
