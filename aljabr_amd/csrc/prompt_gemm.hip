// prompt_gemm.hip - the prompt GEMM's activation image, plan and dispatch
// (the kernels: prompt_gemm.hpp and prompt_{nf4,q40,q80,q4k,q6k}.hip).
#include <algorithm>

#include "prompt_gemm.hpp"

namespace aljabr {

template <> void prompt_pack<kPgNF4>(const PgArgs &, hipStream_t);
template <> void prompt_pack<kPgQ40>(const PgArgs &, hipStream_t);
template <> void prompt_pack<kPgQ80>(const PgArgs &, hipStream_t);
template <> void prompt_pack<kPgQ4K>(const PgArgs &, hipStream_t);
template <> void prompt_pack<kPgQ6K>(const PgArgs &, hipStream_t);
template <> void prompt_multiply<kPgNF4>(const PgArgs &, int, int, hipStream_t);
template <> void prompt_multiply<kPgQ40>(const PgArgs &, int, int, hipStream_t);
template <> void prompt_multiply<kPgQ80>(const PgArgs &, int, int, hipStream_t);
template <> void prompt_multiply<kPgQ4K>(const PgArgs &, int, int, hipStream_t);
template <> void prompt_multiply<kPgQ6K>(const PgArgs &, int, int, hipStream_t);

namespace {

using pg::half8;

// The activations as A fragments: [chunk kb][32-token tile][step j][lane] of
// 8 fp16, lane l = 32h + i holding token 32*tile + i, elements 64kb + 16j +
// 8h + e (NF4 order: 64kb + 32h + 8j + e), zero past M and K; hi = fp16(x)
// and, with xl, lo = fp16(x - hi). One workgroup per (chunk, tile), one wave
// per step. With sums (Q4_K): the sums of each 32-element sub-block of what
// the parts hold, split hi / lo (lane half 0 / 1), [super-block][tile][lane]
// of 8 sub-blocks.
__global__ __launch_bounds__(256) void prompt_pack_kernel(const float *x, u32x4 *xh, u32x4 *xl, _Float16 *sums, int M,
                                                          int K, int tiles, int nf4, const float *scale) {
    __shared__ double part[4][64];
    const int tid = threadIdx.x, lane = tid & 63, j = tid >> 6, h = lane >> 5, i = lane & 31;
    const int tile = blockIdx.x % tiles, kb = blockIdx.x / tiles;
    const int m = 32 * tile + i;
    const int k = 64 * kb + (nf4 ? 32 * h + 8 * j : 16 * j + 8 * h);
    float4 a = {0.0f, 0.0f, 0.0f, 0.0f}, b = a;
    if (m < M && k < K) {                            // K % 32 == 0: the 8 elements are in or out together
        const float4 *src = reinterpret_cast<const float4 *>(x + static_cast<size_t>(m) * K + k);
        a = src[0];
        b = src[1];
    }
    float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    if (scale && m < M) {
        const float inv = 1.0f / scale[m];           // powers of two: exact
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] *= inv;
    }
    half8 hi, lo;
    double t = 0.0;                              // the min term is several times the result: no rounding here
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        hi[e] = static_cast<_Float16>(v[e]);
        lo[e] = isinf(static_cast<float>(hi[e])) ? static_cast<_Float16>(0.0f)
                                                 : static_cast<_Float16>(v[e] - static_cast<float>(hi[e]));
        t += static_cast<double>(xl ? v[e] : static_cast<float>(hi[e]));
    }
    const size_t at = (static_cast<size_t>(blockIdx.x) * 4 + j) * 64 + lane;
    xh[at] = __builtin_bit_cast(u32x4, hi);
    if (xl) xl[at] = __builtin_bit_cast(u32x4, lo);
    if (!sums) return;
    part[j][lane] = t;
    __syncthreads();
    if (tid < 64) {
        const int sb = tid >> 5;                     // sub-block of the chunk: steps 2sb and 2sb + 1
        const double s = (part[2 * sb][i] + part[2 * sb][32 + i]) + (part[2 * sb + 1][i] + part[2 * sb + 1][32 + i]);
        const _Float16 sh = static_cast<_Float16>(static_cast<float>(s));
        _Float16 *dst = sums + ((static_cast<size_t>(kb >> 2) * tiles + tile) * 64 + i) * 8 + 2 * (kb & 3) + sb;
        dst[0] = sh;
        dst[32 * 8] = static_cast<_Float16>(static_cast<float>(s - static_cast<double>(sh)));
    }
}

// Y = the K slices' partial sums, added in double: up to 32 of them would add
// as many roundings to the result as the slices save. Loads in flight as in
// slice_sum (device.hpp).
template <int U>
__device__ __forceinline__ double slice_sum_f64(const float *p, size_t stride, int slices) {
    double acc = 0.0;
    for (int s0 = 0; s0 < slices; s0 += U) {
        float v[U];
#pragma unroll
        for (int j = 0; j < U; ++j) v[j] = p[static_cast<size_t>(min(s0 + j, slices - 1)) * stride];
#pragma unroll
        for (int j = 0; j < U; ++j)
            if (s0 + j < slices) acc += static_cast<double>(v[j]);
    }
    return acc;
}

// The arguments fill the 14 preloaded dwords.
__global__ __launch_bounds__(256) void prompt_sum_kernel(const float *part, int M, int N, int slices, int nseg, float *y0,
                                                         float *y1, float *y2, int end0, int end1) {
    const int n = blockIdx.x * 256 + threadIdx.x, m = blockIdx.y;
    if (n >= N) return;
    const float *p = part + static_cast<size_t>(m) * N + n;
    const size_t stride = static_cast<size_t>(M) * N;
    const double v = slices <= 4   ? slice_sum_f64<4>(p, stride, slices)
                     : slices <= 8 ? slice_sum_f64<8>(p, stride, slices)
                                   : slice_sum_f64<16>(p, stride, slices);
    const int s = min((n >= end0) + (n >= end1), nseg - 1);
    const int start = s == 0 ? 0 : s == 1 ? end0 : end1;
    const int rows = (s == nseg - 1 ? N : s == 0 ? end0 : end1) - start;
    (s == 0 ? y0 : s == 1 ? y1 : y2)[static_cast<size_t>(m) * rows + (n - start)] = static_cast<float>(v);
}

// What a call holds of the stream's scratch: the activation image of a pass of
// tokens, the weight image of a panel of rows, the K slices' partial sums over
// all panels.
constexpr int kPassTokens = 4096;
constexpr size_t kImageBytes = size_t{512} << 20;     // bounds the activation image
constexpr size_t kPanelBytes = size_t{128} << 20;     // bounds the weight image
constexpr float kPartialMb = 128.0f;                  // bounds the K slices' partial sums
constexpr size_t kMaxScratch = size_t{1} << 30;       // a call past it keeps the passes (K past 10^6)

// The plan's constants are fits of a sweep over tiles, slices and formats
// (4096 x 14336 and 2560-wide layers, 64 to 2048 tokens): a chunk of four
// token tiles took 1.65 us for two products (NF4, Q8_0), 2.4 us for Q6_K's
// three; the slice sum moves ~5 TB/s.
constexpr float kFixedUs = 3.0f, kReduceUs = 3.0f, kMbPerUs = 5.0f;

// Tiles of 32 tokens per wave (2 or 4) and K slices for M tokens over N
// stacked rows. Two tiles leave less idle in the last token group, four
// decode and read the weights half as often.
//
// K slices trade idle CUs and ragged last rounds against the partial sums'
// traffic: the least of rounds * (chunks * chunk time + fixed) + slice sum.
// N is the rows of one panel, `all` those whose partial sums are held.
struct Plan {
    int mt, mt_groups, n_groups, per, slices;
};

Plan make_plan(int f, int xp, int M, int N, int all, int chunks, int cus) {
    const int quantum = f == kPgQ4K || f == kPgQ6K ? 4 : 1;
    // Microseconds of a workgroup's chunk: 32 cycles per product and its share
    // of the decode and the scaling.
    const float products = f == kPgQ6K ? 3.0f : f == kPgQ4K ? 1.12f * xp : f == kPgNF4 ? 1.0f + xp : 2.0f;
    Plan best{};
    float best_us = 0.0f;
    const float out_mb = 4e-6f * static_cast<float>(M) * static_cast<float>(N);
    const float held_mb = 4e-6f * static_cast<float>(M) * static_cast<float>(all);
    const int n_groups = (N + 64 * kPgWaves - 1) / (64 * kPgWaves);
    for (int mt = 4; mt >= 2; mt -= 2) {
        const float chunk_us = (0.4f + 0.68f * products) * (mt == 4 ? 1.0f : 0.55f);
        const int mt_groups = (M + 32 * mt - 1) / (32 * mt);
        for (int s = 1; s <= 32; ++s) {
            if (s > 1 && (s * held_mb > kPartialMb || chunks / s < quantum)) break;
            Plan p{mt, mt_groups, n_groups, 0, 0};
            p.per = (chunks + s - 1) / s;
            p.per = (p.per + quantum - 1) / quantum * quantum;
            p.slices = (chunks + p.per - 1) / p.per;
            const long long rounds = (static_cast<long long>(mt_groups) * n_groups * p.slices + cus - 1) / cus;
            const float us = static_cast<float>(rounds) * (static_cast<float>(p.per) * chunk_us + kFixedUs) +
                             (p.slices > 1 ? kReduceUs + static_cast<float>(2 * p.slices + 1) * out_mb / kMbPerUs : 0.0f);
            if (best_us == 0.0f || us < best_us) {
                best = p;
                best_us = us;
            }
        }
    }
    return best;
}

void pack_panel(int f, const PgArgs &a, hipStream_t s) {
    switch (f) {
    case kPgNF4: return prompt_pack<kPgNF4>(a, s);
    case kPgQ40: return prompt_pack<kPgQ40>(a, s);
    case kPgQ80: return prompt_pack<kPgQ80>(a, s);
    case kPgQ4K: return prompt_pack<kPgQ4K>(a, s);
    default: return prompt_pack<kPgQ6K>(a, s);
    }
}

void multiply_panel(int f, const PgArgs &a, int xp, int mt, hipStream_t s) {
    switch (f) {
    case kPgNF4: return prompt_multiply<kPgNF4>(a, xp, mt, s);
    case kPgQ40: return prompt_multiply<kPgQ40>(a, xp, mt, s);
    case kPgQ80: return prompt_multiply<kPgQ80>(a, xp, mt, s);
    case kPgQ4K: return prompt_multiply<kPgQ4K>(a, xp, mt, s);
    default: return prompt_multiply<kPgQ6K>(a, xp, mt, s);
    }
}

// Whether the passes that the call replaces run any of its tokens in fp32:
// shapes and alignments that the matrix-core passes do not take, and the last
// single token left by the GGUF passes of 8 or 32. Those tokens keep fp32's
// range and relative accuracy, so the rows are scaled (unscaled, an element
// past 65504 is infinite and one under 2^-14 loses its last bits).
bool fp32_passes(const RowsOut *outs, int nseg, int f, int K, int M) {
    bool aligned_all = true;
    for (int i = 0; i < nseg; ++i)
        aligned_all = aligned_all && (f == kPgNF4 ? aligned(outs[i].absmax, 8) : aligned(outs[i].w, 16));
    if (!aligned_all || K % (f == kPgNF4 ? 256 : 512) != 0) return true;
    return f == kPgNF4 ? false : M % (f == kPgQ40 || f == kPgQ80 ? 8 : 32) == 1;
}

}  // namespace

int enqueue_prompt_gemm(const RowsOut *outs, int nseg, const float *A, int K, int type, int xparts, int M) {
    const int f = type == ALJABR_ROCM_TYPE_NF4    ? kPgNF4
                  : type == ALJABR_ROCM_TYPE_Q4_0 ? kPgQ40
                  : type == ALJABR_ROCM_TYPE_Q8_0 ? kPgQ80
                  : type == ALJABR_ROCM_TYPE_Q4_K ? kPgQ4K
                  : type == ALJABR_ROCM_TYPE_Q6_K ? kPgQ6K
                                                  : -1;
    const int block = f == kPgNF4 ? 64 : f == kPgQ40 || f == kPgQ80 ? 32 : 256;
    if (f < 0 || nseg < 1 || nseg > 3 || M < 2 || K < block || K % block != 0 || !aligned(A, 16) || !mfma_enabled())
        return ALJABR_ROCM_ERR_UNSUPPORTED;
    PgArgs a{};
    long long end = 0;
    for (int i = 0; i < 3; ++i) {
        a.end[i] = 0x7fffffff;
        if (i >= nseg) continue;
        const RowsOut &o = outs[i];
        // NF4 codes are read 16 bytes at a time; the K-quants' callers refuse
        // weights off 16 bytes at every batch size.
        const size_t wa = f == kPgQ40 || f == kPgQ80 ? 4 : 16;
        if (o.n <= 0 || !aligned(o.w, wa) || (i < nseg - 1 && o.n % 32 != 0)) return ALJABR_ROCM_ERR_UNSUPPORTED;
        end += o.n;
        if (end > 0x7fff0000LL) return ALJABR_ROCM_ERR_UNSUPPORTED;
        a.w[i] = o.w;
        a.absmax[i] = o.absmax;
        a.end[i] = static_cast<int>(end);
    }
    // Q4_K's rows always are: a sub-block's sum of 32 activations leaves fp16's
    // range before they do, and its parts would be inf - inf. Scaled it is
    // below 2^14.
    const bool scaled = f == kPgQ4K || (xparts == 2 && fp32_passes(outs, nseg, f, K, M));
    a.nseg = nseg;
    a.N = static_cast<int>(end);
    a.K = K;
    a.chunks = (K + kPgChunk - 1) / kPgChunk;
    const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
    hipStream_t s = current_stream();
    // Weight image bytes of a row tile, and the panels that bound it.
    const size_t tile_codes = static_cast<size_t>(a.chunks) * (f == kPgQ80 || f == kPgQ6K ? 2048 : 1024);
    const size_t tile_aux = static_cast<size_t>(a.chunks) * (f == kPgQ6K ? 256 : 128) +
                            (f == kPgQ4K ? static_cast<size_t>(a.chunks / 4) * pg::kMinWords * 4 : 0);
    const int all_tiles = (a.N + 31) / 32;
    const int panels = static_cast<int>((all_tiles * (tile_codes + tile_aux) + kPanelBytes - 1) / kPanelBytes);
    const int panel = (all_tiles + panels - 1) / panels;
    const size_t image = (panel * (tile_codes + tile_aux) + 255) & ~size_t{255};
    const size_t fit = kImageBytes / (static_cast<size_t>(xparts) * a.chunks * 128) / 128 * 128;
    const int pass = static_cast<int>(std::min(static_cast<size_t>(kPassTokens), std::max(fit, size_t{128})));
    // Bytes of a pass: its planes, sub-block sums, row scales and partial sums.
    struct Layout {
        size_t plane, sums, scales, parts;
    };
    const auto layout = [&](const Plan &p, int mm) {
        const size_t tiles = static_cast<size_t>(p.mt_groups) * p.mt;
        return Layout{a.chunks * tiles * 4096, f == kPgQ4K ? (a.chunks / 4) * tiles * 1024 : 0,
                      scaled ? tiles * 32 * sizeof(float) : 0,
                      p.slices > 1 ? static_cast<size_t>(p.slices) * mm * a.N * sizeof(float) : 0};
    };
    const auto plan = [&](int mm) { return make_plan(f, xparts, mm, std::min(panel * 32, a.N), a.N, a.chunks, cus); };
    // One buffer for all passes, before any launch: a whole pass's and the
    // last one's, whose plan may take more slices.
    size_t bytes = 0;
    for (const int mm : {std::min(M, pass), (M - 1) % pass + 1}) {
        const Layout l = layout(plan(mm), mm);
        bytes = std::max(bytes, xparts * l.plane + l.sums + image + l.scales + l.parts);
    }
    if (bytes > kMaxScratch) return ALJABR_ROCM_ERR_UNSUPPORTED;
    uint8_t *buf = static_cast<uint8_t *>(stream_scratch_try(bytes, kScratchPartials));
    if (!buf) return ALJABR_ROCM_ERR_UNSUPPORTED;
    for (int m0 = 0; m0 < M; m0 += pass) {
        const int mm = std::min(M - m0, pass);
        const Plan p = plan(mm);
        const auto [plane, sums, scales, parts] = layout(p, mm);
        a.M = mm;
        a.per = p.per;
        a.slices = p.slices;
        a.mt_groups = p.mt_groups;
        a.tiles = p.mt_groups * p.mt;
        uint8_t *xl = xparts == 2 ? buf + plane : nullptr;
        uint8_t *next = buf + xparts * plane;
        a.xh = buf;
        a.xl = xl;
        a.sums = sums ? next : nullptr;
        a.codes = next + sums;
        a.scale = scaled ? reinterpret_cast<const float *>(next + sums + image) : nullptr;
        a.part = parts ? reinterpret_cast<float *>(next + sums + image + scales) : nullptr;
        for (int i = 0; i < nseg; ++i) a.y[i] = outs[i].y + static_cast<size_t>(m0) * outs[i].n;
        const float *x = A + static_cast<size_t>(m0) * K;
        a.x = x;
        for (a.tile0 = 0; a.tile0 < all_tiles; a.tile0 += panel) {
            a.ntiles = std::min(panel, all_tiles - a.tile0);
            a.n_groups = (a.ntiles + 2 * kPgWaves - 1) / (2 * kPgWaves);
            a.aux = reinterpret_cast<const uint32_t *>(a.codes + a.ntiles * tile_codes);
            a.scale_rows = scaled && a.tile0 == 0 ? mm : 0;
            pack_panel(f, a, s);
            if (a.tile0 == 0)
                hipLaunchKernelGGL(prompt_pack_kernel, dim3(static_cast<unsigned>(a.chunks * a.tiles)), dim3(256), 0, s, x,
                                   reinterpret_cast<u32x4 *>(buf), reinterpret_cast<u32x4 *>(xl),
                                   reinterpret_cast<_Float16 *>(const_cast<uint8_t *>(a.sums)), mm, K, a.tiles,
                                   f == kPgNF4, a.scale);
            multiply_panel(f, a, xparts, p.mt, s);
        }
        if (a.part)
            hipLaunchKernelGGL(prompt_sum_kernel, dim3(static_cast<unsigned>((a.N + 255) / 256), static_cast<unsigned>(mm)),
                               dim3(256), 0, s, a.part, mm, a.N, p.slices, nseg, a.y[0], a.y[1], a.y[2], a.end[0], a.end[1]);
    }
    return ALJABR_ROCM_OK;
}

}  // namespace aljabr
