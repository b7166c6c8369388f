// Key prepack and per-token append of PopKV retrieval metadata (gfx950).
//
// head_dim 128, token groups of 8 .. 128 (powers of two): pack128_block_kernel
// (pack128_block in pack128.h), one workgroup per 64 rows (128 for 128-token
// groups).  Other group sizes, one short group and the append: pack128_kernel,
// one workgroup per (KV head, token group), one wave per chunk of max(G, 32)
// dimensions (pack128_group in pack128.h).  In both, the extrema of each dimension over
// its token group come first (thresholds 0.5*max / 0.5*min in LDS), then one
// token per lane: the sign/magnitude words and the representatives, reduced
// in one lane's registers in the production tree order, so the bit-exact
// sums need no cross-lane shuffles.  Other head sizes of whole 32-dimension
// words: pack_rows_kernel, one workgroup per 64 rows, a lane per (token,
// chunk).  Everything else (pack_kernel) uses 256 threads per group:
// per-dimension extrema by (dimension, token stripe), then one token per
// thread.
//
// Semantics follow the reference packers: popkv_ext.cu:79-143 (G32),
// :376-500 (fused G16/G64, head_dim 128), :283-374 (generic G16/G64), with
// output rows token_offset + t (the in-place append of :1075-1092,
// :1177-1206).
#include <type_traits>

#include "device_common.h"
#include "kernels.h"
#include "pack128.h"

namespace popkv {
namespace {

constexpr int kPackThreads = 256;
constexpr int kMaxStaticLds = 64 * 1024;  // LDS a launch may ask for without an attribute

// Encodes one chunk of CH = max(G, 32) dimensions of one token.
// dims [c0, c0 + CH); `valid_d` = number of real dims in the head.
template <typename T, int G, bool FAST>
__device__ __forceinline__ void encode_chunk(const T* __restrict__ row, int c0, int d,
                                             const float* s_hi, const float* s_lo,
                                             uint32_t* sw, uint32_t* mw, float* lows, float* deltas) {
    constexpr int CH = G > 32 ? G : 32;
    float v[CH];
    if constexpr (FAST) {
#pragma unroll
        for (int i = 0; i < CH; i += 8) load8<T>(row + c0 + i, v + i);
    } else {
#pragma unroll
        for (int i = 0; i < CH; ++i) v[i] = (c0 + i < d) ? Elem<T>::load(row, c0 + i) : 0.0f;
    }
    bool mag[CH];
#pragma unroll
    for (int wi = 0; wi < CH / 32; ++wi) {
        uint32_t s = 0, m = 0;
#pragma unroll
        for (int j = 0; j < 32; ++j) {
            const int i = wi * 32 + j;
            const int dim = FAST ? c0 + i : min(c0 + i, 255);
            const bool valid = FAST || (c0 + i) < d;
            const bool sg = valid && v[i] >= 0.0f;
            const bool mg = valid && (sg ? (v[i] > s_hi[dim]) : (v[i] < s_lo[dim]));
            mag[i] = mg;
            s |= static_cast<uint32_t>(sg) << j;
            m |= static_cast<uint32_t>(mg) << j;
        }
        sw[wi] = s;
        mw[wi] = m;
    }
#pragma unroll
    for (int rr = 0; rr < CH / G; ++rr) {
        float xl[G], xh[G];
        int ln = 0, hn = 0;
#pragma unroll
        for (int j = 0; j < G; ++j) {
            const int i = rr * G + j;
            const bool valid = FAST || (c0 + i) < d;
            const float a = fabsf(v[i]);
            xl[j] = (valid && !mag[i]) ? a : 0.0f;
            xh[j] = (valid && mag[i]) ? a : 0.0f;
            ln += (valid && !mag[i]) ? 1 : 0;
            hn += (valid && mag[i]) ? 1 : 0;
        }
        const float ls = rep_tree_sum<G>(xl);
        const float hs = rep_tree_sum<G>(xh);
        finish_rep(ls, ln, hs, hn, lows[rr], deltas[rr]);
    }
}

template <typename T, int G>
__global__ __launch_bounds__(kPackThreads) void pack_kernel(
    const T* __restrict__ keys, int64_t head_stride, int64_t tokens, int D, int tg,
    int32_t* __restrict__ k_sign, int32_t* __restrict__ k_mag,
    uint16_t* __restrict__ k_low, uint16_t* __restrict__ k_delta,
    int64_t cap, int64_t offset) {
    const int W = (D + 31) / 32;
    const int R = (D + G - 1) / G;
    const int64_t kvh = blockIdx.y;
    const int64_t gs = static_cast<int64_t>(blockIdx.x) * tg;
    const int64_t ge = min(gs + static_cast<int64_t>(tg), tokens);
    const T* base = keys + kvh * head_stride;

    __shared__ float s_hi[256], s_lo[256];
    __shared__ float s_mx[kPackThreads], s_mn[kPackThreads];

    // Phase 1: per-dimension extrema over the token group.
    const int tid = threadIdx.x;
    const int nstripe = kPackThreads / D;
    if (tid < nstripe * D) {
        const int dim = tid % D, stripe = tid / D;
        float mn = INFINITY, mx = -INFINITY;
        for (int64_t t = gs + stripe; t < ge; t += nstripe) {
            const float x = Elem<T>::load(base, t * D + dim);
            mn = fminf(mn, x);
            mx = fmaxf(mx, x);
        }
        s_mn[tid] = mn;
        s_mx[tid] = mx;
    }
    __syncthreads();
    if (tid < D) {
        float mn = s_mn[tid], mx = s_mx[tid];
        for (int s = 1; s < nstripe; ++s) {
            mn = fminf(mn, s_mn[s * D + tid]);
            mx = fmaxf(mx, s_mx[s * D + tid]);
        }
        s_lo[tid] = mn * 0.5f;
        s_hi[tid] = mx * 0.5f;
    }
    __syncthreads();

    // Phase 2: one token per lane.
    constexpr int CH = G > 32 ? G : 32;
    for (int64_t t = gs + tid; t < ge; t += kPackThreads) {
        const T* row = base + t * D;
        const int64_t orow = kvh * cap + offset + t;
        for (int c0 = 0; c0 < D; c0 += CH) {
            uint32_t sw[CH / 32], mw[CH / 32];
            float lows[CH / G], deltas[CH / G];
            encode_chunk<T, G, false>(row, c0, D, s_hi, s_lo, sw, mw, lows, deltas);
#pragma unroll
            for (int wi = 0; wi < CH / 32; ++wi) {
                const int w = c0 / 32 + wi;
                if (w < W) {
                    k_sign[orow * W + w] = static_cast<int32_t>(sw[wi]);
                    k_mag[orow * W + w] = static_cast<int32_t>(mw[wi]);
                }
            }
#pragma unroll
            for (int rr = 0; rr < CH / G; ++rr) {
                const int r = c0 / G + rr;
                if (r < R) {
                    k_low[orow * R + r] = f16_rne(lows[rr]);
                    k_delta[orow * R + r] = f16_rne(deltas[rr]);
                }
            }
        }
    }
}

// Two consecutive elements at an address aligned to the pair.
__device__ __forceinline__ float2 load_pair(const float* p) { return *reinterpret_cast<const float2*>(p); }
__device__ __forceinline__ float2 load_pair(const bf16_t* p) {
    const uint32_t u = *reinterpret_cast<const uint32_t*>(p);
    return make_float2(__uint_as_float(u << 16), __uint_as_float(u & 0xffff0000u));
}
__device__ __forceinline__ float2 load_pair(const f16_t* p) {
    const uint32_t u = *reinterpret_cast<const uint32_t*>(p);
    return make_float2(bits_f16(u & 0xffffu), bits_f16(u >> 16));
}

constexpr int kRowsBlock = 64;  // rows a workgroup of pack_rows_kernel takes at most
constexpr int kRowsStripe = 8;  // rows per extrema stripe

// LDS of pack_rows_kernel: the rows (16 bytes of padding each, so that lanes
// at one offset of neighbouring rows spread over the banks), the stripes'
// maxima and minima (4 floats of padding), and the packed rows.
__host__ __device__ constexpr int pack_rows_pitch(int d, int esize) { return d * esize + 16; }
__host__ __device__ constexpr int pack_rows_ext(int d) { return kRowsBlock / kRowsStripe * (d + 4); }
__host__ __device__ constexpr int pack_rows_lds(int d, int g, int esize) {
    return kRowsBlock * pack_rows_pitch(d, esize) + 2 * pack_rows_ext(d) * 4 + kRowsBlock * (2 * (d / 32) * 4 + 2 * (d / g) * 2);
}

// Prepack of head sizes other than 128 that whole chunks of CH = max(G, 32)
// dimensions fill: block (x, y) encodes rows [rpb x, rpb x + rpb) of KV head y,
// rpb the whole token groups (a multiple of 8 tokens each) within 64 rows.  A
// workgroup per token group that read each row by single elements, once for
// the extrema and once a lane, was bound by the latency of those loads with
// 32-token groups filling 32 of 256 encode lanes.  Here the rows cross memory
// once, 16 bytes a lane, into LDS; extrema run over stripes of 8 rows there;
// each (row, chunk) is a lane's; and the packed rows leave whole.
// Measured (8 heads, graph replay, the general kernel -> this one): 64
// dimensions, G32 / 32 tokens fp16, 8191 tokens 25.0 -> 8.3 us, 1000 tokens
// 20.2 -> 7.3; 96 dimensions, 16383 tokens, G16 / 32 tokens fp16 76.4 -> 19.5,
// G32 / 64 tokens bf16 63.6 -> 22.3; 64 dimensions, G64 / 64 tokens fp32, 16384
// tokens 53.0 -> 32.3; 256 dimensions, G32 / 32 tokens bf16, 8191 tokens 104 ->
// 29.7.
template <typename T, int G>
__global__ __launch_bounds__(kPackThreads) void pack_rows_kernel(
    const T* __restrict__ keys, int64_t head_stride, int64_t tokens, int d, int tg, int rpb,
    int32_t* __restrict__ k_sign, int32_t* __restrict__ k_mag, uint16_t* __restrict__ k_low,
    uint16_t* __restrict__ k_delta, int64_t cap, int64_t offset) {
    constexpr int CH = G > 32 ? G : 32;
    extern __shared__ __align__(16) char lds[];
    const int w = d / 32, r = d / G, pitch = pack_rows_pitch(d, sizeof(T)), ext_pitch = d + 4;
    float* s_mx = reinterpret_cast<float*>(lds + kRowsBlock * pitch);
    float* s_mn = s_mx + pack_rows_ext(d);
    uint32_t* s_sign = reinterpret_cast<uint32_t*>(s_mn + pack_rows_ext(d));
    uint32_t* s_mag = s_sign + kRowsBlock * w;
    uint16_t* s_low = reinterpret_cast<uint16_t*>(s_mag + kRowsBlock * w);
    uint16_t* s_delta = s_low + kRowsBlock * r;

    const int tid = threadIdx.x, nt = blockDim.x;
    const int64_t kvh = blockIdx.y, gs = static_cast<int64_t>(blockIdx.x) * rpb;
    const int n = static_cast<int>(min(static_cast<int64_t>(rpb), tokens - gs));
    const uint4* src = reinterpret_cast<const uint4*>(keys + kvh * head_stride + gs * d);
    const int vpr = d * static_cast<int>(sizeof(T)) / 16;
    for (int i = tid; i < n * vpr; i += nt)
        *reinterpret_cast<uint4*>(lds + i / vpr * pitch + i % vpr * 16) = src[i];
    __syncthreads();

    // extrema of each stripe and pair of dimensions
    const int stripes = (n + kRowsStripe - 1) / kRowsStripe, pairs = d / 2;
    for (int i = tid; i < stripes * pairs; i += nt) {
        const int st = i / pairs, dim = i % pairs * 2, t0 = st * kRowsStripe;
        float2 mx = make_float2(-INFINITY, -INFINITY), mn = make_float2(INFINITY, INFINITY);
#pragma unroll
        for (int j = 0; j < kRowsStripe; ++j) {
            // past the end: the last row again
            const float2 x = load_pair(reinterpret_cast<const T*>(lds + min(t0 + j, n - 1) * pitch) + dim);
            mx = make_float2(fmaxf(mx.x, x.x), fmaxf(mx.y, x.y));
            mn = make_float2(fminf(mn.x, x.x), fminf(mn.y, x.y));
        }
        *reinterpret_cast<float2*>(s_mx + st * ext_pitch + dim) = mx;
        *reinterpret_cast<float2*>(s_mn + st * ext_pitch + dim) = mn;
    }
    __syncthreads();
    // each token group's thresholds, in its first stripe's place
    const int spg = tg / kRowsStripe, groups = (n + tg - 1) / tg;
    for (int i = tid; i < groups * d; i += nt) {
        const int first = i / d * spg, last = min(first + spg, stripes), dim = i % d;
        float mx = s_mx[first * ext_pitch + dim], mn = s_mn[first * ext_pitch + dim];
        for (int st = first + 1; st < last; ++st) {
            mx = fmaxf(mx, s_mx[st * ext_pitch + dim]);
            mn = fminf(mn, s_mn[st * ext_pitch + dim]);
        }
        s_mx[first * ext_pitch + dim] = mx * 0.5f;
        s_mn[first * ext_pitch + dim] = mn * 0.5f;
    }
    __syncthreads();

    for (int i = tid; i < d / CH * kRowsBlock; i += nt) {
        const int t = i % kRowsBlock, c0 = i / kRowsBlock * CH;
        if (t >= n) continue;
        const int ext = t / tg * spg * ext_pitch;
        uint32_t sw[CH / 32], mw[CH / 32];
        float lows[CH / G], deltas[CH / G];
        encode_chunk<T, G, true>(reinterpret_cast<const T*>(lds + t * pitch), c0, d, s_mx + ext, s_mn + ext, sw, mw,
                                 lows, deltas);
#pragma unroll
        for (int wi = 0; wi < CH / 32; ++wi) {
            s_sign[t * w + c0 / 32 + wi] = sw[wi];
            s_mag[t * w + c0 / 32 + wi] = mw[wi];
        }
#pragma unroll
        for (int rr = 0; rr < CH / G; ++rr) {
            s_low[t * r + c0 / G + rr] = f16_rne(lows[rr]);
            s_delta[t * r + c0 / G + rr] = f16_rne(deltas[rr]);
        }
    }
    __syncthreads();
    const int64_t orow = kvh * cap + offset + gs;
    for (int i = tid; i < n * w; i += nt) {
        k_sign[orow * w + i] = static_cast<int32_t>(s_sign[i]);
        k_mag[orow * w + i] = static_cast<int32_t>(s_mag[i]);
    }
    for (int i = tid; i < n * r; i += nt) {
        k_low[orow * r + i] = s_low[i];
        k_delta[orow * r + i] = s_delta[i];
    }
}

// Prefix prepack (APPEND false): block (x, y) encodes token group x of KV
// head y, rows [x*tg, min(x*tg + tg, tokens)) of `keys`, into packed rows
// y*cap + offset + x*tg + t, for the group sizes pack128_block does not
// take and for one group of up to 64 rows.  Fused append (APPEND true): block i appends
// the new token of (sequence, KV head) i (pack128_append).  STAGE (16-bit
// rows; tg <= 64 at G 64, tg <= 128 at G 32 / G 16): the group's rows are
// read from memory once, into LDS, and the encode pass reads them there.
template <typename T, int G, bool APPEND, bool STAGE = false>
__global__ __launch_bounds__(kWave * pack128_waves<G>()) void pack128_kernel(
    const T* __restrict__ keys, int64_t head_stride, int64_t tokens, int tg,
    int32_t* __restrict__ k_sign, int32_t* __restrict__ k_mag,
    uint16_t* __restrict__ k_low, uint16_t* __restrict__ k_delta, int64_t cap, int64_t offset,
    AppendArgs<T> ap) {
    constexpr int D = 128;
    static_assert(2 * D * static_cast<int>(sizeof(T)) / 16 <= kWave * pack128_waves<G>(),
                  "one 16-byte slice of the new K/V rows per thread");
    if constexpr (APPEND)
        args_in_sgprs(ap.counts, ap.kv_heads, ap.cache_rows, ap.new_k, ap.new_v, ap.key_cache, ap.value_cache, tg,
                      k_sign, k_mag, k_low, k_delta, cap);
    else
        args_in_sgprs(keys, head_stride, tokens, tg, k_sign, k_mag, k_low, k_delta, cap, offset);
    if constexpr (!APPEND) {
        const int64_t kvh = blockIdx.y;
        const int64_t gs = static_cast<int64_t>(blockIdx.x) * tg;
        const int n = static_cast<int>(min(gs + static_cast<int64_t>(tg), tokens) - gs);
        const T* base = keys + kvh * head_stride + gs * D;
        auto row_of = [&](int t) -> const T* { return base + static_cast<int64_t>(t) * D; };
        pack128_group<T, G, false, STAGE>(row_of, n, kvh * cap + offset + gs, k_sign, k_mag, k_low, k_delta);
    } else {
        pack128_append<T, G, false, STAGE>(blockIdx.x, ap, tg, k_sign, k_mag, k_low, k_delta, cap);
    }
}

// The append of several layers in one launch (StagePointers): block (KV head
// x, layer y) copies its active rows and the new key to the staged rows and
// encodes them.  A launch per layer, of 8 workgroups each, left the chip idle
// and the host bound: 30 layers of 8 heads, 78-token groups at G16 6.4 us of
// kernel and two launches a layer (610 us for the token); now one launch of 9.1
// us (144 us, the host collecting pointers).
template <typename T, int G, bool STAGE>
__global__ __launch_bounds__(kWave * pack128_waves<G>()) void stage_append_kernel(StagePointers p, int n_active,
                                                                                  int64_t cap, int64_t sealed) {
    constexpr int D = 128, VPR = D * static_cast<int>(sizeof(T)) / 16, NT = kWave * pack128_waves<G>();
    const int kvh = blockIdx.x, layer = blockIdx.y, n = n_active + 1;
    const T* active = static_cast<const T*>(p.active[layer]) + static_cast<int64_t>(kvh) * n_active * D;
    const T* last = static_cast<const T*>(p.new_k[layer]) + static_cast<int64_t>(kvh) * D;
    uint4* staged = reinterpret_cast<uint4*>(static_cast<T*>(p.staged[layer]) + static_cast<int64_t>(kvh) * n * D);
    auto row_of = [&](int t) -> const T* { return t == n_active ? last : active + static_cast<int64_t>(t) * D; };
    for (int i = threadIdx.x; i < n * VPR; i += NT)
        staged[i] = reinterpret_cast<const uint4*>(row_of(i / VPR))[i % VPR];
    pack128_group<T, G, false, STAGE>(row_of, n, kvh * cap + sealed, p.k_sign[layer], p.k_mag[layer],
                                      static_cast<uint16_t*>(p.k_low[layer]), static_cast<uint16_t*>(p.k_delta[layer]));
}

template <typename T, int G>
hipError_t launch_stage_append_t(const StagePointers& p, int layers, int kv_heads, int active_tokens, int64_t capacity,
                                 int64_t sealed, int tg, hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>(kv_heads), static_cast<unsigned>(layers)), block(kWave * pack128_waves<G>());
    constexpr bool kStageable = sizeof(T) == 2;
    if (kStageable && tg <= (G == 64 ? 64 : 128))
        hipLaunchKernelGGL((stage_append_kernel<T, G, kStageable>), grid, block, 0, stream, p, active_tokens, capacity,
                           sealed);
    else
        hipLaunchKernelGGL((stage_append_kernel<T, G, false>), grid, block, 0, stream, p, active_tokens, capacity,
                           sealed);
    return hipGetLastError();
}

// Prefix prepack for token groups of TG = 8 .. 128: block (x, y) encodes rows
// [ROWS x, ROWS x + ROWS) of KV head y (pack128_block).
template <typename T, int G, int TG, bool STAGE>
__global__ __launch_bounds__((pack128_block_threads<G, TG>())) void pack128_block_kernel(
    const T* __restrict__ keys, int64_t head_stride, int64_t tokens, int32_t* __restrict__ k_sign,
    int32_t* __restrict__ k_mag, uint16_t* __restrict__ k_low, uint16_t* __restrict__ k_delta, int64_t cap,
    int64_t offset) {
    args_in_sgprs(keys, head_stride, tokens, k_sign, k_mag, k_low, k_delta, cap, offset);
    const int64_t kvh = blockIdx.y;
    const int64_t gs = static_cast<int64_t>(blockIdx.x) * pack128_block_rows(TG);
    const int n = static_cast<int>(min(static_cast<int64_t>(pack128_block_rows(TG)), tokens - gs));
    pack128_block<T, G, TG, STAGE>(keys + kvh * head_stride + gs * 128, n, kvh * cap + offset + gs, k_sign, k_mag,
                                   k_low, k_delta);
}

template <typename T, int G, int TG>
hipError_t launch_pack_block(const T* keys, int64_t kvh, int64_t tokens, int64_t head_stride, int32_t* ks, int32_t* km,
                             uint16_t* kl, uint16_t* kd, int64_t cap, int64_t off, hipStream_t stream) {
    constexpr int rows = pack128_block_rows(TG);
    const dim3 grid(static_cast<unsigned>((tokens + rows - 1) / rows), static_cast<unsigned>(kvh));
    const dim3 block(pack128_block_threads<G, TG>());
    constexpr bool kStage = sizeof(T) == 2 || TG <= 64;
    hipLaunchKernelGGL((pack128_block_kernel<T, G, TG, kStage>), grid, block, 0, stream,
                       keys, head_stride, tokens, ks, km, kl, kd, cap, off);
    return hipGetLastError();
}

template <typename T, int G>
hipError_t launch_pack_t(const T* keys, int64_t kvh, int64_t tokens, int d, int64_t head_stride,
                         int32_t* ks, int32_t* km, uint16_t* kl, uint16_t* kd, int64_t cap, int64_t off,
                         int tg, hipStream_t stream) {
    const int64_t groups = (tokens + tg - 1) / tg;
    dim3 grid(static_cast<unsigned>(groups), static_cast<unsigned>(kvh));
    const bool fast = d == 128 && (reinterpret_cast<uintptr_t>(keys) % 16 == 0) &&
                      ((head_stride * static_cast<int64_t>(sizeof(T))) % 16 == 0) &&
                      (reinterpret_cast<uintptr_t>(ks) % 16 == 0) && (reinterpret_cast<uintptr_t>(km) % 16 == 0) &&
                      (reinterpret_cast<uintptr_t>(kl) % 16 == 0) && (reinterpret_cast<uintptr_t>(kd) % 16 == 0);
    constexpr bool kStageable = sizeof(T) == 2;
    // the block form (figures at pack128_block), but for one group of up to 64
    // rows (a short prefix, the append of one layer): there a workgroup is
    // the group either way, and the block's 128-row workgroup half empty
    // (us, block and group form, 64 tokens x 8 heads in 128-token groups: G16
    // fp32 5.32 / 4.90, G32 fp32 5.23 / 4.62, G64 bf16 5.71 / 5.57; 100 tokens 6.0 / 6.4)
    if (fast && (tokens > tg || tokens > 64)) {
        switch (tg) {
            case 8: return launch_pack_block<T, G, 8>(keys, kvh, tokens, head_stride, ks, km, kl, kd, cap, off, stream);
            case 16: return launch_pack_block<T, G, 16>(keys, kvh, tokens, head_stride, ks, km, kl, kd, cap, off, stream);
            case 32: return launch_pack_block<T, G, 32>(keys, kvh, tokens, head_stride, ks, km, kl, kd, cap, off, stream);
            case 64: return launch_pack_block<T, G, 64>(keys, kvh, tokens, head_stride, ks, km, kl, kd, cap, off, stream);
            case 128: return launch_pack_block<T, G, 128>(keys, kvh, tokens, head_stride, ks, km, kl, kd, cap, off, stream);
            default: break;  // any other size: one group per workgroup
        }
    }
    if (fast && kStageable && tg <= (G == 64 ? 64 : 128))
        hipLaunchKernelGGL((pack128_kernel<T, G, false, kStageable>), grid, dim3(kWave * pack128_waves<G>()), 0,
                           stream, keys, head_stride, tokens, tg, ks, km, kl, kd, cap, off, AppendArgs<T>{});
    else if (fast)
        hipLaunchKernelGGL((pack128_kernel<T, G, false>), grid, dim3(kWave * pack128_waves<G>()), 0, stream, keys,
                           head_stride, tokens, tg, ks, km, kl, kd, cap, off, AppendArgs<T>{});
    else if (d % (G > 32 ? G : 32) == 0 && tg % kRowsStripe == 0 && tg <= kRowsBlock &&
             pack_rows_lds(d, G, sizeof(T)) <= kMaxStaticLds && reinterpret_cast<uintptr_t>(keys) % 16 == 0 &&
             (head_stride * static_cast<int64_t>(sizeof(T))) % 16 == 0) {
        // whole chunks, whole stripes and 16-byte rows that fit LDS; the rest
        // (partial words, other groups, fp32 rows of 192 dimensions and more) keeps
        // the general kernel
        const int rpb = kRowsBlock / tg * tg, items = d / (G > 32 ? G : 32) * kRowsBlock;
        hipLaunchKernelGGL((pack_rows_kernel<T, G>), dim3(static_cast<unsigned>((tokens + rpb - 1) / rpb), grid.y),
                           dim3(items < kPackThreads ? items : kPackThreads), pack_rows_lds(d, G, sizeof(T)), stream,
                           keys, head_stride, tokens, d, tg, rpb, ks, km, kl, kd, cap, off);
    } else
        hipLaunchKernelGGL((pack_kernel<T, G>), grid, dim3(kPackThreads), 0, stream, keys, head_stride,
                           tokens, d, tg, ks, km, kl, kd, cap, off);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_pack_g(const T* keys, int64_t kvh, int64_t tokens, int d, int64_t hs, int32_t* ks,
                         int32_t* km, uint16_t* kl, uint16_t* kd, int64_t cap, int64_t off, int tg, int g,
                         hipStream_t stream) {
    switch (g) {
        case 16: return launch_pack_t<T, 16>(keys, kvh, tokens, d, hs, ks, km, kl, kd, cap, off, tg, stream);
        case 32: return launch_pack_t<T, 32>(keys, kvh, tokens, d, hs, ks, km, kl, kd, cap, off, tg, stream);
        default: return launch_pack_t<T, 64>(keys, kvh, tokens, d, hs, ks, km, kl, kd, cap, off, tg, stream);
    }
}

template <typename T>
hipError_t launch_append_t(const AppendArgs<T>& ap, int64_t rows, int tg, int g, int32_t* ks, int32_t* km,
                           uint16_t* kl, uint16_t* kd, int64_t cap, hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>(rows));
    switch (g) {
        case 16:
            hipLaunchKernelGGL((pack128_kernel<T, 16, true>), grid, dim3(kWave * pack128_waves<16>()), 0, stream,
                               nullptr, 0, 0, tg, ks, km, kl, kd, cap, 0, ap);
            break;
        case 32:
            hipLaunchKernelGGL((pack128_kernel<T, 32, true>), grid, dim3(kWave * pack128_waves<32>()), 0, stream,
                               nullptr, 0, 0, tg, ks, km, kl, kd, cap, 0, ap);
            break;
        default:
            if constexpr (sizeof(T) == 2) {
                if (tg <= 64) {
                    hipLaunchKernelGGL((pack128_kernel<T, 64, true, true>), grid, dim3(kWave * pack128_waves<64>()), 0,
                                       stream, nullptr, 0, 0, tg, ks, km, kl, kd, cap, 0, ap);
                    break;
                }
            }
            hipLaunchKernelGGL((pack128_kernel<T, 64, true>), grid, dim3(kWave * pack128_waves<64>()), 0, stream,
                               nullptr, 0, 0, tg, ks, km, kl, kd, cap, 0, ap);
            break;
    }
    return hipGetLastError();
}

template <typename T>
hipError_t launch_append_dt(const void* new_k, const void* new_v, void* key_cache, void* value_cache,
                            int64_t cache_rows, const int64_t* counts, int64_t batch, int kv_heads, int32_t* k_sign,
                            int32_t* k_mag, uint16_t* k_low, uint16_t* k_delta, int64_t capacity, int tg, int g,
                            int32_t* status, hipStream_t stream) {
    AppendArgs<T> ap;
    ap.new_k = static_cast<const T*>(new_k);
    ap.new_v = static_cast<const T*>(new_v);
    ap.key_cache = static_cast<T*>(key_cache);
    ap.value_cache = static_cast<T*>(value_cache);
    ap.cache_rows = cache_rows;
    ap.counts = counts;
    ap.kv_heads = kv_heads;
    ap.status = status;
    return launch_append_t<T>(ap, batch * kv_heads, tg, g, k_sign, k_mag, k_low, k_delta, capacity, stream);
}

}  // namespace

hipError_t launch_append(const void* new_k, const void* new_v, int dtype, void* key_cache, void* value_cache,
                         int64_t cache_rows, const int64_t* counts, int64_t batch, int kv_heads, int32_t* k_sign,
                         int32_t* k_mag, uint16_t* k_low, uint16_t* k_delta, int64_t capacity,
                         int token_group_size, int dim_group_size, int32_t* status, hipStream_t stream) {
    if (batch <= 0 || kv_heads <= 0) return hipSuccess;
    switch (dtype) {
        case POPKV_DTYPE_F32:
            return launch_append_dt<float>(new_k, new_v, key_cache, value_cache, cache_rows, counts, batch, kv_heads,
                                           k_sign, k_mag, k_low, k_delta, capacity, token_group_size,
                                           dim_group_size, status, stream);
        case POPKV_DTYPE_F16:
            return launch_append_dt<f16_t>(new_k, new_v, key_cache, value_cache, cache_rows, counts, batch, kv_heads,
                                           k_sign, k_mag, k_low, k_delta, capacity, token_group_size,
                                           dim_group_size, status, stream);
        default:
            return launch_append_dt<bf16_t>(new_k, new_v, key_cache, value_cache, cache_rows, counts, batch,
                                            kv_heads, k_sign, k_mag, k_low, k_delta, capacity, token_group_size,
                                            dim_group_size, status, stream);
    }
}

hipError_t launch_stage_append(const StagePointers& ptrs, int layers, int dtype, int kv_heads, int active_tokens,
                               int64_t capacity, int64_t sealed, int token_group_size, int dim_group_size,
                               hipStream_t stream) {
    auto typed = [&](auto elem) {
        using T = decltype(elem);
        switch (dim_group_size) {
            case 16: return launch_stage_append_t<T, 16>(ptrs, layers, kv_heads, active_tokens, capacity, sealed, token_group_size, stream);
            case 32: return launch_stage_append_t<T, 32>(ptrs, layers, kv_heads, active_tokens, capacity, sealed, token_group_size, stream);
            default: return launch_stage_append_t<T, 64>(ptrs, layers, kv_heads, active_tokens, capacity, sealed, token_group_size, stream);
        }
    };
    switch (dtype) {
        case POPKV_DTYPE_F32: return typed(float{});
        case POPKV_DTYPE_F16: return typed(f16_t{});
        default: return typed(bf16_t{});
    }
}

hipError_t launch_pack(const void* keys, int dtype, int64_t kv_heads, int64_t tokens, int head_dim,
                       int64_t key_head_stride, int32_t* k_sign, int32_t* k_mag, uint16_t* k_low,
                       uint16_t* k_delta, int64_t capacity, int64_t token_offset, int token_group_size,
                       int dim_group_size, hipStream_t stream) {
    if (tokens <= 0) return hipSuccess;
    switch (dtype) {
        case POPKV_DTYPE_F32:
            return launch_pack_g(static_cast<const float*>(keys), kv_heads, tokens, head_dim, key_head_stride,
                                 k_sign, k_mag, k_low, k_delta, capacity, token_offset, token_group_size,
                                 dim_group_size, stream);
        case POPKV_DTYPE_F16:
            return launch_pack_g(static_cast<const f16_t*>(keys), kv_heads, tokens, head_dim, key_head_stride,
                                 k_sign, k_mag, k_low, k_delta, capacity, token_offset, token_group_size,
                                 dim_group_size, stream);
        default:
            return launch_pack_g(static_cast<const bf16_t*>(keys), kv_heads, tokens, head_dim, key_head_stride,
                                 k_sign, k_mag, k_low, k_delta, capacity, token_offset, token_group_size,
                                 dim_group_size, stream);
    }
}

}  // namespace popkv
