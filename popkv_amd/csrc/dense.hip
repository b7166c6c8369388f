// Dense decode attention (the reference's full layers, popkv.py:1022-1038):
// every prefix token attends, one GQA group per workgroup so that each K/V
// row is read once for all its query heads; the current token joins in the
// merge.  head_dim 128, contiguous rows, query head h on KV head h / (QH /
// KVH).  The kernels are bound by the K/V stream: 16-bit types multiply Q.K
// on the matrix cores (attn_dense_mfma_kernel), fp32 takes the VALU
// (attn_dense_gqa_kernel); both merge the splits in the same launch.
#include "attention_common.h"
#include "device_common.h"
#include "kernels.h"

namespace popkv {
namespace {

// Merge of `n` <= 64 states (m, l, acc[128]) of one head, `step` states
// apart, by one wave; DPL dims per lane from d0 on (2: dims lane and lane +
// 64; 1: dim d0 + lane).  The states come from other workgroups of this
// launch (device-coherent loads), NF of them in flight at once.  LAST: with
// the current token's logit and value, num / den being the head's output;
// else (mx, den, num) is their state.
template <typename T, int DPL, bool LAST>
__device__ __forceinline__ void dense_merge(const float* __restrict__ ps, int step, int n, const T* __restrict__ qh,
                                            const T* __restrict__ ck, const T* __restrict__ cv, float scale, int d0,
                                            float& mx, float& den, float (&num)[DPL]) {
    constexpr int S = 128 + 2, NF = 32;
    const int lane = threadIdx.x & (kWave - 1);
    float q0 = 0.0f, q1 = 0.0f, k0 = 0.0f, k1 = 0.0f, v[DPL];
    if constexpr (LAST) {
        q0 = Elem<T>::load(qh, lane), q1 = Elem<T>::load(qh, lane + 64);
        k0 = Elem<T>::load(ck, lane), k1 = Elem<T>::load(ck, lane + 64);
#pragma unroll
        for (int i = 0; i < DPL; ++i) v[i] = Elem<T>::load(cv, d0 + lane + 64 * i);
    }
    float m = -INFINITY, l = 0.0f, a[NF][DPL];  // m, l: state `lane`'s
    if (lane < n) {
        m = ld_f32<true>(ps + static_cast<int64_t>(lane * step) * S);
        l = ld_f32<true>(ps + (static_cast<int64_t>(lane * step) * S + 1));
    }
    auto load_acc = [&](int b) {
#pragma unroll
        for (int j = 0; j < NF; ++j) {
            const float* src = ps + (static_cast<int64_t>(min(b + j, n - 1) * step) * S + 2 + d0 + lane);
#pragma unroll
            for (int i = 0; i < DPL; ++i) a[j][i] = ld_f32<true>(src + 64 * i);
        }
    };
    load_acc(0);
    mx = wave_max(m);
    float wc = 0.0f;
    if constexpr (LAST) {
        const float cur_m = wave_sum(q0 * k0 + q1 * k1) * scale;
        mx = fmaxf(mx, cur_m);
        wc = __expf(cur_m - mx);
    }
    const float w = m == -INFINITY ? 0.0f : __expf(m - mx);
#pragma unroll
    for (int i = 0; i < DPL; ++i) num[i] = LAST ? wc * v[i] : 0.0f;
    for (int b = 0; b < n; b += NF) {
        if (b > 0) load_acc(b);
        auto fold = [&](int j) {
            const float ws = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w), b + j));
#pragma unroll
            for (int i = 0; i < DPL; ++i) num[i] = fmaf(ws, a[j][i], num[i]);
        };
        // past n a[j] repeats the last state, which may hold an infinity: not
        // folded, not even with weight 0
#pragma unroll
        for (int j0 = 0; j0 < NF; j0 += 8) {
            if (b + j0 + 8 <= n) {
#pragma unroll
                for (int j = j0; j < j0 + 8; ++j) fold(j);
            } else {
#pragma unroll
                for (int j = j0; j < j0 + 8; ++j)
                    if (b + j < n) fold(j);
            }
        }
    }
    den = wave_sum(l * w) + wc;
}

// The fused merge, as in the layer step's select + attention kernel: the
// states went out with device-coherent stores; once this block's are
// acknowledged (the gfx942 / gfx950 rule stated at st_f32) it takes a ticket
// of its KV head (zero between calls, reset by the last taker), and the last
// block merges each of the group's heads (WAVES waves for QPK heads: a head
// takes one wave, or two of 64 dims each where there are enough).
//
// One block's bursts of coherent loads, each a memory latency, add up with
// the splits that few KV heads give (up to 256), so more than 64 splits merge
// in two levels: the last block of every set of 32 leaves the set's merged
// state in the place of its first one, and the last of the sets' blocks merges
// those.  Up to 64, two bursts cost less than the second hand-off.  Layer at
// 65536 tokens bf16, one level -> two: 1 KV head of 1 / 4 / 8 query heads
// (256 splits) 19.8 -> 13.9, 24.9 -> 17.0, 33.2 -> 19.9 us, 2 of 4 (128) 22.8
// -> 20.7; at 16384 tokens 4 of 4 (64) it took 17.1 against 15.7.
// Tickets: one per KV head; in two levels one per set and one for the sets, at
// most 12 for the 1 to 3 KV heads that give more than 64 splits (the region
// holds 64 at least).
constexpr int kDenseOneLevel = 64, kDenseSet = 32;

template <typename T, int QPK, int WAVES>
__device__ __forceinline__ void dense_finish(int g, int s, float* partials, int nsplit, uint32_t* tickets,
                                             const T* q, const T* cur_k, const T* cur_v, float scale, T* out) {
    constexpr int D = 128, S = D + 2;
    constexpr int DPL = 2 * QPK <= WAVES ? 1 : 2, WPH = 2 / DPL;  // dims per lane, waves per head
    constexpr int UNITS = QPK * WPH;                               // waves' worth of merging
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    __shared__ uint32_t s_last;
    // whether this block is the last of `n` to come here
    auto last_of = [&](uint32_t* ticket, int n) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0) {
            const uint32_t old = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            s_last = old + 1u == static_cast<uint32_t>(n) ? 1u : 0u;
            if (s_last != 0u) __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        return s_last != 0u;
    };
    auto state = [&](int h, int split) { return partials + (static_cast<int64_t>(h) * nsplit + split) * S; };
    float mx, den, num[DPL];
    int n = nsplit, step = 1;
    if (nsplit <= kDenseOneLevel) {
        if (!last_of(tickets + g, n)) return;
    } else {
        const int sets = (nsplit + kDenseSet - 1) / kDenseSet, set = s / kDenseSet, first = set * kDenseSet;
        uint32_t* tk = tickets + g * (sets + 1);
        n = min(kDenseSet, nsplit - first);
        if (!last_of(tk + set, n)) return;
        for (int u0 = 0; u0 < UNITS; u0 += WAVES) {
            const int u = u0 + wave, d0 = 64 * (u % WPH);
            float* dst = state(g * QPK + u / WPH, first);
            if (u < UNITS) dense_merge<T, DPL, false>(dst, 1, n, q, cur_k, cur_v, scale, d0, mx, den, num);
            // a head's two waves read the same m and l: both are past their
            // loads before either stores
            if constexpr (WPH == 2) __syncthreads();
            if (u < UNITS) {
                if (d0 == 0 && lane == 0) {
                    st_f32<true>(dst, mx);
                    st_f32<true>(dst + 1, den);
                }
#pragma unroll
                for (int i = 0; i < DPL; ++i) st_f32<true>(dst + 2 + d0 + lane + 64 * i, num[i]);
            }
        }
        n = sets;
        step = kDenseSet;
        if (!last_of(tk + sets, n)) return;
    }
    for (int u = wave; u < UNITS; u += WAVES) {
        const int h = g * QPK + u / WPH, d0 = 64 * (u % WPH);
        dense_merge<T, DPL, true>(state(h, 0), step, n, q + static_cast<int64_t>(h) * D,
                                  cur_k + static_cast<int64_t>(g) * D, cur_v + static_cast<int64_t>(g) * D, scale, d0,
                                  mx, den, num);
#pragma unroll
        for (int i = 0; i < DPL; ++i)
            Elem<T>::store(out + static_cast<int64_t>(h) * D, d0 + lane + 64 * i, num[i] / den);
    }
}

// VALU form (fp32; at the copy rate: 32 query heads over 8 KV heads at 32767
// tokens 54.2 us for 268 MB, 56.9 with a merge launch): workgroup (s, g) reads
// each row of its split once and folds it into QPK online-softmax states (one
// Q.K dot and one V update per head per row).  The last pass apart for 1 and
// 2 heads, in the loop for 4 and 8 (the better one for each: 8 KV heads at
// 65536 tokens, 2 heads 96.7 us apart and 99.7 in the loop, 8 heads 112.6 and
// 108.7).
template <typename T, int NB, int QPK>
__global__ __launch_bounds__(kAttnThreads) void attn_dense_gqa_kernel(
    const T* __restrict__ q, const T* __restrict__ kc, const T* __restrict__ vc, int64_t k_hs, int64_t v_hs,
    int64_t tokens, int split, float scale, float* __restrict__ partials, int nsplit, uint32_t* __restrict__ tickets,
    const T* __restrict__ cur_k, const T* __restrict__ cur_v, T* __restrict__ out) {
    constexpr int D = 128, LPR = 16, SLOTS = kWave / LPR, ROWS_PER_PASS = SLOTS * kAttnWaves;
    const int g = blockIdx.y;
    const int s = blockIdx.x;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const int slot = wave * SLOTS + lane / LPR;
    const int dim0 = (lane % LPR) * 8;
    Raw8<T> qr[QPK];
#pragma unroll
    for (int j = 0; j < QPK; ++j) qr[j].load(q + static_cast<int64_t>(g * QPK + j) * D + dim0);
    const int64_t t0 = static_cast<int64_t>(s) * split;
    const int n_rows = static_cast<int>(min<int64_t>(split, tokens - t0));
    const char* kb = reinterpret_cast<const char*>(kc + g * k_hs + t0 * D + dim0);
    const char* vb = reinterpret_cast<const char*>(vc + g * v_hs + t0 * D + dim0);
    SoftmaxState st[QPK];
#pragma unroll
    for (int j = 0; j < QPK; ++j) init_state(st[j]);
    // tail: the split's last pass, where it is not whole.  Its dead rows
    // re-read the split's first one; their values are cleared, since a weight
    // of 0 would make NaN of an infinite one.
    constexpr int PASS = ROWS_PER_PASS * NB;
    auto pass = [&](int base, bool tail) __attribute__((always_inline)) {
        Raw8<T> kr[NB], vr[NB];
        bool live[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int r = base + b * ROWS_PER_PASS + slot;
            live[b] = !tail || r < n_rows;
            const uint32_t off = static_cast<uint32_t>(live[b] ? r : 0) * (D * sizeof(T));
            kr[b].load(reinterpret_cast<const T*>(kb + off));
            vr[b].load(reinterpret_cast<const T*>(vb + off));
        }
        if (tail) {  // uniform
#pragma unroll
            for (int b = 0; b < NB; ++b)
                if (!live[b]) vr[b].zero();
        }
#pragma unroll
        for (int j = 0; j < QPK; ++j) fold_rows<T, NB>(st[j], qr[j], kr, vr, live, scale);
    };
    if constexpr (QPK <= 2) {
        int base = 0;
        for (; base + PASS <= n_rows; base += PASS) pass(base, false);
        if (base < n_rows) pass(base, true);
    } else {
        for (int base = 0; base < n_rows; base += PASS) pass(base, base + PASS > n_rows);
    }
#pragma unroll
    for (int j = 0; j < QPK; ++j) {
        store_partial<LPR>(st[j], lane, wave, dim0, D,
                           partials + (static_cast<int64_t>(g * QPK + j) * nsplit + s) * (D + 2), true);
        __syncthreads();  // store_partial's LDS is reused by the next head
    }
    dense_finish<T, QPK, kAttnWaves>(g, s, partials, nsplit, tickets, q, cur_k, cur_v, scale, out);
}

// Matrix-core form (16-bit types): per 16-token tile one v_mfma_f32_16x16x32
// chain (4 steps of 32 dims) multiplies A = the group's query rows (rows QPK
// .. 15 zero) by B = the tile's K rows (column n = token n), so lane group
// l / 16 ends with the logits of heads 4 (l / 16) .. + 3 for token l % 16 (C
// layout: lane l holds rows 4*(l/16) .. +3 of column l % 16; A and B: lane l
// holds k-elements 8*(l/16) .. +7 of row / column l % 16).  The tile's
// softmax runs on those lanes (DPP row maxima, one running max per head and
// wave), the weights go through LDS to the four 16-lane row slots, and each
// slot folds 4 of the tile's V rows into its accumulators (8 dims per lane)
// with the VALU, in fp32 as the weights are.
// Workgroup (split, KV head): 8 waves taking the split's tiles in turn,
// each with the next tile's K and V loads in flight while it folds one.
// Measured (HIP graph, before -> now, the whole layer): 64 query heads over 8
// KV heads at 50001 tokens bf16 97.7 (VALU kernel and a merge launch) -> 45.9
// us (4.5 TB/s; a copy's rate would take 40); 16 over 2 at 2000 tokens 28.6 ->
// 9.9; 32 over 8 at 32767 34.4 -> 31.2; 32 over 32 at 8191 fp16 29.1 -> 28.4.
template <typename T> struct MfmaVec8;
template <> struct MfmaVec8<bf16_t> { typedef __bf16 type __attribute__((ext_vector_type(8))); };
template <> struct MfmaVec8<f16_t> { typedef _Float16 type __attribute__((ext_vector_type(8))); };
typedef float mfma_f32x4 __attribute__((ext_vector_type(4)));

template <typename T>
__device__ __forceinline__ mfma_f32x4 mfma_16x16x32(uint4 a, uint4 b, mfma_f32x4 c) {
    using V = typename MfmaVec8<T>::type;
    if constexpr (std::is_same_v<T, bf16_t>)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(V, a), __builtin_bit_cast(V, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(V, a), __builtin_bit_cast(V, b), c, 0, 0, 0);
}

// Row 0 of the 16-lane rows: a of rows 0 and 1 added, row 1: b of rows 0 and
// 1, row 2: a of rows 2 and 3, row 3: b of rows 2 and 3 (swap_add32: the same
// for the wave's halves: a's in the lower one, b's in the upper).
__device__ __forceinline__ float swap_add16(float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                                                    false, false);
    const uint32_t x = r[0], y = r[1];
    return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
}
__device__ __forceinline__ float swap_add32(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                                                    false, false);
    const uint32_t x = r[0], y = r[1];
    return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
}

constexpr int kDenseWaves = 8;
constexpr int kDenseThreads = kDenseWaves * kWave;
constexpr int kDenseTile = 16;

template <typename T, int QPK>
__global__ __launch_bounds__(kDenseThreads) void attn_dense_mfma_kernel(
    const T* __restrict__ q, const T* __restrict__ kc, const T* __restrict__ vc, int64_t k_hs, int64_t v_hs,
    int64_t tokens, int split, float scale, float* __restrict__ partials, int nsplit, uint32_t* __restrict__ tickets,
    const T* __restrict__ cur_k, const T* __restrict__ cur_v, T* __restrict__ out) {
    constexpr int D = 128, TILE = kDenseTile, W = kDenseWaves;
    constexpr int HL = QPK < 4 ? QPK : 4;  // heads per softmax lane
    const int g = blockIdx.y;
    const int s = blockIdx.x;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int col = lane & 15;  // MFMA row / column; the V dim slice 8*col
    const int grp = lane >> 4;  // MFMA k-group; the V row slot
    const int64_t t0 = static_cast<int64_t>(s) * split;
    const int n_rows = static_cast<int>(min<int64_t>(split, tokens - t0));
    uint4 qa[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        qa[i] = col < QPK ? *reinterpret_cast<const uint4*>(q + static_cast<int64_t>(g * QPK + col) * D + 32 * i + 8 * grp)
                          : make_uint4(0u, 0u, 0u, 0u);
    const char* kb = reinterpret_cast<const char*>(kc + g * k_hs + t0 * D + 8 * grp);
    const char* vb = reinterpret_cast<const char*>(vc + g * v_hs + t0 * D + 8 * col);
    // rows past the split's end re-read the split's first row: the fold masks
    // their logits and clears their values (a weight of 0 would make NaN of
    // an infinite one)
    auto load_tile = [&](int r0, uint4 (&kt)[4], uint4 (&vt)[4]) {
        const int rk = r0 + col;
        const uint32_t ko = static_cast<uint32_t>(rk < n_rows ? rk : 0) * (D * sizeof(T));
#pragma unroll
        for (int i = 0; i < 4; ++i) kt[i] = *reinterpret_cast<const uint4*>(kb + ko + 32 * i * sizeof(T));
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int rv = r0 + 4 * grp + r;
            const uint32_t vo = static_cast<uint32_t>(rv < n_rows ? rv : 0) * (D * sizeof(T));
            vt[r] = *reinterpret_cast<const uint4*>(vb + vo);
        }
    };
    __shared__ __align__(16) float s_p[W][TILE][QPK];
    float m_run[HL], lsum[HL], acc[QPK][8];
#pragma unroll
    for (int j = 0; j < HL; ++j) {
        m_run[j] = -INFINITY;
        lsum[j] = 0.0f;
    }
#pragma unroll
    for (int j = 0; j < QPK; ++j)
#pragma unroll
        for (int d = 0; d < 8; ++d) acc[j][d] = 0.0f;
    auto fold_tile = [&](int r0, const uint4 (&kt)[4], uint4 (&vt)[4]) {
        if (r0 + TILE > n_rows) {  // uniform: the split's last tile
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (r0 + 4 * grp + r >= n_rows) vt[r] = make_uint4(0u, 0u, 0u, 0u);
        }
        mfma_f32x4 c = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < 4; ++i) c = mfma_16x16x32<T>(qa[i], kt[i], c);
        const bool live = r0 + col < n_rows;
        float p[HL], alpha[HL];
        bool moved = false;
#pragma unroll
        for (int j = 0; j < HL; ++j) {
            const float sj = live ? c[j] * scale : -INFINITY;
            float mx = fmaxf(sj, dpp_mov<0xB1>(sj));
            mx = fmaxf(mx, dpp_mov<0x4E>(mx));
            mx = fmaxf(mx, dpp_mov<0x141>(mx));
            mx = fmaxf(mx, dpp_mov<0x140>(mx));
            const float mn = fmaxf(m_run[j], mx);
            alpha[j] = mn == -INFINITY ? 1.0f : __expf(m_run[j] - mn);  // m_run = -inf gives 0
            // dead rows and logits of -inf give 0; a NaN logit stays NaN, also
            // where no logit of the wave has been a number yet (mn = -inf)
            p[j] = sj == -INFINITY ? 0.0f : __expf(sj - mn);
            moved = moved || mn != m_run[j];
            m_run[j] = mn;
            lsum[j] = fmaf(lsum[j], alpha[j], p[j]);
        }
        if (QPK > 4 ? lane < 2 * TILE : lane < TILE) {
            if constexpr (HL == 4) *reinterpret_cast<float4*>(&s_p[wave][col][QPK > 4 ? 4 * grp : 0]) = make_float4(p[0], p[1], p[2], p[3]);
            else if constexpr (HL == 2) *reinterpret_cast<float2*>(&s_p[wave][col][0]) = make_float2(p[0], p[1]);
            else s_p[wave][col][0] = p[0];
        }
        // the wave reads its own weights next: one wave's LDS operations complete in order
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (__ballot(moved) != 0) {  // some head's running max moved
#pragma unroll
            for (int j = 0; j < QPK; ++j) {
                const float al = __builtin_bit_cast(
                    float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, alpha[j % 4]), TILE * (j / 4)));
#pragma unroll
                for (int d = 0; d < 8; ++d) acc[j][d] *= al;
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float pj[QPK];
            const float* src = &s_p[wave][4 * grp + r][0];
            if constexpr (QPK >= 4) {
#pragma unroll
                for (int j = 0; j < QPK; j += 4) {
                    const float4 x = *reinterpret_cast<const float4*>(src + j);
                    pj[j] = x.x; pj[j + 1] = x.y; pj[j + 2] = x.z; pj[j + 3] = x.w;
                }
            } else {
#pragma unroll
                for (int j = 0; j < QPK; ++j) pj[j] = src[j];
            }
            Raw8<T> v;
            v.u = vt[r];
#pragma unroll
            for (int d = 0; d < 8; ++d) {
                const float vf = v.get(d);
#pragma unroll
                for (int j = 0; j < QPK; ++j) acc[j][d] = fmaf(pj[j], vf, acc[j][d]);
            }
        }
        // the next tile's weights overwrite s_p[wave] only after every lane has read
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    constexpr int STEP = W * TILE;
    uint4 ka[4], va[4], kn[4], vn[4];
    int r0 = wave * TILE;
    if (r0 < n_rows) load_tile(r0, ka, va);
    while (r0 < n_rows) {
        if (r0 + STEP < n_rows) load_tile(r0 + STEP, kn, vn);
        fold_tile(r0, ka, va);
        r0 += STEP;
        if (r0 >= n_rows) break;
        if (r0 + STEP < n_rows) load_tile(r0 + STEP, ka, va);
        fold_tile(r0, kn, vn);
        r0 += STEP;
    }
    // the waves' states meet in LDS: every lane of a wave shares the head's
    // running max, so its row slots add up
    __shared__ float s_m[W][QPK], s_l[W][QPK];
    __shared__ float s_acc[W][QPK][D];
#pragma unroll
    for (int j = 0; j < HL; ++j) {
        const float l = row_sum<16>(lsum[j]);
        const int h = (QPK > 4 ? 4 * grp : 0) + j;
        if (col == 0 && grp < (QPK + 3) / 4) {
            s_m[wave][h] = m_run[j];
            s_l[wave][h] = l;
        }
    }
    // four values at a time: a lane-row swap and an add halve two registers
    // into one, twice, and row r of the lanes ends with the sum of value r
#pragma unroll
    for (int k = 0; k < 2 * QPK; ++k) {
        const float* x = &acc[k / 2][4 * (k & 1)];
        const float a = swap_add16(x[0], x[1]), b = swap_add16(x[2], x[3]);
        s_acc[wave][k / 2][8 * col + 4 * (k & 1) + grp] = swap_add32(a, b);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < QPK * D; i += kDenseThreads) {
        const int j = i / D, d = i % D;
        float mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < W; ++w) mx = fmaxf(mx, s_m[w][j]);
        float a = 0.0f, l = 0.0f;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const float f = s_m[w][j] == -INFINITY ? 0.0f : __expf(s_m[w][j] - mx);
            a = fmaf(f, s_acc[w][j][d], a);
            l = fmaf(f, s_l[w][j], l);
        }
        float* dst = partials + (static_cast<int64_t>(g * QPK + j) * nsplit + s) * (D + 2);
        st_f32<true>(dst + 2 + d, a);
        if (d == 0) {
            st_f32<true>(dst, mx);
            st_f32<true>(dst + 1, l);
        }
    }
    dense_finish<T, QPK, W>(g, s, partials, nsplit, tickets, q, cur_k, cur_v, scale, out);
}

// Splits of a dense layer: a workgroup per CU in all (a second one per CU
// only adds its epilogue: 32 query heads over 8 KV heads at 32767 tokens
// 31.1 us with 256 workgroups, 41.6 with 512; 64 over 8 at 50001 48.1 and
// 56.7; 32 over 32 at 8191 27.7 and 29.2; fp32, 64 over 8 at 65536 108.7 and
// 115.0, 8 over 4 at 16384 19.9 and 20.6), of whole tiles and at least one
// per wave.
constexpr int kDenseBlocks = 256;
constexpr int kDenseLeast = kDenseWaves * kDenseTile;

struct DensePlan {
    int splits, tokens;
};
DensePlan dense_plan(int64_t tokens, int kv_heads) {
    if (tokens <= 0) return {1, kDenseLeast};
    int64_t want = kDenseBlocks / kv_heads;
    if (want <= 1) {
        // A workgroup per KV head can leave most CUs idle in its last round:
        // three of a third each where those take at most 0.8 of the rounds'
        // time (4096 tokens bf16, one and three: 144 heads 59.4 and 51.3 us,
        // 300 147 and 118; 176, two thirds of a round either way, 70.6 and 82).
        const int one = (kv_heads + kDenseBlocks - 1) / kDenseBlocks;
        const int three = (3 * kv_heads + kDenseBlocks - 1) / kDenseBlocks;
        if (5 * three <= 12 * one) want = 3;
    }
    if (want > dense_max_splits(tokens)) want = dense_max_splits(tokens);
    if (want < 1) want = 1;
    int64_t per = ((tokens + want - 1) / want + kDenseTile - 1) / kDenseTile * kDenseTile;
    if (per < kDenseLeast) per = kDenseLeast;
    return {static_cast<int>((tokens + per - 1) / per), static_cast<int>(per)};
}

template <typename T>
hipError_t launch_dense_t(const void* q, const void* kc, const void* vc, int64_t k_hs, int64_t v_hs, int64_t tokens,
                          int q_heads, int kv_heads, float* partials, uint32_t* tickets, const void* current_k,
                          const void* current_v, void* output, hipStream_t stream) {
    const float scale = static_cast<float>(1.0 / sqrt(128.0));
    const DensePlan p = dense_plan(tokens, kv_heads);
    const dim3 grid(static_cast<unsigned>(p.splits), static_cast<unsigned>(kv_heads));
    const T *q_ = static_cast<const T*>(q), *k_ = static_cast<const T*>(kc), *v_ = static_cast<const T*>(vc);
    const T *ck = static_cast<const T*>(current_k), *cv = static_cast<const T*>(current_v);
    T* o_ = static_cast<T*>(output);
#define POPKV_DENSE_LAUNCH(KERNEL, THREADS)                                                                        \
    hipLaunchKernelGGL(KERNEL, grid, dim3(THREADS), 0, stream, q_, k_, v_, k_hs, v_hs, tokens, p.tokens, scale,  \
                       partials, p.splits, tickets, ck, cv, o_)
    const int qpk = q_heads / kv_heads;
    if constexpr (sizeof(T) == 2) {
        switch (qpk) {
            case 1: POPKV_DENSE_LAUNCH((attn_dense_mfma_kernel<T, 1>), kDenseThreads); break;
            case 2: POPKV_DENSE_LAUNCH((attn_dense_mfma_kernel<T, 2>), kDenseThreads); break;
            case 4: POPKV_DENSE_LAUNCH((attn_dense_mfma_kernel<T, 4>), kDenseThreads); break;
            default: POPKV_DENSE_LAUNCH((attn_dense_mfma_kernel<T, 8>), kDenseThreads); break;
        }
    } else {
        switch (qpk) {
            case 1: POPKV_DENSE_LAUNCH((attn_dense_gqa_kernel<T, 8, 1>), kAttnThreads); break;
            case 2: POPKV_DENSE_LAUNCH((attn_dense_gqa_kernel<T, 8, 2>), kAttnThreads); break;
            case 4: POPKV_DENSE_LAUNCH((attn_dense_gqa_kernel<T, 4, 4>), kAttnThreads); break;
            default: POPKV_DENSE_LAUNCH((attn_dense_gqa_kernel<T, 4, 8>), kAttnThreads); break;
        }
    }
#undef POPKV_DENSE_LAUNCH
    return hipGetLastError();
}

}  // namespace

int64_t dense_max_splits(int64_t tokens) {
    const int64_t least = (tokens + kDenseLeast - 1) / kDenseLeast;
    return least < 1 ? 1 : least < kDenseBlocks ? least : kDenseBlocks;
}

hipError_t launch_attention_dense(const void* queries, int dtype, const void* prefix_k, const void* prefix_v,
                                  int64_t k_head_stride, int64_t v_head_stride, int64_t tokens, int q_heads,
                                  int kv_heads, float* partials, uint32_t* tickets, const void* current_k,
                                  const void* current_v, void* output, hipStream_t stream) {
#define POPKV_DENSE_T(T)                                                                                          \
    launch_dense_t<T>(queries, prefix_k, prefix_v, k_head_stride, v_head_stride, tokens, q_heads, kv_heads, partials, \
                      tickets, current_k, current_v, output, stream)
    switch (dtype) {
        case POPKV_DTYPE_F32: return POPKV_DENSE_T(float);
        case POPKV_DTYPE_F16: return POPKV_DENSE_T(f16_t);
        default: return POPKV_DENSE_T(bf16_t);
    }
#undef POPKV_DENSE_T
}

}  // namespace popkv
