// Device pieces shared by the sparse (attention.hip) and dense (dense.hip)
// attention kernels: online-softmax states, the fold of gathered rows into
// them, and the device-coherent hand-off and merge of partial states.
#pragma once

#include <type_traits>

#include "device_common.h"

namespace popkv {
namespace {

constexpr int kAttnThreads = 256;
constexpr int kAttnWaves = kAttnThreads / kWave;

struct SoftmaxState {
    float m, l, acc[8];
};

__device__ __forceinline__ void merge_state(SoftmaxState& a, float m2, float l2, const float* acc2) {
    const float mm = fmaxf(a.m, m2);
    if (mm == -INFINITY) return;
    const float wa = a.m == -INFINITY ? 0.0f : __expf(a.m - mm);
    const float wb = m2 == -INFINITY ? 0.0f : __expf(m2 - mm);
    a.l = a.l * wa + l2 * wb;
#pragma unroll
    for (int i = 0; i < 8; ++i) a.acc[i] = a.acc[i] * wa + acc2[i] * wb;
    a.m = mm;
}

// Writes a workgroup's (m, l, acc[d]) to dst: the row slots of each wave
// (lanes with equal dim slice) merge through shuffles, the waves through LDS.
// All threads of the block call it.
// Partial states handed from one workgroup to another inside a kernel (the
// layer step's fused merge) are written and read as device-scope relaxed
// atomics: plain global stores / loads with the device-coherence bit, which
// go through to memory instead of staying in one XCD's L2, so no L2
// write-back or invalidate is needed for them.
// The fused merges hand chunk states from workgroup to workgroup with no
// release/acquire pair: the states are stored with relaxed agent-scope
// atomic stores, each wave then waits with "s_waitcnt vmcnt(0)", the block
// meets at a barrier, and one relaxed agent-scope atomic add takes the
// ticket; the last block reads the states with relaxed agent-scope atomic
// loads.  That is correct on gfx942 / gfx950 because (1) an agent-scope
// atomic store or load is a global store / load with the sc1 bit, which
// writes through and reads past the XCD's non-coherent L2 to the device's
// coherence point, and (2) stores count in vmcnt on these targets, so
// vmcnt(0) returns only once every store of the wave is acknowledged by
// that point -- before the ticket is taken.  On targets that count stores
// in a separate vscnt (gfx10 and later) or that cache agent-scope stores,
// the wait would not cover the states: the build refuses them.
#if defined(__HIP_DEVICE_COMPILE__) && !defined(__gfx950__) && !defined(__gfx942__)
#error "the fused merge's hand-off relies on gfx942/gfx950 store acknowledgement (vmcnt) and sc1 write-through"
#endif

template <bool COH>
__device__ __forceinline__ void st_f32(float* p, float v) {
    if constexpr (COH) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else *p = v;
}
template <bool COH>
__device__ __forceinline__ float ld_f32(const float* p) {
    if constexpr (COH) return __hip_atomic_load(const_cast<float*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else return *p;
}

template <int LPR>
__device__ __forceinline__ void store_partial(SoftmaxState st, int lane, int wave, int dim0, int d, float* dst,
                                              bool coherent = false) {
    auto merge_xor = [&](auto mtag) {
        constexpr int M = decltype(mtag)::value;
        const float m2 = lane_xor<M>(st.m);
        const float l2 = lane_xor<M>(st.l);
        float a2[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) a2[i] = lane_xor<M>(st.acc[i]);
        merge_state(st, m2, l2, a2);
    };
    if constexpr (LPR <= 8) merge_xor(std::integral_constant<int, 8>{});
    if constexpr (LPR <= 16) merge_xor(std::integral_constant<int, 16>{});
    merge_xor(std::integral_constant<int, 32>{});
    __shared__ float s_m[kAttnWaves], s_l[kAttnWaves];
    __shared__ float s_acc[kAttnWaves][256];
    if (lane < LPR) {
#pragma unroll
        for (int i = 0; i < 8; ++i) s_acc[wave][dim0 + i] = st.acc[i];
        if (lane == 0) { s_m[wave] = st.m; s_l[wave] = st.l; }
    }
    __syncthreads();
    const int dim = threadIdx.x;
    float mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < kAttnWaves; ++w) mx = fmaxf(mx, s_m[w]);
    float l = 0.0f, a = 0.0f;
#pragma unroll
    for (int w = 0; w < kAttnWaves; ++w) {
        if (s_m[w] == -INFINITY) continue;
        const float wt = __expf(s_m[w] - mx);
        l += s_l[w] * wt;
        if (dim < d) a += s_acc[w][dim] * wt;
    }
    if (coherent) {
        if (dim < d) st_f32<true>(dst + 2 + dim, a);
        if (dim == 0) {
            st_f32<true>(dst, mx);
            st_f32<true>(dst + 1, l);
        }
    } else {
        if (dim < d) dst[2 + dim] = a;
        if (dim == 0) {
            dst[0] = mx;
            dst[1] = l;
        }
    }
}

// Split states a merge loads in its first burst (and per batch after it).
constexpr int kMergeFirst = 16;

// Merge of one head by one wave (lane l owning dims l and l + 64): the
// head's nsplit states ps[s] = (m, l, acc[128]) plus the current token
// (logit qh . ck * scale, value cv), written to outh in the query dtype.
// No LDS or barrier: the split maxima and denominators are wave reductions
// (lane s holds split s of each 64-split group), and the weights reach the
// accumulation through readlane.  qh, ck, cv, the first group's maxima and
// denominators and the first NF splits' accumulators are loaded in one
// burst, so a layer step's merge pays one memory latency for all of them;
// further splits follow in batches of NF.  Accumulation
// order: the current token, then the splits in ascending order.  COH: the
// states are read with device-coherent loads (written by other workgroups
// of the same kernel).
template <typename T, bool COH, int NF = kMergeFirst>
__device__ __forceinline__ void merge_head(const float* __restrict__ ps, int nsplit, const T* __restrict__ qh,
                                           const T* __restrict__ ck, const T* __restrict__ cv, float scale,
                                           T* __restrict__ outh) {
    constexpr int S = 128 + 2;
    const int lane = threadIdx.x & (kWave - 1);
    // the burst (with nsplit == 0 the accumulator loads read split 0's slot,
    // which every workspace holds, and are not used)
    const float q0 = Elem<T>::load(qh, lane), q1 = Elem<T>::load(qh, lane + 64);
    const float k0 = Elem<T>::load(ck, lane), k1 = Elem<T>::load(ck, lane + 64);
    const float v0 = Elem<T>::load(cv, lane), v1 = Elem<T>::load(cv, lane + 64);
    float m0 = -INFINITY, l0 = 0.0f;  // split `lane`
    if (lane < nsplit) {
        m0 = ld_f32<COH>(ps + (static_cast<int64_t>(lane) * S));
        l0 = ld_f32<COH>(ps + (static_cast<int64_t>(lane) * S + 1));
    }
    const int nf = min(nsplit, NF);
    float a0[NF], a1[NF];
#pragma unroll
    for (int j = 0; j < NF; ++j) {
        const int64_t so = static_cast<int64_t>(max(min(j, nf - 1), 0)) * S + 2;
        a0[j] = ld_f32<COH>(ps + (so + lane));
        a1[j] = ld_f32<COH>(ps + (so + lane + 64));
    }
    // the maxima of every split and the current token's logit
    float mx = m0;
    for (int s0 = kWave; s0 < nsplit; s0 += kWave)
        if (s0 + lane < nsplit) mx = fmaxf(mx, ld_f32<COH>(ps + (static_cast<int64_t>(s0 + lane) * S)));
    const float cur_m = wave_sum(q0 * k0 + q1 * k1) * scale;
    mx = fmaxf(wave_max(mx), cur_m);
    const float wc = __expf(cur_m - mx);
    const float w0 = m0 == -INFINITY ? 0.0f : __expf(m0 - mx);
    float den = l0 * w0, num0 = wc * v0, num1 = wc * v1;
#pragma unroll
    for (int j = 0; j < NF; ++j) {
        if (j < nf) {
            const float ws = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w0), j));
            num0 = fmaf(ws, a0[j], num0);
            num1 = fmaf(ws, a1[j], num1);
        }
    }
    for (int s0 = 0; s0 < nsplit; s0 += kWave) {
        float w = w0;
        if (s0 > 0) {
            float m = -INFINITY, l = 0.0f;
            if (s0 + lane < nsplit) {
                m = ld_f32<COH>(ps + (static_cast<int64_t>(s0 + lane) * S));
                l = ld_f32<COH>(ps + (static_cast<int64_t>(s0 + lane) * S + 1));
            }
            w = m == -INFINITY ? 0.0f : __expf(m - mx);
            den += l * w;
        }
        const int n = min(kWave, nsplit - s0);
        for (int b = s0 == 0 ? nf : 0; b < n; b += NF) {
            float c0[NF], c1[NF];
#pragma unroll
            for (int j = 0; j < NF; ++j) {
                const int64_t so = static_cast<int64_t>(s0 + min(b + j, n - 1)) * S + 2;
                c0[j] = ld_f32<COH>(ps + (so + lane));
                c1[j] = ld_f32<COH>(ps + (so + lane + 64));
            }
#pragma unroll
            for (int j = 0; j < NF; ++j) {
                if (b + j < n) {
                    const float ws =
                        __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w), b + j));
                    num0 = fmaf(ws, c0[j], num0);
                    num1 = fmaf(ws, c1[j], num1);
                }
            }
        }
    }
    den = wave_sum(den) + wc;
    Elem<T>::store(outh, lane, num0 / den);
    Elem<T>::store(outh, lane + 64, num1 / den);
}

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

// Dot product of 8 packed 16-bit elements with v_dot2 (fp32 accumulation).
template <typename T>
__device__ __forceinline__ float dot8(const uint4& a, const uint4& b) {
    auto d2 = [](uint32_t x, uint32_t y, float c) {
        if constexpr (Elem<T>::kDtype == POPKV_DTYPE_BF16)
            return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, x), __builtin_bit_cast(bf16x2_t, y), c,
                                                   false);
        else
            return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2_t, x), __builtin_bit_cast(f16x2_t, y), c, false);
    };
    return d2(a.w, b.w, d2(a.z, b.z, d2(a.y, b.y, d2(a.x, b.x, 0.0f))));
}

__device__ __forceinline__ void init_state(SoftmaxState& st) {
    st.m = -INFINITY;
    st.l = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) st.acc[i] = 0.0f;
}

// Folds NB gathered rows (this lane's 8-element slices of K and V; the 16
// lanes of a row slot hold one row) into the lane's online-softmax state.
// Rows with live[b] false get weight exactly 0.
template <typename T, int NB>
__device__ __forceinline__ void fold_rows(SoftmaxState& st, const Raw8<T>& qr, const Raw8<T> (&kr)[NB],
                                          const Raw8<T> (&vr)[NB], const bool (&live)[NB], float scale) {
    float logit[NB];
    float bm = -INFINITY;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        float dot;
        if constexpr (sizeof(T) == 2) {
            dot = dot8<T>(qr.u, kr[b].u);
        } else {
            dot = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i) dot = fmaf(qr.get(i), kr[b].get(i), dot);
        }
        dot = row_sum<16>(dot);
        logit[b] = live[b] ? dot * scale : -INFINITY;
        bm = fmaxf(bm, logit[b]);
    }
    // The compiler sinks the V loads into this branch, so a batch's V rows
    // are requested only once its K rows have arrived.  A branch-free form
    // with every K and V request in flight at once measured slower on the
    // layer step's gathers (C1 select + attention kernel 18.6 vs 17.1 us).
    const float mnew = fmaxf(st.m, bm);
    if (mnew != -INFINITY) {
        const float alpha = __expf(st.m - mnew);  // st.m = -inf gives 0
        st.l *= alpha;
#pragma unroll
        for (int i = 0; i < 8; ++i) st.acc[i] *= alpha;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const float p = __expf(logit[b] - mnew);  // -inf logit gives 0
            st.l += p;
#pragma unroll
            for (int i = 0; i < 8; ++i) st.acc[i] = fmaf(p, vr[b].get(i), st.acc[i]);
        }
        st.m = mnew;
    }
}

}  // namespace
}  // namespace popkv
