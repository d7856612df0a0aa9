// Decode schedules over an MFMA body (decode_mfma.h): the fixed-split and
// balanced kernels, and the group-size table of the tuned instantiations.
// Included by the per-pool-type translation units only.
#pragma once

#include <hip/hip_runtime.h>

#include "decode_kernels.h"
#include "decode_mfma.h"

namespace llkv {
namespace {

// Streaming (nontemporal) loads, in the kernels that may use them (Body::kStream;
// kStreamBytes in decode.hip): for batches that read more than stream_units
// page-units by their actual lengths, and segments whose middle page is no other
// sequence's too.  A page that several sequences read (a cached prefix) is read
// again from the caches, where streaming loads leave nothing: 256 sequences of
// 32/8/128 fp16 on one prefix of 2048 tokens 265 us, 332 streamed.  A prefix lies at
// the same place of each table, so one entry per sequence tells.  The choice costs 1
// to 2 us: 16 x 32768 tokens of 14/2/64 fp16 51.3 -> 52.6, 55.8 without streaming loads.
// shares_page: whether this lane's part (of `lanes`) of the other sequences has page
// pg of sequence b.
template <class Pages>
__device__ inline bool shares_page(const DecodeArgs& a, int b, int pg, int lane, int lanes, Pages pages) {
    const int id = a.bt[(int64_t)b * a.max_blocks + pg];
    bool same = false;
    for (int j = lane; j < a.B; j += lanes)
        same |= (a.bt[(int64_t)j * a.max_blocks + pg] == id) & (pages(j) > pg) & (j != b);
    return same;
}

// Fixed split schedule: grid (S_max, Hkv, B), Body::W waves per work-group,
// one segment each.
template <class Body>
__global__ __launch_bounds__(Body::kThreads) __attribute__((amdgpu_waves_per_eu(Body::kWavesPerEU)))
void decode_split_kernel(DecodeArgs a) {
    __shared__ typename Body::Smem sm;
    __shared__ SegDesc segs[1];
    using T = typename Body::T;
    LLKV_TRACE_POINT(0);
    const int split = blockIdx.x, kvh = blockIdx.y, b = blockIdx.z;
    const SplitGeo geo = split_geo(a, b);
    const int hq0 = kvh * Body::GQ;
    if (geo.npages == 0) {   // empty sequence: zeros, as the reference (:224-227)
        if (split == 0) {
            T* out = reinterpret_cast<T*>(a.out) + ((int64_t)b * a.Hq + hq0) * Body::HD;
            for (int i = threadIdx.x; i < Body::GQ * Body::HD; i += blockDim.x)
                out[i] = Elem<T>::from_f32(0.0f);
        }
        return;
    }
    if (split >= geo.nsplit) return;
    if (threadIdx.x == 0) {
        SegDesc& d = segs[0];
        d.b = b;
        d.kvh = kvh;
        d.pg_begin = split * geo.pps;
        d.npages = min(geo.pps, geo.npages - d.pg_begin);
        d.cum = 0;
        d.tok_end = min((d.pg_begin + d.npages) * kPage, geo.L);
        d.direct = geo.nsplit == 1;
        d.new_tok = seg_new_tok(a, b, d.pg_begin, d.tok_end, geo.L);
        const int64_t bh0 = (int64_t)b * a.Hq + hq0;
        d.po_off = (bh0 * a.S_max + split) * a.D;
        d.pl_off = bh0 * a.S_max + split;
    }
    bool stream = false;   // the same in every wave
    if constexpr (Body::kStream) {
        // (as if every sequence were as long, so that small batches under a large
        // bound load nothing here; then the actual lengths)
        if ((int64_t)geo.npages * a.B * a.Hkv > a.stream_units) {
            const int lane = threadIdx.x & 63;
            const int pg = split * geo.pps, n = min(geo.pps, geo.npages - pg);
            const int warm = a.bt[(int64_t)b * a.max_blocks + pg + min((int)threadIdx.x, n - 1)];   // for round()
            auto pages = [&](int j) { return (clamp_len(a, j) + kPage - 1) / kPage; };
            int64_t units = 0;
            for (int j = lane; j < a.B; j += 64) units += pages(j);
            const bool same = shares_page(a, b, pg + n / 2, lane, 64, pages);
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) units += __shfl_xor(units, off, 64);
            stream = units * a.Hkv > a.stream_units && __builtin_amdgcn_ballot_w64(same) == 0;
            asm volatile("" ::"v"(warm));
        }
    }
    __syncthreads();
    store_new_row<T, Body::HD>(a, segs[0]);
    if constexpr (Body::kStream) {
        if (stream) {
            Body::template round<true>(a, sm, segs, 1, (int64_t)a.S_max * a.D, a.S_max);
            return;
        }
    }
    Body::template round<false>(a, sm, segs, 1, (int64_t)a.S_max * a.D, a.S_max);
}

// Balanced schedule: grid (nwg), 4 waves per work-group.  Every work-group
// scans the lengths itself (the batch is at most kBalanceMaxB sequences) and
// cuts its share into segments, run kSegMax segments per round.  A unit
// (sequence, kv head) inside one share is written directly; the others are
// merged by decode_merge_balanced_kernel.  Work-group 0 stores the page
// prefix sums for that kernel; empty sequences get zeros from the work-group
// with their index modulo nwg.
template <class Body>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(Body::kWavesPerEU)))
void decode_balanced_kernel(DecodeArgs a) {
    using T = typename Body::T;
    constexpr int D = Body::HD;
    __shared__ typename Body::Smem sm;
    __shared__ int sP[kBalanceMaxB + 1];
    __shared__ int sL[kBalanceMaxB];
    __shared__ SegDesc segs[Body::kSegMax];
    __shared__ int s_n, s_shared;
    __shared__ int64_t s_next;
    LLKV_TRACE_POINT(0);
    scan_pages(a, sP, sL);
    LLKV_TRACE_POINT(4);
    const int tid = threadIdx.x;
    if (blockIdx.x == 0)
        for (int i = tid; i <= a.B; i += blockDim.x) a.plan[i] = sP[i];
    const int64_t T_ = (int64_t)a.Hkv * sP[a.B];
    const int64_t wg = blockIdx.x;
    for (int b = (int)wg; b < a.B; b += a.nwg) {   // the reference's seq_len == 0 rule (:224-227)
        if (sP[b + 1] != sP[b]) continue;
        T* out = reinterpret_cast<T*>(a.out) + (int64_t)b * a.Hq * D;
        for (int i = tid; i < a.Hq * D; i += blockDim.x) out[i] = Elem<T>::from_f32(0.0f);
    }
    const int64_t r1 = share_begin(wg + 1, T_, a.nwg);
    int64_t p = share_begin(wg, T_, a.nwg);
    int stream = -1;   // not decided
    while (p < r1) {
        if (tid == 0) {
            int n = 0;
            s_next = build_segments(a, sP, sL, p, r1, wg, Body::kSegMax, segs, &n);
            s_n = n;
            s_shared = 0;
        }
        __syncthreads();
        const int n = s_n;
        p = s_next;
        for (int i = 0; i < n; ++i) store_new_row<T, D>(a, segs[i]);
        if constexpr (Body::kStream) {
            if (T_ > a.stream_units && stream < 0) {   // uniform; by the share's first segments
                const SegDesc& d = segs[0];
                const int warm = a.bt[(int64_t)d.b * a.max_blocks + d.pg_begin + min(tid, d.npages - 1)];   // for round()
                bool same = false;
                for (int i = 0; i < n; ++i)
                    same |= shares_page(a, segs[i].b, segs[i].pg_begin + segs[i].npages / 2, tid, blockDim.x,
                                        [&](int j) { return sP[j + 1] - sP[j]; });
                asm volatile("" ::"v"(warm));
                if (same) s_shared = 1;
                __syncthreads();
                stream = s_shared == 0;
            }
            if (stream > 0) {
                Body::template round<true>(a, sm, segs, n, D, 1);   // ends with a barrier
                continue;
            }
        }
        Body::template round<false>(a, sm, segs, n, D, 1);   // ends with a barrier
    }
}

template <class Body>
Kernels kernels_of() {
    Kernels k;
    if constexpr (!Body::kStream) k.split = decode_split_kernel<Body>;
    k.balanced = decode_balanced_kernel<Body>;
    return k;
}

// head_dim 64 / 128 also get the unit schedule's kUnitWaves-wave kernel,
// except fp32 at head_dim 128, whose body does not fit the 128 registers of
// four waves per SIMD (~50 would spill).
template <typename T, int D, int G, bool A, bool ST>
Kernels kernels_with_unit() {
    Kernels k = kernels_of<MfmaDecode<T, D, G, A, kDecodeWaves, ST>>();
    constexpr bool kF32 = Elem<T>::kDtype == LLKV_DTYPE_F32;
    if constexpr (!(kF32 && D == 128) && (!ST || (D == 64 && !kF32)))
        k.unit = decode_split_kernel<MfmaDecode<T, D, G, A, kUnitWaves, ST>>;
    return k;
}

template <typename T, int D, bool A, bool ST>
Kernels tuned_g(int G) {
    switch (G) {
        case 1: return kernels_with_unit<T, D, 1, A, ST>();
        case 2: return kernels_with_unit<T, D, 2, A, ST>();
        case 3: return kernels_with_unit<T, D, 3, A, ST>();
        case 4: return kernels_with_unit<T, D, 4, A, ST>();
        case 5: return kernels_with_unit<T, D, 5, A, ST>();
        case 6: return kernels_with_unit<T, D, 6, A, ST>();
        case 7: return kernels_with_unit<T, D, 7, A, ST>();
        case 8: return kernels_with_unit<T, D, 8, A, ST>();
        case 12: return kernels_with_unit<T, D, 12, A, ST>();
        case 16: return kernels_with_unit<T, D, 16, A, ST>();
    }
    return Kernels();
}

// head_dim 96 (Phi-3 layouts) and 256 (Gemma-2 / Gemma-3 layouts): group
// sizes 1, 2, 4, 8.
template <typename T, int D, bool A, bool ST>
Kernels tuned_g_few(int G) {
    switch (G) {
        case 1: return kernels_of<MfmaDecode<T, D, 1, A, kDecodeWaves, ST>>();
        case 2: return kernels_of<MfmaDecode<T, D, 2, A, kDecodeWaves, ST>>();
        case 4: return kernels_of<MfmaDecode<T, D, 4, A, kDecodeWaves, ST>>();
        case 8: return kernels_of<MfmaDecode<T, D, 8, A, kDecodeWaves, ST>>();
    }
    return Kernels();
}

// ST: the kernels that may stream, where they measured faster (kStreamBytes in
// decode.hip); the others stay null and the plain ones run.
template <typename T, bool ST>
Kernels tuned(int D, int G, bool append) {
    constexpr bool kF32 = Elem<T>::kDtype == LLKV_DTYPE_F32;
    if (D == 64) return append ? tuned_g<T, 64, true, ST>(G) : tuned_g<T, 64, false, ST>(G);
    if constexpr (!ST) {
        if (D == 128) return append ? tuned_g<T, 128, true, false>(G) : tuned_g<T, 128, false, false>(G);
    } else if constexpr (!kF32) {
        if (D == 128 && !append) return tuned_g<T, 128, false, true>(G);
    }
    if (D == 256) return append ? tuned_g_few<T, 256, true, ST>(G) : tuned_g_few<T, 256, false, ST>(G);
    if constexpr (!ST || kF32)
        if (D == 96) return append ? tuned_g_few<T, 96, true, ST>(G) : tuned_g_few<T, 96, false, ST>(G);
    return Kernels();
}

}  // namespace
}  // namespace llkv
