// gemm_f32_store.h — epilogue shared by the FP32 products (gemm_x3.hip, gemm_f32_ws.hip):
// four consecutive columns of one row per lane, straight from C^T accumulators.
#ifndef CF_GEMM_F32_STORE_H_
#define CF_GEMM_F32_STORE_H_

#include "cdna4.h"
#include "kernels.h"

namespace cdna4 {

// The per-segment fields of a launch, each as the first segment's value and the distances
// of the others': a select among the fields of the argument block (or of a struct holding
// them) is turned into an indexed load, for which the whole block is copied to scratch.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <typename T> __device__ __forceinline__ T scalar(T v) {
    asm volatile("" : "+s"(v));
    return v;
}
#pragma clang diagnostic pop
struct SegPtr {
    uint64_t p;                                // addresses as integers: p may be null
    int64_t d1, d2;
    __device__ __forceinline__ void load(const void* p0, const void* p1, const void* p2) {
        p = scalar((uint64_t)(uintptr_t)p0);
        d1 = scalar((int64_t)((uintptr_t)p1 - (uintptr_t)p0));
        d2 = scalar((int64_t)((uintptr_t)p2 - (uintptr_t)p0));
    }
    __device__ __forceinline__ CF_GLOBAL float* at(int s) const {
        return (CF_GLOBAL float*)(p + (uint64_t)(s == 1 ? d1 : (int64_t)0) + (uint64_t)(s == 2 ? d2 : (int64_t)0));
    }
};
struct Segs {
    SegPtr w, bias, out;
    int n0, dn1, dn2, start1, start2, total;
    __device__ __forceinline__ int of(int c) const { return (c >= start1 ? 1 : 0) + (c >= start2 ? 1 : 0); }
    __device__ __forceinline__ int width(int s) const { return n0 + (s == 1 ? dn1 : 0) + (s == 2 ? dn2 : 0); }
    __device__ __forceinline__ int start(int s) const { return (s >= 1 ? start1 : 0) + (s == 2 ? start2 - start1 : 0); }
};
__device__ __forceinline__ Segs load_segs(const cf_gemm_args_t& a) {
    Segs s;
    const int k1 = a.nseg > 1 ? 1 : 0, k2 = a.nseg > 2 ? 2 : k1;
    s.w.load(a.w[0], a.w[k1], a.w[k2]);
    s.bias.load(a.bias[0], a.bias[k1], a.bias[k2]);
    s.out.load(a.out[0], a.out[k1], a.out[k2]);
    s.n0 = scalar(a.n[0]);
    s.dn1 = scalar(a.n[k1] - a.n[0]);
    s.dn2 = scalar(a.n[k2] - a.n[0]);
    s.start1 = scalar(a.nseg > 1 ? a.n[0] : 0x7fffffff);
    s.start2 = scalar(a.nseg > 2 ? a.n[0] + a.n[1] : 0x7fffffff);
    s.total = scalar(a.n[0] + (a.nseg > 1 ? a.n[1] : 0) + (a.nseg > 2 ? a.n[2] : 0));
    return s;
}

// acc[i][j][e] = C[m0 + 16 i + lr][n0 + 16 j + 4 lq + e] of the wave; columns are the
// segments side by side (widths multiples of 16).  part: this range of k's plane of fp32
// sums, [M][columns]; else bias and residual are added and the result goes out row-major
// (or row-concatenated), or head-major as q, k (B, H, S, d) and v^T (B, H, d, S).
template <int MI, int NJ>
__device__ __forceinline__ void store_f32_ct(const cf_gemm_args_t& a, const Segs& sg, int m0, int n0, int lr, int lq,
                                             const f4_t (&acc)[MI][NJ], float* part) {
    const int ntot = sg.total;
    const CF_GLOBAL float* const res = (const CF_GLOBAL float*)a.residual;
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int n = n0 + 16 * j + 4 * lq;
        if (n >= ntot) continue;
        if (part) {
#pragma unroll
            for (int i = 0; i < MI; i++) {
                const int m = m0 + 16 * i + lr;
                if (m < a.M) *(f4_t*)(part + (size_t)m * ntot + n) = acc[i][j];
            }
            continue;
        }
        const int seg = sg.of(n), col = n - sg.start(seg);
        const CF_GLOBAL float* bias = sg.bias.at(seg);
        const f4_t b = bias ? *(const CF_GLOBAL f4_t*)(bias + col) : f4_t{0.f, 0.f, 0.f, 0.f};
        if (a.out_kind != CF_GEMM_OUT_QKV) {
#pragma unroll
            for (int i = 0; i < MI; i++) {
                const int m = m0 + 16 * i + lr;
                if (m >= a.M) continue;
                f4_t v = acc[i][j] + b;
                if (res) v += *(const CF_GLOBAL f4_t*)(res + (size_t)m * ntot + n);
                *(CF_GLOBAL f4_t*)(sg.out.at(0) + (size_t)m * ntot + n) = v;
            }
        } else {
            // d % 4 == 0: the four columns are dims of one head.
            const int H = seg == 0 ? a.H_q : a.H_kv, h = col / a.d, dd = col - h * a.d;
            CF_GLOBAL float* const o = sg.out.at(seg);
#pragma unroll
            for (int i = 0; i < MI; i++) {
                const int m = m0 + 16 * i + lr;
                if (m >= a.M) continue;
                const f4_t v = acc[i][j] + b;
                const int bb = m / a.S, s = m - bb * a.S;
                if (seg < 2) *(CF_GLOBAL f4_t*)(o + (((size_t)bb * H + h) * a.S + s) * a.d + dd) = v;
                else
#pragma unroll
                    for (int e = 0; e < 4; e++) o[(((size_t)bb * H + h) * a.d + dd + e) * a.S + s] = v[e];
            }
        }
    }
}

// Position of workgroup blk in an XCD-aware order of tiles_m x tiles_n tiles: each XCD
// takes a contiguous range, column-major over groups of 4 row tiles.
__device__ __forceinline__ void xcd_tile(int blk, int tiles_m, int tiles_n, int& tm, int& tn) {
    const int T = tiles_m * tiles_n, xc = blk & 7, t = xc * (T / 8) + min(xc, T % 8) + (blk >> 3);
    const int per = 4 * tiles_n, g = t / per, first = 4 * g, gm = min(tiles_m - first, 4), r = t - g * per;
    tn = r / gm;
    tm = first + (r - tn * gm);
}

}  // namespace cdna4

#endif  // CF_GEMM_F32_STORE_H_
