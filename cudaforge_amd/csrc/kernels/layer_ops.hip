// layer_ops.hip — the operators next to attention in an FP16 transformer layer that
// keep it on the device: LayerNorm (layernorm.c:85-122, norm_f16_cuda.cu:47-108), the
// Cast conversions (cast_cuda.cu:6-64) and the transpose the MatMul op needs for its
// transposed operands (matmul_cuda.cu:320-352).  All HBM-bound, so: one wave per
// LayerNorm row with 8-byte vector accesses and the row kept in registers, grid-stride
// elementwise loops, and an LDS-tiled transpose.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.h"
#include "cdna4.h"

namespace {

using cdna4::wave_sum;   // DPP and row swaps: no LDS round trip per reduction step

template <typename T> struct Vec4;
template <> struct Vec4<float> { typedef float type __attribute__((ext_vector_type(4))); };
template <> struct Vec4<_Float16> { typedef _Float16 type __attribute__((ext_vector_type(4))); };

// LayerNorm, WPR waves (1 or 4) per row; thread r of the row holds VPL groups of 4
// consecutive elements (group j: elements 4*(64*WPR*j + r) .. +3, masked past the end).
// Requires D % 4 == 0 and 8/16-byte aligned rows.  Every load is unconditional (clamped to
// the row's last group), gain and bias included, so a row costs one round trip to memory:
// under a branch each group's load was waited for before the next (16 rows x 4096, 16
// groups per lane: 16.0 us in a kernel trace; 4.8 us with four waves per row).
constexpr int kRowsX = 65536;                      // rows along x of a grid with a workgroup per row
template <typename T, int VPL, int WPR>
__global__ __launch_bounds__(256) void layernorm_vec(cf_layernorm_args_t a) {
    typedef typename Vec4<T>::type V;
    constexpr int TPR = 64 * WPR;                  // threads per row
    __shared__ float red[2][4];
    const int r = threadIdx.x % TPR, wave = threadIdx.x >> 6;
    // kRowsX and not gridDim.x: a kernel that reads its grid's size gets it in hidden arguments
    // behind its own, and short launches one after another took 3.2 us each instead of 2.7.
    const int64_t row = WPR == 4 ? (int64_t)blockIdx.y * kRowsX + blockIdx.x
                                 : (int64_t)blockIdx.x * (256 / TPR) + threadIdx.x / TPR;
    if (row >= a.N) return;                        // WPR == 4: the whole workgroup
    const int D = a.D, ng = D >> 2;
    const V* x = (const V*)((const T*)a.x + row * D);
    const V* g = (const V*)a.gamma;
    const V* b = (const V*)a.beta;
    V q[VPL], gv[VPL], bv[VPL];
#pragma unroll
    for (int j = 0; j < VPL; j++) q[j] = x[min(TPR * j + r, ng - 1)];
#pragma unroll
    for (int j = 0; j < VPL; j++) {
        gv[j] = g[min(TPR * j + r, ng - 1)];
        bv[j] = b[min(TPR * j + r, ng - 1)];
    }
    auto row_sum = [&](float s, int k) {
        s = wave_sum(s);
        if constexpr (WPR == 1) return s;
        if ((threadIdx.x & 63) == 0) red[k][wave] = s;
        __syncthreads();
        return (red[k][0] + red[k][1]) + (red[k][2] + red[k][3]);
    };
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < VPL; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) s += TPR * j + r < ng ? (float)q[j][e] : 0.0f;
    const float mean = row_sum(s, 0) / (float)D;
    float q2 = 0.0f;
#pragma unroll
    for (int j = 0; j < VPL; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float dv = (float)q[j][e] - mean;
            q2 += TPR * j + r < ng ? dv * dv : 0.0f;
        }
    const float inv_std = 1.0f / sqrtf(row_sum(q2, 1) / (float)D + a.eps);
    V* y = (V*)((T*)a.y + row * D);
#pragma unroll
    for (int j = 0; j < VPL; j++) {
        const int gi = TPR * j + r;
        V o;
#pragma unroll
        for (int e = 0; e < 4; e++) o[e] = (T)(((float)q[j][e] - mean) * inv_std * (float)gv[j][e] + (float)bv[j][e]);
        if (gi < ng) y[gi] = o;
    }
}

// Any D: one wave per row, three passes over the row (it stays in L1/L2).
template <typename T>
__global__ __launch_bounds__(256) void layernorm_any(cf_layernorm_args_t a) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= a.N) return;
    const int D = a.D;
    const T* x = (const T*)a.x + row * D;
    float s = 0.0f;
    for (int i = lane; i < D; i += 64) s += (float)x[i];
    const float mean = wave_sum(s) / (float)D;
    float q2 = 0.0f;
    for (int i = lane; i < D; i += 64) { const float dv = (float)x[i] - mean; q2 += dv * dv; }
    const float inv_std = 1.0f / sqrtf(wave_sum(q2) / (float)D + a.eps);
    const T* g = (const T*)a.gamma;
    const T* b = (const T*)a.beta;
    T* y = (T*)a.y + row * D;
    for (int i = lane; i < D; i += 64) y[i] = (T)(((float)x[i] - mean) * inv_std * (float)g[i] + (float)b[i]);
}

template <typename T, int VPL>
void launch_layernorm_vec(const cf_layernorm_args_t& a, bool wide, hipStream_t s) {
    // A workgroup per row: beyond kRowsX rows along y, as a launch holds fewer than 2^32 threads
    // along x (2^24 rows, which four rows per workgroup do not reach).
    if (wide)
        hipLaunchKernelGGL((layernorm_vec<T, VPL, 4>),
                           dim3((unsigned)(a.N < kRowsX ? a.N : kRowsX), (unsigned)((a.N + kRowsX - 1) / kRowsX)),
                           dim3(256), 0, s, a);
    else hipLaunchKernelGGL((layernorm_vec<T, VPL, 1>), dim3((unsigned)((a.N + 3) / 4)), dim3(256), 0, s, a);
}

template <typename T>
hipError_t launch_layernorm(const cf_layernorm_args_t& a, hipStream_t s) {
    const uintptr_t al = (uintptr_t)a.x | (uintptr_t)a.y | (uintptr_t)a.gamma | (uintptr_t)a.beta;
    const bool vec = a.D % 4 == 0 && al % (4 * sizeof(T)) == 0;
    // Four waves per row for long rows (a wave would hold more than 8 groups per lane in fp16,
    // 6 in fp32: with gain and bias 8 take 96 registers, and 4096 rows of 1792 took 11.6 us
    // against 9.9, 8192 of 2048 21.6 and 20.0) and while one wave per row gives the CUs less
    // than two waves each.
    const int g1 = (a.D / 4 + 63) / 64;
    const bool wide = g1 > (sizeof(T) == 4 ? 6 : 8) || (g1 > 1 && a.N < 2LL * cdna4::cu_count());
    const int groups = wide ? (a.D / 4 + 255) / 256 : g1;
    if (!vec || groups > 8 || (wide && a.N > 0x7fffffffLL))
        hipLaunchKernelGGL((layernorm_any<T>), dim3((unsigned)((a.N + 3) / 4)), dim3(256), 0, s, a);
    else if (groups <= 1) launch_layernorm_vec<T, 1>(a, wide, s);
    else if (groups <= 2) launch_layernorm_vec<T, 2>(a, wide, s);
    else if (groups <= 3) launch_layernorm_vec<T, 3>(a, wide, s);
    else if (groups <= 4) launch_layernorm_vec<T, 4>(a, wide, s);
    else if (groups <= 6) launch_layernorm_vec<T, 6>(a, wide, s);
    else launch_layernorm_vec<T, 8>(a, wide, s);
    return hipGetLastError();
}

// Cast: grid-stride elementwise.  Between f32 and f16, 2048 elements per workgroup: where both
// ends are 16-byte aligned (`vec`) eight per thread with 16-byte accesses (the last n % 8 one by
// one), else eight passes over consecutive ones.  67 million to fp16 and back: aligned 68 and
// 71 us, misaligned 97 and 120 (one per thread, grid-stride, 108 and 143); eight consecutive ones per thread one by one, which touch a
// line per lane and access, took 214 and 212.
template <typename I, typename O>
__device__ __forceinline__ void cast2048(const I* __restrict__ in, O* __restrict__ out, int64_t i0, int64_t n, bool vec) {
    typedef I i8_t __attribute__((ext_vector_type(8)));
    typedef O o8_t __attribute__((ext_vector_type(8)));
    if (vec) {
        const int64_t i = i0 + 8 * threadIdx.x;
        if (i + 8 <= n) {
            *(o8_t*)(out + i) = __builtin_convertvector(*(const i8_t*)(in + i), o8_t);
        } else {
            for (int64_t j = i; j < n; j++) out[j] = (O)in[j];
        }
    } else {
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int64_t i = i0 + 256 * k + threadIdx.x;
            if (i < n) out[i] = (O)in[i];
        }
    }
}
template <typename I, typename O>
__global__ __launch_bounds__(256) void cast8_kernel(const I* __restrict__ in, O* __restrict__ out, int64_t n, bool vec,
                                                    int64_t stride) {
    for (int64_t i = (int64_t)blockIdx.x * 2048; i < n; i += stride) cast2048(in, out, i, n, vec);
}

// Several f32 -> f16 arrays in one launch (the mixed-precision prefill's ten operands, whose
// ten launches of 1.5-3.2 us took longer than its products): entry e owns workgroups
// first[e] .. first[e+1] - 1 of 2048 elements each.
struct CastMany {
    cf_cast_many_args_t a;
    unsigned first[CF_CAST_MANY + 1];
    unsigned vec;                      // bit e: entry e's ends are aligned
};
__global__ __launch_bounds__(256) void cast_many_kernel(CastMany c) {
    int e = 0;
#pragma unroll
    for (int k = 1; k < CF_CAST_MANY; k++) e += blockIdx.x >= c.first[k] ? 1 : 0;
    cast2048((const float*)c.a.in[e], (_Float16*)c.a.out[e], (int64_t)(blockIdx.x - c.first[e]) * 2048, c.a.n[e],
             (c.vec >> e) & 1u);
}

template <typename I, typename O>
__global__ __launch_bounds__(256) void cast_kernel(const I* __restrict__ in, O* __restrict__ out, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
        out[i] = (O)in[i];
}

// Transpose through a 64 x 65 LDS tile (the pad keeps column reads conflict-free).
template <typename T>
__global__ __launch_bounds__(256) void transpose_kernel(const T* __restrict__ in, T* __restrict__ out,
                                                        int64_t rows, int64_t cols, int64_t in_stride,
                                                        int64_t out_stride) {
    __shared__ T tile[64][65];
    const int64_t b = blockIdx.z;
    const int64_t r0 = (int64_t)blockIdx.y * 64, c0 = (int64_t)blockIdx.x * 64;
    const T* src = in + b * in_stride;
    T* dst = out + b * out_stride;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    for (int r = ty; r < 64; r += 4)
        if (r0 + r < rows && c0 + tx < cols) tile[r][tx] = src[(r0 + r) * cols + c0 + tx];
    __syncthreads();
    for (int c = ty; c < 64; c += 4)
        if (c0 + c < cols && r0 + tx < rows) dst[(c0 + c) * rows + r0 + tx] = tile[tx][c];
}

unsigned grid_1d(int64_t n) {
    const int64_t blocks = (n + 255) / 256;
    return (unsigned)(blocks < 65536 ? (blocks > 0 ? blocks : 1) : 65536);
}

}  // namespace

extern "C" int cf_launch_layernorm(const cf_layernorm_args_t* a, void* stream) {
    if (!a || !a->x || !a->gamma || !a->beta || !a->y || a->N < 0 || a->D <= 0) return (int)hipErrorInvalidValue;
    if (a->N == 0) return 0;
    if ((a->N + 3) / 4 > 0x7fffffffLL) return (int)hipErrorInvalidValue;
    hipStream_t s = (hipStream_t)stream;
    return (int)(a->elem == CF_ELEM_F16 ? launch_layernorm<_Float16>(*a, s) : launch_layernorm<float>(*a, s));
}

extern "C" int cf_launch_cast(const void* in, void* out, int64_t n, int32_t kind, void* stream) {
    if (!in || !out || n < 0) return (int)hipErrorInvalidValue;
    if (n == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    const dim3 g(grid_1d(n)), g8(grid_1d((n + 7) / 8)), b(256);
    const bool vec = ((uintptr_t)in | (uintptr_t)out) % 16 == 0;
    const int64_t stride = 2048 * (int64_t)g8.x;           // passed: gridDim.x is a hidden argument (layernorm_vec)
    switch (kind) {
        case CF_CAST_I64_F32: hipLaunchKernelGGL((cast_kernel<int64_t, float>), g, b, 0, s, (const int64_t*)in, (float*)out, n); break;
        case CF_CAST_F32_I64: hipLaunchKernelGGL((cast_kernel<float, int64_t>), g, b, 0, s, (const float*)in, (int64_t*)out, n); break;
        case CF_CAST_F32_F16: hipLaunchKernelGGL((cast8_kernel<float, _Float16>), g8, b, 0, s, (const float*)in, (_Float16*)out, n, vec, stride); break;
        case CF_CAST_F16_F32: hipLaunchKernelGGL((cast8_kernel<_Float16, float>), g8, b, 0, s, (const _Float16*)in, (float*)out, n, vec, stride); break;
        default: return (int)hipErrorInvalidValue;
    }
    return (int)hipGetLastError();
}

extern "C" int cf_launch_cast_many(const cf_cast_many_args_t* a, void* stream) {
    CastMany c;
    c.a = *a;
    c.vec = 0;
    unsigned long long at = 0;
    for (int e = 0; e < CF_CAST_MANY; e++) {
        c.first[e] = (unsigned)at;
        if (a->n[e] < 0 || (a->n[e] > 0 && (!a->in[e] || !a->out[e]))) return (int)hipErrorInvalidValue;
        if (((uintptr_t)a->in[e] | (uintptr_t)a->out[e]) % 16 == 0) c.vec |= 1u << e;
        at += ((unsigned long long)a->n[e] + 2047) / 2048;
        if (at > 0x7fffffffULL) return (int)hipErrorInvalidValue;
    }
    c.first[CF_CAST_MANY] = (unsigned)at;
    if (at == 0) return 0;
    hipLaunchKernelGGL(cast_many_kernel, dim3((unsigned)at), dim3(256), 0, (hipStream_t)stream, c);
    return (int)hipGetLastError();
}

extern "C" int cf_launch_transpose(const void* in, void* out, int64_t rows, int64_t cols, int64_t batch,
                                   int64_t in_stride, int64_t out_stride, int32_t elem_bytes, void* stream) {
    if (!in || !out || rows < 0 || cols < 0 || batch < 1 || (elem_bytes != 2 && elem_bytes != 4))
        return (int)hipErrorInvalidValue;
    if (rows == 0 || cols == 0) return 0;
    const int64_t gx = (cols + 63) / 64, gy = (rows + 63) / 64;
    if (gx > 0x7fffffffLL || gy > 65535 || batch > 65535) return (int)hipErrorInvalidValue;
    const dim3 g((unsigned)gx, (unsigned)gy, (unsigned)batch), b(256);
    hipStream_t s = (hipStream_t)stream;
    if (elem_bytes == 2)
        hipLaunchKernelGGL(transpose_kernel<uint16_t>, g, b, 0, s, (const uint16_t*)in, (uint16_t*)out, rows, cols,
                           in_stride, out_stride);
    else
        hipLaunchKernelGGL(transpose_kernel<uint32_t>, g, b, 0, s, (const uint32_t*)in, (uint32_t*)out, rows, cols, in_stride,
                           out_stride);
    return (int)hipGetLastError();
}
