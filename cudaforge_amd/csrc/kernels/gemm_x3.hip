// gemm_x3.hip — FP32 products on the bf16 matrix cores (gfx950).
//
// The fp32 MFMA runs at 1/16 of the bf16 one's rate (157 against 2500 TFLOP/s), so large
// FP32 products are computed from a three-way split (Henry, Tang and Heinecke, "Leveraging the
// bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations", 2019):
// x = h + m + l exactly, h the nearest bf16 to x, m the nearest to the rest, l what is left, and
//   a b = ah bh + (ah bm + am bh) + (am bm + ah bl + al bh) + dropped,
// six bf16 MFMAs with fp32 accumulation for one fp32 product at 1/6 of 2500 TFLOP/s.  With
// |m| <= 2^-8 |x| and |l| <= 2^-17 |x| the three dropped terms are below 2^-24 |a b| together, of
// either sign.  (Cut instead of rounded parts drop up to 2^-21 |a b|, always towards zero: sums of
// one sign were 4.2e-8 too small on average, now 2e-10.)
// The bf16 MFMA cuts (towards minus infinity) what its products and C have below the last
// place of the largest.  With one running sum, six times per 32 k, all-positive operands of
// K = 4096 were off by 3.0e-6 and 14336 by 8.2e-6, against 0.9e-6 and 1.8e-6 of the fp32 kernel.
// So the six MFMAs of a 32-k stage start from zero and their sum is added to the running one by
// a rounded fp32 add (4096 x 2304 x 768 76 -> 81 us; placing the adds among the next column
// tile's MFMAs, or reading its operands ahead, gave nothing: 83-85 us).  What they still cut
// has one sign too (columns' means of 4096 rows were off by 1.9e-6, the fp32 kernel's by 5.1e-7),
// so the parts of A are stored negated for every second stage and that stage's sum is
// subtracted: 1.3e-7, at no cost.
// Relative 2-norm error against float64, N(0, 1) x N(0, 0.02), fp32 MFMA kernel -> this one:
// K = 768 5.0e-7 -> 1.0e-7, 4096 1.1e-6 -> 1.6e-7, 14336 2.1e-6 -> 2.0e-7; all-positive operands
// 4.3e-7 -> 0.8e-7, 9.3e-7 -> 0.9e-7, 1.8e-6 -> 0.9e-7.
// Times, the 128 x 128 fp32 MFMA kernel (gemm.hip) -> this one with the splitting launch:
// 4096 x 2304 x 768 170 -> 81 us, 4096 x 768 x 768 68 -> 37, 2048 x 1024 x 4096 383 -> 111.
// What bounds it: the stage of one compute wave per SIMD.  On 256 x 144 tiles that is 216 MFMAs
// (3456 clk), 144 fp32 adds and 39 LDS reads of 1 KB that one wave does not overlap whole: by
// the counters the matrix cores are busy 44 % of the 4096 x 2304 x 768 product (1.14 PFLOP/s of
// bf16) and 35 % of 4096 x 768 x 768 on 128 x 96; the chip itself holds 2.4 PFLOP/s of 16-bit
// MFMAs.  Beside it, about 11 and 8 us of splitting at those shapes.
//
// 1. split_kernel writes both operands' parts in MFMA fragment order: units of 16 rows (of
//    A, or columns of W) x 32 k, 1 KB each, lane (lr, lq)'s 16 bytes at lane * 16 = row lr,
//    k 8 lq .. +7.  A unit is one direct-to-LDS load instruction of contiguous memory and
//    one conflict-free ds_read_b128, whatever the layout of the operand was.
// 2. gemm_x3: 4 loader and 4 compute waves as in gemm_f16_ws, 32-k stages of (BM + BN) / 16
//    x 3 units.
// Infinities and NaN cannot be split (inf - inf is NaN, and so is every sum it enters): a
// compute wave whose sums are not all finite computes its part of the tile again from the
// original operands on the fp32 MFMA, with the results the fp32 kernel would have.  Nothing is
// kept for another tile, launch or replay of a recording.
// Very small numbers cannot be split either: the bf16 MFMA takes subnormal operands as zero, so
// below 2^-103 the last part is lost, below 2^-118 the second (1e-37 x 1e5 was off by 1e-3).  Where a
// row's 32 k hold such a number and nothing from 2^-95 on, its parts are stored as NaN, with the
// same consequence; beside a larger number what is lost is below 2^-31 of that.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "kernels.h"
#include "cdna4.h"
#include "gemm_f32_store.h"
#include "gemm_x3.h"

namespace {

using namespace cdna4;

typedef __bf16 b8_t __attribute__((ext_vector_type(8)));
constexpr int kUnit = 512;                 // halves per unit (16 rows x 32 k)

struct X3Args {
    cf_gemm_args_t g;
    uint16_t* ap;                          // A's parts, [row tile][k tile][3] units
    uint16_t* wp;                          // W's, [column tile][k tile][3], segments side by side
    int       mt, nt, kt;                  // tiles of 16 rows, 16 columns, 32 k
    int       tiles_m, tiles_n;
    int       ks, per;                     // ranges of k (blockIdx.y) and their 32-k stages
    float*    part;                        // ks > 1: sums [range][M][columns]
};

// x to the nearest bf16 (ties to even), as the upper half of a float.
__device__ __forceinline__ uint32_t nearest_bf16(float x) {
    const uint32_t u = __float_as_uint(x);
    return (u + 0x7fffu + ((u >> 16) & 1u)) & 0xffff0000u;
}
// The three parts of x, as the upper halves of three floats.  Where rounding up would leave the
// finite numbers h is cut instead (and an infinity's or NaN's m is NaN).
__device__ __forceinline__ void split3(float x, uint32_t& h, uint32_t& m, uint32_t& l) {
    h = nearest_bf16(x);
    h = (h & 0x7f800000u) == 0x7f800000u ? __float_as_uint(x) & 0xffff0000u : h;
    const float r = x - __uint_as_float(h);
    m = (__float_as_uint(r) & 0x7f800000u) == 0x7f800000u ? 0x7fc00000u : nearest_bf16(r);
    l = __float_as_uint(r - __uint_as_float(m));          // at most 7 bits: its lower half is zero
}
__device__ __forceinline__ uint32_t pack_hi(uint32_t a, uint32_t b) { return (a >> 16) | (b & 0xffff0000u); }

constexpr uint32_t kTiny = (127u - 103u) << 23, kSmall = (127u - 95u) << 23;     // 2^-103, 2^-95

// One unit per wave: lane (lr, lq) takes row lr's k 8 lq .. +7.  Workgroups 0 .. (A's row
// tiles x k tile groups) - 1 split A, the rest W.  Bound by memory (4 bytes in, 6 out).
__global__ __launch_bounds__(256)
void split_kernel(X3Args x, int a_wgs) {
    const cf_gemm_args_t& a = x.g;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lr = lane & 15, lq = lane >> 4;
    const int K = a.K, kg = (x.kt + 3) / 4;               // k tile groups of 4 (one per wave)
    int id = blockIdx.x;
    const bool is_w = id >= a_wgs;
    if (is_w) id -= a_wgs;
    const int t = id / kg, kt = (id - t * kg) * 4 + wave;
    if (kt >= x.kt) return;
    const int k0 = 32 * kt + 8 * lq;
    float v[8];
    uint16_t* dst;
    if (!is_w || a.w_nk) {
        // Rows contiguous along k: A, or W given as (N, K).
        const int rows = is_w ? a.n[0] : a.M;
        const float* src = (const float*)(is_w ? a.w[0] : a.a) + (size_t)min(16 * t + lr, rows - 1) * K + k0;
        const f4_t v0 = *(const f4_t*)src, v1 = *(const f4_t*)(src + 4);
#pragma unroll
        for (int e = 0; e < 4; e++) { v[e] = v0[e]; v[4 + e] = v1[e]; }
        dst = is_w ? x.wp : x.ap;
    } else {
        // W (K, N): eight rows of one column; segment widths are multiples of 16.
        const Segs sg = load_segs(a);
        const int c = 16 * t, seg = sg.of(c), N = sg.width(seg);
        const CF_GLOBAL float* src = sg.w.at(seg) + (size_t)k0 * N + (c - sg.start(seg)) + lr;
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = src[(size_t)e * N];
        dst = x.wp;
    }
    uint32_t h[8], m[8], l[8];
#pragma unroll
    for (int e = 0; e < 8; e++) split3(v[e], h[e], m[e], l[e]);
    // The bf16 MFMA takes subnormal operands as zero, and parts go down to 2^-23 of x: see the top.
    uint32_t least = 0xffffffffu, most = 0;                // of 2 |x| - 1 (0: the largest), and |x|, as bits
#pragma unroll
    for (int e = 0; e < 8; e++) {
        least = min(least, (__float_as_uint(v[e]) << 1) - 1u);
        most = max(most, __float_as_uint(v[e]) & 0x7fffffffu);
    }
    if (__builtin_amdgcn_ballot_w64(least < 2u * kTiny)) {
        most = max(most, (uint32_t)__shfl_xor((int)most, 16));
        most = max(most, (uint32_t)__shfl_xor((int)most, 32));     // of the row's 32 k
        if (most > 0 && most < kSmall)
#pragma unroll
            for (int e = 0; e < 8; e++) m[e] = 0x7fc00000u;
    }
    const uint32_t neg = !is_w && (kt & 1) ? 0x80008000u : 0u;       // every second stage of A: see the top
    uint4* const o = (uint4*)(dst + (size_t)(t * x.kt + kt) * (3 * kUnit)) + lane;
    auto put = [&](int part, const uint32_t (&v)[8]) {
        o[64 * part] = uint4{pack_hi(v[0], v[1]) ^ neg, pack_hi(v[2], v[3]) ^ neg, pack_hi(v[4], v[5]) ^ neg,
                             pack_hi(v[6], v[7]) ^ neg};
    };
    put(0, h);
    put(1, m);
    put(2, l);
}

// NCW compute waves, WMC of them along M.  Two per SIMD (8) where the tile divides among
// them: one's MFMAs cover the other's LDS reads.
template <int BM, int BN, int NCW, int WMC>
struct X3Shape {
    static constexpr int WM = BM / WMC, WN = BN * WMC / NCW;   // rows and columns of a compute wave
    static constexpr int MI = WM / 16, NJ = WN / 16;
    static constexpr int AU = BM / 16 * 3, WU = BN / 16 * 3, U = AU + WU;   // units per stage
    static constexpr int PW = (U + 3) / 4;            // load instructions per loader wave, at most
    static constexpr int ST = U * kUnit;              // halves per stage
    static_assert(WM % 16 == 0 && BN * WMC % (16 * NCW) == 0, "wave tile");
};
template <int BM, int BN, int NCW, int WMC, int S>
constexpr unsigned x3_lds_bytes() { return (unsigned)S * X3Shape<BM, BN, NCW, WMC>::ST * 2u; }

// The product.  Stages of 32 k; a compute wave owns MI x NJ tiles of 16 x 16 and runs 6 MI
// MFMAs per 16 columns and stage, the smallest terms first.  Results go out straight from
// the accumulators (C^T: four consecutive columns per lane, 16 bytes).
template <int BM, int BN, int NCW, int WMC, int S>
__global__ __launch_bounds__(64 * (NCW + 4), 1)
void gemm_x3(X3Args x) {
    using SH = X3Shape<BM, BN, NCW, WMC>;
    constexpr int MI = SH::MI, NJ = SH::NJ, U = SH::U, AU = SH::AU, PW = SH::PW, ST = SH::ST;
    extern __shared__ __attribute__((aligned(16))) uint16_t smem_x3[];
    const cf_gemm_args_t& a = x.g;
    int tm, tn;
    xcd_tile((int)blockIdx.x, x.tiles_m, x.tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN, K = a.K;
    const int kt0 = (int)blockIdx.y * x.per, nk = min(x.kt - kt0, x.per);    // no range is empty
    const Segs sg = load_segs(a);
    const int ntot = sg.total;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    if (wave >= NCW) {
        const int cw = wave & 3;
        uint32_t off[PW];
        int nu = 0;
#pragma unroll
        for (int v = 0; v < PW; v++) {
            const int u = cw + 4 * v;
            nu += u < U ? 1 : 0;
            const int tl = u < AU ? min(m0 / 16 + u / 3, x.mt - 1) : min(n0 / 16 + min(u - AU, SH::WU - 1) / 3, x.nt - 1);
            off[v] = (uint32_t)tl * (uint32_t)x.kt * 3072u + (uint32_t)(u % 3) * 1024u + (uint32_t)lane * 16u;
        }
        const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_offset(smem_x3) + (uint32_t)cw * 1024u);
        auto issue = [&](int kt, int stage) {
            const uint16_t* ab = x.ap + (size_t)(kt0 + kt) * (3 * kUnit);
            const uint16_t* wb = x.wp + (size_t)(kt0 + kt) * (3 * kUnit);
            const uint32_t so = lds0 + (uint32_t)stage * (ST * 2u);
#pragma unroll
            for (int v = 0; v < PW; v++)
                if (v < nu) lds_dma16_s(off[v], cw + 4 * v < AU ? ab : wb, so + 4096u * v);
        };
        auto wait = [&](int ahead) {
            if (nu == PW) wait_ahead<PW, S - 2>(ahead);
            else wait_ahead<PW - 1, S - 2>(ahead);
        };
        for (int s = 0; s < S - 1 && s < nk; s++) issue(s, s);
        wait(min(S - 2, nk - 1));
        ring_barrier();
        for_each_stage<S>(nk, [&](int kt, auto stage_c) {
            constexpr int stage = decltype(stage_c)::value;
            if (kt + S - 1 < nk) issue(kt + S - 1, (stage + S - 1) % S);
            if (kt + 1 < nk) wait(min(S - 2, nk - 2 - kt));
            ring_barrier();
        });
        return;
    }

    const int wm = SH::WM * (wave % WMC), wn = SH::WN * (wave / WMC);
    f4_t acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[i][j] = f4_t{0.f, 0.f, 0.f, 0.f};

    {
        const uint16_t* const a_rd = smem_x3 + (wm / 16) * (3 * kUnit) + lane * 8;
        const uint16_t* const w_rd = smem_x3 + (AU + (wn / 16) * 3) * kUnit + lane * 8;
        ring_barrier();
        for_each_stage<S % 2 ? 2 * S : S>(nk, [&](int, auto stage_c) {
            constexpr int stage = decltype(stage_c)::value % S;
            constexpr bool odd = decltype(stage_c)::value % 2;     // kt0 is even
            b8_t af[MI][3];
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int p = 0; p < 3; p++) af[i][p] = *(const b8_t*)(a_rd + stage * ST + (3 * i + p) * kUnit);
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                b8_t bf[3];
#pragma unroll
                for (int p = 0; p < 3; p++) bf[p] = *(const b8_t*)(w_rd + stage * ST + (3 * j + p) * kUnit);
                constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};
                f4_t sum[MI];              // from zero: see the top
#pragma unroll
                for (int i = 0; i < MI; i++) sum[i] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int q = 0; q < 6; q++)
#pragma unroll
                    for (int i = 0; i < MI; i++)
                        sum[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[PB[q]], af[i][PA[q]], sum[i], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < MI; i++) {
                    if constexpr (odd) acc[i][j] -= sum[i];
                    else acc[i][j] += sum[i];
                }
            }
            ring_barrier();
        });
    }
    // 0 x sum: NaN where the sum is not finite.  A row (column) with a non-finite operand has no
    // finite sum at all, so one column of every row and one row of every column tell.
    float test[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) test[e] = __builtin_fmaf(acc[0][j][e], 0.0f, test[e]);
#pragma unroll
    for (int i = 1; i < MI; i++) test[i & 3] = __builtin_fmaf(acc[i][0][0], 0.0f, test[i & 3]);
    if (__builtin_amdgcn_ballot_w64(__float_as_uint((test[0] + test[1]) + (test[2] + test[3])) << 1)) {
        // From the original operands: lane (lr, lq) loads row (column) lr's k0 + lq.
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++) acc[i][j] = f4_t{0.f, 0.f, 0.f, 0.f};
        const float* ar[MI];
        const CF_GLOBAL float* wr[NJ];
        size_t wst[NJ];
#pragma unroll
        for (int i = 0; i < MI; i++) ar[i] = (const float*)a.a + (size_t)min(m0 + wm + 16 * i + lr, a.M - 1) * K + 32 * kt0 + lq;
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const int c = min(n0 + wn + 16 * j + lr, ntot - 1);
            const int seg = sg.of(c), N = sg.width(seg), col = c - sg.start(seg);
            wr[j] = sg.w.at(seg) + (a.w_nk ? (size_t)col * K + 32 * kt0 + lq : (size_t)(32 * kt0 + lq) * N + col);
            wst[j] = a.w_nk ? 4 : (size_t)4 * N;
        }
        for (int k = 0; k < 32 * nk; k += 4) {
            float av[MI];
#pragma unroll
            for (int i = 0; i < MI; i++) av[i] = ar[i][k];
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                const float bv = *wr[j];
                wr[j] += wst[j];
#pragma unroll
                for (int i = 0; i < MI; i++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bv, av[i], acc[i][j], 0, 0, 0);
            }
        }
    }

    store_f32_ct<MI, NJ>(a, sg, m0 + wm, n0 + wn, lr, lq, acc,
                         x.ks > 1 ? x.part + (size_t)blockIdx.y * a.M * ntot : nullptr);
}

template <int BM, int BN, int NCW, int WMC, int S>
hipError_t launch_x3(dim3 grid, hipStream_t st, const X3Args& x) {
    constexpr unsigned lds = x3_lds_bytes<BM, BN, NCW, WMC, S>();
    static std::atomic<uint64_t> raised{0};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev >= 64 || !((raised.load(std::memory_order_acquire) >> dev) & 1u)) {
        e = hipFuncSetAttribute((const void*)gemm_x3<BM, BN, NCW, WMC, S>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        if (dev < 64) raised.fetch_or(1ull << dev, std::memory_order_release);
    }
    hipLaunchKernelGGL((gemm_x3<BM, BN, NCW, WMC, S>), grid, dim3(64 * (NCW + 4)), lds, st, x);
    return hipSuccess;
}

struct X3Candidate {
    int bm, bn;
    hipError_t (*launch)(dim3, hipStream_t, const X3Args&);
};
const X3Candidate kX3Shapes[] = {
    {256, 160, launch_x3<256, 160, 8, 4, 2>}, {256, 144, launch_x3<256, 144, 4, 4, 2>},
    {256, 128, launch_x3<256, 128, 8, 4, 2>}, {256, 96, launch_x3<256, 96, 8, 4, 2>},
    {256, 64, launch_x3<256, 64, 8, 4, 2>},   {128, 192, launch_x3<128, 192, 8, 2, 2>},
    {128, 128, launch_x3<128, 128, 8, 2, 3>}, {128, 96, launch_x3<128, 96, 8, 4, 3>},
    {128, 64, launch_x3<128, 64, 8, 4, 4>},   {64, 64, launch_x3<64, 64, 8, 2, 6>},
};
constexpr int kX3Count = (int)(sizeof(kX3Shapes) / sizeof(kX3Shapes[0]));
constexpr int kX3MaxSplit = 16;
// Stages of each of ks ranges: even, so that every range starts with a stage of A as it is.
inline int x3_per(int kt, int ks) { return ks == 1 ? kt : (kt + 2 * ks - 1) / (2 * ks) * 2; }
int g_x3_mode = 0, g_x3_bm = 0, g_x3_bn = 0, g_x3_ks = 0;

}  // namespace

extern "C" void cf_gemm_set_x3(int32_t mode, int32_t bm, int32_t bn, int32_t ks) {
    g_x3_mode = mode;
    g_x3_ks = ks;
    g_x3_bm = bm;
    g_x3_bn = bn;
}

int gemm_x3_pick(const cf_gemm_args_t* a, int* ks_out, float* clk) {
    if (g_x3_mode == 1 || a->elem != CF_ELEM_F32 || a->out_f32) return -1;
    if (a->K % 32 != 0 || (uintptr_t)a->a % 16 != 0) return -1;
    if (a->w_nk && (a->nseg != 1 || a->out_kind != CF_GEMM_OUT_ROWMAJOR || (uintptr_t)a->w[0] % 16 != 0)) return -1;
    if (a->out_kind == CF_GEMM_OUT_QKV && a->d % 4 != 0) return -1;
    uintptr_t al = (uintptr_t)a->residual;
    long long ntot = 0;
    for (int s = 0; s < a->nseg; s++) {
        if (a->n[s] % 16 != 0) return -1;
        ntot += a->n[s];
        al |= (uintptr_t)a->bias[s];
        if (s == 0 || a->out_kind == CF_GEMM_OUT_QKV) al |= (uintptr_t)a->out[s];
    }
    if (al % 16 != 0) return -1;
    const long long mt = (a->M + 15LL) / 16, nt = ntot / 16, kt = a->K / 32;
    // 32-bit unit offsets, and the splitting grid.
    if (mt * kt * 3072 >= (1LL << 32) || nt * kt * 3072 >= (1LL << 32)) return -1;
    const bool may_split = a->out_kind != CF_GEMM_OUT_QKV && (long long)a->M * ntot < (1LL << 30);
    const int cus = cu_count();
    int best = -1;
    *ks_out = 1;
    float best_cost = 0.0f;
    for (int i = 0; i < kX3Count; i++) {
        const X3Candidate& c = kX3Shapes[i];
        const long long tiles = (a->M + c.bm - 1LL) / c.bm * ((ntot + c.bn - 1) / c.bn);
        if (tiles > 0x7fffffffLL) continue;
        // Measured per 32-k stage with every CU busy: 450 clk plus 2900 FLOP/clk of MFMA
        // work (1.4-1.6 PFLOP/s over the chip; torch's bf16 8192^3 product ran at 1.2 here),
        // for tiles of 64 x 64 to 256 x 160 within 6 %; about 4000 clk per tile around it.
        // Ranges of k add a second launch (8900 clk) and the sums' way through memory.
        const float stage = 450.0f + (float)(c.bm * c.bn) * (32.0f * 2.0f * 6.0f / 2900.0f);
        for (int ks = 1; ks <= kX3MaxSplit; ks++) {
            const int per = x3_per((int)kt, ks);
            if (ks > 1 && (!may_split || tiles * ks > 2LL * cus || per < 4)) break;
            if (ks > 1 && (long long)(ks - 1) * per >= kt) continue;
            float cost = (float)((tiles * ks + cus - 1) / cus) * (stage * (float)per + 4000.0f);
            if (ks > 1) cost += 8900.0f + (float)ks * (float)a->M * (float)ntot * (8.0f / 1900.0f);
            if (c.bm == g_x3_bm && c.bn == g_x3_bn && (g_x3_ks == 0 ? ks == 1 : ks == g_x3_ks)) cost = -1.0f;
            if (best < 0 || cost < best_cost) {
                best = i;
                best_cost = cost;
                *ks_out = ks;
            }
        }
    }
    // ... and the splitting launch: 10 bytes of traffic per operand element.
    *clk = best_cost + 8900.0f + ((float)a->M * (float)a->K + (float)a->K * (float)ntot) * (10.0f / 2100.0f);
    if (g_x3_mode == 2) *clk = 0.0f;
    return best;
}

size_t gemm_x3_floats(const cf_gemm_args_t* a) {
    size_t ntot = 0;
    for (int s = 0; s < a->nseg; s++) ntot += (size_t)a->n[s];
    const size_t units = ((size_t)(a->M + 15) / 16 + ntot / 16) * (size_t)(a->K / 32) * 3;
    // 1 KB per unit, then the ranges' sums.
    return units * 256 + (a->ksplit > 1 ? (size_t)a->ksplit * (size_t)a->M * ntot : 0);
}

int gemm_x3_launch(const cf_gemm_args_t* a, int pick, hipStream_t st) {
    X3Args x;
    x.g = *a;
    int ntot = 0;
    for (int s = 0; s < a->nseg; s++) ntot += a->n[s];
    x.mt = (a->M + 15) / 16;
    x.nt = ntot / 16;
    x.kt = a->K / 32;
    x.ap = (uint16_t*)a->partials;
    x.wp = x.ap + (size_t)x.mt * x.kt * (3 * kUnit);
    const X3Candidate& c = kX3Shapes[pick];
    x.tiles_m = (a->M + c.bm - 1) / c.bm;
    x.tiles_n = (ntot + c.bn - 1) / c.bn;
    const int kg = (x.kt + 3) / 4;
    const long long wgs = (long long)(x.mt + x.nt) * kg;
    if (wgs > 0x7fffffffLL) return (int)hipErrorInvalidValue;
    hipLaunchKernelGGL(split_kernel, dim3((unsigned)wgs), dim3(256), 0, st, x, x.mt * kg);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
    x.ks = a->ksplit;
    x.per = x3_per(x.kt, x.ks);
    x.part = (float*)(x.wp + (size_t)x.nt * x.kt * (3 * kUnit));
    e = c.launch(dim3((unsigned)(x.tiles_m * x.tiles_n), (unsigned)x.ks), st, x);
    if (e == hipSuccess) e = hipGetLastError();
    if (e != hipSuccess || x.ks == 1) return (int)e;
    x.g.partials = x.part;
    return gemm_splitk_sum_launch(&x.g, st);
}
