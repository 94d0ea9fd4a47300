// gemm_f32_ws.hip — FP32 products of few rows on the fp32 MFMA (gfx950).
//
// Below a few hundred rows an FP32 product is bound by reading W, or by the latency of its
// k loop on the few CUs its tiles reach: the 128 x 128 register-staged kernel (gemm.hip)
// took 58 us for 8 x 768 x 768 and 1212 us for 16 x 14336 x 4096, whatever the rows.  Here 16-,
// 32- and 64-row tiles of 64 columns (or 32) stream both operands by DMA through a ring of
// 32-k stages (4 loader waves; 4 compute waves, as gemm_f16_ws), A in rows of 128 bytes, W as
// it is given ((K, N) rows, or (N, K) rows like A).  Every element sums its k in ascending
// order, four per MFMA step, like the reference's loop; only products with K >= 2048 split k
// over workgroups (fp32 partial sums, gemm_splitk_sum), in ranges of at least 1024.
// The same tiles also run FP16 products whose operands are still FP32 in memory (MIX: the
// mixed-precision prefill of few tokens): a lane rounds its fragments to fp16 (nearest even)
// as it reads them from LDS and feeds v_mfma_f32_16x16x32_f16, one per 16 x 16 tile and
// stage, in the k order and ranges of gemm_f16_ws, so the bits are those of rounding the
// operands first.  A weight moves 4 bytes, once, instead of 8 with a casting launch before
// (read 4, write 2, read 2).  The whole op, cast first against this: 8 tokens x 768 19.3 and
// 16.1 us, 8 x 4096 (268 MB of weights) 66 and 47.
// 8 x 768 x 768: 58 -> 7.5 us (24 MFMA stages of one dependent chain per wave); 16 x 14336 x
// 4096 (235 MB of W): 353 -> 36 us, 6.5 TB/s; 16 x 4096 x 14336: 1212 -> 38 us.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "kernels.h"
#include "cdna4.h"
#include "gemm_f32_store.h"
#include "gemm_x3.h"

namespace {

using namespace cdna4;

constexpr int BK = 32;                     // k per stage: 128 bytes of an A row

struct F32Args {
    cf_gemm_args_t g;
    int   tiles_m, tiles_n;
    int   ks, per;                         // ranges of k (blockIdx.y) and their stages
    float* part;
};

// What a product computes in: fp32; or fp16 from fp32 operands, A too or A already fp16.
enum { IN_F32 = 0, MIX_A32 = 1, MIX_A16 = 2 };

// NWN compute waves along N (each BN / NWN columns), 4 / NWN along M.
template <int BM, int BN, int NWN, int MODE = IN_F32>
struct FShape {
    static constexpr int WM = BM * NWN / 4, WN = BN / NWN, MI = WM / 16, NJ = WN / 16;
    static constexpr int A_ST = MODE == MIX_A16 ? BM * BK / 2 : BM * BK;        // floats per stage
    static constexpr int W_ST = BN * BK, ST = A_ST + W_ST;
    static constexpr int AI = A_ST / 256, WI = W_ST / 256;                      // 1 KB instructions
    static constexpr int U = AI + WI, PW = (U + 3) / 4;
    static_assert(MI >= 1 && NJ >= 1 && WM % 16 == 0 && WN % 16 == 0, "wave tile");
};

// W (K, N) rows of BN floats: chunk (16 bytes) c of row k is stored at c ^ kswz(k), which
// spreads the four rows of an MFMA operand read (lanes lq: rows 4 t + lq, 16 floats each)
// over the 64 banks (MIX: the rows of a read are 8 lq + e).
template <int BN, bool MIX = false>
__device__ __forceinline__ int kswz(int k) {
    if (MIX) return BN >= 64 ? 4 * ((k >> 3) & 3) : 4 * ((k >> 3) & 1);
    return BN >= 64 ? 4 * (k & 3) : 4 * ((k >> 1) & 1);
}
__device__ __forceinline__ int rswz(int row) { return (row >> 1) & 7; }

template <int BM, int BN, int NWN, int S, bool WT, int MODE = IN_F32>
__global__ __launch_bounds__(512, 1)
void gemm_f32_ws(F32Args x) {
    using SH = FShape<BM, BN, NWN, MODE>;
    constexpr bool MIX = MODE != IN_F32;
    static_assert(!MIX || !WT, "mixed products: W (K, N)");
    constexpr int MI = SH::MI, NJ = SH::NJ, A_ST = SH::A_ST, ST = SH::ST, U = SH::U, PW = SH::PW;
    extern __shared__ __attribute__((aligned(16))) float smem_f[];
    const cf_gemm_args_t& a = x.g;
    int tm, tn;
    xcd_tile((int)blockIdx.x, x.tiles_m, x.tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN, K = a.K;
    const int kt0 = (int)blockIdx.y * x.per, nk = min(K / BK - kt0, x.per);
    const Segs sg = load_segs(a);
    const int ntot = sg.total;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), cw = wave & 3;

    if (wave >= 4) {
        // Instruction u of a stage: 8 rows x 128 bytes of A (u < AI) or of W (N, K), or 1 KB
        // of W (K, N) rows.  Rows and columns past the end re-read the last ones.
        const char* src[PW];
        uint32_t step[PW];
        int nu = 0;
#pragma unroll
        for (int v = 0; v < PW; v++) {
            const int u = cw + 4 * v;
            nu += u < U ? 1 : 0;
            if (MODE == MIX_A16 && u < SH::AI) {
                // 16 rows x 64 bytes of fp16 A, chunk c of row r at c ^ (r / 4) % 4.
                const int row = 16 * u + (lane >> 2), pc = (lane & 3) ^ ((row >> 2) & 3);
                src[v] = (const char*)((const _Float16*)a.a + (size_t)min(m0 + row, a.M - 1) * K + (size_t)kt0 * BK + 8 * pc);
                step[v] = BK * 2;
            } else if (u < SH::AI || WT) {
                const bool isa = u < SH::AI;
                const int row = 8 * (isa ? u : min(u - SH::AI, SH::WI - 1)) + (lane >> 3), pc = (lane & 7) ^ rswz(row);
                const float* p = isa ? (const float*)a.a + (size_t)min(m0 + row, a.M - 1) * K
                                     : (const float*)a.w[0] + (size_t)min(n0 + row, ntot - 1) * K;
                src[v] = (const char*)(p + (size_t)kt0 * BK + 4 * pc);
                step[v] = BK * 4;
            } else {
                constexpr int CPR = BN / 4;               // chunks per W row
                const int q = 64 * min(u - SH::AI, SH::WI - 1) + lane, k = q / CPR, pc = (q % CPR) ^ kswz<BN, MIX>(k);
                const int c = min(n0 + 4 * pc, ntot - 4);
                const int seg = sg.of(c), N = sg.width(seg);
                src[v] = (const char*)(const float*)(sg.w.at(seg) + (size_t)(kt0 * BK + k) * N + (c - sg.start(seg)));
                step[v] = (uint32_t)N * (BK * 4);
            }
        }
        const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_offset(smem_f) + (uint32_t)cw * 1024u);
        auto issue = [&](int stage) {
            const uint32_t so = lds0 + (uint32_t)stage * (ST * 4u);
#pragma unroll
            for (int v = 0; v < PW; v++)
                if (v < nu) {
                    lds_dma16(src[v], so + 4096u * v);
                    src[v] += step[v];
                }
        };
        auto wait = [&](int ahead) {
            if (nu == PW) wait_ahead<PW, S - 2>(ahead);
            else wait_ahead<PW - 1, S - 2>(ahead);
        };
        for (int s = 0; s < S - 1 && s < nk; s++) issue(s);
        wait(min(S - 2, nk - 1));
        ring_barrier();
        for_each_stage<S>(nk, [&](int kt, auto stage_c) {
            constexpr int stage = decltype(stage_c)::value;
            if (kt + S - 1 < nk) issue((stage + S - 1) % S);
            if (kt + 1 < nk) wait(min(S - 2, nk - 2 - kt));
            ring_barrier();
        });
        return;
    }

    const int wn = SH::WN * (cw % NWN), wm = SH::WM * (cw / NWN);
    f4_t acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[i][j] = f4_t{0.f, 0.f, 0.f, 0.f};
    ring_barrier();
    for_each_stage<S>(nk, [&](int, auto stage_c) {
        constexpr int stage = decltype(stage_c)::value;
        const float* const As = smem_f + stage * ST;
        const float* const Ws = As + A_ST;
        if constexpr (MIX) {
            h8_t af[MI], bf[NJ];
#pragma unroll
            for (int i = 0; i < MI; i++) {
                const int row = wm + 16 * i + lr;
                if constexpr (MODE == MIX_A16) {
                    af[i] = *(const h8_t*)((const _Float16*)As + row * BK + 8 * (lq ^ ((row >> 2) & 3)));
                } else {
                    const f4_t lo = *(const f4_t*)(As + row * BK + 4 * ((2 * lq) ^ rswz(row)));
                    const f4_t hi = *(const f4_t*)(As + row * BK + 4 * ((2 * lq + 1) ^ rswz(row)));
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        af[i][e] = (_Float16)lo[e];
                        af[i][4 + e] = (_Float16)hi[e];
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                const int n = wn + 16 * j + lr;
#pragma unroll
                for (int e = 0; e < 8; e++)
                    bf[j][e] = (_Float16)Ws[(8 * lq + e) * BN + 4 * ((n >> 2) ^ kswz<BN, true>(8 * lq + e)) + (n & 3)];
            }
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < NJ; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bf[j], af[i], acc[i][j], 0, 0, 0);
            ring_barrier();
            return;
        }
#pragma unroll
        for (int t = 0; t < BK / 4; t++) {                 // k = 4 t + lq
            float af[MI], bf[NJ];
#pragma unroll
            for (int i = 0; i < MI; i++) {
                const int row = wm + 16 * i + lr;
                af[i] = As[row * BK + 4 * (t ^ rswz(row)) + lq];
            }
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                const int n = wn + 16 * j + lr, k = 4 * t + lq;
                bf[j] = WT ? Ws[n * BK + 4 * (t ^ rswz(n)) + lq] : Ws[k * BN + 4 * ((n >> 2) ^ kswz<BN>(k)) + (n & 3)];
            }
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < NJ; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bf[j], af[i], acc[i][j], 0, 0, 0);
        }
        ring_barrier();
    });
    if constexpr (MIX) {
        if (x.ks == 1) {
            // Bias and residual rounded to fp16, added in fp32, one rounding of the result:
            // fp16 row-major (or row-concatenated), or widened to fp32 again.
            const CF_GLOBAL float* const res = (const CF_GLOBAL float*)a.residual;
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                const int n = n0 + wn + 16 * j + 4 * lq;
                if (n >= ntot) continue;
                const int seg = sg.of(n);
                const CF_GLOBAL float* bias = sg.bias.at(seg);
                const f4_t b = bias ? *(const CF_GLOBAL f4_t*)(bias + (n - sg.start(seg))) : f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < MI; i++) {
                    const int m = m0 + wm + 16 * i + lr;
                    if (m >= a.M) continue;
                    const f4_t r = res ? *(const CF_GLOBAL f4_t*)(res + (size_t)m * ntot + n) : f4_t{0.f, 0.f, 0.f, 0.f};
                    h4_t o;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        float f = acc[i][j][e] + (float)(_Float16)b[e];
                        if (res) f += (float)(_Float16)r[e];
                        o[e] = (_Float16)f;
                    }
                    if (a.out_f32) *(CF_GLOBAL f4_t*)(sg.out.at(0) + (size_t)m * ntot + n) = __builtin_convertvector(o, f4_t);
                    else *(CF_GLOBAL h4_t*)((CF_GLOBAL _Float16*)sg.out.at(0) + (size_t)m * ntot + n) = o;
                }
            }
            return;
        }
    }
    store_f32_ct<MI, NJ>(a, sg, m0 + wm, n0 + wn, lr, lq, acc,
                         x.ks > 1 ? x.part + (size_t)blockIdx.y * a.M * ntot : nullptr);
}

template <int BM, int BN, int NWN, int S, bool WT, int MODE = IN_F32>
hipError_t launch_f(dim3 grid, hipStream_t st, const F32Args& x) {
    constexpr unsigned lds = (unsigned)S * FShape<BM, BN, NWN, MODE>::ST * 4u;
    static std::atomic<uint64_t> raised{0};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev >= 64 || !((raised.load(std::memory_order_acquire) >> dev) & 1u)) {
        e = hipFuncSetAttribute((const void*)gemm_f32_ws<BM, BN, NWN, S, WT, MODE>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        if (dev < 64) raised.fetch_or(1ull << dev, std::memory_order_release);
    }
    hipLaunchKernelGGL((gemm_f32_ws<BM, BN, NWN, S, WT, MODE>), grid, dim3(512), lds, st, x);
    return hipSuccess;
}

struct F32Candidate {
    int bm, bn, per_cu;        // workgroups whose rings fit one CU
    hipError_t (*launch)(dim3, hipStream_t, const F32Args&);
    hipError_t (*launch_nk)(dim3, hipStream_t, const F32Args&);
};
#define CF_F32_TILE(BM, BN, NWN, S) {BM, BN, 160 * 1024 / (S * FShape<BM, BN, NWN>::ST * 4), launch_f<BM, BN, NWN, S, false>, launch_f<BM, BN, NWN, S, true>}
const F32Candidate kF32Shapes[] = {
    CF_F32_TILE(16, 64, 4, 6), CF_F32_TILE(32, 64, 4, 6), CF_F32_TILE(64, 64, 2, 6),
    CF_F32_TILE(32, 32, 2, 6), CF_F32_TILE(128, 64, 2, 4), CF_F32_TILE(16, 128, 4, 6),
};
#undef CF_F32_TILE
constexpr int kF32Count = (int)(sizeof(kF32Shapes) / sizeof(kF32Shapes[0]));
// Mixed products: rows, columns, and the launches with A in fp32 and in fp16.
struct MixCandidate {
    int bm, bn;
    hipError_t (*a32)(dim3, hipStream_t, const F32Args&);
    hipError_t (*a16)(dim3, hipStream_t, const F32Args&);
};
#define CF_MIX_TILE(BM, BN, NWN, S) \
    {BM, BN, launch_f<BM, BN, NWN, S, false, MIX_A32>, launch_f<BM, BN, NWN, S, false, MIX_A16>}
const MixCandidate kMixShapes[] = {CF_MIX_TILE(32, 32, 2, 8), CF_MIX_TILE(16, 64, 4, 6), CF_MIX_TILE(32, 64, 4, 6),
                                   CF_MIX_TILE(64, 64, 2, 6), CF_MIX_TILE(128, 64, 2, 5)};
#undef CF_MIX_TILE
constexpr int kF32MaxSplit = 16;
int g_mix_bm = 0, g_mix_bn = 0;
int g_f32_bm = 0, g_f32_bn = 0, g_f32_ks = 0, g_f32_mode = 0;

}  // namespace

extern "C" void cf_gemm_set_mix(int32_t bm, int32_t bn) {
    g_mix_bm = bm;
    g_mix_bn = bn;
}

extern "C" void cf_gemm_set_f32(int32_t mode, int32_t bm, int32_t bn, int32_t ks) {
    g_f32_mode = mode;
    g_f32_bm = bm;
    g_f32_bn = bn;
    g_f32_ks = ks;
}

int gemm_f32_ws_pick(const cf_gemm_args_t* a, int* ks_out, float* clk) {
    if (g_f32_mode == 1 || a->elem != CF_ELEM_F32 || a->out_f32) return -1;
    if (a->K % BK != 0 || (uintptr_t)a->a % 16 != 0 || !gemm_w_steps_fit(a)) return -1;
    if (a->w_nk && (a->nseg != 1 || a->out_kind != CF_GEMM_OUT_ROWMAJOR)) return -1;
    if (a->out_kind == CF_GEMM_OUT_QKV && a->d % 4 != 0) return -1;
    uintptr_t al = (uintptr_t)a->residual;
    long long ntot = 0;
    for (int s = 0; s < a->nseg; s++) {
        if (a->n[s] % 4 != 0) return -1;
        ntot += a->n[s];
        al |= (uintptr_t)a->bias[s] | (uintptr_t)a->w[s];
        if (s == 0 || a->out_kind == CF_GEMM_OUT_QKV) al |= (uintptr_t)a->out[s];
    }
    if (al % 16 != 0) return -1;
    const bool may_split = a->out_kind != CF_GEMM_OUT_QKV && (long long)a->M * ntot < (1LL << 30);
    const int cus = cu_count(), nk = a->K / BK;
    const float bytes = ((float)a->M * (float)a->K + (float)a->K * (float)ntot) * 4.0f;
    int best = -1;
    float best_cost = 0.0f;
    *ks_out = 1;
    for (int i = 0; i < kF32Count; i++) {
        const F32Candidate& c = kF32Shapes[i];
        const long long tiles = (a->M + c.bm - 1LL) / c.bm * ((ntot + c.bn - 1) / c.bn);
        if (tiles > 0x7fffffffLL) continue;
        for (int ks = 1; ks <= kF32MaxSplit; ks++) {
            const int per = (nk + ks - 1) / ks;
            if (ks > 1 && (!may_split || tiles * ks > 4LL * cus || per < 1024 / BK)) break;
            if (ks > 1 && (ks - 1) * per >= nk) continue;
            // Per stage: fp32 MFMA at 256 FLOP/clk per CU or the DMA, plus about 250 clk of
            // issue, LDS latency and barrier, which the workgroups sharing a CU hide for
            // one another; the whole at least its bytes from memory.
            const float mfma = (float)(c.bm * c.bn) * (BK * 2.0f / 256.0f);
            const float dma = (float)((c.bm + c.bn) * BK * 4) * (1.0f / 34.0f);
            const float rate = 31.0f * (float)(tiles * ks);
            const float mem = bytes / (rate < 2500.0f ? rate : 2500.0f);
            const int rounds = (int)((tiles * ks + cus - 1) / cus), share = rounds < c.per_cu ? rounds : c.per_cu;
            float t = (float)rounds * (float)per * ((dma > mfma ? dma : mfma) + 250.0f / (float)share);
            t = mem > t ? mem + 0.05f * t : t + 0.05f * mem;
            if (ks > 1) t += 8900.0f + (float)ks * (float)a->M * (float)ntot * (8.0f / 1900.0f);
            if (c.bm == g_f32_bm && c.bn == g_f32_bn && (g_f32_ks == 0 ? ks == 1 : ks == g_f32_ks)) t = -1.0f;
            if (best < 0 || t < best_cost) {
                best = i;
                best_cost = t;
                *ks_out = ks;
            }
        }
    }
    *clk = 1.3f * best_cost;      // measured times are up to a third above the model's
    return best;
}

size_t gemm_f32_ws_floats(const cf_gemm_args_t* a) {
    size_t ntot = 0;
    for (int s = 0; s < a->nseg; s++) ntot += (size_t)a->n[s];
    return a->ksplit > 1 ? (size_t)a->ksplit * (size_t)a->M * ntot : 0;
}

int gemm_f32_ws_launch(const cf_gemm_args_t* a, int pick, hipStream_t st) {
    F32Args x;
    x.g = *a;
    if (!a->partials) x.g.ksplit = 1;
    int ntot = 0;
    for (int s = 0; s < a->nseg; s++) ntot += a->n[s];
    const F32Candidate& c = kF32Shapes[pick];
    x.tiles_m = (a->M + c.bm - 1) / c.bm;
    x.tiles_n = (ntot + c.bn - 1) / c.bn;
    x.ks = x.g.ksplit;
    x.per = (a->K / BK + x.ks - 1) / x.ks;
    x.part = a->partials;
    const dim3 grid((unsigned)((long long)x.tiles_m * x.tiles_n), (unsigned)x.ks);
    hipError_t e = (a->w_nk ? c.launch_nk : c.launch)(grid, st, x);
    if (e == hipSuccess) e = hipGetLastError();
    if (e != hipSuccess || x.ks == 1) return (int)e;
    return gemm_splitk_sum_launch(&x.g, st);
}

int32_t gemm_mix_ok(const cf_gemm_args_t* a) {
    uintptr_t al = (uintptr_t)a->a | (uintptr_t)a->residual | (uintptr_t)a->out[0];
    for (int s = 0; s < a->nseg; s++) {
        if (a->n[s] % 4 != 0) return 0;
        al |= (uintptr_t)a->bias[s] | (uintptr_t)a->w[s];
    }
    return a->K % 64 == 0 && gemm_w_steps_fit(a) && a->out_kind != CF_GEMM_OUT_QKV && al % 16 == 0;
}

int gemm_mix_launch(const cf_gemm_args_t* a, hipStream_t st) {
    if (!gemm_mix_ok(a)) return (int)hipErrorInvalidValue;
    F32Args x;
    x.g = *a;
    x.ks = a->partials && a->ksplit > 1 ? a->ksplit : 1;
    x.g.ksplit = x.ks;
    // The ranges of gemm_f16_ws (whole 64-k stages), so that the sums have its bits.
    x.per = 2 * ((a->K / 64 + x.ks - 1) / x.ks);
    x.part = a->partials;
    int ntot = 0;
    for (int s = 0; s < a->nseg; s++) ntot += a->n[s];
    // Per stage the DMA of (BM + BN) x 128 bytes, at least 300 clk, times the rounds of tiles;
    // 32 columns spread a small weight over more CUs (2304 columns in 64s reach 36).
    const int cus = cu_count();
    const MixCandidate* c = nullptr;
    float best = 0.0f;
    for (const MixCandidate& k : kMixShapes) {
        const long long tiles = (a->M + k.bm - 1LL) / k.bm * ((ntot + k.bn - 1) / k.bn) * x.ks;
        const float dma = (float)((k.bm + k.bn) * BK * 4) * (1.0f / 34.0f);
        const float hbm = (float)a->K * (float)ntot * 4.0f / (31.0f * (float)(tiles < cus ? tiles : cus));
        float t = (float)((tiles + cus - 1) / cus) * (float)x.per * (dma > 300.0f ? dma : 300.0f);
        t = hbm > t ? hbm + 0.05f * t : t + 0.05f * hbm;
        if (g_mix_bm ? k.bm == g_mix_bm && k.bn == g_mix_bn : !c || t < best) {
            c = &k;
            best = t;
        }
    }
    if (!c) c = &kMixShapes[0];
    x.tiles_m = (a->M + c->bm - 1) / c->bm;
    x.tiles_n = (ntot + c->bn - 1) / c->bn;
    const dim3 grid((unsigned)((long long)x.tiles_m * x.tiles_n), (unsigned)x.ks);
    hipError_t e = (a->mix == CF_GEMM_MIX_A32 ? c->a32 : c->a16)(grid, st, x);
    if (e == hipSuccess) e = hipGetLastError();
    if (e != hipSuccess || x.ks == 1) return (int)e;
    return gemm_splitk_sum_launch(&x.g, st);
}
