/*
 * adjoint.hip -- the per-sample AMICA log-likelihood and its adjoint
 * (include/amica_adjoint.h).
 *
 * The forward terms are the reference's E-step quantities
 * (fraimondo/cudamica src/kernels.cu:251-450: y, the generalized-Gaussian
 * log density Q, the log-sum-exp over components and over models).  The
 * adjoint weights each sample's model posterior v_ht by the upstream
 * gradient dll_t and re-evaluates the responsibilities u = dll v z (nothing
 * is stored between the passes); the gradients are then the reference's
 * sufficient statistics of those weighted responsibilities:
 *   dalpha = sum u / alpha                  dmu  = sum sqrt(beta) u f
 *   dbeta  = sum u (1 - f y) / (2 beta)     drho = sum u (psi(1+1/rho)/rho^2 - |y|^rho ln|y|)
 *   dgm    = sum dll v / gm                 g    = sum_j sqrt(beta) u f   (per sample)
 *   dW_h   = (sum_t dll v_h) W_h^-T - sum_t g_t (x_t - c_h)^T
 *   dc_h   = W_h^T sum_t g_t
 * with f = rho sign(y)|y|^(rho-1).
 *
 * Kernels: the inverse and log|det W| (the M-step's Gauss-Jordan), prep (W c,
 * the constant part of Q, GEMM operands), then per chunk of samples the
 * unmixing GEMM b = W x - W c on MFMA (the engine's FP64 or plain FP32
 * kernels, into a [T][M NP] buffer), ll (one wave per (model, 64-channel
 * block) over a range of samples, all M ceil(n/64) waves in one workgroup
 * where they fit in 8, else three passes through per-sample buffers; the
 * allocation-free forward instead forms b there, 16 samples at a time on
 * MFMA), gx (sum_t g_t x_t^T on FP32 or FP64 MFMA over sample chunks) and the
 * sums of their partials onto the chunks' running totals, from which finish
 * assembles the gradients.
 * Every reduction is in a fixed order, so results repeat bit for bit.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <string>
#include <vector>

#include "../../../include/amica_adjoint.h"
#include "../../../include/amica_engine.h"
#include "common.h"
#include "engine_internal.h"
#include "linalg_dev.h"

namespace amica {

namespace {

struct AdjArgs {
    const void* x;
    long T;
    int n, NP, M, m;
    const double *W, *c, *alpha, *mu, *beta, *rho, *gm;
    double ldetS;
    const double* dll;   /* null: forward only */
    double* ll;          /* [T] or null */
    /* workspace */
    double* Winv;        /* [M][n][n] column-major */
    double* ldet;        /* [M] -log|det W_h| */
    double* cq;          /* [M][m][n] log alpha + .5 log beta - log2 - lgamma(1+1/rho) */
    double* wc;          /* [M][NP] W_h c_h */
    void* g;             /* [T][M NP] (adjoint) */
    double* part;        /* [nblocks][pstride] */
    long chunk;          /* samples per workgroup, a multiple of 4 */
    size_t pstride;
    /* split passes (M ceil(n/64) > 8 waves): workgroups of pg (model,
     * channel-block) pairs, blockIdx.y = pair group; qbuf [T][M CW] the
     * pairs' channel sums of q, vbuf [T][M] dll_t v_ht */
    double* qbuf;
    double* vbuf;
    int pg;
    /* b = W x - W c from the unmixing GEMM, [T][M NP] Real (BSRC 0) */
    const void* bbuf;
};

/* kLlFused: a workgroup holds all M ceil(n/64) (model, channel-block) pairs of
 * a sample range and exchanges the channel sums in LDS.  kLlM1: one model,
 * whose posterior is 1 (the exchange serves ll alone).  Where the pairs do not
 * fit one workgroup the same body runs in three passes: kLlQ writes each
 * pair's channel sum of q per sample (qbuf), ll_post_kernel forms L_h, ll_t and
 * dll_t v_ht (vbuf), and kLlGrad re-evaluates the densities and accumulates
 * the gradients. */
enum { kLlFused = 0, kLlQ = 1, kLlGrad = 2, kLlM1 = 3 };

/* raw sums per pair (h, i): su_j, su|y|^(rho-1)sgn_j, su|y|^rho_j,
 * su|y|^rho log|y|_j (j < m), gsum; then Omega_h */
__host__ __device__ inline int pair_stride(int m) { return 4 * m + 1; }

/* What every sample needs of the model: W c, the constant part of Q, and
 * (Wg not null) the unmixing GEMM's operands Wg[h NP + i][k] = W_h[i][k] (zero
 * past n) and W c in its precision.  Grid (eb + NP / 4, M): workgroups below
 * eb take the elementwise parts, the others four rows of W c, one per wave. */
template <typename Real>
__global__ __launch_bounds__(256) void adj_prep_kernel(AdjArgs a, int eb, Real* __restrict__ Wg,
                                                       Real* __restrict__ wcr) {
    const int h = blockIdx.y, n = a.n, m = a.m, NP = a.NP;
    const double* W = a.W + (size_t)h * n * n;
    if ((int)blockIdx.x >= eb) {
        const int lane = threadIdx.x & 63, i = ((int)blockIdx.x - eb) * 4 + ((int)threadIdx.x >> 6);
        if (i >= NP) return;
        const double* c = a.c + (size_t)h * n;
        double s = 0.0;
        if (i < n)
            for (int k = lane; k < n; k += 64) s += W[i + (size_t)k * n] * c[k];
        s = wave_sum_f64(s);
        if (lane == 0) {
            a.wc[(size_t)h * NP + i] = s;
            if (Wg) wcr[(size_t)h * NP + i] = (Real)s;
        }
        return;
    }
    const int nm = n * m, total = Wg ? NP * NP : 0;
    for (int q = (int)blockIdx.x * 256 + threadIdx.x; q < max(nm, total); q += eb * 256) {
        if (q < nm) {
            const size_t e = (size_t)h * nm + q;
            a.cq[e] = log(a.alpha[e]) + 0.5 * log(a.beta[e]) - AMICA_LOG2_REF - lgamma(1.0 + 1.0 / a.rho[e]);
        }
        if (q < total) {
            /* rows along the threads: the column-major W is read in order */
            const int i = q % NP, k = q / NP;
            Wg[((size_t)h * NP + i) * NP + k] = (i < n && k < n) ? (Real)W[(size_t)k * n + i] : (Real)0;
        }
    }
}

/* Base-2 logarithm and exponential on the FP32 variant (v_log_f32, v_exp_f32;
 * arguments here are normal or underflow to 0), natural ones in FP64: kLn is
 * the logarithm of the variant's base, kUnit its reciprocal. */
template <typename Real> struct Base;
template <> struct Base<float> {
    static constexpr double kLn = 0.6931471805599453, kUnit = 1.4426950408889634;
    static constexpr float kTiny = 1.17549435e-38f;
    static __device__ __forceinline__ float log(float v) { return __builtin_amdgcn_logf(v); }
    static __device__ __forceinline__ float exp(float v) { return __builtin_amdgcn_exp2f(v); }
    static __device__ __forceinline__ float rcp(float v) { return __builtin_amdgcn_rcpf(v); }
};
template <> struct Base<double> {
    static constexpr double kLn = 1.0, kUnit = 1.0;
    static constexpr double kTiny = 2.2250738585072014e-308;
    static __device__ __forceinline__ double log(double v) { return ::log(v); }
    static __device__ __forceinline__ double exp(double v) { return ::exp(v); }
    static __device__ __forceinline__ double rcp(double v) { return 1.0 / v; }
};

/* Samples per tile, held in registers between the densities and the gradient
 * sums (4 values per component and sample on the adjoint), about what 256 VGPRs
 * hold.  The adjoint goes past them into scratch memory in FP64 at m = 3, 5, 7
 * and 8 (several models: 84 to 216 bytes a lane; one: 52 and 60 at m = 5 and 8)
 * and in FP32 at m = 5, 7 and 8 (56 to 196; one: 92 at m = 8, where the split
 * pass takes 20).  In FP32 at m = 3, which fits, tiles of two took 14.9 ms a call
 * where these take 13.4 (128 ch x 2M x 4 models); smaller tiles where it spills
 * have not been timed. */
template <typename Real, int MJ, bool ADJ> constexpr int tile_samples() {
    return sizeof(Real) == 4 ? (MJ <= 5 || !ADJ ? 4 : 2) : (!ADJ || MJ <= 3 ? 4 : MJ <= 5 ? 2 : 1);
}

/* 64-bit value of the lane a row rotation by R brings in (rows of 16) */
template <int R> __device__ __forceinline__ double row_ror(double v) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const int lo = __builtin_amdgcn_mov_dpp((int)(uint32_t)u, 0x120 + R, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_mov_dpp((int)(uint32_t)(u >> 32), 0x120 + R, 0xf, 0xf, false);
    return __builtin_bit_cast(double, ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}

__device__ __forceinline__ double row_sum(double v) {
    v += row_ror<8>(v);
    v += row_ror<4>(v);
    v += row_ror<2>(v);
    return v + row_ror<1>(v);
}

__device__ __forceinline__ double row_max(double v) {
    v = fmax(v, row_ror<8>(v));
    v = fmax(v, row_ror<4>(v));
    v = fmax(v, row_ror<2>(v));
    return fmax(v, row_ror<1>(v));
}

/* Two values folded onto each other across the halves (H 32) or the row pairs
 * (H 16) of the wave: swapping a's odd halves (rows) with b's even ones and
 * adding leaves a's pair sums in the even ones, b's in the odd ones. */
template <int H> __device__ __forceinline__ double fold(double a, double b) {
    const uint64_t ua = __builtin_bit_cast(uint64_t, a), ub = __builtin_bit_cast(uint64_t, b);
    auto swap = [](uint32_t p, uint32_t q) {
        if constexpr (H == 32) return __builtin_amdgcn_permlane32_swap(p, q, false, false);
        else return __builtin_amdgcn_permlane16_swap(p, q, false, false);
    };
    const auto lo = swap((uint32_t)ua, (uint32_t)ub), hi = swap((uint32_t)(ua >> 32), (uint32_t)(ub >> 32));
    return __builtin_bit_cast(double, ((uint64_t)hi[0] << 32) | lo[0]) +
           __builtin_bit_cast(double, ((uint64_t)hi[1] << 32) | lo[1]);
}

/* Wave sums of S samples' values at once: every lane of row r ends with the
 * total of sample sample_of_row(r). */
template <int S> __device__ __forceinline__ double wave_totals(const double (&q)[S]) {
    double v;
    if constexpr (S == 4) v = fold<16>(fold<32>(q[0], q[1]), fold<32>(q[2], q[3]));
    else if constexpr (S == 2) { v = fold<32>(q[0], q[1]); v = fold<16>(v, v); }
    else { v = fold<32>(q[0], q[0]); v = fold<16>(v, v); }
    return row_sum(v);
}

template <int S> __device__ __forceinline__ int sample_of_row(int r) {
    return S == 4 ? ((r & 1) << 1) | (r >> 1) : S == 2 ? r >> 1 : 0;
}

__device__ __forceinline__ double readlane_f64(double v, int l) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), l);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

/* 16 samples x this wave's 64 channels of W_h x by MFMA into the wave's LDS
 * tile [16][64]: x rows and W straight from global memory as fragments
 * (element (l % 16, l / 16) per lane), rows past T and inputs past n as
 * zeros. */
template <typename Real>
__device__ __forceinline__ void unmix_tile(const AdjArgs& a, const double* __restrict__ Wh, int ch0, long t0,
                                           Real* __restrict__ tile) {
    const int lane = threadIdx.x & 63, l15 = lane & 15, kq = lane >> 4, n = a.n;
    const Real* xr = (const Real*)a.x + (size_t)min(t0 + l15, a.T - 1) * n;
    const bool row = t0 + l15 < a.T;
    typedef Real R4 __attribute__((ext_vector_type(4)));
    R4 acc[4];
    const double* wp[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        acc[q] = (R4){(Real)0, (Real)0, (Real)0, (Real)0};
        wp[q] = Wh + min(ch0 + 16 * q + l15, n - 1);       /* columns past n are not used */
    }
#pragma unroll 4
    for (int k0 = 0; k0 < n; k0 += 4) {
        const int k = min(k0 + kq, n - 1);
        const Real xv = xr[k];
        const Real av = row && k0 + kq < n ? xv : (Real)0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            /* a repeated W entry meets a zero; one that is not finite is met
             * at its own k as well */
            const Real wv = (Real)wp[q][(size_t)k * n];
            if constexpr (sizeof(Real) == 4) acc[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, wv, acc[q], 0, 0, 0);
            else acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, wv, acc[q], 0, 0, 0);
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            tile[(sizeof(Real) == 4 ? 4 * kq + r : kq + 4 * r) * 64 + 16 * q + l15] = acc[q][r];
}

/* One wave per (model, 64-channel block), lane = channel, over a range of
 * samples in tiles of S.  Per component and sample, with la = log|y| in the
 * variant's base: p = |y|^(rho-1), |y|^rho = p |y|, Q = cq - |y|^rho; the
 * score is rho p sgn(y).  A tile's S channel sums of q reduce together
 * (wave_totals) and cross the waves through one double-buffered LDS slot and
 * one barrier, after which every wave evaluates the model posteriors of the
 * tile for itself (row = sample, lane in row = model): no second barrier, and
 * the tile's densities stay in registers for the gradient sums.  Those are
 * FP64 throughout; the factors rho, sqrt(beta), psi are applied to the totals.
 * The next tile's b (and dll) are loaded before a tile's arithmetic.  Bound by
 * VALU issue (three transcendentals and, on the adjoint, 12 FP64 operations
 * and conversions per component). */
template <typename Real, int MJ, bool ADJ, int MODE, int BSRC>
__global__ __launch_bounds__(512) void ll_kernel(AdjArgs a) {
    constexpr int S = tile_samples<Real, MJ, ADJ>();
    using B = Base<Real>;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int n = a.n, NP = a.NP, M = a.M;
    const int tid = threadIdx.x, lane = tid & 63, nw = blockDim.x >> 6;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int CW = NP / 64;
    int pair = wv;
    if constexpr (MODE == kLlQ || MODE == kLlGrad) {
        pair = (int)blockIdx.y * a.pg + wv;
        if (pair >= M * CW) return;                  /* no barriers in these modes */
    }
    const int h = pair / CW;
    const int i = (pair - h * CW) * 64 + lane;
    const bool act = i < n;
    /* LDS: qp[2][S][nw] (double), and with BSRC 1 a [16][64] tile per wave */
    double* qp = (double*)smem_raw;
    Real* tile = (Real*)(qp + 2 * S * nw) + wv * 1024;

    Real sb[MJ], mu[MJ], rm1[MJ], cq[MJ];
    double sbr[ADJ ? MJ : 1];
#pragma unroll
    for (int j = 0; j < MJ; ++j) {
        const size_t e = ((size_t)h * MJ + j) * n + (act ? i : 0);
        const double be = a.beta[e], rh = a.rho[e];
        sb[j] = (Real)sqrt(be);
        mu[j] = (Real)a.mu[e];
        rm1[j] = (Real)(rh - 1.0);
        cq[j] = (Real)(a.cq[e] * B::kUnit);
        if constexpr (ADJ) sbr[j] = sqrt(be) * rh;
    }
    const Real wci = BSRC ? (Real)a.wc[(size_t)h * NP + i] : (Real)0;
    /* lane (row, hh): the constant of model hh */
    const int hh = lane & 15, row = lane >> 4;
    double lc = -HUGE_VAL;
    if constexpr (MODE == kLlFused || MODE == kLlM1)
        if (hh < M) lc = log(a.gm[hh]) - a.ldet[hh] + a.ldetS;
    double su[ADJ ? MJ : 1], sup[ADJ ? MJ : 1], suy[ADJ ? MJ : 1], sul[ADJ ? MJ : 1];
    double gsum = 0.0, om = 0.0;
#pragma unroll
    for (int j = 0; j < (ADJ ? MJ : 1); ++j) su[j] = sup[j] = suy[j] = sul[j] = 0.0;

    const long t0 = (long)blockIdx.x * a.chunk;
    const long t1 = min(a.T, t0 + a.chunk);
    const size_t ldb = (size_t)M * NP;
    const Real* const bb = (const Real*)a.bbuf + (size_t)h * NP + i;
    Real bn[S];
    double dn[ADJ ? S : 1];
    auto load = [&](long tb) {
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const long t = min(tb + s, t1 - 1);      /* past the range: the last sample again, weight 0 */
            if constexpr (BSRC == 0) bn[s] = bb[(size_t)t * ldb];
            if constexpr (ADJ && MODE == kLlGrad) dn[s] = a.vbuf[(size_t)t * M + h];
            if constexpr (ADJ && MODE == kLlM1) dn[s] = a.dll[t];
        }
        if constexpr (ADJ && MODE == kLlFused) dn[0] = a.dll[min(tb + min(row, S - 1), t1 - 1)];
    };
    load(t0);
    int buf = 0;
    for (long tb = t0; tb < t1; tb += S) {
        Real bv[S];
        double dv[ADJ ? S : 1];
        if constexpr (BSRC == 1) {
            if (((tb - t0) & 15) == 0) {
                unmix_tile<Real>(a, a.W + (size_t)h * n * n, (pair - h * CW) * 64, tb, tile);
                __builtin_amdgcn_wave_barrier();
            }
#pragma unroll
            for (int s = 0; s < S; ++s) bv[s] = tile[(((tb - t0) & 15) + s) * 64 + lane] - wci;
            __builtin_amdgcn_wave_barrier();
        } else {
#pragma unroll
            for (int s = 0; s < S; ++s) bv[s] = bn[s];
        }
        if constexpr (ADJ) {
#pragma unroll
            for (int s = 0; s < S; ++s) dv[s] = dn[s];
        }
        load(tb + S);
        /* densities */
        Real ez[S][MJ], ps[S][MJ], yr[S][MJ], la[S][MJ], rse[S];
        double q[S];
#pragma unroll
        for (int s = 0; s < S; ++s) {
            Real Qj[MJ], mx = (Real)0, se = (Real)0;
#pragma unroll
            for (int j = 0; j < MJ; ++j) {
                const Real y = sb[j] * (bv[s] - mu[j]);
                const Real ay = fmax(fabs(y), B::kTiny);
                la[s][j] = B::log(ay);
                const Real p = B::exp(rm1[j] * la[s][j]);         /* |y|^(rho-1) */
                yr[s][j] = p * fabs(y);       /* not ay, which is kTiny for a NaN */
                if constexpr (ADJ) ps[s][j] = y > (Real)0 ? p : y < (Real)0 ? -p : y;   /* 0 at 0, NaN stays */
                Qj[j] = fma(yr[s][j], (Real)-B::kUnit, cq[j]);
                mx = (j == 0) ? Qj[j] : fmax(mx, Qj[j]);
            }
#pragma unroll
            for (int j = 0; j < MJ; ++j) {
                ez[s][j] = B::exp(Qj[j] - mx);
                se += ez[s][j];
            }
            if constexpr (ADJ) rse[s] = B::rcp(se);
            if constexpr (MODE != kLlGrad) q[s] = act ? (double)mx + (double)B::log(se) : 0.0;
        }
        /* channel sums, and per sample the models' log-sum-exp */
        double w = 0.0;                              /* lane (row, hh): dll v of sample row, model hh */
        if constexpr (MODE != kLlGrad) {
            const double tot = wave_totals<S>(q) * B::kLn;
            const int ts = sample_of_row<S>(row);
            if constexpr (MODE == kLlQ) {
                if (hh == 0 && tb + ts < t1) a.qbuf[(size_t)(tb + ts) * M * CW + pair] = tot;
            } else {
                if (hh == 0) qp[(buf * S + ts) * nw + wv] = tot;
                __syncthreads();
                if (MODE == kLlFused || wv == 0) {
                    const int sr = min(row, S - 1);
                    double L = lc;
                    if (hh < M)
                        for (int c = 0; c < CW; ++c) L += qp[(buf * S + sr) * nw + hh * CW + c];
                    const bool out = a.ll && wv == 0 && hh == 0 && row < S && tb + row < t1;
                    if constexpr (MODE == kLlM1) {
                        if (out) a.ll[tb + row] = L;
                    } else {
                        const double mx = row_max(L);
                        const double e = exp(L - mx), se = row_sum(e);
                        if (ADJ) w = tb + row < t1 ? dv[0] * (e / se) : 0.0;
                        if (wv == 0) {
                            const double P = mx + log(se);
                            if (out) a.ll[tb + row] = P;
                        }
                    }
                }
                buf ^= 1;
            }
        }
        if constexpr (ADJ) {
            Real* g = (Real*)a.g + (size_t)h * NP + i;
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const bool in = tb + s < t1;         /* uniform */
                double omh;
                if constexpr (MODE == kLlFused) omh = readlane_f64(w, 16 * s + h);
                else omh = in ? dv[s] : 0.0;
                double gv = 0.0;
#pragma unroll
                for (int j = 0; j < MJ; ++j) {
                    const double u = omh * (double)(ez[s][j] * rse[s]);
                    const double up = u * (double)ps[s][j], uy = u * (double)yr[s][j];
                    su[j] += u;
                    sup[j] += up;
                    suy[j] += uy;
                    sul[j] = fma(uy, (double)la[s][j], sul[j]);
                    gv = fma(sbr[j], up, gv);
                }
                if (!act) gv = 0.0;
                if (in) g[(size_t)(tb + s) * ldb] = (Real)gv;
                gsum += gv;
                om += omh;
            }
        }
    }
    if constexpr (ADJ && MODE != kLlQ) {
        double* base = a.part + (size_t)blockIdx.x * a.pstride;
        double* pp = base + ((size_t)h * NP + i) * pair_stride(MJ);
#pragma unroll
        for (int j = 0; j < MJ; ++j) {
            pp[j] = su[j];
            pp[MJ + j] = sup[j];
            pp[2 * MJ + j] = suy[j];
            pp[3 * MJ + j] = sul[j] * B::kLn;
        }
        pp[4 * MJ] = gsum;
        if (i == 0) base[(size_t)M * NP * pair_stride(MJ) + h] = om;
    }
}

/* The split passes' middle step, one thread per sample: L_h = log gm_h +
 * log|det W_h| + ldetS + the pairs' sums of q, ll_t = logsumexp_h L_h and
 * (adjoint) dll_t v_ht. */
__global__ __launch_bounds__(256) void ll_post_kernel(AdjArgs a) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= a.T) return;
    const int M = a.M, CW = a.NP / 64;
    const double* q = a.qbuf + (size_t)t * M * CW;
    auto model = [&](int hh) {
        double L = log(a.gm[hh]) - a.ldet[hh] + a.ldetS;
        for (int c = 0; c < CW; ++c) L += q[hh * CW + c];
        return L;
    };
    double mx = -HUGE_VAL;
    for (int hh = 0; hh < M; ++hh) mx = fmax(mx, model(hh));
    double se = 0.0;
    for (int hh = 0; hh < M; ++hh) se += exp(model(hh) - mx);
    const double P = mx + log(se);
    if (a.ll) a.ll[t] = P;
    if (a.dll) {
        const double w = a.dll[t];
        for (int hh = 0; hh < M; ++hh) a.vbuf[(size_t)t * M + hh] = w * exp(model(hh) - P);
    }
}

/* FP64 statistic GEMM part[chunk][r][k] = sum_{t in chunk} g[t][r] x[t][k]
 * (r < ldg, k < n) on the FP64 MFMA units: 64 x 64 per workgroup, whose four
 * waves take every fourth group of two 4-sample steps and add their tiles
 * through LDS in wave order; fragments come straight from memory, a group
 * ahead. */
__global__ __launch_bounds__(256, 2) void adj_gx_kernel(const double* __restrict__ g,
                                                        const double* __restrict__ x, long T, int n, int ldg,
                                                        long chunk, double* __restrict__ part) {
    constexpr int kU = 2;
    __shared__ double sum[16][256];
    const int tid = threadIdx.x, lane = tid & 63, l15 = lane & 15, kq = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rb = blockIdx.y * 64, kb = blockIdx.z * 64;
    const long ts = (long)blockIdx.x * chunk, te = min(T, ts + chunk);
    int ck[4];
    bool vk[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int k = kb + 16 * q + l15;
        vk[q] = k < n;
        ck[q] = vk[q] ? k : n - 1;
    }
    f64x4 acc[4][4];
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[p][q] = (f64x4){0.0, 0.0, 0.0, 0.0};
    double fa[kU][4], fb[kU][4];
    auto load = [&](long t0) {
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const long t = t0 + 4 * u + kq, tc = t < te ? t : te - 1;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                fa[u][p] = g[(size_t)tc * ldg + rb + 16 * p + l15];
                fb[u][p] = x[(size_t)tc * n + ck[p]];
            }
        }
    };
    const long step = 4 * 4 * kU;
    long t0 = ts + (long)w * 4 * kU;
    if (t0 < te) load(t0);
    for (; t0 < te; t0 += step) {
        double av[kU][4], bv[kU][4];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const bool ok = t0 + 4 * u + kq < te;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                av[u][p] = ok ? fa[u][p] : 0.0;
                bv[u][p] = ok && vk[p] ? fb[u][p] : 0.0;
            }
        }
        if (t0 + step < te) load(t0 + step);
#pragma unroll
        for (int u = 0; u < kU; ++u)
#pragma unroll
            for (int p = 0; p < 4; ++p)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    acc[p][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[u][p], bv[u][q], acc[p][q], 0, 0, 0);
    }
    for (int v = 0; v < 4; ++v) {
        if (v == w) {
#pragma unroll
            for (int p = 0; p < 4; ++p)
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        double* s = &sum[p * 4 + q][(kq + 4 * r) * 16 + l15];
                        *s = v == 0 ? acc[p][q][r] : *s + acc[p][q][r];
                    }
        }
        __syncthreads();
    }
    double* out = part + (size_t)blockIdx.x * ldg * n;
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        const int r = rb + (t >> 2) * 16 + (tid >> 4), k = kb + (t & 3) * 16 + (tid & 15);
        if (k < n) out[(size_t)r * n + k] = sum[t][tid];
    }
}

/* x [T][n] into [T][NP] with zero columns past n (the GEMMs' row layout) */
template <typename Real>
__global__ __launch_bounds__(256) void adj_pad_kernel(const Real* __restrict__ x, Real* __restrict__ xp,
                                                      long T, int n, int NP) {
    const long total = T * NP;
    for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < total; q += (long)gridDim.x * blockDim.x) {
        const long t = q / NP;
        const int k = (int)(q - t * NP);
        xp[q] = k < n ? x[(size_t)t * n + k] : (Real)0;
    }
}

struct AdjOut {
    double *dW, *dc, *dalpha, *dmu, *dbeta, *drho, *dgm;
};

/* The gradients from the totals of the raw sums (raw) and of sum_t g_t x_t^T (G,
 * rows of gxs).  Grid (eb + n / 4, M): workgroups below eb take dW and the
 * densities' gradients, the others four entries of dc, one per wave. */
__global__ __launch_bounds__(256) void adj_finish_kernel(AdjArgs a, int eb, const double* __restrict__ raw,
                                                         const double* __restrict__ G, int gxs, AdjOut o) {
    const int h = blockIdx.y, n = a.n, m = a.m, NP = a.NP, ps = pair_stride(m);
    const int nm = n * m, nn = n * n;
    const size_t ldg = (size_t)a.M * NP;
    auto gsum = [&](int i) { return raw[((size_t)h * NP + i) * ps + 4 * m]; };
    const double* W = a.W + (size_t)h * nn;
    if ((int)blockIdx.x >= eb) {
        const int lane = threadIdx.x & 63, k = ((int)blockIdx.x - eb) * 4 + ((int)threadIdx.x >> 6);
        if (k >= n) return;
        double s = 0.0;
        for (int i = lane; i < n; i += 64) s += W[i + (size_t)k * n] * gsum(i);
        s = wave_sum_f64(s);
        if (lane == 0) o.dc[(size_t)h * n + k] = s;
        return;
    }
    const double om = raw[ldg * ps + h];
    for (int q = (int)blockIdx.x * 256 + threadIdx.x; q < nn + nm; q += eb * 256) {
        if (q >= nn) {
            const int e0 = q - nn, j = e0 / n, i = e0 - j * n;
            const size_t e = (size_t)h * nm + e0, off = ((size_t)h * NP + i) * ps + j;
            const double be = a.beta[e], rh = a.rho[e];
            const double su = raw[off], sup = raw[off + m], suy = raw[off + 2 * m], sul = raw[off + 3 * m];
            o.dalpha[e] = su / a.alpha[e];
            o.dmu[e] = sqrt(be) * rh * sup;
            o.dbeta[e] = (su - rh * suy) / (2.0 * be);
            o.drho[e] = su * psi_dev(1.0 + 1.0 / rh) / (rh * rh) - sul;
        } else {
            const int i = q % n, k = q / n;
            o.dW[(size_t)h * nn + q] = om * a.Winv[(size_t)h * nn + k + (size_t)i * n] -
                                       (G[((size_t)h * NP + i) * gxs + k] - gsum(i) * a.c[(size_t)h * n + k]);
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) o.dgm[h] = om / a.gm[h];
}

template <typename Real, bool ADJ, int MODE, int BSRC>
int launch_ll_mode(int MJ, const AdjArgs& a, dim3 grid, dim3 block, hipStream_t st) {
    const size_t nw = block.x / 64;
    const size_t shm = 2 * 4 * nw * 8 + (BSRC ? nw * 1024 * sizeof(Real) : 0);
#define AMICA_LL_CASE(J)                                                                           \
    case J:                                                                                        \
        if (shm > 65536 &&                                                                         \
            hipFuncSetAttribute((const void*)ll_kernel<Real, J, ADJ, MODE, BSRC>,                  \
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm) != hipSuccess) \
            return -1;                                                                             \
        hipLaunchKernelGGL((ll_kernel<Real, J, ADJ, MODE, BSRC>), grid, block, shm, st, a);        \
        break;
    switch (MJ) {
        AMICA_LL_CASE(1)
        AMICA_LL_CASE(2)
        AMICA_LL_CASE(3)
        AMICA_LL_CASE(4)
        AMICA_LL_CASE(5)
        AMICA_LL_CASE(6)
        AMICA_LL_CASE(7)
        AMICA_LL_CASE(8)
        default: return -1;
    }
#undef AMICA_LL_CASE
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <typename Real, bool ADJ>
int launch_ll(int MJ, const AdjArgs& a, int nblocks, hipStream_t st) {
    const int pairs = a.M * (a.NP / 64);
    if (!a.qbuf) {
        const dim3 grid(nblocks), block(64 * pairs);
        if constexpr (!ADJ)
            if (!a.bbuf)
                return a.M == 1 ? launch_ll_mode<Real, ADJ, kLlM1, 1>(MJ, a, grid, block, st)
                                : launch_ll_mode<Real, ADJ, kLlFused, 1>(MJ, a, grid, block, st);
        return a.M == 1 ? launch_ll_mode<Real, ADJ, kLlM1, 0>(MJ, a, grid, block, st)
                        : launch_ll_mode<Real, ADJ, kLlFused, 0>(MJ, a, grid, block, st);
    }
    const dim3 grid(nblocks, (pairs + a.pg - 1) / a.pg), block(64 * a.pg);
    if (launch_ll_mode<Real, false, kLlQ, 0>(MJ, a, grid, block, st)) return -1;
    hipLaunchKernelGGL(ll_post_kernel, dim3((unsigned)((a.T + 255) / 256)), dim3(256), 0, st, a);
    if (hipGetLastError() != hipSuccess) return -1;
    return ADJ ? launch_ll_mode<Real, true, kLlGrad, 0>(MJ, a, grid, block, st) : 0;
}

/* One block of device memory per call, from a pool that outlives it: hipMalloc
 * and hipFree of a call's buffers took longer than its kernels (up to 30 ms for
 * a gigabyte).  A call owns its block until its stream has drained (the
 * destructor waits where the call did not), so blocks in the pool are idle and
 * any thread and stream may take one.  At most kPoolBlocks stay per device, of
 * kPoolBytes in all; the rest goes back to the device, and every idle block on
 * request (amica_ll_release_workspace) and where an allocation of this library
 * fails (device_malloc). */
constexpr size_t kPoolBytes = (size_t)1 << 30;
constexpr int kPoolBlocks = 2;

struct PoolBlock {
    int dev;
    void* p;
    size_t bytes;
};
std::mutex g_pool_mu;
std::vector<PoolBlock> g_pool;

/* frees the idle blocks of device dev (-1: of all) */
hipError_t release_pool(int dev) {
    hipError_t first = hipSuccess;
    for (;;) {
        void* p = nullptr;
        {
            std::lock_guard<std::mutex> lock(g_pool_mu);
            for (size_t k = 0; k < g_pool.size() && !p; ++k) {
                if (dev >= 0 && g_pool[k].dev != dev) continue;
                p = g_pool[k].p;
                g_pool.erase(g_pool.begin() + k);
            }
        }
        if (!p) return first;
        const hipError_t e = hipFree(p);
        if (first == hipSuccess) first = e;
    }
}

class Workspace {
public:
    Workspace(int dev, hipStream_t st) : dev_(dev), st_(st) {}
    Workspace(const Workspace&) = delete;
    Workspace& operator=(const Workspace&) = delete;
    ~Workspace() {
        if (!b_.p) return;
        if (!drained_ && hipStreamSynchronize(st_) != hipSuccess) {
            /* the stream's work may still run: not for another call (hipFree waits
             * for the device) */
            (void)hipFree(b_.p);
            return;
        }
        /* at most one block more than the pool keeps per device leaves at a time */
        void* drop[kPoolBlocks + 2];
        int nd = 0;
        {
            std::lock_guard<std::mutex> lock(g_pool_mu);
            try {
                g_pool.push_back(b_);
            } catch (...) {                 /* no host memory to remember it in */
                drop[nd++] = b_.p;
            }
            /* the smallest blocks leave first */
            for (;;) {
                size_t sum = 0, least = 0;
                int cnt = 0;
                for (size_t k = 0; k < g_pool.size(); ++k) {
                    if (g_pool[k].dev != dev_) continue;
                    if (!cnt || g_pool[k].bytes < g_pool[least].bytes) least = k;
                    sum += g_pool[k].bytes;
                    ++cnt;
                }
                if ((cnt <= kPoolBlocks && sum <= kPoolBytes) || nd == kPoolBlocks + 2) break;
                drop[nd++] = g_pool[least].p;
                g_pool.erase(g_pool.begin() + least);
            }
        }
        for (int k = 0; k < nd; ++k) (void)hipFree(drop[k]);
    }
    /* the smallest idle block of at least `bytes`, or a new one */
    void* take(size_t bytes) {
        bytes = (bytes + ((size_t)1 << 20) - 1) >> 20 << 20;
        {
            std::lock_guard<std::mutex> lock(g_pool_mu);
            size_t best = g_pool.size();
            for (size_t k = 0; k < g_pool.size(); ++k)
                if (g_pool[k].dev == dev_ && g_pool[k].bytes >= bytes &&
                    (best == g_pool.size() || g_pool[k].bytes < g_pool[best].bytes))
                    best = k;
            if (best < g_pool.size()) {
                b_ = g_pool[best];
                g_pool.erase(g_pool.begin() + best);
                return b_.p;
            }
        }
        void* p = nullptr;
        if (device_malloc(&p, bytes) != hipSuccess) return nullptr;
        b_ = PoolBlock{dev_, p, bytes};
        return p;
    }
    void drained() { drained_ = true; }

private:
    PoolBlock b_ = {0, nullptr, 0};
    int dev_;
    hipStream_t st_;
    bool drained_ = false;
};

/* The buffers of a call as offsets into its block (base null: only the size) */
struct Carve {
    char* base;
    size_t off = 0;
    template <typename T> T* take(size_t count) {
        T* p = base ? (T*)(base + off) : nullptr;
        off += (count * sizeof(T) + 255) / 256 * 256;
        return p;
    }
};

/* The fixed device workspace of amica_ll_forward_noalloc (callers that
 * cannot allocate: code under hipGraph capture, tight serving loops).  It
 * holds, in doubles: W^-1 (M n n), the inverse's scratch (M n n + 8 and
 * inverse_work_doubles), the per-(h, j, i) constants (M m n), W c (M NP) and
 * log|det W| (M).  Limits: M n n <= kNoAllocNN (e.g. 256 channels x 1 model,
 * 128 x 4), plus the forward's own M ceil(n/64) 64 <= 512, m <= 8.  1.6 MB per
 * device, held until the process ends; every call on a device shares it. */
constexpr size_t kNoAllocNN = 65536;
constexpr size_t kNoAllocNM = 4096;        /* 8 components x 512 padded channels */
constexpr size_t kNoAllocNP = 512;
constexpr size_t kNoAllocM = 8;
constexpr size_t kNoAllocWork = 2 * kNoAllocNN + 8 + 2 * kNoAllocNP;   /* M n <= M NP */
constexpr size_t kNoAllocDoubles = kNoAllocNN + kNoAllocWork + kNoAllocNM + kNoAllocNP + kNoAllocM;

__device__ __align__(256) double scratch[kNoAllocDoubles];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {nullptr};

/* The device address of `scratch` on the current device, looked up once per
 * device (each GPU holds its own copy of the array at its own address; the
 * array's name in host code is only a handle for the lookup). */
int noalloc_scratch(double** out) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return report_error(AMICA_E_DEVICE, "no HIP device");
    if (dev < 0 || dev >= kMaxDevices) return report_error(AMICA_E_DEVICE, "device ordinal out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        double* ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr)
            return report_error(AMICA_E_DEVICE, (std::string("hipGetSymbolAddress(scratch): ") +
                                                 hipGetErrorString(e)).c_str());
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return 0;
}

/* W^-1, log|det W|, W c, the constants of Q and (Wg) the GEMM operands */
template <typename Real>
int prepare_model(const AdjArgs& a, double* work, Real* Wg, Real* wcr, hipStream_t st) {
    if (launch_gj_inverse(a.W, a.Winv, a.ldet, a.n, a.M, work, st))
        return report_error(AMICA_E_DEVICE, "inverse launch failed");
    const long items = std::max((long)a.n * a.m, Wg ? (long)a.NP * a.NP : 0L);
    const int eb = (int)std::min<long>(1024, (items + 255) / 256);
    hipLaunchKernelGGL(adj_prep_kernel<Real>, dim3(eb + a.NP / 4, a.M), dim3(256), 0, st, a, eb, Wg, wcr);
    return hipGetLastError() == hipSuccess ? 0 : report_error(AMICA_E_DEVICE, "prep launch failed");
}

/* Workgroups of the likelihood kernel over T samples and the samples of each
 * (whole tiles of 4): 16 waves per CU, which its registers allow on the
 * forward passes; where the adjoint's allow half, the rest queue.  A short
 * call runs one tile per wave (a tile is a chain of ~5 us in FP64). */
int ll_grid(long T, int pairs, int cus, long* chunk) {
    const long waves = pairs <= 8 ? pairs : 8L * ((pairs + 7) / 8);
    const long nb = std::max(1L, std::min(16L * cus / waves, (T + 3) / 4));
    *chunk = ((T + nb - 1) / nb + 3) / 4 * 4;
    return (int)((T + *chunk - 1) / *chunk);
}

/* b is formed in the likelihood kernel, 16 samples at a time on MFMA: nothing
 * of the size of the data is stored, and the call only enqueues. */
template <typename Real>
int forward_noalloc(AdjArgs a, const void* x, long T, double* ll, double* work, int cus, hipStream_t st) {
    const int rc = prepare_model<Real>(a, work, nullptr, nullptr, st);
    if (rc) return rc;
    a.x = x;
    a.T = T;
    a.ll = ll;
    const int nb = ll_grid(T, a.M * (a.NP / 64), cus, &a.chunk);
    return launch_ll<Real, false>(a.m, a, nb, st) ? report_error(AMICA_E_DEVICE, "likelihood kernel launch failed")
                                                  : 0;
}

/* Per-sample buffers (b, g, padded x) of one chunk of samples: small enough
 * that what one kernel writes the next reads from the 256 MB last-level
 * cache, large enough that a chunk's launches fill the GPU. */
constexpr size_t kChunkBytes = (size_t)256 << 20;

template <typename Real>
int run_chunks(AdjArgs a, const void* x, long T, const double* dll, double* ll, const AdjOut* out, bool split,
               int dev, int cus, hipStream_t st) {
    const bool adj = out != nullptr;
    const int n = a.n, NP = a.NP, M = a.M, m = a.m, ldb = M * NP, pairs = ldb / 64;
    const size_t nn = (size_t)n * n;
    constexpr size_t rb = sizeof(Real);
    const size_t per = rb * ((size_t)ldb * (adj ? 2 : 1) + (n != NP ? NP : 0)) + (split ? 8 * (size_t)(pairs + M) : 0);
    const long most = std::max(4096L, (long)(kChunkBytes / per));
    const long nc = (T + most - 1) / most;
    const long Tc = nc == 1 ? T : ((T + nc - 1) / nc + 63) / 64 * 64;
    const int C = (int)((T + Tc - 1) / Tc);
    const int nb = ll_grid(Tc, pairs, cus, &a.chunk);
    /* the statistic GEMM sum_t g_t x_t^T: FP32 MFMA over padded rows of x
     * (gx_f32_slab_kernel, row stride NP) on the FP32 variant, FP64 MFMA over
     * the unpadded rows (row stride n) on the FP64 one */
    const bool gx32 = rb == 4;
    const int slabs = (ldb / 64) * ((n + 63) / 64);
    const GxChunks gc32 = gx32 ? gx_f32_chunks(Tc, NP, ldb, cus, cus) : GxChunks{0, 0, 1, 0, 2};
    const int gchunks = gx32 ? gc32.n
                             : (int)std::max(1L, std::min(std::max(1L, 2L * cus / slabs), (Tc + 255) / 256));
    const int gxs = gx32 ? NP : n;
    const size_t pcount = (size_t)ldb * pair_stride(m) + M, gcount = (size_t)ldb * gxs;
    Workspace ws(dev, st);
    Real *Wg, *wcr, *bb, *xpad;
    double *work, *gxpart, *ptot, *gtot, *tmp;
    auto carve = [&](char* base) {
        Carve k{base};
        a.Winv = k.take<double>(M * nn);
        a.ldet = k.take<double>(M);
        a.cq = k.take<double>((size_t)M * m * n);
        a.wc = k.take<double>(ldb);
        work = k.take<double>(8 + M * nn + inverse_work_doubles(n, M));
        Wg = k.take<Real>((size_t)ldb * NP);
        wcr = k.take<Real>(ldb);
        bb = k.take<Real>((size_t)Tc * ldb);
        xpad = n != NP ? k.take<Real>((size_t)Tc * NP) : nullptr;
        if (split) {
            a.qbuf = k.take<double>((size_t)Tc * pairs);
            a.vbuf = k.take<double>((size_t)Tc * M);
        }
        if (adj) {
            a.g = k.take<Real>((size_t)Tc * ldb);
            a.part = k.take<double>((size_t)nb * a.pstride);
            gxpart = k.take<double>((size_t)gchunks * gcount);
            ptot = k.take<double>(pcount);
            gtot = k.take<double>(gcount);
            tmp = k.take<double>(sum_tmp_doubles(nb, pcount) + sum_tmp_doubles(gchunks, gcount));
        }
        return k.off;
    };
    char* base = (char*)ws.take(carve(nullptr));
    if (!base) return report_error(AMICA_E_NOMEM, "workspace allocation failed");
    carve(base);
    const int prc = prepare_model<Real>(a, work, Wg, wcr, st);
    if (prc) return prc;
    for (int c = 0; c < C; ++c) {
        const long t0 = (long)c * Tc, Tn = std::min(Tc, T - t0);
        AdjArgs k = a;
        const Real* xc = (const Real*)x + (size_t)t0 * n;
        const Real* xp = xc;
        k.x = xc;
        k.T = Tn;
        k.dll = adj ? dll + t0 : nullptr;
        k.ll = ll ? ll + t0 : nullptr;
        k.bbuf = bb;
        if (n != NP) {
            const unsigned pg = (unsigned)std::min<long>(65536, (Tn * NP + 255) / 256);
            hipLaunchKernelGGL(adj_pad_kernel<Real>, dim3(pg), dim3(256), 0, st, xc, xpad, Tn, n, NP);
            xp = xpad;
        }
        /* b = W x - W c by the unmixing GEMM on MFMA */
        int urc;
        if constexpr (rb == 8) urc = launch_unmix_f64(xp, Wg, wcr, bb, Tn, NP, ldb, cus, st);
        else urc = launch_unmix_f32(xp, Wg, wcr, bb, Tn, NP, ldb, cus, st);
        if (urc || hipGetLastError() != hipSuccess)
            return report_error(AMICA_E_DEVICE, "unmixing GEMM launch failed");
        const int nbn = (int)((Tn + a.chunk - 1) / a.chunk);
        if (adj ? launch_ll<Real, true>(m, k, nbn, st) : launch_ll<Real, false>(m, k, nbn, st))
            return report_error(AMICA_E_DEVICE, "likelihood kernel launch failed");
        if (!adj) continue;
        int gc = gchunks;
        if constexpr (rb == 4) {
            GxChunks last = gc32;
            last.n = gc = (int)((Tn + gc32.chunk - 1) / gc32.chunk) * gc32.spread;
            if (launch_gx_f32((const float*)a.g, xp, gxpart, Tn, NP, ldb, last, st))
                return report_error(AMICA_E_DEVICE, "statistic GEMM launch failed");
        } else {
            const long gch = ((Tn + gchunks - 1) / gchunks + 31) / 32 * 32;
            gc = (int)((Tn + gch - 1) / gch);
            hipLaunchKernelGGL(adj_gx_kernel, dim3(gc, ldb / 64, (n + 63) / 64), dim3(256), 0, st,
                               (const double*)a.g, xc, Tn, n, ldb, gch, gxpart);
        }
        /* onto the chunks' running totals, in their order */
        if (hipGetLastError() != hipSuccess ||
            launch_sum_parts(a.part, nbn, a.pstride, pcount, ptot, gxpart, gc, gcount, gtot, tmp, c > 0, st))
            return report_error(AMICA_E_DEVICE, "adjoint launch failed");
    }
    if (adj) {
        const int eb = (int)std::min<size_t>(1024, (nn + (size_t)n * m + 255) / 256);
        hipLaunchKernelGGL(adj_finish_kernel, dim3(eb + (n + 3) / 4, M), dim3(256), 0, st, a, eb, ptot, gtot, gxs,
                           *out);
        if (hipGetLastError() != hipSuccess) return report_error(AMICA_E_DEVICE, "adjoint launch failed");
    }
    const hipError_t e = hipStreamSynchronize(st);
    if (e != hipSuccess) return report_error(AMICA_E_DEVICE, hipGetErrorString(e));
    ws.drained();
    return 0;
}

int ll_call(int real_bits, const void* x, long T, int n, int M, int m, const double* W,
            const double* c, const double* alpha, const double* mu, const double* beta,
            const double* rho, const double* gm, double ldetS, const double* dll, double* ll,
            const AdjOut* out, void* stream, bool noalloc = false) {
    const bool adj = out != nullptr;
    if (real_bits != 32 && real_bits != 64) return report_error(AMICA_E_INVALID, "real_bits must be 32 or 64");
    if (!x || !W || !c || !alpha || !mu || !beta || !rho || !gm || (adj && !dll))
        return report_error(AMICA_E_INVALID, "null argument");
    if (adj && (!out->dW || !out->dc || !out->dalpha || !out->dmu || !out->dbeta || !out->drho || !out->dgm))
        return report_error(AMICA_E_INVALID, "null gradient output");
    if (!adj && !ll) return report_error(AMICA_E_INVALID, "null ll output");
    if (T < 1 || n < 1 || M < 1 || m < 1 || m > 8)
        return report_error(AMICA_E_INVALID, "need T >= 1, n >= 1, M >= 1, 1 <= m <= 8");
    if (n > 1024 || M > 16) return report_error(AMICA_E_INVALID, "need n <= 1024 and M <= 16");
    const int NP = (n + 63) / 64 * 64;
    /* all (model, channel-block) pairs in one workgroup, else the split passes */
    const bool split = (long)M * NP > 512;
    if (split && noalloc)
        return report_error(AMICA_E_INVALID, "M * ceil(n/64) * 64 must be <= 512 without allocation");
    hipStream_t st = (hipStream_t)stream;
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return report_error(AMICA_E_DEVICE, "no HIP device");

    AdjArgs a = {};
    a.n = n; a.NP = NP; a.M = M; a.m = m;
    a.W = W; a.c = c; a.alpha = alpha; a.mu = mu; a.beta = beta; a.rho = rho; a.gm = gm;
    a.ldetS = ldetS;
    a.pstride = ((size_t)M * NP * pair_stride(m) + M + 31) & ~(size_t)31;
    a.pg = 8;
    if (noalloc) {
        /* forward only, workspace carved from the static device array */
        if ((size_t)M * n * n > kNoAllocNN)
            return report_error(AMICA_E_INVALID, "M * n * n exceeds the allocation-free workspace (65536)");
        double* sp = nullptr;
        const int rc = noalloc_scratch(&sp);
        if (rc) return rc;
        a.Winv = sp;
        double* work = sp + kNoAllocNN;
        a.cq = work + kNoAllocWork;
        a.wc = a.cq + kNoAllocNM;
        a.ldet = a.wc + kNoAllocNP;
        return real_bits == 64 ? forward_noalloc<double>(a, x, T, ll, work, cus, st)
                               : forward_noalloc<float>(a, x, T, ll, work, cus, st);
    }
    return real_bits == 64 ? run_chunks<double>(a, x, T, dll, ll, out, split, dev, cus, st)
                           : run_chunks<float>(a, x, T, dll, ll, out, split, dev, cus, st);
}

}  // namespace

hipError_t device_malloc(void** p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        int dev = 0;
        if (hipGetDevice(&dev) == hipSuccess && release_pool(dev) == hipSuccess) e = hipMalloc(p, bytes);
    }
    if (e != hipSuccess) (void)hipGetLastError();     /* reported by the caller, not by a later launch */
    return e;
}

}  // namespace amica

extern "C" int amica_ll_release_workspace(void) {
    const hipError_t e = amica::release_pool(-1);
    return e == hipSuccess ? 0 : amica::report_error(AMICA_E_DEVICE, hipGetErrorString(e));
}

extern "C" int amica_ll_forward(int real_bits, const void* x, long T, int n, int M, int m,
                                const double* W, const double* c, const double* alpha,
                                const double* mu, const double* beta, const double* rho,
                                const double* gm, double ldetS, double* ll, void* stream) {
    return amica::ll_call(real_bits, x, T, n, M, m, W, c, alpha, mu, beta, rho, gm, ldetS, nullptr,
                          ll, nullptr, stream);
}

extern "C" int amica_ll_forward_noalloc(int real_bits, const void* x, long T, int n, int M, int m,
                                        const double* W, const double* c, const double* alpha,
                                        const double* mu, const double* beta, const double* rho,
                                        const double* gm, double ldetS, double* ll, void* stream) {
    return amica::ll_call(real_bits, x, T, n, M, m, W, c, alpha, mu, beta, rho, gm, ldetS, nullptr,
                          ll, nullptr, stream, true);
}

extern "C" int amica_ll_adjoint(int real_bits, const void* x, long T, int n, int M, int m,
                                const double* W, const double* c, const double* alpha,
                                const double* mu, const double* beta, const double* rho,
                                const double* gm, double ldetS, const double* dll, double* ll,
                                double* dW, double* dc, double* dalpha, double* dmu, double* dbeta,
                                double* drho, double* dgm, void* stream) {
    const amica::AdjOut out = {dW, dc, dalpha, dmu, dbeta, drho, dgm};
    return amica::ll_call(real_bits, x, T, n, M, m, W, c, alpha, mu, beta, rho, gm, ldetS, dll, ll,
                          &out, stream);
}
