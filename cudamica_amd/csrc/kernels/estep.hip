/*
 * estep.hip -- fused AMICA E-step for gfx950.
 *
 * One kernel computes, for every sample t, model h, channel i and mixture
 * component j, everything the reference spreads over ten kernels and two
 * cuBLAS calls per block (fraimondo/cudamica src/amica.cu:1109-1606):
 *   y    = sqrt(beta) (b - mu)                         betabyxminusmu   kernels.cu:251-272
 *   Q    = log a + .5 log beta - log2 - lgamma(1+1/rho) - |y|^rho
 *                                                      logalogblogpfun  kernels.cu:282-307
 *   q    = logsumexp_j Q, z = exp(Q - q), L_h += sum_i q     updateltz  kernels.cu:317-366
 *   P    = logsumexp_h L, v = exp(L - P), LL += P             updatell  kernels.cu:376-450
 *   u    = v z, f = rho sign(y)|y|^(rho-1), g = sum_j sqrt(beta) u f
 *                                   computeu / computefp / computeg  kernels.cu:473-574
 *   usum, kappa, lambda, mu, beta, rho numerators         getusum ... getdrhonumer
 *   vsum, sigma2 = sum v b^2, cnew = sum v x               amica.cu:1280-1323, 1584
 * and writes g for the statistic GEMM (float32 [T][ldb], or bf16 packed 8
 * samples per column, [T/8][ldb][8], the layout the BF16 statistic GEMM
 * reads its MFMA fragments in).
 *
 * Layout: b and g are [T][ldb] with column h*NP + i; x is [T][NP]; NP is n
 * rounded up to 64.  Lane = channel, wave = (model h, 64-channel block cb);
 * a workgroup of M*CW waves owns a contiguous range of samples, so the
 * cross-channel sum (DPP row sums + LDS) and the cross-model logsumexp
 * stay on chip.  Per-element transcendentals are cut to three:
 *   la  = log2|y|
 *   ym2 = 2^((rho-2) la) = |y|^(rho-2),  sy = ym2 y = sign(y)|y|^(rho-1),
 *   yr  = sy y = |y|^rho
 *   e_j = 2^Q2_j  with Q2 = Q log2(e) (shifted by max_j Q2 only when
 *         every component underflows)
 * and every statistic becomes a product of these with u, with the constant
 * per-(h,j,i) factors (rho, sqrt(beta), ln 2) applied once in the reduction:
 *   usum   = sum u                       mu_numer  = rho  sum u sy
 *   kappa  = beta rho^2 sum u sy^2        mu_denom  = sqrt(beta) rho sum u ym2   (rho <= 2)
 *   beta_d = rho sum u yr                            sqrt(beta) rho^2 sum u sy^2 (rho > 2)
 *   lambda = rho^2 sum u yr^2 - 2 rho sum u yr + usum
 *   rho_n  = rho ln2 sum u yr la
 * Statistics are summed in FP32 registers over 32 samples, those partials in
 * FP32 per lane in LDS over 1024 samples, and those in FP64 in the
 * workgroup's own slot of the partial buffer, which the reduction kernel
 * sums over workgroups in a fixed order (no atomics, run-to-run identical).
 *
 * Bound: the vector ALU.  The arithmetic alone takes about 310 cycles per
 * sample and wave at m = 3 (three transcendentals at 8.3 and some fifteen
 * FP32 operations at 2.8-3.4 cycles each, per component), the kernel about
 * 450: the rest is loads, the row sums, the exchange between the waves (about
 * 40) and the flushes.  So the fixed work is shared out: tiles of four samples
 * (two for m = 4 from FP32 b and for m = 3 from FP64 b in large workgroups, one
 * above) pass the two barriers that publish the channel sums and then the model
 * posteriors, which one wave evaluates for the workgroup, a row of 16 lanes to
 * a sample; one underflow test serves a tile, and with four samples decides
 * before the densities are evaluated; b loads are issued a tile ahead, x loads
 * before the tile's densities, or with less than four samples ahead as well.
 * What that costs in registers comes back by keeping only what an FMA or two
 * cannot form again; one-sample tiles keep it all.  The per-lane LDS footprint (FP32 level-2 totals) leaves room
 * for two 512-thread workgroups per CU.  Against tiles of two samples (one for
 * m = 4) with every intermediate kept, in us: 128 ch x 1M x 4 models m = 3
 * 1526 -> 1463, 256 ch x 500k x 2 models m = 4 1036 -> 961, 128 ch x 500k x 2
 * models with FP64 b 469 -> 440, the split launch's passes (300 ch x 60k x 3
 * models) 515 -> 350.  One barrier with the posteriors formed in every wave
 * (1628) or a tile later (1754) is slower than either.
 *
 * B64 = true (FP32 path): b is FP64 and y = sqrt(beta)(b - mu) is formed in
 * FP64 before the FP32 density math, so |y| near 0 -- where mu_denom's
 * weight |y|^(rho-2) is singular for rho < 2 -- keeps full relative
 * precision.
 */
#include <algorithm>

#include "common.h"
#include "engine_internal.h"

namespace amica {

namespace {

constexpr int kBufferRsrcWord3 = 0x00020000;   /* raw 32-bit buffer, gfx9-family format */
constexpr int kFlush2 = 32;    /* register flushes summed in FP32 LDS */

__device__ __forceinline__ float fast_log2(float x) { return __builtin_amdgcn_logf(x); }
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float fast_rcp(float x) { return __builtin_amdgcn_rcpf(x); }

template <int CTRL, int ROWS, int BANKS, bool BOUND>
__device__ __forceinline__ float dpp(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v),
                                                                 CTRL, ROWS, BANKS, BOUND));
}

/* max of v and the value a row rotation by R (1, 2, 4, 8) brings in; every
 * lane of every row has a source, so the DPP move keeps no old value */
template <int R>
__device__ __forceinline__ float row_ror_max(float v) {
    const float o = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v),
                                                                       0x120 + R, 0xf, 0xf, false));
    return fmaxf(v, o);
}

/* Sum over each row of 16 lanes; the row total lands in the row's lane 15
 * (the other lanes hold partial sums).  Row shifts by 1, 2, 4 and 8 with
 * zeros shifted in, each one v_add_f32 with a DPP source. */
__device__ __forceinline__ float row_sum_lane15(float v) {
    v += dpp<0x111, 0xf, 0xf, true>(v);
    v += dpp<0x112, 0xf, 0xf, true>(v);
    v += dpp<0x114, 0xf, 0xf, true>(v);
    v += dpp<0x118, 0xf, 0xf, true>(v);
    return v;
}

/* Floor of |y| before log2|y|.  FP32 path (y formed in FP64 from FP64 b):
 * the smallest normal float.  Split-BF16 and FP8 paths (y = sb b - sb mu in
 * FP32 from FP32 b): 2^-24, the FP32 spacing at |sb mu| ~ 1.  There b can
 * round exactly onto mu, and the y that cancels to 0 would give
 * |y|^(rho-2) = 2^63 for rho = 1.5 and swamp the mu denominator
 * sum(u |y|^(rho-2)), which is singular at y = 0 for rho < 2; at the FP32
 * spacing the weight stays of the size FP64 gives its smallest |y|.  (A
 * floor at the ~2^-17 error of the BF16 GEMM would cap the weights of all
 * |y| below it and bias mu_denom low.) */
template <bool B64>
__device__ __forceinline__ constexpr float y_floor() { return B64 ? 1.17549435e-38f : 0x1p-24f; }

/* two floats -> two round-to-nearest-even bf16 in one dword (a low): one
 * v_cvt_pk_bf16_f32 */
__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2){a, b}, bf2));
}

/* The FP64 level of a lane's NS statistic sums: l3[s] = l3[s] + add(s)
 * (add(s) the first time), or 0 where keep is false.  The loads go out B
 * at a time before their adds, so a flush costs ceil(NS / B) memory round
 * trips instead of one per sum, for 2 B transient registers. */
template <int NS, int B, typename F>
__device__ __forceinline__ void l3_accumulate(double* l3, bool started, bool keep, F add) {
#pragma unroll
    for (int s0 = 0; s0 < NS; s0 += B) {
        double cur[B];
        if (started) {                  /* wave-uniform */
#pragma unroll
            for (int k = 0; k < B; ++k) cur[k] = s0 + k < NS ? l3[s0 + k] : 0.0;
        } else {
#pragma unroll
            for (int k = 0; k < B; ++k) cur[k] = 0.0;
        }
#pragma unroll
        for (int k = 0; k < B; ++k)
            if (s0 + k < NS) l3[s0 + k] = keep ? cur[k] + add(s0 + k) : 0.0;
    }
}

/* Samples per tile: as many as keep the kernel at 4 waves per SIMD (128 VGPRs).
 * With FP64 b at m = 3, where y is kept, four samples take 151 VGPRs and leave 3:
 * faster for workgroups of up to four waves, which pack three waves a SIMD
 * (estep of 128 ch x 500k x 2 models: 440 us, 469 with two), slower for larger
 * ones, of which a CU then holds one instead of two or three (128 ch x 130k x
 * 4 models 1.24 times, 64 ch x 208k x 5 models 1.35 times), and in the split
 * launch (300 ch x 74k x 3 models 1.08 times). */
constexpr int estep_tile_samples(int MJ, bool B64, bool small) {
    return MJ <= 3 ? (B64 && MJ == 3 && !small ? 2 : 4) : MJ == 4 && !B64 ? 2 : 1;
}
constexpr int kSmallWaves = 4;      /* waves of a fused workgroup that counts as small */

/* Whether sy and |y|^rho (and with FP32 b, y) are kept between the phases
 * instead of formed again, by a product or two each.  One-sample tiles have the
 * registers for it, but not the split launch's statistics pass up to m = 6, and
 * not m = 5 on the plain path in workgroups of 5 to 7 waves: kept, it takes 148
 * VGPRs, and one such workgroup fits a CU where two do with 124 (E-step of 64
 * ch x 5 models, kept / formed again: 1.5 times; at 2 waves 0.83 times). */
constexpr bool estep_keeps(int MJ, bool B64, int mode, bool GB, bool mid) {
    return (MJ >= 5 || (MJ == 4 && B64)) && (mode == kEstepFused ? !(mid && MJ == 5 && !B64 && !GB) : MJ >= 7);
}

/* MODE selects the launch the kernel serves (GB: g as packed bf16):
 *   kEstepFused  all M models x CW channel blocks in one workgroup (M CW <= 8):
 *                the cross-channel and cross-model sums stay on chip;
 *   kEstepLsum   split launch, first pass: a workgroup holds a group of models
 *                x channel blocks (blockIdx.y), and writes each model's sum of
 *                q over its channel blocks per sample (lq);
 *   kEstepStats  split launch, last pass: the densities again, the model
 *                posteriors read from vq (written between the passes by
 *                estep_post_kernel), then the statistics and g. */
template <int MJ, bool B64, int MODE, bool GB, int kS, bool kKeep, bool kThree>
__global__ __launch_bounds__(512) void estep_kernel(EstepArgs a) {
    static_assert(8 % kS == 0 && 7 + kS <= kEstepRowPad, "the unchecked loads past a range stay in the padding rows");
    /* a register past the 128 that four waves per SIMD leave: three then */
    if constexpr (kThree) __asm__ volatile("" ::: "v130");
    static_assert(!kKeep || kS == 1, "larger tiles have no registers to keep more");
    constexpr bool kRecY = !B64 && !kKeep;
    /* a tile of four samples is long enough for its own x to arrive behind its
     * densities; with one or two, x is loaded a tile ahead, as b is (E-step of
     * 64 ch x 2 models on the FP32 path, us at m = 4, 5, 6, 8 against loads in
     * the tile: 0.84, 0.82, 0.80, 0.87 times) */
    constexpr bool kXAhead = kS <= 2;
    /* the underflow test before the densities (below) */
    constexpr bool kShiftFirst = kS == 4 && MODE == kEstepFused;
    constexpr int kFlush = 32 / kS;     /* tiles summed in FP32 registers (32 samples) */
    /* FP64 flushes with batched loads, except in the split launch's
     * statistics pass, which they would push past 128 VGPRs on the FP32
     * path */
    constexpr bool kL3Batched = MODE != kEstepStats;
    constexpr int NSJ = kStatsPerJ;
    constexpr int NS = NSJ * MJ + kStatsPerI;
    constexpr bool kSplit = MODE != kEstepFused;
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   /* wave-uniform */
    int h, cb, hg = 0, cg = 0;
    bool wreal = true;                  /* wave-uniform: the wave owns real columns */
    if constexpr (kSplit) {
        hg = blockIdx.y / a.ncg;
        cg = blockIdx.y - hg * a.ncg;
        const int hl = w / a.cwg;
        h = hg * a.mg + hl;
        cb = cg * a.cwg + (w - hl * a.cwg);
        wreal = h < a.M && cb < a.CW;
        /* a wave past the last model or channel block reads a real column and
         * runs as padding channels (q = 0, no statistics, nothing written) */
        h = min(h, a.M - 1);
        cb = min(cb, a.CW - 1);
    } else {
        h = w / a.CW;
        cb = w - h * a.CW;
    }
    const int i = cb * 64 + lane;
    const bool act = wreal && i < a.n;

    /* per-row channel sums of one tile, double buffered:
     * [buf][wave][sample][row of 16 lanes] (a sample's 4 rows in 16 bytes),
     * and the tile's model posteriors [buf][model][sample] */
    __shared__ __align__(16) float Lp[2][kMaxEstepWaves][kS][4];
    __shared__ __align__(16) float Vp[2][kMaxEstepWaves][kS];
    __shared__ float dc2[AMICA_MAX_M];
    /* per-lane FP32 level-2 totals, [blockDim.x][NSP] (odd stride: the
     * lanes of a wave hit distinct banks) */
    constexpr int NSP = NS | 1;
    extern __shared__ float tot2_all[];
    float* const tot2 = tot2_all + threadIdx.x * NSP;

    /* L'_h = (log gm + ldet + ldetS) - c0 with c0 = max_h of that constant,
     * so that only differences enter FP32 (in log2 units). */
    if ((int)threadIdx.x < a.M) {
        double c0 = a.lconst[0];
        for (int hh = 1; hh < a.M; ++hh) c0 = fmax(c0, a.lconst[hh]);
        dc2[threadIdx.x] = (float)((a.lconst[threadIdx.x] - c0) * 1.4426950408889634);
    }

    float sb[MJ], nsbmu[MJ], rm2[MJ], cq2[MJ], rsb[MJ];
    double sb64[B64 ? MJ : 1], nsbmu64[B64 ? MJ : 1];
    /* FP32 path, m = 3: the FP64 constants live in LDS ([j][2][thread],
     * conflict-free, each thread its own slots), read for every sample, instead
     * of in 12 VGPRs */
    constexpr bool kC64Lds = B64 && MJ == 3;
    __shared__ double c64s[kC64Lds ? 2 * MJ * 512 : 1];
#pragma unroll
    for (int j = 0; j < MJ; ++j) {
        const float* cj = a.cst + ((size_t)h * kNumCst * MJ + j) * a.NP + i;
        const size_t ks = (size_t)MJ * a.NP;
        if (act) {
            sb[j] = cj[kCstSb * ks];
            nsbmu[j] = cj[kCstNsbmu * ks];
            rm2[j] = cj[kCstRm2 * ks];
            cq2[j] = cj[kCstCq2 * ks];
            rsb[j] = cj[kCstRsb * ks];
        } else {
            /* a padding channel: b = 0 gives y = 1, |y|^rho = 1, so
             * q2 = (0, -1e30, ...) and the component sum is exactly 1: its
             * log (the channel's share of L) is exactly 0, and g = 0 */
            sb[j] = 0.f; nsbmu[j] = 1.f; rm2[j] = 0.f; cq2[j] = j == 0 ? AMICA_L2E : -1e30f;
            rsb[j] = 0.f;
        }
        if constexpr (B64) {
            const double* dj = a.cst64 + ((size_t)h * kNumCst64 * MJ + j) * a.NP + i;
            sb64[j] = act ? dj[kCst64Sb * ks] : 0.0;
            nsbmu64[j] = act ? dj[kCst64Nsbmu * ks] : 1.0;
            if constexpr (kC64Lds) {
                c64s[(2 * j) * 512 + threadIdx.x] = sb64[j];
                c64s[(2 * j + 1) * 512 + threadIdx.x] = nsbmu64[j];
            }
        }
    }
    if constexpr (MODE != kEstepLsum) {
#pragma unroll
        for (int s = 0; s < NS; ++s) tot2[s] = 0.f;
    }

    float acc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) acc[s] = 0.f;
    double vsum_acc = 0.0, ll_acc = 0.0;
    double* const base = a.part + (size_t)blockIdx.x * a.pstride;
    /* this lane's FP64 totals: [M][NP][NS], contiguous per lane */
    double* const l3 = base + ((size_t)h * a.NP + i) * NS;
    bool l3_started = false;

    const long t0 = (long)blockIdx.x * a.chunk;
    const long t1 = min(a.T, t0 + a.chunk);
    const size_t bcol = (size_t)h * a.NP + i;
    int buf = 0, tiles = 0, flushes = 0;
    /* bf16 g, 8 samples packed per column: [t/8][ldb][8], one 16-byte store
     * per 8-sample group (t0 is a multiple of 8) */
    uint4* const g8 = (uint4*)a.g;

    /* the loads of the first tile.  Loads carry no channel check: lanes
     * i in [n, NP) read the padding columns of b and x, which hold zeros
     * (the padding rows of W and entries of W c are zero, and x's padding
     * columns are written as zero), so every load is unconditional and the
     * wait for a prefetch can sit where its value is first used. */
    float bn[kS], xn[kXAhead ? kS : 1];
    double bn64[B64 ? kS : 1];
    /* b and x through buffer resources based at row t0: the lane's byte
     * offset is fixed, the row's a scalar (launch_estep bounds it below
     * 2^31), so a load costs no address arithmetic on the vector ALU */
    constexpr int kEb = B64 ? 8 : 4;
    const char* const bbase = (const char*)(B64 ? (const void*)a.b64 : (const void*)a.b);
    auto rsrc_b = [&](long t) {
        return __builtin_amdgcn_make_buffer_rsrc((void*)(bbase + (size_t)t * a.ldb * kEb), (short)0,
                                                 (int)0xffffffff, kBufferRsrcWord3);
    };
    auto rsrc_x = [&](long t) {
        return __builtin_amdgcn_make_buffer_rsrc((void*)(a.x + (size_t)t * a.NP), (short)0,
                                                 (int)0xffffffff, kBufferRsrcWord3);
    };
    /* rows are addressed relative to tbase: the workgroup's first row (fused
     * launch, whose row offsets launch_estep bounds), or in the split
     * launches -- whose rows may be far wider -- the current 8-sample group */
    long tbase = t0;
    __amdgpu_buffer_rsrc_t rb = rsrc_b(t0), rx = rsrc_x(t0);
    const int vob = (int)bcol * kEb, vox = i * 4;
    const int browb = a.ldb * kEb, xrowb = a.NP * 4;
    auto load_tile = [&](long t, int s) {
        const int r = (int)(t - tbase);
        if constexpr (B64)
            bn64[s] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rb, vob, r * browb, 0));
        else
            bn[s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, vob, r * browb, 0));
        if constexpr (kXAhead && MODE != kEstepLsum)
            xn[s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, vox, r * xrowb, 0));
    };
#pragma unroll
    for (int s = 0; s < kS; ++s) load_tile(t0 + s, s);

    constexpr int kTPG = 8 / kS;               /* tiles per packed 8-sample group */
    for (long tg = t0; tg < t1; tg += 8) {
        if constexpr (kSplit) {
            /* loads already in flight keep the resources they were issued with */
            tbase = tg;
            rb = rsrc_b(tg);
            rx = rsrc_x(tg);
        }
        /* the group's packed g words (2 samples each); tiles past t1 in the
         * last group run with posterior 0 and so give g = 0 */
        uint32_t gw[4] = {0u, 0u, 0u, 0u};
        float gpend = 0.f;
#pragma unroll
        for (int sub = 0; sub < kTPG; ++sub) {
            const long tb = tg + sub * kS;
            /* kept per component and sample: |y|^(rho-2), log2|y|, 2^Q, where it
             * is formed in FP64 y, and with kKeep sy and |y|^rho */
            float E[kS][MJ], Y[kS][MJ], YM2[kS][MJ], LA[kS][MJ], SY[kKeep ? kS : 1][MJ], YR[kKeep ? kS : 1][MJ];
            float RS[kS], BV[kS], XV[kS], SE[kS];
            double BV64[B64 ? kS : 1];
#pragma unroll
            for (int s = 0; s < kS; ++s) {
                if constexpr (B64) { BV64[s] = bn64[s]; BV[s] = (float)bn64[s]; }
                else BV[s] = bn[s];
                if constexpr (kXAhead && MODE != kEstepLsum) XV[s] = xn[s];
            }
            /* issue the next tile's b loads and, unless they were ahead too,
             * this one's x loads (first used after the exchange) now; they
             * complete under this tile's math.  Rows past t1 are read without a check (the next range's
             * samples, or the kEstepRowPad zero rows after the last one) and
             * get posterior 0. */
            if constexpr (!kXAhead && MODE != kEstepLsum) {
#pragma unroll
                for (int s = 0; s < kS; ++s)
                    XV[s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                          rx, vox, (int)(tb - tbase + s) * xrowb, 0));
            }
#pragma unroll
            for (int s = 0; s < kS; ++s) load_tile(tb + kS + s, s);
            /* ---- phase 1: densities, component posteriors, channel sums ---- */
            float QS[kS];
            /* q2 <= log2(alpha sqrt(beta) / (2 Gamma(1 + 1/rho))), a few units,
             * so 2^q2 needs no max shift unless every component underflows (a
             * sample far from all of them: sum 2^q2 < 2^-100): then, for the
             * whole wave, that sample's are shifted by the per-lane max.  The
             * max alone says so (2^off <= sum <= 8 * 2^off) but for a narrow
             * band, in which the sum is formed to see.  Heavy-tailed data shift
             * some lane of nearly every wave's samples, so the densities are
             * evaluated once, after that is known, and not again with the shift: 3.42
             * -> 3.04 ms a launch at 128 ch x 2M x 4 models of super-Gaussian
             * sources, no change where none is that far out.  Smaller tiles and
             * the split launch, with fewer samples to overlap, evaluate first
             * and shift afterwards: 961 instead of 1000 us at 256 ch x 500k x 2
             * models m = 4, 350 instead of 369 at 300 ch x 60k x 3 models.  Both
             * give the same bits. */
            if constexpr (kShiftFirst) {
            float off[kS];
#pragma unroll
            for (int s = 0; s < kS; ++s) {
#pragma unroll
                for (int j = 0; j < MJ; ++j) {
                    float y;
                    if constexpr (kC64Lds)
                        y = (float)fma(c64s[(2 * j) * 512 + threadIdx.x], BV64[s],
                                       c64s[(2 * j + 1) * 512 + threadIdx.x]);
                    else if constexpr (B64) y = (float)fma(sb64[j], BV64[s], nsbmu64[j]);
                    else y = fmaf(sb[j], BV[s], nsbmu[j]);
                    const float la = fast_log2(fmaxf(fabsf(y), y_floor<B64>()));
                    const float ym2 = fast_exp2(rm2[j] * la);
                    const float yr = (ym2 * y) * y;
                    E[s][j] = fmaf(yr, -AMICA_L2E, cq2[j]);               /* q2 */
                    off[s] = j == 0 ? E[s][0] : fmaxf(off[s], E[s][j]);
                    Y[s][j] = y; YM2[s][j] = ym2; LA[s][j] = la;
                }
            }
            float omin = off[0];
#pragma unroll
            for (int s = 1; s < kS; ++s) omin = fminf(omin, off[s]);
            const bool far = __builtin_expect(__any(omin < -99.5f), 0);
            if (far) {
#pragma unroll
                for (int s = 0; s < kS; ++s) {
                    bool shift = __any(off[s] < -103.5f);
                    if (!shift && __any(off[s] < -99.5f)) {
                        float se = 0.f;
#pragma unroll
                        for (int j = 0; j < MJ; ++j) se = j == 0 ? fast_exp2(E[s][0]) : se + fast_exp2(E[s][j]);
                        shift = __any(se < 0x1p-100f);
                    }
                    off[s] = shift ? off[s] : 0.f;
#pragma unroll
                    for (int j = 0; j < MJ; ++j) E[s][j] -= off[s];
                }
            }
#pragma unroll
            for (int s = 0; s < kS; ++s) {
#pragma unroll
                for (int j = 0; j < MJ; ++j) {
                    E[s][j] = fast_exp2(E[s][j]);
                    SE[s] = j == 0 ? E[s][j] : SE[s] + E[s][j];
                }
                QS[s] = fast_log2(SE[s]);         /* exactly 0 on padding channels */
            }
            if (far)
#pragma unroll
                for (int s = 0; s < kS; ++s) QS[s] += off[s];
            } else {
#pragma unroll
            for (int s = 0; s < kS; ++s) {
                SE[s] = 0.f;
#pragma unroll
                for (int j = 0; j < MJ; ++j) {
                    float y;
                    if constexpr (kC64Lds)
                        y = (float)fma(c64s[(2 * j) * 512 + threadIdx.x], BV64[s],
                                       c64s[(2 * j + 1) * 512 + threadIdx.x]);
                    else if constexpr (B64) y = (float)fma(sb64[j], BV64[s], nsbmu64[j]);
                    else y = fmaf(sb[j], BV[s], nsbmu[j]);
                    const float la = fast_log2(fmaxf(fabsf(y), y_floor<B64>()));
                    const float ym2 = fast_exp2(rm2[j] * la);
                    const float yr = (ym2 * y) * y;
                    E[s][j] = fast_exp2(fmaf(yr, -AMICA_L2E, cq2[j]));
                    SE[s] = j == 0 ? E[s][j] : SE[s] + E[s][j];
                    Y[s][j] = y; YM2[s][j] = ym2; LA[s][j] = la;
                    if constexpr (kKeep) { SY[s][j] = ym2 * y; YR[s][j] = yr; }
                }
                QS[s] = fast_log2(SE[s]);         /* exactly 0 on padding channels */
            }
            /* (the empty asm, here and before phase 2, keeps the compiler from
             * holding on to the y it could form again) */
            if constexpr (kRecY)
#pragma unroll
                for (int s = 0; s < kS; ++s) __asm__ volatile("" : "+v"(BV[s]));
            float smin = SE[0];
#pragma unroll
            for (int s = 1; s < kS; ++s) smin = fminf(smin, SE[s]);
            if (__builtin_expect(__any(smin < 0x1p-100f), 0)) {
#pragma unroll
                for (int s = 0; s < kS; ++s) {
                    if (!__any(SE[s] < 0x1p-100f)) continue;
                    float q2[MJ], off = 0.f;
#pragma unroll
                    for (int j = 0; j < MJ; ++j) {
                        const float yv = kRecY ? fmaf(sb[j], BV[s], nsbmu[j]) : Y[s][j];
                        const float yr = (YM2[s][j] * yv) * yv;
                        q2[j] = fmaf(yr, -AMICA_L2E, cq2[j]);
                        off = j == 0 ? q2[0] : fmaxf(off, q2[j]);
                    }
#pragma unroll
                    for (int j = 0; j < MJ; ++j) {
                        E[s][j] = fast_exp2(q2[j] - off);
                        SE[s] = j == 0 ? E[s][j] : SE[s] + E[s][j];
                    }
                    QS[s] = off + fast_log2(SE[s]);
                }
            }
            }
#pragma unroll
            for (int s = 0; s < kS; ++s) RS[s] = fast_rcp(SE[s]);
            const int nval = (int)min(t1 - tb, (long)kS);    /* samples of the tile before t1 */
            float GV[kS], VV[kS];
            if constexpr (MODE == kEstepStats) {
                /* the posteriors of the split launch's middle pass */
#pragma unroll
                for (int s = 0; s < kS; ++s) VV[s] = s < nval ? a.vq[(size_t)(tb + s) * a.M + h] : 0.f;
            } else {
#pragma unroll
            for (int s = 0; s < kS; ++s) QS[s] = row_sum_lane15(QS[s]);
            if ((lane & 15) == 15) {
#pragma unroll
                for (int s = 0; s < kS; ++s) Lp[buf][w][s][lane >> 4] = QS[s];
            }
            __syncthreads();
            if constexpr (MODE == kEstepLsum) {
                /* wave 0: lane 16 s + hl adds the row sums of local model hl
                 * for sample s and writes them for the posterior pass */
                if (w == 0) {
                    const int hl = lane & 15, s = lane >> 4;
                    const int hh = hg * a.mg + hl;
                    if (s < kS && s < nval && hl < a.mg && hh < a.M) {
                        float l = 0.f;
                        for (int c = 0; c < a.cwg; ++c)
#pragma unroll
                            for (int row = 0; row < 4; ++row) l += Lp[buf][hl * a.cwg + c][s][row];
                        a.lq[((size_t)(tb + s) * a.M + hh) * a.ncg + cg] = l;
                    }
                }
                buf ^= 1;
                continue;
            } else {
            /* ---- model posteriors, by wave 0 alone: row s of 16 lanes holds
             * sample s, lane hh of it model hh (M <= 8), so that row rotations
             * by 1, 2, 4 (and 8) reach every model; the other waves read them
             * from LDS after a second barrier.  For m <= 3 lane hh + 8 holds
             * model hh again, else nothing: the order the models' sum has been
             * formed in with tiles of two samples and of one. ---- */
            constexpr bool kRow16 = MJ >= 4;
            if (w == 0) {
                /* the other waves wait for this one at the next barrier: let it
                 * issue ahead of the other workgroup's waves on its SIMD */
                __builtin_amdgcn_s_setprio(3);
                /* two-sample tiles for m <= 3 use all four rows, the pairs in
                 * turn: vsum and the LL sum then add up in the order they have
                 * with tiles of four, to the last bit */
                constexpr bool kPairs = kS == 2 && MJ <= 3;
                const int row = lane >> 4, hh = lane & (kRow16 ? 15 : 7);
                const int s = kPairs ? row & 1 : min(row, kS - 1);
                float l = -3.0e38f;
                if (hh < a.M) {
                    l = dc2[hh];
                    for (int c = 0; c < a.CW; ++c) {
                        const float4 r = *(const float4*)Lp[buf][hh * a.CW + c][s];
                        l += r.x;
                        l += r.y;
                        l += r.z;
                        l += r.w;
                    }
                }
                float lmax = row_ror_max<1>(l);
                lmax = row_ror_max<2>(lmax);
                lmax = row_ror_max<4>(lmax);
                if constexpr (kRow16) lmax = row_ror_max<8>(lmax);
                /* lanes hh >= M hold l = -3e38: e = 0 */
                const float e = fast_exp2(l - lmax);
                float esum = e;
                esum += dpp<0x121, 0xf, 0xf, false>(esum);
                esum += dpp<0x122, 0xf, 0xf, false>(esum);
                esum += dpp<0x124, 0xf, 0xf, false>(esum);
                if constexpr (kRow16) esum += dpp<0x128, 0xf, 0xf, false>(esum);
                const bool mine = (lane & 8) == 0 && (kPairs ? row >> 1 == (sub & 1) : row < kS), valid = s < nval;
                const float vl = valid ? e * fast_rcp(esum) : 0.f;
                if (mine) Vp[buf][hh][s] = vl;
                if (mine && valid && hh < a.M) {
                    vsum_acc += (double)vl;
                    if (hh == 0) ll_acc += (double)(lmax + fast_log2(esum)) * AMICA_LN2;
                    if (a.ltall) a.ltall[(size_t)hh * a.T + tb + s] = l * (float)AMICA_LN2;
                }
                __builtin_amdgcn_s_setprio(0);
            }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < kS; ++q) VV[q] = Vp[buf][h][q];
            }
            }
            /* ---- phase 2: responsibilities and statistics ---- */
            if constexpr (kRecY)
#pragma unroll
                for (int s = 0; s < kS; ++s) __asm__ volatile("" : "+v"(BV[s]));
#pragma unroll
            for (int s = 0; s < kS; ++s) {
                const float v = VV[s];
                const float vrs = v * RS[s];
                float g = 0.f;
#pragma unroll
                for (int j = 0; j < MJ; ++j) {
                    float u = E[s][j] * vrs;
                    float sy, yr;
                    if constexpr (kKeep) {
                        sy = SY[s][j];
                        yr = YR[s][j];
                    } else {
                        const float yv = kRecY ? fmaf(sb[j], BV[s], nsbmu[j]) : Y[s][j];
                        sy = YM2[s][j] * yv;
                        yr = sy * yv;
                    }
                    float uf = u * sy;
                    /* two of the sums round u and u f before they add them (the
                     * empty asm), or take the products into an FMA: which one is
                     * fixed here, as it has been for these m and samples, so that
                     * no other tiling moves a fit's FP32 rounding */
                    if (MJ >= 5 || (MJ <= 3 && s % 2 == 0)) __asm__ volatile("" : "+v"(u), "+v"(uf));
                    g = fmaf(uf, rsb[j], g);
                    float* aj = acc + j * NSJ;
                    aj[0] += u;
                    aj[1] += uf;
                    aj[2] = fmaf(uf, sy, aj[2]);
                    aj[3] = fmaf(u, YM2[s][j], aj[3]);
                    const float uyr = u * yr;
                    aj[4] += uyr;
                    aj[5] = fmaf(uyr, yr, aj[5]);
                    aj[6] = fmaf(uyr, LA[s][j], aj[6]);
                }
                /* g is 0 on padding channels (rsb = 0) and past t1 (v = 0) */
                const float vb = v * BV[s];
                acc[NSJ * MJ + 0] = fmaf(vb, BV[s], acc[NSJ * MJ + 0]);
                acc[NSJ * MJ + 1] = fmaf(v, XV[s], acc[NSJ * MJ + 1]);
                acc[NSJ * MJ + 2] += g;
                GV[s] = g;
                /* one sample at a time: the sums are complete here (empty asm
                 * with them as operands, no instruction), or the compiler would
                 * keep several samples' products live, beyond 128 VGPRs */
                if constexpr (!kKeep) {
#pragma unroll
                    for (int q = 0; q < NS; ++q) __asm__ volatile("" : "+v"(acc[q]));
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if constexpr (!GB) {
                if (wreal)
#pragma unroll
                    for (int s = 0; s < kS; ++s)
                        if (s < nval) ((float*)a.g)[(size_t)(tb + s) * a.ldb + bcol] = GV[s];
            } else if constexpr (kS >= 2) {
#pragma unroll
                for (int s = 0; s < kS; s += 2) gw[(sub * kS + s) >> 1] = pack_bf16x2(GV[s], GV[s + 1]);
            } else if (sub & 1) gw[sub >> 1] = pack_bf16x2(gpend, GV[0]);
            else gpend = GV[0];
            buf ^= 1;
            if (++tiles == kFlush) {
                tiles = 0;
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    tot2[s] += acc[s];
                    acc[s] = 0.f;
                }
                if (++flushes == kFlush2) {
                    flushes = 0;
                    if constexpr (kL3Batched) {
                        if (wreal)
                            l3_accumulate<NS, 8>(l3, l3_started, true, [&](int s) { return (double)tot2[s]; });
#pragma unroll
                        for (int s = 0; s < NS; ++s) tot2[s] = 0.f;
                    } else {
#pragma unroll
                        for (int s = 0; s < NS; ++s) {
                            const double v = (double)tot2[s];
                            if (wreal) l3[s] = l3_started ? l3[s] + v : v;
                            tot2[s] = 0.f;
                        }
                    }
                    l3_started = true;
                }
            }
        }
        if constexpr (MODE != kEstepLsum)
            if (GB && wreal) g8[(size_t)(tg >> 3) * a.ldb + bcol] = make_uint4(gw[0], gw[1], gw[2], gw[3]);
    }
    if constexpr (MODE == kEstepLsum) return;
    if constexpr (kL3Batched) {
        if (wreal)
            l3_accumulate<NS, 8>(l3, l3_started, act, [&](int s) { return (double)tot2[s] + (double)acc[s]; });
    } else {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const double v = (double)tot2[s] + (double)acc[s];
            const double r = l3_started ? l3[s] + v : v;
            if (wreal) l3[s] = act ? r : 0.0;
        }
    }
    if constexpr (MODE == kEstepStats) return;   /* vsum and the LL sum: estep_post_kernel */
    /* per-model vsum (lanes 16 s + hh of wave 0) and the LL sum (lanes 16 s) */
    if (w == 0) {
        const size_t tail = (size_t)a.M * NS * a.NP;
        for (int hh = 0; hh < a.M; ++hh) {
            const double vs = wave_sum_f64((lane & 15) == hh ? vsum_acc : 0.0);
            if (lane == 0) base[tail + hh] = vs;
        }
        const double ls = wave_sum_f64(ll_acc);
        if (lane == 0) base[tail + a.M] = ls;
    }
}

/* the kernel of a launch, by the workgroup's waves (fused: 2; up to
 * kSmallWaves; 5 to 7).  With FP64 b at m = 4 it takes 126 VGPRs, four waves per
 * SIMD, but the sample ranges are cut for three (estep_blocks_per_cu).  Workgroups
 * of two waves then crowd some SIMDs; held to three they spread evenly (E-step
 * of 64 ch x 2 models 1.10 times the time otherwise); larger ones use the room
 * (64 ch x 3 models 0.75 times). */
template <int MJ, bool B64, int MODE, bool GB, bool SMALL = false, bool MID = false, bool TWO = false>
constexpr auto estep_variant() {
    return &estep_kernel<MJ, B64, MODE, GB, estep_tile_samples(MJ, B64, SMALL), estep_keeps(MJ, B64, MODE, GB, MID),
                         TWO && MJ == 4 && B64>;
}

/* 4 x 4 transpose between the registers r[0..3] and the four rows of 16 lanes */
__device__ __forceinline__ void transpose_rows(uint32_t& r0, uint32_t& r1, uint32_t& r2, uint32_t& r3) {
    auto p = __builtin_amdgcn_permlane32_swap(r0, r2, false, false);
    auto q = __builtin_amdgcn_permlane32_swap(r1, r3, false, false);
    auto s = __builtin_amdgcn_permlane16_swap(p[0], q[0], false, false);
    auto t = __builtin_amdgcn_permlane16_swap(p[1], q[1], false, false);
    r0 = s[0]; r1 = s[1]; r2 = t[0]; r3 = t[1];
}

/* elements 2 q and 2 q + 1 in row q of a and b -> element q in a's row q and
 * 4 + q in b's */
__device__ __forceinline__ void swap_pairs(uint32_t& a, uint32_t& b) {
    auto p = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    auto q = __builtin_amdgcn_permlane32_swap(p[0], p[1], false, false);
    a = q[0]; b = q[1];
}

/* d[s] = sum_k W[lane][k] x[tb + s][k] for 16 samples of a 64-channel block:
 * v_mfma_f64_16x16x4f64 in the order of unmix_f64_lds_kernel (the same b), whose
 * results -- register r of lane l holds sample l/16 + 4 r of channel l%16 of
 * each 16 -- turn into a channel per lane by row transposes.  wfrag: the W
 * fragments, [k / 4][16-channel block][lane]. */
__device__ __forceinline__ void unmix_tile64(const double* __restrict__ x64, const double* wfrag, long tb,
                                             long T, int lane, double (&d)[16]) {
    typedef double f64x4 __attribute__((ext_vector_type(4)));
    const double* const xr = x64 + (size_t)min(tb + (lane & 15), T - 1) * 64 + 2 * (lane >> 4);
    uint4 xv[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) xv[k] = *(const uint4*)(xr + 8 * k);
    double xa[16];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        uint32_t lo0 = xv[k].x, hi0 = xv[k].y, lo1 = xv[k].z, hi1 = xv[k].w;
        swap_pairs(lo0, lo1);
        swap_pairs(hi0, hi1);
        xa[2 * k] = __builtin_bit_cast(double, (uint64_t)lo0 | (uint64_t)hi0 << 32);
        xa[2 * k + 1] = __builtin_bit_cast(double, (uint64_t)lo1 | (uint64_t)hi1 << 32);
    }
    f64x4 acc[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] = (f64x4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < 16; ++k)
#pragma unroll
        for (int c = 0; c < 4; ++c)
            acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(xa[k], wfrag[(k * 4 + c) * 64 + lane], acc[c], 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint64_t v = __builtin_bit_cast(uint64_t, (double)acc[c][r]);
            lo[c] = (uint32_t)v;
            hi[c] = (uint32_t)(v >> 32);
        }
        transpose_rows(lo[0], lo[1], lo[2], lo[3]);
        transpose_rows(hi[0], hi[1], hi[2], hi[3]);
#pragma unroll
        for (int q = 0; q < 4; ++q)
            d[4 * r + q] = __builtin_bit_cast(double, (uint64_t)lo[q] | (uint64_t)hi[q] << 32);
    }
}

/* M = 1: the model posterior v is 1, so the waves of a workgroup (the
 * 64-channel blocks of one range of samples) never exchange anything: no
 * barrier, no LDS, and phase 2 of a sample follows its phase 1 in
 * registers.  One sample per iteration, loads 3-4 samples ahead; the
 * statistics are summed in FP32 registers over 32 samples, in FP32 per lane
 * in LDS over 1024 samples (odd stride: distinct banks) and in FP64 in the
 * workgroup's slot of the partial buffer.  The log-likelihood sum is sum_t sum_i q_ti (the
 * model constant is added by the reduction); vsum is the sample count.
 * Not used when per-sample L is recorded (ltall). */
template <int MJ, bool B64, bool FUSE>
__device__ __forceinline__ void estep_m1_body(const EstepArgs& a, const long t0, const long t1,
                                              const int slot, const double* wfrag, float* const tot2_all,
                                              const double* c64s) {
    constexpr int NSJ = kStatsPerJ;
    constexpr int NS = NSJ * MJ + kStatsPerI;
    constexpr int G = 8;
    const bool gpacked = !FUSE && a.g_bf16;
    const int lane = threadIdx.x & 63, w = FUSE ? 0 : threadIdx.x >> 6;
    const int i = w * 64 + lane;
    const bool act = i < a.n;
    constexpr int NSP = NS | 1;
    float* const tot2 = tot2_all + threadIdx.x * NSP;
    /* FP32 path, m = 3: the FP64 constants live in LDS ([2 j + k][thread]
     * after the totals, each thread its own slots), read once per sample:
     * 12 VGPRs fewer, so that 4 waves per SIMD fit */
    constexpr bool kC64Lds = B64 && !FUSE && MJ == 3;
    double* const c64 = (double*)((char*)tot2_all + ((size_t)blockDim.x * NSP * sizeof(float) + 7) / 8 * 8);

    float sb[MJ], nsbmu[MJ], rm2[MJ], cq2[MJ], rsb[MJ];
    double sb64[B64 ? MJ : 1], nsbmu64[B64 ? MJ : 1];
#pragma unroll
    for (int j = 0; j < MJ; ++j) {
        const float* cj = a.cst + (size_t)j * a.NP + i;
        const size_t ks = (size_t)MJ * a.NP;
        /* a padding channel: y = 1, so q2 = (0, -1e30, ...) and the
         * component sum is exactly 1 (log 0 to the LL, g = 0) */
        sb[j] = act ? cj[kCstSb * ks] : 0.f;
        nsbmu[j] = act ? cj[kCstNsbmu * ks] : 1.f;
        rm2[j] = act ? cj[kCstRm2 * ks] : 0.f;
        cq2[j] = act ? cj[kCstCq2 * ks] : (j == 0 ? AMICA_L2E : -1e30f);
        rsb[j] = act ? cj[kCstRsb * ks] : 0.f;
        if constexpr (B64 && !FUSE) {
            const double* dj = a.cst64 + (size_t)j * a.NP + i;
            sb64[j] = act ? dj[kCst64Sb * ks] : 0.0;
            nsbmu64[j] = act ? dj[kCst64Nsbmu * ks] : 1.0;
            if constexpr (kC64Lds) {
                c64[(size_t)(2 * j) * blockDim.x + threadIdx.x] = sb64[j];
                c64[(size_t)(2 * j + 1) * blockDim.x + threadIdx.x] = nsbmu64[j];
            }
        }
    }
    float acc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        acc[s] = 0.f;
        tot2[s] = 0.f;
    }
    float qacc = 0.f;
    double qtot = 0.0;
    double* const base = a.part + (size_t)slot * a.pstride;
    double* const l3 = base + (size_t)i * NS;
    bool l3_started = false;

    const size_t bcol = (size_t)i;
    uint4* const g8 = (uint4*)a.g;

    /* a ring of PF prefetched samples; the loop runs whole packed
     * 8-sample groups with the sample loop unrolled, so that ring slots and
     * packed g words are fixed registers (PF divides 8) */
    constexpr int PF = 4;
    static_assert(G % PF == 0, "ring slots must repeat every group");
    float bq[PF], xq[PF];
    double dq[PF];
    /* Unconditional loads through buffer resources based at row t0 (scalar
     * row offsets, bounded by launch_estep): samples past T read row T, the
     * first of the zero padding rows (a range's samples past t1 below T are
     * only ever prefetched, never used), and lanes i in [n, NP) the zero
     * padding columns of b and x (the padding rows of W and entries of W c
     * are zero, and x's padding columns are written as zero). */
    constexpr int kEb = B64 ? 8 : 4;
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((const char*)(B64 ? (const void*)a.b64 : (const void*)a.b) + (size_t)t0 * a.ldb * kEb),
        (short)0, (int)0xffffffff, kBufferRsrcWord3);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.x + (size_t)t0 * a.NP), (short)0, (int)0xffffffff, kBufferRsrcWord3);
    const int vob = (int)bcol * kEb, vox = i * 4;
    auto ld = [&](long t, float& bqv, double& dqv, float& xqv) {
        const int r = (int)(min(t, a.T) - t0);
        if constexpr (FUSE) {
        } else if constexpr (B64)
            dqv = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rb, vob, r * a.ldb * kEb, 0));
        else
            bqv = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, vob, r * a.ldb * kEb, 0));
        xqv = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, vox, r * a.NP * 4, 0));
    };
#pragma unroll
    for (int p = 0; p < PF; ++p) {
        bq[p] = 0.f;
        dq[p] = 0.0;
        ld(t0 + p, bq[p], dq[p], xq[p]);
    }
    const long tend = t0 + (t1 - t0 + G - 1) / G * G;   /* whole 8-sample groups */
    int grp = 0;
    double d16[FUSE ? 16 : 1];
    double bias = 0.0;
    if constexpr (FUSE) bias = a.wc64[lane];
#pragma unroll 1
    for (long tg = t0; tg < tend; tg += G, ++grp) {
        uint32_t gw[G / 2];                           /* packed bf16 g, 2 samples a word */
        float gprev = 0.f;
        if constexpr (FUSE) {
            if ((grp & 1) == 0) unmix_tile64(a.x64, wfrag, tg, a.T, lane, d16);
            else
#pragma unroll
                for (int u = 0; u < 8; ++u) d16[u] = d16[8 + u];
        }
#pragma unroll
        for (int u = 0; u < G; ++u) {
            const long t = tg + u;
            const bool valid = t < t1;                /* wave-uniform */
            const int sl = u % PF;
            const float bcur = B64 ? 0.f : bq[sl];
            double dcur;
            if constexpr (FUSE) dcur = valid ? d16[u] - bias : 0.0;
            else dcur = dq[sl];
            const float xcur = xq[sl];
            ld(t + PF, bq[sl], dq[sl], xq[sl]);
            const float bv = B64 ? (float)dcur : bcur;
            /* the constants' LDS reads stay in the loop (not hoisted back into
             * registers): a compiler-only fence, no instruction */
            if constexpr (kC64Lds || FUSE) __asm__ volatile("" ::: "memory");
            float q2[MJ], E[MJ], SY[MJ], YM2[MJ], YR[MJ], LA[MJ];
#pragma unroll
            for (int j = 0; j < MJ; ++j) {
                float y;
                if constexpr (FUSE) y = (float)fma(c64s[2 * j * 64 + lane], dcur, c64s[(2 * j + 1) * 64 + lane]);
                else if constexpr (kC64Lds)
                    y = (float)fma(c64[(size_t)(2 * j) * blockDim.x + threadIdx.x], dcur,
                                   c64[(size_t)(2 * j + 1) * blockDim.x + threadIdx.x]);
                else if constexpr (B64) y = (float)fma(sb64[j], dcur, nsbmu64[j]);
                else y = fmaf(sb[j], bv, nsbmu[j]);
                LA[j] = fast_log2(fmaxf(fabsf(y), y_floor<B64>()));
                YM2[j] = fast_exp2(rm2[j] * LA[j]);
                SY[j] = YM2[j] * y;
                YR[j] = SY[j] * y;
                q2[j] = fmaf(YR[j], -AMICA_L2E, cq2[j]);
            }
            float se = 0.f, off = 0.f;
#pragma unroll
            for (int j = 0; j < MJ; ++j) {
                E[j] = fast_exp2(q2[j]);
                se += E[j];
            }
            if (__builtin_expect(__any(se < 0x1p-100f), 0)) {
                off = q2[0];
#pragma unroll
                for (int j = 1; j < MJ; ++j) off = fmaxf(off, q2[j]);
                se = 0.f;
#pragma unroll
                for (int j = 0; j < MJ; ++j) {
                    E[j] = fast_exp2(q2[j] - off);
                    se += E[j];
                }
            }
            /* samples past t1 (the last range's last group) count nothing */
            const float rs = valid ? fast_rcp(se) : 0.f;
            qacc += valid ? off + fast_log2(se) : 0.f;
            float g = 0.f;
#pragma unroll
            for (int j = 0; j < MJ; ++j) {
                const float u_ = E[j] * rs;
                const float uf = u_ * SY[j];
                g = fmaf(uf, rsb[j], g);
                float* aj = acc + j * NSJ;
                aj[0] += u_;
                aj[1] += uf;
                aj[2] = fmaf(uf, SY[j], aj[2]);
                aj[3] = fmaf(u_, YM2[j], aj[3]);
                const float uyr = u_ * YR[j];
                aj[4] += uyr;
                aj[5] = fmaf(uyr, YR[j], aj[5]);
                aj[6] = fmaf(uyr, LA[j], aj[6]);
            }
            acc[NSJ * MJ + 0] = fmaf(bv, bv, acc[NSJ * MJ + 0]);
            acc[NSJ * MJ + 1] += xcur;
            acc[NSJ * MJ + 2] += g;
            if (gpacked) {
                if (u & 1) gw[u >> 1] = pack_bf16x2(gprev, g);
                gprev = g;
            } else if (valid) {
                ((float*)a.g)[(size_t)t * a.ldb + bcol] = g;
            }
            /* one sample at a time: the sums are complete here (empty asm
             * with them as operands, no instruction) and the scheduler may
             * not interleave the unrolled samples -- deferring the sums would
             * keep every sample's values live, beyond 128 VGPRs */
#pragma unroll
            for (int s = 0; s < NS; ++s) __asm__ volatile("" : "+v"(acc[s]));
            __asm__ volatile("" : "+v"(qacc));
            __builtin_amdgcn_sched_barrier(0);
        }
        /* t0 is a multiple of 8: the group's packed word */
        if (gpacked) g8[(size_t)((tg) >> 3) * a.ldb + bcol] = make_uint4(gw[0], gw[1], gw[2], gw[3]);
        if ((grp & 3) == 3) {                         /* 32 samples */
#pragma unroll
            for (int s = 0; s < NS; ++s) { tot2[s] += acc[s]; acc[s] = 0.f; }
            qtot += (double)qacc;
            qacc = 0.f;
            if ((grp & 127) == 127) {                 /* 1024 samples */
                l3_accumulate<NS, 8>(l3, l3_started, true, [&](int s) { return (double)tot2[s]; });
#pragma unroll
                for (int s = 0; s < NS; ++s) tot2[s] = 0.f;
                l3_started = true;
            }
        }
    }
    l3_accumulate<NS, 8>(l3, l3_started, act, [&](int s) { return (double)tot2[s] + (double)acc[s]; });
    qtot += (double)qacc;
    const double ls = wave_sum_f64(qtot);
    const size_t tail = (size_t)NS * a.NP;
    if constexpr (FUSE) {
        if (lane == 0) {
            base[tail] = (double)(t1 - t0);
            base[tail + 1] = ls * AMICA_LN2;
        }
    } else {
        __shared__ double llw[kMaxEstepWaves];
        if (lane == 0) llw[w] = ls;
        __syncthreads();
        if (threadIdx.x == 0) {
            double l = 0.0;
            for (int c = 0; c < (int)(blockDim.x >> 6); ++c) l += llw[c];
            base[tail] = (double)(t1 - t0);
            base[tail + 1] = l * AMICA_LN2;
        }
    }
}

template <int MJ, bool B64>
__global__ __launch_bounds__(512) void estep_m1_kernel(EstepArgs a) {
    extern __shared__ float tot2_all[];
    const long t0 = (long)blockIdx.x * a.chunk;
    estep_m1_body<MJ, B64, false>(a, t0, min(a.T, t0 + a.chunk), (int)blockIdx.x, nullptr, tot2_all, nullptr);
}

/* n <= 64 channels, one model, FP32 path: each wave forms b of its own samples,
 * 16 at a time, and b never goes to memory -- two of the five passes of the
 * separate unmixing and E-step (x read and b written; b and x read, g
 * written), which are bound by HBM at 4.3-5 TB/s.  W's fragments and the FP64
 * constants are in LDS, once for the workgroup's waves, which share nothing else
 * (a range of samples each).  What bounds it is issue on the SIMDs: up to 55 %
 * of the cycles the vector ALU (99 instructions a sample at m = 3), 31 % the FP64
 * MFMAs, one after the other in a wave; the next tile's x loaded ahead and wave
 * priorities by phase changed nothing.  64 ch x 1M, us, unmixing and E-step
 * together: m = 1 436 -> 355, m = 2 440 -> 332, m = 3 482 -> 400; 16 ch x 20k 35
 * -> 32; 40 ch x 5k 28 and 28.  For m > 3 the kernel needs more than 128 VGPRs,
 * and for NP > 64 W does not fit LDS: those keep the two launches. */
template <int MJ>
__global__ __launch_bounds__(1024, MJ == 1 ? 5 : 4) void estep_m1_unmix_kernel(EstepArgs a, int nranges, int nw) {
    __shared__ double wfrag[64 * 64];
    __shared__ double c64s[2 * MJ * 64];
    extern __shared__ float tot2_all[];
    /* two of W's entries a load, four loads in flight */
#pragma unroll 4
    for (int e = threadIdx.x; e < 32 * 64; e += blockDim.x) {
        const int col = e >> 5, k = 2 * (e & 31);
        const double2 v = *(const double2*)(a.Wg64 + (size_t)col * 64 + k);
        double* const f = wfrag + ((k >> 2) * 4 + (col >> 4)) * 64 + (k & 3) * 16 + (col & 15);
        f[0] = v.x;
        f[16] = v.y;
    }
    for (int e = threadIdx.x; e < 2 * MJ * 64; e += blockDim.x) {
        const int i = e & 63, k = (e >> 6) & 1, j = e >> 7;
        c64s[e] = i < a.n ? a.cst64[((size_t)(k == 0 ? kCst64Sb : kCst64Nsbmu) * MJ + j) * 64 + i]
                          : (k == 0 ? 0.0 : 1.0);
    }
    __syncthreads();
    /* waves past nw only help with the copies above */
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = blockIdx.x * nw + w;
    if (w >= nw || r >= nranges) return;
    const long t0 = (long)r * a.chunk;
    estep_m1_body<MJ, true, true>(a, t0, min(a.T, t0 + a.chunk), r, wfrag, tot2_all, c64s);
}

/* Many recordings in one launch: workgroup b runs work item b, a range of
 * samples of one recording (args[item.rec]) into that recording's partial
 * slot item.slot.  Every recording of a launch has the same NP (blockDim). */
template <int MJ, bool B64>
__global__ __launch_bounds__(512) void estep_m1_batch_kernel(const EstepArgs* __restrict__ args,
                                                             const BatchItem* __restrict__ items) {
    const BatchItem it = items[blockIdx.x];
    const EstepArgs a = args[it.rec];
    extern __shared__ float tot2_all[];
    estep_m1_body<MJ, B64, false>(a, it.t0, it.t1, it.slot, nullptr, tot2_all, nullptr);
}

/* The split launch's middle pass: per sample, the model log-likelihoods
 * L_h = (log gm_h + ldet_h + ldetS) + sum of q over all channels (the
 * channel-group sums of the first pass), their log-sum-exp (the sample's
 * log-likelihood, as updatell, kernels.cu:376-450) and the posteriors
 * v_h = exp(L_h - logsumexp) for the statistics pass.  One workgroup per
 * sample chunk (the chunks of the other passes): vsum per model and the LL
 * sum go to the tail of the chunk's partial slot, in FP64. */
__global__ __launch_bounds__(256) void estep_post_kernel(EstepArgs a) {
    __shared__ float dc2[AMICA_MAX_M];
    __shared__ double red[4][AMICA_MAX_M + 1];
    const int M = a.M, ncg = a.ncg;
    if ((int)threadIdx.x < M) {
        double c0 = a.lconst[0];
        for (int hh = 1; hh < M; ++hh) c0 = fmax(c0, a.lconst[hh]);
        dc2[threadIdx.x] = (float)((a.lconst[threadIdx.x] - c0) * 1.4426950408889634);
    }
    __syncthreads();
    const long t0 = (long)blockIdx.x * a.chunk;
    const long t1 = min(a.T, t0 + a.chunk);
    double ll = 0.0, vs[AMICA_MAX_M];
#pragma unroll
    for (int hh = 0; hh < AMICA_MAX_M; ++hh) vs[hh] = 0.0;
    for (long t = t0 + threadIdx.x; t < t1; t += blockDim.x) {
        float l[AMICA_MAX_M];
        float lmax = -3.0e38f;
#pragma unroll
        for (int hh = 0; hh < AMICA_MAX_M; ++hh) {
            if (hh < M) {
                float v = dc2[hh];
                const float* q = a.lq + ((size_t)t * M + hh) * ncg;
                for (int c = 0; c < ncg; ++c) v += q[c];
                l[hh] = v;
                lmax = fmaxf(lmax, v);
            }
        }
        float esum = 0.f;
#pragma unroll
        for (int hh = 0; hh < AMICA_MAX_M; ++hh)
            if (hh < M) esum += fast_exp2(l[hh] - lmax);
        const float r = fast_rcp(esum);
#pragma unroll
        for (int hh = 0; hh < AMICA_MAX_M; ++hh) {
            if (hh < M) {
                const float v = fast_exp2(l[hh] - lmax) * r;
                a.vq[(size_t)t * M + hh] = v;
                vs[hh] += (double)v;
                if (a.ltall) a.ltall[(size_t)hh * a.T + t] = l[hh] * (float)AMICA_LN2;
            }
        }
        ll += (double)(lmax + fast_log2(esum)) * AMICA_LN2;
    }
    /* fixed-order block sums: waves, then the 4 wave totals */
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const double lls = wave_sum_f64(ll);
    if (lane == 0) red[w][M] = lls;
#pragma unroll
    for (int hh = 0; hh < AMICA_MAX_M; ++hh) {
        if (hh < M) {
            const double v = wave_sum_f64(vs[hh]);
            if (lane == 0) red[w][hh] = v;
        }
    }
    __syncthreads();
    if ((int)threadIdx.x <= M) {
        const double tot = (red[0][threadIdx.x] + red[1][threadIdx.x]) + (red[2][threadIdx.x] + red[3][threadIdx.x]);
        const int NS = kStatsPerJ * a.mj + kStatsPerI;
        a.part[(size_t)blockIdx.x * a.pstride + (size_t)M * NS * a.NP + threadIdx.x] = tot;
    }
}

}  // namespace

void estep_split_shape(int M, int CW, int* mg, int* cwg, int* ncg, int* ngroups) {
    /* channel blocks per group: all of a model's if they fit one workgroup,
     * else the fewest groups of at most kMaxEstepWaves blocks, balanced */
    const int g = (CW + kMaxEstepWaves - 1) / kMaxEstepWaves;
    const int c = (CW + g - 1) / g;
    const int models = std::max(1, std::min(M, kMaxEstepWaves / c));
    *cwg = c;
    *ncg = g;
    *mg = models;
    *ngroups = ((M + models - 1) / models) * g;
}

int estep_configure(int MJ, size_t lds_bytes) {
    /* one attribute per kernel for the whole process: keep the largest that
     * any engine asked for (engines of other shapes launch with less) */
    static size_t granted[AMICA_MAX_MJ + 1] = {0};
    if (MJ < 1 || MJ > AMICA_MAX_MJ) return -1;
    if (lds_bytes <= granted[MJ]) return 0;
    granted[MJ] = lds_bytes;
    hipError_t r = hipSuccess;
#define AMICA_ESTEP_ATTR(J)                                                                       \
    case J:                                                                                       \
        for (const void* fn : {(const void*)estep_variant<J, true, kEstepFused, false, true, false, true>(), \
                               (const void*)estep_variant<J, true, kEstepFused, false, true>(),   \
                               (const void*)estep_variant<J, true, kEstepFused, false>(),         \
                               (const void*)estep_variant<J, false, kEstepFused, false, false, true>(), \
                               (const void*)estep_variant<J, false, kEstepFused, false>(),        \
                               (const void*)estep_variant<J, false, kEstepFused, true>(),         \
                               (const void*)estep_variant<J, true, kEstepStats, false>(),         \
                               (const void*)estep_variant<J, false, kEstepStats, false>(),        \
                               (const void*)estep_variant<J, false, kEstepStats, true>()})        \
            if (r == hipSuccess)                                                                  \
                r = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,           \
                                        (int)lds_bytes);                                          \
        if (r == hipSuccess)                                                                      \
            r = hipFuncSetAttribute((const void*)estep_m1_batch_kernel<J, false>,                \
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);  \
        if (r == hipSuccess)                                                                      \
            r = hipFuncSetAttribute((const void*)estep_m1_kernel<J, true>,                       \
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);  \
        if (r == hipSuccess)                                                                      \
            r = hipFuncSetAttribute((const void*)estep_m1_kernel<J, false>,                      \
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);  \
        break;
    switch (MJ) {
        AMICA_ESTEP_ATTR(1)
        AMICA_ESTEP_ATTR(2)
        AMICA_ESTEP_ATTR(3)
        AMICA_ESTEP_ATTR(4)
        AMICA_ESTEP_ATTR(5)
        AMICA_ESTEP_ATTR(6)
        AMICA_ESTEP_ATTR(7)
        AMICA_ESTEP_ATTR(8)
        default: return -1;
    }
#undef AMICA_ESTEP_ATTR
    if (MJ <= 3 && r == hipSuccess)
        r = hipFuncSetAttribute(MJ == 1   ? (const void*)estep_m1_unmix_kernel<1>
                                : MJ == 2 ? (const void*)estep_m1_unmix_kernel<2>
                                          : (const void*)estep_m1_unmix_kernel<3>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)estep_lds_bytes(MJ, 1024));
    return r == hipSuccess ? 0 : -1;
}

size_t estep_lds_bytes(int MJ, int threads, bool m1b64) {
    const size_t tot = (size_t)((kStatsPerJ * MJ + kStatsPerI) | 1) * threads * sizeof(float);
    /* the single-model FP32-path kernel at m = 3 also keeps its FP64
     * constants there (2 m doubles per thread after the totals) */
    return (m1b64 && MJ == 3) ? (tot + 7) / 8 * 8 + (size_t)2 * MJ * threads * sizeof(double) : tot;
}

/* Workgroups per CU that the sample ranges are cut for.  A range decides where
 * its FP32 sums round, so for the kernels that exchange posteriors it follows
 * from the shape alone -- these waves per SIMD and LDS bytes -- and not from the
 * registers a build happens to use; where fewer workgroups fit, the rest of
 * the ranges run in a second wave of equal length. */
int estep_blocks_per_cu(int MJ, bool b64, int threads, bool m1, bool split) {
    if (MJ < 1 || MJ > AMICA_MAX_MJ || threads < 64) return -1;
    if (!m1) {
        static const int fused[2][AMICA_MAX_MJ] = {{4, 4, 4, 4, 3, 3, 2, 2}, {4, 4, 4, 3, 3, 2, 2, 2}};
        static const int stats[2][AMICA_MAX_MJ] = {{5, 4, 3, 4, 3, 3, 2, 2}, {6, 4, 4, 4, 3, 3, 2, 2}};
        const int waves = 4 * (split ? stats : fused)[b64][MJ - 1];
        const size_t lds = estep_lds_bytes(MJ, threads) + (MJ <= 3 ? 832 : 576) + (b64 && MJ == 3 ? 24576 : 0);
        return (int)std::max<size_t>(1, std::min<size_t>(waves / (threads / 64), 163840 / lds));
    }
    int nb = 0;
    const size_t shm = estep_lds_bytes(MJ, threads, b64);
    hipError_t r = hipErrorInvalidValue;
#define AMICA_ESTEP_OCC(J)                                                                        \
    case J:                                                                                       \
        r = b64 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, estep_m1_kernel<J, true>,     \
                                                               threads, shm)                      \
                : hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, estep_m1_kernel<J, false>,    \
                                                               threads, shm);                     \
        break;
    switch (MJ) {
        AMICA_ESTEP_OCC(1)
        AMICA_ESTEP_OCC(2)
        AMICA_ESTEP_OCC(3)
        AMICA_ESTEP_OCC(4)
        AMICA_ESTEP_OCC(5)
        AMICA_ESTEP_OCC(6)
        AMICA_ESTEP_OCC(7)
        AMICA_ESTEP_OCC(8)
        default: return -1;
    }
#undef AMICA_ESTEP_OCC
    return r == hipSuccess ? nb : -1;
}

static int launch_estep_split(const EstepArgs& a, int MJ, int nblocks, hipStream_t st) {
    int mg = 0, cwg = 0, ncg = 0, ngroups = 0;
    estep_split_shape(a.M, a.CW, &mg, &cwg, &ncg, &ngroups);
    if (a.mg != mg || a.cwg != cwg || a.ncg != ncg || !a.lq || !a.vq || a.mj != MJ || (a.chunk % 8) != 0)
        return -1;
    const dim3 grid(nblocks, ngroups), block(64 * mg * cwg);
    const size_t shm = estep_lds_bytes(MJ, (int)block.x);
    const bool b64 = a.b64 != nullptr;
#define AMICA_ESTEP_SPLIT(J)                                                                          \
    case J:                                                                                           \
        if (b64) hipLaunchKernelGGL((estep_variant<J, true, kEstepLsum, false>()), grid, block, 0, st, a); \
        else hipLaunchKernelGGL((estep_variant<J, false, kEstepLsum, false>()), grid, block, 0, st, a); \
        hipLaunchKernelGGL(estep_post_kernel, dim3(nblocks), dim3(256), 0, st, a);                   \
        if (b64) hipLaunchKernelGGL((estep_variant<J, true, kEstepStats, false>()), grid, block, shm, st, a); \
        else if (a.g_bf16) hipLaunchKernelGGL((estep_variant<J, false, kEstepStats, true>()), grid, block, shm, st, a); \
        else hipLaunchKernelGGL((estep_variant<J, false, kEstepStats, false>()), grid, block, shm, st, a); \
        break;
    switch (MJ) {
        AMICA_ESTEP_SPLIT(1)
        AMICA_ESTEP_SPLIT(2)
        AMICA_ESTEP_SPLIT(3)
        AMICA_ESTEP_SPLIT(4)
        AMICA_ESTEP_SPLIT(5)
        AMICA_ESTEP_SPLIT(6)
        AMICA_ESTEP_SPLIT(7)
        AMICA_ESTEP_SPLIT(8)
        default: return -1;
    }
#undef AMICA_ESTEP_SPLIT
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

/* where it is faster than unmixing and E-step apart (estep_m1_unmix_kernel) */
bool estep_unmixes(int M, int NP, int MJ) { return M == 1 && NP == 64 && MJ <= 3; }

/* Waves per workgroup of estep_m1_unmix_kernel: a CU's share of the ranges up to
 * 16, and where it is more (m = 1: five waves per SIMD) half of it, an even
 * number, for two workgroups */
static int estep_unmix_waves(int nranges, int cus) {
    const int per = std::max(1, (nranges + cus - 1) / cus);
    return per <= 16 ? per : std::min(16, (per + 3) / 4 * 2);
}

int launch_estep_m1_batch(const EstepArgs* args, const BatchItem* items, int nitems, int MJ, int NP,
                          hipStream_t st) {
    if (nitems < 1 || NP % 64 || NP > 64 * kMaxEstepWaves) return -1;
    const dim3 grid(nitems), block(NP);
    const size_t shm = estep_lds_bytes(MJ, NP);
#define AMICA_ESTEP_BATCH(J)                                                                        \
    case J:                                                                                         \
        hipLaunchKernelGGL((estep_m1_batch_kernel<J, false>), grid, block, shm, st, args, items); \
        break;
    switch (MJ) {
        AMICA_ESTEP_BATCH(1)
        AMICA_ESTEP_BATCH(2)
        AMICA_ESTEP_BATCH(3)
        AMICA_ESTEP_BATCH(4)
        AMICA_ESTEP_BATCH(5)
        AMICA_ESTEP_BATCH(6)
        AMICA_ESTEP_BATCH(7)
        AMICA_ESTEP_BATCH(8)
        default: return -1;
    }
#undef AMICA_ESTEP_BATCH
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_estep(const EstepArgs& a, int MJ, int nblocks, int cus, hipStream_t st) {
    if (a.split) return launch_estep_split(a, MJ, nblocks, st);
    if (a.M * a.CW > kMaxEstepWaves || a.M > 8 || (a.chunk % 8) != 0) return -1;
    /* byte offsets of the rows a workgroup reads (its chunk and the next
     * tile past it) must fit the 31-bit scalar offsets of its buffer loads */
    if ((a.chunk + kEstepRowPad) * (long)a.ldb * 8 >= (1L << 31)) return -1;
    dim3 grid(nblocks), block(64 * a.M * a.CW);
    const bool b64 = a.b64 != nullptr;
    const bool m1 = a.M == 1 && a.ltall == nullptr;
    const size_t shm = estep_lds_bytes(MJ, (int)block.x, m1 && b64);
    if (a.Wg64 && m1 && estep_unmixes(a.M, a.NP, MJ)) {
        const int nw = estep_unmix_waves(nblocks, cus);
        const dim3 ug((nblocks + nw - 1) / nw), ub(64 * std::max(nw, 4));
        const size_t us = estep_lds_bytes(MJ, (int)ub.x);
        if (MJ == 1) hipLaunchKernelGGL((estep_m1_unmix_kernel<1>), ug, ub, us, st, a, nblocks, nw);
        else if (MJ == 2) hipLaunchKernelGGL((estep_m1_unmix_kernel<2>), ug, ub, us, st, a, nblocks, nw);
        else hipLaunchKernelGGL((estep_m1_unmix_kernel<3>), ug, ub, us, st, a, nblocks, nw);
        return hipGetLastError() == hipSuccess ? 0 : -1;
    }
    const int waves = (int)block.x / 64;
    const bool small = waves <= kSmallWaves, mid = waves > 4 && waves < 8;
#define AMICA_ESTEP_CASE(J)                                                                   \
    case J:                                                                                   \
        if (m1) {                                                                             \
            if (b64) hipLaunchKernelGGL((estep_m1_kernel<J, true>), grid, block, shm, st, a); \
            else hipLaunchKernelGGL((estep_m1_kernel<J, false>), grid, block, shm, st, a);    \
        } else {                                                                              \
            hipLaunchKernelGGL((b64 && waves == 2 ? estep_variant<J, true, kEstepFused, false, true, false, true>() \
                                : b64 && small ? estep_variant<J, true, kEstepFused, false, true>()           \
                                : b64        ? estep_variant<J, true, kEstepFused, false>()                   \
                                : a.g_bf16   ? estep_variant<J, false, kEstepFused, true>()                   \
                                : mid        ? estep_variant<J, false, kEstepFused, false, false, true>()     \
                                             : estep_variant<J, false, kEstepFused, false>()),                \
                               grid, block, shm, st, a);                                      \
        }                                                                                     \
        break;
    switch (MJ) {
        AMICA_ESTEP_CASE(1)
        AMICA_ESTEP_CASE(2)
        AMICA_ESTEP_CASE(3)
        AMICA_ESTEP_CASE(4)
        AMICA_ESTEP_CASE(5)
        AMICA_ESTEP_CASE(6)
        AMICA_ESTEP_CASE(7)
        AMICA_ESTEP_CASE(8)
        default: return -1;
    }
#undef AMICA_ESTEP_CASE
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace amica
