/*
 * sphere.hip -- preprocessing on the GPU (fraimondo/cudamica
 * src/preprocess.cu:31-420, which uses cublasDsyrk + magma_dsyevd_gpu +
 * magma_dgesv_gpu) and the final output transform (src/amica.cu:2564-2668).
 *
 *   mean     = sum_t x_t / T                      FP64 partial sums per chunk
 *   C        = sum_t (x_t - mean)(x_t - mean)^T / T   FP64 tiles
 *   S        = 2 C^-1/2 (do_sphere 1)             Newton-Schulz products (FP64 MFMA), or where
 *              they do not converge (condition number past ~1e9, singular C)
 *              V diag(2/sqrt(d)) V^T from a parallel cyclic Jacobi C = V diag(d) V^T
 *              diag(1/std) (do_sphere 2), I otherwise
 *   ldetS    = -log|det S|
 *   x_white  = S (x - mean), stored float32 [T][NP] (+ bf16 copy)
 */
#include <algorithm>
#include <cmath>

#include "common.h"
#include "engine_internal.h"

namespace amica {

namespace {

/* per-chunk FP64 column sums of x (T x n float32), 256 columns per
 * blockIdx.y: the workgroup's threads cover as many whole rows at once as fit
 * (consecutive addresses), kRowUnroll passes of loads in flight, and the rows'
 * sums meet in LDS in a fixed order.  Bound by the read of x: 0.13 ms at
 * 128 ch x 1M, 4.0 TB/s (0.82 ms with one thread per column, which left half
 * the workgroup idle and one load in flight). */
constexpr int kRowUnroll = 8;

__global__ __launch_bounds__(256) void colsum_kernel(const float* __restrict__ x, long T, int n,
                                                     long chunk, double* __restrict__ part) {
    __shared__ double red[256];
    const long ts = (long)blockIdx.x * chunk, te = min(T, ts + chunk);
    const int c0 = blockIdx.y * 256, cols = min(256, n - c0), rows = 256 / cols;
    const int tid = threadIdx.x, r = tid / cols, i = c0 + tid - r * cols;
    double s = 0.0;
    if (r < rows) {
        long t = ts + r;
        for (; t + (long)(kRowUnroll - 1) * rows < te; t += (long)kRowUnroll * rows) {
            float v[kRowUnroll];
#pragma unroll
            for (int u = 0; u < kRowUnroll; ++u) v[u] = x[(size_t)(t + (long)u * rows) * n + i];
#pragma unroll
            for (int u = 0; u < kRowUnroll; ++u) s += (double)v[u];
        }
        for (; t < te; t += rows) s += (double)x[(size_t)t * n + i];
    }
    red[tid] = s;
    __syncthreads();
    if (tid < cols) {
        for (int q = 1; q < rows; ++q) s += red[q * cols + tid];
        part[(size_t)blockIdx.x * n + i] = s;
    }
}

/* Fixed-order totals of per-chunk partials: 64 entries (lanes) per workgroup,
 * wave w takes the chunks w, w + 16, ..., the waves' sums are added in order. */
__device__ __forceinline__ double chunk_total(const double* __restrict__ part, int nchunks, size_t stride,
                                              size_t e, bool valid) {
    __shared__ double red[16][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    double s = 0.0;
    if (valid) {
#pragma unroll 4
        for (int c = w; c < nchunks; c += 16) s += part[(size_t)c * stride + e];
    }
    red[w][lane] = s;
    __syncthreads();
    double t = 0.0;
    if (w == 0)
        for (int q = 0; q < 16; ++q) t += red[q][lane];
    return t;
}

__global__ __launch_bounds__(1024) void finish_mean_kernel(const double* __restrict__ part, int nchunks, int n,
                                                           long T, double* __restrict__ mean) {
    const int i = blockIdx.x * 64 + (threadIdx.x & 63);
    const double s = chunk_total(part, nchunks, n, i, i < n);
    if (threadIdx.x < 64 && i < n) mean[i] = s / (double)T;
}

/* Upper triangle of the covariance over one chunk of samples: blockIdx.y is
 * the pair (bi <= bk) of 16 TI-channel blocks, each of the four waves takes
 * every fourth group of kU 4-sample steps, TI x TI FP64 MFMA tiles; their sums
 * meet in LDS in wave order.  Fragments are loaded straight from x (lane
 * (i, k) = channel l % 16, sample l / 16: 64-byte runs), kU steps ahead of
 * their use, and centred in registers, so that nothing but the sums goes
 * through LDS (the loads in flight spill 36 bytes a lane at TI = 2, 24 at 4).  Bound by the FP64 MFMA rate (64 cycles per 1024 FMAs), and
 * only one triangle is formed: 0.57 ms at 128 ch x 1M, 1.86 ms at 256 ch (44
 * TFLOP/s of 73; 1.31 ms for both triangles by FMAs from LDS at 128 ch). */
template <int TI>
__global__ __launch_bounds__(256, 2) void cov_kernel(const float* __restrict__ x,
                                                  const double* __restrict__ mean, long T, int n,
                                                  long chunk, int nblk, double* __restrict__ part) {
    constexpr int W = 16 * TI, kU = TI == 4 ? 2 : 4;
    __shared__ double sum[TI * TI][256];
    int bi = 0, bk = (int)blockIdx.y;
    while (bk >= nblk - bi) { bk -= nblk - bi; ++bi; }
    bk += bi;
    const int tid = threadIdx.x, lane = tid & 63, l15 = lane & 15, kq = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool diag = bi == bk;                          /* block-uniform */
    const long ts = (long)blockIdx.x * chunk, te = min(T, ts + chunk);
    int ci[TI], ck[TI];
    double mi[TI], mk[TI];
    bool vi[TI], vk[TI];
#pragma unroll
    for (int p = 0; p < TI; ++p) {
        const int i = bi * W + 16 * p + l15, k = bk * W + 16 * p + l15;
        vi[p] = i < n;
        vk[p] = k < n;
        ci[p] = vi[p] ? i : n - 1;
        ck[p] = vk[p] ? k : n - 1;
        mi[p] = mean[ci[p]];
        mk[p] = mean[ck[p]];
    }
    f64x4 acc[TI][TI];
#pragma unroll
    for (int p = 0; p < TI; ++p)
#pragma unroll
        for (int q = 0; q < TI; ++q) acc[p][q] = (f64x4){0.0, 0.0, 0.0, 0.0};
    float fa[kU][TI], fb[kU][TI];
    auto load = [&](long t0) {
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const long t = t0 + 4 * u + kq;
            const float* row = x + (size_t)(t < te ? t : te - 1) * n;
#pragma unroll
            for (int p = 0; p < TI; ++p) {
                fa[u][p] = row[ci[p]];
                if (!diag) fb[u][p] = row[ck[p]];
            }
        }
    };
    const long step = 4 * 4 * kU;
    long t0 = ts + (long)w * 4 * kU;
    if (t0 < te) load(t0);
    for (; t0 < te; t0 += step) {
        double a[kU][TI], b[kU][TI];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const bool ok = t0 + 4 * u + kq < te;
#pragma unroll
            for (int p = 0; p < TI; ++p) {
                a[u][p] = ok && vi[p] ? (double)fa[u][p] - mi[p] : 0.0;
                b[u][p] = diag ? a[u][p] : (ok && vk[p] ? (double)fb[u][p] - mk[p] : 0.0);
            }
        }
        if (t0 + step < te) load(t0 + step);
#pragma unroll
        for (int u = 0; u < kU; ++u)
#pragma unroll
            for (int p = 0; p < TI; ++p)
#pragma unroll
                for (int q = 0; q < TI; ++q)
                    acc[p][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u][p], b[u][q], acc[p][q], 0, 0, 0);
    }
    /* register r of lane l: row l / 16 + 4 r, column l % 16 */
    for (int v = 0; v < 4; ++v) {
        if (v == w) {
#pragma unroll
            for (int p = 0; p < TI; ++p)
#pragma unroll
                for (int q = 0; q < TI; ++q)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        double* s = &sum[p * TI + q][l15 * 16 + kq + 4 * r];
                        *s = v == 0 ? acc[p][q][r] : *s + acc[p][q][r];
                    }
        }
        __syncthreads();
    }
    double* out = part + ((size_t)blockIdx.x * gridDim.y + blockIdx.y) * (W * W);
#pragma unroll
    for (int t = 0; t < TI * TI; ++t) out[t * 256 + tid] = sum[t][tid];
}

/* C from the chunks' block pairs, mirrored: entry e = (pair, tile, row and
 * column) of the layout above */
__global__ __launch_bounds__(1024) void finish_cov_kernel(const double* __restrict__ part, int nchunks, int n,
                                                          int TI, int nblk, int npairs, long T,
                                                          double* __restrict__ C) {
    const int W = 16 * TI;
    const size_t len = (size_t)npairs * W * W, e = (size_t)blockIdx.x * 64 + (threadIdx.x & 63);
    const double s = chunk_total(part, nchunks, len, e, e < len);
    if (threadIdx.x >= 64 || e >= len) return;
    int bk = (int)(e / (W * W)), bi = 0;
    const int f = (int)(e % (W * W));
    while (bk >= nblk - bi) { bk -= nblk - bi; ++bi; }
    bk += bi;
    const int t = f >> 8, g = f & 255;
    const int i = bi * W + (t / TI) * 16 + (g & 15), k = bk * W + (t % TI) * 16 + (g >> 4);
    if (i >= n || k >= n) return;
    C[i + (size_t)k * n] = s / (double)T;
    if (bi != bk) C[k + (size_t)i * n] = s / (double)T;
}

/* Parallel cyclic Jacobi (Brent-Luk round-robin ordering): each round
 * rotates N/2 disjoint (p, q) pairs at once.  A (n x n, overwritten) and V
 * are column-major in global memory; one workgroup. */
__global__ __launch_bounds__(256) void eigh_kernel(double* __restrict__ A, double* __restrict__ V,
                                                   double* __restrict__ d, int n) {
    __shared__ double cs[512], sn[512];
    __shared__ int pp[512], qq[512];
    __shared__ double red[8];
    __shared__ int done;
    const int tid = threadIdx.x;
    const int N = n + (n & 1);
    const int half = N / 2;
    for (long q = tid; q < (long)n * n; q += blockDim.x) V[q] = ((q % n) == (q / n)) ? 1.0 : 0.0;
    __syncthreads();
    for (int sweep = 0; sweep < 40; ++sweep) {
        /* convergence: off-diagonal Frobenius norm relative to the diagonal */
        double off = 0.0, dia = 0.0;
        for (long q = tid; q < (long)n * n; q += blockDim.x) {
            const double v = A[q];
            if ((q % n) == (q / n)) dia += v * v; else off += v * v;
        }
        off = wave_sum_f64(off);
        dia = wave_sum_f64(dia);
        if ((tid & 63) == 0) { red[tid >> 6] = off; red[4 + (tid >> 6)] = dia; }
        __syncthreads();
        if (tid == 0) {
            double o = 0.0, dd = 0.0;
            for (int w = 0; w < (int)(blockDim.x >> 6); ++w) { o += red[w]; dd += red[4 + w]; }
            done = (o <= 1e-30 * dd || o == 0.0) ? 1 : 0;
        }
        __syncthreads();
        if (done) break;
        for (int r = 0; r < N - 1; ++r) {
            for (int k = tid; k < half; k += blockDim.x) {
                /* circle method: position 0 fixed, the others rotate */
                const int a0 = (k == 0) ? 0 : ((k - 1 + r) % (N - 1)) + 1;
                const int b0 = ((N - 1 - k - 1 + r) % (N - 1)) + 1;
                int p = min(a0, b0), q = max(a0, b0);
                double c = 1.0, s = 0.0;
                if (q < n) {
                    const double apq = A[p + (long)q * n];
                    if (apq != 0.0) {
                        const double app = A[p + (long)p * n], aqq = A[q + (long)q * n];
                        const double th = (aqq - app) / (2.0 * apq);
                        const double t = (th >= 0 ? 1.0 : -1.0) / (fabs(th) + sqrt(th * th + 1.0));
                        c = 1.0 / sqrt(t * t + 1.0);
                        s = t * c;
                    }
                } else {
                    q = p;   /* pair with the padding index: identity */
                }
                cs[k] = c; sn[k] = s; pp[k] = p; qq[k] = q;
            }
            __syncthreads();
            /* A <- A J (columns p, q) and V <- V J */
            for (long e = tid; e < (long)half * n; e += blockDim.x) {
                const int k = (int)(e / n), i = (int)(e % n);
                const int p = pp[k], q = qq[k];
                if (p == q) continue;
                const double c = cs[k], s = sn[k];
                const double ap = A[i + (long)p * n], aq = A[i + (long)q * n];
                A[i + (long)p * n] = c * ap - s * aq;
                A[i + (long)q * n] = s * ap + c * aq;
                const double vp = V[i + (long)p * n], vq = V[i + (long)q * n];
                V[i + (long)p * n] = c * vp - s * vq;
                V[i + (long)q * n] = s * vp + c * vq;
            }
            __syncthreads();
            /* A <- J^T A (rows p, q) */
            for (long e = tid; e < (long)half * n; e += blockDim.x) {
                const int k = (int)(e / n), j = (int)(e % n);
                const int p = pp[k], q = qq[k];
                if (p == q) continue;
                const double c = cs[k], s = sn[k];
                const double ap = A[p + (long)j * n], aq = A[q + (long)j * n];
                A[p + (long)j * n] = c * ap - s * aq;
                A[q + (long)j * n] = s * ap + c * aq;
            }
            __syncthreads();
        }
    }
    for (int i = tid; i < n; i += blockDim.x) d[i] = A[i + (long)i * n];
}

/* S = 2 C^-1/2 without an eigendecomposition: the coupled Newton-Schulz
 * iteration Y -> C^1/2, Z -> C^-1/2 from Y = C / |C|_F, Z = I,
 *   R = r/2 (3 I - r^2 Z Y),   Y <- Y R,   Z <- R Z,
 * with r chosen for the interval [l, 1] that the eigenvalues of (Z Y)^1/2 are
 * taken to lie in (Chen and Chow's scaling: r = sqrt(3 / (1 + l + l^2)), then
 * l <- r l (3 - r^2 l^2) / 2); eigenvalues below l only take more steps.  In
 * this order of the factors the iteration is stable (with Z Y formed as
 * Z Y^T it is not: the skew part of the rounding errors grows).  Against
 * 80-bit results its error is 0.2 .. 0.8 of the Jacobi eigensolver's for
 * condition numbers of C from 1e2 to 1e8.  Bound by the latency of its
 * dependent products: 14 to 19 iterations of two 5 us launches (7 + 11 us at
 * 256 channels) replace ~9 sweeps of n - 1 barrier-separated rounds in one
 * workgroup: 46 ms -> 0.2 ms at 128 channels, 356 ms -> 0.5 ms at 260. */

/* scal[0] = |C|_F (one workgroup) and the residual slots cleared */
constexpr int kNsSlots = 32;

__global__ __launch_bounds__(1024) void ns_norm_kernel(const double* __restrict__ C, int n,
                                                       double* __restrict__ scal,
                                                       unsigned long long* __restrict__ rmax) {
    __shared__ double red[16];
    const int tid = threadIdx.x;
    double s = 0.0;
    for (long q = tid; q < (long)n * n; q += blockDim.x) s += C[q] * C[q];
    s = wave_sum_f64(s);
    if ((tid & 63) == 0) red[tid >> 6] = s;
    if (tid < kNsSlots) rmax[tid] = 0;
    __syncthreads();
    if (tid == 0) {
        double t = 0.0;
        for (int w = 0; w < 16; ++w) t += red[w];
        scal[0] = sqrt(t);
    }
}

__global__ __launch_bounds__(256) void ns_init_kernel(const double* __restrict__ C, int n,
                                                      const double* __restrict__ scal,
                                                      double* __restrict__ Y, double* __restrict__ Z) {
    const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (long)n * n) return;
    Y[q] = C[q] / scal[0];
    Z[q] = (q % n) == (q / n) ? 1.0 : 0.0;
}

/* One 16 TI x 16 TI tile of A B per workgroup (column-major n x n, FP64 MFMA):
 * the four waves take every fourth 4-step of the inner index and add their
 * tiles through LDS in wave order.  Loads go straight to the fragments, kU
 * k-steps of them in flight: the matrices sit in L2 and each is read n / 16
 * TI times.  blockIdx.z 0: A0 B0 -> out0, 1: A1 B1 -> out1.  RESID: out0
 * receives rho/2 (3 I - rho^2 A B) instead, and *rmax the largest |I - A B|
 * (as the bits of a non-negative double, which order like it; NaN above all). */
template <int TI, bool RESID>
__global__ __launch_bounds__(256) void ns_product_kernel(const double* __restrict__ A0, const double* __restrict__ B0,
                                                         double* __restrict__ out0,
                                                         const double* __restrict__ A1, const double* __restrict__ B1,
                                                         double* __restrict__ out1, int n, double rho,
                                                         unsigned long long* __restrict__ rmax) {
    constexpr int kU = 4;
    __shared__ double part[4][TI * TI][256];
    const double* A = blockIdx.z ? A1 : A0;
    const double* B = blockIdx.z ? B1 : B0;
    double* out = blockIdx.z ? out1 : out0;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int i0 = blockIdx.x * 16 * TI, j0 = blockIdx.y * 16 * TI;
    const int l15 = lane & 15, kq = lane >> 4;
    f64x4 acc[TI][TI];
#pragma unroll
    for (int p = 0; p < TI; ++p)
#pragma unroll
        for (int q = 0; q < TI; ++q) acc[p][q] = (f64x4){0.0, 0.0, 0.0, 0.0};
    const int steps = (n + 3) / 4;
    for (int s0 = w; s0 < steps; s0 += 4 * kU) {
        double a[kU][TI], b[kU][TI];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int k = (s0 + 4 * u) * 4 + kq;
#pragma unroll
            for (int p = 0; p < TI; ++p) {
                const int i = i0 + 16 * p + l15, j = j0 + 16 * p + l15;
                a[u][p] = (k < n && i < n) ? A[i + (size_t)k * n] : 0.0;
                b[u][p] = (k < n && j < n) ? B[k + (size_t)j * n] : 0.0;
            }
        }
#pragma unroll
        for (int u = 0; u < kU; ++u)
#pragma unroll
            for (int p = 0; p < TI; ++p)
#pragma unroll
                for (int q = 0; q < TI; ++q)
                    acc[p][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u][p], b[u][q], acc[p][q], 0, 0, 0);
    }
    /* D: register r of lane l holds row l / 16 + 4 r, column l % 16 */
#pragma unroll
    for (int p = 0; p < TI; ++p)
#pragma unroll
        for (int q = 0; q < TI; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) part[w][p * TI + q][l15 * 16 + kq + 4 * r] = acc[p][q][r];
    __syncthreads();
    double worst = 0.0;
#pragma unroll
    for (int t = 0; t < TI * TI; ++t) {
        double v = 0.0;
#pragma unroll
        for (int q = 0; q < 4; ++q) v += part[q][t][tid];
        const int i = i0 + (t / TI) * 16 + (tid & 15), j = j0 + (t % TI) * 16 + (tid >> 4);
        if (i >= n || j >= n) continue;
        if constexpr (RESID) {
            const double one = i == j ? 1.0 : 0.0;
            const double e = fabs(one - v);
            worst = e > worst || e != e ? e : worst;    /* NaN stays */
            v = 0.5 * rho * (3.0 * one - rho * rho * v);
        }
        out[i + (size_t)j * n] = v;
    }
    if constexpr (RESID) {
        unsigned long long bits = __builtin_bit_cast(unsigned long long, worst);
        for (int off = 32; off >= 1; off >>= 1) {
            const unsigned long long o = __shfl_xor(bits, off, 64);
            bits = o > bits ? o : bits;
        }
        if (lane == 0) atomicMax(rmax, bits);
    }
}

/* S = 2 Z / sqrt(|C|_F), its two halves averaged */
__global__ __launch_bounds__(256) void ns_sphere_kernel(const double* __restrict__ Z, int n,
                                                        const double* __restrict__ scal,
                                                        double* __restrict__ S) {
    const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (long)n * n) return;
    const int i = (int)(q % n), k = (int)(q / n);
    S[q] = (Z[q] + Z[k + (size_t)i * n]) / sqrt(scal[0]);
}

/* S from the eigen-decomposition (do_sphere 1), ldetS = -log|det S|. */
__global__ __launch_bounds__(256) void sphere_from_eig_kernel(const double* __restrict__ V,
                                                              const double* __restrict__ d, int n,
                                                              double* __restrict__ S,
                                                              double* __restrict__ ldetS) {
    for (long q = threadIdx.x; q < (long)n * n; q += blockDim.x) {
        const int i = (int)(q % n), k = (int)(q / n);
        double s = 0.0;
        for (int j = 0; j < n; ++j) s += V[i + (long)j * n] * (2.0 / sqrt(d[j])) * V[k + (long)j * n];
        S[q] = s;
    }
    if (threadIdx.x == 0) {
        double l = 0.0;
        for (int j = 0; j < n; ++j) l += log(2.0 / sqrt(d[j]));
        *ldetS = -l;
    }
}

/* per-chunk FP64 sums of (x - mean) and (x - mean)^2 for do_sphere 2 */
__global__ __launch_bounds__(256) void var_kernel(const float* __restrict__ x,
                                                  const double* __restrict__ mean, long T, int n,
                                                  long chunk, double* __restrict__ part) {
    const long ts = (long)blockIdx.x * chunk, te = min(T, ts + chunk);
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        double s1 = 0.0, s2 = 0.0;
        for (long t = ts; t < te; ++t) {
            const double v = (double)x[(size_t)t * n + i] - mean[i];
            s1 += v;
            s2 += v * v;
        }
        part[(size_t)blockIdx.x * 2 * n + i] = s1;
        part[(size_t)blockIdx.x * 2 * n + n + i] = s2;
    }
}

/* do_sphere 2: S = diag(1/sqrt(var)) with the unbiased variance of the
 * centred data (getvariance, kernels.cu:148-161); otherwise S = I. */
__global__ __launch_bounds__(256) void sphere_diag_kernel(const double* __restrict__ part,
                                                          int nchunks, int n, long T, int do_var,
                                                          double* __restrict__ S,
                                                          double* __restrict__ ldetS) {
    __shared__ double lsum[256];
    double acc = 0.0;
    for (long q = threadIdx.x; q < (long)n * n; q += blockDim.x) S[q] = 0.0;
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        double sii = 1.0;
        if (do_var) {
            double s1 = 0.0, s2 = 0.0;
            for (int c = 0; c < nchunks; ++c) {
                s1 += part[(size_t)c * 2 * n + i];
                s2 += part[(size_t)c * 2 * n + n + i];
            }
            const double m2 = s2 - s1 * s1 / (double)T;
            sii = 1.0 / sqrt(m2 / (double)(T - 1));
        }
        S[i + (long)i * n] = sii;
        acc += log(fabs(sii));
    }
    lsum[threadIdx.x] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double l = 0.0;
        for (int k = 0; k < (int)blockDim.x; ++k) l += lsum[k];
        *ldetS = -l;
    }
}

/* x_white[t][i] = sum_k S[i][k] (x[t][k] - mean[k]) in FP64, stored float32
 * with the channel dimension padded to NP (zeros), plus optional split bf16
 * copies: xbf[0 .. T NP) = bf16(x), xbf[T NP .. 2 T NP) = bf16(x - bf16(x)). */
__device__ __forceinline__ void store_split_bf16(uint16_t* xbf, size_t lo_ofs, size_t e, float f) {
    const uint16_t hi = f32_to_bf16_bits(f);
    xbf[e] = hi;
    xbf[lo_ofs + e] = f32_to_bf16_bits(f - bf16_bits_to_f32(hi));
}

/* A workgroup takes 16 RT WR samples x all channels: x is staged in LDS as it
 * is (float32, rows of stride = 4 mod 64 words: the 64 lanes of an A fragment
 * hit 64 banks), centred in FP64 as the fragments are read, and multiplied by
 * S from L2 on the FP64 MFMA units; wave (wr, wc) forms the 16 RT samples wr x
 * the 64-channel groups wc, wc + WC, ...  A wave's results pass through its
 * own LDS tile of 16 samples so that every copy -- float32, split bf16, bf16
 * packed by 8 samples -- leaves in 16-byte stores and the packed copy needs no
 * pass of its own.  Bound by the FP64 MFMA rate (2 n per value) and its
 * stores: 1.12 ms at 128 ch x 1M, 3.0 ms at 256 ch (44 TFLOP/s; 7.6 and 27 ms
 * with one thread per value, S from L2, and 0.18 ms more for the packing). */
struct WhitenArgs {
    const float* x;
    const double* mean;
    const double* S;
    long T;
    int n, NP, WR, WC;
    float* xw;
    double* xw64;
    uint16_t* xbf;
    uint16_t* x8;
};

constexpr int kWhitenRow = 68;                 /* floats per row of a wave's LDS tile */
constexpr int kWhitenRT = 2;                   /* 16-sample tiles per wave: 4 leave one workgroup per CU */

__global__ __launch_bounds__(512) void whiten_kernel(WhitenArgs a) {
    constexpr int RT = kWhitenRT;
    extern __shared__ __align__(16) float wlds[];
    const int n = a.n, NP = a.NP, stride = NP + 4, K4 = (n + 3) / 4;
    const int tid = threadIdx.x, lane = tid & 63, l15 = lane & 15, kq = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), nw = blockDim.x >> 6;
    const int wr = w / a.WC, wc = w - wr * a.WC;
    const int TS = 16 * RT * a.WR;
    float* xs = wlds;                                              /* [TS][stride] */
    double* ms = (double*)(wlds + (size_t)TS * stride);            /* [NP] */
    float* tile = (float*)(ms + NP) + w * 16 * kWhitenRow;         /* [16][kWhitenRow] */
    const long t0 = (long)blockIdx.x * TS;
    for (int s = w; s < TS; s += nw)
        for (int k = lane; k < 4 * K4; k += 64)
            xs[s * stride + k] = (t0 + s < a.T && k < n) ? a.x[(size_t)(t0 + s) * n + k] : 0.f;
    for (int k = tid; k < NP; k += blockDim.x) ms[k] = k < n ? a.mean[k] : 0.0;
    __syncthreads();
    const long tw = t0 + (long)wr * 16 * RT;
    const float* xa = xs + (wr * 16 * RT + l15) * stride + kq;
    for (int cg = wc; cg < NP / 64; cg += a.WC) {
        f64x4 acc[RT][4];
#pragma unroll
        for (int p = 0; p < RT; ++p)
#pragma unroll
            for (int q = 0; q < 4; ++q) acc[p][q] = (f64x4){0.0, 0.0, 0.0, 0.0};
        /* past the last row and column the loads repeat it: x - mean is 0
         * there, and the padding channels are cleared on the way out */
        const double* Sc[4];
        bool vc[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int c = cg * 64 + 16 * q + l15;
            vc[q] = c < n;
            Sc[q] = a.S + min(c, n - 1);
        }
        double bn[4];
        auto loadS = [&](int s) {
            const size_t k = (size_t)min(4 * s + kq, n - 1) * n;
#pragma unroll
            for (int q = 0; q < 4; ++q) bn[q] = Sc[q][k];
        };
        loadS(0);
#pragma unroll 2
        for (int s = 0; s < K4; ++s) {
            double bc[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) bc[q] = bn[q];
            loadS(s + 1);                      /* past the end: the last row again */
            const double mk = ms[4 * s + kq];
#pragma unroll
            for (int p = 0; p < RT; ++p) {
                const double av = (double)xa[p * 16 * stride + 4 * s] - mk;
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    acc[p][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bc[q], acc[p][q], 0, 0, 0);
            }
        }
        /* register r of lane l: sample l / 16 + 4 r, channel l % 16 */
#pragma unroll
        for (int p = 0; p < RT; ++p) {
            const long tp = tw + 16 * p;
            if (tp >= a.T) continue;                               /* wave-uniform */
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int s = kq + 4 * r;
                    const double v = vc[q] ? acc[p][q][r] : 0.0;
                    if (a.xw64 && tp + s < a.T)
                        a.xw64[(size_t)(tp + s) * NP + cg * 64 + 16 * q + l15] = v;
                    tile[s * kWhitenRow + 16 * q + l15] = tp + s < a.T ? (float)v : 0.f;
                }
            __builtin_amdgcn_wave_barrier();
            {
                const int s = lane >> 2, c = (lane & 3) * 16;      /* 16 channels of one sample */
                const float4* src = (const float4*)(tile + s * kWhitenRow + c);
                if (tp + s < a.T) {
                    float4* dst = (float4*)(a.xw + (size_t)(tp + s) * NP + cg * 64 + c);
                    float f[16];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const float4 v = src[u];
                        dst[u] = v;
                        f[4 * u] = v.x; f[4 * u + 1] = v.y; f[4 * u + 2] = v.z; f[4 * u + 3] = v.w;
                    }
                    if (a.xbf) {
                        __align__(16) uint16_t hi[16], lo[16];
#pragma unroll
                        for (int u = 0; u < 16; ++u) {
                            hi[u] = f32_to_bf16_bits(f[u]);
                            lo[u] = f32_to_bf16_bits(f[u] - bf16_bits_to_f32(hi[u]));
                        }
                        const size_t e = (size_t)(tp + s) * NP + cg * 64 + c;
                        uint4* dh = (uint4*)(a.xbf + e);
                        uint4* dl = (uint4*)(a.xbf + (size_t)a.T * NP + e);
                        dh[0] = ((const uint4*)hi)[0]; dh[1] = ((const uint4*)hi)[1];
                        dl[0] = ((const uint4*)lo)[0]; dl[1] = ((const uint4*)lo)[1];
                    }
                }
            }
            if (a.x8) {                                            /* lane = channel */
#pragma unroll
                for (int gr = 0; gr < 2; ++gr) {
                    if (tp + 8 * gr >= a.T) continue;              /* wave-uniform */
                    __align__(16) uint16_t h[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) h[u] = f32_to_bf16_bits(tile[(8 * gr + u) * kWhitenRow + lane]);
                    *(uint4*)(a.x8 + ((size_t)((tp >> 3) + gr) * NP + cg * 64 + lane) * 8) = *(const uint4*)h;
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
}

__global__ void white_from_f64_kernel(const double* __restrict__ xin, long T, int n, int NP,
                                      float* __restrict__ xw, double* __restrict__ xw64,
                                      uint16_t* __restrict__ xbf) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)T * NP) return;
    const long t = (long)(e / NP);
    const int i = (int)(e % NP);
    const double d = (i < n) ? xin[(size_t)t * n + i] : 0.0;
    const float f = (float)d;
    xw[e] = f;
    if (xw64) xw64[e] = d;
    if (xbf) store_split_bf16(xbf, (size_t)T * NP, e, f);
}

/* FP8 storage of the whitened data (per-channel scales s_i = max_t |x_ti| /
 * 448, the largest finite e4m3 value): colmaxabs over sample chunks, then
 * the scales (order-free max: deterministic), then per element q =
 * e4m3(x / s) (hardware conversion, round to nearest even), the data the
 * algorithm runs on x^ = s dequant(q) written back into xw, and bf16(q)
 * (exact) packed 8 samples per channel for the statistic GEMM. */
__global__ __launch_bounds__(256) void colmaxabs_kernel(const float* __restrict__ xw, long T, int NP,
                                                         long chunk, float* __restrict__ part) {
    const int i = blockIdx.y * 256 + threadIdx.x;
    if (i >= NP) return;
    const long t0 = (long)blockIdx.x * chunk, t1 = min(T, t0 + chunk);
    float mx = 0.f;
    for (long t = t0; t < t1; ++t) mx = fmaxf(mx, fabsf(xw[(size_t)t * NP + i]));
    part[(size_t)blockIdx.x * NP + i] = mx;
}

__global__ void fp8_scale_kernel(const float* __restrict__ part, int nchunks, int NP,
                                 float* __restrict__ scale) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= NP) return;
    float mx = 0.f;
    for (int c = 0; c < nchunks; ++c) mx = fmaxf(mx, part[(size_t)c * NP + i]);
    scale[i] = mx > 0.f ? mx / 448.f : 1.f;
}

__global__ void quantize_fp8_kernel(float* __restrict__ xw, long T, int NP,
                                    const float* __restrict__ scale, uint8_t* __restrict__ xq,
                                    uint16_t* __restrict__ x8) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)T * NP) return;
    const long t = (long)(e / NP);
    const int i = (int)(e % NP);
    const float s = scale[i];
    const int packed = __builtin_amdgcn_cvt_pk_fp8_f32(xw[e] / s, 0.f, 0, false);
    const f2 d = __builtin_amdgcn_cvt_pk_f32_fp8(packed, false);
    xq[e] = (uint8_t)(packed & 0xff);
    xw[e] = d.x * s;
    x8[((size_t)(t >> 3) * NP + i) * 8 + (t & 7)] = (uint16_t)(__float_as_uint(d.x) >> 16);
}

__global__ void bf16_from_f32_kernel(const float* __restrict__ x, size_t count,
                                     uint16_t* __restrict__ out) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < count) out[e] = f32_to_bf16_bits(x[e]);
}

/* The end of the output transform, one wave per entry of grid (n / 4, M, 2):
 * column k of A_out = S^-1 A_h divided by its norm (blockIdx.z 0), entry k of
 * c_out = S^-1 c_h + mean (1). */
__global__ __launch_bounds__(256) void output_finish_kernel(const double* __restrict__ Sinv,
                                                            const double* __restrict__ mean,
                                                            const double* __restrict__ c, int n,
                                                            double* __restrict__ A_out,
                                                            double* __restrict__ c_out) {
    const int h = blockIdx.y, lane = threadIdx.x & 63;
    const int k = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (k >= n) return;
    double s = 0.0;
    if (blockIdx.z == 0) {
        double* col = A_out + (size_t)h * n * n + (size_t)k * n;
        for (int i = lane; i < n; i += 64) s += col[i] * col[i];
        const double nu = sqrt(wave_sum_f64(s));
        for (int i = lane; i < n; i += 64) col[i] /= nu;
    } else {
        for (int l = lane; l < n; l += 64) s += Sinv[k + (size_t)l * n] * c[(size_t)h * n + l];
        s = wave_sum_f64(s);
        if (lane == 0) c_out[(size_t)h * n + k] = s + mean[k];
    }
}

long chunk_of(long T, int nchunks) { return (T + nchunks - 1) / nchunks; }

}  // namespace

/* chunks of the column sums: about eight workgroups per CU, at least 256 samples each */
static int mean_chunks(long T, int cus) { return (int)std::max(1L, std::min(8L * cus, T / 256)); }

/* channel blocks of 16 TI, their pairs, and chunks for about two workgroups
 * per CU in all (each wave holds one SIMD's MFMA pipe busy), at least 256 samples each */
static void cov_shape(long T, int n, int cus, int* TI, int* nblk, int* npairs, int* nchunks) {
    *TI = std::min(4, (n + 15) / 16);
    if (*TI == 3) *TI = 4;
    *nblk = (n + 16 * *TI - 1) / (16 * *TI);
    *npairs = *nblk * (*nblk + 1) / 2;
    *nchunks = (int)std::max(1L, std::min(2L * cus / *npairs, T / 256));
}

size_t sphere_part_doubles(long T, int n, int cus) {
    int TI, nblk, npairs, nchunks;
    cov_shape(T, n, cus, &TI, &nblk, &npairs, &nchunks);
    return std::max((size_t)nchunks * npairs * 256 * TI * TI, (size_t)mean_chunks(T, cus) * n);
}

int launch_colmean(const float* x, long T, int n, double* part, int cus, double* mean, hipStream_t st) {
    const int nc = mean_chunks(T, cus);
    const long chunk = chunk_of(T, nc);
    const int used = (int)((T + chunk - 1) / chunk);
    hipLaunchKernelGGL(colsum_kernel, dim3(used, (n + 255) / 256), dim3(256), 0, st, x, T, n, chunk, part);
    hipLaunchKernelGGL(finish_mean_kernel, dim3((n + 63) / 64), dim3(1024), 0, st, part, used, n, T, mean);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_cov(const float* x, const double* mean, long T, int n, double* part, int cus, double* C,
               hipStream_t st) {
    int TI, nblk, npairs, nchunks;
    cov_shape(T, n, cus, &TI, &nblk, &npairs, &nchunks);
    const long chunk = chunk_of(T, nchunks);
    nchunks = (int)((T + chunk - 1) / chunk);
    const dim3 grid(nchunks, npairs), blk(256);
    if (TI == 1) hipLaunchKernelGGL(cov_kernel<1>, grid, blk, 0, st, x, mean, T, n, chunk, nblk, part);
    else if (TI == 2) hipLaunchKernelGGL(cov_kernel<2>, grid, blk, 0, st, x, mean, T, n, chunk, nblk, part);
    else hipLaunchKernelGGL(cov_kernel<4>, grid, blk, 0, st, x, mean, T, n, chunk, nblk, part);
    const size_t len = (size_t)npairs * 256 * TI * TI;
    hipLaunchKernelGGL(finish_cov_kernel, dim3((unsigned)((len + 63) / 64)), dim3(1024), 0, st, part, nchunks, n,
                       TI, nblk, npairs, T, C);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

size_t inv_sqrt_doubles(int n) { return 7 * (size_t)n * n + 2 * (size_t)n + 64 + 2 * kNsSlots; }

int launch_inv_sqrt(const double* C, int n, double* S, double* ldetS, double* ws, hipStream_t st) {
    if (n < 1 || n > 1024) return -1;
    const size_t nn = (size_t)n * n;
    double* scal = ws;
    unsigned long long* rmax = (unsigned long long*)(ws + 8);
    double* m = ws + 8 + kNsSlots;
    double *Y = m, *Z = m + nn, *Yn = m + 2 * nn, *Zn = m + 3 * nn, *R = m + 4 * nn;
    const unsigned eb = (unsigned)((nn + 255) / 256);
    hipLaunchKernelGGL(ns_norm_kernel, dim3(1), dim3(1024), 0, st, C, n, scal, rmax);
    hipLaunchKernelGGL(ns_init_kernel, dim3(eb), dim3(256), 0, st, C, n, scal, Y, Z);
    /* l = 1e-3 covers condition numbers to 1e6 at the fastest rate; 24
     * iterations reach ~1e9, past which (or with a covariance that is
     * singular or not finite) the caller takes the eigensolver.  |I - Z Y| <=
     * 1e-7 in every entry is two steps from the rounding level. */
    constexpr int kFirst = 14, kMore = 5, kCap = 24;
    static_assert(kCap <= kNsSlots, "a residual slot per iteration");
    const double kNear = 1e-7;
    double l = 1e-3;
    for (int it = 0, stop = kFirst; it < kCap;) {
        for (; it < stop; ++it) {
            const double rho = sqrt(3.0 / (1.0 + l + l * l));
            l = std::min(1.0, 0.5 * rho * l * (3.0 - rho * rho * l * l));
            /* 16 x 16 tiles fill more CUs; past 192 channels 32 x 32 tiles
             * halve the L2 reads and there are enough of them */
            const unsigned g1 = (unsigned)((n + 15) / 16), g2 = (unsigned)((n + 31) / 32);
            if (n <= 192) {
                hipLaunchKernelGGL((ns_product_kernel<1, true>), dim3(g1, g1, 1), dim3(256), 0, st, Z, Y, R,
                                   nullptr, nullptr, nullptr, n, rho, rmax + it);
                hipLaunchKernelGGL((ns_product_kernel<1, false>), dim3(g1, g1, 2), dim3(256), 0, st, Y, R, Yn, R, Z,
                                   Zn, n, 0.0, nullptr);
            } else {
                hipLaunchKernelGGL((ns_product_kernel<2, true>), dim3(g2, g2, 1), dim3(256), 0, st, Z, Y, R,
                                   nullptr, nullptr, nullptr, n, rho, rmax + it);
                hipLaunchKernelGGL((ns_product_kernel<2, false>), dim3(g2, g2, 2), dim3(256), 0, st, Y, R, Yn, R, Z,
                                   Zn, n, 0.0, nullptr);
            }
            std::swap(Y, Yn);
            std::swap(Z, Zn);
        }
        double res[kNsSlots];
        if (hipGetLastError() != hipSuccess || hipStreamSynchronize(st) != hipSuccess ||
            hipMemcpy(res, rmax, sizeof(res), hipMemcpyDeviceToHost) != hipSuccess)
            return -1;
        for (int k = 0; k + 2 <= it; ++k) {
            if (!(res[k] <= kNear)) continue;
            hipLaunchKernelGGL(ns_sphere_kernel, dim3(eb), dim3(256), 0, st, Z, n, scal, S);
            /* ldetS = -log|det S|, which the inverse leaves as its own log-determinant */
            if (launch_gj_inverse(S, Y, ldetS, n, 1, R, st)) return -1;
            return hipGetLastError() == hipSuccess ? 0 : -1;
        }
        stop = std::min(kCap, it + kMore);
    }
    return 1;
}

int launch_eigh(double* C, double* V, double* d, int n, double* work, hipStream_t st) {
    (void)work;
    if (n > 1024) return -1;
    hipLaunchKernelGGL(eigh_kernel, dim3(1), dim3(256), 0, st, C, V, d, n);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_sphere_matrix(const double* V, const double* d, const double* C, int n,
                         const float* x, const double* mean, long T, int do_sphere, double* S,
                         double* ldetS_out, double* part, int nchunks, hipStream_t st) {
    (void)C;
    if (do_sphere == 1) {
        hipLaunchKernelGGL(sphere_from_eig_kernel, dim3(1), dim3(256), 0, st, V, d, n, S,
                           ldetS_out);
    } else if (do_sphere == 2) {
        hipLaunchKernelGGL(var_kernel, dim3(nchunks), dim3(256), 0, st, x, mean, T, n,
                           chunk_of(T, nchunks), part);
        hipLaunchKernelGGL(sphere_diag_kernel, dim3(1), dim3(256), 0, st, part, nchunks, n, T, 1,
                           S, ldetS_out);
    } else {
        hipLaunchKernelGGL(sphere_diag_kernel, dim3(1), dim3(256), 0, st, part, 0, n, T, 0, S,
                           ldetS_out);
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_whiten(const float* x, const double* mean, const double* S, long T, int n, int NP,
                  float* xw, double* xw64, uint16_t* xbf, uint16_t* x8, hipStream_t st) {
    /* one wave per 64-channel group up to eight (four where the LDS tiles of
     * eight would not fit beside the rows), and rows of four waves in all where
     * the groups are one or two */
    const int WC = NP <= 768 ? std::min(NP / 64, 8) : 4, WR = std::max(1, 4 / WC);
    const int TS = 16 * kWhitenRT * WR;
    const size_t shm = (size_t)TS * (NP + 4) * sizeof(float) + NP * sizeof(double) +
                       (size_t)WR * WC * 16 * kWhitenRow * sizeof(float);
    const WhitenArgs a = {x, mean, S, T, n, NP, WR, WC, xw, xw64, xbf, x8};
    if (hipFuncSetAttribute((const void*)whiten_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm) != hipSuccess) return -1;
    const dim3 grid((unsigned)((T + TS - 1) / TS)), blk(64 * WR * WC);
    hipLaunchKernelGGL(whiten_kernel, grid, blk, shm, st, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_white_from_f64(const double* xin, long T, int n, int NP, float* xw, double* xw64,
                          uint16_t* xbf, hipStream_t st) {
    const size_t cnt = (size_t)T * NP;
    hipLaunchKernelGGL(white_from_f64_kernel, dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0,
                       st, xin, T, n, NP, xw, xw64, xbf);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_quantize_fp8(float* xw, long T, int NP, float* scale, uint8_t* xq, uint16_t* x8,
                        float* part, int nchunks, hipStream_t st) {
    const long chunk = (T + nchunks - 1) / nchunks;
    hipLaunchKernelGGL(colmaxabs_kernel, dim3(nchunks, (NP + 255) / 256), dim3(256), 0, st, xw, T, NP,
                       chunk, part);
    hipLaunchKernelGGL(fp8_scale_kernel, dim3((NP + 255) / 256), dim3(256), 0, st, part, nchunks, NP,
                       scale);
    const size_t cnt = (size_t)T * NP;
    hipLaunchKernelGGL(quantize_fp8_kernel, dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0, st, xw,
                       T, NP, scale, xq, x8);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_bf16_from_f32(const float* x, size_t count, uint16_t* out, hipStream_t st) {
    hipLaunchKernelGGL(bf16_from_f32_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0,
                       st, x, count, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

/* Sinv = S^-1 (the M-step's Gauss-Jordan, over the GPU), S^-1 A_h as FP64
 * MFMA products of two models per launch, then norms and centres: 0.13 ms at
 * 128 channels (4.2 ms in one workgroup with an LU and a thread per value). */
int launch_output_transform(const double* S, const double* mean, const double* A,
                            const double* c, int n, int M, double* work, double* Sinv,
                            double* A_out, double* c_out, hipStream_t st) {
    if (n < 1 || n > 1024) return -1;
    const size_t nn = (size_t)n * n;
    double* ldet = work;
    if (launch_gj_inverse(S, Sinv, ldet, n, 1, work + 8, st)) return -1;
    const unsigned g = (unsigned)((n + 15) / 16);
    for (int h = 0; h < M; h += 2)
        hipLaunchKernelGGL((ns_product_kernel<1, false>), dim3(g, g, std::min(2, M - h)), dim3(256), 0, st, Sinv,
                           A + h * nn, A_out + h * nn, Sinv, A + (h + 1) * nn, A_out + (h + 1) * nn, n, 0.0,
                           nullptr);
    hipLaunchKernelGGL(output_finish_kernel, dim3((unsigned)((n + 3) / 4), M, 2), dim3(256), 0, st, Sinv, mean, c, n,
                       A_out, c_out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace amica
