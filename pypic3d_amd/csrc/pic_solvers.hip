// Electrostatic Poisson CG (FP32 iterations inside an FP64 refinement loop)
// and the FP64 energy diagnostics.
//
// CG follows solve_poisson_with_conjugate_gradient (electrostatic_yee.py:71-156):
// r0 = rho/eps + lapl(phi), p0 = r0, alpha = r.r / p.(-lapl p), phi += alpha p,
// r -= alpha (-lapl p), beta = r'.r'/r.r, p = r' + beta p.  The reference runs
// it in FP64 to an absolute tolerance of 1e-12 on ||r||.  Here the potential
// is held in FP64 and the residual r = rho/eps + lapl(phi) is recomputed from
// it in FP64 (mixed-precision iterative refinement): each outer pass solves
// -lapl e = r with FP32 CG vectors and FP64 dot products to a relative
// residual of kInnerRtol, then phi += e in FP64.  The outer loop stops at the
// reference's test ||r|| <= max(tol, rtol ||r0||) on the FP64 residual, when a
// pass no longer halves it (the FP64 rounding floor), or after max_iter inner
// iterations in total.
//
// Ghost handling: phi and p are refreshed by _apply_tiled_phi_constant_
// boundaries (:26-43) before every Laplacian in the reference.  Only the face
// neighbours of interior cells enter the 7-point Laplacian, and after that
// sequence a face neighbour across axis a is: the periodic partner (periodic
// axis; a reduced periodic axis is its own partner), the cell itself (the
// last conducting axis, whose ghosts copy the adjacent plane) or zero (an
// earlier conducting axis, whose ghosts the later calls' refresh zeroes).
// The kernels read neighbours through that map on interior-only arrays.
// Without a zero-neighbour axis the operator is singular (constants); the
// mean of the FP64 residual is then removed before each pass (the k = 0
// mode, a neutralising background), so a deposit whose net charge is zero
// only up to FP32 rounding still converges; the reference's FP64 CG relies
// on the net charge being zero to its own rounding.
// The scalars live on the device; every iteration kernel returns at once when
// the device `done` flag is set, so the host queues iterations in batches and
// reads the flag once per batch.
//
// Direct passes.  The operator is separable and its eigenvectors along an axis
// are known (periodic: real Fourier, self neighbour: DCT-II, zero neighbour:
// DST-I), so a pass that is to converge can be solved outright: three dense
// transforms, a division by the eigenvalues and three transforms back, in FP64
// on the matrix cores.  64^3 with the default limits takes two such passes of
// six 3.4 us launches, where CG takes 448 iterations of five (an electrostatic
// step with 8 and 8 particles per cell 12.5 -> 1.25 ms).  CG stays for iteration
// limits that may end it before it has converged (its unconverged potential is
// then the answer) and for axes whose dense tables would not pay (kMaxDirect).
#include "pic_common.h"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <mutex>

int pic_refresh_fields(const PicDesc* d, float* f0, float* f1, float* f2, int bc_type, hipStream_t s);
extern "C" int pic_constant_boundary(const PicDesc* desc, float* field, int axis, void* stream);

// Scratch of the allocation-free energy entry point (pic_energy_noalloc):
// the FP64 partial sums of its three reductions, 3 x 1024 doubles = 24 KiB,
// held by every GPU the library runs on until the process ends.  Every
// partial a call reads is written earlier in the same call, so nothing needs
// clearing; calls that overlap on one GPU share the array and race.
static __device__ __align__(256) double scratch[3 * 1024];

namespace {

constexpr int kBlock = 256;
constexpr int kMaxPartials = 1024;
static_assert(sizeof(scratch) == 3 * kMaxPartials * sizeof(double), "energy scratch holds its three partial arrays");
constexpr int kBatch = 32;
constexpr int kMaxOuter = 30;
constexpr double kInnerRtol = 1.0e-5;

enum NeighbourMode : int { NB_PERIODIC = 0, NB_SELF = 1, NB_ZERO = 2 };

struct CGScalars {
    double rr, pAp, alpha, beta, tol2, rr_true, mean;
    int32_t done, iter, max_iter, pad;
    double target, prev;      // of the direct passes
};

// interior-array geometry and the face-neighbour map
struct LapMap {
    int n[3];
    int mode[3];
    int singular;   // no zero-neighbour axis: constants span the null space
    int64_t sx, sy;
    double i2[3];   // 1/d^2
};

LapMap lap_map(const PicDesc* d) {
    LapMap M;
    int last = -1;
    for (int a = 0; a < 3; ++a)
        if (d->bc[a] == 1) last = a;
    for (int a = 0; a < 3; ++a) {
        M.n[a] = d->n[a];
        M.mode[a] = d->bc[a] != 1 ? NB_PERIODIC : (a == last ? NB_SELF : NB_ZERO);
        M.i2[a] = 1.0 / (d->d[a] * d->d[a]);
    }
    M.singular = M.mode[0] != NB_ZERO && M.mode[1] != NB_ZERO && M.mode[2] != NB_ZERO;
    M.sy = d->n[2];
    M.sx = (int64_t)d->n[1] * d->n[2];
    return M;
}

__device__ inline double block_sum(double v) {
    __shared__ double sh[kBlock];
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int s = kBlock / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
        __syncthreads();
    }
    double out = sh[0];
    __syncthreads();
    return out;
}

// value of the face neighbour at offset dir (+-1) along an axis of the
// interior array: index q, extent n, stride st
template <class T>
__device__ inline T face_nb(const T* __restrict__ f, int64_t c, int q, int n, int64_t st, int mode, int dir, T fc) {
    int qq = q + dir;
    if (qq >= 0 && qq < n) return f[c + dir * st];
    if (mode == NB_PERIODIC) return f[c + (dir > 0 ? -(int64_t)(n - 1) : (int64_t)(n - 1)) * st];
    if (mode == NB_SELF) return fc;
    return (T)0;
}

// lapl f at interior cell (i, j, k) (electrostatic_yee.py:98-103) in T
template <class T>
__device__ inline T lapl_at(const T* __restrict__ f, const LapMap& M, int64_t c, int i, int j, int k) {
    const T fc = f[c];
    const T two = (T)2;
    T lx = face_nb(f, c, i, M.n[0], M.sx, M.mode[0], 1, fc) + face_nb(f, c, i, M.n[0], M.sx, M.mode[0], -1, fc) -
           two * fc;
    T ly = face_nb(f, c, j, M.n[1], M.sy, M.mode[1], 1, fc) + face_nb(f, c, j, M.n[1], M.sy, M.mode[1], -1, fc) -
           two * fc;
    T lz = face_nb(f, c, k, M.n[2], (int64_t)1, M.mode[2], 1, fc) +
           face_nb(f, c, k, M.n[2], (int64_t)1, M.mode[2], -1, fc) - two * fc;
    return lx * (T)M.i2[0] + ly * (T)M.i2[1] + lz * (T)M.i2[2];
}

__device__ inline void split(const LapMap& M, int64_t t, int& i, int& j, int& k) {
    k = (int)(t % M.n[2]);
    int64_t r = t / M.n[2];
    j = (int)(r % M.n[1]);
    i = (int)(r / M.n[1]);
}

__device__ inline void interior_coords(const PicDesc& d, int64_t t, int& i, int& j, int& k) {
    k = (int)(t % d.n[2]);
    int64_t r = t / d.n[2];
    j = (int)(r % d.n[1]);
    i = (int)(r / d.n[1]);
    i += d.g;
    j += d.g;
    k += d.g;
}

// phi_d <- interior of phi (ghosted FP32)
__global__ void cg_load_kernel(PicDesc d, const float* __restrict__ phi, double* __restrict__ phid) {
    int64_t total = (int64_t)d.n[0] * d.n[1] * d.n[2];
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        interior_coords(d, t, i, j, k);
        phid[t] = (double)phi[fidx(d, i, j, k)];
    }
}

// sum of the FP64 residual rho/eps + lapl(phi_d) (its mean is removed when
// the operator is singular)
__global__ void cg_residual_sum_kernel(PicDesc d, LapMap M, const float* __restrict__ rho,
                                       const double* __restrict__ phid, double* partials, double inv_eps) {
    int64_t total = (int64_t)M.n[0] * M.n[1] * M.n[2];
    double acc = 0.0;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        split(M, t, i, j, k);
        acc += (double)rho[fidx(d, i + d.g, j + d.g, k + d.g)] * inv_eps + lapl_at(phid, M, t, i, j, k);
    }
    double s = block_sum(acc);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

__global__ void cg_mean_kernel(const double* partials, int nparts, CGScalars* sc, double inv_n) {
    double acc = 0.0;
    for (int b = threadIdx.x; b < nparts; b += blockDim.x) acc += partials[b];
    acc = block_sum(acc);
    if (threadIdx.x == 0) sc->mean = acc * inv_n;
}

// FP64 residual r = rho/eps + lapl(phi_d) - mean; starts an inner solve: r
// (FP32), p = r, e = 0; partials of r.r in FP64 (of the FP64 residual)
__global__ void cg_residual_kernel(PicDesc d, LapMap M, const float* __restrict__ rho, const double* __restrict__ phid,
                                   float* __restrict__ r, float* __restrict__ p, float* __restrict__ e,
                                   double* partials, double inv_eps, const CGScalars* sc) {
    int64_t total = (int64_t)M.n[0] * M.n[1] * M.n[2];
    const double mean = M.singular ? sc->mean : 0.0;
    double acc = 0.0;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        split(M, t, i, j, k);
        double rv = (double)rho[fidx(d, i + d.g, j + d.g, k + d.g)] * inv_eps + lapl_at(phid, M, t, i, j, k) - mean;
        float rf = (float)rv;
        r[t] = rf;
        p[t] = rf;
        e[t] = 0.0f;
        acc += rv * rv;
    }
    double s = block_sum(acc);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

// r.r of the FP64 residual, and the inner solve's start: the inner residual
// is r cast to FP32, its stop threshold max(target, kInnerRtol ||r||)
__global__ void cg_start_kernel(const double* partials, int nparts, CGScalars* sc, double target, int max_iter) {
    double acc = 0.0;
    for (int b = threadIdx.x; b < nparts; b += blockDim.x) acc += partials[b];
    double rr = block_sum(acc);
    if (threadIdx.x == 0) {
        double t = fmax(target, kInnerRtol * sqrt(rr));
        sc->rr_true = rr;
        sc->rr = rr;
        sc->tol2 = t * t;
        sc->iter = 0;
        sc->max_iter = max_iter;
        sc->done = (max_iter <= 0 || !(rr > sc->tol2)) ? 1 : 0;
    }
}

__global__ void cg_ap_kernel(LapMap M, const float* __restrict__ p, float* __restrict__ Ap, double* partials,
                             const CGScalars* sc) {
    if (sc->done) return;
    int64_t total = (int64_t)M.n[0] * M.n[1] * M.n[2];
    double acc = 0.0;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        split(M, t, i, j, k);
        float ap = -lapl_at(p, M, t, i, j, k);
        Ap[t] = ap;
        acc += (double)p[t] * (double)ap;
    }
    double s = block_sum(acc);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

__global__ void cg_alpha_kernel(const double* partials, int nparts, CGScalars* sc) {
    if (sc->done) return;
    double acc = 0.0;
    for (int b = threadIdx.x; b < nparts; b += blockDim.x) acc += partials[b];
    double pAp = block_sum(acc);
    if (threadIdx.x == 0) {
        sc->pAp = pAp;
        sc->alpha = sc->rr / pAp;
    }
}

__global__ void cg_update_kernel(int64_t total, float* __restrict__ e, float* __restrict__ r,
                                 const float* __restrict__ p, const float* __restrict__ Ap, double* partials,
                                 const CGScalars* sc) {
    if (sc->done) return;
    float alpha = (float)sc->alpha;
    double acc = 0.0;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
        e[t] += alpha * p[t];
        float rn = r[t] - alpha * Ap[t];
        r[t] = rn;
        acc += (double)rn * (double)rn;
    }
    double s = block_sum(acc);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

__global__ void cg_beta_kernel(const double* partials, int nparts, CGScalars* sc) {
    if (sc->done) return;
    double acc = 0.0;
    for (int b = threadIdx.x; b < nparts; b += blockDim.x) acc += partials[b];
    double rr_new = block_sum(acc);
    if (threadIdx.x == 0) {
        sc->beta = rr_new / sc->rr;
        sc->rr = rr_new;
        sc->iter += 1;
        if (sc->iter >= sc->max_iter || !(rr_new > sc->tol2)) sc->done = 1;
    }
}

__global__ void cg_p_kernel(int64_t total, const float* __restrict__ r, float* __restrict__ p, const CGScalars* sc) {
    if (sc->done) return;
    float beta = (float)sc->beta;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x)
        p[t] = r[t] + beta * p[t];
}

// ---- direct passes ----

constexpr int kMaxDirect = 1024;    // longest axis: 8 MB per table

// Tables of one axis: Q (eigenvectors in columns, orthonormal), its transpose
// and the eigenvalues of -d^2/dx^2.
struct AxisTable {
    int n, mode;
    double i2;
    double *q, *qt, *lam;
};

struct DirectTables {
    AxisTable a[3];
};

__global__ void direct_tables_kernel(DirectTables D) {
    const AxisTable T = D.a[blockIdx.y];
    const int n = T.n;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < (int64_t)n * n;
         t += (int64_t)gridDim.x * blockDim.x) {
        const int j = (int)(t / n), k = (int)(t % n);
        double q, s;      // eigenvector k at node j; lam = 4 s^2 / d^2
        if (T.mode == NB_PERIODIC) {
            const int m = (k + 1) / 2;
            const double x = (double)((2 * (int64_t)m * j) % (2 * n)) / n;        // angle / pi
            if (k == 0) q = sqrt(1.0 / n);
            else if (2 * m == n) q = (j & 1) ? -sqrt(1.0 / n) : sqrt(1.0 / n);
            else q = sqrt(2.0 / n) * ((k & 1) ? cospi(x) : sinpi(x));
            s = sinpi((double)m / n);
        } else if (T.mode == NB_SELF) {
            const double x = (double)(((2 * (int64_t)j + 1) * k) % (4 * n)) / (2 * n);
            q = k == 0 ? sqrt(1.0 / n) : sqrt(2.0 / n) * cospi(x);
            s = sinpi(0.5 * k / n);
        } else {
            const double x = (double)(((int64_t)(j + 1) * (k + 1)) % (2 * (n + 1))) / (n + 1);
            q = sqrt(2.0 / (n + 1)) * sinpi(x);
            s = sinpi(0.5 * (k + 1) / (n + 1));
        }
        T.q[t] = q;
        T.qt[(int64_t)k * n + j] = q;
        if (j == 0) T.lam[k] = 4.0 * s * s * T.i2;
    }
}

// FP64 residual of a direct pass, its mean removed, and the partials of r.r.
__global__ void direct_residual_kernel(PicDesc d, LapMap M, const float* __restrict__ rho,
                                       const double* __restrict__ phid, double* __restrict__ r, double* partials,
                                       double inv_eps, const CGScalars* sc) {
    int64_t total = (int64_t)M.n[0] * M.n[1] * M.n[2];
    const double mean = M.singular ? sc->mean : 0.0;
    double acc = 0.0;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        split(M, t, i, j, k);
        double rv = (double)rho[fidx(d, i + d.g, j + d.g, k + d.g)] * inv_eps + lapl_at(phid, M, t, i, j, k) - mean;
        r[t] = rv;
        acc += rv * rv;
    }
    double s = block_sum(acc);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

// Ends the passes by the tests of the CG loop: ||r|| at the target, or a pass
// that did not halve it.  pass counts the corrections made so far.
__global__ void direct_check_kernel(const double* partials, int nparts, CGScalars* sc, double tol, double rtol,
                                    int pass) {
    if (pass > 0 && sc->done) return;
    double acc = 0.0;
    for (int b = threadIdx.x; b < nparts; b += blockDim.x) acc += partials[b];
    const double rr = block_sum(acc);
    if (threadIdx.x == 0) {
        const double last = sqrt(rr);
        if (pass == 0) sc->target = fmax(tol, rtol * last);
        sc->rr_true = rr;
        sc->iter = pass;
        sc->done = !(last > sc->target) || (pass > 0 && !(last < 0.5 * sc->prev)) ? 1 : 0;
        sc->prev = last;
    }
}

// C = A B per batch (blockIdx.z), all row-major FP64: a transform along the
// last axis has the data as A (rows of it) and the table as B, one along an
// earlier axis the table as A and the data as B.  A wave owns kW x kW MFMA tiles
// of 16 x 16, a block 2 x 2 waves; 16 values of the contraction are in LDS at a
// time and the next 16 in flight.  kDivide: by the sum of the axes' eigenvalues
// (zero for the constant of a singular operator); kAdd: C += A B.
enum TransformEnd { kStore, kDivide, kAdd };
struct Transform {
    const double *A, *B;
    double* C;
    int M, N, K;
    int64_t lda, ldb, ldc, batch_b, batch_c;
};
typedef double v4d __attribute__((ext_vector_type(4)));

template <int kW, int kEnd>
__global__ __launch_bounds__(kBlock) void transform_kernel(Transform T, LapMap M, DirectTables D, const CGScalars* sc) {
    constexpr int kT = 32 * kW, kK = 16, kQ = kT * kK / kBlock;
    __shared__ double As[kK][kT + 1], Bs[kK][kT];
    if (sc->done) return;
    const int m0 = blockIdx.y * kT, n0 = blockIdx.x * kT;
    const double* __restrict__ B = T.B + blockIdx.z * T.batch_b;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = (wave >> 1) * 16 * kW, wn = (wave & 1) * 16 * kW;
    v4d acc[kW][kW];
#pragma unroll
    for (int a = 0; a < kW; ++a)
#pragma unroll
        for (int b = 0; b < kW; ++b) acc[a][b] = v4d{0.0, 0.0, 0.0, 0.0};
    double ra[kQ], rb[kQ];
    const auto load = [&](int k0) {
#pragma unroll
        for (int q = 0; q < kQ; ++q) {
            const int e = (int)threadIdx.x + q * kBlock;
            const int am = m0 + e / kK, ak = k0 + e % kK, bk = k0 + e / kT, bn = n0 + e % kT;
            ra[q] = am < T.M && ak < T.K ? T.A[am * T.lda + ak] : 0.0;
            rb[q] = bk < T.K && bn < T.N ? B[bk * T.ldb + bn] : 0.0;
        }
    };
    load(0);
    for (int k0 = 0; k0 < T.K; k0 += kK) {
#pragma unroll
        for (int q = 0; q < kQ; ++q) {
            const int e = (int)threadIdx.x + q * kBlock;
            As[e % kK][e / kK] = ra[q];
            Bs[e / kT][e % kT] = rb[q];
        }
        __syncthreads();
        if (k0 + kK < T.K) load(k0 + kK);
#pragma unroll
        for (int kk = 0; kk < kK; kk += 4) {
            double a[kW], b[kW];
#pragma unroll
            for (int q = 0; q < kW; ++q) {
                a[q] = As[kk + (lane >> 4)][wm + 16 * q + (lane & 15)];
                b[q] = Bs[kk + (lane >> 4)][wn + 16 * q + (lane & 15)];
            }
#pragma unroll
            for (int p = 0; p < kW; ++p)
#pragma unroll
                for (int q = 0; q < kW; ++q)
                    acc[p][q] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[p], b[q], acc[p][q], 0, 0, 0);
        }
        __syncthreads();
    }
#pragma unroll
    for (int p = 0; p < kW; ++p)
#pragma unroll
        for (int q = 0; q < kW; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int m = m0 + wm + 16 * p + 4 * v + (lane >> 4), n = n0 + wn + 16 * q + (lane & 15);
                if (m >= T.M || n >= T.N) continue;
                const int64_t t = blockIdx.z * T.batch_c + m * T.ldc + n;
                double c = acc[p][q][v];
                if constexpr (kEnd == kDivide) {
                    int i, j, k;
                    split(M, t, i, j, k);
                    const double lam = D.a[0].lam[i] + D.a[1].lam[j] + D.a[2].lam[k];
                    c = M.singular && i + j + k == 0 ? 0.0 : c / lam;
                }
                if constexpr (kEnd == kAdd) c += T.C[t];
                T.C[t] = c;
            }
}

// phi_d += e (FP64 accumulation of the FP32 correction)
__global__ void cg_accumulate_kernel(int64_t total, double* __restrict__ phid, const float* __restrict__ e) {
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x)
        phid[t] += (double)e[t];
}

// phi interior <- phi_d rounded to FP32
__global__ void cg_store_kernel(PicDesc d, const double* __restrict__ phid, float* __restrict__ phi) {
    int64_t total = (int64_t)d.n[0] * d.n[1] * d.n[2];
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        interior_coords(d, t, i, j, k);
        phi[fidx(d, i, j, k)] = (float)phid[t];
    }
}

// ---- energy (utils.py:108-187) ----

__global__ void energy_fields_kernel(PicDesc d, const float* ex, const float* ey, const float* ez, const float* bx,
                                     const float* by, const float* bz, double* partials) {
    int64_t total = (int64_t)d.n[0] * d.n[1] * d.n[2];
    double e2 = 0.0, b2 = 0.0;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        interior_coords(d, t, i, j, k);
        int64_t c = fidx(d, i, j, k);
        double a = ex[c], b = ey[c], cc = ez[c];
        e2 += a * a + b * b + cc * cc;
        a = bx[c];
        b = by[c];
        cc = bz[c];
        b2 += a * a + b * b + cc * cc;
    }
    double se = block_sum(e2);
    double sb = block_sum(b2);
    if (threadIdx.x == 0) {
        partials[2 * blockIdx.x] = se;
        partials[2 * blockIdx.x + 1] = sb;
    }
}

// f(species, v^2) of the active slots from index i of a plane: four slots by one
// 16-byte load a plane where the planes allow it, the rest one at a time.
template <class F>
__device__ inline void each_speed2(const PicSpecies& sp, const PicParticles& in, int64_t n, int vec_ok, const F& f) {
    const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t groups = vec_ok ? n / 4 : 0;
    const auto speed2 = [](float x, float y, float z) {
        const double vx = x, vy = y, vz = z;
        return vx * vx + vy * vy + vz * vz;
    };
    for (int64_t q = t0; q < groups; q += stride) {
        const float4 x = reinterpret_cast<const float4*>(in.u[0])[q];
        const float4 y = reinterpret_cast<const float4*>(in.u[1])[q];
        const float4 z = reinterpret_cast<const float4*>(in.u[2])[q];
        const uchar4 on = reinterpret_cast<const uchar4*>(in.active)[q];
        int s = species_of(4 * q, sp.slots, sp.count);
        const int64_t left = (int64_t)(s + 1) * sp.slots - 4 * q;   // slots of species s from here
        const bool one = left >= 4 || s + 1 == sp.count;
        if (on.x) f(s, speed2(x.x, y.x, z.x));
        if (on.y) f(one ? s : species_of(4 * q + 1, sp.slots, sp.count), speed2(x.y, y.y, z.y));
        if (on.z) f(one ? s : species_of(4 * q + 2, sp.slots, sp.count), speed2(x.z, y.z, z.z));
        if (on.w) f(one ? s : species_of(4 * q + 3, sp.slots, sp.count), speed2(x.w, y.w, z.w));
    }
    for (int64_t i = 4 * groups + t0; i < n; i += stride)
        if (in.active[i]) f(species_of(i, sp.slots, sp.count), speed2(in.u[0][i], in.u[1][i], in.u[2][i]));
}

int velocities_aligned(const PicParticles& in) {
    const uintptr_t planes = (uintptr_t)in.u[0] | (uintptr_t)in.u[1] | (uintptr_t)in.u[2];
    return (planes & 15u) == 0 && ((uintptr_t)in.active & 3u) == 0;
}

// sqrt((m gamma v)^2 C^2 + m^2 C^4) - m C^2 = |m| C^2 gamma - m C^2, with
// C^2 (gamma - 1) = v^2 / (r (1 + r)) for r = 1/gamma = sqrt(1 - v^2/C^2): one
// square root and no cancellation in place of two roots.  Bound by FP64 arithmetic
// (a root and two divisions a slot): 16.8M slots 98.7 -> 52.7 us (4.1 TB/s).
__global__ void energy_kinetic_kernel(PicSpecies sp, PicParticles in, double C, double* partials, int64_t n,
                                      int vec_ok) {
    __shared__ double mass[PIC_MAX_SPECIES], rest[PIC_MAX_SPECIES];
    const double C2 = C * C;
    if ((int)threadIdx.x < sp.count) {
        const double m = sp.mass[threadIdx.x] * sp.weight[threadIdx.x];
        mass[threadIdx.x] = fabs(m);
        rest[threadIdx.x] = (fabs(m) - m) * C2;     // 0 for any mass that is not negative
    }
    __syncthreads();
    double ke = 0.0;
    each_speed2(sp, in, n, vec_ok, [&](int s, double v2) {
        const double r2 = 1.0 - v2 / C2;
        ke += mass[s] * (v2 / (sqrt(r2) + r2)) + rest[s];
    });
    double s = block_sum(ke);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

__global__ void energy_finalize(const double* fpart, int nf, const double* kpart, int nk, double ce, double cb,
                                double* out) {
    double e = 0.0, b = 0.0, k = 0.0;
    for (int i = threadIdx.x; i < nf; i += blockDim.x) {
        e += fpart[2 * i];
        b += fpart[2 * i + 1];
    }
    for (int i = threadIdx.x; i < nk; i += blockDim.x) k += kpart[i];
    e = block_sum(e);
    b = block_sum(b);
    k = block_sum(k);
    if (threadIdx.x == 0) {
        out[0] = ce * e;
        out[1] = cb * b;
        out[2] = k;
    }
}

// compute_total_momentum (utils.py:190-202): sum active |v| mass weight
// Bound by its reads, 13 bytes a slot: 16.8M slots 60.8 -> 35.9 us (6.1 TB/s).
__global__ void momentum_kernel(PicSpecies sp, PicParticles in, double* partials, int64_t n, int vec_ok) {
    __shared__ double mass[PIC_MAX_SPECIES];
    if ((int)threadIdx.x < sp.count) mass[threadIdx.x] = sp.mass[threadIdx.x] * sp.weight[threadIdx.x];
    __syncthreads();
    double acc = 0.0;
    each_speed2(sp, in, n, vec_ok, [&](int s, double v2) { acc += sqrt(v2) * mass[s]; });
    double s = block_sum(acc);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

// sum of rho over the interior (the total charge is this times dV)
__global__ void charge_kernel(PicDesc d, const float* __restrict__ rho, double* partials) {
    int64_t total = (int64_t)d.n[0] * d.n[1] * d.n[2];
    double acc = 0.0;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
        int i, j, k;
        interior_coords(d, t, i, j, k);
        acc += (double)rho[fidx(d, i, j, k)];
    }
    double s = block_sum(acc);
    if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

__global__ void sum_finalize(const double* partials, int n, double scale, double* out) {
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) acc += partials[i];
    acc = block_sum(acc);
    if (threadIdx.x == 0) out[0] = scale * acc;
}

int partial_blocks(int64_t work) {
    int64_t b = (work + kBlock - 1) / kBlock;
    if (b < 1) b = 1;
    if (b > kMaxPartials) b = kMaxPartials;
    return (int)b;
}

bool desc_ok(const PicDesc* d) {
    if (!d || d->g < 1) return false;
    for (int a = 0; a < 3; ++a)
        if (d->n[a] < 1 || d->dims[a] != d->n[a] + 2 * d->g) return false;
    return true;
}

// _apply_tiled_phi_constant_boundaries (electrostatic_yee.py:26-43)
int phi_bc(const PicDesc* d, float* f, hipStream_t s) {
    bool any = false;
    for (int a = 0; a < 3; ++a) {
        if (d->bc[a] == 1) {
            int rc = pic_constant_boundary(d, f, a, (void*)s);
            if (rc) return rc;
            any = true;
        }
    }
    if (!any) return pic_refresh_fields(d, f, nullptr, nullptr, 0, s);
    return 0;
}

struct CGLayout {
    int64_t phid_off, p_off, r_off, ap_off, e_off, part_off, sc_off, table_off, total;
};

// Longest axis and the square root of the operator's condition number.
bool direct_possible(const LapMap& M, double& kappa) {
    double top = 0.0, zero = 0.0, low = 0.0;
    bool active = false;
    for (int a = 0; a < 3; ++a) {
        const int n = M.n[a];
        if (n > kMaxDirect) return false;
        active = active || n > 1;
        if (n > 1 || M.mode[a] == NB_ZERO) top += 4.0 * M.i2[a];
        const double angle = M.mode[a] == NB_ZERO ? 0.5 / (n + 1) : (M.mode[a] == NB_SELF ? 0.5 / n : 1.0 / n);
        const double s = std::sin(M_PI * angle), lam = 4.0 * s * s * M.i2[a];
        if (M.mode[a] == NB_ZERO) zero += lam;
        else if (n > 1 && (low == 0.0 || lam < low)) low = lam;
    }
    if (!active) return false;
    kappa = std::sqrt(top / (zero > 0.0 ? zero : low));
    return true;
}

// workspace: phi_d (FP64) and p, r, Ap, e (FP32) over the interior, FP64
// partial sums, the scalar block, the axis tables of the direct passes (whose
// two FP64 arrays lie over p, r and Ap, e)
CGLayout cg_layout(const PicDesc* d) {
    auto up = [](int64_t b) { return ((b + 255) / 256) * 256; };
    const int64_t n = (int64_t)d->n[0] * d->n[1] * d->n[2];
    CGLayout L;
    L.phid_off = 0;
    L.p_off = up(n * 8);
    L.r_off = L.p_off + up(n * 4);
    L.ap_off = L.r_off + up(n * 4);
    L.e_off = L.ap_off + up(n * 4);
    L.part_off = L.e_off + up(n * 4);
    L.sc_off = L.part_off + kMaxPartials * 8;
    L.table_off = L.sc_off + 256;
    L.total = L.table_off;
    double kappa;
    if (direct_possible(lap_map(d), kappa))
        for (int a = 0; a < 3; ++a) L.total += up((int64_t)d->n[a] * (2 * d->n[a] + 1) * 8);
    return L;
}

// compute_energy's three FP64 reductions with their partial sums in ws
// (2 * kMaxPartials field partials, then kMaxPartials kinetic partials)
int energy_launch(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in, const float* const E[3],
                  const float* const B[3], double* out, double* ws, hipStream_t s) {
    double* fpart = ws;
    double* kpart = fpart + 2 * kMaxPartials;
    int64_t interior = (int64_t)desc->n[0] * desc->n[1] * desc->n[2];
    int nf = partial_blocks(interior);
    int64_t n = (int64_t)sp->count * sp->slots;
    int nk = partial_blocks(n);
    hipLaunchKernelGGL(energy_fields_kernel, dim3(nf), dim3(kBlock), 0, s, *desc, E[0], E[1], E[2], B[0], B[1], B[2],
                       fpart);
    PIC_CHECK_LAUNCH();
    hipLaunchKernelGGL(energy_kinetic_kernel, dim3(nk), dim3(kBlock), 0, s, *sp, *in, desc->C, kpart, n,
                       velocities_aligned(*in));
    PIC_CHECK_LAUNCH();
    double dV = desc->d[0] * desc->d[1] * desc->d[2];
    hipLaunchKernelGGL(energy_finalize, dim3(1), dim3(kBlock), 0, s, fpart, nf, kpart, nk, 0.5 * desc->eps * dV,
                       0.5 / desc->mu * dV, out);
    PIC_CHECK_LAUNCH();
    return 0;
}

// Device address of `scratch` on the current device, looked up once per
// device with that device current (each GPU holds its own copy of the array
// at its own address; the array's name is not a device address in host code).
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
double* g_scratch_ptr[kMaxDevices] = {};

int scratch_address(double** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= kMaxDevices) return -1;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return (int)e;
        g_scratch_ptr[dev] = static_cast<double*>(p);
    }
    *out = g_scratch_ptr[dev];
    return 0;
}

// One direct pass, phi_d += solution of -lapl e = r: forward along z, y, x, back along x, y, z,
// between r and tmp.  Axes of one cell have nothing to transform.
int direct_solve(const LapMap& M, const DirectTables& D, double* r, double* tmp, double* phid, const CGScalars* sc,
                 hipStream_t s) {
    int axes[6], n = 0;
    for (int a = 2; a >= 0; --a)
        if (M.n[a] > 1) axes[n++] = a;
    for (int q = n - 1, f = n; q >= 0; --q) axes[f++] = axes[q];
    double *src = r, *dst = tmp;
    for (int q = 0; q < 2 * n; ++q) {
        const int a = axes[q];
        const bool back = q >= n, last = q == 2 * n - 1, divide = q == n - 1;
        const AxisTable& X = D.a[a];
        int64_t inner = 1, outer = 1;
        for (int b = a + 1; b < 3; ++b) inner *= M.n[b];
        for (int b = 0; b < a; ++b) outer *= M.n[b];
        Transform T;
        int batches = 1;
        T.C = last ? phid : dst;
        if (inner == 1) {          // rows of data times the table
            T.A = src;
            T.B = back ? X.qt : X.q;
            T.M = (int)outer;
            T.N = T.K = X.n;
            T.lda = T.ldb = T.ldc = X.n;
            T.batch_b = T.batch_c = 0;
        } else {                   // the table times columns of data
            T.A = back ? X.q : X.qt;
            T.B = src;
            T.M = T.K = X.n;
            T.N = (int)inner;
            T.lda = X.n;
            T.ldb = T.ldc = inner;
            T.batch_b = T.batch_c = X.n * inner;
            batches = (int)outer;
        }
        // 64 x 64 tiles where they make a block for every second CU at least; smaller problems
        // take 32 x 32 tiles to fill the chip
        const auto grid = [&](int tile) {
            return dim3((T.N + tile - 1) / tile, (T.M + tile - 1) / tile, batches);
        };
        const dim3 g64 = grid(64), g32 = grid(32);
        const bool wide = (int64_t)g64.x * g64.y * g64.z >= 128;
#define PIC_TRANSFORM(W, END) \
    hipLaunchKernelGGL((transform_kernel<W, END>), W == 2 ? g64 : g32, dim3(kBlock), 0, s, T, M, D, sc)
#define PIC_TRANSFORM_END(END)              \
    do {                                    \
        if (wide) PIC_TRANSFORM(2, END);    \
        else PIC_TRANSFORM(1, END);         \
    } while (0)
        if (last) PIC_TRANSFORM_END(kAdd);
        else if (divide) PIC_TRANSFORM_END(kDivide);
        else PIC_TRANSFORM_END(kStore);
#undef PIC_TRANSFORM_END
#undef PIC_TRANSFORM
        PIC_CHECK_LAUNCH();
        std::swap(src, dst);
    }
    return 0;
}

int read_scalars(CGScalars* host, const CGScalars* dev, hipStream_t s) {
    hipError_t e = hipMemcpyAsync(host, dev, sizeof(CGScalars), hipMemcpyDeviceToHost, s);
    if (e != hipSuccess) return (int)e;
    e = hipStreamSynchronize(s);
    return e == hipSuccess ? 0 : (int)e;
}

}  // namespace

extern "C" {

int64_t pic_cg_workspace_bytes(const PicDesc* desc) {
    if (!desc_ok(desc)) return -1;
    return cg_layout(desc).total;
}

int pic_poisson_cg(const PicDesc* desc, const float* rho, float* phi, double tol, double rtol, int32_t max_iter,
                   void* workspace, int64_t workspace_bytes, int32_t* iterations, double* residual_norm,
                   void* stream) {
    PIC_REQUIRE(desc_ok(desc) && rho && phi && workspace && rho != phi && max_iter >= 0);
    PIC_REQUIRE(tol >= 0.0 && rtol >= 0.0);
    CGLayout Lw = cg_layout(desc);
    PIC_REQUIRE(workspace_bytes >= Lw.total);
    hipStream_t s = as_stream(stream);
    char* base = static_cast<char*>(workspace);
    double* phid = reinterpret_cast<double*>(base + Lw.phid_off);
    float* p = reinterpret_cast<float*>(base + Lw.p_off);
    float* r = reinterpret_cast<float*>(base + Lw.r_off);
    float* Ap = reinterpret_cast<float*>(base + Lw.ap_off);
    float* e = reinterpret_cast<float*>(base + Lw.e_off);
    double* partials = reinterpret_cast<double*>(base + Lw.part_off);
    CGScalars* sc = reinterpret_cast<CGScalars*>(base + Lw.sc_off);

    const LapMap M = lap_map(desc);
    const int64_t interior = (int64_t)desc->n[0] * desc->n[1] * desc->n[2];
    const int nb = partial_blocks(interior);
    const double inv_eps = 1.0 / desc->eps;

    int rc = phi_bc(desc, phi, s);          // phi = apply_bc(phi) (:139)
    if (rc) return rc;
    hipLaunchKernelGGL(cg_load_kernel, dim3(nb), dim3(kBlock), 0, s, *desc, phi, phid);
    PIC_CHECK_LAUNCH();

    CGScalars host;
    int total_iter = 0;
    double target = tol, prev = 0.0, last = 0.0;
    // CG reduces the residual by e^-2 in kappa iterations at least: 16 kappa cover the FP64 range and the restarts
    // of its passes (64^3 periodic: 448 iterations, 12.7 kappa).  Under smaller limits CG itself runs
    double kappa = 0.0;
    const bool direct = direct_possible(M, kappa) && (double)max_iter >= 16.0 * kappa + 64.0;
    if (direct) {
        double *r64 = reinterpret_cast<double*>(base + Lw.p_off), *t64 = reinterpret_cast<double*>(base + Lw.ap_off);
        DirectTables D;
        int64_t off = Lw.table_off;
        int longest = 1;
        for (int a = 0; a < 3; ++a) {
            const int n = M.n[a];
            double* q = reinterpret_cast<double*>(base + off);
            D.a[a] = AxisTable{n, M.mode[a], M.i2[a], q, q + (int64_t)n * n, q + 2 * (int64_t)n * n};
            off += (((int64_t)n * (2 * n + 1) * 8 + 255) / 256) * 256;
            longest = std::max(longest, n);
        }
        hipLaunchKernelGGL(direct_tables_kernel, dim3(grid_1d((int64_t)longest * longest, kBlock), 3), dim3(kBlock), 0,
                           s, D);
        PIC_CHECK_LAUNCH();
        const auto check = [&](int pass) {
            if (M.singular) {
                hipLaunchKernelGGL(cg_residual_sum_kernel, dim3(nb), dim3(kBlock), 0, s, *desc, M, rho, phid, partials,
                                   inv_eps);
                hipLaunchKernelGGL(cg_mean_kernel, dim3(1), dim3(kBlock), 0, s, partials, nb, sc,
                                   1.0 / (double)interior);
            }
            hipLaunchKernelGGL(direct_residual_kernel, dim3(nb), dim3(kBlock), 0, s, *desc, M, rho, phid, r64, partials,
                               inv_eps, sc);
            hipLaunchKernelGGL(direct_check_kernel, dim3(1), dim3(kBlock), 0, s, partials, nb, sc, tol, rtol, pass);
        };
        // one pass brings the residual to the rounding of FP64, the second to its floor: both are
        // queued before the flag is read, the second returning at once if the first was enough
        check(0);
        int pass = 0;
        do {
            for (int q = 0; q < 2; ++q) {
                rc = direct_solve(M, D, r64, t64, phid, sc, s);
                if (rc) return rc;
                check(++pass);
            }
            PIC_CHECK_LAUNCH();
            rc = read_scalars(&host, sc, s);
            if (rc) return rc;
        } while (!host.done && pass < kMaxOuter);
        total_iter = host.iter;
        last = sqrt(host.rr_true);
    }
    for (int outer = 0; !direct && outer < kMaxOuter; ++outer) {
        if (M.singular) {
            hipLaunchKernelGGL(cg_residual_sum_kernel, dim3(nb), dim3(kBlock), 0, s, *desc, M, rho, phid, partials,
                               inv_eps);
            hipLaunchKernelGGL(cg_mean_kernel, dim3(1), dim3(kBlock), 0, s, partials, nb, sc, 1.0 / (double)interior);
        }
        hipLaunchKernelGGL(cg_residual_kernel, dim3(nb), dim3(kBlock), 0, s, *desc, M, rho, phid, r, p, e, partials,
                           inv_eps, sc);
        hipLaunchKernelGGL(cg_start_kernel, dim3(1), dim3(kBlock), 0, s, partials, nb, sc, target,
                           (int)(max_iter - total_iter));
        PIC_CHECK_LAUNCH();
        rc = read_scalars(&host, sc, s);
        if (rc) return rc;
        last = sqrt(host.rr_true);
        if (outer == 0) target = fmax(tol, rtol * last);
        if (!(last > target) || total_iter >= max_iter) break;
        if (outer > 0 && !(last < 0.5 * prev)) break;    // at the FP64 rounding floor
        prev = last;
        // inner FP32 CG on -lapl e = r, e0 = 0, to max(target, kInnerRtol ||r||)
        hipLaunchKernelGGL(cg_start_kernel, dim3(1), dim3(kBlock), 0, s, partials, nb, sc, target,
                           (int)(max_iter - total_iter));
        PIC_CHECK_LAUNCH();
        for (;;) {
            for (int b = 0; b < kBatch; ++b) {
                hipLaunchKernelGGL(cg_ap_kernel, dim3(nb), dim3(kBlock), 0, s, M, p, Ap, partials, sc);
                hipLaunchKernelGGL(cg_alpha_kernel, dim3(1), dim3(kBlock), 0, s, partials, nb, sc);
                hipLaunchKernelGGL(cg_update_kernel, dim3(nb), dim3(kBlock), 0, s, interior, e, r, p, Ap, partials,
                                   sc);
                hipLaunchKernelGGL(cg_beta_kernel, dim3(1), dim3(kBlock), 0, s, partials, nb, sc);
                hipLaunchKernelGGL(cg_p_kernel, dim3(nb), dim3(kBlock), 0, s, interior, r, p, sc);
                PIC_CHECK_LAUNCH();
            }
            rc = read_scalars(&host, sc, s);
            if (rc) return rc;
            if (host.done) break;
        }
        total_iter += host.iter;
        hipLaunchKernelGGL(cg_accumulate_kernel, dim3(nb), dim3(kBlock), 0, s, interior, phid, e);
        PIC_CHECK_LAUNCH();
    }
    hipLaunchKernelGGL(cg_store_kernel, dim3(nb), dim3(kBlock), 0, s, *desc, phid, phi);
    PIC_CHECK_LAUNCH();
    rc = phi_bc(desc, phi, s);
    if (rc) return rc;
    if (iterations) *iterations = total_iter;
    if (residual_norm) *residual_norm = last;
    return 0;
}

int64_t pic_energy_workspace_bytes(const PicDesc* desc, const PicSpecies* sp) {
    if (!desc_ok(desc) || !sp) return -1;
    return (int64_t)(2 * kMaxPartials + kMaxPartials) * 8;
}

int pic_energy(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in, const float* const E[3],
               const float* const B[3], double* out, void* workspace, int64_t workspace_bytes, void* stream) {
    PIC_REQUIRE(desc_ok(desc) && sp && in && E && B && out && workspace);
    for (int a = 0; a < 3; ++a) PIC_REQUIRE(E[a] && B[a]);
    PIC_REQUIRE(particles_ok(sp, in));
    PIC_REQUIRE(workspace_bytes >= pic_energy_workspace_bytes(desc, sp));
    return energy_launch(desc, sp, in, E, B, out, static_cast<double*>(workspace), as_stream(stream));
}

int pic_energy_noalloc(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in, const float* const E[3],
                       const float* const B[3], double* out, void* stream) {
    PIC_REQUIRE(desc_ok(desc) && sp && in && E && B && out);
    for (int a = 0; a < 3; ++a) PIC_REQUIRE(E[a] && B[a]);
    PIC_REQUIRE(particles_ok(sp, in));
    // the partial sums this call needs; never more than the scratch holds
    // (the partial count is capped at kMaxPartials per reduction)
    const int64_t need = pic_energy_workspace_bytes(desc, sp);
    if (need < 0 || need > (int64_t)sizeof(scratch)) {
        fprintf(stderr, "pic_energy_noalloc: needs %lld scratch bytes, the static scratch holds %zu\n",
                (long long)need, sizeof(scratch));
        return -2;
    }
    double* ws = nullptr;
    int rc = scratch_address(&ws);
    if (rc) return rc;
    return energy_launch(desc, sp, in, E, B, out, ws, as_stream(stream));
}

/* compute_total_momentum (utils.py:190-202), FP64 accumulation. */
int pic_total_momentum(const PicSpecies* sp, const PicParticles* in, double* out, void* workspace,
                       int64_t workspace_bytes, void* stream) {
    PIC_REQUIRE(sp && in && out && workspace);
    PIC_REQUIRE(particles_ok(sp, in));
    PIC_REQUIRE(workspace_bytes >= (int64_t)kMaxPartials * 8);
    hipStream_t s = as_stream(stream);
    double* part = static_cast<double*>(workspace);
    int64_t n = (int64_t)sp->count * sp->slots;
    int nk = partial_blocks(n);
    hipLaunchKernelGGL(momentum_kernel, dim3(nk), dim3(kBlock), 0, s, *sp, *in, part, n, velocities_aligned(*in));
    PIC_CHECK_LAUNCH();
    hipLaunchKernelGGL(sum_finalize, dim3(1), dim3(kBlock), 0, s, part, nk, 1.0, out);
    PIC_CHECK_LAUNCH();
    return 0;
}

/* Total charge sum_interior rho dV, FP64 accumulation of the FP32 density. */
int pic_total_charge(const PicDesc* desc, const float* rho, double* out, void* workspace, int64_t workspace_bytes,
                     void* stream) {
    PIC_REQUIRE(desc_ok(desc) && rho && out && workspace);
    PIC_REQUIRE(workspace_bytes >= (int64_t)kMaxPartials * 8);
    hipStream_t s = as_stream(stream);
    double* part = static_cast<double*>(workspace);
    int nf = partial_blocks((int64_t)desc->n[0] * desc->n[1] * desc->n[2]);
    hipLaunchKernelGGL(charge_kernel, dim3(nf), dim3(kBlock), 0, s, *desc, rho, part);
    PIC_CHECK_LAUNCH();
    hipLaunchKernelGGL(sum_finalize, dim3(1), dim3(kBlock), 0, s, part, nf, desc->d[0] * desc->d[1] * desc->d[2],
                       out);
    PIC_CHECK_LAUNCH();
    return 0;
}

}  // extern "C"
