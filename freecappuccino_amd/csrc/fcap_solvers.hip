// Krylov solver drivers: DIC-PCG (src/iccg.f90), Jacobi-PCG (src/dpcg.f90),
// DILU-BiCGStab (src/bicgstab.f90) in FP64 with the reference's update order,
// and FP32 inner solves inside FP64 iterative refinement.
//
// All scalars of an iteration live on the device (struct Scalars).  Each
// reduction is written as per-block partials by the kernel that produces the
// vector (fused), summed by a one-block "finalize" kernel that also performs
// the scalar update of the algorithm (beta, alpha, omega, convergence test).
// Every kernel returns at once when `done` is set, so the host enqueues
// iterations in batches and reads one flag per batch.
//
// Fused iterations (every solve without O-C couplings and with tree-order sums): the
// finalisers are folded into the kernels that need the sums, each block of which adds
// the partials itself, in the same order, so all blocks have the same scalars; block 0
// records them.  An iteration is rotated to begin with A p (PCG) or the new direction
// (BiCGStab), so that the kernel that ends it also tests for convergence; the
// recurrences are those of the finalisers.

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <functional>
#include <mutex>

#include "fcap_solvers.h"
#include "fcap_gnn.h"

namespace fcap {

namespace {

inline int grid_for(long long n, int block) {
    long long g = (n + block - 1) / block;
    return (int)std::max<long long>(1, std::min<long long>(g, 1 << 30));
}

enum FinStep : int {
    kFinRes0 = 0,     // initial residual: res0, early exit
    kFinSk = 1,       // sk = r.z, bet = sk/s0
    kFinAlf = 2,      // pkapk = p.q, alf = sk/pkapk
    kFinPcgEnd = 3,   // resl, s0 = sk, iteration count, convergence
    kFinBet = 4,      // BiCGStab: bet, om, beto
    kFinGam = 5,      // BiCGStab: ukreso, gam
    kFinAlfB = 6,     // BiCGStab: alf = vr/(vv+small)
    kFinBicgEnd = 7,  // BiCGStab: resl, iteration count, convergence
    kFinOuter = 8,    // refinement: true residual norms
    kFinFcgBeta = 9,  // FCG: bet_s = -(z.q_s)/(p_s.q_s) for every stored direction s
    kFinFcgAlf = 10,  // FCG: alf = p.r / p.q, p.q stored in this iteration's slot
    kFinFcgEnd = 11   // FCG: residual, convergence, stagnation at the end of each window
};

// FCG stagnation: window length in fc_context::fcg_stag_window (64 by default)

__device__ inline void converge_test(Scalars *sc) {
    sc->iters += 1;
    sc->rsm = sc->resl / (sc->res0 + sc->small);
    bool finite = isfinite(sc->resl) && isfinite(sc->rnorm2);
    bool conv;
    if (sc->stop_rule == 0) conv = sc->rsm < sc->resmax;
    else if (sc->stop_rule == 1) {
        sc->rel = sqrt(sc->rnorm2 / sc->bnorm2);
        conv = sc->rel < sc->resmax;
    } else conv = sc->rnorm2 <= sc->inner_tol2;
    if (!finite) { sc->done = 1; sc->status = FC_ERR_NONFINITE; }
    else if (conv) { sc->done = 1; sc->status = FC_OK; }
    else if (sc->iters >= sc->nsw) { sc->done = 1; sc->status = FC_NOT_CONVERGED; }
}

// np2: partials of pb (nparts but where said)
__global__ __launch_bounds__(kFinBlock) void k_fin(int step, int nparts, const double *__restrict__ pa, int np2,
                                                  const double *__restrict__ pb, Scalars *__restrict__ sc) {
    __shared__ double sh[kFinBlock / kWave];
    if (sc->done) return;
    if (step == kFinFcgBeta) {
        // partials of slot s at pa[s * nparts + block]
        const int nwin = min(sc->iters, sc->fcg_m);
        for (int s = 0; s < nwin; ++s) {
            double v = 0.0;
            for (int i = threadIdx.x; i < nparts; i += kFinBlock) v += pa[(size_t)s * nparts + i];
            v = block_sum<kFinBlock>(v, sh);
            if (threadIdx.x == 0) sc->fcg_bet[s] = -v / sc->fcg_pqh[s];
        }
        return;
    }
    double a = 0.0, b = 0.0;
    for (int i = threadIdx.x; i < nparts; i += kFinBlock) a += pa[i];
    if (pb)
        for (int i = threadIdx.x; i < np2; i += kFinBlock) b += pb[i];
    a = block_sum<kFinBlock>(a, sh);
    if (pb) b = block_sum<kFinBlock>(b, sh);
    if (threadIdx.x != 0) return;
    switch (step) {
    case kFinRes0:
        sc->res0 = a;
        sc->resl = a;
        sc->rnorm2 = b;
        sc->rel = sc->bnorm2 > 0.0 ? sqrt(b / sc->bnorm2) : 0.0;
        if (!isfinite(a) || !isfinite(b)) { sc->done = 1; sc->status = FC_ERR_NONFINITE; }
        else if (sc->early_exit && a < (double)1e-13f) { sc->done = 1; sc->status = FC_EARLY_EXIT; }
        else if (sc->stop_rule == 1 && sc->rel < sc->resmax) { sc->done = 1; sc->status = FC_OK; }
        else if (sc->stop_rule == 2 && b <= sc->inner_tol2) { sc->done = 1; sc->status = FC_OK; }
        break;
    case kFinSk:
        sc->sk = a;
        sc->bet = a / sc->s0;
        break;
    case kFinAlf:
        sc->pkapk = a;
        sc->alf = sc->sk / a;
        break;
    case kFinPcgEnd:
        sc->resl = a;
        sc->rnorm2 = b;
        sc->s0 = sc->sk;
        converge_test(sc);
        break;
    case kFinBet:
        sc->om = (a * sc->gam) / ((sc->alf * sc->beto) + sc->small);
        sc->beto = a;
        sc->sk = a;
        break;
    case kFinGam:
        sc->ukreso = a;
        sc->gam = sc->sk / a;
        break;
    case kFinAlfB:
        sc->vr = a;
        sc->vv = b;
        sc->alf = a / (b + sc->small);
        break;
    case kFinBicgEnd:
        sc->resl = a;
        sc->rnorm2 = b;
        converge_test(sc);
        break;
    case kFinOuter:
        sc->rnorm2 = b;
        sc->resl = a;
        sc->rel = sqrt(b / sc->bnorm2);
        break;
    case kFinFcgAlf:   // pb: the partials of p.r
        sc->fcg_pr = b;
        sc->pkapk = a;
        sc->alf = b / a;
        sc->fcg_pqh[sc->iters % sc->fcg_m] = a;
        break;
    case kFinFcgEnd:
        sc->resl = a;
        sc->rnorm2 = b;
        converge_test(sc);
        sc->stag_min = fmin(sc->stag_min, b);
        if (!sc->done && sc->stag_every > 0 && sc->iters % sc->stag_every == 0) {
            // CG's residual 2-norm is not monotone: on a graded 192^3 mesh it rises to
            // ~13x ||r0|| within a few iterations of the learned preconditioner and is
            // back below ||r0|| only after ~100 (~3x with IC(0)).  The first window
            // only sets the reference; every later window's best must beat the best
            // before it by the factor.
            const bool first = sc->iters == sc->stag_every;
            if (!first && !(sc->stag_min < sc->stag_factor * sc->stag_ref)) {
                sc->done = 1;
                sc->status = FC_FALLBACK_USED;
            }
            sc->stag_ref = first ? sc->stag_min : fmin(sc->stag_ref, sc->stag_min);
            sc->stag_min = 1e300;
        }
        break;
    }
}

// Flexible CG with the last m = sc->fcg_m <= kFcgM directions.  Direction of
// iteration t lives in slot t % m of ph (and A p in qh); at iteration k
// (= sc->iters) the slots s < min(k, m) hold the directions of iterations
// k-1, ..., k-min(k, m).

// Up to kFcgFold directions k_fcg_p adds the partials of their dot products itself, in every
// block; more of them go through a finaliser (a launch of 5 us against 2 us a block).
constexpr int kFcgFold = 4;

// partials of z.q_s for every stored slot s, at pa[s * gridDim.x + block], or at
// pa[M * block + s] for k_fcg_p; M = sc->fcg_m
template <int M>
__global__ __launch_bounds__(kRedBlock) void k_fcg_dots(int n, const float *__restrict__ z,
                                                        const float *__restrict__ qh, const Scalars *__restrict__ sc,
                                                        double *__restrict__ pa) {
    __shared__ double sh[kRedBlock / kWave];
    if (sc->done) return;
    const int nwin = min(sc->iters, M);
    if (nwin == 0) return;
    double acc[M];
#pragma unroll
    for (int s = 0; s < M; ++s) acc[s] = 0.0;
    if (nwin == M) {
        for (int i = blockIdx.x * kRedBlock + threadIdx.x; i < n; i += gridDim.x * kRedBlock) {
            const double zi = (double)z[i];
#pragma unroll
            for (int s = 0; s < M; ++s) acc[s] += zi * (double)qh[(size_t)s * n + i];
        }
    } else {
        for (int i = blockIdx.x * kRedBlock + threadIdx.x; i < n; i += gridDim.x * kRedBlock) {
            const double zi = (double)z[i];
#pragma unroll
            for (int s = 0; s < M; ++s)
                if (s < nwin) acc[s] += zi * (double)qh[(size_t)s * n + i];
        }
    }
#pragma unroll
    for (int s = 0; s < M; ++s) {
        if (s < nwin) {
            const double v = block_sum<kRedBlock>(acc[s], sh);
            if (threadIdx.x == 0) pa[M <= kFcgFold ? (size_t)M * blockIdx.x + s : (size_t)s * gridDim.x + blockIdx.x] = v;
        }
    }
}

// p = z + sum_s bet_s p_s (bet_s = -z.q_s / p_s.q_s) and the partial of p.r; M = sc->fcg_m
template <int M>
__global__ __launch_bounds__(kRedBlock) void k_fcg_p(int n, float *__restrict__ p, const float *__restrict__ z,
                                                     const float *__restrict__ r, const float *__restrict__ ph,
                                                     const Scalars *__restrict__ sc, const double *__restrict__ pd,
                                                     int nd, double *__restrict__ pa) {
    constexpr bool kFold = M <= kFcgFold;
    __shared__ double sh[(kFold ? M : 1) * (kRedBlock / kWave)];
    if (sc->done) return;
    const int nwin = min(sc->iters, M);
    float bet[M];
    if constexpr (kFold) {
        double t[M];
        parts_total<kRedBlock, M, M>(pd, nd, sh, t);   // (those of slots not yet stored are not used)
#pragma unroll
        for (int s = 0; s < M; ++s) bet[s] = s < nwin ? (float)(-t[s] / sc->fcg_pqh[s]) : 0.f;
    } else {
#pragma unroll
        for (int s = 0; s < M; ++s) bet[s] = s < nwin ? (float)sc->fcg_bet[s] : 0.f;
    }
    double acc = 0.0;
    if (nwin == M) {
        for (int i = blockIdx.x * kRedBlock + threadIdx.x; i < n; i += gridDim.x * kRedBlock) {
            float pv = z[i];
#pragma unroll
            for (int s = 0; s < M; ++s) pv = pv + bet[s] * ph[(size_t)s * n + i];
            p[i] = pv;
            acc += (double)pv * (double)r[i];
        }
    } else {
        for (int i = blockIdx.x * kRedBlock + threadIdx.x; i < n; i += gridDim.x * kRedBlock) {
            float pv = z[i];
#pragma unroll
            for (int s = 0; s < M; ++s)
                if (s < nwin) pv = pv + bet[s] * ph[(size_t)s * n + i];
            p[i] = pv;
            acc += (double)pv * (double)r[i];
        }
    }
    acc = block_sum<kRedBlock>(acc, sh);
    if (threadIdx.x == 0) pa[blockIdx.x] = acc;
}

// x += alf p ; r -= alf q ; p, q stored in this iteration's slot ; partials |r| and r^2
__global__ __launch_bounds__(kRedBlock) void k_fcg_xr(int n, float *__restrict__ x, float *__restrict__ r,
                                                      const float *__restrict__ p, const float *__restrict__ q,
                                                      float *__restrict__ ph, float *__restrict__ qh,
                                                      const Scalars *__restrict__ sc, double *__restrict__ pa,
                                                      double *__restrict__ pb) {
    __shared__ double sh[kRedBlock / kWave];
    if (sc->done) return;
    const float alf = (float)sc->alf;
    const size_t slot = (size_t)(sc->iters % sc->fcg_m) * n;
    double a = 0.0, b = 0.0;
    for (int i = blockIdx.x * kRedBlock + threadIdx.x; i < n; i += gridDim.x * kRedBlock) {
        const float pv = p[i], qv = q[i];
        x[i] = x[i] + alf * pv;
        const float rv = r[i] - alf * qv;
        r[i] = rv;
        ph[slot + i] = pv;
        qh[slot + i] = qv;
        a += fabs((double)rv);
        b += (double)rv * (double)rv;
    }
    a = block_sum<kRedBlock>(a, sh);
    b = block_sum<kRedBlock>(b, sh);
    if (threadIdx.x == 0) { pa[blockIdx.x] = a; pb[blockIdx.x] = b; }
}

// x += alf p ; r -= alf q ; partials |r| and r^2 (src/iccg.f90:147-154)
__global__ __launch_bounds__(kRedBlock) void k_pcg_xr64(int n, double *__restrict__ x, double *__restrict__ r,
                                                       const double *__restrict__ p, const double *__restrict__ q,
                                                       const Scalars *__restrict__ sc, double *__restrict__ pa,
                                                       double *__restrict__ pb) {
    __shared__ double sh[kRedBlock / kWave];
    if (sc->done) return;
    const double alf = sc->alf;
    double a = 0.0, b = 0.0;
    for (int i = blockIdx.x * kRedBlock + threadIdx.x; i < n; i += gridDim.x * kRedBlock) {
        x[i] = x[i] + alf * p[i];
        double rv = r[i] - alf * q[i];
        r[i] = rv;
        a += fabs(rv);
        b += rv * rv;
    }
    a = block_sum<kRedBlock>(a, sh);
    b = block_sum<kRedBlock>(b, sh);
    if (threadIdx.x == 0) { pa[blockIdx.x] = a; pb[blockIdx.x] = b; }
}

template <class T>
__global__ void k_p_update(int n, T *__restrict__ p, const T *__restrict__ z, const Scalars *__restrict__ sc) {
    if (sc->done) return;
    const T bet = (T)sc->bet;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = z[i] + bet * p[i];
}

template <class T>
__global__ __launch_bounds__(kRedBlock) void k_dot(int n, const T *__restrict__ x, const T *__restrict__ y,
                                                   const Scalars *__restrict__ sc, double *__restrict__ pa) {
    __shared__ double sh[kRedBlock / kWave];
    if (sc && sc->done) return;
    double a = 0.0;
    for (int i = blockIdx.x * kRedBlock + threadIdx.x; i < n; i += gridDim.x * kRedBlock)
        a += (double)x[i] * (double)y[i];
    a = block_sum<kRedBlock>(a, sh);
    if (threadIdx.x == 0) pa[blockIdx.x] = a;
}

// Jacobi: z = r / a(diag) and the partial of r.z (src/dpcg.f90:85-90)
template <class T, class AT>
__global__ __launch_bounds__(kRedBlock) void k_jacobi(int n, const T *__restrict__ r, const AT *__restrict__ a,
                                                      const int *__restrict__ diag, T *__restrict__ z,
                                                      const Scalars *__restrict__ sc, double *__restrict__ pa) {
    __shared__ double sh[kRedBlock / kWave];
    if (sc->done) return;
    double s = 0.0;
    for (int i = blockIdx.x * kRedBlock + threadIdx.x; i < n; i += gridDim.x * kRedBlock) {
        T zv = r[i] / (T)a[diag[i]];
        z[i] = zv;
        s += (double)r[i] * (double)zv;
    }
    s = block_sum<kRedBlock>(s, sh);
    if (threadIdx.x == 0) pa[blockIdx.x] = s;
}

// pk = res + om*(pk - alf*uk)  (src/bicgstab.f90:111)
template <class T>
__global__ void k_bicg_p(int n, T *__restrict__ pk, const T *__restrict__ res, const T *__restrict__ uk,
                         const Scalars *__restrict__ sc) {
    if (sc->done) return;
    const T om = (T)sc->om, alf = (T)sc->alf;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        T t = alf * uk[i];
        t = pk[i] - t;
        t = om * t;
        pk[i] = res[i] + t;
    }
}

// fi += gam*zk ; res -= gam*uk  (src/bicgstab.f90:160-161)
template <class T, class X>
__global__ void k_bicg_xr1(int n, X *__restrict__ fi, T *__restrict__ res, const T *__restrict__ zk,
                           const T *__restrict__ uk, const Scalars *__restrict__ sc) {
    if (sc->done) return;
    const T gam = (T)sc->gam;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        fi[i] = fi[i] + (X)(gam * zk[i]);
        res[i] = res[i] - gam * uk[i];
    }
}

// ------------------------------------------------- fused solver iterations

// the end of an iteration with ||r||_1 = a and ||r||_2^2 = b, sc->iters counting it:
// the status (kStatusRunning: go on), the same in every block
__device__ inline int end_test(const Scalars *sc, double a, double b, double &rsm, double &rel) {
    rsm = a / (sc->res0 + sc->small);
    rel = sc->stop_rule == 1 ? sqrt(b / sc->bnorm2) : sc->rel;
    const bool conv = sc->stop_rule == 0 ? rsm < sc->resmax : sc->stop_rule == 1 ? rel < sc->resmax : b <= sc->inner_tol2;
    if (!(isfinite(a) && isfinite(b))) return FC_ERR_NONFINITE;
    if (conv) return FC_OK;
    return sc->iters >= sc->nsw ? FC_NOT_CONVERGED : kStatusRunning;
}

__device__ inline void record_end(Scalars *sc, double a, double b, double rsm, double rel, int status) {
    sc->resl = a;
    sc->rnorm2 = b;
    sc->rsm = rsm;
    sc->rel = rel;
    if (status != kStatusRunning) {
        sc->done = 1;
        sc->status = status;
    }
}

// Whether the solve has ended, for a kernel whose first block may set `done` while others still
// begin: read once a block, so a block goes on or returns as a whole (one that goes on comes to
// the same end by its own test, and returns there).
__device__ inline bool ended(const Scalars *sc, int *sh) {
    if (threadIdx.x == 0) *sh = sc->done;
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(*sh) != 0;
}

// Partials of the fused vector kernels: block b's |r|_1, |r|_2^2 and r.z (or res.reso) at
// pv[kVecParts b ..]; one reduction adds what a kernel needs of them.
__device__ inline void vec_part(double *pv, double a, double b, double c) {
    double *p = pv + (size_t)kVecParts * blockIdx.x;
    p[0] = a;
    p[1] = b;
    p[2] = c;
}

// block sums of three values, valid in thread 0
__device__ inline void block_sum3(double &a, double &b, double &c, double *sh) {
    constexpr int kW = kRedBlock / kWave;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_down(a, off, kWave);
        b += __shfl_down(b, off, kWave);
        c += __shfl_down(c, off, kWave);
    }
    if ((threadIdx.x & (kWave - 1)) == 0) {
        const int w = threadIdx.x / kWave;
        sh[w] = a;
        sh[kW + w] = b;
        sh[2 * kW + w] = c;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        a = b = c = 0.0;
        for (int w = 0; w < kW; ++w) {
            a += sh[w];
            b += sh[kW + w];
            c += sh[2 * kW + w];
        }
    }
}

constexpr int kVecShared = 3 * (kRedBlock / kWave);

// Convergence test (not on the first call), bet = r.z / (r.z of the iteration before),
// p = z + bet p (src/iccg.f90:114-125).  JAC: z = r / d formed here, z then is r, and the
// partials of r.z are those of pv; otherwise they are pz's (nz of them).
template <class T, bool JAC>
__global__ __launch_bounds__(kRedBlock) void k_cg_p(int n, T *__restrict__ p, const T *__restrict__ z,
                                                   const T *__restrict__ d, Scalars *__restrict__ sc,
                                                   const double *__restrict__ pv, int nv,
                                                   const double *__restrict__ pz, int nz, int first) {
    __shared__ double sh[kVecShared];
    __shared__ int stop;
    if (ended(sc, &stop)) return;
    const bool rec = blockIdx.x == 0 && threadIdx.x == 0;
    double t[3];
    if (JAC || !first) parts_total<kRedBlock, 3, kVecParts>(pv, nv, sh, t);
    if (!first) {
        double rsm, rel;
        const int status = end_test(sc, t[0], t[1], rsm, rel);
        if (rec) record_end(sc, t[0], t[1], rsm, rel, status);
        if (status != kStatusRunning) return;
    }
    double rz[1] = {t[2]};
    if (!JAC) parts_total<kRedBlock, 1, 1>(pz, nz, sh, rz);
    const double bet64 = rz[0] / sc->sk;
    if (rec) {
        sc->sk_next = rz[0];
        sc->bet = bet64;
    }
    const T bet = (T)bet64;
    for (int i = blockIdx.x * kRedBlock + threadIdx.x; i < n; i += gridDim.x * kRedBlock)
        p[i] = (JAC ? z[i] / d[i] : z[i]) + bet * p[i];
}

// alf = r.z / p.q; x += alf p ; r -= alf q (src/iccg.f90:143-154); partials |r|, r^2 and,
// JAC, r.z of the next z = r / d.
template <class T, class X, bool JAC>
__global__ __launch_bounds__(kRedBlock) void k_cg_xr(int n, X *__restrict__ x, T *__restrict__ r,
                                                    const T *__restrict__ p, const T *__restrict__ q,
                                                    const T *__restrict__ d, Scalars *__restrict__ sc,
                                                    const double *__restrict__ pq, int nq, double *__restrict__ pv) {
    __shared__ double sh[kVecShared];
    if (sc->done) return;
    double pkapk[1];
    parts_total<kRedBlock, 1, 1>(pq, nq, sh, pkapk);
    const double sk = sc->sk_next, alf64 = sk / pkapk[0];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc->sk = sk;
        sc->pkapk = pkapk[0];
        sc->alf = alf64;
        sc->iters += 1;
    }
    const T alf = (T)alf64;
    double a = 0.0, b = 0.0, c = 0.0;
    for (int i = blockIdx.x * kRedBlock + threadIdx.x; i < n; i += gridDim.x * kRedBlock) {
        x[i] = x[i] + (X)(alf * p[i]);
        const T rv = r[i] - alf * q[i];
        r[i] = rv;
        a += fabs((double)rv);
        b += (double)rv * (double)rv;
        if (JAC) c += (double)rv * (double)(T)(rv / d[i]);
    }
    block_sum3(a, b, c, sh);
    if (threadIdx.x == 0) vec_part(pv, a, b, c);
}

// Convergence test (not on the first call), bet = res.reso, om = bet gam / (alf beto +
// small), pk = res + om (pk - alf uk) (src/bicgstab.f90:101-111)
template <class T>
__global__ __launch_bounds__(kRedBlock) void k_bi_p(int n, T *__restrict__ pk, const T *__restrict__ res,
                                                   const T *__restrict__ uk, Scalars *__restrict__ sc,
                                                   const double *__restrict__ pv, int nv, int first) {
    __shared__ double sh[kVecShared];
    __shared__ int stop;
    if (ended(sc, &stop)) return;
    const bool rec = blockIdx.x == 0 && threadIdx.x == 0;
    double t[3];
    parts_total<kRedBlock, 3, kVecParts>(pv, nv, sh, t);
    if (!first) {
        double rsm, rel;
        const int status = end_test(sc, t[0], t[1], rsm, rel);
        if (rec) record_end(sc, t[0], t[1], rsm, rel, status);
        if (status != kStatusRunning) return;
    }
    const double bet = t[2];
    const double om64 = (bet * sc->gam) / ((sc->alf * sc->beto) + sc->small);
    if (rec) {
        sc->om = om64;
        sc->sk_next = bet;
        sc->beto_next = bet;
    }
    const T om = (T)om64, alf = (T)sc->alf;
    for (int i = blockIdx.x * kRedBlock + threadIdx.x; i < n; i += gridDim.x * kRedBlock) {
        T t1 = alf * uk[i];
        t1 = pk[i] - t1;
        t1 = om * t1;
        pk[i] = res[i] + t1;
    }
}

// gam = bet / uk.reso; fi += gam zk ; res -= gam uk (src/bicgstab.f90:152-161)
template <class T, class X>
__global__ __launch_bounds__(kRedBlock) void k_bi_xr1(int n, X *__restrict__ fi, T *__restrict__ res,
                                                     const T *__restrict__ zk, const T *__restrict__ uk,
                                                     Scalars *__restrict__ sc, const double *__restrict__ pq, int nq) {
    __shared__ double sh[kVecShared];
    if (sc->done) return;
    double ukreso[1];
    parts_total<kRedBlock, 1, 1>(pq, nq, sh, ukreso);
    const double sk = sc->sk_next, gam64 = sk / ukreso[0];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc->ukreso = ukreso[0];
        sc->sk = sk;
        sc->gam = gam64;
        sc->beto = sc->beto_next;
    }
    const T gam = (T)gam64;
    for (int i = blockIdx.x * kRedBlock + threadIdx.x; i < n; i += gridDim.x * kRedBlock) {
        fi[i] = fi[i] + (X)(gam * zk[i]);
        res[i] = res[i] - gam * uk[i];
    }
}

// alf = vk.res / (vk.vk + small); fi += alf zk ; res -= alf vk (src/bicgstab.f90:200-208);
// partials |res|, res^2 and res.reso of the next iteration
template <class T, class X>
__global__ __launch_bounds__(kRedBlock) void k_bi_xr2(int n, X *__restrict__ fi, T *__restrict__ res,
                                                     const T *__restrict__ zk, const T *__restrict__ vk,
                                                     const T *__restrict__ reso, Scalars *__restrict__ sc,
                                                     const double *__restrict__ pvr, const double *__restrict__ pvv,
                                                     int nv, double *__restrict__ pv) {
    __shared__ double sh[kVecShared];
    if (sc->done) return;
    double vr[1], vv[1];
    parts_total<kRedBlock, 1, 1>(pvr, nv, sh, vr);
    parts_total<kRedBlock, 1, 1>(pvv, nv, sh, vv);
    const double alf64 = vr[0] / (vv[0] + sc->small);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc->vr = vr[0];
        sc->vv = vv[0];
        sc->alf = alf64;
        sc->iters += 1;
    }
    const T alf = (T)alf64;
    double a = 0.0, b = 0.0, c = 0.0;
    for (int i = blockIdx.x * kRedBlock + threadIdx.x; i < n; i += gridDim.x * kRedBlock) {
        fi[i] = fi[i] + (X)(alf * zk[i]);
        const T rv = res[i] - alf * vk[i];
        res[i] = rv;
        a += fabs((double)rv);
        b += (double)rv * (double)rv;
        c += (double)rv * (double)reso[i];
    }
    block_sum3(a, b, c, sh);
    if (threadIdx.x == 0) vec_part(pv, a, b, c);
}

// the SpMV's partials as one value each
__global__ __launch_bounds__(kFinBlock) void k_parts_one(int np, const double *__restrict__ pa,
                                                        const double *__restrict__ pb, double *__restrict__ out,
                                                        const Scalars *__restrict__ sc) {
    __shared__ double sh[kFinBlock / kWave];
    if (sc->done) return;
    double a[1], b[1] = {0.0};
    parts_total<kFinBlock, 1, 1>(pa, np, sh, a);
    if (pb) parts_total<kFinBlock, 1, 1>(pb, np, sh, b);
    if (threadIdx.x == 0) {
        out[0] = a[0];
        out[1] = b[0];
    }
}

// The first iteration's partials: x.y, or with d x.(y / d)
template <class T>
__global__ __launch_bounds__(kRedBlock) void k_first_dot(int n, const T *__restrict__ x, const T *__restrict__ y,
                                                         const T *__restrict__ d, const Scalars *__restrict__ sc,
                                                         double *__restrict__ pv) {
    __shared__ double sh[kVecShared];
    if (sc->done) return;
    double a = 0.0, b = 0.0, c = 0.0;
    for (int i = blockIdx.x * kRedBlock + threadIdx.x; i < n; i += gridDim.x * kRedBlock)
        c += (double)x[i] * (double)(d ? (T)(y[i] / d[i]) : y[i]);
    block_sum3(a, b, c, sh);
    if (threadIdx.x == 0) vec_part(pv, a, b, c);
}

// d = a(diag)
__global__ void k_diag(int n, const double *__restrict__ a, const int *__restrict__ diag, double *__restrict__ d) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) d[i] = a[diag[i]];
}

template <class T>
__global__ void k_copy(int n, const T *__restrict__ x, T *__restrict__ y) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) y[i] = x[i];
}

template <class T>
__global__ void k_zero(int n, T *__restrict__ y) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) y[i] = T(0);
}

template <class TI, class TO>
__global__ void k_cast(long long n, const TI *__restrict__ x, TO *__restrict__ y) {
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        y[i] = (TO)x[i];
}

// x(fp64) += scale * e(fp32)
__global__ void k_refine(int n, double *__restrict__ x, const float *__restrict__ e, double scale) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        x[i] = x[i] + scale * (double)e[i];
}

// r32 = (float)(r * inv): each inner solve sees a unit-norm right-hand side, so
// the algorithms' absolute guards (small) and FP32's range stay scale-free
__global__ void k_scale_cast(int n, const double *__restrict__ r, float *__restrict__ r32, double inv) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        r32[i] = (float)(r[i] * inv);
}

// ----------------------------------------------------------------- helpers

struct Ctx {
    fc_context *ctx;
    hipStream_t s;
    Workspace *ws;   // the context's workspace (null for the allocation-free solve)
    int n;
    Scalars *sc;
    double *pa, *pb;
    // fused iterations: the vector kernels' partials, r.z, the SpMV's, and the sums of those
    double *pv, *pz, *pq, *pq2, *one;
    int gv;   // grid of the vector kernels
    int gf;   // grid of the fused ones
    SweepCfg sw;   // how the triangular sweeps run
};

Scalars init_scalars(const SolveArgs &args, double small) {
    Scalars h;
    std::memset(&h, 0, sizeof(h));
    h.small = small;
    h.resmax = (args.variant == FC_VARIANT_TESTS) ? (double)1e-13f : args.sor;
    h.nsw = (args.variant == FC_VARIANT_TESTS) ? 100 : args.nsw;
    h.s0 = kS0;
    h.sk = kS0;   // fused iterations: the r.z before the first
    h.alf = 1.0;
    h.beto = 1.0;
    h.gam = 1.0;
    h.early_exit = (args.variant == FC_VARIANT_TESTS) ? 0 : 1;
    h.stop_rule = (args.variant == FC_VARIANT_TESTS) ? 0 : (args.stop_rule == FC_STOP_L2 ? 1 : 0);
    h.status = kStatusRunning;
    return h;
}

void upload_scalars(Ctx &c, const Scalars &h) {
    FC_HIP_CHECK(hipMemcpyAsync(c.sc, &h, sizeof(Scalars), hipMemcpyHostToDevice, c.s));
}

Scalars read_scalars(Ctx &c) {
    Scalars h;
    FC_HIP_CHECK(hipMemcpyAsync(&h, c.sc, sizeof(Scalars), hipMemcpyDeviceToHost, c.s));
    FC_HIP_CHECK(hipStreamSynchronize(c.s));
    return h;
}

int read_done(Ctx &c) {
    int *hf = c.ctx->host_flags;
    FC_HIP_CHECK(hipMemcpyAsync(hf, &c.sc->done, sizeof(int), hipMemcpyDeviceToHost, c.s));
    FC_HIP_CHECK(hipStreamSynchronize(c.s));
    return hf[0];
}

// the SpMV's partials (pq, and pq2 with two) as the fused kernels read them
struct SpmvSums {
    const double *a, *b;
    int n;
};
SpmvSums spmv_sums(Ctx &c, bool two) {
    const int gs = spmv_grid(c.n);
    if (gs <= kDirectParts) return {c.pq, c.pq2, gs};
    k_parts_one<<<1, kFinBlock, 0, c.s>>>(gs, c.pq, two ? c.pq2 : nullptr, c.one, c.sc);
    return {c.one, c.one + 1, 1};
}

// whether a solve's iterations are the fused ones
bool fused(const Ctx &c, const OcView &oc) { return !c.ctx->reduce_seq && !oc.noc; }

// four rows a thread where that still gives every CU two blocks
int fused_grid(int n) { return std::min(kVecGrid, grid_for(n, n >= 512 * 4 * kRedBlock ? 4 * kRedBlock : 2 * kRedBlock)); }

void fin(Ctx &c, int step, int nparts, bool two) {
    k_fin<<<1, kFinBlock, 0, c.s>>>(step, nparts, c.pa, nparts, two ? c.pb : nullptr, c.sc);
}

// Sums in index order, as the reference forms them (sum(res*zk), sum(abs(res)):
// one running sum from the first entry to the last, src/iccg.f90:65,114,143,154).
// One wave loads 64 terms at a time and adds them to the running sum one by one
// through lane broadcasts, so the sum has the reference's rounding; it goes to
// pa[0] (and pb[0]) for a finaliser that reads one partial.
//   OP 0: a = sum x_i y_i;  OP 1: a = sum |x_i|, b = sum x_i x_i;  OP 2: a = sum x_i y_i, b = sum y_i y_i
template <int OP>
__global__ __launch_bounds__(64) void k_seq_sum(int n, const double *__restrict__ x, const double *__restrict__ y,
                                                double *__restrict__ pa, double *__restrict__ pb,
                                                const Scalars *__restrict__ sc) {
    if (sc && sc->done) return;
    const int lane = threadIdx.x;
    double a = 0.0, b = 0.0;
    for (int base = 0; base < n; base += 64) {
        const int i = base + lane;
        double ta = 0.0, tb = 0.0;
        if (i < n) {
            const double xv = x[i];
            const double yv = OP == 1 ? 0.0 : y[i];
            ta = OP == 1 ? fabs(xv) : xv * yv;
            tb = OP == 1 ? xv * xv : yv * yv;
        }
        const int cnt = min(64, n - base);
        for (int l = 0; l < cnt; ++l) {
            a = a + __shfl(ta, l, 64);
            if (OP != 0) b = b + __shfl(tb, l, 64);
        }
    }
    if (lane == 0) {
        pa[0] = a;
        if (OP != 0) pb[0] = b;
    }
}

// The partial count for the finaliser of a reduction whose per-block partials
// the kernels just wrote: with sequential reductions (fc_set_reduction_order)
// the same sums are formed again in index order into one partial.
int seq_or(Ctx &c, int nparts, int op, const double *x, const double *y) {
    if (!c.ctx->reduce_seq) return nparts;
    if (op == 0) k_seq_sum<0><<<1, 64, 0, c.s>>>(c.n, x, y, c.pa, c.pb, c.sc);
    else if (op == 1) k_seq_sum<1><<<1, 64, 0, c.s>>>(c.n, x, y, c.pa, c.pb, c.sc);
    else k_seq_sum<2><<<1, 64, 0, c.s>>>(c.n, x, y, c.pa, c.pb, c.sc);
    return 1;
}

// b-norm^2 into sc->bnorm2 (host-side read; used by L2 stopping)
double norm2_host(Ctx &c, const double *v) {
    dot_launch64(c.s, c.n, v, v, c.pa);
    sum_parts_launch(c.s, red_grid(c.n), c.pa, nullptr, c.ws->sums.as<double>());
    double h[2];
    FC_HIP_CHECK(hipMemcpyAsync(h, c.ws->sums.get(), sizeof(double) * 2, hipMemcpyDeviceToHost, c.s));
    FC_HIP_CHECK(hipStreamSynchronize(c.s));
    return h[0];
}

// Runs `iter` until the device sets `done`, `per_graph` iterations captured into a HIP
// graph and `launches` of them a batch; the null stream cannot be captured, so it launches
// directly.  Between two graphs the GPU idles 5 to 7 us, inside one it does not: 8
// Jacobi-PCG iterations a graph instead of 1 (four launches a batch) took 24.5 against
// 27.7 ms on 97 x 83 x 61 (4: 25.7, 16: 24.1), 4 DIC-PCG iterations 10.8 against 11.4 ms
// on 40^3 (2: 11.1, 6: 10.9) and 1.60 against 1.73 ms on 20 x 20 x 1 (6: 1.68, 8: 1.75:
// what a batch launches past the end returns at once, but not for nothing).  One a graph
// where an iteration is many launches (level sweeps) or a solve few iterations (BiCGStab:
// 6.1 against 6.2 to 6.5 ms with 2 to 4), which a larger graph's set-up outweighs.
constexpr int kDirect = 5;
struct GraphExec {
    hipGraphExec_t exec = nullptr;
    ~GraphExec() { if (exec) (void)hipGraphExecDestroy(exec); }
};

struct Events {
    hipEvent_t e[2] = {nullptr, nullptr};
    Events() {
        for (hipEvent_t &x : e) FC_HIP_CHECK(hipEventCreateWithFlags(&x, hipEventDisableTiming));
    }
    ~Events() {
        for (hipEvent_t x : e)
            if (x) (void)hipEventDestroy(x);
    }
};

// The first `direct` iterations are launched one by one, and the graph is set up, while the
// last of them runs, only if the solve goes on after the others: a momentum or correction
// solve often ends there.  On 20 x 20 x 1 and 40^3 one DIC-PCG iteration through the host
// takes 0.37 and 0.66 ms, with the graph set up first 0.52 to 0.60 and 0.75 to 0.84.
// `kept`, when given, keeps the graph for the solve's next call with the same iterations
// (refinement cycles: 170 us a cycle to capture one at 128^3).
void run_batches(Ctx &c, int direct, int per_graph, int launches, const std::function<void()> &iter,
                 GraphExec *kept = nullptr) {
    GraphExec own;
    GraphExec &ge = kept ? *kept : own;
    // The flag of a batch is read while the next one runs, so the GPU does not idle for
    // the host's round trip (25 us a batch); past the end it finds `done` set and every
    // kernel returns.
    Events ev;
    int *flags = c.ctx->host_flags;
    int b = 0;   // batches launched
    auto flag = [&]() {
        FC_HIP_CHECK(hipGetLastError());
        FC_HIP_CHECK(hipMemcpyAsync(flags + (b & 1), &c.sc->done, sizeof(int), hipMemcpyDeviceToHost, c.s));
        FC_HIP_CHECK(hipEventRecord(ev.e[b & 1], c.s));
        ++b;
    };
    auto ended = [&](int batch) {
        FC_HIP_CHECK(hipEventSynchronize(ev.e[batch & 1]));
        return flags[batch & 1] != 0;
    };
    bool done = false;
    if (!ge.exec) {
        for (int k = 0; k < direct && !done; ++k) {
            iter();
            flag();
            done = b > 1 && ended(b - 2);
        }
        if (!done && c.ctx->use_graphs && c.s != nullptr) {
            hipGraph_t g = nullptr;
            FC_HIP_CHECK(hipStreamBeginCapture(c.s, hipStreamCaptureModeThreadLocal));
            try {
                for (int k = 0; k < per_graph; ++k) iter();
            } catch (...) {
                (void)hipStreamEndCapture(c.s, &g);
                if (g) (void)hipGraphDestroy(g);
                throw;
            }
            FC_HIP_CHECK(hipStreamEndCapture(c.s, &g));
            hipError_t e = hipGraphInstantiate(&ge.exec, g, nullptr, nullptr, 0);
            (void)hipGraphDestroy(g);
            FC_HIP_CHECK(e);
        }
    }
    while (!done) {
        for (int k = 0; k < (ge.exec ? launches : launches * per_graph); ++k) {
            if (ge.exec) FC_HIP_CHECK(hipGraphLaunch(ge.exec, c.s));
            else iter();
        }
        flag();
        done = b > 1 && ended(b - 2);
    }
    FC_HIP_CHECK(hipStreamSynchronize(c.s));
}

}  // namespace

void cast_d2f(hipStream_t s, long long n, const double *x, float *y) {
    k_cast<double, float><<<std::min(grid_for(n, 256), 8192), 256, 0, s>>>(n, x, y);
    FC_HIP_CHECK(hipGetLastError());
}

void Workspace::ensure(int n_, int nnz_) {
    const size_t D = sizeof(double) * (size_t)std::max(n_, 1), F = sizeof(float) * (size_t)std::max(n_, 1);
    for (DevBuf *b : {&r, &z, &p, &q, &x, &reso, &uk, &vk, &d, &tmp}) b->ensure(D);
    for (DevBuf *b : {&r32, &z32, &p32, &q32, &e32, &d32}) b->ensure(F);
    a32.ensure(sizeof(float) * (size_t)std::max(nnz_, 1));
    const int parts = std::max(kFcgM * kMaxRedGrid, spmv_grid(n_));   // kFcgM dot products at once (FCG)
    pa.ensure(sizeof(double) * parts);
    pb.ensure(sizeof(double) * parts);
    pv.ensure(sizeof(double) * kVecParts * kVecGrid);
    pz.ensure(sizeof(double) * kVecGrid);
    pq.ensure(sizeof(double) * spmv_grid(n_));
    pq2.ensure(sizeof(double) * spmv_grid(n_));
    sums.ensure(sizeof(double) * 4);
    sc.ensure(sizeof(Scalars));
    err.ensure(sizeof(int) * 4);
    sf.ensure(sizeof(SyncFree));
    sf_tmp.ensure(D);
    n = n_;
    nnz = nnz_;
}

static Ctx make_ctx(fc_context *ctx, int n) {
    Workspace &ws = *ctx->ws;
    Ctx c{ctx, ctx->stream, &ws, n, ws.sc.as<Scalars>(), ws.pa.as<double>(), ws.pb.as<double>(), ws.pv.as<double>(), ws.pz.as<double>(),
          ws.pq.as<double>(), ws.pq2.as<double>(), ws.sums.as<double>() + 2, red_grid(n), fused_grid(n), {}};
    return c;
}

static void setup_sweeps(Ctx &c, const Structure &st) {
    const SweepChoice ch = choose_sweeps(c.ctx, st);
    if (ch.dep) {
        syncfree_reset(c.ctx, c.s, c.ws->sf.as<SyncFree>());
        c.sw.sf = c.ws->sf.as<SyncFree>();
        c.sw.tmp = c.ws->sf_tmp.get();
        c.sw.waves = syncfree_wave_count(c.ctx, st);
        if (ch.parts) {
            c.ws->sf_tmp.ensure(sizeof(double) * (size_t)st.pt_npk);
            c.ws->sf_zp.ensure(sizeof(double) * (size_t)st.pt_npk);
            c.sw.tmp = c.ws->sf_tmp.get();
            c.sw.zp = c.ws->sf_zp.get();
            c.sw.parts = true;
            c.sw.waves = part_wave_count(c.ctx);
        }
    }
}

static void check_sweeps(Ctx &c) {
    if (!c.sw.sf) return;
    SyncFree h;
    FC_HIP_CHECK(hipMemcpyAsync(&h, c.sw.sf, sizeof(SyncFree), hipMemcpyDeviceToHost, c.s));
    FC_HIP_CHECK(hipStreamSynchronize(c.s));
    if (h.abort) throw Error(FC_ERR_HIP, "dependency-driven sweep: a wait exceeded its time limit");
}

// The factor (a, pivots d) in level-packed order for this solve's sweeps; empty
// (sweeps over the CSR rows) when the structure is not packed.
template <class T>
static PackedFactor<T> pack_for_solve(Ctx &c, const Structure &st, const T *a, const T *d) {
    PackedFactor<T> pf;
    if (!packed_sweeps(st)) return pf;
    Workspace &ws = *c.ws;
    constexpr bool f32 = sizeof(T) == sizeof(float);
    DevBuf &af = f32 ? ws.pk_af32 : ws.pk_af, &df = f32 ? ws.pk_df32 : ws.pk_df;
    DevBuf &ab = f32 ? ws.pk_ab32 : ws.pk_ab, &db = f32 ? ws.pk_db32 : ws.pk_db;
    if (c.sw.parts) {
        af.ensure(sizeof(T) * part_factor_count(st, false));
        ab.ensure(sizeof(T) * part_factor_count(st, true));
        T *tmp = static_cast<T *>(c.sw.tmp);
        if constexpr (f32) pack_factor_parts32(c.s, st, a, d, af.as<float>(), ab.as<float>(), tmp);
        else pack_factor_parts64(c.s, st, a, d, af.as<double>(), ab.as<double>(), tmp);
        pf.af = af.as<T>();
        pf.ab = ab.as<T>();
        return pf;
    }
    if (c.sw.sf) {
        T *tmp = static_cast<T *>(c.sw.tmp);
        if constexpr (f32) mark_sweep_input32(c.s, st.n, tmp);
        else mark_sweep_input64(c.s, st.n, tmp);
    }
    const size_t n = (size_t)st.n;
    af.ensure(sizeof(T) * n * (size_t)st.ell_f);
    ab.ensure(sizeof(T) * n * (size_t)st.ell_b);
    df.ensure(sizeof(T) * n);
    db.ensure(sizeof(T) * n);
    if constexpr (f32)
        pack_factor32(c.s, st, a, d, af.as<float>(), df.as<float>(), ab.as<float>(), db.as<float>());
    else
        pack_factor64(c.s, st, a, d, af.as<double>(), df.as<double>(), ab.as<double>(), db.as<double>());
    pf.af = af.as<T>();
    pf.df = df.as<T>();
    pf.ab = ab.as<T>();
    pf.db = db.as<T>();
    return pf;
}

// The matrix of a solve as its iterations multiply by it: in slices where the structure has
// them, else the CSR arrays.
template <class T> struct Matrix {
    SliceView S;
    const T *v = nullptr;          // sliced values
    const int *ptr, *ja;
    const T *a = nullptr;          // CSR values
};
static Matrix<double> matrix64(Ctx &c, const Structure &st, const double *a) {
    Matrix<double> A{{}, nullptr, st.ioffset.as<int>(), st.ja.as<int>(), a};
    A.S = slices_for(c.ctx, const_cast<Structure &>(st));
    if (A.S.w) {
        c.ws->as64.ensure(sizeof(double) * slice_count(st.n, A.S));
        slice_values64(c.s, st.n, A.S, a, c.ws->as64.as<double>());
        A.v = c.ws->as64.as<double>();
    }
    return A;
}
// csr: the FP32 CSR values are wanted too
static Matrix<float> matrix32(Ctx &c, const Structure &st, const double *a, bool csr) {
    Matrix<float> A{{}, nullptr, st.ioffset.as<int>(), st.ja.as<int>(), c.ws->a32.as<float>()};
    A.S = slices_for(c.ctx, const_cast<Structure &>(st));
    if (A.S.w) {
        c.ws->as32.ensure(sizeof(float) * slice_count(st.n, A.S));
        slice_values32(c.s, st.n, A.S, a, c.ws->as32.as<float>());
        A.v = c.ws->as32.as<float>();
    }
    if (csr || !A.S.w)
        k_cast<double, float><<<std::min(grid_for(st.nnz, 256), 8192), 256, 0, c.s>>>(st.nnz, a,
                                                                                     c.ws->a32.as<float>());
    return A;
}
// y = A x with partials of y.b (pa) and, with pb, of y.y
static void product(Ctx &c, const Matrix<double> &A, const double *x, const double *b, double *y, double *pa,
                    double *pb = nullptr) {
    if (A.S.w) sliced_product64(c.s, c.n, A.S, A.v, x, b, y, pa, pb, c.sc);
    else spmv_launch64(c.s, pb ? 3 : 2, c.n, A.ptr, A.ja, A.a, x, nullptr, b, y, nullptr, pa, pb, c.sc);
}
static void product(Ctx &c, const Matrix<float> &A, const float *x, const float *b, float *y, double *pa,
                    double *pb = nullptr) {
    if (A.S.w) sliced_product32(c.s, c.n, A.S, A.v, x, b, y, pa, pb, c.sc);
    else spmv_launch32(c.s, pb ? 3 : 2, c.n, A.ptr, A.ja, A.a, x, nullptr, b, y, pa, pb, c.sc);
}

static void check_pivots(Ctx &c) {
    int h = 0;
    FC_HIP_CHECK(hipMemcpyAsync(&h, c.ws->err.get(), sizeof(int), hipMemcpyDeviceToHost, c.s));
    FC_HIP_CHECK(hipStreamSynchronize(c.s));
    if (h) throw Error(FC_ERR_ZERO_PIVOT, "incomplete factorisation: zero or non-finite pivot");
}

double true_rel_l2(fc_context *ctx, const SolveArgs &args) {
    Workspace &ws = *ctx->ws;
    const Structure &st = *args.st;
    Ctx c = make_ctx(ctx, st.n);
    double *r = ws.tmp.as<double>();
    spmv_launch64(c.s, 1, st.n, st.ioffset.as<int>(), st.ja.as<int>(), args.a, args.fi, args.su, nullptr, r, nullptr,
                  c.pa, c.pb, nullptr);
    if (args.oc.noc) oc_launch64(c.s, st.n, args.oc, args.fi, r, -1, nullptr);
    double rr = norm2_host(c, r);
    double bb = norm2_host(c, args.su);
    return bb > 0 ? std::sqrt(rr / bb) : std::sqrt(rr);
}

static void fill_info(fc_solve_info *info, const Scalars &h, double setup_ms, double solve_ms) {
    if (!info) return;
    info->res0 = h.res0;
    info->resl = h.resl;
    info->rsm = h.rsm;
    info->iters = h.iters;
    info->status = h.status;
    info->setup_ms = setup_ms;
    info->solve_ms = solve_ms;
}

// Initial residual r = su - A fi (+ O-C), norms, early exit.
static void initial_residual(Ctx &c, const SolveArgs &args, double *r) {
    const Structure &st = *args.st;
    if (!args.oc.noc) {
        spmv_launch64(c.s, 1, c.n, st.ioffset.as<int>(), st.ja.as<int>(), args.a, args.fi, args.su, nullptr, r,
                      nullptr, c.pa, c.pb, nullptr);
        fin(c, kFinRes0, seq_or(c, spmv_grid(c.n), 1, r, nullptr), true);
    } else {
        spmv_launch64(c.s, 1, c.n, st.ioffset.as<int>(), st.ja.as<int>(), args.a, args.fi, args.su, nullptr, r,
                      nullptr, c.pa, c.pb, nullptr);
        oc_launch64(c.s, c.n, args.oc, args.fi, r, -1, nullptr);
        norms_launch64(c.s, c.n, r, c.pa, c.pb);
        fin(c, kFinRes0, seq_or(c, red_grid(c.n), 1, r, nullptr), true);
    }
}

fc_status solve_pcg64(fc_context *ctx, const SolveArgs &args, bool dic, fc_solve_info *info) {
    const Structure &st = *args.st;
    Workspace &ws = *ctx->ws;
    Ctx c = make_ctx(ctx, st.n);
    setup_sweeps(c, st);
    const int n = st.n;
    const double small = args.variant == FC_VARIANT_TESTS ? kSmallTests : kSmallSrc;
    double *r = ws.r.as<double>(), *z = ws.z.as<double>(), *p = ws.p.as<double>(), *q = ws.q.as<double>();
    double *d = ws.d.as<double>();
    const bool fuse = fused(c, args.oc);
    Scalars h = init_scalars(args, small);
    if (h.stop_rule == 1) h.bnorm2 = norm2_host(c, args.su);
    ctx->timer.start(c.s);
    upload_scalars(c, h);
    k_zero<double><<<c.gv, 256, 0, c.s>>>(n, p);
    FC_HIP_CHECK(hipMemsetAsync(ws.err.get(), 0, sizeof(int), c.s));
    initial_residual(c, args, r);
    PackedFactor<double> pf;
    if (dic) {
        pivots_launch(c.s, st, args.a, d, false, ws.err.as<int>(), &c.sw);
        pf = pack_for_solve<double>(c, st, args.a, d);
    }
    double setup_ms = ctx->timer.stop_ms(c.s);
    if (dic) check_pivots(c);
    if (read_done(c)) {
        Scalars hs = read_scalars(c);
        fill_info(info, hs, setup_ms, 0.0);
        return (fc_status)hs.status;
    }
    const int *ptr = st.ioffset.as<int>(), *ja = st.ja.as<int>(), *dg = st.diag.as<int>();
    const int gs = spmv_grid(n);
    ctx->timer.start(c.s);
    if (fuse) {
        const Matrix<double> A = matrix64(c, st, args.a);
        if (!dic) k_diag<<<c.gv, 256, 0, c.s>>>(n, args.a, dg, z);   // z holds the diagonal
        auto precondition = [&](int first) {
            if (dic) {
                lu_launch64(c.s, st, args.a, d, small, r, z, c.sc, &c.sw, pf.af ? &pf : nullptr);
                k_dot<double><<<c.gf, kRedBlock, 0, c.s>>>(n, r, z, c.sc, c.pz);
                k_cg_p<double, false><<<c.gf, kRedBlock, 0, c.s>>>(n, p, z, nullptr, c.sc, c.pv, c.gf, c.pz, c.gf, first);
            } else {
                if (first) k_first_dot<double><<<c.gf, kRedBlock, 0, c.s>>>(n, r, r, z, c.sc, c.pv);
                k_cg_p<double, true><<<c.gf, kRedBlock, 0, c.s>>>(n, p, r, z, c.sc, c.pv, c.gf, nullptr, 0, first);
            }
        };
        precondition(1);
        const bool level = dic && !c.sw.sf;
        run_batches(c, level ? 0 : kDirect, level ? 1 : dic ? 4 : 8, 1, [&]() {
            product(c, A, p, p, q, c.pq);
            const SpmvSums pq = spmv_sums(c, false);
            if (dic)
                k_cg_xr<double, double, false><<<c.gf, kRedBlock, 0, c.s>>>(n, args.fi, r, p, q, nullptr, c.sc, pq.a,
                                                                           pq.n, c.pv);
            else
                k_cg_xr<double, double, true><<<c.gf, kRedBlock, 0, c.s>>>(n, args.fi, r, p, q, z, c.sc, pq.a, pq.n,
                                                                          c.pv);
            precondition(0);
        });
        const double solve_ms = ctx->timer.stop_ms(c.s);
        check_sweeps(c);
        Scalars hs = read_scalars(c);
        fill_info(info, hs, setup_ms, solve_ms);
        return (fc_status)hs.status;
    }
    auto iter = [&]() {
        if (dic) {
            lu_launch64(c.s, st, args.a, d, small, r, z, c.sc, &c.sw, pf.af ? &pf : nullptr);
            k_dot<double><<<c.gv, kRedBlock, 0, c.s>>>(n, r, z, c.sc, c.pa);
        } else {
            k_jacobi<double, double><<<c.gv, kRedBlock, 0, c.s>>>(n, r, args.a, dg, z, c.sc, c.pa);
        }
        fin(c, kFinSk, seq_or(c, c.gv, 0, r, z), false);
        k_p_update<double><<<c.gv, 256, 0, c.s>>>(n, p, z, c.sc);
        if (!args.oc.noc) {
            spmv_launch64(c.s, 2, n, ptr, ja, args.a, p, nullptr, p, q, nullptr, c.pa, nullptr, c.sc);
            fin(c, kFinAlf, seq_or(c, gs, 0, p, q), false);
        } else {
            spmv_launch64(c.s, 0, n, ptr, ja, args.a, p, nullptr, nullptr, q, nullptr, c.pa, nullptr, c.sc);
            oc_launch64(c.s, n, args.oc, p, q, +1, c.sc);
            k_dot<double><<<c.gv, kRedBlock, 0, c.s>>>(n, p, q, c.sc, c.pa);
            fin(c, kFinAlf, seq_or(c, c.gv, 0, p, q), false);
        }
        k_pcg_xr64<<<c.gv, kRedBlock, 0, c.s>>>(n, args.fi, r, p, q, c.sc, c.pa, c.pb);
        fin(c, kFinPcgEnd, seq_or(c, c.gv, 1, r, nullptr), true);
    };
    const bool level = dic && !c.sw.sf;
    run_batches(c, level ? 0 : kDirect, 1, level ? 1 : dic ? 2 : 4, iter);
    double solve_ms = ctx->timer.stop_ms(c.s);
    check_sweeps(c);
    Scalars hs = read_scalars(c);
    fill_info(info, hs, setup_ms, solve_ms);
    return (fc_status)hs.status;
}

fc_status solve_bicgstab64(fc_context *ctx, const SolveArgs &args, fc_solve_info *info) {
    const Structure &st = *args.st;
    Workspace &ws = *ctx->ws;
    Ctx c = make_ctx(ctx, st.n);
    setup_sweeps(c, st);
    const int n = st.n;
    const double small = args.variant == FC_VARIANT_TESTS ? kSmallTests : kSmallSrc;
    double *res = ws.r.as<double>(), *reso = ws.reso.as<double>(), *pk = ws.p.as<double>();
    double *uk = ws.uk.as<double>(), *zk = ws.z.as<double>(), *vk = ws.vk.as<double>(), *d = ws.d.as<double>();
    build_tpos(ctx, const_cast<Structure &>(st));
    Scalars h = init_scalars(args, small);
    if (h.stop_rule == 1) h.bnorm2 = norm2_host(c, args.su);
    ctx->timer.start(c.s);
    upload_scalars(c, h);
    FC_HIP_CHECK(hipMemsetAsync(ws.err.get(), 0, sizeof(int), c.s));
    initial_residual(c, args, res);
    pivots_launch(c.s, st, args.a, d, true, ws.err.as<int>(), &c.sw);
    const PackedFactor<double> pf = pack_for_solve<double>(c, st, args.a, d);
    const PackedFactor<double> *ppf = pf.af ? &pf : nullptr;
    k_copy<double><<<c.gv, 256, 0, c.s>>>(n, res, reso);
    k_zero<double><<<c.gv, 256, 0, c.s>>>(n, pk);
    k_zero<double><<<c.gv, 256, 0, c.s>>>(n, uk);
    double setup_ms = ctx->timer.stop_ms(c.s);
    check_pivots(c);
    if (read_done(c)) {
        Scalars hs = read_scalars(c);
        fill_info(info, hs, setup_ms, 0.0);
        return (fc_status)hs.status;
    }
    const int *ptr = st.ioffset.as<int>(), *ja = st.ja.as<int>();
    const int gs = spmv_grid(n);
    ctx->timer.start(c.s);
    if (!c.ctx->reduce_seq) {   // (the reference's BiCGStab applies its O-C couplings to the initial residual alone)
        const Matrix<double> A = matrix64(c, st, args.a);
        auto direction = [&](int first) {
            k_bi_p<double><<<c.gf, kRedBlock, 0, c.s>>>(n, pk, res, uk, c.sc, c.pv, c.gf, first);
        };
        k_first_dot<double><<<c.gf, kRedBlock, 0, c.s>>>(n, res, reso, nullptr, c.sc, c.pv);
        direction(1);
        run_batches(c, c.sw.sf ? kDirect : 0, 1, c.sw.sf ? 2 : 1, [&]() {
            lu_launch64(c.s, st, args.a, d, small, pk, zk, c.sc, &c.sw, ppf);
            product(c, A, zk, reso, uk, c.pq);
            const SpmvSums ur = spmv_sums(c, false);
            k_bi_xr1<double, double><<<c.gf, kRedBlock, 0, c.s>>>(n, args.fi, res, zk, uk, c.sc, ur.a, ur.n);
            lu_launch64(c.s, st, args.a, d, small, res, zk, c.sc, &c.sw, ppf);
            product(c, A, zk, res, vk, c.pq, c.pq2);
            const SpmvSums v = spmv_sums(c, true);
            k_bi_xr2<double, double><<<c.gf, kRedBlock, 0, c.s>>>(n, args.fi, res, zk, vk, reso, c.sc, v.a, v.b, v.n,
                                                                 c.pv);
            direction(0);
        });
        const double solve_ms = ctx->timer.stop_ms(c.s);
        check_sweeps(c);
        Scalars hs = read_scalars(c);
        fill_info(info, hs, setup_ms, solve_ms);
        return (fc_status)hs.status;
    }
    auto iter = [&]() {
        k_dot<double><<<c.gv, kRedBlock, 0, c.s>>>(n, res, reso, c.sc, c.pa);
        fin(c, kFinBet, seq_or(c, c.gv, 0, res, reso), false);
        k_bicg_p<double><<<c.gv, 256, 0, c.s>>>(n, pk, res, uk, c.sc);
        lu_launch64(c.s, st, args.a, d, small, pk, zk, c.sc, &c.sw, ppf);
        spmv_launch64(c.s, 2, n, ptr, ja, args.a, zk, nullptr, reso, uk, nullptr, c.pa, nullptr, c.sc);
        fin(c, kFinGam, seq_or(c, gs, 0, uk, reso), false);
        k_bicg_xr1<double, double><<<c.gv, 256, 0, c.s>>>(n, args.fi, res, zk, uk, c.sc);
        lu_launch64(c.s, st, args.a, d, small, res, zk, c.sc, &c.sw, ppf);
        spmv_launch64(c.s, 3, n, ptr, ja, args.a, zk, nullptr, res, vk, nullptr, c.pa, c.pb, c.sc);
        fin(c, kFinAlfB, seq_or(c, gs, 2, res, vk), true);
        k_pcg_xr64<<<c.gv, kRedBlock, 0, c.s>>>(n, args.fi, res, zk, vk, c.sc, c.pa, c.pb);
        fin(c, kFinBicgEnd, seq_or(c, c.gv, 1, res, nullptr), true);
    };
    run_batches(c, c.sw.sf ? kDirect : 0, 1, c.sw.sf ? 2 : 1, iter);
    double solve_ms = ctx->timer.stop_ms(c.s);
    check_sweeps(c);
    Scalars hs = read_scalars(c);
    fill_info(info, hs, setup_ms, solve_ms);
    return (fc_status)hs.status;
}

// FP32 inner solve of A e = r32 to ||r_inner||_2 <= eta ||r32||_2, e32 out.
// s0_carry (PCG only, may be null): on entry the r.z of the previous cycle's last
// iteration (<= 0: none), on exit this cycle's.  With a previous value the search
// direction p is kept and the first step continues it (beta = r.z / s0_carry), so
// the refinement replaces the residual without discarding the Krylov direction.
static int inner_solve32(Ctx &c, const Structure &st, const Matrix<float> &A, bool bicg, double eta, double r32norm2,
                         int cap, const PackedFactor<float> *pf, double *s0_carry, GraphExec &graph) {
    Workspace &ws = *c.ws;
    const int n = c.n;
    float *a32 = ws.a32.as<float>(), *d32 = ws.d32.as<float>();
    float *r = ws.r32.as<float>(), *z = ws.z32.as<float>(), *p = ws.p32.as<float>(), *q = ws.q32.as<float>();
    float *e = ws.e32.as<float>();
    const float small = (float)kSmallSrc;
    Scalars h;
    std::memset(&h, 0, sizeof(h));
    const bool keep = !bicg && s0_carry && *s0_carry > 0.0;
    h.small = kSmallSrc;
    h.sk = keep ? *s0_carry : kS0;
    h.alf = 1.0;
    h.beto = 1.0;
    h.gam = 1.0;
    h.nsw = cap;
    h.stop_rule = 2;
    h.inner_tol2 = eta * eta * r32norm2;
    h.res0 = std::sqrt(r32norm2);
    h.status = kStatusRunning;
    upload_scalars(c, h);
    k_zero<float><<<c.gv, 256, 0, c.s>>>(n, e);
    if (!keep) k_zero<float><<<c.gv, 256, 0, c.s>>>(n, p);
    if (!bicg) {
        auto precondition = [&](int first) {
            lu_launch32(c.s, st, a32, d32, small, r, z, c.sc, &c.sw, pf);
            k_dot<float><<<c.gf, kRedBlock, 0, c.s>>>(n, r, z, c.sc, c.pz);
            k_cg_p<float, false><<<c.gf, kRedBlock, 0, c.s>>>(n, p, z, nullptr, c.sc, c.pv, c.gf, c.pz, c.gf, first);
        };
        precondition(1);
        run_batches(c, c.sw.sf ? kDirect : 0, c.sw.sf ? 4 : 1, 1, [&]() {
            product(c, A, p, p, q, c.pq);
            const SpmvSums pq = spmv_sums(c, false);
            k_cg_xr<float, float, false><<<c.gf, kRedBlock, 0, c.s>>>(n, e, r, p, q, nullptr, c.sc, pq.a, pq.n, c.pv);
            precondition(0);
        }, &graph);
    } else {
        float *reso = reinterpret_cast<float *>(ws.tmp.get());   // n floats fit in n doubles
        float *uk = q, *vk = reinterpret_cast<float *>(ws.vk.get());
        k_copy<float><<<c.gv, 256, 0, c.s>>>(n, r, reso);
        k_zero<float><<<c.gv, 256, 0, c.s>>>(n, uk);
        auto direction = [&](int first) {
            k_bi_p<float><<<c.gf, kRedBlock, 0, c.s>>>(n, p, r, uk, c.sc, c.pv, c.gf, first);
        };
        k_first_dot<float><<<c.gf, kRedBlock, 0, c.s>>>(n, r, reso, nullptr, c.sc, c.pv);
        direction(1);
        run_batches(c, c.sw.sf ? kDirect : 0, 1, c.sw.sf ? 2 : 1, [&]() {
            lu_launch32(c.s, st, a32, d32, small, p, z, c.sc, &c.sw, pf);
            product(c, A, z, reso, uk, c.pq);
            const SpmvSums ur = spmv_sums(c, false);
            k_bi_xr1<float, float><<<c.gf, kRedBlock, 0, c.s>>>(n, e, r, z, uk, c.sc, ur.a, ur.n);
            lu_launch32(c.s, st, a32, d32, small, r, z, c.sc, &c.sw, pf);
            product(c, A, z, r, vk, c.pq, c.pq2);
            const SpmvSums v = spmv_sums(c, true);
            k_bi_xr2<float, float><<<c.gf, kRedBlock, 0, c.s>>>(n, e, r, z, vk, reso, c.sc, v.a, v.b, v.n, c.pv);
            direction(0);
        }, &graph);
    }
    Scalars hs = read_scalars(c);
    if (s0_carry) *s0_carry = bicg || hs.status != FC_OK ? 0.0 : hs.sk;
    return hs.iters;
}

fc_status solve_mixed(fc_context *ctx, const SolveArgs &args, bool bicg, fc_solve_info *info) {
    const Structure &st = *args.st;
    Workspace &ws = *ctx->ws;
    Ctx c = make_ctx(ctx, st.n);
    setup_sweeps(c, st);
    const int n = st.n;
    double *r = ws.r.as<double>(), *d = ws.d.as<double>();
    // set-up: FP64 pivots, FP32 copies of the matrix and pivots
    ctx->timer.start(c.s);
    FC_HIP_CHECK(hipMemsetAsync(ws.err.get(), 0, sizeof(int), c.s));
    if (bicg) build_tpos(ctx, const_cast<Structure &>(st));
    pivots_launch(c.s, st, args.a, d, bicg, ws.err.as<int>(), &c.sw);
    const Matrix<float> A = matrix32(c, st, args.a, true);
    k_cast<double, float><<<c.gv, 256, 0, c.s>>>(n, d, ws.d32.as<float>());
    const PackedFactor<float> pf = pack_for_solve<float>(c, st, ws.a32.as<float>(), ws.d32.as<float>());
    double setup_ms = ctx->timer.stop_ms(c.s);
    check_pivots(c);
    Scalars h0 = init_scalars(args, kSmallSrc);
    h0.bnorm2 = norm2_host(c, args.su);
    const double bnorm = std::sqrt(h0.bnorm2);
    const bool l2 = args.stop_rule == FC_STOP_L2;
    int total_inner = 0, outer = 0;
    double res0 = 0.0, resl = 0.0, rel = 0.0;
    double scale = 1.0, s0c = 0.0;   // FP32 residual scale; r.z carried between PCG cycles
    GraphExec graph;                 // the inner iterations, the same in every cycle
    fc_status status = FC_NOT_CONVERGED;
    ctx->timer.start(c.s);
    for (;;) {
        // FP64 refinement residual r = su - A fi, its FP32 copy, L1 and L2 norms
        h0.done = 0;
        upload_scalars(c, h0);
        spmv_launch64(c.s, 1, n, st.ioffset.as<int>(), st.ja.as<int>(), args.a, args.fi, args.su, nullptr, r,
                      nullptr, c.pa, c.pb, nullptr);
        fin(c, kFinOuter, spmv_grid(n), true);
        Scalars ho = read_scalars(c);
        if (outer == 0) res0 = ho.resl;
        resl = ho.resl;
        rel = bnorm > 0 ? std::sqrt(ho.rnorm2) / bnorm : std::sqrt(ho.rnorm2);
        if (!std::isfinite(rel)) { status = FC_ERR_NONFINITE; break; }
        bool conv = l2 ? rel < args.sor : (res0 > 0 ? resl / (res0 + kSmallSrc) < args.sor : true);
        if (conv) { status = FC_OK; break; }
        if (outer >= args.max_outer || total_inner >= args.nsw) { status = FC_NOT_CONVERGED; break; }
        int cap = std::max(1, args.nsw - total_inner);
        // PCG: every cycle's FP32 residual is scaled by the first cycle's norm, so that the
        // kept search direction and r.z stay on one scale; BiCGStab: each cycle starts
        // afresh on a unit-norm right-hand side
        const double rn = std::sqrt(ho.rnorm2);
        if (outer == 0 || bicg) scale = rn;
        k_scale_cast<<<c.gv, 256, 0, c.s>>>(n, r, ws.r32.as<float>(), 1.0 / scale);
        total_inner += inner_solve32(c, st, A, bicg, args.inner_eta, ho.rnorm2 / (scale * scale), cap,
                                     pf.af ? &pf : nullptr, &s0c, graph);
        k_refine<<<c.gv, 256, 0, c.s>>>(n, args.fi, ws.e32.as<float>(), scale);
        ++outer;
    }
    double solve_ms = ctx->timer.stop_ms(c.s);
    check_sweeps(c);
    if (info) {
        info->res0 = res0;
        info->resl = resl;
        info->rsm = res0 > 0 ? resl / (res0 + kSmallSrc) : 0.0;
        info->iters = total_inner;
        info->outer = outer;
        info->status = status;
        info->setup_ms = setup_ms;
        info->solve_ms = solve_ms;
    }
    return status;
}

// Directions kept by flexible CG: the context's setting rounded up to a window
// the kernels are compiled for (4, 8, 12 or 16); by default 4 with the coarse
// correction (192^3: 104 iterations with 4, 8 or 12 kept, 4 the cheapest) and 12
// without it (416 iterations against 512 with 4).  The ring buffers hold exactly
// this many slots, and every kernel and finaliser uses the same count.
// Iterations per network application: the context's setting, by default 2 with
// the coarse correction (192^3: 130 iterations, every second one without the
// network, against 104 with it every time, and 15 % less time) and 1 without it.
static int fcg_network_period(const fc_context *ctx) {
    return ctx->fcg_net_period > 0 ? ctx->fcg_net_period : ctx->fcg_coarse > 0 ? 2 : 1;
}

static int fcg_window(const fc_context *ctx) {
    const int m = ctx->fcg_m > 0 ? ctx->fcg_m : ctx->fcg_coarse > 0 ? 4 : 12;
    return m <= 4 ? 4 : m <= 8 ? 8 : m <= 12 ? 12 : 16;
}

// Truncated FCG in FP32 on A e = r32 (unit-norm r32), preconditioner P.
// Returns the inner status (FC_OK, FC_NOT_CONVERGED, FC_FALLBACK_USED on
// stagnation, FC_ERR_NONFINITE) and adds the iterations to `iters`.
static int inner_fcg32(Ctx &c, const Matrix<float> &A, const PrecondHook &P, double eta, int cap, int &iters,
                       GraphExec &graph) {
    Workspace &ws = *c.ws;
    const int n = c.n;
    float *r = ws.r32.as<float>(), *z = ws.z32.as<float>(), *p = ws.p32.as<float>(), *q = ws.q32.as<float>();
    float *e = ws.e32.as<float>(), *ph = ws.ph.as<float>(), *qh = ws.qh.as<float>();
    const int gs = spmv_grid(n);
    Scalars h;
    std::memset(&h, 0, sizeof(h));
    h.small = kSmallSrc;
    h.nsw = cap;
    h.stop_rule = 2;
    h.inner_tol2 = eta * eta;
    h.res0 = 1.0;
    h.stag_ref = 1e300;    // set by the first window
    h.stag_min = 1e300;
    h.stag_every = c.ctx->fcg_stag_window;
    h.stag_factor = c.ctx->fcg_stag_factor;
    h.fcg_m = fcg_window(c.ctx);
    h.status = kStatusRunning;
    upload_scalars(c, h);
    k_zero<float><<<c.gv, 256, 0, c.s>>>(n, e);
    // the window is compiled in (h.fcg_m is one of 4, 8, 12, 16: fcg_window)
    const int gd = h.fcg_m <= kFcgFold ? c.gf : c.gv;
    auto dots = [&]() {
        switch (h.fcg_m) {
        case 4: k_fcg_dots<4><<<gd, kRedBlock, 0, c.s>>>(n, z, qh, c.sc, c.pa); break;
        case 8: k_fcg_dots<8><<<gd, kRedBlock, 0, c.s>>>(n, z, qh, c.sc, c.pa); break;
        case 12: k_fcg_dots<12><<<gd, kRedBlock, 0, c.s>>>(n, z, qh, c.sc, c.pa); break;
        default: k_fcg_dots<16><<<gd, kRedBlock, 0, c.s>>>(n, z, qh, c.sc, c.pa); break;
        }
        if (h.fcg_m > kFcgFold) fin(c, kFinFcgBeta, gd, false);
    };
    auto pupd = [&]() {   // the partials of p.r go to pb
        switch (h.fcg_m) {
        case 4: k_fcg_p<4><<<gd, kRedBlock, 0, c.s>>>(n, p, z, r, ph, c.sc, c.pa, gd, c.pb); break;
        case 8: k_fcg_p<8><<<gd, kRedBlock, 0, c.s>>>(n, p, z, r, ph, c.sc, nullptr, 0, c.pb); break;
        case 12: k_fcg_p<12><<<gd, kRedBlock, 0, c.s>>>(n, p, z, r, ph, c.sc, nullptr, 0, c.pb); break;
        default: k_fcg_p<16><<<gd, kRedBlock, 0, c.s>>>(n, p, z, r, ph, c.sc, nullptr, 0, c.pb); break;
        }
    };
    // The network runs on the first of every `period` iterations; the others take the
    // Jacobi guess in its place (flexible CG allows a preconditioner that changes from
    // one iteration to the next).  One captured graph holds `period` iterations.
    const int period = fcg_network_period(c.ctx);
    bool light = false;
    auto iter = [&]() {
        P.apply(P.obj, c.s, r, z, c.sc, light);
        dots();
        pupd();
        product(c, A, p, p, q, c.pq);
        k_fin<<<1, kFinBlock, 0, c.s>>>(kFinFcgAlf, gs, c.pq, gd, c.pb, c.sc);
        k_fcg_xr<<<c.gv, kRedBlock, 0, c.s>>>(n, e, r, p, q, ph, qh, c.sc, c.pa, c.pb);
        fin(c, kFinFcgEnd, c.gv, true);
    };
    auto group = [&]() {
        for (int k = 0; k < period; ++k) {
            light = k > 0;
            iter();
        }
    };
    run_batches(c, 1 + (kDirect + period - 2) / period, 1, std::max(1, 2 / period), group, &graph);
    Scalars hs = read_scalars(c);
    iters += hs.iters;
    return hs.status;
}

fc_status solve_fcg(fc_context *ctx, const SolveArgs &args, const PrecondHook &P, fc_solve_info *info) {
    FC_REQUIRE(P.apply != nullptr, FC_ERR_ARGUMENT, "no network attached (fc_sys_set_network)");
    const Structure &st = *args.st;
    Workspace &ws = *ctx->ws;
    Ctx c = make_ctx(ctx, st.n);
    const int n = st.n;
    double *r = ws.r.as<double>(), *xgood = ws.tmp.as<double>();
    const int m = fcg_window(ctx);
    ws.ph.ensure(sizeof(float) * (size_t)m * (size_t)n);
    ws.qh.ensure(sizeof(float) * (size_t)m * (size_t)n);
    ctx->timer.start(c.s);
    const Matrix<float> A = matrix32(c, st, args.a, false);
    double setup_ms = ctx->timer.stop_ms(c.s);
    Scalars h0 = init_scalars(args, kSmallSrc);
    h0.bnorm2 = norm2_host(c, args.su);
    const double bnorm = std::sqrt(h0.bnorm2);
    const bool l2 = args.stop_rule == FC_STOP_L2;
    int total_inner = 0, outer = 0, fallback_iters = 0;
    double res0 = 0.0, resl = 0.0, fallback_ms = 0.0;
    bool fell_back = false;
    GraphExec graph;   // the inner iterations, the same in every cycle
    fc_status status = FC_NOT_CONVERGED;
    ctx->timer.start(c.s);
    for (;;) {
        h0.done = 0;
        upload_scalars(c, h0);
        spmv_launch64(c.s, 1, n, st.ioffset.as<int>(), st.ja.as<int>(), args.a, args.fi, args.su, nullptr, r,
                      nullptr, c.pa, c.pb, nullptr);
        fin(c, kFinOuter, spmv_grid(n), true);
        Scalars ho = read_scalars(c);
        if (outer == 0) res0 = ho.resl;
        resl = ho.resl;
        const double rel = bnorm > 0 ? std::sqrt(ho.rnorm2) / bnorm : std::sqrt(ho.rnorm2);
        if (!std::isfinite(rel)) { status = FC_ERR_NONFINITE; break; }
        const bool conv = l2 ? rel < args.sor : (res0 > 0 ? resl / (res0 + kSmallSrc) < args.sor : true);
        if (conv) { status = FC_OK; break; }
        if (outer >= args.max_outer || total_inner >= args.nsw) { status = FC_NOT_CONVERGED; break; }
        FC_HIP_CHECK(hipMemcpyAsync(xgood, args.fi, sizeof(double) * n, hipMemcpyDeviceToDevice, c.s));
        const double rn = std::sqrt(ho.rnorm2);
        k_scale_cast<<<c.gv, 256, 0, c.s>>>(n, r, ws.r32.as<float>(), 1.0 / rn);
        const int cap = std::max(1, args.nsw - total_inner);
        const int ist = inner_fcg32(c, A, P, args.inner_eta, cap, total_inner, graph);
        ++outer;
        if (ist == FC_FALLBACK_USED || ist == FC_ERR_NONFINITE) {
            // plain IC(0)-PCG (FP64) finishes the solve from the last refined iterate;
            // it runs its own timer, so the learned part is timed up to here
            FC_HIP_CHECK(hipMemcpyAsync(args.fi, xgood, sizeof(double) * n, hipMemcpyDeviceToDevice, c.s));
            fallback_ms = ctx->timer.stop_ms(c.s);
            fell_back = true;
            // The fallback gets what is left of the caller's nsw, and keeps the caller's
            // stopping rule: the L2 rule is relative to ||su|| already; the L1 rule is
            // relative to the first refinement's ||r0||_1, so the fallback's tolerance is
            // rescaled from its own start (resl: ||r||_1 at that iterate).
            SolveArgs fb = args;
            fb.nsw = std::max(1, args.nsw - total_inner);
            if (!l2) fb.sor = args.sor * (res0 + kSmallSrc) / (resl + kSmallSrc);
            fc_solve_info fi;
            std::memset(&fi, 0, sizeof fi);
            ensure_levels(ctx, const_cast<Structure &>(st));
            fc_status fs = solve_pcg64(ctx, fb, true, &fi);
            fallback_iters = fi.iters;
            fallback_ms += fi.setup_ms + fi.solve_ms;
            resl = fi.resl;
            status = (fs == FC_OK || fs == FC_EARLY_EXIT) ? FC_FALLBACK_USED : fs;
            break;
        }
        k_refine<<<c.gv, 256, 0, c.s>>>(n, args.fi, ws.e32.as<float>(), rn);
    }
    const double solve_ms = fell_back ? fallback_ms : ctx->timer.stop_ms(c.s);
    if (info) {
        info->res0 = res0;
        info->resl = resl;
        info->rsm = res0 > 0 ? resl / (res0 + kSmallSrc) : 0.0;
        info->iters = total_inner;
        info->outer = outer;
        info->fallback_iters = fallback_iters;
        info->status = status;
        info->setup_ms = setup_ms;
        info->solve_ms = solve_ms;
    }
    return status;
}

// ====================================== allocation-free Jacobi-PCG (fc_dpcg_noalloc)
//
// dpcg (src/dpcg.f90) on caller-owned device arrays for callers that cannot
// allocate device memory.  Every buffer beyond the caller's arrays -- the search
// direction, the preconditioned residual, A p, the residual when the caller
// passes none, the reduction partials and the solver scalars -- is carved from
// one file-scope device array.  The 1-based CSR arrays are read in place: the
// kernels index a, ja and x with 1-based positions and columns through pointers
// shifted back by one entry, while ioffset and diag are indexed by 0-based row
// and hold 1-based positions.  The kernels and sums are those of solve_pcg64,
// so the result is bitwise that of fc_dpcg on the same inputs.

constexpr int kNoAllocCells = 1 << 20;
constexpr size_t kNoAllocVec = sizeof(double) * (size_t)kNoAllocCells;
constexpr int kNoAllocParts = kNoAllocCells / kSpmvRows > kMaxRedGrid ? kNoAllocCells / kSpmvRows : kMaxRedGrid;
constexpr size_t kNoAllocPartBytes = sizeof(double) * (size_t)kNoAllocParts;
constexpr size_t kNoAllocTail = 1024;   // Scalars, then three sums
static_assert(kVecParts * kVecGrid <= kNoAllocParts, "scratch partials");
static_assert(sizeof(Scalars) + 3 * sizeof(double) <= kNoAllocTail, "scratch tail");
constexpr size_t kNoAllocBytes = 4 * kNoAllocVec + 4 * kNoAllocPartBytes + kNoAllocTail;

// Each GPU holds its own copy of this array until the process ends.  Host code
// never uses its name as an address: it uses the per-device pointer that
// hipGetSymbolAddress returns (g_noalloc).
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

constexpr int kNoAllocDevices = 64;
static void *g_noalloc[kNoAllocDevices];
static std::mutex g_noalloc_mu;

size_t noalloc_bytes() { return kNoAllocBytes; }
int noalloc_max_cells() { return kNoAllocCells; }

void noalloc_init(int device) {
    FC_REQUIRE(device >= 0 && device < kNoAllocDevices, FC_ERR_ARGUMENT, "device index beyond 63");
    std::lock_guard<std::mutex> lock(g_noalloc_mu);
    if (g_noalloc[device]) return;
    FC_HIP_CHECK(hipSetDevice(device));
    void *ptr = nullptr;
    FC_HIP_CHECK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    FC_REQUIRE(ptr != nullptr, FC_ERR_HIP, "no device address for the allocation-free scratch");
    g_noalloc[device] = ptr;
}

fc_status solve_dpcg_noalloc(fc_context *ctx, int n, int nnz, const int *ioffset, const int *ja, const int *diag,
                             const double *a, const double *su, double *fi, double *res, double sor, int nsw,
                             fc_solve_info *info) {
    FC_REQUIRE(n >= 1 && n <= kNoAllocCells, FC_ERR_ARGUMENT,
               "fc_dpcg_noalloc: numCells must be 1..1048576 (the size of its scratch)");
    FC_REQUIRE(nnz >= n, FC_ERR_ARGUMENT, "nnz < numCells");
    void *base = ctx->device >= 0 && ctx->device < kNoAllocDevices ? g_noalloc[ctx->device] : nullptr;
    FC_REQUIRE(base != nullptr, FC_ERR_HIP, "allocation-free scratch not set up on this device");
    const hipStream_t s = ctx->stream;
    // the CSR bounds, read with two 4-byte copies into host variables
    int first = 0, last = 0;
    FC_HIP_CHECK(hipMemcpyAsync(&first, ioffset, sizeof(int), hipMemcpyDeviceToHost, s));
    FC_HIP_CHECK(hipMemcpyAsync(&last, ioffset + n, sizeof(int), hipMemcpyDeviceToHost, s));
    FC_HIP_CHECK(hipStreamSynchronize(s));
    FC_REQUIRE(first == 1 && last == nnz + 1, FC_ERR_STRUCTURE, "ioffset is not 1-based with ioffset(n+1) = nnz+1");
    const auto t0 = std::chrono::steady_clock::now();
    unsigned char *b = static_cast<unsigned char *>(base);
    double *r = res ? res : reinterpret_cast<double *>(b);
    double *z = reinterpret_cast<double *>(b + kNoAllocVec);
    double *p = reinterpret_cast<double *>(b + 2 * kNoAllocVec);
    double *q = reinterpret_cast<double *>(b + 3 * kNoAllocVec);
    double *pa = reinterpret_cast<double *>(b + 4 * kNoAllocVec);
    double *pb = reinterpret_cast<double *>(b + 4 * kNoAllocVec + kNoAllocPartBytes);
    double *pv = reinterpret_cast<double *>(b + 4 * kNoAllocVec + 2 * kNoAllocPartBytes);
    double *pq = reinterpret_cast<double *>(b + 4 * kNoAllocVec + 3 * kNoAllocPartBytes);
    Scalars *sc = reinterpret_cast<Scalars *>(b + 4 * kNoAllocVec + 4 * kNoAllocPartBytes);
    double *sums = reinterpret_cast<double *>(b + 4 * kNoAllocVec + 4 * kNoAllocPartBytes + sizeof(Scalars));
    const double *a1 = a - 1;    // a1[k], k a 1-based position
    const int *ja1 = ja - 1;     // ja1[k] a 1-based column
    Ctx c{ctx, s, nullptr, n, sc, pa, pb, pv, nullptr, pq, nullptr, sums, red_grid(n), fused_grid(n), {}};
    SolveArgs args;
    args.sor = sor;
    args.nsw = nsw;
    args.variant = ctx->variant;
    args.stop_rule = FC_STOP_L1;
    const double small = args.variant == FC_VARIANT_TESTS ? kSmallTests : kSmallSrc;
    const Scalars h = init_scalars(args, small);
    upload_scalars(c, h);
    k_zero<double><<<c.gv, 256, 0, s>>>(n, p);
    spmv_launch64(s, 1, n, ioffset, ja1, a1, fi - 1, su, nullptr, r, nullptr, pa, pb, nullptr);
    fin(c, kFinRes0, seq_or(c, spmv_grid(n), 1, r, nullptr), true);
    const int gs = spmv_grid(n);
    if (!read_done(c) && !ctx->reduce_seq) {
        // the fused iterations of solve_pcg64, the diagonal in z
        k_diag<<<c.gv, 256, 0, s>>>(n, a1, diag, z);
        k_first_dot<double><<<c.gf, kRedBlock, 0, s>>>(n, r, r, z, sc, pv);
        k_cg_p<double, true><<<c.gf, kRedBlock, 0, s>>>(n, p, r, z, sc, pv, c.gf, nullptr, 0, 1);
        for (;;) {
            for (int k = 0; k < 8; ++k) {
                spmv_launch64(s, 2, n, ioffset, ja1, a1, p - 1, nullptr, p, q, nullptr, pq, nullptr, sc);
                const SpmvSums v = spmv_sums(c, false);
                k_cg_xr<double, double, true><<<c.gf, kRedBlock, 0, s>>>(n, fi, r, p, q, z, sc, v.a, v.n, pv);
                k_cg_p<double, true><<<c.gf, kRedBlock, 0, s>>>(n, p, r, z, sc, pv, c.gf, nullptr, 0, 0);
            }
            FC_HIP_CHECK(hipGetLastError());
            if (read_done(c)) break;
        }
    } else if (!read_done(c)) {
        for (;;) {
            for (int k = 0; k < 8; ++k) {
                k_jacobi<double, double><<<c.gv, kRedBlock, 0, s>>>(n, r, a1, diag, z, sc, pa);
                fin(c, kFinSk, seq_or(c, c.gv, 0, r, z), false);
                k_p_update<double><<<c.gv, 256, 0, s>>>(n, p, z, sc);
                spmv_launch64(s, 2, n, ioffset, ja1, a1, p - 1, nullptr, p, q, nullptr, pa, nullptr, sc);
                fin(c, kFinAlf, seq_or(c, gs, 0, p, q), false);
                k_pcg_xr64<<<c.gv, kRedBlock, 0, s>>>(n, fi, r, p, q, sc, pa, pb);
                fin(c, kFinPcgEnd, seq_or(c, c.gv, 1, r, nullptr), true);
            }
            FC_HIP_CHECK(hipGetLastError());
            if (read_done(c)) break;
        }
    }
    const Scalars hs = read_scalars(c);
    const double ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    fill_info(info, hs, 0.0, ms);
    if (info) {
        // ||su - A fi||_2 / ||su||_2 from scratch: the true residual into z (q's partials)
        spmv_launch64(s, 1, n, ioffset, ja1, a1, fi - 1, su, nullptr, z, nullptr, pa, pb, nullptr);
        sum_parts_launch(s, gs, pb, nullptr, sums);
        norms_launch64(s, n, su, pa, pb);
        sum_parts_launch(s, red_grid(n), pb, nullptr, sums + 1);
        double hsum[3] = {0.0, 0.0, 0.0};
        FC_HIP_CHECK(hipMemcpyAsync(hsum, sums, sizeof(double) * 3, hipMemcpyDeviceToHost, s));
        FC_HIP_CHECK(hipStreamSynchronize(s));
        info->rel_l2 = hsum[1] > 0.0 ? std::sqrt(hsum[0] / hsum[1]) : std::sqrt(hsum[0]);
    }
    return (fc_status)hs.status;
}

}  // namespace fcap
