// SpMV, reductions, level-scheduled incomplete factorisations and sweeps.
//
// SpMV: one wavefront per block of 64 consecutive rows.  The wave stages the
// block's slice of a/ja (contiguous in CSR) into LDS with coalesced loads,
// then each lane walks its own row from LDS in CSR order, gathering x from
// global memory.  The per-row order of operations is the reference's
// (src/iccg.f90:129-134), so the FP64 result is bit-identical.
//
// Triangular sweeps and pivot recurrences are level-scheduled: the rows of a
// level of the lower (forward) or upper (backward) dependency DAG have no
// mutual dependencies; each level is one launch over its rows, each row
// computed in the reference's order (src/iccg.f90:77-111, src/bicgstab.f90:68-79).

#include <algorithm>

#include "fcap_internal.h"
#include "fcap_kernels.h"
#include "fcap_linalg.h"
#include "fcap_syncfree.h"

namespace fcap {

namespace {

inline int grid_for(long long n, int block) {
    long long g = (n + block - 1) / block;
    return (int)std::max<long long>(1, std::min<long long>(g, 1 << 30));
}

}  // namespace

int red_grid(int n) { return std::min(kMaxRedGrid, grid_for(n, kRedBlock)); }
int spmv_grid(int n) { return grid_for(n, kSpmvRows); }
// launch grid of a kernel with an XCD-aware block order: `blocks` rounded up to a multiple of kXcds
static int xcd_grid(int blocks) { return (blocks + kXcds - 1) / kXcds * kXcds; }

// SpMV block order: workgroup b takes row block b.  (An XCD-aware order, each
// XCD sweeping one contiguous eighth of the rows, measured slower at 192^3:
// 4.86 against 5.10 TB/s.)
constexpr int g_spmv_xcd = 0;

// ------------------------------------------------------------------- SpMV

template <class T, class AT, int MODE>
__global__ __launch_bounds__(kSpmvRows) void k_spmv(int n, const int *__restrict__ ptr, const int *__restrict__ ja,
                                                    const AT *__restrict__ a, const T *__restrict__ x,
                                                    const T *__restrict__ b, const T *__restrict__ v,
                                                    T *__restrict__ y, float *__restrict__ y32,
                                                    double *__restrict__ partA, double *__restrict__ partB,
                                                    const Scalars *__restrict__ sc, int xcd, float omega) {
    // MODE 0: y = A x; 1: y = b - A x with |y| and y^2 partials; 2: y = A x with y.v
    // partials; 3: y = A x with y.v and y^2 partials; 4: y = x + omega (b - A x) / v;
    // 5: y = b - A x
    constexpr bool kRes = MODE == 1 || MODE == 4 || MODE == 5;
    __shared__ AT sa[kSpmvWaves][kSpmvCap];
    __shared__ int sj[kSpmvWaves][kSpmvCap];
    __shared__ double red[kSpmvWaves];
    if (sc && sc->done) return;
    // xcd = 1, XCD-aware order: workgroups go to the 8 XCDs round-robin, so
    // workgroup b takes row block (b % 8) * per + b / 8 and each XCD sweeps one
    // contiguous eighth of the rows (the grid is then a multiple of 8).
    const int nblk = (int)(((long long)n + kSpmvRows - 1) / kSpmvRows);
    const int per = gridDim.x / kXcds;
    const int blk = xcd ? (int)(blockIdx.x % kXcds) * per + (int)(blockIdx.x / kXcds) : (int)blockIdx.x;
    if (blk >= nblk) return;
    const int w = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const long long row0 = (long long)blk * kSpmvRows + (long long)w * kWave;
    const long long rowl = row0 + lane;
    const bool valid = rowl < n;
    const int row = (int)rowl;
    int nrows = (int)std::min<long long>(std::max<long long>(n - row0, 0), kWave);
    int s0 = 0, cnt = 0;
    if (nrows > 0) {
        s0 = ptr[row0];
        cnt = ptr[row0 + nrows] - s0;
    }
    const bool staged = nrows > 0 && cnt <= kSpmvCap;
    if (staged) {
        // all loads of the slice are issued before the first LDS store, so a
        // wave keeps up to 2*kSpmvCap/64 loads in flight; a and ja are read
        // once, so they are streamed (non-temporal) and leave the caches to x
        constexpr int kChunks = kSpmvCap / kWave;
        AT va[kChunks];
        int vj[kChunks];
#pragma unroll
        for (int c = 0; c < kChunks; ++c) {
            const int j = c * kWave + lane;
            if (j < cnt) {
                va[c] = __builtin_nontemporal_load(a + s0 + j);
                vj[c] = __builtin_nontemporal_load(ja + s0 + j);
            }
        }
#pragma unroll
        for (int c = 0; c < kChunks; ++c) {
            const int j = c * kWave + lane;
            if (j < cnt) {
                sa[w][j] = va[c];
                sj[w][j] = vj[c];
            }
        }
    }
    __syncthreads();
    double pa = 0.0, pb = 0.0;
    if (valid) {
        const int rs = ptr[row], re = ptr[row + 1];
        T acc = kRes ? b[row] : T(0);
        if (staged) {
            // gathers issued four at a time; the sum still runs in CSR order
            int k = rs - s0;
            const int ke = re - s0;
            for (; k + 4 <= ke; k += 4) {
                const T x0 = x[sj[w][k]], x1 = x[sj[w][k + 1]], x2 = x[sj[w][k + 2]], x3 = x[sj[w][k + 3]];
                const T p0 = (T)sa[w][k] * x0, p1 = (T)sa[w][k + 1] * x1;
                const T p2 = (T)sa[w][k + 2] * x2, p3 = (T)sa[w][k + 3] * x3;
                if (kRes) { acc = acc - p0; acc = acc - p1; acc = acc - p2; acc = acc - p3; }
                else { acc = acc + p0; acc = acc + p1; acc = acc + p2; acc = acc + p3; }
            }
            for (; k < ke; ++k) {
                T prod = (T)sa[w][k] * x[sj[w][k]];
                acc = kRes ? acc - prod : acc + prod;
            }
        } else {
            for (int k = rs; k < re; ++k) {
                T prod = (T)a[k] * x[ja[k]];
                acc = kRes ? acc - prod : acc + prod;
            }
        }
        if (MODE == 4)
            y[row] = x[row] + (T)omega * (acc / v[row]);
        else
            y[row] = acc;
        if (MODE == 1) {
            if (y32) y32[row] = (float)acc;
            pa = fabs((double)acc);
            pb = (double)acc * (double)acc;
        } else if (MODE == 2) {
            pa = (double)acc * (double)v[row];
        } else if (MODE == 3) {
            pa = (double)acc * (double)v[row];
            pb = (double)acc * (double)acc;
        }
    }
    if (MODE != 0 && MODE != 4 && MODE != 5) {
        pa = wave_sum(pa);
        if (lane == 0) red[w] = pa;
        __syncthreads();
        if (threadIdx.x == 0) {
            double s = 0.0;
            for (int i = 0; i < kSpmvWaves; ++i) s += red[i];
            partA[blk] = s;
        }
        if (MODE == 1 || MODE == 3) {
            __syncthreads();
            pb = wave_sum(pb);
            if (lane == 0) red[w] = pb;
            __syncthreads();
            if (threadIdx.x == 0) {
                double s = 0.0;
                for (int i = 0; i < kSpmvWaves; ++i) s += red[i];
                partB[blk] = s;
            }
        }
    }
}

// O-C couplings in cut order, per cell (src/iccg.f90:59-62,137-140):
// sign -1 for the residual form, +1 for the product form.
template <class T>
__global__ void k_oc_apply(int n, const int *__restrict__ co_ptr, const int *__restrict__ co_idx,
                           const int *__restrict__ ijl, const int *__restrict__ ijr, const double *__restrict__ al,
                           const double *__restrict__ ar, const T *__restrict__ x, T *__restrict__ y, int sign,
                           const Scalars *__restrict__ sc) {
    if (sc && sc->done) return;
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int s = co_ptr[i], e = co_ptr[i + 1];
    if (s == e) return;
    T acc = y[i];
    for (int q = s; q < e; ++q) {
        int code = co_idx[q], o = code >> 1;
        T prod = (code & 1) ? (T)al[o] * x[ijl[o]] : (T)ar[o] * x[ijr[o]];
        acc = sign < 0 ? acc - prod : acc + prod;
    }
    y[i] = acc;
}

void spmv_launch64(hipStream_t s, int mode, int n, const int *ptr, const int *ja, const double *a, const double *x,
                   const double *b, const double *v, double *y, float *y32, double *pa, double *pb,
                   const Scalars *sc) {
    const int xo = g_spmv_xcd;
    const int g = xo ? xcd_grid(spmv_grid(n)) : spmv_grid(n);
    switch (mode) {
    case 0: k_spmv<double, double, 0><<<g, kSpmvRows, 0, s>>>(n, ptr, ja, a, x, b, v, y, y32, pa, pb, sc, xo, 0.f); break;
    case 1: k_spmv<double, double, 1><<<g, kSpmvRows, 0, s>>>(n, ptr, ja, a, x, b, v, y, y32, pa, pb, sc, xo, 0.f); break;
    case 2: k_spmv<double, double, 2><<<g, kSpmvRows, 0, s>>>(n, ptr, ja, a, x, b, v, y, y32, pa, pb, sc, xo, 0.f); break;
    default: k_spmv<double, double, 3><<<g, kSpmvRows, 0, s>>>(n, ptr, ja, a, x, b, v, y, y32, pa, pb, sc, xo, 0.f); break;
    }
}

void spmv_launch32(hipStream_t s, int mode, int n, const int *ptr, const int *ja, const float *a, const float *x,
                   const float *b, const float *v, float *y, double *pa, double *pb, const Scalars *sc) {
    const int xo = g_spmv_xcd;
    const int g = xo ? xcd_grid(spmv_grid(n)) : spmv_grid(n);
    switch (mode) {
    case 0: k_spmv<float, float, 0><<<g, kSpmvRows, 0, s>>>(n, ptr, ja, a, x, b, v, y, nullptr, pa, pb, sc, xo, 0.f); break;
    case 1: k_spmv<float, float, 1><<<g, kSpmvRows, 0, s>>>(n, ptr, ja, a, x, b, v, y, nullptr, pa, pb, sc, xo, 0.f); break;
    case 2: k_spmv<float, float, 2><<<g, kSpmvRows, 0, s>>>(n, ptr, ja, a, x, b, v, y, nullptr, pa, pb, sc, xo, 0.f); break;
    default: k_spmv<float, float, 3><<<g, kSpmvRows, 0, s>>>(n, ptr, ja, a, x, b, v, y, nullptr, pa, pb, sc, xo, 0.f); break;
    }
}

void jacobi_step32(hipStream_t s, int n, const int *ptr, const int *ja, const float *a, const float *x, const float *b,
                   const float *d, float omega, float *y, const Scalars *sc) {
    const int xo = g_spmv_xcd;
    const int g = xo ? xcd_grid(spmv_grid(n)) : spmv_grid(n);
    k_spmv<float, float, 4><<<g, kSpmvRows, 0, s>>>(n, ptr, ja, a, x, b, d, y, nullptr, nullptr, nullptr, sc, xo,
                                                    omega);
}

void residual32(hipStream_t s, int n, const int *ptr, const int *ja, const float *a, const float *x, const float *b,
                float *y, const Scalars *sc) {
    const int xo = g_spmv_xcd;
    const int g = xo ? xcd_grid(spmv_grid(n)) : spmv_grid(n);
    k_spmv<float, float, 5><<<g, kSpmvRows, 0, s>>>(n, ptr, ja, a, x, b, nullptr, y, nullptr, nullptr, nullptr, sc,
                                                    xo, 0.f);
}

void oc_launch64(hipStream_t s, int n, const OcView &oc, const double *x, double *y, int sign, const Scalars *sc) {
    if (!oc.noc) return;
    k_oc_apply<double><<<grid_for(n, 256), 256, 0, s>>>(n, oc.co_ptr, oc.co_idx, oc.ijl, oc.ijr, oc.al, oc.ar, x, y,
                                                        sign, sc);
}

// ------------------------------------------------------- pivots and sweeps

__global__ void k_dic_level(const int *__restrict__ rows, int beg, int cnt, const int *__restrict__ ptr,
                            const int *__restrict__ ja, const int *__restrict__ diag, const double *__restrict__ a,
                            double *__restrict__ d, int *__restrict__ err) {
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= cnt) return;
    int i = rows[beg + t];
    double di = a[diag[i]];
    for (int k = ptr[i]; k < diag[i]; ++k) {
        double ak = a[k];
        di = di - (ak * ak) * d[ja[k]];
    }
    if (!(di != 0.0) || !isfinite(di)) atomicOr(err, 1);
    d[i] = 1.0 / di;
}

__global__ void k_dilu_level(const int *__restrict__ rows, int beg, int cnt, const int *__restrict__ ptr,
                             const int *__restrict__ ja, const int *__restrict__ diag, const int *__restrict__ tpos,
                             const double *__restrict__ a, double *__restrict__ d, int *__restrict__ err) {
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= cnt) return;
    int i = rows[beg + t];
    double di = a[diag[i]];
    for (int k = ptr[i]; k < diag[i]; ++k) di = di - (a[k] * d[ja[k]]) * a[tpos[k]];
    if (!(di != 0.0) || !isfinite(di)) atomicOr(err, 1);
    d[i] = 1.0 / di;
}

// forward sweep of (D+L) w = rhs: w_i = (rhs_i - sum_{k<diag} a_k w_j) d_i
template <class T>
__global__ void k_fwd_level(const int *__restrict__ rows, int beg, int cnt, const int *__restrict__ ptr,
                            const int *__restrict__ ja, const int *__restrict__ diag, const T *__restrict__ a,
                            const T *__restrict__ d, const T *__restrict__ rhs, T *__restrict__ w,
                            const Scalars *__restrict__ sc) {
    if (sc && sc->done) return;
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= cnt) return;
    int i = rows[beg + t];
    T acc = rhs[i];
    for (int k = ptr[i]; k < diag[i]; ++k) acc = acc - a[k] * w[ja[k]];
    w[i] = acc * d[i];
}

// backward sweep in place: z_i = (w_i/(d_i+small) - sum_{k>diag} a_k z_j) d_i
template <class T>
__global__ void k_bwd_level(const int *__restrict__ rows, int beg, int cnt, const int *__restrict__ ptr,
                            const int *__restrict__ ja, const int *__restrict__ diag, const T *__restrict__ a,
                            const T *__restrict__ d, T small, T *__restrict__ w, const Scalars *__restrict__ sc) {
    if (sc && sc->done) return;
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= cnt) return;
    int i = rows[beg + t];
    T di = d[i];
    T acc = w[i] / (di + small);
    for (int k = diag[i] + 1; k < ptr[i + 1]; ++k) acc = acc - a[k] * w[ja[k]];
    w[i] = acc * di;
}

template <int W>
void pivots_syncfree_w(hipStream_t s, const Structure &st, const double *a, double *d, bool dilu, int *err,
                       const SweepCfg &cfg);

void pivots_launch(hipStream_t s, const Structure &st, const double *a, double *d, bool dilu, int *err,
                   const SweepCfg *cfg) {
    if (cfg && cfg->sf && syncfree_sweeps(st)) {
        FC_REQUIRE(!dilu || st.tpos.get(), FC_ERR_ARGUMENT, "DILU pivots need the transpose positions");
        switch (st.ell_f) {
        case 3: pivots_syncfree_w<3>(s, st, a, d, dilu, err, *cfg); break;
        case 4: pivots_syncfree_w<4>(s, st, a, d, dilu, err, *cfg); break;
        default: pivots_syncfree_w<8>(s, st, a, d, dilu, err, *cfg); break;
        }
        FC_HIP_CHECK(hipGetLastError());
        return;
    }
    const int *rows = st.rows_f.as<int>();
    for (int l = 0; l < st.nlev_f; ++l) {
        int beg = st.lvl_f[l], cnt = st.lvl_f[l + 1] - beg;
        if (dilu)
            k_dilu_level<<<grid_for(cnt, 256), 256, 0, s>>>(rows, beg, cnt, st.ioffset.as<int>(), st.ja.as<int>(),
                                                             st.diag.as<int>(), st.tpos.as<int>(), a, d, err);
        else
            k_dic_level<<<grid_for(cnt, 256), 256, 0, s>>>(rows, beg, cnt, st.ioffset.as<int>(), st.ja.as<int>(),
                                                            st.diag.as<int>(), a, d, err);
    }
    FC_HIP_CHECK(hipGetLastError());
}

// ------------------------------------------------- level-packed sweeps

// packed row p of a level: operands at [k * n + p] (coalesced across the
// level's threads); all of a row's slots are loaded, then all gathers of w
// issued, then the sum runs in CSR order over the row's own entries only, so
// the arithmetic is that of k_fwd_level / k_bwd_level.  Padding slots hold
// column 0 and value 0 and are never added.
template <class T, int W>
__global__ void k_fwd_packed(int beg, int cnt, int n, const int *__restrict__ rows, const int *__restrict__ cntp,
                             const int *__restrict__ col, const T *__restrict__ av, const T *__restrict__ dv,
                             const T *__restrict__ rhs, T *__restrict__ w, int ell, const Scalars *__restrict__ sc) {
    if (sc && sc->done) return;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= cnt) return;
    const int p = beg + t;
    const int i = rows[p];
    const int c = cntp[p];
    T acc = rhs[i];
    if (W > 0) {
        int cj[W > 0 ? W : 1];
        T ak[W > 0 ? W : 1], wk[W > 0 ? W : 1];
#pragma unroll
        for (int k = 0; k < W; ++k) {
            cj[k] = col[(size_t)k * n + p];
            ak[k] = av[(size_t)k * n + p];
        }
#pragma unroll
        for (int k = 0; k < W; ++k) wk[k] = w[cj[k]];
#pragma unroll
        for (int k = 0; k < W; ++k)
            if (k < c) acc = acc - ak[k] * wk[k];
    } else {
        for (int k = 0; k < c; ++k) acc = acc - av[(size_t)k * n + p] * w[col[(size_t)k * n + p]];
    }
    (void)ell;
    w[i] = acc * dv[p];
}

template <class T, int W>
__global__ void k_bwd_packed(int beg, int cnt, int n, const int *__restrict__ rows, const int *__restrict__ cntp,
                             const int *__restrict__ col, const T *__restrict__ av, const T *__restrict__ dv, T small,
                             T *__restrict__ w, const Scalars *__restrict__ sc) {
    if (sc && sc->done) return;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= cnt) return;
    const int p = beg + t;
    const int i = rows[p];
    const int c = cntp[p];
    const T di = dv[p];
    if (W > 0) {
        int cj[W > 0 ? W : 1];
        T ak[W > 0 ? W : 1], wk[W > 0 ? W : 1];
#pragma unroll
        for (int k = 0; k < W; ++k) {
            cj[k] = col[(size_t)k * n + p];
            ak[k] = av[(size_t)k * n + p];
        }
#pragma unroll
        for (int k = 0; k < W; ++k) wk[k] = w[cj[k]];
        T acc = w[i] / (di + small);
#pragma unroll
        for (int k = 0; k < W; ++k)
            if (k < c) acc = acc - ak[k] * wk[k];
        w[i] = acc * di;
    } else {
        T acc = w[i] / (di + small);
        for (int k = 0; k < c; ++k) acc = acc - av[(size_t)k * n + p] * w[col[(size_t)k * n + p]];
        w[i] = acc * di;
    }
}

// values of the factor into packed order (one pass per solve)
template <class T>
__global__ void k_pack_factor(int n, int ell, const int *__restrict__ rows, const int *__restrict__ cntp,
                              const int *__restrict__ kpos, const T *__restrict__ a, const T *__restrict__ d,
                              T *__restrict__ av, T *__restrict__ dv) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const int c = cntp[p];
    for (int k = 0; k < ell; ++k) {
        const size_t o = (size_t)k * n + p;
        av[o] = k < c ? a[kpos[o]] : T(0);
    }
    dv[p] = d[rows[p]];
}

// Each triangle's ELL is stored at exactly the width its kernel reads (3, 4 or
// 8 slots per row, or its widest row for the generic W = 0 kernel).
template <class T, int W>
void fwd_packed_w(hipStream_t s, const Structure &st, const PackedFactor<T> &pf, const T *rhs, T *w,
                  const Scalars *sc) {
    const int *rf = st.rows_f.as<int>();
    for (int l = 0; l < st.nlev_f; ++l) {
        const int beg = st.lvl_f[l], cnt = st.lvl_f[l + 1] - beg;
        k_fwd_packed<T, W><<<grid_for(cnt, 256), 256, 0, s>>>(beg, cnt, st.n, rf, st.cnt_f.as<int>(),
                                                              st.col_f.as<int>(), pf.af, pf.df, rhs, w, st.ell_f, sc);
    }
}

template <class T, int W>
void bwd_packed_w(hipStream_t s, const Structure &st, const PackedFactor<T> &pf, T small, T *w, const Scalars *sc) {
    const int *rb = st.rows_b.as<int>();
    for (int l = 0; l < st.nlev_b; ++l) {
        const int beg = st.lvl_b[l], cnt = st.lvl_b[l + 1] - beg;
        k_bwd_packed<T, W><<<grid_for(cnt, 256), 256, 0, s>>>(beg, cnt, st.n, rb, st.cnt_b.as<int>(),
                                                              st.col_b.as<int>(), pf.ab, pf.db, small, w, sc);
    }
}

template <class T>
void sweeps_packed(hipStream_t s, const Structure &st, const PackedFactor<T> &pf, T small, const T *rhs, T *w,
                   const Scalars *sc) {
    switch (st.ell_f) {
    case 3: fwd_packed_w<T, 3>(s, st, pf, rhs, w, sc); break;
    case 4: fwd_packed_w<T, 4>(s, st, pf, rhs, w, sc); break;
    case 8: fwd_packed_w<T, 8>(s, st, pf, rhs, w, sc); break;
    default: fwd_packed_w<T, 0>(s, st, pf, rhs, w, sc); break;
    }
    switch (st.ell_b) {
    case 3: bwd_packed_w<T, 3>(s, st, pf, small, w, sc); break;
    case 4: bwd_packed_w<T, 4>(s, st, pf, small, w, sc); break;
    case 8: bwd_packed_w<T, 8>(s, st, pf, small, w, sc); break;
    default: bwd_packed_w<T, 0>(s, st, pf, small, w, sc); break;
    }
}

template <class T>
void pack_factor_t(hipStream_t s, const Structure &st, const T *a, const T *d, T *af, T *df, T *ab, T *db) {
    FC_REQUIRE(packed_sweeps(st), FC_ERR_ARGUMENT, "structure has no level-packed sweeps");
    const int n = st.n;
    k_pack_factor<T><<<grid_for(n, 256), 256, 0, s>>>(n, st.ell_f, st.rows_f.as<int>(), st.cnt_f.as<int>(),
                                                      st.kpos_f.as<int>(), a, d, af, df);
    k_pack_factor<T><<<grid_for(n, 256), 256, 0, s>>>(n, st.ell_b, st.rows_b.as<int>(), st.cnt_b.as<int>(),
                                                      st.kpos_b.as<int>(), a, d, ab, db);
    FC_HIP_CHECK(hipGetLastError());
}

// ------------------------------------------- dependency-driven sweeps
// One launch per sweep.  Persistent one-wave workgroups take blocks of 64
// consecutive packed rows (level order) from kSfTickets ticket counters: counter c
// hands out blocks c, c + kSfTickets, ... in turn, workgroup g takes from counter
// g % kSfTickets.  (One counter for all cost 10 ns a ticket one after the other: with
// marks in launches of their own 34 us a sweep on the 24^3 tets, now 25, on the 40^3
// tets 90 and 39.)  A sweep clears the other direction's counters.
//
// The waits end whichever workgroups run: the smallest unfinished block has only
// finished inputs, so the wave that holds it goes on; and if none has taken it, because
// its counter's workgroups have not started, every wave that waits comes to take it --
// one whose inputs are late sets its block aside and takes the smallest block before it
// that is left, from whichever counter.  A block set aside is begun anew later; the
// blocks a wave holds are of different counters (a counter's later blocks are larger),
// so there are at most kSfTickets of them.  Fewer workgroups than counters take from all
// of them from the start.
//
// The output starts filled with a
// signalling-NaN pattern that arithmetic never produces; a row polls the
// outputs of the rows it reads until none holds the pattern, computes exactly
// as k_fwd_packed / k_bwd_packed (same operands, same order), and stores its
// value with one coherent store, which is also its "ready" signal.  A wave
// whose wait exceeds the time limit, or that sees the abort flag, raises the
// flag and leaves; the host then reports the solve as failed.

// Waves in flight poll the coherent level of the memory system; the fewer there
// are, the faster the chain of levels advances, as long as they hold a level
// (syncfree_wave_count: twice an average level, at least one a CU).  Per sweep: Kuhn
// tets 24^3, 14 levels of 5,925 rows, 256 waves 25 us, 512 26, 1,024 28; 40^3, 14 of
// 27,429, 256 62, 428 46, 768 39, 1,024 38, 2,048 44; 96^3 box, 286 of 3,094, 256 468,
// 512 527, 1,024 627.

template <class T>
__global__ void k_sf_mark(int n, T *__restrict__ w, const Scalars *__restrict__ sc) {
    if (sc && sc->done) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) sf_mark(w + i);
}

// Takes the smallest block below `limit` that is left, from any counter; `limit`: there is none.
__device__ inline unsigned sf_take_before(unsigned (*tickets)[32], unsigned limit) {
    const unsigned lane = threadIdx.x, c = lane & (kSfTickets - 1);
    for (;;) {
        unsigned t = __hip_atomic_load(&tickets[c][0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned mine = t * kSfTickets + c;
        unsigned least = mine;
#pragma unroll
        for (int off = kSfTickets / 2; off > 0; off >>= 1) least = min(least, (unsigned)__shfl_xor(least, off));
        if (least >= limit) return limit;
        bool got = false;
        if (lane < kSfTickets && mine == least)
            got = __hip_atomic_compare_exchange_strong(&tickets[c][0], &t, t + 1u, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_AGENT);
        if (__any(got)) return least;   // else another wave has moved that counter on
    }
}

// The other sweep's output takes its marks here: the forward sweep marks w, whose values
// are spent, the backward one its right-hand side once read (a pass of its own for each
// took 4.4 us on 83 K rows, beside sweeps of 26 us) and puts it back for a block set aside;
// mark_sweep_input does it before the first sweep.
// BWD == false: out[i] = (rhs[i] - sum a w) d over the strict lower triangle;
// BWD == true:  out[i] = (fwd[i] / (d + small) - sum a w) d over the strict upper one.
template <class T, int W, bool BWD>
__global__ __launch_bounds__(64) void k_sweep_syncfree(int n, const int *__restrict__ rows,
                                                        const int *__restrict__ cntp, const int *__restrict__ col,
                                                        const T *__restrict__ av, const T *__restrict__ dv,
                                                        const T *in, T small, T *out, T *mk, SyncFree *sf,
                                                        const Scalars *__restrict__ sc) {
    if (sc && sc->done) return;
    using U = typename SfBits<T>::U;
    const int lane = threadIdx.x;
    const unsigned nblk = (unsigned)((n + 63) / 64);
    const unsigned long long limit = sf_wait_ticks(sf, sf->rate_khz);
    const unsigned mine = blockIdx.x % kSfTickets;
    const bool few = gridDim.x < kSfTickets;
    // after how many polls (less one) a wave looks for a block to compute first: a level takes
    // one or two
    const int patience = few ? 0 : 63;
    unsigned aside = 0;   // the blocks set aside: the k-th in lane k
    int naside = 0;
    if (blockIdx.x == 0 && lane < kSfTickets)
        __hip_atomic_store(&sf->tickets[!BWD][lane][0], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (;;) {
        unsigned b = 0;
        if (naside > 0) {
            b = __shfl(aside, --naside);
        } else if (few) {
            b = sf_take_before(sf->tickets[BWD], nblk);
        } else {
            if (lane == 0)
                b = __hip_atomic_fetch_add(&sf->tickets[BWD][mine][0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            b = __shfl(b, 0) * kSfTickets + mine;
        }
        if (b >= nblk) break;
        const int p = (int)b * 64 + lane;
        bool done = p >= n;
        int i = 0, c = 0;
        int cj[W];
        T ak[W], wk[W];
        T rhs = T(0), acc = T(0), di = T(0);
        unsigned ready = 0;
        if (!done) {
            i = rows[p];
            c = cntp[p];
            di = dv[p];
#pragma unroll
            for (int k = 0; k < W; ++k) {
                cj[k] = col[(size_t)k * n + p];
                ak[k] = av[(size_t)k * n + p];
                wk[k] = T(0);
            }
            rhs = in[i];
            acc = BWD ? rhs / (di + small) : rhs;
            sf_mark(mk + i);   // behind the load of in[i] (mk may be in)
        }
        int spins = 0;
        const unsigned long long t0 = wall_clock64();
        unsigned before = b;   // a block taken to be computed first
        for (;;) {
            if (!done) {
                bool all = true;
#pragma unroll
                for (int k = 0; k < W; ++k) {
                    if (k < c && !((ready >> k) & 1u)) {
                        const U bits = sf_load_bits(out + cj[k]);
                        if (bits != SfBits<T>::kMark) {
                            T v;
                            __builtin_memcpy(&v, &bits, sizeof(U));
                            wk[k] = v;
                            ready |= 1u << k;
                        } else {
                            all = false;
                        }
                    }
                }
                if (all) {
                    T r = acc;
#pragma unroll
                    for (int k = 0; k < W; ++k)
                        if (k < c) r = r - ak[k] * wk[k];
                    sf_store(out + i, r * di);
                    done = true;
                }
            }
            if (__all(done)) break;
            ++spins;
            bool give_up = false;
            if ((spins & 63) == 0) {
                give_up = wall_clock64() - t0 > limit ||
                          __hip_atomic_load(&sf->abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
            }
            if (__any(give_up)) {
                if (lane == 0) __hip_atomic_store(&sf->abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
            if ((spins & patience) == 0 && (before = sf_take_before(sf->tickets[BWD], b)) < b) break;
            __builtin_amdgcn_s_sleep(1);
        }
        if (before < b) {
            if (p < n) mk[i] = rhs;   // read again where mk is in
            if (lane == naside) aside = b;
            if (lane == naside + 1) aside = before;
            naside += 2;
        }
    }
}

// The pivot recurrences of k_dic_level / k_dilu_level with the same schedule:
// d_i = 1 / (a_ii - sum over the strict lower row, in CSR order, of a_k^2 d_j
// (DIC) or (a_k d_j) a_kT (DILU)); W bounds the strict lower row (the packed
// width of the forward triangle).
template <int W, bool DILU>
__global__ __launch_bounds__(64) void k_pivots_syncfree(int n, const int *__restrict__ rows, const int *__restrict__ ptr,
                                                        const int *__restrict__ ja, const int *__restrict__ diag,
                                                        const int *__restrict__ tpos, const double *__restrict__ a,
                                                        double *d, int *__restrict__ err, SyncFree *sf) {
    using U = SfBits<double>::U;
    const int lane = threadIdx.x;
    const unsigned nblk = (unsigned)((n + 63) / 64);
    const unsigned long long limit = sf_wait_ticks(sf, sf->rate_khz);
    for (;;) {
        unsigned b = 0;
        if (lane == 0) b = __hip_atomic_fetch_add(&sf->ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        b = __shfl(b, 0);
        if (b >= nblk) break;
        const int p = (int)b * 64 + lane;
        bool done = p >= n;
        int i = 0, c = 0;
        int cj[W];
        double a1[W], a2[W], dk[W];
        double di = 0.0;
        unsigned ready = 0;
        if (!done) {
            i = rows[p];
            const int k0 = ptr[i], kd = diag[i];
            c = kd - k0;
            di = a[kd];
#pragma unroll
            for (int k = 0; k < W; ++k) {
                const bool in = k < c;
                cj[k] = in ? ja[k0 + k] : 0;
                a1[k] = in ? a[k0 + k] : 0.0;
                a2[k] = in && DILU ? a[tpos[k0 + k]] : 0.0;
                dk[k] = 0.0;
            }
            if (c > W) {   // not a structure these sweeps were set up for: report, never wait
                atomicOr(err, 2);
                sf_store(d + i, __builtin_nan(""));
                done = true;
            }
        }
        int spins = 0;
        const unsigned long long t0 = wall_clock64();
        for (;;) {
            if (!done) {
                bool all = true;
#pragma unroll
                for (int k = 0; k < W; ++k) {
                    if (k < c && !((ready >> k) & 1u)) {
                        const U bits = sf_load_bits(d + cj[k]);
                        if (bits != SfBits<double>::kMark) {
                            __builtin_memcpy(&dk[k], &bits, sizeof(U));
                            ready |= 1u << k;
                        } else {
                            all = false;
                        }
                    }
                }
                if (all) {
                    double v = di;
#pragma unroll
                    for (int k = 0; k < W; ++k) {
                        if (k < c) v = DILU ? v - (a1[k] * dk[k]) * a2[k] : v - (a1[k] * a1[k]) * dk[k];
                    }
                    if (!(v != 0.0) || !isfinite(v)) atomicOr(err, 1);
                    sf_store(d + i, 1.0 / v);
                    done = true;
                }
            }
            if (__all(done)) break;
            ++spins;
            bool give_up = false;
            if ((spins & 63) == 0) {
                give_up = wall_clock64() - t0 > limit ||
                          __hip_atomic_load(&sf->abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
            }
            if (__any(give_up)) {
                if (lane == 0) __hip_atomic_store(&sf->abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
    }
    if (lane == 0) {
        const unsigned f = __hip_atomic_fetch_add(&sf->fin, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        if (f == gridDim.x - 1) {
            __hip_atomic_store(&sf->ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&sf->fin, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

template <int W>
void pivots_syncfree_w(hipStream_t s, const Structure &st, const double *a, double *d, bool dilu, int *err,
                       const SweepCfg &cfg) {
    const int n = st.n;
    const int waves = std::max(1, std::min(cfg.waves, (n + 63) / 64));
    k_sf_mark<double><<<grid_for(n, 256), 256, 0, s>>>(n, d, nullptr);
    if (dilu)
        k_pivots_syncfree<W, true><<<waves, 64, 0, s>>>(n, st.rows_f.as<int>(), st.ioffset.as<int>(),
                                                         st.ja.as<int>(), st.diag.as<int>(), st.tpos.as<int>(), a, d,
                                                         err, cfg.sf);
    else
        k_pivots_syncfree<W, false><<<waves, 64, 0, s>>>(n, st.rows_f.as<int>(), st.ioffset.as<int>(),
                                                          st.ja.as<int>(), st.diag.as<int>(), nullptr, a, d, err,
                                                          cfg.sf);
}

void syncfree_reset(fc_context *ctx, hipStream_t s, SyncFree *sf) {
    SyncFree h{};
    h.wait_us = ctx->sf_wait_us;
    h.rate_khz = (unsigned)ctx->wall_clock_khz;
    FC_HIP_CHECK(hipMemcpyAsync(sf, &h, sizeof(SyncFree), hipMemcpyHostToDevice, s));
    FC_HIP_CHECK(hipStreamSynchronize(s));   // h lives on this stack frame
}

bool syncfree_sweeps(const Structure &st) {
    auto ok = [](int w) { return w == 3 || w == 4 || w == 8; };
    return packed_sweeps(st) && ok(st.ell_f) && ok(st.ell_b);
}

// Why half: us a sweep part-wise and row-wise, by the share of entries read from the part's
// own LDS.  Box in reverse Cuthill-McKee order 24^3 (0.93) 48 and 82, 32^3 (0.87) 96 and
// 112, 40^3 (0.40) 168 and 142, 48^3 (0.22) 255 and 172, 56^3 (0.14) 350 and 202; Kuhn tets
// in that order 16^3 (0.92) 66 and 126, 28^3 (0.73) 133 and 229, 40^3 (0.47) 255 and 327, in
// natural order 16^3 (0.94) 64 and 77, 28^3 (0.70) 170 and 143, 40^3 (0.63) 327 and 199;
// boxes shuffled within runs of 300 to 500 cells (0.81, 0.57; five entries a triangle) 147
// and 485, 313 and 513; Morton order (0.96) 45 to 136 and 131 to 406.  No share parts them
// all: the part-wise time is that of the longest chain through parts, not of the share.
// A ring of 4,096 slots would count 0.79, 0.69 and 0.58 of the Cuthill-McKee boxes' entries
// as inside, and take them to the slower schedule: the times are the same to 1 % with rings
// of 1,024, 2,048 and 4,096 (129 and 147 us on one of the shuffled boxes).
bool part_sweeps(const Structure &st) {
    return syncfree_sweeps(st) && st.parts && st.int_frac_f >= 0.5 && st.int_frac_b >= 0.5;
}

template <class T, int WF, int WB>
void lu_syncfree_w(hipStream_t s, const Structure &st, const PackedFactor<T> &pf, T small, const T *rhs, T *w,
                   const Scalars *sc, const SweepCfg &cfg) {
    const int n = st.n;
    T *tmp = static_cast<T *>(cfg.tmp);
    const int waves = std::max(1, std::min(cfg.waves, (n + 63) / 64));
    k_sweep_syncfree<T, WF, false><<<waves, 64, 0, s>>>(n, st.rows_f.as<int>(), st.cnt_f.as<int>(),
                                                          st.col_f.as<int>(), pf.af, pf.df, rhs, small, tmp, w,
                                                          cfg.sf, sc);
    k_sweep_syncfree<T, WB, true><<<waves, 64, 0, s>>>(n, st.rows_b.as<int>(), st.cnt_b.as<int>(),
                                                         st.col_b.as<int>(), pf.ab, pf.db, tmp, small, w, tmp, cfg.sf,
                                                         sc);
}

template <class T, int WF>
void lu_syncfree_b(hipStream_t s, const Structure &st, const PackedFactor<T> &pf, T small, const T *rhs, T *w,
                   const Scalars *sc, const SweepCfg &cfg) {
    switch (st.ell_b) {
    case 3: lu_syncfree_w<T, WF, 3>(s, st, pf, small, rhs, w, sc, cfg); break;
    case 4: lu_syncfree_w<T, WF, 4>(s, st, pf, small, rhs, w, sc, cfg); break;
    default: lu_syncfree_w<T, WF, 8>(s, st, pf, small, rhs, w, sc, cfg); break;
    }
}

template <class T>
void lu_syncfree(hipStream_t s, const Structure &st, const PackedFactor<T> &pf, T small, const T *rhs, T *w,
                 const Scalars *sc, const SweepCfg &cfg) {
    FC_REQUIRE(syncfree_sweeps(st) && cfg.tmp && cfg.sf, FC_ERR_ARGUMENT, "dependency-driven sweeps not set up");
    switch (st.ell_f) {
    case 3: lu_syncfree_b<T, 3>(s, st, pf, small, rhs, w, sc, cfg); break;
    case 4: lu_syncfree_b<T, 4>(s, st, pf, small, rhs, w, sc, cfg); break;
    default: lu_syncfree_b<T, 8>(s, st, pf, small, rhs, w, sc, cfg); break;
    }
    FC_HIP_CHECK(hipGetLastError());
}

template <class T>
void lu_launch_t(hipStream_t s, const Structure &st, const T *a, const T *d, T small, const T *rhs, T *w,
                 const Scalars *sc, const SweepCfg *cfg, const PackedFactor<T> *pf) {
    if (cfg && cfg->sf && cfg->parts && pf && pf->af) {
        if constexpr (sizeof(T) == sizeof(double)) lu_parts64(s, st, *pf, small, rhs, w, sc, *cfg);
        else lu_parts32(s, st, *pf, small, rhs, w, sc, *cfg);
        return;
    }
    if (cfg && cfg->sf && pf && pf->af) {
        lu_syncfree<T>(s, st, *pf, small, rhs, w, sc, *cfg);
        return;
    }
    if (pf && pf->af) {
        sweeps_packed<T>(s, st, *pf, small, rhs, w, sc);
        return;
    }
    const int *ptr = st.ioffset.as<int>(), *ja = st.ja.as<int>(), *dg = st.diag.as<int>();
    const int *rf = st.rows_f.as<int>(), *rb = st.rows_b.as<int>();
    for (int l = 0; l < st.nlev_f; ++l) {
        int beg = st.lvl_f[l], cnt = st.lvl_f[l + 1] - beg;
        k_fwd_level<T><<<grid_for(cnt, 256), 256, 0, s>>>(rf, beg, cnt, ptr, ja, dg, a, d, rhs, w, sc);
    }
    for (int l = 0; l < st.nlev_b; ++l) {
        int beg = st.lvl_b[l], cnt = st.lvl_b[l + 1] - beg;
        k_bwd_level<T><<<grid_for(cnt, 256), 256, 0, s>>>(rb, beg, cnt, ptr, ja, dg, a, d, small, w, sc);
    }
}

void lu_launch64(hipStream_t s, const Structure &st, const double *a, const double *d, double small,
                 const double *rhs, double *w, const Scalars *sc, const SweepCfg *cfg,
                 const PackedFactor<double> *pf) {
    lu_launch_t<double>(s, st, a, d, small, rhs, w, sc, cfg, pf);
}

void lu_launch32(hipStream_t s, const Structure &st, const float *a, const float *d, float small, const float *rhs,
                 float *w, const Scalars *sc, const SweepCfg *cfg, const PackedFactor<float> *pf) {
    lu_launch_t<float>(s, st, a, d, small, rhs, w, sc, cfg, pf);
}

void mark_sweep_input64(hipStream_t s, int n, double *tmp) {
    k_sf_mark<double><<<grid_for(n, 256), 256, 0, s>>>(n, tmp, nullptr);
    FC_HIP_CHECK(hipGetLastError());
}
void mark_sweep_input32(hipStream_t s, int n, float *tmp) {
    k_sf_mark<float><<<grid_for(n, 256), 256, 0, s>>>(n, tmp, nullptr);
    FC_HIP_CHECK(hipGetLastError());
}

bool packed_sweeps(const Structure &st) { return st.levels_ready && st.ell_f > 0 && st.ell_b > 0; }

void pack_factor64(hipStream_t s, const Structure &st, const double *a, const double *d, double *af, double *df,
                   double *ab, double *db) {
    pack_factor_t<double>(s, st, a, d, af, df, ab, db);
}

void pack_factor32(hipStream_t s, const Structure &st, const float *a, const float *d, float *af, float *df,
                   float *ab, float *db) {
    pack_factor_t<float>(s, st, a, d, af, df, ab, db);
}

// ----------------------------------------------------------- reductions

__global__ void k_sum_parts(int nparts, const double *__restrict__ pa, const double *__restrict__ pb,
                            double *__restrict__ out) {
    __shared__ double sh[kFinBlock / kWave];
    double a = 0.0, b = 0.0;
    for (int i = threadIdx.x; i < nparts; i += kFinBlock) {
        a += pa[i];
        if (pb) b += pb[i];
    }
    a = block_sum<kFinBlock>(a, sh);
    b = block_sum<kFinBlock>(b, sh);
    if (threadIdx.x == 0) {
        out[0] = a;
        out[1] = b;
    }
}

template <class TA, class TB, int OP>
__global__ __launch_bounds__(kRedBlock) void k_reduce(long long n, const TA *__restrict__ x, const TB *__restrict__ y,
                                                      double *__restrict__ pa, double *__restrict__ pb) {
    __shared__ double sh[kRedBlock / kWave];
    double a = 0.0, b = 0.0;
    for (long long i = blockIdx.x * (long long)kRedBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kRedBlock) {
        double xv = (double)x[i];
        if (OP == 0) a += xv * (double)y[i];        // dot
        else if (OP == 1) { a += fabs(xv); b += xv * xv; }   // L1 and L2^2
    }
    a = block_sum<kRedBlock>(a, sh);
    if (OP == 1) b = block_sum<kRedBlock>(b, sh);
    if (threadIdx.x == 0) {
        pa[blockIdx.x] = a;
        if (OP == 1) pb[blockIdx.x] = b;
    }
}

void dot_launch64(hipStream_t s, int n, const double *x, const double *y, double *pa) {
    k_reduce<double, double, 0><<<red_grid(n), kRedBlock, 0, s>>>(n, x, y, pa, nullptr);
}

void norms_launch64(hipStream_t s, int n, const double *x, double *pa, double *pb) {
    k_reduce<double, double, 1><<<red_grid(n), kRedBlock, 0, s>>>(n, x, x, pa, pb);
}

void sum_parts_launch(hipStream_t s, int nparts, const double *pa, const double *pb, double *out) {
    k_sum_parts<<<1, kFinBlock, 0, s>>>(nparts, pa, pb, out);
}

}  // namespace fcap
