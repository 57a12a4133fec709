// The library's kernels on the CPU (wave_emu.h): their text, cut from the sources by the test
// that builds this file, and an entry point for each.
#include "fcap.h"
#include "fcap_kernels.h"

namespace fcap {
#include "cut_syncfree.inc"
namespace parts {
#include "cut_parts.inc"
}
namespace rows {
#include "cut_rows.inc"
}
namespace slices {
#include "cut_slices.inc"
}
namespace solver {
#include "cut_solver.inc"
}
}  // namespace fcap

using namespace fcap;

namespace {

struct Run {
    int grid, seed, resident, freeze_steps;
    double freeze, freeze_store;
    long long wait_ticks, max_steps;
    const unsigned *order;   // or null
};
emu::Policy policy(const Run &r) {
    emu::Policy p;
    p.seed = (unsigned)r.seed;
    p.freeze = r.freeze;
    p.freeze_store = r.freeze_store;
    p.freeze_steps = r.freeze_steps;
    if (r.resident > 0) p.resident = (unsigned)r.resident;
    if (r.order) p.order.assign(r.order, r.order + r.grid);
    p.max_steps = r.max_steps;
    return p;
}
SyncFree state(const Run &r) {
    SyncFree sf{};
    sf.wait_us = (int)r.wait_ticks;
    sf.rate_khz = 1000;
    return sf;
}

template <class T, int W>
void sliced_w(int mode, int grid, int n, const slices::SliceView &S, const T *v, const T *x, const T *b, const T *d, T *y,
              double *pa, double *pb) {
    const Run r{grid, 1, 2, 1, 0.0, 0.0, 0, 1000000000, nullptr};
    emu::launch((unsigned)grid, kSpmvRows, policy(r), [&]() {
        if (mode == 2) slices::k_sliced<T, W, 2>(n, S, v, x, b, d, y, pa, pb, nullptr, 0.f);
        else if (mode == 3) slices::k_sliced<T, W, 3>(n, S, v, x, b, d, y, pa, pb, nullptr, 0.f);
        else slices::k_sliced<T, W, 4>(n, S, v, x, b, d, y, pa, pb, nullptr, 0.7f);
    });
}
// y (modes 2, 3: A x; 4: a damped Jacobi step) by the sliced kernels; wide slices found
template <class T>
int sliced(int mode, int n, int w, const int *ptr, const int *ja, const double *a, const T *x, const T *b, const T *d,
           T *y, double *pa, double *pb) {
    const int ns = (n + 63) / 64, grid = (n + kSpmvRows - 1) / kSpmvRows;
    std::vector<int> base((size_t)ns * w);
    std::vector<unsigned> off((size_t)ns * ((w + 1) / 2) * 64, 0xffffffffu);
    std::vector<T> v((size_t)ns * 64 * w);
    int wide = 0;
    const Run r{grid, 1, 2, 1, 0.0, 0.0, 0, 1000000000, nullptr};
    emu::launch((unsigned)grid, 256, policy(r), [&]() {
        slices::k_slice_columns(n, w, ptr, ja, base.data(), off.data(), &wide);
    });
    emu::launch((unsigned)grid, 256, policy(r), [&]() { slices::k_slice_values<T>(n, w, ptr, a, v.data()); });
    slices::SliceView S;
    S.w = w;
    S.base = base.data();
    S.off = off.data();
    S.ptr = ptr;
    S.ja = ja;
    switch (w) {
    case 4: sliced_w<T, 4>(mode, grid, n, S, v.data(), x, b, d, y, pa, pb); break;
    case 5: sliced_w<T, 5>(mode, grid, n, S, v.data(), x, b, d, y, pa, pb); break;
    case 7: sliced_w<T, 7>(mode, grid, n, S, v.data(), x, b, d, y, pa, pb); break;
    default: sliced_w<T, 8>(mode, grid, n, S, v.data(), x, b, d, y, pa, pb); break;
    }
    return wide;
}

template <int W>
int rows_sweeps(const Run &r, int n, const int *const rows[2], const int *const cnt[2], const int *const col[2],
                const double *const val[2], const double *const piv[2], const double *rhs, double small, double *tmp,
                double *w) {
    SyncFree sf = state(r);
    bool ended = emu::launch((unsigned)r.grid, 64, policy(r), [&]() {
        rows::k_sweep_syncfree<double, W, false>(n, rows[0], cnt[0], col[0], val[0], piv[0], rhs, small, tmp, w, &sf,
                                                 nullptr);
    });
    if (ended && !sf.abort)
        ended = emu::launch((unsigned)r.grid, 64, policy(r), [&]() {
            rows::k_sweep_syncfree<double, W, true>(n, rows[1], cnt[1], col[1], val[1], piv[1], tmp, small, w, tmp,
                                                    &sf, nullptr);
        });
    return !ended ? 2 : sf.abort ? 1 : 0;
}

template <class T, int W, bool BWD>
int parts_sweep(const Run &r, int nparts, int npk, const int *codes, const unsigned char *step, const int *win,
                const T *vals, const T *in, double small, T *out, T *mk, T *z) {
    SyncFree sf = state(r);
    const parts::PartView P{npk, codes, step};
    const bool ended = emu::launch((unsigned)r.grid, parts::PartShape<W>::kBlock, policy(r), [&]() {
        parts::k_sweep_parts<T, W, BWD>(nparts, P, win, vals, in, (T)small, out, mk, z, &sf, nullptr);
    });
    return !ended ? 2 : sf.abort ? 1 : 0;
}
template <class T, int W>
int parts_either(const Run &r, int bwd, int nparts, int npk, const int *codes, const unsigned char *step,
                 const int *win, const void *vals, const void *in, double small, void *out, void *mk, void *z) {
    auto f = [&](auto b) {
        return parts_sweep<T, W, decltype(b)::value>(r, nparts, npk, codes, step, win, (const T *)vals, (const T *)in,
                                                     small, (T *)out, (T *)mk, (T *)z);
    };
    return bwd ? f(std::true_type{}) : f(std::false_type{});
}

}  // namespace

extern "C" {

// the kernels that begin an iteration and end the solve (k_cg_p<float>, k_bi_p<float>), with
// residual sums a, b in every one of the nv partials; what they leave of `done` and the direction
int emu_begin(const Run *r, int bicg, int n, float *p, const float *z, double a, double b, double resmax, int nv,
              int *done) {
    Scalars sc{};
    sc.resmax = resmax;
    sc.res0 = sc.sk = sc.gam = sc.alf = sc.beto = 1.0;
    sc.nsw = 100;
    sc.status = kStatusRunning;
    std::vector<double> pv((size_t)kVecParts * nv), pz(nv, 1.0);
    for (int i = 0; i < nv; ++i) {
        pv[(size_t)kVecParts * i] = a;
        pv[(size_t)kVecParts * i + 1] = b;
        pv[(size_t)kVecParts * i + 2] = 1.0;
    }
    const bool ended = emu::launch((unsigned)r->grid, kRedBlock, policy(*r), [&]() {
        if (bicg) solver::k_bi_p<float>(n, p, z, z, &sc, pv.data(), nv, 0);
        else solver::k_cg_p<float, false>(n, p, z, nullptr, &sc, pv.data(), nv, pz.data(), nv, 0);
    });
    *done = sc.done;
    return !ended;
}

int emu_rows(const Run *r, int width, int n, const int *const rows[2], const int *const cnt[2], const int *const col[2],
             const double *const val[2], const double *const piv[2], const double *rhs, double small, double *tmp,
             double *w) {
    if (width == 3) return rows_sweeps<3>(*r, n, rows, cnt, col, val, piv, rhs, small, tmp, w);
    return rows_sweeps<8>(*r, n, rows, cnt, col, val, piv, rhs, small, tmp, w);
}

// The forward part-wise sweep (W = 3, FP64) of one part, with values put into its output from
// outside: value k at slot at[k] after step when[k].
int emu_parts_fed(const Run *r, int npk, const int *codes, const unsigned char *step, const int *win,
                  const double *vals, const double *in, double *out, double *mk, int nfed, const int *at,
                  const double *value, const long long *when) {
    SyncFree sf = state(*r);
    const parts::PartView P{npk, codes, step};
    emu::Policy p = policy(*r);
    p.each_step = [&](long long t) {
        for (int k = 0; k < nfed; ++k)
            if (t == when[k]) out[at[k]] = value[k];
    };
    const bool ended = emu::launch(1, parts::PartShape<3>::kBlock, p, [&]() {
        parts::k_sweep_parts<double, 3, false>(1, P, win, vals, in, 0.0, out, mk, nullptr, &sf, nullptr);
    });
    return !ended ? 2 : sf.abort ? 1 : 0;
}

int emu_sliced32(int mode, int n, int w, const int *ptr, const int *ja, const double *a, const float *x, const float *b,
                 const float *d, float *y, double *pa, double *pb) {
    return sliced<float>(mode, n, w, ptr, ja, a, x, b, d, y, pa, pb);
}

int emu_ring() { return parts::kRing; }

int emu_parts(const Run *r, int f32, int width, int bwd, int nparts, int npk, const int *codes,
              const unsigned char *step, const int *win, const void *vals, const void *in, double small, void *out,
              void *mk, void *z) {
#define CALL(T, W) parts_either<T, W>(*r, bwd, nparts, npk, codes, step, win, vals, in, small, out, mk, z)
    if (f32) return width == 3 ? CALL(float, 3) : width == 4 ? CALL(float, 4) : CALL(float, 8);
    return width == 3 ? CALL(double, 3) : width == 4 ? CALL(double, 4) : CALL(double, 8);
#undef CALL
}

}  // extern "C"
