// Matrix rows in slices of 64 for the products inside the solvers' iterations: entry k of
// the slice's rows together (64 values of one load each), the columns as 16-bit offsets
// from the smallest column of the entry in the slice.  A row's entries keep the CSR order
// and its padding is skipped, so every result equals the CSR kernel's (k_spmv) bit for bit,
// the partial sums included (one per 256 rows, added in the same order).
//
// Bound by the bytes of the matrix: at seven entries a row 4 + 2.3 B an entry in FP32
// instead of 4 + 4 and a row pointer, and one round of loads before the gathers of x
// instead of three (pointer, entries, LDS).  Matrix loads are non-temporal (temporal: FCG
// at 192^3 186 against 183 ms).  With CSR products and now: Jacobi-PCG 97 x 83 x 61 24.5 and
// 21.0 ms, DIC-PCG 128^3 142.6 and 137.2, flexible CG without a network at 128^3 24.2 and
// 20.0, with it at 192^3 203 and 183.
#include <algorithm>

#include "fcap_kernels.h"
#include "fcap_linalg.h"

namespace fcap {

namespace {

constexpr unsigned kPad = 0xffffu;      // offset of a padding entry
constexpr int kMinWidth = 4, kMaxWidth = 8;
// Rows from which a matrix whose slices are mostly wide (below) keeps the CSR rows
constexpr int kWideRows = 200000;

inline int grid_for(long long n, int block) { return (int)std::max<long long>(1, (n + block - 1) / block); }
__host__ __device__ inline int slices_of(int n) { return (n + kWave - 1) / kWave; }

__global__ void k_row_width(int n, const int *__restrict__ ptr, int *__restrict__ w) {
    int len = 0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        len = max(len, ptr[i + 1] - ptr[i]);
#pragma unroll
    for (int off = 32; off; off >>= 1) len = max(len, __shfl_xor(len, off));
    if ((threadIdx.x & 63) == 0) atomicMax(w, len);
}

// Bases and offsets of a slice, one wave each; base -1: some entry's columns span more
// than 16 bits, the slice then reads its columns from the CSR array (a wide slice; counted).
__global__ void k_slice_columns(int n, int width, const int *__restrict__ ptr, const int *__restrict__ ja,
                                int *__restrict__ base, unsigned *__restrict__ off, int *__restrict__ nwide) {
    const int slice = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, lane = threadIdx.x & 63;
    if (slice * kWave >= n) return;
    const int row = slice * kWave + lane;
    const int s = row < n ? ptr[row] : 0, len = row < n ? ptr[row + 1] - s : 0;
    bool wide = false;
    for (int k = 0; k < width; ++k) {
        const int col = k < len ? ja[s + k] : -1;
        int lo = col < 0 ? 0x7fffffff : col, hi = col;
#pragma unroll
        for (int o = 32; o; o >>= 1) {
            lo = min(lo, __shfl_xor(lo, o));
            hi = max(hi, __shfl_xor(hi, o));
        }
        if (hi < 0) lo = 0;   // padding only
        wide |= hi - lo >= (int)kPad;
        if (lane == 0) base[slice * width + k] = lo;
        const unsigned d = col < 0 ? kPad : (unsigned)(col - lo) & 0xffffu;
        unsigned short *o16 = reinterpret_cast<unsigned short *>(
            off + ((size_t)slice * ((width + 1) / 2) + k / 2) * kWave + lane);
        o16[k & 1] = (unsigned short)d;
    }
    if (wide && lane == 0) {
        for (int k = 0; k < width; ++k) base[slice * width + k] = -1;
        atomicAdd(nwide, 1);
    }
}

template <class T>
__global__ void k_slice_values(int n, int width, const int *__restrict__ ptr, const double *__restrict__ a,
                               T *__restrict__ v) {
    const int row = blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= slices_of(n) * kWave) return;
    const int s = row < n ? ptr[row] : 0, len = row < n ? ptr[row + 1] - s : 0;
    T *o = v + (size_t)(row >> 6) * width * kWave + (row & 63);
    for (int k = 0; k < width; ++k) o[(size_t)k * kWave] = k < len ? (T)a[s + k] : T(0);
}

// MODE 2: y = A x with y.b partials; 3: and y^2 partials; 4: y = x + omega (b - A x) / d
template <class T, int W, int MODE>
__global__ __launch_bounds__(kSpmvRows) void k_sliced(int n, SliceView S, const T *__restrict__ val,
                                                      const T *__restrict__ x, const T *__restrict__ b,
                                                      const T *__restrict__ d, T *__restrict__ y,
                                                      double *__restrict__ partA, double *__restrict__ partB,
                                                      const Scalars *__restrict__ sc, float omega) {
    __shared__ double red[2][kSpmvWaves];
    if (sc && sc->done) return;
    constexpr int W2 = (W + 1) / 2;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int slice = blockIdx.x * kSpmvWaves + w;
    const int row = slice * kWave + lane;
    double pa = 0.0, pb = 0.0;
    if (slice * kWave < n) {
        const bool valid = row < n;
        const T *v = val + (size_t)slice * W * kWave + lane;
        const unsigned *o = S.off + (size_t)slice * W2 * kWave + lane;
        unsigned o2[W2];
        T av[W], xv[W];
#pragma unroll
        for (int k = 0; k < W2; ++k) o2[k] = __builtin_nontemporal_load(o + k * kWave);
#pragma unroll
        for (int k = 0; k < W; ++k) av[k] = __builtin_nontemporal_load(v + k * kWave);
        const T bv = valid ? b[row] : T(0);
        const int *base = S.base + slice * W;
        bool in[W];
        if (base[0] >= 0) {
#pragma unroll
            for (int k = 0; k < W; ++k) {
                const unsigned t = (k & 1) ? o2[k / 2] >> 16 : o2[k / 2] & 0xffffu;
                in[k] = t != kPad;
                xv[k] = in[k] ? x[base[k] + (int)t] : T(0);
            }
        } else {
            const int s = valid ? S.ptr[row] : 0, len = valid ? S.ptr[row + 1] - s : 0;
#pragma unroll
            for (int k = 0; k < W; ++k) {
                in[k] = k < len;
                xv[k] = in[k] ? x[S.ja[s + k]] : T(0);
            }
        }
        T acc = MODE == 4 ? bv : T(0);
#pragma unroll
        for (int k = 0; k < W; ++k) {
            const T p = av[k] * xv[k], t = MODE == 4 ? acc - p : acc + p;
            acc = in[k] ? t : acc;
        }
        if (valid) {
            if (MODE == 4) {
                y[row] = x[row] + (T)omega * (acc / d[row]);
            } else {
                y[row] = acc;
                pa = (double)acc * (double)bv;
                if (MODE == 3) pb = (double)acc * (double)acc;
            }
        }
    }
    if (MODE != 4) {
        pa = wave_sum(pa);
        if (MODE == 3) pb = wave_sum(pb);
        if (lane == 0) {
            red[0][w] = pa;
            red[1][w] = pb;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            double s = 0.0, t = 0.0;
            for (int i = 0; i < kSpmvWaves; ++i) {
                s += red[0][i];
                t += red[1][i];
            }
            partA[blockIdx.x] = s;
            if (MODE == 3) partB[blockIdx.x] = t;
        }
    }
}

template <class T, int MODE>
void sliced(hipStream_t s, int n, const SliceView &S, const T *v, const T *x, const T *b, const T *d, T *y, double *pa,
            double *pb, const Scalars *sc, float omega) {
    const int g = spmv_grid(n);
    switch (S.w) {
    case 4: k_sliced<T, 4, MODE><<<g, kSpmvRows, 0, s>>>(n, S, v, x, b, d, y, pa, pb, sc, omega); break;
    case 5: k_sliced<T, 5, MODE><<<g, kSpmvRows, 0, s>>>(n, S, v, x, b, d, y, pa, pb, sc, omega); break;
    case 6: k_sliced<T, 6, MODE><<<g, kSpmvRows, 0, s>>>(n, S, v, x, b, d, y, pa, pb, sc, omega); break;
    case 7: k_sliced<T, 7, MODE><<<g, kSpmvRows, 0, s>>>(n, S, v, x, b, d, y, pa, pb, sc, omega); break;
    default: k_sliced<T, 8, MODE><<<g, kSpmvRows, 0, s>>>(n, S, v, x, b, d, y, pa, pb, sc, omega); break;
    }
}

}  // namespace

// Slices up to eight entries a row (what the kernels hold in registers) where padding is at
// most a quarter of them: 16-bit columns save as much.  Not where most slices are wide (a
// scattered numbering) and the matrix is large: their columns come a row at a time instead of
// a wave at a time through LDS, beside offsets read for nothing.  In ms, CSR and slices, 200
// Jacobi-PCG and 60 flexible CG iterations, randomly numbered boxes and tets: 97,336 rows 3.46
// and 3.48, 4.35 and 4.23; 131,712 (tets) 3.72 and 3.56, 4.43 and 4.35; 195,112 4.75 and 4.78,
// 5.69 and 5.76; 262,144 5.48 and 5.73, 6.54 and 6.76; 884,736 16.4 and 17.6, 13.6 and 15.4;
// 2,097,152 46.8 and 48.9, 41.3 and 45.5.
SliceView slices_for(fc_context *ctx, Structure &st) {
    if (!st.sl_ready) {
        hipStream_t s = ctx->stream;
        DevBuf wd(sizeof(int));
        fill_int(ctx, wd.as<int>(), 1, 0);
        k_row_width<<<std::min(grid_for(st.n, 256), 256), 256, 0, s>>>(st.n, st.ioffset.as<int>(), wd.as<int>());
        int w = 0;
        FC_HIP_CHECK(hipMemcpyAsync(&w, wd.get(), sizeof(int), hipMemcpyDeviceToHost, s));
        FC_HIP_CHECK(hipStreamSynchronize(s));
        w = std::max(w, kMinWidth);
        st.sl_w = w <= kMaxWidth && 4ll * st.nnz >= 3ll * st.n * w ? w : 0;
        if (st.sl_w) {
            const size_t ns = (size_t)slices_of(st.n);
            fill_int(ctx, wd.as<int>(), 1, 0);   // now the wide slices
            st.sl_base.alloc(sizeof(int) * ns * w);
            st.sl_off.alloc(sizeof(unsigned) * ns * ((w + 1) / 2) * kWave);
            FC_HIP_CHECK(hipMemsetAsync(st.sl_off.get(), 0xff, sizeof(unsigned) * ns * ((w + 1) / 2) * kWave, s));
            k_slice_columns<<<grid_for((long long)ns * kWave, 256), 256, 0, s>>>(
                st.n, w, st.ioffset.as<int>(), st.ja.as<int>(), st.sl_base.as<int>(), st.sl_off.as<unsigned>(),
                wd.as<int>());
            FC_HIP_CHECK(hipGetLastError());
            if (st.n >= kWideRows) {
                int wide = 0;
                FC_HIP_CHECK(hipMemcpyAsync(&wide, wd.get(), sizeof(int), hipMemcpyDeviceToHost, s));
                FC_HIP_CHECK(hipStreamSynchronize(s));
                if (2ll * wide > (long long)ns) {
                    st.sl_w = 0;
                    st.sl_base.release();
                    st.sl_off.release();
                }
            }
        }
        st.sl_ready = true;
    }
    SliceView S;
    S.w = st.sl_w;
    S.base = st.sl_base.as<int>();
    S.off = st.sl_off.as<unsigned>();
    S.ptr = st.ioffset.as<int>();
    S.ja = st.ja.as<int>();
    return S;
}

size_t slice_count(int n, const SliceView &S) { return (size_t)slices_of(n) * kWave * (size_t)S.w; }

void slice_values64(hipStream_t s, int n, const SliceView &S, const double *a, double *v) {
    k_slice_values<double><<<grid_for((long long)slices_of(n) * kWave, 256), 256, 0, s>>>(n, S.w, S.ptr, a, v);
    FC_HIP_CHECK(hipGetLastError());
}
void slice_values32(hipStream_t s, int n, const SliceView &S, const double *a, float *v) {
    k_slice_values<float><<<grid_for((long long)slices_of(n) * kWave, 256), 256, 0, s>>>(n, S.w, S.ptr, a, v);
    FC_HIP_CHECK(hipGetLastError());
}

void sliced_product64(hipStream_t s, int n, const SliceView &S, const double *v, const double *x, const double *b,
                      double *y, double *pa, double *pb, const Scalars *sc) {
    if (pb) sliced<double, 3>(s, n, S, v, x, b, nullptr, y, pa, pb, sc, 0.f);
    else sliced<double, 2>(s, n, S, v, x, b, nullptr, y, pa, nullptr, sc, 0.f);
}
void sliced_product32(hipStream_t s, int n, const SliceView &S, const float *v, const float *x, const float *b,
                      float *y, double *pa, double *pb, const Scalars *sc) {
    if (pb) sliced<float, 3>(s, n, S, v, x, b, nullptr, y, pa, pb, sc, 0.f);
    else sliced<float, 2>(s, n, S, v, x, b, nullptr, y, pa, nullptr, sc, 0.f);
}
void sliced_jacobi32(hipStream_t s, int n, const SliceView &S, const float *v, const float *x, const float *b,
                     const float *d, float omega, float *y, const Scalars *sc) {
    sliced<float, 4>(s, n, S, v, x, b, d, y, nullptr, nullptr, sc, omega);
}

}  // namespace fcap
