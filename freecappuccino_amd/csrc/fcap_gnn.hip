// Learned preconditioner: a message-passing network over the cell graph,
// evaluated and trained with hand-written kernels.
//
// Network (H = 32, L = 4), for a residual r on a system with diagonal a_ii:
//   s = rms(r/a_ii), u = (r/a_ii)/s, h0 = relu(w_enc u + b_enc)
//   layer l: c_k = g0 + g1 e1_k + g2 e2_k (edge gate of CSR entry k = (i, j))
//            agg_i = sum_k c_k h_j ;  h_i <- h_i + relu(Ws h_i + Wm agg_i + b)
//   y = w_dec . h + b_dec, z = s (u + y)
// Edge features of entry (i, j), face f: e1 = (|S_f|/|x_j - x_i|)/a_ii, e2 = 1 - |cos(S_f, x_j - x_i)|.
//
// Precision: weights, stored activations and the aggregated messages are
// BF16; each layer's node GEMM [h | agg] (64) -> 32 runs on MFMA
// (v_mfma_f32_16x16x16_bf16, FP32 accumulation); gathers, gates and the
// epilogue are FP32.  One wavefront owns 64 consecutive cells: each lane
// gathers its cell's messages, the wave stages [h | agg] in LDS, four 16-cell
// tiles x two 16-output tiles x four K steps of MFMA produce the layer output.
//
// Training minimises the energy norm of the preconditioned error,
// (z - e)^T A (z - e) / (e^T A e), over (r, e) pairs generated by IC(0)-PCG
// iterates; the backward pass mirrors the forward (MFMA for the input and
// weight gradients, gather over transposed entries for the messages) and
// writes per-wave / per-block partials that a reduction kernel sums in a fixed
// order.  Adam updates an FP32 master copy; the BF16 copy feeds the kernels.

#include <algorithm>
#include <atomic>
#include <climits>
#include <numeric>
#include <thread>
#include <cmath>
#include <cstring>
#include <random>
#include <vector>

#include "fcap_gnn.h"
#include "fcap_linalg.h"
#include "fcap_solvers.h"
#include "fcap_system.h"

using fcap::DevBuf;

namespace fcap {

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short bf16_t;

constexpr int H = kGnnH;
constexpr int kWaves = 4;        // waves per workgroup of the backward kernels
constexpr int kLayerWaves = 1;   // waves per workgroup of the forward layer kernel
constexpr int kLdA = 72;   // padded row of the [h | agg] tile, bf16 elements (144 bytes)
constexpr int kLdC = 36;   // the same bytes viewed as an FP32 output tile row
constexpr int kLdD = 40;   // padded row of the d_out tile, bf16 elements

inline int grid_for(long long n, int block) {
    long long g = (n + block - 1) / block;
    return (int)std::max<long long>(1, std::min<long long>(g, 1 << 30));
}

__device__ inline float bf2f(bf16_t b) { return __uint_as_float(((unsigned)b) << 16); }

// round to nearest even; NaN stays NaN
// (gfx950's v_cvt_pk_bf16_f32: round to nearest even, NaN stays NaN)
__device__ inline bf16_t f2bf(float f) { return __builtin_bit_cast(bf16_t, (__bf16)f); }

// two floats -> packed BF16 pair (lo, hi), one conversion instruction
__device__ inline unsigned f2bf2(float lo, float hi) {
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    const bf16x2_t v = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(unsigned, v);
}

__device__ inline float bfround(float f) { return bf2f(f2bf(f)); }

__device__ inline void store_row_bf16(bf16_t *__restrict__ dst, const float *src) {
    uint4 *p = reinterpret_cast<uint4 *>(dst);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        unsigned ww[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) ww[t] = f2bf2(src[v * 8 + 2 * t], src[v * 8 + 2 * t + 1]);
        p[v] = make_uint4(ww[0], ww[1], ww[2], ww[3]);
    }
}

// Activation rows in HBM (h0..h4) keep a cell's 32 BF16 channels in the order
// [4g .. 4g+3, 16+4g .. 16+4g+3] for g = 0..3 (16 bytes per group g); the
// LDS tiles of the layer kernels keep the natural order, and a group goes
// there as two 8-byte halves.
__device__ inline int hrow_channel(int g, int t) { return t < 4 ? 4 * g + t : 16 + 4 * g + (t - 4); }

// 16 bytes of a stored row (group g) -> its 8 channels, local order t = 0..7
__device__ inline void unpack8(uint4 w, float *v) {
    const unsigned ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        v[2 * t] = __uint_as_float(ww[t] << 16);
        v[2 * t + 1] = __uint_as_float(ww[t] & 0xffff0000u);
    }
}

__device__ inline uint4 pack8(const float *v) {
    return make_uint4(f2bf2(v[0], v[1]), f2bf2(v[2], v[3]), f2bf2(v[4], v[5]), f2bf2(v[6], v[7]));
}

// whole stored row <-> natural channel order
__device__ inline void load_hrow(const bf16_t *__restrict__ src, float *dst) {
    const uint4 *p = reinterpret_cast<const uint4 *>(src);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        float v[8];
        unpack8(p[g], v);
#pragma unroll
        for (int t = 0; t < 8; ++t) dst[hrow_channel(g, t)] = v[t];
    }
}

__device__ inline void store_hrow(bf16_t *__restrict__ dst, const float *src) {
    uint4 *p = reinterpret_cast<uint4 *>(dst);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        float v[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) v[t] = src[hrow_channel(g, t)];
        p[g] = pack8(v);
    }
}

// agg (natural order) += cg * stored row given as its four 16-byte groups
__device__ inline void add_hrow(const uint4 *raw, float cg, float *agg) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        float v[8];
        unpack8(raw[g], v);
#pragma unroll
        for (int t = 0; t < 8; ++t) agg[hrow_channel(g, t)] = fmaf(cg, v[t], agg[hrow_channel(g, t)]);
    }
}

// --------------------------------------------------------------- graph data

__global__ void k_gnn_edges(int n, const int *__restrict__ ptr, const int *__restrict__ ja,
                            const int *__restrict__ diagpos, const int *__restrict__ kface,
                            const double *__restrict__ arx, const double *__restrict__ ary,
                            const double *__restrict__ arz, const double *__restrict__ xc,
                            const double *__restrict__ yc, const double *__restrict__ zc,
                            const double *__restrict__ a, uint32_t *__restrict__ ef, float *__restrict__ dg) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int dp = diagpos[i];
    const double di = a[dp];
    dg[i] = (float)di;
    for (int k = ptr[i]; k < ptr[i + 1]; ++k) {
        const int e = kface[k];   // (face << 1) | side, -1 on the diagonal
        if (k == dp || e < 0) {
            ef[k] = 0u;
            continue;
        }
        const int f = e >> 1;
        const int j = ja[k];
        const double sx = arx[f], sy = ary[f], sz = arz[f];
        const double dx = xc[j] - xc[i], dy = yc[j] - yc[i], dz = zc[j] - zc[i];
        const double sa = sqrt(sx * sx + sy * sy + sz * sz), dd = sqrt(dx * dx + dy * dy + dz * dz);
        const double e1 = (sa / dd) / di;
        const double e2 = 1.0 - fabs(sx * dx + sy * dy + sz * dz) / (sa * dd);
        ef[k] = (uint32_t)f2bf((float)e1) | ((uint32_t)f2bf((float)e2) << 16);
    }
}

// entries that are neither a face pair nor a diagonal (none on a plain mesh) map to themselves
__global__ void k_gnn_trans_init(int nnz, int *__restrict__ trans) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < nnz) trans[k] = k;
}

__global__ void k_gnn_trans(int nif, const int *__restrict__ ij, const int *__restrict__ ji, int *__restrict__ trans) {
    int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nif) return;
    trans[ij[f]] = ji[f];
    trans[ji[f]] = ij[f];
}

__global__ void k_gnn_trans_diag(int n, const int *__restrict__ diagpos, int *__restrict__ trans) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) trans[diagpos[i]] = diagpos[i];
}

__global__ void k_gnn_width(int n, const int *__restrict__ ptr, int *__restrict__ wmax) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) atomicMax(wmax, ptr[i + 1] - ptr[i] - 1);
}

__global__ void k_gnn_ell(int n, int ew, const int *__restrict__ ptr, const int *__restrict__ ja,
                          const int *__restrict__ diagpos, const uint32_t *__restrict__ ef,
                          const int *__restrict__ trans, int *__restrict__ ecnt, int *__restrict__ enbr,
                          uint32_t *__restrict__ eef, uint32_t *__restrict__ eeft) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int dp = diagpos[i];
    int slot = 0;
    for (int k = ptr[i]; k < ptr[i + 1] && slot < ew; ++k) {
        if (k == dp) continue;
        const size_t o = (size_t)slot * n + i;
        enbr[o] = ja[k];
        eef[o] = ef[k];
        eeft[o] = ef[trans[k]];
        ++slot;
    }
    ecnt[i] = slot;
    for (int k = slot; k < ew; ++k) {
        const size_t o = (size_t)k * n + i;
        enbr[o] = i;
        eef[o] = 0u;
        eeft[o] = 0u;
    }
}

// centroid of each block of 64 consecutive cells (mean of the cell centres)
__global__ void k_gnn_block_centre(int n, int nblk, const double *__restrict__ xc, const double *__restrict__ yc,
                                   const double *__restrict__ zc, float *__restrict__ cen) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nblk) return;
    const int i0 = b * 64, i1 = min(n, i0 + 64);
    double sx = 0.0, sy = 0.0, sz = 0.0;
    for (int i = i0; i < i1; ++i) {
        sx += xc[i];
        sy += yc[i];
        sz += zc[i];
    }
    const double inv = 1.0 / (double)(i1 - i0);
    cen[3 * b] = (float)(sx * inv);
    cen[3 * b + 1] = (float)(sy * inv);
    cen[3 * b + 2] = (float)(sz * inv);
}

// 21-bit coordinate spread to every third bit of a 63-bit Morton code
__host__ __device__ inline uint64_t spread3(uint64_t v) {
    v &= 0x1fffffull;
    v = (v | v << 32) & 0x1f00000000ffffull;
    v = (v | v << 16) & 0x1f0000ff0000ffull;
    v = (v | v << 8) & 0x100f00f00f00f00full;
    v = (v | v << 4) & 0x10c30c30c30c30c3ull;
    v = (v | v << 2) & 0x1249249249249249ull;
    return v;
}

// the blocks sorted by the Morton code of their centroid (ties by block index)
std::vector<int> block_order(const std::vector<float> &cen, int nblk) {
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int b = 0; b < nblk; ++b)
        for (int d = 0; d < 3; ++d) {
            lo[d] = std::min(lo[d], cen[3 * (size_t)b + d]);
            hi[d] = std::max(hi[d], cen[3 * (size_t)b + d]);
        }
    std::vector<std::pair<uint64_t, int>> key(nblk);
    const double top = (double)((1 << 21) - 1);
    for (int b = 0; b < nblk; ++b) {
        uint64_t code = 0;
        for (int d = 0; d < 3; ++d) {
            const double ext = (double)hi[d] - (double)lo[d];
            const double t = ext > 0.0 ? ((double)cen[3 * (size_t)b + d] - (double)lo[d]) / ext : 0.0;
            const uint64_t q = (uint64_t)std::min(top, std::max(0.0, t * top));
            code |= spread3(q) << (2 - d);
        }
        key[b] = {code, b};
    }
    std::sort(key.begin(), key.end());
    std::vector<int> order(nblk);
    for (int b = 0; b < nblk; ++b) order[b] = key[b].second;
    return order;
}

__global__ void k_cast_df(long long n, const double *__restrict__ x, float *__restrict__ y) {
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        y[i] = (float)x[i];
}

// ----------------------------------------------------------------- input

__global__ __launch_bounds__(256) void k_gnn_norm_part(int n, const float *__restrict__ r, const float *__restrict__ dg,
                                                       double *__restrict__ part, const Scalars *__restrict__ sc) {
    __shared__ double sh[256 / 64];
    if (sc && sc->done) return;
    double s = 0.0;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        double v = (double)r[i] / (double)dg[i];
        s += v * v;
    }
    s = block_sum<256>(s, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ __launch_bounds__(256) void k_gnn_norm_fin(int nparts, const double *__restrict__ part, int n,
                                                      float *__restrict__ s_out, const Scalars *__restrict__ sc) {
    __shared__ double sh[256 / 64];
    if (sc && sc->done) return;
    double s = 0.0;
    for (int i = threadIdx.x; i < nparts; i += 256) s += part[i];
    s = block_sum<256>(s, sh);
    if (threadIdx.x == 0) s_out[0] = (float)(sqrt(s / (double)n) + 1e-30);
}

// u = (r / a_ii) / s and the encoder output h0 = relu(w_enc u + b_enc) (BF16 rows).
// Four threads per cell, one 16-byte channel group each, so that a wave
// writes 16 whole rows (1 KiB) per store.
__global__ __launch_bounds__(256) void k_gnn_input(int n, const float *__restrict__ r, const float *__restrict__ dg,
                                                   const float *__restrict__ s, const bf16_t *__restrict__ w,
                                                   float *__restrict__ u, bf16_t *__restrict__ h0,
                                                   const Scalars *__restrict__ sc) {
    if (sc && sc->done) return;
    const float sv = s[0];
    const long long total = 4LL * n;
    for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < total;
         t += (long long)gridDim.x * blockDim.x) {
        const int i = (int)(t >> 2), g = (int)(t & 3);
        const float uv = (r[i] / dg[i]) / sv;
        if (g == 0) u[i] = uv;
        float hv[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int c = hrow_channel(g, k);
            hv[k] = fmaxf(bf2f(w[kGnnOffEncW + c]) * uv + bf2f(w[kGnnOffEncB + c]), 0.f);
        }
        reinterpret_cast<uint4 *>(h0 + (size_t)i * H)[g] = pack8(hv);
    }
}

// u only, for the first layer that computes the encoder rows itself
__global__ __launch_bounds__(256) void k_gnn_u(int n, const float *__restrict__ r, const float *__restrict__ dg,
                                               const float *__restrict__ s, float *__restrict__ u,
                                               const Scalars *__restrict__ sc) {
    if (sc && sc->done) return;
    const float sv = s[0];
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) u[i] = (r[i] / dg[i]) / sv;
}

// -------------------------------------------------------------- forward

// Neighbour lists of the layer kernels (GnnGraph's ELL, slot k of cell i at [k * n + i]).
struct GnnEll {
    int n;
    const int *cnt, *nbr;
    const uint32_t *ef, *eft;   // packed BF16 features of entry (i, j), and of (j, i)
};

// Edge gate c = g0 + g1 e1 + g2 e2, rounded to BF16 (the messages multiply BF16
// by BF16).  Messages and gates use fused multiply-adds, written out: the
// library is built without FP contraction.
__device__ inline float edge_gate(float g0, float g1, float g2, uint32_t e) {
    return bfround(fmaf(g2, bf2f((bf16_t)(e >> 16)), fmaf(g1, bf2f((bf16_t)(e & 0xffffu)), g0)));
}

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

// agg (natural order) += c1 row1 + c2 row2 for two stored rows given as their
// 16-byte groups, with BF16 gates c packed as (c1, c2): for each channel the two
// rows' values are paired into one register and v_dot2_f32_bf16 adds both
// products at once (two products of BF16 values are exact in FP32)
__device__ inline void add_hrow_pair(const uint4 *r1, const uint4 *r2, unsigned cpair, float *agg) {
    const bf16x2_t cp = __builtin_bit_cast(bf16x2_t, cpair);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const unsigned a[4] = {r1[g].x, r1[g].y, r1[g].z, r1[g].w};
        const unsigned b[4] = {r2[g].x, r2[g].y, r2[g].z, r2[g].w};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            // byte permutes: (a.lo, b.lo) for the channel of position 2t, (a.hi, b.hi) for 2t+1
            const unsigned lo = __builtin_amdgcn_perm(b[t], a[t], 0x05040100u);
            const unsigned hi = __builtin_amdgcn_perm(b[t], a[t], 0x07060302u);
            float &al = agg[hrow_channel(g, 2 * t)];
            float &ah = agg[hrow_channel(g, 2 * t + 1)];
            al = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, lo), cp, al, false);
            ah = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, hi), cp, ah, false);
        }
    }
}

// Fills the lane's [h | agg] features (FP32, BF16-rounded as stored) for the
// backward pass: a loop over the cell's own count.  The first layer rebuilds
// h0 of the cell and its neighbours from u (4 bytes per gather).
template <bool FIRST>
__device__ inline void gather_features(int node, bool valid, const GnnEll &E, const float *__restrict__ u,
                                       const bf16_t *__restrict__ h_in, const bf16_t *__restrict__ w,
                                       const bf16_t *__restrict__ lw, float *hv, float *agg) {
    const float g0 = bf2f(lw[2 * H * H + H]), g1 = bf2f(lw[2 * H * H + H + 1]), g2 = bf2f(lw[2 * H * H + H + 2]);
    if (FIRST) {
        const float uv = valid ? u[node] : 0.f;
#pragma unroll
        for (int c = 0; c < H; ++c)
            hv[c] = bfround(fmaxf(bf2f(w[kGnnOffEncW + c]) * uv + bf2f(w[kGnnOffEncB + c]), 0.f));
    } else {
        if (valid) load_hrow(h_in + (size_t)node * H, hv);
        else {
#pragma unroll
            for (int c = 0; c < H; ++c) hv[c] = 0.f;
        }
    }
#pragma unroll
    for (int c = 0; c < H; ++c) agg[c] = 0.f;
    if (!valid) return;
    const int cnt = E.cnt[node];
    for (int k = 0; k < cnt; ++k) {
        const int j = E.nbr[(size_t)k * E.n + node];
        const float c = edge_gate(g0, g1, g2, E.ef[(size_t)k * E.n + node]);
        if (FIRST) {
            const float uj = u[j];
#pragma unroll
            for (int ch = 0; ch < H; ++ch)
                agg[ch] = fmaf(c, bfround(fmaxf(bf2f(w[kGnnOffEncW + ch]) * uj + bf2f(w[kGnnOffEncB + ch]), 0.f)),
                               agg[ch]);
        } else {
            uint4 raw[4];
            const uint4 *p = reinterpret_cast<const uint4 *>(h_in + (size_t)j * H);
#pragma unroll
            for (int v = 0; v < 4; ++v) raw[v] = p[v];
            add_hrow(raw, c, agg);
        }
    }
}

// out(64 nodes x 32) = [h | agg](64 x 64) * [Ws^T ; Wm^T](64 x 32) on MFMA; result left in registers
// B fragments of [Ws^T ; Wm^T] for the lane: for K step kk and output tile ot,
// B[k][o] with o = ot*16 + lane%16, k = kk*16 + 4*(lane/16) .. +3 -- four
// consecutive weights of row o of Ws (k < 32) or Wm, one 8-byte load each.
__device__ inline void load_b_frags(const bf16_t *__restrict__ lw, int lane, bf16x4 bfr[4][2]) {
    const int q = lane >> 4, r16 = lane & 15;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int ot = 0; ot < 2; ++ot) {
            const int o = ot * 16 + r16, k = kk * 16 + 4 * q;
            const bf16_t *src = k < H ? lw + o * H + k : lw + H * H + o * H + (k - H);
            bfr[kk][ot] = *reinterpret_cast<const bf16x4 *>(src);
        }
}

// out(64 nodes x 32) = [h | agg](64 x 64, LDS) * [Ws^T ; Wm^T](64 x 32) on MFMA
__device__ inline void layer_gemm(const bf16_t *A, const bf16x4 bfr[4][2], int lane, f32x4 acc[4][2]) {
    const int q = lane >> 4, r16 = lane & 15;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int ot = 0; ot < 2; ++ot) acc[t][ot] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            // A[m][k]: m = 16t + lane%16, k = kk*16 + 4*(lane/16) .. +3 (one 8-byte LDS read)
            const bf16x4 afr = *reinterpret_cast<const bf16x4 *>(A + (16 * t + r16) * kLdA + kk * 16 + 4 * q);
#pragma unroll
            for (int ot = 0; ot < 2; ++ot)
                acc[t][ot] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(afr, bfr[kk][ot], acc[t][ot], 0, 0, 0);
        }
    }
}

// the lane's row of [h | agg] into the LDS tile as BF16, 16 bytes per store
__device__ inline void stage_row(bf16_t *A, int lane, const float *hv, const float *agg) {
    store_row_bf16(A + lane * kLdA, hv);
    store_row_bf16(A + lane * kLdA + H, agg);
}

__device__ inline void store_gemm_out(float *C, int lane, const f32x4 acc[4][2]) {
    const int q = lane >> 4, r16 = lane & 15;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int ot = 0; ot < 2; ++ot)
#pragma unroll
            for (int j = 0; j < 4; ++j) C[(16 * t + 4 * q + j) * kLdC + ot * 16 + r16] = acc[t][ot][j];
}

// One wavefront per workgroup: each wave only uses its own LDS tile, so its
// barriers couple no other wave's gather latency.
// channel c (natural order) of a stored row held as its four 16-byte groups
__device__ inline float hraw_channel(const uint4 *raw, int c) {
    const int g = (c & 15) >> 2, t = c & 3;
    const unsigned wd = c < 16 ? (t < 2 ? raw[g].x : raw[g].y) : (t < 2 ? raw[g].z : raw[g].w);
    return __uint_as_float((t & 1) ? (wd & 0xffff0000u) : (wd << 16));
}

// The lane's own stored row (raw, 16 VGPRs) and its aggregated messages
// (FP32, natural order).  With W > 0 (the ELL width) every slot's neighbour
// row is loaded before any is added, so a lane has all its gathers in flight
// at once; padding slots point at the cell itself and get gate 0.  W = 0: a
// loop over the cell's own count.
template <int W>
__device__ inline void gather_rows(int node, bool valid, const GnnEll &E, const bf16_t *__restrict__ h_in,
                                   const bf16_t *__restrict__ lw, uint4 *hraw, float *agg) {
    const float g0 = bf2f(lw[2 * H * H + H]), g1 = bf2f(lw[2 * H * H + H + 1]), g2 = bf2f(lw[2 * H * H + H + 2]);
#pragma unroll
    for (int c = 0; c < H; ++c) agg[c] = 0.f;
#pragma unroll
    for (int v = 0; v < 4; ++v) hraw[v] = make_uint4(0u, 0u, 0u, 0u);
    if (!valid) return;
    const uint4 *own = reinterpret_cast<const uint4 *>(h_in + (size_t)node * H);
#pragma unroll
    for (int v = 0; v < 4; ++v) hraw[v] = own[v];
    const int cnt = E.cnt[node];
    if constexpr (W > 0) {
        int jn[W];
        float cg[W];
#pragma unroll
        for (int k = 0; k < W; ++k) {
            jn[k] = E.nbr[(size_t)k * E.n + node];
            cg[k] = k < cnt ? edge_gate(g0, g1, g2, E.ef[(size_t)k * E.n + node]) : 0.f;
        }
        uint4 raw[W][4];
#pragma unroll
        for (int k = 0; k < W; ++k) {
            const uint4 *p = reinterpret_cast<const uint4 *>(h_in + (size_t)jn[k] * H);
#pragma unroll
            for (int v = 0; v < 4; ++v) raw[k][v] = p[v];
        }
#pragma unroll
        for (int k = 0; k < W; ++k) add_hrow(raw[k], cg[k], agg);
    } else {
        for (int k = 0; k < cnt; ++k) {
            const int j = E.nbr[(size_t)k * E.n + node];
            const float c = edge_gate(g0, g1, g2, E.ef[(size_t)k * E.n + node]);
            uint4 raw[4];
            const uint4 *p = reinterpret_cast<const uint4 *>(h_in + (size_t)j * H);
#pragma unroll
            for (int v = 0; v < 4; ++v) raw[v] = p[v];
            add_hrow(raw, c, agg);
        }
    }
}

// One wavefront per workgroup and one lane per cell: each wave only uses its
// own LDS tile, so its barriers couple no other wave's gather latency.  The
// own row stays in its stored BF16 form (16 VGPRs) from the load to the
// epilogue; its halves go to the LDS tile in the natural channel order.
template <bool LAST, bool STORE, int W>
__global__ __launch_bounds__(64 * kLayerWaves) void k_gnn_layer(int n, GnnEll E, const float *__restrict__ u,
                                                                const bf16_t *__restrict__ h_in,
                                                                bf16_t *__restrict__ h_out, float *__restrict__ z_out,
                                                                const float *__restrict__ s_ptr,
                                                                const bf16_t *__restrict__ w, int layer,
                                                                const Scalars *__restrict__ sc, int xcd,
                                                                const int *__restrict__ order) {
    __shared__ __attribute__((aligned(16))) bf16_t smem[kLayerWaves][64 * kLdA];
    if (sc && sc->done) return;
    // xcd = 1: workgroups are dealt to the 8 XCDs round-robin, so workgroup b takes
    // position (b % 8) * per + b / 8 of the block sequence and each XCD works
    // through one contiguous eighth of it (the grid is a multiple of 8).  The
    // sequence is `order` (blocks by the Morton code of their centroid) or the
    // block index itself; either way the rows that neighbours gather are mostly
    // still in that XCD's own L2.
    static_assert(kLayerWaves == 1, "the block order is over 64-cell blocks");
    const int nblk = (n + 63) / 64;
    const int per = gridDim.x / kXcds;
    const int pos = xcd ? (int)(blockIdx.x % kXcds) * per + (int)(blockIdx.x / kXcds) : (int)blockIdx.x;
    if (pos >= nblk) return;
    const int blk = order ? order[pos] : pos;
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int node = (blk * kLayerWaves + wv) * 64 + lane;
    const bool valid = node < n;
    const bf16_t *lw = w + kGnnOffLayer0 + layer * kGnnLayerStride;
    uint4 hraw[4];
    float agg[H];
    gather_rows<W>(node, valid, E, h_in, lw, hraw, agg);
    bf16_t *A = smem[wv];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        *reinterpret_cast<uint2 *>(A + lane * kLdA + 4 * g) = make_uint2(hraw[g].x, hraw[g].y);
        *reinterpret_cast<uint2 *>(A + lane * kLdA + 16 + 4 * g) = make_uint2(hraw[g].z, hraw[g].w);
    }
    store_row_bf16(A + lane * kLdA + H, agg);
    // loaded after the gathers, so they hold no registers while those are in flight
    bf16x4 bfr[4][2];
    load_b_frags(lw, lane, bfr);
    __syncthreads();
    f32x4 acc[4][2];
    layer_gemm(A, bfr, lane, acc);
    __syncthreads();
    float *C = reinterpret_cast<float *>(A);
    store_gemm_out(C, lane, acc);
    __syncthreads();
    float hn[H];
    const float4 *crow = reinterpret_cast<const float4 *>(C + lane * kLdC);   // 16-byte LDS reads
#pragma unroll
    for (int v = 0; v < H / 4; ++v) {
        const float4 o4 = crow[v];
        const float ov[4] = {o4.x, o4.y, o4.z, o4.w};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int c = 4 * v + t;
            const float out = ov[t] + bf2f(lw[2 * H * H + c]);
            hn[c] = hraw_channel(hraw, c) + fmaxf(out, 0.f);   // rounded to BF16 below
        }
    }
    if (!valid) return;
    if (!LAST || STORE) store_hrow(h_out + (size_t)node * H, hn);
    if (LAST) {
        float y = bf2f(w[kGnnOffDecB]);
#pragma unroll
        for (int c = 0; c < H; ++c) y = fmaf(bf2f(w[kGnnOffDecW + c]), bfround(hn[c]), y);
        z_out[node] = s_ptr[0] * (u[node] + y);
    }
}

// The layer with the rows gathered by quads of lanes, for ELL widths 4, 6 and 8.
// A lane's 16-byte load of a scattered row costs the texture path as much as a
// 64-byte one, so with one lane per cell the four loads per row keep that path
// busy.  Here lane l = 4 m + g loads 16-byte group g of a row, so four adjacent
// lanes read one row's 64 contiguous bytes and a load instruction covers 16
// whole rows.  The block's 64 cells are four sub-tiles of 16 (cell 16 i + m);
// the neighbour indices and gates are loaded one lane per cell and handed to
// the quads with cross-lane shuffles.  Persistent waves walk the block
// sequence with a stride of `waves` (the waves per XCD), so the blocks in
// flight on an XCD stay consecutive in the sequence, and the next block's
// neighbour indices, features and count are loaded before the current block's
// gathers are waited for.  Aggregation, the LDS tile, the MFMA GEMM and the
// epilogue give the values of k_gnn_layer (the decoder sums its 32 products
// in another order).
template <int W>
struct QuadIdx {
    int cnt;
    int jn[W];
    uint32_t ef[W];
};

template <int W>
__device__ inline void load_quad_idx(const GnnEll &E, int node_c, QuadIdx<W> &b) {
    b.cnt = E.cnt[node_c];
#pragma unroll
    for (int k = 0; k < W; ++k) {
        b.jn[k] = E.nbr[(size_t)k * E.n + node_c];
        b.ef[k] = E.ef[(size_t)k * E.n + node_c];
    }
}

// agg8 (the 8 channels of group g, local order) += c1 row1 + c2 row2 (one 16-byte group each)
__device__ inline void add_group_pair(uint4 r1, uint4 r2, unsigned cpair, float *agg8) {
    const bf16x2_t cp = __builtin_bit_cast(bf16x2_t, cpair);
    const unsigned a[4] = {r1.x, r1.y, r1.z, r1.w};
    const unsigned b[4] = {r2.x, r2.y, r2.z, r2.w};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const unsigned lo = __builtin_amdgcn_perm(b[t], a[t], 0x05040100u);
        const unsigned hi = __builtin_amdgcn_perm(b[t], a[t], 0x07060302u);
        agg8[2 * t] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, lo), cp, agg8[2 * t], false);
        agg8[2 * t + 1] =
            __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, hi), cp, agg8[2 * t + 1], false);
    }
}

// group g of the encoder row of a cell with input v: the BF16 values k_gnn_input stores
__device__ inline uint4 enc_group(float v, const float *wenc, const float *benc) {
    float hv[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) hv[t] = fmaxf(wenc[t] * v + benc[t], 0.f);
    return pack8(hv);
}

// FIRST: the input rows are the encoder rows, computed from u of the cell and of
// its neighbours instead of being read (4 bytes gathered per row instead of 64)
template <bool LAST, bool STORE, int W, bool FIRST = false>
__global__ __launch_bounds__(64, 2) void k_gnn_layer_quad(int n, GnnEll E, const float *__restrict__ u,
                                                       const bf16_t *__restrict__ h_in, bf16_t *__restrict__ h_out,
                                                       float *__restrict__ z_out, const float *__restrict__ s_ptr,
                                                       const bf16_t *__restrict__ w, int layer,
                                                       const Scalars *__restrict__ sc, int waves,
                                                       const int *__restrict__ order) {
    static_assert(W > 0 && W <= 8 && W % 2 == 0, "compiled ELL width, rows added in pairs");
    __shared__ __attribute__((aligned(16))) bf16_t smem[64 * kLdA];
    if (sc && sc->done) return;
    const int nblk = (n + 63) / 64;
    const int per = (nblk + kXcds - 1) / kXcds;
    const int x = (int)(blockIdx.x % kXcds), lw_idx = (int)(blockIdx.x / kXcds);
    const int end = min(nblk, (x + 1) * per);
    int pos = x * per + lw_idx;
    if (pos >= end) return;
    const int lane = threadIdx.x;
    const int m = lane >> 2, g = lane & 3;
    const bf16_t *lw = w + kGnnOffLayer0 + layer * kGnnLayerStride;
    const float g0 = bf2f(lw[2 * H * H + H]), g1 = bf2f(lw[2 * H * H + H + 1]), g2 = bf2f(lw[2 * H * H + H + 2]);
    // bias and decoder weights of the lane's 8 channels (group g, local order), and
    // the encoder's weights and biases of the same channels for FIRST
    float bias[8], wdec[8], wenc[8], benc[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        bias[t] = bf2f(lw[2 * H * H + hrow_channel(g, t)]);
        wdec[t] = LAST ? bf2f(w[kGnnOffDecW + hrow_channel(g, t)]) : 0.f;
        wenc[t] = FIRST ? bf2f(w[kGnnOffEncW + hrow_channel(g, t)]) : 0.f;
        benc[t] = FIRST ? bf2f(w[kGnnOffEncB + hrow_channel(g, t)]) : 0.f;
    }
    int blk = order ? order[pos] : pos;
    QuadIdx<W> cur;
    load_quad_idx<W>(E, min(blk * 64 + lane, n - 1), cur);
    for (;;) {
        const int base = blk * 64;
        // gate pairs of the lane's own cell (lane = cell in this phase)
        const bool lvalid = base + lane < n;
        unsigned cp[W / 2];
#pragma unroll
        for (int q = 0; q < W / 2; ++q) {
            const float c1 = lvalid && 2 * q < cur.cnt ? edge_gate(g0, g1, g2, cur.ef[2 * q]) : 0.f;
            const float c2 = lvalid && 2 * q + 1 < cur.cnt ? edge_gate(g0, g1, g2, cur.ef[2 * q + 1]) : 0.f;
            cp[q] = f2bf2(c1, c2);
        }
        // gathers: sub-tile i, slot k -> group g of the row of neighbour k of cell 16 i + m
        uint4 own[4];
        uint4 raw[4][W];
        float uq[4];        // u of the sub-tiles' cells (last layer, FIRST), loaded with the rows
        float un[4][W];     // u of the neighbours (FIRST)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int src = 16 * i + m;
            if (!FIRST) own[i] = reinterpret_cast<const uint4 *>(h_in + (size_t)min(base + src, n - 1) * H)[g];
            uq[i] = LAST || FIRST ? u[min(base + src, n - 1)] : 0.f;
#pragma unroll
            for (int k = 0; k < W; ++k) {
                const int j = __shfl(cur.jn[k], src, 64);
                if (FIRST)
                    un[i][k] = u[j];
                else
                    raw[i][k] = reinterpret_cast<const uint4 *>(h_in + (size_t)j * H)[g];
            }
        }
        // the next block's indices (this block's again on the last trip)
        const int npos = pos + waves;
        const bool more = npos < end;
        const int nb = more ? (order ? order[npos] : npos) : blk;
        QuadIdx<W> nxt;
        load_quad_idx<W>(E, min(nb * 64 + lane, n - 1), nxt);
        if (FIRST) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                own[i] = enc_group(uq[i], wenc, benc);
#pragma unroll
                for (int k = 0; k < W; ++k) raw[i][k] = enc_group(un[i][k], wenc, benc);
            }
        }
        // messages, and [h | agg] of each cell into the LDS tile (natural channel order)
        bf16_t *A = smem;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int src = 16 * i + m;
            float agg[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) agg[t] = 0.f;
#pragma unroll
            for (int q = 0; q < W / 2; ++q)
                add_group_pair(raw[i][2 * q], raw[i][2 * q + 1], (unsigned)__shfl((int)cp[q], src, 64), agg);
            bf16_t *row = A + src * kLdA;
            *reinterpret_cast<uint2 *>(row + 4 * g) = make_uint2(own[i].x, own[i].y);
            *reinterpret_cast<uint2 *>(row + 16 + 4 * g) = make_uint2(own[i].z, own[i].w);
            *reinterpret_cast<uint2 *>(row + H + 4 * g) = make_uint2(f2bf2(agg[0], agg[1]), f2bf2(agg[2], agg[3]));
            *reinterpret_cast<uint2 *>(row + H + 16 + 4 * g) =
                make_uint2(f2bf2(agg[4], agg[5]), f2bf2(agg[6], agg[7]));
        }
        bf16x4 bfr[4][2];
        load_b_frags(lw, lane, bfr);
        __syncthreads();
        f32x4 acc[4][2];
        layer_gemm(A, bfr, lane, acc);
        __syncthreads();
        float *C = reinterpret_cast<float *>(A);
        store_gemm_out(C, lane, acc);
        __syncthreads();
        // epilogue in the quad layout: channels of group g of cell 16 i + m
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int rowi = 16 * i + m;
            const int node = base + rowi;
            const float4 o0 = *reinterpret_cast<const float4 *>(C + rowi * kLdC + 4 * g);
            const float4 o1 = *reinterpret_cast<const float4 *>(C + rowi * kLdC + 16 + 4 * g);
            const float ov[8] = {o0.x, o0.y, o0.z, o0.w, o1.x, o1.y, o1.z, o1.w};
            float hv[8], hn[8];
            unpack8(own[i], hv);
#pragma unroll
            for (int t = 0; t < 8; ++t) hn[t] = hv[t] + fmaxf(ov[t] + bias[t], 0.f);   // rounded to BF16 below
            if (!LAST || STORE) {
                if (node < n) reinterpret_cast<uint4 *>(h_out + (size_t)node * H)[g] = pack8(hn);
            }
            if (LAST) {
                float y = 0.f;
#pragma unroll
                for (int t = 0; t < 8; ++t) y = fmaf(wdec[t], bfround(hn[t]), y);
                y += __shfl_xor(y, 1, 64);
                y += __shfl_xor(y, 2, 64);
                if (node < n && g == 0) z_out[node] = s_ptr[0] * (uq[i] + (bf2f(w[kGnnOffDecB]) + y));
            }
        }
        // the C tile is read: the next trip may overwrite the LDS tile
        __syncthreads();
        if (!more) break;
        pos = npos;
        blk = nb;
        cur = nxt;
    }
}

// ---------------------------------------------------- cluster layout

// Set-up of the cluster layout (GnnGraph::cperm ...).  Per axis, the cells
// sorted by centroid coordinate give each cell its rank; the Morton code of the
// three ranks (21 bits each) then orders the cells.  Ranks instead of
// coordinates make the order follow the cell counts along each axis, so a
// graded mesh gets bricks of cells, not bricks of space.

// order-preserving 64-bit key of a double, and the cell index as the value
__global__ void k_cl_axis_keys(int n, const double *__restrict__ x, unsigned long long *__restrict__ key,
                               int *__restrict__ idx) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const unsigned long long b = (unsigned long long)__double_as_longlong(x[i]);
        key[i] = (b >> 63) ? ~b : (b | (1ull << 63));
        idx[i] = i;
    }
}

__global__ void k_cl_rank(int n, const int *__restrict__ sorted_idx, int *__restrict__ rank) {
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) rank[sorted_idx[p]] = p;
}

__global__ void k_cl_morton(int n, const int *__restrict__ rx, const int *__restrict__ ry, const int *__restrict__ rz,
                            unsigned long long *__restrict__ key, int *__restrict__ idx) {
    const unsigned long long top = (1ull << 21) - 1;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const unsigned long long qx = (unsigned long long)rx[i] * top / (unsigned long long)n;
        const unsigned long long qy = (unsigned long long)ry[i] * top / (unsigned long long)n;
        const unsigned long long qz = (unsigned long long)rz[i] * top / (unsigned long long)n;
        key[i] = (spread3(qx) << 2) | (spread3(qy) << 1) | spread3(qz);
        idx[i] = i;
    }
}

// cinv[cell] = position; cperm past n is -1
__global__ void k_cl_inverse(int n, int n_pad, int *__restrict__ cperm, int *__restrict__ cinv) {
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n_pad; p += gridDim.x * blockDim.x) {
        if (p < n) cinv[cperm[p]] = p;
        else cperm[p] = -1;
    }
}

// One workgroup per cluster: the distinct outside neighbours of its cells (the
// halo, sorted by position), and for every ELL slot the LDS row it reads --
// p - base for a cell of the cluster, kGnnClCells + (halo rank) outside, 0xffff
// for a padding slot -- as 16-bit pairs.  The candidates are sorted in LDS
// (bitonic, padded to a power of two with INT_MAX) and the first of each run
// counted; *hmax becomes the largest halo (above kGnnClHalo the layer kernel is
// not used for the graph).
template <int W>
__global__ __launch_bounds__(kGnnClCells) void k_cl_halo(int n, int n_pad, const int *__restrict__ cperm,
                                                        const int *__restrict__ cinv, const int *__restrict__ ecnt,
                                                        const int *__restrict__ enbr, int *__restrict__ hcnt,
                                                        int *__restrict__ halo, uint32_t *__restrict__ lidx,
                                                        int *__restrict__ hmax) {
    constexpr int SZ = kGnnClCells * W <= 1024 ? 1024 : 2048;
    constexpr int PER = SZ / kGnnClCells;
    static_assert(kGnnClCells * W <= SZ, "candidate array");
    __shared__ int cand[SZ];
    __shared__ int wpart[kGnnClCells / 64];
    const int c = blockIdx.x, t = threadIdx.x, base = c * kGnnClCells, pos = base + t;
    const int cell = pos < n ? cperm[pos] : -1;
    const int cnt = cell >= 0 ? ecnt[cell] : 0;
    int pj[W];
#pragma unroll
    for (int k = 0; k < W; ++k) {
        pj[k] = k < cnt ? cinv[enbr[(size_t)k * n + cell]] : -1;
        const bool out = k < cnt && (pj[k] < base || pj[k] >= base + kGnnClCells);
        cand[t * W + k] = out ? pj[k] : INT_MAX;
    }
    for (int i = kGnnClCells * W + t; i < SZ; i += kGnnClCells) cand[i] = INT_MAX;
    __syncthreads();
    for (int k = 2; k <= SZ; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int i = t; i < SZ; i += kGnnClCells) {
                const int ixj = i ^ j;
                if (ixj > i) {
                    const int a = cand[i], b = cand[ixj];
                    if ((a > b) == ((i & k) == 0)) {
                        cand[i] = b;
                        cand[ixj] = a;
                    }
                }
            }
            __syncthreads();
        }
    // first of each run: thread t owns candidates t*PER .. t*PER + PER - 1
    int flags = 0, mine = 0;
#pragma unroll
    for (int e = 0; e < PER; ++e) {
        const int i = t * PER + e;
        const int v = cand[i];
        if (v != INT_MAX && (i == 0 || cand[i - 1] != v)) {
            flags |= 1 << e;
            ++mine;
        }
    }
    // exclusive prefix of the counts over the workgroup
    const int lane = t & 63, wv = t >> 6;
    int incl = mine;
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(incl, o, 64);
        if (lane >= o) incl += y;
    }
    if (lane == 63) wpart[wv] = incl;
    __syncthreads();
    int off = incl - mine, total = 0;
    for (int w2 = 0; w2 < kGnnClCells / 64; ++w2) {
        if (w2 < wv) off += wpart[w2];
        total += wpart[w2];
    }
    int uv[PER];
#pragma unroll
    for (int e = 0; e < PER; ++e) uv[e] = cand[t * PER + e];
    __syncthreads();
    // the distinct values, in order, back into cand[0 .. total) (and the halo list)
#pragma unroll
    for (int e = 0; e < PER; ++e)
        if ((flags >> e) & 1) {
            cand[off] = uv[e];
            if (off < kGnnClHalo) halo[(size_t)c * kGnnClHalo + off] = uv[e];
            ++off;
        }
    if (t == 0) {
        hcnt[c] = total;
        atomicMax(hmax, total);
    }
    __syncthreads();
    unsigned short li[W];
#pragma unroll
    for (int k = 0; k < W; ++k) {
        if (k >= cnt) {
            li[k] = 0xffff;
        } else if (pj[k] >= base && pj[k] < base + kGnnClCells) {
            li[k] = (unsigned short)(pj[k] - base);
        } else {
            int lo = 0, hi = total - 1;   // binary search in the sorted distinct list
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (cand[mid] < pj[k]) lo = mid + 1;
                else hi = mid;
            }
            li[k] = (unsigned short)(kGnnClCells + min(lo, kGnnClHalo - 1));
        }
    }
#pragma unroll
    for (int q = 0; q < W / 2; ++q) lidx[(size_t)q * n_pad + pos] = (uint32_t)li[2 * q] | ((uint32_t)li[2 * q + 1] << 16);
}

// The edge features of the ELL slots in position order (every assembly).
__global__ void k_cl_feats(int n, int n_pad, int w, const int *__restrict__ cperm, const uint32_t *__restrict__ eef,
                           uint32_t *__restrict__ efc) {
    const long long total = (long long)w * n_pad;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total;
         i += (long long)gridDim.x * blockDim.x) {
        const int k = (int)(i / n_pad), p = (int)(i - (long long)k * n_pad);
        efc[i] = p < n ? eef[(size_t)k * n + cperm[p]] : 0u;
    }
}

// u = (r / a_ii) / s in position order (the values k_gnn_u computes): read in cell
// order, written to each cell's position (the positions of nearby cells are nearby)
__global__ __launch_bounds__(256) void k_gnn_u_cl(int n, const int *__restrict__ cinv, const float *__restrict__ r,
                                                  const float *__restrict__ dg, const float *__restrict__ s,
                                                  float *__restrict__ u, const Scalars *__restrict__ sc) {
    if (sc && sc->done) return;
    const float sv = s[0];
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        u[cinv[i]] = (r[i] / dg[i]) / sv;
}

// Gate pairs of every layer in the cluster layout, for the weights of one
// network: for layer l, slot pair q and position p, {the two slots' LDS rows (a
// padding slot reads the cell's own row), their two BF16 gates (0 for a padding
// slot)} at [(l * W/2 + q) * n_pad + p] -- the values the quad kernel forms in
// every launch.  Rebuilt when the weights or the features change.
__global__ void k_cl_gates(int n_pad, int w, const uint32_t *__restrict__ lidx, const uint32_t *__restrict__ efc,
                           const bf16_t *__restrict__ wts, uint2 *__restrict__ out) {
    const int halfw = w / 2;
    const long long total = (long long)kGnnL * halfw * n_pad;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total;
         i += (long long)gridDim.x * blockDim.x) {
        const int lq = (int)(i / n_pad), p = (int)(i - (long long)lq * n_pad);
        const int q = lq % halfw, l = lq / halfw;
        const bf16_t *lw = wts + kGnnOffLayer0 + l * kGnnLayerStride;
        const float g0 = bf2f(lw[2 * H * H + H]), g1 = bf2f(lw[2 * H * H + H + 1]), g2 = bf2f(lw[2 * H * H + H + 2]);
        const uint32_t lp = lidx[(size_t)q * n_pad + p];
        const unsigned l1 = lp & 0xffffu, l2 = lp >> 16, own = (unsigned)(p % kGnnClCells);
        const float c1 = l1 != 0xffffu ? edge_gate(g0, g1, g2, efc[(size_t)(2 * q) * n_pad + p]) : 0.f;
        const float c2 = l2 != 0xffffu ? edge_gate(g0, g1, g2, efc[(size_t)(2 * q + 1) * n_pad + p]) : 0.f;
        out[i] = make_uint2((l1 != 0xffffu ? l1 : own) | ((l2 != 0xffffu ? l2 : own) << 16), f2bf2(c1, c2));
    }
}

// Workgroup barrier that orders LDS only: global loads and stores in flight stay
// in flight across it (__syncthreads would wait for all of them)
__device__ inline void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// LDS slot of 16-byte group g of row r: the groups of a row rotate with r / 4,
// so that rows read together spread over the banks
__device__ inline int cl_slot(int r, int g) { return 4 * r + (g ^ ((r >> 2) & 3)); }

// Per-cluster inputs of the layer kernel, loaded one cluster ahead: the halo
// positions (two clusters ahead: the halo rows' loads need them), the gate pairs
// of the quad layout's cells and (LAST) u and cell of the MFMA layout's cells,
// and the rows themselves (FIRST: u of the cluster's cells and of its halo).
template <int HJ>
struct ClHalo {
    int nh;
    int hp[HJ];
};
template <int W>
struct ClMeta {
    uint2 gp[4][W / 2];
    float uz[4];
    int cz[4];
};
template <int HJ, bool FIRST>
struct ClRows {
    uint4 own[4];    // !FIRST: group qq of rows 16 t + r16 of the wave
    uint4 hr[HJ];    // !FIRST: group qq of halo rows 64 j + 16 wv + r16
    float uo[4];     // FIRST: u of the same cells
    float uh[HJ];
};

template <int HJ>
__device__ inline ClHalo<HJ> cl_load_halo(const int *__restrict__ hcnt, const int *__restrict__ halo, int c, int wv,
                                          int r16) {
    // every load unconditional (entries past the count hold 0, a valid position), so
    // that they are all in flight together
    ClHalo<HJ> h;
    h.nh = min(hcnt[c], kGnnClHalo);
#pragma unroll
    for (int j = 0; j < HJ; ++j) h.hp[j] = halo[(size_t)c * kGnnClHalo + min(64 * j + 16 * wv + r16, kGnnClHalo - 1)];
    return h;
}

template <int W, bool LAST>
__device__ inline ClMeta<W> cl_load_meta(const uint2 *__restrict__ lg, const int *__restrict__ cperm,
                                         const float *__restrict__ u, int n, int n_pad, int base, int wv, int m,
                                         int r16) {
    ClMeta<W> mt;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int q = 0; q < W / 2; ++q) mt.gp[i][q] = lg[(size_t)q * n_pad + base + wv * 64 + 16 * i + m];
    if constexpr (LAST) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int p = min(base + wv * 64 + 16 * t + r16, n - 1);
            mt.uz[t] = u[p];
            mt.cz[t] = cperm[p];
        }
    }
    return mt;
}

template <int HJ, bool FIRST>
__device__ inline ClRows<HJ, FIRST> cl_load_rows(const ClHalo<HJ> &h, const float *__restrict__ u,
                                                 const bf16_t *__restrict__ h_in, int n, int base, int wv, int qq,
                                                 int r16) {
    // unconditional loads (a branch around a load makes the compiler wait for every
    // load in flight); the cluster's cells past n take the row of cell n - 1, which only
    // they read (their slots are padding) and which is never stored for them
    ClRows<HJ, FIRST> r;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int pc = min(base + wv * 64 + 16 * t + r16, n - 1);
        if constexpr (FIRST) r.uo[t] = u[pc];
        else r.own[t] = reinterpret_cast<const uint4 *>(h_in + (size_t)pc * H)[qq];
    }
#pragma unroll
    for (int j = 0; j < HJ; ++j) {
        if constexpr (FIRST) r.uh[j] = u[h.hp[j]];
        else r.hr[j] = reinterpret_cast<const uint4 *>(h_in + (size_t)h.hp[j] * H)[qq];
    }
    return r;
}

// The rows into LDS (FIRST: encoded from u); returns the lane's own groups.
template <int HJ, bool FIRST>
__device__ inline void cl_store_rows(uint4 *rows, const ClRows<HJ, FIRST> &r, int nh, const float *wenc,
                                     const float *benc, int wv, int qq, int r16, uint4 *own) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        own[t] = FIRST ? enc_group(r.uo[t], wenc, benc) : r.own[t];
        rows[cl_slot(wv * 64 + 16 * t + r16, qq)] = own[t];
    }
#pragma unroll
    for (int j = 0; j < HJ; ++j) {
        const int hr = 64 * j + 16 * wv + r16;
        if (hr < nh) rows[cl_slot(kGnnClCells + hr, qq)] = FIRST ? enc_group(r.uh[j], wenc, benc) : r.hr[j];
    }
}

// The inference layer over clusters (ELL widths 4, 6, 8), on rows in position
// order.  Persistent workgroups of four waves; XCD x walks the x-th eighth of
// the clusters (compact in the Morton order) with a stride of its workgroups.
// Wave v owns a cluster's cells 64 v .. 64 v + 63 as four sub-tiles of 16.  Per
// cluster:
//  1. lane r + 16 q holds group q of its wave's rows 16 t + r (t = 0..3) in
//     registers -- the layout of the MFMA operand and of the epilogue -- and
//     writes them to LDS; the halo rows follow, 64 contiguous bytes a row
//     (FIRST: the encoder rows computed from u of the cluster and of the halo);
//  2. lane 4 m + g adds the messages of cell 16 i + m, group g, reading every
//     neighbour row from LDS (four lanes read one row's 64 bytes; slot pairs
//     through v_dot2 as in the quad kernel, with the gate pairs of k_cl_gates);
//     the sums move to the MFMA layout with cross-lane permutes;
//  3. [h | agg] times [Ws ; Wm] on MFMA, the weights the A operand and the
//     cells' features the B operand, straight from registers: a lane ends with
//     one 16-byte output group of a cell;
//  4. epilogue: h + relu(out + b), 16 bytes per lane (LAST: the decoder, z
//     scattered back to cell order).
// The next cluster's rows, gates and halo positions are loaded into registers
// before step 2 (its halo positions one cluster earlier), so their latency
// hides behind this cluster's work.  Each value is formed with the same
// operations in the same order as k_gnn_layer_quad, so the rows and z are
// bitwise those of the cell-order path.
template <int W, bool FIRST, bool LAST>
__global__ __launch_bounds__(kGnnClCells, 2) void k_gnn_layer_cl(int n, int ncl, int wg_per_xcd,
                                                                const int *__restrict__ hcnt,
                                                                const int *__restrict__ halo,
                                                                const uint2 *__restrict__ gates,
                                                                const int *__restrict__ cperm,
                                                                const float *__restrict__ u,
                                                                const bf16_t *__restrict__ h_in,
                                                                bf16_t *__restrict__ h_out, float *__restrict__ z_out,
                                                                const float *__restrict__ s_ptr,
                                                                const bf16_t *__restrict__ w, int layer,
                                                                const Scalars *__restrict__ sc) {
    static_assert(W == 4 || W == 6 || W == 8, "compiled ELL widths");
    constexpr int ROWS = kGnnClCells + kGnnClHalo;
    constexpr int HJ = (kGnnClHalo + 63) / 64;   // halo rows per lane, at most
    __shared__ uint4 rows[ROWS * 4];
    if (sc && sc->done) return;
    const int per = (ncl + kXcds - 1) / kXcds;
    const int x = (int)(blockIdx.x % kXcds);
    const int cend = min(ncl, (x + 1) * per);
    int c = x * per + (int)(blockIdx.x / kXcds);
    if (c >= cend) return;
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
    const int n_pad = ncl * kGnnClCells;
    const int qq = lane >> 4, r16 = lane & 15;   // MFMA layout: cell 16 t + r16 of the wave, group qq
    const int m = lane >> 2, g = lane & 3;       // quad layout: cell 16 i + m of the wave, group g
    const bf16_t *lw = w + kGnnOffLayer0 + layer * kGnnLayerStride;
    const uint2 *lg = gates + (size_t)layer * (W / 2) * n_pad;

    // weights: MFMA A fragments, bias and decoder of group qq, encoder of group qq (FIRST)
    bf16x4 afr[4][2];
    load_b_frags(lw, lane, afr);
    float bias[8], wdec[8], wenc[8], benc[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        bias[t] = bf2f(lw[2 * H * H + hrow_channel(qq, t)]);
        wdec[t] = LAST ? bf2f(w[kGnnOffDecW + hrow_channel(qq, t)]) : 0.f;
        wenc[t] = FIRST ? bf2f(w[kGnnOffEncW + hrow_channel(qq, t)]) : 0.f;
        benc[t] = FIRST ? bf2f(w[kGnnOffEncB + hrow_channel(qq, t)]) : 0.f;
    }
    const float sv = LAST ? s_ptr[0] : 0.f;
    const float bdec = LAST ? bf2f(w[kGnnOffDecB]) : 0.f;

    // the first cluster, and the halo positions of the second
    uint4 own[4];
    ClMeta<W> mt = cl_load_meta<W, LAST>(lg, cperm, u, n, n_pad, c * kGnnClCells, wv, m, r16);
    {
        const ClHalo<HJ> h0 = cl_load_halo<HJ>(hcnt, halo, c, wv, r16);
        const ClRows<HJ, FIRST> r0 = cl_load_rows<HJ, FIRST>(h0, u, h_in, n, c * kGnnClCells, wv, qq, r16);
        cl_store_rows<HJ, FIRST>(rows, r0, h0.nh, wenc, benc, wv, qq, r16, own);
    }
    int c1 = c + wg_per_xcd;
    ClHalo<HJ> h1 = cl_load_halo<HJ>(hcnt, halo, min(c1, cend - 1), wv, r16);
    lds_barrier();

    for (;;) {
        const int base = c * kGnnClCells;
        const bool more = c1 < cend;
        const int cn = more ? c1 : c;   // a last trip loads its own cluster again (in bounds, unused)
        // next cluster's inputs in flight while this one is computed
        const ClRows<HJ, FIRST> rn = cl_load_rows<HJ, FIRST>(h1, u, h_in, n, cn * kGnnClCells, wv, qq, r16);
        const ClMeta<W> mn = cl_load_meta<W, LAST>(lg, cperm, u, n, n_pad, cn * kGnnClCells, wv, m, r16);
        const int c2 = c1 + wg_per_xcd;
        const ClHalo<HJ> h2 = cl_load_halo<HJ>(hcnt, halo, min(c2, cend - 1), wv, r16);

        // 2. messages (quad layout), then to the MFMA layout: lane r16 + 16 qq takes
        // cell 16 t + r16, group qq from quad lane 4 r16 + qq
        uint4 aggm[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float agg[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) agg[t] = 0.f;
#pragma unroll
            for (int q = 0; q < W / 2; ++q) {
                const unsigned l = mt.gp[i][q].x;
                add_group_pair(rows[cl_slot((int)(l & 0xffffu), g)], rows[cl_slot((int)(l >> 16), g)],
                               mt.gp[i][q].y, agg);
            }
            const uint4 pk = pack8(agg);
            const int src = 4 * r16 + qq;
            aggm[i] = make_uint4((unsigned)__shfl((int)pk.x, src, 64), (unsigned)__shfl((int)pk.y, src, 64),
                                 (unsigned)__shfl((int)pk.z, src, 64), (unsigned)__shfl((int)pk.w, src, 64));
        }

        // 3. out^T(32 x 64 cells) = [Ws | Wm](32 x 64) [h | agg]^T on MFMA: A = the weights
        // (rows o = 16 ot + lane % 16, k = 16 kk + 4 (lane / 16) .. + 3), B = the cells'
        // features (column cell 16 t + lane % 16, the same four k: half kk % 2 of group qq)
        // 4. epilogue: lane (r16, qq) holds outputs 4 qq + v (tile 0) and 16 + 4 qq + v
        // (tile 1) of cell 16 t + r16 -- stored group qq of the cell's new row
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            f32x4 acc[2];
#pragma unroll
            for (int ot = 0; ot < 2; ++ot) acc[ot] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const uint4 gv = kk < 2 ? own[t] : aggm[t];
                const uint2 hv = (kk & 1) ? make_uint2(gv.z, gv.w) : make_uint2(gv.x, gv.y);
                const bf16x4 bfr = __builtin_bit_cast(bf16x4, hv);
#pragma unroll
                for (int ot = 0; ot < 2; ++ot)
                    acc[ot] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(afr[kk][ot], bfr, acc[ot], 0, 0, 0);
            }
            const int p = base + wv * 64 + 16 * t + r16;
            float hv[8], hn[8];
            unpack8(own[t], hv);
            const float ov[8] = {acc[0][0], acc[0][1], acc[0][2], acc[0][3], acc[1][0], acc[1][1], acc[1][2], acc[1][3]};
#pragma unroll
            for (int k = 0; k < 8; ++k) hn[k] = hv[k] + fmaxf(ov[k] + bias[k], 0.f);
            if constexpr (!LAST) {
                if (p < n) reinterpret_cast<uint4 *>(h_out + (size_t)p * H)[qq] = pack8(hn);
            } else {
                float y = 0.f;
#pragma unroll
                for (int k = 0; k < 8; ++k) y = fmaf(wdec[k], bfround(hn[k]), y);
                y += __shfl_xor(y, 16, 64);
                y += __shfl_xor(y, 32, 64);
                if (p < n && qq == 0) z_out[mt.cz[t]] = sv * (mt.uz[t] + (bdec + y));
            }
        }
        if (!more) break;
        // every wave is done with this cluster's LDS rows: the next cluster's go in
        lds_barrier();
        cl_store_rows<HJ, FIRST>(rows, rn, h1.nh, wenc, benc, wv, qq, r16, own);
        mt = mn;
        h1 = h2;
        c = c1;
        c1 = c2;
        lds_barrier();
    }
}

// ------------------------------------------------------------- backward

// dz = coef * q (coef = 2 / (e^T A e * batch)); d = z - e
__global__ void k_gnn_diff(int n, const float *__restrict__ z, const float *__restrict__ e, float *__restrict__ d) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) d[i] = z[i] - e[i];
}

__global__ void k_gnn_scale(int n, const float *__restrict__ q, float coef, float *__restrict__ dz) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) dz[i] = coef * q[i];
}

// y = x / d (div) or y = x * d
template <bool DIV>
__global__ void k_gnn_diag(int n, const float *__restrict__ x, const float *__restrict__ d, float *__restrict__ y) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        y[i] = DIV ? x[i] / d[i] : x[i] * d[i];
}

// Block sums of N values a thread (256 threads), column c's in FP64 to put(c, sum) by one
// thread each: 32 columns at a time go through an LDS tile whose columns four threads sum a
// quarter of each, so the block has two barriers per 32 columns (a block_sum per column had
// three per column and took most of the first layer's and the decoder's time).
constexpr int kColTile = 32, kColPad = 257;
template <int N, class Put>
__device__ inline void block_columns(const float *v, float *tile, Put &&put) {
    const int t = threadIdx.x;
#pragma unroll
    for (int c0 = 0; c0 < N; c0 += kColTile) {
        __syncthreads();
#pragma unroll
        for (int c = 0; c < kColTile; ++c)
            if (c0 + c < N) tile[c * kColPad + t] = v[c0 + c];
        __syncthreads();
        double s = 0.0;
        const int c = (t >> 2) & (kColTile - 1), part = t & 3;
        if (t < 4 * kColTile && c0 + c < N)
            for (int k = 0; k < 64; ++k) s += (double)tile[c * kColPad + 4 * k + part];
        s += __shfl_down(s, 2, 4);
        s += __shfl_down(s, 1, 4);
        if (t < 4 * kColTile && part == 0 && c0 + c < N) put(c0 + c, s);
    }
}

// decoder: dy = s dz ; dh4 = dy w_dec ; partials of d w_dec (32) and d b_dec (1) per block
__global__ __launch_bounds__(256) void k_gnn_dec_bwd(int n, const bf16_t *__restrict__ h4, const float *__restrict__ dz,
                                                     const float *__restrict__ s_ptr, const bf16_t *__restrict__ w,
                                                     float *__restrict__ dh, float *__restrict__ part) {
    __shared__ float tile[kColTile * kColPad];
    const float sv = s_ptr[0];
    float acc[H + 1];
#pragma unroll
    for (int c = 0; c <= H; ++c) acc[c] = 0.f;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        const float dy = sv * dz[i];
        float hv[H];
        load_hrow(h4 + (size_t)i * H, hv);
#pragma unroll
        for (int c = 0; c < H; ++c) {
            dh[(size_t)i * H + c] = dy * bf2f(w[kGnnOffDecW + c]);
            acc[c] += dy * hv[c];
        }
        acc[H] += dy;
    }
    block_columns<H + 1>(acc, tile, [&](int c, double v) { part[(size_t)blockIdx.x * (H + 1) + c] = (float)v; });
}

// Layer backward, part 1 (one wave per 64 cells, chunks strided over the grid):
// recompute [h | agg] and out, d_out = dh_out * (out > 0),
// [d_self | d_agg] = d_out * [Ws | Wm] (MFMA), dh_part = dh_out + d_self,
// per-wave partials of dWs, dWm (d_out^T [h | agg], MFMA over cells) and db.
template <bool FIRST>
__global__ __launch_bounds__(256) void k_gnn_bwd1(int n, GnnEll E, const float *__restrict__ u,
                                                  const bf16_t *__restrict__ h_in, const float *__restrict__ dh_out,
                                                  const bf16_t *__restrict__ w, int layer, float *__restrict__ dh_part,
                                                  float *__restrict__ dagg, float *__restrict__ wpart) {
    __shared__ __attribute__((aligned(16))) bf16_t smx[kWaves][64 * kLdA];
    __shared__ __attribute__((aligned(16))) bf16_t smd[kWaves][64 * kLdD];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int q = lane >> 4, r16 = lane & 15;
    const bf16_t *lw = w + kGnnOffLayer0 + layer * kGnnLayerStride;
    f32x4 gacc[2][4];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) gacc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float dbacc[H];
#pragma unroll
    for (int c = 0; c < H; ++c) dbacc[c] = 0.f;
    const int nchunks = (n + 255) / 256;
    for (int chunk = blockIdx.x; chunk < nchunks; chunk += gridDim.x) {
        const int node = chunk * 256 + wv * 64 + lane;
        const bool valid = node < n;
        float hv[H], agg[H];
        gather_features<FIRST>(node, valid, E, u, h_in, w, lw, hv, agg);
        bf16_t *X = smx[wv];
        bf16_t *D = smd[wv];
        stage_row(X, lane, hv, agg);
        __syncthreads();
        f32x4 acc[4][2];
        bf16x4 bfr[4][2];
        load_b_frags(lw, lane, bfr);
        layer_gemm(X, bfr, lane, acc);
        __syncthreads();
        // d_out needs out of the lane's own cell: stage out in the D tile region as FP32? D is
        // 64 x 40 bf16 = 5120 bytes < 64 x 32 floats; so stage out in X temporarily (X is
        // re-written from registers afterwards).
        float *C = reinterpret_cast<float *>(X);
        store_gemm_out(C, lane, acc);
        __syncthreads();
        float dout[H];
#pragma unroll
        for (int c = 0; c < H; ++c) {
            const float out = C[lane * kLdC + c] + bf2f(lw[2 * H * H + c]);
            const float g = valid ? dh_out[(size_t)node * H + c] : 0.f;
            dout[c] = out > 0.f ? g : 0.f;
            dbacc[c] += dout[c];
        }
        __syncthreads();
        // restore [h | agg] and stage d_out (BF16)
        stage_row(X, lane, hv, agg);
        store_row_bf16(D + lane * kLdD, dout);
        __syncthreads();
        // weight gradients: G[o][c] += sum_cells D[cell][o] X[cell][c]
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            bf16x4 afr[2], bfr[4];
#pragma unroll
            for (int mt = 0; mt < 2; ++mt)
#pragma unroll
                for (int qq = 0; qq < 4; ++qq) afr[mt][qq] = (short)D[(kk * 16 + 4 * q + qq) * kLdD + mt * 16 + r16];
#pragma unroll
            for (int nt = 0; nt < 4; ++nt)
#pragma unroll
                for (int qq = 0; qq < 4; ++qq) bfr[nt][qq] = (short)X[(kk * 16 + 4 * q + qq) * kLdA + nt * 16 + r16];
#pragma unroll
            for (int mt = 0; mt < 2; ++mt)
#pragma unroll
                for (int nt = 0; nt < 4; ++nt)
                    gacc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(afr[mt], bfr[nt], gacc[mt][nt], 0, 0, 0);
        }
        // input gradients: [d_self | d_agg](cell, 64) = d_out(cell, 32) * Wcat(32, 64), Wcat[o][c] = Ws[o][c] | Wm[o][c-32]
        f32x4 iacc[4][4];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) iacc[t][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            bf16x4 bfr[4];
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) {
                const int c = nt * 16 + r16;
#pragma unroll
                for (int qq = 0; qq < 4; ++qq) {
                    const int o = kk * 16 + 4 * q + qq;
                    bfr[nt][qq] = (short)(c < H ? lw[o * H + c] : lw[H * H + o * H + (c - H)]);
                }
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                bf16x4 afr;
#pragma unroll
                for (int qq = 0; qq < 4; ++qq) afr[qq] = (short)D[(16 * t + r16) * kLdD + kk * 16 + 4 * q + qq];
#pragma unroll
                for (int nt = 0; nt < 4; ++nt)
                    iacc[t][nt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(afr, bfr[nt], iacc[t][nt], 0, 0, 0);
            }
        }
        __syncthreads();
        // two passes through the 64 x 36 FP32 view of X: d_self, then d_agg
#pragma unroll
        for (int half = 0; half < 2; ++half) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int nn = 0; nn < 2; ++nn)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        C[(16 * t + 4 * q + j) * kLdC + nn * 16 + r16] = iacc[t][2 * half + nn][j];
            __syncthreads();
            // eight lanes a row: whole rows per store
#pragma unroll
            for (int it = 0; it < 8; ++it) {
                const int rr = 8 * it + (lane >> 3), c4 = 4 * (lane & 7);
                const int cell = chunk * 256 + wv * 64 + rr;
                if (cell < n) {
                    float4 v = *reinterpret_cast<const float4 *>(C + rr * kLdC + c4);
                    const size_t o = (size_t)cell * H + c4;
                    if (half == 0) {
                        const float4 g = *reinterpret_cast<const float4 *>(dh_out + o);
                        v = make_float4(g.x + v.x, g.y + v.y, g.z + v.z, g.w + v.w);
                        *reinterpret_cast<float4 *>(dh_part + o) = v;
                    } else {
                        *reinterpret_cast<float4 *>(dagg + o) = v;
                    }
                }
            }
            __syncthreads();
        }
    }
    // per-wave partial: [dWs (32x32) | dWm (32x32) | db (32)], element G[o][c] at o*64 + c
    float *wp = wpart + (size_t)(blockIdx.x * kWaves + wv) * (2 * H * H + H);
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int o = mt * 16 + 4 * q + j, c = nt * 16 + r16;
                const int dst = c < H ? o * H + c : H * H + o * H + (c - H);
                wp[dst] = gacc[mt][nt][j];
            }
#pragma unroll
    for (int c = 0; c < H; ++c) {
        float v = wave_sum(dbacc[c]);
        if (lane == 0) wp[2 * H * H + c] = v;
    }
}

// Layer backward, part 2 (eight lanes per cell j, four channels each, so that a row is
// read and written whole): messages flow back along the transposed entries, dh_in_j =
// dh_part_j + sum_{k in row j} c_{t(k)} d_agg_{ja[k]}, and the gate gradient dc_t =
// d_agg_i . h_j (linear in the lanes' parts, which are added at the end).  First layer:
// encoder gradients.  Bound by the rows gathered (6 x 128 B a cell): 33 us at
// 64^3, with a thread per cell and a wave per SIMD 48 us (81 us in the first layer).
template <bool FIRST>
__global__ __launch_bounds__(256) void k_gnn_bwd2(int n, GnnEll E, const float *__restrict__ u,
                                                  const bf16_t *__restrict__ h_in, const float *__restrict__ dh_part,
                                                  const float *__restrict__ dagg, const bf16_t *__restrict__ w,
                                                  int layer, float *__restrict__ dh_in, float *__restrict__ gpart) {
    __shared__ double sh[4][3 + 2 * H];
    const bf16_t *lw = w + kGnnOffLayer0 + layer * kGnnLayerStride;
    const float g0 = bf2f(lw[2 * H * H + H]), g1 = bf2f(lw[2 * H * H + H + 1]), g2 = bf2f(lw[2 * H * H + H + 2]);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, q = lane & 7, c0 = 4 * q;
    float ew[4], eb[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        ew[t] = bf2f(w[kGnnOffEncW + c0 + t]);
        eb[t] = bf2f(w[kGnnOffEncB + c0 + t]);
    }
    float dg[3] = {0.f, 0.f, 0.f}, denc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int j = blockIdx.x * 32 + (threadIdx.x >> 3); j < n; j += gridDim.x * 32) {
        float hj[4], pre[4], uj = 0.f;
        if (FIRST) {
            uj = u[j];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                pre[t] = ew[t] * uj + eb[t];
                hj[t] = bfround(fmaxf(pre[t], 0.f));
            }
        } else {
            // channels 4q .. 4q + 3 of a stored row: half q / 4 of its group q % 4
            const uint2 raw = *reinterpret_cast<const uint2 *>(h_in + (size_t)j * H + 8 * (q & 3) + 4 * (q >> 2));
            hj[0] = __uint_as_float(raw.x << 16);
            hj[1] = __uint_as_float(raw.x & 0xffff0000u);
            hj[2] = __uint_as_float(raw.y << 16);
            hj[3] = __uint_as_float(raw.y & 0xffff0000u);
        }
        const float4 dp = *reinterpret_cast<const float4 *>(dh_part + (size_t)j * H + c0);
        float d[4] = {dp.x, dp.y, dp.z, dp.w};
        const int cnt = E.cnt[j];
        for (int k = 0; k < cnt; ++k) {
            // slot k of cell j: neighbour i, and the features of entry (i, j) of row i
            const int i = E.nbr[(size_t)k * E.n + j];
            const uint32_t e = E.eft[(size_t)k * E.n + j];
            const float4 da = *reinterpret_cast<const float4 *>(dagg + (size_t)i * H + c0);
            const float e1 = bf2f((bf16_t)(e & 0xffffu)), e2 = bf2f((bf16_t)(e >> 16));
            const float ct = edge_gate(g0, g1, g2, e);
            d[0] += ct * da.x;
            d[1] += ct * da.y;
            d[2] += ct * da.z;
            d[3] += ct * da.w;
            const float dc = (da.x * hj[0] + da.y * hj[1]) + (da.z * hj[2] + da.w * hj[3]);
            dg[0] += dc;
            dg[1] += dc * e1;
            dg[2] += dc * e2;
        }
        if (!FIRST) {
            *reinterpret_cast<float4 *>(dh_in + (size_t)j * H + c0) = make_float4(d[0], d[1], d[2], d[3]);
        } else {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const float dp_ = pre[t] > 0.f ? d[t] : 0.f;
                denc[t] += dp_ * uj;
                denc[4 + t] += dp_;
            }
        }
    }
    // block sums in FP64: the lanes of one channel group, then the four waves
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const double v = wave_sum((double)dg[c]);
        if (lane == 0) sh[wv][c] = v;
    }
    if (FIRST) {
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            double v = (double)denc[t];
#pragma unroll
            for (int off = 32; off >= 8; off >>= 1) v += __shfl_down(v, off, kWave);
            if (lane < 8) sh[wv][3 + (t >> 2) * H + c0 + (t & 3)] = v;
        }
    }
    __syncthreads();
    const int stride = 3 + 2 * H;
    const int c = threadIdx.x;
    if (c < (FIRST ? stride : 3))
        gpart[(size_t)blockIdx.x * stride + c] = (float)((sh[0][c] + sh[1][c]) + (sh[2][c] + sh[3][c]));
}

// grad[off + c] += sum_p part[p * stride + col0 + c], c < width (fixed order over p): a
// block takes 64 columns, sixteen waves a sixteenth of the partials each, eight rows in
// flight: 9.5 us for 2,048 rows of 2,080 columns (one thread per column adding 1,024 rows
// one by one took 134 us a launch, ten launches a gradient)
constexpr int kReduceRows = 16;
__global__ __launch_bounds__(64 * kReduceRows) void k_gnn_reduce(int nparts, int stride, int col0, int width,
                                                                 const float *__restrict__ part,
                                                                 float *__restrict__ grad, int off) {
    __shared__ double sh[kReduceRows][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int c = blockIdx.x * 64 + lane;
    const int per = (nparts + kReduceRows - 1) / kReduceRows;
    const int p1 = min(nparts, (w + 1) * per);
    double s = 0.0;
    if (c < width) {
        const float *src = part + col0 + c;
        int p = w * per;
        for (; p + 8 <= p1; p += 8) {
            float v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = src[(size_t)(p + k) * stride];
#pragma unroll
            for (int k = 0; k < 8; ++k) s += (double)v[k];
        }
        for (; p < p1; ++p) s += (double)src[(size_t)p * stride];
    }
    sh[w][lane] = s;
    __syncthreads();
    if (w == 0 && c < width) {
        double t = 0.0;
#pragma unroll
        for (int k = 0; k < kReduceRows; ++k) t += sh[k][lane];
        grad[off + c] += (float)t;
    }
}

__global__ void k_gnn_adam(int np, float *__restrict__ th, const float *__restrict__ g, float *__restrict__ m,
                           float *__restrict__ v, float lr, float b1, float b2, float eps, float bc1, float bc2,
                           bf16_t *__restrict__ wbf) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float t = th[i] - lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
    th[i] = t;
    wbf[i] = f2bf(t);
}

__global__ void k_gnn_to_bf16(int np, const float *__restrict__ th, bf16_t *__restrict__ wbf) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < np) wbf[i] = f2bf(th[i]);
}

__global__ void k_f2d_axpy(int n, const float *__restrict__ x, double *__restrict__ acc) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) acc[i] += (double)x[i];
}

}  // namespace

// ---------------------------------------------------------------- graph

namespace {

// The cluster layout of a graph whose ELL is built (GnnGraph::cperm ...): four
// radix sorts (one per axis for the ranks, one of the Morton codes) and one
// workgroup per cluster for the halos.  Leaves cl_ok false when a halo exceeds
// kGnnClHalo.
void build_clusters(hipStream_t s, GnnGraph &g, const double *xc, const double *yc, const double *zc) {
    const int n = g.n;
    g.ncl = (n + kGnnClCells - 1) / kGnnClCells;
    const int n_pad = g.ncl * kGnnClCells;
    const int gb = std::min(grid_for(n, 256), 8192);
    DevBuf ka(sizeof(unsigned long long) * n), kb(sizeof(unsigned long long) * n), ia(sizeof(int) * n),
        ib(sizeof(int) * n), rk(sizeof(int) * 3 * (size_t)n), tmp;
    const double *axis[3] = {xc, yc, zc};
    for (int d = 0; d < 3; ++d) {
        k_cl_axis_keys<<<gb, 256, 0, s>>>(n, axis[d], ka.as<unsigned long long>(), ia.as<int>());
        sort_pairs_u64(s, ka.as<unsigned long long>(), kb.as<unsigned long long>(), ia.as<int>(), ib.as<int>(), n,
                       tmp);
        k_cl_rank<<<gb, 256, 0, s>>>(n, ib.as<int>(), rk.as<int>() + (size_t)d * n);
    }
    k_cl_morton<<<gb, 256, 0, s>>>(n, rk.as<int>(), rk.as<int>() + n, rk.as<int>() + 2 * (size_t)n,
                                   ka.as<unsigned long long>(), ia.as<int>());
    g.cperm.ensure(sizeof(int) * (size_t)n_pad);
    g.cinv.ensure(sizeof(int) * (size_t)n);
    sort_pairs_u64(s, ka.as<unsigned long long>(), kb.as<unsigned long long>(), ia.as<int>(), g.cperm.as<int>(), n,
                   tmp);
    k_cl_inverse<<<std::min(grid_for(n_pad, 256), 8192), 256, 0, s>>>(n, n_pad, g.cperm.as<int>(), g.cinv.as<int>());
    g.hcnt.ensure(sizeof(int) * (size_t)g.ncl);
    g.halo.ensure(sizeof(int) * (size_t)g.ncl * kGnnClHalo);
    g.lidx.ensure(sizeof(uint32_t) * (size_t)(g.ew / 2) * n_pad);
    DevBuf ovf(sizeof(int));
    FC_HIP_CHECK(hipMemsetAsync(ovf.get(), 0, sizeof(int), s));
    FC_HIP_CHECK(hipMemsetAsync(g.halo.get(), 0, sizeof(int) * (size_t)g.ncl * kGnnClHalo, s));
#define FC_CL_HALO(W)                                                                                              \
    k_cl_halo<W><<<g.ncl, kGnnClCells, 0, s>>>(n, n_pad, g.cperm.as<int>(), g.cinv.as<int>(), g.ecnt.as<int>(),      \
                                               g.enbr.as<int>(), g.hcnt.as<int>(), g.halo.as<int>(),                 \
                                               g.lidx.as<uint32_t>(), ovf.as<int>())
    if (g.ew == 4) FC_CL_HALO(4);
    else if (g.ew == 6) FC_CL_HALO(6);
    else FC_CL_HALO(8);
#undef FC_CL_HALO
    FC_HIP_CHECK(hipGetLastError());
    int over = 0;
    FC_HIP_CHECK(hipMemcpyAsync(&over, ovf.get(), sizeof(int), hipMemcpyDeviceToHost, s));
    FC_HIP_CHECK(hipStreamSynchronize(s));
    g.cl_ok = over <= kGnnClHalo;
    g.cl_halo_max = over;
    g.cl_n = n;
}

}  // namespace

void gnn_prepare_graph(fc_context *ctx, GnnGraph &g, Structure &st, const int *kface, const int *owner0,
                       const int *ij, const int *ji, int nif, const double *arx, const double *ary, const double *arz,
                       const double *xc, const double *yc, const double *zc, const double *a) {
    (void)owner0;
    hipStream_t s = ctx->stream;
    g.n = st.n;
    g.nnz = st.nnz;
    g.ptr = st.ioffset.as<int>();
    g.ja = st.ja.as<int>();
    g.diagpos = st.diag.as<int>();
    // what depends on the structure and geometry only is built once per structure:
    // the transposed-entry index, the ELL width, the block order and the cluster layout
    const bool new_structure = !g.ready || g.skey != st.key || g.n_struct != st.n;
    g.ef.ensure(sizeof(uint32_t) * (size_t)st.nnz);
    g.dg.ensure(sizeof(float) * (size_t)st.n);
    g.a32.ensure(sizeof(float) * (size_t)st.nnz);
    k_gnn_edges<<<grid_for(st.n, 256), 256, 0, s>>>(st.n, g.ptr, g.ja, g.diagpos, kface, arx, ary, arz, xc, yc, zc, a,
                                                    g.ef.as<uint32_t>(), g.dg.as<float>());
    k_cast_df<<<std::min(grid_for(st.nnz, 256), 8192), 256, 0, s>>>(st.nnz, a, g.a32.as<float>());
    g.slices = slices_for(ctx, st);
    if (g.slices.w) {
        g.as32.ensure(sizeof(float) * slice_count(st.n, g.slices));
        slice_values32(s, st.n, g.slices, a, g.as32.as<float>());
    }
    if (new_structure) {
        g.trans.ensure(sizeof(int) * (size_t)st.nnz);
        k_gnn_trans_init<<<grid_for(st.nnz, 256), 256, 0, s>>>(st.nnz, g.trans.as<int>());
        if (nif) k_gnn_trans<<<grid_for(nif, 256), 256, 0, s>>>(nif, ij, ji, g.trans.as<int>());
        k_gnn_trans_diag<<<grid_for(st.n, 256), 256, 0, s>>>(st.n, g.diagpos, g.trans.as<int>());
        // ELL of the off-diagonal entries
        DevBuf wmax(sizeof(int));
        FC_HIP_CHECK(hipMemsetAsync(wmax.get(), 0, sizeof(int), s));
        k_gnn_width<<<grid_for(st.n, 256), 256, 0, s>>>(st.n, g.ptr, wmax.as<int>());
        int ew = 0;
        FC_HIP_CHECK(hipMemcpyAsync(&ew, wmax.get(), sizeof(int), hipMemcpyDeviceToHost, s));
        FC_HIP_CHECK(hipStreamSynchronize(s));
        // stored width = the width the layer kernels are compiled for (4, 6, 8), or the
        // largest count for the generic kernel; slots past a cell's count are padding
        g.ew = ew <= 4 ? 4 : ew <= 6 ? 6 : ew <= 8 ? 8 : ew;
    }
    const size_t en = (size_t)g.ew * (size_t)st.n;
    g.ecnt.ensure(sizeof(int) * (size_t)st.n);
    g.enbr.ensure(sizeof(int) * en);
    g.eef.ensure(sizeof(uint32_t) * en);
    g.eeft.ensure(sizeof(uint32_t) * en);
    k_gnn_ell<<<grid_for(st.n, 256), 256, 0, s>>>(st.n, g.ew, g.ptr, g.ja, g.diagpos, g.ef.as<uint32_t>(),
                                                  g.trans.as<int>(), g.ecnt.as<int>(), g.enbr.as<int>(),
                                                  g.eef.as<uint32_t>(), g.eeft.as<uint32_t>());
    // block order: Morton code of the block centroids, 21 bits per axis over the bounding box
    if (new_structure) {
        g.nblk = (st.n + 63) / 64;
        DevBuf cen(sizeof(float) * 3 * (size_t)g.nblk);
        k_gnn_block_centre<<<grid_for(g.nblk, 256), 256, 0, s>>>(st.n, g.nblk, xc, yc, zc, cen.as<float>());
        FC_HIP_CHECK(hipGetLastError());
        std::vector<float> hc(3 * (size_t)g.nblk);
        FC_HIP_CHECK(hipMemcpyAsync(hc.data(), cen.get(), sizeof(float) * hc.size(), hipMemcpyDeviceToHost, s));
        FC_HIP_CHECK(hipStreamSynchronize(s));
        const std::vector<int> order = block_order(hc, g.nblk);
        g.border.ensure(sizeof(int) * (size_t)g.nblk);
        FC_HIP_CHECK(
            hipMemcpyAsync(g.border.get(), order.data(), sizeof(int) * (size_t)g.nblk, hipMemcpyHostToDevice, s));
        FC_HIP_CHECK(hipStreamSynchronize(s));
        g.cl_n = -1;   // the cluster layout follows the structure
    }
    // cluster layout of the inference layers: the order and halos once per structure,
    // the features at every assembly
    if (g.ew == 4 || g.ew == 6 || g.ew == 8) {
        if (g.cl_n != st.n) build_clusters(s, g, xc, yc, zc);
        g.gate_wver = -1;
        if (g.cl_ok) {
            const int n_pad = g.ncl * kGnnClCells;
            g.efc.ensure(sizeof(uint32_t) * (size_t)g.ew * n_pad);
            k_cl_feats<<<std::min(grid_for((long long)g.ew * n_pad, 256), 8192), 256, 0, s>>>(
                st.n, n_pad, g.ew, g.cperm.as<int>(), g.eef.as<uint32_t>(), g.efc.as<uint32_t>());
            FC_HIP_CHECK(hipGetLastError());
        }
    } else {
        g.cl_ok = false;
    }
    g.skey = st.key;
    g.n_struct = st.n;
    g.ready = true;
}

void ensure_coarse(fc_system *sys, GnnGraph &g);

GnnGraph &system_graph(fc_system *sys) {
    if (sys->graph_version != sys->assembly_version || !sys->graph.ready) {
        GeometryDev &g = sys->mesh.g;
        gnn_prepare_graph(sys->ctx, sys->graph, sys->st, sys->kface.as<int>(), sys->mesh.owner.as<int>(),
                          sys->ij.as<int>(), sys->ji.as<int>(), sys->mesh.nif, g.arx.as<double>(), g.ary.as<double>(),
                          g.arz.as<double>(), g.xc.as<double>(), g.yc.as<double>(), g.zc.as<double>(),
                          sys->a.as<double>());
        sys->graph_version = sys->assembly_version;
    }
    return sys->graph;
}

}  // namespace fcap

// ================================================================ network

using namespace fcap;

// versions of network weights, unique over the process (GnnGraph::gate_wver)
long long next_wver() {
    static std::atomic<long long> v{0};
    return ++v;
}

struct GnnSample {
    fc_system *sys;
    DevBuf r, e;      // FP32 residual and error
    double eAe;       // e^T A e with the FP32 matrix
};

struct fc_gnn {
    fc_context *ctx = nullptr;
    DevBuf master, wbf, grad, m, v;
    int step = 0;
    long long wver = 0;   // version of wbf: a new value at every change of the weights (next_wver)
    // damped-Jacobi steps after the network that training takes into the loss
    // (fc_gnn_set_training_smoothing; 0: the network's own output)
    int train_smooth = 0;
    float train_omega = 0.8f;
    // the coarse correction after the steps in the loss (fc_gnn_set_training_coarse)
    int train_coarse = 0;
    std::vector<GnnSample> data;
    // scratch
    int cap_n = 0;
    DevBuf u, s, part, h[kGnnL + 1], dha, dhb, dagg, zbuf, dz, dvec, qvec, wpart, gpart, lossacc, sma, smb, zero;
    void ensure(int n) {
        if (n <= cap_n) return;
        const size_t F = sizeof(float) * (size_t)n;
        u.alloc(F);
        s.alloc(sizeof(float) * 4);
        // partials of the grid-capped reductions and of one SpMV block per kSpmvRows rows
        part.alloc(sizeof(double) * std::max(kMaxRedGrid, spmv_grid(n)));
        for (auto &b : h) b.alloc(sizeof(bf16_t) * (size_t)n * kGnnH);
        dha.alloc(F * kGnnH);
        dhb.alloc(F * kGnnH);
        dagg.alloc(F * kGnnH);
        zbuf.alloc(F);
        dz.alloc(F);
        dvec.alloc(F);
        qvec.alloc(F);
        lossacc.alloc(sizeof(double) * 4);
        sma.alloc(F);
        smb.alloc(F);
        zero.alloc(F);
        FC_HIP_CHECK(hipMemset(zero.get(), 0, F));
        cap_n = n;
    }
};

namespace {

// blocks of the backward kernels (grid-strided over cells): what fits the CUs at once
// (layer part 1 holds 57 KB of LDS)
constexpr int kBwdGrid = 512, kBwd2Grid = 2048, kDecGrid = 1024;

void gnn_normalise(fc_gnn *net, hipStream_t s, const GnnGraph &g, const float *r, const Scalars *sc) {
    const int gp = std::min(kMaxRedGrid, grid_for(g.n, 256));
    k_gnn_norm_part<<<gp, 256, 0, s>>>(g.n, r, g.dg.as<float>(), net->part.as<double>(), sc);
    k_gnn_norm_fin<<<1, 256, 0, s>>>(gp, net->part.as<double>(), g.n, net->s.as<float>(), sc);
    k_gnn_input<<<std::min(grid_for(4LL * g.n, 256), 8192), 256, 0, s>>>(g.n, r, g.dg.as<float>(), net->s.as<float>(),
                                                                  net->wbf.as<bf16_t>(), net->u.as<float>(),
                                                                  net->h[0].as<bf16_t>(), sc);
}

GnnEll ell_of(const GnnGraph &g) {
    GnnEll e;
    e.n = g.n;
    e.cnt = g.ecnt.as<int>();
    e.nbr = g.enbr.as<int>();
    e.ef = g.eef.as<uint32_t>();
    e.eft = g.eeft.as<uint32_t>();
    return e;
}

// One layer launch.  ELL widths 4, 6 and 8 (hex and tet meshes) run the
// persistent quad kernel with the width compiled in; wider cells (polyhedral
// meshes) run the one-lane-per-cell kernel over each cell's own count.  last:
// the decoder writes z (and, with store, the layer's rows too); hin == nullptr:
// the first layer computes the encoder rows from u (quad kernel, inference).
template <int W>
void launch_layer_w(fc_gnn *net, hipStream_t s, const GnnGraph &g, int l, const bf16_t *hin, bf16_t *hout, float *z,
                    const Scalars *sc, bool last, bool store) {
    const int nblk = grid_for(g.n, 64);
    const GnnEll E = ell_of(g);
    const int *ord = g.nblk == nblk ? g.border.as<int>() : nullptr;
    const bf16_t *w = net->wbf.as<bf16_t>();
    const float *u = net->u.as<float>();
    const float *sp = net->s.as<float>();
    if constexpr (W > 0) {
        // persistent waves, as many as are resident (two per SIMD), walking each XCD's
        // eighth of the Morton-ordered blocks
        const int pw = std::max(1, net->ctx->num_cus / kXcds) * 4 * 2;
        const int pgrid = kXcds * pw;
        if (hin == nullptr) {
            FC_REQUIRE(!last, FC_ERR_ARGUMENT, "the fused first layer is not the last one");
            k_gnn_layer_quad<false, false, W, true><<<pgrid, 64, 0, s>>>(g.n, E, u, nullptr, hout, nullptr, sp, w, l,
                                                                         sc, pw, ord);
        } else if (!last) {
            k_gnn_layer_quad<false, false, W><<<pgrid, 64, 0, s>>>(g.n, E, u, hin, hout, nullptr, sp, w, l, sc, pw,
                                                                   ord);
        } else if (store) {
            k_gnn_layer_quad<true, true, W><<<pgrid, 64, 0, s>>>(g.n, E, u, hin, hout, z, sp, w, l, sc, pw, ord);
        } else {
            k_gnn_layer_quad<true, false, W><<<pgrid, 64, 0, s>>>(g.n, E, u, hin, nullptr, z, sp, w, l, sc, pw, ord);
        }
        return;
    }
    FC_REQUIRE(hin != nullptr, FC_ERR_ARGUMENT, "only the quad layer kernel computes the encoder rows");
    const int grid = (nblk + kXcds - 1) / kXcds * kXcds;
    const int block = 64 * kLayerWaves;
    if (!last)
        k_gnn_layer<false, false, W><<<grid, block, 0, s>>>(g.n, E, u, hin, hout, nullptr, sp, w, l, sc, 1, ord);
    else if (store)
        k_gnn_layer<true, true, W><<<grid, block, 0, s>>>(g.n, E, u, hin, hout, z, sp, w, l, sc, 1, ord);
    else
        k_gnn_layer<true, false, W><<<grid, block, 0, s>>>(g.n, E, u, hin, nullptr, z, sp, w, l, sc, 1, ord);
}

void launch_layer(fc_gnn *net, hipStream_t s, const GnnGraph &g, int l, const bf16_t *hin, bf16_t *hout, float *z,
                  const Scalars *sc, bool last, bool store) {
    switch (g.ew) {
    case 4: launch_layer_w<4>(net, s, g, l, hin, hout, z, sc, last, store); break;
    case 6: launch_layer_w<6>(net, s, g, l, hin, hout, z, sc, last, store); break;
    case 8: launch_layer_w<8>(net, s, g, l, hin, hout, z, sc, last, store); break;
    default: launch_layer_w<0>(net, s, g, l, hin, hout, z, sc, last, store); break;
    }
}

// Inference: the first layer computes the encoder rows itself (quad kernel).
bool fused_first_layer(const GnnGraph &g) { return (g.ew == 4 || g.ew == 6 || g.ew == 8) && kGnnL > 1; }

// The inference layers run over the cluster layout when the graph has one and
// the context does not ask for cell order (fc_set_network_layout).
bool cluster_layers(const fc_gnn *net, const GnnGraph &g) {
    return g.cl_ok && net->ctx->gnn_layout == FC_NET_CLUSTERS && kGnnL > 1;
}

// The gate pairs of the cluster layout for the network's current weights (once
// per change of weights or features; the learned solve builds them before it
// captures its iterations).
void ensure_cl_gates(fc_gnn *net, hipStream_t s, const GnnGraph &gc) {
    if (gc.gate_wver == net->wver) return;
    GnnGraph &g = const_cast<GnnGraph &>(gc);
    const int n_pad = g.ncl * kGnnClCells;
    const long long total = (long long)kGnnL * (g.ew / 2) * n_pad;
    g.cgate.ensure(sizeof(uint2) * (size_t)total);
    k_cl_gates<<<std::min(grid_for(total, 256), 8192), 256, 0, s>>>(n_pad, g.ew, g.lidx.as<uint32_t>(),
                                                                     g.efc.as<uint32_t>(), net->wbf.as<bf16_t>(),
                                                                     g.cgate.as<uint2>());
    FC_HIP_CHECK(hipGetLastError());
    g.gate_wver = net->wver;
}

template <int W>
void launch_layer_cl_w(fc_gnn *net, hipStream_t s, const GnnGraph &g, int l, const bf16_t *hin, bf16_t *hout,
                       float *z, const Scalars *sc) {
    // persistent: two workgroups per CU (the registers of the next cluster's inputs
    // leave room for two), dealt round-robin to the XCDs
    const int wpx = std::max(1, net->ctx->num_cus / kXcds) * 2;
    const int grid = wpx * kXcds;
    const int *hc = g.hcnt.as<int>(), *hl = g.halo.as<int>(), *cp = g.cperm.as<int>();
    const uint2 *gt = g.cgate.as<uint2>();
    const float *u = net->u.as<float>(), *sp = net->s.as<float>();
    const bf16_t *w = net->wbf.as<bf16_t>();
    if (l == 0)
        k_gnn_layer_cl<W, true, false><<<grid, kGnnClCells, 0, s>>>(g.n, g.ncl, wpx, hc, hl, gt, cp, u, nullptr, hout,
                                                                    nullptr, sp, w, l, sc);
    else if (l < kGnnL - 1)
        k_gnn_layer_cl<W, false, false><<<grid, kGnnClCells, 0, s>>>(g.n, g.ncl, wpx, hc, hl, gt, cp, u, hin, hout,
                                                                     nullptr, sp, w, l, sc);
    else
        k_gnn_layer_cl<W, false, true><<<grid, kGnnClCells, 0, s>>>(g.n, g.ncl, wpx, hc, hl, gt, cp, u, hin, nullptr, z,
                                                                    sp, w, l, sc);
}

void launch_layer_cl(fc_gnn *net, hipStream_t s, const GnnGraph &g, int l, const bf16_t *hin, bf16_t *hout, float *z,
                     const Scalars *sc) {
    switch (g.ew) {
    case 4: launch_layer_cl_w<4>(net, s, g, l, hin, hout, z, sc); break;
    case 6: launch_layer_cl_w<6>(net, s, g, l, hin, hout, z, sc); break;
    default: launch_layer_cl_w<8>(net, s, g, l, hin, hout, z, sc); break;
    }
}

// z = P(r).  training: keep h1..h4 for the backward pass.
void gnn_forward(fc_gnn *net, hipStream_t s, const GnnGraph &g, const float *r, float *z, const Scalars *sc,
                 bool training) {
    net->ensure(g.n);
    const bool fused = !training && fused_first_layer(g);
    if (fused && cluster_layers(net, g)) {
        // u and the rows in position order; the last layer scatters z back to cell order
        ensure_cl_gates(net, s, g);
        const int gp = std::min(kMaxRedGrid, grid_for(g.n, 256));
        k_gnn_norm_part<<<gp, 256, 0, s>>>(g.n, r, g.dg.as<float>(), net->part.as<double>(), sc);
        k_gnn_norm_fin<<<1, 256, 0, s>>>(gp, net->part.as<double>(), g.n, net->s.as<float>(), sc);
        k_gnn_u_cl<<<std::min(grid_for(g.n, 256), 8192), 256, 0, s>>>(g.n, g.cinv.as<int>(), r, g.dg.as<float>(),
                                                                      net->s.as<float>(), net->u.as<float>(), sc);
        bf16_t *hb[2] = {net->h[1].as<bf16_t>(), net->h[2].as<bf16_t>()};
        for (int l = 0; l < kGnnL; ++l)
            launch_layer_cl(net, s, g, l, l == 0 ? nullptr : hb[(l - 1) & 1], l == kGnnL - 1 ? nullptr : hb[l & 1],
                            z, sc);
        FC_HIP_CHECK(hipGetLastError());
        return;
    }
    if (fused) {
        const int gp = std::min(kMaxRedGrid, grid_for(g.n, 256));
        k_gnn_norm_part<<<gp, 256, 0, s>>>(g.n, r, g.dg.as<float>(), net->part.as<double>(), sc);
        k_gnn_norm_fin<<<1, 256, 0, s>>>(gp, net->part.as<double>(), g.n, net->s.as<float>(), sc);
        k_gnn_u<<<std::min(grid_for(g.n, 256), 8192), 256, 0, s>>>(g.n, r, g.dg.as<float>(), net->s.as<float>(),
                                                                 net->u.as<float>(), sc);
    } else {
        gnn_normalise(net, s, g, r, sc);
    }
    bf16_t *hb[kGnnL + 1];
    for (int l = 0; l <= kGnnL; ++l) hb[l] = net->h[l].as<bf16_t>();
    for (int l = 0; l < kGnnL; ++l) {
        // h0 (written by k_gnn_input, or computed inside the fused first layer) is
        // in h[0]; inference then ping-pongs between h[1] and h[2], training keeps
        // one buffer per layer
        const bf16_t *hin = training ? hb[l] : (l == 0 ? (fused ? nullptr : hb[0]) : hb[1 + ((l - 1) & 1)]);
        bf16_t *hout = training ? hb[l + 1] : (l == kGnnL - 1 ? nullptr : hb[1 + (l & 1)]);
        launch_layer(net, s, g, l, hin, hout, z, sc, l == kGnnL - 1, training);
    }
    FC_HIP_CHECK(hipGetLastError());
}

void reduce_parts(hipStream_t s, int nparts, int stride, int col0, int width, const float *part, float *grad, int off) {
    k_gnn_reduce<<<grid_for(width, 64), 64 * kReduceRows, 0, s>>>(nparts, stride, col0, width, part, grad, off);
}

// Loss of one pair and its gradient, accumulated into net->grad (scaled by coef_batch).
void gnn_backward_pair(fc_gnn *net, hipStream_t s, GnnGraph &g, const float *r, const float *e, double eAe,
                       float batch, double *loss_dev_slot) {
    const int n = g.n;
    gnn_forward(net, s, g, r, net->zbuf.as<float>(), nullptr, true);
    float *z = net->zbuf.as<float>();
    float *d = net->dvec.as<float>(), *q = net->qvec.as<float>();
    const int gv = std::min(grid_for(n, 256), 8192);
    // the preconditioner's damped-Jacobi steps after the network, when training takes them
    // into the loss: z_{k+1} = M z_k + omega D^-1 r, M = I - omega D^-1 A
    const int steps = net->train_smooth;
    float *sb[2] = {net->sma.as<float>(), net->smb.as<float>()};
    const float *zs = z;
    for (int k = 0; k < steps; ++k) {
        jacobi_step32(s, n, g.ptr, g.ja, g.a32.as<float>(), zs, r, g.dg.as<float>(), net->train_omega, sb[k & 1],
                      nullptr);
        zs = sb[k & 1];
    }
    // and the coarse correction z_c = z + P A_c^-1 P^T (r - A z), when training takes it in
    const bool coarse = net->train_coarse && g.coarse.ok;
    if (coarse) {
        float *zc = sb[steps & 1];   // the buffer zs does not occupy
        coarse_apply(s, g.coarse, r, zs, zc, nullptr);
        zs = zc;
    }
    k_gnn_diff<<<gv, 256, 0, s>>>(n, zs, e, d);
    // q = A d with the partial of d.q
    spmv_launch32(s, 2, n, g.ptr, g.ja, g.a32.as<float>(), d, nullptr, d, q, net->part.as<double>(), nullptr, nullptr);
    sum_parts_launch(s, spmv_grid(n), net->part.as<double>(), nullptr, loss_dev_slot);
    const float coef = (float)(2.0 / (eAe * (double)batch));
    k_gnn_scale<<<gv, 256, 0, s>>>(n, q, coef, net->dz.as<float>());
    if (coarse) {
        // back through the correction: dz <- (I - P A_c^-1 P^T A)^T dz = dz - A w,
        // w = P A_c^-1 P^T dz (A and A_c symmetric; the correction of a zero vector)
        coarse_apply(s, g.coarse, net->dz.as<float>(), net->zero.as<float>(), sb[0], nullptr);
        residual32(s, n, g.ptr, g.ja, g.a32.as<float>(), sb[0], net->dz.as<float>(), sb[1], nullptr);
        FC_HIP_CHECK(hipMemcpyAsync(net->dz.get(), sb[1], sizeof(float) * (size_t)n, hipMemcpyDeviceToDevice, s));
    }
    if (steps > 0) {
        // back through the steps: dz <- (M^T)^k dz = D M^k D^-1 dz (A symmetric); M t is a
        // Jacobi step of t with a zero right-hand side
        k_gnn_diag<true><<<gv, 256, 0, s>>>(n, net->dz.as<float>(), g.dg.as<float>(), sb[0]);
        for (int k = 0; k < steps; ++k)
            jacobi_step32(s, n, g.ptr, g.ja, g.a32.as<float>(), sb[k & 1], net->zero.as<float>(), g.dg.as<float>(),
                          net->train_omega, sb[(k + 1) & 1], nullptr);
        k_gnn_diag<false><<<gv, 256, 0, s>>>(n, sb[steps & 1], g.dg.as<float>(), net->dz.as<float>());
    }
    // decoder
    const bf16_t *w = net->wbf.as<bf16_t>();
    float *grad = net->grad.as<float>();
    net->gpart.ensure(sizeof(float) * (size_t)kBwd2Grid * (3 + 2 * kGnnH));
    k_gnn_dec_bwd<<<kDecGrid, 256, 0, s>>>(n, net->h[kGnnL].as<bf16_t>(), net->dz.as<float>(), net->s.as<float>(), w,
                                           net->dha.as<float>(), net->gpart.as<float>());
    reduce_parts(s, kDecGrid, kGnnH + 1, 0, kGnnH + 1, net->gpart.as<float>(), grad, kGnnOffDecW);
    // layers, last to first
    net->wpart.ensure(sizeof(float) * (size_t)kBwdGrid * kWaves * (2 * kGnnH * kGnnH + kGnnH));
    const GnnEll E = ell_of(g);
    const float *u = net->u.as<float>();
    float *dh_out = net->dha.as<float>(), *dh_in = net->dhb.as<float>();
    for (int l = kGnnL - 1; l >= 0; --l) {
        const bf16_t *hin = net->h[l].as<bf16_t>();
        float *dpart = dh_in;   // dh_part written here, then dh_in overwrites dh_out's role
        if (l == 0)
            k_gnn_bwd1<true><<<kBwdGrid, 256, 0, s>>>(n, E, u, hin, dh_out, w, l, dpart, net->dagg.as<float>(),
                                                      net->wpart.as<float>());
        else
            k_gnn_bwd1<false><<<kBwdGrid, 256, 0, s>>>(n, E, u, hin, dh_out, w, l, dpart, net->dagg.as<float>(),
                                                       net->wpart.as<float>());
        const int loff = kGnnOffLayer0 + l * kGnnLayerStride;
        const int wstride = 2 * kGnnH * kGnnH + kGnnH;
        reduce_parts(s, kBwdGrid * kWaves, wstride, 0, wstride, net->wpart.as<float>(), grad, loff);
        // dh_in of this layer goes into dh_out's buffer (no longer needed)
        if (l == 0)
            k_gnn_bwd2<true><<<kBwd2Grid, 256, 0, s>>>(n, E, u, hin, dpart, net->dagg.as<float>(), w, l, dh_out,
                                                      net->gpart.as<float>());
        else
            k_gnn_bwd2<false><<<kBwd2Grid, 256, 0, s>>>(n, E, u, hin, dpart, net->dagg.as<float>(), w, l, dh_out,
                                                       net->gpart.as<float>());
        const int gstride = 3 + 2 * kGnnH;
        reduce_parts(s, kBwd2Grid, gstride, 0, 3, net->gpart.as<float>(), grad, loff + 2 * kGnnH * kGnnH + kGnnH);
        if (l == 0)
            reduce_parts(s, kBwd2Grid, gstride, 3, 2 * kGnnH, net->gpart.as<float>(), grad, kGnnOffEncW);
    }
    FC_HIP_CHECK(hipGetLastError());
}

// z = r / a_ii: the preconditioner's start on the iterations that leave the network out
__global__ void k_jacobi_guess(int n, const float *__restrict__ r, const float *__restrict__ dg, float *__restrict__ z,
                               const Scalars *__restrict__ sc) {
    if (sc && sc->done) return;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) z[i] = r[i] / dg[i];
}

__global__ void k_copy_f(int n, const float *__restrict__ x, float *__restrict__ y, const Scalars *__restrict__ sc) {
    if (sc && sc->done) return;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) y[i] = x[i];
}

// The preconditioner of flexible CG: the network, then `gnn_smooth` damped-Jacobi
// steps z <- z + omega (r - A z) / a_ii (the network is trained on smooth errors;
// the steps damp the rough part of what it leaves), then the coarse correction
// z <- z + P A_c^{-1} P^T (r - A z) over aggregates of the mesh (what neither
// reaches: the error's components that vary only across the whole domain).
// Each step is one pass of the SpMV kernel, alternating between z and a scratch
// vector.
// After the network (or the Jacobi guess in its place) in z: the damped-Jacobi
// steps and the coarse correction.
void precondition_tail(fc_system *sys, hipStream_t s, const float *r, float *z, const Scalars *sc) {
    GnnGraph &g = sys->graph;
    const fc_context *c = sys->ctx;
    const int steps = c->gnn_smooth;
    float *buf[2] = {z, g.zscratch.as<float>()};
    for (int k = 0; k < steps; ++k)
        if (g.slices.w)
            sliced_jacobi32(s, g.n, g.slices, g.as32.as<float>(), buf[k & 1], r, g.dg.as<float>(), c->gnn_omega,
                            buf[(k + 1) & 1], sc);
        else
            jacobi_step32(s, g.n, g.ptr, g.ja, g.a32.as<float>(), buf[k & 1], r, g.dg.as<float>(), c->gnn_omega,
                          buf[(k + 1) & 1], sc);
    float *zf = buf[steps & 1];
    if (g.coarse.ok)
        coarse_apply(s, g.coarse, r, zf, z, sc);
    else if (steps & 1)
        k_copy_f<<<std::min(grid_for(g.n, 256), 8192), 256, 0, s>>>(g.n, zf, z, sc);
}

void gnn_apply_hook(void *obj, hipStream_t s, const float *r, float *z, const Scalars *sc, bool light) {
    fc_system *sys = static_cast<fc_system *>(obj);
    GnnGraph &g = sys->graph;
    if (light)
        k_jacobi_guess<<<std::min(grid_for(g.n, 256), 8192), 256, 0, s>>>(g.n, r, g.dg.as<float>(), z, sc);
    else
        gnn_forward(sys->net, s, g, r, z, sc, false);
    precondition_tail(sys, s, r, z, sc);
}

// FC_METHOD_FCG_JACOBI: the same preconditioner with the Jacobi guess on every iteration
void jacobi_apply_hook(void *obj, hipStream_t s, const float *r, float *z, const Scalars *sc, bool) {
    gnn_apply_hook(obj, s, r, z, sc, true);
}

template <class F>
fc_status gnn_guard(fc_context *ctx, F &&f) {
    if (!ctx) return FC_ERR_ARGUMENT;
    try {
        FC_HIP_CHECK(hipSetDevice(ctx->device));
        return f();
    } catch (const Error &e) {
        ctx->last_error = e.what();
        return e.code;
    } catch (const std::exception &e) {
        ctx->last_error = e.what();
        return FC_ERR_ALLOC;
    }
}

}  // namespace

namespace fcap {
// The coarse space of the system's current matrix, with the context's aggregate
// size (kept while neither changes; switched off by an aggregate size of 0).
void ensure_coarse(fc_system *sys, GnnGraph &g) {
    fc_context *ctx = sys->ctx;
    if (ctx->fcg_coarse <= 0) {
        g.coarse.ok = false;
        g.coarse.version = -1;
        return;
    }
    const int agg = coarse_aggregate_cells(g.n, ctx->fcg_coarse);
    const bool morton = g.cl_n == g.n;
    const int *perm = morton ? g.cperm.as<int>() : nullptr, *inv = morton ? g.cinv.as<int>() : nullptr;
    if (g.coarse.version == sys->assembly_version && g.coarse.agg == agg && g.coarse.n == g.n &&
        g.coarse.perm == perm && g.coarse.inv == inv)
        return;
    coarse_setup(ctx, g.coarse, g.n, g.nnz, g.ptr, g.ja, sys->a.as<double>(), g.a32.as<float>(), g.trans.as<int>(),
                 perm, inv, agg, g.ew + 1, sys->assembly_version);
}

PrecondHook gnn_hook(fc_system *sys) {
    PrecondHook h;
    if (!sys || !sys->net) return h;
    GnnGraph &g = system_graph(sys);
    sys->net->ensure(sys->st.n);
    g.zscratch.ensure(sizeof(float) * (size_t)g.n);
    if (fused_first_layer(g) && cluster_layers(sys->net, g)) ensure_cl_gates(sys->net, sys->ctx->stream, g);
    ensure_coarse(sys, g);
    h.obj = sys;
    h.apply = gnn_apply_hook;
    return h;
}

PrecondHook jacobi_hook(fc_system *sys) {
    PrecondHook h;
    if (!sys) return h;
    GnnGraph &g = system_graph(sys);
    g.zscratch.ensure(sizeof(float) * (size_t)g.n);
    ensure_coarse(sys, g);
    h.obj = sys;
    h.apply = jacobi_apply_hook;
    return h;
}
}  // namespace fcap

extern "C" int fc_gnn_num_params(void) { return kGnnParams; }

extern "C" fc_status fc_gnn_create(fc_context *ctx, fc_gnn **out, const float *params) {
    if (!out) return FC_ERR_ARGUMENT;
    *out = nullptr;
    fc_gnn *net = new fc_gnn();
    net->ctx = ctx;
    fc_status st = gnn_guard(ctx, [&]() {
        net->master.alloc(sizeof(float) * kGnnParams);
        net->wbf.alloc(sizeof(bf16_t) * kGnnParams);
        net->grad.alloc(sizeof(float) * kGnnParams);
        net->m.alloc(sizeof(float) * kGnnParams);
        net->v.alloc(sizeof(float) * kGnnParams);
        std::vector<float> p(kGnnParams, 0.f);
        if (params) std::memcpy(p.data(), params, sizeof(float) * kGnnParams);
        h2d(net->master.get(), p.data(), sizeof(float) * kGnnParams, ctx->stream);
        FC_HIP_CHECK(hipMemsetAsync(net->m.get(), 0, sizeof(float) * kGnnParams, ctx->stream));
        FC_HIP_CHECK(hipMemsetAsync(net->v.get(), 0, sizeof(float) * kGnnParams, ctx->stream));
        k_gnn_to_bf16<<<grid_for(kGnnParams, 256), 256, 0, ctx->stream>>>(kGnnParams, net->master.as<float>(),
                                                                          net->wbf.as<bf16_t>());
        net->wver = next_wver();
        FC_HIP_CHECK(hipStreamSynchronize(ctx->stream));
        return FC_OK;
    });
    if (st != FC_OK) {
        delete net;
        return st;
    }
    *out = net;
    return FC_OK;
}

extern "C" fc_status fc_gnn_destroy(fc_gnn *net) {
    if (!net) return FC_ERR_ARGUMENT;
    if (net->ctx) (void)hipStreamSynchronize(net->ctx->stream);
    delete net;
    return FC_OK;
}

extern "C" fc_status fc_gnn_set_params(fc_gnn *net, const float *params) {
    if (!net || !params) return FC_ERR_ARGUMENT;
    return gnn_guard(net->ctx, [&]() {
        h2d(net->master.get(), params, sizeof(float) * kGnnParams, net->ctx->stream);
        k_gnn_to_bf16<<<grid_for(kGnnParams, 256), 256, 0, net->ctx->stream>>>(kGnnParams, net->master.as<float>(),
                                                                               net->wbf.as<bf16_t>());
        net->wver = next_wver();
        FC_HIP_CHECK(hipMemsetAsync(net->m.get(), 0, sizeof(float) * kGnnParams, net->ctx->stream));
        FC_HIP_CHECK(hipMemsetAsync(net->v.get(), 0, sizeof(float) * kGnnParams, net->ctx->stream));
        net->step = 0;
        FC_HIP_CHECK(hipStreamSynchronize(net->ctx->stream));
        return FC_OK;
    });
}

extern "C" fc_status fc_gnn_get_params(fc_gnn *net, float *params) {
    if (!net || !params) return FC_ERR_ARGUMENT;
    return gnn_guard(net->ctx, [&]() {
        d2h(params, net->master.get(), sizeof(float) * kGnnParams, net->ctx->stream);
        return FC_OK;
    });
}

extern "C" fc_status fc_gnn_edge_features(fc_gnn *net, fc_system *sys, float *e1, float *e2, float *diag) {
    if (!net || !sys) return FC_ERR_ARGUMENT;
    return gnn_guard(net->ctx, [&]() {
        GnnGraph &g = system_graph(sys);
        std::vector<uint32_t> ef(g.nnz);
        d2h(ef.data(), g.ef.get(), sizeof(uint32_t) * g.nnz, net->ctx->stream);
        for (int k = 0; k < g.nnz; ++k) {
            uint32_t lo = (ef[k] & 0xffffu) << 16, hi = ef[k] & 0xffff0000u;
            std::memcpy(&e1[k], &lo, 4);
            std::memcpy(&e2[k], &hi, 4);
        }
        if (diag) d2h(diag, g.dg.get(), sizeof(float) * g.n, net->ctx->stream);
        return FC_OK;
    });
}

extern "C" fc_status fc_gnn_apply(fc_gnn *net, fc_system *sys, const float *r, float *z) {
    if (!net || !sys || !r || !z) return FC_ERR_ARGUMENT;
    return gnn_guard(net->ctx, [&]() {
        GnnGraph &g = system_graph(sys);
        net->ensure(g.n);
        hipStream_t s = net->ctx->stream;
        DevBuf dr(sizeof(float) * g.n), dz(sizeof(float) * g.n);
        h2d(dr.get(), r, sizeof(float) * g.n, s);
        gnn_forward(net, s, g, dr.as<float>(), dz.as<float>(), nullptr, false);
        d2h(z, dz.get(), sizeof(float) * g.n, s);
        return FC_OK;
    });
}

// Average milliseconds of one network application (device-resident residual:
// the system's FP64 RHS cast to FP32), timed with events on the library's
// stream over `reps` back-to-back applications; -1 on error.
extern "C" double fc_gnn_bench(fc_gnn *net, fc_system *sys, int reps) {
    if (!net || !sys || reps <= 0) return -1.0;
    double out = -1.0;
    fc_status st = gnn_guard(net->ctx, [&]() {
        GnnGraph &g = system_graph(sys);
        net->ensure(g.n);
        hipStream_t s = net->ctx->stream;
        DevBuf dr(sizeof(float) * g.n), dz(sizeof(float) * g.n);
        k_cast_df<<<std::min(grid_for(g.n, 256), 8192), 256, 0, s>>>(g.n, sys->su.as<double>(), dr.as<float>());
        gnn_forward(net, s, g, dr.as<float>(), dz.as<float>(), nullptr, false);   // warm-up
        net->ctx->timer.start(s);
        for (int k = 0; k < reps; ++k) gnn_forward(net, s, g, dr.as<float>(), dz.as<float>(), nullptr, false);
        out = net->ctx->timer.stop_ms(s) / reps;
        return FC_OK;
    });
    return st == FC_OK ? out : -1.0;
}

extern "C" fc_status fc_sys_network_layout(fc_system *sys, int *clusters, int *halo_max, long long *halo_total) {
    if (!sys || !clusters || !halo_max || !halo_total) return FC_ERR_ARGUMENT;
    return gnn_guard(sys->ctx, [&]() {
        GnnGraph &g = system_graph(sys);
        *clusters = g.cl_ok ? g.ncl : 0;
        *halo_max = g.cl_n == g.n ? g.cl_halo_max : 0;
        *halo_total = 0;
        if (g.cl_n == g.n && g.ncl > 0) {
            std::vector<int> hc(g.ncl);
            d2h(hc.data(), g.hcnt.get(), sizeof(int) * (size_t)g.ncl, sys->ctx->stream);
            for (int v : hc) *halo_total += v;
        }
        return FC_OK;
    });
}

extern "C" fc_status fc_sys_coarse_space(fc_system *sys, int *aggregates, int *cells_per_aggregate, int *factored,
                                         int *cell_aggregate, double *matrix) {
    if (!sys || !aggregates || !cells_per_aggregate || !factored) return FC_ERR_ARGUMENT;
    return gnn_guard(sys->ctx, [&]() {
        GnnGraph &g = system_graph(sys);
        ensure_coarse(sys, g);
        const CoarseSpace &cs = g.coarse;
        const bool on = sys->ctx->fcg_coarse > 0;
        *aggregates = on ? cs.nc : 0;
        *cells_per_aggregate = on ? cs.agg : 0;
        *factored = on && cs.ok ? 1 : 0;
        if (on && cell_aggregate) {
            std::vector<int> pos(g.n);
            if (cs.inv)
                d2h(pos.data(), cs.inv, sizeof(int) * (size_t)g.n, sys->ctx->stream);
            else
                for (int i = 0; i < g.n; ++i) pos[i] = i;
            for (int i = 0; i < g.n; ++i) cell_aggregate[i] = pos[i] / cs.agg;
        }
        if (on && matrix) coarse_matrix_host(sys->ctx, cs, matrix);
        return FC_OK;
    });
}

extern "C" fc_status fc_sys_precondition(fc_system *sys, const float *r, float *z) {
    if (!sys || !r || !z) return FC_ERR_ARGUMENT;
    return gnn_guard(sys->ctx, [&]() {
        if (!sys->net) throw Error(FC_ERR_ARGUMENT, "no network attached (fc_sys_set_network)");
        PrecondHook P = gnn_hook(sys);
        const int n = sys->st.n;
        hipStream_t s = sys->ctx->stream;
        DevBuf dr(sizeof(float) * (size_t)n), dz(sizeof(float) * (size_t)n);
        h2d(dr.get(), r, sizeof(float) * (size_t)n, s);
        P.apply(P.obj, s, dr.as<float>(), dz.as<float>(), nullptr, false);
        FC_HIP_CHECK(hipGetLastError());
        d2h(z, dz.get(), sizeof(float) * (size_t)n, s);
        return FC_OK;
    });
}

extern "C" double fc_gnn_bench_layer(fc_gnn *net, fc_system *sys, int reps) {
    if (!net || !sys || reps <= 0) return -1.0;
    double out = -1.0;
    fc_status st = gnn_guard(net->ctx, [&]() {
        GnnGraph &g = system_graph(sys);
        net->ensure(g.n);
        hipStream_t s = net->ctx->stream;
        DevBuf dr(sizeof(float) * g.n), dz(sizeof(float) * g.n);
        k_cast_df<<<std::min(grid_for(g.n, 256), 8192), 256, 0, s>>>(g.n, sys->su.as<double>(), dr.as<float>());
        gnn_forward(net, s, g, dr.as<float>(), dz.as<float>(), nullptr, false);   // rows of layers 0..2
        const bf16_t *hin = net->h[1].as<bf16_t>();
        bf16_t *hout = net->h[2].as<bf16_t>();
        const bool cl = fused_first_layer(g) && cluster_layers(net, g);
        if (cl) ensure_cl_gates(net, s, g);
        auto layer = [&]() {
            if (cl) launch_layer_cl(net, s, g, 1, hin, hout, nullptr, nullptr);
            else launch_layer(net, s, g, 1, hin, hout, nullptr, nullptr, false, false);
        };
        layer();   // warm-up
        net->ctx->timer.start(s);
        for (int k = 0; k < reps; ++k) layer();
        out = net->ctx->timer.stop_ms(s) / reps;
        FC_HIP_CHECK(hipGetLastError());
        return FC_OK;
    });
    return st == FC_OK ? out : -1.0;
}

extern "C" fc_status fc_gnn_loss_grad(fc_gnn *net, fc_system *sys, const float *r, const float *e, double *loss,
                                      float *grad) {
    if (!net || !sys || !r || !e) return FC_ERR_ARGUMENT;
    return gnn_guard(net->ctx, [&]() {
        GnnGraph &g = system_graph(sys);
        net->ensure(g.n);
        hipStream_t s = net->ctx->stream;
        DevBuf dr(sizeof(float) * g.n), de(sizeof(float) * g.n);
        h2d(dr.get(), r, sizeof(float) * g.n, s);
        h2d(de.get(), e, sizeof(float) * g.n, s);
        // e^T A e with the FP32 matrix
        spmv_launch32(s, 2, g.n, g.ptr, g.ja, g.a32.as<float>(), de.as<float>(), nullptr, de.as<float>(),
                      net->qvec.as<float>(), net->part.as<double>(), nullptr, nullptr);
        sum_parts_launch(s, spmv_grid(g.n), net->part.as<double>(), nullptr, net->lossacc.as<double>() + 2);
        double hs[4];
        d2h(hs, net->lossacc.get(), sizeof(double) * 4, s);
        const double eAe = hs[2];
        FC_HIP_CHECK(hipMemsetAsync(net->grad.get(), 0, sizeof(float) * kGnnParams, s));
        if (net->train_coarse) ensure_coarse(sys, g);
        gnn_backward_pair(net, s, g, dr.as<float>(), de.as<float>(), eAe, 1.0f, net->lossacc.as<double>());
        d2h(hs, net->lossacc.get(), sizeof(double) * 4, s);
        if (loss) *loss = hs[0] / eAe;
        if (grad) d2h(grad, net->grad.get(), sizeof(float) * kGnnParams, s);
        return FC_OK;
    });
}

// Residual/error pairs of IC(0)-PCG iterates on the homogeneous system
// A x = 0 (exact solution 0) from seeded standard-normal starts x0: after
// iters[t] iterations, e_t = -x_t and r_t = -A x_t.  Starting from random
// vectors covers the whole spectrum, from rough errors (few iterations) to
// the smooth errors IC(0)-PCG leaves behind (many).
extern "C" fc_status fc_gnn_add_samples(fc_gnn *net, fc_system *sys, int nk, const int *iters, unsigned seed) {
    if (!net || !sys || nk <= 0 || !iters) return FC_ERR_ARGUMENT;
    for (int t = 0; t < nk; ++t)
        if (iters[t] < 0) return FC_ERR_ARGUMENT;
    return gnn_guard(net->ctx, [&]() {
        fc_context *ctx = net->ctx;
        hipStream_t s = ctx->stream;
        GnnGraph &g = system_graph(sys);
        net->ensure(g.n);
        const int n = g.n;
        DevBuf zero(sizeof(double) * n), rk(sizeof(double) * n);
        FC_HIP_CHECK(hipMemsetAsync(zero.get(), 0, sizeof(double) * n, s));
        SolveArgs args;
        args.st = &sys->st;
        args.a = sys->a.as<double>();
        args.su = zero.as<double>();
        args.fi = sys->fi.as<double>();
        args.stop_rule = FC_STOP_L1;
        args.sor = 1e-30;   // never met: exactly iters[t] iterations
        std::vector<double> hx(n), hr(n);
        for (int t = 0; t < nk; ++t) {
            std::mt19937_64 rng((uint64_t)seed * 1000003ull + (uint64_t)t);
            std::normal_distribution<double> normal(0.0, 1.0);
            for (int i = 0; i < n; ++i) hx[i] = normal(rng);
            h2d(sys->fi.get(), hx.data(), sizeof(double) * n, s);
            if (iters[t] > 0) {
                args.nsw = iters[t];
                fc_solve_info info;
                solve_pcg64(ctx, args, true, &info);
            }
            // r = 0 - A x (FP64)
            spmv_launch64(s, 1, n, sys->st.ioffset.as<int>(), sys->st.ja.as<int>(), args.a, args.fi, args.su, nullptr,
                          rk.as<double>(), nullptr, ctx->ws->pa.as<double>(), ctx->ws->pb.as<double>(), nullptr);
            d2h(hr.data(), rk.get(), sizeof(double) * n, s);
            d2h(hx.data(), sys->fi.get(), sizeof(double) * n, s);
            GnnSample smp;
            smp.sys = sys;
            smp.r.alloc(sizeof(float) * n);
            smp.e.alloc(sizeof(float) * n);
            std::vector<float> fr(n), fe(n);
            for (int i = 0; i < n; ++i) {
                fr[i] = (float)hr[i];
                fe[i] = (float)(-hx[i]);
            }
            h2d(smp.r.get(), fr.data(), sizeof(float) * n, s);
            h2d(smp.e.get(), fe.data(), sizeof(float) * n, s);
            spmv_launch32(s, 2, n, g.ptr, g.ja, g.a32.as<float>(), smp.e.as<float>(), nullptr, smp.e.as<float>(),
                          net->qvec.as<float>(), net->part.as<double>(), nullptr, nullptr);
            sum_parts_launch(s, spmv_grid(n), net->part.as<double>(), nullptr, net->lossacc.as<double>() + 2);
            double hs[4];
            d2h(hs, net->lossacc.get(), sizeof(double) * 4, s);
            smp.eAe = hs[2];
            if (smp.eAe > 0.0 && std::isfinite(smp.eAe)) net->data.push_back(std::move(smp));
        }
        FC_HIP_CHECK(hipMemsetAsync(sys->fi.get(), 0, sizeof(double) * n, s));
        return FC_OK;
    });
}

extern "C" int fc_gnn_num_samples(fc_gnn *net) { return net ? (int)net->data.size() : -1; }

extern "C" fc_status fc_gnn_get_sample(fc_gnn *net, int index, float *r, float *e, int n) {
    if (!net || index < 0 || index >= (int)net->data.size() || !r || !e) return FC_ERR_ARGUMENT;
    return gnn_guard(net->ctx, [&]() {
        GnnSample &smp = net->data[index];
        FC_REQUIRE(n == smp.sys->st.n, FC_ERR_ARGUMENT, "sample length differs from n");
        d2h(r, smp.r.get(), sizeof(float) * n, net->ctx->stream);
        d2h(e, smp.e.get(), sizeof(float) * n, net->ctx->stream);
        return FC_OK;
    });
}

extern "C" fc_status fc_gnn_clear_samples(fc_gnn *net) {
    if (!net) return FC_ERR_ARGUMENT;
    net->data.clear();
    return FC_OK;
}

extern "C" fc_status fc_gnn_drop_system(fc_gnn *net, fc_system *sys) {
    if (!net || !sys) return FC_ERR_ARGUMENT;
    net->data.erase(std::remove_if(net->data.begin(), net->data.end(),
                                   [&](const GnnSample &s) { return s.sys == sys; }),
                    net->data.end());
    return FC_OK;
}

// Adam over mini-batches of `batch` samples drawn with a seeded generator;
// loss_out (may be NULL) receives the mean batch loss of every step.
extern "C" fc_status fc_gnn_train(fc_gnn *net, int steps, int batch, float lr, unsigned seed, float *loss_out) {
    if (!net || steps <= 0 || batch <= 0) return FC_ERR_ARGUMENT;
    return gnn_guard(net->ctx, [&]() {
        FC_REQUIRE(!net->data.empty(), FC_ERR_ARGUMENT, "no training samples");
        hipStream_t s = net->ctx->stream;
        std::mt19937 rng(seed);
        std::uniform_int_distribution<int> pick(0, (int)net->data.size() - 1);
        DevBuf losses(sizeof(double) * 2 * std::max(batch, 1));
        std::vector<double> hl(2 * batch);
        for (int it = 0; it < steps; ++it) {
            FC_HIP_CHECK(hipMemsetAsync(net->grad.get(), 0, sizeof(float) * kGnnParams, s));
            std::vector<double> dens(batch);
            for (int b = 0; b < batch; ++b) {
                GnnSample &smp = net->data[pick(rng)];
                GnnGraph &g = system_graph(smp.sys);
                net->ensure(g.n);
                if (net->train_coarse) ensure_coarse(smp.sys, g);
                dens[b] = smp.eAe;
                gnn_backward_pair(net, s, g, smp.r.as<float>(), smp.e.as<float>(), smp.eAe, (float)batch,
                                  losses.as<double>() + 2 * b);
            }
            net->step += 1;
            const float b1 = 0.9f, b2 = 0.999f;
            const float bc1 = 1.f - std::pow(b1, (float)net->step), bc2 = 1.f - std::pow(b2, (float)net->step);
            k_gnn_adam<<<grid_for(kGnnParams, 256), 256, 0, s>>>(kGnnParams, net->master.as<float>(),
                                                                 net->grad.as<float>(), net->m.as<float>(),
                                                                 net->v.as<float>(), lr, b1, b2, 1e-8f, bc1, bc2,
                                                                 net->wbf.as<bf16_t>());
            net->wver = next_wver();
            FC_HIP_CHECK(hipGetLastError());
            if (loss_out) {
                d2h(hl.data(), losses.get(), sizeof(double) * 2 * batch, s);
                double sum = 0.0;
                for (int b = 0; b < batch; ++b) sum += hl[2 * b] / dens[b];
                loss_out[it] = (float)(sum / batch);
            }
        }
        FC_HIP_CHECK(hipStreamSynchronize(s));
        return FC_OK;
    });
}

extern "C" fc_status fc_gnn_set_training_smoothing(fc_gnn *net, int steps, double omega) {
    if (!net || steps < 0 || steps > 8 || !(omega > 0.0 && omega < 2.0)) return FC_ERR_ARGUMENT;
    net->train_smooth = steps;
    net->train_omega = (float)omega;
    return FC_OK;
}

extern "C" fc_status fc_gnn_set_training_coarse(fc_gnn *net, int on) {
    if (!net || (on != 0 && on != 1)) return FC_ERR_ARGUMENT;
    net->train_coarse = on;
    return FC_OK;
}

extern "C" fc_status fc_sys_set_network(fc_system *sys, fc_gnn *net) {
    if (!sys) return FC_ERR_ARGUMENT;
    sys->net = net;
    return FC_OK;
}
