// Part-wise triangular sweeps (FC_SWEEP_PARTS): the analysis that splits the rows
// into parts and windows, the packed factor, and the sweep kernel.
//
// A sweep is a chain of levels (3N - 2 on an N^3 box), so its time is the chain's
// latency, not its bytes.  One persistent workgroup computes a part 64 rows (a window)
// at a time; what it reads of its own part comes from LDS, so the chain inside a
// part costs LDS round trips, and only the chain from part to part costs round
// trips through the coherent level of the memory system.  The parts are therefore
// chosen to have few hops between them and full windows inside:
//
//   * pencils (pencil_parts), where the numbering has the runs of a structured
//     block: rows in lines (each coupled to the row before it), lines in sheets,
//     sheets in stacks; a part is 64 lines, 8 lines x 8 sheets (64 lines of one
//     sheet in 2D).  A level of a part then has at most 64 rows, one per line: a
//     window is a level and takes one step.  192^3 box: 576 parts, a chain of 47
//     hops of 8 levels; 128^3 box: 256 parts, 31 hops.
//   * runs of kPartRows consecutive rows otherwise (meshes numbered with locality).
//
// Both give parts whose rows read only rows of the same or an earlier part in part
// order (the backward sweep: the same or a later one).  Tickets hand the parts out
// in that order, so every part a part reads has been handed to a wave that is
// running or has finished, and every wait ends.
#include <algorithm>
#include <cstring>
#include <vector>

#include "fcap_linalg.h"
#include "fcap_syncfree.h"

namespace fcap {

namespace {

constexpr int kBlock = 256;
// values of a part kept in the wave's LDS: a ring over its packed slots (an entry
// further back than the ring reaches is read from memory like another part's)
constexpr int kRing = 1024;

inline int grid_for(long long n, int block = kBlock) {
    return (int)std::max<long long>(1, (n + block - 1) / block);
}

// Packed operands of a slot: W + 1 values of E in 16-byte blocks, block b of slot s
// at [b * npk + s], the remaining ones as single values after the blocks.
template <class E>
__host__ __device__ inline size_t packed_at(int e, int width, size_t npk, size_t slot) {
    constexpr int V = 16 / (int)sizeof(E);
    const int blocks = (width + 1) / V;
    return e < blocks * V ? ((size_t)(e / V) * npk + slot) * V + e % V
                          : (size_t)blocks * V * npk + (size_t)(e - blocks * V) * npk + slot;
}

// flag[u] = 1 when row start[u] reads row start[u - 1] (start null: row u)
__global__ void k_run_links(int m, const int *__restrict__ start, const int *__restrict__ ptr,
                            const int *__restrict__ ja, const int *__restrict__ diag, unsigned char *__restrict__ flag) {
    const int u = blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= m) return;
    unsigned char f = 0;
    if (u > 0) {
        const int r = start ? start[u] : u, t = start ? start[u - 1] : u - 1;
        for (int k = ptr[r]; k < diag[r]; ++k)
            if (ja[k] == t) f = 1;
    }
    flag[u] = f;
}

// slot of every row (a window's padding lanes repeat its last row: not theirs)
__global__ void k_part_slots(int npk, const int *__restrict__ rows, int *__restrict__ slot_of) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= npk) return;
    if ((q & 63) != 0 && rows[q] == rows[q - 1]) return;
    slot_of[rows[q]] = q;
}

// Code of each entry of each slot: its LDS ring slot when the entry's row is of the
// same part and still in the ring, else its packed slot with the top bit set; kRing
// (which holds zero) for the padding entries.  The row itself follows the codes.
// Also checks the schedule (an entry's row comes earlier in the sweep) and counts
// the entries read from the ring.
__global__ __launch_bounds__(kBlock) void k_part_codes(int npk, int width, bool upper, const int *__restrict__ rows,
                                                       const int *__restrict__ slot_of,
                                                       const int *__restrict__ win_part,
                                                       const unsigned char *__restrict__ step,
                                                       const int *__restrict__ ptr, const int *__restrict__ ja,
                                                       const int *__restrict__ diag, int *__restrict__ codes,
                                                       unsigned long long *__restrict__ count, int *__restrict__ err) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    int in = 0, all = 0;
    if (q < npk) {
        const int i = rows[q], own = slot_of[i], w = q >> 6, part = win_part[w];
        const int s = upper ? diag[i] + 1 : ptr[i];
        const int c = upper ? ptr[i + 1] - s : diag[i] - s;
        for (int k = 0; k < width; ++k) {
            int code = kRing;
            if (k < c) {
                const int e = slot_of[ja[s + k]];
                const bool same = win_part[e >> 6] == part;
                const bool ordered = upper ? e > own : e < own;
                const bool stepped = (e >> 6) != w || (upper ? step[e] > step[own] : step[e] < step[own]);
                if (!ordered || !stepped) atomicOr(err, 1);
                const bool inside = same && (upper ? (long long)e < 64ll * w + kRing
                                                   : (long long)e + kRing >= 64ll * (w + 1));
                code = inside ? (e & (kRing - 1)) : (int)(0x80000000u | (unsigned)e);
                if (q == own) {
                    all += 1;
                    in += inside;
                }
            }
            codes[packed_at<int>(k, width, npk, q)] = code;
        }
        codes[packed_at<int>(width, width, npk, q)] = i;
    }
    for (int off = 32; off > 0; off >>= 1) {
        in += __shfl_down(in, off, kWave);
        all += __shfl_down(all, off, kWave);
    }
    if ((threadIdx.x & 63) == 0 && all) {
        atomicAdd(count, (unsigned long long)in);
        atomicAdd(count + 1, (unsigned long long)all);
    }
}

// the factor's values in the packed order: a row's strict-triangle entries in CSR
// order (zero past its last), then its pivot
template <class T>
__global__ void k_part_vals(int npk, int width, bool upper, const int *__restrict__ rows, const int *__restrict__ ptr,
                            const int *__restrict__ diag, const T *__restrict__ a, const T *__restrict__ d,
                            T *__restrict__ vals) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= npk) return;
    const int i = rows[q];
    const int s = upper ? diag[i] + 1 : ptr[i];
    const int c = upper ? ptr[i + 1] - s : diag[i] - s;
    for (int k = 0; k < width; ++k) vals[packed_at<T>(k, width, npk, q)] = k < c ? a[s + k] : T(0);
    vals[packed_at<T>(width, width, npk, q)] = d[i];
}

template <class T>
__global__ void k_part_mark(int npk, T *__restrict__ w) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q < npk) sf_mark(w + q);
}

// ------------------------------------------------------------------- kernel

struct PartView {
    int npk;
    const int *codes;
    const unsigned char *step;
};

// A workgroup computes a part.  Wave 0 does nothing but the chain: per window it reads
// its operands and the inputs' values from LDS, forms the rows' values, puts them into
// the ring and publishes them.  The pollers fetch the inputs from other parts, each a
// window in turn.  The feeders stage the windows, each kBatch in turn: operands and
// right-hand side from memory, kStage windows ahead at most; they also store what need
// not be early (the result in row order, the marks for the next sweep).  A wave issues
// one instruction in four cycles at most: with one wave per part doing all of it a window
// took 330 ns (of about 110 instructions), with the chain apart 160 ns.  The polls are
// apart from the feeders because memory answers a wave in order: a poll repeated behind
// the prefetch of the next windows waits for that prefetch, which cost about 1 us more at
// each entry of the chain into another part.
//
// What bounds a sweep: the windows along its longest chain, 160 to 180 ns each, and 2 to
// 3 us where the chain enters another part (40^3 2.8, 128^3 3.1, 192^3 2.0, over 8, 30 and
// 47 entries; a value stored by one workgroup is seen by another's poll 0.6 to 0.75 us
// later); from some 5 M rows also the feeders' loads (about 80 B a row at W = 3 in FP64: the
// 192^3 box's 0.57 GB take 118 us at a copy's rate and 165 us here with every input there).
// Per sweep, with the
// polls in three feeders and now: 40^3 box 45 and 36 us, 96 x 80 x 72 98 and 77, 128^3 190
// and 139, 192^3 315 and 261, 163 x 75 x 1 49 and 43.  Feeders x batch, pollers at 128^3:
// 3 x 3, 2 pollers of 4 windows 173; 6 x 2, 2 of 4 167; 6 x 2, 4 of 2 142; 6 x 2, 6 of 1
// 139; 6 x 2, 8 of 1 142; 4 x 3, 11 of 1 148 us.
template <int W> struct PartShape {
    // waves that stage windows and windows a turn of one; waves that poll for inputs.  Thirteen
    // waves leave 128 registers a lane (W = 3 takes 106), twelve 168, eight 256.
    static constexpr int kFeeders = W <= 4 ? 6 : 3, kBatch = 2;
    static constexpr int kPollers = W <= 3 ? 6 : W <= 4 ? 5 : 4;
    static constexpr int kStage = kFeeders * kBatch;
    static constexpr int kBlock = 64 * (1 + kPollers + kFeeders);
    // a window's values are read from the ring at the latest when the window kStage further
    // is staged, so at most kStage - 1 windows have been written since
    static_assert(kStage <= kRing / 64, "the ring holds every window that is not retired");
};

template <class T, int W>
struct PartLds {
    static constexpr int K = PartShape<W>::kStage;
    static constexpr int V = 16 / (int)sizeof(T);
    // codes and step; values, pivot and right-hand side: 16-byte pieces, then single ones
    static constexpr int kIntVecs = (W + 1) / 4, kIntRest = (W + 1) % 4;
    static constexpr int kValVecs = (W + 2) / V, kValRest = (W + 2) % V;
    typedef T vec __attribute__((ext_vector_type(V)));
    struct Slot {
        int4 ints[kIntVecs][64];
        vec vals[kValVecs][64];
        T val1[kValRest ? kValRest : 1][64];
        int int1[kIntRest ? kIntRest : 1][64];
    } stage[K];
    // the ring of the part's values, a zero (padding entries), and the staged inputs from
    // other parts: everything a staged code points to (byte offsets)
    T x[kRing + 2 + K * W * 64];
    int fed[K];      // window index + 1 when the stage holds its operands
    int flag[K];     // the same when its inputs from other parts are there too
    int progress;    // windows the chain has finished
    int give_up, ticket;
};

template <class E, int W>
__device__ __forceinline__ void load_packed(E *out, const E *__restrict__ p, size_t npk, size_t q) {
    constexpr int V = 16 / (int)sizeof(E), B = (W + 1) / V, R = (W + 1) % V;
    typedef E vec __attribute__((ext_vector_type(V)));
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const vec v = reinterpret_cast<const vec *>(p)[(size_t)b * npk + q];
#pragma unroll
        for (int t = 0; t < V; ++t) out[b * V + t] = v[t];
    }
#pragma unroll
    for (int t = 0; t < R; ++t) out[B * V + t] = p[(size_t)B * V * npk + (size_t)t * npk + q];
}

// LDS is served in order, so a wave's data and then its flag are seen in that order by
// a wave that reads the flag and then the data: only the compiler has to keep them so.
__device__ __forceinline__ void lds_order() { __asm__ volatile("" ::: "memory"); }
__device__ __forceinline__ int lds_get(const int *p) {
    return __builtin_amdgcn_readfirstlane(__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
}
__device__ __forceinline__ void lds_set(int *p, int v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <class T, int W>
struct PartRow {
    int code[W + 1];   // the entries' codes, then the row
    T val[W + 1];      // the entries' values, then the pivot
    int step;
};
template <class T>
struct PartRun {
    int w0, nw;   // the part's first window and its windows
    PartView P;
    const T *vals, *in;
    T *out, *mk, *z;
    T small;
    SyncFree *sf;
    unsigned long long limit;
    template <bool BWD>
    __device__ __forceinline__ int at(int j) const {   // packed window of the j-th in sweep order
        j = min(j, nw - 1);
        return BWD ? w0 + nw - 1 - j : w0 + j;
    }
};

// A window's inputs from other parts: their codes (a code < 0 names a packed slot of
// another part) and the bits found there so far.
template <class T, int W>
struct PartIn {
    int code[W];
    typename SfBits<T>::U pb[W];
};

// polls of the inputs that are not there yet
template <class T, int W>
__device__ __forceinline__ void part_poll(PartIn<T, W> &I, const T *out) {
#pragma unroll
    for (int k = 0; k < W; ++k)
        if (I.code[k] < 0 && I.pb[k] == SfBits<T>::kMark) I.pb[k] = sf_load_bits(out + (I.code[k] & 0x7fffffff));
}

template <class T, int W>
__device__ __forceinline__ bool part_missing(const PartIn<T, W> &I) {
    bool miss = false;
#pragma unroll
    for (int k = 0; k < W; ++k) miss |= I.code[k] < 0 && I.pb[k] == SfBits<T>::kMark;
    return __any(miss);
}

// waits until the chain has finished window j of the part; false: gave up
template <class T, int W>
__device__ __forceinline__ bool part_finished(const PartLds<T, W> &L, int j) {
    while (lds_get(&L.progress) <= j)
        if (lds_get(&L.give_up)) return false;
    lds_order();
    return true;
}

// The backward sweep's value of this lane's row in a finished window, while the ring holds
// it: a window's slots are written again kRing / 64 windows later.
template <class T, int W, bool BWD>
__device__ __forceinline__ T part_result(const PartRun<T> &R, const PartLds<T, W> &L, int j) {
    const int q = R.template at<BWD>(j) * 64 + (int)(threadIdx.x & 63);
    return BWD ? L.x[q & (kRing - 1)] : T(0);
}

// the results of a finished window that need not be early
template <class T, bool BWD>
__device__ __forceinline__ void part_retire(const PartRun<T> &R, int j, int row, T result) {
    const int q = R.template at<BWD>(j) * 64 + (int)(threadIdx.x & 63);
    // the other direction's output takes its mark for the next sweep: the forward sweep
    // marks the backward one's slots, the backward sweep those it has read
    sf_mark(R.mk + q);
    if (BWD) R.z[row] = result;
}

template <class T, int W>
__device__ __forceinline__ void stage_put(typename PartLds<T, W>::Slot &s, int lane, const int *ints, const T *vals) {
    using L = PartLds<T, W>;
#pragma unroll
    for (int b = 0; b < L::kIntVecs; ++b)
        s.ints[b][lane] = make_int4(ints[4 * b], ints[4 * b + 1], ints[4 * b + 2], ints[4 * b + 3]);
#pragma unroll
    for (int t = 0; t < L::kIntRest; ++t) s.int1[t][lane] = ints[4 * L::kIntVecs + t];
#pragma unroll
    for (int b = 0; b < L::kValVecs; ++b) {
        typename L::vec v;
#pragma unroll
        for (int t = 0; t < L::V; ++t) v[t] = vals[L::V * b + t];
        s.vals[b][lane] = v;
    }
#pragma unroll
    for (int t = 0; t < L::kValRest; ++t) s.val1[t][lane] = vals[L::V * L::kValVecs + t];
}

template <class T, int W, bool BWD>
__device__ __forceinline__ void part_feed(const PartRun<T> &R, PartLds<T, W> &L, int feeder) {
    using S = PartShape<W>;
    using U = typename SfBits<T>::U;
    constexpr int B = S::kBatch, K = S::kStage;
    const int lane = threadIdx.x & 63;
    PartRow<T, W> cur[B], nxt[B];
    int row[B];            // rows of the batch before the current one
    int before = -1;       // first window of that batch
    auto load = [&](PartRow<T, W> &o, int j) {
        const size_t q = (size_t)R.template at<BWD>(j) * 64 + lane;
        load_packed<int, W>(o.code, R.P.codes, R.P.npk, q);
        load_packed<T, W>(o.val, R.vals, R.P.npk, q);
        o.step = R.P.step[q];
    };
    int j0 = feeder * B;
#pragma unroll
    for (int u = 0; u < B; ++u) {
        load(cur[u], j0 + u);
        row[u] = 0;
    }
    for (; j0 < R.nw; j0 += K) {
        T rhs[B];
#pragma unroll
        for (int u = 0; u < B; ++u)
            rhs[u] = BWD ? R.in[(size_t)R.template at<BWD>(j0 + u) * 64 + lane] : R.in[cur[u].code[W]];
#pragma unroll
        for (int u = 0; u < B; ++u) load(nxt[u], j0 + K + u);
#pragma unroll
        for (int u = 0; u < B; ++u) {
            const int j = j0 + u;
            T vals[W + 2];
#pragma unroll
            for (int k = 0; k < W; ++k) vals[k] = cur[u].val[k];
            vals[W] = cur[u].val[W];
            vals[W + 1] = BWD ? rhs[u] / (cur[u].val[W] + R.small) : rhs[u];
            // room in the stage
            if (!part_finished(L, j - K)) return;
            // Window j - kStage, which this wave fed too, is finished.  Its values are read
            // before window j is staged: from then on the chain runs on as far as the other
            // feeders have staged, past where the ring holds them.
            const T result = before >= 0 ? part_result<T, W, BWD>(R, L, j - K) : T(0);
            if (j < R.nw) {
                const int slot = j % K;
                const int xbase = kRing + 2 + slot * W * 64 + lane;
                int ints[W + 1];
#pragma unroll
                for (int k = 0; k < W; ++k) {
                    const bool outside = cur[u].code[k] < 0;
                    ints[k] = (int)sizeof(T) * (outside ? xbase + k * 64 : cur[u].code[k]);
                    // the slot's code until the poller puts its value there
                    reinterpret_cast<U *>(L.x)[xbase + k * 64] = (U)(unsigned)cur[u].code[k];
                }
                const int top = __builtin_amdgcn_readlane(cur[u].step, 63);
                ints[W] = (BWD ? top - cur[u].step : cur[u].step) | top << 8;
                stage_put<T, W>(L.stage[slot], lane, ints, vals);
                lds_order();
                lds_set(&L.fed[slot], j + 1);
            }
            if (before >= 0) part_retire<T, BWD>(R, j - K, row[u], result);
        }
        before = j0;
#pragma unroll
        for (int u = 0; u < B; ++u) {
            row[u] = cur[u].code[W];
            cur[u] = nxt[u];
        }
    }
    // the windows of the last round
    if (before < 0) return;
#pragma unroll
    for (int u = 0; u < B; ++u) {
        if (before + u < R.nw) {
            if (!part_finished(L, before + u)) return;
            part_retire<T, BWD>(R, before + u, row[u], part_result<T, W, BWD>(R, L, before + u));
        }
    }
}

// The inputs from other parts, a window per turn of a poller: polled until they are there
// and put where the staged codes point to.  By the first poller alone while the part has
// not begun: a part that waits must not flood the memory system.  The window's operands
// are waited for here (fed), so the chain waits for one flag only.
template <class T, int W>
__device__ __forceinline__ void part_inputs(const PartRun<T> &R, PartLds<T, W> &L, int poller) {
    using U = typename SfBits<T>::U;
    constexpr int K = PartShape<W>::kStage;
    const int lane = threadIdx.x & 63;
    for (int j = poller; j < R.nw; j += PartShape<W>::kPollers) {
        const int slot = j % K, xbase = kRing + 2 + slot * W * 64 + lane;
        while (lds_get(&L.fed[slot]) != j + 1)
            if (lds_get(&L.give_up)) return;
        lds_order();
        PartIn<T, W> in;
#pragma unroll
        for (int k = 0; k < W; ++k) {
            in.code[k] = (int)reinterpret_cast<const U *>(L.x)[xbase + k * 64];
            in.pb[k] = SfBits<T>::kMark;
        }
        if (part_missing<T, W>(in)) {
            unsigned long long t0 = wall_clock64();
            int polls = 0;
            do {
                bool late = false;
                if (j > 0 && lds_get(&L.flag[0]) == 0) {
                    __builtin_amdgcn_s_sleep(1);
                    t0 = wall_clock64();   // the first poller's wait, not this one's
                } else {
                    part_poll<T, W>(in, R.out);
                    if ((++polls & 7) == 0)
                        late = __any(wall_clock64() - t0 > R.limit ||
                                     __hip_atomic_load(&R.sf->abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0);
                }
                if (late || lds_get(&L.give_up)) {
                    if (late) __hip_atomic_store(&R.sf->abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    lds_set(&L.give_up, 1);
                    return;
                }
            } while (part_missing<T, W>(in));
        }
#pragma unroll
        for (int k = 0; k < W; ++k)
            if (in.code[k] < 0) L.x[xbase + k * 64] = __builtin_bit_cast(T, in.pb[k]);
        lds_order();
        lds_set(&L.flag[slot], j + 1);
    }
}

template <class T, int W>
struct PartOps {
    int i[W + 1];
    T v[W + 2];
    __device__ __forceinline__ void read(const typename PartLds<T, W>::Slot &s, int lane) {
        using L = PartLds<T, W>;
#pragma unroll
        for (int b = 0; b < L::kIntVecs; ++b) {
            const int4 q = s.ints[b][lane];
            i[4 * b] = q.x;
            i[4 * b + 1] = q.y;
            i[4 * b + 2] = q.z;
            i[4 * b + 3] = q.w;
        }
#pragma unroll
        for (int t = 0; t < L::kIntRest; ++t) i[4 * L::kIntVecs + t] = s.int1[t][lane];
#pragma unroll
        for (int b = 0; b < L::kValVecs; ++b) {
            const typename L::vec q = s.vals[b][lane];
#pragma unroll
            for (int t = 0; t < L::V; ++t) v[L::V * b + t] = q[t];
        }
#pragma unroll
        for (int t = 0; t < L::kValRest; ++t) v[L::V * L::kValVecs + t] = s.val1[t][lane];
    }
};

template <class T, int W>
__device__ __forceinline__ T part_row(const PartOps<T, W> &o, const T *x) {
    T r = o.v[W + 1];
#pragma unroll
    for (int k = 0; k < W; ++k) r = r - o.v[k] * x[k];
    return r * o.v[W];
}

template <class T, int W>
struct Chain {
    int j, nw;        // the current window and the part's
    int ring;         // ring index of this lane's row
    T *out;           // its output
    bool have;        // the next window's operands are read (or on their way)
};

// One window of the chain, its operands in `o`.  Those of the next one are in `n`
// (c.have) or are waited for here; those of the one after it are read into `n2` if
// the stage holds it, behind the chain's own LDS accesses and a window ahead of their
// use.  false: the part is finished, or gave up.
template <class T, int W, bool BWD, int SLOT>
__device__ __forceinline__ bool part_step(PartLds<T, W> &L, Chain<T, W> &c, const PartOps<T, W> &o, PartOps<T, W> &n,
                                          PartOps<T, W> &n2) {
    constexpr int K = PartShape<W>::kStage, S1 = (SLOT + 1) % K, S2 = (SLOT + 2) % K;
    const int lane = threadIdx.x;
    const char *xs = reinterpret_cast<const char *>(L.x);
    T x[W], v;
#pragma unroll
    for (int k = 0; k < W; ++k) x[k] = *reinterpret_cast<const T *>(xs + o.i[k]);
    const int seen = __hip_atomic_load(&L.flag[S2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    const int top = __builtin_amdgcn_readfirstlane(o.i[W]) >> 8;
    if (top == 0) {
        v = part_row<T, W>(o, x);
        L.x[c.ring] = v;
    } else {   // levels of the window in turn, each reading what the ones before it wrote
        const int step = o.i[W] & 255;
        v = T(0);
        for (int st = 0; st <= top; ++st) {
            lds_order();
            if (step == st) {
#pragma unroll
                for (int k = 0; k < W; ++k) x[k] = *reinterpret_cast<const T *>(xs + o.i[k]);
                v = part_row<T, W>(o, x);
                L.x[c.ring] = v;
            }
        }
    }
    lds_order();
    sf_store(c.out, v);
    lds_set(&L.progress, c.j + 1);
    if (c.j + 1 >= c.nw) return false;
    if (!c.have) {
        while (lds_get(&L.flag[S1]) != c.j + 2)
            if (lds_get(&L.give_up)) return false;
        lds_order();
        n.read(L.stage[S1], lane);
    }
    c.have = __builtin_amdgcn_readfirstlane(seen) == c.j + 3;
    lds_order();
    if (c.have) n2.read(L.stage[S2], lane);
    c.j += 1;
    c.ring = (c.ring + (BWD ? -64 : 64)) & (kRing - 1);
    c.out += BWD ? -64 : 64;
    return true;
}

template <class T, int W, bool BWD, int SLOT>
__device__ __forceinline__ bool part_round(PartLds<T, W> &L, Chain<T, W> &c, PartOps<T, W> (&o)[3]) {
    if constexpr (SLOT == PartShape<W>::kStage) {
        return true;
    } else {
        if (!part_step<T, W, BWD, SLOT>(L, c, o[SLOT % 3], o[(SLOT + 1) % 3], o[(SLOT + 2) % 3])) return false;
        return part_round<T, W, BWD, SLOT + 1>(L, c, o);
    }
}

template <class T, int W, bool BWD>
__device__ __forceinline__ void part_chain(const PartRun<T> &R, PartLds<T, W> &L) {
    static_assert(PartShape<W>::kStage % 3 == 0, "three sets of operands in rotation");
    const int q = R.template at<BWD>(0) * 64 + (int)threadIdx.x;
    Chain<T, W> c;
    c.j = 0;
    c.nw = R.nw;
    c.ring = q & (kRing - 1);
    c.out = R.out + q;
    c.have = false;
    PartOps<T, W> o[3];
    while (lds_get(&L.flag[0]) != 1)
        if (lds_get(&L.give_up)) return;
    lds_order();
    o[0].read(L.stage[0], threadIdx.x);
    while (part_round<T, W, BWD, 0>(L, c, o)) {
    }
}

// One sweep over all parts.  The output (packed order) is full of marks on entry; a
// value is published with one coherent store, which is also its "ready" signal.  `in`
// is the right-hand side in row order (forward) or the forward sweep's packed output
// (backward), which takes its marks again; `mk` the array to mark; `z` the backward
// sweep's result in row order.  A row's step in its window is the rank of its level
// there, so its inputs inside the part are in LDS by then.  A row's value is formed as
// k_sweep_syncfree forms it: padding entries subtract 0 * 0, which leaves every value
// as it is.
template <class T, int W, bool BWD>
__global__ __launch_bounds__(PartShape<W>::kBlock) void k_sweep_parts(int nparts, PartView P, const int *__restrict__ win_ptr,
                                                            const T *__restrict__ vals, const T *in, T small, T *out,
                                                            T *mk, T *z, SyncFree *sf,
                                                            const Scalars *__restrict__ sc) {
    __shared__ PartLds<T, W> L;
    if (sc && sc->done) return;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    PartRun<T> R;
    R.P = P;
    R.vals = vals;
    R.in = in;
    R.out = out;
    R.mk = mk;
    R.z = z;
    R.small = small;
    R.sf = sf;
    R.limit = sf_wait_ticks(sf, sf->rate_khz);
    if (threadIdx.x == 0) {
        L.x[kRing] = T(0);
        L.give_up = 0;
    }
    for (;;) {
        if (threadIdx.x == 0) {
            L.ticket = (int)__hip_atomic_fetch_add(&sf->ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            L.progress = 0;
        }
        if (threadIdx.x < (unsigned)PartShape<W>::kStage) {
            L.fed[threadIdx.x] = 0;
            L.flag[threadIdx.x] = 0;
        }
        __syncthreads();
        const int t = __builtin_amdgcn_readfirstlane(L.ticket);
        if ((unsigned)t >= (unsigned)nparts) break;
        const int part = BWD ? nparts - 1 - t : t;
        R.w0 = win_ptr[part];
        R.nw = win_ptr[part + 1] - R.w0;
        if (wave == 0)
            part_chain<T, W, BWD>(R, L);
        else if (wave <= PartShape<W>::kPollers)
            part_inputs<T, W>(R, L, wave - 1);
        else
            part_feed<T, W, BWD>(R, L, wave - 1 - PartShape<W>::kPollers);
        __syncthreads();
        if (L.give_up) break;
    }
    if (threadIdx.x == 0) {
        const unsigned f = __hip_atomic_fetch_add(&sf->fin, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        if (f == gridDim.x - 1) {
            __hip_atomic_store(&sf->ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&sf->fin, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// ----------------------------------------------------------------- analysis

// Lines of rows (their first rows) and the part of each, parts numbered in an order
// in which every part's inputs come first; false when the numbering has no such runs.
struct PartLines {
    std::vector<int> start, part;
    int nparts = 0;
};

void consecutive_parts(int n, PartLines &L) {
    L.nparts = (n + kPartRows - 1) / kPartRows;
    L.start.resize(L.nparts);
    L.part.resize(L.nparts);
    for (int p = 0; p < L.nparts; ++p) {
        L.start[p] = p * kPartRows;
        L.part[p] = p;
    }
}

std::vector<unsigned char> run_links(fc_context *ctx, const Structure &st, int m, const std::vector<int> *start) {
    hipStream_t s = ctx->stream;
    DevBuf flag((size_t)m), ds;
    if (start) {
        ds.alloc(sizeof(int) * (size_t)m);
        h2d(ds.get(), start->data(), sizeof(int) * (size_t)m, s);
    }
    k_run_links<<<grid_for(m), kBlock, 0, s>>>(m, start ? ds.as<int>() : nullptr, st.ioffset.as<int>(),
                                               st.ja.as<int>(), st.diag.as<int>(), flag.as<unsigned char>());
    FC_HIP_CHECK(hipGetLastError());
    std::vector<unsigned char> h((size_t)m);
    d2h(h.data(), flag.get(), (size_t)m, s);
    return h;
}

// Pencils of 64 lines.  A line is a run of rows each reading the one before it; a
// sheet a run of lines whose first rows do; a stack a run of sheets of as many lines
// whose first rows do.  Parts are numbered stack by stack, within a stack along the
// diagonals of (line block, sheet block): the order in which the sweep reaches them.
bool pencil_parts(fc_context *ctx, const Structure &st, PartLines &L) {
    const int n = st.n;
    const std::vector<unsigned char> linked = run_links(ctx, st, n, nullptr);
    for (int r = 0; r < n; ++r)
        if (!linked[r]) L.start.push_back(r);
    const int lines = (int)L.start.size();
    if ((long long)lines * 4 > n) return false;   // runs of fewer than four rows: not a structured numbering
    const std::vector<unsigned char> lf = run_links(ctx, st, lines, &L.start);
    std::vector<int> sheet;   // first line of every sheet
    for (int l = 0; l < lines; ++l)
        if (!lf[l]) sheet.push_back(l);
    const int sheets = (int)sheet.size();
    std::vector<int> first(sheets);
    for (int k = 0; k < sheets; ++k) first[k] = L.start[sheet[k]];
    const std::vector<unsigned char> sf = run_links(ctx, st, sheets, &first);
    auto lines_of = [&](int k) { return (k + 1 < sheets ? sheet[k + 1] : lines) - sheet[k]; };
    L.part.assign(lines, 0);
    L.nparts = 0;
    for (int s0 = 0; s0 < sheets;) {
        const int J = lines_of(s0);
        int s1 = s0 + 1;
        while (s1 < sheets && sf[s1] && lines_of(s1) == J) ++s1;
        const int K = s1 - s0;
        int bk = std::min(8, K), bj = std::min(J, 64 / bk);
        bk = std::min(K, 64 / bj);
        const int nj = (J + bj - 1) / bj, nk = (K + bk - 1) / bk;
        std::vector<int> id((size_t)nj * nk);
        int next = L.nparts;
        for (int d = 0; d < nj + nk - 1; ++d)
            for (int b = std::max(0, d - nj + 1); b < std::min(nk, d + 1); ++b) id[(size_t)b * nj + (d - b)] = next++;
        for (int k = 0; k < K; ++k)
            for (int j = 0; j < J; ++j)   // blocks of nearly equal size
                L.part[sheet[s0 + k] + j] = id[(size_t)((long long)k * nk / K) * nj + (size_t)((long long)j * nj / J)];
        L.nparts = next;
        s0 = s1;
    }
    // many small blocks (an unstructured numbering with accidental runs): no gain
    return (long long)L.nparts * 512 <= (long long)n + 64 * 512;
}

// The packed order: parts in their order, a part's rows by (level, row) in windows of
// 64.  A window takes whole levels while they fit; a level of more than 64 rows fills
// windows of its own.  The backward sweep walks the same windows the other way round.
bool pack_part_order(fc_context *ctx, Structure &st, const PartLines &L) {
    hipStream_t s = ctx->stream;
    const int n = st.n, np = L.nparts;
    std::vector<int> part((size_t)n), byrow((size_t)n), order((size_t)n), lev((size_t)n);
    for (size_t l = 0; l < L.start.size(); ++l) {
        const int e = l + 1 < L.start.size() ? L.start[l + 1] : n;
        std::fill(part.begin() + L.start[l], part.begin() + e, L.part[l]);
    }
    d2h(byrow.data(), st.rows_f.get(), sizeof(int) * (size_t)n, s);
    std::vector<int> at((size_t)np + 1, 0);
    for (int r = 0; r < n; ++r) at[part[r] + 1] += 1;
    for (int p = 0; p < np; ++p) at[p + 1] += at[p];
    const std::vector<int> begin(at);
    for (int v = 0; v < st.nlev_f; ++v)
        for (int p = st.lvl_f[v]; p < st.lvl_f[v + 1]; ++p) {
            const int o = at[part[byrow[p]]]++;
            order[o] = byrow[p];
            lev[o] = v;
        }
    std::vector<int> rows, win((size_t)np + 1, 0), win_part;
    std::vector<unsigned char> step;
    rows.reserve((size_t)n + (size_t)n / 8);
    step.reserve((size_t)n + (size_t)n / 8);
    int used = 64, rank = 0;   // lanes of the open window, rank of its last level
    auto close = [&]() {
        while (used < 64) {
            rows.push_back(rows.back());
            step.push_back(step.back());
            ++used;
        }
    };
    for (int p = 0; p < np; ++p) {
        for (int b = begin[p]; b < begin[p + 1];) {
            int e = b + 1;
            while (e < begin[p + 1] && lev[e] == lev[b]) ++e;
            if (used + (e - b) > 64) close();
            else ++rank;
            for (; b < e; ++b) {
                if (used == 64) {
                    used = 0;
                    rank = 0;
                    win_part.push_back(p);
                }
                rows.push_back(order[b]);
                step.push_back((unsigned char)rank);
                ++used;
            }
        }
        close();
        win[p + 1] = (int)win_part.size();
    }
    if (rows.size() > (size_t)0x7fffffc0) return false;
    const int npk = (int)rows.size();
    st.pt_npk = npk;
    st.pt_nparts = np;
    st.pt_rows.alloc(sizeof(int) * (size_t)npk);
    h2d(st.pt_rows.get(), rows.data(), sizeof(int) * (size_t)npk, s);
    st.pt_step.alloc((size_t)npk);
    h2d(st.pt_step.get(), step.data(), (size_t)npk, s);
    st.pt_win.alloc(sizeof(int) * win.size());
    h2d(st.pt_win.get(), win.data(), sizeof(int) * win.size(), s);
    DevBuf wp(sizeof(int) * win_part.size()), slot(sizeof(int) * (size_t)n), cnt(sizeof(unsigned long long) * 4),
        err(sizeof(int));
    h2d(wp.get(), win_part.data(), sizeof(int) * win_part.size(), s);
    FC_HIP_CHECK(hipMemsetAsync(cnt.get(), 0, sizeof(unsigned long long) * 4, s));
    FC_HIP_CHECK(hipMemsetAsync(err.get(), 0, sizeof(int), s));
    k_part_slots<<<grid_for(npk), kBlock, 0, s>>>(npk, st.pt_rows.as<int>(), slot.as<int>());
    for (int upper = 0; upper < 2; ++upper) {
        const int width = upper ? st.ell_b : st.ell_f;
        DevBuf &codes = upper ? st.pt_codes_b : st.pt_codes_f;
        codes.alloc(sizeof(int) * (size_t)(width + 1) * npk);
        k_part_codes<<<grid_for(npk), kBlock, 0, s>>>(npk, width, upper != 0, st.pt_rows.as<int>(), slot.as<int>(),
                                                      wp.as<int>(), st.pt_step.as<unsigned char>(),
                                                      st.ioffset.as<int>(), st.ja.as<int>(), st.diag.as<int>(),
                                                      codes.as<int>(), cnt.as<unsigned long long>() + 2 * upper,
                                                      err.as<int>());
    }
    FC_HIP_CHECK(hipGetLastError());
    unsigned long long c[4];
    int bad = 0;
    d2h(c, cnt.get(), sizeof c, s);
    d2h(&bad, err.get(), sizeof bad, s);
    st.int_frac_f = c[1] ? (double)c[0] / (double)c[1] : 0.0;
    st.int_frac_b = c[3] ? (double)c[2] / (double)c[3] : 0.0;
    return bad == 0;
}

template <class T, int WF, int WB>
void lu_parts_w(hipStream_t s, const Structure &st, const PackedFactor<T> &pf, T small, const T *rhs, T *w,
                const Scalars *sc, const SweepCfg &cfg) {
    T *tmp = static_cast<T *>(cfg.tmp), *zp = static_cast<T *>(cfg.zp);
    const int np = st.pt_nparts;
    const int waves = std::max(1, std::min(cfg.waves, np));
    const PartView F{st.pt_npk, st.pt_codes_f.as<int>(), st.pt_step.as<unsigned char>()};
    const PartView B{st.pt_npk, st.pt_codes_b.as<int>(), st.pt_step.as<unsigned char>()};
    const int *win = st.pt_win.as<int>();
    k_sweep_parts<T, WF, false><<<waves, PartShape<WF>::kBlock, 0, s>>>(np, F, win, pf.af, rhs, small, tmp, zp, nullptr, cfg.sf, sc);
    k_sweep_parts<T, WB, true><<<waves, PartShape<WB>::kBlock, 0, s>>>(np, B, win, pf.ab, tmp, small, zp, tmp, w, cfg.sf, sc);
}

template <class T, int WF>
void lu_parts_b(hipStream_t s, const Structure &st, const PackedFactor<T> &pf, T small, const T *rhs, T *w,
                const Scalars *sc, const SweepCfg &cfg) {
    switch (st.ell_b) {
    case 3: lu_parts_w<T, WF, 3>(s, st, pf, small, rhs, w, sc, cfg); break;
    case 4: lu_parts_w<T, WF, 4>(s, st, pf, small, rhs, w, sc, cfg); break;
    default: lu_parts_w<T, WF, 8>(s, st, pf, small, rhs, w, sc, cfg); break;
    }
}

template <class T>
void lu_parts_t(hipStream_t s, const Structure &st, const PackedFactor<T> &pf, T small, const T *rhs, T *w,
                const Scalars *sc, const SweepCfg &cfg) {
    FC_REQUIRE(part_sweeps(st) && cfg.tmp && cfg.zp && cfg.sf, FC_ERR_ARGUMENT, "part-wise sweeps not set up");
    switch (st.ell_f) {
    case 3: lu_parts_b<T, 3>(s, st, pf, small, rhs, w, sc, cfg); break;
    case 4: lu_parts_b<T, 4>(s, st, pf, small, rhs, w, sc, cfg); break;
    default: lu_parts_b<T, 8>(s, st, pf, small, rhs, w, sc, cfg); break;
    }
    FC_HIP_CHECK(hipGetLastError());
}

template <class T>
void pack_parts_t(hipStream_t s, const Structure &st, const T *a, const T *d, T *af, T *ab, T *tmp) {
    FC_REQUIRE(st.parts && packed_sweeps(st), FC_ERR_ARGUMENT, "structure has no part-wise sweeps");
    const int npk = st.pt_npk;
    k_part_vals<T><<<grid_for(npk), kBlock, 0, s>>>(npk, st.ell_f, false, st.pt_rows.as<int>(), st.ioffset.as<int>(),
                                                    st.diag.as<int>(), a, d, af);
    k_part_vals<T><<<grid_for(npk), kBlock, 0, s>>>(npk, st.ell_b, true, st.pt_rows.as<int>(), st.ioffset.as<int>(),
                                                    st.diag.as<int>(), a, d, ab);
    k_part_mark<T><<<grid_for(npk), kBlock, 0, s>>>(npk, tmp);
    FC_HIP_CHECK(hipGetLastError());
}

}  // namespace

void analyse_parts(fc_context *ctx, Structure &st) {
    st.parts = false;
    auto compiled = [](int w) { return w == 3 || w == 4 || w == 8; };
    if (!compiled(st.ell_f) || !compiled(st.ell_b)) return;
    PartLines pencils;
    if (pencil_parts(ctx, st, pencils) && pack_part_order(ctx, st, pencils)) {
        st.parts = true;
        return;
    }
    PartLines runs;
    consecutive_parts(st.n, runs);
    st.parts = pack_part_order(ctx, st, runs);
}

size_t part_factor_count(const Structure &st, bool upper) {
    return (size_t)((upper ? st.ell_b : st.ell_f) + 1) * (size_t)st.pt_npk;
}

void pack_factor_parts64(hipStream_t s, const Structure &st, const double *a, const double *d, double *af, double *ab,
                         double *tmp) {
    pack_parts_t<double>(s, st, a, d, af, ab, tmp);
}

void pack_factor_parts32(hipStream_t s, const Structure &st, const float *a, const float *d, float *af, float *ab,
                         float *tmp) {
    pack_parts_t<float>(s, st, a, d, af, ab, tmp);
}

void lu_parts64(hipStream_t s, const Structure &st, const PackedFactor<double> &pf, double small, const double *rhs,
                double *w, const Scalars *sc, const SweepCfg &cfg) {
    lu_parts_t<double>(s, st, pf, small, rhs, w, sc, cfg);
}

void lu_parts32(hipStream_t s, const Structure &st, const PackedFactor<float> &pf, float small, const float *rhs,
                float *w, const Scalars *sc, const SweepCfg &cfg) {
    lu_parts_t<float>(s, st, pf, small, rhs, w, sc, cfg);
}

}  // namespace fcap
