// Workgroups of a HIP kernel on the CPU, for tests of what waves may do to each other.
//
// Every lane is a fiber.  A wave's lanes meet at the wave-wide operations (votes, shuffles,
// first-lane reads, sleeps, workgroup-scope stores, barriers), and between two of them its
// lanes run one after the other.  After each such meeting the scheduler chooses the next
// wave at random, of any resident workgroup, and may leave one aside for a long time
// (`freeze`): every order of the waves' steps that the hardware may take, the unlikely ones
// made likely.  LDS starts as garbage; a wave that has returned no longer counts in
// barriers.  wall_clock64() counts the scheduler's steps.  Memory is sequentially
// consistent here: what a missing fence would do is not seen.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <memory>
#include <random>
#include <vector>

#include <sys/mman.h>

extern "C" void emu_switch(void **save, void *to);
asm(R"(
.text
.globl emu_switch
.type emu_switch,@function
emu_switch:
    pushq %rbp
    pushq %rbx
    pushq %r12
    pushq %r13
    pushq %r14
    pushq %r15
    movq %rsp, (%rdi)
    movq %rsi, %rsp
    popq %r15
    popq %r14
    popq %r13
    popq %r12
    popq %rbx
    popq %rbp
    ret
)");
extern char __start_emu_lds[] __attribute__((weak));
extern char __stop_emu_lds[] __attribute__((weak));

namespace emu {

struct Dim { unsigned x; };
enum Op : int { kNone, kPoint, kStore, kValue, kBarrier };

struct Wave;
struct Lane {
    void *sp = nullptr;
    char *stack = nullptr;
    Wave *wave = nullptr;
    unsigned tid = 0;
    int lane = 0, op = kNone;
    unsigned ops = 0;
    bool ended = false;
};
struct Block;
struct Wave {
    Block *block = nullptr;
    std::vector<Lane> lanes;
    bool ended = false, barrier = false;
    uint64_t ex[2][64], with[2] = {0, 0};   // values brought to an operation, and by which lanes
    unsigned op_of[2] = {~0u, ~0u};
    long long frozen = 0;   // left aside until this step
};
struct Block {
    unsigned id = 0;
    std::vector<Wave> waves;
    std::vector<char> lds;
    bool ended = false;
};

struct Policy {
    unsigned seed = 1;
    double freeze = 0.0;           // chance that a wave is left aside after a step (one in three starts late),
    double freeze_store = 0.0;     // and after a workgroup-scope store (a flag just set)
    int freeze_steps = 0;          // for at most so many steps
    std::vector<unsigned> order;   // workgroups in the order in which they become resident
    unsigned resident = ~0u;       // at once
    long long max_steps = 200000000;
    std::function<void(long long)> each_step;
};

inline Lane *cur = nullptr;
inline void *sched_sp = nullptr;
inline const std::function<void()> *body = nullptr;
inline unsigned grid_size = 0, block_size = 0;
inline long long clock_steps = 0;

inline void meet(int op) {
    Lane *l = cur;
    l->op = op;
    emu_switch(&l->sp, sched_sp);
    cur = l;
}
inline void lane_main() {
    (*body)();
    cur->ended = true;
    Lane *l = cur;
    emu_switch(&l->sp, sched_sp);
    std::abort();
}
inline void die(const char *what) {
    std::fprintf(stderr, "wave emulation: %s\n", what);
    std::abort();
}

// the values the wave's live lanes bring to a wave-wide operation
template <class T>
struct Brought {
    const uint64_t *v;
    uint64_t with;
    bool has(int lane) const { return with >> lane & 1; }
    T at(int lane) const {
        T r;
        std::memcpy(&r, &v[lane & 63], sizeof(T));
        return r;
    }
};
template <class T>
inline Brought<T> bring(T v) {
    static_assert(sizeof(T) <= 8, "");
    Lane *l = cur;
    Wave &w = *l->wave;
    const unsigned set = l->ops & 1;
    if (w.op_of[set] != l->ops) {
        w.op_of[set] = l->ops;
        w.with[set] = 0;
    }
    l->ops += 1;
    w.with[set] |= 1ull << l->lane;
    w.ex[set][l->lane] = 0;
    std::memcpy(&w.ex[set][l->lane], &v, sizeof(T));
    meet(kValue);
    return Brought<T>{w.ex[set], w.with[set]};
}
template <class T>
inline T first(T v) {
    const Brought<T> b = bring(v);
    return b.at(__builtin_ctzll(b.with));
}

// Runs a kernel; false: max_steps ran out
inline bool launch(unsigned grid, unsigned threads, Policy p, const std::function<void()> &f) {
    constexpr size_t kStack = 64 * 1024;
    body = &f;
    grid_size = grid;
    block_size = threads;
    clock_steps = 0;
    std::mt19937 rng(p.seed);
    if (p.order.empty())
        for (unsigned b = 0; b < grid; ++b) p.order.push_back(b);
    const size_t lds = (size_t)(__stop_emu_lds - __start_emu_lds);
    Block *in_lds = nullptr;
    std::vector<std::unique_ptr<Block>> live;
    std::vector<char *> stacks, spare;
    size_t next = 0;
    auto start = [&](unsigned id) {
        auto b = std::make_unique<Block>();
        b->id = id;
        b->lds.resize(lds);
        const float garbage = 1e30f;
        for (size_t i = 0; i + 4 <= lds; i += 4) std::memcpy(&b->lds[i], &garbage, 4);
        b->waves.resize((threads + 63) / 64);
        for (size_t w = 0; w < b->waves.size(); ++w) {
            Wave &wv = b->waves[w];
            wv.block = b.get();
            if (p.freeze > 0 && rng() % 3 == 0) wv.frozen = clock_steps + rng() % (unsigned)p.freeze_steps;
            wv.lanes.resize(std::min(64u, threads - 64 * (unsigned)w));
            for (size_t l = 0; l < wv.lanes.size(); ++l) {
                Lane &ln = wv.lanes[l];
                ln.wave = &wv;
                ln.lane = (int)l;
                ln.tid = (unsigned)(64 * w + l);
                if (spare.empty()) {
                    void *m = mmap(nullptr, kStack, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
                    if (m == MAP_FAILED) die("no memory for a lane's stack");
                    stacks.push_back((char *)m);
                    spare.push_back((char *)m);
                }
                ln.stack = spare.back();
                spare.pop_back();
                void **top = (void **)(ln.stack + kStack - 16);
                *--top = nullptr;                  // return address of lane_main: none
                *--top = (void *)&lane_main;
                for (int r = 0; r < 6; ++r) *--top = nullptr;
                ln.sp = top;
            }
        }
        live.push_back(std::move(b));
    };
    bool ok = true;
    std::vector<Wave *> ready;
    while (true) {
        while (live.size() < p.resident && next < p.order.size()) start(p.order[next++]);
        if (live.empty()) break;
        if (++clock_steps > p.max_steps) {
            ok = false;
            break;
        }
        if (p.each_step) p.each_step(clock_steps);
        ready.clear();
        for (auto &b : live)
            for (Wave &w : b->waves)
                if (!w.ended && !w.barrier && w.frozen <= clock_steps) ready.push_back(&w);
        if (ready.empty()) continue;   // the ones left aside come back
        Wave &w = *ready[rng() % ready.size()];
        if (in_lds != w.block) {
            if (in_lds) std::memcpy(in_lds->lds.data(), __start_emu_lds, lds);
            std::memcpy(__start_emu_lds, w.block->lds.data(), lds);
            in_lds = w.block;
        }
        int op = kNone;
        bool any = false;
        for (Lane &l : w.lanes) {
            if (l.ended) continue;
            cur = &l;
            emu_switch(&sched_sp, l.sp);
            if (l.ended) continue;
            if (any && l.op != op) die("the lanes of a wave met at different operations");
            op = l.op;
            any = true;
        }
        if (!any) w.ended = true;
        else if (op == kBarrier) w.barrier = true;
        if (std::uniform_real_distribution<>(0, 1)(rng) < (op == kStore ? p.freeze_store : p.freeze))
            w.frozen = clock_steps + 1 + (long long)(rng() % (unsigned)p.freeze_steps);
        Block &b = *w.block;
        bool all = true, none = true;
        for (Wave &x : b.waves) {
            all = all && (x.ended || x.barrier);
            none = none && x.ended;
        }
        if (none) {
            in_lds = nullptr;
            for (auto it = live.begin(); it != live.end(); ++it)
                if (it->get() == &b) {
                    for (Wave &x : b.waves)
                        for (Lane &l : x.lanes) spare.push_back(l.stack);
                    live.erase(it);
                    break;
                }
        } else if (all) {
            for (Wave &x : b.waves) x.barrier = false;
        }
    }
    for (char *s : stacks) munmap(s, kStack);
    return ok;
}

template <class T> inline T load(const T *p) { return *const_cast<const volatile T *>(p); }
template <class T, class V> inline void store(T *p, V v, int scope) {
    *const_cast<volatile T *>(p) = (T)v;
    if (scope == 2) meet(kStore);
}
template <class T, class V> inline T add(T *p, V v) {
    const T old = *p;
    *p = old + (T)v;
    return old;
}

template <class T, class V> inline bool cas(T *p, T *expected, V v) {
    if (*p == *expected) {
        *p = (T)v;
        return true;
    }
    *expected = *p;
    return false;
}

}  // namespace emu

struct int4 { int x, y, z, w; };
inline int4 make_int4(int x, int y, int z, int w) { return {x, y, z, w}; }

#define __global__ static
#define __device__
#define __host__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ static __attribute__((section("emu_lds"), aligned(16)))
#define threadIdx (emu::Dim{emu::cur->tid})
#define blockIdx (emu::Dim{emu::cur->wave->block->id})
#define blockDim (emu::Dim{emu::block_size})
#define gridDim (emu::Dim{emu::grid_size})
#define __HIP_MEMORY_SCOPE_AGENT 1
#define __HIP_MEMORY_SCOPE_WORKGROUP 2
#define __hip_atomic_load(p, order, scope) emu::load(p)
#define __hip_atomic_store(p, v, order, scope) emu::store(p, v, scope)
#define __hip_atomic_fetch_add(p, v, order, scope) emu::add(p, v)
#define __hip_atomic_compare_exchange_strong(p, e, v, order, order2, scope) emu::cas(p, e, v)
#define atomicAdd(p, v) emu::add(p, v)
#define atomicOr(p, v) (*(p) |= (v))
#define atomicMax(p, v) (*(p) = std::max(*(p), (v)))
#define __builtin_amdgcn_readfirstlane(v) emu::first(v)
#define __builtin_amdgcn_readlane(v, l) emu::bring(v).at(l)
#define __builtin_amdgcn_s_sleep(n) emu::meet(emu::kPoint)
#define __syncthreads() emu::meet(emu::kBarrier)
#define wall_clock64() ((unsigned long long)emu::clock_steps)

constexpr int kEmuWave = 64;
template <class T> inline T __shfl(T v, int l, int = kEmuWave) { return emu::bring(v).at(l); }
template <class T> inline T __shfl_down(T v, int o, int width = kEmuWave) {
    const int l = emu::cur->lane;
    return emu::bring(v).at((l & (width - 1)) + o < width ? l + o : l);
}
template <class T> inline T __shfl_xor(T v, int o, int = kEmuWave) {
    const int l = emu::cur->lane;
    return emu::bring(v).at(l ^ o);
}
inline bool __any(bool v) {
    const auto b = emu::bring(v);
    for (int l = 0; l < kEmuWave; ++l)
        if (b.has(l) && b.at(l)) return true;
    return false;
}
inline bool __all(bool v) {
    const auto b = emu::bring(v);
    for (int l = 0; l < kEmuWave; ++l)
        if (b.has(l) && !b.at(l)) return false;
    return true;
}
using std::isfinite;
using std::max;
using std::min;
