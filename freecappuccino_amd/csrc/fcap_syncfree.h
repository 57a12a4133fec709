// Device primitives of the dependency-driven sweeps: values published with one
// coherent store, polled until they differ from a mark arithmetic never produces.
#pragma once

#include "fcap_linalg.h"

namespace fcap {

// A wait is bounded in wall-clock time (wall_clock64(), a constant-rate counter), not in
// polls, so the bound does not shrink with a deeper chain or a faster clock: it only ends
// waits that cannot end otherwise.
constexpr unsigned long long kSfWaitUs = 2000000ull;   // 2 s

// the wait limit in wall-clock ticks (sf->wait_us microseconds, 0: kSfWaitUs)
__device__ inline unsigned long long sf_wait_ticks(const SyncFree *sf, unsigned long long rate_khz) {
    const unsigned long long us = sf->wait_us > 0 ? (unsigned long long)sf->wait_us : kSfWaitUs;
    return us * rate_khz / 1000ull + 1ull;
}

template <class T> struct SfBits;
template <> struct SfBits<double> {
    using U = unsigned long long;
    static constexpr U kMark = 0x7FF4DEADBEEF0001ull;   // signalling NaN
};
template <> struct SfBits<float> {
    using U = unsigned;
    static constexpr U kMark = 0x7FA0BEEFu;               // signalling NaN
};

template <class T>
__device__ inline typename SfBits<T>::U sf_load_bits(const T *p) {
    return __hip_atomic_load(reinterpret_cast<const typename SfBits<T>::U *>(p), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
}

// A plain store of the mark, of the array's own type: a sweep marks what it has read through
// that type, and a store of the integer type might be moved before the read.
template <class T>
__device__ inline void sf_mark(T *p) {
    *p = __builtin_bit_cast(T, SfBits<T>::kMark);
}

template <class T>
__device__ inline void sf_store(T *p, T v) {
    using U = typename SfBits<T>::U;
    U b;
    __builtin_memcpy(&b, &v, sizeof(U));
    __hip_atomic_store(reinterpret_cast<U *>(p), b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace fcap
