// Reads from LDS with hand-counted waits, for kernels that have direct-to-LDS loads under way: the compiler cannot tell the
// two apart and waits for every read it has issued (lgkmcnt(0)) ahead of each use.  A register is not touched between its
// read and lds_arrived, which the compiler does not know: no such read may be under way where the code branches (it may copy
// one there).  The build refuses these kernels if they spill (build.py), and if their generated code touches such a register
// ahead of its wait (inflight.py).
#pragma once

#include "common.h"

#include <type_traits>

namespace {

template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>());
        static_for<I + 1, N>(f);
    }
}

// 16, 8 or 2 bytes at `at` + OFF
template <typename T, int OFF>
__device__ __forceinline__ T lds_read(uint32_t at) {
    T v;
    if constexpr (sizeof(T) == 16)
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(at), "n"(OFF));
    else if constexpr (sizeof(T) == 8)
        asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(v) : "v"(at), "n"(OFF));
    else
        asm volatile("ds_read_u16 %0, %1 offset:%2" : "=v"(v) : "v"(at), "n"(OFF));
    return v;
}
// v has arrived, with at most LATER of the reads issued behind it still under way
template <int LATER, typename T>
__device__ __forceinline__ void lds_arrived(T &v) {
    asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(v) : "n"(LATER < 15 ? LATER : 15));
}

}  // namespace
