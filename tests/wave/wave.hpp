// A wave of 64 lanes on the CPU, for tests of the library's device functions as they
// stand: include this before a HIP source, compiled by the host compiler.  Each lane is a
// coroutine that runs from one cross-lane operation to the next; at such an operation
// every lane still running leaves its value, and all go on with what the others left
// (run_wave).  Memory is plain host memory, so a test can put its arrays at the end of
// mapped pages or check indices.
#pragma once

#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime.h>
#undef hipLaunchKernelGGL
#define hipLaunchKernelGGL(...) ((void)0)  // entry points are parsed, kernels never launched
#undef __shared__
#define __shared__ static
#undef __align__
#define __align__(n) __attribute__((aligned(n)))
#undef __launch_bounds__
#define __launch_bounds__(...)

#include <ucontext.h>

#include <algorithm>
#include <bit>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <vector>

namespace wave {
constexpr int kLanes = 64;
constexpr size_t kStack = 256 << 10;

inline int g_lane = 0;
inline int g_wave = 0;  // the wave's place in its workgroup
inline uint64_t g_slot[2][kLanes], g_here[2];
inline int g_round = 0;
inline ucontext_t g_main, g_ctx[kLanes];
inline bool g_done[kLanes];
inline std::function<void(int)>* g_body;

inline void entry() {
    const int lane = g_lane;
    (*g_body)(lane);
    g_done[lane] = true;
    swapcontext(&g_ctx[lane], &g_main);
}

// Leaves v and waits for the other lanes; afterwards got(l) is lane l's value, `mask`
// the lanes that took part.
struct Exchange {
    const uint64_t* slot;
    uint64_t mask;
    uint64_t got(int l) const { return slot[l & 63]; }
};
inline Exchange exchange(uint64_t v) {
    const int lane = g_lane, at = g_round & 1;
    g_slot[at][lane] = v;
    g_here[at] |= 1ull << lane;
    swapcontext(&g_ctx[lane], &g_main);
    return {g_slot[at], g_here[at]};
}

// Runs body(lane) on the 64 lanes of one wave.
inline void run_wave(std::function<void(int)> body) {
    static std::vector<char> stacks(kLanes * kStack);
    g_body = &body;
    g_round = 0;
    g_here[0] = g_here[1] = 0;
    for (int l = 0; l < kLanes; ++l) {
        g_done[l] = false;
        getcontext(&g_ctx[l]);
        g_ctx[l].uc_stack.ss_sp = &stacks[l * kStack];
        g_ctx[l].uc_stack.ss_size = kStack;
        g_ctx[l].uc_link = nullptr;
        makecontext(&g_ctx[l], entry, 0);
    }
    for (bool live = true; live; ++g_round) {
        live = false;
        g_here[g_round & 1] = 0;
        for (g_lane = 0; g_lane < kLanes; ++g_lane)
            if (!g_done[g_lane]) {
                swapcontext(&g_main, &g_ctx[g_lane]);
                live = true;
            }
    }
}

template <typename T>
inline uint64_t bits(T v) {
    uint64_t u = 0;
    std::memcpy(&u, &v, sizeof(T));
    return u;
}
template <typename T>
inline T value(uint64_t u) {
    T v;
    std::memcpy(&v, &u, sizeof(T));
    return v;
}
}  // namespace wave

// ------------------------------------------------ the device functions the sources use
using std::max;
using std::min;
inline uint3 wave_thread() { return {(unsigned)(64 * wave::g_wave + wave::g_lane), 0, 0}; }
#define threadIdx wave_thread()
inline uint3 blockIdx;
inline dim3 blockDim(wave::kLanes), gridDim;
inline int __lane_id() { return wave::g_lane; }
inline int __popcll(uint64_t m) { return std::popcount(m); }
inline float __int_as_float(int v) { return std::bit_cast<float>(v); }
inline int __float_as_int(float v) { return std::bit_cast<int>(v); }
inline float __uint_as_float(uint32_t v) { return std::bit_cast<float>(v); }
inline uint32_t __float_as_uint(float v) { return std::bit_cast<uint32_t>(v); }
inline float __fadd_rn(float a, float b) { return a + b; }
inline float __fmul_rn(float a, float b) { return a * b; }
inline uint64_t __ballot(bool p) {
    const auto x = wave::exchange(p);
    uint64_t m = 0;
    for (int l = 0; l < wave::kLanes; ++l) m |= (x.mask >> l & 1) && x.got(l) ? 1ull << l : 0;
    return m;
}
template <typename T>
inline T __shfl(T v, int src, int width = 64) {
    const int me = wave::g_lane;
    return wave::value<T>(wave::exchange(wave::bits(v)).got((me & ~(width - 1)) + (src & (width - 1))));
}
template <typename T>
inline T __shfl_xor(T v, int m, int width = 64) {
    const int me = wave::g_lane, src = me ^ m;
    const auto x = wave::exchange(wave::bits(v));
    return wave::value<T>(x.got((src & ~(width - 1)) == (me & ~(width - 1)) ? src : me));
}
template <typename T>
inline T __shfl_up(T v, int d, int width = 64) {
    const int me = wave::g_lane;
    const auto x = wave::exchange(wave::bits(v));
    return wave::value<T>(x.got((me & (width - 1)) >= d ? me - d : me));
}
template <typename T>
inline T __shfl_down(T v, int d, int width = 64) {
    const int me = wave::g_lane;
    const auto x = wave::exchange(wave::bits(v));
    return wave::value<T>(x.got((me & (width - 1)) + d < width ? me + d : me));
}
inline int wave_readlane(int v, int lane) { return wave::value<int>(wave::exchange(wave::bits(v)).got(lane)); }
inline int wave_readfirstlane(int v) {
    const auto x = wave::exchange(wave::bits(v));
    return wave::value<int>(x.got(std::countr_zero(x.mask)));
}
// row_ror:n of a DPP row of 16 lanes (control 0x120 + n), all lanes taking part
inline int wave_dpp(int v, int ctrl) {
    if ((ctrl & 0x1f0) != 0x120) std::abort();
    const int me = wave::g_lane, n = ctrl & 15;
    return wave::value<int>(wave::exchange(wave::bits(v)).got((me & ~15) | ((me - n) & 15)));
}
inline void wave_sync() { wave::exchange(0); }
struct WavePair {
    uint32_t a[2];
    uint32_t operator[](int i) const { return a[i]; }
};
struct WaveFloats {
    float a[2];
    float operator[](int i) const { return a[i]; }
};
#define __builtin_amdgcn_readfirstlane(v) wave_readfirstlane(v)
#define __builtin_amdgcn_readlane(v, l) wave_readlane(v, l)
#define __builtin_amdgcn_update_dpp(o, v, c, rm, bm, bc) wave_dpp(v, c)
#define __builtin_amdgcn_fence(...) ((void)0)
#define __builtin_amdgcn_wave_barrier() wave_sync()
#define __builtin_amdgcn_s_setprio(p) ((void)0)
#define __builtin_amdgcn_sbfe(v, at, n) ((int)((uint32_t)(v) << (32 - (at) - (n))) >> (32 - (n)))
#define __builtin_nontemporal_load(p) (*(p))
#define __builtin_nontemporal_store(v, p) ((void)(*(p) = (v)))
// Waves of a workgroup run one after the other, if a test runs them: what one leaves in LDS
// before a barrier the others do not see.
inline void __syncthreads() { wave_sync(); }
// (not emulated, parsed only)
template <typename T>
inline T atomicAdd(T*, T) { std::abort(); }
template <typename T>
inline T atomicMax(T*, T) { std::abort(); }
template <typename T>
inline T atomicOr(T*, T) { std::abort(); }
template <typename T>
inline T atomicCAS(T*, T, T) { std::abort(); }
inline uint32_t __umulhi(uint32_t a, uint32_t b) { return (uint32_t)((uint64_t)a * b >> 32); }
#define __builtin_amdgcn_permlane32_swap(...) (WavePair{})
#define __builtin_amdgcn_cvt_pk_f32_fp8(...) (WaveFloats{})
