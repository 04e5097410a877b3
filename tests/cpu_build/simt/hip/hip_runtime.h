// Runs whole HIP kernels on the CPU for the test-suite: a workgroup is a set of fibers in one OS thread, a barrier hands over
// to the next fiber, `__shared__` is thread-local storage (static, and legal behind `extern`).  Translation units that include
// this in the place of the HIP runtime launch through the same hipLaunchKernelGGL lines as on the GPU, so index maps, barriers
// and dispatch can be checked against the oracle, and under AddressSanitizer over buffers of exactly the stated sizes.
//
// Dynamic LDS (`extern __shared__`) needs its definition beside the include; atomics are plain, as one fiber runs at a time.
#pragma once
#include <stddef.h>
#include <stdint.h>
#include <string.h>
#include <sys/mman.h>
#include <ucontext.h>

#include <cstdio>
#include <cstdlib>
#include <functional>
#include <map>
#include <vector>

#define __global__
#define __device__
#define __constant__ static
#define __host__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __align__(n) __attribute__((aligned(n)))
#define __shared__ thread_local
#define ext_vector_type(n) vector_size(4 * (n))                       // 32-bit elements only

struct dim3 {
    unsigned x, y, z;
    dim3(unsigned x_ = 1, unsigned y_ = 1, unsigned z_ = 1) : x(x_), y(y_), z(z_) {}
};
struct alignas(16) ulonglong2 { unsigned long long x, y; };
inline uint64_t __umul64hi(uint64_t a, uint64_t b) { return (uint64_t)((unsigned __int128)a * b >> 64); }
struct alignas(8) uint2 { uint32_t x, y; };
struct alignas(16) uint4 { uint32_t x, y, z, w; };
inline uint4 make_uint4(uint32_t x, uint32_t y, uint32_t z, uint32_t w) { return uint4{x, y, z, w}; }

inline dim3 threadIdx, blockIdx, blockDim, gridDim;

namespace simt {

constexpr size_t STACK = 256 << 10;
enum State { READY, AT_WAVE, AT_LANES, AT_VOTE, AT_GROUP, DONE };
struct Fiber {
    ucontext_t ctx;
    State state;
};
inline std::vector<Fiber> fibers;
inline ucontext_t scheduler;
inline unsigned current;
inline const std::function<void()> *body;
inline long launches = 0;

inline void run_body() {
    (*body)();
    fibers[current].state = DONE;
    swapcontext(&fibers[current].ctx, &scheduler);
}
inline void wait_at(State s) {
    const unsigned me = current;
    fibers[me].state = s;
    swapcontext(&fibers[me].ctx, &scheduler);
}

// releases the fibers lo .. hi - 1 when every one that is not done waits at `s`
inline bool release(unsigned lo, unsigned hi, State s) {
    bool any = false;
    for (unsigned i = lo; i < hi; ++i) {
        if (fibers[i].state == DONE) continue;
        if (fibers[i].state != s) return false;
        any = true;
    }
    for (unsigned i = lo; any && i < hi; ++i)
        if (fibers[i].state == s) fibers[i].state = READY;
    return any;
}

// what the lanes of a branch do together (a vote, a shuffle) while the others wait behind it: releases the fibers at `s` when every
// one that is not done waits somewhere
inline bool release_some(unsigned lo, unsigned hi, State s) {
    bool any = false;
    for (unsigned i = lo; i < hi; ++i) {
        if (fibers[i].state == READY) return false;
        any |= fibers[i].state == s;
    }
    for (unsigned i = lo; any && i < hi; ++i)
        if (fibers[i].state == s) fibers[i].state = READY;
    return any;
}

inline void run_group(unsigned n) {
    static char *stacks = (char *)mmap(nullptr, 1024 * STACK, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    fibers.resize(1024);
    for (unsigned i = 0; i < n; ++i) {
        getcontext(&fibers[i].ctx);
        fibers[i].ctx.uc_stack.ss_sp = stacks + i * STACK;
        fibers[i].ctx.uc_stack.ss_size = STACK;
        fibers[i].ctx.uc_link = &scheduler;
        makecontext(&fibers[i].ctx, run_body, 0);
        fibers[i].state = READY;
    }
    for (;;) {
        bool ran = false, left = false;
        for (unsigned i = 0; i < n; ++i) {
            if (fibers[i].state == READY) {
                current = i;
                threadIdx = dim3(i % blockDim.x, i / blockDim.x);
                swapcontext(&scheduler, &fibers[i].ctx);
                ran = true;
            }
            left |= fibers[i].state != DONE;
        }
        if (!left) return;
        for (unsigned w = 0; w < n; w += 64) {
            const unsigned end = w + 64 < n ? w + 64 : n;
            // votes stand in branches, so their lanes go before those that wait at a shuffle behind the branch
            ran |= release(w, end, AT_WAVE) || release_some(w, end, AT_VOTE) || release_some(w, end, AT_LANES) || release_some(w, end, AT_WAVE);
        }
        ran |= release(0, n, AT_GROUP);
        if (!ran) {
            fprintf(stderr, "a barrier that not every thread reaches\n");
            abort();
        }
    }
}

inline std::function<void()> before_launch;                           // once, in front of the next launch: another thread's call

inline void launch(dim3 grid, dim3 block, const std::function<void()> &f) {
    if (before_launch) {
        const std::function<void()> other = std::move(before_launch);
        before_launch = nullptr;
        other();
    }
    if (block.x * block.y > 1024 || grid.x == 0 || grid.y == 0 || grid.x > 0x7FFFFFFFu || grid.y > 65535) {
        fprintf(stderr, "launch outside the limits\n");
        abort();
    }
    ++launches;
    gridDim = grid;
    blockDim = block;
    body = &f;
    for (unsigned y = 0; y < grid.y; ++y)
        for (unsigned x = 0; x < grid.x; ++x) {
            blockIdx = dim3(x, y);
            run_group(block.x * block.y);
        }
}

inline std::map<const void *, int> system_stores;                     // how often a word was stored for the host to see at once
inline int any_true, wave_any[16];
inline uint64_t wave_v[16][64];                                       // of shuffles, by wavefront and lane
inline int32_t wave_a[16][64][4], wave_b[16][64][4];                  // operands of a matrix instruction, by wavefront and lane

}  // namespace simt

#define hipLaunchKernelGGL(K, GRID, BLOCK_, LDS, STREAM, ...) simt::launch(GRID, BLOCK_, [&] { K(__VA_ARGS__); })

inline void __syncthreads() { simt::wait_at(simt::AT_GROUP); }
inline int __syncthreads_or(int v) {
    simt::any_true = 0;
    __syncthreads();
    simt::any_true |= v != 0;
    __syncthreads();
    const int r = simt::any_true;
    __syncthreads();
    return r;
}
inline int __any(int v) {                                             // over the threads of a wavefront that are still there
    int &any = simt::wave_any[threadIdx.x >> 6];
    any = 0;
    simt::wait_at(simt::AT_VOTE);
    any |= v != 0;
    simt::wait_at(simt::AT_VOTE);
    const int r = any;
    simt::wait_at(simt::AT_VOTE);
    return r;
}
// the value of lane `from` of the wavefront, the own one where there is no such lane
inline uint64_t simt_lane(uint64_t v, int from) {
    uint64_t *lanes = simt::wave_v[threadIdx.x >> 6];
    lanes[threadIdx.x & 63] = v;
    simt::wait_at(simt::AT_LANES);
    const uint64_t r = from >= 0 && from < 64 ? lanes[from] : v;
    simt::wait_at(simt::AT_LANES);
    return r;
}
inline uint64_t __shfl(uint64_t v, int lane, int) { return simt_lane(v, lane); }
inline uint64_t __shfl_xor(uint64_t v, int mask, int) { return simt_lane(v, (int)(threadIdx.x & 63) ^ mask); }
inline uint64_t __shfl_up(uint64_t v, unsigned d, int) { return simt_lane(v, (int)(threadIdx.x & 63) - (int)d); }
inline uint64_t __shfl_down(uint64_t v, unsigned d, int) { return simt_lane(v, (int)(threadIdx.x & 63) + (int)d); }
// the lanes of four, permuted: ctrl has two bits per lane (the row and bank masks leave no lane out)
inline int __builtin_amdgcn_mov_dpp(int v, int ctrl, int, int, bool) {
    const int lane = threadIdx.x & 63;
    return (int)simt_lane((uint32_t)v, (lane & ~3) | ((ctrl >> (2 * (lane & 3))) & 3));
}
inline uint32_t __builtin_amdgcn_alignbit(uint32_t hi, uint32_t lo, uint32_t n) { return (uint32_t)(((uint64_t)hi << 32 | lo) >> (n & 31)); }
inline void __threadfence_system() {}
#define __builtin_amdgcn_fence(...) ((void)0)
#define __builtin_amdgcn_wave_barrier() simt::wait_at(simt::AT_WAVE)
#define __builtin_nontemporal_load(p) (*(p))
#define __hip_atomic_load(p, order, scope) (*(p))
enum { __HIP_MEMORY_SCOPE_AGENT = 4, __HIP_MEMORY_SCOPE_SYSTEM = 5 };
template <class T, class V>
void simt_store(T *p, V v, int scope) {
    *p = (T)v;
    if (scope == __HIP_MEMORY_SCOPE_SYSTEM) ++simt::system_stores[p];
}
#define __hip_atomic_store(p, v, order, scope) simt_store(p, v, scope)
#define __builtin_nontemporal_store(v, p) (*(p) = (v))

template <class T, class V>
T atomicAdd(T *p, V v) { T was = *p; *p += (T)v; return was; }
template <class T, class V>
T atomicOr(T *p, V v) { T was = *p; *p |= (T)v; return was; }
template <class T, class V>
T atomicMin(T *p, V v) { T was = *p; if ((T)v < was) *p = (T)v; return was; }
template <class T, class E, class V>
T atomicCAS(T *p, E expect, V v) { T was = *p; if (was == (T)expect) *p = (T)v; return was; }

inline uint32_t __builtin_amdgcn_readfirstlane(uint32_t v) { return v; }   // of values that are the same for the wavefront
inline uint32_t __brev(uint32_t v) {
    uint32_t r = 0;
    for (int b = 0; b < 32; ++b) r |= ((v >> b) & 1) << (31 - b);
    return r;
}
inline uint32_t __umul24(uint32_t a, uint32_t b) { return (a & 0xFFFFFF) * (b & 0xFFFFFF); }
inline uint32_t __umulhi(uint32_t a, uint32_t b) { return (uint32_t)(((uint64_t)a * b) >> 32); }
inline uint32_t __float_as_uint(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }
inline uint32_t min(uint32_t a, uint32_t b) { return a < b ? a : b; }
inline uint32_t max(uint32_t a, uint32_t b) { return a > b ? a : b; }
inline int min(int a, int b) { return a < b ? a : b; }

// sum of the products of four signed bytes, plus c
inline int __builtin_amdgcn_sdot4(int a, int b, int c, bool) {
    for (int i = 0; i < 4; ++i) c += (int)(int8_t)(a >> (8 * i)) * (int)(int8_t)(b >> (8 * i));
    return c;
}
// bytes of {a, b} (b is the low word) picked by the four bytes of the selector, 12: zero
inline uint32_t __builtin_amdgcn_perm(uint32_t a, uint32_t b, uint32_t sel) {
    uint32_t r = 0;
    for (int i = 0; i < 4; ++i) {
        const uint32_t s = (sel >> (8 * i)) & 0xFF;
        r |= (s == 12 ? 0 : (s < 4 ? b >> (8 * s) : a >> (8 * (s - 4))) & 0xFF) << (8 * i);
    }
    return r;
}
// 32 x 32 x 32 on signed bytes: lane l holds row (column) l % 32 of A (B), the sixteen inner indices from 16 (l / 32); register r of
// the result is row 8 (r / 4) + 4 (l / 32) + r % 4 of column l % 32
template <class A, class C>
void simt_mfma_i32_32x32x32_i8(const A &a, const A &b, C &c) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int i = 0; i < 4; ++i) {
        simt::wave_a[wave][lane][i] = a[i];
        simt::wave_b[wave][lane][i] = b[i];
    }
    __builtin_amdgcn_wave_barrier();
    for (int r = 0; r < 16; ++r) {
        const int row = 8 * (r / 4) + 4 * (lane / 32) + r % 4, col = lane % 32;
        int sum = 0;
        for (int half = 0; half < 2; ++half)
            for (int i = 0; i < 4; ++i)
                sum = __builtin_amdgcn_sdot4(simt::wave_a[wave][row + 32 * half][i], simt::wave_b[wave][col + 32 * half][i], sum, false);
        c[r] += sum;
    }
    __builtin_amdgcn_wave_barrier();
}
// the accumulator is updated where it lies, as the kernels do
#define __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, x, y, z) (simt_mfma_i32_32x32x32_i8(a, b, c), c)

typedef void *hipStream_t;
typedef int hipError_t;
enum { hipSuccess = 0, hipErrorNotReady = 1, hipFuncAttributeMaxDynamicSharedMemorySize = 0, hipMemcpyHostToDevice = 1, hipMemcpyDeviceToDevice = 3 };
inline hipError_t hipGetLastError() { return hipSuccess; }
inline const char *hipGetErrorString(hipError_t) { return ""; }
inline hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
enum hipStreamCaptureStatus { hipStreamCaptureStatusNone = 0 };
inline hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) { *s = hipStreamCaptureStatusNone; return hipSuccess; }
inline hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
inline hipError_t hipFuncSetAttribute(const void *, int, int) { return hipSuccess; }
#define HIP_SYMBOL(s) s
template <class T>
hipError_t hipGetSymbolAddress(void **p, T &symbol) { *p = (void *)&symbol; return hipSuccess; }
enum hipDeviceAttribute_t { hipDeviceAttributeMultiprocessorCount };
// SIMT_CUS: a smaller chip, on which launches of the resident grid go round several times at small sizes
inline hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
    const char *cus = getenv("SIMT_CUS");
    *v = cus ? atoi(cus) : 256;
    return hipSuccess;
}
template <class K>
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, K, int, size_t) { *n = 4; return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipMalloc(void **p, size_t n) { *p = malloc(n); return hipSuccess; }
inline hipError_t hipFree(void *p) { free(p); return hipSuccess; }
inline hipError_t hipMemcpy(void *to, const void *from, size_t n, int) { memcpy(to, from, n); return hipSuccess; }
inline hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, int, hipStream_t) { memcpy(to, from, n); return hipSuccess; }
