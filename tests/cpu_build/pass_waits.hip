// The long pass of a sumcheck proof by itself, for a look at what the compiler makes of its waits (test_cpu_build_waits.py).
#include <algorithm>
#include <mutex>

#include "../../verinf_amd/csrc/common.hpp"
#include "../../verinf_amd/csrc/gl_field.hpp"

namespace {
constexpr int BLOCK = 256, MAX_BLOCKS = 2048, NSAMP = 8;
__device__ __forceinline__ void put_sample(u64 *out, u64 v) { *out = v; }
__device__ __forceinline__ u64 wave_sum(u64 v) {
    for (int off = 32; off > 0; off >>= 1) v = gl::addc(v, __shfl_xor(v, off, 64));
    return v;
}
template <typename K>
int resident_blocks(K, int) { return 1; }
inline int blocks_for(i64) { return 1; }
}  // namespace

#include "../../verinf_amd/csrc/sumcheck_fast.hpp"

namespace {
template __global__ void k_pass3_long<2, 1, false, false>(const FastDesc, i64, u64, u64, u64, u64 *, const u64 *, int, u64 *);
template __global__ void k_pass3_long<3, 1, true, false>(const FastDesc, i64, u64, u64, u64, u64 *, const u64 *, int, u64 *);
}  // namespace
