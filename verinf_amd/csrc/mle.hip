// Multilinear helpers that feed and close the sumchecks, on the device:
//   eq_vector(z)[i] = prod_j (bit_j(i) ? z_j : 1 - z_j) (layergkr/logup.py:61-69; its doubling
//                     loop puts z_0 on the LEAST significant index bit);
//   mle_eval(f, r)  = sum_i f[i] * prod_j (bit_j(i) ? r_j : 1 - r_j) with r_0 on the MOST
//                     significant bit (layergkr/sumcheck.py:40-48 computes it by folding f once
//                     per variable).
// Inside this file a point is stored most significant variable first; vi_eq_vector reverses
// its argument unless asked for the mle_eval order.
// The reference builds eq by n doublings of a Python list and evaluates by n folds; here a
// thread derives sixteen entries from one running product -- the n - 4 factors of the bits
// it shares, then a 4-level split e -> (e - e z, e z) -- so eq costs about 3 multiplications
// per entry and one coalesced store, and mle_eval is ONE streaming pass over f that never
// writes eq or any folded table.
#include "common.hpp"
#include "gl_field.hpp"

namespace {

constexpr int BLOCK = 256;
constexpr int MAX_VARS = 32;
constexpr int PARTIAL_BLOCKS = 1024;

struct Point {
    u64 z[MAX_VARS];          // canonical
};

// e[j], j < 2^JB: eq entries of the indices (j << (n - JB)) | g.
// Indices into pt.z are the same for all threads, so that the by-value argument stays in the kernarg segment.
template <int JB>
__device__ __forceinline__ void eq_entries(const Point &pt, int n, i64 g, u64 (&e)[1 << JB]) {
    // two running products, whose chains are interleaved (gl::mul_lazy2), as are the products of the split: one table of 2^26 evaluated in
    // 211 -> 178 us, eq_vector of 2^24 34 -> 32.  A loop, as a small call waits for its instructions: unrolled for all MAX_VARS variables, those that
    // are not there stepped over, k_mle_partial<3> was 39 KB and is 20: an evaluation over 2^3 entries 7.8 -> 5.3 us, 2^10 7.9 -> 6.1, 39 tables of 2^14
    // 12.4 -> 10.6 (one running product, unrolled: 6.7, 7.5 and 12.2)
    u64 even = 1, odd = 1;
    auto factor = [&](int zi) {
        const u64 z = pt.z[zi], other = z <= 1 ? 1 - z : gl::P + 1 - z;        // the same for all threads
        return (g >> (n - 1 - zi)) & 1 ? z : other;
    };
#pragma unroll 1
    for (int zi = JB; zi < n; zi += 2) gl::mul_lazy2(even, factor(zi), even, odd, zi + 1 < n ? factor(zi + 1) : 1, odd);
    e[0] = gl::mul(even, odd);
#pragma unroll
    for (int zi = JB - 1; zi >= 0; --zi) {
        // variable zi is bit (JB - 1 - zi) of j; entries with lower bits of j are already split
        const int step = 1 << (JB - 1 - zi);
        const u64 z = pt.z[zi];
        if (step == 1) {
            const u64 hi = gl::mul(e[0], z);
            e[step] = hi;
            e[0] = gl::sub(e[0], hi);
        }
#pragma unroll
        for (int x = 0; x + 1 < step; x += 2) {
            gl::mul2(e[x], z, e[x + step], e[x + 1], z, e[x + 1 + step]);
            gl::sub2(e[x], e[x + step], e[x], e[x + 1], e[x + 1 + step], e[x + 1]);
        }
    }
}

template <int JB>
__global__ __launch_bounds__(BLOCK) void k_eq_vector(const Point pt, int n, u64 *__restrict__ out) {
    const i64 threads = (i64)1 << (n - JB);
    const i64 g = (i64)blockIdx.x * BLOCK + threadIdx.x;
    if (g >= threads) return;
    u64 e[1 << JB];
    eq_entries<JB>(pt, n, g, e);
#pragma unroll
    for (int j = 0; j < (1 << JB); ++j) out[((i64)j << (n - JB)) | g] = e[j];
}

__device__ __forceinline__ u64 block_sum(u64 v, u64 *lds4) {
    for (int off = 32; off > 0; off >>= 1) v = gl::add(v, __shfl_xor(v, off, 64));
    if ((threadIdx.x & 63) == 0) lds4[threadIdx.x >> 6] = v;
    __syncthreads();
    u64 r = 0;
    if (threadIdx.x == 0) {
        r = lds4[0];
        for (int i = 1; i < BLOCK / 64; ++i) r = gl::add(r, lds4[i]);
    }
    __syncthreads();
    return r;
}

// partial[row * gridDim.x + block] = sum over this block's share of f_row[i] * eq[i], for the up to TB
// tables row = blockIdx.y * TB + 0 .. TB-1: the eq entries of an index are computed once and used for all
// of them.  A table's words are requested while those of the table before it are used (the first table's before the eq entries are
// computed), the products of a table are added up as one integer of five words, and the tables' sums over the workgroup go
// side by side: 39 tables of 2^18 entries 27.5 -> 22 us (3.7 TB/s), of 2^20 90 -> 78 a call, one of 2^26 265 -> 212.
constexpr int TB = 4;

template <int JB>
__global__ __launch_bounds__(BLOCK) void k_mle_partial(const Point pt, int n, const u64 *__restrict__ tables, i64 row_stride,
                                                       int n_tables, u64 *__restrict__ partial) {
    __shared__ u64 lds[BLOCK / 64][TB];
    const i64 threads = (i64)1 << (n - JB);
    const int row0 = blockIdx.y * TB;
    const int rows = n_tables - row0 < TB ? n_tables - row0 : TB;
    u64 acc[TB];
#pragma unroll
    for (int r = 0; r < TB; ++r) acc[r] = 0;
    for (i64 g = (i64)blockIdx.x * BLOCK + threadIdx.x; g < threads; g += (i64)gridDim.x * BLOCK) {
        u64 e[1 << JB], v[2][1 << JB];
        // read once: with the streaming hint (three tables of 2^24 104 -> 97 us, 39 of 2^20 75.7 -> 74.4, smaller ones within 2 % either way)
        auto fetch = [&](int r) {
            const u64 *f = tables + (i64)(row0 + r) * row_stride;
#pragma unroll
            for (int j = 0; j < (1 << JB); ++j) v[r & 1][j] = __builtin_nontemporal_load(&f[((i64)j << (n - JB)) | g]);
        };
        fetch(0);
        VI_SCHED_FENCE();                      // the loads stay in front of what they are to hide behind
        eq_entries<JB>(pt, n, g, e);
#pragma unroll
        for (int r = 0; r < TB; ++r) {
            if (r >= rows) break;
            VI_SCHED_FENCE();
            if (r + 1 < rows) fetch(r + 1);
            VI_SCHED_FENCE();
            gl::Wide sum;
            gl::wide_zero(sum);
#pragma unroll
            for (int j = 0; j < (1 << JB); ++j) gl::wide_mul_acc(sum, e[j], v[r & 1][j]);
            acc[r] = gl::addc(acc[r], gl::wide_reduce(sum));
        }
    }
    // the tables' sums side by side: their shuffles are in flight together, one barrier
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        u64 o[TB];
#pragma unroll
        for (int r = 0; r < TB; ++r) o[r] = __shfl_xor(acc[r], off, 64);
#pragma unroll
        for (int r = 0; r < TB; ++r) acc[r] = gl::addc(acc[r], o[r]);
    }
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int r = 0; r < TB; ++r) lds[threadIdx.x >> 6][r] = acc[r];
    }
    __syncthreads();
    if ((int)threadIdx.x < rows) {
        u64 s = lds[0][threadIdx.x];
        for (int i = 1; i < BLOCK / 64; ++i) s = gl::addc(s, lds[i][threadIdx.x]);
        partial[(i64)(row0 + threadIdx.x) * gridDim.x + blockIdx.x] = s;
    }
}

__global__ __launch_bounds__(BLOCK) void k_mle_final(const u64 *__restrict__ partial, int nb, u64 *__restrict__ out) {
    __shared__ u64 lds4[BLOCK / 64];
    u64 acc = 0;
    for (int i = threadIdx.x; i < nb; i += BLOCK) acc = gl::add(acc, partial[(i64)blockIdx.x * nb + i]);
    const u64 r = block_sum(acc, lds4);
    // straight through to memory: `out` may be host memory that is being polled
    if (threadIdx.x == 0) __hip_atomic_store(&out[blockIdx.x], r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

int load_point(const char *who, const uint64_t *z, int n, bool msb_first, Point &pt) {
    if (n < 0 || n > MAX_VARS) return vi::fail(VI_EINVAL, "%s: %d variables (0 .. %d supported)", who, n, MAX_VARS);
    if (n > 0 && !z) return vi::fail(VI_EINVAL, "%s: null point", who);
    for (int i = 0; i < MAX_VARS; ++i) pt.z[i] = i < n ? gl::canon(z[msb_first ? i : n - 1 - i]) : 0;
    return VI_OK;
}

}  // namespace

extern "C" {

int vi_eq_vector(const uint64_t *z, int n_vars, int msb_first, uint64_t *out, void *stream) {
    Point pt;
    int rc = load_point("vi_eq_vector", z, n_vars, msb_first != 0, pt);
    if (rc) return rc;
    if (!out) return vi::fail(VI_EINVAL, "vi_eq_vector: null out");
    const int jb = n_vars < 4 ? n_vars : 4;
    const i64 threads = (i64)1 << (n_vars - jb);
    const dim3 grid((unsigned)((threads + BLOCK - 1) / BLOCK)), block(BLOCK);
    hipStream_t s = (hipStream_t)stream;
    switch (jb) {
        case 0: hipLaunchKernelGGL(k_eq_vector<0>, grid, block, 0, s, pt, n_vars, out); break;
        case 1: hipLaunchKernelGGL(k_eq_vector<1>, grid, block, 0, s, pt, n_vars, out); break;
        case 2: hipLaunchKernelGGL(k_eq_vector<2>, grid, block, 0, s, pt, n_vars, out); break;
        case 3: hipLaunchKernelGGL(k_eq_vector<3>, grid, block, 0, s, pt, n_vars, out); break;
        default: hipLaunchKernelGGL(k_eq_vector<4>, grid, block, 0, s, pt, n_vars, out); break;
    }
    VI_LAUNCH_CHECK("k_eq_vector");
    return VI_OK;
}

size_t vi_mle_eval_workspace_bytes(int64_t n_tables) {
    return n_tables <= 0 ? 0 : (size_t)n_tables * PARTIAL_BLOCKS * sizeof(u64);
}

int vi_mle_eval(const uint64_t *tables, int64_t n_tables, int64_t row_stride, const uint64_t *z, int n_vars,
                uint64_t *out, void *ws, size_t ws_bytes, void *stream) {
    Point pt;
    int rc = load_point("vi_mle_eval", z, n_vars, true, pt);
    if (rc) return rc;
    if (n_tables < 0 || n_tables > 65535) return vi::fail(VI_EINVAL, "vi_mle_eval: n_tables = %lld (0 .. 65535)", (long long)n_tables);
    if (n_tables == 0) return VI_OK;
    if (!tables || !out) return vi::fail(VI_EINVAL, "vi_mle_eval: null pointer");
    if (n_tables > 1 && row_stride < ((int64_t)1 << n_vars)) return vi::fail(VI_EINVAL, "vi_mle_eval: row_stride below the table length");
    if (!ws || ws_bytes < vi_mle_eval_workspace_bytes(n_tables)) return vi::fail(VI_ENOMEM, "vi_mle_eval: workspace too small");
    // sixteen entries to a thread where that still fills the chip, eight below (39 tables of 2^16: 28.0 -> 26.7 us a call, of 2^20: 78
    // with sixteen, 81 with eight)
    const int most = n_vars >= 18 ? 4 : 3, jb = n_vars < most ? n_vars : most;
    const i64 threads = (i64)1 << (n_vars - jb);
    i64 nb = (threads + BLOCK - 1) / BLOCK;
    if (nb > PARTIAL_BLOCKS) nb = PARTIAL_BLOCKS;
    const dim3 block(BLOCK);
    hipStream_t s = (hipStream_t)stream;
    u64 *partial = (u64 *)ws;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)nb, (unsigned)((n_tables + TB - 1) / TB)), block, 0, s, pt, n_vars, tables, (i64)row_stride, (int)n_tables,
                           partial);
    };
    switch (jb) {
        case 0: launch(k_mle_partial<0>); break;
        case 1: launch(k_mle_partial<1>); break;
        case 2: launch(k_mle_partial<2>); break;
        case 3: launch(k_mle_partial<3>); break;
        default: launch(k_mle_partial<4>); break;
    }
    VI_LAUNCH_CHECK("k_mle_partial");
    hipLaunchKernelGGL(k_mle_final, dim3((unsigned)n_tables), block, 0, s, (const u64 *)partial, (int)nb, out);
    VI_LAUNCH_CHECK("k_mle_final");
    return VI_OK;
}

}  // extern "C"
