// Elementwise Goldilocks kernels and the field sum reduction.
//
// All of these are pure HBM streaming (24 B per element for a binary op) with a
// handful of integer VALU ops per element; they use 64-bit indexing and a
// grid-stride loop sized to keep every CU busy (the reference kernels index with
// int, prover/cuda_primitives.py:208-233).
#include "common.hpp"
#include "gl_field.hpp"

namespace {

constexpr int BLOCK = 256;
constexpr int MAX_BLOCKS = 256 * 16;      // 16 workgroups per CU

inline unsigned grid_for(i64 n) {
    i64 b = (n + BLOCK - 1) / BLOCK;
    return (unsigned)(b < 1 ? 1 : (b > MAX_BLOCKS ? MAX_BLOCKS : b));
}

template <int OP>
__device__ __forceinline__ u64 apply(u64 a, u64 b) {
    return OP == 0 ? gl::add(a, b) : OP == 1 ? gl::sub(a, b) : gl::mul(a, b);
}

template <int OP>
__global__ __launch_bounds__(BLOCK) void k_binop(const u64 *a, const u64 *b, u64 *out, i64 n) {
    i64 stride = (i64)gridDim.x * BLOCK;
    for (i64 i = (i64)blockIdx.x * BLOCK + threadIdx.x; i < n; i += stride)
        __builtin_nontemporal_store(apply<OP>(__builtin_nontemporal_load(a + i), __builtin_nontemporal_load(b + i)), out + i);
}

// two elements per lane through 16-byte accesses (operands 16-byte aligned); the last of an odd number by itself
template <int OP>
__global__ __launch_bounds__(BLOCK) void k_binop_v2(const ulonglong2 *a, const ulonglong2 *b, ulonglong2 *out, i64 n) {
    const i64 stride = (i64)gridDim.x * BLOCK, n2 = n >> 1;
    if ((n & 1) && blockIdx.x == gridDim.x - 1 && threadIdx.x == BLOCK - 1) {
        const u64 *x = (const u64 *)a, *y = (const u64 *)b;
        ((u64 *)out)[n - 1] = apply<OP>(x[n - 1], y[n - 1]);
    }
    for (i64 i = (i64)blockIdx.x * BLOCK + threadIdx.x; i < n2; i += stride) {
        // operands read once, result not read back by this launch: streaming hints (2^24 elements 5.1 -> 5.9 TB/s,
        // 2^27 4.40 -> 4.50 TB/s)
        typedef u64 v2 __attribute__((ext_vector_type(2)));
        const v2 xv = __builtin_nontemporal_load(reinterpret_cast<const v2 *>(a + i));
        const v2 yv = __builtin_nontemporal_load(reinterpret_cast<const v2 *>(b + i));
        v2 rv;
        rv.x = apply<OP>(xv.x, yv.x);
        rv.y = apply<OP>(xv.y, yv.y);
        __builtin_nontemporal_store(rv, reinterpret_cast<v2 *>(out + i));
    }
}

template <int OP>
__global__ __launch_bounds__(BLOCK) void k_binop_bcast(const u64 *a, const u64 *b, i64 period, u64 *out, i64 n) {
    i64 stride = (i64)gridDim.x * BLOCK;
    for (i64 i = (i64)blockIdx.x * BLOCK + threadIdx.x; i < n; i += stride) out[i] = apply<OP>(a[i], b[i % period]);
}

__global__ __launch_bounds__(BLOCK) void k_unop(int op, const u64 *a, u64 arg, u64 *out, i64 n) {
    i64 stride = (i64)gridDim.x * BLOCK;
    for (i64 i = (i64)blockIdx.x * BLOCK + threadIdx.x; i < n; i += stride) {
        u64 v = a[i];
        out[i] = op == 0 ? gl::neg(v) : gl::pow(v, arg);
    }
}

// One device field primitive applied elementwise, for the test-suite: the transforms use these through fully
// unrolled code with compile-time exponents, so this is the only place they can be driven with chosen operands.
template <int E>
__device__ __forceinline__ u64 shift_by(u64 v, int e) {
    if constexpr (E >= 96) return 0;
    else {
        if (e == E) return gl::mul_pow2c<E>(v);
        return shift_by<E + 1>(v, e);
    }
}

// the same through the form used inside the coset loop of the fused LDE launch: any exponent below 192, 2^96 = -1
template <int E>
__device__ __forceinline__ u64 shift_pinned_by(u64 v, int e) {
    if constexpr (E >= 192) return 0;
    else {
        if (e == E) return gl::mul_pow2c_pinned<E>(v);
        return shift_pinned_by<E + 1>(v, e);
    }
}

__global__ __launch_bounds__(BLOCK) void k_probe(int op, const u64 *a, const u64 *b, u64 *out, i64 n) {
    i64 stride = (i64)gridDim.x * BLOCK;
    for (i64 i = (i64)blockIdx.x * BLOCK + threadIdx.x; i < n; i += stride) {
        const u64 x = a[i], y = b ? b[i] : 0;
        u64 s, d, r;
        gl::bfly(x, y, s, d);
        if (op == 0) r = gl::addc(x, y);
        else if (op == 1) r = gl::sub(x, y);
        else if (op == 2) r = s;
        else if (op == 3) r = d;
        else if (op == 4) r = gl::canon(x);
        else if (op == 5) r = gl::mul(x, y);
        else if (op == 6) r = gl::reduce128(x, y);
        else if (op == 7) r = gl::canon(gl::mul_lazy(x, y));
        else if (op == 8) r = gl::mul_add(x, y, ((x << 17) | (x >> 47)) ^ y);
        else if (op == 9) r = gl::canon(gl::mul_add_lazy(x, y, ((x << 17) | (x >> 47)) ^ y));
        else if (op == 10 || op == 11) {
            gl::Wide A;
            gl::wide_zero(A);
            if (op == 10) {
                gl::wide_mul_acc(A, x, y);
                gl::wide_mul_acc(A, y, y);
                gl::wide_mul_acc(A, x, x);
                gl::wide_mul_acc(A, ~x, ~y);
                gl::wide_mul_acc(A, ~0ull, ~0ull);
            } else {
                for (int k = 0; k < 40; ++k) gl::wide_mul_acc(A, x, y);      // carries into the fifth word
            }
            r = gl::wide_reduce(A);
        }
        else if (op >= 20 && op < 36) {
            // two at once: the first result, and the second (of other operands)
            u64 p, q;
            const u64 e = ((x << 17) | (x >> 47)) ^ y;
            if (op < 22) gl::sub2(x, y, p, y, x, q);
            else if (op < 24) gl::addc2(x, y, p, y, y, q);
            else if (op < 26) gl::mul2(x, y, p, y, y, q);
            else if (op < 28) gl::mul_lazy2(x, y, p, y, y, q);
            else if (op < 30) gl::mul_add2(x, y, e, p, y, y, x, q);
            else if (op >= 32) {
                u64 s, d, t, v;
                gl::bfly2(x, y, s, d, y, x, t, v);
                p = op < 34 ? s : d;
                q = op < 34 ? t : v;
            }
            else {
                gl::Wide A, B;
                gl::wide_zero(A);
                gl::wide_zero(B);
                for (int k = 0; k < 40; ++k) gl::wide_mul_acc2(A, x, y, B, ~0ull, ~y);
                p = gl::wide_reduce(A);
                q = gl::wide_reduce(B);
            }
            r = op & 1 ? q : p;
            if (op == 26 || op == 27) r = gl::canon(r);
        }
        else if (op >= 300) r = shift_pinned_by<0>(x, op - 300);
        else r = shift_by<0>(x, op - 100);
        out[i] = r;
    }
}

// Inverses of a whole array by Montgomery's trick (the batching of layergkr/field.py:84-101 at the scale of one
// workgroup): a thread takes INV_E elements, one from each of INV_E equal slabs of the array so that a wavefront's
// accesses stay contiguous, and multiplies them up; the first wavefront does the same with the products of all threads
// and inverts ONE product per lane (74 multiplications in a chain); the single inverses are peeled off in turn.  A
// wavefront that inverts costs the same however many of its lanes do, so the chain is paid once per
// workgroup and not once per wavefront.  Workgroups of 256 rather than 512 have the shorter chain and fill the SIMDs while one wavefront of each
// inverts (1.5 M elements 13.6 -> 12.4 us, 16 M 89 -> 71).  Zeros are taken out of the product and map to zero, so every output
// equals the Fermat power a^(p-2) of the reference kernel (prover/cuda_primitives.py:289-303).
//
// A call lasts as long as a thread's chain of products, up to a few million elements; beyond that VALU issue.  The thread's
// elements run as two halves side by side and what feeds another product is only reduced to a congruent word: us per call in a
// queue, one half and canonical words -> now: 200000 elements 8.0 -> 6.8, 700001 9.4 -> 8.3, 1.5 M 12.0 -> 10.5, 6 M 30.0 -> 26.6,
// 16 M 71.0 -> 62.3 (one inversion to an element, lazily reduced words alone: 100000 7.5 -> 6.6).
//
// Elements of a thread: four while the chip has SIMDs to spare, then eight, then twelve, which share an inversion (us with 4, 8 and 12,
// measured with one half:
// 300000 8.7, 9.7, 10.7; 700001 9.6, 10.9, 11.3; 1.5 M 13.3, 12.4, 13.3; 3 M 21.8, 22.0, 17.5; 6 M 33.6, 32.4, 29.4; 16 M 78.6, 70.8, 68.0).
constexpr int INV_THREADS = 256;

// Few elements: an inversion each.  A launch lasts as long as one thread's chain while a SIMD has a wavefront or two, and
// without products before and after it the chain is the shortest (us per call in a queue: 1000 elements 9.5 -> 6.3, 2^16 10.5
// -> 6.4, 2^17 10.6 -> 7.4, 200000 with a third wavefront 10.6 -> 11.5).
constexpr i64 INV_FEW = (i64)1 << 17;

__global__ __launch_bounds__(64) void k_inv_each(const u64 *a, u64 *out, i64 n) {
    const i64 i = (i64)blockIdx.x * 64 + threadIdx.x;
    if (i < n) out[i] = gl::inv(gl::canon(a[i]));
}

template <int INV_E>
__global__ __launch_bounds__(INV_THREADS) void k_inv_batched(const u64 *a, u64 *out, i64 n, i64 groups) {
    __shared__ u64 prod[INV_THREADS];
    const int tid = threadIdx.x;
    const i64 g = (i64)blockIdx.x * INV_THREADS + tid;
    u64 x[INV_E], pre[INV_E];
    unsigned zero = 0;
#pragma unroll
    for (int j = 0; j < INV_E; ++j) {
        const i64 i = (i64)j * groups + g;
        x[j] = g < groups && i < n ? a[i] : 1;
    }
#pragma unroll
    for (int j = 0; j < INV_E; ++j) {
        u64 v = gl::canon(x[j]);
        if (v == 0) { zero |= 1u << j; v = 1; }
        x[j] = v;
    }
    // two halves of the elements with interleaved products (gl::mul2)
    constexpr int H = INV_E / 2;
    pre[0] = x[0];
    pre[H] = x[H];
#pragma unroll
    for (int j = 1; j < H; ++j) gl::mul_lazy2(pre[j - 1], x[j], pre[j], pre[H + j - 1], x[H + j], pre[H + j]);
    prod[tid] = gl::mul_lazy(pre[H - 1], pre[INV_E - 1]);
    __syncthreads();
    if (tid < 64) {
        static_assert(INV_THREADS == 256, "four products to a lane");
        u64 y[4], low, high, r[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) y[j] = prod[tid + 64 * j];
        gl::mul_lazy2(y[0], y[1], low, y[2], y[3], high);
        const u64 all = gl::inv(gl::mul_lazy(low, high));
        u64 a01, a23;                          // 1 / (y0 y1), 1 / (y2 y3)
        gl::mul_lazy2(all, high, a01, all, low, a23);
        gl::mul_lazy2(a01, y[1], r[0], a01, y[0], r[1]);
        gl::mul_lazy2(a23, y[3], r[2], a23, y[2], r[3]);
#pragma unroll
        for (int j = 0; j < 4; ++j) prod[tid + 64 * j] = r[j];
    }
    __syncthreads();
    u64 low = prod[tid], high;
    gl::mul_lazy2(low, pre[INV_E - 1], low, low, pre[H - 1], high);            // 1 / (x0 .. x(H-1)) and 1 / (xH ..)
    auto put = [&](int j, u64 r) {
        const i64 i = (i64)j * groups + g;
        if (g < groups && i < n) out[i] = (zero >> j) & 1 ? 0 : r;
    };
#pragma unroll
    for (int j = H - 1; j >= 1; --j) {
        u64 r, q;
        gl::mul2(low, pre[j - 1], r, high, pre[H + j - 1], q);
        gl::mul_lazy2(low, x[j], low, high, x[H + j], high);
        put(j, r);
        put(H + j, q);
    }
    put(0, gl::canon(low));
    put(H, gl::canon(high));
}

__global__ __launch_bounds__(BLOCK) void k_axpy(u64 *y, u64 alpha, const u64 *x, i64 n) {
    i64 stride = (i64)gridDim.x * BLOCK;
    for (i64 i = (i64)blockIdx.x * BLOCK + threadIdx.x; i < n; i += stride) y[i] = gl::add(y[i], gl::mul(alpha, x[i]));
}

__device__ __forceinline__ u64 wave_sum(u64 v) {
    for (int off = 32; off > 0; off >>= 1) v = gl::add(v, __shfl_xor(v, off, 64));
    return v;
}

// block-wide field sum; the result is valid in thread 0
__device__ __forceinline__ u64 block_sum(u64 v, u64 *lds4) {
    v = wave_sum(v);
    int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) lds4[w] = v;
    __syncthreads();
    u64 r = 0;
    if (threadIdx.x == 0) {
        r = lds4[0];
        for (int i = 1; i < BLOCK / 64; ++i) r = gl::add(r, lds4[i]);
    }
    __syncthreads();
    return r;
}

constexpr int SUM_BLOCKS = 1024;

__global__ __launch_bounds__(BLOCK) void k_sum_partial(const u64 *a, i64 n, u64 *partial) {
    __shared__ u64 lds4[BLOCK / 64];
    i64 stride = (i64)gridDim.x * BLOCK;
    u64 acc = 0;
    i64 i = (i64)blockIdx.x * BLOCK + threadIdx.x;
    for (; i + 3 * stride < n; i += 4 * stride) {     // four loads in flight
        u64 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = __builtin_nontemporal_load(&a[i + u * stride]);     // read once: streaming
#pragma unroll
        for (int u = 0; u < 4; ++u) acc = gl::add(acc, v[u] >= gl::P ? v[u] - gl::P : v[u]);
    }
    for (; i < n; i += stride) {
        u64 v = a[i];
        acc = gl::add(acc, v >= gl::P ? v - gl::P : v);
    }
    u64 r = block_sum(acc, lds4);
    if (threadIdx.x == 0) partial[blockIdx.x] = r;
}

__global__ __launch_bounds__(BLOCK) void k_sum_final(const u64 *partial, int nb, u64 *out) {
    __shared__ u64 lds4[BLOCK / 64];
    u64 acc = 0;
    for (int i = threadIdx.x; i < nb; i += BLOCK) acc = gl::add(acc, partial[i]);
    u64 r = block_sum(acc, lds4);
    if (threadIdx.x == 0) out[0] = r;
}

// words of a small result to pinned host memory, then the tag the host polls (one workgroup, so that one barrier and one
// fence order the data before the tag)
__global__ __launch_bounds__(BLOCK) void k_read_back(const u32 *src, int words, u32 *host, u64 *flag, u64 tag) {
    for (int i = threadIdx.x; i < words; i += BLOCK) host[i] = src[i];
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(flag, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

struct Words {
    u64 w[VI_UPLOAD_WORDS];
};
__global__ __launch_bounds__(BLOCK) void k_upload(const Words W, int n, u64 *dst) {
    for (int i = threadIdx.x; i < n; i += BLOCK) dst[i] = W.w[i];
}

inline bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

extern "C" {

const char *vi_last_error(void) { return vi::err_buf(); }
const char *vi_version(void) { return "0.2"; }

int vi_read_back(const void *src, int64_t bytes, void *host, size_t host_bytes, void *stream) {
    if (bytes <= 0 || bytes > (1 << 20) || (bytes & 3)) return vi::fail(VI_EINVAL, "vi_read_back: %lld bytes (a multiple of 4 up to 2^20)", (long long)bytes);
    const size_t data = ((size_t)bytes + 7) & ~(size_t)7;
    if (!src || !host || ((uintptr_t)src & 3) || ((uintptr_t)host & 7)) return vi::fail(VI_EINVAL, "vi_read_back: null or unaligned pointer");
    if (host_bytes < data + 8) return vi::fail(VI_ENOMEM, "vi_read_back: host buffer below %zu bytes", data + 8);
    u64 *flag = (u64 *)((char *)host + data);
    const u64 tag = vi::new_tag();
    *(volatile u64 *)flag = 0;
    std::atomic_thread_fence(std::memory_order_seq_cst);
    hipLaunchKernelGGL(k_read_back, dim3(1), dim3(BLOCK), 0, (hipStream_t)stream, (const u32 *)src, (int)(bytes / 4), (u32 *)host, flag, tag);
    VI_LAUNCH_CHECK("k_read_back");
    return vi::wait_for_tag("vi_read_back", flag, tag, (hipStream_t)stream);
}

int vi_wait_words(const uint64_t *words, int64_t rows, int64_t row_words, int64_t n, void *stream) {
    if (rows < 0 || n < 0 || row_words < n) return vi::fail(VI_EINVAL, "vi_wait_words: %lld of %lld words in %lld rows", (long long)n, (long long)row_words, (long long)rows);
    if (rows == 0 || n == 0) return VI_OK;
    if (!words || ((uintptr_t)words & 7)) return vi::fail(VI_EINVAL, "vi_wait_words: null or unaligned pointer");
    const volatile uint64_t *w = words;
    int64_t r = 0, i = 0;
    return vi::wait_until("vi_wait_words", [&] {
        for (; r < rows; ++r, i = 0)
            for (; i < n; ++i)
                if (w[r * row_words + i] == VI_NO_WORD) return false;
        return true;
    }, (hipStream_t)stream);
}

int vi_upload_words(const uint64_t *host, int64_t n, uint64_t *dst, void *stream) {
    if (n < 0 || n > VI_UPLOAD_WORDS) return vi::fail(VI_EINVAL, "vi_upload_words: n = %lld (0 .. %d)", (long long)n, VI_UPLOAD_WORDS);
    if (n == 0) return VI_OK;
    if (!host || !dst) return vi::fail(VI_EINVAL, "vi_upload_words: null pointer");
    Words W;
    for (i64 i = 0; i < VI_UPLOAD_WORDS; ++i) W.w[i] = i < n ? host[i] : 0;
    hipLaunchKernelGGL(k_upload, dim3(1), dim3(BLOCK), 0, (hipStream_t)stream, W, (int)n, dst);
    VI_LAUNCH_CHECK("k_upload");
    return VI_OK;
}

int vi_gl_binop(int op, const uint64_t *a, const uint64_t *b, uint64_t *out, int64_t n, void *stream) {
    if (op < 0 || op > 2) return vi::fail(VI_EINVAL, "vi_gl_binop: op %d", op);
    if (n < 0) return vi::fail(VI_EINVAL, "vi_gl_binop: n = %lld", (long long)n);
    if (n == 0) return VI_OK;
    if (!a || !b || !out) return vi::fail(VI_EINVAL, "vi_gl_binop: null pointer");
    hipStream_t s = (hipStream_t)stream;
    if (aligned16(a) && aligned16(b) && aligned16(out)) {
        const i64 n2 = (n + 1) / 2;
        auto A = (const ulonglong2 *)a, B = (const ulonglong2 *)b;
        auto O = (ulonglong2 *)out;
        if (op == 0) hipLaunchKernelGGL(k_binop_v2<0>, dim3(grid_for(n2)), dim3(BLOCK), 0, s, A, B, O, (i64)n);
        if (op == 1) hipLaunchKernelGGL(k_binop_v2<1>, dim3(grid_for(n2)), dim3(BLOCK), 0, s, A, B, O, (i64)n);
        if (op == 2) hipLaunchKernelGGL(k_binop_v2<2>, dim3(grid_for(n2)), dim3(BLOCK), 0, s, A, B, O, (i64)n);
    } else {
        if (op == 0) hipLaunchKernelGGL(k_binop<0>, dim3(grid_for(n)), dim3(BLOCK), 0, s, a, b, out, (i64)n);
        if (op == 1) hipLaunchKernelGGL(k_binop<1>, dim3(grid_for(n)), dim3(BLOCK), 0, s, a, b, out, (i64)n);
        if (op == 2) hipLaunchKernelGGL(k_binop<2>, dim3(grid_for(n)), dim3(BLOCK), 0, s, a, b, out, (i64)n);
    }
    VI_LAUNCH_CHECK("k_binop");
    return VI_OK;
}

int vi_gl_binop_bcast(int op, const uint64_t *a, const uint64_t *b, int64_t period, uint64_t *out,
                      int64_t n, void *stream) {
    if (op < 0 || op > 2) return vi::fail(VI_EINVAL, "vi_gl_binop_bcast: op %d", op);
    if (n < 0 || period <= 0) return vi::fail(VI_EINVAL, "vi_gl_binop_bcast: n = %lld period = %lld", (long long)n, (long long)period);
    if (n == 0) return VI_OK;
    if (!a || !b || !out) return vi::fail(VI_EINVAL, "vi_gl_binop_bcast: null pointer");
    hipStream_t s = (hipStream_t)stream;
    if (op == 0) hipLaunchKernelGGL(k_binop_bcast<0>, dim3(grid_for(n)), dim3(BLOCK), 0, s, a, b, (i64)period, out, (i64)n);
    if (op == 1) hipLaunchKernelGGL(k_binop_bcast<1>, dim3(grid_for(n)), dim3(BLOCK), 0, s, a, b, (i64)period, out, (i64)n);
    if (op == 2) hipLaunchKernelGGL(k_binop_bcast<2>, dim3(grid_for(n)), dim3(BLOCK), 0, s, a, b, (i64)period, out, (i64)n);
    VI_LAUNCH_CHECK("k_binop_bcast");
    return VI_OK;
}

int vi_gl_unop(int op, const uint64_t *a, uint64_t arg, uint64_t *out, int64_t n, void *stream) {
    if (op < 0 || op > 2) return vi::fail(VI_EINVAL, "vi_gl_unop: op %d", op);
    if (n < 0) return vi::fail(VI_EINVAL, "vi_gl_unop: n = %lld", (long long)n);
    if (n == 0) return VI_OK;
    if (!a || !out) return vi::fail(VI_EINVAL, "vi_gl_unop: null pointer");
    if (op == 2) {
        if (n <= INV_FEW) {
            hipLaunchKernelGGL(k_inv_each, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, (hipStream_t)stream, a, out, (i64)n);
            VI_LAUNCH_CHECK("k_inv_each");
            return VI_OK;
        }
        const int each = n <= ((i64)1 << 20) ? 4 : n <= ((i64)1 << 21) ? 8 : 12;
        const i64 groups = (n + each - 1) / each;
        const i64 blocks = (groups + INV_THREADS - 1) / INV_THREADS;
        if (blocks > 0x7FFFFFFF) return vi::fail(VI_EINVAL, "vi_gl_unop: n = %lld", (long long)n);
        const dim3 grid((unsigned)blocks), block(INV_THREADS);
        if (each == 4) hipLaunchKernelGGL(k_inv_batched<4>, grid, block, 0, (hipStream_t)stream, a, out, (i64)n, groups);
        else if (each == 8) hipLaunchKernelGGL(k_inv_batched<8>, grid, block, 0, (hipStream_t)stream, a, out, (i64)n, groups);
        else hipLaunchKernelGGL(k_inv_batched<12>, grid, block, 0, (hipStream_t)stream, a, out, (i64)n, groups);
        VI_LAUNCH_CHECK("k_inv_batched");
        return VI_OK;
    }
    hipLaunchKernelGGL(k_unop, dim3(grid_for(n)), dim3(BLOCK), 0, (hipStream_t)stream, op, a, (u64)arg, out, (i64)n);
    VI_LAUNCH_CHECK("k_unop");
    return VI_OK;
}

int vi_gl_axpy(uint64_t *y, uint64_t alpha, const uint64_t *x, int64_t n, void *stream) {
    if (n < 0) return vi::fail(VI_EINVAL, "vi_gl_axpy: n = %lld", (long long)n);
    if (n == 0) return VI_OK;
    if (!y || !x) return vi::fail(VI_EINVAL, "vi_gl_axpy: null pointer");
    hipLaunchKernelGGL(k_axpy, dim3(grid_for(n)), dim3(BLOCK), 0, (hipStream_t)stream, y, (u64)alpha, x, (i64)n);
    VI_LAUNCH_CHECK("k_axpy");
    return VI_OK;
}

int vi_gl_probe(int op, const uint64_t *a, const uint64_t *b, uint64_t *out, int64_t n, void *stream) {
    const bool shift = (op >= 100 && op < 196) || (op >= 300 && op < 492);
    if (!shift && (op < 0 || (op > 11 && op < 20) || op > 35)) return vi::fail(VI_EINVAL, "vi_gl_probe: op = %d", op);
    if (n < 0) return vi::fail(VI_EINVAL, "vi_gl_probe: n = %lld", (long long)n);
    if (n == 0) return VI_OK;
    const bool needs_b = !shift && op != 4;
    if (!a || !out || (needs_b && !b)) return vi::fail(VI_EINVAL, "vi_gl_probe: null pointer");
    hipLaunchKernelGGL(k_probe, dim3(grid_for(n)), dim3(BLOCK), 0, (hipStream_t)stream, op, a, needs_b ? b : nullptr, out, (i64)n);
    VI_LAUNCH_CHECK("k_probe");
    return VI_OK;
}

size_t vi_gl_sum_workspace_bytes(int64_t n) {
    (void)n;
    return SUM_BLOCKS * sizeof(u64);
}

int vi_gl_sum(const uint64_t *a, int64_t n, uint64_t *out, void *ws, size_t ws_bytes, void *stream) {
    if (n < 0) return vi::fail(VI_EINVAL, "vi_gl_sum: n = %lld", (long long)n);
    if (!out || (n > 0 && !a)) return vi::fail(VI_EINVAL, "vi_gl_sum: null pointer");
    if (!ws || ws_bytes < SUM_BLOCKS * sizeof(u64)) return vi::fail(VI_ENOMEM, "vi_gl_sum: workspace below %zu bytes", SUM_BLOCKS * sizeof(u64));
    i64 b = (n + BLOCK - 1) / BLOCK;
    int nb = (int)(b < 1 ? 1 : (b > SUM_BLOCKS ? SUM_BLOCKS : b));
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(k_sum_partial, dim3(nb), dim3(BLOCK), 0, s, a, (i64)n, (u64 *)ws);
    VI_LAUNCH_CHECK("k_sum_partial");
    hipLaunchKernelGGL(k_sum_final, dim3(1), dim3(BLOCK), 0, s, (const u64 *)ws, nb, out);
    VI_LAUNCH_CHECK("k_sum_final");
    return VI_OK;
}

}  // extern "C"
