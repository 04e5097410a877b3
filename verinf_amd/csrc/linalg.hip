// Dense field products over Goldilocks: C = A B, w = M v, and Horner evaluation.
//
// The reference kernels reduce after every term (s = add(s, mul(a, b)),
// prover/kernels/gl_matmul.cuh:29-59).  Here a dot product is accumulated as an exact
// integer -- 128-bit running sum plus a count of its wrap-arounds -- and reduced once
// at the end: per term four v_mad_u64_u32 and a carry chain instead of a full modular
// multiply-add.  Results are the same canonical residues.
//
// k_matmul is built for few rows of A (1 for the projection seam `chi^T W`, layergkr/projection.py:150-167, and for
// combine_t, layergkr/gpu.py:301-308) against a tall B that is streamed once per eight rows of A.  Lanes run along the
// columns of B (coalesced), the inner dimension is split across wavefronts and workgroups so that even a single output
// row fills the GPU, and a second small kernel adds the partial sums of the workgroups.  Products of many rows go to
// the matrix cores (matmul_rns.hip).
#include "common.hpp"
#include "gl_field.hpp"
#include "matmul_rns.hpp"

namespace {

constexpr int BLOCK = 256;

// exact running sum of 64x64-bit products: value = lo + hi*2^64 + wraps*2^128
struct WideAcc {
    u64 lo = 0, hi = 0;
    u32 wraps = 0;
    __device__ __forceinline__ void fma(u64 a, u64 b) {
        u64 pl, ph;
        gl::mul_wide(a, b, pl, ph);
        u64 nl = lo + pl;
        u64 c = nl < pl ? 1 : 0;
        u64 nh = hi + ph;
        u32 w = nh < ph ? 1u : 0u;
        u64 nh2 = nh + c;
        w += nh2 < nh ? 1u : 0u;
        lo = nl;
        hi = nh2;
        wraps += w;
    }
    // 2^128 = 2^96 * 2^32 = -2^32 (mod p)
    __device__ __forceinline__ u64 reduce() const {
        u64 r = gl::reduce128(lo, hi);
        return gl::sub(r, gl::mul((u64)wraps, (u64)1 << 32));
    }
};

// sum of a[l] b[l] with a[l] the same for the whole wavefront, as three 64-bit sums of 32 x 32-bit products (weights 1,
// 2^32, 2^64) and the counts of their wrap-arounds: the multiply-add leaves its carry in a scalar pair and one
// instruction counts it, 8 instructions per term where a 160-bit accumulator takes 13 (the carry has to ripple).  The
// carries are read four instructions after they were written (two wait states are needed).
struct UniformDot {
    u64 lo = 0, mid = 0, hi = 0;
    u32 n_lo = 0, n_mid = 0, n_hi = 0;
    __device__ __forceinline__ void fma(u64 a, u64 b) {
        u64 c0, c1, c2, c3;
        asm("v_mad_u64_u32 %[lo], %[c0], %[a0], %[b0], %[lo]\n\t"
            "v_mad_u64_u32 %[mid], %[c1], %[a0], %[b1], %[mid]\n\t"
            "v_mad_u64_u32 %[hi], %[c2], %[a1], %[b1], %[hi]\n\t"
            "v_mad_u64_u32 %[mid], %[c3], %[a1], %[b0], %[mid]\n\t"
            "v_addc_co_u32 %[n0], %[c0], 0, %[n0], %[c0]\n\t"
            "v_addc_co_u32 %[n1], %[c1], 0, %[n1], %[c1]\n\t"
            "v_addc_co_u32 %[n2], %[c2], 0, %[n2], %[c2]\n\t"
            "v_addc_co_u32 %[n1], %[c3], 0, %[n1], %[c3]"
            : [lo] "+v"(lo), [mid] "+v"(mid), [hi] "+v"(hi), [n0] "+v"(n_lo), [n1] "+v"(n_mid), [n2] "+v"(n_hi), [c0] "=&s"(c0),
              [c1] "=&s"(c1), [c2] "=&s"(c2), [c3] "=&s"(c3)
            : [a0] "s"((u32)a), [a1] "s"((u32)(a >> 32)), [b0] "v"((u32)b), [b1] "v"((u32)(b >> 32)));
    }
    // 2^64 = 2^32 - 1, 2^96 = -1, 2^128 = -2^32 (mod p)
    __device__ __forceinline__ u64 reduce() const {
        u64 r = gl::add(gl::canon(lo), gl::mul(mid, (u64)1 << 32));                  // lo + 2^32 mid
        r = gl::add(r, gl::mul(gl::add(gl::canon(hi), n_lo), gl::EPS));             // + 2^64 (hi + n_lo)
        r = gl::sub(r, n_mid);                                                      // - n_mid
        return gl::sub(r, gl::canon((u64)n_hi << 32));                              // - 2^32 n_hi
    }
};

// partial[s][i][j] = sum over the s-th slice of the inner dimension of A[i][l] * B[l][j]
// A lane owns column j for MB consecutive rows of A, so B is streamed once per MB rows, and requests UN elements of its
// column before it uses the first (one row of A against a 4096 x 65536 B: 5.5 TB/s with eight loads in flight, 4.9 TB/s
// with the loop left to the compiler; with the streaming hint 6.3 TB/s, what a kernel that only reads reaches).
// The slice is divided again over the KS wavefronts of a workgroup, which add up through LDS: a product of few columns
// fills the chip in one launch.
template <int MB, int UN, int KS>
__global__ __launch_bounds__(64 * KS) void k_matmul(const u64 *__restrict__ A, const u64 *__restrict__ B, u64 *__restrict__ out, i64 m, i64 k,
                                                    i64 n, i64 k_per_split) {
    __shared__ u64 part[KS > 1 ? KS : 1][MB][64];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const i64 j = (i64)blockIdx.x * 64 + lane;
    const i64 i0 = (i64)blockIdx.y * MB, s = blockIdx.z;
    const i64 s0 = s * k_per_split, s1 = (s0 + k_per_split < k) ? s0 + k_per_split : k;
    const i64 per = (s1 - s0 + KS - 1) / KS;
    const i64 l0 = s0 + w * per, l1 = (l0 + per < s1) ? l0 + per : s1;
    const int rows = (m - i0 < MB) ? (int)(m - i0) : MB;
    UniformDot acc[MB];
    if (j < n) {
        const u64 *b_col = B + j;
        i64 l = l0;
        for (; l + UN <= l1; l += UN) {
            u64 b[UN];
#pragma unroll
            for (int u = 0; u < UN; ++u) b[u] = __builtin_nontemporal_load(&b_col[(l + u) * n]);
#pragma unroll
            for (int r = 0; r < MB; ++r) {
                const u64 *a = A + (i0 + (r < rows ? r : 0)) * k + l;
#pragma unroll
                for (int u = 0; u < UN; ++u) acc[r].fma(a[u], b[u]);
            }
        }
        for (; l < l1; ++l) {
            const u64 b = b_col[l * n];
#pragma unroll
            for (int r = 0; r < MB; ++r) acc[r].fma(A[(i0 + (r < rows ? r : 0)) * k + l], b);
        }
    }
    if (KS == 1) {
        if (j < n) {
#pragma unroll
            for (int r = 0; r < MB; ++r)
                if (r < rows) out[(s * m + i0 + r) * n + j] = acc[r].reduce();
        }
        return;
    }
#pragma unroll
    for (int r = 0; r < MB; ++r) part[w][r][lane] = acc[r].reduce();
    __syncthreads();
    // row r of the tile is added up by wavefront r mod KS
    for (int r = w; r < rows; r += KS) {
        u64 v = part[0][r][lane];
#pragma unroll
        for (int q = 1; q < KS; ++q) v = gl::add(v, part[q][r][lane]);
        if (j < n) out[(s * m + i0 + r) * n + j] = v;
    }
}

// an empty inner dimension gives the zero matrix (a kernel, not a memset: the call may be under stream capture)
__global__ __launch_bounds__(BLOCK) void k_zero(u64 *__restrict__ out, i64 n) {
    const i64 e = (i64)blockIdx.x * BLOCK + threadIdx.x;
    if (e < n) out[e] = 0;
}

// The sums of the slices: 64 entries per workgroup, the slices dealt over its four wavefronts, eight of them in flight (one thread
// per entry going through all of them: 13 us for 46 slices of 2804 entries, 18 for 64 of 1000; 4 this way).
__global__ __launch_bounds__(BLOCK) void k_add_partials(const u64 *__restrict__ partial, u64 *__restrict__ out, i64 mn, int splits) {
    __shared__ u64 part[BLOCK / 64][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const i64 e = (i64)blockIdx.x * 64 + lane;
    u64 acc = 0;
    if (e < mn) {
        constexpr int UN = 8;
        for (int s0 = w; s0 < splits; s0 += UN * (BLOCK / 64)) {
            u64 v[UN];
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                const int s = s0 + u * (BLOCK / 64);
                v[u] = s < splits ? partial[(i64)s * mn + e] : 0;
            }
#pragma unroll
            for (int u = 0; u < UN; ++u) acc = gl::add(acc, v[u]);
        }
    }
    part[w][lane] = acc;
    __syncthreads();
    if (w == 0 && e < mn) out[e] = gl::add(gl::add(part[0][lane], part[1][lane]), gl::add(part[2][lane], part[3][lane]));
}

// TPR threads per row of M (a wavefront, or the whole workgroup when there are too few rows for a wavefront
// each to fill the GPU): they stride over the columns with four row elements requested before the first is
// used, exact accumulation, shuffle tree, and for a workgroup a last sum over its wavefronts in LDS.
// 1024 x 262144: 2.01 ms with a wavefront per row and one load in flight, 0.72 ms with four, TPR = 256 below.
// The matrix is read once, with the streaming hint (4096 x 65536: 4.7 -> 4.8 TB/s, 65536 x 4096: 5.0 -> 5.2 TB/s).
template <int TPR>
__global__ __launch_bounds__(BLOCK) void k_matvec(const u64 *__restrict__ M, const u64 *__restrict__ v, u64 *__restrict__ w, i64 m, i64 n) {
    __shared__ u64 part[BLOCK / 64];
    const int lane = threadIdx.x & 63, t = threadIdx.x & (TPR - 1);
    const i64 row = ((i64)blockIdx.x * BLOCK + threadIdx.x) / TPR;
    u64 x = 0;
    if (row < m) {
        const u64 *r = M + row * n;
        WideAcc acc;
        i64 j = t;
        for (; j + 3 * TPR < n; j += 4 * TPR) {
            u64 a[4], b[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) { a[u] = __builtin_nontemporal_load(&r[j + u * TPR]); b[u] = v[j + u * TPR]; }
#pragma unroll
            for (int u = 0; u < 4; ++u) acc.fma(a[u], b[u]);
        }
        for (; j < n; j += TPR) acc.fma(r[j], v[j]);
        x = acc.reduce();
    }
    for (int off = 32; off > 0; off >>= 1) x = gl::add(x, __shfl_xor(x, off, 64));
    if (TPR == 64) {
        if (lane == 0 && row < m) w[row] = x;
    } else {
        if (lane == 0) part[threadIdx.x >> 6] = x;
        __syncthreads();
        if (threadIdx.x == 0 && row < m) {
            u64 sum = part[0];
            for (int i = 1; i < BLOCK / 64; ++i) sum = gl::add(sum, part[i]);
            w[row] = sum;
        }
    }
}

// out[r][p] = sum_i coeffs[r][i] x_p^i by Horner's rule (prover/kernels/gl_extras.cuh:93-108)
__global__ __launch_bounds__(BLOCK) void k_poly_eval(const u64 *__restrict__ coeffs, i64 m, i64 d, const u64 *__restrict__ points, i64 kp,
                                                     u64 *__restrict__ out) {
    const i64 p = (i64)blockIdx.x * BLOCK + threadIdx.x;
    const i64 r = blockIdx.y;
    if (p >= kp) return;
    const u64 x = points[p];
    const u64 *row = coeffs + r * d;
    u64 acc = 0;
    for (i64 i = d - 1; i >= 0; --i) acc = gl::add(gl::mul(acc, x), row[i]);
    out[r * kp + p] = acc;
}

// How a product on the VALU is cut up: rows of A a lane takes together (mb), wavefronts of a workgroup along the inner
// dimension (ks), and slices of it over workgroups (splits), whose partial sums a second launch adds up.  The rows are dealt
// evenly over as few blocks of at most eight as there have to be, so that B is read no more often than that and no row is computed
// twice (3 x 4096 x 16384: 161 -> 91 us, which two rows to a lane read twice; 5 rows 179 -> 109; 9 x 12000 x 12000, two blocks of 8,
// 643 -> 427; seven rows to a lane are slower than
// eight, 20 x 12000 x 12000 1205 against 945, and seven rows alone fastest as four and three).  About 8192
// wavefronts in all, eight to a SIMD, with at least 16 terms each (4096 and 16384 measured within 10 % of it from one row
// to 32, 32768 up to 25 % slower; 4096 is up to 15 % faster at 10 M entries of B and 40 % slower at 288 M); fewer rows to a
// lane while even so there would be less than two wavefronts to a SIMD
// (24 x 760 x 1070: 21 -> 18 us).  One row against 32768 columns or more streams fastest with one wavefront to a workgroup
// (1 x 4096 x 65536: 312 us, 6.9 TB/s; 360 us with four along the inner dimension); everything else takes four (12 x 4096
// x 4096: 90 us, 103 with sixteen, which saves the second launch now and then but leaves CUs idle).
struct DirectPlan {
    int mb, ks, splits;
};
DirectPlan plan_direct(i64 m, i64 k, i64 n) {
    DirectPlan D;
    const i64 cols = (n + 63) / 64, most = k / 16 > 1 ? k / 16 : 1;
    const i64 blocks = (m + 7) / 8;
    D.mb = (int)((m + blocks - 1) / blocks);
    if (D.mb == 7) D.mb = m == 7 ? 4 : 8;
    while (D.mb > 1 && cols * ((m + D.mb - 1) / D.mb) * most < 4096) D.mb = (D.mb + 1) / 2;
    i64 want = 8192 / (cols * ((m + D.mb - 1) / D.mb));
    if (want > most) want = most;
    D.ks = (m == 1 && cols >= 512) || want < 3 ? 1 : 4;
    const i64 splits = want / D.ks;
    D.splits = (int)(splits < 1 ? 1 : (splits > 64 ? 64 : splits));
    if (D.ks > 1 && D.splits == 2) D.splits = 1;           // a second launch for twice the wavefronts does not pay
    return D;
}

template <int MB, int UN>
void launch_direct(const DirectPlan &D, const u64 *A, const u64 *B, u64 *dst, i64 m, i64 k, i64 n, hipStream_t s) {
    const i64 per = (k + D.splits - 1) / D.splits;
    dim3 grid((unsigned)((n + 63) / 64), (unsigned)((m + MB - 1) / MB), (unsigned)D.splits);
    if (D.ks == 4) hipLaunchKernelGGL((k_matmul<MB, UN, 4>), grid, dim3(256), 0, s, A, B, dst, m, k, n, per);
    else hipLaunchKernelGGL((k_matmul<MB, UN, 1>), grid, dim3(64), 0, s, A, B, dst, m, k, n, per);
}

}  // namespace

extern "C" {

size_t vi_gl_matmul_workspace_bytes(int64_t m, int64_t k, int64_t n) {
    if (m <= 0 || k <= 0 || n <= 0) return 0;
    if (vi::rns_matmul_pays(m, k, n)) return vi::rns_matmul_workspace_bytes(m, k, n);
    const int s = plan_direct(m, k, n).splits;
    return s > 1 ? (size_t)s * (size_t)m * (size_t)n * sizeof(u64) : 0;
}

int vi_gl_matmul(const uint64_t *A, const uint64_t *B, uint64_t *C, int64_t m, int64_t k, int64_t n, void *ws,
                 size_t ws_bytes, void *stream) {
    if (m < 0 || k < 0 || n < 0) return vi::fail(VI_EINVAL, "vi_gl_matmul: negative dimension");
    if (m == 0 || n == 0) return VI_OK;
    if (!C || (k > 0 && (!A || !B))) return vi::fail(VI_EINVAL, "vi_gl_matmul: null pointer");
    if (m > 65535) return vi::fail(VI_EINVAL, "vi_gl_matmul: at most 65535 rows of A per call, got %lld", (long long)m);
    hipStream_t s = (hipStream_t)stream;
    if (k == 0) {
        const i64 mn = m * n;
        hipLaunchKernelGGL(k_zero, dim3((unsigned)((mn + BLOCK - 1) / BLOCK)), dim3(BLOCK), 0, s, C, mn);
        VI_LAUNCH_CHECK("k_zero");
        return VI_OK;
    }
    if (vi::rns_matmul_pays(m, k, n)) {
        const size_t need = vi::rns_matmul_workspace_bytes(m, k, n);
        if (!ws || ws_bytes < need) return vi::fail(VI_ENOMEM, "vi_gl_matmul: workspace below %zu bytes", need);
        return vi::rns_matmul(A, B, C, m, k, n, ws, s);
    }
    const DirectPlan D = plan_direct(m, k, n);
    const int splits = D.splits;
    if (splits > 1 && (!ws || ws_bytes < vi_gl_matmul_workspace_bytes(m, k, n)))
        return vi::fail(VI_ENOMEM, "vi_gl_matmul: workspace below %zu bytes", vi_gl_matmul_workspace_bytes(m, k, n));
    u64 *dst = splits > 1 ? (u64 *)ws : C;
    switch (D.mb) {
        case 1: launch_direct<1, 8>(D, A, B, dst, m, k, n, s); break;
        case 2: launch_direct<2, 8>(D, A, B, dst, m, k, n, s); break;
        case 3: launch_direct<3, 8>(D, A, B, dst, m, k, n, s); break;
        case 4: launch_direct<4, 8>(D, A, B, dst, m, k, n, s); break;
        case 5: launch_direct<5, 8>(D, A, B, dst, m, k, n, s); break;
        case 6: launch_direct<6, 8>(D, A, B, dst, m, k, n, s); break;
        default: launch_direct<8, 8>(D, A, B, dst, m, k, n, s); break;
    }
    VI_LAUNCH_CHECK("k_matmul");
    if (splits > 1) {
        const i64 mn = m * n;
        hipLaunchKernelGGL(k_add_partials, dim3((unsigned)((mn + 63) / 64)), dim3(BLOCK), 0, s, (const u64 *)ws, C, mn, splits);
        VI_LAUNCH_CHECK("k_add_partials");
    }
    return VI_OK;
}

int vi_gl_matvec(const uint64_t *M, const uint64_t *v, uint64_t *w, int64_t m, int64_t n, void *stream) {
    if (m < 0 || n < 0) return vi::fail(VI_EINVAL, "vi_gl_matvec: negative dimension");
    if (m == 0) return VI_OK;
    if (!w || (n > 0 && (!M || !v))) return vi::fail(VI_EINVAL, "vi_gl_matvec: null pointer");
    const bool wide = m < 8192 && n >= 4096;          // few long rows: a workgroup per row
    const i64 blocks = wide ? m : (m * 64 + BLOCK - 1) / BLOCK;
    if (blocks > 0x7FFFFFFF) return vi::fail(VI_EINVAL, "vi_gl_matvec: too many rows");
    if (wide) hipLaunchKernelGGL(k_matvec<BLOCK>, dim3((unsigned)blocks), dim3(BLOCK), 0, (hipStream_t)stream, M, v, w, (i64)m, (i64)n);
    else hipLaunchKernelGGL(k_matvec<64>, dim3((unsigned)blocks), dim3(BLOCK), 0, (hipStream_t)stream, M, v, w, (i64)m, (i64)n);
    VI_LAUNCH_CHECK("k_matvec");
    return VI_OK;
}

int vi_poly_eval(const uint64_t *coeffs, int64_t m, int64_t d, const uint64_t *points, int64_t k, uint64_t *out,
                 void *stream) {
    if (m < 0 || d < 0 || k < 0) return vi::fail(VI_EINVAL, "vi_poly_eval: negative dimension");
    if (m == 0 || k == 0) return VI_OK;
    if (!out || !points || (d > 0 && !coeffs)) return vi::fail(VI_EINVAL, "vi_poly_eval: null pointer");
    if (m > 65535) return vi::fail(VI_EINVAL, "vi_poly_eval: at most 65535 polynomials per call, got %lld", (long long)m);
    dim3 grid((unsigned)((k + BLOCK - 1) / BLOCK), (unsigned)m);
    hipLaunchKernelGGL(k_poly_eval, grid, dim3(BLOCK), 0, (hipStream_t)stream, coeffs, (i64)m, (i64)d, points, (i64)k, out);
    VI_LAUNCH_CHECK("k_poly_eval");
    return VI_OK;
}

}  // extern "C"
