// Transforms and coset extensions of few short rows: one launch, four points per thread.
//
// k_ntt_fast and its relatives give a thread sixteen points, which is right when every SIMD has wavefronts to choose
// from.  A batch that does not fill the chip waits for ONE wavefront's chain instead: two 16-point transforms, two trips
// to memory for twiddles and a trip through LDS, 8 to 12 us per launch however little there is to do.  Here a row of
// N <= 4096 points is spread over N / 4 threads: radix-4 levels through LDS, each a dozen dependent instructions deep, with
// every twiddle of the thread requested together with the data.  An extension keeps its coefficients in registers
// between the inverse and the forward transform: decimation in frequency leaves a thread the four consecutive slots
// (bit-reversed coefficients) that decimation in time starts from, so there is no reordering in between.
//
// A SIMD has one or two wavefronts here, so a chain's length is what counts, and a thread's butterflies and products go two at once
// (gl::bfly2, gl::mul2).  One at a time the corrections by multiply-adds were the longer chains: extensions of 2^7 points by two, 2^20 points, 11.6 us
// with corrections by additions and 12.1, by four 14.8 and 15.4.  us, calls in a queue, additions one at a time -> multiply-adds two at
// once: 2^7 by two, 2^20 points, 11.2 -> 10.9, by four 14.4 -> 13.1, 2^8 by four 15.7 -> 13.1, 2^10 by two 16.7 -> 15.6; 12 rows of 2^7 by two 6.2 -> 5.9;
// a first pass over sixteen rows of 2^12 4.67 -> 4.37, the last the same; 2^18 points as passes 13.2 -> 12.7.
//
// Rows of more points take the passes of ntt_plan.hpp, digit by digit, with the same four points per thread (k_small_pass): a
// launch takes 4.3 us where one of k_ntt_fast takes 8, and the cosets of an extension run side by side.  One row of 2^16
// extended to 2^18: 57 -> 21 us; 16 rows of 2^12 transformed, calls in a queue: 11.6 -> 8.6 us (two launches where k_ntt_row is
// one: a program that transforms them there and back with a copy in between takes 25 us either way).
#pragma once

namespace {

constexpr int SMALL_MIN_LOG = 3, SMALL_MAX_LOG = 12;

// LOGN: log2 of the row length
template <int LOGN>
struct SmallShape {
    static constexpr int N = 1 << LOGN, TR = N / 4;                    // threads per row
    static constexpr int WG = TR < 256 ? 256 : TR, ROWS = WG / TR;     // workgroup, and rows it holds
    static constexpr int PITCH = N + N / 16 + 1;                       // LDS words per row
    static constexpr int LEVELS = (LOGN + 1) / 2;
};

// slot s of a row in LDS: one word of padding every sixteen
__device__ __forceinline__ int small_pad(int s) { return s + (s >> 4); }

// every thread's LDS writes before any later read; rows of up to 256 points live inside one wavefront, whose LDS accesses
// are in order, unless their threads are dealt over the workgroup (SPREAD)
template <int LOGN, bool SPREAD = false>
__device__ __forceinline__ void small_sync() {
    if (SPREAD || SmallShape<LOGN>::TR > 64) __syncthreads();
    else {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// span of level l (0 = first) of the decimation in frequency; an odd LOGN starts with a radix-2 level
template <int LOGN>
constexpr int small_span(int l) {
    return (LOGN & 1) ? (l == 0 ? 1 << LOGN : (1 << (LOGN + 1)) >> (2 * l)) : (1 << LOGN) >> (2 * l);
}

// The twiddles w_L^j, w_L^2j, w_L^3j of a thread at every level with one (w: w_4096^e at [e], 4096 entries).
template <int LOGN>
struct SmallTwiddles {
    u64 w[SmallShape<LOGN>::LEVELS][3];
    __device__ __forceinline__ void load(const u64 *__restrict__ tab, int t) {
        static_for<0, SmallShape<LOGN>::LEVELS>([&](auto l_) {
            constexpr int l = decltype(l_)::value, L = small_span<LOGN>(l), step = 4096 / L;
            if constexpr ((LOGN & 1) && l == 0) {
                w[l][0] = tab[t * step];
            } else if constexpr (L > 4) {
                const int j = t & (L / 4 - 1);
                w[l][0] = tab[j * step];
                w[l][1] = tab[2 * j * step];
                w[l][2] = tab[3 * j * step];
            }
        });
    }
};

// v w_4, w_4 = 2^48 (inverse transform: w_4^-1 = -2^48, so the caller's sum and difference change places)
__device__ __forceinline__ u64 small_i(u64 v) { return gl::mul_pow2c<48>(v); }

// slot of element c of thread t at a level of span L
template <int L>
__device__ __forceinline__ int small_slot(int t, int c) {
    constexpr int Q = L / 4;
    return (t / Q) * L + (t & (Q - 1)) + c * Q;
}

// Decimation in frequency over a row: x[c] = point t + c N / 4 on entry, slot 4 t + c of the bit-reversed result on return.
template <int LOGN, bool INV, bool SPREAD = false>
__device__ __forceinline__ void small_dif(u64 (&x)[4], const SmallTwiddles<LOGN> &W, int t, u64 *row) {
    constexpr int LEVELS = SmallShape<LOGN>::LEVELS, N = SmallShape<LOGN>::N;
    static_for<0, LEVELS>([&](auto l_) {
        constexpr int l = decltype(l_)::value, L = small_span<LOGN>(l);
        if constexpr ((LOGN & 1) && l == 0) {
            // (x0, x2) and (x1, x3) with w^t and w^(t + N/4) = w_4 w^t
            u64 s0, d0, s1, d1;
            gl::bfly2(x[0], x[2], s0, d0, x[1], x[3], s1, d1);
            if constexpr (INV) d1 = gl::neg(d1);
            x[0] = s0;
            x[1] = s1;
            gl::mul2(d0, W.w[l][0], x[2], small_i(d1), W.w[l][0], x[3]);
        } else {
            u64 s0, d0, s1, d1;
            gl::bfly2(x[0], x[2], s0, d0, x[1], x[3], s1, d1);
            d1 = small_i(d1);
            u64 y1, y3;
            // outputs 0 and 2 mod 4 of the span, and 1 and 3
            gl::bfly2(s0, s1, x[0], x[1], d0, d1, INV ? y3 : y1, INV ? y1 : y3);
            x[2] = y1;
            x[3] = y3;
            if constexpr (L > 4) {
                gl::mul2(x[1], W.w[l][1], x[1], x[2], W.w[l][0], x[2]);
                x[3] = gl::mul(x[3], W.w[l][2]);
            }
        }
        if constexpr (l + 1 < LEVELS) {
            // the radix-2 level's elements lie as those of a span N
            constexpr int LW = (LOGN & 1) && l == 0 ? N : L, LR = small_span<LOGN>(l + 1);
#pragma unroll
            for (int c = 0; c < 4; ++c) row[small_pad(small_slot<LW>(t, c))] = x[c];
            small_sync<LOGN, SPREAD>();
#pragma unroll
            for (int c = 0; c < 4; ++c) x[c] = row[small_pad(small_slot<LR>(t, c))];
        }
    });
}

// Decimation in time, forward: x[c] = slot 4 t + c of bit-reversed points on entry, point t + c N / 4 on return.
template <int LOGN>
__device__ __forceinline__ void small_dit(u64 (&x)[4], const SmallTwiddles<LOGN> &W, int t, u64 *row) {
    constexpr int LEVELS = SmallShape<LOGN>::LEVELS, N = SmallShape<LOGN>::N;
    static_for<0, LEVELS>([&](auto b_) {
        constexpr int l = LEVELS - 1 - decltype(b_)::value, L = small_span<LOGN>(l);
        if constexpr ((LOGN & 1) && l == 0) {
            u64 o0, o1, s0, d0, s1, d1;
            gl::mul2(x[2], W.w[l][0], o0, x[3], W.w[l][0], o1);
            gl::bfly2(x[0], o0, s0, d0, x[1], small_i(o1), s1, d1);
            x[0] = s0;
            x[1] = s1;
            x[2] = d0;
            x[3] = d1;
        } else {
            // the quarters of a span hold the points 0, 2, 1, 3 mod 4
            u64 t2 = x[1], t1 = x[2], t3 = x[3];
            if constexpr (L > 4) {
                gl::mul2(t1, W.w[l][0], t1, t3, W.w[l][2], t3);
                t2 = gl::mul(t2, W.w[l][1]);
            }
            u64 s0, d0, s1, d1;
            gl::bfly2(x[0], t2, s0, d0, t1, t3, s1, d1);
            gl::bfly2(s0, s1, x[0], x[2], d0, small_i(d1), x[1], x[3]);
        }
        if constexpr (l > 0) {
            constexpr int LW = L, LR = (LOGN & 1) && l == 1 ? N : small_span<LOGN>(l - 1);
#pragma unroll
            for (int c = 0; c < 4; ++c) row[small_pad(small_slot<LW>(t, c))] = x[c];
            small_sync<LOGN>();
#pragma unroll
            for (int c = 0; c < 4; ++c) x[c] = row[small_pad(small_slot<LR>(t, c))];
        }
    });
}

__device__ __forceinline__ int small_brev(int s, int bits) { return (int)(__brev((u32)s) >> (32 - bits)); }

// In-place transform of m rows: natural order in and out.
template <int LOGN, bool INV>
__global__ __launch_bounds__(SmallShape<LOGN>::WG) void k_small_ntt(u64 *rows, i64 m, const u64 *__restrict__ tab, u64 scale) {
    using S = SmallShape<LOGN>;
    __shared__ u64 lds[S::ROWS * S::PITCH];
    const int t = threadIdx.x & (S::TR - 1), r = threadIdx.x / S::TR;
    const i64 row = (i64)blockIdx.x * S::ROWS + r;
    const bool there = row < m;
    u64 *p = rows + row * S::N, *mine = lds + r * S::PITCH;
    u64 x[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) x[c] = there ? p[t + c * S::TR] : 0;
    SmallTwiddles<LOGN> W;
    W.load(tab, t);
#pragma unroll
    for (int c = 0; c < 4; ++c) x[c] = gl::canon(x[c]);
    small_dif<LOGN, INV>(x, W, t, mine);
    // slots back to natural order through LDS, so that the stores are contiguous
    small_sync<LOGN>();
#pragma unroll
    for (int c = 0; c < 4; ++c) mine[small_pad(4 * t + c)] = x[c];
    small_sync<LOGN>();
#pragma unroll
    for (int c = 0; c < 4; ++c) x[c] = mine[small_pad(small_brev(t + c * S::TR, LOGN))];
    if constexpr (INV) {
#pragma unroll
        for (int c = 0; c < 4; c += 2) gl::mul2(x[c], scale, x[c], x[c + 1], scale, x[c + 1]);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
        if (there) p[t + c * S::TR] = x[c];
}

struct SmallLde {
    const u64 *in;                             // values at w_K^c, or coefficients when COEFFS
    i64 m, width, in_stride;
    u64 *coeffs;                               // where the coefficients go, or null
    i64 coeffs_stride;
    u64 *out;                                  // codewords, or null
    i64 out_stride;
    const u64 *tab_inv, *tab_fwd, *pre;        // w_4096^-e, w_4096^e, (shift w_N^t)^i at [t][i]
    u64 scale;                                 // 1 / K
    int log_rho, cosets;                       // cosets a workgroup takes: 1, or all when the coefficients overwrite `in`
};

// Coset extension of m rows of K = 2^LOGN points: a workgroup per group of rows and coset, each with its own inverse
// transform (cheap here, and nothing is handed over).
template <int LOGN, bool COEFFS>
__global__ __launch_bounds__(SmallShape<LOGN>::WG) void k_small_lde(const SmallLde A) {
    using S = SmallShape<LOGN>;
    __shared__ u64 lds[S::ROWS * S::PITCH];
    const int t = threadIdx.x & (S::TR - 1), r = threadIdx.x / S::TR;
    const int log_groups = A.cosets == 1 ? A.log_rho : 0;              // workgroups per group of rows, log2
    const i64 row = (i64)(blockIdx.x >> log_groups) * S::ROWS + r;
    const int first = A.cosets == 1 ? (int)(blockIdx.x & ((1u << log_groups) - 1)) : 0;
    const bool there = row < A.m;
    u64 *mine = lds + r * S::PITCH;
    const u64 *src = A.in + row * A.in_stride;
    u64 coef[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int i = COEFFS ? small_brev(4 * t + c, LOGN) : t + c * S::TR;
        coef[c] = there && i < A.width ? src[i] : 0;
    }
    SmallTwiddles<LOGN> F;
    F.load(A.tab_fwd, t);
    if constexpr (!COEFFS) {
        SmallTwiddles<LOGN> W;
        W.load(A.tab_inv, t);
#pragma unroll
        for (int c = 0; c < 4; ++c) coef[c] = gl::canon(coef[c]);
        small_dif<LOGN, true>(coef, W, t, mine);
#pragma unroll
        for (int c = 0; c < 4; c += 2) gl::mul2(coef[c], A.scale, coef[c], coef[c + 1], A.scale, coef[c + 1]);
        if (A.coeffs && first == 0 && there) {
#pragma unroll
            for (int c = 0; c < 4; ++c) A.coeffs[row * A.coeffs_stride + small_brev(4 * t + c, LOGN)] = coef[c];
        }
    } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) coef[c] = gl::canon(coef[c]);
    }
    if (!A.out) return;
    for (int k = first; k < first + A.cosets; ++k) {
        u64 x[4];
#pragma unroll
        for (int c = 0; c < 4; c += 2) {
            const u64 *pre = A.pre + ((i64)k << LOGN);
            gl::mul2(coef[c], pre[small_brev(4 * t + c, LOGN)], x[c], coef[c + 1], pre[small_brev(4 * t + c + 1, LOGN)], x[c + 1]);
        }
        small_sync<LOGN>();                                            // the transform before this one has read the row
        small_dit<LOGN>(x, F, t, mine);
        if (there) {
            u64 *o = A.out + row * A.out_stride + k;
#pragma unroll
            for (int c = 0; c < 4; ++c) o[(i64)(t + c * S::TR) << A.log_rho] = x[c];
        }
    }
}

// One pass (digit of 2^A points, PassArgs of ntt_pass.hpp) of a transform whose rows are too long for the single launch, in
// batches that leave the chip idle: the same four points per thread, 1024 points and so many columns per workgroup.  A
// non-final pass deals the threads of a sub-transform over the workgroup, so that neighbouring lanes read neighbouring
// columns; a final pass reads its contiguous digits row by row.  Both store along the columns, through LDS.  The cosets of a
// first forward pass are workgroups of their own.
template <int A>
struct SmallPassShape {
    static constexpr int N = 1 << A, TR = N / 4, COLS = 256 / TR, PITCH = N + N / 16 + 1;
};

template <int A, bool INV, bool FINAL>
__global__ __launch_bounds__(256) void k_small_pass(const PassArgs P, const u64 *__restrict__ full) {
    using S = SmallPassShape<A>;
    __shared__ u64 lds[S::COLS * S::PITCH];
    const int tid = threadIdx.x;
    const int t = FINAL ? tid & (S::TR - 1) : tid / S::COLS, c = FINAL ? tid / S::TR : tid & (S::COLS - 1);
    const i64 g0 = (i64)blockIdx.x * S::COLS, coset = blockIdx.y;
    const int lc = P.B + (FINAL ? P.log_rho : P.logR);                 // columns per row, log2
    u64 *mine = lds + c * S::PITCH;

    // gather: element l of the column at src[base + idx0 + l * step]
    const i64 g = g0 + c, row = g >> lc, col = g & (((i64)1 << lc) - 1);
    i64 base = row * P.src_row_stride, idx0, step;
    if (FINAL) {
        base += (col & (((i64)1 << P.log_rho) - 1)) * P.src_coset_stride;
        idx0 = storage_prefix(P, col >> P.log_rho) << A;
        step = 1;
    } else {
        idx0 = ((col >> P.logR) << (A + P.logR)) + (col & (((i64)1 << P.logR) - 1));
        step = (i64)1 << P.logR;
    }
    u64 x[4], f[4], w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const i64 idx = idx0 + (t + i * S::TR) * step;
        x[i] = row < P.n_rows && idx < P.src_width ? P.src[base + idx] : 0;
        if (!FINAL) f[i] = P.pre ? P.pre[(coset << P.logn) + idx] : 1;
    }
    // scatter: column oc of the workgroup, outputs k0 + i * 256 / COLS; the inter-pass twiddles are requested here
    const int oc = tid & (S::COLS - 1), k0 = tid / S::COLS;
    const i64 og = g0 + oc, orow = og >> lc, ocol = og & (((i64)1 << lc) - 1);
    const i64 r = ocol & (((i64)1 << P.logR) - 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = FINAL ? P.scale : P.tw[((i64)(k0 + i * S::TR) << P.logR) + r];
    SmallTwiddles<A> W;
    W.load(full, t);

    if (P.canon_src) {
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = gl::canon(x[i]);
    }
    if (!FINAL && P.pre) {
#pragma unroll
        for (int i = 0; i < 4; i += 2) gl::mul2(x[i], f[i], x[i], x[i + 1], f[i + 1], x[i + 1]);
    }
    small_dif<A, INV, !FINAL>(x, W, t, mine);
#pragma unroll
    for (int i = 0; i < 4; ++i) mine[small_pad(4 * t + i)] = x[i];      // the slots this thread read last
    __syncthreads();
    if (orow >= P.n_rows) return;
    u64 *o = P.dst + orow * P.dst_row_stride;
    if (!FINAL) o += coset * P.dst_coset_stride + ((ocol >> P.logR) << (A + P.logR)) + r;
    else o += ocol;
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = lds[oc * S::PITCH + small_pad(small_brev(k0 + i * S::TR, A))];
    if (!FINAL || P.scale != 1) {
#pragma unroll
        for (int i = 0; i < 4; i += 2) gl::mul2(x[i], w[i], x[i], x[i + 1], w[i + 1], x[i + 1]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) o[(i64)(k0 + i * S::TR) << (FINAL ? lc : P.logR)] = x[i];
}

template <int A>
void launch_small_pass(const PassArgs &P, const u64 *full, hipStream_t s) {
    const i64 cols = P.n_rows << (P.is_final ? P.B + P.log_rho : P.B + P.logR);
    const dim3 grid((unsigned)((cols + SmallPassShape<A>::COLS - 1) / SmallPassShape<A>::COLS), !P.is_final && P.loop_cosets ? 1u << P.log_rho : 1u);
    switch ((P.inverse ? 2 : 0) + (P.is_final ? 1 : 0)) {
        case 0: hipLaunchKernelGGL((k_small_pass<A, false, false>), grid, dim3(256), 0, s, P, full); break;
        case 1: hipLaunchKernelGGL((k_small_pass<A, false, true>), grid, dim3(256), 0, s, P, full); break;
        case 2: hipLaunchKernelGGL((k_small_pass<A, true, false>), grid, dim3(256), 0, s, P, full); break;
        default: hipLaunchKernelGGL((k_small_pass<A, true, true>), grid, dim3(256), 0, s, P, full); break;
    }
}

template <int LOGN>
void launch_small_ntt(u64 *rows, i64 m, const u64 *tab, u64 scale, bool inv, hipStream_t s) {
    const dim3 grid((unsigned)((m + SmallShape<LOGN>::ROWS - 1) / SmallShape<LOGN>::ROWS)), block(SmallShape<LOGN>::WG);
    if (inv) hipLaunchKernelGGL((k_small_ntt<LOGN, true>), grid, block, 0, s, rows, m, tab, scale);
    else hipLaunchKernelGGL((k_small_ntt<LOGN, false>), grid, block, 0, s, rows, m, tab, scale);
}

template <int LOGN>
void launch_small_lde(const SmallLde &A, bool coeffs_in, hipStream_t s) {
    const unsigned groups = (unsigned)((A.m + SmallShape<LOGN>::ROWS - 1) / SmallShape<LOGN>::ROWS);
    const dim3 grid(A.cosets == 1 ? groups << A.log_rho : groups), block(SmallShape<LOGN>::WG);
    if (coeffs_in) hipLaunchKernelGGL((k_small_lde<LOGN, true>), grid, block, 0, s, A);
    else hipLaunchKernelGGL((k_small_lde<LOGN, false>), grid, block, 0, s, A);
}

// dispatch over the row length: f(std::integral_constant<int, LOGN>)
template <class F>
void small_dispatch(int logn, F f) {
    switch (logn) {
        case 3: f(std::integral_constant<int, 3>()); break;
        case 4: f(std::integral_constant<int, 4>()); break;
        case 5: f(std::integral_constant<int, 5>()); break;
        case 6: f(std::integral_constant<int, 6>()); break;
        case 7: f(std::integral_constant<int, 7>()); break;
        case 8: f(std::integral_constant<int, 8>()); break;
        case 9: f(std::integral_constant<int, 9>()); break;
        case 10: f(std::integral_constant<int, 10>()); break;
        case 11: f(std::integral_constant<int, 11>()); break;
        default: f(std::integral_constant<int, 12>()); break;
    }
}

}  // namespace
