// Sumcheck proofs of a sum under a common factor, three rounds per pass:
//
//     S = common * ( c0 + sum_j d_j L_j + sum_k c_k A_k B_k )
//
// which is what the batched gate check of a layer comes to (layergkr/relations.py:104-124: eq(z, .) times products of two tables,
// a hadamard or booleanity gate, and many single tables).  As in sumcheck_fast.hpp the challenges are known before the first launch
// and the eight entries i + c n / 8 of a table are closed under three rounds of folding.  The terms are dealt over rows of
// workgroups: a row holds one product, or a few of the single tables, and the common factor.  Its samples are sums over its own
// terms and add up with those of the other rows, so a thread's walk is three tables long whatever the number of terms.
//
//   k_sum3      a pass: three rounds, an eighth of the entries written.  The single tables of a row become one table,
//               Lambda = sum_j d_j L_j, which is folded like any other (folding is linear), in the first pass.
//   k_sum_tail  the last rounds, from 512 entries or fewer on: a wavefront per row, its entries in registers, eight to a lane for
//               up to three rounds and one to a lane for the last six, partners fetched by lane shuffles
//   k_finish    sums of the rows, claims, samples (sumcheck_fast.hpp)
//
// What bounds it.  15 gates of 2^18 entries (40 tables, 8 products, 29 single tables): 82 us in five launches where a launch or two per
// round took 218 in 24.  The first pass 30 (84 MB read at 2.8 TB/s; its instructions are 14 us at the issue rate, and twelve rows read the
// common factor again), two passes of 11 and 10, the tail 18 and k_finish 12: those are a wavefront's chain of loads and some 1,300
// dependent instructions each, whatever the size.  Whole proofs through prove_terms, before -> after: these gates at 2^10 147 -> 101 us, at
// 2^14 200 -> 111, at 2^22 848 -> 662; two hadamard gates (7 tables) at 2^22 425 -> 198; 97 tables with 18 products at 2^22 1653 -> 1446.
#pragma once

namespace {

constexpr int SUM_PRODUCTS = 64;            // products a descriptor holds
constexpr int SUM_SINGLES = 128;            // single tables a descriptor holds
constexpr int SUM_ROW_SINGLES = 4, SUM_ROW_SINGLES_LONG = 8;          // single tables of a row, more where that would be too many rows
constexpr int SUM_SINGLE_ROWS = 16;
constexpr i64 SUM_TAIL = 512;               // entries per table that the tail takes

struct SumDesc {
    const u64 *common;
    u64 *common_dst;                        // written by row 0
    // row n_single_rows + k: product k
    const u64 *a[SUM_PRODUCTS], *b[SUM_PRODUCTS];
    u64 *a_dst[SUM_PRODUCTS], *b_dst[SUM_PRODUCTS];         // NULL: another row writes this table
    u64 coeff[SUM_PRODUCTS];
    // rows below n_single_rows: tables per_row r .. of the list, and their sum
    const u64 *single[SUM_SINGLES];
    u64 single_coeff[SUM_SINGLES];
    u64 *single_dst[SUM_SINGLE_ROWS];
    u64 c0;                                 // belongs to row 0
    int n_products, n_singles, n_single_rows, per_row, n_rows;
};

// Entries i + c cols, c < entries, of a table as they are there, and taken as residues (FIRST: caller data, any 64-bit word).  Apart, so that a
// thread asks for all its words before it looks at one: canon_all() ends in a branch, in front of which the words of its table are waited
// for, and the scheduler puts every load of a sum in front of its use otherwise (24 gates of 2^20, first pass 192 -> 131 us; 15 of 2^18 29.3 -> 28).
__device__ __forceinline__ void request(const u64 *f, i64 i, i64 cols, int entries, u64 (&v)[8]) {
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] = c < entries ? f[i + c * cols] : 0;
}
template <bool FIRST>
__device__ __forceinline__ void take(u64 (&v)[8]) {
    if (FIRST) canon_all(v);
}
// the same of the sum of a row's single tables: plain integers of five words, reduced once
__device__ __forceinline__ void load_singles(const SumDesc &D, int row, i64 i, i64 cols, int entries, u64 (&v)[8]) {
    gl::Wide sum[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) gl::wide_zero(sum[c]);
    const int k0 = row * D.per_row, k1 = min(D.n_singles, k0 + D.per_row);
    u64 w[8], y[8];
    if (k0 < k1) request(D.single[k0], i, cols, entries, w);
    for (int k = k0; k < k1; k += 2) {                     // a table's words on their way while those of the one before are added
        const bool two = k + 1 < k1;
        request(D.single[two ? k + 1 : k], i, cols, entries, y);
        VI_SCHED_FENCE();
        const u64 d = D.single_coeff[k], e = two ? D.single_coeff[k + 1] : 0;
#pragma unroll
        for (int c = 0; c < 8; c += 2) gl::wide_mul_acc2(sum[c], d, w[c], sum[c + 1], d, w[c + 1]);
        VI_SCHED_FENCE();
        if (k + 2 < k1) request(D.single[k + 2], i, cols, entries, w);
        VI_SCHED_FENCE();
#pragma unroll
        for (int c = 0; c < 8; c += 2) gl::wide_mul_acc2(sum[c], e, y[c], sum[c + 1], e, y[c + 1]);
    }
    const u64 c0 = row == 0 ? D.c0 : 0;
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] = gl::addc(gl::wide_reduce(sum[c]), c0);
}

// part: three regions of gridDim.x * n_rows rows of NSAMP words, one per round.  A row of workgroups behind those of the terms adds up
// the regions of the pass before.
template <bool FIRST, bool ONE>
__global__ __launch_bounds__(BLOCK) void k_sum3(const SumDesc D, i64 cols, u64 r0, u64 r1, u64 r2, u64 *part, const u64 *prev_part, int prev_rows,
                                                u64 *prev_sums) {
    constexpr int NS = 4;
    __shared__ u64 red[BLOCK / 64][3 * NS];
    __shared__ u64 red_prev[BLOCK / 64][NSAMP];
    const int row = blockIdx.y, id = blockIdx.y * gridDim.x + blockIdx.x;
    if (row == D.n_rows) {
        for (int j = blockIdx.x; j < 3; j += gridDim.x) block_sum_rows<NS>(prev_part + (i64)j * prev_rows * NSAMP, prev_rows, prev_sums + j * NSAMP, red_prev);
        return;
    }
    SampleAcc<true> acc0[NS], acc1[NS], acc2[NS];
#pragma unroll
    for (int x = 0; x < NS; ++x) { acc0[x].zero(); acc1[x].zero(); acc2[x].zero(); }
    const i64 stride = (i64)gridDim.x * BLOCK;
    const int k = row - D.n_single_rows;
    for (i64 i = (i64)blockIdx.x * BLOCK + threadIdx.x; i < cols; i += stride) {
        u64 common;
        if (k < 0) {
            u64 v[2][8], folded[2];
            request(D.common, i, cols, 8, v[0]);
            load_singles(D, row, i, cols, 8, v[1]);
            take<FIRST>(v[0]);
            three_rounds<2, 3, ONE>(v, r0, r1, r2, acc0, acc1, acc2, folded);
            D.single_dst[row][i] = folded[1];
            common = folded[0];
        } else {
            u64 v[3][8], folded[3];
            request(D.common, i, cols, 8, v[0]);
            request(D.a[k], i, cols, 8, v[1]);
            request(D.b[k], i, cols, 8, v[2]);
            VI_SCHED_FENCE();
#pragma unroll
            for (int t = 0; t < 3; ++t) take<FIRST>(v[t]);
            three_rounds<3, 1, ONE>(v, r0, r1, r2, acc0, acc1, acc2, folded);
            if (D.a_dst[k]) D.a_dst[k][i] = folded[1];
            if (D.b_dst[k]) D.b_dst[k][i] = folded[2];
            common = folded[0];
        }
        if (row == 0) D.common_dst[i] = common;
    }
    const u64 scale = k >= 0 ? D.coeff[k] : 1;
    pass_sums<NS>(acc0, acc1, acc2, red, part + (i64)id * NSAMP, (i64)gridDim.x * D.n_rows * NSAMP, scale);
}

// challenges of the rounds on 2 h entries, h = 2^level
struct TailCoins {
    u64 r[9];
};

// a round on P pairs of every lane: their samples, and the entries folded
template <int P, bool ONE>
__device__ __forceinline__ void lane_round(u64 (&v)[3][8], u64 r, u64 (&total)[4]) {
    SampleAcc<false> acc[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) acc[x].zero();
    u64 lo[3], hi[3], dif[3];
#pragma unroll
    for (int c = 0; c < P; ++c) {
#pragma unroll
        for (int t = 0; t < 3; ++t) { lo[t] = v[t][c]; hi[t] = v[t][c + P]; }
        eval_pair<3, 1, !ONE, false>(lo, hi, dif, acc);
        folds(r, dif, lo, lo);
#pragma unroll
        for (int t = 0; t < 3; ++t) v[t][c] = lo[t];
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) total[x] = acc[x].v;
}

// size: entries per table, a power of two up to SUM_TAIL.  part: a region of n_rows rows of NSAMP words per round, in the order of
// the rounds.  Workgroups behind those of the rows add up the three regions of the pass before.
// FIRST: the tables are the caller's.  ONE: every round sums S(1) (the first of the launch is the one that it is used of).
template <bool FIRST, bool ONE>
__global__ __launch_bounds__(BLOCK) void k_sum_tail(const SumDesc D, int size, const TailCoins C, u64 *part, const u64 *prev_part, int prev_rows, u64 *prev_sums) {
    __shared__ u64 red_prev[BLOCK / 64][NSAMP];
    const int lane = threadIdx.x & 63, n_rows = D.n_rows, groups = (n_rows + BLOCK / 64 - 1) / (BLOCK / 64);
    if ((int)blockIdx.x >= groups) {
        const int j = blockIdx.x - groups;
        block_sum_rows<4>(prev_part + (i64)j * prev_rows * NSAMP, prev_rows, prev_sums + j * NSAMP, red_prev);
        return;
    }
    const int row = blockIdx.x * (BLOCK / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (row >= n_rows) return;
    const int entries = size >> 6;                         // of a lane; below 64 only the first lanes have one
    u64 v[3][8];
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
        for (int c = 0; c < 8; ++c) v[t][c] = 0;
    if (lane < size) {
        const int n = entries > 0 ? entries : 1, k = row - D.n_single_rows;
        request(D.common, lane, 64, n, v[0]);
        if (k < 0) {
            load_singles(D, row, lane, 64, n, v[1]);
#pragma unroll
            for (int c = 0; c < 8; ++c) v[2][c] = 1;       // a third factor: one walk over the rounds for both kinds of rows
        } else {
            request(D.a[k], lane, 64, n, v[1]);
            request(D.b[k], lane, 64, n, v[2]);
            VI_SCHED_FENCE();
            take<FIRST>(v[1]);
            take<FIRST>(v[2]);
        }
        take<FIRST>(v[0]);
    }
    u64 total[9][4];                                       // [8 - log2 of the pairs of a round]
#pragma unroll
    for (int q = 0; q < 9; ++q)
#pragma unroll
        for (int x = 0; x < 4; ++x) total[q][x] = 0;
    if (entries >= 8) lane_round<4, ONE>(v, C.r[8], total[0]);
    if (entries >= 4) lane_round<2, ONE>(v, C.r[7], total[1]);
    if (entries >= 2) lane_round<1, ONE>(v, C.r[6], total[2]);
#pragma unroll
    for (int level = 5; level >= 0; --level) {
        const int h = 1 << level;
        if (size >= 2 * h) {
            SampleAcc<false> acc[4];
            u64 lo[3], hi[3], dif[3];
#pragma unroll
            for (int x = 0; x < 4; ++x) acc[x].zero();
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                lo[t] = v[t][0];
                hi[t] = __shfl_down(v[t][0], (unsigned)h, 64);         // lanes past the pairs compute on what they get and drop it
            }
            eval_pair<3, 1, !ONE, false>(lo, hi, dif, acc);
            folds(C.r[level], dif, lo, lo);
#pragma unroll
            for (int t = 0; t < 3; ++t) v[t][0] = lo[t];
#pragma unroll
            for (int x = 0; x < 4; ++x) total[8 - level][x] = lane < h ? acc[x].v : 0;
        }
    }
    u64 flat[36];
#pragma unroll
    for (int q = 0; q < 9; ++q)
#pragma unroll
        for (int x = 0; x < 4; ++x) flat[4 * q + x] = total[q][x];
    int slot;
    u64 sum = wave_totals<36>(flat, 32, slot);
    if (row >= D.n_single_rows) sum = gl::mul(sum, D.coeff[row - D.n_single_rows]);
    // the round with 2^level pairs is the (log2(size) - 1 - level)-th of this launch
    const int first_level = 31 - __builtin_clz((unsigned)size) - 1, level = 8 - slot / 4;
    if (slot >= 0 && level <= first_level) part[((i64)(first_level - level) * n_rows + row) * NSAMP + (slot & 3)] = sum;
}

// ---- the host side ----------------------------------------------------------------------------------------------
struct SumShape {
    struct Product {
        int a, b;
        u64 coeff;
    };
    int common;
    std::vector<Product> products;
    std::vector<int> singles;
    std::vector<u64> single_coeff;
    u64 c0;
};

// whether the sum is one of this form that the descriptor holds (indices and term lengths have been checked)
bool sum_shape(int n_tables, const int *term_off, const int *factor_idx, const uint64_t *coeffs, int n_terms, SumShape &S) {
    if (n_terms < 2) return false;
    S.common = -1;
    for (int j = term_off[0]; j < term_off[1] && S.common < 0; ++j) {
        bool everywhere = true;
        for (int k = 1; k < n_terms && everywhere; ++k)
            everywhere = std::find(factor_idx + term_off[k], factor_idx + term_off[k + 1], factor_idx[j]) != factor_idx + term_off[k + 1];
        if (everywhere) S.common = factor_idx[j];
    }
    if (S.common < 0) return false;
    std::vector<int> at(n_tables, -1);
    S.c0 = 0;
    for (int k = 0; k < n_terms; ++k) {
        const int n_rest = term_off[k + 1] - term_off[k] - 1;
        if (n_rest > 2) return false;
        const u64 c = coeffs[k] % gl::P;
        int rest[2] = {0, 0}, n = 0;
        bool dropped = false;
        for (int j = term_off[k]; j < term_off[k + 1]; ++j) {
            if (!dropped && factor_idx[j] == S.common) dropped = true;
            else rest[n++] = factor_idx[j];
        }
        if (n_rest == 0) {
            S.c0 = gl::add(S.c0, c);
        } else if (n_rest == 1) {
            int &p = at[rest[0]];
            if (p < 0) {
                p = (int)S.singles.size();
                S.singles.push_back(rest[0]);
                S.single_coeff.push_back(0);
            }
            S.single_coeff[p] = gl::add(S.single_coeff[p], c);
        } else {
            S.products.push_back({rest[0], rest[1], c});
        }
    }
    return S.products.size() <= (size_t)SUM_PRODUCTS && S.singles.size() <= (size_t)SUM_SINGLES && S.products.size() + S.singles.size() > 0;
}

template <bool FIRST, bool ONE>
int sum_resident() {
    static std::mutex mu;
    static int caps[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
    std::lock_guard<std::mutex> lock(mu);
    if (!caps[dev]) caps[dev] = resident_blocks(k_sum3<FIRST, ONE>, 64);
    return caps[dev];
}

// The whole proof.  tables and work are different buffers.  part: workspace of (n_rounds + 1) * MAX_BLOCKS * NSAMP words; C arrives with r, winv, deg, n_rounds set.
// A pass writes behind what the pass before it wrote in the tables' buffers (size / 2 words each: an eighth, a 64th, ... of the
// size), as other rows may still be reading that; the sums of single tables have the upper halves of the buffers.
int prove_sum(const SumShape &S, const uint64_t *const *tables, uint64_t *const *work, i64 size, ChainDesc &C, u64 *part, u64 *out, hipStream_t s) {
    SumDesc D;
    D.c0 = S.c0;
    D.n_products = (int)S.products.size();
    D.n_singles = (int)S.singles.size();
    D.common = tables[S.common];
    for (int k = 0; k < D.n_products; ++k) {
        D.a[k] = tables[S.products[k].a];
        D.b[k] = tables[S.products[k].b];
        D.coeff[k] = S.products[k].coeff;
    }
    for (int k = 0; k < D.n_singles; ++k) {
        D.single[k] = tables[S.singles[k]];
        D.single_coeff[k] = S.single_coeff[k];
    }
    // a pass over few entries is bound by a thread's walk over its row, one over many by the work of all rows (15 gates of 2^18 entries,
    // 29 single tables: 36 us with 4 to a row in the first pass, 31 with 8, 42 with 16)
    auto deal_singles = [&] {
        D.per_row = std::max(size > (i64)1 << 15 ? SUM_ROW_SINGLES_LONG : SUM_ROW_SINGLES, (D.n_singles + SUM_SINGLE_ROWS - 1) / SUM_SINGLE_ROWS);
        D.n_single_rows = (D.n_singles + D.per_row - 1) / D.per_row;
        if (D.n_singles == 0 && D.c0 != 0) D.n_single_rows = 1;
        D.n_rows = D.n_single_rows + D.n_products;
    };
    deal_singles();
    if (C.deg == 3) fill_inf_node(C, 3);
    fill_late(C, size > SUM_TAIL);
    const unsigned sums_off = (unsigned)C.n_rounds * MAX_BLOCKS * NSAMP;
    const i64 upper = size >> 2;
    const u64 *prev_part = nullptr;
    int prev_rows = 0, k = 0;
    unsigned off = 0;
    i64 written = 0;
    bool first = true;
    // the rounds from k on have left n rows each; the three before that are single rows now
    auto note = [&](int rounds, int n) {
        if (prev_rows > 0)
            for (int j = 0; j < 3; ++j) {
                C.off[k - 3 + j] = sums_off + (unsigned)(k - 3 + j) * NSAMP;
                C.nb[k - 3 + j] = 1;
            }
        for (int j = 0; j < rounds; ++j) {
            C.off[k + j] = off + (unsigned)j * (unsigned)n * NSAMP;
            C.nb[k + j] = (unsigned short)n;
        }
    };
    while (size > SUM_TAIL) {
        const i64 cols = size >> 3;
        std::vector<char> owned((size_t)S.common + 1, 0);
        auto own = [&](int t) -> u64 * {                   // the first row that holds a table writes it
            if ((size_t)t >= owned.size()) owned.resize(t + 1, 0);
            if (owned[t]) return nullptr;
            owned[t] = 1;
            return work[t] + written;
        };
        D.common_dst = own(S.common);
        for (int q = 0; q < D.n_products; ++q) {
            D.a_dst[q] = own(S.products[q].a);
            D.b_dst[q] = own(S.products[q].b);
        }
        for (int q = 0; q < D.n_single_rows; ++q) D.single_dst[q] = work[q] + upper + written;
        const bool one = k == C.late;
        const int rows = D.n_rows, cap = first ? (one ? sum_resident<true, true>() : sum_resident<true, false>())
                                               : (one ? sum_resident<false, true>() : sum_resident<false, false>());
        int gx = blocks_for(cols);
        if (gx * rows > cap) gx = std::max(1, cap / rows);
        u64 *prev_sums = part + sums_off + (unsigned)std::max(k - 3, 0) * NSAMP;
        const dim3 grid((unsigned)gx, (unsigned)(rows + (prev_rows > 0 ? 1 : 0)));
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3(BLOCK), 0, s, D, cols, C.r[k], C.r[k + 1], C.r[k + 2], part + off, prev_part, prev_rows, prev_sums);
        };
        if (first && one) launch(k_sum3<true, true>);
        else if (first) launch(k_sum3<true, false>);
        else if (one) launch(k_sum3<false, true>);
        else launch(k_sum3<false, false>);
        VI_LAUNCH_CHECK("sumcheck pass (sum under a common factor)");
        note(3, gx * rows);
        prev_part = part + off;
        prev_rows = gx * rows;
        off += 3u * (unsigned)prev_rows * NSAMP;
        // the tables of the next pass
        D.common = work[S.common] + written;
        for (int q = 0; q < D.n_products; ++q) {
            D.a[q] = work[S.products[q].a] + written;
            D.b[q] = work[S.products[q].b] + written;
        }
        D.n_singles = D.n_single_rows;
        for (int q = 0; q < D.n_singles; ++q) {
            D.single[q] = D.single_dst[q];
            D.single_coeff[q] = 1;
        }
        D.c0 = 0;
        written += cols;
        k += 3;
        size >>= 3;
        first = false;
        deal_singles();
    }
    const int rows = D.n_rows, rounds = C.n_rounds - k;
    TailCoins T;
    for (int level = 0; level < 9; ++level) T.r[level] = level < rounds ? C.r[C.n_rounds - 1 - level] : 0;
    u64 *prev_sums = part + sums_off + (unsigned)std::max(k - 3, 0) * NSAMP;
    const dim3 grid((unsigned)((rows + BLOCK / 64 - 1) / (BLOCK / 64) + (prev_rows > 0 ? 3 : 0)));
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(BLOCK), 0, s, D, (int)size, T, part + off, prev_part, prev_rows, prev_sums);
    };
    if (first) launch(k_sum_tail<true, true>);
    else if (k == C.late) launch(k_sum_tail<false, true>);
    else launch(k_sum_tail<false, false>);
    VI_LAUNCH_CHECK("sumcheck tail (sum under a common factor)");
    note(rounds, rows);
    C.n_prior = C.n_rounds;
    hipLaunchKernelGGL(k_finish, dim3(1), dim3(TAIL_THREADS), 0, s, C, (const u64 *)part, out);
    VI_LAUNCH_CHECK("sumcheck finish");
    return VI_OK;
}

}  // namespace
