// Sumcheck proofs whose challenges are all known before the first launch.
//
// The reference's prover asks its verifier coin for a challenge by round number only
// (layergkr/gpu.py:403, layergkr/sumcheck.py:217: `r = coin(rnd)`) and every caller draws the coins before
// the proof starts (layergkr/full_layer.py:222-224, layergkr/relations.py:122-123), so nothing the host
// contributes to a round depends on that round's samples.  With the challenges in hand the rounds need no
// host round trip, and more than that: several rounds fit in ONE pass over the tables.  The fold pairs index
// i with i + n/2 (most significant variable first), so the 2^R entries i + c n/2^R, c < 2^R, of a table are
// closed under R rounds of folding.  A thread of k_pass3 loads those eight entries of every table (eight
// coalesced streams), evaluates round k on the four pairs (c, c + 4), folds them by r_k, evaluates round
// k + 1 on the two pairs of folded values, folds by r_(k+1), evaluates round k + 2 on the last pair and
// writes ONE folded value per table: a table is read once and an eighth of it written per three rounds,
// instead of read once and half of it written per round.  When the tables have become small enough for one
// workgroup's LDS, k_tail runs every remaining round in a single launch, adds up the per-workgroup partial
// sums the passes left behind, and finishes all samples of the proof: S_k(1) = claim_k - S_k(0), where
// claim_(k+1) = S_k(r_k) follows from the samples by Lagrange interpolation -- a chain over the rounds that a
// launch per round used to carry through the host.
//
// Shapes with their own unrolled evaluation (the ones the layer proof consists of): a single product of up to
// four distinct tables (a matmul contraction, eq * a * b, the three-factor benchmark instance) and the hadamard
// gate batch eq * (a * b + c' * c).  Sums of products of two tables and single tables under a common factor have passes of three rounds
// too (sumcheck_sum.hpp).  Other sums keep one launch per round (k_round / k_eval_mem) but are queued back to back in the same way
// and finished by k_finish.
#pragma once

namespace {

constexpr int MAX_ROUNDS = 40;              // tables of up to 2^40 words
constexpr int TAIL_THREADS = 1024;
constexpr int TAIL_WORDS = 6144;            // table words a tail workgroup keeps in LDS (48 KiB)

// What the kernel that finishes a proof needs to know about its rounds.
struct ChainDesc {
    u64 r[MAX_ROUNDS];                      // challenges, canonical
    u64 winv[NSAMP];                        // Lagrange weights of the points 0..deg
    u64 scale;                              // factor of every summed sample (1 = none)
    u64 skip_mask;                          // bit k: round k did not sum S(1); it is claim_k - S_k(0)
    // inf_node: slot deg of a round holds the leading coefficient L of S_k (the "value at infinity": the sum of
    // the products of the differences hi - lo) instead of S_k(deg), which costs the kernels one step less of every
    // table's ladder; S(deg) = sum_{j<deg} cinf[j] S(j) + deg! L  (the polynomial through the values at 0..deg-1,
    // extrapolated to deg, plus L x (x-1) ... (x-deg+1) there)
    u64 cinf[NSAMP];
    u64 dfact;
    int inf_node;
    // late: the round that sums S(1) where round 0 does not (0 = round 0 does): it has an eighth of the pairs.  The claims before it are
    // affine in the first, claim_late = A claim_0 + B, and late_inv = 1 / A
    int late;
    u64 late_inv;
    unsigned off[MAX_ROUNDS];               // word offset of round k's per-workgroup partial sums in the workspace
    unsigned short nb[MAX_ROUNDS];          // rows of NSAMP words round k left there
    int n_rounds, n_prior, deg;             // rounds of the proof; rounds whose partial sums are in the workspace
};

struct FinishShared {
    u64 raw[MAX_ROUNDS][NSAMP];             // summed samples per round, before scale and chain
    u64 lag[MAX_ROUNDS][NSAMP];             // Lagrange basis of the points 0..deg at r_k
};

// The sums over the wavefront of N values per lane: a step adds the halves of the lanes and halves the values, each half of the
// lanes going on with its own (N / 2 + N / 4 + ... shuffles instead of 6 N; a pass over few entries 14.9 -> 11.2 us).  Returns one total per lane; slot: whose, -1 for none.
template <int N>
__device__ __forceinline__ u64 wave_totals(u64 (&v)[N], int off, int &slot) {
    const int lane = threadIdx.x & 63;
    if constexpr (N == 1) {
        u64 s = v[0];
        for (; off > 0; off >>= 1) s = gl::addc(s, __shfl_xor(s, off, 64));
        slot = 0;
        return s;
    } else {
        constexpr int H = (N + 1) / 2;
        const bool upper = (lane & off) != 0;
        u64 half[H];
#pragma unroll
        for (int i = 0; i < H; ++i) {
            const u64 lo = v[i], hi = i + H < N ? v[i + H] : 0;
            const u64 keep = upper ? hi : lo, give = upper ? lo : hi;
            half[i] = gl::addc(keep, __shfl_xor(give, off, 64));
        }
        const u64 s = wave_totals<H>(half, off >> 1, slot);
        if (slot >= 0 && upper) slot = slot + H < N ? slot + H : -1;
        return s;
    }
}

// Lagrange basis at the challenges (one thread per round and point) and the sums of the partials the earlier launches left
// (one wavefront per round).  The caller synchronises the workgroup before finish_samples().
__device__ __forceinline__ void finish_begin(const ChainDesc &C, const u64 *part, FinishShared &sh) {
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, nw = blockDim.x >> 6;
    for (int e = tid; e < C.n_rounds * NSAMP; e += blockDim.x) {
        const int k = e / NSAMP, x = e % NSAMP;
        if (x <= C.deg) {
            const u64 r = C.r[k];
            u64 num = C.winv[x];
            for (int j = 0; j <= C.deg; ++j)
                if (j != x) num = gl::mul(num, gl::sub(r, (u64)j));
            sh.lag[k][x] = num;
        }
    }
    for (int k = w; k < C.n_prior; k += nw) {
        const u64 *p = part + C.off[k];
        const int nb = C.nb[k];
        u64 v[NSAMP];
#pragma unroll
        for (int x = 0; x < NSAMP; ++x) v[x] = 0;
        // four rows per lane in flight (a lane's loads are otherwise a chain of round trips to memory)
        for (int b0 = lane; b0 < nb; b0 += 256) {
            u64 t[4][NSAMP];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int b = b0 + 64 * u;
#pragma unroll
                for (int x = 0; x < NSAMP; ++x) t[u][x] = (x <= C.deg && b < nb) ? p[(i64)b * NSAMP + x] : 0;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int x = 0; x < NSAMP; ++x)
                    if (x <= C.deg) v[x] = gl::addc(v[x], t[u][x]);
        }
        int slot;
        const u64 sum = wave_totals<NSAMP>(v, 32, slot);
        if (slot >= 0 && slot <= C.deg) sh.raw[k][slot] = sum;
    }
}

// sh.raw holds every round's sums (the workgroup has synchronised): scale, chain the claims, store the samples.
// out: n_rounds rows of NSAMP words, S_k(x) at out[k * NSAMP + x].
__device__ __forceinline__ void finish_samples(const ChainDesc &C, FinishShared &sh, u64 *out) {
    const int k = threadIdx.x;
    const bool mine = k < C.n_rounds;
    const bool skip = mine && ((C.skip_mask >> k) & 1);
    const bool inf = C.inf_node != 0;
    u64 y[NSAMP];
    u64 top_a = 0, top_b = 0;                // S_k(deg) = top_a claim_k + top_b when it is not summed itself
    u64 a = 0, b = 0;                        // claim_(k+1) = a claim_k + b
#pragma unroll
    for (int x = 0; x < NSAMP; ++x) y[x] = 0;
    if (mine) {
        // every sample is a + b claim_k for known a, b: S(1) = claim - S(0) where it was skipped, S(deg) from
        // the leading coefficient; so claim_(k+1) = sum_x L_x(r_k) S_k(x) = a claim_k + b
#pragma unroll
        for (int x = 0; x < NSAMP; ++x) {
            if (x <= C.deg && !(skip && x == 1)) {
                y[x] = sh.raw[k][x];
                if (C.scale != 1) y[x] = gl::mul(y[x], C.scale);
            }
        }
        // S(1) = claim - S(0) when skipped: its part that does not depend on the claim
        const u64 one_b = skip ? gl::neg(y[0]) : y[1];
        if (inf) {
            u64 lead = 0;
#pragma unroll
            for (int x = 0; x < NSAMP; ++x) {
                if (x == C.deg) lead = y[x];
                if (x < C.deg && x != 1) top_b = gl::addc(top_b, gl::mul(C.cinf[x], y[x]));
            }
            top_b = gl::addc(top_b, gl::mul(C.cinf[1], one_b));
            top_b = gl::addc(top_b, gl::mul(C.dfact, lead));
            top_a = skip ? C.cinf[1] : 0;
        }
#pragma unroll
        for (int x = 0; x < NSAMP; ++x) {
            if (x <= C.deg) {
                const u64 l = sh.lag[k][x];
                if (x == 1) {
                    b = gl::addc(b, gl::mul(l, one_b));
                    if (skip) a = gl::addc(a, l);
                } else if (inf && x == C.deg) {
                    b = gl::addc(b, gl::mul(l, top_b));
                    a = gl::addc(a, gl::mul(l, top_a));
                } else {
                    b = gl::addc(b, gl::mul(l, y[x]));
                }
            }
        }
    }
    // claim_(k+1) in terms of claim_0, a prefix product of affine maps in the first wavefront (one after the other, 18 rounds
    // took 3 us)
    if (k >= 64) return;
    for (int d = 1; d < C.n_rounds; d <<= 1) {
        const u64 pa = __shfl_up(a, (unsigned)d, 64), pb = __shfl_up(b, (unsigned)d, 64);
        if (k >= d) {
            b = gl::mul_add(a, pb, b);
            a = gl::mul(a, pa);
        }
    }
    u64 first = 0;                           // a round that summed every sample does not read it
    if (C.late > 0) first = gl::mul(gl::sub(__shfl(gl::addc(y[0], y[1]), C.late, 64), __shfl(b, C.late - 1, 64)), C.late_inv);
    const u64 prev_a = __shfl_up(a, 1, 64), prev_b = __shfl_up(b, 1, 64);
    if (mine) {
        const u64 claim = k == 0 ? first : gl::mul_add(prev_a, first, prev_b);
        if (skip) y[1] = gl::sub(claim, y[0]);
#pragma unroll
        for (int x = 0; x < NSAMP; ++x) {
            if (x <= C.deg) {
                u64 v = y[x];
                if (inf && x == C.deg) v = gl::addc(gl::mul(top_a, claim), top_b);
                put_sample(out + (i64)k * NSAMP + x, v);
            }
        }
    }
}

// finishes a proof whose rounds all left partial sums in the workspace
__global__ __launch_bounds__(TAIL_THREADS) void k_finish(const ChainDesc C, const u64 *part, u64 *out) {
    __shared__ FinishShared sh;
    finish_begin(C, part, sh);
    __syncthreads();
    finish_samples(C, sh, out);
}

// ---- the fixed shapes ------------------------------------------------------------------------------------------
// SHAPE 1: the product of the NT tables (degree NT, NT + 1 samples).
// SHAPE 2: four tables [eq, a, b, c]: eq (a b + c) (degree 3); the coefficient of c is multiplied into the table
//          when the caller's words are first loaded, so that every later round sees a plain sum.
struct FastDesc {
    const u64 *src[4];
    u64 *dst[4];
    u64 lin_coeff;
};

// SHAPE 3: the product of two tables as part of a sum of degree 3: S(2) is taken as well, the leading coefficient is 0.
template <int NT, int SHAPE>
struct FastShape {
    static constexpr int NS = SHAPE >= 2 ? 4 : NT + 1;
    // degree >= 2: the last slot takes the leading coefficient instead of S(deg) (ChainDesc::inf_node)
    static constexpr bool INF = NS >= 3;
};

// accumulators of the samples of one round: plain integers of five words (a product is added without being
// reduced, gl::wide_mul_acc) in the passes, canonical field elements in the tail, where a thread adds few pairs
template <bool WIDE>
struct SampleAcc;
template <>
struct SampleAcc<true> {
    gl::Wide v;
    __device__ __forceinline__ void zero() { gl::wide_zero(v); }
    __device__ __forceinline__ void add_product(u64 a, u64 b) { gl::wide_mul_acc(v, a, b); }
    __device__ __forceinline__ u64 value() const { return gl::wide_reduce(v); }
    // x += a b and y += c d
    static __device__ __forceinline__ void add_two(SampleAcc &x, u64 a, u64 b, SampleAcc &y, u64 c, u64 d) { gl::wide_mul_acc2(x.v, a, b, y.v, c, d); }
};
template <>
struct SampleAcc<false> {
    u64 v;
    __device__ __forceinline__ void zero() { v = 0; }
    __device__ __forceinline__ void add_product(u64 a, u64 b) { v = gl::addc(v, gl::mul(a, b)); }
    __device__ __forceinline__ u64 value() const { return v; }
    static __device__ __forceinline__ void add_two(SampleAcc &x, u64 a, u64 b, SampleAcc &y, u64 c, u64 d) {
        u64 p, q;
        gl::mul2(a, b, p, c, d, q);
        gl::addc2(x.v, p, x.v, y.v, q, y.v);
    }
};

// the same operation on N independent pairs, two at once (gl::mul2 and its neighbours)
template <int N>
__device__ __forceinline__ void differences(const u64 (&hi)[N], const u64 (&lo)[N], u64 (&dif)[N]) {
#pragma unroll
    for (int t = 0; t + 1 < N; t += 2) gl::sub2(hi[t], lo[t], dif[t], hi[t + 1], lo[t + 1], dif[t + 1]);
    if constexpr (N & 1) dif[N - 1] = gl::sub(hi[N - 1], lo[N - 1]);
}
template <int N>
__device__ __forceinline__ void sums(const u64 (&a)[N], const u64 (&b)[N], u64 (&out)[N]) {
#pragma unroll
    for (int t = 0; t + 1 < N; t += 2) gl::addc2(a[t], b[t], out[t], a[t + 1], b[t + 1], out[t + 1]);
    if constexpr (N & 1) out[N - 1] = gl::addc(a[N - 1], b[N - 1]);
}
// lo + r (hi - lo)
template <int N>
__device__ __forceinline__ void folds(u64 r, const u64 (&dif)[N], const u64 (&lo)[N], u64 (&out)[N]) {
#pragma unroll
    for (int t = 0; t + 1 < N; t += 2) gl::mul_add2(r, dif[t], lo[t], out[t], r, dif[t + 1], lo[t + 1], out[t + 1]);
    if constexpr (N & 1) out[N - 1] = gl::mul_add(r, dif[N - 1], lo[N - 1]);
}

// One pair (lo, hi) of every table: adds S(x) of the pair to acc[x] for x = 0..deg-1 (x = 1 left out when SKIP1)
// and the pair's leading coefficient to acc[deg] (or S(deg) when the degree is 1), and returns the differences
// hi - lo, which the fold needs again.  All values canonical.
template <int NT, int SHAPE, bool SKIP1, bool WIDE>
__device__ __forceinline__ void eval_pair(const u64 (&lo)[NT], const u64 (&hi)[NT], u64 (&dif)[NT],
                                          SampleAcc<WIDE> (&acc)[FastShape<NT, SHAPE>::NS]) {
    constexpr int NS = FastShape<NT, SHAPE>::NS;
    constexpr bool INF = FastShape<NT, SHAPE>::INF;
    u64 cur[NT];
    differences(hi, lo, dif);
    if constexpr (NT == 2) {
        // samples two at once as well
        constexpr int second = SHAPE == 3 ? 2 : NS - 1;
        if (SHAPE == 3) sums(hi, dif, cur);
        const u64 (&other)[NT] = SHAPE == 3 ? cur : dif;
        SampleAcc<WIDE>::add_two(acc[0], lo[0], lo[1], acc[second], other[0], other[1]);
        if (!SKIP1) acc[1].add_product(hi[0], hi[1]);
        return;
    }
    if constexpr (NT == 3) {
        u64 v, w;
        sums(hi, dif, cur);                                // S(2)
        if (SKIP1) {
            gl::mul_lazy2(lo[0], lo[1], v, dif[0], dif[1], w);
            SampleAcc<WIDE>::add_two(acc[0], v, lo[2], acc[3], w, dif[2]);
            acc[2].add_product(gl::mul_lazy(cur[0], cur[1]), cur[2]);
        } else {
            gl::mul_lazy2(lo[0], lo[1], v, hi[0], hi[1], w);
            SampleAcc<WIDE>::add_two(acc[0], v, lo[2], acc[1], w, hi[2]);
            gl::mul_lazy2(cur[0], cur[1], v, dif[0], dif[1], w);
            SampleAcc<WIDE>::add_two(acc[2], v, cur[2], acc[3], w, dif[2]);
        }
        return;
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) cur[t] = lo[t];
#pragma unroll
    for (int x = 0; x < NS; ++x) {
        const bool at_inf = INF && x == NS - 1;
        if (!(SKIP1 && x == 1)) {
            if constexpr (SHAPE == 2) {
                // eq (a b + c): the c term has degree 2 and does not reach the leading coefficient
                if (at_inf) acc[x].add_product(gl::mul_lazy(dif[1], dif[2]), dif[0]);
                else acc[x].add_product(gl::mul_add_lazy(cur[1], cur[2], cur[3]), cur[0]);
            } else if constexpr (NT == 1) {
                acc[x].add_product(cur[0], 1);
            } else {
                u64 v = at_inf ? dif[0] : cur[0];
#pragma unroll
                for (int t = 1; t + 1 < NT; ++t) v = gl::mul_lazy(v, at_inf ? dif[t] : cur[t]);
                acc[x].add_product(v, at_inf ? dif[NT - 1] : cur[NT - 1]);
            }
        }
        if (x + 1 < NS - (INF ? 1 : 0)) {
            // f(1) is the upper value itself: the first step of the ladder costs nothing
#pragma unroll
            for (int t = 0; t < NT; ++t) cur[t] = (x == 0) ? hi[t] : gl::addc(cur[t], dif[t]);
        }
    }
}

// Caller data, any 64-bit word is taken as its residue.  Words at or above p have all of the upper half set, as few others have:
// where no lane of the wavefront holds such a word, one maximum per two words is all that this costs.
template <int N>
__device__ __forceinline__ void canon_all(u64 (&v)[N]) {
    u32 top = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) top = max(top, (u32)(v[i] >> 32));
    if (__any(top == 0xFFFFFFFFu)) {
#pragma unroll
        for (int i = 0; i < N; ++i) v[i] = gl::canon(v[i]);
    }
}

template <int N>
__device__ __forceinline__ void canon_pairs(u64 (&lo)[N], u64 (&hi)[N]) {
    u32 top = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) top = max(max(top, (u32)(lo[i] >> 32)), (u32)(hi[i] >> 32));
    if (__any(top == 0xFFFFFFFFu)) {
#pragma unroll
        for (int i = 0; i < N; ++i) { lo[i] = gl::canon(lo[i]); hi[i] = gl::canon(hi[i]); }
    }
}

template <int NT, int SHAPE, bool FIRST>
__device__ __forceinline__ u64 fast_load(const FastDesc &D, int t, i64 idx) {
    u64 v = D.src[t][idx];
    if (FIRST) {
        v = gl::canon(v);                    // caller data: any 64-bit word is taken as its residue
        if (SHAPE == 2 && t == 3) v = gl::mul(v, D.lin_coeff);
    }
    return v;
}

// sum over the rows of NSAMP words at `rows` -> out[0..ns), by one workgroup of THREADS threads
template <int NS, int THREADS = BLOCK>
__device__ __forceinline__ void block_sum_rows(const u64 *rows, int n_rows, u64 *out, u64 (*red)[NSAMP]) {
    u64 v[NS];
#pragma unroll
    for (int x = 0; x < NS; ++x) v[x] = 0;
    for (int b0 = threadIdx.x; b0 < n_rows; b0 += 2 * THREADS) {         // two rows per thread in flight
        u64 t[2][NS];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int x = 0; x < NS; ++x) t[u][x] = (b0 + u * THREADS < n_rows) ? rows[(i64)(b0 + u * THREADS) * NSAMP + x] : 0;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int x = 0; x < NS; ++x) v[x] = gl::addc(v[x], t[u][x]);
    }
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int x = 0; x < NS; ++x) {
        const u64 sum = wave_sum(v[x]);
        if (lane == 0) red[w][x] = sum;
    }
    __syncthreads();
    if (threadIdx.x < NS) {
        u64 sum = red[0][threadIdx.x];
        for (int i = 1; i < THREADS / 64; ++i) sum = gl::addc(sum, red[i][threadIdx.x]);
        out[threadIdx.x] = sum;
    }
    __syncthreads();
}

// a pass's sums of its three rounds over the workgroup, times scale -> row at `row`, region_words apart
template <int NS, int WAVES = BLOCK / 64>
__device__ __forceinline__ void pass_sums(const SampleAcc<true> (&acc0)[NS], const SampleAcc<true> (&acc1)[NS], const SampleAcc<true> (&acc2)[NS],
                                          u64 (*red)[3 * NS], u64 *row, i64 region_words, u64 scale) {
    u64 v[3 * NS];
#pragma unroll
    for (int x = 0; x < NS; ++x) {
        v[x] = acc0[x].value();
        v[NS + x] = acc1[x].value();
        v[2 * NS + x] = acc2[x].value();
    }
    int slot;
    const u64 sum = wave_totals<3 * NS>(v, 32, slot);
    if (slot >= 0) red[threadIdx.x >> 6][slot] = sum;
    __syncthreads();
    if (threadIdx.x < 3 * NS) {
        u64 s = red[0][threadIdx.x];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) s = gl::addc(s, red[w][threadIdx.x]);
        if (scale != 1) s = gl::mul(s, scale);
        row[threadIdx.x / NS * region_words + threadIdx.x % NS] = s;
    }
}

// Three rounds on eight entries of every table: load(c, lo, hi), called for c = 0 .. 3 in turn, gives entries i + c cols and i + (c + 4) cols
// (canonical).  The samples of the seven pairs go into the rounds' accumulators, the entry folded three times into `folded`.  ONE: the
// first round sums S(1) too.
template <int NT, int SHAPE, bool ONE, class Load>
__device__ __forceinline__ void three_rounds_from(Load load, u64 r0, u64 r1, u64 r2, SampleAcc<true> (&acc0)[FastShape<NT, SHAPE>::NS],
                                                  SampleAcc<true> (&acc1)[FastShape<NT, SHAPE>::NS], SampleAcc<true> (&acc2)[FastShape<NT, SHAPE>::NS],
                                                  u64 (&folded)[NT]) {
    // the scheduler is kept from interleaving the pairs: each one's temporaries die before the next starts
    u64 lo[NT], hi[NT], dif[NT], v[4][NT];
    static_for<0, 4>([&](auto c_) {
        constexpr int c = decltype(c_)::value;
        VI_SCHED_FENCE();
        load(c_, lo, hi);
        eval_pair<NT, SHAPE, !ONE, true>(lo, hi, dif, acc0);
        folds(r0, dif, lo, v[c]);
    });
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        VI_SCHED_FENCE();
#pragma unroll
        for (int t = 0; t < NT; ++t) { lo[t] = v[c][t]; hi[t] = v[c + 2][t]; }
        eval_pair<NT, SHAPE, true, true>(lo, hi, dif, acc1);
        folds(r1, dif, lo, v[c]);
    }
    VI_SCHED_FENCE();
    eval_pair<NT, SHAPE, true, true>(v[0], v[1], dif, acc2);
    folds(r2, dif, v[0], folded);
}

// the same of entries in registers, v[t][c] = entry i + c cols
template <int NT, int SHAPE, bool ONE>
__device__ __forceinline__ void three_rounds(const u64 (&v)[NT][8], u64 r0, u64 r1, u64 r2, SampleAcc<true> (&acc0)[FastShape<NT, SHAPE>::NS],
                                             SampleAcc<true> (&acc1)[FastShape<NT, SHAPE>::NS], SampleAcc<true> (&acc2)[FastShape<NT, SHAPE>::NS],
                                             u64 (&folded)[NT]) {
    auto load = [&](auto c_, u64 (&lo)[NT], u64 (&hi)[NT]) {
        constexpr int c = decltype(c_)::value;
#pragma unroll
        for (int t = 0; t < NT; ++t) { lo[t] = v[t][c]; hi[t] = v[t][c + 4]; }
    };
    three_rounds_from<NT, SHAPE, ONE>(load, r0, r1, r2, acc0, acc1, acc2, folded);
}

// 64 words at src into LDS, by one wavefront and without a register in between; src and dst are the same for all its lanes.  Two
// loads of four bytes a lane, which ask for no more than the alignment of a word.  The compiler does not wait for them: loads_arrived()
// does.  M0 has its value back afterwards (the compiler does not accept it in a list of clobbered registers).
// ONCE: words that nothing reads again, with the streaming hint.
template <bool ONCE>
__device__ __forceinline__ void words_to_lds(const u64 *src, u64 *dst, int lane) {
#ifdef __HIP_DEVICE_COMPILE__
    const u32 at = __builtin_amdgcn_readfirstlane((u32)(uintptr_t)(__attribute__((address_space(3))) u64 *)dst);
    u32 m0;
    if (ONCE)
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %3, %5 nt\n\t"
                     "s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %4, %5 nt\n\ts_mov_b32 m0, %0"
                     : "=&s"(m0) : "s"(at), "s"(at + 256), "v"((u32)lane * 4), "v"((u32)lane * 4 + 256), "s"(src) : "memory");
    else
        asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %3, %5\n\t"
                     "s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %4, %5\n\ts_mov_b32 m0, %0"
                     : "=&s"(m0) : "s"(at), "s"(at + 256), "v"((u32)lane * 4), "v"((u32)lane * 4 + 256), "s"(src) : "memory");
#else
    dst[lane] = src[lane];
#endif
}
// all but the LATER youngest of the wavefront's loads and stores are complete
template <int LATER>
__device__ __forceinline__ void loads_arrived() {
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(LATER) : "memory");
#endif
}
// the wavefront's LDS reads are complete
__device__ __forceinline__ void lds_reads_done() {
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
#endif
}

// Waits for the loads of v, here and not at its first use.  The compiler counts its own loads only, and loads end in order: its wait for
// v behind words_to_lds() is one for all the younger words on their way to LDS as well.
template <int N>
__device__ __forceinline__ void used_from_here(u64 (&v)[N][2]) {
#ifdef __HIP_DEVICE_COMPILE__
#pragma unroll
    for (int t = 0; t < N; ++t) asm volatile("" : "+v"(v[t][0]), "+v"(v[t][1]) : : "memory");
#endif
}

// Three rounds in one pass.  cols = n / 8 for tables of n words; thread i < cols owns entries i + c cols.
// FIRST: the tables are the caller's (words reduced on load).  ONE: the first of the rounds sums every sample.
// part: three regions of gridDim.x rows of NSAMP words, one per round.
// prev_part / prev_rows / prev_sums: the previous pass's three regions of prev_rows rows each; workgroup j < 3 adds
// region j up into row j of prev_sums before it starts on its own columns, so that the kernel that finishes the
// proof finds one row per round instead of a thousand (prev_rows = 0: nothing to add up).
template <int NT, int SHAPE, bool FIRST, bool ONE>
__global__ __launch_bounds__(BLOCK) void k_pass3(const FastDesc D, i64 cols, u64 r0, u64 r1, u64 r2, u64 *part,
                                                 const u64 *prev_part, int prev_rows, u64 *prev_sums) {
    constexpr int NS = FastShape<NT, SHAPE>::NS;
    __shared__ u64 red[BLOCK / 64][3 * NS];
    __shared__ u64 red_prev[BLOCK / 64][NSAMP];
    if (prev_rows > 0 && blockIdx.x < 3)
        block_sum_rows<NS>(prev_part + (i64)blockIdx.x * prev_rows * NSAMP, prev_rows, prev_sums + blockIdx.x * NSAMP, red_prev);
    SampleAcc<true> acc0[NS], acc1[NS], acc2[NS];
#pragma unroll
    for (int x = 0; x < NS; ++x) { acc0[x].zero(); acc1[x].zero(); acc2[x].zero(); }
    if (const i64 i = (i64)blockIdx.x * BLOCK + threadIdx.x; i < cols) {
        u64 v[NT][8];
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int c = 0; c < 8; ++c) v[t][c] = D.src[t][i + c * cols];
        if (FIRST) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if (SHAPE == 2 && t == 3) {
#pragma unroll
                    for (int c = 0; c < 8; ++c) {
                        v[t][c] = gl::mul(v[t][c], D.lin_coeff);
                        VI_SCHED_FENCE();
                    }
                } else {
                    canon_all(v[t]);
                }
            }
        }
        u64 folded[NT];
        three_rounds<NT, SHAPE, ONE>(v, r0, r1, r2, acc0, acc1, acc2, folded);
#pragma unroll
        for (int t = 0; t < NT; ++t) D.dst[t][i] = folded[t];
    }
    pass_sums<NS>(acc0, acc1, acc2, red, part + (i64)blockIdx.x * NSAMP, (i64)gridDim.x * NSAMP, 1);
}

// The same for more columns than fit the chip at once.  Two things keep the plain loop from either of its bounds there: a SIMD
// serves its oldest wavefront first, so of four workgroups of a CU with the same share the first was done after 250 us and the last
// after 450 (three tables of 2^26), alone by then; and a wavefront's loads wait for its arithmetic.  So a workgroup has all the wavefronts
// of a CU, which take pieces of 64 columns from a counter in LDS, and a piece's entries are on their way into LDS while
// the piece before it is worked on (18 of 24 words a lane for three tables; the last pair's go to registers, and are waited for in front of
// the next piece's request, two pairs after their own: used_from_here).
// Where the pieces lie decides the rate of memory: 24 streams of three tables of 2^26 and an eighth as much written take 384 us with
// sixteen pieces of a workgroup in a row, 346 with the workgroups' pieces beside each other, 315 with the streaming hint on the loads
// besides (without the writes 290, 256 and 224: 7.2 TB/s; one stream 5.9).  The proof over them 559 -> 475 us; with equal shares of the
// columns and this staging 543, with pieces in rows of sixteen 510.  The first pass takes 342 us, near what its loads and stores take alone.  Where
// the last pair's words were waited for at their use, behind the request, its wavefronts waited 31.7 % of their time and now 28.5, over
// 1.5 % fewer cycles; the time is the same within its noise.
template <int NT>
struct LongPass {
    static constexpr int THREADS = NT <= 3 ? 1024 : 768;               // 128 and 168 registers
};

template <int NT, int SHAPE, bool FIRST, bool ONE>
__global__ __launch_bounds__(LongPass<NT>::THREADS) void k_pass3_long(const FastDesc D, i64 cols, u64 r0, u64 r1, u64 r2, u64 *part,
                                                 const u64 *prev_part, int prev_rows, u64 *prev_sums) {
    constexpr int NS = FastShape<NT, SHAPE>::NS;
    constexpr int WAVES = LongPass<NT>::THREADS / 64;
    __shared__ u64 red[WAVES][3 * NS];
    __shared__ u64 red_prev[WAVES][NSAMP];
    __shared__ u64 stage[WAVES][6 * NT][64];
    __shared__ int next;
    if (threadIdx.x == 0) next = WAVES;
    __syncthreads();
    if (prev_rows > 0 && blockIdx.x < 3)
        block_sum_rows<NS, 64 * WAVES>(prev_part + (i64)blockIdx.x * prev_rows * NSAMP, prev_rows, prev_sums + blockIdx.x * NSAMP, red_prev);
    SampleAcc<true> acc0[NS], acc1[NS], acc2[NS];
#pragma unroll
    for (int x = 0; x < NS; ++x) { acc0[x].zero(); acc1[x].zero(); acc2[x].zero(); }
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    u64 (&mine)[6 * NT][64] = stage[wave];
    // entries c and c + 4 of table t are rows 2 (3 t + c) and 2 (3 t + c) + 1 of the wavefront's stage; c = 3 goes to registers
    auto fetch = [&](i64 first) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                words_to_lds<FIRST>(D.src[t] + first + c * cols, mine[2 * (3 * t + c)], lane);
                words_to_lds<FIRST>(D.src[t] + first + (c + 4) * cols, mine[2 * (3 * t + c) + 1], lane);
            }
    };
    // piece j of the workgroup, the workgroups' pieces beside each other
    auto piece = [&](int j) { return ((i64)j * gridDim.x + blockIdx.x) * 64; };
    i64 first = piece(wave), following = 0;
    if (first < cols) fetch(first);
    for (; first < cols; first = following) {
        const i64 i = first + lane;
        u64 last[NT][2];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const u64 *p = D.src[t] + i + 3 * cols, *q = D.src[t] + i + 7 * cols;
            last[t][0] = FIRST ? __builtin_nontemporal_load(p) : *p;
            last[t][1] = FIRST ? __builtin_nontemporal_load(q) : *q;
        }
        loads_arrived<2 * NT>();
        auto load = [&](auto c_, u64 (&lo)[NT], u64 (&hi)[NT]) {
            constexpr int c = decltype(c_)::value;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                lo[t] = c < 3 ? mine[2 * (3 * t + c % 3)][lane] : last[t][0];
                hi[t] = c < 3 ? mine[2 * (3 * t + c % 3) + 1][lane] : last[t][1];
            }
            if constexpr (c == 2) {
                int j = 0;
                if (lane == 0) j = atomicAdd(&next, 1);
                following = piece((int)__builtin_amdgcn_readfirstlane((u32)__shfl((u64)j, 0, 64)));
                lds_reads_done();
                used_from_here(last);
                if (following < cols) fetch(following);
            }
            if (FIRST) {
                canon_pairs(lo, hi);
                if (SHAPE == 2) {
                    lo[NT - 1] = gl::mul(lo[NT - 1], D.lin_coeff);
                    hi[NT - 1] = gl::mul(hi[NT - 1], D.lin_coeff);
                }
            }
        };
        u64 folded[NT];
        three_rounds_from<NT, SHAPE, ONE>(load, r0, r1, r2, acc0, acc1, acc2, folded);
#pragma unroll
        for (int t = 0; t < NT; ++t) D.dst[t][i] = folded[t];
    }
    pass_sums<NS, WAVES>(acc0, acc1, acc2, red, part + (i64)blockIdx.x * NSAMP, (i64)gridDim.x * NSAMP, 1);
}

// pairs per table a tail workgroup holds after its first fold
template <int NT>
struct TailCap {
    static constexpr int HALF = NT == 1 ? 4096 : (NT <= 3 ? 2048 : 1024);
    static_assert(NT * HALF <= TAIL_WORDS, "tail tables exceed their LDS share");
};

// Every remaining round in one workgroup: tables of `size` <= 2 TailCap<NT>::HALF words; rounds C.n_prior .. C.n_rounds - 1.
// FIRST: the proof starts here (the tables are the caller's).  ONE: the launch's first round sums S(1).  The folded tables live in LDS and are not written back.
// A round costs its longest thread and a barrier, so what can wait is kept off that path:
//  - every round leaves its threads' sums in LDS, and a wavefront per round adds them up at the end, all at once (summed across
//    the workgroup as they went, the rounds of more than 256 pairs took 1 us longer each);
//  - once a table fits the lanes of one wavefront (64 entries) the first wavefront goes on alone, a table entry per lane and
//    partners fetched by lane shuffles, and only folds: it leaves the tables of those rounds behind, and a wavefront per round
//    takes the samples from them at the end.
// 12 rounds over two tables 21.0 -> 15.2 us, the last 11 of 26 over three 35.4 -> 24.4.
constexpr int TAIL_SMALL = 6;                // rounds of 32, 16, .. 1 pairs

template <int NT, int SHAPE, bool FIRST, bool ONE>
__global__ __launch_bounds__(TAIL_THREADS) void k_tail(const FastDesc D, i64 size, const ChainDesc C, const u64 *part, u64 *out) {
    constexpr int NS = FastShape<NT, SHAPE>::NS;
    constexpr int HALF = TailCap<NT>::HALF;
    // sums of the round of h pairs: min(h, TAIL_THREADS) words at [h, 2 h), or one after the other beyond 2 TAIL_THREADS
    constexpr int SUMS = HALF <= TAIL_THREADS ? 2 * TAIL_THREADS : (HALF == 2 * TAIL_THREADS ? 3 : 4) * TAIL_THREADS;
    auto sums_at = [](int h) { return h <= 2 * TAIL_THREADS ? h : 3 * TAIL_THREADS; };
    static_assert(HALF <= 4 * TAIL_THREADS, "rounds of more pairs need more room for their sums");
    __shared__ u64 tab[NT][HALF];
    __shared__ u64 lane_sums[NS][SUMS];
    __shared__ u64 small[NT][128];           // the table of s <= 64 entries at [s, 2 s)
    __shared__ FinishShared sh;
    finish_begin(C, part, sh);

    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    int k = C.n_prior;
    int h = (int)(size >> 1);
    const int h_first = h;
    SampleAcc<false> acc[NS];
    u64 lo[NT], hi[NT], dif[NT];
    auto leave_sums = [&]() {
        if (tid < h) {
#pragma unroll
            for (int x = 0; x < NS; ++x) lane_sums[x][sums_at(h) + tid] = acc[x].v;
        }
        __syncthreads();
    };
    {
        // first round of this launch: pairs from memory, folded values into LDS
#pragma unroll
        for (int x = 0; x < NS; ++x) acc[x].zero();
        const u64 r = C.r[k];
        for (int i = tid; i < h; i += TAIL_THREADS) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                lo[t] = fast_load<NT, SHAPE, FIRST>(D, t, i);
                hi[t] = fast_load<NT, SHAPE, FIRST>(D, t, (i64)h + i);
            }
            eval_pair<NT, SHAPE, !ONE, false>(lo, hi, dif, acc);
            if (h > 1) {
                folds(r, dif, lo, lo);
#pragma unroll
                for (int t = 0; t < NT; ++t) tab[t][i] = lo[t];
            }
        }
        leave_sums();
    }
    // rounds on tables of more than 64 entries: pairs from LDS, a workgroup barrier per round
    for (h >>= 1; h >= 64; h >>= 1) {
        ++k;
#pragma unroll
        for (int x = 0; x < NS; ++x) acc[x].zero();
        const u64 r = C.r[k];
        for (int i = tid; i < h; i += TAIL_THREADS) {
#pragma unroll
            for (int t = 0; t < NT; ++t) { lo[t] = tab[t][i]; hi[t] = tab[t][h + i]; }
            eval_pair<NT, SHAPE, true, false>(lo, hi, dif, acc);
            folds(r, dif, lo, lo);
#pragma unroll
            for (int t = 0; t < NT; ++t) tab[t][i] = lo[t];
        }
        leave_sums();
    }
    // tables of at most 64 entries: the first wavefront alone, lane i holding entry i of every table
    const int h_small = h;
    if (w == 0) {
        u64 val[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) val[t] = (lane < 2 * h) ? tab[t][lane] : 0;
        for (; h >= 1; h >>= 1) {
            const u64 r = C.r[++k];
            u64 up[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if (lane < 2 * h) small[t][2 * h + lane] = val[t];
                up[t] = __shfl_down(val[t], (unsigned)h, 64);              // lanes past the pairs compute on what they get and drop it
            }
            differences(up, val, up);
            folds(r, up, val, val);
        }
    }
    __syncthreads();
    // wavefront w < TAIL_SMALL: the round of 32 >> w pairs; the others a round of h_small < 2^j <= h_first pairs
    auto keep = [&](u64 (&v)[NS], int pairs) {
        int slot;
        const u64 sum = wave_totals<NS>(v, 32, slot);
        const int kd = C.n_rounds - 1 - (31 - __builtin_clz((unsigned)pairs));
        if (slot >= 0) sh.raw[kd][slot] = sum;
    };
    u64 v[NS];
    if (w < TAIL_SMALL) {
        const int pairs = 32 >> w;
        if (pairs <= h_small) {
#pragma unroll
            for (int x = 0; x < NS; ++x) acc[x].zero();
            if (lane < pairs) {
#pragma unroll
                for (int t = 0; t < NT; ++t) { lo[t] = small[t][2 * pairs + lane]; hi[t] = small[t][3 * pairs + lane]; }
                eval_pair<NT, SHAPE, true, false>(lo, hi, dif, acc);
            }
#pragma unroll
            for (int x = 0; x < NS; ++x) v[x] = acc[x].v;
            keep(v, pairs);
        }
    } else {
        const int pairs = h_first >> (w - TAIL_SMALL);
        if (pairs > h_small) {
            const int words = pairs < TAIL_THREADS ? pairs : TAIL_THREADS, at = sums_at(pairs);
#pragma unroll
            for (int x = 0; x < NS; ++x) v[x] = 0;
            for (int i = lane; i < words; i += 64)
#pragma unroll
                for (int x = 0; x < NS; ++x) v[x] = gl::addc(v[x], lane_sums[x][at + i]);
            keep(v, pairs);
        }
    }
    __syncthreads();
    finish_samples(C, sh, out);
}

// k_pass3 has a column a thread where all of them are resident at once, k_pass3_long what is more, and first passes over three and four
// tables from four workgroups a CU on.  us of a pass and of the one behind it, which has fewer rows to add up, long and with a workgroup for 256
// columns: one table of 2^23 19.0 + 5.5 and 21.0 + 7.9, 2^26 103 + 18 and 122 + 21; two of 2^22 21.4 + 7.2 and 22.0 + 9.6, 2^26 219 + 31 and 246 + 36 (2^24 61 +
// 12 and 53 + 13 where they stay in the last-level cache from proof to proof); three of 2^21 23.5 + 10.4 and 21.1 + 12.1, the proofs 63.7 and 64.6; 2^22
// 33.9 + 10.4 and 35.1 + 13.4; four of 2^21 proofs 90.1 and 94.2, gates of 2^21 72.3 and 75.0 on one box, 79.0 and 77.0 on another; 2^22 42.7 + 11.8 and
// 41.2 + 15.1, 2^26 459 + 65 and 527 + 83.  Second passes of four workgroups a CU: 2^24, three tables 21.2 + 9.8 and 18.4 + 10.7, gates 23.6 + 11.4 and
// 21.5 + 12.3.
template <int NT, int SHAPE, bool FIRST, bool ONE>
int launch_pass3(const FastDesc &F, i64 cols, const u64 *r, u64 *part, const u64 *prev_part, int prev_rows,
                 u64 *prev_sums, hipStream_t s) {
    static std::mutex mu;
    static int caps[64] = {0}, cus[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
    int cap, n_cus;
    {
        std::lock_guard<std::mutex> lock(mu);
        if (!caps[dev]) {
            caps[dev] = resident_blocks(k_pass3<NT, SHAPE, FIRST, ONE>, FIRST && NT >= 3 ? 3 : 64);
            cus[dev] = resident_blocks(k_pass3<NT, SHAPE, FIRST, ONE>, 1);
        }
        cap = caps[dev];
        n_cus = cus[dev];
    }
    const int least = prev_rows > 0 ? 3 : 1; // the first three workgroups add up the previous pass's sums
    if (cols > (i64)cap * BLOCK) {
        const int nb = std::max(n_cus, least);
        hipLaunchKernelGGL((k_pass3_long<NT, SHAPE, FIRST, ONE>), dim3(nb), dim3(LongPass<NT>::THREADS), 0, s, F, cols, r[0], r[1], r[2], part,
                           prev_part, prev_rows, prev_sums);
        return nb;
    }
    const int nb = std::max(blocks_for(cols), least);
    hipLaunchKernelGGL((k_pass3<NT, SHAPE, FIRST, ONE>), dim3(nb), dim3(BLOCK), 0, s, F, cols, r[0], r[1], r[2], part,
                       prev_part, prev_rows, prev_sums);
    return nb;
}

// constants of ChainDesc::inf_node for degree d: S(d) = sum_{j<d} cinf[j] S(j) + d! L
void fill_inf_node(ChainDesc &C, int d) {
    C.inf_node = 1;
    C.dfact = 1;
    for (int m = 1; m <= d; ++m) C.dfact = gl::mul(C.dfact, (u64)m);
    for (int j = 0; j < NSAMP; ++j) C.cinf[j] = 0;
    for (int j = 0; j < d; ++j) {
        // Lagrange basis of the nodes 0..d-1 at x = d
        u64 num = 1, den = 1;
        for (int m = 0; m < d; ++m) {
            if (m == j) continue;
            num = gl::mul(num, (u64)(d - m));
            den = gl::mul(den, gl::sub((u64)j, (u64)m));
        }
        C.cinf[j] = gl::mul(num, gl::inv(den));
    }
}

// Round 3 sums S(1) in the place of round 0, for a proof whose first launch does three rounds: C.late, C.late_inv, C.skip_mask.  A
// challenge at which S(1) does not enter the next claim (0, and 2 in degree 2 and 3) leaves round 0 as it is.  Called with r, winv
// and the constants of inf_node set.
void fill_late(ChainDesc &C, bool passes) {
    C.late = 0;
    C.late_inv = 0;
    if (passes) {
        u64 product = 1;
        for (int k = 0; k < 3; ++k) {
            auto basis = [&](int x) {
                u64 l = C.winv[x];
                for (int j = 0; j <= C.deg; ++j)
                    if (j != x) l = gl::mul(l, gl::sub(C.r[k], (u64)j));
                return l;
            };
            u64 a = basis(1);
            if (C.inf_node) a = C.deg == 1 ? 0 : gl::add(a, gl::mul(basis(C.deg), C.cinf[1]));
            product = gl::mul(product, a);
        }
        if (product != 0) {
            C.late = 3;
            C.late_inv = gl::inv(product);
        }
    }
    C.skip_mask = 0;
    for (int j = 0; j < C.n_rounds; ++j)
        if (j != C.late) C.skip_mask |= 1ull << j;
}

// The whole proof of a fixed shape: passes of three rounds while the tables exceed a tail workgroup, then the tail.
// part: workspace of at least (n_rounds + 1) * MAX_BLOCKS * NSAMP words; C arrives with r, winv, scale, deg, n_rounds set.
template <int NT, int SHAPE>
int prove_fast_shape(FastDesc F, i64 size, ChainDesc &C, u64 *part, u64 *out, hipStream_t s) {
    constexpr i64 TAIL_MAX = 2 * (i64)TailCap<NT>::HALF;
    int k = 0;
    unsigned off = 0;
    bool first = true;
    if (FastShape<NT, SHAPE>::INF) fill_inf_node(C, C.deg);
    fill_late(C, size > TAIL_MAX);
    // one row per round for the sums that a pass adds up for the pass before it: the last MAX_ROUNDS rows of the workspace
    const unsigned sums_off = (unsigned)C.n_rounds * MAX_BLOCKS * NSAMP;
    const u64 *prev_part = nullptr;
    int prev_rows = 0, prev_k = 0;
    while (size > TAIL_MAX) {
        const i64 cols = size >> 3;
        u64 *prev_sums = part + sums_off + (unsigned)prev_k * NSAMP;
        const bool one = k == C.late;
        auto launch = [&](auto kernel_of) { return kernel_of(F, cols, C.r + k, part + off, prev_part, prev_rows, prev_sums, s); };
        const int nb = first ? (one ? launch(launch_pass3<NT, SHAPE, true, true>) : launch(launch_pass3<NT, SHAPE, true, false>))
                             : (one ? launch(launch_pass3<NT, SHAPE, false, true>) : launch(launch_pass3<NT, SHAPE, false, false>));
        VI_LAUNCH_CHECK("sumcheck pass (three rounds)");
        if (prev_rows > 0) {
            for (int j = 0; j < 3; ++j) {    // this launch has left the previous pass's rounds as one row each
                C.off[prev_k + j] = sums_off + (unsigned)(prev_k + j) * NSAMP;
                C.nb[prev_k + j] = 1;
            }
        }
        for (int j = 0; j < 3; ++j) {
            C.off[k + j] = off + (unsigned)j * (unsigned)nb * NSAMP;
            C.nb[k + j] = (unsigned short)nb;
        }
        prev_part = part + off;
        prev_rows = nb;
        prev_k = k;
        off += 3u * (unsigned)nb * NSAMP;
        k += 3;
        size >>= 3;
        if (first) {
            for (int t = 0; t < NT; ++t) F.src[t] = F.dst[t];    // later passes fold the work buffers in place
            first = false;
        }
    }
    C.n_prior = k;
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(1), dim3(TAIL_THREADS), 0, s, F, size, C, (const u64 *)part, out); };
    if (first) launch(k_tail<NT, SHAPE, true, true>);
    else if (k == C.late) launch(k_tail<NT, SHAPE, false, true>);
    else launch(k_tail<NT, SHAPE, false, false>);
    VI_LAUNCH_CHECK("sumcheck tail");
    return VI_OK;
}

}  // namespace
