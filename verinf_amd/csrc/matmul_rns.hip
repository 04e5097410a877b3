// Dense products over the field on the int8 matrix cores.
//
// A 64 x 64-bit multiply-accumulate is at least 8 VALU instructions, so a product of many rows of A is bound by VALU
// issue at 2 to 2.6 T multiply-adds per second whatever its tiling.  Here the exact integer product is computed modulo 18
// pairwise coprime numbers m_i <= 256 instead and put together by the Chinese remainder theorem (the residue-number
// form of integer matrix products; Ozaki, Uchino, Imamura 2024 use it for floating point).  Modulo one m_i an operand
// is a signed byte, so each residue is ONE int8 matrix product on v_mfma_i32_32x32x32_i8: 18 byte multiply-adds per
// field multiply-add, where splitting both operands into bytes would take 64.
//
// What bounds it at 1000 x 4096 x 4096 (8240 us on the VALU, 423 here): the int8 products 308 us, 2.0 POP/s of the 2.9 to 3.5 that a
// loop of nothing else holds on random bytes -- the matrix cores are busy 53 % of the cycles and the LDS 20 %, neither at its limit: with
// 2.5 wavefronts to a SIMD (registers) the barrier and the operand reads of a step are not all covered by the others' products; the
// residues 113 us, 0.54 GB read and written and 77 % of the VALU issue rate; the reconstruction 23 us.
//
// Operands that are 16-bit signed numbers take fewer byte products (matmul_i16.hpp): k_cut looks at them, k_product does their
// product, and the kernels behind it leave at once when it is done.
//
//   k_cut, k_product, k_residues words -> 18 planes of signed bytes
//   k_residue_gemm    per plane an int8 product; the 32-bit sums are reduced mod m_i to one byte
//   k_from_residues   18 bytes -> the integer mod p
//
// Range.  A word is taken as the integer D = w or w - p with eight balanced digits (bytes in [-128, 127]), |D| <=
// 2^63.006, so a sum of K products is below 2^126.012 K in size; the product M of the moduli is 2^140.45, and for K <=
// MAX_K = 8192 the sum stays within 0.37 M of zero: the multiple of M to take off is the nearest integer to
// sum_i y_i / m_i and a sum of 20-bit fractions finds it (error below 0.003, room 0.13).  A longer inner dimension is
// cut into slices whose results are added mod p.  The 32-bit sums stay below 2^14 K = 2^27.
//
// Layout.  A plane holds units of 16 consecutive inner indices: [unit][row of A or column of B][16 bytes].  A unit is
// what one lane of the MFMA takes (16 of the 32 inner indices of a step), the global loads, the LDS tile and the
// operand reads are all contiguous 16-byte accesses in this order, and B is transposed on the way without a pass.
#include "matmul_rns.hpp"

#include <algorithm>
#include <utility>

#include "common.hpp"
#include "gl_field.hpp"
#include "matmul_i16.hpp"

namespace {

constexpr int BLOCK = 256;
constexpr int NMOD = 18;
constexpr int MODS[NMOD] = {256, 255, 253, 251, 247, 241, 239, 233, 229, 227, 223, 217, 211, 199, 197, 193, 191, 181};
constexpr int MAX_K = 8192;                    // inner indices of one slice
constexpr int UNIT = 16;                       // inner indices of a unit
constexpr unsigned RESIDUE_BLOCKS = 768;       // workgroups of k_product where it makes residues: what is resident at once
constexpr unsigned FEW_SLABS = 340;            // up to so many slabs k_cut takes three workgroups each for the residues

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// ---- constants of the residues, all at compile time -------------------------------------------------------------
constexpr u64 mulmod(u64 a, u64 b) { return (u64)((unsigned __int128)a * b % gl::P); }

// prod of the moduli other than i, mod q (q < 2^16)
constexpr int others_mod(int i, int q) {
    int r = 1 % q;
    for (int j = 0; j < NMOD; ++j)
        if (j != i) r = r * (MODS[j] % q) % q;
    return r;
}
// (M / m_i)^-1 mod m_i
constexpr int crt_factor(int i) {
    const int m = MODS[i], c = others_mod(i, m);
    for (int x = 1; x < m; ++x)
        if (c * x % m == 1) return x;
    return 0;
}
// M / m_i mod p (i = NMOD: M mod p)
constexpr u64 others_mod_p(int i) {
    u64 r = 1;
    for (int j = 0; j < NMOD; ++j)
        if (j != i) r = mulmod(r, (u64)MODS[j]);
    return r;
}
constexpr int balanced(int v, int m) { return v > m / 2 || (v == m / 2 && m == 256) ? v - m : v; }

// the weights 256^j f mod m_i of four digits j = first .. first + 3, as signed bytes
constexpr u32 digit_weights(int i, int first, int f) {
    const int m = MODS[i];
    int pw = 1 % m;
    for (int j = 0; j < first; ++j) pw = pw * 256 % m;
    u32 w = 0;
    for (int j = 0; j < 4; ++j) {
        w |= (u32)(balanced(pw * f % m, m) & 0xFF) << (8 * j);
        pw = pw * 256 % m;
    }
    return w;
}

// ---- words to residues ------------------------------------------------------------------------------------------
// the eight balanced digits of D(w) as signed bytes: w, or w - p = w + 2^32 - 1 - 2^64 for the upper half, plus 128 per
// digit with carries, minus 128 per digit without
__device__ __forceinline__ void balanced_digits(u64 w, int &lo, int &hi) {
    constexpr u64 BIAS = 0x8080808080808080ull;
    u64 t = w > ~BIAS ? w + gl::EPS : w;
    t = (t + BIAS) ^ BIAS;
    lo = (int)(u32)t;
    hi = (int)(u32)(t >> 32);
}

// a word whose low byte is the residue mod MODS[I] (signed, of f D): two byte dot products with the digits' weights give
// |x| <= 2^17, and x - m round(x / m) needs only the low bits of the quotient, which the addition of 1.5 * 2^23 leaves
// in the low mantissa bits
template <int I, bool CRT>
__device__ __forceinline__ u32 residue(int lo, int hi) {
    constexpr int m = MODS[I], f = CRT ? crt_factor(I) : 1;
    constexpr u32 wl = digit_weights(I, 0, f), wh = digit_weights(I, 4, f);
    const int x = __builtin_amdgcn_sdot4(hi, (int)wh, __builtin_amdgcn_sdot4(lo, (int)wl, 0, false), false);
    const u32 q = __float_as_uint(__builtin_fmaf((float)x, 1.0f / (float)m, 12582912.0f));
    return (u32)x + __umul24(q, (1u << 24) - (u32)m);
}

__device__ __forceinline__ u32 pack_bytes(u32 a, u32 b, u32 c, u32 d) {
    return __builtin_amdgcn_perm(b, a, 0x0c0c0400u) | __builtin_amdgcn_perm(d, c, 0x04000c0cu);
}

template <int I, bool CRT>
__device__ __forceinline__ void store_residues(const int (&lo)[UNIT], const int (&hi)[UNIT], v4i *planes, i64 plane, i64 at) {
    v4i v;
#pragma unroll
    for (int g = 0; g < 4; ++g)
        v[g] = (int)pack_bytes(residue<I, CRT>(lo[4 * g], hi[4 * g]), residue<I, CRT>(lo[4 * g + 1], hi[4 * g + 1]),
                               residue<I, CRT>(lo[4 * g + 2], hi[4 * g + 2]), residue<I, CRT>(lo[4 * g + 3], hi[4 * g + 3]));
    planes[I * plane + at] = v;
}
template <bool CRT, int FIRST, int... I>
__device__ __forceinline__ void store_some(const int (&lo)[UNIT], const int (&hi)[UNIT], v4i *planes, i64 plane, i64 at,
                                           std::integer_sequence<int, I...>) {
    (store_residues<FIRST + I, CRT>(lo, hi, planes, plane, at), ...);
}
// share `share` of `shares` = 1 or 3 of the moduli
template <bool CRT>
__device__ __forceinline__ void store_share(const int (&lo)[UNIT], const int (&hi)[UNIT], v4i *planes, i64 plane, i64 at, unsigned share, unsigned shares) {
    constexpr auto third = std::make_integer_sequence<int, NMOD / 3>();
    if (shares == 1 || share == 0) store_some<CRT, 0>(lo, hi, planes, plane, at, third);
    if (shares == 1 || share == 1) store_some<CRT, NMOD / 3>(lo, hi, planes, plane, at, third);
    if (shares == 1 || share == 2) store_some<CRT, 2 * NMOD / 3>(lo, hi, planes, plane, at, third);
}

// ---- cutting up the operands --------------------------------------------------------------------------------------
// An item is four units (64 inner indices) of 64 rows of A or columns of B; a wavefront takes one unit, its lanes along the rows or
// columns, so that the sixteen words that a lane reads of B and all stores are contiguous over the wavefront.  A is read along the
// inner dimension into LDS for that and picked up with the lanes along the rows (an odd pitch in words: no bank conflicts); read by
// each lane from its own row, 1000 x 4096 words took 37 us, 15 this way.  Inner indices from k to the padded length count as zeros.
// Residues are made in slabs: the items of A and, for longer runs of memory, one unit of 256 columns of B (in items of B, 128 x 4096 x
// 4096 94 us, 90 in slabs).
// The residues of A carry the factor of the remainder theorem, so that the sums of the products come out as its y_i.
constexpr int ITEM_UNITS = 4, LINES = 64, TILE_PITCH = ITEM_UNITS * UNIT + 1;

struct Operand {
    const u64 *src;                            // first word of the slice
    i64 ld, count, pitch;                      // row length in memory; rows of A or columns of B; the same padded
    v4i *planes;
    unsigned groups;                           // items along rows or columns
};
struct Cut {
    Operand A, B;
    i64 k;                                     // inner indices of the slice
    int units;
    unsigned b_items, items;                   // items of B (first), of both
    unsigned wide, b_slabs, slabs;             // slabs of B along its columns, of B (first), of both
};

// the sixteen words that a thread holds of an item: of its own column of B, or of A in the order of memory
__device__ __forceinline__ void load_item(const Cut &D, unsigned it, u64 (&w)[UNIT]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const bool is_b = it < D.b_items;
    const unsigned id = is_b ? it : it - D.b_items, groups = is_b ? D.B.groups : D.A.groups;
    const i64 l0 = (i64)(id / groups) * (ITEM_UNITS * UNIT), first = (i64)(id % groups) * LINES;
    if (is_b) {
        const i64 l = l0 + wave * UNIT, at = first + lane;
        const u64 *src = D.B.src + l * D.B.ld + at;
#pragma unroll
        for (int u = 0; u < UNIT; ++u) w[u] = at < D.B.count && l + u < D.k ? __builtin_nontemporal_load(&src[u * D.B.ld]) : 0;
    } else {
        const i64 l = l0 + lane;
        const u64 *src = D.A.src + (first + wave) * D.A.ld + l;
#pragma unroll
        for (int i = 0; i < UNIT; ++i) w[i] = first + wave + 4 * i < D.A.count && l < D.k ? src[4 * i * D.A.ld] : 0;
    }
}
// words of an item of A -> those of the thread's own row
__device__ __forceinline__ void turn_item(u64 (&w)[UNIT], u64 *tile) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();                                       // the tile of the item before has been read
#pragma unroll
    for (int i = 0; i < UNIT; ++i) tile[(wave + 4 * i) * TILE_PITCH + lane] = w[i];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < UNIT; ++u) w[u] = tile[lane * TILE_PITCH + wave * UNIT + u];
}
// residues of a slab, a share of the moduli
__device__ __forceinline__ void residues(const Cut &D, unsigned slab, u64 *tile, unsigned share, unsigned shares) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const bool is_b = slab < D.b_slabs;
    const Operand &S = is_b ? D.B : D.A;
    u64 w[UNIT];
    i64 unit, at;
    if (is_b) {
        unit = slab / D.wide;
        at = (i64)(slab - (unsigned)unit * D.wide) * BLOCK + tid;
        const u64 *src = S.src + unit * UNIT * S.ld + at;
#pragma unroll
        for (int u = 0; u < UNIT; ++u) w[u] = at < S.count && unit * UNIT + u < D.k ? __builtin_nontemporal_load(&src[u * S.ld]) : 0;
    } else {
        const unsigned id = slab - D.b_slabs;
        load_item(D, D.b_items + id, w);
        turn_item(w, tile);
        unit = (i64)(id / S.groups) * ITEM_UNITS + wave;
        at = (i64)(id % S.groups) * LINES + lane;
    }
    if (at >= S.count) return;
    int lo[UNIT], hi[UNIT];
#pragma unroll
    for (int u = 0; u < UNIT; ++u) balanced_digits(w[u], lo[u], hi[u]);
    if (is_b) store_share<false>(lo, hi, S.planes, (i64)D.units * S.pitch, unit * S.pitch + at, share, shares);
    else store_share<true>(lo, hi, S.planes, (i64)D.units * S.pitch, unit * S.pitch + at, share, shares);
}
// done: whether matmul_i16.hpp has finished the product (NULL: it was not tried)
__global__ __launch_bounds__(BLOCK) void k_residues(const Cut D, const u32 *done) {
    __shared__ u64 tile[LINES * TILE_PITCH];
    if (done && *done) return;
    residues(D, blockIdx.x, tile, 0, 1);
}

// The first launch of a product that matmul_i16.hpp may be able to do.  Sixteen runs of sixteen words of either operand, the same for every
// workgroup, decide whether to try (all words of 1000 x 4096 x 4096 read and cut up for nothing would be 37 us; 256 words of either in as
// many lines cost 2 us more for bytes and 4 for residues, as every workgroup reads them).
//
// Bytes: n_flags workgroups, what is resident at once, go over the items, the next item's words on their way while this one's are cut up
// (128 x 4096 x 4096 32 us, a workgroup per item 39).  flags: FITS where all words of a workgroup's items fitted, TOO_LARGE where one
// did not (the workgroup leaves).
//
// Residues, of the first block: a workgroup per slab (1020 workgroups for all of them 104 us for 128 x 4096 x 4096, 93 this way), of few slabs
// three that share the moduli (512 x 512 x 512 16 -> 12).  Only flags[0] is written.
//
// Products of arbitrary words pay for the look and for k_product, which then finds nothing to do, 3 to 5 us; us with neither, and now:
// 128 x 4096 x 4096 170 and 175, 64 x 4096 x 4096 156 and 161, 100 x 760 x 1070 28 and 31, 512 x 512 x 512 26.5 and 27.5, 300 x 9000 x 500 117
// and 124; with the products' loads straight into LDS 500 x 2048 x 2048 89 and 87, 1000 x 4096 x 4096 467 and 423.  Where only
// few words are too large and the sample misses them, the bytes have been cut for nothing as well: 128 x 4096 x 4096 209, 512 x 512 x 512 33.5,
// 1000 x 4096 x 4096 457.
constexpr int SAMPLE_RUN = 16;
enum { FITS = 0, TOO_LARGE = 1, CUT_TO_RESIDUES = 2 };                // CUT_TO_RESIDUES: by the sample, in flags[0]

__global__ __launch_bounds__(BLOCK, 4) void k_cut(const Cut D, const Cut first_block, const i16::Job J, unsigned shares) {
    __shared__ u64 tile[LINES * TILE_PITCH];
    __shared__ int part[BLOCK];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    u32 beyond = 0;
    {
        const i64 na = D.A.count * D.k, nb = D.k * D.B.count;
        const u64 run = (u64)(tid / SAMPLE_RUN + 1) * 0x9E3779B97F4A7C15ull;
        const i64 ea = (i64)__umul64hi(run, (u64)na) + tid % SAMPLE_RUN, eb = (i64)__umul64hi(run, (u64)nb) + tid % SAMPLE_RUN;
        const u64 wa = ea < na ? D.A.src[ea] : 0, wb = eb < nb ? D.B.src[eb] : 0;
        i16::signed_low(wa, beyond);
        i16::signed_low(wb, beyond);
    }
    if (__syncthreads_or((int)beyond)) {
        if (tid == 0 && blockIdx.x == 0) J.flags[0] = CUT_TO_RESIDUES;
        const unsigned share = blockIdx.x / first_block.slabs;
        if (share < shares) residues(first_block, blockIdx.x - share * first_block.slabs, tile, share, shares);
        return;
    }
    const unsigned step = (unsigned)J.n_flags;
    if (blockIdx.x >= step) return;
    u64 w[UNIT];
    load_item(D, blockIdx.x, w);
    for (unsigned it = blockIdx.x; it < D.items; it += step) {
        if (it >= D.b_items) turn_item(w, tile);
        u64 now[UNIT];
#pragma unroll
        for (int u = 0; u < UNIT; ++u) now[u] = w[u];
        if (it + step < D.items) load_item(D, it + step, w);
        const bool is_b = it < D.b_items;
        const i16::Side &S = is_b ? J.B : J.A;
        const unsigned id = is_b ? it : it - D.b_items, groups = is_b ? D.B.groups : D.A.groups;
        const i64 chunk = id / groups, at = (i64)(id % groups) * LINES + lane;          // pitch: a multiple of LINES
        part[tid] = i16::store_digits(now, S.planes + (chunk * ITEM_UNITS + wave) * S.pitch + at, (i64)D.units * S.pitch, beyond);
        if (__syncthreads_or((int)beyond)) {
            if (tid == 0) J.flags[blockIdx.x] = TOO_LARGE;
            return;
        }
        if (tid < LINES) S.sums[chunk * S.pitch + at] = part[tid] + part[tid + 64] + part[tid + 128] + part[tid + 192];
        __syncthreads();
    }
    if (tid == 0) J.flags[blockIdx.x] = FITS;
}

// The launch behind k_cut: the product of 16-bit numbers; or the residues of the first block, where a word has turned out not to fit
// after the sample did; or nothing.
template <int MT, int NT>
__global__ __launch_bounds__(BLOCK, 3) void k_product(const Cut D, const i16::Job J) {
    __shared__ union {
        i16::Lds<MT, NT> product;
        u64 tile[LINES * TILE_PITCH];
    } lds;
    u32 seen = J.flags[0];
    const bool cut = seen == CUT_TO_RESIDUES;
    if (!cut)
        for (int i = threadIdx.x; i < J.n_flags; i += BLOCK) seen |= J.flags[i];
    const bool fits = !cut && !__syncthreads_or((int)seen);
    if (blockIdx.x == 0 && threadIdx.x == 0) *J.done = fits;
    if (cut) return;
    if (!fits) {
        for (unsigned it = blockIdx.x; it < D.slabs; it += gridDim.x) residues(D, it, lds.tile, 0, 1);
    } else if (blockIdx.x < (unsigned)(J.tiles * J.slices)) {
        i16::product<MT, NT>(J, lds.product);
    }
}

// ---- the int8 products ------------------------------------------------------------------------------------------
// per modulus: m, floor(2^32 / m), a multiple of m above 2^28
struct ModConst {
    u32 m[NMOD], inv[NMOD], off[NMOD];
};

// One 64 WM x 64 WN tile of one plane per workgroup: four wavefronts in a 2 x 2 square, each WM x WN MFMA tiles of
// 32 x 32.  BKU units of the inner dimension per step through two LDS buffers.  The next step's loads are in registers while the
// current one is multiplied, or, STRAIGHT, go straight into the other buffer, which leaves room for another workgroup on a CU.  With 128 x
// 256 tiles straight is faster at all sizes (1000 x 4096 x 4096 369 us through registers, 308; three buffers 375), with the smaller ones at
// inner dimensions below some 4000 (us a call: 500 x 2048 x 2048 98 and 91, 777 x 1234 x 2345 136 and 126, 256 x 4096 x 3000 167 and 163; 256 x
// 4096 x 4096 236 and 242, 128 x 8000 x 4096 396 and 412), 64 x 64 only where there are several rounds of workgroups (64 x 1000 x 12000
// 114 and 112, 64 x 4096 x 4096 165 and 169; the launch of 512 x 512 x 512 10.2 and 12.0).
template <int WM, int WN, int BKU, int OCC, bool STRAIGHT>
__global__ __launch_bounds__(BLOCK, OCC) void k_residue_gemm(const v4i *__restrict__ Ap, const v4i *__restrict__ Bp, u32 *__restrict__ Cp,
                                                             int units, i64 mpad, i64 npad, int mt, int nt, ModConst K, const u32 *done) {
    constexpr int TM = 64 * WM, TN = 64 * WN;
    constexpr int LA = BKU * TM / BLOCK, LB = BKU * TN / BLOCK;
    constexpr int LOADS = LA + LB;                                     // loads of 64 16-byte words of a step per wavefront
    __shared__ v4i As[2][BKU * TM];
    __shared__ v4i Bs[2][BKU * TN];
    if (done && *done) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // consecutive ids of one XCD take tiles that share their columns of B
    u32 id = blockIdx.x;
    const u32 total = gridDim.x;
    if ((total & 7) == 0) id = (id & 7) * (total >> 3) + (id >> 3);
    const int mod = id / (mt * nt), rest = id - mod * (mt * nt);
    const int tn = rest / mt, tm = rest - tn * mt;
    const v4i *a_src = Ap + (i64)mod * units * mpad + (i64)tm * TM;
    const v4i *b_src = Bp + (i64)mod * units * npad + (i64)tn * TN;

    // through registers
    v4i ra[LA], rb[LB];
    auto fetch = [&](int u0) {
#pragma unroll
        for (int i = 0; i < LA; ++i) {
            const int c = tid + i * BLOCK;
            ra[i] = a_src[(i64)(u0 + c / TM) * mpad + c % TM];
        }
#pragma unroll
        for (int i = 0; i < LB; ++i) {
            const int c = tid + i * BLOCK;
            rb[i] = b_src[(i64)(u0 + c / TN) * npad + c % TN];
        }
    };
    auto put = [&](int buf) {
#pragma unroll
        for (int i = 0; i < LA; ++i) As[buf][tid + i * BLOCK] = ra[i];
#pragma unroll
        for (int i = 0; i < LB; ++i) Bs[buf][tid + i * BLOCK] = rb[i];
    };
    // straight: load j of the wavefront is chunk wave LOADS + j of a step: [A or B][unit][64 rows]
    auto fetch_straight = [&](int u0, int buf) {
#pragma unroll
        for (int j = 0; j < LOADS; ++j) {
            const int c = wave * LOADS + j, ca = BKU * TM / 64, cb = c - ca;
            if (c < ca) i16::fetch_to_lds(a_src + (i64)(u0 + c / (TM / 64)) * mpad + c % (TM / 64) * 64, &As[buf][c * 64], lane);
            else i16::fetch_to_lds(b_src + (i64)(u0 + cb / (TN / 64)) * npad + cb % (TN / 64) * 64, &Bs[buf][cb * 64], lane);
        }
    };

    v16i acc[WM][WN];
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;
    const int row0 = (wave >> 1) * (32 * WM) + (lane & 31), col0 = (wave & 1) * (32 * WN) + (lane & 31), half = lane >> 5;

    if constexpr (STRAIGHT) {
        fetch_straight(0, 0);
    } else {
        fetch(0);
        put(0);
        __syncthreads();
    }
    int buf = 0;
    for (int u0 = 0; u0 < units; u0 += BKU, buf ^= 1) {
        const bool more = u0 + BKU < units;
        if constexpr (STRAIGHT) {
            i16::wait_and_meet();
            if (more) fetch_straight(u0 + BKU, buf ^ 1);
        } else {
            if (more) fetch(u0 + BKU);
        }
#pragma unroll
        for (int s = 0; s < BKU / 2; ++s) {
            v4i a[WM], b[WN];
#pragma unroll
            for (int i = 0; i < WM; ++i) a[i] = As[buf][(2 * s + half) * TM + row0 + 32 * i];
#pragma unroll
            for (int j = 0; j < WN; ++j) b[j] = Bs[buf][(2 * s + half) * TN + col0 + 32 * j];
#pragma unroll
            for (int i = 0; i < WM; ++i)
#pragma unroll
                for (int j = 0; j < WN; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        if constexpr (!STRAIGHT) {
            if (more) put(buf ^ 1);
            __syncthreads();
        }
    }

    // y = sum mod m in [0, m); register r of a tile is row 8 (r / 4) + 4 half + r % 4: four rows make a word of C's plane
    const u32 m = K.m[mod], inv = K.inv[mod], off = K.off[mod];
    u32 *dst = Cp + (i64)mod * (mpad / 4) * npad + (i64)tn * TN + col0;
    const i64 q0 = ((i64)tm * TM + (wave >> 1) * (32 * WM)) / 4 + half;
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                u32 y[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const u32 u = (u32)acc[i][j][4 * g + r] + off;
                    const u32 v = u - __umulhi(u, inv) * m;
                    y[r] = min(v, v - m);
                }
                dst[(q0 + 8 * i + 2 * g) * npad + 32 * j] = pack_bytes(y[0], y[1], y[2], y[3]);
            }
}

// ---- residues to words ------------------------------------------------------------------------------------------
struct CrtSum {
    u64 lo, hi;                                // sum of y_i (M / m_i mod p), by halves of the constant
    u32 q;                                     // sum of y_i / m_i in 2^-20
};
template <int I>
__device__ __forceinline__ void crt_add(CrtSum &S, u32 y) {
    constexpr u64 c = others_mod_p(I);
    constexpr u32 fr = (u32)(((1 << 21) / MODS[I] + 1) / 2);       // round(2^20 / m)
    S.lo += (u64)y * (u32)c;
    S.hi += (u64)y * (u32)(c >> 32);
    S.q += __umul24(y, fr);
}
template <int... I>
__device__ __forceinline__ void crt_all(CrtSum (&S)[4], const u32 (&w)[NMOD], std::integer_sequence<int, I...>) {
    ((crt_add<I>(S[0], w[I] & 0xFF), crt_add<I>(S[1], (w[I] >> 8) & 0xFF), crt_add<I>(S[2], (w[I] >> 16) & 0xFF), crt_add<I>(S[3], w[I] >> 24)), ...);
}

// Four rows of one column per thread: eighteen words in, four words of C out (added to what is there when `accumulate`).  After a
// product of 16-bit numbers in slices, J.slices > 1, the launch adds up the slices.
__global__ __launch_bounds__(BLOCK) void k_from_residues(const u32 *__restrict__ Cp, i64 plane, i64 npad, u64 *C, i64 ld, i64 m, i64 width, int accumulate, const i16::Job J) {
    if (J.done && *J.done) {
        if (J.slices > 1) i16::add_slices(J, ((i64)blockIdx.y * gridDim.x + blockIdx.x) * BLOCK + threadIdx.x, (i64)gridDim.x * gridDim.y * BLOCK);
        return;
    }
    const i64 j = (i64)blockIdx.x * BLOCK + threadIdx.x, r4 = blockIdx.y;
    if (j >= width) return;
    u32 w[NMOD];
#pragma unroll
    for (int i = 0; i < NMOD; ++i) w[i] = __builtin_nontemporal_load(&Cp[i * plane + r4 * npad + j]);
    CrtSum S[4] = {};
    crt_all(S, w, std::make_integer_sequence<int, NMOD>());
    constexpr u64 neg_m = gl::P - others_mod_p(NMOD);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const i64 row = 4 * r4 + r;
        if (row >= m) break;
        const u32 q = (S[r].q + (1u << 19)) >> 20;                  // the multiple of M to take off
        const u64 lo = S[r].lo + (u64)q * (u32)neg_m, hi = S[r].hi + (u64)q * (u32)(neg_m >> 32);
        const u64 low = lo + (hi << 32);
        u64 v = gl::reduce128(low, (hi >> 32) + (low < lo ? 1 : 0));
        u64 *out = C + row * ld + j;
        if (accumulate) v = gl::add(v, *out);
        *out = v;
    }
}

// ---- the host side ----------------------------------------------------------------------------------------------
inline i64 round_up(i64 v, i64 to) { return (v + to - 1) / to * to; }

struct Plan {
    int wm, wn;                                // MFMA tiles per wavefront
    i64 kc, mb, nb;                            // slice of the inner dimension, block of rows, block of columns
    size_t a_bytes, b_bytes, c_bytes;
};

constexpr int STEP_UNITS = 4;

// The tile is the largest that still gives the 256 CUs a few workgroups each: 128 x 256 (its operands cross the LDS
// least; 1000 x 4096 x 4096: 448 us, 495 with 128 x 128, 665 with 64 x 64; 256 x 256 leaves one wavefront to a SIMD,
// 475 us), then 128 x 128 (128 x 4096 x 4096: 165 us, 200 with 64 x 64), and 64 x 64 for up to 64 rows or few tiles
// (300 x 9000 x 500: 118 us, 130 and 148 with the larger two).
Plan make_plan(i64 m, i64 k, i64 n) {
    Plan L;
    auto tiles = [&](int wm, int wn) { return (m + 64 * wm - 1) / (64 * wm) * ((n + 64 * wn - 1) / (64 * wn)) * NMOD; };
    L.wm = m <= 64 || tiles(2, 2) < 400 ? 1 : 2;
    L.wn = L.wm == 1 ? 1 : (tiles(2, 4) < 2048 ? 2 : 4);
    const i64 tm = 64 * L.wm, tn = 64 * L.wn;
    const i64 slices = (k + MAX_K - 1) / MAX_K;
    L.kc = round_up((k + slices - 1) / slices, STEP_UNITS * UNIT);
    // bytes of the planes of one operand, and of the result: smaller blocks mean more, shorter launches (64 MiB: twice the
    // time at 1000 x 4096 x 4096, 160 MiB: 3 % more)
    constexpr i64 CAP = (i64)384 << 20;
    L.mb = CAP / (NMOD * L.kc) / tm * tm;
    if (L.mb > 8192) L.mb = 8192;
    if (L.mb < tm) L.mb = tm;
    if (L.mb > m) L.mb = m;
    const i64 mpad = round_up(L.mb, tm);
    L.nb = CAP / (NMOD * (L.kc > mpad ? L.kc : mpad)) / tn * tn;
    if (L.nb < tn) L.nb = tn;
    L.nb = round_up((n + (n + L.nb - 1) / L.nb - 1) / ((n + L.nb - 1) / L.nb), tn);      // blocks of about the same width
    if (L.nb > n) L.nb = n;
    const i64 npad = round_up(L.nb, tn);
    L.a_bytes = (size_t)NMOD * L.kc * mpad;
    L.b_bytes = (size_t)NMOD * L.kc * npad;
    L.c_bytes = (size_t)NMOD * mpad * npad;
    return L;
}

template <int WM, int WN, int OCC, bool STRAIGHT>
void launch_gemm(const v4i *A, const v4i *B, u32 *C, int units, i64 mpad, i64 npad, const ModConst &K, const u32 *done, hipStream_t s) {
    const int mt = (int)(mpad / (64 * WM)), nt = (int)(npad / (64 * WN));
    hipLaunchKernelGGL((k_residue_gemm<WM, WN, STEP_UNITS, OCC, STRAIGHT>), dim3((unsigned)(mt * nt * NMOD)), dim3(BLOCK), 0, s, A, B, C, units, mpad, npad, mt, nt, K, done);
}

}  // namespace

namespace vi {

// Estimates in us fitted to measurements of both paths from 1 x 64 x 64 to 2048 x 4096 x 2048 (within a third of the
// times): here three launches, 36 bytes through memory per word of A, B and C, and 52 T multiply-adds per second; on the
// VALU 2.6 T.  They meet at 32 rows for a 4096 x 4096 matrix (155 us each) and at 45 rows for 760 x 1070 (27 us).
bool rns_matmul_pays(int64_t m, int64_t k, int64_t n) {
    const double macs = (double)m * (double)k * (double)n;
    const double words = (double)m * (double)k + (double)k * (double)n + (double)m * (double)n;
    return 18.0 + words / 112e3 + macs / 52e6 < 8.0 + macs / 2.6e6;
}

size_t rns_matmul_workspace_bytes(int64_t m, int64_t k, int64_t n) {
    const Plan L = make_plan(m, k, n);
    const size_t own = L.a_bytes + L.b_bytes + L.c_bytes + i16::GATE_BYTES, small = i16::takes(m, k, n) ? i16::workspace_bytes(m, k, n) : 0;
    return (own > small ? own : small) + WS_SLACK;
}

int rns_matmul(const uint64_t *A, const uint64_t *B, uint64_t *C, int64_t m, int64_t k, int64_t n, void *ws, hipStream_t s) {
    const Plan L = make_plan(m, k, n);
    ws = align16(ws);
    // the planes of the residues lie over the bytes of k_cut: they are written when those are of no use
    v4i *Ap = (v4i *)((char *)ws + i16::GATE_BYTES), *Bp = (v4i *)((char *)Ap + L.a_bytes);
    u32 *Cp = (u32 *)((char *)Bp + L.b_bytes);
    ModConst K;
    for (int i = 0; i < NMOD; ++i) {
        K.m[i] = (u32)MODS[i];
        K.inv[i] = (u32)((1ull << 32) / (u32)MODS[i]);
        K.off[i] = (u32)MODS[i] * ((1u << 28) / (u32)MODS[i] + 1);
    }
    auto cut = [&](i64 i0, i64 mb, i64 l0, i64 kc, i64 j0, i64 nb, bool with_a) {
        Cut D;
        D.A = {A + i0 * k + l0, (i64)k, mb, round_up(mb, 64 * L.wm), Ap, (unsigned)((mb + LINES - 1) / LINES)};
        D.B = {B + l0 * n + j0, (i64)n, nb, round_up(nb, 64 * L.wn), Bp, (unsigned)((nb + LINES - 1) / LINES)};
        D.k = kc;
        D.units = (int)(round_up(kc, STEP_UNITS * UNIT) / UNIT);
        const unsigned chunks = (unsigned)(D.units / ITEM_UNITS);
        D.b_items = D.B.groups * chunks;
        D.items = D.b_items + (with_a ? D.A.groups * chunks : 0);
        D.wide = (unsigned)((nb + BLOCK - 1) / BLOCK);
        D.b_slabs = D.wide * (unsigned)D.units;
        D.slabs = D.b_slabs + D.items - D.b_items;
        return D;
    };
    i16::Job J = {};
    const bool small = i16::takes(m, k, n);
    if (small) {
        J = i16::make_job(C, m, k, n, ws);
        const Cut D = cut(0, m, 0, k, 0, n, true), first = cut(0, L.mb, 0, k < L.kc ? k : L.kc, 0, L.nb, true);
        J.n_flags = (int)std::min(D.items, (unsigned)i16::MAX_CUT_BLOCKS);
        const unsigned shares = first.slabs <= FEW_SLABS ? 3 : 1;
        hipLaunchKernelGGL(k_cut, dim3(std::max((unsigned)J.n_flags, first.slabs * shares)), dim3(BLOCK), 0, s, D, first, J, shares);
        VI_LAUNCH_CHECK("k_cut");
    }
    for (i64 l0 = 0; l0 < k; l0 += L.kc) {
        const i64 kc = k - l0 < L.kc ? k - l0 : L.kc;
        for (i64 i0 = 0; i0 < m; i0 += L.mb) {
            const i64 mb = m - i0 < L.mb ? m - i0 : L.mb, mpad = round_up(mb, 64 * L.wm);
            for (i64 j0 = 0; j0 < n; j0 += L.nb) {
                const i64 nb = n - j0 < L.nb ? n - j0 : L.nb, npad = round_up(nb, 64 * L.wn);
                const Cut D = cut(i0, mb, l0, kc, j0, nb, j0 == 0);
                if (small && l0 == 0 && i0 == 0 && j0 == 0) {
                    const unsigned tiles = (unsigned)(J.tiles * J.slices), most = std::min(D.slabs, RESIDUE_BLOCKS);
                    const dim3 grid(tiles > most ? tiles : most);
                    if (m <= 64) hipLaunchKernelGGL((k_product<1, 2>), grid, dim3(BLOCK), 0, s, D, J);
                    else hipLaunchKernelGGL((k_product<2, 1>), grid, dim3(BLOCK), 0, s, D, J);
                    VI_LAUNCH_CHECK("k_product");
                } else {
                    hipLaunchKernelGGL(k_residues, dim3(D.slabs), dim3(BLOCK), 0, s, D, (const u32 *)J.done);
                    VI_LAUNCH_CHECK("k_residues");
                }
                const bool straight = kc < 4000 && (L.wm == 2 || mpad / 64 * (npad / 64) * NMOD > 2048);
                if (L.wn == 4) launch_gemm<2, 4, 2, true>(Ap, Bp, Cp, D.units, mpad, npad, K, J.done, s);
                else if (L.wn == 2 && straight) launch_gemm<2, 2, 3, true>(Ap, Bp, Cp, D.units, mpad, npad, K, J.done, s);
                else if (L.wn == 2) launch_gemm<2, 2, 3, false>(Ap, Bp, Cp, D.units, mpad, npad, K, J.done, s);
                else if (straight) launch_gemm<1, 1, 4, true>(Ap, Bp, Cp, D.units, mpad, npad, K, J.done, s);
                else launch_gemm<1, 1, 4, false>(Ap, Bp, Cp, D.units, mpad, npad, K, J.done, s);
                VI_LAUNCH_CHECK("k_residue_gemm");
                hipLaunchKernelGGL(k_from_residues, dim3((unsigned)((nb + BLOCK - 1) / BLOCK), (unsigned)((mb + 3) / 4)), dim3(BLOCK), 0, s, (const u32 *)Cp,
                                   mpad / 4 * npad, npad, C + i0 * n + j0, (i64)n, mb, nb, l0 > 0 ? 1 : 0, J);
                VI_LAUNCH_CHECK("k_from_residues");
                J.slices = 1;                              // added up by the first of these launches
            }
        }
    }
    return VI_OK;
}

}  // namespace vi
