// Dense products over the field whose operands are 16-bit signed numbers, on the int8 matrix cores.
//
// What a prover multiplies in a layer are quantised weights and activations: field elements x or p - |x| with |x| < 2^15.  Their
// products need 4 byte products per multiply-add where arbitrary words take 18 (matmul_rns.hip) and 64 as plain digits.  Whether the
// operands are such numbers is looked at on the device in every call, by the launch that cuts them into bytes:
//
//   k_cut      (matmul_rns.hip) words -> two planes of signed bytes, sums along the inner dimension, and per workgroup whether a word
//              did not fit
//   product()  all four byte products of a tile at once, put together as 64-bit integers and taken mod p
//
// 1000 x 4096 x 4096: 423 us through residues, 111 to 114 here: k_cut 37 (0.21 GB read and written, the rate of a copy), the product 71,
// two launches that find nothing left to do 4.5 each.  The product runs at 1.9 POP/s, 2.3 without its first loads and last stores, with the
// matrix cores busy 44 % of the cycles, the LDS 17 %; a loop of nothing but these matrix instructions on random bytes holds 2.9 to 3.5
// POP/s on this card (power), of a nominal 5.  Deeper prefetch (3
// or 4 buffers), wavefronts of 64 x 64 (half the LDS reads) and operands read a quarter step ahead made no difference.  Other sizes,
// before -> after: 2048 x 4096 x 2048 450 -> 108 us, 64 x 4096 x 4096 152 -> 58, 300 x 9000 x 500 117 -> 56, 100 x 760 x 1070 28.5 -> 25.5.
//
// Bytes.  x = 256 h + l + 128 with h, l in [-128, 127] covers exactly the 16-bit numbers (balanced digits reach 32639 only).  With
// x' = x - 128 a sum of products is sum a'b' + 128 (sum a' + sum b') + 2^14 K: the sums along the inner dimension come out of
// k_cut (per 64 inner indices), a tile adds them up while its first operands are under way.
//
// Range.  l l' and h h' sums stay below 2^14 K and the middle one, l h' + h l', below 2^15 K: K <= MAX_K = 32768 fits 32 bits.
//
// Layout.  As in matmul_rns.hip, units of 16 inner indices: [digit][unit][row of A or column of B][16 bytes]; global loads, the LDS
// tile and the operand reads of the matrix instruction are contiguous 16-byte accesses in this order.
#pragma once

#include <type_traits>

#include "common.hpp"
#include "gl_field.hpp"

namespace i16 {

constexpr int BLOCK = 256;
constexpr int MAX_K = 32768;
constexpr int UNIT = 16;                       // inner indices of a unit
constexpr int STEP = 4;                        // units of a step of the product, and of a sum of k_cut
constexpr int MAX_CUT_BLOCKS = 1020;           // workgroups that cut words into bytes, what is resident at once; each leaves a word that says what it saw
constexpr size_t GATE_BYTES = 16 + 4 * MAX_CUT_BLOCKS;   // whole lines: planes across lines cost their readers and writers 8 %
static_assert(GATE_BYTES % 128 == 0, "");

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// ---- words to bytes ---------------------------------------------------------------------------------------------
struct Side {
    i64 count, pitch;                          // rows of A or columns of B; the same padded
    v4i *planes;                               // [2][units][pitch]
    int *sums;                                 // [units / STEP][pitch]
};

// the low 32 bits of the signed number a word stands for (w, or w - p for the upper half); `beyond` collects bits that are set
// when it has more than 16 bits
__device__ __forceinline__ u32 signed_low(u64 w, u32 &beyond) {
    const u64 s = w + ((i64)w < 0 ? gl::EPS : 0);
    const u64 t = s + 0x8000;
    beyond |= (u32)(t >> 32) | ((u32)t >> 16);
    return (u32)s;
}

// sixteen words of one row or column -> its 16 bytes in either plane; returns the sum of x' = x - 128
__device__ __forceinline__ int store_digits(const u64 (&w)[UNIT], v4i *at, i64 plane, u32 &beyond) {
    v4i lo, hi;
    int sl = 0, sh = 0;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        u32 x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = signed_low(w[4 * g + u], beyond);
        const u32 p01 = __builtin_amdgcn_perm(x[1], x[0], 0x05010400u), p23 = __builtin_amdgcn_perm(x[3], x[2], 0x05010400u);
        lo[g] = (int)(__builtin_amdgcn_perm(p23, p01, 0x05040100u) ^ 0x80808080u);
        hi[g] = (int)__builtin_amdgcn_perm(p23, p01, 0x07060302u);
        sl = __builtin_amdgcn_sdot4(lo[g], 0x01010101, sl, false);
        sh = __builtin_amdgcn_sdot4(hi[g], 0x01010101, sh, false);
    }
    at[0] = lo;
    at[plane] = hi;
    return sl + 256 * sh;
}

// ---- the products -----------------------------------------------------------------------------------------------
// 64 lanes' 16 bytes at base + 16 lane into 1 KiB of LDS, without a register in between; base and dst are the same for the wavefront.
// As an instruction of its own the compiler does not wait for it before the next LDS read, as it does for its builtin: the waits are
// wait_and_meet's.  M0, which it takes its LDS address from, has its value back afterwards: the compiler does not accept it in a list
// of clobbered registers.
__device__ __forceinline__ void fetch_to_lds(const v4i *base, v4i *dst, int lane) {
#ifdef __HIP_DEVICE_COMPILE__
    const u32 at = __builtin_amdgcn_readfirstlane((u32)(uintptr_t)(__attribute__((address_space(3))) v4i *)dst);
    const u32 off = (u32)lane * 16;
    u32 m0;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3\n\ts_mov_b32 m0, %0"
                 : "=&s"(m0) : "s"(at), "v"(off), "s"(base) : "memory");
#else
    dst[lane] = base[lane];
#endif
}
// the wavefront's loads have arrived and its LDS reads are done, then the workgroup's barrier
__device__ __forceinline__ void wait_and_meet() {
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" : : : "memory");
#else
    __syncthreads();
#endif
}

// What k_cut and the launches behind it need to know.
struct Job {
    Side A, B;
    u64 *C;
    i64 *partial;                              // [slices][m][n] sums, for more than one slice of the inner dimension
    u32 *flags;                                // what each workgroup of k_cut saw
    u32 *done;                                 // for the launches behind the product: whether C is finished; NULL: it was not tried
    int units, mt, tiles, slices, steps_per_slice, n_flags;
};

// A tile of 64 MT x 64 NT of C by four wavefronts in a square, MT x NT matrix instructions each: the inner dimension is cut into slices where a product has few tiles.  A step is four units (64 inner indices) of both digits of
// both operands, loaded straight into the one LDS buffer while the other is multiplied.  Three workgroups to a CU cover each other's
// barriers, first loads and last stores (128 x 128 with eight wavefronts and one workgroup to a CU: 2048 x 700 x 11000 108 us, 90 this
// way).  As k_product<1, 2> (matmul_rns.hip) 10 of its 168 registers go to scratch.
template <int MT, int NT>
struct Lds {
    v4i buf[2][2 * STEP * 64 * (MT + NT)];
    int sums[64 * (MT + NT)];
};

template <int MT, int NT>
__device__ __forceinline__ void product(const Job &J, Lds<MT, NT> &lds) {
    constexpr int TM = 64 * MT, TN = 64 * NT;
    constexpr int LOADS = 2 * STEP * (MT + NT) / 4;                    // loads of 64 16-byte words of a step per wavefront
    const Side &A = J.A, &B = J.B;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // consecutive ids of one XCD take tiles that share their columns of B
    const u32 total = (u32)J.tiles, slice = blockIdx.x / total;
    u32 id = blockIdx.x - slice * total;
    if ((total & 7) == 0) id = (id & 7) * (total >> 3) + (id >> 3);
    const int tn = id / J.mt, tm = id - tn * J.mt;
    const int steps = J.units / STEP, s0 = slice * J.steps_per_slice, s1 = min((u32)(s0 + J.steps_per_slice), (u32)steps);

    // load j of the wavefront is chunk wave LOADS + j of the step: [A or B][digit][unit][64 rows]
    const v4i *src[LOADS];
    i64 ahead[LOADS];
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
        int c = wave * LOADS + j;
        const bool is_a = c < 2 * STEP * TM / 64;
        if (!is_a) c -= 2 * STEP * TM / 64;
        const int per = is_a ? TM / 64 : TN / 64, part = c % per, unit = c / per % STEP, digit = c / per / STEP;
        const i64 pitch = is_a ? A.pitch : B.pitch, first = is_a ? (i64)tm * TM : (i64)tn * TN;
        src[j] = (is_a ? A.planes : B.planes) + ((i64)digit * J.units + s0 * STEP + unit) * pitch + first + part * 64;
        ahead[j] = STEP * pitch;
    }
    auto fetch = [&](int stage) {
#pragma unroll
        for (int j = 0; j < LOADS; ++j) {
            fetch_to_lds(src[j], &lds.buf[stage][(wave * LOADS + j) * 64], lane);
            src[j] += ahead[j];
        }
    };

    fetch(0);
    // the sums along the inner dimension: for the whole of it, by the first slice
    if (tid < TM + TN) {
        const bool is_a = tid < TM;
        const i64 pitch = is_a ? A.pitch : B.pitch;
        const int *p = is_a ? A.sums + (i64)tm * TM + tid : B.sums + (i64)tn * TN + tid - TM;
        u32 v = 0;                             // padded rows and columns hold anything: their sums wrap around
        if (slice == 0) {
#pragma unroll 16
            for (int q = 0; q < steps; ++q) v += (u32)p[q * pitch];
        }
        lds.sums[tid] = (int)v;
    }

    v16i ll[MT][NT], mid[MT][NT], hh[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) ll[i][j][r] = mid[i][j][r] = hh[i][j][r] = 0;
    const int row0 = (wave / 2) * (32 * MT) + (lane & 31), col0 = (wave % 2) * (32 * NT) + (lane & 31), half = lane >> 5;
    for (int s = s0; s < s1; ++s) {
        wait_and_meet();
        const v4i *as = lds.buf[(s - s0) & 1], *bs = as + 2 * STEP * TM;
        if (s + 1 < s1) fetch((s - s0 + 1) & 1);
#pragma unroll
        for (int t = 0; t < STEP / 2; ++t) {
            v4i a[2][MT], b[2][NT];
#pragma unroll
            for (int d = 0; d < 2; ++d) {
#pragma unroll
                for (int i = 0; i < MT; ++i) a[d][i] = as[(d * STEP + 2 * t + half) * TM + row0 + 32 * i];
#pragma unroll
                for (int j = 0; j < NT; ++j) b[d][j] = bs[(d * STEP + 2 * t + half) * TN + col0 + 32 * j];
            }
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    ll[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[0][i], b[0][j], ll[i][j], 0, 0, 0);
                    mid[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[0][i], b[1][j], mid[i][j], 0, 0, 0);
                    hh[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[1][i], b[1][j], hh[i][j], 0, 0, 0);
                    mid[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[1][i], b[0][j], mid[i][j], 0, 0, 0);
                }
        }
    }

    // register r of a tile is row 8 (r / 4) + 4 half + r % 4
    const i64 base = slice == 0 ? (i64)J.units * UNIT << 14 : 0;
    auto store = [&](auto whole) {                                     // whole: no row or column of the tile is padding
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int lcol = col0 + 32 * j;
            const i64 col = (i64)tn * TN + lcol;
            if (!whole && col >= B.count) continue;
            const int cs = lds.sums[TM + lcol];
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int lrow = (wave / 2) * (32 * MT) + 32 * i + 8 * (r / 4) + 4 * half + r % 4;
                    const i64 row = (i64)tm * TM + lrow;
                    if (!whole && row >= A.count) continue;
                    const i64 v = (i64)ll[i][j][r] + (i64)mid[i][j][r] * 256 + (i64)hh[i][j][r] * 65536 + ((i64)lds.sums[lrow] + cs) * 128 + base;
                    if (J.slices == 1) J.C[row * B.count + col] = (u64)v + (v < 0 ? gl::P : 0);
                    else J.partial[((i64)slice * A.count + row) * B.count + col] = v;
                }
        }
    };
    if ((i64)(tm + 1) * TM <= A.count && (i64)(tn + 1) * TN <= B.count) store(std::true_type());
    else store(std::false_type());
}

// the sums of the slices -> C, by the threads of a whole launch
__device__ __forceinline__ void add_slices(const Job &J, i64 thread, i64 threads) {
    const i64 mn = J.A.count * J.B.count;
    for (i64 e = thread; e < mn; e += threads) {
        i64 v = 0;
#pragma unroll 4
        for (int q = 0; q < J.slices; ++q) v += J.partial[q * mn + e];
        J.C[e] = (u64)v + (v < 0 ? gl::P : 0);
    }
}

// ---- the host side ----------------------------------------------------------------------------------------------
struct Plan {
    int mt, nt, slices, steps_per_slice;       // 64 mt x 64 nt tiles
    i64 units, mpad, npad;
    size_t a_bytes, b_bytes, sa_bytes, sb_bytes, partial_bytes;
};

inline i64 round_up(i64 v, i64 to) { return (v + to - 1) / to * to; }

inline Plan make_plan(i64 m, i64 k, i64 n) {
    Plan L;
    L.mt = m <= 64 ? 1 : 2;
    L.nt = 3 - L.mt;
    L.mpad = round_up(m, 64 * L.mt);
    L.npad = round_up(n, 64 * L.nt);
    const i64 steps = (k + STEP * UNIT - 1) / (STEP * UNIT), tiles = (L.mpad / (64 * L.mt)) * (L.npad / (64 * L.nt));
    L.units = steps * STEP;
    // slices of the inner dimension until there is a tile for every CU, of at least 8 steps: 16 to 2000 rows, inner dimensions 100 to
    // 12000, twice the tiles or half the steps are within 5 % of it, faster or slower
    i64 slices = 1;
    while (tiles * slices * 2 <= 256 && steps / (slices * 2) >= 8) slices *= 2;
    L.steps_per_slice = (int)((steps + slices - 1) / slices);
    L.slices = (int)((steps + L.steps_per_slice - 1) / L.steps_per_slice);
    L.a_bytes = (size_t)(2 * UNIT) * L.units * L.mpad;
    L.b_bytes = (size_t)(2 * UNIT) * L.units * L.npad;
    L.sa_bytes = (size_t)round_up(4 * steps * L.mpad, 16);
    L.sb_bytes = (size_t)round_up(4 * steps * L.npad, 16);
    L.partial_bytes = L.slices > 1 ? (size_t)8 * L.slices * m * n : 0;
    return L;
}

// the 32-bit sums hold MAX_K inner indices; 1 GiB of bytes is about the scratch that the products through residues take
inline bool takes(i64 m, i64 k, i64 n) {
    if (k > MAX_K) return false;
    const Plan L = make_plan(m, k, n);
    return L.a_bytes + L.b_bytes <= (size_t)1 << 30;
}

// flags first (GATE_BYTES); the rest may be written over once a word has not fitted
inline size_t workspace_bytes(i64 m, i64 k, i64 n) {
    const Plan L = make_plan(m, k, n);
    return GATE_BYTES + L.a_bytes + L.b_bytes + L.sa_bytes + L.sb_bytes + L.partial_bytes;
}

// the places of a job in 16-byte aligned scratch
inline Job make_job(u64 *C, i64 m, i64 k, i64 n, void *ws) {
    const Plan L = make_plan(m, k, n);
    Job J;
    char *p = (char *)ws;
    J.done = (u32 *)p;
    J.flags = J.done + 4;
    p += GATE_BYTES;
    v4i *a = (v4i *)p, *b = (v4i *)(p + L.a_bytes);
    p += L.a_bytes + L.b_bytes;
    J.A = {m, L.mpad, a, (int *)p};
    p += L.sa_bytes;
    J.B = {n, L.npad, b, (int *)p};
    p += L.sb_bytes;
    J.C = C;
    J.partial = (i64 *)p;
    J.units = (int)L.units;
    J.mt = (int)(L.mpad / (64 * L.mt));
    J.tiles = J.mt * (int)(L.npad / (64 * L.nt));
    J.slices = L.slices;
    J.steps_per_slice = L.steps_per_slice;
    J.n_flags = 0;
    return J;
}

}  // namespace i16
