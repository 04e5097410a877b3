// Goldilocks field p = 2^64 - 2^32 + 1 for gfx950 wavefronts.
//
// The VALU has no 64-bit multiplier, so a product is built from four 32x32->64
// partial products (v_mad_u64_u32) and reduced with the two identities
//     2^64 = 2^32 - 1   and   2^96 = -1   (mod p).
// Canonical-in / canonical-out; for arbitrary 64-bit inputs add/sub/mul return the
// same word the reference device functions return
// (prover/kernels/goldilocks.cuh:28-81), so elementwise results agree bit for bit
// even on non-canonical operands.
//
// The same header compiles for the host (VI_HD empty) so that the kernels' index
// logic and arithmetic can be exercised by a CPU build in the test-suite.
#pragma once
#include <stdint.h>

#include <type_traits>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define VI_HD __host__ __device__ __forceinline__
#else
#define VI_HD inline
#endif

// Fence for the instruction scheduler (device code only): keeps it from hoisting a
// whole phase's loads above the arithmetic of the previous one, which costs more
// live registers than the latency it hides.
#if defined(__HIP_DEVICE_COMPILE__)
#define VI_SCHED_FENCE() __builtin_amdgcn_sched_barrier(0)
#else
#define VI_SCHED_FENCE() ((void)0)
#endif

typedef uint64_t u64;
typedef uint32_t u32;
typedef int64_t i64;

namespace gl {

constexpr u64 P = 0xFFFFFFFF00000001ull;
constexpr u64 EPS = 0xFFFFFFFFull;   // 2^32 - 1 = 2^64 mod p

#if defined(__HIP_DEVICE_COMPILE__)
// Hand-scheduled gfx950 sequences.  Written from 64-bit C++ the compiler spends a 64-bit compare (two issue
// slots) and two selects on every carry test and builds register pairs with moves: 29 VALU instructions (42
// issue slots) for a product, 7 (11) for a modular sum.  Here a product is 15, a sum 5, a difference 4 and a butterfly 9.
// Corrections by 2^32 - 1 are multiply-adds, which take the same 4.2 cycles as any instruction with a carry: + (2^32 - 1) with its
// carry is 1 * (2^32 - 1) + x, and - (2^32 - 1) behind a borrow is 3 * (-0x55555555) + x with a factor of 3 or 0.  With 32-bit
// additions and masks in their places (18, 6, 5 and 11 instructions; cycles per operation and SIMD at eight wavefronts) a product took 74,
// now 66; a butterfly 44.5, now 36; a 16-point transform 2049, now 1782.  1024 rows 2^16 -> 2^18 2124 -> 2040 us (the clock gives
// some of it back: 2.0 to 2.1 GHz under these loads), proofs over three tables of 2^26 567 -> 559.
// On this chip a VALU instruction that reads a carry or mask needs two
// wait states after the VALU instruction that wrote it; inside an asm block the assembler does not add
// them, so every such pair below is separated by two instructions or an s_nop.  s_or_b64 also writes SCC, which the
// compiler may be holding a loop condition in: the blocks that use it say so in their clobber lists.  A carry that leaves a
// block in an SGPR pair is only read by a scalar instruction, or by a vector instruction at least two
// instructions into the next block.
namespace dev {

__device__ __forceinline__ u64 pack(u32 lo, u32 hi) { return ((u64)hi << 32) | lo; }

// mask ? a : b.  The long encoding, with the mask in a pair of scalar registers: with the mask in VCC a select is the short one,
// which takes 2.8 cycles where an instruction with a carry stands before it but was seen at 23 behind a multiply-add
__device__ __forceinline__ u64 select(u64 mask, u64 a, u64 b) {
    u32 r0 = (u32)a, r1 = (u32)(a >> 32);
    asm("v_cndmask_b32_e64 %[r0], %[b0], %[r0], %[m]\n\t"
        "v_cndmask_b32_e64 %[r1], %[b1], %[r1], %[m]"
        : [r0] "+v"(r0), [r1] "+v"(r1)
        : [b0] "v"((u32)b), [b1] "v"((u32)(b >> 32)), [m] "s"(mask));
    return pack(r0, r1);
}

// d - (2^32 - 1) where a block before has put 3 in m, d itself where it has put 0: 2^32 - 1 = 3 * 0x55555555, so that both
// factors are signed 32-bit words and the first one is an inline constant of a select on the borrow
constexpr int BORROWED = 3;
__device__ __forceinline__ u64 minus_eps(u64 d, u32 m) {
    u64 r;
    asm("v_mad_i64_i32 %[r], vcc, %[m], %[k], %[d]" : [r] "=v"(r) : [m] "v"(m), [k] "s"(-0x55555555), [d] "v"(d) : "vcc");
    return r;
}

// w, plus 2^64 when the carry `cin` is set, lies in [0, 2p): subtract p when it is >= p.
// r = w + (2^32 - 1) mod 2^64 is that difference, and it is the answer exactly when one of the two additions wrapped.
__device__ __forceinline__ u64 canon_tail(u64 w, u64 cin) {
    u64 st, r;
    asm("v_mad_u64_u32 %[r], %[st], 1, -1, %[w]\n\t"
        "s_or_b64 %[st], %[st], %[cin]"
        : [r] "=v"(r), [st] "=&s"(st)
        : [w] "v"(w), [cin] "s"(cin)
        : "scc");
    return select(st, r, w);
}

__device__ __forceinline__ u64 addc(u64 a, u64 b) {
    u32 a0 = (u32)a, a1 = (u32)(a >> 32), b0 = (u32)b, b1 = (u32)(b >> 32);
    u32 s0, s1;
    u64 st;
    asm("v_add_co_u32 %[s0], vcc, %[a0], %[b0]\n\t"
        "s_nop 1\n\t"
        "v_addc_co_u32 %[s1], %[st], %[a1], %[b1], vcc"
        : [s0] "=&v"(s0), [s1] "=v"(s1), [st] "=s"(st)
        : [a0] "v"(a0), [a1] "v"(a1), [b0] "v"(b0), [b1] "v"(b1)
        : "vcc");
    return canon_tail(pack(s0, s1), st);
}

// a - b, minus 2^32 - 1 more when it borrowed
__device__ __forceinline__ u64 sub(u64 a, u64 b) {
    u32 a0 = (u32)a, a1 = (u32)(a >> 32), b0 = (u32)b, b1 = (u32)(b >> 32);
    u32 d0, d1, m;
    asm("v_sub_co_u32 %[d0], vcc, %[a0], %[b0]\n\t"
        "s_nop 1\n\t"
        "v_subb_co_u32 %[d1], vcc, %[a1], %[b1], vcc\n\t"
        "s_nop 1\n\t"
        "v_cndmask_b32_e64 %[m], 0, %[k], vcc"
        : [d0] "=&v"(d0), [d1] "=&v"(d1), [m] "=v"(m)
        : [a0] "v"(a0), [a1] "v"(a1), [b0] "v"(b0), [b1] "v"(b1), [k] "n"(BORROWED)
        : "vcc");
    return minus_eps(pack(d0, d1), m);
}

// (u + v, u - v) of canonical u, v: the two carry chains are interleaved, and the first select waits behind the sum's
// correction, so that no wait has to be inserted but one
__device__ __forceinline__ void bfly(u64 u, u64 v, u64 &sum, u64 &dif) {
    u32 u0 = (u32)u, u1 = (u32)(u >> 32), v0 = (u32)v, v1 = (u32)(v >> 32);
    u32 s0, s1, d0, d1, m;
    u64 st, sb, r, d;
    asm("v_add_co_u32 %[s0], vcc, %[u0], %[v0]\n\t"
        "v_sub_co_u32 %[d0], %[sb], %[u0], %[v0]\n\t"
        "s_nop 0\n\t"
        "v_addc_co_u32 %[s1], %[st], %[u1], %[v1], vcc\n\t"
        "v_subb_co_u32 %[d1], %[sb], %[u1], %[v1], %[sb]"
        : [s0] "=&v"(s0), [s1] "=&v"(s1), [d0] "=&v"(d0), [d1] "=&v"(d1), [st] "=&s"(st), [sb] "=&s"(sb)
        : [u0] "v"(u0), [u1] "v"(u1), [v0] "v"(v0), [v1] "v"(v1)
        : "vcc");
    asm("v_mad_u64_u32 %[r], vcc, 1, -1, %[s]\n\t"
        "s_or_b64 %[st], %[st], vcc\n\t"
        "v_cndmask_b32_e64 %[m], 0, %[n], %[sb]\n\t"
        "v_mad_i64_i32 %[d], vcc, %[m], %[k], %[dd]"
        : [r] "=&v"(r), [m] "=&v"(m), [st] "+s"(st), [d] "=v"(d)
        : [s] "v"(pack(s0, s1)), [dd] "v"(pack(d0, d1)), [sb] "s"(sb), [n] "n"(BORROWED), [k] "s"(-0x55555555)
        : "vcc", "scc");
    sum = select(st, r, pack(s0, s1));
    dif = d;
}

__device__ __forceinline__ u64 canon(u64 x) {
    u64 st, r;
    asm("v_mad_u64_u32 %[r], %[st], 1, -1, %[x]\n\t"
        "s_nop 1"
        : [r] "=v"(r), [st] "=s"(st)
        : [x] "v"(x));
    return select(st, r, x);
}

// (hi:lo) given as four words l0 l1 hl hh, minus the borrow-in `bin`: lo - hh - bin + hl (2^32 - 1) as a word w and a carry st of
// 2^64, together in [0, 2p).  hh + bin must be below 2^32.
__device__ __forceinline__ u64 reduce_words_open(u32 l0, u32 l1, u32 hl, u32 hh, u64 bin, u64 *st) {
    u32 x0, x1, m;
    asm("v_subb_co_u32 %[x0], vcc, %[l0], %[hh], %[bin]\n\t"
        "s_nop 1\n\t"
        "v_subbrev_co_u32 %[x1], vcc, 0, %[l1], vcc\n\t"
        "s_nop 1\n\t"
        "v_cndmask_b32_e64 %[m], 0, %[k], vcc"
        : [x0] "=&v"(x0), [x1] "=&v"(x1), [m] "=v"(m)
        : [l0] "v"(l0), [l1] "v"(l1), [hh] "v"(hh), [bin] "s"(bin), [k] "n"(BORROWED)
        : "vcc");
    u64 w;
    const u64 x = minus_eps(pack(x0, x1), m);
    asm("v_mad_u64_u32 %[w], %[st], %[hl], -1, %[x]"
        : [w] "=v"(w), [st] "=&s"(*st)
        : [hl] "v"(hl), [x] "v"(x));
    return w;
}

// the same -> [0, p)
__device__ __forceinline__ u64 reduce_words(u32 l0, u32 l1, u32 hl, u32 hh, u64 bin) {
    u64 st;
    const u64 w = reduce_words_open(l0, l1, hl, hh, bin, &st);
    return canon_tail(w, st);
}

__device__ __forceinline__ u64 mul(u64 a, u64 b) {
    u32 a0 = (u32)a, a1 = (u32)(a >> 32), b0 = (u32)b, b1 = (u32)(b >> 32);
    u64 p00, mm, p11, st;
    asm("v_mad_u64_u32 %[p00], vcc, %[a0], %[b0], 0\n\t"
        "v_mad_u64_u32 %[mm], vcc, %[a1], %[b0], 0\n\t"
        "v_mad_u64_u32 %[p11], vcc, %[a1], %[b1], 0\n\t"
        "v_mad_u64_u32 %[mm], %[st], %[a0], %[b1], %[mm]"
        : [p00] "=&v"(p00), [mm] "=&v"(mm), [p11] "=&v"(p11), [st] "=&s"(st)
        : [a0] "v"(a0), [a1] "v"(a1), [b0] "v"(b0), [b1] "v"(b1)
        : "vcc");
    // words of the 128-bit product: p00.lo, p00.hi + mm.lo, p11.lo + mm.hi + carry, p11.hi + carry.  The carry of the
    // cross sum (in st) weighs 2^96 = -1: it goes into the reduction as a borrow.
    u32 w1 = (u32)(p00 >> 32), hl, hh;
    asm("v_add_co_u32 %[w1], vcc, %[w1], %[m0]\n\t"
        "s_nop 1\n\t"
        "v_addc_co_u32 %[hl], vcc, %[q0], %[m1], vcc\n\t"
        "s_nop 1\n\t"
        "v_addc_co_u32 %[hh], vcc, 0, %[q1], vcc"
        : [w1] "+v"(w1), [hl] "=&v"(hl), [hh] "=&v"(hh)
        : [m0] "v"((u32)mm), [m1] "v"((u32)(mm >> 32)), [q0] "v"((u32)p11), [q1] "v"((u32)(p11 >> 32))
        : "vcc");
    return reduce_words((u32)p00, w1, hl, hh, st);
}

// the reduction of reduce_words() without its last step: a 64-bit word congruent to the value, not necessarily
// below p; good as an operand of a further product.  The borrow of lo - hh and the carry of + hl (2^32 - 1) weigh -2^64 and 2^64: where one
// of them is set, 2^32 - 1 comes off or on at the end (one correction where reduce_words() has two, and a shorter chain).  The word cannot
// wrap by that: with the carry alone it is at most 2^64 - 2^33, with the borrow alone at least 2^64 - 2^32.
__device__ __forceinline__ u64 reduce_words_lazy(u32 l0, u32 l1, u32 hl, u32 hh, u64 bin) {
    u32 x0, x1, m;
    u64 bo, st, w;
    asm("v_subb_co_u32 %[x0], vcc, %[l0], %[hh], %[bin]\n\t"
        "s_nop 1\n\t"
        "v_subbrev_co_u32 %[x1], %[bo], 0, %[l1], vcc"
        : [x0] "=&v"(x0), [x1] "=v"(x1), [bo] "=s"(bo)
        : [l0] "v"(l0), [l1] "v"(l1), [hh] "v"(hh), [bin] "s"(bin)
        : "vcc");
    asm("v_mad_u64_u32 %[w], %[st], %[hl], -1, %[x]\n\t"
        "s_xor_b64 vcc, %[bo], %[st]\n\t"
        "s_nop 0\n\t"
        "v_cndmask_b32_e64 %[m], %[k3], -%[k3], %[st]\n\t"
        "v_cndmask_b32_e64 %[m], 0, %[m], vcc"
        : [w] "=&v"(w), [m] "=&v"(m), [st] "=&s"(st)
        : [hl] "v"(hl), [x] "v"(pack(x0, x1)), [bo] "s"(bo), [k3] "n"(BORROWED)
        : "vcc", "scc");
    return minus_eps(w, m);
}

// the four partial products of a * b (+ c, a 64-bit addend of the lowest one) as the words l0 l1 hl hh of the
// 128-bit result; *st receives the carry of the cross sum, which weighs 2^96 = -1 and goes into the reduction as a
// borrow
template <bool ADD>
__device__ __forceinline__ void mul_words(u64 a, u64 b, u64 c, u32 &l0, u32 &l1, u32 &hl, u32 &hh, u64 &st) {
    u32 a0 = (u32)a, a1 = (u32)(a >> 32), b0 = (u32)b, b1 = (u32)(b >> 32);
    u64 p00, mm, p11, cy = 0;
    if (ADD) {
        asm("v_mad_u64_u32 %[p00], %[cy], %[a0], %[b0], %[c]\n\t"
            "v_mad_u64_u32 %[mm], vcc, %[a1], %[b0], 0\n\t"
            "v_mad_u64_u32 %[p11], vcc, %[a1], %[b1], 0\n\t"
            "v_mad_u64_u32 %[mm], %[st], %[a0], %[b1], %[mm]"
            : [p00] "=&v"(p00), [mm] "=&v"(mm), [p11] "=&v"(p11), [st] "=&s"(st), [cy] "=&s"(cy)
            : [a0] "v"(a0), [a1] "v"(a1), [b0] "v"(b0), [b1] "v"(b1), [c] "v"(c)
            : "vcc");
    } else {
        asm("v_mad_u64_u32 %[p00], vcc, %[a0], %[b0], 0\n\t"
            "v_mad_u64_u32 %[mm], vcc, %[a1], %[b0], 0\n\t"
            "v_mad_u64_u32 %[p11], vcc, %[a1], %[b1], 0\n\t"
            "v_mad_u64_u32 %[mm], %[st], %[a0], %[b1], %[mm]"
            : [p00] "=&v"(p00), [mm] "=&v"(mm), [p11] "=&v"(p11), [st] "=&s"(st)
            : [a0] "v"(a0), [a1] "v"(a1), [b0] "v"(b0), [b1] "v"(b1)
            : "vcc");
    }
    u32 q0 = (u32)p11, q1 = (u32)(p11 >> 32);
    if (ADD) {
        // the carry of the lowest product plus c weighs 2^64: into a1 b1 <= (2^32 - 1)^2, which cannot overflow
        asm("v_addc_co_u32 %[q0], vcc, 0, %[q0], %[cy]\n\t"
            "s_nop 1\n\t"
            "v_addc_co_u32 %[q1], vcc, 0, %[q1], vcc"
            : [q0] "+v"(q0), [q1] "+v"(q1)
            : [cy] "s"(cy)
            : "vcc");
    }
    u32 w1 = (u32)(p00 >> 32);
    asm("v_add_co_u32 %[w1], vcc, %[w1], %[m0]\n\t"
        "s_nop 1\n\t"
        "v_addc_co_u32 %[hl], vcc, %[q0], %[m1], vcc\n\t"
        "s_nop 1\n\t"
        "v_addc_co_u32 %[hh], vcc, 0, %[q1], vcc"
        : [w1] "+v"(w1), [hl] "=&v"(hl), [hh] "=&v"(hh)
        : [m0] "v"((u32)mm), [m1] "v"((u32)(mm >> 32)), [q0] "v"(q0), [q1] "v"(q1)
        : "vcc");
    l0 = (u32)p00;
    l1 = w1;
}

// a * b + c -> [0, p): the addend rides on the first partial product (17 instructions against 20 for mul + add)
__device__ __forceinline__ u64 mul_add(u64 a, u64 b, u64 c) {
    u32 l0, l1, hl, hh;
    u64 st;
    mul_words<true>(a, b, c, l0, l1, hl, hh, st);
    return reduce_words(l0, l1, hl, hh, st);
}

// a * b + c as a 64-bit word congruent to it, not necessarily below p
__device__ __forceinline__ u64 mul_add_lazy(u64 a, u64 b, u64 c) {
    u32 l0, l1, hl, hh;
    u64 st;
    mul_words<true>(a, b, c, l0, l1, hl, hh, st);
    return reduce_words_lazy(l0, l1, hl, hh, st);
}

// a * b as a 64-bit word congruent to the product, not necessarily below p
__device__ __forceinline__ u64 mul_lazy(u64 a, u64 b) {
    u32 l0, l1, hl, hh;
    u64 st;
    mul_words<false>(a, b, 0, l0, l1, hl, hh, st);
    return reduce_words_lazy(l0, l1, hl, hh, st);
}

// five words w[0..4] (an integer below 2^160) += a * b, the full 128-bit product, nothing reduced: 13 instructions
// against the 20 of a product reduced to [0, p) followed by a modular addition.  The two carry chains (the words
// of the product, the words of the sum) are interleaved so that each carry is read two slots after it was written.
__device__ __forceinline__ void mul_acc(u32 (&w)[5], u64 a, u64 b) {
    u32 a0 = (u32)a, a1 = (u32)(a >> 32), b0 = (u32)b, b1 = (u32)(b >> 32);
    u64 p00, mm, p11, st;
    asm("v_mad_u64_u32 %[p00], vcc, %[a0], %[b0], 0\n\t"
        "v_mad_u64_u32 %[mm], vcc, %[a1], %[b0], 0\n\t"
        "v_mad_u64_u32 %[p11], vcc, %[a1], %[b1], 0\n\t"
        "v_mad_u64_u32 %[mm], %[st], %[a0], %[b1], %[mm]"
        : [p00] "=&v"(p00), [mm] "=&v"(mm), [p11] "=&v"(p11), [st] "=&s"(st)
        : [a0] "v"(a0), [a1] "v"(a1), [b0] "v"(b0), [b1] "v"(b1)
        : "vcc");
    // product words: p00.lo | p00.hi + mm.lo | p11.lo + mm.hi + carry | p11.hi + carry + st (st = carry of the cross
    // sum; the product is below 2^128, so the top word cannot overflow)
    u32 w1 = (u32)(p00 >> 32), hl, hh;
    u64 cb;
    asm("v_add_co_u32 %[w1], vcc, %[w1], %[m0]\n\t"
        "v_add_co_u32 %[A0], %[cb], %[A0], %[w0]\n\t"
        "s_nop 0\n\t"
        "v_addc_co_u32 %[hl], vcc, %[q0], %[m1], vcc\n\t"
        "v_addc_co_u32 %[A1], %[cb], %[A1], %[w1], %[cb]\n\t"
        "s_nop 0\n\t"
        "v_addc_co_u32 %[hh], vcc, 0, %[q1], vcc\n\t"
        "v_addc_co_u32 %[A2], %[cb], %[A2], %[hl], %[cb]\n\t"
        "s_nop 0\n\t"
        "v_addc_co_u32 %[hh], vcc, 0, %[hh], %[st]\n\t"
        "v_addc_co_u32 %[A3], %[cb], %[A3], %[hh], %[cb]\n\t"
        "s_nop 1\n\t"
        "v_addc_co_u32 %[A4], %[cb], 0, %[A4], %[cb]"
        : [w1] "+v"(w1), [hl] "=&v"(hl), [hh] "=&v"(hh), [cb] "=&s"(cb), [A0] "+v"(w[0]), [A1] "+v"(w[1]),
          [A2] "+v"(w[2]), [A3] "+v"(w[3]), [A4] "+v"(w[4])
        : [w0] "v"((u32)p00), [m0] "v"((u32)mm), [m1] "v"((u32)(mm >> 32)), [q0] "v"((u32)p11),
          [q1] "v"((u32)(p11 >> 32)), [st] "s"(st)
        : "vcc");
}

// canonical v times 2^E, 0 <= E < 96, canonical result; s = 32 q + r moves v into limbs m0 m1 m2 at phi^q
// PIN: the three shifts as one asm block.  Plain shifts of a loop-invariant value are hoisted out of a loop even from
// a branch that is not always taken (they are safe to speculate), and then stay live in registers across it; an asm
// block stays where it is written.
// NEG: minus the product, i.e. v times 2^(E + 96); for E >= 32 the last step is a subtraction whose operands swap, so
// the sign is free.
template <int E, bool PIN = false, bool NEG = false>
__device__ __forceinline__ u64 mul_pow2(u64 v) {
    static_assert(E >= 0 && E < 96, "shift out of range");
    if (E == 0) return NEG ? sub(0, v) : v;
    constexpr int q = E >> 5, r = E & 31;
    const u32 v0 = (u32)v, v1 = (u32)(v >> 32);
    if constexpr (q == 1 && r != 0 && !NEG) {
        // v phi 2^r = v0 2^r phi + v1 2^r (phi - 1) = Q phi - R with R = v1 2^r and Q = v0 2^r + R < 2^(33 + r), two
        // multiply-adds in the place of three shifts; Q phi - R = (Q0 + Q1) phi - (Q1 + R).  The carry of Q0 + Q1 and the borrow
        // of the difference cancel where both are set; a borrow alone takes 2^32 - 1 off, a carry alone adds it
        u64 R, Q, T, c, bo, st;
        u32 S, d0, d1, m;
        asm("v_mad_u64_u32 %[R], vcc, %[v1], %[c], 0\n\t"
            "v_mad_u64_u32 %[Q], vcc, %[v0], %[c], %[R]"
            : [R] "=&v"(R), [Q] "=v"(Q)
            : [v0] "v"(v0), [v1] "v"(v1), [c] "s"(1u << r)
            : "vcc");
        const u32 q0 = (u32)Q, q1 = (u32)(Q >> 32);
        asm("v_mad_u64_u32 %[T], vcc, %[q1], 1, %[R]\n\t"
            "v_add_co_u32 %[S], %[c], %[q0], %[q1]"
            : [T] "=&v"(T), [S] "=v"(S), [c] "=&s"(c)
            : [q0] "v"(q0), [q1] "v"(q1), [R] "v"(R)
            : "vcc");
        asm("v_sub_co_u32 %[d0], vcc, 0, %[t0]\n\t"
            "s_nop 1\n\t"
            "v_subb_co_u32 %[d1], vcc, %[S], %[t1], vcc\n\t"
            "s_andn2_b64 %[bo], vcc, %[c]\n\t"
            "s_andn2_b64 %[st], %[c], vcc\n\t"
            "v_cndmask_b32_e64 %[m], 0, %[k], %[bo]"
            : [d0] "=&v"(d0), [d1] "=&v"(d1), [m] "=v"(m), [bo] "=&s"(bo), [st] "=&s"(st)
            : [t0] "v"((u32)T), [t1] "v"((u32)(T >> 32)), [S] "v"(S), [c] "s"(c), [k] "n"(BORROWED)
            : "vcc", "scc");
        return canon_tail(minus_eps(pack(d0, d1), m), st);
    }
    u32 m0, m1, m2;
    if constexpr (PIN && r != 0) {
        asm("v_lshlrev_b32 %[m0], %[r], %[v0]\n\t"
            "v_alignbit_b32 %[m1], %[v1], %[v0], %[c]\n\t"
            "v_lshrrev_b32 %[m2], %[c], %[v1]"
            : [m0] "=&v"(m0), [m1] "=&v"(m1), [m2] "=&v"(m2)
            : [v0] "v"(v0), [v1] "v"(v1), [r] "n"(r), [c] "n"(32 - r));
    } else {
        m0 = v0 << r;
        m1 = r ? __builtin_amdgcn_alignbit(v1, v0, (32 - r) & 31) : v1;
        m2 = r ? (v1 >> ((32 - r) & 31)) : 0u;
    }
    if (q == 0) {
        // m0 + m1 phi + m2 phi^2 = (m1:m0) + m2 (2^32 - 1)
        u64 w, st;
        asm("v_mad_u64_u32 %[w], %[st], %[m2], -1, %[x]"
            : [w] "=&v"(w), [st] "=&s"(st)
            : [m2] "v"(m2), [x] "v"(pack(m0, m1)));
        const u64 x = canon_tail(w, st);
        return NEG ? sub(0, x) : x;
    } else if (q == 1) {
        // m0 phi + m1 phi^2 + m2 phi^3 = (m0:0) + m1 (2^32 - 1) - m2
        u64 w, st;
        asm("v_mad_u64_u32 %[w], %[st], %[m1], -1, %[x]"
            : [w] "=&v"(w), [st] "=&s"(st)
            : [m1] "v"(m1), [x] "v"(pack(0u, m0)));
        const u64 x = canon_tail(w, st);
        if (NEG) return sub((u64)m2, x);                   // m2 = 0 when r = 0
        return r ? sub(x, (u64)m2) : x;
    } else {
        // m0 phi^2 + m1 phi^3 + m2 phi^4 = m0 (2^32 - 1) - (m2:m1); both operands are below p
        u64 e;
        asm("v_mad_u64_u32 %[e], vcc, %[m0], -1, 0" : [e] "=v"(e) : [m0] "v"(m0) : "vcc");
        return NEG ? sub(pack(m1, m2), e) : sub(e, pack(m1, m2));
    }
}

// ---- two at once ------------------------------------------------------------------------------------------------
// The same operations on two independent sets of operands, their instructions interleaved: where a SIMD has four wavefronts, a
// product takes 77 cycles alone and 66 beside another (66 and 64 with eight wavefronts), as its carries are waited for otherwise.

__device__ __forceinline__ void sub2(u64 a, u64 b, u64 &x, u64 c, u64 d, u64 &y) {
    u32 x0, x1, y0, y1, m, n;
    u64 t;
    asm("v_sub_co_u32 %[x0], vcc, %[a0], %[b0]\n\t"
        "v_sub_co_u32 %[y0], %[t], %[c0], %[d0]\n\t"
        "s_nop 0\n\t"
        "v_subb_co_u32 %[x1], vcc, %[a1], %[b1], vcc\n\t"
        "v_subb_co_u32 %[y1], %[t], %[c1], %[d1], %[t]\n\t"
        "s_nop 0\n\t"
        "v_cndmask_b32_e64 %[m], 0, %[k], vcc\n\t"
        "v_cndmask_b32_e64 %[n], 0, %[k], %[t]"
        : [x0] "=&v"(x0), [x1] "=&v"(x1), [y0] "=&v"(y0), [y1] "=&v"(y1), [m] "=&v"(m), [n] "=v"(n), [t] "=&s"(t)
        : [a0] "v"((u32)a), [a1] "v"((u32)(a >> 32)), [b0] "v"((u32)b), [b1] "v"((u32)(b >> 32)), [c0] "v"((u32)c), [c1] "v"((u32)(c >> 32)),
          [d0] "v"((u32)d), [d1] "v"((u32)(d >> 32)), [k] "n"(BORROWED)
        : "vcc");
    x = minus_eps(pack(x0, x1), m);
    y = minus_eps(pack(y0, y1), n);
}

// as bfly: the first carries are read three slots after they were written, the masks of the corrections later still
__device__ __forceinline__ void bfly2(u64 u, u64 v, u64 &sum, u64 &dif, u64 x, u64 y, u64 &sum2, u64 &dif2) {
    u32 s0, s1, d0, d1, t0, t1, e0, e1, m, n;
    u64 st, sb, tt, tb, r, d, z, e;
    asm("v_add_co_u32 %[s0], vcc, %[u0], %[v0]\n\t"
        "v_sub_co_u32 %[d0], %[sb], %[u0], %[v0]\n\t"
        "v_add_co_u32 %[t0], %[tt], %[x0], %[y0]\n\t"
        "v_sub_co_u32 %[e0], %[tb], %[x0], %[y0]\n\t"
        "v_addc_co_u32 %[s1], %[st], %[u1], %[v1], vcc\n\t"
        "v_subb_co_u32 %[d1], %[sb], %[u1], %[v1], %[sb]\n\t"
        "v_addc_co_u32 %[t1], %[tt], %[x1], %[y1], %[tt]\n\t"
        "v_subb_co_u32 %[e1], %[tb], %[x1], %[y1], %[tb]"
        : [s0] "=&v"(s0), [s1] "=&v"(s1), [d0] "=&v"(d0), [d1] "=&v"(d1), [t0] "=&v"(t0), [t1] "=&v"(t1), [e0] "=&v"(e0), [e1] "=&v"(e1),
          [st] "=&s"(st), [sb] "=&s"(sb), [tt] "=&s"(tt), [tb] "=&s"(tb)
        : [u0] "v"((u32)u), [u1] "v"((u32)(u >> 32)), [v0] "v"((u32)v), [v1] "v"((u32)(v >> 32)), [x0] "v"((u32)x), [x1] "v"((u32)(x >> 32)),
          [y0] "v"((u32)y), [y1] "v"((u32)(y >> 32))
        : "vcc");
    asm("v_mad_u64_u32 %[r], vcc, 1, -1, %[s]\n\t"
        "s_or_b64 %[st], %[st], vcc\n\t"
        "v_mad_u64_u32 %[z], vcc, 1, -1, %[t]\n\t"
        "s_or_b64 %[tt], %[tt], vcc\n\t"
        "v_cndmask_b32_e64 %[m], 0, %[k3], %[sb]\n\t"
        "v_cndmask_b32_e64 %[n], 0, %[k3], %[tb]\n\t"
        "v_mad_i64_i32 %[d], vcc, %[m], %[k], %[dd]\n\t"
        "v_mad_i64_i32 %[e], vcc, %[n], %[k], %[ee]"
        : [r] "=&v"(r), [z] "=&v"(z), [m] "=&v"(m), [n] "=&v"(n), [st] "+&s"(st), [tt] "+&s"(tt), [d] "=&v"(d), [e] "=v"(e)
        : [s] "v"(pack(s0, s1)), [dd] "v"(pack(d0, d1)), [t] "v"(pack(t0, t1)), [ee] "v"(pack(e0, e1)), [sb] "s"(sb), [tb] "s"(tb), [k3] "n"(BORROWED),
          [k] "s"(-0x55555555)
        : "vcc", "scc");
    sum = select(st, r, pack(s0, s1));
    sum2 = select(tt, z, pack(t0, t1));
    dif = d;
    dif2 = e;
}

// two words with their carries, as canon_tail
__device__ __forceinline__ void canon_tail2(u64 w, u64 st, u64 &x, u64 v, u64 tt, u64 &y) {
    u64 r, z;
    asm("v_mad_u64_u32 %[r], vcc, 1, -1, %[w]\n\t"
        "s_or_b64 %[st], %[st], vcc\n\t"
        "v_mad_u64_u32 %[z], vcc, 1, -1, %[v]\n\t"
        "s_or_b64 %[tt], %[tt], vcc"
        : [r] "=&v"(r), [z] "=v"(z), [st] "+s"(st), [tt] "+s"(tt)
        : [w] "v"(w), [v] "v"(v)
        : "vcc", "scc");
    x = select(st, r, w);
    y = select(tt, z, v);
}

__device__ __forceinline__ void addc2(u64 a, u64 b, u64 &x, u64 c, u64 d, u64 &y) {
    u32 s0, s1, t0, t1;
    u64 st, tt;
    asm("v_add_co_u32 %[s0], vcc, %[a0], %[b0]\n\t"
        "v_add_co_u32 %[t0], %[tt], %[c0], %[d0]\n\t"
        "s_nop 0\n\t"
        "v_addc_co_u32 %[s1], %[st], %[a1], %[b1], vcc\n\t"
        "v_addc_co_u32 %[t1], %[tt], %[c1], %[d1], %[tt]"
        : [s0] "=&v"(s0), [s1] "=&v"(s1), [t0] "=&v"(t0), [t1] "=&v"(t1), [st] "=&s"(st), [tt] "=&s"(tt)
        : [a0] "v"((u32)a), [a1] "v"((u32)(a >> 32)), [b0] "v"((u32)b), [b1] "v"((u32)(b >> 32)), [c0] "v"((u32)c), [c1] "v"((u32)(c >> 32)),
          [d0] "v"((u32)d), [d1] "v"((u32)(d >> 32))
        : "vcc");
    canon_tail2(pack(s0, s1), st, x, pack(t0, t1), tt, y);
}

// partial products of a b and c d as in mul_words, ADD: with the addends e and f
template <bool ADD>
__device__ __forceinline__ void partial_products2(u64 a, u64 b, u64 e, u64 c, u64 d, u64 f, u64 &p00, u64 &mm, u64 &p11, u64 &st, u64 &cy, u64 &q00, u64 &nn,
                                                  u64 &q11, u64 &tt, u64 &cz) {
    const u32 a0 = (u32)a, a1 = (u32)(a >> 32), b0 = (u32)b, b1 = (u32)(b >> 32), c0 = (u32)c, c1 = (u32)(c >> 32), d0 = (u32)d, d1 = (u32)(d >> 32);
    if (ADD) {
        asm("v_mad_u64_u32 %[mm], vcc, %[a1], %[b0], 0\n\t"
            "v_mad_u64_u32 %[nn], vcc, %[c1], %[d0], 0\n\t"
            "v_mad_u64_u32 %[p00], %[cy], %[a0], %[b0], %[e]\n\t"
            "v_mad_u64_u32 %[q00], %[cz], %[c0], %[d0], %[f]\n\t"
            "v_mad_u64_u32 %[mm], %[st], %[a0], %[b1], %[mm]\n\t"
            "v_mad_u64_u32 %[nn], %[tt], %[c0], %[d1], %[nn]\n\t"
            "v_mad_u64_u32 %[p11], vcc, %[a1], %[b1], 0\n\t"
            "v_mad_u64_u32 %[q11], vcc, %[c1], %[d1], 0"
            : [p00] "=&v"(p00), [mm] "=&v"(mm), [p11] "=&v"(p11), [st] "=&s"(st), [cy] "=&s"(cy), [q00] "=&v"(q00), [nn] "=&v"(nn), [q11] "=&v"(q11),
              [tt] "=&s"(tt), [cz] "=&s"(cz)
            : [a0] "v"(a0), [a1] "v"(a1), [b0] "v"(b0), [b1] "v"(b1), [c0] "v"(c0), [c1] "v"(c1), [d0] "v"(d0), [d1] "v"(d1), [e] "v"(e), [f] "v"(f)
            : "vcc");
    } else {
        asm("v_mad_u64_u32 %[mm], vcc, %[a1], %[b0], 0\n\t"
            "v_mad_u64_u32 %[nn], vcc, %[c1], %[d0], 0\n\t"
            "v_mad_u64_u32 %[p00], vcc, %[a0], %[b0], 0\n\t"
            "v_mad_u64_u32 %[q00], vcc, %[c0], %[d0], 0\n\t"
            "v_mad_u64_u32 %[mm], %[st], %[a0], %[b1], %[mm]\n\t"
            "v_mad_u64_u32 %[nn], %[tt], %[c0], %[d1], %[nn]\n\t"
            "v_mad_u64_u32 %[p11], vcc, %[a1], %[b1], 0\n\t"
            "v_mad_u64_u32 %[q11], vcc, %[c1], %[d1], 0"
            : [p00] "=&v"(p00), [mm] "=&v"(mm), [p11] "=&v"(p11), [st] "=&s"(st), [q00] "=&v"(q00), [nn] "=&v"(nn), [q11] "=&v"(q11), [tt] "=&s"(tt)
            : [a0] "v"(a0), [a1] "v"(a1), [b0] "v"(b0), [b1] "v"(b1), [c0] "v"(c0), [c1] "v"(c1), [d0] "v"(d0), [d1] "v"(d1)
            : "vcc");
    }
}

// x = a b (+ e), y = c d (+ f).  LAZY: words congruent to them, not necessarily below p
template <bool ADD, bool LAZY>
__device__ __forceinline__ void mul2(u64 a, u64 b, u64 e, u64 &x, u64 c, u64 d, u64 f, u64 &y) {
    u64 p00, mm, p11, st, cy, q00, nn, q11, tt, cz;
    partial_products2<ADD>(a, b, e, c, d, f, p00, mm, p11, st, cy, q00, nn, q11, tt, cz);
    u32 g0 = (u32)p11, g1 = (u32)(p11 >> 32), h0 = (u32)q11, h1 = (u32)(q11 >> 32);
    if (ADD) {
        asm("v_addc_co_u32 %[g0], vcc, 0, %[g0], %[cy]\n\t"
            "v_addc_co_u32 %[h0], %[cz], 0, %[h0], %[cz]\n\t"
            "s_nop 0\n\t"
            "v_addc_co_u32 %[g1], vcc, 0, %[g1], vcc\n\t"
            "v_addc_co_u32 %[h1], vcc, 0, %[h1], %[cz]"
            : [g0] "+&v"(g0), [g1] "+&v"(g1), [h0] "+&v"(h0), [h1] "+&v"(h1), [cz] "+&s"(cz)
            : [cy] "s"(cy)
            : "vcc");
    }
    u32 w1 = (u32)(p00 >> 32), v1 = (u32)(q00 >> 32), hl, hh, kl, kh, x0, x1, y0, y1, m, n;
    u64 t, bo;
    asm("v_add_co_u32 %[w1], vcc, %[w1], %[m0]\n\t"
        "v_add_co_u32 %[v1], %[t], %[v1], %[n0]\n\t"
        "s_nop 0\n\t"
        "v_addc_co_u32 %[hl], vcc, %[g0], %[m1], vcc\n\t"
        "v_addc_co_u32 %[kl], %[t], %[h0], %[n1], %[t]\n\t"
        "s_nop 0\n\t"
        "v_addc_co_u32 %[hh], vcc, 0, %[g1], vcc\n\t"
        "v_subb_co_u32 %[x0], vcc, %[l0], %[hh], %[st]\n\t"
        "v_addc_co_u32 %[kh], %[t], 0, %[h1], %[t]\n\t"
        "v_subb_co_u32 %[y0], %[t], %[k0], %[kh], %[tt]\n\t"
        "v_subbrev_co_u32 %[x1], %[bo], 0, %[w1], vcc\n\t"
        "s_nop 0\n\t"
        "v_subbrev_co_u32 %[y1], %[t], 0, %[v1], %[t]"
        : [w1] "+&v"(w1), [v1] "+&v"(v1), [hl] "=&v"(hl), [hh] "=&v"(hh), [kl] "=&v"(kl), [kh] "=&v"(kh), [x0] "=&v"(x0), [x1] "=&v"(x1),
          [y0] "=&v"(y0), [y1] "=&v"(y1), [t] "=&s"(t), [bo] "=&s"(bo)
        : [l0] "v"((u32)p00), [m0] "v"((u32)mm), [m1] "v"((u32)(mm >> 32)), [g0] "v"(g0), [g1] "v"(g1), [st] "s"(st),
          [k0] "v"((u32)q00), [n0] "v"((u32)nn), [n1] "v"((u32)(nn >> 32)), [h0] "v"(h0), [h1] "v"(h1), [tt] "s"(tt)
        : "vcc");
    u64 w, v;
    if (LAZY) {
        asm("v_mad_u64_u32 %[w], %[st], %[hl], -1, %[x]\n\t"
            "v_mad_u64_u32 %[v], %[tt], %[kl], -1, %[y]\n\t"
            "s_xor_b64 %[bo], %[bo], %[st]\n\t"
            "s_xor_b64 %[t], %[t], %[tt]\n\t"
            "v_cndmask_b32_e64 %[m], %[k3], -%[k3], %[st]\n\t"
            "v_cndmask_b32_e64 %[n], %[k3], -%[k3], %[tt]\n\t"
            "v_cndmask_b32_e64 %[m], 0, %[m], %[bo]\n\t"
            "v_cndmask_b32_e64 %[n], 0, %[n], %[t]"
            : [w] "=&v"(w), [v] "=&v"(v), [m] "=&v"(m), [n] "=&v"(n), [st] "=&s"(st), [tt] "=&s"(tt), [bo] "+&s"(bo), [t] "+&s"(t)
            : [hl] "v"(hl), [kl] "v"(kl), [x] "v"(pack(x0, x1)), [y] "v"(pack(y0, y1)), [k3] "n"(BORROWED)
            : "scc");
        x = minus_eps(w, m);
        y = minus_eps(v, n);
    } else {
        u64 X, Y;
        asm("s_nop 0\n\t"
            "v_cndmask_b32_e64 %[m], 0, %[k3], %[bo]\n\t"
            "v_cndmask_b32_e64 %[n], 0, %[k3], %[t]\n\t"
            "v_mad_i64_i32 %[X], vcc, %[m], %[k], %[x]\n\t"
            "v_mad_i64_i32 %[Y], vcc, %[n], %[k], %[y]\n\t"
            "v_mad_u64_u32 %[w], %[st], %[hl], -1, %[X]\n\t"
            "v_mad_u64_u32 %[v], %[tt], %[kl], -1, %[Y]"
            : [X] "=&v"(X), [Y] "=&v"(Y), [w] "=&v"(w), [v] "=&v"(v), [m] "=&v"(m), [n] "=&v"(n), [st] "=&s"(st), [tt] "=&s"(tt)
            : [bo] "s"(bo), [t] "s"(t), [hl] "v"(hl), [kl] "v"(kl), [x] "v"(pack(x0, x1)), [y] "v"(pack(y0, y1)), [k3] "n"(BORROWED), [k] "s"(-0x55555555)
            : "vcc");
        canon_tail2(w, st, x, v, tt, y);
    }
}

// A += a b, B += c d as in mul_acc
__device__ __forceinline__ void mul_acc2(u32 (&A)[5], u64 a, u64 b, u32 (&B)[5], u64 c, u64 d) {
    u64 p00, mm, p11, st, cy, q00, nn, q11, tt, cz;
    partial_products2<false>(a, b, 0, c, d, 0, p00, mm, p11, st, cy, q00, nn, q11, tt, cz);
    u32 w1 = (u32)(p00 >> 32), v1 = (u32)(q00 >> 32), hl, hh, kl, kh;
    u64 ca, cb, t;
    asm("v_add_co_u32 %[w1], vcc, %[w1], %[m0]\n\t"
        "v_add_co_u32 %[v1], %[t], %[v1], %[n0]\n\t"
        "v_add_co_u32 %[A0], %[ca], %[A0], %[l0]\n\t"
        "v_add_co_u32 %[B0], %[cb], %[B0], %[k0]\n\t"
        "v_addc_co_u32 %[hl], vcc, %[g0], %[m1], vcc\n\t"
        "v_addc_co_u32 %[kl], %[t], %[h0], %[n1], %[t]\n\t"
        "v_addc_co_u32 %[A1], %[ca], %[A1], %[w1], %[ca]\n\t"
        "v_addc_co_u32 %[B1], %[cb], %[B1], %[v1], %[cb]\n\t"
        "v_addc_co_u32 %[hh], vcc, 0, %[g1], vcc\n\t"
        "v_addc_co_u32 %[kh], %[t], 0, %[h1], %[t]\n\t"
        "v_addc_co_u32 %[A2], %[ca], %[A2], %[hl], %[ca]\n\t"
        "v_addc_co_u32 %[B2], %[cb], %[B2], %[kl], %[cb]\n\t"
        "v_addc_co_u32 %[hh], vcc, 0, %[hh], %[st]\n\t"
        "v_addc_co_u32 %[kh], vcc, 0, %[kh], %[tt]\n\t"
        "v_addc_co_u32 %[A3], %[ca], %[A3], %[hh], %[ca]\n\t"
        "v_addc_co_u32 %[B3], %[cb], %[B3], %[kh], %[cb]\n\t"
        "s_nop 0\n\t"
        "v_addc_co_u32 %[A4], vcc, 0, %[A4], %[ca]\n\t"
        "v_addc_co_u32 %[B4], vcc, 0, %[B4], %[cb]"
        : [w1] "+&v"(w1), [v1] "+&v"(v1), [hl] "=&v"(hl), [hh] "=&v"(hh), [kl] "=&v"(kl), [kh] "=&v"(kh), [t] "=&s"(t), [ca] "=&s"(ca), [cb] "=&s"(cb),
          [A0] "+&v"(A[0]), [A1] "+&v"(A[1]), [A2] "+&v"(A[2]), [A3] "+&v"(A[3]), [A4] "+&v"(A[4]),
          [B0] "+&v"(B[0]), [B1] "+&v"(B[1]), [B2] "+&v"(B[2]), [B3] "+&v"(B[3]), [B4] "+&v"(B[4])
        : [l0] "v"((u32)p00), [m0] "v"((u32)mm), [m1] "v"((u32)(mm >> 32)), [g0] "v"((u32)p11), [g1] "v"((u32)(p11 >> 32)), [st] "s"(st),
          [k0] "v"((u32)q00), [n0] "v"((u32)nn), [n1] "v"((u32)(nn >> 32)), [h0] "v"((u32)q11), [h1] "v"((u32)(q11 >> 32)), [tt] "s"(tt)
        : "vcc");
}

}  // namespace dev
#endif

VI_HD u64 add(u64 a, u64 b) {
    u64 s = a + b;
    if (s < a) s += EPS;             // wrapped past 2^64: add 2^64 mod p
    if (s >= P) s -= P;
    return s;
}

VI_HD u64 sub(u64 a, u64 b) {
#if defined(__HIP_DEVICE_COMPILE__)
    return dev::sub(a, b);
#endif
    u64 d = a - b;
    if (a < b) d -= EPS;             // borrowed 2^64: take 2^64 mod p back out
    return d;
}

VI_HD u64 neg(u64 a) { return a == 0 ? 0 : P - a; }

// Sum of two CANONICAL values (cheaper than add(): the wrap past 2^64 and the
// overshoot past p take the same correction, + (2^32 - 1) mod 2^64, so one select
// serves both).  Not for arbitrary words: with both operands >= p it can be wrong.
VI_HD u64 addc(u64 a, u64 b) {
#if defined(__HIP_DEVICE_COMPILE__)
    return dev::addc(a, b);
#endif
    u64 s = a + b;
    u64 r = s + EPS;
    return ((s < a) | (r < s)) ? r : s;
}

// (u + v, u - v) for canonical u, v
VI_HD void bfly(u64 u, u64 v, u64 &sum, u64 &dif) {
#if defined(__HIP_DEVICE_COMPILE__)
    dev::bfly(u, v, sum, dif);
#else
    sum = addc(u, v);
    dif = sub(u, v);
#endif
}

// x mod p for an arbitrary 64-bit word
VI_HD u64 canon(u64 x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return dev::canon(x);
#endif
    u64 r = x + EPS;
    return (r < x) ? r : x;
}

// (hi:lo) -> [0, p).  hi = hh*2^32 + hl  =>  value = lo - hh + hl*(2^32 - 1).
VI_HD u64 reduce128(u64 lo, u64 hi) {
#if defined(__HIP_DEVICE_COMPILE__)
    return dev::reduce_words((u32)lo, (u32)(lo >> 32), (u32)hi, (u32)(hi >> 32), 0);
#endif
    u32 hh = (u32)(hi >> 32), hl = (u32)hi;
    u64 t0 = lo - hh;
    if (lo < hh) t0 -= EPS;
    u64 t1 = ((u64)hl << 32) - hl;   // hl * (2^32 - 1), no multiplier needed
    u64 r = t0 + t1;
    if (r < t0) r += EPS;
    if (r >= P) r -= P;
    return r;
}

// (hi:lo) -> some 64-bit word congruent to it (not necessarily below p): reduce128 without
// its last conditional subtraction.  Good enough as an operand of mul / mul_wide.
VI_HD u64 reduce128_lazy(u64 lo, u64 hi) {
    u32 hh = (u32)(hi >> 32), hl = (u32)hi;
    u64 t0 = lo - hh;
    if (lo < hh) t0 -= EPS;
    u64 t1 = ((u64)hl << 32) - hl;
    u64 r = t0 + t1;
    if (r < t0) r += EPS;
    return r;
}

// 64x64 -> 128 from 32-bit halves; every line is one v_mad_u64_u32 (the addends
// cannot overflow: (2^32-1)^2 + 2*(2^32-1) < 2^64).
VI_HD void mul_wide(u64 a, u64 b, u64 &lo, u64 &hi) {
    u32 a0 = (u32)a, a1 = (u32)(a >> 32), b0 = (u32)b, b1 = (u32)(b >> 32);
    u64 p00 = (u64)a0 * b0;
    u64 p01 = (u64)a0 * b1 + (p00 >> 32);
    u64 p10 = (u64)a1 * b0 + (u32)p01;
    u64 p11 = (u64)a1 * b1 + (p01 >> 32) + (p10 >> 32);
    lo = (p10 << 32) | (u32)p00;
    hi = p11;
}

VI_HD u64 mul(u64 a, u64 b) {
#if defined(__HIP_DEVICE_COMPILE__)
    return dev::mul(a, b);
#endif
    u64 lo, hi;
    mul_wide(a, b, lo, hi);
    return reduce128(lo, hi);
}

// a * b + c in [0, p) for any words a, b, c
VI_HD u64 mul_add(u64 a, u64 b, u64 c) {
#if defined(__HIP_DEVICE_COMPILE__)
    return dev::mul_add(a, b, c);
#endif
    return add(mul(a, b), canon(c));
}

// a * b + c as a word congruent to it, not necessarily below p
VI_HD u64 mul_add_lazy(u64 a, u64 b, u64 c) {
#if defined(__HIP_DEVICE_COMPILE__)
    return dev::mul_add_lazy(a, b, c);
#endif
    return mul_add(a, b, c);
}

// product as a non-canonical word (see reduce128_lazy): for chains of multiplications
VI_HD u64 mul_lazy(u64 a, u64 b) {
#if defined(__HIP_DEVICE_COMPILE__)
    return dev::mul_lazy(a, b);
#endif
    u64 lo, hi;
    mul_wide(a, b, lo, hi);
    return reduce128_lazy(lo, hi);
}

// two at once (dev::mul2 and its neighbours): x from the first operands, y from the second
VI_HD void sub2(u64 a, u64 b, u64 &x, u64 c, u64 d, u64 &y) {
#if defined(__HIP_DEVICE_COMPILE__)
    dev::sub2(a, b, x, c, d, y);
#else
    const u64 first = sub(a, b);
    y = sub(c, d);
    x = first;
#endif
}
VI_HD void addc2(u64 a, u64 b, u64 &x, u64 c, u64 d, u64 &y) {
#if defined(__HIP_DEVICE_COMPILE__)
    dev::addc2(a, b, x, c, d, y);
#else
    const u64 first = addc(a, b);
    y = addc(c, d);
    x = first;
#endif
}
VI_HD void bfly2(u64 u, u64 v, u64 &sum, u64 &dif, u64 x, u64 y, u64 &sum2, u64 &dif2) {
#if defined(__HIP_DEVICE_COMPILE__)
    dev::bfly2(u, v, sum, dif, x, y, sum2, dif2);
#else
    const u64 s = addc(u, v), d = sub(u, v);
    bfly(x, y, sum2, dif2);
    sum = s;
    dif = d;
#endif
}
VI_HD void mul2(u64 a, u64 b, u64 &x, u64 c, u64 d, u64 &y) {
#if defined(__HIP_DEVICE_COMPILE__)
    dev::mul2<false, false>(a, b, 0, x, c, d, 0, y);
#else
    const u64 first = mul(a, b);
    y = mul(c, d);
    x = first;
#endif
}
VI_HD void mul_lazy2(u64 a, u64 b, u64 &x, u64 c, u64 d, u64 &y) {
#if defined(__HIP_DEVICE_COMPILE__)
    dev::mul2<false, true>(a, b, 0, x, c, d, 0, y);
#else
    const u64 first = mul_lazy(a, b);
    y = mul_lazy(c, d);
    x = first;
#endif
}
VI_HD void mul_add2(u64 a, u64 b, u64 e, u64 &x, u64 c, u64 d, u64 f, u64 &y) {
#if defined(__HIP_DEVICE_COMPILE__)
    dev::mul2<true, false>(a, b, e, x, c, d, f, y);
#else
    const u64 first = mul_add(a, b, e);
    y = mul_add(c, d, f);
    x = first;
#endif
}

// Sums of products kept as plain integers: five 32-bit words, reduced once at the end.
struct Wide {
    u32 w[5];
};
VI_HD void wide_zero(Wide &A) {
    for (int i = 0; i < 5; ++i) A.w[i] = 0;
}
// A += a * b (any 64-bit words); the caller keeps the number of products below 2^32
VI_HD void wide_mul_acc(Wide &A, u64 a, u64 b) {
#if defined(__HIP_DEVICE_COMPILE__)
    dev::mul_acc(A.w, a, b);
#else
    u64 lo, hi;
    mul_wide(a, b, lo, hi);
    const u64 add[4] = {(u32)lo, lo >> 32, (u32)hi, hi >> 32};
    u64 carry = 0;
    for (int i = 0; i < 5; ++i) {
        const u64 t = (u64)A.w[i] + (i < 4 ? add[i] : 0) + carry;
        A.w[i] = (u32)t;
        carry = t >> 32;
    }
#endif
}
// A += a * b and B += c * d
VI_HD void wide_mul_acc2(Wide &A, u64 a, u64 b, Wide &B, u64 c, u64 d) {
#if defined(__HIP_DEVICE_COMPILE__)
    dev::mul_acc2(A.w, a, b, B.w, c, d);
#else
    wide_mul_acc(A, a, b);
    wide_mul_acc(B, c, d);
#endif
}
// the integer mod p: words 0..3 as a 128-bit value, word 4 weighs 2^128 = -2^32
VI_HD u64 wide_reduce(const Wide &A) {
    const u64 x = reduce128(((u64)A.w[1] << 32) | A.w[0], ((u64)A.w[3] << 32) | A.w[2]);
    return sub(x, (u64)A.w[4] << 32);
}

VI_HD u64 pow(u64 base, u64 e) {
    u64 r = 1;
    while (e) {
        if (e & 1) r = mul(r, base);
        base = mul(base, base);
        e >>= 1;
    }
    return r;
}

VI_HD u64 sqr_n(u64 x, int n) {
    for (int i = 0; i < n; ++i) x = mul_lazy(x, x);
    return x;
}

// x^(p-2) by a fixed addition chain: p - 2 = (2^31 - 1) * 2^33 + (2^32 - 1), and x^(2^k - 1)
// doubles its k with k squarings and one product.  64 squarings + 10 products instead of the
// 63 + 62 of square-and-multiply; 0 -> 0 like the Fermat power.  Every value but the last only feeds a product, so the
// chain runs on lazily reduced words (its length is what a wavefront that inverts waits for).
VI_HD u64 inv(u64 x) {
    u64 a2 = mul_lazy(sqr_n(x, 1), x);            // 2^2 - 1
    u64 a4 = mul_lazy(sqr_n(a2, 2), a2);
    u64 a8 = mul_lazy(sqr_n(a4, 4), a4);
    u64 a16 = mul_lazy(sqr_n(a8, 8), a8);
    u64 a24 = mul_lazy(sqr_n(a16, 8), a8);
    u64 a28 = mul_lazy(sqr_n(a24, 4), a4);
    u64 a30 = mul_lazy(sqr_n(a28, 2), a2);
    u64 a31 = mul_lazy(sqr_n(a30, 1), x);         // 2^31 - 1
    u64 a32 = mul_lazy(sqr_n(a31, 1), x);         // 2^32 - 1
    return mul(sqr_n(a31, 33), a32);
}

// canonical x times 2^s for 0 <= s < 96, as shifts: the 64-bit value moved left by
// s bits occupies at most three 32-bit limbs L[q..q+2] (s = 32q + r) of
//   L0 + L1*phi + L2*phi^2 + L3*phi^3 + L4*phi^4,  phi = 2^32,
// and phi^2 = phi - 1, phi^3 = -1, phi^4 = -phi fold it back to two limbs.
VI_HD u64 mul_pow2(u64 x, u32 s) {
    u32 q = s >> 5, r = s & 31;
    u32 x0 = (u32)x, x1 = (u32)(x >> 32);
    u32 m0 = x0 << r;
    u32 m1 = r ? ((x1 << r) | (x0 >> (32 - r))) : x1;
    u32 m2 = r ? (x1 >> (32 - r)) : 0;
    if (q == 0) return reduce128(((u64)m1 << 32) | m0, (u64)m2);            // m0 + m1 phi + m2 phi^2
    if (q == 1) return reduce128((u64)m0 << 32, ((u64)m2 << 32) | m1);      // m0 phi + m1 phi^2 + m2 phi^3
    // q == 2: m0 phi^2 + m1 phi^3 + m2 phi^4 = (m0 - m2) phi - (m0 + m1)
    u64 pos = (u64)m0 << 32;                       // m0 * phi            < p
    u64 negv = (u64)m2 << 32;                      // m2 * phi            < p
    u64 small = (u64)m0 + (u64)m1;                 // < 2^33              < p
    return sub(sub(pos, negv), small);
}

// the same with the exponent fixed at compile time
template <int E>
VI_HD u64 mul_pow2c(u64 x) {
#if defined(__HIP_DEVICE_COMPILE__)
    return dev::mul_pow2<E>(x);
#else
    return mul_pow2(x, (u32)E);
#endif
}

// x times 2^E for any exponent (2^192 = 1, 2^96 = -1), for use inside a branch of a loop on a value the loop does
// not change (see dev::mul_pow2)
template <int E>
VI_HD u64 mul_pow2c_pinned(u64 x) {
    constexpr int e = ((E % 192) + 192) % 192;
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (e < 96) return dev::mul_pow2<e, true, false>(x);
    else return dev::mul_pow2<e - 96, true, true>(x);
#else
    return e < 96 ? mul_pow2(x, (u32)e) : sub(0, mul_pow2(x, (u32)(e - 96)));
#endif
}

}  // namespace gl

// compile-time loop: f(std::integral_constant<int, I>) for I in [I0, N)
template <int I0, int N, class F>
VI_HD void static_for(F &&f) {
    if constexpr (I0 < N) {
        f(std::integral_constant<int, I0>{});
        static_for<I0 + 1, N>(f);
    }
}
