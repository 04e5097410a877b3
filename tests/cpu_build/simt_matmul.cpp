// Field products through residues (verinf_amd/csrc/matmul_rns.hip) and of small numbers (matmul_i16.hpp) on the CPU, launches and all.
#include <hip/hip_runtime.h>
#include "../../verinf_amd/csrc/matmul_rns.hip"

extern "C" size_t simt_matmul_workspace(int64_t m, int64_t k, int64_t n) { return vi::rns_matmul_workspace_bytes(m, k, n); }
extern "C" int simt_matmul(const uint64_t *A, const uint64_t *B, uint64_t *C, int64_t m, int64_t k, int64_t n, void *ws) {
    return vi::rns_matmul(A, B, C, m, k, n, ws, nullptr);
}

// One workgroup tile of the larger shapes, which rns_matmul takes for many of them only: m <= 128, n <= 256 (wn = 4) or 128 (2), any k
// of one slice.
template <int WN, int OCC, bool STRAIGHT>
static void one_tile(const u64 *A, const u64 *B, u64 *C, i64 m, i64 k, i64 n, void *ws) {
    const i64 mpad = 128, npad = 64 * WN, units = round_up(k, STEP_UNITS * UNIT) / UNIT;
    v4i *Ap = (v4i *)vi::align16(ws), *Bp = Ap + NMOD * units * mpad;
    u32 *Cp = (u32 *)(Bp + NMOD * units * npad);
    ModConst K;
    for (int i = 0; i < NMOD; ++i) {
        K.m[i] = (u32)MODS[i];
        K.inv[i] = (u32)((1ull << 32) / (u32)MODS[i]);
        K.off[i] = (u32)MODS[i] * ((1u << 28) / (u32)MODS[i] + 1);
    }
    const Operand OA = {A, k, m, mpad, Ap, (unsigned)((m + LINES - 1) / LINES)}, OB = {B, n, n, npad, Bp, (unsigned)((n + LINES - 1) / LINES)};
    const unsigned chunks = (unsigned)(units / ITEM_UNITS), b_items = OB.groups * chunks;
    const unsigned wide = (unsigned)((n + BLOCK - 1) / BLOCK), b_slabs = wide * (unsigned)units;
    const Cut D = {OA, OB, k, (int)units, b_items, b_items + OA.groups * chunks, wide, b_slabs, b_slabs + OA.groups * chunks};
    hipLaunchKernelGGL(k_residues, dim3(D.slabs), dim3(BLOCK), 0, nullptr, D, (const u32 *)nullptr);
    launch_gemm<2, WN, OCC, STRAIGHT>(Ap, Bp, Cp, (int)units, mpad, npad, K, nullptr, nullptr);
    hipLaunchKernelGGL(k_from_residues, dim3((unsigned)((n + BLOCK - 1) / BLOCK), (unsigned)((m + 3) / 4)), dim3(BLOCK), 0, nullptr, (const u32 *)Cp,
                       mpad / 4 * npad, npad, C, n, m, n, 0, i16::Job{});
}
extern "C" size_t simt_tile_workspace(int64_t k, int wn) {
    return NMOD * (size_t)(round_up(k, STEP_UNITS * UNIT) * (128 + 64 * wn) + 128 * 64 * wn) + vi::WS_SLACK;
}
extern "C" void simt_tile(const uint64_t *A, const uint64_t *B, uint64_t *C, int64_t m, int64_t k, int64_t n, int wn, void *ws) {
    if (wn == 4) one_tile<4, 2, true>(A, B, C, m, k, n, ws);
    else if (k < 4000) one_tile<2, 3, true>(A, B, C, m, k, n, ws);
    else one_tile<2, 3, false>(A, B, C, m, k, n, ws);
}
