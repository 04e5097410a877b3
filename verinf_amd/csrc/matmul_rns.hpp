// C = A B over the field on the matrix cores (matmul_rns.hip), behind vi_gl_matmul in linalg.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace vi {

// whether this path is the faster one for the shape (see the rule in matmul_rns.hip)
bool rns_matmul_pays(int64_t m, int64_t k, int64_t n);
size_t rns_matmul_workspace_bytes(int64_t m, int64_t k, int64_t n);
// m, k, n >= 1; ws holds rns_matmul_workspace_bytes()
int rns_matmul(const uint64_t *A, const uint64_t *B, uint64_t *C, int64_t m, int64_t k, int64_t n, void *ws, hipStream_t s);

}  // namespace vi
