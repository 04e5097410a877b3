// Sumcheck proofs (verinf_amd/csrc/sumcheck.hip) on the CPU, launches and all.
#include <hip/hip_runtime.h>
#include "../../verinf_amd/csrc/sumcheck.hip"
extern "C" const char *simt_error() { return vi::err_buf(); }
extern "C" long simt_launches() { return simt::launches; }
extern "C" int simt_system_stores(const void *p) {
    const auto it = simt::system_stores.find(p);
    return it == simt::system_stores.end() ? 0 : it->second;
}
