// The look-up counts (verinf_amd/csrc/lookup.hip) on the CPU, launches and all.
#include <hip/hip_runtime.h>

namespace {
thread_local uint4 lds_counts[163840 / 16];                            // the dynamic LDS of its kernels
}
#include "../../verinf_amd/csrc/lookup.hip"

extern "C" const char *simt_error() { return vi::err_buf(); }
extern "C" long simt_launches() { return simt::launches; }
