// Multilinear helpers (verinf_amd/csrc/mle.hip) on the CPU, launches and all.
#include <hip/hip_runtime.h>
#include "../../verinf_amd/csrc/mle.hip"
extern "C" const char *simt_error() { return vi::err_buf(); }
