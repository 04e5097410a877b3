#include <hip/hip_runtime.h>
#include "../../verinf_amd/csrc/ntt.hip"
extern "C" const char *simt_error() { return vi::err_buf(); }
extern "C" long simt_launches() { return simt::launches; }
