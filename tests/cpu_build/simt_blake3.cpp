// Column digests, trees and pads (verinf_amd/csrc/blake3.hip) on the CPU, launches and all.
#include <hip/hip_runtime.h>
#include "../../verinf_amd/csrc/blake3.hip"
extern "C" const char *simt_error() { return vi::err_buf(); }
