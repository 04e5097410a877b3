#include <hip/hip_runtime.h>
#include "../../verinf_amd/csrc/ntt.hip"
extern "C" const char *simt_error() { return vi::err_buf(); }
extern "C" long simt_launches() { return simt::launches; }

// In front of the next launch, extensions with `count` other shifts, as another thread may make them there.
extern "C" void simt_other_shifts(int count) {
    simt::before_launch = [count] {
        std::vector<u64> in(8, 1), out(16), ws(vi_coset_lde_workspace_bytes(1, 8, 16) / 8);
        for (int i = 0; i < count; ++i)
            if (vi_coset_lde(in.data(), 1, 8, 8, 8, 16, 1000 + (u64)i, out.data(), 16, ws.data(), ws.size() * 8, nullptr)) abort();
    };
}
