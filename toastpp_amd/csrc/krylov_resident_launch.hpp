// Cooperative launch of a resident solve kernel.
#pragma once
#include "krylov_resident.hpp"

namespace tmi {

// All RES_WG workgroups must run at once (they wait for each other), which a
// cooperative launch guarantees or refuses.  false: refused -- the kernel
// does not fit one workgroup per CU, or the device has fewer CUs.
template <class F>
inline bool coop_launch(F *kernel, size_t lds, const ResArgs &a, hipStream_t st)
{
    int per_cu = 0;
    if (Context::get().num_cu < RES_WG) return false;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)kernel, RES_NT, lds) != hipSuccess ||
        per_cu < 1) {
        (void)hipGetLastError();
        return false;
    }
    ResArgs args = a;
    void *params[] = {&args};
    const hipError_t e = hipLaunchCooperativeKernel((const void *)kernel, dim3(RES_WG), dim3(RES_NT), params,
                                                    (unsigned)lds, st);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    ++g_launch_calls;
    return true;
}

}  // namespace tmi
