// Resident PCG (real) and COCG (complex symmetric) solves: instantiations of
// k_resident and their cooperative launch.
#include "krylov_resident.hpp"
#include "krylov_resident_launch.hpp"

namespace tmi {

bool launch_resident_cg(VKind vk, int cl, int E, bool cocg, bool mf, const ResArgs &a, size_t lds, hipStream_t st)
{
#define ONE(V, CL, EE, M, MF) \
    if (cl == CL && E == EE) return coop_launch(k_resident<V, CL, EE, M, MF>, lds, a, st);
#define ALL8(V, M, MF)                                                              \
    ONE(V, 1, 1, M, MF) ONE(V, 1, 2, M, MF) ONE(V, 1, 4, M, MF) ONE(V, 1, 8, M, MF) \
    ONE(V, 4, 1, M, MF) ONE(V, 4, 2, M, MF) ONE(V, 4, 4, M, MF)
#define ALL16(V, M, MF)                                                             \
    ONE(V, 1, 1, M, MF) ONE(V, 1, 2, M, MF) ONE(V, 1, 4, M, MF) ONE(V, 1, 8, M, MF) \
    ONE(V, 2, 1, M, MF) ONE(V, 2, 2, M, MF) ONE(V, 2, 4, M, MF)
    if (cocg) {
        if (vk == VK_C32) {
            if (mf) { ALL8(float2, RES_COCG, true) }
            else { ALL8(float2, RES_COCG, false) }
        } else if (vk == VK_C64) {
            if (mf) { ALL16(double2, RES_COCG, true) }
            else { ALL16(double2, RES_COCG, false) }
        }
    } else if (vk == VK_R32) { ALL8(float, RES_CG, false) }
    else if (vk == VK_R64) { ALL8(double, RES_CG, false) }
    return false;
}

}  // namespace tmi
