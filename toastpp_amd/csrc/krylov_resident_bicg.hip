// Resident BiCGSTAB solves: instantiations of k_resident and their
// cooperative launch.
#include "krylov_resident.hpp"
#include "krylov_resident_launch.hpp"

namespace tmi {

bool launch_resident_bicg(VKind vk, int cl, int E, const ResArgs &a, size_t lds, hipStream_t st)
{
#define ONE(V, CL, EE) \
    if (cl == CL && E == EE) return coop_launch(k_resident<V, CL, EE, RES_BICG, false>, lds, a, st);
#define ALL8(V) ONE(V, 1, 1) ONE(V, 1, 2) ONE(V, 1, 4) ONE(V, 1, 8) ONE(V, 4, 1) ONE(V, 4, 2)
#define ALL16(V) ONE(V, 1, 1) ONE(V, 1, 2) ONE(V, 1, 4) ONE(V, 2, 1) ONE(V, 2, 2)
    switch (vk) {
    case VK_C32: ALL8(float2) break;
    case VK_C64: ALL16(double2) break;
    case VK_R32: ALL8(float) break;
    case VK_R64: ALL8(double) break;
    }
    return false;
}

}  // namespace tmi
