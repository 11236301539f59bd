// The Q4_K GEMV family over half activations: the caller's half vectors are widened as the workgroup stages them and the
// results rounded where they are stored, in the one launch.  (Widening into f32 staging, the f32 kernel and a narrowing
// launch were three, at 3.5 us a launch from a stream.)  Arithmetic between the two is the f32 kernel's.  Built for the
// schedules the defaults choose (1 or 2 rows per wave, 4 or 8 waves, byte converts or three digit planes); a handle
// bound to another one goes through the conversions (half_boundary.hip).
// One decode layer of eight operators on half buffers, launched one by one (hidden 2048, ffn 8192, 700 cached rows):
// 88 us with the conversions, 39 us without.
#include "q4k_gemv.hpp"

namespace ksh {

bool q4k_gemv_half_built(const Q4kGeom &G) { return G.R <= 2 && (G.NW == 4 || G.NW == 8) && G.var != kXI2; }

namespace {
template <int NM, int XF>
int launch_half_rn(const Q4kGeom &G, const MatvecParams &p, int total_waves, hipStream_t st)
{
    if (G.R == 1) return G.NW == 4 ? launch_inst<1, 4, NM, XF, true>(G.half, p, total_waves, st) : launch_inst<1, 8, NM, XF, true>(G.half, p, total_waves, st);
    return G.NW == 4 ? launch_inst<2, 4, NM, XF, true>(G.half, p, total_waves, st) : launch_inst<2, 8, NM, XF, true>(G.half, p, total_waves, st);
}
}  // namespace

int launch_q4k_gemv_half(const Q4kGeom &G, int nm, const MatvecParams &p, int total_waves, hipStream_t st)
{
    if (nm == 2) return G.var == kXI8 ? launch_half_rn<2, kXI8>(G, p, total_waves, st) : launch_half_rn<2, kXF32>(G, p, total_waves, st);
    return G.var == kXI8 ? launch_half_rn<1, kXI8>(G, p, total_waves, st) : launch_half_rn<1, kXF32>(G, p, total_waves, st);
}

}  // namespace ksh
