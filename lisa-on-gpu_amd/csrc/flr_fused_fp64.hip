// flr_fused_fp64.hip -- fused projection + TDI kernels with FP64 storage (complex128 in,
// double out): exact stencils (bitwise the unfused path) or the fast form, 512-sample tiles.
#include "flr_fused.hpp"

namespace flr {

hipError_t launch_fused_fp64(const ProjConfig &pc, const TdiConfig &tc,
                             const Batch<FusedSource> &b, const OrbitView &orb,
                             const LagrangeView &lg, bool exact, int grid_per_cu,
                             const StockTdi &st, hipStream_t stream)
{
    // the projection's windows reach lowest: the TDI window's start less the projection's halo
    const int64_t lowest = (int64_t)b.min_start - tc.halo_lo - pc.halo_lo;
    return by_form(stencil_form(exact, lowest, lg.h), [&](auto form) {
        return launch_fused_variant<decltype(form)::value, double2, double, 2>(
            pc, tc, b, orb, lg, st, grid_per_cu, stream);
    });
}

}  // namespace flr
