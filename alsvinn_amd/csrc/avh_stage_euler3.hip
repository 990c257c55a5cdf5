// Stage kernels for euler3 (hll and hll3 fluxes).
#include "avh_stage_inst.hpp"
namespace avh {
Launchers get_launchers_euler3(int recon, int flux, int dim) {
    if (dim == 3) {
        switch (recon) {
        case RECON_NONE: return get_launchers_euler3_3d_none(flux);
        case RECON_WENO2: return get_launchers_euler3_3d_weno2(flux);
        case RECON_ENO2: return get_launchers_euler3_3d_eno2(flux);
        case RECON_ENO3: return get_launchers_euler3_3d_eno3(flux);
        }
        return Launchers();
    }
    if (flux == 1) return pick_dim<EulerEq<3>, HLLFlux, 2>(recon, dim);
    if (flux == 2) return pick_dim<EulerEq<3>, HLL3Flux, 2>(recon, dim);
    return Launchers();
}
}  // namespace avh
