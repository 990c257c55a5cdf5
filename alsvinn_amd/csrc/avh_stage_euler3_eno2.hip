// Stage kernels for euler3 on three active axes, eno2 reconstruction.
#include "avh_stage_inst.hpp"
namespace avh {
Launchers get_launchers_euler3_3d_eno2(int flux) {
    if (flux == 1) return launchers_of<EulerEq<3>, RECON_ENO2, HLLFlux, 3>();
    if (flux == 2) return launchers_of<EulerEq<3>, RECON_ENO2, HLL3Flux, 3>();
    return Launchers();
}
}  // namespace avh
