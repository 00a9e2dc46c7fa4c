// Ring kernel on MXFP8 / MXFP4 with row-major B.
#include "ring_launch.hpp"

namespace qg {

hipError_t launch_ring_mx(const RingArgs& a, bool fp4, int mb, int nb, bool panel, int batch, hipStream_t s) {
    return fp4 ? ring::launch<kFmtFp4, ScaleKind::MX, BLay::RAW>(a, mb, nb, panel, batch, s)
               : ring::launch<kFmtFp8, ScaleKind::MX, BLay::RAW>(a, mb, nb, panel, batch, s);
}

}  // namespace qg
