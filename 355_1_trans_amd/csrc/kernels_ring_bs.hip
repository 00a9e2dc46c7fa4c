// Ring kernel on fp8 with fp32 block scales (B' or B'') and on MXFP4 in
// aiter's formats (W16 B has B'' bytes, e8m0_shuffle scales).
#include "ring_launch.hpp"

namespace qg {

hipError_t launch_ring_bs(const RingArgs& a, bool frag, int mb, int nb, bool panel, int batch, hipStream_t s) {
    return frag ? ring::launch<kFmtFp8, ScaleKind::BSF32, BLay::FRAG>(a, mb, nb, panel, batch, s)
                : ring::launch<kFmtFp8, ScaleKind::BSF32, BLay::KPANEL>(a, mb, nb, panel, batch, s);
}

hipError_t launch_ring_mx4s(const RingArgs& a, int mb, int nb, int batch, hipStream_t s) {
    return ring::launch<kFmtFp4, ScaleKind::MXS, BLay::FRAG>(a, mb, nb, true, batch, s);
}

}  // namespace qg
