// Launch helpers of the ring kernel, shared by its instantiation units.
#pragma once
#include "launch.hpp"
#include "ring_gemm.hpp"

namespace qg {
namespace ring {

template <int FMT, ScaleKind SK, BLay BL, int MB, int NB>
hipError_t go(const RingArgs& a, bool panel, int batch, hipStream_t s) {
    const dim3 grid(a.n_tiles * a.splitk, batch);
    if (panel) ring_gemm_kernel<FMT, SK, BL, MB, NB, true><<<grid, 512, 0, s>>>(a);
    else if constexpr (SK != ScaleKind::MXS) ring_gemm_kernel<FMT, SK, BL, MB, NB, false><<<grid, 512, 0, s>>>(a);
    else return hipErrorInvalidValue;
    trace_launch("ring_gemm<%s,%s,%s,mb%d,nb%d,%s,splitk%d>", FMT == kFmtFp4 ? "fp4" : "fp8", scale_name(SK),
                 SK == ScaleKind::MXS ? "W16" : layout_name(BL), MB, NB, a.bf16 ? "bf16" : "fp32", a.splitk);
    return hipGetLastError();
}

// tiles of mb x nb 16-row blocks, (mb, nb) in {1, 2} x {1, 2, 4} or 4 x {1, 2}
template <int FMT, ScaleKind SK, BLay BL>
hipError_t launch(const RingArgs& a, int mb, int nb, bool panel, int batch, hipStream_t s) {
#define QG_RING(MBV, NBV) \
    if (mb == MBV && nb == NBV) return go<FMT, SK, BL, MBV, NBV>(a, panel, batch, s);
    QG_RING(1, 1) QG_RING(1, 2) QG_RING(1, 4) QG_RING(2, 1) QG_RING(2, 2) QG_RING(2, 4) QG_RING(4, 1) QG_RING(4, 2)
#undef QG_RING
    return hipErrorInvalidValue;
}

}  // namespace ring
}  // namespace qg
