"""The 128 x 128 kernel's pipeline at its edges: the ring of four stages (one
workgroup per CU) and the two-stage form (more workgroups than CUs), from one
K-tile up, with the scales in 4-K-tile panels and K-tile by K-tile.

A scale pitch that is not a multiple of 16 bytes keeps the panels off, so the
same problem with padded scale rows has to give the same bits; both are
checked against the GPU reference GEMM over all outputs."""
import ctypes

import pytest
import torch

from helpers import assert_close_all

pytestmark = pytest.mark.gpu

KID_MID = 2


def _padded(s, extra):
    wide = torch.zeros((s.shape[0], s.shape[1] + extra), dtype=s.dtype, device=s.device)
    wide[:, :s.shape[1]] = s
    return wide


def _run(qgemm, kind, a, b, sa, sb, m, n, k, out_dtype, extra, split):
    """kid MID through the C ABI, scale rows padded by `extra` elements."""
    sa, sb = _padded(sa, extra), _padded(sb, extra)
    c = torch.full((m, n), float("nan"), dtype=out_dtype, device=a.device)
    la, lb = sa.shape[1], sb.shape[1]
    L, fp4 = qgemm.lib(), kind == "mxfp4"
    kb = k // 2 if fp4 else k
    if kind == "bypass":
        args = qgemm.LdsBypassKargs(a.data_ptr(), None, b.data_ptr(), c.data_ptr(), m, n, k, 1, k, 128, n, m * k, n * k,
                                    m * n, sa.data_ptr(), sb.data_ptr(), 1, lb, m * la, sb.numel(), b.numel())
        name = "gemm_a8w8_blockscale_ldsbypass_kid"
    elif kind == "bs":
        args = qgemm.Kargs(a.data_ptr(), b.data_ptr(), c.data_ptr(), m, n, k, 1, k, 128, n, m * k, n * k, m * n,
                           sa.data_ptr(), sb.data_ptr(), 1, lb, m * la, sb.numel())
        name = "gemm_a8w8_blockscale_bpreshuffle_kid"
    else:
        args = qgemm.Kargs(a.data_ptr(), b.data_ptr(), c.data_ptr(), m, n, k, 1, kb, kb, n, m * kb, n * kb, m * n,
                           sa.data_ptr(), sb.data_ptr(), la, lb, sa.numel(), sb.numel())
        name = "gemm_a4w4_mxfp4_kid" if fp4 else "gemm_a8w8_mxfp8_kid"
    need = getattr(L, name + "_workspace_bytes")(ctypes.byref(args), KID_MID) if split else 0
    ws = torch.zeros(max(need, 1), dtype=torch.uint8, device=a.device)
    st = getattr(L, name)(ctypes.byref(args), 1 if out_dtype == torch.bfloat16 else 0, KID_MID,
                          ws.data_ptr() if need else None, need,
                          ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert st == 0, f"{name}: error {st}"
    trace = qgemm.last_launch()
    assert trace.startswith("mid_gemm<"), trace
    torch.cuda.synchronize()
    return c, trace


# K-tiles: below, at and past the ring's four stages and a panel, an odd
# count (no panels), and 40 and 44 (split: in slices of eight, and of nine,
# which start inside a panel)
@pytest.mark.parametrize("ktiles,m,n,split", [(1, 130, 70, False), (2, 65, 130, False), (3, 70, 200, False),
                                              (4, 129, 129, False), (5, 200, 100, False), (8, 100, 300, False),
                                              (12, 70, 70, False), (40, 150, 260, True), (44, 300, 1500, True),
                                              (4, 2100, 2180, False), (8, 2100, 2180, False), (9, 2100, 2180, False)])
@pytest.mark.parametrize("kind", ["mxfp8", "mxfp4", "bs", "bypass"])
def test_mid_pipeline_edges(qgemm, gpu, kind, ktiles, m, n, split):
    k = ktiles * (256 if kind == "mxfp4" else 128)
    g = torch.Generator(gpu).manual_seed(1000 * ktiles + m)
    x, w = (torch.randn((r, k), generator=g, device=gpu) for r in (m, n))
    if kind in ("bs", "bypass"):
        (a, sa), (braw, sb) = qgemm.quant_fp8_blockscale(x), qgemm.quant_fp8_blockscale(w, block="128x128")
        ref = qgemm.reference_gemm("bs_fp32", a, braw, sa, sb)
        b = qgemm.shuffle_b_kpanel(braw) if kind == "bs" else qgemm.ldsbypass_pack_b(braw)
    else:
        fn = qgemm.quant_mxfp4 if kind == "mxfp4" else qgemm.quant_mxfp8
        (a, sa), (b, sb) = fn(x), fn(w)
        ref = qgemm.reference_gemm(kind, a, b, sa, sb)
    outs = []
    # fp32 scales: the entries take dense row-major A scales only (pitch K/128), so only MX pads its rows
    for extra in ((0, 4) if kind.startswith("mx") else (0,)):
        for dtype in (torch.float32, torch.bfloat16):
            y, trace = _run(qgemm, kind, a, b, sa, sb, m, n, k, dtype, extra, split)
            assert ("st2" in trace) == (m > 2000) and ("splitk1>" in trace) == (not split), trace
            assert_close_all(ref, y, f"{kind} {m}x{n}x{k} +{extra} {dtype} ({trace})")
            outs.append(y)
    for y in outs[2:]:
        assert torch.equal(y, outs[0] if y.dtype == torch.float32 else outs[1])
