"""The ring decode kernel (QGEMM_KID_RING) at its edges: K-tile counts around
its stages of four (one K-tile up to more stages than the ring holds, partial
last stages), ragged M and N across the 16 / 32 / 64-row tiles, K split over
workgroups and not, both output types, batches.

Scale rows come in panels where their pitch and K allow it and dword by dword
otherwise; a padded pitch (MX) or the column-major A scales (fp32) force the
second form, which reads the same numbers in the same order, so both give the
same bits.  All outputs are checked against the GPU reference GEMM."""
import ctypes

import pytest
import torch

from helpers import assert_close_all

pytestmark = pytest.mark.gpu

KID_RING = 11


def _operands(qgemm, kind, m, n, k, g, gpu):
    x, w = (torch.randn((r, k), generator=g, device=gpu) for r in (m, n))
    if kind in ("bs", "bypass"):
        (a, sa), (braw, sb) = qgemm.quant_fp8_blockscale(x), qgemm.quant_fp8_blockscale(w, block="128x128")
        ref = qgemm.reference_gemm("bs_fp32", a, braw, sa, sb)
        b = qgemm.shuffle_b_kpanel(braw) if kind == "bs" else qgemm.ldsbypass_pack_b(braw)
    else:
        fn = qgemm.quant_mxfp8 if kind == "mxfp8" else qgemm.quant_mxfp4
        (a, sa), (b, sb) = fn(x), fn(w)
        ref = qgemm.reference_gemm("mxfp8" if kind == "mxfp8" else "mxfp4", a, b, sa, sb)
        if kind == "aiter":
            b, sa, sb = qgemm.shuffle_weight_16x16(b), qgemm.e8m0_shuffle(sa), qgemm.e8m0_shuffle(sb)
    return a, b, sa, sb, ref


def _stack(ops, i):
    return torch.stack([o[i].contiguous().view(torch.uint8) for o in ops]).contiguous()


def _run(qgemm, kind, ops, m, n, k, out_dtype, narrow, split, kid=KID_RING):
    """The id through the C ABI over a batch of operand sets; `narrow` pads
    the MX scale rows by 4 bytes / takes the fp32 A scales column-major."""
    dev, batch = ops[0][0].device, len(ops)
    a, b = _stack(ops, 0), _stack(ops, 1)
    sa = torch.stack([o[2].contiguous() for o in ops])
    sb = torch.stack([o[3].contiguous() for o in ops])
    c = torch.full((batch, m, n), float("nan"), dtype=out_dtype, device=dev)
    L, kb = qgemm.lib(), k if kind in ("mxfp8", "bs", "bypass") else k // 2
    if kind in ("bs", "bypass"):
        lb, stride_sfa = sb.shape[2], 1 if m > 1 else m
        if narrow:
            sa, stride_sfa = sa.transpose(1, 2).contiguous(), m
        common = (m, n, k, batch, k, 128, n, m * k, n * k, m * n, sa.data_ptr(), sb.data_ptr(), stride_sfa, lb,
                  sa[0].numel(), sb[0].numel())
        if kind == "bs":
            args = qgemm.Kargs(a.data_ptr(), b.data_ptr(), c.data_ptr(), *common)
            name = "gemm_a8w8_blockscale_bpreshuffle_kid"
        else:
            args = qgemm.LdsBypassKargs(a.data_ptr(), None, b.data_ptr(), c.data_ptr(), *common, b[0].numel())
            name = "gemm_a8w8_blockscale_ldsbypass_kid"
    else:
        sa, sb = sa.view(torch.uint8), sb.view(torch.uint8)
        if narrow:
            sa, sb = (torch.nn.functional.pad(s, (0, 4)) for s in (sa, sb))
        # (e8m0_shuffle: bytes per 32-row block)
        lsa, lsb = (k, k) if kind == "aiter" else (sa.shape[2], sb.shape[2])
        vals = (a.data_ptr(), b.data_ptr(), c.data_ptr(), m, n, k, batch, kb, kb, n, m * kb, n * kb, m * n,
                sa.data_ptr(), sb.data_ptr(), lsa, lsb, sa[0].numel(), sb[0].numel())
        args = qgemm.Mxfp4Kargs(*vals, 0) if kind == "aiter" else qgemm.Kargs(*vals)
        name = {"aiter": "gemm_a4w4_mxfp4_bpreshuffle_kid", "mxfp4": "gemm_a4w4_mxfp4_kid",
                "mxfp8": "gemm_a8w8_mxfp8_kid"}[kind]
    need = getattr(L, name + "_workspace_bytes")(ctypes.byref(args), kid) if split else 0
    ws = torch.full((max(need, 1),), 0xFF, dtype=torch.uint8, device=dev)    # any contents will do
    st = getattr(L, name)(ctypes.byref(args), 1 if out_dtype == torch.bfloat16 else 0, kid,
                          ws.data_ptr() if need else None, need,
                          ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert st == 0, f"{name}: error {st}"
    trace = qgemm.last_launch()
    torch.cuda.synchronize()
    return c, trace, need


# K-tiles: one, under / at / past one stage of four, past the ring (8 stages),
# many; 31 and 46: a partial last stage, also in a split's last slice
@pytest.mark.parametrize("ktiles,m,n", [(1, 1, 16), (2, 17, 112), (3, 33, 96), (4, 16, 64), (5, 64, 144), (9, 40, 272),
                                        (31, 64, 304), (32, 32, 1008), (46, 50, 528), (56, 64, 1536), (64, 5, 80),
                                        (128, 24, 2112), (13, 8, 16400)])
@pytest.mark.parametrize("kind", ["mxfp8", "mxfp4", "bs", "bypass", "aiter"])
def test_ring_edges(qgemm, gpu, kind, ktiles, m, n):
    k = ktiles * (256 if kind in ("mxfp4", "aiter") else 128)
    if kind != "aiter":
        n -= 3 if ktiles % 2 else 0    # (aiter: N % 16 == 0)
    g = torch.Generator(gpu).manual_seed(1000 * ktiles + m)
    op = _operands(qgemm, kind, m, n, k, g, gpu)
    for split in (False, True):
        first = {}
        for narrow in ((False,) if kind == "aiter" else (False, True)):
            for dtype in (torch.float32, torch.bfloat16):
                y, trace, need = _run(qgemm, kind, [op], m, n, k, dtype, narrow, split)
                assert trace.startswith("ring_gemm<") and ("splitk1>" in trace) == (need == 0), trace
                assert_close_all(op[4], y[0], f"{kind} {m}x{n}x{k} narrow {narrow} {dtype} ({trace})")
                assert torch.equal(first.setdefault(dtype, y), y), f"the scale forms differ ({trace})"


@pytest.mark.parametrize("kind", ["mxfp8", "mxfp4", "bs", "bypass", "aiter"])
def test_ring_batch(qgemm, gpu, kind):
    """Batch 3, K split: every batch entry's operands, planes and output."""
    m, n, k = 20, 144, 8192
    g = torch.Generator(gpu).manual_seed(7)
    ops = [_operands(qgemm, kind, m, n, k, g, gpu) for _ in range(3)]
    y, trace, need = _run(qgemm, kind, ops, m, n, k, torch.bfloat16, False, True)
    assert need > 0 and "splitk1>" not in trace, trace
    for i, op in enumerate(ops):
        assert_close_all(op[4], y[i], f"{kind} batch {i} ({trace})")


# AUTO at shapes inside the kernel's rules and one step outside, with and
# without the workspace (without: the ring only unsplit, else another kernel)
@pytest.mark.parametrize("kind,m,n,k,ring", [
    ("mxfp8", 8, 2112, 4096, True), ("mxfp8", 4, 2112, 4096, False), ("mxfp4", 1, 7168, 7168, True),
    ("mxfp4", 9, 7168, 7168, False), ("mxfp8", 16, 16384, 4096, True), ("mxfp8", 32, 1536, 7168, True),
    ("mxfp4", 64, 6144, 16384, True), ("mxfp8", 64, 12288, 4096, False), ("bs", 32, 4096, 7168, True),
    ("bs", 32, 1536, 7168, False), ("bypass", 33, 1536, 16384, True), ("bypass", 64, 7168, 2048, False),
    ("aiter", 33, 2112, 6144, True), ("aiter", 33, 1536, 6144, False), ("aiter", 32, 4096, 7168, False)])
def test_ring_auto(qgemm, gpu, kind, m, n, k, ring):
    g = torch.Generator(gpu).manual_seed(m + n)
    op = _operands(qgemm, kind, m, n, k, g, gpu)
    y, trace, need = _run(qgemm, kind, [op], m, n, k, torch.bfloat16, False, True, kid=0)
    if torch.cuda.get_device_properties(gpu).multi_processor_count == 256:
        assert trace.startswith("ring_gemm<") == ring, trace
    assert_close_all(op[4], y[0], f"{kind} {m}x{n}x{k} ({trace})")
    y, trace0, _ = _run(qgemm, kind, [op], m, n, k, torch.bfloat16, False, False, kid=0)
    assert not trace0.startswith("ring_gemm<") or trace0 == trace, (trace, trace0)
    assert_close_all(op[4], y[0], f"{kind} {m}x{n}x{k}, no workspace ({trace0})")
