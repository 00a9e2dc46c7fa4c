"""C ABI of libqgemm.so without a GPU: every symbol declared in
include/qgemm.h is exported, argument validation rejects bad calls before
any device call, the host layout helpers equal their numpy forms, and the
split-K workspace queries follow the documented contract."""
import ctypes
import re
from pathlib import Path

import numpy as np
import pytest
import torch

import oracle as O

ROOT = Path(__file__).resolve().parent.parent
HIP_INVALID_VALUE = 1


def _declared_functions():
    text = (ROOT / "include" / "qgemm.h").read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"^[A-Za-z_][\w \*]*?\b(\w+)\s*\(", text, flags=re.M)))


def test_library_exports_every_declared_symbol(qgemm):
    names = _declared_functions()
    assert len(names) >= 18, names
    L = ctypes.CDLL(str(qgemm.LIB_PATH))
    missing = [n for n in names if not hasattr(L, n)]
    assert not missing, missing
    assert set(names) <= set(qgemm.EXPORTS), set(names) - set(qgemm.EXPORTS)
    assert qgemm.lib().qgemm_version().startswith(b"qgemm gfx950")


def _kargs(qgemm, m=32, n=256, k=512, **kw):
    buf = [ctypes.create_string_buffer(1 << 16) for _ in range(5)]
    base = dict(ptr_a=ctypes.addressof(buf[0]), ptr_b=ctypes.addressof(buf[1]), ptr_c=ctypes.addressof(buf[2]),
                m=m, n=n, k=k, batch=1, stride_a=k, stride_b=k, stride_c=n, stride_a_batch=m * k,
                stride_b_batch=n * k, stride_c_batch=m * n, ptr_sfa=ctypes.addressof(buf[3]),
                ptr_sfb=ctypes.addressof(buf[4]), stride_sfa=k // 32, stride_sfb=k // 32,
                stride_sfa_batch=m * (k // 32), stride_sfb_batch=n * (k // 32))
    base.update(kw)
    a = qgemm.Kargs(**base)
    a._keep = buf
    return a


@pytest.mark.parametrize("change", [
    dict(ptr_a=None), dict(ptr_c=None), dict(k=100), dict(m=0), dict(n=-1), dict(batch=0),
    dict(stride_a=256), dict(stride_c=100), dict(stride_sfa=8), dict(stride_b=520),
])
def test_mxfp8_rejects_bad_arguments(qgemm, change):
    a = _kargs(qgemm, **change)
    assert qgemm.lib().gemm_a8w8_mxfp8(ctypes.byref(a), 1, None, 0, None) == HIP_INVALID_VALUE


def test_rejects_bad_flags_null_args_and_overlap(qgemm):
    L = qgemm.lib()
    a = _kargs(qgemm)
    assert L.gemm_a8w8_mxfp8(None, 1, None, 0, None) == HIP_INVALID_VALUE
    assert L.gemm_a8w8_mxfp8(ctypes.byref(a), 2, None, 0, None) == HIP_INVALID_VALUE
    a.ptr_c = a.ptr_a + 64                                   # C overlapping A
    assert L.gemm_a8w8_mxfp8(ctypes.byref(a), 1, None, 0, None) == HIP_INVALID_VALUE
    a4 = _kargs(qgemm, k=384, stride_a=192, stride_b=192)    # K % 256 != 0 for fp4
    assert L.gemm_a4w4_mxfp4(ctypes.byref(a4), 1, None, 0, None) == HIP_INVALID_VALUE


def test_blockscale_e8m0_contract(qgemm):
    """SNAP launcher: M, N multiples of 256, dense strides, tiles in {0, 1}."""
    L = qgemm.lib()
    ok = dict(m=256, n=256, k=256, stride_a=256, stride_b=256, stride_c=256, stride_a_batch=65536,
              stride_b_batch=65536, stride_c_batch=65536, stride_sfa=256, stride_sfb=2, stride_sfa_batch=512,
              stride_sfb_batch=4)
    for bad in (dict(m=128), dict(n=384, stride_c=384), dict(stride_sfa=128), dict(k=200)):
        a = _kargs(qgemm, **{**ok, **bad})
        assert L.launch_blockscale_bpreshuffle(ctypes.byref(a), 1, 0, None) == HIP_INVALID_VALUE
    a = _kargs(qgemm, **ok)
    assert L.launch_blockscale_bpreshuffle(ctypes.byref(a), 1, 2, None) == HIP_INVALID_VALUE
    assert L.launch_blockscale_bpreshuffle(ctypes.byref(a), 3, 0, None) == HIP_INVALID_VALUE


def test_bpreshuffle_requires_kpanel_stride(qgemm):
    a = _kargs(qgemm, stride_b=512, stride_sfa=32, stride_sfb=4)
    assert qgemm.lib().gemm_a8w8_blockscale_bpreshuffle(ctypes.byref(a), 1, None, 0, None) == HIP_INVALID_VALUE


def test_workspace_queries(qgemm):
    L = qgemm.lib()
    # large M runs the 256 x 256 tile kernel: 2 KB of counters, then both
    # operands' E8M0 scales copied panel-major ((M + N) * K/32 bytes, each
    # operand's share rounded up to 256) -- only when K % 512 == 0
    assert L.gemm_a8w8_mxfp8_workspace_bytes(ctypes.byref(_kargs(qgemm, m=8192, n=8192, k=8192))) == \
        2048 + 2 * 8192 * 256
    assert L.gemm_a4w4_mxfp4_workspace_bytes(ctypes.byref(_kargs(qgemm, m=1000, n=8192, k=4096))) == \
        2048 + 1000 * 128 + 8192 * 128
    assert L.gemm_a8w8_mxfp8_workspace_bytes(ctypes.byref(_kargs(qgemm, m=8192, n=8192, k=8320))) == 0
    # decode (M <= 64) with too few N tiles for the skinny kernel: the decode
    # kernel splits K -- 2 KB of counters + splitk * M * N fp32 partials
    for m, n, k in [(1, 1536, 7168), (32, 1536, 7168), (4, 1000, 7168), (64, 1536, 7168)]:
        a = _kargs(qgemm, m=m, n=n, k=k)
        ws = L.gemm_a8w8_mxfp8_workspace_bytes(ctypes.byref(a))
        assert ws >= 2048 + 2 * m * n * 4 and (ws - 2048) % (m * n * 4) == 0, (m, n, k, ws)
    # enough N tiles for the skinny kernel -> no split
    assert L.gemm_a8w8_mxfp8_workspace_bytes(ctypes.byref(_kargs(qgemm, m=1, n=7168, k=16384))) == 0
    # M > 64 with few 256 x 256 tiles: the 128 x 128 kernel, 64 tiles; K of
    # 32 K-tiles split in four (8-K-tile slices while one workgroup per CU
    # holds them: 256 / 64 = 4)
    assert L.gemm_a8w8_mxfp8_workspace_bytes(ctypes.byref(_kargs(qgemm, m=128, n=8192, k=4096))) == \
        2048 + 4 * 128 * 8192 * 4
    assert L.gemm_a8w8_mxfp8_workspace_bytes(ctypes.byref(_kargs(qgemm, m=128, n=8192, k=1024))) == 0
    # 56 tiles of 128 x 128 at N = 7168: split capped at kCUs / tiles = 4
    # (one workgroup per CU), not 512 / 56 = 9; MXFP4 K-tiles are 256 deep
    assert L.gemm_a8w8_mxfp8_workspace_bytes(ctypes.byref(_kargs(qgemm, m=128, n=7168, k=16384))) == \
        2048 + 4 * 128 * 7168 * 4
    assert L.gemm_a4w4_mxfp4_workspace_bytes(ctypes.byref(_kargs(qgemm, m=128, n=7168, k=16384))) == \
        2048 + 4 * 128 * 7168 * 4
    # M > 256 on 96 256 x 256 tiles: the four-wave kernel's K split in two
    # (MXFP8 56 K-tiles, MXFP4 64), whole scale panels per slice: counters,
    # both operands' panel copies, then two fp32 partial planes
    assert L.gemm_a8w8_mxfp8_workspace_bytes(ctypes.byref(_kargs(qgemm, m=512, n=12288, k=7168))) == \
        2048 + 512 * 224 + 12288 * 224 + 2 * 512 * 12288 * 4
    assert L.gemm_a4w4_mxfp4_workspace_bytes(ctypes.byref(_kargs(qgemm, m=512, n=12288, k=16384))) == \
        2048 + 512 * 512 + 12288 * 512 + 2 * 512 * 12288 * 4
    # 136 tiles (> kCUs / 2): two workgroups per CU, 56 K-tiles / 16 -> 3 slices
    assert L.gemm_a8w8_mxfp8_workspace_bytes(ctypes.byref(_kargs(qgemm, m=1024, n=2112, k=7168))) == \
        2048 + 3 * 1024 * 2112 * 4
    # too few K-tiles to split (8 per slice at least)
    assert L.gemm_a8w8_mxfp8_workspace_bytes(ctypes.byref(_kargs(qgemm, m=1, n=1536, k=1024))) == 0
    assert L.gemm_a8w8_mxfp8_workspace_bytes(None) == 0
    # fp4 K-tiles hold 256 elements: K = 16384 gives 64 of them, enough for 16-tile slices
    assert L.gemm_a4w4_mxfp4_workspace_bytes(ctypes.byref(_kargs(qgemm, m=1, n=1536, k=16384))) > 0


# ----------------------------------------------------------------- host layout helpers
def test_product_layout_helpers_match_numpy(qgemm):
    L = qgemm.lib()
    rng = np.random.default_rng(21)
    b = rng.integers(0, 256, (48, 384), dtype=np.uint8)
    out = np.empty_like(b)
    assert L.qgemm_shuffle_b_kpanel(b.ctypes.data, out.ctypes.data, 48, 384) == 0
    assert np.array_equal(out.reshape(3, 48, 128), b.reshape(48, 3, 128).transpose(1, 0, 2))
    assert L.qgemm_shuffle_weight_16x16(b.ctypes.data, out.ctypes.data, 48, 384) == 0
    assert np.array_equal(out, b.reshape(3, 16, 24, 16).transpose(0, 2, 1, 3).reshape(48, 384))
    e = rng.integers(0, 255, (64, 24), dtype=np.uint8)
    nbytes = L.qgemm_e8m0_shuffle_bytes(64, 24)
    eo = np.empty(nbytes, np.uint8)
    assert L.qgemm_e8m0_shuffle(e.ctypes.data, eo.ctypes.data, 64, 24) == 0
    assert np.array_equal(eo, e.reshape(2, 2, 16, 3, 2, 4).transpose(0, 3, 5, 2, 4, 1).reshape(-1))
    assert L.qgemm_shuffle_b_kpanel(b.ctypes.data, out.ctypes.data, 48, 100) == HIP_INVALID_VALUE


@pytest.mark.parametrize("n,k", [(48, 256), (37, 384), (16, 128)])
def test_ldsbypass_host_pack_matches_permutation(qgemm, n, k):
    """B'' = [ceil(N/16)][K/128][h][lane = 16q + r][16] with chunk q + 4h of row 16nb + r."""
    b = np.random.default_rng(n * k).integers(0, 256, (n, k), dtype=np.uint8)
    got = qgemm.ldsbypass_pack_b(torch.from_numpy(b)).numpy()
    nb = (n + 15) // 16
    pad = np.zeros((nb * 16, k), np.uint8)
    pad[:n] = b
    ref = pad.reshape(nb, 16, k // 128, 2, 4, 16).transpose(0, 2, 3, 4, 1, 5).reshape(-1)
    assert got.size == qgemm.ldsbypass_b_bytes(n, k) == nb * 16 * k
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("n,k", [(16, 128), (48, 512), (256, 1024)])
def test_ldsbypass_b_is_shuffle_weight_16x16(qgemm, n, k):
    """For N % 16 == 0 the LDS-bypass B'' is byte for byte aiter's
    shuffle_weight(16,16) of B (the 16x16x128 fragment order): aiter-shuffled
    weights feed gemm_a8w8_blockscale_ldsbypass as they are."""
    b = np.random.default_rng(n + k).integers(0, 256, (n, k), dtype=np.uint8)
    assert np.array_equal(qgemm.ldsbypass_pack_b(torch.from_numpy(b)).numpy().reshape(-1),
                          O.shuffle_weight_16x16(b).reshape(-1))


def test_python_layout_helpers(qgemm):
    b = torch.from_numpy(np.random.default_rng(22).integers(0, 256, (32, 256), dtype=np.uint8))
    assert np.array_equal(qgemm.shuffle_b_kpanel(b).numpy(), O.shuffle_b_kpanel(b.numpy()))
    assert np.array_equal(qgemm.shuffle_weight_16x16(b).numpy(), O.shuffle_weight_16x16(b.numpy()))


def test_no_cpu_fallback(qgemm):
    a = torch.zeros(16, 128, dtype=torch.uint8).view(torch.float8_e4m3fn)
    s = torch.zeros(16, 4, dtype=torch.uint8)
    with pytest.raises(ValueError, match="GPU"):
        qgemm.gemm_a8w8_mxfp8(a, a, s, s)


# ----------------------------------------------------------------- workspace rule
def _far_kargs(qgemm, m, n, k, fp4=False, out_bytes=2):
    """Kargs whose operands sit at widely separated, 256-byte aligned fake
    addresses (never dereferenced: every call below is rejected before any
    device work, or, on a machine without a GPU, fails the device check)."""
    kb = k // 2 if fp4 else k
    base = [(1 << 44) + (i << 38) for i in range(5)]
    return qgemm.Kargs(base[0], base[1], base[2], m, n, k, 1, kb, kb, n, m * kb, n * kb, m * n,
                       base[3], base[4], k // 32, k // 32, m * (k // 32), n * (k // 32))


# one shape per route: wide (panel copy), 128 x 128 split-K, decode split-K,
# row-streaming split-K
WS_ROUTES = [("gemm_a8w8_mxfp8", 8192, 8192, 8192, False), ("gemm_a8w8_mxfp8", 128, 7168, 16384, False),
             ("gemm_a8w8_mxfp8", 32, 1536, 7168, False), ("gemm_a8w8_mxfp8", 4, 7168, 32768, False),
             ("gemm_a4w4_mxfp4", 8192, 8192, 8192, True), ("gemm_a4w4_mxfp4", 128, 7168, 16384, True),
             ("gemm_a4w4_mxfp4", 4, 7168, 65536, True)]


@pytest.mark.parametrize("name,m,n,k,fp4", WS_ROUTES)
def test_workspace_rule_is_uniform(qgemm, name, m, n, k, fp4):
    """Every route applies one rule before launching: a non-NULL workspace
    smaller than the query, misaligned, or overlapping C or an input is
    rejected with hipErrorInvalidValue."""
    L = qgemm.lib()
    a = _far_kargs(qgemm, m, n, k, fp4)
    need = getattr(L, name + "_workspace_bytes")(ctypes.byref(a))
    assert need > 0, (name, m, n, k)
    ws = (1 << 44) + (7 << 38)
    fn = getattr(L, name)
    assert fn(ctypes.byref(a), 1, ws, need - 1, None) == HIP_INVALID_VALUE         # too small
    assert fn(ctypes.byref(a), 1, ws + 16, need, None) == HIP_INVALID_VALUE        # not 256-byte aligned
    assert fn(ctypes.byref(a), 1, a.ptr_c, need, None) == HIP_INVALID_VALUE        # overlaps C
    assert fn(ctypes.byref(a), 1, a.ptr_b, need, None) == HIP_INVALID_VALUE        # overlaps B
    if not torch.cuda.is_available():
        # a conforming workspace passes validation and stops at the device check
        assert fn(ctypes.byref(a), 1, ws, need, None) != HIP_INVALID_VALUE


def test_blockscale_workspace_rule(qgemm):
    L = qgemm.lib()
    m, n, k = 32, 1536, 7168
    base = [(1 << 44) + (i << 38) for i in range(5)]
    a = qgemm.Kargs(base[0], base[1], base[2], m, n, k, 1, k, 128, n, m * k, n * k, m * n, base[3], base[4],
                    1, k // 128, m * (k // 128), (n // 128) * (k // 128))
    need = L.gemm_a8w8_blockscale_bpreshuffle_workspace_bytes(ctypes.byref(a))
    assert need > 0
    ws = (1 << 44) + (7 << 38)
    assert L.gemm_a8w8_blockscale_bpreshuffle(ctypes.byref(a), 1, ws, need - 4, None) == HIP_INVALID_VALUE
    assert L.gemm_a8w8_blockscale_bpreshuffle(ctypes.byref(a), 1, a.ptr_a, need, None) == HIP_INVALID_VALUE


def test_misaligned_output_rejected(qgemm):
    """C must be aligned to its element size; wider vector stores are chosen
    from the actual alignment of ptr_c, the row pitch and the batch stride."""
    L = qgemm.lib()
    a = _far_kargs(qgemm, 32, 256, 512)
    a.ptr_c += 1
    assert L.gemm_a8w8_mxfp8(ctypes.byref(a), 1, None, 0, None) == HIP_INVALID_VALUE
    a.ptr_c += 1                                            # 2-byte aligned: fine for bf16, not fp32
    assert L.gemm_a8w8_mxfp8(ctypes.byref(a), 0, None, 0, None) == HIP_INVALID_VALUE
    if not torch.cuda.is_available():
        assert L.gemm_a8w8_mxfp8(ctypes.byref(a), 1, None, 0, None) != HIP_INVALID_VALUE


def test_last_launch_empty_after_rejection(qgemm):
    L = qgemm.lib()
    assert L.gemm_a8w8_mxfp8(None, 1, None, 0, None) == HIP_INVALID_VALUE
    assert qgemm.last_launch() == ""


def test_e8m0_adapter_rejects_before_launch(qgemm):
    f = qgemm.blockscale_bpreshuffle.gemm_a8w8_blockscale_bpreshuffle
    x = torch.zeros(256, 256, dtype=torch.uint8)
    with pytest.raises(ValueError, match="2-D"):
        f(x[0], x, x, x)
    with pytest.raises(ValueError, match="GPU"):
        f(x.view(torch.float8_e4m3fn), x, x[:, :2], x[:2, :2])


# ----------------------------------------------------------------- quantizer entries
def test_quantizers_reject_bad_arguments(qgemm):
    """Bad sources, pitches, alignments, scale layouts and overlaps return
    hipErrorInvalidValue before any device work (fake, separated addresses)."""
    L = qgemm.lib()
    x, q, s = 1 << 44, (1 << 44) + (1 << 38), (1 << 44) + (2 << 38)
    m, k = 64, 1024
    act = L.qgemm_quant_fp8_blockscale_act
    assert act(None, 0, m, k, k, q, k, s, k // 128, 1, None) == HIP_INVALID_VALUE
    assert act(x, 2, m, k, k, q, k, s, k // 128, 1, None) == HIP_INVALID_VALUE          # dtype code
    assert act(x, 0, m, 1000, 1000, q, 1000, s, 8, 1, None) == HIP_INVALID_VALUE      # K % 128
    assert act(x, 0, m, k, k - 4, q, k, s, k // 128, 1, None) == HIP_INVALID_VALUE     # pitch < K
    assert act(x + 4, 0, m, k, k, q, k, s, k // 128, 1, None) == HIP_INVALID_VALUE     # fp32 source not 16-B aligned
    assert act(x, 0, m, k, k, q, k, s, 2, 1, None) == HIP_INVALID_VALUE                # scale rows overlap
    assert act(x, 0, m, k, k, q, k, s, 1, m - 1, None) == HIP_INVALID_VALUE            # column-major pitch < M
    assert act(x, 0, m, k, k, x + 64, k, s, k // 128, 1, None) == HIP_INVALID_VALUE    # q overlaps x
    mx = L.qgemm_quant_mxfp4
    assert mx(x, 0, m, 100, 100, q, 50, s, 3, 0, None) == HIP_INVALID_VALUE             # K % 32
    assert mx(x, 0, m, 96, 96, q, 47, s, 3, 0, None) == HIP_INVALID_VALUE               # q pitch < K/2
    assert mx(x, 0, m, 96, 96, q, 48, s, 2, 0, None) == HIP_INVALID_VALUE               # scale pitch < K/32
    assert mx(x, 0, m, 96, 96, q, 48, s, 3, 2, None) == HIP_INVALID_VALUE               # shuffle flag
    lay = L.qgemm_shuffle_weight_16x16_device
    assert lay(x, q, 40, 256, 256, None) == HIP_INVALID_VALUE                            # N % 16
    assert L.qgemm_shuffle_b_kpanel_device(x, q, 40, 200, 208, None) == HIP_INVALID_VALUE   # K % 128
    assert L.qgemm_shuffle_b_kpanel_device(x, x + 256, 40, 256, 256, None) == HIP_INVALID_VALUE  # overlap


def test_extreme_dimensions_do_not_overflow(qgemm):
    """Dimensions near INT_MAX through the workspace queries, the entries and
    the host layout helpers (found with a host AddressSanitizer /
    UndefinedBehaviorSanitizer build: rounding-up helpers overflowed int):
    queries stay defined, entries reject, sizes are computed in 64 bits."""
    L = qgemm.lib()
    big = (1 << 31) - 1
    for m, n in [(1, big), (big, 1), (64, big - 15), (big, big)]:
        a = _kargs(qgemm, m=m, n=n)
        for kid in range(-1, 9):
            L.gemm_a8w8_mxfp8_kid_workspace_bytes(ctypes.byref(a), kid)
            L.gemm_a4w4_mxfp4_kid_workspace_bytes(ctypes.byref(a), kid)
            L.gemm_a8w8_blockscale_bpreshuffle_kid_workspace_bytes(ctypes.byref(a), kid)
        assert L.gemm_a8w8_mxfp8(ctypes.byref(a), 1, None, 0, None) == HIP_INVALID_VALUE
        assert L.gemm_a8w8_blockscale_bpreshuffle(ctypes.byref(a), 1, None, 0, None) == HIP_INVALID_VALUE
    # e8m0_shuffle image: rows to 32, groups to 8, in 64 bits
    assert L.qgemm_e8m0_shuffle_bytes(big, 8) == (big + 31) // 32 * 32 * 8
    assert L.qgemm_e8m0_shuffle_bytes(32, big) == 32 * ((big + 7) // 8 * 8)
    assert L.qgemm_ldsbypass_b_bytes(big, 128) == (big + 15) // 16 * 16 * 128


def test_mxfp8_opus_rejects_2d_out_for_batches(qgemm):
    """A 2-D ``out`` holds one batch entry: with batch > 1 the kernel would
    write batch * M * N values into it, so the wrapper refuses it before any
    device work (CPU tensors: the shape check comes first)."""
    from importlib import import_module
    opus = import_module("355_1_trans_amd.opus")
    b, m, n, k = 2, 16, 32, 128
    A = torch.zeros(b, m, k, dtype=torch.uint8).view(torch.float8_e4m3fn)
    B = torch.zeros(b, n, k, dtype=torch.uint8).view(torch.float8_e4m3fn)
    sa, sb = torch.zeros(b, m, k // 32, dtype=torch.uint8), torch.zeros(b, n, k // 32, dtype=torch.uint8)
    with pytest.raises(ValueError, match="only when batch is 1"):
        opus.gemm_a8w8_mxfp8_opus(A, B, sa, sb, out=torch.empty(m, n, dtype=torch.float32))
    # batch 1 may pass [M, N]; it gets as far as the device check
    with pytest.raises(ValueError, match="GPU"):
        opus.gemm_a8w8_mxfp8_opus(A[0], B[0], sa[0], sb[0], out=torch.empty(m, n, dtype=torch.float32))


def test_noalloc_plans_as_the_query(qgemm):
    """gemm_a4w4_mxfp4_noalloc runs exactly the plan gemm_a4w4_mxfp4 runs with
    the queried workspace: it is refused wherever that query exceeds the
    static scratch -- here a four-wave K split whose partial planes (55 MB)
    do not fit 32 MiB -- instead of silently planning another kernel; a split
    whose planes fit is accepted (stops at the device check without a GPU)."""
    L = qgemm.lib()
    cap = L.gemm_a4w4_mxfp4_noalloc_max_workspace_bytes()
    big = _far_kargs(qgemm, 768, 8192, 16384, fp4=True)
    assert L.gemm_a4w4_mxfp4_workspace_bytes(ctypes.byref(big)) > cap
    assert L.gemm_a4w4_mxfp4_noalloc(ctypes.byref(big), 1, None) == HIP_INVALID_VALUE
    fit = _far_kargs(qgemm, 129, 18432, 16384, fp4=True)
    need = L.gemm_a4w4_mxfp4_workspace_bytes(ctypes.byref(fit))
    assert 2 * 129 * 18432 * 4 < need <= cap                # two fp32 planes + panels
    if not torch.cuda.is_available():
        assert L.gemm_a4w4_mxfp4_noalloc(ctypes.byref(fit), 1, None) != HIP_INVALID_VALUE


def test_cached_workspace_outlives_its_replacement(qgemm, monkeypatch):
    """The address that a call takes from a workspace cache keeps its buffer
    alive: another thread's larger call may replace it before the launch."""
    import types
    import weakref

    opus, stream, dev = qgemm.opus, types.SimpleNamespace(cuda_stream=0), torch.device("cpu")
    monkeypatch.setattr(qgemm, "_WORKSPACES", {})
    monkeypatch.setattr(opus, "_WS", {})
    for cache, take in ((qgemm._WORKSPACES, lambda need: qgemm._workspace(lambda a: need, qgemm.Kargs(), None, dev, stream)),
                        (opus._WS, lambda need: opus._scratch("splitk", need, dev, stream))):
        address, nbytes = take(1000)
        first = weakref.ref(next(iter(cache.values())))
        assert nbytes == 1024 and address == first().data_ptr()
        assert ctypes.c_void_p.from_param(address) is not None
        take(5000)
        assert next(iter(cache.values())) is not first() and first() is not None
        del address
        assert first() is None


# ----------------------------------------------------------------- grouped entries
def _group(qgemm, shapes, fp4=False, bs=False):
    """An array of far-apart fake kargs blocks (never dereferenced)."""
    ks = []
    for i, (m, n, k) in enumerate(shapes):
        base = [(1 << 44) + ((5 * i + j) << 36) for j in range(5)]
        if bs:
            kg = k // 128
            ks.append(qgemm.Kargs(base[0], base[1], base[2], m, n, k, 1, k, 128, n, m * k, n * k, m * n, base[3],
                                  base[4], 1, kg, m * kg, ((n + 127) // 128) * kg))
        else:
            kb = k // 2 if fp4 else k
            ks.append(qgemm.Kargs(base[0], base[1], base[2], m, n, k, 1, kb, kb, n, m * kb, n * kb, m * n, base[3],
                                  base[4], k // 32, k // 32, m * (k // 32), n * (k // 32)))
    return (qgemm.Kargs * len(ks))(*ks)


def test_grouped_validation_and_workspace(qgemm):
    """Grouped calls: 1..16 problems of M <= 64 and batch 1; outputs must not
    overlap another problem's operands; the workspace query is 0 unless a
    problem splits K, and a split plan's workspace rule is the single
    entries' (too small / misaligned / overlapping rejected)."""
    L = qgemm.lib()
    fn, query = L.gemm_a8w8_blockscale_bpreshuffle_grouped, L.gemm_a8w8_blockscale_bpreshuffle_grouped_workspace_bytes
    ok = _group(qgemm, [(16, 2112, 7168), (16, 4096, 7168), (16, 7168, 2048)], bs=True)
    assert query(ok, 3) == 0                                             # one slice each: no workspace
    split = _group(qgemm, [(64, 2112, 16384), (8, 512, 2048)], bs=True)
    need = query(split, 2)
    assert need >= 256 + 4 * 64 * 2112 * 4                               # counters + >= 4 planes of problem 0
    for bad in (0, 17, -1):
        assert fn(ok, bad, 1, 0, None, 0, None) == HIP_INVALID_VALUE
        assert query(ok, bad) == 0
    assert fn(None, 1, 1, 0, None, 0, None) == HIP_INVALID_VALUE
    assert fn(ok, 3, 1, -1, None, 0, None) == HIP_INVALID_VALUE          # grid_blocks < 0
    big = _group(qgemm, [(16, 2112, 7168), (65, 512, 2048)], bs=True)
    assert fn(big, 2, 1, 0, None, 0, None) == HIP_INVALID_VALUE          # M > 64
    b2 = _group(qgemm, [(16, 2112, 7168)], bs=True)
    b2[0].batch = 2
    assert fn(b2, 1, 1, 0, None, 0, None) == HIP_INVALID_VALUE           # batch > 1
    ov = _group(qgemm, [(16, 2112, 7168), (16, 512, 2048)], bs=True)
    ov[1].ptr_c = ov[0].ptr_a                                            # C of problem 1 on A of problem 0
    assert fn(ov, 2, 1, 0, None, 0, None) == HIP_INVALID_VALUE
    ws = (1 << 44) + (90 << 36)
    assert fn(split, 2, 1, 0, ws, need - 1, None) == HIP_INVALID_VALUE   # too small
    assert fn(split, 2, 1, 0, ws + 16, need, None) == HIP_INVALID_VALUE  # misaligned
    assert fn(split, 2, 1, 0, split[0].ptr_b, need, None) == HIP_INVALID_VALUE
    mx = _group(qgemm, [(1, 7168, 16384), (32, 4096, 8192)], fp4=True)
    assert L.gemm_a4w4_mxfp4_grouped(mx, 2, 1, 0, None, 0, None) != HIP_INVALID_VALUE or torch.cuda.is_available()
    mx[1].k = 8000                                                      # K % 256 for fp4
    assert L.gemm_a4w4_mxfp4_grouped(mx, 2, 1, 0, None, 0, None) == HIP_INVALID_VALUE
    if not torch.cuda.is_available():
        assert fn(ok, 3, 1, 0, None, 0, None) != HIP_INVALID_VALUE       # valid: stops at the device check
        assert fn(split, 2, 1, 256, ws, need, None) != HIP_INVALID_VALUE


def test_layout_entry_contract(qgemm):
    """NN / TT / TN read their operands in place: the workspace query is 0
    for every layout, and the entry refuses (before any device work) a
    layout code out of range, strides that do not match the layout, and
    M or N not a multiple of 256."""
    L = qgemm.lib()
    m, n, k = 512, 768, 1024
    base = [(1 << 44) + (i << 38) for i in range(5)]

    def kargs(layout, **over):
        at, bn = layout in (2, 3), layout in (1, 3)
        a = qgemm.Kargs(base[0], base[1], base[2], m, n, k, 1, m if at else k, n if bn else k, n, m * k, n * k,
                        m * n, base[3], base[4], m, k // 128, m * (k // 128), (n // 128) * (k // 128))
        for f, v in over.items():
            setattr(a, f, v)
        return a

    for layout in range(4):
        assert L.gemm_a8w8_blockscale_layout_workspace_bytes(ctypes.byref(kargs(layout)), layout) == 0
    assert L.gemm_a8w8_blockscale_layout(ctypes.byref(kargs(1)), 4, 1, None, 0, None) == HIP_INVALID_VALUE
    assert L.gemm_a8w8_blockscale_layout(ctypes.byref(kargs(1)), 2, 1, None, 0, None) == HIP_INVALID_VALUE
    assert L.gemm_a8w8_blockscale_layout(ctypes.byref(kargs(3, stride_b=k)), 3, 1, None, 0, None) == HIP_INVALID_VALUE
    assert L.gemm_a8w8_blockscale_layout(ctypes.byref(kargs(1, n=640, stride_c=640, stride_b=640)), 1, 1, None, 0,
                                         None) == HIP_INVALID_VALUE
    if not torch.cuda.is_available():
        # conforming arguments pass validation and stop at the device check
        for layout in (1, 2, 3):
            assert L.gemm_a8w8_blockscale_layout(ctypes.byref(kargs(layout)), layout, 1, None, 0, None) \
                != HIP_INVALID_VALUE


def test_runs_kernel_id_contract(qgemm):
    """QGEMM_KID_RUNS (9): M <= 64, 16-byte aligned scale rows; a K split
    (more than 64 K-tiles, or narrow N) sizes its workspace as counters +
    fp32 planes; other shapes answer 0 / hipErrorInvalidValue."""
    L = qgemm.lib()
    kid = 9
    q = lambda a: L.gemm_a4w4_mxfp4_kid_workspace_bytes(ctypes.byref(a), kid)
    assert q(_far_kargs(qgemm, 65, 7168, 16384, fp4=True)) == 0                  # M > 64
    assert q(_far_kargs(qgemm, 32, 7168, 256, fp4=True)) == 0                    # 8-byte scale rows
    assert q(_far_kargs(qgemm, 32, 7168, 16384, fp4=True)) == 0                  # unsplit: no workspace
    m, n, k = 40, 256, 32768                                                     # 128 K-tiles: split
    need = q(_far_kargs(qgemm, m, n, k, fp4=True))
    assert need > 2048 and (need - 2048) % (m * n * 4) == 0
    a = _far_kargs(qgemm, 32, 7168, 256, fp4=True)
    assert L.gemm_a4w4_mxfp4_kid(ctypes.byref(a), 1, kid, None, 0, None) == HIP_INVALID_VALUE
    a = _far_kargs(qgemm, m, n, k, fp4=True)
    assert L.gemm_a4w4_mxfp4_kid(ctypes.byref(a), 1, kid, None, 0, None) == HIP_INVALID_VALUE   # split needs ws


def test_slice_kernel_id_contract(qgemm):
    """QGEMM_KID_SLICE (10): M <= 64, 16-byte aligned scale rows; K past one
    slice (64 / 32 / 16 K-tiles for 16 / 32 / 64 A rows) splits and sizes the
    workspace as counters + fp32 planes; other shapes answer 0 /
    hipErrorInvalidValue."""
    L = qgemm.lib()
    kid = 10
    q = lambda a: L.gemm_a4w4_mxfp4_kid_workspace_bytes(ctypes.byref(a), kid)
    assert q(_far_kargs(qgemm, 65, 7168, 16384, fp4=True)) == 0                  # M > 64
    assert q(_far_kargs(qgemm, 32, 7168, 256, fp4=True)) == 0                    # 8-byte scale rows
    assert q(_far_kargs(qgemm, 16, 7168, 16384, fp4=True)) == 0                  # one slice: unsplit
    for m, n, k in ((32, 7168, 16384), (64, 7168, 16384), (40, 256, 8192)):     # split
        need = q(_far_kargs(qgemm, m, n, k, fp4=True))
        assert need > 2048 and (need - 2048) % (m * n * 4) == 0, (m, n, k, need)
    a = _far_kargs(qgemm, 32, 7168, 256, fp4=True)
    assert L.gemm_a4w4_mxfp4_kid(ctypes.byref(a), 1, kid, None, 0, None) == HIP_INVALID_VALUE
    a = _far_kargs(qgemm, 32, 7168, 16384, fp4=True)
    assert L.gemm_a4w4_mxfp4_kid(ctypes.byref(a), 1, kid, None, 0, None) == HIP_INVALID_VALUE   # split needs ws


def test_ring_kernel_id_contract(qgemm):
    """QGEMM_KID_RING (11): M <= 64 in every family; a split sizes its
    workspace as counters + fp32 planes and needs it aligned; without one the
    id runs unsplit; other shapes answer 0 / hipErrorInvalidValue, dimensions
    near INT_MAX included."""
    L = qgemm.lib()
    kid, big = 11, (1 << 31) - 1
    q = lambda a: L.gemm_a8w8_mxfp8_kid_workspace_bytes(ctypes.byref(a), kid)
    assert q(_far_kargs(qgemm, 65, 7168, 16384)) == 0                            # M > 64
    assert q(_far_kargs(qgemm, 64, 16384, 2048)) == 0                            # tiles for every CU: unsplit
    for m, n, k in ((1, 512, 16384), (32, 1536, 7168), (64, 2112, 8192)):       # split
        a = _far_kargs(qgemm, m, n, k)
        need, ws = q(a), (1 << 44) + (7 << 38)
        assert need > 2048 and (need - 2048) % (m * n * 4) == 0, (m, n, k, need)
        call = lambda p, size: L.gemm_a8w8_mxfp8_kid(ctypes.byref(a), 1, kid, p, size, None)
        for p, size in ((ws, need - 1), (ws + 16, need), (a.ptr_c, need)):
            assert call(p, size) == HIP_INVALID_VALUE, (m, n, k)
        if not torch.cuda.is_available():
            assert call(ws, need) != HIP_INVALID_VALUE and call(None, 0) != HIP_INVALID_VALUE
    a = _far_kargs(qgemm, 65, 7168, 16384)
    assert L.gemm_a8w8_mxfp8_kid(ctypes.byref(a), 1, kid, None, 0, None) == HIP_INVALID_VALUE
    for m, n in ((1, big), (64, big - 15), (big, 1)):
        a = _kargs(qgemm, m=m, n=n)
        for query in ("gemm_a8w8_mxfp8", "gemm_a4w4_mxfp4", "gemm_a8w8_blockscale_bpreshuffle"):
            getattr(L, query + "_kid_workspace_bytes")(ctypes.byref(a), kid)
        assert L.gemm_a8w8_mxfp8_kid(ctypes.byref(a), 1, kid, None, 0, None) == HIP_INVALID_VALUE
