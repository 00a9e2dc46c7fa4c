"""Threads on one stream share its cached split-K workspace: plans of two
launches over it (partial planes, then their sum) give every thread the bits
of a call made alone."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def _linear(q, kind, m, n, k, seed, gpu):
    g = torch.Generator(gpu).manual_seed(seed)
    x, w = (torch.randn((r, k), generator=g, device=gpu).bfloat16() for r in (m, n))
    if kind == "bs":
        (a, sa), (b, sb) = q.quant_fp8_blockscale(x), q.quant_fp8_blockscale(w, block="128x128")
        ops, fn = (a, q.shuffle_b_kpanel(b), sa, sb), q.gemm_a8w8_bpreshuffle
    else:
        (a, sa), (b, sb) = q.quant_mxfp8(x), q.quant_mxfp8(w)
        ops, fn = (a, b, sa, sb), q.gemm_a8w8_mxfp8
    return lambda **kw: fn(*ops, **kw)


# ring kernel with a K split (two launches), 128 x 128 kernel with one, and a plan that counts in its only launch
@pytest.mark.parametrize("python", [False, True])
def test_threads_share_a_workspace(qgemm, gpu, python):
    calls = [_linear(qgemm, kind, m, n, k, i, gpu) for i, (kind, m, n, k) in enumerate(
        [("mxfp8", 32, 1536, 7168), ("bs", 64, 2112, 7168), ("mxfp8", 128, 2112, 7168), ("bs", 32, 1536, 7168)])]
    want = [c() for c in calls]
    # an `out` of the caller's takes the wrappers' Python code, which shares the workspace
    outs = [torch.empty_like(y) if python else None for y in want]
    bad, errors = [0] * len(calls), []
    start = threading.Barrier(len(calls))

    def worker(i):
        try:
            start.wait()
            for _ in range(200):
                y = calls[i](out=outs[i])
                bad[i] += not torch.equal(y, want[i])
        except Exception as e:    # noqa: BLE001 -- reported by the test's own thread
            errors.append(e)

    threads = [threading.Thread(target=worker, args=(i,)) for i in range(len(calls))]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not errors and bad == [0] * len(calls), (errors, bad)
