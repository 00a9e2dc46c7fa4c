"""The layout kernels at their tile edges -- 16 rows x 2 K-tiles per workgroup
for small weights, x 8 for large ones -- against the layouts' definitions:
partial last K-tile pairs, W16 rows that end inside a K-tile, ragged N, and a
padded source pitch.  Bytes, so every comparison is exact."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _source(n, k, pad, gpu):
    g = torch.Generator(gpu).manual_seed(n * 131 + k)
    return torch.randint(0, 256, (n, k + pad), dtype=torch.uint8, generator=g, device=gpu)[:, :k]


# 16384 row blocks x K-tiles is where the larger workgroups begin, 4096 for K-panel
SIZES = [(16, 128), (48, 384), (80, 1152), (1024, 8064), (1024, 8192), (4096, 8064), (4096, 8192), (4112, 9344)]


@pytest.mark.parametrize("pad", [0, 16])
@pytest.mark.parametrize("n,k", SIZES + [(16, 16), (32, 144), (4096, 8208)])
def test_w16(qgemm, gpu, n, k, pad):
    src = _source(n, k, pad, gpu)
    want = src.reshape(n // 16, 16, k // 16, 16).transpose(1, 2).reshape(n, k)
    assert torch.equal(qgemm.shuffle_weight_16x16(src), want)


@pytest.mark.parametrize("pad", [0, 16])
@pytest.mark.parametrize("n,k", SIZES + [(1, 128), (17, 256), (4101, 8320)])
def test_kpanel_and_fragment_order(qgemm, gpu, n, k, pad):
    src = _source(n, k, pad, gpu)
    want = src.reshape(n, k // 128, 128).transpose(0, 1)
    assert torch.equal(qgemm.shuffle_b_kpanel(src), want)
    rows = torch.nn.functional.pad(src, (0, 0, 0, -n % 16))
    frag = rows.reshape(-1, 16, k // 16, 16).transpose(1, 2).reshape(-1)    # zero rows past N
    assert torch.equal(qgemm.ldsbypass_pack_b(src).reshape(-1), frag)
