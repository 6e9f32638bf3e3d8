"""Several byte keep masks packed in one launch (mxs_keep_pack_group) against the one-mask launch,
with rows that break the 16-byte path and a mask at an odd address."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,M,K", [(1, 3, 31), (2, 5, 33), (3, 37, 1536), (4, 2, 100)])
def test_group_equals_single_packs(cuda, n, M, K):
    from mindxsoup_amd import _lib, kernels

    g = torch.Generator(device=cuda)
    g.manual_seed(n * 100 + K)
    buf = (torch.rand((n * M * K + 1,), device=cuda, generator=g) >= 0.3).to(torch.uint8)
    masks = [buf[1 + i * M * K:1 + (i + 1) * M * K].view(M, K) for i in range(n)]
    bits = [torch.empty((M, (K + 31) // 32), dtype=torch.int32, device=cuda) for _ in masks]
    _lib.call("mxs_keep_pack_group", n, kernels._ptr_array(masks), M, K,
              kernels._ptr_array(bits), _lib.stream_of(cuda))
    for m, b in zip(masks, bits):
        assert torch.equal(b, kernels.keep_bits(m, M, K))
