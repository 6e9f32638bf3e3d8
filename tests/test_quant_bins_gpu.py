"""The quantizer's bin lookup and in-kernel mean against the oracle quantizer: values at and around
every midpoint and bin edge, zero blocks, one block, and weights whose mean takes one partial, the
last that fits the in-kernel sum, and the launch of its own."""

import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _check(cuda, w):
    from mindxsoup_amd.quant import quantize_4bit

    packed, st = quantize_4bit(torch.from_numpy(w).to(cuda))
    q = O.quantize(w)
    assert np.array_equal(packed.view(-1).cpu().numpy(), q.packed)
    assert np.array_equal(st.absmax.cpu().numpy(), q.absmax8)
    assert np.array_equal(st.state2.absmax.cpu().numpy(), q.absmax2)
    assert float(st.offset.item()) == np.float32(q.offset)


def test_codes_around_every_midpoint_and_edge(cuda):
    from mindxsoup_amd.nf4 import NF4_VALUES

    mids = ((NF4_VALUES[:-1].astype(np.float64) + NF4_VALUES[1:]) / 2).astype(np.float16)
    edges = (np.arange(-16, 17) / 16).astype(np.float16)
    pts = []
    for c in np.concatenate([mids, edges]):
        u = np.array([c], np.float16).view(np.int16).astype(np.int32)
        pts.append((u + np.arange(-12, 13)).astype(np.int16).view(np.float16))
    v = np.concatenate(pts)
    v = v[np.isfinite(v) & (np.abs(v) <= 1)]
    v = np.resize(v, ((v.size + 62) // 63) * 63).reshape(-1, 63)
    one = np.ones((v.shape[0], 1), np.float16)  # the block's maximum: x = v exactly
    w = np.concatenate([one, v], axis=1)
    _check(cuda, np.concatenate([w, -w, np.zeros((2, 64), np.float16)]))


@pytest.mark.parametrize("n_blocks", [1, 257, 4096, 4097, 256 * 4096, 256 * 4096 + 1])
def test_mean_of_partials(cuda, n_blocks):
    rng = np.random.default_rng(n_blocks)
    small = (rng.standard_normal((min(n_blocks, 5000), 64)) * 0.02).astype(np.float16)
    _check(cuda, np.resize(small, (n_blocks, 64)))
