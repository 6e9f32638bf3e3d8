"""The SwiGLU forms of a GEMM (mxs_nf4_linear_fwd_glu, mxs_nf4_linear_bwd_dx_glu) against the plain
GEMM and the elementwise kernel at many tokens, at shapes where decoding the weight pays for one
form and not for the other, or splits the reduction in one and not the other: the same bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _operands(dev, n, k, M, seed):
    from mindxsoup_amd.quant import quantize_4bit

    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    rnd = lambda *s: torch.randn(s, device=dev, generator=g)  # noqa: E731
    return rnd, *quantize_4bit((rnd(n, k) * 0.02).half())


# N, K, tokens: square, wide and long, first counts of the route and partial row bands
SHAPES = [(3392, 1408, 4663), (3776, 1472, 5130), (4096, 4096, 1080), (4096, 2048, 844),
          (1536, 8960, 8192), (1536, 8960, 769)]


@pytest.mark.parametrize("n,k,M", SHAPES)
def test_input_gradient(cuda, n, k, M):
    from mindxsoup_amd import kernels

    print(f"case swiglu dX n={n} k={k} M={M}", flush=True)
    assert kernels.glu_fused(M, n, k, True)
    rnd, packed, st = _operands(cuda, n, k, M, 1)
    dy, gate, up = rnd(M, n).half(), rnd(M, k).half(), rnd(M, k).half()
    dhp = rnd(1, (M + 7) // 8 * 8, 16)
    at = (rnd(k, 16) * 0.1).half()
    keep = (torch.rand((M, k), device=cuda) >= 0.05).to(torch.uint8)
    dh, dht = kernels.nf4_linear_bwd_dx_hp(dy, packed, st, dhp, at, keep, 1 / 0.95)
    g1, u1 = gate.clone(), up.clone()
    kernels.silu_mul_bwd_(dh, g1, u1)
    dht2 = kernels.nf4_linear_bwd_dx_glu_(dy, packed, st, gate, up, dhp, at, keep, 1 / 0.95)
    assert torch.equal(gate, g1) and torch.equal(up, u1) and torch.equal(dht, dht2)


@pytest.mark.parametrize("n,k,M", [(2048, 4096, 1300), (3328, 5632, 2400), (1728, 12800, 1100),
                                   (4096, 4096, 1080), (8960, 1536, 2048)])
def test_forward(cuda, n, k, M):
    from mindxsoup_amd import kernels

    print(f"case swiglu forward n={n} k={k} M={M}", flush=True)
    assert kernels.glu_fused(M, n, k, False)
    rnd, packed, st = _operands(cuda, n, k, M, 2)
    x, gate, b = rnd(M, k).half(), rnd(M, n).half(), (rnd(n, 16) * 0.1).half()
    hp = rnd(1, (M + 7) // 8 * 8, 16)
    y, ht = kernels.nf4_linear_fwd_hp(x, packed, st, hp, b)
    y2, h2, ht2 = kernels.nf4_linear_fwd_glu(x, packed, st, gate, hp, b)
    assert torch.equal(y, y2) and torch.equal(ht, ht2)
    assert torch.equal(h2, kernels.silu_mul(gate, y))
