"""Forward GEMMs of up to 16 tokens (k_nf4_skinny) against the fused tile kernels and the float64
product, and the LoRA row products' side outputs when the row blocks are few.

The two kernels add the same fp32 products in another order; over a reduction of K products of
unit-variance inputs that differs by a few fp32 roundings of the running sum, far below the fp16
output's half ulp, so two outputs differ by at most one fp16 rounding step: 2^-10 of the value plus
2^-20 of the largest (where terms cancel)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _close(got, want):
    d = (got.float() - want.float()).abs()
    bound = 2.0 ** -10 * want.float().abs() + 2.0 ** -20 * want.float().abs().max()
    assert bool((d <= bound).all()), (d - bound).max().item()


# M: the 16-row block's edges; N: whole 16-column groups (partial ones, which only the C ABI takes:
# test_few_tokens_abi_gpu.py); K: shorter than one 128-wide chunk, a half chunk at the end, more
# chunks than one batch per wave
@pytest.mark.parametrize("M", [1, 5, 16, 17])
@pytest.mark.parametrize("n,k,r", [(64, 64, 16), (1536, 1536, 16), (256, 1472, 32),
                                   (1536, 8960, 16), (192, 320, 128)])
def test_few_tokens_match_the_tile_kernel(cuda, M, n, k, r):
    from mindxsoup_amd import kernels
    from mindxsoup_amd.quant import quantize_4bit

    print(f"case few tokens M={M} n={n} k={k} r={r}", flush=True)
    g = torch.Generator(device=cuda)
    g.manual_seed(M + n + k)
    rnd = lambda *s: torch.randn(s, device=cuda, generator=g)  # noqa: E731
    packed, st = quantize_4bit((rnd(n, k) * 0.02).half())
    x, bias = rnd(M, k).half(), rnd(n).half()
    a, b = (rnd(r, k) / k ** 0.5).half(), (rnd(n, r) * 0.1).half()
    _close(kernels.nf4_linear_fwd(x, packed, st, bias),
           kernels.nf4_linear_fwd(x, packed, st, bias, cfg=10, splits=1))
    hp, at, bt = kernels.lora_h_partials(x, a, 2.0, lora_b=b)
    assert torch.equal(at, a.t()) and torch.equal(bt, b.t())
    y, ht = kernels.nf4_linear_fwd_hp(x, packed, st, hp, b, bias)
    y0, ht0 = kernels.nf4_linear_fwd_hp(x, packed, st, hp, b, bias, cfg=10, splits=1)
    assert torch.equal(ht, ht0)
    _close(y, y0)
    if M > 16:  # past the few-token kernel: a group and a single launch plan their own tiles
        return
    # a group of two problems: each as alone
    outs = kernels.nf4_linear_fwd_hp_group([x] * 2, [packed] * 2, [st] * 2, [hp, hp], [b, b],
                                           [bias, None])
    assert torch.equal(outs[0][0], y) and torch.equal(outs[0][1], ht)
    assert torch.equal(outs[1][0], kernels.nf4_linear_fwd_hp(x, packed, st, hp, b)[0])


@pytest.mark.parametrize("M", [1, 16])
def test_pair_and_glu_equal_single_launches(cuda, M):
    from mindxsoup_amd import kernels
    from mindxsoup_amd.quant import quantize_4bit

    k, n = 1536, 8960
    ws = [quantize_4bit((torch.randn((n, k), device=cuda) * 0.02).half()) for _ in range(2)]
    x = torch.randn((M, k), device=cuda).half()
    ab = [((torch.randn((16, k), device=cuda) / 40).half(),
           (torch.randn((n, 16), device=cuda) * 0.1).half()) for _ in range(2)]
    rows = kernels.lora_h_partials_group([x] * 2, [t[0] for t in ab], 2.0, None, 1.0,
                                         [t[1] for t in ab])
    pair = kernels.nf4_linear_fwd_hp_pair(x, [w[0] for w in ws], [w[1] for w in ws],
                                          [o[0] for o in rows], [t[1] for t in ab])
    for (pk, st), (a, b), (hp, at, bt), (y, ht) in zip(ws, ab, rows, pair):
        y1, ht1 = kernels.nf4_linear_fwd_hp(x, pk, st, hp, b)
        assert torch.equal(y, y1) and torch.equal(ht, ht1)
        assert torch.equal(at, a.t()) and torch.equal(bt, b.t())
    up, h, _ = kernels.nf4_linear_fwd_glu(x, ws[1][0], ws[1][1], pair[0][0], rows[1][0], ab[1][1])
    assert torch.equal(up, pair[1][0])
    assert torch.equal(h, kernels.silu_mul(pair[0][0], pair[1][0]))
    y = torch.empty_like(up)
    kernels.nf4_linear_fwd_noalloc(x, ws[0][0], ws[0][1], y)
    assert torch.equal(y, kernels.nf4_linear_fwd(x, ws[0][0], ws[0][1]))


def test_split_plan_without_a_workspace(cuda):
    """A wide, long projection splits at few tokens; a caller without a workspace gets the plan
    that needs none."""
    from mindxsoup_amd import _lib, kernels
    from mindxsoup_amd.quant import quantize_4bit

    M, k, n = 64, 11008, 4096
    print("case split plan without a workspace", flush=True)
    packed, st = quantize_4bit((torch.randn((n, k), device=cuda) * 0.02).half())
    x = torch.randn((M, k), device=cuda).half()
    y = torch.empty((M, n), device=cuda, dtype=torch.float16)
    _lib.call("mxs_nf4_linear_fwd", _lib.ptr(x), M, k, n, *kernels._nf4_args(packed, st), None,
              None, None, 0, _lib.ptr(y), None, -1, 1, _lib.stream_of(x.device))
    _close(y, kernels.nf4_linear_fwd(x, packed, st))
