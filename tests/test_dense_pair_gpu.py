"""The summed input gradient of gate and up at many tokens (mxs_nf4_linear_bwd_dx_hp_pair): from
decoded weights (k_dense_gemm over two reductions) with a keep mask on both or on neither, on the
fused kernel with a mask on one; ranks staged through LDS (16) and read from memory, unequal widths.

Reference: the two projections' single input gradients on the fused kernels, each rounded to fp16,
added in fp32.  The summed launch rounds once, so the two differ by the parts' roundings (half an
ulp each), its own, and the fp32 sums' other order (2^-18 of the largest value)."""

import pytest
import torch

pytestmark = pytest.mark.gpu

S, MS = 2.0, 1 / 0.95
K = 1536


def _proj(dev, n, M, r, seed):
    from mindxsoup_amd.quant import quantize_4bit

    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    rnd = lambda *s: torch.randn(s, device=dev, generator=g)  # noqa: E731
    packed, st = quantize_4bit((rnd(n, K) * 0.02).half())
    return dict(n=n, packed=packed, st=st, a=(rnd(r, K) / K ** 0.5).half(),
                b=(rnd(n, r) * 0.01).half(), dy=rnd(M, n).half(),
                ht=rnd(r, (M + 7) // 8 * 8).half(),
                keep=(torch.rand((M, K), device=dev, generator=g) >= 0.05).to(torch.uint8))


def _bound(parts, two):
    return 2.0 ** -11 * (sum(t.float().abs() for t in parts) + two.abs()) * 1.01 + \
        2.0 ** -18 * two.abs().max()


@pytest.mark.parametrize("widths", [(8960, 8960), (8960, 6144)])
@pytest.mark.parametrize("r", [16, 32, 64])
@pytest.mark.parametrize("masked", [(True, False), (False, True), (False, False), (True, True)])
def test_masks_of_either_projection(cuda, masked, r, widths):
    from mindxsoup_amd import kernels

    M = 1430  # the last row band holds 150 rows
    print(f"case dense dX pair masked={masked} r={r} widths={widths}", flush=True)
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the plans of another CU count")
    assert kernels.gemm_route("dx", M, widths[0], K, widths[1]) == "dense"
    ps = [_proj(cuda, n, M, r, 20 + i) for i, n in enumerate(widths)]
    keeps = [p["keep"] if m else None for p, m in zip(ps, masked)]
    dhps = [kernels.lora_dh_partials(p["dy"], p["b"].t().contiguous(), S) for p in ps]
    ats = [p["a"].t().contiguous() for p in ps]
    dys = [p["dy"] for p in ps]
    nf4 = ([p["packed"] for p in ps], [p["st"] for p in ps])
    dx, dhts = kernels.nf4_linear_bwd_dx_hp_pair(dys, *nf4, dhps, ats, keeps, MS)
    parts = [kernels.nf4_linear_bwd_dx_hp(d, p["packed"], p["st"], h, at, kp, MS, cfg=11,
                                          splits=4)
             for d, p, h, at, kp in zip(dys, ps, dhps, ats, keeps)]
    two = parts[0][0].float() + parts[1][0].float()
    assert bool(((dx.float() - two).abs() <= _bound([t[0] for t in parts], two)).all())
    for (_, want), dht in zip(parts, dhts):
        assert torch.equal(dht, want)
    if widths[0] != widths[1]:  # one launch for both gradients needs equal widths
        return
    x, hts = torch.randn((M, K), device=cuda).half(), [p["ht"] for p in ps]
    dx2, dhts2, grads = kernels.nf4_linear_bwd_dx_hp_pair_grads(dys, *nf4, dhps, ats, hts, x,
                                                                keeps, MS)
    assert torch.equal(dx, dx2)
    for (da, db), p, dht, ht, kp in zip(grads, ps, dhts2, hts, keeps):
        da1, db1 = kernels.lora_grads(dht, ht, x, p["dy"], kp, MS)
        assert torch.equal(da, da1) and torch.equal(db, db1)


@pytest.mark.parametrize("M", [64, 1430, 3001, 3200, 8192])
def test_callers_workspace(cuda, M):
    """A workspace of projection_workspace_bytes serves the summed gradient at every token count,
    whatever the faster plan would take (more fp32 planes at few tokens, the decoded weights at
    many), and nothing past its end is written; a smaller one than four planes is refused."""
    from mindxsoup_amd import kernels
    from mindxsoup_amd.linear4bit import lora_backward_group

    print(f"case dX pair in a caller's workspace M={M}", flush=True)
    x = torch.randn((M, K), device=cuda).half()
    ps = [_proj(cuda, 8960, M, 16, 30 + i) for i in range(2)]
    items = [dict(dy=p["dy"], x2d=x, keep=p["keep"], ht=p["ht"], at=p["a"].t().contiguous(),
                  bt=p["b"].t().contiguous(), packed=p["packed"], state=p["st"], mask_scale=MS,
                  s=S, wants=(True, True, True)) for p in ps]
    nbytes = kernels.projection_workspace_bytes(M, K, 8960)
    whole = torch.full((nbytes + 4096,), 7, dtype=torch.uint8, device=cuda)
    got = lora_backward_group(items, ws=whole[:nbytes], sum_dx=True)
    assert bool((whole[nbytes:] == 7).all())
    parts = [r[0] for r in lora_backward_group(items)]
    two = parts[0].float() + parts[1].float()
    for dx in (got[0][0], lora_backward_group(items, sum_dx=True)[0][0]):
        assert bool(((dx.float() - two).abs() <= _bound(parts, two)).all())
    dhps = [kernels.lora_dh_partials(it["dy"], it["bt"], S) for it in items]
    with pytest.raises(ValueError, match="workspace"):
        kernels.nf4_linear_bwd_dx_hp_pair([p["dy"] for p in ps], [p["packed"] for p in ps],
                                          [p["st"] for p in ps], dhps, [it["at"] for it in items],
                                          ws=whole[:16 * M * K - 4])
