"""The dense route of the NF4 GEMMs (weights decoded once into the workspace, then one plain fp16
GEMM), taken by the planner at many tokens, against the fused kernels.

Unsplit it accumulates the same products in the same order from the same start, so the outputs
are the fused kernels' bits.  A split reduction adds fp32 partial sums in another order: each sum
differs by at most a few fp32 roundings of its partials, so the fp16 outputs differ by at most one
rounding step: |a - b| <= 2^-10 |b| plus, where terms cancel, 2^-20 of the largest output.
Shapes: partial row bands and column tiles, one and several splits, ranks 16 and 32, with and
without masks and bias."""

import pytest
import torch

pytestmark = pytest.mark.gpu

S, MS = 2.0, 1 / 0.95


def _proj(dev, n, k, M, r, seed, x=None, bias=False):
    from mindxsoup_amd.quant import quantize_4bit

    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    packed, st = quantize_4bit((torch.randn((n, k), device=dev, generator=g) * 0.02).half())
    rnd = lambda *s: torch.randn(s, device=dev, generator=g)  # noqa: E731
    return dict(n=n, k=k, packed=packed, st=st, x=rnd(M, k).half() if x is None else x,
                a=(rnd(r, k) / k ** 0.5).half(), b=(rnd(n, r) * 0.01).half(),
                dy=rnd(M, n).half(), bias=rnd(n).half() if bias else None,
                keep=(torch.rand((M, k), device=dev, generator=g) >= 0.05).to(torch.uint8))


def _on_dense_route(op, M, n, k, n1=0):
    """The planned call runs on decoded weights (else, on another CU count, the test is skipped)."""
    from mindxsoup_amd import kernels

    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the plans of another CU count")
    assert kernels.gemm_route(op, M, n, k, n1) == "dense"


def _close(got, want):
    d = (got.float() - want.float()).abs()
    bound = 2.0 ** -10 * want.float().abs() + 2.0 ** -20 * want.float().abs().max()
    assert bool((d <= bound).all()), (d - bound).max().item()


def _same(got, want, split):
    if split:
        _close(got, want)
    else:
        assert torch.equal(got, want)


# (N, K, M, rank, bias, dense splits): square; a partial column tile; split; wide
FWD = [(1536, 1536, 8100, 16, True, 1), (1600, 4096, 8190, 32, False, 1),
       (1536, 8960, 3001, 16, False, 3), (8960, 1536, 2047, 16, True, 1)]


@pytest.mark.parametrize("n,k,M,r,bias,splits", FWD)
def test_forward(cuda, n, k, M, r, bias, splits):
    from mindxsoup_amd import kernels

    print(f"case dense fwd n={n} k={k} M={M} r={r}", flush=True)
    p = _proj(cuda, n, k, M, r, 1, bias=bias)
    _on_dense_route("fwd", M, n, k)
    hp, _, _ = kernels.lora_h_partials(p["x"], p["a"], S, p["keep"], MS, lora_b=p["b"])
    y, ht = kernels.nf4_linear_fwd_hp(p["x"], p["packed"], p["st"], hp, p["b"], p["bias"])
    y0, ht0 = kernels.nf4_linear_fwd_hp(p["x"], p["packed"], p["st"], hp, p["b"], p["bias"],
                                        cfg=10, splits=1)
    assert torch.equal(ht, ht0)
    _same(y, y0, splits > 1)
    _same(kernels.nf4_linear_fwd(p["x"], p["packed"], p["st"], p["bias"]),
          kernels.nf4_linear_fwd(p["x"], p["packed"], p["st"], p["bias"], cfg=10, splits=1),
          splits > 1)


# (N, K, M, rank, masked, split): dX is [M, K]
BWD = [(1536, 8960, 2047, 16, True, False), (1536, 8960, 2048, 32, True, False),
       (1536, 1536, 8100, 16, False, False), (8960, 1536, 3001, 16, True, True)]


@pytest.mark.parametrize("n,k,M,r,masked,split", BWD)
def test_input_gradient(cuda, n, k, M, r, masked, split):
    from mindxsoup_amd import kernels

    print(f"case dense dx n={n} k={k} M={M} r={r}", flush=True)
    p = _proj(cuda, n, k, M, r, 2)
    _on_dense_route("dx", M, n, k)
    keep = p["keep"] if masked else None
    dhp = kernels.lora_dh_partials(p["dy"], p["b"].t().contiguous(), S)
    at = p["a"].t().contiguous()
    args = (p["dy"], p["packed"], p["st"], dhp, at, keep, MS)
    dx, dht = kernels.nf4_linear_bwd_dx_hp(*args)
    dx0, dht0 = kernels.nf4_linear_bwd_dx_hp(*args, cfg=10, splits=1)
    assert torch.equal(dht, dht0)
    _same(dx, dx0, split)
    if not split and kernels.glu_fused(M, n, k, True):  # the SwiGLU adjoint in the epilogue
        gate, up = (torch.randn((M, k), device=cuda).half() for _ in range(2))
        g1, u1 = gate.clone(), up.clone()
        kernels.silu_mul_bwd_(dx0, g1, u1)
        kernels.nf4_linear_bwd_dx_glu_(p["dy"], p["packed"], p["st"], gate, up, dhp, at, keep, MS)
        assert torch.equal(gate, g1) and torch.equal(up, u1)


@pytest.mark.parametrize("M,T,r", [(6144, 2048, 16), (8190, 1638, 32)])
def test_qkv_group_with_rope_and_summed_dx(cuda, M, T, r):
    """q, k, v forward with the rotation, and their summed dX, from decoded weights."""
    from mindxsoup_amd import kernels
    from mindxsoup_amd.rope import as_rows, qkv_rope

    print(f"case dense qkv M={M} r={r}", flush=True)
    shapes = (1536, 256, 256)
    x = torch.randn((M, 1536), device=cuda).half()
    ps = [_proj(cuda, n, 1536, M, r, 3 + i, x=x, bias=True) for i, n in enumerate(shapes)]
    if not kernels._group_workspace_bytes(M, shapes, 1536, 2):
        pytest.skip("this device's CU count plans the fused kernel")
    rows = kernels.lora_h_partials_group([x] * 3, [p["a"] for p in ps], S,
                                         [p["keep"] for p in ps], MS, [p["b"] for p in ps])
    ang = torch.arange(T, device=cuda).float()[:, None] * torch.rand(128, device=cuda)
    cos, sin = ang.cos()[None].contiguous(), ang.sin()[None].contiguous()
    outs = kernels.nf4_linear_fwd_hp_group([x] * 3, [p["packed"] for p in ps],
                                           [p["st"] for p in ps], [o[0] for o in rows],
                                           [p["b"] for p in ps], [p["bias"] for p in ps],
                                           rope=(2, cos, sin))
    ref = [kernels.nf4_linear_fwd_hp(x, p["packed"], p["st"], o[0], p["b"], p["bias"], cfg=10,
                                     splits=1) for p, o in zip(ps, rows)]
    B = M // T
    q, k_, v = (o[0].view(B, T, -1) for o in ref)
    qr, kr, _ = qkv_rope(q, None, k_, v, None, cos, sin, 12, 2)
    assert torch.equal(outs[0][0].view(B, T, -1), as_rows(qr))
    assert torch.equal(outs[1][0].view(B, T, -1), as_rows(kr))
    assert torch.equal(outs[2][0], ref[2][0])
    assert all(torch.equal(o[1], r_[1]) for o, r_ in zip(outs, ref))
    if r != 16:  # the summed launch takes rank 16
        return
    dhs = kernels.lora_dh_group([p["dy"] for p in ps], [o[2] for o in rows], S)
    dx, _ = kernels.nf4_linear_bwd_dx_grads_sum(
        [p["dy"] for p in ps], [p["packed"] for p in ps], [p["st"] for p in ps],
        [d[0] for d in dhs], [o[1] for o in rows], [d[1] for d in dhs], [o[1] for o in ref], x,
        [p["keep"] for p in ps], MS, grads=False)
    parts = [kernels.nf4_linear_bwd_dx(p["dy"], p["packed"], p["st"], d[0], None, p["keep"], MS,
                                       cfg=10, splits=1, lora_at=o[1])
             for p, d, o in zip(ps, dhs, rows)]
    two = parts[0].float() + parts[1].float() + parts[2].float()
    # the parts' own fp16 roundings (half an ulp each of at most the largest part) and one more
    bound = 2.0 ** -11 * (sum(t.float().abs() for t in parts) + two.abs()) * 1.01 + 1e-6
    assert bool(((dx.float() - two).abs() <= bound).all())


# which of the two is on decoded weights: the summed dX in five splits, the forward, both (two
# splits, and unsplit)
@pytest.mark.parametrize("M,dense", [(1430, ("dx",)), (3001, ("fwd",)), (3200, ("fwd", "dx")),
                                     (8192, ("fwd", "dx"))])
def test_gate_up_pair(cuda, M, dense):
    """gate and up: forward in one launch (the bits of two), the summed dX and both projections'
    gradients."""
    from mindxsoup_amd import kernels

    print(f"case dense pair M={M}", flush=True)
    for op in dense:
        _on_dense_route(op, M, 8960, 1536, 8960)
    x = torch.randn((M, 1536), device=cuda).half()
    ps = [_proj(cuda, 8960, 1536, M, 16, 9 + i, x=x) for i in range(2)]
    rows = kernels.lora_h_partials_group([x] * 2, [p["a"] for p in ps], S,
                                         [p["keep"] for p in ps], MS, [p["b"] for p in ps])
    nf4 = ([p["packed"] for p in ps], [p["st"] for p in ps])
    outs = kernels.nf4_linear_fwd_hp_pair(x, *nf4, [o[0] for o in rows], [p["b"] for p in ps])
    for p, o, (y, ht) in zip(ps, rows, outs):
        y0, ht0 = kernels.nf4_linear_fwd_hp(x, p["packed"], p["st"], o[0], p["b"], cfg=7,
                                            splits=1)
        assert torch.equal(y, y0) and torch.equal(ht, ht0)
    dhps = kernels.lora_dh_partials_group([p["dy"] for p in ps], [o[2] for o in rows], S)
    ats, hts = [o[1] for o in rows], [o[1] for o in outs]
    keeps = [p["keep"] for p in ps]
    dys = [p["dy"] for p in ps]
    dx, dhts, grads = kernels.nf4_linear_bwd_dx_hp_pair_grads(dys, *nf4, dhps, ats, hts, x, keeps,
                                                              MS)
    dx2, dhts2 = kernels.nf4_linear_bwd_dx_hp_pair(dys, *nf4, dhps, ats, keeps, MS)
    assert torch.equal(dx, dx2) and all(torch.equal(a, b) for a, b in zip(dhts, dhts2))
    apart = kernels.lora_grads_group(dhts, hts, [x, x], dys, keeps, MS)
    for (a1, b1), (a2, b2) in zip(grads, apart):
        assert torch.equal(a1, a2) and torch.equal(b1, b2)
    parts = [kernels.nf4_linear_bwd_dx_hp(d, p["packed"], p["st"], h, at, kp, MS, cfg=11,
                                          splits=4)[0]
             for d, p, h, at, kp in zip(dys, ps, dhps, ats, keeps)]
    two = parts[0].float() + parts[1].float()
    bound = 2.0 ** -11 * (sum(t.float().abs() for t in parts) + two.abs()) * 1.01 + \
        2.0 ** -18 * two.abs().max()  # and the fp32 sums' other order
    assert bool(((dx.float() - two).abs() <= bound).all())


@pytest.mark.parametrize("op,n,k,n1", [("fwd", 1536, 8960, 0), ("fwd", 8960, 1536, 0),
                                       ("dx", 1536, 8960, 0), ("dx", 8960, 1536, 0),
                                       ("dx", 8960, 1536, 8960)])
def test_first_planned_token_count(cuda, op, n, k, n1):
    """The fewest tokens that decode the weight, and one fewer: within the split sums' bound."""
    from mindxsoup_amd import kernels

    first = next((M for M in range(2, 8192) if kernels.gemm_route(op, M, n, k, n1) == "dense"), 0)
    if not first:
        pytest.skip("the plans of another CU count")
    print(f"case first dense {op} n={n} k={k} n1={n1} M={first}", flush=True)
    for M in (first, first - 1):
        ps = [_proj(cuda, n, k, M, 16, 40 + i) for i in range(2 if n1 else 1)]
        if op == "fwd":
            args = (ps[0]["x"], ps[0]["packed"], ps[0]["st"])
            _close(kernels.nf4_linear_fwd(*args), kernels.nf4_linear_fwd(*args, cfg=10, splits=1))
            continue
        dhps = [kernels.lora_dh_partials(p["dy"], p["b"].t().contiguous(), S) for p in ps]
        ats = [p["a"].t().contiguous() for p in ps]
        parts = [kernels.nf4_linear_bwd_dx_hp(p["dy"], p["packed"], p["st"], h, at, p["keep"], MS,
                                              cfg=10, splits=1)[0]
                 for p, h, at in zip(ps, dhps, ats)]
        if not n1:
            _close(kernels.nf4_linear_bwd_dx_hp(ps[0]["dy"], ps[0]["packed"], ps[0]["st"], dhps[0],
                                                ats[0], ps[0]["keep"], MS)[0], parts[0])
            continue
        dx, _ = kernels.nf4_linear_bwd_dx_hp_pair(
            [p["dy"] for p in ps], [p["packed"] for p in ps], [p["st"] for p in ps], dhps, ats,
            [p["keep"] for p in ps], MS)
        two = parts[0].float() + parts[1].float()
        bound = 2.0 ** -11 * (sum(t.float().abs() for t in parts) + two.abs()) * 1.01 + \
            2.0 ** -18 * two.abs().max()
        assert bool(((dx.float() - two).abs() <= bound).all())
