"""The few-token forward kernel (k_nf4_skinny) behind the C ABI, in the forms the package's own
callers never use: any number of output columns, any row length of the transposed LoRA operand."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _weight(dev, n, k, seed):
    from mindxsoup_amd.quant import quantize_4bit

    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    return g, *quantize_4bit((torch.randn((n, k), device=dev, generator=g) * 0.02).half())


@pytest.mark.parametrize("M,ldt", [(1, 8), (5, 16), (5, 64), (16, 24), (16, 136), (3, 512)])
@pytest.mark.parametrize("r", [16, 48])
def test_transposed_operand_has_zeros_past_the_rows(cuda, M, ldt, r):
    from mindxsoup_amd import _lib, kernels

    print(f"case few tokens ht M={M} ldt={ldt} r={r}", flush=True)
    n, k, S = 128, 192, 2
    g, packed, st = _weight(cuda, n, k, M + ldt)
    rnd = lambda *s: torch.randn(s, device=cuda, generator=g)  # noqa: E731
    x, b = rnd(M, k).half(), rnd(n, r).half()
    hp = rnd(S, ldt, r)
    y = torch.empty((M, n), dtype=torch.float16, device=cuda)
    ht = torch.full((r * ldt + 64,), 7.0, dtype=torch.float16, device=cuda)
    _lib.call("mxs_nf4_linear_fwd_hp", _lib.ptr(x), M, k, n, *kernels._nf4_args(packed, st), None,
              _lib.ptr(hp), S, ldt, _lib.ptr(b), r, _lib.ptr(ht), _lib.ptr(y), None, -1, 1,
              _lib.stream_of(x.device))
    assert bool((ht[r * ldt:] == 7).all())
    got = ht[:r * ldt].view(r, ldt)
    assert torch.equal(got[:, :M], (hp[0, :M] + hp[1, :M]).half().t())
    assert bool((got[:, M:] == 0).all())


@pytest.mark.parametrize("M", [1, 16])
@pytest.mark.parametrize("n,k", [(1, 64), (15, 128), (40, 64), (72, 192), (1000, 1536)])
def test_partial_column_groups(cuda, M, n, k):
    """Output widths that end inside a group of 16 columns, against the tile kernel: the same
    products in another order, at most one fp16 rounding step apart."""
    from mindxsoup_amd import kernels

    print(f"case few tokens columns M={M} n={n} k={k}", flush=True)
    g, packed, st = _weight(cuda, n, k, n)
    x = torch.randn((M, k), device=cuda, generator=g).half()
    bias = torch.randn((n,), device=cuda, generator=g).half()
    got = kernels.nf4_linear_fwd(x, packed, st, bias)
    want = kernels.nf4_linear_fwd(x, packed, st, bias, cfg=10, splits=1).float()
    bound = 2.0 ** -10 * want.abs() + 2.0 ** -20 * want.abs().max()
    assert bool(((got.float() - want).abs() <= bound).all())


# gate / up widths (N > K), where one projection alone must not split what the pair sums whole; and
# long reductions (K >= N), where it does split and the pair runs as two launches
@pytest.mark.parametrize("M,n,k", [(17, 11008, 4096), (64, 11008, 4096), (200, 11008, 4096),
                                   (200, 14336, 4096), (64, 4096, 4096), (1024, 4096, 4096),
                                   (40, 4096, 14336), (40, 8960, 1536)])
def test_forward_pair_has_the_bits_of_single_launches(cuda, M, n, k):
    from mindxsoup_amd import kernels, ops

    print(f"case forward pair M={M} n={n} k={k}", flush=True)
    g, p0, s0 = _weight(cuda, n, k, 1)
    _, p1, s1 = _weight(cuda, n, k, 2)
    rnd = lambda *s: torch.randn(s, device=cuda, generator=g)  # noqa: E731
    x, bias = rnd(M, k).half(), rnd(n).half()
    As = [(rnd(16, k) / k ** 0.5).half() for _ in range(2)]
    Bs = [(rnd(n, 16) * 0.1).half() for _ in range(2)]
    rows = kernels.lora_h_partials_group([x, x], As, 2.0, None, 1.0, Bs)
    hps = [o[0] for o in rows]
    assert kernels.fwd_pair_ok(M, n, n, k) == (n > k)
    pair = kernels.nf4_linear_fwd_hp_pair(x, [p0, p1], [s0, s1], hps, Bs, [bias, None])
    both = ops.load().lora_fwd_group(
        x, As, Bs, *map(list, zip(ops.nf4(p0, s0), ops.nf4(p1, s1))), [bias, None], [None, None],
        1.0, 2.0, False, None, None, 0)
    for i, (p, s, b) in enumerate(((p0, s0, bias), (p1, s1, None))):
        y, ht = kernels.nf4_linear_fwd_hp(x, p, s, hps[i], Bs[i], b)
        assert torch.equal(pair[i][0], y) and torch.equal(pair[i][1], ht)
        assert torch.equal(both[0][i], y) and torch.equal(both[1][i], ht)


@pytest.mark.parametrize("M", [1, 16, 17])
def test_swiglu_forward_refused_where_it_was(cuda, M):
    """A width whose plan has no SwiGLU epilogue is refused at few tokens too, nothing written."""
    from mindxsoup_amd import kernels

    n, k = 256, 1536
    print(f"case glu refused M={M}", flush=True)
    _, packed, st = _weight(cuda, n, k, 3)
    assert not kernels.glu_fused(M, n, k, False)
    x, gate = (torch.randn((M, w), device=cuda).half() for w in (k, n))
    with pytest.raises(RuntimeError, match="shape outside"):
        kernels.nf4_linear_fwd_glu(x, packed, st, gate)
