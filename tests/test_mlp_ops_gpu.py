"""The MLP block through torch.ops.mxs_nf4.mlp_fwd / mlp_bwd against the Python launch sequence: the
same kernels in the same order, so output and gradients are equal bit for bit."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _mlp(dev, hidden, inter, r, dropout):
    from mindxsoup_amd.linear4bit import Linear4bit, LoraLinear4bit
    from mindxsoup_amd.mlp import MLP

    layers = []
    for n, k in ((inter, hidden), (inter, hidden), (hidden, inter)):
        base = Linear4bit.from_weight((torch.randn((n, k), device=dev) * 0.02).half())
        layers.append(LoraLinear4bit(base, r=r, lora_alpha=2 * r, lora_dropout=dropout))
        torch.nn.init.normal_(layers[-1].lora_B["default"].weight, std=0.02)
    return MLP(*layers)


@pytest.mark.parametrize("M,hidden,inter,r,dropout,frozen", [
    (5, 1536, 8960, 16, 0.0, ()), (37, 1536, 8960, 16, 0.05, ()),
    (300, 1536, 4224, 32, 0.05, ("gate_proj", "x")), (1024, 1536, 8960, 16, 0.05, ("down_proj",)),
    (130, 1536, 1536, 16, 0.05, ())])
def test_compiled_block_equals_python_sequence(cuda, monkeypatch, M, hidden, inter, r, dropout,
                                               frozen):
    from mindxsoup_amd import ops

    print(f"case mlp op M={M} inter={inter} r={r} frozen={frozen}", flush=True)
    torch.manual_seed(M)
    mlp = _mlp(cuda, hidden, inter, r, dropout).train()
    for name in frozen:
        if name != "x":
            for p in getattr(mlp, name).parameters():
                p.requires_grad_(False)
    x = torch.randn((1, M, hidden), device=cuda)
    dy = torch.randn((1, M, hidden), device=cuda) * 1e-2
    got = {}
    for enabled in (True, False):
        monkeypatch.setattr(ops, "ENABLED", enabled)
        mlp.zero_grad(set_to_none=True)
        torch.manual_seed(7)  # the same dropout draws
        xl = x.clone().requires_grad_("x" not in frozen)
        y = mlp(xl)
        y.backward(dy)
        with torch.no_grad():
            mlp.eval()
            e = mlp(x)
            mlp.train()
        got[enabled] = [y.detach(), e, xl.grad] + [p.grad for p in mlp.parameters()]
    for i, (a, b) in enumerate(zip(got[True], got[False])):
        assert (a is None) == (b is None), i
        assert a is None or torch.equal(a, b), i


def test_unequal_scalings_pack_masks_once(cuda, monkeypatch):
    """gate and up with scalings of their own take the Python sequence: each byte keep mask is
    packed once for the forward's launches and the backward's."""
    from mindxsoup_amd import kernels

    print("case mlp unequal scalings", flush=True)
    packed, pack = [], kernels.keep_bits
    monkeypatch.setattr(kernels, "keep_bits", lambda m, M, K: (
        packed.append((M, K)) if m is not None and m.dtype != torch.int32 else None) or pack(m, M, K))
    torch.manual_seed(3)
    mlp = _mlp(cuda, 1536, 2048, 16, 0.05).train()
    mlp.up_proj.scaling["default"] = 1.0
    x = torch.randn((1, 37, 1536), device=cuda, requires_grad=True)
    y = mlp(x)
    y.backward(torch.randn_like(y))
    assert packed == [(37, 1536), (37, 1536), (37, 2048)]


@pytest.mark.parametrize("name", ["gate_proj", "down_proj"])
def test_wrong_keep_mask_is_a_value_error(cuda, monkeypatch, name):
    """A caller's keep mask of another shape or dtype is refused with one error on both paths,
    before anything is launched."""
    from mindxsoup_amd import ops

    print(f"case mlp wrong keep {name}", flush=True)
    mlp = _mlp(cuda, 1536, 2048, 16, 0.05).train()
    x = torch.randn((1, 37, 1536), device=cuda, requires_grad=True)
    width = getattr(mlp, name).base_layer.in_features
    for enabled in (True, False):
        monkeypatch.setattr(ops, "ENABLED", enabled)
        for keep in (torch.ones((37, width - 1), dtype=torch.uint8, device=cuda),
                     torch.ones((37, width), dtype=torch.int64, device=cuda)):
            getattr(mlp, name).next_keep = keep
            with pytest.raises(ValueError, match="keep mask"):
                mlp(x)
