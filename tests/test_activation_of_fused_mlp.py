"""Which activations a fused gated MLP block takes for SiLU: by what their class computes, not by its name or base."""
import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F


class Scaled(nn.SiLU):
    def forward(self, x):
        return super().forward(x) * 0.5 + 0.25


def _namesake():
    class SiLU(nn.Module):
        def forward(self, x):
            return torch.tanh(x)
    return SiLU


def _same_code_other_function():
    class SiLUActivation(nn.Module):
        pass
    ns = {"nn": type("nn", (), {"functional": type("functional", (), {"silu": staticmethod(torch.tanh)})})}
    exec("def forward(self, input):\n    return nn.functional.silu(input)", ns)
    SiLUActivation.forward = ns["forward"]
    return SiLUActivation


class Called(nn.SiLU):
    def __call__(self, x):
        return torch.tanh(x)


class Inherited(nn.SiLU):
    pass


OTHERS = {"subclass": Scaled, "namesake": _namesake(), "same code": _same_code_other_function(), "call": Called}


def test_activation_is_judged_by_what_it_computes():
    from transformers.activations import SiLUActivation
    from alpaca_lora_4bit_amd.model_attn_mlp_patch import _is_silu
    for act in (nn.SiLU(), nn.SiLU(inplace=True), Inherited(), SiLUActivation(), F.silu):
        assert _is_silu(act)
    for cls in OTHERS.values():
        assert not _is_silu(cls())
    instance = nn.SiLU()
    instance.forward = torch.tanh
    assert not _is_silu(instance) and not _is_silu(nn.GELU()) and not _is_silu(None) and not _is_silu(torch.tanh)


@pytest.mark.gpu
@pytest.mark.parametrize("name", [*OTHERS, "replaced"])
def test_other_activations_keep_the_blocks_own_forward(oracle, name):
    """Decode at 1, 4 and 16 rows, prefill and training at 40: what the block's own modules give, forward and gradient."""
    from conftest import rel_err, to_cuda_layer
    from alpaca_lora_4bit_amd.autograd_4bit import Autograd4bitQuantLinear
    from alpaca_lora_4bit_amd.model_attn_mlp_patch import make_fused_mlp

    class Gated(nn.Module):
        def forward(self, x):
            return self.down_proj(self.act_fn(self.gate_proj(x)) * self.up_proj(x))

    H, I, gs = 256, 384, 128
    own, fused = Gated(), Gated()
    for m in (own, fused):
        for i, (layer, k, n) in enumerate((("gate_proj", H, I), ("up_proj", H, I), ("down_proj", I, H))):
            lin = Autograd4bitQuantLinear(k, n, groupsize=gs)
            for key, v in to_cuda_layer(oracle.make_layer(k, n, gs, seed=30 + i)).items():
                if isinstance(v, torch.Tensor):
                    setattr(lin, key, v)
            lin.bias = torch.zeros(n, dtype=torch.float16, device="cuda")
            setattr(m, layer, lin)
        m.act_fn = nn.SiLU() if name == "replaced" else OTHERS[name]()
    assert make_fused_mlp(fused) == 1
    if name == "replaced":                                   # after the block was grouped, and after its first steps
        with torch.no_grad():
            for M in (1, 16):
                fused(torch.zeros(M, H, dtype=torch.float16, device="cuda"))
        own.act_fn = fused.act_fn = Scaled()
    for M in (1, 4, 16, 40):
        x = torch.from_numpy(oracle.make_activations(M, H, seed=M)).cuda()
        with torch.no_grad():
            # the same products, alone and grouped, and the same activation
            assert rel_err(fused(x).cpu().numpy(), own(x).double().cpu().numpy()) <= 1e-3
    res = []
    for m in (fused, own):
        leaf = x.clone().requires_grad_(True)
        y = m(leaf)
        y.backward(torch.ones_like(y))
        res.append((y.detach(), leaf.grad))
    for a, b in zip(*res):
        assert rel_err(a.cpu().numpy(), b.double().cpu().numpy()) <= 3e-3          # grouped grad-input: the sums in another order
