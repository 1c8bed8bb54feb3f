"""silu(gate) * up in one pass, forward and backward, against torch's own operations on the same fp16 tensors."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _close(got, want):
    """One fp16 rounding may fall the other way (2^-10 of the value, the smallest subnormal near zero): both sides round the
    same expressions, from exponentials that differ in the last bits of fp32.  Backward rounds twice in a row."""
    import torch
    got, want = got.float(), want.float()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    fin = torch.isfinite(want) & torch.isfinite(got)
    assert torch.equal(got[~fin & ~torch.isnan(want)], want[~fin & ~torch.isnan(want)])
    assert bool(((got[fin] - want[fin]).abs() <= 2.0 ** -9 * want[fin].abs() + 2.0 ** -23).all())


@pytest.mark.parametrize("shape", [(1,), (7,), (8,), (9,), (3, 5, 683), (2047,), (2048 + 8,), (64, 11008), (129, 13824)])
def test_silu_mul_matches_torch(shape):
    import torch
    import torch.nn.functional as F
    from alpaca_lora_4bit_amd import quant_hip
    gen = torch.Generator(device="cuda").manual_seed(sum(shape))
    gate, up, dout = (torch.randn(shape, device="cuda", generator=gen).half() * s for s in (4.0, 1.0, 0.01))
    special = torch.tensor([0.0, -0.0, 65504.0, -65504.0, float("inf"), float("-inf"), float("nan"), 6e-8, -88.0, 89.0, -20.0], device="cuda").half()
    k = min(gate.numel(), special.numel())
    gate.view(-1)[:k] = special[:k]
    assert quant_hip.silu_mul_takes(gate, up)
    g, u = gate.clone().requires_grad_(True), up.clone().requires_grad_(True)
    want = F.silu(g) * u
    want.backward(dout)
    _close(quant_hip.silu_mul(gate, up), want.detach())
    dg, du = quant_hip.silu_mul_bwd(dout, gate, up)
    _close(dg, g.grad)
    _close(du, u.grad)


def test_gated_block_trains_like_its_own_forward(oracle):
    """A block grouped by make_fused_mlp above the decode sizes: outputs and gradients of its own forward, also with an
    expanded output gradient, a hooked activation (own forward), a graph of the backward and checkpointing."""
    import torch
    import torch.nn as nn
    from torch.utils.checkpoint import checkpoint
    from conftest import rel_err, to_cuda_layer
    from alpaca_lora_4bit_amd import quant_hip
    from alpaca_lora_4bit_amd.autograd_4bit import Autograd4bitQuantLinear
    from alpaca_lora_4bit_amd.model_attn_mlp_patch import make_fused_mlp

    class Gated(nn.Module):
        def __init__(self):
            super().__init__()
            self.act_fn = nn.SiLU()

        def forward(self, x):
            return self.down_proj(self.act_fn(self.gate_proj(x)) * self.up_proj(x))

    H, I, gs, M = 256, 384, 128, 40
    blocks = []
    for _ in range(2):
        m = Gated()
        for i, (name, k, n) in enumerate((("gate_proj", H, I), ("up_proj", H, I), ("down_proj", I, H))):
            lin = Autograd4bitQuantLinear(k, n, groupsize=gs)
            for key, v in to_cuda_layer(oracle.make_layer(k, n, gs, seed=20 + i)).items():
                if isinstance(v, torch.Tensor):
                    setattr(lin, key, v)
            lin.bias = torch.zeros(n, dtype=torch.float16, device="cuda")
            setattr(m, name, lin)
        blocks.append(m)
    own, fused = blocks
    assert make_fused_mlp(fused) == 1
    xh = torch.from_numpy(oracle.make_activations(M, H, seed=4)).cuda()
    seen = []
    real = quant_hip.silu_mul

    def counted(*a):
        seen.append(1)
        return real(*a)
    quant_hip.silu_mul = counted
    try:
        def run(block, dy, wrap=None):
            x = xh.clone().requires_grad_(True)
            with torch.amp.autocast("cuda", dtype=torch.float16):
                y = block(x) if wrap is None else checkpoint(block, x, use_reentrant=False)
            y.backward(dy)
            return y.detach(), x.grad
        dense = torch.from_numpy(oracle.make_activations(M, H, seed=5)).cuda()
        for dy in (dense, torch.ones(1, 1, dtype=torch.float16, device="cuda").expand(M, H)):
            want = run(own, dy)
            assert not seen
            for wrap in (None, checkpoint):
                got = run(fused, dy, wrap)
                assert seen
                seen.clear()
                # the same sums over 256 and 384 products, from intermediates one fp16 rounding apart at most
                for a, b in zip(got, want):
                    assert rel_err(a.cpu().numpy(), b.double().cpu().numpy()) <= 3e-3
        with torch.no_grad():
            assert rel_err(fused(xh).cpu().numpy(), own(xh).double().cpu().numpy()) <= 3e-3 and seen
        seen.clear()
        handle = fused.act_fn.register_forward_hook(lambda *a: None)
        got = run(fused, dense)
        handle.remove()
        assert not seen and rel_err(got[1].cpu().numpy(), run(own, dense)[1].double().cpu().numpy()) <= 3e-3
        # second derivatives through the product of the two
        from alpaca_lora_4bit_amd.model_attn_mlp_patch import _SiluMul
        res = []
        for f in (_SiluMul.apply, lambda a, b: nn.functional.silu(a) * b):
            g = xh.clone().requires_grad_(True)
            u = dense.clone().requires_grad_(True)
            dg, = torch.autograd.grad(f(g, u).float().sum(), g, create_graph=True)
            res.append(torch.autograd.grad(dg.float().sum(), (g, u)))
        for a, b in zip(*res):
            assert torch.equal(a, b)
    finally:
        quant_hip.silu_mul = real


def test_silu_mul_has_the_bits_of_the_separate_operations():
    """Every fp16 value of gate with some of up and of the output gradient: the one pass forms the same fp32 expressions as torch's
    silu, silu_backward and products, so nothing but the sign and payload of a NaN may differ."""
    import torch
    import torch.nn.functional as F
    from alpaca_lora_4bit_amd import quant_hip
    gate = torch.arange(-2 ** 15, 2 ** 15, device="cuda", dtype=torch.int32).to(torch.int16).view(torch.float16).repeat(8, 1)
    gen = torch.Generator(device="cuda").manual_seed(11)
    up, dout = (torch.randn(gate.shape, device="cuda", generator=gen).half() for _ in range(2))
    dout *= 0.01
    g, u = gate.clone().requires_grad_(True), up.clone().requires_grad_(True)
    want = F.silu(g) * u
    want.backward(dout)
    dg, du = quant_hip.silu_mul_bwd(dout, gate, up)
    for got, ref in ((quant_hip.silu_mul(gate, up), want.detach()), (dg, g.grad), (du, u.grad)):
        num = ~torch.isnan(ref)
        assert torch.equal(torch.isnan(got), ~num) and torch.equal(got.view(torch.int16)[num], ref.view(torch.int16)[num])
