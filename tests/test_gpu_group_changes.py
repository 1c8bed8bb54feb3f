"""Grouped projections and fused MLP blocks whose layers change between calls give what the same layers give ungrouped: what the
group and the block keep from one call to the next follows the tensors."""
import copy

import pytest

pytestmark = pytest.mark.gpu


def _close(a, b):
    """The same products, in groups or with the rows of an act-order layer sorted: sums in another order, one fp16 rounding apart."""
    from conftest import rel_err
    assert rel_err(a.float().cpu().numpy(), b.double().cpu().numpy()) <= 3e-3


def _mlp(oracle, H, I, gs):
    import torch
    import torch.nn as nn
    from conftest import to_cuda_layer
    from alpaca_lora_4bit_amd.autograd_4bit import Autograd4bitQuantLinear

    class Gated(nn.Module):
        def forward(self, x):
            return self.down_proj(self.act_fn(self.gate_proj(x)) * self.up_proj(x))

    m = Gated()
    m.act_fn = nn.SiLU()
    for i, (name, k, n) in enumerate((("gate_proj", H, I), ("up_proj", H, I), ("down_proj", I, H))):
        lin = Autograd4bitQuantLinear(k, n, groupsize=gs)
        for key, v in to_cuda_layer(oracle.make_layer(k, n, gs, seed=50 + i)).items():
            if isinstance(v, torch.Tensor):
                setattr(lin, key, v)
        lin.bias = torch.zeros(n, dtype=torch.float16, device="cuda")
        setattr(m, name, lin)
    return m


def _shuffled(g_idx):
    import torch
    return g_idx[torch.randperm(g_idx.numel(), generator=torch.Generator().manual_seed(9)).to(g_idx.device)]


def _change(block, what):
    """One change of one of the block's layers, the same for the grouped and the ungrouped block."""
    from alpaca_lora_4bit_amd import quant_hip
    layer, buffer, how = what
    m = getattr(block, layer)
    t = getattr(m, buffer)
    new = _shuffled(t) if buffer == "g_idx" else t * 0.5 if t.is_floating_point() else t.roll(1, -1)
    if how == "replaced":
        setattr(m, buffer, new)
    elif how == "written":
        t.copy_(new)
    else:                                                    # behind the version counter's back, and said so
        t.data.copy_(new)
        quant_hip.invalidate(m)


CHANGES = [(layer, buffer, how) for how in ("replaced", "written", "invalidated") for layer, buffer in
           (("down", "scales"), ("up", "qzeros"), ("gate", "scales"), ("down", "qweight"), ("up", "g_idx"), ("down", "g_idx"))]


@pytest.mark.parametrize("rows", [1, 8, 40])
@pytest.mark.parametrize("layer,buffer,how", CHANGES)
def test_mlp_step_follows_its_layers(oracle, rows, layer, buffer, how):
    import torch
    from alpaca_lora_4bit_amd.model_attn_mlp_patch import make_fused_mlp
    own = _mlp(oracle, 256, 384, 128)
    fused = copy.deepcopy(own)
    assert make_fused_mlp(fused) == 1
    x = torch.from_numpy(oracle.make_activations(rows, 256, seed=rows)).cuda()
    with torch.no_grad():
        before = own(x)
        _close(fused(x), before)
        for m in (own, fused):
            _change(m, (layer + "_proj", buffer, how))
        want = own(x)
        assert not torch.equal(want, before)
        _close(fused(x), want)


@pytest.mark.parametrize("rows,N", [(3, 512), (200, 4096)])
@pytest.mark.parametrize("layer,buffer,how", [("k", "qzeros", "replaced"), ("k", "qweight", "written"), ("v", "scales", "written"), ("q", "g_idx", "written"), ("v", "g_idx", "replaced"),
                                              ("k", "g_idx", "invalidated")])
def test_grouped_projections_follow_their_layers(oracle, rows, N, layer, buffer, how):
    """Also when a member changes after another of the group was called for the same input."""
    import torch
    from alpaca_lora_4bit_amd.model_attn_mlp_patch import make_quant_attn
    from test_gpu_gemm_grouped import _Block
    grouped, plain = (_Block(oracle, 1024, N, 128, 0.0, 70).eval() for _ in range(2))
    assert make_quant_attn(grouped) == 1
    x = torch.from_numpy(oracle.make_activations(rows, 1024, seed=rows)).cuda()
    others = [n for n in ("q_proj", "k_proj", "v_proj") if n != layer + "_proj"]
    with torch.no_grad():
        for a, b in zip(grouped(x), plain(x)):
            _close(a, b)
        _close(getattr(grouped, others[0])(x), getattr(plain, others[0])(x))
        for b in (grouped, plain):
            _change(b, (layer + "_proj", buffer, how))
        for name in (layer + "_proj", others[1], others[0]):
            _close(getattr(grouped, name)(x), getattr(plain, name)(x))


@pytest.mark.parametrize("matrix", ["lora_A", "lora_B"])
@pytest.mark.parametrize("how", ["storage", "invalidated", "version"])
def test_adapter_changed_between_two_members(oracle, matrix, how):
    """v's adapter is added together with q's; a change of it in between is followed."""
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    from alpaca_lora_4bit_amd.model_attn_mlp_patch import make_quant_attn
    from test_gpu_gemm_grouped import _Block
    grouped, plain = (_Block(oracle, 1024, 512, 128, 0.0, 80).eval() for _ in range(2))
    for b in (grouped, plain):
        b.v_proj.bias.zero_()
    assert make_quant_attn(grouped) == 1
    x = torch.from_numpy(oracle.make_activations(2, 1024, seed=8)).cuda()
    with torch.no_grad():
        _close(grouped.q_proj(x), plain.q_proj(x))
        for b in (grouped, plain):
            w = getattr(b.v_proj, matrix)["default"].weight
            if how == "storage":
                w.data = w.data * -3.0
            elif how == "version":
                w.mul_(-3.0)
            else:
                w.data.mul_(-3.0)
                quant_hip.invalidate(b.v_proj)
        _close(grouped.v_proj(x), plain.v_proj(x))


@pytest.mark.parametrize("rows,N", [(1, 512), (3, 512), (200, 4096)])
def test_grouped_blocks_under_inference_mode(oracle, rows, N):
    """Inference tensors have no version counter: members run by themselves, and a write to the input between them is followed."""
    import torch
    from alpaca_lora_4bit_amd.model_attn_mlp_patch import make_fused_mlp, make_quant_attn
    from test_gpu_gemm_grouped import _Block
    grouped, plain = (_Block(oracle, 1024, N, 128, 0.0, 90).eval() for _ in range(2))
    mlp = _mlp(oracle, 256, 384, 128)
    fused = copy.deepcopy(mlp)
    assert make_quant_attn(grouped) == 1 and make_fused_mlp(fused) == 1
    wide = copy.deepcopy(mlp)
    assert make_fused_mlp(wide, concatenate=True) == 1
    with torch.inference_mode():
        x = torch.from_numpy(oracle.make_activations(rows, 1024, seed=rows)).cuda()
        assert x.is_inference()
        for a, b in zip(grouped(x), plain(x)):
            _close(a, b)
        _close(grouped.q_proj(x), plain.q_proj(x))
        x.mul_(-2.0)
        _close(grouped.v_proj(x), plain.v_proj(x))
        _close(grouped.k_proj(x), plain.k_proj(x))
        y = x[:, :256].contiguous()
        _close(fused(y), mlp(y))
        _close(wide(y), mlp(y))


def _attention(oracle, rows, seed):
    import torch
    from alpaca_lora_4bit_amd.model_attn_mlp_patch import make_quant_attn
    from test_gpu_gemm_grouped import _Block
    grouped, plain = (_Block(oracle, 1024, 4096 if rows > 16 else 512, 128, 0.0, seed).eval() for _ in range(2))
    for b in (grouped, plain):
        b.v_proj.bias.zero_()
    assert make_quant_attn(grouped) == 1
    x = torch.from_numpy(oracle.make_activations(rows, 1024, seed=seed)).cuda()
    with torch.no_grad():
        want = plain(x)
        for a, b in zip(grouped(x), want):
            _close(a, b)
    torch.cuda.synchronize()
    return grouped, x, want


@pytest.mark.parametrize("rows", [3, 200])
def test_members_called_on_another_stream(oracle, rows):
    """q is queued behind other work of one stream; k and v, called on another one meanwhile, do not take what is not there yet."""
    import torch
    grouped, x, want = _attention(oracle, rows, 110)
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.no_grad():
        with torch.cuda.stream(first):
            torch.cuda._sleep(100_000_000)                   # some tens of milliseconds
            q = grouped.q_proj(x)
        with torch.cuda.stream(second):
            v, k = grouped.v_proj(x).clone(), grouped.k_proj(x).clone()
            second.synchronize()
            assert not first.query()
        first.synchronize()
        for a, b in zip((q, k, v), want):
            _close(a, b)


@pytest.mark.parametrize("rows", [3, 200])
def test_members_called_after_a_capture_that_left_them(oracle, rows):
    """What a capture queued was not computed: an eager call on the same stream and input computes its own."""
    import torch
    grouped, x, want = _attention(oracle, rows, 120)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.stream(stream):
        grouped(x)
        stream.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            q = grouped.q_proj(x)
        k = grouped.k_proj(x)
        stream.synchronize()
        _close(k, want[1])
        for _ in range(3):
            q.fill_(float("nan"))
            graph.replay()
            stream.synchronize()
            _close(q, want[0])


@pytest.mark.parametrize("rows", [3, 200])
def test_members_called_from_two_threads(oracle, rows):
    """Two threads with inputs of their own, and one input, call the members of one group in turn."""
    import threading
    import torch
    grouped, x, want = _attention(oracle, rows, 130)
    other = torch.from_numpy(oracle.make_activations(rows, 1024, seed=131)).cuda()
    with torch.no_grad():
        want_other = grouped(other)
    torch.cuda.synchronize()
    failed, barrier = [], threading.Barrier(2, timeout=60)

    def work(t, results):
        try:
            with torch.no_grad():
                for rep in range(40):
                    inp, ref = results[rep % len(results)]
                    for name, r in zip(("q_proj", "k_proj", "v_proj"), ref):
                        if rep % 2:
                            barrier.wait()
                        _close(getattr(grouped, name)(inp), r)
        except BaseException as e:                           # noqa: B902
            failed.append(e)
            barrier.abort()
    threads = [threading.Thread(target=work, args=(t, ((x, want), (other, want_other))[::1 - 2 * t])) for t in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed[0]
