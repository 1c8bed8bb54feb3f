"""Fused MLP decode step (q4_mlp_decode_f16: gate|up -> silu * up -> down in one launch) vs the CPU oracle and vs
the three separate products.  Tolerance for y: max|y - ref| <= 1e-2 * max|ref| against the float64 result computed
from the oracle's dequantized weights with the intermediate rounded to fp16 where the unfused modules round it."""
import ctypes

import numpy as np
import pytest

from conftest import rel_err, to_cuda_layer

pytestmark = pytest.mark.gpu
TOL = 1e-2


def _layers(oracle, H, I, gs, seed):
    gate = oracle.make_layer(H, I, gs, seed=seed)
    up = oracle.make_layer(H, I, gs, seed=seed + 1)
    down = oracle.make_layer(I, H, gs, seed=seed + 2)
    return gate, up, down


def _dense(oracle, layer):
    return oracle.dequant_v2(layer["qweight"], layer["qzeros"], layer["scales"], layer["g_idx"]).astype(np.float64)


def _reference(oracle, x, gate, up, down):
    """float64 products; fp16 roundings of gate, up, silu(gate) and the product, as the modules apply them."""
    g = (x.astype(np.float64) @ _dense(oracle, gate)).astype(np.float16)
    u = (x.astype(np.float64) @ _dense(oracle, up)).astype(np.float16)
    g32 = g.astype(np.float32)
    h = (g32 / (1.0 + np.exp(-g32))).astype(np.float16)
    inter = (h.astype(np.float32) * u.astype(np.float32)).astype(np.float16)
    return g, u, inter, inter.astype(np.float64) @ _dense(oracle, down)


def _tuple(t):
    return (t["qweight"], t["qzeros"], t["scales"])


@pytest.mark.parametrize("H,I,gs", [(4096, 11008, 128), (256, 384, 128), (128, 128, 128), (512, 1408, 128),
                                    (1024, 2816, 256), (2048, 1024, 1024)])
@pytest.mark.parametrize("M", [1, 3, 4, 16])
def test_mlp_decode_matches_oracle_and_separate_products(oracle, H, I, gs, M):
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    gate, up, down = _layers(oracle, H, I, gs, seed=H + I + M)
    tg, tu, td = (to_cuda_layer(l) for l in (gate, up, down))
    x = oracle.make_activations(M, H, seed=M + 5)
    xt = torch.from_numpy(x).cuda()
    g_ref, u_ref, inter_ref, y_ref = _reference(oracle, x, gate, up, down)

    y, g, u = quant_hip.mlp_decode(xt, _tuple(tg), _tuple(tu), _tuple(td), gs, intermediates=True)
    assert y.shape == (M, H) and g.shape == (M, I) and u.shape == (M, I)
    assert rel_err(g.cpu().numpy(), g_ref.astype(np.float64)) <= 2e-3
    assert rel_err(u.cpu().numpy(), u_ref.astype(np.float64)) <= 2e-3
    assert rel_err(y.cpu().numpy(), y_ref) <= TOL, rel_err(y.cpu().numpy(), y_ref)
    assert rel_err(y.cpu().numpy(), y_ref) <= 3e-3

    # the two projections are the GEMV's values (the same bits when K is long enough for the same eight-wavefront
    # split, one fp16 rounding apart otherwise); the output agrees with the unfused chain
    g2 = quant_hip.gemv(xt, tg["qweight"], tg["qzeros"], tg["scales"], None, gs)
    u2 = quant_hip.gemv(xt, tu["qweight"], tu["qzeros"], tu["scales"], None, gs)
    if H >= 1024:
        assert torch.equal(g, g2) and torch.equal(u, u2)
    assert rel_err(g.cpu().numpy(), g2.float().cpu().numpy().astype(np.float64)) <= 1e-3
    assert rel_err(u.cpu().numpy(), u2.float().cpu().numpy().astype(np.float64)) <= 1e-3
    y2 = quant_hip.gemv(torch.nn.functional.silu(g2) * u2, td["qweight"], td["qzeros"], td["scales"], None, gs)
    assert rel_err(y.cpu().numpy(), y2.float().cpu().numpy().astype(np.float64)) <= 3e-3

    # every launch advances the ticket; results do not depend on it, with or without the intermediates
    for _ in range(4):
        assert torch.equal(y, quant_hip.mlp_decode(xt, _tuple(tg), _tuple(tu), _tuple(td), gs))
    assert not quant_hip.mlp_decode_gave_up()
    assert quant_hip.workspaces_are_zero()


def test_mlp_decode_many_launches_back_to_back_and_changing_inputs(oracle):
    """300 launches on one workspace without a synchronisation in between, inputs alternating between two tensors:
    a consumer never picks up a word of an earlier launch (the tag in the hand-over words) and the accumulators end
    at zero every time."""
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    H, I, gs = 1024, 2816, 128
    gate, up, down = _layers(oracle, H, I, gs, seed=77)
    tg, tu, td = (to_cuda_layer(l) for l in (gate, up, down))
    xs = [torch.from_numpy(oracle.make_activations(2, H, seed=s)).cuda() for s in (1, 2)]
    want = [quant_hip.mlp_decode(x, _tuple(tg), _tuple(tu), _tuple(td), gs).clone() for x in xs]
    for x, w in zip(xs, want):
        ref = _reference(oracle, x.cpu().numpy(), gate, up, down)[3]
        assert rel_err(w.cpu().numpy(), ref) <= 3e-3
    outs = [quant_hip.mlp_decode(xs[i & 1], _tuple(tg), _tuple(tu), _tuple(td), gs) for i in range(300)]
    torch.cuda.synchronize()
    for i, o in enumerate(outs):
        assert torch.equal(o, want[i & 1]), i
    assert not quant_hip.mlp_decode_gave_up()


def test_mlp_decode_through_the_c_abi_and_in_a_hip_graph(oracle):
    """Direct call of q4_mlp_decode_f16 with a caller-owned zeroed workspace; the same call captured in a HIP graph and
    replayed (the ticket lives in device memory, so replays of identical launch arguments still get fresh tags)."""
    import torch
    from alpaca_lora_4bit_amd import _lib, quant_hip
    H, I, gs, M = 512, 1408, 128, 4
    gate, up, down = _layers(oracle, H, I, gs, seed=5)
    tg, tu, td = (to_cuda_layer(l) for l in (gate, up, down))
    x = torch.from_numpy(oracle.make_activations(M, H, seed=9)).cuda()
    want = quant_hip.mlp_decode(x, _tuple(tg), _tuple(tu), _tuple(td), gs)
    L = _lib.lib()
    need = L.q4_mlp_decode_workspace_bytes(M, H, I)
    assert need >= 8 * M * (2 * I + H) + 8 * M * I
    ws = torch.zeros(need, dtype=torch.uint8, device="cuda")
    y = torch.empty(M, H, dtype=torch.float16, device="cuda")
    desc = [_lib.Layer(t["qweight"].data_ptr(), t["qzeros"].data_ptr(), t["scales"].data_ptr()) for t in (tg, tu, td)]

    def call(stream):
        return L.q4_mlp_decode_f16(x.data_ptr(), ctypes.byref(desc[0]), ctypes.byref(desc[1]), ctypes.byref(desc[2]), gs,
                                   None, None, y.data_ptr(), M, H, I, ws.data_ptr(), need, stream)

    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert call(side.cuda_stream) == 0
        side.synchronize()
        assert torch.equal(y, want)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            assert call(torch.cuda.current_stream().cuda_stream) == 0
            assert call(torch.cuda.current_stream().cuda_stream) == 0
    for _ in range(5):
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
    off = L.q4_mlp_decode_status_offset(M, H, I)
    assert int(ws[off:off + 4].view(torch.int32).item()) == 0
    # argument validation
    assert L.q4_mlp_decode_f16(x.data_ptr(), ctypes.byref(desc[0]), ctypes.byref(desc[1]), ctypes.byref(desc[2]), gs,
                               None, None, y.data_ptr(), M, H, I, ws.data_ptr(), need - 1, None) == -3
    assert L.q4_mlp_decode_f16(x.data_ptr(), ctypes.byref(desc[0]), ctypes.byref(desc[1]), ctypes.byref(desc[2]), 64,
                               None, None, y.data_ptr(), M, H, I, ws.data_ptr(), need, None) == -2
    assert L.q4_mlp_decode_f16(None, ctypes.byref(desc[0]), ctypes.byref(desc[1]), ctypes.byref(desc[2]), gs,
                               None, None, y.data_ptr(), M, H, I, ws.data_ptr(), need, None) == -1


@pytest.mark.parametrize("H,I,gs", [(128, 128, 128), (256, 384, 128), (1152, 640, 128), (1024, 2816, 256), (640, 1024, 1024), (4096, 11008, 128)])
@pytest.mark.parametrize("M", [1, 4, 5, 8, 9, 16])
def test_gate_up_launch_and_two_launch_step(oracle, H, I, gs, M):
    """q4_mlp_gate_up_f16 at the edges of its range (one chunk of the reduction, a last block of less than 8 chunks, a group
    beyond H, every number of outputs per thread) and quant_hip.mlp_rows_prepared, the step with down as its second launch."""
    import torch
    from alpaca_lora_4bit_amd import _lib, quant_hip
    gate, up, down = _layers(oracle, H, I, gs, seed=H + I + M)
    tg, tu, td = (to_cuda_layer(l) for l in (gate, up, down))
    x = oracle.make_activations(M, H, seed=M + 5)
    xt = torch.from_numpy(x).cuda()
    _, _, inter_ref, y_ref = _reference(oracle, x, gate, up, down)
    h = torch.full((M + 1, I), 7.0, dtype=torch.float16, device="cuda")            # one row beyond: stays as it is
    desc = [_lib.Layer(t["qweight"].data_ptr(), t["qzeros"].data_ptr(), t["scales"].data_ptr()) for t in (tg, tu)]
    L, stream = _lib.lib(), torch.cuda.current_stream().cuda_stream
    assert L.q4_mlp_gate_up_f16(xt.data_ptr(), ctypes.byref(desc[0]), ctypes.byref(desc[1]), gs, h.data_ptr(), M, H, I, stream) == 0
    assert bool((h[M] == 7.0).all())
    # gate and up are within one fp16 rounding (2^-11) of the reference's, |silu'| <= 1.1 and two more roundings follow
    assert rel_err(h[:M].cpu().numpy(), inter_ref.astype(np.float64)) <= 4.2 * 2.0 ** -11
    y = quant_hip.mlp_rows_prepared(xt, _tuple(tg), _tuple(tu), _tuple(td), gs, (1, M, H))
    assert y.shape == (1, M, H)
    assert rel_err(y[0].cpu().numpy(), y_ref) <= 3e-3
    assert torch.equal(y, quant_hip.mlp_rows_prepared(xt, _tuple(tg), _tuple(tu), _tuple(td), gs, (1, M, H)))
    assert quant_hip.workspaces_are_zero()
    for args, rc in (((xt.data_ptr(), 64, h.data_ptr(), M, H, I), -2), ((xt.data_ptr(), gs, h.data_ptr(), 17, H, I), -2),
                     ((None, gs, h.data_ptr(), M, H, I), -1), ((xt.data_ptr() + 2, gs, h.data_ptr(), M, H, I), -5)):
        assert L.q4_mlp_gate_up_f16(args[0], ctypes.byref(desc[0]), ctypes.byref(desc[1]), *args[1:], None) == rc


def test_mlp_block_above_four_rows_keeps_its_own_forward_where_it_must(oracle, monkeypatch):
    """5..16 rows take the fused step only when the block's forward is the gated expression and nobody watches its steps;
    replayed as a graph the step gives what it gives eagerly."""
    import torch
    import torch.nn as nn
    from alpaca_lora_4bit_amd import quant_hip
    from alpaca_lora_4bit_amd.autograd_4bit import Autograd4bitQuantLinear
    from alpaca_lora_4bit_amd.model_attn_mlp_patch import make_fused_mlp, ungroup

    class Gated(nn.Module):
        def __init__(self):
            super().__init__()
            self.act_fn = nn.SiLU()

        def forward(self, x):
            return self.down_proj(self.act_fn(self.gate_proj(x)) * self.up_proj(x))

    class Clamped(Gated):
        def forward(self, x):
            return self.down_proj(self.act_fn(self.gate_proj(x)).clamp(max=0.0) * self.up_proj(x))

    H, I, gs = 256, 384, 128
    layers = _layers(oracle, H, I, gs, seed=3)
    calls = []
    real = quant_hip.mlp_rows_prepared
    monkeypatch.setattr(quant_hip, "mlp_rows_prepared", lambda *a: (calls.append(1), real(*a))[1])

    def block(cls):
        m = cls()
        for name, layer in zip(("gate_proj", "up_proj", "down_proj"), layers):
            lin = Autograd4bitQuantLinear(layer["qweight"].shape[0] * 8, layer["qweight"].shape[1], groupsize=gs)
            for k, v in to_cuda_layer(layer).items():
                if isinstance(v, torch.Tensor):
                    setattr(lin, k, v)
            lin.bias = torch.zeros(lin.out_features, dtype=torch.float16, device="cuda")
            setattr(m, name, lin)
        return m

    with torch.no_grad():
        for M in (5, 16):
            x = torch.from_numpy(oracle.make_activations(M, H, seed=M)).cuda()
            for cls in (Gated, Clamped):
                m = block(cls)
                want = m(x)
                assert make_fused_mlp(m) == 1
                calls.clear()
                got = m(x)
                assert len(calls) == (cls is Gated)
                assert rel_err(got.cpu().numpy(), want.double().cpu().numpy()) <= 3e-3
                seen = []
                handle = m.act_fn.register_forward_hook(lambda *a: seen.append(1))
                m(x)
                handle.remove()
                assert len(seen) == 1 and len(calls) == (cls is Gated)
                if cls is Gated:
                    side = torch.cuda.Stream()
                    graph = torch.cuda.CUDAGraph()
                    with torch.cuda.stream(side):
                        m(x)
                        side.synchronize()
                        with torch.cuda.graph(graph, stream=side):
                            y = m(x)
                    for rep in range(4):
                        y.fill_(float("nan"))
                        (x.float() @ x.float().t()).sum().item()
                        torch.cuda.synchronize()
                        graph.replay()
                        torch.cuda.synchronize()
                        assert torch.equal(y, got)
                assert ungroup(m) == 1 and "_q4_mlp_gated" not in m.__dict__
    assert quant_hip.workspaces_are_zero()


@pytest.mark.parametrize("H,I,gs", [(256, 192, 128), (1024, 128, 128), (1152, 192, 384), (4096, 11008, 128), (5120, 13824, 128), (9216, 128, 1024),
                                    (2048, 16640, 128)])
@pytest.mark.parametrize("M", [1, 3, 4, 5, 8, 9, 16])
def test_gate_up_launch_has_the_bits_of_the_separate_calls(oracle, H, I, gs, M):
    """silu(gate) * up out of one launch against the two projections by themselves and torch's activation and product: one block
    of the reduction, a last block of one chunk, as many blocks as fit in LDS together and more, more strips than compute units."""
    import torch
    import torch.nn.functional as F
    from alpaca_lora_4bit_amd import _lib, quant_hip
    gen = torch.Generator(device="cuda").manual_seed(H + I + M)
    layers = []
    for _ in range(2):
        G = -(-H // gs)
        qweight = torch.randint(-2 ** 31, 2 ** 31 - 1, (H // 8, I), device="cuda", dtype=torch.int32, generator=gen)
        qzeros = torch.randint(-2 ** 31, 2 ** 31 - 1, (G, I // 8), device="cuda", dtype=torch.int32, generator=gen)
        layers.append((qweight, qzeros, (0.02 * torch.rand((G, I), device="cuda", generator=gen)).half()))
    x = torch.randn((M, H), device="cuda", generator=gen).half()
    gate, up = (quant_hip.gemv(x, *l, None, gs) for l in layers)
    h = torch.empty_like(gate)
    desc = [_lib.Layer(*(t.data_ptr() for t in l)) for l in layers]
    _lib.check(_lib.lib().q4_mlp_gate_up_f16(x.data_ptr(), ctypes.byref(desc[0]), ctypes.byref(desc[1]), gs, h.data_ptr(), M, H, I,
                                             torch.cuda.current_stream().cuda_stream), "q4_mlp_gate_up_f16")
    assert bool(torch.isfinite(gate).all()) and float(gate.abs().max()) > 1.0
    assert torch.equal(h, F.silu(gate) * up)
