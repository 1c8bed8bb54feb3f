"""Grouped GEMMs (q4_gemm_grouped_fwd_f16 / q4_gemm_grouped_bwd_dx_f16: q|k|v or gate|up of a block in one launch on the
layers' own tensors) against the CPU oracle and against the per-layer entry points.  Tolerance 1e-2 * max|ref|."""
import numpy as np
import pytest

from conftest import rel_err, to_cuda_layer

pytestmark = pytest.mark.gpu
TOL = 1e-2


def _t(a):
    import torch
    return torch.from_numpy(a).cuda()


@pytest.mark.parametrize("M,K,Ns,gs,lora", [
    (1024, 4096, (4096, 4096, 4096), 128, (8, 0, 8)),          # q|k|v of config 4: 192 wide tiles, adapters on q and v
    (1024, 4096, (11008, 11008), 128, (0, 0)),                 # gate|up of config 4
    (600, 1024, (4096, 2048, 1024, 2048), 256, (16, 8, 0, 0)),  # four layers, ragged rows, 24 narrow tiles in eight shares, some across layers
    (2048, 512, (4096, 4096), 64, (0, 8)),                     # groups of 64 rows
])
def test_grouped_forward_and_grad_input(oracle, M, K, Ns, gs, lora):
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    assert quant_hip.gemm_grouped_applicable(True, M, K, Ns) and quant_hip.gemm_grouped_applicable(False, M, K, Ns)
    layers = [oracle.make_layer(K, N, gs, seed=K + N + i) for i, N in enumerate(Ns)]
    ts = [to_cuda_layer(l) for l in layers]
    xh = oracle.make_activations(M, K, seed=M)
    x = _t(xh)
    rng = np.random.default_rng(M + K)
    biases, As, Bs, xas = [], [], [], []
    for i, (N, r) in enumerate(zip(Ns, lora)):
        biases.append(torch.randn(N, device="cuda").half() if i % 2 == 0 else None)
        if r:
            A, B = oracle.make_lora(K, N, r, seed=i + 1)
            As.append(_t(A)); Bs.append(_t(B))
            xas.append(quant_hip.lora_down(x, As[-1]))
        else:
            As.append(None); Bs.append(None); xas.append(None)
    fwd_layers = [(t["qweight"], t["qzeros"], t["scales"], b, xa, None if B is None else B.t(), 2.0)
                  for t, b, xa, B in zip(ts, biases, xas, Bs)]
    ys = quant_hip.gemm_grouped_fwd(x, fwd_layers, gs)
    ys2 = quant_hip.gemm_grouped_fwd(x, fwd_layers, gs)
    rows = np.array([0, 1, M // 2, M - 1])
    for i, (lay, t, y) in enumerate(zip(layers, ts, ys)):
        assert y.shape == (M, Ns[i]) and torch.equal(y, ys2[i])
        single = quant_hip.gemm_fwd(x, t["qweight"], t["qzeros"], t["scales"], None, gs, bias=biases[i], xa=xas[i],
                                    lora_bt=None if Bs[i] is None else Bs[i].t(), lora_scale=2.0)
        assert float((y.float() - single.float()).abs().max() / single.float().abs().max()) <= 2e-3
        ref = oracle.matmul_recons(xh[rows], lay["qweight"], lay["qzeros"], lay["scales"], lay["g_idx"])
        if biases[i] is not None:
            ref = ref + biases[i].float().cpu().numpy()
        if lora[i]:
            ref = ref + 2.0 * (xas[i].float().cpu().numpy()[rows].astype(np.float64) @ Bs[i].half().float().cpu().numpy().astype(np.float64).T)
        assert rel_err(y.cpu().numpy()[rows], ref) <= 2e-3

    dyhs = [oracle.make_activations(M, N, seed=M + 7 + i) for i, N in enumerate(Ns)]
    dys = [_t(d) for d in dyhs]
    dybs = [None if B is None else quant_hip.lora_down(dy, B.t()) for dy, B in zip(dys, Bs)]
    for drops in ([None] * len(Ns), [(77 + i, 0.1) if lora[i] else None for i in range(len(Ns))]):
        bwd_layers = [(t["qweight"], t["qzeros"], t["scales"], dyb, A, 2.0, dr) for t, dyb, A, dr in zip(ts, dybs, As, drops)]
        dx = quant_hip.gemm_grouped_bwd_dx(dys, bwd_layers, gs)
        assert dx.shape == (M, K) and torch.equal(dx, quant_hip.gemm_grouped_bwd_dx(dys, bwd_layers, gs))
        want = torch.zeros(M, K, device="cuda")
        for t, dy, dyb, A, dr in zip(ts, dys, dybs, As, drops):
            want += quant_hip.gemm_bwd_dx(dy, t["qweight"], t["qzeros"], t["scales"], None, gs, dyb=dyb, lora_a=A, lora_scale=2.0,
                                          dropout=dr).float()
        assert float((dx.float() - want).abs().max() / want.abs().max()) <= 2e-3
        if drops[0] is None and not any(drops):
            ref = np.zeros((len(rows), K))
            for lay, dyh, dyb, A in zip(layers, dyhs, dybs, As):
                ref += oracle.matmul_recons_t(dyh[rows], lay["qweight"], lay["qzeros"], lay["scales"], lay["g_idx"])
                if A is not None:
                    ref += 2.0 * (dyb.float().cpu().numpy()[rows].astype(np.float64) @ A.half().float().cpu().numpy().astype(np.float64))
            assert rel_err(dx.cpu().numpy()[rows], ref) <= 2e-3


def test_grouped_gemm_refuses_what_it_does_not_take(oracle):
    import ctypes
    import torch
    from alpaca_lora_4bit_amd import _lib, quant_hip
    assert not quant_hip.gemm_grouped_applicable(True, 128, 4096, (4096, 4096, 4096))      # 128 rows: the per-layer kernels
    assert not quant_hip.gemm_grouped_applicable(True, 1024, 4096, (4096,))                # one layer is not a group
    assert not quant_hip.gemm_grouped_applicable(True, 256, 1024, (128, 128))              # too few tiles for a launch
    assert not quant_hip.gemm_grouped_applicable(False, 1024, 4096 + 64, (4096, 4096))
    L = _lib.lib()
    lay = to_cuda_layer(oracle.make_layer(256, 128, 128, seed=1))
    x = torch.zeros(256, 256, device="cuda", dtype=torch.float16)
    y = torch.zeros(256, 128, device="cuda", dtype=torch.float16)
    desc = (_lib.GemmLayer * 2)()
    for d in desc:
        d.act, d.qweight, d.qzeros, d.scales, d.out, d.N = (x.data_ptr(), lay["qweight"].data_ptr(), lay["qzeros"].data_ptr(),
                                                            lay["scales"].data_ptr(), y.data_ptr(), 128)
    assert L.q4_gemm_grouped_fwd_f16(desc, 2, 128, 256, 256, None) == -2                   # not enough tiles
    assert L.q4_gemm_grouped_fwd_f16(None, 2, 128, 256, 256, None) == -1
    assert L.q4_gemm_grouped_bwd_dx_f16(desc, 2, 128, None, 256, 256, None, 0, None) == -1


class _Block:
    """Stands for an attention block: three projections of one input, two of them with LoRA adapters."""

    def __new__(cls, oracle, K, N, gs, dropout, seed):
        import torch
        import torch.nn as nn
        from alpaca_lora_4bit_amd import autograd_4bit as ag, models

        class Block(nn.Module):
            def __init__(self):
                super().__init__()
                for i, name in enumerate(("q_proj", "k_proj", "v_proj")):
                    lay = oracle.make_layer(K, N, gs, seed=seed + i)
                    if name == "k_proj":
                        m = ag.Autograd4bitQuantLinear(K, N, groupsize=gs)
                    else:
                        m = models.Linear4bitLt("default", K, N, gs, False, r=8, lora_alpha=16, lora_dropout=dropout)
                        A, B = oracle.make_lora(K, N, 8, seed=seed + 10 + i)
                        m.lora_A["default"].weight.data = torch.from_numpy(A)
                        m.lora_B["default"].weight.data = torch.from_numpy(B)
                    m.qweight.data = torch.from_numpy(lay["qweight"])
                    m.qzeros.data = torch.from_numpy(lay["qzeros"])
                    m.scales = torch.from_numpy(lay["scales"])
                    m.g_idx.data = torch.from_numpy(lay["g_idx"])
                    m.bias = torch.zeros(N, dtype=torch.float16) if name != "v_proj" else (torch.arange(N) % 7 - 3).half() * 0.25
                    setattr(self, name, m)

            def forward(self, x):
                return self.q_proj(x), self.k_proj(x), self.v_proj(x)
        return Block().cuda()


@pytest.mark.parametrize("dropout", [0.0, 0.1])
def test_grouped_block_matches_the_ungrouped_block_forward_and_gradients(oracle, dropout, monkeypatch):
    """make_quant_attn on a block above the decode sizes: q|k|v (LoRA on q and v, a bias on v) run as ONE grouped
    forward launch and, in backward, ONE grouped grad-input launch.  Outputs, grad_input and adapter gradients
    against the same block ungrouped (whose layers are held to the oracle in test_gpu_autograd.py); with adapter
    dropout both draw their mask seeds in the same order, so the masks are the same."""
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    from alpaca_lora_4bit_amd.model_attn_mlp_patch import make_quant_attn, ungroup
    K, N, gs, M = 1024, 4096, 128, 512
    grouped, plain = _Block(oracle, K, N, gs, dropout, 40), _Block(oracle, K, N, gs, dropout, 40)
    assert make_quant_attn(grouped) == 1
    grouped.train(); plain.train()
    calls = {"fwd": 0, "bwd": 0}
    for name, key in (("gemm_grouped_fwd", "fwd"), ("gemm_grouped_bwd_dx", "bwd")):
        real = getattr(quant_hip, name)
        monkeypatch.setattr(quant_hip, name, (lambda real, key: lambda *a, **k: (calls.__setitem__(key, calls[key] + 1), real(*a, **k))[1])(real, key))
    xh = oracle.make_activations(M, K, seed=3)
    gys = [_t(oracle.make_activations(M, N, seed=4 + i)).view(2, M // 2, N) for i in range(3)]
    results = []
    for block in (grouped, plain):
        torch.manual_seed(1234)
        x = _t(xh).view(2, M // 2, K).requires_grad_(True)
        with torch.amp.autocast(device_type="cuda", dtype=torch.float16):
            ys = block(x)
        torch.autograd.backward(ys, gys)
        grads = [p.grad.clone() for p in block.parameters() if p.requires_grad]
        results.append(([y.detach() for y in ys], x.grad.clone(), grads))
        block.zero_grad()
    assert calls == {"fwd": 1, "bwd": 1}
    (ys_g, dx_g, gr_g), (ys_p, dx_p, gr_p) = results
    for a, b in zip(ys_g, ys_p):
        assert a.shape == (2, M // 2, N)
        assert float((a.float() - b.float()).abs().max() / b.float().abs().max()) <= 2e-3
    assert float((dx_g.float() - dx_p.float()).abs().max() / dx_p.float().abs().max()) <= 3e-3
    assert len(gr_g) == 4
    for a, b in zip(gr_g, gr_p):
        assert float((a.float() - b.float()).abs().max() / b.float().abs().max()) <= 3e-3
    # no grad, eval: the same grouped launch for a prefill-sized input; 8 rows go to the grouped GEMV
    grouped.eval(); plain.eval()
    with torch.no_grad():
        for rows in (M, 8):
            x = _t(xh)[:rows]
            for a, b in zip(grouped(x), plain(x)):
                assert float((a.float() - b.float()).abs().max() / b.float().abs().max()) <= 2e-3
    assert calls["fwd"] == 2
    assert ungroup(grouped) == 1 and "_q4_group" not in grouped.k_proj.__dict__


@pytest.mark.parametrize("K,N,M,streams", [(4096, 4096, 200, True),        # 96 tiles, one row tile, all three layers stream
                                           (1024, 5120, 200, False)])      # 120 tiles, too many strips to stream at this many rows
def test_one_row_tile_is_grouped_by_what_there_is_to_train(oracle, K, N, M, streams, monkeypatch):
    """129..256 rows of q|k|v: one grouped launch when something needs a gradient, when an adapter rides along or when the
    layers have no streaming kernel of their own; a forward alone of layers that stream stays with them, whether or not
    gradients are switched on.  Values and gradients against the block without grouping in every case."""
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    from alpaca_lora_4bit_amd.model_attn_mlp_patch import make_quant_attn
    grouped, plain = _Block(oracle, K, N, 128, 0.0, 60), _Block(oracle, K, N, 128, 0.0, 60)
    assert make_quant_attn(grouped) == 1
    assert quant_hip.streams_forward(M, K, (N, N, N), 128) == streams
    count = {"fwd": 0, "bwd": 0}
    for name, key in (("gemm_grouped_fwd", "fwd"), ("gemm_grouped_bwd_dx", "bwd")):
        real = getattr(quant_hip, name)
        monkeypatch.setattr(quant_hip, name, (lambda real, key: lambda *a, **k: (count.__setitem__(key, count[key] + 1), real(*a, **k))[1])(real, key))
    xh, gys = oracle.make_activations(M, K, seed=5), [_t(oracle.make_activations(M, N, seed=6 + i)) for i in range(3)]

    def compare(grad_mode, x_needs_grad, want_fwd, want_bwd):
        count.update(fwd=0, bwd=0)
        results = []
        for block in (grouped, plain):
            block.zero_grad()
            x = _t(xh).requires_grad_(x_needs_grad)
            with torch.set_grad_enabled(grad_mode):
                ys = block(x)
            if any(y.requires_grad for y in ys):
                torch.autograd.backward([y for y in ys if y.requires_grad], [g for y, g in zip(ys, gys) if y.requires_grad])
            results.append([y.detach() for y in ys] + [g for g in [x.grad] + [p.grad for p in block.parameters() if p.requires_grad] if g is not None])
        assert count == {"fwd": want_fwd, "bwd": want_bwd}
        assert len(results[0]) == len(results[1])
        for a, b in zip(*results):
            assert float((a.float() - b.float()).abs().max() / b.float().abs().max()) <= 3e-3

    compare(True, True, 1, 1)                          # training: grad_input and the adapters
    compare(True, False, 1, 0)                         # the first block: adapters only
    compare(False, False, 1, 0)                        # inference with the adapters
    for block in (grouped, plain):
        for m in (block.q_proj, block.v_proj):
            for p in list(m.lora_A.parameters()) + list(m.lora_B.parameters()):
                p.requires_grad_(False)
    compare(True, False, 1, 0)                         # frozen adapters still ride in the launch
    for block in (grouped, plain):
        for m in (block.q_proj, block.v_proj):
            m.enable_adapters(False)
    alone = 0 if streams else 1
    compare(True, True, 1, 1)
    compare(True, False, alone, 0)                     # an evaluation that left gradients on
    compare(False, False, alone, 0)


def _dense(quant_hip, t, gs):
    return quant_hip.dequant(t["qweight"], t["qzeros"], t["scales"], t["g_idx"], gs).float()


@pytest.mark.parametrize("M,K,Ns,gs,r,p,bare,splits,tail_cols", [
    (200, 4096, (256, 384), 128, 8, 0.05, 1, 1, 0),                    # 10 steps in all, walked whole
    (1000, 4096, (1024, 640, 512), 64, 16, 0.05, 1, 1, 0),             # ragged rows, walked whole, no scale / zero table
    (200, 4096, (2048, 1152, 1024), 128, 8, 0.05, 1, 6, 0),            # layers begin at steps 32 and 50, shares at multiples of 11
    (200, 4096, (2048, 1152, 1024), 64, 16, 0.0, None, 6, 0),          # the same without the table, every layer with an adapter
    (1000, 4096, (2048, 1152, 640), 64, 16, 0.05, 0, 2, 0),            # the second share begins in layer 0 and holds 1 and 2 whole
    (4500, 4096, (512, 256), 128, 8, 0.1, 1, 1, 4),                    # 288 wide tiles: whole rounds and a remainder launch
    (4500, 4096, (2048, 640), 128, 8, 0.1, None, 3, 4),                # its reduction in three shares, the last across both layers
    (4500, 4096, (1152, 640), 128, 8, 0.0, None, 2, 4),                # unmasked adapters on the wide layer walk and on two shares
    (300, 384, (1024, 1024), 128, 0, 0.0, None, 4, 0),                 # K not a multiple of 256: narrow tiles only
])
def test_grouped_grad_input_is_one_reduction_over_the_layers(oracle, M, K, Ns, gs, r, p, bare, splits, tail_cols):
    """dx over the concatenated reduction (adapter terms and their dropout masks included) against fp32 products with
    the bit-exact dense weights.  Bound: inputs and weights are the same fp16 values on both sides, so what differs is the
    fp16 rounding of the result (2^-11), of the scaled adapter matrix (2^-11 of the smaller adapter term) and the order
    of the 32-bit sums: 2e-3 of the largest value (an adapter term left out or counted twice is 10 to 40 times that).
    The scratch query shows that the plan is the one the case stands for: `splits` shares of the whole output, or of the
    last `tail_cols` column tiles.  `bare`: the layer without an adapter."""
    import ctypes
    import torch
    from alpaca_lora_4bit_amd import _lib, quant_hip
    scratch = splits * M * (tail_cols * 128 or K) * 4 if splits > 1 else 0
    assert _lib.lib().q4_gemm_grouped_workspace_bytes(0, len(Ns), M, K, (ctypes.c_int * len(Ns))(*Ns)) == scratch
    ts = [to_cuda_layer(oracle.make_layer(K, N, gs, seed=K + N + i)) for i, N in enumerate(Ns)]
    g = torch.Generator(device="cuda").manual_seed(M)
    dys, layers, ref = [], [], 0.0
    for i, (t, N) in enumerate(zip(ts, Ns)):
        dy = torch.randn((M, N), device="cuda", generator=g).half()
        dyb = A = drop = None
        ref = ref + dy.float() @ _dense(quant_hip, t, gs).t()
        if r and i != bare:
            A = torch.randn((r, K), device="cuda", generator=g) * 0.05
            dyb = torch.randn((M, r), device="cuda", generator=g).half()
            term = 2.0 * (dyb.float() @ A)
            if p:
                drop = (77 + i, p)
                term = term * quant_hip.dropout_keep_mask(M, K, 77 + i, p, dy.device).float() * quant_hip.dropout_scale(p)
            ref = ref + term
        dys.append(dy)
        layers.append((t["qweight"], t["qzeros"], t["scales"], dyb, A, 2.0 if A is not None else 1.0, drop))
    dx = quant_hip.gemm_grouped_bwd_dx(dys, layers, gs)
    assert float((dx.float() - ref).abs().max() / ref.abs().max()) <= 2e-3
    assert torch.equal(dx, quant_hip.gemm_grouped_bwd_dx(dys, layers, gs))


def test_grouped_forward_remainder_launch(oracle):
    """344 wide tiles: 256 of them as they are, the columns left over (inside the second layer) as 256 x 128 tiles."""
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    M, K, Ns = 1000, 512, (11008, 11008)
    ts = [to_cuda_layer(oracle.make_layer(K, N, 128, seed=N + i)) for i, N in enumerate(Ns)]
    x = torch.randn((M, K), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1)).half()
    bias = [None, torch.randn(Ns[1], device="cuda").half()]
    ys = quant_hip.gemm_grouped_fwd(x, [(t["qweight"], t["qzeros"], t["scales"], b, None, None, 1.0) for t, b in zip(ts, bias)], 128)
    for t, b, y in zip(ts, bias, ys):
        ref = x.float() @ _dense(quant_hip, t, 128) + (0.0 if b is None else b.float())
        assert float((y.float() - ref).abs().max() / ref.abs().max()) <= 2e-3


@pytest.mark.parametrize("M,red,nout,gs,act,tail_cols,splits", [
    (2000, 512, 11008, 128, False, 22, 1),      # 8 x 43 wide tiles: 11 columns left, one round of narrow tiles
    (2000, 512, 11008, 64, False, 22, 1),
    (4500, 1536, 4096, 128, True, 4, 3),        # 18 x 32 narrow tiles (indexed groups): 4 columns left, reduction split
    (4096, 2048, 5120, 256, False, 8, 2),       # 16 x 20: 4 columns left (64 tiles)
])
def test_wide_tiles_with_a_remainder_launch(oracle, M, red, nout, gs, act, tail_cols, splits):
    """Forward (bias, adapter) and grad-input (adapter with dropout) where the last columns are a launch of narrow tiles."""
    import torch
    from alpaca_lora_4bit_amd import _lib, quant_hip
    r = 8
    for fwd in (True, False):
        K, N = (red, nout) if fwd else (nout, red)
        want = splits * M * tail_cols * 128 * 4 if splits > 1 else 0
        assert _lib.lib().q4_gemm_workspace_bytes(int(fwd), M, K, N) == want
        t = to_cuda_layer(oracle.make_layer(K, N, gs, act_order=act, seed=M))
        W = _dense(quant_hip, t, gs)
        g = torch.Generator(device="cuda").manual_seed(M)
        A, B = (torch.randn(s, device="cuda", generator=g) * 0.05 for s in ((r, K), (N, r)))
        a = torch.randn((M, red), device="cuda", generator=g).half()
        small = torch.randn((M, r), device="cuda", generator=g).half()
        if fwd:
            bias = torch.randn(N, device="cuda", generator=g).half()
            got = quant_hip.gemm_fwd(a, t["qweight"], t["qzeros"], t["scales"], t["g_idx"] if act else None, gs, bias=bias,
                                     xa=small, lora_bt=B.t(), lora_scale=2.0)
            ref = a.float() @ W + bias.float() + 2.0 * (small.float() @ B.t())
        else:
            drop = None if act else (5, 0.1)
            got = quant_hip.gemm_bwd_dx(a, t["qweight"], t["qzeros"], t["scales"], t["g_idx"] if act else None, gs, dyb=small,
                                        lora_a=A, lora_scale=2.0, dropout=drop)
            term = 2.0 * (small.float() @ A)
            if drop:
                term = term * quant_hip.dropout_keep_mask(M, K, 5, 0.1, a.device).float() * quant_hip.dropout_scale(0.1)
            ref = a.float() @ W.t() + term
        assert float((got.float() - ref).abs().max() / ref.abs().max()) <= 2e-3
