"""The tiles of the GEMMs whose operands are built in registers (csrc/q4_gemm_wide.hip) at the edges of their pipeline: reductions
shorter than, equal to and just past the ring of activation tiles, ragged last row tiles of 256 and of 128 rows, groups of 64, 128 and 256 rows, adapters
of every number of 16-deep sub-steps in both types, with and without a dropout mask.
Tolerance: outputs are rounded to fp16 (2^-11 of a value), adapter matrices and their scaling too; sums of a few hundred such terms
average out to below 2e-3 of the largest output.  Weights are the dense kernel's, bit for bit."""
import numpy as np
import pytest

from conftest import rel_err, to_cuda_layer

pytestmark = pytest.mark.gpu
TOL = 2e-3


def _t(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _rows(M):
    return np.unique(np.minimum([0, 1, 31, 32, 127, 128, 255, 256, M - 2, M - 1], M - 1))


@pytest.mark.parametrize("red,gs,rank,f32", [(128, 128, 0, False), (128, 64, 8, True), (256, 64, 24, False), (384, 128, 0, True),
                                             (512, 256, 40, True), (640, 128, 64, False)])
@pytest.mark.parametrize("M", [130, 200, 256, 257, 300, 512])
def test_forward(oracle, M, red, gs, rank, f32):
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    N = 18432                                     # 72 column tiles: 144 tiles of 256 x 256 from 257 rows on, of 128 x 256 below
    layer = oracle.make_layer(red, N, gs, seed=red + gs)
    t = to_cuda_layer(layer)
    xh = oracle.make_activations(M, red, seed=M)
    bias = torch.randn(N, device="cuda", generator=torch.Generator("cuda").manual_seed(3)).half()
    xa = B = None
    if rank:
        A, B = oracle.make_lora(red, N, rank, seed=5)
        xa, B = quant_hip.lora_down(_t(xh), _t(A)), _t(B).to(torch.float32 if f32 else torch.float16)
    y = quant_hip.gemm_fwd(_t(xh), t["qweight"], t["qzeros"], t["scales"], None, gs, bias=bias, xa=xa,
                           lora_bt=None if B is None else B.t(), lora_scale=2.0)
    rows = _rows(M)
    ref = oracle.matmul_recons(xh[rows], layer["qweight"], layer["qzeros"], layer["scales"], layer["g_idx"]) + bias.float().cpu().numpy()
    if rank:
        ref = ref + 2.0 * xa.cpu().numpy()[rows].astype(np.float64) @ B.double().cpu().numpy().T
    assert y.shape == (M, N) and rel_err(y.cpu().numpy()[rows], ref) <= TOL
    # every row, against the float64 product with the dense weights
    W = quant_hip.dequant(t["qweight"], t["qzeros"], t["scales"], None, gs).double()
    full = _t(xh).double() @ W + bias.double()
    if rank:
        full += 2.0 * xa.double() @ B.double().t()
    assert float((y.double() - full).abs().max() / full.abs().max()) <= TOL


@pytest.mark.parametrize("red,gs,rank,f32,p", [(128, 128, 0, False, 0.0), (128, 64, 8, True, 0.1), (256, 64, 24, False, 0.0),
                                               (384, 128, 64, True, 0.5), (512, 256, 0, False, 0.0), (640, 128, 40, False, 0.05)])
@pytest.mark.parametrize("M", [257, 300, 512])
def test_grad_input(oracle, M, red, gs, rank, f32, p):
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    K = 18432
    layer = oracle.make_layer(K, red, gs, seed=red + gs)
    t = to_cuda_layer(layer)
    dyh = oracle.make_activations(M, red, seed=M)
    dyb = A = None
    if rank:
        A, B = oracle.make_lora(K, red, rank, seed=5)
        dyb, A = quant_hip.lora_down(_t(dyh), _t(B).t()), _t(A).to(torch.float32 if f32 else torch.float16)
    drop = (987654321 + M, p) if p else None
    dx = quant_hip.gemm_bwd_dx(_t(dyh), t["qweight"], t["qzeros"], t["scales"], None, gs, dyb=dyb, lora_a=A, lora_scale=2.0, dropout=drop)
    W = quant_hip.dequant(t["qweight"], t["qzeros"], t["scales"], None, gs).double()
    full = _t(dyh).double() @ W.t()
    term = None
    if rank:
        term = 2.0 * dyb.double() @ A.double()
        if p:
            keep, scale = oracle.dropout_keep_counter(M, K, drop[0], p)
            term = term * _t(keep).double() * scale
        full += term
    assert dx.shape == (M, K) and float((dx.double() - full).abs().max() / full.abs().max()) <= TOL
    rows = _rows(M)
    ref = oracle.matmul_recons_t(dyh[rows], layer["qweight"], layer["qzeros"], layer["scales"], layer["g_idx"])
    if rank:
        ref = ref + term.cpu().numpy()[rows]
    assert rel_err(dx.cpu().numpy()[rows], ref) <= TOL


# (forward?, rows, reduction, outputs, group size) of every kernel that multiplies fp16 weights:
ROUTES = [(True, 257, 128, 18432, 128), (True, 200, 128, 18432, 64),      # tiles of 256 x 256, of 128 x 256 with operands in registers
          (True, 600, 4096, 2048, 128),                                  # the latter with their reduction in five shares
          (True, 200, 128, 18560, 128), (True, 100, 4096, 1024, 64), (True, 128, 128, 18432, 64),    # 256 x 128, 128 x 128 (split, unsplit)
          (True, 17, 256, 8192, 128), (True, 48, 128, 18432, 128), (True, 150, 128, 4096, 128), (True, 300, 1024, 2048, 128),   # streaming
          (False, 257, 128, 18432, 128), (False, 200, 128, 18432, 128), (False, 200, 128, 18432, 64),
          (False, 600, 4096, 2048, 128), (False, 600, 1024, 2048, 64), (False, 100, 4096, 1024, 64), (False, 128, 128, 18432, 128)]


def _layer_of(codes, zero, gs, gen):
    """Tensors of a layer with these codes [K, N] and one zero code for all, and its weights rn16(rn16(s * code) - rn16(s * (zero + 1)))."""
    import torch
    K, N = codes.shape
    q = torch.zeros(K // 8, N, dtype=torch.int64, device="cuda")
    for e in range(8):
        q |= codes[e::8].long() << (4 * e)
    qweight = torch.where(q >= 2 ** 31, q - 2 ** 32, q).to(torch.int32)
    word = sum(zero << (4 * j) for j in range(8))
    qzeros = torch.full((K // gs, N // 8), word - 2 ** 32 if word >= 2 ** 31 else word, dtype=torch.int32, device="cuda")
    scales = (0.001 + 0.02 * torch.rand(K // gs, N, device="cuda", generator=gen)).half()
    s = scales.double().repeat_interleave(gs, 0)
    W = ((s * codes.double()).half().double() - (s * (zero + 1)).half().double()).half()
    return qweight, qzeros, scales, W


@pytest.mark.parametrize("z", range(16))
@pytest.mark.parametrize("route", ROUTES)
def test_every_code_and_zero(route, z):
    """A one-hot x reads single weights: every code of every zero point, in every nibble of a word, both directions, on every route.
    The weight has the three roundings of the dense kernel, bit for bit."""
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    fwd, M, red, out, gs = route
    gen = torch.Generator("cuda").manual_seed(z)
    codes = torch.randint(0, 16, (red, out) if fwd else (out, red), device="cuda", generator=gen)
    qweight, qzeros, scales, W = _layer_of(codes, z, gs, gen)
    assert torch.equal(quant_hip.dequant(qweight, qzeros, scales, None, gs), W)
    at = (torch.arange(M, device="cuda") * 37 + z) % red              # 37: every row of a word within 8 rows, every word within 128
    x = torch.zeros(M, red, dtype=torch.float16, device="cuda")
    x[torch.arange(M), at] = 1.0
    y = (quant_hip.gemm_fwd if fwd else quant_hip.gemm_bwd_dx)(x, qweight, qzeros, scales, None, gs)
    assert torch.equal(y, (W if fwd else W.t())[at])


@pytest.mark.parametrize("route", ROUTES)
def test_weights_at_their_zero_point_are_zero(route):
    """Columns (forward) or rows (grad-input) whose codes are all z + 1 give exactly the bias or zero, whatever the input's mean."""
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    fwd, M, red, out, gs = route
    gen = torch.Generator("cuda").manual_seed(M)
    codes = torch.randint(0, 16, (red, out) if fwd else (out, red), device="cuda", generator=gen)
    none = torch.arange(3, out, 7, device="cuda")
    if fwd:
        codes[:, none] = 8
    else:
        codes[none] = 8
    qweight, qzeros, scales, _ = _layer_of(codes, 7, gs, gen)
    x = (torch.randn(M, red, device="cuda", generator=gen) + 0.5).half()
    if fwd:
        bias = torch.randn(out, device="cuda", generator=gen).half()
        y = quant_hip.gemm_fwd(x, qweight, qzeros, scales, None, gs, bias=bias)
        assert torch.equal(y[:, none], bias[none].expand(M, -1))
    else:
        y = quant_hip.gemm_bwd_dx(x, qweight, qzeros, scales, None, gs)
        assert not y[:, none].any()
    assert float(y.double().abs().mean()) > 0.1
