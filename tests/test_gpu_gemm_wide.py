"""The tiles of the GEMMs whose operands are built in registers (csrc/q4_gemm_wide.hip) at the edges of their pipeline: reductions
shorter than, equal to and just past the ring of activation tiles, ragged last row tiles of 256 and of 128 rows, groups of 64, 128 and 256 rows, adapters
of every number of 16-deep sub-steps in both types, with and without a dropout mask.
Tolerance: outputs are rounded to fp16 (2^-11 of a value) and weights to fp16 twice (together at most 2^-10 of the largest
|scale * code|, about twice the largest weight); sums of a few hundred such terms average out to below 2e-3 of the largest output."""
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


@pytest.mark.parametrize("z", range(16))
def test_every_code_and_zero(z):
    """A one-hot x reads single weights: every code of every zero point, in every nibble of a word, both directions.  The weight
    is rn(scale * code - rn(scale * (zero + 1))), off by half a unit in the last place of each of the two roundings."""
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    gs, D, M = 64, 18432, 257
    gen = torch.Generator("cuda").manual_seed(z)
    for fwd in (True, False):
        K, N = (128, D) if fwd else (D, 128)
        codes = torch.randint(0, 16, (K // 8, 8, N), device="cuda", generator=gen)
        q = torch.zeros(K // 8, N, dtype=torch.int64, device="cuda")
        for e in range(8):
            q |= codes[:, e] << (4 * e)
        qweight = torch.where(q >= 2 ** 31, q - 2 ** 32, q).to(torch.int32)
        word = sum(z << (4 * j) for j in range(8))
        qzeros = torch.full((K // gs, N // 8), word - 2 ** 32 if word >= 2 ** 31 else word, dtype=torch.int32, device="cuda")
        scales = (0.001 + 0.02 * torch.rand(K // gs, N, device="cuda", generator=gen)).half()
        s = scales.double().repeat_interleave(gs, 0)
        zt = (s * (z + 1)).half().double()
        W = (s * codes.reshape(K, N).double() - zt).half()
        x = torch.zeros(M, 128, dtype=torch.float16, device="cuda")
        x[torch.arange(M), torch.arange(M) % 128] = 1.0
        y = (quant_hip.gemm_fwd if fwd else quant_hip.gemm_bwd_dx)(x, qweight, qzeros, scales, None, gs)
        assert torch.equal(y, (W if fwd else W.t())[torch.arange(M, device="cuda") % 128])
