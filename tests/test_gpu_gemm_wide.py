"""The tiles of the GEMMs whose operands are built in registers (csrc/q4_gemm_wide.hip) at the edges of their pipeline: shares of the
reduction shorter than the ring of activation tiles and of every length modulo its four steps, ragged last row tiles of 256 and of 128 rows,
groups of 64, 128 and 256 rows, adapters of every number of 16-deep sub-steps in both types, with and without a dropout mask.
Tolerance: outputs are rounded to fp16 (2^-11 of a value), adapter matrices and their scaling too; sums of a few hundred such terms
average out to below 2e-3 of the largest output.  Weights are the dense kernel's, bit for bit."""
import numpy as np
import pytest

from conftest import rel_err, to_cuda_layer
from test_gemm_plan import _group_plan, _plan, plans  # noqa: F401

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


def _indexed(fwd, x, layer, gs, out_cols, bias=None, la=None, lb=None, drop=None):
    """The same product by the kernels that look every row's group up (csrc/q4_gemm.hip)."""
    import ctypes
    import torch
    from alpaca_lora_4bit_amd import _lib, quant_hip
    L = _lib.lib()
    qweight, qzeros, scales = layer
    K, N, M = 8 * qweight.shape[0], qweight.shape[1], x.shape[0]
    g_idx = (torch.arange(K, device="cuda") // gs).to(torch.int32)
    out = torch.empty(M, out_cols, dtype=torch.float16, device="cuda")
    need = L.q4_gemm_workspace_bytes(int(fwd), M, K, N)
    ws = torch.empty(max(need, 256), dtype=torch.uint8, device="cuda")
    lora = (None, None, 0, 0, 0, 0.0, 0) if la is None else (la.data_ptr(), lb.data_ptr(), lb.stride(0), lb.stride(1),
                                                             int(lb.dtype == torch.float32), 2.0, la.shape[1])
    common = (x.data_ptr(), qweight.data_ptr(), qzeros.data_ptr(), scales.data_ptr(), g_idx.data_ptr(), gs)
    tail = (out.data_ptr(), M, K, N, K // gs)
    stream = torch.cuda.current_stream().cuda_stream
    if fwd:
        rc = L.q4_gemm_fwd_f16(*common, None if bias is None else bias.data_ptr(), *lora, *tail, ws.data_ptr(), ws.numel(), stream)
    else:
        d = quant_hip._drop_arg(drop)
        rc = L.q4_gemm_bwd_dx_f16(*common, *lora, *tail, quant_hip._drop_ref(d), ws.data_ptr(), ws.numel(), stream)
    torch.cuda.synchronize()
    assert rc == 0
    return out


def _random_layer(K, N, gs, gen):
    import torch
    qweight = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 8, N), device="cuda", dtype=torch.int32, generator=gen)
    qzeros = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // gs, N // 8), device="cuda", dtype=torch.int32, generator=gen)
    return qweight, qzeros, (0.001 + 0.01 * torch.rand(K // gs, N, device="cuda", generator=gen)).half()


def _lengths(steps, shares):
    return {steps // shares, -(-steps // shares)}


# rows, reduction, outputs; which grid; reduction steps of its shares
GRIDS = [(600, 1024, 18432, "256 x 256", {16}), (600, 1024, 10240, "128 x 256", {16}), (600, 4096, 2048, "128 x 256 in shares", {12, 13}),
         (600, 4736, 2048, "128 x 256 in shares", {14, 15}), (1000, 4096, 8448, "128 x 256, remainder in shares", {64, 8}),
         (520, 1024, 11008, "256 x 128, one column left in shares", {16, 8}), (300, 1152, 18432, "256 x 256", {18}), (1024, 11008, 4096, "128 x 256 in shares", {86})]


@pytest.mark.parametrize("rank,f32", [(0, False), (8, True), (24, False), (64, True)])
@pytest.mark.parametrize("M,red,out,what,steps", GRIDS)
def test_bits_are_those_of_the_indexed_kernels(plans, M, red, out, what, steps, rank, f32):
    """Weights, the order of the reduction (rotated per 256 rows), its shares and the place of the adapter term are the same in both
    files, so an explicit index of the same groups gives the same bits; every length of a share modulo the four steps of the loop."""
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    cfg, splits, tail, tail_splits = _plan(plans, M, red, out, indexed=2)
    assert (cfg == 3) == (what == "256 x 256") and (splits > 1) == ("in shares" in what and tail == 0) and (tail > 0) == ("in shares" in what and splits == 1)
    assert _lengths(red // 64, splits) | (_lengths(red // 64, tail_splits) if tail else set()) == steps
    gen = torch.Generator("cuda").manual_seed(M + out + rank)
    x = torch.randn(M, red, device="cuda", generator=gen).half()
    for fwd, drop in ((True, None), (False, None), (False, (4321, 0.25))):
        if drop and not rank:
            continue
        K, N = (red, out) if fwd else (out, red)
        layer = _random_layer(K, N, 64, gen)
        la = lb = None
        if rank:
            la = torch.randn(M, rank, device="cuda", generator=gen).half()
            lb = (torch.randn(out, rank, device="cuda", generator=gen).t() if fwd else torch.randn(rank, out, device="cuda", generator=gen))
            lb = lb if f32 else lb.half()
        bias = torch.randn(out, device="cuda", generator=gen).half() if fwd else None
        if fwd:
            got = quant_hip.gemm_fwd(x, *layer, None, 64, bias=bias, xa=la, lora_bt=lb, lora_scale=2.0)
            if rank:                                                  # the matrix as [N, R] rows, as [R, N] rows and off the 16-byte grid
                other = torch.empty(rank * out + 1, dtype=lb.dtype, device="cuda")[1:].view(rank, out).copy_(lb)
                assert torch.equal(got, quant_hip.gemm_fwd(x, *layer, None, 64, bias=bias, xa=la, lora_bt=other, lora_scale=2.0))
                odd = torch.empty(rank * out + 1, dtype=lb.dtype, device="cuda")[1:].view(out, rank).copy_(lb.t()).t()
                assert torch.equal(got, quant_hip.gemm_fwd(x, *layer, None, 64, bias=bias, xa=la, lora_bt=odd, lora_scale=2.0))
        else:
            got = quant_hip.gemm_bwd_dx(x, *layer, None, 64, dyb=la, lora_a=lb, lora_scale=2.0, dropout=drop)
        assert torch.equal(got, _indexed(fwd, x, layer, 64, out, bias, la, lb, drop))
        W = quant_hip.dequant(*layer, None, 64).double()
        full = x.double() @ (W if fwd else W.t()) + (bias.double() if fwd else 0.0)
        if rank:
            term = 2.0 * la.double() @ lb.double()
            full += term if drop is None else term * quant_hip.dropout_keep_mask(M, K, *drop, x.device).double() * quant_hip.dropout_scale(drop[1])
        assert float((got.double() - full).abs().max() / full.abs().max()) <= TOL


# rows, outputs, columns of the layers; steps of the shares' parts of the layers
SHARED = [(300, 5120, (1280, 3712, 640, 2304), [20, 1, 21, 21, 15, 6, 4, 16, 20]), (300, 5120, (3200, 2048, 2688), [21, 21, 8, 13, 19, 2, 20, 20]),
          (300, 5120, (3840, 4096), [21, 21, 18, 3, 21, 20, 20])]


@pytest.mark.parametrize("M,K,Ns,parts", SHARED)
@pytest.mark.parametrize("rank,p", [(0, 0.0), (16, 0.0), (40, 0.1)])
def test_grouped_grad_input_in_shares(plans, M, K, Ns, parts, rank, p):
    """Shares of 256 x 256 tiles that end in the middle of a layer, down to one, two and three steps of it, against float64 over all rows."""
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    cfg, splits, tail, _ = _group_plan(plans, 0, M, K, Ns)
    assert cfg == 3 and splits > 1 and tail == 0
    ends, total, begin, seen = np.cumsum([n // 64 for n in Ns]), sum(Ns) // 64, 0, []
    for z in range(splits):
        end = begin + total // splits + (z < total % splits)
        seen += [int(min(end, e) - max(begin, e - n // 64)) for e, n in zip(ends, Ns) if min(end, e) > max(begin, e - n // 64)]
        begin = end
    assert seen == parts
    gen = torch.Generator("cuda").manual_seed(rank + len(Ns))
    layers = [_random_layer(K, n, 128, gen) for n in Ns]
    dys = [torch.randn(M, n, device="cuda", generator=gen).half() for n in Ns]
    dybs = [torch.randn(M, rank, device="cuda", generator=gen).half() if rank else None for _ in Ns]
    As = [torch.randn(rank, K, device="cuda", generator=gen) if rank else None for _ in Ns]
    drops = [(100 + i, p) if p and i != 1 else None for i in range(len(Ns))]
    dx = quant_hip.gemm_grouped_bwd_dx(dys, [(*l, b, A, 2.0, d) for l, b, A, d in zip(layers, dybs, As, drops)], 128)
    full = torch.zeros(M, K, dtype=torch.float64, device="cuda")
    for l, dy, b, A, d in zip(layers, dys, dybs, As, drops):
        full += dy.double() @ quant_hip.dequant(*l, None, 128).double().t()
        if rank:
            term = 2.0 * b.double() @ A.double()
            full += term if d is None else term * quant_hip.dropout_keep_mask(M, K, *d, dy.device).double() * quant_hip.dropout_scale(p)
    assert float((dx.double() - full).abs().max() / full.abs().max()) <= TOL


@pytest.mark.parametrize("ranks", [(0, 0), (8, 64), (0, 24)])
def test_grouped_bits(ranks):
    """Forward: the bits of the layers one by one, whose tiles are unsplit too, in wide tiles and their remainder of 128 x 256.  Grad-input:
    128 more outputs keep the group on the tiles of csrc/q4_gemm.hip; the outputs that both have are the same."""
    import torch
    from alpaca_lora_4bit_amd import _lib, quant_hip
    gen = torch.Generator("cuda").manual_seed(sum(ranks))
    M, K, N, gs = 300, 640, 18432, 128
    x = torch.randn(M, K, device="cuda", generator=gen).half()
    layers = [_random_layer(K, N, gs, gen) for _ in ranks]
    xas = [torch.randn(M, r, device="cuda", generator=gen).half() if r else None for r in ranks]
    Bs = [torch.randn(N, r, device="cuda", generator=gen).t() if r else None for r in ranks]
    assert _lib.lib().q4_gemm_workspace_bytes(1, M, K, N) == 0
    ys = quant_hip.gemm_grouped_fwd(x, [(*l, None, xa, B, 2.0) for l, xa, B in zip(layers, xas, Bs)], gs)
    for y, l, xa, B in zip(ys, layers, xas, Bs):
        assert torch.equal(y, _indexed(True, x, l, gs, N, None, xa, B))

    Ns, K = (384, 256), 18432
    dys = [torch.randn(M, n, device="cuda", generator=gen).half() for n in Ns]
    more = [_random_layer(K + 128, n, gs, gen) for n in Ns]
    less = [(q[:K // 8].contiguous(), z[:K // gs].contiguous(), s[:K // gs].contiguous()) for q, z, s in more]
    dybs = [torch.randn(M, r, device="cuda", generator=gen).half() if r else None for r in ranks]
    As = [torch.randn(r, K + 128, device="cuda", generator=gen) if r else None for r in ranks]
    for drops in ((None, None), ((11, 0.1), (12, 0.5)), (None, (13, 0.25))):
        def dx(ls, k):
            arr = (__import__("ctypes").c_int * 2)(*Ns)
            assert _lib.lib().q4_gemm_grouped_workspace_bytes(0, 2, M, k, arr) == 0
            return quant_hip.gemm_grouped_bwd_dx(dys, [(*l, b, None if A is None else A[:, :k].contiguous(), 2.0, d if b is not None else None)
                                                       for l, b, A, d in zip(ls, dybs, As, drops)], gs)
        assert torch.equal(dx(less, K), dx(more, K + 128)[:, :K])
