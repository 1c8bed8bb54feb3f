"""HIP GEMV (M <= 16) vs the CPU oracle.  Tolerance: max|y - ref| <= 1e-2 * max|ref| against
the fp32-accumulated reference result."""
import numpy as np
import pytest

from conftest import rel_err, to_cuda_layer

pytestmark = pytest.mark.gpu
TOL = 1e-2


def _gemv(layer, x, use_gidx=True):
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    t = to_cuda_layer(layer)
    y = quant_hip.gemv(torch.from_numpy(x).cuda(), t["qweight"], t["qzeros"], t["scales"],
                       t["g_idx"] if use_gidx else None, t["groupsize"])
    torch.cuda.synchronize()
    return y.cpu().numpy()


@pytest.mark.parametrize("K,N,gs", [(4096, 4096, 128), (4096, 11008, 128), (11008, 4096, 128),
                                    (256, 128, 128), (64, 64, 32), (1024, 320, 64), (2048, 192, 2048)])
@pytest.mark.parametrize("M", [1, 4, 16])
def test_gemv_sequential_groups(oracle, K, N, gs, M):
    layer = oracle.make_layer(K, N, gs, seed=K * 7 + N)
    x = oracle.make_activations(M, K, seed=M)
    ref = oracle.matmul_recons(x, layer["qweight"], layer["qzeros"], layer["scales"], layer["g_idx"])
    for use_gidx in (True, False):
        got = _gemv(layer, x, use_gidx)
        assert got.shape == (M, N)
        assert rel_err(got, ref) <= TOL, (use_gidx, rel_err(got, ref))
    # typical error is far below the tolerance: fp32 accumulation, fp16 output rounding only
    assert rel_err(got, ref) <= 2e-3


@pytest.mark.parametrize("K,N,M", [(5120, 13824, 1), (5120, 13824, 16), (256, 128, 3), (512, 192, 7)])
def test_gemv_act_order(oracle, K, N, M):
    layer = oracle.make_layer(K, N, 128, act_order=True, seed=K + 3 * N)
    x = oracle.make_activations(M, K, seed=M + 11)
    ref = oracle.matmul_recons(x, layer["qweight"], layer["qzeros"], layer["scales"], layer["g_idx"])
    got = _gemv(layer, x)
    assert rel_err(got, ref) <= TOL
    ref32 = oracle.gemv_v2_fp32(x, layer["qweight"], layer["qzeros"], layer["scales"], layer["g_idx"])
    assert rel_err(got, ref32) <= TOL


def test_gemv_repeatable_and_workspace_left_clean(oracle):
    """The split-K reduction adds partials in a fixed order: repeated calls are bit-identical,
    and the counters in the workspace are back to zero after every call."""
    layer = oracle.make_layer(4096, 4096, 128, seed=2)
    x = oracle.make_activations(4, 4096, seed=2)
    a = _gemv(layer, x)
    for _ in range(5):
        assert np.array_equal(a.view(np.uint16), _gemv(layer, x).view(np.uint16))
    from alpaca_lora_4bit_amd import quant_hip
    assert quant_hip.workspaces_are_zero()


def test_gemv_linearity_full_size(oracle):
    """Size-independent property at a full benchmark shape: (a*x1 + x2) @ W == a*(x1 @ W) + x2 @ W."""
    layer = oracle.make_layer(4096, 11008, 128, seed=4)
    x1 = oracle.make_activations(1, 4096, seed=21)
    x2 = oracle.make_activations(1, 4096, seed=22)
    xs = (2.0 * x1.astype(np.float32) + x2.astype(np.float32)).astype(np.float16)
    y1, y2, ys = _gemv(layer, x1), _gemv(layer, x2), _gemv(layer, xs)
    lin = 2.0 * y1.astype(np.float32) + y2.astype(np.float32)
    assert rel_err(ys, lin) <= 5e-3


def test_quant_cuda_compatible_matmuls(oracle):
    """vecquant4matmul / _faster / _old_faster: accumulate into a pre-zeroed `mul` in its dtype."""
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    layer = oracle.make_layer(512, 256, 128, seed=8)
    t = to_cuda_layer(layer)
    x = oracle.make_activations(2, 512, seed=8)
    ref = oracle.matmul_recons(x, layer["qweight"], layer["qzeros"], layer["scales"], layer["g_idx"])
    xt = torch.from_numpy(x).cuda()
    y32 = torch.zeros((2, 256), dtype=torch.float32, device="cuda")
    quant_hip.vecquant4matmul(xt.float(), t["qweight"], y32, t["scales"].float(), t["qzeros"], t["g_idx"])
    assert rel_err(y32.cpu().numpy(), ref) <= TOL
    y32.zero_()
    quant_hip.vecquant4matmul_old_faster(xt, t["qweight"], y32, t["scales"].float(), t["qzeros"], 128, 256)
    assert rel_err(y32.cpu().numpy(), ref) <= TOL
    y16 = torch.zeros((2, 256), dtype=torch.float16, device="cuda")
    quant_hip.vecquant4matmul_faster(xt, t["qweight"], y16, t["scales"], t["qzeros"], t["g_idx"], 256)
    assert rel_err(y16.cpu().numpy(), ref) <= TOL
    quant_hip.vecquant4matmul_faster(xt, t["qweight"], y16, t["scales"], t["qzeros"], t["g_idx"], 256)
    assert rel_err(y16.cpu().numpy(), 2 * ref) <= TOL      # second call accumulated


def test_gemv_accumulate_flag(oracle):
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    layer = oracle.make_layer(4096, 256, 128, seed=3)
    t = to_cuda_layer(layer)
    x = oracle.make_activations(3, 4096, seed=3)
    ref = oracle.matmul_recons(x, layer["qweight"], layer["qzeros"], layer["scales"], layer["g_idx"])
    base = torch.full((3, 256), 1.5, dtype=torch.float16, device="cuda")
    quant_hip.gemv(torch.from_numpy(x).cuda(), t["qweight"], t["qzeros"], t["scales"], None, 128, out=base,
                   accumulate=True)
    assert rel_err(base.cpu().numpy(), ref + 1.5) <= TOL


def test_two_streams_and_two_threads_use_separate_workspaces(oracle):
    """The split-K accumulators (GEMV) and partial-sum scratch (GEMM) are cached per stream: products launched
    concurrently on two streams, from two Python threads, give the bits of the same products run one by one."""
    import threading
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    layers = [to_cuda_layer(oracle.make_layer(4096, 2048, 128, seed=50 + i)) for i in range(2)]
    xs = [torch.from_numpy(oracle.make_activations(m, 4096, seed=60 + i)).cuda() for i, m in enumerate((1, 16))]
    xg = [torch.from_numpy(oracle.make_activations(40, 4096, seed=70 + i)).cuda() for i in range(2)]
    want = [quant_hip.gemv(x, t["qweight"], t["qzeros"], t["scales"], None, 128) for x, t in zip(xs, layers)]
    want_g = [quant_hip.gemm_fwd(x, t["qweight"], t["qzeros"], t["scales"], None, 128) for x, t in zip(xg, layers)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = [[None] * 30, [None] * 30]
    got_g = [[None] * 30, [None] * 30]

    def work(i):
        with torch.cuda.stream(streams[i]):
            for r in range(30):
                got[i][r] = quant_hip.gemv(xs[i], layers[i]["qweight"], layers[i]["qzeros"], layers[i]["scales"], None, 128)
                got_g[i][r] = quant_hip.gemm_fwd(xg[i], layers[i]["qweight"], layers[i]["qzeros"], layers[i]["scales"],
                                                 None, 128)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    torch.cuda.synchronize()
    for i in range(2):
        assert all(torch.equal(y, want[i]) for y in got[i])
        assert all(torch.equal(y, want_g[i]) for y in got_g[i])


@pytest.mark.parametrize("M", [1, 3, 16])
@pytest.mark.parametrize("K,Ns,gs", [(4096, (11008, 11008), 128), (4096, (4096, 1024, 1024), 128), (512, (64, 192, 128, 320), 64),
                                     (11008, (4096,), 128), (256, (128, 64), 32)])
def test_gemv_grouped_matches_single_launches_and_oracle(oracle, K, Ns, gs, M):
    """q4_gemv_grouped_f16: several layers in one launch, each read from its own tensors.  Same kernels and the same
    fixed-order integer reduction as q4_gemv_f16, so each output is bit-identical to the single-layer launch;
    both are held to the oracle."""
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    layers = [oracle.make_layer(K, N, gs, seed=K + 5 * N + i) for i, N in enumerate(Ns)]
    ts = [to_cuda_layer(l) for l in layers]
    xh = oracle.make_activations(M, K, seed=M + 3)
    x = torch.from_numpy(xh).cuda()
    outs = quant_hip.gemv_grouped(x, [(t["qweight"], t["qzeros"], t["scales"]) for t in ts], gs)
    torch.cuda.synchronize()
    assert len(outs) == len(Ns)
    for lay, t, y in zip(layers, ts, outs):
        single = quant_hip.gemv(x, t["qweight"], t["qzeros"], t["scales"], None, gs)
        assert torch.equal(y, single)
        ref = oracle.matmul_recons(xh, lay["qweight"], lay["qzeros"], lay["scales"], lay["g_idx"])
        assert rel_err(y.cpu().numpy(), ref) <= TOL
    # one activation tensor per layer, g_idx given (sequential), accumulate into existing outputs
    xs = [torch.from_numpy(oracle.make_activations(M, K, seed=40 + i)).cuda() for i in range(len(Ns))]
    base = [torch.full((M, N), 0.5, dtype=torch.float16, device="cuda") for N in Ns]
    quant_hip.gemv_grouped(xs, [(t["qweight"], t["qzeros"], t["scales"], t["g_idx"]) for t in ts], gs, outs=base,
                           accumulate=True)
    for lay, xi, y in zip(layers, xs, base):
        ref = oracle.matmul_recons(xi.cpu().numpy(), lay["qweight"], lay["qzeros"], lay["scales"], lay["g_idx"]) + 0.5
        assert rel_err(y.cpu().numpy(), ref) <= TOL
    assert quant_hip.workspaces_are_zero()                    # accumulators left zeroed


def test_gemv_grouped_rejects_act_order_and_mismatched_layers(oracle):
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    a = to_cuda_layer(oracle.make_layer(256, 128, 128, act_order=True, seed=1))
    b = to_cuda_layer(oracle.make_layer(512, 128, 128, seed=2))
    c = to_cuda_layer(oracle.make_layer(256, 128, 128, seed=3))
    x = torch.zeros((1, 256), dtype=torch.float16, device="cuda")
    with pytest.raises(ValueError):
        quant_hip.gemv_grouped(x, [(a["qweight"], a["qzeros"], a["scales"], a["g_idx"])], 128)
    with pytest.raises(ValueError):
        quant_hip.gemv_grouped(x, [(c["qweight"], c["qzeros"], c["scales"]), (b["qweight"], b["qzeros"], b["scales"])], 128)
    with pytest.raises(ValueError):
        quant_hip.gemv_grouped(x, [(c["qweight"], c["qzeros"], c["scales"])] * 5, 128)


@pytest.mark.parametrize("K,Ns,gs", [(128, (64, 128), 128), (1152, (64, 192), 128), (1152, (128, 64), 2048), (2176, (64, 64), 64),
                                     (1408, (64, 128), 32), (5120, (1024, 5120, 5120, 4096), 128), (11008, (2048, 2048), 128)])
@pytest.mark.parametrize("M", [1, 4, 5, 8, 9, 16])
def test_gemv_same_bits_however_the_reduction_is_split(oracle, K, Ns, gs, M):
    """Edges of the streaming kernel: one chunk of 128 rows, a last block with fewer than 8 chunks, groups of 32 and 64 rows, a group
    beyond K, and groups of layers that take longer shares of the reduction than each of them alone.  Blocks are added as
    integers, so the split never shows; rows past M (1..16 of the 16 of an operand) and neighbouring strips stay untouched."""
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    layers = [oracle.make_layer(K, N, gs, seed=K + 3 * N + i) for i, N in enumerate(Ns)]
    ts = [to_cuda_layer(l) for l in layers]
    xh = oracle.make_activations(M, K, seed=M + 7)
    x = torch.from_numpy(xh).cuda()
    outs = quant_hip.gemv_grouped(x, [(t["qweight"], t["qzeros"], t["scales"]) for t in ts], gs)
    for lay, t, y in zip(layers, ts, outs):
        assert torch.equal(y, quant_hip.gemv(x, t["qweight"], t["qzeros"], t["scales"], None, gs))
    ref = oracle.matmul_recons(xh, layers[0]["qweight"], layers[0]["qzeros"], layers[0]["scales"], layers[0]["g_idx"])
    assert rel_err(outs[0].cpu().numpy(), ref) <= 2e-3
    assert quant_hip.workspaces_are_zero()


def test_gemv_longest_reduction(oracle):
    """More than 255 blocks of 1024 rows: shares of several blocks keep the arrival count within 8 bits."""
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    K, N, gs, M = 262144 + 128, 64, 128, 3
    layer = oracle.make_layer(K, N, gs, seed=5)
    t = to_cuda_layer(layer)
    x = oracle.make_activations(M, K, seed=5)
    y = quant_hip.gemv(torch.from_numpy(x).cuda(), t["qweight"], t["qzeros"], t["scales"], None, gs)
    ref = oracle.matmul_recons(x, layer["qweight"], layer["qzeros"], layer["scales"], layer["g_idx"])
    assert rel_err(y.cpu().numpy(), ref) <= 2e-3
    assert quant_hip.workspaces_are_zero()


def _offset_heavy(M, K, gs, gen):
    """Activations whose plain sums are exact in fp32 in any order (multiples of 2^-9, partial sums below 2^14) while their sums
    with the operand offsets (1024 on even rows, 64 on odd ones) need more than 24 bits, and their sum per group."""
    import torch
    G = K // gs
    x = torch.zeros((M, G, gs), dtype=torch.float64)
    big = torch.randint(256, 512, (M, G, gs // 4), generator=gen).double()
    x[:, :, 0:gs // 2:2] = big
    x[:, :, gs // 2::2] = -big.flip(-1)
    x[:, :, 1::2] = torch.randint(-500, 500, (M, G, gs // 2), generator=gen).double() / 512
    return x.view(M, K), x.sum(-1)


@pytest.mark.parametrize("route,K,gs", [("stream", 4096, 128), ("stream", 1152, 64), ("stream", 1152, 32), ("grouped", 2176, 128),
                                        ("burst", 2080, 32), ("burst", 2112, 64), ("sorted", 2048, 128), ("sorted", 2048, 32), ("v1", 2048, 2048)])
@pytest.mark.parametrize("M", [1, 2, 3, 7, 16])
def test_gemv_offsets_of_the_operands_cancel_exactly(route, K, gs, M):
    """With all codes 0 the sum with the codes and the sum of the offsets are the same operations, so what is left is
    -s * (z + 1) * sum x, exact in fp32 here: nothing of the rounding of the offset products may stay in the result."""
    import torch
    from alpaca_lora_4bit_amd import _lib, quant_hip
    if route == "sorted" and M > 3:
        pytest.skip("the gathering kernel takes up to three rows")
    gen = torch.Generator().manual_seed(K + gs + M)
    N, G = 128, K // gs
    x, sums = _offset_heavy(M, K, min(gs, 128), gen)
    qw = torch.zeros((K // 8, N), dtype=torch.int32, device="cuda")
    z = torch.randint(0, 16, (G, N), generator=gen)
    qz = torch.zeros((G, N // 8), dtype=torch.int64)
    for b in range(8):
        qz |= z[:, b::8] << (4 * b)
    qz = torch.where(qz >= 2 ** 31, qz - 2 ** 32, qz).int().cuda()
    sc = torch.full((G, N), 0.125, dtype=torch.float16, device="cuda")
    want = (-0.125 * (sums @ (z + 1).double())).half().cuda() if route != "v1" else None
    xt = x.half().cuda()
    assert torch.equal(xt.double().cpu(), x)
    if route == "grouped":
        got = quant_hip.gemv_grouped(xt, [(qw, qz, sc)] * 2, gs)[1]
    elif route == "v1":
        zeros = torch.full((N, 1), 0.75, dtype=torch.float16, device="cuda")
        got = quant_hip.gemv_v1(xt, qw, torch.ones_like(zeros), zeros)
        want = (-0.75 * sums.sum(1, keepdim=True)).half().expand(M, N).cuda()
    elif route == "sorted":
        perm = torch.randperm(K, generator=gen)
        inverse = torch.empty_like(perm)
        inverse[perm] = torch.arange(K)
        xt = xt[:, inverse.cuda()].contiguous()              # gathered through perm it is x again
        got = torch.empty((M, N), dtype=torch.float16, device="cuda")
        ws = torch.zeros(_lib.lib().q4_gemv_workspace_bytes(M, K, N), device="cuda", dtype=torch.uint8)
        perm = perm.int().cuda()
        _lib.check(_lib.lib().q4_gemv_sorted_f16(xt.data_ptr(), qw.data_ptr(), qz.data_ptr(), sc.data_ptr(), perm.data_ptr(), gs, got.data_ptr(),
                                                 0, M, K, N, G, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream), "sorted")
    else:
        got = quant_hip.gemv(xt, qw, qz, sc, None, gs)
    assert torch.equal(got, want)


@pytest.mark.parametrize("K,Ns,gs", [(128, (64,), 128), (384, (64, 128), 128), (896, (192,), 32), (1152, (64, 64), 64), (4096, (4096,), 128),
                                     (4096, (8192,), 128), (4096, (4096, 4096, 64), 128), (5120, (128,), 64), (2048, (8192, 64), 32), (3200, (13824,), 640)])
def test_one_and_two_rows_have_the_bits_of_the_first_of_three(K, Ns, gs):
    """One and two rows go through eight wavefronts of one chunk or through the stream, by groups and number of workgroups; three
    rows through the stream: the same sums in the same order, alone and in a group."""
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    gen = torch.Generator(device="cuda").manual_seed(K + sum(Ns))
    G = -(-K // gs)
    layers = [(torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 8, N), device="cuda", dtype=torch.int32, generator=gen),
               torch.randint(-2 ** 31, 2 ** 31 - 1, (G, N // 8), device="cuda", dtype=torch.int32, generator=gen),
               torch.rand((G, N), device="cuda", generator=gen).half()) for N in Ns]
    x = torch.randn((3, K), device="cuda", generator=gen).half()
    three = [quant_hip.gemv(x, *l, None, gs) for l in layers]
    for M in (1, 2):
        grouped = quant_hip.gemv_grouped(x[:M].contiguous(), layers, gs)
        for l, want, got in zip(layers, three, grouped):
            assert bool(torch.isfinite(want).all())
            assert torch.equal(quant_hip.gemv(x[:M].contiguous(), *l, None, gs), want[:M]) and torch.equal(got, want[:M])
    assert quant_hip.workspaces_are_zero()


@pytest.mark.parametrize("blocks,gs,M", [(257, 64, 2), (257, 64, 7), (258, 64, 16), (300, 32, 3), (300, 32, 5), (600, 128, 1), (600, 1024, 16), (1020, 128, 3),
                                         (1020, 32, 9)])
def test_gemv_of_more_blocks_than_arrivals(oracle, blocks, gs, M):
    """Shares of several blocks, up to the longest reduction that is taken, for every number of groups per chunk and of outputs per
    thread, alone and in a group: the exchange holds them, the result is the sum and the accumulators are left zero.  The last
    block has one chunk."""
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    K, N = blocks * 1024 - 896, 64
    layer = oracle.make_layer(K, N, gs, seed=blocks)
    t = to_cuda_layer(layer)
    x = oracle.make_activations(M, K, seed=M)
    xt, packed = torch.from_numpy(x).cuda(), (t["qweight"], t["qzeros"], t["scales"])
    y = quant_hip.gemv(xt, *packed, None, gs)
    assert all(torch.equal(y, other) for other in quant_hip.gemv_grouped(xt, [packed] * 2, gs))
    ref = oracle.matmul_recons(x, layer["qweight"], layer["qzeros"], layer["scales"], layer["g_idx"])
    assert rel_err(y.cpu().numpy(), ref) <= 2e-3
    assert quant_hip.workspaces_are_zero()


@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_gemv_shares_beyond_the_exchange_saturate(sign):
    """1020 blocks of sums beyond 2^22 in 255 workgroups: the most the exchange can be asked to hold, in either direction."""
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    K, N = 1020 * 1024, 64
    qw = torch.full((K // 8, N), -1, dtype=torch.int32, device="cuda")                # codes 15, zero points 1
    qz = torch.zeros((K // 128, N // 8), dtype=torch.int32, device="cuda")
    x = torch.full((1, K), sign * 60000.0, dtype=torch.float16, device="cuda")
    y = quant_hip.gemv(x, qw, qz, torch.full((K // 128, N), 2.0, dtype=torch.float16, device="cuda"), None, 128)
    assert torch.equal(y, torch.full_like(y, sign * float("inf")))
    assert quant_hip.workspaces_are_zero()


@pytest.mark.parametrize("route,K,gs", [("burst", 131104, 32), ("burst", 131136, 96), ("grouped", 262208, 64), ("gidx", 65312, 32), ("gidx", 524352, 64),
                                        ("v1", 131104, 131104), ("v1", 524416, 524416)])
@pytest.mark.parametrize("M", [1, 6])
def test_long_reductions_of_odd_chunks(oracle, route, K, gs, M):
    """Reductions of more chunks than 255 workgroups of one chunk per wavefront hold, by every kernel that takes such sizes."""
    import torch
    from alpaca_lora_4bit_amd import _lib, quant_hip
    N = 64
    layer = oracle.make_layer(K, N, gs, act_order=route == "gidx", seed=M)
    t = to_cuda_layer(layer)
    x = oracle.make_activations(M, K, seed=M)
    xt = torch.from_numpy(x).cuda()
    if route == "grouped":
        y = quant_hip.gemv_grouped(xt, [(t["qweight"], t["qzeros"], t["scales"])] * 2, gs)[1]
    elif route == "v1":
        zeros = torch.from_numpy(layer["scales"] * (layer["zcodes"] + 1).astype("float16")).cuda()      # scale * (q - z - 1)
        y = torch.empty((M, N), dtype=torch.float16, device="cuda")
        ws = torch.zeros(M * N * 8 + 256, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        _lib.check(_lib.lib().q4_gemv_v1_f16(xt.data_ptr(), t["qweight"].data_ptr(), t["scales"].data_ptr(), zeros.data_ptr(), y.data_ptr(), 0,
                                             M, K, N, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream), "q4_gemv_v1_f16")
        assert not bool(ws.any())
        weights = layer["codes"].astype("float64") * layer["scales"].astype("float64") - zeros.cpu().numpy().astype("float64")
        assert rel_err(y.cpu().numpy(), x.astype("float64") @ weights) <= 2e-3
        return
    else:
        try:
            quant_hip.actorder_repack = False
            y = quant_hip.gemv(xt, t["qweight"], t["qzeros"], t["scales"], t["g_idx"] if route == "gidx" else None, gs)
        finally:
            quant_hip.actorder_repack = True
    ref = oracle.matmul_recons(x, layer["qweight"], layer["qzeros"], layer["scales"], layer["g_idx"])
    assert rel_err(y.cpu().numpy(), ref) <= 3e-3             # the gathering kernel multiplies fp16 weights
    assert quant_hip.workspaces_are_zero()


# shares of 3, 5 and 6 blocks in two teams, of 7 and 8 (their sums beyond the LDS beside two teams' tiles) in one; 6 and 8 fill all 160 KB
@pytest.mark.parametrize("K", [3072, 5120, 6144, 7168, 8192])
@pytest.mark.parametrize("M", [7, 8, 9, 16])
def test_longer_shares_in_two_teams_have_the_bits_of_single_blocks(oracle, K, M):
    """216 strips at 7 rows and more: one workgroup takes the whole reduction, its blocks in turn to two teams of wavefronts.  Up to
    four rows every block has a workgroup of its own; the sums of a row are the same integers either way."""
    import torch
    from alpaca_lora_4bit_amd import quant_hip
    N = 13824
    layer = oracle.make_layer(K, N, 128, seed=K + M)
    t = to_cuda_layer(layer)
    xh = oracle.make_activations(M, K, seed=M)
    x = torch.from_numpy(xh).cuda()
    args = (t["qweight"], t["qzeros"], t["scales"], None, 128)
    y = quant_hip.gemv(x, *args)
    for lo in range(0, M, 4):
        assert torch.equal(y[lo:lo + 4], quant_hip.gemv(x[lo:lo + 4].contiguous(), *args))
    assert torch.equal(y, quant_hip.gemv(x, *args))
    grouped = quant_hip.gemv_grouped(x, [(t["qweight"], t["qzeros"], t["scales"])], 128)[0]
    assert torch.equal(y, grouped)
    rows = [0, M - 1]
    ref = oracle.matmul_recons(xh[rows], layer["qweight"], layer["qzeros"], layer["scales"], layer["g_idx"])
    assert rel_err(y.cpu().numpy()[rows], ref) <= 2e-3
