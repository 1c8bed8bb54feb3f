"""The adapters of layers that run together: grouped down projections, gradients and the one-launch update of a few rows give the
bits of the separate launches (same operands, same order of sums), and a decode block hands out what its members ask for."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,Cs,rs,dtypes,ps", [
    (1, (4096, 4096), (8, 8), ("float32", "float32"), (0.0, 0.0)),
    (200, (4096, 4096), (8, 8), ("float32", "float32"), (0.05, 0.05)),           # one launch, 4 rows a workgroup
    (1037, (5120, 5120, 1024), (16, 16, 16), ("float16", "float16", "float16"), (0.1, 0.0, 0.3)),
    (33, (256, 256, 96, 256), (8, 16, 16, 5), ("float32", "float32", "float16", "float16"), (0.0, 0.1, 0.0, 0.0)),   # several launches
])
def test_grouped_down_projections_are_the_single_ones(M, Cs, rs, dtypes, ps):
    from alpaca_lora_4bit_amd import quant_hip
    g = torch.Generator(device="cuda").manual_seed(M)
    specs = []
    for i, (C, r, dt, p) in enumerate(zip(Cs, rs, dtypes, ps)):
        w = torch.randn((r, C), device="cuda", generator=g).mul_(0.1).to(getattr(torch, dt))
        x = torch.randn((M, C), device="cuda", generator=g).half()
        specs.append((x, w if i % 2 == 0 else w.t().contiguous().t(), (7 + i, p) if p else None))
    for order in (specs, specs[::2]):
        for got, (x, w, drop) in zip(quant_hip.lora_down_grouped(order), order):
            assert torch.equal(got, quant_hip.lora_down(x, w, dropout=drop))


@pytest.mark.parametrize("M,Cs,R,p", [(200, ((4096, 4096), (4096, 1024)), 8, 0.05), (1024, ((4096, 4096),) * 3, 8, 0.0),
                                      (300, ((512, 1408), (512, 264), (512, 8), (512, 128)), 40, 0.1), (1, ((64, 64), (64, 128)), 2, 0.0)])
def test_grouped_gradients_are_the_pairs(M, Cs, R, p):
    from alpaca_lora_4bit_amd import quant_hip
    g = torch.Generator(device="cuda").manual_seed(M + R)
    x = torch.randn((M, Cs[0][0]), device="cuda", generator=g).half()
    specs = []
    for i, (_, c2) in enumerate(Cs):
        p1, p2 = (torch.randn((M, R), device="cuda", generator=g).half() for _ in range(2))
        specs.append((p1, x, p2, torch.randn((M, c2), device="cuda", generator=g).half(), 0.5 + i, (3 + i, p) if p else None))
    for (da, db), (p1, in1, p2, in2, alpha, drop) in zip(quant_hip.lora_grad_grouped(specs), specs):
        want_a, want_b = quant_hip.lora_grad_pair(p1, in1, p2, in2, alpha, dropout=drop)
        assert torch.equal(da, want_a) and torch.equal(db, want_b)


@pytest.mark.parametrize("M,K,Ns,r,dtype", [(1, 4096, (4096, 4096), 8, "float32"), (4, 4096, (4096, 1024), 8, "float16"),
                                            (16, 5120, (65, 13824, 256), 16, "float32"), (5, 32, (257,), 4, "float16"),
                                            (15, 13824, (300, 5, 255, 256), 12, "float32")])
def test_update_of_a_few_rows_in_one_launch(M, K, Ns, r, dtype):
    """Edges of the 256-column blocks and of the four row groups, against the two launches it stands for."""
    from alpaca_lora_4bit_amd import _lib, quant_hip
    g = torch.Generator(device="cuda").manual_seed(M * K + r)
    x = torch.randn((M, K), device="cuda", generator=g).half()
    specs, want, guards = [], [], []
    for i, N in enumerate(Ns):
        A = torch.randn((r, K), device="cuda", generator=g).mul_(0.1).to(getattr(torch, dtype))
        B = torch.randn((N, r), device="cuda", generator=g).mul_(0.1).to(getattr(torch, dtype))
        guard = torch.randn((M + 1, N), device="cuda", generator=g).half()
        ref = guard.clone()
        xa = quant_hip.lora_down(x, A)
        _lib.check(_lib.lib().q4_lora_up_f16(xa.data_ptr(), B.data_ptr(), r, 1, int(dtype == "float32"), ref.data_ptr(), 0.5 + i, M, N, r,
                                             torch.cuda.current_stream().cuda_stream), "q4_lora_up_f16")
        specs.append((A, B, guard[:M], 0.5 + i)); want.append(ref); guards.append(guard)
    quant_hip.lora_update_grouped(x, specs)
    for got, ref in zip(guards, want):
        assert torch.equal(got, ref)


def test_update_takes_other_ranks_and_layouts_in_two_launches():
    from alpaca_lora_4bit_amd import quant_hip
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn((6, 128), device="cuda", generator=g).half()
    specs, want = [], []
    for r, dtype, strided in ((8, torch.float32, False), (3, torch.float32, False), (8, torch.float16, True), (64, torch.float16, False)):
        A = torch.randn((r, 128), device="cuda", generator=g).mul_(0.1).to(dtype)
        B = torch.randn((r, 96) if strided else (96, r), device="cuda", generator=g).mul_(0.1).to(dtype)
        B = B.t() if strided else B
        y = torch.randn((6, 96), device="cuda", generator=g).half()
        want.append(y.double() + 1.5 * (quant_hip.lora_down(x, A).double() @ B.double().t()))
        specs.append((A, B, y, 1.5))
    quant_hip.lora_update_grouped(x, specs)
    for (_, _, y, _), ref in zip(specs, want):
        assert bool(((y.double() - ref).abs() <= 2.0 ** -11 * ref.abs() + 1e-5).all())       # one rounding of y


def test_decode_block_hands_out_the_adapter_that_is_asked_for(oracle):
    """q|k|v with adapters on q and v, 3 rows: v's output is finished together with q's; a member whose adapter changes, is
    switched off or is called twice in between gets the product of that moment, as the ungrouped block does."""
    from alpaca_lora_4bit_amd.model_attn_mlp_patch import make_quant_attn
    from test_gpu_gemm_grouped import _Block
    grouped, plain = (_Block(oracle, 1024, 512, 128, 0.0, 40).eval() for _ in range(2))
    for b in (grouped, plain):
        b.v_proj.bias.zero_()
    assert make_quant_attn(grouped) == 1
    x = torch.from_numpy(oracle.make_activations(3, 1024, seed=3)).cuda()

    def same(a, b):
        assert float((a.float() - b.float()).abs().max() / b.float().abs().max()) <= 2e-3    # sums of the products in another order

    with torch.no_grad():
        for a, b in zip(grouped(x), plain(x)):
            same(a, b)
        for change in ("weight", "scaling", "off", "twice"):
            same(grouped.q_proj(x), plain.q_proj(x))
            for b in (grouped, plain):
                v = b.v_proj
                if change == "weight":
                    v.lora_B["default"].weight.mul_(-3.0)
                elif change == "scaling":
                    v.scaling["default"] = 4.0
                elif change == "off":
                    v._disable_adapters = True
                else:
                    v(x)
            same(grouped.v_proj(x), plain.v_proj(x))
            same(grouped.k_proj(x), plain.k_proj(x))
            for b in (grouped, plain):
                b.v_proj._disable_adapters = False
