"""End-to-end parity of the drop-in layers against the CPU oracle.

Layer-level parity is against this repository's restatement of the reference semantics: the reference's
own MoE test (sharktank/tests/models/llama/moe_block_test.py:17-30) only checks that the block exports."""

import pytest
import torch
import torch.nn.functional as F

from oracle import moe_oracle as O
import moe_cases as MC

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 1e-5, torch.float16: 1e-3, torch.bfloat16: 1e-3}
# Limits on the MoE contribution y - h alone (the residual h ~ N(0, 1) is as large as the contribution and would hide an
# FFN error in a check of y).  fp32 and fp16: the north-star figures.  bf16 keeps 8 significant bits and the gated
# intermediate, the down projection and the weighted slot values are each rounded to it: a different order of the fp32
# sums moves a value across a rounding boundary now and then, and on these small layers (hidden size 512, where few terms
# average the flips out) the kernels measure 1.6e-3 to 2.1e-3 against the oracle; two formulations of the oracle itself
# that differ only in that order are up to 8e-3 apart (tests/test_oracle_golden.py).  The layer output y itself is held to
# the north-star 1e-3 (measured: under 1e-4); at the full BASELINE shapes the contribution alone is, too
# (tests/test_gpu_full_configs.py).
MOE_TOL = {torch.float32: 1e-4, torch.float16: 1e-3, torch.bfloat16: 3e-3}


def run_block(case, device, variant=0):
    from sharktank_amd.layers import MoeBlock

    theta = MC.make_theta(case, device)
    block = MoeBlock(theta, case.E, case.k, case.eps, moe_activation=case.activation)
    block.experts.kernel_variant = variant
    h = case.planes["h"].reshape(1, case.T, case.K).to(device)
    y, idx, gate = block(h, return_routing=True)
    return y.reshape(case.T, case.K).cpu(), idx.cpu(), gate.cpu()


def check_case(case, device, variant=0, tol=None, moe_tol=None):
    """Routing bit-exact; the layer output y within `tol`; the MoE contribution y - h on its own within `moe_tol`."""
    case = MC.build(case)
    y, idx, gate = run_block(case, device, variant)
    want_y, want_idx, want_gate = MC.oracle_block(case)
    assert torch.equal(idx.long(), want_idx), "routing indices differ"
    h = case.planes["h"]
    err = O.rel_l2(y.float() - h.float(), want_y.float() - h.float())
    err_y = O.rel_l2(y, want_y)
    tol = tol or TOL[case.dtype]
    moe_tol = moe_tol or MOE_TOL[case.dtype]
    print(f"  {case.fmt} {case.dtype} T={case.T} variant {variant}: layer rel-L2 {err_y:.2e}, MoE contribution {err:.2e} (limits {tol:.0e}, {moe_tol:.0e})")
    assert err_y < tol, f"layer output rel-L2 {err_y:.3e}"
    assert err < moe_tol, f"MoE contribution rel-L2 {err:.3e} (limit {moe_tol:.0e})"
    return err, err_y


def exact_block(case):
    """The layer with the oracle's routing and the same quantised operands, every product and sum in float64 and no
    rounding of intermediates to the activation dtype: what both the reference's arithmetic and the kernels approximate."""
    case = MC.build(case)
    wg, wu, wd = (w.double() for w in MC.dense_weights(case))
    h = case.planes["h"]
    x = O.rms_norm_ordered(h, case.planes["ffn_norm"], case.eps)
    idx, gate, _ = O.route(O.router_logits_ordered(x, case.planes["router"]), case.k)
    xs, zs = case.planes["x_rscale"], case.planes["z_rscale"]
    xq = (O.fake_quant_per_tensor(x, xs) if xs is not None else x).double()
    out = torch.zeros(case.T, case.K, dtype=torch.float64)
    for t in range(case.T):
        for j in range(case.k):
            e = int(idx[t, j])
            z = case.activation(wg[e] @ xq[t]) * (wu[e] @ xq[t])
            if zs is not None:
                z = O.fake_quant_per_tensor(z.float(), zs).double()
            out[t] += gate[t, j].double() * (wd[e] @ z)
    return out


def test_toy_fp32_config(device):
    """64 tokens, hidden 512, FFN 1024, 8 experts, top-2, fp32, SiLU, seed 0."""
    case = MC.Case(T=64, K=512, N=1024, fmt="dense", dtype=torch.float32, seed=0)
    err, err_y = check_case(case, device)
    assert err < 1e-4


def test_toy_fp32_matches_reference_operation_order(device):
    case = MC.build(MC.Case(T=64, K=512, N=1024, fmt="dense", dtype=torch.float32, seed=0))
    y, idx, _ = run_block(case, device)
    want_y, want_idx, _ = MC.oracle_block(case, formulation="gather")
    assert torch.equal(idx.long(), want_idx)
    assert O.rel_l2(y, want_y) < 1e-5


@pytest.mark.parametrize("fmt", ["q8_0", "q4_1", "fp8", "dense"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_small_quantized_layers(device, fmt, dtype):
    case = MC.Case(T=96, K=512, N=768, fmt=fmt, dtype=dtype, seed=21)
    check_case(case, device)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("T", [1, 24, 200, 700])
def test_fp8_weights_and_fp8_activations(device, dtype, T):
    """fp8 tensor-scaled weights with static fp8 quantizers on the FFN input and the gated intermediate.  The
    step-by-step path quantises and dequantises the activations and multiplies in the activation dtype, which is the
    reference's own arithmetic: the MoE contribution itself (without the residual) matches the oracle to the 16-bit
    tolerance.  (The automatic choice equals it for bf16 and for launches of fewer than 320 rows; larger fp16 launches go
    to the fp8 matrix cores: test_fp8_matrix_core_layer.)"""
    from sharktank_amd import _hip

    case = MC.Case(T=T, K=512, N=768, fmt="fp8", dtype=dtype, act_quant=True, seed=40 + T)
    err, err_y = check_case(case, device, variant=_hip.VARIANT_STEP_BY_STEP, tol=1e-3)
    if dtype == torch.bfloat16 or T * 2 < 320:
        built = MC.build(MC.Case(T=T, K=512, N=768, fmt="fp8", dtype=dtype, act_quant=True, seed=40 + T))
        assert torch.equal(run_block(built, device, _hip.VARIANT_AUTO)[0], run_block(built, device, _hip.VARIANT_STEP_BY_STEP)[0])
    assert err < (1e-3 if dtype == torch.float16 else 3e-3), f"MoE contribution rel-L2 {err:.3e}"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("T", [40, 200, 700])
def test_fp8_matrix_core_layer(device, dtype, T):
    """The same layers with both operands on the fp8 matrix cores (kernel variant 5): the dot product of the quantised
    samples is scaled once, skipping the reference's rounding of the dequantised samples to the activation dtype (2^-11
    relative for fp16, 2^-8 for bf16, on both operands).  With fp16 activations the MoE contribution stays within the fp8
    tolerance of 2e-2 of the reference's arithmetic.  With bf16 activations the two arithmetics are up to 6e-2 apart,
    and neither is the better one: the gated intermediate is quantised to e4m3 (3 mantissa bits), so a value that the
    two compute slightly differently lands in a different bucket now and then.  Measured against a float64 evaluation of
    the same quantised operands both are about 4e-2 off; the kernel must be no further off than the oracle (within 5 %)."""
    from sharktank_amd import _hip

    case = MC.Case(T=T, K=512, N=768, fmt="fp8", dtype=dtype, act_quant=True, seed=40 + T)
    err, err_y = check_case(case, device, variant=_hip.VARIANT_FP8_MFMA, tol=2e-2, moe_tol=2e-2 if dtype == torch.float16 else 6e-2)
    if dtype == torch.float16 and T * 2 >= 320:  # what the automatic choice takes for such a launch
        built = MC.build(MC.Case(T=T, K=512, N=768, fmt="fp8", dtype=dtype, act_quant=True, seed=40 + T))
        assert torch.equal(run_block(built, device, _hip.VARIANT_AUTO)[0], run_block(built, device, _hip.VARIANT_FP8_MFMA)[0])
    if dtype == torch.bfloat16:
        case = MC.build(case)
        y, _, _ = run_block(case, device, _hip.VARIANT_FP8_MFMA)
        want_y, _, _ = MC.oracle_block(case)
        exact = exact_block(MC.Case(T=T, K=512, N=768, fmt="fp8", dtype=dtype, act_quant=True, seed=40 + T))
        h = case.planes["h"].double()
        kernel_vs_exact = O.rel_l2(y.double() - h, exact)
        oracle_vs_exact = O.rel_l2(want_y.double() - h, exact)
        print(f"  MoE contribution against float64: kernel {kernel_vs_exact:.2e}, oracle {oracle_vs_exact:.2e}")
        assert kernel_vs_exact <= oracle_vs_exact * 1.05 + 2e-3


@pytest.mark.parametrize("variant_name,down_packed", [("VARIANT_FP8_MFMA", False), ("VARIANT_FP8_MFMA", True), ("VARIANT_FP8_TILE", True)])
def test_fp8_matrix_core_path_is_exact_up_to_dequant_rounding(device, variant_name, down_packed):
    """With activations that are exactly representable after quantisation (integers times the scale) and power-of-two
    scales, scaling the fp32 dot product once equals dequantise-then-multiply: the fp8 path must then agree with the
    16-bit path to the rounding of the result only."""
    from sharktank_amd import _hip
    from sharktank_amd.ops import device_weight
    import sharktank_amd.types as ST

    g = torch.Generator().manual_seed(3)
    T, K, N, E, k = 256, 256, 512, 4, 2
    def w8(shape):
        q = torch.randint(-8, 9, shape, generator=g).float()
        return q.to(torch.float8_e4m3fn)
    planes = {n: w8(s) for n, s in (("gate", (E, N, K)), ("up", (E, N, K)), ("down", (E, K, N)))}
    d = torch.tensor(2.0 ** -6)
    x = (torch.randint(-6, 7, (T, K), generator=g).float() * 0.25).to(torch.float16)
    experts = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)])
    dw = [device_weight(ST.PlanarQuantizedTensor(name=n, shape=list(q.shape),
                                                 layout=ST.TensorScaledLayout(shape=list(q.shape), d=d.to(device), qs=q.to(device))),
                        stacked=True, prepack=pp)
          for (n, q), pp in zip(planes.items(), (True, True, down_packed))]
    _, offsets, perm, inv = _hip.dispatch_build(experts.to(device), E)
    xs = torch.tensor(0.25)
    zs = torch.tensor(2.0 ** -4)
    got = _hip.grouped_ffn(x.to(device), *dw, _hip.ACT_SILU, offsets, perm, k, variant=getattr(_hip, variant_name),
                           x_scale=xs.to(device), z_scale=zs.to(device)).cpu()
    dense = [O.dequant_tensor_scaled(d, q).to(torch.float16) for q in planes.values()]
    want_pairs = torch.zeros(T * k, K, dtype=torch.float16)
    xq = O.fake_quant_per_tensor(x, xs)
    for p_sorted, pair in enumerate(perm.cpu().tolist()):
        t, e = pair // k, int(experts.reshape(-1)[pair])
        z = F.silu(O._mm_rt(xq[t:t + 1], dense[0][e])) * O._mm_rt(xq[t:t + 1], dense[1][e])
        want_pairs[p_sorted] = O._mm_rt(O.fake_quant_per_tensor(z, zs), dense[2][e])[0]
    assert O.rel_l2(got, want_pairs) < 1e-3


@pytest.mark.parametrize("T", [3, 32, 64, 65])
def test_narrow_unquantized_layer_with_a_long_reduction(device, T):
    """32 units of 64 features at most: up to 64 tokens the streaming kernel (which builds its own dispatch up to 64 pairs), from 65 on
    the kernel of unquantized weights."""
    check_case(MC.Case(T=T, K=3328, N=256, fmt="dense", dtype=torch.float16, seed=60 + T), device)


def test_a_subclass_that_overrides_device_weights_is_asked_every_time(device):
    from sharktank_amd.layers import MoeBlock, PreGatherFFNMOE

    case = MC.build(MC.Case(T=8, K=256, N=256, fmt="q8_0", dtype=torch.float16, seed=61))
    block = MoeBlock(MC.make_theta(case, device), case.E, case.k, case.eps)

    class Counting(PreGatherFFNMOE):
        calls = 0

        def device_weights(self):
            self.calls += 1
            return super().device_weights()

    block.experts.__class__ = Counting
    h = case.planes["h"].reshape(1, 8, 256).to(device)
    for n in (1, 2, 3):
        block(h)
        assert block.experts.calls == n


def test_gelu_and_output_norm(device):
    """Grok-style block: exact-erf GELU and a layer_output_norm (sharktank/sharktank/models/grok/grok.py:102-109)."""
    case = MC.Case(T=80, K=384, N=512, fmt="q4_1", dtype=torch.float16, act="gelu", out_norm=True, seed=22)
    check_case(case, device)


def test_decode_sizes(device):
    for T in (1, 8, 32):
        check_case(MC.Case(T=T, K=512, N=1024, fmt="q8_0", dtype=torch.float16, seed=30 + T), device)


def test_pre_gather_ffn_moe_signature(device):
    """PreGatherFFNMOE.forward(h [T,K], experts [T,k] int64, expert_gate [T,k]) -> [T,K]."""
    from sharktank_amd.layers import PreGatherFFNMOE

    case = MC.build(MC.Case(T=50, K=256, N=512, fmt="q8_0", dtype=torch.float16, seed=23))
    theta = MC.make_theta(case, device)
    layer = PreGatherFFNMOE(theta, activation=F.silu)
    g = torch.Generator().manual_seed(5)
    experts = torch.stack([torch.randperm(case.E, generator=g)[: case.k] for _ in range(case.T)])
    gate = torch.rand(case.T, case.k, generator=g).to(case.dtype)
    got = layer(case.planes["h"].to(device), experts.to(device), gate.to(device)).cpu()
    wg, wu, wd = MC.dense_weights(case)
    want = O.pre_gather_ffn_moe(case.planes["h"], experts, gate, wg, wu, wd)
    assert O.rel_l2(got, want) < 1e-3


def test_host_tensors_are_refused():
    from sharktank_amd import _hip

    with pytest.raises(RuntimeError, match="GPU only"):
        _hip.rms_norm(torch.zeros(2, 8), torch.ones(8), 1e-5)


@pytest.mark.parametrize("fmt,T", [("q8_0", 32), ("q8_0", 600), ("q4_1", 8)])
def test_forward_under_hip_graph_capture(device, fmt, T):
    """The fused forward allocates nothing, never synchronises and records no memset, so it can be captured in a HIP
    graph once the kernels have run eagerly on the device.  Every replay (with eager work and synchronisations of the
    program's own between the replays) must reproduce the eager result bit for bit."""
    from sharktank_amd import _hip
    from sharktank_amd.layers import MoeBlock
    from sharktank_amd.types import unbox_tensor

    case = MC.build(MC.Case(T=T, K=512, N=1024, fmt=fmt, dtype=torch.float16, seed=61))
    theta = MC.make_theta(case, device)
    block = MoeBlock(theta, expert_count=case.E, expert_used_count=case.k, rms_epsilon=case.eps)
    wg, wu, wd = block.experts.device_weights()
    norm_w = unbox_tensor(block.ffn_norm.weight)
    router = block._router_weight(torch.float16)
    g = torch.Generator().manual_seed(62)
    inputs = [torch.randn(T, case.K, generator=g).to(torch.float16).to(device) for _ in range(3)]
    ws = torch.empty(_hip.moe_forward_workspace_bytes(T, case.k, case.E, case.K, case.N, torch.float16), dtype=torch.uint8, device=device)

    def forward(x, out):
        _hip.moe_forward(x, norm_w, None, case.eps, router, wg, wu, wd, block.experts._act, case.k, workspace=ws, out=out)

    eager = []
    for x in inputs:  # also the warm-up that capture needs
        out = torch.empty_like(x)
        forward(x, out)
        eager.append(out)
    torch.cuda.synchronize()

    static_in, static_out = torch.empty_like(inputs[0]), torch.empty_like(inputs[0])
    graph = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        static_in.copy_(inputs[0])
        with torch.cuda.graph(graph, stream=side):
            forward(static_in, static_out)
    torch.cuda.current_stream().wait_stream(side)
    for rep in range(2):
        for x, want in zip(inputs, eager):
            static_in.copy_(x)
            graph.replay()
            got = static_out.clone()
            torch.cuda.synchronize()
            scratch = torch.randn(256, 256, device=device) @ torch.randn(256, 256, device=device)  # unrelated eager work
            assert torch.equal(got, want), f"replay {rep} differs from the eager result"
            del scratch


@pytest.mark.parametrize("fmt", ["dense", "q8_0", "q4_1"])
def test_ffnmoe_single_expert_and_cross_check(device, fmt):
    """FFNMOE (one expert as three linears, sharktank/sharktank/layers/ffn_moe_block.py:77-127) against the oracle's
    dense arithmetic, against its own three LinearLayers composed with torch's element-wise ops, and as the second
    formulation of the MoE sum: sum_j gate[t, j] * FFNMOE_{e(t, j)}(x_t) equals PreGatherFFNMOE's output."""
    from sharktank_amd.layers import FFNMOE, PreGatherFFNMOE

    case = MC.build(MC.Case(T=40, K=256, N=512, fmt=fmt, dtype=torch.float16, seed=77))
    theta = MC.make_theta(case, device)
    wg, wu, wd = MC.dense_weights(case)
    x = case.planes["h"].to(torch.float16)
    xd = x.to(device)
    outs = []
    for e in range(case.E):
        layer = FFNMOE(theta, expert_idx=e)
        got = layer(xd)
        want = O._mm_rt(F.silu(O._mm_rt(x, wg[e])) * O._mm_rt(x, wu[e]), wd[e])
        assert got.shape == (case.T, case.K) and O.rel_l2(got.cpu(), want) < 1e-3
        composed = layer.ffn_down(F.silu(layer.ffn_gate(xd)) * layer.ffn_up(xd))  # the reference's forward, op by op
        assert O.rel_l2(got.cpu(), composed.cpu()) < 1e-3
        assert layer.ffn_gate.weight.name == f"blk.0.ffn_gate.{e}.weight" or ".ffn_gate." in layer.ffn_gate.weight.name
        outs.append(got)
    g = torch.Generator().manual_seed(78)
    experts = torch.stack([torch.randperm(case.E, generator=g)[: case.k] for _ in range(case.T)]).to(device)
    gate = torch.rand(case.T, case.k, generator=g).to(torch.float16).to(device)
    fused = PreGatherFFNMOE(theta)(xd, experts, gate)
    stacked = torch.stack(outs)  # [E, T, K]
    second = torch.zeros(case.T, case.K, dtype=torch.float32, device=device)
    for j in range(case.k):
        picked = stacked[experts[:, j], torch.arange(case.T, device=device)]
        second += (gate[:, j:j + 1] * picked).float()
    assert O.rel_l2(fused.float().cpu(), second.cpu()) < 2e-3


def test_trace_hooks_dump_routing_and_output(device, tmp_path, capsys):
    """With golden dumps switched on (the reference's TURBINE_LLM_DEBUG=save_goldens_path=...), a forward of the block
    leaves one file holding its routing and its output, equal to what the call returns and to a forward without
    dumps; a model's own `trace_tensor` calls go through the same switchboard."""
    from safetensors.torch import load_file
    from sharktank_amd.layers import MoeBlock
    from sharktank_amd.utils import debugging

    case = MC.build(MC.Case(T=24, K=256, N=512, fmt="q4_1", dtype=torch.float16, seed=63))
    theta = MC.make_theta(case, device)
    block = MoeBlock(theta, expert_count=case.E, expert_used_count=case.k, rms_epsilon=case.eps)
    h = case.planes["h"].reshape(2, 12, case.K).to(device)
    plain = block(h)
    saved = debugging.DebugFlags(**vars(debugging.flags))
    try:
        debugging.flags.save_goldens_path = tmp_path
        debugging.flags.golden_sequence_value = 0
        debugging.flags.enable_nan_checks = True
        out, idx, gate = block(h, return_routing=True)
        block.trace_golden("mixtral.moe_block.0.output", out)
    finally:
        for k, v in vars(saved).items():
            setattr(debugging.flags, k, v)
    assert torch.equal(out, plain)
    files = sorted(p.name for p in tmp_path.iterdir())
    assert files == ["0000_moe_block.safetensors", "0001_mixtral.moe_block.0.output.safetensors"]
    dump = load_file(tmp_path / files[0])
    assert torch.equal(dump["output"], out.cpu())
    assert torch.equal(dump["top_k_experts"], idx.cpu()) and torch.equal(dump["expert_gate"], gate.cpu())
    assert torch.equal(load_file(tmp_path / files[1])["default"], out.cpu())


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,dtype", [("q8_0", torch.float16), ("q4_1", torch.bfloat16)])
@pytest.mark.parametrize("T", [3, 10, 48, 400])
def test_sixty_four_experts_against_the_oracle(device, fmt, dtype, T):
    """64 experts with top-6 routing (the most the one-wavefront kernels take: a lane per expert, the last lane holds
    expert 63), from a few tokens (streaming kernels, dispatch in one wavefront up to 64 pairs) to a prefill (many experts
    with partial token tiles and some without rows)."""
    # (bf16: the six weighted slot outputs of this small layer add up to about a hundredth of the residual they are added
    # to, so a single flip of the final bf16 rounding, 2^-9 of the residual, is a large fraction of the contribution: the
    # contribution is held to 2e-2 here, the layer output to 1e-3 as everywhere)
    check_case(MC.Case(T=T, K=512, N=256, E=64, k=6, fmt=fmt, dtype=dtype, seed=6400 + T), device,
               moe_tol=2e-2 if dtype == torch.bfloat16 else None)


@pytest.mark.parametrize("E,k", [(8, 2), (3, 3), (16, 4), (4, 1), (64, 6)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_single_token_forward_equals_staged_calls(device, E, k, dtype):
    """A forward of one token lets the router launch write the dispatch arrays itself; the result must be the same bits
    as router, dispatch_build, grouped_ffn and combine called one after the other."""
    from sharktank_amd import _hip
    from sharktank_amd.layers import MoeBlock
    from sharktank_amd.types import unbox_tensor

    case = MC.build(MC.Case(T=1, K=512, N=256, E=E, k=k, fmt="q8_0", dtype=dtype, seed=700 + E))
    theta = MC.make_theta(case, device)
    block = MoeBlock(theta, expert_count=E, expert_used_count=k, rms_epsilon=case.eps)
    wg, wu, wd = block.experts.device_weights()
    h = case.planes["h"].to(device)
    fused, idx_f, gate_f = block(h.reshape(1, 1, case.K), return_routing=True)

    xn = _hip.rms_norm(h, unbox_tensor(block.ffn_norm.weight), case.eps)
    idx, gate, _ = _hip.router_topk(xn, block._router_weight(dtype), k)
    assert torch.equal(idx.cpu().to(torch.int64), idx_f.cpu().to(torch.int64)) and torch.equal(gate, gate_f)
    counts, offsets, perm, inv = _hip.dispatch_build(idx, E)
    assert counts.sum().item() == k and offsets[-1].item() == k
    y = _hip.grouped_ffn(xn, wg, wu, wd, block.experts._act, offsets, perm, k)
    staged = _hip.combine(y, gate, inv, 1, k, residual=h)
    assert torch.equal(staged.view(torch.int16), fused.reshape(1, case.K).view(torch.int16))


@pytest.mark.parametrize("T", [2, 10, 11, 31, 32, 33, 200, 256, 257, 700])
@pytest.mark.parametrize("E,k", [(8, 2), (64, 6)])
@pytest.mark.parametrize("K,N", [(512, 256), (1024, 256), (512, 96)])
def test_small_batch_forward_equals_staged_calls(device, T, E, k, K, N):
    """The fused forward (one C-ABI call, one workspace) must give the same bits as router, dispatch_build, grouped_ffn and
    combine called one after the other, also when called again on the same workspace and whatever the workspace held
    before (nothing in it needs an initial value).  Forwards of at most 64 (token, slot) pairs have no dispatch launch: the
    wavefronts of the streaming gate/up launch sort the router's choices themselves and the first one writes the arrays
    the down and combine launches read (2 to 32 tokens with top-2, 2 and 10 with top-6; 33 and 11 tokens are the first
    forwards with a dispatch launch again).  The three shapes take that launch through the three streaming kernels: token
    rows shared through LDS; the reduction split over a workgroup's wavefronts (few items, four chunks or more);
    independent wavefronts (a tile count that is no multiple of four)."""
    from sharktank_amd import _hip
    from sharktank_amd.layers import MoeBlock
    from sharktank_amd.types import unbox_tensor

    if (K, N) != (512, 256) and T > 33:
        pytest.skip("the larger forwards are covered at the first shape")
    dtype = torch.float16
    case = MC.build(MC.Case(T=T, K=K, N=N, E=E, k=k, fmt="q8_0", dtype=dtype, seed=800 + T + E))
    theta = MC.make_theta(case, device)
    block = MoeBlock(theta, expert_count=E, expert_used_count=k, rms_epsilon=case.eps)
    wg, wu, wd = block.experts.device_weights()
    h = case.planes["h"].to(device)
    block.reserve_workspace(T, dtype, device)
    block._workspace.fill_(0xFF)
    fused, idx_f, gate_f = block(h.reshape(1, T, case.K), return_routing=True)
    again = block(h.reshape(1, T, case.K))
    block._workspace.fill_(0x01)
    third = block(h.reshape(1, T, case.K))

    xn = _hip.rms_norm(h, unbox_tensor(block.ffn_norm.weight), case.eps)
    idx, gate, _ = _hip.router_topk(xn, block._router_weight(dtype), k)
    assert torch.equal(idx.cpu().to(torch.int64), idx_f.cpu().to(torch.int64)) and torch.equal(gate, gate_f)
    counts, offsets, perm, inv = _hip.dispatch_build(idx, E)
    y = _hip.grouped_ffn(xn, wg, wu, wd, block.experts._act, offsets, perm, k)
    staged = _hip.combine(y, gate, inv, T, k, residual=h)
    for got in (fused, again, third):
        assert torch.equal(staged.view(torch.int16), got.reshape(T, case.K).view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize("norm_in_act_dtype", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("T,K,E,k", [(256, 2048, 8, 2), (301, 4096, 8, 2), (2051, 4096, 8, 2), (515, 6144, 16, 4), (260, 8192, 3, 3)])
def test_prefill_front_end_equals_staged_calls(device, dtype, T, K, E, k, norm_in_act_dtype):
    """Launches of many tokens run ffn_norm + router with one wavefront per token (rows of 2048 / 4096 / 6144 / 8192
    elements).  Its normalised rows, routing indices and gates must have the bits of rms_norm + router_topk called one
    after the other (whose own bits the oracle's ordered restatements pin), and so must the layer output."""
    from sharktank_amd import _hip
    from sharktank_amd import types as ST
    from sharktank_amd.layers import MoeBlock
    from sharktank_amd.types import unbox_tensor

    case = MC.build(MC.Case(T=T, K=K, N=256, E=E, k=k, fmt="q8_0", dtype=dtype, seed=900 + T + E))
    if T == 301 and dtype == torch.float16:
        case.planes["h"][:7] *= 1e-4  # rows whose squares and products reach down to fp16 subnormals
        case.planes["h"][7:9] *= 200.0
    theta = MC.make_theta(case, device)
    if norm_in_act_dtype:
        flat = theta.flatten()
        flat["ffn_norm.weight"] = ST.DefaultPrimitiveTensor(name="ffn_norm.weight", data=case.planes["ffn_norm"].to(dtype).to(device))
        theta = ST.Theta(flat)
    block = MoeBlock(theta, expert_count=E, expert_used_count=k, rms_epsilon=case.eps)
    wg, wu, wd = block.experts.device_weights()
    h = case.planes["h"].to(device)
    fused, idx_f, gate_f = block(h.reshape(1, T, K), return_routing=True)

    norm_w = unbox_tensor(block.ffn_norm.weight)
    xn = _hip.rms_norm(h, norm_w, case.eps)
    if not norm_in_act_dtype:  # (the oracle restates the fp32-weight form)
        want_xn = O.rms_norm_ordered(case.planes["h"], case.planes["ffn_norm"], case.eps)
        assert torch.equal(xn.cpu().view(torch.int16), want_xn.view(torch.int16))
    idx, gate, _ = _hip.router_topk(xn, block._router_weight(dtype), k)
    assert torch.equal(idx.cpu().to(torch.int64), idx_f.cpu().to(torch.int64))
    assert torch.equal(gate.view(torch.int16), gate_f.view(torch.int16))
    counts, offsets, perm, inv = _hip.dispatch_build(idx, E)
    y = _hip.grouped_ffn(xn, wg, wu, wd, block.experts._act, offsets, perm, k)
    staged = _hip.combine(y, gate, inv, T, k, residual=h)
    assert torch.equal(staged.view(torch.int16), fused.reshape(T, K).view(torch.int16))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("fmt,T,K,N", [("fp8", 40, 512, 768), ("fp8", 300, 512, 768), ("q8_0", 1100, 2048, 512), ("q8_0", 2300, 3328, 512), ("fp8", 700, 512, 256)])
def test_fused_activation_quantizers_equal_separate_passes(device, fmt, dtype, T, K, N):
    """Static e4m3fn quantizers of the experts' input and of the gated intermediate are applied where those tensors are
    produced (the norm launch writes the fake-quantised rows, the gate/up kernels write the fake-quantised intermediate).
    The result must have the bits of the same forward with each quantizer as a pass of its own over the finished tensor
    (stmoe_fake_quant_fp8, itself bit-exact against the oracle): the streaming kernel, the register kernel (1100 tokens), the
    prefill kernels with ride-along rows and split units (2300 tokens), and both front-end kernels are covered by the shapes."""
    from sharktank_amd import _hip
    from sharktank_amd.layers import MoeBlock
    from sharktank_amd.types import unbox_tensor

    case = MC.build(MC.Case(T=T, K=K, N=N, fmt=fmt, dtype=dtype, act_quant=True, seed=300 + T))
    theta = MC.make_theta(case, device)
    block = MoeBlock(theta, case.E, case.k, case.eps)
    block.experts.kernel_variant = _hip.VARIANT_STEP_BY_STEP  # (the fp8 matrix cores take real samples, not these values)
    wg, wu, wd = block.experts.device_weights()
    h = case.planes["h"].to(device)
    fused, idx_f, gate_f = block(h.reshape(1, T, K), return_routing=True)
    xs, zs = block.experts.activation_scales()
    assert xs is not None and zs is not None

    xn = _hip.rms_norm(h, unbox_tensor(block.ffn_norm.weight), case.eps)
    idx, gate, _ = _hip.router_topk(xn, block._router_weight(dtype), case.k)
    assert torch.equal(idx, idx_f) and torch.equal(gate, gate_f)
    counts, offsets, perm, inv = _hip.dispatch_build(idx, case.E)
    xq = _hip.fake_quant_fp8(xn, xs)
    z = _hip.grouped_gate_up(xq, wg, wu, block.experts._act, offsets, perm, case.k)
    zq = _hip.fake_quant_fp8(z, zs)
    y = _hip.grouped_down(zq, wd, offsets, T, case.k)
    staged = _hip.combine(y, gate, inv, T, case.k, residual=h)
    assert torch.equal(staged.view(torch.int16), fused.reshape(T, K).view(torch.int16))
    # the grouped FFN on its own takes both scales too
    y2 = _hip.grouped_ffn(xn, wg, wu, wd, block.experts._act, offsets, perm, case.k, x_scale=xs, z_scale=zs,
                          variant=_hip.VARIANT_STEP_BY_STEP)
    assert torch.equal(y2.view(torch.int16), y.view(torch.int16))
