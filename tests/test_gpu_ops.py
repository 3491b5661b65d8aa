"""The `sharktank.ops`-level surface on the GPU: quantized matmul/linear with the generators of the reference's own
kernel tests, dispatch selection, and layout dequant through the layout classes."""

import pytest
import torch

from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu


def test_mmt_block_scaled_q8_reference_generator(device):
    """The shapes and the seed of sharktank/tests/kernels/mmt_block_scaled_q8_test.py:24-41 (a [4,16,3200], d [3200,100,1],
    qs [3200,100,32], seed 42; expected = a @ (d*qs).flatten(1).T) through ops.matmul, with two stated changes: a and d
    are drawn as rand / 64 where the reference draws rand * 64 (with * 64 every fp16 output is +inf, which compares equal
    and checks nothing; test_kernels_mmt_block_scaled_q8 below runs the reference's own * 64 generator in fp32), and the
    tolerances are atol 1e-2 with rtol 1e-4 (fp32) / 2e-3 (fp16) instead of atol 1e-3, rtol 1e-5: the reference compares
    an fp32 kernel with an fp32 matmul, here the fp16 case rounds the dequantised weights and the result to fp16."""
    from sharktank_amd import ops, types as ST

    torch.manual_seed(42)
    for dtype, atol, rtol in ((torch.float32, 1e-3, 1e-5), (torch.float16, 1.0, 1e-3)):
        a = (torch.rand([4, 16, 3200], dtype=torch.float32) / 64).to(dtype)
        d = (torch.rand([3200, 100, 1], dtype=torch.float32) / 64).to(torch.float16)
        qs = (torch.rand([3200, 100, 32], dtype=torch.float32) * 32.0).to(torch.int8)
        w = ST.PlanarQuantizedTensor(shape=[3200, 3200], layout=ST.BlockScaledLayout([3200, 3200], d.to(device), qs.to(device)))
        ops._test_enable_last_op_dispatch(True)
        try:
            got = ops.matmul(a.to(device), w, transpose_rhs=True)
            assert ops._test_get_last_op_dispatch().__name__ == "matmul_tensor_quantized"
        finally:
            ops._test_enable_last_op_dispatch(False)
        assert got.shape == (4, 16, 3200) and got.dtype == dtype
        b = O.dequant_block_scaled(d, qs).flatten(1).to(dtype)
        ref = O.mmt(a, b)
        torch.testing.assert_close(got.cpu(), ref, atol=atol * 1e-2, rtol=max(rtol, 2e-3 if dtype == torch.float16 else 1e-4))


def test_mmt_block_scaled_offset_q4_reference_generator(device):
    """sharktank/tests/kernels/mmt_block_scaled_offset_q4_test.py:25-44: a/256, d/256, qs uint8*255, m + 16."""
    from sharktank_amd import ops, types as ST

    torch.manual_seed(42)
    a = torch.rand([4, 16, 3200], dtype=torch.float32) / 256.0
    d = (torch.rand([3200, 100, 1], dtype=torch.float32) / 256.0).to(torch.float16)
    qs = (torch.rand([3200, 100, 16], dtype=torch.float32) * 255.0).to(torch.uint8)
    m = (torch.rand([3200, 100, 1], dtype=torch.float32) + 16.0).to(torch.float16)
    w = ST.PlanarQuantizedTensor(shape=[3200, 3200], layout=ST.BlockScaledI4Layout(
        [3200, 3200], d.to(device), qs.to(device), m=m.to(device), signed=False))
    got = ops.matmul(a.to(device), w, transpose_rhs=True)
    b = O.dequant_block_scaled_i4(d, qs, m).flatten(1).float()
    ref = torch.matmul(a, b.T)
    torch.testing.assert_close(got.cpu(), ref, atol=1e-2, rtol=1e-3)


def test_linear_and_dense_matmul(device):
    from sharktank_amd import ops, types as ST

    g = torch.Generator().manual_seed(1)
    x = torch.randn(33, 256, generator=g).to(torch.float16)
    w = torch.randn(48, 256, generator=g) * 0.05  # f32 weight, cast to the activation dtype as linear_default does
    got = ops.linear(x.to(device), ST.DefaultPrimitiveTensor(data=w.to(device)))
    ref = O.mmt(x, w)
    assert got.dtype == torch.float16 and O.rel_l2(got.cpu(), ref) < 1e-3
    with pytest.raises(NotImplementedError):
        ops.matmul(x.to(device), w.to(device), transpose_rhs=False)


@pytest.mark.parametrize("fmt", ["q8_0", "q4_1", "fp8"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N", [(1, 96), (7, 96), (16, 256), (17, 96), (32, 256), (33, 96), (40, 256), (64, 256), (80, 96), (81, 256)])
def test_quantized_linear_few_rows(device, fmt, dtype, M, N):
    """One quantized matrix times a handful of rows (a Llama-style projection at decode): the streaming kernel runs
    without an expert offsets array (up to 32 rows by itself, beyond that on request), from planar and from packed
    planes, with the same bits from both."""
    import moe_cases as MC
    from sharktank_amd import _hip
    from sharktank_amd.ops import device_weight

    K = 1024
    case = MC.build(MC.Case(T=4, K=K, N=N, E=1, k=1, fmt=fmt, dtype=dtype, seed=90 + M))
    it = MC.to_inference_tensor(fmt, case.planes["gate"], [1, N, K], "w", device)
    x = (torch.randn(M, K, generator=torch.Generator().manual_seed(M)) * 0.5).to(dtype)
    w_ref = MC.dense_weights(case)[0][0].to(dtype)
    ref = O.mmt(x, w_ref)
    outs = []
    for prepack in (False, True):
        dw = device_weight(it, stacked=True, prepack=prepack)
        auto = _hip.mmt(x.to(device), dw)
        assert O.rel_l2(auto.cpu(), ref) < (1e-3 if dtype == torch.float16 else 8e-3)
        forced = _hip.mmt(x.to(device), dw, variant=_hip.VARIANT_SKINNY)
        if M <= 32:  # the automatic choice for so few rows is the streaming kernel (N = 256: its LDS-sharing form)
            assert torch.equal(auto.view(torch.int16), forced.view(torch.int16))
        else:
            assert O.rel_l2(forced.cpu(), ref) < (1e-3 if dtype == torch.float16 else 8e-3)
        outs.append(forced.cpu())
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


@pytest.mark.parametrize("fmt", ["q8_0", "q4_1"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M", [33, 48, 129, 200, 256, 300, 512])
def test_quantized_linear_few_hundred_rows_splits_the_reduction(device, fmt, dtype, M):
    """A few hundred rows of one matrix make too few 256 x 256 units for the chip: with a workspace the units are cut along
    the reduction and the chunk that finishes last adds the fp32 partial tiles.  Checked against the oracle's dense product
    and against the launch without a workspace (one fp32 sum per output instead of four: equal to the rounding of the
    output), twice in a row (the tickets that elect the adding workgroup must be back at zero)."""
    import moe_cases as MC
    from sharktank_amd import _hip
    from sharktank_amd.ops import device_weight

    K, N = 2048, 1792  # 7 column units: every one of them is split
    case = MC.build(MC.Case(T=4, K=K, N=N, E=1, k=1, fmt=fmt, dtype=dtype, seed=300 + M))
    it = MC.to_inference_tensor(fmt, case.planes["gate"], [1, N, K], "w", device)
    x = (torch.randn(M, K, generator=torch.Generator().manual_seed(M)) * 0.5).to(dtype)
    ref = O.mmt(x, MC.dense_weights(case)[0][0].to(dtype))
    dw = device_weight(it, stacked=True, prepack=True)
    lib = _hip.load_library()
    need = int(lib.stmoe_mmt_workspace_bytes(M))
    assert need > 0 and int(lib.stmoe_mmt_workspace_bytes(32)) == 0
    ws = torch.full((need,), 0xA5, dtype=torch.uint8, device=device)  # stale contents must not matter
    tol = 1e-3 if dtype == torch.float16 else 8e-3
    # (the 256 x 256 kernel is named: the automatic choice takes this matrix to the register kernel up to 128 rows and to 64 x 256 tiles
    # from 129 on, neither of which splits)
    ws_kernel = _hip.VARIANT_MFMA_WS
    plain = _hip.mmt(x.to(device), dw, workspace=torch.empty(0, dtype=torch.uint8, device=device), variant=ws_kernel)
    assert O.rel_l2(plain.cpu(), ref) < tol
    first = _hip.mmt(x.to(device), dw, workspace=ws, variant=ws_kernel)
    second = _hip.mmt(x.to(device), dw, workspace=ws, variant=ws_kernel)
    own = _hip.mmt(x.to(device), dw, variant=ws_kernel)  # the binding's own buffer
    assert O.rel_l2(first.cpu(), ref) < tol
    assert torch.equal(first.view(torch.int16), second.view(torch.int16)) and torch.equal(first.view(torch.int16), own.view(torch.int16))
    assert not torch.equal(first.view(torch.int16), plain.view(torch.int16))  # (the reduction was split)
    assert O.rel_l2(first.float().cpu(), plain.float().cpu()) < (5e-4 if dtype == torch.float16 else 4e-3)
    # (narrow tiles keep one running sum per output like `plain`)
    auto = _hip.mmt(x.to(device), dw)
    assert torch.equal(auto.view(torch.int16), (_hip.mmt(x.to(device), dw, variant=_hip.VARIANT_MFMA_REG) if M <= 128 else plain).view(torch.int16))


@pytest.mark.parametrize("fmt", ["q8_0", "q4_1", "fp8"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_quantized_linear_narrow_tiles(device, fmt, dtype):
    """A single matrix with a few hundred rows runs on tiles of 64 output features x 256 rows (kernel variant 9): enough
    tiles for the CUs without cutting the reduction.  Against the oracle's dense product, bit for bit against the
    128 x 128 tile kernel (both keep one fp32 running sum per output, in the same order), and as the automatic choice from
    129 rows on; ragged row counts on both sides of the 256-row tile; a matrix whose feature count is no multiple of 64
    goes to the other kernels."""
    import moe_cases as MC
    from sharktank_amd import _hip
    from sharktank_amd.ops import device_weight

    K, N = 1024, 448  # 7 feature tiles
    case = MC.build(MC.Case(T=4, K=K, N=N, E=1, k=1, fmt=fmt, dtype=dtype, seed=410))
    dw = device_weight(MC.to_inference_tensor(fmt, case.planes["gate"], [1, N, K], "w", device), stacked=True, prepack=True)
    wd = MC.dense_weights(case)[0][0].to(dtype)
    tol = 1e-3 if dtype == torch.float16 else 8e-3
    for M in (1, 64, 129, 200, 255, 256, 257, 300, 512, 700):
        x = (torch.randn(M, K, generator=torch.Generator().manual_seed(M)) * 0.5).to(dtype)
        ref = O.mmt(x, wd)
        narrow = _hip.mmt(x.to(device), dw, variant=_hip.VARIANT_MFMA_NARROW)
        tile = _hip.mmt(x.to(device), dw, variant=_hip.VARIANT_MFMA_TILE)
        assert torch.isfinite(narrow.float()).all()
        assert O.rel_l2(narrow.cpu(), ref) < tol, (M, O.rel_l2(narrow.cpu(), ref))
        assert torch.equal(narrow.view(torch.int16), tile.view(torch.int16)), M
        if M > 128:
            assert torch.equal(_hip.mmt(x.to(device), dw).view(torch.int16), narrow.view(torch.int16)), M
    # 96 output features: no whole 64-feature tiles, the request falls through to the kernels that take the shape
    case = MC.build(MC.Case(T=4, K=K, N=96, E=1, k=1, fmt=fmt, dtype=dtype, seed=411))
    dw = device_weight(MC.to_inference_tensor(fmt, case.planes["gate"], [1, 96, K], "w", device), stacked=True, prepack=True)
    x = (torch.randn(200, K, generator=torch.Generator().manual_seed(5)) * 0.5).to(dtype)
    got = _hip.mmt(x.to(device), dw, variant=_hip.VARIANT_MFMA_NARROW)
    assert O.rel_l2(got.cpu(), O.mmt(x, MC.dense_weights(case)[0][0].to(dtype))) < tol


@pytest.mark.parametrize("fmt,dtype", [("q8_0", torch.float16), ("q4_1", torch.bfloat16)])
@pytest.mark.parametrize("act", ["silu", "gelu"])
def test_gated_ffn_on_narrow_tiles(device, fmt, dtype, act):
    """The gated form of the narrow tiles (32 gate + the same 32 up features x 256 rows, the gated product formed in
    registers) and the down projection on them: one expert through the grouped FFN with kernel variant 9 named, against the
    oracle's down(act(gate x) * up x) and against the 128 x 128 tile kernel."""
    import moe_cases as MC
    from sharktank_amd import _hip
    from sharktank_amd.ops import device_weight

    K, N = 512, 768
    case = MC.build(MC.Case(T=4, K=K, N=N, E=1, k=1, fmt=fmt, dtype=dtype, act=act, seed=420))
    dws = [device_weight(MC.to_inference_tensor(fmt, case.planes[n], shape, n, device), stacked=True, prepack=True)
           for n, shape in (("gate", [1, N, K]), ("up", [1, N, K]), ("down", [1, K, N]))]
    dense = MC.dense_weights(case)
    wg, wu, wdn = (dense[i][0].to(dtype) for i in range(3))
    fn = torch.nn.functional.silu if act == "silu" else torch.nn.functional.gelu
    act_id = _hip.ACT_SILU if act == "silu" else _hip.ACT_GELU_ERF
    for M in (130, 256, 300, 513):
        x = (torch.randn(M, K, generator=torch.Generator().manual_seed(M))).to(dtype)
        want = O._mm_rt(fn(O._mm_rt(x, wg)) * O._mm_rt(x, wu), wdn)
        got = _hip.grouped_ffn(x.to(device), *dws, act_id, None, None, 1, variant=_hip.VARIANT_MFMA_NARROW)
        tile = _hip.grouped_ffn(x.to(device), *dws, act_id, None, None, 1, variant=_hip.VARIANT_MFMA_TILE)
        assert torch.isfinite(got.float()).all()
        assert O.rel_l2(got.cpu(), want) < (1e-3 if dtype == torch.float16 else 8e-3), (M, O.rel_l2(got.cpu(), want))
        assert O.rel_l2(got.float().cpu(), tile.float().cpu()) < (2e-4 if dtype == torch.float16 else 4e-3)


def test_quantized_linear_split_reduction_under_hip_graph_capture(device):
    """A product of a few dozen rows cuts its reduction over several workgroups, which elect the adding one through counters
    in the workspace.  Captured in a HIP graph (the capture brings its own buffer, cleared inside the graph by a kernel: no
    memset node) every replay must give the eager result bit for bit, with eager products, which use the kept buffer,
    between the replays."""
    import moe_cases as MC
    from sharktank_amd import _hip
    from sharktank_amd.ops import device_weight

    K, N, M = 2048, 1792, 64
    case = MC.build(MC.Case(T=4, K=K, N=N, E=1, k=1, fmt="q8_0", dtype=torch.float16, seed=77))
    it = MC.to_inference_tensor("q8_0", case.planes["gate"], [1, N, K], "w", device)
    dw = device_weight(it, stacked=True, prepack=True)
    g = torch.Generator().manual_seed(78)
    inputs = [(torch.randn(M, K, generator=g) * 0.5).to(torch.float16).to(device) for _ in range(3)]
    # (the prefill kernel is named: the automatic choice takes this matrix to the register kernel, which does not split)
    split = lambda x, **kw: _hip.mmt(x, dw, variant=_hip.VARIANT_MFMA_WS, **kw)  # noqa: E731
    eager = [split(x) for x in inputs]  # (also the warm-up that capture needs)
    unsplit = split(inputs[0], workspace=torch.empty(0, dtype=torch.uint8, device=device))
    assert not torch.equal(eager[0].view(torch.int16), unsplit.view(torch.int16))
    torch.cuda.synchronize()
    static_in = torch.empty_like(inputs[0])
    graph = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        static_in.copy_(inputs[0])
        with torch.cuda.graph(graph, stream=side):
            static_out = split(static_in)
    torch.cuda.current_stream().wait_stream(side)
    for rep in range(2):
        for x, want in zip(inputs, eager):
            static_in.copy_(x)
            graph.replay()
            got = static_out.clone()
            torch.cuda.synchronize()
            assert torch.equal(got.view(torch.int16), want.view(torch.int16))
            again = split(x)  # eager work between the replays
            assert torch.equal(again.view(torch.int16), want.view(torch.int16))


def test_layout_classes_dequant_on_device(device):
    from sharktank_amd import types as ST

    g = torch.Generator().manual_seed(2)
    w = torch.randn(3, 64, 128, generator=g) * 0.02
    d, qs = O.quantize_q8_0(w)
    lay = ST.BlockScaledLayout([3, 64, 128], d.to(device), qs.to(device))
    assert torch.equal(lay.dequant().cpu(), O.dequant_block_scaled(d, qs).reshape(3, 64, 128))
    d4, m4, q4 = O.quantize_q4_1(w)
    lay4 = ST.BlockScaledI4Layout([3, 64, 128], d4.to(device), q4.to(device), m=m4.to(device))
    assert torch.equal(lay4.dequant(torch.float32).cpu(), O.dequant_block_scaled_i4(d4, q4, m4, dtype=torch.float32).reshape(3, 64, 128))
    assert torch.equal(lay4.qs.cpu(), O.promote_linear_i4_block_to_i8(q4))
    # GGUF raw blocks -> planar planes -> device
    raw = torch.cat([d.view(torch.uint8).reshape(-1, 2), qs.view(torch.uint8).reshape(-1, 32)], dim=1).reshape(-1)
    q8 = ST.Q8_0(raw=raw, shape=[3, 64, 128]).to_planar().to(device="cuda:0")
    assert torch.equal(q8.unpack().dequant().cpu(), O.dequant_block_scaled(d, qs).reshape(3, 64, 128))


def test_static_scaled_quantizer_fp8(device):
    from sharktank_amd import types as ST

    x = torch.randn(64, 32, generator=torch.Generator().manual_seed(3)).to(torch.float16)
    rscale = torch.tensor(0.0118, dtype=torch.float32)
    q = ST.StaticScaledQuantizer(scale=(1.0 / rscale).to(device), reciprocal_scale=rscale.to(device), dtype=torch.float8_e4m3fn)
    qt = q.quantize(x.to(device))
    want_qs, _, _ = O.static_quantize_per_tensor(x, rscale, torch.float8_e4m3fn)
    assert torch.equal(qt.unpack().qs.cpu().view(torch.uint8), want_qs.view(torch.uint8))
    deq = qt.unpack().dequant()
    assert deq.dtype == torch.float16
    assert torch.equal(deq.cpu(), O.dequant_tensor_scaled(rscale, want_qs, layout_dtype=torch.float16))


@pytest.mark.parametrize("fmt", ["q8_0", "q4_1", "fp8", "dense"])
@pytest.mark.parametrize("dtype,T", [(torch.float16, 40), (torch.bfloat16, 9), (torch.float32, 12)])
def test_gathered_expert_einsums(device, fmt, dtype, T):
    """`weights[experts]` + einsum_2args for the three einsum strings of PreGatherFFNMOE
    (shapes as in sharktank/tests/kernels/einsum_q4_test.py:32-89, enlarged), against the materialised gather."""
    import moe_cases as MC
    from sharktank_amd import ops, types as ST

    case = MC.build(MC.Case(T=T, K=128, N=96 if fmt == "dense" else 256, fmt=fmt, dtype=dtype, seed=70))
    E, N, K, k = case.E, case.N, case.K, case.k
    g = torch.Generator().manual_seed(71)
    experts = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)])
    x = case.planes["h"]
    wg, wu, wd = MC.dense_weights(case)
    w_it = MC.to_inference_tensor(fmt, case.planes["gate"], [E, N, K], "w", device)
    gathered = w_it[experts.to(device), :, :] if fmt != "dense" else ops.gather_experts(w_it, experts.to(device))
    assert isinstance(gathered, ST.GatheredExpertsTensor) and gathered.shape == [T, k, N, K]
    got = ops.einsum_2args(x.to(device), gathered, "mk,menk->men")
    want = O._mm_rt(x.unsqueeze(1), wg[experts].reshape(T, k * N, K)).reshape(T, k, N)
    tol = 1e-5 if dtype == torch.float32 else (1e-3 if dtype == torch.float16 else 8e-3)
    assert got.shape == (T, k, N) and O.rel_l2(got.cpu(), want) < tol
    # "mek,menk->men" with the down matrix
    z = torch.randn(T, k, N, generator=g).to(dtype)
    wd_it = MC.to_inference_tensor(fmt, case.planes["down"], [E, K, N], "wd", device)
    got2 = ops.einsum_2args(z.to(device), ops.gather_experts(wd_it, experts.to(device)), "mek,menk->men")
    want2 = O._mm_rt(z.reshape(T * k, 1, N), wd[experts].reshape(T * k, K, N)).reshape(T, k, K)
    assert O.rel_l2(got2.cpu(), want2) < tol
    # "me,men->men"
    gate = torch.rand(T, k, generator=g).to(dtype)
    got3 = ops.einsum_2args(gate.to(device), got2, "me,men->men")
    assert torch.equal(got3.cpu(), (gate.unsqueeze(-1) * got2.cpu()))
    with pytest.raises(NotImplementedError):
        ops.einsum_2args(x.to(device), gathered, "mk,bnk->bmn")


def test_forward_unfused_equals_fused(device):
    import moe_cases as MC
    from sharktank_amd.layers import PreGatherFFNMOE

    case = MC.build(MC.Case(T=70, K=256, N=512, fmt="q4_1", dtype=torch.float16, act="gelu", seed=72))
    layer = PreGatherFFNMOE(MC.make_theta(case, device), activation=torch.nn.functional.gelu)
    g = torch.Generator().manual_seed(73)
    experts = torch.stack([torch.randperm(case.E, generator=g)[: case.k] for _ in range(case.T)]).to(device)
    gate = torch.rand(case.T, case.k, generator=g).to(case.dtype).to(device)
    h = case.planes["h"].to(device)
    a = layer(h, experts, gate)
    b = layer.forward_unfused(h, experts, gate)
    assert O.rel_l2(b.cpu(), a.cpu()) < 1e-3
    wg, wu, wd = MC.dense_weights(case)
    want = O.pre_gather_ffn_moe(case.planes["h"], experts.cpu(), gate.cpu(), wg, wu, wd, torch.nn.functional.gelu)
    assert O.rel_l2(b.cpu(), want) < 1e-3


# ---- the reference's custom-op layer: same operand sets and argument checks ---------------------------------------
# Generators as in sharktank/tests/kernels/mmt_block_scaled_q8_test.py:31-41, mmt_block_scaled_offset_q4_test.py:32-44
# and einsum_q4_test.py:32-89 (fp16 scales); expected values from the layouts' dequantisation (in the scales' dtype,
# as the eager reference path dequantises) followed by an fp32 product.
@pytest.mark.parametrize("a_dtype", [torch.float32, torch.float16])
def test_kernels_mmt_block_scaled_q8(device, a_dtype):
    from sharktank_amd import kernels

    torch.manual_seed(42)
    # (the reference's factors of 64 overflow an fp16 result to inf on both sides; fp16 runs use 1/16 instead)
    amp = 64.0 if a_dtype == torch.float32 else 1.0 / 16
    a = torch.rand([4, 16, 3200], dtype=a_dtype) * amp
    d = torch.rand([3200, 100, 1], dtype=torch.float16) * amp
    qs = (torch.rand([3200, 100, 32], dtype=torch.float32) * 32.0).to(torch.int8)
    got = kernels.mmt_block_scaled_q8(a.to(device), d.to(device), qs.to(device))
    b = O.dequant_block_scaled(d, qs).reshape(3200, 3200).to(a_dtype)
    want = torch.matmul(a.float(), b.float().T)
    assert got.shape == (4, 16, 3200) and got.dtype == a_dtype
    assert O.rel_l2(got.float().cpu(), want) < (1e-5 if a_dtype == torch.float32 else 1e-3)
    with pytest.raises(RuntimeError, match="Expected 3d tensor"):
        kernels.mmt_block_scaled_q8(a[0].to(device), d.to(device), qs.to(device))
    with pytest.raises(RuntimeError, match="arg 'qs': Incorrect shape"):
        kernels.mmt_block_scaled_q8(a.to(device), d.to(device), qs[:, :50].to(device))


@pytest.mark.parametrize("a_dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("batched", [False, True])
def test_kernels_mmt_block_scaled_offset_q4_unsigned(device, a_dtype, batched):
    from sharktank_amd import kernels

    torch.manual_seed(42)
    n = 320 if batched else 3200
    lead = [4] if batched else []
    a = torch.rand([4, 16, 3200], dtype=a_dtype) / 256.0
    d = torch.rand(lead + [n, 100, 1], dtype=torch.float16) / 256.0
    qs = (torch.rand(lead + [n, 100, 16], dtype=torch.float32) * 255.0).to(torch.uint8)
    m = torch.rand(lead + [n, 100, 1], dtype=torch.float16) + 16.0
    got = kernels.mmt_block_scaled_offset_q4_unsigned(a.to(device), d.to(device), qs.to(device), m.to(device))
    b = O.dequant_block_scaled_i4(d, qs, m).reshape(lead + [n, 3200]).to(a_dtype)
    want = torch.matmul(a.float(), b.float().transpose(-1, -2))
    assert got.shape == (4, 16, n) and got.dtype == a_dtype
    assert O.rel_l2(got.float().cpu(), want) < (1e-5 if a_dtype == torch.float32 else 1e-3)
    with pytest.raises(RuntimeError, match="arg 'm': Incorrect shape"):
        kernels.mmt_block_scaled_offset_q4_unsigned(a.to(device), d.to(device), qs.to(device), m[..., :50, :].to(device))


@pytest.mark.parametrize("a_dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("es", ["mk,menk->men", "mek,menk->men", "me,men->men"])
def test_kernels_einsum_2args_q4(device, a_dtype, es):
    from sharktank_amd import kernels

    torch.manual_seed(42)
    if es == "me,men->men":
        a = torch.rand([2, 4], dtype=a_dtype) / 256.0
        planes = [2, 4, 10]
    else:
        a = torch.rand([2, 320] if es.startswith("mk") else [2, 4, 320], dtype=a_dtype) / 256.0
        planes = [2, 4, 8, 10]
    d = torch.rand(planes + [1], dtype=torch.float16) / 256.0
    qs = (torch.rand(planes + [16], dtype=torch.float32) * 255.0).to(torch.uint8)
    m = torch.rand(planes + [1], dtype=torch.float16) + 16.0
    got = kernels.einsum_2args_q4(a.to(device), d.to(device), qs.to(device), m.to(device), es)
    b = O.dequant_block_scaled_i4(d, qs, m).flatten(len(planes) - 1).to(a_dtype)
    want = torch.einsum(es, a.float(), b.float())
    assert got.shape == want.shape and got.dtype == a_dtype
    assert O.rel_l2(got.float().cpu(), want) < (1e-5 if a_dtype == torch.float32 else 1e-3)
    with pytest.raises(NotImplementedError):
        kernels.einsum_2args_q4(a.to(device), d.to(device), qs.to(device), m.to(device), "ij,jk->ik")


def test_quantized_matmul_descriptor_is_built_once_and_packed(device):
    """ops.matmul / ops.linear / LinearLayer on a quantized weight build the device descriptor on the first call (planes made
    contiguous, re-ordered into the streaming order) and reuse it afterwards, so they run the packed kernels; a changed
    plane invalidates it."""
    from sharktank_amd import ops, types as ST
    from sharktank_amd.layers import LinearLayer

    g = torch.Generator().manual_seed(12)
    N, K = 512, 1024
    d, qs = O.quantize_q8_0(torch.randn(N, K, generator=g) * 0.02)
    w = ST.PlanarQuantizedTensor(name="weight", shape=[N, K], layout=ST.BlockScaledLayout([N, K], d.to(device), qs.to(device)))
    x = torch.randn(3, 40, K, generator=g).to(torch.float16)
    y1 = ops.matmul(x.to(device), w, transpose_rhs=True)
    store = w.__dict__["_stmoe_descriptors"]
    (key, dw), = store.values()
    assert dw.is_packed
    y2 = LinearLayer(ST.Theta({"weight": w}))(x.to(device))
    assert next(iter(store.values()))[1] is dw, "the descriptor must be reused, not rebuilt"
    want = O.mmt(x, O.dequant_block_scaled(d, qs).reshape(N, K).to(torch.float16))
    assert torch.equal(y1, y2) and O.rel_l2(y1.cpu(), want) < 1e-3
    # an in-place change of a plane gives a new descriptor and the new product
    w.unpack().d.mul_(2.0)
    y3 = ops.matmul(x.to(device), w, transpose_rhs=True)
    assert next(iter(store.values()))[1] is not dw
    assert O.rel_l2(y3.cpu(), O.mmt(x, O.dequant_block_scaled(d * 2, qs).reshape(N, K).to(torch.float16))) < 1e-3


@pytest.mark.parametrize("fmt", ["q8_0", "q4_1"])
@pytest.mark.parametrize("M", [1, 32, 33, 100, 2048])  # 33 (down), 100: the prefill kernel with its reductions split (scratch appended to the workspace)
def test_ffn_layer_llama_shape(device, fmt, M):
    """FFN (sharktank/sharktank/layers/ffn_block.py:21-51) at a Llama-8B shape, hidden 4096, FFN 14336, quantized weights:
    the gated form on the fused kernels against the closed form down(silu(gate x) * up x) of the oracle, row by row."""
    import moe_cases as MC
    from sharktank_amd import types as ST
    from sharktank_amd.layers import FFN

    K, N = 4096, 14336
    gg = torch.Generator(device=device).manual_seed(20)
    planes, tensors = {}, {}
    for name, shape in (("ffn_gate", [N, K]), ("ffn_up", [N, K]), ("ffn_down", [K, N])):
        w = torch.randn(shape, generator=gg, device=device) * 0.02
        q = O.quantize_q8_0(w) if fmt == "q8_0" else O.quantize_q4_1(w)
        p = {"d": q[0], "qs": q[1]} if fmt == "q8_0" else {"d": q[0], "m": q[1], "qs": q[2]}
        planes[name] = {k: v.cpu() for k, v in p.items()}
        tensors[f"{name}.weight"] = MC.to_inference_tensor(fmt, p, shape, f"{name}.weight", device)
    ffn = FFN(ST.Theta(tensors))
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(21)).to(torch.float16)
    got = ffn(x.reshape(1, M, K).to(device)).reshape(M, K).cpu()
    rows = list(range(M)) if M <= 32 else [r for r in (0, 1, 31, 32, 63, 64, 99, 255, 256, 257, 1023, 1024, 2047) if r < M]
    xs = x[rows]
    dense = {n: MC.dense_from_planes(fmt, planes[n], [N, K] if n != "ffn_down" else [K, N], torch.float16) for n in planes}
    z = torch.nn.functional.silu(O._mm_rt(xs, dense["ffn_gate"])) * O._mm_rt(xs, dense["ffn_up"])
    want = O._mm_rt(z, dense["ffn_down"])
    assert torch.isfinite(got.float()).all()
    assert O.rel_l2(got[rows], want) < 1e-3


def test_ffn_layer_ungated_and_with_bias(device):
    """The forms without a fused kernel compose the linears as the reference does: an un-gated FFN, and a gated one whose
    projections carry a bias (ops.linear adds it after the product, sharktank/sharktank/ops/default_impls.py:328-341)."""
    import moe_cases as MC
    from sharktank_amd import types as ST
    from sharktank_amd.layers import FFN

    g = torch.Generator().manual_seed(22)
    K, N, M = 256, 512, 24
    up = torch.randn(N, K, generator=g) * 0.05
    down = torch.randn(K, N, generator=g) * 0.05
    theta = ST.Theta({"ffn_up.weight": ST.DefaultPrimitiveTensor(name="ffn_up.weight", data=up.to(torch.float16).to(device)),
                      "ffn_down.weight": ST.DefaultPrimitiveTensor(name="ffn_down.weight", data=down.to(torch.float16).to(device))})
    x = torch.randn(M, K, generator=g).to(torch.float16)
    got = FFN(theta, is_gated=False, activation_fn=torch.nn.functional.gelu)(x.to(device)).cpu()
    want = O._mm_rt(torch.nn.functional.gelu(O._mm_rt(x, up.to(torch.float16))), down.to(torch.float16))
    assert O.rel_l2(got, want) < 1e-3

    # gated, Q8_0 weights, a bias on the gate and on the down projection
    gate = torch.randn(N, K, generator=g) * 0.05
    b_gate, b_down = (torch.randn(N, generator=g) * 0.1).to(torch.float16), (torch.randn(K, generator=g) * 0.1).to(torch.float16)
    planes = {n: MC._quantize("q8_0", w) for n, w in (("ffn_gate", gate), ("ffn_up", up), ("ffn_down", down))}
    tensors = {f"{n}.weight": MC.to_inference_tensor("q8_0", planes[n], [N, K] if n != "ffn_down" else [K, N], f"{n}.weight", device)
               for n in planes}
    tensors["ffn_gate.bias"] = ST.DefaultPrimitiveTensor(name="ffn_gate.bias", data=b_gate.to(device))
    tensors["ffn_down.bias"] = ST.DefaultPrimitiveTensor(name="ffn_down.bias", data=b_down.to(device))
    got = FFN(ST.Theta(tensors))(x.to(device)).cpu()
    dense = {n: MC.dense_from_planes("q8_0", planes[n], [N, K] if n != "ffn_down" else [K, N], torch.float16) for n in planes}
    z = torch.nn.functional.silu(O._mm_rt(x, dense["ffn_gate"]) + b_gate) * O._mm_rt(x, dense["ffn_up"])
    want = O._mm_rt(z, dense["ffn_down"]) + b_down
    assert got.dtype == torch.float16 and O.rel_l2(got, want) < 1e-3


@pytest.mark.parametrize("y_dtype,b_dtype", [(torch.float16, torch.float16), (torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32),
                                             (torch.float32, torch.bfloat16), (torch.float16, torch.bfloat16)])
def test_linear_bias_add_bit_exact(device, y_dtype, b_dtype):
    """ops.linear with a bias: the product is rounded to the input's dtype, then `result + bias` in torch's promoted dtype
    (sharktank/sharktank/ops/default_impls.py:328-341).  The add itself is checked bit for bit against torch on the host."""
    from sharktank_amd import _hip, ops
    from sharktank_amd import types as ST

    g = torch.Generator().manual_seed(31)
    y = (torch.randn(37, 200, generator=g) * 3).to(y_dtype)
    b = (torch.randn(200, generator=g) * 3).to(b_dtype)
    got = _hip.add_bias(y.to(device), b.to(device)).cpu()
    want = y + b
    assert got.dtype == want.dtype and torch.equal(got, want)
    if y_dtype != torch.float32:
        w = (torch.randn(200, 64, generator=g) * 0.1).to(y_dtype)
        x = torch.randn(5, 3, 64, generator=g).to(y_dtype)
        out = ops.linear(x.to(device), ST.DefaultPrimitiveTensor(name="w", data=w.to(device)), b.to(device)).cpu()
        ref = O._mm_rt(x.reshape(15, 64), w).reshape(5, 3, 200) + b
        assert out.dtype == ref.dtype and O.rel_l2(out, ref) < 1e-3


@pytest.mark.parametrize("in_dtype,out_dtype", [(torch.float16, torch.float32), (torch.bfloat16, torch.float32), (torch.float32, None),
                                                (torch.float16, None)])
@pytest.mark.parametrize("shape,dim", [((300, 8), 1), ((300, 8), -1), ((5, 64), 1), ((7, 1000), 1), ((4, 6, 40), 1), ((3, 100), 0)])
def test_softmax_op(device, in_dtype, out_dtype, shape, dim):
    """ops.softmax (sharktank/sharktank/ops/signatures.py:974-993; F.softmax in default_impls.py:426-432) against torch on the
    host in fp32; on router-sized rows, ranking its probabilities reproduces the router kernel's choice."""
    from sharktank_amd import _hip, ops

    g = torch.Generator().manual_seed(33)
    x = (torch.randn(*shape, generator=g) * 4).to(in_dtype)
    got = ops.softmax(x.to(device), dim=dim, dtype=out_dtype).cpu()
    want = torch.nn.functional.softmax(x.float(), dim=dim).to(out_dtype or in_dtype)
    assert got.dtype == want.dtype and got.shape == want.shape
    assert torch.allclose(got.float(), want.float(), rtol=1e-5 if got.dtype == torch.float32 else 4e-3, atol=1e-7)
    assert torch.allclose(got.float().sum(dim=dim), torch.ones(()), atol=2e-3 if got.dtype != torch.float32 else 1e-5)


def test_softmax_of_router_logits_ranks_like_the_router(device):
    from sharktank_amd import _hip, ops

    g = torch.Generator().manual_seed(34)
    T, K, E, k = 500, 512, 8, 2
    x = torch.randn(T, K, generator=g).to(torch.float16).to(device)
    wr = (torch.randn(E, K, generator=g) * 0.02).to(torch.float16).to(device)
    idx, gate, logits = _hip.router_topk(x, wr, k, want_logits=True)
    probs = ops.softmax(logits, dim=1, dtype=torch.float32).cpu()
    want_idx, want_gate, want_probs = O.route(logits.cpu(), k)
    assert torch.equal(idx.cpu().long(), want_idx)
    assert torch.allclose(probs, want_probs, rtol=1e-6, atol=1e-9)
    # ranking the op's probabilities (descending, lower index first on ties) is the kernel's choice
    order = torch.sort(probs, dim=1, descending=True, stable=True).indices[:, :k]
    assert torch.equal(order, idx.cpu().long())


def test_bigger_mmg_is_the_per_pair_gathered_product(device):
    """PreGatherFFNMOE.bigger_mmg = weights[experts] + "mek,menk->men" (sharktank/sharktank/layers/ffn_moe_block.py:43-47)."""
    import moe_cases as MC
    from sharktank_amd.layers import PreGatherFFNMOE

    case = MC.build(MC.Case(T=40, K=256, N=512, fmt="q4_1", dtype=torch.float16, seed=71))
    ffn = PreGatherFFNMOE(MC.make_theta(case, device))
    g = torch.Generator().manual_seed(72)
    idx = torch.stack([torch.randperm(case.E, generator=g)[:case.k] for _ in range(case.T)])
    z = torch.randn(case.T, case.k, case.N, generator=g).to(torch.float16)
    got = ffn.bigger_mmg(z.to(device), ffn.ffn_down, idx.to(device)).cpu()
    wd = MC.dense_weights(case)[2]
    want = torch.stack([torch.stack([O._mm_rt(z[t, j:j + 1], wd[idx[t, j]])[0] for j in range(case.k)]) for t in range(case.T)])
    assert got.shape == (case.T, case.k, case.K) and O.rel_l2(got, want) < 1e-3


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("scale_dtype", ["same", torch.float32])
@pytest.mark.parametrize("shape,axis", [((40, 96), 1), ((40, 96), 0), ((3, 17, 64), 1), ((3, 17, 64), 2)])
def test_static_scaled_quantizer_per_axis(device, dtype, scale_dtype, shape, axis):
    """StaticScaledQuantizer with a 1-d scale (sharktank/sharktank/types/quantizers.py:184-230): samples bit for bit those
    of the oracle's per-axis branch (the product in the dtype torch promotes the two tensors to), and the layout's dequant
    with the broadcast reciprocal scale bit for bit the oracle's TensorScaledLayout dequant."""
    from sharktank_amd import types as ST

    g = torch.Generator().manual_seed(31 + axis)
    sdt = dtype if scale_dtype == "same" else scale_dtype
    t = (torch.randn(shape, generator=g) * 3).to(dtype)
    t.view(-1)[0] = 1000.0  # saturates
    scale = (torch.rand(shape[axis], generator=g) * 60 + 20).to(sdt)
    q = ST.StaticScaledQuantizer(scale=scale.to(device), dtype=torch.float8_e4m3fn, axis=axis)
    assert q.axis == axis
    qt = q.quantize(t.to(device))
    layout = qt.unpack()
    want_qs, want_d, _ = O.static_quantize_per_axis(t, scale, axis, torch.float8_e4m3fn)
    assert torch.equal(layout.qs.cpu().view(torch.uint8), want_qs.view(torch.uint8))
    assert list(layout.d.shape) == list(want_d.shape) and torch.equal(layout.d.cpu(), want_d)
    want = O.dequant_tensor_scaled(want_d, want_qs, layout_dtype=dtype)
    got = layout.dequant()
    assert got.dtype == want.dtype
    view = torch.int32 if want.dtype == torch.float32 else torch.int16
    assert torch.equal(got.cpu().view(view), want.view(view))


@pytest.mark.parametrize("kind", ["dynamic", "per_axis"])
def test_pre_gather_ffn_moe_with_dynamic_and_per_axis_input_quantizers(device, kind):
    """ffn_gate_exps.q_input as a DynamicScaledQuantizer (scale from the input's own maximum) or as a per-axis static
    quantizer (one scale per hidden feature): the layer quantises and dequantises its input with the quantizer's own
    arithmetic and must match the oracle fed with the same fake-quantised input."""
    import moe_cases as MC
    from sharktank_amd import types as ST
    from sharktank_amd.layers import PreGatherFFNMOE

    case = MC.build(MC.Case(T=48, K=512, N=768, fmt="q8_0", dtype=torch.float16, seed=61))
    x = case.planes["h"]
    g = torch.Generator().manual_seed(62)
    idx = torch.stack([torch.randperm(case.E, generator=g)[:case.k] for _ in range(case.T)])
    gate = torch.full((case.T, case.k), 0.5, dtype=torch.float16)
    flat = MC.make_theta(case, device).flatten()
    if kind == "dynamic":
        flat["ffn_gate_exps.q_input"] = ST.DynamicScaledQuantizer(name="ffn_gate_exps.q_input", dtype=torch.float8_e4m3fn)
        qs, rscale = O.dynamic_quantize(x, torch.float8_e4m3fn)
        xq = O.dequant_tensor_scaled(rscale, qs, layout_dtype=torch.float16)
    else:
        scale = (torch.rand(case.K, generator=g) * 40 + 60).to(torch.float32)
        flat["ffn_gate_exps.q_input"] = ST.StaticScaledQuantizer(name="ffn_gate_exps.q_input", scale=scale.to(device),
                                                                 dtype=torch.float8_e4m3fn, axis=1)
        qs, d, _ = O.static_quantize_per_axis(x, scale, 1, torch.float8_e4m3fn)
        xq = O.dequant_tensor_scaled(d, qs, layout_dtype=torch.float16).to(torch.float16)
    ffn = PreGatherFFNMOE(ST.Theta(flat))
    got = ffn(x.to(device), idx.to(device), gate.to(device)).cpu()
    wg, wu, wd = MC.dense_weights(case)
    want = O.grouped_ffn_moe(xq.to(torch.float16), idx, gate, wg, wu, wd, case.activation)
    assert O.rel_l2(got, want) < 1e-3


@pytest.mark.parametrize("kind", ["dynamic", "per_axis"])
@pytest.mark.parametrize("through", ["PreGatherFFNMOE", "MoeBlock"])
def test_dynamic_and_per_axis_quantizers_of_the_intermediate(device, kind, through):
    """ffn_down_exps.q_input as a DynamicScaledQuantizer (sharktank/sharktank/types/quantizers.py:338-389: its scale is the
    maximum of the whole gated intermediate) or as a static quantizer with one scale per feature: the gate/up projection,
    the quantizer's quantise + dequantise and the down projection run as three steps, and the result must match the oracle
    taken through the same three steps.  Through MoeBlock the forward takes its staged form (no quantizer may be dropped),
    which is also checked with a dynamic quantizer of the input."""
    import moe_cases as MC
    from sharktank_amd import types as ST
    from sharktank_amd.layers import MoeBlock, PreGatherFFNMOE

    case = MC.build(MC.Case(T=48, K=512, N=768, fmt="q8_0", dtype=torch.float16, seed=63))
    g = torch.Generator().manual_seed(64)
    flat = MC.make_theta(case, device).flatten()
    if kind == "dynamic":
        flat["ffn_down_exps.q_input"] = ST.DynamicScaledQuantizer(name="ffn_down_exps.q_input", dtype=torch.float8_e4m3fn)

        def fake_quant(z):
            qs, rscale = O.dynamic_quantize(z, torch.float8_e4m3fn)
            return O.dequant_tensor_scaled(rscale, qs, layout_dtype=torch.float16).to(torch.float16)
    else:
        scale = (torch.rand(case.N, generator=g) * 200 + 300).to(torch.float32)
        flat["ffn_down_exps.q_input"] = ST.StaticScaledQuantizer(name="ffn_down_exps.q_input", scale=scale.to(device),
                                                                 dtype=torch.float8_e4m3fn, axis=-1)

        def fake_quant(z):
            qs, d, _ = O.static_quantize_per_axis(z, scale, 1, torch.float8_e4m3fn)
            return O.dequant_tensor_scaled(d, qs, layout_dtype=torch.float16).to(torch.float16)
    wg, wu, wd = MC.dense_weights(case)

    def oracle_ffn(x, idx, gate):
        T, k = idx.shape
        pairs_x = x.repeat_interleave(k, dim=0)
        e = idx.reshape(-1)
        z = torch.stack([(case.activation(O._mm_rt(pairs_x[p:p + 1], wg[e[p]])) * O._mm_rt(pairs_x[p:p + 1], wu[e[p]]))[0] for p in range(T * k)])
        zq = fake_quant(z)
        y = torch.stack([O._mm_rt(zq[p:p + 1], wd[e[p]])[0] for p in range(T * k)]).reshape(T, k, -1)
        return torch.sum(gate.to(torch.float16).unsqueeze(-1) * y, dim=1)

    if through == "PreGatherFFNMOE":
        x = case.planes["h"]
        idx = torch.stack([torch.randperm(case.E, generator=g)[:case.k] for _ in range(case.T)])
        gate = torch.full((case.T, case.k), 0.5, dtype=torch.float16)
        got = PreGatherFFNMOE(ST.Theta(flat))(x.to(device), idx.to(device), gate.to(device)).cpu()
        assert O.rel_l2(got, oracle_ffn(x, idx, gate)) < 1e-3
        return
    block = MoeBlock(ST.Theta(flat), case.E, case.k, case.eps)
    h = case.planes["h"]
    out, idx, gate = block(h.reshape(1, case.T, case.K).to(device), return_routing=True)
    xn = O.rms_norm_ordered(h, case.planes["ffn_norm"], case.eps)
    want_idx, want_gate, _ = O.route(O.router_logits_ordered(xn, case.planes["router"]), case.k)
    assert torch.equal(idx.cpu().long(), want_idx)
    moe = oracle_ffn(xn, want_idx, want_gate.to(torch.float16))
    out = out.reshape(case.T, case.K).cpu()
    # (MoeBlock adds the residual, which is some thirty times the experts' contribution here: the contribution itself is
    # held to 1e-3 by the PreGatherFFNMOE form of this test; here the staged forward must add the right one)
    assert O.rel_l2(out, h + moe) < 3e-4
    plain_out = MoeBlock(MC.make_theta(case, device), case.E, case.k, case.eps)(h.reshape(1, case.T, case.K).to(device)).reshape(case.T, case.K).cpu()
    assert not torch.equal(out, plain_out), "the intermediate's quantizer left no trace in the output"
    # a dynamic quantizer of the input reaches the experts through MoeBlock too
    flat.pop("ffn_down_exps.q_input")
    flat["ffn_gate_exps.q_input"] = ST.DynamicScaledQuantizer(name="ffn_gate_exps.q_input", dtype=torch.float8_e4m3fn)
    out2 = MoeBlock(ST.Theta(flat), case.E, case.k, case.eps)(h.reshape(1, case.T, case.K).to(device)).reshape(case.T, case.K).cpu()
    qs, rscale = O.dynamic_quantize(xn, torch.float8_e4m3fn)
    xq = O.dequant_tensor_scaled(rscale, qs, layout_dtype=torch.float16).to(torch.float16)
    want2 = O.grouped_ffn_moe(xq, want_idx, want_gate.to(torch.float16), wg, wu, wd, case.activation)
    assert O.rel_l2(out2, h + want2) < 3e-4
    assert not torch.equal(out2, plain_out), "the input quantizer left no trace in the output"


@pytest.mark.parametrize("fmt", ["dense", "q8_0", "q4_1", "fp8"])
@pytest.mark.parametrize("T,K,N,E,k", [(1, 64, 32, 8, 2), (5, 96, 160, 3, 2), (40, 512, 96, 8, 2), (77, 352, 224, 4, 2), (150, 128, 320, 2, 2)])
def test_f32_layers_against_the_general_kernel_and_fp64(device, fmt, T, K, N, E, k):
    """fp32 activations: the matrix-core kernel (token tiles of 16, 32 and 64 rows, a last pass with fewer, reduction lengths
    with a partial chunk of 64, feature counts with a partial tile of 32) against the general kernel and against fp64."""
    import moe_cases as MC
    from sharktank_amd import _hip
    from sharktank_amd.ops import device_weight

    case = MC.build(MC.Case(T=T, K=K, N=N, E=E, k=k, fmt=fmt, dtype=torch.float32, seed=900 + T))
    idx = torch.stack([torch.randperm(E, generator=torch.Generator().manual_seed(t))[:k] for t in range(T)]).to(torch.int32)
    dws = [device_weight(MC.to_inference_tensor(fmt, case.planes[n], shp, n, device), stacked=True)
           for n, shp in (("gate", [E, N, K]), ("up", [E, N, K]), ("down", [E, K, N]))]
    x = case.planes["h"].to(device)
    _, offsets, perm, inv = _hip.dispatch_build(idx.to(device), E)
    got = _hip.grouped_ffn(x, *dws, _hip.ACT_SILU, offsets, perm, k)
    other = _hip.grouped_ffn(x, *dws, _hip.ACT_SILU, offsets, perm, k, variant=_hip.VARIANT_GENERIC)
    wg, wu, wd = (w.double() for w in MC.dense_weights(case))
    pairs = perm.cpu().long()
    e, t = idx.reshape(-1)[pairs].long(), pairs // k
    xs = case.planes["h"].double()[t]
    z = torch.nn.functional.silu(torch.einsum("rk,rnk->rn", xs, wg[e])) * torch.einsum("rk,rnk->rn", xs, wu[e])
    want = torch.einsum("rn,rkn->rk", z, wd[e])
    # sums of up to 512 fp32 products: half a unit in the last place per addition at worst, three chained sums
    tol = 3 * 512 ** 0.5 * 2.0 ** -24 * 4
    for y in (got, other):
        assert O.rel_l2(y.cpu().double(), want) < tol


@pytest.mark.parametrize("K", [64, 128, 512, 1024, 2048, 4096])
def test_f32_products_are_no_further_from_fp64_than_the_general_kernel(device, K):
    """Rounding error of the fp32 matrix-core kernel's sums against that of the general kernel, whose lanes add 1/64 of the
    products each (tiles of 64, 32 and 16 rows, dense weights)."""
    from sharktank_amd import _hip

    g = torch.Generator().manual_seed(K)
    x, w = torch.randn(112, K, generator=g), torch.randn(256, K, generator=g) / K ** 0.5
    want = x.double() @ w.double().T
    dw = _hip.DeviceWeight(_hip.W_DENSE, 1, 256, K, w.to(device), None, None, _hip.F32)
    err = {v: O.rel_l2(_hip.mmt(x.to(device), dw, variant=v).cpu().double(), want) for v in (_hip.VARIANT_AUTO, _hip.VARIANT_GENERIC)}
    # a mean over 28672 rounding errors: 1 % of itself, so 5 % are room enough
    assert err[_hip.VARIANT_AUTO] < 1.05 * err[_hip.VARIANT_GENERIC], err


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,K,N,act", [
    ((1, 0, 15, 16), 64, 64, "silu"),               # one K step; fewer weight rows than one wide unit
    ((17, 63, 64, 65), 128, 128, "gelu"),
    ((127, 128, 129, 0), 256, 320, "silu"),         # the two unit shapes; 128-row units of a width 256 does not divide
    ((192, 193, 256, 257), 256, 256, "silu"),       # three and four column blocks, a full tile, one row more
    ((0, 513, 640, 3), 384, 192, "gelu"),           # several tiles per expert with a rest of 1 and of 128 rows
    ((385, 511, 0), 128, 192, "silu"),              # two tiles of equal size (a remainder of 129 and of 255 rows)
    ((650, 700), 256, 128, "gelu"),                 # three
    ((70,) * 32, 128, 4096, "silu"),                # enough units for 256 weight rows each
    ((300,), 512, 768, "silu"),                     # a single expert
])
def test_dense_16_bit_kernel_against_the_tile_kernel_and_fp64(device, rows, K, N, act, dtype):
    """Unquantized weights: row counts on both sides of the column blocks, the token groups, the two unit shapes and the tile,
    against fp64 and (both add in the same order) bit for bit against the 128 x 128 kernel."""
    from sharktank_amd import _hip

    E, T = len(rows), sum(rows)
    g = torch.Generator().manual_seed(1000 + T)
    x, wg, wu = (torch.randn(s, generator=g).to(dtype) for s in ([T, K], [E, N, K], [E, N, K]))
    wg, wu = wg / K ** 0.5, wu / K ** 0.5
    wd = (torch.randn([E, K, N], generator=g) / N ** 0.5).to(dtype)
    dg, du, dd = (_hip.DeviceWeight(_hip.W_DENSE, E, w.shape[1], w.shape[2], w.to(device), None, None, _hip.dtype_enum(dtype)) for w in (wg, wu, wd))
    idx = torch.repeat_interleave(torch.arange(E), torch.tensor(rows))[torch.randperm(T, generator=g)].to(torch.int32).reshape(T, 1)
    _, offsets, perm, _ = _hip.dispatch_build(idx.to(device), E)
    act_id = _hip.ACT_SILU if act == "silu" else _hip.ACT_GELU_ERF
    z, z_tile = (_hip.grouped_gate_up(x.to(device), dg, du, act_id, offsets, perm, 1, variant=v) for v in (_hip.VARIANT_DENSE, _hip.VARIANT_MFMA_TILE))
    assert torch.equal(z.view(torch.int16), z_tile.view(torch.int16))  # (the same sums, and the activation function as precise)
    pairs = perm.cpu().long()
    xs, e = x[pairs].double(), idx.reshape(-1)[pairs].long()
    want = torch.empty(T, N, dtype=torch.float64)
    for ee in range(E):
        a, b = xs[e == ee] @ wg[ee].double().T, xs[e == ee] @ wu[ee].double().T
        # (four roundings to 16 bits on the way, of at most eps / 2 each)
        want[e == ee] = (torch.nn.functional.silu(a) if act == "silu" else torch.nn.functional.gelu(a)) * b
    eps = 2.0 ** (-11 if dtype == torch.float16 else -8)
    assert O.rel_l2(z.cpu().double(), want) < 2 * eps
    down = {v: _hip.grouped_down(z, dd, offsets, T, 1, variant=v).cpu() for v in (_hip.VARIANT_DENSE, _hip.VARIANT_MFMA_TILE)}
    bits = torch.int16
    assert N % 64 == 0 and (K % 128 == 0 or K == 64)  # (K = 64: the down projection has no tile and runs on the 128 x 128 kernel)
    assert torch.equal(down[_hip.VARIANT_DENSE].view(bits), down[_hip.VARIANT_MFMA_TILE].view(bits))
    auto = _hip.grouped_ffn(x.to(device), dg, du, dd, act_id, offsets, perm, 1)
    y = torch.empty(T, K, dtype=torch.float64)
    for ee in range(E):
        y[e == ee] = z.cpu().double()[e == ee] @ wd[ee].double().T
    assert O.rel_l2(down[_hip.VARIANT_DENSE].double(), y) < eps
    assert O.rel_l2(auto.cpu().double(), y) < 2 * eps  # (a z element may round the other way under another kernel)


@pytest.mark.parametrize("fmt,dtype", [("q8_0", torch.float16), ("q4_1", torch.bfloat16)])
@pytest.mark.parametrize("rows,n_out", [(1, 4096), (16, 4096), (17, 4128), (32, 32), (32, 4096), (5, 1056)])
def test_streamed_single_matrix_items_of_16_and_32_features(device, rows, n_out, fmt, dtype):
    """A single matrix with few rows: items of 16 output features up to 4096 of them, of 32 beyond, one and two token tiles."""
    import moe_cases as MC
    from sharktank_amd import _hip
    from sharktank_amd.ops import device_weight

    g = torch.Generator().manual_seed(rows + n_out)
    w = torch.randn(n_out, 1280, generator=g) * 0.03
    planes = dict(zip(("d", "qs"), O.quantize_q8_0(w))) if fmt == "q8_0" else dict(zip(("d", "m", "qs"), O.quantize_q4_1(w)))
    dw = device_weight(MC.to_inference_tensor(fmt, planes, [n_out, 1280], "w", device), stacked=False, prepack=True)
    x = torch.randn(rows, 1280, generator=g).to(dtype).to(device)
    got, tile = _hip.mmt(x, dw), _hip.mmt(x, dw, variant=_hip.VARIANT_MFMA_TILE)
    # the same products in another order: a value moves by one unit of the last place where the sum sits at a rounding boundary
    assert O.rel_l2(got.cpu().double(), tile.cpu().double()) < 2.0 ** (-11 if dtype == torch.float16 else -8) / 4


@pytest.mark.parametrize("rows", [1, 16, 17])
@pytest.mark.parametrize("N", [12288, 12544, 16384, 16640])
def test_streamed_gate_up_on_both_sides_of_its_splits(device, rows, N):
    """Gate/up of 768 and 1024 items and one tile more: reduction split over a workgroup, whole items, items through LDS."""
    import moe_cases as MC
    from sharktank_amd import _hip
    from sharktank_amd.ops import device_weight

    g = torch.Generator().manual_seed(N + rows)
    dws = []
    for shape in ([N, 1024], [N, 1024], [1024, N]):
        w = torch.randn(shape, generator=g) * 0.03
        dws.append(device_weight(MC.to_inference_tensor("q8_0", dict(zip(("d", "qs"), O.quantize_q8_0(w))), shape, "w", device), stacked=False, prepack=True))
    x = torch.randn(rows, 1024, generator=g).to(torch.float16).to(device)
    got, tile = (_hip.grouped_ffn(x, *dws, _hip.ACT_SILU, None, None, 1, variant=v) for v in (_hip.VARIANT_AUTO, _hip.VARIANT_MFMA_TILE))
    # (see above; the intermediate is rounded as well)
    assert O.rel_l2(got.cpu().double(), tile.cpu().double()) < 2.0 ** -11 / 2


@pytest.mark.parametrize("fmt,dtype", [("q8_0", torch.float16), ("q4_1", torch.bfloat16), ("fp8", torch.float16)])
@pytest.mark.parametrize("rows", [257, 300, 512, 700])
def test_narrow_tiles_of_128_features(device, fmt, dtype, rows):
    """A single matrix whose tiles of 64 features are more than the CUs: tiles of 128 (bit for bit against the 128 x 128 kernel: both
    keep one running sum in the same order), and tiles of 64 where 128 does not divide its features; the gated form beside it."""
    import moe_cases as MC
    from sharktank_amd import _hip
    from sharktank_amd.ops import device_weight

    x = torch.randn(rows, 256, generator=torch.Generator().manual_seed(rows)).to(dtype).to(device)
    for N in (8320, 8384):  # 130 and 131 tiles of 64, two or three tiles of rows
        case = MC.build(MC.Case(T=4, K=256, N=N, E=1, k=1, fmt=fmt, dtype=dtype, seed=430))
        dws = [device_weight(MC.to_inference_tensor(fmt, case.planes[n], [1, N, 256], n, device), stacked=True, prepack=True) for n in ("gate", "up")]
        narrow, tile = (_hip.mmt(x, dws[0], variant=v) for v in (_hip.VARIANT_MFMA_NARROW, _hip.VARIANT_MFMA_TILE))
        assert torch.equal(narrow.view(torch.int16), tile.view(torch.int16))
        idx = torch.zeros(rows, 1, dtype=torch.int32, device=device)
        _, offsets, perm, _ = _hip.dispatch_build(idx, 1)
        got, want = (_hip.grouped_gate_up(x, *dws, _hip.ACT_SILU, offsets, perm, 1, variant=v) for v in (_hip.VARIANT_MFMA_NARROW, _hip.VARIANT_MFMA_TILE))
        # (the same sums; the gated product may be rounded once more or less on the way: one unit of the last place)
        assert O.rel_l2(got.cpu().double(), want.cpu().double()) < 2.0 ** (-11 if dtype == torch.float16 else -8)


@pytest.mark.parametrize("fmt,dtype", [("q8_0", torch.float16), ("q4_1", torch.bfloat16), ("fp8", torch.float16)])
@pytest.mark.parametrize("rows", [1, 49, 192, 193, 257, 384, 385])
def test_narrow_tiles_of_equal_rows(device, fmt, dtype, rows):
    """Narrow tiles of at most 192 rows spread their rows over the four token-row groups: on both sides of every change of the tiling, bit
    for bit against the 128 x 128 kernel (one running sum per output in the same order), 64 and 128 features per tile, plain and gated."""
    import moe_cases as MC
    from sharktank_amd import _hip
    from sharktank_amd.ops import device_weight

    K = 512
    x = torch.randn(rows, K, generator=torch.Generator().manual_seed(rows)).to(dtype).to(device)
    for N in (512, 16640):  # tiles of 64 features; 260 of them are more than the CUs from the first row on: tiles of 128
        case = MC.build(MC.Case(T=4, K=K, N=N, E=1, k=1, fmt=fmt, dtype=dtype, seed=440))
        dws = [device_weight(MC.to_inference_tensor(fmt, case.planes[n], [1, N, K], n, device), stacked=True, prepack=True) for n in ("gate", "up")]
        narrow, tile = (_hip.mmt(x, dws[0], variant=v) for v in (_hip.VARIANT_MFMA_NARROW, _hip.VARIANT_MFMA_TILE))
        assert torch.equal(narrow.view(torch.int16), tile.view(torch.int16))
        got, want = (_hip.grouped_gate_up(x, *dws, _hip.ACT_SILU, None, None, 1, variant=v) for v in (_hip.VARIANT_MFMA_NARROW, _hip.VARIANT_MFMA_TILE))
        # (the same sums; the gated product may be rounded once more or less on the way: one unit of the last place)
        assert O.rel_l2(got.cpu().double(), want.cpu().double()) < 2.0 ** (-11 if dtype == torch.float16 else -8)


def test_probe_takes_a_device_without_an_index(device):
    from sharktank_amd import _hip

    for dev in ("cuda", torch.device("cuda"), device):
        assert _hip.probe_mfma(dev, iters=100, launches=1, warm_launches=1) > 0
