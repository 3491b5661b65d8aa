"""Host-side mirror of the reference interfaces: dispatch protocol, Theta, tensor wrappers (no GPU needed)."""

import pytest
import torch

import moe_cases as MC
from sharktank_amd import ops
from sharktank_amd import types as ST
from sharktank_amd.ops._registry import AllOfType, AnyOfType, overridable


def test_override_protocol_and_failure_message():
    @overridable
    def myop(a, b):
        ...

    @myop.trampoline
    def _t(d, a, b):
        for o in d.find_overrides((a, b)):
            r = o(a, b)
            if r is not NotImplemented:
                return o, r
        d.fail((a, b))

    calls = []

    @myop.override(torch.Tensor, torch.Tensor)
    def first(a, b):
        calls.append("first")
        return "first"

    @myop.override(torch.Tensor, torch.Tensor)
    def second(a, b):
        calls.append("second")
        return NotImplemented

    t = torch.zeros(1)
    assert myop(t, t) == "first" and calls == ["second", "first"]  # later registration is tried first
    # PrimitiveTensor auto-unboxes to Tensor; QuantizedTensor does not unless auto_dequant
    assert myop(ST.DefaultPrimitiveTensor(data=t), t) == "first"
    q = ST.PlanarQuantizedTensor(shape=[1, 32], layout=ST.BlockScaledLayout([1, 32], torch.zeros(1, 1, 1), torch.zeros(1, 1, 32, dtype=torch.int8)))
    # message format pinned by the reference's test (sharktank/tests/ops/ops_test.py:109-116)
    with pytest.raises(NotImplementedError, match=r"Overridable operator.+does not have an implementation for argument types:.+"):
        myop(t, q)

    @myop.override(AllOfType(torch.Tensor, ST.QuantizedTensor), salience=5)
    def high(a, b):
        return "high"

    assert myop(t, q) == "high" and myop(t, t) == "high"
    assert AnyOfType(int)(str, int) and not AnyOfType(int)(str, str)


def test_last_op_dispatch_hook():
    ops._test_enable_last_op_dispatch(True)
    try:
        t = ST.DefaultPrimitiveTensor(data=torch.zeros(2, 3))
        ops.view(t, (3, 2))
        assert ops._test_get_last_op_dispatch().__name__ == "view_default"
    finally:
        ops._test_enable_last_op_dispatch(False)


def test_quantized_matmul_without_kernel_raises_not_implemented():
    # matmul(Tensor, QuantizedTensor) with transpose_rhs=False has no kernel: every override declines
    q = ST.PlanarQuantizedTensor(shape=[4, 32], layout=ST.BlockScaledLayout([4, 32], torch.zeros(4, 1, 1, dtype=torch.float16), torch.zeros(4, 1, 32, dtype=torch.int8)))
    with pytest.raises(NotImplementedError, match="does not have an implementation"):
        ops.matmul(torch.zeros(2, 32), q, transpose_rhs=False)


def test_theta_accessors():
    a = ST.DefaultPrimitiveTensor(name="ffn_norm.weight", data=torch.ones(4))
    b = ST.DefaultPrimitiveTensor(name="ffn_gate_exps.weight", data=torch.ones(2, 3, 4))
    theta = ST.Theta([a, b])
    assert set(theta.keys) == {"ffn_norm", "ffn_gate_exps"}
    assert theta.tensor("ffn_gate_exps", "weight") is b
    assert theta("ffn_norm").tensor("weight") is a
    assert theta.optional_tensor("layer_output_norm") is None
    with pytest.raises(KeyError):
        theta.tensor("nope")
    assert set(theta.flatten()) == {"ffn_norm.weight", "ffn_gate_exps.weight"}


def test_planar_globals_and_clone():
    d = torch.ones(2, 1, 1, dtype=torch.float16)
    m = torch.zeros(2, 1, 1, dtype=torch.float16)
    qs = torch.zeros(2, 1, 16, dtype=torch.uint8)
    q = ST.PlanarQuantizedTensor(name="w", shape=[2, 32], layout=ST.BlockScaledI4Layout([2, 32], d, qs, m=m, signed=False))
    assert set(q.globals) == {"w:d", "w:m", "w:qs"}
    moved = q.to(device="cpu")
    assert isinstance(moved.unpack(), ST.BlockScaledI4Layout) and moved.unpack().signed is False
    assert moved.layout_type is ST.BlockScaledI4Layout


def test_gguf_raw_views_carry_no_arithmetic():
    raw = torch.zeros(2 * 34, dtype=torch.uint8)
    lay = ST.Q8_0(raw=raw, shape=[2, 32]).unpack()
    assert lay.d.shape == (2, 1, 1) and lay.qs.shape == (2, 1, 32) and lay.d.dtype == torch.float16
    raw4 = torch.zeros(2 * 20, dtype=torch.uint8)
    lay4 = ST.Q4_1(raw=raw4, shape=[2, 32]).unpack()
    assert lay4.qs_bit_packed.shape == (2, 1, 16) and lay4.m.shape == (2, 1, 1)


def test_layers_refuse_host_tensors():
    from sharktank_amd.layers import RMSNormLayer

    theta = ST.Theta([ST.DefaultPrimitiveTensor(name="weight", data=torch.ones(8))])
    with pytest.raises(RuntimeError, match="GPU only"):
        RMSNormLayer(theta)(torch.zeros(2, 8))


def test_unknown_activation_is_rejected():
    from sharktank_amd.layers.ffn_moe_block import activation_enum

    with pytest.raises(NotImplementedError):
        activation_enum(torch.tanh)


def _tiny_theta(**extra):
    E, N, K = 2, 32, 64
    tensors = {
        "ffn_gate_inp.weight": ST.DefaultPrimitiveTensor(name="ffn_gate_inp.weight", data=torch.zeros(E, K)),
        "ffn_norm.weight": ST.DefaultPrimitiveTensor(name="ffn_norm.weight", data=torch.ones(K)),
        "ffn_gate_exps.weight": ST.DefaultPrimitiveTensor(name="ffn_gate_exps.weight", data=torch.zeros(E, N, K)),
        "ffn_up_exps.weight": ST.DefaultPrimitiveTensor(name="ffn_up_exps.weight", data=torch.zeros(E, N, K)),
        "ffn_down_exps.weight": ST.DefaultPrimitiveTensor(name="ffn_down_exps.weight", data=torch.zeros(E, K, N)),
    }
    tensors.update(extra)
    return ST.Theta(tensors)


def test_router_with_bias_is_refused():
    """The fused forward reads the router matrix only; a bias that a LinearLayer would add must not vanish silently."""
    from sharktank_amd.layers import MoeBlock

    MoeBlock(_tiny_theta(), 2, 1, 1e-5)  # a plain router builds
    bias = ST.DefaultPrimitiveTensor(name="ffn_gate_inp.bias", data=torch.zeros(2))
    with pytest.raises(NotImplementedError, match="ffn_gate_inp"):
        MoeBlock(_tiny_theta(**{"ffn_gate_inp.bias": bias}), 2, 1, 1e-5)


def test_unused_reference_alternatives_are_named():
    """PreGatherFFNMOE.one_hot_matmul exists in the reference (with a hard-wired 8 experts) and is never called by its forward."""
    from sharktank_amd.layers import PreGatherFFNMOE

    ffn = PreGatherFFNMOE(_tiny_theta())
    with pytest.raises(NotImplementedError, match="unused by forward"):
        ffn.one_hot_matmul(None, None, None)


def _ffn_weights(K, N, N_up=None, N_down=None, d_dtype=torch.float16):
    def q8(rows, cols):
        layout = ST.BlockScaledLayout([rows, cols], torch.ones(rows, cols // 32, 1, dtype=d_dtype), torch.zeros(rows, cols // 32, 32, dtype=torch.int8))
        return ST.PlanarQuantizedTensor(shape=[rows, cols], layout=layout)

    return q8(N, K), q8(N_up or N, K), q8(K, N_down or N)


@pytest.mark.parametrize("K,N,width", [(256, 256, None), (256, 704, 768), (256, 160, 256), (256, 128, None), (256, 320, 512), (256, 288, None),
                                       (288, 288, None), (2880, 2880, None), (512, 2880, 3072)])
def test_ffn_widths_that_are_padded(K, N, width):
    from sharktank_amd.ops.hip_impls import padded_ffn_width

    assert padded_ffn_width(*_ffn_weights(K, N)) == width


def test_ffn_weights_of_different_widths_are_not_padded_to_one():
    """Gate, up and down of widths that round up to the same multiple of 256 do not fit each other; the calls must get to see that."""
    from sharktank_amd.ops.hip_impls import padded_ffn_width

    assert padded_ffn_width(*_ffn_weights(256, 704, N_up=736)) is None
    assert padded_ffn_width(*_ffn_weights(256, 704, N_down=736)) is None


@pytest.mark.parametrize("refusing", [0, 1, 2, None])
def test_a_refused_padding_is_given_back_and_remembered(monkeypatch, refusing):
    """A weight whose values keep it out of the streaming order (Q4_1 block scales): the other two keep no padded copy beside the
    descriptors that are used, and later calls build nothing."""
    from types import SimpleNamespace

    from sharktank_amd.ops import hip_impls

    weights = _ffn_weights(256, 704)
    built = []

    def device_weight(w, *, stacked, prepack=False, pad=(None, None)):
        i = next(i for i, x in enumerate(weights) if x is w)
        built.append((i, pad))
        return SimpleNamespace(is_packed=i != refusing, pad=pad, weight=i)

    monkeypatch.setattr(hip_impls, "device_weight", device_weight)
    first = hip_impls.ffn_device_weights(*weights, stacked=False, prepack=True, cache=True)
    n_built = len(built)
    assert hip_impls.ffn_device_weights(*weights, stacked=False, prepack=True, cache=True) == first and len(built) == n_built
    assert [d.weight for d in first] == [0, 1, 2]
    if refusing is None:
        assert [d.pad for d in first] == [(768, None), (768, None), (None, 768)] and n_built == 3
    else:
        assert [d.pad for d in first] == [(None, None)] * 3 and n_built == 3 + refusing + 1
    for w, used in zip(weights, first):  # (nothing is kept that is not used)
        kept = [d for _, d in hip_impls._descriptor_store(w).values() if d is not None]
        assert kept == [used]


def test_planes_of_64_gb_stay_planar():
    """stmoe_prepack refuses them, so a weight of that size must not be sent there."""
    from sharktank_amd import _hip

    w = object.__new__(_hip.DeviceWeight)
    w.format, w.experts, w.rows, w.cols = _hip.W_Q8_0, 64, 32768, 32768 - 256
    assert w.can_prepack()
    assert not w.can_prepack(cols=32768)
    w.cols = 32768
    assert not w.can_prepack()
    assert _hip.packable_size(_hip.W_Q4_1, 64, 32768, 32768) and not _hip.packable_size(_hip.W_Q4_1, 128, 32768, 32768)


def test_padded_layers_that_fitted_the_built_in_workspace_still_do():
    """A layer of a padded width is called with that width: what its own width needed of 16 MiB must not become too much."""
    from sharktank_amd import _hip

    for dtype in (torch.float16, torch.float32):
        for T, k in ((1, 2), (64, 2), (128, 1), (21, 6), (200, 1)):
            for K in (256, 2048, 8192):
                need = lambda n: _hip.moe_forward_workspace_bytes(T, k, 8, K, n, dtype)
                for n in range(32, 1 << 18, 1024 + 32):
                    if need(n) > 16 << 20:
                        break
                    assert need((n + 255) // 256 * 256) <= _hip.STATIC_SCRATCH_BYTES, (T, k, K, n)


@pytest.mark.parametrize("counts,rows", [
    ([65, 65, 65, 65, 64, 64, 64, 64], 96),      # 192 units of 64 rows: one round; 128 of 96: half a round
    ([129, 129, 129, 49, 40, 20, 10, 10], 64),   # 224 and 176: one round either way
    ([97, 97, 97, 97, 97, 10, 10, 11], 64),      # 208 and 208
    ([172, 172, 172, 0, 0, 0, 0, 0], 96),        # 144 and 96
    ([200, 200, 116, 0, 0, 0, 0, 0], 96),        # 160 and 128
])
def test_units_of_the_register_kernel_follow_the_rows_of_the_experts(counts, rows):
    """A launch that the automatic choice gives units of up to 96 rows takes them only where they save half a round; the sizes alone (8 experts
    of 1024 x 2048, 516 pairs) do not tell."""
    assert sum(counts) == 516
    assert MC.unit_rows("q4_1", torch.float16, True, 8, 4, 129, 1024, 2048) == 96
    assert MC.unit_rows("q4_1", torch.float16, True, 8, 4, 129, 1024, 2048, counts) == rows


@pytest.mark.parametrize("E,k,T,n_out,rows", [
    (4, 2, 120, 7168, 96),    # 60 rows on each of 4 experts, 224 units
    (4, 2, 121, 7168, 0),     # from 61 on an expert of an uneven routing spills into a second round too often
    (4, 2, 160, 6144, 96),    # 192 units
    (8, 2, 310, 3584, 96),    # eight experts
    (32, 4, 608, 1024, 96),   # 76 rows on each of 32 experts, 256 units
    (32, 4, 609, 1024, 0),
])
def test_nearly_full_rounds_of_wide_units(E, k, T, n_out, rows):
    """Where one unit per expert and feature tile nearly fills a round of the CUs and the experts are few or very many."""
    assert MC.unit_rows("q4_1", torch.bfloat16, True, E, k, T, 4096, n_out) == rows


def test_one_unit_per_expert_up_to_56_rows():
    """226 pairs on 4 experts, 136 units: a seventh more than the average is 64.57 rows, which counts as one unit of 64."""
    assert MC.unit_rows("fp8", torch.float16, True, 4, 2, 113, 2048, 4352) == 64


@pytest.mark.parametrize("fmt,dtype,gate_up,T,kred,n_out,rows", [
    ("q8_0", torch.float16, False, 160, 4096, 14336, 80),    # 168 units of 64 rows; 112 of 80 run as halves
    ("q8_0", torch.float16, False, 300, 4096, 14336, 75),    # 280; 224 of 75 fit one round
    ("q8_0", torch.float16, False, 256, 4096, 14336, 0),     # 224 of 64
    ("q8_0", torch.float16, False, 385, 4096, 14336, 0),     # 280 of 96
    ("q8_0", torch.float16, False, 100, 4096, 14336, 64),    # 112 of 64
    ("q4_1", torch.bfloat16, True, 130, 4096, 8192, 65),     # gate/up: 192 of 64; 128 of 65
    ("q8_0", torch.float16, False, 272, 8192, 13568, 68),
    ("q8_0", torch.float16, False, 272, 8448, 13568, 0),     # reductions that the prefill kernel cuts
    ("q8_0", torch.bfloat16, False, 272, 6144, 13568, 68),
    ("q8_0", torch.bfloat16, False, 272, 6400, 13568, 0),    # ... from shorter ones on where the conversion is slowest
    ("q4_1", torch.bfloat16, False, 272, 8192, 13568, 68),
    ("q8_0", torch.bfloat16, False, 160, 8192, 14336, 80),   # (halves: all formats)
    ("q8_0", torch.float16, False, 160, 2048, 14336, 0),     # from 129 rows on, more than 2048 elements
    ("q8_0", torch.float16, False, 128, 2048, 14336, 64),
])
def test_units_of_a_single_matrix(fmt, dtype, gate_up, T, kred, n_out, rows):
    """One matrix on both sides of the lines around tiles of 64 and of up to 96 rows: as few tiles as run as halves, or as many as fit one round."""
    assert MC.unit_rows(fmt, dtype, gate_up, 1, 1, T, kred, n_out) == rows


@pytest.mark.parametrize("fmt,dtype,gate_up,E,k,T,kred,n_out,scratch,rows", [
    ("q4_1", torch.bfloat16, True, 8, 2, 208, 1024, 8192, True, 64),    # 52 rows per expert
    ("q4_1", torch.bfloat16, True, 8, 2, 212, 1024, 8192, True, 96),    # 53: some expert has more than 64
    ("q4_1", torch.bfloat16, True, 8, 2, 288, 1024, 8192, True, 96),    # 72 ...
    ("q4_1", torch.bfloat16, True, 8, 2, 292, 1024, 8192, True, 0),
    ("q4_1", torch.bfloat16, True, 8, 2, 320, 2048, 8192, True, 96),    # ... and 80 with 2048 elements
    ("q4_1", torch.bfloat16, True, 8, 2, 324, 2048, 8192, True, 0),
    ("q8_0", torch.float16, True, 8, 2, 240, 1792, 4096, True, 0),      # a short reduction of a format that converts fast
    ("q8_0", torch.float16, True, 8, 2, 240, 2048, 4096, True, 96),
    ("q8_0", torch.float16, False, 8, 2, 560, 3072, 3072, True, 96),    # two tiles of 140 rows: 192 units
    ("q8_0", torch.float16, False, 8, 2, 560, 9216, 2304, True, 0),     # 144 leave CUs idle
    ("fp8", torch.bfloat16, False, 8, 2, 560, 3072, 2048, True, 96),    # 128 run as halves
    ("q8_0", torch.bfloat16, True, 33, 2, 396, 2048, 1024, True, 64),   # several rounds: 24 rows per expert with up to 2048 elements
    ("q8_0", torch.bfloat16, True, 33, 2, 397, 2048, 1024, True, 0),
    ("q8_0", torch.bfloat16, True, 33, 2, 397, 2304, 1024, True, 64),
    ("fp8", torch.bfloat16, False, 4, 2, 67, 8448, 1024, True, 0),      # units for a quarter of the CUs, a reduction that can be cut
    ("fp8", torch.bfloat16, False, 4, 2, 67, 8448, 1024, False, 64),    # ... where there is scratch
    ("q4_1", torch.bfloat16, False, 8, 2, 16, 3072, 4096, True, 64),    # streamed launches
    ("q8_0", torch.float16, True, 8, 2, 16, 4096, 14336, True, 0),
])
def test_units_of_grouped_launches(fmt, dtype, gate_up, E, k, T, kred, n_out, scratch, rows):
    """Several experts on both sides of the lines."""
    assert MC.unit_rows(fmt, dtype, gate_up, E, k, T, kred, n_out, scratch=scratch) == rows
