"""The C-ABI library loads without a GPU and exports every symbol the public header declares."""

import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "sharktank_moe_hip.h")


def declared_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(stmoe_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_expected_entry_points():
    syms = declared_symbols()
    for name in ("stmoe_router_topk", "stmoe_dispatch_build", "stmoe_grouped_ffn", "stmoe_combine", "stmoe_moe_forward",
                 "stmoe_dequant_block_scaled", "stmoe_dequant_block_scaled_i4", "stmoe_dequant_tensor_scaled", "stmoe_mmt"):
        assert name in syms


def test_library_exports_every_declared_symbol():
    from sharktank_amd import _hip

    lib = ctypes.CDLL(_hip.library_path())
    for name in declared_symbols():
        assert hasattr(lib, name), f"{name} declared in the header but not exported"


def test_binding_table_matches_header():
    from sharktank_amd import _hip

    assert sorted(_hip.SIGNATURES) == declared_symbols()


def test_argument_validation_without_a_gpu():
    """Status codes come back before any launch, so these calls are safe on a host without a GPU."""
    from sharktank_amd import _hip

    lib = _hip.load_library()
    assert lib.stmoe_abi_version() == 1
    assert lib.stmoe_router_topk(None, None, _hip.F16, 4, 30, 8, 2, None, None, None, None, None) == 2  # K % 8
    assert b"multiple of 8" in lib.stmoe_last_error()
    assert lib.stmoe_router_topk(None, None, _hip.F16, 4, 64, 8, 9, None, None, None, None, None) == 2  # k > E
    assert lib.stmoe_router_topk(None, None, _hip.F16, 4, 64, 8, 2, None, None, None, None, None) == 1  # NULL
    assert lib.stmoe_router_topk(None, None, _hip.F16, 0, 64, 8, 2, None, None, None, None, None) == 0  # zero tokens
    assert lib.stmoe_dispatch_build(None, 0, 0, None, None, None, None, None) == 2
    assert lib.stmoe_dequant_block_scaled(None, None, _hip.F16, None, 0, 32, None, _hip.F16, None) == 0
    assert lib.stmoe_grouped_ffn_workspace_bytes(32, 2, 4096, 14336, _hip.F16) == 32 * 2 * 14336 * 2 + 32 * 4096 * 2 + 32 * 2 * 14336  # z, copy of x, fp8 z
    w = _hip.StmoeWeight(format=_hip.W_Q8_0, dtype=0, experts=8, rows=64, cols=48, qs=16, d=16, m=None, d_count=1)
    rc = lib.stmoe_grouped_ffn(None, _hip.F16, 4, 48, 64, 8, 2, ctypes.byref(w), ctypes.byref(w), ctypes.byref(w), 0,
                               None, None, None, None, None, None, 0, 0, None)
    assert rc == 2 and b"32" in lib.stmoe_last_error()  # Q8_0 needs cols % 32 == 0
    assert lib.stmoe_dynamic_quantize_fp8_scratch_bytes() == 4096
    assert lib.stmoe_probe_mfma(0, 1, 400, None, None, None) == 1  # NULL sink
    assert lib.stmoe_probe_mfma(2, 1, 400, 16, None, None) == 2  # unknown kind
    assert lib.stmoe_probe_mfma(0, 1, 402, 16, None, None) == 2  # iters not a multiple of 4
    assert lib.stmoe_dynamic_quantize_fp8(None, _hip.F16, 8, None, 16, 16, 16, None) == 6  # scratch too small
    assert lib.stmoe_dynamic_quantize_fp8(None, _hip.F16, 8, None, 16, 16, 4096, None) == 1  # NULL x
    # raw GGUF blocks: shape, format pairing and streaming-order constraints are checked before any launch
    assert lib.stmoe_gguf_ingest(16, _hip.GGUF_Q8_0, ctypes.byref(w), None) == 2
    w2 = _hip.StmoeWeight(format=_hip.W_Q4_1, dtype=0, experts=1, rows=16, cols=64, qs=16, d=16, m=16, d_count=1)
    assert lib.stmoe_gguf_ingest(16, _hip.GGUF_Q8_0, ctypes.byref(w2), None) == 5  # Q8_0 blocks cannot become Q4_1 planes
    assert lib.stmoe_gguf_ingest(17, _hip.GGUF_Q4_1, ctypes.byref(w2), None) == 4  # odd address
    w2.format = _hip.W_Q4_1_PACKED
    assert lib.stmoe_gguf_ingest(16, _hip.GGUF_Q4_1, ctypes.byref(w2), None) == 2 and b"256" in lib.stmoe_last_error()
    w2.rows = 0
    assert lib.stmoe_gguf_ingest(16, _hip.GGUF_Q4_1, ctypes.byref(w2), None) == 2  # still not whole 256-column pieces
    w2.format, w2.cols = _hip.W_Q4_1, 64
    assert lib.stmoe_gguf_ingest(16, _hip.GGUF_Q4_1, ctypes.byref(w2), None) == 0  # nothing to do


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    from sharktank_amd import _hip

    monkeypatch.setattr(_hip, "_lib", None)
    monkeypatch.setattr(_hip, "_LIB_PATH", str(tmp_path / "nope.so"))
    with pytest.raises(RuntimeError, match="is missing"):
        _hip.load_library()


def test_hand_scheduled_kernels_get_no_scratch_accesses_from_the_compiler():
    """The prefill and register kernels and the one of unquantized weights issue loads by hand and wait for them with counted `s_waitcnt vmcnt(N)`.  That count only
    holds while the compiler adds no vector-memory instruction of its own to those wavefronts: a register spilled to scratch
    memory would be one (and a spill of a register with a load in flight would read it too early).  The build keeps the
    compiler's per-kernel resource report beside the library; every instance of those kernels must show no scratch and no
    spilled vector register."""
    from sharktank_amd import _hip

    report = os.path.splitext(_hip.library_path())[0] + ".resources.txt"
    assert os.path.exists(report), f"{report} is missing: build with the Makefile (make -C shark-platform_amd/csrc)"
    kernels, name = {}, None
    for line in open(report):
        key, _, value = line.strip().partition(": ")
        if key == "Function Name":
            name = value
            kernels[name] = {}
        elif name is not None:
            kernels[name][key] = value
    instances = {
        "grouped_mfma_ws_kernel": 2 * 3 * 2,  # types x formats x (gate/up, down)
        "grouped_mfma_reg_kernel": 2 * 3 * 2 * 2,  # ... x units of up to 64 and of up to 96 rows
        "grouped_fp8_ws_kernel": 2 * 2,
        "grouped_dense_kernel": 2 * 2 * 2,  # types x (gate/up, down) x 128 or 256 weight rows
    }
    hand = {n: r for n, r in kernels.items() if any(k in n for k in instances)}
    for kernel, count in instances.items():
        assert sum(kernel in n for n in hand) == count, (kernel, sorted(hand))
    for n, r in hand.items():
        assert r["ScratchSize [bytes/lane]"] == "0", (n, r)
        assert r["VGPRs Spill"] == "0", (n, r)
        if "grouped_mfma_ws_kernel" in n:
            assert int(r["VGPRs"]) <= 168, (n, r)  # 12 wavefronts per CU
    # The fp32 kernel keeps two chunks of loads in flight by their order alone; a register in scratch memory would come back behind them.
    f32 = {n: r for n, r in kernels.items() if "grouped_f32_kernel" in n}
    assert len(f32) == 9 * 3 * 2, sorted(f32)  # weight formats x (gate/up, down of 32 and of 16 features) x whole or ragged reductions
    for n, r in f32.items():
        assert r["ScratchSize [bytes/lane]"] == "0", (n, r)


def test_hand_issued_loads_wait_for_their_base(tmp_path):
    """A vector-memory instruction may read a scalar register that a vector instruction wrote only five wait states later.  The compiler
    sees to that for its own instructions, not for those inside inline assembly.  In the built library no vector-memory instruction
    reads such a register too early, and in the kernels whose bases pass through vector instructions (or come back from a scalar spill,
    the same thing) every load into LDS carries the wait states itself, so that no register allocation can break one."""
    import re
    import shutil
    import subprocess

    from sharktank_amd import _hip

    objdump = "/opt/rocm/llvm/bin/llvm-objdump"
    if not os.path.exists(objdump):
        pytest.skip("no llvm-objdump")
    lib = str(tmp_path / "lib.so")
    shutil.copy(_hip.library_path(), lib)
    subprocess.run([objdump, "--offloading", lib], check=True, stdout=subprocess.DEVNULL, cwd=tmp_path)
    memory = re.compile(r"(?:global|buffer|scratch)_\w+ .*?s\[(\d+):(\d+)\]")
    vector_write = re.compile(r"v_(?:readlane_b32|readfirstlane_b32|cmp\w*) s(?:(\d+)|\[(\d+):(\d+)\]),")
    scalar_write = re.compile(r"s_\w+ s(?:(\d+)|\[(\d+):(\d+)\]),")
    span = lambda m: [int(m[1])] if m[1] else range(int(m[2]), int(m[3]) + 1)  # noqa: E731
    waiting, bad = {"grouped_fp8_ws_kernel": 0, "grouped_mfma_reg_kernel": 0}, []
    for obj in sorted(tmp_path.glob("*gfx950")):
        text = subprocess.run([objdump, "-d", "--no-show-raw-insn", str(obj)], check=True, capture_output=True, text=True).stdout
        if "global_load_lds_dwordx4" not in text:  # (the kernels that issue loads by hand all have some of these)
            continue
        written, last_nop = {}, 0  # scalar register -> wait states since a vector instruction wrote it; those of a directly preceding s_nop
        kernel = None
        for line in text.splitlines():
            if not line.startswith("\t"):  # (a label: what precedes it in the listing still counts, as if fallen through)
                if line.endswith(">:") and "L0" not in line:
                    kernel = next((k for k in waiting if k in line), None)
                continue
            ins = line.split("//")[0].strip()
            if kernel and ins.startswith("global_load_lds_dwordx4"):
                waiting[kernel] += 1
                if last_nop < 5:
                    bad.append((kernel, ins))
            m = memory.match(ins)
            if m and any(written.get(r, 5) < 5 for r in span((None, None, m[1], m[2]))):
                bad.append(ins)
            nop = re.match(r"s_nop (\w+)", ins)
            last_nop = int(nop[1], 0) + 1 if nop else 0
            written = {r: n + max(last_nop, 1) for r, n in written.items() if n < 5}
            m = vector_write.match(ins)
            if m:
                written.update((r, 0) for r in span(m))
            m = scalar_write.match(ins)
            if m:
                for r in span(m):
                    written.pop(r, None)
    assert all(waiting.values()) and not bad, (waiting, len(bad), bad[:5])
