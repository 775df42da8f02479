"""CPU checks of the native artefacts: the C-ABI library loads and exports
every symbol include/wush_int4.h declares; argument validation rejects bad
calls before any device work; the torch module exposes the reference's 16 ops
(reference csrc/bindings.cpp:28-68) and rejects CPU tensors like the
reference does.  No kernel is launched here (there is no GPU)."""
from __future__ import annotations

import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "wush_int4.h")
INVALID = 1  # hipErrorInvalidValue

REFERENCE_OPS = [
    "quant_int4_tensor_scale", "quant_int4_tensor_scale_dev", "quant_int4", "w4a4_gemm",
    "w4a4_gemm_v1", "w4a4_gemm_cutlass", "w4a4_gemm_cutlass_dev", "w4a4_gemm_s4",
    "s4_atom_selftest", "w4a4_gemv", "w4a4_gemv_multi", "fused_transform_quant_int4_v3",
    "fused_transform_quant_int4_smallm", "fused_transform_quant_int4", "w4a4_gemm_v2",
    "fused_transform_quant_int4_wmma",
]


def declared_symbols():
    text = open(HEADER).read()
    return sorted(set(re.findall(r"^\s*(?:const\s+)?[a-z_0-9]+\s*\*?\s*(wush_[a-z0-9_]+)\s*\(", text, re.M)))


@pytest.fixture(scope="module")
def capi():
    import torch  # noqa: F401
    from wush_int4_kernel_amd import capi as c
    c.load()
    return c


def test_header_declares_expected_entry_points():
    syms = declared_symbols()
    for s in ["wush_quant_int4", "wush_fused_tq", "wush_gemv_int4", "wush_gemm_s4",
              "wush_gemm_s4_workspace_bytes", "wush_mfma_selftest", "wush_quant_int4_tensor_scale",
              "wush_gemm_s4_tensor_scale", "wush_abi_version", "wush_error_string",
              "wush_gemv_int4_supported"]:
        assert s in syms, s


def test_library_exports_every_declared_symbol(capi):
    lib = capi.load()
    for s in declared_symbols():
        assert hasattr(lib, s), s
    assert set(declared_symbols()) == set(capi.SIGNATURES)
    assert lib.wush_abi_version() == 1


def test_library_exports_no_undeclared_c_symbols():
    import subprocess
    out = subprocess.run(["nm", "-D", "--defined-only", os.path.join(ROOT, "wush_int4_kernel_amd", "libwush_int4.so")],
                         capture_output=True, text=True).stdout
    exported = sorted(set(re.findall(r" T (wush_[a-z0-9_]+)$", out, re.M)))
    assert exported == declared_symbols()


def test_lds_dma_waits_for_its_m0_write(tmp_path):
    # gfx950 needs one wait state between a scalar write of M0 and the LDS DMA
    # that takes its LDS address from M0.  The compiler inserts it for its own
    # instructions, not inside the asm strings of wush_device.h, so the built
    # code is checked: no DMA directly behind a write of M0.  Nor does it see
    # that such an asm reads an SGPR as a vector memory address, which needs
    # five wait states after a VALU write of that SGPR.
    import glob
    import shutil
    import subprocess
    objdump = "/opt/rocm/llvm/bin/llvm-objdump"
    lib = shutil.copy(os.path.join(ROOT, "wush_int4_kernel_amd", "libwush_int4.so"), tmp_path)
    subprocess.run([objdump, "--offloading", lib], cwd=tmp_path, capture_output=True, check=True)
    dmas, early = 0, []
    for obj in sorted(glob.glob(str(tmp_path / "*gfx950"))):
        text = subprocess.run([objdump, "-d", "--no-show-raw-insn", obj], capture_output=True, text=True,
                              check=True).stdout
        ins = [line.split("//")[0].strip() for line in text.splitlines() if line.startswith("\t")]
        for i, op in enumerate(ins):
            if not re.match(r"(global|buffer|flat|scratch)_", op):
                continue
            if re.match(r"global_load_lds_|buffer_load_\w+ .*\blds\b", op):
                dmas += 1
                if re.match(r"s_\w+ m0,", ins[i - 1]):
                    early.append((ins[i - 1], op))
            sgprs = {r for a, b in re.findall(r"\bs\[(\d+):(\d+)\]", op) for r in range(int(a), int(b) + 1)}
            waited = 0
            for prev in reversed(ins[max(0, i - 5):i]):
                wrote = re.match(r"v_\w+ s(?:(\d+)|\[(\d+):(\d+)\]),", prev)
                if wrote and waited < 5:
                    lo, hi = (int(wrote[1] or wrote[2]), int(wrote[1] or wrote[3]))
                    if sgprs & set(range(lo, hi + 1)):
                        early.append((prev, op))
                nop = re.match(r"s_nop (\d+)", prev)
                waited += int(nop[1]) + 1 if nop else 1
    assert dmas > 500                    # every DMA kernel was seen
    assert not early, f"{len(early)} of {dmas}: {early[:3]}"


def test_argument_validation_without_device(capi):
    lib = capi.load()
    P = ctypes.c_void_p
    # empty work succeeds without touching the device
    assert lib.wush_quant_int4(None, 0, None, None, 0, None) == 0
    assert lib.wush_fused_tq(None, None, None, None, 0, 32, None) == 0
    assert lib.wush_gemm_s4(None, None, None, None, None, 0, 8, 64, None, 0, None) == 0
    # bad arguments are rejected before any launch
    assert lib.wush_quant_int4(None, 0, None, None, 4, None) == INVALID
    assert lib.wush_quant_int4(P(16), 9, P(16), P(16), 4, None) == INVALID       # dtype
    assert lib.wush_quant_int4(P(8), 0, P(16), P(16), 4, None) == INVALID        # misaligned x
    assert lib.wush_fused_tq(P(16), P(16), P(16), P(16), 1, 48, None) == INVALID  # K % 32
    assert lib.wush_gemv_int4(P(16), P(16), P(16), P(16), P(16), 9, 4, 64, None) == INVALID  # M > 8
    assert lib.wush_gemv_int4(P(16), P(16), P(16), P(16), P(16), 8, 4, 1 << 20, None) == INVALID  # LDS
    assert lib.wush_gemm_s4(P(16), P(16), P(16), P(16), P(16), 4, 4, 40, None, 0, None) == INVALID
    # rows at a time: a multiple of 64 or all of them, the workspace whole
    assert lib.wush_gemm_s4_rows(None, None, None, None, None, 0, 8, 64, 64, None, 0, None) == 0
    for M, rows in ((100, 33), (100, 0), (64, -64)):
        assert lib.wush_gemm_s4_rows(P(16), P(16), P(16), P(16), P(16), M, 4, 64, rows, None, 0, None) == INVALID
    need = lib.wush_gemm_s4_rows_workspace_bytes(P(16), P(16), P(16), P(16), 2048, 4096, 4096, 64)
    assert 0 < need < lib.wush_gemm_s4_best_workspace_bytes(2048, 4096, 4096)
    assert lib.wush_gemm_s4_rows(P(16), P(16), P(16), P(16), P(16), 2048, 4096, 4096, 64, P(16), need - 1, None) == INVALID
    assert lib.wush_gemm_s4_tensor_scale(P(16), P(16), P(16), 4, 4, 1 << 21, 1.0, None, None) == INVALID
    # int32 bound of the per-tensor GEMM: 256 * 64 * K < 2^31 for K <= 131040
    assert 256 * 64 * 131040 < 2 ** 31 <= 256 * 64 * (131040 + 32)
    assert lib.wush_gemm_s4_tensor_scale(P(16), P(16), P(16), 4, 4, 131040 + 32, 1.0, None, None) == INVALID
    assert lib.wush_gemm_s4_tensor_scale(P(16), P(16), P(16), 0, 4, 131040, 1.0, None, None) == 0  # empty, valid
    assert lib.wush_quant_int4_tensor_scale(P(16), P(16), 40, 1.0, None, None) == INVALID
    assert lib.wush_mfma_selftest(None, None, None, None) == INVALID
    assert b"invalid argument" in lib.wush_error_string(INVALID)


def test_workspace_plan_is_host_only(capi):
    # split-K across workgroups only for skinny shapes with few row blocks and
    # a long K (each wavefront of the in-workgroup K split keeps >= 2 stages)
    assert capi.gemm_s4_workspace_bytes(8, 1024, 16384) > 0
    assert capi.gemm_s4_workspace_bytes(8, 4096, 4096) == 0
    assert capi.gemm_s4_workspace_bytes(4096, 4096, 4096) == 0
    assert capi.gemm_s4_workspace_bytes(0, 4096, 4096) == 0
    assert capi.gemm_s4_workspace_bytes(8, 4096, 40) == 0


def test_best_workspace_bytes_against_the_base(capi):
    # never less than wush_gemm_s4_workspace_bytes; equal wherever the same
    # plan runs (M <= 64, K % 64 != 0, wide weights, little work), above it
    # where the converted-activation plan takes over
    for M, N, K in [(8, 1024, 16384), (64, 4096, 4096), (2048, 4096, 4128), (4096, 57344, 8192), (203, 8192, 8192),
                    (96, 4096, 4096), (0, 4096, 4096), (8, 4096, 40)]:
        assert capi.gemm_s4_best_workspace_bytes(M, N, K) == capi.gemm_s4_workspace_bytes(M, N, K), (M, N, K)
    for M, N, K in [(65, 4096, 16384), (2048, 4096, 4096), (1000, 4096, 12288), (4096, 512, 4096),
                    (2048, 4096, 4160)]:
        best = capi.gemm_s4_best_workspace_bytes(M, N, K)
        assert best > capi.gemm_s4_workspace_bytes(M, N, K) and best >= 2 * M * K, (M, N, K)


def test_plan_queries_are_host_only(capi):
    # the kernel, tile and K slices a call runs, at the workspace it is given
    def plan(M, N, K, ws):
        return capi.gemm_s4_plan(M, N, K, ws)
    shape = (203, 8195, 8192)
    need = capi.gemm_s4_workspace_bytes(*shape)
    kernel, rows, cols, splits = plan(*shape, need)
    assert (kernel, cols) == (capi.FP16_CONVERTED, 256) and rows in (64, 128, 256)
    # exactly what that plan holds: partials, then activations and shifts
    partial = (splits * 203 * 8195 * 4 if splits > 1 else 0) + 255 & ~255
    assert need == partial + 256 * 8192 * 2 + splits * (256 + 8448) * 4
    assert plan(*shape, 0)[0] != capi.FP16_CONVERTED
    assert plan(16, 4096, 4096, 0) == (capi.INT8_STREAM, 32, 32, 1)
    assert plan(64, 57344, 8192, 0)[0] == capi.FP16_STREAM
    assert plan(4096, 4096, 4096, 0) == (capi.FP16_TILES, 256, 256, 1)
    assert plan(100, 64, 96, 0)[0] == capi.INT8_TILES
    assert capi.gemm_s4_tensor_scale_plan(512, 24576, 4096)[0] == capi.TENSOR_TILES
    assert capi.gemm_s4_tensor_scale_plan(64, 96, 96)[0] == capi.INT8_TILES
    for bad in [(0, 64, 64), (4, 0, 64), (4, 64, 40)]:
        with pytest.raises(RuntimeError, match="invalid argument"):
            capi.gemm_s4_plan(*bad, 0)
        with pytest.raises(RuntimeError, match="invalid argument"):
            capi.gemm_s4_tensor_scale_plan(*bad)


def test_torch_module_exposes_reference_ops():
    from my_int4 import _C
    import my_int4
    from wush_int4_kernel_amd import _C as C2
    for op in REFERENCE_OPS:
        assert callable(getattr(_C, op)), op
        assert getattr(_C, op) is getattr(C2, op)
    assert my_int4.quant_int4 is C2.quant_int4
    assert _C.abi_version() == 1


def test_torch_ops_reject_cpu_tensors():
    import torch
    from my_int4 import _C
    x = torch.zeros(4, 64, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="CUDA"):
        _C.quant_int4(x)
    with pytest.raises(RuntimeError, match="CUDA"):
        _C.fused_transform_quant_int4(x, torch.zeros(2, 32, 32, dtype=torch.bfloat16))
    q = torch.zeros(4, 32, dtype=torch.uint8)
    s = torch.zeros(4, 2, dtype=torch.bfloat16)
    for op in ["w4a4_gemm_s4", "w4a4_gemv_multi", "w4a4_gemm", "w4a4_gemm_v1", "w4a4_gemm_v2"]:
        with pytest.raises(RuntimeError, match="CUDA"):
            getattr(_C, op)(q, s, q, s)
    with pytest.raises(RuntimeError, match="CUDA"):
        _C.w4a4_gemm_cutlass(q, q, 1.0)


def test_reference_python_modules_exposed():
    # reference my_int4/rtn_int4.py and my_int4/wush_transform.py: same names
    # and parameters; rtn_int4's quant/product refuse CPU tensors (no CPU path)
    import inspect
    import torch
    from my_int4 import rtn_int4, wush_transform
    assert list(inspect.signature(rtn_int4.quant_int4).parameters) == ["x", "group_size"]
    assert list(inspect.signature(rtn_int4.dequant_int4).parameters) == ["q_byte", "scale", "group_size"]
    assert list(inspect.signature(rtn_int4.w4a4_matmul_reference).parameters) == ["x_q", "x_s", "w_q", "w_s"]
    for name in ("compute_wush_transform", "transform_weights", "transform_activations_reference"):
        assert callable(getattr(wush_transform, name))
    assert list(inspect.signature(wush_transform.compute_wush_transform).parameters)[:4] == \
        ["X_cal", "W", "group_size", "use_hadamard"]
    with pytest.raises(RuntimeError, match="GPU"):
        rtn_int4.quant_int4(torch.zeros(2, 64, dtype=torch.bfloat16))
    # dequant decodes the packed format: byte 0xD3 = codes (+3, -3), scale 0.5
    q = torch.tensor([[0xD3] * 16], dtype=torch.uint8)
    s = torch.tensor([[0.5]], dtype=torch.bfloat16)
    d = rtn_int4.dequant_int4(q, s)
    assert d.shape == (1, 32) and d[0, 0].item() == 1.5 and d[0, 1].item() == -1.5


def test_tuning_defines_parsing(monkeypatch):
    # WUSH_DEFINES becomes -D flags on the hipcc lines; only WUSH_* names with
    # plain values pass, so the variable cannot smuggle other compiler flags in
    from wush_int4_kernel_amd import _build

    monkeypatch.setenv("WUSH_DEFINES", "WUSH_TQ_SMALLM_PAIRS=0  WUSH_GEMV_WAVES=8 WUSH_X")
    assert _build.tuning_defines() == ["-DWUSH_TQ_SMALLM_PAIRS=0", "-DWUSH_GEMV_WAVES=8", "-DWUSH_X"]
    monkeypatch.delenv("WUSH_DEFINES")
    assert _build.tuning_defines() == []
    for bad in ("-fsanitize=address", "WUSH_A=1;rm", "OTHER=1", "WUSH_A=$(x)", "wush_a=1"):
        monkeypatch.setenv("WUSH_DEFINES", bad)
        with pytest.raises(ValueError):
            _build.tuning_defines()


# (M, N, K) on both sides of every term of the GEMV shape rule: the staged
# kernel's 64 KiB LDS limit, the K-split kernel's M, N and K bounds
GEMV_RULE_SHAPES = [(M, N, K) for M in (1, 4, 6, 7, 8, 9) for N in (4096, 32768, 32769, 57344)
                    for K in (4096, 8192, 16384, 32768, 34816, 65536)] + [(0, 4096, 4096), (8, 57344, 8200)]


def _check_gemv_rule(lib):
    """wush_gemv_int4 rejects (before touching a device) exactly the shapes
    wush_gemv_int4_supported reports as unsupported; returns the supported set."""
    P = ctypes.c_void_p
    lib.wush_gemv_int4_supported.argtypes = [ctypes.c_int64] * 3
    lib.wush_gemv_int4.argtypes = [P] * 5 + [ctypes.c_int64] * 3 + [P]
    ok = set()
    for M, N, K in GEMV_RULE_SHAPES:
        sup = lib.wush_gemv_int4_supported(M, N, K)
        st = lib.wush_gemv_int4(P(16), P(16), P(16), P(16), P(16), M, N, K, None)
        assert sup in (0, 1)
        assert (st == INVALID) == (sup == 0), (M, N, K, sup, st)
        if sup:
            ok.add((M, N, K))
    return ok


def test_gemv_rule_is_the_librarys(capi, tmp_path):
    # The _C product ops route to wush_gemv_int4 only where the library says
    # it runs the shape (bindings.cpp asks wush_gemv_int4_supported), so a
    # build with other tuning macros cannot send a shape the GEMV rejects.
    # Default build: the K-split kernel takes M = 7, 8 at L70 and K = 16384.
    default = _check_gemv_rule(capi.load())
    assert (8, 57344, 8192) in default and (8, 57344, 16384) in default and (7, 32769, 32768) in default
    assert (8, 32768, 16384) not in default and (6, 57344, 16384) not in default
    assert (1, 4096, 65536) in default and (4, 4096, 16384) in default and (6, 4096, 16384) not in default
    # A build with the K-split kernel off (WUSH_GEMV_KS_MIN_M=9, the documented
    # off value) keeps only the LDS-staged shapes.
    from wush_int4_kernel_amd import _build
    lib_path = str(tmp_path / "libwush_int4_ks_off.so")
    _build.build_capi(lib_path=lib_path, build_dir=str(tmp_path / "obj"), defines="WUSH_GEMV_KS_MIN_M=9")
    off = _check_gemv_rule(ctypes.CDLL(lib_path))
    assert (8, 57344, 16384) not in off and (7, 57344, 32768) not in off and (7, 57344, 8192) in off
    assert off == {s for s in default if s[0] * (s[2] // 2) + s[0] * (s[2] // 32) * 8 <= 64 * 1024}
