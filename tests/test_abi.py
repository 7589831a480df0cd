"""The C-ABI library and the Python dispatch layer (CPU only: no kernel is launched here)."""
from __future__ import annotations

import ctypes
import re
import shutil
import subprocess
import warnings
from pathlib import Path

import pytest
import torch

from qwen_triton import _native
from qwen_triton import kernels as K
from qwen_triton.kernels import _common

ROOT = Path(__file__).resolve().parents[1]


def _declared():
    text = "\n".join(p.read_text() for p in (ROOT / "include").glob("*.h"))
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return re.findall(r"\b(qh_\w+)\s*\(", text)


def test_library_loads_and_exports_every_declared_symbol():
    lib = ctypes.CDLL(str(_native.LIB_PATH))
    names = _declared()
    assert len(names) >= 30
    for name in names:
        assert hasattr(lib, name), name
    assert _native.available()
    assert "gfx950" in _native.version()


def test_header_signatures_bind():
    sigs = _native.parse_header()
    assert sigs["qh_gemm"] == ("i", "iilllplplplpiip")
    assert sigs["qh_last_error"] == ("s", "")
    assert set(sigs) == set(_declared())


def test_workspace_queries_are_host_only():
    assert _native.call("qh_rmsnorm_bwd_workspace", 16384, 1024, _native.BF16) > 0
    # id sort space: keys and token positions, in and out (no per-row table)
    assert _native.call("qh_embedding_bwd_workspace", 16384, 151936) >= 4 * 16384 * 4
    # Delta and log2-scale LSE per query, rows padded to a multiple of 64 plus one 64-query tile
    assert _native.call("qh_flash_bwd_workspace", 8, 16, 4096) == 2 * 8 * 16 * (4096 + 64) * 4
    assert _native.call("qh_flash_bwd_workspace", 1, 2, 65) == 2 * 1 * 2 * (128 + 64) * 4
    # 64 sequences x 8 kv-heads at head dim 128: one workgroup per pair, partials combined on chip
    assert _native.call("qh_flash_decode_workspace", 64, 16, 8, 2049, 128) == 0
    assert _native.call("qh_flash_decode_workspace", 8, 32, 8, 2900, 128) > 0


def test_argument_errors_are_reported_without_launching():
    with pytest.raises(_native.NativeError, match="rotary dim"):
        _native.call("qh_rope", 0, 1, 1, 1, 1, 0, 0, 1, 1, 1, 1, 0, 1, 1, 1, 4, 3, 0, _native.BF16, _native.BF16, 0)
    with pytest.raises(_native.NativeError, match="k=5 > C=4"):
        _native.call("qh_topk", 0, 0, 0, 1, 4, 5, _native.F32, 0)
    with pytest.raises(_native.NativeError, match="N and ldc multiples of 8"):  # 16-byte output rows
        _native.call("qh_moe_down", 0, 8, 1, 8, 0, 8, 100, 0, 0, 1, 0, 100, 0, _native.BF16, 0)
    with pytest.raises(_native.NativeError, match="head dim"):
        _native.call("qh_flash_fwd", 0, 0, 0, 8, 0, 0, 0, 8, 0, 0, 0, 8, 0, 0, 0, 8, 0, 1, 1, 1, 1, 1, 200, 1.0, 1,
                     0, _native.BF16, 0)


def test_cpu_tensors_use_torch_path_like_the_reference():
    x, w = torch.randn(3, 8), torch.randn(8)
    torch.testing.assert_close(K.rmsnorm(x, w), K.rmsnorm(x, w, use_triton=False))


def test_forced_native_on_cpu_falls_back_with_one_warning(monkeypatch):
    monkeypatch.delenv("QWEN_TRITON_STRICT", raising=False)
    from qwen_triton.kernels import swiglu

    swiglu._GUARD.reset()
    try:
        with warnings.catch_warnings(record=True) as rec:
            warnings.simplefilter("always")
            a, b = torch.randn(4), torch.randn(4)
            out = K.silu_mul(a, b, use_triton=True)
            out2 = K.silu_mul(a, b, use_triton=True)
        torch.testing.assert_close(out, torch.nn.functional.silu(a) * b)
        torch.testing.assert_close(out2, out)
        msgs = [str(r.message) for r in rec if "[Qwen-Triton fallback]" in str(r.message)]
        assert len(msgs) == 1
        # CPU tensors are inputs the kernels do not take, not a kernel failure: the operator stays on
        # the kernels for later GPU calls (the reference's flag would stick here)
        assert swiglu._GUARD.runtime_ok is True
    finally:
        swiglu._GUARD.reset()


def test_strict_mode_raises(monkeypatch):
    monkeypatch.setenv("QWEN_TRITON_STRICT", "1")
    from qwen_triton.kernels import softmax

    softmax._GUARD.reset()
    try:
        with pytest.raises(RuntimeError, match="strict"):
            K.triton_softmax(torch.randn(2, 3), use_triton=True)
    finally:
        softmax._GUARD.reset()


def test_missing_library_is_loud_for_gpu_tensors(monkeypatch):
    guard = _common.OpGuard("Probe")

    class FakeCuda:
        is_cuda = True

    monkeypatch.setattr(_native, "available", lambda: False)
    with pytest.raises(RuntimeError, match="could not be loaded"):
        guard.use_native(None, FakeCuda())


@pytest.mark.parametrize("lda,ldb", [(1 << 27, 64), (64, 1 << 27)])
def test_grouped_products_refuse_rows_past_their_lane_offsets(lda, ldb):
    """The grouped launch reaches the rows of a load with 32-bit lane offsets: strides that would wrap
    are an argument error before any launch."""
    arr = lambda t, *v: (t * len(v))(*v)  # noqa: E731
    b, c = arr(ctypes.c_void_p, 4096, 4096), arr(ctypes.c_void_p, 8192, 8192)
    ldb_, n, ldc = arr(ctypes.c_int64, 64, ldb), arr(ctypes.c_int64, 3072, 3072), arr(ctypes.c_int64, 3072, 3072)
    with pytest.raises(_native.NativeUnsupported, match="elements apart"):
        _native.call("qh_gemm_group", 517, 64, 4096, lda, 2, ctypes.addressof(b), ctypes.addressof(ldb_),
                     ctypes.addressof(n), ctypes.addressof(c), ctypes.addressof(ldc), None, 0, _native.BF16, 0)


@pytest.mark.parametrize("ldx,ldw", [(1 << 25, 64), (64, 1 << 25)])
def test_fused_loss_refuses_rows_past_its_lane_offsets(ldx, ldw):
    """The logits kernel's loading waves reach 39 rows past a load's base with 32-bit lane offsets."""
    with pytest.raises(_native.NativeUnsupported, match="elements apart"):
        _native.call("qh_lmce_rows_fwd", 4096, ldx, 4096, ldw, 4096, 512, 1024, 64, -100, 4096, 1024, 4096, 4096,
                     4096, 1 << 30, _native.BF16, 0)


@pytest.mark.parametrize("wide", [0, 1])
def test_loss_products_refuse_rows_past_their_lane_offsets(wide):
    ld = [64, 64]
    ld[wide] = 1 << 27
    with pytest.raises(_native.NativeUnsupported, match="elements apart"):
        _native.call("qh_lmce_fwd", 4096, ld[0], 4096, ld[1], 4096, 512, 1024, 64, -100, 4096, 4096, 4096, 4096, 4096,
                     1 << 30, _native.BF16, 0)
    with pytest.raises(_native.NativeUnsupported, match="elements apart"):
        _native.call("qh_gemm_acc", 0, 0, 256, 256, 64, 4096, ld[0], 4096, ld[1], 4096, 256, _native.BF16, 0)


def test_grouped_products_leave_split_k_alone():
    n = (ctypes.c_int64 * 2)(3072, 3072)
    ok = lambda K: _native.call("qh_gemm_group_ok", 517, K, 2, ctypes.addressof(n), 1)  # noqa: E731
    assert ok(1024) and ok(8184) and not ok(8192)
    assert not _native.call("qh_gemm_workspace", 517, 3072, 8184, _native.BF16)
    assert _native.call("qh_gemm_workspace", 517, 3072, 8192, _native.BF16)


_LDS_LIMIT_PROGRAM = r"""
#include "qh_lds_limit.h"
#include <cstdio>
static int device = 0, calls = 0, failures = 0;
extern "C" hipError_t hipGetDevice(int* d) { *d = device; return hipSuccess; }
extern "C" hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) {
  ++calls;
  return failures-- > 0 ? hipErrorUnknown : hipSuccess;
}
extern "C" const char* hipGetErrorString(hipError_t) { return "injected"; }
namespace qh { void set_error(const char*, ...) {} }
int main() {
  static qh::LdsLimit limit;
  failures = 1;
  const int first = limit.raise("k", 1 << 17, "t");  // the attribute call fails: reported, not remembered
  for (int i = 0; i < 3; ++i)
    if (limit.raise("k", 1 << 17, "t") != QH_OK) return 1;
  const int on0 = calls;
  device = 1;
  for (int i = 0; i < 3; ++i)
    if (limit.raise("k", 1 << 17, "t") != QH_OK) return 1;
  device = 64;
  std::printf("%d %d %d %d", first != QH_OK, on0, calls, limit.raise("k", 1 << 17, "t") != QH_OK);
  return 0;
}
"""


def test_lds_limit_is_raised_on_every_device(tmp_path):
    """A kernel's dynamic LDS limit belongs to a device: every place that raises it looks at the current
    one, and the helper sets it once on each and again after a failure."""
    csrc = ROOT / "qwen-triton_amd" / "csrc"
    for f in [*csrc.glob("*.h"), *csrc.glob("*.hip")]:
        assert ("hipFuncSetAttribute" in f.read_text()) <= ("hipGetDevice" in f.read_text()), f.name
    if shutil.which("hipcc") is None and not Path("/opt/rocm/bin/hipcc").exists():
        pytest.skip("no hipcc")
    (tmp_path / "t.cpp").write_text(_LDS_LIMIT_PROGRAM)
    exe = tmp_path / "t"
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    subprocess.run([hipcc, "-x", "hip", "--offload-host-only", "-std=c++17", "-fPIE", f"-I{csrc}",
                    f"-I{ROOT / 'include'}", "-c", str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t.o")], check=True)
    subprocess.run(["g++", str(tmp_path / "t.o"), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout == "1 2 3 1"
