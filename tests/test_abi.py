"""The C-ABI library loads without a GPU and exports every symbol include/kuiper_hip.h declares;
argument validation happens before any device call.  CPU only (no compute)."""
import ctypes as C
import os
import re

import pytest

from conftest import ROOT, load_golden
from kuiperllama_amd import _ffi, build


@pytest.fixture(scope="module")
def lib():
    build.build_lib()
    return _ffi.lib()


def _declared_functions():
    src = open(os.path.join(ROOT, "include", "kuiper_hip.h")).read()
    src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
    return sorted(set(re.findall(r"\b(kh_[a-z0-9_]+)\s*\(", src)))


def test_every_declared_symbol_is_exported(lib):
    names = _declared_functions()
    assert len(names) >= 28
    for n in names:
        assert hasattr(lib, n), f"{n} declared in kuiper_hip.h but not exported"
    assert sorted(_ffi.EXPORTS) == names


def test_version_and_error_strings(lib):
    assert lib.kh_version() == 110
    assert _ffi.error_string(0) == "success"
    assert "invalid" in _ffi.error_string(-1)
    assert "exception" in _ffi.error_string(_ffi.KH_ERR_INTERNAL)  # no C++ exception crosses the C ABI (kh_api_guard)
    assert lib.kh_kclass_name(3).decode() == "ffn13"


def test_invalid_arguments_are_rejected_without_touching_the_device(lib):
    assert lib.kh_add_f32(None, None, None, 4, None) == -1
    assert lib.kh_matmul_f32(None, None, None, 4, 4, 1.0, None) == -1
    assert lib.kh_matmul_q8(None, None, None, 64, None, 64, 4, None) == -1
    assert lib.kh_rmsnorm_f32(None, None, None, 0, 1e-5, None) == -1
    assert lib.kh_argmax_f32(None, 0, None, None) == -1
    assert lib.kh_model_get_config(None, None) == -1
    h = C.c_void_p()
    assert lib.kh_model_create_from_file(b"/nonexistent/model.bin",
                                         C.byref(_ffi.ModelOpts(0, 0, 0, 1e4, 1e-5, 0, 0, 0)),
                                         C.byref(h)) == -3  # KH_ERR_IO (reference: PathNotValid)


def test_model_creation_fails_loudly_without_gpu(lib):
    import torch
    if torch.cuda.is_available():
        pytest.skip("GPU present")
    from kuiperllama_amd.model import KuiperModel
    spec, img, _, _ = load_golden("ref_llama_gqa_tied")
    with pytest.raises(_ffi.KhError) as ei:
        KuiperModel.from_host_image(img, spec)
    assert ei.value.code == -5  # KH_ERR_NO_DEVICE: no silent CPU fallback


def test_ops_refuse_cpu_tensors():
    import torch
    from kuiperllama_amd import ops
    a = torch.zeros(4)
    with pytest.raises(ValueError):
        ops.add(a, a, a)


def test_debug_hooks_live_in_one_table_not_in_getenv(lib, monkeypatch):
    """Tuning / test hooks: set, read back, listed, cleared through kh_debug_*; the launch-plan entry
    points honour a hook set through the API; no translation unit of the library calls getenv."""
    assert lib.kh_debug_set(b"NOT_A_HOOK", b"1") == -1
    assert _ffi.debug_get("KH_TEST_HOOK") is None
    _ffi.debug_set("KH_TEST_HOOK", "abc")
    assert _ffi.debug_get("KH_TEST_HOOK") == "abc"
    n = lib.kh_debug_list(None, 0)
    buf = C.create_string_buffer(int(n))
    lib.kh_debug_list(buf, n)
    assert "KH_TEST_HOOK" in buf.value.decode().split("\n")
    _ffi.debug_set("KH_TEST_HOOK", None)
    assert _ffi.debug_get("KH_TEST_HOOK") is None
    # a shape hook set through the API changes the plan and SURVIVES the binding's environment mirror
    # (sync_env only manages the keys it took from os.environ); an environment variable of the same name
    # overrides it while it exists; clearing goes through the API again
    base = _ffi.plan_decode_shapes(2048, 8192, 512, 128256, False)["ffn13"]
    _ffi.debug_set("KH_SHAPE_FFN", "1,4,256,256")
    out = (C.c_int32 * 20)()
    assert lib.kh_plan_decode_shapes(2048, 8192, 512, 128256, 0, out) == 0
    assert list(out[8:12]) == [1, 4, 256, 256]
    assert _ffi.plan_decode_shapes(2048, 8192, 512, 128256, False)["ffn13"]["grid"] == 256  # sync_env left it alone
    monkeypatch.setenv("KH_SHAPE_FFN", "1,4,512,256")
    assert _ffi.plan_decode_shapes(2048, 8192, 512, 128256, False)["ffn13"]["grid"] == 512
    monkeypatch.delenv("KH_SHAPE_FFN")
    assert _ffi.plan_decode_shapes(2048, 8192, 512, 128256, False)["ffn13"] == base  # the mirrored key is cleared
    _ffi.debug_set("KH_SHAPE_FFN", None)
    # the LDS-DMA ring plan: int8 geometries whose input vector the 256-thread staging holds take it, KH_RING=0 turns it off
    assert _ffi.plan_decode_ring(4096, 11008, 32000, True) == {"ffn13": {"slots": 2, "grid": 512}, "cls": {"slots": 2, "grid": 512}}
    assert _ffi.plan_decode_ring(512, 1408, 501, True) == {"ffn13": {"slots": 2, "grid": 352}, "cls": {"slots": 2, "grid": 63}}
    assert _ffi.plan_decode_ring(2048, 8192, 128256, False)["ffn13"]["slots"] == 0   # fp32
    assert _ffi.plan_decode_ring(448, 1216, 3000, True)["cls"] == {"slots": 2, "grid": 375}  # partial pieces are fine
    assert _ffi.plan_decode_ring(8192, 28672, 128256, True)["ffn13"]["slots"] == 0  # 32 floats per staging thread
    monkeypatch.setenv("KH_RING", "0")
    assert _ffi.plan_decode_ring(4096, 11008, 32000, True)["ffn13"]["slots"] == 0
    monkeypatch.delenv("KH_RING")
    # a KH_SHAPE_FFN / KH_SHAPE_CLS hook names a register-tile launch: the ring must not take that launch over
    # (the B-token prefill follows the hook, decode silently ignored it)
    monkeypatch.setenv("KH_SHAPE_FFN", "1,4,512,256")
    r = _ffi.plan_decode_ring(4096, 11008, 32000, True)
    assert r["ffn13"]["slots"] == 0 and r["cls"]["slots"] == 2
    monkeypatch.delenv("KH_SHAPE_FFN")
    monkeypatch.setenv("KH_SHAPE_CLS", "1,4,512,256")
    r = _ffi.plan_decode_ring(4096, 11008, 32000, True)
    assert r["ffn13"]["slots"] == 2 and r["cls"]["slots"] == 0
    monkeypatch.delenv("KH_SHAPE_CLS")
    assert _ffi.plan_decode_ring(4096, 11008, 32000, True)["cls"]["slots"] == 2
    _ffi.sync_env()
    csrc = os.path.join(ROOT, "kuiperllama_amd", "csrc")
    for f in os.listdir(csrc):
        assert "getenv" not in open(os.path.join(csrc, f)).read(), f


def test_every_hook_of_the_sources_is_mirrored_from_the_environment(lib, monkeypatch):
    """A hook whose prefix the mirror does not know is set in os.environ and never reaches the library."""
    csrc = os.path.join(ROOT, "kuiperllama_amd", "csrc")
    hooks = set()
    for f in os.listdir(csrc):
        if f.endswith((".h", ".hip", ".cpp")):
            with open(os.path.join(csrc, f)) as src:
                hooks.update(re.findall(r'"(KH_[A-Z0-9]+_[A-Z0-9_]*[A-Z0-9]|KH_[A-Z0-9]+)"', src.read()))
    assert {"KH_PAIR_SHAPE", "KH_PAIR_ATTN", "KH_PG_PAIR", "KH_RING", "KH_HY_ROWS"} <= hooks
    for h in sorted(hooks):
        monkeypatch.setenv(h, "7")
        _ffi.sync_env()
        got = _ffi.debug_get(h)
        monkeypatch.delenv(h)
        _ffi.sync_env()
        assert got == "7", h
        assert _ffi.debug_get(h) is None, h
