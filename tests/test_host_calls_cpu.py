"""The native host calls (csrc/host_calls.cpp) bound to a stub of the C ABI, on CPU tensors:
what each does with a status of the launch, and how often it launches."""

import ctypes
import importlib.machinery
import importlib.util
import os
import shutil
import subprocess
from pathlib import Path

import pytest
import torch

from mimir_amd import _capi

INCLUDE = Path(__file__).resolve().parents[1] / "include" / "mimir_prefixlm.h"
STUB = f'#include "{INCLUDE}"\n' + r"""
extern "C" {
int stub_status = 0, stub_calls = 0;
static int launched() { ++stub_calls; return stub_status; }
const char* mimir_prefixlm_last_error(void) { return "stub launch failed"; }
int mimir_prefixlm_fwd(const MimirPrefixLMFwdParams*, void*) { return launched(); }
int mimir_prefixlm_bwd(const MimirPrefixLMBwdParams*, void*) { return launched(); }
int mimir_prefixlm_rope(const MimirRopeParams* p, void*) {  // in place: every launch shows
  for (int i = 0; i < p->total_tokens; ++i) ((float*)p->y)[i * p->y_stride_token] = ((const float*)p->x)[i * p->x_stride_token] + 1;
  return launched();
}
int mimir_prefixlm_cache_attn(const MimirCacheAttnParams*, void*) { return launched(); }
size_t mimir_prefixlm_fwd_workspace_size(const MimirPrefixLMFwdParams*) { return 64; }
size_t mimir_prefixlm_fwd_workspace_bytes(int32_t, int32_t, int32_t) { return 64; }
size_t mimir_prefixlm_bwd_workspace_size(const MimirPrefixLMBwdParams*) { return 64; }
size_t mimir_prefixlm_bwd_dscore_bytes(const MimirPrefixLMBwdParams*) { return 0; }
size_t mimir_prefixlm_cache_attn_workspace_bytes(const MimirCacheAttnParams*) { return 64; }
}
"""


@pytest.fixture(scope="module")
def bound(tmp_path_factory):
    """(the native calls, the stub): a copy of the module of their own, bound for CPU tensors."""
    if not _capi.HOST_PATH.exists():
        from mimir_amd.build import build

        build(verbose=False)
    tmp = tmp_path_factory.mktemp("host")
    subprocess.run([os.environ.get("CXX", "g++"), "-shared", "-fPIC", "-x", "c++", "-", "-o", str(tmp / "stub.so")],
                   input=STUB, text=True, check=True)
    copy = shutil.copy(_capi.HOST_PATH, tmp / "_host_calls.so")
    loader = importlib.machinery.ExtensionFileLoader("_host_calls", str(copy))
    host = importlib.util.module_from_spec(importlib.util.spec_from_loader("_host_calls", loader))
    loader.exec_module(host)
    host.bind(str(tmp / "stub.so"), "cpu")
    return host, ctypes.CDLL(str(tmp / "stub.so"))


def _calls(host):
    T, d = 5, 64
    q, k, v = torch.zeros(T, 4, d), torch.zeros(T, 2, d), torch.zeros(T, 2, d)
    meta = [torch.tensor(x, dtype=torch.int32) for x in ([2], [3], [0, T])]
    no_flag = torch.zeros(0, dtype=torch.int32)
    cos = torch.zeros(T, d)
    new, cache = torch.zeros(2, 1, 2, d, dtype=torch.bfloat16), torch.zeros(2, 9, 2, d, dtype=torch.bfloat16)
    return {
        "fwd": lambda: host.fwd(q, k, v, False, *meta, T, 1, T, 0.125, 0, True, False, None, None, torch.empty, 0),
        "bwd": lambda: host.bwd(q, q, k, v, q, torch.zeros(4, T), q.new_empty(0), no_flag, False, *meta, T, 1, T, 0.125, 0, True,
                                0, 0, None, None, torch.empty, 0),
        "rope": lambda: host.rope(q, cos, cos, True, q, 0),
        "cache_attn": lambda: host.cache_attn(torch.zeros(2, 1, 4, d, dtype=torch.bfloat16), new, new, cache, cache.clone(),
                                              torch.tensor([3, 4]), True, None, 0.125, torch.empty, 0),
    }


@pytest.mark.parametrize("name", ["fwd", "bwd", "rope", "cache_attn"])
def test_status_of_the_launch(bound, name):
    host, stub = bound
    status, calls = (ctypes.c_int.in_dll(stub, x) for x in ("stub_status", "stub_calls"))
    call = _calls(host)[name]
    calls.value, status.value = 0, _capi.OK
    assert call() is not None and calls.value == 1
    for refused in (_capi.ERR_INVALID_ARGUMENT, _capi.ERR_UNSUPPORTED_DTYPE, _capi.ERR_UNSUPPORTED_SHAPE):
        status.value = refused  # before any launch: the general path raises it
        assert call() is None
    calls.value, status.value = 0, _capi.ERR_HIP
    with pytest.raises(RuntimeError, match="stub launch failed"):
        call()
    assert calls.value == 1


def test_a_failed_in_place_rope_is_not_run_again(bound, monkeypatch):
    """Kernels of a failed launch may have run: nothing else launches the call again."""
    import mimir_amd
    from mimir_amd import prefixlm as P

    host, stub = bound
    monkeypatch.setattr(_capi, "host", lambda: host)
    monkeypatch.setattr(P, "_check_device_tensor", lambda name, t: None)
    monkeypatch.setattr(P, "_stream", lambda device: 0)
    monkeypatch.setattr(_capi, "load", lambda: pytest.fail("the general path ran"))
    ctypes.c_int.in_dll(stub, "stub_status").value = _capi.ERR_HIP
    x, cos = torch.zeros(5, 2, 64), torch.zeros(5, 64)
    with pytest.raises(RuntimeError, match="stub launch failed"):
        mimir_amd.rope(x, cos, cos, inverse=True, out=x)
    assert x[:, 0, 0].tolist() == [1.0] * 5


def test_tensors_of_another_device_take_the_general_path(bound):
    host, stub = bound
    ctypes.c_int.in_dll(stub, "stub_status").value = _capi.OK
    x, cos = torch.zeros(5, 2, 64, device="meta"), torch.zeros(5, 64, device="meta")
    assert host.rope(x, cos, cos, False, None, 0) is None


@pytest.mark.parametrize("form", ["missing", "another torch", "not a module"])
def test_without_the_native_calls_the_general_path_runs(monkeypatch, tmp_path, form):
    monkeypatch.setattr(_capi, "_host", None)
    if form == "missing":
        monkeypatch.setattr(_capi, "HOST_PATH", tmp_path / "_host_calls.so")
    elif form == "another torch":
        monkeypatch.setattr(torch, "__version__", "1.0")
    else:
        (tmp_path / "_host_calls.so").write_bytes(b"no shared object")
        monkeypatch.setattr(_capi, "HOST_PATH", tmp_path / "_host_calls.so")
    with pytest.warns(RuntimeWarning, match="general path"):
        host = _capi.host()
    assert host.fwd(1) is host.bwd(1) is host.rope(1) is host.cache_attn(1) is None
    assert _capi.host() is host  # and without another warning


def test_the_built_module_fits(monkeypatch):
    if not _capi.HOST_PATH.exists():
        pytest.skip("the native host calls are not built")
    monkeypatch.setattr(_capi, "_host", None)
    assert _capi.host() is not _capi._GeneralPath


def test_build_without_a_compiler_keeps_the_library(monkeypatch, tmp_path, capsys):
    from mimir_amd import build

    stale = tmp_path / "_host_calls.so"
    stale.write_bytes(b"of other sources")
    monkeypatch.setattr(build, "HOST_PATH", stale)
    monkeypatch.setenv("CXX", str(tmp_path / "no_such_compiler"))
    build._build_host()
    assert not stale.exists() and "general path" in capsys.readouterr().err
