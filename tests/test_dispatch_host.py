"""The dispatch extension is connected to the Python implementations whichever module of the package is imported first (an
internal-layout call of a known signature packs its weight through them)."""
import subprocess
import sys
import threading
import time
import weakref

import pytest
import torch

from conftest import ROOT


@pytest.mark.parametrize("first", ["runtime.hip_blocked_backend", "runtime.snn_custom_ops", "runtime.hip_pool_backend", "fx_temporal_rewrite"])
def test_extension_is_connected_by_whoever_loads_it(snnf_lib, first):
    code = (f"import importlib, triton_snn_fusion_amd\nimportlib.import_module('triton_snn_fusion_amd.{first}')\n"
            "from triton_snn_fusion_amd import _dispatch\nassert _dispatch.module().connected()\n")
    done = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=120)
    assert done.returncode == 0, done.stderr[-2000:]


def test_internal_layout_tensors_take_attributes_and_weak_references():
    from triton_snn_fusion_amd.runtime import hip_blocked_backend as B
    x = B.Blocked(torch.empty(0), B.BITS, 1, 1, 8, 2, 2, torch.bfloat16)
    x.note = "a host program's own mark"
    assert weakref.ref(x)() is x and x.note


def test_two_threads_that_learn_at_once_file_their_own_statistics(monkeypatch):
    """The index that a first call hands to the native dispatch names the events of that call, whatever another thread files meanwhile."""
    from triton_snn_fusion_amd.runtime import snn_custom_ops as ops

    class Slow(list):
        def append(self, item):
            super().append(item)
            time.sleep(0.05)                                # room for the other thread

    filed = Slow()
    monkeypatch.setattr(ops, "_SIGNATURE_EVENTS", filed)
    start = threading.Barrier(2)

    def implementation(key):
        start.wait()
        ops._bump("triton", key)
        return ()

    answers = {}
    for name in ("a", "b"):
        monkeypatch.setitem(ops.OPERATORS, name, ("", implementation, None, None))
    threads = [threading.Thread(target=lambda n=n: answers.update({n: ops._slow_dispatch(f"snn_custom::{n}", [f"counter_{n}"], True)[1]})) for n in ("a", "b")]
    try:
        for t in threads:
            t.start()
        for t in threads:
            t.join(10)
    finally:
        ops.reset_fused_op_call_stats()
    assert len(filed) == 2
    assert all(("count", f"counter_{n}") in filed[answers[n]] for n in ("a", "b")), (answers, list(filed))


@pytest.mark.parametrize("state", ["not built", "not loadable"])
@pytest.mark.parametrize("first", ["runtime.hip_blocked_backend", "runtime.snn_custom_ops"])
def test_without_the_extension(snnf_lib, tmp_path, state, first):
    """libsnnf.so alone is enough: the operators register with their Python implementations for the CPU and the GPU, and an extension
    that does not load (built against another PyTorch, say) is one warning."""
    broken = tmp_path / "_snnf_dispatch.so"
    if state == "not loadable":
        broken.write_bytes(b"no library")
    code = f"""
import importlib, pathlib, warnings
import torch, triton_snn_fusion_amd
from triton_snn_fusion_amd import _dispatch, _lib
_dispatch.DISPATCH_PATH = pathlib.Path({str(broken)!r})
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    importlib.import_module('triton_snn_fusion_amd.{first}')
    assert _dispatch.module().blocked_conv(1, 2) is None and _dispatch.loaded() is None
    ops = importlib.import_module('triton_snn_fusion_amd.runtime.snn_custom_ops')
assert [w.category for w in seen if "_snnf_dispatch" in str(w.message)] == [RuntimeWarning] * {int(state == "not loadable")}, [str(w.message) for w in seen]
assert _lib.library_available()
ops._require_library()
for name in ops.OPERATORS:
    for key in ("CPU", "CUDA", "Meta"):
        assert torch._C._dispatch_has_kernel_for_dispatch_key("snn_custom::" + name, key), (name, key)
ops.configure_fused_op("hip")
x = torch.randn(4, 2, 8, 3, 3)
out = torch.ops.snn_custom.fused_temporal_lif_state(x, torch.zeros(()), 1.0, 0.0, 2.0, False)
assert torch.equal(out[0], ops.fused_temporal_lif_state_torch(x, torch.zeros(()), 1.0, 0.0, 2.0, False)[0])
assert ops.get_fused_op_call_stats()["total"] == 1
ops.reset_fused_op_call_stats()
"""
    done = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=120)
    assert done.returncode == 0, done.stderr[-2000:]
