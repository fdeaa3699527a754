"""The dispatch extension is connected to the Python implementations whichever module of the package is imported first (an
internal-layout call of a known signature packs its weight through them)."""
import subprocess
import sys
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
