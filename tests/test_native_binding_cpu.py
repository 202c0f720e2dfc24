"""The native module beside the Python binding is an addition to it: without the
module, or with one built for another PyTorch, every launcher still works
through ctypes, and the C++ library builds without Python or PyTorch."""

from __future__ import annotations

import os
import subprocess
import sys
import threading

import pytest

from conftest import ROOT

# A process of its own: a module that is loaded once stays for the process.
PROGRAM = """
import sys, types, warnings
sys.path.insert(0, {package!r})
import cuvit_amd, torch
{setup}
x = torch.zeros(4, 4)
with warnings.catch_warnings(record=True) as caught:
    warnings.simplefilter("always")
    for call in (lambda: cuvit_amd.layer_norm(x, x[0], x[0], x, 4, 4),
                 lambda: cuvit_amd.softmax(x, x, 4, 4),
                 lambda: cuvit_amd.softmax(None, None, 4, 4),
                 lambda: cuvit_amd.softmax(None, None, -1, 4),
                 lambda: cuvit_amd.gemm(x, x, None, x, cuvit_amd.gemm_problem(4, 4, 4)),
                 lambda: cuvit_amd.attention(x, x, 1, 1, 1, 64)):
        try:
            call()
        except cuvit_amd.InvalidArgument:
            continue
        raise SystemExit("a call that the library refuses was not refused by it")
    cuvit_amd.softmax(None, None, 0, 4)  # an empty extent returns first
warned = [w for w in caught if "native binding" in str(w.message)]
print("warnings", len(warned))
"""


@pytest.mark.parametrize("setup,warnings", [
    ("sys.modules['cuvit_amd._native'] = None", 1),
    ("m = types.ModuleType('cuvit_amd._native'); m.built_for = ('1.0.0', 3, 0);"
     " sys.modules['cuvit_amd._native'] = cuvit_amd._native = m", 1),
    ("m = types.ModuleType('cuvit_amd._native'); sys.modules['cuvit_amd._native'] = cuvit_amd._native = m", 1),
    ("", 0),
], ids=["missing", "other_torch", "no_stamp", "built"])
def test_launchers_without_a_usable_module(setup, warnings):
    program = PROGRAM.format(package=os.path.join(ROOT, "cu-vit_amd"), setup=setup)
    result = subprocess.run([sys.executable, "-c", program], capture_output=True, text=True, timeout=110)
    assert result.returncode == 0, result.stderr
    assert f"warnings {warnings}" in result.stdout


def test_first_use_from_several_threads():
    import cuvit_amd
    import torch

    calls = cuvit_amd._NativeCalls()
    x = torch.zeros(4)
    answers, start = [], threading.Barrier(8)

    def use():
        start.wait()
        answers.append(calls.softmax(x, x, 1, 4, None, None))

    threads = [threading.Thread(target=use) for _ in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert answers == [-1] * 8  # a CPU tensor is left to the Python code


def test_the_library_builds_without_python():
    plan = subprocess.run(["make", "-n", "-B", "-C", os.path.join(ROOT, "cu-vit_amd")],
                          capture_output=True, text=True, check=True).stdout
    assert "libcuvit_amd.so" in plan
    assert "native.cpp" not in plan and "python" not in plan
