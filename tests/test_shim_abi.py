"""The device library loads without a GPU and exports every symbol its header declares (no compute calls)."""
import os
import re
import subprocess
import sys

import pytest

from armnn_amd import shim

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "armnn_mi355x.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(mi355x_[a-z0-9_]+)\s*\(", text)))


def test_header_and_binding_agree():
    assert _declared_symbols() == sorted(shim.EXPORTS)


def test_library_exports_every_declared_symbol():
    if not os.path.exists(shim.LIB_PATH):
        pytest.skip("device library not built yet (run __graft_entry__.build())")
    lib = shim.load_library()
    for name in _declared_symbols():
        assert hasattr(lib, name), name
    assert lib.mi355x_abi_version() == 1


def test_device_count_without_gpu_is_not_an_error():
    if not os.path.exists(shim.LIB_PATH):
        pytest.skip("device library not built yet")
    assert shim.Device.count() >= 0


@pytest.mark.parametrize("what", ["missing", "not_loadable", "built"])
def test_the_library_loads_with_and_without_the_cpython_calls(what, tmp_path):
    """_calls.so belongs to the Python that built it; elsewhere the same calls go through ctypes."""
    if not os.path.exists(shim.LIB_PATH):
        pytest.skip("device library not built yet")
    calls = tmp_path / "_calls.so"
    if what == "not_loadable":
        calls.write_bytes(b"built for something else")
    program = ("from armnn_amd import shim\n"
               + ("" if what == "built" else f"shim.CALLS_PATH = {str(calls)!r}\n") +
               "shim.load_library()\n"
               "for cls, plan in ((shim.Conv2dPlan, 'plan'), (shim.FullyConnectedPlan, 'plan')):\n"
               "    p = object.__new__(cls)\n"
               "    p.lib, p.plan = shim.load_library(), None\n"
               "    try:\n"
               "        p.run(1, 0, 0)\n"
               "    except shim.ShimError as e:\n"
               "        print(e)\n"
               "print('through', 'ctypes' if shim._calls is None else '_calls')\n")
    r = subprocess.run([sys.executable, "-c", program], cwd=ROOT, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    lines = r.stdout.split("\n")
    assert lines[0] == lines[1] and lines[0].endswith("plan is null"), r.stdout
    if what != "built" or os.path.exists(shim.CALLS_PATH):
        assert lines[2] == ("through _calls" if what == "built" else "through ctypes")
