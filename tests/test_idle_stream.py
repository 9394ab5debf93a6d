"""The stream that plan uploads leave behind for the next plan (csrc/idle_stream.h): threads of one process may be on different
devices, and none may be handed another device's stream."""
import os
import subprocess

from tests.conftest import ROOT

PROGRAM = r"""
#include "idle_stream.h"
#include <cstdio>
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)
int main()
{
    int a = 0, b = 0;
    mi355x::IdleStream<int*> idle;
    CHECK(idle.Take(0) == nullptr);
    CHECK(idle.Put(0, &a) == nullptr);
    CHECK(idle.Take(1) == nullptr);              // a thread on device 1 makes a stream of its own
    CHECK(idle.Put(1, &b) == &a);                // ... and leaves it: one waits at most
    CHECK(idle.Take(0) == nullptr);
    CHECK(idle.Take(1) == &b);
    CHECK(idle.Take(1) == nullptr);
    CHECK(idle.Put(1, &b) == nullptr);
    CHECK(idle.TakeAny() == &b);
    CHECK(idle.TakeAny() == nullptr);
    return 0;
}
"""


def test_a_stream_goes_to_its_own_device_only(tmp_path):
    src, exe = tmp_path / "idle.cpp", tmp_path / "idle"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{os.path.join(ROOT, 'armnn_amd', 'csrc')}", str(src), "-o", str(exe), "-pthread"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
