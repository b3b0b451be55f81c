"""The large-LDS attribute of a kernel (csrc/gptq4_lds.h), on the CPU with the two HIP calls it makes replaced: set once per kernel
AND device, tried again after an error."""
import os
import re
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "gptq-triton_amd" / "csrc"

PROGRAM = r'''
#include "gptq4_lds.h"
#include <cstdio>

static int g_device = 0, g_calls = 0, g_device_error = 0, g_set_error = 0;
extern "C" hipError_t hipGetDevice(int *d) { *d = g_device; return (hipError_t)g_device_error; }
extern "C" hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int bytes) {
    g_calls += bytes == 100000;
    return (hipError_t)g_set_error;
}

#define EXPECT(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

int main() {
    LdsGrant a, b;
    auto ask = [&](LdsGrant &g, int device) { g_device = device; return allow_lds(g, &g, 100000); };
    EXPECT(ask(a, 0) == 0 && g_calls == 1);
    EXPECT(ask(a, 0) == 0 && g_calls == 1);
    EXPECT(ask(a, 1) == 0 && g_calls == 2);   // another device: the kernel is loaded there anew
    EXPECT(ask(a, 63) == 0 && g_calls == 3);
    EXPECT(ask(a, 1) == 0 && ask(a, 0) == 0 && g_calls == 3);
    g_set_error = 1;
    EXPECT(ask(b, 1) == 1 && g_calls == 4);
    g_set_error = 0;
    EXPECT(ask(b, 1) == 0 && g_calls == 5 && ask(b, 1) == 0 && g_calls == 5);
    EXPECT(ask(a, 64) != 0 && ask(a, -1) != 0 && g_calls == 5);
    g_device_error = 3;
    EXPECT(ask(a, 0) == 3);
    return 0;
}
'''


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_once_per_kernel_and_device(tmp_path):
    src, exe = tmp_path / "grant.cpp", tmp_path / "grant"
    src.write_text(PROGRAM)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{CSRC}", f"-isystem{rocm}/include", str(src), "-o", str(exe)], check=True)
    done = subprocess.run([str(exe)], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout


def test_every_launch_asks_through_it():
    for path in sorted(CSRC.glob("*.hip")):
        assert not re.search(r"hipFuncSetAttribute|static bool", path.read_text()), path.name
