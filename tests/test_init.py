"""esp_attn_init's promise, without a GPU: after it no call of the library has anything but launches left to do, so that the first
launch of any variant may be recorded into a graph. The library runs over recording_hip.cpp in a process of its own."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

CHILD = """
import ctypes as C, sys
sys.path.insert(0, sys.argv[1])
hip = C.CDLL(sys.argv[2], mode=C.RTLD_GLOBAL)
from espetero_amd import abi
lib, err = abi.attn_lib(), C.create_string_buffer(256)
if sys.argv[3] == "init":
    abi.check(lib.esp_attn_init(0, err, 256), err)
first = hip.recorded_attributes()
assert (first > 0) == (sys.argv[3] == "init")
p, n = abi.GateParams(), 0
for dt in (abi.ESP_F16, abi.ESP_BF16):
    for H in (1, 16, 17, 40, 64):
        for O in (0x1000, None):
            p.H, p.head_dim, p.D, p.dtype, p.q_ld, p.x_ld = H, 64, 128, dt, 64 * H, 128
            before = hip.recorded_attributes()
            abi.check(lib.esp_head_gate(C.byref(p), O, 0x2000, 0x3000, 0x4000, 5, None, err, 256), err)
            n += 1
            assert hip.recorded_launches() == n
            # without init the first call that needs the set-up does all of it
            assert hip.recorded_attributes() == before or (sys.argv[3] != "init" and O is None and before == 0), (dt, H, O)
assert hip.recorded_over_limit() == 0
print("ok")
"""


@pytest.mark.parametrize("how", ["init", "first use"])
def test_gate_calls_only_launch(how, tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    if cxx is None or not os.path.exists(os.path.join(rocm, "include", "hip", "hip_runtime_api.h")):
        pytest.skip("no C++ compiler or no HIP headers")
    so = str(tmp_path / "recording_hip.so")
    subprocess.run([cxx, "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"),
                    os.path.join(HERE, "recording_hip.cpp"), "-o", so], check=True)
    r = subprocess.run([sys.executable, "-c", CHILD, os.path.dirname(HERE), so, how], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "ok" in r.stdout, r.stdout + r.stderr
