"""The order of calls on one stager, whichever stream each names, on the CPU:
the library enqueues into a recording stand-in for the HIP runtime
(tests/order/hip_recorder.cpp), which says what every kernel and copy follows."""
import json
import os
import shutil
import subprocess
import sys
from pathlib import Path

import pytest

from paceserve_amd import _native

HERE = Path(__file__).resolve().parent / "order"
ROCM = Path(os.environ.get("ROCM_PATH", "/opt/rocm"))


@pytest.fixture(scope="module")
def recorder(tmp_path_factory):
    if shutil.which("g++") is None or not (ROCM / "include" / "hip").exists():
        pytest.skip("g++ or the HIP headers not available")
    out = tmp_path_factory.mktemp("order") / "libhip_recorder.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM / 'include'}",
                    str(HERE / "hip_recorder.cpp"), "-o", str(out)], check=True, timeout=300)
    return out


def run(recorder, *calls):
    r = subprocess.run([sys.executable, str(HERE / "calls.py"), str(recorder), str(_native.LIB_PATH), *calls],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
    return json.loads(r.stdout)


def pages(call):
    """The operations of a call that read or write pages."""
    ops = [o for o in call if "page_copy" in o["name"] or "host_leg" in o["name"]]
    assert ops
    return ops


def in_order(earlier, later):
    return all(e["op"] in o["after"] for o in pages(later) for e in pages(earlier))


@pytest.mark.parametrize("host", ["pinned", "pageable"])
@pytest.mark.parametrize("second", ["trip:6", "trip:2"])
@pytest.mark.parametrize("first", ["trip:6", "trip:2"])
def test_a_round_trip_follows_the_round_trip_before_it(recorder, first, second, host):
    """Of one chunk (on the caller's stream) or three (on the stager's): every
    pack and unpack follows those of the call before, and what writes the host
    buffer follows what read it."""
    a, b = run(recorder, f"{first}:a:{host}", f"{second}:b:{host}")["calls"]
    assert in_order(a, b)
    assert all(e["op"] in o["after"] for o in b for e in a)
    for call in (a, b):
        assert all(o["joined"] for o in call)    # the caller's stream follows everything
