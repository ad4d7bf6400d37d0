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


def pages_of(call):
    """The operations of a call that read or write pages."""
    return [o for o in call if "page_copy" in o["name"] or "host_leg" in o["name"]]


def pages(call):
    assert pages_of(call)
    return pages_of(call)


def in_order(earlier, later):
    return all(e["op"] in o["after"] for o in pages(later) for e in pages(earlier))


KINDS = ["pack", "unpack", "trip"]
OPPOSITE = {("pack", "unpack"), ("unpack", "pack")}    # leave each other alone


@pytest.mark.parametrize("host", ["pinned", "pageable"])
@pytest.mark.parametrize("chunks", [(1, 1), (1, 3), (3, 1), (3, 3)])
@pytest.mark.parametrize("second", KINDS)
@pytest.mark.parametrize("first", KINDS)
def test_a_call_follows_the_call_before_it(recorder, first, second, chunks, host):
    """Two calls on two streams, of one chunk (on the caller's stream) or three
    (on the stager's too): what the second does with pages follows what the
    first does with them, and what writes a host buffer follows what used it,
    but for a pack to host beside an unpack from host."""
    k1, k2 = (6 // c for c in chunks)
    a, b = run(recorder, f"{first}:{k1}:a:{host}", f"{second}:{k2}:b:pinned")["calls"]
    if (first, second) in OPPOSITE:
        assert not any(e["op"] in o["after"] for o in b for e in a)
    else:
        assert in_order(a, b)
        if second != "unpack":    # an unpack's copies read the host buffer
            assert all(e["op"] in o["after"] for o in b for e in a)
    for call in (a, b):
        assert all(o["joined"] for o in call)    # the caller's stream follows everything


@pytest.mark.parametrize("call", ["pack:6", "unpack:6", "trip:6"])
def test_a_captured_call_leaves_the_order_of_calls_alone(recorder, call):
    """A pinned one-chunk call under capture waits for no event of earlier
    calls, which belong to no graph, and the calls after it follow those."""
    first, captured, last = run(recorder, "trip:6:a", "capture:g", f"{call}:g", "end:g", "trip:6:b")["calls"]
    assert not any(e["op"] in o["after"] for o in captured for e in first)
    assert in_order(first, last) and not any(e["op"] in o["after"] for o in last for e in captured)


@pytest.mark.parametrize("host", ["pinned", "pageable"])
@pytest.mark.parametrize("call", ["pack:6", "unpack:6", "trip:6", "pack:2", "unpack:2", "trip:2"])
def test_destroy_waits_for_everything_before_it_frees(recorder, call, host):
    """What every call enqueued has finished when a stager gives its memory
    back, and with it the host tensors that Stager kept alive."""
    assert run(recorder, f"{call}:a:{host}")["unwaited"] == 0
    assert run(recorder, f"{call}:a:{host}", "trip:6:b", f"{call}:c:{host}")["unwaited"] == 0


@pytest.mark.parametrize("host", ["pinned", "pageable"])
@pytest.mark.parametrize("k", [6, 2])
@pytest.mark.parametrize("kind", ["pack", "unpack", "inline-pack", "inline-unpack", "trip-null-src", "trip-null-dst"])
def test_missing_page_ids_are_refused(recorder, kind, k, host):
    """NULL ids are an error of the caller's, not pages 0 to n - 1, however
    many chunks a call has and whatever its host memory is."""
    kind = kind if "null" in kind else f"{kind}-null"
    got = run(recorder, f"{kind}:{k}:a:{host}", f"trip:6:b:{host}")
    assert got["status"] == [_native.PACE_KV_EINVAL]
    assert not pages_of(got["calls"][0]) or kind == "trip-null-dst"    # the way out comes first
    assert all(e["op"] in o["after"] for o in pages(got["calls"][1]) for e in got["calls"][0])
