"""The host layer's use of workspaces (CPU only): the built library driven by tests/cpp/workspace_regions.cpp, which
stands in for its kernel launchers and HIP calls."""
from __future__ import annotations

import os
import subprocess
from pathlib import Path

import ascq

ROOT = Path(__file__).resolve().parent.parent
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def _run(tmp_path, name):
    exe = tmp_path / name
    libdir = Path(ascq.LIB_PATH).parent
    subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-host-only", "-x", "hip", "-std=c++17", "-O1", "-I", str(ROOT / "include"),
                    str(ROOT / "tests" / "cpp" / f"{name}.cpp"), "-rdynamic", "-L", str(libdir), "-lascq",
                    f"-Wl,-rpath,{libdir}", "-Wl,-rpath,/opt/rocm/lib", "-o", str(exe)],
                   check=True)
    return subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)


def test_regions_of_a_call_are_disjoint(tmp_path):
    """int8 and fp8, org x single shape x layout x alignment, in a handle's own workspace, a caller's of the reported
    size, a larger one and the static scratch: packed operands, operand copies and split partials share no byte"""
    r = _run(tmp_path, "workspace_regions")
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-2000:]


def test_captured_memory_outlives_eager_calls(tmp_path):
    """A graph captured over a handle that uses its own workspace, then eager calls whose operands are packed: the memory
    that the graph uses stays allocated, and captured calls pack into a caller's workspace only"""
    r = _run(tmp_path, "workspace_lifetime")
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-2000:]


def test_overlapping_streams_share_no_room(tmp_path):
    """Calls of one handle on several streams and devices pack into rooms of their own (four at most), allocated and freed
    without harm to captures of other streams"""
    r = _run(tmp_path, "workspace_streams")
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-2000:]


def test_allocation_free_calls_pack_nothing(tmp_path):
    """IterateAllNoAlloc with operands off their alignment does not pack them into the scratch that all handles share"""
    r = _run(tmp_path, "workspace_noalloc")
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-2000:]


def test_workspace_off_its_alignment_is_not_packed_into(tmp_path):
    """A caller's workspace off 16 bytes: calls whose operands would be packed there run without, and none is refused"""
    r = _run(tmp_path, "workspace_offset")
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-2000:]
