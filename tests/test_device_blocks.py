"""The library's device memory on the CPU: idle table blocks go back where they
are needed. tests/blocks/blocks_check.cpp stands in for the HIP calls that
allocate; the library is the built one."""
from __future__ import annotations

import re
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CSRC = ROOT / "process_amd" / "csrc"


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    from process_amd import _lib
    _lib.lib()  # built if it is not there
    exe = tmp_path_factory.mktemp("blocks") / "blocks_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", str(ROOT / "include"), "-I", str(CSRC),
                    "-isystem", "/opt/rocm/include", str(ROOT / "tests" / "blocks" / "blocks_check.cpp"),
                    str(ROOT / "process_amd" / "libpsx.so"), f"-Wl,-rpath,{ROOT / 'process_amd'}",
                    "-rdynamic", "-Wl,--allow-shlib-undefined", "-o", str(exe)], check=True)

    def run(what: str):
        out = subprocess.run([str(exe), what], capture_output=True, text=True, timeout=120)
        assert out.returncode == 0 and "blocks ok" in out.stdout, out.stdout + out.stderr

    return run


def test_callers_buffers_take_the_memory_of_idle_blocks(check):
    check("alloc")


def test_trim_gives_idle_blocks_back(check):
    check("trim")


def test_idle_blocks_are_not_reported_free(check):
    check("info")


def test_a_table_freed_during_a_capture_leaves_no_error(check):
    check("capture")


def test_device_memory_is_allocated_in_one_place():
    """psx_dev_malloc gives idle blocks back when memory runs out; nothing allocates past it."""
    calls = [f"{f.name}: {line.strip()}" for f in sorted(CSRC.iterdir()) for line in f.read_text().splitlines()
             if re.search(r"\bhipMalloc(Async)?\s*\(", line.split("//")[0])]
    assert len(calls) == 2 and all(c.startswith("psx_host.cpp:") for c in calls), calls
