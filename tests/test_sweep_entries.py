"""The accessors of the sweeps' vector entries, as the compiler sees them (built here, host
only): they touch double arrays through an integer type, so their accesses must not carry
a type that excludes a double at the same address."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "swcholesky_amd", "csrc")

SOURCE = """#include <hip/hip_runtime.h>
namespace {
#include "sweep_entries.h"
}
__global__ void mark(double* x, double* y) { const double b = *x; mark_pending(x); *y = b; }
__global__ void put(double* x, double v) { publish(x, v); }
__global__ void get(double* x, unsigned long long* y) { *y = load_entry(x); }
"""


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="no hipcc")
def test_entry_accesses_may_alias_doubles(tmp_path):
    src = tmp_path / "entries.hip"
    src.write_text(SOURCE)
    ir = subprocess.run(["hipcc", "--offload-arch=gfx950", "-O1", "--cuda-device-only", "-emit-llvm", "-S", "-I", CSRC,
                         "-o", "-", str(src)], check=True, capture_output=True, text=True).stdout
    bodies = dict(re.findall(r"^define [^@]*@_Z\d+(mark|put|get)P\S*\([^{]*\{(.*?)^\}", ir, re.S | re.M))
    accesses = {"mark": r"store i64 .*", "put": r"store atomic i64 .*", "get": r"load atomic i64, .*"}
    for name, pattern in accesses.items():
        lines = re.findall(pattern, bodies[name])
        assert len(lines) == 1, (name, bodies[name])
        tag = re.search(r"!tbaa !(\d+)", lines[0])
        if tag:  # the access type it names, or none
            node = re.search(rf"^!{tag.group(1)} = !{{!(\d+),", ir, re.M).group(1)
            kind = re.search(rf'^!{node} = !{{!"([^"]*)"', ir, re.M).group(1)
            assert kind == "omnipotent char", (name, kind)
