"""The stand-alone measurement programs under benchmarks/ compile against the library's headers as they are.  No GPU."""
import glob
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.parametrize("program", sorted(os.path.basename(p) for p in glob.glob(os.path.join(ROOT, "intrasm_engine_amd", "benchmarks", "*.hip"))))
def test_it_compiles(program):
    proc = subprocess.run([HIPCC, "--offload-arch=gfx950", "-std=c++17", "-fsyntax-only", "-w",
                           os.path.join(ROOT, "intrasm_engine_amd", "benchmarks", program)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert proc.returncode == 0, proc.stdout[-3000:]
