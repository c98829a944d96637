"""The ring of pinned memory that carries the engine's tables to the device: past a
half, through growth, with a slow stream, and without pinned memory (each table must
arrive as it was).  Compiled for the host against a model of the runtime."""
import os
import subprocess

import pytest

from ptb_amd.build import CSRC, HIPCC, ROOT

SRC = os.path.join(ROOT, "tests", "native", "table_ring.cpp")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_tables_through_the_pinned_ring(tmp_path):
    exe = str(tmp_path / "table_ring")
    flags = ["-O1", "-std=c++20", "-fPIC", "-Wno-unused-result", "-I", CSRC, "-I", os.path.join(ROOT, "include")]
    objs = []
    for src in (os.path.join(CSRC, "api.hip"), SRC):
        obj = str(tmp_path / (os.path.basename(src) + ".o"))
        subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "--offload-arch=gfx950", *flags, "-c", src, "-o", obj],
                       check=True)
        objs.append(obj)
    # (the runtime's other functions, and the engine's kernels, are never called)
    subprocess.run(["g++", "-o", exe, *objs, "-lpthread", "-Wl,--unresolved-symbols=ignore-all"], check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    print(run.stdout)
    assert run.returncode == 0, run.stdout
