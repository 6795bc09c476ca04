"""Failed device allocations, on the CPU: the library's host code compiled without its kernels
and linked to host/hip_runtime.cpp, which fails the n-th allocation.  What a call leaves
behind must be usable: a buffer that was given back and not replaced is not taken for the
one it was."""
import shutil
import subprocess
from pathlib import Path

import pytest

from shiokaze_amd import build as B

HERE = Path(__file__).resolve().parent / "host"

pytestmark = pytest.mark.skipif(shutil.which("g++") is None or not Path(B.HIPCC).exists(), reason="no compilers")


def _run(tmp_path, program, sources):
    objs = []
    jobs = []
    for s in sources:
        o = tmp_path / f"{s}.o"
        objs.append(str(o))
        jobs.append([B.HIPCC, *B.COMMON, "-O1", "-w", "--offload-host-only", "-c", str(B.CSRC / f"{s}.hip"), "-o", str(o)])
    for s in (program, "hip_runtime"):
        o = tmp_path / f"{s}.o"
        objs.append(str(o))
        jobs.append([B.HIPCC, *B.COMMON, "-O1", "-w", "-x", "hip" if s == program else "c++", "--offload-host-only", "-c",
                     str(HERE / f"{s}.cpp"), "-o", str(o)])
    procs = [subprocess.Popen(j, stderr=subprocess.PIPE, text=True) for j in jobs]
    for p in procs:
        err = p.communicate(timeout=300)[1]
        assert p.returncode == 0, err
    exe = tmp_path / "prog"
    # kernels and the functions that the program does not reach stay undefined
    subprocess.run(["g++", "-no-pie", *objs, "-o", str(exe), "-Wl,--unresolved-symbols=ignore-all"], check=True)
    r = subprocess.run([str(exe), str(tmp_path / "file")], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


def test_training_step(tmp_path):
    _run(tmp_path, "unet_alloc", ("unet", "unet_kernels"))


def test_multigrid_tables(tmp_path):
    _run(tmp_path, "mg_alloc", ("mgsolve", "mg"))


def test_csr_multigrid_hierarchy(tmp_path):
    _run(tmp_path, "amg_alloc", ("amg",))


def test_learned_preconditioner(tmp_path):
    _run(tmp_path, "precond_alloc", ("unet", "unet_kernels"))
