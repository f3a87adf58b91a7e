"""The dispatch of the row kernels and the quantizer over every accepted width and extreme row counts, on the CPU
(row_dispatch.hip): each call launches something, every row is covered once, no grid reaches HIP's limit of 2^32
threads, and every row kernel that is built can be chosen."""
from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

from v7multiplikator_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    """(exit code, output, the kernels in the program)."""
    d = tmp_path_factory.mktemp("row_dispatch")
    obj, exe = str(d / "row_dispatch.o"), str(d / "row_dispatch")
    flags = [f for f in build.HIP_FLAGS if f not in ("-shared", "-O3", "-Wall")]
    res = subprocess.run([build.hipcc(), *flags, "-O1", "--offload-host-only", "-c", "-o", obj,
                          os.path.join(HERE, "row_dispatch.hip")], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    # no HIP runtime and no device code: the launch symbols stay unresolved and are never called
    res = subprocess.run(["g++", "-rdynamic", "-no-pie", "-Wl,-z,lazy", "-Wl,--unresolved-symbols=ignore-all", "-o", exe,
                          obj, "-ldl"], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    run = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    nm = subprocess.run([shutil.which("nm"), exe], capture_output=True, text=True, check=True).stdout
    built = {line.split()[-1] for line in nm.splitlines()
             if re.search(r"_ZN3v7g\d+(rmsnorm_(row|padded_row|q8_row)_kernel|norm_q8_row16_kernel)I", line)}
    return run.returncode, run.stdout + run.stderr, built


def test_every_shape_is_launched_within_the_grid_limit(probe):
    rc, out, _ = probe
    assert "FAULT" not in out, out[:4000]
    assert rc == 0 and out.rstrip().endswith("0 faults")


def test_every_built_row_kernel_is_reachable(probe):
    _, out, built = probe
    chosen = set(re.findall(r"KERNEL (\S+)", out))
    assert len(built) > 100
    assert built <= chosen, sorted(built - chosen)
