"""What the library asks of the allocators, and what it does without their
memory: child processes with tests/alloc_shim.c before the HIP runtime's
hipMalloc, hipFree and hipHostMalloc."""
import os
import shutil
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    gcc = shutil.which("gcc")
    assert gcc, "gcc is needed to build the allocation shim"
    so = str(tmp_path_factory.mktemp("shim") / "alloc_shim.so")
    subprocess.run([gcc, "-std=gnu11", "-O1", "-Wall", "-Werror", "-fPIC", "-shared",
                    os.path.join(HERE, "alloc_shim.c"), "-o", so, "-ldl"], check=True)
    return so


def _child(shim, *args):
    print("[gpu-case] allocations", *args, flush=True)
    r = subprocess.run([sys.executable, "-u", os.path.join(HERE, "alloc_child.py"), shim, *map(str, args)],
                       capture_output=True, text=True, timeout=100)
    print(r.stdout[-4000:], r.stderr[-4000:], sep="\n")
    assert r.returncode == 0 and r.stdout.rstrip().endswith("ok")


def test_pinned_slots_are_coherent(shim):
    _child(shim, "coherent")


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [1, (1 << 20) // 24, (1 << 20) // 24 + 1, (1 << 20) // 8 + 1])  # around a chunk's end
def test_transfers_without_pinned_memory(shim, precision, n):
    _child(shim, "no_pinned", precision, n)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("how", ["stages", "fused"])
def test_without_memory_for_records_and_filter(shim, precision, how):
    _child(shim, "tight", precision, how)
