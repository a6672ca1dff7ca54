"""The (unit, sample) items of the strip and batch launches (csrc/work_items.h),
on the CPU: every item of the grid is work, each (unit, sample) comes once, a
chunk's items of one unit are consecutive, and the eight contiguous stretches of
the grid that the XCDs take hold equal shares also where the samples do not fill
a chunk."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("items") / "work_items_host.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC",
                    "-I" + os.path.join(ROOT, "pisco4cmb_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "work_items_host.cpp"), "-o", so],
                   check=True)
    lib = ctypes.CDLL(so)
    lib.launch_items.restype = ctypes.c_long
    lib.launch_items.argtypes = [ctypes.c_long] * 4 + [ctypes.c_void_p] * 2
    return lib


@pytest.mark.parametrize("nsamp", [1, 7, 250, 1023, 1024, 1025, 2500])
@pytest.mark.parametrize("nunits,chunk", [(1, 1024), (2, 1024), (6, 1024), (2, 512), (33, 1024)])
def test_every_item_is_work(host, nsamp, nunits, chunk):
    cap = 2 * nsamp * nunits + 10 * chunk * nunits
    unit, sample = np.full(cap, -2, np.int64), np.full(cap, -2, np.int64)
    n = host.launch_items(nsamp, nunits, chunk, cap, unit.ctypes.data, sample.ctypes.data)
    assert n == nsamp * nunits
    unit, sample = unit[:n], sample[:n]
    assert unit.min() >= 0 and unit.max() < nunits
    assert np.array_equal(np.sort(unit * nsamp + sample), np.arange(n))
    key = (sample // chunk) * nunits + unit          # chunk by chunk, unit by unit
    assert np.all(np.diff(key) >= 0)
    same = np.diff(key) == 0
    assert np.all(np.diff(sample)[same] == 1)
