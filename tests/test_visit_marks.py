"""The walk's run marks (csrc/visit_marks.h), on the CPU: every lane of a lane
group, with a visit or idling beside a group with more segments of marks, reads
an entry of its own table, and a lane with a visit the entry of its visit's run
(numpy's searchsorted)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("marks") / "visit_marks_host.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC",
                    "-I" + os.path.join(ROOT, "pisco4cmb_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "visit_marks_host.cpp"), "-o", so],
                   check=True)
    return ctypes.CDLL(so)


@pytest.mark.parametrize("lanes,vcap,rpp", [(8, 256, 24), (8, 256, 8), (16, 1024, 32),
                                           (16, 512, 16), (32, 1024, 32)])
def test_lanes_read_their_own_runs(host, lanes, vcap, rpp):
    rng = np.random.default_rng(lanes + rpp)
    for nrun in (0, 0, 1, 2, rpp - 1, rpp):
        for longest in (1, lanes, 3 * vcap // rpp + 1):
            ln = rng.integers(1, longest + 1, nrun)
            pref = np.concatenate([[0], np.cumsum(ln)]).astype(np.int32)
            total = int(pref[-1])
            for wtot in (max(total, 1), vcap, vcap + 1, 3 * vcap + 5):
                if wtot < total:
                    continue
                run = np.full(wtot, -99, np.int32)
                host.visit_runs(lanes, vcap, nrun, pref.ctypes.data_as(ctypes.c_void_p), wtot,
                                run.ctypes.data_as(ctypes.c_void_p))
                assert run.min() >= 0 and run.max() < max(nrun, 1)
                want = np.searchsorted(pref[:nrun], np.arange(total), side="right") - 1
                assert np.array_equal(run[:total], want)
