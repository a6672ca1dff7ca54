"""The map-maker's path for a pointing shared by the detectors against the
oracle, bit for bit: pixels hit by 1, 15, 16, 17, 64 and 70 samples (around
the lanes of a group; with 33 detectors the last two take a whole wave), sample counts around a sort tile (1,024 and, from 2^20
samples, 4,096), skipped samples, data that are infinite, and a pass smaller
than the pointing, which takes the general path."""
import math

import numpy as np
import pytest
import torch

from pisco4cmb_amd._lib import check, lib
from pisco4cmb_amd.mapmaker import DeviceSkyMap

pytestmark = pytest.mark.gpu


def t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


@pytest.mark.parametrize("n,ndet,chunk", [(1, 2, None), (49, 2, None), (49, 16, 48), (1023, 3, None),
                                          (1024, 5, None), (1025, 33, None), (20000, 2, None),
                                          ((1 << 20) + 1, 2, None)])
def test_shared_pointing_bits(oracle, n, ndet, chunk):
    nside = 16
    rng = np.random.default_rng(n)
    ra = rng.uniform(0, 2 * math.pi, n).astype(np.float32)
    dec = np.arcsin(rng.uniform(-1, 1, n)).astype(np.float32)
    pa = rng.uniform(-math.pi, math.pi, n).astype(np.float32)
    k = 0
    more = ((70, 0.9), (64, -0.9)) if n > 1000 else ()
    for m, centre in ((15, 0.1), (16, 0.5), (17, -0.4)) + more:   # m samples of one pixel
        ra[k:k + m] = np.float32(1.0)
        dec[k:k + m] = np.float32(centre)
        k += m
    if n > 100:
        dec[n // 2] = 2.0   # skipped
        ra[n // 2 + 3] = np.inf
    pol = rng.uniform(-math.pi, math.pi, ndet).astype(np.float32)
    data = rng.normal(0, 30, (ndet, n)).astype(np.float32)
    if n > 1000:
        data[1, n - 9] = np.inf
    m = DeviceSkyMap(nside)
    if chunk:
        check(lib.pisco_skymap_set_chunk(m.handle, chunk))
    for _ in range(2):   # the second call adds onto the first one's sums
        m.accumulate(t(ra), t(dec), t(pa), t(pol), t(data), shared_pointing=True)
    AtA = AtD = None
    for _ in range(2):
        AtA, AtD, skipped = oracle.skymap_accumulate(nside, ra, dec, pa, pol, data, AtA, AtD,
                                                     shared_pointing=True)
    a, d = np.empty((12 * nside ** 2, 9)), np.empty((12 * nside ** 2, 3))
    torch.cuda.synchronize()
    check(lib.pisco_skymap_get_normal(m.handle, a.ctypes.data, d.ctypes.data))
    assert np.array_equal(a, AtA)
    assert np.array_equal(d, AtD, equal_nan=True)
    assert m.skipped() == 2 * skipped == (4 * ndet if n > 100 else 0)
    m.close()
