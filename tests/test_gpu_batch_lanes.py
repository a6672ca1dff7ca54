"""Per-pair batch items: a pair's TOD has the same bits whatever other pairs are
in the batch.  The lanes per sample, and with them the order of a sample's FP64
sums, follow the pair's own disc; before, they followed the batch's largest.

Sky NSIDE 64: discs of 86 pixels (4.8 deg) alone, and beside one of 2,500 pixels
(26 deg, 64 lanes).  The beams are flat and every 64th sky pixel holds 2^60, the
next one -2^60: a sum over a disc that holds both loses the low bits of what the
same lane has added, so that another order of the additions shows in the TOD."""
import math

import numpy as np
import pytest
import torch

from pisco4cmb_amd import inputs, pypisco
from pisco4cmb_amd.batched import DetectorBatch

pytestmark = pytest.mark.gpu


def t(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to("cuda")


@pytest.mark.parametrize("n", [40, 2100])
@pytest.mark.parametrize("per_pair", [True, False])
def test_tod_does_not_depend_on_the_other_pairs(n, per_pair):
    ns, nb = 64, 256
    sky = [x.copy() for x in inputs.iid_sky(ns, seed=3)[:3]]
    sky[0][::64] = 2.0 ** 60
    sky[0][1::64] = -(2.0 ** 60)
    small, large = (pypisco.beam_npix_for_radius(nb, math.radians(c)) for c in (4.8, 26.0))

    def spec(npix, off):
        beam = np.zeros((4, npix), np.float32)
        beam[0] = 1.0
        return t(beam), t(beam), nb, off

    ra, dec, pa = inputs.ces_scan(n, t0=700.0)
    I, Q, U = (t(x) for x in sky)

    def forward(specs):
        batch = DetectorBatch(specs)
        batch.set_tuning("batch_group", 1)
        batch.set_tuning("batch_pair_major", 0)
        p = [np.stack([x] * len(specs)) if per_pair else x for x in (ra, dec, pa)]
        out = batch.forward(I, Q, U, *(t(x) for x in p), ns).cpu().numpy()
        batch.close()
        return out

    alone = forward([spec(small, 0.3)])[0]
    beside = forward([spec(large, -1.0), spec(small, 0.3), spec(large, 0.1)])[1]
    assert np.isfinite(alone).all() and np.abs(alone).max() > 0
    assert np.array_equal(alone.view(np.int32), beside.view(np.int32))
