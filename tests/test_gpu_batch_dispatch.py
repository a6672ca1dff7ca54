"""The batched forward's automatic choice of pairs per wave: pairs whose packed
beams are large leave the groups of four, whose gathers from four beams then miss
the L2.  Shapes (sky NSIDE, beam NSIDE, cap; beam, disc): 64, 256, 30 deg (1.6 MiB,
3,300 pixels: groups of two, and of four from 2,048 to 6,143 samples), 64, 256, 36 deg (2.3 MiB, 4,700: a pair's items), 48,
512, 18 deg (2.4 MiB, 680: a pair's items) and 64, 256, 12 deg (0.3 MiB, 540: four).

The choice shows in the order of the FP64 sums: with flat beams and a sky that
holds 2^60 at every 64th pixel and -2^60 beside it, the default has the bits of
the group that is named, and not those of the other groups.  With ordinary beams
and skies every pair agrees with the oracle to relative RMS 1e-6, the bound of the
other batched tests; unequal discs in one block of four included."""
import math

import numpy as np
import pytest
import torch

from pisco4cmb_amd import inputs, pypisco
from pisco4cmb_amd.batched import DetectorBatch

pytestmark = pytest.mark.gpu


def t(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to("cuda")


def rel_rms(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.sqrt(np.mean((a - b) ** 2)) / max(np.sqrt(np.mean(b ** 2)), 1e-300))


@pytest.mark.parametrize("ns,nb,cap,group,n",
                         [(64, 256, 30.0, 2, 300), (64, 256, 30.0, 2, 2047), (64, 256, 30.0, 4, 2048),
                          (64, 256, 30.0, 4, 6143), (64, 256, 30.0, 2, 6144), (64, 256, 36.0, 1, 300),
                          (64, 256, 36.0, 1, 3000), (48, 512, 18.0, 1, 300), (64, 256, 12.0, 4, 300)])
def test_default_group(ns, nb, cap, group, n):
    sky = [x.copy() for x in inputs.iid_sky(ns, seed=3)[:3]]
    sky[0][::64] = 2.0 ** 60
    sky[0][1::64] = -(2.0 ** 60)
    ra, dec, pa = (t(x) for x in inputs.ces_scan(n, t0=700.0))
    beams = []
    for f in (1.0, 0.99, 0.95, 0.94):   # a group walks the disc of its largest pair
        beam = np.zeros((4, pypisco.beam_npix_for_radius(nb, math.radians(f * cap))), np.float32)
        beam[0] = 1.0
        beams.append(t(beam))
    out = {}
    for g in (0, 1, 2, 4):   # 0: the default
        batch = DetectorBatch([(b, b, nb, 0.3 * k) for k, b in enumerate(beams)])
        batch.set_tuning("batch_pair_major", 0)
        if g:
            batch.set_tuning("batch_group", g)
        out[g] = batch.forward(*(t(x) for x in sky), ra, dec, pa, ns).cpu().numpy()
        assert batch.get_tuning("batch_group") == (g or 4)
        batch.close()
    for g in (1, 2, 4):
        same = np.array_equal(out[0].view(np.int32), out[g].view(np.int32))
        assert same == (g == group), g


@pytest.mark.parametrize("ns,nb,caps", [(64, 256, [30.0] * 4), (64, 256, [36.0] * 4 + [30.0] * 2),
                                        (48, 512, [18.0] * 3), (64, 256, [37.0, 36.0, 27.0, 24.0]),
                                        (64, 256, [36.0, 30.0, 12.0, 4.0, 3.0])])
def test_every_choice_vs_oracle(oracle, ns, nb, caps):
    n = 33
    sky = [x.copy() for x in inputs.iid_sky(ns, seed=5)[:3]]
    sky[0] = np.abs(sky[0]) + 1   # no cancellation in the sums
    ra, dec, pa = inputs.ces_scan(n, t0=321.0)
    dec[:4] = np.array([89.9, -89.9, 88.0, -85.0], np.float32) * np.float32(math.pi / 180)
    beams = [inputs.make_polbeam("crosspolar" if k % 2 else "copolar", nb, c, c / 3, 0.05, 0.01,
                                 nside_sky=ns) for k, c in enumerate(caps)]
    offs = [0.4 * k - 1.0 for k in range(len(caps))]
    batch = DetectorBatch([(t(np.stack(b.aBeams)), t(np.stack(b.bBeams)), nb, o)
                           for b, o in zip(beams, offs)])
    batch.set_tuning("batch_pair_major", 0)
    tod = batch.forward(*(t(x) for x in sky), t(ra), t(dec), t(pa), ns).cpu().numpy()
    batch.close()
    for k, (b, o) in enumerate(zip(beams, offs)):
        p = (pa + np.float32(o)).astype(np.float32)
        ref = oracle.convolve(ns, *sky, nb, list(b.aBeams) + list(b.bBeams), ra, dec, p)
        assert rel_rms(tod[k, 0], ref[0]) < 1e-6 and rel_rms(tod[k, 1], ref[1]) < 1e-6
