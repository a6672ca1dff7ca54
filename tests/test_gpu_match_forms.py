"""Accuracy of the kernels' cos, sin(2chi) in single precision, against the oracle's
chi, and of the sky gradient over small discs against the oracle's FP64 adjoint.

The float form is within 2.3e-6 |eta| + 4e-8 of FP64, where eta < 0.026 tan|dec|
over a 1.5-degree disc: at |dec| < 0.17, |eta| < 0.0045, 5e-8 (the half unit in the
last place of a result near 1 is 3e-8; a phase rounded to float before the turn by
2 psi reached 5.9e-8).  Near the poles 2.5e-7: the FP64 form beyond |eta| = 0.078, also
in the sky adjoint with several samples per wave, whose Q and U gradients of
1.5-degree discs at 86 degrees were 1.2 times less accurate with 0.38.  Their bound
here, relative RMS 6.5e-8, is the error of an FP64 geometry with every product
rounded to float, over ten seeds 6.4e-8 and 6.6e-8."""
import math

import numpy as np
import pytest

from test_gpu_strips import Calls, rel_rms
from pisco4cmb_amd import inputs

pytestmark = pytest.mark.gpu


def pointings(n, seed, dec):
    rng = np.random.default_rng(seed)
    return (rng.uniform(0, 2 * math.pi, n).astype(np.float32),
            (np.resize(dec, n) + rng.uniform(-0.01, 0.01, n)).astype(np.float32),
            rng.uniform(-math.pi, math.pi, n).astype(np.float32))


@pytest.mark.parametrize("dec,tol", [([0.0, 0.15, -0.15], 5e-8),
                                     ([1.2, -1.3, 1.45, -1.5, 1.55, -1.56], 2.5e-7)])
@pytest.mark.parametrize("ns,nb", [(256, 2048), (512, 4096)])
def test_phase_in_single_precision(gpu, oracle, ns, nb, dec, tol):
    ra, dec, pa = pointings(600, ns, np.array(dec))
    off, pix = oracle.query_disc_many(ns, ra, dec, math.radians(1.5))
    want, chi = oracle.match(ns, nb, ra, dec, pa, off, pix)
    bp, c2, s2 = gpu.match_fast(ns, nb, ra, dec, pa, off, pix, mode=4)
    assert np.array_equal(bp, want)
    assert np.abs(c2 - np.cos(2 * chi)).max() <= tol
    assert np.abs(s2 - np.sin(2 * chi)).max() <= tol


@pytest.mark.parametrize("lanes", [8, 16])
@pytest.mark.parametrize("dec", [0.5, 1.1, 1.35, 1.5])
def test_gradient_of_small_discs(oracle, lanes, dec):
    ns, nb, cap, n = 256, 2048, 1.5, 2000
    beam = inputs.make_polbeam("crosspolar", nb, cap, cap / 2, 0.05, 0.01, nside_sky=ns)
    beams = list(beam.aBeams) + list(beam.bBeams)
    c = Calls(ns, nb, beam, inputs.iid_sky(ns, seed=1))
    c.tune(adjmap_lanes=lanes)
    err = []
    for seed in range(4):
        ra, d, pa = pointings(n, seed, np.array([dec]))
        g = np.random.default_rng(100 + seed).normal(size=(2, n)).astype(np.float32)
        ref = oracle.adjoint_map(ns, nb, beams, ra, d, pa, *g)
        err.append([rel_rms(x, r) for x, r in zip(c.adjoint(ra, d, pa, *g), ref)])
    c.tune(adjmap_lanes=0)
    err = np.mean(err, axis=0)
    print("I, Q, U", err)
    assert err.max() <= 6.5e-8


@pytest.mark.parametrize("ns,nb,cap,n", [(512, 2048, 3.0, 500), (512, 4096, 5.0, 200),
                                         (2048, 8192, 1.0, 150), (64, 512, 10.0, 500),
                                         (64, 64, 35.0, 60), (256, 8192, 2.0, 300)])
@pytest.mark.parametrize("polar", [False, True])
def test_batched_form(gpu, oracle, ns, nb, cap, n, polar):
    """The batched kernels' single-precision form: every pixel that it certifies is
    the oracle's.  It declines where a floor's argument lies within 4e-6 tmp + 2e-6
    of an integer, tmp <= sqrt(3 (1 - cos cap)) nside, three floors with two sides
    each, the arguments of ip larger by up to 4: at most 6 x 1.7 times that, and
    what the pole of the beam and the end of its polar cap add."""
    rng = np.random.default_rng(ns + nb)
    if polar:
        ra, dec, pa = pointings(n, ns, np.array([1.2, -1.3, 1.45, -1.5, 1.55, -1.56, 1.5707]))
    else:
        ra, dec, pa = pointings(n, ns, math.pi / 2 - np.arccos(rng.uniform(-1, 1, n)))
    off, pix = oracle.query_disc_many(ns, ra, dec, math.radians(cap))
    want, chi = oracle.match(ns, nb, ra, dec, pa, off, pix)
    bp, c2, s2 = gpu.match_fast(ns, nb, ra, dec, pa, off, pix, mode=6)
    sure = bp != -2
    assert np.array_equal(bp[sure], want[sure])
    assert np.abs(c2 - np.cos(2 * chi))[sure].max() <= 2.5e-7
    assert np.abs(s2 - np.sin(2 * chi))[sure].max() <= 2.5e-7
    tmp = math.sqrt(3 * (1 - math.cos(math.radians(cap)))) * nb
    # a declination beyond the pole has the exact form for every visit
    regular = np.repeat(np.abs(dec.astype(np.float64)) <= math.pi / 2, np.diff(off))
    assert not sure[~regular].any()
    declined = 1 - sure[regular].mean()
    print("declined %.2e, bound %.2e" % (declined, 10.2 * (4e-6 * tmp + 2e-6)))
    assert declined <= 10.2 * (4e-6 * tmp + 2e-6) + 2e-3
