"""The record form of the beam adjoint with bands that are patches of the polar
cap (rings by pixels of a quadrant) against the oracle: patches of 8, 9, 10 and
17 rings, a beam that ends in its first, middle or last ring block and at the
edge of the polar cap, and one beyond it (consecutive rows).  Tolerance:
relative RMS 1e-6 per column, as for the other forms."""
import numpy as np
import pytest

from pisco4cmb_amd import inputs, pypisco

pytestmark = pytest.mark.gpu


def rel_rms(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return float(np.sqrt(np.mean((a - b) ** 2)) / max(np.sqrt(np.mean(b ** 2)), 1e-300))


@pytest.mark.parametrize("nb,cap,rows", [(256, 4.0, 64), (256, 4.0, 81), (256, 4.0, 100),
                                         (256, 3.75, 64), (64, 47.9, 300), (64, 60.0, 300)])
def test_patches_vs_oracle(oracle, nb, cap, rows):
    ns = 128 if cap < 10 else 16
    sky = inputs.iid_sky(ns, seed=91)
    beam = inputs.make_polbeam("crosspolar", nb, cap, cap / 2, 0.05, 0.01, nside_sky=ns)
    ra, dec, pa = inputs.ces_scan(301, t0=50.0)
    ga, gb = (np.random.default_rng(k).normal(size=ra.size).astype(np.float32) for k in (92, 93))
    G = oracle.adjoint_beam(ns, *sky[:3], nb, list(beam.aBeams) + list(beam.bBeams), ra, dec, pa,
                            ga, gb)
    conv = pypisco.GPUConvolver(pypisco.default_run_config())
    conv.configure_execution()
    conv.update_sky(pypisco.Sky(ns, *sky))
    conv.update_beam(beam)
    conv.update_scan(pypisco.Scan(ra.size, ra, dec, pa))
    conv.set_tuning("adjbeam_rows", rows)
    for pool in (8192, 1):   # one chunk, several
        conv.set_tuning("adjbeam_pool_mb", pool)
        oa, ob = conv.exec_adjoint_beam(ga, gb)
        for k in range(3):
            assert rel_rms(oa[k], G[:, k]) < 1e-6
            assert rel_rms(ob[k], G[:, 3 + k]) < 1e-6
    conv.close()
