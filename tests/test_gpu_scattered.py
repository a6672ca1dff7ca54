"""Sky adjoint of pointings in no order: a block's samples lie all over the sky or
some radii apart, its windows would hold the gaps between them, and its sums go to
global memory instead.  Samples all over the sky, in a few far groups, on a coarse
grid, and along a scan (which keep their windows), with and without strips, and
batched; both kinds of sums.  Tolerance: relative RMS 1e-6 of the oracle, the bound
of the other sky adjoint tests."""

import numpy as np
import pytest
import torch

from pisco4cmb_amd import inputs, pypisco
from pisco4cmb_amd.batched import DetectorBatch
from test_gpu_strips import Calls, make, rel_rms
from test_launch_shape import shape

pytestmark = pytest.mark.gpu
N = 700


def pointings(kind):
    r = np.random.default_rng(17)
    if kind == "sky":
        x = r.uniform(0, 2 * np.pi, N), np.arcsin(r.uniform(-1, 1, N)), r.uniform(-np.pi, np.pi, N)
    elif kind == "groups":      # samples by turns at five places
        k = np.arange(N) % 5
        x = 1.3 * k + 0.01 * r.normal(size=N), 0.5 * (k - 2) + 0.01 * r.normal(size=N), 0.3 * k
    elif kind == "grid":        # about a disc's radius from sample to sample
        k = np.arange(N)
        x = 0.1 * (k % 27), -1.2 + 0.1 * (k // 27), 0.2 * k
    else:
        x = inputs.ces_scan(N, t0=321.0)
    return [np.ascontiguousarray(v, np.float32) for v in x]


@pytest.mark.parametrize("kind", ["sky", "groups", "grid", "scan"])
@pytest.mark.parametrize("ns,nb,cap,strips", [(128, 1024, 20.0, 2), (128, 1024, 6.0, 1), (64, 512, 3.0, 1)])
def test_single(oracle, kind, ns, nb, cap, strips):
    assert shape(ns, nb, cap, N)[2:4] == [64, strips]
    sky, beam, _, _, _, g = make(ns, nb, cap, N, 19)
    ra, dec, pa = pointings(kind)
    conv = pypisco.GPUConvolver(pypisco.default_run_config())
    conv.configure_execution()
    c = Calls(ns, nb, beam, sky)
    c.ctx = conv.ctx
    ref = oracle.adjoint_map(ns, nb, list(beam.aBeams) + list(beam.bBeams), ra, dec, pa, *g)
    for det in (0, 1):
        for lanes in (0, 64, 16, 8):
            c.tune(adjmap_deterministic=det, adjmap_lanes=lanes)
            for x, r in zip(c.adjoint(ra, dec, pa, *g), ref):
                assert rel_rms(x, r) < 1e-6, (det, lanes)


@pytest.mark.parametrize("kind", ["sky", "groups", "grid", "scan"])
def test_batched(oracle, kind):
    ns, nb = 64, 512
    ra, dec, pa = pointings(kind)
    beams = [inputs.make_polbeam("crosspolar" if k % 2 else "copolar", nb, c, c / 3, 0.05, 0.01,
                                 nside_sky=ns) for k, c in enumerate((6.0, 2.0, 9.0))]
    def t(a):
        return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to("cuda")

    g = np.random.default_rng(3).normal(size=(3, 2, N)).astype(np.float32)
    ref = 0.0
    off = [0.0, 0.4, -1.0]
    for k, b in enumerate(beams):
        p = (pa + np.float32(off[k])).astype(np.float32)
        ref = ref + np.asarray(oracle.adjoint_map(ns, nb, list(b.aBeams) + list(b.bBeams), ra, dec, p, g[k, 0], g[k, 1]),
                               np.float64)
    for pair_major in (0, 1):
        batch = DetectorBatch([(t(np.stack(b.aBeams)), t(np.stack(b.bBeams)), nb, off[k])
                               for k, b in enumerate(beams)])
        batch.set_tuning("batch_pair_major", pair_major)
        out = batch.adjoint_map(t(g), t(ra), t(dec), t(pa), ns)
        for x, r in zip(out, ref):
            assert rel_rms(x.cpu().numpy(), r) < 1e-6, pair_major
        batch.close()
