"""A forward with strips has the same bits with and without its workspace: where
the workspace may not grow (a frozen context, a captured stream) the strips of a
disc are summed one after the other in the same order.  Before, such a call took
whole discs, and a call captured after a smaller one could not be captured at all.

Sky NSIDE 64, beam NSIDE 512 with a flat cap of 36 deg (9.2 MB, 4,700 pixels: five
strips); every 64th sky pixel holds 2^60, the next one -2^60, so that another order
of the additions shows in the TOD."""
import math

import numpy as np
import pytest
import torch

from pisco4cmb_amd import inputs, pypisco, torch_ops
from pisco4cmb_amd._lib import check, lib
from test_launch_shape import shape

pytestmark = pytest.mark.gpu
NS, NB, CAP = 64, 512, 36.0


def t(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to("cuda")


class Forward:
    def __init__(self, n):
        self.n = n
        sky = [x.copy() for x in inputs.iid_sky(NS, seed=3)]
        sky[0][::64] = 2.0 ** 60
        sky[0][1::64] = -(2.0 ** 60)
        self.sky = [t(x) for x in sky]
        npix = pypisco.beam_npix_for_radius(NB, math.radians(CAP))
        self.beam8 = torch.zeros((npix, 8), device="cuda")
        self.beam8[:, 0] = 1.0
        self.beam8[:, 3] = 1.0
        self.beam8[:, 6] = 0.5
        self.ptg = [t(x) for x in inputs.ces_scan(n, t0=700.0)]
        self.out = [torch.empty(n, device="cuda") for _ in range(2)]

    def __call__(self, ctx, n=None, v=False):
        args = [s.data_ptr() for s in self.sky[:4 if v else 3]]
        f = lib.pisco_dev_forward_v if v else lib.pisco_dev_forward
        check(f(ctx, torch_ops._stream(torch.device("cuda:0")), NS, *args, NB,
                self.beam8.shape[0], self.beam8.data_ptr(), n or self.n,
                *[x.data_ptr() for x in self.ptg], *[o.data_ptr() for o in self.out]))

    def bits(self):
        torch.cuda.synchronize()
        return [o.cpu().numpy().view(np.int32).copy() for o in self.out]


def same(x, y):
    return all(np.array_equal(a, b) for a, b in zip(x, y))


@pytest.fixture
def ctx():
    c = torch_ops.new_ctx(torch.device("cuda:0"))
    yield c
    torch.cuda.synchronize()
    lib.pisco_destroy(c)


@pytest.mark.parametrize("n", [1, 201, 1500])
@pytest.mark.parametrize("v", [False, True])
def test_frozen_without_workspace(ctx, n, v):
    assert shape(NS, NB, CAP)[:2] == [64, 5]
    f = Forward(n)
    check(lib.pisco_set_tuning(ctx, b"forward_lanes", 8))
    f(ctx, v=v)                                             # no strips yet
    check(lib.pisco_freeze_buffers(ctx, 1))
    check(lib.pisco_set_tuning(ctx, b"forward_lanes", 0))
    for o in f.out:
        o.fill_(float("nan"))
    f(ctx, v=v)
    frozen = f.bits()
    check(lib.pisco_freeze_buffers(ctx, 0))
    f(ctx, v=v)
    assert same(frozen, f.bits())


def test_captured_after_a_call_without_strips(ctx):
    n = 700
    f = Forward(n)
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        check(lib.pisco_set_tuning(ctx, b"forward_lanes", 8))
        f(ctx)                                              # ring table and packed sky
        check(lib.pisco_set_tuning(ctx, b"forward_lanes", 0))
        st.synchronize()
        g = torch.cuda.CUDAGraph()
        g.capture_begin()
        f(ctx)
        g.capture_end()
        ref = Forward(n)
        other = torch_ops.new_ctx(torch.device("cuda:0"))
        ref(other)
        want = ref.bits()
        for k in range(3):                                  # eager work between the replays
            for o in f.out:
                o.fill_(float("nan"))
            g.replay()
            assert same(f.bits(), want), k
            ref(other)
            assert same(ref.bits(), want)
    torch.cuda.synchronize()
    lib.pisco_destroy(other)


def test_workspace_is_the_size_of_the_call():
    """500 samples of five strips need 112 kB; a context held 27 MB for them, and the
    fixed array of the forward without allocations 32 MiB beside its sky."""
    import re
    f = Forward(500)
    ctx = torch_ops.new_ctx(torch.device("cuda:0"))
    check(lib.pisco_set_tuning(ctx, b"forward_lanes", 8))
    f(ctx)                                                  # everything but the strips
    check(lib.pisco_set_tuning(ctx, b"forward_lanes", 0))
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    f(ctx)
    torch.cuda.synchronize()
    assert free - torch.cuda.mem_get_info()[0] <= 4 << 20
    lib.pisco_destroy(ctx)
    rc = lib.pisco_dev_forward_noalloc(None, 1024, *[s.data_ptr() for s in f.sky[:3]], NB,
                                       f.beam8.shape[0], f.beam8.data_ptr(), 0, None, None, None,
                                       None, None)
    assert rc != 0
    size = int(re.search(r"(\d+)-byte", lib.pisco_last_error().decode()).group(1))
    assert size <= 48.2 * 2 ** 20 + (8 << 20)


@pytest.mark.parametrize("ns", [64, 512])
def test_noalloc_launches_of_what_its_workspace_holds(ns):
    """More samples than one launch's (sky NSIDE 512: 37,000 of six strips): the bits
    of the forward with allocations."""
    nb, cap, n = (512, 36.0, 3000) if ns == 64 else (4096, 5.0, 40001)
    f = Forward(n)
    if ns == 512:
        f.sky = [t(x) for x in inputs.iid_sky(ns, seed=4)]
        npix = pypisco.beam_npix_for_radius(nb, math.radians(cap))
        f.beam8 = torch.rand((npix, 8), device="cuda")
    args = (ns, *[s.data_ptr() for s in f.sky[:3]], nb, f.beam8.shape[0], f.beam8.data_ptr(), n,
            *[x.data_ptr() for x in f.ptg], *[o.data_ptr() for o in f.out])
    dev = torch.device("cuda:0")
    check(lib.pisco_dev_forward(torch_ops._ctx(dev), torch_ops._stream(dev), *args))
    want = f.bits()
    for o in f.out:
        o.fill_(float("nan"))
    check(lib.pisco_dev_forward_noalloc(torch_ops._stream(dev), *args))
    assert same(f.bits(), want)
