"""Flux rows are ordered by photon energy before neighbours share integrand
factors: in buckets of 0.27 %, ordered by a wavefront up to 128 rows, by a workgroup
up to 1,024, and by row number through a bitmap of 262,144 rows at a time beyond.
Equal calls give equal bits (the order decides which rows expand J1 together), a
point is what a small call makes of it (1e-11: see the other routes' tests), and
points that crowd into few buckets do not cost more to order than to integrate."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CFG = dict(flux_point=0, breakup_mode=2, nm=3, ny=3)


def _points(n, width, seed):
    """n points at (10 GeV, 0.5), M within `width` of it."""
    rng = np.random.default_rng(seed)
    return 10.0 * np.exp(width * rng.uniform(-1, 1, n)), np.full(n, 0.5)


# rows a bucket: about 50, 130, 500, 2,000; more than 1,024 from two windows of the bitmap
@pytest.mark.parametrize("n,width", [(4100, 0.11), (4100, 0.042), (4100, 0.011), (8200, 0.004), (140000, 0.1),
                                     (140000, 0.0)])
def test_order_is_the_same_every_time(gpu, n, width):
    import torch
    M, Y = (torch.as_tensor(v, device="cuda") for v in _points(n, width, 3))
    bits = lambda x: x.view(torch.int64)
    with gpu.Context(**CFG) as c, gpu.Context(**CFG) as d:
        L = c.lumi_points(M, Y)
        assert c.info.qags_bad == 0
        for again in (c, c, d):
            assert torch.equal(bits(again.lumi_points(M, Y)), bits(L))
        idx = torch.as_tensor(np.random.default_rng(4).choice(n, 690, replace=False), device="cuda")
        one = c.lumi_points(M[idx].contiguous(), Y[idx].contiguous())
        assert float((L[idx] / one - 1).abs().max()) <= 1e-11


def test_batch_orders_as_its_context(gpu):
    """A job whose bins crowd into a few buckets, between two others."""
    import torch
    narrow = dict(CFG, nm=120, ny=100, mmin=10.0, mmax=10.05, ymin=0.0, ymax=0.004)
    jobs = [gpu.Config.make(**dict(CFG, nm=100, ny=90)), gpu.Config.make(**narrow), gpu.Config.make(**CFG)]
    b = gpu.Batch(jobs)
    first = [o.clone() for o in b.run(graph=False)]
    for got, L in zip(b.run(graph=False), first):
        assert torch.equal(got.view(torch.int64), L.view(torch.int64))
    b.close()
    for L, cfg in zip(first, jobs):
        with gpu.Context(cfg) as c:
            ref = c.lumi_grid()
        nan = torch.isnan(ref)
        assert torch.equal(nan, torch.isnan(L))
        assert float((L[~nan] / ref[~nan] - 1).abs().max()) <= 1e-12


def test_crowded_rows_are_ordered_in_time(gpu):
    """8,192 rows in four or five buckets: what precedes the integrals takes less than
    half of their time (the best of five; 1.2 of it when one wavefront looked
    through all rows for those of its bucket)."""
    import torch
    M, Y = (torch.as_tensor(v, device="cuda") for v in _points(4096, 0.002, 5))
    with gpu.Context(**CFG) as c:
        c.lumi_points(M, Y)
        c.set_timing(True)
        share = []
        for _ in range(5):
            c.timings(reset=True)
            c.lumi_points(M, Y)
            t = c.timings(reset=True)
            share.append(t["flux"][0] / t["qags"][0])
        assert min(share) < 0.5, share
