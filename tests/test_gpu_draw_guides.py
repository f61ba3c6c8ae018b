"""Draws from prefix tables go through guides where a call makes many of them,
and through the plain search where it makes few.  The bin of a draw is unique,
so a call's events are, bit for bit, those of small calls at the same offsets:
tables with empty first, middle and last bins, single bins, and rows that are
all NaN (an empty z histogram)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _prefix(w):
    return np.concatenate([[0.0], np.cumsum(w / w.sum())])


def _tables(cfg, rng, pol):
    import torch
    ym = rng.gamma(0.2, size=cfg["nm"] * cfg["ny"])
    ym[rng.random(ym.size) < 0.3] = 0.0
    ym[0] = ym[-1] = 0.0
    if not ym.any():
        ym[:] = 1.0

    def rows():
        t = []
        for i in range(cfg["nm"]):
            z = rng.gamma(0.5, size=cfg["nz"])
            z[rng.random(z.size) < 0.3] = 0.0
            t.append(np.full(cfg["nz"] + 1, np.nan) if i % 7 == 3 or not z.any() else _prefix(z))
        return torch.as_tensor(np.array(t), device="cuda")

    out = dict(sum_ym=torch.as_tensor(_prefix(ym).reshape(1, -1), device="cuda"))
    if pol:
        out.update(sum_zs=rows(), sum_zp=rows(),
                   ratio=torch.as_tensor(rng.random((cfg["ny"], cfg["nm"])), device="cuda"))
    else:
        out.update(sum_z=rows())
    return out


@pytest.mark.parametrize("nm,ny,nz,pol", [(37, 5, 9, 0), (33, 4, 100, 1), (1, 2, 1, 0), (130, 65, 64, 0)])
def test_guided_draws_are_the_searched_ones(gpu, nm, ny, nz, pol):
    import torch
    cfg = dict(nm=nm, ny=ny, nz=nz)
    t = _tables(cfg, np.random.default_rng(nm), pol)
    c = gpu.Context(flux_point=1, breakup_mode=1, use_polarized=pol, proc_id=13, **cfg)
    n, part = 60_000, 400
    if nm == 1:
        part = 3  # a guide of a few entries
    bits = lambda x: x.view(torch.int64) if x.dtype == torch.float64 else x
    whole = c.sample_events(**t, n=n, seed=9)
    for off in (0, 777, n - part):
        got = c.sample_events(**t, n=part, seed=9, offset=off)
        for a, b in zip(got, whole):
            assert torch.equal(bits(a), bits(b[off:off + part]))
    c.photon_pt_tables(c.info.g1)
    opts = gpu.EventOpts(1, 0, 0.0, 0, 0.0, 0.0)
    p, pdg, ok = c.generate_pairs(**t, n=n, seed=9, opts=opts)
    drawn = ok != 0  # an event without a bin leaves its momenta unwritten
    for off in (0, 777, n - part):
        q, qdg, qok = c.generate_pairs(**t, n=part, seed=9, offset=off, opts=opts)
        d = drawn[off:off + part]
        assert torch.equal(qok, ok[off:off + part])
        assert torch.equal(bits(q)[d], bits(p[off:off + part])[d])
        assert torch.equal(qdg[d], pdg[off:off + part][d])
