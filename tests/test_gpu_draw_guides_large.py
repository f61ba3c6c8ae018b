"""Guided draws from tables of realistic sizes: (Y, M) guides of many cells, z
guides behind them, and cells that hold several bins (more than 2^18 (Y, M) bins,
more than 2^10 z bins).  Bit for bit the events of small calls, which search.
test_host_paths.py checks that N draws from these tables take the guides and
PART draws do not."""
import numpy as np
import pytest

from test_gpu_draw_guides import _tables

pytestmark = pytest.mark.gpu

PART = 400
CASES = [  # nm, ny, nz, polarised, N
    (130, 65, 64, 0, 200_000),
    (130, 65, 64, 1, 200_000),
    (3, 2, 1500, 1, 60_000),
    (601, 443, 2, 0, 800_000),
]


@pytest.mark.parametrize("nm,ny,nz,pol,n", CASES)
def test_guided_draws_are_the_searched_ones(gpu, nm, ny, nz, pol, n):
    import torch
    t = _tables(dict(nm=nm, ny=ny, nz=nz), np.random.default_rng(nm + pol), pol)
    bits = lambda x: x.view(torch.int64) if x.dtype == torch.float64 else x
    opts = gpu.EventOpts(1, 0, 0.0, 0, 0.0, 0.0)
    with gpu.Context(flux_point=1, breakup_mode=1, use_polarized=pol, proc_id=13, nm=nm, ny=ny, nz=nz) as c:
        c.photon_pt_tables(c.info.g1)
        whole = c.sample_events(**t, n=n, seed=9)
        p, pdg, ok = c.generate_pairs(**t, n=n, seed=9, opts=opts)
        drawn = ok != 0  # an event without a bin leaves its momenta unwritten
        for off in range(0, n - PART + 1, (n - PART) // 25):
            at = slice(off, off + PART)
            for a, b in zip(c.sample_events(**t, n=PART, seed=9, offset=off), whole):
                assert torch.equal(bits(a), bits(b[at]))
            q, qdg, qok = c.generate_pairs(**t, n=PART, seed=9, offset=off, opts=opts)
            d = drawn[at]
            assert torch.equal(qok, ok[at])
            assert torch.equal(bits(q)[d], bits(p[at])[d])
            assert torch.equal(qdg[d], pdg[at][d])
