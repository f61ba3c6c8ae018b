"""A z table of more than 2^30 bins (8.6 GB): positions in it need more than 31
bits where two are added.  A uniform table draws z = zmin + r (zmax - zmin),
which is what one bin draws from the same seed; rounding of the table's entries
moves a draw by less than a bin."""
import pytest

pytestmark = pytest.mark.gpu

NZ = (1 << 30) + 5


def test_draws_from_a_long_z_table(gpu):
    import torch
    f64 = dict(dtype=torch.float64, device="cuda")
    n = 5000
    sum_ym = torch.tensor([[0.0, 1.0]], **f64)
    long = torch.arange(NZ + 1, **f64).div_(NZ).reshape(1, -1)
    short = torch.tensor([[0.0, 1.0]], **f64)
    kw = dict(flux_point=1, breakup_mode=1, proc_id=13, nm=1, ny=1)
    opts = gpu.EventOpts(0, 0, 0.0, 0, 0.0, 0.0)
    with gpu.Context(nz=1, **kw) as c:
        want = c.sample_events(sum_ym=sum_ym, sum_z=short, n=n, seed=4)
        pairs = c.generate_pairs(sum_ym=sum_ym, sum_z=short, n=n, seed=4, opts=opts)
    with gpu.Context(nz=NZ, **kw) as c:
        got = c.sample_events(sum_ym=sum_ym, sum_z=long, n=n, seed=4)
        pairs_long = c.generate_pairs(sum_ym=sum_ym, sum_z=long, n=n, seed=4, opts=opts)
    assert float(want[2].max() - want[2].min()) > 1.9  # both halves of the table
    for a, b in zip(got, want):
        assert float((a - b).abs().max()) <= 4.0 / NZ
    # cos(theta) moves by a bin, sin(theta) by the root of twice that near the ends (1e-4)
    assert bool((pairs_long[2] == 1).all()) and bool((pairs[2] == 1).all())
    scale = pairs[0].abs().amax(dim=(1, 2), keepdim=True)
    assert float(((pairs_long[0] - pairs[0]).abs() / scale).max()) <= 2e-4
