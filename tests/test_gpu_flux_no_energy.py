"""Points without a photon energy (M = 0): their flux integrals are NaN and
count as failed, whatever rows they share a wavefront with.  Among points that
all have the same b grid, and among points at one (M, Y)."""
import pytest

pytestmark = pytest.mark.gpu

N = 4200  # 8,400 flux rows: shared integrand factors; parts of 350 take a team of lanes per integral


@pytest.mark.parametrize("base", [10.0, 300.0])
@pytest.mark.parametrize("zeros", [(7,), (0, 2100, 4199)])
def test_integrals_without_an_energy_fail(gpu, base, zeros):
    import torch
    M = torch.full((N,), base, dtype=torch.float64, device="cuda")
    Y = torch.zeros(N, dtype=torch.float64, device="cuda")
    M[list(zeros)] = 0.0
    with gpu.Context(flux_point=0, breakup_mode=2, nm=3, ny=3) as c:
        L = c.lumi_points(M, Y)
        bad, evals = c.info.qags_bad, c.info.qags_evals
        assert bool(torch.isnan(L[list(zeros)]).all()) and int(torch.isnan(L).sum()) == len(zeros)
        part_bad = part_evals = 0
        for a in range(0, N, 350):
            c.lumi_points(M[a:a + 350].clone(), Y[a:a + 350].clone())
            part_bad += c.info.qags_bad
            part_evals += c.info.qags_evals
        assert part_bad >= 2 * len(zeros)
        assert (bad, evals) == (part_bad, part_evals)
