"""Point sets whose flux rows are not spread evenly in photon energy, large enough
to share integrand factors: a dense cluster and distant points, so that groups of
neighbouring rows lie far apart.  A point's luminosity is that of a small call,
which takes a team of lanes per integral: 1e-11 relative (the integrand may
differ by rounding, which the contraction of these Pb-Pb points amplifies by less
than 1e3), and every QAGS decision is the same, so the evaluations add up."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _cluster(rng, n, width):
    """n points within `width` of (10 GeV, 0.5), and 40 anywhere."""
    M = np.concatenate([10.0 * np.exp(width * rng.uniform(-1, 1, n)), np.exp(rng.uniform(np.log(1.0), np.log(100.0), 40))])
    Y = np.concatenate([0.5 + width * rng.uniform(-1, 1, n), rng.uniform(-5.0, 5.0, 40)])
    return M, Y


@pytest.mark.parametrize("width", [0.0, 1e-4, 0.02])
def test_cluster_and_distant_points(gpu, width):
    import torch
    rng = np.random.default_rng(21)
    M, Y = _cluster(rng, 4700, width)
    p = rng.permutation(len(M))
    M, Y = (torch.as_tensor(v[p].copy(), device="cuda") for v in (M, Y))
    with gpu.Context(flux_point=0, breakup_mode=2, nm=3, ny=3) as c:
        L = c.lumi_points(M, Y)
        evals, total = c.info.qags_evals, 0
        assert c.info.qags_bad == 0
        for a in range(0, len(M), 600):
            one = c.lumi_points(M[a:a + 600].clone(), Y[a:a + 600].clone())
            total += c.info.qags_evals
            assert float((L[a:a + 600] / one - 1).abs().max()) <= 1e-11
        assert total == evals
