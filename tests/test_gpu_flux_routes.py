"""The form-factor flux integrals take one of several kernels by their number
(teams of 64, 16 or 8 lanes per integral, one lane per integral with rows
grouped by photon energy, or that with shared integrand factors).  Every route runs the same dqagse arithmetic, so a
point's luminosity must not depend on how many points were asked for with it:
1e-11 relative between routes (the integrand may differ by rounding, which
the contraction of these Pb-Pb points amplifies by less than 1e3), and 1e-9
against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CFG = dict(flux_point=0, breakup_mode=2, nm=3, ny=3)
NMAX = 1500  # 3000 rows: one lane per integral, last group of 64 rows partly filled


@pytest.fixture(scope="module")
def data(gpu):
    import torch
    rng = np.random.default_rng(77)
    M = np.exp(rng.uniform(np.log(2.0), np.log(60.0), NMAX))
    Y = rng.uniform(-3.5, 3.5, NMAX)
    c = gpu.Context(**CFG)
    t = lambda x: torch.as_tensor(x, device="cuda")
    L = c.lumi_points(t(M), t(Y)).cpu().numpy()
    return c, M, Y, L, c.info.qags_evals


# one point; row groups of 64 and their neighbours; both sides of every change of route
@pytest.mark.parametrize("n", [1, 14, 15, 31, 32, 33, 175, 176, 702, 703, 1499])
def test_route_does_not_change_a_point(gpu, data, n):
    import torch
    c, M, Y, L, _ = data
    t = lambda x: torch.as_tensor(x, device="cuda")
    got = c.lumi_points(t(M[:n]), t(Y[:n])).cpu().numpy()
    assert c.info.qags_bad == 0
    assert np.max(np.abs(got - L[:n]) / np.abs(L[:n])) <= 1e-11


def test_evaluation_counts_add_up(gpu, data):
    """Every QAGS decision is the same on every route: the integrand
    evaluations of the parts sum to those of the whole."""
    import torch
    c, M, Y, _, evals = data
    t = lambda x: torch.as_tensor(x, device="cuda")
    total = 0
    for a, b in ((0, 14), (14, 189), (189, 500), (500, 1500)):
        c.lumi_points(t(M[a:b].copy()), t(Y[a:b].copy()))
        total += c.info.qags_evals
    assert total == evals


# the fewest rows that share factors, one group and one row more, and more
# than one launch's groups (262,144 rows)
@pytest.mark.parametrize("n", [4096, 4129, 131105])
def test_shared_factors_do_not_change_a_point(gpu, data, n):
    import torch
    c = data[0]
    rng = np.random.default_rng(n)
    M = np.exp(rng.uniform(np.log(2.0), np.log(60.0), n))
    Y = rng.uniform(-3.5, 3.5, n)
    t = lambda x: torch.as_tensor(x, device="cuda")
    L = c.lumi_points(t(M), t(Y)).cpu().numpy()
    assert c.info.qags_bad == 0
    idx = rng.choice(n, 700, replace=False)
    one = c.lumi_points(t(M[idx]), t(Y[idx])).cpu().numpy()
    assert np.max(np.abs(L[idx] - one) / np.abs(one)) <= 1e-11


def test_shared_factors_evaluation_counts(gpu, data):
    import torch
    c = data[0]
    rng = np.random.default_rng(3)
    M = np.exp(rng.uniform(np.log(2.0), np.log(60.0), 6150))
    Y = rng.uniform(-3.5, 3.5, 6150)
    t = lambda x: torch.as_tensor(x, device="cuda")
    c.lumi_points(t(M), t(Y))  # 12,300 rows share factors, 2,460 do not
    whole, total = c.info.qags_evals, 0
    for a in range(0, 6150, 1230):
        c.lumi_points(t(M[a:a + 1230].copy()), t(Y[a:a + 1230].copy()))
        total += c.info.qags_evals
    assert total == whole


@pytest.mark.parametrize("cap", [9, 8, 3, 1])
def test_shared_factors_hand_integrals_on(gpu, data, cap):
    """Integrals that outgrow the lists (or a smaller cap) go to the
    1000-interval kernel: the same decisions and, to rounding, values."""
    import torch
    rng = np.random.default_rng(8)
    t = lambda x: torch.as_tensor(x, device="cuda")
    M, Y = t(np.exp(rng.uniform(np.log(2.0), np.log(60.0), 4100))), t(rng.uniform(-3.5, 3.5, 4100))
    with gpu.Context(**CFG) as c:
        L = c.lumi_points(M, Y).cpu().numpy()
        evals = c.info.qags_evals
        c.set_qags_cap(cap)
        got = c.lumi_points(M, Y).cpu().numpy()
        assert c.info.qags_evals == evals
        assert np.max(np.abs(got - L) / np.abs(L)) <= 1e-11


def test_points_against_oracle(data, oracle_ctx):
    _, M, Y, L, _ = data
    o = oracle_ctx(**CFG)
    for i in (0, 1, 700, NMAX - 1):
        assert abs(L[i] / o.lumi(M[i], Y[i]) - 1) <= 1e-9


@pytest.mark.parametrize("n", [1, 2048, 2049, 24576, 24577, 98304, 98305])
def test_flux_form_routes(gpu, data, n):
    """Bit for bit: the per-point routes evaluate every node alike."""
    import torch
    c = data[0]
    rng = np.random.default_rng(5)
    b = torch.as_tensor(rng.uniform(0.3, 16.0, 98305), device="cuda")
    k = torch.as_tensor(10 ** rng.uniform(-2.0, 2.5, 98305), device="cuda")
    full, ier = c.flux_form(b, k)
    got, ier_n = c.flux_form(b[:n].clone(), k[:n].clone())
    assert torch.equal(got.view(torch.int64), full[:n].view(torch.int64))
    assert torch.equal(ier_n, ier[:n])
