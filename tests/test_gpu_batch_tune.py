"""The launch shapes a batch times run its integrals several times over: what it
reports afterwards is one pass.  One job's photon energy puts the first QK21 node
q0 of every integral between the form factor's last knot and Q2max (t = q0^2 +
(k / gamma)^2 = 2 - 1e-6), where an integral ends as failed."""
import math

import pytest

pytestmark = pytest.mark.gpu


def test_failure_counts_after_tuning(gpu):
    g = 5020.0 / (2.0 * 0.9382720813)
    q0 = 5.0 * (1.0 - 0.995657163025808080735527280689003)
    M = 2.0 * g * math.sqrt(2.0 - 1e-6 - q0 * q0)
    kw = dict(flux_point=0, breakup_mode=2)
    jobs = [gpu.Config.make(nm=1, ny=1, mmin=M, mmax=1.1 * M, ymin=0.0, ymax=1.0, **kw),
            gpu.Config.make(nm=21, ny=11, **kw)]
    b = gpu.Batch(jobs)
    b.run(graph=False)
    want = b.job_failures()
    assert want[0] > 0 and want[1] == 0 and b.stats().qags_bad == want[0]
    b.autotune()
    assert b.job_failures() == want and b.stats().qags_bad == want[0]
    b.close()
