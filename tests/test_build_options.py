"""Build options compile (CPU only)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


# the ends of its range and both sides of the entries that one store keeps in LDS
@pytest.mark.parametrize("cap", [2, 7, 8, 9, 16])
def test_qags_fast_cap(cap):
    from upcgen_amd import build as B
    runs = [subprocess.Popen([B.HIPCC] + B._hip_flags(src) + [f"-DUPC_QAGS_FAST_CAP={cap}", "-fsyntax-only", "-x", "hip",
                                                             os.path.join(B.CSRC, src)],
                             stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
            for src in ("upc_flux_lumi.hip", "upc_flux_rows.hip", "upc_batch.hip", "upc_noalloc.hip")]
    for r in runs:
        out = r.communicate()[0]
        assert r.returncode == 0, out
