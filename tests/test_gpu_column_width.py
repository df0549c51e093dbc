"""Ensembles whose tuned FP64 column pass has transforms of 1024 points: the
widths tried up to eight columns are all powers of two."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("backend,Ns,count", [("fft", 512, 3), ("periodic", 1024, 2)])
def test_tuned_ensemble(backend, Ns, count):
    import aspher_amd as hc
    gaps = [hc.surfaces.rough_gap(Ns, seed=i) for i in range(count)]
    rs, _ = hc.solve_ensemble([dict(backend=backend, grid_size=Ns, gap=g, p_nominal=0.01)
                               for g in gaps], tol=1e-9, precision="double")
    op = (O.FreeSpaceOperator if backend == "fft" else O.PeriodicOperator)(Ns)
    for g, r in zip(gaps, rs):
        assert r.status == "converged"
        d = O.diagnose(op.matvec, g, r.pressure.ravel(), 0.01 * Ns * Ns, np.ptp(g))
        assert d["fw_error"] <= 1.01e-9 and d["penetration"] <= 1.01e-9
