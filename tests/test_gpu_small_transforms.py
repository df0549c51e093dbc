"""Short power-of-two transforms (4 elements per thread): every length that
takes them, both precisions, and the operator table shared between plans of
the two layouts. Tolerances (relative L2): FP64 1e-13 (a few tens of roundings
per value, ~1e-15), FP32 1e-6 (5e-7 for twice 20 butterfly levels at half an
ulp each, random signs)."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hc():
    import aspher_amd
    return aspher_amd


@pytest.mark.parametrize("backend,Ns", [("fft", 16), ("fft", 32), ("fft", 64), ("fft", 128),
                                        ("fft", 256), ("fft", 512), ("periodic", 32),
                                        ("periodic", 64), ("periodic", 128), ("periodic", 256),
                                        ("periodic", 512), ("periodic", 1024)])
def test_responses(hc, backend, Ns):
    from aspher_amd.device import DeviceArray
    s = hc.ContactSolver(Ns, domain_size=0.8, E_star=1.9, backend=backend)
    op = (O.FreeSpaceOperator if backend == "fft" else O.PeriodicOperator)(Ns, 0.8, 1.9)
    x = np.random.default_rng(Ns).uniform(-0.5, 1, Ns * Ns)
    ref = op.matvec(x)
    assert np.linalg.norm(s.matvec(x) - ref) < 1e-13 * np.linalg.norm(ref)
    xd = DeviceArray.from_numpy(x.astype(np.float32))
    s.matvec_device(xd.ptr, xd.ptr, 32)
    assert np.linalg.norm(xd.numpy().astype(np.float64) - ref) < 1e-6 * np.linalg.norm(ref)


def test_operator_shared_by_plans_of_both_layouts(hc):
    """Eight 256^2 instances transform their columns in 16 elements per thread,
    a single solver in 4: the cached operator serves both."""
    Ns, n = 256, 8
    x = np.random.default_rng(2).uniform(0, 1, Ns * Ns)
    ref = O.FreeSpaceOperator(Ns).matvec(x)
    s = hc.ContactSolver(Ns, backend="fft", shared_operator=True)
    first = s.matvec(x)
    gaps = [hc.surfaces.rough_gap(Ns, seed=i) for i in range(n)]
    rs, _ = hc.solve_ensemble([dict(backend="fft", grid_size=Ns, gap=g, p_nominal=0.01)
                               for g in gaps], tol=1e-9, precision="double")
    assert all(r.status == "converged" for r in rs)
    d = O.diagnose(O.FreeSpaceOperator(Ns).matvec, gaps[3], rs[3].pressure.ravel(),
                   0.01 * Ns * Ns, np.ptp(gaps[3]))
    assert d["fw_error"] <= 1.01e-9 and d["penetration"] <= 1.01e-9
    again = s.matvec(x)
    assert np.array_equal(first, again)
    assert np.linalg.norm(again - ref) < 1e-13 * np.linalg.norm(ref)


@pytest.mark.parametrize("backend,Ns,precond", [
    ("fft", 16, "none"), ("fft", 64, "fourier"), ("fft", 256, "none"), ("fft", 512, "fourier-fft"),
    ("periodic", 32, "fourier"), ("periodic", 512, "fourier"), ("periodic", 1024, "fourier-fft")])
def test_solves_with_folded_passes(hc, backend, Ns, precond):
    """Solves whose passes finish each other's reductions (up to 512 partial
    rows: 512^2 has 256, the 1024^2 response 512) and whose evaluation and line
    search are folded into the response. The certificate is the oracle's."""
    op = (O.FreeSpaceOperator if backend == "fft" else O.PeriodicOperator)(Ns)
    g0 = hc.surfaces.rough_gap(Ns, k_high=min(64, Ns // 4), seed=Ns)
    r = hc.ContactSolver(Ns, backend=backend).solve(g0, 0.01, tol=1e-9, precond=precond)
    assert r.status == "converged"
    d = O.diagnose(op.matvec, g0, r.pressure.ravel(), 0.01 * Ns * Ns, np.ptp(g0))
    assert d["fw_error"] <= 1.01e-9 and d["penetration"] <= 1.01e-9


@pytest.mark.parametrize("Ns", [16, 32, 64, 128, 256, 512])
def test_two_component_columns(hc, Ns):
    """Column transforms of 32 .. 1024 in 16 elements per thread, forward and
    inverse: last stages of radix 2, 4, 8 and 16."""
    from aspher_amd import tangential
    q = np.random.default_rng(Ns).uniform(-1, 1, 2 * Ns * Ns)
    u = tangential.TangentialFFTOperator(Ns, 0.7, 1.6, 0.3).matvec(q)
    ref = O.TangentialOperator(Ns, 0.7, 1.6, 0.3).matvec(q)
    assert np.linalg.norm(u - ref) < 1e-13 * np.linalg.norm(ref)
