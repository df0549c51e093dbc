"""Free-space grids whose torus is a power of two wider than 2 Ns (the next
smooth even side from 2 Ns - 1 on): the register-blocked kernels on grids that
are not a power of two, odd ones among them. Tolerances (relative L2) are those
of the register-blocked transforms at power-of-two grids: FP64 1e-13 (a few tens
of roundings per value, ~1e-15), FP32 1e-6 (5e-7 for twice 20 butterfly levels
at half an ulp each, random signs)."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hc():
    import aspher_amd
    return aspher_amd


@pytest.mark.parametrize("Ns", [31, 127, 253, 254, 255, 508, 511, 1015, 1020, 1023, 2029, 2047])
def test_response(hc, Ns):
    from aspher_amd.device import DeviceArray
    s = hc.ContactSolver(Ns, domain_size=1.3, E_star=0.7, backend="fft")
    x = np.random.default_rng(Ns).uniform(-0.5, 1, Ns * Ns)
    ref = O.FreeSpaceOperator(Ns, 1.3, 0.7).matvec(x)
    assert np.linalg.norm(s.matvec(x) - ref) < 1e-13 * np.linalg.norm(ref)
    xd = DeviceArray.from_numpy(x.astype(np.float32))
    s.matvec_device(xd.ptr, xd.ptr, 32)
    assert np.linalg.norm(xd.numpy().astype(np.float64) - ref) < 1e-6 * np.linalg.norm(ref)


@pytest.mark.parametrize("Ns,precond", [(31, "none"), (127, "fourier"), (254, "fourier-fft"),
                                        (255, "fourier"), (511, "none"), (511, "fourier")])
def test_solve(hc, Ns, precond):
    """Short rows: the passes folded into them move pairs of values, which an
    odd grid has no place for."""
    g0 = hc.surfaces.rough_gap(Ns, k_high=min(64, Ns // 4), seed=Ns)
    r = hc.ContactSolver(Ns, backend="fft").solve(g0, 0.01, tol=1e-9, precond=precond)
    assert r.status == "converged"
    d = O.diagnose(O.FreeSpaceOperator(Ns).matvec, g0, r.pressure.ravel(), 0.01 * Ns * Ns,
                   np.ptp(g0))
    assert d["fw_error"] <= 1.01e-9 and d["penetration"] <= 1.01e-9


def test_nested_solve_through_them(hc):
    """Levels 127 (odd), 254 and 508."""
    Ns = 508
    g0 = hc.surfaces.rough_gap(Ns, k_high=64, seed=1)
    r = hc.solve_nested(Ns, g0, 0.01, coarsest=127, backend="fft", tol=1e-9)
    assert r.status == "converged"
    d = O.diagnose(O.FreeSpaceOperator(Ns).matvec, g0, r.pressure.ravel(), 0.01 * Ns * Ns,
                   np.ptp(g0))
    assert d["fw_error"] <= 1.01e-9 and d["penetration"] <= 1.01e-9


@pytest.mark.parametrize("Ns", [100, 127, 254])
def test_matvec_without_allocation_takes_powers_of_two_only(hc, Ns):
    """Whatever torus a grid is embedded in."""
    import ctypes as C
    from aspher_amd import _capi
    from aspher_amd.device import DeviceArray
    s = hc.ContactSolver(Ns, backend="fft")
    xd = DeviceArray.from_numpy(np.zeros(Ns * Ns))
    s.matvec_device(xd.ptr, xd.ptr, 64)
    rc = _capi.lib().aspher_solver_matvec_device_noalloc(s._h, C.c_void_p(xd.ptr),
                                                         C.c_void_p(xd.ptr), 64)
    assert rc == _capi.ERR_LOGIC
    assert b"power-of-two grids" in _capi.lib().aspher_last_error()
