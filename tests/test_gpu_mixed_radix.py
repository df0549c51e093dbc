"""Grid sides that are not a power of two in [32, 8192]: mixed-radix and chirp
transforms against the oracle's scipy.fft operators.

Tolerances (relative L2). The transforms' own error, from the same passes run
on a host in the two precisions over every length up to 700 and the largest
ones, is at most 1.7e-15 and 3.6e-7 for a forward-inverse pair; an operator
takes one pair per direction, so 1e-13 and 2e-6 leave a margin of several.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hc():
    import aspher_amd
    return aspher_amd


def _check(hc, backend, Ns, L=1.3, E=0.7, fp32=True):
    s = hc.ContactSolver(Ns, domain_size=L, E_star=E, backend=backend)
    op = (O.FreeSpaceOperator if backend == "fft" else O.PeriodicOperator)(Ns, L, E)
    x = np.random.default_rng(Ns).uniform(-0.5, 1, Ns * Ns)
    ref = op.matvec(x)
    scale = np.linalg.norm(ref)
    assert np.linalg.norm(s.matvec(x) - ref) < 1e-13 * scale
    if fp32:
        from aspher_amd.device import DeviceArray
        xd = DeviceArray.from_numpy(x.astype(np.float32))
        s.matvec_device(xd.ptr, xd.ptr, 32)          # in place
        assert np.linalg.norm(xd.numpy().astype(np.float64) - ref) < 2e-6 * scale


# 2 Ns: every radix, one to five passes, a larger smooth side (17, 59, 331),
# one row and column, several rows per workgroup
@pytest.mark.parametrize("Ns", [1, 2, 3, 5, 7, 11, 13, 17, 33, 45, 59, 100, 129, 143, 150, 169,
                                240, 331, 625, 1000])
def test_free_space(hc, Ns):
    _check(hc, "fft", Ns)


# even and odd sides, direct and chirp (17, 31, 257, 501, 1009), powers of two
# below the register-blocked range
@pytest.mark.parametrize("Ns", [2, 3, 4, 5, 8, 9, 13, 15, 16, 17, 31, 34, 99, 121, 169, 257, 360,
                                501, 1009, 1215, 1500, 2018])
def test_periodic(hc, Ns):
    _check(hc, "periodic", Ns)


def test_largest_sides_and_refusals(hc):
    """The largest sides FP64 takes: free space 2559 (embedded in 5120) and a
    prime torus side whose chirp convolution fills the LDS."""
    _check(hc, "fft", 2559, fp32=False)
    _check(hc, "periodic", 5011, fp32=False)
    for backend, Ns in (("fft", 2560), ("periodic", 5120), ("periodic", 5121)):
        with pytest.raises(ValueError):
            hc.ContactSolver(Ns, backend=backend)


@pytest.mark.parametrize("Ns", [5, 12, 33, 100, 129, 257, 300])
def test_fourier_preconditioner(hc, Ns):
    """Masked input and output with the per-block sums, and the two-row packing
    of odd sides with a row left over."""
    import ctypes as C
    from aspher_amd._capi import check, dptr, lib
    rng = np.random.default_rng(Ns)
    mask = rng.random(Ns * Ns) < 0.4
    mask[:2] = True
    g = np.ascontiguousarray(rng.uniform(-1, 1, Ns * Ns))
    m = mask.astype(np.uint8)
    ref = O.FourierPreconditioner(Ns)
    for bits, tol, dt in ((64, 1e-12, np.float64), (32, 1e-5, np.float32)):
        z = np.empty(Ns * Ns)
        check(lib().aspher_precond_apply(Ns, b"fourier-fft", 2, bits, dptr(g),
                                         m.ctypes.data_as(C.POINTER(C.c_uint8)), dptr(z)))
        r = ref.apply(g.astype(dt), mask).astype(np.float64)
        assert np.linalg.norm(z - r) <= tol * np.linalg.norm(r), bits


def test_solve_odd_side(hc):
    """A certified solve on an odd torus: convolution, preconditioner and their
    reductions together."""
    Ns = 63
    g0 = hc.surfaces.rough_gap(Ns, k_high=16, seed=3)
    r = hc.ContactSolver(Ns, backend="periodic").solve(g0, 0.01, tol=1e-10, precond="fourier-fft")
    assert r.status == "converged"
    d = O.diagnose(O.PeriodicOperator(Ns).matvec, g0, r.pressure.ravel(), 0.01 * Ns * Ns,
                   np.ptp(g0))
    assert d["fw_error"] <= 1.01e-10 and d["penetration"] <= 1.01e-10
