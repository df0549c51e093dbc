"""Rounding error of the responses on sides that are not a power of two: no
larger than that of direct DFT passes of every prime factor with one correctly
rounded twiddle table, which these transforms replaced.

FP32, against the FP64 response of the same library: the bounds are the errors
of those passes (relative L2, mean over fields of the same distribution). FP64: a
constant field has only the frequency that a torus operator drops, and every
DFT of equal inputs leaves exact zeros in the others, so its response is 0."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Ns,bound", [(27, 1.44e-7), (81, 1.72e-7), (143, 2.41e-7),
                                      (243, 2.07e-7), (405, 2.25e-7), (625, 2.54e-7),
                                      # prime factors above 13
                                      (17, 1.73e-7), (34, 1.89e-7), (51, 1.99e-7),
                                      (62, 2.58e-7), (136, 2.30e-7), (323, 3.16e-7),
                                      (340, 2.67e-7), (510, 2.81e-7), (820, 4.10e-7),
                                      (1020, 3.67e-7), (1180, 4.91e-7)])
def test_fp32_response(Ns, bound):
    import aspher_amd
    from aspher_amd.device import DeviceArray
    s = aspher_amd.ContactSolver(Ns, backend="periodic")
    err = []
    for seed in range(40 if Ns < 100 else 10 if Ns < 700 else 3):
        # the pressure of a partial contact
        x = np.random.default_rng(seed).standard_normal(Ns * Ns) - 0.8
        x = np.maximum(x, 0.0).astype(np.float32)
        ref = s.matvec(x.astype(np.float64))
        xd = DeviceArray.from_numpy(x)
        s.matvec_device(xd.ptr, xd.ptr, 32)
        err.append(np.linalg.norm(xd.numpy() - ref) / np.linalg.norm(ref))
    assert np.mean(err) <= bound


@pytest.mark.parametrize("Ns,former", [(17, 3.33e-16), (34, 3.60e-16), (51, 3.67e-16),
                                       (136, 4.54e-16), (340, 5.21e-16), (510, 5.35e-16),
                                       # the smallest power of two, in 4 x 4 x 2
                                       # points where it was 16 x 2
                                       (32, 2.90e-16)])
def test_fp64_response(Ns, former):
    """Against 80-bit sums; 1.1 times the former passes' error (the mean of a few
    fields moves by a few percent)."""
    import aspher_amd
    import scipy.fft
    ld = np.longdouble
    k = np.arange(Ns)
    my = np.where(k < (Ns + 1) // 2, k, k - Ns).astype(ld)
    m2 = k[:Ns // 2 + 1].astype(ld)[None] ** 2 + my[:, None] ** 2
    m2[0, 0] = 1
    W = 1 / (np.arccos(ld(-1)) * np.sqrt(m2))
    W[0, 0] = 0
    s = aspher_amd.ContactSolver(Ns, backend="periodic")
    err = []
    for seed in range(40 if Ns < 100 else 8):
        x = np.maximum(np.random.default_rng(seed).standard_normal((Ns, Ns)) - 0.8, 0)
        ref = scipy.fft.irfft2(scipy.fft.rfft2(x.astype(ld)) * W, s=(Ns, Ns))
        d = s.matvec(x.ravel()).reshape(Ns, Ns) - ref
        err.append(float(np.sqrt((d ** 2).sum() / (ref ** 2).sum())))
    assert np.mean(err) <= 1.1 * former


# one, two and three prime passes, the largest and the first chirp prime of each
# precision (67, 71, 97, 101), one row and column and many per workgroup
@pytest.mark.parametrize("Ns", [17, 19, 34, 58, 67, 71, 94, 97, 101, 194, 202, 289, 323, 391, 646,
                                1122, 1156, 2346, 4913])
def test_prime_factors(Ns):
    """Against the oracle: FP64 1e-13, FP32 2e-6 as for every such side."""
    import aspher_amd
    from aspher_amd.device import DeviceArray
    from oracle import oracle as O
    s = aspher_amd.ContactSolver(Ns, domain_size=1.3, E_star=0.7, backend="periodic")
    x = np.random.default_rng(Ns).uniform(-0.5, 1, Ns * Ns)
    ref = O.PeriodicOperator(Ns, 1.3, 0.7).matvec(x)
    assert np.linalg.norm(s.matvec(x) - ref) < 1e-13 * np.linalg.norm(ref)
    xd = DeviceArray.from_numpy(x.astype(np.float32))
    s.matvec_device(xd.ptr, xd.ptr, 32)
    assert np.linalg.norm(xd.numpy().astype(np.float64) - ref) < 2e-6 * np.linalg.norm(ref)


@pytest.mark.parametrize("Ns", [17, 34, 51, 97, 289, 323])
def test_fourier_preconditioner_of_prime_factors(Ns):
    """Masked rows and their sums: FP64 1e-12, FP32 1e-5 as for every such side."""
    import ctypes as C
    from aspher_amd._capi import check, dptr, lib
    from oracle import oracle as O
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


@pytest.mark.parametrize("Ns", [27, 45, 100, 135, 143, 243, 343, 500, 625, 1210])
def test_fp64_response_to_a_constant(Ns):
    import aspher_amd
    u = aspher_amd.ContactSolver(Ns, backend="periodic").matvec(np.full(Ns * Ns, 0.7))
    assert np.all(u == 0.0)
