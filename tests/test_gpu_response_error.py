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
                                      (243, 2.07e-7), (405, 2.25e-7), (625, 2.54e-7)])
def test_fp32_response(Ns, bound):
    fp32_response(Ns, bound)


def fp32_response(Ns, bound):
    import aspher_amd
    from aspher_amd.device import DeviceArray
    s = aspher_amd.ContactSolver(Ns, backend="periodic")
    err = []
    for seed in range(40 if Ns < 100 else 10):
        # the pressure of a partial contact
        x = np.random.default_rng(seed).standard_normal(Ns * Ns) - 0.8
        x = np.maximum(x, 0.0).astype(np.float32)
        ref = s.matvec(x.astype(np.float64))
        xd = DeviceArray.from_numpy(x)
        s.matvec_device(xd.ptr, xd.ptr, 32)
        err.append(np.linalg.norm(xd.numpy() - ref) / np.linalg.norm(ref))
    assert np.mean(err) <= bound


@pytest.mark.parametrize("Ns", [27, 45, 100, 135, 143, 243, 343, 500, 625, 1210])
def test_fp64_response_to_a_constant(Ns):
    import aspher_amd
    u = aspher_amd.ContactSolver(Ns, backend="periodic").matvec(np.full(Ns * Ns, 0.7))
    assert np.all(u == 0.0)
