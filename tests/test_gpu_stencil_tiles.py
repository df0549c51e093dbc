"""Stencil preconditioner on both sides of the tile rule (64 x 4 tiles up to
512^2, 64 x 16 above): one tile, two tiles per workgroup, odd sides read byte
by byte, overhanging last tiles, empty tiles. Tolerances (relative L2) of the
sums of at most 81 taps: FP64 1e-12 as for the other sizes, FP32 1e-5."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Ns,radius", [(5, 2), (61, 1), (68, 3), (509, 4), (512, 1), (512, 5),
                                       (513, 1), (516, 3), (520, 4), (577, 5)])
def test_stencil_tiles(Ns, radius):
    from aspher_amd._capi import check, dptr, lib
    rng = np.random.default_rng(Ns + radius)
    mask = rng.random((Ns, Ns)) < 0.5
    mask[Ns // 3:2 * Ns // 3] = False          # whole tiles without a contact point
    mask[0, 0] = mask[-1, -1] = True
    mask = mask.ravel()
    g = np.ascontiguousarray(rng.uniform(-1, 1, Ns * Ns))
    m = mask.astype(np.uint8)
    ref = O.StencilPreconditioner(Ns, radius)
    for bits, tol, dt in ((64, 1e-12, np.float64), (32, 1e-5, np.float32)):
        z = np.empty(Ns * Ns)
        check(lib().aspher_precond_apply(Ns, b"fourier", radius, bits, dptr(g),
                                         m.ctypes.data_as(C.POINTER(C.c_uint8)), dptr(z)))
        r = ref.apply(g.astype(dt), mask).astype(np.float64)
        assert np.all(z[~mask] == 0.0)
        assert np.linalg.norm(z - r) <= tol * np.linalg.norm(r), bits
