"""Amplitudes and residuals through device arrays: one kernel for both parts (and tau) against
the host path; results are the same bits."""
import ctypes

import numpy as np
import pytest

from spinorb_ccsd import mpqc_blocks, random_hamiltonian

pytestmark = pytest.mark.gpu


# one orbital of a kind; odd o (single loads); even o with arrays aligned to 16 bytes (pairs) and
# 8 bytes beyond that; more elements than one pass of the grid (o^2 v^2 > 2^22)
@pytest.mark.parametrize("no,nv,offset", [(1, 1, 0), (1, 6, 0), (3, 7, 0), (4, 9, 0), (4, 9, 1), (12, 180, 0)])
def test_device_arrays_match_host(no, nv, offset):
    import torch
    from mpqc_amd import _lib
    from mpqc_amd.ccsd import CCSD, Integrals
    rng = np.random.default_rng(no + nv)
    t1, t2 = rng.normal(0, 0.02, (nv, no)), rng.normal(0, 0.02, (nv, nv, no, no))

    def device(x):
        buf = torch.zeros(x.size + 2, dtype=torch.float64, device="cuda")
        buf[offset:offset + x.size] = torch.from_numpy(x.ravel())
        return buf, buf[offset:offset + x.size]

    def ptr(t):
        return ctypes.cast(t.data_ptr(), ctypes.POINTER(ctypes.c_double))

    (b1, d1), (b2, d2) = device(t1), device(t2)
    (o1, e1), (o2, e2) = device(np.zeros_like(t1)), device(np.zeros_like(t2))
    torch.cuda.synchronize()
    small = no * nv < 100
    with CCSD(no, nv) as c:
        if small:
            f, g = random_hamiltonian(no, nv, seed=no + nv, eri_scale=0.03)
            c.set_integrals(Integrals(**mpqc_blocks(f, g, no)))
            want = c.compute_residuals(t1, t2)  # host arrays
        c._check(c.lib.mpqc_ccsd_set_amplitudes(c.ctx, ptr(d1), ptr(d2), _lib.LAYOUT_DENSE, _lib.MEM_DEVICE))
        got = c.get_amplitudes()
        assert np.array_equal(got[0], t1) and np.array_equal(got[1], t2)
        c._check(c.lib.mpqc_ccsd_get_amplitudes(c.ctx, ptr(e1), ptr(e2), _lib.LAYOUT_DENSE, _lib.MEM_DEVICE))
        assert torch.equal(e1, d1) and torch.equal(e2, d2)
        for o, b in ((o1, b1), (o2, b2)):  # nothing written around the arrays
            assert torch.equal(o, b)
        if small:
            c.residual()  # on the tau that the device path built
            c._check(c.lib.mpqc_ccsd_get_residuals(c.ctx, ptr(e1), ptr(e2), _lib.LAYOUT_DENSE, _lib.MEM_DEVICE))
            assert np.array_equal(e1.cpu().numpy().reshape(want[0].shape), want[0])
            assert np.array_equal(e2.cpu().numpy().reshape(want[1].shape), want[1])


def test_one_part_alone():
    """One part of the pair asked for."""
    import torch
    from mpqc_amd import _lib
    from mpqc_amd.ccsd import CCSD
    no, nv = 2, 5
    rng = np.random.default_rng(1)
    t1, t2 = rng.normal(0, 1, (nv, no)), rng.normal(0, 1, (nv, nv, no, no))
    null = ctypes.POINTER(ctypes.c_double)()
    out = torch.zeros(t2.size, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    with CCSD(no, nv) as c:
        c._check(c.lib.mpqc_ccsd_set_amplitudes(c.ctx, *(x.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
                                                          for x in (t1, t2)), _lib.LAYOUT_DENSE, _lib.MEM_HOST))
        p = ctypes.cast(out.data_ptr(), ctypes.POINTER(ctypes.c_double))
        c._check(c.lib.mpqc_ccsd_get_amplitudes(c.ctx, null, p, _lib.LAYOUT_DENSE, _lib.MEM_DEVICE))
    assert np.array_equal(out.cpu().numpy().reshape(t2.shape), t2)
