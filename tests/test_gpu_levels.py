"""Small FP64 residuals by levels of independent ops (option "levels") against the oracle and
against one launch per op, whose kernels the small sizes would not reach otherwise."""
import numpy as np
import pytest

from oracle import ccsd as O
from spinorb_ccsd import mpqc_blocks, random_hamiltonian

pytestmark = pytest.mark.gpu


def _problem(no, nv, symmetric=True):
    f, g = random_hamiltonian(no, nv, seed=no * 100 + nv, eri_scale=0.03)
    b = mpqc_blocks(f, g, no)
    rng = np.random.default_rng(no + nv)
    if not symmetric:
        for k in ("Giabc", "Gabcd", "Gijab", "Fia"):
            b[k] = b[k] + rng.normal(0, 0.01, b[k].shape)
    t1 = rng.normal(0, 0.02, (nv, no))
    t2 = rng.normal(0, 0.02, (nv, nv, no, no))
    return f, b, t1, t2


def _oracle(b, t1, t2, fov_sign=1.0):
    ints = O.Integrals(**b)
    tau = O.make_tau(t1, t2)
    return O.cs_ccsd_r1(t1, t2, tau, ints), O.cs_ccsd_r2(t1, t2, tau, ints, fov_sign)


# one orbital of a kind; odd sizes; tiles of transposes (v o >= 1024); split sums of up to 16
# and more partials (K = o v^2); contractions launched by themselves; the pair-symmetric
# ladder (o^2 v^4 >= 3e8) with and without symmetric integrals; the last size below the limit
@pytest.mark.parametrize("no,nv,symmetric", [(1, 1, True), (1, 9, True), (7, 1, True), (3, 17, True), (6, 33, True),
                                             (9, 45, True), (9, 45, False), (12, 85, True)])
def test_levels_match_oracle_and_single_launches(no, nv, symmetric):
    from mpqc_amd.ccsd import CCSD, Integrals
    f, b, t1, t2 = _problem(no, nv, symmetric)
    ref = _oracle(b, t1, t2)
    got = {}
    with CCSD(no, nv) as c:
        c.set_integrals(Integrals(**b))
        for levels in (1, 0):
            c.set_option("levels", levels)
            runs = [c.compute_residuals(t1, t2) for _ in range(4)]  # eager, captured, replayed
            for r in runs[1:]:
                assert np.array_equal(r[0], runs[0][0]) and np.array_equal(r[1], runs[0][1])
            got[levels] = runs[0] + c.get_dressed_fock()
    # FP64 sums of at most o v^2 + v^2 products in another order: 1e-12 of the largest element, as the parity tests
    for levels, (r1, r2, _, _) in got.items():
        assert np.abs(r1 - ref[0]).max() <= 1e-12 * max(np.abs(ref[0]).max(), 1e-3), levels
        assert np.abs(r2 - ref[1]).max() <= 1e-12 * max(np.abs(ref[1]).max(), 1e-3), levels
    for x, y in zip(got[1][2:], got[0][2:]):
        assert np.abs(x - y).max() <= 1e-12 * max(np.abs(y).max(), 1.0)


def test_levels_replan_on_new_integrals_and_options():
    """New integrals, new amplitudes and an option change on one context."""
    from mpqc_amd.ccsd import CCSD, Integrals
    no, nv = 4, 21
    _, b, t1, t2 = _problem(no, nv)
    _, b2, u1, u2 = _problem(no, nv, symmetric=False)
    with CCSD(no, nv) as c:
        for blocks, a1, a2, sign in ((b, t1, t2, 1.0), (b, u1, u2, 1.0), (b2, u1, u2, 1.0), (b2, u1, u2, -1.0)):
            c.set_integrals(Integrals(**blocks))
            c.set_option("fov_sign", sign)
            ref = _oracle(blocks, a1, a2, sign)
            for _ in range(3):
                r = c.compute_residuals(a1, a2)
                assert np.abs(r[0] - ref[0]).max() <= 1e-12 * np.abs(ref[0]).max()
                assert np.abs(r[1] - ref[1]).max() <= 1e-12 * np.abs(ref[1]).max()


# o^4 up to 2^23 and beyond it, where every op has a launch of its own with the option on too
@pytest.mark.parametrize("no,nv,by_levels", [(53, 3, True), (54, 3, False)])
def test_many_occupied_orbitals(no, nv, by_levels):
    from mpqc_amd.ccsd import CCSD, Integrals
    _, b, t1, t2 = _problem(no, nv)
    ref = _oracle(b, t1, t2)
    got = []
    with CCSD(no, nv) as c:
        c.set_integrals(Integrals(**b))
        for levels in (1, 0):
            c.set_option("levels", levels)
            got.append(c.compute_residuals(t1, t2))
    for r1, r2 in got:
        assert np.abs(r1 - ref[0]).max() <= 1e-12 * max(np.abs(ref[0]).max(), 1e-3)
        assert np.abs(r2 - ref[1]).max() <= 1e-12 * max(np.abs(ref[1]).max(), 1e-3)
    assert np.array_equal(got[0][1], got[1][1]) != by_levels
