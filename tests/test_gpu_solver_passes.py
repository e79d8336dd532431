"""The solver loop's fused passes (energy with the DIIS overlaps; Jacobi step with the
extrapolation and tau) against the step-by-step entry points, which keep them apart."""
import numpy as np
import pytest

from spinorb_ccsd import mpqc_blocks, random_hamiltonian

pytestmark = pytest.mark.gpu

E_TOL, T_TOL = 1e-10, 1e-9  # the lockstep bounds against the oracle


# histories of one vector, a short one that rolls over, and one never full; one orbital of a kind;
# odd o (scalar loads); even o below and above o^2 v^2 = 2^19 (two elements per load); fp16
# planes, whose extrapolation pass also forms the maxima
@pytest.mark.parametrize("no,nv,scale,n_diis,prec", [
    (1, 1, 0.02, 8, "f64"), (1, 7, 0.02, 1, "f64"), (5, 13, 0.02, 2, "f64"), (4, 18, 0.02, 16, "f64"),
    (5, 19, 0.02, 3, "f16x3"), (12, 60, 0.003, 3, "f64"), (12, 61, 0.003, 3, "f64")])
def test_solve_matches_single_steps(no, nv, scale, n_diis, prec):
    from mpqc_amd.ccsd import CCSD, Integrals
    f, g = random_hamiltonian(no, nv, seed=no + nv, eri_scale=scale)
    b = mpqc_blocks(f, g, no)
    with CCSD(no, nv, n_diis=n_diis, max_iter=60, precision=prec) as c:
        c.set_integrals(Integrals(**b))
        c.set_orbital_energies(np.diag(f)[:no], np.diag(f)[no:])
        E = c.compute_ccsd(target_precision=1e-9)
        rows = c.trace()
        t1, t2 = c.get_amplitudes()
    with CCSD(no, nv, n_diis=n_diis, max_iter=60, precision=prec) as c:
        c.set_integrals(Integrals(**b))
        c.set_orbital_energies(np.diag(f)[:no], np.diag(f)[no:])
        c.init_guess()
        for k in range(len(rows) + 1):  # the trace begins at the second energy
            e, err = c.energy_error()
            if k > 0:
                assert abs(e - rows[k - 1].energy) < E_TOL, k
                assert abs(err - rows[k - 1].error) < T_TOL, k
            if k < len(rows):
                c.update()
                c.residual()
        t1s, t2s = c.get_amplitudes()
    assert abs(E - e) < E_TOL
    assert np.abs(t1 - t1s).max() < T_TOL and np.abs(t2 - t2s).max() < T_TOL
