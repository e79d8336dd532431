"""(T) on the GPU (mpqc_ccsd_triples; CCSD_T::compute_ccsd_t_straight,
ccsd_t.h:1127-1167) against the oracle (oracle/ccsd_t.py) at arbitrary
amplitudes, and the reference's golden (T) energy of the DF water.

Bar: 1e-12 relative to |E(T)| at FP64 (the sum runs in a different order).
"""
import numpy as np
import pytest

from oracle import ccsd as O
from oracle import ccsd_t as T
from spinorb_ccsd import mpqc_blocks, random_hamiltonian
from test_golden import FIX

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("no,nv,block_bytes", [(1, 4, 0), (2, 7, 0), (3, 6, 0), (5, 13, 0), (6, 20, 1 << 20)])
def test_triples_match_oracle_at_random_amplitudes(no, nv, block_bytes):
    from mpqc_amd.ccsd import CCSD, Integrals
    f, g = random_hamiltonian(no, nv, seed=no * 13 + nv, eri_scale=0.05)
    b = mpqc_blocks(f, g, no)
    rng = np.random.default_rng(no + 7 * nv)
    t1 = rng.normal(0, 0.05, (nv, no))
    t2 = rng.normal(0, 0.05, (nv, nv, no, no))   # no permutational symmetry assumed
    eo, ev = np.diag(f)[:no], np.diag(f)[no:]
    ref = T.ccsd_t_straight(t1, t2, b["Gijab"], b["Giabc"], b["Gijka"], eo, ev)
    print(f"o={no} v={nv} block_bytes={block_bytes}", flush=True)
    with CCSD(no, nv) as c:
        c.set_integrals(Integrals(**b))
        c.set_orbital_energies(eo, ev)
        if block_bytes:
            c.set_option("triples_block_bytes", block_bytes)
        c.set_amplitudes(t1, t2)
        et, sec = c.triples()
    print(f"  GPU {et:.15e} oracle {ref:.15e} ({sec * 1e3:.2f} ms)")
    if no == 1:  # two electrons: no triples (closed form E(T) = 0)
        assert abs(et) < 1e-16 and abs(ref) < 1e-16
    else:
        assert abs(et - ref) < 1e-12 * abs(ref)


def test_triples_of_converged_water_match_oracle():
    from mpqc_amd.ccsd import CCSD, Integrals
    from test_golden import _inputs
    case = FIX["cases"][1]  # cc-pVDZ, all electrons
    _, inp = _inputs(case)
    with CCSD(inp.o, inp.v) as c:
        c.set_integrals(Integrals(**inp.blocks))
        c.set_orbital_energies(inp.eps_occ, inp.eps_vir)
        c.compute_ccsd(target_precision=1e-11)
        t1, t2 = c.get_amplitudes()
        et, _ = c.triples()
    b = inp.blocks
    ref = T.ccsd_t_straight(t1, t2, b["Gijab"], b["Giabc"], b["Gijka"], inp.eps_occ, inp.eps_vir)
    print(f"H2O cc-pVDZ (T): GPU {et:.15e} oracle {ref:.15e}")
    assert abs(et - ref) < 1e-12 * abs(ref)


def test_gpu_df_triples_match_reference():
    """DF-CCSD then (T) with <ia|bc> built on the device from the factors."""
    from mpqc_amd.ccsd import CCSD
    from test_oracle_df import _df_inputs
    case = FIX["df_cases"][0]
    tcase = FIX["triples_cases"][0]
    _, inp = _df_inputs(case)
    with CCSD(inp.o, inp.v, occ_block_size=2, unocc_block_size=2) as c:
        c.set_df_basis(inp.naux)
        c.set_integrals(inp.df_blocks())
        c.set_orbital_energies(inp.base.eps_occ, inp.base.eps_vir)
        E = c.compute_ccsd(target_precision=case["precision"])
        et, _ = c.triples()
        giabc = c.get_integral("Giabc")
    print(f"GPU DF-CCSD {E:.15f}, (T) {et:.15e}; reference (T) {tcase['e_triples']:.15e}")
    assert np.abs(giabc - inp.base.blocks["Giabc"]).max() < 1e-13
    assert abs(et - tcase["e_triples"]) < 2e-12


@pytest.mark.parametrize("prec,tol", [("f16x3", 5e-8), ("bf16x3", 1e-6)])  # measured <= 5.6e-9 / 7.7e-8
def test_triples_split_precision_forms(prec, tol):
    """The W GEMMs on 16-bit planes: E(T) within the form's precision of the
    FP64 oracle (random amplitudes, several i blocks) and of FP64 at converged
    water amplitudes."""
    from mpqc_amd.ccsd import CCSD, Integrals
    from test_golden import _inputs
    no, nv = 6, 20
    f, g = random_hamiltonian(no, nv, seed=77, eri_scale=0.05)
    b = mpqc_blocks(f, g, no)
    rng = np.random.default_rng(78)
    t1 = rng.normal(0, 0.05, (nv, no))
    t2 = rng.normal(0, 0.05, (nv, nv, no, no))
    eo, ev = np.diag(f)[:no], np.diag(f)[no:]
    ref = T.ccsd_t_straight(t1, t2, b["Gijab"], b["Giabc"], b["Gijka"], eo, ev)
    with CCSD(no, nv, precision=prec) as c:
        c.set_integrals(Integrals(**b))
        c.set_orbital_energies(eo, ev)
        c.set_option("triples_block_bytes", 1 << 20)
        c.set_amplitudes(t1, t2)
        et, _ = c.triples()
    print(f"{prec} random: {et:.12e} oracle {ref:.12e} rel {abs(et - ref) / abs(ref):.2e}")
    assert abs(et - ref) < tol * abs(ref)
    case = FIX["cases"][1]
    _, inp = _inputs(case)
    with CCSD(inp.o, inp.v) as c:
        c.set_integrals(Integrals(**inp.blocks))
        c.set_orbital_energies(inp.eps_occ, inp.eps_vir)
        c.compute_ccsd(target_precision=1e-10)
        e64, _ = c.triples()
        c.set_option("precision", {"f16x3": 3, "bf16x3": 2}[prec])
        esp, _ = c.triples()
    print(f"{prec} water: {esp:.12e} f64 {e64:.12e} diff {esp - e64:.2e}")
    assert abs(esp - e64) < tol * abs(e64)


# tiles of the summed t3s: one column block, v on either side of a block's edge, wide tiles,
# two tiles of columns (v > 144), K = v + o short of, at and past a multiple of 16; blocks of a few
# triples with a shorter last one
@pytest.mark.parametrize("no,nv,block_bytes", [(3, 13, 0), (4, 16, 1 << 20), (3, 17, 0), (5, 31, 1 << 20), (2, 81, 0),
                                               (2, 145, 0)])
def test_triples_sums_at_tile_edges(no, nv, block_bytes):
    from mpqc_amd.ccsd import CCSD
    rng = np.random.default_rng(no + nv)
    naux = 6  # density-fitted blocks: <ia|bc> is built on the device, and no v^4 block is needed
    X = rng.normal(0, 0.1, (naux, no + nv, no + nv))
    X = 0.5 * (X + X.transpose(0, 2, 1))
    o, v = slice(0, no), slice(no, no + nv)
    eri = lambda p, q, r, s: np.einsum("Kpr,Kqs->pqrs", X[:, p, r], X[:, q, s])  # noqa: E731  <pq|rs>
    eo, ev = np.sort(rng.uniform(-1.5, -0.4, no)), np.sort(rng.uniform(0.3, 2.5, nv))
    b = {"Fia": np.zeros((no, nv)), "Fij": np.diag(eo), "Fab": np.diag(ev), "Gijab": eri(o, o, v, v),
         "Gijkl": eri(o, o, o, o), "Giajb": eri(o, v, o, v), "Gijka": eri(o, o, o, v),
         "Xai": X[:, v, o], "Xij": X[:, o, o], "Xab": X[:, v, v]}
    t1, t2 = rng.normal(0, 0.05, (nv, no)), rng.normal(0, 0.05, (nv, nv, no, no))
    ref = T.ccsd_t_straight(t1, t2, b["Gijab"], eri(o, v, v, v), b["Gijka"], eo, ev)
    with CCSD(no, nv) as c:
        c.set_df_basis(naux)
        c.set_integrals({k: np.ascontiguousarray(x) for k, x in b.items()})
        c.set_orbital_energies(eo, ev)
        if block_bytes:
            c.set_option("triples_block_bytes", block_bytes)
        c.set_amplitudes(t1, t2)
        et, _ = c.triples()
        again, _ = c.triples()
    assert et == again
    assert abs(et - ref) < 1e-12 * abs(ref)


# W of every ordering from 16-bit planes (v + o above the limit up to which the FP64 sums are the
# faster, K not a multiple of 8) against the FP64 sums; on the other side of that limit the sums
# themselves run
@pytest.mark.parametrize("prec,tol", [("f16x3", 5e-8), ("bf16x3", 1e-6)])  # as the split forms' test above
@pytest.mark.parametrize("no,nv,planes", [(2, 161, True), (21, 124, True), (21, 123, False), (21, 125, False), (2, 158, False)])
def test_triples_from_planes_of_a_large_k(no, nv, planes, prec, tol):
    from mpqc_amd.ccsd import CCSD
    naux = 6
    rng = np.random.default_rng(no + nv)
    X = rng.normal(0, 0.1, (naux, no + nv, no + nv))
    X = 0.5 * (X + X.transpose(0, 2, 1))
    o, v = slice(0, no), slice(no, no + nv)
    eri = lambda p, q, r, s: np.einsum("Kpr,Kqs->pqrs", X[:, p, r], X[:, q, s])  # noqa: E731  <pq|rs>
    eo, ev = np.sort(rng.uniform(-1.5, -0.4, no)), np.sort(rng.uniform(0.3, 2.5, nv))
    b = {"Fia": np.zeros((no, nv)), "Fij": np.diag(eo), "Fab": np.diag(ev), "Gijab": eri(o, o, v, v),
         "Gijkl": eri(o, o, o, o), "Giajb": eri(o, v, o, v), "Gijka": eri(o, o, o, v),
         "Xai": X[:, v, o], "Xij": X[:, o, o], "Xab": X[:, v, v]}
    t1, t2 = rng.normal(0, 0.05, (nv, no)), rng.normal(0, 0.05, (nv, nv, no, no))
    et = {}
    for p in ("f64", prec):
        with CCSD(no, nv, precision=p) as c:
            c.set_df_basis(naux)
            c.set_integrals({k: np.ascontiguousarray(x) for k, x in b.items()})
            c.set_orbital_energies(eo, ev)
            c.set_amplitudes(t1, t2)
            et[p], _ = c.triples()
    if planes:
        assert 0 < abs(et[prec] - et["f64"]) < tol * abs(et["f64"])
    else:
        assert et[prec] == et["f64"]


def test_triples_operands_in_parts():
    """Operands that are set up a few occupied orbitals at a time (o max(v, o)^2 v > 2^24): the energy
    against that from fp16 planes, and no more device memory than one A with K = v + o, its
    o v^3 temporary, six B, the six orderings of W for one i and a permuted Gijka."""
    import ctypes
    import torch
    from mpqc_amd import _lib as L
    from mpqc_amd.ccsd import CCSD
    no, nv, naux = 12, 160, 6
    gen = torch.Generator(device="cuda").manual_seed(3)
    new = lambda *s: torch.randn(s, dtype=torch.float64, device="cuda", generator=gen)  # noqa: E731
    X = 0.05 * new(naux, no + nv, no + nv)
    X = X + X.transpose(1, 2)
    o, v = slice(0, no), slice(no, no + nv)

    def eri(p, q, r, s):  # <pq|rs>
        A, B = X[:, p, r], X[:, q, s]
        g = A.reshape(naux, -1).T @ B.reshape(naux, -1)
        return g.reshape(A.shape[1], A.shape[2], B.shape[1], B.shape[2]).permute(0, 2, 1, 3).contiguous()

    rng = np.random.default_rng(4)
    eo, ev = np.sort(rng.uniform(-1.5, -0.4, no)), np.sort(rng.uniform(0.3, 2.5, nv))
    dev = lambda x: torch.from_numpy(x).cuda()  # noqa: E731
    blocks = {"Fia": dev(np.zeros((no, nv))), "Fij": dev(np.diag(eo)), "Fab": dev(np.diag(ev)),
              "Gijab": eri(o, o, v, v), "Gijkl": eri(o, o, o, o), "Giajb": eri(o, v, o, v),
              "Giabc": eri(o, v, v, v), "Gijka": eri(o, o, o, v), "Gabcd": eri(v, v, v, v)}
    t1, t2 = 0.05 * new(nv, no), 0.05 * new(nv, nv, no, no)
    torch.cuda.synchronize()
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    et = {}
    for prec in ("f64", "f16x3"):
        with CCSD(no, nv, precision=prec) as c:
            for name, t in blocks.items():
                c._check(c.lib.mpqc_ccsd_set_integral(c.ctx, L.INTEGRAL_IDS[name], p(t), L.LAYOUT_DENSE, L.MEM_DEVICE))
            c.set_orbital_energies(eo, ev)
            c.set_option("triples_block_bytes", 1 << 20)
            c.init_guess()  # derived integral layouts exist
            c._check(c.lib.mpqc_ccsd_set_amplitudes(c.ctx, p(t1), p(t2), L.LAYOUT_DENSE, L.MEM_DEVICE))
            before = torch.cuda.mem_get_info()[0]
            et[prec], _ = c.triples()
            if prec == "f64":  # (the context keeps up to 4 GiB of temporaries)
                used = before - torch.cuda.mem_get_info()[0]
                k, v3 = nv + no, nv ** 3
                most = no * nv * nv * k + no * v3 + 6 * no * no * nv * k + 6 * v3 + no * no * nv * nv
                print(f"scratch {used / 2**20:.0f} MiB of {most * 8 / 2**20:.0f}")
                assert used <= 8 * most
    assert 0 < abs(et["f16x3"] - et["f64"]) < 5e-8 * abs(et["f64"])  # as the split forms' test above
