"""The flattened local energy (k_el_prep / k_el_kinetic / k_el_points) against the oracle where its tiles end:
walker counts around the groups of four walkers and 64 electrons, meshes that fill a wave differently, every
orbital form (up to 16, 32, 48, 64 and more MOs, different MOs per spin, AO orbitals), f shells; Cartesian closed
shells (the other forms: test_gpu_forms.py).  Tolerance: 1e-9 of 1 + |T| + |V| (the parts cancel in e_L; G^-1 of these small
random wavefunctions loses at most a few digits)."""

import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _with_mos(system, n_up, same):
    """The system's Hamiltonian with n_up MOs per spin (dn MOs differ unless same), full pairing matrix."""
    from jqmc_amd.determinant import Geminal_data
    from jqmc_amd.molecular_orbital import MOs_data

    ham = system.hamiltonian_data
    gem = ham.wavefunction_data.geminal_data
    rng = np.random.default_rng(5)
    aos = gem.aos_data
    C = [rng.standard_normal((n_up, aos.num_ao)) / np.sqrt(aos.num_ao) for _ in range(2)]
    up = MOs_data(num_mo=n_up, aos_data=aos, mo_coefficients=C[0])
    dn = up if same else MOs_data(num_mo=n_up, aos_data=aos, mo_coefficients=C[1])
    lam = np.hstack([np.eye(n_up) + 0.2 * rng.standard_normal((n_up, n_up)),
                     rng.standard_normal((n_up, gem.num_electron_up - gem.num_electron_dn))])
    g = Geminal_data(gem.num_electron_up, gem.num_electron_dn, up, dn, lam)
    wf = dataclasses.replace(ham.wavefunction_data, geminal_data=g)
    return dataclasses.replace(ham, wavefunction_data=wf)


CASES = [("water_ae", None, 6, 1), ("water_ae", None, 6, 13), ("chain10", None, 4, 9), ("chain10", None, 18, 7),
         ("benzene_ecp", None, 12, 5), ("chain56", None, 6, 3), ("chain96", None, 6, 2), ("water4_ecp", None, 12, 3),
         ("water4_jagp", None, 6, 2), ("chain30", (20, True), 6, 3), ("chain30", (17, False), 12, 3),
         ("chain30", (50, False), 6, 2), ("chain30", (60, True), 6, 3), ("chain30", (70, True), 6, 3),
         ("chain30", (66, False), 4, 2)]


@pytest.mark.parametrize("name,mos,nv,W", CASES)
def test_local_energy_matches_oracle(name, mos, nv, W):
    import torch

    from jqmc_amd import synthetic
    from jqmc_amd._api import WalkerState
    from jqmc_amd._pack import SystemPack
    from oracle import coulomb as oc
    from oracle import wf as owf

    if name.startswith("chain"):
        system = synthetic.chain_ecp(int(name[5:]), 1)
    elif name == "water4_jagp":
        system = synthetic.water4_ecp(0, jagp=True)
    else:
        system = synthetic.WORKLOADS[name](0)
    ham = system.hamiltonian_data if mos is None else _with_mos(system, mos[0], mos[1])
    r_up, r_dn = system.initial_walkers(W, seed=11)
    ws = WalkerState(SystemPack(ham, Nv=nv), W).init(r_up, r_dn)
    RT = ws.rotations(3, 0)
    e, kin, pot, tel = ws.local_energy(RT, with_parts=True)
    assert torch.isfinite(e).all()
    assert ((tel.sum(1) - kin).abs() <= 1e-11 * tel.abs().sum(1)).all()
    for w in sorted({0, W - 1}):
        G = owf.geminal(ham.wavefunction_data.geminal_data, r_up[w], r_dn[w])
        Gi = owf.geminal_inverse(G)
        tu, td = owf.kinetic_all_elements_fast(ham.wavefunction_data, r_up[w], r_dn[w], Gi)
        T = float(np.sum(tu) + np.sum(td))
        V = oc.coulomb_potential_fast(ham.coulomb_potential_data, ham.wavefunction_data, r_up[w], r_dn[w],
                                      RT[w].cpu().numpy(), Gi, 1, nv)
        tol = 1e-9 * (1.0 + abs(T) + abs(V))
        assert abs(float(kin[w]) - T) <= tol, (w, float(kin[w]), T)
        assert abs(float(pot[w]) - V) <= tol, (w, float(pot[w]), V)


@pytest.mark.parametrize("name,mos,nv,W", [("water_ae", None, 6, 3), ("chain10", None, 6, 11), ("chain56", None, 6, 2),
                                           ("chain30", (70, True), 6, 2)])
def test_lattice_elements_match_oracle(name, mos, nv, W):
    from jqmc_amd import synthetic
    from jqmc_amd._api import WalkerState
    from jqmc_amd._pack import SystemPack
    from oracle import gfmc as og
    from oracle import wf as owf

    system = synthetic.chain_ecp(int(name[5:]), 1) if name.startswith("chain") else synthetic.WORKLOADS[name](0)
    ham = system.hamiltonian_data if mos is None else _with_mos(system, mos[0], mos[1])
    r_up, r_dn = system.initial_walkers(W, seed=12)
    ws = WalkerState(SystemPack(ham, Nv=nv), W).init(r_up, r_dn)
    RT = ws.rotations(4, 0)
    for move in ("tmove", "dltmove") if ham.coulomb_potential_data.ecp_flag else ("tmove",):
        Vd, Vn = ws.lrdmc_local_energy(WalkerState.lrdmc_params(0.25, non_local_move=move), RT)
        w = W - 1
        Gi = owf.geminal_inverse(owf.geminal(ham.wavefunction_data.geminal_data, r_up[w], r_dn[w]))
        d, n, _, _ = og.hamiltonian_elements(ham, r_up[w], r_dn[w], Gi, RT[w].cpu().numpy(), 0.25, move, Nv=nv)
        tol = 1e-9 * (1.0 + abs(d) + abs(n))
        assert abs(float(Vd[w]) - d) <= tol and abs(float(Vn[w]) - n) <= tol, (move, float(Vd[w]), d, float(Vn[w]), n)


def test_batch_companions_change_no_bit():
    """A system of 50 orbitals (four waves per block of the kinetic kernel) has the same bits alone and in one call
    with a system of 60 orbitals (two waves) of the same orbital class, and with one of another class."""
    import torch

    from jqmc_amd import synthetic
    from jqmc_amd._api import WalkerState, lrdmc_projection_multi
    from jqmc_amd._pack import SystemPack

    base = synthetic.chain_ecp(30, 1)
    packs = [SystemPack(_with_mos(base, n, True)) for n in (50, 60, 18)]
    prm = WalkerState.lrdmc_params(0.3, n_steps=2)

    def run(n_systems):
        states = []
        for k, W in zip(range(n_systems), (5, 3, 2)):
            states.append(WalkerState(packs[k], W).init(*base.initial_walkers(W, seed=21 + k)))
        outs = lrdmc_projection_multi(states, [prm] * n_systems, 17, [100] * n_systems)
        torch.cuda.synchronize()
        return states[0], outs[0]

    s1, o1 = run(1)
    for n in (2, 3):
        s, o = run(n)
        for key in ("V_diag", "V_nondiag", "w_L", "RT"):
            assert torch.equal(o[key], o1[key]), (n, key)
        for key in ("r_up", "r_dn", "Ginv", "jfield"):
            assert torch.equal(getattr(s, key), getattr(s1, key)), (n, key)


def test_more_walkers_than_a_row_of_blocks():
    """12 million walkers of H2: the grids of k_el_prep and k_dlnpsi_small go on along y.  Every walker has the bits
    that it has in a small set."""
    import torch

    from jqmc_amd import synthetic
    from jqmc_amd._api import WalkerState
    from jqmc_amd._pack import SystemPack

    st = synthetic._structure(["H", "H"], [[0.0, 0.0, 0.0], [0.0, 0.0, 1.4]])
    system = synthetic._assemble("h2", st, {"H": "1s"}, 1, use_j3=False)
    pack, n, rep = SystemPack(system.hamiltonian_data), 1000, 12000
    r_up, r_dn = (torch.as_tensor(r, device="cuda") for r in system.initial_walkers(n, seed=2))
    small = WalkerState(pack, n).init(r_up, r_dn)
    large = WalkerState(pack, n * rep).init(r_up.repeat(rep, 1, 1), r_dn.repeat(rep, 1, 1))
    assert torch.equal(large.local_energy().view(rep, n), small.local_energy().expand(rep, n))
    O, ref = large.dln_psi_dparams(), small.dln_psi_dparams()
    for k in ref:
        assert torch.equal(O[k].view(rep, n, -1), ref[k].view(1, n, -1).expand(rep, n, ref[k][0].numel())), k
