"""Every form of wavefunction through the flattened local energy, lattice elements, position derivatives and
parameter derivatives, against the oracle: open shells (unpaired orbitals, no dn electron at all), with and without
J3 for MO and AO orbitals, every pair of Jastrow functions at quadrature points, spherical shells, shells of more
than twelve AOs and of more than four primitives, meshes of more than 64 points; and the forms whose AOs go through
the general tables in the mixed (FP32) form.

Tolerances as in the tests of the same kernels on closed Cartesian shells: 1e-9 of 1 + |T| + |V| (lattice: of
1 + |V_diag| + |V_nondiag|; derivatives: of the largest element, at least 1); mixed form 2e-5 of the same scales."""

import dataclasses
import functools

import numpy as np
import pytest
import torch

from jqmc_amd import synthetic

pytestmark = pytest.mark.gpu


def _with_spins(system, n_up, n_dn, jagp=False):
    """The system with n_up / n_dn electrons, random MOs (two more than n_up) or AO orbitals and a full pairing
    matrix."""
    from jqmc_amd.determinant import Geminal_data
    from jqmc_amd.molecular_orbital import MOs_data

    ham = system.hamiltonian_data
    aos = ham.wavefunction_data.geminal_data.aos_data
    rng = np.random.default_rng(5)
    n = aos.num_ao if jagp else n_up + 2
    orb = aos if jagp else MOs_data(num_mo=n, aos_data=aos, mo_coefficients=synthetic.random_orthonormal_rows(rng, n, aos.num_ao))
    lam = np.hstack([np.eye(n) + 0.2 * rng.standard_normal((n, n)), rng.standard_normal((n, n_up - n_dn))])
    gem = Geminal_data(n_up, n_dn, orb, orb, lam)
    wf = dataclasses.replace(ham.wavefunction_data, geminal_data=gem)
    return dataclasses.replace(ham, wavefunction_data=wf)


def _cn(**kw):
    st = synthetic._structure(["C", "N"], [[0.0, 0.0, 0.0], [0.0, 0.0, 2.3]])
    return synthetic._assemble("cn", st, {"C": "3s2p1d", "N": "3s3p"}, 2, ecp_elements={"C": 2, "N": 2}, **kw)


def _shells(spec, n_prim=3, **kw):
    plain = synthetic.build_cart_basis
    synthetic.build_cart_basis = functools.partial(plain, n_prim=n_prim)
    try:
        st = synthetic._structure(["N", "H"], [[0.0, 0.0, 0.0], [0.0, 0.4, 1.9]])
        return synthetic._assemble("nh", st, {"N": spec, "H": "2s1p"}, 3, ecp_elements={"N": 2}, **kw).hamiltonian_data
    finally:
        synthetic.build_cart_basis = plain


def _spherical():
    from jqmc_amd.hamiltonians import Hamiltonian_data
    from test_golden_turborvb import build_case

    st, cp, wf, _, _, _ = build_case("test_comparison_with_TurboRVB_w_2b_3b_Jastrow_w_ecp")
    return Hamiltonian_data(st, cp, wf)


EE, PE, PP = ("exp", 1.2), ("pade", 0.9), ("pade", 1.1)
FORMS = {
    "doublet": lambda: _cn().hamiltonian_data,
    "doublet_jagp": lambda: _cn(jagp=True, lam_rank=8).hamiltonian_data,
    "septet": lambda: _with_spins(_cn(), 7, 1),
    "all_up": lambda: _with_spins(_cn(), 5, 0),
    "all_up_jagp": lambda: _with_spins(_cn(), 4, 0, jagp=True),
    "one_electron": lambda: _with_spins(_cn(), 1, 0),
    "no_j3": lambda: _cn(use_j3=False).hamiltonian_data,
    "no_j3_jagp": lambda: _cn(use_j3=False, jagp=True, lam_rank=8).hamiltonian_data,
    "no_jastrow": lambda: _cn(use_j3=False, j1=None, j2=None).hamiltonian_data,
    "j3_alone": lambda: _cn(j1=None, j2=None).hamiltonian_data,
    "exp_exp": lambda: _cn(j1=EE, j2=EE).hamiltonian_data,
    "pade_exp": lambda: _cn(j1=PE, j2=EE).hamiltonian_data,
    "pade_pade": lambda: _cn(j1=PE, j2=PP).hamiltonian_data,
    "spherical": _spherical,
    "g_shell": lambda: _shells("3s2p1d1f1g"),
    "g_shell_jagp": lambda: _shells("2s1p1g", jagp=True, lam_rank=8),
    "six_primitives": lambda: _shells("3s2p1d1f", n_prim=6),
    "one_primitive": lambda: _shells("3s2p1d1f", n_prim=1),
}


@functools.lru_cache(maxsize=None)
def _form(name):
    return FORMS[name]()


def _walkers(ham, W, seed=9):
    gem, pos = ham.wavefunction_data.geminal_data, ham.structure_data.positions
    rng = np.random.default_rng(seed)
    nuc = np.arange(gem.num_electron_up + gem.num_electron_dn) % len(pos)
    r = pos[nuc][None] + 0.8 * rng.standard_normal((W, len(nuc), 3))
    n = gem.num_electron_up
    return np.ascontiguousarray(r[:, :n]), np.ascontiguousarray(r[:, n:])


def _check_energies(ham, W, nv, precision, rtol):
    from jqmc_amd import _lib
    from jqmc_amd._api import WalkerState
    from jqmc_amd._pack import SystemPack
    from oracle import coulomb as oc
    from oracle import gfmc as og
    from oracle import wf as owf

    pack = SystemPack(ham, Nv=nv, precision=precision)
    if precision == "mixed":  # the flattened kernels' own values
        _lib.call("jqmc_system_set_mixed_guard", pack.handle, 0.0, 0.0)
    r_up, r_dn = _walkers(ham, W)
    ws = WalkerState(pack, W).init(r_up, r_dn)
    RT = ws.rotations(3, 0)
    e, kin, pot, _ = ws.local_energy(RT, with_parts=True)
    lattice = {m: ws.lrdmc_local_energy(WalkerState.lrdmc_params(0.25, non_local_move=m), RT)
               for m in ("tmove", "dltmove")}
    for w in (0, W - 1):
        R = RT[w].cpu().numpy()
        Gi = owf.geminal_inverse(owf.geminal(ham.wavefunction_data.geminal_data, r_up[w], r_dn[w]))
        tu, td = owf.kinetic_all_elements_fast(ham.wavefunction_data, r_up[w], r_dn[w], Gi)
        T = float(np.sum(tu) + np.sum(td))
        V = oc.coulomb_potential_fast(ham.coulomb_potential_data, ham.wavefunction_data, r_up[w], r_dn[w], R, Gi, 1, nv)
        tol = rtol * (1.0 + abs(T) + abs(V))
        assert abs(float(kin[w]) - T) <= tol and abs(float(pot[w]) - V) <= tol, (w, float(kin[w]), T, float(pot[w]), V)
        for m, (Vd, Vn) in lattice.items():
            d, n, _, _ = og.hamiltonian_elements(ham, r_up[w], r_dn[w], Gi, R, 0.25, m, Nv=nv)
            tol = rtol * (1.0 + abs(d) + abs(n))
            assert abs(float(Vd[w]) - d) <= tol and abs(float(Vn[w]) - n) <= tol, (m, w, float(Vd[w]), d, float(Vn[w]), n)


@pytest.mark.parametrize("name", sorted(FORMS))
def test_energies_match_oracle(name):
    _check_energies(_form(name), 7, 6, "fp64", 1e-9)


@pytest.mark.parametrize("name", ["spherical", "g_shell", "six_primitives", "doublet_jagp", "all_up", "pade_exp", "no_j3"])
def test_mixed_energies_match_oracle(name):
    _check_energies(_form(name), 5, 6, "mixed", 2e-5)


@pytest.mark.parametrize("name", sorted(FORMS))
def test_position_derivatives_match_oracle(name):
    from jqmc_amd._api import WalkerState
    from jqmc_amd._pack import SystemPack
    from oracle import forces as of

    ham = _form(name)
    W = 6
    r_up, r_dn = _walkers(ham, W)
    ws = WalkerState(SystemPack(ham), W).init(r_up, r_dn)
    RT = ws.rotations(3, 0)
    out = {k: v.cpu().numpy() for k, v in ws.position_grads(RT).items()}
    for w in (0, W - 1):
        R = RT[w].cpu().numpy()
        ref = of.local_energy_position_grads(ham, r_up[w], r_dn[w], R)
        ref.update(of.force_terms(ham, r_up[w], r_dn[w], R))
        for k in ("e_L", "dE_dr", "dE_dR", "dlnpsi_dr", "dlnpsi_dR", "force_HF", "force_PP"):
            a, b = np.asarray(out[k][w]), np.asarray(ref[k])
            err = float(np.abs(a - b).max()) / max(1.0, float(np.abs(b).max()))
            assert err <= 1e-9, (w, k, err)


@pytest.mark.parametrize("name", sorted(FORMS))
def test_parameter_derivatives_match_oracle(name):
    from jqmc_amd._api import WalkerState
    from jqmc_amd._pack import SystemPack
    from oracle import derivs as od

    ham = _form(name)
    W = 5
    r_up, r_dn = _walkers(ham, W)
    O = {k: v.cpu().numpy() for k, v in WalkerState(SystemPack(ham), W).init(r_up, r_dn).dln_psi_dparams().items()}
    for w in (0, W - 1):
        ref = od.dln_psi_dparams(ham.wavefunction_data, r_up[w], r_dn[w])
        assert set(ref) == set(O)
        for k, b in ref.items():
            b = np.asarray(b)
            assert O[k][w].shape == b.shape
            assert float(np.abs(O[k][w] - b).max()) <= 1e-9 * max(1e-300, float(np.abs(b).max())), (w, k)


@pytest.mark.parametrize("nv", [64, 65, 130])
def test_meshes_of_many_points_match_oracle(nv, monkeypatch):
    """Up to a wave of points and more, where an electron's points are taken in parts."""
    import jqmc_amd._pack
    import oracle.coulomb
    import oracle.forces
    from jqmc_amd._api import WalkerState
    from jqmc_amd._pack import SystemPack
    from jqmc_amd.coulomb_potential import _Mesh

    i = np.arange(nv) + 0.5
    th, ph = np.arccos(1.0 - 2.0 * i / nv), np.pi * (1.0 + 5.0**0.5) * i
    pts = np.stack([np.sin(th) * np.cos(ph), np.sin(th) * np.sin(ph), np.cos(th)], 1)
    mesh = _Mesh(nv, np.full(nv, 1.0 / nv), pts)
    for module in (jqmc_amd._pack, oracle.coulomb, oracle.forces):
        if hasattr(module, "get_mesh"):
            monkeypatch.setattr(module, "get_mesh", lambda n: mesh)
    ham = _form("doublet")
    _check_energies(ham, 6, nv, "fp64", 1e-9)
    r_up, r_dn = _walkers(ham, 6)
    ws = WalkerState(SystemPack(ham, Nv=nv), 6).init(r_up, r_dn)
    RT = ws.rotations(3, 0)
    out = {k: v.cpu().numpy() for k, v in ws.position_grads(RT).items()}
    for w in (0, 5):
        ref = oracle.forces.local_energy_position_grads(ham, r_up[w], r_dn[w], RT[w].cpu().numpy(), Nv=nv)
        for k in ("dE_dr", "dE_dR", "dlnpsi_dr", "dlnpsi_dR"):
            assert float(np.abs(out[k][w] - ref[k]).max()) <= 1e-9 * max(1.0, float(np.abs(ref[k]).max())), (w, k)


CHAINS = ["all_up", "doublet", "doublet_jagp", "g_shell", "no_j3", "no_jastrow", "one_electron", "pade_exp", "septet",
          "six_primitives"]


@pytest.mark.parametrize("name", CHAINS)
def test_moves_match_oracle(name):
    """Metropolis decisions and positions, then two lattice projections from there, on the oracle's stream (to
    1e-10; the weights to 1e-8: G^-1 after the moves)."""
    from jqmc_amd._api import WalkerState
    from jqmc_amd._pack import SystemPack
    from oracle import mcmc as om
    from test_gpu_lrdmc import _oracle_chain

    ham = _form(name)
    W, n_moves, seed = 3, 30, 77
    r_up, r_dn = _walkers(ham, W)
    ws = WalkerState(SystemPack(ham), W).init(r_up, r_dn)
    ws.sweep(n_moves, 0.5, 1e-4, seed, 0)
    ru, rd = ws.r_up.cpu().numpy(), ws.r_dn.cpu().numpy()
    for w in range(W):
        G, Gi = om.init_walker(ham, r_up[w], r_dn[w])
        acc, rej, ou, od, _, _ = om.metropolis_walker(ham, r_up[w], r_dn[w], Gi, G, seed, w, 0, n_moves, 0.5, 1e-4)
        assert ws.accepted[w].item() == acc and ws.rejected[w].item() == rej
        np.testing.assert_allclose(ru[w], ou, rtol=0, atol=1e-10)
        np.testing.assert_allclose(rd[w], od, rtol=0, atol=1e-10)
    ws.refresh()
    for move in ("tmove", "dltmove"):
        ws.init(ru, rd)
        out = ws.lrdmc_projection(WalkerState.lrdmc_params(0.3, E_scf=-10.0, n_steps=2, non_local_move=move), seed, 5)
        for w in range(W):
            a, b, _, _, wgt, _, _, _ = _oracle_chain(ham, ru[w], rd[w], 2, 0.3, -10.0, seed, w, 5, move)
            np.testing.assert_allclose(ws.r_up[w].cpu().numpy(), a, rtol=0, atol=1e-10)
            np.testing.assert_allclose(ws.r_dn[w].cpu().numpy(), b, rtol=0, atol=1e-10)
            assert abs(out["w_L"][w].item() - wgt) <= 1e-8 * abs(wgt)
