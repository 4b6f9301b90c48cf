"""The flattened position derivatives (k_fr_kinetic / k_fr_points / k_fr_adjoint / k_fr_pairing / k_fr_orbital /
k_fr_out) against the oracle where their tiles end: walker counts around the groups of four walkers and 64
electrons, meshes that fill a wave differently, up to 16 and more than 64 MOs, different MOs per spin, Cartesian
closed shells (the other forms: test_gpu_forms.py); and a call longer than the walkers taken at a time against short calls.
Tolerance: 1e-9 of the largest element, as for the other checks of these derivatives."""

import numpy as np
import pytest
import torch

from test_gpu_el_flattened import _with_mos
from test_gpu_forces import _err, _rotations

pytestmark = pytest.mark.gpu

CASES = [("water_ae", None, 6, 13), ("chain10", None, 4, 9), ("chain10", None, 18, 7), ("benzene_ecp", None, 12, 3),
         ("chain56", None, 6, 2), ("chain30", (17, False), 12, 3), ("chain30", (70, True), 6, 2)]


def _state(name, mos, nv, W):
    from jqmc_amd import synthetic
    from jqmc_amd._api import WalkerState
    from jqmc_amd._pack import SystemPack

    system = synthetic.chain_ecp(int(name[5:]), 1) if name.startswith("chain") else synthetic.WORKLOADS[name](0)
    ham = system.hamiltonian_data if mos is None else _with_mos(system, mos[0], mos[1])
    r_up, r_dn = system.initial_walkers(W, seed=13, sigma=0.8)
    return ham, WalkerState(SystemPack(ham, Nv=nv), W).init(r_up, r_dn), r_up, r_dn


@pytest.mark.parametrize("name,mos,nv,W", CASES)
def test_position_grads_match_oracle(name, mos, nv, W):
    from oracle import forces as of

    ham, ws, r_up, r_dn = _state(name, mos, nv, W)
    RT = _rotations(W)
    out = {k: v.cpu().numpy() for k, v in ws.position_grads(torch.as_tensor(RT)).items()}
    assert all(np.isfinite(v).all() for v in out.values())
    for w in sorted({0, W - 1}):
        ref = of.local_energy_position_grads(ham, r_up[w], r_dn[w], RT[w], Nv=nv)
        ref.update(of.force_terms(ham, r_up[w], r_dn[w], RT[w], Nv=nv))
        assert abs(out["e_L"][w] - ref["e_L"]) <= 1e-10 * max(1.0, abs(ref["e_L"]))
        for k in ("dE_dr", "dE_dR", "dlnpsi_dr", "dlnpsi_dR", "force_HF", "force_PP"):
            assert _err(out[k][w], ref[k]) < 1e-9, (w, k, _err(out[k][w], ref[k]))


def test_long_call_matches_short_calls():
    """A call of 13112 walkers of 10 electrons (more than 2^17 electrons) is taken in two parts; every walker's
    results are those of a short call."""
    from jqmc_amd._api import WalkerState

    W = 13112
    _, ws, r_up, r_dn = _state("water_ae", None, 6, W)
    out = ws.position_grads(None)
    for a, b in ((0, 3), (6550, 6560), (W - 4, W)):
        sub = WalkerState(ws.pack, b - a).init(r_up[a:b], r_dn[a:b])
        ref = sub.position_grads(None)
        for k, v in ref.items():
            scale = max(1.0, float(v.abs().max()))
            assert float((out[k][a:b] - v).abs().max()) <= 1e-9 * scale, k


@pytest.mark.parametrize("name", ["h2", "water_ae", "chain10"])
def test_number_of_walkers_changes_no_bit(name):
    """The waves that k_fr_out and k_fr_pairing give a walker, the J3 product's form and the parts of a call depend on
    how many walkers there are; their results do not."""
    from jqmc_amd import synthetic
    from jqmc_amd._api import WalkerState
    from jqmc_amd._pack import SystemPack

    if name == "h2":
        st = synthetic._structure(["H", "H"], [[0.0, 0.0, 0.0], [0.0, 0.0, 1.4]])
        system = synthetic._assemble("h2", st, {"H": "2s1p"}, 1)
    else:
        system = synthetic.chain_ecp(10, 1) if name == "chain10" else synthetic.water_ae(0)
    pack, n, rep = SystemPack(system.hamiltonian_data), 5, 4000
    r_up, r_dn = (torch.as_tensor(r, device="cuda") for r in system.initial_walkers(n, seed=2, sigma=0.8))
    small = WalkerState(pack, n).init(r_up, r_dn).position_grads()
    large = WalkerState(pack, n * rep).init(r_up.repeat(rep, 1, 1), r_dn.repeat(rep, 1, 1)).position_grads()
    for k, v in small.items():
        assert torch.equal(large[k].view(rep, *v.shape), v.expand(rep, *v.shape)), k
