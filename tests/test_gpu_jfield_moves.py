"""J3 fields after moves (k_sweep_jfield_mfma) where its tiles end: walker counts around the segments of 64 and
their groups of 16 movers, AO counts that are no multiple of 16, symmetric and non-symmetric J3, Metropolis
sweeps and LRDMC moves.  Against the fields of the same walkers built anew from their positions: the increments
add up to n_moves (n_ao + n_el) roundings of sums of |J a| (at most 1e-10 of the largest field here)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _system(name, sym):
    import dataclasses

    from jqmc_amd import synthetic

    system = synthetic.chain_ecp(10, 1) if name == "chain10" else synthetic.WORKLOADS[name](0)
    ham = system.hamiltonian_data
    if sym:
        jas = ham.wavefunction_data.jastrow_data
        j3 = jas.jastrow_three_body_data
        m = j3.j_matrix.copy()
        m[:, :-1] = 0.5 * (m[:, :-1] + m[:, :-1].T)
        j3 = dataclasses.replace(j3, j_matrix=m)
        jas = dataclasses.replace(jas, jastrow_three_body_data=j3)
        ham = dataclasses.replace(ham, wavefunction_data=dataclasses.replace(ham.wavefunction_data, jastrow_data=jas))
    return system, ham


@pytest.mark.parametrize("sym", [False, True])
@pytest.mark.parametrize("name,W", [("water_ae", 1), ("water_ae", 15), ("water_ae", 65), ("chain10", 129),
                                    ("benzene_ecp", 17), ("benzene_ecp", 600)])
def test_fields_after_moves(name, W, sym):
    from jqmc_amd._api import WalkerState
    from jqmc_amd._pack import SystemPack

    system, ham = _system(name, sym)
    pack = SystemPack(ham, Nv=6)
    r_up, r_dn = system.initial_walkers(W, seed=5)

    def check(ws):
        ref = WalkerState(pack, W).init(ws.r_up.cpu().numpy(), ws.r_dn.cpu().numpy()).jfield
        assert float((ws.jfield - ref).abs().max()) <= 1e-10 * float(ref.abs().max())

    ws = WalkerState(pack, W).init(r_up, r_dn)
    ws.sweep(24, 2.0, 1.0e-2, 11, 0)
    assert int(ws.accepted.sum()) > 0
    check(ws)
    if not sym:
        ws.lrdmc_projection(WalkerState.lrdmc_params(0.3, n_steps=3), 7, 0)
        check(ws)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("sym", [False, True])
@pytest.mark.parametrize("name,W", [("water_ae", 49153), ("benzene_ecp", 6593)])
def test_many_walkers_give_the_bits_of_few(name, W, sym, precision):
    """Many walkers take two tiles of 16 AOs a wave and the proposal with fewer loads in flight; the sums of an element
    stay the same, and the draws of a walker depend on its index alone, so the first walkers of a large set end as
    those of a small one do.  25 and 228 AOs: the last pair of tiles holds 25 and 4 columns."""
    from jqmc_amd._api import WalkerState
    from jqmc_amd._pack import SystemPack

    system, ham = _system(name, sym)
    pack = SystemPack(ham, Nv=6, precision=precision)
    r_up, r_dn = system.initial_walkers(W, seed=5)

    def run(n):
        ws = WalkerState(pack, n).init(r_up[:n], r_dn[:n])
        ws.sweep(12, 2.0, 1.0e-2, 11, 0)
        return ws

    many, few = run(W), run(300)
    assert W > 5 * 4 * 256 and -(-W // 64) * -(-pack.n_ao // 16) >= 6 * 256 and int(few.accepted.sum()) > 0
    assert torch.equal(many.r_up[:300], few.r_up) and torch.equal(many.jfield[:300], few.jfield)
    if precision == "fp64":
        ref = WalkerState(pack, W).init(many.r_up.cpu().numpy(), many.r_dn.cpu().numpy()).jfield
        assert float((many.jfield - ref).abs().max()) <= 1e-10 * float(ref.abs().max())
