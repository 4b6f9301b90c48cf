"""J3 fields built from positions (k_init_jfield_mfma) against the defining sums on the cached AO values, at
sizes around the 64 x 64 x 16 tiles: fewer AOs than a tile, a last partial row tile, one walker."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,W,sym", [("water_ae", 1, False), ("water_ae", 13, True), ("benzene_ecp", 3, False),
                                        ("benzene_ecp", 32, True), ("water4_ecp", 5, False)])
def test_fields_from_positions(name, W, sym):
    import torch

    from jqmc_amd import synthetic
    from jqmc_amd._api import WalkerState
    from jqmc_amd._pack import system_for

    system = synthetic.WORKLOADS[name](0, j3_symmetric=sym)
    ws = WalkerState(system_for(system.hamiltonian_data), W).init(*system.initial_walkers(W))
    jm = system.hamiltonian_data.wavefunction_data.jastrow_data.jastrow_three_body_data.j_matrix
    J = torch.as_tensor(np.asarray(jm), dtype=torch.float64)
    A = ws.ao.cpu()
    after = A.flip(1).cumsum(1).flip(1) - A
    before = A.cumsum(1) - A
    ref = J[:, -1] + after @ J[:, :-1].T + before @ J[:, :-1]
    # each output sums 2 n_ao products of magnitude |J| |S|, S itself a sum over the electrons
    scale = J[:, -1].abs() + A.abs().sum(1, keepdim=True) @ (J[:, :-1].abs() + J[:, :-1].abs().T)
    bound = 2.0**-52 * (2 * A.shape[2] + 2 * A.shape[1]) * scale
    assert ((ws.jfield.cpu() - ref).abs() <= bound).all()


@pytest.mark.parametrize("n_ao,sym", [(1, False), (15, True), (17, False), (64, False), (64, True), (65, False)])
def test_small_and_large_sets_have_the_same_bits(n_ao, sym):
    """The tile form of small systems and the 64 x 64 form (from 65536 electrons on) add in the same order: a
    walker's fields do not depend on how many are set up together."""
    import torch

    from jqmc_amd import synthetic
    from jqmc_amd._api import WalkerState
    from jqmc_amd._pack import SystemPack

    st = synthetic._structure(["H", "H"], [[0.0, 0.0, 0.0], [0.0, 0.0, 1.4]])
    half = [n_ao // 2, n_ao - n_ao // 2]
    st.element_symbols = ["H", "N"]  # two shell lists, one electron each
    system = synthetic._assemble("x", st, {"H": f"{half[0]}s" if half[0] else "", "N": f"{half[1]}s"}, 1, j3_symmetric=sym)
    pack, n, rep = SystemPack(system.hamiltonian_data), 3, 12000
    assert pack.n_ao == n_ao and 2 * n * rep > 65536
    r_up, r_dn = (torch.as_tensor(r, device="cuda") for r in system.initial_walkers(n, seed=2))
    small = WalkerState(pack, n).init(r_up, r_dn)
    large = WalkerState(pack, n * rep).init(r_up.repeat(rep, 1, 1), r_dn.repeat(rep, 1, 1))
    assert torch.equal(large.jfield.view(rep, n, 2, n_ao), small.jfield.expand(rep, n, 2, n_ao))
    A, j3 = small.ao.cpu(), system.hamiltonian_data.wavefunction_data.jastrow_data.jastrow_three_body_data.j_matrix
    J = torch.as_tensor(np.asarray(j3), dtype=torch.float64)
    ref = J[:, -1] + torch.stack((A[:, 1] @ J[:, :-1].T, A[:, 0] @ J[:, :-1]), 1)
    size = J[:, -1].abs() + A.abs().flip(1) @ (J[:, :-1].abs() + J[:, :-1].abs().T)
    assert ((small.jfield.cpu() - ref).abs() <= 2.0**-52 * (2 * n_ao + 4) * size).all()
