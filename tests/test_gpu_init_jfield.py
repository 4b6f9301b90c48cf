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
