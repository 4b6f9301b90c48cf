"""The column reductions of the SR step and the per-walker outer products of the parameter derivatives at the
edges of their tiles.

Statistics: against extended precision.  The mean is a sum of S products in FP64: |error| <= (S + 4) u sum |w O|
(u = 2^-53); the centred squares are merged from groups with their own means: |error| <= 4 (S + 16) u (var +
u mean^2) up to the weights' own sum.  Projection: (S + 4) u sum |terms|.  Outer products: K + 2 roundings of
sum |L R|."""

import numpy as np
import pytest
import torch

from jqmc_amd import _lib
from jqmc_amd._api import _ptr, stream_handle

pytestmark = pytest.mark.gpu
U = 2.0**-53


@pytest.mark.parametrize("S,P,ld,shift", [(1, 1, 1, 0.0), (2, 63, 70, 1e6), (8, 64, 64, 0.0), (63, 65, 65, 1e6),
                                          (65, 130, 137, -3.0), (1030, 7, 9, 1e8)])
def test_column_statistics_and_projection(S, P, ld, shift):
    rng = np.random.default_rng(S + P)
    O = np.full((S, ld), np.nan)
    O[:, :P] = rng.normal(size=(S, P)) + shift
    wn = rng.uniform(0.0, 1.0, size=S)
    wn[::3] *= 1e-8
    if S > 2:
        wn[1] = 0.0
    wn /= wn.sum()
    X, w = O[:, :P].astype(np.longdouble), wn.astype(np.longdouble)
    m_ref = w @ X
    v_ref = w @ (X - m_ref) ** 2
    Od, wd = torch.as_tensor(O, device="cuda"), torch.as_tensor(wn, device="cuda")
    mean = torch.full((P,), np.nan, dtype=torch.float64, device="cuda")
    var = torch.full_like(mean, np.nan)
    _lib.call("jqmc_sr_colstats", _ptr(Od), S, P, ld, _ptr(wd), _ptr(mean), _ptr(var), stream_handle())
    dm = np.abs(mean.cpu().numpy() - m_ref)
    dv = np.abs(var.cpu().numpy() - v_ref)
    size = np.abs(X).max(axis=0)
    assert (dm <= (S + 4) * U * (w @ np.abs(X))).all()
    assert (dv <= 4 * (S + 16) * U * (v_ref + U * size**2)).all()
    rs, cs, x = rng.uniform(0.5, 1.5, size=S), rng.uniform(0.5, 1.5, size=P), rng.normal(size=S)
    args = [torch.as_tensor(np.ascontiguousarray(t), device="cuda") for t in (m_ref.astype(np.float64), rs, cs, x)]
    out = torch.full((P,), np.nan, dtype=torch.float64, device="cuda")
    _lib.call("jqmc_sr_project", _ptr(Od), S, P, ld, *[_ptr(t) for t in args], _ptr(out), stream_handle())
    terms = (X - m_ref.astype(np.float64)) * (rs * x)[:, None] * cs
    assert (np.abs(out.cpu().numpy() - terms.sum(axis=0)) <= (S + 8) * U * (np.abs(terms).sum(axis=0) + U)).all()


@pytest.mark.parametrize("S,zero", [(64, slice(0, 8)), (200, slice(0, 64)), (200, slice(64, 128)), (1030, slice(0, 700)),
                                    (70, slice(0, 69)), (130, slice(8, 130))])
def test_column_statistics_with_rows_of_no_weight(S, zero):
    """Whole groups of rows with weight exactly 0 (walkers that are out), wherever they stand; the bound of the
    statistics above.  A constant column has no negative variance."""
    rng = np.random.default_rng(S)
    P = 70
    O = rng.normal(size=(S, P)) + 1e7
    O[:, 3] = -0.1
    O[:, 4] = 1e5 / 3.0
    wn = rng.uniform(0.2, 1.0, size=S)
    wn[zero] = 0.0
    wn /= wn.sum()
    X, w = O.astype(np.longdouble), wn.astype(np.longdouble)
    m_ref = w @ X
    v_ref = w @ (X - m_ref) ** 2
    Od, wd = torch.as_tensor(O, device="cuda"), torch.as_tensor(wn, device="cuda")
    mean = torch.full((P,), np.nan, dtype=torch.float64, device="cuda")
    var = torch.full_like(mean, np.nan)
    _lib.call("jqmc_sr_colstats", _ptr(Od), S, P, P, _ptr(wd), _ptr(mean), _ptr(var), stream_handle())
    m, v = mean.cpu().numpy(), var.cpu().numpy()
    assert (np.abs(m - m_ref) <= (S + 4) * U * (w @ np.abs(X))).all()
    assert (np.abs(v - v_ref) <= 4 * (S + 16) * U * (v_ref + U * np.abs(X).max(axis=0) ** 2)).all()
    assert (v >= 0.0).all()


@pytest.mark.parametrize("name,W", [("water_ae", 1), ("water_ae", 17), ("chain10", 9), ("benzene_ecp", 8),
                                    ("water4_jagp", 3)])
def test_parameter_blocks_are_the_outer_products(name, W):
    from jqmc_amd import synthetic

    if name == "chain10":
        system = synthetic.chain_ecp(10, 1)
    elif name == "water4_jagp":
        system = synthetic.water4_ecp(0, jagp=True)
    else:
        system = synthetic.WORKLOADS[name](0)
    _check_parameter_blocks(system, W)


@pytest.mark.parametrize("jagp", [False, True])
@pytest.mark.parametrize("n_ao,W", [(16, 3), (17, 5), (32, 2), (33, 7), (112, 3), (113, 3)])
def test_parameter_blocks_around_the_narrow_tiles(n_ao, W, jagp):
    """AO counts around the 16- and 32-column tiles of the narrow form and its largest size; an open shell."""
    from jqmc_amd import synthetic

    st = synthetic._structure(["N"], [[0.0, 0.0, 0.0]])
    _check_parameter_blocks(synthetic._assemble("n", st, {"N": f"{n_ao}s"}, 1, jagp=jagp, lam_rank=12), W)


def _check_parameter_blocks(system, W):
    """The J3 and Lambda_p blocks against outer products of the cached rows."""
    from jqmc_amd._api import WalkerState
    from jqmc_amd._pack import SystemPack

    r_up, r_dn = system.initial_walkers(W, seed=21)
    ws = WalkerState(SystemPack(system.hamiltonian_data), W).init(r_up, r_dn)
    O = {k: v.reshape(W, -1) for k, v in ws.dln_psi_dparams().items()}
    A = ws.ao
    na, no = A.shape[2], ws.orb.shape[2]
    nu, nd = ws.Ginv.shape[1], A.shape[1] - ws.Ginv.shape[1]
    after = A.flip(1).cumsum(1).flip(1) - A
    for key, L, R, off in (("j3_matrix", A, after, 1),
                           ("lambda_matrix", (ws.Ginv @ ws.orb[:, :nu])[:, :nd], ws.orb[:, nu:], nu - nd)):
        ref, size = L.transpose(1, 2) @ R, L.abs().transpose(1, 2) @ R.abs()
        got = O[key].reshape(W, L.shape[2], R.shape[2] + off)[:, :, : R.shape[2]]
        if key == "lambda_matrix":  # Z is a rounded product itself
            size = (ws.Ginv.abs() @ ws.orb[:, :nu].abs())[:, :nd].transpose(1, 2) @ R.abs()
        else:  # so are the sums over the electrons after
            size = L.abs().transpose(1, 2) @ A.abs().sum(1, keepdim=True).expand_as(R)
        assert ((got - ref).abs() <= (2 * A.shape[1] + 8) * U * size).all(), key
    assert na and no
