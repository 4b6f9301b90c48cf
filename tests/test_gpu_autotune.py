"""Launch-shape knobs and the autotuner (jqmc_amd/autotune.py): every proposal walkers-per-block setting
takes identical decisions (bit-identical positions), the local-energy knobs are taken and change
nothing, bad knob values are refused, and autotune() applies a valid choice and round-trips through its
JSON cache, older ones included."""

import json

import pytest
import torch

from jqmc_amd import _lib, synthetic
from jqmc_amd._api import WalkerState
from jqmc_amd._pack import system_for
from jqmc_amd.autotune import CANDIDATES, autotune, get_tuning, set_tuning

pytestmark = pytest.mark.gpu


def _state(prec="fp64", W=96):
    s = synthetic.chain_ecp(10, seed=1)
    pack = system_for(s.hamiltonian_data, Nv=6, precision=prec)
    ru, rd = s.initial_walkers(W, seed=3)
    return pack, ru, rd


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_knobs_change_no_result_bit(prec):
    pack, ru, rd = _state(prec)
    pos = {}
    for w in (0,) + CANDIDATES["sweep_walkers_per_block"]:
        set_tuning(pack, sweep_walkers_per_block=w)
        wk = WalkerState(pack, len(ru)).init(ru, rd)
        wk.sweep(12, 0.5, 1e-4, 7, 0)
        pos[w] = (wk.r_up.clone(), wk.r_dn.clone(), wk.accepted.clone())
    for w in CANDIDATES["sweep_walkers_per_block"]:
        assert all(torch.equal(a, b) for a, b in zip(pos[w], pos[0])), w


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_local_energy_knobs_are_taken_and_change_nothing(prec):
    """Both knobs of the local energy keep their values and reach no launch."""
    pack, ru, rd = _state(prec)
    ws = WalkerState(pack, len(ru)).init(ru, rd)
    RT = ws.rotations(4, 0)
    ref = ws.local_energy(RT).clone()
    for knob in ("el_walkers_per_block", "el_waves_per_walker"):
        assert knob not in CANDIDATES
        for v in (1, 2, 4, 0):
            set_tuning(pack, **{knob: v})
            assert get_tuning(pack)[knob] == v
            assert torch.equal(ws.local_energy(RT), ref), (knob, v)


def test_bad_knob_values_are_refused():
    pack, _, _ = _state()
    with pytest.raises(_lib.JqmcError):
        set_tuning(pack, el_waves_per_walker=3)
    with pytest.raises(_lib.JqmcError):
        set_tuning(pack, el_walkers_per_block=3)
    with pytest.raises(_lib.JqmcError):
        set_tuning(pack, sweep_walkers_per_block=3)
    with pytest.raises(_lib.JqmcError):
        _lib.call("jqmc_system_set_tuning", pack.handle, 99, 1)


def test_autotune_applies_and_caches(tmp_path):
    pack, ru, rd = _state(W=128)
    ws = WalkerState(pack, len(ru)).init(ru, rd)
    r0 = ws.r_up.clone()
    cache = tmp_path / "tune.json"
    out = autotune(ws, reps=1, cache_path=str(cache))
    assert not out["cached"]
    assert set(out["best"]) == set(CANDIDATES)
    for k, v in out["best"].items():
        assert v in CANDIDATES[k] and get_tuning(pack)[k] == v, (k, v)
    assert torch.equal(ws.r_up, r0), "the caller's walkers do not move"
    assert len(out["sweep_ms"]) == 3
    set_tuning(pack, sweep_walkers_per_block=0)
    again = autotune(ws, cache_path=str(cache))
    assert again["cached"] and get_tuning(pack)["sweep_walkers_per_block"] == out["best"]["sweep_walkers_per_block"]
    (key, best), = json.loads(cache.read_text()).items()
    assert best == out["best"]
    # a file of an earlier version, with the local-energy knobs
    older = {"el_walkers_per_block": 2, "sweep_walkers_per_block": 1, "el_waves_per_walker": 2}
    cache.write_text(json.dumps({key: older}))
    assert autotune(ws, cache_path=str(cache))["cached"] and get_tuning(pack) == older
