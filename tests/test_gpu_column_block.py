"""GPU parity of the acoustic column block (62 columns of a row by waves of four w levels) with
the CPU oracle at the sizes where its tiling can go wrong: the column counts around one and two
workgroups, one row, the fewest levels, level counts that leave the last wave one to four
levels, the deepest grid it takes (63 levels) and the first that runs the column march instead
(64).  Every value is computed by the oracle's operations in the oracle's order, so the
comparison is exact.  The mixed form, which has no oracle, is compared with the column march
in the same precision form.  The damping of w where the vertical Courant number exceeds 1 is
run by winds that reach it."""

import dataclasses

import numpy as np
import pytest

from tests.parity_util import FIELDS

pytestmark = pytest.mark.gpu

SPECIES = ("qv", "qc", "qr", "qi", "qs", "qg")


def _case(nx, ny, nz, ns=4):
    from wrf_gpu_amd import ic

    return ic.stratified_terrain_3d(nx=nx, ny=ny, nz=nz, dx=3000.0, ns=ns, u_sigma=1.0, sigma=0.5)


def _step(case, n):
    import torch
    from wrf_gpu_amd.dycore import Dycore, state_to_device, state_to_host

    print(f"[block] {case.metrics.nx}x{case.metrics.ny}x{case.metrics.nz} moist={case.namelist.moist}", flush=True)
    st = state_to_device(case.state, "cuda")
    dyn = Dycore(case.metrics, case.namelist)
    dyn.step(st, n)
    torch.cuda.synchronize()
    dyn.close()
    return state_to_host(st)


@pytest.mark.parametrize("grid", [(4, 1, 4), (61, 3, 5), (62, 2, 6), (63, 2, 7), (125, 3, 8), (21, 7, 47),
                                  (21, 7, 48), (21, 7, 63), (21, 7, 64)])
def test_column_block_matches_oracle(oracle_lib, grid):
    case = _case(*grid)
    ref = oracle_lib.run(case.metrics, case.namelist, case.state, 2)
    got = _step(case, 2)
    for k in FIELDS:
        assert np.array_equal(got[k], ref[k]), k


def test_moist_column_block_matches_oracle(oracle_lib):
    from wrf_gpu_amd import ic

    case = ic.with_moisture(_case(63, 5, 50), moist_adv_opt=2)
    ref = oracle_lib.run(case.metrics, case.namelist, case.state, 1)
    got = _step(case, 1)
    for k in FIELDS + SPECIES:
        assert np.array_equal(got[k], ref[k]), k


def test_mixed_column_block_matches_the_march(monkeypatch):
    """The block of the eager step (four levels a wave) and of the persistent step (13) against the
    march in both, mixed form; the persistent ones say which they ran, the eager one's launches are
    counted."""
    import torch
    from wrf_gpu_amd.dycore import Dycore, Ensemble, state_to_device, state_to_host

    case = _case(63, 5, 50)
    out = {}
    for choice in ("block", "march"):
        monkeypatch.setenv("WRFDYN_COLUMN_TILE", "" if choice == "block" else choice)
        for persistent in (False, True):
            print(f"[block] 63x5x50 mixed {choice} persistent={persistent}", flush=True)
            st = state_to_device(case.state, "cuda")
            dyn = Dycore(case.metrics, case.namelist, precision="mixed")
            if persistent:
                ens = Ensemble([(dyn, st)], persistent=True)
                assert ens.column_form(0) == choice
                ens.step(2)
                ens.status()
                ens.close()
            else:
                dyn.profile(["k_column_block", "k_column_w"])
                dyn.step(st, 2)
                assert list(dyn.profile_read()) == ["k_column_block" if choice == "block" else "k_column_w"]
            torch.cuda.synchronize()
            out[choice, persistent] = state_to_host(st)
            dyn.close()
    for key, got in out.items():
        for k in FIELDS:
            assert np.array_equal(got[k], out["march", False][k]), (key, k)


@pytest.mark.parametrize("form", ["dry", "moist", "mixed"])
def test_the_march_choice_runs_the_march(oracle_lib, monkeypatch, form):
    """WRFDYN_COLUMN_TILE=march selects the column march on a grid that the block holds, in every
    form and beside a choice of the workgroup order; without it the same grid runs the block."""
    import torch
    from wrf_gpu_amd import ic
    from wrf_gpu_amd.dycore import Dycore, state_to_device, state_to_host

    case = _case(63, 5, 50)
    if form == "moist":
        case = ic.with_moisture(case, moist_adv_opt=2)
    fields = FIELDS + (SPECIES if form == "moist" else ())
    names = ["k_column_block", "k_column_mu", "k_column_w"]
    out = {}
    for choice in ("march", ""):
        print(f"[block] 63x5x50 {form} WRFDYN_COLUMN_TILE={choice!r}", flush=True)
        monkeypatch.setenv("WRFDYN_COLUMN_TILE", choice)
        dyn = Dycore(case.metrics, case.namelist, precision="mixed" if form == "mixed" else "fp64")
        if choice == "march":
            dyn.set_tuned_config(-1, 0)
        st = state_to_device(case.state, "cuda")
        dyn.profile(names)
        dyn.step(st, 1)
        torch.cuda.synchronize()
        counts = {k: n for k, (_, n) in dyn.profile_read().items()}
        dyn.close()
        out[choice] = state_to_host(st)
        substeps = 1 + 2 + 4
        want = {"k_column_mu": substeps, "k_column_w": substeps} if choice else {"k_column_block": substeps}
        assert counts == want, counts
    for k in fields:
        assert np.array_equal(out["march"][k], out[""][k]), k
    if form != "mixed":
        ref = oracle_lib.run(case.metrics, case.namelist, case.state, 1)
        for k in fields:
            assert np.array_equal(out["march"][k], ref[k]), k


@pytest.mark.parametrize("nz,column,persistent", [(47, "", False), (63, "", False), (47, "", True), (47, "march", False),
                                                  (64, "", False), (47, "16x16", False)])
def test_w_damping_above_a_courant_number_of_one_matches_oracle(oracle_lib, monkeypatch, nz, column, persistent):
    """Winds that diverge from face to face and turn with height drive the vertical Courant number
    of the acoustic omega above 1 in most columns and leave it below 1 in others."""
    import torch
    from wrf_gpu_amd.dycore import Dycore, Ensemble, state_to_device, state_to_host

    base = _case(20, 6, nz)
    z = (np.arange(nz) + 0.5) / nz
    state = dict(base.state)
    state["u"] = state["u"] + 40.0 * np.cos(np.pi * z)[:, None, None] * np.where(np.arange(21) % 2 == 0, 1.0, -1.0)
    nl = dataclasses.replace(base.namelist, dt_s=12.0, w_damping=1)
    ref = oracle_lib.run(base.metrics, nl, state, 1)
    off = oracle_lib.run(base.metrics, dataclasses.replace(nl, w_damping=0), state, 1)
    acted = ref["w"] != off["w"]
    assert acted.any() and not acted[1:nz].all()
    print(f"[block] 20x6x{nz} Courant {column!r} persistent={persistent}", flush=True)
    monkeypatch.setenv("WRFDYN_COLUMN_TILE", column)
    dyn = Dycore(base.metrics, nl)
    st = state_to_device(state, "cuda")
    if persistent:
        ens = Ensemble([(dyn, st)], persistent=True)
        assert ens.column_form(0) == "block"
        ens.step(1)
        ens.status()
        ens.close()
    else:
        dyn.step(st, 1)
    torch.cuda.synchronize()
    dyn.close()
    got = state_to_host(st)
    for k in FIELDS:
        assert np.array_equal(got[k], ref[k]), k
