"""GPU parity of the level runs with the CPU oracle.  A k-marching kernel whose launch has few
waves splits the levels into runs, each of which rebuilds the carried values of its lowest level
(vertical face flux, pressure windows, dpn, ph); the column sums and the gamma recurrence run
across the waves of a workgroup instead of up one thread.  Covered: level counts that leave the
last run one or two levels, one row and one column tile, column counts around a workgroup's 64,
the deepest grid of the block forms and the first beyond them, the moist instances, and grids on
both sides of the launch sizes at which the runs and the block forms stop (2048 waves; 512
workgroups of k_rom, 256 of k_col_setup).  Every value is computed by the oracle's operations in the oracle's order, so the
comparison is exact."""

import numpy as np
import pytest

from tests.parity_util import FIELDS

pytestmark = pytest.mark.gpu

SPECIES = ("qv", "qc", "qr", "qi", "qs", "qg")


@pytest.mark.parametrize("grid,moist", [((4, 1, 4), False), ((64, 1, 5), False), ((65, 2, 9), True),
                                        ((63, 5, 21), False), ((30, 9, 63), True), ((30, 9, 64), False),
                                        ((124, 256, 7), False), ((124, 257, 7), False), ((62, 256, 5), False),
                                        ((62, 257, 5), False), ((62, 256, 5), True), ((362, 361, 5), False),
                                        ((363, 363, 5), False)])
def test_level_runs_match_oracle(oracle_lib, grid, moist):
    import torch
    from wrf_gpu_amd import ic
    from wrf_gpu_amd.dycore import Dycore, state_to_device, state_to_host

    nx, ny, nz = grid
    case = ic.stratified_terrain_3d(nx=nx, ny=ny, nz=nz, dx=3000.0, ns=4, u_sigma=1.0, sigma=0.5)
    if moist:
        case = ic.with_moisture(case, moist_adv_opt=1)
    print(f"[runs] {nx}x{ny}x{nz} moist={moist}", flush=True)
    ref = oracle_lib.run(case.metrics, case.namelist, case.state, 1)
    st = state_to_device(case.state, "cuda")
    dyn = Dycore(case.metrics, case.namelist)
    dyn.step(st, 1)
    torch.cuda.synchronize()
    dyn.close()
    got = state_to_host(st)
    for k in FIELDS + (SPECIES if moist else ()):
        assert np.array_equal(got[k], ref[k]), k
