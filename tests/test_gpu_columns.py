"""GPU: y and z sweeps of whole columns, 6 to 8 of them per block, against marches
of 4: the same bits, dt and error word included.  tests/test_host_engine.py holds
the widths that the size rule gives these boxes."""
import numpy as np
import pytest

from gpluto_dev_amd import ic
from gpluto_dev_amd.stage import Definitions, RuntimeSetup, StageUpdate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,phys,solver,lim", [
    ((34, 29, 42), "MHD", "hlld", "MC_LIM"),          # y 6, z 5
    ((48, 20, 36), "MHD", "hll", "VANLEER_LIM"),      # y 7, z 4
    ((69, 20, 28), "MHD", "hllc", "MC_LIM"),          # y 8, z 6
    ((20, 65, 24), "MHD", "hlld", "VANLEER_LIM"),     # y marches, z 7
    ((62, 29, 20), "RMHD", "hll", "MC_LIM"),          # y 6, z 8
    ((48, 20, 36), "RMHD", "hlld", "VANLEER_LIM")])
def test_wide_columns_match_marches(n, phys, solver, lim, monkeypatch):
    rel = phys == "RMHD"
    state = ic.rmhd_turbulence(n, 5, lorentz_max=2.0, sigma=0.3) if rel else ic.mhd_turbulence(n, 5)
    res = []
    for march in ("", "4"):
        if march:
            monkeypatch.setenv("GPL_MARCH", march)
        print(f"case n={n} {phys} {solver} {lim} march={march}", flush=True)
        g = StageUpdate(Definitions(physics=phys, time_stepping="RK3", limiter=lim),
                        RuntimeSetup(n=n, solver=solver, cfl=0.2, gamma=4 / 3 if rel else 5 / 3))
        g.upload(*state)
        res.append((g.run(3, 1e-3), *g.download()))
        g.close()
    assert res[0][0] == res[1][0]
    assert all(np.array_equal(a, b) for a, b in zip(res[0][1:], res[1][1:]))
