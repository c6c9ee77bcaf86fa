"""GPU: HD boxes that take their stages direction by direction, against the
oracle, at the edges of the kernel's blocks and with every side type."""
import numpy as np
import pytest

from gpluto_dev_amd import ic
from gpluto_dev_amd.stage import Definitions, RuntimeSetup, StageUpdate

pytestmark = pytest.mark.gpu

SIDES = ["periodic", "outflow", "reflective"]


@pytest.mark.parametrize("n,ts,lim,solver", [
    ((3, 1501, 1), "RK2", "MC_LIM", "hllc"),             # the last block short
    ((16, 4096, 1), "RK3", "VANLEER_LIM", "hll"),        # 65536 cells: blocks of one wavefront
    ((5, 13108, 1), "RK2", "VANLEER_LIM", "hllc"),       # above: blocks of four
    ((3, 3, 1500), "RK2", "MC_LIM", "hll"), ((3, 100, 200), "RK3", "MC_LIM", "hllc"),
    ((11, 23, 260), "RK2", "VANLEER_LIM", "hllc"), ((65, 8, 201), "RK3", "MC_LIM", "hll")])
@pytest.mark.parametrize("sides", [0, 1, 2])
def test_narrow_boxes_match_oracle(n, ts, lim, solver, sides):
    import oracle
    dims = 2 if n[2] == 1 else 3
    t = []
    for d in range(3):
        if d >= dims or sides == 0:
            t += ["periodic", "periodic"]
        else:
            t += [SIDES[1 + (sides + d) % 2], SIDES[1 + (sides + d + 1) % 2]]
    vc = ic.hd_blast(n, 6)
    print(f"case n={n} {ts} {lim} {solver} {t}", flush=True)
    g = StageUpdate(Definitions(physics="HD", dimensions=dims, time_stepping=ts, limiter=lim),
                    RuntimeSetup(n=n, solver=solver, sides=tuple(t), gamma=1.4))
    g.upload(vc)
    g.set_timing(True)
    dt0 = 0.02/max(n)
    res = g.run(4, dt0)
    assert all(g.kernel_stats()[k][0] for k in ("k_hd_sweep_x", "k_hd_sweep_y", "k_dt"))
    g.set_timing(False)
    inv = g.advance_step(dt0)
    gvc, _, guc = g.download()
    g.close()
    o = oracle.Oracle(phys="hd", n=n, gamma=1.4, solver=solver, limiter=lim, time_stepping=int(ts[-1]),
                      sides=t)
    o.set_state(vc)
    assert res == o.run(4, dt0)
    assert inv == o.advance(dt0)
    ovc, _, ouc = o.get_state()
    assert np.array_equal(gvc, ovc) and np.array_equal(guc, ouc)
