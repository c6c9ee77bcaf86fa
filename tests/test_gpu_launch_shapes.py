"""GPU: every launch shape that the size rules can pick gives the same bits as
the oracle (FP64) or as one fixed shape (mixed precision), at sizes where a
shape leaves remainders."""
import numpy as np
import pytest

from gpluto_dev_amd import ic
from gpluto_dev_amd.stage import Definitions, RuntimeSetup, StageUpdate

pytestmark = pytest.mark.gpu


def _run(n, steps, first_dt, precision="fp64", ts="RK2", lim="MC_LIM", sides=()):
    vc, vs = ic.mhd_turbulence(n, 17)
    print(f"case n={n} {precision} {ts} {lim} {sides}", flush=True)
    g = StageUpdate(Definitions(time_stepping=ts, limiter=lim), RuntimeSetup(n=n, sides=tuple(sides)),
                    precision=precision)
    g.upload(vc, vs)
    res = g.run(steps, first_dt)
    vc, vs, uc = g.download()
    g.close()
    return res, vc, vs, uc


@pytest.mark.parametrize("march", ["", "1", "2", "4", "8", "32", "64"])
def test_march_lengths_match_oracle(march, monkeypatch):
    """y and z marches of every length, remainders included, in FP64."""
    import oracle
    if march:
        monkeypatch.setenv("GPL_MARCH", march)
    n = (19, 23, 37)
    (err, t, dt), vc, vs, _ = _run(n, 4, 1e-3)
    o = oracle.Oracle(phys="mhd", n=n, gamma=5 / 3)
    o.set_state(*ic.mhd_turbulence(n, 17))
    assert (err, t, dt) == o.run(4, 1e-3)
    ovc, ovs, _ = o.get_state()
    assert np.array_equal(vc, ovc) and np.array_equal(vs, ovs)


@pytest.mark.parametrize("n", [(19, 23, 37), (64, 17, 33)])
def test_march_lengths_mixed(n, monkeypatch):
    """The mixed form's x+y kernel and z march: the same bits at every length."""
    monkeypatch.setenv("GPL_MARCH", "16")
    ref = _run(n, 4, 1e-3, precision="mixed")
    for march in ("", "1", "2", "4", "8"):
        monkeypatch.setenv("GPL_MARCH", march)
        got = _run(n, 4, 1e-3, precision="mixed")
        assert got[0] == ref[0]
        assert all(np.array_equal(a, b) for a, b in zip(got[1:], ref[1:])), march


@pytest.mark.parametrize("n", [(15, 11, 9), (80, 10, 7), (130, 101, 79)])
@pytest.mark.parametrize("lim", ["MC_LIM", "VANLEER_LIM"])
def test_emf_choice_matches_tiles(n, lim, monkeypatch):
    """The EMF kernel of the box's size (flat or 64 x 4 edges, tiles of 8 above
    a million cells) against tiles of 16 planes."""
    got = _run(n, 2, 1e-3, lim=lim)
    monkeypatch.setenv("GPL_EMF_MARCH", "-16")
    ref = _run(n, 2, 1e-3, lim=lim)
    assert got[0] == ref[0] and got[0][0] == 0
    assert all(np.array_equal(a, b) for a, b in zip(got[1:], ref[1:]))


@pytest.mark.parametrize("n", [(3, 70, 1), (65, 19, 1), (130, 37, 1), (128, 515, 1)])
@pytest.mark.parametrize("sides", [(), ("outflow", "reflective", "reflective", "outflow", "periodic", "periodic")])
def test_one_2d_box_matches_oracle(n, sides):
    """One 2D box: the y march's length follows from its size."""
    import oracle
    vc, vs = ic.mhd_turbulence(n, 4)
    g = StageUpdate(Definitions(dimensions=2), RuntimeSetup(n=n, sides=sides))
    g.upload(vc, vs)
    res = g.run(4, 5e-4)
    gvc, gvs, _ = g.download()
    g.close()
    o = oracle.Oracle(phys="mhd", n=n, gamma=5 / 3, sides=sides or None)
    o.set_state(vc, vs)
    assert res == o.run(4, 5e-4)
    ovc, ovs, _ = o.get_state()
    assert np.array_equal(gvc, ovc) and np.array_equal(gvs, ovs)


@pytest.mark.parametrize("n", [(3, 4, 5), (9, 3, 3)])
@pytest.mark.parametrize("sides", [
    ("outflow", "reflective", "reflective", "reflective", "outflow", "outflow"),
    ("periodic", "periodic", "outflow", "reflective", "reflective", "outflow"),
    ("reflective", "outflow", "periodic", "periodic", "periodic", "periodic")])
def test_sides_of_the_smallest_boxes(n, sides):
    """Every side type on boxes whose two ghost fills reach the same cells."""
    import oracle
    vc, vs = ic.mhd_turbulence(n, 4)
    g = StageUpdate(Definitions(), RuntimeSetup(n=n, sides=sides))
    g.upload(vc, vs)
    res = g.run(3, 5e-4)
    gvc, gvs, _ = g.download()
    g.close()
    o = oracle.Oracle(phys="mhd", n=n, gamma=5 / 3, sides=sides)
    o.set_state(vc, vs)
    assert res == o.run(3, 5e-4)
    ovc, ovs, _ = o.get_state()
    assert np.array_equal(gvc, ovc) and np.array_equal(gvs, ovs)


HD_SIDES = ["periodic", "outflow", "reflective"]


@pytest.mark.parametrize("n,ts,lim,solver", [
    # 1D: one wavefront per block up to 16384 zones (56 or 52 zones each), four above
    ((3, 1, 1), "RK2", "MC_LIM", "hllc"), ((5, 1, 1), "RK3", "VANLEER_LIM", "hll"),
    ((52, 1, 1), "RK3", "MC_LIM", "hllc"), ((56, 1, 1), "RK2", "VANLEER_LIM", "hllc"),
    ((113, 1, 1), "RK2", "MC_LIM", "hll"), ((16385, 1, 1), "RK3", "MC_LIM", "hllc"),
    ((16617, 1, 1), "RK2", "MC_LIM", "hllc"),
    # 2D: 63 columns per wavefront
    ((3, 3, 1), "RK2", "MC_LIM", "hllc"), ((62, 7, 1), "RK3", "MC_LIM", "hll"),
    ((63, 40, 1), "RK2", "VANLEER_LIM", "hllc"), ((64, 33, 1), "RK2", "MC_LIM", "hllc"),
    ((127, 190, 1), "RK3", "VANLEER_LIM", "hllc"),
    # 3D: 64 x 7 cells per block
    ((3, 3, 3), "RK3", "MC_LIM", "hllc"), ((63, 8, 5), "RK2", "VANLEER_LIM", "hllc"),
    ((64, 7, 4), "RK2", "MC_LIM", "hll"), ((65, 15, 33), "RK3", "MC_LIM", "hllc"),
    ((66, 6, 70), "RK2", "MC_LIM", "hllc")])
@pytest.mark.parametrize("sides", [0, 1, 2])
def test_hd_launch_shapes_match_oracle(n, ts, lim, solver, sides):
    """HD boxes at the edges of the kernels' blocks; every side type in turn on
    every direction, from a noisy blast."""
    import oracle
    dims = 1 if n[1] == 1 else 2 if n[2] == 1 else 3
    t = []
    for d in range(3):
        if d >= dims or sides == 0:
            t += ["periodic", "periodic"]
        else:
            t += [HD_SIDES[1 + (sides + d) % 2], HD_SIDES[1 + (sides + d + 1) % 2]]
    vc = ic.hd_blast(n, 6)
    print(f"case n={n} {ts} {lim} {solver} {t}", flush=True)
    g = StageUpdate(Definitions(physics="HD", dimensions=dims, time_stepping=ts, limiter=lim),
                    RuntimeSetup(n=n, solver=solver, sides=tuple(t), gamma=1.4))
    g.upload(vc)
    dt0 = 0.02/max(n)
    res = g.run(5, dt0)
    more = g.run(2, -1.0)                      # goes on from the device's dt
    inv = g.advance_step(dt0)
    gvc, _, guc = g.download()
    g.close()
    o = oracle.Oracle(phys="hd", n=n, gamma=1.4, solver=solver, limiter=lim, time_stepping=int(ts[-1]),
                      sides=t)
    o.set_state(vc)
    assert res == o.run(5, dt0)
    dt = res[2]
    err, time = 0, res[1]
    for _ in range(2):
        e, i = o.advance(dt)
        err |= e
        time += dt
        dt = min(0.4/i, 1.1*dt)
    assert more == (err, time, dt)
    assert inv == o.advance(dt0)
    ovc, _, ouc = o.get_state()
    assert np.array_equal(gvc, ovc) and np.array_equal(guc, ouc)


@pytest.mark.parametrize("n,phys,solver,lim,sides", [
    ((5, 3, 4), "MHD", "hlld", "MC_LIM", ()),                    # columns shorter than a wavefront's rows
    ((9, 64, 5), "MHD", "hll", "VANLEER_LIM", ()),               # the longest column, 4 per block
    ((33, 17, 64), "MHD", "hlld", "MC_LIM", ()),                 # remainders in x and in the last wavefront
    ((13, 65, 32), "MHD", "hllc", "MC_LIM", ()),                 # y marches, z in columns of 8
    ((18, 14, 21), "MHD", "hlld", "VANLEER_LIM", ("outflow", "reflective", "outflow", "outflow",
                                                  "reflective", "reflective")),
    ((21, 30, 11), "RMHD", "hll", "MC_LIM", ()),
    ((14, 19, 38), "RMHD", "hlld", "VANLEER_LIM", ()),
])
def test_columns_match_marches(n, phys, solver, lim, sides, monkeypatch):
    """y and z sweeps of whole columns against marches of 4: the same bits, dt
    and error word included."""
    rel = phys == "RMHD"
    state = ic.rmhd_turbulence(n, 5, lorentz_max=2.0, sigma=0.3) if rel else ic.mhd_turbulence(n, 5)
    res = []
    for march in ("", "4"):
        if march:
            monkeypatch.setenv("GPL_MARCH", march)
        print(f"case n={n} {phys} {solver} {lim} {sides} march={march}", flush=True)
        g = StageUpdate(Definitions(physics=phys, time_stepping="RK3", limiter=lim),
                        RuntimeSetup(n=n, solver=solver, sides=tuple(sides), cfl=0.2,
                                     gamma=4 / 3 if rel else 5 / 3))
        g.upload(*state)
        res.append((g.run(3, 1e-3), *g.download()))
        g.close()
    assert res[0][0] == res[1][0]
    assert all(np.array_equal(a, b) for a, b in zip(res[0][1:], res[1][1:]))


@pytest.mark.parametrize("n", [(5, 21, 37), (20, 23, 29), (72, 17, 19)])
def test_rows_per_block_match_oracle(n):
    """x sweeps of 4, 3 and 2 rows per block, the last block short of a row."""
    import oracle
    (err, t, dt), vc, vs, _ = _run(n, 3, 1e-3)
    o = oracle.Oracle(phys="mhd", n=n, gamma=5 / 3)
    o.set_state(*ic.mhd_turbulence(n, 17))
    assert (err, t, dt) == o.run(3, 1e-3)
    ovc, ovs, _ = o.get_state()
    assert np.array_equal(vc, ovc) and np.array_equal(vs, ovs)


@pytest.mark.parametrize("n,lim", [((4, 300, 1), "MC_LIM"), ((31, 9, 1), "VANLEER_LIM"), ((32, 8, 1), "MC_LIM"),
                                   ((33, 17, 1), "MC_LIM"), ((65, 7, 1), "VANLEER_LIM"),
                                   ((301, 190, 1), "MC_LIM"), ((520, 513, 1), "MC_LIM")])
def test_2d_tiles_match_oracle(n, lim):
    """The 2D EMF and update tiles: narrow boxes of whole rows, one tile, remainders of
    a cell or a row; the larger tiles; a box past one round of blocks (two launches)."""
    import oracle
    vc, vs = ic.mhd_turbulence(n, 17)
    print(f"case n={n} {lim}", flush=True)
    g = StageUpdate(Definitions(dimensions=2, limiter=lim), RuntimeSetup(n=n))
    g.upload(vc, vs)
    res = g.run(3, 1e-3)
    gvc, gvs, _ = g.download()
    g.close()
    o = oracle.Oracle(phys="mhd", n=n, gamma=5 / 3, limiter=lim)
    o.set_state(vc, vs)
    assert res == o.run(3, 1e-3)
    ovc, ovs, _ = o.get_state()
    assert np.array_equal(gvc, ovc) and np.array_equal(gvs, ovs)
