"""GPU: downloads of the active layout, chunked through pinned buffers, against
the array layout's (element by element on the host), around the sizes where a
transfer changes its form: direct up to 2^17 doubles, then slots of an eighth of
the state, then of 16 MiB; gathered when the state is FP32 or padded."""
import ctypes as C

import numpy as np
import pytest

from gpluto_dev_amd import _lib, ic
from gpluto_dev_amd.stage import Definitions, RuntimeSetup, StageUpdate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,physics,precision,sides", [
    ((18, 17, 16), "MHD", "fp64", ()),               # below 2^17 doubles: direct
    ((23, 19, 41), "MHD", "fp64", ()),               # above: slots of an eighth
    ((11, 10, 9), "MHD", "mixed", ()),
    ((37, 41, 29), "MHD", "mixed", ()),
    ((19, 21, 23), "MHD", "fp64", ("outflow", "reflective", "periodic", "periodic", "outflow", "outflow")),
    ((19, 21, 23), "MHD", "mixed", ("outflow", "reflective", "periodic", "periodic", "outflow", "outflow")),
    ((130, 121, 117), "MHD", "fp64", ()),            # slots of 16 MiB, helper threads
    ((301, 77, 1), "MHD", "fp64", ()),
    ((301, 77, 1), "MHD", "mixed", ("outflow", "outflow", "reflective", "reflective", "periodic", "periodic")),
    ((61, 1, 1), "HD", "fp64", ()),
    ((151, 149, 33), "HD", "fp64", ("outflow",)*6)])
def test_active_layout_matches_array_layout(n, physics, precision, sides):
    nx, ny, nz = n
    dims = 1 if ny == 1 else 2 if nz == 1 else 3
    hd = physics == "HD"
    print(f"case {n} {physics} {precision} {sides}", flush=True)
    g = StageUpdate(Definitions(physics=physics, dimensions=dims),
                    RuntimeSetup(n=n, sides=sides, solver="hllc" if hd else "hlld"), precision=precision)
    if hd:
        g.upload(ic.hd_blast(n, 3))
    else:
        rng = np.random.default_rng(5)
        vc = 1.0 + 0.1*rng.random((8, nz, ny, nx))
        g.upload(vc, 0.1*rng.random((dims, nz, ny, nx)))
    g.run(2, 1e-5)
    vc, vs, uc = g.download()
    again = g.download()
    assert np.array_equal(vc, again[0]) and np.array_equal(uc, again[2])
    # a subset: only one face component
    if not hd:
        one = np.zeros((nz, ny, nx))
        ptr = (C.c_void_p*3)(None, one.ctypes.data, None)
        _lib.check(g._L.gpl_download(g._h, None, ptr, None, _lib.GPL_LAYOUT_ACTIVE), "gpl_download")
        assert np.array_equal(one, vs[1])
    gh = [2 if d < dims else 0 for d in range(3)]
    t = [n[d] + 2*gh[d] for d in range(3)]
    nv = 5 if hd else 8
    av, au = np.zeros((nv, t[2], t[1], t[0])), np.zeros((nv, t[2], t[1], t[0]))
    faces = [np.zeros((t[2] + (d == 2), t[1] + (d == 1), t[0] + (d == 0))) for d in range(3)]
    ptr = None if hd else (C.c_void_p*3)(*[f.ctypes.data for f in faces])
    _lib.check(g._L.gpl_download(g._h, av.ctypes.data, ptr, au.ctypes.data, _lib.GPL_LAYOUT_ARY4D),
               "gpl_download")
    g.close()
    box = (slice(gh[2], gh[2] + nz), slice(gh[1], gh[1] + ny), slice(gh[0], gh[0] + nx))
    assert np.array_equal(vc, av[(slice(None),) + box]) and np.array_equal(uc, au[(slice(None),) + box])
    for d in range(0 if hd else dims):
        assert np.array_equal(vs[d], faces[d][box]), f"face component {d}"
