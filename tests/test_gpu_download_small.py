"""GPU: downloads in the active layout at the line between one launch (states of
at most 2^17 doubles, Uc included) and chunks, against the array layout."""
import numpy as np
import pytest

import test_gpu_download
from gpluto_dev_amd import _lib, ic
from gpluto_dev_amd.stage import Definitions, RuntimeSetup, StageUpdate

pytestmark = pytest.mark.gpu
SIDES = ("outflow", "reflective", "periodic", "periodic", "outflow", "outflow")


@pytest.mark.parametrize("n,physics,precision,sides", [
    ((3, 1, 1), "HD", "fp64", ()),
    ((13107, 1, 1), "HD", "fp64", ()), ((13108, 1, 1), "HD", "fp64", ()),            # 131070, 131080 doubles
    ((2427, 3, 1), "MHD", "mixed", ()), ((1821, 4, 1), "MHD", "mixed", SIDES),       # 131058, 131112
    ((19, 33, 11), "MHD", "fp64", SIDES), ((19, 11, 34), "MHD", "mixed", ()),        # 131043, 135014
    ((24, 24, 24), "MHD", "mixed", ()), ((24, 24, 24), "MHD", "fp64", SIDES)])       # three chunks
def test_small_states(n, physics, precision, sides):
    test_gpu_download.test_active_layout_matches_array_layout(n, physics, precision, sides)


@pytest.mark.parametrize("n", [(3, 1, 1), (61, 17, 1), (20, 20, 20)])
def test_vc_of_a_small_hd_state(n):
    """Vc by itself, one array on the device, against Vc beside Uc."""
    dims = 1 if n[1] == 1 else 2 if n[2] == 1 else 3
    g = StageUpdate(Definitions(physics="HD", dimensions=dims), RuntimeSetup(n=n, solver="hllc"))
    g.upload(ic.hd_blast(n, 3))
    for _ in range(2):                               # 1D: both buffers
        g.run(1, 1e-5)
        vc = np.zeros((5, n[2], n[1], n[0]))
        _lib.check(g._L.gpl_download(g._h, vc.ctypes.data, None, None, _lib.GPL_LAYOUT_ACTIVE), "gpl_download")
        assert np.array_equal(vc, g.download()[0]) and vc[0].min() > 0
    g.close()
