"""GPU: downloads in the active layout at the line between one launch (states of
at most 2^17 doubles, Uc included) and chunks, against the array layout."""
import pytest

import test_gpu_download

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
