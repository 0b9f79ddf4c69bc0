"""PPM CT steps form their edge EMFs in the step: the same bits as the step that fills the
workspace slots for the separate edge pass."""
import pytest

import test_gpu_parity as parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(33, 13, 17), (16, 12, 5), (8, 5, 3)])
@pytest.mark.parametrize("riemann", ["hlld", "hll", "llf"])
def test_ppm_step_forming_edges_equals_the_workspace_path(dims, riemann):
    parity.test_ct_step_forming_edges_in_kernel_equals_the_workspace_path(dims, "ppm", riemann)
