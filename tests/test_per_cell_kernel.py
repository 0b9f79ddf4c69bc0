"""The per-cell kernel of the :ref GLM steps (pmf_set_ct_kernel; otherwise the fused kernel runs
most of them): the repository's parity tests of :ref steps against the oracle, the fixtures, the
known answers and the fused kernel, with every GLM state on the per-cell kernel."""
import pytest

import pmfmhd as M
from test_fullsize import (state256, test_fused_and_per_cell_glm_steps_agree,  # noqa: F401
                           test_mach15_512_fused_equals_per_cell_and_keeps_the_ledger)
from test_golden import test_library_ct_and_coupled_steps_match_fixtures, test_library_steps_match_fixtures  # noqa: F401
from test_gpu_parity import (test_config1_50_steps_float32_vs_float64_oracle,  # noqa: F401
                             test_config1_one_step_float32_vs_float32_oracle,
                             test_evolve_alfven_float32_matches_recorded,
                             test_fused_boundaries_float32_match_float32_oracle_and_ref_kernel,
                             test_fused_float32_config1_gates, test_fused_step_equals_the_per_cell_step_bitwise,
                             test_ref_step_boundaries_match_oracle, test_ref_step_float64_matches_oracle)
from test_mach15 import (test_mach15_float32_one_step_matches_float32_oracle,  # noqa: F401
                         test_mach15_float64_ten_steps_match_oracle)
from test_sources import (test_drag_ref_and_cube_agree_float32, test_drag_step_matches_oracle_float64,  # noqa: F401
                          test_radiation_float32_against_float32_oracle,
                          test_radiation_step_with_tracking_matches_oracle_float64,
                          test_ref_drag_with_a_moving_target_and_boundaries_matches_oracle)

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def per_cell(monkeypatch):
    allocate = M.allocate_state

    def on_the_per_cell_kernel(*args, **kw):
        s = allocate(*args, **kw)
        if not s.uses_ct:
            M.set_ct_kernel(s, True)
        return s

    monkeypatch.setattr(M, "allocate_state", on_the_per_cell_kernel)
