"""Per-event post-fit outputs of more than four polarisation states, which the kernels take four
at a time: whole groups and a remainder, against the oracle as for fewer states."""
import pytest

import test_gpu_post_pols

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npol,precision,n", [(6, "fp64", 65), (8, "mixed", 64), (9, "fp64", 1)])
def test_outputs_four_states_at_a_time(npol, precision, n, oracle_lib):
    pol = "[" + ", ".join(["1", "0", "-1"][k % 3] for k in range(npol)) + "]"
    test_gpu_post_pols.test_post_fit_outputs(pol, precision, n, oracle_lib)
