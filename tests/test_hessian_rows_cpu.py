"""Source of the Hessian's rows form: phase-space events have no u row, and only models of small
blocks branch around its stores (a branch at every store of a long block cuts its code up)."""
import pytest

from helpers import plan_of
from test_gpu_group_counts import chains
from ctpwa_amd import _native
from ctpwa_amd import workloads as W


@pytest.mark.parametrize("text,branches", [
    (W.JPSI_3PI, True),                # blocks of one amplitude and two free parameters
    (chains("k1p_rho"), False),        # two blocks of four amplitudes and four free parameters
    (chains("k1p"), False),            # three of them
    (W.JPSI_KKPIPI, False),            # 20 amplitudes
], ids=["three pions", "8 amplitudes", "12 amplitudes", "20 amplitudes"])
def test_u_stores_branch_in_small_blocks_only(text, branches):
    src = _native.generate_hessian_source(plan_of(text).to_text(), "mixed")
    assert "at(Uk + " in src
    assert ("if (cls != 0) at(Uk + " in src) == branches
