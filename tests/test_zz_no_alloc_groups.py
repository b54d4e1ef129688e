"""ctpwa_nll_grad_noalloc at the limit of its scratch for a model evaluated in wave groups:
a handle within the contract (accumulators of every propagator times workgroups of 256 events)
is accepted, with the bits of ctpwa_nll_grad, however the kernel splits the events; one past it
is rejected."""
import re

import numpy as np
import pytest

from helpers import perturbed, plan_of, samples
from test_zz_no_alloc import _eval
from ctpwa_amd import _native
from ctpwa_amd import workloads as W

pytestmark = pytest.mark.gpu

MASSES = W.WORKLOADS["jpsi_kkpipi_wide"]["masses"]


def many_amplitudes():
    """the 149-amplitude cascade with 60 more K1 states in its two charge-conjugate chains and
    one free resonance parameter"""
    new = ["K1_x%d" % k for k in range(60)]
    text = W.JPSI_KKPIPI_WIDE.replace("[K1_1270, K1_1400, K1_1650]", "[K1_1270, K1_1400, K1_1650, " + ", ".join(new) + "]")
    text = re.sub(r", free: \[[^\]]*\]", "", text).replace("[1.253, 0.090]", "[1.253, 0.090], free: [0]")
    return text + "".join("  %s: {J: 1, P: 1, model: BWR, parameters: [%.3f, 0.12]}\n" % (x, 1.3 + 0.01 * k) for k, x in enumerate(new))


@pytest.mark.parametrize("n_ph,n_da,accepted", [(45_000, 5_000, True), (60_000, 5_000, True), (120_000, 5_000, False)])
def test_noalloc_limit_counts_the_contract(n_ph, n_da, accepted):
    # about 1270 accumulators: 262144 doubles hold some 200 workgroups of 256 to 384 events
    # (whole 128-event steps) and the totals
    plan = plan_of(many_amplitudes())
    assert plan.n_amp == 629
    p = perturbed(W.nominal_params(plan, 4), plan, 9)
    L = _native.lib()
    ph, da, _ = samples(n_ph, n_da, 0, 75, masses=MASSES)
    print("case no-alloc contract", n_ph, n_da, flush=True)
    h = _native.Handle(plan.to_text(), ph, da, None, device=0)
    if accepted:
        ref = _eval(h, L.ctpwa_nll_grad, p)
        assert np.all(np.isfinite(ref))
        assert np.array_equal(_eval(h, L.ctpwa_nll_grad_noalloc, p), ref)
    else:
        with pytest.raises(_native.NativeError, match="scratch"):
            _eval(h, L.ctpwa_nll_grad_noalloc, p)
    h.close()
