"""Events per pass of the Hessian's rows form: their byte offsets (eight bytes per event) are
32-bit numbers in the generated kernel, so no row budget may allow 2^29 events of a class or
more.  The workspace estimate shows it: two columns of weights (16 bytes) and, for one amplitude
and two parameters, six FP32 and four FP64 columns per event."""
import pytest

from helpers import plan_of
from ctpwa_amd import _native


@pytest.mark.parametrize("jbytes", [None, 1 << 36, 1 << 45])
def test_pass_is_bounded_whatever_the_budget(jbytes, monkeypatch):
    if jbytes:
        monkeypatch.setenv("CTPWA_HESS_JBYTES", str(jbytes))
    n = 1 << 31
    plan = plan_of("jpsi_rho")
    assert plan.n_amp == 1
    text = plan.to_text()
    need = _native.lib().ctpwa_hessian_workspace_bytes(text.encode(), n, n, 0)
    per_event = 2 * 6 * 4 + 4 * 8 + 2 * 8
    assert 0 < need < (1 << 29) * per_event
