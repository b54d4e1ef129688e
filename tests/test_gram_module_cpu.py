"""The amplitude Gram's generated module (compiled when a handle first needs it) is part of the
sources and compiles that can be checked without a device."""
import pytest

from helpers import plan_of
from ctpwa_amd import _native
from ctpwa_amd import workloads as W

CUSTOM = W.JPSI_3PI.replace("f2_1270: {J: 2, P: 1,  model: BWR, parameters: [1.275, 0.185], free: [0, 1]}",
                            'f2_1270: {J: 2, P: 1, model: Custom, paramValues: [1.275, 0.185], paramNames: [p0, p1], free: [0], '
                            'expression: "BWR(p0, p1, 2, 3.0)"}')


@pytest.mark.parametrize("text", [W.JPSI_RHO, W.JPSI_KKPIPI_WIDE, CUSTOM], ids=["rho", "wide", "custom"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_sources_hold_the_gram_module(text, precision):
    src = _native.generate_hessian_source(plan_of(text).to_text(), precision)
    head, gram = src.split("// ---- module: ctpwa_amp_gram ----")
    assert "ctpwa_hess_" in head and "ctpwa_amp_gram" not in head
    gram = gram.split("// ---- module: ctpwa_custom2 ----")[0]
    assert gram.count('extern "C" __global__') == 1 and " ctpwa_amp_gram(" in gram

