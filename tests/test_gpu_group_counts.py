"""The fused kernel in two to seven wave groups (25 to 133 amplitudes), against the oracle,
and the number of its workgroups.

The models are the 149-amplitude cascade with some of its decay chains.  Tolerances as for
the eight groups of the whole model: 1e-9 (NLL) and 1e-7 (gradient) of the oracle, the NLL
relative to the larger of its value and ten per data event (it is a difference of sums of
logarithms below 10).
"""
import re

import numpy as np
import pytest
import torch

from helpers import perturbed, plan_of, rel, samples
from ctpwa_amd import workloads as W

pytestmark = pytest.mark.gpu

MASSES = W.WORKLOADS["jpsi_kkpipi_wide"]["masses"]


def chains(*names):
    """the 149-amplitude configuration with these decay chains only"""
    head, rest = W.JPSI_KKPIPI_WIDE.split("DecayChains:\n")
    body, tail = rest.split("Resonances:\n")
    parts = re.split(r"(?m)^(  \w+:\n)", body)[1:]
    kept = [n + b for n, b in zip(parts[::2], parts[1::2]) if n.strip(" :\n") in names]
    assert len(kept) == len(names)
    return head + "DecayChains:\n" + "".join(kept) + "Resonances:\n" + tail


MODELS = {
    2: chains("k1p", "f2ppipi"),
    3: chains("k1p", "k1m", "k1p_rho", "k1m_rho"),
    4: chains("k1p", "kstkst"),
    5: chains("k1p", "k1m", "kstkst"),
    6: chains("k1p", "k1m", "k1p_rho", "kstkst", "f2ppipi"),
    7: chains("k1p", "k1m", "k1p_rho", "k1m_rho", "phipipi", "f2ppipi", "kstkst"),
}


def groups(h):
    return len(set(re.findall(r"void eval_g(\d+)\(", h.kernel_source())))


@pytest.mark.parametrize("ng", sorted(MODELS))
def test_group_counts_against_oracle(ng, oracle_lib):
    from ctpwa_amd import _native
    plan = plan_of(MODELS[ng])
    ph, da, bk = samples(1_283, 321, 65, 171, masses=MASSES)
    w = np.random.default_rng(3).uniform(0.5, 1.0, 65)
    print("case group count", ng, plan.n_amp, flush=True)
    h = _native.Handle(plan.to_text(), ph, da, bk, None, None, w)
    assert groups(h) == ng
    O = oracle_lib.Oracle(plan.to_text(), 4, ph, da, bk, w_bkg=w)
    p = perturbed(W.nominal_params(plan, 4), plan, 5)
    nll_o, g_o = O.nll_grad(p)
    t = torch.tensor(p, dtype=torch.float64, device="cuda")
    out = torch.empty(1 + h.n_params, dtype=torch.float64, device="cuda")
    h.nll_grad(t.data_ptr(), out.data_ptr(), torch.cuda.current_stream().cuda_stream)
    got = out.cpu().numpy()
    assert abs(got[0] - nll_o) <= 1e-9 * max(abs(nll_o), 10.0 * len(da))
    assert rel(got[1:], g_o) <= 1e-7
    h.close()


@pytest.mark.parametrize("ng", [2, 3])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_few_groups_fill_the_simds(ng, precision):
    """With enough events there is a wave for each of a CU's four SIMDs (less the rounding of
    the classes' shares), also where a workgroup has only two or three."""
    from ctpwa_amd import _native
    plan = plan_of(MODELS[ng])
    ph, da, _ = samples(130_000, 20_000, 0, 173, masses=MASSES)
    print("case group fill", ng, precision, flush=True)
    h = _native.Handle(plan.to_text(), ph, da, None, precision=precision)
    waves = h.layout()["n_workgroups"] * groups(h)
    assert waves >= 0.9 * 4 * torch.cuda.get_device_properties(0).multi_processor_count
    h.close()
