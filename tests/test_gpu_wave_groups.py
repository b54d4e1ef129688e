"""The fused kernel's wave groups (models of more than 24 amplitudes: the waves of a
workgroup share 64 events and each evaluates its own blocks) against the oracle.

Sizes sit at the edges of its split: one event, a workgroup's iteration less or more by one
event, several workgroups of several iterations with a partial last one.  Models: the
149-amplitude cascade in both storage forms, with a weight per background event, with three
polarisations (nothing folded), and with a Custom lineshape in one group.  Tolerances: the
fused kernel's usual bars, 1e-9 (NLL) and 1e-7 (gradient) of the oracle, 1e-6 and 1e-5 in
the mixed form (FP32 storage), relative to the larger of the value and the sum of the terms'
magnitudes the NLL is the difference of (n_data x 10, since |ln I| stays below 10 here).
"""
import numpy as np
import pytest
import torch

from helpers import perturbed, plan_of, rel, samples
from ctpwa_amd import workloads as W

MASSES = W.WORKLOADS["jpsi_kkpipi_wide"]["masses"]
F0_1500 = "  f0_1500:  {J: 0, P: 1, model: BWR, parameters: [1.506, 0.112], free: [0]}"
TEXTS = {
    "wide": W.JPSI_KKPIPI_WIDE,
    "three_pol": W.JPSI_KKPIPI_WIDE.replace("polarization: [1, -1]", "polarization: [1, 0, -1]"),
    "custom": W.JPSI_KKPIPI_WIDE.replace(F0_1500, '  f0_1500:  {J: 0, P: 1, model: Custom, paramValues: [1.506, 0.112], '
                                                  'paramNames: [p0, p1], free: [0], expression: "BWR(p0, p1, 0, 3.0)"}'),
}


def test_groups_cover_the_model_once():
    """Every amplitude's accumulators appear in exactly one group's code, each group's code
    in one branch, and the model's equal propagators are evaluated once per group."""
    import re
    from ctpwa_amd import _native
    plan = plan_of("jpsi_kkpipi_wide")
    src = _native.generate_source(plan.to_text(), "fp64")
    bodies = re.split(r"__device__ __forceinline__ void eval_g(\d+)\(", src)[1::2], \
        re.split(r"__device__ __forceinline__ void eval_g\d+\(", src)[1:]
    assert bodies[0] == [str(g) for g in range(8)]
    seen = []
    for k, text in enumerate(bodies[1]):
        text = text[:text.index("\n}\n")]
        seen += [int(a) for a in re.findall(r"double ax(\d+)r = 0\.0", text)]
        assert text.count("__syncthreads();") == 2           # one in the loop, one before the reduction
    assert sorted(seen) == list(range(plan.n_amp))
    assert plan_of("jpsi_3pi").n_amp <= 24
    assert "eval_g0" not in _native.generate_source(plan_of("jpsi_3pi").to_text(), "fp64")


@pytest.mark.gpu
@pytest.mark.parametrize("model,precision,n3,weighted", [
    ("wide", "fp64", (1, 1, 0), False),
    ("wide", "fp64", (64, 63, 65), True),
    ("wide", "mixed", (129, 127, 1), True),
    ("wide", "mixed", (40_001, 7_000, 130), False),
    ("three_pol", "fp64", (1_000, 200, 65), True),
    ("custom", "fp64", (1_000, 193, 64), False),
])
def test_wave_groups_against_oracle(oracle_lib, model, precision, n3, weighted):
    from ctpwa_amd import _native
    plan = plan_of(TEXTS[model])
    assert plan.n_amp > 24
    ph, da, bk = samples(*n3, 91, masses=MASSES)
    w = None
    if n3[2]:
        w = np.random.default_rng(5).uniform(0.5, 1.0, n3[2]) if weighted else np.full(n3[2], 0.8)
    print("case wave groups", model, precision, n3, weighted, flush=True)
    h = _native.Handle(plan.to_text(), ph, da, bk, None, None, w, precision=precision)
    O = oracle_lib.Oracle(plan.to_text(), 4, ph, da, bk, w_bkg=w)
    p = perturbed(W.nominal_params(plan, 4), plan, 5)
    nll_o, g_o = O.nll_grad(p)
    t = torch.tensor(p, dtype=torch.float64, device="cuda")
    out = torch.empty(1 + h.n_params, dtype=torch.float64, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    h.nll_grad(t.data_ptr(), out.data_ptr(), s)
    got = out.cpu().numpy()
    tol = (1e-9, 1e-7) if precision == "fp64" else (1e-6, 1e-5)
    assert abs(got[0] - nll_o) <= tol[0] * max(abs(nll_o), 10.0 * n3[1])
    assert rel(got[1:], g_o) <= tol[1]
    # the grouped launch of a batch gives the same bits
    b = _native.Batch(2)
    out2 = torch.zeros_like(out)
    b.nll_grad([h], [t.data_ptr()], [out2.data_ptr()], s)
    assert np.array_equal(out2.cpu().numpy(), got)
    b.close()
    h.close()
