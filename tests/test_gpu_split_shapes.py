"""Hessian and amplitude Gram of 25 to 107 amplitudes against the oracle: the panel Gram with a
last panel of one to eight tiles (columns 129 to 258 of the Jacobian, 112 to 236 of u), a wide
Jacobian with a narrow u, sets of amplitudes with a Custom lineshape, with three and with twelve
polarisations, and the fused and narrow forms of models of more than 24 amplitudes without free
resonance parameters.

Tolerances as for the other Hessian shapes: 1e-6 (FP64), 1e-5 (mixed) of the largest element;
Gram 1e-10 and 1e-6.
"""
import re

import numpy as np
import pytest
import torch

from helpers import perturbed, plan_of, rel, samples
from test_gpu_group_counts import MASSES, chains
from ctpwa_amd import workloads as W

pytestmark = pytest.mark.gpu

F0 = "  f0_1500:  {J: 0, P: 1, model: BWR, parameters: [1.506, 0.112], free: [0]}"
CUSTOM = '  f0_1500:  {J: 0, P: 1, model: Custom, paramValues: [1.506, 0.112], paramNames: [p0, p1], free: [0], ' \
         'expression: "BWR(p0, p1, 0, 3.0)"}'


def states(text, npol):
    return text.replace("polarization: [1, -1]", "polarization: [" + ", ".join(["1", "0", "-1"][k % 3] for k in range(npol)) + "]")


def fixed(text):
    return re.sub(r", +free: \[[^\]]*\]", "", text)


CASES = {
    # name: configuration, amplitudes, free resonance parameters
    "tiles_5_4": (chains("k1p_rho", "phipipi"), 25, 14),
    "tiles_8_7": (chains("k1p", "k1m", "phipipi"), 41, 18),
    "tiles_9_8": (chains("k1p", "phipipi", "k2kst"), 50, 22),
    "tiles_10_9": (chains("k1p_rho", "kstkst"), 65, 12),
    "tiles_12_11": (chains("phipipi", "kstkst"), 74, 16),
    "tiles_14_14": (chains("k1p", "k1p_rho", "kstkst", "k2kst"), 98, 14),
    "tiles_15_13": (chains("k1p", "k1p_rho", "f2ppipi", "kstkst"), 91, 22),
    "tiles_17_15": (chains("k1p", "phipipi", "kstkst", "k2kst"), 107, 22),
    "custom": (chains("k1p", "phipipi", "f2ppipi").replace(F0, CUSTOM), 43, 20),
    "three_states": (states(chains("k1p", "phipipi"), 3), 29, 18),
    "twelve_states": (states(chains("k1p", "phipipi"), 12), 29, 18),
    "fixed": (fixed(chains("k1p", "f2ppipi")), 26, 0),
}


@pytest.mark.parametrize("case,precision,n3", [
    ("tiles_5_4", "fp64", (65, 33, 17)), ("tiles_5_4", "mixed", (31, 65, 0)),
    ("tiles_8_7", "fp64", (63, 129, 1)), ("tiles_9_8", "fp64", (129, 64, 0)), ("tiles_9_8", "mixed", (129, 65, 31)),
    ("tiles_10_9", "fp64", (17, 33, 0)), ("tiles_12_11", "mixed", (65, 15, 17)), ("tiles_14_14", "fp64", (33, 65, 0)),
    ("tiles_15_13", "fp64", (129, 31, 16)), ("tiles_17_15", "mixed", (63, 33, 1)),
    ("custom", "fp64", (129, 65, 17)), ("custom", "mixed", (65, 33, 0)),
    ("three_states", "fp64", (129, 65, 33)), ("twelve_states", "mixed", (65, 17, 1)),
    ("fixed", "fp64", (129, 65, 1)), ("fixed", "mixed", (65, 64, 63)),
])
def test_hessian_and_gram(case, precision, n3, oracle_lib):
    from ctpwa_amd import _native
    text, namp, ntheta = CASES[case]
    plan = plan_of(text)
    assert (plan.n_amp, plan.n_theta) == (namp, ntheta)
    ph, da, bk = samples(*n3, 181, masses=MASSES)
    rng = np.random.default_rng(17)
    wd = rng.uniform(0.5, 1.5, n3[1])
    wb = rng.uniform(0.2, 1.0, n3[2]) if n3[2] else None
    print("case split shapes", case, precision, n3, flush=True)
    h = _native.Handle(plan.to_text(), ph, da, bk, None, wd, wb, precision=precision)
    O = oracle_lib.Oracle(plan.to_text(), 4, ph, da, bk, w_data=wd, w_bkg=wb)
    p = perturbed(W.nominal_params(plan, 1), plan, 13, 0.1)
    _, _, Ho = O.hessian(p)
    t = torch.tensor(p, dtype=torch.float64, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    H = torch.full((h.n_params, h.n_params), float("nan"), dtype=torch.float64, device="cuda")
    h.hessian(t.data_ptr(), H.data_ptr(), s)
    tol, gtol = (1e-6, 1e-10) if precision == "fp64" else (1e-5, 1e-6)
    assert rel(H.cpu().numpy(), Ho) <= tol
    A = O.amplitudes(p, 1).reshape(-1, plan.n_amp)
    Q = A.conj().T @ A
    G = torch.full((plan.n_amp, plan.n_amp, 2), float("nan"), dtype=torch.float64, device="cuda")
    h.amplitude_gram(t.data_ptr(), 1, G.data_ptr(), s)
    g = G.cpu().numpy()
    assert np.max(np.abs(g[..., 0] + 1j * g[..., 1] - Q)) <= gtol * np.max(np.abs(Q))
    h.close()
