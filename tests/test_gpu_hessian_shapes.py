"""Hessian and amplitude Gram at the edges of their kernels' shapes, against the oracle.

The generated kernel has a fused form (FP64, up to 64 columns: Jacobian tile in LDS, matrix
cores in the same kernel) and a row form (FP32 Jacobian, or more columns), one to eight wave
groups, and three classes of events per launch; the row form's Gram has one kernel up to 64
columns and one for more (panels of 128).  The cases are one event, 64-event steps less or
more by one event, several steps with a partial last one, weights per event, three
polarisations (nothing folded), and several passes (a small row buffer).

Tolerances, relative to the largest element: 1e-6 (FP64) as in the other Hessian tests; 1e-5
in the mixed form, whose FP32 inputs (6e-8) enter divided by the square of |S| over the sum
of |v A|, some 1e-1 at the worst of these few events.  Gram: 1e-10 and 1e-6, as for the other
post-fit outputs.
"""
import numpy as np
import pytest
import torch

from helpers import perturbed, plan_of, rel, samples
from ctpwa_amd import workloads as W

pytestmark = pytest.mark.gpu

TEXTS = {n: W.WORKLOADS[n]["config"] for n in W.WORKLOADS}
TEXTS["three_pol"] = TEXTS["jpsi_3pi"].replace("polarization: [1, -1]", "polarization: [1, 0, -1]")


@pytest.mark.parametrize("model,precision,n3,weighted,jbytes", [
    ("jpsi_rho", "fp64", (1, 1, 1), False, None),
    ("jpsi_3pi", "fp64", (1, 1, 0), False, None),
    ("jpsi_3pi", "fp64", (64, 63, 65), True, None),
    ("jpsi_3pi", "fp64", (70_001, 193, 1), True, None),
    ("jpsi_3pi", "mixed", (65, 63, 31), True, None),
    ("jpsi_3pi", "mixed", (20_011, 9_001, 4_001), True, 1 << 20),
    ("three_pol", "fp64", (129, 127, 64), False, None),
    ("three_pol", "mixed", (129, 127, 64), True, None),
    ("jpsi_kkpipi", "fp64", (4_001, 129, 33), True, None),
    ("jpsi_kkpipi", "mixed", (257, 129, 33), False, None),
    ("jpsi_kkpipi_wide", "fp64", (1, 65, 0), False, None),
    ("jpsi_kkpipi_wide", "fp64", (1_500, 300, 33), True, 1 << 21),
    ("jpsi_kkpipi_wide", "mixed", (301, 129, 17), True, None),
])
def test_hessian_and_gram_shapes(model, precision, n3, weighted, jbytes, oracle_lib, monkeypatch):
    from ctpwa_amd import _native
    if jbytes:
        monkeypatch.setenv("CTPWA_HESS_JBYTES", str(jbytes))
    plan = plan_of(TEXTS[model])
    four = model.startswith("jpsi_kkpipi")
    ph, da, bk = samples(*n3, 57, masses=W.WORKLOADS[model]["masses"] if four else None)
    rng = np.random.default_rng(11)
    wd = rng.uniform(0.5, 1.5, n3[1]) if weighted else None
    wb = rng.uniform(0.2, 1.0, n3[2]) if n3[2] else None
    print("case shapes", model, precision, n3, weighted, jbytes, flush=True)
    h = _native.Handle(plan.to_text(), ph, da, bk, None, wd, wb, precision=precision)
    O = oracle_lib.Oracle(plan.to_text(), 4 if four else 3, ph, da, bk, w_data=wd, w_bkg=wb)
    p = perturbed(W.nominal_params(plan, None if model == "jpsi_rho" else 1), plan, 13, 0.1)
    _, _, Ho = O.hessian(p)
    t = torch.tensor(p, dtype=torch.float64, device="cuda")
    H = torch.empty((h.n_params, h.n_params), dtype=torch.float64, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    tol, gtol = (1e-6, 1e-10) if precision == "fp64" else (1e-5, 1e-6)
    for _ in range(2):                                # the second call reuses the buffers
        H.fill_(float("nan"))
        h.hessian(t.data_ptr(), H.data_ptr(), s)
        got = H.cpu().numpy()
        assert rel(got, Ho) <= tol
        assert np.array_equal(got, got.T)
    for cls in range(3 if n3[2] else 2):
        A = O.amplitudes(p, cls).reshape(-1, plan.n_amp)
        Q = A.conj().T @ A
        G = torch.full((plan.n_amp, plan.n_amp, 2), float("nan"), dtype=torch.float64, device="cuda")
        h.amplitude_gram(t.data_ptr(), cls, G.data_ptr(), s)
        g = G.cpu().numpy()
        assert np.max(np.abs(g[..., 0] + 1j * g[..., 1] - Q)) <= gtol * np.max(np.abs(Q)), cls
    h.close()
