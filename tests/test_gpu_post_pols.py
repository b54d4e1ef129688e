"""Per-event post-fit outputs for one to five polarisation states and at the edges of a
workgroup (one event, 63, 64 and 65), against the oracle's amplitudes.

Up to four polarisations the kernels know the count at compile time, beyond that they take
any count, or groups of four (partial amplitudes).  Tolerances, relative to the largest
value: FP64 1e-10, mixed 1e-6 (FP32 inputs), times ten for sums over waves, as in the other
tests of these outputs.
"""
import numpy as np
import pytest
import torch

from helpers import perturbed, plan_of, samples
from ctpwa_amd import results as R
from ctpwa_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pol,precision,n", [
    ("[1]", "fp64", 1), ("[1, -1]", "fp64", 63), ("[1, -1]", "mixed", 65), ("[1, 0, -1]", "fp64", 64),
    ("[1, 0, -1]", "mixed", 129), ("[1, 0, -1, 1]", "fp64", 65), ("[1, 0, -1, 1, 0]", "fp64", 65),
])
def test_post_fit_outputs(pol, precision, n, oracle_lib):
    from ctpwa_amd import _native
    plan = plan_of(W.JPSI_3PI.replace("polarization: [1, -1]", "polarization: " + pol))
    ph, da, _ = samples(200, n, 0, 23)
    print("case post", pol, precision, n, flush=True)
    h = _native.Handle(plan.to_text(), ph, da, None, precision=precision)
    O = oracle_lib.Oracle(plan.to_text(), 3, ph, da)
    p = perturbed(W.nominal_params(plan, 1), plan, 17)
    t = torch.tensor(p, dtype=torch.float64, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    tol = 1e-10 if precision == "fp64" else 1e-6
    A = O.amplitudes(p, 1)
    npol, v, nb = A.shape[1], R.coupling_vector(plan, p), len(plan.blocks)
    assert npol == pol.count(",") + 1
    P = np.stack([np.einsum("epa,a->ep", A[:, :, B.site:B.site + B.nsl], v[B.site:B.site + B.nsl]) for B in plan.blocks])
    top = np.max(np.abs(P))
    out = torch.full((nb, n, npol, 2), float("nan"), dtype=torch.float64, device="cuda")
    h.partial_amplitudes(t.data_ptr(), 1, out.data_ptr(), s)
    g = out.cpu().numpy()
    assert np.max(np.abs(g[..., 0] + 1j * g[..., 1] - P)) <= 10 * tol * top
    out = torch.full((nb + 1, n), float("nan"), dtype=torch.float64, device="cuda")
    h.partial_intensities(t.data_ptr(), 1, out.data_ptr(), s)
    g, I = out.cpu().numpy(), np.sum(np.abs(np.sum(P, axis=0)) ** 2, axis=1)
    scale = np.max(np.sum(np.abs(P), axis=0)) ** 2 * npol
    assert np.max(np.abs(g[:nb] - np.sum(np.abs(P) ** 2, axis=2))) <= 10 * tol * scale
    assert np.max(np.abs(g[nb] - I)) <= 10 * tol * scale
    out = torch.full((n,), float("nan"), dtype=torch.float64, device="cuda")
    h.intensity(t.data_ptr(), 1, out.data_ptr(), s)
    assert np.max(np.abs(out.cpu().numpy() - I)) <= 10 * tol * scale
    out = torch.full((n, npol, plan.n_amp, 2), float("nan"), dtype=torch.float64, device="cuda")
    h.amplitudes(t.data_ptr(), 1, out.data_ptr(), s)
    g = out.cpu().numpy()
    assert np.max(np.abs(g[..., 0] + 1j * g[..., 1] - A)) <= tol * np.max(np.abs(A))
    h.close()
