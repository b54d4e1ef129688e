"""The Gram of up to 64 columns (Hessians of the mixed form, and of FP64 models whose many
polarisations do not fit the fused form) where its last tile has columns of its own and missing
ones, and its last slab rows: one to four tiles, row counts around a slab of 16 or 32 rows, two
classes one behind the other.  Against the oracle, tolerances as for the other Hessian shapes:
1e-6 (FP64), 1e-5 (FP32 rows) of the largest element.
"""
import numpy as np
import pytest
import torch

from helpers import perturbed, plan_of, rel, samples
from ctpwa_amd import workloads as W

pytestmark = pytest.mark.gpu


def three_pions(rhos, pol="[1, -1]"):
    """the three-pion model with this many rho states per charge: 3 rhos + 1 amplitudes and
    2 rhos + 4 free parameters"""
    names = ["rho770", "rho1450", "rho1700"][:rhos] + ["rho_x%d" % k for k in range(3, rhos)]
    text = W.JPSI_3PI.replace("[rho770, rho1450, rho1700]", "[" + ", ".join(names) + "]")
    text = text.replace("polarization: [1, -1]", "polarization: " + pol)
    return text + "".join("  rho_x%d: {J: 1, P: -1, model: BWR, parameters: [%.2f, 0.2], free: [0, 1]}\n" % (k, 1.0 + 0.1 * k)
                          for k in range(3, rhos))


MANY = "[" + ", ".join(["1", "0", "-1"][k % 3] for k in range(12)) + "]"


@pytest.mark.parametrize("rhos,pol,precision,n3", [
    (1, "[1, -1]", "mixed", (17, 1, 15)),
    (2, "[1, -1]", "mixed", (31, 33, 16)),
    (3, "[1, -1]", "mixed", (1_025, 1, 33)),
    (4, "[1, -1]", "mixed", (1, 65, 31)),
    (4, "[1, -1]", "mixed", (4_099, 1_027, 0)),
    (5, "[1, -1]", "mixed", (129, 63, 1)),
    (5, "[1]", "mixed", (33, 31, 17)),
    (1, MANY, "fp64", (15, 17, 1)),
    (3, MANY, "fp64", (1, 33, 64)),
    (4, MANY, "fp64", (131, 65, 0)),
])
def test_columns_and_rows_past_the_end(rhos, pol, precision, n3, oracle_lib):
    from ctpwa_amd import _native
    plan = plan_of(three_pions(rhos, pol))
    assert plan.n_amp == 3 * rhos + 1
    ph, da, bk = samples(*n3, 61)
    wb = np.random.default_rng(2).uniform(0.2, 1.0, n3[2]) if n3[2] else None
    print("case gram tails", rhos, pol, precision, n3, flush=True)
    h = _native.Handle(plan.to_text(), ph, da, bk, None, None, wb, precision=precision)
    O = oracle_lib.Oracle(plan.to_text(), 3, ph, da, bk, w_bkg=wb)
    p = perturbed(W.nominal_params(plan, 1), plan, 13, 0.1)
    _, _, Ho = O.hessian(p)
    t = torch.tensor(p, dtype=torch.float64, device="cuda")
    H = torch.full((h.n_params, h.n_params), float("nan"), dtype=torch.float64, device="cuda")
    h.hessian(t.data_ptr(), H.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert rel(H.cpu().numpy(), Ho) <= (1e-6 if precision == "fp64" else 1e-5)
    h.close()
