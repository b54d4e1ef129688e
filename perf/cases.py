"""The work a fit with this framework consists of, as cases that can be timed.

A fit evaluates the likelihood and its gradient a few hundred times (``getNLL`` and
``torch.autograd.grad``), takes Hessians for Newton steps and errors (``getHessian``), and
afterwards the amplitude Gram behind fit fractions (``getAmplitudeGram``) and per-event
quantities for projections (``getPartialAmplitudes``, ``getPartialIntensities``,
``getIntensity``).  Toy ensembles evaluate many likelihoods of one model together
(``Batch.nll_grad``).  The cases run these calls on the repository's own models from the
smallest fit (60 thousand events, launches and latency count) to the benchmark sizes
(3 million events, ten amplitudes) and the 149-amplitude model, in both storage forms.

``exact`` restates the likelihood in plain torch, in 64 bits and without this
repository's code: Clebsch-Gordan coefficients by the Racah sum, Wigner rotations as
exp(-i psi n.J), lineshapes and barriers per event, gradients by automatic differentiation.
"""
import itertools
import math

import numpy as np
import torch

import ctpwa_amd
from ctpwa_amd import _native, workloads
from ctpwa_amd.config import ConfigParser
from ctpwa_amd.model import build_plan

SQRT_S = 3.0969
RADIUS = 3.0                       # barrier radius of every vertex (the configurations' default)

# ---------------------------------------------------------------------------
# the models, as exact() and the samples need them
# ---------------------------------------------------------------------------
# resonance: lineshape, parameters, free parameters, Flatte channels


def _bwr(m, g, free=(0, 1)):
    return dict(shape="BWR", par=(m, g), free=free)


_F0 = dict(shape="Flatte", par=(0.99, 0.2, 0.4), free=(0, 1, 2), ch=((0.13957, 0.13957), (0.493677, 0.493677)))
_PI3 = dict(pip=0.13975, pim=0.13975, pi0=0.13495)
_KKPP = dict(Kp=0.493677, Km=0.493677, pip=0.13957, pim=0.13957)

# chain: name, decay steps (mother, daughter 1, daughter 2), intermediates with their
# (J, P) choices and the resonances of each
_RHOS = ["rho770", "rho1450", "rho1700"]


def _pair_chain(name, bachelor, tag, pair, jps):
    return (name, [("Jpsi", bachelor, tag), (tag,) + pair], [(tag, jps)])


def _k1_chain(name, spect, k1, k1_res, kst, kst_res, bach, pair):
    return (name, [("Jpsi", spect, k1), (k1,) + bach, (kst,) + pair],
            [(k1, [((1, 1), k1_res)]), (kst, [((1, -1), kst_res)])])


def _two_chain(name, a, pa, ja, b, pb, jb):
    return (name, [("Jpsi", a, b), (a,) + pa, (b,) + pb], [(b, jb), (a, ja)])


_KST = ["Kst892", "Kst1410", "Kst1680"]
_K1S = ["K1_1270", "K1_1400", "K1_1650"]
MODELS = {
    "jpsi_rho": dict(
        final=_PI3, chains=[_pair_chain("c0", "pi0", "R_pm", ("pip", "pim"), [((1, -1), ["rho770"])])],
        res=dict(rho770=_bwr(0.775, 0.149))),
    "jpsi_3pi": dict(
        final=_PI3,
        chains=[_pair_chain("c1", "pi0", "R_pm", ("pip", "pim"),
                            [((1, -1), _RHOS), ((0, 1), ["f0_980"]), ((2, 1), ["f2_1270"])]),
                _pair_chain("c1", "pip", "R_m0", ("pim", "pi0"), [((1, -1), _RHOS)]),
                _pair_chain("c1", "pim", "R_p0", ("pip", "pi0"), [((1, -1), _RHOS)])],
        res=dict(rho770=_bwr(0.775, 0.149), rho1450=_bwr(1.465, 0.40), rho1700=_bwr(1.72, 0.25),
                 f0_980=_bwr(0.99, 0.05), f2_1270=_bwr(1.275, 0.185))),
    "jpsi_kkpipi": dict(
        final=_KKPP,
        chains=[_k1_chain("k1p", "Km", "K1p", _K1S[:1], "Kst0", _KST[:1], ("Kst0", "pip"), ("Kp", "pim")),
                _k1_chain("k1m", "Kp", "K1m", _K1S[:1], "Kstb0", _KST[:1], ("Kstb0", "pim"), ("Km", "pip")),
                _two_chain("phipipi", "R_KK", ("Kp", "Km"), [((1, -1), ["phi1020"])], "R_pipi", ("pip", "pim"),
                           [((0, 1), ["f0_980"]), ((2, 1), ["f2_1270"])]),
                _two_chain("kstk2", "R_Kpim", ("Kp", "pim"), [((1, -1), ["Kst892"])], "R_Kmpip", ("Km", "pip"),
                           [((2, 1), ["K2st1430"])])],
        res=dict(K1_1270=_bwr(1.253, 0.090), Kst892=_bwr(0.8955, 0.0473), phi1020=_bwr(1.0195, 0.0045, ()),
                 f0_980=_F0, f2_1270=_bwr(1.275, 0.185), K2st1430=_bwr(1.4273, 0.100))),
    "jpsi_kkpipi_wide": dict(
        final=_KKPP,
        chains=[_k1_chain("k1p", "Km", "K1p", _K1S, "Kst0", _KST[:1], ("Kst0", "pip"), ("Kp", "pim")),
                _k1_chain("k1m", "Kp", "K1m", _K1S, "Kstb0", _KST[:1], ("Kstb0", "pim"), ("Km", "pip")),
                _k1_chain("k1p_rho", "Km", "K1pr", _K1S[1:], "R_pp", ["rho770"], ("Kp", "R_pp"), ("pip", "pim")),
                _k1_chain("k1m_rho", "Kp", "K1mr", _K1S[1:], "R_mm", ["rho770"], ("Km", "R_mm"), ("pip", "pim")),
                _two_chain("phipipi", "R_KK", ("Kp", "Km"), [((1, -1), ["phi1020"])], "R_pipi", ("pip", "pim"),
                           [((0, 1), ["f0_980", "f0_1500"]), ((1, -1), ["rho770", "rho1450"]), ((2, 1), ["f2_1270"])]),
                _two_chain("f2ppipi", "R_KK2", ("Kp", "Km"), [((2, 1), ["f2p_1525"])], "R_pipi2", ("pip", "pim"),
                           [((0, 1), ["f0_980", "f0_1500"]), ((1, -1), ["rho770", "rho1450"])]),
                _two_chain("kstkst", "R_Kpim", ("Kp", "pim"), [((1, -1), _KST)], "R_Kmpip", ("Km", "pip"),
                           [((1, -1), _KST), ((2, 1), ["K2st1430"]), ((0, 1), ["K0st1430"])]),
                _two_chain("k2kst", "R_K2pim", ("Kp", "pim"), [((2, 1), ["K2st1430"]), ((0, 1), ["K0st1430"])],
                           "R_Kstmpip", ("Km", "pip"), [((1, -1), _KST)])],
        res=dict(K1_1270=_bwr(1.253, 0.090), K1_1400=_bwr(1.403, 0.174), K1_1650=_bwr(1.650, 0.150),
                 Kst892=_bwr(0.8955, 0.0473), Kst1410=_bwr(1.414, 0.232), Kst1680=_bwr(1.718, 0.322, ()),
                 rho770=_bwr(0.775, 0.149), rho1450=_bwr(1.465, 0.40), phi1020=_bwr(1.0195, 0.0045, ()),
                 f2p_1525=_bwr(1.5174, 0.086), f0_980=_F0, f0_1500=_bwr(1.506, 0.112, (0,)),
                 f2_1270=_bwr(1.275, 0.185), K2st1430=_bwr(1.4273, 0.100), K0st1430=_bwr(1.425, 0.270, ()))),
}
# per event: SL tensors, stored polarisations, FP64-stored and narrowed invariants, amplitudes,
# propagators, free resonance parameters, partial waves
SHAPE = {
    "jpsi_rho": dict(nu=1, nps=1, inv64=1, inv32=1, amp=1, den=1, th=2, wave=1),
    "jpsi_3pi": dict(nu=4, nps=1, inv64=3, inv32=4, amp=10, den=10, th=10, wave=11),
    "jpsi_kkpipi": dict(nu=20, nps=1, inv64=6, inv32=11, amp=20, den=10, th=11, wave=5),
    "jpsi_kkpipi_wide": dict(nu=52, nps=1, inv64=8, inv32=19, amp=149, den=80, th=24, wave=40),
}


def _enumerate(name, fixed):
    """Topologies (nodes with their (S, L) waves), blocks, amplitudes and parameter slots of a
    model in the order of the configuration."""
    M = MODELS[name]
    final = list(M["final"])
    topos, blocks, slots, owner, amps = [], [], [], {}, []
    for cname, steps, inter in M["chains"]:
        for comb in itertools.product(*[[(tag, jp, rs) for jp, rs in jps] for tag, jps in inter]):
            jp = {tag: q for tag, q, _ in comb}
            jp["Jpsi"] = (1, -1)
            nodes = []
            mothers = [s[0] for s in steps]
            for mo, a, b in steps:
                (J, P), (j1, p1), (j2, p2) = [jp.get(x, (0, -1)) for x in (mo, a, b)]
                sl = [(S, L) for S in range(abs(j1 - j2), j1 + j2 + 1) for L in range(abs(J - S), J + S + 1)
                      if P == p1 * p2 * (-1) ** L]
                nodes.append(dict(mother=mo, d=(a, b), J=(J, j1, j2), sl=sl, lmin=min([L for _, L in sl], default=0)))
            combos = list(itertools.product(*[n["sl"] for n in nodes]))
            topos.append(dict(nodes=nodes, combos=combos, mothers=mothers))
            for rcombo in itertools.product(*[rs for _, _, rs in comb]):
                inst = {}
                for (tag, _, _), rn in zip(comb, rcombo):
                    if rn not in owner:
                        owner[rn] = {}
                        for p in (() if fixed else M["res"][rn]["free"]):
                            owner[rn][p] = len(slots)
                            slots.append((rn, p))
                    inst[tag] = rn
                key = "%s_%s" % (cname, comb[0][0]) + "".join("_%s[%s]" % (c[0], rn) for c, rn in zip(comb, rcombo))
                blocks.append(dict(topo=len(topos) - 1, res=inst, key=key, first=len(amps)))
                amps += [(len(blocks) - 1, c) for c in range(len(combos))]
    # coupling order: as the amplitudes where every chain has one wave, else by chain key
    n_of = {}
    for b, _ in amps:
        n_of[blocks[b]["key"]] = n_of.get(blocks[b]["key"], 0) + 1
    order = list(range(len(amps)))
    if any(n > 1 for n in n_of.values()):
        order = sorted(order, key=lambda a: (blocks[amps[a][0]]["key"], a))
    free_of = [0] * len(amps)
    for f, a in enumerate(order):
        free_of[a] = f
    init = [M["res"][rn]["par"][p] for rn, p in slots]
    return dict(final=final, mass=M["final"], res=M["res"], topos=topos, blocks=blocks, amps=amps, free_of=free_of,
                owner=owner, init=init, n=len(amps), nt=len(slots))


# ---------------------------------------------------------------------------
# samples: phase space, and data shaped by the model's resonance peaks
# ---------------------------------------------------------------------------
def _pdk(a, b, c):
    x = (a - b - c) * (a + b + c) * (a - b + c) * (a + b - c)
    return torch.sqrt(torch.clamp(x, min=0.0)) / (2.0 * a)


def _boost(p, beta):
    b2 = (beta * beta).sum(-1, keepdim=True)
    g = 1.0 / torch.sqrt(1.0 - b2)
    bp = (beta * p[..., 1:]).sum(-1, keepdim=True)
    E = p[..., :1]
    return torch.cat([g * (E + bp), p[..., 1:] + ((g - 1.0) / b2.clamp(min=1e-300) * bp + g * E) * beta], -1)


def _phase_space(gen, n, masses):
    """Uniform n-body phase space [n, k, 4] (E, px, py, pz): ordered uniform subsystem
    masses, accepted by the product of the breakup momenta."""
    k, dev = len(masses), gen.device
    cum = torch.tensor(np.cumsum(masses), dtype=torch.float64, device=dev)
    T = SQRT_S - sum(masses)
    wmax, lo, hi = 1.0, 0.0, T + masses[0]
    for i in range(1, k):
        lo, hi = lo + masses[i - 1], hi + masses[i]
        t = [torch.tensor(v, dtype=torch.float64) for v in (hi, lo, masses[i])]
        wmax *= float(_pdk(*t))
    out, have = [], 0
    while have < n:
        m = int(min(4_000_000, 3.5 * (n - have) + 4096))
        rnd = lambda *s: torch.rand(*s, generator=gen, dtype=torch.float64, device=dev)  # noqa: E731
        r = torch.sort(rnd(m, k - 2), dim=1).values
        one = torch.ones(m, 1, dtype=torch.float64, device=dev)
        Mk = cum + T * torch.cat([0 * one, r, one], 1)
        q = [_pdk(Mk[:, i], Mk[:, i - 1], torch.as_tensor(masses[i], dtype=torch.float64)) for i in range(1, k)]
        keep = torch.stack(q).prod(0) > rnd(m) * wmax
        Mk, q = Mk[keep], [x[keep] for x in q]
        m = Mk.shape[0]
        p = []
        for i in range(1, k):
            c, phi = 2.0 * rnd(m) - 1.0, 2.0 * math.pi * rnd(m)
            s = torch.sqrt(1.0 - c * c)
            v = q[i - 1][:, None] * torch.stack([s * torch.cos(phi), s * torch.sin(phi), c], 1)
            vec = lambda mass, w: torch.cat([torch.sqrt((w * w).sum(1, keepdim=True) + mass * mass), w], 1)  # noqa: E731
            if i == 1:
                p = [vec(masses[0], -v), vec(masses[1], v)]
            else:
                beta = -v / torch.sqrt(q[i - 1] ** 2 + Mk[:, i - 1] ** 2)[:, None]
                p = [_boost(x, beta) for x in p] + [vec(masses[i], v)]
        out.append(torch.stack(p, 1))
        have += m
    return torch.cat(out)[:n]


def _peaks(E, ev):
    """Sum of the model's squared Breit-Wigner factors over its two-body resonances; with three
    spinless particles times |p1 x p2|^2, since every amplitude of a spin-1 state to them
    vanishes on the boundary of the Dalitz plot.  Returns it with an upper bound."""
    w, seen = 0.2, set()
    for blk in E["blocks"]:
        for node in E["topos"][blk["topo"]]["nodes"][1:]:
            if all(d in E["final"] for d in node["d"]):
                rn = blk["res"][node["mother"]]
                if (rn, node["d"]) in seen:
                    continue
                seen.add((rn, node["d"]))
                a, b = (E["final"].index(d) for d in node["d"])
                P = ev[:, a] + ev[:, b]
                s = P[:, 0] ** 2 - (P[:, 1:] ** 2).sum(1)
                r = E["res"][rn]
                m0, g0 = r["par"][0], r["par"][1] if r["shape"] == "BWR" else 0.05
                w = w + (m0 * g0) ** 2 / ((s - m0 * m0) ** 2 + (m0 * g0) ** 2)
    if len(E["final"]) > 3:
        return w, 0.2 + len(seen)
    return w * (torch.linalg.cross(ev[:, 0, 1:], ev[:, 1, 1:]) ** 2).sum(1), 0.35 * (0.2 + len(seen))


def _events(E, gen, n_data, n_phsp, n_bkg):
    masses = [E["mass"][f] for f in E["final"]]
    kept, have, eff = [], 0, 0.2
    while have < n_data:
        c = _phase_space(gen, int(min(4_000_000, 1.3 * (n_data - have) / eff + 4096)), masses)
        w, top = _peaks(E, c)
        c = c[w > 0.5 * top * torch.rand(c.shape[0], generator=gen, dtype=torch.float64, device=gen.device)]
        kept.append(c)
        have += c.shape[0]
        eff = 0.05
    return dict(phsp=_phase_space(gen, n_phsp, masses), data=torch.cat(kept)[:n_data],
                bkg=_phase_space(gen, n_bkg, masses) if n_bkg else None)


def _params(E, rng, points):
    """Fit parameters [Re p, Im p, theta]: coupling magnitudes U[0.1, 1], any phase, resonance
    parameters within a per cent of their configured values."""
    n = E["n"]
    mag, ph = rng.uniform(0.1, 1.0, (points, n)), rng.uniform(0.0, 2.0 * math.pi, (points, n))
    th = np.asarray(E["init"]) * (1.0 + 0.01 * rng.standard_normal((points, E["nt"])).clip(-2.0, 2.0))
    return np.concatenate([mag * np.cos(ph), mag * np.sin(ph), th], axis=1)


def _toy_sizes(case, rng):
    """Events of each toy of an ensemble: data log-uniform in [n_data / 10, n_data]."""
    return [max(500, int(case["n_data"] * 10.0 ** (-rng.random()))) for _ in range(case["toys"])]


def _inputs(case, seed):
    """Model, samples (device tensors), weights and parameter points of a case."""
    E = _enumerate(case["model"], case["fixed"])
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    gen = torch.Generator(device=dev).manual_seed(1000003 * seed + 17)
    rng = np.random.default_rng(seed)
    if case["op"] == "toys":
        f, g = case["n_phsp"] / case["n_data"], case["n_bkg"] / case["n_data"]
        smp = [_events(E, gen, nd, int(f * nd), int(g * nd)) for nd in _toy_sizes(case, rng)]
    else:
        smp = [_events(E, gen, case["n_data"], case["n_phsp"], case["n_bkg"])]
    for s in smp:
        nb = 0 if s["bkg"] is None else s["bkg"].shape[0]
        s["bkg_weights"] = None if not nb else rng.uniform(0.6, 1.0, nb) if case["weighted"] else np.full(nb, 0.8)
    return E, smp, _params(E, rng, len(smp))


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _case(op, model, precision, n_data, n_phsp, n_bkg=0, fixed=False, weighted=False, toys=0, name=None):
    c = dict(op=op, model=model, precision=precision, n_data=n_data, n_phsp=n_phsp, n_bkg=n_bkg, fixed=fixed,
             weighted=weighted, toys=toys)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # one fit step (likelihood and gradient), which a fit repeats a few hundred times:
        # the smallest model at the size of a first look at a channel
        _case("step", "jpsi_rho", "fp64", 10_000, 50_000, name="step_rho"),
        # the benchmark workload in both storage forms
        _case("step", "jpsi_3pi", "fp64", 500_000, 2_500_000, 50_000, name="step_3pi"),
        _case("step", "jpsi_3pi", "mixed", 500_000, 2_500_000, 50_000, name="step_3pi_mixed"),
        # couplings only (every resonance parameter fixed), background with a weight per event
        _case("step", "jpsi_3pi", "mixed", 333_333, 1_666_667, 33_331, fixed=True, weighted=True, name="step_3pi_fixed"),
        # four-body cascades with Wigner rotations and a Flatte: 20 and 149 amplitudes
        _case("step", "jpsi_kkpipi", "fp64", 200_003, 1_000_001, name="step_kkpipi"),
        _case("step", "jpsi_kkpipi_wide", "fp64", 250_000, 1_250_000, name="step_wide"),
        # the Hessian: a Newton step of a toy fit, the error matrix of the benchmark fit and
        # of the 149-amplitude fit
        _case("hessian", "jpsi_3pi", "mixed", 50_000, 250_000, 5_000, name="hessian_3pi_mixed"),
        _case("hessian", "jpsi_3pi", "fp64", 500_000, 2_500_000, 50_000, name="hessian_3pi"),
        _case("hessian", "jpsi_kkpipi_wide", "fp64", 100_003, 500_009, name="hessian_wide"),
        # one round of a toy ensemble: 24 likelihoods of 5 to 50 thousand data events
        _case("toys", "jpsi_3pi", "mixed", 50_000, 250_000, 2_500, toys=24, name="toys_3pi"),
        # after the fit: the amplitude Gram behind fit fractions, and the per-event
        # partial-wave amplitudes behind projections
        _case("gram", "jpsi_kkpipi", "fp64", 2_000, 1_000_000, name="gram_kkpipi"),
        _case("waves", "jpsi_3pi", "fp64", 2_000, 1_000_000, name="waves_3pi"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# per operation: models, and the range of the data (steps, Hessians, toys) or phase-space
# (post-fit) events for each
_RANGE = {
    "step": {"jpsi_rho": (2_000, 500_000), "jpsi_3pi": (2_000, 500_000), "jpsi_kkpipi": (2_000, 200_000),
             "jpsi_kkpipi_wide": (2_000, 200_000)},
    "hessian": {"jpsi_rho": (5_000, 200_000), "jpsi_3pi": (5_000, 300_000), "jpsi_kkpipi": (5_000, 200_000),
                "jpsi_kkpipi_wide": (2_000, 80_000)},
    "toys": {"jpsi_3pi": (10_000, 50_000), "jpsi_kkpipi": (5_000, 20_000)},
    "gram": {"jpsi_3pi": (20_000, 1_000_000), "jpsi_kkpipi": (20_000, 1_000_000), "jpsi_kkpipi_wide": (20_000, 200_000)},
    "waves": {"jpsi_3pi": (20_000, 1_000_000), "jpsi_kkpipi": (20_000, 1_000_000)},
    "weights": {"jpsi_3pi": (20_000, 1_000_000), "jpsi_kkpipi": (20_000, 500_000)},
    "intensity": {"jpsi_3pi": (20_000, 1_000_000), "jpsi_kkpipi": (20_000, 1_000_000), "jpsi_kkpipi_wide": (20_000, 200_000)},
}


def draw(rng):
    op = rng.choice(["step", "step", "step", "step", "hessian", "hessian", "toys", "gram", "waves", "weights", "intensity"])
    model = rng.choice(sorted(_RANGE[op]))
    lo, hi = _RANGE[op][model]
    n = _log(rng, lo, hi)
    precision = rng.choice(["fp64", "mixed"])
    if op in ("gram", "waves", "weights", "intensity"):
        return _case(op, model, precision, 2_000, n)
    n_phsp = int(n * rng.uniform(3.0, 5.0))
    n_bkg = int(n * rng.uniform(0.02, 0.1)) if rng.random() < 0.5 else 0
    fixed = op == "step" and model != "jpsi_rho" and rng.random() < 0.25    # (one coupling alone has no gradient)
    return _case(op, model, precision, n, n_phsp, n_bkg, fixed=fixed, weighted=n_bkg > 0 and rng.random() < 0.4,
                 toys=rng.randint(4, 24) if op == "toys" else 0)


def _config(case):
    text = workloads.WORKLOADS[case["model"]]["config"]
    return workloads.fixed_theta_config(text) if case["fixed"] else text


def _host(sample):
    return {k: v.cpu().numpy() if isinstance(v, torch.Tensor) else v for k, v in sample.items() if v is not None}


class _Analysis(ctpwa_amd.analysis):
    """``ctpwa_amd.analysis`` of a configuration held as text."""

    def __init__(self, text, samples, precision):
        import os
        import tempfile
        with tempfile.TemporaryDirectory() as d:
            path = os.path.join(d, "config.yml")
            with open(path, "w") as f:
                f.write(text)
            super().__init__(path, samples=samples, precision=precision)


def prepare(case, seed):
    E, smp, pts = _inputs(case, seed)
    host = [_host(s) for s in smp]
    p = torch.tensor(pts, dtype=torch.float64, device="cuda")
    if case["op"] == "toys":
        text = build_plan(ConfigParser("", text=_config(case))).to_text()
        hs = [_native.Handle(text, s["phsp"], s["data"], s.get("bkg"), None, None, s.get("bkg_weights"),
                             precision=case["precision"]) for s in host]
        out = torch.zeros(len(hs), 1 + p.shape[1], dtype=torch.float64, device="cuda")
        return dict(op="toys", handles=hs, batch=_native.Batch(len(hs)), p=p, out=out,
                    pp=[p[j].data_ptr() for j in range(len(hs))], po=[out[j].data_ptr() for j in range(len(hs))])
    text = _config(case)
    if not case["n_bkg"]:
        text = "\n".join(x for x in text.splitlines() if not x.strip().startswith(("bkg:", "bkg_weights:"))) + "\n"
    return dict(op=case["op"], ana=_Analysis(text, host[0], case["precision"]),
                p=p[0].clone().requires_grad_(case["op"] == "step"))


def run(state):
    op, p = state["op"], state["p"]
    if op == "toys":
        state["batch"].nll_grad(state["handles"], state["pp"], state["po"], torch.cuda.current_stream().cuda_stream)
        return state["out"]
    ana = state["ana"]
    if op == "step":
        nll = ana.getNLL(p)
        (grad,) = torch.autograd.grad(nll, p)
        return {"nll": nll.detach(), "grad": grad}
    if op == "hessian":
        return ana.getHessian(p)
    if op == "gram":
        return ana.getAmplitudeGram(p, 0)
    if op == "waves":
        return ana.getPartialAmplitudes(p, 0)
    if op == "weights":
        return ana.getPartialIntensities(p, 0)
    return ana.getIntensity(p, 0)


def work(case):
    """Bytes of the stored event inputs (each read once) and of the per-event outputs, and the
    real operations of the sums (multiply and add counted apart)."""
    m = SHAPE[case["model"]]
    mixed = case["precision"] == "mixed"
    ev = m["nu"] * m["nps"] * (8 if mixed else 16) + m["inv64"] * 8 + m["inv32"] * (4 if mixed else 8)
    op, n_all = case["op"], case["n_data"] + case["n_phsp"] + case["n_bkg"]
    if op == "toys":
        n_all = int(n_all * case["toys"] * 0.9 / math.log(10.0))
    if op in ("step", "toys"):
        if case["fixed"]:
            n_all -= case["n_phsp"]
        return {"bytes": n_all * ev, "flops": n_all * (40.0 * m["amp"] + 20.0 * m["den"] + 16.0 * m["nu"] * 2)}
    if op == "hessian":
        return {"bytes": n_all * ev, "flops": n_all * 2 * 4.0 * (m["amp"] + m["th"]) ** 2}
    n = case["n_phsp"]
    if op == "gram":
        return {"bytes": n * ev, "flops": n * 2 * 4.0 * m["amp"] ** 2}
    out = {"waves": 32 * m["wave"], "weights": 8 * (m["wave"] + 1), "intensity": 8}[op]
    return {"bytes": n * (ev + out), "flops": n * (20.0 * m["amp"] + 20.0 * m["den"])}


# ---------------------------------------------------------------------------
# the same quantities in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _cg(j1, m1, j2, m2, J, M):
    f = math.factorial
    if m1 + m2 != M or not abs(j1 - j2) <= J <= j1 + j2 or abs(m1) > j1 or abs(m2) > j2 or abs(M) > J:
        return 0.0
    pre = math.sqrt((2 * J + 1) * f(j1 + j2 - J) * f(j1 - j2 + J) * f(J + j2 - j1) / f(j1 + j2 + J + 1)
                    * f(J + M) * f(J - M) * f(j1 - m1) * f(j1 + m1) * f(j2 - m2) * f(j2 + m2))
    s = 0.0
    for k in range(j1 + j2 - J + 1):
        d = [k, j1 + j2 - J - k, j1 - m1 - k, j2 + m2 - k, J - j2 + m1 + k, J - j1 - m2 + k]
        if min(d) >= 0:
            s += (-1) ** k / math.prod(f(x) for x in d)
    return pre * s


def _ylm(L, m, n):
    """Y_L^m of the unit vector n [N, 3] (Condon-Shortley), L <= 4."""
    am, z = abs(m), n[:, 2]
    xy = torch.complex(n[:, 0], n[:, 1]) ** am                  # sin^m e^{i m phi}
    p0 = torch.full_like(z, (-1.0) ** am * math.prod(range(1, 2 * am, 2)))   # P_m^m / sin^m
    p1 = z * (2 * am + 1) * p0
    for l in range(am + 1, L + 1):
        if l > am + 1:
            p0, p1 = p1, ((2 * l - 1) * z * p1 - (l + am - 1) * p0) / (l - am)
    P = p0 if L == am else p1
    y = math.sqrt((2 * L + 1) / (4 * math.pi) * math.factorial(L - am) / math.factorial(L + am)) * P * xy
    return y if m >= 0 else (-1) ** am * y.conj()


def _rotation(P, p, j):
    """exp(-i psi n.J): the Wigner rotation of a spin-j daughter p inside the moving pair P,
    in the basis m = j .. -j; [N, 2j+1, 2j+1]."""
    d = 2 * j + 1
    eye = torch.eye(d, dtype=torch.complex128, device=P.device)
    h = torch.linalg.cross(P[:, 1:], p[:, 1:])
    hn = h.norm(dim=1)
    flat = h.abs().amax(1) < 1e-10
    mass = lambda v: torch.sqrt(v[:, 0] ** 2 - (v[:, 1:] ** 2).sum(1))  # noqa: E731
    g1, g2 = P[:, 0] / mass(P), p[:, 0] / mass(p)
    cs = -(P[:, 1:] * p[:, 1:]).sum(1)
    k = torch.sqrt(1.0 / ((g1 + 1.0) * (g2 + 1.0))) / (mass(P) * mass(p))
    k = k / torch.sqrt((g1 + 1.0) * (g2 + 1.0))                 # sqrt((g-1)/(g+1)) = |p| / (m (g+1))
    psi = 2.0 * torch.atan2(hn * k, 1.0 + cs * k)
    n = h / torch.where(flat, torch.ones_like(hn), hn)[:, None]
    ms = [j - i for i in range(d)]
    jp = torch.zeros(d, d, dtype=torch.complex128, device=P.device)
    for i in range(1, d):
        jp[i - 1, i] = math.sqrt(j * (j + 1) - ms[i] * (ms[i] + 1))
    jx, jy, jz = (jp + jp.T) / 2, (jp - jp.T) / 2j, torch.diag(torch.tensor(ms, dtype=torch.complex128, device=P.device))
    X = n[:, 0, None, None] * jx + n[:, 1, None, None] * jy + n[:, 2, None, None] * jz
    R = torch.zeros_like(X)
    for m in ms:                                                # projectors on the eigenvalues of n.J
        pr = eye.expand_as(X)
        for q in ms:
            if q != m:
                pr = pr @ (X - q * eye) / (m - q)
        R = R + torch.exp(-1j * m * psi)[:, None, None] * pr
    return torch.where(flat[:, None, None], eye.expand_as(X), R)


def _bf(L, z):
    """Blatt-Weisskopf polynomial N_L(z)."""
    u = z * z
    return {0: 1.0 + 0.0 * u, 1: 1.0 + u, 2: 9.0 + 3.0 * u + u * u, 3: 225.0 + 45.0 * u + 6.0 * u ** 2 + u ** 3,
            4: 11025.0 + 1575.0 * u + 135.0 * u ** 2 + 10.0 * u ** 3 + u ** 4}[L]


def _breakup(m, a, b):
    x = (m * m - (a + b) ** 2) * (m * m - (a - b) ** 2)
    up = x > 0.0                                                # 0, without derivatives, below threshold
    return torch.where(up, torch.sqrt(torch.where(up, x, torch.ones_like(x))), torch.zeros_like(x)) / (2.0 * m)


class _Exact:
    """Amplitudes of a model over a chunk of events, differentiable in the parameters."""

    def __init__(self, E, ev):
        self.E, self.n = E, ev.shape[0]
        self.dev = ev.device
        self.cache = {}
        mom = {f: ev[:, i] for i, f in enumerate(E["final"])}
        self.sl, self.kin = [], []
        for T in E["topos"]:
            pm = dict(mom)
            for node in reversed(T["nodes"]):
                pm[node["mother"]] = pm[node["d"][0]] + pm[node["d"][1]]
            kin = []
            for node in T["nodes"]:
                m = [torch.sqrt(torch.clamp(v[:, 0] ** 2 - (v[:, 1:] ** 2).sum(1), min=0.0))
                     for v in (pm[node["mother"]],) + tuple(pm[d] for d in node["d"])]
                kin.append((m[0], _breakup(*m)))
            self.kin.append(kin)
            self.sl.append([self._tensor(T, pm, combo, kin) for combo in T["combos"]])

    def _node(self, node, pm, S, L, key):
        J, j1, j2 = node["J"]
        p1, p2 = pm[node["d"][0]], pm[node["d"][1]]
        P = p1 + p2
        k = ("dir",) + key
        if k not in self.cache:
            m = torch.sqrt(P[:, 0] ** 2 - (P[:, 1:] ** 2).sum(1))
            # daughter 1 in the pair's rest frame
            e = (p1[:, 0] * P[:, 0] - (p1[:, 1:] * P[:, 1:]).sum(1)) / m
            q = p1[:, 1:] - ((p1[:, 0] + e) / (P[:, 0] + m))[:, None] * P[:, 1:]
            qn = q.norm(dim=1)
            self.cache[k] = (qn, q / qn[:, None], [_rotation(P, x, j) if j else None for x, j in ((p1, j1), (p2, j2))])
        qn, n, R = self.cache[k]
        t = torch.zeros(self.n, 2 * J + 1, 2 * j1 + 1, 2 * j2 + 1, dtype=torch.complex128, device=self.dev)
        for a, s in enumerate(range(J, -J - 1, -1)):
            for b, s1 in enumerate(range(j1, -j1 - 1, -1)):
                for c, s2 in enumerate(range(j2, -j2 - 1, -1)):
                    M = s - s1 - s2
                    cg = _cg(j1, s1, j2, s2, S, s1 + s2) * _cg(S, s1 + s2, L, M, J, s) if abs(M) <= L else 0.0
                    if cg:
                        t[:, a, b, c] = 10.0 * cg / math.sqrt(2 * J + 1) * qn ** L * _ylm(L, M, n).conj()
        if R[0] is not None:
            t = torch.einsum("nob,naoc->nabc", R[0], t)
        if R[1] is not None:
            t = torch.einsum("noc,nabo->nabc", R[1], t)
        return t

    def _tensor(self, T, pm, combo, kin):
        """SL tensor of one (S, L) combination at m = +1, -1, with the event part of every barrier."""
        nodes = T["nodes"]
        at = {node["mother"]: k for k, node in enumerate(nodes)}

        def expand(k):                                          # [N, 2J+1] of node k's decay below it
            S, L = combo[k]
            t = self._node(nodes[k], pm, S, L, (tuple(nodes[k]["d"]), nodes[k]["J"], id(T)))
            below = [expand(at[d]) if d in at else None for d in nodes[k]["d"]]
            t = t[..., 0] if below[1] is None else (t * below[1][:, None, None, :]).sum(-1)
            return t[..., 0] if below[0] is None else (t * below[0][:, None, :]).sum(-1)

        t = expand(0)[:, [0, 2]]
        for k in range(len(nodes)):
            t = t / torch.sqrt(_bf(combo[k][1], kin[k][1] * RADIUS))[:, None]
        return t

    def factors(self, theta):
        """F_a = K_a Psi_b of every amplitude: list of [N] complex, differentiable in theta."""
        E, out = self.E, []
        val = lambda rn, p: theta[E["owner"][rn][p]] if p in E["owner"][rn] else torch.tensor(  # noqa: E731
            E["res"][rn]["par"][p], dtype=torch.float64, device=self.dev)
        for blk in E["blocks"]:
            T = E["topos"][blk["topo"]]
            mass = {f: torch.tensor(m, dtype=torch.float64, device=self.dev) for f, m in E["mass"].items()}
            mass["Jpsi"] = torch.tensor(SQRT_S, dtype=torch.float64, device=self.dev)
            for tag, rn in blk["res"].items():
                mass[tag] = val(rn, 0)
            psi = torch.ones((), dtype=torch.complex128, device=self.dev)
            q0s = []
            if T["combos"]:
                for k, node in enumerate(T["nodes"]):
                    q0 = _breakup(mass[node["mother"]], mass[node["d"][0]], mass[node["d"][1]])
                    q0s.append(q0)
                    if k == 0:
                        continue
                    rn = blk["res"][node["mother"]]
                    r, (m, q), m0 = E["res"][rn], self.kin[blk["topo"]][k], val(rn, 0)
                    s = m * m
                    if r["shape"] == "BWR":
                        l = node["lmin"]
                        re = m0 * m0 - s
                        im = (val(rn, 1) * m0 * m0 * _bf(l, q0 * RADIUS) / q0 ** (2 * l + 1)
                              * q ** (2 * l + 1) / (m * _bf(l, q * RADIUS)))
                    else:
                        re, im = m0 * m0 - s, 0.0
                        for i, (ma, mb) in enumerate(r["ch"]):
                            f1, f2 = 1.0 - (ma + mb) ** 2 / s, 1.0 - (ma - mb) ** 2 / s
                            rho = torch.sqrt(f1.abs() * f2.clamp(min=0.0))
                            b = m0 * val(rn, 1 + i) / 2.0
                            re = re + b * torch.where(f1 < 0, rho, torch.zeros_like(rho))
                            im = im + b * torch.where(f1 >= 0, rho, torch.zeros_like(rho))
                    psi = psi * torch.complex(re, im) / (re * re + im * im)
            for combo in T["combos"]:
                K = 1.0
                for k in range(len(T["nodes"])):
                    K = K * torch.sqrt(_bf(combo[k][1], q0s[k] * RADIUS))
                out.append(K * psi)
        return out

    def amplitudes(self, p):
        """[N, 2, n_amp] without couplings."""
        F = self.factors(p[2 * self.E["n"]:])
        return torch.stack([F[a][:, None] * self.sl[self.E["blocks"][b]["topo"]][c]
                            for a, (b, c) in enumerate(self.E["amps"])], dim=2)

    def couplings(self, p):
        n = self.E["n"]
        idx = torch.tensor(self.E["free_of"], device=self.dev)
        return torch.complex(p[:n], p[n:2 * n])[idx]

    def waves(self, p):
        """[n_wave, N, 2]: the couplings-weighted sum of each block's amplitudes."""
        A, v = self.amplitudes(p), self.couplings(p)
        out = torch.zeros(len(self.E["blocks"]), self.n, 2, dtype=torch.complex128, device=self.dev)
        for a, (b, _) in enumerate(self.E["amps"]):
            out[b] += v[a] * A[:, :, a]
        return out

    def intensity(self, p):
        F, v = self.factors(p[2 * self.E["n"]:]), self.couplings(p)
        y = {}
        for a, (b, c) in enumerate(self.E["amps"]):
            k = (self.E["blocks"][b]["topo"], c)
            t = v[a] * F[a]
            y[k] = t if k not in y else y[k] + t
        S = sum(t[:, None] * self.sl[k[0]][k[1]] for k, t in y.items())
        return (S.real ** 2 + S.imag ** 2).sum(1)


def _chunks(ev, w, step):
    for s in range(0, ev.shape[0], step):
        yield ev[s:s + step], None if w is None else w[s:s + step]


def _class_sum(E, ev, w, p, step, hessian):
    """Sum, gradient and (optionally) Hessian over a sample of w ln I, or of I where w is None."""
    P, n = p.numel(), E["n"]
    f, g = 0.0, torch.zeros_like(p)
    H = torch.zeros(P, P, dtype=torch.float64, device=p.device)
    inv = torch.tensor(E["free_of"], device=p.device)
    for e, we in _chunks(ev, w, step):
        X = _Exact(E, e)
        x = p.detach().clone().requires_grad_(True)
        I = X.intensity(x)
        t = (I if we is None else we * torch.log(I)).sum()
        gr = torch.autograd.grad(t, x, create_graph=hessian)[0]
        f += float(t.detach())
        g += gr.detach()
        if hessian:
            for j in range(2 * n, P):                           # rows of the resonance parameters
                H[j] += torch.autograd.grad(gr[j], x, retain_graph=True)[0]
            with torch.no_grad():                               # the couplings' block in closed form
                A = X.amplitudes(p)
                S = (A * X.couplings(p)).sum(2)
                I = (S.real ** 2 + S.imag ** 2).sum(1)
                al = torch.ones_like(I) if we is None else we / I
                B = torch.empty(A.shape[0], 2, n, dtype=torch.complex128, device=p.device)
                B[:, :, inv] = A
                B = torch.cat([B, 1j * B], dim=2)
                D = (B * torch.sqrt(al)[:, None, None]).reshape(-1, 2 * n)
                D = torch.cat([D.real, D.imag])
                h = 2.0 * D.T @ D
                if we is not None:
                    u = 2.0 * (S.conj()[:, :, None] * B).sum(1).real * (torch.sqrt(we) / I)[:, None]
                    h -= u.T @ u
                H[:2 * n, :2 * n] += h
        del X
    H[:2 * n, 2 * n:] = H[2 * n:, :2 * n].T
    return f, g, H


def _likelihood(E, s, p, hessian):
    step = 200_000 if E["n"] < 30 else 25_000
    dev = p.device
    one = torch.ones(s["data"].shape[0], dtype=torch.float64, device=dev)
    fd, gd, Hd = _class_sum(E, s["data"], one, p, step, hessian)
    fb, gb, Hb, Wb = 0.0, 0.0, 0.0, 0.0
    if s["bkg"] is not None:
        w = torch.tensor(s["bkg_weights"], dtype=torch.float64, device=dev)
        fb, gb, Hb = _class_sum(E, s["bkg"], w, p, step, hessian)
        Wb = float(w.sum())
    z, gz, Hz = _class_sum(E, s["phsp"], None, p, step, hessian)
    neff = s["data"].shape[0] - Wb
    nll = -fd + fb + neff * math.log(z / s["phsp"].shape[0])
    grad = -gd + gb + neff * gz / z
    H = -Hd + Hb + neff * (Hz / z - torch.outer(gz, gz) / z ** 2) if hessian else None
    return nll, grad, H


def exact(case, seed):
    E, smp, pts = _inputs(case, seed)
    dev = smp[0]["phsp"].device
    P = torch.tensor(pts, dtype=torch.float64, device=dev)
    op, p = case["op"], P[0]
    if op == "toys":
        rows = [_likelihood(E, s, P[j], False) for j, s in enumerate(smp)]
        return torch.stack([torch.cat([g.new_tensor([f]), g]) for f, g, _ in rows])
    if op == "step":
        f, g, _ = _likelihood(E, smp[0], p, False)
        return {"nll": torch.tensor(f, dtype=torch.float64), "grad": g}
    if op == "hessian":
        return _likelihood(E, smp[0], p, True)[2]
    ev, got = smp[0]["phsp"], []
    with torch.no_grad():
        for e, _ in _chunks(ev, None, 200_000 if E["n"] < 30 else 25_000):
            X = _Exact(E, e)
            if op == "gram":
                A = X.amplitudes(p).reshape(-1, E["n"])
                got.append(A.conj().T @ A)
            elif op == "intensity":
                got.append(X.intensity(p))
            else:
                W = X.waves(p)
                if op == "weights":
                    tot = W.sum(0)
                    W = torch.cat([(W.real ** 2 + W.imag ** 2).sum(2), (tot.real ** 2 + tot.imag ** 2).sum(1)[None]])
                got.append(W)
    if op == "gram":
        return sum(got).cpu().numpy()
    return torch.cat(got, dim=0 if op == "intensity" else 1)
