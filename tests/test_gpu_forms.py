"""Every form of an FP64 evaluation on the register passes (density in and
potential out; trial points phi_t = ca u + cb v in with the potential, the
signed dE/dphi or the Newton product out), one request and two in a launch set,
with one and two spin channels, with alpha != beta and with WGC, against the
staged LDS passes.

Outputs within 1e-13 of the largest value that enters them, the bound the other
register passes are held to; the Newton product divides a difference by eps =
1e-3, so 1e-13 / eps of the largest dE/dphi. Energy sums within 1e-12 of the
largest. The optimizer's sums against numpy on the outputs themselves, within
1e-13 of the sum of magnitudes (32 levels of pairwise rounding are 4e-15). Two
requests in a launch set give the bits of each alone."""
import numpy as np
import pytest

from tests import eval_forms as F

pytestmark = pytest.mark.gpu

CASES = [((36, 21, 63), "spin", "three"), ((20, 24, 18), "spin4", "general"), ((32, 32, 24), "spin", "plane"),
         ((32, 32, 24), "spin4", "plane"), ((20, 24, 18), "wt4", "three"), ((128, 28, 25), "wt", "three"),
         ((18, 125, 16), "wt4", "general"), ((200, 27, 20), "wt", "general"), ((20, 24, 18), "wgc", "general"),
         ((256, 18, 16), "wgc", "general"), ((128, 128, 24), "wgc", "plane"), ((64, 64, 256), "wt4", "plane"),
         ((32, 32, 192), "wt", "plane")]
EPS = 1e-3


def request(grid, kind, seed, phi_in, newton_ch=None):
    rng = np.random.default_rng(seed)
    shape = grid[::-1]
    nc = (grid[0] // 2 + 1) * grid[1] * grid[2]
    spin = kind.startswith("spin")
    ab = dict(wt=(5 / 6, 5 / 6), spin=(5 / 6, 5 / 6), wt4=(0.9, 0.7), spin4=(0.9, 0.7), wgc=(1.2, 0.46))[kind]
    q = dict(alpha=ab[0], beta=ab[1], vion=0.1 + rng.random(shape))
    if kind == "wgc":
        q["wgck"] = (0.1 + rng.random(4 * nc)) * 0.1
    else:
        q["wtk"] = (0.1 + rng.random(nc)) / (grid[0] * grid[1] * grid[2])
    for s, name in enumerate(("u", "u2") if spin else ("u",)):
        rho = (0.55, 0.45)[s] * 0.027 * (1.0 + 0.3 * (2.0 * rng.random(shape) - 1.0))
        q[name] = np.sqrt(rho) if phi_in else rho
    if not phi_in:
        return q
    names = ("v", "v2") if spin else ("v",)
    if newton_ch is None:   # a point of a line search
        for s, n in enumerate(names):
            q[n] = 0.03 * (2.0 * rng.random(shape) - 1.0)
        q.update(ca=0.96, cb=0.28, s1=-0.28, s2=0.96, mu0=0.11)
        if spin:
            q.update(ca2=0.96, cb2=0.28, s1b=-0.28, s2b=0.96, mu0b=0.13)
        return q
    q[names[newton_ch]] = 0.5 * (2.0 * rng.random(shape) - 1.0)
    q.update(bvec=rng.random(shape) - 0.5, w=rng.random(shape) - 0.5, eps=EPS, mu0=0.11, newton_ch=newton_ch, ca=1.0)
    q["cb2" if newton_ch else "cb"] = EPS
    if spin:
        q["ca2"] = 1.0
        del q["w"]   # the spin solver takes that sum itself
    return q


def check_sums(q, outs, sums, outmode, spin):
    def holds(k, *terms):
        t = [a for a in terms]
        assert abs(sums[k] - sum(a.sum() for a in t)) <= 1e-13 * sum(np.abs(a).sum() for a in t), k
    if outmode == F.OUT_SIGNED:
        t = q["ca"] * q["u"] + q["cb"] * q["v"]
        holds(6, outs[0] * (q["s1"] * q["u"] + q["s2"] * q["v"]))
        holds(8, outs[0] * t)
        sq = [(outs[0] - 2.0 * q["mu0"] * t) ** 2]
        if spin:
            t2 = q["ca2"] * q["u2"] + q["cb2"] * q["v2"]
            sq.append((outs[1] - 2.0 * q["mu0b"] * t2) ** 2)
            holds(9, outs[1] * (q["s1b"] * q["u2"] + q["s2b"] * q["v2"]))
            holds(10, outs[1] * t2)
        else:
            holds(9, outs[0] ** 2)
            holds(10, t * t)
        holds(7, *sq)
    elif outmode == F.OUT_NEWTON:
        p = q["v2" if q["newton_ch"] else "v"]
        holds(6, p * outs[0])
        if "w" in q:
            holds(7, q["w"] * outs[0])
            holds(8, outs[0] ** 2)


@pytest.mark.parametrize("grid,kind,family", CASES)
def test_forms(monkeypatch, grid, kind, family):
    print(grid, kind, family, flush=True)
    spin = kind.startswith("spin")
    F.environment(monkeypatch, False)
    ev = F.Evaluator(grid, kind)
    F.environment(monkeypatch, True)
    staged = F.Evaluator(grid, kind)
    forms = [(F.IN_RHO, F.OUT_POT, None), (F.IN_PHI, F.OUT_POT, None), (F.IN_PHI, F.OUT_SIGNED, None),
             (F.IN_PHI, F.OUT_NEWTON, 0)] + ([(F.IN_PHI, F.OUT_NEWTON, 1)] if spin else [])
    scale = None
    for inmode, outmode, ch in forms:
        print("  form", inmode, outmode, ch, flush=True)
        reqs = [request(grid, kind, seed, inmode == F.IN_PHI, ch) for seed in (1, 2)]
        got, ref = ev.run(reqs, inmode, outmode), staged.run(reqs, inmode, outmode)
        for q, (o, e), (o0, e0) in zip(reqs, got, ref):
            n = 1 if outmode == F.OUT_NEWTON else len(o)   # the Newton form writes one channel's product
            big = max(np.max(np.abs(x)) for x in o0[:n])
            if (inmode, outmode) == (F.IN_PHI, F.OUT_POT):
                scale = big
            bound = 1e-13 * (scale / EPS if outmode == F.OUT_NEWTON else big)
            for x, x0 in zip(o[:n], o0[:n]):
                assert np.max(np.abs(x - x0)) <= bound, (inmode, outmode, np.max(np.abs(x - x0)), bound)
            assert np.max(np.abs(e[:6] - e0[:6])) <= 1e-12 * np.max(np.abs(e0[:6]))
            check_sums(q, o, e, outmode, spin)
        for i in range(2):
            (o, e), = ev.run(reqs[i:i + 1], inmode, outmode)
            n = 1 if outmode == F.OUT_NEWTON else len(o)
            assert np.array_equal(e, got[i][1]) and all(np.array_equal(a, b) for a, b in zip(o[:n], got[i][0]))
