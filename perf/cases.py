"""The solver's performance cases: the work a user of this library has it do,
through its public entry points (sw-mpdec_amd/swm.py over include/swm.h).

A pass is a user's call between two outputs:

  solve   the state goes to the handle, `steps` steps of the time scheme run
          with the device's own time steps (swm_run_steps), the state comes back
  loop    the same with the host's time loop, as the drop-in in the reference's
          program drives it: swm_timestep and one swm_step_* call per step
  batch   a handful of uneven independent grids in one engine: submitted by
          their family's parameters, run until all are done, fetched, released

listed() gives the fixed cases, draw() more of the same ranges.  exact() is the
same computation in plain torch FP64, written from the scheme's formulas.
"""
from __future__ import annotations

import math
import random
import sys
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parent.parent
sys.path.insert(0, str(ROOT / "sw-mpdec_amd"))

import problems as P  # noqa: E402
import swm  # noqa: E402

G = 9.81
CFL = 0.5
# FVTD evaluations and Patankar solves of one step, by timescheme
FVTDS = {1: 1, 2: 5, 3: 6, 4: 13, 5: 13, 6: 1, 7: 2}
SOLVES = {1: 0, 2: 0, 3: 0, 4: 0, 5: 13, 6: 1, 7: 2}
# the most a drawn case may cost, in FVTD evaluations of one cell: the largest listed case
MOST_WORK = 2048 * 2048 * 13 * 5


def listed():
    return [
        # the smallest call: a 32^2 grid (the low end of the batched mix), where latency counts
        dict(name="vortex_32", call="solve", family="vortex", nx=32, ny=32, scheme=5, recfix=4,
             steps=20),
        # the drop-in's time loop on a small odd rectangle: one timestep and one step call a step
        dict(name="loop_101x67", call="loop", family="vortex", nx=101, ny=67, scheme=5, recfix=4,
             steps=10),
        # the size the reference itself is run at on a CPU: its lake at rest, well-balanced
        dict(name="lake_128", call="solve", family="lake", nx=128, ny=128, scheme=5, recfix=4,
             steps=10),
        # first-order fix on the cells the shock indicator flags, on a dam break
        dict(name="dam_192_fix1", call="solve", family="dam", nx=192, ny=160, scheme=5, recfix=1,
             steps=10),
        # an ordinary request of the served stream, odd
        dict(name="vortex_257", call="solve", family="vortex", nx=257, ny=257, scheme=5, recfix=4,
             steps=10),
        # the explicit scheme most used without the Patankar build, lake without well-balancing
        dict(name="ssprk4_300x417", call="solve", family="lake_nowb", nx=300, ny=417, scheme=2,
             recfix=4, steps=10),
        # the second-order modified-Patankar scheme
        dict(name="mpdec2_640x360", call="solve", family="lake", nx=640, ny=360, scheme=7,
             recfix=4, steps=10),
        # a dam break with the MUSCL fix at the middle of the served sizes
        dict(name="dam_512_fix2", call="solve", family="dam", nx=512, ny=512, scheme=5, recfix=2,
             steps=5),
        # the explicit fifth-order scheme on a wide grid
        dict(name="dec5_1000x700", call="solve", family="vortex", nx=1000, ny=700, scheme=4,
             recfix=4, steps=4),
        # the largest served request: a dam break, with the many Jacobi sweeps it asks for
        dict(name="dam_1024", call="solve", family="dam", nx=1024, ny=1024, scheme=5, recfix=4,
             steps=4),
        # the benchmark's headline grid: well-balanced lake over bumps
        dict(name="lake_2048", call="solve", family="lake", nx=2048, ny=2048, scheme=5, recfix=4,
             steps=5),
        # a batch of uneven solves in one engine (a slice of the benchmark's batched mix)
        dict(name="batch_16", call="batch", mix=2024, jobs=16, nmin=32, nmax=256, scheme=5,
             recfix=4, steps=16),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    if rng.random() < 0.15:
        return dict(call="batch", mix=rng.randrange(1 << 20), jobs=rng.randint(4, 20), nmin=32,
                    nmax=_log_int(rng, 96, 400), scheme=5, recfix=4, steps=rng.randint(10, 30))
    call = "loop" if rng.random() < 0.15 else "solve"
    scheme = rng.choice((5, 5, 5, 5, 5, 5, 4, 2, 3, 1, 7, 6))
    family = rng.choice(("vortex", "lake", "dam", "lake_nowb") if scheme < 5 else
                        ("vortex", "vortex", "lake", "lake", "dam"))
    recfix = rng.choice((4, 4, 4, 1, 2)) if family == "dam" else 4
    size = _log_int(rng, 24, 1500)
    aspect = math.exp(rng.uniform(-0.5, 0.5))
    nx = max(17, int(size * math.sqrt(aspect)) + rng.randint(0, 2))
    ny = max(17, int(size / math.sqrt(aspect)) + rng.randint(0, 2))
    most = MOST_WORK // (2 * nx * ny * FVTDS[scheme])
    steps = max(1, min(rng.randint(4, 20), most))
    return dict(call=call, family=family, nx=nx, ny=ny, scheme=scheme, recfix=recfix, steps=steps)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _device():
    return torch.device("cuda") if torch.cuda.is_available() else torch.device("cpu")


def _params(family, seed):
    """The family's parameters from the seed, in the ranges the benchmark draws."""
    r = random.Random(seed * 7919 + 17)
    if family == "vortex":
        return dict(eps=r.uniform(0.5, 1.5))
    if family == "dam":
        return dict(radius=r.uniform(0.2, 0.3), h_in=1.0, h_out=r.uniform(0.1, 0.2))
    q = dict(A=[r.uniform(0.05, 0.11) for _ in range(8)], s=[r.uniform(0.05, 0.2) for _ in range(8)],
             cx=[r.random() for _ in range(8)], cy=[r.random() for _ in range(8)],
             amp=1e-3, px=r.random(), py=r.random(), ps=r.uniform(0.05, 0.2))
    return q


def _axis(n, dev):
    """(dx, x at the 4 Gauss points of every cell (4, n)) of n cells on [0, 1]."""
    nodes, _ = _gauss()
    dx = 1.0 / n
    bary = torch.arange(n, dtype=torch.float64, device=dev) * dx + 0.5 * dx
    return dx, torch.stack([bary + c * dx for c in nodes])


def _gauss():
    a = 2. / 7. * math.sqrt(6. / 5.)
    o, i = 0.5 * math.sqrt(3. / 7. + a), 0.5 * math.sqrt(3. / 7. - a)
    s = math.sqrt(30.)
    return (-o, -i, i, o), ((18. - s) / 72., (18. + s) / 72., (18. + s) / 72., (18. - s) / 72.)


def _hump(x, c, s):
    """sum over three periodic images of exp(-(x-c-a)^2/s^2), and its derivative."""
    g, d = 0., 0.
    for a in (-1, 0, 1):
        t = x - (c + a)
        e = torch.exp(-(t * t) / (s * s))
        g = g + e
        d = d - e * t * (2. / (s * s))
    return g, d


def _inputs(family, nx, ny, q, dev):
    """U0 (3, ny, nx), and for the lakes Uwb and the bathymetry gradients
    (16, ny, nx) at the Gauss points, plane yg*4 + xg."""
    _, w = _gauss()
    _, X = _axis(nx, dev)
    _, Y = _axis(ny, dev)
    U0 = torch.zeros(3, ny, nx, dtype=torch.float64, device=dev)
    lake = family.startswith("lake")
    Uwb = torch.zeros_like(U0) if lake else None
    bx = torch.zeros(16, ny, nx, dtype=torch.float64, device=dev) if lake else None
    by = torch.zeros_like(bx) if lake else None
    if lake:
        hx = [[_hump(X[a], c, s) for a in range(4)] for c, s in zip(q["cx"], q["s"])]
        hy = [[_hump(Y[a], c, s) for a in range(4)] for c, s in zip(q["cy"], q["s"])]
        px = [_hump(X[a], q["px"], q["ps"])[0] for a in range(4)]
        py = [_hump(Y[a], q["py"], q["ps"])[0] for a in range(4)]
    for xg in range(4):
        for yg in range(4):
            c = w[xg] * w[yg]
            if family == "vortex":
                xp, yp = (X[xg][None, :] - 0.5) / 0.1, (Y[yg][:, None] - 0.5) / 0.1
                r2 = xp * xp + yp * yp
                h = 1.0 - q["eps"] * q["eps"] / (2.0 * G) * torch.exp(1.0 - r2)
                s = q["eps"] * torch.exp(0.5 * (1.0 - r2))
                U0 += c * torch.stack([h, h * (-s * yp), h * (s * xp)])
            elif family == "dam":
                r2 = (X[xg][None, :] - 0.5) ** 2 + (Y[yg][:, None] - 0.5) ** 2
                U0[0] += c * torch.where(r2 < q["radius"] * q["radius"],
                                         torch.full_like(r2, q["h_in"]),
                                         torch.full_like(r2, q["h_out"]))
            else:
                b = torch.zeros_like(U0[0])
                for k in range(8):
                    (gx, dgx), (gy, dgy) = hx[k][xg], hy[k][yg]
                    b += q["A"][k] * gx[None, :] * gy[:, None]
                    bx[yg * 4 + xg] += q["A"][k] * dgx[None, :] * gy[:, None]
                    by[yg * 4 + xg] += q["A"][k] * gx[None, :] * dgy[:, None]
                Uwb[0] += c * (1.0 - b)
                U0[0] += c * (1.0 - b + q["amp"] * px[xg][None, :] * py[yg][:, None])
    return U0, Uwb, bx, by


def _host(U):
    """(3, ny, nx) on the device -> the boundary's (ny, nx, 3) host array."""
    return np.ascontiguousarray(U.permute(1, 2, 0).cpu().numpy())


def _jobs(case, seed):
    """The batch's jobs: sizes and step counts of the case, parameters of the seed."""
    r = random.Random(case["mix"])
    jobs = []
    for k in range(case["jobs"]):
        n = _log_int(r, case["nmin"], case["nmax"])
        steps = r.randint(max(1, case["steps"] // 4), case["steps"])
        family = ("vortex", "lake")[k % 2]
        jobs.append((family, n, steps, _params(family, seed + 101 * k)))
    return jobs


def prepare(case, seed):
    if case["call"] == "batch":
        kind = {"vortex": P.FAMILY_VORTEX, "lake": P.FAMILY_LAKE_BUMPS}
        specs = [(P.FamilySpec(kind[f], n, q, steps=steps, cfl=CFL, gravity=G), steps)
                 for f, n, steps, q in _jobs(case, seed)]
        return dict(call="batch", engine=swm.Engine(), specs=specs)
    nx, ny = case["nx"], case["ny"]
    U0, Uwb, bx, by = _inputs(case["family"], nx, ny, _params(case["family"], seed), _device())
    wb = case["family"] == "lake"
    s = swm.Solver(nx, ny, 1.0 / nx, 1.0 / ny, G, CFL, wb, np.array(_gauss()[1]))
    s.set_timescheme(case["scheme"])
    s.set_hp_association(swm.HP_BY_NODE)
    if case["recfix"] != 4:
        s.set_reconstruction_fix(case["recfix"])
    if bx is not None:
        s.set_bathy_grad(bx.cpu().numpy(), by.cpu().numpy())
    if wb:
        s.init_wb(_host(Uwb))
    return dict(call=case["call"], solver=s, U0=_host(U0), steps=case["steps"])


def run(state):
    if state["call"] == "batch":
        eng = state["engine"]
        ids = [eng.submit_family(spec, steps) for spec, steps in state["specs"]]
        while eng.run(16)[0]:
            pass
        out = {"U%02d" % k: eng.fetch(j) for k, j in enumerate(ids)}
        for j in ids:
            eng.release(j)
        return out
    s = state["solver"]
    s.upload(state["U0"])
    if state["call"] == "loop":
        hist, U = s.run(state["steps"])
        return {"U": U, "dt": np.array([h[0] for h in hist]),
                "sweeps": np.array([h[3] for h in hist], dtype=np.int64)}
    dts, sweeps, _ = s.run_steps(state["steps"])
    return {"U": s.download(), "dt": dts, "sweeps": sweeps.astype(np.int64)}


def _work(cells, steps, scheme, lake, wb):
    # one step reads and writes the state once, and reads the bathymetry and
    # the well-balanced tables once; a pass also takes the state in and out
    step_bytes = 48. + (256. if lake else 0.) + (64. if wb else 0.)
    # per face: ConsToPrim 4, three first and six second WENO sweeps 1668,
    # limiter 70, Rusanov at four Gauss points 264; per cell of an FVTD two
    # faces, and over bathymetry five depth sweeps 1100 and 16 x 10 for the
    # source; per Patankar system of a cell 16 divisions with 6 operations
    # each, and at least one sweep of 10
    fvtd = 2. * 2006. + 20. + (1260. if lake else 0.)
    flops = FVTDS[scheme] * fvtd + SOLVES[scheme] * 122.
    return cells * (steps * step_bytes + 48.), cells * steps * flops


def work(case):
    if case["call"] == "batch":
        parts = [_work(n * n, steps, case["scheme"], f == "lake", f == "lake")
                 for f, n, steps, _ in _jobs(case, 0)]
    else:
        f = case["family"]
        parts = [_work(case["nx"] * case["ny"], case["steps"], case["scheme"],
                       f.startswith("lake"), f == "lake")]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


# ---------------------------------------------------------------------------
# the same computation in plain torch FP64: tensors (..., ny, nx)
# ---------------------------------------------------------------------------
EPS = 1e-24
HMIN = 1e-6
GAMMA2 = ((0.2658420974778319, 0.6112504900322486, 0.1229074124899195),
          (0.1281641584355059, 0.5219691498503563, 0.3498666917141379),
          (0.3498666917141379, 0.5219691498503563, 0.1281641584355059),
          (0.1229074124899195, 0.6112504900322486, 0.2658420974778319))
# candidate coefficients on (q-2, q-1, q0), (q-1, q0, q+1), (q0, q+1, q+2)
CAND2 = (((-0.1642562761719537, 0.7590807081409336, 0.4051755680310201),
          (0.2663118796250726, 0.8979443965468811, -0.1642562761719537),
          (1.6968800354220990, -0.9631919150471715, 0.2663118796250726)),
         ((-0.1122135388132497, 0.3944175994189276, 0.7177959393943222),
          (0.0577769829791784, 1.0544365558340714, -0.1122135388132497),
          (1.2277675047716066, -0.2855444877507849, 0.0577769829791784)),
         ((0.0577769829791784, -0.2855444877507849, 1.2277675047716066),
          (-0.1122135388132497, 1.0544365558340714, 0.0577769829791784),
          (0.7177959393943222, 0.3944175994189276, -0.1122135388132497)),
         ((0.2663118796250726, -0.9631919150471715, 1.6968800354220990),
          (-0.1642562761719537, 0.8979443965468811, 0.2663118796250726),
          (0.4051755680310201, 0.7590807081409336, -0.1642562761719537)))
THETA = {5: ((0., 0., 0., 0.),
             (0.1103005664791649049, 0.1896994335208351257, -0.0339073642291439076,
              0.0103005664791649201),
             (0.0730327668541684294, 0.4505740308958107176, 0.2269672331458314485,
              -0.0269672331458315692),
             (0.0833333333333333287, 0.4166666666666666852, 0.4166666666666666852,
              0.0833333333333333287)),
         7: ((0., 0.), (0.5, 0.5))}
THETA[4] = THETA[5]
THETA[6] = THETA[7]
SSPRK4 = (((0, 1.0, ), 0.39175222700392),
          ((0, 0.44437049406734, 1, 0.55562950593266), 0.36841059262959),
          ((0, 0.62010185138540, 2, 0.37989814861460), 0.25189177424738),
          ((0, 0.17807995410773, 3, 0.82192004589227), 0.54497475021237))
SSPRK4_LAST = ((0, 0.00683325884039), (2, 0.51723167208978), (3, 0.12759831133288),
               (4, 0.34833675773694))
ARK65 = ((0.25,), (0.125, 0.125), (0., 0., 0.5), (0.1875, -0.375, 0.375, 0.5625),
         (-0.42857142857142855, 1.1428571428571428, 0.8571428571428571, -1.7142857142857142,
          1.1428571428571428))
BRK65 = (0.077777777777777778, 0., 0.35555555555555556, 0.13333333333333333, 0.35555555555555556,
         0.077777777777777778)


def _five(q, axis):
    return [torch.roll(q, -o, axis) for o in (-2, -1, 0, 1, 2)]


def _alphas(q):
    a, b, c, d, e = q
    b1 = (1. / 3.) * (4. * a * a - 19. * a * b + 25. * b * b + 11. * a * c - 31. * b * c
                      + 10. * c * c)
    b2 = (1. / 3.) * (4. * b * b - 13. * b * c + 13. * c * c + 5. * b * d - 13. * c * d
                      + 4. * d * d)
    b3 = (1. / 3.) * (10. * c * c - 31. * c * d + 25. * d * d + 11. * c * e - 19. * d * e
                      + 4. * e * e)
    return [(EPS + t) * (EPS + t) for t in (b1, b2, b3)]


def _blend(gam, den, w):
    al = [torch.full_like(t, g) / t for g, t in zip(gam, den)]
    s = al[0] + al[1] + al[2]
    return al[0] / s * w[0] + al[1] / s * w[1] + al[2] / s * w[2]


def _first(q):
    a, b, c, d, e = q
    den = _alphas(q)
    m = _blend((.3, .6, .1), den, ((1. / 6.) * (-a + 5. * b + 2. * c),
                                   (1. / 6.) * (2. * b + 5. * c - d),
                                   (1. / 6.) * (11. * c - 7. * d + 2. * e)))
    p = _blend((.1, .6, .3), den, ((1. / 6.) * (2. * a - 7. * b + 11. * c),
                                   (1. / 6.) * (-b + 5. * c + 2. * d),
                                   (1. / 6.) * (2. * c + 5. * d - e)))
    return m, p


def _second(q):
    a, b, c, d, e = q
    den = _alphas(q)
    return [_blend(gam, den, (k[0][0] * a + k[0][1] * b + k[0][2] * c,
                              k[1][0] * b + k[1][1] * c + k[1][2] * d,
                              k[2][0] * c + k[2][1] * d + k[2][2] * e))
            for gam, k in zip(GAMMA2, CAND2)]


def _primitives(U):
    ht = U[0] + torch.full_like(U[0], HMIN) / U[0]
    return torch.stack([U[0], U[1] / ht, U[2] / ht])


class _Plain:
    """One grid: U is (3, M, ny, nx) for M states at once."""

    def __init__(self, nx, ny, Uwb, bx, by, recfix):
        self.nx, self.ny, self.bx, self.by, self.recfix = nx, ny, bx, by, recfix
        self.d = {-1: 1.0 / nx, -2: 1.0 / ny}
        self.w = _gauss()[1]
        self.wb = None
        if Uwb is not None:
            self.wb = self.parts(Uwb[:, None])

    def faces(self, V, axis):
        """Fluxes of the n + 1 faces along axis (-1: x, -2: y)."""
        other = -3 - axis
        n = V.shape[axis]
        m, p = _first(_five(V, axis))
        WM, WP = _second(_five(m, other)), _second(_five(p, other))  # lists over Gauss points
        if self.recfix != 4:
            WM, WP = self.fixed(V, WM, WP, axis, n)
        else:
            WM, WP = ([torch.cat([W.narrow(axis, n - 1, 1), W, W.narrow(axis, 0, 1)], axis)
                       for W in WW] for WW in (WM, WP))
        # cells 0..n+1 from here on; the limiter leaves out cell n+1
        h = V[0]
        h = torch.cat([h.narrow(axis, n - 1, 1), h], axis)
        wm = [W[0].narrow(axis, 0, n + 1) for W in WM]
        wp = [W[0].narrow(axis, 0, n + 1) for W in WP]
        al = sum(w * x for w, x in zip(self.w, wm))
        be = sum(w * x for w, x in zip(self.w, wp))
        lob = 1. / 12.
        csi = (h - lob * al - lob * be) / torch.full_like(h, 1. - 2. * lob)
        total = 0.
        for g in range(4):
            mn = torch.minimum(torch.minimum(csi, wm[g]), wp[g])
            th = torch.where(h == mn, torch.ones_like(h),
                             torch.clamp(torch.abs((h - HMIN) / (h - mn)), max=1.))
            hl = h + th * (wp[g] - h)
            lm = h + th * (wm[g] - h)
            hr = torch.cat([lm.narrow(axis, 1, n), WM[g][0].narrow(axis, n + 1, 1)], axis)
            L, R = WP[g].narrow(axis, 0, n + 1), WM[g].narrow(axis, 1, n + 1)
            un = 1 if axis == -1 else 2
            F = self.rusanov(hl, L[un], L[3 - un], hr, R[un], R[3 - un])
            F = torch.stack(F if axis == -1 else (F[0], F[2], F[1]))
            total = total + self.w[g] * F
        return total

    def fixed(self, V, WM, WP, axis, n):
        """Cells 0..n+1 with the fix on the flagged ones: cell c takes the
        verdict of the indicator at min(c + 1, n)."""
        up, dn = torch.roll(V, -1, axis), torch.roll(V, 1, axis)
        a, b, c = dn[0], V[0], up[0]
        ind = torch.abs(a + c - 2. * b) / (torch.abs(a) + torch.abs(c) + torch.abs(2. * b))
        at = torch.clamp(torch.arange(1, n + 3, device=V.device), max=n) - 1
        flag = (ind > 0.5e-3).index_select(axis if axis >= 0 else ind.dim() + axis, at)
        ext = lambda T: torch.cat([T.narrow(axis, n - 1, 1), T, T.narrow(axis, 0, 1)], axis)  # noqa: E731
        fm = fp = V
        if self.recfix == 2:
            d = torch.full_like(V, self.d[axis])
            sp, sm = (up - V) / d, (V - dn) / d
            one = torch.ones_like(V)
            slope = 0.5 * (torch.copysign(one, sm) + torch.copysign(one, sp)) * torch.minimum(
                torch.abs(sm), torch.abs(sp))
            fm, fp = V - 0.5 * slope * d, V + 0.5 * slope * d
        fm, fp = ext(fm), ext(fp)
        return ([torch.where(flag, fm, ext(W)) for W in WM],
                [torch.where(flag, fp, ext(W)) for W in WP])

    @staticmethod
    def rusanov(hl, ul, tl, hr, ur, tr):
        """Flux along the normal: (mass, normal momentum, tangential momentum);
        the reference's wave speed is |u + sqrt(g h)|."""
        out = []
        lam = torch.maximum(torch.abs(ul + torch.sqrt(G * hl)), torch.abs(ur + torch.sqrt(G * hr)))
        fl = (hl * ul, hl * (ul * ul) + (0.5 * G) * (hl * hl), (hl * ul) * tl)
        fr = (hr * ur, hr * (ur * ur) + (0.5 * G) * (hr * hr), (hr * ur) * tr)
        cl, cr = (hl, hl * ul, hl * tl), (hr, hr * ur, hr * tr)
        for k in range(3):
            out.append(0.5 * ((fl[k] + fr[k]) - lam * (cr[k] - cl[k])))
        return tuple(out)

    def source(self, h):
        S2, S3 = torch.zeros_like(h), torch.zeros_like(h)
        if self.bx is None:
            return S2, S3
        hgp = [_second(_five(v, -1)) for v in _second(_five(h, -2))]  # [yg][xg]
        for xg in range(4):
            for yg in range(4):
                w = self.w[xg] * self.w[yg]
                S2 = S2 + w * (-G * hgp[yg][xg] * self.bx[yg * 4 + xg])
                S3 = S3 + w * (-G * hgp[yg][xg] * self.by[yg * 4 + xg])
        return S2, S3

    def parts(self, U):
        V = _primitives(U)
        return self.faces(V, -1), self.faces(V, -2), self.source(U[0])

    def fvtd(self, U):
        """(Ut (3, M, ny, nx), mass fluxes over dx (M, ny, nx+1), over dy (M, ny+1, nx))."""
        FX, FY, (S2, S3) = self.parts(U)
        if self.wb is not None:
            FX, FY, S2, S3 = FX - self.wb[0], FY - self.wb[1], S2 - self.wb[2][0], S3 - self.wb[2][1]
        dx = torch.full_like(S2, self.d[-1])
        dy = torch.full_like(S2, self.d[-2])
        out = []
        for k, S in enumerate((torch.zeros_like(S2), S2, S3)):
            out.append(S - (FX[k][..., 1:] - FX[k][..., :-1]) / dx
                       - (FY[k][..., 1:, :] - FY[k][..., :-1, :]) / dy)
        return (torch.stack(out), FX[0] / torch.full_like(FX[0], self.d[-1]),
                FY[0] / torch.full_like(FY[0], self.d[-2]))

    def dt(self, U):
        V = _primitives(U)
        c = torch.sqrt(G * V[0])
        lx, ly = float(torch.abs(V[1] + c).max()), float(torch.abs(V[2] + c).max())
        return max(CFL * min(self.d[-1] / lx, self.d[-2] / ly), 1e-30)

    # -- the explicit schemes -------------------------------------------------
    def explicit(self, U, dt, scheme):
        f = lambda W: self.fvtd(W[:, None])[0][:, 0]  # noqa: E731
        if scheme == 1:
            return U + f(U) * dt
        if scheme == 2:
            X = [U]
            for terms, cf in SSPRK4:
                F = f(X[-1])
                acc = None
                for s, c in zip(terms[::2], terms[1::2]):
                    acc = c * X[s] if acc is None else acc + c * X[s]
                X.append(acc + (cf * F) * dt)
                last = F
            new = f(X[4])
            acc = None
            for s, c in SSPRK4_LAST:
                acc = c * X[s] if acc is None else acc + c * X[s]
            return acc + (0.08460416338212 * last) * dt + (0.22600748319395 * new) * dt
        if scheme == 3:
            K = [f(U)]
            for row in ARK65 + (BRK65,):
                s = row[0] * K[0]
                for a, k in zip(row[1:], K[1:]):
                    s = s + a * k
                X = U + s * dt
                if row is BRK65:
                    return X
                K.append(f(X))
        th = THETA[4]
        F = [f(U)] * 4
        for kk in range(1, 6):
            X = []
            for m in range(1, 4):
                acc = U
                for r in range(4):
                    acc = acc + (dt * th[m][r]) * F[r]
                X.append(acc)
            if kk == 5:
                return X[2]
            new = self.fvtd(torch.stack(X, 1))[0]
            F = [F[0]] + [new[:, i] for i in range(3)]
        return None

    # -- the modified-Patankar schemes ----------------------------------------
    def patankar(self, U, dt, scheme):
        th = THETA[scheme]
        R = len(th)
        kcorr = {5: 5, 6: 1, 7: 2}[scheme]
        ut, qx, qy = self.fvtd(U[:, None])
        F = [ut[:, 0]] * R
        Q = [(qx[0], qy[0])] * R
        h = {m: U[0] for m in range(1, R)}
        for kk in range(1, kcorr + 1):
            X = {}
            for m in range(1, R) if kk < kcorr else (R - 1,):
                X[m] = torch.stack([self.solve(U[0], h[m], Q, th[m], dt),
                                    self.moment(U[1], F, 1, th[m], dt),
                                    self.moment(U[2], F, 2, th[m], dt)])
            if kk == kcorr:
                return X[R - 1]
            new, qx, qy = self.fvtd(torch.stack([X[m] for m in range(1, R)], 1))
            F = [F[0]] + [new[:, i] for i in range(R - 1)]
            Q = [Q[0]] + [(qx[i], qy[i]) for i in range(R - 1)]
            h = {m: X[m][0] for m in X}
        return None

    @staticmethod
    def moment(u, F, v, th, dt):
        for r, c in enumerate(th):
            u = u + (dt * c) * F[r][v]
        return u

    @staticmethod
    def solve(b, hp, Q, th, dt):
        """One Patankar system by Jacobi from x = b (tolerance 1e-16, at most 1000 sweeps)."""
        roll = lambda T: (torch.roll(T, 1, -2), torch.roll(T, 1, -1),  # noqa: E731
                          torch.roll(T, -1, -1), torch.roll(T, -1, -2))
        pos = lambda t: torch.where(t > 0., t, torch.zeros_like(t))  # noqa: E731

        def quot(a, hh):
            q = (2. * hh) * a / (hh * hh + torch.clamp(hh * hh, min=HMIN))
            return torch.where(hh < HMIN, torch.zeros_like(q), q)

        hn = roll(hp)
        D = torch.ones_like(b)
        M = []
        for sl in range(4):
            m = torch.zeros_like(b)
            for r, c0 in enumerate(th):
                qx, qy = Q[r]
                s = (qy[:-1, :], qx[:, :-1], -qx[:, 1:], -qy[1:, :])[sl]
                into, out = pos(s), pos(-s)
                c = dt * c0
                if c0 > 0.:
                    m = m - c * quot(into, hn[sl])
                    D = D + c * quot(out, hp)
                else:
                    m = m + c * quot(out, hn[sl])
                    D = D - c * quot(into, hp)
            M.append(m)
        n = b.numel()
        if not 1e-16 < float(b.abs().sum()) / n:
            return torch.zeros_like(b)
        x = b
        for _ in range(1000):
            acc = torch.zeros_like(b)
            for m, t in zip(M, roll(x)):
                acc = acc + m * t
            new = (b - acc) / D
            left = float((new - x).abs().sum()) / n
            x = new
            if not 1e-16 < left:
                break
        return x

    def run(self, U, scheme, steps):
        dts = []
        for _ in range(steps):
            dt = self.dt(U)
            dts.append(dt)
            U = self.explicit(U, dt, scheme) if scheme < 5 else self.patankar(U, dt, scheme)
        return U, dts


def exact(case, seed):
    dev = _device()
    if case["call"] == "batch":
        out = {}
        for k, (family, n, steps, q) in enumerate(_jobs(case, seed)):
            if sum(j[2] for j in _jobs(case, seed)) > 200:
                return None  # the plain form is bound by its many small calls: over 20 s
            U0, Uwb, bx, by = _inputs(family, n, n, q, dev)
            U, _ = _Plain(n, n, Uwb, bx, by, 4).run(U0, case["scheme"], steps)
            out["U%02d" % k] = _host(U)
        return out
    nx, ny, steps = case["nx"], case["ny"], case["steps"]
    if nx * ny * steps * FVTDS[case["scheme"]] > 2.5e7:
        return None
    U0, Uwb, bx, by = _inputs(case["family"], nx, ny, _params(case["family"], seed), dev)
    wb = case["family"] == "lake"
    U, dts = _Plain(nx, ny, Uwb if wb else None, bx, by, case["recfix"]).run(
        U0, case["scheme"], steps)
    return {"U": _host(U), "dt": np.array(dts), "sweeps": None}
