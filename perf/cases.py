"""Performance cases of the all-bead-pairs path, through the package's public entry points.

Every case is He-4 at 0.02198 A^-3 with the Aziz 1979 pair potential (pimc_amd.workloads).
The worldlines are those of a liquid that has settled: a path integral of atoms bound
harmonically to distinct sites of a jittered cubic lattice, so links have the free-particle
variance 2 lambda tau per axis, atoms spread by about 0.6 A per axis and few pairs overlap.

listed() names what each case stands for; draw() gives more of the same ranges.
"""
import math

import numpy as np
import torch

import pimc_amd
from pimc_amd.workloads import DENSITY, LAMBDA, batched_walkers, box_side, lattice_q

PRIMITIVE = ((1.0, 1.0), (0.0, 0.0), 1)
GSF = ((2.0 / 3.0, 4.0 / 3.0), (0.0, 2.0 / 9.0), 2)
SEGMENTS = (8, 16, 32)          # Bisection segments of one Monte Carlo step
F_PAIR, F_QB, F_QMT = 50, 9, 4  # flops per pair term, per (q, bead), per (q, m, tau)


def listed():
    return [
        # the smallest system, one sample: the action with V per slice and S(q) of 729 q (|n| <= 4);
        # launches and host time set it
        {"name": "sample_n16_m125", "kind": "sample", "N": 16, "M": 125, "nmax": 4},
        # one Monte Carlo step of an ordinary walker: the full action and the Delta V of three
        # Bisection segments
        {"name": "step_n256_m167", "kind": "step", "N": 256, "M": 167, "mode": 0, "gsf": False},
        # the same step under the GSF action (gradient-corrected, the reference's default action)
        {"name": "step_gsf_n256_m166", "kind": "step", "N": 256, "M": 166, "mode": 0, "gsf": True},
        # a centre-of-mass move: Delta V of a whole worldline, odd sizes, exact table values
        {"name": "com_n181_m143_table", "kind": "com", "N": 181, "M": 143, "mode": 2},
        # the energy estimators of one sample under the GSF action: thermodynamic and virial
        {"name": "energy_n256_m166", "kind": "energy", "N": 256, "M": 166},
        # F(q, tau) of an ordinary walker: every lattice q with |q| <= 3 A^-1, all lags
        {"name": "isf_n256_m167", "kind": "isf", "N": 256, "M": 167, "qmax": 3.0},
        # many uneven walkers in one launch, tiles as the batch sets them, graph replay
        {"name": "batch_512_walkers", "kind": "batch", "walkers": 512},
        # an ensemble of device-resident Markov chains: staging, bisection and centre-of-mass moves
        {"name": "chains_128_n64_m96", "kind": "chains", "chains": 128, "N": 64, "M": 96, "moves": 12},
        # a burst of Delta V requests and a few S(q) requests against the server's resident chains
        {"name": "served_64_chains", "kind": "served", "chains": 64, "requests": 96},
        # odd sizes in the FP64 mode: the full action after a bead has moved
        {"name": "action_n777_m61_fp64", "kind": "action", "N": 777, "M": 61, "mode": 1},
        # the large system (rc = L/2): the full action after a bead has moved
        {"name": "action_n2048_m250", "kind": "action", "N": 2048, "M": 250, "mode": 0},
        # the large system's structure factors: S(q) and F(q, tau) on the 100 401 q with |q| <= 4 A^-1
        {"name": "sq_isf_n2048_m250", "kind": "sq_isf", "N": 2048, "M": 250, "qmax": 4.0},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["sample", "step", "step", "com", "energy", "isf", "batch", "chains", "served",
                       "action", "action", "sq_isf"])
    if kind == "sample":
        return {"kind": kind, "N": _log(rng, 8, 64), "M": _log(rng, 20, 256), "nmax": rng.randint(2, 5)}
    if kind == "step":
        return {"kind": kind, "N": _log(rng, 16, 512), "M": _log(rng, 40, 320), "mode": rng.choice([0, 0, 1, 2]),
                "gsf": rng.random() < 0.5}
    if kind == "com":
        return {"kind": kind, "N": _log(rng, 16, 1024), "M": _log(rng, 20, 320), "mode": rng.choice([0, 0, 1, 2])}
    if kind == "energy":
        return {"kind": kind, "N": _log(rng, 16, 512), "M": 2 * _log(rng, 16, 128)}
    if kind == "isf":
        return {"kind": kind, "N": _log(rng, 16, 512), "M": _log(rng, 40, 320), "qmax": round(rng.uniform(1.0, 3.0), 2)}
    if kind == "batch":
        return {"kind": kind, "walkers": _log(rng, 8, 512)}
    if kind == "chains":
        return {"kind": kind, "chains": _log(rng, 4, 128), "N": _log(rng, 16, 128), "M": _log(rng, 48, 128),
                "moves": 3 * rng.randint(2, 6)}
    if kind == "served":
        return {"kind": kind, "chains": _log(rng, 8, 64), "requests": _log(rng, 8, 128)}
    if kind == "action":
        N = _log(rng, 128, 2048)
        return {"kind": kind, "N": N, "M": _log(rng, 16, 250), "mode": rng.choice([0, 0, 0, 1, 2])}
    return {"kind": kind, "N": _log(rng, 256, 2048), "M": _log(rng, 40, 250), "qmax": round(rng.uniform(1.5, 4.0), 2)}


# ---- inputs -------------------------------------------------------------------------------------
def _tau(M):
    return 0.004 if M >= 40 else 0.01


def _wrap(r, L):
    return r - L * np.floor(r / L + 0.5)


def _worldlines(rng, L, M, N, tau):
    """beads [M][N][3]: harmonically bound path integrals around the sites of a jittered cubic lattice."""
    k = int(math.ceil(N ** (1.0 / 3.0) - 1e-9))
    site = rng.permutation(k ** 3)[:N]
    c = np.stack([site // (k * k), (site // k) % k, site % k], axis=-1)
    centre = (c + 0.5) * (L / k) - 0.5 * L + rng.normal(scale=0.15, size=(N, 3))
    modes = np.arange(M // 2 + 1)
    # a chain of M links of stiffness 1 / (2 lambda tau); the binding spreads a bead by about 0.6 A
    link = (2.0 - 2.0 * np.cos(2.0 * np.pi * modes / M)) / (2.0 * LAMBDA * tau)
    bind = 2.0 * LAMBDA * tau / (4.0 * 0.6 ** 4)
    sd = np.sqrt(M / (link + bind))
    z = rng.normal(size=(modes.size, N, 3, 2)) * math.sqrt(0.5)
    coef = (z[..., 0] + 1j * z[..., 1]) * sd[:, None, None]
    coef[0] = math.sqrt(2.0) * z[0, ..., 0] * sd[0]
    if M % 2 == 0:
        coef[-1] = math.sqrt(2.0) * z[-1, ..., 0] * sd[-1]
    return np.ascontiguousarray(_wrap(np.fft.irfft(coef, n=M, axis=0) + centre[None], L))


def _segment(rng, beads, L, tau, seg, M, N):
    """A Bisection proposal: the seg - 1 beads between two fixed ends of a worldline, redrawn as a free bridge."""
    start, p = int(rng.integers(M)), int(rng.integers(N))
    seg = min(seg, M - 1)
    sl = np.array([(start + k) % M for k in range(1, seg)], dtype=np.int32)
    a, span = beads[start, p], _wrap(beads[(start + seg) % M, p] - beads[start, p], L)
    w = np.cumsum(rng.normal(scale=math.sqrt(2.0 * LAMBDA * tau), size=(seg, 3)), axis=0)
    f = (np.arange(1, seg) / seg)[:, None]
    new = a + f * span + w[:-1] - f * w[-1]
    return np.stack([sl, np.full(seg - 1, p, dtype=np.int32)], axis=-1), _wrap(new, L)


def _com(rng, beads, L, M, N):
    p = int(rng.integers(N))
    sp = np.stack([np.arange(M, dtype=np.int32), np.full(M, p, dtype=np.int32)], axis=-1)
    return sp, _wrap(beads[:, p] + rng.normal(scale=0.3, size=3), L)


def _system(case, rng):
    N, M = case["N"], case["M"]
    L, tau = box_side(N, DENSITY), _tau(M)
    return N, M, L, tau, _worldlines(rng, L, M, N, tau)


def _context(L, M, N, tau, beads, rc_frac=1.0, mode=0, action=PRIMITIVE):
    ctx = pimc_amd.Context(L, M, N, tau, LAMBDA, rc_frac * L, v_mode=mode)
    ctx.upload_path(beads)
    if action is not PRIMITIVE:
        ctx.set_action_factors(*action)
    return ctx


def _walkers(case, seed):
    ws = batched_walkers(case["walkers"], seed=seed)
    rng = np.random.default_rng(seed)
    return ws, [_worldlines(rng, w["side"], w["M"], w["N"], w["tau"]) for w in ws]


def _served(case, seed):
    """Chains of uneven sizes and a burst of requests: one in 16 an S(q), one in 10 of the others a whole worldline."""
    rng = np.random.default_rng(seed)
    chains, reqs = [], []
    for _ in range(case["chains"]):
        N, M = int(rng.integers(32, 513)), int(rng.integers(64, 257))
        L, tau = box_side(N, DENSITY), 1.0 / (M * rng.uniform(1.0, 3.0))
        chains.append((L, M, N, tau, _worldlines(rng, L, M, N, tau)))
    for k in range(case["requests"]):
        c = int(rng.integers(case["chains"]))
        L, M, N, tau, beads = chains[c]
        if k % 16 == 15:
            reqs.append((c, lattice_q(L, nmax=2)))
        elif rng.random() < 0.1:
            reqs.append((c,) + _com(rng, beads, L, M, N))
        else:
            reqs.append((c,) + _segment(rng, beads, L, tau, int(rng.integers(4, 65)), M, N))
    return chains, reqs


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "batch":
        ws, beads = _walkers(case, seed)
        bt = pimc_amd.Batch(ws)
        for k, b in enumerate(beads):
            bt.upload(k, b)
        bt.use_graph(True)
        s["batch"] = bt
        return s
    if kind == "chains":
        rng = np.random.default_rng(seed)
        s["ctx"], s["chains"] = [], []
        for c in range(case["chains"]):
            N, M, L, tau, beads = _system(case, rng)
            s["ctx"].append(_context(L, M, N, tau, beads))
            s["chains"].append(pimc_amd.Chain(s["ctx"][-1], 5000 + seed % 100000 + c, 16, 4, True, 1, 0.1))
        s["kinds"] = ["staging", "bisection", "com"] * (case["moves"] // 3)
        return s
    if kind == "served":
        chains, reqs = _served(case, seed)
        sv = pimc_amd.Server(sum(64 * M * N + 65536 for _, M, N, _, _ in chains))
        ids = [sv.add_chain(L, M, N, tau, LAMBDA, L, b) for L, M, N, tau, b in chains]
        s["server"], s["requests"] = sv, [(ids[r[0]],) + r[1:] for r in reqs]
        return s
    rng = np.random.default_rng(seed)
    N, M, L, tau, beads = _system(case, rng)
    if kind == "sample":
        s["ctx"], s["q"] = _context(L, M, N, tau, beads), lattice_q(L, nmax=case["nmax"])
    elif kind == "step":
        s["ctx"] = _context(L, M, N, tau, beads, 1.0, case["mode"], GSF if case["gsf"] else PRIMITIVE)
        s["moves"] = [s["ctx"].prepare_delta(*_segment(rng, beads, L, tau, g, M, N)) for g in SEGMENTS]
    elif kind == "com":
        s["ctx"] = _context(L, M, N, tau, beads, 1.0, case["mode"])
        s["move"] = _com(rng, beads, L, M, N)
    elif kind == "energy":
        s["ctx"] = _context(L, M, N, tau, beads, 1.0, 0, GSF)
    elif kind == "isf":
        s["ctx"], s["q"] = _context(L, M, N, tau, beads), lattice_q(L, qmag_max=case["qmax"])
        s["out"] = pimc_amd.pinned_empty((s["q"].shape[0], M))
    elif kind == "action":
        s["ctx"] = _context(L, M, N, tau, beads, 0.5 if N >= 1024 else 1.0, case["mode"])
        s["bead"], s["pos"] = np.array([[M // 2, N // 3]], dtype=np.int32), _moved(beads, M, N, L)
    else:
        s["ctx"], s["q"] = _context(L, M, N, tau, beads, 0.5), lattice_q(L, qmag_max=case["qmax"])
        s["out"] = pimc_amd.pinned_empty((s["q"].shape[0], M))
    return s


def _moved(beads, M, N, L):
    return _wrap(beads[M // 2, N // 3] + np.array([0.1, -0.05, 0.07]), L)[None]


def run(s):
    kind = s["kind"]
    if kind == "sample":
        action, v = s["ctx"].potentialAction(with_slices=True)
        return {"action": action, "v": v, "sq": s["ctx"].ssf(s["q"])}
    if kind == "step":
        out = {"action": s["ctx"].potentialAction()}
        for g, m in zip(SEGMENTS, s["moves"]):
            out["dv%d" % g] = s["ctx"].delta_action_prepared(m)[:3].copy()
        return out
    if kind == "com":
        return {"dv": s["ctx"].delta_action(*s["move"])}
    if kind == "energy":
        e, v = s["ctx"].energy(), s["ctx"].virial_energy(5)
        return {"energy": np.array(list(e.values())), "virial": np.array(list(v.values()))}
    if kind == "isf":
        return {"isf": s["ctx"].isf(s["q"], out=s["out"])}
    if kind == "batch":
        return {"actions": s["batch"].potentialAction()}
    if kind == "chains":
        acc, info, _ = pimc_amd.run_chains_device(s["chains"], s["kinds"])
        return {"accepted": acc, "info": info, "beads": np.stack([c.positions() for c in s["chains"]])}
    if kind == "served":
        sv = s["server"]
        ids = [sv.submit_ssf(*r) if len(r) == 2 else sv.submit(*r) for r in s["requests"]]
        dv, sq = [], []
        for rid, r in zip(ids, s["requests"]):
            if len(r) == 2:
                sq.append(sv.wait_ssf(rid)[0])
            else:
                dv.append(sv.wait(rid)["raw"][:3])
        return {"dv": np.array(dv), "sq": np.concatenate(sq) if sq else np.zeros(1)}
    if kind == "action":
        s["ctx"].update_beads(s["bead"], s["pos"])
        action, v = s["ctx"].potentialAction(with_slices=True)
        return {"action": action, "v": v}
    return {"sq": s["ctx"].ssf(s["q"]), "isf": s["ctx"].isf(s["q"], out=s["out"])}


# ---- what a pass cannot do without -------------------------------------------------------------
def _nq(case, L):
    if "nmax" in case:
        return lattice_q(L, nmax=case["nmax"]).shape[0]
    return lattice_q(L, qmag_max=case["qmax"]).shape[0]


def work(case):
    kind = case["kind"]
    if kind == "batch":
        # the first 512 walkers of a seed stand for every seed's
        ws = batched_walkers(case["walkers"], seed=1)
        return {"bytes": sum(24 * w["M"] * w["N"] + 8 for w in ws),
                "flops": sum(F_PAIR * w["M"] * w["N"] * (w["N"] - 1) // 2 for w in ws)}
    if kind == "served":
        chains, reqs = _served(case, 1)
        b = f = 0
        for r in reqs:
            L, M, N, _, _ = chains[r[0]]
            if len(r) == 2:
                b += 24 * M * N + 32 * len(r[1])
                f += len(r[1]) * (F_QB * M * N + F_QMT * M)
            else:
                b += 24 * N * len(r[1]) + 32 * len(r[1]) + 24
                f += F_PAIR * 2 * len(r[1]) * (N - 1)
        return {"bytes": b, "flops": f}
    N, M = case["N"], case["M"]
    L, beads = box_side(N, DENSITY), 24 * M * N
    pairs = M * N * (N - 1) // 2
    if kind == "chains":
        # a rotation moves about 12 + 11 + M beads, each scored at its old and its new position
        moved = (23 + M) * (case["moves"] // 3)
        return {"bytes": case["chains"] * 2 * beads, "flops": case["chains"] * F_PAIR * 2 * moved * (N - 1)}
    if kind == "com":
        return {"bytes": beads + 48 * M, "flops": F_PAIR * 2 * M * (N - 1)}
    if kind == "step":
        dv = 2 * (N - 1) * sum(g - 1 for g in SEGMENTS)
        if not case["gsf"]:
            return {"bytes": beads + 8, "flops": F_PAIR * (pairs + dv)}
        # gradients of the pairs of the corrected (odd) slices, and the three-body terms of the moved beads there
        three = 2 * (N - 1) * (N - 2) // 2 * sum(g - 1 for g in SEGMENTS) // 2
        return {"bytes": beads + 8, "flops": F_PAIR * (pairs + pairs // 2 + dv + three)}
    if kind == "energy":
        return {"bytes": 2 * beads + 28 * 8, "flops": F_PAIR * (2 * pairs + pairs // 2 + 2 * pairs)}
    if kind == "action":
        return {"bytes": beads + 16 * M, "flops": F_PAIR * pairs}
    nq = _nq(case, L)
    rho = nq * (F_QB * M * N + F_QMT * M)
    if kind == "sample":
        return {"bytes": 2 * beads + 16 * M + 32 * nq, "flops": F_PAIR * pairs + rho}
    # q and -q have the same S and F: one of each pair has to be computed
    if kind == "isf":
        return {"bytes": beads + 24 * nq + 8 * nq * M, "flops": (rho + F_QMT * nq * M * M) // 2}
    return {"bytes": 2 * beads + 56 * nq + 8 * nq * M, "flops": (2 * rho + F_QMT * nq * M * M) // 2}


# ---- the same in 64 bits, plain torch ----------------------------------------------------------
_AZ = {"eps": 10.8, "rm": 2.9673, "D": 1.241314, "alpha": 13.353384, "C6": 1.3732412, "C8": 0.4253785,
       "C10": 0.1781, "A": 0.5448504e6}
_radius = {}


def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _t(a):
    return torch.as_tensor(np.asarray(a), device=_dev())


def _bin_radius(L):
    """r of every bin of the pair potential's step table: dr = 1e-6 rm, added up bin by bin."""
    n = int(0.5 * math.sqrt(3.0) * L / (1e-6 * _AZ["rm"])) + 2
    if _radius.get("n", 0) < n:
        _radius.update(n=n, r=_t(np.concatenate([[0.0], np.cumsum(np.full(n, 1e-6 * _AZ["rm"]))])))
    return _radius["r"]


def _aziz(r, L, what):
    """V, dV/dr or d2V/dr2 of the Aziz 1979 potential at the bins of the separations r (r > 0)."""
    a = _AZ
    k = (r / (1e-6 * a["rm"])).to(torch.int64)
    x = _bin_radius(L)[k] / a["rm"]
    rep = a["A"] * torch.exp(-a["alpha"] * x)
    i = 1.0 / x
    t = a["D"] * i - 1.0
    near = x < a["D"]
    F = torch.where(near, torch.exp(-t * t), torch.ones_like(x))
    i2 = i * i
    c6 = i2 * i2 * i2
    c8, c10 = c6 * i2, c6 * i2 * i2
    p0 = a["C6"] * c6 + a["C8"] * c8 + a["C10"] * c10
    if what == 0:
        return a["eps"] * (rep - p0 * F)
    dF = torch.where(near, 2.0 * a["D"] * i2 * t * F, torch.zeros_like(x))
    p1 = (6.0 * a["C6"] * c6 + 8.0 * a["C8"] * c8 + 10.0 * a["C10"] * c10) * i
    if what == 1:
        return a["eps"] / a["rm"] * (-a["alpha"] * rep + p1 * F - p0 * dF)
    D = a["D"]
    d2F = torch.where(near, 2.0 * D * i2 * i * (2.0 * D ** 3 * i2 * i - 4.0 * D * D * i2 - D * i + 2.0) * F,
                      torch.zeros_like(x))
    p2 = (42.0 * a["C6"] * c6 + 72.0 * a["C8"] * c8 + 110.0 * a["C10"] * c10) * i2
    return a["eps"] / a["rm"] ** 2 * (a["alpha"] ** 2 * rep - p2 * F + 2.0 * p1 * dF - p0 * d2F)


def _sep(a, b, L):
    d = a - b
    return d - L * torch.floor(d * (1.0 / L) + 0.5)


def _slices(M, N):
    step = max(1, 24_000_000 // (N * N))
    return [slice(m, min(M, m + step)) for m in range(0, M, step)]


def _v_slices(beads, L):
    """V of each slice: every pair once."""
    b = _t(beads)
    M, N = b.shape[:2]
    out = []
    for s in _slices(M, N):
        r = torch.linalg.vector_norm(_sep(b[s, :, None], b[s, None, :], L), dim=-1)
        eye = torch.eye(N, dtype=torch.bool, device=r.device)
        v = _aziz(r.masked_fill(eye, _AZ["rm"]), L, 0).masked_fill(eye, 0.0)
        out.append(0.5 * v.sum(dim=(1, 2)))
    return torch.cat(out)


def _forces(beads, L):
    """gradV of the pair potential per bead [M][N][3] and the T-matrix applied to it."""
    b = _t(beads)
    M, N = b.shape[:2]
    F, TF = [], []
    for s in _slices(M, 3 * N):
        d = _sep(b[s, :, None], b[s, None, :], L)
        eye = torch.eye(N, dtype=torch.bool, device=d.device)
        r = torch.linalg.vector_norm(d, dim=-1).masked_fill(eye, _AZ["rm"])
        g = _aziz(r, L, 1).masked_fill(eye, 0.0)
        h = _aziz(r, L, 2).masked_fill(eye, 0.0)
        f = (g / r)[..., None] * d
        F.append(f.sum(dim=2))
        m = g.abs()
        T = torch.einsum("mij,mija,mijb->miab", h / r ** 2 - m / r ** 3, d, d)
        T = T + (m / r).sum(dim=2)[..., None, None] * torch.eye(3, dtype=d.dtype, device=d.device)
        TF.append((T * F[-1][..., None, :]).sum(dim=-1))
    return torch.cat(F), torch.cat(TF)


def _vfactor(action, M):
    return _t(np.array([action[0][m % 2] for m in range(M)])), _t(np.array([action[1][m % 2] for m in range(M)]))


def _total(beads, L, tau, action, v=None):
    vf, gf = _vfactor(action, beads.shape[0])
    a = (vf * tau * (_v_slices(beads, L) if v is None else v)).sum()
    if max(action[1]) > 0:
        F, _ = _forces(beads, L)
        a = a + (gf * tau ** 3 * LAMBDA * (F * F).sum(dim=(1, 2))).sum()
    return float(a)


def _bead_action(beads, sp, pos, L, tau, action):
    """Sum over the listed beads at the positions pos: Vnn, and the change of the slice's force sum with the GSF factors."""
    b = _t(beads)
    vf, gf = _vfactor(action, beads.shape[0])
    tot = 0.0
    for (m, i), p in zip(np.asarray(sp).tolist(), _t(pos)):
        o = torch.cat([b[m, :i], b[m, i + 1:]])
        d = _sep(o, p, L)
        r = torch.linalg.vector_norm(d, dim=-1)
        tot += float(vf[m] * tau * _aziz(r, L, 0).sum())
        if float(gf[m]) > 0:
            f1 = (_aziz(r, L, 1) / r)[:, None] * d                 # force on each other bead from this one
            R, _ = _forces(o[None].cpu().numpy(), L)
            g2 = (f1 * f1).sum() + 2.0 * (f1 * R[0]).sum() + f1.sum(dim=0).square().sum()
            tot += float(gf[m] * tau ** 3 * LAMBDA * g2)
    return tot


def _delta(beads, sp, new, L, tau, action=PRIMITIVE):
    old = beads[np.asarray(sp)[:, 0], np.asarray(sp)[:, 1]]
    a, b = (_bead_action(beads, sp, p, L, tau, action) for p in (old, new))
    return np.array([a, b, b - a])


def _rho(beads, L, q):
    """Density modes [nq][M] of lattice q."""
    n = torch.as_tensor(np.rint(q * L / (2.0 * math.pi)).astype(np.int64), device=_dev())
    b = _t(beads) / L
    h = int(n.abs().max())
    rows, row = torch.unique(n[:, :2], dim=0, return_inverse=True)
    k = torch.arange(-h, h + 1, device=b.device, dtype=torch.float64)
    out = torch.empty((n.shape[0], b.shape[0]), dtype=torch.complex128, device=b.device)
    for m in range(b.shape[0]):
        turn = b[m].T[:, None, :] * k[None, :, None]                # [3][2h + 1][N]
        turn = 2.0 * math.pi * (turn - torch.round(turn))
        ph = torch.complex(torch.cos(turn), torch.sin(turn))
        xy = ph[0][rows[:, 0] + h] * ph[1][rows[:, 1] + h]
        out[:, m] = (xy @ ph[2].T.contiguous())[row, n[:, 2] + h]
    return out


def _sq(rho, N):
    return ((rho.real ** 2 + rho.imag ** 2).sum(dim=1) / N).cpu().numpy()


def _isf(rho, N):
    out = []
    for c in torch.split(rho, 8192):
        f = torch.fft.fft(c, dim=1)
        out.append((torch.fft.ifft(f.real ** 2 + f.imag ** 2, dim=1).real / N).cpu())
    return torch.cat(out).numpy()


def _estimators(beads, L, tau, W=5):
    """The thermodynamic (9) and virial (19) columns under the GSF action, closed worldlines, mu = 0."""
    vfac, gfac, period = GSF
    M, N = beads.shape[:2]
    vf, gf = _vfactor(GSF, M)
    b, v = _t(beads), _v_slices(beads, L)
    F, TF = _forces(beads, L)
    g2 = (F * F).sum(dim=(1, 2))
    vol, x = L ** 3, _AZ["rm"] / L
    tail = N * N / vol * -2.0 * math.pi * _AZ["eps"] * _AZ["rm"] ** 3 * (
        _AZ["C6"] * x ** 3 / 3.0 + _AZ["C8"] * x ** 5 / 5.0 + _AZ["C10"] * x ** 7 / 7.0)
    vel = _sep(torch.roll(b, -1, 0), b, L)
    vel2 = float((vel * vel).sum())
    t1 = float((gf * tau ** 3 * g2).sum()) * LAMBDA / (tau * M)
    dU = vf * v + 3.0 * gf * tau * tau * LAMBDA * g2
    t2 = float(dU.sum()) / M
    K = -vel2 / (4.0 * LAMBDA * tau) / (tau * M) + 1.5 / tau * N + t1
    V, vop = t2 - t1 + tail, float(v[::period].sum()) / (M // period) + tail
    energy = [K, V, 0.0, vop, K + V, K + V, K / N, V / N, (K + V) / N]
    more, less = torch.zeros_like(b), torch.zeros_like(b)
    com, fwd = torch.zeros_like(b), torch.zeros_like(b)
    for g in range(W):
        if g:
            more = more + torch.roll(vel, -(g - 1), 0)
            less = less - torch.roll(vel, g, 0)
        com = com + 2.0 * b + more + less
        fwd = fwd + torch.roll(vel, -g, 0)
    delta = _sep(b, com / (2.0 * W), L)
    c2 = 2.0 * gf * tau ** 3 * LAMBDA

    def dot(u, w):
        return (u * w).sum(dim=(1, 2))
    beta = M * tau
    T1 = 1.5 * N / (W * tau)
    T2 = -float((fwd * vel).sum()) / (4.0 * W * tau ** 2 * LAMBDA * M)
    T3 = float((vf * tau * dot(F, delta)).sum()) / (2.0 * beta)
    T4 = float((c2 * dot(TF, delta)).sum()) / beta
    T5 = float(dU.sum()) / M
    vkin = float((gf * tau ** 3 * LAMBDA * g2).sum()) / (0.5 * beta)
    P = 3.0 * N - vel2 / (2.0 * LAMBDA * tau * M)
    P -= float((vf * tau * dot(F, b) + c2 * dot(TF, b)).sum()) / (2.0 * M)
    P /= 3.0 * tau * vol
    th = -vel2 / (4.0 * LAMBDA * tau) / (tau * M) + 1.5 / tau * N + T5 + tail
    vo = float(v[::2].sum()) / (0.5 * M) + tail
    E, Kcv = T1 + T2 + T3 + T4 + T5 + tail, T1 + T2 + T3 + T4 + vkin
    dE = (-T1 - 2.0 * T2 + 2.0 * T4) / tau + float((6.0 * gf * tau * LAMBDA * g2).sum()) / M
    dE *= beta * beta / M
    EE = E * th * beta * beta
    virial = [E - vo + E * beta * dE, Kcv, vo, E - Kcv, E, E, (E - vo) / N, Kcv / N, vo / N, (E - Kcv) / N, E / N,
              EE, E * beta, dE, EE * E * beta, 0.0, EE * dE, th, P]
    return {"energy": np.array(energy), "virial": np.array(virial)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "chains":
        return None     # a Markov chain's decisions follow its own random stream
    if kind == "batch":
        ws, beads = _walkers(case, seed)
        return {"actions": np.array([_total(b, w["side"], w["tau"], PRIMITIVE) for w, b in zip(ws, beads)])}
    if kind == "served":
        chains, reqs = _served(case, seed)
        dv, sq = [], []
        for r in reqs:
            L, M, N, tau, beads = chains[r[0]]
            if len(r) == 2:
                sq.append(_sq(_rho(beads, L, r[1]), N))
            else:
                dv.append(_delta(beads, r[1], r[2], L, tau))
        return {"dv": np.array(dv), "sq": np.concatenate(sq) if sq else np.zeros(1)}
    rng = np.random.default_rng(seed)
    N, M, L, tau, beads = _system(case, rng)
    if kind == "step":
        act = GSF if case["gsf"] else PRIMITIVE
        out = {"action": _total(beads, L, tau, act)}
        for g in SEGMENTS:
            out["dv%d" % g] = _delta(beads, *_segment(rng, beads, L, tau, g, M, N), L, tau, act)
        return out
    if kind == "com":
        return {"dv": _delta(beads, *_com(rng, beads, L, M, N), L, tau)}
    if kind == "energy":
        return _estimators(beads, L, tau)
    if kind in ("sample", "action"):
        if kind == "action":
            beads[M // 2, N // 3] = _moved(beads, M, N, L)[0]
        v = _v_slices(beads, L)
        out = {"action": _total(beads, L, tau, PRIMITIVE, v),
               "v": torch.stack([torch.zeros_like(v), v], dim=1).cpu().numpy()}
        if kind == "sample":
            out["sq"] = _sq(_rho(beads, L, lattice_q(L, nmax=case["nmax"])), N)
        return out
    rho = _rho(beads, L, lattice_q(L, qmag_max=case["qmax"]))
    if kind == "isf":
        return {"isf": _isf(rho, N)}
    return {"sq": _sq(rho, N), "isf": _isf(rho, N)}
