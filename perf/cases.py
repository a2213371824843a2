"""The calls that a user of this framework has it do, as cases to be timed and compared.

A case names one public entry point, the bodies it is given and its options.  listed() holds the
cases, draw() gives more of the same ranges, prepare() makes the bodies and the context a program
keeps, run() is one pass through the entry point, exact() the same result from plain torch in 64
bits.  Bodies come from taichi_collisional_amd.ics, the initial conditions that the benchmark and
the tests use; every context gets a root shift of its own from the seed, so that one state gives
the same tree on every pass.
"""
import math

import numpy as np
import torch

import taichi_collisional_amd as tca
from taichi_collisional_amd import flops, ics, learn

# the path's options by kind:
#   eval       Fmm.eval: force, potential and jerk (direct sum below direct_below bodies)
#   clusters   Fmm.eval_clusters: many independent clusters in one evaluation
#   bodies     Fmm.get_force_and_potential on host Body records, both copies included
#   master     Fmm.master_eval: all-pairs force and potential, with the time-step estimate or without
#   evolve     Fmm.master_evolve: one do_evolve of the step loop


def listed():
    return [
        # a few stars: below direct_below the call is the direct sum, launches and latency count
        {"name": "eval_direct_n1009", "kind": "eval", "model": "plummer", "n": 1009, "p": 12,
         "theta": 0.4},
        # the smallest systems that take the tree path, an odd size
        {"name": "eval_n10007_p12", "kind": "eval", "model": "plummer", "n": 10007, "p": 12,
         "theta": 0.4},
        # an ordinary star cluster at the smaller order
        {"name": "eval_n65536_p10", "kind": "eval", "model": "plummer", "n": 65536, "p": 10,
         "theta": 0.5},
        # the reference's Makefiles build orders 20 and 24: a high-accuracy run
        {"name": "eval_n131072_p20", "kind": "eval", "model": "plummer", "n": 131072, "p": 20,
         "theta": 0.5},
        # the reference's default pass: p = 2 pre-pass and error-controlled opening
        {"name": "eval_error_mac_n300007_p12", "kind": "eval", "model": "plummer", "n": 300007,
         "p": 12, "theta": 0.4, "mac": "error"},
        # the benchmark's workload
        {"name": "eval_n1048576_p12", "kind": "eval", "model": "plummer", "n": 1048576, "p": 12,
         "theta": 0.4},
        # a mass spectrum with binaries and the mixed-precision near field, the largest system
        {"name": "eval_kroupa_mixed_n4194304_p12", "kind": "eval", "model": "kroupa",
         "n": 4194304, "p": 12, "theta": 0.4, "near": "hilo"},
        # opening angle chosen per leaf by the trained network, a cuspy model with a deep tree
        {"name": "eval_learned_n262144_p12", "kind": "eval", "model": "dehnen", "n": 262144,
         "p": 12, "theta": 0.4, "learned": True},
        # 256 clusters of 2^10 .. 2^16 bodies in one evaluation
        {"name": "clusters_256_p8", "kind": "clusters", "ncl": 256, "lo": 1024, "hi": 65536,
         "p": 8, "theta": 0.5},
        # a host program's Body records in and out
        {"name": "bodies_n250000_p12", "kind": "bodies", "model": "plummer", "n": 250000, "p": 12,
         "theta": 0.4},
        # the master build's default call: all pairs and time steps over the leaves
        {"name": "master_steps_n65536", "kind": "master", "model": "plummer", "n": 65536,
         "ncrit": 300, "steps": True},
        # one step of the hierarchical integrator
        {"name": "evolve_n4096", "kind": "evolve", "model": "plummer", "n": 4096, "ncrit": 300,
         "dt": 1.0 / 1024},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["eval", "eval", "eval", "high", "direct", "error", "mixed", "learned",
                       "clusters", "bodies", "master", "evolve"])
    model = rng.choice(["plummer", "plummer", "dehnen", "kroupa"])
    theta = round(rng.uniform(0.4, 0.65), 2)
    if kind == "eval":
        return {"kind": "eval", "model": model, "n": _log_int(rng, 8001, 1 << 20),
                "p": rng.randint(6, 14), "theta": theta, "masked": rng.random() < 0.25}
    if kind == "high":
        return {"kind": "eval", "model": model, "n": _log_int(rng, 8001, 1 << 17),
                "p": rng.choice([16, 18, 20, 22, 24]), "theta": max(theta, 0.5)}
    if kind == "direct":
        return {"kind": "eval", "model": model, "n": _log_int(rng, 16, 7999), "p": 12,
                "theta": 0.4, "masked": rng.random() < 0.25}
    if kind == "error":
        return {"kind": "eval", "model": model, "n": _log_int(rng, 8001, 1 << 19),
                "p": rng.choice([10, 12, 14]), "theta": 0.4, "mac": "error"}
    if kind == "mixed":
        return {"kind": "eval", "model": "kroupa", "n": _log_int(rng, 1 << 15, 1 << 20), "p": 12,
                "theta": round(rng.uniform(0.4, 0.5), 2), "near": rng.choice(["float", "hilo"])}
    if kind == "learned":
        return {"kind": "eval", "model": rng.choice(["plummer", "dehnen"]),
                "n": _log_int(rng, 1 << 15, 1 << 19), "p": 12, "theta": 0.4, "learned": True}
    if kind == "clusters":
        return {"kind": "clusters", "ncl": _log_int(rng, 4, 128), "lo": 1024, "hi": 65536,
                "p": rng.choice([8, 10]), "theta": 0.5}
    if kind == "bodies":
        return {"kind": "bodies", "model": model, "n": _log_int(rng, 8001, 1 << 18), "p": 12,
                "theta": theta}
    if kind == "master":
        return {"kind": "master", "model": model, "n": _log_int(rng, 500, 1 << 16),
                "ncrit": rng.choice([64, 128, 300]), "steps": rng.random() < 0.75}
    return {"kind": "evolve", "model": "plummer", "n": _log_int(rng, 256, 4096), "ncrit": 300,
            "dt": 1.0 / 1024}


# ---- inputs -------------------------------------------------------------------------------------
def _bodies(model, n, seed):
    if model == "dehnen":
        return ics.dehnen(n, gamma=1.5, seed=seed)
    return {"plummer": ics.plummer, "kroupa": ics.kroupa_binaries}[model](n, seed=seed)


def _cluster_starts(case):
    """The clusters' sizes are the case's own: every seed has the same ones."""
    rng = np.random.default_rng(case["ncl"])
    sizes = np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]), case["ncl"]))
    return np.concatenate([[0], np.cumsum(sizes.astype(np.int64))]).astype(np.int32)


def _inputs(case, seed):
    """(x, v, m, flags or None) on the host."""
    if case["kind"] == "clusters":
        st = _cluster_starts(case)
        x, v, m = (np.concatenate(a) for a in zip(*[
            ics.plummer(int(b - a), seed=[seed, k]) for k, (a, b) in enumerate(zip(st, st[1:]))]))
    else:
        x, v, m = _bodies(case["model"], case["n"], seed)
    flags = None
    if case.get("masked"):
        # a subsystem's force call: some bodies take no force, some exert none
        rng = np.random.default_rng([seed, 5])
        flags = ((rng.random(m.size) < 0.8) | ((rng.random(m.size) < 0.9).astype(np.uint8) << 1)
                 ).astype(np.uint8)
    return x, v, m, flags


def _context(case, seed):
    fmm = tca.Fmm(p=case.get("p", 12), ncrit=case.get("ncrit", 64), theta=case.get("theta", 0.4),
                  mac=tca.TC_MAC_ERROR if case.get("mac") == "error" else tca.TC_MAC_THETA,
                  direct_below=0 if case["kind"] in ("clusters", "master", "evolve") else 8000)
    fmm.set_shift(np.random.default_rng([seed, 3]).uniform(-0.5, 0.49, 3))
    if case.get("near"):
        fmm.set_precision({"float": tca.TC_P2P_MIXED, "hilo": tca.TC_P2P_MIXED_HILO}[case["near"]])
    if case.get("learned"):
        learn.apply_model(fmm, learn.load_model())
    return fmm


_EVOLVE = (("pos", 3), ("pos_e", 3), ("vel", 3), ("acc", 3), ("mass", 1), ("timestep", 1),
           ("pot", 1), ("acc_old", 1))


def _views(flat, n):
    out, at = {}, 0
    for key, width in _EVOLVE:
        part = flat[at * n:(at + width) * n]
        out[key] = part.view(n, 3) if width == 3 else part
        at += width
    return out


def prepare(case, seed):
    x, v, m, flags = _inputs(case, seed)
    s = {"case": case, "fmm": _context(case, seed)}
    if case["kind"] == "bodies":
        b = np.zeros(m.size, dtype=tca.body_dtype)
        b["X"], b["V"], b["q"] = x, v, m
        b["index"] = np.arange(m.size)
        b["issink"] = b["issource"] = 1
        s["bodies"] = b
        return s
    x, v, m = (torch.from_numpy(a).cuda() for a in (x, v, m))
    if case["kind"] == "evolve":
        n = m.shape[0]
        s["start"] = torch.zeros(14 * n + 2 * n, dtype=torch.float64, device="cuda")
        first = _views(s["start"], n)
        first["pos"].copy_(x)
        first["vel"].copy_(v)
        first["mass"].copy_(m)
        s["flat"] = s["start"].clone()
        s["state"] = _views(s["flat"], n)
        return s
    s["args"] = (x, v, m)
    s["flags"] = None if flags is None else torch.from_numpy(flags).cuda()
    if case["kind"] == "clusters":
        s["starts"] = _cluster_starts(case)
    return s


def run(state):
    case, fmm = state["case"], state["fmm"]
    kind = case["kind"]
    if kind == "eval":
        return dict(zip(("pot", "acc", "jerk"), fmm.eval(*state["args"], flags=state["flags"])))
    if kind == "clusters":
        return dict(zip(("pot", "acc", "jerk"),
                        fmm.eval_clusters(state["starts"], *state["args"])))
    if kind == "bodies":
        b = fmm.get_force_and_potential(state["bodies"])
        return {"pot": b["p"], "acc": b["F"], "jerk": b["J"]}
    if kind == "master":
        out = fmm.master_eval(*state["args"], get_steps=case["steps"])
        return {k: t for k, t in zip(("pot", "acc", "timestep"), out) if t is not None}
    # every pass is the same step: the state goes back to its start in one copy
    state["flat"].copy_(state["start"])
    t = fmm.master_evolve(state["state"], case["dt"])
    return {"time": t, **{k: state["state"][k] for k in ("pos", "vel", "acc", "timestep")}}


# ---- what a pass cannot do without --------------------------------------------------------------
def _fmm_flops(n, p, theta, mac="theta"):
    """Flops of one evaluation of n bodies: pair counts per body as Plummer spheres and Dehnen
    cusps show them (ncrit 64): M2L pairs 38 (1 - (2000/n)^(1/3)) at theta = 0.4, body pairs
    5200; they fall with theta to the powers 2.8 and 3.9; the error-controlled walk 20 and 3500."""
    far = 38.0 * max(0.05, 1.0 - (2000.0 / n) ** (1.0 / 3.0)) * (0.4 / theta) ** 2.8
    near = min(float(n), 5200.0 * (0.4 / theta) ** 3.9)
    if mac == "error":
        far, near = min(far, 20.0), min(near, 3500.0)
    return flops.eval_flops(p, n, near * n, far * n, 0.06 * n)["total"]


def work(case):
    kind = case["kind"]
    if kind == "clusters":
        sizes = np.diff(_cluster_starts(case)).tolist()
        return {"bytes": 112.0 * sum(sizes),
                "flops": sum(_fmm_flops(n, case["p"], case["theta"]) for n in sizes)}
    n = float(case["n"])
    if kind == "master":
        # 23 flops a pair for force and potential, 55 more for the two time scales
        return {"bytes": (56 + 32 + 8 * case["steps"]) * n,
                "flops": (78.0 if case["steps"] else 23.0) * n * n}
    if kind == "evolve":
        # five kicks over all pairs, one of them with the time steps: what one level does
        return {"bytes": 2 * 16 * 8 * n, "flops": (4 * 23.0 + 78.0) * n * n}
    if kind == "eval" and n < 8000:
        return {"bytes": 112.0 * n, "flops": 44.0 * n * n}
    return {"bytes": (304.0 if kind == "bodies" else 112.0) * n,
            "flops": _fmm_flops(n, case["p"], case["theta"], case.get("mac", "theta"))}


def tolerance(case):
    """Seen with the near field's sums cut another way: 3e-15 (one value 1e-13); the rotations of
    the far field against the direct sum where nothing is truncated: 2e-14 (4e-13) at order 20, and
    a rotation in another form moves a local expansion by 7e-14 at order 12.  Mixed near field, cut
    another way: 2e-10 (5e-9) with offsets in float pairs."""
    if case.get("learned"):
        # the network picks an angle per leaf in 32 bits: another order of its sums turns a tie,
        # which moves one leaf's forces by the error that the angle stands for (1e-7)
        return {"rel": 4e-9, "max": 1e-6}
    if case.get("near"):
        # 32-bit body pairs, sums of at most a tile in 32 bits
        return {"rel": 1e-9, "max": 2e-8} if case["near"] == "hilo" else {"rel": 4e-7, "max": 1e-5}
    if case.get("mac") == "error":
        # the pre-pass sums in 32 bits: another order turns a tie of the walk
        return {"rel": 1e-10, "max": 1e-8}
    if case["kind"] == "eval" and case["p"] >= 16:
        return {"rel": 4e-13, "max": 1e-11}
    if case["kind"] in ("master", "evolve"):
        # a step is a sum of fourth powers of minima
        return {"rel": 4e-13, "max": 1e-11}
    return {"rel": 1e-13, "max": 1e-12}


# ---- the same in plain torch, 64 bits -----------------------------------------------------------
def _direct(x, v, m, live, jerk):
    """All-pairs potential, acceleration and jerk (live: the sources' mask or None)."""
    n = m.shape[0]
    q = m if live is None else m * live
    pot = torch.empty(n, dtype=torch.float64, device="cuda")
    acc, jrk = torch.empty_like(x), torch.empty_like(x)
    step = max(1, (1 << 25) // n)
    for a in range(0, n, step):
        b = min(n, a + step)
        d = [x[:, k][None, :] - x[a:b, k][:, None] for k in range(3)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        ri = torch.where(r2 > 0, r2.rsqrt(), torch.zeros_like(r2))
        f = ri * q[None, :]
        pot[a:b] = f.sum(1)
        ri *= ri
        f *= ri
        if jerk:
            vr = torch.zeros_like(r2)
            for k in range(3):
                w = v[:, k][None, :] - v[a:b, k][:, None]
                vr.addcmul_(d[k], w)
                w *= f
                jrk[a:b, k] = w.sum(1)
            vr.mul_(f).mul_(ri).mul_(-3.0)
            for k in range(3):
                jrk[a:b, k] += (d[k] * vr).sum(1)
        for k in range(3):
            acc[a:b, k] = (d[k] * f).sum(1)
    return pot, acc, jrk


def exact(case, seed):
    kind = case["kind"]
    sizes = np.diff(_cluster_starts(case)).tolist() if kind == "clusters" else [case["n"]]
    # the step loop's steps come from the tree's own leaves; 1e11 pairs take about 20 seconds
    if kind == "evolve" or sum(float(n) ** 2 for n in sizes) > 1e11:
        return None
    x, v, m, flags = _inputs(case, seed)
    x, v, m = (torch.from_numpy(a).cuda() for a in (x, v, m))
    live = sink = None
    if flags is not None:
        fl = torch.from_numpy(flags).cuda()
        sink, live = (fl & 1).double(), ((fl >> 1) & 1).double()
    parts, at = [], 0
    for n in sizes:
        cut = slice(at, at + n)
        parts.append(_direct(x[cut], v[cut], m[cut], live, kind != "master"))
        at += n
    pot, acc, jerk = (torch.cat(t) for t in zip(*parts))
    if sink is not None:
        pot, acc, jerk = pot * sink, acc * sink[:, None], jerk * sink[:, None]
    out = {"pot": pot, "acc": acc}
    if kind == "master":
        return dict(out, timestep=None) if case["steps"] else out
    return dict(out, jerk=jerk)
