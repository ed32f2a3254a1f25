"""Measured cases of the lane engine, each through its public entry points
(espice_amd.lanes) with values on the host in and results on the host out,
as a program that sweeps a circuit calls them.

A case is a dict:
  path      "op" (Engine.solve_op), "tran" (Engine.solve_tran), "adaptive"
            (Engine.solve_tran_adaptive), "batch" (solve_batch), "replay"
            (Tape.replay)
  family    the circuit family (espice_amd/circuits.py), size its size
  points    sweep points (rows of live values, drawn from the seed); batch:
            instances over all templates
  mode      "op": cold, given (x0: the nominal operating point, the warm
            start of a point sweep), learned (x0 from a trained network)
  fp32      "op": FP32 factors with FP64 refinement
  measures  "op": return a few probed unknowns instead of every unknown
  ladder    "op": points the plain Newton leaves unconverged climb the ladder
  steps     "tran", "batch": fixed time steps; "adaptive": the stop time in
            steps of the family's dt

`exact` solves the same circuits in 64-bit torch, with the device equations
written out here: Newton to the last digit over a block tridiagonal
ordering. The engine stops inside Newton's tolerance, so it sits up to about
1e-4 from that solution.
"""
import math

import numpy as np
import torch

from espice_amd import circuits, lanes

# dt of each family's transient (seconds)
DT = {"rc_ladder": 10e-12, "inverter_chain": 2e-12, "diffpair_array": 20e-12, "mirror_tree": 20e-12,
      "rc_mesh": 1e-12}
MAX_ITER = {"inverter_chain": 1000, "inverter_chain_tran": 1000}


def listed():
    return [
        # one designer's quick look: a few dozen points of a small circuit
        {"name": "op_diodes_few", "path": "op", "family": "diode_stack", "size": 8, "points": 37, "mode": "cold",
         "fp32": False, "measures": False, "ladder": False},
        # the small Monte Carlo that a CPU also runs: 16 CMOS stages, 256 points
        {"name": "op_chain_small", "path": "op", "family": "inverter_chain", "size": 16, "points": 256,
         "mode": "cold", "fp32": False, "measures": False, "ladder": False},
        # the bipolar Monte Carlo with FP32 factors and FP64 refinement
        {"name": "op_pairs_fp32", "path": "op", "family": "diffpair_array", "size": 64, "points": 2048,
         "mode": "cold", "fp32": True, "measures": True, "ladder": False},
        # the large Monte Carlo, plain FP64 from a cold start
        {"name": "op_ota_cold", "path": "op", "family": "ota_array", "size": 64, "points": 16384, "mode": "cold",
         "fp32": False, "measures": True, "ladder": False},
        # the same sweep with learned starts and FP32 factors (bench.py's headline mode)
        {"name": "op_ota_learned_fp32", "path": "op", "family": "ota_array", "size": 64, "points": 16384,
         "mode": "learned", "fp32": True, "measures": True, "ladder": False},
        # a sweep around a known operating point, every unknown returned, a ragged count
        {"name": "op_mirrors_given", "path": "op", "family": "mirror_tree", "size": 6, "points": 5003,
         "mode": "given", "fp32": False, "measures": False, "ladder": False},
        # interconnect delay: an RC line with clamps, waveforms and .meas cards
        {"name": "tran_ladder", "path": "tran", "family": "rc_ladder", "size": 182, "points": 1000, "steps": 100},
        # a switching transient of bipolar pairs
        {"name": "tran_pairs", "path": "tran", "family": "diffpair_array", "size": 16, "points": 1536, "steps": 60},
        # step control per lane: CMOS stages switching one after another
        {"name": "adaptive_chain", "path": "adaptive", "family": "inverter_chain", "size": 12, "points": 777,
         "steps": 150},
        # a power grid beyond a workgroup's LDS
        {"name": "tran_mesh_big", "path": "tran", "family": "rc_mesh", "size": 64, "points": 256, "steps": 4},
        # the uneven batch: several templates and both analyses in one launch
        {"name": "batch_mixed", "path": "batch", "family": "mixed", "size": 64, "points": 600, "steps": 50},
        # the LU boundary alone: one pivot sequence over many matrices
        {"name": "replay_mesh", "path": "replay", "family": "rc_mesh", "size": 16, "points": 3000},
    ]


def _spread(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    path = rng.choice(["op", "op", "op", "tran", "tran", "adaptive", "big", "batch", "replay"])
    if path == "op":
        fam, lo, hi = rng.choice([("diode_stack", 2, 24), ("inverter_chain", 4, 24), ("diffpair_array", 4, 64),
                                  ("ota_array", 2, 64), ("mirror_tree", 2, 7), ("rc_ladder", 16, 256)])
        size = _spread(rng, lo, hi) if hi > 8 else rng.randint(lo, hi)
        mode = rng.choice(["cold", "cold", "given"])
        fp32 = fam in ("diffpair_array", "ota_array") and rng.random() < 0.4
        return {"path": "op", "family": fam, "size": size, "points": _spread(rng, 1, 16384), "mode": mode,
                "fp32": fp32, "measures": rng.random() < 0.5, "ladder": not fp32 and rng.random() < 0.3}
    if path == "tran":
        fam, lo, hi = rng.choice([("rc_ladder", 16, 400), ("inverter_chain", 4, 24), ("diffpair_array", 4, 32),
                                  ("mirror_tree", 2, 6), ("rc_mesh", 4, 16)])
        size = _spread(rng, lo, hi) if hi > 8 else rng.randint(lo, hi)
        return {"path": "tran", "family": fam, "size": size, "points": _spread(rng, 1, 1500),
                "steps": rng.randint(5, 60)}
    if path == "adaptive":
        fam, lo, hi = rng.choice([("rc_ladder", 16, 128), ("inverter_chain", 4, 12), ("diffpair_array", 4, 16)])
        return {"path": "adaptive", "family": fam, "size": _spread(rng, lo, hi), "points": _spread(rng, 1, 777),
                "steps": rng.randint(20, 120)}
    if path == "big":
        return {"path": "tran", "family": "rc_mesh", "size": rng.randint(36, 64), "points": _spread(rng, 16, 256),
                "steps": rng.randint(1, 4)}
    if path == "batch":
        return {"path": "batch", "family": "mixed", "size": rng.randint(16, 64), "points": _spread(rng, 40, 600),
                "steps": rng.randint(10, 50)}
    return {"path": "replay", "family": "rc_mesh", "size": rng.randint(4, 20), "points": _spread(rng, 1, 3000)}


# ---- inputs -----------------------------------------------------------------
def _family(case):
    f, k = case["family"], case["size"]
    if case["path"] in ("tran", "adaptive"):
        return {"rc_ladder": lambda: circuits.rc_ladder(k, tran=True),
                "inverter_chain": lambda: circuits.inverter_chain_tran(k),
                "diffpair_array": lambda: circuits.diffpair_array_tran(k),
                "mirror_tree": lambda: circuits.mirror_tree(k, tran=True),
                "rc_mesh": lambda: circuits.rc_mesh(k)}[f]()
    return circuits.FAMILIES[f](k)


def _probe_nodes(fam):
    """The unknowns a user would look at: a spread of the named nodes."""
    nodes = list(range(1, fam.deck.n_nodes))
    step = max(1, len(nodes) // 64)
    return np.array(nodes[::step][:64], dtype=np.uint32)


def _tran_probes(fam):
    n = fam.deck.n_nodes
    return [min(3, n - 1), 1 + n // 16, n // 4]   # where a step at the source has arrived


def _meas(fam):
    """Delay, extremes and mean of a waveform, as a delay study asks for."""
    n = fam.deck.n_nodes
    mid = 1 + (n - 2) // 8
    c = lanes.meas_clause
    return [lanes.meas_card("when", c(node=mid, val=0.1, rise=1)), lanes.meas_card("max", c(node=mid)),
            lanes.meas_card("avg", c(node=n - 1)), lanes.meas_card("pp", c(node=mid))]


def _mixed_groups(case):
    """Templates of the uneven batch up to the case's size, the instances
    dealt over them unevenly (each template at least one)."""
    grid = [(f, s) for f in circuits.MIXED_FAMILIES for s in f[2] if s <= case["size"] * (4 if "rc" in f[0] else 1)]
    keep = grid[::max(1, len(grid) // 24)]
    idx = np.arange(case["points"], dtype=np.uint64)
    pick = (circuits.uniform01(2024, idx, 1) * len(keep)).astype(np.int64)
    pick[:min(len(keep), len(pick))] = np.arange(min(len(keep), len(pick)))
    return [(f, s, idx[pick == g]) for g, (f, s) in enumerate(keep) if (pick == g).any()]


def _replay_inputs(case, seed):
    """Matrices of an RC mesh's pattern with the conductances, the
    capacitive companions and the source branch of a transient step, one
    draw per lane; the first is the lead."""
    k, m = case["size"], case["points"]
    fam = circuits.rc_mesh(k)
    eng = lanes.Engine(fam.deck.arrays())
    cp, ri, q = eng.pattern()
    eng.close()
    a = fam.deck.arrays()
    vals = fam.sample(seed, m)
    n = len(cp) - 1
    slot = {}
    for c in range(n):
        for p in range(cp[c], cp[c + 1]):
            slot[int(ri[p]), c] = p
    out = np.zeros((m, int(cp[-1])))
    bound = {int(d): int(l) for d, l in zip(a["bind_dev"], a["bind_live"])}
    branch = a["n_nodes"]
    for d, kind in enumerate(a["kind"]):
        p, t = int(a["nodes"][d][0]), int(a["nodes"][d][1])
        v = vals[:, bound[d]] if d in bound else np.full(m, a["params"][d][0])
        if kind == 2:
            for rc, g in (((p, branch), 1.0), ((t, branch), -1.0), ((branch, p), 1.0), ((branch, t), -1.0)):
                if rc in slot:
                    out[:, slot[rc]] += g
            continue
        g = 1.0 / v if kind == 0 else v * 2e12 if kind == 1 else np.full(m, 1e-12)
        for rc, sg in (((p, p), 1.0), ((p, t), -1.0), ((t, p), -1.0), ((t, t), 1.0)):
            if rc in slot:
                out[:, slot[rc]] += sg * g
    out[:, slot[0, 0]] += 1.0
    rhs = 1e-3 * circuits.normal(seed, np.arange(m * n, dtype=np.uint64), 9999).reshape(m, n)
    rhs[:, 0] = 0.0
    return cp, ri, q, out, rhs


def prepare(case, seed):
    path = case["path"]
    if path == "replay":
        cp, ri, q, a, rhs = _replay_inputs(case, seed)
        return {"case": case, "tape": lanes.Tape(cp, ri, a[0], q), "a": a, "rhs": rhs}
    if path == "batch":
        jobs = []
        for f, s, inst in _mixed_groups(case):
            fam = f[1](s)
            j = {"engine": lanes.Engine(fam.deck.arrays()), "values": fam.sample_at(seed, inst)}
            t = lanes.default_options().tol
            t.max_iter = MAX_ITER.get(f[0], t.max_iter)
            j.update(tol=t, ladder=True)
            if f[3] == "tran":
                j.update(analysis=lanes.BATCH_TRAN, dt=f[4], steps=case["steps"], probes=_tran_probes(fam))
            else:
                j.update(analysis=lanes.BATCH_OP)
            jobs.append(j)
        return {"case": case, "jobs": jobs}
    fam = _family(case)
    eng = lanes.Engine(fam.deck.arrays())
    s = {"case": case, "fam": fam, "eng": eng, "values": fam.sample(seed, case["points"])}
    if path == "op":
        if case["family"] in MAX_ITER:
            s["tol"] = lanes.default_options().tol
            s["tol"].max_iter = MAX_ITER[case["family"]]
        if case["measures"]:
            s["probes"] = _probe_nodes(fam)
        if case["mode"] != "cold":
            x_nom = eng.solve_op(fam.nominal()[None, :], tol=s.get("tol"))["x"][0]
            if case["mode"] == "given":
                s["x0"] = np.repeat(x_nom[None, :], case["points"], 0)
            else:
                # the network that a sweep keeps for its template, trained on
                # operating points of another draw
                tv = fam.sample(7, 16384)
                sol = eng.solve_op(tv, x0=np.repeat(x_nom[None, :], len(tv), 0), tiling=lanes.TILING_WAVE)
                ok = sol["reasons"] == 0
                tv, xs = tv[ok], sol["x"][ok]
                net = lanes.Mlp(tv.shape[1], eng.n - 1, seed=7)
                net.set_scaling(tv.mean(0), tv.std(0) + 1e-30, xs[:, 1:].mean(0), xs[:, 1:].std(0) + 1e-12)
                net.train(tv, xs, epochs=20, batch=512)
                eng.set_warm_start(net, x_nom)
    else:
        s["probes"] = _tran_probes(fam)
        if path == "tran":
            s["meas"] = _meas(fam)
    return s


# ---- one pass ---------------------------------------------------------------
def run(s):
    c = s["case"]
    if c["path"] == "replay":
        return s["tape"].replay(s["a"], s["rhs"])
    if c["path"] == "batch":
        out, _ = lanes.solve_batch(s["jobs"])
        res = {}
        for an, name in ((lanes.BATCH_OP, "op"), (lanes.BATCH_TRAN, "tran")):
            r = [o for o, j in zip(out, s["jobs"]) if j["analysis"] == an]
            if r:
                res[name] = {k: np.concatenate([v[k].reshape(-1) for v in r]) for k in r[0]}
        return res
    eng = s["eng"]
    if c["path"] == "op":
        return eng.solve_op(s["values"], x0=s.get("x0"), learned=c["mode"] == "learned", probes=s.get("probes"),
                            precision=lanes.FP32_REFINED if c["fp32"] else lanes.FP64, tol=s.get("tol"),
                            ladder=c["ladder"])
    dt = DT[c["family"]]
    if c["path"] == "adaptive":
        return eng.solve_tran_adaptive(s["values"], c["steps"] * dt, dt, probes=s["probes"], max_steps=400)
    if c["family"] == "rc_mesh" and c["size"] > 20:
        return eng.solve_tran(s["values"], dt, c["steps"], probes=s["probes"])
    return eng.solve_tran(s["values"], dt, c["steps"], probes=s["probes"], meas=s["meas"])


# ---- what a pass cannot do without ------------------------------------------
_DEV_FLOPS = {0: 7, 1: 5, 2: 6, 3: 2, 4: 40, 5: 148, 6: 190}
_OP_ITERS = {"diode_stack": 20, "inverter_chain": 40, "diffpair_array": 11, "ota_array": 11, "mirror_tree": 6,
             "rc_ladder": 6}


def _iteration_flops(a):
    """Devices, a sparse solve at the fill of a good order (planar meshes:
    n log n entries), the update."""
    n = a["n_nodes"] + int((a["kind"] == 2).sum())
    dev = sum(_DEV_FLOPS[int(k)] for k in a["kind"])
    if len(a["kind"]) > 2.8 * n and int((a["kind"] == 0).sum()) > 1.5 * n:
        return dev + 20 * n ** 1.5
    return dev + 20 * n


def _job_work(a, points, iters, steps, outs):
    n = a["n_nodes"] + int((a["kind"] == 2).sum())
    return {"bytes": 8.0 * points * (a["n_live"] + n + outs),
            "flops": float(points) * _iteration_flops(a) * (iters + 2 * steps)}


def work(case):
    if case["path"] == "replay":
        k, m = case["size"], case["points"]
        n = k * k + 3
        fill = n + 2 * 2.0 * n * max(1.0, math.log2(k))
        return {"bytes": 8.0 * m * (5 * n + 2 * n + fill), "flops": m * 20.0 * n ** 1.5}
    if case["path"] == "batch":
        tot = {"bytes": 0.0, "flops": 0.0}
        for f, s, inst in _mixed_groups(case):
            w = _job_work(f[1](s).deck.arrays(), len(inst), 20, case["steps"] if f[3] == "tran" else 0,
                          3 * case["steps"] if f[3] == "tran" else 0)
            tot = {k: tot[k] + w[k] for k in tot}
        return tot
    fam = _family(case)
    a = fam.deck.arrays()
    if case["path"] == "op":
        it = 4 if case["mode"] != "cold" else _OP_ITERS[case["family"]]
        return _job_work(a, case["points"], it, 0, 0)
    return _job_work(a, case["points"], 10, case["steps"], 3 * case["steps"])


# ---- how far another correct implementation may be ----------------------------
# Measured with another column order of the factors (sums in another order).
# Where no Newton gate turns over, x moves by 1e-16 to 1e-15 (FP32 factors
# refined to 1e-12 of a step: 7e-14; a switching transient: 1.5e-12). In the
# inverter chains, whose stages have gain, a point meets a gate an iteration
# earlier or later: 2.1e-7 on x (6e-6 V at most) at an operating point, 6e-5
# on the waveforms of an adaptive run, and more counts differ than can be
# allowed for.
def tolerance(case):
    if case["path"] == "replay":
        return {"rel": 1e-13, "max": 1e-11}
    if case["path"] == "batch":
        return {"rel": 1e-6, "max": 5e-5, "differ": 0.01}
    gain = case["family"] == "inverter_chain"
    if case["path"] == "op":
        if case["mode"] == "learned":
            # the starts come from a BF16 network; two Newton steps follow
            return {"rel": 1e-5, "max": 1e-3, "differ": 0.01}
        if case["fp32"]:
            return {"rel": 3e-13, "max": 3e-11, "differ": 0.002}
        if gain:
            return {"rel": 1e-6, "max": 5e-5, "differ": 0.01}
        return {"rel": 1e-14, "max": 1e-12, "differ": 0.002}
    if gain:
        return {"rel": 2.5e-4, "max": 1e-2, "differ": 0.01} if case["path"] == "adaptive" else \
            {"rel": 6e-12, "max": 1e-9, "differ": 0.01}
    return {"rel": 1e-13, "max": 1e-11, "differ": 0.002}


# ---- the same circuits in 64 bits, without the engine --------------------------
_VT = 300.15 * (1.3806226e-23 / 1.6021918e-19)


def _junction(v, isat, vt):
    """isat (exp(v / vt) - 1) with a linear tail above 80 vt."""
    u = v / vt
    ul = torch.clamp(u, max=80.0)
    return isat * (torch.exp(ul) * (1.0 + (u - ul)) - 1.0)


def _junction_spice(v, isat, vt):
    """The junction law with the cubic reverse tail below -3 vt."""
    vn = torch.clamp(v, max=-1e-3)
    tail = -isat * (1.0 + (3.0 * vt / (vn * math.e)) ** 3)
    return torch.where(v >= -3.0 * vt, _junction(torch.clamp(v, min=-3.0 * vt), isat, vt), tail)


def _mos(v, p):
    """Terminal currents (into d, g, s, b) of level-1 devices without body
    effect; v [..., 4] terminal voltages."""
    tp, gmin, isat = p["type"], p["gmin"], p["is"]
    d, g, s, b = (v[..., i] * tp for i in range(4))
    vds, vbs, vbd = d - s, b - s, b - d

    def bulk(u):
        return torch.where(u > -3.0 * _VT, _junction(torch.clamp(u, min=-3.0 * _VT), isat, _VT), -isat + 0 * u) \
            + gmin * u

    ibs, ibd = bulk(vbs), bulk(vbd)
    fwd = vds >= 0
    vgst = torch.where(fwd, g - s, g - d) - p["vto"] * tp
    av = torch.abs(vds)
    beta = p["kp"] * p["m"] * p["w"] / p["l"]
    bp = beta * (1.0 + p["lambda"] * av)
    on = torch.clamp(vgst, min=0.0)
    idc = torch.where(on <= av, 0.5 * bp * on * on, bp * av * (on - 0.5 * av))
    ich = torch.where(fwd, idc, -idc)
    return tp[..., None] * torch.stack([ich - ibd, 0 * ich, -ich - ibs, ibd + ibs], -1)


def _bjt(v, p):
    """Terminal currents (into c, b, e, s): Gummel-Poon with the Early
    effect, no high-level injection or leakage."""
    tp, gm = p["type"], p["gmin"]
    c, b, e, s = (v[..., i] * tp for i in range(4))
    vbe, vbc, vsub = b - e, b - c, s - c
    cbe, cbc = _junction_spice(vbe, p["is"], _VT), _junction_spice(vbc, p["is"], _VT)
    icc = (cbe - cbc) * (1.0 - vbc / p["vaf"])
    ibe, ibc = cbe / p["bf"] + gm * vbe, cbc / p["br"] + gm * vbc
    isub = gm * vsub
    return tp[..., None] * torch.stack([icc - ibc - isub, ibe + ibc, -icc - ibe, isub], -1)


class _Plain:
    """One circuit over B points in float64 torch: unknown voltages of the
    nodes no grounded source fixes, ordered in breadth-first levels, so the
    Jacobian is block tridiagonal."""

    def __init__(self, fam, values, device):
        a = fam.deck.arrays()
        self.dev, self.a = device, a
        self.nn = a["n_nodes"]
        v = torch.tensor(values, dtype=torch.float64, device=device)
        self.B = B = v.shape[0]
        par = torch.tensor(a["params"], dtype=torch.float64, device=device)
        over = {}
        for d, p, l in zip(a["bind_dev"], a["bind_param"], a["bind_live"]):
            over[int(d), int(p)] = v[:, int(l)]
        nodes = a["nodes"].astype(np.int64)
        self.groups = {}
        for kind in range(7):
            ids = np.nonzero(a["kind"] == kind)[0]
            if len(ids):
                self.groups[kind] = (ids, torch.tensor(nodes[ids], device=device))

        def field(kind, slot):
            ids = self.groups[kind][0]
            out = par[ids, slot].expand(B, -1).clone()
            for k, d in enumerate(ids):
                if (int(d), slot) in over:
                    out[:, k] = over[int(d), slot]
            return out

        from espice_amd import deck as dk
        self.f = {}
        for kind, slots in ((0, {"r": 0}), (1, {"c": 0}), (2, {"v": 0, "wave": 1, "v2": 2}), (3, {"i": 0}),
                            (4, {k: dk.D_SLOTS[k] for k in ("is", "gmin")}),
                            (5, {k: dk.M_SLOTS[k] for k in ("type", "vto", "kp", "lambda", "w", "l", "m", "is",
                                                            "gmin")}),
                            (6, {k: dk.Q_SLOTS[k] for k in ("type", "is", "bf", "br", "vaf", "gmin")})):
            if kind in self.groups:
                self.f[kind] = {name: field(kind, s) for name, s in slots.items()}
        src = self.groups[2][0]
        self.fixed = [0] + [int(nodes[d][0]) for d in src]
        free = [i for i in range(self.nn) if i not in set(self.fixed)]
        # breadth-first levels over shared devices
        adj = {i: set() for i in free}
        for kind in (0, 1, 4, 5, 6):
            if kind in self.groups:
                for t in nodes[self.groups[kind][0]]:
                    ts = [int(x) for x in set(t[:2 if kind < 5 else 4].tolist()) if int(x) in adj]
                    for i in ts:
                        adj[i].update(j for j in ts if j != i)
        levels, seen = [], set()
        for root in sorted(free, key=lambda i: len(adj[i])):
            if root in seen:
                continue
            lev = [root]
            seen.add(root)
            while lev:
                levels.append(lev)
                nxt = []
                for i in lev:
                    for j in sorted(adj[i]):
                        if j not in seen:
                            seen.add(j)
                            nxt.append(j)
                lev = nxt
        blocks = [[]]
        for lev in levels:
            if blocks[-1] and len(blocks[-1]) + len(lev) > 24:
                blocks.append([])
            blocks[-1] += lev
        self.free = [i for b in blocks for i in b]
        where = {n: k for k, n in enumerate(self.free)}
        self.cuts = np.cumsum([0] + [len(b) for b in blocks])
        self.free_t = torch.tensor(self.free, device=device)
        blk = np.searchsorted(self.cuts, np.arange(len(self.free)), side="right") - 1
        # where each device entry (row terminal, column terminal) goes
        self.put = {}
        for kind, (ids, _) in self.groups.items():
            if kind in (2, 3):
                continue
            nt = 2 if kind < 5 else 4
            ent = {}
            for k, d in enumerate(ids):
                for ri in range(nt):
                    for ci in range(nt):
                        r, c = where.get(int(nodes[d][ri])), where.get(int(nodes[d][ci]))
                        if r is None or c is None:
                            continue
                        br, bc = int(blk[r]), int(blk[c])
                        ent.setdefault((br, bc), []).append((r - self.cuts[br], c - self.cuts[bc], k, ri, ci))
            self.put[kind] = {key: torch.tensor(np.array(v), device=device).T for key, v in ent.items()}

    def currents(self, x, grad):
        """{kind: (I [B, nd, 4], dI/dv [B, nd, 4, 4])} of the static devices."""
        out = {}
        for kind, (ids, t) in self.groups.items():
            if kind in (1, 2, 3):
                continue
            p = self.f[kind]
            v = x[:, t]
            if kind == 0:
                g = 1.0 / p["r"]
                i = g * (v[..., 0] - v[..., 1])
                out[kind] = (torch.stack([i, -i], -1), self._pair(g))
                continue
            v = v.detach().requires_grad_(grad)
            with torch.enable_grad():
                if kind == 4:
                    u = v[..., 0] - v[..., 1]
                    i = _junction_spice(u, p["is"], _VT) + p["gmin"] * u
                    cur = torch.stack([i, -i], -1)
                else:
                    cur = _mos(v, p) if kind == 5 else _bjt(v, p)
                jac = None
                if grad:
                    nt = cur.shape[-1]
                    jac = torch.stack([torch.autograd.grad(cur[..., k].sum(), v, retain_graph=True)[0][..., :nt]
                                       for k in range(nt)], -2)
            out[kind] = (cur.detach(), jac)
        return out

    @staticmethod
    def _pair(g):
        return torch.stack([torch.stack([g, -g], -1), torch.stack([-g, g], -1)], -2)

    def charges(self, x):
        q = torch.zeros(self.B, self.nn, dtype=torch.float64, device=self.dev)
        if 1 in self.groups:
            t, c = self.groups[1][1], self.f[1]["c"]
            qq = c * (x[:, t[:, 0]] - x[:, t[:, 1]])
            q.index_add_(1, t[:, 0], qq)
            q.index_add_(1, t[:, 1], -qq)
        return q

    def rows(self, x, cur):
        """Current out of every node through the static devices."""
        f = torch.zeros(self.B, self.nn, dtype=torch.float64, device=self.dev)
        for kind, (i, _) in cur.items():
            t = self.groups[kind][1]
            for k in range(i.shape[-1]):
                f.index_add_(1, t[:, k], i[..., k])
        if 3 in self.groups:
            t, i = self.groups[3][1], self.f[3]["i"]
            f.index_add_(1, t[:, 0], i)
            f.index_add_(1, t[:, 1], -i)
        return f

    def newton(self, x, ag0=0.0, const=None, iters=300):
        """Newton with steps of at most 0.25 V, shrinking to 0.02 V; const: what the companion
        adds to the rows beside ag0 q(x)."""
        nb = len(self.cuts) - 1
        for it in range(iters):
            cur = self.currents(x, True)
            f = self.rows(x, cur)
            if ag0:
                f = f + ag0 * self.charges(x) + const
            f = f[:, self.free_t]
            blocks = {}
            parts = [(kind, j) for kind, (_, j) in cur.items()]
            if ag0 and 1 in self.groups:
                parts.append((1, self._pair(ag0 * self.f[1]["c"])))
            for kind, j in parts:
                for key, e in self.put[kind].items():
                    if key not in blocks:
                        blocks[key] = torch.zeros(self.B, int(self.cuts[key[0] + 1] - self.cuts[key[0]]),
                                                  int(self.cuts[key[1] + 1] - self.cuts[key[1]]),
                                                  dtype=torch.float64, device=self.dev)
                    m = blocks[key]
                    m.view(self.B, -1).index_add_(1, e[0] * m.shape[2] + e[1], j[:, e[2], e[3], e[4]])
            # block Thomas
            up, rhs = [], []
            for b in range(nb):
                d, r = blocks[b, b], -f[:, self.cuts[b]:self.cuts[b + 1], None]
                if b and (b, b - 1) in blocks:
                    if up[-1] is not None:
                        d = d - blocks[b, b - 1] @ up[-1]
                    r = r - blocks[b, b - 1] @ rhs[-1]
                u = blocks.get((b, b + 1))
                s = torch.linalg.solve(d, r if u is None else torch.cat([r, u], -1))
                rhs.append(s[..., :1])
                up.append(None if u is None else s[..., 1:])
            dx = [None] * nb
            for b in range(nb - 1, -1, -1):
                dx[b] = rhs[b] if up[b] is None else rhs[b] - up[b] @ dx[b + 1]
            step = torch.cat(dx, 1)[..., 0]
            big = step.abs().amax()
            x = x.clone()
            cap = max(0.25 * 0.98 ** it, 0.02)
            x[:, self.free_t] = x[:, self.free_t] + step.clamp(-cap, cap)
            if float(big) < 1e-11:
                return x
        return None

    def set_sources(self, x, after):
        ids, t = self.groups[2]
        p = self.f[2]
        x = x.clone()
        x[:, t[:, 0]] = torch.where((p["wave"] == 1) & after, p["v2"], p["v"])
        return x

    def op(self):
        x = torch.zeros(self.B, self.nn, dtype=torch.float64, device=self.dev)
        return self.newton(self.set_sources(x, False))

    def branches(self, x, dyn=None):
        """Branch currents of the grounded sources: what their nodes' other
        devices take from them."""
        f = self.rows(x, self.currents(x, False))
        if dyn is not None:
            f = f + dyn
        return -f[:, self.groups[2][1][:, 0]]


def _exact_op(fam, values, probes, device):
    out = []
    m = max(1, min(4096, len(values)))
    for k in range(0, len(values), m):
        p = _Plain(fam, values[k:k + m], device)
        x = p.op()
        if x is None:
            return None
        full = torch.cat([x, p.branches(x)], 1)
        out.append((full if probes is None else full[:, torch.tensor(probes.astype(np.int64), device=device)]).cpu())
    return torch.cat(out)


def _exact_tran(fam, values, dt, steps, probes, device):
    p = _Plain(fam, values, device)
    x = p.op()
    if x is None:
        return None, None
    q1 = p.charges(x)
    ip = torch.zeros_like(q1)
    rows = []
    for s in range(steps):
        ag0, ag1 = (1.0 / dt, 0.0) if s == 0 else (2.0 / dt, 1.0)
        x = p.newton(p.set_sources(x, True), ag0, -ag0 * q1 - ag1 * ip)
        if x is None:
            return None, None
        q = p.charges(x)
        ip = ag0 * (q - q1) - ag1 * ip
        q1 = q
        rows.append(x[:, probes])
    return torch.cat([x, p.branches(x, ip)], 1).cpu(), torch.stack(rows, 1).cpu()


def exact(case, seed):
    device = "cuda" if torch.cuda.is_available() else "cpu"
    path = case["path"]
    if path == "replay":
        cp, ri, _, a, rhs = _replay_inputs(case, seed)
        n = len(cp) - 1
        col = np.repeat(np.arange(n), np.diff(cp.astype(np.int64)))
        dx = np.zeros((len(a), n))
        for k in range(0, len(a), 256):
            m = np.zeros((len(a[k:k + 256]), n, n))
            m[:, ri, col] = a[k:k + 256]
            dx[k:k + 256] = -np.linalg.solve(m, rhs[k:k + 256, :, None])[..., 0]
        return {"lx": None, "ux": None, "udiag": None, "dx": dx, "fail": None}
    # an adaptive run chooses its own time points, a batch solves dozens of
    # templates; long chains of high-gain stages and the largest transients
    # take the plain solver too long
    if path in ("batch", "adaptive"):
        return None
    fam = _family(case)
    values = fam.sample(seed, case["points"])
    if path == "op":
        if case["family"] == "inverter_chain" and case["size"] > 32:
            return None
        probes = _probe_nodes(fam) if case["measures"] else None
        x = _exact_op(fam, values, probes, device)
        return None if x is None else {"x": x, "iterations": None, "reasons": None}
    if case["size"] * case["steps"] > 20000 and case["family"] == "rc_ladder":
        return None
    x, rows = _exact_tran(fam, values, DT[case["family"]], case["steps"], _tran_probes(fam), device)
    if x is None:
        return None
    out = {"x": x, "probes": rows, "iterations": None, "reasons": None}
    if not (case["family"] == "rc_mesh" and case["size"] > 20):
        out.update(meas=None, steps_done=None)
    return out
