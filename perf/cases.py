"""The work that programs built on this package have it do, as timed cases.

Kinds:
  ccp       a simulation of ccp's own force field (lamina binding sites, A/B
            domains): frames of steps handed to the caller
  lj        a simulation of the WCA + het LJ set in the tuned kernel shape:
            blocks of steps, then the positions
  batch     many independent single-chain systems stepped together
  contacts  the binned contact map of a state
  analysis  ccp's frame analysis: observables, d(s) / P(s), packed contact map
  cells     the allocation-free cell list of a device position array
  predict   the surrogate's contact map and radial density of B sequences
  train     one training step of the surrogate

Inputs are made from the seed alone: conformations are crumpled chains (a
Hilbert curve mapped into the nucleus) relaxed by a few dozen steps of
overdamped dynamics written in torch with a fixed order of every sum, so that
the same seed gives the same bits. `exact` steps the same physics in float64
(pair lists by cells, Philox4x32-10 noise).
"""
import ctypes
import math

import numpy as np
import torch

import tfm_amd
from tfm_amd import ccp, surrogate

RCO, ACO, LCO, K_E, L_0, E_P, E_L, K_B, T = (float(np.float32(v)) for v in
                                             (1.154701, 2.0, 0.5, 128.0, 1.0, 0.5, 8.0, 0.003356, 298.0))
HET, LAD = 1, 2
CHROMOSOMES = (0, 2284, 4599, 6687, 9338, 12508, 15193, 17477, 19792, 21880, 24531, 27701, 30386)
LJ_SHAPE = {"lanes_per_bead": 8, "cell_reach": 2, "cell_size": 1.25}     # bench.py's tuned shape
BATCH_SHAPE = {"lanes_per_bead": 8, "cell_reach": 2, "cell_size": 1.375}  # the ensemble's tuned shape


# ---------------------------------------------------------------- cases
def listed():
    return [
        # the smallest of ccp's own timing runs with enough beads for a domain
        # structure: every step is launch and dependency latency
        {"name": "ccp_1k", "kind": "ccp", "n": 1024, "vf": 0.125, "steps": 128},
        # ccp's default nucleus: 12 chromosomes, 30386 beads, a frame to the caller
        {"name": "ccp_30k", "kind": "ccp", "n": 30386, "vf": 0.15, "steps": 128},
        # one 16384-bead chain of the WCA + het LJ set
        {"name": "lj_16k", "kind": "lj", "n": 16384, "chains": 1, "vf": 0.2, "steps": 100},
        # the large nucleus of bench.py, 8 chains of 16384 beads
        {"name": "lj_131k", "kind": "lj", "n": 131072, "chains": 8, "vf": 0.3, "steps": 100},
        # one batch of the parameter sweep: 256 chains of 2048 beads
        {"name": "sweep_256x2048", "kind": "batch", "systems": 256, "lo": 2048, "hi": 2048, "draw": 1, "steps": 100},
        # an ensemble of uneven chains, log-uniform 512 to 16384 beads
        {"name": "ensemble_64", "kind": "batch", "systems": 64, "lo": 512, "hi": 16384, "draw": 2, "steps": 100},
        # a contact sample of the large nucleus into 1024 x 1024 bins, read by the host
        {"name": "contacts_131k", "kind": "contacts", "n": 131072, "chains": 8, "vf": 0.3, "cutoff": 1.5},
        # ccp-analyze's work on one frame of the default nucleus
        {"name": "analysis_30k", "kind": "analysis", "n": 30386, "vf": 0.15},
        # the cell list of a device position array for callers that cannot allocate
        {"name": "cells_100k", "kind": "cells", "n": 100003, "vf": 0.2, "side": 2.0},
        # the smallest network of the tests: a handful of short sequences
        {"name": "predict_small", "kind": "predict", "c_in": 5, "width": 32, "layers": 3, "d": 8, "L": 16, "rd": 8,
         "B": 3},
        # scoring candidates in the sweep: 64 sequences of 128 bins
        {"name": "predict_b64", "kind": "predict", "c_in": 5, "width": 256, "layers": 6, "d": 64, "L": 128, "rd": 32,
         "B": 64},
        # one step of the sweep's training loop
        {"name": "train_b64", "kind": "train", "c_in": 5, "width": 256, "layers": 6, "d": 64, "L": 128, "rd": 32,
         "B": 64},
    ]


def _log_int(rng, lo, hi):
    """A whole number of [lo, hi], uniform over the logarithm, odd as often as even."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("ccp", "lj", "batch", "contacts", "analysis", "cells", "predict", "train"))
    if kind == "ccp":
        return {"kind": kind, "n": _log_int(rng, 256, 32768), "vf": rng.uniform(0.08, 0.25),
                "steps": rng.randint(16, 128)}
    if kind == "lj":
        return {"kind": kind, "n": _log_int(rng, 1024, 131072), "chains": rng.randint(1, 8),
                "vf": rng.uniform(0.1, 0.3), "steps": rng.randint(16, 100)}
    if kind == "batch":
        hi = rng.choice((2048, 4096, 16384))
        return {"kind": kind, "systems": _log_int(rng, 4, 64 if hi > 4096 else 128), "lo": rng.choice((512, 1000, 2048)),
                "hi": hi, "draw": rng.randint(1, 1 << 20), "steps": rng.randint(16, 100)}
    if kind == "contacts":
        return {"kind": kind, "n": _log_int(rng, 1024, 131072), "chains": rng.randint(1, 8),
                "vf": rng.uniform(0.1, 0.3), "cutoff": rng.choice((1.2, 1.5, 2.0))}
    if kind == "analysis":
        return {"kind": kind, "n": _log_int(rng, 512, 16384), "vf": rng.uniform(0.08, 0.25)}
    if kind == "cells":
        return {"kind": kind, "n": _log_int(rng, 1000, 131072), "vf": rng.uniform(0.1, 0.3),
                "side": rng.choice((1.25, 2.0, 2.5))}
    return {"kind": kind, "c_in": 5, "width": rng.choice((32, 64, 100, 128, 256)), "layers": rng.randint(2, 6),
            "d": rng.choice((8, 32, 64)), "L": rng.choice((16, 50, 64, 100, 128)), "rd": rng.choice((8, 32)),
            "B": _log_int(rng, 1, 64)}


# ---------------------------------------------------------------- geometry and patterns
def _radius(n, vf):
    """The nucleus radius of volume fraction vf, to the six digits of a parameter file."""
    return float(f"{RCO / 2 + RCO / 2 * (n / vf) ** (1.0 / 3.0):.6f}")


def _chains(case, n):
    if case["kind"] == "lj" or case["kind"] == "contacts":
        k = case["chains"]
        return np.cumsum([0] + [n // k + (1 if c < n % k else 0) for c in range(k)])
    return np.array(CHROMOSOMES if n == 30386 else (0, n))


def _pattern(rng, n, het_fraction, lad_fraction, mean=20.0):
    """Alternating het blocks of geometric lengths; LAD blocks near the ends (lad_fraction) or on the het beads."""
    out = np.zeros(n, np.uint8)
    i, het = 0, rng.random() < het_fraction
    while i < n:
        k = int(rng.geometric(1.0 / (mean if het else mean * (1 - het_fraction) / het_fraction)))
        if het:
            out[i:i + k] |= HET | (LAD if lad_fraction is None else 0)
        i, het = i + k, not het
    if lad_fraction is not None:
        k = int(round(lad_fraction * n / 2))
        out[:k] |= LAD
        out[n - k:] |= LAD
    return out


def _hilbert(bits):
    """The Hilbert curve through a cube of 2^bits points a side (Skilling 2004): [8^bits, 3] whole numbers."""
    t = np.arange(1 << (3 * bits), dtype=np.int64)
    x = [np.zeros_like(t) for _ in range(3)]
    for b in range(bits):
        for a in range(3):
            x[a] |= ((t >> (3 * b + 2 - a)) & 1) << b
    g = x[2] >> 1
    for a in (2, 1):
        x[a] ^= x[a - 1]
    x[0] ^= g
    q = 2
    while q != 1 << bits:
        p = q - 1
        for a in (2, 1, 0):
            on = (x[a] & q) != 0
            s = np.where(on, 0, (x[0] ^ x[a]) & p)
            x[0] = np.where(on, x[0] ^ p, x[0] ^ s)
            x[a] = x[a] ^ s
        q <<= 1
    return np.stack(x, 1)


_curves = {}


def _start(n, radius, rng):
    """n points along a Hilbert curve through a cube, the cube mapped onto a ball of `radius`, turned at random."""
    bits = max(1, math.ceil(math.log(max(n, 8), 8) - 0.2))
    if bits not in _curves:
        _curves[bits] = _hilbert(bits).astype(np.float64) * (2.0 / ((1 << bits) - 1)) - 1.0
    c = _curves[bits]
    u = np.linspace(0, len(c) - 1, n)
    k = np.minimum(u.astype(np.int64), len(c) - 2)
    p = c[k] + (u - k)[:, None] * (c[k + 1] - c[k])
    norm = np.linalg.norm(p, axis=1, keepdims=True)
    p = p * (np.abs(p).max(axis=1, keepdims=True) / np.maximum(norm, 1e-9))
    q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
    return radius * (p @ q)


class _Cells:
    """Cell lists of several systems in torch: system s holds sys_of == s, inside a ball of radius R[s]."""

    OFFSETS = [(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)]

    def __init__(self, x, sys_of, R, side):
        cps = 2 * torch.ceil(R / side).long() + 4
        off = torch.cumsum(cps ** 3, 0) - cps ** 3
        self.cps = cps[sys_of]
        c = torch.floor(x / side).long() + (self.cps // 2)[:, None]
        c = torch.minimum(c.clamp(min=1), (self.cps - 2)[:, None])
        self.key = off[sys_of] + (c[:, 2] * self.cps + c[:, 1]) * self.cps + c[:, 0]
        key, self.order = torch.sort(self.key, stable=True)
        count = torch.bincount(key, minlength=int((cps ** 3).sum()) + 1)
        self.start = torch.cumsum(count, 0) - count
        self.count = count
        self.cap = int(count.max())

    def around(self, who=None):
        """(j, valid) of [n, cap] for each of the 27 cells around every bead of `who`."""
        key, cps = (self.key, self.cps) if who is None else (self.key[who], self.cps[who])
        slot = torch.arange(self.cap, device=key.device)
        for a, b, c in self.OFFSETS:
            k = key + (c * cps + b) * cps + a
            ok = slot[None] < self.count[k][:, None]
            j = self.order[torch.where(ok, self.start[k][:, None] + slot[None], 0)]
            yield j, ok


def _relaxed(starts, radii, chain_starts, seed, steps=60):
    """Overdamped chains (bonds, soft repulsion, wall) from `starts`; the positions of all systems, float32 on the GPU."""
    dev = torch.device("cuda")
    sys_of = torch.cat([torch.full((len(s),), k, dtype=torch.long) for k, s in enumerate(starts)]).to(dev)
    x = torch.tensor(np.concatenate(starts), dtype=torch.float32, device=dev)
    R = torch.tensor(radii, dtype=torch.float32, device=dev)
    first = torch.zeros(len(x), dtype=torch.bool, device=dev)
    first[torch.tensor(chain_starts, device=dev)] = True
    i = torch.arange(len(x), device=dev)
    g = torch.Generator(device=dev).manual_seed(seed)
    limit = (R - 0.95)[sys_of][:, None]
    for s in range(steps):
        f = torch.zeros_like(x)
        bond = torch.zeros_like(x)
        v = x[1:] - x[:-1]
        d = v.norm(dim=1, keepdim=True).clamp(min=1e-3)
        bond[1:] = torch.where(first[1:, None], torch.zeros_like(v), 128.0 * (1.0 - 1.0 / d) * v)
        f -= bond
        f[:-1] += bond[1:]
        for j, ok in _Cells(x, sys_of, R, 1.15).around():
            w = x[:, None] - x[j]
            r = w.norm(dim=2).clamp(min=1e-2)
            on = ok & (r < 1.1) & ((i[:, None] - j).abs() > 1)
            f += (torch.where(on, 160.0 * (1.1 - r) / r, torch.zeros_like(r))[:, :, None] * w).sum(1)
        move = 0.002 * f
        move *= (0.12 / move.norm(dim=1, keepdim=True).clamp(min=1e-9)).clamp(max=1.0)
        x = x + move
        if s < steps - 12:
            x = x + 0.06 * torch.randn(x.shape, generator=g, device=dev)
        r = x.norm(dim=1, keepdim=True)
        x = x * torch.clamp(limit / r.clamp(min=1e-6), max=1.0)
    return x


def _systems(case):
    """The systems of a batch: bead counts and parameters from the case alone, as a sweep draws them."""
    rng = np.random.default_rng(case["draw"])
    lo, hi = min(case["lo"], case["hi"]), case["hi"]
    return [{"n_beads": int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))))),
             "volume_fraction": float(rng.uniform(0.1, 0.35)), "eps_het": float(rng.uniform(0.2, 1.0)),
             "eps_lam": float(rng.uniform(0.2, 1.5)), "het_fraction": 0.3, "lad_fraction": 0.1,
             "seed": 4000 + k} for k in range(case["systems"])]


def _inputs(case, seed):
    """What the program has in hand: positions, flags, sites (host arrays) and the geometry."""
    rng = np.random.default_rng([seed, 77])
    kind = case["kind"]
    if kind == "batch":
        systems = _systems(case)
        n = [s["n_beads"] for s in systems]
        # the library takes the radius from the float32 volume fraction
        R = [_radius(k, float(np.float32(s["volume_fraction"]))) for k, s in zip(n, systems)]
        off = np.cumsum([0] + n)
        x = _relaxed([_start(k, r - 1.0, rng) for k, r in zip(n, R)], R, off[:-1], seed)
        flags = np.concatenate([_pattern(rng, k, 0.3, 0.1) for k in n])
        return {"x": x.cpu().numpy(), "flags": flags, "systems": systems, "R": R, "off": off, "chains": off}
    n = case["n"]
    R = _radius(n, case["vf"])
    chains = _chains(case, n)
    x = _relaxed([_start(n, R - 1.0, rng)], [R], chains[:-1], seed).cpu().numpy()
    out = {"x": x, "R": [R], "off": np.array([0, n]), "chains": chains}
    if kind in ("ccp", "analysis"):
        out["flags"] = np.concatenate([_pattern(rng, b - a, 0.5, None) for a, b in zip(chains[:-1], chains[1:])])
    else:
        out["flags"] = np.concatenate([_pattern(rng, b - a, 0.3, 0.15) for a, b in zip(chains[:-1], chains[1:])])
    if kind == "ccp":
        n_l = int(0.25 * 4.0 / (LCO / (R - RCO)) ** 2)
        d = rng.normal(size=(n_l, 3))
        out["lbs"] = ((R - RCO) * d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    return out


def _net(case, seed):
    return surrogate.Surrogate(c_in=case["c_in"], width=case["width"], n_layers=case["layers"], d=case["d"],
                               L=case["L"], rd_bins=case["rd"], B=case["B"], seed=seed)


def _sequences(case, seed):
    """Per-bin het and LAD fractions and three constant channels, contact maps and densities, as float32 arrays."""
    rng = np.random.default_rng([seed, 5])
    B, L = case["B"], case["L"]
    x = np.zeros((case["c_in"], B, L), np.float32)
    for b in range(B):
        f = _pattern(rng, 16 * L, 0.3, 0.1)
        x[0, b] = ((f & HET) > 0).reshape(L, 16).mean(axis=1)
        x[1, b] = ((f & LAD) > 0).reshape(L, 16).mean(axis=1)
    for c in range(2, case["c_in"]):
        x[c] = rng.uniform(-1.7, 1.7, size=(B, 1))
    s = np.abs(np.arange(L)[:, None] - np.arange(L)[None])
    y = (-1.0 - 1.2 * np.log10(1.0 + s) + rng.normal(0, 0.3, size=(B, L, L)))
    y = np.maximum((0.5 * (y + y.transpose(0, 2, 1))).astype(np.float32), -4.0)
    r = rng.uniform(0.05, 0.4, size=(case["rd"], B)).astype(np.float32)
    return x.reshape(case["c_in"], B * L), y, r


def _moments(net, seed):
    """Adam's moments of a training run under way (the seventieth step or so), and the step number."""
    g = torch.Generator().manual_seed(seed)
    for k in net.names:
        shape = net.p[k].shape
        net.m[k].copy_(1e-3 * torch.randn(shape, generator=g))
        net.v[k].copy_(1e-5 * (0.5 + torch.rand(shape, generator=g)))
    net.t = 70


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("predict", "train"):
        net = _net(case, seed)
        x, y, r = _sequences(case, seed)
        state = {"kind": kind, "net": net, "x": torch.tensor(x, device="cuda")}
        if kind == "train":
            _moments(net, seed)
            state["y"], state["r"] = torch.tensor(y, device="cuda"), torch.tensor(r, device="cuda")
        return state
    got = _inputs(case, seed)
    if kind == "batch":
        batch = tfm_amd.Batch(got["systems"], dict(timestep=0.001, contact_interval=1000, contact_cutoff=1.5,
                                                   contact_bins=128, radial_bins=32, graph_steps=100, **BATCH_SHAPE))
        batch.set_state(got["x"], got["flags"])
        return {"kind": kind, "batch": batch, "steps": case["steps"]}
    n, R = case["n"], got["R"][0]
    if kind == "cells":
        cps = max(4, 2 * math.ceil(R / case["side"]))
        new = lambda k: torch.zeros(k, dtype=torch.int32, device="cuda")
        return {"kind": kind, "x": torch.tensor(got["x"].reshape(-1), device="cuda"), "n": n, "side": case["side"],
                "cps": cps, "sci": new(n), "soi": new(n), "beg": new(cps ** 3), "end": new(cps ** 3)}
    par = {"number_of_particles": n, "nucleus_radius": f"{R:.6f}", "seed": 9}
    if kind in ("ccp", "analysis"):
        par.update(number_of_lbs=len(got["lbs"]) if kind == "ccp" else 0, steps_per_frame=case.get("steps", 64))
    else:
        par.update(force_field="lj", epsilon_het=0.6, epsilon_lamina=1.0, timestep=0.001, graph_steps=100,
                   number_of_chains=case["chains"], contact_interval=1000, number_of_lbs=0,
                   contact_cutoff=case.get("cutoff", 1.5), **LJ_SHAPE)
    sim = tfm_amd.Simulation(par)
    sim.flags = got["flags"]
    sim.positions = got["x"]
    if kind == "ccp":
        sim.lbs = got["lbs"]
    sim.set_time(0, 0.0, 0)
    return {"kind": kind, "sim": sim, "x": got["x"], "steps": case.get("steps"),
            "chromosomes": 6 if n == 30386 else 1}


def run(state):
    kind = state["kind"]
    if kind == "ccp":
        frames = []
        state["sim"].run_frames(1, lambda i_f, t, xyz: frames.append(xyz))
        return frames[0]
    if kind == "lj":
        state["sim"].run_steps(state["steps"])
        state["sim"].synchronize()
        return state["sim"].positions
    if kind == "batch":
        state["batch"].run_steps(state["steps"])
        state["batch"].synchronize()
        return state["batch"].state()[0]
    if kind == "contacts":
        sim = state["sim"]
        sim.contact_reset()
        sim.contact_sample()
        return sim.contact_map()[0]
    if kind == "analysis":
        sim = state["sim"]
        sim.positions = state["x"]
        scalars, density = sim.observables(64)
        by_s = [sim.distance_contact(c) for c in range(state["chromosomes"])]
        return {"scalars": scalars, "density": density, "d": [v[0] for v in by_s], "p": [v[1] for v in by_s],
                "map": sim.frame_contact_map()}
    if kind == "cells":
        u32p, f32p = ctypes.POINTER(ctypes.c_uint32), ctypes.POINTER(ctypes.c_float)
        out = [state[k] for k in ("sci", "soi", "beg", "end")]
        rc = ccp.lib().ccp_cell_list_noalloc(ctypes.cast(state["x"].data_ptr(), f32p), state["n"], state["side"],
                                             state["cps"], *(ctypes.cast(t.data_ptr(), u32p) for t in out),
                                             ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        if rc:
            raise RuntimeError(ccp.lib().ccp_last_error(None).decode())
        return out
    net = state["net"]
    if kind == "predict":
        return list(net.predict(state["x"]))
    net.zero_grad()
    loss = net.loss_backward(state["x"], state["y"], state["r"])
    net.step(lr=1e-3, wd=1e-4)
    return {"loss": loss, "grad": dict(net.g), "weight": dict(net.p)}


# ---------------------------------------------------------------- what a pass cannot do without
def _conv_macs(case):
    P, W, L = case["B"] * case["L"], case["width"], case["L"]
    enc = 3 * case["c_in"] * W + (case["layers"] - 1) * 3 * W * W
    return P * (enc + 2 * case["d"] * W + case["d"] * L) + case["rd"] * W * case["B"]


def work(case):
    kind = case["kind"]
    if kind in ("ccp", "lj", "batch"):
        n = sum(s["n_beads"] for s in _systems(case)) if kind == "batch" else case["n"]
        # a bead and step: both stages read and write the positions, the cell list and the noise state (176 bytes),
        # and take about twenty candidate partners of 25 operations each, twice
        return {"bytes": 176.0 * n * case["steps"], "flops": 1000.0 * n * case["steps"]}
    if kind == "contacts":
        bins = -(-case["n"] // max(1, -(-case["n"] // 1024)))
        return {"bytes": 16.0 * case["n"] + 4.0 * bins * bins, "flops": 250.0 * case["n"]}
    if kind == "analysis":
        n = case["n"]
        half = n // 2 if n == 30386 else n
        spans = [b - a for a, b in zip(CHROMOSOMES[:6], CHROMOSOMES[1:7])] if n == 30386 else [n]
        copies = 2 if n == 30386 else 1
        pairs = copies * (sum(k * k * 3 // 8 for k in spans) + half * half // 2)
        return {"bytes": 12.0 * n + 4.0 * (half // 4) * (half // 4 + 1) / 2 + 8.0 * sum(spans) / 2,
                "flops": 10.0 * pairs}
    if kind == "cells":
        cps = max(4, 2 * math.ceil(_radius(case["n"], case["vf"]) / case["side"]))
        return {"bytes": 20.0 * case["n"] + 8.0 * cps ** 3, "flops": 10.0 * case["n"]}
    W = case["width"]
    params = 3 * case["c_in"] * W + (case["layers"] - 1) * 3 * W * W + 2 * case["d"] * W + case["rd"] * W
    io = 4.0 * case["B"] * case["L"] * (case["c_in"] + case["L"])
    if kind == "predict":
        return {"bytes": 2.0 * params + io, "flops": 2.0 * _conv_macs(case)}
    return {"bytes": 28.0 * params + 2 * io, "flops": 6.0 * _conv_macs(case)}


# ---------------------------------------------------------------- the same in 64 bits
def _philox_normals(bead, step, k0, k1):
    """Unit normal triples of a step: Philox4x32-10 counter {bead, step, 0, attempt}, Box-Muller, redrawn while any
    exceeds 5."""
    mask = 0xFFFFFFFF
    z = torch.empty(len(bead), 3, dtype=torch.float64, device=bead.device)
    todo = torch.arange(len(bead), device=bead.device)
    for attempt in range(64):
        c = [bead[todo], torch.full_like(todo, step & mask), torch.full_like(todo, step >> 32),
             torch.full_like(todo, attempt)]
        a, b = k0[todo], k1[todo]
        for _ in range(10):
            p0, p1 = 0xD2511F53 * c[0], 0xCD9E8D57 * c[2]
            c = [((p1 >> 32) & mask) ^ c[1] ^ a, p1 & mask, ((p0 >> 32) & mask) ^ c[3] ^ b, p0 & mask]
            a, b = (a + 0x9E3779B9) & mask, (b + 0xBB67AE85) & mask
        u = [((v >> 8) + 1).double() * 2.0 ** -24 for v in c]
        r, q = torch.sqrt(-2 * torch.log(u[0])), torch.sqrt(-2 * torch.log(u[2]))
        t = torch.stack((r * torch.cos(2 * math.pi * u[1]), r * torch.sin(2 * math.pi * u[1]),
                         q * torch.cos(2 * math.pi * u[3])), 1)
        z[todo] = t
        todo = todo[(t.abs() > 5.0).any(1)]
        if not len(todo):
            break
    return z


class _Exact:
    """The simulation's forces and stochastic-Heun step in float64 for one or several systems."""

    SKIN = 0.8

    def __init__(self, case, got):
        dev = torch.device("cuda")
        self.lj = case["kind"] != "ccp"
        n = got["off"][-1]
        self.x = torch.tensor(got["x"], dtype=torch.float64, device=dev)
        self.sys_of = torch.tensor(np.repeat(np.arange(len(got["R"])), np.diff(got["off"])), device=dev)
        self.R = torch.tensor(np.array(got["R"], np.float32).astype(np.float64), device=dev)
        fl = torch.tensor(got["flags"], device=dev)
        self.het, self.lad = (fl & HET) > 0, (fl & LAD) > 0
        self.local = torch.tensor(np.arange(n) - np.repeat(got["off"][:-1], np.diff(got["off"])), device=dev)
        f32 = lambda v: float(np.float32(v))
        self.dt = f32(0.001) if self.lj else 1.0 / 2048
        self.sd = f32(math.sqrt(2.0 * K_B * T * self.dt))
        self.cap = f32(np.float32(0.2) / np.float32(self.dt)) if self.lj else None
        if case["kind"] == "batch":
            seeds = torch.tensor([s["seed"] for s in got["systems"]], device=dev)
            par = lambda k: torch.tensor([f32(s[k]) for s in got["systems"]], dtype=torch.float64, device=dev)
            self.eps_het, self.eps_lam = par("eps_het")[self.sys_of], par("eps_lam")[self.sys_of]
        else:
            seeds = torch.tensor([9], device=dev)
            full = lambda v: torch.full((n,), f32(v), dtype=torch.float64, device=dev)
            self.eps_het, self.eps_lam = full(0.6), full(1.0)
        self.k0, self.k1 = seeds[self.sys_of] & 0xFFFFFFFF, seeds[self.sys_of] >> 32
        self.first = torch.zeros(n + 1, dtype=torch.bool, device=dev)
        self.first[torch.tensor(np.asarray(got["chains"]), device=dev)] = True
        self.lbs = torch.tensor(got["lbs"], dtype=torch.float64, device=dev) if "lbs" in got else None
        self.built = None

    def _pairs(self, x, radius, who):
        cells = _Cells(x[who], self.sys_of[who], self.R, radius)
        a, b = [], []
        for j, ok in cells.around():
            ok &= (x[who][:, None] - x[who][j]).square().sum(2) < radius * radius
            i = torch.arange(len(who), device=x.device)[:, None].expand_as(j)[ok]
            a.append(who[i])
            b.append(who[j[ok]])
        i, j = torch.cat(a), torch.cat(b)
        keep = (i - j).abs() > 1
        return i[keep], j[keep]

    def _lists(self, x):
        if self.built is not None and float((x - self.built).square().sum(1).max()) < (0.49 * self.SKIN) ** 2:
            return
        self.built = x.clone()
        short = 2.0 ** (1 / 6) if self.lj else RCO
        every = torch.arange(len(x), device=x.device)
        self.short = self._pairs(x, short + self.SKIN, every)
        self.long = self._pairs(x, (2.5 if self.lj else ACO) + self.SKIN, torch.nonzero(self.het)[:, 0])
        if self.lbs is not None:
            near = torch.nonzero(self.lad & (x.norm(dim=1) > float(self.R[0]) - RCO - LCO - self.SKIN))[:, 0]
            hit = torch.nonzero(torch.cdist(x[near], self.lbs) < LCO + self.SKIN)
            self.sites = near[hit[:, 0]], hit[:, 1]

    def _add_pairs(self, f, x, pairs, factor):
        i, j = pairs
        v = x[i] - x[j]
        f.index_add_(0, i, factor(v.square().sum(1), i, j)[:, None] * v)

    def forces(self, x):
        self._lists(x)
        f = torch.zeros_like(x)
        wf = lambda e, d2: e * (18.0 * d2 * d2 - 96.0 * d2 + 96.0) / d2 ** 4
        lj = lambda e, d2: e * 24.0 * (2.0 * d2 ** -6 - d2 ** -3) / d2
        zero = torch.zeros((), dtype=x.dtype, device=x.device)
        if self.lj:
            rm2, rc2 = 2.0 ** (1 / 3), 6.25
            self._add_pairs(f, x, self.short, lambda d2, i, j: torch.where(d2 < rm2, lj(1.0, d2), zero))
            self._add_pairs(f, x, self.long, lambda d2, i, j: torch.where((d2 >= rm2) & (d2 < rc2),
                                                                        lj(self.eps_het[i], d2), zero))
        else:
            self._add_pairs(f, x, self.short, lambda d2, i, j: torch.where(d2.sqrt() <= RCO, wf(E_P, d2), zero))
            self._add_pairs(f, x, self.long, lambda d2, i, j: torch.where((d2.sqrt() > RCO) & (d2.sqrt() <= ACO),
                                                                        wf(E_P, d2), zero))
            i, l = self.sites
            v = x[i] - self.lbs[l]
            d = v.norm(dim=1)
            fac = torch.where(d <= LCO, E_L * 8.0 / (3.0 * LCO * LCO) * ((d / LCO) ** 6 - 1.0), zero)
            f.index_add_(0, i, fac[:, None] * v)
        # bonds and bending: v[k] = x[k] - x[k - 1], zero where a chain starts
        n = len(x)
        v = torch.zeros(n + 3, 3, dtype=x.dtype, device=x.device)
        v[2:n + 1] = x[1:] - x[:-1]
        gone = torch.ones(n + 3, dtype=torch.bool, device=x.device)
        gone[1:n + 2] = self.first
        v[gone] = 0.0
        il = torch.where(gone, zero, 1.0 / v.norm(dim=1))
        v0, v1, v2, v3 = (v[k:k + n] for k in range(4))
        i0, i1, i2, i3 = (il[k:k + n, None] for k in range(4))
        f += K_E * (1.0 - L_0 * i2) * v2 - K_E * (1.0 - L_0 * i1) * v1
        c0, c1, c2 = ((a * b).sum(1, keepdim=True) * p * q for a, b, p, q in
                      ((v1, v0, i1, i0), (v2, v1, i2, i1), (v3, v2, i3, i2)))
        a0, a1, a3, q1, q2 = i1 * i0, i1 * i2, i2 * i3, i1 * i1, i2 * i2
        bend = a0 * v0 - (c0 * q1 + c1 * q1 + a1) * v1 + (a1 + c1 * q2 + c2 * q2) * v2 - a3 * v3
        f += (2.0 if self.lj else 1.0) * (bend if self.lj else torch.where(self.het[:, None], bend, zero))
        # wall
        r = x.norm(dim=1, keepdim=True)
        w = -(self.R[self.sys_of][:, None] / r - 1.0) * x
        d2 = w.square().sum(1)
        if self.lj:
            fac = torch.where(d2 < rm2, lj(1.0, d2), torch.where(self.lad & (d2 < rc2), lj(self.eps_lam, d2), zero))
        else:
            fac = torch.where(d2.sqrt() <= RCO, wf(1.0, d2), zero)
        f += torch.where(torch.isfinite(fac), fac, zero)[:, None] * torch.where(torch.isfinite(w), w, zero)
        if self.cap:
            f *= torch.clamp(self.cap / f.norm(dim=1, keepdim=True).clamp(min=1e-30), max=1.0)
        return f

    def run(self, steps):
        x = self.x
        for s in range(steps):
            noise = self.sd * _philox_normals(self.local, s, self.k0, self.k1)
            f = self.forces(x)
            e = self.forces(x + f * self.dt + noise)
            x = x + 0.5 * self.dt * (f + e) + noise
        return x


def _exact_analysis(case, got):
    x = torch.tensor(got["x"], dtype=torch.float64, device="cuda")
    n, R = len(x), float(np.float32(got["R"][0]))
    com = x.mean(0)
    d = x.norm(dim=1)
    bond = x[1:] - x[:-1]
    cos = (bond * x[:-1]).sum(1) / (bond.norm(dim=1) * d[:-1])
    scalars = [com.norm(), x.square().sum() / n - com.square().sum(), 0.5 * (3.0 * cos * cos - 1.0).mean(),
               (x[:, 2] < R).double().mean()]
    a, nb = RCO / 2.0, 64
    vb = 4.0 / 3.0 * math.pi * a ** 3
    het = torch.tensor((got["flags"] & HET) > 0, device="cuda")
    inside = torch.zeros(3, nb + 1, dtype=torch.float64, device="cuda")
    for k in range(1, nb + 1):
        rb = R * (k / nb) ** (1.0 / 3.0)
        ca = (d * d + a * a - rb * rb) / (2.0 * d * a)
        cb = (rb * rb + d * d - a * a) / (2.0 * rb * d)
        lens = math.pi / 3.0 * (a ** 3 * (2 + ca) * (1 - ca) ** 2 + rb ** 3 * (2 + cb) * (1 - cb) ** 2)
        v = torch.where(d - a > rb, torch.zeros_like(d), torch.where(d + a < rb, torch.full_like(d, vb), lens))
        inside[:, k] = torch.stack((v[het].sum(), v[~het].sum(), v.sum()))
    density = inside.diff(dim=1) / (4.0 / 3.0 * math.pi * R ** 3 / nb)
    copies = [0, n // 2] if n == 30386 else [0]
    spans = list(zip(CHROMOSOMES[:6], CHROMOSOMES[1:7])) if n == 30386 else [(0, n)]
    ds, ps = [], []
    for b, e in spans:
        sd, sp = [], []
        for s in range(1, (e - b) // 2 + 1):
            r = torch.cat([(x[b + s + c:e + c] - x[b + c:e + c - s]).norm(dim=1) for c in copies])
            sd.append(r.mean())
            sp.append(1000.0 * (r < 2.0).double().mean())
        ds.append(torch.stack(sd))
        ps.append(torch.stack(sp))
    side = n // len(copies) // 4
    rows = torch.zeros(side, side, dtype=torch.float64, device="cuda")
    for c in copies:
        p = x[c:c + 4 * side]
        for k in range(0, side, 256):
            q = p[4 * k:4 * min(side, k + 256)]
            close = ((q[:, None] - p[None]).square().sum(2) < 4.0).double()
            rows[k:k + 256] += 1000.0 / (16 * len(copies)) * close.reshape(-1, 4, side, 4).sum((1, 3))
    low = torch.tril_indices(side, side, device="cuda")
    return {"scalars": torch.stack(scalars), "density": density, "d": ds, "p": ps, "map": rows[low[0], low[1]]}


def _forward64(case, p, x):
    B, L = case["B"], case["L"]
    h = None
    y = x.reshape(case["c_in"], B, L).permute(1, 0, 2)
    for k in range(1, case["layers"] + 1):
        w = p[f"W{k}"].reshape(case["width"], -1, 3)
        z = torch.nn.functional.pad(y, (1, 1))
        cols = torch.stack((z[:, :, :-2], z[:, :, 1:-1], z[:, :, 2:]), 2).reshape(B, -1, L)
        g = torch.matmul(w.reshape(case["width"], -1), cols) + p[f"b{k}"][:, None]
        g = torch.nn.functional.gelu(g, approximate="tanh")
        h = g if h is None else h + g
        y = h
    u, v = torch.matmul(p["Wu"], h), torch.matmul(p["Wv"], h)
    raw = torch.matmul(u.transpose(1, 2).contiguous(), v) / math.sqrt(case["d"])
    i = torch.arange(L, device=x.device)
    S = 0.5 * (raw + raw.transpose(1, 2)) + p["dist"][(i[:, None] - i[None]).abs()] + p["c0"]
    return S, torch.matmul(p["Wr"], h.mean(2).t().contiguous()) + p["br"][:, None]


def _exact_net(case, seed):
    net = _net(case, seed)
    if case["kind"] == "train":
        _moments(net, seed)
    x, y, r = (torch.tensor(v, dtype=torch.float64, device="cuda") for v in _sequences(case, seed))
    p = {k: net.p[k].double().requires_grad_() for k in net.names}
    S, rd = _forward64(case, p, x)
    if case["kind"] == "predict":
        return [S.detach(), rd.detach()]
    L = case["L"]
    upper = torch.triu_indices(L, L, device="cuda")
    loss = (S - y)[:, upper[0], upper[1]].square().mean() + (rd - r).square().mean()
    loss.backward()
    lr, b1, b2, eps = (float(np.float32(v)) for v in (1e-3, 0.9, 0.999, 1e-8))
    t = net.t + 1
    new = {}
    for k in net.names:
        wd = float(np.float32(1e-4)) if k.startswith("W") else 0.0
        g = p[k].grad
        m = b1 * net.m[k].double() + (1 - b1) * g
        v = b2 * net.v[k].double() + (1 - b2) * g * g
        new[k] = p[k].detach() * (1 - lr * wd) - lr * (m / (1 - b1 ** t)) / ((v / (1 - b2 ** t)).sqrt() + eps)
    return {"loss": loss.detach().reshape(1), "grad": {k: p[k].grad for k in net.names}, "weight": new}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("contacts", "cells"):
        return None  # whole numbers only
    if kind in ("predict", "train"):
        return _exact_net(case, seed)
    got = _inputs(case, seed)
    if kind == "analysis":
        return _exact_analysis(case, got)
    return _Exact(case, got).run(case["steps"])
