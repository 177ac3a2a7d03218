"""The work that users of gadget_ng_pm_hip have it do, as cases that can be timed.

A case is a dict of plain values; `prepare` makes what a program holds before
the call (particles, the plan, the network), `run` makes one call through the
package's public entry points, `work` counts what that call cannot do without
and `exact` computes the same outputs in 64 bits with torch alone.

Kinds of case:
  pm        one PM force solve: "entry" host (the GravitySolver drop-in on host
            Vec3 arrays), f64 (device Vec3), soa64 or f32 (device SoA arrays)
  ensemble  many small boxes in one call
  pk        the power spectrum of a particle set
  ic        second-order initial conditions into device memory
  sr        the TreePM short-range sum
  learned   PM solve, network input, inference and correction of one box
  train     one training step of the network
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gadget-ng_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DEV = "cuda"
F64 = torch.float64
CHUNK = 1 << 23  # particles handled at a time in the generators and references


def listed():
    return [
        # the reference's own GPU-against-CPU bench input: one host call on a
        # 32^3 mesh, where latency and launches are all there is
        {"name": "host_curve_32", "kind": "pm", "entry": "host", "nm": 32, "n": 1024, "box": 20.0, "dist": "curve",
         "r_split_cells": 0.0, "eps_cells": 0.0, "deconvolve": False, "subset": False},
        # the FP64 parity configuration: 32^3 uniform particles on a 64^3 mesh, device resident
        {"name": "uniform_64", "kind": "pm", "entry": "f64", "nm": 64, "n": 32768, "box": 100.0, "dist": "uniform",
         "r_split_cells": 0.0, "eps_cells": 0.0, "deconvolve": False, "subset": False},
        # a TreePM long-range call on a radix-3 mesh, particles in no spatial
        # order, forces wanted for the active quarter (a block time step)
        {"name": "treepm_active_192", "kind": "pm", "entry": "f32", "nm": 192, "n": 884735, "box": 96.0,
         "dist": "shuffled", "r_split_cells": 1.25, "eps_cells": 0.0, "deconvolve": True, "subset": True},
        # the drop-in on host arrays at an everyday size: transfers, conversion and the solve
        {"name": "host_lattice_256", "kind": "pm", "entry": "host", "nm": 256, "n": 2097152, "box": 128.0,
         "dist": "lattice", "r_split_cells": 0.0, "eps_cells": 0.25, "deconvolve": False, "subset": False},
        # the headline: 256^3 Zel'dovich particles on a 512^3 mesh, device Vec3 arrays
        {"name": "lattice_512", "kind": "pm", "entry": "f64", "nm": 512, "n": 16777216, "box": 256.0,
         "dist": "lattice", "r_split_cells": 0.0, "eps_cells": 0.0, "deconvolve": False, "subset": False},
        # the largest: 512^3 clustered particles on a 1024^3 mesh, TreePM long range
        {"name": "clustered_1024", "kind": "pm", "entry": "f64", "nm": 1024, "n": 134217728, "box": 512.0,
         "dist": "clustered", "r_split_cells": 1.25, "eps_cells": 0.0, "deconvolve": False, "subset": False},
        # an ensemble of boxes of uneven size (meshes 64^3 to 256^3) in one call
        {"name": "ensemble_16", "kind": "ensemble", "boxes": 16},
        # analysis in the loop: P(k) of 160^3 particles on a 256^3 mesh
        {"name": "pk_256", "kind": "pk", "nm": 256, "n": 4096000, "box": 256.0, "dist": "clustered"},
        # 2LPT initial conditions of 256^3 particles
        {"name": "ic_2lpt_256", "kind": "ic", "nm": 256, "box": 100.0},
        # TreePM short range of a clustered 96^3 box (r_s = 1.25 cells, r_cut = 5 r_s)
        {"name": "short_range_96", "kind": "sr", "n": 884736, "box": 96.0, "r_split": 1.25, "eps": 0.05,
         "split": "exact"},
        # the learned correction applied to one full 256^3 box
        {"name": "learned_256", "kind": "learned", "nm": 256},
        # its training step: 8 boxes of 64^3, forward, loss, backward and update
        {"name": "train_8x64", "kind": "train", "nm": 64, "boxes": 8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pm"] * 6 + ["ensemble", "pk", "ic", "sr", "learned", "train"])
    if kind == "pm":
        entry = rng.choice(["host", "f64", "f32", "soa64"])
        nm = rng.choice([16, 32, 48, 64, 96, 128, 192, 256, 384, 512] if entry != "host" else [16, 32, 64, 128, 256])
        n = _log_int(rng, 500, min(nm ** 3 // 4 + 500, 16 << 20))
        cells = rng.choice([0.0, 1.25, 2.5])
        return {"kind": "pm", "entry": entry, "nm": nm, "n": n, "box": round(rng.uniform(10.0, 500.0), 3),
                "dist": rng.choice(["uniform", "clustered", "shuffled"]), "r_split_cells": cells,
                "eps_cells": rng.choice([0.0, 0.0, 0.3]), "deconvolve": cells > 0.0 and rng.random() < 0.5,
                "subset": rng.random() < 0.3}
    if kind == "ensemble":
        return {"kind": "ensemble", "boxes": rng.randint(3, 20)}
    if kind == "pk":
        nm = rng.choice([64, 96, 128, 256, 384])
        return {"kind": "pk", "nm": nm, "n": _log_int(rng, 5000, nm ** 3 // 2), "box": round(rng.uniform(50.0, 500.0), 3),
                "dist": rng.choice(["uniform", "clustered"])}
    if kind == "ic":
        return {"kind": "ic", "nm": rng.choice([32, 48, 64, 96, 128, 192, 256]), "box": round(rng.uniform(20.0, 500.0), 3)}
    if kind == "sr":
        side = rng.randint(24, 96)
        return {"kind": "sr", "n": side ** 3 - rng.randint(0, side), "box": float(side),
                "r_split": round(rng.uniform(0.8, 1.4), 3), "eps": rng.choice([0.02, 0.05, 0.2]),
                "split": rng.choice(["exact", "exact", "reference"])}
    if kind == "learned":
        return {"kind": "learned", "nm": rng.choice([32, 48, 64, 96, 128, 192])}
    return {"kind": "train", "nm": rng.choice([32, 48, 64]), "boxes": rng.randint(1, 8)}


# ---------------------------------------------------------------------------
# particle sets
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _freqs(n):
    return torch.fft.fftfreq(n, 1.0 / n, device=DEV, dtype=F64)


def _rfreqs(n):
    return torch.arange(n // 2 + 1, device=DEV, dtype=F64)


def _lattice(side, box, rms, gen):
    """(side^3, 3) lattice, z slowest, displaced by a Zel'dovich field of
    P(k) ~ k^-2 with 3-D rms displacement `rms`, wrapped into [0, box)."""
    m = 16
    while m < min(side, 256):
        m *= 2
    dk = torch.fft.rfftn(torch.randn(m, m, m, device=DEV, generator=gen))
    k = (_freqs(m)[:, None, None], _freqs(m)[None, :, None], _rfreqs(m)[None, None, :])
    k2 = (k[0] ** 2 + k[1] ** 2 + k[2] ** 2).float()
    k2[0, 0, 0] = 1.0
    dk = torch.where(k2 <= (m / 2 - 1) ** 2, dk * k2 ** -1.5, torch.zeros_like(dk))
    dk[0, 0, 0] = 0.0
    psi = torch.stack([torch.fft.irfftn(1j * ka.float() * dk, s=(m, m, m)) for ka in (k[2], k[1], k[0])])
    if m != side:
        psi = torch.nn.functional.interpolate(psi[None], size=(side,) * 3, mode="trilinear", align_corners=False)[0]
    psi *= rms / torch.sqrt((psi ** 2).sum(0).mean())
    q = torch.arange(side, device=DEV, dtype=F64) * (box / side)
    pos = torch.empty(side, side, side, 3, device=DEV, dtype=F64)
    pos[..., 0] = q[None, None, :] + psi[0]
    pos[..., 1] = q[None, :, None] + psi[1]
    pos[..., 2] = q[:, None, None] + psi[2]
    return pos.reshape(-1, 3).remainder_(box)


def _spheres(n, count, box, a, gen):
    """(n, 3) members of `count` Plummer spheres of scale radius a (cut at 20 a),
    uniform centres, log-normal populations, sphere after sphere."""
    centres = torch.rand(count, 3, device=DEV, dtype=F64, generator=gen) * box
    w = torch.exp(torch.randn(count, device=DEV, dtype=F64, generator=gen))
    edges = torch.cumsum(w, 0) / w.sum()
    pos = torch.empty(n, 3, device=DEV, dtype=F64)
    umax = 20.0 ** 3 / (20.0 ** 2 + 1.0) ** 1.5
    for lo in range(0, n, CHUNK):
        hi = min(n, lo + CHUNK)
        t = (torch.arange(lo, hi, device=DEV, dtype=F64) + 0.5) / n
        owner = torch.searchsorted(edges, t).clamp_(max=count - 1)
        u = torch.rand(hi - lo, 3, device=DEV, dtype=F64, generator=gen)
        r = a / torch.sqrt((u[:, 0] * umax).clamp_(min=1e-9) ** (-2.0 / 3.0) - 1.0)
        cz = 2.0 * u[:, 1] - 1.0
        s = torch.sqrt(1.0 - cz * cz)
        p = torch.stack([r * s * torch.cos(2 * math.pi * u[:, 2]), r * s * torch.sin(2 * math.pi * u[:, 2]), r * cz], 1)
        pos[lo:hi] = (centres[owner] + p).remainder_(box)
    return pos


def _clustered(n, box, rms, a, spheres, gen):
    """70 % of n on a displaced lattice, the rest in Plummer spheres."""
    side = max(2, int((0.698 * n) ** (1.0 / 3.0)))
    return torch.cat([_lattice(side, box, rms, gen), _spheres(n - side ** 3, spheres, box, a, gen)])


def _positions(case, seed):
    """(n, 3) f64 positions of a "pm" or "pk" case."""
    n, box, nm, dist = case["n"], case["box"], case["nm"], case["dist"]
    gen = _gen(seed)
    if dist == "curve":
        t = 0.37 * torch.arange(n, device=DEV, dtype=F64) + torch.rand(1, device=DEV, dtype=F64, generator=gen)
        return torch.stack([torch.sin(t), torch.cos(t), torch.sin(0.5 * t)], 1) * (0.5 * box)
    if dist == "uniform":
        return torch.rand(n, 3, device=DEV, dtype=F64, generator=gen) * box
    if dist == "lattice":
        return _lattice(round(n ** (1.0 / 3.0)), box, 0.5 * box / nm, gen)
    pos = _clustered(n, box, 0.5 * box / nm, 0.4 * box / nm, max(1, n // 65536), gen)
    if dist == "shuffled":
        pos = pos[torch.randperm(n, device=DEV, generator=gen)]
    return pos


def _subset(case, seed):
    """Indices of the active quarter, ascending, or None."""
    if not case.get("subset"):
        return None
    pick = torch.randperm(case["n"], device=DEV, generator=_gen(seed + 7))[: max(1, case["n"] // 4)]
    return torch.sort(pick).values


def _pm_inputs(case, seed):
    """(pos, idx): f64 positions, rounded to f32 where the entry takes f32."""
    pos = _positions(case, seed)
    if case["entry"] == "f32":
        pos = pos.float()
    return pos, _subset(case, seed)


def _ensemble_inputs(case, seed):
    """Boxes of mesh 2 s for s cycling over the sides, and their f32 particles."""
    sides = (32, 48, 64, 96, 128)
    out = []
    for b in range(case["boxes"]):
        s = sides[(b * 3) % 5]
        out.append((s, _lattice(s, float(s), 0.25, _gen(seed * 1009 + b)).float()))
    return out


def _learned_inputs(case, seed):
    """One particle per cell, Plummer spheres of 0.2 cells (f32), and the weights."""
    nm = case["nm"]
    pos = _clustered(nm ** 3, float(nm), 0.5, 0.2, max(1, round(250 * (nm / 256) ** 3)), _gen(seed)).float()
    pos[pos >= nm] = 0.0
    return pos, _weights(seed)


def _weights(seed):
    """He-normal weights of the network's three layers, the last at a tenth."""
    g = np.random.default_rng(seed)
    p = {}
    for k, (ci, co) in enumerate(((8, 16), (16, 16), (16, 3)), start=1):
        std = math.sqrt(2.0 / (27 * ci)) * (0.1 if k == 3 else 1.0)
        p["w%d" % k] = g.normal(0.0, std, (27, ci, co)).astype(np.float32)
        p["b%d" % k] = (0.05 * g.normal(size=co)).astype(np.float32)
    return p


def _train_inputs(case, seed):
    """Network input of each box (bf16 mesh, 8 channels, two of them zero) and
    the cell-sorted training records (x, y, z, box) and (target, weight)."""
    nm, nb = case["nm"], case["boxes"]
    gen = _gen(seed)
    x0 = torch.zeros(nb, nm, nm, nm, 8, device=DEV, dtype=torch.bfloat16)
    x0[..., :6] = torch.randn(nb, nm, nm, nm, 6, device=DEV, generator=gen)
    pos, tgt = [], []
    for b in range(nb):
        p = _clustered(nm ** 3, float(nm), 0.5, 0.2, max(1, nm ** 3 // 65536), gen).float()
        p[p >= nm] = 0.0
        c = p.floor().long() % nm
        key = (c[:, 2] * nm + c[:, 1]) * nm + c[:, 0]
        order = torch.argsort(key, stable=True)
        dense = torch.bincount(key, minlength=nm ** 3)[key] > 9
        t = torch.randn(nm ** 3, 4, device=DEV, generator=gen)
        t[:, 3] = torch.where(dense, 0.0, 1.0 / (t[:, 3] ** 2 + 1.0))
        pos.append(torch.cat([p, torch.full((nm ** 3, 1), float(b), device=DEV)], 1)[order])
        tgt.append(t[order])
    return x0, torch.cat(pos), torch.cat(tgt), _weights(seed + 1)


def _ic_sigma(nm):
    """Amplitudes of P(k) ~ k^-2 at every integer |n|^2, about half a cell of rms displacement."""
    n2 = np.arange(3 * (nm // 2 - 1) ** 2 + 1, dtype=np.float64)
    n2[0] = 1.0
    s = 0.1 * float(nm) ** 3 / np.sqrt(n2)
    s[0] = 0.0
    return s


IC = {"vel1": 0.32, "vel2": -0.27, "d2": -3.0 / 7.0, "scale": 0.6}  # momentum factors, D2/D1^2, D(a)/D(1)


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------

class State:
    pass


def _soa(pos):
    return [pos[:, a].contiguous() for a in range(3)]


def prepare(case, seed):
    import gadget_ng_pm_hip as pkg
    from gadget_ng_pm_hip import learned

    st = State()
    st.case = case
    kind = case["kind"]
    if kind == "pm":
        nm, box, n = case["nm"], case["box"], case["n"]
        cell = box / nm
        pos, idx = _pm_inputs(case, seed)
        st.k = n if idx is None else int(idx.numel())
        opts = {"r_split": case["r_split_cells"] * cell, "plummer_eps": case["eps_cells"] * cell,
                "deconvolve": case["deconvolve"]}
        if case["entry"] == "host":
            st.pos = pos.cpu().numpy()
            st.mass = np.full(n, 1.0 / n)
            st.idx = np.arange(n) if idx is None else idx.cpu().numpy()
            st.out = np.zeros((st.k, 3))
            if opts["r_split"] > 0.0:
                st.plan = pkg.Plan(nm, box, **opts)
            else:
                st.solver = pkg.PmSolver(nm, box, plummer_eps=opts["plummer_eps"] or None, deconvolve=case["deconvolve"])
                st.plan = None
            return st
        st.plan = pkg.Plan(nm, box, **opts)
        st.idx = idx
        if case["entry"] == "f64":
            st.pos, st.mass = pos, torch.ones(n, device=DEV, dtype=F64)
            st.out = torch.empty(st.k, 3, device=DEV, dtype=F64)
        else:
            st.pos, st.mass = _soa(pos), torch.ones(n, device=DEV)
            st.out = [torch.empty(st.k, device=DEV) for _ in range(3)]
    elif kind == "ensemble":
        boxes = _ensemble_inputs(case, seed)
        st.batch = pkg.Batch([{"grid_size": 2 * s, "box_size": float(s)} for s, _ in boxes])
        st.offsets = np.concatenate([[0], np.cumsum([p.shape[0] for _, p in boxes])])
        st.pos = _soa(torch.cat([p for _, p in boxes]))
        st.mass = torch.ones_like(st.pos[0])
        st.out = [torch.empty_like(st.mass) for _ in range(3)]
    elif kind == "pk":
        st.pos = _soa(_positions(case, seed).float())
        st.mass = torch.ones(case["n"], device=DEV)
        st.plan = pkg.Plan(case["nm"], case["box"])
    elif kind == "ic":
        st.plan = pkg.Plan(case["nm"], case["box"])
        st.sigma = _ic_sigma(case["nm"])
        st.seed = seed
        st.out = [torch.empty(case["nm"] ** 3, 3, device=DEV, dtype=F64) for _ in range(2)]
    elif kind == "sr":
        pos = _clustered(case["n"], case["box"], 0.5, 0.2, max(1, case["n"] // 65536), _gen(seed)).float()
        st.pos = _soa(pos)
        st.mass = torch.ones(case["n"], device=DEV)
        st.sr = learned.ShortRange()
        st.split = learned.SR_EXACT if case["split"] == "exact" else learned.SR_REFERENCE
        st.out = [torch.empty_like(st.mass) for _ in range(3)]
    elif kind == "learned":
        nm = case["nm"]
        pos, weights = _learned_inputs(case, seed)
        st.pos, st.mass = _soa(pos), torch.ones(nm ** 3, device=DEV)
        st.plan = pkg.Plan(nm, float(nm), keep_density=True, keep_potential=True)
        st.net = learned.Net(nm)
        st.net.set_params(weights)
        st.moments = torch.empty(nm ** 3 * 5, device=DEV, dtype=F64)
        st.out = [torch.empty_like(st.mass) for _ in range(3)]
    else:
        nm, nb = case["nm"], case["boxes"]
        x0, st.pos4, st.tgt4, weights = _train_inputs(case, seed)
        st.net = learned.Net(nm, max_boxes=nb)
        st.net.set_params(weights)
        torch.cuda.synchronize()
        learned._dcopy(st.net.device_buffer("x0"), x0.data_ptr(), x0.numel() * 2)
    return st


def run(st):
    case = st.case
    kind = case["kind"]
    if kind == "pm":
        if case["entry"] == "host":
            if st.plan is None:
                return st.solver.accelerations_for_indices(st.pos, st.mass, 0.0, 1.0, st.idx, out=st.out)
            return st.plan.accelerations_f64(st.pos, st.mass, 1.0, st.idx, out=st.out)
        idx = None if st.idx is None else st.idx.data_ptr()
        if case["entry"] == "f64":
            st.plan.solve_device_f64(st.pos.data_ptr(), st.mass.data_ptr(), case["n"], st.out.data_ptr(), 1.0,
                                     idx_ptr=idx, k=st.k)
        else:
            solve = st.plan.solve_device if case["entry"] == "f32" else st.plan.solve_device_soa64
            solve(*(p.data_ptr() for p in st.pos), st.mass.data_ptr(), case["n"], *(o.data_ptr() for o in st.out), 1.0,
                  idx_ptr=idx, k=st.k)
        return st.out
    if kind == "ensemble":
        st.batch.solve_device(*(p.data_ptr() for p in st.pos), st.mass.data_ptr(), st.offsets, 1.0,
                              *(o.data_ptr() for o in st.out))
        return st.out
    if kind == "pk":
        from gadget_ng_pm_hip import analysis
        k, pk, modes = analysis.power_spectrum_device(st.plan, *(p.data_ptr() for p in st.pos), st.mass.data_ptr(),
                                                      case["n"])
        return [k, pk, modes.astype(np.int64)]
    if kind == "ic":
        from gadget_ng_pm_hip import ic
        ic.zeldovich_2lpt_ics_device(st.plan, st.seed, st.sigma, IC["vel1"], IC["vel2"], IC["d2"], IC["scale"],
                                     st.out[0].data_ptr(), st.out[1].data_ptr())
        return st.out
    if kind == "sr":
        st.sr.accelerations_device(*(p.data_ptr() for p in st.pos), st.mass.data_ptr(), case["n"], case["box"],
                                   case["r_split"], 5.0 * case["r_split"], case["eps"] ** 2, 1.0, st.split,
                                   *(o.data_ptr() for o in st.out))
        return st.out
    if kind == "learned":
        nm = case["nm"]
        n, box = nm ** 3, float(nm)
        x, y, z = (p.data_ptr() for p in st.pos)
        out = [o.data_ptr() for o in st.out]
        st.plan.solve_device(x, y, z, st.mass.data_ptr(), n, *out, 1.0)
        rho, phi = st.plan.device_meshes()
        st.plan.cell_moments_device(st.moments.data_ptr())
        st.net.input_from_moments(0, rho, phi, 1.0, 100.0, st.moments.data_ptr())
        st.net.infer(1)
        st.net.apply_field(0, x, y, z, n, box, OUT_SCALE, rho, RHO_MAX, *out)
        return st.out
    nb = case["boxes"]
    st.net.train_step(nb, st.pos4.data_ptr(), st.tgt4.data_ptr(), st.pos4.shape[0], float(case["nm"]), OUT_SCALE, 1e-3)
    return [st.net.read("grad"), st.net.loss()]


OUT_SCALE = 3.0  # the typical force of a field particle in these units
RHO_MAX = 9.0    # cells above nine times the mean mass keep the PM force


# ---------------------------------------------------------------------------
# work: each input read once, each output written once
# ---------------------------------------------------------------------------

def _pm_flops(nm, n, k):
    m = nm ** 3
    fft = 2.5 * m * math.log2(m)  # one real transform
    return 4 * fft + 14 * m + 60 * n + 80 * k


def work(case):
    kind = case["kind"]
    if kind == "pm":
        n = case["n"]
        k = max(1, n // 4) if case["subset"] else n
        per = {"host": (32, 24), "f64": (32, 24), "soa64": (28, 12), "f32": (16, 12)}[case["entry"]]
        return {"bytes": n * per[0] + k * per[1] + (8 * k if case["subset"] else 0), "flops": _pm_flops(case["nm"], n, k)}
    if kind == "ensemble":
        sides = [(32, 48, 64, 96, 128)[(b * 3) % 5] for b in range(case["boxes"])]
        return {"bytes": sum(28 * s ** 3 for s in sides), "flops": sum(_pm_flops(2 * s, s ** 3, s ** 3) for s in sides)}
    if kind == "pk":
        m = case["nm"] ** 3
        return {"bytes": 16 * case["n"], "flops": 2.5 * m * math.log2(m) + 6 * m + 60 * case["n"]}
    if kind == "ic":
        m = case["nm"] ** 3
        # 3 + 6 inverse transforms, one forward and 3 inverse; half a mode per cell drawn
        return {"bytes": 48 * m, "flops": 13 * 2.5 * m * math.log2(m) + 1500 * m}
    if kind == "sr":
        # pairs inside the cut at the mean density (clustering adds to them), 25 operations each
        n, rc = case["n"], 5.0 * case["r_split"]
        return {"bytes": 28 * n, "flops": 25.0 * n * (4.0 / 3.0 * math.pi * rc ** 3 * n / case["box"] ** 3)}
    if kind == "learned":
        m = case["nm"] ** 3
        return {"bytes": 28 * m, "flops": _pm_flops(case["nm"], m, m) + 2.0 * 27 * (6 * 16 + 16 * 16 + 16 * 3) * m}
    m = case["nm"] ** 3 * case["boxes"]
    macs = 27 * (2 * 6 * 16 + 3 * 16 * 16 + 3 * 16 * 3)  # forward, weight gradient, data gradient
    return {"bytes": (12 + 32) * m + 4 * 11699 * 6, "flops": 2.0 * macs * m}


# ---------------------------------------------------------------------------
# the same outputs in 64 bits
# ---------------------------------------------------------------------------

def _cic(pos, box, nm):
    """Base cell (n, 3) and in-cell fraction of f64 positions."""
    c = (pos * (nm / box)).remainder(nm)
    i = c.floor()
    return i.long() % nm, c - i


def _corners(i, f, nm):
    for a in range(8):
        b = [(a >> s) & 1 for s in range(3)]
        j = [(i[:, s] + b[s]) % nm for s in range(3)]
        w = 1.0
        for s in range(3):
            w = w * (f[:, s] if b[s] else 1.0 - f[:, s])
        yield (j[2] * nm + j[1]) * nm + j[0], w


def _add(acc, node, w):
    """acc[node] += w for |w| <= 1, in units of 2^-40 (integer sums: exact and quick where many share a node)."""
    acc.index_add_(0, node, torch.round(w * 2.0 ** 40).long())


def _deposit(pos, mass, box, nm):
    rho = torch.zeros(nm ** 3, device=DEV, dtype=torch.int64)
    for lo in range(0, pos.shape[0], CHUNK):
        i, f = _cic(pos[lo:lo + CHUNK].to(F64), box, nm)
        for node, w in _corners(i, f, nm):
            _add(rho, node, w)
    return (rho.to(F64) * (mass * 2.0 ** -40)).view(nm, nm, nm)


def _gather(meshes, pos, box, nm):
    """(n, len(meshes)) interpolated values."""
    out = torch.empty(pos.shape[0], len(meshes), device=DEV, dtype=F64)
    for lo in range(0, pos.shape[0], CHUNK):
        i, f = _cic(pos[lo:lo + CHUNK].to(F64), box, nm)
        part = torch.zeros(i.shape[0], len(meshes), device=DEV, dtype=F64)
        for node, w in _corners(i, f, nm):
            for c, m in enumerate(meshes):
                part[:, c] += w * m.reshape(-1)[node]
        out[lo:lo + CHUNK] = part
    return out


def _phi_hat(rho, box, nm, g, r_s=0.0, eps=0.0, deconvolve=False):
    """The potential factor phi of each mode: the force is IFFT(-i n phi), unnormalised."""
    hat = torch.fft.rfftn(rho)
    n = (_freqs(nm)[:, None, None], _freqs(nm)[None, :, None], _rfreqs(nm)[None, None, :])
    n2 = n[0] ** 2 + n[1] ** 2 + n[2] ** 2
    n2[0, 0, 0] = 1.0
    kf = 2.0 * math.pi / box
    hat *= -(2.0 * g / box ** 2) * torch.exp(-kf * kf * (0.5 * r_s ** 2 + eps ** 2) * n2) / n2
    hat[0, 0, 0] = 0.0
    if deconvolve:
        for a in n:
            hat *= torch.sinc(a / nm) ** -4
    return hat


def _force_meshes(phi, nm):
    """(F_x, F_y, F_z) meshes [z, y, x]; the Nyquist plane of each axis has no derivative."""
    out = []
    for axis in (2, 1, 0):
        n = _rfreqs(nm) if axis == 2 else _freqs(nm)
        n = n.clone()
        n[nm // 2] = 0.0
        shape = [1, 1, 1]
        shape[axis] = n.numel()
        out.append(torch.fft.irfftn(phi * (-1j * n.view(shape)), s=(nm, nm, nm), norm="forward"))
    return out


def _pm_exact(pos, mass, box, nm, at, g=1.0, **filters):
    rho = _deposit(pos, mass, box, nm)
    phi = _phi_hat(rho, box, nm, g, **filters)
    del rho
    meshes = _force_meshes(phi, nm)
    del phi
    return _gather(meshes, at, box, nm)


def _pk_exact(case, seed):
    nm, box, n = case["nm"], case["box"], case["n"]
    hat = torch.fft.rfftn(_deposit(_positions(case, seed).float(), 1.0, box, nm))
    a, h = _freqs(nm), _rfreqs(nm)
    n2 = a[:, None, None] ** 2 + a[None, :, None] ** 2 + h[None, None, :] ** 2
    p = (hat.real ** 2 + hat.imag ** 2) * (box ** 3 / n) ** 2
    for f in (a[:, None, None], a[None, :, None], h[None, None, :]):
        p = p / torch.sinc(f / nm) ** 2
    weight = torch.full((nm // 2 + 1,), 2.0, device=DEV, dtype=F64)
    weight[0] = weight[-1] = 1.0
    shell = (n2.sqrt() - 0.5).floor().long()
    ok = (n2 > 0) & (shell < nm // 2) & (n2.sqrt() < nm / 2 + 0.5)
    wt = weight.expand_as(n2)[ok]
    sums = torch.bincount(shell[ok], weights=p[ok] * wt, minlength=nm // 2)
    modes = torch.bincount(shell[ok], weights=wt, minlength=nm // 2)
    k = (torch.arange(nm // 2, device=DEV, dtype=F64) + 1.0) * (2.0 * math.pi / box)
    have = modes > 0
    return [k[have], (sums / modes)[have], None]


def _s64(v):
    """A 64-bit pattern as the signed integer torch holds it in."""
    return v - (1 << 64) if v >= 1 << 63 else v


def _shr(x, r):
    return (x >> r) & ((1 << (64 - r)) - 1)


def _hash(x):
    """murmur3's 64-bit finaliser."""
    x = (x ^ _shr(x, 33)) * _s64(0xFF51AFD7ED558CCD)
    x = (x ^ _shr(x, 33)) * _s64(0xC4CEB9FE1A85EC53)
    return x ^ _shr(x, 33)


def _gaussian(seed):
    """One normal value for each 64-bit seed: ChaCha12 keyed by eight PCG32
    outputs, two 53-bit uniforms, the cosine branch of Box-Muller."""
    m32 = 0xFFFFFFFF
    key = []
    st = seed
    for _ in range(8):
        st = st * 6364136223846793005 + _s64(11634580027462260723)
        xs = _shr(_shr(st, 18) ^ st, 27) & m32
        rot = _shr(st, 59)
        key.append(((xs >> rot) | (xs << ((32 - rot) & 31))) & m32)
    const = [0x61707865, 0x3320646E, 0x79622D32, 0x6B206574]
    x = [torch.full_like(seed, c) for c in const] + key + [torch.zeros_like(seed) for _ in range(4)]

    def rotl(v, r):
        return ((v << r) | (v >> (32 - r))) & m32

    def quarter(a, b, c, d):
        x[a] = (x[a] + x[b]) & m32
        x[d] = rotl(x[d] ^ x[a], 16)
        x[c] = (x[c] + x[d]) & m32
        x[b] = rotl(x[b] ^ x[c], 12)
        x[a] = (x[a] + x[b]) & m32
        x[d] = rotl(x[d] ^ x[a], 8)
        x[c] = (x[c] + x[d]) & m32
        x[b] = rotl(x[b] ^ x[c], 7)

    for _ in range(6):
        for q in ((0, 4, 8, 12), (1, 5, 9, 13), (2, 6, 10, 14), (3, 7, 11, 15),
                  (0, 5, 10, 15), (1, 6, 11, 12), (2, 7, 8, 13), (3, 4, 9, 14)):
            quarter(*q)
    w = [(x[i] + const[i]) & m32 for i in range(4)]
    u1 = ((w[1] << 21) | (w[0] >> 11)).to(F64) / 9007199254740992.0
    u2 = ((w[3] << 21) | (w[2] >> 11)).to(F64) / 9007199254740992.0
    return torch.sqrt(-2.0 * torch.log(u1.clamp(min=1e-300))) * torch.cos(2.0 * math.pi * u2)


def _ic_exact(case, seed):
    nm, box = case["nm"], case["box"]
    h = nm // 2
    a = torch.arange(nm, device=DEV)
    ix, iy, iz = a[:, None, None], a[None, :, None], torch.arange(h + 1, device=DEV)[None, None, :]
    flat = (ix * nm + iy) * nm + iz
    other = ((-ix % nm) * nm + (-iy % nm)) * nm + (-iz % nm)
    ms = _hash(_hash(torch.minimum(flat, other)) ^ _s64(seed))
    re = _gaussian(ms)
    im = _gaussian(_hash(ms ^ _s64(0x9E3779B97F4A7C15))) * torch.where(flat < other, 1.0, -1.0)
    n = (_freqs(nm)[:, None, None], _freqs(nm)[None, :, None], _rfreqs(nm)[None, None, :])
    n2 = n[0] ** 2 + n[1] ** 2 + n[2] ** 2
    live = (n2 > 0) & (ix != h) & (iy != h) & (iz != h)
    sigma = torch.from_numpy(_ic_sigma(nm)).to(DEV)
    amp = torch.where(live, sigma[n2.long().clamp(max=sigma.numel() - 1)], 0.0)
    n2[0, 0, 0] = 1.0
    pot = torch.complex(amp * re, amp * im) / n2  # delta-hat / |n|^2

    def back(v):
        return torch.fft.irfftn(v, s=(nm, nm, nm))  # with the 1 / nm^3

    d = box / nm
    der = {(p, q): back(-n[p] * n[q] * pot) for p, q in ((0, 0), (1, 1), (2, 2), (0, 1), (1, 2), (0, 2))}
    src = der[0, 0] * der[1, 1] + der[1, 1] * der[2, 2] + der[2, 2] * der[0, 0]
    src -= der[0, 1] ** 2 + der[1, 2] ** 2 + der[0, 2] ** 2
    del der
    s_hat = torch.where(live, torch.fft.rfftn(src) / n2, 0.0)
    pos = torch.empty(nm ** 3, 3, device=DEV, dtype=F64)
    vel = torch.empty_like(pos)
    for c in range(3):
        p1 = back(1j * n[c] * pot) * (d * IC["scale"])
        p2 = back(-1j * n[c] * s_hat) * (d * IC["scale"] ** 2)
        shape = [1, 1, 1]
        shape[c] = nm
        q = ((a.to(F64) + 0.5) * d).view(shape)
        pos[:, c] = (q + p1 + IC["d2"] * p2).reshape(-1).remainder(box)
        vel[:, c] = (p1 * IC["vel1"] + p2 * IC["vel2"]).reshape(-1)
    return [pos, vel]


def _sr_exact(case, seed):
    """Every pair inside the cut, cell by cell over a chaining mesh."""
    n, box, rs = case["n"], case["box"], case["r_split"]
    rc, eps2 = 5.0 * rs, case["eps"] ** 2
    pos = _clustered(n, box, 0.5, 0.2, max(1, n // 65536), _gen(seed)).float().to(F64)
    nc = int(box / rc)
    c = (pos * (nc / box)).floor().long() % nc
    cell = (c[:, 2] * nc + c[:, 1]) * nc + c[:, 0]
    order = torch.argsort(cell)
    srt = pos[order]
    start = torch.searchsorted(cell[order], torch.arange(nc ** 3 + 1, device=DEV)).tolist()
    acc = torch.zeros(n, 3, device=DEV, dtype=F64)
    for cz in range(nc):
        for cy in range(nc):
            for cx in range(nc):
                lo, hi = start[(cz * nc + cy) * nc + cx], start[(cz * nc + cy) * nc + cx + 1]
                if lo == hi:
                    continue
                near = []
                for o in range(27):
                    u = ((cz + o // 9 - 1) % nc * nc + (cy + o // 3 % 3 - 1) % nc) * nc + (cx + o % 3 - 1) % nc
                    if start[u + 1] > start[u]:
                        near.append(srt[start[u]:start[u + 1]])
                near = torch.cat(near)
                step = max(1, (1 << 25) // near.shape[0])
                for b in range(lo, hi, step):
                    e = min(hi, b + step)
                    dv = near[None, :, :] - srt[b:e, None, :]
                    dv -= box * torch.round(dv / box)
                    r2 = (dv ** 2).sum(2)
                    ok = (r2 <= rc * rc) & (r2 > 0)
                    r = torch.sqrt(r2 + eps2)
                    x = r / (math.sqrt(2.0) * rs)
                    s = torch.special.erfc(x)
                    if case["split"] == "exact":
                        s = s + 2.0 / math.sqrt(math.pi) * x * torch.exp(-x * x)
                    w = torch.where(ok, s / r ** 3, 0.0)
                    acc[b:e] = torch.einsum("ij,ijc->ic", w, dv)
    out = torch.empty_like(acc)
    out[order] = acc
    return [out[:, a].contiguous() for a in range(3)]


def _conv(x, w, b):
    """Periodic 3^3 convolution of [z, y, x, c] (leading box axis allowed), tap (dz, dy, dx) reading cell + offset."""
    shifts = [(1 - t // 9, 1 - t // 3 % 3, 1 - t % 3) for t in range(27)]
    if x.numel() <= 1 << 23:  # all taps side by side: one product
        taps = torch.cat([torch.roll(x, s, dims=(-4, -3, -2)) for s in shifts], -1)
        return taps @ w.reshape(-1, w.shape[-1]) + b
    out = b.expand(*x.shape[:-1], b.numel())
    for t, s in enumerate(shifts):
        out = out + torch.roll(x, s, dims=(-4, -3, -2)) @ w[t]
    return out


def _network(x, p):
    silu = torch.nn.functional.silu
    h = silu(_conv(x, p["w1"], p["b1"]))
    h = silu(_conv(h, p["w2"], p["b2"]))
    return _conv(h, p["w3"], p["b3"])


def _weights64(p):
    return {k: torch.from_numpy(v).to(DEV).to(F64) for k, v in p.items()}


def _learned_exact(case, seed):
    nm = case["nm"]
    box = float(nm)
    pos, weights = _learned_inputs(case, seed)
    rho = _deposit(pos, 1.0, box, nm)
    hat = _phi_hat(rho, box, nm, 1.0)
    acc = _gather(_force_meshes(hat, nm), pos, box, nm)
    pot = torch.fft.irfftn(hat, s=(nm, nm, nm), norm="forward") * (box / (2.0 * math.pi))
    del hat
    smooth = pot
    for dim in range(3):
        smooth = sum(torch.roll(smooth, s, dims=dim) for s in range(-3, 4)) / 7.0
    i, f = _cic(pos.to(F64), box, nm)
    base = (i[:, 2] * nm + i[:, 1]) * nm + i[:, 0]
    f = f - 0.5

    def total(v):
        acc = torch.zeros(nm ** 3, device=DEV, dtype=torch.int64)
        _add(acc, base, v)
        return acc.to(F64) * 2.0 ** -40

    m0, dip = total(torch.ones_like(f[:, 0])), [total(f[:, a].contiguous()) for a in range(3)]
    spread = total((f ** 2).sum(1)) - sum(v * v for v in dip) / m0.clamp(min=1e-300)
    x = torch.stack([rho.view(-1) - 1.0, (pot - smooth).view(-1) / 100.0, *dip,
                     torch.where(m0 > 0, spread.clamp(min=0.0), 0.0)], 1).view(nm, nm, nm, 6)
    p = _weights64(weights)
    p["w1"] = p["w1"][:, :6]
    y = _network(x, p)
    corr = _gather([y[..., a].contiguous() for a in range(3)], pos, box, nm)
    acc += torch.where((rho.view(-1)[base] <= RHO_MAX)[:, None], OUT_SCALE * corr, 0.0)
    return [acc[:, a].contiguous() for a in range(3)]


def _train_exact(case, seed):
    nm = case["nm"]
    x0, pos4, tgt4, weights = _train_inputs(case, seed)
    p = {k: v.requires_grad_() for k, v in _weights64(weights).items()}
    n = pos4.shape[0]
    loss = 0.0
    for b in range(case["boxes"]):  # the loss is a sum over the boxes, and so are the gradients
        mine = pos4[:, 3] == b
        y = _network(x0[b].to(F64), p).reshape(-1, 3)
        i, f = _cic(pos4[mine, :3].to(F64), float(nm), nm)
        v = sum(w[:, None] * y[node] for node, w in _corners(i, f, nm))
        t = tgt4[mine].to(F64)
        part = (t[:, 3:] * (OUT_SCALE * v - t[:, :3]) ** 2).sum() / n
        part.backward()
        loss += float(part.detach())
    grad = torch.cat([p[k].grad.reshape(-1) for k in ("w1", "b1", "w2", "b2", "w3", "b3")])
    return [grad, loss]


def exact(case, seed):
    kind = case["kind"]
    if kind == "pm":
        pos, idx = _pm_inputs(case, seed)
        cell = case["box"] / case["nm"]
        mass = float(np.float32(1.0 / case["n"])) if case["entry"] == "host" else 1.0
        acc = _pm_exact(pos, mass, case["box"], case["nm"], pos if idx is None else pos[idx],
                        r_s=case["r_split_cells"] * cell, eps=case["eps_cells"] * cell, deconvolve=case["deconvolve"])
        return acc if case["entry"] in ("host", "f64") else [acc[:, a].contiguous() for a in range(3)]
    if kind == "ensemble":
        acc = torch.cat([_pm_exact(p, 1.0, float(s), 2 * s, p) for s, p in _ensemble_inputs(case, seed)])
        return [acc[:, a].contiguous() for a in range(3)]
    return {"pk": _pk_exact, "ic": _ic_exact, "sr": _sr_exact, "learned": _learned_exact,
            "train": _train_exact}[kind](case, seed)
