"""The workloads that say how fast this framework is: calls that its users make, through its
public entry points, over the sizes of its own configurations, tests and benchmark.

A case is a dict of plain values.  Its "kind" names the call:

  points      ops.field_points: the field at a few points (point_field, point_mag)
  grid        ops.field_grid: field and / or potential on a box grid (volume, volume_ESP)
  volumes     batch.batch_volume: the grids of several MD frames in one call
  topo        ops.topo: streamlines and their histogram (topo, topo_GPU), Euler or RK4
  dipole      ops.topo_dipole: streamlines in the field of point dipoles
  topos       batch.batch_topo: the streamlines of several MD frames in one call
  residues    residue_breakdown.residue_counts: each residue's streamlines over shared starts
  cluster     clusterhist: shared bins, histograms and chi-square matrix of many frames

Charges are "ball" (uniform in a ball, 3 A clear of the box, q ~ N(0, 0.4) e) or "md"
(residue-like clusters with charges anywhere, in the box too, and Gaussian jitter), as
pycpet_amd.workloads makes them.  Inputs are float32 (the library's only input type) and lie
on the GPU, except where the entry point takes host arrays by its nature (residues, cluster).
"""
import math

import numpy as np
import torch

from pycpet_amd import batch, clusterhist, ops, residue_breakdown
from pycpet_amd import workloads as W

K = 14.3996451  # eV A / e^2


def listed():
    return [
        # the field at the box centre of a whole protein frame: the smallest call, one
        # point; examples' 7,890 charges
        {"name": "point_field_8k", "kind": "points", "charges": 7890, "points": 1},
        # the plain volume configuration: field and ESP on the 21^3 grid of 2,000 charges
        {"name": "volume_2k_21", "kind": "grid", "charges": 2000, "layout": "ball", "radius": 25.0,
         "nx": 21, "ny": 21, "nz": 21, "step": 0.2, "E": True, "phi": True},
        # an anisotropic box of an MD frame: ragged charge count and odd grid sizes
        {"name": "volume_12k_ragged", "kind": "grid", "charges": 12345, "layout": "md",
         "radius": 45.0, "nx": 61, "ny": 47, "nz": 38, "step": 0.1, "E": True, "phi": False},
        # the largest volume configuration: 30,000 clustered charges on 101^3 points
        {"name": "volume_30k_101", "kind": "grid", "charges": 30000, "layout": "md",
         "radius": 45.0, "nx": 101, "ny": 101, "nz": 101, "step": 0.1, "E": True, "phi": False},
        # the same frame for the volume_ESP method
        {"name": "esp_30k_101", "kind": "grid", "charges": 30000, "layout": "md",
         "radius": 45.0, "nx": 101, "ny": 101, "nz": 101, "step": 0.1, "E": False, "phi": True},
        # eight volume jobs of the mixed MD set in one call (3k-40k atoms, 21^3 to 81^3)
        {"name": "volumes_md_8", "kind": "volumes", "frames": 8, "min_charges": 3000,
         "max_charges": 40000},
        # the streamline benchmark: 5,000 charges, 100,000 starts, h = 0.001 A, 20 x 20 bins
        {"name": "topo_5k_100k", "kind": "topo", "charges": 5000, "layout": "ball",
         "radius": 35.0, "starts": 100000, "box": 1.5, "h": 0.001, "cap": 2000, "rk4": False,
         "bins": 20},
        # one frame of the options-file topo driver: 22^3 starts, h = 0.005 A
        {"name": "topo_10k_driver", "kind": "topo", "charges": 10000, "layout": "ball",
         "radius": 35.0, "starts": 10648, "box": 1.5, "h": 0.005, "cap": 0, "rk4": False,
         "bins": 0},
        # the streamline configuration's RK4 integrator at the MD frames' 20,000 starts
        {"name": "topo_5k_rk4", "kind": "topo", "charges": 5000, "layout": "ball",
         "radius": 35.0, "starts": 20000, "box": 1.5, "h": 0.001, "cap": 2000, "rk4": True,
         "bins": 0},
        # eight streamline jobs of the mixed MD set in one call, with the driver's starts
        {"name": "topos_md_8", "kind": "topos", "frames": 8, "min_charges": 3000,
         "max_charges": 40000, "starts": 10648, "h": 0.005, "cap": 0},
        # the residue breakdown of a frame: 200 residues of 8-24 charges over 20,000 starts
        {"name": "residues_200x20k", "kind": "residues", "residues": 200, "starts": 20000,
         "h": 0.001, "cap": 2000},
        # the cluster step after topo: 256 frames of 20,000 feature rows
        {"name": "cluster_256x20k", "kind": "cluster", "frames": 256, "rows": 20000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# pairs of charge and field evaluation that the largest listed case has, about
_MOST_PAIRS = 4.0e11


def draw(rng):
    kind = rng.choice(["points", "grid", "grid", "grid", "volumes", "topo", "topo", "dipole",
                       "topos", "residues", "cluster"])
    if kind == "points":
        return {"kind": kind, "charges": _log(rng, 500, 60000), "points": _log(rng, 1, 3000)}
    if kind == "grid":
        what = rng.choice(["E", "E", "phi", "both"])
        return {"kind": kind, "charges": _log(rng, 1000, 40000),
                "layout": rng.choice(["ball", "md"]), "radius": rng.choice([25.0, 35.0, 45.0]),
                "nx": _log(rng, 11, 101), "ny": _log(rng, 11, 101), "nz": _log(rng, 11, 101),
                "step": rng.choice([0.05, 0.1, 0.2]) if what != "both" else 0.1,
                "E": what != "phi", "phi": what != "E"}
    if kind == "volumes":
        lo = _log(rng, 1000, 10000)
        return {"kind": kind, "frames": rng.randint(2, 12), "min_charges": lo,
                "max_charges": min(40000, 4 * lo)}
    if kind in ("topo", "dipole"):
        c = {"kind": kind, "charges": _log(rng, 300, 20000), "layout": "ball", "radius": 35.0,
             "starts": _log(rng, 2000, 100000), "box": rng.choice([0.6, 1.0, 1.5]),
             "h": rng.choice([0.001, 0.005, 0.01]), "cap": rng.choice([0, 1000, 2000])}
        if kind == "topo":
            c["rk4"] = rng.random() < 0.3
            c["bins"] = rng.choice([0, 20, 33])
            c["layout"] = rng.choice(["ball", "ball", "md"])
        while _pairs(c) > _MOST_PAIRS / 4:
            c["starts"] = c["starts"] * 2 // 3
        return c
    if kind == "topos":
        lo = _log(rng, 500, 5000)
        return {"kind": kind, "frames": rng.randint(2, 6), "min_charges": lo,
                "max_charges": 3 * lo, "starts": _log(rng, 2000, 20000),
                "h": rng.choice([0.001, 0.005]), "cap": 2000}
    if kind == "residues":
        return {"kind": kind, "residues": rng.randint(20, 300), "starts": _log(rng, 2000, 20000),
                "h": rng.choice([0.001, 0.005]), "cap": 2000}
    return {"kind": kind, "frames": rng.randint(20, 256), "rows": _log(rng, 2000, 20000)}


# ---- inputs ---------------------------------------------------------------


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _axes(c):
    """The reference's inclusive box grid: nx points over +-(nx - 1) step / 2."""
    half = [0.5 * (n - 1) * c["step"] for n in (c["nx"], c["ny"], c["nz"])]
    return [np.linspace(-d, d, n).astype(np.float32)
            for d, n in zip(half, (c["nx"], c["ny"], c["nz"]))]


def _charges(layout, n, radius, box, seed):
    if layout == "ball":
        return W.ball_exclusion(n, radius, box, 3.0, seed)
    x, q = W.clustered(-(-n // 10), 10, radius, 1.5, -3.0, seed)
    return np.ascontiguousarray(x[:n]), np.ascontiguousarray(q[:n])


def _starts(c, seed):
    return W.topo_starts(c["starts"], (c["box"],) * 3, c["h"], c["cap"] or None,
                         seed=seed % (1 << 31), start_seed=(seed + 1) % (1 << 31))[:2]


def _md_set(c, seed, kind):
    """Frames of the mixed MD-like set: atom counts uniform in the case's range, grid edges
    21, 41, 61 and 81 in turn."""
    rng = np.random.default_rng(seed)
    base = W.md_base(c["max_charges"], seed)
    out = []
    for i in range(c["frames"]):
        n = int(rng.integers(c["min_charges"], c["max_charges"] // 10 * 10 + 1)) // 10 * 10
        out.append(W.md_frame(base, i, kind, max(n, 10), edge=(21, 41, 61, 81)[i % 4],
                              seed=seed % 100000, rng=rng,
                              topo_starts_per_frame=c.get("starts", 0), h=c.get("h", 0.001),
                              cap=c.get("cap") or None))
    return out


def _residue_sets(c, seed):
    rng = np.random.default_rng(seed)
    xs, qs = [], []
    for _ in range(c["residues"]):
        n = int(rng.integers(8, 25))
        centre = rng.standard_normal(3)
        centre *= rng.uniform(5.0, 14.0) / np.linalg.norm(centre)
        xs.append((centre + rng.normal(0.0, 1.2, (n, 3))).astype(np.float32))
        qs.append(rng.normal(0.0, 0.4, n).astype(np.float32))
    return xs, qs


def _feature_frames(c, seed):
    """Frames of feature rows, like .top files.  The rows of the whole set depend on the sizes
    alone, so that the shared bins (and the shapes of the results) do too; the seed puts frames
    and rows in order."""
    rng = np.random.default_rng(c["frames"] * 1000003 + c["rows"])
    feats = [np.column_stack([np.abs(rng.normal(1.0 + 0.002 * f, 0.3, c["rows"])),
                              np.abs(rng.normal(5.0, 2.0, c["rows"]))])
             for f in range(c["frames"])]
    rng = np.random.default_rng(seed)
    return [feats[f][rng.permutation(c["rows"])] for f in rng.permutation(c["frames"])]


def prepare(case, seed):
    c, kind = case, case["kind"]
    s = {"case": c}
    if kind == "points":
        x, q = W.ball_exclusion(c["charges"], 35.0, 1.0, 1.0, seed)
        pts = np.random.default_rng(seed + 1).uniform(-1.0, 1.0, (c["points"], 3))
        if c["points"] == 1:
            pts *= 0.0  # the box centre
        s.update(x=_dev(x), q=_dev(q), pts=_dev(pts.astype(np.float32)))
    elif kind == "grid":
        axes = _axes(c)
        x, q = _charges(c["layout"], c["charges"], c["radius"],
                        max(float(a[-1]) for a in axes), seed)
        s.update(x=_dev(x), q=_dev(q), axes=[_dev(a) for a in axes])
    elif kind == "volumes":
        s["frames"] = [{"x": _dev(f["x"]), "q": _dev(f["q"]),
                        "axes": tuple(_dev(a) for a in f["axes"])}
                       for f in _md_set(c, seed, "volume")]
    elif kind in ("topo", "dipole"):
        x, q = _charges(c["layout"], c["charges"], c["radius"], c["box"], seed)
        st, it = _starts(c, seed)
        s.update(x=_dev(x), q=_dev(q), starts=_dev(st), n_iter=_dev(it),
                 dims=np.full(3, c["box"], np.float32))
        if kind == "dipole":
            s["q"] = _dev(np.random.default_rng(seed + 2)
                          .standard_normal((c["charges"], 3)).astype(np.float32))
        elif c["bins"]:
            # distances up to the box diagonal, curvatures up to that of a 0.5 A circle
            s["edges"] = (_dev(np.linspace(0.0, 2 * math.sqrt(3.0) * c["box"], c["bins"] + 1)),
                          _dev(np.linspace(0.0, 2.0, c["bins"] + 1)))
    elif kind == "topos":
        s["frames"] = [{"x": _dev(f["x"]), "q": _dev(f["q"]), "starts": _dev(f["starts"]),
                        "n_iter": _dev(f["n_iter"]), "h": f["h"], "dims": f["dims"]}
                       for f in _md_set(c, seed, "topo")]
    elif kind == "residues":
        s["xs"], s["qs"] = _residue_sets(c, seed)
        s["starts"], s["n_iter"] = _starts(dict(c, box=1.5), seed)
        s["edges"] = (np.linspace(0.0, 3.2, 21), np.linspace(0.0, 40.0, 21))
    elif kind == "cluster":
        s["feats"] = _feature_frames(c, seed)
    return s


# ---- one pass -------------------------------------------------------------


def _streams(r):
    out = {"feats": r.feats, "steps": r.steps, "exited": r.exited}
    if r.hist is not None:
        out["hist"] = r.hist
    return out


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "points":
        return {"E": ops.field_points(s["pts"], s["x"], s["q"], soften=False)[0]}
    if kind == "grid":
        E, phi = ops.field_grid(*s["axes"], s["x"], s["q"], want_E=c["E"], want_phi=c["phi"])
        return {k: v for k, v in (("E", E), ("phi", phi)) if v is not None}
    if kind == "volumes":
        return [E for E, _ in batch.batch_volume(s["frames"])]
    if kind == "topo":
        return _streams(ops.topo(s["starts"], s["n_iter"], c["h"], s["dims"], s["x"], s["q"],
                                 edges=s.get("edges"),
                                 integrator="rk4" if c["rk4"] else "euler"))
    if kind == "dipole":
        return _streams(ops.topo_dipole(s["starts"], s["n_iter"], c["h"], s["dims"], s["x"],
                                        s["q"]))
    if kind == "topos":
        return [_streams(r) for r in batch.batch_topo(s["frames"])]
    if kind == "residues":
        return {"counts": residue_breakdown.residue_counts(
            s["xs"], s["qs"], s["starts"], s["n_iter"], c["h"], (1.5,) * 3, s["edges"])}
    hist = clusterhist.histograms_from_features(s["feats"])
    return {"hist": hist, "dist": clusterhist.construct_distance_matrix(hist)}


# ---- what a pass cannot do without ----------------------------------------


def _mean_steps(c):
    """Steps of a streamline, about: the mean step limit, shortened by the streamlines that
    leave the box (a path of about 1.7 half-widths)."""
    box = c.get("box", 1.5)
    top = 2 * math.sqrt(3.0) * box / c["h"]
    cap = min(c["cap"] or top, top)
    mean = cap - 0.5 * cap * cap / top
    return 1.0 / (1.0 / mean + c["h"] / (1.7 * box))


def _pairs(c):
    """Pairs of source and field evaluation of the sums that the call is defined by."""
    kind = c["kind"]
    if kind == "points":
        return float(c["points"]) * c["charges"]
    if kind == "grid":
        return float(c["nx"]) * c["ny"] * c["nz"] * c["charges"]
    if kind == "volumes":  # edges 21, 41, 61 and 81 in turn
        return c["frames"] * (21**3 + 41**3 + 61**3 + 81**3) / 4 * (
            0.5 * (c["min_charges"] + c["max_charges"]))
    if kind in ("topo", "dipole"):
        return float(c["starts"]) * (_mean_steps(c) * (4 if c.get("rk4") else 1) + 4) * c["charges"]
    if kind == "topos":
        return c["frames"] * c["starts"] * _mean_steps(c) * (
            0.5 * (c["min_charges"] + c["max_charges"]))
    if kind == "residues":
        return c["residues"] * c["starts"] * _mean_steps(c) * 16.0
    return 0.0


def work(case):
    """Inputs once and outputs once; 18 operations a pair for the field, 11 for the
    potential, 20 for both, 33 for a dipole, 5 a bin of two histograms."""
    c, kind = case, case["kind"]
    per = 18
    if kind == "points":
        b = 16 * c["charges"] + 24 * c["points"]
    elif kind == "grid":
        m = c["nx"] * c["ny"] * c["nz"]
        b = 16 * c["charges"] + m * (12 * c["E"] + 4 * c["phi"])
        per = 20 if c["E"] and c["phi"] else 18 if c["E"] else 11
    elif kind == "volumes":
        b = c["frames"] * (8 * (c["min_charges"] + c["max_charges"])
                           + 3 * (21**3 + 41**3 + 61**3 + 81**3))
    elif kind in ("topo", "dipole"):
        b = (24 if kind == "dipole" else 16) * c["charges"] + 40 * c["starts"]
        per = 33 if kind == "dipole" else 18
    elif kind == "topos":
        b = c["frames"] * (8 * (c["min_charges"] + c["max_charges"]) + 40 * c["starts"])
    elif kind == "residues":
        b = c["residues"] * (16 * 16 + 8 * 400) + 16 * c["starts"]
    else:
        rows, bins = c["frames"] * c["rows"], 6700 * (c["rows"] / 20000.0) ** (2 / 3)
        return {"bytes": 16 * rows + 8 * c["frames"] * (bins + c["frames"]),
                "flops": 5.0 * c["frames"] ** 2 / 2 * bins}
    return {"bytes": float(b), "flops": per * _pairs(c)}


# ---- the same results in 64 bits ------------------------------------------

_MOST_EXACT_PAIRS = 4.0e10


def _field64(p, x, q, floor, E=True, phi=False):
    """Field and potential at the FP64 points p of FP64 charges, in slabs of points."""
    oE = torch.empty((p.shape[0], 3), dtype=torch.float64, device=p.device) if E else None
    oP = torch.empty(p.shape[0], dtype=torch.float64, device=p.device) if phi else None
    per = max(1, 30_000_000 // x.shape[0])
    for a in range(0, p.shape[0], per):
        d = [p[a:a + per, k, None] - x[None, :, k] for k in range(3)]
        r2 = d[0] * d[0]
        r2 += d[1] * d[1]
        r2 += d[2] * d[2]
        if phi:
            oP[a:a + per] = K * (r2.rsqrt() @ q)
        if E:
            if floor:
                r2.clamp_(min=1e-6)
            w = r2.rsqrt_()
            w = w * w * w * q
            for k in range(3):
                oE[a:a + per, k] = K * (w * d[k]).sum(1)
    return oE, oP


def _mesh64(axes):
    return torch.stack(torch.meshgrid(*[a.double() for a in axes], indexing="ij"),
                       -1).reshape(-1, 3)


def _unit64(p, x, q):
    E = _field64(p, x, q, False)[0]
    return E / E.norm(dim=1, keepdim=True)


def _step64(p, x, q, h, rk4):
    u = _unit64(p, x, q)
    if not rk4:
        return p + h * u
    v = _unit64(p + 0.5 * h * u, x, q)
    w = _unit64(p + 0.5 * h * v, x, q)
    z = _unit64(p + h * w, x, q)
    return p + h / 6.0 * (u + 2.0 * v + 2.0 * w + z)


def _curvature64(p, x, q, h, rk4):
    p1 = _step64(p, x, q, h, rk4)
    p2 = _step64(p1, x, q, h, rk4)
    v1, v2 = p1 - p, p2 - 2.0 * p1 + p
    return torch.linalg.cross(v1, v2).norm(dim=1) / v1.norm(dim=1) ** 3


def _topo64(s, c):
    x, q = s["x"].double(), s["q"].double()
    h = float(np.float32(c["h"]))
    box = torch.from_numpy(s["dims"].astype(np.float64)).cuda()
    p0 = s["starts"].double()
    p, left = p0.clone(), s["n_iter"].long().clone()
    live = (left > 0).nonzero().ravel()
    while live.numel():
        n = _step64(p[live], x, q, h, c["rk4"])
        p[live] = n
        left[live] -= 1
        live = live[(n.abs() <= box).all(1) & (left[live] > 0)]
    kappa = 0.5 * (_curvature64(p0, x, q, h, c["rk4"]) + _curvature64(p, x, q, h, c["rk4"]))
    return torch.stack([(p0 - p).norm(dim=1), kappa], 1)


def _edges64(v, n):
    """numpy.histogram2d's edges for the width 2 IQR / n^(1/3) over [min, max]."""
    lo, hi = v.min(), v.max()
    p25, p75 = np.percentile(v, [25, 75])
    return np.linspace(lo, hi, int((hi - lo) / (2 * (p75 - p25) / n ** (1 / 3))) + 1)


def exact(case, seed):
    c, kind = case, case["kind"]
    if _pairs(c) > _MOST_EXACT_PAIRS or kind in ("dipole", "topos", "residues"):
        return None
    s = prepare(c, seed)
    if kind == "points":
        return {"E": _field64(s["pts"].double(), s["x"].double(), s["q"].double(), False)[0]}
    if kind == "grid":
        E, phi = _field64(_mesh64(s["axes"]), s["x"].double(), s["q"].double(), True, c["E"],
                          c["phi"])
        return {k: v for k, v in (("E", E), ("phi", phi)) if v is not None}
    if kind == "volumes":
        return [_field64(_mesh64(f["axes"]), f["x"].double(), f["q"].double(), True)[0]
                for f in s["frames"]]
    if kind == "topo":
        # charges inside the box end streamlines in a walk to and fro about them, whose end
        # depends on every rounding
        if c["layout"] != "ball":
            return None
        out = {"feats": _topo64(s, c), "steps": None, "exited": None}
        return dict(out, hist=None) if c["bins"] else out
    allf = np.concatenate(s["feats"])
    edges = [_edges64(allf[:, k], c["rows"]) for k in range(2)]
    hist = np.stack([np.histogram2d(f[:, 0], f[:, 1], bins=edges)[0].ravel() for f in s["feats"]])
    hist = torch.from_numpy(hist / hist.sum(1, keepdims=True)).cuda()
    dist = torch.zeros((len(hist), len(hist)), dtype=torch.float64, device="cuda")
    for i in range(len(hist)):
        t = hist[i] + hist
        dist[i] = 0.5 * ((hist[i] - hist) ** 2 / torch.where(t == 0, 1.0, t)).sum(1)
    return {"hist": hist.cpu().numpy(), "dist": dist.cpu().numpy()}
