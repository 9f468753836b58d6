"""Workloads of this framework: what a localisation, mapping or simulation program
asks of it through the public Python surface, from one lidar scan to whole tables.

``listed()`` names the standing cases, ``draw(rng)`` gives others of the same
ranges.  ``prepare(case, seed)`` makes what the program holds before the call,
``run(state)`` is one pass, ``work(case)`` the bytes and operations it cannot do
without and ``exact(case, seed)`` the same outputs in 64 bits (None where an
output is a step function of rounded values: sensor weights index a table by
truncated ranges, CDDT bins round projections, training iterates in bf16).

Kinds
  scan     a host program casts lidar scans from numpy arrays (a simulator, a ROS node)
  step     a particle filter's update with inputs in HBM: ranges and weights
  queries  independent rays with inputs in HBM (planning, visibility)
  batch    the filters of several robots, each on its own map, in one launch
  map      a new occupancy grid arrives (SLAM): distance transform, then a scan match
  glt      a GiantLUTCast table is built for a map and answers a filter update
  cddt     CDDT tables are built and pruned for a map and answer a filter update
  train    the learned surrogate is fitted to a map for some steps
  infer    the surrogate proposes ranges, which are checked against the map
"""
from __future__ import annotations

import math

import numpy as np
import torch

import range_libc_amd as rl
from range_libc_amd import workloads as W

METHODS = {"rm": rl.RL_METHOD_RM, "bl": rl.RL_METHOD_BL, "cddt": rl.RL_METHOD_CDDT, "glt": rl.RL_METHOD_GLT}
WORLD = (0.05, 0.3, -7.5, 4.25)  # metres per cell, angle, origin of a map recorded in the field


def listed():
    return [
        # one 60-beam scan of one robot from host arrays: the smallest call, all latency
        dict(name="scan_1x60", kind="scan", map="rect_disk", w=512, h=512, n=1, m=60, R=500, world=False, weights=False),
        # the standard particle-filter update: 4000 particles, 60 beams, 2048^2 corridors
        dict(name="step_4000x60", kind="step", method="rm", map="corridor", w=2048, h=2048, n=4000, m=60, R=500,
             td=0, world=False),
        # a large filter of odd sizes on a map that is not square, in a rotated world frame
        dict(name="step_20011x107_world", kind="step", method="rm", map="rect_disk", w=1531, h=1999, n=20011, m=107,
             R=400, td=0, world=True),
        # 100 k independent queries of a 512^2 map
        dict(name="queries_rm_100k", kind="queries", method="rm", map="rect_disk", w=512, h=512, n=100000, R=500,
             world=False),
        # 1 M Bresenham queries with a long range
        dict(name="queries_bl_1m", kind="queries", method="bl", map="corridor", w=2048, h=2048, n=1000000, R=1000,
             world=False),
        # the standard update answered by pruned CDDT tables
        dict(name="step_pcddt_4000x60", kind="step", method="cddt", map="corridor", w=2048, h=2048, n=4000, m=60,
             R=500, td=108, world=False),
        # sixteen maps of uneven sides, particles and beams in one launch
        dict(name="batch_16_maps", kind="batch", maps=16, spec=4, side_max=2048, p_max=8000, b_max=120, R=500),
        # a new 2048^2 grid from the host, and 4096 rays cast in it
        dict(name="map_2048", kind="map", map="corridor", w=2048, h=2048, n=4096, R=500),
        # the whole lookup table of a 2048^2 map, 108 headings
        dict(name="glt_2048x108", kind="glt", map="corridor", w=2048, h=2048, n=4000, m=60, R=500, td=108),
        # CDDT tables of the same map, pruned
        dict(name="cddt_2048x108", kind="cddt", map="corridor", w=2048, h=2048, n=4000, m=60, R=500, td=108),
        # sixteen training steps of the surrogate on 16384 marched rays each
        dict(name="train_16x16384", kind="train", map="corridor", w=2048, h=2048, batch=16384, steps=16, R=500),
        # the standard update's rays proposed by the surrogate and checked
        dict(name="infer_4000x60", kind="infer", map="corridor", w=2048, h=2048, n=4000, m=60, R=500),
    ]


def draw(rng):
    """One more case of these ranges, odd and ragged sizes among them."""
    def size(lo, hi):  # spread over the logarithm
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["scan", "step", "queries", "batch", "map", "glt", "cddt", "train", "infer"])
    world = rng.random() < 0.4
    c = dict(kind=kind)
    if kind == "batch":
        c.update(maps=rng.randint(2, 16), spec=rng.randint(0, 10**6), side_max=size(300, 2048),
                 p_max=size(600, 8000), b_max=rng.randint(31, 120), R=rng.randint(100, 500))
        return c
    c.update(map=rng.choice(["corridor", "rect_disk"]), w=size(200, 2048), h=size(200, 2048), R=rng.randint(40, 500))
    if kind == "scan":
        c.update(n=size(1, 4000), m=rng.randint(9, 120), world=world, weights=rng.random() < 0.5)
    elif kind == "step":
        c.update(method=rng.choice(["rm", "rm", "cddt", "glt", "bl"]), n=size(1, 20000), m=rng.randint(9, 110),
                 td=rng.randint(36, 180), world=world)
        if c["method"] == "glt":  # the table stays within the largest listed one
            c["td"] = min(c["td"], 108)
    elif kind == "queries":
        c.update(method=rng.choice(["rm", "bl"]), n=size(1000, 1000000), R=rng.randint(40, 1000), world=world)
    elif kind == "map":
        c.update(n=size(64, 4096))
    elif kind in ("glt", "cddt"):
        c.update(n=size(100, 4000), m=60, td=rng.randint(36, 108))
    elif kind == "train":
        c.update(batch=size(1000, 16384), steps=rng.randint(4, 16))
    elif kind == "infer":
        c.update(n=size(50, 4000), m=60)
    return c


# --- inputs -------------------------------------------------------------------

_STREAM = None


def _context():
    """The library's context on a torch stream that is current in this program."""
    global _STREAM
    ctx = rl.default_context(0)
    if _STREAM is None:
        _STREAM = torch.cuda.Stream()
        torch.cuda.set_stream(_STREAM)
        ctx.set_stream(_STREAM.cuda_stream)
    return ctx


def _image(case, seed):
    """img[y, x], h x w, cut from a square map of the case's kind."""
    img = W.make_map(case["map"], max(case["w"], case["h"]), 1000 + seed)
    return np.ascontiguousarray(img[: case["h"], : case["w"]])


def _world(case):
    if not case.get("world"):
        return (1.0, 0.0, 0.0, 0.0, 0.0, 1.0)
    scale, angle, ox, oy = WORLD
    return (scale, angle, ox, oy, math.sin(angle), math.cos(angle))


def _poses(case, img, n, seed):
    """n poses in free cells, in the world frame that the case's map is in."""
    ins = W.world_poses(img, n, seed)
    if case.get("world"):
        scale, _, ox, oy, s, c = _world(case)
        u, v = ins[:, 0].astype(np.float64), ins[:, 1].astype(np.float64)
        ins[:, 0] = (c * u + s * v) * scale + ox
        ins[:, 1] = (-s * u + c * v) * scale + oy
    return ins


def _dmap(case, img):
    m = rl.DeviceMap(_context(), np.ascontiguousarray(img.T))
    m.set_world(*_world(case))
    return m


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def _observation(case, m, seed):
    """Ranges a lidar saw: between a few cells and max_range, in world units."""
    r = np.random.default_rng(seed + 77)
    obs = np.minimum(r.gamma(2.0, 25.0, size=m), case["R"])
    return (obs * _world(case)[0]).astype(np.float32)


def _table(case):
    return W.sensor_table(case["R"] + 1)


def _params(seed):
    """Surrogate parameters: He-normal layers, range head around a tenth of max_range, bound head around one cell."""
    r = np.random.default_rng(seed + 5)
    p = []
    for fout, fin in ((256, 64), (256, 256), (256, 256)):
        p += [r.normal(0.0, math.sqrt(2.0 / fin), fout * fin), np.zeros(fout)]
    p += [r.normal(0.0, 0.01, 2 * 256), np.array([0.1, 0.0])]
    freq = r.normal(0.0, 1.0, (32, 4)) * np.array([2.0, 2.0, 1.0, 1.0])
    return np.concatenate(p).astype(np.float32), freq.astype(np.float32)


def _step_state(case, img, seed):
    """Poses, beams, observation and output buffers of a filter update, in HBM."""
    n, m = case["n"], case["m"]
    return {
        "ins": _dev(_poses(case, img, n, seed)), "angles": _dev(W.beam_angles(m)),
        "obs": _dev(_observation(case, m, seed)),
        "ranges": torch.zeros(n * m, dtype=torch.float32, device="cuda"),
        "weights": torch.zeros(n, dtype=torch.float64, device="cuda"),
    }


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "R": float(case["R"])}
    if kind == "batch":
        return _prepare_batch(s, case, seed)
    img = _image(case, seed)
    if kind == "scan":
        omap = rl.PyOMap(img)
        if case["world"]:
            scale, angle, ox, oy, sn, cs = _world(case)
            omap.set_world(scale, angle, ox, oy, sn, cs)
        _context()
        s["rm"] = rl.PyRayMarchingGPU(omap, case["R"])
        s.update(ins=_poses(case, img, case["n"], seed), angles=W.beam_angles(case["m"]),
                 obs=_observation(case, case["m"], seed))
        if case["weights"]:
            s["rm"].set_sensor_model(_table(case))
            s["out"] = np.zeros(case["n"], np.float64)
        else:
            s["out"] = np.zeros(case["n"] * case["m"], np.float32)
        return s
    if kind == "map":
        _context()
        s["occ"] = np.ascontiguousarray(img.T)
        s["ins"] = _dev(W.grid_poses(img, case["n"], seed))
        s["ranges"] = torch.zeros(case["n"], dtype=torch.float32, device="cuda")
        return s
    s["map"] = m = _dmap(case, img)
    if kind in ("step", "glt", "cddt"):
        m.set_sensor_table(_table(case))
        s.update(_step_state(case, img, seed))
        if case.get("method") == "cddt":
            m.build_cddt(case["td"])
            m.prune_cddt(s["R"])
        elif case.get("method") == "glt":
            m.build_giant_lut(s["R"], case["td"])
    elif kind == "queries":
        s["ins"] = _dev(_poses(case, img, case["n"], seed))
        s["ranges"] = torch.zeros(case["n"], dtype=torch.float32, device="cuda")
    else:  # train, infer
        s["net"] = rl.Surrogate(m, seed=seed)
        s["net"].set_params(*_params(seed))
        s["seed"] = seed
        if kind == "infer":
            s.update(_step_state(case, img, seed))
    return s


def _batch_specs(case, seed):
    """Sizes by the case, maps and poses by the seed."""
    specs = W.uneven_batch_specs(case["maps"], case["spec"], side_min=256, side_max=case["side_max"], p_min=500,
                                 p_max=case["p_max"], b_min=30, b_max=case["b_max"])
    return [dict(p, map_seed=p["map_seed"] ^ seed, pose_seed=p["pose_seed"] ^ seed) for p in specs]


def _prepare_batch(s, case, seed):
    ctx = _context()
    specs = _batch_specs(case, seed)
    rays = sum(p["particles"] * p["beams"] for p in specs)
    s["ranges"] = torch.zeros(rays, dtype=torch.float32, device="cuda")
    s["weights"] = torch.zeros(sum(p["particles"] for p in specs), dtype=torch.float64, device="cuda")
    s["keep"], jobs, r0, w0 = [], [], 0, 0
    table = _table(case)
    for p in specs:
        img = W.make_map(p["kind"], p["side"], p["map_seed"])
        m = rl.DeviceMap(ctx, np.ascontiguousarray(img.T))
        m.set_sensor_table(table)
        n, b = p["particles"], p["beams"]
        held = (_dev(W.world_poses(img, n, p["pose_seed"])), _dev(W.beam_angles(b)),
                _dev(_observation(case, b, p["pose_seed"])))
        s["keep"].append((m, held))
        jobs.append(dict(map=m, max_range=s["R"], ins=held[0].data_ptr(), angles=held[1].data_ptr(),
                         obs=held[2].data_ptr(), ranges=s["ranges"][r0:].data_ptr(),
                         weights=s["weights"][w0:].data_ptr(), num_particles=n, num_angles=b))
        r0, w0 = r0 + n * b, w0 + n
    s["batch"] = rl.Batch(ctx, rl.RL_METHOD_RM)
    s["batch"].set_jobs(jobs)
    return s


# --- one pass -----------------------------------------------------------------


class _DeviceArray:
    """A device buffer of a map as torch takes it; a tensor of it keeps the map."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": "<f4", "version": 2}


def _pf_step(s, method):
    c = s["case"]
    s["map"].pf_step_dev(METHODS[method], s["R"], s["ins"].data_ptr(), s["angles"].data_ptr(), s["obs"].data_ptr(),
                         s["ranges"].data_ptr(), s["weights"].data_ptr(), c["n"], c["m"])
    return {"ranges": s["ranges"], "weights": s["weights"]}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "scan":
        if case["weights"]:
            s["rm"].calc_range_repeat_angles_eval_sensor_model(s["ins"], s["angles"], s["obs"], s["out"])
            return {"weights": s["out"]}
        s["rm"].calc_range_repeat_angles(s["ins"], s["angles"], s["out"])
        return {"ranges": s["out"]}
    if kind == "step":
        return _pf_step(s, case["method"])
    if kind == "queries":
        s["map"].numpy_calc_range_dev(METHODS[case["method"]], s["R"], s["ins"].data_ptr(), s["ranges"].data_ptr(),
                                      case["n"])
        return {"ranges": s["ranges"]}
    if kind == "batch":
        s["batch"].launch()
        return {"ranges": s["ranges"], "weights": s["weights"]}
    if kind == "map":
        # the map of the pass before is let go when its successor is there
        s["map"] = m = rl.DeviceMap(_context(), s["occ"])
        m.calc_range_many_dev(rl.RL_METHOD_RM, s["R"], s["ins"].data_ptr(), s["ranges"].data_ptr(), case["n"])
        edt = torch.as_tensor(_DeviceArray(m, m.device_buffers()[0], (case["w"], case["h"])), device="cuda")
        return {"edt": edt, "ranges": s["ranges"]}
    if kind == "glt":
        s["map"].build_giant_lut(s["R"], case["td"])
        return _pf_step(s, "glt")
    if kind == "cddt":
        s["map"].build_cddt(case["td"])
        s["map"].prune_cddt(s["R"])
        return _pf_step(s, "cddt")
    if kind == "train":
        curve = s["net"].train(s["R"], case["batch"] * case["steps"], batch=case["batch"], lr=1e-3, seed=s["seed"])
        return {"loss": curve, "params": s["net"].params()[0]}
    st = s["net"].calc_range_angles_dev(s["R"], s["ins"].data_ptr(), s["angles"].data_ptr(), s["ranges"].data_ptr(),
                                        case["n"], case["m"], bound_max=2.0)
    return {"ranges": s["ranges"], "stats": [st[k] for k in sorted(st)]}


def work(case):
    kind = case["kind"]
    if kind == "batch":  # means of the specs' distributions
        rays = case["maps"] * (500 + case["p_max"]) / 2 * (30 + case["b_max"]) / 2
        side2 = (case["side_max"] ** 2 - 256 ** 2) / max(2 * math.log(case["side_max"] / 256), 1e-3)
        return {"bytes": case["maps"] * side2 + rays * 4, "flops": 0}
    cells = case["w"] * case["h"]
    if kind == "train":
        rays = case["batch"] * case["steps"]
        return {"bytes": min(cells, 8 * rays) + case["steps"] * 148738 * 4 * 6, "flops": 3 * 296960 * rays}
    if kind in ("map", "queries"):
        n = case["n"]
        b = min(cells, 8 * n) + 16 * n
        if kind == "map":
            b += cells * 5
        return {"bytes": b, "flops": 0}
    n, rays = case["n"], case["n"] * case["m"]
    b = 12 * n + 8 * case["m"] + min(cells, 8 * rays)
    if kind == "infer":
        return {"bytes": b + 4 * rays, "flops": 296960 * rays}
    if kind == "scan" and not case["weights"]:
        return {"bytes": b + 4 * rays, "flops": 0}
    b += min(8 * (case["R"] + 1) ** 2, 8 * rays) + 8 * n
    if kind != "scan":
        b += 4 * rays
    if kind == "glt":
        b += cells + 2 * cells * case["td"]
    elif kind == "cddt":  # about one cell in twenty is at a wall's face: an entry for each heading of a half turn
        b += cells + 0.05 * cells * (case["td"] / 2) * 4
    return {"bytes": b, "flops": 0}


# --- the same in 64 bits ---------------------------------------------------------


def _edt64(occ):
    """Euclidean distance to the nearest occupied cell, occ (w, h) bool."""
    w, h = occ.shape
    y = torch.arange(h, dtype=torch.float64, device=occ.device).expand(w, h)
    inf = torch.tensor(math.inf, dtype=torch.float64, device=occ.device)
    before = torch.cummax(torch.where(occ, y, -inf), 1).values
    after = torch.cummin(torch.where(occ, y, inf).flip(1), 1).values.flip(1)
    g = torch.minimum(y - before, after - y) ** 2
    best = g.clone()
    d = 1
    while d < w and d * d < best.max().item():
        best[d:] = torch.minimum(best[d:], g[:-d] + d * d)
        best[:-d] = torch.minimum(best[:-d], g[d:] + d * d)
        d += 1
    return best.sqrt()


def _march64(edt, x0, y0, heading, R):
    """Sphere tracing with steps max(0.999 d, 1) until a cell of distance 0; R past the range or the map."""
    w, h = edt.shape
    dx, dy = heading.cos(), heading.sin()
    out = torch.full_like(x0, R)
    t = torch.zeros_like(x0)
    at = torch.arange(x0.numel(), device=x0.device)
    while at.numel():
        px, py = (x0[at] + dx[at] * t[at]).trunc(), (y0[at] + dy[at] * t[at]).trunc()
        go = (t[at] < R) & (px >= 0) & (px < w) & (py >= 0) & (py < h)
        at, px, py = at[go], px[go], py[go]
        d = edt[px.long(), py.long()]
        hit = d <= 0
        out[at[hit]] = torch.sqrt((px[hit] - x0[at[hit]]) ** 2 + (py[hit] - y0[at[hit]]) ** 2)
        at, d = at[~hit], d[~hit]
        t[at] += (d * 0.999).clamp(min=1.0)
    return out


def _bresenham64(occ, x, y, heading, R):
    """The error-accumulating walk from (y, x) in rows, steps of one cell along the longer axis."""
    w, h = occ.shape
    x0, y0 = y, x
    x1, y1 = y + R * heading.sin(), x + R * heading.cos()
    steep = (y1 - y0).abs() > (x1 - x0).abs()
    x0, y0, x1, y1 = (torch.where(steep, a, b) for a, b in ((y0, x0), (x0, y0), (y1, x1), (x1, y1)))
    dx, dy = (x1 - x0).abs(), (y1 - y0).abs()
    sx = torch.where(x0 < x1, 1.0, -1.0).double()
    sy = torch.where(y0 < y1, 1.0, -1.0).double()
    end = (x1 + sx).trunc()
    px, py, err = x0.clone(), y0.clone(), torch.zeros_like(x0)
    out = torch.full_like(x0, float(R))
    at = torch.arange(x0.numel(), device=x0.device)

    def cell(u, v, st):
        gx, gy = torch.where(st, u, v), torch.where(st, v, u)
        inside = (gx >= 0) & (gx < w) & (gy >= 0) & (gy < h)
        return inside & occ[gx.clamp(0, w - 1).long(), gy.clamp(0, h - 1).long()]

    start = cell(x0, y0, steep)
    out[start] = 0.0
    at = at[~start]
    at = at[px[at].trunc() != end[at]]
    while at.numel():
        u = px[at] + sx[at]
        e = err[at] + dy[at]
        adv = e * 2.0 >= dx[at]
        v = torch.where(adv, py[at] + sy[at], py[at])
        px[at], py[at], err[at] = u, v, torch.where(adv, e - dx[at], e)
        hit = cell(u, v, steep[at])
        k = at[hit]
        out[k] = torch.sqrt((px[k] - x0[k]) ** 2 + (py[k] - y0[k]) ** 2)
        at = at[~hit & (u.trunc() != end[at])]
    return out


def _rays64(case, ins, angles=None):
    """Grid-frame origins and headings of world-frame poses (and beams), flattened particle by particle."""
    scale, angle, ox, oy, sn, cs = (float(np.float32(v)) for v in _world(case))
    p = torch.from_numpy(ins.astype(np.float64)).to("cuda")
    x, y = (p[:, 0] - ox) / scale, (p[:, 1] - oy) / scale
    gx, gy = cs * x - sn * y, sn * x + cs * y
    h = -p[:, 2] - angle - 1.5 * math.pi
    if angles is not None:
        a = torch.from_numpy(angles.astype(np.float64)).to("cuda")
        h = (h[:, None] - a[None, :]).reshape(-1)
        gx, gy = (v[:, None].expand(-1, a.numel()).reshape(-1) for v in (gx, gy))
    return gy, gx, h, scale


def _glt64(edt, x, y, heading, R, td):
    """The march from the cell's corner along the nearest of td headings, in 65535ths of R."""
    b = torch.remainder(torch.round(torch.remainder(heading, 2 * math.pi) * td / (2 * math.pi)), td)
    r = _march64(edt, x.trunc(), y.trunc(), b * (2 * math.pi / td), float(R)).clamp(max=R)
    return (r * (65535.0 / R)).trunc() * (R / 65535.0)


def _batch64(case, seed):
    out = []
    for p in _batch_specs(case, seed):
        img = W.make_map(p["kind"], p["side"], p["map_seed"])
        edt = _edt64(torch.from_numpy(np.ascontiguousarray(img.T) != 0).to("cuda"))
        ins = W.world_poses(img, p["particles"], p["pose_seed"])
        x, y, h, _ = _rays64({}, ins, W.beam_angles(p["beams"]))
        out.append(_march64(edt, x, y, h, float(case["R"])))
    return torch.cat(out)


def exact(case, seed):
    kind = case["kind"]
    method = case.get("method", "glt" if kind == "glt" else "rm")
    if kind == "batch":
        return {"ranges": _batch64(case, seed), "weights": None}
    if kind in ("cddt", "train") or method == "cddt" or (kind == "scan" and case["weights"]):
        return None
    img = _image(case, seed)
    occ = torch.from_numpy(np.ascontiguousarray(img.T) != 0).to("cuda")
    R = float(case["R"])
    if kind == "map":
        edt = _edt64(occ)
        p = torch.from_numpy(W.grid_poses(img, case["n"], seed).astype(np.float64)).to("cuda")
        return {"edt": edt, "ranges": _march64(edt, p[:, 0].contiguous(), p[:, 1].contiguous(), p[:, 2], R)}
    angles = None if kind == "queries" else W.beam_angles(case["m"])
    x, y, h, scale = _rays64(case, _poses(case, img, case["n"], seed), angles)
    if method == "bl":
        r = _bresenham64(occ, x, y, h, R)
    elif method == "glt":
        r = _glt64(_edt64(occ), x, y, h, R, case["td"])
    else:
        r = _march64(_edt64(occ), x, y, h, R)
    r = r * scale
    if kind in ("scan", "queries"):
        return {"ranges": r}
    return {"ranges": r, "stats" if kind == "infer" else "weights": None}
