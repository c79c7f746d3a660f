"""Performance cases: the work programs have the engines do, through the public
entry points of include/pattern.h and its Python mirror.

Families (the "kind" of a case):
  heat       the tuned heat3D engine: a field on the device advanced `steps`
             sweeps by a Stencil handle
  app        an application's own stencil functor, compiled through the
             functor-table templates, on the handle's generic sweep
  moldyn     velocity-Verlet LJ dynamics over a fixed half pair list
  minimd     the same with the neighbour list rebuilt on the device
  csr        the inspector: a half edge list reordered into rows by node
  kmeans     Lloyd iterations on points resident in device memory
  keyed      a generalized reduction with an application's own map / reduce
             functors and a keyed reduction object
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "ipdps15-pattern_amd"))
import pattern_amd as pa  # noqa: E402

ALPHA = 0.1
RHO = 0.8442
RC, SKIN, EVERY, DT = 2.5, 0.3, 20, 0.005
HIST_KEYS = 5003  # apps/regular/regular.h
KMEANS3_K = 40
CSR_PAIRS = 26  # per atom: a random part of the about 27 within the cutoff, so that every seed has as many


def listed():
    return [
        # a small field, as in a stream of small jobs: launches and latencies
        {"name": "heat_64", "kind": "heat", "nx": 64, "ny": 64, "nz": 64, "steps": 100},
        # the heat3D workload at its two benchmark sizes
        {"name": "heat_128", "kind": "heat", "nx": 128, "ny": 128, "nz": 128, "steps": 100},
        {"name": "heat_384", "kind": "heat", "nx": 384, "ny": 384, "nz": 384, "steps": 100},
        # a user's own functor (the W = 3 star) on a ragged field
        {"name": "star_200", "kind": "app", "functor": "star", "nx": 200, "ny": 186, "nz": 210, "steps": 20},
        # the moldyn benchmark: 256,000 molecules, 6.9 M pairs, 50 steps
        {"name": "moldyn_40", "kind": "moldyn", "cells": 40, "steps": 50},
        # miniMD: 1 M atoms, two rebuilds in 40 steps
        {"name": "minimd_64", "kind": "minimd", "cells": 64, "steps": 40},
        # set-up of a new edge list (an irregular runtime's initialisation)
        {"name": "csr_40", "kind": "csr", "cells": 40, "order": "node"},
        # a small clustering, a few launches' worth of work
        {"name": "kmeans_20k_8", "kind": "kmeans", "n": 20000, "d": 8, "k": 16, "iters": 10},
        # the kmeans benchmark (5 of its iterations)
        {"name": "kmeans_16m_32", "kind": "kmeans", "n": 1 << 24, "d": 32, "k": 256, "iters": 5},
        # many wide centres: the largest jobs of the serving mix
        {"name": "kmeans_1m_128", "kind": "kmeans", "n": 1 << 20, "d": 128, "k": 1000, "iters": 10},
        # kmeans' map1 at the reference's sizes as a user's functor: 40 keys
        {"name": "keyed_kmeans3", "kind": "keyed", "functor": "kmeans3", "n": 1000000},
        # a user's histogram of 5,003 keys, more than an LDS object holds
        {"name": "keyed_hist", "kind": "keyed", "functor": "hist", "n": 500000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["heat", "heat", "app", "moldyn", "minimd", "csr", "kmeans", "kmeans", "keyed"])
    if kind == "heat":
        side = _log(rng, 32, 360)
        n = [max(16, min(384, int(side * rng.uniform(0.8, 1.25)))) for _ in range(3)]
        return {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "steps": rng.choice([50, 75, 99, 100])}
    if kind == "app":
        side = _log(rng, 32, 220)
        n = [max(16, int(side * rng.uniform(0.8, 1.25))) for _ in range(3)]
        return {"kind": kind, "functor": rng.choice(["star", "heat", "heat_ref"]), "nx": n[0], "ny": n[1], "nz": n[2],
                "steps": rng.randrange(5, 21)}
    if kind == "moldyn":
        return {"kind": kind, "cells": _log(rng, 8, 40), "steps": rng.randrange(20, 51)}
    if kind == "minimd":
        return {"kind": kind, "cells": _log(rng, 8, 56), "steps": rng.randrange(20, 61)}
    if kind == "csr":
        return {"kind": kind, "cells": _log(rng, 8, 40), "order": rng.choice(["edge", "node"])}
    if kind == "kmeans":
        d = rng.choice([8, 16, 32, 64, 128])
        k = _log(rng, 16, 1024)
        n = min(_log(rng, 10000, 4000000), (1 << 34) // (d * k) * 8)
        return {"kind": kind, "n": n, "d": d, "k": k, "iters": rng.randrange(5, 11)}
    return {"kind": kind, "functor": rng.choice(["kmeans3", "hist"]), "n": _log(rng, 20000, 1000000)}


# ------------------------------------------------------------------ inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _width(case):
    return 3 if case.get("functor") == "star" else 1


def _field(case, seed):
    """Interior uniform in [0, 1), zero halo; (z, y, x)."""
    w = _width(case)
    dt = torch.float64 if case.get("functor") == "heat_ref" else torch.float32
    u = torch.zeros((case["nz"] + 2 * w, case["ny"] + 2 * w, case["nx"] + 2 * w), dtype=dt, device="cuda")
    u[w:-w, w:-w, w:-w] = torch.rand((case["nz"], case["ny"], case["nx"]), generator=_gen(seed), dtype=dt,
                                     device="cuda")
    return u


def _lattice(case, seed):
    """FCC atoms of a cubic box: jittered and at rest for moldyn's fixed list,
    on the lattice with Maxwell velocities for miniMD."""
    c = case["cells"]
    if case["kind"] == "minimd":
        pos, box = pa.gen_fcc(c, c, c, RHO, 0.0, seed)
        return pos, pa.gen_velocities(len(pos), 1.44, seed), float(box[0])
    pos, box = pa.gen_fcc(c, c, c, RHO, 0.05, seed)
    return pos, None, float(box[0])


def _points(case, seed):
    """A Gaussian mixture of k components (sigma 1, centres in [-10, 10]^d)."""
    n, d, k = case["n"], case["d"], case["k"]
    g = _gen(seed)
    centres = torch.rand((k, d), generator=g, device="cuda") * 20 - 10
    x = torch.randn((n, d), generator=g, device="cuda")
    x += centres[torch.randint(0, k, (n,), generator=g, device="cuda")]
    return x


def _units(case, seed):
    """(units, functor parameter) of a keyed reduction, host arrays."""
    rng = np.random.default_rng(seed)
    if case["functor"] == "hist":
        return rng.integers(0, 1 << 31, case["n"], dtype=np.uint32), None
    centres = rng.uniform(-10, 10, (KMEANS3_K, 3)).astype(np.float32)
    x = rng.standard_normal((case["n"], 3)).astype(np.float32)
    x += centres[rng.integers(0, KMEANS3_K, case["n"])]
    return x, x[:KMEANS3_K].copy()


# ------------------------------------------------------------------ state

class _View:
    """A device buffer of a handle as torch reads it (no copy).  The tensor
    holds this object, and so the handle that owns the memory."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (int(ptr), False),
                                         "version": 2}


def _view(owner, ptr, shape, typestr="<f4"):
    return torch.as_tensor(_View(owner, ptr, shape, typestr), device="cuda")


def prepare(case, seed):
    pa.init(0)
    kind = case["kind"]
    s = {"case": case}
    if kind in ("heat", "app"):
        u = _field(case, seed)
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        if kind == "heat":
            h = pa.Stencil(nx, ny, nz, alpha=ALPHA)
        elif case["functor"] == "star":
            h = pa.Stencil(nx, ny, nz, width=3, table=pa.app_table("stencil2"), idx=0)
        elif case["functor"] == "heat":
            h = pa.Stencil(nx, ny, nz, alpha=ALPHA, table=pa.app_table("heat3d"), idx=0)
            h.set_variant(pa.PAT_STENCIL_GENERIC)
        else:
            h = pa.Stencil(nx, ny, nz, dtype=np.float64, param=np.zeros(5), table=pa.app_table("heat3d"), idx=1)
        h.upload(u.cpu().numpy())
        torch.cuda.synchronize()
        s.update(h=h, start=u)
    elif kind in ("moldyn", "minimd"):
        pos, vel, box = _lattice(case, seed)
        if kind == "moldyn":
            edges = pa.gen_pairs(pos, box, RC, shuffle=True, seed=seed + 1)
            h = pa.MD(pos, vel, edges, box, RC, DT)
        else:
            h = pa.MD(pos, vel, None, box, RC, DT, skin=SKIN, every=EVERY)
        s.update(h=h)
    elif kind == "csr":
        pos, _, box = _lattice(case, seed)
        n = len(pos)
        edges = pa.gen_pairs(pos, box, RC, shuffle=True, seed=seed + 1)[:CSR_PAIRS * n].copy()
        e = len(edges)
        wb = pa.c_i64(0)
        pa.call("pat_ir_csr_workspace", n, e, pa.ctypes.byref(wb))
        s.update(n=n, e=e, wb=wb.value, edges=torch.from_numpy(edges).cuda(),
                 work=torch.empty(wb.value, dtype=torch.uint8, device="cuda"),
                 rowptr=torch.empty(n + 1, dtype=torch.int32, device="cuda"),
                 cols=torch.empty(2 * e, dtype=torch.int32, device="cuda"),
                 order=pa.PAT_IR_ORDER_NODE if case["order"] == "node" else pa.PAT_IR_ORDER_EDGE)
    elif kind == "kmeans":
        x = _points(case, seed)
        torch.cuda.synchronize()
        xd = pa.DeviceArray((case["n"], case["d"]), np.float32)
        pa.call("pat_memcpy_d2d", xd.ptr, x.data_ptr(), xd.nbytes, None)
        pa.sync()
        h = pa.KMeans(xd, case["k"])
        s.update(h=h, c0=h.centroids())
    else:
        units, param = _units(case, seed)
        h = pa.Regular(units, len(units), units.itemsize * (1 if units.ndim == 1 else units.shape[1]),
                       table=pa.app_table("regular", "gr"))
        m = 3 if case["functor"] == "hist" else 1
        if case["functor"] == "hist":
            h.set_capacity(8192, 32)
        pa.call("pat_regular_set_map_idx", h.h, m)
        pa.call("pat_regular_set_reduce_idx", h.h, m)
        if param is not None:
            pa.call("pat_regular_set_param", h.h, pa.ptr(param), param.nbytes)
        s.update(h=h)
    return s


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind in ("heat", "app"):
        # a new field of the same shape, already on the device, advanced
        h, p = s["h"], pa.c_vp()
        pa.call("pat_stencil_device_ptr", h.h, pa.ctypes.byref(p))
        pa.call("pat_memcpy_d2d", p, s["start"].data_ptr(), s["start"].numel() * s["start"].element_size(), None)
        pa.sync()
        h.run(case["steps"])
        pa.call("pat_stencil_device_ptr", h.h, pa.ctypes.byref(p))
        return _view(h, p.value, h.shape, "<f8" if h.dtype == np.float64 else "<f4")
    if kind in ("moldyn", "minimd"):
        h = s["h"]
        h.run(case["steps"])
        b = [pa.c_vp() for _ in range(3)]
        pa.call("pat_md_device_buffers", h.h, *[pa.ctypes.byref(x) for x in b])
        return {name: _view(h, x.value, (h.n, 4))[:, :3] for name, x in zip(("pos", "vel", "force"), b)}
    if kind == "csr":
        pa.call("pat_ir_csr_build_dev", s["edges"].data_ptr(), s["e"], s["n"], s["order"], s["rowptr"].data_ptr(),
                s["cols"].data_ptr(), s["work"].data_ptr(), s["wb"], None)
        return s["rowptr"], s["cols"]
    if kind == "kmeans":
        h = s["h"]
        h.set_centroids(s["c0"])
        h.run(case["iters"])
        sums, counts, dsums, shift, dshift = h.get_object()
        return {"centroids": h.centroids(), "sums": sums, "counts": counts, "dsums": dsums,
                "shifts": np.array([shift, dshift], np.int64)}
    h = s["h"]
    pa.call("pat_regular_start", h.h)
    nk, kb, vb = pa.c_i64(0), pa.c_i64(0), pa.c_i64(0)
    ref = pa.ctypes.byref
    pa.call("pat_regular_get_output", h.h, ref(nk), ref(kb), ref(vb), None, None, None, None, None, None)
    keys, vals = np.empty(kb.value, np.uint8), np.empty(vb.value, np.uint8)
    ki, ks, vi, vs = (np.empty(nk.value, np.uint32) for _ in range(4))
    pa.call("pat_regular_get_output", h.h, ref(nk), ref(kb), ref(vb), pa.ptr(keys), pa.ptr(ki), pa.ptr(ks),
            pa.ptr(vals), pa.ptr(vi), pa.ptr(vs))
    keys = keys.view(np.uint32).astype(np.int64)
    if case["functor"] == "hist":
        v = vals.reshape(-1, 16)
        return {"keys": keys, "counts": np.ascontiguousarray(v[:, :8]).view(np.int64)[:, 0],
                "sums": np.ascontiguousarray(v[:, 8:]).view(np.float64)[:, 0]}
    v = vals.view(np.float32).reshape(-1, 5)
    return {"keys": keys, "counts": v[:, 3].astype(np.int64), "sums": np.ascontiguousarray(v[:, [0, 1, 2, 4]])}


# ------------------------------------------------------------------ what a pass cannot do without

def _pairs_per_atom(r):
    return RHO * 4.0 / 3.0 * math.pi * r ** 3 / 2


def work(case):
    kind = case["kind"]
    if kind in ("heat", "app"):
        unit = 8 if case.get("functor") == "heat_ref" else 4
        cells = case["nx"] * case["ny"] * case["nz"]
        ops = {"heat": 9, "star": 13, "heat_ref": 14}[case.get("functor", "heat")]
        return {"bytes": 2 * unit * cells, "flops": ops * cells * case["steps"]}
    if kind in ("moldyn", "minimd"):
        n = 4 * case["cells"] ** 3
        pairs = n * _pairs_per_atom(RC)
        listed_pairs = pairs if kind == "moldyn" else 0  # miniMD's list is made from the positions
        return {"bytes": 8 * listed_pairs + (24 + 36) * n, "flops": case["steps"] * (27 * pairs + 12 * n)}
    if kind == "csr":
        n = 4 * case["cells"] ** 3
        return {"bytes": 16 * n * CSR_PAIRS + 4 * n, "flops": 0}
    if kind == "kmeans":
        n, d, k = case["n"], case["d"], case["k"]
        return {"bytes": case["iters"] * 4 * (n * d + k * d) + 8 * k * (d + 2),
                "flops": case["iters"] * n * (2 * k * d + 2 * d)}
    if case["functor"] == "hist":
        return {"bytes": 4 * case["n"] + 20 * HIST_KEYS, "flops": 3 * case["n"]}
    return {"bytes": 12 * case["n"] + 24 * KMEANS3_K, "flops": case["n"] * (KMEANS3_K * 9 + 5)}


def tolerance(case):
    """Bits, where the entry points promise them: the sweeps, the in-order
    forces (the serial scatter over the list), rows of a CSR and the
    fixed-point object of kmeans.  A keyed object's floating sums may be
    folded in another order."""
    if case["kind"] != "keyed":
        return "exact"
    if case["functor"] == "hist":  # FP64 sums of up to a few hundred values a key
        return {"rel": 2e-15, "max": 2e-14}
    return {"rel": 1e-6, "max": 4e-5}  # FP32 sums of up to 25,000 values a key


# ------------------------------------------------------------------ the same in 64 bits

def _exact_stencil(case, seed):
    w = _width(case)
    u = _field(case, seed).double()

    def at(dz, dy, dx):
        n = u.shape
        return u[w + dz:n[0] - w + dz, w + dy:n[1] - w + dy, w + dx:n[2] - w + dx]

    faces = [(0, 0, -1), (0, 0, 1), (0, -1, 0), (0, 1, 0), (-1, 0, 0), (1, 0, 0)]
    for _ in range(case["steps"]):
        c = at(0, 0, 0)
        if case.get("functor") == "star":
            v = sum(at(m * z, m * y, m * x) for z, y, x in faces for m in (1, 2)) / 36
        elif case.get("functor") == "heat_ref":
            v = 0.234 * (sum(at(*f) for f in faces) + 3 * 0.234 * c)
        else:
            v = c + ALPHA * (sum(at(*f) for f in faces) - 6 * c)
        u[w:-w, w:-w, w:-w] = v
    return u


def _pairs(x, box, cut):
    """All pairs i < j within cut under the minimum image, by cells."""
    n = x.shape[0]
    nc = int(box // cut)
    if nc < 4:
        i, j = torch.triu_indices(n, n, 1, device=x.device)
        d = x[i] - x[j]
        d -= box * torch.round(d / box)
        near = (d * d).sum(1) < cut * cut
        return i[near], j[near]
    cell = (x * (nc / box)).long().clamp(0, nc - 1)
    cid = (cell[:, 2] * nc + cell[:, 1]) * nc + cell[:, 0]
    order = torch.argsort(cid)
    count = torch.bincount(cid, minlength=nc ** 3)
    first = torch.cumsum(count, 0) - count
    slots = torch.full((nc ** 3, int(count.max())), -1, dtype=torch.int64, device=x.device)
    slots[cid[order], torch.arange(n, device=x.device) - first[cid[order]]] = order
    grid = torch.arange(nc ** 3, device=x.device).reshape(nc, nc, nc)
    got = []
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                other = slots[torch.roll(grid, (dz, dy, dx), (0, 1, 2)).reshape(-1)]
                a, b = torch.broadcast_tensors(slots[:, :, None], other[:, None, :])
                keep = (a >= 0) & (a < b)
                i, j = a[keep], b[keep]
                d = x[i] - x[j]
                d -= box * torch.round(d / box)
                near = (d * d).sum(1) < cut * cut
                got.append((i[near], j[near]))
    return torch.cat([g[0] for g in got]), torch.cat([g[1] for g in got])


def _exact_md(case, seed):
    pos, vel, box = _lattice(case, seed)
    x = torch.from_numpy(pos).cuda().double()
    v = torch.zeros_like(x) if vel is None else torch.from_numpy(vel).cuda().double()

    def force(i, j):
        d = x[i] - x[j]
        d -= box * torch.round(d / box)
        r2 = (d * d).sum(1)
        q = torch.where(r2 < RC * RC, 1.0 / r2, torch.zeros_like(r2))
        q3 = q * q * q
        d *= (48.0 * (q3 - 0.5) * q3 * q)[:, None]
        f = torch.zeros_like(x)
        f.index_add_(0, i, d)
        f.index_add_(0, j, -d)
        return f

    cut = RC if case["kind"] == "moldyn" else RC + SKIN
    i, j = _pairs(x, box, cut)
    f = force(i, j)
    for k in range(1, case["steps"] + 1):
        v += 0.5 * DT * f
        x += DT * v
        x = torch.where(x < 0, x + box, torch.where(x >= box, x - box, x))
        if case["kind"] == "minimd" and k % EVERY == 0:
            i, j = _pairs(x, box, cut)
        f = force(i, j)
        v += 0.5 * DT * f
    return {"pos": x, "vel": v, "force": f}


def _exact_kmeans(case, seed):
    x = _points(case, seed)
    k, d = case["k"], case["d"]
    c = x[:k].double()
    rows = max(1, (1 << 28) // (k + d))
    for _ in range(case["iters"]):
        sums, count = torch.zeros_like(c), torch.zeros(k, dtype=torch.float64, device="cuda")
        for part in torch.split(x, rows):
            p = part.double()
            near = ((c * c).sum(1) - 2 * (p @ c.t().contiguous())).argmin(1)
            sums.index_add_(0, near, p)
            count += torch.bincount(near, minlength=k)
        c = torch.where(count[:, None] > 0, sums / count.clamp(min=1)[:, None], c)
    return {"centroids": c, "sums": None, "counts": None, "dsums": None, "shifts": None}


def _exact_keyed(case, seed):
    units, param = _units(case, seed)
    if case["functor"] == "hist":
        key, value, n = (units % HIST_KEYS).astype(np.int64), units.astype(np.float64)[:, None] / 1000.0, HIST_KEYS
    else:
        d2 = ((units[:, None, :].astype(np.float64) - param[None]) ** 2).sum(2)
        key, n = d2.argmin(1), KMEANS3_K
        value = np.concatenate([units.astype(np.float64), np.sqrt(d2.min(1))[:, None]], 1)
    sums = np.stack([np.bincount(key, weights=value[:, c], minlength=n) for c in range(value.shape[1])], 1)
    sums = sums[np.bincount(key, minlength=n) > 0]
    # records come out by the keys' bytes
    keys = np.flatnonzero(np.bincount(key, minlength=n)).astype(np.uint32)
    at = sorted(range(len(keys)), key=lambda i: keys[i].tobytes())
    sums = np.ascontiguousarray(sums[at])
    return {"keys": None, "counts": None, "sums": sums[:, 0] if case["functor"] == "hist" else sums}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("heat", "app"):
        return _exact_stencil(case, seed)
    if kind in ("moldyn", "minimd"):
        return _exact_md(case, seed)
    if kind == "kmeans":
        return _exact_kmeans(case, seed)
    if kind == "keyed":
        return _exact_keyed(case, seed)
    return None  # whole numbers
