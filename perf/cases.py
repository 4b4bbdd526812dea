"""The work whose speed is measured: halopot's paths as a halo finder calls them.

Paths (a case's "path"):
  drop_in    compute_potential + compute_kinetic_energy on one halo's host
             records, as the halo finder's own loop over halos calls them
  host       bound_pass_host: a batch of calls from host buffers and back
  bound      Plan.run: potential and bound pass of a batch on device records,
             into which the pristine records are copied first (the pass
             reorders them in place, and a program fills them anew each time)
  potential  Plan.potential, the eager driver, with the caller's arithmetic
  props      Plan.props on the results of a bound pass
  gather     gather_calls: a batch's records from the particle copies
  subfof     find_subfofs: the phase-space sub-FOF step of FOF groups (in
             place, so the groups' particles are copied in first)

Sizes are those of halopot.catalog's configurations, of the tests' batches
and of bench.py's legs.  The number of records of a case follows from its
fields alone; positions and velocities come from the seed (NFW haloes with
Jeans velocities, made on the GPU).
"""
import math
import pathlib
import sys

import numpy as np
import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parent.parent / "mpi-rockstar_amd"))

import halopot  # noqa: E402
from halopot import catalog  # noqa: E402

DEV = "cuda"
ACC = {"compensated": halopot.ACC_COMPENSATED, "naive": halopot.ACC_NAIVE, "f64": halopot.ACC_F64}
CATALOGUE_MASS = catalog.CRITICAL_DENSITY * 250.0 ** 3 * 0.27 / 16_777_216


def listed():
    return [
        # the most common call of the reference's loop: a halo of the one-GPU
        # catalogue's mean size, from host memory (latency)
        {"name": "drop_in_134", "path": "drop_in", "records": 134, "mass": CATALOGUE_MASS},
        # one well resolved halo with background from host memory
        {"name": "drop_in_11000", "path": "drop_in", "records": 11_000, "mass": 1e9},
        # a work unit of a small region: a few dozen calls, half of them
        # sub-haloes, some with their host as potential-only records
        {"name": "bound_48_calls", "path": "bound", "calls": 48, "lo": 5, "hi": 4_000,
         "records": 6_007, "contam": 0.05, "potential_only": 0.1, "mass": 1e9,
         "acc": "compensated", "deep": 0},
        # a region's batch: 2,000 calls with unbound contaminants
        {"name": "bound_2000_calls", "path": "bound", "calls": 2_000, "lo": 20, "hi": 200_000,
         "records": 530_001, "contam": 0.05, "potential_only": 0.0, "mass": 1e9,
         "acc": "compensated", "deep": 0},
        # the whole one-GPU catalogue
        {"name": "bound_catalogue", "path": "bound", "calls": 50_000, "lo": 20, "hi": 500_000,
         "records": 6_710_886, "contam": 0.0, "potential_only": 0.0, "mass": CATALOGUE_MASS,
         "acc": "compensated", "deep": 0},
        # one 2M-particle host with 30 embedded sub-haloes: a deep tree
        {"name": "bound_deep_host", "path": "bound", "calls": 31, "lo": 200, "hi": 2_000_000,
         "records": 2_390_017, "contam": 0.0, "potential_only": 0.0, "mass": 4.2e8,
         "acc": "compensated", "deep": 1},
        # potentials alone in FP64, as the precision sweep takes them
        {"name": "potential_f64", "path": "potential", "calls": 500, "lo": 20, "hi": 100_000,
         "records": 150_011, "contam": 0.05, "potential_only": 0.0, "mass": 1e9, "acc": "f64",
         "deep": 0},
        # halo properties, shapes and fits of the whole catalogue
        {"name": "props_catalogue", "path": "props", "calls": 50_000, "lo": 20, "hi": 500_000,
         "records": 6_710_886, "contam": 0.0, "potential_only": 0.0, "mass": CATALOGUE_MASS,
         "acc": "compensated", "deep": 0},
        # record assembly of 4,000 FOF groups with sub-haloes to depth 3
        {"name": "gather_4000_groups", "path": "gather", "groups": 4_000, "lo": 200, "hi": 50_000,
         "subs": 1.5, "mass": 1e9},
        # the sub-FOF step of those groups, and of one group on its own
        {"name": "subfof_4000_groups", "path": "subfof", "groups": 4_000, "lo": 200, "hi": 50_000,
         "subs": 1.5, "mass": 1e9},
        {"name": "subfof_one_group", "path": "subfof", "groups": 1, "lo": 5_003, "hi": 5_003,
         "subs": 3.0, "mass": 1e9},
        # a region's batch from host buffers, planned, copied in and out
        {"name": "host_2000_calls", "path": "host", "calls": 2_000, "lo": 20, "hi": 200_000,
         "records": 530_001, "contam": 0.05, "potential_only": 0.0, "mass": 1e9,
         "acc": "compensated", "deep": 0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["drop_in", "bound", "bound", "potential", "props", "gather", "subfof",
                       "subfof", "host"])
    mass = math.exp(rng.uniform(math.log(4e8), math.log(7e10)))
    if path == "drop_in":
        return {"path": path, "records": _log_int(rng, 20, 60_000), "mass": mass}
    if path in ("gather", "subfof"):
        lo = _log_int(rng, 100, 2_000)
        return {"path": path, "groups": _log_int(rng, 1, 3_000), "lo": lo,
                "hi": _log_int(rng, 2 * lo, 50_000), "subs": round(rng.uniform(0.5, 2.5), 3),
                "mass": mass}
    calls = _log_int(rng, 3, 2_000 if path == "host" else 20_000)
    lo = rng.choice([5, 20, 20, 50])
    hi = _log_int(rng, 2_000, 500_000)
    per = math.exp(rng.uniform(math.log(3.0 * lo), math.log(max(4.0 * lo, 0.2 * hi))))
    top = 500_000 if path in ("host", "potential") else 4_000_000
    return {"path": path, "calls": calls, "lo": lo, "hi": hi,
            "records": min(int(calls * per) + rng.randrange(64), top) | 1,
            "contam": rng.choice([0.0, 0.05]), "potential_only": rng.choice([0.0, 0.0, 0.1]),
            "mass": mass, "acc": rng.choice(["compensated", "compensated", "naive", "f64"])
            if path in ("bound", "potential") else "compensated", "deep": 0}


# ------------------------------------------------------------------ inputs

def _params(case):
    return catalog.Params(particle_mass=case["mass"])


def _shape_rng(*sizes):
    """Counts and hierarchies depend on a case's sizes only, so that every
    seed's inputs are the same amount of work."""
    return np.random.Generator(np.random.Philox(int(sum(int(s) * 7919 ** k
                                                        for k, s in enumerate(sizes))) % 2 ** 62))


def _scaled(raw, total, lo):
    """Counts of at least lo in the proportions of raw, `total` together (or
    lo each, where that is more)."""
    a, b = 0.0, 1.0
    count = lambda s: np.maximum(lo, np.floor(raw * s)).astype(np.int64)  # noqa: E731
    while count(b).sum() <= total and b < 1e12:
        b *= 2.0
    for _ in range(100):
        m = 0.5 * (a + b)
        a, b = (m, b) if count(m).sum() <= total else (a, m)
    n = count(a)
    n[int(np.argmax(n))] += max(0, total - int(n.sum()))
    return n


def _call_counts(case):
    """Per call: halo particles, contaminants, potential-only records."""
    rng = _shape_rng(case["calls"], case["lo"], case["hi"], case["records"])
    if case["deep"]:  # a host call that holds its sub-haloes' particles too
        k = case["calls"] - 1
        host = case["records"] / (1.0 + 2.0 * 2.15e-3 * k)
        sub = np.maximum(20, host * np.exp(rng.uniform(math.log(1e-4), math.log(1e-2), k)))
        n = np.concatenate([[0], sub.astype(np.int64)])
        n[0] = case["records"] - int(n.sum())
    else:
        raw = catalog.power_law_counts(rng, case["calls"], case["lo"], case["hi"])
        n = _scaled(raw.astype(np.float64), case["records"], case["lo"])
    nc = np.round(case["contam"] * n).astype(np.int64)
    npot = np.round(case["potential_only"] * n * (rng.uniform(size=n.shape) < 0.5)).astype(np.int64)
    keep = np.maximum(n - nc - npot, 1)
    return keep, nc, npot


_TABLES = None


def _tables():
    """Inverse enclosed mass and Jeans dispersion of an NFW halo, on the GPU."""
    global _TABLES
    if _TABLES is None:
        x = np.exp(np.linspace(math.log(1e-5), math.log(1e3), 32768))
        _TABLES = tuple(torch.from_numpy(v).to(DEV) for v in
                        (catalog.nfw_m(x), x, np.sqrt(catalog.jeans_sigma2(x))))
    return _TABLES


def _interp(v, xs, ys):
    k = torch.searchsorted(xs, v).clamp(1, xs.shape[0] - 1)
    t = (v - xs[k - 1]) / (xs[k] - xs[k - 1])
    return ys[k - 1] + t * (ys[k] - ys[k - 1])


def _unit(n, gen):
    u = torch.rand(n, generator=gen, device=DEV, dtype=torch.float64) * 2 - 1
    phi = torch.rand(n, generator=gen, device=DEV, dtype=torch.float64) * (2 * math.pi)
    s = torch.sqrt(1 - u * u)
    return torch.stack([s * torch.cos(phi), s * torch.sin(phi), u], 1)


def _nfw(call, conc, rvir, mvir, cen, bulk, gen):
    """One particle per entry of `call` (its halo): positions, velocities."""
    m, x, sig = _tables()
    c = conc[call]
    mc = torch.log1p(c) - c / (1 + c)
    u = torch.rand(call.shape[0], generator=gen, device=DEV, dtype=torch.float64)
    xi = _interp(u * mc, m, x)
    rs = rvir[call] / c
    pos = cen[call] + (xi * rs)[:, None] * _unit(call.shape[0], gen)
    s = _interp(xi, x, sig) * torch.sqrt(catalog.GC * mvir[call] / mc / rs)
    vel = bulk[call] + s[:, None] * torch.randn(call.shape[0], 3, generator=gen, device=DEV,
                                                dtype=torch.float64)
    return pos, vel


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _virial(n, prm):
    mvir = np.maximum(n, 1) * prm.particle_mass
    rvir = catalog.virial_radius(prm, mvir)
    return mvir, rvir, catalog.sigma_vir(mvir, rvir)


def _fill(rec, pos, vel, cen32):
    """struct potential records (as 12 floats each) with r2 about cen32."""
    rec[:, 0:3] = pos.float()
    rec[:, 3:6] = vel.float()
    d = rec[:, 0:3] - cen32
    d = d * d
    rec[:, 6] = (d[:, 0] + d[:, 1]) + d[:, 2]


def _batch(case, seed):
    """A batch's records on the device (48 bytes each, as 12 floats) and its
    descriptors on the host."""
    prm = _params(case)
    keep, nc, npot = _call_counts(case)
    n = keep + nc + npot
    H, total = n.shape[0], int(n.sum())
    rng = np.random.Generator(np.random.Philox(int(seed)))
    gen = _gen(seed)
    conc = np.exp(rng.normal(math.log(8.0), 0.3, H))
    mvir, rvir, sv = _virial(keep, prm)
    cen = rng.uniform(0.0, 250.0, (H, 3))
    bulk = rng.normal(0.0, 200.0, (H, 3))
    first = np.concatenate([[0], np.cumsum(n)[:-1]])
    if case["deep"]:  # the sub-haloes lie inside the host
        off = rng.standard_normal((H - 1, 3))
        off /= np.linalg.norm(off, axis=1, keepdims=True)
        cen[1:] = cen[0] + rvir[0] * rng.uniform(0.05, 0.8, (H - 1, 1)) * off
        bulk[1:] = bulk[0] + sv[0] * rng.standard_normal((H - 1, 3))
    call = torch.repeat_interleave(torch.arange(H, device=DEV), _dev(n))
    slot = torch.arange(total, device=DEV) - _dev(first)[call]
    dcen, dbulk, drv = _dev(cen), _dev(bulk), _dev(rvir)
    halo = call
    if case["deep"]:  # the tail of the host's call is its sub-haloes' particles
        subs = int(n[1:].sum())
        halo = call.clone()
        halo[int(n[0]) - subs:int(n[0])] = call[int(n[0]):]
    pos, vel = _nfw(halo, _dev(conc), drv, _dev(mvir), dcen, dbulk, gen)
    rec = torch.zeros(total, 12, dtype=torch.float32, device=DEV)
    kd, kc = _dev(keep)[call], _dev(keep + nc)[call]
    bg = torch.nonzero((slot >= kd) & (slot < kc)).flatten()
    if bg.numel():
        b = call[bg]
        pos[bg] = dcen[b] + drv[b, None] * (2 * torch.rand(bg.numel(), 3, generator=gen, device=DEV,
                                                           dtype=torch.float64) - 1)
        vel[bg] = dbulk[b] + 3 * _dev(sv)[b, None] * torch.randn(
            bg.numel(), 3, generator=gen, device=DEV, dtype=torch.float64)
    po = torch.nonzero(slot >= kc).flatten()
    if po.numel():
        pos[po] = dcen[call[po]] + 2 * (pos[po] - dcen[call[po]])
        rec[po, 10] = -1.0
    _fill(rec, pos, vel, _dev(cen.astype(np.float32))[call])
    rec.view(torch.int32)[:, 11] = 1
    halos = np.zeros(H, catalog.HALO_DTYPE)
    halos["first"], halos["count"] = first, n
    halos["pos"][:, :3], halos["pos"][:, 3:] = cen, bulk
    halos["corevel"] = halos["bulkvel"] = bulk
    halos["is_sub"] = (rng.uniform(size=H) < 0.5) if not case["deep"] else np.arange(H) > 0
    return rec, halos


def _hierarchy(case):
    """FOF groups with sub-haloes to depth 3 (counts and links only)."""
    rng = _shape_rng(case["groups"], case["lo"], case["hi"], 1000 * case["subs"])
    n = catalog.power_law_counts(rng, case["groups"], case["lo"], case["hi"])
    group, parent = np.arange(case["groups"]), np.full(case["groups"], -1)
    level = (n, group, np.arange(case["groups"]))
    at, cols = case["groups"], [(n, group, parent)]
    for depth in range(3):
        ln, lg, lid = level
        kids = np.minimum(6, rng.poisson(case["subs"] / (depth + 1), ln.shape[0])) * (ln > 20)
        p = np.repeat(np.arange(ln.shape[0]), kids)
        u = rng.uniform(size=p.shape[0])
        share = np.exp(rng.uniform(math.log(0.005), math.log(0.5), p.shape[0]))
        share = np.where(u < 0.15, rng.uniform(0.45, 0.9, p.shape[0]), share)
        cn = (ln[p] * np.where(u > 0.97, 0.0, share)).astype(np.int64)
        cols.append((cn, lg[p], lid[p]))
        level = (cn, lg[p], at + np.arange(p.shape[0]))
        at += p.shape[0]
    n, group, parent = (np.concatenate([c[k] for c in cols]) for k in range(3))
    order = np.argsort(group, kind="stable")  # a group's haloes together, parents first
    place = np.empty_like(order)
    place[order] = np.arange(order.shape[0])
    n, group = n[order], group[order]
    parent = np.where(parent[order] < 0, -1, place[parent[order]])
    tree = np.zeros(n.shape[0], catalog.TREE_DTYPE)
    tree["p_start"] = np.concatenate([[0], np.cumsum(n)[:-1]])
    tree["num_p"], tree["sub_of"] = n, parent
    tree["child"] = tree["next_cochild"] = -1
    kin = np.argsort(parent, kind="stable")
    kin = kin[parent[kin] >= 0]
    same = parent[kin][1:] == parent[kin][:-1]
    tree["next_cochild"][kin[:-1][same]] = kin[1:][same]
    heads = kin[np.concatenate([[True], ~same])] if kin.size else kin
    tree["child"][parent[heads]] = heads
    below = n.copy()
    for h in range(n.shape[0] - 1, -1, -1):  # children come after their parent
        if parent[h] >= 0:
            below[parent[h]] += below[h]
    tree["num_child_particles"] = below
    return tree, group


def _groups(case, seed, shuffle):
    """The groups' particle copies on the device (32 bytes, as 8 floats)."""
    prm = _params(case)
    tree, group = _hierarchy(case)
    n = tree["num_p"]
    rng = np.random.Generator(np.random.Philox(int(seed)))
    gen = _gen(seed)
    H = n.shape[0]
    mvir, rvir, sv = _virial(n, prm)
    cen, bulk = rng.uniform(0.0, 100.0, (H, 3)), rng.normal(0.0, 200.0, (H, 3))
    off = rng.standard_normal((H, 3))
    off *= rng.uniform(0.05, 0.8, (H, 1)) / np.linalg.norm(off, axis=1, keepdims=True)
    kick = rng.standard_normal((H, 3))
    todo = np.flatnonzero(tree["sub_of"] >= 0)
    for h in todo:  # parents come first
        p = tree["sub_of"][h]
        cen[h] = cen[p] + rvir[p] * off[h]
        bulk[h] = bulk[p] + sv[p] * kick[h]
    tree["pos"][:, :3], tree["pos"][:, 3:] = cen, bulk
    halo = torch.repeat_interleave(torch.arange(H, device=DEV), _dev(n))
    conc = np.exp(rng.normal(math.log(8.0), 0.3, H))
    pos, vel = _nfw(halo, _dev(conc), _dev(rvir), _dev(mvir), _dev(cen), _dev(bulk), gen)
    total = pos.shape[0]
    if shuffle:  # a FOF pass leaves a group's particles in no order
        key = _dev(group)[halo].double() + 0.999 * torch.rand(total, generator=gen, device=DEV,
                                                              dtype=torch.float64)
        o = torch.argsort(key)
        pos, vel = pos[o], vel[o]
    parts = torch.zeros(total, 8, dtype=torch.float32, device=DEV)
    parts.view(torch.int64)[:, 0] = torch.arange(total, device=DEV)
    parts[:, 2:5], parts[:, 5:8] = pos.float(), vel.float()
    return parts, tree, group


def _to_host(rec):
    return np.ascontiguousarray(rec.cpu().numpy()).view(catalog.POTENTIAL_DTYPE).reshape(-1)


def _host_fields(po):
    return {k: po[k] for k in ("pos", "r2", "pe", "ke", "flags")}


def _dev_fields(rec):
    return {"pos": rec[:, 0:6], "r2": rec[:, 6], "pe": rec.view(torch.float64)[:, 4],
            "ke": rec[:, 10], "flags": rec.view(torch.int32)[:, 11]}


HALO_OUT = ("pos", "corevel", "bulkvel", "min_vel_err", "min_bulkvel_err", "n_core", "kept",
            "n_bound")


def _fields(buf, dtype, names):
    """Views of the fields of packed device rows (a uint8 tensor)."""
    out, size = {}, dtype.itemsize
    kinds = {"f4": torch.float32, "i4": torch.int32, "i8": torch.int64, "f8": torch.float64}
    for f in names:
        dt, at = dtype.fields[f][:2]
        base, w = dt.base.str[1:], int(np.prod(dt.shape)) if dt.shape else 1
        step = dt.base.itemsize
        v = buf.view(kinds[base]).view(-1, size // step)
        out[f] = v[:, at // step:at // step + w] if dt.shape else v[:, at // step]
    return out


def prepare(case, seed):
    path, prm = case["path"], _params(case)
    halopot.set_config(prm)
    if path == "drop_in":
        one = dict(case, calls=1, lo=case["records"], hi=case["records"] + 1, contam=0.09,
                   potential_only=0.0, deep=0)
        rec, halos = _batch(one, seed)
        po = _to_host(rec)
        return {"path": path, "src": po, "po": po.copy(), "vel": halos["bulkvel"][0].copy(),
                "cen": halos["pos"][0].copy(), "a": prm.scale_now}
    if path in ("gather", "subfof"):
        parts, tree, group = _groups(case, seed, path == "subfof")
        if path == "subfof":
            hosts = np.flatnonzero(tree["sub_of"] < 0)
            g = np.zeros(hosts.shape[0], catalog.FOF_GROUP_DTYPE)
            g["first"], g["num_p"] = tree["p_start"][hosts], tree["num_child_particles"][hosts]
            subs = np.zeros((2, parts.shape[0] // 10 + 1), np.int64)  # room for every sub-FOF
            return {"path": path, "src": parts, "parts": parts.clone(), "groups": g, "subs": subs}
        base = np.flatnonzero(tree["num_p"] >= 1).astype(np.int64)
        cap = int(sum(_gather_counts(tree, base)))
        rec = torch.zeros(cap, 12, dtype=torch.float32, device=DEV)
        return {"path": path, "parts": parts, "tree": tree, "base": base, "rec": rec,
                "out": _dev_fields(rec)}
    rec, halos = _batch(case, seed)
    if path == "host":
        po = _to_host(rec)
        return {"path": path, "src": po, "po": po.copy(), "halos": halos, "h": halos.copy()}
    st = {"path": path, "src": rec, "rec": rec.clone(), "H": halos.shape[0],
          "opts": halopot.options(accumulate=ACC[case["acc"]],
                                  use_graph=1 if path == "bound" else 0)}
    st["plan"] = halopot.Plan(halos, st["opts"])
    st["hsrc"] = torch.from_numpy(halos.view(np.uint8).reshape(-1)).to(DEV)
    st["halos"] = st["hsrc"].clone()
    st["bound"] = torch.zeros(rec.shape[0], dtype=torch.uint8, device=DEV)
    st["out"] = _dev_fields(st["rec"])
    if path == "potential":
        return st
    st["out"].update({"halo_" + k: v for k, v in
                      _fields(st["halos"], catalog.HALO_DTYPE, HALO_OUT).items()})
    st["out"]["bound"] = st["bound"]
    if path == "props":
        st["plan"].run(st["rec"].data_ptr(), st["halos"].data_ptr(), st["bound"].data_ptr())
        st["defs"] = halopot.mass_definitions()
        st["props"] = torch.zeros(st["H"] * catalog.PROPS_DTYPE.itemsize, dtype=torch.uint8,
                                  device=DEV)
        st["out"] = _fields(st["props"], catalog.PROPS_DTYPE, catalog.PROPS_DTYPE.names)
    return st


def run(s):
    path = s["path"]
    if path == "drop_in":
        np.copyto(s["po"], s["src"])
        halopot.compute_potential(s["po"])
        halopot.compute_kinetic_energy(s["po"], s["vel"], s["cen"][:3], s["a"])
        return _host_fields(s["po"])
    if path == "host":
        np.copyto(s["po"], s["src"])
        np.copyto(s["h"], s["halos"])
        bound = halopot.bound_pass_host(s["po"], s["h"])
        out = _host_fields(s["po"])
        out.update({"halo_" + k: s["h"][k] for k in HALO_OUT})
        out["bound"] = bound
        return out
    if path == "gather":
        calls, n = halopot.gather_calls(s["tree"], s["base"], s["parts"].data_ptr(),
                                        s["parts"].shape[0], s["rec"].data_ptr(),
                                        s["rec"].shape[0])
        return dict(s["out"], first=calls["first"], count=calls["count"], records=n)
    if path == "subfof":
        s["parts"].copy_(s["src"])
        g, subs = halopot.find_subfofs(s["parts"].data_ptr(), s["parts"].shape[0], s["groups"])
        s["subs"][0, :subs.shape[0]], s["subs"][1, :subs.shape[0]] = subs["first"], subs["num_p"]
        return {"id": s["parts"].view(torch.int64)[:, 0], "pos": s["parts"][:, 2:8],
                "target_r": g["target_r"], "first_sub": g["first_sub"], "num_sub": g["num_sub"],
                "subs": s["subs"], "nsubs": subs.shape[0]}
    if path == "props":
        s["plan"].props(s["rec"].data_ptr(), s["halos"].data_ptr(), s["props"].data_ptr(),
                        s["defs"])
        return s["out"]
    s["rec"].copy_(s["src"])
    if path == "potential":
        s["plan"].potential(s["rec"].data_ptr())
        return s["out"]
    s["halos"].copy_(s["hsrc"])
    s["plan"].run(s["rec"].data_ptr(), s["halos"].data_ptr(), s["bound"].data_ptr())
    return s["out"]


# ------------------------------------------------------------ work and check

def _gather_segments(tree, b):
    """The haloes whose particles call b holds, in order, as the recursion of
    calc_particle_radii visits them: (halo, potential-only)."""
    out, path = [], []

    def visit(h, only):
        if h in path:
            return
        path.append(h)
        out.append((h, only))
        c = int(tree["child"][h])
        while c > -1:
            visit(c, only)
            c = int(tree["next_cochild"][c])
        p = int(tree["sub_of"][h])
        if h == b and p > -1 and (tree["num_child_particles"][p] * 0.3
                                  < tree["num_child_particles"][h]):
            visit(p, True)
        path.pop()

    visit(int(b), False)
    return out


def _gather_counts(tree, base):
    """Records of each call.  The host's subtree, when it joins, leaves out
    the call's own (it is on the descent path)."""
    own, up = tree["num_child_particles"], tree["sub_of"][base]
    joins = (up > -1) & (own[up] * 0.3 < own[base])
    return own[base] + np.where(joins, own[up] - own[base], 0)


def work(case):
    """Bytes: inputs read and outputs written once.  Operations: 11 per pair
    and 10 per monopole term of the walk at the catalogues' counts per record
    (24 pairs, 8 monopoles per level), 18 per 6D distance of one leaf."""
    path = case["path"]
    if path in ("gather", "subfof"):
        tree, _ = _hierarchy(case)
        if path == "gather":
            n = int(sum(_gather_counts(tree, np.flatnonzero(tree["num_p"] >= 1))))
            return {"bytes": 32.0 * int(tree["num_p"].sum()) + 48.0 * n, "flops": 8.0 * n}
        n = int(tree["num_p"].sum())
        return {"bytes": 64.0 * n, "flops": 2.0 * 18 * 40 * n}
    if path == "drop_in":
        n = np.array([case["records"]])
    else:
        n = sum(_call_counts(case))
    N = float(n.sum())
    walk = float((n * (24.0 * 11 + 80.0 * np.log2(np.maximum(n / 10.0, 1.0)))).sum())
    if path == "props":
        return {"bytes": 48.0 * N + 328.0 * n.shape[0], "flops": 150.0 * N}
    if path == "drop_in":
        return {"bytes": 96.0 * N, "flops": walk + 20.0 * N}
    if path == "potential":
        return {"bytes": 96.0 * N, "flops": walk}
    return {"bytes": 97.0 * N + 208.0 * n.shape[0], "flops": walk + 60.0 * N}


def _segments(v, n, op):
    """Per segment (n rows of v each, in order) the sum, amin or amax, 64 rows
    at a time (a reduction straight into one row per segment would serialise)."""
    none = {"sum": 0.0, "amin": math.inf, "amax": -math.inf}[op]
    while True:
        own = torch.repeat_interleave(torch.arange(n.shape[0], device=DEV), n)
        k = torch.arange(own.shape[0], device=DEV) - (torch.cumsum(n, 0) - n)[own]
        last = int(n.max()) <= 64 if n.numel() else True
        c = torch.ones_like(n) if last else (n + 63) // 64
        at = own if last else (torch.cumsum(c, 0) - c)[own] + k // 64
        rows = int(c.sum())
        out = torch.full((rows,) + v.shape[1:], none, dtype=v.dtype, device=DEV)
        out.scatter_reduce_(0, at if v.dim() == 1 else at[:, None].expand(-1, v.shape[1]), v, op)
        if last:
            return out
        v, n = out, c


def _barnes_hut(x, first, count, pm, fr):
    """Potentials, in tree order, and that order, of the reference's tree (split at the midpoint of the widest
    side, 10 points per leaf, float centres and opening distances) with every
    term and sum in 64 bits."""
    N = x.shape[0]
    xd = x.double()
    order = torch.arange(N, device=DEV)
    nf, nn = first.clone(), count.clone()             # per node: first position, points
    left = torch.full_like(nf, -1)
    ids = torch.arange(nf.shape[0], device=DEV)       # the level's nodes
    levels, base = [], nf.shape[0]
    while ids.numel():
        n = nn[ids]
        own = torch.repeat_interleave(torch.arange(ids.shape[0], device=DEV), n)
        start = torch.cumsum(n, 0) - n
        at = nf[ids][own] + (torch.arange(own.shape[0], device=DEV) - start[own])
        p = x[order[at]]
        levels.append((ids, own, at))
        lo, hi = _segments(p, n, "amin"), _segments(p, n, "amax")
        w = hi - lo
        dim = torch.full((ids.shape[0],), 2, device=DEV)
        best = w[:, 2].clone()
        for k in (0, 1):
            up = w[:, k] > best
            dim[up], best[up] = k, w[up, k]
        lim = 0.5 * (hi.gather(1, dim[:, None]) + lo.gather(1, dim[:, None])).flatten()
        big = p.gather(1, dim[own][:, None]).flatten() > lim[own]
        cs = torch.nn.functional.pad(torch.cumsum(~big, 0), (1, 0))
        nl = cs[start + n] - cs[start]
        split = (n > 10) & (nl > 0) & (nl < n)
        mv = torch.nonzero(split[own]).flatten()
        # the in-place partition's order (a point above the plane is swapped
        # with the last slot), from the stable listing st of the two sides
        ow, rel, bg = own[mv], (at - nf[ids][own])[mv], big[mv]
        o = torch.argsort(ow * 2 + bg, stable=True)
        st, lst = rel[o], torch.empty_like(o)
        lst[o] = torch.arange(o.shape[0], device=DEV)
        size = torch.where(split, n, 0)
        sm, ns, nw = (torch.cumsum(size, 0) - size)[ow], nl[ow], n[ow]
        rank = lst - sm - torch.where(bg, ns, 0)
        look = lambda k: st[(sm + k).clamp(0, max(0, st.shape[0] - 1))]  # noqa: E731
        dest = torch.where(bg, torch.where(rel > ns, rel, torch.where(
            rank == 0, nw, look(ns - rank))) - 1, torch.where(rel < ns, rel, look(2 * ns - 1 - rank)))
        order[nf[ids][ow] + dest] = order[at[mv]]
        par = ids[split]
        kids = base + torch.arange(2 * par.shape[0], device=DEV)
        left[par] = kids[0::2]
        f = torch.stack([nf[par], nf[par] + nl[split]], 1).flatten()
        c = torch.stack([nl[split], nn[par] - nl[split]], 1).flatten()
        nf, nn = torch.cat([nf, f]), torch.cat([nn, c])
        left = torch.cat([left, torch.full_like(f, -1)])
        base, ids = base + kids.shape[0], kids
    M = nf.shape[0]
    com, mass = torch.zeros(M, 3, device=DEV), torch.zeros(M, device=DEV)
    dmin2 = torch.zeros(M, device=DEV)
    for ids, own, at in reversed(levels):
        p = x[order[at]]
        n = nn[ids]
        s, seg, n = _segments(p.double(), n, "sum"), n, n.double()
        cm, ms = (s / n[:, None].clamp(min=1)).float(), (pm * n).float()
        inner = left[ids] >= 0
        L = left[ids][inner]
        m = mass[L] + mass[L + 1]
        ms[inner] = m
        cm[inner] = (com[L + 1] * mass[L + 1, None] + com[L] * mass[L, None]) / m[:, None]
        com[ids], mass[ids] = cm, ms
        d2 = (cm[own] - p).double().square().sum(1)
        tot, far = _segments(d2, seg, "sum"), _segments(d2, seg, "amax").clamp(min=0)
        b = far.sqrt() / 2
        dm = (b + (b * b + tot / n.clamp(min=1)).sqrt()).float()
        dmin2[ids] = dm * dm
    pe = torch.zeros(N, dtype=torch.float64, device=DEV)
    xo = xd[order]

    def pairs(a, b, kind):
        """Adds the terms of leaves a with nodes b to the leaves' points."""
        size = nn[a] * (nn[b] if kind else 1)
        for part in torch.split(torch.arange(a.shape[0], device=DEV), 2_000_000):
            rep = torch.repeat_interleave(part, size[part])
            if not rep.numel():
                continue
            k = torch.arange(rep.shape[0], device=DEV) - (torch.cumsum(size[part], 0)
                                                          - size[part])[rep - part[0]]
            if kind:
                q = nn[b[rep]]
                i, j = nf[a[rep]] + k // q, nf[b[rep]] + k % q
                r = (xo[i] - xo[j]).square().sum(1).sqrt().clamp(min=fr)
                t = torch.where(i == j, 0.0, pm / r)
            else:
                i = nf[a[rep]] + k
                t = mass[b[rep]].double() / (xo[i] - com[b[rep]].double()).square().sum(1).sqrt()
            pe.index_add_(0, i, t)

    leaves = torch.nonzero((left < 0) & (nn > 0)).flatten()
    root = torch.searchsorted(first[count > 0], nf[leaves], right=True) - 1
    root = torch.nonzero(count > 0).flatten()[root]
    for a, b in zip(torch.split(leaves, 100_000), torch.split(root, 100_000)):
        while a.numel():
            own = (nf[a] >= nf[b]) & (nf[a] < nf[b] + nn[b])
            d2 = (com[a] - com[b]).double().square().sum(1).float()
            take = ~own & (d2 > dmin2[b])
            pairs(a[take], b[take], 0)
            leaf = ~take & (left[b] < 0) & ~((a == b) & (nn[b] > 20))
            pairs(a[leaf], b[leaf], 1)
            go = ~take & (left[b] >= 0)
            a, b = a[go].repeat(2), torch.cat([left[b[go]], left[b[go]] + 1])
    return pe, order


def _core_velocities(rec, halos, first, kept, prm):
    """Core and bulk velocity of each call's r2-sorted records, in 64 bits."""
    H, dev = first.shape[0], rec.device
    call = torch.repeat_interleave(torch.arange(H, device=dev), kept)
    j = torch.arange(call.shape[0], device=dev) - (torch.cumsum(kept, 0) - kept)[call]
    r2, v = rec[:, 6], rec[:, 3:6].double()
    thr = prm.particle_rvir_dens * 4.0 * math.pi / 3.0
    r6 = (r2 * r2 * r2).double()

    def pick(ok, value, op, none):  # one value per call from the records that qualify
        got = _segments(torch.where(ok, value.double(), none), kept, op)
        return got.long() if value.dtype == torch.int64 else got

    last = pick(j.double() ** 2 > r6 * thr * thr, j, "amax", -1.0).clamp(min=-1)
    start = torch.cumsum(kept, 0) - kept
    edge = r2[(start + last.clamp(min=0)).clamp(max=max(0, r2.shape[0] - 1))].double()
    core = pick(r2.double() * 100.0 < edge[call], j, "amax", -1.0).clamp(min=100)
    d = v - _dev(halos["bulkvel"].astype(np.float64))[call]  # small numbers: no cancellation
    zero = torch.zeros(1, 3, dtype=torch.float64, device=dev)

    def prefix(t):
        s = torch.cat([zero, torch.cumsum(t, 0)])
        return s[1:] - s[start][call]

    s1, s2 = prefix(d), prefix(d * d)
    n = (j + 1).double()
    var = (s2 - s1 * s1 / n[:, None]).sum(1)
    score = var / ((j - 3) * j).clamp(min=1).double()
    out = []
    for limit in (torch.minimum(last, core), last):
        use = (j < limit[call]) & ((j >= 9) | (j == limit[call] - 1))
        use &= (j >= 9) | (limit[call] <= 10)
        best = pick(use, score, "amin", math.inf)
        at = pick(use & (score == best[call]), j, "amin", 1e15)
        ok = (at < 10 ** 12) & (last >= 1)
        base = _dev(halos["bulkvel"].astype(np.float64))
        k = (start + torch.where(ok, at, 0)).clamp(max=max(0, r2.shape[0] - 1))
        out.append(torch.where(ok[:, None], base + s1[k] / n[k][:, None], base))
    return out


def exact(case, seed):
    path, prm = case["path"], _params(case)
    if path in ("props", "subfof"):
        return None  # orders, lengths and shapes that float roundings decide step by step
    if path == "gather":
        parts, tree, _ = _groups(case, seed, False)
        base = np.flatnonzero(tree["num_p"] >= 1)
        if base.shape[0] > 30_000:
            return None
        at, cen = [], []
        for b in base:
            segs = [h for h, _ in _gather_segments(tree, b)]
            at += [np.arange(tree["p_start"][h], tree["p_start"][h] + tree["num_p"][h])
                   for h in segs]
            cen.append(np.full(int(tree["num_p"][segs].sum()), b))
        at, cen = _dev(np.concatenate(at)), _dev(np.concatenate(cen))
        c = _dev(tree["pos"][:, :3].astype(np.float64))
        r2 = (parts[at, 2:5].double() - c[cen]).square().sum(1)
        return {"pos": parts[at, 2:8].double(), "r2": r2, "pe": torch.zeros_like(r2), "ke": None,
                "flags": None, "first": None, "count": None, "records": None}
    if path == "drop_in":
        rec, halos = _batch(dict(case, calls=1, lo=case["records"], hi=case["records"] + 1,
                                 contam=0.09, potential_only=0.0, deep=0), seed)
    else:
        rec, halos = _batch(case, seed)
    first, count = _dev(halos["first"]), _dev(halos["count"])
    pe, order = _barnes_hut(rec[:, 0:3].contiguous(), first, count, prm.particle_mass,
                            prm.force_res)
    rec = rec[order]  # compute_potential leaves a call's records in tree order
    hub = 100.0 * prm.hubble_scaling(0.0)
    if path == "potential":
        return {"pos": rec[:, 0:6].double(), "r2": rec[:, 6].double(), "pe": pe, "ke": None,
                "flags": None}
    if path == "drop_in":
        c = _dev(halos["pos"][0].astype(np.float64))
        vc = _dev(halos["bulkvel"][0].astype(np.float64))
        dv = rec[:, 3:6].double() - vc + hub * (rec[:, 0:3].double() - c[:3])
        return {"pos": rec[:, 0:6].double(), "r2": rec[:, 6].double(), "pe": pe,
                "ke": 0.5 / catalog.GC * dv.square().sum(1), "flags": None}
    # a call's kept records by r2, then its potential-only ones (in no set order)
    call = torch.repeat_interleave(torch.arange(first.shape[0], device=DEV), count)
    only = rec[:, 10] < 0
    o = torch.argsort(rec[:, 6], stable=True)
    o = o[torch.argsort((call * 2 + only)[o], stable=True)]
    rec, pe, only, call = rec[o], pe[o], only[o], call[o]
    kept = count - torch.zeros_like(count).scatter_add_(0, call, only.long())
    core, bulk = _core_velocities(rec[~only], halos, first, kept, prm)
    sub = _dev(halos["is_sub"].astype(np.int64)) > 0
    vc = torch.where(sub[:, None], core, bulk)
    c = _dev(halos["pos"][:, :3].astype(np.float64))
    dv = rec[:, 3:6].double() - vc[call] + hub * (rec[:, 0:3].double() - c[call])
    ke = torch.where(only, -1.0, 0.5 / catalog.GC * dv.square().sum(1))
    out = {"pos": None, "r2": rec[:, 6].double() if not bool(only.any()) else None,
           "pe": pe if not bool(only.any()) else None, "ke": ke, "flags": None, "bound": None}
    out.update({"halo_" + k: None for k in HALO_OUT})
    out["halo_corevel"], out["halo_bulkvel"] = core, bulk
    return out
