"""The measured cases of the collision-query framework: what an optimizer does with it, through its
public Python entry points, from one small batch of sampled placements to a full plan over a large
layout.

A case is a dict of plain values.  `kind` names the call:

    detect      CDEngine.detect_batch, one item's sampled placements against one layout
    collect     CDEngine.collect_batch, the hazard set of every placement
    plan        QueryPlan.detect over many items (and layouts) in one launch sequence
    plan_sets   QueryPlan.collect, the hazard sets of a plan's queries
    search      PlacementSearch.run + results, sampled placement search on the GPU
    place       register an item, query the changed layout, take the item out again
    overlap     PoleOverlap.forward_backward, one evaluation of an optimizer step
    surrogates  SPolygon.new_batch, shape import with its pole (and pier) searches

Inputs are synthetic and come from the seed alone; sizes are those of the benchmark's workloads
and of the tests.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "jagua-rs_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import jagua_amd as J  # noqa: E402
from jagua_amd import synth as S  # noqa: E402

F32 = np.float32


def listed():
    return [
        # a few candidate poses of one small item in a small strip layout: a caller's latency
        dict(name="detect_small", kind="detect", layout="strip", items=40, queries=64, nv=16, filter="none", host=False),
        # the samples lbf draws for one item (5000 by default) against a large layout
        dict(name="detect_item", kind="detect", layout="sheet", items=2000, queries=5000, nv=64, filter="none", host=False),
        # the same call with host arrays and the item's own key filtered out (a feasibility check)
        dict(name="detect_host", kind="detect", layout="sheet", items=600, queries=1000, nv=48, filter="keys", host=True),
        # which hazards a set of placements would collide with, for an overlap-minimizing optimizer
        dict(name="collect_item", kind="collect", layout="sheet", items=2000, queries=4096, nv=64, capacity=16, host=False),
        # every item type of an instance sampled at once over a large sheet (the benchmark's workload)
        dict(name="plan_sheet", kind="plan", layout="sheet", items=2000, layouts=1, polys=64, queries=16384, nv=512, filter="none"),
        # many independent star-shaped bins, each query with its own random hazard filter
        dict(name="plan_bins", kind="plan", layout="bins", items=200, layouts=16, polys=16, queries=2048, nv=256, filter="hashed"),
        # concave items of many vertices, a deep quadtree
        dict(name="plan_concave", kind="plan", layout="concave", items=2500, layouts=1, polys=32, queries=16384, nv=1024, filter="none"),
        # the hazard sets of a plan's queries
        dict(name="plan_sets", kind="plan_sets", layout="sheet", items=2000, layouts=1, polys=32, queries=8192, nv=512, capacity=8),
        # lbf's sampled search of 64 item types at once, 10 rounds of 500 samples each
        dict(name="search", kind="search", layout="sheet", items=2000, searches=64, samples=500, uniform=8, local=2, nv=512),
        # the constructive loop: place an item, sample the next one, undo
        dict(name="place", kind="place", layout="sheet", items=1000, queries=2000, nv=64),
        # Q and its gradient over all items of a layout
        dict(name="overlap", kind="overlap", items=4096, poles_lo=16, poles_hi=64),
        # the shapes of an instance, imported with the default surrogate configuration
        dict(name="surrogates", kind="surrogates", polys=192, nv=256, piers=0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["detect", "detect", "collect", "plan", "plan", "plan_sets", "search", "place", "overlap", "surrogates"])
    if kind in ("detect", "collect"):
        layout = rng.choice(["strip", "sheet"])
        c = dict(kind=kind, layout=layout, items=_log_int(rng, 10, 60) if layout == "strip" else _log_int(rng, 100, 2000),
                 queries=_log_int(rng, 1, 40000 if kind == "detect" else 10000), nv=_log_int(rng, 8, 256),
                 host=rng.random() < 0.25)
        if kind == "detect":
            c["filter"] = rng.choice(["none", "none", "keys", "hashed"])
        else:
            c["capacity"] = rng.choice([0, 4, 8, 16, 32])
        return c
    if kind == "plan":
        layout = rng.choice(["sheet", "bins", "concave"])
        return dict(kind=kind, layout=layout, items=_log_int(rng, 50, 200) if layout == "bins" else _log_int(rng, 200, 2000),
                    layouts=rng.randint(2, 12) if layout == "bins" else 1, polys=rng.randint(1, 48 if layout != "bins" else 12),
                    queries=_log_int(rng, 50, 12000 if layout != "bins" else 2000), nv=_log_int(rng, 16, 512),
                    filter=rng.choice(["none", "none", "keys", "hashed"]))
    if kind == "plan_sets":
        return dict(kind=kind, layout="sheet", items=_log_int(rng, 200, 2000), layouts=1, polys=rng.randint(1, 32),
                    queries=_log_int(rng, 50, 6000), nv=_log_int(rng, 16, 512), capacity=rng.choice([0, 4, 8, 16]))
    if kind == "search":
        return dict(kind=kind, layout=rng.choice(["strip", "sheet"]), items=_log_int(rng, 30, 60), searches=_log_int(rng, 4, 64),
                    samples=_log_int(rng, 100, 500), uniform=rng.randint(2, 8), local=rng.randint(0, 2), nv=_log_int(rng, 16, 256))
    if kind == "place":
        return dict(kind=kind, layout="sheet", items=_log_int(rng, 50, 1500), queries=_log_int(rng, 50, 5000), nv=_log_int(rng, 8, 256))
    if kind == "overlap":
        return dict(kind=kind, items=_log_int(rng, 16, 4000), poles_lo=rng.randint(1, 16), poles_hi=rng.randint(17, 90))
    return dict(kind=kind, polys=_log_int(rng, 1, 120), nv=_log_int(rng, 8, 200), piers=rng.choice([0, 0, 1]))


# ------------------------------------------------------------------------------------ layouts


def _scene(case, seed, k=0):
    """One layout: container, holes and placed items."""
    s, n = (seed * 131 + 17 * k) & 0x3FFFFFFF, case["items"]
    if case["layout"] == "strip":
        # 1000 x 400 strip of twelve-vertex stars placed left-bottom-fill, rotations of 45 degrees
        return S.generate_scene(depth=5, seed=s, container_kind=0, cw=1000.0, ch=400.0, n_items=n, item_nv_lo=12,
                                item_nv_hi=12, item_r_lo=20.0, item_r_hi=40.0, item_shape=0, rot_kind=1, placement=1,
                                lbf_samples=2000, min_sep=0.0), (0.0, 0.0, 1000.0, 400.0)
    if case["layout"] == "bins":
        # a star-shaped bin filled with star and concave polygons
        r = 40.0 * math.sqrt(n)
        sc = S.generate_scene(depth=7, seed=s, container_kind=1, cw=0.7 * r, ch=r, container_nv_lo=64, container_nv_hi=2048,
                              n_items=n, item_nv_lo=8, item_nv_hi=256, item_r_lo=10.0, item_r_hi=30.0, item_shape=2,
                              min_sep=0.0, rot_kind=0, placement=0, max_attempts=600)
        c = sc.container
        return sc, (float(c[:, 0].min()), float(c[:, 1].min()), float(c[:, 0].max()), float(c[:, 1].max()))
    # sheets keep the density of 2000 items on 4000 x 1500 (polygons of radius 10-30) and of
    # 20000 on 6000 x 2000 (concave ones of radius 6-12)
    if case["layout"] == "sheet":
        f = math.sqrt(n / 2000.0)
        w, h = 4000.0 * f, 1500.0 * f
        sc = S.generate_scene(depth=8, seed=s, container_kind=0, cw=w, ch=h, n_holes=5, hole_kind=0, hole_lo=50.0 * f,
                              hole_hi=300.0 * f, n_items=n, item_nv_lo=8, item_nv_hi=256, item_r_lo=10.0, item_r_hi=30.0,
                              item_shape=2, min_sep=0.5, rot_kind=0, placement=0, max_attempts=2000)
        return sc, (0.0, 0.0, w, h)
    f = math.sqrt(n / 20000.0)
    w, h = 6000.0 * f, 2000.0 * f
    rng = np.random.default_rng(s)
    nx = int(math.ceil(math.sqrt(n * w / h)))
    ny = int(math.ceil(n / nx))
    gx, gy = w / nx, h / ny
    items = []
    for i in range(n):
        lim = 0.5 * min(gx, gy)
        p = S.polygon(s * 7 + i, 64, 1024, 0.55 * lim, 0.9 * lim, 1)
        x, y = (i % nx + 0.5) * gx + rng.uniform(-0.08, 0.08) * gx, (i // nx + 0.5) * gy + rng.uniform(-0.08, 0.08) * gy
        items.append((p, np.array([rng.uniform(0, 2 * math.pi), x, y], dtype=F32)))
    cont = np.array([[0, 0], [w, 0], [w, h], [0, h]], dtype=F32)
    return S.Scene(cont, [], items, 10, 16), (0.0, 0.0, w, h)


def _polys(seed, n, nv, layout):
    """Query polygons of 8 to nv vertices (log-uniform), sized like the layout's items."""
    lo, hi, shape = {"strip": (15.0, 35.0, 0), "concave": (6.0, 12.0, 2)}.get(layout, (10.0, 30.0, 2))
    return [S.polygon(seed * 100003 + 31 * i + 1, min(8, nv), nv, lo, hi, shape) for i in range(n)]


def _mats(seed, n, box, layout):
    return J.compose(S.transforms(seed, n, box, 1 if layout == "strip" else 0))


def _filter(case, keys, seed):
    kind = case.get("filter", "none")
    if kind == "keys":
        return J.HazKeyFilter(keys[:: max(1, len(keys) // 5)])
    return J.HashedFilter(seed & 0xFFFF, 0.1) if kind == "hashed" else None


# ------------------------------------------------------------------------------------ prepare


def prepare(case, seed):
    dev = torch.device("cuda:0")
    kind = case["kind"]
    if kind == "surrogates":
        cfg = J.SPSurrogateConfig(n_ff_piers=case["piers"])
        return dict(kind=kind, polys=_polys(seed, case["polys"], case["nv"], "sheet"), cfg=cfg)
    if kind == "overlap":
        w = _overlap_inputs(case, seed)
        pairs = J.candidate_pairs(w["pose"], w["rad"], [0.0, 0.0, w["w"], w["h"]], 8)
        ov = J.PoleOverlap(w["poles"], w["off"], pairs, w["cedges"])
        return dict(kind=kind, ov=ov, pose=torch.from_numpy(w["pose"]).to(dev),
                    q=torch.empty(1, dtype=torch.float32, device=dev),
                    grad=torch.empty((case["items"], 3), dtype=torch.float32, device=dev))
    scenes = [_scene(case, seed, k) for k in range(case.get("layouts", 1))]
    engines = [S.build_cde(sc) for sc, _ in scenes]
    for cde, _ in engines:
        cde.sync()
    (cde, keys), (scene, box), layout = engines[0], scenes[0], case["layout"]
    if kind in ("detect", "collect", "place"):
        item = J.SPolygon.new_batch([S.polygon(seed * 7919 + 11, case["nv"], case["nv"], 15.0, 30.0, 0)])[0][0]
        m = _mats(seed * 7919 + 12, case["queries"], box, layout)
        n = len(m)
        st = dict(kind=kind, cde=cde, item=item, m=m if case.get("host") else torch.from_numpy(m).to(dev), host=case.get("host", False),
                  filter=_filter(case, keys, seed), capacity=case.get("capacity", 0))
        if kind == "place":
            dt = S.transforms(seed * 7919 + 13, 1, box, 0)[0]
            shape = J.SPolygon.new(S.polygon(seed * 7919 + 14, 64, 64, 10.0, 30.0, 2)).transform_clone(dt)
            st["hazard"] = J.Hazard(J.HazardEntity.placed_item(1 << 20, dt, 1 << 20), shape, True)
        if not st["host"]:
            st["out"] = torch.empty(n, dtype=torch.uint8, device=dev)
            cap = max(1, st["capacity"])
            st["sets"] = (torch.empty(n, dtype=torch.int32, device=dev), torch.empty(n, dtype=torch.int64, device=dev),
                          torch.full((n, cap), -1, dtype=torch.int32, device=dev))
        return st
    if kind == "search":
        polys = _polys(seed, case["searches"], case["nv"], layout)
        items, _ = J.SPolygon.new_batch(polys)
        rots = ["continuous", [0.0, math.pi], None]
        ps = J.PlacementSearch([(cde, it, rots[i % 3], None) for i, it in enumerate(items)], samples_per_round=case["samples"],
                               uniform_rounds=case["uniform"], local_rounds=case["local"], seed=seed)
        return dict(kind=kind, search=ps)
    polys = _polys(seed, case["polys"], case["nv"], layout)
    items, _ = J.SPolygon.new_batch(polys)
    sets, mats, at = [], [], 0
    for k, ((cde, keys), (_, box)) in enumerate(zip(engines, scenes)):
        for i, it in enumerate(items):
            mats.append(_mats(seed * 100003 + 64 * k + i, case["queries"], box, layout))
            sets.append((cde, it, at, case["queries"], _filter(case, keys, seed + k)))
            at += case["queries"]
    m = torch.from_numpy(np.concatenate(mats)).to(dev)
    st = dict(kind=kind, plan=J.QueryPlan(sets), m=m, out=torch.empty(at, dtype=torch.uint8, device=dev))
    if kind == "plan_sets":
        cap = case["capacity"]
        st.update(capacity=cap, count=torch.empty(at, dtype=torch.int32, device=dev), hash=torch.empty(at, dtype=torch.int64, device=dev),
                  keys=torch.empty((at, cap), dtype=torch.int32, device=dev) if cap else None)
    return st


# ------------------------------------------------------------------------------------ run


def run(st):
    kind = st["kind"]
    if kind == "detect":
        if st["host"]:
            return {"status": st["cde"].detect_batch(st["item"], st["m"], st["filter"])}
        return {"status": st["cde"].detect_batch(st["item"], st["m"], st["filter"], out=st["out"])}
    if kind == "collect":
        if st["host"]:
            cnt, hsh, keys = st["cde"].collect_batch(st["item"], st["m"], capacity=st["capacity"])
            hsh = hsh.view(np.int64)
        else:
            cnt, hsh, keys = st["cde"].collect_batch(st["item"], st["m"], capacity=st["capacity"], out=st["sets"])
        return {"count": cnt, "hash": hsh, "keys": keys if st["capacity"] else None}
    if kind == "place":
        key = st["cde"].register_hazard(st["hazard"])
        status = st["cde"].detect_batch(st["item"], st["m"], out=st["out"])
        st["cde"].deregister_hazard_by_key(key)
        return {"status": status, "slot": key.idx}
    if kind == "plan":
        return {"status": st["plan"].detect(st["m"], st["out"])}
    if kind == "plan_sets":
        cnt, hsh, keys = st["plan"].collect(st["m"], st["capacity"], count=st["count"], hash=st["hash"], keys=st["keys"])
        return {"count": cnt, "hash": hsh, "keys": keys}
    if kind == "search":
        res = st["search"].run(graph=True).results()
        return {k: np.array([r[k] for r in res], dtype=np.float32 if k not in ("found", "samples") else np.int32)
                for k in ("found", "rotation", "tx", "ty", "cost", "x_max", "y_max", "samples")}
    if kind == "overlap":
        q, grad = st["ov"].forward_backward(st["pose"], q=st["q"], grad=st["grad"])
        return {"q": q, "grad": grad}
    shapes, _ = J.SPolygon.new_batch(st["polys"], st["cfg"])
    infos = [p.info() for p in shapes]
    poles = np.zeros((len(shapes), 100, 3), dtype=np.float32)      # at most 100 poles each (SPSurrogateConfig)
    for row, p, i in zip(poles, shapes, infos):
        row[: i.n_poles] = p.poles
    return {"n_poles": np.array([i.n_poles for i in infos], dtype=np.int32), "poles": poles,
            "piers": np.concatenate([p.piers for p in shapes]),
            "area": np.array([i.area for i in infos], dtype=np.float32),
            "poi": np.array([i.poi[:] for i in infos], dtype=np.float32)}


# ------------------------------------------------------------------------------------ overlap inputs


def _overlap_inputs(case, seed):
    """Items on a jittered grid (the density of 4096 on 2000 x 800), each with its inscribed circles:
    one large pole near the middle, the further ones smaller and further out."""
    rng = np.random.default_rng(seed)
    n = case["items"]
    f = math.sqrt(n / 4096.0)
    w, h = 2000.0 * f, 800.0 * f
    nx = int(math.ceil(math.sqrt(n * w / h)))
    ny = int(math.ceil(n / nx))
    gx, gy = w / nx, h / ny
    radius = rng.uniform(6.0, 11.5, n)
    count = rng.integers(case["poles_lo"], case["poles_hi"] + 1, n)
    off = np.zeros(n + 1, dtype=np.uint32)
    off[1:] = np.cumsum(count)
    item = np.repeat(np.arange(n), count)
    k = np.arange(len(item)) - off[item]
    r = radius[item] * 0.6 * (1.0 + k) ** -0.6 * rng.uniform(0.7, 1.0, len(item))
    d = (radius[item] - r) * np.sqrt(rng.uniform(0.0, 1.0, len(item))) * np.where(k == 0, 0.3, 1.0)
    a = rng.uniform(0.0, 2.0 * math.pi, len(item))
    poles = np.stack([d * np.cos(a), d * np.sin(a), r], axis=1).astype(F32)
    i = np.arange(n)
    pose = np.stack([(i % nx + 0.5) * gx + rng.uniform(-3.0, 3.0, n), (i // nx + 0.5) * gy + rng.uniform(-3.0, 3.0, n),
                     rng.uniform(0.0, 2.0 * math.pi, n)], axis=1).astype(F32)
    rad = np.array([np.max(np.hypot(p[:, 0], p[:, 1]) + p[:, 2]) for p in np.split(poles, off[1:-1])], dtype=F32)
    cedges = np.array([[0, 0, w, 0], [w, 0, w, h], [w, h, 0, h], [0, h, 0, 0]], dtype=F32)
    return dict(poles=poles, off=off, item=item, count=count, pose=pose, rad=rad, cedges=cedges, w=w, h=h)


# ------------------------------------------------------------------------------------ exact


def exact(case, seed):
    """The overlap and its gradient, and the imported polygons' areas, in 64 bits.  The queries
    return whole numbers; a pole search's or a placement search's result is the outcome of a long
    chain of comparisons, which has no value of its own in 64 bits."""
    if case["kind"] == "surrogates":
        area = []
        for p in _polys(seed, case["polys"], case["nv"], "sheet"):
            x, y = p[:, 0].astype(np.float64), p[:, 1].astype(np.float64)
            area.append(abs(0.5 * float(np.sum(x * np.roll(y, -1) - np.roll(x, -1) * y))))
        return {"n_poles": None, "poles": None, "piers": None, "area": np.array(area), "poi": None}
    if case["kind"] != "overlap":
        return None
    w = _overlap_inputs(case, seed)
    n = case["items"]
    rad = w["rad"].astype(np.float64)
    pose = torch.from_numpy(w["pose"].astype(np.float64)).requires_grad_(True)
    width = int(w["count"].max())
    pad = torch.zeros((n, width, 3), dtype=torch.float64)
    pad[..., 2] = -1.0
    pad[torch.from_numpy(w["item"]), torch.from_numpy((np.arange(len(w["item"])) - w["off"][w["item"]]).astype(np.int64))] = \
        torch.from_numpy(w["poles"].astype(np.float64))
    c, s = torch.cos(pose[:, 2:3]), torch.sin(pose[:, 2:3])
    cx = c * pad[..., 0] - s * pad[..., 1] + pose[:, 0:1]
    cy = s * pad[..., 0] + c * pad[..., 1] + pose[:, 1:2]
    r, real = pad[..., 2], pad[..., 2] >= 0
    # pairs of items whose bounding circles come near each other: others cannot overlap
    p32 = w["pose"].astype(np.float64)
    ia, ib = [], []
    for i in range(n):
        d = np.hypot(p32[i + 1:, 0] - p32[i, 0], p32[i + 1:, 1] - p32[i, 1])
        j = np.nonzero(d <= (rad[i + 1:] + rad[i]) * 1.001)[0] + i + 1
        ia.append(np.full(len(j), i))
        ib.append(j)
    ia, ib = np.concatenate(ia), np.concatenate(ib)
    q = torch.zeros((), dtype=torch.float64)
    for k in range(0, len(ia), 2048):
        a, b = torch.from_numpy(ia[k:k + 2048]), torch.from_numpy(ib[k:k + 2048])
        dx, dy = cx[a][:, :, None] - cx[b][:, None, :], cy[a][:, :, None] - cy[b][:, None, :]
        sq = dx * dx + dy * dy
        sr = r[a][:, :, None] + r[b][:, None, :]
        hit = real[a][:, :, None] & real[b][:, None, :] & (sq < sr * sr)
        pen = sr[hit] - torch.sqrt(sq[hit])
        part = (pen * pen).sum()
        part.backward(retain_graph=True)
        q = q + part.detach()
    # the container is a rectangle: signed distance to its boundary, positive inside
    x, y, ri = cx[real], cy[real], r[real]
    cw, ch = float(w["cedges"][0, 2]), float(w["cedges"][1, 3])
    inner = torch.minimum(torch.minimum(x, cw - x), torch.minimum(y, ch - y))
    ox, oy = torch.clamp(torch.maximum(-x, x - cw), min=0.0), torch.clamp(torch.maximum(-y, y - ch), min=0.0)
    outer = torch.sqrt(torch.clamp(ox * ox + oy * oy, min=1e-300))
    dist = torch.where(inner >= 0, inner, -outer)
    pen = torch.clamp(ri - dist, min=0.0)
    part = (pen * pen).sum()
    part.backward()
    q = q + part.detach()
    return {"q": q.reshape(1), "grad": pose.grad}


# ------------------------------------------------------------------------------------ work


def work(case):
    """Every transform (or polygon, or pole) read once, every result written once and the layout's
    edges read once, with the transformation of the entities each query tests at the least (its two
    fail-fast poles; the vertices too where sets are collected)."""
    kind = case["kind"]
    if kind == "surrogates":
        v = case["polys"] * case["nv"] * 0.35            # vertices: log-uniform from 8 up
        return {"bytes": 8.0 * v + 16.0 * 20 * case["polys"], "flops": 20.0 * v * 20 * 100}
    if kind == "overlap":
        mean = 0.5 * (case["poles_lo"] + case["poles_hi"])
        pairs = 1.47 * case["items"]                     # candidate pairs at this density
        return {"bytes": 16.0 * mean * case["items"] + 24.0 * case["items"], "flops": 8.0 * pairs * mean * mean}
    edges = case["items"] * {"strip": 12, "bins": 72, "sheet": 72, "concave": 346}[case["layout"]] * case.get("layouts", 1)
    if kind == "search":
        n = case["searches"] * case["samples"] * (case["uniform"] + case["local"])
        return {"bytes": 16.0 * edges + 16.0 * n, "flops": 16.0 * n}
    n = case["queries"] * case.get("polys", 1) * case.get("layouts", 1)
    if kind in ("collect", "plan_sets"):
        nv = case["nv"] if kind == "collect" else 0.35 * case["nv"]
        return {"bytes": 16.0 * edges + n * (24.0 + 12.0 + 4.0 * case["capacity"]), "flops": n * (16.0 + 8.0 * nv)}
    return {"bytes": 16.0 * edges + 25.0 * n, "flops": 16.0 * n}
