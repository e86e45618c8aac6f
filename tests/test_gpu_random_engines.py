"""Random engines (depth, threshold, container, root box, scale, place; hazards across every border), items
(sizes, poles, piers), filters and placements in and around the container, through every query form,
against the oracle, bit for bit."""
import numpy as np
import pytest
import torch

import jagua_amd as J
from jagua_amd import synth as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _engine(rng, seed, to_world):
    w, h = 100.0, 100.0 * rng.choice([1.0, 0.5, 1.7])
    cont = np.array([[0, 0], [w, 0], [w, h], [0, h]]) if seed % 4 else S.polygon(seed, 8, 40, 0.35 * min(w, h), 0.5 * min(w, h)) + (w / 2, h / 2)
    cont = to_world(cont)
    bbox = S.Scene(cont).cde_bbox() if seed % 5 else np.concatenate([cont.min(0), cont.max(0)])
    haz = [(O.KIND_EXTERIOR, cont)]
    if seed % 7 == 3:
        haz.append((O.KIND_EXTERIOR, to_world(S.polygon(seed + 5, 4, 12, 10.0, 30.0) + (0.6 * w, 0.5 * h))))
    for i in range(int(rng.choice([0, 3, 20, 80]))):
        r = rng.uniform(1.0, 12.0) * (3.0 if i % 17 == 0 else 1.0)
        haz.append((O.KIND_HOLE, to_world(S.polygon(seed * 100 + i, 3 if i % 9 == 0 else 4, 24, 0.5 * r, r, int(rng.integers(0, 3)))
                                          + rng.uniform((-5, -5), (w + 5, h + 5)))))
    depth, threshold = int(rng.integers(0, 13)), int(rng.choice([0, 1, 4, 16, 64, 255]))
    oc = O.OracleCDE.from_hazards(bbox, depth, threshold, [(k, i, 0, v) for i, (k, v) in enumerate(haz)])
    cde = J.CDEngine(bbox, [J.Hazard(J.HazardEntity(k, i), J.SPolygon.new(v), False) for i, (k, v) in enumerate(haz)],
                     J.CDEConfig(depth, threshold, J.SPSurrogateConfig()))
    return cde, oc, len(haz), w, h


@pytest.mark.parametrize("seed", [1, 2, 3, 5, 10, 14, 15, 17, 24, 31])
def test_random_engine(cuda, seed):
    rng = np.random.default_rng(seed)
    scale = 10.0 ** rng.uniform(-2, 3) if seed % 3 else 1.0
    off = np.zeros(2) if seed % 2 else rng.uniform(-1, 1, 2) * scale * 100.0 * 10.0 ** rng.uniform(0, 2.5)
    cde, oc, n_haz, w, h = _engine(rng, seed, lambda v: (np.asarray(v, np.float64) * scale + off).astype(np.float32))
    sets, mats, detect, collect, first = [], [], [], [], 0
    for j in range(3):
        r, nv = float(rng.choice([0.5, 3, 8, 30])), int(rng.choice([4, 12, 40, 130]))
        poles, piers = int(rng.integers(1, 4)), int(rng.choice([0, 0, 2]))
        poly = (S.polygon(seed * 31 + j, nv, nv, 0.5 * r, r, int(rng.integers(0, 3))) * np.float32(scale)).astype(np.float32)
        n = int(rng.choice([1, 17, 300, 2500]))
        xy = rng.uniform((-0.15 * w, -0.15 * h), (1.15 * w, 1.15 * h), (n, 2)) * scale + off
        m = J.compose(np.concatenate([rng.uniform(0, 6.28, (n, 1)), xy], 1).astype(np.float32))
        kind, f, of = int(rng.integers(0, 3)), None, None
        if kind == 1:
            f = J.HashedFilter(int(rng.integers(0, 99)), float(rng.uniform(0, 1)))
            of = O.make_filter(2, f.seed, f.threshold)
        elif kind == 2:
            keys = [k for k in range(1, n_haz + 1) if rng.random() < 0.4]
            f, of = J.HazKeyFilter([J.HazKey(k, 1) for k in keys]), O.make_filter(1, keys=keys)
        try:
            oitem = O.OracleItem(poly, n_ff_poles=poles, n_ff_piers=piers)
        except RuntimeError:                             # (no pier found)
            continue
        item = S.make_items([poly], J.SPSurrogateConfig(n_ff_poles=poles, n_ff_piers=piers))[0]
        detect.append(O.query(oc, oitem, mats=m, mode=1, filt=of, threads=8)["status"])
        collect.append(O.query(oc, oitem, mats=m, mode=2, keys_cap=6, threads=8))
        t = torch.from_numpy(m).to(cuda)
        np.testing.assert_array_equal(cde.detect_batch(item, t, f).cpu().numpy(), detect[-1])
        _same_sets(cde.collect_batch(item, t, capacity=6), collect[-1:])
        sets.append((cde, item, first, n, f))
        mats.append(m)
        first += n
    assert sets
    m, ref = torch.from_numpy(np.concatenate(mats)).to(cuda), np.concatenate(detect)
    out = torch.empty(first, dtype=torch.uint8, device=cuda)
    for cfg in ({}, {"lanes_per_query": 8}, {"lanes_per_query": 64, "chunk": 16}, {"stages": 1}, {"workgroups": 5}):
        out.fill_(99)
        J.QueryPlan(sets, **cfg).detect(m, out)
        np.testing.assert_array_equal(out.cpu().numpy(), ref, str(cfg))
    out.fill_(99)
    cde.sync()
    J.detect_sets_noalloc(sets, m, out)
    np.testing.assert_array_equal(out.cpu().numpy(), ref)
    _same_sets(J.QueryPlan([(*s[:4], None) for s in sets]).collect(m, capacity=6), collect)


def _same_sets(got, ref):
    cnt, hsh, keys = (t.cpu().numpy() for t in got)
    np.testing.assert_array_equal(cnt.astype(np.uint32), np.concatenate([r["count"] for r in ref]))
    np.testing.assert_array_equal(hsh.view(np.uint64), np.concatenate([r["hash"] for r in ref]))
    np.testing.assert_array_equal(keys.view(np.uint32), np.concatenate([r["keys"] for r in ref]))
