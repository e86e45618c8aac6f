"""Hazard collection where queries have more hazards than the wave traversal's collector holds: every
query of a batch (by the per-query kernel) or some of them (left to the second launch), against
the oracle, bit for bit, at the sizes where the second launch's shares change; and how their time
grows with the batch."""
import numpy as np
import pytest
import torch

import jagua_amd as J
from jagua_amd import synth as S
from oracle import oracle as O

from helpers import engines, items

pytestmark = pytest.mark.gpu

W, H = 1000.0, 800.0
WAVES = 256 * 16


@pytest.fixture(scope="module")
def cluster():
    """120 small items on one another in a spot of a wide sheet, and 40 all over it."""
    rng = np.random.default_rng(7)
    xy = np.concatenate([rng.uniform(-12, 12, (120, 2)) + (300.0, 250.0), rng.uniform((30, 30), (W - 30, H - 30), (40, 2))])
    its = [(S.polygon(40 + i % 8, 5, 12, 2.0, 6.0, 0), np.array([rng.uniform(0, 6.28), *p], np.float32)) for i, p in enumerate(xy)]
    sc = S.Scene(np.array([[0, 0], [W, 0], [W, H], [0, H]], np.float32), [], its, 7, 16)
    return engines(sc)


def _mats(seed, n, spot):
    """n placements, all over the sheet but for the share `spot` of them on the cluster."""
    rng = np.random.default_rng(seed)
    xy = rng.uniform((0, 0), (W, H), (n, 2))
    on = rng.random(n) < spot
    xy[on] = rng.uniform(-15, 15, (on.sum(), 2)) + (300.0, 250.0)
    return J.compose(np.concatenate([rng.uniform(0, 6.28, (n, 1)), xy], 1).astype(np.float32))


def _check(cuda, cde, oc, item, oitem, mats, capacity=12):
    n = len(mats)
    out = (torch.full((n + 8,), -7, dtype=torch.int32, device=cuda), torch.full((n + 8,), -7, dtype=torch.int64, device=cuda),
           torch.full((n + 8, capacity), -7, dtype=torch.int32, device=cuda))
    cde.collect_batch(item, torch.from_numpy(mats).to(cuda), capacity=capacity, out=tuple(t[:n] for t in out))
    ref = O.query(oc, oitem, mats=mats, mode=2, keys_cap=capacity, threads=8)
    got = [t.cpu().numpy() for t in out]
    np.testing.assert_array_equal(got[0][:n].astype(np.uint32), ref["count"])
    np.testing.assert_array_equal(got[1][:n].view(np.uint64), ref["hash"])
    np.testing.assert_array_equal(got[2][:n].view(np.uint32), ref["keys"])
    assert all((g[n:] == -7).all() for g in got), "written past the batch"
    return ref["count"]


@pytest.mark.parametrize("n,spot", [(1, 1.0), (64, 1.0), (65, 0.5), (3000, 0.2), (64 * WAVES // 2 + 1, 0.02), (64 * WAVES + 1, 0.01)])
def test_some_queries_left(cuda, cluster, n, spot):
    cde, _, oc = cluster
    (item,), (oitem,) = items([S.polygon(90, 6, 6, 8.0, 12.0, 0)])
    count = _check(cuda, cde, oc, item, oitem, _mats(n, n, spot))
    assert (count > 16).sum() >= min(n * spot * 0.3, 500)


def test_shallow_virtual_roots(cuda):
    """More candidates than a query's list (8) but not than its set (16): across the middle lines the
    virtual root is the root, and the whole wave scans its entries for containment."""
    sc = S.config2_scene(seed=71, n_items=300)
    cde, _, oc = engines(sc)
    w, h = float(sc.container[:, 0].max()), float(sc.container[:, 1].max())
    (item,), (oitem,) = items([S.polygon(91, 24, 24, 60.0, 140.0, 2)])
    rng = np.random.default_rng(8)
    for n in (1, 700, 9000):
        xy = np.where(rng.random((n, 1)) < 0.5, np.stack([np.full(n, w / 2), rng.uniform(0, h, n)], 1), rng.uniform((0, 0), (w, h), (n, 2)))
        mats = J.compose(np.concatenate([rng.uniform(0, 6.28, (n, 1)), xy], 1).astype(np.float32))
        _check(cuda, cde, oc, item, oitem, mats)


@pytest.mark.parametrize("spread", [True, False])
def test_time_of_a_batch(cuda, cluster, spread):
    """64 queries, each with more hazards than the collector holds, take a few times as long as the
    slowest of them, as they are spread over waves (in one wave they took up to 62 times as long)."""
    if spread:                                           # every query: a large item over a full sheet
        sc = S.config2_scene(seed=2, n_items=2000)
        cde, _ = S.build_cde(sc)
        item = S.make_items([S.polygon(76, 24, 24, 200.0, 400.0, 2)])[0]
        mats = J.compose(S.transforms(141, 64, (0.0, 0.0, float(sc.container[:, 0].max()), float(sc.container[:, 1].max())), 0))
    else:                                                # queries on the cluster
        cde = cluster[0]
        item = S.make_items([S.polygon(90, 6, 6, 8.0, 12.0, 0)])[0]
        mats = _mats(3, 64, 1.0)

    def best(m):
        t = []
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            cde.collect_batch(item, m, capacity=0)
            b.record()
            b.synchronize()
            t.append(a.elapsed_time(b))
        return min(t)

    m = torch.from_numpy(mats).to(cuda)
    one = max(best(m[i:i + 1].contiguous()) for i in range(0, 64, 8))
    assert best(m) < 6.0 * one
