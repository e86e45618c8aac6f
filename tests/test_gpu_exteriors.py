"""Engines with more than one hazard of exterior scope: each is met everywhere outside its shape, also far
from its box.  Detection and collection against the oracle, bit for bit."""
import numpy as np
import pytest
import torch

import jagua_amd as J
from jagua_amd import synth as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu

BOX = np.array([0.0, 0.0, 100.0, 100.0], np.float32)
SQUARE = np.array([[0, 0], [100, 0], [100, 100], [0, 100]], np.float32)


def _check(cuda, cde, oc, seed):
    rng = np.random.default_rng(seed)
    for nv, r, n in ((6, 2.0, 2000), (40, 15.0, 500)):
        poly = S.polygon(70 + nv, nv, nv, 0.5 * r, r, 2)
        item, oitem = S.make_items([poly])[0], O.OracleItem(poly)
        mats = J.compose(np.stack([rng.uniform(0, 6.28, n), rng.uniform(-5, 105, n), rng.uniform(-5, 105, n)], 1).astype(np.float32))
        m = torch.from_numpy(mats).to(cuda)
        ref = O.query(oc, oitem, mats=mats, mode=3, threads=8)
        plan = J.QueryPlan([(cde, item, 0, n, None)])
        for cnt, hsh, _ in (cde.collect_batch(item, m, capacity=0), plan.collect(m, capacity=0)):
            np.testing.assert_array_equal(cnt.cpu().numpy().astype(np.uint32), ref["count"])
            np.testing.assert_array_equal(hsh.cpu().numpy().view(np.uint64), ref["hash"])
        np.testing.assert_array_equal(cde.detect_batch(item, m).cpu().numpy(), ref["status"])
    return ref


def test_second_exterior(cuda):
    diamond = np.array([[60, 30], [90, 60], [60, 90], [30, 60]], np.float32)
    holes = [S.polygon(50 + i, 5, 12, 2.0, 6.0, 0) + np.float32(p) for i, p in enumerate(((15, 15), (70, 60), (40, 85)))]
    haz = [(1, SQUARE), (1, diamond)] + [(2, h) for h in holes]
    cde = J.CDEngine(BOX, [J.Hazard(J.HazardEntity(k, i), J.SPolygon.new(v), False) for i, (k, v) in enumerate(haz)],
                     J.CDEConfig(6, 4, J.SPSurrogateConfig()))
    oc = O.OracleCDE.from_hazards(BOX, 6, 4, [(k, i, 0, v) for i, (k, v) in enumerate(haz)])
    _check(cuda, cde, oc, 1)


def test_exterior_registered_later_and_taken_out(cuda):
    """The rule follows the registered hazards: a second exterior comes, and the first one goes."""
    cde = J.CDEngine(BOX, [J.Hazard(J.HazardEntity.exterior(), J.SPolygon.new(SQUARE), False)], J.CDEConfig(6, 2, J.SPSurrogateConfig()))
    oc = O.OracleCDE.from_hazards(BOX, 6, 2, [(1, 0, 0, SQUARE)])
    first = cde.hkey_exterior
    _check(cuda, cde, oc, 2)
    inner = np.array([[50, 50], [80, 50], [80, 80], [50, 80]], np.float32)
    cde.register_hazard(J.Hazard(J.HazardEntity(1, 7), J.SPolygon.new(inner), False))
    oc2 = O.OracleCDE.from_hazards(BOX, 6, 2, [(1, 0, 0, SQUARE), (1, 7, 0, inner)])
    _check(cuda, cde, oc2, 3)
    cde.deregister_hazard_by_key(first)
    oc2.deregister_key((first.idx, first.version))
    _check(cuda, cde, oc2, 4)
