"""Boxes, edges and queries that lie partly or wholly outside the engine's box: the start cells on the
CPU (tests/outside_cells_check.cpp) and the collections against the oracle, bit for bit."""
import os
import subprocess

import numpy as np
import pytest
import torch

import jagua_amd as J
from jagua_amd import synth as S
from oracle import oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BOX = np.array([0.0, 0.0, 100.0, 100.0], np.float32)


def _ring(x0, y0, x1, y1):
    return np.array([[x0, y0], [x1, y0], [x1, y1], [x0, y1]], np.float32)


def _engines(hazards, depth=7, threshold=16):
    """Product and oracle engines of static hazards [(kind, vertices)] over BOX, after its exterior."""
    haz = [(O.KIND_EXTERIOR, _ring(*BOX))] + hazards
    cde = J.CDEngine(BOX, [J.Hazard(J.HazardEntity(k, i), J.SPolygon.new(v), False) for i, (k, v) in enumerate(haz)],
                     J.CDEConfig(depth, threshold, J.SPSurrogateConfig()))
    return cde, O.OracleCDE.from_hazards(BOX, depth, threshold, [(k, i, 0, v) for i, (k, v) in enumerate(haz)])


def _mats(xy, rot=None):
    xy = np.asarray(xy, np.float32)
    r = np.zeros(len(xy), np.float32) if rot is None else np.asarray(rot, np.float32)
    return J.compose(np.concatenate([r[:, None], xy], 1).astype(np.float32))


def _check_sets(cuda, cde, oc, poly, mats, capacity=8):
    """collect_batch and QueryPlan.collect of one item against the oracle."""
    item, oitem = S.make_items([poly])[0], O.OracleItem(poly)
    m = torch.from_numpy(np.ascontiguousarray(mats)).to(cuda)
    ref = O.query(oc, oitem, mats=mats, mode=3, keys_cap=capacity, threads=8)
    plan = J.QueryPlan([(cde, item, 0, len(mats), None)])
    for cnt, hsh, keys in (cde.collect_batch(item, m, capacity=capacity), plan.collect(m, capacity=capacity)):
        np.testing.assert_array_equal(cnt.cpu().numpy().astype(np.uint32), ref["count"])
        np.testing.assert_array_equal(hsh.cpu().numpy().view(np.uint64), ref["hash"])
        np.testing.assert_array_equal(keys.cpu().numpy().view(np.uint32), ref["keys"])
    np.testing.assert_array_equal(cde.detect_batch(item, m).cpu().numpy(), ref["status"])
    return ref


def test_cells_outside_the_root_box(tmp_path):
    exe = tmp_path / "outside_cells_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "outside_cells_check.cpp"), "-o", str(exe)], check=True, capture_output=True)
    for seed in (1, 2):
        out = subprocess.run([str(exe), str(seed), "20000"], capture_output=True, text=True)
        assert out.returncode == 0, out.stdout + out.stderr
        ok, outside, inside, leave, cells, nans = out.stdout.split()
        assert ok == "ok" and int(outside) > 100000 and int(inside) > 50000
        assert int(leave) > 100000 and int(cells) > 20000 and int(nans) > 100000


@pytest.mark.gpu
def test_collection_from_the_root_outside(cuda):
    """A placed item hangs over the border, and queries lie between its arm and the border: their
    virtual root is the root, whose hazards they are tested against for containment."""
    arm = np.array([[-40, 0], [-30, 0], [-30, 40], [10, 40], [10, 60], [-40, 60]], np.float32)
    cde, oc = _engines([(O.KIND_HOLE, arm)])
    ref = _check_sets(cuda, cde, oc, _ring(-2, -2, 2, 2), _mats([[-35, 8], [-35, 30], [-20, 50], [-60, 8], [5, 50], [-1, 20]]))
    assert ref["count"].tolist()[:3] == [2, 2, 2]


@pytest.mark.gpu
def test_collection_of_edges_outside(cuda):
    """Queries in the notch of a hazard that reaches over the border, whose cells beside them are
    Entire: their edges, outside the box, reach no node (the root itself does not collect)."""
    notch = np.array([[-50, 20], [30, 20], [30, 80], [-50, 80], [-50, 60], [-2, 60], [-2, 40], [-50, 40]], np.float32)
    cde, oc = _engines([(O.KIND_HOLE, notch)], threshold=2)
    ref = _check_sets(cuda, cde, oc, _ring(-0.2, -0.2, 0.2, 0.2), _mats([[-8, 51.17], [-30, 48.83], [-2.5, 51.17], [-20, 30], [-1, 51.17]]))
    assert ref["count"].tolist()[:3] == [1, 1, 1]


@pytest.mark.gpu
@pytest.mark.parametrize("depth,nv,r", [(7, 5, 2.0), (7, 24, 12.0), (10, 9, 5.0), (3, 40, 40.0)])
def test_queries_around_the_border(cuda, depth, nv, r):
    """Hazards across every border and in the middle, queries in and around the box."""
    rng = np.random.default_rng(5 + depth)
    c = np.concatenate([np.stack([rng.uniform(0, 100, 6), rng.choice([0.0, 100.0], 6)], 1),
                        np.stack([rng.choice([0.0, 100.0], 6), rng.uniform(0, 100, 6)], 1), rng.uniform(0, 100, (6, 2))])
    cde, oc = _engines([(O.KIND_HOLE, S.polygon(60 + i, 5, 20, 3.0, 20.0, i % 3) + p.astype(np.float32)) for i, p in enumerate(c)], depth)
    n = 3000
    mats = _mats(rng.uniform(-60, 160, (n, 2)), rng.uniform(0, 6.28, n))
    ref = _check_sets(cuda, cde, oc, S.polygon(80 + nv, nv, nv, 0.5 * r, r, 2), mats)
    assert len(np.unique(ref["count"])) > 2
