"""Transforms with NaN, infinite, huge and tiny entries through every query form, against the oracle,
bit for bit (but for the transforms on which the reference would panic)."""
import numpy as np
import pytest
import torch

import jagua_amd as J
from jagua_amd import synth as S
from oracle import oracle as O

from helpers import engines, items

pytestmark = pytest.mark.gpu

VALUES = np.array([np.nan, np.inf, -np.inf, 3e38, -3e38, 1e30, 1e-40, 0.0], np.float32)


@pytest.mark.parametrize("nv", [5, 40])
def test_non_finite_transforms(cuda, nv):
    sc = S.config2_scene(seed=71, n_items=300)
    cde, _, oc = engines(sc)
    (item,), (oitem,) = items([S.polygon(76, nv, nv, 10.0, 30.0, 2)])
    rng = np.random.default_rng(3 + nv)
    mats = J.compose(S.transforms(7, 1500, (0.0, 0.0, float(sc.container[:, 0].max()), float(sc.container[:, 1].max())), 0)).copy()
    for row in mats:
        k = rng.integers(1, 4)
        row[rng.choice(6, k, replace=False)] = VALUES[rng.integers(len(VALUES), size=k)]
    keep, ref = [], []
    for i in range(len(mats)):
        try:
            ref.append(O.query(oc, oitem, mats=mats[i:i + 1], mode=3))
        except RuntimeError:
            continue
        keep.append(i)
    status, count, hashes = (np.concatenate([r[k] for r in ref]) for k in ("status", "count", "hash"))
    assert len(keep) > 700 and len(np.unique(count)) > 4
    mats = np.ascontiguousarray(mats[keep])
    m = torch.from_numpy(mats).to(cuda)
    plan = J.QueryPlan([(cde, item, 0, len(mats), None)])
    out = torch.empty(len(mats), dtype=torch.uint8, device=cuda)
    plan.detect(m, out)
    np.testing.assert_array_equal(out.cpu().numpy(), status)
    np.testing.assert_array_equal(cde.detect_batch(item, m).cpu().numpy(), status)
    for cnt, hsh, _ in (cde.collect_batch(item, m, capacity=0), plan.collect(m, capacity=0)):
        np.testing.assert_array_equal(cnt.cpu().numpy().astype(np.uint32), count)
        np.testing.assert_array_equal(hsh.cpu().numpy().view(np.uint64), hashes)
