"""The sharing-out of work units and survivor groups (jg_plan.hpp) where its branches meet: a
workgroup per item or claims, fewer workgroups than counter streams, and launch after launch on
one table (the group counts alternate between two sets), against the oracle."""
import numpy as np
import pytest
import torch

import jagua_amd as J
from jagua_amd import synth as S
from oracle import oracle as O

from helpers import engines, items

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def layout():
    sc = S.config2_scene(seed=91, n_items=250)
    cde, _, oc = engines(sc)
    polys = [S.polygon(92 + i, nv, nv, 10.0, 30.0, 2) for i, nv in enumerate((9, 70, 400))]
    prod, orc = items(polys)
    box = (0.0, 0.0, float(sc.container[:, 0].max()), float(sc.container[:, 1].max()))
    return cde, oc, prod, orc, box


@pytest.mark.parametrize("n,workgroups,stages", [(1, 0, 2), (700, 0, 2), (700, 1, 2), (700, 15, 2), (700, 16, 2), (700, 17, 2),
                                                 (700, 3, 1), (30000, 0, 2), (30000, 333, 2)])
def test_every_item_is_taken(cuda, layout, n, workgroups, stages):
    cde, oc, prod, orc, box = layout
    sets = [(cde, it, i * n, n, None) for i, it in enumerate(prod)]
    plan = J.QueryPlan(sets, workgroups=workgroups, stages=stages)
    m = torch.empty((3 * n, 6), dtype=torch.float32, device=cuda)
    out = torch.empty(3 * n, dtype=torch.uint8, device=cuda)
    for rnd in range(4):
        mats = [J.compose(S.transforms(93 + 7 * rnd + i, n, box, 0)) for i in range(3)]
        m.copy_(torch.from_numpy(np.concatenate(mats)))
        out.fill_(99)
        plan.detect(m, out)
        ref = [O.query(oc, o, mats=mt, mode=3 if rnd == 2 else 1, threads=8) for o, mt in zip(orc, mats)]
        np.testing.assert_array_equal(out.cpu().numpy(), np.concatenate([r["status"] for r in ref]))
        if rnd == 2:                                     # the collection between two detections
            cnt, hsh, _ = plan.collect(m, capacity=0)
            np.testing.assert_array_equal(cnt.cpu().numpy().astype(np.uint32), np.concatenate([r["count"] for r in ref]))
            np.testing.assert_array_equal(hsh.cpu().numpy().view(np.uint64), np.concatenate([r["hash"] for r in ref]))


@pytest.mark.parametrize("item", [1, 2])
def test_noalloc_takes_what_its_scratch_was_sized_for(cuda, layout, item):
    """33 B of table per 4 queries (a unit per 64, a group per 2), whatever lanes the default
    schedule would give the item: about 4.066 million queries fit 32 MiB."""
    cde, oc, prod, orc, box = layout
    cde.sync()
    base = J.compose(S.transforms(97, 40000, box, 0))
    n = 4_064_000
    m = torch.from_numpy(base).to(cuda).repeat(n // 40000 + 1, 1)[:4_069_000].contiguous()
    out = torch.full((4_069_000,), 99, dtype=torch.uint8, device=cuda)
    with pytest.raises(J.JaguaError, match="scratch"):
        J.detect_sets_noalloc([(cde, prod[item], 0, 4_069_000, None)], m, out)
    J.detect_sets_noalloc([(cde, prod[item], 0, n, None)], m, out)
    ref = O.query(oc, orc[item], mats=base, mode=1, threads=8)["status"]
    got = out.cpu().numpy()
    np.testing.assert_array_equal(got[:n], np.tile(ref, n // 40000 + 1)[:n])
    assert (got[n:] == 99).all()


@pytest.mark.parametrize("item,n_sets,chunk,most", [(0, 1, 0, 7894076), (1, 1, 0, 4066590), (2, 1, 0, 4066302),
                                                    (2, 3, 0, 4066204), (2, 1, 16, 3727422)])
def test_noalloc_limit_to_the_query(cuda, layout, item, n_sets, chunk, most):
    """The largest call that the fixed scratch takes is part of the interface: descriptors, the item's
    record, a unit per 64 queries (or the chunk) and a group per 8 or 2, whatever form the table has."""
    cde, oc, prod, orc, box = layout
    cde.sync()
    m = torch.zeros((most + 1, 6), dtype=torch.float32, device=cuda)
    out = torch.empty(most + 1, dtype=torch.uint8, device=cuda)

    def call(n):
        per = n // n_sets
        J.detect_sets_noalloc([(cde, prod[item], k * per, per if k < n_sets - 1 else n - per * k, None) for k in range(n_sets)],
                              m, out, chunk=chunk)

    call(most)
    with pytest.raises(J.JaguaError, match="scratch"):
        call(most + 1)
    torch.cuda.synchronize()
