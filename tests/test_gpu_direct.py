"""Batches of one item (detect_batch, collect_batch) against the oracle, bit for bit, at the
sizes where the queries per wave change and where the last wave's unit is ragged."""
import numpy as np
import pytest
import torch

import jagua_amd as J
from jagua_amd import synth as S
from oracle import oracle as O

from helpers import engines, items

pytestmark = pytest.mark.gpu

CUS16 = 256 * 16


@pytest.fixture(scope="module")
def sheet():
    sc = S.config2_scene(seed=71, n_items=300)
    return engines(sc) + (sc.container,)


@pytest.mark.parametrize("n", [1, 65, CUS16, CUS16 + 1, 2 * CUS16 + 3, 16 * CUS16 + 17])
@pytest.mark.parametrize("filt", ["none", "keys", "hashed"])
def test_detect_sizes(cuda, sheet, n, filt):
    cde, keys, oc, cont = sheet
    (item,), (oitem,) = items([S.polygon(72, 40, 40, 10.0, 30.0, 2)])
    mats = J.compose(S.transforms(73 + n, n, (0.0, 0.0, float(cont[:, 0].max()), float(cont[:, 1].max())), 0))
    hf = J.HashedFilter(5, 0.1)
    f, of = {"none": (None, None), "hashed": (hf, O.make_filter(2, hf.seed, hf.threshold)),
             "keys": (J.HazKeyFilter(keys[::4]), O.make_filter(1, keys=[k.idx for k in keys[::4]]))}[filt]
    out = torch.full((n + 64,), 99, dtype=torch.uint8, device=cuda)
    cde.detect_batch(item, torch.from_numpy(mats).to(cuda), f, out=out)
    ref = O.query(oc, oitem, mats=mats, mode=1, filt=of, threads=8)
    got = out.cpu().numpy()
    np.testing.assert_array_equal(got[:n], ref["status"])
    assert (got[n:] == 99).all(), "written past the batch"


@pytest.mark.parametrize("n,nv,filt", [(48 * CUS16, 24, False), (48 * CUS16 + 1, 24, True), (96 * CUS16 + 1, 64, True),
                                       (96 * CUS16 + 1, 65, False), (96 * CUS16 + 1, 65, True)])
def test_detect_full_waves(cuda, sheet, n, nv, filt):
    """16, 32 and 64 queries per wave; 16 at most for filtered queries of more than 64 vertices."""
    cde, keys, oc, cont = sheet
    (item,), (oitem,) = items([S.polygon(78, nv, nv, 10.0, 30.0, 2)])
    mats = J.compose(S.transforms(79, n, (0.0, 0.0, float(cont[:, 0].max()), float(cont[:, 1].max())), 0))
    out = torch.full((n + 8,), 99, dtype=torch.uint8, device=cuda)
    cde.detect_batch(item, torch.from_numpy(mats).to(cuda), J.HashedFilter(5, 0.1) if filt else None, out=out[:n])
    ref = O.query(oc, oitem, mats=mats, mode=1, filt=O.make_filter(2, 5, J.HashedFilter(5, 0.1).threshold) if filt else None, threads=8)
    got = out.cpu().numpy()
    np.testing.assert_array_equal(got[:n], ref["status"])
    assert (got[n:] == 99).all()


@pytest.mark.parametrize("n,nv,r", [(1, 40, 20.0), (5 * CUS16 // 4, 40, 20.0), (5 * CUS16 // 4 + 1, 12, 20.0),
                                    (40 * CUS16 // 4 + 3, 9, 15.0), (130, 24, 400.0)])
def test_collect_sizes(cuda, sheet, n, nv, r):
    """The last item covers more hazards than a query's collector holds (16): those queries are
    collected by the second launch."""
    cde, keys, oc, cont = sheet
    (item,), (oitem,) = items([S.polygon(76, nv, nv, 0.5 * r, r, 2)])
    mats = J.compose(S.transforms(77 + n, n, (0.0, 0.0, float(cont[:, 0].max()), float(cont[:, 1].max())), 0))
    out = (torch.full((n + 8,), -7, dtype=torch.int32, device=cuda), torch.full((n + 8,), -7, dtype=torch.int64, device=cuda),
           torch.full((n + 8, 20), -7, dtype=torch.int32, device=cuda))
    cde.collect_batch(item, torch.from_numpy(mats).to(cuda), capacity=20, out=tuple(t[:n] for t in out))
    ref = O.query(oc, oitem, mats=mats, mode=3, keys_cap=20, threads=8)
    got = [t.cpu().numpy() for t in out]
    np.testing.assert_array_equal(got[0][:n].astype(np.uint32), ref["count"])
    np.testing.assert_array_equal(got[1][:n].view(np.uint64), ref["hash"])
    np.testing.assert_array_equal(got[2][:n].view(np.uint32), ref["keys"])
    assert all((g[n:] == -7).all() for g in got), "written past the batch"
    assert r < 100.0 or (ref["count"] > 16).sum() > 20


def test_detect_captured(cuda, sheet):
    """One call captured and replayed on new transforms in the same buffer."""
    cde, keys, oc, cont = sheet
    (item,), (oitem,) = items([S.polygon(74, 12, 12, 10.0, 30.0, 2)])
    n = 5000
    m = torch.empty((n, 6), dtype=torch.float32, device=cuda)
    out = torch.empty(n, dtype=torch.uint8, device=cuda)
    s = torch.cuda.Stream()
    for k in range(3):
        mats = J.compose(S.transforms(75 + k, n, (0.0, 0.0, float(cont[:, 0].max()), float(cont[:, 1].max())), 0))
        m.copy_(torch.from_numpy(mats))
        torch.cuda.synchronize()
        if k == 0:
            cde.detect_batch(item, m, out=out)
            torch.cuda.synchronize()
            with J.Graph.capture(s) as g:
                cde.detect_batch(item, m, out=out, stream=s)
        out.fill_(99)
        torch.cuda.synchronize()
        g.launch()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out.cpu().numpy(), O.query(oc, oitem, mats=mats, mode=1, threads=8)["status"])
