"""The per-query detection kernel, which takes the engines and batches past the wave traversal's packed
formats (2^24 nodes, 2^29 hazard edges, 2^32 - 1 queries): too large to be met in a test, so
jg_check_detect_batch_plain calls it.  Against the oracle, bit for bit."""
import ctypes as C

import numpy as np
import pytest
import torch

import jagua_amd as J
from jagua_amd import _native as N
from jagua_amd import synth as S
from oracle import oracle as O

from helpers import engines, items

pytestmark = pytest.mark.gpu


def _plain(cde, item, m, filt, flags, out):
    f = (filt or J.NoFilter())._filter()
    fn = N.lib().jg_check_detect_batch_plain
    N.check(fn(cde._h, item._h, C.c_void_p(m.data_ptr()), C.c_uint64(m.shape[0]), C.byref(f), C.c_uint32(flags),
               C.c_void_p(out.data_ptr()), None))


@pytest.mark.parametrize("n", [1, 256, 4097])
@pytest.mark.parametrize("filt", ["none", "keys", "hashed"])
@pytest.mark.parametrize("piers", [0, 2])
def test_plain_kernel(cuda, n, filt, piers):
    sc = S.config2_scene(seed=71, n_items=300)
    cde, keys, oc = engines(sc)
    (item,), (oitem,) = items([S.polygon(72, 40, 40, 10.0, 30.0, 2)], n_ff_piers=piers)
    w, h = float(sc.container[:, 0].max()), float(sc.container[:, 1].max())
    mats = J.compose(S.transforms(73 + n, n, (-30.0, -30.0, w + 30.0, h + 30.0), 0))
    hf = J.HashedFilter(5, 0.1)
    f, of = {"none": (None, None), "hashed": (hf, O.make_filter(2, hf.seed, hf.threshold)),
             "keys": (J.HazKeyFilter(keys[::4]), O.make_filter(1, keys=[k.idx for k in keys[::4]]))}[filt]
    m = torch.from_numpy(mats).to(cuda)
    ref = O.query(oc, oitem, mats=mats, mode=1, filt=of, threads=8)
    out = torch.full((n + 300,), 99, dtype=torch.uint8, device=cuda)
    _plain(cde, item, m, f, 0, out)
    got = out.cpu().numpy()
    np.testing.assert_array_equal(got[:n], ref["status"])
    assert (got[n:] == 99).all(), "written past the batch"
    for flags in (1, 2):                                 # one stage alone: as the wave traversal answers
        _plain(cde, item, m, f, flags, out)
        np.testing.assert_array_equal(out.cpu().numpy()[:n], cde.detect_batch(item, m, f, flags).cpu().numpy())
