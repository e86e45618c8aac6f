"""The pole searches on the device to their end: what they finish without the host routine, and full
cell trees, which are emptied in the middle of a polygon's searches, bit for bit with the host
construction.  No polygon fills the library's trees (24576 blocks of 4 nodes) before its frontier
overflows, so jg_check_spolygon_new_batch runs the same kernels with smaller ones."""
import concurrent.futures as cf
import ctypes as C

import numpy as np
import pytest

import jagua_amd as J
from jagua_amd import _native as N
from jagua_amd import synth as S

pytestmark = pytest.mark.gpu


def _fixed(n):
    return J.SPSurrogateConfig(((n, 0.0), (n, 0.0), (n, 0.0)), n_ff_poles=2)


def _arc(n, r0, r1):
    a = np.linspace(0.05, 2.0 * np.pi - 0.05, n)
    out = np.stack([r1 * np.cos(a), r1 * np.sin(a)], 1)
    inn = np.stack([r0 * np.cos(a[::-1]), r0 * np.sin(a[::-1])], 1)
    return np.concatenate([out, inn]).astype(np.float32)


def _check(got, polys, cfg):
    with cf.ThreadPoolExecutor(8) as ex:
        ref = list(ex.map(lambda p: J.SPolygon.new(p).generate_surrogate(cfg), polys))
    for g, r in zip(got, ref):
        np.testing.assert_array_equal(g.poles.view(np.uint32), r.poles.view(np.uint32))
        np.testing.assert_array_equal(np.array(g.info().poi[:], np.float32).view(np.uint32),
                                      np.array(r.info().poi[:], np.float32).view(np.uint32))


def _with_trees_of(blocks, polys, cfg):
    """(polygons, finished by the host routine, trees emptied)"""
    off = np.zeros(len(polys) + 1, np.uint32)
    off[1:] = np.cumsum([len(p) for p in polys])
    xy = np.ascontiguousarray(np.concatenate(polys), np.float32)
    hs, n_host, n_emptied, c = (C.c_void_p * len(polys))(), C.c_uint32(), C.c_uint32(), cfg._c()
    N.check(N.lib().jg_check_spolygon_new_batch(xy.ctypes.data_as(C.c_void_p), off.ctypes.data_as(C.c_void_p), C.c_uint32(len(polys)),
                                                C.byref(c), hs, C.byref(n_host), C.c_uint32(blocks), C.byref(n_emptied)))
    return [J.SPolygon(h) for h in hs], n_host.value, n_emptied.value


@pytest.mark.parametrize("polys,cfg,n_host", [
    ([S.polygon(82, 2049, 2049, 20.0, 30.0, 0), S.polygon(83, 10, 10, 10.0, 20.0, 0)], _fixed(3), 0),
    # levels of up to 8068 and 6076 new cells (the list of new cells holds 1024, a frontier 8192)
    ([_arc(60, 85.0, 100.0), _arc(40, 60.0, 100.0)], _fixed(4), 0),
    # a level of 8636: finished by the host routine
    ([_arc(60, 90.0, 100.0)], _fixed(2), 1),
    ([S.polygon(8400 + i, 3 + i % 14, 3 + i % 14, 5.0, 15.0, 0) for i in range(513)], _fixed(4), 0),
])
def test_finished_on_the_device(cuda, polys, cfg, n_host):
    got, n = J.SPolygon.new_batch(polys, cfg)
    assert n == n_host
    _check(got, polys, cfg)


@pytest.mark.parametrize("blocks", [1, 1800, 2500, 24576])
@pytest.mark.parametrize("n_small", [0, 520])
def test_full_trees(cuda, blocks, n_small):
    """Trees of one block hold no search at all; those of 1800 and 2500 fill up over a
    polygon's 100 searches (both workgroup sizes)."""
    cfg = _fixed(100)
    polys = [S.polygon(83, 10, 10, 10.0, 20.0, 0), S.polygon(84, 40, 40, 10.0, 20.0, 0)]
    polys += [np.array([[0, 0], [4, 0], [4, 3 + 0.01 * i], [0, 3]], np.float32) for i in range(n_small)]
    if n_small:
        cfg = _fixed(30)
    got, n_host, n_emptied = _with_trees_of(blocks, polys, cfg)
    print(blocks, n_small, "host", n_host, "emptied", n_emptied)
    if blocks == 1:
        assert n_host == len(polys) and n_emptied == len(polys)
    elif blocks == 24576:
        assert n_host == 0 and n_emptied == 0
    elif blocks == 1800 or not n_small:
        assert n_host == 0 and n_emptied >= 2
    _check(got, polys, cfg)


@pytest.mark.parametrize("blocks", [0, 24577])
def test_tree_sizes_out_of_range(cuda, blocks):
    with pytest.raises(J.JaguaError, match="out of range"):
        _with_trees_of(blocks, [S.polygon(83, 10, 10, 10.0, 20.0, 0)], _fixed(2))
