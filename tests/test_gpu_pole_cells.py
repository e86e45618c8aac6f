"""The pole searches' cell tree (jg_spolygon_new_batch) against the host construction, bit for
bit, where the kernel's ranges end: vertices and poles past the part held in local memory, more
new cells on a level than its list holds, and both workgroup sizes."""
import concurrent.futures as cf

import numpy as np
import pytest

import jagua_amd as J
from jagua_amd import synth as S

pytestmark = pytest.mark.gpu


def _arc(n, r0, r1):
    """A ring open at one end: every point of its middle line is as far from the border, so the
    first search keeps cells along all of it."""
    a = np.linspace(0.05, 2.0 * np.pi - 0.05, n)
    out = np.stack([r1 * np.cos(a), r1 * np.sin(a)], 1)
    inn = np.stack([r0 * np.cos(a[::-1]), r0 * np.sin(a[::-1])], 1)
    return np.concatenate([out, inn]).astype(np.float32)


def _fixed(n):
    return J.SPSurrogateConfig(((n, 0.0), (n, 0.0), (n, 0.0)), n_ff_poles=2)


CASES = {
    "triangle": ([np.array([[0, 0], [5, 0], [1, 7]], np.float32)], None),
    "vertices_2048": ([S.polygon(81, 2048, 2048, 20.0, 30.0, 0)], _fixed(3)),
    "vertices_2049": ([S.polygon(82, 2049, 2049, 20.0, 30.0, 0)], _fixed(3)),
    "poles_140": ([S.polygon(83, 10, 10, 10.0, 20.0, 0)], _fixed(140)),
    "new_cells": ([_arc(60, 90.0, 100.0), _arc(40, 60.0, 100.0)], _fixed(6)),
    "many": ([S.polygon(8400 + i, 3 + i % 14, 3 + i % 14, 5.0, 15.0, 0) for i in range(513)], _fixed(4)),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_pole_searches_match_host(cuda, name):
    polys, cfg = CASES[name]
    got, n_host = J.SPolygon.new_batch(polys, cfg)
    print(name, "finished on the host:", n_host)
    with cf.ThreadPoolExecutor(8) as ex:
        ref = list(ex.map(lambda p: J.SPolygon.new(p).generate_surrogate(cfg), polys))
    for g, r in zip(got, ref):
        np.testing.assert_array_equal(g.poles.view(np.uint32), r.poles.view(np.uint32))
        np.testing.assert_array_equal(np.array(g.info().poi[:], np.float32).view(np.uint32),
                                      np.array(r.info().poi[:], np.float32).view(np.uint32))
