"""Stable-partition builds whose levels hold few chunks: partial last chunks,
the last size of the few-chunk kernels' tables and one key past it, every key
on one side, ties, ids, weights, both level modes, and a weighted cell of more
chunks than one table holds, against the CPU oracle, bit for bit."""
import numpy as np
import pytest
from gpu_helpers import assert_heaps_equal, fbits

import inputs

pytestmark = pytest.mark.gpu


def check(orb, oracle, xyz, d, levels=1, ids=False, w=None, graph=True):
    n = len(xyz[0])
    with orb.Context(n, d, generate=False) as ctx:
        ctx.set_semantics(1, 1)
        ctx.set_particles(*xyz)
        if ids:
            ctx.enable_ids()
        if w is not None:
            ctx.set_weights(w)
        ctx.enable_graph(graph)
        r = oracle.build(*xyz, d, levels_mode=levels, cmp=1, partition=1, weights=w, ids=ids, threads=8)
        try:
            info = ctx.build(orb.FORM_BATCHED, levels)
        except orb.OrbError as e:
            assert (e.code, e.error_cell) == (r.rc, r.error_cell)
            return
        assert r.rc == 0
        assert info["level_passes"] == list(r.level_passes)
        assert np.array_equal(ctx.exists(), r.exists)
        assert_heaps_equal(ctx.heap(), r.heap, r.exists)
        assert np.array_equal(ctx.ranges(), r.ranges)
        for a, b in zip(ctx.get_particles(), (r.x, r.y, r.z)):
            assert np.array_equal(fbits(a), fbits(b))
        if ids:
            assert np.array_equal(ctx.ids(), r.ids)
        if w is not None:
            assert np.array_equal(ctx.weights(), r.weights)


@pytest.mark.parametrize("n,d", [(1, 1), (300, 2), (4096, 3), (4097, 8), (70001, 64), (2097148, 2),
                                 (2097149, 2), (131072, 1024)])
@pytest.mark.parametrize("levels", [0, 1])
@pytest.mark.parametrize("weighted", [False, True])
def test_few_chunks(orb, oracle, n, d, levels, weighted):
    w = np.random.default_rng(n).integers(1, 9, n).astype(np.uint32) if weighted else None
    check(orb, oracle, inputs.clustered(n, n_spheres=7, a=0.04, seed=d), d, levels, ids=n < 100000, w=w,
          graph=levels == 1)


@pytest.mark.parametrize("keys", ["grid", "one_value", "sorted"])
def test_ties(orb, oracle, keys):
    n = 150001
    if keys == "grid":
        xyz = inputs.quantized(n, levels=9, seed=3)
    elif keys == "sorted":
        xyz = tuple(np.sort(a) for a in oracle.generate(n))
    else:
        xyz = (np.full(n, 0.125, np.float32),) + oracle.generate(n)[1:]
    check(orb, oracle, xyz, 8, ids=True)


# nearly all the weight on a thousandth of the keys: the cells of the levels
# below the root hold up to 3.9M keys where half a million is expected
def test_cell_of_several_tables(orb, oracle):
    n = 3900001
    xyz = oracle.generate(n)
    w = np.ones(n, np.uint32)
    w[(xyz[0] < np.float32(-0.499))] = 100000
    check(orb, oracle, xyz, 16, w=w)


@pytest.mark.parametrize("n,d", [(9000001, 40), (17000003, 300)])
@pytest.mark.parametrize("weighted", [False, True])
def test_many_chunks(orb, oracle, n, d, weighted):
    w = np.random.default_rng(n).integers(1, 9, n).astype(np.uint32) if weighted else None
    check(orb, oracle, inputs.clustered(n, n_spheres=7, a=0.04, seed=d), d, w=w)
