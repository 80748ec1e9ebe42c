"""Levels whose cells one block takes whole (keys in registers), and levels of
few chunks: sizes at the edges of their capacities, of the waves' parts, of
the 64-key rows and of the chunks, both block shapes, ids, ties, and cells
larger than the level expected, against the CPU oracle, bit for bit."""
import numpy as np
import pytest
from gpu_helpers import assert_heaps_equal, bin_edge_keys, fbits

import inputs

pytestmark = pytest.mark.gpu


def check(orb, oracle, xyz, d, cmp=0, ids=False, subtree=None):
    n = len(xyz[0])
    with orb.Context(n, d, generate=False) as ctx:
        ctx.set_semantics(cmp, 0)
        ctx.set_particles(*xyz)
        if ids:
            ctx.enable_ids()
        if subtree is not None:
            ctx.set_tuning({"subtree_max_keys": subtree})
        ctx.enable_trace(True)
        r = oracle.build(*xyz, d, levels_mode=1, cmp=cmp, pass_counts=True, ids=ids)
        try:
            info = ctx.build(orb.FORM_BATCHED, orb.LEVELS_FULL)
        except orb.OrbError as e:
            assert (e.code, e.error_cell) == (r.rc, r.error_cell)
            return False
        assert r.rc == 0
        assert info["level_passes"] == list(r.level_passes)
        assert np.array_equal(ctx.exists(), r.exists)
        assert_heaps_equal(ctx.heap(), r.heap, r.exists)
        assert np.array_equal(ctx.ranges(), r.ranges)
        assert np.array_equal(ctx.pass_counts(), r.pass_counts)
        for a, b in zip(ctx.get_particles(), (r.x, r.y, r.z)):
            assert np.array_equal(fbits(a), fbits(b))
        if ids:
            assert np.array_equal(ctx.ids(), r.ids)
    return True


# the root's size: 1 past the subtree kernel's, around a wave part's end
# (multiples of 4096 and of 64), the two capacities less what the level rule
# keeps free, and just past them (the chunk path)
@pytest.mark.parametrize("n", [8833, 12288, 12289, 16383, 20476, 20477, 24641, 40955, 40956, 40957])
@pytest.mark.parametrize("cmp", [0, 1])
def test_one_cell(orb, oracle, n, cmp):
    assert check(orb, oracle, inputs.clustered(n, n_spheres=5, a=0.05, seed=n), 2, cmp=cmp, ids=True)


# levels of few chunks: partial last chunks, one chunk more or less, the largest
# cell of their tables (512 chunks less what the level rule keeps free) and one past it
@pytest.mark.parametrize("n,d", [(40961, 2), (65537, 3), (8 * 4096 * 64 - 1, 5), (2097148, 2), (2097149, 2),
                                 (1500007, 30)])
@pytest.mark.parametrize("cmp", [0, 1])
def test_few_chunks(orb, oracle, n, d, cmp):
    assert check(orb, oracle, inputs.clustered(n, n_spheres=9, a=0.03, seed=d), d, cmp=cmp, ids=n < 100000)


# no subtree kernel: every level of every size, down to cells of two leaves of
# a few keys; d = 1024 has more than 256 cells on its last levels
@pytest.mark.parametrize("n,d", [(1, 1), (300, 2), (5000, 7), (70001, 64), (131072, 1024), (200003, 1000)])
def test_every_level(orb, oracle, n, d):
    assert check(orb, oracle, oracle.generate(n), d, ids=True, subtree=0)


# the half-sized subtree blocks: their largest cell, a key more, partial
# 64-key pieces, and cells below
@pytest.mark.parametrize("n,d", [(4224, 64), (4225, 64), (8440, 32), (4161, 3), (100003, 1000), (513, 8)])
@pytest.mark.parametrize("cmp", [0, 1])
def test_half_subtree_blocks(orb, oracle, n, d, cmp):
    assert check(orb, oracle, inputs.clustered(n, n_spheres=5, a=0.05, seed=n), d, cmp=cmp, subtree=4224)


@pytest.mark.parametrize("keys", ["grid", "edges", "one_value", "sorted"])
@pytest.mark.parametrize("cmp", [0, 1])
@pytest.mark.parametrize("n", [30011, 150001])
def test_ties(orb, oracle, keys, cmp, n):
    rng = np.random.default_rng(5)
    if keys == "grid":
        xyz = inputs.quantized(n, levels=9, seed=3)
    elif keys == "edges":
        xyz = tuple(bin_edge_keys(n, rng) for _ in range(3))
    elif keys == "sorted":  # the window's keys lie side by side
        xyz = tuple(np.sort(a) for a in oracle.generate(n))
    else:  # every x the same: one side of the first cut is empty
        xyz = (np.full(n, 0.125, np.float32),) + oracle.generate(n)[1:]
    check(orb, oracle, xyz, 8, cmp=cmp, subtree=0)


# x holds one value in most particles: the first split is uneven, its larger
# child exceeds what its level expected (on a level without chunk kernels) and
# the build is finished by a second run of the levels
@pytest.mark.parametrize("n,d,subtree", [(75000, 4, None), (17000, 4, None), (75000, 4, 0)])
def test_larger_than_expected(orb, oracle, n, d, subtree):
    x, y, z = oracle.generate(n)
    x[np.random.default_rng(2).random(n) < 0.7] = np.float32(0.21)
    assert check(orb, oracle, (x, y, z), d, ids=True, subtree=subtree)


# weighted builds on levels of few chunks: even weights, many zeros, and a few
# heavy particles (cells of very uneven sizes; with 3 of them a cell outgrows
# the tables of a level of few chunks and the levels run again)
@pytest.mark.parametrize("n,d,kind", [(5121, 2, "even"), (40961, 8, "even"), (150001, 24, "zeros"),
                                      (150001, 8, "grid"), (1000003, 16, "heavy"), (2000003, 8, "three")])
@pytest.mark.parametrize("cmp", [0, 1])
def test_weighted_few_chunks(orb, oracle, n, d, kind, cmp):
    rng = np.random.default_rng(n)
    x, y, z = inputs.quantized(n, levels=64, seed=1) if kind == "grid" else oracle.generate(n)
    w = rng.integers(1, 1000, n).astype(np.uint32)
    if kind == "zeros":
        w[rng.random(n) < 0.9] = 0
    elif kind in ("heavy", "three"):
        w[:] = 1
        w[rng.integers(0, n, 3 if kind == "three" else 50)] = 1 << 24
    with orb.Context(n, d, generate=False) as ctx:
        ctx.set_semantics(cmp, 0)
        ctx.set_particles(x, y, z)
        ctx.enable_ids()
        ctx.set_weights(w)
        ctx.enable_trace(True)
        r = oracle.build(x, y, z, d, levels_mode=1, cmp=cmp, ids=True, weights=w, pass_weights=True)
        try:
            info = ctx.build(orb.FORM_BATCHED, orb.LEVELS_FULL)
        except orb.OrbError as e:
            assert (e.code, e.error_cell) == (r.rc, r.error_cell)
            return
        assert r.rc == 0
        assert info["level_passes"] == list(r.level_passes)
        assert_heaps_equal(ctx.heap(), r.heap, r.exists)
        assert np.array_equal(ctx.ranges(), r.ranges)
        assert np.array_equal(ctx.pass_weights(), r.pass_weights)
        for a, b in zip(ctx.get_particles(), (r.x, r.y, r.z)):
            assert np.array_equal(fbits(a), fbits(b))
        assert np.array_equal(ctx.ids(), r.ids)
        assert np.array_equal(ctx.weights(), r.weights)


# levels of many chunks whose cells still fit the few-chunk kernels' tables
@pytest.mark.parametrize("n,d", [(9000001, 40), (17000003, 300)])
@pytest.mark.parametrize("cmp", [0, 1])
def test_many_chunks(orb, oracle, n, d, cmp):
    assert check(orb, oracle, inputs.clustered(n, n_spheres=9, a=0.03, seed=d), d, cmp=cmp)
