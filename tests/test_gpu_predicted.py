"""Large levels whose cut is found from a sampled window (builds without a
trace): exact against the CPU oracle, bit for bit, on even, clustered, ordered
and tied keys, and where the sample misses."""
import numpy as np
import pytest
from gpu_helpers import assert_heaps_equal, fbits

import inputs

pytestmark = pytest.mark.gpu

N = 16800011  # a build large enough for predicted windows


def check(orb, oracle, xyz, d, cmp=0, ids=False):
    n = len(xyz[0])
    with orb.Context(n, d, generate=False) as ctx:
        ctx.set_semantics(cmp, 0)
        ctx.set_particles(*xyz)
        if ids:
            ctx.enable_ids()
        ctx.save_particles()
        r = oracle.build(*xyz, d, levels_mode=1, cmp=cmp, ids=ids, threads=8)
        for _ in range(2):  # captured, then replayed
            ctx.restore_particles()
            try:
                info = ctx.build(orb.FORM_BATCHED, orb.LEVELS_FULL)
            except orb.OrbError as e:
                assert (e.code, e.error_cell) == (r.rc, r.error_cell)
                continue
            assert r.rc == 0
            assert info["level_passes"] == list(r.level_passes)
            assert np.array_equal(ctx.exists(), r.exists)
            assert_heaps_equal(ctx.heap(), r.heap, r.exists)
            assert np.array_equal(ctx.ranges(), r.ranges)
            for a, b in zip(ctx.get_particles(), (r.x, r.y, r.z)):
                assert np.array_equal(fbits(a), fbits(b))
            if ids:
                assert np.array_equal(ctx.ids(), r.ids)


# d = 128: cells from the whole set down to 131000 keys (every number of sample
# lines a chunk); 37: uneven shares
@pytest.mark.parametrize("d", [128, 37])
@pytest.mark.parametrize("cmp", [0, 1])
@pytest.mark.parametrize("keys", ["uniform", "clustered", "sorted", "reversed", "grid", "far"])
def test_keys(orb, oracle, keys, cmp, d):
    rng = np.random.default_rng(7)
    if keys == "clustered":
        xyz = inputs.clustered(N, n_spheres=11, a=0.003, seed=4)
    elif keys == "grid":  # many keys tie at a cut (few levels: the cells keep several values)
        xyz, d = inputs.quantized(N, levels=300, seed=2), 32
    else:
        xyz = tuple((rng.random(N, np.float32) - np.float32(0.5)) for _ in range(3))
        if keys in ("sorted", "reversed"):
            xyz = tuple(np.sort(a)[:: -1 if keys == "reversed" else 1].copy() for a in xyz)
        elif keys == "far":  # the cut lies a few floats from the first midpoint
            xyz = tuple((a * np.float32(2.0 ** -20)).astype(np.float32) for a in xyz)
    check(orb, oracle, xyz, d, cmp=cmp, ids=keys == "uniform")


# every sampled line of the root level holds keys far from the rest: the counts
# contradict the window, and the levels run again
def test_sample_misses(orb, oracle):
    x, y, z = oracle.generate(N)
    for q in range(N // 4096):
        p = 4096 * q + ((((q * 0x9E3779B1) & 0xFFFFFFFF) >> 20) & 4095 & ~63)
        x[p:p + 64] = np.float32(-0.45)
    check(orb, oracle, (x, y, z), 64, ids=True)
