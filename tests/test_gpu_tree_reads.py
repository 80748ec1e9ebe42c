"""Reading a built tree back, in parts and in any order."""
import itertools

import numpy as np
import pytest
from gpu_helpers import assert_heaps_equal

pytestmark = pytest.mark.gpu


# 8192 slots: above the size at which the ranges bring the whole tree
@pytest.mark.parametrize("d", [16, 4096])
def test_ranges_leave_the_trace(orb, oracle, d):
    """Reading the ranges reads no pass counts: with the trace off again they are
    not there, as after reading nothing."""
    n = 100 * d
    with orb.Context(n, d) as ctx:
        ctx.enable_trace(True)
        ctx.build(orb.FORM_BATCHED, orb.LEVELS_FULL)
        want = oracle.build(*oracle.generate(n), d, levels_mode=1)
        assert np.array_equal(ctx.ranges(), want.ranges)
        ctx.enable_trace(False)
        with pytest.raises(orb.OrbError) as e:
            ctx.pass_counts()
        assert e.value.code == orb.ERR_STATE


@pytest.mark.parametrize("d", [16, 4096])
def test_reads_in_any_order(orb, oracle, d):
    n = 100 * d
    want = oracle.build(*oracle.generate(n), d, levels_mode=1)
    root = np.zeros((len(want.ranges), 2), np.uint32)
    root[0, 1] = n
    with orb.Context(n, d) as ctx:
        ctx.save_particles()
        for order in itertools.permutations(("ranges", "heap", "exists")):
            ctx.restore_particles()
            assert np.array_equal(ctx.ranges(), root)
            ctx.build(orb.FORM_BATCHED, orb.LEVELS_FULL)
            for what in order + ("ranges",):
                if what == "ranges":
                    assert np.array_equal(ctx.ranges(), want.ranges)
                elif what == "heap":
                    assert_heaps_equal(ctx.heap(), want.heap, want.exists)
                else:
                    assert np.array_equal(ctx.exists(), want.exists)
            ctx.reset_ranges()
            assert np.array_equal(ctx.ranges(), root)
            # a service call that moves ranges
            cells = ctx.heap()[:1].copy()
            ctx.partition(cells)
            moved = ctx.ranges()
            assert moved[1, 1] == moved[2, 0] and moved[2, 1] == n and 0 < moved[1, 1] < n
