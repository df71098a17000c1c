"""The order in which the kernels of a call enter a stream's queue, without a GPU (tests/launch_log.py)."""
import pytest

from tests.launch_log import record
from tests.test_merge_launch_gpu import MERGING

# launches in several parts with a fold kernel behind, and with the fold in a launch that merges
SPLIT = dict(B=1, Sq=900, H=2, D=128, lens=[2600], jobs=[[0]], merged=0)
SPLIT_MERGING = dict(B=2, Sq=100, H=516, D=64, lens=[2560, 2500], jobs=None, max_jobs=2, merged=2)


@pytest.mark.parametrize("other", [SPLIT, SPLIT_MERGING])
def test_no_parts_come_between_parts_and_their_fold(tmp_path, other):
    """Two threads on one stream share its workspace: behind a launch whose parts a fold kernel reads comes that kernel, and no other
    launch that writes parts."""
    alone, pair, both = record(tmp_path, [SPLIT, other], [SPLIT, other], 20)
    assert [k.startswith("_ZN2dt21attn_tail_fold_kernel") for _, k in alone] == [False, True]
    assert len(pair) == (2 if other is SPLIT else 1)
    split = alone[0][1]
    assert sum(k == split for _, k in both) == (40 if other is SPLIT else 20)
    assert len({t for t, _ in both}) == 2
    for (t0, k0), (t1, k1) in zip(both, both[1:]):
        if k0 == split:
            assert (t1, k1) == (t0, alone[1][1])


def _masked(H, Sq, D, states, jobs, keys=None, B=1):
    """A device-listed call: ``jobs`` of ``states`` chunks of ``keys`` keys (the queries' number)."""
    return dict(B=B, Sq=Sq, H=H, D=D, lens=[keys or Sq] * states, jobs=None, max_jobs=jobs, merged=states)


def _listed(H, Sq, D, states, jobs, keys=None, B=1):
    """The same with jobs of one chunk each that the host lists."""
    return dict(_masked(H, Sq, D, max(states, jobs), 0, keys, B), jobs=[[j] for j in range(jobs)], merged=states)


# both sides of every line of the rule: whether the launch merges the states itself
MERGES = [
    # items of one job: 24 and 48 an XCD; items in all: 216 and 270
    (_masked(24, 1861, 128, 16, 15), False), (_masked(24, 4000, 128, 8, 8), True), (_masked(24, 1861, 64, 16, 15), False),
    (_masked(24, 4000, 64, 16, 15), True), (_masked(48, 2222, 64, 8, 4), False), (_masked(48, 2222, 64, 8, 5), True),
    (_masked(24, 14882, 128, 8, 4), True), (_masked(24, 119056, 128, 32, 3, 3721), True),
    # key tiles: 9 and 10 at D = 64, 19 and 20 at D = 128
    (_masked(24, 6000, 64, 16, 8, 9 * 64), False), (_masked(24, 6000, 64, 16, 8, 9 * 64 + 1), True),
    (_masked(24, 6000, 128, 16, 8, 19 * 64), False), (_masked(24, 6000, 128, 16, 8, 19 * 64 + 1), True),
    # short launches: queries, items, key tiles, states, parts
    (_masked(48, 128, 64, 4, 4), True), (_masked(48, 129, 64, 4, 2), True), (_masked(48, 129, 64, 4, 3), False), (_masked(4, 512, 64, 4, 2), True),
    (_masked(48, 512, 64, 2, 2), False), (_masked(12, 7732, 64, 4, 2), True), (_masked(24, 1735, 64, 4, 2), False),
    (_masked(24, 5000, 64, 4, 2, 9 * 64), False), (_masked(24, 5000, 64, 4, 2, 9 * 64 + 1), True), (_masked(24, 5000, 64, 5, 2), False),
    (_masked(24, 96, 128, 2, 2), True), (_masked(24, 129, 128, 2, 2), False), (_masked(24, 160, 128, 2, 2, 128), True),
    (_masked(24, 161, 128, 2, 2, 128), False), (_masked(48, 128, 128, 3, 2), True),
    (_masked(48, 128, 128, 3, 3), False), (_masked(3, 128, 128, 2, 2, 256), True), (_masked(3, 128, 128, 2, 2, 257), False),
    (_masked(4, 96, 64, 4, 1), True), (_masked(4, 96, 64, 5, 1), False), (_masked(3, 1706, 64, 3, 1), False),
    # one job whose items all merge
    (_masked(32, 1479, 64, 2, 1), True), (_masked(32, 1479, 64, 2, 1, 23 * 64), False), (_masked(32, 1479, 64, 2, 2), False),
    # the host's list: items, key tiles
    (_listed(48, 400, 64, 4, 4), True), (_listed(48, 600, 64, 4, 3), False), (_listed(48, 254, 128, 4, 4), True),
    (_listed(48, 254, 128, 3, 3, B=2), False), (_listed(24, 256, 128, 2, 2), True), (_listed(24, 257, 128, 2, 2), False),
    (_listed(12, 300, 64, 5, 2), False),
]


def test_the_gpu_tests_of_merging_launches_merge(tmp_path):
    for call, kernels in zip(MERGING, record(tmp_path, MERGING)):
        assert len(kernels) == 1, call


def test_which_launches_merge_their_states(tmp_path):
    """A launch merges where that is the faster form for its sizes: one kernel, an instantiation of its own; else the attention
    kernel, the fold kernel where items are split, and the merge kernel."""
    for (call, merges), kernels in zip(MERGES, record(tmp_path, [call for call, _ in MERGES])):
        names = [k for _, k in kernels]
        own = f"_ZN2dt15attn_fwd_kernelILi{call['D']}ELb0ELb0ELb1EEE"
        if merges:
            assert len(names) == 1 and names[0].startswith(own), call
        else:
            assert not names[0].startswith(own) and names[-1].startswith("_ZN2dt19merge_states_kernel"), call
