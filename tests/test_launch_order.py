"""The order in which the kernels of a call enter a stream's queue, without a GPU (tests/launch_log.py)."""
import pytest

from tests.launch_log import record

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
