"""K/V of all ring positions at once: what ``kv_chunk`` gives and raises one by one."""
import pytest
import torch

from ditango_amd.core.parallel_state import LocalRingGroup


def _one_by_one(group, n, local, key, value):
    kv = [(key, value) if c == local else group.kv_chunk(c) for c in range(n)]
    return [k for k, _ in kv], [v for _, v in kv]


@pytest.mark.parametrize("patched", [False, True])
@pytest.mark.parametrize("missing", [None, 0, 2])
@pytest.mark.parametrize("n,local", [(3, -1), (3, 0), (3, 2), (2, -1), (2, 1), (4, -1), (0, -1)])
def test_lists_are_the_chunks_one_by_one(n, local, missing, patched):
    group = LocalRingGroup(3)
    ks, vs = ([torch.full((1,), float(10 * s + i)) for i in range(3)] for s in (1, 2))
    if missing is not None:
        vs[missing] = None
    group.set_kv_chunks(ks, vs)
    if patched:
        group.kv_chunk = lambda c: (ks[0], ks[c])
    key, value = torch.zeros(1), torch.ones(1)
    try:
        want = _one_by_one(group, n, local, key, value)
    except Exception as e:
        with pytest.raises(type(e), match=str(e)[:20].replace("(", r"\(")):
            group.kv_lists(n, local, key, value)
        return
    got = group.kv_lists(n, local, key, value)
    assert all(a is b for g, w in zip(got, want) for a, b in zip(g, w)) and [len(g) for g in got] == [n, n]
    assert got[0] is not group._k and all(a is b for a, b in zip(group._k, ks))


def test_a_lookup_replaced_on_the_class_is_called(monkeypatch):
    group = LocalRingGroup(3)
    ks, vs = ([torch.full((1,), float(10 * s + i)) for i in range(3)] for s in (1, 2))
    group.set_kv_chunks(ks, vs)
    asked = []

    def lookup(self, c):
        asked.append(c)
        return ks[0], vs[c]

    monkeypatch.setattr(LocalRingGroup, "kv_chunk", lookup)
    key, value = torch.zeros(1), torch.ones(1)
    got = group.kv_lists(3, 1, key, value)
    assert asked == [0, 2]
    assert all(a is b for g, w in zip(got, ([ks[0], key, ks[0]], [vs[0], value, vs[2]])) for a, b in zip(g, w))
