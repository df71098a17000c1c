"""The start of a work item of ``attn_fwd_kernel`` as a host-side model (no GPU): Q comes through the LDS, and half of it through V buffers 2 and 3.

``tests/test_attn_schedule_model.py`` replays the waits, barriers, loads and reads of a work item and holds the rules for K and V.  Its prologue
is that of a kernel that reads Q from memory: four calls of the trailing group, then one wait, and a share of V in the first call.  Here
the prologue is the kernel's (a test compares its order with the source), the loop and the end are those of that model, and besides its
rules

  (iv) a wavefront reads its rows of Q behind a wait of its own that covers their loads (they are nobody else's, no barrier is needed);
  (v)  what a wavefront loads into a place that holds rows of Q is issued behind a barrier behind its reads of them (the barrier waits for the
       LDS, too), and nothing is loaded there between the rows' own load and their reads.

A quarter of the wavefront's 32 rows is a share: as many load instructions as its share of a K or V tile, in the same place of the buffer."""
import re

import pytest

from tests import test_attn_schedule_model as model

LOOP = model.wave_program
STAGING = [("staging", 0), ("staging", 1)]
PLACES = STAGING + [("V", 3), ("V", 2)]   # of the quarters of Q, in the order of their loads


def kernel_program(s, group, n_tiles, end=model.END_PLAIN, places=PLACES, first_call_has_v=False, call_before_q=False, call_before_barrier=False):
    """As ``model.wave_program``, with ("load", "Q", -1 - quarter, place) and ("read own", quarter, place); the last three arguments are mistakes."""
    ops = [("load", "Q", -1 - i, place) for i, place in enumerate(places)]

    def load_tile(y):
        if y > 0 or first_call_has_v:
            ops.append(("load", "V", y - 1, (y - 1) % s.num_buf))
        ops.append(("load", "K", y, y % s.num_buf))

    def trailing_calls():
        if group == 1:
            for y in range(s.prologue_calls[0], s.prologue_calls[1]):
                load_tile(y)

    for y in range(s.prologue_calls[0]):
        load_tile(y)
    if call_before_q:
        trailing_calls()
    ops.append(("wait", s.prologue_inflight[0]))
    ops += [("read own", i, place) for i, place in enumerate(places)]
    if call_before_barrier:
        trailing_calls()
    ops.append(("barrier",))
    if group == 1:
        if not (call_before_q or call_before_barrier):
            trailing_calls()
        ops.append(("barrier",))
    if n_tiles > 0:
        ops.append(("read", "K", 0, 0))
    if group == 1 and s.trailing_k1_inflight is not None:
        ops.append(("wait", s.trailing_k1_inflight))
    ops.append(("barrier",))
    theirs = LOOP(s, group, n_tiles, end)
    loop = 2 * s.prologue_calls[group] + 2 + (group == 1) + (n_tiles > 0) + (group == 1 and s.trailing_k1_inflight is not None) + 1
    assert theirs[loop - 1] == ("barrier",)
    return ops + theirs[loop:]


def q_violations(program):
    bad, issued, landed, holds, read_behind = [], [], 0, {}, {}   # holds: place -> quarter not read yet; read_behind: place -> barriers at the read
    barriers = 0
    for op in program:
        if op[0] == "barrier":
            barriers += 1
        elif op[0] == "wait":
            landed = max(landed, len(issued) - op[1])
        elif op[0] == "load":
            place = op[3] if op[1] == "Q" else (op[1], op[3])
            if place in holds:
                bad.append(("load over rows of Q that have not been read", op))
            elif read_behind.get(place) == barriers:
                bad.append(("load over rows of Q without a barrier behind their reads", op))
            if op[1] == "Q":
                holds[place] = len(issued)
            issued.append(op)
        elif op[0] == "read own":
            if holds.get(op[2], landed) >= landed:
                bad.append(("rows of Q are read that may not have landed", op))
            holds.pop(op[2], None)
            read_behind[op[2]] = barriers
    return bad


def violations(s, n_tiles, monkeypatch, end=model.END_PLAIN, **mistake):
    program = lambda s, group, n, end=model.END_PLAIN: kernel_program(s, group, n, end, **mistake)   # noqa: E731
    with monkeypatch.context() as m:
        m.setattr(model, "wave_program", program)
        bad, _ = model.replay(s, n_tiles, end)
    return bad + [b for group in (0, 1) for b in q_violations(program(s, group, n_tiles, end))]


@pytest.mark.parametrize("end", [model.END_PLAIN, model.END_SHARED_KEYS], ids=["plain", "shared keys"])
@pytest.mark.parametrize("D", [128, 64])
def test_the_kernels_start_is_race_free(monkeypatch, D, end):
    s = model.Schedule(model.read_table(), D)
    for n in model.TILE_COUNTS:
        assert not violations(s, n, monkeypatch, end), (D, n)
        shares = [sum(op[0] == "load" and op[1] != "Q" for op in kernel_program(s, g, n, end)) for g in (0, 1)]
        assert shares == [2 * (s.prologue_calls[g] + n) - 1 for g in (0, 1)]


MISTAKES = [dict(call_before_q=True), dict(call_before_barrier=True), dict(first_call_has_v=True), dict(places=STAGING + [("V", 0), ("V", 2)]),
            dict(places=STAGING + [("V", 3), ("V", 1)])]


@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("mistake", MISTAKES, ids=lambda m: next(iter(m)))
def test_loads_over_rows_of_q_are_rejected(monkeypatch, D, mistake):
    s = model.Schedule(model.read_table(), D)
    assert all(violations(s, n, monkeypatch, **mistake) for n in model.TILE_COUNTS)


@pytest.mark.parametrize("D", [128, 64])
def test_weaker_waits_are_rejected(monkeypatch, D):
    base = model.read_table()
    suffix = "D64" if D == 64 else "D128"
    for key, delta in ((f"VECTOR_BARRIER_INFLIGHT_{suffix}", 1), ("PROLOGUE_INFLIGHT_LEADING", 1), ("TRAILING_K1_INFLIGHT", 1), ("NUM_BUF", -1), ("CALL_AHEAD", 1)):
        s = model.Schedule(dict(base, **{key: base[key] + delta}), D)
        assert any(violations(s, n, monkeypatch) for n in range(1, 13)), (D, key)
    # the wait that Q needs by itself: one share more than the calls behind it
    s = model.Schedule(dict(base, PROLOGUE_INFLIGHT_LEADING=2 * base["PROLOGUE_CALLS_LEADING"]), D)
    assert all(any("Q" in b[0] for b in violations(s, n, monkeypatch)) for n in model.TILE_COUNTS)


def _item():
    code = re.sub(r"//[^\n]*", "", open(model.KERNEL).read())
    return code[code.index("void attn_item("):code.index("__global__", code.index("void attn_item("))]


def test_the_kernel_starts_as_the_model_does():
    """Loads, waits, reads of Q and barriers in front of the loop, in the order of the source."""
    item = _item()
    start = item[:item.index("for (int t = 0; t < n_tiles; t += 4)")]
    start = start[:start.index("auto load_tile = ")] + start[start.index("load_tile(y)") - 200:start.index("auto iteration = ")]
    steps = [r"load_rows_to_lds\(", r"y = 0; y < DT_SCHED_PROLOGUE_CALLS_LEADING; \+\+y\) load_tile\(y\)", r"wait_tile_loads<DT_SCHED_PROLOGUE_INFLIGHT_LEADING \* T::kLoads>",
             r"qf\[s\] = \*reinterpret_cast", r"phase_barrier\(\);", r"if \(group == 1\) \{",
             r"y = DT_SCHED_PROLOGUE_CALLS_LEADING; y < DT_SCHED_PROLOGUE_CALLS_TRAILING; \+\+y\) load_tile\(y\)", r"phase_barrier\(\);", r"qk_only\(\);",
             r"if \(group == 1\) wait_tile_loads<DT_SCHED_TRAILING_K1_INFLIGHT \* T::kLoads>", r"phase_barrier_after_matrix\("]
    anything = r"load_rows_to_lds\(|load_tile\(y\)|wait_tile_loads<|qf\[s\] = \*|phase_barrier\w*\(|qk_only\(\);"
    at = 0
    for step in steps:
        found = re.compile(step).search(start, at)
        assert found, step
        between = re.search(anything, start[at:found.start()])
        assert between is None, (step, between)
        at = found.end()
    assert re.search(anything, start[at:]) is None


def test_places_and_first_call_are_those_of_the_model():
    item = re.sub(r"\s+", " ", _item())
    assert "constexpr int kQuarter = T::kLoads;" in item
    quarters = re.search(r"q_quarter\[4\] = \{(.*?)\};", item).group(1)
    assert re.findall(r"T::kOffV \+ (\d) \* T::kBytesV \+ wave \* kQuarter \* 1024", quarters) == [str(b) for kind, b in PLACES if kind == "V"]
    assert quarters.count("T::kLdsTiles + wave * T::kStageBytes") == 2
    assert "const uint32_t vdst = lds_base + T::kOffV + vbuf * T::kBytesV + wave * (1024 * T::kLoads);" in item
    assert "no_v = true;" in item and "if (no_v) { no_v = false; } else if (__builtin_expect(v_lags, 0)) {" in item
