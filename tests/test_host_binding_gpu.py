"""The extension module between Python and the C ABI (ditango_amd/csrc/host_binding.cpp)."""
import os
import re
import shutil
import subprocess
import sys
import textwrap
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_CALLS = """
    import importlib.util, sys, threading, time
    import torch
    spec = importlib.util.spec_from_file_location("_ditango_host", sys.argv[1])
    host = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(host)
    q = torch.zeros(1, 8, 2, 64, dtype=torch.bfloat16, device="cuda")
    o, l = torch.zeros_like(q), torch.zeros(1, 2, 8, device="cuda")
    table = host.ChunkTable([q], [q], 0, None)
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device="cuda")
    seg = host.Segments(i32(0, 8), [i32(0, 8)], 8)
    jobs = lambda **kw: host.attn_jobs(q, table, [[0]], [o], [l], 0.0, None, None, None, 0, kw.get("no_alloc", False),
                                       kw.get("seg"), [0] if "seg" in kw else None, 0)
    sched = lambda s: host.attn_sched(q, table, i32(0), i32(1), 0, 1, o[None], l[None], -1, None, None, 0.0, None, None, None, 0, s, 0)
    calls = {
        "jobs": jobs, "noalloc": lambda: jobs(no_alloc=True), "varlen": lambda: jobs(seg=seg),
        "states": lambda: host.attn_states(q, [q], [q], [[0]], 32, None, None, None, 0, None, None, 0),
        "f32": lambda: host.attn_states_f32(q.float(), [q.float()], [q.float()], [[0]], 0.0, 0),
        "sched": lambda: sched(None), "sched varlen": lambda: sched(seg),
        "merge": lambda: host.merge([o], [l], None, None, torch.float32, True, 0),
        "arena": lambda: host.merge_arena(o[None], l[None], -1, o, l, torch.float32, 0),
        "store": lambda: host.cache_store(o.float(), l, o, l, 0),
        "load": lambda: host.cache_load(o, l, torch.float32, True, None, None, 0),
        "zero": lambda: host.zero_rows_from(o, i32(0), 0),
    }
    torch.cuda.synchronize()
    ticks = 0
    def tick():
        global ticks
        while True:
            ticks += 1
            time.sleep(0.002)
    threading.Thread(target=tick, daemon=True).start()
    for name, call in calls.items():
        before = ticks
        call()
        print(name, ticks - before, flush=True)
    torch.cuda.synchronize()
"""


def test_other_python_threads_run_while_a_launch_waits(tmp_path):
    """The module next to a library of the same entry points that do nothing but wait 200 ms: a second thread that wakes up every
    2 ms gets on in the meantime, so no call holds the interpreter lock (50 of the 100 wake-ups leave room for a slow
    machine; with the lock held there is one at most)."""
    shutil.copy(os.path.join(ROOT, "ditango_amd", "lib", "_ditango_host.so"), tmp_path)
    names = set(re.findall(r"^int (dt_\w+)\(", open(os.path.join(ROOT, "include", "ditango_hip.h")).read(), re.M))
    (tmp_path / "stub.cpp").write_text(
        "#include <unistd.h>\nextern \"C\" {\nconst char* dt_last_error(void) { return \"\"; }\n"
        + "".join(f"int {n}(...) {{ usleep(200000); return 0; }}\n" for n in sorted(names)) + "}\n")
    subprocess.run(["g++", "-shared", "-fPIC", "-o", str(tmp_path / "libditango_hip.so"), str(tmp_path / "stub.cpp")], check=True)
    (tmp_path / "calls.py").write_text(textwrap.dedent(_CALLS))
    run = subprocess.run([sys.executable, "-u", str(tmp_path / "calls.py"), str(tmp_path / "_ditango_host.so")],
                         capture_output=True, text=True, timeout=100)
    assert run.returncode == 0, run.stderr[-2000:]
    counts = dict(line.rsplit(" ", 1) for line in run.stdout.splitlines())
    assert len(counts) == 12 and all(int(n) >= 50 for n in counts.values()), counts


@pytest.mark.parametrize("jobs,max_chunks,cu_q,cu_kv,says", [
    ([[0, 2]], 32, [0, 8], [[0, 8], [0, 8]], "outside the table of 2"),
    ([[-1]], 32, [0, 8], [[0, 8], [0, 8]], "outside the table of 2"),
    ([[5]], 32, None, None, "outside the table of 2"),
    ([[0, 1]], 0, None, None, "at least one chunk"),
    ([[0, 1]], -1, None, None, "at least one chunk"),
    ([[0]], 32, [], [[], []], "at least one entry"),
    ([[0]], 32, [0, 8], [[0, 8]], "one cu_seqlens_kv per chunk"),
    ([[0]], 32, [0, 4, 8], [[0, 8], [0, 4, 8]], "as many entries"),
])
def test_states_of_malformed_jobs_are_refused(hip, jobs, max_chunks, cu_q, cu_kv, says):
    """Everything is checked before it is used as an index or a step: an error, not a stray read or a loop without an end."""
    q = torch.zeros(1, 8, 2, 64, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(hip.DitangoHipError, match=says):
        hip.attn_states(q, [q, q], [q, q], jobs, max_chunks, None, False, cu_q, cu_kv)


def test_boundaries_of_a_chunk_behind_the_last_query_segment_are_not_read(hip):
    """A chunk's host boundaries may go on behind the segments of the queries, in the state's launch as under a reuse mask."""
    gen = torch.Generator(device="cuda").manual_seed(6)
    q, k, v = (torch.randn(1, n, 2, 64, generator=gen, device="cuda", dtype=torch.bfloat16) for n in (70, 90, 90))
    state = lambda cu_kv: hip.attn_states(q, [k], [v], [[0]], 32, None, False, [0, 30, 70], [cu_kv])[0]
    for got, want in zip(state([0, 40, 80, 90]), state([0, 40, 80])):
        assert torch.equal(got, want)


def test_threads_that_launch_on_one_stream_share_its_workspace(hip):
    """Launches that are split, from two threads on one stream and so with one workspace: what one thread launches may not come
    between the partial states of the other and their fold.  Bit for bit what one thread alone gets."""
    gen = torch.Generator(device="cuda").manual_seed(5)
    rnd = lambda *s: torch.randn(*s, generator=gen, device="cuda", dtype=torch.bfloat16)
    sizes = [(700, 2100, 3, 64), (900, 2600, 2, 64)]   # of less than a round: every item in several parts
    inputs = [[rnd(1, sq, h, d), rnd(1, sk, h, d), rnd(1, sk, h, d)] for sq, sk, h, d in sizes]
    run = lambda q, k, v: hip.attn_states(q, [k], [v], [[0]], 32, hip.attn_workspace("cuda"))[0]
    want = [run(*i) for i in inputs]
    plain = [hip.attn_states(q, [k], [v], [[0]], 32, None)[0] for q, k, v in inputs]
    assert all(not torch.equal(w[0], p[0]) for w, p in zip(want, plain))   # they are split
    torch.cuda.synchronize()
    got, errors = [[], []], []
    start = threading.Barrier(2)

    def work(i):
        try:
            start.wait()
            for _ in range(150):
                got[i].append(run(*inputs[i]))
        except Exception as e:   # noqa: BLE001 (reported by the assertion below)
            errors.append(e)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors
    for i in range(2):
        assert len(got[i]) == 150
        assert all(torch.equal(o, want[i][0]) and torch.equal(l, want[i][1]) for o, l in got[i])


def test_a_launch_that_folds_its_own_parts_shares_the_workspace_too(hip):
    """As above, the second thread's launches merging their states and folding their parts themselves (tests/test_launch_order.py
    has the order of the launches)."""
    gen = torch.Generator(device="cuda").manual_seed(5)
    rnd = lambda *s: torch.randn(*s, generator=gen, device="cuda", dtype=torch.bfloat16)
    q, k, v = rnd(1, 900, 2, 128), rnd(1, 2600, 2, 128), rnd(1, 2600, 2, 128)
    q2, ks, vs = rnd(2, 100, 516, 64), [rnd(2, n, 516, 64) for n in (2560, 2500)], [rnd(2, n, 516, 64) for n in (2560, 2500)]
    runs = [lambda: hip.attn_states(q, [k], [v], [[0]], 32, hip.attn_workspace("cuda"))[0],
            lambda: hip.attn_states_merge(q2, ks, vs, [[0], [1]], 32, [], [], [0, 1], torch.float32, hip.attn_workspace("cuda"))[1:]]
    want = [run() for run in runs]
    plain = hip.attn_states(q, [k], [v], [[0]], 32, None)[0]
    assert not torch.equal(want[0][0], plain[0])   # it is split
    torch.cuda.synchronize()
    errors = []
    start = threading.Barrier(2)

    def work(i):
        try:
            start.wait()
            for _ in range(60):
                out, lse = runs[i]()
                assert torch.equal(out, want[i][0]) and torch.equal(lse, want[i][1])
        except BaseException as e:   # noqa: BLE001 (reported by the assertion below)
            errors.append(e)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors


def test_a_schedule_of_its_own_may_be_a_strided_count_and_a_list_of_any_shape(hip):
    g = torch.Generator().manual_seed(7)
    q, k, v = (torch.randn(1, 96, 2, 64, generator=g).bfloat16().cuda() for _ in range(3))
    table = hip.ChunkTable([k, v, q], [v, k, q])
    counts = torch.tensor([[2, 1], [0, 0]], dtype=torch.int32, device="cuda")
    ids = torch.tensor([2, 0, -1], dtype=torch.int32, device="cuda")
    states = []
    for i, c in ((ids, counts[0, :1]), (ids, counts[:, 0]), (ids[:, None], counts[0, :1]), (ids[:2, None], counts)):
        out, lse = torch.zeros(3, 1, 96, 2, 64, dtype=q.dtype, device="cuda"), torch.zeros(3, 1, 2, 96, device="cuda")
        hip.attn_sched_fwd(q, table, i, c, 2, out, lse, -1, None, None)
        states.append((out, lse))
    for out, lse in states[1:]:
        assert torch.equal(out, states[0][0]) and torch.equal(lse, states[0][1])
    assert states[0][0][0].any() and states[0][0][2].any() and not states[0][0][1].any()


def test_counters_are_asked_for_by_launches_that_merge_only(hip, monkeypatch):
    """The counters of a merging launch are host work, and memory of the stream's: calls that cannot merge (segments, a prescaled q,
    states of another type) and calls whose sizes go to the merge kernel never ask for them."""
    asked = []
    counters = hip._stream_counters
    monkeypatch.setattr(hip, "_stream_counters", lambda *a: asked.append(a) or counters(*a))
    rnd = lambda *s, dtype=torch.bfloat16: torch.randn(*s, device="cuda").to(dtype)

    def call(Sq, D, states=(), **k):
        q, ks, vs = rnd(1, Sq, 2, D), [rnd(1, 300, 2, D)] * 2, [rnd(1, 300, 2, D)] * 2
        outs, lses = [s[0] for s in states], [s[1] for s in states]
        asked.clear()
        _, out, _ = hip.attn_states_merge(q, ks, vs, [[0], [1]], 32, outs, lses, [0, 1], torch.float32, hip.attn_workspace("cuda"), **k)
        assert torch.isfinite(out).all()
        return len(asked)

    state = lambda dtype: (rnd(1, 200, 2, 64, dtype=dtype), rnd(1, 2, 200, dtype=torch.float32))
    assert call(200, 64) == 1 and call(200, 64, [state(torch.bfloat16)]) == 1
    assert call(200, 64, [state(torch.float32)]) == 0
    assert call(200, 64, [state(torch.bfloat16)] * 3) == 0      # 5 states
    assert call(200, 128) == 0
    assert call(200, 64, q_prescaled=True) == 0
    assert call(200, 64, cu_q=[0, 200], cu_kv=[[0, 300]] * 2) == 0
    cu, cu_kv = torch.tensor([0, 200], dtype=torch.int32, device="cuda"), torch.tensor([0, 300], dtype=torch.int32, device="cuda")
    assert call(200, 64, dev_segments=hip.DeviceSegments(cu, [cu_kv] * 2, 200)) == 0

    def scheduled(Sq, D, **k):
        q, ks = rnd(1, Sq, 2, D), [rnd(1, 300, 2, D)] * 2
        so, sl = rnd(2, 1, Sq, 2, D), rnd(2, 1, 2, Sq, dtype=torch.float32)
        ids = torch.tensor([0, 1], dtype=torch.int32, device="cuda")
        asked.clear()
        hip.attn_sched_merge(q, hip.ChunkTable(ks, ks), ids, ids[1:], 1, so, sl, -1, so[0], sl[0], torch.float32, hip.attn_workspace("cuda"), **k)
        return len(asked)

    assert scheduled(200, 64) == 1 and scheduled(200, 128) == 0 and scheduled(200, 64, q_prescaled=True) == 0
