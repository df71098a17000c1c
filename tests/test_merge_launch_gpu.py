"""Launches that merge (``dt_attn_sched_merge_fwd``, ``dt_attn_jobs_merge_fwd``) against the same launch without a merge and
the merge kernel behind it: the two compute one thing, in fp32 from the same 16-bit states.  Such a call merges in the launch for some
sizes and in a kernel behind it for others; tests/test_launch_order.py checks, without a GPU, that those of ``MERGING`` below are
of the first kind."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from ditango_amd import _hip
    _hip.load_library()
    return _hip


def _inputs(B, Sq, H, D, lens, dtype, strided=False):
    g = torch.Generator(device="cuda").manual_seed(Sq * 131 + H * 7 + D)

    def make(n):
        if strided:   # slices of a fused projection
            return torch.randn(B, n, 3, H, D, generator=g, device="cuda").to(dtype)[:, :, 1]
        return torch.randn(B, n, H, D, generator=g, device="cuda").to(dtype)

    return make(Sq), [make(n) for n in lens], [make(n) for n in lens]


def _close(got, want, dtype, what):
    """fp32 results of the same states: products and sums of n terms in another order and another exp's last bits, 2^-20 of the
    largest value here.  A 16-bit result, or states that were folded from parts (another order under their rounding), may differ by one
    rounding of a state: 2^-8 (bf16) or 2^-11 (fp16) of the value's binade."""
    tol = {torch.float32: 2.0 ** -20, torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}[dtype]
    got, want = got.float(), want.float()
    got, want = got.masked_fill(got == want, 0.0), want.masked_fill(got == want, 0.0)   # (the lse of a chunk without keys: -inf in both)
    assert torch.isfinite(got).all(), what
    err, scale = (got - want).abs().max().item(), max(1.0, want.abs().max().item())
    assert err <= tol * scale, what


# rows: one, the edges of a 32-row slice, of half a tile and of a tile, several tiles; chunks without keys, of less than a key
# tile, of the sizes at which a launch is cut along its rows (8 key tiles) and along its keys (16 and more); some of them merge
SHAPES = [
    (1, 1, 3, 64, (40, 0, 64), (0, 2)), (1, 31, 2, 128, (64, 65, 1), (0, 1, 2)), (2, 33, 3, 64, (200, 130), (1,)),
    (1, 127, 4, 128, (512, 512, 512), (0, 2)), (1, 129, 4, 64, (512, 512, 512), (0, 2)), (1, 512, 4, 64, (512,) * 4, (0, 3)),
    (1, 255, 2, 128, (1500, 700), (0, 1)), (2, 257, 3, 64, (2000, 1999, 2000), (0, 1)), (1, 300, 2, 64, (4000, 4000), (0,)),
    (2, 100, 516, 64, (2560, 2500), (0, 1)), (2, 100, 516, 128, (1700, 1600), (1, 0)),   # long enough to merge and fold items of several parts
    (1, 700, 5, 128, (1100,) * 11, (0, 4, 10)), (1, 1861, 6, 64, (1861,) * 3 + (1860,) * 2, (0, 3)), (1, 96, 1, 128, (96,) * 40, (7,)),
]


# launches that merge: short ones, one job a chunk, and ...
SHORT = [SHAPES[i] for i in (0, 1, 2, 4, 5)] + [(1, 128, 6, 128, (250, 30), (0, 1)), (1, 700, 3, 64, (700, 650), (1, 0))]   # (the last along its rows)
# ... long ones, of enough items and key tiles: whole items of one, several and many tiles, items cut in two along the rows, and in 2, 4 and 5
# parts along the keys; 2 ... 6 states; the last in few rounds
LONG = [
    (1, 31, 1040, 128, (1290, 90), (0, 1)), (1, 300, 560, 128, (1300, 90), (1, 0)), (1, 1861, 66, 128, (1300, 90, 64, 0), (0, 2, 3)),
    (1, 300, 528, 128, (1300, 90), (0, 1)), (1, 300, 540, 64, (700, 90), (0,)), (1, 100, 1080, 128, (2600, 90), (0, 1)),
    (1, 300, 352, 128, (2600, 90, 90), (0, 1, 2)), (2, 300, 262, 64, (2600, 90), (0, 1)), (1, 289, 200, 64, (700, 90, 90, 1, 90, 0), (0, 4)),
    (1, 300, 130, 64, (700, 600), (0, 1)),
]


@pytest.mark.parametrize("B,Sq,H,D,lens,computed", SHAPES + SHORT[-2:] + LONG)
@pytest.mark.parametrize("dtype,out", [(torch.bfloat16, torch.float32), (torch.float16, torch.float16)])
def test_scheduled_launch_that_merges(hip, B, Sq, H, D, lens, computed, dtype, out):
    q, ks, vs = _inputs(B, Sq, H, D, lens, dtype, strided=Sq % 2 == 1)
    C, diag = len(lens), computed[0]
    table = hip.ChunkTable(ks, vs)
    ids = torch.tensor(list(computed) + [-1] * (C - len(computed)), dtype=torch.int32, device="cuda")
    count = torch.tensor([len(computed), 0], dtype=torch.int32, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(5)
    slots = torch.randn(C, B, Sq, H, D, generator=g, device="cuda").to(dtype)
    lses = 2 * torch.randn(C, B, H, Sq, generator=g, device="cuda")
    ws = hip.attn_workspace("cuda")

    def run(merging):
        so, sl = slots.clone(), lses.clone()
        do, dl = torch.zeros_like(so[0]), torch.zeros_like(sl[0])
        args = (q, table, ids, count, C, so, sl, diag, do, dl)   # (more jobs than the schedule lists)
        if merging:
            return (*hip.attn_sched_merge(*args, out, ws), so, sl, do, dl)
        hip.attn_sched_fwd(*args, workspace=ws)
        return (*hip.merge_arena(so, sl, diag, do, dl, out), so, sl, do, dl)

    want, got, again = run(False), run(True), run(True)
    split = len(computed) * max(lens) >= 16 * 64 * len(computed)
    for i, name in enumerate(("out", "lse", "slots", "slot lse", "local", "local lse")):
        assert torch.equal(got[i], again[i]), name
        loose = dtype if i in (2, 4) or (i == 0 and (split or out != torch.float32)) else torch.float32
        _close(got[i], want[i], loose, name)
    assert not hip.attn_counters("cuda", q).any()



NUMBERS = [1, 4, 5, 8, 9, 16, 17]


def _of_states(n, D):
    """Rows that end in the middle of a load instruction's; heads and keys enough that the launch merges any number of states."""
    return 1, 70, 520 if n >= 5 else 2080, D, (1290 if D == 128 else 650,) + (90,) * (n - 1), (n // 2,)


@pytest.mark.parametrize("n", NUMBERS)
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dtype,out", [(torch.bfloat16, torch.float32), (torch.float16, torch.float16)])
def test_numbers_of_states_that_merge(hip, n, D, dtype, out):
    """The edges of the merge's batches of states."""
    test_scheduled_launch_that_merges(hip, *_of_states(n, D), dtype, out)


# host-listed jobs and cached states; those from the fifth on merge 2, 6, 9, 16, 5 and 3 states in the launch
JOBS = [
    (1, 65, 3, 64, (100, 100), [[0], [1]], 0), (1, 512, 4, 128, (512,) * 4, [[2], [0, 1, 3]], 3), (2, 333, 2, 64, (900, 1700, 64), [[0, 1, 2]], 1),
    (1, 288, 5, 128, (2300, 1), [[0], [1], [0, 1]], 14),
    (1, 600, 3, 64, (500, 200), [[0, 1]], 0), (1, 288, 352, 128, (700, 600, 64), [[0, 1], [2], [1]], 2), (1, 70, 800, 64, (650, 90), [[1, 0], [0], [1]], 5),
    (1, 300, 352, 128, (1300, 1), [[0], [1], [0, 1]], 14), (1, 100, 1080, 64, (2600, 90), [[0], [1]], 2), (1, 128, 5, 128, (190, 56), [[0, 1]], 1),
]


def _merged_jobs(jobs, cached):
    which = list(range(len(jobs))) + [0]   # (a state may be merged twice)
    return which[:2] if cached + len(which) > 16 else which


@pytest.mark.parametrize("B,Sq,H,D,lens,jobs,cached", JOBS)
def test_jobs_that_merge_with_cached_states(hip, B, Sq, H, D, lens, jobs, cached):
    dtype = torch.bfloat16
    q, ks, vs = _inputs(B, Sq, H, D, lens, dtype)
    g = torch.Generator(device="cuda").manual_seed(9)
    outs = [torch.randn(B, Sq, H, D, generator=g, device="cuda").to(dtype) for _ in range(cached)]
    lses = [2 * torch.randn(B, H, Sq, generator=g, device="cuda") for _ in range(cached)]
    which = _merged_jobs(jobs, cached)
    ws = hip.attn_workspace("cuda")
    states, out, lse = hip.attn_states_merge(q, ks, vs, jobs, 32, outs, lses, which, torch.float32, ws)
    plain = hip.attn_states(q, ks, vs, jobs, 32, ws)
    for (o, l), (po, pl) in zip(states, plain):
        _close(o, po, dtype, "state")
        _close(l, pl, torch.float32, "state lse")
    want, want_lse = hip.merge_states(outs + [states[i][0] for i in which], lses + [states[i][1] for i in which], dst_lse_bsh=True)
    _close(out, want, torch.float32, "out")
    _close(lse, want_lse, torch.float32, "lse")
    assert not hip.attn_counters("cuda", q).any()


def test_rows_without_any_state_and_infinite_values(hip):
    """A row whose states are all empty is 0 with lse -inf; an infinity in a state of weight is one in the result."""
    q, ks, vs = _inputs(1, 40, 2, 64, (64, 64), torch.bfloat16)
    so = torch.randn(2, 1, 40, 2, 64, device="cuda").bfloat16()
    sl = torch.full((2, 1, 2, 40), float("-inf"), device="cuda")
    ids = torch.zeros(2, dtype=torch.int32, device="cuda")
    none = torch.zeros(2, dtype=torch.int32, device="cuda")
    table = hip.ChunkTable(ks, vs)
    out, lse = hip.attn_sched_merge(q, table, ids, none, 1, so, sl, -1, so[0], sl[0], torch.float32)
    assert (out == 0).all() and (lse == float("-inf")).all()
    sl.fill_(0.5)
    so[1, 0, 7, 1, 3] = float("inf")
    out, lse = hip.attn_sched_merge(q, table, ids, none, 1, so, sl, -1, so[0], sl[0], torch.float32)
    assert out[0, 7, 1, 3] == float("inf") and torch.isinf(out).sum() == 1
    _close(lse, torch.full_like(lse, 0.5 + 0.6931472), torch.float32, "lse")


def _infinite(n, D):
    """One job, with heads and keys enough that its launch merges; 32 rows and 8."""
    return 1, 40, 2048, D, (1290 if D == 128 else 650,) + (64,) * (n - 1)


@pytest.mark.parametrize("n", [1, 2, 3, 5, 9])
@pytest.mark.parametrize("D", [64, 128])
def test_infinities_of_the_last_state(hip, n, D):
    """The lists of states go on behind the last one with copies of it that are not to be read: an infinity of its own, in every
    row, is one in the result, and nothing else is."""
    B, Sq, H, D, lens = _infinite(n, D)
    q, ks, vs = _inputs(B, Sq, H, D, lens, torch.bfloat16)
    g = torch.Generator(device="cuda").manual_seed(n)
    so = torch.randn(n, 1, Sq, H, D, generator=g, device="cuda").bfloat16()
    sl = 2 * torch.randn(n, 1, H, Sq, generator=g, device="cuda")
    col = ((5 * torch.arange(Sq, device="cuda")[:, None] + 3 * torch.arange(H, device="cuda")) % D)[None, :, :, None]
    so[-1].scatter_(-1, col, float("inf"))
    ids = torch.zeros(n, dtype=torch.int32, device="cuda")
    out, lse = hip.attn_sched_merge(q, hip.ChunkTable(ks, vs), ids, ids[:1].clone(), 1, so, sl, -1, so[0], sl[0], torch.float32)
    assert not torch.isnan(out).any()
    assert torch.equal(torch.isinf(out), torch.zeros_like(out, dtype=torch.bool).scatter_(-1, col, True))
    want, want_lse = hip.merge_arena(so, sl, -1, so[0], sl[0])
    finite = ~torch.isinf(out)
    _close(out[finite], want[finite], torch.float32, "out")
    _close(lse, want_lse, torch.float32, "lse")


def _call(B, Sq, H, D, lens, states, jobs=None, max_jobs=0, **k):
    """The arguments of ``record`` in tests/launch_log.py."""
    return dict(B=B, Sq=Sq, H=H, D=D, lens=list(lens), jobs=jobs, max_jobs=max_jobs, merged=states)


GRAPH = (1, 129, 4, 64, (512,) * 3)
MERGING = [_call(B, Sq, H, D, lens, len(lens), max_jobs=len(lens)) for B, Sq, H, D, lens, _ in
           SHORT + LONG + [_of_states(n, D) for n in NUMBERS for D in (64, 128)] + [(*GRAPH, ())]]
MERGING += [_call(*_infinite(n, D), n, max_jobs=1) for n in (1, 2, 3, 5, 9) for D in (64, 128)]
MERGING += [_call(B, Sq, H, D, lens, cached + len(_merged_jobs(jobs, cached)), jobs) for B, Sq, H, D, lens, jobs, cached in JOBS[:1] + JOBS[4:]]


def test_captured_merging_launch_replays(hip):
    """A launch that merges, captured with counters of the graph's own: they are at zero after every replay, with eager launches that
    have theirs in between.  (A layer call under capture runs the merge kernel: its counters would have to be cleared by the graph.)"""
    B, Sq, H, D, lens = GRAPH
    q, ks, vs = _inputs(B, Sq, H, D, lens, torch.bfloat16)
    table = hip.ChunkTable(ks, vs)
    ids, count = torch.tensor([2, 0, 1], dtype=torch.int32, device="cuda"), torch.tensor([2], dtype=torch.int32, device="cuda")
    ws = hip.attn_workspace("cuda").clone()
    own = torch.zeros(hip.attn_counters("cuda", q).numel(), dtype=torch.int32, device="cuda")
    asked = []

    def run(counters, workspace, so, sl):
        return hip._host().attn_sched_merge(q, table.native, ids, count, 0, 3, so, sl, -1, so[0], sl[0], torch.float32, workspace, counters,
                                            0, hip._stream())

    g = torch.Generator(device="cuda").manual_seed(3)
    states = lambda: (torch.randn(3, B, Sq, H, D, generator=g, device="cuda").bfloat16(), torch.randn(3, B, H, Sq, generator=g, device="cuda"))
    slots, eager_slots = states(), states()
    eager = lambda: run(lambda need: hip.attn_counters("cuda", q), hip.attn_workspace("cuda"), *eager_slots)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        run(lambda need: own, ws, *slots)
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            got = run(lambda need: asked.append(need) or own, ws, *slots)
    assert asked and asked[0] <= own.numel()
    for _ in range(5):
        q.copy_(torch.randn(q.shape, generator=g, device="cuda").bfloat16())
        for mine, others in zip(slots, eager_slots):
            mine.copy_(torch.randn(mine.shape, generator=g, device="cuda").to(mine.dtype))
            others.copy_(mine)
        graph.replay()
        want = eager()
        torch.cuda.synchronize()
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
        assert all(torch.equal(mine, others) for mine, others in zip(slots, eager_slots))
        assert not own.any() and not hip.attn_counters("cuda", q).any()


def test_layer_call_replays_in_a_graph(hip):
    """Under capture the states are merged by the kernel behind the launch."""
    q, ks, vs = _inputs(1, 600, 3, 64, (1500, 1500), torch.bfloat16)
    run = lambda: hip.attn_states_merge(q, ks, vs, [[0], [1]], 32, [], [], [0, 1], torch.float32, hip.attn_workspace("cuda"))[1:]
    want = run()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        run()
        graph = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            got = run()
    for _ in range(4):
        q.copy_(torch.randn(q.shape, device="cuda").bfloat16())
        graph.replay()
        want = run()
        torch.cuda.synchronize()
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
