"""fp32 attention on the bf16 matrix pipe: both widths of a workgroup, keys shared by several workgroups, numbers that do not split."""
import ctypes

import pytest
import torch

from oracle import attention_math as om

pytestmark = pytest.mark.gpu


def _check(hip, q, ks, vs, jobs, bsh, bound=1e-5):
    """Against the closed form in fp64, 1e-5 as for the other fp32 tests: sums of at most some thousand terms in fp32."""
    got = hip.attn_jobs_f32_fwd(q.cuda(), [k.cuda() for k in ks], [v.cuda() for v in vs], jobs, lse_bsh=bsh)
    torch.cuda.synchronize()
    for job, (out, lse) in zip(jobs, got):
        k, v = (torch.cat([t[c] for c in job] or [t[0][:, :0]], 1) for t in (ks, vs))
        lse = lse.squeeze(-1).transpose(1, 2) if bsh else lse
        if k.shape[1] == 0:
            assert (out == 0).all() and torch.isneginf(lse).all()
            continue
        ref_out, ref_lse = om.chunk_attention(q, k, v, compute_dtype=torch.float64)
        scale = v.abs().max().item()
        assert (out.double().cpu() - ref_out).abs().max().item() <= bound * scale, job
        assert (lse.double().cpu() - ref_lse).abs().max().item() <= bound, job
    return got


@pytest.mark.parametrize("B,Sq,H,D,lens,jobs,bsh", [
    (1, 1, 1, 64, [1], [[0]], True),                                   # one query, one key
    (1, 65, 2, 64, [31, 0, 33, 70, 1], [[0, 1, 2, 3, 4, 0]], True),    # chunks that end inside tiles, an empty one, one twice
    (1, 33, 1, 128, [1030], [[0]], True),                              # 33 tiles in parts that do not divide them
    (2, 129, 3, 128, [64, 65], [[0, 1], [1], []], False),              # jobs of unequal length, one without keys
    (1, 512, 4, 64, [512, 512, 512, 512], [[0, 1, 2, 3]], True),       # 8 parts
    (1, 700, 12, 64, [700, 701], [[0, 1]], True),                      # four query tiles a workgroup
    (1, 847, 10, 128, [847, 846], [[0, 1]], False),
])
def test_split_products_match_fp64_closed_form(hip, B, Sq, H, D, lens, jobs, bsh):
    g = torch.Generator().manual_seed(Sq + D)
    q = torch.randn(B, Sq, H, D, generator=g)
    ks, vs = ([torch.randn(B, n, H, D, generator=g) for n in lens] for _ in range(2))
    _check(hip, q, ks, vs, jobs, bsh)


@pytest.mark.parametrize("D,q_scale,k_scale,v_scale", [
    (64, 2.0 ** 100, 2.0 ** -100, 1.0),      # the low parts of K end below the exponent range
    (128, 2.0 ** -110, 2.0 ** 110, 1.0),     # ... of Q
    (64, 1.0, 1.0, 2.0 ** -118),             # ... of V, and the result is as small
    (128, 1.0, 1.0, 2.0 ** 100),
    (64, 1.0, 1.0, 0.0),
])
def test_magnitudes_at_the_ends_of_the_range(hip, D, q_scale, k_scale, v_scale):
    g = torch.Generator().manual_seed(D)
    q = torch.randn(1, 70, 2, D, generator=g) * q_scale
    ks, vs = ([torch.randn(1, 300, 2, D, generator=g) * s] for s in (k_scale, v_scale))
    _check(hip, q, ks, vs, [[0]], True)


@pytest.mark.parametrize("D,column", [(64, 3), (64, 60), (128, 5), (128, 77)])
def test_one_small_element_of_q_that_a_large_one_of_k_makes_count(hip, D, column):
    """The rest of the row is of ordinary size, and so are the scores."""
    g = torch.Generator().manual_seed(column)
    q, k, v = (torch.randn(1, n, 2, D, generator=g) for n in (70, 300, 300))
    q[..., column] *= 2.0 ** -122
    k[..., column] *= 2.0 ** 124
    _check(hip, q, [k], [v], [[0]], True)


def _us(call):
    best = float("inf")
    for _ in range(5):
        start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        start.record()
        for _ in range(10):
            call()
        end.record()
        end.synchronize()
        best = min(best, start.elapsed_time(end) * 100)
    return best


def _c_call(hip, q, k, v, scratch, falling):
    """dt_attn_jobs_f32_ws_fwd on one chunk, with scratch or without, and with the keys in falling order: what 64-bit offsets are for, beside
    chunks of 2 GiB and more."""
    lib = hip.load_library()
    B, Sq, H, D = q.shape
    out, lse = torch.empty_like(q), torch.empty(B, H, Sq, device="cuda")
    one = lambda t, x: (t * 1)(x)
    i32, i64, vp = ctypes.c_int32, ctypes.c_int64, ctypes.c_void_p
    last = (k.shape[1] - 1) * k.stride(1) * 4 if falling else 0
    ws = hip.attn_workspace(q.device) if scratch else None
    counters = torch.zeros(1 << 14, dtype=torch.int32, device="cuda") if scratch else None

    def call():
        rc = lib.dt_attn_jobs_f32_ws_fwd(
            q.data_ptr(), B, Sq, H, D, *q.stride()[:3], 1, one(vp, k.data_ptr() + last), one(vp, v.data_ptr() + last), one(i32, k.shape[1]),
            one(i64, k.stride(0)), one(i64, -k.stride(1) if falling else k.stride(1)), one(i64, k.stride(2)), 1, (i32 * 2)(0, 1), one(i32, 0),
            one(vp, out.data_ptr()), one(vp, lse.data_ptr()), 0, 0.0, ws.data_ptr() if scratch else None, ws.numel() if scratch else 0,
            counters.data_ptr() if scratch else None, counters.numel() if scratch else 0, torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        return out, lse

    return call


# (one, two and four query tiles a workgroup, one part and several)
@pytest.mark.parametrize("H,Sq,Sk,D", [(4, 512, 2048, 64), (5, 130, 1040, 64), (12, 355, 3071, 64), (12, 700, 1401, 64), (2, 65, 33, 64),
                                       (4, 512, 2048, 128), (12, 700, 1401, 128), (9, 990, 222, 128), (3, 33, 31, 128)])
@pytest.mark.parametrize("scratch", [True, False])
@pytest.mark.parametrize("falling", [False, True])
def test_accuracy_of_every_form(hip, H, Sq, Sk, D, scratch, falling):
    """The 2-norm of the error against fp64: 1.6 to 2.4e-7 with all six terms of a product; without the smallest of them, with their
    sums in fp64, 2.2e-6 and more.  The lse is rounded to fp32 (3.4e-8)."""
    g = torch.Generator().manual_seed(Sq + Sk)
    q, k, v = (torch.randn(1, n, H, D, generator=g) for n in (Sq, Sk, Sk))
    out, lse = _c_call(hip, q.cuda(), k.cuda(), v.cuda(), scratch, falling)()
    torch.cuda.synchronize()
    ref_out, ref_lse = om.chunk_attention(q, k, v, compute_dtype=torch.float64)
    error = lambda x, ref: ((x.double().cpu() - ref).norm() / ref.norm()).item()
    assert error(out, ref_out) <= 6e-7 and error(lse, ref_lse) <= 1.5e-7


def test_calls_without_scratch_are_spread_over_the_workgroup(hip):
    """4 heads x 512 x 2048: with one query tile and four groups of keys a workgroup 2.0 times the call that shares keys between
    workgroups, 3.1 times with two query tiles."""
    g = torch.Generator(device="cuda").manual_seed(9)
    q, k, v = (torch.randn(1, n, 4, 64, generator=g, device="cuda") for n in (512, 2048, 2048))
    shared, alone = (_us(_c_call(hip, q, k, v, scratch, False)) for scratch in (True, False))
    assert alone < 2.5 * shared


def test_infinities_in_one_part_of_the_keys(hip):
    """An infinity of V leaves the other columns, and a key of infinite score the other rows, bit for bit what they are."""
    g = torch.Generator().manual_seed(5)
    q = torch.randn(1, 96, 2, 64, generator=g)
    k, v = (torch.randn(1, 1500, 2, 64, generator=g) for _ in range(2))
    [(want, want_lse)] = hip.attn_jobs_f32_fwd(q.cuda(), [k.cuda()], [v.cuda()], [[0]])
    v2 = v.clone()
    v2[0, 1300, 1, 7] = float("-inf")
    [(out, lse)] = hip.attn_jobs_f32_fwd(q.cuda(), [k.cuda()], [v2.cuda()], [[0]])
    want = want.clone()
    want[:, :, 1, 7] = float("-inf")
    assert torch.equal(out, want) and torch.equal(lse, want_lse)


@pytest.mark.parametrize("D", [64, 128])
def test_zeros_split_as_well_as_other_numbers(hip, D):
    """Scores of zero from a row of Q that is zero, and from one that meets a zero column of K: the same numbers on the same way, bit for
    bit; a zero column of V is zero, and the other columns are what they are beside another column."""
    g = torch.Generator().manual_seed(D)
    q, k, v = (torch.randn(1, n, 3, D, generator=g) for n in (130, 700, 700))
    k[..., 3] = 0
    q[:, ::7] = 0
    e3 = q.clone()
    e3[:, ::7, :, 3] = 1
    run = lambda q, v: hip.attn_jobs_f32_fwd(q.cuda(), [k.cuda()], [v.cuda()], [[0]])[0]
    out, lse = run(q, v)
    want, want_lse = run(e3, v)
    assert torch.equal(out, want) and torch.equal(lse, want_lse)
    v0 = v.clone()
    v0[..., 40] = 0
    out, lse = run(e3, v0)
    want = want.clone()
    want[..., 40] = 0
    assert torch.equal(out, want) and torch.equal(lse, want_lse)


@pytest.mark.parametrize("H,Sq,Sk,D", [(12, 1053, 4212, 64), (10, 847, 1694, 128)])
def test_zeros_do_not_send_wavefronts_through_their_keys_again(hip, H, Sq, Sk, D):
    """A padded row of Q in every tile, a padded column of V, padded keys, terms that cancel: as long as without (2.2 to 2.6 times where a
    wavefront computes once more; half as long again is allowed, runs differ by some per cent)."""
    g = torch.Generator(device="cuda").manual_seed(9)
    q, k, v = (torch.randn(1, n, H, D, generator=g, device="cuda") for n in (Sq, Sk, Sk))

    us = lambda q, k, v: _us(lambda: hip.attn_jobs_f32_fwd(q, [k], [v], [[0]]))
    q0, k0, v0, v1 = q.clone(), k.clone(), v.clone(), v.clone()
    q0[:, ::32] = 0
    v0[..., 5] = 0
    k0[:, -Sk // 4:] = 0
    v1[:, -Sk // 4:] = 0
    # in every tile of 32 keys two equal ones, whose V in one column are opposite and the others' zero: a sum of exactly zero
    k2, v2 = k.clone(), v0.clone()
    k2[:, 1::32] = k2[:, 0::32][:, :k2[:, 1::32].shape[1]]
    v2[:, 0::32, :, 5] = 1
    v2[:, 1::32, :, 5] = -1
    v2[:, -(Sk % 32) or Sk:, :, 5] = 0
    assert (hip.attn_jobs_f32_fwd(q, [k2], [v2], [[0]])[0][0][..., 5] == 0).all()
    us(q, k, v)
    plain = us(q, k, v)
    for case in ((q0, k, v), (q, k, v0), (q, k0, v1), (q, k2, v2)):
        assert us(*case) < 1.5 * plain


def test_scores_whose_reference_leaves_the_range(hip):
    """The largest score is finite and the next multiple of the grid above it is not: one key has all the weight."""
    q, k = torch.zeros(1, 40, 1, 64), torch.zeros(1, 70, 1, 64)
    q[..., 3] = 2.0 ** 63
    k[0, 50, 0, 3] = 1.75 * 2.0 ** 63
    v = torch.randn(1, 70, 1, 64, generator=torch.Generator().manual_seed(8))
    [(out, _)] = hip.attn_jobs_f32_fwd(q.cuda(), [k.cuda()], [v.cuda()], [[0]], softmax_scale=8.0)
    assert torch.equal(out.cpu(), v[:, 50:51].expand_as(out))


def test_result_under_graph_capture(hip):
    """Parts, counters and all: every replay equals the eager call, with other launches of the stream between them."""
    g = torch.Generator(device="cuda").manual_seed(6)
    q, k, v = (torch.randn(1, n, 4, 64, generator=g, device="cuda") for n in (200, 2000, 2000))
    run = lambda: hip.attn_jobs_f32_fwd(q, [k], [v], [[0]], lse_bsh=True)[0]
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out, lse = run()
    for i in range(4):
        q.copy_(torch.randn(q.shape, generator=g, device="cuda"))
        graph.replay()
        want, want_lse = run()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(lse, want_lse), i
