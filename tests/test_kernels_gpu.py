"""Parity of the HIP kernels (through the C ABI) against the CPU oracle.

Tolerances (the stated bar): out max-abs <= 2e-2 (bf16), lse <= 1e-3 (fp32).
The tests additionally bound the error relative to the magnitude of the exact
result, because attention outputs over thousands of keys are far smaller than 1.
"""
import math

import numpy as np
import pytest
import torch

from oracle import attention_math as om
from oracle import mask_schedule as ms

pytestmark = pytest.mark.gpu

OUT_TOL = 2e-2
LSE_TOL = 1e-3


def _qkv(B, Sq, Sk, H, D, seed, norm=None):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(B, Sq, H, D, generator=g)
    k = torch.randn(B, Sk, H, D, generator=g)
    v = torch.randn(B, Sk, H, D, generator=g)
    if norm == "rms":
        q = q / q.pow(2).mean(-1, keepdim=True).sqrt()
        k = k / k.pow(2).mean(-1, keepdim=True).sqrt()
    elif norm == "layer":
        q = torch.nn.functional.layer_norm(q, (D,))
        k = torch.nn.functional.layer_norm(k, (D,))
    return q.bfloat16(), k.bfloat16(), v.bfloat16()


def _check_state(out, lse, ref_out, ref_lse, what=""):
    out = out.float().cpu()
    lse = lse.float().cpu()
    err = (out - ref_out).abs().max().item()
    lerr = (lse - ref_lse).abs().max().item()
    rel = (out - ref_out).norm().item() / max(ref_out.norm().item(), 1e-30)
    print(f"{what} out max-abs {err:.3e} rel-l2 {rel:.3e} lse max-abs {lerr:.3e}", flush=True)
    assert err <= OUT_TOL, f"{what}: out max-abs {err}"
    assert lerr <= LSE_TOL, f"{what}: lse max-abs {lerr}"
    assert rel <= 1e-2, f"{what}: out relative l2 {rel}"


@pytest.mark.parametrize("B,Sq,Sk,H,D", [
    (1, 128, 64, 1, 128),
    (1, 128, 128, 2, 128),
    (1, 100, 77, 3, 128),      # ragged Sq and Sk
    (2, 257, 333, 2, 128),     # batch > 1, several tiles, ragged
    (1, 1, 1, 1, 128),         # smallest
    (1, 128, 64, 1, 64),
    (2, 190, 201, 3, 64),
    (1, 33, 1000, 2, 64),
])
def test_chunk_attention_matches_oracle(hip, B, Sq, Sk, H, D):
    print(f"case chunk B={B} Sq={Sq} Sk={Sk} H={H} D={D}", flush=True)
    q, k, v = _qkv(B, Sq, Sk, H, D, seed=B * 1000 + Sq + Sk + D)
    ref_out, ref_lse = om.chunk_attention(q, k, v)
    out, lse = hip.attn_chunk_fwd(q.cuda(), k.cuda(), v.cuda())
    torch.cuda.synchronize()
    _check_state(out, lse, ref_out, ref_lse, "chunk")


@pytest.mark.parametrize("B,Sq,Sk,H,D", [
    (1, 512, 512, 4, 64),      # the CPU-runnable configuration's chunk
    (2, 100, 77, 3, 128),      # ragged queries and keys, batch > 1
    (1, 1, 1, 1, 64),
    (1, 65, 130, 2, 128),
    (1, 33, 0, 2, 64),         # empty chunk: out = 0, lse = -inf
])
def test_fp32_chunk_attention_matches_fp64_closed_form(hip, B, Sq, Sk, H, D):
    """dt_attn_chunk_f32_fwd computes in fp32 from fp32 inputs: it must agree with the closed form in
    fp64 to fp32 rounding error (1e-5), far inside the bar of the bf16 path."""
    g = torch.Generator().manual_seed(Sq * 7 + Sk)
    q = torch.randn(B, Sq, H, D, generator=g) * 1.5
    k = torch.randn(B, Sk, H, D, generator=g)
    v = torch.randn(B, Sk, H, D, generator=g)
    ref_out, ref_lse = om.chunk_attention(q, k, v, compute_dtype=torch.float64)
    out, lse = hip.attn_chunk_f32_fwd(q.cuda(), k.cuda(), v.cuda())
    torch.cuda.synchronize()
    assert out.dtype == torch.float32 and tuple(lse.shape) == (B, H, Sq)
    if Sk == 0:
        assert (out == 0).all() and torch.isinf(lse).all() and (lse < 0).all()
        return
    assert (out.double().cpu() - ref_out).abs().max().item() <= 1e-5
    assert (lse.double().cpu() - ref_lse).abs().max().item() <= 1e-5
    # strided inputs (slices of a fused projection) give the same numbers
    qkv = torch.stack([q, k[:, :Sq] if Sk >= Sq else q, q], dim=2).cuda() if Sk >= Sq else None
    if qkv is not None:
        out2, lse2 = hip.attn_chunk_f32_fwd(qkv[:, :, 0], k.cuda(), v.cuda())
        torch.cuda.synchronize()
        assert torch.equal(out2, out) and torch.equal(lse2, lse)


@pytest.mark.parametrize("B,Sq,H,D,lens,jobs", [
    (1, 97, 2, 64, [33, 1, 0, 128], [[0, 1], [2], [3, 2, 0], [1]]),   # tiles that end inside a chunk, an empty chunk, one key
    (1, 32, 1, 128, [31, 32, 65], [[0, 1, 2], [2]]),
    (2, 1024, 48, 64, [70], [[0]]),                                   # the form without a key split: 3072 query tiles
    (1, 1025, 48, 128, [40, 33], [[0, 1], [1]]),
])
def test_fp32_jobs_match_fp64_closed_form(hip, B, Sq, H, D, lens, jobs):
    """Several fp32 states of one launch, chunks with strides of their own (every second one a slice of a fused
    projection).  Bound as above: 1e-5, fp32 rounding of sums over at most 256 keys."""
    g = torch.Generator().manual_seed(Sq + D)
    q = torch.randn(B, Sq, H, D, generator=g)
    kv = [torch.randn(B, n, 2, H, D, generator=g) for n in lens]
    dev = [t.cuda() if i % 2 else t.transpose(1, 2).contiguous().cuda().transpose(1, 2) for i, t in enumerate(kv)]
    got = hip.attn_jobs_f32_fwd(q.cuda(), [t[:, :, 0] for t in dev], [t[:, :, 1] for t in dev], jobs)
    torch.cuda.synchronize()
    for job, (out, lse) in zip(jobs, got):
        k, v = (torch.cat([kv[c][:, :, i] for c in job], 1) for i in (0, 1))
        if k.shape[1] == 0:
            assert (out == 0).all() and torch.isneginf(lse).all()
            continue
        ref_out, ref_lse = om.chunk_attention(q, k, v, compute_dtype=torch.float64)
        assert (out.double().cpu() - ref_out).abs().max().item() <= 1e-5, job
        assert (lse.double().cpu() - ref_lse).abs().max().item() <= 1e-5, job


@pytest.mark.parametrize("B,Sq,H,D,lens,job", [
    (1, 64, 2, 64, [33], [0]),            # the key behind the last whole tile
    (1, 40, 1, 128, [63, 5], [0, 1]),     # both chunks end inside a tile
    (2, 1024, 48, 64, [70], [0]),         # the form without a key split
    (1, 1025, 48, 128, [40, 97], [1, 0]),
])
def test_fp32_infinite_values_stay_what_the_formula_gives(hip, B, Sq, H, D, lens, job):
    """V holds +inf / -inf in one element of the last key of every chunk: every probability is positive, so that column of the
    output is that infinity and every other one the same as with a finite value there."""
    g = torch.Generator().manual_seed(Sq + D)
    q = torch.randn(B, Sq, H, D, generator=g)
    ks, vs = ([torch.randn(B, n, H, D, generator=g) for n in lens] for _ in range(2))
    dq, dk, dv = q.cuda(), [k.cuda() for k in ks], [v.cuda() for v in vs]
    [(want, want_lse)] = hip.attn_jobs_f32_fwd(dq, dk, dv, [job])
    for i, v in enumerate(dv):
        v[:, -1, :, 3 + i] = float("inf") if i == 0 else float("-inf")
    [(out, lse)] = hip.attn_jobs_f32_fwd(dq, dk, dv, [job])
    want = want.clone()
    for i in range(len(dv)):
        want[..., 3 + i] = float("inf") if i == 0 else float("-inf")
    torch.cuda.synchronize()
    assert torch.equal(out, want) and torch.equal(lse, want_lse)


@pytest.mark.parametrize("B,Sq,H,D,lens,job,dead", [
    (1, 40, 2, 64, [64], [0], [(0, 0, 32)]),                  # the first tile of one wavefront's keys, the second is another's
    (1, 33, 1, 128, [300, 70], [0, 1], [(0, 0, 40), (0, 128, 160), (1, 32, 70)]),
    (2, 1024, 48, 64, [64], [0], [(0, 0, 32)]),               # the form without a key split
    (2, 1024, 48, 64, [64], [0], [(0, 0, 64)]),               # no key at all is left
])
def test_fp32_scores_of_minus_infinity_weigh_nothing(hip, B, Sq, H, D, lens, job, dead):
    """Whole key tiles whose scores are -inf (their K overflows against a positive q) leave the softmax over the other keys,
    to the 1e-5 of fp32 sums; rows without any other key get the empty state."""
    g = torch.Generator().manual_seed(Sq + D)
    q = torch.randn(B, Sq, H, D, generator=g)
    q[..., 0] = q[..., 0].abs() + 2.0
    ks, vs = ([torch.randn(B, n, H, D, generator=g) for n in lens] for _ in range(2))
    keep = [torch.ones(n, dtype=torch.bool) for n in lens]
    for c, a, b in dead:
        ks[c][:, a:b] = 0.0
        ks[c][:, a:b, :, 0] = float("-inf")
        keep[c][a:b] = False
    [(out, lse)] = hip.attn_jobs_f32_fwd(q.cuda(), [k.cuda() for k in ks], [v.cuda() for v in vs], [job])
    if not any(k.any() for k in keep):
        assert (out == 0).all() and torch.isneginf(lse).all()
        return
    k, v = (torch.cat([t[c][:, keep[c]] for c in job], 1) for t in (ks, vs))
    rows = torch.arange(0, Sq, max(1, Sq // 64))
    ref_out, ref_lse = om.chunk_attention(q[:, rows], k, v, compute_dtype=torch.float64)
    assert (out[:, rows.cuda()].double().cpu() - ref_out).abs().max().item() <= 1e-5
    assert (lse[:, :, rows.cuda()].double().cpu() - ref_lse).abs().max().item() <= 1e-5


def test_fp32_token_strides_beyond_32_bits(hip):
    """Keys 2^30 elements apart (4 GiB), in tiles that end inside the chunk and in whole ones: the same states as from a
    dense copy."""
    Sk, D, stride = 33, 64, 2 ** 30
    need = (Sk - 1) * stride + 2 * D
    if torch.cuda.mem_get_info()[0] < 4 * need + (32 << 30):
        pytest.skip("needs 160 GiB of device memory")
    g = torch.Generator().manual_seed(30)
    q = torch.randn(1, 40, 1, D, generator=g).cuda()
    kv = torch.randn(2, 1, Sk, 1, D, generator=g).cuda()
    far = torch.empty(need, device="cuda")
    try:
        k, v = (far.as_strided((1, Sk, 1, D), (Sk * stride, stride, D, 1), i * D) for i in (0, 1))
        k.copy_(kv[0])
        v.copy_(kv[1])
        [(out, lse)] = hip.attn_jobs_f32_fwd(q, [k], [v], [[0]])
        [(want, want_lse)] = hip.attn_jobs_f32_fwd(q, [kv[0]], [kv[1]], [[0]])
        assert torch.equal(out, want) and torch.equal(lse, want_lse)
    finally:
        del far, k, v
        torch.cuda.empty_cache()


def test_chunk_attention_strided_inputs(hip):
    """q/k/v as slices of a fused [B,S,3,H,D] projection (non-contiguous token stride)."""
    B, S, H, D = 1, 300, 2, 128
    g = torch.Generator().manual_seed(5)
    qkv = torch.randn(B, S, 3, H, D, generator=g).bfloat16()
    q, k, v = qkv[:, :, 0], qkv[:, :, 1], qkv[:, :, 2]
    ref_out, ref_lse = om.chunk_attention(q, k, v)
    dq = qkv.cuda()
    out, lse = hip.attn_chunk_fwd(dq[:, :, 0], dq[:, :, 1], dq[:, :, 2])
    torch.cuda.synchronize()
    _check_state(out, lse, ref_out, ref_lse, "strided")


def test_multi_chunk_job_equals_merge_of_chunks(hip):
    """One job over several chunks == folding per-chunk states with update_out_and_lse."""
    B, Sq, H, D = 1, 200, 2, 128
    lens = [64, 130, 0, 77, 1]
    g = torch.Generator().manual_seed(11)
    q = torch.randn(B, Sq, H, D, generator=g).bfloat16()
    ks = [torch.randn(B, n, H, D, generator=g).bfloat16() for n in lens]
    vs = [torch.randn(B, n, H, D, generator=g).bfloat16() for n in lens]
    # oracle: literal fold
    o = l = None
    for k, v in zip(ks, vs):
        if k.shape[1] == 0:
            continue
        bo, bl = om.chunk_attention(q, k, v)
        o, l = om.update_out_and_lse(o, l, bo.bfloat16(), bl)
    ref_out, ref_lse = o, l.squeeze(-1).transpose(1, 2)
    full_out, full_lse = om.full_attention(q, ks, vs)
    assert (full_out - ref_out).abs().max() < 5e-3  # the fold itself is pinned by full attention

    dq = q.cuda()
    table = hip.ChunkTable([k.cuda() for k in ks], [v.cuda() for v in vs])
    outs = [torch.empty(B, Sq, H, D, dtype=torch.bfloat16, device="cuda") for _ in range(3)]
    lses = [torch.empty(B, H, Sq, dtype=torch.float32, device="cuda") for _ in range(3)]
    hip.attn_jobs_fwd(dq, table, [[0, 1, 2, 3, 4], [3], [2]], outs, lses)
    torch.cuda.synchronize()
    _check_state(outs[0], lses[0], full_out, full_lse, "job all chunks")
    r3o, r3l = om.chunk_attention(q, ks[3], vs[3])
    _check_state(outs[1], lses[1], r3o, r3l, "job chunk 3")
    # a job whose only chunk is empty yields the neutral state
    assert torch.isinf(lses[2]).all() and (lses[2] < 0).all()
    assert (outs[2].float() == 0).all()


@pytest.mark.parametrize("D,n,src_fp32", [(128, 1, False), (128, 5, False), (64, 8, False), (128, 3, True), (64, 33, False),
                                          (128, 6, False), (128, 7, True), (64, 9, True), (64, 4, False), (64, 7, False), (128, 8, False)])
def test_merge_states_matches_closed_form(hip, D, n, src_fp32):
    B, Sq, H = 2, 150, 3
    g = torch.Generator().manual_seed(n * 7 + D)
    outs = [torch.randn(B, Sq, H, D, generator=g) for _ in range(n)]
    lses = [torch.randn(B, H, Sq, generator=g) * 3 for _ in range(n)]
    if n >= 3:
        lses[1][:, :, ::5] = -math.inf   # partially empty state
    if not src_fp32:
        outs = [o.bfloat16() for o in outs]
    ref_out, ref_lse = om.merge_states_closed_form(outs, lses)
    d_out, d_lse = hip.merge_states([o.cuda() for o in outs], [l.cuda() for l in lses])
    torch.cuda.synchronize()
    assert (d_out.cpu() - ref_out).abs().max() < 1e-5 * max(1, n)
    assert (d_lse.cpu() - ref_lse).abs().max() < 1e-5
    # literal sigmoid/logsigmoid fold of the reference agrees with the fused kernel
    o = l = None
    for bo, bl in zip(outs, lses):
        o, l = om.update_out_and_lse(o, l, bo, bl)
    finite = torch.isfinite(l.squeeze(-1).transpose(1, 2))
    assert (d_lse.cpu()[finite] - l.squeeze(-1).transpose(1, 2)[finite]).abs().max() < 1e-4


def test_merge_all_empty_and_layouts(hip):
    B, Sq, H, D = 1, 70, 2, 128
    g = torch.Generator().manual_seed(3)
    outs = [torch.randn(B, Sq, H, D, generator=g).bfloat16() for _ in range(2)]
    lses = [torch.full((B, H, Sq), -math.inf) for _ in range(2)]
    d_out, d_lse = hip.merge_states([o.cuda() for o in outs], [l.cuda() for l in lses])
    torch.cuda.synchronize()
    assert (d_out == 0).all() and torch.isinf(d_lse).all()
    # running layout [B,S,H,1] in, [B,S,H,1] out, bf16 destination, in place
    lses = [torch.randn(B, H, Sq, generator=g) for _ in range(2)]
    ref_out, ref_lse = om.merge_states_closed_form(outs, lses)
    a_out = outs[0].cuda()
    a_lse = lses[0].transpose(1, 2).contiguous().unsqueeze(-1).cuda()   # [B,S,H,1]
    b_out, b_lse = outs[1].cuda(), lses[1].cuda()
    r_out, r_lse = hip.merge_states([a_out, b_out], [a_lse, b_lse], dst_out=a_out, dst_lse=a_lse)
    torch.cuda.synchronize()
    assert r_out.data_ptr() == a_out.data_ptr()
    assert (a_out.float().cpu() - ref_out).abs().max() < 2e-2
    assert (a_lse.cpu().squeeze(-1).transpose(1, 2) - ref_lse).abs().max() < 1e-5


@pytest.mark.parametrize("B,Sq,H", [(1, 77, 5), (2, 150, 8), (1, 37, 24), (1, 19, 48), (3, 9, 16)])
@pytest.mark.parametrize("D,n", [(64, 2), (64, 8), (128, 3), (128, 8), (128, 17)])
def test_merge_row_mappings(hip, B, Sq, H, D, n):
    """The merge hands rows to workgroups in memory order or as tiles of queries x heads, depending on the
    head count, the head dimension and the number of states; at D = 64 two neighbouring rows share a lane
    group.  Head counts that do and do not divide into tiles, an odd row count, query counts that leave
    partial tiles; fp32 and bf16 destinations; one state fp32, one lse in the [B,S,H,1] layout."""
    g = torch.Generator().manual_seed(B * 1000 + Sq * 10 + H + D + n)
    outs = [torch.randn(B, Sq, H, D, generator=g).bfloat16() for _ in range(n)]
    lses = [torch.randn(B, H, Sq, generator=g) * 3 for _ in range(n)]
    lses[0][:, :, ::4] = -math.inf
    lses[n - 1][:, ::2, :] = -math.inf
    ref_out, ref_lse = om.merge_states_closed_form([o.float() for o in outs], lses)
    d_outs = [o.cuda() for o in outs]
    d_lses = [l.cuda() for l in lses]
    def lse_close(got, tol=1e-5):   # rows without any state keep -inf
        fin = torch.isfinite(ref_lse)
        return bool((got[~fin] == ref_lse[~fin]).all()) and float((got[fin] - ref_lse[fin]).abs().max()) < tol

    o, l = hip.merge_states(d_outs, d_lses)
    torch.cuda.synchronize()
    assert (o.cpu() - ref_out).abs().max() < 1e-5 * n and lse_close(l.cpu())
    d_outs[1] = d_outs[1].float()
    d_lses[n - 1] = d_lses[n - 1].transpose(1, 2).contiguous().unsqueeze(-1)
    dst_l = torch.empty(B, Sq, H, 1, device="cuda")
    o2, l2 = hip.merge_states(d_outs, d_lses, dst_dtype=torch.bfloat16, dst_lse=dst_l)
    torch.cuda.synchronize()
    assert l2.data_ptr() == dst_l.data_ptr()
    assert (o2.float().cpu() - ref_out).abs().max() <= 2.0 ** -8 * float(ref_out.abs().max())
    assert lse_close(dst_l.cpu().squeeze(-1).transpose(1, 2))


@pytest.mark.parametrize("D,H", [(64, 8), (128, 4), (128, 3)])
@pytest.mark.parametrize("order", ["ascending", "descending", "spiky"])
def test_merge_rescales_across_batches(hip, D, H, order):
    """States are folded in batches of 8 with a running maximum.  lse values that grow (every batch rescales what was
    accumulated), shrink (later batches underflow to nothing) or jump by +-60 between neighbours: against the closed
    form in fp64."""
    B, Sq, n = 1, 41, 29
    g = torch.Generator().manual_seed(17 + D + H)
    outs = [torch.randn(B, Sq, H, D, generator=g).bfloat16() for _ in range(n)]
    base = torch.randn(B, H, Sq, generator=g)
    if order == "ascending":
        lses = [base + 7.0 * i for i in range(n)]
    elif order == "descending":
        lses = [base - 7.0 * i for i in range(n)]
    else:
        lses = [base + (60.0 if i % 3 == 0 else -60.0 if i % 3 == 1 else 0.0) + torch.randn(B, H, Sq, generator=g) for i in range(n)]
    lw = torch.stack([l.double() for l in lses])                       # [n,B,H,Sq]
    ref_lse = torch.logsumexp(lw, 0)
    w = torch.exp(lw - ref_lse).permute(0, 1, 3, 2).unsqueeze(-1)      # [n,B,Sq,H,1]
    ref_out = (w * torch.stack([o.double() for o in outs])).sum(0)
    o, l = hip.merge_states([x.cuda() for x in outs], [x.cuda() for x in lses])
    torch.cuda.synchronize()
    assert (l.cpu().double() - ref_lse).abs().max() < 1e-4 * max(1.0, float(ref_lse.abs().max()) / 16)
    assert (o.cpu().double() - ref_out).abs().max() < 1e-5


def test_merge_large_launch_d64(hip):
    """A D = 64 launch of more than 2^20 lane groups takes two tile passes per workgroup."""
    B, Sq, H, D, n = 1, 16400, 128, 64, 2
    g = torch.Generator(device="cuda").manual_seed(5)
    outs = [torch.randn(B, Sq, H, D, generator=g, device="cuda").bfloat16() for _ in range(n)]
    lses = [torch.randn(B, H, Sq, generator=g, device="cuda") * 2 for _ in range(n)]
    o, l = hip.merge_states(outs, lses)
    torch.cuda.synchronize()
    rows = torch.randperm(Sq)[:257]
    ref_out, ref_lse = om.merge_states_closed_form([x[:, rows].float().cpu() for x in outs],
                                                   [x[:, :, rows].cpu() for x in lses])
    assert (o[:, rows].cpu() - ref_out).abs().max() < 1e-5 and (l[:, :, rows].cpu() - ref_lse).abs().max() < 1e-5
    # every row was written: the lse of all rows against torch's logaddexp
    assert (l - torch.logaddexp(lses[0], lses[1])).abs().max() < 1e-5


@pytest.mark.parametrize("D", [64, 128])
def test_merge_many_states_in_place_with_row_layout_lse(hip, D):
    """Six states and more take the kernel's other row-to-workgroup mapping: in place into the first
    state (bf16 destination), lse of that state in the running [B,S,H,1] layout, a repeated pointer."""
    B, Sq, H, n = 2, 77, 5, 7
    g = torch.Generator().manual_seed(D)
    outs = [torch.randn(B, Sq, H, D, generator=g).bfloat16() for _ in range(n)]
    lses = [torch.randn(B, H, Sq, generator=g) * 2 for _ in range(n)]
    lses[3][:, :, 1::3] = -math.inf
    ref_out, ref_lse = om.merge_states_closed_form(outs + [outs[2]], lses + [lses[2]])
    d_outs = [o.cuda() for o in outs]
    d_lses = [l.cuda() for l in lses]
    a_lse = lses[0].transpose(1, 2).contiguous().unsqueeze(-1).cuda()
    hip.merge_states(d_outs + [d_outs[2]], [a_lse] + d_lses[1:] + [d_lses[2]], dst_out=d_outs[0], dst_lse=a_lse)
    torch.cuda.synchronize()
    assert (d_outs[0].float().cpu() - ref_out).abs().max() < 2e-2
    assert (a_lse.cpu().squeeze(-1).transpose(1, 2) - ref_lse).abs().max() < 1e-5


@pytest.mark.parametrize("B,Sq,H,D", [(2, 131, 3, 64), (2, 131, 8, 64), (1, 19, 48, 64), (3, 77, 16, 128), (1, 5, 5, 128)])
def test_cache_store_load_roundtrip(hip, B, Sq, H, D):
    """fp32 state with a [B,S,H,1] lse -> slot -> fp32.  At D = 64 head counts that divide into tiles of 8 heads
    take the kernel that moves two neighbouring rows per lane group, the others the row-mapped one."""
    g = torch.Generator().manual_seed(9 + H)
    src = torch.randn(B, Sq, H, D, generator=g)
    lse = torch.randn(B, Sq, H, 1, generator=g)
    slot_out = torch.empty(B, Sq, H, D, dtype=torch.bfloat16, device="cuda")
    slot_lse = torch.empty(B, H, Sq, dtype=torch.float32, device="cuda")
    hip.cache_store(src.cuda(), lse.cuda(), slot_out, slot_lse)
    torch.cuda.synchronize()
    assert torch.equal(slot_out.cpu(), src.bfloat16())            # round-to-nearest-even, bit exact
    assert torch.equal(slot_lse.cpu(), lse.squeeze(-1).transpose(1, 2))
    o, l = hip.cache_load(slot_out, slot_lse, torch.float32, dst_lse_bsh=True)
    torch.cuda.synchronize()
    assert torch.equal(o.cpu(), src.bfloat16().float())
    assert torch.equal(l.cpu(), lse)


@pytest.mark.parametrize("B,Sq,H,D", [(1, 1, 1, 64), (2, 131, 3, 64), (1, 64, 24, 128), (3, 700, 7, 128), (1, 65, 300, 64),
                                      (2, 1000, 48, 64)])
@pytest.mark.parametrize("lse_bsh", [False, True])
def test_cache_load_widens_bit_exactly_in_both_lse_layouts(hip, B, Sq, H, D, lse_bsh):
    """bf16 slot -> fp32 state: the flat widening pass and the lse's trip through the LDS (runs of 64 query
    positions x all heads; fewer positions per run above 256 heads), ragged last run included."""
    g = torch.Generator().manual_seed(B * 1000 + Sq + H)
    slot_out = torch.randn(B, Sq, H, D, generator=g).bfloat16()
    slot_lse = torch.randn(B, H, Sq, generator=g)
    slot_lse[0, 0, 0] = float("-inf")
    o, l = hip.cache_load(slot_out.cuda(), slot_lse.cuda(), torch.float32, dst_lse_bsh=lse_bsh)
    torch.cuda.synchronize()
    assert torch.equal(o.cpu(), slot_out.float())
    want = slot_lse.transpose(1, 2).unsqueeze(-1).contiguous() if lse_bsh else slot_lse
    assert l.shape == want.shape and torch.equal(l.cpu(), want)


@pytest.mark.parametrize("B,Sq,H,D", [(1, 1, 1, 64), (2, 131, 3, 64), (1, 77, 3, 128), (1, 2222, 5, 64), (3, 700, 7, 128)])
def test_same_format_copies_are_bit_exact(hip, B, Sq, H, D):
    """State copies whose two sides share dtype and lse layout take the flat-range path: slot -> slot
    (bf16 / [B,H,S]) and fp32 -> fp32 loads in either lse layout, with sizes that are no multiple of the
    4 KB a wavefront moves, destinations inside larger buffers (nothing outside the state may be
    written) and lse slices that are not 16-byte aligned."""
    g = torch.Generator().manual_seed(B * 1000 + Sq)
    rows = B * Sq * H
    src_o = torch.randn(B, Sq, H, D, generator=g).bfloat16().cuda()
    src_l = torch.randn(B, H, Sq, generator=g).cuda()
    # destinations: slices of poisoned arenas, so that a write outside the state shows
    pad = 3
    arena_o = torch.full((3, B, Sq, H, D), 7.0, dtype=torch.bfloat16, device="cuda")
    arena_l = torch.full((3 * rows + 2 * pad,), 7.0, dtype=torch.float32, device="cuda")
    dst_l = arena_l[rows + pad: 2 * rows + pad].view(B, H, Sq)          # 12 bytes off a 16-byte boundary (for odd sizes)
    hip.cache_store(src_o, src_l, arena_o[1], dst_l)
    torch.cuda.synchronize()
    assert torch.equal(arena_o[1], src_o) and torch.equal(dst_l, src_l)
    assert (arena_o[0].float() == 7).all() and (arena_o[2].float() == 7).all()
    assert (arena_l[:rows + pad] == 7).all() and (arena_l[2 * rows + pad:] == 7).all()
    back_o, back_l = hip.cache_load(arena_o[1], dst_l.contiguous(), torch.bfloat16, dst_lse_bsh=False)
    torch.cuda.synchronize()
    assert torch.equal(back_o, src_o) and torch.equal(back_l, src_l)


@pytest.mark.parametrize("T,L,C,p,diag", [(3, 4, 8, 0.5, 0), (2, 3, 32, 0.9, -1), (2, 2, 1, 0.5, 0), (1, 2, 100, 0.3, 77), (2, 2, 64, 0.0, 3), (1, 1, 65, 1.0, 64)])
def test_schedule_builder_bit_exact(hip, T, L, C, p, diag):
    mask = ms.seeded_mask(T, L, C, p, seed=C + T, diag=diag, cold_first_step=False)
    comp, reu, cnt = ms.build_schedule_table(mask, diag)
    dmask = torch.from_numpy(mask).cuda()
    dcomp, dreu, dcnt = hip.build_schedule_table(dmask, diag)
    torch.cuda.synchronize()
    assert np.array_equal(dcomp.cpu().numpy(), comp)
    assert np.array_equal(dreu.cpu().numpy(), reu)
    assert np.array_equal(dcnt.cpu().numpy(), cnt)
    t, l = T - 1, L - 1
    c1, r1, n1 = hip.build_schedule(dmask, t, l, diag)
    torch.cuda.synchronize()
    assert np.array_equal(c1.cpu().numpy(), comp[t, l])
    assert np.array_equal(r1.cpu().numpy(), reu[t, l])
    assert np.array_equal(n1.cpu().numpy(), cnt[t, l])


def test_rel_l1_sums(hip):
    g = torch.Generator().manual_seed(2)
    a = torch.randn(1, 77, 3, 64, generator=g)
    b = a + 0.05 * torch.randn(1, 77, 3, 64, generator=g)
    a[0, 3, 1, 5] = float("nan")
    b[0, 9, 2, 7] = float("nan")
    ref = om.rel_l1(a, b)
    s = hip.rel_l1_sums(a.cuda(), b.cuda()).cpu()
    val = (s[0] / s[3]).item() / ((s[2] / s[3]).item() + 1e-8)
    assert s[3].item() == a.numel() - 2
    assert abs(val - ref) < 1e-5 * max(1.0, abs(ref))


@pytest.mark.parametrize("case", ["ramp", "huge", "late_outlier", "descending"])
def test_chunk_attention_with_drifting_maximum(hip, case):
    """The kernel keeps a reference maximum that may lag behind the true row maximum and only
    redoes a tile when its row sum overflows a bound: drive that logic with scores that grow
    steadily along the keys, scores of huge magnitude, and one dominant key at the very end."""
    B, Sq, Sk, H, D = 1, 130, 1000, 2, 128
    g = torch.Generator().manual_seed(42)
    q = torch.randn(B, Sq, H, D, generator=g)
    k = torch.randn(B, Sk, H, D, generator=g)
    v = torch.randn(B, Sk, H, D, generator=g)
    qdir = q / q.norm(dim=-1, keepdim=True)
    if case == "ramp":          # score of key j grows linearly from about -40 to +40
        ramp = torch.linspace(-40, 40, Sk).view(1, Sk, 1, 1) * math.sqrt(D)
        k = 0.1 * k + ramp * qdir.mean(dim=1, keepdim=True) / qdir.mean(dim=1, keepdim=True).norm(dim=-1, keepdim=True)
        q = qdir.mean(dim=1, keepdim=True).expand_as(q) / qdir.mean(dim=1, keepdim=True).norm(dim=-1, keepdim=True) + 0.05 * q
    elif case == "descending":  # the first tile holds the maximum, later probabilities shrink to nothing
        ramp = torch.linspace(40, -40, Sk).view(1, Sk, 1, 1) * math.sqrt(D)
        d0 = qdir.mean(dim=1, keepdim=True) / qdir.mean(dim=1, keepdim=True).norm(dim=-1, keepdim=True)
        k = 0.1 * k + ramp * d0
        q = d0.expand_as(q) + 0.05 * q
    elif case == "huge":        # natural-log scores of magnitude in the hundreds
        q = q * 6
        k = k * 6
    elif case == "late_outlier":
        k[:, -1] = 30 * qdir[:, 7]
    q, k, v = q.bfloat16(), k.bfloat16(), v.bfloat16()
    ref_out, ref_lse = om.chunk_attention(q, k, v, compute_dtype=torch.float64)
    out, lse = hip.attn_chunk_fwd(q.cuda(), k.cuda(), v.cuda())
    torch.cuda.synchronize()
    assert torch.isfinite(out.float()).all() and torch.isfinite(lse).all()
    err = (out.float().cpu() - ref_out.float()).abs().max().item()
    lerr = ((lse.cpu().double() - ref_lse).abs() / ref_lse.abs().clamp_min(1.0)).max().item()
    print(f"{case}: out max-abs {err:.3e}, lse max rel/abs {lerr:.3e}, lse range [{ref_lse.min():.1f}, {ref_lse.max():.1f}]", flush=True)
    assert err <= OUT_TOL
    assert lerr <= LSE_TOL


@pytest.mark.parametrize("D", [128, 64])
def test_short_work_items_repeat_bit_exactly(hip, D):
    """Work items of two key tiles, many per launch, many launches on K/V just copied in from the host: every launch
    must return the bits of the first one, and the first one the oracle's numbers.

    With two tiles the trailing half of a workgroup has no softmax phase of its own before the leading
    half reads K of the second tile, so its share of that tile needs a wait of its own: the loads were
    issued long before and nearly always land in time, which is why only repetition shows a missing one
    (some rows of one head lose a few per cent of their softmax mass, about once in 40 000 work items)."""
    B, Sq, H, Sk, n_chunks, launches = 1, 90, 3, 90, 40, 2500
    g = torch.Generator().manual_seed(90 + D)
    q = torch.randn(B, Sq, H, D, generator=g).bfloat16()
    k_all = torch.randn(n_chunks, B, Sk, H, D, generator=g).bfloat16()
    v_all = torch.randn(n_chunks, B, Sk, H, D, generator=g).bfloat16()
    dq = q.cuda()
    jobs = [[c] for c in range(n_chunks)]

    def launch():
        dk, dv = k_all.cuda(), v_all.cuda()      # copied by the DMA engine: in no cache of the GPU, new addresses
        table = hip.ChunkTable(list(dk.unbind(0)), list(dv.unbind(0)))
        out = torch.empty(n_chunks, B, Sq, H, D, dtype=torch.bfloat16, device="cuda")
        lse = torch.empty(n_chunks, B, H, Sq, dtype=torch.float32, device="cuda")
        hip.attn_jobs_fwd(dq, table, jobs, list(out.unbind(0)), list(lse.unbind(0)))
        return out, lse, (dk, dv)

    out0, lse0, _ = launch()
    torch.cuda.synchronize()
    for c in (0, 17, n_chunks - 1):
        ref_out, ref_lse = om.chunk_attention(q, k_all[c], v_all[c])
        _check_state(out0[c], lse0[c], ref_out, ref_lse, f"chunk {c}")
    differing = torch.zeros((), dtype=torch.int64, device="cuda")
    keep = []                                                   # a few generations stay allocated: addresses vary
    for i in range(launches):
        out, lse, kv = launch()
        differing += ((out != out0).flatten(1).any(1) | (lse != lse0).flatten(1).any(1)).sum()
        keep.append(kv)
        if len(keep) > (i % 7) + 1:
            keep.clear()
    torch.cuda.synchronize()
    assert int(differing) == 0, f"{int(differing)} chunk states of {launches * n_chunks} differ from the first launch"


def test_scheduled_launch_with_split_tail_and_merge_repeat_bit_exactly(hip):
    """The device-scheduled launch with its tail run as parts, the fold kernel behind it and the merge of the
    resulting states, 150 times on K/V just copied in from the host: every repetition returns the bits of
    the first (the kernels share nothing but the workspace, and its users are ordered on the stream)."""
    B, H, D, Sq, lens, diag = 1, 24, 128, 3000, [2000, 1500, 1800], 1
    C = len(lens)
    g = torch.Generator().manual_seed(77)
    q = torch.randn(B, Sq, H, D, generator=g).bfloat16()
    ks = [torch.randn(B, n, H, D, generator=g).bfloat16() for n in lens]
    vs = [torch.randn(B, n, H, D, generator=g).bfloat16() for n in lens]
    ids = torch.arange(C, dtype=torch.int32, device="cuda")
    cnt = torch.tensor([C], dtype=torch.int32, device="cuda")
    ws = hip.attn_workspace("cuda")
    dq = q.cuda()

    def run():
        dk, dv = [k.cuda() for k in ks], [v.cuda() for v in vs]
        so = torch.zeros(C, B, Sq, H, D, dtype=torch.bfloat16, device="cuda")
        sl = torch.zeros(C, B, H, Sq, device="cuda")
        do = torch.zeros(B, Sq, H, D, dtype=torch.bfloat16, device="cuda")
        dl = torch.zeros(B, H, Sq, device="cuda")
        hip.attn_sched_fwd(dq, hip.ChunkTable(dk, dv), ids, cnt, C, so, sl, diag, do, dl, workspace=ws)
        out, lse = hip.merge_states([so[c] if c != diag else do for c in range(C)],
                                    [sl[c] if c != diag else dl for c in range(C)])
        return so, sl, do, dl, out, lse

    first = run()
    torch.cuda.synchronize()
    full_out, full_lse = om.full_attention(q, ks, vs)
    _check_state(first[4], first[5], full_out, full_lse, "merged")
    differing = torch.zeros((), dtype=torch.int64, device="cuda")
    for _ in range(150):
        for a, b in zip(run(), first):
            differing += (a != b).any().long()
    torch.cuda.synchronize()
    assert int(differing) == 0


def test_rel_l1_sums_at_the_hunyuan_shape(hip):
    """The profiling mode's reduction over two fp32 outputs of the HunyuanVideo per-rank shape (45.7 M elements each,
    a few NaN among them) against the oracle's rel_l1 on the host."""
    B, S, H, D = 1, 14882, 24, 128
    g = torch.Generator(device="cuda").manual_seed(31)
    a = torch.randn(B, S, H, D, generator=g, device="cuda")
    b = a + 0.05 * torch.randn(B, S, H, D, generator=g, device="cuda")
    a[0, 7, 3, 5] = float("nan")
    b[0, 9000, 20, 100] = float("nan")
    sums = hip.rel_l1_sums(b, a).cpu()
    torch.cuda.synchronize()
    d, sa, sb, cnt = [float(x) for x in sums]
    assert cnt == a.numel() - 2
    got = (d / cnt) / (sb / cnt + 1e-8)                 # mean|new - ori| / (mean|ori| + 1e-8), new = b, ori = a
    want = om.rel_l1(b.cpu(), a.cpu())
    assert abs(got - want) <= 1e-5 * want


@pytest.mark.parametrize("rows", [1, 12288, 12289, 65536, 65537])
def test_running_state_from_one_row_to_256_mib(hip, rows):
    """fp32 destinations of one state and of an update, from one row to 256 MiB (65536 rows of 8 heads of 128) and a row more."""
    from ditango_amd.utils import update_out_and_lse
    g = torch.Generator(device="cuda:0").manual_seed(rows)
    blocks = [(torch.randn(1, rows, 8, 128, generator=g, device="cuda:0").bfloat16(), torch.randn(1, 8, rows, generator=g, device="cuda:0"))
              for _ in range(2)]
    out, lse = update_out_and_lse(None, None, *blocks[0])
    assert torch.equal(out, blocks[0][0].float())
    torch.testing.assert_close(lse[..., 0], blocks[0][1].transpose(1, 2), rtol=0, atol=1e-6)   # one exp / log pair of fp32
    out, lse = update_out_and_lse(out, lse, *blocks[1])
    w = torch.sigmoid(blocks[1][1] - blocks[0][1]).transpose(1, 2).unsqueeze(-1)
    ref = blocks[0][0].float() * (1 - w) + blocks[1][0].float() * w
    torch.testing.assert_close(out, ref, rtol=2e-6, atol=4e-6)   # the weights carry a few ulp, the terms are below 6
    torch.testing.assert_close(lse[..., 0], torch.logaddexp(blocks[0][1], blocks[1][1]).transpose(1, 2), rtol=0, atol=2e-6)


@pytest.mark.parametrize("B,Sq,H,D", [(1, 1, 1, 64), (1, 1, 1, 128), (3, 7, 1, 64), (1, 1, 37, 128), (2, 5, 3, 128), (1, 300, 7, 64),
                                      (1, 523, 24, 128), (2, 1031, 48, 64)])
@pytest.mark.parametrize("layouts", [(1, 0, 1), (0, 1, 0), (1, 1, 1)])
def test_running_state_and_a_block(hip, B, Sq, H, D, layouts):
    """The update of an fp32 running state has a kernel of its own: one row, one head, one query, odd counts, enough workgroups
    for their reordering and a remainder behind it; every lse layout; empty rows on either side and on both; in place.
    Against the closed form in 64 bits: three roundings of fp32 an element (2^-22 of the largest, here below 8) and the exp's."""
    gen = torch.Generator().manual_seed(B + Sq * 3 + H * 5 + D)
    for dtype in (torch.bfloat16, torch.float16):
        run, blk = torch.randn(B, Sq, H, D, generator=gen), torch.randn(B, Sq, H, D, generator=gen).to(dtype)
        lses = [4 * torch.randn(B, H, Sq, generator=gen) for _ in range(2)]
        lses[0][:, :, ::3] = -math.inf
        lses[1][:, :, ::2] = -math.inf
        store = lambda l, bsh: (l.transpose(1, 2).contiguous().unsqueeze(-1) if bsh else l).cuda()
        w = torch.stack(lses).double()
        ref_lse = torch.logsumexp(w, 0)
        p = torch.nan_to_num(torch.exp(w - ref_lse)).permute(0, 1, 3, 2).unsqueeze(-1)
        ref = p[0] * run.double() + p[1] * blk.double()
        for in_place in (False, True):
            d_run, d_lse = run.cuda(), store(lses[0], layouts[0])
            out, lse = (d_run, d_lse) if in_place else (torch.full_like(d_run, math.nan), store(torch.zeros(B, H, Sq), layouts[2]))
            hip.merge_states([d_run, blk.cuda()], [d_lse, store(lses[1], layouts[1])], dst_out=out, dst_lse=lse)
            got = (lse.squeeze(-1).transpose(1, 2) if lse.dim() == 4 else lse).cpu().double()
            assert (out.cpu().double() - ref).abs().max() <= 4e-6
            none = torch.isinf(ref_lse)
            assert (got[none] == -math.inf).all()
            assert torch.where(none, 0.0, got - ref_lse).abs().max() <= 4e-6


@pytest.mark.parametrize("rows_less", [0, 8])
def test_running_state_of_64_gib(hip, rows_less):
    """The largest state that the update's own kernel has lanes for, and the first that goes to the general one, in place.
    Constant values: both weights are 1/2 to the last bits, the result is 1.5."""
    H, D, Sq = 1, 128, (1 << 27) - rows_less
    need = Sq * (6 * D + 8)
    if torch.cuda.mem_get_info()[0] < need + (4 << 30):
        torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < need + (4 << 30):
        pytest.skip("needs 104 GiB of free GPU memory")
    run = torch.full((1, Sq, H, D), 1.0, device="cuda")
    blk = torch.full((1, Sq, H, D), 2.0, dtype=torch.bfloat16, device="cuda")
    run_lse = torch.zeros(1, Sq, H, 1, device="cuda")
    blk_lse = torch.zeros(1, H, Sq, device="cuda")
    hip.merge_states([run, blk], [run_lse, blk_lse], dst_out=run, dst_lse=run_lse)
    for got, want in ((run, 1.5), (run_lse, 0.6931472)):
        assert abs(got.amin().item() - want) <= 1e-6 and abs(got.amax().item() - want) <= 1e-6
    del run, blk
    torch.cuda.empty_cache()


@pytest.mark.parametrize("B,Sq,H,D", [(1, 1, 1, 64), (1, 1, 1, 128), (3, 7, 1, 64), (1, 1, 37, 128), (2, 5, 3, 128), (1, 300, 7, 64),
                                      (1, 2185, 30, 128), (1, 4369, 15, 64), (2, 2048, 16, 64), (1, 4096, 16, 128)])
@pytest.mark.parametrize("bsh", [True, False])
def test_states_convert_exactly(hip, B, Sq, H, D, bsh):
    """fp32 states rounded and 16-bit ones widened, either lse layout outside the cache: one row, one head, one query, odd counts, the last sizes of
    short loads (65 535 rows) and the first of longer ones.  One rounding to nearest, and exact widening: bits as torch's."""
    gen = torch.Generator().manual_seed(B + Sq * 3 + H * 5 + D)
    store = lambda l, bsh: (l.transpose(1, 2).contiguous().unsqueeze(-1) if bsh else l).cuda()
    wide, lse = torch.randn(B, Sq, H, D, generator=gen), 4 * torch.randn(B, H, Sq, generator=gen)
    lse[:, :, ::3] = -math.inf
    wide.view(-1)[::53] = math.inf
    for dtype in (torch.bfloat16, torch.float16):
        slot, slot_lse = torch.full((B, Sq, H, D), math.nan, dtype=dtype, device="cuda"), torch.zeros(B, H, Sq, device="cuda")
        hip.cache_store(wide.cuda(), store(lse, bsh), slot, slot_lse)
        assert torch.equal(slot.cpu(), wide.to(dtype)) and torch.equal(slot_lse.cpu(), lse)
        back, back_lse = hip.cache_load(slot, slot_lse, torch.float32, dst_lse_bsh=bsh)
        assert torch.equal(back.cpu(), wide.to(dtype).float()) and torch.equal(back_lse.cpu(), store(lse, bsh).cpu())
