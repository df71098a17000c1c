"""Launches of few query rows: workgroups of 32 queries whose eight or four wavefronts take every eighth or fourth key tile each (``short_rows`` and
``attn_rows32`` in ditango_amd/csrc/attn_fwd.hip).  Without a GPU: which launches these are.  On it: every number of rows and keys at
which a slice, a tile or a wavefront's turn begins or ends, against fp64 on the CPU.

Tolerances: a result is one rounding to its type away from a sum of values below 4.5 (2^-9 of them, 9e-3; fp16 2^-12), whose
probabilities are rounded to the same type (2^-9 of a weighted mean of such values): 2e-2, as in the kernels' other tests.  The lse
is fp32: 1e-3."""
import json

import pytest
import torch

from ditango_amd import build
from oracle import attention_math as om
from tests.launch_log import record

OUT_TOL, LSE_TOL = 2e-2, 1e-3


def _listed(D, H, Sq, jobs, keys, B=1, **k):
    return dict(B=B, Sq=Sq, H=H, D=D, lens=[keys] * jobs, jobs=[[j] for j in range(jobs)], merged=0, **k)


RULE = [   # the launch, wavefronts of a workgroup of 32 rows (0: other workgroups)
    # slices of an XCD, 32 CUs: at D = 64 128 for up to 6 key tiles and 96 beyond, at D = 128 64; ragged slices count whole
    (_listed(64, 32, 1024, 1, 384), 4), (_listed(64, 33, 1024, 1, 384), 0), (_listed(64, 32, 1025, 1, 64), 0),
    (_listed(64, 24, 1024, 1, 385), 4), (_listed(64, 25, 1024, 1, 385), 0), (_listed(64, 2, 33, 1, 2048, B=192), 4), (_listed(64, 2, 33, 1, 2048, B=193), 0),
    (_listed(128, 16, 1024, 1, 64), 4), (_listed(128, 17, 1024, 1, 64), 0), (_listed(128, 4, 500, 8, 64), 4), (_listed(128, 4, 500, 9, 64), 0),
    # eight wavefronts: one workgroup a CU, more than 4 tiles
    (_listed(64, 8, 1024, 1, 256), 4), (_listed(64, 8, 1024, 1, 257), 8), (_listed(64, 8, 1025, 1, 257), 4),
    (_listed(128, 8, 1024, 1, 256), 4), (_listed(128, 8, 1024, 1, 257), 8), (_listed(128, 8, 1025, 1, 257), 4),
    # key tiles of the longest job: 32, and 8 at D = 128 with more workgroups than CUs
    (_listed(64, 4, 100, 2, 2048), 8), (_listed(64, 4, 100, 2, 2049), 0), (_listed(128, 4, 100, 2, 2048), 8),
    (_listed(128, 4, 100, 2, 2049), 0), (_listed(128, 8, 1025, 1, 512), 4), (_listed(128, 8, 1025, 1, 513), 0),
    (dict(B=1, Sq=40, H=3, D=64, lens=[1000, 1000, 48], jobs=[[0, 1, 2], [2]], merged=0), 0),
    (dict(B=1, Sq=40, H=3, D=64, lens=[1000, 1000, 0], jobs=[[0, 1, 2], [2]], merged=0), 8),
    (dict(B=1, Sq=300, H=3, D=64, lens=[300, 2049], jobs=None, max_jobs=1, merged=0), 0),
    (dict(B=1, Sq=300, H=3, D=64, lens=[300, 2048], jobs=None, max_jobs=2, merged=0), 8),
    # fp16; without a workspace items stay whole
    (_listed(128, 4, 100, 1, 7, fp16=True), 4), (_listed(128, 4, 100, 1, 7, workspace=False), 0),
]


def test_which_launches_take_32_rows_a_workgroup(tmp_path):
    for (call, waves), kernels in zip(RULE, record(tmp_path, [call for call, _ in RULE])):
        assert [w for w in (4, 8) if f"AttnRows{w}E" in kernels[0][1]] == [waves] * (waves > 0), call
        assert not waves or len(kernels) == 1, call


def _view(x, order):
    """x [B,S,H,D] on the GPU: contiguous, a slice of a fused buffer, or laid out [B,H,S,D]; NaN around it."""
    B, S, H, D = x.shape
    if order == "plain":
        return x.cuda()
    shape = (B, S + 2, 3, H, D + 8) if order == "fused" else (B, H + 1, S + 5, D)
    buf = torch.full(shape, float("nan"), dtype=x.dtype, device="cuda")
    view = buf[:, 1:1 + S, 1, :, :D] if order == "fused" else buf[:, 1:, 4:4 + S].permute(0, 2, 1, 3)
    view.copy_(x)
    return view


@pytest.mark.gpu
@pytest.mark.parametrize("order", ["plain", "fused", "heads"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
def test_edges_of_slices_and_tiles(hip, D, dtype, order):
    B = 2
    g = torch.Generator().manual_seed(D + (dtype == torch.float16))
    for rows, H in ((1, 2), (31, 2), (32, 2), (33, 2), (100, 2), (257, 2), (257, 16)):   # (the last: more workgroups than CUs)
        q = torch.randn(B, rows, H, D, generator=g).to(dtype)
        dq = _view(q, order)
        # one chunk; several with short and empty ones between, so that turns end inside and between chunks
        for lens in ((1,), (31,), (33,), (64,), (65,), (256,), (257,), (448,), (512,), (513,), (2048,), (0, 1, 0, 64, 63), (130, 0, 300, 5, 700)):
            print(f"case D={D} {dtype} {order} rows={rows} heads={H} keys={lens}", flush=True)
            ks, vs = ([torch.randn(B, n, H, D, generator=g).to(dtype) for n in lens] for _ in range(2))
            laid = "plain" if order == "heads" and len(lens) > 1 else order   # (the chunks of a table share their strides)
            table = hip.ChunkTable([_view(k, laid) for k in ks], [_view(v, laid) for v in vs])
            out = torch.full((B, rows, H, D), 7.0, dtype=dtype, device="cuda")
            lse = torch.full((B, H, rows), 7.0, device="cuda")
            hip.attn_jobs_fwd(dq, table, [list(range(len(lens)))], [out], [lse], workspace=hip.attn_workspace("cuda"))
            torch.cuda.synchronize()
            ref_out, ref_lse = om.chunk_attention(q, torch.cat(ks, 1), torch.cat(vs, 1))
            assert (out.float().cpu() - ref_out).abs().max().item() <= OUT_TOL, (rows, lens)
            assert (lse.cpu() - ref_lse).abs().max().item() <= LSE_TOL, (rows, lens)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
def test_jobs_of_a_segment_write_their_rows_only(hip, D):
    B, H, Sq = 1, 3, 200
    g = torch.Generator().manual_seed(D)
    q, k, v = (torch.randn(B, n, H, D, generator=g).bfloat16() for n in (Sq, 700, 700))
    table = hip.ChunkTable([k.cuda()], [v.cuda()])
    rows, keys = [(3, 33), (40, 1), (41, 64), (150, 0)], [(5, 64), (0, 700), (699, 1), (0, 700)]
    out, lse = torch.full((B, Sq, H, D), 7.0, dtype=torch.bfloat16, device="cuda"), torch.full((B, H, Sq), 7.0, device="cuda")
    hip.attn_jobs_fwd(q.cuda(), table, [[0]] * 4, [out] * 4, [lse] * 4, q_ranges=rows, kv_ranges=[[r] for r in keys],
                      workspace=hip.attn_workspace("cuda"))
    torch.cuda.synchronize()
    out, lse, rest = out.float().cpu(), lse.cpu(), torch.ones(Sq, dtype=torch.bool)
    for (q0, n), (k0, m) in zip(rows, keys):
        rest[q0:q0 + n] = False
        if n == 0:
            continue
        ref_out, ref_lse = om.chunk_attention(q[:, q0:q0 + n], k[:, k0:k0 + m], v[:, k0:k0 + m])
        assert (out[:, q0:q0 + n] - ref_out).abs().max().item() <= OUT_TOL
        assert (lse[:, :, q0:q0 + n] - ref_lse).abs().max().item() <= LSE_TOL
    assert (out[:, rest] == 7.0).all() and (lse[:, :, rest] == 7.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dst", [torch.float32, None])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("rows", [1, 33, 100])
def test_merging_launch_is_the_merge_of_its_states(hip, rows, D, dst):
    """States computed and merged in one launch, three times over the same counters, against the merge kernel on the same states: fp32
    sums of four terms, 2^-20 of the largest value, and one rounding where the result is 16 bits."""
    H = 3
    g = torch.Generator(device="cuda").manual_seed(rows + D)
    make = lambda n: torch.randn(1, n, H, D, generator=g, device="cuda").bfloat16()
    q, ks, vs = make(rows), [make(n) for n in (100, 3, 64)], [make(n) for n in (100, 3, 64)]
    cached, cached_lse = make(rows), torch.randn(1, H, rows, generator=g, device="cuda")
    for _ in range(3):
        states, out, lse = hip.attn_states_merge(q, ks, vs, [[0], [1], [2]], 32, [cached], [cached_lse], [0, 1, 2], dst or q.dtype,
                                                 hip.attn_workspace(q.device))
        torch.cuda.synchronize()
        want, want_lse = hip.merge_states([cached] + [s[0] for s in states], [cached_lse] + [s[1] for s in states])
        assert (out.float() - want.float()).abs().max().item() <= (2.0 ** -17 if dst else 2.0 ** -6)
        assert (lse.reshape(-1) - want_lse.permute(0, 2, 1).reshape(-1) if lse.shape != want_lse.shape else lse - want_lse).abs().max().item() <= 2.0 ** -17


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128])
def test_scores_of_minus_infinity_and_nan(hip, D):
    """Whole tiles of some wavefronts without a finite score, rows without any, and a NaN, which stays in its own row and head."""
    g = torch.Generator().manual_seed(5)
    q = torch.rand(1, 70, 2, D, generator=g).bfloat16() + 0.5
    k, v = (torch.randn(1, 900, 2, D, generator=g).bfloat16() for _ in range(2))
    k[:, 64:640, 0] = float("-inf")
    k[:, :, 1] = float("-inf")
    q[:, 40, 0, 3] = float("nan")
    out, lse = torch.empty(1, 70, 2, D, dtype=torch.bfloat16, device="cuda"), torch.empty(1, 2, 70, device="cuda")
    hip.attn_jobs_fwd(q.cuda(), hip.ChunkTable([k.cuda()], [v.cuda()]), [[0]], [out], [lse], workspace=hip.attn_workspace("cuda"))
    out, lse = out.float().cpu(), lse.cpu()
    keep = torch.cat([torch.arange(64), torch.arange(640, 900)])
    ref_out, ref_lse = om.chunk_attention(q[:, :, :1], k[:, keep, :1], v[:, keep, :1])
    fine = torch.arange(70) != 40
    assert (out[:, fine, :1] - ref_out[:, fine]).abs().max().item() <= OUT_TOL
    assert (lse[:, :1, fine] - ref_lse[:, :, fine]).abs().max().item() <= LSE_TOL
    assert out[:, 40, 0].isnan().all()
    assert (out[:, :, 1] == 0).all() and (lse[:, 1] == float("-inf")).all()


def test_no_form_is_built_that_no_launch_takes(tmp_path):
    """At D = 128 eight wavefronts take more than 4 key tiles and a merging launch up to 4: no call, whoever lists its jobs, takes both, and the
    kernel for it is not there.  Every other form is taken by some call."""
    calls = [dict(B=1, Sq=Sq, H=H, D=D, lens=[64 * tiles] * 4, jobs=listed, max_jobs=0 if listed else jobs, merged=merged, fp16=fp16)
             for D in (64, 128) for Sq, H in ((32, 1), (96, 24), (128, 16), (160, 20), (512, 4), (300, 16)) for tiles in (1, 2, 4, 5, 8)
             for jobs in (1, 2) for listed in (None, [[j] for j in range(jobs)]) for merged in (0, 2) for fp16 in (False, True)]
    taken = {k for kernels in record(tmp_path, calls) for _, k in kernels if "AttnRows" in k}
    built = {k for kernels in json.loads(build.RESOURCES_PATH.read_text()).values() for k in kernels if "AttnRows" in k}
    assert taken == built


# at D = 64 with more workgroups than CUs: key tiles by the slices of a head (one, two, two of heads side by side, more)
LONG_JOBS = [
    (_listed(64, 24, 32, 2, 2048, B=7), 4), (_listed(64, 24, 32, 1, 2048, B=11), 4), (_listed(64, 24, 32, 2, 2049, B=7), 0),
    (_listed(64, 24, 33, 1, 1024, B=8), 4), (_listed(64, 24, 33, 1, 1025, B=8), 0), (_listed(64, 24, 64, 1, 1025, B=8), 0),
    (_listed(64, 24, 64, 1, 640, B=16), 4), (_listed(64, 24, 64, 1, 641, B=16), 0),
    (_listed(64, 2, 64, 1, 2048, B=190), 4), (_listed(64, 3, 64, 1, 2048, B=127), 0), (_listed(64, 2, 65, 1, 641, B=120), 0),
    (_listed(64, 24, 65, 1, 2048, B=4), 4), (_listed(64, 16, 1024, 1, 2048), 4), (_listed(64, 16, 1025, 1, 640), 4), (_listed(64, 16, 1025, 1, 641), 0),
    (_listed(64, 48, 109, 1, 1830, B=4), 0), (_listed(64, 24, 969, 1, 1984), 0), (_listed(64, 8, 1024, 1, 2048), 8),
]


def test_long_jobs_of_more_workgroups_than_cus_keep_256_rows(tmp_path):
    for (call, waves), kernels in zip(LONG_JOBS, record(tmp_path, [call for call, _ in LONG_JOBS])):
        assert [w for w in (4, 8) if f"AttnRows{w}E" in kernels[0][1]] == [waves] * (waves > 0), call
