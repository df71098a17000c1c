"""What the attention kernel takes off its scores: the reference maximum that the accumulators are scaled to, which at D = 128 the MFMAs
start from.  First tiles without a key for some wavefront, references far below and above what follows, references beyond the size
that the MFMAs take (64 in log2 units, 44 in natural ones), and rows of one wavefront on either side of it.
Tolerances: one rounding to the element type of the result and of the probabilities, as in the kernels' other tests; the lse of scores of
size s is an fp32 sum of products of that size, 128 * 2^-24 * s with room to spare below 1e-3 up to s = 100."""
import pytest
import torch

from oracle import attention_math as om

pytestmark = pytest.mark.gpu
OUT_TOL, LSE_TOL = 2e-2, 1e-3


def _case(hip, D, dtype, rows, chunks, scales, seed):
    """One job over chunks of ``chunks`` keys; the keys of chunk i lie along the queries' common direction, so that all of its scores are
    about ``scales[i]`` for the even rows and minus that for the odd ones."""
    B, H = 1, 2
    g = torch.Generator().manual_seed(seed)
    base = torch.randn(B, 1, H, D, generator=g)
    base /= base.norm(dim=-1, keepdim=True)
    q = torch.randn(B, rows, H, D, generator=g) * 0.3 + 6 * base
    q[:, 1::2] -= 12 * base
    ks = [torch.randn(B, n, H, D, generator=g) * 0.5 + base * (s * D ** 0.5 / 6) for n, s in zip(chunks, scales)]
    vs = [torch.randn(B, n, H, D, generator=g) for n in chunks]
    q, ks, vs = q.to(dtype), [k.to(dtype) for k in ks], [v.to(dtype) for v in vs]
    ref_out, ref_lse = om.chunk_attention(q, torch.cat(ks, 1), torch.cat(vs, 1))
    table = hip.ChunkTable([k.cuda() for k in ks], [v.cuda() for v in vs])
    for workspace in (None, hip.attn_workspace("cuda")):
        out = torch.empty(B, rows, H, D, dtype=dtype, device="cuda")
        lse = torch.empty(B, H, rows, device="cuda")
        hip.attn_jobs_fwd(q.cuda(), table, [list(range(len(chunks)))], [out], [lse], workspace=workspace)
        torch.cuda.synchronize()
        assert torch.isfinite(out.float()).all()
        assert (out.float().cpu() - ref_out).abs().max().item() <= OUT_TOL
        assert (lse.cpu() - ref_lse).abs().max().item() <= LSE_TOL


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("scales", [(0, 0, 0), (-30, 0, 20), (-60, 0, 3), (-100, 5, 0), (60, 0, 80), (100, 0, -100), (0, 50, 90)])
def test_reference_moves(hip, D, dtype, scales):
    for rows in (40, 100, 300):              # shared keys (up to 128 rows), and not
        for first in (1, 20, 33, 64, 200):   # keys of the first chunk: none for the wavefronts of the second half of a tile below 33
            print(f"case D={D} {dtype} {scales} rows={rows} first={first}", flush=True)
            _case(hip, D, dtype, rows, (first, 70, 500), scales, seed=rows + first)


@pytest.mark.parametrize("D", [64, 128])
def test_rows_whose_first_tiles_hold_no_finite_score(hip, D):
    """Keys at -inf scores for every row, then ordinary ones: the result is the ordinary keys' alone."""
    B, H, rows = 1, 1, 70
    g = torch.Generator().manual_seed(3)
    q = torch.rand(B, rows, H, D, generator=g).bfloat16() + 0.5
    dead = torch.full((B, 130, H, D), float("-inf")).bfloat16()
    k, v = (torch.randn(B, 300, H, D, generator=g).bfloat16() for _ in range(2))
    table = hip.ChunkTable([dead.cuda(), k.cuda()], [torch.zeros_like(dead).cuda(), v.cuda()])
    out = torch.empty(B, rows, H, D, dtype=torch.bfloat16, device="cuda")
    lse = torch.empty(B, H, rows, device="cuda")
    hip.attn_jobs_fwd(q.cuda(), table, [[0, 1]], [out], [lse])
    ref_out, ref_lse = om.chunk_attention(q, k, v)
    torch.cuda.synchronize()
    assert (out.float().cpu() - ref_out).abs().max().item() <= OUT_TOL
    assert (lse.cpu() - ref_lse).abs().max().item() <= LSE_TOL


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
def test_scores_behind_a_reference_far_below_keep_their_bits(hip, D, dtype):
    """A first tile of scores about -``below`` for every row, then keys of ordinary ones: the lse is that of the ordinary keys alone, and its
    error that of their own sums, however far below the first reference lies.  Tolerance: |q| |k| / sqrt(D) is below 5, so 128 roundings of
    2^-24 of it are below 4e-5; a reference that the MFMAs take (up to 64 log2 units, 44 natural ones) adds D / 16 roundings of 2^-18 log2
    units, 2.2e-5 in all."""
    H = 2
    for below in (38.0, 60.0, 1e3, 3e4) + ((1e5, 1e7) if dtype == torch.bfloat16 else ()):
        for rows in (40, 100, 300):
            for keys in (1, 3, 150):
                print(f"case D={D} {dtype} below={below} rows={rows} keys={keys}", flush=True)
                g = torch.Generator().manual_seed(rows + keys)
                base = torch.randn(1, 1, H, D, generator=g)
                base /= base.norm(dim=-1, keepdim=True)
                q = (torch.randn(1, rows, H, D, generator=g) * 0.3 + 6 * base).to(dtype)
                first = (-base * (below * D ** 0.5 / 6)).expand(1, 64, H, D).to(dtype)
                k = (torch.randn(1, keys, H, D, generator=g) * 0.4).to(dtype)
                v = [torch.randn(1, n, H, D, generator=g).to(dtype) for n in (64, keys)]
                assert (q.float().norm(dim=-1).max() * k.float().norm(dim=-1).max() / D ** 0.5).item() < 5
                ref_out, ref_lse = om.chunk_attention(q, torch.cat([first, k], 1), torch.cat(v, 1), compute_dtype=torch.float64)
                table = hip.ChunkTable([first.cuda(), k.cuda()], [x.cuda() for x in v])
                for workspace in (None, hip.attn_workspace("cuda")):
                    out = torch.empty(1, rows, H, D, dtype=dtype, device="cuda")
                    lse = torch.empty(1, H, rows, device="cuda")
                    hip.attn_jobs_fwd(q.cuda(), table, [[0, 1]], [out], [lse], workspace=workspace)
                    torch.cuda.synchronize()
                    assert (out.double().cpu() - ref_out).abs().max().item() <= OUT_TOL
                    assert (lse.double().cpu() - ref_lse).abs().max().item() <= (6.2e-5 if below < 44 else 4e-5)
