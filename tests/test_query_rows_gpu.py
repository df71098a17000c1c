"""The rows of q of a work item on their way into registers, and its rows of the result on their way out.

A wavefront brings its 32 rows of q through parts of the LDS that K/V tiles take later, so short key ranges matter (the tile that
takes a row's place is then the next one, or there is none), and so do rows that do not exist: they repeat the last one, and nothing
is written for them.  q is a view with strides of its own whose other rows and columns are NaN; destinations hold a value
that has to stay where a job has no rows.  Tolerances as in the kernels' other tests: one rounding to the element type of
values below 4 (2^-9 of them: 8e-3) beside probabilities rounded likewise."""
import pytest
import torch

from oracle import attention_math as om

pytestmark = pytest.mark.gpu
OUT_TOL, LSE_TOL = 2e-2, 1e-3


def _strided(x, order):
    """x [B,S,H,D] on the GPU as a view of a NaN-filled buffer: ``fused`` a slice of [B,S,3,H,D], ``heads`` laid out [B,H,S,D]."""
    B, S, H, D = x.shape
    if order == "fused":
        buf = torch.full((B, S + 3, 3, H, D + 8), float("nan"), dtype=x.dtype, device="cuda")
        view = buf[:, 2:2 + S, 1, :, :D]
    else:
        buf = torch.full((B, H + 1, S + 5, D), float("nan"), dtype=x.dtype, device="cuda")
        view = buf[:, 1:, 4:4 + S].permute(0, 2, 1, 3)
    view.copy_(x)
    return view


@pytest.mark.parametrize("order", ["fused", "heads"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
def test_every_number_of_rows_and_tiles(hip, D, dtype, order):
    """Jobs of 1 ... 257 query rows at odd places, against 1 ... 600 keys; with and without a workspace (items cut along the keys)."""
    B, H = 2, 3
    g = torch.Generator().manual_seed(D + (dtype == torch.float16))
    rows = [1, 8, 9, 23, 24, 31, 32, 33, 127, 128, 129, 255, 256, 257]
    begins = [sum(rows[:i]) + 3 * i + 1 for i in range(len(rows))]
    Sq = begins[-1] + rows[-1] + 2
    q = torch.randn(B, Sq, H, D, generator=g).to(dtype)
    dq = _strided(q, order)
    for keys in (1, 64, 65, 130, 200, 600):
        print(f"case D={D} {dtype} {order} keys={keys}", flush=True)
        k, v = (torch.randn(B, keys, H, D, generator=g).to(dtype) for _ in range(2))
        table = hip.ChunkTable([k.cuda()], [v.cuda()])
        ref_out, ref_lse = om.chunk_attention(q, k, v)
        live = torch.zeros(Sq, dtype=torch.bool)
        for begin, n in zip(begins, rows):
            live[begin:begin + n] = True
        for workspace in (None, hip.attn_workspace(dq.device)):
            out = torch.full((B, Sq, H, D), 7.0, dtype=dtype, device="cuda")
            lse = torch.full((B, H, Sq), 7.0, dtype=torch.float32, device="cuda")
            hip.attn_jobs_fwd(dq, table, [[0]] * len(rows), [out] * len(rows), [lse] * len(rows), q_ranges=list(zip(begins, rows)),
                              workspace=workspace)
            torch.cuda.synchronize()
            out, lse = out.float().cpu(), lse.cpu()
            assert (out[:, ~live] == 7.0).all() and (lse[:, :, ~live] == 7.0).all(), keys
            assert (out[:, live] - ref_out[:, live]).abs().max().item() <= OUT_TOL, keys
            assert (lse[:, :, live] - ref_lse[:, :, live]).abs().max().item() <= LSE_TOL, keys


@pytest.mark.parametrize("D", [64, 128])
def test_launches_that_merge_read_strided_rows(hip, D):
    """The same through a launch that merges its states (short, few states), bit for bit with contiguous q."""
    B, H, Sq = 1, 4, 100
    g = torch.Generator().manual_seed(9 + D)
    q = torch.randn(B, Sq, H, D, generator=g).bfloat16()
    ks, vs = ([torch.randn(B, n, H, D, generator=g).bfloat16().cuda() for n in (100, 97)] for _ in range(2))
    results = []
    for dq in (q.cuda(), _strided(q, "fused"), _strided(q, "heads")):
        states, out, lse = hip.attn_states_merge(dq, ks, vs, [[0], [1]], 32, [], [], [0, 1], torch.float32, hip.attn_workspace(dq.device))
        results.append([out, lse] + [t for state in states for t in state])
    for other in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(results[0], other))
