"""Cache stores of fp32 states and loads into fp32 (``state_convert_kernel``): every element is one rounding or its exact widening, so
results equal torch's conversion bit for bit.  Sizes on either side of what a launch is cut into: 2048 elements a workgroup, lse
tiles of 16 ... 256 query positions x up to 256 heads, 2^18 rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (2, 15, 1), (1, 257, 1), (3, 16, 3), (1, 33, 7), (2, 65, 12), (1, 17, 48), (1, 70, 129), (1, 16, 256), (2, 19, 257), (1, 5, 600),
         (1, 2731, 96), (2, 1366, 100), (1, 1040, 260), (1, 5500, 48)]


def _lse(B, S, H, bsh, g):
    x = 3 * torch.randn(B, H, S, generator=g, device="cuda")
    x[..., ::7] = float("-inf")
    return x, (x.transpose(1, 2).unsqueeze(-1).contiguous() if bsh else x.contiguous())


@pytest.mark.parametrize("bsh", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
def test_store_and_load_are_one_rounding_and_its_widening(hip, D, dtype, bsh):
    for B, S, H in SIZES:
        print(f"case {D} {dtype} bsh={bsh} {B} x {S} x {H}", flush=True)
        g = torch.Generator(device="cuda").manual_seed(S * H)
        out = torch.randn(B, S, H, D, generator=g, device="cuda") * torch.exp2(torch.randint(-12, 13, (B, S, H, 1), generator=g, device="cuda").float())
        out.view(-1)[::1013] = float("inf")
        lse, given = _lse(B, S, H, bsh, g)
        slot_out = torch.full((B, S, H, D), 7.0, dtype=dtype, device="cuda")
        slot_lse = torch.full((B, H, S), 7.0, device="cuda")
        hip.cache_store(out, given, slot_out, slot_lse)
        assert torch.equal(slot_out, out.to(dtype)) and torch.equal(slot_lse, lse)
        back_out, back_lse = hip.cache_load(slot_out, slot_lse, torch.float32, bsh)
        assert torch.equal(back_out, slot_out.float())
        assert torch.equal(back_lse.reshape(given.shape), given)


# 2^14 rows: below, a lane moves one value of the lse, from there on it goes in tiles
DIRECT_EDGE = [(1, 16383, 1), (1, 16384, 1), (2, 8192, 1), (1, 2340, 7), (1, 2341, 7), (3, 1820, 3), (3, 1821, 3), (3, 455, 12), (1, 63, 257), (1, 64, 257),
               (2, 13, 600), (2, 14, 600), (1, 40000, 1)]


@pytest.mark.parametrize("src_bsh", [False, True])
@pytest.mark.parametrize("dst_bsh", [False, True])
def test_few_rows_and_tiles_move_every_value_of_the_lse(hip, src_bsh, dst_bsh):
    for B, S, H in DIRECT_EDGE:
        print(f"case {src_bsh} -> {dst_bsh} {B} x {S} x {H}", flush=True)
        g = torch.Generator(device="cuda").manual_seed(S * H)
        out = torch.randn(B, S, H, 64, generator=g, device="cuda")
        lse, given = _lse(B, S, H, src_bsh, g)
        slot_out = torch.full((B, S, H, 64), 7.0, dtype=torch.bfloat16, device="cuda")
        slot_lse = torch.full((B, H, S), 7.0, device="cuda")
        hip.cache_store(out, given, slot_out, slot_lse)
        assert torch.equal(slot_out, out.bfloat16()) and torch.equal(slot_lse, lse)
        back_out, back_lse = hip.cache_load(slot_out, slot_lse, torch.float32, dst_bsh)
        assert torch.equal(back_out, slot_out.float())
        want = lse.transpose(1, 2).unsqueeze(-1) if dst_bsh else lse
        assert torch.equal(back_lse.reshape(want.shape), want)
