"""q, k and v in one launch (``dt_qkv_project``) against the projections, the norm and the rotation in fp64, and the calls that go to
the modules instead."""
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu


def _layer(H, K, dtype, bias=True, affine=True, seed=0):
    torch.manual_seed(seed)
    attn = SimpleNamespace(heads=H, is_cross_attention=False)
    for name in ("to_q", "to_k", "to_v"):
        setattr(attn, name, torch.nn.Linear(K, H * 64, bias=bias, device="cuda", dtype=dtype))
    for name in ("norm_q", "norm_k"):
        m = torch.nn.LayerNorm(64, eps=1e-6, elementwise_affine=affine, device="cuda", dtype=dtype)
        if affine:
            with torch.no_grad():
                m.weight.copy_(1 + 0.1 * torch.randn(64))
                m.bias.copy_(0.1 * torch.randn(64))
        setattr(attn, name, m)
    return attn


def _tokens(B, T, V, K, dtype, seed=1, strided=False):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def make(n):
        if strided:   # every other row of a longer tensor
            return torch.randn(B, 2 * n, K, generator=g, device="cuda").to(dtype)[:, ::2]
        return torch.randn(B, n, K, generator=g, device="cuda").to(dtype)

    angle = (6.28 * torch.rand(V, 32, generator=g, device="cuda")).repeat_interleave(2, -1)
    return make(T), make(V), (angle.cos().contiguous(), angle.sin().contiguous())


def _exact(attn, text, video, rope, norms=True):
    x = torch.cat([text, video], 1).double()
    out = []
    for name, norm in (("to_q", "norm_q"), ("to_k", "norm_k"), ("to_v", None)):
        m = getattr(attn, name)
        y = x @ m.weight.double().t() + (m.bias.double() if m.bias is not None else 0)
        y = y.view(*y.shape[:2], attn.heads, 64)
        if norm and norms:
            n = getattr(attn, norm)
            y = torch.nn.functional.layer_norm(y, (64,), n.weight.double() if n.weight is not None else None,
                                               n.bias.double() if n.bias is not None else None, n.eps)
        if norm and rope is not None:
            cos, sin = (t.double()[None, :, None] for t in rope)
            z = y[:, text.shape[1]:]
            turned = torch.stack([-z[..., 1::2], z[..., ::2]], -1).flatten(-2)
            y = torch.cat([y[:, :text.shape[1]], z * cos + turned * sin], 1)
        out.append(y)
    return out


def _check(got, want, dtype):
    """Three roundings to 16 bits on the way (projection, norm, rotation), each half a unit at most: of a value, or of the row's largest
    where a mean was subtracted; the 2-norm of three independent ones is below one unit's half."""
    unit = 2.0 ** -8 if dtype is torch.bfloat16 else 2.0 ** -11
    for a, b in zip(got, want):
        assert torch.isfinite(a).all()
        assert (a.double() - b).norm() <= unit * b.norm()
        assert (a.double() - b).abs().max() <= 4 * unit * b.abs().max()


@pytest.mark.parametrize("B,T,V,H,K,dtype", [
    (1, 1, 1, 1, 64, torch.bfloat16),          # fewer steps than buffers
    (2, 26, 170, 3, 128, torch.float16),       # a sample's rows end inside a tile; columns end inside one
    (1, 28, 37, 8, 192, torch.bfloat16),       # one row more than a tile of 64
    (3, 5, 300, 5, 320, torch.bfloat16),       # rows of three samples in one tile
    (1, 113, 2500, 24, 1536, torch.bfloat16),  # 192 x 256
    (1, 28, 2212, 48, 3072, torch.float16),    # 320 x 256, 7 full tiles of rows
    (1, 28, 1893, 48, 3072, torch.bfloat16),   # ... one row more than 6
    (1, 28, 3301, 48, 3072, torch.bfloat16),   # 256 x 256, one row more than 13 tiles
    # columns of 22.5 tiles of 256, in each of the large tiles; rows of two samples in one tile
    (1, 30, 1970, 30, 1920, torch.bfloat16),
    (1, 30, 2970, 30, 1920, torch.float16),
    (1, 30, 4970, 30, 1920, torch.bfloat16),
    (2, 30, 1470, 30, 1920, torch.bfloat16),
    (2, 30, 1970, 30, 1920, torch.float16),
    (2, 30, 3970, 30, 1920, torch.bfloat16),
])
@pytest.mark.parametrize("bias,rotated", [(True, True), (False, False)])
def test_projections_match_fp64(hip, B, T, V, H, K, dtype, bias, rotated):
    from ditango_amd.executor.cogvideox.projection import project_qkv
    attn = _layer(H, K, dtype, bias, affine=bias)
    text, video, rope = _tokens(B, T, V, K, dtype, strided=not bias)
    rope = rope if rotated else None
    with torch.no_grad():
        got = project_qkv(attn, text, video, rope)
        assert got is not None
        _check(got, _exact(attn, text, video, rope), dtype)


@pytest.mark.parametrize("B,T,V,H,K", [
    (2, 26, 170, 3, 128),
    (2, 30, 1500, 30, 1920),     # columns of 22.5 tiles of 256; rows of two samples in one tile
    (1, 113, 2500, 24, 1536),
    (1, 28, 2194, 48, 3072),
    (1, 28, 3301, 48, 3072),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_norm_and_rotation_are_the_producers_bit_for_bit(hip, B, T, V, H, K, dtype):
    """The projections alone, then ``prepare_qk`` as the adapter calls it, against all of it in one launch; and the modules' products,
    which the library adds up in one chain at these sizes."""
    from ditango_amd.executor.cogvideox.projection import project_qkv
    from ditango_amd.producer import prepare_qk
    attn = _layer(H, K, dtype)
    text, video, rope = _tokens(B, T, V, K, dtype)
    bare = SimpleNamespace(**{**vars(attn), "norm_q": None, "norm_k": None})
    x = torch.cat([text, video], 1)
    with torch.no_grad():
        got = project_qkv(attn, text, video, rope)
        plain = project_qkv(bare, text, video, None)
        for m, y in zip((attn.to_q, attn.to_k, attn.to_v), plain):
            assert torch.equal(m(x).view_as(y), y)
        for y, n, z in zip(plain, (attn.norm_q, attn.norm_k), got):
            want = prepare_qk(y, norm="layer_norm", weight=n.weight, bias=n.bias, eps=n.eps, match_eager_rounding=True, rope="interleaved",
                              freqs_cis=rope, rope_begin=T)
            assert torch.equal(want, z)
        for y, n, z in zip(plain, (attn.norm_q, attn.norm_k), project_qkv(attn, text, video, None)):
            assert torch.equal(prepare_qk(y, norm="layer_norm", weight=n.weight, bias=n.bias, eps=n.eps, match_eager_rounding=True), z)
        for y, z in zip(plain[:2], project_qkv(bare, text, video, rope)):
            assert torch.equal(prepare_qk(y, rope="interleaved", freqs_cis=rope, rope_begin=T, match_eager_rounding=True), z)
        assert torch.equal(plain[2], got[2])


@pytest.mark.parametrize("T,V,H,K", [
    (5, 100, 3, 64),           # one projection's columns end inside a tile
    (113, 2500, 24, 1536),
    (28, 2194, 48, 3072),
    (28, 3301, 48, 3072),
])
@pytest.mark.parametrize("which", range(3))
def test_rotation_of_one_projection_alone(hip, T, V, H, K, which):
    """Every tile form, and each of the three places: bit for bit the producer's rotation of the bare product, the others untouched."""
    from ditango_amd.producer import prepare_qk
    attn = _layer(H, K, torch.bfloat16)
    text, video, rope = _tokens(1, T, V, K, torch.bfloat16)
    with torch.no_grad():
        table = lambda turned: [(m.weight, m.bias, hip.DT_NORM_NONE, None, None, 0.0, i in turned)
                                for i, m in enumerate((attn.to_q, attn.to_k, attn.to_v))]
        plain = hip.qkv_project(text, video, H, table(()))
        got = hip.qkv_project(text, video, H, table((which,)), *rope)
        for i, (a, b) in enumerate(zip(plain, got)):
            want = prepare_qk(a, rope="interleaved", freqs_cis=rope, rope_begin=T) if i == which else a
            assert torch.equal(want, b), i


@pytest.mark.parametrize("H,K,V", [(2, 128, 150), (24, 1536, 2500), (48, 3072, 2194), (48, 3072, 3272)])
def test_a_row_depends_on_its_own_tokens_only(hip, H, K, V):
    """Every tile form: rows one by one, in another tile and beside other rows, come out bit for bit the same (one order of the sums)."""
    from ditango_amd.executor.cogvideox.projection import project_qkv
    attn = _layer(H, K, torch.bfloat16)
    text, video, rope = _tokens(1, 28, V, K, torch.bfloat16)
    with torch.no_grad():
        whole = project_qkv(attn, text, video, rope)
        part = project_qkv(attn, text[:, :3], video[:, 40:75], tuple(t[40:75].contiguous() for t in rope))
    for a, b in zip(whole, part):
        assert torch.equal(a[:, :3], b[:, :3]) and torch.equal(a[:, 68:103], b[:, 3:])


def test_modules_that_are_more_than_their_arithmetic_are_called(hip):
    from ditango_amd.executor.cogvideox.projection import project_qkv

    class Adapted(torch.nn.Linear):
        pass

    text, video, rope = _tokens(1, 4, 60, 128, torch.bfloat16)
    attn = _layer(2, 128, torch.bfloat16)
    take = lambda a=attn, t=text, v=video, r=rope: project_qkv(a, t, v, r)
    assert take() is None   # gradients are asked for
    with torch.no_grad():
        assert take() is not None
        handle = attn.to_v.register_forward_hook(lambda m, i, o: o + 1)
        assert take() is None
        handle.remove()
        handle = attn.norm_k.register_forward_pre_hook(lambda m, i: None)
        assert take() is None
        handle.remove()
        with torch.autocast("cuda", torch.float16):
            assert take() is None
        odd = _layer(2, 128, torch.bfloat16)
        odd.to_k = Adapted(128, 128, device="cuda", dtype=torch.bfloat16)
        assert take(odd) is None
        odd = _layer(2, 128, torch.bfloat16)
        odd.norm_q = odd.norm_q.float()
        assert take(odd) is None
        assert take(t=text.half()) is None and take(t=text.float(), v=video.float()) is None
        assert take(r=(rope[0][:, :32], rope[1][:, :32])) is None
        assert take(v=video[:, :, 4:]) is None
        assert take() is not None


def test_captured_projections_replay(hip):
    from ditango_amd.executor.cogvideox.projection import project_qkv
    attn = _layer(6, 384, torch.bfloat16)
    text, video, rope = _tokens(1, 17, 400, 384, torch.bfloat16)
    with torch.no_grad():
        project_qkv(attn, text, video, rope)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got = project_qkv(attn, text, video, rope)
        for i in range(3):
            video.copy_(torch.randn_like(video))
            graph.replay()
            want = project_qkv(attn, text, video, rope)
            torch.cuda.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(got, want)), i
