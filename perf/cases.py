"""The work that users of this package have it do, as cases that can be timed.

A sampler calls the cached block attention once per layer and denoising step, through one of four entries:
``proAttention.attn`` (directly, under a reuse mask or under the stride schedule) or one of the three model adapters.
Around it run the QK-norm / RoPE producer, the running-state merge and the state cache.  ``listed`` holds one case
for each, from a toy problem to a sequence of 119 056 tokens on one GPU; ``draw`` gives more of the same ranges.

Kinds:

* ``mask``      one layer call under a per-chunk reuse mask: ``computed`` of ``N`` KV chunks are recomputed, the cached
                states of the others (made by the cold first step, which is preparation) are merged
* ``block``     the same call through the CogVideoX attention processor: projections, LayerNorm + RoPE, attention,
                output projection
* ``stride``    a short generation of one layer under the stride schedule, from a cold full-stride step to the last one
                (``strides``: chunks recomputed at each step), through ``proAttention.attn``, the Step-Video adapter
                (``entry`` = ``step``) or the HunyuanVideo one (``varlen``: packed tokens, boundaries on the GPU, the
                last ``pad`` rows padding in a segment of their own)
* ``exact``     fp32 tensors computed in fp32: one full-stride call
* ``update``    the running (out, lse) of a ring loop over ``N`` block states, as ``update_out_and_lse`` folds them
* ``cache``     fp32 states stored in the cache and loaded back
* ``producer``  QK norm + RoPE of the q and k slices of a fused projection
"""
import math
from types import SimpleNamespace

import torch

from ditango_amd import utils
from ditango_amd.core import config, parallel_state, redundancy_map
from ditango_amd.core.attention import proAttention
from ditango_amd.core.cache import proCache
from ditango_amd.executor.cogvideox.attention_processor import CVX_oCacheAttnProcessor
from ditango_amd.executor.hunyuanvideo.attention_hunyuan import Hunyuan_DiTangoProcessor
from ditango_amd.executor.step.attentions import Attention as StepAttention
from ditango_amd.producer import prepare_qk

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "f32": torch.float32}


def listed():
    return [
        # a user's first run and the unit tests' size: the reference's CPU-runnable configuration (4 heads of 64, 512
        # queries, 4 chunks of 512), where a call is latency and launches
        dict(name="toy_mask", kind="mask", B=1, H=4, D=64, Sq=512, N=4, ragged=False, computed=2, dtype="bf16", out="f32"),
        # the same configuration in the precision it is stated in
        dict(name="toy_exact", kind="exact", B=1, H=4, D=64, Sq=512, N=4, dtype="f32"),
        # a preview: a short, low-resolution clip (an eighth of the HunyuanVideo share's tokens), two samples of a guided
        # batch, chunks of unequal length
        dict(name="preview_mask", kind="mask", B=2, H=24, D=128, Sq=1861, N=8, ragged=True, computed=3, dtype="bf16",
             out="act"),
        # the CogVideoX-5B share of one of 8 ranks, half of the chunks recomputed
        dict(name="cogvideox_mask", kind="mask", B=1, H=48, D=64, Sq=2222, N=8, ragged=False, computed=5, dtype="bf16",
             out="f32"),
        # the same share through the model's attention processor (226 text tokens split over 8 ranks)
        dict(name="cogvideox_block", kind="block", B=1, H=48, D=64, Sq=2222, N=8, ragged=False, computed=4, text=28,
             dtype="bf16"),
        # the Step-Video-T2V share in fp16 over a short generation
        dict(name="stepvideo_stride", kind="stride", entry="step", B=1, H=48, D=128, Sq=6851, N=8, strides="8,2,2,4,8",
             rank=3, dtype="fp16", out="act"),
        # HunyuanVideo as the model calls it: packed, 64 padding rows, boundaries on the GPU
        dict(name="hunyuan_varlen", kind="stride", entry="varlen", B=1, H=24, D=128, Sq=14882, N=8, strides="8,2,2,2,4,8",
             rank=0, pad=64, dtype="bf16", out="f32"),
        # the benchmark's layer call
        dict(name="hunyuan_mask", kind="mask", B=1, H=24, D=128, Sq=14882, N=8, ragged=False, computed=4, dtype="bf16",
             out="f32"),
        # a whole sequence on one GPU at high reuse: 3 of 32 chunks recomputed, 29 cached states of 743 MB merged
        dict(name="sweep_reuse", kind="mask", B=1, H=24, D=128, Sq=119056, Sk=3721, N=32, ragged=True, computed=3,
             dtype="bf16", out="f32"),
        # a caller's own ring loop at the Step-Video share
        dict(name="running_update", kind="update", B=1, H=48, D=128, Sq=6851, N=3, dtype="bf16"),
        # one fp32 state into the cache and back at the CogVideoX share
        dict(name="cache_roundtrip", kind="cache", B=1, H=48, D=64, Sq=2222, dtype="bf16"),
        # RMSNorm + interleaved RoPE of the HunyuanVideo share's q and k
        dict(name="producer_qk", kind="producer", B=1, H=24, D=128, Sq=14882, norm="rms", rope="interleaved", begin=0,
             dtype="bf16"),
    ]


# of a drawn case: below the largest listed ones (fp32 on the vector ALU is the slowest path by far)
_MOST_FLOPS, _MOST_FLOPS_F32, _MOST_BYTES = 4.0e13, 4.0e10, 6.0e9


def draw(rng):
    """One more case: tokens over their logarithm from one query tile to the largest share, any head count."""
    while True:
        kind = rng.choice(["mask", "mask", "mask", "stride", "stride", "varlen", "block", "exact", "update", "cache", "producer"])
        D = rng.choice([64, 128])
        H = rng.choice([1, 2, 3, 4, 6, 8, 10, 12, 16, 20, 24, 30, 32, 40, 48])
        B = rng.choice([1, 1, 1, 2])
        Sq = int(math.exp(rng.uniform(math.log(96), math.log(15000))))
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
        N = rng.choice([2, 4, 8])
        case = dict(kind=kind, B=B, H=H, D=D, Sq=Sq, N=N, dtype=dtype)
        if kind == "mask":
            case.update(N=rng.choice([2, 3, 4, 6, 8, 16]), ragged=rng.random() < 0.5, out=rng.choice(["act", "f32"]))
            case["computed"] = rng.randint(1, case["N"])
            if rng.random() < 0.25:
                case["Sk"] = -(-Sq // case["N"])
        elif kind == "stride":
            case.update(entry=rng.choice(["attn", "step"]), strides=_draw_strides(rng, N), rank=rng.randrange(N),
                        out=rng.choice(["act", "f32"]))
            if case["entry"] == "step":
                case["out"] = "act"
        elif kind == "varlen":
            case.update(kind="stride", entry="varlen", B=1, strides=_draw_strides(rng, N), rank=rng.randrange(N),
                        pad=rng.choice([0, 17, 64, 200]), out=rng.choice(["act", "f32"]))
            if case["pad"] >= Sq // 2:
                case["pad"] = 16
        elif kind == "block":
            case.update(H=rng.choice([8, 16, 24, 30, 48]), D=64, ragged=False, text=rng.choice([16, 28, 113]), N=rng.choice([4, 8]))
            case["Sq"] = int(math.exp(rng.uniform(math.log(300), math.log(6000))))
            case["computed"] = rng.randint(1, case["N"])
        elif kind == "exact":
            case.update(dtype="f32", B=1, H=min(H, 12), Sq=int(math.exp(rng.uniform(math.log(96), math.log(2048)))))
        elif kind == "update":
            case.update(N=rng.randint(2, 4))
        elif kind == "cache":
            del case["N"]
            case["dtype"] = "bf16"
        else:
            del case["N"]
            case.update(norm=rng.choice(["rms", "layer_norm"]), rope=rng.choice(["interleaved", "rotate_half"]),
                        begin=rng.choice([0, 0, 16]))
        w = work(case)
        if w["flops"] <= (_MOST_FLOPS_F32 if kind == "exact" else _MOST_FLOPS) and w["bytes"] <= _MOST_BYTES:
            return case


def _draw_strides(rng, N):
    """Strides of a short generation that a refined divider map can hold: full first and last, never finer again in between."""
    middle = sorted(rng.choice([s for s in (1, 2, 4, 8) if s <= N // 2]) for _ in range(rng.randint(1, 4)))
    return ",".join(str(s) for s in [N] + middle + [N])


# ---- the process-wide schedule and step counter that a sampler keeps -------------------------------------------------------

_installed = None


def _schedule(case):
    """The redundancy map of the case, installed once as a sampler does before its first step."""
    global _installed
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if _installed is not None and _installed[0] == key and redundancy_map.get_redundancy_map() is _installed[1]:
        return
    redundancy_map.destroy_redundancy_map()
    strides = [int(s) for s in case["strides"].split(",")] if "strides" in case else [case["N"]] * 2
    parallel_state.init_local_groups(case["N"], case.get("rank", 0))
    cfg = config.init_config(None, num_inference_steps=len(strides), num_layers=2, ditango_base="-")
    rm = redundancy_map.init_redundancy_map(cfg, quiet=True)
    if "computed" in case:
        # step 0 is cold; step 1 recomputes the local chunk and computed - 1 others, spread over the ring
        N, n = case["N"], case["computed"] - 1
        fresh = {1 + (i * (N - 1)) // n for i in range(n)} if n else set()
        mask = torch.zeros(2, 2, N, dtype=torch.uint8)
        for c in range(1, N):
            mask[1, :, c] = 0 if c in fresh else 1
        rm.set_chunk_mask(mask.numpy(), diag=0)
    else:
        for t, s in enumerate(strides):
            rm.set_pattern_for_row(t, [], [case["N"] // s])
    _installed = (key, rm)


def _lengths(case):
    """Tokens of every KV chunk: equal shards, or the second half of them one token shorter where the sequence does not divide."""
    N = case["N"]
    n = case.get("Sk", case["Sq"])            # (Sk: all queries on one GPU, the chunks split the same sequence)
    return [n - (1 if case.get("ragged") and i >= N // 2 else 0) for i in range(N)]


def _normed(shape, g, dtype):
    """Queries and keys as the models hand them over: normalised over the head dimension."""
    x = torch.randn(shape, generator=g, device="cuda")
    x *= torch.rsqrt(x.pow(2).mean(-1, keepdim=True))
    return x.to(dtype)


def _plain(shape, g, dtype):
    return torch.randn(shape, generator=g, device="cuda").to(dtype)


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    kind, B, H, D, Sq = case["kind"], case["B"], case["H"], case["D"], case["Sq"]
    dtype = _DTYPES[case["dtype"]]
    st = SimpleNamespace(case=case, kind=kind)
    if kind == "update":
        st.blocks = [(_plain((B, Sq, H, D), g, dtype), 2.0 + torch.randn(B, H, Sq, generator=g, device="cuda"))
                     for _ in range(case["N"])]
        return st
    if kind == "cache":
        st.out = torch.randn(B, Sq, H, D, generator=g, device="cuda")
        st.lse = 2.0 + torch.randn(B, Sq, H, 1, generator=g, device="cuda")
        st.cache = proCache(isp_size=8, layer_id=1)
        return st
    if kind == "producer":
        qkv = _plain((B, Sq, 3, H, D), g, dtype)
        st.q, st.k = qkv[:, :, 0], qkv[:, :, 1]
        st.norm = dict(norm=case["norm"], weight=1.0 + 0.1 * torch.randn(D, generator=g, device="cuda"))
        if case["norm"] == "layer_norm":
            st.norm["bias"] = 0.1 * torch.randn(D, generator=g, device="cuda")
        rows = Sq - case["begin"]
        angle = torch.rand(rows, D // 2, generator=g, device="cuda") * 6.28
        wide = angle.repeat_interleave(2, -1) if case["rope"] == "interleaved" else torch.cat([angle, angle], -1)
        st.rope = dict(rope=case["rope"], freqs_cis=(wide.cos().contiguous(), wide.sin().contiguous()), rope_begin=case["begin"])
        return st

    _schedule(case)
    rank = case.get("rank", 0)
    lens = _lengths(case)
    packed = case.get("entry") == "varlen"

    def shape(n):
        return (n, H, D) if packed else (B, n, H, D)

    ks = [_normed(shape(n), g, dtype) for n in lens]
    vs = [_plain(shape(n), g, dtype) for n in lens]
    parallel_state.init_local_groups(case["N"], rank)
    group = parallel_state.get_usp_group()
    if kind == "block":
        channels = H * D
        lin = SimpleNamespace(heads=H, is_cross_attention=False)
        for name in ("to_q", "to_k", "to_v", "to_out"):
            m = torch.nn.Linear(channels, channels, device="cuda", dtype=dtype)
            with torch.no_grad():
                m.weight.copy_(torch.randn(channels, channels, generator=g, device="cuda") * channels ** -0.5)
                m.bias.copy_(0.1 * torch.randn(channels, generator=g, device="cuda"))
            setattr(lin, name, torch.nn.ModuleList([m, torch.nn.Dropout(0.0)]) if name == "to_out" else m)
        for name in ("norm_q", "norm_k"):
            m = torch.nn.LayerNorm(D, eps=1e-6, device="cuda", dtype=dtype)
            with torch.no_grad():
                m.weight.copy_(1.0 + 0.1 * torch.randn(D, generator=g, device="cuda"))
                m.bias.copy_(0.1 * torch.randn(D, generator=g, device="cuda"))
            setattr(lin, name, m)
        st.modules = lin
        n_video = Sq - case["text"]
        st.hidden = _plain((B, n_video, channels), g, dtype)
        st.text = _plain((B, case["text"], channels), g, dtype)
        angle = (torch.rand(n_video, D // 2, generator=g, device="cuda") * 6.28).repeat_interleave(2, -1)
        st.rope = (angle.cos().contiguous(), angle.sin().contiguous())
        st.proc = CVX_oCacheAttnProcessor(1)
        group.set_kv_chunks([None] + ks[1:], [None] + vs[1:])   # what the other ranks send
        utils.update_timestep(0)
        with torch.no_grad():
            st.proc(lin, st.hidden, st.text, image_rotary_emb=st.rope)
        return st

    st.q = _normed(shape(Sq), g, dtype)
    st.k, st.v = ks[rank], vs[rank]
    if packed:
        bounds = [0, Sq - case["pad"], Sq] if case["pad"] else [0, Sq]
        st.cu = torch.tensor(bounds, dtype=torch.int32, device="cuda")
        group.set_kv_chunks(ks, vs, cu_seqlens_kv=[st.cu] * case["N"])
        st.entry = Hunyuan_DiTangoProcessor(1)
        st.entry.oAttn.out_dtype = torch.float32 if case["out"] == "f32" else dtype
        st.q, st.k, st.v = (x.unsqueeze(0) for x in (st.q, st.k, st.v))
        st.steps = len(case["strides"].split(","))
        return st
    group.set_kv_chunks(ks, vs)
    if case.get("entry") == "step":
        st.entry = StepAttention(1)
    else:
        st.entry = proAttention(1, group)
        if kind != "exact":
            st.entry.out_dtype = torch.float32 if case["out"] == "f32" else dtype
    if kind == "mask":
        utils.update_timestep(0)
        st.entry.attn(st.q, st.k, st.v)
    elif kind == "exact":
        st.entry.fp32_inputs = "exact"
    else:
        st.steps = len(case["strides"].split(","))
    return st


@torch.no_grad()
def run(st):
    case, kind = st.case, st.kind
    if kind == "update":
        out = lse = None
        for block_out, block_lse in st.blocks:
            out, lse = utils.update_out_and_lse(out, lse, block_out, block_lse)
        return [out, lse]
    if kind == "cache":
        st.cache.store_block(3, st.out, st.lse)
        return list(st.cache.load_block(3))
    if kind == "producer":
        return [prepare_qk(st.q, **st.norm, **st.rope), prepare_qk(st.k, **st.norm, **st.rope)]
    _schedule(case)
    if kind == "mask":
        utils.update_timestep(1)
        out = st.entry.attn(st.q, st.k, st.v)
        return [out, st.entry.last_lse]
    if kind == "block":
        utils.update_timestep(1)
        return list(st.proc(st.modules, st.hidden, st.text, image_rotary_emb=st.rope))
    if kind == "exact":
        utils.update_timestep(0)
        out = st.entry.attn(st.q, st.k, st.v)
        return [out, st.entry.last_lse]
    outs = []
    for t in range(st.steps):
        utils.update_timestep(t)
        if case["entry"] == "varlen":
            n = case["Sq"]
            outs.append(st.entry.ringfusion_attn(st.q, st.k, st.v, cu_seqlens_q=st.cu, cu_seqlens_kv=st.cu, max_seqlen_q=n,
                                                 max_seqlen_kv=n))
        elif case["entry"] == "step":
            outs.append(st.entry.o_attn_func(st.q, st.k, st.v))
        else:
            outs.append(st.entry.attn(st.q, st.k, st.v))
    return outs


def _computed_chunks(case):
    """Chunks a stride generation recomputes at each step: the stride, and the local chunk where the target block is another."""
    N, rank, strides = case["N"], case["rank"], [int(s) for s in case["strides"].split(",")]
    done, target = [], 0
    for t, s in enumerate(strides):
        if s == N:
            target = rank
            done.append(N)
            continue
        first = (target // s) * s
        local = target != rank
        done.append(s + (1 if local and not first <= rank < first + s else 0))
        target = (target + s) % N
    return done


def work(case):
    kind, B, H, D, Sq = case["kind"], case["B"], case["H"], case["D"], case["Sq"]
    rows = B * Sq * H
    e = 4 if case["dtype"] == "f32" else 2
    state = rows * (2 * D + 4)
    result = rows * ((e if case.get("out") == "act" else 4) * D + 4)
    if kind == "update":
        return {"bytes": float(case["N"] * state + rows * (4 * D + 4)), "flops": float(case["N"] * rows * 2 * D)}
    if kind == "cache":
        return {"bytes": float(2 * rows * (4 * D + 4) + state), "flops": float(rows * D)}
    if kind == "producer":
        return {"bytes": float(4 * rows * D * 2 + 2 * (Sq - case["begin"]) * D * 4), "flops": float(2 * rows * D * 10)}
    lens = _lengths(case)
    if kind == "exact":
        kv = sum(lens)
        return {"bytes": float(rows * D * 4 + 2 * B * kv * H * D * 4 + result), "flops": 4.0 * rows * kv * D}
    if kind in ("mask", "block"):
        N, n = case["N"], case["computed"]
        kv = sum(lens) * n / N
        total = {"bytes": rows * D * 2 + 2 * B * kv * H * D * 2 + (n - 1) * state + (N - n) * state + result,
                 "flops": 4.0 * rows * kv * D}
        if kind == "block":   # projections of q, k, v and the output; hidden states in and out, weights
            total["flops"] += 4 * 2.0 * B * Sq * (H * D) ** 2
            total["bytes"] = 2 * rows * D * 2 + 4 * (H * D) ** 2 * 2 + 2 * B * (kv - Sq) * H * D * 2 + (n - 1) * state + (N - n) * state
        return {k: float(v) for k, v in total.items()}
    # a generation: every step reads its q and the K / V it recomputes, reads the states it reuses, writes the result
    N, steps = case["N"], [int(s) for s in case["strides"].split(",")]
    done = _computed_chunks(case)
    pad = case.get("pad", 0)
    pairs = float((Sq - pad) ** 2 + pad ** 2)
    total_bytes = 0.0
    for t, s in enumerate(steps):
        nxt = steps[t + 1] if t + 1 < len(steps) else N
        reused = N // s - 1
        kept = 0 if nxt == N else (N if s == N else 1)
        total_bytes += rows * D * 2 + 2 * done[t] * rows * D * 2 + (reused + kept) * state + result - rows * 4
    return {"bytes": total_bytes, "flops": 4.0 * B * H * D * pairs * sum(done)}


def tolerance(case):
    """About four times what the present code shows against the same computation in 64 bits (2-norm / largest element)."""
    kind, half = case["kind"], case["dtype"] == "fp16"
    if kind == "cache":
        return "exact"                                  # one rounding to bf16 and its exact widening
    if kind == "exact":
        return {"rel": 2.5e-6, "max": 1.5e-5}           # fp32 sums and exponentials: 5.9e-7 / 3.5e-6
    if kind == "update":
        return {"rel": 5e-7, "max": 4e-6}               # three fp32 products a value: 7e-8 / 5e-7
    if kind == "producer":                              # one rounding of the result: bf16 1.7e-3 / 3.9e-3, fp16 2.1e-4 / 4.9e-4
        return {"rel": 8e-4, "max": 2e-3} if half else {"rel": 6.5e-3, "max": 1.6e-2}
    # rounded probabilities and states: bf16 2.9e-3 / 1.4e-2, fp16 3.6e-4 / 1.9e-3
    return {"rel": 1.5e-3, "max": 8e-3} if half else {"rel": 1.1e-2, "max": 6e-2}
