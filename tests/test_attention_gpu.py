"""End-to-end parity of the drop-in API (proAttention / proCache / RedundancyMap on the
HIP kernels) against the numeric oracle on identical seeded inputs.

Bar: out max-abs <= 2e-2 (bf16 states), lse max-abs <= 1e-3 (fp32), schedule bit-exact.
"""
import numpy as np
import pytest
import torch

from oracle import attention_math as om
from oracle import mask_schedule as ms
from oracle.state_machine import RingOracle, strides_from_dividers

pytestmark = pytest.mark.gpu

OUT_TOL, LSE_TOL = 2e-2, 1e-3


@pytest.fixture
def env(hip):
    from ditango_amd.core import config, parallel_state, redundancy_map as rmod
    from ditango_amd import utils

    def make(N, rank, T, L, **cfg):
        parallel_state.init_local_groups(N, rank)
        config.init_config(None, num_inference_steps=T, num_layers=L, **cfg)
        rmod.destroy_redundancy_map()
        rmod._redundancy_map = rmod.RedundancyMap(config.get_config())
        return rmod.get_redundancy_map()

    yield make
    from ditango_amd.core import parallel_state, redundancy_map as rmod
    rmod.destroy_redundancy_map()
    parallel_state.destroy_local_groups()
    utils.update_timestep(0)


def _inputs(B, Sq, lens, H, D, seed, norm=None):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(B, Sq, H, D, generator=g)
    ks = [torch.randn(B, n, H, D, generator=g) for n in lens]
    vs = [torch.randn(B, n, H, D, generator=g) for n in lens]
    if norm == "rms":
        q = q / q.pow(2).mean(-1, keepdim=True).sqrt()
        ks = [k / k.pow(2).mean(-1, keepdim=True).sqrt() for k in ks]
    return q, ks, vs


def _perturb(x, g):
    return x + 0.01 * torch.randn(x.shape, generator=g)


def _cmp(out, lse_bsh1, ref_out, ref_lse_bhs, what):
    out = out.float().cpu()
    lse = lse_bsh1.cpu().squeeze(-1).transpose(1, 2)
    err = (out - ref_out).abs().max().item()
    lerr = (lse - ref_lse_bhs).abs().max().item()
    rel = (out - ref_out).norm().item() / max(ref_out.norm().item(), 1e-30)
    print(f"{what}: out max-abs {err:.3e} rel-l2 {rel:.3e} lse max-abs {lerr:.3e}", flush=True)
    assert err <= OUT_TOL and lerr <= LSE_TOL and rel <= 1e-2, what


@pytest.mark.parametrize("N,rank,D,col,max_job_chunks", [
    (4, 1, 128, (1, 1, 1, 2, 2, 2, 1, 4, 2, 2, 1, 1), None),     # includes the stride-1 -> 2 misalignment
    (8, 3, 64, (1, 1, 1, 4, 4, 4, 2, 2, 2, 2, 1, 1), None),
    (8, 0, 128, (1, 1, 1, 8, 8, 4, 4, 2, 1, 8, 1, 1), None),
    # the same with blocks of more than 3 chunks computed in pieces that are folded into the block's state
    # (what a ring of 128 positions and more needs at the real limit of 32 chunks per job)
    (8, 5, 128, (1, 1, 1, 4, 4, 2, 2, 2, 1, 2, 1, 1), 3),
    # a ring of 64 positions (strides 64 / 32 / 16 / 8, two-level ring above 8): a full-stride step that
    # announces stride 8 files 64 fine-grained states, more than one merge launch or chunk table holds
    (64, 37, 64, (1, 1, 1, 8, 8, 4, 4, 2, 1, 8, 1, 1), None),
])
def test_stride_mode_matches_numeric_oracle(env, N, rank, D, col, max_job_chunks):
    from ditango_amd.core.attention import proAttention
    from ditango_amd.core.parallel_state import get_usp_group
    from ditango_amd.utils import update_timestep

    T, B, H, S = len(col), 1, 2, 100
    rm = env(N, rank, T, 1)
    rm.divider_map[:, 0] = torch.tensor(col)
    curr, nxt = strides_from_dividers(N, col)
    g = torch.Generator().manual_seed(17)
    q, ks, vs = _inputs(B, S, [S] * N, H, D, seed=N * 10 + rank)
    state = {}

    def attn_fn(r, c):
        if r != rank:
            return (c,)
        o, l = om.chunk_attention(state["q"], state["ks"][c], state["vs"][c])
        return (o, l)

    def merge_fn(a, b):
        if isinstance(b[0], int):
            return tuple(b) if a is None else tuple(a) + tuple(b)
        return om.update_out_and_lse(None if a is None else a[0], None if a is None else a[1], b[0], b[1])

    def store_fn(s):
        if isinstance(s[0], int):
            return s
        return (om.bf16_round(s[0]), s[1])

    ring = RingOracle(N, attn_fn=attn_fn, merge_fn=merge_fn, store_fn=store_fn)
    attn = proAttention(0, get_usp_group())
    if max_job_chunks is not None:
        attn._MAX_JOB_CHUNKS = max_job_chunks
    group = get_usp_group()
    for t in range(T):
        print(f"case stride N={N} rank={rank} D={D} t={t} curr={curr[t]} next={nxt[t]}", flush=True)
        qb, kb, vb = q.bfloat16(), [k.bfloat16() for k in ks], [v.bfloat16() for v in vs]
        state.update(q=qb, ks=kb, vs=vb)
        tr = ring.call(t, curr[t], nxt[t])[rank]
        update_timestep(t)
        dk = [k.cuda() for k in kb]
        dv = [v.cuda() for v in vb]
        group.set_kv_chunks(dk, dv)
        out = attn.attn(qb.cuda(), dk[rank], dv[rank])
        torch.cuda.synchronize()
        p = attn.last_plan
        assert p.computed == tr.computed and p.reuse_merged == tr.reuse_merged and p.stores == tr.stores
        assert p.target_after == tr.target_after and p.occupancy_after == tr.occupancy_after
        assert out.dtype == torch.float32 and tuple(out.shape) == (B, S, H, D)
        ref_out, ref_lse = tr.out
        _cmp(out, attn.last_lse, ref_out, ref_lse.squeeze(-1).transpose(1, 2), f"t={t}")
        q, ks, vs = _perturb(q, g), [_perturb(k, g) for k in ks], [_perturb(v, g) for v in vs]


@pytest.mark.parametrize("N,rank,D,col,trip", [
    (8, 3, 128, (1, 1, 1, 4, 4, 2, 2, 1, 1), {2}),        # trips on the step that announces stride 2
    (8, 0, 64, (1, 1, 1, 2, 2, 2, 2, 2, 1, 1), {4}),      # mid-run: one of two blocks held, the other predicted
    (4, 2, 128, (1, 1, 1, 2, 2, 2, 4, 4, 1, 1), {2, 5}),
])
def test_stride_mode_memory_guard_fallback_matches_numeric_oracle(env, N, rank, D, col, trip):
    """The stride-mode fallback of the memory guard (core/attention.py:97-98 with core/cache.py:103-128),
    run on the kernels with an injected memory reading against the lock-step ring with the same reading:
    on the tripping call the announced stride becomes N, nothing is stored and the cache is reset to N
    empty slots; the NEXT call reads its stride from the map again, probes blocks of the empty cache and
    computes only its target block, so the other chunks are missing from its softmax -- schedule and
    numbers (out, lse of the partial softmax) must equal the oracle's."""
    from ditango_amd.core.attention import proAttention
    from ditango_amd.core.parallel_state import get_usp_group
    from ditango_amd.utils import update_timestep

    T, B, H, S = len(col), 1, 2, 100
    rm = env(N, rank, T, 1)
    rm.divider_map[:, 0] = torch.tensor(col)
    curr, nxt = strides_from_dividers(N, col)
    g = torch.Generator().manual_seed(29)
    q, ks, vs = _inputs(B, S, [S] * N, H, D, seed=N * 7 + rank)
    state, now = {}, {"t": 0}
    probe = lambda: 950.0 if now["t"] in trip else 0.0       # MB allocated; budget 1000 MB, one block 100 MB

    def attn_fn(r, c):
        if r != rank:
            return (c,)
        return om.chunk_attention(state["q"], state["ks"][c], state["vs"][c])

    def merge_fn(a, b):
        if isinstance(b[0], int):
            return tuple(b) if a is None else tuple(a) + tuple(b)
        return om.update_out_and_lse(None if a is None else a[0], None if a is None else a[1], b[0], b[1])

    def store_fn(s):
        return s if isinstance(s[0], int) else (om.bf16_round(s[0]), s[1])

    ring = RingOracle(N, attn_fn=attn_fn, merge_fn=merge_fn, store_fn=store_fn,
                      memory_probe=probe, block_size_mb=100.0, memory_constraint=1000.0)
    group = get_usp_group()
    attn = proAttention(0, group)
    attn.cache.block_size_mb, attn.cache.memory_constraint, attn.cache.memory_probe = 100.0, 1000.0, probe
    tripped, dropped = set(), 0
    for t in range(T):
        print(f"case guard N={N} rank={rank} D={D} t={t} curr={curr[t]} next={nxt[t]} trip={t in trip}", flush=True)
        now["t"] = t
        qb, kb, vb = q.bfloat16(), [k.bfloat16() for k in ks], [v.bfloat16() for v in vs]
        state.update(q=qb, ks=kb, vs=vb)
        tr = ring.call(t, curr[t], nxt[t])[rank]
        update_timestep(t)
        dk, dv = [k.cuda() for k in kb], [v.cuda() for v in vb]
        group.set_kv_chunks(dk, dv)
        out = attn.attn(qb.cuda(), dk[rank], dv[rank])
        torch.cuda.synchronize()
        p = attn.last_plan
        assert (p.curr_stride, p.next_stride) == (tr.curr_stride, tr.next_stride)
        assert p.computed == tr.computed and p.reuse_probed == tr.reuse_probed and p.reuse_merged == tr.reuse_merged
        assert p.stores == tr.stores and p.flushes == tr.flushes
        assert (p.target_after, p.nblk_after, p.occupancy_after) == (tr.target_after, tr.nblk_after, tr.occupancy_after)
        if tr.next_stride != nxt[t]:
            tripped.add(t)
            assert p.next_stride == N and p.stores == [] and attn.cache.curr_block_num == N
            assert all(o is None for o in attn.cache.out_block_cache) and all(l is None for l in attn.cache.lse_block_cache)
        if t - 1 in tripped and curr[t] != N:
            assert p.reuse_probed and p.reuse_merged == []
            dropped += N - len({c for c, _ in p.computed})
        ref_out, ref_lse = tr.out
        _cmp(out, attn.last_lse, ref_out, ref_lse.squeeze(-1).transpose(1, 2), f"guard t={t}")
        q, ks, vs = _perturb(q, g), [_perturb(k, g) for k in ks], [_perturb(v, g) for v in vs]
    assert tripped == trip and dropped > 0


@pytest.mark.parametrize("C,diag,D,p,lens", [
    (8, 0, 128, 0.5, None),
    (8, 5, 64, 0.6, None),
    (6, -1, 128, 0.75, [70, 69, 69, 70, 1, 64]),     # ragged chunks, no local chunk
    (48, 5, 128, 0.5, None),                         # more chunks than one launch addresses: two windows
    (70, 43, 64, 0.6, None),                         # local chunk in the second window; 70-way merge
    (48, 5, 128, 0.5, [90] * 40 + [0] * 8),          # the second window holds no key at all: it is not launched,
                                                     # its scheduled chunks get the empty state (out 0, lse -inf)
])
def test_mask_mode_matches_numeric_oracle(env, C, diag, D, p, lens):
    from ditango_amd.core.attention import proAttention
    from ditango_amd.core.parallel_state import get_usp_group
    from ditango_amd.utils import update_timestep

    T, L, B, H, Sq = 5, 2, 1, 3, 90
    lens = lens or [Sq] * C
    rank = max(diag, 0)
    rm = env(C, rank, T, L)
    mask = ms.seeded_mask(T, L, C, p, seed=C + D, diag=diag)
    rm.set_chunk_mask(mask, diag=diag)
    comp, reu, cnt = ms.build_schedule_table(mask, diag)
    assert np.array_equal(rm.sched_compute_ids.cpu().numpy(), comp)      # schedule bit-exact
    assert np.array_equal(rm.sched_reuse_ids.cpu().numpy(), reu)
    assert np.array_equal(rm.sched_counts.cpu().numpy(), cnt)
    group = get_usp_group()
    layers = [proAttention(l, group) for l in range(L)]
    oracles = [ms.MaskCacheOracle(C, diag) for _ in range(L)]
    g = torch.Generator().manual_seed(23)
    q, ks, vs = _inputs(B, Sq, lens, H, D, seed=C, norm="rms")
    for t in range(T):
        update_timestep(t)
        for l in range(L):
            print(f"case mask C={C} diag={diag} D={D} t={t} l={l} row={mask[t, l].tolist()}", flush=True)
            qb, kb, vb = q.bfloat16(), [k.bfloat16() for k in ks], [v.bfloat16() for v in vs]
            (ref_out, ref_lse), c_ids, r_ids = oracles[l].call(
                mask[t, l], lambda c: om.chunk_attention(qb, kb[c], vb[c]),
                lambda sts: om.merge_states_closed_form([s[0] for s in sts], [s[1] for s in sts]),
                lambda s: (om.bf16_round(s[0]), s[1]))
            dk, dv = [k.cuda() for k in kb], [v.cuda() for v in vb]
            group.set_kv_chunks(dk, dv)
            out = layers[l].attn(qb.cuda(), dk[rank], dv[rank])
            torch.cuda.synchronize()
            _cmp(out, layers[l].last_lse, ref_out, ref_lse, f"t={t} l={l}")
            q, ks, vs = _perturb(q, g), [_perturb(k, g) for k in ks], [_perturb(v, g) for v in vs]


@pytest.mark.parametrize("N,rank,S_total,D", [(8, 7, 8 * 90 - 3, 128), (4, 3, 4 * 130 - 1, 64)])
def test_zero_padded_shards_of_an_uneven_sequence(env, N, rank, S_total, D):
    """The callers shard an uneven sequence with ``split_tensor_uneven`` (utils.py:86-136): the last shards
    carry a zero-padded row, and the dense path does not mask it (utils.py:120-127) -- a padded key takes
    part in the softmax with score 0, a padded query row is computed like any other.  Shards built by the
    drop-in ``split_tensor_uneven`` go through ``attn`` (a full-stride call and a cached one) and must equal
    the oracle on those same zero-padded chunks; and against attention over the UNPADDED sequence the merged
    lse must be off by exactly the padded keys: exp(lse) = exp(lse_unpadded) + number of padded keys."""
    from ditango_amd.core.attention import proAttention
    from ditango_amd.core.parallel_state import get_usp_group
    from ditango_amd.utils import get_padding_dict, split_tensor_uneven, update_timestep

    B, H = 1, 3
    col = (1, 1, 2, 2, 1)
    T = len(col)
    rm = env(N, rank, T, 1)
    rm.divider_map[:, 0] = torch.tensor(col)
    curr, nxt = strides_from_dividers(N, col)
    g = torch.Generator().manual_seed(S_total)
    q_full = torch.randn(B, S_total, H, D, generator=g).bfloat16()
    k_full = torch.randn(B, S_total, H, D, generator=g).bfloat16()
    v_full = torch.randn(B, S_total, H, D, generator=g).bfloat16()
    qs = split_tensor_uneven(q_full, N, dim=1, tensor_name="q")
    ks = split_tensor_uneven(k_full, N, dim=1, tensor_name="k")
    vs = split_tensor_uneven(v_full, N, dim=1, tensor_name="v")
    pads = get_padding_dict()["k"]
    n_pad = sum(pads)
    assert n_pad == N - S_total % N and pads[rank] == 1 and all(k.shape[1] == -(-S_total // N) for k in ks)
    state = dict(q=qs[rank], ks=ks, vs=vs)

    def attn_fn(r, c):
        return (c,) if r != rank else om.chunk_attention(state["q"], state["ks"][c], state["vs"][c])

    def merge_fn(a, b):
        if isinstance(b[0], int):
            return tuple(b) if a is None else tuple(a) + tuple(b)
        return om.update_out_and_lse(None if a is None else a[0], None if a is None else a[1], b[0], b[1])

    ring = RingOracle(N, attn_fn=attn_fn, merge_fn=merge_fn,
                      store_fn=lambda s: s if isinstance(s[0], int) else (om.bf16_round(s[0]), s[1]))
    group = get_usp_group()
    attn = proAttention(0, group)
    dk, dv = [k.cuda() for k in ks], [v.cuda() for v in vs]
    group.set_kv_chunks(dk, dv)
    # attention of the local queries over the unpadded sequence (the padded query row attends like a zero query)
    ex_out, ex_lse = om.chunk_attention(qs[rank], k_full, v_full)
    for t in range(T):
        print(f"case padded shards N={N} rank={rank} D={D} t={t} curr={curr[t]}", flush=True)
        tr = ring.call(t, curr[t], nxt[t])[rank]
        update_timestep(t)
        out = attn.attn(qs[rank].cuda(), dk[rank], dv[rank])
        torch.cuda.synchronize()
        assert attn.last_plan.computed == tr.computed and attn.last_plan.stores == tr.stores
        ref_out, ref_lse = tr.out
        _cmp(out, attn.last_lse, ref_out, ref_lse.squeeze(-1).transpose(1, 2), f"padded t={t}")
        # inputs do not change between the steps, so every step sees all N chunks: padded keys add exactly n_pad
        lse = attn.last_lse.cpu().squeeze(-1).transpose(1, 2).double()
        assert torch.allclose(lse.exp(), ex_lse.double().exp() + n_pad, rtol=2e-3)
        w = (ex_lse.double().exp() / (ex_lse.double().exp() + n_pad)).transpose(1, 2).unsqueeze(-1)
        assert (out.cpu().double() - ex_out.double() * w).abs().max() <= OUT_TOL
    # the padded query row (a zero query: uniform attention over all keys, padded ones included)
    mean_v = torch.cat(vs, dim=1).float().sum(1) / (N * ks[0].shape[1])
    assert (out.cpu()[:, -1] - mean_v).abs().max() <= OUT_TOL


@pytest.mark.parametrize("T,layer,step,same_as", [(3, 0, -1, (0, 2)), (3, 1, -2, (1, 1)), (3, -1, 1, (1, 1)), (4, -2, -1, (0, 3))])
def test_mask_mode_steps_and_layers_count_from_the_end(env, T, layer, step, same_as):
    """A step or layer number below zero means the mask's row counted from the end, for the host's lists and for the row of the
    device schedule alike: the same chunks are recomputed and the same result comes out, bit for bit."""
    from ditango_amd import utils
    from ditango_amd.core import parallel_state
    from ditango_amd.core.attention import proAttention
    rm = env(4, 0, T, 2)
    mask = np.zeros((T, 2, 4), dtype=np.uint8)
    for t in range(1, T):
        for l in range(2):
            mask[t, l, 1 + (t + l) % 3] = 1
    rm.set_chunk_mask(mask, diag=0)
    q, ks, vs = _inputs(1, 200, [90] * 4, 2, 64, seed=3)
    q = q.bfloat16().cuda()
    outs = []
    for l, t in ((same_as[0], same_as[1]), (layer, step)):
        g = torch.Generator().manual_seed(5)
        attn = proAttention(l, parallel_state.get_usp_group())
        for now in (0, t):                       # other K and V at the second step: the reused chunk shows in the result
            k, v = ([x.bfloat16().cuda() + 0.5 * torch.randn(x.shape, generator=g).bfloat16().cuda() for x in xs] for xs in (ks, vs))
            parallel_state.get_usp_group().set_kv_chunks(k, v)
            utils.update_timestep(now)
            out = attn.attn(q, k[0], v[0])
        outs.append((out, attn.last_lse))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


def test_mask_mode_cold_reuse_is_an_error(env):
    from ditango_amd.core.attention import proAttention
    from ditango_amd.core.parallel_state import get_usp_group
    rm = env(4, 0, 2, 1)
    mask = np.zeros((2, 1, 4), dtype=np.uint8)
    mask[0, 0, 2] = 1      # reuse at the very first step: nothing stored yet
    rm.set_chunk_mask(mask, diag=0)
    q, ks, vs = _inputs(1, 64, [64] * 4, 1, 64, seed=1)
    group = get_usp_group()
    group.set_kv_chunks([k.bfloat16().cuda() for k in ks], [v.bfloat16().cuda() for v in vs])
    with pytest.raises(RuntimeError, match="reuse chunk 2"):
        proAttention(0, group).attn(q.bfloat16().cuda(), group.kv_chunk(0)[0], group.kv_chunk(0)[1])


def test_config1_cpu_plumbing_case(env):
    """B=1, H=4, D=64, Q 512 tokens, KV 2048 in 4 chunks of 512,
    N(0,1) seed 0; chunks 1 and 3 come from states cached at step t-1 on inputs that differ
    by 1% Gaussian noise, chunks 0 and 2 are recomputed and LSE-merged.  (The configuration
    is stated for fp32 on the reference's torch path; the kernels take bf16, so inputs are
    rounded to bf16 for both sides.)"""
    from ditango_amd.core.attention import proAttention
    from ditango_amd.core.parallel_state import get_usp_group
    from ditango_amd.utils import update_timestep
    B, H, D, Sq, C = 1, 4, 64, 512, 4
    rm = env(C, 0, 2, 1)
    mask = np.zeros((2, 1, C), dtype=np.uint8)
    mask[1, 0, [1, 3]] = 1
    rm.set_chunk_mask(mask, diag=0)
    g0 = torch.Generator().manual_seed(0)
    q1 = torch.randn(B, Sq, H, D, generator=g0)
    k1 = [torch.randn(B, 512, H, D, generator=g0) for _ in range(C)]
    v1 = [torch.randn(B, 512, H, D, generator=g0) for _ in range(C)]
    g1 = torch.Generator().manual_seed(1)
    q0, k0, v0 = _perturb(q1, g1), [_perturb(k, g1) for k in k1], [_perturb(v, g1) for v in v1]   # step t-1
    group = get_usp_group()
    attn = proAttention(0, group)
    orc = ms.MaskCacheOracle(C, 0)
    merge = lambda sts: om.merge_states_closed_form([s[0] for s in sts], [s[1] for s in sts])
    for t, (q, ks, vs) in enumerate([(q0, k0, v0), (q1, k1, v1)]):
        qb, kb, vb = q.bfloat16(), [k.bfloat16() for k in ks], [v.bfloat16() for v in vs]
        (ref_out, ref_lse), comp, reuse = orc.call(mask[t, 0], lambda c: om.chunk_attention(qb, kb[c], vb[c]), merge,
                                                   lambda s: (om.bf16_round(s[0]), s[1]))
        update_timestep(t)
        dk, dv = [k.cuda() for k in kb], [v.cuda() for v in vb]
        group.set_kv_chunks(dk, dv)
        out = attn.attn(qb.cuda(), dk[0], dv[0])
        torch.cuda.synchronize()
        _cmp(out, attn.last_lse, ref_out, ref_lse, f"config1 t={t}")
    assert comp == [0, 2] and reuse == [1, 3]
    # stale-but-close: the cached result stays near exact attention on the step-t inputs
    exact, _ = om.full_attention(q1.bfloat16(), [k.bfloat16() for k in k1], [v.bfloat16() for v in v1])
    assert (out.cpu() - exact).abs().max() < 5e-2


def test_config1_fp32_inputs_as_stated(env):
    """BASELINE configuration 1 with the fp32 tensors handed over as they are: the driver rounds them
    to bf16 at the kernel boundary (flash_attn_func itself takes no fp32).  Two comparisons: the strict
    bar against the oracle on the rounded inputs (same numbers as test_config1_cpu_plumbing_case), and
    the distance to fp32 attention of the UNROUNDED inputs, which is the price of the bf16 inputs:
    observed 8.6e-4 in out and 1.3e-3 in lse for N(0,1) inputs at D = 64; the test allows 5e-3 / 5e-3."""
    from ditango_amd.core.attention import proAttention
    from ditango_amd.core.parallel_state import get_usp_group
    from ditango_amd.utils import update_timestep
    B, H, D, Sq, C = 1, 4, 64, 512, 4
    rm = env(C, 0, 2, 1)
    mask = np.zeros((2, 1, C), dtype=np.uint8)
    mask[1, 0, [1, 3]] = 1
    rm.set_chunk_mask(mask, diag=0)
    g0 = torch.Generator().manual_seed(0)
    q1 = torch.randn(B, Sq, H, D, generator=g0)
    k1 = [torch.randn(B, 512, H, D, generator=g0) for _ in range(C)]
    v1 = [torch.randn(B, 512, H, D, generator=g0) for _ in range(C)]
    g1 = torch.Generator().manual_seed(1)
    q0, k0, v0 = _perturb(q1, g1), [_perturb(k, g1) for k in k1], [_perturb(v, g1) for v in v1]
    group = get_usp_group()
    attn = proAttention(0, group)
    merge = lambda sts: om.merge_states_closed_form([s[0] for s in sts], [s[1] for s in sts])
    orc_rounded, orc_fp32 = ms.MaskCacheOracle(C, 0), ms.MaskCacheOracle(C, 0)
    for t, (q, ks, vs) in enumerate([(q0, k0, v0), (q1, k1, v1)]):
        qb, kb, vb = q.bfloat16(), [k.bfloat16() for k in ks], [v.bfloat16() for v in vs]
        (ref_out, ref_lse), _, _ = orc_rounded.call(mask[t, 0], lambda c: om.chunk_attention(qb, kb[c], vb[c]), merge,
                                                    lambda s: (om.bf16_round(s[0]), s[1]))
        (f_out, f_lse), _, _ = orc_fp32.call(mask[t, 0], lambda c: om.chunk_attention(q, ks[c], vs[c]), merge)
        update_timestep(t)
        dk, dv = [k.cuda() for k in ks], [v.cuda() for v in vs]          # fp32 on the device
        group.set_kv_chunks(dk, dv)
        out = attn.attn(q.cuda(), dk[0], dv[0])
        torch.cuda.synchronize()
        assert out.dtype == torch.float32
        _cmp(out, attn.last_lse, ref_out, ref_lse, f"config1 fp32 inputs t={t}, oracle on rounded inputs")
        err = (out.cpu() - f_out).abs().max().item()
        lerr = (attn.last_lse.cpu().squeeze(-1).transpose(1, 2) - f_lse).abs().max().item()
        print(f"config1 fp32 inputs t={t}: distance to fp32 attention of the unrounded inputs: out {err:.3e} lse {lerr:.3e}",
              flush=True)
        assert err <= 5e-3 and lerr <= 5e-3
    with pytest.raises(TypeError):
        attn.attn(q1.double().cuda(), dk[0], dv[0])


def test_config1_fp32_exact_mode_meets_the_stated_bar(env):
    """BASELINE configuration 1 as stated, fp32 end to end: with ``fp32_inputs = "exact"`` every fresh state is
    computed and merged in fp32 from the fp32 tensors (dt_attn_chunk_f32_fwd); only the states that go into the
    cache (chunks 1 and 3, reused at step t) are rounded to bf16, the cache's storage format.  Two references:
    (a) the same flow restated on the CPU (fresh fp32, cached bf16): agreement to fp32 rounding error, plus at
    most one bf16 ulp of a cached element where the two fp32 values round to different neighbours; (b) the
    reference's torch math path proper, fp32 with nothing rounded anywhere: the stated bar (out 2e-2, lse 1e-3)
    holds with almost two (out) and three (lse) orders of magnitude to spare.  The schedule is bit-exact."""
    from ditango_amd.core.attention import proAttention
    from ditango_amd.core.parallel_state import get_usp_group
    from ditango_amd.utils import update_timestep
    B, H, D, Sq, C = 1, 4, 64, 512, 4
    rm = env(C, 0, 2, 1)
    mask = np.zeros((2, 1, C), dtype=np.uint8)
    mask[1, 0, [1, 3]] = 1
    rm.set_chunk_mask(mask, diag=0)
    g0 = torch.Generator().manual_seed(0)
    q1 = torch.randn(B, Sq, H, D, generator=g0)
    k1 = [torch.randn(B, 512, H, D, generator=g0) for _ in range(C)]
    v1 = [torch.randn(B, 512, H, D, generator=g0) for _ in range(C)]
    g1 = torch.Generator().manual_seed(1)
    q0, k0, v0 = _perturb(q1, g1), [_perturb(k, g1) for k in k1], [_perturb(v, g1) for v in v1]
    group = get_usp_group()
    attn = proAttention(0, group)
    attn.fp32_inputs = "exact"
    merge = lambda sts: om.merge_states_closed_form([s[0] for s in sts], [s[1] for s in sts])
    cached_bf16, cached_fp32 = {}, {}
    for t, (q, ks, vs) in enumerate([(q0, k0, v0), (q1, k1, v1)]):
        comp, reuse = ms.build_schedule(mask[t, 0], 0)
        fresh = {c: om.chunk_attention(q, ks[c], vs[c]) for c in comp}
        ref_out, ref_lse = merge([cached_bf16[c] for c in reuse] + [fresh[c] for c in comp])      # (a)
        pure_out, pure_lse = merge([cached_fp32[c] for c in reuse] + [fresh[c] for c in comp])    # (b)
        for c in comp:
            if c != 0:
                cached_bf16[c] = (om.bf16_round(fresh[c][0]), fresh[c][1])
                cached_fp32[c] = fresh[c]
        update_timestep(t)
        dk, dv = [k.cuda() for k in ks], [v.cuda() for v in vs]
        group.set_kv_chunks(dk, dv)
        out = attn.attn(q.cuda(), dk[0], dv[0])
        torch.cuda.synchronize()
        got_lse = attn.last_lse.cpu().squeeze(-1).transpose(1, 2)
        err, lerr = (out.cpu() - ref_out).abs().max().item(), (got_lse - ref_lse).abs().max().item()
        perr, plerr = (out.cpu() - pure_out).abs().max().item(), (got_lse - pure_lse).abs().max().item()
        print(f"config1 fp32 exact t={t}: vs same flow on the CPU out {err:.3e} lse {lerr:.3e}; "
              f"vs fp32 with nothing rounded out {perr:.3e} lse {plerr:.3e}", flush=True)
        assert err <= (1e-5 if t == 0 else 2e-3) and lerr <= 1e-5
        assert perr <= 2e-3 and plerr <= 1e-5
        assert perr <= OUT_TOL and plerr <= LSE_TOL            # the stated bar
    assert comp == [0, 2] and reuse == [1, 3]
    assert attn.last_plan is None                              # mask mode: the schedule is the committed mask's


def test_stride_mode_fp32_exact(env):
    """The exact-fp32 mode under the reference's stride schedule (ring of 4): fresh block states are
    fp32, stored blocks are rounded to bf16 as they enter the cache; against the lock-step oracle."""
    from ditango_amd.core.attention import proAttention
    from ditango_amd.core.parallel_state import get_usp_group
    from ditango_amd.utils import update_timestep
    N, rank, D, col = 4, 2, 64, (1, 1, 1, 4, 2, 2, 1, 2, 1, 1)
    T, B, H, S = len(col), 1, 2, 70
    rm = env(N, rank, T, 1)
    rm.divider_map[:, 0] = torch.tensor(col)
    curr, nxt = strides_from_dividers(N, col)
    g = torch.Generator().manual_seed(5)
    q, ks, vs = _inputs(B, S, [S] * N, H, D, seed=77)
    state = {}

    def attn_fn(r, c):
        return (c,) if r != rank else om.chunk_attention(state["q"], state["ks"][c], state["vs"][c])

    def merge_fn(a, b):
        if isinstance(b[0], int):
            return tuple(b) if a is None else tuple(a) + tuple(b)
        return om.update_out_and_lse(None if a is None else a[0], None if a is None else a[1], b[0], b[1])

    ring = RingOracle(N, attn_fn=attn_fn, merge_fn=merge_fn,
                      store_fn=lambda s: s if isinstance(s[0], int) else (om.bf16_round(s[0]), s[1]))
    group = get_usp_group()
    attn = proAttention(0, group)
    attn.fp32_inputs = "exact"
    for t in range(T):
        state.update(q=q, ks=ks, vs=vs)
        tr = ring.call(t, curr[t], nxt[t])[rank]
        update_timestep(t)
        dk, dv = [k.cuda() for k in ks], [v.cuda() for v in vs]
        group.set_kv_chunks(dk, dv)
        out = attn.attn(q.cuda(), dk[rank], dv[rank])
        torch.cuda.synchronize()
        assert attn.last_plan.computed == tr.computed and attn.last_plan.stores == tr.stores
        ref_out, ref_lse = tr.out
        _cmp(out, attn.last_lse, ref_out, ref_lse.squeeze(-1).transpose(1, 2), f"stride fp32 exact t={t}")
        q, ks, vs = _perturb(q, g), [_perturb(k, g) for k in ks], [_perturb(v, g) for v in vs]


def test_mask_mode_memory_guard_recomputes_without_arena(env):
    """A layer whose state arena does not fit under the memory budget keeps no states and computes
    every chunk on every call (what the reference's guard falls back to, core/attention.py:97-98):
    the result is full attention whatever the mask says, and no arena is allocated."""
    from ditango_amd.core.attention import proAttention
    from ditango_amd.core.parallel_state import get_usp_group
    from ditango_amd.utils import update_timestep
    B, H, D, Sq, C, T = 1, 2, 128, 80, 5, 3
    rm = env(C, 0, T, 2)
    mask = ms.seeded_mask(T, 2, C, 0.6, seed=3, diag=0)
    rm.set_chunk_mask(mask, diag=0)
    q, ks, vs = _inputs(B, Sq, [Sq, 70, 1, 64, 90], H, D, seed=9)
    group = get_usp_group()
    tight, roomy = proAttention(0, group), proAttention(1, group)
    tight.cache.memory_probe = lambda: 1000.0
    tight.cache.memory_constraint = 1000.2          # the arena (6 states of 80 KB) would not fit
    g = torch.Generator().manual_seed(2)
    for t in range(T):
        update_timestep(t)
        qb, kb, vb = q.bfloat16(), [k.bfloat16() for k in ks], [v.bfloat16() for v in vs]
        dk, dv = [k.cuda() for k in kb], [v.cuda() for v in vb]
        group.set_kv_chunks(dk, dv)
        out = tight.attn(qb.cuda(), dk[0], dv[0])
        roomy.attn(qb.cuda(), dk[0], dv[0])
        torch.cuda.synchronize()
        ref_out, ref_lse = om.full_attention(qb, kb, vb)
        _cmp(out, tight.last_lse, ref_out, ref_lse, f"no arena t={t}")
        q, ks, vs = _perturb(q, g), [_perturb(k, g) for k in ks], [_perturb(v, g) for v in vs]
    assert tight.cache.arena_out is None and roomy.cache.arena_out is not None


def test_fp16_inputs_run_as_fp16(env):
    """flash_attn_func takes fp16 as well as bf16: fp16 tensors run on the fp16 MFMA with fp16 states, they are
    not rounded to bf16 at the boundary.  The result is fp32 attention of the fp16 inputs to an fp16 pipeline's
    accuracy (1e-3 / 2e-4 here; rounding the inputs to bf16 first would cost 5e-3).  More in test_fp16_gpu.py."""
    from ditango_amd.core.attention import proAttention
    from ditango_amd.core.parallel_state import get_usp_group
    B, H, D, S, N = 1, 2, 128, 200, 2
    env(N, 0, 1, 1)
    g = torch.Generator().manual_seed(12)
    q = torch.randn(B, S, H, D, generator=g).half()
    ks = [torch.randn(B, S, H, D, generator=g).half() for _ in range(N)]
    vs = [torch.randn(B, S, H, D, generator=g).half() for _ in range(N)]
    group = get_usp_group()
    group.set_kv_chunks([k.cuda() for k in ks], [v.cuda() for v in vs])
    attn = proAttention(0, group)
    out = attn.attn(q.cuda(), ks[0].cuda(), vs[0].cuda())
    torch.cuda.synchronize()
    assert out.dtype == torch.float32
    f_out, f_lse = om.full_attention(q.float(), [k.float() for k in ks], [v.float() for v in vs])
    lse = attn.last_lse.cpu().squeeze(-1).transpose(1, 2)
    assert (out.cpu() - f_out).abs().max() <= 1e-3 and (lse - f_lse).abs().max() <= 2e-4


def test_update_out_and_lse_dropin(hip):
    from ditango_amd.utils import update_out_and_lse
    g = torch.Generator().manual_seed(4)
    B, S, H, D = 1, 77, 2, 128
    blocks = [(torch.randn(B, S, H, D, generator=g).bfloat16(), torch.randn(B, H, S, generator=g)) for _ in range(3)]
    o = l = ro = rl = None
    for bo, bl in blocks:
        o, l = update_out_and_lse(o, l, bo.cuda(), bl.cuda())
        ro, rl = om.update_out_and_lse(ro, rl, bo, bl)
    torch.cuda.synchronize()
    assert o.dtype == torch.float32 and tuple(l.shape) == (B, S, H, 1)
    assert (o.cpu() - ro).abs().max() < 1e-5 and (l.cpu() - rl).abs().max() < 1e-5


def test_cache_coarsening_in_place(hip):
    """proCache._merge_blocks on the GPU == closed-form merge of the member states."""
    from ditango_amd.core.cache import proCache
    g = torch.Generator().manual_seed(5)
    B, S, H, D, N = 1, 65, 2, 64, 8
    cache = proCache(N, 0)
    states = {}
    for i in (0, 1, 3, 4, 5, 6):      # block 2 and 7 empty
        o, l = torch.randn(B, S, H, D, generator=g), torch.randn(B, S, H, 1, generator=g)
        cache.store_block(i, o.cuda(), l.cuda())        # fp32 + [B,S,H,1]: goes through dt_cache_store
        states[i] = (om.bf16_round(o), l.squeeze(-1).transpose(1, 2))
    cache.update_cache_blocks(4, 1)                      # 8 -> 2 blocks of 4, block 1 invalidated
    torch.cuda.synchronize()
    assert cache.curr_block_num == 2 and cache.out_block_cache[1] is None
    ref_out, ref_lse = om.merge_states_closed_form([states[i][0] for i in (0, 1, 3)], [states[i][1] for i in (0, 1, 3)])
    o, l = cache.get_block(0)
    assert o.dtype == torch.bfloat16 and (o.float().cpu() - ref_out).abs().max() < 2e-2
    assert (l.cpu() - ref_lse).abs().max() < 1e-5
    lo, ll = cache.load_block(0)
    assert lo.dtype == torch.float32 and tuple(ll.shape) == (B, S, H, 1)
    with pytest.raises(IndexError):
        cache.get_block(5)


def test_profiling_mode_records_rel_l1(env):
    from ditango_amd.core.attention import proAttention
    from ditango_amd.core.parallel_state import get_usp_group
    from ditango_amd.utils import update_timestep
    N, T = 2, 3
    rm = env(N, 0, T, 1)
    rm.enable_auto_setting()
    group = get_usp_group()
    attn = proAttention(0, group)
    g = torch.Generator().manual_seed(9)
    q, ks, vs = _inputs(1, 80, [80, 80], 2, 64, seed=3)
    outs = []
    for t in range(T):
        update_timestep(t)
        qb, kb, vb = q.bfloat16(), [k.bfloat16() for k in ks], [v.bfloat16() for v in vs]
        group.set_kv_chunks([k.cuda() for k in kb], [v.cuda() for v in vb])
        assert attn.last_plan is None or attn.last_plan.curr_stride == N   # profiling forces full stride
        outs.append(attn.attn(qb.cuda(), group.kv_chunk(0)[0], group.kv_chunk(0)[1]).cpu())
        q, ks, vs = _perturb(q, g), [_perturb(k, g) for k in ks], [_perturb(v, g) for v in vs]
    rm._sync_redundancy()
    assert rm.redundancy_map[0, 0] == 0
    for t in (1, 2):
        assert abs(rm.redundancy_map[t, 0].item() - om.rel_l1(outs[t], outs[t - 1])) < 1e-5


def test_bf16_result_and_producer_feed_the_attention(env):
    """The caller-side chain in one piece: q/k/v read in place from a fused QKV projection, RMSNorm +
    RoPE by dt_qk_norm_rope, cached block attention, result written as bf16 by the merge
    (out_dtype); against the oracle's norm + RoPE + full attention on the same inputs."""
    from oracle import producer as P
    from ditango_amd.core.attention import proAttention
    from ditango_amd.core.parallel_state import get_usp_group
    from ditango_amd.producer import prepare_qk
    from ditango_amd.utils import update_timestep

    C, B, H, D, Sq = 4, 1, 5, 128, 96
    rm = env(C, 0, 2, 1)
    rm.set_chunk_mask(np.zeros((2, 1, C), dtype=np.uint8), diag=0)
    g = torch.Generator().manual_seed(31)
    qkv = torch.randn(B, C * Sq, 3, H, D, generator=g).bfloat16()
    wq, wk = torch.rand(D, generator=g) + 0.5, torch.rand(D, generator=g) + 0.5
    th = torch.rand(C * Sq, D // 2, generator=g) * 6.28
    cos, sin = th.cos().repeat_interleave(2, -1), th.sin().repeat_interleave(2, -1)
    # oracle
    qn = P.qk_norm_rope(qkv[:, :, 0], P.NORM_RMS, wq, None, 1e-6, P.ROPE_INTERLEAVED, cos, sin).bfloat16()
    kn = P.qk_norm_rope(qkv[:, :, 1], P.NORM_RMS, wk, None, 1e-6, P.ROPE_INTERLEAVED, cos, sin).bfloat16()
    ref_out, ref_lse = om.chunk_attention(qn[:, :Sq], kn, qkv[:, :, 2])
    # product
    dev = qkv.cuda()
    qd = prepare_qk(dev[:, :, 0], norm="rms", weight=wq, rope="interleaved", freqs_cis=(cos, sin))
    kd = prepare_qk(dev[:, :, 1], norm="rms", weight=wk, rope="interleaved", freqs_cis=(cos, sin))
    vd = prepare_qk(dev[:, :, 2])
    group = get_usp_group()
    group.set_kv_chunks(list(kd.split(Sq, dim=1)), list(vd.split(Sq, dim=1)))
    layer = proAttention(0, group)
    layer.out_dtype = torch.bfloat16
    update_timestep(0)
    out = layer.attn(qd[:, :Sq], kd[:, :Sq], vd[:, :Sq])
    torch.cuda.synchronize()
    assert out.dtype == torch.bfloat16 and out.shape == (B, Sq, H, D)
    _cmp(out, layer.last_lse, ref_out, ref_lse, "producer + attention + bf16 result")


def test_profiling_to_divider_map_end_to_end(hip, tmp_path):
    """redundancy_preprocess (two "prompts") -> finish_auto_setting -> .pt on disk -> init_redundancy_map
    -> dividers -> a generation pass that reuses cached states.  The recorded map equals the oracle's
    rel_l1 sums, the dividers equal the oracle's generate + refine on that map, and the cached pass
    follows the lock-step oracle of the state machine."""
    from oracle import divider_map as od
    from ditango_amd.core import config, parallel_state, redundancy_map as rmod
    from ditango_amd.core.attention import proAttention
    from ditango_amd.utils import update_timestep

    N, T, L, B, H, D, S = 4, 8, 2, 1, 2, 64, 72
    pct, dv = [0, 40, 90], [4, 2, 1, 1]
    parallel_state.init_local_groups(N, 1)
    cfg = config.init_config(None, num_inference_steps=T, num_layers=L, stride_percentiles=pct, stride_dividers=dv,
                             ditango_base=str(tmp_path), model_name="toy")
    rmod.destroy_redundancy_map()
    try:
        rm = rmod.init_redundancy_map(cfg, quiet=True)          # nothing on disk yet: full stride
        group = parallel_state.get_usp_group()
        recorded = torch.zeros(T, L)

        def make_inputs(seed):
            g = torch.Generator().manual_seed(seed)
            base = _inputs(B, S, [S] * N, H, D, seed=seed, norm="rms")
            steps = []
            q, ks, vs = base
            for t in range(T):
                steps.append((q.bfloat16(), [k.bfloat16() for k in ks], [v.bfloat16() for v in vs]))
                q, ks, vs = _perturb(q, g), [_perturb(k, g) for k in ks], [_perturb(v, g) for v in vs]
            return steps

        def generate(prompt, seed_of, check=None):
            layers = [proAttention(l, group) for l in range(L)]
            steps = make_inputs(seed_of[prompt])
            prev = [None] * L
            for t in range(T):
                update_timestep(t)
                qb, kb, vb = steps[t]
                group.set_kv_chunks([k.cuda() for k in kb], [v.cuda() for v in vb])
                for l in range(L):
                    out = layers[l].attn(qb.cuda(), group.kv_chunk(1)[0], group.kv_chunk(1)[1]).cpu()
                    if check is None:
                        if prev[l] is not None:
                            recorded[t, l] += om.rel_l1(out, prev[l])
                        prev[l] = out
                    else:
                        check(t, l, layers[l], out, steps[t])

        seeds = {"a": 5, "b": 6}
        rmod.redundancy_preprocess(generate, {"seed_of": seeds}, prompt_list=["a", "b"])
        assert not rm.auto_setting
        path = tmp_path / "configs" / "toy" / f"redundancy_map_{T}_{L}.pt"
        saved = torch.load(str(path), weights_only=True)
        assert saved.shape == (T, L) and (saved[0] == 0).all()
        assert (saved - recorded).abs().max() < 2e-5
        # a fresh process would now find the file
        rmod.destroy_redundancy_map()
        rm = rmod.init_redundancy_map(cfg, quiet=True)
        div, _ = od.generate_divider_map(saved.numpy(), N, pct, dv)
        refined, _ = od.refine_divider_map(div)
        assert np.array_equal(rm.divider_map.numpy(), refined)
        assert (refined[3:T - 2] > 1).any(), "the toy map should leave something to reuse"
        # the cached pass follows the state-machine oracle call by call
        oracles = [RingOracle(N) for _ in range(L)]

        def check(t, l, layer, out, step):
            qb, kb, vb = step
            curr, nxt = od.curr_stride(refined, N, t, l), od.next_stride(refined, N, t, l)
            traces = oracles[l].call(t, curr, nxt)
            tr = traces[1]
            assert list(layer.last_plan.computed) == list(tr.computed), (t, l)

        generate("a", seeds, check=check)
    finally:
        rmod.destroy_redundancy_map()
        parallel_state.destroy_local_groups()
        update_timestep(0)
