"""What the host side of a call accepts, as far as it shows without a GPU."""
import numpy as np
import pytest
import torch

from ditango_amd import _hip
from ditango_amd.core import config, parallel_state, redundancy_map
from ditango_amd.core.attention import proAttention
from ditango_amd.executor.cogvideox import projection
from ditango_amd.executor.hunyuanvideo import attention_hunyuan


@pytest.mark.parametrize("kind", ["list", "tuple", "iterator", "generator", "stacked", "values"])
def test_chunk_table_takes_any_iterable_of_chunks(kind):
    """Each of them gets as far as the check of the first chunk."""
    chunks = [torch.zeros(1, 4, 1, 64, dtype=torch.bfloat16) for _ in range(2)]
    make = {"list": list, "tuple": tuple, "iterator": iter, "generator": lambda c: (x for x in c), "stacked": torch.stack,
            "values": lambda c: dict(enumerate(c)).values()}[kind]
    with pytest.raises(_hip.DitangoHipError, match=r"k\[0\] must live on the GPU"):
        _hip.ChunkTable(make(chunks), make(chunks))


class _OwnMap(redundancy_map.RedundancyMap):
    def get_curr_isp_stride(self, timestep, layer_id):
        return 7


@pytest.fixture(params=[True, False], ids=["host module", "no host module"])
def strides(request, monkeypatch):
    """proAttention's strides of a layer call from a map of 4 steps and 2 layers on a ring of 8."""
    if request.param:
        _hip._host()
    else:
        monkeypatch.setattr(_hip, "_host_module", None)
        monkeypatch.setattr(_hip, "HOST_PATH", _hip.HOST_PATH.with_name("absent.so"))
    parallel_state.init_local_groups(8, 0)
    cfg = config.init_config(None, num_inference_steps=4, num_layers=2)

    def of(timestep, layer_id, kind=redundancy_map.RedundancyMap, divider_map=None):
        rm = kind(cfg) if callable(kind) else kind
        if callable(kind):
            rm.base_weight = 8
            rm.divider_map = torch.tensor([[1, 2], [2, 4], [4, 8], [8, 1]]) if divider_map is None else divider_map
        monkeypatch.setattr(redundancy_map, "_redundancy_map", rm)
        attention = proAttention.__new__(proAttention)
        attention.layer_id = layer_id
        return attention._strides(timestep)

    return of


def test_strides_of_every_step_and_layer(strides):
    assert [[strides(t, i) for i in range(2)] for t in range(4)] == [[(8, 4), (4, 2)], [(4, 2), (2, 1)], [(2, 1), (1, 8)], [(1, 8), (8, 8)]]
    assert strides(-2, 1) == (1, 8) and strides(torch.tensor(1), 0) == (4, 2) and strides(np.int64(1), 0) == (4, 2)
    for outside in ((9, 0), (0, 5)):
        with pytest.raises(IndexError):
            strides(*outside)


@pytest.mark.parametrize("convert", [torch.Tensor.int, torch.Tensor.float, torch.Tensor.numpy, lambda m: torch.stack([m, m])[0].t().contiguous().t()])
def test_strides_from_other_maps(strides, convert):
    """Any array that is indexed by step and layer."""
    assert strides(1, 1, divider_map=convert(torch.tensor([[1, 2], [2, 4], [4, 8], [8, 1]]))) == (2, 1)


def test_strides_are_asked_of_the_map(strides):
    """A map of one's own overrides either of them, and needs nothing else."""
    assert strides(1, 1, kind=_OwnMap) == (7, 1)

    class Bare:
        get_curr_isp_stride = staticmethod(lambda timestep, layer_id: 3)
        get_next_isp_stride = staticmethod(lambda timestep, layer_id: 5)

    assert strides(0, 0, kind=Bare()) == (3, 5)


def test_producer_refuses_host_tensors_itself():
    with pytest.raises(_hip.DitangoHipError, match="x must be"):
        _hip.qk_norm_rope(torch.zeros(1, 4, 2, 64, dtype=torch.bfloat16))


@pytest.mark.parametrize("place", ["processor", "attention", "class", "own class"])
def test_hunyuan_processor_calls_a_replaced_varlen_attn(monkeypatch, place):
    """One packed sample takes a way without views, unless somebody listens at ``varlen_attn``."""
    parallel_state.init_local_groups(1, 0)
    seen = []

    def listen(*args, **kwargs):
        seen.append(tuple(args[-7].shape))
        return args[-7]

    monkeypatch.setattr(proAttention, "varlen_sample", lambda self, q, *args: seen.append("sample") or q)
    if place == "class":
        monkeypatch.setattr(proAttention, "varlen_attn", listen)
    processor = attention_hunyuan.Hunyuan_DiTangoProcessor(0)
    if place == "processor":
        processor.varlen_Attn = listen
    elif place == "attention":
        monkeypatch.setattr(processor.oAttn, "varlen_attn", listen)
        processor.varlen_Attn = processor.oAttn.varlen_attn
    elif place == "own class":
        processor.oAttn.__class__ = type("Own", (proAttention,), {"varlen_attn": listen})
        processor.varlen_Attn = processor.oAttn.varlen_attn
    q = torch.zeros(1, 6, 2, 64)
    cu = torch.tensor([0, 4, 6], dtype=torch.int32)
    out = processor.ringfusion_attn(q, q, q, cu_seqlens_q=cu, cu_seqlens_kv=cu, max_seqlen_q=6, max_seqlen_kv=6)
    assert out.shape == (1, 6, 128) and seen == [(6, 2, 64)]


def test_hunyuan_processor_of_one_sample_makes_no_views(monkeypatch):
    parallel_state.init_local_groups(1, 0)
    seen = []
    monkeypatch.setattr(proAttention, "varlen_sample", lambda self, q, *args: seen.append(tuple(q.shape)) or q)
    q = torch.zeros(1, 6, 2, 64)
    cu = torch.tensor([0, 4, 6], dtype=torch.int32)
    attention_hunyuan.Hunyuan_DiTangoProcessor(0).ringfusion_attn(q, q, q, cu_seqlens_q=cu, cu_seqlens_kv=cu, max_seqlen_q=6, max_seqlen_kv=6)
    assert seen == [(1, 6, 2, 64)]


def test_fused_projections_step_aside_for_whoever_sees_the_modules(monkeypatch):
    """Forward-mode derivatives (v carries its tangent to the caller of project_qkv) and a patched nn.Linear."""
    linear = torch.nn.Linear(64, 64)
    assert projection._only_arithmetic() and projection._plain(linear, torch.nn.Linear)
    with torch.autograd.forward_ad.dual_level():
        assert not projection._only_arithmetic()
    monkeypatch.setattr(torch.nn.Linear, "forward", lambda self, x: x)
    assert not projection._plain(linear, torch.nn.Linear)
