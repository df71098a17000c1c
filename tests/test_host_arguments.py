"""What the host side of a call accepts, as far as it shows without a GPU."""
import numpy as np
import pytest
import torch

from ditango_amd import _hip
from ditango_amd.core import config, parallel_state, redundancy_map
from ditango_amd.core.attention import proAttention


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
