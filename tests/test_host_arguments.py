"""What the host side of a call accepts, as far as it shows without a GPU."""
import pytest
import torch

from ditango_amd import _hip


@pytest.mark.parametrize("kind", ["list", "tuple", "iterator", "generator", "stacked", "values"])
def test_chunk_table_takes_any_iterable_of_chunks(kind):
    """Each of them gets as far as the check of the first chunk."""
    chunks = [torch.zeros(1, 4, 1, 64, dtype=torch.bfloat16) for _ in range(2)]
    make = {"list": list, "tuple": tuple, "iterator": iter, "generator": lambda c: (x for x in c), "stacked": torch.stack,
            "values": lambda c: dict(enumerate(c)).values()}[kind]
    with pytest.raises(_hip.DitangoHipError, match=r"k\[0\] must live on the GPU"):
        _hip.ChunkTable(make(chunks), make(chunks))
