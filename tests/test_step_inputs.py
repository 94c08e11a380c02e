"""A captured step's inputs, copied in one launch that has no order, end up as if they had been copied one after the other."""

import ctypes

import pytest
import torch

from lite_llama_amd.executor import slots


@pytest.fixture(autouse=True)
def backwards(monkeypatch):
    """The launch on the host, last vector first."""
    def copy(todo):
        for to, of, words in reversed(todo):
            ctypes.memmove(to, of, 4 * words)
    monkeypatch.setattr(slots, "copy_words", copy)


def _vectors():
    return (torch.arange(8).view(8, 1), torch.arange(100, 108).view(8, 1), torch.arange(200, 208, dtype=torch.int32),
            torch.arange(300, 308, dtype=torch.int32), torch.arange(400, 408, dtype=torch.int32))


def _in_order(dst, src, batch):
    for d, s in zip(dst, src):
        if s.data_ptr() != d.data_ptr():
            d[:batch].copy_(s.view(d[:batch].shape))


@pytest.mark.parametrize("batch", [1, 3, 8])
@pytest.mark.parametrize("case", ["apart", "kept", "crossed", "shifted", "other types"])
def test_inputs_arrive_as_if_one_by_one(batch, case):
    def sources(d):
        own = [torch.full((batch, *v.shape[1:]), 7 + i, dtype=v.dtype) for i, v in enumerate(d)]
        if case == "kept":
            own[2], own[3] = d[2][:batch], d[3][:batch]
        elif case == "crossed":   # positions from where the ids go, lengths from where the slots go
            own[1], own[3] = d[0][:batch], d[2][:batch]
        elif case == "shifted":
            own[4] = d[3][8 - batch:]
        elif case == "other types":
            own[0], own[3] = own[0].int(), own[3].long()
        return own

    a, b = _vectors(), _vectors()
    slots.feed(tuple(zip(a, sources(a))), batch)
    _in_order(b, sources(b), batch)
    for x, y in zip(a, b):
        assert torch.equal(x, y)


def test_a_vector_of_another_length_is_refused():
    d = torch.arange(8).view(8, 1)
    with pytest.raises(RuntimeError):
        slots.feed(((d, torch.zeros(3, dtype=torch.int64)),), 2)
