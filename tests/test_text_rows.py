"""Batches of texts put together row by row against the same batches put together from tensors, for every form of a text that either
takes, on the CPU."""
import numpy as np
import pytest
import torch

from m2_amd.embed import M2BertTextEncoder


class _Encoder(M2BertTextEncoder):
    def __init__(self, length):
        self.max_seq_len = length


def _both(texts, masks=None, length=6):
    enc = _Encoder(length)
    out = []
    for f in (enc._assemble, enc._assemble_tensors):
        try:
            out.append(f(texts, masks, 0, len(texts)))
        except Exception as e:
            out.append(e)
    return out


@pytest.mark.parametrize("texts", [
    [[1, 2, 3], list(range(9)), [4]], [(1, 2), [True, 2], [3]], [[1], []], [[1], torch.tensor([2, 3])], [torch.arange(12).view(3, 4)], [np.arange(4)],
    [torch.tensor([1, 2], dtype=torch.int32), [5]], [[1.5, 2.5]], [[1, 2.7]], [[1, 2 ** 40]], [[-1, 3]], [[np.int64(3), 4]], [[[1, 2], [3, 4]]],
    [torch.empty(0, dtype=torch.long)], [torch.arange(20)[::3]], [torch.tensor(7)], [["1", "2"]], [[1, "2"]], [[1, None]], [[2 ** 63]], [[1, [2]]], [5], ["12"]])
def test_rows_and_tensors_agree(texts):
    rows, tensors = _both(texts)
    if isinstance(tensors, Exception):
        assert type(rows) is type(tensors)
    else:
        assert all(torch.equal(a, b) and a.dtype == b.dtype for a, b in zip(rows, tensors))


@pytest.mark.parametrize("masks", [[[1, 0], [1] * 8], [torch.tensor([1, 1]), [0] * 8], [[1, 1], [1.0] * 8], [[1], [1] * 8], [[1, 2, 3], [1] * 8]])
def test_masks(masks):
    rows, tensors = _both([[3, 4], list(range(8))], masks)
    if isinstance(tensors, Exception):
        assert type(rows) is type(tensors) and str(rows) == str(tensors)
    else:
        assert all(torch.equal(a, b) for a, b in zip(rows, tensors))
