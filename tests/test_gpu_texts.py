"""Texts encoded with batches enqueued ahead of the GPU: the results and the errors of one batch after the other."""
import weakref

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _encoder(gpu, length=128):
    import m2_amd
    cfg = m2_amd.m2_bert_80m(length)
    cfg.num_hidden_layers = 2
    model = m2_amd.BertModel(cfg)
    model.load_state_dict(m2_amd.seeded_state_dict(cfg, 11))
    return m2_amd.M2BertTextEncoder(model.to(gpu), max_seq_len=length)


def _texts(n, vocab=30000):
    g = torch.Generator().manual_seed(n)
    return [torch.randint(1, vocab, (int(k),), generator=g).tolist() for k in torch.randint(1, 160, (n,), generator=g)]


@pytest.mark.parametrize("n,batch", [(0, 4), (1, 4), (23, 3), (9, 1), (40, 16)])
def test_same_as_one_batch_at_a_time(gpu, n, batch):
    enc = _encoder(gpu)
    texts = _texts(n)
    got = enc.encode_token_ids(texts, batch)
    hook = enc.model.register_forward_hook(lambda *a: None)      # (a hook sees what it always saw)
    want = enc.encode_token_ids(texts, batch)
    hook.remove()
    assert got.shape == (n, 768) and got.dtype == np.float32 and np.array_equal(got, want)
    assert np.array_equal(enc.encode_token_ids([torch.tensor(t) for t in texts], batch), got)
    odd = [t if i % 3 else np.array(t) for i, t in enumerate(texts)]      # rows that torch.as_tensor is asked about
    assert np.array_equal(enc.encode_token_ids(odd, batch), got)
    masks = [[1] * len(t) for t in texts]
    assert np.array_equal(enc.encode_token_ids(texts, batch, attention_masks=masks), got)


def test_ids_and_masks_on_the_gpu(gpu):
    enc = _encoder(gpu)
    texts = _texts(11)
    masks = [[1 - i % 2 for i in range(len(t))] for t in texts]
    want = enc.encode_token_ids(texts, 4, attention_masks=masks)
    there = [torch.tensor(t).to(gpu) for t in texts]
    mthere = [torch.tensor(m).to(gpu) for m in masks]
    assert np.array_equal(enc.encode_token_ids(there, 4), want)      # (the mask is not used by the plain pooler)
    assert np.array_equal(enc.encode_token_ids(there, 4, attention_masks=mthere), want)
    assert np.array_equal(enc.encode_token_ids(there, 4, attention_masks=masks), want)
    assert np.array_equal(enc.encode_token_ids(texts, 4, attention_masks=mthere), want)
    assert np.array_equal(enc.encode_token_ids([t.int() for t in there], 4), want)


def test_pinned_memory_does_not_grow_with_the_texts(gpu, monkeypatch):
    enc = _encoder(gpu)
    texts, kept, most, empty = _texts(60), [], [0], torch.empty

    def counting(*args, **kw):
        t = empty(*args, **kw)
        if kw.get("pin_memory"):
            kept.append(weakref.ref(t))
            most[0] = max(most[0], sum(r() is not None for r in kept))
        return t

    monkeypatch.setattr(torch, "empty", counting)
    enc.encode_token_ids(texts, 2)
    # ids of the batch being put together and of the last, results of three
    assert len(kept) == 60 and most[0] <= 5 and not any(r() is not None for r in kept)


def test_what_a_caller_put_around_the_model_sees_every_call(gpu):
    import m2_amd
    enc = _encoder(gpu)
    texts, seen = _texts(9), []
    want = enc.encode_token_ids(texts, 4)
    hook = torch.nn.modules.module.register_module_forward_pre_hook(lambda m, a: seen.append(m))
    assert np.abs(enc.encode_token_ids(texts, 4) - want).max() < 2e-6      # (such a hook is to see the pooler's modules too)
    hook.remove()
    assert seen.count(enc.model) == 3

    class Counting(m2_amd.BertModel):
        def __call__(self, *args, **kwargs):
            seen.append(sorted(kwargs))
            return super().__call__(*args, **kwargs)

    enc.model.__class__ = Counting
    del seen[:]
    assert np.array_equal(enc.encode_token_ids(texts, 4), want) and seen == 3 * [["attention_mask", "input_ids"]]
    enc.model.__class__ = m2_amd.BertModel
    enc.model._compiled_call_impl = lambda *args, **kwargs: (seen.append(args), enc.model.forward(*args, **kwargs))[1]
    del seen[:]
    assert np.array_equal(enc.encode_token_ids(texts, 4), want) and len(seen) == 3
    enc.model._compiled_call_impl = None
    # a forward takes what it always took, and no keyword puts its check off
    with pytest.raises(IndexError):
        enc.model(torch.full((1, 128), 10 ** 6, device=gpu), ids_checked_later=True)


def test_errors(gpu):
    enc = _encoder(gpu)
    texts = _texts(20)
    want = enc.encode_token_ids(texts, 4)
    bad = list(texts)
    bad[9] = [5, 10 ** 6, 7]
    with pytest.raises(IndexError):
        enc.encode_token_ids(bad, 4)
    masks = [[1] * len(t) for t in texts]
    masks[18] = [1]
    texts[18] = [1, 2, 3]
    with pytest.raises(ValueError, match="text 18"):
        enc.encode_token_ids(texts, 4, attention_masks=masks)
    with pytest.raises(IndexError):                               # of an earlier batch, ahead of a later one's
        enc.encode_token_ids(bad[:18] + texts[18:], 4, attention_masks=[[1] * len(t) for t in bad[:18]] + masks[18:])
    texts = _texts(20)
    assert np.array_equal(enc.encode_token_ids(texts, 4), want)  # nothing of it is left
    enc.model.validate_ids = False
    assert np.isfinite(enc.encode_token_ids(bad, 4)).all()
    enc.model.validate_ids = True
    with pytest.raises(IndexError):                               # what nobody asked about is still there
        enc.model.embeddings.check_indices()
    assert np.isfinite(enc.encode_token_ids(texts, 4)).all()
    # ... and is not the error of a call that has looked nothing up
    enc.model.validate_ids = False
    enc.encode_token_ids(bad, 4)
    enc.model.validate_ids = True
    assert enc.encode_token_ids([], 4).shape == (0, 768)
    with pytest.raises(ValueError, match="text 0"):
        enc.encode_token_ids([[1, 2]], 4, attention_masks=[[1]])
    with pytest.raises(IndexError):
        enc.encode_token_ids(texts, 4)
    assert np.array_equal(enc.encode_token_ids(texts, 4), want)
