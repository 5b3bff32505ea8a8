"""Embedding-inference caller: batches of texts -> pooled embeddings, the loop of the reference's
`M2_BERT_Encoder.encode_queries` / `encode_corpus` (bert/embeddings_inference.py:267-351).

The reference tokenises with a Hugging Face tokenizer it downloads; here the tokenizer is whatever
callable the caller passes (`tokenizer([text], return_tensors="pt")` -> mapping with `input_ids` and
`attention_mask` of shape (1, n), which is the Hugging Face calling convention), or the caller passes
token ids directly to `encode_token_ids`.
"""
from __future__ import annotations

from array import array
from collections import deque
from typing import Callable, Dict, Iterable, List, Optional, Sequence

import numpy as np
import torch
import torch.nn as nn
import torch.nn.functional as F

from .encoder import BertModel, called_plainly


def split_list(items: Sequence, chunk_size: int) -> Iterable[Sequence]:
    """Consecutive chunks of at most chunk_size items (bert/embeddings_inference.py:60-62)."""
    for i in range(0, len(items), chunk_size):
        yield items[i:i + chunk_size]


def pad_or_truncate(ids: torch.Tensor, length: int) -> torch.Tensor:
    """(1, n) -> (1, length): zero padding on the right, or truncation (`expand_tensor` followed by the slice,
    bert/embeddings_inference.py:38-43,278-283)."""
    if ids.shape[1] < length:
        ids = F.pad(ids, [0, length - ids.shape[1]])
    return ids[:, :length]


def _host_row(row) -> Optional[np.ndarray]:
    """A list or tuple of whole numbers, or an integer CPU tensor, as a flat int64 array; None for anything else, which torch.as_tensor
    is asked about (floats, empty and nested lists, strings, ...)."""
    if isinstance(row, torch.Tensor):
        return row.detach().reshape(-1).numpy() if row.dtype == torch.int64 and row.device.type == "cpu" else None
    if type(row) in (list, tuple) and len(row) > 0:
        try:
            return np.frombuffer(array("q", row), np.int64)
        except (TypeError, OverflowError):
            return None
    return None


class M2BertTextEncoder:
    """`model`: a BertModel with a pooler, on the GPU, in eval mode.  Every text is padded or cut to
    `max_seq_len` tokens (the reference's `evaluation_max_seq_len`), texts are run `batch_size` at a time and the
    pooled outputs are collected on the host."""

    def __init__(self, model: BertModel, max_seq_len: int, tokenizer: Optional[Callable] = None,
                 device: Optional[torch.device] = None):
        if model.pooler is None:
            raise ValueError("the embedding caller needs a BertModel built with add_pooling_layer=True")
        self.model = model.eval()
        self.max_seq_len = int(max_seq_len)
        self.tokenizer = tokenizer
        self.device = device if device is not None else next(model.parameters()).device

    # -- the loop ----------------------------------------------------------------------------------
    def encode_token_ids(self, token_ids: Sequence, batch_size: int,
                         attention_masks: Optional[Sequence] = None) -> np.ndarray:
        """token_ids: one 1-D sequence of ids per text (any lengths, may be empty); returns (len(token_ids), d)
        fp32.  Without attention_masks every given token counts as real and the padding as masked."""
        out = [torch.empty(0, self.model.config.hidden_size)]
        if self._plain_model():
            self._run_ahead(token_ids, batch_size, attention_masks, out)
        else:
            for lo in range(0, len(token_ids), batch_size):
                hi = min(lo + batch_size, len(token_ids))
                ids_b, mask_b = self._assemble(token_ids, attention_masks, lo, hi)
                with torch.no_grad():
                    _, pooled = self.model(input_ids=ids_b.to(self.device), attention_mask=mask_b.to(self.device))
                out.append(pooled.detach().float().cpu())
        out = torch.cat(out, 0)
        if torch.isnan(out).any():
            raise ValueError("NaNs in the encoded texts")
        return out.numpy()

    def _plain_model(self) -> bool:
        """The model's forward is the one of this package, with nothing around it that would see its call."""
        m = self.model
        return (type(m).forward is BertModel.forward and type(m).__call__ is nn.Module.__call__ and called_plainly(m)
                and torch.device(self.device).type == "cuda")

    def _run_ahead(self, token_ids: Sequence, batch_size: int, attention_masks: Optional[Sequence], out: List[torch.Tensor]) -> None:
        """The batches enqueued up to two ahead of the GPU: while one is computed the next is put together, in pinned memory that the GPU
        fetches by itself, and nothing is waited for but the batch before the last (waiting for each batch's copies and for its check
        of the token ids left the GPU idle for 0.7 ms between two batches of 32 x 512: 75 texts 9.7 ms, now 8.7; 512 texts 60.9, now 48.1).  The ids are checked
        once, behind the last batch or ahead of another error."""
        emb, pending, asked = self.model.embeddings, deque(), False

        def finish():
            host, done = pending.popleft()
            done.synchronize()
            out.append(host.clone())      # (pageable: the pinned block goes back for the batch after the next)

        try:
            for lo in range(0, len(token_ids), batch_size):
                hi = min(lo + batch_size, len(token_ids))
                both = torch.empty(2, hi - lo, self.max_seq_len, dtype=torch.int64, pin_memory=True)
                rows = self._assemble(token_ids, attention_masks, lo, hi, both)
                with torch.no_grad():
                    if rows[0].data_ptr() == both.data_ptr():
                        ids_b, mask_b = both.to(self.device, non_blocking=True).unbind(0)
                    else:      # (put together from tensors, wherever those are)
                        ids_b, mask_b = (t.to(self.device) for t in rows)
                    asked = True
                    _, pooled = self.model._forward(ids_b, None, mask_b, None, False, None, check_ids=False)
                host = torch.empty(pooled.shape, dtype=torch.float32, pin_memory=True)
                host.copy_(pooled.detach().float(), non_blocking=True)
                done = torch.cuda.Event()
                done.record(torch.cuda.current_stream(pooled.device))
                pending.append((host, done))
                if len(pending) > 2:
                    finish()
            while pending:
                finish()
        finally:
            if asked and self.model.validate_ids:      # (without a batch, an earlier unchecked forward's flag is nobody's error here)
                emb.check_indices()

    def _assemble(self, token_ids: Sequence, attention_masks: Optional[Sequence], lo: int, hi: int, into: Optional[torch.Tensor] = None):
        """Texts [lo, hi) as padded or cut (hi - lo, max_seq_len) ids and mask.  Rows are written into two arrays, the halves of `into` where
        given, 7 us a text of up to 512 tokens; a torch tensor per text, its mask, both padded and all of them concatenated took 41 (3 ms of
        75 texts).  Rows that no array can be written from (on the GPU, of floats, ...) come as tensors of their own."""
        L = self.max_seq_len
        both = np.empty((2, hi - lo, L), np.int64) if into is None else into.numpy()
        both[...] = 0
        ids_b, mask_b = both
        for k in range(lo, hi):
            ids = _host_row(token_ids[k])
            mask = None if attention_masks is None else _host_row(attention_masks[k])
            if ids is None or (mask is None and attention_masks is not None):
                return self._assemble_tensors(token_ids, attention_masks, lo, hi)
            if mask is not None and mask.shape != ids.shape:
                raise ValueError(f"text {k}: {ids.shape[0]} token ids but {mask.shape[0]} mask entries")
            n = min(ids.shape[0], L)
            ids_b[k - lo, :n] = ids[:n]
            mask_b[k - lo, :n] = 1 if mask is None else mask[:n]
        return torch.from_numpy(ids_b), torch.from_numpy(mask_b)

    def _assemble_tensors(self, token_ids: Sequence, attention_masks: Optional[Sequence], lo: int, hi: int):
        """The same for whatever torch.as_tensor takes."""
        ids_rows, mask_rows = [], []
        for k in range(lo, hi):
            ids = torch.as_tensor(token_ids[k], dtype=torch.long).reshape(1, -1)
            mask = torch.ones_like(ids) if attention_masks is None else \
                torch.as_tensor(attention_masks[k], dtype=torch.long).reshape(1, -1)
            if mask.shape != ids.shape:
                raise ValueError(f"text {k}: {ids.shape[1]} token ids but {mask.shape[1]} mask entries")
            ids_rows.append(pad_or_truncate(ids, self.max_seq_len))
            mask_rows.append(pad_or_truncate(mask, self.max_seq_len))
        return torch.cat(ids_rows, 0), torch.cat(mask_rows, 0)

    def _encode_texts(self, texts: List[str], batch_size: int) -> np.ndarray:
        if self.tokenizer is None:
            raise ValueError("no tokenizer was given: use encode_token_ids, or pass tokenizer= to the constructor")
        ids, masks = [], []
        for text in texts:
            enc = self.tokenizer([text], return_tensors="pt")
            ids.append(enc["input_ids"].reshape(-1))
            masks.append(enc["attention_mask"].reshape(-1))
        return self.encode_token_ids(ids, batch_size, attention_masks=masks)

    # -- the reference's two entry points ------------------------------------------------------------
    def encode_queries(self, queries: List[str], batch_size: int, **kwargs) -> np.ndarray:
        return self._encode_texts(list(queries), batch_size)

    def encode_corpus(self, corpus: List[Dict[str, str]], batch_size: int, **kwargs) -> np.ndarray:
        """Passages are dicts with 'title' and 'text'; the title is prepended when the model reads at least
        512 tokens (bert/embeddings_inference.py:316-319)."""
        if self.max_seq_len >= 512:
            texts = [p["title"] + " " + p["text"] for p in corpus]
        else:
            texts = [p["text"] for p in corpus]
        return self._encode_texts(texts, batch_size)
