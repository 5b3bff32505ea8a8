"""The native schedule of an encoder: embeddings, filter generation and all layers enqueued by three library calls.

`BertEncoder._run_layers` walks over its layers in Python, about 170 us of host time per layer and 0.2 ms more for the
filter table, which is what a short forward then costs whatever the GPU does (L = 128, B = 1: 2.4 ms for 0.75 ms of
kernels).  A `StackPlan` holds what the calls need: the layers' device pointers, the bf16 and packed copies of the
weights, the filter pointer table.  It is made once and, before each use, compared with what the modules hold now, tensor
by tensor (storage, address and shape, and version counter for the weights that copies were made from) and value by value:
`_param_check.Checker`.

Same kernels in the same order on the current stream as the Python schedule, hence the same bits.  It serves row counts
whose projections run on the library's own kernels; larger forwards, whose host time hides behind the GPU's, and encoders
with per-layer options, modules of other classes or computed weights stay with the Python schedule.
"""
from __future__ import annotations

import ctypes
import warnings
from typing import List, Optional

import torch

from . import encoder as _encoder, ops
from ._lib import LayerParams, check, lib
from .blockdiag import BlockdiagLinear
from .hyena import HyenaFilter
from .mixer import MonarchMixerSequenceMixing

try:
    from . import _param_check
except ImportError as e:
    # built against torch's internals, unlike the library with its plain C interface: without it everything runs, short forwards
    # with the Python schedule's host time
    _param_check = None
    warnings.warn(f"m2_amd/_param_check.so is missing or does not fit this torch ({e}): short forwards take the slower Python schedule; "
                  "build it with `python m2_amd/build.py`", RuntimeWarning)


_IN_PLACE, _COPIED = False, True       # read at its address / a copy was made from it: compare the version too


class _Slots:
    """(dict, key) of every module, (dict, key, compare the version) of every tensor and (dict, key) of every plain value that
    something depends on.  What is not there, or not what the modules are built with, is a ValueError: the Python schedule asks
    the modules themselves."""

    def __init__(self):
        self.modules, self.tensors, self.values = [], [], []

    def child(self, mod, key, kind=None):
        found = mod._modules.get(key)
        if found is None or (kind is not None and type(found) is not kind):
            raise ValueError(f"{key} is not the module it was built as")
        self.modules.append((mod._modules, key))
        return found

    def tensor(self, mod, key, how=_IN_PLACE, shape=None):
        where = mod._parameters if key in mod._parameters else mod._buffers
        t = where.get(key)
        if t is None:                                  # absent, or computed (a parametrisation, weight_norm, pruning)
            raise ValueError(f"{key} is not a plain parameter")
        self.tensors.append((where, key, how))
        if not (t.is_cuda and t.dtype == torch.float32 and t.is_contiguous()):
            raise ValueError("parameters that are not plain fp32")
        if shape is not None and t.shape != shape:      # the kernels take sizes, not shapes: never read beyond a tensor
            raise ValueError(f"{key} of shape {tuple(t.shape)} where {shape} is expected")
        return t

    def value(self, obj, key):
        if key not in obj.__dict__:
            raise ValueError(f"no plain attribute {key}")
        self.values.append((obj.__dict__, key))
        return obj.__dict__[key]

    def checker(self):
        return _param_check.Checker(self.modules, self.tensors, self.values)


class EmbedPart:
    """Device pointers of the embeddings in front of a stack.  Host work only: it can be made at any time."""

    def __init__(self, e, d: int):
        slots = _Slots()
        child, tensor, value = slots.child, slots.tensor, slots.value
        word, typ = tensor(child(e, "word_embeddings"), "weight"), tensor(child(e, "token_type_embeddings"), "weight")
        pos = tensor(child(e, "position_embeddings"), "weight") if value(e, "use_positional_encodings") else None
        if any(t is not None and (t.dim() != 2 or t.shape[1] != d) for t in (word, typ, pos)):
            raise ValueError("embedding tables of another width")
        ln = child(e, "LayerNorm")
        g, b = tensor(ln, "weight", shape=(d,)), tensor(ln, "bias", shape=(d,))
        slots.tensors.append((e._buffers, "_bad_index", _IN_PLACE))
        self.of, self.d = e, d
        self.args = (word.data_ptr(), typ.data_ptr(), None if pos is None else pos.data_ptr(), word.shape[0], typ.shape[0],
                     0 if pos is None else pos.shape[0], g.data_ptr(), b.data_ptr(), float(value(ln, "eps")))
        self.bad_index = e._bad_index.data_ptr()
        self.checker = slots.checker()

    def __reduce__(self):
        return type(None), ()


def embed_part(model, d: int) -> Optional[EmbedPart]:
    """The part of `model`'s embeddings as they are now, made or re-used, or None where their own forward serves."""
    part = model._embed_part
    if part is None or part.of is not model.embeddings or part.d != d or not part.checker.unchanged():
        try:
            part = EmbedPart(model.embeddings, d)
        except ValueError:
            return None
        model._embed_part = part
    return part


class StackPlan:
    """Device pointers of an encoder's layers for one length, for every row count: what any of them reads is made with the plan, so
    that a forward of another batch size needs nothing that a stream capture could not make."""

    def __init__(self, encoder, L: int):
        slots = _Slots()
        slots.modules.append((encoder._modules, "layer"))
        child, tensor, value = slots.child, slots.tensor, slots.value
        stack = encoder._modules["layer"]
        n = len(stack._modules)
        self.layers = n
        self.arrays = [(LayerParams * n)(), None, None]        # plain; with the streaming product's packed weights; with the MLP's
        self.keep: List[torch.Tensor] = []
        rows, skips = [], []
        for i, key in enumerate(stack._modules):
            lay = child(stack, key)
            at, mlp = child(lay, "attention"), child(lay, "mlp")
            for name in ("filter_fn", "filter_fn2")[:2 if value(at, "residual_long_conv") else 1]:
                f = child(at, name, HyenaFilter)
                skips.append(tensor(f, "bias"))
                emb = child(f, "pos_emb")
                fwd = child(f, "implicit_filter")
                mod = child(f, "modulation")
                for key_ in ("order", "emb_dim", "w_mod"):
                    value(f, key_)
                value(mod, "shift")
                row = [tensor(emb, "z"), tensor(emb, "t"), tensor(child(fwd, "1"), "freq"), tensor(mod, "deltas")]
                for seq in (fwd, child(f, "implicit_filter_rev") if value(f, "bidirectional") else None):
                    if seq is None:
                        row += [None] * 7
                        continue
                    for k in "024":
                        lin = child(seq, k)
                        row += [tensor(lin, "weight"), tensor(lin, "bias")]
                    row.append(tensor(child(seq, "6"), "weight"))
                rows.append(row)
            lin_in, lin_out, short = child(at, "in_linear"), child(at, "out_linear"), child(at, "short_filter")
            gated, wo, ln = child(mlp, "gated_layers", BlockdiagLinear), child(mlp, "wo", BlockdiagLinear), child(mlp, "layernorm")
            cfg = value(mlp, "config")
            d, I, nb = value(at, "d_model"), value(cfg, "intermediate_size"), value(cfg, "monarch_mlp_nblocks")
            if d % nb or I % nb:
                raise ValueError("padded blocks")
            in_place = [tensor(lin_in, "bias", shape=(3 * d,)), tensor(lin_out, "bias", shape=(d,)),
                        tensor(short, "weight", shape=(3 * d, 1, 3)), tensor(short, "bias", shape=(3 * d,)),
                        tensor(wo, "bias", shape=(d,)), tensor(ln, "weight", shape=(d,)), tensor(ln, "bias", shape=(d,))]
            for m, shape in ((lin_in, (3 * d, d)), (lin_out, (d, d)), (gated, (nb, 2 * I // nb, d // nb)), (wo, (nb, d // nb, I // nb))):
                tensor(m, "weight", _COPIED, shape)
            w_in, w_out = at._cast("in_w", lin_in.weight, torch.bfloat16), at._cast("out_w", lin_out.weight, torch.bfloat16)
            wg16, wo16 = gated.weight_bf16(), wo.weight_bf16()
            self.keep += [w_in, w_out, wg16, wo16]
            p = self.arrays[0][i]
            p.in_w, p.out_w, p.w_gated, p.w_out = w_in.data_ptr(), w_out.data_ptr(), wg16.data_ptr(), wo16.data_ptr()
            (p.in_b, p.out_b, p.short_w, p.short_b, p.wo_b, p.ln_gamma, p.ln_beta) = [t.data_ptr() for t in in_place]
            p.residual = 1 if at.residual_long_conv else 0
            value(at, "bidirectional")
            sizes = (d, I, nb, float(value(ln, "eps")))
            if i == 0:
                f0 = at.filter_fn
                self.d, self.I, self.nb, self.eps = sizes
                self.w_mod, self.shift = float(f0.w_mod), float(f0.modulation.shift)
                if ops.glu_stream_supported(self.d, self.I, self.nb):
                    self.arrays[1] = (LayerParams * n)()
                if ops.mlp_fused_supported(self.d, self.I, self.nb):
                    self.arrays[2] = (LayerParams * n)()
            elif sizes != (self.d, self.I, self.nb, self.eps):
                raise ValueError("layers that differ")
            if self.arrays[1] is not None:
                self.arrays[1][i] = p
                self.keep.append(mlp.packed_glu(wg16))
                self.arrays[1][i].glu_packed = self.keep[-1].data_ptr()
            if self.arrays[2] is not None:
                self.arrays[2][i] = p
                self.keep.append(mlp.packed_mlp(wg16, wo16))
                self.arrays[2][i].mlp_packed = self.keep[-1].data_ptr()
        self.table = ops.FilterTable.of_rows(rows, skips, len(rows) // n, L, self.d, f0.order, f0.emb_dim)
        self.checker = slots.checker()
        self.device = self.table.table.device
        ready = torch.cuda.Event()
        ready.record()
        self._use = ops.StreamUse(self.keep, ready)
        self.L = L
        self.spec_bytes = lib.m2_filter_spectrum_bytes(self.d, L)
        self.filter_ws = lib.m2_mixer_filters_workspace_bytes(n, self.table.fpm, L, self.d, self.table.order)
        self.filter_ws_layer = max(1, lib.m2_mixer_filters_workspace_bytes(1, self.table.fpm, L, self.d, self.table.order))

    def use_on_current_stream(self) -> None:
        self.table.use_on_current_stream()
        self._use.use_on_current_stream()

    def route(self, mlp, M: int) -> Optional[int]:
        """Which of `arrays` serves M rows."""
        fused, few = mlp.mlp_route(M)
        which = 2 if fused else 1 if not few and self.arrays[1] is not None else 0
        return which if self.arrays[which] is not None else None

    def current(self, encoder) -> bool:
        return self.layers == len(encoder._modules["layer"]._modules) and self.checker.unchanged()

    def __reduce__(self):                    # a plan belongs to its modules: copies and pickles of them make their own
        return type(None), ()

    def run(self, which: int, B: int, all_layers: bool, h16: Optional[torch.Tensor], hT: Optional[torch.Tensor],
            part: Optional[EmbedPart] = None, ids=None, tt=None, pos=None):
        """Enqueues the stack on the current stream; input either as h16 / hT or as token ids for the embeddings (`part`)."""
        n, L, d = self.layers, self.L, self.d
        M = B * L
        dev = ids.device if ids is not None else h16.device
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        self.use_on_current_stream()
        up = lambda v: (v + 255) & ~255      # noqa: E731
        o_spec = up(self.filter_ws)
        o_act = o_spec + up(n * self.spec_bytes)
        o_in = o_act + up(lib.m2_encoder_layers_workspace_bytes(M, d, self.I))
        ws = torch.empty(o_in + (up(2 * M * d) + 4 * M * d if ids is not None else 0), dtype=torch.uint8, device=dev)
        base = ws.data_ptr()
        outs = [torch.empty(M, d, dtype=torch.float32, device=dev) for _ in range(n if all_layers else 1)]
        ptrs = (ctypes.c_void_p * n)()
        for i, o in enumerate(outs):
            ptrs[n - len(outs) + i] = o.data_ptr()
        t = self.table
        check(lib.m2_mixer_filters_fwd(t.table.data_ptr(), t.skip.data_ptr(), n, t.fpm, L, d, t.order, t.emb_dim, self.w_mod, self.shift,
                                       base, base + o_spec, stream))
        if ids is not None:
            p16, pT = base + o_in, base + o_in + up(2 * M * d)
            check(lib.m2_embed_layernorm_fwd(ids.data_ptr(), None if tt is None else tt.data_ptr(), None if pos is None else pos.data_ptr(),
                                             *part.args, None, p16, pT, part.bad_index, B, L, d, stream))
        else:
            p16, pT = h16.data_ptr(), hT.data_ptr()
        check(lib.m2_encoder_layers_fwd(self.arrays[which], n, base + o_spec, p16, pT, ptrs, base + o_act, B, L, d, self.I, self.nb, self.eps, stream))
        return outs


def stack_plan(encoder, B: int, L: int, device: torch.device):
    """(the plan for L, made or re-used, and which of its arrays serves B L rows), or None where the Python schedule serves."""
    if _param_check is None or not encoder.native_schedule or not encoder.batch_filters or encoder.overlap_filters not in (None, False):
        return None
    M = B * L
    for lay in encoder._modules["layer"]._modules.values():
        if type(lay) is not _encoder.BertLayer:
            return None
        at, mlp = lay._modules.get("attention"), lay._modules.get("mlp")
        # classes of a caller's own run their own methods
        if type(at) is not MonarchMixerSequenceMixing or type(mlp) is not _encoder.BertGatedLinearUnitMLP:
            return None
        if (at.cache_filters or at.hyena_training_additions or mlp.fuse_wo_layernorm or not mlp.fuse_mlp or not mlp.bf16_presum
                or not mlp.stream_glu):
            return None
    d = at.d_model
    w = at.in_linear.weight
    if w.dtype != torch.float32 or not w.is_cuda:
        return None
    if not ops.own_to_channels(M, d) or not ops.own_from_channels(M, d):
        return None
    plan = encoder._native_plans.get(L)
    if plan is None or not plan.current(encoder):
        if torch.cuda.is_current_stream_capturing():
            return None                              # the filter table is copied from the host: not inside a capture
        groups = encoder._batched_filter_groups(L)   # the same rule: layers alike, spectra small enough, ...
        if groups is None or len(groups) != 1:
            return None
        try:
            plan = StackPlan(encoder, L)
        except ValueError:
            return None
        # What changed for one length changed for others: none of them keeps copies of replaced weights.  (At most one plan for
        # each of the nine lengths.)
        for other, p in list(encoder._native_plans.items()):
            if p is None or not p.current(encoder):
                encoder._native_plans.pop(other, None)
        encoder._native_plans[L] = plan
    elif (plan.layers * plan.spec_bytes > encoder.UPFRONT_MAX_BYTES                     # (limits that were lowered since)
          or encoder.FILTER_WORKSPACE_BYTES // plan.filter_ws_layer < plan.layers):
        return None
    which = plan.route(mlp, M)
    return None if which is None or plan.device != device else (plan, which)
