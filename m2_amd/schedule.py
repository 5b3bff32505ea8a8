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
        if found is None:
            self.values.append((mod._modules, key))
            raise ValueError(f"no module {key}")
        self.modules.append((mod._modules, key))
        if kind is not None and type(found) is not kind:
            raise ValueError(f"{key} is not the module it was built as")
        return found

    def tensor(self, mod, key, how=_IN_PLACE, shape=None):
        where = mod._parameters if key in mod._parameters else mod._buffers
        t = where.get(key)
        if t is None:                                  # absent, or computed (a parametrisation, weight_norm, pruning)
            self.values += [(mod._parameters, key), (mod._buffers, key)]
            raise ValueError(f"{key} is not a plain parameter")
        self.tensors.append((where, key, how))
        if not (t.is_cuda and t.dtype == torch.float32 and t.is_contiguous()):
            raise ValueError("parameters that are not plain fp32")
        if shape is not None and t.shape != shape:      # the kernels take sizes, not shapes: never read beyond a tensor
            raise ValueError(f"{key} of shape {tuple(t.shape)} where {shape} is expected")
        return t

    def value(self, obj, key):
        self.values.append((obj.__dict__, key))
        if key not in obj.__dict__:
            raise ValueError(f"no plain attribute {key}")
        return obj.__dict__[key]

    def option(self, obj, key):
        """An attribute of the object, or of its class where the object has none of its own."""
        self.values.append((obj.__dict__, key))
        return getattr(obj, key)

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


# (options of the MLP that the native schedule has a path for)
_MLP_OPTIONS = {"fuse_wo_layernorm": False, "fuse_mlp": True, "bf16_presum": True, "stream_glu": True}


def _class_options() -> tuple:
    return tuple(bool(getattr(_encoder.BertGatedLinearUnitMLP, key)) for key in _MLP_OPTIONS)


class NoPlan:
    """That an encoder as it is has no plan: what was looked at before that was clear, so as not to look at it again each time."""

    usable, keep = False, ()

    def __init__(self, encoder, slots: _Slots):
        self.layers = len(encoder._modules["layer"]._modules)
        self.class_options = _class_options()
        self.checker = slots.checker()

    def current(self, encoder) -> bool:
        return (self.layers == len(encoder._modules["layer"]._modules) and self.class_options == _class_options()
                and self.checker.unchanged())

    def __reduce__(self):                    # a plan belongs to its modules: copies and pickles of them make their own
        return type(None), ()


class StackPlan(NoPlan):
    """Device pointers of an encoder's layers for one length, for every row count.  The packed weights of a route come with its first
    use outside a stream capture; a capture that wants them earlier takes the Python schedule, and the table from here."""

    usable = True

    def __init__(self, encoder, L: int, slots: _Slots):
        child, tensor, value = slots.child, slots.tensor, slots.value
        stack = encoder._modules["layer"]
        n = len(stack._modules)
        plain = (LayerParams * n)()
        self.keep: List[torch.Tensor] = []
        self.mlps = []
        rows, skips = [], []
        for i, key in enumerate(stack._modules):
            lay = child(stack, key, _encoder.BertLayer)
            # classes of a caller's own run their own methods
            at, mlp = child(lay, "attention", MonarchMixerSequenceMixing), child(lay, "mlp", _encoder.BertGatedLinearUnitMLP)
            if (slots.option(at, "cache_filters") or slots.option(at, "hyena_training_additions")
                    or any(bool(slots.option(mlp, k)) is not v for k, v in _MLP_OPTIONS.items())):
                raise ValueError("options of the Python schedule")
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
            p = plain[i]
            p.in_w, p.out_w, p.w_gated, p.w_out = w_in.data_ptr(), w_out.data_ptr(), wg16.data_ptr(), wo16.data_ptr()
            (p.in_b, p.out_b, p.short_w, p.short_b, p.wo_b, p.ln_gamma, p.ln_beta) = [t.data_ptr() for t in in_place]
            p.residual = 1 if at.residual_long_conv else 0
            value(at, "bidirectional")
            sizes = (d, I, nb, float(value(ln, "eps")))
            if i == 0:
                f0 = at.filter_fn
                self.d, self.I, self.nb, self.eps = sizes
                self.w_mod, self.shift = float(f0.w_mod), float(f0.modulation.shift)
                self.supported = (True, ops.glu_stream_supported(self.d, self.I, self.nb), ops.mlp_fused_supported(self.d, self.I, self.nb))
            elif sizes != (self.d, self.I, self.nb, self.eps):
                raise ValueError("layers that differ")
            self.mlps.append(mlp)
        self.table = ops.FilterTable.of_rows(rows, skips, len(rows) // n, L, self.d, f0.order, f0.emb_dim)
        super().__init__(encoder, slots)
        self.device = self.table.table.device
        # the layers' pointers with the memory they need: plain, with the streaming product's packed weights, with the one-kernel MLP's
        self.routes: list = [(plain, self._made_here(self.keep)), None, None]
        self.L = L
        self.spec_bytes = lib.m2_filter_spectrum_bytes(self.d, L)
        self.filter_ws = lib.m2_mixer_filters_workspace_bytes(n, self.table.fpm, L, self.d, self.table.order)
        self.taps_ws = lib.m2_mixer_taps_workspace_bytes(n, self.table.fpm, L, self.d, self.table.order)
        self.filter_ws_layer = max(1, lib.m2_mixer_filters_workspace_bytes(1, self.table.fpm, L, self.d, self.table.order))

    @staticmethod
    def _made_here(tensors) -> ops.StreamUse:
        ready = torch.cuda.Event()
        ready.record()
        return ops.StreamUse(tensors, ready)

    def use_on(self, handle: int) -> None:
        self.table.use_on(handle)
        for route in self.routes:
            if route is not None:
                route[1].use_on(handle)

    def route(self, M: int):
        """The one of `routes` that serves M rows, or None where it would have to be made during a stream capture."""
        fused, few = self.mlps[-1].mlp_route(M)
        which = 2 if fused else 1 if not few and self.supported[1] else 0
        found = self.routes[which]
        if found is None and self.supported[which] and not torch.cuda.is_current_stream_capturing():
            packs, array = [], (LayerParams * self.layers)()
            for i, mlp in enumerate(self.mlps):
                array[i] = self.routes[0][0][i]
                wg16, wo16 = self.keep[4 * i + 2], self.keep[4 * i + 3]
                packs.append(mlp.packed_glu(wg16) if which == 1 else mlp.packed_mlp(wg16, wo16))
                setattr(array[i], "glu_packed" if which == 1 else "mlp_packed", packs[-1].data_ptr())
            self.routes[which] = found = (array, self._made_here(packs))
        return found

    def run(self, route, B: int, all_layers: bool, h16: Optional[torch.Tensor], hT: Optional[torch.Tensor],
            part: Optional[EmbedPart] = None, ids=None, tt=None, pos=None):
        """Enqueues the stack on the current stream; input either as h16 / hT or as token ids for the embeddings (`part`)."""
        n, L, d = self.layers, self.L, self.d
        M = B * L
        dev = ids.device if ids is not None else h16.device
        current = ops._stream()
        t = self.table
        t.use_on(current)
        self.routes[0][1].use_on(current)
        route[1].use_on(current)
        stream = ctypes.c_void_p(current)
        up = lambda v: (v + 255) & ~255      # noqa: E731
        taps = ops.taps_pay(B, L, torch.bfloat16)
        o_spec = up(self.taps_ws if taps else self.filter_ws)
        o_act = o_spec + up(n * (8 * t.fpm * d * L if taps else self.spec_bytes))
        o_in = o_act + up(lib.m2_encoder_layers_workspace_bytes(M, d, self.I))
        ws = torch.empty(o_in + (up(2 * M * d) + 4 * M * d if ids is not None else 0), dtype=torch.uint8, device=dev)
        base = ws.data_ptr()
        outs = [torch.empty(M, d, dtype=torch.float32, device=dev) for _ in range(n if all_layers else 1)]
        ptrs = (ctypes.c_void_p * n)()
        for i, o in enumerate(outs):
            ptrs[n - len(outs) + i] = o.data_ptr()
        if taps:
            check(lib.m2_mixer_taps_fwd(t.table.data_ptr(), n, t.fpm, L, d, t.order, t.emb_dim, self.w_mod, self.shift, base, base + o_spec, stream))
        else:
            check(lib.m2_mixer_filters_fwd(t.table.data_ptr(), t.skip.data_ptr(), n, t.fpm, L, d, t.order, t.emb_dim, self.w_mod, self.shift,
                                           base, base + o_spec, stream))
        if ids is not None:
            p16, pT = base + o_in, base + o_in + up(2 * M * d)
            check(lib.m2_embed_layernorm_fwd(ids.data_ptr(), None if tt is None else tt.data_ptr(), None if pos is None else pos.data_ptr(),
                                             *part.args, None, p16, pT, part.bad_index, B, L, d, stream))
        else:
            p16, pT = h16.data_ptr(), hT.data_ptr()
        if taps:
            check(lib.m2_encoder_layers_taps_fwd(route[0], n, base + o_spec, t.skip.data_ptr(), t.fpm, p16, pT, ptrs, base + o_act, B, L, d,
                                                 self.I, self.nb, self.eps, stream))
        else:
            check(lib.m2_encoder_layers_fwd(route[0], n, base + o_spec, p16, pT, ptrs, base + o_act, B, L, d, self.I, self.nb, self.eps, stream))
        return outs


def stack_plan(encoder, B: int, L: int, device: torch.device):
    """(the plan for L, made or re-used, and the route of it that serves B L rows), or None where the Python schedule serves."""
    if _param_check is None or not encoder.native_schedule or not encoder.batch_filters or encoder.overlap_filters not in (None, False):
        return None
    M = B * L
    plan = encoder._native_plans.get(L)
    if plan is not None and plan.current(encoder):
        if not plan.usable:
            return None
        d = plan.d
    else:
        plan, first = None, next(iter(encoder._modules["layer"]._modules.values()), None)
        if type(first) is not _encoder.BertLayer or type(first.attention) is not MonarchMixerSequenceMixing:
            return None
        d = first.attention.d_model
    if not ops.native_rows(M, d):
        return None
    if plan is None:
        if torch.cuda.is_current_stream_capturing():
            return None                              # the filter table is copied from the host: not inside a capture
        groups = encoder._batched_filter_groups(L)   # the same rule: layers alike, spectra small enough, ...
        if groups is None or len(groups) != 1:
            return None
        slots = _Slots()
        slots.modules.append((encoder._modules, "layer"))
        try:
            plan = StackPlan(encoder, L, slots)
        except ValueError:
            try:
                plan = NoPlan(encoder, slots)
            except (KeyError, ValueError):
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
    if not plan.usable or plan.device != device:
        return None
    route = plan.route(M)
    return None if route is None else (plan, route)
