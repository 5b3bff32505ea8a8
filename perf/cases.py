"""Work that a user of m2_amd has it do, as cases that can be prepared, run and timed.

A case is a dict of plain values:

    entry    "model"    BertModel on token ids, last hidden state and pooled output (the default call)
             "hidden"   BertEncoder on hidden states, every layer's output (what a masked-LM head is put on)
             "texts"    M2BertTextEncoder on ragged token-id lists in host memory, pooled vectors back in host memory
             "layer"    one BertLayer
             "mixer"    one MonarchMixerSequenceMixing
    width    768, 960, 1536 or 1792: the four models of the configuration helpers
    layers   how many layers
    L, B     sequence length and batch ("texts": tokens a text is padded or cut to, texts per forward)
    l_max    the length the model was built for (L unless said otherwise)
    f32      True: fp32 activations outside autocast; False: bf16 GEMMs
    graph    True: the model replays one captured HIP graph per input shape
    texts    "texts" only: how many texts
"""
from __future__ import annotations

import math

import torch

import m2_amd

HELPERS = {768: m2_amd.m2_bert_80m, 960: m2_amd.m2_bert_110m, 1536: m2_amd.m2_bert_large, 1792: m2_amd.m2_bert_341m}
LENGTHS = [128, 256, 512, 1024, 2048, 4096, 8192, 16384, 32768]


def _case(name, entry, width, layers, L, B, f32=False, graph=False, l_max=None, texts=0):
    case = {"entry": entry, "width": width, "layers": layers, "L": L, "B": B, "l_max": l_max or L, "f32": f32,
            "graph": graph, "texts": texts}
    return dict(case, name=name) if name else case


def listed():
    return [
        # one query embedded as it comes in: latency and launches
        _case("query_L128_B1", "model", 768, 12, 128, 1),
        # one mixer in fp32, the first benchmark configuration
        _case("mixer_f32_L128_B16", "mixer", 768, 1, 128, 16, f32=True),
        # one whole layer in fp32 (checking a checkpoint, or a user who wants no bf16), odd batch
        _case("layer_f32_L512_B5", "layer", 768, 1, 512, 5, f32=True),
        # sentence batches in a serving loop, the second benchmark configuration
        _case("sentences_L128_B32_graph", "model", 768, 12, 128, 32, graph=True),
        # passages of any length from the host, embedded 32 at a time with a short last batch (retrieval)
        _case("passages_512", "texts", 768, 12, 512, 32, texts=75),
        # the reference's benchmark form: hidden states in, all layers out, here with an odd batch
        _case("hidden_L1024_B31", "hidden", 768, 12, 1024, 31),
        # one document at a time
        _case("document_L4096_B1", "model", 768, 12, 4096, 1),
        # the headline workload: long documents in a batch
        _case("documents_L8192_B4_graph", "model", 768, 12, 8192, 4, graph=True),
        # the longest context, one sequence
        _case("book_L32768_B1", "model", 768, 12, 32768, 1),
        # the large model on sentence batches: the GEMM-heavy end
        _case("large_L128_B64_graph", "model", 1536, 24, 128, 64, graph=True),
        # the two other widths at the length their checkpoints are used at
        _case("width960_L2048_B16", "model", 960, 12, 2048, 16),
        _case("width1792_L2048_B5", "model", 1792, 12, 2048, 5),
    ]


def draw(rng):
    """One more case of the ranges above: any width, any supported length, any batch (odd ones included) up to the
    token counts of the largest listed cases, each option on and off."""
    entry = rng.choice(["model"] * 5 + ["hidden", "hidden", "texts", "layer", "mixer"])
    width = rng.choice([768, 768, 768, 960, 1536, 1792])
    if entry in ("layer", "mixer"):
        L = rng.choice(LENGTHS[:7])
        most, layers = (16384 if width <= 960 else 8192), 1
    elif entry == "texts":
        L = rng.choice(LENGTHS[:6])
        most, layers = 8192, (24 if width == 1536 else 12)
    else:
        L = rng.choice(LENGTHS if width == 768 else LENGTHS[:7])
        most, layers = (32768 if width == 768 else 16384 if width == 960 else 8192), (24 if width == 1536 else 12)
    B = max(1, int(round(math.exp(rng.uniform(0.0, math.log(max(1.0, most / L)))))))
    l_max = L
    if entry == "model" and L < 8192 and rng.random() < 0.25:      # a model built for longer sequences
        l_max = 2 * L
    graph = entry in ("model", "hidden") and rng.random() < 0.5
    f32 = entry in ("layer", "mixer") and rng.random() < 0.6
    texts = rng.randint(B, 3 * B) if entry == "texts" else 0
    return _case(None, entry, width, layers, L, B, f32=f32, graph=graph, l_max=l_max, texts=texts)


def _config(case):
    cfg = HELPERS[case["width"]](case["l_max"])
    cfg.num_hidden_layers = case["layers"]
    return cfg


def _fill(module, gen, l_max):
    """N(0, 0.02) weights, zero biases, unit LayerNorms: the initial values of the models.  The output projections of
    the implicit filters are scaled by 128 / l_max, which keeps the gain of the long convolutions what it is at the
    shortest model; unscaled, random taps of the same size at every length make a long-context stack amplify bf16
    rounding by 1.3x per layer, which no trained model does."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            leaf = name.rsplit(".", 1)[-1]
            if leaf in ("z", "t", "deltas", "freq"):
                continue
            if "norm" in name.lower():
                p.fill_(1.0 if leaf == "weight" else 0.0)
            elif leaf == "bias" and "filter_fn" not in name and "pooler" not in name:
                p.zero_()
            elif ".bias" in name and "implicit_filter" in name:
                p.zero_()
            else:
                p.normal_(0.0, 0.02, generator=gen)
                if "implicit_filter" in name and name.endswith(".6.weight"):
                    p.mul_(128.0 / l_max)


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    cfg = _config(case)
    B, L, entry = case["B"], case["L"], case["entry"]
    state = {"case": case, "seed": seed}
    with torch.device(dev):
        if entry == "mixer":
            module = m2_amd.MonarchMixerSequenceMixing(
                cfg.hidden_size, l_max=cfg.long_conv_l_max, bidirectional=True, hyena_w=cfg.hyena_w,
                hyena_emb_dim=cfg.hyena_emb_dim, hyena_filter_order=cfg.hyena_filter_order, residual_long_conv=True)
        elif entry == "layer":
            module = m2_amd.BertLayer(cfg)
        elif entry == "hidden":
            module = m2_amd.BertEncoder(cfg, use_hip_graph=case["graph"])
        else:
            module = m2_amd.BertModel(cfg, use_hip_graph=case["graph"])
    module = module.to(dev).eval()
    _fill(module, gen, cfg.long_conv_l_max)
    state["module"] = module
    if entry == "texts":
        host = torch.Generator().manual_seed(seed)
        lengths = torch.randint(max(1, L // 16), L + L // 8, (case["texts"],), generator=host)   # some are cut
        state["ids"] = [torch.randint(1, cfg.vocab_size, (int(n),), generator=host).tolist() for n in lengths]
        state["encoder"] = m2_amd.M2BertTextEncoder(module, max_seq_len=L)
    elif entry == "model":
        # padded batches: sequences fill between half and all of L
        ids = torch.randint(1, cfg.vocab_size, (B, L), generator=gen, device=dev)
        lengths = torch.randint(max(1, L // 2), L + 1, (B, 1), generator=gen, device=dev)
        mask = (torch.arange(L, device=dev)[None] < lengths).long()
        state["ids"], state["mask"] = ids * mask, mask
    else:
        dtype = torch.bfloat16 if entry in ("layer", "mixer") and not case["f32"] else torch.float32
        state["u"] = torch.randn(B, L, cfg.hidden_size, generator=gen, device=dev).to(dtype)
    return state


def run(state):
    entry = state["case"]["entry"]
    with torch.no_grad():
        if entry == "texts":
            return state["encoder"].encode_token_ids(state["ids"], state["case"]["B"])
        if entry == "model":
            return state["module"](state["ids"], attention_mask=state["mask"])
        if entry == "mixer":
            return state["module"](state["u"])[0]
        return state["module"](state["u"])


def work(case):
    """Bytes: parameters and inputs once, outputs once.  Flops: the matrix products, the filter MLPs and
    5 N log2 N per complex transform of N = 2L points (a forward and an inverse one per channel of a sequence, one per
    channel for the filters)."""
    cfg = _config(case)
    d, I, nb, L, n = cfg.hidden_size, cfg.intermediate_size, cfg.monarch_mlp_nblocks, case["L"], case["layers"]
    order, emb = cfg.hyena_filter_order, cfg.hyena_emb_dim
    tokens = (case["texts"] or case["B"]) * L
    forwards = -(-case["texts"] // case["B"]) if case["texts"] else 1
    act = 4 if case["f32"] or case["entry"] in ("model", "hidden", "texts") else 2

    mixer_params = 4 * d * d + 4 * (order * (emb + 2 * order + 3) + d * order) + 2 * emb * L + 20 * d
    mlp_params = 3 * d * I // nb + 3 * d
    fft = 5 * 2 * L * math.log2(2 * L)
    filters = 4 * L * 2 * (emb * order + 2 * order * order + order * d) + d * fft
    mixer = tokens * 8 * d * d + forwards * filters + (tokens // L) * d * 2 * fft
    mlp = tokens * 6 * d * I // nb
    if case["entry"] == "mixer":
        return {"bytes": 4 * mixer_params + 2 * act * tokens * d, "flops": mixer}
    params = n * (mixer_params + mlp_params)
    if case["entry"] == "layer":
        return {"bytes": 4 * params + tokens * d * (act + 4), "flops": mixer + mlp}
    flops = n * (mixer + mlp)
    if case["entry"] == "hidden":
        return {"bytes": 4 * params + 4 * tokens * d * (1 + n), "flops": flops}
    rows = min(cfg.vocab_size, tokens)                                   # table rows that are read
    out = 0 if case["entry"] == "texts" else 4 * tokens * d
    return {"bytes": 4 * (params + rows * d + L * d + d * d) + 16 * tokens + out, "flops": flops}


def tolerance(case):
    """Measured against the same path in fp64 (relative 2-norm, over the listed cases and drawn ones): fp32 4e-6 for one
    mixer or layer; bf16 GEMMs 3e-3 after one layer, 6e-3 ... 8e-3 after twelve (9e-3 at width 1792), 1.5e-2 after
    twenty-four."""
    if case["f32"]:
        return {"rel": 1.6e-5}
    return {"rel": 1e-2 if case["layers"] == 1 else 2.5e-2 if case["layers"] <= 12 else 5e-2}
