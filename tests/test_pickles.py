"""Modules pickled whole by earlier versions load."""
import pickle

import m2_amd


def _encoder():
    cfg = m2_amd.m2_bert_80m(128)
    cfg.num_hidden_layers = 1
    return m2_amd.BertEncoder(cfg)


def test_an_encoder_from_before_there_were_plans():
    enc = _encoder()
    for key in ("native_schedule", "_native_plans"):
        del enc.__dict__[key]
    got = pickle.loads(pickle.dumps(enc))
    assert got.native_schedule is True and got._native_plans == {}


def test_modules_from_when_the_parts_of_a_weight_were_kept():
    enc = _encoder()
    at, mlp = enc.layer[0].attention, enc.layer[0].mlp

    class Parts:
        def __reduce__(self):
            return m2_amd.ops.WeightParts, ()

    at._in_parts, at._out_parts, mlp.wo._parts, mlp.gated_layers._parts = Parts(), Parts(), Parts(), Parts()
    data = pickle.dumps(enc)
    assert b"WeightParts" in data
    got = pickle.loads(data)
    assert got.layer[0].attention._in_parts is None
