"""The tensors of an implicit filter's MLPs, on the CPU: those of the modules as they are at the time of the call."""
import torch


def test_mlp_tensors_are_those_of_the_modules():
    import m2_amd
    fn = m2_amd.HyenaFilter(64, emb_dim=5, order=128, seq_len=32, bidirectional=True)
    seq = fn.implicit_filter

    def same(s):
        want = [s[0].weight, s[0].bias, s[2].weight, s[2].bias, s[4].weight, s[4].bias, s[6].weight]
        got = fn._mlp_tensors(s)
        return len(got) == len(want) and all(a is b for a, b in zip(got, want))

    assert same(seq) and same(fn.implicit_filter_rev)
    seq[2] = torch.nn.Linear(128, 128)
    assert same(seq)
    seq[6].weight = torch.nn.Parameter(torch.zeros(64, 128))
    assert same(seq)
    seq.append(torch.nn.Identity())
    assert same(seq) and same(torch.nn.ModuleList(seq))
    p = fn.kernel_params("both")
    assert all(a.data_ptr() == b.data_ptr() for a, b in zip(p["fwd"] + p["rev"], fn._mlp_tensors(seq) + fn._mlp_tensors(fn.implicit_filter_rev)))
