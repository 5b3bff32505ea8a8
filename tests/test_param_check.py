"""The check behind the plans of the native schedule (m2_amd/csrc/param_check.cpp), on CPU tensors: what a plan depends on is
recognised as changed whichever way it was changed."""
import os

import numpy as np
import pytest
import torch

from m2_amd import _param_check


def _checker(mod, key="weight", version=True):
    return _param_check.Checker([], [(mod._parameters, key, version)], [])


def test_another_tensor_at_the_same_address_is_another():
    """As when the allocator gives the address of a freed weight out again: same address, same version, another storage."""
    memory = np.zeros((8, 8), dtype=np.float32)
    lin = torch.nn.Linear(8, 8)
    lin.weight = torch.nn.Parameter(torch.from_numpy(memory))
    check, address, version = _checker(lin), lin.weight.data_ptr(), lin.weight._version
    assert check.unchanged()
    lin.weight = None
    assert not check.unchanged()
    lin.weight = torch.nn.Parameter(torch.from_numpy(memory))
    assert (lin.weight.data_ptr(), lin.weight._version) == (address, version)
    assert not check.unchanged()


def test_a_view_of_the_recorded_storage_is_the_recorded_tensor():
    lin = torch.nn.Linear(8, 8)
    check = _checker(lin)
    lin.weight = torch.nn.Parameter(lin.weight.detach())
    assert check.unchanged()


def test_data_assigned_twice_is_noticed():
    lin = torch.nn.Linear(8, 8)
    check, version = _checker(lin), lin.weight._version
    lin.weight.data = lin.weight.data * 2
    assert lin.weight._version == version and not check.unchanged()
    check = _checker(lin)
    lin.weight.data = lin.weight.data * 2
    lin.weight.data = lin.weight.data * 2
    assert not check.unchanged()


def test_versions_count_where_a_copy_was_made():
    lin = torch.nn.Linear(8, 8)
    copied, in_place = _checker(lin), _checker(lin, version=False)
    with torch.no_grad():
        lin.weight.add_(1)
    assert not copied.unchanged() and in_place.unchanged()


@pytest.mark.parametrize("value,others", [(1e-12, (1e-5, 1, None)), (3, (4, 3.0, True)), (None, (0, 0.0)), (True, (False, 1)),
                                          (float(2.5), (2.25,)), ("a", ("b", 1))])
def test_plain_values_are_compared(value, others):
    lin = torch.nn.LayerNorm(8)
    lin.eps = value
    check = _param_check.Checker([], [], [(lin.__dict__, "eps")])
    assert check.unchanged()
    for other in others:
        lin.eps = other
        assert not check.unchanged(), other
    lin.eps = float(str(value)) if isinstance(value, float) else value          # an equal number, another object
    assert check.unchanged()
    del lin.eps
    assert not check.unchanged()
    absent = _param_check.Checker([], [], [(lin.__dict__, "eps")])          # and the absence of one
    assert absent.unchanged()
    lin.eps = None
    assert not absent.unchanged()


def test_a_part_of_the_recorded_tensor_is_another():
    """Same storage, same address, fewer rows, other strides or another type."""
    for change in (lambda w: w[:4], lambda w: w.t(), lambda w: w.view(64), lambda w: w.view(torch.int32)):
        lin = torch.nn.Linear(8, 8)
        check, address = _checker(lin, version=False), lin.weight.data_ptr()
        new = change(lin.weight.detach())
        lin.weight = torch.nn.Parameter(new, requires_grad=new.is_floating_point())
        assert lin.weight.data_ptr() == address and not check.unchanged()


def test_tensors_without_memory_are_errors_and_changes():
    """Sparse and fake tensors have no address: a change before a plan is used, an error when one is made, never an exception out of
    the C entry."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode():
        fake = torch.empty(8, 8)
    lin = torch.nn.Linear(8, 8)
    check = _checker(lin)
    where = lin._parameters
    was, where["weight"] = where["weight"], fake
    assert not check.unchanged()
    for other in (None, 3, torch.ones(8, 8).to_sparse(), torch.ones(8, 8).to_sparse_csr(), torch.ones(8, 8).to_mkldnn()):
        where["weight"] = other
        assert not check.unchanged()
        with pytest.raises((KeyError, ValueError)):
            _checker(lin)
    where["weight"] = was
    assert check.unchanged()


def test_another_module_or_another_class_in_its_place():
    seq = torch.nn.Sequential(torch.nn.Linear(8, 8))
    check = _param_check.Checker([(seq._modules, "0")], [], [])
    assert check.unchanged()
    seq[0].__class__ = type("Other", (torch.nn.Linear,), {})
    assert not check.unchanged()
    seq[0].__class__ = torch.nn.Linear
    assert check.unchanged()
    seq[0] = torch.nn.Linear(8, 8)
    assert not check.unchanged()


def test_a_cycle_through_the_check_is_collected():
    import gc
    import weakref
    for slots in (lambda m: ([(m._modules, "0")], [], []), lambda m: ([], [(m[0]._parameters, "weight", True)], []),
                  lambda m: ([], [], [(m.__dict__, "training")])):
        seq = torch.nn.Sequential(torch.nn.Linear(8, 8))
        seq[0].__dict__["_parameters"]["weight"].owner = seq       # and back
        seq[0].owner_dict = {"owner": seq}
        seq.check = _param_check.Checker(*slots(seq))
        gone = weakref.ref(seq)
        del seq
        gc.collect()
        assert gone() is None


def test_the_package_works_without_the_extension():
    """Only plans need it: a package without it (or with one that does not fit torch) imports with a warning and makes no plans."""
    import subprocess
    import sys
    code = ("import sys, warnings\n"
            "sys.modules['m2_amd._param_check'] = None\n"
            "with warnings.catch_warnings(record=True) as seen:\n"
            "    warnings.simplefilter('always')\n"
            "    import m2_amd\n"
            "assert any('_param_check' in str(w.message) for w in seen)\n"
            "from m2_amd import schedule\n"
            "assert schedule._param_check is None\n"
            "assert schedule.stack_plan(m2_amd.BertEncoder(m2_amd.m2_bert_80m(128)), 1, 128, None) is None\n")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", code], cwd=root, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
