"""FFITrainStep.step and step_bce call the methods that a subclass or an attribute replaces."""
import pytest
import torch

from haste_amd import step as step_mod
from haste_amd.step import FFITrainStep


def bare(cls):
    """An instance without buffers on a device."""
    st = object.__new__(cls)
    st.grad_dtype, st.ldo, st.loss_buf = torch.float32, 64, torch.zeros(())
    st._joins = {(64, 0): 1}
    st.logits_buf = torch.zeros(4, 64, dtype=torch.bfloat16)
    st.dY_buf = torch.zeros(4, 64, dtype=torch.bfloat16)
    return st


def recorder(name, calls):
    return lambda self, *a, **k: calls.append(name)


@pytest.mark.parametrize("how", ["subclass", "attribute", "patch"])
@pytest.mark.parametrize("method", ["step", "step_bce"])
def test_replaced_methods_are_called(monkeypatch, method, how):
    calls = []
    monkeypatch.setattr(step_mod._lib, "call", lambda name, *a: calls.append(name))
    names = ["forward" if method == "step" else "forward_bce", "backward_features",
             "backward_weights_sgd"]
    cls = type("Sub", (FFITrainStep,), {n: recorder(n, calls) for n in names}) \
        if how == "subclass" else FFITrainStep
    st = bare(cls)
    for n in names:
        if how == "attribute":
            setattr(st, n, lambda *a, _n=n, **k: calls.append(_n))
        elif how == "patch":
            monkeypatch.setattr(FFITrainStep, n, recorder(n, calls))
    if method == "step":
        st.step(torch.zeros(4, 8), torch.zeros(4, 64, dtype=torch.bfloat16), 64)
    else:
        st.step_bce(torch.zeros(4, 8), torch.zeros(3, 2, dtype=torch.int32))
    assert calls == names


def test_the_class_itself_replaces_none():
    st = object.__new__(FFITrainStep)
    assert not st._replaced("forward", "forward_bce", "backward_weights_sgd")
    st.forward = lambda x: None
    assert st._replaced("forward") and not st._replaced("forward_bce")
