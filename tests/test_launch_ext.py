"""The C function behind the call of a loaded kernel: what it takes, and what it hands back to the
checks in Python."""

import ctypes
import os
import sys

import pytest
import torch

from deca_amd.driver.build_lib import EXT_PATH, LIB_PATH, build_extension, build_library
from deca_amd.driver.driver import LaunchPlan


@pytest.fixture(scope="module")
def launch():
    if not os.path.exists(LIB_PATH):
        build_library()
    if not os.path.exists(EXT_PATH):
        build_extension()
    from deca_amd._launch import launch

    return launch


def test_arguments_it_cannot_take_launch_nothing(launch):
    """(a plan without a kernel: a launch would give hipErrorInvalidValue = 1)"""
    plan = LaunchPlan(None, (1, 1, 1), (64, 1, 1), 0, 2)
    at = ctypes.addressof(plan)
    t = torch.zeros(4, 4)

    class Wrapped(torch.Tensor):
        pass

    for args in ((t, t), (t,), (t, t, t), (t.t()[:2], t), (1, 2), (None, t), (t.as_subclass(Wrapped), t)):
        assert launch(at, *args) == -1
    with pytest.raises(TypeError):
        launch()
    with pytest.raises(ValueError):
        launch(0, t, t)
    with pytest.raises(TypeError):
        launch("plan", t, t)


def test_an_extension_that_cannot_serve_is_left_aside(launch, monkeypatch):
    """Not built, or built for another torch: `None` and a warning, no error."""
    from deca_amd.driver import driver

    load = driver._load_launch.__wrapped__
    assert load() is launch
    with monkeypatch.context() as m:
        m.setattr(torch, "__version__", "0.1")
        with pytest.warns(RuntimeWarning, match="built for torch"):
            assert load() is None
    with monkeypatch.context() as m:
        m.delattr(sys.modules["deca_amd"], "_launch", raising=False)
        m.setitem(sys.modules, "deca_amd._launch", None)
        with pytest.warns(RuntimeWarning, match="take a few microseconds more"):
            assert load() is None


@pytest.mark.gpu
def test_a_kernel_is_called_without_the_extension_too(monkeypatch):
    from deca_amd.driver import driver
    from deca_amd.kernels.rowwise_hip import RowConfig, build_rowwise, make_rowwise

    monkeypatch.setattr(driver, "_load_launch", lambda: None)
    kern = build_rowwise(make_rowwise("softmax", 512, 4096, "float16", RowConfig(128, 1, 8)))
    assert not kern._plan_address
    x = torch.randn(512, 4096, device="cuda").half()
    y = torch.zeros_like(x)
    kern(x, y)
    assert (y.float() - torch.softmax(x.float(), -1)).abs().max().item() <= 2e-3
    with pytest.raises(ValueError, match="contiguous device tensors"):
        kern(x.cpu(), y)


@pytest.mark.gpu
def test_a_call_says_what_it_cannot_take():
    from deca_amd.kernels.rowwise_hip import RowConfig, build_rowwise, make_rowwise

    kern = build_rowwise(make_rowwise("softmax", 512, 4096, "float16", RowConfig(128, 1, 8)))
    assert kern._plan_address
    x = torch.randn(512, 4096, device="cuda").half()
    y = torch.zeros_like(x)
    with pytest.raises(ValueError, match="2 tensors"):
        kern(x)
    with pytest.raises(ValueError, match="contiguous device tensors"):
        kern(x.cpu(), y)
    with pytest.raises(ValueError, match="contiguous device tensors"):
        kern(x, torch.zeros(4096, 512, device="cuda", dtype=torch.float16).t())
    with pytest.raises(AttributeError):
        kern(x, 0)
    torch.cuda.synchronize()
    assert y.abs().max().item() == 0
    kern(x, torch.nn.Parameter(y, requires_grad=False))  # the parameter shares y's memory
    assert (y.float() - torch.softmax(x.float(), -1)).abs().max().item() <= 2e-3
