"""The packed-weight cache (PersistentLSTM.packed_blob) holds what the module's attributes hold: a weight that is
computed from parameters of other names (pruning, norms, parametrizations) is packed anew when it changes.  CPU
only: the packer is a stub that keeps copies of what it is given."""
from __future__ import annotations

import pytest
import torch
import torch.nn as nn
from torch.nn.utils import parametrize, prune, spectral_norm, weight_norm

from persistent_lstm_hip_amd import model as model_module
from persistent_lstm_hip_amd.model import PersistentLSTM

NAMES = ("weight_ih", "weight_hh", "bias_ih", "bias_hh")


class _Packer:
    def __init__(self):
        self.calls = 0

    def pack(self, w_ih, w_hh, b_ih, b_hh, lin_w, lin_b):
        self.calls += 1
        return [[t.detach().clone() for t in ts] for ts in (w_ih, w_hh, b_ih, b_hh)]


class _Scale(nn.Module):
    def __init__(self, factor):
        super().__init__()
        self.register_buffer("factor", torch.tensor(factor))

    def forward(self, w):
        return w * self.factor


@pytest.fixture
def packer(monkeypatch):
    p = _Packer()
    monkeypatch.setattr(model_module, "require_extension", lambda: p)
    return p


def _module(layers=2):
    torch.manual_seed(3)
    return PersistentLSTM.from_native_module(nn.LSTM(5, 8, layers, batch_first=True)).eval()


def _forward(m):
    """The blob of a forward: its pre-hooks (which recompute pruned and normed weights), then the pack."""
    for hook in list(m._forward_pre_hooks.values()):
        hook(m, ())
    return m.packed_blob(torch.device("cpu"))


def _check(m, blob):
    for kind, packed in zip(NAMES, blob):
        for l, t in enumerate(packed):
            assert torch.equal(t, getattr(m, f"{kind}_l{l}")), f"{kind}_l{l} is stale"


def test_unchanged_parameters_are_packed_once_and_changes_again(packer):
    m = _module()
    blob = _forward(m)
    assert _forward(m) is blob and packer.calls == 1
    for name in ("weight_hh_l1", "bias_ih_l0"):
        with torch.no_grad():
            getattr(m, name).mul_(2.0)
        _check(m, _forward(m))
    m.weight_ih_l0 = nn.Parameter(torch.zeros_like(m.weight_ih_l0))
    _check(m, _forward(m))
    assert packer.calls == 4


@pytest.mark.parametrize("name", ["weight_ih_l0", "weight_hh_l1", "bias_hh_l1"])
def test_pruning_step_by_step(packer, name):
    """Each pass keeps the number of parameters, the second one also the parameter objects."""
    m = _module()
    _check(m, _forward(m))
    for _ in range(2):
        prune.random_unstructured(m, name, amount=0.4)
        _check(m, _forward(m))
    getattr(m, f"{name}_mask").zero_()  # a mask written in place
    _check(m, _forward(m))
    prune.remove(m, name)
    _check(m, _forward(m))


@pytest.mark.parametrize("norm", [spectral_norm, weight_norm])
def test_normed_weight(packer, norm):
    m = _module()
    _check(m, _forward(m))
    norm(m, "weight_hh_l0")
    m.train()  # a spectral norm's power iteration moves the weight at every forward
    for _ in range(2):
        _check(m, _forward(m))


def test_parametrized_weight_beside_an_added_parameter(packer):
    """A parametrization takes its parameter out of the module; another registered one makes up the number."""
    m = _module()
    _check(m, _forward(m))
    m.register_parameter("temperature", nn.Parameter(torch.ones(())))
    parametrize.register_parametrization(m, "weight_hh_l0", _Scale(0.5))
    _check(m, _forward(m))
    m.parametrizations.weight_hh_l0[0].factor.fill_(0.25)
    _check(m, _forward(m))
