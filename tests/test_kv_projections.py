"""Which q/k/v projections the KV recalibration finds, against ``named_modules()``
of the same model: shared and aliased modules, missing children, modules with a
traversal of their own, and models that only delegate to a module."""

from __future__ import annotations

import weakref

import pytest
import torch.nn as nn

from lumenrl_amd.quantization.fp8_kv_cache import _projections


def lin():
    return nn.Linear(4, 4, bias=False, device="meta")


class Attention(nn.Module):
    def __init__(self, **children):
        super().__init__()
        for name in ("q_proj", "k_proj", "v_proj", "o_proj"):
            self.add_module(name, children.get(name, lin()))


class Renames(Attention):
    """Its projections go by other names, and one module that is no child is among them."""

    def named_modules(self, memo=None, prefix="", remove_duplicate=True):
        yield prefix, self
        yield prefix + ".q_proj", self.o_proj
        yield prefix + ".other", self.q_proj


class Delegates:
    def __init__(self, model):
        self.model = model

    def __getattr__(self, name):
        return getattr(self.model, name)


def plain():
    return nn.Sequential(Attention(), nn.ModuleDict({"attn": Attention(), "k_proj": lin()}), lin())


def shared():
    one = lin()
    return nn.Sequential(nn.ModuleDict({"dense": one, "q_proj": one}), Attention(q_proj=one), nn.ModuleList([Attention()] * 2))


def missing():
    return nn.Sequential(Attention(k_proj=None, v_proj=nn.Identity()), Attention())


def own_traversal_below():
    return nn.Sequential(Attention(), Renames(), Attention())


def own_traversal_of_an_instance():
    model = plain()
    model[1].attn.named_modules = lambda *a, **k: iter([("x.v_proj", model[2])])
    return model


def projection_as_model():
    return lin()


MODELS = [plain, shared, missing, own_traversal_below, own_traversal_of_an_instance, projection_as_model, Renames]
WRAPS = [lambda m: m, weakref.proxy, Delegates]


@pytest.mark.parametrize("wrap", WRAPS, ids=["itself", "proxy", "delegate"])
@pytest.mark.parametrize("make", MODELS)
def test_projections_are_those_of_named_modules(make, wrap):
    model = make()
    seen = wrap(model)
    want = [(name.rpartition(".")[2], module) for name, module in seen.named_modules()
            if isinstance(module, nn.Linear) and name.rpartition(".")[2] in ("q_proj", "k_proj", "v_proj")]
    got = _projections(seen)
    assert [n for n, _ in got] == [n for n, _ in want]
    assert all(a is b for (_, a), (_, b) in zip(got, want))
