"""When a decoder's step may leave torch's operations for products of a few rows: the parts that need no device."""
import functools

import pytest
import torch
from torch import nn

from cascading_kv_cache_amd import row_products as rp
from cascading_kv_cache_amd.cascade_attention import CascadeAttention
from cascading_kv_cache_amd.decoder import PRESETS, CascadeDecoder, DecoderLayer, GatedMLP, RMSNorm
from cascading_kv_cache_amd.latency import ProjectedCascadeAttention

MAKE = {nn.Linear: lambda: nn.Linear(4, 4), RMSNorm: lambda: RMSNorm(4, 1e-5, torch.float32, "cpu"),
        GatedMLP: lambda: GatedMLP(PRESETS["tiny"], torch.float32, "cpu"),
        ProjectedCascadeAttention: lambda: ProjectedCascadeAttention(64, 2, 1, 32, dtype=torch.float32, device="cpu")}


@pytest.mark.parametrize("kind,home,name", [(nn.Linear, nn.Linear, "forward"), (RMSNorm, RMSNorm, "forward"), (GatedMLP, GatedMLP, "forward"),
                                            (ProjectedCascadeAttention, ProjectedCascadeAttention, "qkv"),
                                            (ProjectedCascadeAttention, CascadeAttention, "forward"),
                                            (ProjectedCascadeAttention, CascadeAttention, "forward_cascade"),
                                            (GatedMLP, nn.Module, "__call__"), (nn.Linear, nn.Module, "_call_impl")])
def test_methods_put_on_a_class_or_an_object_are_seen(kind, home, name, monkeypatch):
    module = MAKE[kind]()
    assert rp.plain(module, kind)
    own = getattr(home, name)

    @functools.wraps(own)
    def other(self, *args, **kw):
        return own(self, *args, **kw)

    monkeypatch.setattr(home, name, other)
    assert not rp.plain(module, kind)
    monkeypatch.undo()
    assert rp.plain(module, kind)
    object.__setattr__(module, name, other)
    assert not rp.plain(module, kind)


def test_a_method_put_on_torchs_class_before_is_seen(monkeypatch):
    own = nn.Linear.forward
    monkeypatch.setattr(nn.Linear, "forward", functools.wraps(own)(lambda self, x: own(self, x)))
    monkeypatch.setattr(rp, "_OWN", dict(rp._OWN))
    rp.own_methods(nn.Linear)
    assert not rp.plain(nn.Linear(4, 4), nn.Linear)


def test_a_layer_saved_without_orders_keeps_torchs_operations():
    layer = DecoderLayer(PRESETS["tiny"], 0, torch.float32, "cpu")
    vars(layer).pop("_orders", None)   # as an object pickled before there were any
    assert layer._as_rows(torch.zeros(1, 1, 256), None) is False


@pytest.mark.parametrize("k,same", [(64, 1), (128, 2), (192, 3), (256, 3), (512, 4), (4096, 4)])
def test_orders_that_are_one_for_short_rows(k, same):
    chains = {order: rp._chains(order, k) for order in rp.ORDERS}
    assert len(set(chains.values())) == same
    for found in chains.values():
        assert sorted(s for c in found for s in c) == list(range(k // 64))


def test_nothing_is_tried_on_tensors_without_memory():
    from torch._subclasses.fake_tensor import FakeTensorMode

    with FakeTensorMode(allow_non_fake_inputs=True):
        weight = torch.empty(4096, 4096, dtype=torch.bfloat16, device="cuda")
        assert rp.library_orders(weight) == {}


@pytest.mark.parametrize("path", ["layers.0.self_attn.o_proj", "layers.0.mlp.down_proj", "lm_head", "layers.0.input_layernorm", "norm"])
def test_projections_are_fused_beside_modules_of_somebody_elses(path):
    model = CascadeDecoder(PRESETS["tiny"], torch.float32, "cpu")
    parent, name = path.rpartition(".")[::2]
    setattr(model.get_submodule(parent), name, nn.Identity())   # no weight, no eps
    model.fuse_projections()
    assert model.layers[0].mlp._w_gate_up is not None and (path.startswith("layers") == (model.layers[0]._orders is None))


@pytest.mark.parametrize("kind", list(MAKE))
def test_a_compiled_module_is_called(kind):
    module = MAKE[kind]()
    module._compiled_call_impl = module._call_impl   # what Module.compile() sets
    assert not rp.plain(module, kind)


def test_numbers_of_workgroups_that_cut_alike_are_one():
    """501 tiles of 256 rows and 64 stretches: runs of 126, whether 256 workgroups share them or 255.  4752 of 32 rows and 14: 250 leave
    4500 whole ones, and the rest in runs of 15."""
    assert (1, 1, 256) in rp._cut_orders(128256, 4096, 256) and (1, 1, 255) not in rp._cut_orders(128256, 4096, 256)
    assert (4, 1, 250) in rp._cut_orders(152064, 3584, 256)
    assert rp._cut_orders(256 * 32, 4096, 256) == [o for o in rp._cut_orders(256 * 32, 4096, 256) if o[2] < 256]   # one round, nothing to cut
    assert not any(o[0] == 4 for o in rp._cut_orders(128256, 64 * 3, 256))   # stretches of 256 elements
