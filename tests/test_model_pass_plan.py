"""What the whole-model pass keeps between calls (model_pass._Plan), looked at on the CPU: the plan of a model is made again
when what it was derived from changes, and a pass it does not cover is left to the modules."""
import pytest
import torch
from torch import nn

from crystalframer_amd import encoder, latticeformer, model_pass, params


@pytest.fixture
def planned(monkeypatch):
    """A model and its plan."""
    monkeypatch.setattr(model_pass, "_on_device", lambda weight: True)
    torch.manual_seed(0)
    model = latticeformer.Latticeformer(params.ModelParams(num_layers=2))
    plan = model_pass._Plan(model)
    assert plan.ok and plan.current()
    return model, plan


def test_an_added_or_removed_module_makes_the_plan_anew(planned):
    model, plan = planned
    layer = encoder.CrystalformerEncoderLayerCUDA(128, 8, 512, 0.0, no_layer_norm=True,
                                                  params=model.encoder.lattice_params.getLayerParameters(2))
    model.encoder.layers.append(layer)
    assert not plan.current()
    again = model_pass._Plan(model)
    assert again.ok and len(again.attn) == 3 and again.current()
    del model.encoder.layers[2]                      # (puts another dict of modules in the place of the old one)
    assert not again.current()
    plan = model_pass._Plan(model)
    assert plan.ok and len(plan.attn) == 2
    model.mlp.append(nn.Tanh())
    assert not plan.current() and not model_pass._Plan(model).ok
    del model.mlp[-1]
    plan = model_pass._Plan(model)
    assert plan.ok
    model.mlp.insert(1, nn.ReLU())
    assert not plan.current()
