"""What the whole-model pass keeps between calls (model_pass._Plan), looked at on the CPU: the plan of a model is made again
when what it was derived from changes, and a pass it does not cover is left to the modules."""
import copy

import pytest
import torch
import torch.autograd.forward_ad as fwAD
import torch.nn.utils.prune  # noqa: F401
from torch import nn
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from crystalframer_amd import encoder, latticeformer, model_pass, params, synthetic


@pytest.fixture
def planned(monkeypatch):
    """A model and its plan."""
    monkeypatch.setattr(model_pass, "_on_device", lambda weight: True)
    torch.manual_seed(0)
    model = latticeformer.Latticeformer(params.ModelParams(num_layers=2))
    for layer in model.encoder.layers:
        layer.self_attn.gauss_scale.data.fill_(0.5)
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


def test_another_layout_at_the_same_address_makes_the_plan_anew(planned):
    model, plan = planned
    at, head = model.encoder.layers[1].self_attn, model.mlp[0]
    for p in (at.out_proj.weight, head.weight):
        p.data = p.data.t()                          # square: same address, same sizes
        assert not plan.current() and not model_pass._Plan(model).ok
        p.data = p.data.t()
        assert plan.current()
    lin = model.encoder.layers[0].linear1
    lin.weight.data = lin.weight.data.view(128, 512)
    assert not plan.current() and not model_pass._Plan(model).ok
    lin.weight.data = lin.weight.data.view(512, 128)
    at.gauss_scale.data = torch.zeros(4)[::2]
    assert not plan.current() and not model_pass._Plan(model).ok


@pytest.mark.parametrize("name,value", [
    ("value_pe_dist_max", -8.0), ("value_pe_dist_wscale", 1.5), ("value_pe_dist_coef", 2.0), ("value_pe_angle_wscale", 5.0),
    ("value_pe_angle_coef", 3.0), ("cos_abs", 1), ("scale_real", 1.3), ("adaptive_cutoff_sigma", 2.5), ("gauss_lb_real", 0.4),
    ("positive_func_beta", 0.2), ("normalize_gauss", False), ("frame_method", "pca"), ("value_pe_angle_real", 0),
    ("value_pe_dist_real", 0)])
def test_another_setting_of_a_layer_makes_the_plan_anew(planned, name, value):
    model, plan = planned
    P = model.encoder.layers[1].self_attn.params
    old = getattr(P, name)
    setattr(P, name, value)
    assert not plan.current()
    model_pass._Plan(model)                          # (covered or not, it can be asked)
    setattr(P, name, old)
    assert plan.current()
    setattr(P, name, torch.tensor(1.0))              # may change in place: not covered
    assert not plan.current() and not model_pass._Plan(model).ok


def test_weights_of_another_shape_are_not_covered(planned):
    """The library reads as many words as the widths say."""
    model, plan = planned
    lin = model.mlp[3]                               # 128 -> 1
    lin.out_features = 4
    assert model_pass._Plan(model).out_features == 1
    lin.bias = nn.Parameter(torch.zeros(2))
    assert not plan.current() and not model_pass._Plan(model).ok
    lin.bias = nn.Parameter(torch.zeros(1))
    assert model_pass._Plan(model).ok
    at = model.encoder.layers[0].self_attn
    at.proj_angle2 = nn.Parameter(torch.zeros(1, 8, 16, 32))
    assert not model_pass._Plan(model).ok
    at.proj_angle2 = nn.Parameter(torch.zeros(8, 16, 64))
    assert model_pass._Plan(model).ok


def test_shared_projection_weights_are_not_covered(planned):
    """The library reads the query, key and value weights as one matrix, from the address of the first."""
    model, plan = planned
    first, second = (layer.self_attn for layer in model.encoder.layers)
    own = first.k_proj_weight
    first.k_proj_weight = first.q_proj_weight
    assert not plan.current() and not model_pass._Plan(model).ok
    first.k_proj_weight = own
    assert model_pass._Plan(model).ok
    second.q_proj_weight = first.q_proj_weight
    assert not model_pass._Plan(model).ok


@pytest.mark.parametrize("where", ["input_embeddings", "mlp.0", "mlp.3", "encoder.layers.1.linear2",
                                   "encoder.layers.0.self_attn.out_proj"])
def test_reparametrised_weights_are_not_covered(planned, where):
    model, plan = planned
    module = model.get_submodule(where)
    nn.utils.parametrizations.weight_norm(module)
    assert not plan.current() and not model_pass._Plan(model).ok
    nn.utils.parametrize.remove_parametrizations(module, "weight")
    assert model_pass._Plan(model).ok
    nn.utils.prune.l1_unstructured(module, "weight", amount=0.5)
    assert not model_pass._Plan(model).ok


def test_an_embedding_with_a_bias_is_not_covered(planned):
    model, plan = planned
    model.input_embeddings.bias = nn.Parameter(torch.ones(128))
    assert not plan.current() and not model_pass._Plan(model).ok
    nn.utils.parametrize.register_parametrization(model.input_embeddings, "bias", nn.Identity())
    assert model.input_embeddings.bias is not None and not model_pass._Plan(model).ok


def _batch():
    return synthetic.make_config("C1", seed=5, num_crystals=3)


def test_forward_derivatives_tracers_and_modes_are_left_to_the_modules(planned):
    model, plan = planned
    cb = _batch()
    covered = lambda data=cb: model_pass.covered(model, data) is not None  # noqa: E731
    assert covered()
    with fwAD.dual_level():
        assert not covered()
    seen = []
    look = lambda t: (seen.append(covered()), t.sum())[1]  # noqa: E731
    torch.func.grad(look)(torch.ones(3))
    torch.func.vmap(look)(torch.ones(3, 2))
    torch.func.jvp(look, (torch.ones(3),), (torch.ones(3),))
    torch.jit.trace(look, (torch.ones(3),), check_trace=False)
    make_fx(look)(torch.ones(3))
    assert len(seen) >= 5 and not any(seen)
    with FakeTensorMode():
        assert not covered()

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    for mode in (Dispatch(), Function()):
        with mode:
            assert not covered()
    with torch.device("cpu"):                        # only chooses the device of new tensors
        assert covered()
        with Function():
            assert not covered()
    assert covered()


def test_hooks_on_saved_tensors_are_left_to_the_modules(planned):
    model, plan = planned
    cb = _batch()
    with torch.autograd.graph.save_on_cpu():         # (activation checkpointing is one of these as well)
        assert model_pass.covered(model, cb) is None
        with torch.no_grad():                        # nothing is saved
            assert model_pass.covered(model, cb) is not None
    with torch.autograd.graph.disable_saved_tensors_hooks("none"):
        assert model_pass.covered(model, cb) is not None


@pytest.mark.parametrize("where", ["encoder", "proj_before_pooling"])
def test_hooks_and_own_forwards_of_the_called_modules_are_left_to_the_modules(planned, where):
    model, plan = planned
    cb = _batch()
    module = model.get_submodule(where)
    covered = lambda: model_pass.covered(model, cb) is not None  # noqa: E731
    for register in (module.register_forward_hook, module.register_forward_pre_hook, module.register_full_backward_hook,
                     module.register_full_backward_pre_hook):
        handle = register(lambda *a: None)
        assert not covered()
        handle.remove()
        assert covered()
    module.forward = module.forward
    assert not covered()
    del module.forward
    assert covered()
    module.compile()
    assert not covered()

    class Other(type(module)):
        pass

    if where == "proj_before_pooling":
        model.proj_before_pooling = Other()
        assert not covered()


def test_hooks_of_all_modules_are_left_to_the_modules(planned):
    model, plan = planned
    cb = _batch()
    for register in (nn.modules.module.register_module_forward_hook, nn.modules.module.register_module_forward_pre_hook,
                     nn.modules.module.register_module_full_backward_hook,
                     nn.modules.module.register_module_full_backward_pre_hook):
        handle = register(lambda *a: None)
        assert model_pass.covered(model, cb) is None
        handle.remove()
        assert model_pass.covered(model, cb) is not None


def test_an_attention_with_methods_of_its_own_is_left_to_the_modules(planned):
    model, plan = planned
    at = model.encoder.layers[1].self_attn
    at.attention_core = at.attention_core
    assert not plan.current() and not model_pass._Plan(model).ok
    del at.attention_core
    assert plan.current()


@pytest.mark.parametrize("name,change", [
    ("pos", lambda t: t[:-1]), ("pos", lambda t: t[:, :2].contiguous()), ("batch", lambda t: t[:-1]), ("sizes", lambda t: t[:-1]),
    ("sizes", lambda t: t[None]), ("trans_vec", lambda t: t.reshape(-1, 9)), ("trans_vec", lambda t: t.flatten()),
    ("pos", lambda t: t.t().contiguous().t()), ("x", lambda t: t[:-1])])
def test_batches_of_other_shapes_are_left_to_the_modules(planned, name, change):
    model, plan = planned
    cb = _batch()
    assert model_pass.covered(model, cb) is not None
    setattr(cb, name, change(getattr(cb, name)))
    assert model_pass.covered(model, cb) is None


def test_a_plan_made_in_inference_mode_leaves_the_parameters_trainable(monkeypatch):
    monkeypatch.setattr(model_pass, "_on_device", lambda weight: True)
    model = latticeformer.Latticeformer(params.ModelParams(num_layers=2))
    with torch.inference_mode():
        assert model_pass._Plan(model).ok
    for n, p in model.named_parameters():
        assert not p.is_inference() and not p.data.is_inference(), n
        assert p.requires_grad == (not n.endswith("_scale")), n
    assert model_pass._Plan(model).native.wanted() == 2


def test_a_shallow_copy_has_a_plan_of_its_own(planned):
    model, plan = planned
    cb = _batch()
    assert model_pass.covered(model, cb) is not None
    other = copy.copy(model)
    assert model_pass.covered(other, cb)[0] is not model_pass.covered(model, cb)[0]
    other = copy.copy(model)
    other.pooling_layer = latticeformer.max_pool
    assert model_pass.covered(other, cb) is None and model_pass.covered(model, cb) is not None
