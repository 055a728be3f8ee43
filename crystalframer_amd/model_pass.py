"""The whole model in one library call per direction (cfh_model_forward / cfh_model_backward).

``Latticeformer.forward`` comes here first.  When the model and the batch are of the kind the library call covers (the
default architecture: no layer norm, no dropout, ReLU, "max" frames, mean pooling, a head of linear layers; float32
batches whose pair count is known on the host), the pass is ONE autograd function: embedding, geometry, layers, pooling and head
are enqueued by native code, the backward pass with all parameter gradients likewise.  Everything else takes the modules'
own forward: same kernels, one autograd function per operator.

The modules' path makes some thirty (inference) to eighty (training) calls from Python, each with its own allocations,
argument structures and autograd nodes: 755 us of host time per inference pass and 2330 us per training step of the
4-layer model, whatever the batch, where the GPU is busy for 168 us (one crystal) and 515 us (training step on 13).
"""
from __future__ import annotations

import ctypes
import math

import torch
import torch.autograd.forward_ad as fwAD
from torch import nn
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext

from . import _lib

ENABLED = True

# hooks of all modules of the program
_GLOBAL_HOOKS = [getattr(torch.nn.modules.module, n) for n in (
    "_global_forward_hooks", "_global_forward_pre_hooks", "_global_backward_hooks", "_global_backward_pre_hooks")]

# what a layer's pass takes from its attention's hyper-parameters
_SETTINGS = ("value_pe_dist_real", "value_pe_dist_max", "value_pe_dist_wscale", "value_pe_dist_coef", "value_pe_angle_real",
             "value_pe_angle_wscale", "value_pe_angle_coef", "cos_abs", "scale_real", "adaptive_cutoff_sigma", "gauss_lb_real",
             "positive_func_beta", "normalize_gauss", "frame_method")


def _on_device(weight) -> bool:
    return weight.is_cuda


def _no_plan():
    return None


class _Plan:
    """What a model's passes share: its parameters in the library's order, the structures that hold their addresses, and
    the objects all of it was derived from.  ``current()`` is False as soon as a module or parameter was added, removed or
    exchanged, a parameter got another storage or layout, or a layer another setting; the plan is then made again.  The native
    part keeps the storages whose addresses the library has, and a backward pass keeps the native part's."""

    def __init__(self, model):
        self.owner = model.__dict__
        self.links = []          # (dict, key, value): the plan holds while dict[key] is value
        self.walked = []         # (dict, entries): ... and while the dicts whose entries were walked have as many of them
        self.seen = set()
        self.params = []         # in the order of the library's gradients
        self.ok = False
        self.tables = {}         # kernel constants -> (layer structures, objects kept alive)
        self.hooks = []          # hooks of the modules that a pass calls as modules: dicts that have to be empty
        self.attn = []
        self._collect(model)
        del self.seen
        self.native = None
        if self.ok:
            self.native = _lib.load_host().Plan(self.links, self.walked, self.params, self.gauss, self.feat, self.D, self.H,
                                                  self.out_features)
        else:
            self.ptrs = [p.data_ptr() for p in self.params if p is not None]

    def __reduce_ex__(self, protocol):       # copies and pickles of a model carry no plan (addresses of the original)
        return _no_plan, ()

    def current(self) -> bool:
        if self.native is not None:
            return self.native.current()
        return (all(d.get(k) is v for d, k, v in self.links) and all(len(d) == n for d, n in self.walked)
                and [p.data_ptr() for p in self.params if p is not None] == self.ptrs)

    def _dict(self, module, name):
        """A module's ``_modules`` or ``_parameters``: taking an entry out of a ModuleList puts another dict in its place."""
        d = module.__dict__[name]
        if (id(module), name) not in self.seen:
            self.seen.add((id(module), name))
            self.links.append((module.__dict__, name, d))
        return d

    def _child(self, module, name):
        d = self._dict(module, "_modules")
        child = d.get(name)
        self.links.append((d, name, child))
        return child

    def _children(self, module):
        """The names of all children, in the order in which a forward pass goes through them."""
        d = self._dict(module, "_modules")
        self.walked.append((d, len(d)))
        return list(d)

    def _param(self, module, name):
        d = self._dict(module, "_parameters")
        p = d.get(name)
        self.links.append((d, name, p))
        return p

    def _setting(self, owner, name):
        v = owner.__dict__.get(name)
        self.links.append((owner.__dict__, name, v))
        return v

    def _called(self, module, kind) -> bool:
        """A module that the modules' path calls, so that hooks, a forward of its own and compilation count."""
        if type(module) is not kind:
            return False
        for n in ("_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks"):
            self.hooks.append(self._setting(module, n))
        own = [self._setting(module, n) for n in ("forward", "_compiled_call_impl")]
        return own == [None, None]

    def _collect(self, model):
        from . import cuda_funcs
        from .attention import CrystalformerMultiheadAttentionCUDA
        from .encoder import CrystalformerEncoderCUDA
        from .latticeformer import avr_pool
        enc = self._child(model, "encoder")
        emb = self._child(model, "input_embeddings")
        mlp = self._child(model, "mlp")
        pre = self._child(model, "proj_before_pooling")
        self.links.append((model.__dict__, "pooling_layer", model.__dict__.get("pooling_layer")))
        if not (isinstance(emb, nn.Linear) and isinstance(mlp, nn.Sequential) and self._called(pre, nn.Identity)
                and self._called(enc, CrystalformerEncoderCUDA) and model.__dict__.get("pooling_layer") is avr_pool and self._child(enc, "norm") is None):
            return
        layers = self._child(enc, "layers")
        self._setting(enc, "d_model")
        We = self._param(emb, "weight")
        # (a weight that a parametrization or a pruning mask makes is no parameter of its module)
        if We is None or self._param(emb, "bias") is not None or emb.bias is not None or len(layers) < 1:
            return
        self.params.append(We)
        self.layers = []
        for name in self._children(layers):
            layer = self._child(layers, name)
            at = self._child(layer, "self_attn")
            out_proj = self._child(at, "out_proj")
            l1, l2 = self._child(layer, "linear1"), self._child(layer, "linear2")
            for n in ("norm1", "norm2", "dropout", "dropout1", "dropout2"):
                if not isinstance(self._child(layer, n), nn.Identity):
                    return
            self.links.append((layer.__dict__, "activation", layer.activation))
            P = self._setting(at, "params")
            for n in ("num_heads", "head_dim", "kdim", "vdim"):
                self._setting(at, n)
            # (compared by identity from call to call: a value that can change in place is left to the modules)
            if type(at) is not CrystalformerMultiheadAttentionCUDA or [
                    n for n in ("attention_core", "project_inputs") if self._setting(at, n) is not None]:
                return
            if not all([isinstance(self._setting(P, n), (bool, int, float, str)) for n in _SETTINGS]):
                return
            A = P.value_pe_angle_real
            if not (layer.activation is torch.nn.functional.relu and P.frame_method == "max" and at.kdim == at.vdim == enc.d_model
                    and P.value_pe_dist_real > 0 and at.head_dim == 16
                    and cuda_funcs.AttentionInputsHIP.supported(at.num_heads, at.head_dim)):
                return
            names = ["q_proj_weight", "k_proj_weight", "v_proj_weight", "in_proj_bias"]
            ps = [self._param(at, n) for n in names] + [self._param(out_proj, "weight"), self._param(out_proj, "bias"),
                                                        self._param(at, "lattice_pos_weights"), self._param(at, "pe_dist_proj")]
            if A > 0:
                ps += [self._param(at, f"proj_angle{n}") for n in (1, 2, 3)]
            ps += [self._param(l1, "weight"), self._param(l1, "bias"), self._param(l2, "weight"), self._param(l2, "bias")]
            gauss = self._param(at, "gauss_scale")
            if any(p is None for p in ps):
                return
            if not (cuda_funcs.LayerBridgeHIP.supported(enc.d_model, ps[-4].shape[0], at.num_heads)
                    and cuda_funcs.PeriodicAttentionCoreHIP.supported(
                        P.value_pe_dist_real, A, P.value_pe_dist_wscale, P.value_pe_angle_wscale, at.pe_dist_proj,
                        at.proj_angle1 if A > 0 else None)):
                return
            self.params += ps
            self.attn.append(at)
            self.layers.append((at, ps, gauss, A))
        self.head = []
        mods = []
        for name in self._children(mlp):
            m = self._child(mlp, name)
            if isinstance(m, nn.Linear):
                W, b = self._param(m, "weight"), self._param(m, "bias")
                if W is None or b is None:
                    return
                mods.append([W, b, 0])
            elif isinstance(m, nn.ReLU) and mods and not mods[-1][2]:
                mods[-1][2] = 1
            elif not isinstance(m, nn.Identity):
                return
        D = enc.d_model
        if not 1 <= len(mods) <= _lib.MODEL_MAX_LINEARS or mods[-1][2] or D > _lib.MODEL_MAX_WIDTH or len(self.attn) > 64:
            return
        width = D
        for m in mods:
            W, b, relu = m
            if W.dim() != 2 or W.shape[1] != width or width % 16 or b.shape != W.shape[:1] or W.shape[0] > _lib.MODEL_MAX_WIDTH:
                return
            width = W.shape[0]
            self.params += [W, b]
        self.head, self.out_features = mods, width
        self.D, self.F, self.H, self.feat = D, self.layers[0][1][-4].shape[0], self.attn[0].num_heads, We.shape[1]
        dev = We.device
        if not _on_device(We) or not 1 <= self.feat <= 512 or We.shape[0] != D:
            return
        for p in self.params:
            if p.dtype != torch.float32 or p.device != dev or not p.is_contiguous():
                return
        for at, ps, gauss, A in self.layers:
            F, H = self.F, self.H
            shapes = [(D, D)] * 3 + [(3 * D,), (D, D), (D,), (D,), (1, H, 16, 64)] + [(1, H, 16, A)] * (3 if A > 0 else 0)
            shapes += [(F, D), (F,), (D, F), (D,)]
            # (the value encodings with or without their leading dimension)
            if (at.num_heads != H or A != self.layers[0][3]
                    or any(tuple(w.shape) != s and (1,) + tuple(w.shape) != s for w, s in zip(ps, shapes))
                    or gauss.device != dev or gauss.dtype != torch.float32 or gauss.numel() != 2 or not gauss.is_contiguous()):
                return
            at._stacked_in_proj()            # query, key and value weights as adjacent rows of one storage
        for at, ps, gauss, A in self.layers:
            q, k, v = ps[:3]                 # (they cannot be where a weight is shared, in a layer or between layers)
            if not (k.data_ptr() == q.data_ptr() + 4 * D * D and v.data_ptr() == k.data_ptr() + 4 * D * D):
                return
        self.in_proj = self.attn[0]._in_proj_stack.detach()
        # the gradients lie one behind the other: every one but the last starts on 16 bytes
        if any(p.numel() % 4 for p in self.params[:-1]):
            return
        self.gauss = [g for _, _, g, _ in self.layers]
        self.embedding, self.in_proj_bias = We.detach(), self.layers[0][1][3].detach()
        self.device = dev
        self.ok = True

    # ---- structures of the library call
    def constants(self):
        """What the attention cores take from KernelManager, as a key of ``tables``."""
        from .cuda_funcs import KernelManager as K
        sd = K.NOISE_SEED_DEVICE
        return (K.LATTICE_RANGE, K.MINIMUM_RANGE, K.CORE_WINDOW_MODE, K.PRUNE_LOG2, K.SYMM_BREAK_NOISE, K.NOISE_SEED,
                None if sd is None else sd.data_ptr(), bool(K.COLLECT_STATS))

    def table(self):
        key = self.constants()
        got = self.tables.get(key)
        if got is None:
            if len(self.tables) >= 8:
                self.tables.clear()
            got = self.tables[key] = self._build_table()
        return got

    def _build_table(self):
        from . import cuda_funcs
        K = cuda_funcs.KernelManager
        arr = (_lib.CfhModelLayer * len(self.layers))()
        seed = K.NOISE_SEED
        for S, (at, ps, gauss, A) in zip(arr, self.layers):
            P = at.params
            dist_max = P.value_pe_dist_max if P.value_pe_dist_max >= 0 else -P.value_pe_dist_max * P.scale_real
            cutoff = None
            if P.adaptive_cutoff_sigma != 0:
                cutoff = (P.adaptive_cutoff_sigma if P.adaptive_cutoff_sigma < 0
                          else P.scale_real * P.gauss_lb_real ** (-0.5) * P.adaptive_cutoff_sigma)
            p = cuda_funcs._params(at.num_heads, at.head_dim, P.value_pe_dist_real, A, P.cos_abs, dist_max,
                                   P.value_pe_dist_wscale, P.value_pe_angle_wscale, P.value_pe_dist_coef,
                                   P.value_pe_angle_coef, cutoff, noise_seed=0 if seed is None else seed)
            p.window_mode = int(K.CORE_WINDOW_MODE)
            S.core = p
            q, _, _, bq, Wo, bo, lw, Wd = ps[:8]
            S.Wqkv, S.bqkv, S.lattice_w = q.data_ptr(), bq.data_ptr(), lw.data_ptr()
            S.gauss_scale_dev = gauss.data_ptr() if P.normalize_gauss else None
            S.W_dist, S.Wo, S.bo = Wd.data_ptr(), Wo.data_ptr(), bo.data_ptr()
            if A > 0:
                S.W_axis1, S.W_axis2, S.W_axis3 = (w.data_ptr() for w in ps[8:11])
            S.W1, S.b1, S.W2, S.b2 = (w.data_ptr() for w in ps[-4:])
            S.c1, S.lb, S.c2 = at._gauss_constants()
            S.q_scale = 1.0 / math.sqrt(at.head_dim)
            S.adaptive = 1 if cutoff is not None else 0
        m = _lib.CfhModel()
        m.struct_size = ctypes.sizeof(_lib.CfhModel)
        m.layers, m.heads, m.D, m.F, m.feat, m.linears = len(self.layers), self.H, self.D, self.F, self.feat, len(self.head)
        m.We = self.params[0].data_ptr()
        m.layer = ctypes.cast(arr, ctypes.POINTER(_lib.CfhModelLayer))
        for T, (W, b, relu) in zip(m.head, self.head):
            T.W, T.b, T.K, T.O, T.relu = W.data_ptr(), b.data_ptr(), W.shape[1], W.shape[0], relu
        return m, arr, (K.NOISE_SEED_DEVICE, list(self.gauss)), ctypes.addressof(m)


def _switches_default() -> bool:
    """The switches that choose between the kernels' variants from Python stand where this path stands."""
    from . import attention, cuda_funcs, encoder, geometry
    K = cuda_funcs.KernelManager
    return (ENABLED and attention.FUSED_CORE and attention.FUSED_INPUTS and encoder.FUSED_LAYER_BRIDGE and geometry.USE_LIBRARY
            and cuda_funcs.LayerBridgeHIP.FUSED_BACKWARD and K.DEFER_WEIGHT_GRADS and K.DEFER_CORE_WEIGHT_GRADS
            and K.DETERMINISTIC_WEIGHT_GRADIENTS and not K.GRAD_COEF_QUIRK and K.EVENT_LOG is None)


def _forward(plan, args, keep: bool):
    from .cuda_funcs import KernelManager as K, LinearHIP
    table = plan.table()
    m, arr = table[0], table[1]
    dev = plan.device
    x = args[0]
    first = ()
    if keep and x.shape[0] > LinearHIP.SMALL_ROWS:
        # the embedding and the first projection of a long batch as the modules' path makes them, by the framework's
        # GEMM: a training step is then the same to the last bit whichever path makes it
        with torch.no_grad():
            x0 = torch.nn.functional.linear(x, plan.embedding)
            first = (x0, torch.nn.functional.linear(x0, plan.in_proj, plan.in_proj_bias))
    seeds = ()
    if K.NOISE_SEED is None and K.SYMM_BREAK_NOISE > 0:
        seeds = [int(torch.randint(0, 2 ** 62, (1,)).item()) for _ in arr]
    return plan.native.forward(table[3], table, *args, keep, lambda n: _lib.workspace(dev, n), seeds, first)


def _eager(host, keep: bool) -> bool:
    """Whether what the pass does to tensors is seen by nobody but autograd's backward pass: one native call has no forward-mode
    derivative, no batching rule and nothing that a tracer or a mode could record."""
    seen = host.watchers()
    if seen == 0 and fwAD._current_level < 0:
        return True
    if fwAD._current_level >= 0 or seen & host.WATCHED or (keep and seen & host.SAVED_TENSOR_HOOKS):
        return False
    # a function mode that only chooses the device of new tensors (torch.set_default_device) changes nothing here
    return not seen & host.FUNCTION_MODE or all(type(m) is DeviceContext for m in _get_current_function_mode_stack())


def covered(model, data):
    """(plan, arguments, keep) of the native call for ``data``, or None when the pass is not one this path covers."""
    if torch.compiler.is_compiling() or not _switches_default():
        return None
    host = _lib.load_host()
    keep = torch.is_grad_enabled()
    if not _eager(host, keep):
        return None
    plan = model.__dict__.get("_pass_plan")
    if plan is None or plan.owner is not model.__dict__ or not plan.current():      # (a shallow copy has its original's plan)
        plan = model.__dict__["_pass_plan"] = _Plan(model)
    if not plan.ok:
        return None
    x, pos, batch, trans, sizes = data.x, data.pos, data.batch, data.trans_vec, data.sizes
    if sizes is None or torch.is_autocast_enabled() or not plan.native.accepts(x, pos, batch, trans, sizes):
        return None
    for at in plan.attn:
        if at.frame_sink is not None or at.grad_sink is not None:
            return None
        if at.params.normalize_gauss and not at._gauss_scale_ready():
            return None
    if any(plan.hooks) or any(_GLOBAL_HOOKS):
        return None
    if not getattr(data, "zero_based", False):       # the reference subtracts batch[0]
        batch = batch - batch[0]
    E = getattr(data, "num_pairs", -1)
    if E is None or E < 0:                           # not known on the host: read back, as the modules' path does
        E = int((sizes * sizes).sum().item())
    if E < 1:
        return None
    lim = 1 << 30
    if x.shape[0] * plan.D >= lim or E * max(plan.H, 3) >= lim:
        return None
    if keep:
        if x.requires_grad or pos.requires_grad or trans.requires_grad:
            return None
        wanted = plan.native.wanted()
        if wanted == 1:
            return None
        keep = wanted == 2
    return plan, (x, pos, batch, trans, sizes, int(E)), keep


def run(model, data):
    """The model's output for ``data``, or None when the pass is not one this path covers."""
    found = covered(model, data)
    if found is None:
        return None
    plan, args, keep = found
    if torch.cuda.current_device() != plan.device.index:
        with torch.cuda.device(plan.device):
            return _forward(plan, args, keep)
    return _forward(plan, args, keep)
