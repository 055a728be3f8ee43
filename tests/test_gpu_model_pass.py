"""The whole-model library call (cfh_model_forward / cfh_model_backward) against the modules' own path, which makes the
same kernels' calls one operator at a time: the same bits where both use the library's kernels throughout, float32
rounding where the modules' path hands a product to the framework's GEMM."""
import copy

import pytest
import torch

import helpers as Hh

pytestmark = pytest.mark.gpu


def _model(mp, cb, seed=1, change=None):
    from crystalframer_amd import latticeformer
    dev = torch.device("cuda:0")
    torch.manual_seed(seed)
    model = latticeformer.Latticeformer(mp).to(dev)
    if change is not None:
        change(model)
    cb = cb.to(dev)
    model.train()
    model(cb)                                   # stores the normalisation of alpha (modules' path)
    return model, cb


def _both(mp, cb, seed=1, change=None, before=None):
    """Outputs and gradients of the native call and of the modules.  change: of the model; before: each of the passes."""
    from crystalframer_amd import model_pass
    dev = torch.device("cuda:0")
    model, cb = _model(mp, cb, seed, change)
    target = torch.linspace(-1, 1, cb.num_crystals * model.mlp[-1].out_features, device=dev).view(cb.num_crystals, -1)
    results = []
    for on in (True, False):
        model_pass.ENABLED = on
        try:
            model.zero_grad(set_to_none=True)
            if before is not None:
                before()
            out = model(cb)
            torch.nn.functional.mse_loss(out, target).backward()
            if before is not None:
                before()
            with torch.no_grad():
                ev = model(cb)
        finally:
            model_pass.ENABLED = True
        assert (out.grad_fn.name() == "ModelPassHIPBackward") == on
        results.append((out.detach(), ev, {n: p.grad.clone() for n, p in model.named_parameters() if p.grad is not None}))
    return model, cb, results


# one atom; a tile of 16 atoms and its edges; one crystal; more crystals than a workgroup of the tail takes (1, 4, 16);
# around the 512 rows where the modules' path hands the first projection to the framework's GEMM
@pytest.mark.parametrize("B,hi,bins,layers", [(1, 1, 64, 1), (1, 16, 64, 2), (3, 6, 16, 2), (16, 2, 0, 1), (17, 9, 64, 4),
                                              (97, 9, 0, 4), (120, 9, 16, 3), (513, 3, 64, 2), (2050, 2, 0, 1)])
def test_one_call_equals_the_modules_path(B, hi, bins, layers):
    from crystalframer_amd import params, synthetic
    kw = dict(value_pe_angle_wscale=1.0, value_pe_dist_coef=1.5, value_pe_angle_coef=6.0) if bins == 16 else {}
    mp = params.ModelParams(num_layers=layers, value_pe_angle_real=bins, symm_break_noise=0.0, **kw)
    cb = synthetic.make_batch(B, atoms="uniform", atoms_lo=1, atoms_hi=hi, len_lo=3.0, len_hi=9.0, ang_lo=65.0, ang_hi=115.0,
                              seed=B)
    model, cb, ((o1, e1, g1), (o2, e2, g2)) = _both(mp, cb)
    assert g1.keys() == g2.keys() and len(g1) == (4 + 15 * layers if bins else 4 + 12 * layers) + 1
    if B <= 512:                                # (above, the modules' head goes through the framework's GEMM)
        assert torch.equal(o1, o2)
        for n in g1:
            assert torch.equal(g1[n], g2[n]), n
    assert Hh.rel_err(o1, o2.double()) < 1e-6 and Hh.rel_err(e1, e2.double()) < 1e-6
    for n in g1:                                # (a rectifier whose input rounds to the other sign moves one atom's share)
        assert Hh.rel_err(g1[n], g2[n].double()) < (1e-5 if B <= 512 else 2e-3), n


# The sums over the pairs that point at an atom, four atoms per wavefront from 18 432 items on (here of 13 and 14 atoms each),
# with rows of more than 24 pairs from 10 240 on; the modules' pairs are looked at first and rows of up to 24 take one.
@pytest.mark.parametrize("B,lo,hi", [(177, 13, 14), (168, 13, 14), (46, 27, 31), (42, 27, 31)])
def test_column_sums_of_a_batch(B, lo, hi):
    from crystalframer_amd import params, synthetic
    mp = params.ModelParams(num_layers=2, value_pe_angle_real=0, symm_break_noise=0.0)
    cb = synthetic.make_batch(B, atoms="uniform", atoms_lo=lo, atoms_hi=hi, len_lo=4.0, len_hi=9.0, ang_lo=65.0, ang_hi=115.0, seed=B)
    N = cb.pos.shape[0]
    assert (8 * N >= (10240 if lo > 24 else 18432)) == (B in (177, 46))
    _, _, ((o1, _, g1), (o2, _, g2)) = _both(mp, cb)
    assert torch.equal(o1, o2)
    for n in g1:
        assert torch.equal(g1[n], g2[n]), n


# (from 445 features on, a workgroup of the tail takes more than 64 KB of LDS; 480 is the widest head it takes)
@pytest.mark.parametrize("widths", [[64, 208], [448], [464], [480, 16, 480]])
def test_head_of_several_layers_and_targets(widths):
    from crystalframer_amd import params, synthetic
    mp = params.ModelParams(num_layers=1, symm_break_noise=0.0, embedding_dim=widths, targets=["a", "b", "c"])
    cb = synthetic.make_batch(21, atoms="uniform", atoms_lo=1, atoms_hi=5, len_lo=3.0, len_hi=9.0, ang_lo=65.0, ang_hi=115.0,
                              seed=4)
    model, cb, ((o1, e1, g1), (o2, e2, g2)) = _both(mp, cb)
    assert o1.shape == (21, 3)
    assert Hh.rel_err(o1, o2.double()) < 1e-6 and Hh.rel_err(e1, e2.double()) < 1e-6
    for n in g1:
        assert Hh.rel_err(g1[n], g2[n].double()) < 1e-5, n


def test_copies_exchanged_weights_and_changes_before_the_backward_pass():
    from crystalframer_amd import params, synthetic
    mp = params.ModelParams(num_layers=1, symm_break_noise=0.0)
    cb = synthetic.make_batch(5, atoms="uniform", atoms_lo=1, atoms_hi=5, len_lo=3.0, len_hi=9.0, ang_lo=65.0, ang_hi=115.0,
                              seed=6)
    model, cb, _ = _both(mp, cb)
    with torch.no_grad():
        ref = model(cb)
        assert torch.equal(copy.deepcopy(model)(cb), ref)
        layer = model.encoder.layers[0]
        old = layer.linear1.weight
        layer.linear1.weight = torch.nn.Parameter(old * 2.0)           # another parameter
        changed = model(cb)
        assert not torch.equal(changed, ref)
        layer.linear1.weight.data = old.detach().clone()               # another storage
        assert torch.equal(model(cb), ref)
    out = model(cb)
    with torch.no_grad():
        layer.linear1.weight.mul_(1.5)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.sum().backward()


def test_backward_pass_after_the_storages_of_the_weights_were_exchanged():
    """The gradients are those of what the forward pass computed, whatever the parameters hold by then."""
    from crystalframer_amd import params, synthetic
    mp = params.ModelParams(num_layers=2, symm_break_noise=0.0)
    cb = synthetic.make_batch(5, atoms="uniform", atoms_lo=1, atoms_hi=5, len_lo=3.0, len_hi=9.0, ang_lo=65.0, ang_hi=115.0,
                              seed=6)
    model, cb, ((_, _, want), _) = _both(mp, cb)
    target = torch.linspace(-1, 1, 5, device="cuda").view(5, 1)
    model.zero_grad(set_to_none=True)
    loss = torch.nn.functional.mse_loss(model(cb), target)
    with torch.no_grad():
        for p in model.parameters():
            p.data = p.data * 3.0 + 1.0
        model(cb)                                    # (the plan is made again)
        for n in ("x", "pos", "trans_vec", "sizes", "batch"):
            t = getattr(cb, n)
            t.data = t.clone()
        # takes the memory given back
        fill = [torch.full_like(p, 7.0) for p in model.parameters() for _ in range(3)]
        fill += [torch.full_like(getattr(cb, n), 7) for n in ("x", "pos", "trans_vec", "sizes", "batch") for _ in range(3)]
    loss.backward()
    for n, p in model.named_parameters():
        if n in want:
            assert torch.equal(p.grad, want[n]), n
    assert len(fill) > 0
    # memory that is no longer there is not read
    for t in (cb.pos, model.mlp[0].weight):
        out, copy_of_t, size = model(cb), t.detach().clone(), t.untyped_storage().nbytes()
        t.untyped_storage().resize_(0)
        with pytest.raises(RuntimeError, match="resized or given back"):
            out.sum().backward()
        t.untyped_storage().resize_(size)
        t.detach().copy_(copy_of_t)


@pytest.fixture
def kernel_constants():
    """The constants of the kernels, put back after a test."""
    from crystalframer_amd.cuda_funcs import KernelManager as K
    names = ("NOISE_SEED", "NOISE_SEED_DEVICE", "SYMM_BREAK_NOISE", "LATTICE_RANGE", "MINIMUM_RANGE")
    saved = {n: getattr(K, n) for n in names}
    yield K
    for n, v in saved.items():
        setattr(K, n, v)


# few items, of which a wavefront takes each from its record to the sums, and more (5120 items and 8 heads: 640 atoms)
@pytest.mark.parametrize("B,hi", [(7, 6), (97, 16)])
@pytest.mark.parametrize("seeds", ["fixed", "drawn", "on the device"])
def test_noise_of_the_frame_search(kernel_constants, B, hi, seeds):
    """The same seeds for the same layers as in the modules' path: fixed, drawn per layer and pass, or mixed with a word on the
    device that every search advances."""
    from crystalframer_amd import params, synthetic
    K = kernel_constants
    mp = params.ModelParams(num_layers=3, symm_break_noise=1e-2)      # (large: another seed is another frame)
    cb = synthetic.make_batch(B, atoms="uniform", atoms_lo=1, atoms_hi=hi, len_lo=3.0, len_hi=9.0, ang_lo=65.0, ang_hi=115.0,
                              seed=B)
    word = torch.zeros(1, dtype=torch.int64, device="cuda")
    K.NOISE_SEED = None if seeds == "drawn" else 77

    def before(start=5):
        torch.manual_seed(start)
        K.NOISE_SEED_DEVICE = word if seeds == "on the device" else None
        word.fill_(start)

    model, cb, ((o1, e1, g1), (o2, e2, g2)) = _both(mp, cb, before=before)
    assert torch.equal(o1, o2)
    for n in g1:
        # (with seeds of their own the modules' path sums the layers' core weights in separate launches, the atoms in other
        # slices: a rounding of 6e-8 per atom at worst)
        sliced = seeds == "drawn" and ("proj_angle" in n or "pe_dist" in n)
        err = Hh.rel_err(g1[n], g2[n].double())
        assert err < 6e-8 * cb.pos.shape[0] if sliced else torch.equal(g1[n], g2[n]), (n, err)
    assert Hh.rel_err(e1, e2.double()) < 1e-4
    if seeds != "fixed":
        before(6)
        assert not torch.equal(model(cb), o1)


def test_wide_model():
    from crystalframer_amd import params, synthetic
    mp = params.ModelParams(num_layers=2, symm_break_noise=0.0, model_dim=256, ff_dim=384, head_num=16, embedding_dim=[256])
    cb = synthetic.make_batch(19, atoms="uniform", atoms_lo=1, atoms_hi=7, len_lo=3.0, len_hi=9.0, ang_lo=65.0, ang_hi=115.0,
                              seed=4)
    model, cb, ((o1, e1, g1), (o2, e2, g2)) = _both(mp, cb)
    assert torch.equal(o1, o2) and Hh.rel_err(e1, e2.double()) < 1e-6
    for n in g1:
        assert torch.equal(g1[n], g2[n]), n


# (half-width of the layers' usual box without and with the adaptive cutoff): the tables of one serve some layers only
@pytest.mark.parametrize("fixed,adaptive", [(2, 1), (2, 0), (1, 2)])
@pytest.mark.parametrize("rules", ["fa", "af", "faf", "afa", "aaf"])
def test_layers_with_different_box_rules(kernel_constants, fixed, adaptive, rules):
    from crystalframer_amd import params, synthetic
    mp = params.ModelParams(num_layers=len(rules), symm_break_noise=0.0)
    cb = synthetic.make_batch(9, atoms="uniform", atoms_lo=1, atoms_hi=6, len_lo=3.0, len_hi=9.0, ang_lo=65.0, ang_hi=115.0,
                              seed=4)

    def change(model):
        kernel_constants.LATTICE_RANGE, kernel_constants.MINIMUM_RANGE = fixed, adaptive
        for layer, rule in zip(model.encoder.layers, rules):
            if rule == "f":
                layer.self_attn.params.adaptive_cutoff_sigma = 0.0

    model, cb, ((o1, e1, g1), (o2, e2, g2)) = _both(mp, cb, change=change)
    assert torch.equal(o1, o2) and Hh.rel_err(e1, e2.double()) < 1e-6
    for n in g1:
        assert torch.equal(g1[n], g2[n]), n
    out = model(cb)
    g = torch.ones_like(out)
    first = torch.autograd.grad(out, [model.mlp[0].weight, model.input_embeddings.weight], g, retain_graph=True)
    second = torch.autograd.grad(out, [model.mlp[0].weight, model.input_embeddings.weight], g)
    assert torch.equal(first[0], second[0]) and torch.equal(first[1], second[1])


# few atoms and more than the slow lists' leading wavefronts serve
@pytest.mark.parametrize("B,hi,bins", [(7, 6, 64), (150, 20, 64), (150, 20, 0), (60, 12, 16)])
def test_backward_passes_as_autograd_makes_them(B, hi, bins):
    """A second pass over a kept graph, gradients of some parameters only, accumulation, another stream, and a graph that is
    used up."""
    from crystalframer_amd import params, synthetic
    kw = dict(value_pe_angle_wscale=1.0, value_pe_dist_coef=1.5, value_pe_angle_coef=6.0) if bins == 16 else {}
    mp = params.ModelParams(num_layers=2, value_pe_angle_real=bins, symm_break_noise=0.0, **kw)
    cb = synthetic.make_batch(B, atoms="uniform", atoms_lo=1, atoms_hi=hi, len_lo=3.0, len_hi=9.0, ang_lo=65.0, ang_hi=115.0,
                              seed=B)
    model, cb = _model(mp, cb)
    named = {n: p for n, p in model.named_parameters() if p.requires_grad}
    gout = torch.linspace(-1, 1, B, device="cuda").view(B, 1)
    out = model(cb)
    assert out.grad_fn.name() == "ModelPassHIPBackward"
    want = dict(zip(named, torch.autograd.grad(out, list(named.values()), gout, retain_graph=True)))
    some = [n for n in named if n.endswith("linear1.weight") or n == "input_embeddings.weight"]
    for n, g in zip(some, torch.autograd.grad(out, [named[n] for n in some], gout, retain_graph=True)):
        assert torch.equal(g, want[n]), n
    out.backward(gout)                               # .grad made
    for n, p in named.items():
        assert torch.equal(p.grad, want[n]), n
    with pytest.raises(RuntimeError, match="second time"):
        out.backward(gout)
    model(cb).backward(gout)                         # added to .grad
    for n, p in named.items():
        assert torch.equal(p.grad, 2.0 * want[n]), n
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        model.zero_grad(set_to_none=True)
        here = model(cb)
        assert torch.equal(here, out)
        here.backward(gout)
    torch.cuda.current_stream().wait_stream(side)
    for n, p in named.items():
        assert torch.equal(p.grad, want[n]), n
    # two passes over other batches between a forward pass and its backward pass
    model.zero_grad(set_to_none=True)
    out = model(cb)
    other = synthetic.make_batch(3, atoms="uniform", atoms_lo=1, atoms_hi=4, len_lo=3.0, len_hi=9.0, ang_lo=65.0, ang_hi=115.0,
                                 seed=1).to("cuda")
    model(other)
    torch.autograd.grad(model(other).sum(), list(named.values()))
    out.backward(gout)
    for n, p in named.items():
        assert torch.equal(p.grad, want[n]), n


@pytest.mark.parametrize("bins", [64, 16, 0])
def test_items_in_one_launch_and_in_several(bins):
    """Up to 5120 (atom, head) items a wavefront takes an item through a layer, above the items go through three launches: the
    crystals of the smaller batch are answered alike in the larger one."""
    from crystalframer_amd import params, synthetic
    kw = dict(value_pe_angle_wscale=1.0, value_pe_dist_coef=1.5, value_pe_angle_coef=6.0) if bins == 16 else {}
    mp = params.ModelParams(num_layers=2, value_pe_angle_real=bins, symm_break_noise=0.0, **kw)
    B = 80
    cb = synthetic.make_batch(B + 1, atoms="uniform", atoms_lo=8, atoms_hi=8, len_lo=3.0, len_hi=9.0, ang_lo=65.0, ang_hi=115.0,
                              seed=3)
    less = synthetic.CrystalBatch(cb.x[:8 * B], cb.pos[:8 * B], cb.batch[:8 * B], cb.trans_vec[:B], cb.sizes[:B], zero_based=True)
    model, less = _model(mp, less)
    more = cb.to("cuda")
    assert less.x.shape[0] * 8 == 5120 and more.x.shape[0] * 8 == 5184
    gout = torch.linspace(-1, 1, B, device="cuda").view(B, 1)
    named = [p for p in model.parameters() if p.requires_grad]
    a, b = model(less), model(more)
    assert Hh.rel_err(b[:B], a.double()) < 1e-6
    with torch.no_grad():
        assert Hh.rel_err(model(more)[:B], model(less).double()) < 1e-6
    ga = torch.autograd.grad(a, named, gout)
    gb = torch.autograd.grad(b, named, torch.cat([gout, torch.zeros(1, 1, device="cuda")]))
    for p, q in zip(ga, gb):
        assert Hh.rel_err(q, p.double()) < 2e-5      # (sums over the atoms in other slices)


def test_the_library_times_the_kernels_of_the_model_pass():
    """What bench.py reports per kernel comes from the pass it times."""
    from crystalframer_amd import _lib, params, synthetic
    cb = synthetic.make_batch(7, atoms="uniform", atoms_lo=1, atoms_hi=4, len_lo=3.0, len_hi=9.0, ang_lo=65.0, ang_hi=115.0,
                              seed=1)
    model, cb = _model(params.ModelParams(num_layers=3, symm_break_noise=0.0), cb)
    names = dict(model_forward=1, model_backward=1, model_start=1, layer_front=1, item_pass=3, core_project=3,
                 layer_bridge_forward=3, model_tail=2, layer_bridge_backward=4, core_gbuild=3, fused_core_backward=3,
                 core_bwd_col=3, linear_weight_gradients=1, core_weight_gradients=1, fused_core_forward=0, core_prepare=0)
    for n in names:
        _lib.read_kernel_timing(n)
    _lib.kernel_timing(True)
    try:
        out = model(cb)
        assert out.grad_fn.name() == "ModelPassHIPBackward"
        out.sum().backward()
    finally:
        _lib.kernel_timing(False)
    read = {n: _lib.read_kernel_timing(n) for n in names}
    assert {n: c for n, (ms, c) in read.items()} == names
    assert all(ms > 0.0 for ms, c in read.values() if c)


# (with |cos| the cosines 0 and 1 are nodes of both series: what is left are errors of the same size, measured at some thousand
# outputs)
@pytest.mark.parametrize("cos_abs,slack", [(0, 1.0), (1, 1.15)])
def test_inference_is_as_close_to_float64_as_training(cos_abs, slack):
    """One layer with large angle weights, its atoms' outputs pooled and read through an identity head."""
    from crystalframer_amd import params, synthetic
    from oracle import cpu_model
    wrong = {"inference": 0.0, "training": 0.0}
    for seed in range(4):
        mp = params.ModelParams(num_layers=1, symm_break_noise=0.0, cos_abs=cos_abs)
        cb = synthetic.make_batch(24, atoms="uniform", atoms_lo=1, atoms_hi=6, len_lo=3.0, len_hi=9.0, ang_lo=65.0, ang_hi=115.0,
                                  seed=seed + 50)
        host = cb

        def change(model):
            at = model.encoder.layers[0].self_attn
            model.mlp[3] = torch.nn.Linear(128, 128).cuda()
            with torch.no_grad():
                for n in (1, 2, 3):
                    getattr(at, f"proj_angle{n}").mul_(8.0)
                at.v_proj_weight.mul_(0.1)
                at.pe_dist_proj.mul_(0.1)
                for i in (0, 3):
                    model.mlp[i].weight.copy_(torch.eye(128))
                    model.mlp[i].bias.zero_()

        model, cb = _model(mp, cb, seed, change)
        at = model.encoder.layers[0].self_attn
        at.frame_sink = []
        with torch.no_grad():
            model(cb)
            frames = [[f.detach().cpu().double() for f in at.frame_sink[0]]]
            at.frame_sink = None
            out = {"inference": model(cb)}
        out["training"] = model(cb).detach()
        sd = {k: v.detach().cpu().double() for k, v in model.state_dict().items()}
        ref = cpu_model.model_forward(sd, host, mp, dtype=torch.float64, frames_per_layer=frames, windows="full")
        for k, o in out.items():
            assert Hh.rel_err(o, ref) < 1e-5
            wrong[k] += float(((o.cpu().double() - ref) ** 2).sum())
    assert wrong["inference"] <= slack ** 2 * wrong["training"], {k: v ** 0.5 for k, v in wrong.items()}


# more layers than a launch's table holds: 32 weight gradients of linear layers, 8 of cores, 24 weight streams, 24 layers' weights
@pytest.mark.parametrize("layers,bins", [(7, 16), (9, 64), (13, 0), (26, 64)])
def test_deep_models(layers, bins):
    from crystalframer_amd import params, synthetic
    kw = dict(value_pe_angle_wscale=1.0, value_pe_dist_coef=1.5, value_pe_angle_coef=6.0) if bins == 16 else {}
    mp = params.ModelParams(num_layers=layers, value_pe_angle_real=bins, symm_break_noise=0.0, **kw)
    cb = synthetic.make_batch(5, atoms="uniform", atoms_lo=1, atoms_hi=5, len_lo=3.0, len_hi=9.0, ang_lo=65.0, ang_hi=115.0,
                              seed=layers)
    model, cb, ((o1, e1, g1), (o2, e2, g2)) = _both(mp, cb)
    assert torch.equal(o1, o2) and Hh.rel_err(e1, e2.double()) < 1e-6 * layers
    for n in g1:                                # (sums over the atoms in other slices: a rounding of 6e-8 per atom at worst)
        assert Hh.rel_err(g1[n], g2[n].double()) < 6e-8 * cb.pos.shape[0], n


def test_passes_of_several_threads_on_one_stream():
    """A thread trains, another predicts, both on the default stream, whose scratch they share."""
    import threading
    from crystalframer_amd import params, synthetic
    kw = dict(atoms="uniform", atoms_lo=1, atoms_hi=12, len_lo=3.0, len_hi=9.0, ang_lo=65.0, ang_hi=115.0)
    mp = params.ModelParams(num_layers=2, symm_break_noise=0.0)
    train, cb = _model(mp, synthetic.make_batch(110, seed=1, **kw), seed=1)
    serve, other = _model(mp, synthetic.make_batch(90, seed=2, **kw), seed=2)
    named = [p for p in train.parameters() if p.requires_grad]
    step = lambda: torch.autograd.grad(train(cb).sum(), named)  # noqa: E731
    want = step()
    with torch.no_grad():
        expected = serve(other)
    seen, stop = [], threading.Event()

    def serving():
        with torch.no_grad():
            while not stop.is_set() and len(seen) < 400:
                seen.append(serve(other))

    thread = threading.Thread(target=serving)
    thread.start()
    got = [step() for _ in range(40)]
    stop.set()
    thread.join()
    assert len(seen) > 0 and all(torch.equal(o, expected) for o in seen)
    for g in got:
        assert all(torch.equal(a, b) for a, b in zip(g, want))


def test_training_after_a_first_pass_in_inference_mode():
    from crystalframer_amd import params, synthetic
    cb = synthetic.make_batch(3, atoms="uniform", atoms_lo=1, atoms_hi=4, len_lo=3.0, len_hi=9.0, ang_lo=65.0, ang_hi=115.0,
                              seed=1)
    model, cb = _model(params.ModelParams(num_layers=2, symm_break_noise=0.0), cb)
    for layer in model.encoder.layers:               # storages of their own, as after loading: stacked again by the next pass
        for p in (layer.self_attn.q_proj_weight, layer.self_attn.k_proj_weight, layer.self_attn.v_proj_weight):
            p.data = p.data.clone()
    with torch.inference_mode():
        first = model(cb)
    out = model(cb)
    assert out.grad_fn.name() == "ModelPassHIPBackward" and Hh.rel_err(out, first.double()) < 1e-6
    out.sum().backward()
    assert all(p.grad is not None for p in model.parameters() if p.requires_grad)


def test_forward_derivatives_are_refused():
    import torch.autograd.forward_ad as fwAD
    from crystalframer_amd import params, synthetic
    cb = synthetic.make_batch(3, atoms="uniform", atoms_lo=1, atoms_hi=4, len_lo=3.0, len_hi=9.0, ang_lo=65.0, ang_hi=115.0,
                              seed=1)
    model, cb = _model(params.ModelParams(num_layers=1, symm_break_noise=0.0), cb)
    with fwAD.dual_level():
        cb.pos = fwAD.make_dual(cb.pos, torch.ones_like(cb.pos))
        cb.x = fwAD.make_dual(cb.x, torch.ones_like(cb.x))
        with pytest.raises((NotImplementedError, RuntimeError)):
            model(cb)


# a tile of 16 rows and its edges; either side of the row counts at which the bridge takes one launch instead of two and 32
# rows per workgroup instead of 16; both widths; one and several chunks of the feed-forward block's inside
@pytest.mark.parametrize("D,F,N", [(128, 128, 17), (128, 384, 1), (128, 384, 1361), (128, 384, 1393), (128, 256, 16351),
                                   (128, 256, 16385), (256, 256, 33), (256, 384, 1377)])
def test_bridge_launch_forms(D, F, N):
    from crystalframer_amd.cuda_funcs import LayerBridgeHIP
    H, c1, lb, c2 = D // 16, 0.2, 0.5, -0.25
    gen = torch.Generator().manual_seed(N)
    mk = lambda *s: torch.randn(*s, generator=gen, dtype=torch.float64) * s[-1] ** -0.5
    t64 = dict(attn=mk(N, D), x=mk(N, D), Wo=mk(D, D), bo=mk(D), W1=mk(F, D), b1=mk(F), W2=mk(D, F), b2=mk(D), b=mk(3 * D),
               lw=mk(D), Wq=mk(D, D), Wk=mk(D, D), Wv=mk(D, D))
    t32 = {n: t.float().cuda().requires_grad_(True) for n, t in t64.items()}
    for t in t64.values():
        t.requires_grad_(True)
    lin = torch.nn.functional.linear
    x1 = t64["x"] + lin(t64["attn"], t64["Wo"], t64["bo"])
    z = lin(x1, t64["W1"], t64["b1"])
    x2 = x1 + lin(torch.relu(z), t64["W2"], t64["b2"])
    q, k, v = lin(x2, torch.cat([t64["Wq"], t64["Wk"], t64["Wv"]]), t64["b"]).split(D, 1)
    alpha = (q * t64["lw"]).view(N, H, 16).sum(-1)
    ref = (x2, q * 0.25, k, v, ((1.0 - lb) * torch.nn.functional.elu(alpha * c1) + 1.0) * c2)
    steady = (z.detach().abs().amin(1, keepdim=True) > 3e-6).double()         # no rectifier may round to the other side
    g = [torch.randn(o.shape, generator=gen, dtype=torch.float64) * steady for o in ref]
    sum((o * gi).sum() for o, gi in zip(ref, g)).backward()
    p = t32
    out = LayerBridgeHIP.apply(p["attn"], p["x"], p["Wo"], p["bo"], p["W1"], p["b1"], p["W2"], p["b2"], None, p["b"], p["lw"], None,
                               H, c1, lb, c2, 0.25, p["Wq"], p["Wk"], p["Wv"])
    for o, r in zip(out, ref):
        assert Hh.rel_err(o.reshape(r.shape), r.detach()) < 2e-6
    torch.autograd.backward(out, [gi.float().cuda().view(o.shape) for o, gi in zip(out, g)])
    for n in t64:
        assert Hh.rel_err(p[n].grad, t64[n].grad) < 5e-6, n


# The bridges of inference: a row, a tile of 16 rows and its edges; either side of the row counts where they take one launch
# instead of two (2048 at F = 512, 4096 at F = 256) and 32 rows per workgroup instead of 16 (4096); both widths; one, an odd
# number and more chunks of the feed-forward block's inside than are read at a time; more features than a group of 128.
@pytest.mark.parametrize("D,F,N,feat", [(128, 512, 1, 98), (128, 128, 15, 98), (128, 384, 17, 130), (128, 640, 33, 98),
                                        (128, 512, 2048, 98), (128, 512, 2049, 98), (128, 256, 4096, 98), (128, 512, 4097, 98),
                                        (128, 512, 4129, 200), (256, 512, 31, 98), (256, 512, 2065, 140)])
def test_bridges_of_inference(D, F, N, feat):
    """Against the modules' path (float32 matrix instructions), and, on a part of the atoms, float64."""
    from crystalframer_amd import latticeformer, model_pass, params, synthetic
    from oracle import cpu_model
    mp = params.ModelParams(num_layers=2, symm_break_noise=0.0, value_pe_angle_real=0, model_dim=D, ff_dim=F, head_num=D // 16)
    torch.manual_seed(N)
    sizes = torch.full((N,), 1)
    cb = synthetic.make_batch(N, atoms="uniform", atoms_lo=1, atoms_hi=1, len_lo=3.0, len_hi=6.0, ang_lo=70.0, ang_hi=110.0, seed=N)
    x = torch.zeros(N, feat)
    x[torch.arange(N), torch.arange(N) % feat] = 1.0 + torch.rand(N)
    host = synthetic.CrystalBatch(x, cb.pos, cb.batch, cb.trans_vec, sizes, zero_based=True)
    model = latticeformer.Latticeformer(mp)
    if feat != model.input_embeddings.in_features:
        model.input_embeddings = torch.nn.Linear(feat, D, bias=False)
    model.mlp[0], model.mlp[3] = torch.nn.Linear(D, D), torch.nn.Linear(D, D)
    with torch.no_grad():
        for i in (0, 3):                        # the atoms' outputs, those that the rectifier passes on
            model.mlp[i].weight.copy_(torch.eye(D))
            model.mlp[i].bias.zero_()
    model, cb = model.cuda(), host.to("cuda")
    model.train()
    model(cb)
    model.eval()
    out = []
    for on in (True, False):
        model_pass.ENABLED = on
        try:
            with torch.no_grad():
                out.append(model(cb))
        finally:
            model_pass.ENABLED = True
    limit = 2e-6                                # (sums of up to 640 float32 numbers: 640 ** 0.5 * 2 ** -24)
    assert model_pass.covered(model, cb) and not torch.equal(out[0], out[1])
    assert Hh.rel_err(out[0], out[1].double()) < limit
    some = slice(max(0, N - 40), N)
    part = synthetic.CrystalBatch(host.x[some], host.pos[some], torch.arange(N)[some] - max(0, N - 40), host.trans_vec[some], sizes[some],
                                  zero_based=True)
    sd = {k: v.detach().cpu().double() for k, v in model.state_dict().items()}
    ref = cpu_model.model_forward(sd, part, mp, dtype=torch.float64, windows="full")
    assert Hh.rel_err(out[0][some], ref) < limit


def _one_layer_of_atoms(N, D=128, **kw):
    """N crystals of one atom, one layer, distances alone (nothing that the weights behind the core hold reaches a lattice kernel),
    and a head that passes on the atoms' outputs, those that the rectifier lets through."""
    from crystalframer_amd import params, synthetic
    mp = params.ModelParams(num_layers=1, symm_break_noise=0.0, value_pe_angle_real=0, model_dim=D, head_num=D // 16, **kw)
    cb = synthetic.make_batch(N, atoms="uniform", atoms_lo=1, atoms_hi=1, len_lo=3.0, len_hi=6.0, ang_lo=70.0, ang_hi=110.0, seed=N)

    def outputs_of_atoms(model):
        for i in (0, 3):
            model.mlp[i] = torch.nn.Linear(D, D).cuda()
            with torch.no_grad():
                model.mlp[i].weight.copy_(torch.eye(D))
                model.mlp[i].bias.zero_()

    return _model(mp, cb, change=outputs_of_atoms)


# The bridges of inference and of training in their forms: two launches, one, 32 rows per workgroup
@pytest.mark.parametrize("N", [33, 2065, 4129])
@pytest.mark.parametrize("where,value", [("linear1", float("inf")), ("linear1", float("nan")), ("linear2", float("-inf")),
                                         ("linear2", float("nan")), ("out_proj", float("inf"))])
def test_weights_that_are_no_numbers_show(N, where, value):
    """Where a pass that keeps everything gives no finite number, inference gives none either (an infinity may become a NaN there,
    also one that the rectifier takes away in the other)."""
    model, cb = _one_layer_of_atoms(N)
    layer = model.encoder.layers[0]
    with torch.no_grad():
        (layer.self_attn if where == "out_proj" else layer).get_submodule(where).weight[3, 5] = value
    kept = model(cb).detach()
    model.eval()
    with torch.no_grad():
        out = model(cb)
    lost = ~torch.isfinite(kept)
    assert lost.any() and not torch.isfinite(out[lost]).any()
    if value != value and where == "linear1":
        assert lost.all()


@pytest.mark.parametrize("N", [33, 2065, 4129])
def test_largest_weights(N):
    """A weight that rounds to an infinite bfloat16 number, times a feature that makes a product of ordinary size of it."""
    model, cb = _one_layer_of_atoms(N)
    layer = model.encoder.layers[0]
    with torch.no_grad():
        model.input_embeddings.weight[5] = 2.0 ** -126
        layer.self_attn.out_proj.weight[5] = 0.0
        layer.self_attn.out_proj.bias[5] = 0.0
        layer.linear1.weight[:, 5] = 0.0
        layer.linear1.weight[3, 5] = 3.402e38           # (4 of every atom's third inner feature)
    kept = model(cb).detach()
    model.eval()
    with torch.no_grad():
        out = model(cb)
    assert torch.isfinite(kept).all() and Hh.rel_err(out, kept.double()) < 2e-6      # (sums of up to 512 products)


# Two launches, one, 32 rows per workgroup
@pytest.mark.parametrize("N", [33, 2065, 4129])
def test_bridges_of_inference_use_all_bits_of_their_operands(N):
    """Against float64, with weights large enough that every product shows in the output: 4 to 5e-7 in 2-norm with float32 sums, 2.3
    to 2.8e-6 when one operand is the sum of two bfloat16 numbers instead of three (looked at with the oracle)."""
    from crystalframer_amd import synthetic
    from oracle import cpu_model
    model, cb = _one_layer_of_atoms(N)
    names = ["input_embeddings.weight"] + ["encoder.layers.0." + n + ".weight" for n in ("self_attn.out_proj", "linear1", "linear2")]
    names.append("encoder.layers.0.self_attn.v_proj_weight")
    with torch.no_grad():
        for n in names[1:]:
            model.get_parameter(n).mul_(3.0)
        cb.x.copy_(torch.rand(cb.x.shape, generator=torch.Generator().manual_seed(N)) - 0.5)
        model.eval()
        out = model(cb).cpu().double()
    some = slice(N - 33, N)
    one = torch.ones(33, dtype=torch.long)
    part = synthetic.CrystalBatch(cb.x[some].cpu(), cb.pos[some].cpu(), torch.arange(33), cb.trans_vec[some].cpu(), one, zero_based=True)
    sd = {n: t.detach().cpu().double() for n, t in model.state_dict().items()}

    def oracle(sd, x):
        batch = synthetic.CrystalBatch(x, part.pos, part.batch, part.trans_vec, one, zero_based=True)
        return cpu_model.model_forward(sd, batch, model.params, dtype=torch.float64, windows="full")

    def two_parts(t):
        first = t.float().bfloat16().float()
        return first.double() + (t.float() - first).bfloat16().double()

    ref = oracle(sd, part.x)
    off = lambda t: float((t - ref).norm() / ref.norm())  # noqa: E731
    short = [off(oracle({**sd, n: two_parts(sd[n])}, part.x)) for n in names] + [off(oracle(sd, two_parts(part.x).float()))]
    assert min(short) > 2e-6
    assert off(out[some]) < 1e-6


# Inference of few items: the product of an item's histogram with the weights by its own wavefront.  One atom, a few, either side
# of the item counts where a launch of its own makes it for short rows (10 240 with an angle encoding, 16 384 without).
@pytest.mark.parametrize("bins,B,atoms", [(64, 1, 1), (64, 3, 7), (64, 64, 10), (64, 1280, 1), (64, 1281, 1), (16, 1, 1), (16, 24, 8),
                                          (16, 1280, 1), (16, 1281, 1), (0, 1, 1), (0, 24, 8), (0, 2048, 1), (0, 2049, 1)])
def test_products_of_few_items(bins, B, atoms):
    """Against the same pass with everything kept, whose products have a launch of their own: two sums of 720 float32 products
    (of a 64-bin pass: around other nodes, 1.4e-6 of the basis' peak, a few 1e-6 of a layer's output)."""
    from crystalframer_amd import params, synthetic
    kw = dict(value_pe_angle_wscale=1.0, value_pe_dist_coef=1.5, value_pe_angle_coef=6.0) if bins == 16 else {}
    mp = params.ModelParams(num_layers=1, value_pe_angle_real=bins, symm_break_noise=0.0, **kw)
    cb = synthetic.make_batch(B, atoms="uniform", atoms_lo=atoms, atoms_hi=atoms, len_lo=3.0, len_hi=9.0, ang_lo=65.0,
                              ang_hi=115.0, seed=B)
    model, cb = _model(mp, cb)
    model.eval()
    kept = model(cb).detach()
    with torch.no_grad():
        out = model(cb)
    assert Hh.rel_err(out, kept.double()) < 5e-6


# Very few items (up to 768 on 256 compute units): further wavefronts of an item's workgroup make the product.  One atom, rows of
# several groups of eight pairs whose maximum grows, either side of the line, the absolute value of the cosine, sixteen heads.
@pytest.mark.parametrize("bins,B,atoms,width,cos_abs", [(64, 1, 1, 128, 0), (64, 2, 43, 128, 0), (64, 96, 1, 128, 0), (64, 97, 1, 128, 0),
                                                        (16, 1, 1, 128, 1), (16, 12, 8, 128, 0), (64, 3, 16, 256, 1)])
def test_products_by_further_wavefronts_of_an_item(bins, B, atoms, width, cos_abs):
    """Against the same pass with everything kept (tolerance as above), which has a launch of its own for the products."""
    from crystalframer_amd import params, synthetic
    kw = dict(value_pe_angle_wscale=1.0, value_pe_dist_coef=1.5, value_pe_angle_coef=6.0) if bins == 16 else {}
    mp = params.ModelParams(num_layers=2, value_pe_angle_real=bins, symm_break_noise=0.0, model_dim=width, head_num=width // 16,
                            embedding_dim=[width], cos_abs=cos_abs, **kw)
    cb = synthetic.make_batch(B, atoms="uniform", atoms_lo=atoms, atoms_hi=atoms, len_lo=3.0, len_hi=9.0, ang_lo=65.0,
                              ang_hi=115.0, seed=B)
    model, cb = _model(mp, cb)
    model.eval()
    kept = model(cb).detach()
    with torch.no_grad():
        out = model(cb)
        assert torch.equal(model(cb), out)
    assert Hh.rel_err(out, kept.double()) < 1e-5


# Every form of inference counts its terms: with further wavefronts for the product, one launch without, several launches with the
# products in the main kernel, two and four heads per wavefront.
@pytest.mark.parametrize("bins,B,atoms", [(64, 1, 8), (16, 3, 8), (64, 120, 1), (0, 3, 8), (64, 2200, 1), (0, 2100, 1), (0, 5700, 1)])
def test_inference_counts_its_terms(bins, B, atoms):
    """The same pairs as a pass that keeps everything, and its images within 0.1 % (its inputs differ in their last bits, which
    moves an image across the threshold of a pair now and then)."""
    from crystalframer_amd import _lib, params, synthetic
    from crystalframer_amd.cuda_funcs import KernelManager as KM
    kw = dict(value_pe_angle_wscale=1.0, value_pe_dist_coef=1.5, value_pe_angle_coef=6.0) if bins == 16 else {}
    mp = params.ModelParams(num_layers=1, value_pe_angle_real=bins, symm_break_noise=0.0, **kw)
    cb = synthetic.make_batch(B, atoms="uniform", atoms_lo=atoms, atoms_hi=atoms, len_lo=3.0, len_hi=9.0, ang_lo=65.0,
                              ang_hi=115.0, seed=B)
    model, cb = _model(mp, cb)
    model.eval()
    saved, counts = KM.COLLECT_STATS, []
    KM.COLLECT_STATS = True
    try:
        for keep in (True, False):
            _lib.read_stats(torch.device("cuda:0"), reset=True)
            with torch.set_grad_enabled(keep):
                model(cb)
            counts.append(_lib.read_stats(torch.device("cuda:0"), reset=True))
    finally:
        KM.COLLECT_STATS = saved
    kept, lean = counts
    assert lean["fwd_pairs"] == kept["fwd_pairs"] == 8 * B * atoms * atoms
    for name in ("fwd_evaluated", "fwd_in_box", "fwd_visited"):
        assert kept[name] > 0 and abs(lean[name] - kept[name]) <= (1e-3 if name != "fwd_visited" else 0.5) * kept[name], name


# Inference of many items with the angle encoding: the wavefront that completes sixteen items of a head makes their products, but
# for the last items (a fifth, at least 16 384 on 256 compute units).  One atom short of the first 128 atoms whose products are
# made so, exactly those, a last block of one atom and of 127, rows of mixed lengths, sixteen heads.
@pytest.mark.parametrize("bins,B,atoms,width", [(64, 2175, (1, 1), 128), (64, 2176, (1, 1), 128), (16, 2177, (1, 1), 128),
                                                (64, 2303, (1, 1), 128), (64, 4097, (1, 1), 128), (64, 640, (1, 9), 128),
                                                (16, 700, (1, 9), 128), (64, 60, (30, 61), 128), (64, 1425, (1, 1), 256)])
def test_products_by_the_wavefront_that_completes_sixteen_items(bins, B, atoms, width):
    """Against the same pass with everything kept, whose products have a launch of their own (tolerance as above), and bit for bit
    the same from call to call, on other crystals in between."""
    from crystalframer_amd import params, synthetic
    kw = dict(value_pe_angle_wscale=1.0, value_pe_dist_coef=1.5, value_pe_angle_coef=6.0) if bins == 16 else {}
    mp = params.ModelParams(num_layers=1, value_pe_angle_real=bins, symm_break_noise=0.0, model_dim=width, head_num=width // 16,
                            embedding_dim=[width], **kw)
    make = lambda seed: synthetic.make_batch(B, atoms="uniform", atoms_lo=atoms[0], atoms_hi=atoms[1], len_lo=3.0, len_hi=9.0,  # noqa: E731
                                             ang_lo=65.0, ang_hi=115.0, seed=seed)
    model, cb = _model(mp, make(B))
    other = make(B + 1).to("cuda")
    model.eval()
    kept = model(cb).detach()
    with torch.no_grad():
        out = model(cb)
        for _ in range(3):
            model(other)
            assert torch.equal(model(cb), out)
    assert Hh.rel_err(out, kept.double()) < 5e-6


# Inference without the angle encoding: one head of an atom per wavefront up to 16 383 items, two from there on, four from 45 056
# (from 24 576 with rows of more than 64 pairs).  Either side of the lines; rows of one pair, of a whole group of eight, one more, of
# several groups whose maximum grows, of more than 64; sixteen heads; a few cells so small that their box is not the usual one
# (their heads one after the other).
@pytest.mark.parametrize("B,atoms,width,small", [(2048, (1, 1), 128, 0), (5631, (1, 1), 128, 0), (5632, (1, 1), 128, 3), (704, (8, 8), 128, 0),
                                                 (626, (9, 9), 128, 40), (300, (1, 60), 128, 7), (46, (67, 67), 128, 0), (45, (66, 68), 128, 0),
                                                 (1024, (1, 1), 256, 0), (2816, (1, 1), 256, 5)])
def test_heads_of_an_atom_in_one_wavefront(B, atoms, width, small):
    """Against the same pass with everything kept, which takes one item per wavefront: the same operations per item but for images
    lighter than 2^-32 of their pair's heaviest."""
    from crystalframer_amd import params, synthetic
    mp = params.ModelParams(num_layers=1, value_pe_angle_real=0, model_dim=width, head_num=width // 16, embedding_dim=[width])
    cb = synthetic.make_batch(B, atoms="uniform", atoms_lo=atoms[0], atoms_hi=atoms[1], len_lo=4.0, len_hi=9.0, ang_lo=65.0, ang_hi=115.0,
                              seed=B)
    if small:
        cb.trans_vec[torch.randperm(B, generator=torch.Generator().manual_seed(B))[:small]] *= 0.25
    model, cb = _model(mp, cb)
    model.eval()
    kept = model(cb).detach()
    with torch.no_grad():
        out = model(cb)
        assert torch.equal(model(cb), out)
    assert Hh.rel_err(out, kept.double()) < 2e-6


# ... and many such cells: fewer of them than the leading wavefronts (a sixteenth of the items, at least 256), up to one and two for each
# of the resident wavefronts behind (at most 24 per compute unit), and more, which come from their counters; every head of a cell
# listed or only some (atoms differ in their widths); ordinary cells in front and behind.  {crystals: (from atoms, to atoms, narrow)}
@pytest.mark.parametrize("heads,width,parts", [(2, 128, [(2100, 1, 1, False), (20, 1, 2, True)]), (2, 128, [(2050, 1, 1, True)]),
                                               (2, 128, [(1500, 1, 2, True), (300, 1, 6, False), (200, 1, 2, True)]),
                                               (2, 128, [(1100, 2, 2, True)]), (4, 128, [(5700, 1, 1, True)]), (4, 256, [(2817, 1, 1, True)]),
                                               (4, 128, [(900, 1, 3, True), (3000, 1, 3, False), (1, 17, 17, True)]),
                                               (4, 128, [(20, 17, 30, True), (3500, 1, 3, True)])])
def test_many_cells_with_a_box_of_their_own_beside_several_heads_per_wavefront(heads, width, parts):
    """Against the same pass with everything kept (one item per wavefront; tolerance as above), bit for bit the same from call to call
    with other crystals in between, whose histograms lie where a record that nobody took would find its own."""
    from crystalframer_amd import params, synthetic
    mp = params.ModelParams(num_layers=1, value_pe_angle_real=0, model_dim=width, head_num=width // 16, embedding_dim=[width])

    def make(seed):
        cells = [synthetic.make_batch(B, atoms="uniform", atoms_lo=lo, atoms_hi=hi, ang_lo=65.0, ang_hi=115.0, seed=seed + k,
                                      **(dict(len_lo=1.9, len_hi=2.4) if narrow else dict(len_lo=4.0, len_hi=9.0)))
                 for k, (B, lo, hi, narrow) in enumerate(parts)]
        sizes = torch.cat([c.sizes for c in cells])
        return synthetic.CrystalBatch(torch.cat([c.x for c in cells]), torch.cat([c.pos for c in cells]),
                                      torch.repeat_interleave(torch.arange(len(sizes)), sizes), torch.cat([c.trans_vec for c in cells]),
                                      sizes, zero_based=True)
    model, cb = _model(mp, make(1))
    other = make(50).to("cuda")
    items = cb.pos.shape[0] * width // 16
    assert (45056 if heads == 4 else 16384) <= items and (heads == 4 or items < 45056)
    model.eval()
    kept = model(cb).detach()
    with torch.no_grad():
        model(other)
        out = model(cb)
        for _ in range(2):
            model(other)
            assert torch.equal(model(cb), out)
    assert Hh.rel_err(out, kept.double()) < 2e-6


# Either side of the item counts up to which a layer's items take one launch, crystals of as many atoms as the row has pairs.  With
# everything kept: 5120 with an angle encoding (8 atoms), 6144 from 13 atoms on, 4096 from 33, none from 65; 10 240 without (8
# atoms), 5120 from 17 atoms on.  Inference: 10 240 (8, 24 and 40 atoms), 16 384 without an angle encoding for up to 12 atoms, 5120
# from 101 atoms on.  (And counts between them.)
@pytest.mark.parametrize("bins,atoms,B", [(64, 8, 112), (16, 8, 112), (0, 8, 160), (64, 25, 25), (0, 25, 25), (64, 24, 37), (64, 8, 160),
                                          (0, 8, 256), (64, 8, 80), (16, 8, 80), (64, 24, 32), (16, 13, 59), (64, 40, 12), (64, 65, 2),
                                          (0, 65, 2), (0, 24, 53), (64, 24, 53), (64, 40, 32), (0, 12, 170), (0, 13, 98), (64, 101, 6),
                                          (0, 101, 6)])
def test_item_counts_of_one_launch(bins, atoms, B):
    """The crystals of a batch are answered alike in a batch of one more (no frame changes: the same operations per item, sums of
    the layers' rows in other tiles)."""
    from crystalframer_amd import params, synthetic
    kw = dict(value_pe_angle_wscale=1.0, value_pe_dist_coef=1.5, value_pe_angle_coef=6.0) if bins == 16 else {}
    mp = params.ModelParams(num_layers=1, value_pe_angle_real=bins, symm_break_noise=0.0, **kw)
    cb = synthetic.make_batch(B + 1, atoms="uniform", atoms_lo=atoms, atoms_hi=atoms, len_lo=4.0, len_hi=9.0, ang_lo=65.0, ang_hi=115.0,
                              seed=B)
    n = atoms * B
    less = synthetic.CrystalBatch(cb.x[:n], cb.pos[:n], cb.batch[:n], cb.trans_vec[:B], cb.sizes[:B], zero_based=True)
    model, less = _model(mp, less)
    more = cb.to("cuda")
    a, b = model(less), model(more)
    assert Hh.rel_err(b[:B], a.double()) < 1e-6
    with torch.no_grad():
        assert Hh.rel_err(model(more)[:B], model(less).double()) < 2e-6


# One launch per layer (few items) and several; without and with an angle encoding.  The pairs stated end within the last
# crystal's rows, at its first, and within a crystal before.
@pytest.mark.parametrize("bins", [0, 64])
@pytest.mark.parametrize("B,atoms,cut", [(5, 7, 3), (5, 7, 49), (5, 7, 60), (260, 7, 3), (260, 7, 60), (55, 25, 3), (55, 25, 650)])
def test_fewer_pairs_stated_than_there_are(bins, B, atoms, cut):
    """The atoms whose pairs are not all there have none, the status word says so, every read stays inside the arrays, and the
    crystals before are answered as with the right count."""
    from crystalframer_amd import _lib, params, synthetic
    mp = params.ModelParams(num_layers=2, value_pe_angle_real=bins, symm_break_noise=0.0)
    cb = synthetic.make_batch(B, atoms="uniform", atoms_lo=atoms, atoms_hi=atoms, len_lo=4.0, len_hi=9.0, ang_lo=65.0, ang_hi=115.0, seed=B)
    model, cb = _model(mp, cb)
    dev = torch.device("cuda:0")

    def passes():
        _lib.read_status(dev, reset=True)
        model.zero_grad(set_to_none=True)
        out = model(cb)
        assert out.grad_fn.name() == "ModelPassHIPBackward"
        out.sum().backward()
        with torch.no_grad():
            served = model(cb)
        grads = [p.grad for p in model.parameters() if p.grad is not None]
        return out.detach(), served, grads, _lib.read_status(dev, reset=True)

    want, want_served, _, status = passes()
    assert status == 0
    cb.num_pairs -= cut
    out, served, grads, status = passes()
    assert status & 2 == 2
    whole = B - -(-cut // atoms ** 2)
    assert torch.equal(out[:whole], want[:whole]) and torch.equal(served[:whole], want_served[:whole])
    assert torch.isfinite(out).all() and torch.isfinite(served).all() and all(torch.isfinite(t).all() for t in grads)


# Kernels whose own arrays and dynamic LDS together pass 64 KB while the dynamic part alone does not reach 48: the embedding of
# inference (257 to 384 features at a width of 256, and an edge), and the second launch of training's bridge (F = 512)
@pytest.mark.parametrize("feat,F,N", [(256, 128, 5), (257, 128, 5), (384, 256, 40), (385, 128, 17), (98, 512, 33), (300, 512, 600)])
def test_lds_of_a_kernel_and_of_its_launch_together(feat, F, N):
    """Inference against the pass that keeps everything (float32 matrix instructions), sums of up to 512 products."""
    from crystalframer_amd import params, synthetic
    mp = params.ModelParams(num_layers=2, symm_break_noise=0.0, value_pe_angle_real=0, model_dim=256, head_num=16, ff_dim=F)
    cb = synthetic.make_batch(N, atoms="uniform", atoms_lo=1, atoms_hi=1, len_lo=3.0, len_hi=6.0, ang_lo=70.0, ang_hi=110.0, seed=N)
    x = torch.zeros(N, feat)
    x[torch.arange(N), torch.arange(N) % feat] = 1.0
    x[:, -1] = 0.5
    cb = synthetic.CrystalBatch(x, cb.pos, cb.batch, cb.trans_vec, cb.sizes, zero_based=True)

    def wide_input(model):
        model.input_embeddings = torch.nn.Linear(feat, 256, bias=False).cuda()
        for i in (0, 3):
            model.mlp[i] = torch.nn.Linear(256, 256).cuda()

    model, cb = _model(mp, cb, change=wide_input)
    kept = model(cb)
    assert kept.grad_fn.name() == "ModelPassHIPBackward"
    with torch.no_grad():
        served = model(cb)
    assert Hh.rel_err(served, kept.detach().double()) < 2e-6
