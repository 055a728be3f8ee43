"""Cases that stand for what the framework is used for, from one crystal to batches of thousands.

    listed()             the cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  inputs and weights on the GPU, as a program that uses the framework holds them
    run(state)           one pass through the public entry points
    work(case)           bytes and flop that the pass cannot do without
    tolerance(case)      how far the results of another correct implementation at this precision may be off

Crystals are synthetic: the cell shapes and atom counts of a case are those of the configurations in
``crystalframer_amd.synthetic`` (or parts of their ranges).  The atom counts of a batch are the quantiles of the
distribution in an order drawn from the seed, so that a case has the same number of atoms and pairs for every seed while
cells, positions, species and the order of the crystals differ.
"""
import math
import random
import statistics

import torch

from crystalframer_amd import cuda_funcs, geometry, latticeformer, optim, params, synthetic
from crystalframer_amd.cuda_funcs import KernelManager

# Kinds of pass:
#   infer      the model in evaluation mode on one batch (screening, serving)
#   train      one training step, launched from Python: every batch of an epoch has shapes of its own
#   replay     the same training step on a fixed batch as one captured HIP graph, replayed
#   gradient   forward and backward of the model without the optimizer
#   operators  the operators of the reference's attention layer one by one, forward and backward: code written against
#              the reference's interface that only swaps the import
# The noise that breaks ties between equally good frame axes is on for the large batches, as it is by default, and off
# for the small ones, as a program that wants the same answer for a crystal every time sets it.
# Families: (atoms per crystal, cell edges in angstrom, cell angles in degrees) of synthetic.CONFIGS.
FAMILY = {
    "molecular": dict(atoms="uniform", lo=1, hi=8, edge=(3.0, 10.0), angle=(70.0, 110.0)),       # C1
    "materials": dict(atoms="lognormal", lo=1, hi=60, edge=(3.0, 12.0), angle=(60.0, 120.0)),    # C2, C3
    "large": dict(atoms="uniform", lo=40, hi=200, edge=(8.0, 20.0), angle=(60.0, 120.0)),        # C4
    "small": dict(atoms="uniform", lo=1, hi=10, edge=(3.0, 8.0), angle=(70.0, 110.0)),           # C5
}
MEDIAN, SIGMA = 8.0, 0.6        # of the log-normal atom counts
D, F, H, DH = 128, 512, 8, 16   # model width, feed-forward width, heads, head width of the default model


NOISE = 1e-5        # the default of the frame search's tie-breaking noise; 0: the first of equal candidates wins


def listed():
    return [
        # one crystal at a time: a relaxation loop or an interactive query; launches and host time are all there is
        dict(name="infer_1", kind="infer", family="materials", crystals=1, layers=4, bins=64, noise=0.0),
        # the small forward pass: one attention layer without the angle encoding on 16 small cells
        dict(name="infer_16_one_layer", kind="infer", family="molecular", crystals=16, layers=1, bins=0, noise=0.0),
        # a serving batch of odd size with cells of 1 to 60 atoms
        dict(name="infer_101", kind="infer", family="materials", crystals=101, layers=4, bins=64, noise=0.0),
        # screening of many small cells, with and without the angle encoding
        dict(name="infer_4096", kind="infer", family="small", crystals=4096, layers=4, bins=64, noise=NOISE),
        dict(name="infer_4096_distance", kind="infer", family="small", crystals=4096, layers=4, bins=0, noise=NOISE),
        # fine-tuning in small odd batches
        dict(name="train_13", kind="train", family="materials", crystals=13, layers=4, bins=64, noise=0.0),
        # the default training batch: full model, the lightweight setting (16 angle bins), and distances only
        dict(name="train_256", kind="train", family="materials", crystals=256, layers=4, bins=64, noise=NOISE),
        dict(name="train_256_light", kind="train", family="materials", crystals=256, layers=4, bins=16, noise=NOISE),
        dict(name="train_97_distance", kind="train", family="materials", crystals=97, layers=4, bins=0, noise=0.0),
        # the same step of the full model as one HIP graph (the benchmark's headline)
        dict(name="replay_256", kind="replay", family="materials", crystals=256, layers=4, bins=64, noise=NOISE),
        # cells of 40 to 200 atoms, one layer, forward and backward
        dict(name="gradient_large_cells", kind="gradient", family="large", crystals=32, layers=1, bins=64, noise=0.0),
        # the reference's operators one after the other at the default training batch
        dict(name="operators_256", kind="operators", family="materials", crystals=256, layers=1, bins=64, noise=NOISE),
    ]


def _spread(rng, lo, hi):
    """A whole number between lo and hi, spread over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["infer", "infer", "train", "train", "replay", "gradient", "operators"])
    bins = rng.choice([64, 64, 16, 0])
    layers = 4
    if kind == "infer":
        family = rng.choice(["molecular", "materials", "small"])
        crystals = _spread(rng, 1, {"molecular": 4096, "materials": 1024, "small": 4096}[family])
        layers = rng.choice([4, 4, 4, 2, 1])
    elif kind in ("train", "replay"):
        family, crystals = "materials", _spread(rng, 4, 256)
    elif kind == "gradient":
        family, crystals, layers = "large", _spread(rng, 2, 32), 1
    else:
        family, crystals, layers, bins = "materials", _spread(rng, 4, 256), 1, 64
    return dict(kind=kind, family=family, crystals=crystals, layers=layers, bins=bins,
                noise=NOISE if crystals >= 128 else 0.0)


# ------------------------------------------------------------------------------------------------ inputs
def _sizes(case):
    """Atoms per crystal: quantiles of the family's distribution."""
    f, B = FAMILY[case["family"]], case["crystals"]
    u = [(i + 0.5) / B for i in range(B)]
    if f["atoms"] == "uniform":
        return [f["lo"] + min(int(x * (f["hi"] - f["lo"] + 1)), f["hi"] - f["lo"]) for x in u]
    norm = statistics.NormalDist()
    return [min(max(round(MEDIAN * math.exp(SIGMA * norm.inv_cdf(x))), f["lo"]), f["hi"]) for x in u]


def _batch(case, seed):
    """The crystals of a case in host memory."""
    f, sizes = FAMILY[case["family"]], _sizes(case)
    random.Random(seed).shuffle(sizes)
    sizes = torch.tensor(sizes)
    gen = torch.Generator().manual_seed(seed)
    B, N = len(sizes), int(sizes.sum())
    cells = []
    while sum(len(c) for c in cells) < B:      # angles that no cell can have are drawn again
        edge = f["edge"][0] + (f["edge"][1] - f["edge"][0]) * torch.rand(B, 3, generator=gen, dtype=torch.float64)
        angle = f["angle"][0] + (f["angle"][1] - f["angle"][0]) * torch.rand(B, 3, generator=gen, dtype=torch.float64)
        lattice, ok = synthetic.lattice_from_parameters(edge, angle)
        cells.append(lattice[ok])
    trans = torch.cat(cells)[:B]
    batch = torch.repeat_interleave(torch.arange(B), sizes)
    frac = torch.rand(N, 3, generator=gen, dtype=torch.float64)
    pos = (frac[:, :, None] * trans[batch]).sum(1)
    x = torch.zeros(N, synthetic.ATOM_FEAT_DIM)
    x[torch.arange(N), torch.randint(1, 95, (N,), generator=gen)] = 1.0
    return synthetic.CrystalBatch(x, pos.float(), batch, trans.float(), sizes, zero_based=True)


def _model_params(case):
    kw = dict(num_layers=case["layers"], value_pe_angle_real=case["bins"], symm_break_noise=case["noise"])
    if case["bins"] == 16:      # the reference's lightweight setting
        kw.update(value_pe_angle_wscale=1.0, value_pe_dist_coef=1.5, value_pe_angle_coef=6.0)
    return params.ModelParams(**kw)


def _model(case, seed, dev):
    torch.manual_seed(seed)
    model = latticeformer.Latticeformer(_model_params(case)).to(dev)
    # the first training-mode pass measures the normalisation of the Gaussian widths and stores it with the weights
    model.train()
    with torch.no_grad():
        model(_batch(dict(family="molecular", crystals=16), 1).to(dev))
    return model


_capture_stream = []


def prepare(case, seed):
    dev = torch.device("cuda")
    # the tie-breaking noise of the frame search: a fixed seed, so that a run can be repeated; training advances a
    # word on the device from step to step
    KernelManager.NOISE_SEED = 20240607
    KernelManager.NOISE_SEED_DEVICE = None
    if case["kind"] == "operators":
        return _prepare_operators(case, seed, dev)
    model = _model(case, seed, dev)
    batch = _batch(case, seed).to(dev)
    state = dict(kind=case["kind"], model=model, batch=batch)
    if case["kind"] == "infer":
        model.eval()
        return state
    gen = torch.Generator().manual_seed(seed + 1)
    state["target"] = torch.randn(case["crystals"], 1, generator=gen).to(dev)
    if case["kind"] in ("train", "replay"):
        KernelManager.NOISE_SEED_DEVICE = state["noise"] = torch.zeros(1, dtype=torch.int64, device=dev)
        state["optimizer"] = optim.AdamW(model.parameters(), lr=5e-4, betas=(0.9, 0.98), weight_decay=1e-5)
    if case["kind"] == "replay":
        if not _capture_stream:
            _capture_stream.append(torch.cuda.Stream())
        side = _capture_stream[0]
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(3):
                _step(state)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"], stream=side):
            state["outputs"] = _step(state)
    return state


def _prepare_operators(case, seed, dev):
    """Operands of one attention layer as its projections leave them: unit-variance keys and values, queries divided by
    sqrt(head width), Gaussian coefficients from the same map as the layer's."""
    P = params.ModelParams()
    cuda_funcs.compile_kernels(P.lattice_range, H, DH, 64, 64, DH, P.minimum_range, P.cos_abs, P.value_pe_dist_wscale,
                               P.value_pe_angle_wscale, P.value_pe_dist_coef, P.value_pe_angle_coef, case["noise"])
    cb = _batch(case, seed)
    N, E = cb.pos.shape[0], cb.num_pairs
    gen = torch.Generator().manual_seed(seed + 1)
    rand = lambda *shape: torch.randn(*shape, generator=gen)  # noqa: E731
    lb, beta, scale = P.gauss_lb_real, P.positive_func_beta, P.scale_real[0]
    a = ((1 - lb) * torch.nn.functional.elu(rand(N, H) * (beta / (1 - lb))) + 1) * (-0.5 * scale ** -2)
    s = dict(kind="operators", q=rand(N, H, DH) / math.sqrt(DH), k=rand(N, H, DH), v=rand(N, H, DH), a=a,
             wd=rand(1, H, DH, 64) * 0.1, w1=rand(1, H, DH, 64) * 0.1, w2=rand(1, H, DH, 64) * 0.1,
             w3=rand(1, H, DH, 64) * 0.1)
    s = {n: t.to(dev).requires_grad_(True) if isinstance(t, torch.Tensor) else t for n, t in s.items()}
    s["gout"] = rand(case["crystals"], H, DH).to(dev)
    cb = cb.to(dev)
    geo = geometry.crystal_geometry(cb.pos, cb.batch, cb.trans_vec, cb.sizes, num_edges=E)
    s.update(cb=cb, edges=geo.edges, rpos=geo.rpos, rvlen=geo.rvlen, dist_max=-P.value_pe_dist_max * scale,
             cutoff=P.adaptive_cutoff_sigma)
    return s


# ------------------------------------------------------------------------------------------------ one pass
def _forward_backward(state):
    out = state["model"](state["batch"])
    torch.nn.functional.mse_loss(out, state["target"]).backward()
    # The predictions and the gradient of every parameter but the two biases of the head: with them the list would have
    # more entries than are kept, and both follow from the predictions and the gradients of the head's weights.
    return [out.detach()] + [p.grad for n, p in state["model"].named_parameters()
                             if p.grad is not None and not (n.startswith("mlp.") and n.endswith(".bias"))]


def _step(state):
    """A training step.  The updated weights are what the next pass on the same state predicts with."""
    state["optimizer"].zero_grad(set_to_none=True)
    out = _forward_backward(state)
    state["optimizer"].step()
    return out


def _operators(s):
    """The calls of the reference's layer: two frame axes, Gram-Schmidt, the lattice sums, softmax attention, and the
    mean over the atoms of a crystal."""
    leaves = [s[n] for n in ("q", "k", "v", "a", "wd", "w1", "w2", "w3")]
    q, k, v, a, wd, w1, w2, w3 = leaves
    cb, edges, rpos = s["cb"], s["edges"], s["rpos"]
    search = (q, k, v, a, rpos, None, cb.trans_vec, cb.batch, edges, 64, s["dist_max"], 1.0)
    f1 = cuda_funcs.ComputeFrame1MaximumMethodCUDA.apply(*search, s["rvlen"], s["cutoff"])
    f2 = cuda_funcs.ComputeFrame2MaximumMethodCUDA.apply(*search, f1, s["rvlen"], s["cutoff"])
    f2 = torch.nn.functional.normalize(f2 - (f1 * f2).sum(-1, keepdim=True) * f1, dim=2)
    f3 = torch.linalg.cross(f1, f2)
    z, psi = cuda_funcs.RealEncodingWithFramedProjFuncCUDA.apply(
        a, rpos, None, cb.trans_vec, cb.batch, edges, 64, s["dist_max"], 1.0, wd, w1, w2, w3, f1, f2, f3, 64, 4.0, 0,
        1.0, 1.0, s["rvlen"], s["cutoff"])
    out = cuda_funcs.FusedDotProductAttentionCUDA.apply(q, k, v, z, psi, cb.batch, edges)
    mean = cuda_funcs.IrregularMeanCUDA.apply(out, cb.batch, cb.sizes)
    return [mean.detach(), z.detach(), *torch.autograd.grad(mean, leaves, s["gout"])]


def run(state):
    kind = state["kind"]
    if kind == "infer":
        with torch.no_grad():
            return state["model"](state["batch"])
    if kind == "operators":
        return _operators(state)
    if kind == "train":
        return _step(state)
    if kind == "replay":
        state["graph"].replay()
        return state["outputs"]
    for p in state["model"].parameters():
        p.grad = None
    return _forward_backward(state)


# ------------------------------------------------------------------------------------------------ what it takes
def _images(case):
    """Lattice images that carry weight, per (pair, head): those within the radius sqrt(2^24's logarithm / a) of about
    8 angstrom at the mean Gaussian width, by the mean density of the family's cells."""
    lo, hi = FAMILY[case["family"]]["edge"]
    per_volume = (math.log(hi / lo) / (hi - lo)) ** 3 / 0.9
    return min(125.0, max(1.0, 4.0 / 3.0 * math.pi * 8.06 ** 3 * per_volume))


def work(case):
    """Each input, weight and gradient once; per lattice image the windowed bases of the reference's formulation (9
    distance bins, 33 bins or the whole 16-bin basis per axis), and the dense layers."""
    sizes = _sizes(case)
    B, N, E, L, bins = len(sizes), sum(sizes), sum(n * n for n in sizes), case["layers"], case["bins"]
    terms = E * H * _images(case) * L
    wide = {64: 33, 16: 16, 0: 0}[bins]
    forward = terms * (29 + 4 * 9 + (87 + 27 + 12 * wide if bins else 0))
    backward = terms * (37 + 6 * 9 + (24 + 18 * wide if bins else 0))
    encoding = H * DH * (64 + 3 * bins)
    crystals = 4 * (N * (98 + 3) + 9 * B) + 8 * (N + B)
    if case["kind"] == "operators":
        operands = 4 * (3 * N * H * DH + N * H + encoding)
        pairs = E * (16 + 12)
        outputs = 4 * (B * H * DH + E * H)
        return dict(bytes=2.0 * operands + pairs + outputs, flops=forward + backward + 6.0 * 2 * E * H * DH * 4)
    weights = 98 * D + L * (4 * D * D + 2 * D * F + encoding + 7 * D + F) + D * D + 2 * D + 1
    dense = 2.0 * (N * (98 * D + L * (4 * D * D + 2 * D * F + encoding)) + B * D * (D + 1))
    if case["kind"] == "infer":
        return dict(bytes=crystals + 4.0 * (weights + B), flops=forward + dense)
    moved = 2 if case["kind"] == "gradient" else 7     # read, gradient; with the update also two moments each way, weight
    return dict(bytes=crystals + 4.0 * (moved * weights + 2 * B), flops=forward + backward + 3 * dense)


def tolerance(case):
    """32-bit arithmetic throughout: 1e-6 in 2-norm without the angle encoding and wherever no frame changes.  A frame
    axis is an arg max over candidates: when the weights change in their last bit, the winner of a near tie changes for a
    few of the (atom, head) items of a large batch, and the sum over a crystal with it.  Measured with weights multiplied by
    1 + 1.2e-7 x: predictions up to 2e-4 (largest difference 6e-3), gradients up to 6e-3 (0.35) with the tie-breaking
    noise, 1.2e-4 (5e-3) for gradients without it."""
    if case["bins"] == 0:
        return {"rel": 1e-5, "max": 5e-4}
    if case["kind"] == "infer":
        return {"rel": 1e-3, "max": 0.03} if case["noise"] > 0 else {"rel": 3e-4, "max": 0.01}
    return {"rel": 0.02, "max": 0.5} if case["noise"] > 0 else {"rel": 2e-3, "max": 0.1}
