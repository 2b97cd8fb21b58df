"""The work this framework is measured on, through its public entry points.

A case is one way of calling the library on one kind of batch:

* ``predict``    an eager forward pass, ``model(batch)`` without autograd;
* ``replay``     the forward of a known layout replayed from a HIP graph (``GraphedForward``) on new data;
* ``inflight``   four such graphs on four streams, as a throughput loop keeps them;
* ``serve``      one capacity graph taking batches whose crystal sizes it was not captured with;
* ``train``      a whole training step replayed from a graph (``GraphedTrainStep``);
* ``fit``        the same step launched eagerly (``fused_training_step``);
* ``operators``  the drop-in operator boundary: geometry, periodic encoding, attention and mean as
                 autograd Functions, forward and backward.

Batches are synthetic crystals of the benchmark's distributions (``crystalformer_amd.synthetic``); every
model is the default 128-wide, 8-head architecture with the number of blocks, value bins, domain and
translation rule that the case names, and carries stored exponent statistics as a trained one does.
"""
import math

import torch

from crystalformer_amd import hip_funcs, ops, synthetic
from crystalformer_amd.encoder import compute_lattice_distances_for_cuda
from crystalformer_amd.graphs import GraphedForward, GraphedTrainStep
from crystalformer_amd.latticeformer import Latticeformer, default_params
from crystalformer_amd.training import FusedAdamW, fused_training_step

HEADS, HEAD_DIM, WIDTH, FF, SPECIES = 8, 16, 128, 512, 98
TRANSLATIONS = 125          # the cube of lattice range 2
IN_FLIGHT = 4

# cells: (lattice lengths, angles, long first axis or none), as in the benchmark's workloads
CELLS = {"small": ((3.0, 12.0), (70.0, 110.0), None),
         "usual": ((3.0, 15.0), (60.0, 120.0), None),
         "skewed": ((4.0, 8.0), (50.0, 130.0), (20.0, 40.0))}


def case(name, kind, crystals, lo, hi, spread="log", cells="usual", blocks=4, bins=64, r0=1.4, domain="real",
         adaptive=True):
    """``spread``: sizes log-uniform or uniform over [lo, hi]; ``r0`` 0 stands for the widening scales
    1.4 ... 3.0 of the seven-block model; ``adaptive`` the per-head boxes (the default) or the fixed cube."""
    c = dict(kind=kind, crystals=crystals, lo=lo, hi=hi, spread=spread, cells=cells, blocks=blocks, bins=bins, r0=r0,
             domain=domain, adaptive=adaptive)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one structure at a time, as an interactive prediction asks for it
        case("predict_one", "predict", 1, 12, 12),
        # the simplified model (no value encoding) on a small batch of small crystals
        case("predict_simplified_b32", "predict", 32, 1, 16, spread="uniform", cells="small", bins=0),
        # the default model on a batch never seen before, and at the default settings throughout
        case("predict_default_b128", "predict", 128, 1, 64),
        # the headline benchmark, one batch at a time and with several batches in flight
        case("replay_default_b128", "replay", 128, 1, 64, adaptive=False),
        case("inflight_default_b128", "inflight", 128, 1, 64, adaptive=False),
        # a server with one graph for whatever arrives
        case("serve_default_b128", "serve", 128, 1, 64),
        # half of the heads in reciprocal space
        case("replay_multihead_b96", "replay", 96, 1, 64, domain="multihead", adaptive=False),
        # the deep model on a large batch
        case("replay_7block_b256", "replay", 256, 1, 96, blocks=7, r0=0),
        # large skewed cells: the largest forward
        case("predict_stress_b16", "predict", 16, 200, 444, spread="uniform", cells="skewed", r0=3.0),
        # training: the benchmark's step from a graph, and an epoch's step on an ever new batch
        case("train_default_b128", "train", 128, 1, 64, adaptive=False),
        case("fit_default_b61", "fit", 61, 1, 64),
        # the operators inside someone else's model, crystals up to the reference's limit of 320 atoms
        case("operators_b8", "operators", 8, 150, 320, spread="uniform", cells="skewed", r0=2.0, adaptive=False),
    ]


def draw(rng):
    """One more case: any kind, the sizes spread over the logarithm of their range, odd ones among them."""
    def log_int(a, b):
        return max(a, min(b, int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))))

    kind = rng.choice(["predict", "predict", "replay", "inflight", "serve", "train", "fit", "operators"])
    training = kind in ("train", "fit", "operators")        # (a gradient needs more than one-atom crystals)
    crystals = log_int(4 if training else 1, 256)
    # (at most a million edges of log-uniform or uniform sizes: below the largest listed case)
    hi = log_int(16 if training else 4, max(16, min(444, int(math.sqrt(1.5e6 / crystals)))))
    spread = rng.choice(["log", "uniform"])
    lo = 1 if spread == "log" else log_int(1, hi)
    if spread == "uniform" and crystals * hi * hi > 1.0e6:
        hi = max(2, int(math.sqrt(1.0e6 / crystals)))
        lo = min(lo, hi)
    if kind in ("train", "fit", "inflight", "operators"):   # several passes' worth of work in one
        hi = max(2, min(hi, int(math.sqrt(4.0e5 / crystals))))
        lo = min(lo, hi)
    if kind == "serve":                                     # (capacity for crystals that are all of the largest size)
        hi = max(2, min(hi, int(math.sqrt(1.0e6 / crystals))))
        lo = min(lo, hi)
    cells = "skewed" if hi >= 128 else rng.choice(["small", "usual"])
    domain = "multihead" if kind in ("predict", "replay") and rng.random() < 0.15 else "real"
    bins = 64 if domain == "multihead" or kind == "operators" else rng.choice([64, 64, 64, 32, 0])
    blocks = rng.choice([4, 4, 4, 7]) if kind in ("predict", "replay", "serve") else 4
    r0 = 0 if blocks == 7 else rng.choice([1.4, 1.4, 2.0, 3.0])
    return case(None, kind, crystals, lo, hi, spread, cells, blocks, bins, r0, domain, rng.random() < 0.5)


def _batch(c, seed, with_targets=False):
    lengths, angles, long_axis = CELLS[c["cells"]]
    return synthetic.make_batch(c["crystals"], (c["lo"], c["hi"]), c["spread"] == "log", lengths, angles, seed=seed,
                                long_axis=long_axis, with_targets=with_targets).to("cuda")


def _scales(c):
    return [1.4, 1.4, 2.0, 2.0, 3.0, 3.0, 3.0] if c["r0"] == 0 else [c["r0"]]


def _model(c, seed):
    torch.manual_seed(seed)
    over = {} if c["adaptive"] else {"adaptive_cutoff_sigma": 0.0}
    return Latticeformer(default_params(num_layers=c["blocks"], value_pe_dist_real=c["bins"], scale_real=_scales(c),
                                        domain=c["domain"], **over)).to("cuda")


def _trained(c, seed, batch):
    """A model as training leaves it: features of order one (the initialisation's are near zero, and the
    head's bias would be all of the output) and the exponents' statistics of a batch stored in it."""
    model = _model(c, seed).train()
    with torch.no_grad():
        model.input_embeddings.weight.normal_()
        model(batch)
    return model.eval()


def prepare(c, seed):
    kind = c["kind"]
    s = {"kind": kind}
    if kind in ("train", "fit"):
        s["batch"] = _batch(c, seed, with_targets=True)
        s["model"] = _model(c, seed).train()
        if kind == "train":
            s["step"] = GraphedTrainStep(s["model"], s["batch"])
            s["batch"] = _relabelled(s["batch"], seed)
        else:
            s["opt"] = FusedAdamW(s["model"])
        s["params"] = [p for p in s["model"].parameters() if p.requires_grad]
    elif kind == "operators":
        # (its outputs are per atom: the crystal sizes are the case's, all else the seed's)
        b = _batch(c, 1000 * c["crystals"] + c["hi"])
        g = torch.Generator(device="cuda").manual_seed(seed)
        frac = torch.rand(b.pos.shape, device="cuda", generator=g)
        pos = (frac[:, None, :] @ b.trans_vec[b.batch]).squeeze(1).contiguous()
        batch = s["batch"] = synthetic.CrystalBatch(b.x, pos, b.batch, b.trans_vec, b.sizes)
        N = batch.pos.shape[0]

        def randn(*shape, scale=1.0):
            return torch.randn(*shape, device="cuda", generator=g) * scale
        hip_funcs.compile_kernels(2, HEADS, HEAD_DIM, c["bins"], HEAD_DIM, True)
        rho = 0.5 + torch.rand(N, HEADS, device="cuda", generator=g)          # around one, as normalised exponents are
        s["a"] = (-0.5 * rho / c["r0"] ** 2).requires_grad_()
        s["q"] = randn(N, HEADS, HEAD_DIM, scale=HEAD_DIM ** -0.5).requires_grad_()
        s["k"] = randn(N, HEADS, HEAD_DIM).requires_grad_()
        s["v"] = randn(N, HEADS, HEAD_DIM).requires_grad_()
        s["W"] = randn(1, HEADS, HEAD_DIM, c["bins"], scale=c["bins"] ** -0.5).requires_grad_()
        s["g"] = randn(c["crystals"], HEADS, HEAD_DIM)
        s["bins"], s["dist_max"] = c["bins"], 10.0 * c["r0"]
        s["cutoff"] = -3.5 if c["adaptive"] else 0.0
    else:
        batch = _batch(c, seed)
        model = s["model"] = _trained(c, seed, batch)
        if kind == "predict":
            s["batch"] = batch
        elif kind == "replay":
            s["graph"], s["batch"] = GraphedForward(model, batch), _relabelled(batch, seed)
        elif kind == "inflight":
            s["streams"] = [torch.cuda.Stream() for _ in range(IN_FLIGHT)]
            s["graphs"] = [GraphedForward(model, batch, launch_share=0.75) for _ in range(IN_FLIGHT)]
            s["batches"] = [_relabelled(batch, seed + i) for i in range(IN_FLIGHT)]
        else:
            B, top = c["crystals"], c["hi"]
            s["graph"] = GraphedForward(model, batch, capacity=(B, B * top, B * top * top))
            s["batch"] = _batch(c, seed + 7919)              # other crystal sizes than the graph was captured with
    return s


def _relabelled(batch, seed):
    """Another data set for the same layout: the species change places, the positions move a little."""
    g = torch.Generator(device="cuda").manual_seed(seed + 104729)
    order = torch.randperm(batch.x.shape[0], device="cuda", generator=g)
    pos = batch.pos + 0.1 * torch.randn(batch.pos.shape, device="cuda", generator=g)
    return synthetic.CrystalBatch(batch.x[order], pos, batch.batch, batch.trans_vec, batch.sizes, batch.y)


def run(s):
    kind = s["kind"]
    if kind == "predict":
        with torch.no_grad():
            return s["model"](s["batch"])
    if kind in ("replay", "serve"):
        return s["graph"](s["batch"])
    if kind == "inflight":
        here = torch.cuda.current_stream()
        out = []
        for stream, graph, batch in zip(s["streams"], s["graphs"], s["batches"]):
            stream.wait_stream(here)
            with torch.cuda.stream(stream):
                out.append(graph(batch))
        for stream in s["streams"]:
            here.wait_stream(stream)
        return out
    if kind == "train":
        loss = s["step"](s["batch"])
        return [loss] + [p.grad for p in s["params"]]
    if kind == "fit":
        loss = fused_training_step(s["model"], s["batch"], s["opt"])
        return [loss] + [p.grad for p in s["params"]]
    b = s["batch"]
    rpos, _, _, rvecs, _, edges = compute_lattice_distances_for_cuda(b.pos, b.batch, b.trans_vec, b.sizes, 2)
    adaptive = (torch.norm(rvecs, 2, dim=-1), s["cutoff"]) if s["cutoff"] else (None, None)
    bias, values = hip_funcs.RealPeriodicEncodingWithProjFuncCUDA.apply(
        s["a"], rpos, None, b.trans_vec, b.batch, edges, s["bins"], s["dist_max"], 1.0, s["W"], *adaptive)
    out = hip_funcs.FusedDotProductAttentionCUDA.apply(s["q"], s["k"], s["v"], bias, values, b.batch, edges)
    pooled = hip_funcs.IrregularMeanCUDA.apply(out, b.batch, b.sizes)
    grads = torch.autograd.grad(pooled, [s["a"], s["q"], s["k"], s["v"], s["W"]], s["g"])
    return [pooled.detach(), out.detach(), *grads]


def _counts(c):
    """Expected atoms and edges of the case's batch."""
    lo, hi = c["lo"], c["hi"]
    if c["spread"] == "uniform":
        n = (lo + hi) / 2
        n2 = n * n + ((hi - lo + 1) ** 2 - 1) / 12
    else:                                    # floor of a log-uniform draw over [lo, hi + 1)
        span = math.log((hi + 1) / lo)
        w = [math.log((k + 1) / k) / span for k in range(lo, hi + 1)]
        n = sum(k * p for k, p in zip(range(lo, hi + 1), w))
        n2 = sum(k * k * p for k, p in zip(range(lo, hi + 1), w))
    return c["crystals"] * n, c["crystals"] * n2


def work(c):
    """Per edge and block: half of an atom pair's 125 distances and their weights for 16 (atom, head) columns,
    16 Gaussians of the half of the translations that reach a bin, their products with the weights, and the
    projection of the bins to the head's width; per atom and block the dense layers.  Bytes: batch, weights
    and outputs once (an operator's inputs, outputs and gradients where those are what the call takes)."""
    N, E = _counts(c)
    K = c["bins"]
    enc = TRANSLATIONS / 2 * (23 + 16 * 4)
    if K:
        enc += TRANSLATIONS / 4 * 16 * (3 + 2 * 16) + 2 * HEADS * HEAD_DIM * K
    att = 4 * HEADS * HEAD_DIM + 8 * HEADS
    dense = 2 * (4 * WIDTH * WIDTH + 2 * WIDTH * FF)
    if c["kind"] == "operators":
        # the gradient of the mean spreads over all atoms; encoding twice for its gradients, attention likewise
        return {"bytes": 4 * (2 * 5 * N * HEADS * HEAD_DIM + 2 * N * HEADS + 6 * N + 2 * 3 * E),
                "flops": 3 * E * (enc + att)}
    per_pass = 3 if c["kind"] in ("train", "fit") else IN_FLIGHT if c["kind"] == "inflight" else 1
    weights = 4 * (c["blocks"] * (4 * WIDTH * WIDTH + 2 * WIDTH * FF + WIDTH * K) + SPECIES * WIDTH + WIDTH * WIDTH)
    batch = 4 * (SPECIES + 3) * N + (36 + 8) * c["crystals"] + 8 * N
    moved = weights * (7 if c["kind"] in ("train", "fit") else 1) + batch * (IN_FLIGHT if c["kind"] == "inflight" else 1)
    return {"bytes": moved + 4 * c["crystals"],
            "flops": per_pass * (c["blocks"] * (E * (enc + att) + N * dense) + 2 * SPECIES * WIDTH * N)}


def tolerance(c):
    """Four times the largest difference seen when every crystal's atoms, and with them the sums, are put in
    another order (worst of the listed and twenty drawn cases): 6.5e-7 for a model's output, 7e-7 for an
    operator's gradient.  The gradients of a training step go through some 10^6 ReLU kinks, and through
    optimiser steps that divide by a gradient's own size: there 2.4e-3 of a tensor, 0.13 of an entry."""
    if c["kind"] in ("train", "fit"):
        return {"rel": 1e-2, "max": 0.5}
    return {"rel": 3e-6, "max": 4e-5}
