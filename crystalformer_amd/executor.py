"""Inference forwards as one native call.

:func:`encode` and :func:`forward` run the encoder -- the latter with pooling and the regression
head behind it -- through ``cf_forward``, which issues every launch from C++.  They serve the plain
case (real space, or for 128-wide blocks half of the heads in reciprocal space; no norm layers, ReLU,
softmax attention, exponents from the query, one value projection per head) without autograd and
return ``None`` for everything else: other options, modules or forwards replaced by a user's own,
parameters worked out from others, blocks that do not agree on their mode, inputs of other shapes,
forward hooks (which must see the intermediate outputs), kernel timing and counting.  The callers
then run the modules one by one, with the same operators.
"""
from __future__ import annotations

import math
from typing import Optional, Tuple

import torch
from torch import Tensor, nn
from torch.nn.modules import module as _torch_module

from . import global_config as config
from . import hip_funcs
from . import lib as _lib
from . import ops
from . import pooling
from .attention import CrystalformerMultiheadAttentionCUDA, fused_exponents_spec
from .encoder import CrystalformerEncoderCUDA, CrystalformerEncoderLayerCUDA, _sizes_on_device
from .latticeformer import Latticeformer, is_plain_head
from .lib import device_guard, stream_handle


# What the staged translations of a forward may take: with adaptive boxes 5024 bytes an atom pair, all at once for 1.7 million
# pairs, in the fixed cube 544.  Where they take more they are staged in slices, by every block; results don't depend on it.  An
# `ops.STAGED_RINGS_MAX_BYTES` below its default bounds these too.
STAGED_UNITS_MAX_BYTES = 8 << 30


def _unit_limit() -> int:
    return STAGED_UNITS_MAX_BYTES if ops.STAGED_RINGS_MAX_BYTES >= 1 << 30 \
        else min(STAGED_UNITS_MAX_BYTES, ops.STAGED_RINGS_MAX_BYTES)


def _hooked(module: nn.Module) -> bool:
    return bool(module._forward_hooks or module._forward_pre_hooks)


def _touched(module: nn.Module, backward: bool = False) -> bool:
    """A forward hook (or, with ``backward``, a hook of any kind) or a forward of its own on the module or one below."""
    if module._forward_hooks or module._forward_pre_hooks or "forward" in module.__dict__ \
            or (backward and (module._backward_hooks or module._backward_pre_hooks)):
        return True
    for child in module._modules.values():
        if child is not None and _touched(child, backward):
            return True
    return False


def _ready(t: Optional[Tensor], numel: int, device_index: int) -> bool:
    """A parameter the kernels can read as it is (absent ones are fine)."""
    return t is None or (t.dtype is torch.float32 and t.get_device() == device_index and t.is_contiguous()
                         and t.numel() == numel)


def _address(t: Optional[Tensor]) -> Optional[int]:
    return None if t is None else t.data_ptr()


def _plain(layer: nn.Module, width: int) -> bool:
    """Whether a layer's classes, modes and options are those of the plain case: what costs little to look at, and
    first, so that a model of another kind hardly pays for being asked."""
    if type(layer) is not CrystalformerEncoderLayerCUDA:
        return False
    mods = layer._modules
    attn, lin1, lin2 = mods["self_attn"], mods["linear1"], mods["linear2"]
    if type(attn) is not CrystalformerMultiheadAttentionCUDA or type(lin1) is not nn.Linear \
            or type(lin2) is not nn.Linear or type(attn._modules.get("out_proj")) is not nn.Linear:
        return False
    if type(mods["norm1"]) is not nn.Identity or type(mods["norm2"]) is not nn.Identity \
            or layer.activation is not torch.nn.functional.relu:
        return False
    P = attn.params
    # (every module has a mode of its own: the attention's decides on its dropout and its statistics)
    if (attn.training and attn.dropout > 0) or any(type(mods[d]) is not nn.Identity and (layer.training or mods[d].training)
                                                   for d in ("dropout", "dropout1", "dropout2")):
        return False
    halves = P.domain == "multihead"               # half of the heads in reciprocal space
    if halves and (P.gauss_lb_real != P.gauss_lb_reci or attn.num_heads % 2 or width != 128 or lin1.out_features != 512
                   or ops.current_live_sizes() is not None):
        return False
    if (P.domain != "real" and not halves) or P.norm_func_mode not in (0, "default") or fused_exponents_spec(P) is None \
            or attn.kdim != width or attn.vdim != width or attn.embed_dim != width:
        return False
    if P.value_pe_dist_real <= 0:                      # (without FUSE_..: the two operators asked for one by one)
        return halves or hip_funcs.KernelManager.FUSE_ENCODING_ATTENTION
    return P.value_pe_condproj == "no" and P.value_pe_headed and P.use_low_memory


def _block(layer: nn.Module, width: int, device_index: int):
    """(``cf_forward_block`` fields, heads, feed-forward width, whether it stores its exponents' statistics) of a
    layer, or None when it is not the plain case."""
    if not _plain(layer, width):
        return None
    mods = layer._modules
    attn, lin1, lin2 = mods["self_attn"], mods["linear1"], mods["linear2"]
    P = attn.params
    spec, halves = fused_exponents_spec(P), P.domain == "multihead"
    H = attn.num_heads
    D = width // H
    bins = max(int(P.value_pe_dist_real), 0)
    own = attn._parameters
    out, w1, w2 = attn._modules["out_proj"]._parameters, lin1._parameters, lin2._parameters
    ff = lin1.out_features
    try:
        tensors = (own["q_proj_weight"], own["k_proj_weight"], own["v_proj_weight"], own["in_proj_bias"],
                   own["lattice_pos_weights"], own["gauss_scale"], own["pe_dist_proj"] if bins > 0 else None,
                   out["weight"], out["bias"], w1["weight"], w1["bias"], w2["weight"], w2["bias"])
    except KeyError:                                       # (worked out from others whenever it is read)
        return None
    sq = width * width
    counts = (sq, sq, sq, 3 * width, width, 2, H * D * bins, sq, width, width * ff, ff, width * ff, width)
    if bins > 0 and tensors[6] is None:
        return None
    for t, n in zip(tensors, counts):
        if not _ready(t, n, device_index):
            return None
    dist_max = P.value_pe_dist_max
    if dist_max < 0:
        dist_max = (-dist_max) * P.scale_real
    cutoff = P.adaptive_cutoff_sigma
    if cutoff > 0:
        cutoff = P.scale_real * P.gauss_lb_real ** (-0.5) * cutoff
    fields = [_address(t) for t in tensors]
    fields += [bins, int(bool(P.normalize_gauss)), ops.POSITIVE_FUNCS[spec[0]], dist_max, P.value_pe_width_scale,
               cutoff, -0.5 * P.gauss_lb_real * P.scale_real ** -2 * (1 - 1e-5), -0.5 * P.scale_real ** -2,
               P.gauss_lb_real, spec[1], 1.0 / math.sqrt(D), -0.5 * P.scale_reci ** 2 if halves else 0.0]
    return fields, H, ff, attn.training and bool(P.normalize_gauss)


def pack_for_training(encoder: nn.Module, src: Tensor) -> Optional["ops.PackedBlocks"]:
    """The blocks' weights packed for the one-launch row kernels if every block of a fused training step is one
    they serve (the plain case of this module, 128 wide with 512 hidden units, real domain) and nobody looks into
    the blocks; else None: the blocks then run their operators one by one."""
    if not (hip_funcs.USE_LINEAR_FUNCTION and torch.is_grad_enabled()) or type(src) is not Tensor or src.dim() != 2 \
            or config.REPRODUCIBLITY_STATE < 2 or encoder.d_model != 128 or ops.current_live_sizes() is not None \
            or not _ready(src, src.shape[0] * 128, src.get_device()) or src.get_device() < 0 or src.shape[0] == 0 \
            or _torch_module._global_forward_hooks or _torch_module._global_forward_pre_hooks \
            or _torch_module._global_backward_hooks or _torch_module._global_backward_pre_hooks:
        return None
    blocks, settings = [], []
    for layer in encoder._modules["layers"]._modules.values():
        mods = layer._modules
        if _touched(layer, backward=True):
            return None
        got = _block(layer, 128, src.get_device())
        if got is None or got[2] != 512 or layer.self_attn.params.domain != "real" or 128 // got[1] % 4:
            return None
        attn = mods["self_attn"]
        blocks.append((attn.out_proj.weight, mods["linear1"].weight, mods["linear2"].weight, attn.q_proj_weight,
                       attn.k_proj_weight, attn.v_proj_weight))
        settings.append((got[0], got[1], attn.training))
    if not blocks:
        return None
    pack = ops.PackedBlocks(blocks)
    pack.settings = settings
    return pack


def native_training(encoder: nn.Module, src: Tensor, pack: "ops.PackedBlocks", layout, rpos: Tensor, tvecs: Tensor,
                    rvlen: Tensor):
    """The blocks of a fused training step as one call each way (:class:`hip_funcs.BlockTrainHIP`), in the order of the
    layers, or None where the operators run one by one: under instrumentation, without a pair list, with operands that the
    operators convert or refuse (a row too many or too few among them), or with an encoding other than the one the call
    has."""
    if ops.instrumented() or layout.pairs is None or layout.num_edges == 0 or src.shape[0] != layout.num_atoms \
            or not hip_funcs.KernelManager.DENSE_EDGE_BLOCKS:
        return None
    index, B = layout.batch.get_device(), tvecs.shape[0]
    if not _ready(rpos, 3 * layout.num_edges, index) or not _ready(tvecs, 9 * B, index) or not _ready(rvlen, 3 * B, index) \
            or tvecs.dim() != 3 or layout.atom_start.numel() != B + 1:
        return None
    shared = hip_funcs.TrainGeometry(pack, layout, rpos, tvecs, rvlen)
    blocks = []
    for i, (layer, (fields, heads, training)) in enumerate(zip(encoder.layers, pack.settings)):
        attn = layer.self_attn
        if not attn.params.use_low_memory or "encode_and_attend" in attn.__dict__ or "exponent_settings" in attn.__dict__:
            return None
        blocks.append(hip_funcs.TrainBlock(shared, i, fields, heads, training))
    return blocks


def _head(mlp: nn.Module, width: int, device_index: int) -> Optional[Tuple[tuple, int, int]]:
    """((w_head, b_head, w_last, b_last), hidden, targets) of a head ``Linear, ReLU, Linear`` or ``Linear``
    (identities in between do not count), else None."""
    mods = [m for m in mlp._modules.values() if type(m) is not nn.Identity]
    kinds = [type(m) for m in mods]
    if any(t is nn.Linear and not m._parameters.keys() >= {"weight", "bias"} for t, m in zip(kinds, mods)):
        return None                                        # (as in _block)
    if kinds == [nn.Linear, nn.ReLU, nn.Linear]:
        first, last = mods[0]._parameters, mods[2]._parameters
        hidden = mods[0].out_features
        if hidden % 16 or mods[2].in_features != hidden \
                or not _ready(first["weight"], hidden * width, device_index) \
                or not _ready(first["bias"], hidden, device_index):
            return None
        head = (first["weight"], first["bias"])
    elif kinds == [nn.Linear]:
        last, hidden, head = mods[0]._parameters, 0, (None, None)
    else:
        return None
    targets = mods[-1].out_features
    if not _ready(last["weight"], targets * (hidden or width), device_index) \
            or not _ready(last["bias"], targets, device_index):
        return None
    return head + (last["weight"], last["bias"]), hidden, targets


def _embeds(model: nn.Module, x: Tensor):
    """Whether the native call can embed the atoms itself: a plain, unhooked projection of contiguous rows into
    the one block width that has the kernel, without autocast (which would run it in another type)."""
    embed = model._modules.get("input_embeddings")
    layers = model._modules["encoder"]._modules["layers"]
    return (type(embed) is nn.Linear and not _hooked(embed) and embed.out_features == 128 and len(layers) > 0
            and getattr(layers[0], "linear1", None) is not None and layers[0].linear1.out_features == 512
            and type(x) is Tensor and x.dim() == 2 and x.shape[1] == embed.in_features <= 128
            and not torch.is_autocast_enabled("cuda") and x.get_device() >= 0
            and _ready(x, x.numel(), x.get_device())
            and _ready(embed.weight, embed.in_features * 128, x.get_device())
            and _ready(embed.bias, 128, x.get_device()))


def _blocks(encoder: nn.Module, device_index: int):
    """(fields of all blocks, heads, feed-forward width, whether they store statistics) or None."""
    if torch.is_grad_enabled() or config.REPRODUCIBLITY_STATE < 2 or not hip_funcs.KernelManager.DENSE_EDGE_BLOCKS \
            or ops.instrumented() or encoder._modules.get("norm") is not None:
        return None
    blocks, common = [], None
    for layer in encoder._modules["layers"]._modules.values():
        got = _block(layer, encoder.d_model, device_index)
        if got is None or (blocks and got[1:] != common):
            return None                                # (one setting for all blocks: some frozen, some not)
        blocks.append(got[0])
        common = got[1:]
    if not blocks or _torch_module._global_forward_hooks or _torch_module._global_forward_pre_hooks or _touched(encoder):
        return None
    return (blocks, *common)


def _run(encoder: nn.Module, src: Tensor, pos: Tensor, batch: Tensor, trans: Tensor, sizes: Tensor,
         blocks, head=None, embed: Optional[nn.Module] = None) -> Optional[Tensor]:
    """``blocks`` from :func:`_blocks`, ``head`` from :func:`_head`; ``embed`` where ``src`` is still to be embedded."""
    if blocks is None:
        return None
    blocks, H, ff, store = blocks
    KM = hip_funcs.KernelManager
    width = encoder.d_model
    index = src.get_device()
    if index < 0 or src.dim() != 2 or trans.dim() != 3 or batch.dim() != 1:
        return None
    N, B = src.shape[0], trans.shape[0]
    # (shapes and not counts: what the operators refuse one by one is theirs to refuse)
    if N == 0 or src.shape[1] != (embed.in_features if embed else width) or pos.shape != (N, 3) \
            or trans.shape != (B, 3, 3) or not _ready(src, src.numel(), index) or not _ready(pos, 3 * N, index) \
            or not _ready(trans, 9 * B, index) or batch.get_device() != index or batch.dtype is not torch.int64:
        return None
    dev = src.device
    if not torch.is_tensor(sizes) or sizes.device != dev or sizes.dtype != torch.long:
        sizes = _sizes_on_device(sizes, batch, B, dev)
    layout = ops.batch_layout(sizes, batch)            # index structure: built once per batch
    if layout.pairs is None or layout.num_edges == 0 or layout.num_atoms != N or sizes.numel() > B:
        return None
    tensors, hidden, targets = head if head is not None else ((None,) * 4, 0, 0)
    out = torch.empty((sizes.numel(), targets) if targets else (N, width), dtype=torch.float32, device=dev)
    L = _lib.load()
    sched = ops._scheduling_words(dev) if ops.DYNAMIC_ROUNDS else None
    args = _lib.ForwardArgs(
        N, layout.num_edges, sizes.numel(), len(blocks), H, width, ff, KM.LATTICE_RANGE, KM.MINIMUM_RANGE, 1,
        int(store), int(KM.STAGED_RINGS), int(KM.ADAPTIVE_RINGS), ops.STAGED_RINGS_MAX_BYTES, _unit_limit(), hidden,
        targets, embed.in_features if embed else 0, src.data_ptr(), pos.data_ptr(), trans.data_ptr(),
        layout.batch.data_ptr(), layout.atom_start.data_ptr(), layout.edge_start.data_ptr(), layout.edges.data_ptr(),
        layout.e_start.data_ptr(), layout.pairs.data_ptr(),
        _address(sched), *(_address(t) for t in tensors),
        *((_address(embed.weight), _address(embed.bias)) if embed else (None, None)), out.data_ptr())
    table = (_lib.ForwardBlock * len(blocks))(*(tuple(f) for f in blocks))
    need = L.cf_forward_workspace(_lib.ctypes.byref(args), table)
    if need < 0:
        return None
    ws = torch.empty(need, dtype=torch.uint8, device=dev)
    with device_guard(dev):
        rc = L.cf_forward(_lib.ctypes.byref(args), table, ws.data_ptr(), need, stream_handle(dev))
    if rc == -2:                                       # a shape some kernel does not serve: module by module
        return None
    _lib.check(rc, "cf_forward")
    return out


def encode(encoder: nn.Module, src: Tensor, pos: Tensor, batch: Tensor, trans: Tensor, sizes) -> Optional[Tensor]:
    """The output of ``CrystalformerEncoderCUDA.forward``, or None where it has to run module by module."""
    return _run(encoder, src, pos, batch, trans, sizes, _blocks(encoder, src.get_device()))


def forward(model: nn.Module, data) -> Tuple[Optional[Tensor], Optional[Tensor]]:
    """The output of ``Latticeformer.forward``, or None and the embedded atoms if they are there already."""
    if torch.is_grad_enabled():
        return None, None
    mods = model._modules
    encoder, proj, mlp = mods.get("encoder"), mods.get("proj_before_pooling"), mods.get("mlp")
    # (an encoder of another class computes something else than its layers say)
    if type(encoder) is not CrystalformerEncoderCUDA or "forward" in encoder.__dict__:
        return None, None
    if type(proj) is not nn.Identity or model.pooling_layer is not pooling.avr_pool \
            or _hooked(proj) or not is_plain_head(mlp) \
            or type(model)._head is not Latticeformer._head or "_head" in model.__dict__:
        return None, None
    x = data.x
    blocks = _blocks(encoder, x.get_device())
    if blocks is None or _touched(mlp):
        return None, None
    head = _head(mlp, encoder.d_model, x.get_device())
    if head is None:
        return None, None
    where = data.pos, data.batch, data.trans_vec, data.sizes, blocks, head
    if _embeds(model, x):
        return _run(encoder, x, *where, mods["input_embeddings"]), None
    x = hip_funcs.linear(x, model.input_embeddings.weight, model.input_embeddings.bias)
    return _run(encoder, x, *where), x
