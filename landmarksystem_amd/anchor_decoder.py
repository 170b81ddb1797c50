"""MFMA-backed anchor decoder with the reference's module interface.

`FusedAnchorDecoder` takes the constructor keywords of the reference's
`AnchorDecoder` / `FusedAnchorDecoder` (landmark/nerf_components/
model_components/fields/anchor_decoder.py:49-61) and has the same `forward`
signature (:108-120) and 7-tuple result (:239-242), so the reference's
component-swap map (`kernel_fusion_components_convert_map["AnchorDecoder"]`,
landmark/nerf_components/components_convertor/convert_maps.py:40-47) can point
at it.  Parameters keep the reference's names (`mlp_opacity.0.weight`, ...,
`mlp_feature_bank.0.weight`, cf. tests/test_module/test_util/
test_gs_ckpt_transform.py:24-28) so its checkpoints load unchanged.

Supported: the feature bank (`use_feat_bank`), the level input (`add_level`)
and the training-mode by-products (`neural_opacity`, `mask`); not the
appearance embedding (`appearance_dim > 0`: the reference's own branch
concatenates a 1-D integer tensor to the 2-D input, anchor_decoder.py:204-211,
and cannot run as written).  Without gradients all arithmetic runs in the HIP
kernels behind `gs355_decode`: one call enqueues the whole decode and the
number of Gaussians stays on the device; `forward` waits for that one number
(the reference's boolean-mask indexing synchronises at the same place) only to
give its results their exact shapes, `decode_on_device` never waits.

In training mode with gradients enabled and something to differentiate (a
parameter or an input that requires grad: the training loops of
benchmarks/nerf/scaffold_gs and octree_gs), `forward` is one autograd function
whose two directions run in kernels too (`gs355_decode_train` and its backward
call, fp32), reaching the MLPs, the features, the offsets, the scales and the
anchors.  The feature bank in front of it, heads that were changed (another
activation, a hook on one), tensors of other shapes or types, and second
derivatives are evaluated as the module's own statements
(anchor_decoder.py:147-242) in torch operations -- as in the reference, whose
fused decoder is an inference component and whose training runs the torch
module.  The rasterizer behind it differentiates in HIP.
"""
import ctypes as C
import functools
import threading
import weakref
from collections import OrderedDict
from typing import NamedTuple, Optional

import torch
from torch import nn
from torch.nn.modules import module as _module

from . import _lib
from .pipeline import _raw_stream


def _f32c(t: torch.Tensor, device) -> torch.Tensor:
    if t.dtype is torch.float32 and t.device == device and t.is_contiguous():
        return t
    t = t.detach()
    if t.device != device:
        t = t.to(device)
    if t.dtype != torch.float32:
        t = t.float()
    return t.contiguous()


_counts = threading.local()


def _host_counts(dev: torch.device) -> torch.Tensor:
    """Pinned int32[2] where the kernels of one call on `dev` leave their counts: this thread's own.  A call waits for them
    before it returns or raises, so a thread has one such call under way at most; threads that share a decoder, or replicas of one,
    have a buffer each."""
    kept = _counts.__dict__
    counts = kept.get(dev.index)
    if counts is None:
        with torch.inference_mode(False):
            counts = kept[dev.index] = torch.zeros(2, dtype=torch.int32, device="cpu", pin_memory=True)
    return counts


class DeviceDecode(NamedTuple):
    """Result of `decode_on_device`: tensors with room for A * n_offsets Gaussians, of which the first `count[0]`
    are valid.  `counts` (int32[2], on the device) holds the number of Gaussians and of visible anchors."""
    xyz: torch.Tensor
    color: torch.Tensor
    opacity: torch.Tensor
    scaling: torch.Tensor
    rot: torch.Tensor
    counts: torch.Tensor
    neural_opacity: Optional[torch.Tensor]
    mask: Optional[torch.Tensor]
    first_count: Optional[torch.Tensor] = None

    @property
    def count(self) -> torch.Tensor:  # int32[1]: what the rasterizer takes as its device-side Gaussian count
        return self.counts[0:1] if self.first_count is None else self.first_count


class _TallLinear(torch.autograd.Function):
    """y = x W^T + b for x with hundreds of thousands of rows and a few dozen columns (one row per visible anchor).
    Forward and dL/dx are what nn.Linear computes; dL/dW = dy^T x has its long dimension inside the product, which
    the library's matrix multiply runs on a handful of workgroups (0.8 ms each at 500k anchors): here the rows are
    cut into slabs, one small product per slab in a batched multiply, and the slabs' products are added."""

    SLAB = 4096

    @staticmethod
    def forward(ctx, x, weight, bias):
        x = x.contiguous()
        ctx.save_for_backward(x, weight)
        return torch.addmm(bias, x, weight.t())

    @staticmethod
    def backward(ctx, dy):
        x, weight = ctx.saved_tensors
        dy = dy.contiguous()
        dx = dy @ weight if ctx.needs_input_grad[0] else None
        dw = None
        if ctx.needs_input_grad[1]:
            rows, slab = x.shape[0], _TallLinear.SLAB
            whole = rows // slab * slab
            dw = torch.zeros_like(weight)
            if whole:
                dw += torch.bmm(dy[:whole].view(-1, slab, dy.shape[1]).transpose(1, 2),
                                x[:whole].view(-1, slab, x.shape[1])).sum(dim=0)
            if whole < rows:
                dw += dy[whole:].t() @ x[whole:]
        db = dy.sum(dim=0) if ctx.needs_input_grad[2] else None
        return dx, dw, db


def _train_records(decoder, camera_center, visible, level, anchor, feat, offset, scaling, params):
    """The gs355_decoder and gs355_anchors records of a training decode: pointers into these tensors."""
    d = _lib.Decoder()
    d.feat_dim, d.n_offsets = decoder.feat_dim, decoder.n_offsets
    for j in range(3):
        w0, b0, w1, b1 = params[4 * j:4 * j + 4]
        d.in_dim[j] = w0.shape[1]
        d.w0[j], d.b0[j], d.w1[j], d.b1[j] = w0.data_ptr(), b0.data_ptr(), w1.data_ptr(), b1.data_ptr()
    d.add_level = 1 if decoder.add_level else 0
    an = _lib.Anchors()
    an.A = anchor.shape[0]
    an.anchor, an.feat, an.offset, an.scaling = (t.data_ptr() for t in (anchor, feat, offset, scaling))
    an.campos, an.visible_mask = camera_center.data_ptr(), visible.data_ptr()
    an.level = None if level is None else level.data_ptr()
    return d, an


# The number of visible anchors is on the device until the heads are done: up to this many anchors there is room for every
# one of them (63 MB), beyond, the visible ones are counted and waited for first, so that memory follows them (behind a
# level-of-detail mask they may be few).  The second wait is about 5 % of a step at 5k and 60k anchors (952 -> 1004 us,
# 989 -> 1068), 1 % or less from 200k on (1302 -> 1311).
_ROOM_FOR_ALL = 1 << 16


class _TrainBlock:
    """Where things lie in the block that a training decode keeps for its backward pass: the kernels' workspace, the input
    rows with and without the distance, hidden units and pre-activations of the three heads; every part 256-byte aligned.
    `room`: the most rows (visible anchors) that fit."""

    def __init__(self, A, room, n, widths, compact_feat):
        need, scratch = C.c_size_t(), C.c_size_t()
        _lib.check(_lib.load().gs355_decode_train_bytes(A, 0, n, C.byref(need), C.byref(scratch)))
        sizes = [need.value, room * 36 * 4 if 36 in widths else 0, room * 35 * 4 if 35 in widths else 0]
        sizes += [room * 32 * 4] * 3 + [room * n * k * 4 for k in (1, 7, 3)]
        self.workspace_bytes, self.room, self.sizes, self.compact_feat = need.value, room, sizes, compact_feat
        self.offsets, self.total = [], 0
        for size in sizes:
            self.offsets.append(self.total)
            self.total += (size + 255) // 256 * 256

    def rows(self, block, num_visible):
        """The gs355_train_rows record of the block's parts, and the workspace's address."""
        at = [block.data_ptr() + o for o in self.offsets]
        rows = _lib.TrainRows(num_visible, 1 if self.compact_feat else 0, at[1] if self.sizes[1] else None,
                              at[2] if self.sizes[2] else None)
        for j in range(3):
            rows.hidden[j], rows.pre[j] = at[3 + j], at[6 + j]
        return rows, at[0]


class _DecodeTrain(torch.autograd.Function):
    """The training decode (gs355_decode_train) with its whole backward pass in the kernels
    (gs355_decode_train_backward): differentiable with respect to anchors, features, offsets, scales and the heads'
    parameters.  Workspace, input rows, hidden units and pre-activations (968 bytes a row, 1108 with heads of both widths)
    live until the graph is dropped.  Everything that the backward pass reads goes through save_for_backward and its
    pointers are taken there: saved-tensor hooks (save_on_cpu, checkpointing) hand back other tensors than they were given.

    A backward pass that is itself differentiated (create_graph=True) or batched (is_grads_batched=True) takes the module's
    statements from the visible anchors on, with the forward pass's choice of offsets."""

    @staticmethod
    def forward(ctx, decoder, camera_center, visible, level, compact_feat, anchor, feat, offset, scaling, *params):
        dev, A, n = anchor.device, anchor.shape[0], decoder.n_offsets
        lib = _lib.load()
        stream = _raw_stream(dev)
        dec, an = _train_records(decoder, camera_center, visible, level, anchor, feat, offset, scaling, params)
        f = lambda *shape: torch.empty(shape, dtype=torch.float32, device=dev)  # noqa: E731
        counts = _host_counts(dev)  # (pinned: the kernels' stores land there, nothing is copied)
        o = _lib.Decoded()
        o.num_visible = counts.data_ptr() + 4
        o.count = counts.data_ptr()

        def launch(room):
            parts = _TrainBlock(A, room, n, {params[4 * j].shape[1] for j in range(3)}, compact_feat)
            block = torch.empty(parts.total, dtype=torch.uint8, device=dev)
            rows, workspace = parts.rows(block, room)
            return parts, block, rows, workspace, lib.gs355_decode_train(
                C.byref(dec), C.byref(an), C.byref(rows), 0, C.byref(o), workspace, parts.workspace_bytes, _lib.TRAIN_HEADS,
                stream)

        # How many rows there are is only known on the device, but for features out of the bank.
        room = feat.shape[0] if compact_feat else A
        if not compact_feat and A > _ROOM_FOR_ALL:
            first = launch(0)  # (counts the visible anchors)
            torch.cuda.current_stream(dev).synchronize()
            _lib.check(first[-1])
            room = int(counts[1])
        parts, block, rows, workspace, rc = launch(room)
        # Camera, mask and level are not differentiated, and what a caller does to them after this is nothing to the
        # gradients: the camera is copied, the kernels read neither mask nor level going back (the statements do).
        # (All of this while the heads are evaluated.)
        ctx.decoder, ctx.parts, ctx.visible, ctx.level = decoder, parts, visible, level
        ctx.versions = [_version(t) for t in (visible, level)]
        saved = (camera_center.clone(), block, anchor, feat, offset, scaling, *params)
        ctx.save_for_backward(*saved)
        ctx.shapes = [t.shape for t in saved]
        ctx.set_materialize_grads(False)
        torch.cuda.current_stream(dev).synchronize()
        _lib.check(rc)
        G, V = counts.tolist()
        if V > room:
            raise RuntimeError("%d anchors are visible, %d were a moment ago: the mask changed during the call" % (V, room))
        ctx.num_visible = V
        rows.num_visible = V
        out = (f(G, 3), f(G, 3), f(G, 1), f(G, 3), f(G, 4), f(V * n, 1), torch.empty(V * n, dtype=torch.bool, device=dev))
        if G > 0:
            o.xyz, o.color, o.opacity, o.scaling, o.rot = (t.data_ptr() for t in out[:5])
        o.neural_opacity, o.mask = out[5].data_ptr(), out[6].data_ptr()
        _lib.check(lib.gs355_decode_train(C.byref(dec), C.byref(an), C.byref(rows), G, C.byref(o), workspace,
                                          parts.workspace_bytes, _lib.TRAIN_EMIT, stream))
        ctx.mark_non_differentiable(out[6])
        return out

    @staticmethod
    def backward(ctx, *cotangents):
        given = cotangents[:6]  # (the mask has none)
        if torch.is_grad_enabled() or any(g is not None and _batched(g) for g in given):
            return _DecodeTrain._backward_statements(ctx, given)
        saved = ctx.saved_tensors
        device = ctx.visible.get_device()
        if any(t.shape != shape or t.get_device() != device or t.dtype is not (torch.float32 if k != 1 else torch.uint8)
               for k, (t, shape) in enumerate(zip(saved, ctx.shapes))):
            raise RuntimeError("a tensor that the decode's backward pass reads has another shape, type or device than in its "
                               "forward pass (its .data was replaced in between, or a saved-tensor hook changed it)")
        saved = [t if t.is_contiguous() else t.contiguous() for t in saved]
        camera_center, block, anchor, feat, offset, scaling, *params = saved
        # (the block's parts lie at 256-byte boundaries from its start, feature rows are read 16 bytes at a time)
        block, feat = (t if t.data_ptr() % to == 0 else t.clone() for t, to in ((block, 256), (feat, 16)))
        parts = ctx.parts
        dec, an = _train_records(ctx.decoder, camera_center, ctx.visible, ctx.level, anchor, feat, offset, scaling, params)
        rows, workspace = parts.rows(block, ctx.num_visible)
        dev, A, V = anchor.device, anchor.shape[0], rows.num_visible
        lib = _lib.load()
        ptr = lambda t: None if t is None or t.numel() == 0 else t.data_ptr()  # noqa: E731
        given = [None if g is None else g.contiguous() for g in given]
        cot = _lib.DecodeCotangents(*[ptr(g) for g in given])
        # (anchors that were not decoded have no gradient: their rows stay zero)
        new = torch.empty_like if V == A else torch.zeros_like
        wanted = ctx.needs_input_grad[5:]
        grads = [new(t) if w else None for t, w in zip((anchor, feat, offset, scaling), wanted)]
        grads += [torch.empty_like(p) if w else None for p, w in zip(params, wanted[4:])]
        out = _lib.DecodeGradients(*[ptr(t) for t in grads[:4]])
        for j in range(3):
            out.w0[j], out.b0[j], out.w1[j], out.b1[j] = (ptr(t) for t in grads[4 + 4 * j:8 + 4 * j])
        need, scratch_bytes = C.c_size_t(), C.c_size_t()
        _lib.check(lib.gs355_decode_train_bytes(A, V, ctx.decoder.n_offsets, C.byref(need), C.byref(scratch_bytes)))
        scratch = torch.empty(scratch_bytes.value // 4, dtype=torch.float32, device=dev)
        _lib.check(lib.gs355_decode_train_backward(C.byref(dec), C.byref(an), C.byref(rows), workspace,
                                                   parts.workspace_bytes, C.byref(cot), C.byref(out), scratch.data_ptr(),
                                                   scratch.numel() * 4, _raw_stream(dev)))
        return (None, None, None, None, None, *grads)

    @staticmethod
    def _backward_statements(ctx, given):
        camera_center, block, *tensors = ctx.saved_tensors
        visible, level = ctx.visible, ctx.level
        if ctx.versions != [_version(t) for t in (visible, level)]:
            raise RuntimeError("visible_mask or level was modified in place after the decode, and its gradients are to be "
                               "differentiated")
        decoder, parts = ctx.decoder, ctx.parts
        opacities = block[parts.offsets[6]:][:ctx.num_visible * decoder.n_offsets * 4].view(torch.float32)
        with torch.enable_grad():
            # (aliases: features out of the bank depend on the anchors, and that part is not this function's)
            anchor, feat, offset, scaling, *params = tensors = [t.view_as(t) for t in tensors]
            rows = visible.nonzero(as_tuple=True)[0]
            heads = [_Layers(params[4 * j:4 * j + 4], last) for j, last in enumerate((torch.tanh, None, torch.sigmoid))]
            out = decoder._from_rows(camera_center, anchor.index_select(0, rows),
                                     feat if parts.compact_feat else feat.index_select(0, rows),
                                     offset.index_select(0, rows), scaling.index_select(0, rows),
                                     None if level is None else level.reshape(-1, 1).index_select(0, rows), heads,
                                     mixed=parts.compact_feat, mask=opacities > 0.0)
            wanted = [t for t, w in zip(tensors, ctx.needs_input_grad[5:]) if w]
            pairs = [(o, g) for o, g in zip(out, given) if g is not None and o.requires_grad]
        grads = iter(torch.autograd.grad([o for o, _ in pairs], wanted, [g for _, g in pairs], allow_unused=True,
                                         create_graph=torch.is_grad_enabled()) if pairs else [None] * len(wanted))
        return (None, None, None, None, None, *[next(grads) if w else None for w in ctx.needs_input_grad[5:]])


def _batched(t):
    """Whether t stands for a batch of tensors (vmap, is_grads_batched)."""
    return torch._C._functorch.is_legacy_batchedtensor(t) or torch._C._functorch.is_batchedtensor(t)


def _version(t):
    return None if t is None or t.is_inference() else t._version


class _Layers:
    """A head by its parameters: Linear, ReLU, Linear and the activation `last`."""

    def __init__(self, params, last):
        self.params, self.last = params, last

    def __call__(self, x):
        w0, b0, w1, b1 = self.params
        x = torch.addmm(b1, torch.relu(torch.addmm(b0, x, w0.t())), w1.t())
        return x if self.last is None else self.last(x)


def _mlp(seq, x):
    """The Sequential `seq` (Linear, ReLU, Linear[, activation]) with its Linear layers through _TallLinear."""
    for layer in seq:
        x = _TallLinear.apply(x, layer.weight, layer.bias) if isinstance(layer, torch.nn.Linear) else layer(x)
    return x


class FusedAnchorDecoder(nn.Module):
    def __init__(self, use_feat_bank: bool, add_opacity_dist: bool, add_color_dist: bool, add_cov_dist: bool,
                 view_dim: int, feat_dim: int, n_offsets: int, appearance_dim: int = 0, add_level: bool = False,
                 dist2level: str = None):
        super().__init__()
        if appearance_dim > 0:
            raise NotImplementedError("FusedAnchorDecoder does not take an appearance embedding (appearance_dim=0 only)")
        if view_dim != 3 or feat_dim != 32 or not 1 <= n_offsets <= 10:
            raise NotImplementedError("FusedAnchorDecoder needs view_dim=3, feat_dim=32 and 1..10 offsets")
        self.use_feat_bank, self.add_level, self.dist2level = use_feat_bank, add_level, dist2level
        self.add_opacity_dist, self.add_color_dist, self.add_cov_dist = add_opacity_dist, add_color_dist, add_cov_dist
        self.view_dim, self.feat_dim, self.n_offsets, self.appearance_dim = view_dim, feat_dim, n_offsets, appearance_dim
        level_dim = 1 if add_level else 0

        def head(with_dist: bool, outputs: int, last: Optional[nn.Module]):
            layers = [nn.Linear(feat_dim + view_dim + (1 if with_dist else 0) + level_dim, feat_dim), nn.ReLU(True),
                      nn.Linear(feat_dim, outputs)]
            if last is not None:
                layers.append(last)
            return nn.Sequential(*layers)

        if use_feat_bank:
            self.mlp_feature_bank = nn.Sequential(nn.Linear(view_dim + level_dim, feat_dim), nn.ReLU(True),
                                                  nn.Linear(feat_dim, 3), nn.Softmax(dim=1))
        self.mlp_opacity = head(add_opacity_dist, n_offsets, nn.Tanh())
        self.mlp_cov = head(add_cov_dist, 7 * n_offsets, None)
        self.mlp_color = head(add_color_dist, 3 * n_offsets, nn.Sigmoid())
        # device buffers the decoder keeps between calls, one set per stream that decoded recently (frames of
        # different streams may be in flight together): "workspace" of gs355_decode, "block" of reused outputs
        self._per_stream = OrderedDict()
        self._marshalled = None  # (key, gs355_decoder struct, the tensors it points at)
        self._feat_checked = None  # (the last feature tensor, its state, whether fp16 holds it exactly)

    def __getstate__(self):
        """What a copy or a pickle takes along: not the buffers of past calls and the records of pointers into them."""
        return dict(self.__dict__, _per_stream=OrderedDict(), _marshalled=None, _feat_checked=None)

    # ---- marshalling -----------------------------------------------------------------------------------------
    def _decoder_struct(self, device):
        """The gs355_decoder record of the current parameters, rebuilt only when a parameter was replaced, moved or
        modified in place (tensor identity and version), not per call."""
        key = (device,) + tuple((id(p), p._version, p.data_ptr()) for p in self._parameter_list())
        if self._marshalled is not None and self._marshalled[0] == key:
            return self._marshalled[1]
        keep = []
        d = _lib.Decoder()
        d.feat_dim, d.n_offsets = self.feat_dim, self.n_offsets
        fp16_exact = True  # weights that fp16 cannot hold (fp32-trained checkpoints) go in as hi + lo fp16 pairs
        for j, mlp in enumerate((self.mlp_opacity, self.mlp_cov, self.mlp_color)):
            w0, b0, w1, b1 = (_f32c(t, device) for t in (mlp[0].weight, mlp[0].bias, mlp[2].weight, mlp[2].bias))
            keep += [w0, b0, w1, b1]
            fp16_exact = fp16_exact and all(bool(torch.equal(w.half().float(), w)) for w in (w0, w1))
            d.in_dim[j] = w0.shape[1]
            d.w0[j], d.b0[j], d.w1[j], d.b1[j] = w0.data_ptr(), b0.data_ptr(), w1.data_ptr(), b1.data_ptr()
        d.fp32_weights = 0 if fp16_exact else 1
        d.add_level = 1 if self.add_level else 0
        d.bank_in_dim = 0
        if self.use_feat_bank:
            mlp = self.mlp_feature_bank
            w0, b0, w1, b1 = (_f32c(t, device) for t in (mlp[0].weight, mlp[0].bias, mlp[2].weight, mlp[2].bias))
            keep += [w0, b0, w1, b1]
            d.bank_in_dim = w0.shape[1]
            d.bank_w0, d.bank_b0, d.bank_w1, d.bank_b1 = w0.data_ptr(), b0.data_ptr(), w1.data_ptr(), b1.data_ptr()
        self._marshalled = (key, d, keep)
        return d

    def _parameter_list(self):
        return self._parameters_of(("mlp_opacity", "mlp_cov", "mlp_color") +
                                   (("mlp_feature_bank",) if self.use_feat_bank else ()))

    def _parameters_of(self, names):
        """Weights and biases of the named heads' two layers.  Read from the modules' own tables: the attribute and index
        lookups of nn.Module cost a microsecond each, and every frame asks for a dozen parameters."""
        out = []
        for name in names:
            layers = tuple(self._modules[name]._modules.values())
            for layer in (layers[0], layers[2]):
                p = layer._parameters
                if "weight" in p and "bias" in p:
                    out += (p["weight"], p["bias"])
                else:  # (a reparametrised layer computes them)
                    out += (layer.weight, layer.bias)
        return out

    def _check_level(self, level, A):
        """The reference's behaviour for the level input (anchor_decoder.py:157-186): with add_level and a level
        tensor every head is fed [feat | view | level]; anything else does not match the widths the heads were
        built with and fails in its first matrix product."""
        if not self.add_level:
            return None
        if level is None:
            raise RuntimeError("add_level=True but no level was given: the heads are %d wide, the input without a level "
                               "is not (the reference fails in mlp_opacity with a shape mismatch)"
                               % self.mlp_opacity[0].weight.shape[1])
        for name, flag in (("opacity", self.add_opacity_dist), ("cov", self.add_cov_dist), ("color", self.add_color_dist)):
            if flag:
                raise RuntimeError("add_level=True with add_%s_dist=True: the reference feeds [feat | view | level] "
                                   "(36 columns, anchor_decoder.py:181-182) into a head built 37 wide and fails with a "
                                   "shape mismatch" % name)
        if level.numel() != A:
            raise ValueError("level has %d elements, expected %d" % (level.numel(), A))
        return level.reshape(-1)

    # ---- decode ----------------------------------------------------------------------------------------------
    def _marshal(self, camera_center, anchor, anchor_feat, offset, scaling, visible_mask, level):
        if not anchor.is_cuda:
            raise ValueError("anchor must be a tensor on the GPU (the decoder has no CPU path)")
        dev = anchor.device
        A = anchor.shape[0]
        level = self._check_level(level, A)
        if visible_mask is None:
            visible_mask = torch.ones(A, dtype=torch.bool, device=dev)
        vis = visible_mask
        if vis.dtype is not torch.bool or vis.device != dev or not vis.is_contiguous():
            vis = vis.to(device=dev, dtype=torch.bool).contiguous()
        an = _lib.Anchors()
        tensors = [_f32c(anchor, dev), _f32c(anchor_feat, dev), _f32c(offset, dev), _f32c(scaling, dev),
                   _f32c(camera_center, dev), vis]
        an.A = A
        an.anchor, an.feat, an.offset, an.scaling = (t.data_ptr() for t in tensors[:4])
        an.campos, an.visible_mask = tensors[4].data_ptr(), vis.data_ptr()
        if level is not None:
            tensors.append(_f32c(level, dev))
            an.level = tensors[-1].data_ptr()
        dec = self._decoder_struct(dev)
        # features that fp16 cannot hold exactly (fp32-trained checkpoints) go through the matrix cores as hi + lo
        # pairs; checked once per feature tensor, not per frame
        # (a weak reference: another tensor may have the identity and the address of one that is gone)
        feat_key = (anchor_feat._version, anchor_feat.data_ptr(), tuple(anchor_feat.shape))
        checked = self._feat_checked
        if checked is None or checked[0]() is not anchor_feat or checked[1] != feat_key:
            f32 = tensors[1]
            checked = self._feat_checked = (weakref.ref(anchor_feat), feat_key, bool(torch.equal(f32.half().float(), f32)))
        dec.fp32_features = 0 if checked[2] else 1
        kept = self._kept(dev)
        if kept.get("anchors") != A:
            need = C.c_size_t()
            _lib.check(_lib.load().gs355_decode_workspace_bytes(A, self.n_offsets, 1 if self.use_feat_bank else 0,
                                                                C.byref(need)))
            if kept.get("workspace") is None or kept["workspace"].numel() < need.value:
                kept["workspace"] = torch.empty(max(need.value, 256), dtype=torch.uint8, device=dev)
            kept["anchors"] = A
        return dev, A, dec, an, tensors

    def _kept(self, dev):
        key = (dev, _raw_stream(dev))
        kept = self._per_stream.get(key)
        if kept is None:
            kept = self._per_stream[key] = {}
            while len(self._per_stream) > 4:
                self._per_stream.popitem(last=False)
        else:
            self._per_stream.move_to_end(key)
        return kept

    def _run(self, dec, an, capacity, o, phases, dev):
        ws = self._kept(dev)["workspace"]
        _lib.check(_lib.load().gs355_decode(C.byref(dec), C.byref(an), int(capacity), C.byref(o), ws.data_ptr(),
                                            ws.numel(), int(phases), _raw_stream(dev)))

    def decode_on_device(self, camera_center, anchor, anchor_feat, offset, scaling, visible_mask=None, level=None,
                         want_training_outputs: bool = False, reuse_buffers: bool = False) -> DeviceDecode:
        """The whole decode enqueued on the current stream, nothing read back.  Outputs have room for
        A * n_offsets Gaussians; `counts` says how many are valid.  `reuse_buffers`: the outputs live in one block
        the decoder keeps and overwrites at its next call (a render loop that consumes them at once pays no
        per-frame allocation of the capacity-sized block).  Nothing here is differentiated."""
        dev, A, dec, an, tensors = self._marshal(camera_center, anchor, anchor_feat, offset, scaling, visible_mask, level)
        n = self.n_offsets
        cap = A * n
        # one block for the five outputs (14 floats per Gaussian) and the two counters, carved into views
        kept = self._kept(dev)
        if reuse_buffers and kept.get("block") is not None and kept["block"][0] == cap:
            _, res, o = kept["block"]
        else:
            block = torch.empty(cap * 14 + 2, dtype=torch.float32, device=dev)
            cut = lambda first, width: block[first * cap:(first + width) * cap].view(cap, width)  # noqa: E731
            counts = block[cap * 14:].view(torch.int32)
            res = DeviceDecode(cut(0, 3), cut(3, 3), cut(6, 1), cut(7, 3), cut(10, 4), counts, None, None, counts[0:1])
            o = _lib.Decoded()
            if cap > 0:
                o.xyz, o.color, o.opacity = res.xyz.data_ptr(), res.color.data_ptr(), res.opacity.data_ptr()
                o.scaling, o.rot = res.scaling.data_ptr(), res.rot.data_ptr()
            o.count, o.num_visible = counts.data_ptr(), counts.data_ptr() + 4
            kept["block"] = (cap, res, o) if reuse_buffers else None
        if want_training_outputs:
            res = res._replace(neural_opacity=torch.empty((cap, 1), dtype=torch.float32, device=dev),
                               mask=torch.empty(cap, dtype=torch.bool, device=dev))
            o = _lib.Decoded.from_buffer_copy(o)
            if cap > 0:
                o.neural_opacity, o.mask = res.neural_opacity.data_ptr(), res.mask.data_ptr()
        self._run(dec, an, cap, o, _lib.DECODE_ALL, dev)
        del tensors  # torch's allocator keeps their memory alive for the work already enqueued on this stream
        return res

    def read_counts(self, res):
        """(G, visible anchors) from the device-side counters of a decode: one 8-byte copy to pinned memory, waited
        for.  `res`: a `decode_on_device` result or the int32[2] counter tensor."""
        counts = res.counts if isinstance(res, DeviceDecode) else res
        host = _host_counts(counts.device)
        host.copy_(counts, non_blocking=True)
        torch.cuda.current_stream(counts.device).synchronize()
        return int(host[0]), int(host[1])

    def forward(self, camera_center, anchor, anchor_feat, offset, scaling, visible_mask=None, level=None,
                prog_ratio=None, transition_mask=None, appearance_code=None):
        if self.dist2level == "progressive" and prog_ratio is not None and transition_mask is not None:
            raise NotImplementedError("progressive level-of-detail opacity scaling is not part of this decoder")
        if self.training and torch.is_grad_enabled() and (any(p.requires_grad for p in self.parameters()) or any(
                torch.is_tensor(t) and t.requires_grad for t in (anchor, anchor_feat, offset, scaling))):
            return self._forward_differentiable(camera_center, anchor, anchor_feat, offset, scaling, visible_mask, level)
        with torch.no_grad():
            return self._forward_kernels(camera_center, anchor, anchor_feat, offset, scaling, visible_mask, level)

    _HEAD_LAYERS = {"mlp_opacity": (nn.Linear, nn.ReLU, nn.Linear, nn.Tanh), "mlp_cov": (nn.Linear, nn.ReLU, nn.Linear),
                    "mlp_color": (nn.Linear, nn.ReLU, nn.Linear, nn.Sigmoid)}

    def _heads_as_built(self):
        """Whether the heads are the layers that the constructor made and calling an activation would do nothing but
        evaluate it: the kernels know neither a module that was put in its place nor a hook on it."""
        if any((_module._global_forward_hooks, _module._global_forward_pre_hooks, _module._global_backward_hooks,
                _module._global_backward_pre_hooks)):
            return False
        for name, kinds in self._HEAD_LAYERS.items():
            head = self._modules[name]
            layers = tuple(head._modules.values())
            if type(head) is not nn.Sequential or len(layers) != len(kinds):
                return False
            for layer, kind in zip(layers, kinds):
                if kind is nn.Linear:  # (weight and bias are read, the module is not called)
                    if not isinstance(layer, nn.Linear):
                        return False
                elif (type(layer) is not kind or layer._forward_hooks or layer._forward_pre_hooks or layer._backward_hooks
                      or layer._backward_pre_hooks or "forward" in layer.__dict__):
                    return False
        return True

    def _head_parameters(self):
        return self._parameters_of(("mlp_opacity", "mlp_cov", "mlp_color"))

    def _bank_mix(self, feat, view, level):
        """The feature bank (anchor_decoder.py:163-177): a softmax-weighted mix of strided copies of the features."""
        w = _mlp(self.mlp_feature_bank, view if level is None else torch.cat([view, level], dim=1))  # softmax inside
        return feat[:, ::4].repeat(1, 4) * w[:, 0:1] + feat[:, ::2].repeat(1, 2) * w[:, 1:2] + feat * w[:, 2:3]

    def _kernels_take(self, camera_center, anchor, anchor_feat, offset, scaling, visible_mask, level, params):
        """Whether the training kernels read these tensors as the module's statements do: every one of the shape that the
        kernels assume (they go by the number of anchors alone, rows of fixed widths), fp32, contiguous and on one device;
        camera and level not differentiated.  The statements take more than that (masks of other lengths, scales of more
        columns, heads of other widths) or refuse it themselves."""
        A, n, dim, device, f32 = anchor.shape[0], self.n_offsets, self.feat_dim, anchor.get_device(), torch.float32
        if (A == 0 or anchor.shape != (A, 3) or anchor_feat.shape != (A, dim) or offset.dim() == 0 or offset.shape[0] != A
                or offset.numel() != A * n * 3 or scaling.shape != (A, 6) or visible_mask.shape != (A,)
                or visible_mask.dtype is not torch.bool or visible_mask.get_device() != device
                or (camera_center.shape != (3,) and camera_center.shape != (1, 3)) or camera_center.requires_grad
                or (level is not None and level.requires_grad) or anchor_feat.data_ptr() % 16 != 0):
            return False
        wide = dim + 3 + (level is not None)
        if any(t is None for t in params) or [t.shape for t in params] != [
                (32, wide + bool(self.add_opacity_dist)), (32,), (n, 32), (n,),
                (32, wide + bool(self.add_cov_dist)), (32,), (7 * n, 32), (7 * n,),
                (32, wide + bool(self.add_color_dist)), (32,), (3 * n, 32), (3 * n,)]:
            return False
        tensors = [anchor, anchor_feat, offset, scaling, camera_center]
        if level is not None:
            tensors.append(level)
        if any(t.is_inference() for t in tensors):  # (cannot be saved for the backward pass; the statements need not)
            return False
        for t in tensors + params:
            if t.dtype is not f32 or t.get_device() != device or not t.is_contiguous():
                return False
        return True

    def _forward_differentiable(self, camera_center, anchor, anchor_feat, offset, scaling, visible_mask, level):
        """The training decode: same 7-tuple, the training by-products always present.  On the GPU in the kernels, forward
        and backward, where the heads are what they evaluate (_heads_as_built) and they can take the tensors
        (_kernels_take); else the statements of the reference module as torch operations."""
        level = self._check_level(level, anchor.shape[0])
        if visible_mask is None:
            visible_mask = torch.ones(anchor.shape[0], dtype=torch.bool, device=anchor.device)
        camera_center = camera_center.to(anchor.device)
        params = self._head_parameters() if anchor.is_cuda and self._heads_as_built() else None
        if params is not None and self._kernels_take(camera_center, anchor, anchor_feat, offset, scaling, visible_mask, level,
                                                     params):
            feat = anchor_feat
            if self.use_feat_bank:  # (mixed features of the visible anchors, one row each)
                rows = visible_mask.nonzero(as_tuple=True)[0]
                if rows.shape[0] == 0:  # (no features to hand to the kernels)
                    return self._forward_torch(camera_center, anchor, anchor_feat, offset, scaling, visible_mask, level)
                view = anchor.index_select(0, rows) - camera_center
                view = view / view.norm(dim=1, keepdim=True)
                feat = self._bank_mix(anchor_feat.index_select(0, rows), view,
                                      None if level is None else level.reshape(-1, 1).index_select(0, rows))
                feat = feat.float().contiguous()
            return _DecodeTrain.apply(self, camera_center, visible_mask.contiguous(), level, self.use_feat_bank, anchor,
                                      feat, offset, scaling, *params)
        return self._forward_torch(camera_center, anchor, anchor_feat, offset, scaling, visible_mask, level)

    def _forward_torch(self, camera_center, anchor, anchor_feat, offset, scaling, visible_mask, level):
        """The statements of the reference module (anchor_decoder.py:147-242) as torch operations, for autograd."""
        # Rows are selected with index_select over index lists computed once, not with boolean masks: the results
        # are the same tensors, but the backward of a boolean-mask index is a sorting index_put (3.7 ms per step at
        # 500k anchors), that of index_select an index_add.
        rows = visible_mask.nonzero(as_tuple=True)[0]
        # (an index past the end is an error on the CPU and an assertion on the GPU: the rare call that can have one waits
        # for the largest)
        shortest = min(t.shape[0] for t in (anchor, anchor_feat, offset, scaling))
        if shortest < visible_mask.shape[0] and rows.numel() and int(rows[-1]) >= shortest:
            raise IndexError("anchor %d is visible, a tensor has %d rows" % (int(rows[-1]), shortest))
        a, feat, off, sc = (t.index_select(0, rows) for t in (anchor, anchor_feat, offset, scaling))
        lvl = level.reshape(-1, 1).index_select(0, rows).to(feat.dtype) if level is not None else None
        heads = [functools.partial(_mlp, head) for head in (self.mlp_opacity, self.mlp_cov, self.mlp_color)]
        return self._from_rows(camera_center, a, feat, off, sc, lvl, heads)

    def _from_rows(self, camera_center, a, feat, off, sc, lvl, heads, mixed=False, mask=None):
        """The statements from the rows of the visible anchors on.  `heads`: opacity, covariance and colour, callable;
        `mixed`: the features come out of the feature bank; `mask`: the choice of offsets, where it was made before."""
        mlp_opacity, mlp_cov, mlp_color = heads
        view = a - camera_center.to(a.device)
        dist = view.norm(dim=1, keepdim=True)
        view = view / dist
        if self.use_feat_bank and not mixed:
            feat = self._bank_mix(feat, view, lvl)
        if lvl is not None:  # (:181-182: both inputs become [feat | view | level])
            with_dist = without = torch.cat([feat, view, lvl], dim=1)
        else:
            with_dist, without = torch.cat([feat, view, dist], dim=1), torch.cat([feat, view], dim=1)
        n = self.n_offsets
        neural_opacity = mlp_opacity(with_dist if self.add_opacity_dist else without).reshape(-1, 1)
        if mask is None:
            mask = (neural_opacity > 0.0).view(-1)
        kept = mask.nonzero(as_tuple=True)[0]
        owner = torch.div(kept, n, rounding_mode="floor")  # anchor (among the visible ones) of each kept offset
        off = off.reshape(-1, 3)
        color = mlp_color(with_dist if self.add_color_dist else without).reshape(-1, 3)
        cov = mlp_cov(with_dist if self.add_cov_dist else without).reshape(-1, 7)
        shortest = min(t.shape[0] for t in (off, color, cov))
        if shortest < mask.shape[0] and kept.numel() and int(kept[-1]) >= shortest:
            raise IndexError("offset %d of the visible anchors is kept, a tensor has %d rows" % (int(kept[-1]), shortest))
        color, cov = color.index_select(0, kept), cov.index_select(0, kept)
        sc_kept = sc.index_select(0, owner)
        scaling_out = sc_kept[:, 3:6] * torch.sigmoid(cov[:, 0:3])
        rot = torch.nn.functional.normalize(cov[:, 3:7])
        xyz = a.index_select(0, owner) + off.index_select(0, kept) * sc_kept[:, 0:3]
        return xyz, color, neural_opacity.index_select(0, kept), scaling_out, rot, neural_opacity, mask

    def _forward_kernels(self, camera_center, anchor, anchor_feat, offset, scaling, visible_mask=None, level=None):
        """Returns (xyz[G,3], color[G,3], opacity[G,1], scaling[G,3], rot[G,4], neural_opacity, mask): the neural
        Gaussians of the visible anchors whose decoded opacity is positive, in boolean-mask order; in training mode
        also the opacity of every offset of the visible anchors ([A_vis * n, 1]) and the mask over them, else None.

        The output shapes depend on the data, so the count phase runs first and its two counters are read back
        (the reference's boolean-mask indexing synchronises at the same place); the emit phase then writes into
        tensors of exactly that size."""
        dev, A, dec, an, tensors = self._marshal(camera_center, anchor, anchor_feat, offset, scaling, visible_mask, level)
        # the two counters go straight into pinned host memory (which the GPU addresses like its own): no copy is
        # enqueued, the host waits for the count phase and reads them
        counts = _host_counts(dev)
        o = _lib.Decoded()
        o.count, o.num_visible = counts.data_ptr(), counts.data_ptr() + 4
        try:
            self._run(dec, an, 0, o, _lib.DECODE_COUNT, dev)
        finally:
            torch.cuda.current_stream(dev).synchronize()
        G, a_vis = int(counts[0]), int(counts[1])
        f = lambda *shape: torch.empty(shape, dtype=torch.float32, device=dev)  # noqa: E731
        out = (f(G, 3), f(G, 3), f(G, 1), f(G, 3), f(G, 4))
        extra = (None, None)
        if self.training:
            extra = (f(a_vis * self.n_offsets, 1), torch.empty(a_vis * self.n_offsets, dtype=torch.bool, device=dev))
        if G > 0 or (self.training and a_vis > 0):
            if G > 0:
                o.xyz, o.color, o.opacity, o.scaling, o.rot = (t.data_ptr() for t in out)
            if self.training and a_vis > 0:
                o.neural_opacity, o.mask = extra[0].data_ptr(), extra[1].data_ptr()
            o.count = o.num_visible = None
            self._run(dec, an, G, o, _lib.DECODE_EMIT, dev)
        del tensors
        return out + extra
