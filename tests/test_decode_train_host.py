"""Host side of the training decode, no GPU needed: what is handed to the library, which stands in as a recorder here."""
import copy
import ctypes as C
import pickle
import threading
from collections import OrderedDict
from types import SimpleNamespace

import pytest
import torch

from landmarksystem_amd import _lib, anchor_decoder
from landmarksystem_amd.anchor_decoder import FusedAnchorDecoder, _DecodeTrain


class Recorder:
    """The library's training calls: counts of `visible` rows and `kept` Gaussians, and the records of the backward call."""

    def __init__(self, visible, kept):
        self.visible, self.kept, self.back, self.heads, self.opacities = visible, kept, None, [], None

    def wait(self):
        pass

    def gs355_decode_train_bytes(self, A, num_visible, n, workspace, scratch):
        workspace._obj.value, scratch._obj.value = 1024, 1024
        return 0

    def gs355_decode_train(self, dec, an, rows, capacity, out, workspace, nbytes, phase, stream):
        if phase == _lib.TRAIN_HEADS:
            self.heads.append(rows._obj.num_visible)
            C.c_int32.from_address(out._obj.count).value = self.kept
            C.c_int32.from_address(out._obj.num_visible).value = self.visible
            if self.opacities is not None:  # (pre-activations)
                C.memmove(rows._obj.pre[0], self.opacities.data_ptr(), 4 * self.opacities.numel())
        return 0

    def gs355_decode_train_backward(self, dec, an, rows, workspace, nbytes, cot, grads, scratch, scratch_bytes, stream):
        self.back = SimpleNamespace(dec=dec._obj, an=an._obj, rows=rows._obj, workspace=workspace)
        return 0


@pytest.fixture
def recorder(monkeypatch):
    lib = Recorder(visible=5, kept=11)
    monkeypatch.setattr(_lib, "load", lambda: lib)
    monkeypatch.setattr(anchor_decoder, "_raw_stream", lambda device: 0)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: SimpleNamespace(synchronize=lambda: lib.wait()))
    zeros = torch.zeros
    monkeypatch.setattr(torch, "zeros", lambda *a, pin_memory=False, **kw: zeros(*a, **kw))  # (no GPU to pin for)
    return lib


def decoder(n=10, **kw):
    torch.manual_seed(0)
    dec = FusedAnchorDecoder(**dict(dict(use_feat_bank=False, add_opacity_dist=True, add_cov_dist=True, add_color_dist=True,
                                         view_dim=3, feat_dim=32, n_offsets=n), **kw)).train()
    return dec


def inputs(A=7, n=10):
    return [torch.randn(*s, requires_grad=True) for s in ((A, 3), (A, 32), (A, n, 3), (A, 6))]


def apply(dec, leaves, visible=None, camera=None):
    A = leaves[0].shape[0]
    return _DecodeTrain.apply(dec, torch.zeros(3) if camera is None else camera,
                              torch.ones(A, dtype=torch.bool) if visible is None else visible, None, False, *leaves,
                              *dec._head_parameters())


def pointers(back):
    heads = [p[j] for p in (back.dec.w0, back.dec.b0, back.dec.w1, back.dec.b1) for j in range(3)]
    return [back.an.anchor, back.an.feat, back.an.offset, back.an.scaling, back.an.campos] + heads


def aligned_copy(t, to=256):
    room = torch.empty(t.numel() * t.element_size() + to, dtype=torch.uint8)
    first = -room.data_ptr() % to
    copy = room[first:first + t.numel() * t.element_size()].view(t.dtype).view(t.shape)
    return copy.copy_(t)


def test_backward_reads_what_saved_tensor_hooks_hand_back(recorder):
    """The tensors of the forward pass may be gone by then: every pointer of the backward call is into an unpacked one."""
    handed = []

    def unpack(t):
        handed.append(aligned_copy(t))
        return handed[-1]

    dec, leaves = decoder(), inputs()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.detach().clone(), unpack):
        out = apply(dec, leaves)
    out[0].sum().backward()
    assert set(pointers(recorder.back)) <= {t.data_ptr() for t in handed}
    (block,) = [t for t in handed if t.dtype == torch.uint8]
    parts = [recorder.back.workspace] + list(recorder.back.rows.hidden) + list(recorder.back.rows.pre)
    assert all(block.data_ptr() <= p < block.data_ptr() + block.numel() and p % 256 == 0 for p in parts)


def test_backward_reads_a_replaced_parameter_where_it_is(recorder):
    dec, leaves = decoder(), inputs()
    out = apply(dec, leaves)
    leaves[2].data = leaves[2].data.clone()
    out[0].sum().backward()
    assert recorder.back.an.offset == leaves[2].data_ptr()
    # (of another shape: refused, as the kernels go by the forward pass's)
    leaves = inputs()
    out = apply(dec, leaves)
    leaves[2].data = torch.zeros(5, 10, 3)
    recorder.back = None
    with pytest.raises(RuntimeError, match="shape"):
        out[0].sum().backward()
    assert recorder.back is None


def test_camera_and_mask_may_change_after_the_forward_pass(recorder):
    """A caller that renders several views before one backward pass moves its camera tensor in place."""
    dec, leaves, camera, visible = decoder(), inputs(), torch.zeros(3), torch.ones(7, dtype=torch.bool)
    out = apply(dec, leaves, visible, camera)
    camera.add_(1.0)
    visible.logical_not_()
    out[0].sum().backward()
    assert recorder.back.an.campos != camera.data_ptr()


def _forms():
    """name -> (what differs from the plain call: A = 7 anchors, n = 3 offsets; whether the kernels take it; whether the
    module's statements do)"""
    r = torch.Generator().manual_seed(1)
    rand = lambda *s: torch.randn(*s, generator=r)  # noqa: E731
    mask = torch.tensor([1, 0, 1, 1, 0, 1, 1], dtype=torch.bool)
    return {
        "plain": ({}, True, True),
        "no mask": (dict(visible_mask=None), True, True),
        "mask of bytes": (dict(visible_mask=mask.byte()), False, True),
        "mask as a column": (dict(visible_mask=mask[:, None]), False, True),
        "shorter mask": (dict(visible_mask=mask[:4]), False, True),
        "longer mask, all of it past the end unset": (dict(visible_mask=torch.cat([mask, ~mask.new_ones(5)])), False, True),
        "longer mask": (dict(visible_mask=torch.cat([mask, mask])), False, False),
        "strided mask": (dict(visible_mask=mask.repeat_interleave(2)[::2]), True, True),
        "camera as a row": (dict(camera_center=rand(1, 3)), True, True),
        "camera of one number": (dict(camera_center=rand(1)), False, True),
        "camera per visible anchor": (dict(camera_center=rand(5, 3)), False, True),
        "differentiable camera": (dict(camera_center=rand(3).requires_grad_(True)), False, True),
        "strided anchors": (dict(anchor=rand(3, 7).t()), False, True),
        "anchors of four columns": (dict(anchor=rand(7, 4)), False, False),
        "offsets as rows": (dict(offset=rand(7, 9)), True, True),
        "fewer offsets": (dict(offset=rand(7, 1, 3)), False, False),
        "more offsets": (dict(offset=rand(7, 5, 3)), False, True),
        "offsets of fewer anchors": (dict(offset=rand(5, 3, 3)), False, False),
        "scales of three columns": (dict(scaling=rand(7, 3).exp()), False, False),
        "scales of eight columns": (dict(scaling=rand(7, 8).exp()), False, True),
        "scales of fewer anchors": (dict(scaling=rand(3, 6).exp()), False, False),
        "features of fewer anchors": (dict(anchor_feat=rand(6, 32)), False, False),
        "features of more anchors": (dict(anchor_feat=rand(9, 32)), False, True),
        "wider features": (dict(anchor_feat=rand(7, 64)), False, False),
        "misaligned features": (dict(anchor_feat=rand(7 * 32 + 1)[1:].view(7, 32)), False, True),
        "double features": (dict(anchor_feat=rand(7, 32).double()), False, False),
        "head of another hidden width": (dict(hidden=48), False, True),
        "head of another input width": (dict(inputs=40), False, False),
        "head of more outputs": (dict(outputs=12), False, True),
        "head of fewer outputs": (dict(outputs=6), False, False),
    }


@pytest.mark.parametrize("form", list(_forms()))
def test_what_the_training_kernels_take(form):
    """The kernels are chosen only for what they read as the module's statements do; the rest goes to the statements, which
    take it or refuse it."""
    change, kernels, statements = _forms()[form]
    change = dict(change)
    dec = decoder(n=3)
    if "hidden" in change or "inputs" in change or "outputs" in change:
        first = torch.nn.Linear(change.pop("inputs", 36), change.get("hidden", 32))
        dec.mlp_color = torch.nn.Sequential(first, torch.nn.ReLU(True),
                                            torch.nn.Linear(change.pop("hidden", 32), change.pop("outputs", 9)), torch.nn.Sigmoid())
    with torch.no_grad():
        dec.mlp_opacity[2].bias.fill_(2.0)  # (every offset is kept)
    anchor, feat, offset, scaling = inputs(n=3)
    call = dict(camera_center=torch.tensor([0.3, -4.0, 2.0]), anchor=anchor, anchor_feat=feat, offset=offset,
                scaling=scaling.exp(), visible_mask=torch.tensor([1, 0, 1, 1, 0, 1, 1], dtype=torch.bool))
    call.update(change)
    mask = torch.ones(7, dtype=torch.bool) if call["visible_mask"] is None else call["visible_mask"]
    takes = dec._kernels_take(*[call[k] for k in ("camera_center", "anchor", "anchor_feat", "offset", "scaling")],
                              mask.contiguous() if mask.dim() == 1 else mask, None, dec._head_parameters())
    assert takes == kernels
    if not statements:
        with pytest.raises((RuntimeError, IndexError)):
            dec(**call)
        return
    got = dec(**call)
    assert got[0].shape[0] == int(mask.sum()) * 3
    if kernels:  # as the kernels read them: rows of the fixed widths, one after the other
        rows = dict(camera_center=call["camera_center"].reshape(3), offset=call["offset"].reshape(7, 3, 3))
        for a, b in zip(got, dec(**{**call, **rows})):
            assert torch.equal(a, b)


def test_heads_that_were_changed_take_the_statements():
    """A hook on an activation, a module in its place or a head of other layers: the kernels know nothing of it."""
    called = []
    note = lambda *a: called.append(1)  # noqa: E731
    changes = {
        "forward hook": lambda d: d.mlp_opacity[1].register_forward_hook(note),
        "forward pre-hook": lambda d: d.mlp_color[3].register_forward_pre_hook(note),
        "backward hook": lambda d: d.mlp_color[3].register_full_backward_hook(note),
        "backward pre-hook": lambda d: d.mlp_opacity[3].register_full_backward_pre_hook(note),
        "own forward": lambda d: setattr(d.mlp_cov[1], "forward", torch.relu),
        "another activation": lambda d: d.mlp_color.__setitem__(1, torch.nn.LeakyReLU()),
        "one more layer": lambda d: d.mlp_cov.append(torch.nn.Tanh()),
        "normalised hidden units": lambda d: setattr(d, "mlp_opacity", torch.nn.Sequential(
            d.mlp_opacity[0], torch.nn.LayerNorm(32), torch.nn.ReLU(), d.mlp_opacity[2], torch.nn.Tanh())),
        "hook on all modules": lambda d: torch.nn.modules.module.register_module_forward_hook(note),
    }
    for name, change in changes.items():
        dec, leaves = decoder(n=3), inputs(n=3)
        assert dec._heads_as_built()
        handle = change(dec)
        try:
            assert not dec._heads_as_built(), name
            called.clear()
            out = dec(torch.tensor([0.3, -4.0, 2.0]), *leaves)
            (out[1].sum() + out[5].sum()).backward()
            assert bool(called) == ("hook" in name), name
        finally:
            if handle is not None and hasattr(handle, "remove"):
                handle.remove()
    dec = decoder(n=3)
    dec.mlp_opacity[0].register_forward_hook(note)  # (the linear layers are not called, their parameters are read)
    assert dec._heads_as_built()


def test_parameters_are_found_by_place():
    """Heads whose layers have names of their own."""
    dec = decoder(n=3)
    want = dec._head_parameters()
    names = ("first", "relu", "second", "tanh")
    dec.mlp_opacity = torch.nn.Sequential(OrderedDict(zip(names, dec.mlp_opacity)))
    assert all(a is b for a, b in zip(dec._head_parameters(), want)) and dec._heads_as_built()


@pytest.mark.parametrize("bank", [False, True])
def test_gradients_can_be_differentiated(recorder, bank):
    """A penalty on a gradient: first and second derivatives of a backward pass under create_graph=True are the statements',
    with the forward pass's choice of offsets."""
    dec = decoder(n=3, use_feat_bank=bank).double()
    leaves = [t.detach().double().requires_grad_(True) for t in inputs(n=3)]
    camera, visible = torch.tensor([0.3, -4.0, 2.0]).double(), torch.tensor([1, 0, 1, 1, 0, 1, 1], dtype=torch.bool)
    want = dec._forward_torch(camera, *leaves, visible, None)
    recorder.kept, recorder.opacities = want[0].shape[0], torch.atanh(want[5].detach()).float().contiguous()
    rows = visible.nonzero(as_tuple=True)[0]
    feat = leaves[1]
    if bank:
        view = leaves[0].index_select(0, rows) - camera
        feat = dec._bank_mix(feat.index_select(0, rows), view / view.norm(dim=1, keepdim=True), None)
    got = _DecodeTrain.apply(dec, camera, visible, None, bank, leaves[0], feat, *leaves[2:], *dec._head_parameters())
    weights = [torch.randn(t.shape).double() for t in want[:6]]  # (exact in the outputs' type)
    params = leaves + list(dec.parameters())

    def derivatives(out):
        loss = sum((t.to(w) * w).sum() for t, w in zip(out, weights))
        first = torch.autograd.grad(loss, params, create_graph=True, allow_unused=True)
        second = torch.autograd.grad(sum(f.square().sum() for f in first if f is not None and f.requires_grad), params,
                                     allow_unused=True)
        return [torch.zeros_like(p) if g is None else g for p, g in zip(params * 2, first + second)]

    for a, b in zip(derivatives(got), derivatives(want)):
        assert torch.allclose(a, b, rtol=1e-9, atol=1e-9 * float(b.detach().abs().max()) + 1e-300)
    assert recorder.back is None
    # ... but not behind a mask that has changed since
    got = _DecodeTrain.apply(dec, camera, visible, None, bank, leaves[0], feat, *leaves[2:], *dec._head_parameters())
    visible.logical_not_()
    with pytest.raises(RuntimeError, match="in place"):
        derivatives(got)


def test_batched_cotangents_take_the_statements(recorder):
    dec, leaves = decoder(n=3), inputs(n=3)
    for p in dec.parameters():
        p.requires_grad_(False)
    visible = torch.tensor([1, 0, 1, 1, 0, 1, 1], dtype=torch.bool)
    want = dec._forward_torch(torch.zeros(3), *leaves, visible, None)
    recorder.kept, recorder.opacities = want[0].shape[0], torch.atanh(want[5].detach()).contiguous()
    got = apply(dec, leaves, visible)
    cotangents = torch.randn(4, *want[3].shape)
    for a, b in zip(torch.autograd.grad(got[3], leaves, cotangents, is_grads_batched=True, allow_unused=True),
                    torch.autograd.grad(want[3], leaves, cotangents, is_grads_batched=True, allow_unused=True)):
        assert (a is None) == (b is None) and (a is None or torch.allclose(a, b, rtol=1e-4, atol=1e-5))


def test_threads_that_share_a_decoder_keep_their_counts(recorder, monkeypatch):
    """Both calls have stored their counts before either reads its own (two streams, or replicas over one __dict__)."""
    dec = decoder(n=3)
    both, own = threading.Barrier(2), threading.local()
    store = recorder.gs355_decode_train

    def decode_train(dec, an, rows, capacity, out, *rest):
        recorder.visible, recorder.kept = own.counts
        return store(dec, an, rows, capacity, out, *rest)

    monkeypatch.setattr(recorder, "gs355_decode_train", decode_train)
    monkeypatch.setattr(recorder, "wait", lambda: both.wait(timeout=20))
    shapes = {}

    def train(visible, kept):
        own.counts = (visible, kept)
        shapes[visible] = [t.shape[0] for t in apply(dec, inputs(n=3))]

    threads = [threading.Thread(target=train, args=a) for a in ((5, 11), (6, 13))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert shapes == {5: [11] * 5 + [15] * 2, 6: [13] * 5 + [18] * 2}


@pytest.mark.parametrize("make", [copy.deepcopy, lambda d: pickle.loads(pickle.dumps(d))])
def test_copies_start_without_what_calls_left_behind(recorder, make):
    """Buffers, records of pointers and pinned memory belong to the decoder that made them: a copy makes its own."""
    dec = decoder(n=3)
    apply(dec, inputs(n=3))
    dec._per_stream[("stream",)] = dict(workspace=torch.zeros(4), block=(1, None, _lib.Decoded(1)))
    dec._marshalled, dec._feat_checked = ("key", _lib.Decoder(), []), ("key", True)
    twin = make(dec)
    assert not twin._per_stream and twin._marshalled is None and twin._feat_checked is None
    assert all(torch.equal(a, b) and a is not b for a, b in zip(dec.parameters(), twin.parameters()))
    assert not any(isinstance(v, torch.Tensor) for v in twin.__dict__.values())
    apply(twin, inputs(n=3))


@pytest.mark.parametrize("limit,compact,calls", [(7, False, [7]), (6, False, [0, 5]), (6, True, [5])])
def test_room_for_rows(recorder, monkeypatch, limit, compact, calls):
    """Room for every anchor up to a number of anchors, for the visible ones beyond (counted first, unless the features
    come out of the bank, one row for each)."""
    monkeypatch.setattr(anchor_decoder, "_ROOM_FOR_ALL", limit)
    dec, leaves = decoder(), inputs()
    feat = leaves[1][:5] if compact else leaves[1]
    out = _DecodeTrain.apply(dec, torch.zeros(3), torch.arange(7) < 5, None, compact, leaves[0], feat, *leaves[2:],
                             *dec._head_parameters())
    assert recorder.heads == calls and out[5].shape[0] == 50
    assert out[0].grad_fn.parts.room == calls[-1]


def test_more_rows_than_room_are_refused(recorder, monkeypatch):
    """(the mask changed while the call was under way; the kernels write no row past the room)"""
    monkeypatch.setattr(recorder, "visible", 6)
    dec, leaves = decoder(), inputs()
    with pytest.raises(RuntimeError, match="visible"):
        _DecodeTrain.apply(dec, torch.zeros(3), torch.arange(7) < 5, None, True, leaves[0], leaves[1][:5], *leaves[2:],
                           *dec._head_parameters())
