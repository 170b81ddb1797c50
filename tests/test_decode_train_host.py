"""Host side of the training decode, no GPU needed: what is handed to the library, which stands in as a recorder here."""
import ctypes as C
from types import SimpleNamespace

import pytest
import torch

from landmarksystem_amd import _lib, anchor_decoder
from landmarksystem_amd.anchor_decoder import FusedAnchorDecoder, _DecodeTrain


class Recorder:
    """The library's training calls: counts of `visible` rows and `kept` Gaussians, and the records of the backward call."""

    def __init__(self, visible, kept):
        self.visible, self.kept, self.back, self.heads = visible, kept, None, []

    def gs355_decode_train_bytes(self, A, num_visible, n, workspace, scratch):
        workspace._obj.value, scratch._obj.value = 1024, 1024
        return 0

    def gs355_decode_train(self, dec, an, rows, capacity, out, workspace, nbytes, phase, stream):
        if phase == _lib.TRAIN_HEADS:
            self.heads.append(rows._obj.num_visible)
            C.c_int32.from_address(out._obj.count).value = self.kept
            C.c_int32.from_address(out._obj.num_visible).value = self.visible
        return 0

    def gs355_decode_train_backward(self, dec, an, rows, workspace, nbytes, cot, grads, scratch, scratch_bytes, stream):
        self.back = SimpleNamespace(dec=dec._obj, an=an._obj, rows=rows._obj, workspace=workspace)
        return 0


@pytest.fixture
def recorder(monkeypatch):
    lib = Recorder(visible=5, kept=11)
    monkeypatch.setattr(_lib, "load", lambda: lib)
    monkeypatch.setattr(anchor_decoder, "_raw_stream", lambda device: 0)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: SimpleNamespace(synchronize=lambda: None))
    return lib


def decoder(n=10, **kw):
    torch.manual_seed(0)
    dec = FusedAnchorDecoder(**dict(dict(use_feat_bank=False, add_opacity_dist=True, add_cov_dist=True, add_color_dist=True,
                                         view_dim=3, feat_dim=32, n_offsets=n), **kw)).train()
    dec._host_count = torch.zeros(2, dtype=torch.int32)
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
