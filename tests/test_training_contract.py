"""What the training forward and backward on tile steps refuse, checked without a GPU: the tensors are fake (types, shapes
and devices, no memory), and the first call into the kernels' wrappers ends the test."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from mlp_splatting_amd import ops, tile_ext
from mlp_splatting_amd.tile_ext import TileExt

W, H, N = 20, 12, 7


class Reached(Exception):
    pass


def _scene_tensors():
    f32 = dict(dtype=torch.float32, device="cuda")
    shapes = [(W * H, 3), (W * H, 3), (N, 3), (N, 3), (N, 4), (11,), (7,), (6,), (6,), (N, 32, 72), (N, 32), (N, 32, 32),
              (N, 32), (N, 4, 32), (N, 4)]
    return [torch.empty(s, dtype=torch.int32, device="cuda") if i in (5, 6) else torch.empty(s, **f32)
            for i, s in enumerate(shapes)]


@pytest.fixture
def ext(monkeypatch):
    def stop(*_a, **_k):
        raise Reached
    ext = TileExt()
    for name in ("train_forward", "train_reverse", "train_gradients", "train_group", "validate_tile_lists", "sort_tiles",
                 "prepare_primitives", "pack_mfma_weights_listed"):
        monkeypatch.setattr(ops, name, stop)

    class NoDevice:
        def __init__(self, *_a):
            pass

        def __enter__(self):
            pass

        def __exit__(self, *_a):
            pass
    monkeypatch.setattr(torch.cuda, "device", NoDevice)
    monkeypatch.setattr(tile_ext, "_on_device", NoDevice)
    return ext


# (index of the scene tensor, what replaces it)
def _half(t):
    return t.half()


def _short(t):
    return t[:-1]


def _wide(t):
    return torch.cat([t, t], dim=-1)


def _strided(t):
    return torch.cat([t, t], dim=-1)[..., :t.shape[-1]]


BAD = [([i], _half) for i in (0, 1, 2, 3, 4, 7, 8)] + [([i], _half) for i in range(9, 15)] + [(list(range(9, 15)), _half)]
BAD += [([i], _short) for i in (0, 1, 2, 3, 4, 7, 8, *range(9, 15))]
BAD += [([i], _wide) for i in (1, 3, 4, 7, 9, 10, 11, 12, 13, 14)] + [([7, 8], _wide)]
BAD += [([i], _strided) for i in (0, 1, 2, 9, 11, 13)]
BAD += [([i], lambda t: t.cpu()) for i in (1, 9, 14)] + [([5], lambda t: t.long()), ([6], lambda t: t.long())]


@pytest.mark.parametrize("precision", [None, "float16"])
@pytest.mark.parametrize("which,change", BAD)
def test_the_training_forward_refuses_what_its_kernels_would_misread(ext, which, change, precision):
    with FakeTensorMode():
        x = _scene_tensors()
        for i in which:
            x[i] = change(x[i])
        with pytest.raises(RuntimeError):
            ext.train_forward(x, W, H, 1e-3, precision=precision)


@pytest.mark.parametrize("which,change", BAD)
def test_the_backward_holds_the_saved_tensors_to_the_same_contract(ext, which, change):
    with FakeTensorMode():
        x = _scene_tensors()
        for i in which:
            x[i] = change(x[i])
        frame = ops.TrainFrame(None, 11, W, H, 1, 0, 1)
        with pytest.raises(RuntimeError):
            ext.backward_from_steps(frame, None, x, torch.empty(W * H, 3, device="cuda"), torch.empty(W * H, device="cuda"))


def test_well_formed_tensors_reach_the_kernels(ext):
    with FakeTensorMode():
        x = _scene_tensors()
        frame = ops.TrainFrame(None, 11, W, H, 1, 0, 1)
        with pytest.raises(Reached):
            ext.train_forward(x, W, H, 1e-3)
        with pytest.raises(Reached):
            ext.backward_from_steps(frame, None, x, torch.empty(W * H, 3, device="cuda"), torch.empty(W * H, device="cuda"))
        for bad in (torch.empty(W * H, 3, device="cuda", dtype=torch.float64), torch.empty(W * H - 1, 3, device="cuda"),
                    torch.empty(W * H, 4, device="cuda"), torch.empty(3, W * H, device="cuda").t(), torch.empty(W * H, 3)):
            with pytest.raises(RuntimeError):
                ext.backward_from_steps(frame, None, x, bad, torch.empty(W * H, device="cuda"))
        for bad in (torch.empty(W * H, device="cuda").half(), torch.empty(W * H - 1, device="cuda")):
            with pytest.raises(RuntimeError):
                ext.backward_from_steps(frame, None, x, torch.empty(W * H, 3, device="cuda"), bad)


def test_saved_steps_come_back_whole():
    with FakeTensorMode():
        steps = torch.empty(4096, dtype=torch.uint8, device="cuda")
        frame = ops.TrainFrame(steps, 11, W, H, 1, 0, 1).with_workspace(None)
        assert frame.with_workspace(steps).workspace is steps
        for bad in (steps[:-256], steps.cpu(), steps.half(), torch.empty(8192, dtype=torch.uint8, device="cuda")[::2]):
            with pytest.raises(RuntimeError):
                frame.with_workspace(bad)


def test_the_backward_takes_the_offsets_attributes_and_adjoint_of_its_forward(monkeypatch):
    monkeypatch.setattr(ops._lib, "load", lambda: (_ for _ in ()).throw(Reached()))
    monkeypatch.setattr(ops, "_ptr", lambda t: 0)

    class Feature:
        slots, channels, row_bytes, kept, target_size = 4, 6, 256, 256, (3, 2)
    with FakeTensorMode():
        offsets = torch.empty(3 * 2 + 1, dtype=torch.int32, device="cuda")
        frame = ops.TrainFrame(torch.empty(256, dtype=torch.uint8, device="cuda"), 11, W, H, 1, 0, 1)
        grads = torch.empty(W * H, 3, device="cuda"), torch.empty(W * H, device="cuda")
        calls = (lambda o: ops.train_group(frame, o, N), lambda o: ops.train_reverse(frame, o, *grads))
        for call in calls:
            with pytest.raises(Reached):
                call(offsets)
            for bad in (offsets[:-1], offsets.long(), offsets.cpu(), torch.empty(14, dtype=torch.int32, device="cuda")[::2]):
                with pytest.raises(RuntimeError):
                    call(bad)
        kept, attributes, one = offsets, torch.empty(N, 4, 6, device="cuda"), torch.empty((), device="cuda")
        with pytest.raises(Reached):
            ops.train_feature_gradients(frame, kept, Feature, kept, attributes, one)
        for bad in (attributes.half(), attributes[:, :3].contiguous(), attributes[..., :4], attributes.cpu()):
            with pytest.raises(RuntimeError):
                ops.train_feature_gradients(frame, kept, Feature, kept, bad, one)
        for bad in (one.double(), torch.empty(2, device="cuda"), one.cpu()):
            with pytest.raises(RuntimeError):
                ops.train_feature_gradients(frame, kept, Feature, kept, attributes, bad)


@pytest.mark.parametrize("shape", [(6,), (N, 2, 2, 6)])
def test_the_streamed_loss_refuses_attributes_that_are_no_rows_of_channels(shape):
    """One axis would be read as [N, C] past its end."""
    from mlp_splatting_amd.record_feature_loss import _loss_geometry
    with FakeTensorMode():
        image, target = torch.empty(W * H, 3, device="cuda"), torch.empty(2, 3, 6, device="cuda")
        assert _loss_geometry(torch.empty(N, 6, device="cuda"), target, (image,), W, H) == (2, 3, 6, 1)
        assert _loss_geometry(torch.empty(N, 5, 6, device="cuda"), target, (image,), W, H) == (2, 3, 6, 5)
        with pytest.raises(ValueError, match="1/4/5-slot renderer"):
            _loss_geometry(torch.empty(shape, device="cuda"), target, (image,), W, H)


@pytest.mark.parametrize("asked,calls", [((4,), 1), ((9, 9), 2), ((9, 10), None)])
def test_no_frame_comes_back_without_room_for_its_steps(monkeypatch, asked, calls):
    made = []

    class Lib:
        def mlpsp_train_workspace_bytes(self, *_a):
            return 256

        def mlpsp_train_forward_f32(self, *_a):
            made.append(asked[len(made)])
            return 0
    empty = torch.empty

    def chunks_asked(*shape, **kw):             # (the workspace: the kernels count the chunks that they drew)
        t = empty(*shape, **kw)
        if t.dtype == torch.uint8:
            t.view(torch.int32)[:3] = torch.tensor([asked[min(len(made), 1)], 0, 3])
        return t
    monkeypatch.setattr(ops._lib, "load", Lib)
    monkeypatch.setattr(ops, "_stream", lambda _d: 0)
    monkeypatch.setattr(ops.torch, "empty", chunks_asked)
    x = torch.zeros(1)
    args = (x, x, x, x.int(), x.int(), x, x, [x] * 6, W, H, 1e-3, 64, 8 * ops._lib.STEP_CHUNK)
    if calls is None:
        with pytest.raises(RuntimeError, match="more steps"):
            ops.train_forward(*args)
    else:
        assert ops.train_forward(*args)[2].chunks == asked[-1] and len(made) == calls
