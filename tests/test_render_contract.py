"""What the frames refuse before their kernels read it, checked without a GPU: the tensors are fake (types, shapes and
devices, no memory), and the first call into the kernels' wrappers ends the test."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from mlp_splatting_amd import ops, tile_ext
from mlp_splatting_amd.tile_ext import TileExt

W, H, N = 20, 12, 7
SHAPES = [(W * H, 3), (W * H, 3), (N, 3), (N, 3), (N, 4), (11,), (7,), (6,), (6,), (N, 32, 72), (N, 32), (N, 32, 32),
          (N, 32), (N, 4, 32), (N, 4)]


class Reached(Exception):
    pass


class NoDevice:
    def __init__(self, *_a):
        pass

    def __enter__(self):
        pass

    def __exit__(self, *_a):
        pass


@pytest.fixture
def ext(monkeypatch):
    def stop(*_a, **_k):
        raise Reached

    class Lib:                                   # (prepares and packs; nothing is read or written)
        def __getattr__(self, _name):
            return lambda *_a: 0
    for name in ("render_per_pixel_f32", "render_tilecenter_f32", "render_tilecenter_mfma"):
        monkeypatch.setattr(ops, name, stop)
    monkeypatch.setattr(ops, "sort_tiles", lambda *a, **_k: (a[3], None))
    monkeypatch.setattr(ops, "validate_tile_lists", lambda *_a: None)
    monkeypatch.setattr(ops, "_ptr", lambda _t: 0)
    monkeypatch.setattr(ops, "_stream", lambda _d: 0)
    monkeypatch.setattr(ops._lib, "load", Lib)
    monkeypatch.setattr(torch.cuda, "device", NoDevice)
    monkeypatch.setattr(tile_ext, "_on_device", NoDevice)
    ext = TileExt()
    monkeypatch.setattr(ext, "_caching", lambda: False)
    return ext


def _tensors(changes=()):
    x = [torch.empty(s, dtype=torch.int32 if i in (5, 6) else torch.float32, device="cuda") for i, s in enumerate(SHAPES)]
    for i, shape in changes:
        x[i] = torch.empty(shape, device="cuda")
    return x


def _queued(ext, x, precision="bf16"):
    tail = torch.empty(96, dtype=torch.uint8, device="cuda")
    binned = (x[5], x[6], tail[:32].view(torch.int64), tail, 64, 1, {}, None)
    return ext.render_frame_queued(x[0], x[1], *x[2:5], x[7], x[8], x[9:], None, None, W, H, 1e-3, precision, binned=binned)


CALLS = {
    "tilecenter": lambda ext, x: ext.render_tiles_forward_tilecenter(*x, W, H, 8, 8, 1e-3),
    "per_pixel": lambda ext, x: ext.render_tiles_forward(*x, W, H, 8, 8, 1e-3),
    "queued_f32": lambda ext, x: _queued(ext, x, "f32"),
    "queued_bf16": _queued,
}
SHORT = [[(1, (W * H - 1, 3))], [(3, (N - 1, 3))], [(4, (N - 1, 4))], [(8, (5,))]]
SHORT += [[(i, (N - 1, *SHAPES[i][1:]))] for i in range(9, 15)]
SHORT += [[(10, (N, 16))], [(11, (N, 64, 64))], [(11, (N, 32, 16))], [(12, (N, 31))], [(13, (N, 3, 32))], [(14, (N, 3))],
          [(9, (N, 16, 72))], [(9, (N + 1, 32, 72))], [(i, (N - 1, *SHAPES[i][1:])) for i in range(9, 15)]]


@pytest.mark.parametrize("call", CALLS.values(), ids=CALLS)
@pytest.mark.parametrize("changes", SHORT, ids=str)
def test_frames_refuse_tensors_their_kernels_would_read_past(ext, call, changes):
    with FakeTensorMode():
        with pytest.raises(RuntimeError):
            call(ext, _tensors(changes))


@pytest.mark.parametrize("call", CALLS.values(), ids=CALLS)
def test_frames_take_what_they_took(ext, call):
    more = [(i, (N + 2, *SHAPES[i][1:])) for i in (3, 4, *range(9, 15))]
    for changes in ((), more, [(10, (N, 32, 1)), (14, (N, 1, 4))], [(8, (7,))]):
        with FakeTensorMode(), pytest.raises(Reached):
            call(ext, _tensors(changes))
    with FakeTensorMode(), pytest.raises(Reached):
        x = _tensors()
        call(ext, [t[:0] if t.shape[0] == N and i not in (5, 6) else t for i, t in enumerate(x)])


@pytest.mark.parametrize("precision", ["f32", "bf16"])
def test_a_queued_frame_refuses_rays_its_kernels_would_misread(ext, precision):
    for i in (0, 1):
        for change in (lambda t: t[:1], lambda t: t[0], lambda t: t.double(), lambda t: t.half(), lambda t: t.cpu(),
                       lambda t: torch.cat([t, t], 1)[:, :3]):
            with FakeTensorMode():
                x = _tensors()
                x[i] = change(x[i])
                with pytest.raises(RuntimeError, match="float32"):
                    _queued(ext, x, precision)


@pytest.mark.parametrize("shapes", [((N, 3), (N - 1, 3)), ((N, 2), (N, 3)), ((N, 3), (N, 2)), ((N,), (N,))], ids=str)
def test_binning_refuses_primitives_that_do_not_go_together(ext, shapes):
    from mlp_splatting_amd.camera import ray_cone_candidates
    with FakeTensorMode(allow_non_fake_inputs=True):
        p, s = (torch.empty(x, device="cuda") for x in shapes)
        rays, eye = torch.empty(W * H, 3, device="cuda"), torch.empty(4, 4, device="cuda")
        for call in (lambda: ops.bin_legacy(p, s, eye, eye, W, H, 8, 1e-3),
                     lambda: ops.bin_legacy_async(p, s, eye, eye, W, H, 8, 1e-3, 64),
                     lambda: ops.bin_segments_async(p, s, eye, eye, W, H, 8, 1e-3),
                     lambda: ray_cone_candidates(rays, rays, p, s, W, H, 8, 1e-3),
                     lambda: ops.prepare_primitives(p, s, torch.empty(N, 4, device="cuda"))):
            with pytest.raises(RuntimeError, match="primitive count"):
                call()
