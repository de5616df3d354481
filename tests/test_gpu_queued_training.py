"""Differentiable frames whose lists are queued behind no read-back of their own: what they return is what the frame that waits
for its binning returns, and what was refused is refused."""
import pytest
import torch

from mlp_splatting_amd import cumodel, synthetic
from mlp_splatting_amd.cumodel import NeuralPrimitiveSceneTileCUDA

pytestmark = pytest.mark.gpu

WIDTH, HEIGHT, FOCAL = 61, 43, 60.0


def _scene(device, channels):
    torch.manual_seed(0)
    sc = synthetic.make_scene(400, 32, seed=3, log_scale_mean=-2.0)
    scene = NeuralPrimitiveSceneTileCUDA(num_primitives=sc.n, hidden_dim=32, feature_dim_low=channels).to(device)
    with torch.no_grad():
        for name, value in zip(("positions", "log_scales", "quats", "W1", "b1", "W2", "b2", "W3", "b3"),
                               (sc.positions, sc.log_scales, sc.quats, *sc.mlp())):
            getattr(scene, name).copy_(torch.as_tensor(value))
        if channels:
            scene.feat_attr.normal_(0, 0.1)
    scene.set_image_size(WIDTH, HEIGHT)
    return scene.train()


def _camera(device, eye, on_device=True):
    c2w = synthetic.look_at(eye)
    rays = [torch.as_tensor(r).to(device) for r in synthetic.pinhole_rays(WIDTH, HEIGHT, FOCAL, c2w)]
    matrices = [torch.as_tensor(m) for m in (synthetic.view_matrix(c2w), synthetic.projection_matrix(FOCAL, WIDTH, HEIGHT))]
    return rays, [m.to(device) if on_device else m for m in matrices]


def _step(scene, rays, matrices, target):
    scene.zero_grad(set_to_none=True)
    more = {} if target is None else {"return_feature": True, "feature_target": target}
    out = scene(*rays, score_threshold=1e-3, view_matrix=matrices[0], proj_matrix=matrices[1], **more)
    rgb, loss = (out, 0.0) if target is None else out
    (rgb.square().sum() + loss).backward()
    return [rgb.detach().clone()] + [p.grad.clone() for p in scene.parameters() if p.grad is not None]


@pytest.fixture
def fresh(monkeypatch):
    monkeypatch.setattr(cumodel, "_tile_ext", None)
    monkeypatch.setattr(cumodel, "_tile_ext_key", None)


@pytest.mark.parametrize("on_device", [True, False])
@pytest.mark.parametrize("backend", [None, "scalar", "wmma_fp16"])
def test_queued_lists_give_what_read_back_ones_give(device, fresh, monkeypatch, backend, on_device):
    """With the estimates of other frames, with none, with too little room for the candidates."""
    scene = _scene(device, 20 if backend else 0)
    target = None
    if backend:
        monkeypatch.setenv("MLPSP_CSR_FORWARD_BACKEND", backend)
        target = torch.randn(11, 15, 20, device=device)
    eyes = [(0.2, -0.1, -0.9), (-0.4, 0.3, 0.5)]
    cameras = [_camera(device, eye, on_device) for eye in eyes]
    scene.queued_frames = False
    want = [_step(scene, *camera, target) for camera in cameras]
    del scene.queued_frames
    ext = scene._ensure_tile_ext()
    queued = []
    whole = ext.train_lists_queued
    monkeypatch.setattr(ext, "train_lists_queued", lambda *a: queued.append(whole(*a)) or queued[-1])
    for capacity in (None, 0, 64, None):
        if capacity is not None:
            ext._queue_capacity = capacity
        for camera, expected in zip(cameras, want):
            queued.clear()
            got = _step(scene, *camera, target)
            assert len(queued) == 1 and len(got) == len(expected)
            for a, b in zip(got, expected):
                assert torch.equal(a, b)
    assert queued[0] is not None and ext._queue_capacity > 64


@pytest.mark.parametrize("backend", [None, "wmma_fp16"])
def test_queued_lists_beyond_the_capacity_are_refused(device, fresh, monkeypatch, backend):
    scene = _scene(device, 4 if backend else 0)
    target = None
    if backend:
        monkeypatch.setenv("MLPSP_CSR_FORWARD_BACKEND", backend)
        target = torch.randn(11, 15, 4, device=device)
    camera = _camera(device, (0.2, -0.1, -0.9))
    _step(scene, *camera, target)
    ext = scene._ensure_tile_ext()
    ext.max_tile_prims = 3
    before = ext.training_wmma_safety_stats()
    with pytest.raises(RuntimeError, match="tile candidate capacity 3 exceeded"):
        _step(scene, *camera, target)
    assert ext.training_wmma_safety_stats() == before


def test_queued_frames_with_inputs_that_are_not_finite_are_refused_and_not_counted(device, fresh, monkeypatch):
    monkeypatch.setenv("MLPSP_CSR_FORWARD_BACKEND", "wmma_fp16")
    scene, camera = _scene(device, 4), _camera(device, (0.2, -0.1, -0.9))
    target = torch.randn(11, 15, 4, device=device)
    for turn in range(2):
        _step(scene, *camera, target)
    ext = scene._ensure_tile_ext()
    before = ext.training_wmma_safety_stats()
    assert before[0] == 2
    for name in ("W2", "b3", "positions"):
        with torch.no_grad():
            kept = getattr(scene, name).clone()
            getattr(scene, name)[-1] = float("nan")
        with pytest.raises(RuntimeError, match="input is nonfinite"):
            _step(scene, *camera, target)
        with torch.no_grad():
            getattr(scene, name).copy_(kept)
    assert ext.training_wmma_safety_stats() == before


def test_a_queued_frame_that_overflows_its_operands_is_repeated_in_f32(device, fresh, monkeypatch):
    monkeypatch.setenv("MLPSP_CSR_FORWARD_BACKEND", "wmma_fp16")
    scene, camera = _scene(device, 4), _camera(device, (0.2, -0.1, -0.9))
    target = torch.randn(11, 15, 4, device=device)
    _step(scene, *camera, target)
    with torch.no_grad():
        scene.W2.mul_(1e6)
    ext = scene._ensure_tile_ext()
    with pytest.warns(UserWarning, match="numeric overflow"):
        got = _step(scene, *camera, target)
    assert ext.training_wmma_safety_stats()[:3] == [2, 1, 0]
    scene.queued_frames = False
    with pytest.warns(UserWarning, match="numeric overflow"):
        want = _step(scene, *camera, target)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("what", ["room", "lists", "numbers"])
def test_a_frame_that_is_repeated_gives_its_workspace_up_first(device, fresh, monkeypatch, what):
    """Too little room for the steps, lists cut short, operands beyond fp16: before the repetition makes its workspace, nothing
    holds the one it replaces."""
    import weakref
    from mlp_splatting_amd import _lib, ops
    monkeypatch.setenv("MLPSP_CSR_FORWARD_BACKEND", "wmma_fp16")
    scene, camera = _scene(device, 4), _camera(device, (0.2, -0.1, -0.9))
    target = torch.randn(11, 15, 4, device=device)
    _step(scene, *camera, target)
    ext, lib, made, gone = scene._ensure_tile_ext(), _lib.load(), [], []

    class Buffer(ops.TrainBuffer):
        def __init__(self, *a):
            super().__init__(*a)
            made.append(weakref.ref(self.bytes))

    class Spy:
        def __getattr__(self, name):
            if name == "mlpsp_train_workspace_bytes" and made:
                gone.append([ref() is None for ref in made])
            return getattr(lib, name)
    monkeypatch.setattr(ops, "TrainBuffer", Buffer)
    monkeypatch.setattr(_lib, "load", lambda: Spy())
    if what == "room":
        ext._steps_per_tile = 0.5
    elif what == "lists":
        ext._queue_capacity = 64
    else:
        with torch.no_grad():
            scene.W2.mul_(1e6)
    if what == "numbers":
        with pytest.warns(UserWarning, match="numeric overflow"):
            _step(scene, *camera, target)
    else:
        _step(scene, *camera, target)
    assert gone == [[True]]


@pytest.mark.parametrize("backend", [None, "wmma_fp16"])
def test_lists_have_room_for_what_training_frames_needed(device, fresh, monkeypatch, backend):
    """The lists of a queued training frame hold three tenths more than the frames before needed, a tile, and 65,536: not what a
    frame of many candidates needed that was only rendered.  One that needs more is repeated, and the next one has the room."""
    scene = _scene(device, 4 if backend else 0)
    target = None
    if backend:
        monkeypatch.setenv("MLPSP_CSR_FORWARD_BACKEND", backend)
        target = torch.randn(11, 15, 4, device=device)
    camera = _camera(device, (0.2, -0.1, -0.9))
    want = _step(scene, *camera, target)
    ext = scene._ensure_tile_ext()
    pairs = ext._queue_capacity                        # (1.3 pairs + 65,536 by the first frame)
    ext.note_frame_pairs(50_000_000)
    sizes, whole = [], ext.train_lists_queued
    monkeypatch.setattr(ext, "train_lists_queued", lambda *a: (lambda q: sizes.append(q.candidates.numel()) or q)(whole(*a)))
    for _ in range(3):
        assert all(torch.equal(a, b) for a, b in zip(_step(scene, *camera, target), want))
    assert len(sizes) == 3 and all(abs(size - pairs) <= 2 for size in sizes)
    ext._pairs_per_tile *= 64.0
    _step(scene, *camera, target)
    assert sizes[3] > sizes[2] and ext._pairs_per_tile < 64.0 * (sizes[0] - 65_536) / 48 * 0.99
    ext._pairs_per_tile, ext._queue_capacity = 0.0, 256
    for _ in range(2):
        assert all(torch.equal(a, b) for a, b in zip(_step(scene, *camera, target), want))
    assert sizes[4] == 256 and abs(sizes[5] - pairs) <= 2
