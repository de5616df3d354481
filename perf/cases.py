"""Performance cases of the tile renderer: the work a user's program has it do, through the scene module's public calls.

A case is a dict of plain values:

  kind        frame          one camera, ``scene(rays_o, rays_d, view_matrix=, proj_matrix=)``
              sequence       several cameras in one ``scene.render_frames`` call (an evaluation loop, a fly-through)
              mosaic         four views in one image: tile lists for a view per tile, then ``scene(...)`` on those lists
              feature        one camera, RGB and the gated feature image (``return_feature=True``)
              train          a differentiable RGB frame, L1 image loss, backward: the nine parameter gradients
              train_feature  a training step with the streamed feature loss: ten parameter gradients
  primitives  size of the scene
  width, height, focal, threshold   the camera's image (for the mosaic: of one view) and the score threshold
  hidden      hidden width of the per-primitive MLP: 16 or 32 (the matrix-core renders exist for 32)
  precision   f32 (exact), bf16 or fp16 operands of the MLP
  channels    width of the feature attributes (0: none)
  views       cameras in one call

The scene is what such a program keeps from call to call: it depends on the sizes in the case alone and is made once.
The seed chooses what is new with every call: the cameras (centres inside the scene, as in ``synthetic.random_poses``)
and the training targets.  The scenes are those of ``synthetic.make_scene`` -- primitives uniform in a cube of four units,
30 % of them in a cluster for the mosaic, log-normal scales, weights of 0.1 -- drawn on the device.
"""
import functools
import math
import os

import torch

from mlp_splatting_amd import synthetic
from mlp_splatting_amd.cumodel import NeuralPrimitiveSceneTileCUDA

DEVICE = "cuda"
MLP_FLOPS = {16: 2 * (72 * 16 + 16 * 16 + 4 * 16), 32: 2 * (72 * 32 + 32 * 32 + 4 * 32)}


def _case(name, kind, primitives, width, height, precision, focal=None, threshold=5e-3, hidden=32, channels=0, views=1):
    case = dict(kind=kind, primitives=primitives, width=width, height=height, focal=float(focal or width / 2.0),
                threshold=threshold, hidden=hidden, precision=precision, channels=channels, views=views)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # a thumbnail of a small scene with the narrow MLP, exact arithmetic: the shortest call there is
        _case("frame_5k_160x120_f32", "frame", 5000, 160, 120, "f32", 150.0, 1e-3, hidden=16),
        # an interactive preview: latency of one call decides
        _case("frame_20k_320x240_bf16", "frame", 20000, 320, 240, "bf16", 300.0),
        # a medium scene, image sides that are no multiples of the tile, the other operand type of the matrix cores
        _case("frame_50k_641x479_fp16", "frame", 50000, 641, 479, "fp16", 600.0, 1e-3),
        # the full-size frame of an evaluator on the matrix cores, and with exact arithmetic
        _case("frame_200k_1200x680_bf16", "frame", 200000, 1200, 680, "bf16", 600.0),
        _case("frame_200k_1200x680_f32", "frame", 200000, 1200, 680, "f32", 600.0),
        # an evaluation loop that hands over eight cameras at a time
        _case("sequence_100k_800x450_bf16", "sequence", 100000, 800, 450, "bf16", 400.0, views=8),
        # four full-size views of a clustered scene in one call
        _case("mosaic_200k_2400x1360_bf16", "mosaic", 200000, 1200, 680, "bf16", 600.0, views=4),
        # open-vocabulary evaluation: RGB and the 512-channel feature image
        _case("feature_200k_1200x680_512ch_bf16", "feature", 200000, 1200, 680, "bf16", 600.0, channels=512),
        # a small feature head with exact arithmetic, ragged image and channel count
        _case("feature_30k_333x251_67ch_f32", "feature", 30000, 333, 251, "f32", 300.0, channels=67),
        # training steps: a small image (many launches, little work), the full frame, and the full frame with features
        _case("train_20k_320x240_f32", "train", 20000, 320, 240, "f32", 300.0),
        _case("train_200k_1200x680_f32", "train", 200000, 1200, 680, "f32", 600.0),
        _case("train_feature_200k_1200x680_512ch_fp16", "train_feature", 200000, 1200, 680, "fp16", 600.0, channels=512),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """One more case: scenes of 5,000 to 200,000 primitives and images of 160x120 to 1200x680 pixels of any aspect from
    portrait to wide (mosaic views in whole tiles), every kind with the precisions it is used in.  The small images go
    with the small scenes (at most 1.5 primitives per squared unit of focal length): a tile is then a wide cone, and the
    lists of a large scene would not fit it however small its primitives are."""
    kind = rng.choice(["frame"] * 5 + ["feature"] * 2 + ["train"] * 2 + ["sequence", "mosaic", "train_feature"])
    pixels = _log_uniform(rng, 160 * 120, 1200 * 680)
    aspect = rng.uniform(0.75, 1.8)
    width = max(64, int(math.sqrt(pixels * aspect)))
    height = max(64, int(pixels / width))
    focal = width * rng.uniform(0.5, 0.95)
    primitives = int(_log_uniform(rng, 5000, max(10000.0, min(200000.0, 1.5 * focal * focal))))
    threshold = rng.choice([1e-3, 5e-3])
    hidden, channels, views = 32, 0, 1
    if kind == "frame":
        precision = rng.choice(["f32", "bf16", "fp16"])
        if precision == "f32" and rng.random() < 0.25:
            hidden = 16
    elif kind == "sequence":
        precision, views = rng.choice(["bf16", "fp16"]), rng.randint(3, 8)
    elif kind == "mosaic":
        precision, views = rng.choice(["f32", "bf16", "bf16"]), 4
        width, height = width // 8 * 8, height // 8 * 8
    elif kind == "feature":
        precision, channels = rng.choice(["f32", "bf16", "bf16"]), int(_log_uniform(rng, 16, 512))
    elif kind == "train":
        precision = "f32"
    else:
        precision, channels = rng.choice(["f32", "fp16", "bf16"]), int(_log_uniform(rng, 16, 512))
    return _case(None, kind, primitives, width, height, precision, focal, threshold, hidden, channels, views)


# ---------------------------------------------------------------------------------------------------------------------
# scene and cameras
# ---------------------------------------------------------------------------------------------------------------------
def _reach(case):
    """Standard deviations at which a primitive's falloff reaches the threshold."""
    return math.sqrt(-2.0 * math.log(case["threshold"]))


def _log_scale_mean(case):
    """Mean log-scale: -3, or what keeps the fullest tile's list at about three quarters of the 1,536 candidates that the
    renderer takes.  A primitive is listed where a square of its largest semi-axis overlaps the tile, so a list grows with
    primitives x (support + tile)^2, both seen about two units away; the constant is that of the 200,000-primitive
    1200x680 scene at -3.95."""
    side = 2.0 * 1.6
    reference = 2e5 * (side * 3.255 * math.exp(-3.95) + 8 * 2.0 / 600.0) ** 2
    support = math.sqrt(reference / case["primitives"]) - 8 * 2.0 / case["focal"]
    mean = math.log(max(support, 1e-3) / (side * _reach(case)))
    return min(-3.0, mean) - (2.4 if case["kind"] == "mosaic" else 0.0)


@functools.lru_cache(maxsize=1)
def _scene(primitives, hidden, channels, log_scale_mean, clustered):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(0)
    with torch.device(DEVICE):
        scene = NeuralPrimitiveSceneTileCUDA(num_primitives=primitives, hidden_dim=hidden, feature_dim_low=channels)

    def normal(parameter, std, mean=0.0):
        parameter.normal_(mean, std, generator=gen)

    with torch.no_grad():
        scene.positions.uniform_(-2.0, 2.0, generator=gen)
        if clustered:
            scene.positions[:int(0.3 * primitives)] *= 0.125
        normal(scene.log_scales, 0.5, log_scale_mean)
        normal(scene.quats, 1.0)
        scene.quats.copy_(torch.nn.functional.normalize(scene.quats, dim=-1))
        for weight in (scene.W1, scene.b1, scene.W2, scene.b2, scene.W3, scene.b3):
            normal(weight, 0.1)
        normal(scene.b3[:, 3], 1.0)
        if channels:
            normal(scene.feat_attr, 0.05)
    return scene


def _cameras(case, gen):
    """[(view matrix, rays_o, rays_d)] of the case's cameras, the matrices and rays of ``synthetic`` on the device."""
    width, height, focal = case["width"], case["height"], case["focal"]
    j, i = torch.meshgrid(torch.arange(height, dtype=torch.float32, device=DEVICE),
                          torch.arange(width, dtype=torch.float32, device=DEVICE), indexing="ij")
    pixel = torch.stack([(i - width * 0.5) / focal, (j - height * 0.5) / focal, torch.ones_like(i)], -1).reshape(-1, 3)
    cameras = []
    for _ in range(case["views"]):
        eye = torch.rand(3, generator=gen) * 3.0 - 1.5
        c2w = synthetic.look_at(eye.tolist())
        pose = torch.from_numpy(c2w).to(DEVICE)
        rays_d = (pixel[:, None, :] * pose[None, :3, :3]).sum(-1)
        rays_o = pose[:3, 3].expand_as(rays_d).contiguous()
        cameras.append((torch.from_numpy(synthetic.view_matrix(c2w)).to(DEVICE), rays_o, rays_d))
    return cameras


def _mosaic(case, cameras):
    """(rays_o, rays_d, view of every tile, view matrices) of the 2x2 mosaic, laid out as ``synthetic.mosaic_frame``."""
    width, height, focal = case["width"], case["height"], case["focal"]

    def tiled(images):
        quads = [image.view(height, width, 3) for image in images]
        return torch.cat([torch.cat(quads[:2], 1), torch.cat(quads[2:], 1)], 0).reshape(-1, 3).contiguous()

    columns, rows = 2 * width // 8, 2 * height // 8
    ty, tx = torch.meshgrid(torch.arange(rows, device=DEVICE), torch.arange(columns, device=DEVICE), indexing="ij")
    tile_views = ((ty >= rows // 2) * 2 + (tx >= columns // 2)).reshape(-1).to(torch.int32)
    views = []
    for q, (view, _, _) in enumerate(cameras):
        shear = torch.eye(4, device=DEVICE)
        shear[0, 2] = (q % 2 - 0.5) * width / focal
        shear[1, 2] = (q // 2 - 0.5) * height / focal
        views.append(shear @ view)
    return (tiled([c[1] for c in cameras]), tiled([c[2] for c in cameras]), tile_views, torch.stack(views))


def prepare(case, seed):
    kind = case["kind"]
    scene = _scene(case["primitives"], case["hidden"], case["channels"], _log_scale_mean(case), kind == "mosaic")
    times = 2 if kind == "mosaic" else 1
    width, height = times * case["width"], times * case["height"]
    scene.set_image_size(width, height)
    scene.render_precision = "f32" if kind.startswith("train") else case["precision"]
    host = torch.Generator().manual_seed(seed)
    cameras = _cameras(case, host)
    state = dict(kind=kind, scene=scene, threshold=case["threshold"], size=(width, height), cameras=cameras,
                 proj=torch.from_numpy(synthetic.projection_matrix(case["focal"], width, height)).to(DEVICE))
    if kind == "mosaic":
        state["mosaic"] = _mosaic(case, cameras)
    if kind.startswith("train"):
        gen = torch.Generator(device=DEVICE)
        gen.manual_seed(seed)
        scene.train()
        state["target"] = torch.rand(width * height, 3, device=DEVICE, generator=gen)
        if kind == "train_feature":
            # the feature image of a training view comes at a quarter of the resolution, in half precision
            state["feature_target"] = (torch.randn(height // 4, width // 4, case["channels"], device=DEVICE,
                                                   generator=gen) * 0.05).half()
            backend = {"f32": ("scalar", "float32"), "fp16": ("wmma_fp16", "float16"), "bf16": ("wmma_bf16", "bfloat16")}
            (os.environ["MLPSP_CSR_FORWARD_BACKEND"],
             os.environ["MLPSP_CSR_MLP_PRECISION"]) = backend[case["precision"]]
    else:
        scene.eval()
    return state


def run(state):
    kind, scene, proj, threshold = state["kind"], state["scene"], state["proj"], state["threshold"]
    view, rays_o, rays_d = state["cameras"][0]
    camera = dict(score_threshold=threshold, view_matrix=view, proj_matrix=proj)
    if kind in ("frame", "feature"):
        with torch.inference_mode():
            return scene(rays_o, rays_d, return_feature=kind == "feature", **camera)
    if kind == "sequence":
        with torch.inference_mode():
            return scene.render_frames([(o, d, v, proj) for v, o, d in state["cameras"]], threshold)
    if kind == "mosaic":
        rays_o, rays_d, tile_views, views = state["mosaic"]
        with torch.inference_mode():
            candidates, offsets = scene.build_tilecenter_culling_from_tile_views(tile_views, views, proj, threshold)
            return scene(rays_o, rays_d, score_threshold=threshold, culled_prim_indices=candidates, tile_offsets=offsets)
    scene.zero_grad(set_to_none=True)
    if kind == "train":
        rgb = scene(rays_o, rays_d, **camera)
        loss = (rgb - state["target"]).abs().mean()
    else:
        rgb, feature_loss = scene(rays_o, rays_d, return_feature=True, feature_target=state["feature_target"], **camera)
        loss = (rgb - state["target"]).abs().mean() + 0.5 * feature_loss
    loss.backward()
    out = {name: parameter.grad for name, parameter in scene.named_parameters() if parameter.grad is not None}
    return dict(out, rgb=rgb.detach(), loss=loss.detach())


# ---------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------------
def _hits_per_pixel(case):
    """Primitives that a ray blends: those it meets on the two units or so to the far side of the scene -- density times
    the mean cross-section of the ellipsoids -- or, where there are more, the 45 after which it is opaque."""
    volume = 64.0
    section = math.pi * _reach(case) ** 2 * math.exp(2.0 * _log_scale_mean(case) + 0.25)
    met = 2.0 * case["primitives"] / volume * section
    if case["kind"] == "mosaic":          # 0.3 of the primitives in a 512th of the volume, met over half a unit
        met = 0.7 * met + 0.3 * met * 512.0 * 0.125 * 0.25
    return min(45.0, met)


def work(case):
    """Bytes: geometry (40 per primitive) and rays (24 per pixel) read, images written, training targets read and the
    gradients of every parameter written (the weights that are read are those of the few primitives that rays end in, and
    are left out).  Flops: the MLP of every (pixel, primitive) hit, three times that with its gradient, and the blend of the
    feature channels; hits are estimated."""
    n, pixels = case["primitives"], case["width"] * case["height"] * case["views"]
    hits = _hits_per_pixel(case) * pixels
    hidden, channels = case["hidden"], case["channels"]
    nbytes = 40.0 * n + (24.0 + 12.0) * pixels
    flops = MLP_FLOPS[hidden] * hits
    if case["kind"] == "feature":
        nbytes += 4.0 * channels * pixels
        flops += 2.0 * 4 * channels * hits
    if case["kind"].startswith("train"):
        nbytes += 12.0 * pixels + 4.0 * n * (3 + 3 + 4 + 32 * 72 + 32 + 32 * 32 + 32 + 4 * 32 + 4)
        flops *= 3.0
    if case["kind"] == "train_feature":
        low = (case["width"] // 4) * (case["height"] // 4)
        nbytes += 2.0 * channels * low + 4.0 * n * 4 * channels
        # the four source pixels of every target pixel, forward and adjoint
        flops += 2.0 * 2.0 * 4 * channels * _hits_per_pixel(case) * 4 * low
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """f32: sums in another order; a hit or an opaque pixel decided the other way by a rounding moves one pixel by up to
    the threshold.  bf16/fp16 operands: eight and eleven bits, averaged over a pixel's hits.  Gradients: longer sums, and
    with reduced operands a residual near zero may change the sign that the L1 losses pass on."""
    if case["kind"] == "train":
        return {"rel": 1e-4, "max": 2e-2}
    if case["kind"] == "train_feature":
        return {"rel": 1e-3, "max": 0.3} if case["precision"] == "f32" else {"rel": 1e-2, "max": 0.5}
    if case["precision"] == "f32":
        return {"rel": 1e-5, "max": 1e-2}
    return {"rel": 4e-3 if case["precision"] == "bf16" else 1e-3, "max": 5e-2}
