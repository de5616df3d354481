"""The training-step kernels (one step per tile x primitive) against the per-pixel record pipeline, which the float64
restatement of test_gpu_training.py pins: ragged frames, a frame without hits, a single tile, primitives whose steps
span many chunks, a pool that has to be drawn again, each operand type of the weight gradients."""
import pytest
import torch

from conftest import to_dev
from helpers import Frame

pytestmark = pytest.mark.gpu

#        primitives, width, height, scale of the primitives, camera turned away
CASES = [(40, 5, 3, 2.0, False), (300, 33, 17, 1.0, False), (300, 32, 24, 1.0, True), (3, 96, 80, 30.0, False),
         (1500, 80, 48, 1.0, False)]


def _scene(device, oracle_mod, n, width, height, scale, away):
    import numpy as np
    fr = Frame("cfg1_5k_160x120", n=n, hidden=32, width=width, height=height,
               **({"eye": (0.0, 0.0, -50.0), "target": (0.0, 0.0, -90.0)} if away else {}))
    fr.scene.log_scales += np.float32(np.log(scale))
    cand, off = fr.oracle_lists(oracle_mod)
    base = [to_dev(a, device) for a in fr.base_numpy(cand, off)]
    return fr, base


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 2e-5), (torch.float16, 3e-3), (torch.bfloat16, 3e-2)])
@pytest.mark.parametrize("n,width,height,scale,away", CASES)
def test_gradients_of_steps_are_those_of_records(device, oracle_mod, n, width, height, scale, away, dtype, tol):
    from mlp_splatting_amd import ops
    from mlp_splatting_amd.tile_ext import TileExt
    fr, base = _scene(device, oracle_mod, n, width, height, scale, away)
    ext = TileExt()
    ext._steps_per_tile = 16 if n == 1500 else 96             # 16: too little room, the forward repeats with more
    x = base + [torch.zeros_like(base[0]), torch.zeros(width * height, device=device)]
    records = ext.render_tiles_training_records(x, width, height, 8, fr.thr, 1.5, 2.0, render_order=True)
    rgb, alpha, frame = ext.train_forward(base, width, height, fr.thr)
    assert torch.equal(rgb, records[0]) and torch.equal(alpha, records[1]) and frame.status == 0
    assert (frame.steps == 0) == (records[2].numel() == 0) and not (away and frame.steps)
    torch.manual_seed(3)
    g_rgb, g_t = torch.randn(width * height, 3, device=device), torch.randn(width * height, device=device)
    mlp = base[9:15]
    want = ext.backward_from_records(records, base[2], base[3], base[4], base[7], base[8], *mlp, g_rgb, g_t)
    got = ext.backward_from_steps(frame, ops.train_group(frame, base[6], n), base, g_rgb, g_t, dtype=dtype)
    assert len(got) == 9
    for i, (g, w) in enumerate(zip(got, want)):
        assert g.shape == w.shape and torch.isfinite(g).all()
        bound = tol if i < 6 else 2e-5
        assert float((g - w).norm()) <= bound * float(w.norm()), (i, float((g - w).norm()), float(w.norm()))
        assert torch.equal(g[w.reshape(n, -1).abs().amax(1) == 0], torch.zeros_like(g[w.reshape(n, -1).abs().amax(1) == 0]))


@pytest.mark.parametrize("precision", ["float16", "bfloat16"])
def test_reduced_forward_steps_are_those_of_its_records(device, oracle_mod, precision):
    """The matrix-core forward of the steps against the matrix-core record forward: image, hits and output adjoints."""
    from mlp_splatting_amd import ops
    from mlp_splatting_amd.tile_ext import TileExt
    fr, base = _scene(device, oracle_mod, 300, 33, 17, 1.0, False)
    ext = TileExt()
    x = base + [torch.zeros_like(base[0]), torch.zeros(33 * 17, device=device)]
    records = ext.render_tiles_training_records_wmma(x, 33, 17, 8, fr.thr, 1.5, 2.0, precision)
    rgb, alpha, frame = ext.train_forward(base, 33, 17, fr.thr, render_order=False, precision=precision)
    assert frame.status == 0
    torch.testing.assert_close(rgb, records[0], atol=2e-6, rtol=0)
    torch.testing.assert_close(alpha, records[1], atol=2e-6, rtol=0)
    torch.manual_seed(4)
    g_rgb, g_t = torch.randn(33 * 17, 3, device=device), torch.randn(33 * 17, device=device)
    want = ext.backward_from_records(records, base[2], base[3], base[4], base[7], base[8], *base[9:15], g_rgb, g_t)
    got = ext.backward_from_steps(frame, ops.train_group(frame, base[6], 300), base, g_rgb, g_t)
    for i, (g, w) in enumerate(zip(got, want)):
        assert float((g - w).norm()) <= 1e-4 * float(w.norm()), i


#                target, channels, slots
@pytest.mark.parametrize("wf,hf,channels,slots", [
    (33, 17, 5, 4),        # a target for every pixel: nine taps to a tile and axis, shared between tiles
    (8, 4, 64, 4), (8, 4, 67, 5), (8, 4, 516, 1),     # a quarter; one, two and four lane groups; more than one wavefront
    (13, 7, 130, 5),       # a ratio that is no whole number
    (3, 2, 256, 4),        # more pixels than a tile between two targets: tiles without one
    (33, 17, 144, 4), (8, 4, 128, 4), (13, 7, 528, 4),      # sixteens of channels, whole and with a remainder
    (1, 1, 3, 1)])
@pytest.mark.parametrize("half", [False, True])
def test_feature_loss_of_steps_is_that_of_records(device, oracle_mod, wf, hf, channels, slots, half):
    from mlp_splatting_amd import ops, primitive_csr, record_feature_loss
    from mlp_splatting_amd.tile_ext import TileExt
    fr, base = _scene(device, oracle_mod, 300, 33, 17, 1.0, False)
    ext = TileExt()
    gen = torch.Generator(device=device).manual_seed(7)
    attributes = torch.randn(300, slots, channels, device=device, generator=gen)
    attributes = attributes[:, 0].contiguous() if slots == 1 else attributes
    target = torch.randn(hf, wf, channels, device=device, generator=gen)
    target = target.half() if half else target
    x = base + [torch.zeros_like(base[0]), torch.zeros(33 * 17, device=device)]
    records = ext.render_tiles_training_records(x, 33, 17, 8, fr.thr, 1.5, 2.0)
    want_loss, signs, _ = record_feature_loss.streaming_feature_l1(records, attributes, target, 33, 17)
    csr = primitive_csr.group_records(records[2], records[3], records[3].new_zeros(records[2].numel(), 4), 300, records[5])
    want = record_feature_loss.feature_weight_gradients(records, csr, signs, attributes, 33, 17, mixed=False)
    _, _, frame = ext.train_forward(base, 33, 17, fr.thr, render_order=False)
    loss, feature, kept = ops.train_feature_l1(frame, base[6], attributes, target, 1.5, 2.0)
    got = ops.train_feature_gradients(frame, ops.train_group(frame, base[6], 300), feature, kept, attributes,
                                      torch.tensor(0.75, device=device))
    torch.testing.assert_close(loss, want_loss, rtol=1e-6, atol=0)
    assert got.shape == want.shape
    torch.testing.assert_close(got, want * 0.75, rtol=1e-4, atol=2e-6 * float(want.abs().max()))


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("away", [False, True])
@pytest.mark.parametrize("channels,slots", [(8, 4), (67, 5), (300, 1), (1, 1)])
def test_zeros_of_the_attribute_gradient_beside_the_weight_gradients(device, oracle_mod, channels, slots, away, precision):
    """Rows of primitives without a step from the weight gradients, the others from the attribute gradient: together what the
    attribute gradient writes by itself, and the weight gradients are the same."""
    from mlp_splatting_amd import ops
    from mlp_splatting_amd.tile_ext import TileExt
    fr, base = _scene(device, oracle_mod, 300, 33, 17, 0.3, away)
    _, _, frame = TileExt().train_forward(base, 33, 17, fr.thr)
    gen = torch.Generator(device=device).manual_seed(8)
    attributes = torch.randn(300, slots, channels, device=device, generator=gen)
    target = torch.randn(5, 9, channels, device=device, generator=gen)
    _, feature, kept = ops.train_feature_l1(frame, base[6], attributes, target, 1.5, 2.0)
    groups, one = ops.train_group(frame, base[6], 300), torch.ones(1, device=device)
    d4 = torch.randn(frame.steps, 64, 4, device=device, generator=gen)
    args = (frame, groups, d4, d4[..., 0].contiguous(), base[1], base[7], base[8], base[9:15], base[3], base[4], precision, 1.0)
    rows = torch.full_like(attributes, float("nan"))
    grads, got = ops.train_gradients(*args)[0], ops.train_gradients(*args, rows)[0]
    assert all(torch.equal(a, b) for a, b in zip(grads, got))
    used = torch.zeros(300, dtype=torch.bool, device=device)
    used[groups.view(torch.int32)[320:320 + frame.steps].long()] = True          # (the sorted primitives, behind 301 ints)
    assert (rows[~used] == 0).all() and rows[used].isnan().all() and bool(used.any()) != away and not bool(used.all())
    assert ops.train_feature_gradients(frame, groups, feature, kept, attributes, one, rows) is rows
    assert torch.equal(rows, ops.train_feature_gradients(frame, groups, feature, kept, attributes, one))


def test_feature_training_step_of_an_empty_scene(device, oracle_mod):
    from mlp_splatting_amd.record_training import Frame as TrainingFrame, feature_training_step
    fr, base = _scene(device, oracle_mod, 40, 33, 17, 1.0, False)
    empty = [t[:0].clone() if i in (2, 3, 4, *range(9, 15)) else t for i, t in enumerate(base)]
    empty[5], empty[6] = empty[5][:0].clone(), torch.zeros_like(empty[6])
    leaves = [t.requires_grad_() if i in (2, 3, 4, *range(9, 15)) else t for i, t in enumerate(empty)]
    attributes = torch.zeros(0, 4, 16, device=device, requires_grad=True)
    target = torch.ones(4, 8, 16, device=device)
    rgb, loss = feature_training_step(leaves, attributes, target, TrainingFrame(33, 17, fr.thr, 1.5, 2.0))
    assert float(rgb.detach().abs().max()) == 0.0 and float(loss.detach()) == 1.0
    (rgb.sum() + loss).backward()
    assert attributes.grad.shape == attributes.shape


def test_unit_quaternions_are_those_of_torch(device):
    from mlp_splatting_amd import ops
    gen = torch.Generator(device=device).manual_seed(2)
    q = torch.randn(5000, 4, device=device, generator=gen)
    q[:3] *= torch.tensor([[0.0], [1e-20], [1e18]], device=device)
    g = torch.randn(5000, 4, device=device, generator=gen)
    grads = []
    for f in (ops.unit_quats, lambda t: torch.nn.functional.normalize(t, dim=-1)):
        leaf = q.clone().requires_grad_()
        u = f(leaf)
        u.backward(g)
        grads.append((u.detach(), leaf.grad))
    assert torch.equal(grads[0][0], grads[1][0])
    torch.testing.assert_close(grads[0][1], grads[1][1], rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("backend", ["scalar", "wmma_fp16"])
def test_feature_training_step_refuses_weights_stored_in_half_precision(device, oracle_mod, monkeypatch, backend):
    from mlp_splatting_amd.record_training import Frame as TrainingFrame, feature_training_step
    monkeypatch.setenv("MLPSP_CSR_FORWARD_BACKEND", backend)
    fr, base = _scene(device, oracle_mod, 40, 33, 17, 1.0, False)
    target, attributes = torch.zeros(4, 8, 16, device=device), torch.zeros(40, 4, 16, device=device)
    half = [t.half() if i >= 9 else t for i, t in enumerate(base)]
    short = [t[:39].contiguous() if i in (11, 13) else t for i, t in enumerate(base)]
    for bad, text in ((half, "requires FP32 inputs"), (short, None)):
        with pytest.raises(RuntimeError, match=text):
            feature_training_step(bad, attributes, target, TrainingFrame(33, 17, fr.thr, 1.5, 2.0))


def _frame_with_holes(device, oracle_mod):
    """Small primitives: tiles where some pixels are hit and others by nothing at all."""
    from mlp_splatting_amd.tile_ext import TileExt
    fr, base = _scene(device, oracle_mod, 300, 33, 17, 0.35, False)
    ext = TileExt()
    x = base + [torch.zeros_like(base[0]), torch.zeros(33 * 17, device=device)]
    records = ext.render_tiles_training_records(x, 33, 17, 8, fr.thr, 1.5, 2.0, render_order=True)
    empty = records[7].diff() == 0
    pixel = torch.arange(33 * 17, device=device)
    tile = (pixel // 33) // 8 * 5 + (pixel % 33) // 8
    beside_hits = torch.isin(tile[empty], tile[~empty])
    assert int(beside_hits.sum()) > 20 and int((~empty).sum()) > 20
    return fr, base, ext, records, empty


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf")])
def test_pixels_that_nothing_hits_contribute_nothing_whatever_their_adjoint(device, oracle_mod, value, dtype):
    from mlp_splatting_amd import ops
    fr, base, ext, records, empty = _frame_with_holes(device, oracle_mod)
    _, _, frame = ext.train_forward(base, 33, 17, fr.thr)
    groups = ops.train_group(frame, base[6], 300)
    torch.manual_seed(5)
    g_rgb, g_t = torch.randn(33 * 17, 3, device=device), torch.randn(33 * 17, device=device)
    g_rgb[empty], g_t[empty] = 0.0, 0.0
    want = ext.backward_from_steps(frame, groups, base, g_rgb, g_t, dtype=dtype)
    for rgb_too, t_too in ((True, False), (False, True), (True, True)):
        b_rgb, b_t = g_rgb.clone(), g_t.clone()
        if rgb_too:
            b_rgb[empty] = value
        if t_too:
            b_t[empty] = value
        got = ext.backward_from_steps(frame, groups, base, b_rgb, b_t, dtype=dtype)
        for g, w in zip(got, want):
            assert torch.equal(g, w) and bool(torch.isfinite(g).all())


def test_a_pixel_with_hits_and_a_non_finite_adjoint_is_refused_as_by_the_record_pipeline(device, oracle_mod):
    from mlp_splatting_amd import ops
    fr, base, ext, records, empty = _frame_with_holes(device, oracle_mod)
    _, _, frame = ext.train_forward(base, 33, 17, fr.thr)
    g_rgb, g_t = torch.zeros(33 * 17, 3, device=device), torch.zeros(33 * 17, device=device)
    g_rgb[(~empty).nonzero()[0]] = float("inf")
    with pytest.raises(FloatingPointError):
        ext.backward_from_records(records, base[2], base[3], base[4], base[7], base[8], *base[9:15], g_rgb, g_t)
    with pytest.raises(FloatingPointError):
        ext.backward_from_steps(frame, ops.train_group(frame, base[6], 300), base, g_rgb, g_t)


@pytest.mark.parametrize("background", [None, 0.5])
def test_a_loss_whose_derivative_is_infinite_at_black_pixels_trains(device, background):
    """rgb ** (1 / 2.2) at an empty pixel on black: an infinite adjoint, which ends there."""
    from mlp_splatting_amd import synthetic as syn
    from mlp_splatting_amd.cumodel import NeuralPrimitiveSceneTileCUDA
    sc = syn.make_scene(300, 32, seed=0, log_scale_mean=-4.0)
    scene = NeuralPrimitiveSceneTileCUDA(num_primitives=300, hidden_dim=32).to(device)
    with torch.no_grad():
        for name, value in zip(("positions", "log_scales", "quats", "W1", "b1", "W2", "b2", "W3", "b3"),
                               (sc.positions, sc.log_scales, sc.quats, *sc.mlp())):
            getattr(scene, name).copy_(to_dev(value, device))
    width, height, focal = 64, 48, 60.0
    scene.set_image_size(width, height)
    c2w = syn.look_at((0.2, -0.1, -3.0), (0.0, 0.0, 0.0))
    ro, rd = (to_dev(a, device) for a in syn.pinhole_rays(width, height, focal, c2w))
    args = dict(score_threshold=5e-3, view_matrix=to_dev(syn.view_matrix(c2w), device),
                proj_matrix=to_dev(syn.projection_matrix(focal, width, height), device))
    rgb = scene(ro, rd, bg_color=None if background is None else (0.0, background, 0.0), **args)
    empty = (rgb == 0).any(-1)
    assert 20 < int(empty.sum()) < width * height - 20
    rgb.retain_grad()
    (rgb ** (1 / 2.2)).mean().backward()
    assert not bool(torch.isfinite(rgb.grad[empty]).all())
    for parameter in (scene.positions, scene.log_scales, scene.quats, scene.W1, scene.b3):
        assert bool(torch.isfinite(parameter.grad).all()) and float(parameter.grad.abs().max()) > 0


@pytest.mark.parametrize("channels,slots", [(8, 4), (67, 5), (300, 1)])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_attributes_that_no_target_samples_may_be_anything(device, oracle_mod, value, channels, slots):
    """A primitive that hits a tile, but none of the pixels that the tile's targets take: its attributes reach no target."""
    from mlp_splatting_amd import ops
    fr, base, ext, records, empty = _frame_with_holes(device, oracle_mod)
    wf, hf = 8, 4
    taps = []
    for size, low in ((33, wf), (17, hf)):
        at = ((torch.arange(low, device=device) + 0.5) * (size / low) - 0.5).clamp_min(0).long()
        taps.append(torch.cat([at, (at + 1).clamp_max(size - 1)]).unique())
    sampled = torch.zeros(17, 33, dtype=torch.bool, device=device)
    sampled[taps[1][:, None], taps[0][None, :]] = True
    pixel = torch.repeat_interleave(torch.arange(33 * 17, device=device), records[7].diff())
    is_hit, is_sampled = torch.zeros(300, dtype=torch.bool, device=device), torch.zeros(300, dtype=torch.bool, device=device)
    is_hit[records[2].long()] = True
    is_sampled[records[2].long()[sampled.reshape(-1)[pixel]]] = True
    others = is_hit & ~is_sampled
    assert int(others.sum()) > 5 and int(is_sampled.sum()) > 5
    gen = torch.Generator(device=device).manual_seed(11)
    attributes = torch.randn(300, slots, channels, device=device, generator=gen)
    attributes[others] = 0.0
    target = torch.randn(hf, wf, channels, device=device, generator=gen)
    _, _, frame = ext.train_forward(base, 33, 17, fr.thr, render_order=False)
    groups, one, results = ops.train_group(frame, base[6], 300), torch.ones((), device=device), []
    for fill in (0.0, value):
        attributes[others] = fill
        used = attributes[:, 0].contiguous() if slots == 1 else attributes
        loss, feature, kept = ops.train_feature_l1(frame, base[6], used, target, 1.5, 2.0)
        results.append((loss, ops.train_feature_gradients(frame, groups, feature, kept, used, one)))
    assert torch.equal(results[0][0], results[1][0]) and bool(torch.isfinite(results[1][0]))
    assert torch.equal(results[0][1], results[1][1]) and bool(torch.isfinite(results[1][1]).all())
    attributes[is_sampled] = value
    used = attributes[:, 0].contiguous() if slots == 1 else attributes
    assert not bool(torch.isfinite(ops.train_feature_l1(frame, base[6], used, target, 1.5, 2.0)[0]))


@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("tiles", [1, 3, 4, 5, 15, 16, 17, 31, 129, 255])
def test_weight_gradients_of_runs_of_every_length(device, tiles, precision):
    """The kernels deal a run's half steps to four wavefronts and cut the steps into chunks, here of 16 (those of more are
    test_gpu_weight_gradients.py's): runs of one primitive that are a little shorter and longer, three in a row, against float64
    over the same steps and the forward's phases.  An f32 gradient is a sum of up to 16,000 products of two factors that are f32
    sums of up to 72 terms themselves: a few units of 2^-24 each, 1e-6 of the norm.  In 16 bits (1: fp16, 2: bf16) every factor
    and what it was computed from, eight tensors at the most, is rounded once, by 2^-11 or 2^-8 of it, and a phase moves its sine
    by two roundings, 2^-23 times the largest phase; the adjoints are scaled by 256 and stay above what fp16 holds in full."""
    import numpy as np
    from mlp_splatting_amd import ops, synthetic as syn
    from mlp_splatting_amd.tile_ext import TileExt
    n, width, height = 3, 8 * tiles, 8
    sc = syn.make_scene(n, 32, seed=5, log_scale_mean=2.5)
    sc.positions[:] = np.array([0.0, 0.0, 9.0]) + 0.1 * sc.positions
    sc.b3[:, 3] = -6.0
    c2w = syn.look_at((0.0, 0.0, -3.0), (0.0, 0.0, 5.0))
    ro, rd = syn.pinhole_rays(width, height, 2.0 * width, c2w)
    cand, off = np.tile(np.arange(n, dtype=np.int32), tiles), np.arange(tiles + 1, dtype=np.int32) * n
    base = [to_dev(a, device) for a in (ro, syn.normalize_rays(rd), sc.positions, sc.log_scales, sc.quats, cand, off, sc.freq,
                                        sc.att, *sc.mlp())]
    ext = TileExt()
    x = base + [torch.zeros_like(base[0]), torch.zeros(width * height, device=device)]
    records = ext.render_tiles_training_records(x, width, height, 8, 1e-3, 1.5, 2.0, render_order=True)
    _, _, frame = ext.train_forward(base, width, height, 1e-3)
    assert frame.steps == n * tiles
    g = torch.Generator().manual_seed(6)
    g_rgb, g_t = torch.randn(width * height, 3, generator=g).to(device), torch.randn(width * height, generator=g).to(device)
    d4, falloff = ops.train_reverse(frame, base[6], g_rgb, g_t)
    got, flag = ops.train_gradients(frame, ops.train_group(frame, base[6], n), d4, falloff, base[1], base[7], base[8], base[9:15],
                                    base[3], base[4], precision, 256.0 if precision else 1.0)
    assert int(flag) == 0
    # d4 is [tile, step of the tile, lane]; the records are [pixel, hit], and every pixel hits all three, in the tile's order
    ids, x6 = records[2].view(-1, n), records[3].view(-1, n, 6)
    assert records[2].numel() == n * width * height
    pixel = torch.arange(width * height, device=device)
    tile, lane = (pixel % width) // 8, pixel // width * 8 + pixel % 8
    adjoint = d4.view(tiles, n, 64, 4)[tile[:, None], torch.arange(n, device=device)[None], lane[:, None]].double()
    W1, b1, W2, b2, W3, _ = (w.double() for w in base[9:15])
    for p in range(n):
        at = (ids == p).nonzero(as_tuple=True)
        phase = ((x6[at][:, :, None] * base[7]) * base[8]).reshape(-1, 36).double()
        enc, d = torch.cat([phase.sin(), phase.cos()], 1), adjoint[at]
        z1 = enc @ W1[p].T + b1[p]
        bound = (1e-6, 8 * 2.0 ** -11, 8 * 2.0 ** -8)[precision]
        bound += 2.0 ** -23 * float(phase.abs().max()) if precision else 0.0
        h1 = z1.clamp(min=0.0)
        z2 = h1 @ W2[p].T + b2[p]
        d2 = (d @ W3[p]) * (z2 > 0)
        d1 = (d2 @ W2[p]) * (z1 > 0)
        want = [d1.T @ enc, d1.sum(0), d2.T @ h1, d2.sum(0), d.T @ z2.clamp(min=0.0), d.sum(0)]
        for i, (a, b) in enumerate(zip(got, want)):
            assert float((a[p].double() - b).norm()) <= bound * float(b.norm()), (p, i)


# every tile by a team (40 and 1,681 tiles), then most by one wavefront (2,050 tiles, in rows of 50 and one of 2,050)
@pytest.mark.parametrize("width,height", [(61, 40), (328, 325), (400, 325), (16397, 5)])
def test_tiles_of_every_length_take_the_chunks_they_need(device, width, height):
    """Lists of 0 to 97 primitives that all hit their tile: the steps, and the pool's chunks, of one tile beside another at
    and around the ends of the groups that a tile draws; image and gradients as the records give them."""
    import numpy as np
    from mlp_splatting_amd import _lib, ops, synthetic as syn
    from mlp_splatting_amd.tile_ext import TileExt
    n, tiles = 97, ((width + 7) // 8) * ((height + 7) // 8)
    lengths = np.array([1, 8, 9, 0, 7, 16, 17, 31, 32, 33, 2, 63, 64, 65, 96, 97, 15, 4])[np.arange(tiles) % 18]
    sc = syn.make_scene(n, 32, seed=3, log_scale_mean=1.2)
    sc.positions[:, 2] += 6.0
    sc.b3[:, 3] = -6.0
    c2w = syn.look_at((0.0, 0.0, -3.0), (0.0, 0.0, 5.0))
    ro, rd = syn.pinhole_rays(width, height, float(width), c2w)
    cand = np.concatenate([np.arange(k) for k in lengths]).astype(np.int32)
    off = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    base = [to_dev(a, device) for a in (ro, syn.normalize_rays(rd), sc.positions, sc.log_scales, sc.quats, cand, off, sc.freq,
                                        sc.att, *sc.mlp())]
    ext = TileExt()
    x = base + [torch.zeros_like(base[0]), torch.zeros(width * height, device=device)]
    records = ext.render_tiles_training_records(x, width, height, 8, 1e-3, 1.5, 2.0, render_order=True)
    rgb, alpha, frame = ext.train_forward(base, width, height, 1e-3)
    assert frame.status == 0 and torch.equal(rgb, records[0]) and torch.equal(alpha, records[1])
    # (the primitives of a tile that hit it, as the records have them: the lists but for a few at the image's border)
    pixel = torch.repeat_interleave(torch.arange(width * height, device=device), records[7].diff())
    tile = (pixel // width) // 8 * ((width + 7) // 8) + (pixel % width) // 8
    steps = torch.bincount((tile * n + records[2]).unique() // n, minlength=tiles).cpu().numpy()
    assert (steps <= lengths).all() and (steps == lengths).mean() > 0.9
    assert frame.steps == steps.sum()
    ends = np.array([0, 8, 16, *range(32, 129, 32)])
    assert frame.chunks * _lib.STEP_CHUNK == ends[np.searchsorted(ends, steps)].sum()
    torch.manual_seed(6)
    g_rgb, g_t = torch.randn(width * height, 3, device=device), torch.randn(width * height, device=device)
    want = ext.backward_from_records(records, base[2], base[3], base[4], base[7], base[8], *base[9:15], g_rgb, g_t)
    got = ext.backward_from_steps(frame, ops.train_group(frame, base[6], n), base, g_rgb, g_t)
    for i, (g, w) in enumerate(zip(got, want)):
        assert float((g - w).norm()) <= 1e-4 * float(w.norm()), i      # (up to 107,000 records of a primitive, f32 sums)
    # the same frame from a pool that is too small at first
    ext._steps_per_tile = 3.0
    again, _, frame = ext.train_forward(base, width, height, 1e-3)
    assert torch.equal(again, rgb) and frame.steps == steps.sum()
    for g, w in zip(ext.backward_from_steps(frame, ops.train_group(frame, base[6], n), base, g_rgb, g_t), got):
        assert torch.equal(g, w)


@pytest.mark.parametrize("lengths", [(1, 2, 3, 4, 5, 6, 7, 0, 8, 9), (511, 512, 513, 516), (1024, 1, 1025, 1029)])
def test_the_reverse_walk_of_tiles_of_every_length(device, lengths):
    """The reverse walk asks for four steps ahead and for the places of 512 at a time: lists that end around these, of
    primitives that all hit and hardly cover, against the record pipeline.  A step's adjoint behind up to 1,029 others is a
    chain of as many f32 roundings on either side, 1,029 x 2^-24 = 6e-5 of it at the worst."""
    import numpy as np
    from mlp_splatting_amd import ops, synthetic as syn
    from mlp_splatting_amd.tile_ext import TileExt
    n, width, height = max(lengths), 8 * len(lengths), 8
    sc = syn.make_scene(n, 32, seed=4, log_scale_mean=2.5)
    sc.positions[:] = np.array([0.0, 0.0, 9.0]) + 0.1 * sc.positions
    sc.b3[:, 3] = -8.0
    c2w = syn.look_at((0.0, 0.0, -3.0), (0.0, 0.0, 5.0))
    ro, rd = syn.pinhole_rays(width, height, 2.0 * width, c2w)
    cand = np.concatenate([np.arange(k) for k in lengths]).astype(np.int32)
    off = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    base = [to_dev(a, device) for a in (ro, syn.normalize_rays(rd), sc.positions, sc.log_scales, sc.quats, cand, off, sc.freq,
                                        sc.att, *sc.mlp())]
    ext = TileExt(max_hits=2048)
    x = base + [torch.zeros_like(base[0]), torch.zeros(width * height, device=device)]
    records = ext.render_tiles_training_records(x, width, height, 8, 1e-3, 1.5, 2.0, render_order=True)
    rgb, _, frame = ext.train_forward(base, width, height, 1e-3)
    assert frame.steps == sum(lengths) and torch.equal(rgb, records[0])
    torch.manual_seed(7)
    g_rgb, g_t = torch.randn(width * height, 3, device=device), torch.randn(width * height, device=device)
    want = ext.backward_from_records(records, base[2], base[3], base[4], base[7], base[8], *base[9:15], g_rgb, g_t)
    got = ext.backward_from_steps(frame, ops.train_group(frame, base[6], n), base, g_rgb, g_t)
    for i, (g, w) in enumerate(zip(got, want)):
        assert float((g - w).norm()) <= 6e-5 * float(w.norm()), i


@pytest.mark.parametrize("n,tiles,listed", [(2, 1, 1), (40, 700, 40), (70_000, 700, 40), (600_000, 1030, 80)])
def test_steps_are_sorted_by_primitive(device, n, tiles, listed):
    """The stable sort of a frame's steps, with fewer counts than the sums over blocks and digits take at a time (4,096), with
    several times and, at 600,000 primitives and 82,400 steps, with more than ten times as many (41 blocks x 1,024 digits),
    which are two turns of six."""
    import numpy as np
    from mlp_splatting_amd import ops, synthetic as syn
    from mlp_splatting_amd.tile_ext import TileExt
    width, height, rng = 8 * tiles, 8, np.random.default_rng(n)
    lists = np.stack([np.sort(rng.choice(n, listed, replace=False)) for _ in range(tiles)]).astype(np.int32)
    ro, rd = syn.pinhole_rays(width, height, 2.0 * width, syn.look_at((0.0, 0.0, -3.0), (0.0, 0.0, 5.0)))
    positions = np.array([0.0, 0.0, 9.0], np.float32) + 0.1 * rng.standard_normal((n, 3)).astype(np.float32)
    quats = np.tile(np.array([1.0, 0.0, 0.0, 0.0], np.float32), (n, 1))
    sc = syn.make_scene(1, 32, seed=0)
    base = [to_dev(a, device) for a in (ro, syn.normalize_rays(rd), positions, np.full((n, 3), 2.5, np.float32), quats,
                                        lists.reshape(-1), np.arange(tiles + 1, dtype=np.int32) * listed, sc.freq, sc.att)]
    base += [torch.zeros((n,) + w.shape[1:], device=device) for w in sc.mlp()]
    base[14][:, 3] = -8.0
    _, _, frame = TileExt().train_forward(base, width, height, 1e-3)
    steps = frame.steps
    assert steps == tiles * listed
    words = ops.train_group(frame, base[6], n).view(torch.int32).cpu().numpy()
    ends = np.cumsum([(k + 63) // 64 * 64 for k in (n + 1, steps, 4 * steps)])      # parts in units of 256 bytes
    first, prim, step = words[:n + 1], words[ends[0]:ends[0] + steps], words[ends[1]:ends[1] + 4 * steps].reshape(-1, 4)
    order = np.argsort(lists.reshape(-1), kind="stable")
    tile = order // listed                             # (a tile's steps come in the order of their depths: listed to a tile)
    assert (prim == lists.reshape(-1)[order]).all() and (step[:, 1] // listed == tile).all()
    assert (step[:, 2] == tile).all() and (step[:, 3] == 8 * tile).all() and (np.sort(step[:, 1]) == np.arange(steps)).all()
    assert (first == np.searchsorted(prim, np.arange(n + 1))).all()


@pytest.mark.parametrize("columns,rows", [(3, 1), (2100, 1), (50, 42)])
def test_the_forward_looks_for_what_is_not_finite(device, columns, rows):
    """By its wavefronts behind their tiles (2,100 tiles in a row, of which 244 go to teams, which do not look, and 50x42, of which
    all but 248 do) or, of 3 tiles, in a launch of its own: every element of arrays that begin at any float and of every length
    around a wavefront's and a workgroup's reach, the first and the last ones among them; a flag that is set stays set."""
    from mlp_splatting_amd import ops, synthetic as syn
    from mlp_splatting_amd.tile_ext import TileExt
    n, tiles, width, height = 40, columns * rows, 8 * columns, 8 * rows
    sc = syn.make_scene(n, 32, seed=4, log_scale_mean=-1.0)
    ro, rd = syn.pinhole_rays(width, height, 60.0, syn.look_at((0.0, 0.0, -3.0), (0.0, 0.0, 5.0)))
    base = [to_dev(a, device) for a in (ro, syn.normalize_rays(rd), sc.positions, sc.log_scales, sc.quats)]
    order = torch.arange(n, dtype=torch.int32, device=device).repeat(tiles)
    offsets = torch.arange(tiles + 1, dtype=torch.int32, device=device) * n
    freq, att, ws = to_dev(sc.freq, device), to_dev(sc.att, device), [to_dev(w, device) for w in sc.mlp()]
    records, packed = ops.prepare_primitives(*base[2:5]), ops.pack_mfma_weights(*ws, bf16=False)
    pool = tiles * n + 32 * tiles
    arrays = [torch.ones(length + 3, device=device)[shift:shift + length]
              for length, shift in ((1, 0), (3, 1), (63, 2), (257, 3), (4 * 64 + 1, 0), (70_001, 1), (3_000_000, 2), (0, 0))]

    def run(flag):
        seen = []
        buffer = ops.TrainBuffer(order.numel(), width, height, pool, device)
        buffer.bytes[:256].zero_()
        buffer.flag.fill_(flag)
        out = ops.train_forward(base[0], base[1], records, order, offsets, freq, att, ws, width, height, 1e-3, 128, pool,
                                packed=packed, buffer=buffer, settle=lambda counts, word: seen.append(word) or True, look=arrays)
        return out, seen[0]
    want, flag = run(0)
    assert flag == 0 and run(1)[1] == 1
    plain = ops.train_forward(base[0], base[1], records, order, offsets, freq, att, ws, width, height, 1e-3, 128, pool,
                              packed=packed)
    assert torch.equal(want[0], plain[0]) and torch.equal(want[1], plain[1]) and want[2].steps == plain[2].steps > 0
    for array in arrays[:-1]:
        for at in {0, array.numel() // 2, array.numel() - 1}:
            for value in (float("nan"), float("-inf")):
                array[at] = value
                (rgb, _, _), flag = run(0)
                assert flag == 1 and torch.equal(rgb, want[0])
            array[at] = 1.0


@pytest.mark.parametrize("columns,rows", [(1, 1), (3, 1), (64, 64), (67, 61), (128, 128), (129, 129)])
def test_first_steps_of_many_tiles(device, columns, rows):
    """The sums over the tiles' steps take 4,096 tiles at a time and 16,384 behind a barrier, four to a thread."""
    from mlp_splatting_amd import ops, synthetic as syn
    from mlp_splatting_amd.tile_ext import TileExt
    tiles, width, height = columns * rows, 8 * columns, 8 * rows
    sc = syn.make_scene(40, 32, seed=4, log_scale_mean=-1.0)
    view, proj = syn.view_matrix(syn.look_at((0.0, 0.0, -3.0))), syn.projection_matrix(0.5 * width, width, height)
    ro, rd = syn.pinhole_rays(width, height, 0.5 * width, syn.look_at((0.0, 0.0, -3.0)))
    ro, rd, pos, logs, quats = [to_dev(a, device) for a in (ro, syn.normalize_rays(rd), sc.positions, sc.log_scales, sc.quats)]
    order, offsets = ops.bin_legacy(pos, logs, torch.from_numpy(view)[None], torch.from_numpy(proj), width, height, 8, 1e-3)
    base = [ro, rd, pos, logs, quats, order, offsets] + [to_dev(a, device) for a in (sc.freq, sc.att, *sc.mlp())]
    _, _, frame = TileExt().train_forward(base, width, height, 1e-3)
    words = frame.workspace[256:].view(torch.int32)
    steps, first = words[:tiles].long(), words[(tiles + 63) // 64 * 64:][:tiles + 1].long()
    assert frame.steps == int(steps.sum()) > 0 and int(first[0]) == 0 and torch.equal(first[1:], steps.cumsum(0))


def test_a_frame_of_small_primitives_keeps_little(device, oracle_mod):
    """Storage follows the steps, not the tiles: a tile with a hit takes a chunk, and the first frame reserves no more than
    its lists can need."""
    from mlp_splatting_amd import _lib
    from mlp_splatting_amd.tile_ext import TileExt
    fr, base = _scene(device, oracle_mod, 300, 160, 120, 0.2, False)
    _, _, frame = TileExt().train_forward(base, 160, 120, fr.thr)
    assert frame.steps > 50
    slots = frame.chunks * _lib.STEP_CHUNK
    assert slots <= 2 * frame.steps + _lib.STEP_CHUNK * min(frame.steps, 300)
    pairs = base[5].numel()
    assert frame.nbytes <= (2 * pairs + _lib.STEP_CHUNK * 300 + 32) * 3400 + 65536


def test_captured_launches_replay_like_eager_ones(device, oracle_mod):
    """The launches between two read-backs of a training step, and a matrix-core render, as a captured graph: every replay,
    with eager work in between, gives what the eager calls give, and flags that one replay raised are down in the next."""
    from mlp_splatting_amd import _lib, ops
    from mlp_splatting_amd.tile_ext import TileExt
    fr, base = _scene(device, oracle_mod, 300, 33, 17, 1.0, False)
    ext, mlp = TileExt(), base[9:15]
    _, alpha, frame = ext.train_forward(base, 33, 17, fr.thr)
    rec = ops.prepare_primitives(*base[2:5])
    order, _ = ops.sort_tiles(base[0], base[1], rec, base[5], base[6], 33, 17, 8, 8, _lib.KEY_TSTAR)
    packed = ops.pack_mfma_weights(*mlp)
    g_rgb, g_t = torch.zeros(33 * 17, 3, device=device), torch.zeros(33 * 17, device=device)

    def launches():
        groups = ops.train_group(frame, base[6], 300)
        d4, falloff = ops.train_reverse(frame, base[6], g_rgb, g_t)
        grads, flag = ops.train_gradients(frame, groups, d4, falloff, base[1], base[7], base[8], mlp, base[3], base[4], 0, 1.0)
        image = ops.render_tilecenter_mfma(base[0], base[1], rec, order, base[6], base[7], base[8], *mlp, 33, 17, fr.thr,
                                           packed=packed, check=False)
        return [*grads, flag, *image]
    launches()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = launches()
    hit = int((alpha.reshape(-1) > 0).nonzero()[0])
    gen = torch.Generator(device=device).manual_seed(8)
    for replay in range(5):
        g_rgb.copy_(torch.randn(33 * 17, 3, device=device, generator=gen))
        g_t.copy_(torch.randn(33 * 17, device=device, generator=gen))
        if replay % 2:
            g_rgb[hit] = float("inf")
        want = launches()
        graph.replay()
        torch.cuda.synchronize()
        assert int(captured[9]) == int(want[9]) == replay % 2 and not int(captured[12][0])
        for got, expected in zip(captured[:9] + captured[10:12], want[:9] + want[10:12]):
            assert torch.equal(torch.nan_to_num(got), torch.nan_to_num(expected))


def test_cameras_that_come_round_again_are_not_rendered_twice(device, oracle_mod, monkeypatch):
    """Room for the steps is kept for the largest of the frames, whatever lies between its turns."""
    from mlp_splatting_amd import ops
    from mlp_splatting_amd.tile_ext import TileExt
    lib, asked = ops._lib.load(), []

    class Counting:
        def __getattr__(self, name):
            if name == "mlpsp_train_workspace_bytes":
                asked.append(name)
            return getattr(lib, name)
    frames = [_scene(device, oracle_mod, n, 160, 120, scale, False) for n, scale in ((300, 0.3), (1500, 1.0), (300, 0.2))]
    ext = TileExt()
    monkeypatch.setattr(ops._lib, "load", lambda: Counting())
    for turn in range(4):
        for fr, base in (*frames, frames[0], frames[2]):
            ext.train_forward(base, 160, 120, fr.thr)
        if turn == 0:
            asked.clear()
    assert len(asked) == 3 * 5


# teams of eight, of four, and most tiles by one wavefront with 2,048, 1,536 and 2,560 teams behind them
@pytest.mark.parametrize("columns,rows", [(40, 16), (641, 1), (32, 64), (41, 50), (53, 54), (80, 81)])
@pytest.mark.parametrize("precision", [None, "float16", "bfloat16"])
def test_the_forward_of_every_team_size_is_that_of_the_records(device, oracle_mod, columns, rows, precision):
    """Image and alpha bit for bit, and the number of steps, of the same frame in per-pixel records, whose walk knows no teams."""
    import numpy as np
    from mlp_splatting_amd.tile_ext import TileExt
    width, height = 8 * columns - 3, 8 * rows - 5
    fr, base = _scene(device, oracle_mod, 400, width, height, 0.6, False)
    ext = TileExt()
    rgb, alpha, frame = ext.train_forward(base, width, height, fr.thr, precision=precision)
    x = base + [torch.zeros_like(base[0]), torch.zeros(width * height, device=device)]
    if precision is None:
        records = ext.render_tiles_training_records(x, width, height, 8, fr.thr, 1.5, 2.0, render_order=True)
    else:
        records = ext.render_tiles_training_records_wmma(x, width, height, 8, fr.thr, 1.5, 2.0, precision)
    assert torch.equal(rgb, records[0]) and torch.equal(alpha.reshape(-1), records[1].reshape(-1))
    offsets = records[7].cpu().numpy()
    pixel = np.repeat(np.arange(width * height), np.diff(offsets))
    tile = pixel // width // 8 * columns + pixel % width // 8
    assert frame.steps == len(np.unique(tile.astype(np.int64) * 400 + records[2].cpu().numpy()))
