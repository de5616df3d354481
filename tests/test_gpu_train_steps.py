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
