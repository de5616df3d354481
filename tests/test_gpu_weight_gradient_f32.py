"""The parts of the f32 weight-gradient kernel of training steps, each against float64: the encoding that it forms anew."""
import pytest
import torch

from conftest import to_dev

pytestmark = pytest.mark.gpu


def _frame(device, tiles, lists, n, mlp=None, log_scale_mean=2.5):
    """(base, frame) of a row of ``tiles`` tiles; ``lists[t]``: the primitives of tile t, each of which hits all its pixels."""
    import numpy as np
    from mlp_splatting_amd import synthetic as syn
    from mlp_splatting_amd.tile_ext import TileExt
    width, height = 8 * tiles, 8
    sc = syn.make_scene(n, 32, seed=5, log_scale_mean=log_scale_mean)
    sc.positions[:] = np.array([0.0, 0.0, 9.0]) + 0.1 * sc.positions
    sc.b3[:, 3] = -6.0
    c2w = syn.look_at((0.0, 0.0, -3.0), (0.0, 0.0, 5.0))
    ro, rd = syn.pinhole_rays(width, height, 2.0 * width, c2w)
    cand = np.concatenate(lists).astype(np.int32)
    off = np.concatenate([[0], np.cumsum([len(v) for v in lists])]).astype(np.int32)
    base = [to_dev(a, device) for a in (ro, syn.normalize_rays(rd), sc.positions, sc.log_scales, sc.quats, cand, off, sc.freq,
                                        sc.att, *sc.mlp())]
    if mlp is not None:
        for t, v in zip(base[9:15], mlp):
            t.copy_(v.to(device).expand_as(t))
    _, _, frame = TileExt().train_forward(base, width, height, 1e-3)
    assert frame.steps == cand.size
    return base, frame


def _encoding(device, rays, freq, att, tiles):
    """(sines, cosines, flag) of the phases of ``rays`` [tiles, 3], read off the W1 gradient of one record a primitive whose
    hidden adjoints are all 1: [tiles, 3, 6] each, the value of every hidden unit compared."""
    import numpy as np
    from mlp_splatting_amd import ops
    eye = torch.eye(32)
    first = torch.zeros(4, 32)
    first[0] = 1.0
    mlp = (torch.zeros(32, 72), torch.ones(32), eye, torch.ones(32), first, torch.tensor([0.0, 0.0, 0.0, -6.0]))
    base, frame = _frame(device, tiles, [np.array([t]) for t in range(tiles)], tiles, mlp)
    tile = torch.arange(tiles, device=device)
    lane = 7 * tile % 64
    d4 = torch.zeros(tiles, 64, 4, device=device)
    d4[tile, lane, 0] = 1.0
    rays_d = torch.rand(8 * 8 * tiles, 3, device=device)
    rays_d[(lane // 8) * 8 * tiles + 8 * tile + lane % 8] = rays.to(device)
    grads, flag = ops.train_gradients(frame, ops.train_group(frame, base[6], tiles), d4, torch.zeros(tiles, 64, device=device),
                                      rays_d, freq.to(device), att.to(device), base[9:15], base[3], base[4], 0, 1.0)
    gW1 = grads[0].cpu()
    torch.testing.assert_close(gW1, gW1[:, :1].expand_as(gW1), rtol=0, atol=0, equal_nan=True)
    return gW1[:, 0, :18].reshape(tiles, 3, 6), gW1[:, 0, 36:54].reshape(tiles, 3, 6), int(flag)


# A pair is a table value and a rotation, each to 2^-31 and better, and one rounded sum of the two: half a unit of the last
# place, 2^-25 below 1, and four times 2^-31.  Over all phases that is 2^-25 / sqrt(3) rms for values from 0.5 on and less below.
PAIR_MAX, PAIR_RMS = 2.0 ** -25 + 4 * 2.0 ** -31, 2.0 ** -25 / 3 ** 0.5


@pytest.mark.parametrize("reach", [0.01, 0.9, 60.0, 3000.0])
def test_sines_and_cosines_are_rounded_once(device, reach):
    """Factors that are powers of two: the phases are exact."""
    gen = torch.Generator().manual_seed(1)
    rays = (torch.rand(1024, 3, generator=gen) * 2 - 1) * (reach / 32)
    freq = 2.0 ** torch.arange(6)
    sine, cosine, flag = _encoding(device, rays, freq, torch.ones(6), 1024)
    phase = (rays[:, :, None] * freq).double()
    assert flag == 0
    for got, want in ((sine, phase.sin()), (cosine, phase.cos())):
        error = got.double() - want
        assert float(error.abs().max()) <= PAIR_MAX and float(error.square().mean().sqrt()) <= PAIR_RMS


def _attenuated(device):
    """Frequencies and attenuations of an annealed encoding: neither product with an input is exact."""
    gen = torch.Generator().manual_seed(2)
    return 100.5 ** (torch.arange(6) / 5), 0.3 + 0.7 * torch.rand(6, generator=gen)


def test_phases_are_those_of_the_forward(device):
    """(x freq) att with both roundings, and nothing else: to the rounding of a pair, at phases of up to 60."""
    freq, att = _attenuated(device)
    rays = torch.rand(1024, 3, generator=torch.Generator().manual_seed(3)) * 2 - 1
    sine, cosine, flag = _encoding(device, rays, freq, att, 1024)
    phase = ((rays[:, :, None] * freq) * att).double()
    assert flag == 0
    for got, want in ((sine, phase.sin()), (cosine, phase.cos())):
        assert float((got.double() - want).abs().max()) <= PAIR_MAX


def test_a_phase_out_of_range_ends_its_own_pair(device):
    """65536 is the last phase that the forward takes; the float behind it gives NaN, and so do infinities and NaN."""
    freq = 2.0 ** torch.arange(6)
    edge = 65536.0 / 32
    beyond = float(torch.nextafter(torch.tensor(edge), torch.tensor(1e9)))
    taken = torch.tensor([[edge, -edge, 0.0], [1e-30, -0.0, 2.0]])
    refused = torch.tensor([[beyond, -beyond, 1.0], [4 * edge, 1e30, -1e38], [float("inf"), float("-inf"), float("nan")]])
    for rays in (taken, refused):
        sine, cosine, flag = _encoding(device, rays, freq, torch.ones(6), rays.shape[0])
        phase = (rays[:, :, None] * freq).double()
        phase = torch.where(phase.abs() <= 65536, phase, float("nan"))
        assert flag == int(bool(phase.isnan().any()))
        for got, want in ((sine, phase.sin()), (cosine, phase.cos())):
            assert torch.equal(got.isnan(), want.isnan())
            assert float((got.double() - want).nan_to_num().abs().max()) <= PAIR_MAX


@pytest.mark.parametrize("power", [-120, -112, -100, 40, 100, 110])
def test_gradients_scale_with_the_adjoints(device, power):
    """A loss scaled by a power of two has gradients scaled by it, bit for bit.  Where the sums of a chunk (16 of 16 steps for
    each primitive, of two rows at the ends) fall below the smallest normal number, each is rounded to 2^-149 by half of that,
    and those that stay above may be rounded the other way for it, 2^-24 of the largest each."""
    import numpy as np
    from mlp_splatting_amd import ops
    base, frame = _frame(device, 256, [np.arange(3)] * 256, 3)
    groups = ops.train_group(frame, base[6], 3)
    gen = torch.Generator(device=device).manual_seed(4)
    d4 = torch.randn(frame.steps, 64, 4, device=device, generator=gen)
    scaled = (d4.double() * 2.0 ** power).float()
    d4 = (scaled.double() * 2.0 ** -power).float()
    falloff = torch.zeros(frame.steps, 64, device=device)
    grads = [ops.train_gradients(frame, groups, d, falloff, base[1], base[7], base[8], base[9:15], base[3], base[4], 0, 1.0)
             for d in (d4, scaled)]
    assert int(grads[0][1]) == int(grads[1][1]) == 0
    for want, got in zip(grads[0][0][:6], grads[1][0]):
        want, got = want.double() * 2.0 ** power, got.double()
        bound = 18 * (2.0 ** -150 + 2.0 ** -24 * float(want.abs().max())) if power < -80 else 0.0
        assert float(want.abs().max()) > 0 and float((got - want).abs().max()) <= bound


@pytest.mark.parametrize("value", [float("nan"), float("inf"), 3e38])
def test_sums_out_of_range_are_refused(device, value):
    """... and of the numbers that f32 holds none is refused: a finite adjoint of 3e38 by itself is taken."""
    import numpy as np
    from mlp_splatting_amd import ops
    base, frame = _frame(device, 40, [np.arange(3)] * 40, 3)
    groups = ops.train_group(frame, base[6], 3)
    for copies in (1, 2):
        d4 = torch.zeros(frame.steps, 64, 4, device=device)
        d4[60:60 + 3 * copies:3, 5, 1] = value              # one primitive, one or two of its tiles
        got, flag = ops.train_gradients(frame, groups, d4, torch.zeros(frame.steps, 64, device=device), base[1], base[7],
                                        base[8], base[9:15], base[3], base[4], 0, 1.0)
        taken = value == 3e38 and copies == 1
        assert int(flag) == int(not taken)
        if taken:
            assert sorted(got[5].flatten().tolist())[-1] == torch.tensor(value).item()
