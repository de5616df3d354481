"""The weight-gradient kernels of training steps against float64: the encoding that the f32 kernel forms anew, its range, and
sums over chunks of every length."""
import numpy as np
import pytest
import torch

from helpers import ragged_lists, tile_row

pytestmark = pytest.mark.gpu


def _frame(device, tiles, n, tile, prim, mlp=None):
    from mlp_splatting_amd.tile_ext import TileExt
    base, width, height = tile_row(device, tiles, n, tile, prim, mlp)
    _, _, frame = TileExt().train_forward(base, width, height, 1e-3)
    assert frame.steps == len(tile)
    return base, frame


def _every_tile(tiles, n):
    return np.repeat(np.arange(tiles), n), np.tile(np.arange(n), tiles)


def _encoding(device, rays, freq, att, tiles):
    """(sines, cosines, flag) of the phases of ``rays`` [tiles, 3], read off the W1 gradient of one record a primitive whose
    hidden adjoints are all 1: [tiles, 3, 6] each, the value of every hidden unit compared."""
    from mlp_splatting_amd import ops
    eye = torch.eye(32)
    first = torch.zeros(4, 32)
    first[0] = 1.0
    mlp = (torch.zeros(32, 72), torch.ones(32), eye, torch.ones(32), first, torch.tensor([0.0, 0.0, 0.0, -6.0]))
    base, frame = _frame(device, tiles, tiles, np.arange(tiles), np.arange(tiles), mlp)
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
    from mlp_splatting_amd import ops
    base, frame = _frame(device, 256, 3, *_every_tile(256, 3))
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
    from mlp_splatting_amd import ops
    base, frame = _frame(device, 40, 3, *_every_tile(40, 3))
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


def _two_parts(v):
    """``v`` as the sum of two bf16 numbers: an f32 operand without its third part."""
    v = v.float()
    high = v.bfloat16().float()
    return (high + (v - high).bfloat16().float()).double()


# Steps of a chunk: steps / 2048 in eights, between 16 and 128.
@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("tiles,n,steps", [(2500, 40, 49151), (2500, 40, 49152), (3300, 40, 65536 + 17), (6700, 40, 131072 + 50),
                                           (13200, 40, 262144 - 1), (13200, 40, 262144), (15100, 40, 300001)])
def test_weight_gradients_of_chunks_of_every_length(device, tiles, n, steps, precision):
    """A pixel in 25 has an adjoint, so that blocks without one lie among the others.  An f32 gradient is the sum of up to
    25,000 products, in chains of up to 64 blocks x 12 roundings whose sums, 100 at the most, are added up in turn.  k roundings
    of a sum that grows to s, as a random walk does, add up to sqrt(k / 2) s 2^-24 / sqrt(12): 5.7 units of 2^-24 for a chain,
    2 for its sums, 2 for the factors' own; twelve, which is less than what is lost with the third part of any one operand.  In
    16 bits every factor and what it was computed from, eight tensors at the most, is rounded once, and a phase by a few units
    of 2^-24."""
    from mlp_splatting_amd import ops
    from mlp_splatting_amd.tile_ext import TileExt
    base, width, height = tile_row(device, tiles, n, *ragged_lists(tiles, n, steps))
    ext = TileExt()
    x = base + [torch.zeros_like(base[0]), torch.zeros(width * height, device=device)]
    records = ext.render_tiles_training_records(x, width, height, 8, 1e-3, 1.5, 2.0, render_order=True)
    _, _, frame = ext.train_forward(base, width, height, 1e-3)
    assert frame.steps == steps and records[2].numel() == 64 * steps
    gen = torch.Generator(device=device).manual_seed(9)
    d4 = torch.randn(steps, 64, 4, device=device, generator=gen)
    d4 *= torch.rand(steps, 64, 1, device=device, generator=gen) < 0.04
    got, flag = ops.train_gradients(frame, ops.train_group(frame, base[6], n), d4, torch.zeros(steps, 64, device=device), base[1],
                                    base[7], base[8], base[9:15], base[3], base[4], precision, 256.0 if precision else 1.0)
    assert int(flag) == 0
    # d4 is [step of a tile, lane], the records are [pixel, hit] in the tile's order
    pixel = torch.repeat_interleave(torch.arange(width * height, device=device), records[7].diff())
    hit = torch.arange(64 * steps, device=device) - records[7][:-1][pixel]
    at = (base[6].long()[pixel % width // 8] + hit) * 64 + pixel // width * 8 + pixel % 8
    live = (d4.view(-1, 4)[at] != 0).any(1).nonzero()[:, 0]
    ids, x6, d4 = records[2][live], records[3][live], d4.view(-1, 4)[at[live]]
    active = (records[5][live][:, :, None] >> torch.arange(32, dtype=torch.int32, device=device)) & 1
    W1, b1, W2, b2, W3, _ = (w.double() for w in base[9:15])
    for p in range(n):
        mine = ids == p
        phase = ((x6[mine][:, :, None] * base[7]) * base[8]).reshape(-1, 36).double()
        enc, d, on = torch.cat([phase.sin(), phase.cos()], 1), d4[mine].double(), active[mine].double()
        bound = (12 * 2.0 ** -24, 8 * 2.0 ** -11, 8 * 2.0 ** -8)[precision]
        bound += 2.0 ** -23 * float(phase.abs().max()) if precision else 0.0
        h1 = (enc @ W1[p].T + b1[p]).clamp(min=0.0)
        h2 = (h1 @ W2[p].T + b2[p]).clamp(min=0.0)
        d2 = (d @ W3[p]) * on[:, 1]
        d1 = (d2 @ W2[p]) * on[:, 0]
        want = [d1.T @ enc, d1.sum(0), d2.T @ h1, d2.sum(0), d.T @ h2, d.sum(0)]
        for i, (a, b) in enumerate(zip(got, want)):
            assert float((a[p].double() - b).norm()) <= bound * float(b.norm()), (p, i)
        if precision == 0:
            for i, less in ((0, d1.T @ _two_parts(enc)), (0, _two_parts(d1).T @ enc), (2, d2.T @ _two_parts(h1)),
                            (2, _two_parts(d2).T @ h1)):
                assert float((less - want[i]).norm()) > bound * float(want[i].norm()), (p, i)


@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("tiles,n", [(1, 1), (1, 7), (1, 8), (1, 33), (17, 4099), (40, 999)])
def test_primitives_without_a_step_get_zeros(device, monkeypatch, tiles, n, precision):
    """The wavefronts of the chunks share out the rows of all primitives, eight at a time: fewer groups than wavefronts and
    more, a last group that is not full; every third primitive has steps."""
    from mlp_splatting_amd import ops
    listed = np.arange(0, min(n, 96), 3)
    tile, prim = np.repeat(np.arange(tiles), len(listed)), np.tile(listed, tiles)
    base, frame = _frame(device, tiles, n, tile, prim)
    groups = ops.train_group(frame, base[6], n)
    d4, falloff = torch.ones(frame.steps, 64, 4, device=device), torch.ones(frame.steps, 64, device=device)
    monkeypatch.setattr(torch, "empty_like", lambda t: torch.full_like(t, float("nan")))
    grads, flag = ops.train_gradients(frame, groups, d4, falloff, base[1], base[7], base[8], base[9:15], base[3], base[4],
                                      precision, 1.0)
    monkeypatch.undo()
    without = torch.ones(n, dtype=torch.bool, device=device)
    without[torch.from_numpy(listed).to(device)] = False
    assert int(flag) == 0
    for i, g in enumerate(grads):
        assert bool(torch.isfinite(g).all()) and not bool(g[without].any()), i
    assert bool((grads[5][~without] != 0).all())


@pytest.mark.parametrize("precision,share", [(0, 1 << 20), (1, 448 << 10), (2, 448 << 10)])
@pytest.mark.parametrize("beside", [False, True])
def test_zeros_on_both_sides_of_a_wavefronts_share(device, precision, share, beside):
    """One chunk of 16 steps, four wavefronts: as many primitives as they store the rows of, and one more, whose rows a launch of
    its own writes."""
    from mlp_splatting_amd import ops
    channels = 24 if beside else 0
    most = 4 * share // (4 * (3524 + 10 + channels))
    for n in (most, most + 1):
        base, frame = _frame(device, 1, n, np.zeros(16, int), np.arange(5, 21))
        groups, d4 = ops.train_group(frame, base[6], n), torch.ones(16, 64, 4, device=device)
        rows = torch.full((n, max(channels, 1)), float("nan"), device=device)
        grads, flag = ops.train_gradients(frame, groups, d4, d4[..., 0].contiguous(), base[1], base[7], base[8], base[9:15], base[3],
                                          base[4], precision, 1.0, *((rows,) if beside else ()))
        without = torch.ones(n, dtype=torch.bool, device=device)
        without[5:21] = False
        assert int(flag) == 0 and bool((grads[5][~without] != 0).all())
        for g in grads + ([rows] if beside else []):
            assert not bool(g[without].ne(0).any())
        assert not beside or bool(rows[~without].isnan().all())


@pytest.mark.parametrize("precision", [0, 1])
def test_few_steps_of_many_primitives_do_not_wait_for_their_zeros(device, precision):
    """16 steps, a chunk, of 20,000 primitives: 283 MB of zeros, which one workgroup takes 50 times as long for as the whole
    call of 2,400 steps takes.  With a launch for them it is twice as long; ten times leaves room for a busy host."""
    from mlp_splatting_amd import ops

    def call(tiles):
        listed = np.arange(16) * 700
        base, frame = _frame(device, tiles, 20_000, np.repeat(np.arange(tiles), 16), np.tile(listed, tiles))
        groups, d4 = ops.train_group(frame, base[6], 20_000), torch.ones(frame.steps, 64, 4, device=device)
        args = (frame, groups, d4, d4[..., 0].contiguous(), base[1], base[7], base[8], base[9:15], base[3], base[4], precision, 1.0)
        times = []
        for _ in range(7):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            ops.train_gradients(*args)
            end.record()
            torch.cuda.synchronize()
            times.append(begin.elapsed_time(end))
        return sorted(times)[3]
    assert call(1) <= 10.0 * call(150)
