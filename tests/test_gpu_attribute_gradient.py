"""The feature-attribute gradient of training steps where its kernels part, against the gradient from per-pixel records: a
chunk holds steps x (256s of channels, rounded up) / 16,384 of the sorted steps, between 4 and 64, and the matrix-core kernel
takes rows of more than 64 channels in sixteens where it holds seven and more (fourteen up to 128 channels), eight at a time."""
import pytest
import torch

from helpers import ragged_lists, tile_row

pytestmark = pytest.mark.gpu


#                        tiles, primitives, steps, channels          steps of a chunk
@pytest.mark.parametrize("tiles,n,steps,channels", [
    (300, 40, 7167, 4096),           # 6, FMA
    (300, 40, 7168, 4096),           # 7, matrix cores
    (300, 40, 7168, 4100),           # 7, no sixteens of channels
    (330, 40, 8192, 4096),           # 8: a product of every chunk is full
    (380, 40, 9216, 4096),           # 9: and one step more
    (700, 48, 16700, 2064),          # 9, a last workgroup with one lane of channels
    (420, 40, 11000, 4080),          # 10
    (1400, 48, 33792, 4096),         # 33
    (2100, 48, 65536, 4096),         # 64, the most
    (2100, 48, 70001, 4096),         # 64 and a remainder
    (2048, 56, 114688, 80), (2048, 56, 114688, 144)])       # 7: FMA up to 128 channels, matrix cores above
def test_attribute_gradients_at_the_edges_of_chunks_and_kernels(device, tiles, n, steps, channels):
    from mlp_splatting_amd import ops, primitive_csr, record_feature_loss
    from mlp_splatting_amd.tile_ext import TileExt
    base, width, height = tile_row(device, tiles, n, *ragged_lists(tiles, n, steps))
    ext = TileExt()
    x = base + [torch.zeros_like(base[0]), torch.zeros(width * height, device=device)]
    records = ext.render_tiles_training_records(x, width, height, 8, 1e-3, 1.5, 2.0)
    _, _, frame = ext.train_forward(base, width, height, 1e-3, render_order=False)
    assert frame.steps == steps
    gen = torch.Generator(device=device).manual_seed(7)
    attributes = torch.randn(n, 4, channels, device=device, generator=gen) * 0.05
    # (targets far outside what the attributes blend to: no residual is near zero, where two sums may differ in sign)
    target = 16.0 * torch.randint(0, 2, (2, int(1.7 * tiles), channels), device=device, generator=gen) - 8.0
    _, signs, _ = record_feature_loss.streaming_feature_l1(records, attributes, target, width, height)
    csr = primitive_csr.group_records(records[2], records[3], records[3].new_zeros(records[2].numel(), 4), n, records[5])
    want = record_feature_loss.feature_weight_gradients(records, csr, signs, attributes, width, height, mixed=False)
    _, feature, kept = ops.train_feature_l1(frame, base[6], attributes, target, 1.5, 2.0)
    got = ops.train_feature_gradients(frame, ops.train_group(frame, base[6], n), feature, kept, attributes,
                                      torch.tensor(0.75, device=device))
    # f32 sums of up to 4 x 2,100 terms of either sign in chunks, on both sides: a few units of 2^-24 of the largest sum
    torch.testing.assert_close(got, want * 0.75, rtol=1e-5, atol=2e-6 * float(want.abs().max()))
