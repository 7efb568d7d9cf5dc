"""Fused reconstruction (odie_reconstruct) against the composition of the tested entry points:
route the raster ids, encode the compacted coordinates (odie_grid_forward), run the decoder
(odie_mlp_forward) and put the rows back in raster order -- features, decoder outputs and
predictions bit for bit, over ragged ranges and with tiles that have no expert.  Then the
scoring pipeline (score_image): per-cell totals bit-exact against the oracle's residual of the
fused predictions, the top tiles against the oracle's ranking, the mse against torch's expression;
both the streamed form (odie_reconstruct + score_chunk) and the fused one (odie_reconstruct_scores,
one or several waves per cell)."""
import numpy as np
import pytest
import torch

import oracle
from odie_amd import _lib, synth
from odie_amd.decoder import Decoder
from odie_amd.experts import ExpertGrid, route
from odie_amd.gpu_residual import DeviceScores
from odie_amd.reconstruction import reconstruct, score_image
from odie_amd.selection import topk_tiles

pytestmark = pytest.mark.gpu

ENCODING = dict(n_levels=16, n_features_per_level=2, log2_hashmap_size=10, base_resolution=4, per_level_scale=1.3)


def _model(seed, experts):
    grid = ExpertGrid(ENCODING, experts)
    values = synth.normal(seed, 'recon_table', grid.table.numel()) * 0.5
    grid.table.copy_(torch.from_numpy(values.astype(np.float16)))
    return grid, Decoder(seed=seed)


def _composed(grid, decoder, shape, regions, begin, n, slots=None):
    height, width = shape
    ids = torch.arange(begin, begin + n, dtype=torch.int64, device='cuda')
    routing = route(ids, width, height, *regions)
    features_c = grid.forward(routing.coords, routing.offsets) if slots is None else None
    if slots is not None:
        # tiles without an expert read zero features; others read their slot's table
        table = grid.table.view(grid.experts, -1)
        regrouped = ExpertGrid(ENCODING, regions[0] * regions[1])
        for tile, slot in enumerate(slots.tolist()):
            if 0 <= slot < grid.experts:
                regrouped.table.view(regrouped.experts, -1)[tile].copy_(table[slot])
        features_c = regrouped.forward(routing.coords, routing.offsets)
    output_c = decoder.forward(features_c)
    perm = routing.perm.long()
    features = torch.empty_like(features_c)
    features[perm] = features_c
    output = torch.empty_like(output_c)
    output[perm] = output_c
    return features, output


def _bits(t):
    return t.cpu().numpy().view(np.uint16 if t.dtype == torch.float16 else np.uint32)


@pytest.mark.parametrize('shape,regions,begin,n', [((96, 130), (3, 2), 0, 96 * 130),
                                                   ((96, 130), (3, 2), 1001, 5000 - 7),
                                                   ((200, 64), (2, 5), 12345, 1)])
def test_reconstruction_equals_route_encode_decoder(shape, regions, begin, n):
    grid, decoder = _model(2, regions[0] * regions[1])
    features = torch.empty((n, 32), dtype=torch.float16, device='cuda')
    output = torch.empty((n, 16), dtype=torch.float16, device='cuda')
    prediction = reconstruct(grid, decoder.half, shape, regions, begin, n, prediction=torch.empty(
        (n, 3), dtype=torch.float32, device='cuda'), features=features, output=output)
    want_features, want_output = _composed(grid, decoder, shape, regions, begin, n)
    assert np.array_equal(_bits(features), _bits(want_features))
    assert np.array_equal(_bits(output), _bits(want_output))
    assert np.array_equal(_bits(prediction), _bits(want_output[:, :3].float()))


def test_tiles_without_an_expert_predict_zero():
    shape, regions = (120, 90), (3, 3)
    grid, decoder = _model(3, 5)
    slots = torch.tensor([4, -1, 0, 2, 9, 1, -1, 3, 0], dtype=torch.int32, device='cuda')   # 9 >= experts: none
    n = shape[0] * shape[1]
    features = torch.empty((n, 32), dtype=torch.float16, device='cuda')
    output = torch.empty((n, 16), dtype=torch.float16, device='cuda')
    reconstruct(grid, decoder.half, shape, regions, 0, n, slots=slots, features=features, output=output)
    want_features, want_output = _composed(grid, decoder, shape, regions, 0, n, slots=slots.cpu())
    assert np.array_equal(_bits(features), _bits(want_features))
    assert np.array_equal(_bits(output), _bits(want_output))
    empty = (want_features == 0).all(dim=1)
    assert bool(empty.any()) and bool((output[empty] == 0).all())


@pytest.mark.parametrize('fused', [True, False])
@pytest.mark.parametrize('shape,resolution,tile,batch', [((128, 160), 8, None, 4096), ((128, 128), None, 32, 10000),
                                                         ((90, 77), 5, None, 1000)])
def test_scoring_pipeline_matches_the_oracle(shape, resolution, tile, batch, fused):
    regions = (4, 4) if shape[0] >= 128 else (3, 2)
    grid, decoder = _model(4, regions[0] * regions[1])
    image = synth.image(5, shape[1], shape[0]).reshape(-1, 3)
    target = torch.from_numpy(image).cuda()
    n = shape[0] * shape[1]
    image_out = torch.full((n, 3), float('nan'), dtype=torch.float32, device='cuda') if fused else None
    metrics, scores = score_image(grid, decoder.half, target, shape, regions, resolution=resolution, tile=tile,
                                  batch=batch, fused=fused, prediction=image_out)
    prediction = reconstruct(grid, decoder.half, shape, regions, 0, n).cpu().numpy()
    if fused:
        assert np.array_equal(image_out.cpu().numpy().view(np.uint32), prediction.view(np.uint32))
    expected = oracle.residual(prediction, image, shape[1], scores.resolution, scores.xb.cpu().numpy(),
                               scores.yb.cpu().numpy())
    assert np.array_equal(scores.totals.cpu().numpy().view(np.uint64), expected.view(np.uint64))
    truth = torch.from_numpy(image).cuda().float() / 255.
    reference = ((torch.from_numpy(prediction).cuda() - truth).square().double().sum() / image.size).item()
    assert metrics['mse'] == pytest.approx(reference, rel=1e-12)   # summation order only
    k = scores.resolution ** 2 // 4
    ids = topk_tiles(scores.totals / torch.from_numpy(scores.counts).cuda(), k).cpu().numpy()
    means = expected / scores.counts
    assert np.array_equal(ids, oracle.topk_ids(means, k))


def test_device_image_on_the_gpu_equals_numpy():
    expected = synth.image(7, 300, 170)
    got = synth.image_device(7, 300, 170, device='cuda', rows=64).cpu().numpy()
    assert np.array_equal(got, expected)


@pytest.mark.parametrize('shape,resolution,tile', [
    ((330, 330), None, 33),      # 1089 pixels: several waves per cell, ragged rounds; 100 cells
    ((640, 640), None, 32),      # 1024 pixels exactly; more cells than CUs
    ((96, 1100), 3, None),       # tall and narrow native cells across tile bounds
    ((40, 40), None, 7),         # small cells, one wave each, chunks across row ends
])
def test_scores_of_cells_of_every_size(shape, resolution, tile):
    """Cells on both sides of the large-cell rule against the oracle's sequential totals, bit for bit."""
    regions = (5, 3)
    grid, decoder = _model(6, regions[0] * regions[1])
    image = synth.image(8, shape[1], shape[0]).reshape(-1, 3)
    target = torch.from_numpy(image).cuda()
    n = shape[0] * shape[1]
    _, scores = score_image(grid, decoder.half, target, shape, regions, resolution=resolution, tile=tile)
    prediction = reconstruct(grid, decoder.half, shape, regions, 0, n).cpu().numpy()
    expected = oracle.residual(prediction, image, shape[1], scores.resolution, scores.xb.cpu().numpy(),
                               scores.yb.cpu().numpy())
    assert np.array_equal(scores.totals.cpu().numpy().view(np.uint64), expected.view(np.uint64))


@pytest.mark.parametrize('encoding', [
    dict(n_levels=16, base_resolution=3, log2_hashmap_size=15, per_level_scale=1.9, n_features_per_level=2),
    dict(n_levels=16, base_resolution=16, log2_hashmap_size=9, per_level_scale=1.38, n_features_per_level=2),
    dict(n_levels=16, base_resolution=8, log2_hashmap_size=20, per_level_scale=1.2, n_features_per_level=2),   # all dense
    dict(n_levels=16, base_resolution=40, log2_hashmap_size=6, per_level_scale=2.0, n_features_per_level=2),   # all hashed, past 2^12 cells
])
def test_reconstruction_encode_over_level_kinds(encoding):
    """The reconstruction's own encode against odie_grid_forward on the routed coordinates: dense,
    hashed and mixed lane steps, power-of-two and other level sizes, coordinates of exactly 0 and 1."""
    shape, regions = (77, 201), (4, 3)
    grid = ExpertGrid(encoding, regions[0] * regions[1])
    grid.table.copy_(torch.from_numpy(synth.table(9, grid.table.numel(), -1.0, 1.0, name='kinds')).half())
    decoder = Decoder(seed=9)
    n = shape[0] * shape[1]
    features = torch.empty((n, 32), dtype=torch.float16, device='cuda')
    output = torch.empty((n, 16), dtype=torch.float16, device='cuda')
    reconstruct(grid, decoder.half, shape, regions, 0, n, features=features, output=output)
    want_features, want_output = _composed(grid, decoder, shape, regions, 0, n)
    assert np.array_equal(_bits(features), _bits(want_features))
    assert np.array_equal(_bits(output), _bits(want_output))


def test_infinite_predictions_keep_their_scores():
    """A decoder that overflows fp16 scores infinite and NaN totals exactly as score_chunk does."""
    shape, regions = (64, 96), (2, 2)
    grid, decoder = _model(10, 4)
    decoder.params.mul_(3000.0)
    decoder.sync_weights()
    image = torch.from_numpy(synth.image(3, shape[1], shape[0]).reshape(-1, 3)).cuda()
    n = shape[0] * shape[1]
    prediction = reconstruct(grid, decoder.half, shape, regions, 0, n)
    assert not bool(torch.isfinite(prediction).all())
    streamed = DeviceScores(shape, resolution=4)
    streamed.add(prediction, image, 0)
    expected = oracle.residual(prediction.cpu().numpy(), image.cpu().numpy(), shape[1], 4, streamed.xb.cpu().numpy(),
                               streamed.yb.cpu().numpy())
    got = streamed.totals.cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(expected)) and np.array_equal(np.isinf(got), np.isinf(expected))
    finite = np.isfinite(expected)
    assert np.array_equal(got[finite], expected[finite])


# Past 2^22 cells the reconstruction takes the general geometry in place of its fast encode.
GENERAL = dict(n_levels=16, base_resolution=40, log2_hashmap_size=6, per_level_scale=2.3, n_features_per_level=2)
# A wave a cell, for few pixels and for many cells; several waves a cell, at most and more cells than CUs.
CELL_CLASSES = [((101, 77), 9, None), ((2912, 2912), None, 32), ((330, 330), None, 33), ((640, 640), None, 32)]


def _encoded(encoding, seed, experts):
    grid = ExpertGrid(encoding, experts)
    grid.table.copy_(torch.from_numpy(synth.table(seed, grid.table.numel(), -1.0, 1.0, name='general')).half())
    return grid, Decoder(seed=seed)


def _fused_scores(grid, decoder, target, shape, regions, scores):
    """odie_reconstruct_scores into scores.totals as they stand; the squares per cell."""
    squares = torch.zeros_like(scores.totals)
    xb, yb = scores.xb.to(torch.int32).contiguous(), scores.yb.to(torch.int32).contiguous()
    _lib.check(_lib.library().odie_reconstruct_scores(
        shape[1], shape[0], regions[0], regions[1], None, grid.experts, grid.table.data_ptr(), grid.expert_params,
        grid.levels, len(grid.levels), decoder.half.data_ptr(), target.data_ptr(), scores.resolution, xb.data_ptr(),
        yb.data_ptr(), scores.totals.data_ptr(), squares.data_ptr(), None, _lib.stream_of(target)))
    return squares


def test_general_geometry_reconstruction():
    shape, regions = (77, 201), (4, 3)
    grid, decoder = _encoded(GENERAL, 11, 12)
    assert max(level.resolution for level in grid.levels) >= 1 << 22
    n = shape[0] * shape[1]
    features = torch.empty((n, 32), dtype=torch.float16, device='cuda')
    output = torch.empty((n, 16), dtype=torch.float16, device='cuda')
    reconstruct(grid, decoder.half, shape, regions, 0, n, features=features, output=output)
    want_features, want_output = _composed(grid, decoder, shape, regions, 0, n)
    assert np.array_equal(_bits(features), _bits(want_features))
    assert np.array_equal(_bits(output), _bits(want_output))


@pytest.mark.parametrize('encoding', [ENCODING, GENERAL], ids=['fast', 'general'])
@pytest.mark.parametrize('shape,resolution,tile', CELL_CLASSES)
def test_scores_continue_totals_in_every_cell_class(shape, resolution, tile, encoding):
    """Totals that are not zero are carried on in raster order, bit for bit, whichever kernel scores the
    cells and whichever geometry encodes."""
    regions = (5, 3)
    grid, decoder = _encoded(encoding, 12, 15)
    image = synth.image(13, shape[1], shape[0]).reshape(-1, 3)
    target = torch.from_numpy(image).cuda()
    scores = DeviceScores(shape, resolution=resolution, tile=tile)
    start = synth.uniform(14, 'totals', scores.resolution ** 2).astype(np.float64) * 1e-3 + 0.1
    scores.totals.copy_(torch.from_numpy(start))
    squares = _fused_scores(grid, decoder, target, shape, regions, scores)
    prediction = reconstruct(grid, decoder.half, shape, regions, 0, len(image)).cpu().numpy()
    expected = oracle.residual(prediction, image, shape[1], scores.resolution, scores.xb.cpu().numpy(),
                               scores.yb.cpu().numpy(), totals=start.copy())
    assert np.array_equal(scores.totals.cpu().numpy().view(np.uint64), expected.view(np.uint64))
    error = np.square(prediction - image.astype(np.float32) * np.float32(1 / 255)).astype(np.float64).sum()
    assert float(squares.sum()) == pytest.approx(error, rel=1e-10)   # fp64 sums in another order


@pytest.mark.parametrize('encoding', [ENCODING, GENERAL], ids=['fast', 'general'])
@pytest.mark.parametrize('shape,resolution,tile', CELL_CLASSES)
def test_fused_scores_of_infinite_predictions(shape, resolution, tile, encoding):
    """An expert whose decoder overflows fp16: its cells' infinite and NaN totals, and the others' finite
    ones, as the streamed pass forms them."""
    regions = (5, 3)
    grid, decoder = _encoded(encoding, 15, 15)
    grid.table.view(15, -1)[4] = 6e4
    target = torch.from_numpy(synth.image(16, shape[1], shape[0]).reshape(-1, 3)).cuda()
    fused, streamed = (DeviceScores(shape, resolution=resolution, tile=tile) for _ in range(2))
    _fused_scores(grid, decoder, target, shape, regions, fused)
    prediction = reconstruct(grid, decoder.half, shape, regions, 0, shape[0] * shape[1])
    streamed.add(prediction, target, 0)
    got, want = fused.totals.cpu().numpy(), streamed.totals.cpu().numpy()
    finite = np.isfinite(want)
    assert finite.any() and not finite.all()
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    assert np.array_equal(got[finite].view(np.uint64), want[finite].view(np.uint64))
