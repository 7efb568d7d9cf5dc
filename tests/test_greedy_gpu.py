"""B2 exact greedy on the device (selection_init / selection_chunk) against the oracle's heap
restatement of odie/selection.py:129-207: chosen cells, closure nodes, iteration count and the
order of choices are bit-exact."""
import numpy as np
import pytest
import torch

import oracle
from odie_amd import synth
from odie_amd.selection import align8, select_device

pytestmark = pytest.mark.gpu


def _scores(seed, cells, ties):
    if ties:
        # few distinct values, signed zeros: exercises every tie rule
        values = synth.integers(seed, 'greedy', cells, 6).astype(np.float64) * 0.5
        values[synth.integers(seed, 'negzero', cells, 4) == 0] = -0.0
    else:
        values = synth.uniform(seed, 'greedy', cells).astype(np.float64) ** 3
    return values


def _check(values, resolution, cap, normalize=True, chunk=512):
    trace = []
    selected, nodes, iterations = oracle.select_benefit_cost(values, resolution, cap, normalize_by_cost=normalize,
                                                             trace=trace)
    got_selected, got_nodes, got_iterations, got_trace = select_device(
        torch.from_numpy(values).cuda(), resolution, cap, normalize_by_cost=normalize, trace=True, chunk=chunk)
    assert got_iterations == iterations
    assert np.array_equal(got_trace.cpu().numpy(), np.asarray(trace, dtype=np.int32))
    assert np.array_equal(got_selected.cpu().numpy(), selected)
    assert np.array_equal(got_nodes.cpu().numpy(), nodes)


@pytest.mark.parametrize('resolution', [2, 3, 5, 8])
@pytest.mark.parametrize('ties', [False, True])
def test_tiny_grids_every_cap(resolution, ties):
    values = _scores(resolution, resolution * resolution, ties)
    for cap in range(0, align8(resolution * resolution) + 1, 8):
        _check(values, resolution, cap)


@pytest.mark.parametrize('resolution,cap,ties,normalize', [
    (64, 1024, False, True),      # two tree levels, all in LDS
    (64, 4096, True, True),       # cap = every node: all cells end selected
    (100, 2000, True, True),      # three levels, ragged last node
    (100, 2000, False, False),    # unnormalized: raw score order under the node cap
    (181, 9000, True, True),
])
def test_medium_grids(resolution, cap, ties, normalize):
    _check(_scores(7, resolution * resolution, ties), resolution, cap, normalize)


def test_chunk_boundaries_do_not_change_the_result():
    values = _scores(11, 48 * 48, True)
    _check(values, 48, 512, chunk=1)
    _check(values, 48, 512, chunk=3)


def test_large_grid_with_device_resident_tree_levels():
    # 448^2 cells: the level-0 nodes exceed the LDS-resident part, so the lowest tree level
    # is repaired in device memory
    _check(_scores(5, 448 * 448, False), 448, 8192)


def test_zero_scores_still_fill_capacity():
    values = np.zeros(32 * 32)
    _check(values, 32, 256)


def _bulk_scores(kind, resolution):
    cells = resolution * resolution
    values = synth.uniform(13, 'bulk' + kind, cells).astype(np.float64)
    if kind == 'ties':
        return _scores(13, cells, True)
    if kind == 'thirds':      # score/3, score/2 and score/4 of different cells meet up to rounding
        return np.array([1.0, 2.0, 3.0, 4.0, 6.0, 1 / 3, 2 / 3])[(values * 7).astype(int)]
    if kind == 'patches':     # flat zero ground with a few bright blocks, as a mostly settled residual
        plane = values.reshape(resolution, resolution) * 1e-3
        plane[: resolution // 2] = 0.0
        plane[resolution // 4: resolution // 3, resolution // 4:] += 5.0
        return plane.reshape(-1)
    if kind == 'chain':       # one long row of cells each freed by the last: levels cross every tile
        plane = np.full((resolution, resolution), 1e-9)
        plane[resolution // 2] = 1.0 + 1e-6 * np.arange(resolution)
        plane[resolution // 2, 0] = 4.5
        return plane.reshape(-1)
    if kind == 'nan':
        values[cells // 3] = np.nan
    if kind == 'negative':
        values[::7] *= -1.0
    if kind == 'huge':
        values[::5] *= 1e304
    if kind == 'tiny':
        values *= 5e-324 * 64
    return values


@pytest.mark.parametrize('resolution', [8, 31, 32, 33, 64, 65, 129, 200])
@pytest.mark.parametrize('kind', ['uniform', 'ties', 'thirds', 'patches', 'chain', 'nan', 'negative', 'huge', 'tiny'])
def test_bulk_start_equals_one_choice_at_a_time(kind, resolution):
    """Without a trace most choices are found in parallel; with one each is made in its turn."""
    scores = torch.from_numpy(_bulk_scores(kind, resolution)).cuda()
    points = align8(resolution * resolution)
    for cap in sorted({64, points // 64 * 8, points // 16 * 8, points - 8, points}):
        for normalize in (True, False):
            selected, nodes, iterations, _ = select_device(scores, resolution, cap, normalize, trace=True)
            got = select_device(scores, resolution, cap, normalize)
            what = (kind, resolution, cap, normalize)
            assert got[2] == iterations, what
            assert torch.equal(got[0], selected) and torch.equal(got[1], nodes), what


def test_without_memory_for_the_bulk_start(monkeypatch):
    """No room for the head start's workspace: every choice is made in its turn."""
    scores = torch.from_numpy(_bulk_scores('uniform', 65)).cuda()
    want = select_device(scores, 65, 512)
    empty = torch.empty

    def refusing(*size, **options):
        if options.get('dtype') == torch.uint8 and size and isinstance(size[0], int) and size[0] > 8 * 4225:
            raise torch.cuda.OutOfMemoryError('no room')
        return empty(*size, **options)
    monkeypatch.setattr(torch, 'empty', refusing)
    got = select_device(scores, 65, 512)
    assert got[2] == want[2] and torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


def test_bulk_start_against_the_oracle():
    values = _scores(17, 150 * 150, False)
    selected, nodes, iterations = oracle.select_benefit_cost(values, 150, 4000)
    got = select_device(torch.from_numpy(values).cuda(), 150, 4000)
    assert got[2] == iterations
    assert np.array_equal(got[0].cpu().numpy(), selected) and np.array_equal(got[1].cpu().numpy(), nodes)
