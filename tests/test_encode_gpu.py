"""GPU parity of the grid encode (HIP via the C-ABI) against the CPU oracle.

Forward: bit-exact (fp16 chain and fp32 chain).  Backward: each gradient entry within
1e-4 of the sum of the absolute values of its contributions (summation order is free), plus
half the fixed-point quantum of its own (level, feature) column per contribution (the owner
backward rounds each contribution once; oracle.bounds states the bar and the quantum).
"""
import numpy as np
import pytest
import torch

import oracle
from oracle.bounds import check_gradient as _check, hash_quantum, packed_quantum
from odie_amd import _lib
from odie_amd.config import grid_levels
from odie_amd.encoding import grid_backward, grid_forward
from odie_amd import synth

pytestmark = pytest.mark.gpu


def rows_of(levels):
    return [(r.scale, r.resolution, r.size, r.offset, r.hashed) for r in levels]


def hash_bar(xy, up, levels, features, total, offsets=None, expert_params=None):
    """The oracle's gradient with each entry's bar: (expected, sum|c|, count, quantum)."""
    rows = rows_of(levels)
    expected, magnitude, counts = oracle.hash_backward(xy, up, rows, features, total, offsets=offsets,
                                                       expert_params=expert_params, counts=True)
    return expected, magnitude, counts, hash_quantum(up, rows, features, total, offsets=offsets,
                                                     expert_params=expert_params)


def packed_bar(xy, up, layout, total):
    expected, magnitude, counts = oracle.packed_backward(xy, up, layout, total, counts=True)
    return expected, magnitude, counts, packed_quantum(up, layout, total)


def check_gradient(gpu, bar, label=''):
    _check(gpu.detach().cpu().numpy(), *bar, label=label)


def encoding(levels=16, base=16, log2=19, scale=1.38, features=2):
    return dict(n_levels=levels, base_resolution=base, log2_hashmap_size=log2, per_level_scale=scale,
                n_features_per_level=features)


@pytest.mark.parametrize('dtype', [torch.float16, torch.float32])
def test_single_grid_forward_bit_exact(dtype):
    enc = encoding()
    levels, entries = grid_levels(enc)
    n = 1 << 16
    xy = synth.coordinates(0, n)
    values = synth.table(0, entries * 2)
    table = values.astype(np.float16) if dtype == torch.float16 else values
    out = grid_forward(torch.from_numpy(xy).cuda(), torch.from_numpy(table).cuda(), levels, 2)
    expected = oracle.hash_forward(xy, table, rows_of(levels), 2, threads=0)
    got = out.cpu().numpy()
    view = np.uint16 if dtype == torch.float16 else np.uint32
    mismatch = got.view(view) != expected.view(view)
    assert not mismatch.any(), 'mismatches at %s' % (np.argwhere(mismatch)[:5],)


@pytest.mark.parametrize('log2', [14, 19])
@pytest.mark.parametrize('mode', [0, 1, 2], ids=['single', 'pairs', 'auto'])
def test_forward_corner_pairs_bit_exact(mode, log2):
    """The fp16 forward's 16-byte corner-pair loads (tuning key paired_loads: off, on, and the
    default, on only for tables past 4 MB) against the oracle, on a table that fits one L2
    (2^14 entries) and one that does not (2^19): the odd corner outside its group of four
    entries takes the single load."""
    enc = encoding(log2=log2)
    levels, entries = grid_levels(enc)
    n = 1 << 15
    xy = synth.coordinates(3, n)
    table = synth.table(3, entries * 2).astype(np.float16)
    out = _tuned('paired_loads', mode, 2, lambda: grid_forward(torch.from_numpy(xy).cuda(),
                                                               torch.from_numpy(table).cuda(), levels, 2))
    expected = oracle.hash_forward(xy, table, rows_of(levels), 2, threads=0)
    mismatch = out.cpu().numpy().view(np.uint16) != expected.view(np.uint16)
    assert not mismatch.any(), 'mismatches at %s' % (np.argwhere(mismatch)[:5],)


@pytest.mark.parametrize('experts', [1, 3])
def test_handoff_band_lists_bit_identical(experts):
    """The forward filling the handoff with the owner's band lists (2^19-entry levels, whose
    passes the owner bands) and walking the coordinates in band order, and the backward reading
    them: features and gradient bit-identical to the plain pair, one expert and three."""
    from odie_amd.encoding import grid_handoff_bytes
    enc = encoding(log2=19)
    levels, entries = grid_levels(enc)
    n = (1 << 17) + 333
    params = entries * 2
    xy = torch.from_numpy(synth.coordinates(5, n)).cuda()
    table = torch.from_numpy(synth.table(5, experts * params).astype(np.float16)).cuda()
    upstream = torch.from_numpy(synth.upstream(5, n, 32)).cuda().half()
    offsets = torch.tensor([k * n // experts for k in range(experts + 1)], dtype=torch.int32).cuda()
    size = grid_handoff_bytes(n, levels, 2, experts=experts, expert_params=params)
    assert size >= 12 * n   # band lists: a 4-byte index and an 8-byte (x, y) per coordinate
    handoff = torch.empty(size, dtype=torch.uint8, device='cuda')
    kw = dict(offsets=offsets, experts=experts, expert_params=params)
    plain = grid_forward(xy, table, levels, 2, **kw)
    walked = grid_forward(xy, table, levels, 2, handoff=handoff, **kw)
    assert np.array_equal(walked.cpu().numpy().view(np.uint16), plain.cpu().numpy().view(np.uint16))
    formed = grid_backward(xy, upstream, levels, 2, **kw)
    read = grid_backward(xy, upstream, levels, 2, handoff=handoff, **kw)
    assert np.array_equal(read.cpu().numpy().view(np.uint32), formed.cpu().numpy().view(np.uint32))


@pytest.fixture(params=[(1, 1), (1, 0), (0, 0)], ids=['owner-banded', 'owner', 'atomics'])
def backward_mode(request):
    mode, banded = request.param
    _lib.set_tuning('backward_mode', mode)
    _lib.set_tuning('banded', banded)
    yield mode
    _lib.set_tuning('backward_mode', 1)
    _lib.set_tuning('banded', 2)


def _tuned(key, value, default, call):
    _lib.set_tuning(key, value)
    try:
        return call()
    finally:
        _lib.set_tuning(key, default)


@pytest.mark.parametrize('lds_bytes', [0, 65536])
def test_single_grid_backward_tolerance(lds_bytes, backward_mode):
    enc = encoding()
    levels, entries = grid_levels(enc)
    n = 1 << 16
    xy = synth.coordinates(0, n)
    up = synth.upstream(0, n, 32)
    _lib.set_tuning('lds_bytes', lds_bytes)
    _lib.set_tuning('owner_lds_bytes', 162816 if lds_bytes else 32768)
    try:
        grad = grid_backward(torch.from_numpy(xy).cuda(), torch.from_numpy(up).cuda(), levels, 2,
                             expert_params=entries * 2)
    finally:
        _lib.set_tuning('lds_bytes', 65536)
        _lib.set_tuning('owner_lds_bytes', 162816)
    check_gradient(grad, hash_bar(xy, up, levels, 2, entries * 2),
                   'single grid lds=%d mode=%d' % (lds_bytes, backward_mode))


def test_owner_backward_is_deterministic():
    levels, entries = grid_levels(encoding(log2=14))
    n = 30000
    xy = torch.from_numpy(synth.coordinates(21, n)).cuda()
    up = torch.from_numpy(synth.upstream(21, n, 32)).cuda()
    first = grid_backward(xy, up, levels, 2, expert_params=entries * 2)
    second = grid_backward(xy, up, levels, 2, expert_params=entries * 2)
    assert torch.equal(first, second)


def test_owner_backward_is_order_independent():
    """Coordinates in row bands, x ascending within a band (the order of a stratified draw), and
    the same rows shuffled within each expert give the same fixed-point sums bit for bit: every
    coordinate is added once whichever lane takes it (dense levels spread a wave over its block,
    hashed levels take consecutive coordinates).  The upstream has one magnitude per level and
    random signs, so every range (an expert's, or a split of one) bounds the same fixed-point
    scale in both orders.  The banded order is also checked against the oracle."""
    levels, entries = grid_levels(encoding(log2=14))
    params, experts, per = entries * 2, 64, 4096
    n = experts * per
    xy = synth.coordinates(31, n)
    rng = np.random.default_rng(31)
    magnitude = 2.0 ** -(np.arange(32) // 2 % 4)
    up = (np.where(rng.random((n, 32)) < 0.5, -1.0, 1.0) * magnitude).astype(np.float16)
    banded, shuffled = [], []
    for e in range(experts):
        rows = np.arange(e * per, (e + 1) * per)
        bands = np.floor(xy[rows, 1] * 64).astype(np.int64)
        banded.append(rows[np.lexsort((xy[rows, 0], bands))])
        shuffled.append(rng.permutation(rows))
    offsets = np.arange(0, n + 1, per, dtype=np.int32)
    d_off = torch.from_numpy(offsets).cuda()
    grads = []
    for order in (np.concatenate(banded), np.concatenate(shuffled)):
        grads.append(grid_backward(torch.from_numpy(xy[order]).cuda(), torch.from_numpy(up[order]).cuda(), levels, 2,
                                   offsets=d_off, experts=experts, expert_params=params))
    assert torch.equal(grads[0], grads[1])
    order = np.concatenate(banded)
    check_gradient(grads[0], hash_bar(xy[order], up[order], levels, 2, experts * params, offsets=offsets,
                                      expert_params=params), 'banded')


def _expert_batch(seed, log2, experts, n, outside=False):
    levels, entries = grid_levels(encoding(log2=log2))
    counts = np.random.default_rng(seed).multinomial(n, np.ones(experts) / experts)
    offsets = torch.from_numpy(np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)).cuda()
    xy = synth.coordinates(seed, n)
    if outside:   # off the unit square: the band lists' last slot, visited by every slice
        xy[::97, 0] = 1.5
        xy[5::101, 1] = -0.25
        xy[7::211] = (-3.0, 2.5)
    up = torch.from_numpy(synth.upstream(seed, n, 32)).cuda()
    return levels, entries * 2, offsets, torch.from_numpy(xy).cuda(), up


@pytest.mark.parametrize('log2,experts,n,outside', [(16, 64, 1 << 20, False), (14, 16, 300000, True),
                                                    (19, 1, 1 << 20, False), (12, 3, 5000, True)])
def test_banded_owner_matches_unbanded(log2, experts, n, outside):
    """The banded fine passes skip only coordinates whose corners cannot reach the slice, and
    every pass bounds its fixed-point scale over the expert's coordinates: where the unbanded
    owner does not split a pass either (64 experts of 16384 coordinates), the gradient is the
    same integer sum bit for bit; otherwise both are within fp32 rounding of each other."""
    levels, params, offsets, xy, up = _expert_batch(log2, log2, experts, n, outside)
    run = lambda: grid_backward(xy, up.half(), levels, 2, offsets=offsets, experts=experts, expert_params=params)
    banded = _tuned('banded', 1, 2, run)
    plain = _tuned('banded', 0, 2, run)
    got, want = banded.cpu().numpy(), plain.cpu().numpy()
    if experts == 64:
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    else:
        finite = np.isfinite(want)
        assert np.array_equal(finite, np.isfinite(got))
        assert np.allclose(got[finite], want[finite], rtol=1e-5, atol=1e-6 * np.abs(want[finite]).max())


def test_single_expert_band_order_against_the_oracle():
    """One expert (its offsets dropped: every row is its) with band lists: the backward transposes
    the upstream in band-list order and every pass reads it at the list positions.  Off-square
    coordinates (the lists' last slot) and a ragged last 128-row record; the gradient within the
    oracle's bar, and within fp32 rounding of the index-order (unbanded) owner."""
    levels, entries = grid_levels(encoding(log2=17))
    params, n = entries * 2, 300001
    xy = synth.coordinates(41, n)
    xy[::97, 0] = 1.5
    xy[7::211] = (-3.0, 2.5)
    up = synth.upstream(41, n, 32)
    d_xy, d_up = torch.from_numpy(xy).cuda(), torch.from_numpy(up).cuda().half()
    run = lambda: grid_backward(d_xy, d_up, levels, 2, expert_params=params)
    banded = _tuned('banded', 1, 2, run)
    plain = _tuned('banded', 0, 2, run)
    got, want = banded.cpu().numpy(), plain.cpu().numpy()
    assert np.allclose(got, want, rtol=1e-5, atol=1e-6 * np.abs(want).max())
    check_gradient(banded, hash_bar(xy, up.astype(np.float16), levels, 2, params), 'band order')


@pytest.mark.parametrize('log2,experts,n', [(19, 1, 1 << 20), (14, 16, 300000), (12, 3, 5000)])
def test_banded_splits_are_exact(log2, experts, n):
    """Banded splits write 64-bit partial sums at one scale per pass and are added exactly: the
    gradient is the same bit for bit however finely the passes are split."""
    levels, params, offsets, xy, up = _expert_batch(log2 + 1, log2, experts, n)
    run = lambda: grid_backward(xy, up.half(), levels, 2, offsets=offsets, experts=experts, expert_params=params)
    _lib.set_tuning('banded', 1)
    try:
        auto = run()
        fine = _tuned('split_target', 1024, 0, run)
        whole = _tuned('split_target', 1 << 30, 0, run)
    finally:
        _lib.set_tuning('banded', 2)
    assert torch.equal(auto, fine) and torch.equal(auto, whole)


@pytest.mark.parametrize('log2,experts,n', [(10, 4, 4 * 4096 - 1), (10, 4, 4 * 4096), (9, 16, 200001), (14, 1, 20000),
                                            (14, 1, 1 << 20), (13, 9, 70001)])
def test_unbanded_splits_are_exact(log2, experts, n):
    """Few experts without band lists: every pass splits into shares of at least 2048 coordinates of an
    expert's (the first size is one short of two), whose 64-bit partials add exactly: the gradient equals
    the unsplit one (band lists, one item a pass) bit for bit, added to a gradient with accumulate."""
    levels, params, offsets, xy, up = _expert_batch(log2 + 2, log2, experts, n, outside=True)
    start = torch.linspace(-1, 1, experts * params, device='cuda')
    run = lambda: [grid_backward(xy, up.half(), levels, 2, offsets=offsets, experts=experts, expert_params=params),
                   grid_backward(xy, up.half(), levels, 2, offsets=offsets, experts=experts, expert_params=params,
                                 gradient=start.clone(), accumulate=True)]
    split = _tuned('banded', 0, 2, run)
    whole = _tuned('banded', 1, 2, lambda: _tuned('split_target', 1 << 30, 0, run))
    for got, want in zip(split, whole):
        assert torch.equal(got, want)


@pytest.mark.parametrize('log2,experts,n', [(13, 4, 1 << 20), (14, 4, 1 << 18), (11, 9, 150001), (7, 1, 100000),
                                            (9, 120, 1 << 19), (16, 2, 50000), (14, 15, 120000)])
def test_unbanded_splits_of_one_round_are_exact(log2, experts, n):
    """The group and the fine passes split in different ways (one pass alone, two ways left, no room for a
    second way, the group alone split): the gradient equals the unsplit one bit for bit."""
    levels, params, offsets, xy, up = _expert_batch(log2 + 3, log2, experts, n)
    run = lambda: grid_backward(xy, up.half(), levels, 2, offsets=offsets, experts=experts, expert_params=params)
    split = _tuned('banded', 0, 2, run)
    assert torch.equal(split, _tuned('banded', 1, 2, lambda: _tuned('split_target', 1 << 30, 0, run)))


def test_banded_owner_with_unordered_offsets():
    """Offsets that decrease somewhere make the expert ranges overlap: the band lists are not
    used and the fine passes walk the experts' index ranges, as the unbanded owner does."""
    levels, entries = grid_levels(encoding(log2=14))
    experts, n = 16, 40000
    bounds = np.linspace(0, n, experts + 1).astype(np.int32)
    bounds[5], bounds[6] = bounds[6], bounds[5]
    offsets = torch.from_numpy(bounds).cuda()
    xy = torch.from_numpy(synth.coordinates(41, n)).cuda()
    up = torch.from_numpy(synth.upstream(41, n, 32)).cuda()
    run = lambda: grid_backward(xy, up, levels, 2, offsets=offsets, experts=experts, expert_params=entries * 2)
    assert torch.equal(_tuned('banded', 1, 2, run), _tuned('banded', 0, 2, run))


def test_experts_forward_and_backward(backward_mode):
    enc = encoding(log2=14)
    levels, entries = grid_levels(enc)
    experts, params = 16, entries * 2
    n = 40000
    rng = np.random.default_rng(1)
    counts = rng.multinomial(n, np.r_[np.zeros(2), np.ones(experts - 3), [0.0]] / (experts - 3))
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)   # empty experts 0, 1, 15
    xy = synth.coordinates(3, n)
    table = synth.table(3, experts * params).astype(np.float16)
    up = synth.upstream(3, n, 32)
    d_xy, d_off = torch.from_numpy(xy).cuda(), torch.from_numpy(offsets).cuda()
    out = grid_forward(d_xy, torch.from_numpy(table).cuda(), levels, 2, offsets=d_off, experts=experts,
                       expert_params=params)
    expected = oracle.hash_forward(xy, table, rows_of(levels), 2, offsets=offsets, expert_params=params, threads=0)
    assert np.array_equal(out.cpu().numpy().view(np.uint16), expected.view(np.uint16))
    grad = grid_backward(d_xy, torch.from_numpy(up).cuda(), levels, 2, offsets=d_off, experts=experts,
                         expert_params=params)
    check_gradient(grad, hash_bar(xy, up, levels, 2, experts * params, offsets=offsets, expert_params=params),
                   'experts')


@pytest.mark.parametrize('features,n_levels,width,n', [(1, 5, 5, 1000), (4, 3, 16, 777), (8, 2, 16, 513),
                                                        (2, 20, 40, 3001), (2, 16, 36, 1029), (2, 1, 2, 1)])
def test_shapes_and_padding(features, n_levels, width, n, backward_mode):
    enc = encoding(levels=n_levels, base=3, log2=10, scale=1.7, features=features)
    levels, entries = grid_levels(enc)
    xy = synth.coordinates(5, n)
    xy[0] = (0.0, 0.0)
    if n > 1:
        xy[1] = (1.0, 1.0)
    table = synth.table(5, entries * features, -1.0, 1.0).astype(np.float16)
    out = grid_forward(torch.from_numpy(xy).cuda(), torch.from_numpy(table).cuda(), levels, features, width=width)
    expected = oracle.hash_forward(xy, table, rows_of(levels), features, width=width)
    assert np.array_equal(out.cpu().numpy().view(np.uint16), expected.view(np.uint16))
    up = synth.upstream(5, n, width)
    up[:, ::3] = 0   # zero upstream values are skipped
    grad = grid_backward(torch.from_numpy(xy).cuda(), torch.from_numpy(up).cuda(), levels, features,
                         expert_params=entries * features)
    check_gradient(grad, hash_bar(xy, up, levels, features, entries * features), 'F=%d L=%d' % (features, n_levels))


def test_fp32_upstream_and_accumulate(backward_mode):
    levels, entries = grid_levels(encoding(levels=8, log2=12))
    n = 5000
    xy = synth.coordinates(7, n)
    up = synth.normal(7, 'up32', n * 16).astype(np.float32).reshape(n, 16)
    d_xy = torch.from_numpy(xy).cuda()
    grad = grid_backward(d_xy, torch.from_numpy(up).cuda(), levels, 2, expert_params=entries * 2)
    grad = grid_backward(d_xy, torch.from_numpy(up).cuda(), levels, 2, expert_params=entries * 2, gradient=grad,
                         accumulate=True)
    expected, magnitude, counts, quantum = hash_bar(xy, up, levels, 2, entries * 2)
    check_gradient(grad, (2 * expected, 2 * magnitude, 2 * counts, quantum), 'fp32 upstream x2')


def test_empty_input_and_xcd_order_invariance():
    levels, entries = grid_levels(encoding(levels=4, log2=10))
    empty = torch.zeros((0, 2), device='cuda')
    assert grid_forward(empty, torch.zeros(entries * 2, dtype=torch.float16, device='cuda'), levels, 2).shape == (0, 8)
    grad = grid_backward(empty, torch.zeros((0, 8), dtype=torch.float16, device='cuda'), levels, 2,
                         expert_params=entries * 2)
    assert not grad.any()
    xy = torch.from_numpy(synth.coordinates(9, 3000)).cuda()
    table = torch.from_numpy(synth.table(9, entries * 2).astype(np.float16)).cuda()
    first = grid_forward(xy, table, levels, 2)
    _lib.set_tuning('xcd_remap', 0)
    try:
        second = grid_forward(xy, table, levels, 2)
    finally:
        _lib.set_tuning('xcd_remap', 1)
    assert torch.equal(first, second)


def test_grid_encoding_module_autograd():
    from odie_amd.encoding import GridEncoding
    module = GridEncoding(encoding(levels=6, log2=12), dtype=torch.float16)
    with torch.no_grad():
        module.params.copy_(torch.from_numpy(synth.table(11, module.n_params, -1, 1)))
    xy = torch.from_numpy(synth.coordinates(11, 2048)).cuda()
    out = module(xy)
    weight = torch.from_numpy(synth.upstream(11, 2048, 12)).cuda()
    (out.float() * weight.float()).sum().backward()
    check_gradient(module.params.grad, hash_bar(xy.cpu().numpy(), weight.cpu().numpy(), module.levels, 2,
                                                module.n_params), 'autograd')


def _packed_layout(seed, resolutions=(8, 13, 20, 32, 51, 81), dims=(2, 2, 2, 2, 1, 4), dense=3):
    from odie_amd.model import make_layout, plane_closure
    rng = np.random.default_rng(seed)
    supports, caps = [], []
    for level, r in enumerate(resolutions):
        support = np.ones(r * r, dtype=bool) if level < dense else rng.random(r * r) < 0.3
        nodes = plane_closure(torch.as_tensor(support), r)
        supports.append(torch.as_tensor(support))
        caps.append(min((r * r + 7) // 8 * 8, (nodes.numel() + 7) // 8 * 8 + 8 * level))
    config = dict(resolutions=list(resolutions), n_levels=len(resolutions), representation='xy_planes',
                  coarse_levels=0, gate_topology='shared', gate_position='feature', initial_active_prefix=3)
    return make_layout(config, supports, list(dims), caps)


def _packed_gradient(layout, xy, up, **tuning):
    from odie_amd.model import packed_backward
    dev = {k: layout[k].cuda() for k in ('descriptors', 'node_bitmap', 'node_prefix', 'bitmap')}
    settings = dict(dict(packed_owner=1), **tuning)
    for key, value in settings.items():
        _lib.set_tuning(key, value)
    try:
        return packed_backward(xy, up, dev['descriptors'], dev['node_bitmap'], dev['node_prefix'], dev['bitmap'],
                               layout['params'])
    finally:
        _lib.set_tuning('packed_owner', 0)
        _lib.set_tuning('packed_splits', 0)


# Nine levels of 8..512 cells (the finer ones 30% supported), mixed F1/F2/F4: about 1.4e6
# parameters, so the owner's slices span several levels at the coarse end and split the fine ones.
BIG_PLANES = dict(resolutions=(8, 13, 20, 32, 64, 128, 256, 384, 512), dims=(2, 2, 2, 2, 4, 2, 2, 1, 2), dense=5)


def test_packed_owner_matches_oracle_and_atomics():
    """The owner-computes packed backward against the oracle (multi-slice layout, off-square and
    edge coordinates) and against the global-atomics kernel it replaces (fp32 order only)."""
    layout = _packed_layout(4, **BIG_PLANES)
    n, width = 30000, 32
    xy = synth.coordinates(17, n)
    xy[:4] = [(0, 0), (1, 1), (0, 1), (1, 0)]
    up = synth.upstream(17, n, width)
    d_xy, d_up = torch.from_numpy(xy).cuda(), torch.from_numpy(up).cuda()
    owner = _packed_gradient(layout, d_xy, d_up)
    atomics = _packed_gradient(layout, d_xy, d_up, packed_owner=0)
    host = {k: layout[k].numpy() for k in ('descriptors', 'node_bitmap', 'node_prefix', 'bitmap')}
    bar = packed_bar(xy, up, host, layout['params'])
    check_gradient(owner, bar, 'packed owner')
    check_gradient(atomics, bar, 'packed atomics')


@pytest.mark.parametrize('seed,n', [(5, 30000), (6, 4097), (7, 1)])
def test_packed_owner_splits_are_exact(seed, n):
    """Splits share one fixed-point scale per slice and sum 64-bit partials: the gradient is the
    same bit for bit for any split count, and from run to run."""
    layout = _packed_layout(seed, **BIG_PLANES)
    d_xy = torch.from_numpy(synth.coordinates(seed, n)).cuda()
    d_up = torch.from_numpy(synth.upstream(seed, n, 32)).cuda()
    first = _packed_gradient(layout, d_xy, d_up)
    for splits in (1, 3, 7):
        assert torch.equal(first, _packed_gradient(layout, d_xy, d_up, packed_splits=splits)), splits
    assert torch.equal(first, _packed_gradient(layout, d_xy, d_up))


def test_packed_planes_forward_backward():
    from odie_amd.model import PackedQuery
    layout = _packed_layout(2)
    n, width = 20000, 13
    xy = synth.coordinates(13, n)
    xy[:4] = [(0, 0), (1, 1), (0, 1), (1, 0)]
    grid = synth.table(13, layout['params'], -0.5, 0.5)
    host = {k: layout[k].numpy() for k in ('descriptors', 'node_bitmap', 'node_prefix', 'bitmap')}
    expected, vis = oracle.packed_forward(xy, grid, host, width)
    dev = {k: layout[k].cuda() for k in ('descriptors', 'node_bitmap', 'node_prefix', 'bitmap')}
    d_grid = torch.from_numpy(grid).cuda().requires_grad_(True)
    features, visible = PackedQuery.apply(torch.from_numpy(xy).cuda(), d_grid, dev['descriptors'], dev['node_bitmap'],
                                          dev['node_prefix'], dev['bitmap'], width)
    assert np.array_equal(features.detach().cpu().numpy().view(np.uint16), expected.view(np.uint16))
    assert np.array_equal(visible.cpu().numpy(), vis)
    up = synth.upstream(13, n, width)
    features.backward(torch.from_numpy(up).cuda())
    check_gradient(d_grid.grad, packed_bar(xy, up, host, layout['params']), 'packed')


def test_owner_scale_sees_both_features():
    """Regression: the largest |upstream| of a row block must cover both features of a level.
    Feature 0 carries values ~1e3 while feature 1 is ~1e-3 and largest in a row whose feature 0
    is tiny; a maximum taken over packed 32-bit words follows feature 1 only, picks a scale
    2^40 too fine and saturates the fixed-point contributions of feature 0."""
    levels, entries = grid_levels(encoding(log2=12))
    n = 4096
    xy = synth.coordinates(31, n)
    up = np.empty((n, 32), dtype=np.float32)
    up[:, 0::2] = np.where(synth.uniform(31, 'sign', n * 16).reshape(n, 16) < 0.5, -1000.0, 1000.0)
    up[:, 1::2] = 0.001
    up[7, 1::2] = 0.002
    up[7, 0::2] = 0.0001
    up = up.astype(np.float16)
    grad = grid_backward(torch.from_numpy(xy).cuda(), torch.from_numpy(up).cuda(), levels, 2,
                         expert_params=entries * 2)
    bar = hash_bar(xy, up, levels, 2, entries * 2)
    check_gradient(grad, bar, 'two-scale upstream')
    _check_relative(grad, bar, 'two-scale upstream')


def _check_relative(gpu, bar, label):
    """Every touched entry whose contributions are not all below 10^4 quanta (an entry reached
    only through corner weights of order 1e-5 or less) meets 1e-4 * sum|c| alone, the north
    star's relative bar, with no quantum term; and those exceptions are rare."""
    expected, magnitude, counts, quantum = bar
    got = gpu.detach().cpu().numpy().astype(np.float64)
    touched = counts > 0
    coarse = counts * quantum * 0.5 > 1e-4 * magnitude
    strict = np.abs(got - expected) <= 1e-4 * magnitude
    assert strict[touched & ~coarse].all(), '%s: %d entries miss the relative bar' % (
        label, (touched & ~coarse & ~strict).sum())
    assert (touched & coarse).sum() <= 1e-3 * touched.sum(), '%s: %d of %d entries below 10^4 quanta' % (
        label, (touched & coarse).sum(), touched.sum())


def _level_magnitudes(seed, n, levels, features, magnitude):
    """Upstream [n, levels * features] of random signs, column l * features + c of size
    magnitude[l][c] (1 +- 1/2 per row)."""
    rng = np.random.default_rng(seed)
    scale = np.repeat(np.asarray(magnitude, dtype=np.float64).reshape(1, levels * features), n, axis=0)
    sign = np.where(rng.random((n, levels * features)) < 0.5, -1.0, 1.0)
    return (sign * scale * (0.5 + rng.random((n, levels * features)))).astype(np.float16)


@pytest.mark.parametrize('experts', [1, 16])
def test_owner_scale_per_level_in_the_coarse_group(experts, backward_mode):
    """Levels that share the coarse-group pass carry upstream 10^5 apart (as a router step whose
    coarse gates differ that much can), and the two features of some levels 10^5 apart too.
    Every column has its own fixed-point scale, so the small levels keep their precision: each
    entry within its own bar, and every entry not reached only through tiny corner weights within
    1e-4 of its contribution scale alone."""
    levels, entries = grid_levels(encoding(log2=12))
    n = experts * 6000
    xy = synth.coordinates(43, n)
    magnitude = [[1e3, 1e3] if l % 2 == 0 else [1e-2, 1e-7 if l % 4 == 1 else 1e-2] for l in range(16)]
    up = _level_magnitudes(43, n, 16, 2, magnitude)
    params = entries * 2
    offsets = np.linspace(0, n, experts + 1).astype(np.int32) if experts > 1 else None
    grad = grid_backward(torch.from_numpy(xy).cuda(), torch.from_numpy(up).cuda(), levels, 2,
                         offsets=None if offsets is None else torch.from_numpy(offsets).cuda(), experts=experts,
                         expert_params=params)
    bar = hash_bar(xy, up, levels, 2, experts * params, offsets=offsets, expert_params=params)
    check_gradient(grad, bar, 'levels 10^5 apart, mode %d' % backward_mode)
    _check_relative(grad, bar, 'levels 10^5 apart, mode %d' % backward_mode)


def test_packed_owner_scale_per_level():
    """The packed-plane owner's slices span several coarse levels; their upstream columns are
    10^6 apart (alternating by level, and by feature within the four-feature level): each keeps
    its own scale, for any split count."""
    layout = _packed_layout(8, **BIG_PLANES)
    n, width = 20000, 32
    xy = synth.coordinates(47, n)
    dims = BIG_PLANES['dims']
    magnitude = np.ones(width)
    column = 0
    for level, f in enumerate(dims):
        for c in range(f):
            magnitude[column] = 1e3 if (level + c) % 2 == 0 else 1e-3
            column += 1
    rng = np.random.default_rng(47)
    up = (np.where(rng.random((n, width)) < 0.5, -1.0, 1.0) * magnitude * (0.5 + rng.random((n, width))))
    up = up.astype(np.float16)
    d_xy, d_up = torch.from_numpy(xy).cuda(), torch.from_numpy(up).cuda()
    host = {k: layout[k].numpy() for k in ('descriptors', 'node_bitmap', 'node_prefix', 'bitmap')}
    bar = packed_bar(xy, up, host, layout['params'])
    first = _packed_gradient(layout, d_xy, d_up)
    check_gradient(first, bar, 'packed owner, levels 10^6 apart')
    _check_relative(first, bar, 'packed owner, levels 10^6 apart')
    for splits in (1, 5):
        assert torch.equal(first, _packed_gradient(layout, d_xy, d_up, packed_splits=splits)), splits


@pytest.mark.parametrize('experts,n', [(8, 50000), (1, 4097), (3, 1)])
def test_planes_backward_equals_rows(experts, n):
    """odie_grid_backward_planes on the upstream in the decoder's planes layout (level-major fp16
    pairs and per-column 128-row maxima) gives odie_grid_backward's gradient bit for bit, and
    accumulates into a given gradient."""
    from odie_amd.experts import ExpertGrid
    encoding = dict(n_levels=16, n_features_per_level=2, log2_hashmap_size=12, base_resolution=8, per_level_scale=1.4)
    grid = ExpertGrid(encoding, experts)
    coords = torch.from_numpy(synth.coordinates(51, n)).cuda()
    counts = np.diff(np.linspace(0, n, experts + 1).astype(np.int64))
    offsets = torch.from_numpy(np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)).cuda()
    upstream = torch.from_numpy(synth.upstream(51, n, 32)).cuda()
    planes = upstream.view(torch.int32).t().contiguous()
    records = (n + 127) // 128
    column = torch.zeros((records * 128, 32), dtype=torch.float32, device='cuda')
    column[:n] = upstream.abs().float()
    blockmax = column.view(records, 128, 32).amax(dim=1).contiguous()
    rows = grid.backward(coords, offsets, upstream)
    via_planes = grid.backward_planes(coords, offsets, planes, blockmax)
    assert torch.equal(rows.view(torch.int32), via_planes.view(torch.int32))
    twice = grid.backward_planes(coords, offsets, planes, blockmax, gradient=via_planes.clone(), accumulate=True)
    assert torch.equal(twice, 2 * rows)


@pytest.mark.parametrize('log2,experts,n,outside', [(16, 64, 1 << 20, False), (14, 16, 300000, True),
                                                    (15, 3, 5000, True), (16, 1, 65536, False)])
def test_owner_masks_are_bit_identical(log2, experts, n, outside):
    """Hashed slices that walk only the coordinates whose slice masks reach them form the same
    integer sums as slices that walk every coordinate: the gradient bit for bit (coordinates off
    the unit square included), for 2- to 8-block levels."""
    levels, params, offsets, xy, up = _expert_batch(log2 + 3, log2, experts, n, outside)
    run = lambda: grid_backward(xy, up.half(), levels, 2, offsets=offsets, experts=experts, expert_params=params)
    _lib.set_tuning('banded', 0)
    try:
        masked = _tuned('owner_masks', 1, 1, run)
        plain = _tuned('owner_masks', 0, 1, run)
    finally:
        _lib.set_tuning('banded', 2)
    assert torch.equal(masked.view(torch.int32), plain.view(torch.int32))


# Levels on both sides of the tile pass's limits: coarse (48 and below), the smallest tiles, a level
# whose tile fills LDS several times over (F = 4, 1200 cells a side), mixed features.
TILE_PLANES = dict(resolutions=(8, 47, 48, 49, 50, 65, 130, 333, 1200), dims=(2, 4, 1, 2, 4, 1, 2, 2, 4), dense=4)


def _without_tiles(layout, xy, up):
    _lib.set_tuning('packed_tiles', 0)
    try:
        return _packed_gradient(layout, xy, up, packed_owner=0)
    finally:
        _lib.set_tuning('packed_tiles', 1)


@pytest.mark.parametrize('n,width,spread', [(1024, 22, 'uniform'), (16384, 22, 'uniform'), (20001, 22, 'edges'),
                                            (40000, 22, 'corner'),
                                            (16385, 32, 'outside'), (70000, 20, 'stratified'), (16384, 2, 'uniform')])
def test_packed_tiles_match_the_oracle_and_the_atomics(n, width, spread):
    """The packed backward by spatial tiles: bins' edges, corners that wrap past a row or the plane,
    coordinates off the unit square, every coordinate in one tile, fewer upstream columns than
    features."""
    layout = _packed_layout(21, **TILE_PLANES)
    xy = synth.coordinates(21, n)
    if spread == 'edges':       # bin edges, and the last half cell that wraps
        grid = np.arange(33, dtype=np.float32) / 32
        xy[:33 * 33] = np.stack(np.meshgrid(grid, grid), axis=-1).reshape(-1, 2)
        xy[2000:6000, 0] = 1.0 - np.float32(1e-4) * xy[2000:6000, 0]
        xy[6000:9000, 1] = 1.0 - np.float32(1e-4) * xy[6000:9000, 1]
    elif spread == 'corner':
        xy = xy * np.float32(0.03)
    elif spread == 'outside':
        xy = (xy * 3 - 1).astype(np.float32)
    elif spread == 'stratified':
        side = 256
        j = np.arange(n)
        xy = ((np.stack([j % side, j // side % side], axis=1) + xy) / side).astype(np.float32)
    up = synth.upstream(21, n, width)
    d_xy, d_up = torch.from_numpy(xy).cuda(), torch.from_numpy(up).cuda()
    tiles = _packed_gradient(layout, d_xy, d_up, packed_owner=0)
    atomics = _without_tiles(layout, d_xy, d_up)
    if spread == 'outside':     # the oracle takes the unit square; the kernels clamp the cell
        difference = (tiles.double() - atomics.double()).abs()
        assert float(difference.max()) <= 1e-5 * float(atomics.abs().max())
        return
    host = {k: layout[k].numpy() for k in ('descriptors', 'node_bitmap', 'node_prefix', 'bitmap')}
    columns = np.zeros((n, max(width, 22)), dtype=np.float16)   # a feature past the upstream's columns gets nothing
    columns[:, :width] = up
    bar = packed_bar(xy, columns, host, layout['params'])
    check_gradient(tiles, bar, 'packed tiles, ' + spread)
    check_gradient(atomics, bar, 'packed atomics, ' + spread)


# Planes whose tiles take 2 pieces (1290 cells, F = 2), 3 (1200, F = 4) and 10 (3300, F = 2): summed by
# tiles from 65536 and 98304 coordinates on, and never.
FINE_PLANES = dict(resolutions=(8, 13, 49, 1290, 1200, 3300), dims=(1, 2, 1, 2, 4, 2), dense=3)


@pytest.mark.parametrize('n', [2000, 65535, 65536, 98304])
def test_packed_tiles_of_fine_planes(n):
    layout = _packed_layout(26, **FINE_PLANES)
    xy, up = synth.coordinates(26, n), synth.upstream(26, n, 12)
    xy[:500] = 1.0 - np.float32(1e-4) * xy[:500]     # corners that wrap
    host = {k: layout[k].numpy() for k in ('descriptors', 'node_bitmap', 'node_prefix', 'bitmap')}
    expected, magnitude, counts = oracle.packed_backward(xy, up, host, layout['params'], counts=True)
    got = _packed_gradient(layout, torch.from_numpy(xy).cuda(), torch.from_numpy(up).cuda(), packed_owner=0)
    # an fp32 rounding per contribution added in memory, or per partial sum, and one for the sum
    assert (np.abs(got.cpu().numpy().astype(np.float64) - expected) <= (counts + 33) * 2.0 ** -24 * magnitude).all()


def test_packed_tiles_of_a_fine_plane_cost_no_more_than_the_atomics():
    """6000 cells a side: the level goes to memory (32 pieces a tile took three times as long)."""
    layout = _packed_layout(27, resolutions=(8, 13, 20, 6000), dims=(2, 2, 2, 2), dense=3)
    n = 2048
    d_xy = torch.from_numpy(synth.coordinates(27, n)).cuda()
    d_up = torch.from_numpy(synth.upstream(27, n, 8)).cuda()
    dev = {k: layout[k].cuda() for k in ('descriptors', 'node_bitmap', 'node_prefix', 'bitmap')}
    lib, gradient = _lib.library(), torch.empty(layout['params'], device='cuda')
    scratch = torch.empty(lib.odie_packed_backward_workspace(n, 8), dtype=torch.uint8, device='cuda')

    def best(scratch):
        times = []
        for _ in range(10):
            begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            begin.record()
            _lib.check(lib.odie_packed_backward_scratch(
                d_xy.data_ptr(), n, d_up.data_ptr(), 8, dev['descriptors'].data_ptr(), 4,
                dev['node_bitmap'].data_ptr(), dev['node_prefix'].data_ptr(), dev['bitmap'].data_ptr(),
                gradient.data_ptr(), layout['params'], _lib.ptr(scratch), 0 if scratch is None else scratch.numel(),
                _lib.stream_of(gradient)))
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end))
        return min(times)
    assert best(scratch) < 2 * best(None)


def _planes_of_features(features, dense):
    """A layout's descriptors stretched to another feature count than layouts have (1, 2 or 4)."""
    layout = _packed_layout(28, resolutions=(8, 13, 20, 130, 64), dims=(1,) * 5, dense=dense)
    layout['descriptors'][:, [2, 5, 6]] *= features
    return layout, layout['params'] * features, 5 * features


@pytest.mark.parametrize('features', [3, 6, 8])
@pytest.mark.parametrize('n,dense', [(1000, 5), (5000, 3)])
def test_packed_forward_of_any_feature_count(features, n, dense):
    """Bit for bit, the last feature of the last node among them."""
    from odie_amd.model import packed_forward
    layout, params, width = _planes_of_features(features, dense)
    xy = synth.coordinates(28, n)
    xy[-200:] = 1.0 - np.float32(1e-5) * xy[-200:]
    grid = synth.table(28, params, -0.5, 0.5)
    host = {k: layout[k].numpy() for k in ('descriptors', 'node_bitmap', 'node_prefix', 'bitmap')}
    dev = [layout[k].cuda() for k in ('descriptors', 'node_bitmap', 'node_prefix', 'bitmap')]
    out, visible = packed_forward(torch.from_numpy(xy).cuda(), torch.from_numpy(grid).cuda(), *dev, width)
    want, seen = oracle.packed_forward(xy, grid, host, width)
    assert np.array_equal(out.cpu().numpy().view(np.uint16), want.view(np.uint16))
    assert np.array_equal(visible.cpu().numpy(), seen)


@pytest.mark.parametrize('features', [3, 6, 8])
@pytest.mark.parametrize('n,dense', [(1000, 5), (5000, 3), (5000, 5)])
def test_packed_backward_of_any_feature_count(features, n, dense):
    """With scratch and without: levels whose feature count has no tiles go to memory."""
    layout, params, width = _planes_of_features(features, dense)
    xy, up = synth.coordinates(28, n), synth.upstream(28, n, width)
    xy[-200:] = 1.0 - np.float32(1e-5) * xy[-200:]
    host = {k: layout[k].numpy() for k in ('descriptors', 'node_bitmap', 'node_prefix', 'bitmap')}
    expected, magnitude, counts = oracle.packed_backward(xy, up, host, params, counts=True)
    got = _packed_gradient(dict(layout, params=params), torch.from_numpy(xy).cuda(), torch.from_numpy(up).cuda(),
                           packed_owner=0)
    # an fp32 rounding per contribution added in memory, and one for the sum
    assert (np.abs(got.cpu().numpy() - expected) <= (counts + 1) * 2.0 ** -24 * magnitude).all()


def test_packed_tiles_column_scales_and_zero_upstream():
    """Columns 10^6 apart keep their own scale; an all-zero upstream clears the gradient."""
    layout = _packed_layout(22, **TILE_PLANES)
    n, width = 20000, 22
    xy = synth.coordinates(22, n)
    up = synth.upstream(22, n, width).astype(np.float32) * np.where(np.arange(width) % 2 == 0, 1e3, 1e-3)
    up = up.astype(np.float16)
    d_xy, d_up = torch.from_numpy(xy).cuda(), torch.from_numpy(up).cuda()
    host = {k: layout[k].numpy() for k in ('descriptors', 'node_bitmap', 'node_prefix', 'bitmap')}
    bar = packed_bar(xy, up, host, layout['params'])
    got = _packed_gradient(layout, d_xy, d_up, packed_owner=0)
    check_gradient(got, bar, 'packed tiles, columns 10^6 apart')
    _check_relative(got, bar, 'packed tiles, columns 10^6 apart')
    zero = _packed_gradient(layout, d_xy, torch.zeros_like(d_up), packed_owner=0)
    assert not bool(zero.any())


@pytest.mark.parametrize('case', ['outlier', 'alternate'])
def test_packed_tiles_rows_of_one_column_far_apart(case):
    """Rows of one column 2^20 and more apart: every node keeps the bits that fp32 sums of its own
    contributions have, whatever the largest row of its column is."""
    layout = _packed_layout(25, **TILE_PLANES)
    n, width = 20000, 22
    xy = synth.coordinates(25, n)
    up = synth.upstream(25, n, width).astype(np.float32)
    up *= (1e-2 if case == 'outlier' else np.where(np.arange(n) % 2 == 0, 2.0 ** 10, 2.0 ** -10)[:, None]) / np.abs(up).max()
    if case == 'outlier':
        up[7] = 6e4
    up = up.astype(np.float16)
    host = {k: layout[k].numpy() for k in ('descriptors', 'node_bitmap', 'node_prefix', 'bitmap')}
    expected, magnitude, counts = oracle.packed_backward(xy, up, host, layout['params'], counts=True)
    got = _packed_gradient(layout, torch.from_numpy(xy).cuda(), torch.from_numpy(up).cuda(), packed_owner=0)
    # an fp32 rounding for each contribution that goes to memory by itself, or for each of a node's
    # at most 32 partial sums, and one for the sum
    bound = (counts + 33) * 2.0 ** -24 * magnitude
    error = np.abs(got.cpu().numpy().astype(np.float64) - expected)
    assert (error <= bound).all(), (error / np.maximum(bound, 1e-300)).max()


@pytest.mark.parametrize('case', ['inf', 'nan', 'nan_xy', 'far_xy', 'all_inf'])
def test_packed_tiles_carry_infinities_and_nans_as_the_atomics_do(case):
    layout = _packed_layout(23, **TILE_PLANES)
    n, width = 20000, 22
    xy = synth.coordinates(23, n)
    up = synth.upstream(23, n, width)
    if case == 'inf':
        up[::997, 3] = np.inf
        up[5::1999, 20] = -np.inf
    elif case == 'nan':
        up[::1013, :] = np.nan
    elif case == 'nan_xy':
        xy[::1511, 0] = np.nan
        xy[7::1511, 1] = np.inf
    elif case == 'far_xy':
        xy[::1511, 0] = 1e12
        xy[3::1511, 1] = -1e12
    else:
        up[:, 1] = np.inf
    d_xy, d_up = torch.from_numpy(xy).cuda(), torch.from_numpy(up).cuda()
    got, want = _packed_gradient(layout, d_xy, d_up, packed_owner=0), _without_tiles(layout, d_xy, d_up)
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.isinf(got) * got.sign(), torch.isinf(want) * want.sign())
    fine = torch.isfinite(want)
    assert bool(fine.any()) and bool(fine.all()) == (case == 'far_xy')   # there: huge finite weights
    difference = (got[fine].double() - want[fine].double()).abs()
    # sums of the same fp32 products in another order, beside a rounding to 2^-30 of the column's peak
    assert float(difference.norm() / want[fine].double().norm()) < 1e-5


def test_packed_backward_scratch_is_checked_and_ragged_streams_overlap():
    """Too little scratch is refused; two streams with their own scratch do not disturb each other."""
    layout = _packed_layout(24, **TILE_PLANES)
    n, width = 30000, 22
    d_xy = torch.from_numpy(synth.coordinates(24, n)).cuda()
    d_up = torch.from_numpy(synth.upstream(24, n, width)).cuda()
    lib = _lib.library()
    need = lib.odie_packed_backward_workspace(n, width)
    assert need > 0 and lib.odie_packed_backward_workspace(100, width) == 0
    assert lib.odie_packed_backward_workspace(-1, width) == -1 and lib.odie_packed_backward_workspace(n, 1) == -1
    want = _packed_gradient(layout, d_xy, d_up, packed_owner=0)
    torch.cuda.synchronize()
    streams, results = [torch.cuda.Stream() for _ in range(2)], []
    for stream in streams:
        with torch.cuda.stream(stream):
            for _ in range(3):
                results.append(_packed_gradient(layout, d_xy, d_up, packed_owner=0))
    torch.cuda.synchronize()
    for got in results:   # the wrapped corners' and coarse levels' fp32 atomics sum in any order
        assert float((got - want).abs().max()) <= 1e-5 * float(want.abs().max())
    dev = {k: layout[k].cuda() for k in ('descriptors', 'node_bitmap', 'node_prefix', 'bitmap')}
    scratch, gradient = torch.empty(need, dtype=torch.uint8, device='cuda'), torch.empty_like(want)
    assert lib.odie_packed_backward_scratch(
        d_xy.data_ptr(), n, d_up.data_ptr(), width, dev['descriptors'].data_ptr(), 9, dev['node_bitmap'].data_ptr(),
        dev['node_prefix'].data_ptr(), dev['bitmap'].data_ptr(), gradient.data_ptr(), layout['params'],
        scratch.data_ptr(), need - 1, 0) == -1


@pytest.mark.parametrize('n,log2,levels,features,dtype', [
    (4096, 14, 16, 2, torch.float16), (1, 14, 16, 2, torch.float16), (70001, 16, 16, 2, torch.float16),
    (150000, 19, 16, 2, torch.float16), (150000, 19, 12, 4, torch.float32), (60001, 17, 20, 1, torch.float32)])
def test_grid_encoding_with_its_handoff_equals_the_plain_pair(n, log2, levels, features, dtype):
    """GridEncoding's training forward hands the backward its lists or masks: the features and the gradient
    of odie_grid_forward and odie_grid_backward bit for bit, also on a second backward, after a tuning
    change in between, and without gradients."""
    from odie_amd.encoding import GridEncoding
    module = GridEncoding(dict(n_levels=levels, n_features_per_level=features, log2_hashmap_size=log2,
                               base_resolution=16, per_level_scale=1.38), dtype=dtype)
    with torch.no_grad():
        module.params.copy_(torch.from_numpy(synth.table(31, module.n_params, -1.0, 1.0, name='enc')))
    xy = torch.from_numpy(synth.coordinates(31, n)).cuda()
    up = torch.from_numpy(synth.upstream(31, n, module.n_output_dims)).cuda().to(dtype)
    table = module.params.detach().to(dtype)
    want = grid_forward(xy, table, module.levels, features)
    gradient = grid_backward(xy, up, module.levels, features, expert_params=module.n_params)
    out = module(xy)
    assert torch.equal(out.detach(), want)
    first, = torch.autograd.grad(out, module.params, up, retain_graph=True)
    again, = torch.autograd.grad(out, module.params, up)
    assert torch.equal(first, gradient) and torch.equal(again, gradient)
    out = module(xy)
    _lib.set_tuning('banded', 0)     # another plan: the handoff is not read
    try:
        changed, = torch.autograd.grad(out, module.params, up)
        plain = grid_backward(xy, up, module.levels, features, expert_params=module.n_params)
    finally:
        _lib.set_tuning('banded', 2)
    assert torch.equal(changed, plain)
    with torch.no_grad():
        assert torch.equal(module(xy), want)


@pytest.mark.parametrize('n,log2,levels,features,dtype,formed', [
    (196607, 14, 16, 2, torch.float16, False), (196608, 14, 16, 2, torch.float16, True),    # slice masks
    (65536, 19, 16, 2, torch.float16, False), (196607, 19, 12, 4, torch.float32, False),    # band lists
    (196608, 19, 16, 2, torch.float16, True), (200003, 19, 12, 4, torch.float32, True)])
def test_grid_encoding_forms_its_handoff_where_it_pays(n, log2, levels, features, dtype, formed, monkeypatch):
    """A forward that no backward may follow does not pay for lists that a small batch's backward gains
    little from; either way the pair is the plain one bit for bit, also on a second backward, after a
    tuning change in between, and where there is no memory for the handoff."""
    from odie_amd.encoding import GridEncoding
    module = GridEncoding(dict(n_levels=levels, n_features_per_level=features, log2_hashmap_size=log2,
                               base_resolution=16, per_level_scale=1.38), dtype=dtype)
    with torch.no_grad():
        module.params.copy_(torch.from_numpy(synth.table(33, module.n_params, -1.0, 1.0, name='enc')))
    xy = torch.from_numpy(synth.coordinates(33, n)).cuda()
    up = torch.from_numpy(synth.upstream(33, n, module.n_output_dims)).cuda().to(dtype)
    out = module(xy)
    assert (out.grad_fn.saved_tensors[1] is not None) == formed
    assert torch.equal(out.detach(), grid_forward(xy, module.params.detach().to(dtype), module.levels, features))
    want = grid_backward(xy, up, module.levels, features, expert_params=module.n_params)
    for last in (False, True):
        got, = torch.autograd.grad(out, module.params, up, retain_graph=not last)
        assert torch.equal(got, want)
    out = module(xy)
    changed = _tuned('banded', 0, 2, lambda: [torch.autograd.grad(out, module.params, up)[0], grid_backward(
        xy, up, module.levels, features, expert_params=module.n_params)])
    assert torch.equal(*changed)
    monkeypatch.setattr(_lib, 'optional_bytes', lambda size, device: None)
    got, = torch.autograd.grad(module(xy), module.params, up)
    assert torch.equal(got, want)


def test_without_memory_for_optional_scratch(monkeypatch):
    """No room for the tiles' scratch or the handoff: the passes that need none run instead."""
    from odie_amd.encoding import GridEncoding
    monkeypatch.setattr(_lib, 'optional_bytes', lambda size, device: None)
    layout, n = _packed_layout(21, **TILE_PLANES), 2000
    xy = torch.from_numpy(synth.coordinates(21, n)).cuda()
    up = torch.from_numpy(synth.upstream(21, n, 22)).cuda().half()
    got = _packed_gradient(layout, xy, up, packed_owner=0).cpu().numpy()
    want = _without_tiles(layout, xy, up).cpu().numpy()       # the same kernel: its adds' order differs
    assert np.allclose(got, want, rtol=1e-5, atol=1e-6 * np.abs(want).max())
    module = GridEncoding(dict(n_levels=16, n_features_per_level=2, log2_hashmap_size=16, base_resolution=16,
                               per_level_scale=1.38))
    xy = torch.from_numpy(synth.coordinates(32, 70001)).cuda()
    up = torch.from_numpy(synth.upstream(32, 70001, 32)).cuda().half()
    got, = torch.autograd.grad(module(xy), module.params, up)
    assert torch.equal(got, grid_backward(xy, up, module.levels, 2, expert_params=module.n_params))
