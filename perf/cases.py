"""The measured work of the framework, through its public entry points.

A case is a dict of plain values whose "kind" names the path:

  encode  GridEncoding, forward and backward through autograd (the tcnn.Encoding replacement)
  query   PackedQuery, the on-demand planes' encode, forward and backward through autograd
  step    ExpertTrainer.step, the multi-expert training step (route, encode, heads, backward, Adam)
  native  NativeOptimizer.train_batch, the single-model training step (stratified draw, graph replay)
  live    PackedXYPlanes / HashGrid evaluated over the raster and scored per cell (the live selection's input)
  score   score_image and topk_tiles: the multi-expert reconstruction, its residual and the worst tiles
  select  select_device (exact greedy) or select_mean_rank: the support of the next plane

Inputs come from the seed alone.  exact() restates each path in plain torch at 64 bits from the
same inputs, with the points where the format itself fixes the precision (fp32 cell geometry,
fp16 copies of the weights, the loss scales) kept.
"""
import math

import torch

from odie_amd.config import grid_levels
from odie_amd.decoder import Decoder
from odie_amd.encoding import GridEncoding
from odie_amd.experts import ExpertGrid
from odie_amd.gate import Gate
from odie_amd.gpu_residual import DeviceScores
from odie_amd.hash_grid import HashGrid
from odie_amd.model import PackedPlanes, PackedXYPlanes, plane_closure
from odie_amd.native_backend import NativeModel, NativeOptimizer, make_native_optimizer
from odie_amd.reconstruction import score_image
from odie_amd.sampling import stratified_ids
from odie_amd.selection import select_device, select_mean_rank, topk_tiles
from odie_amd.trainer import ExpertTrainer

# The recorded DIV2K plane layouts of the reference's runs (resolutions, node caps, selected cells,
# levels covered in full), every level of 2 features but the finest, which has 1.
LAYOUTS = {
    'L8': ([8, 16, 32, 64, 128, 255, 510, 1020],
           [64, 256, 1024, 4096, 16384, 65032, 257712, 257712],
           [64, 256, 1024, 4096, 16384, 65025, 257237, 244883], 6),
    'L16': ([8, 11, 15, 21, 29, 40, 56, 77, 106, 147, 203, 280, 387, 534, 738, 1020],
            [64, 128, 232, 448, 848, 1600, 3136, 5936, 11240, 21616, 41216, 78400, 87936, 87936, 87936, 87968],
            [64, 121, 225, 441, 841, 1600, 3136, 5929, 11236, 21609, 41209, 78400, 87044, 84261, 74770, 63937], 12),
    'L20': ([8, 10, 13, 17, 22, 29, 37, 48, 62, 80, 103, 132, 171, 221, 285, 368, 474, 612, 790, 1020],
            [64, 104, 176, 296, 488, 848, 1376, 2304, 3848, 6400, 10616, 17424, 29248, 48848, 63560, 63560, 63560,
             63560, 63560, 63584],
            [64, 100, 169, 289, 484, 841, 1369, 2304, 3844, 6400, 10609, 17424, 29241, 48841, 62401, 62602, 59646,
             54137, 48024, 43053], 14),
}
SHAPE = (1536, 2040)     # height, width of a DIV2K image
BATCH = 65536            # ids of a native step


def listed():
    return [
        # a small batch on a small grid: what a user's unit-sized fit or a preview calls
        dict(name='encode_4k_f16', kind='encode', n=4096, levels=16, features=2, log2_table=14, half=True),
        # a ragged batch in full precision with 4 features per level
        dict(name='encode_300k_f32x4', kind='encode', n=300007, levels=12, features=4, log2_table=19, half=False),
        # one large grid, a large batch: the single-expert configuration
        dict(name='encode_4m_f16', kind='encode', n=1 << 22, levels=16, features=2, log2_table=19, half=True),
        # the on-demand planes' autograd op on a ragged batch (20 levels, 39 columns)
        dict(name='query_100k_L20', kind='query', n=100003, layout='L20'),
        # the 64-expert training step on ids uniform over the image
        dict(name='step_64x4m', kind='step', side_x=2048, side_y=1365, regions_x=8, regions_y=8, n=1 << 22,
             log2_table=16, stratified=False, router=False),
        # the many-expert step on a stratified batch, small tables
        dict(name='step_1024x16m', kind='step', side_x=16384, side_y=16384, regions_x=32, regions_y=32, n=1 << 24,
             log2_table=9, stratified=True, router=False),
        # a ragged batch over few experts with the router gate
        dict(name='step_15x300k_router', kind='step', side_x=2040, side_y=1536, regions_x=5, regions_y=3, n=300007,
             log2_table=14, stratified=False, router=True),
        # the native step on a recorded DIV2K layout
        dict(name='native_L16', kind='native', layout='L16', height=SHAPE[0], width=SHAPE[1], n=BATCH, router=True),
        # the native step on a large hash grid (the no-on-demand ablation)
        dict(name='native_hash21', kind='native', layout='hash', log2_table=21, height=4096, width=8192, n=BATCH,
             router=True),
        # full-image evaluation of the on-demand model with the per-cell residual of the next selection
        dict(name='live_L16', kind='live', layout='L16', height=SHAPE[0], width=SHAPE[1], resolution=1020, router=True),
        # gigapixel-style reconstruction, residual and tile choice
        dict(name='score_8k', kind='score', height=8192, width=8192, regions_x=32, regions_y=32, log2_table=9, tile=256,
             top=64),
        # the exact greedy for a fine plane under its recorded node cap
        dict(name='select_738', kind='select', resolution=738, cap=87936, policy='greedy'),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(['encode', 'query', 'step', 'native', 'live', 'score', 'select'])
    if kind == 'encode':
        features = rng.choice([1, 2, 2, 4])
        half = rng.random() < 0.6
        return dict(kind=kind, n=_log_int(rng, 4096, (1 << 22) if half and features == 2 else (1 << 19)),
                    levels=rng.randint(8, 20 if features < 4 else 16), features=features,
                    log2_table=rng.randint(14, 19), half=half)
    if kind == 'query':
        return dict(kind=kind, n=_log_int(rng, 4096, 1 << 20), layout=rng.choice(sorted(LAYOUTS)))
    if kind == 'step':
        regions_x, regions_y = rng.randint(2, 16), rng.randint(2, 16)
        stratified = rng.random() < 0.5
        return dict(kind=kind, side_x=rng.randint(1500, 4000), side_y=rng.randint(1000, 4000), regions_x=regions_x,
                    regions_y=regions_y, n=1 << rng.choice([16, 18, 20, 22]) if stratified
                    else _log_int(rng, 1 << 16, 1 << 22), log2_table=rng.randint(9, 14), stratified=stratified,
                    router=rng.random() < 0.4)
    if kind == 'native':
        layout = rng.choice(sorted(LAYOUTS) + ['hash'])
        case = dict(kind=kind, layout=layout, height=rng.randint(1000, 2040), width=rng.randint(1000, 2040),
                    n=rng.choice([BATCH, BATCH, _log_int(rng, 4096, BATCH)]), router=rng.random() < 0.7)
        return dict(case, log2_table=rng.randint(14, 21)) if layout == 'hash' else case
    if kind == 'live':
        return dict(kind=kind, layout=rng.choice(sorted(LAYOUTS) + ['hash']), height=_log_int(rng, 128, 1536),
                    width=_log_int(rng, 128, 2040), resolution=_log_int(rng, 8, 128), router=rng.random() < 0.7,
                    log2_table=rng.randint(14, 19))
    if kind == 'score':
        tile = rng.choice([64, 96, 128, 256])
        tiles = rng.randint(4, 24)
        side = tile * tiles - rng.randint(0, tile // 2)
        return dict(kind=kind, height=side, width=side, regions_x=rng.randint(2, 32), regions_y=rng.randint(2, 32),
                    log2_table=rng.randint(9, 12), tile=tile, top=rng.randint(1, tiles * tiles))
    resolution = _log_int(rng, 64, 738)
    cap = int(resolution * resolution * rng.uniform(0.05, 0.15)) // 8 * 8 + 8
    return dict(kind='select', resolution=resolution, cap=cap, policy=rng.choice(['greedy', 'greedy', 'rank']))


# ---------------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------------
def _generator(seed, device='cuda'):
    return torch.Generator(device=device).manual_seed(int(seed) % (1 << 62))


def _smooth(gen, channels, height, width, cells=48):
    """Smooth noise in [0, 1]: a photograph's low frequencies."""
    coarse = torch.rand((1, channels, cells, cells), device='cuda', generator=gen)
    return torch.nn.functional.interpolate(coarse, size=(height, width), mode='bilinear', align_corners=True)[0]


def _image(gen, height, width):
    image = torch.empty((height, width, 3), dtype=torch.uint8, device='cuda')
    coarse = torch.rand((1, 3, 64, 64), device='cuda', generator=gen)
    rows = max(1, (1 << 24) // width)
    for y in range(0, height, rows):      # by bands: a gigapixel image needs no fp32 copy of itself
        n = min(rows, height - y)
        down = torch.linspace(2 * y / height - 1, 2 * (y + n) / height - 1, n, device='cuda')
        across = torch.linspace(-1, 1, width, device='cuda')
        grid = torch.stack(torch.meshgrid(down, across, indexing='ij')[::-1], dim=-1)
        band = torch.nn.functional.grid_sample(coarse, grid[None], align_corners=True, padding_mode='border')[0]
        band = band * 0.8 + 0.2 * torch.rand(band.shape, device='cuda', generator=gen)
        image[y:y + n] = (band * 255).permute(1, 2, 0).to(torch.uint8)
    return image


def _encoding(levels, features, log2_table, base=16, scale=1.38):
    return dict(otype='HashGrid', n_levels=levels, n_features_per_level=features, log2_hashmap_size=log2_table,
                base_resolution=base, per_level_scale=scale)


def _table_entries(encoding):
    return grid_levels(encoding)[1]


def _dims(layout):
    return [2] * (len(LAYOUTS[layout][0]) - 1) + [1]


_SUPPORTS = {}


def _supports(layout):
    """The planes' selected cells: full where the layout says so, else the cells of the largest
    smooth residual whose closure fits the cap (residuals cluster, as an image's do)."""
    if layout not in _SUPPORTS:
        resolutions, caps, allowed, direct = LAYOUTS[layout]
        supports = []
        for level, (r, cap, count) in enumerate(zip(resolutions, caps, allowed)):
            support = torch.ones(r * r, dtype=torch.bool)
            if level >= direct:
                gen = torch.Generator().manual_seed(level)
                coarse = torch.rand((1, 1, 24, 24), generator=gen)
                residual = torch.nn.functional.interpolate(coarse, size=(r, r), mode='bilinear', align_corners=True)
                order = torch.argsort(residual.reshape(-1), descending=True, stable=True)
                while True:
                    support = torch.zeros(r * r, dtype=torch.bool)
                    support[order[:count]] = True
                    if plane_closure(support, r).numel() <= cap:
                        break
                    count = int(count * 0.97)
            supports.append(support)
        _SUPPORTS[layout] = supports
    return _SUPPORTS[layout]


def _align16(value):
    return (value + 15) // 16 * 16


def _model_config(layout, seed, router, log2_table=19):
    if layout == 'hash':
        encoding = _encoding(16, 2, log2_table, base=3, scale=1.84)
        rows, _ = grid_levels(encoding)
        dims, resolutions, direct = [2] * 16, [r.resolution for r in rows], 16
        extra = dict(representation='hash_grid', hash_encoding=encoding)
        caps = [r.size for r in rows]
    else:
        resolutions, caps, _, direct = LAYOUTS[layout]
        dims, extra = _dims(layout), dict(representation='xy_planes')
    levels, width = len(dims), _align16(sum(dims))
    config = dict(extra, resolutions=resolutions, n_levels=levels, coarse_levels=0, gate_coarse_levels_K=0,
                  gate_topology='shared', gate_position='feature', initial_active_prefix=direct,
                  seed=int(seed) % 100003, feature_init_std=1e-2, router_enabled=router,
                  router_output_activation='sigmoid',
                  target_storage='uint8', plane_feature_dimensions=dims, decoder_parameters=64 * width + 5120,
                  gate_parameters=32 * width + 32 * _align16(levels) if router else 0, grid_lr=1e-2, gate_lr=1e-3,
                  decoder_lr=1e-3)
    return config, dims, caps


class _Native:
    """A native optimizer with the stream it runs on, closed with the state.  Every state uses the
    one stream: the library's scratch is shared by the calls of a device."""
    stream = None

    def __init__(self, case, seed):
        if _Native.stream is None:
            _Native.stream = torch.cuda.Stream()
        gen = _generator(seed)
        config, dims, _ = _model_config(case['layout'], seed, case['router'], case.get('log2_table', 19))
        width = _align16(sum(dims))
        decoder = Decoder(seed=int(seed) % 1009, width=width)
        gate = Gate(seed=int(seed) % 1013, features=dims) if case['router'] else None
        self.shape = (case['height'], case['width'])
        self.image = _image(gen, *self.shape)
        self.uniforms = torch.rand((BATCH, 2), device='cuda', generator=gen)
        if case['layout'] == 'hash':
            grid = torch.randn(2 * _table_entries(config['hash_encoding']), device='cuda', generator=gen) * 0.1
            self.model = NativeModel(decoder, gate, grid=grid)
        else:
            planes = PackedPlanes(config, _supports(case['layout']), dims, LAYOUTS[case['layout']][1])
            planes.set_active_prefix(len(dims))
            planes.grid.copy_(torch.randn(planes.grid.shape, device='cuda', generator=gen) * 0.1)
            self.model = NativeModel(decoder, gate, planes=planes)
        torch.cuda.synchronize()
        with torch.cuda.stream(self.stream):
            if case['layout'] == 'hash':
                self.optimizer = NativeOptimizer(self.model, self.image, self.shape, config, [self.model.grid])
            else:
                self.optimizer, self.planes = make_native_optimizer(self.model, self.image, self.shape, config)
            self.optimizer.prepare_epoch()
        self.n = case['n']

    def __del__(self):
        if hasattr(self, 'optimizer'):
            self.optimizer.close()


def prepare(case, seed):
    kind, gen = case['kind'], _generator(seed)
    if kind == 'encode':
        encoding = _encoding(case['levels'], case['features'], case['log2_table'])
        module = GridEncoding(encoding, dtype=torch.float16 if case['half'] else torch.float32)
        with torch.no_grad():
            module.params.copy_(torch.randn(module.params.shape, device='cuda', generator=gen) * 0.1)
        xy = torch.rand((case['n'], 2), device='cuda', generator=gen)
        upstream = torch.randn((case['n'], module.n_output_dims), device='cuda', generator=gen).to(module.dtype)
        return dict(kind=kind, module=module, xy=xy, upstream=upstream)
    if kind == 'query':
        config, dims, caps = _model_config(case['layout'], seed, False)
        planes = PackedPlanes(config, _supports(case['layout']), dims, caps)
        planes.grid = (torch.randn(planes.grid.shape, device='cuda', generator=gen) * 0.1).requires_grad_()
        xy = torch.rand((case['n'], 2), device='cuda', generator=gen)
        upstream = torch.randn((case['n'], planes.input_width), device='cuda', generator=gen).half()
        return dict(kind=kind, planes=planes, xy=xy, upstream=upstream)
    if kind == 'step':
        image = _image(gen, case['side_y'], case['side_x'])
        trainer = ExpertTrainer(image, _encoding(16, 2, case['log2_table']), case['regions_x'], case['regions_y'],
                                case['n'], seed=int(seed) % 1009, router=case['router'])
        trainer.master.copy_(torch.randn(trainer.master.shape, device='cuda', generator=gen) * 0.1)
        trainer.grid.table.copy_(trainer.master)
        if case['stratified']:
            return dict(kind=kind, trainer=trainer, ids=None,
                        uniforms=torch.rand((case['n'], 2), device='cuda', generator=gen))
        ids = torch.randint(0, case['side_x'] * case['side_y'], (case['n'],), device='cuda', generator=gen)
        return dict(kind=kind, trainer=trainer, ids=ids, uniforms=None)
    if kind == 'native':
        return dict(kind=kind, native=_Native(case, seed))
    if kind == 'live':
        config, dims, caps = _model_config(case['layout'], seed, case['router'], case.get('log2_table', 19))
        if case['layout'] == 'hash':
            model = HashGrid(config, [], dims, caps)
            model.grid.copy_(torch.randn(model.grid.shape, device='cuda', generator=gen) * 0.1)
        else:
            model = PackedXYPlanes(config, _supports(case['layout']), dims, caps)
            model.set_active_prefix(len(dims))
            model.grid.copy_(torch.randn(model.grid.shape, device='cuda', generator=gen) * 0.1)
        height, width = case['height'], case['width']
        ids = torch.arange(height * width, device='cuda')
        xy = torch.stack([(ids % width).float() / (width - 1), (ids // width).float() / (height - 1)], dim=1)
        return dict(kind=kind, model=model, xy=xy.contiguous(), shape=(height, width), resolution=case['resolution'],
                    image=_image(gen, height, width).reshape(-1, 3))
    if kind == 'score':
        grid = ExpertGrid(_encoding(16, 2, case['log2_table']), case['regions_x'] * case['regions_y'])
        grid.table.copy_(torch.randn(grid.table.shape, device='cuda', generator=gen) * 0.1)
        image = _image(gen, case['height'], case['width']).reshape(-1, 3)
        return dict(kind=kind, grid=grid, decoder=Decoder(seed=int(seed) % 1009), image=image,
                    shape=(case['height'], case['width']), regions=(case['regions_x'], case['regions_y']),
                    tile=case['tile'], top=case['top'])
    r = case['resolution']
    scores = _smooth(gen, 1, r, r)[0].double() * torch.rand((r, r), device='cuda', generator=gen, dtype=torch.float64)
    return dict(kind='select', scores=scores.reshape(-1).contiguous(), resolution=r, cap=case['cap'],
                policy=case['policy'])


# ---------------------------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------------------------
LIVE_BATCH = 1 << 20     # pixels per evaluated batch


def run(state):
    kind = state['kind']
    if kind == 'encode':
        module = state['module']
        module.params.grad = None
        features = module(state['xy'])
        features.backward(state['upstream'])
        return dict(features=features.detach(), gradient=module.params.grad)
    if kind == 'query':
        planes = state['planes']
        planes.grid.grad = None
        features, visible = planes.query_features(state['xy'])
        features.backward(state['upstream'])
        return dict(features=features.detach(), visible=visible, gradient=planes.grid.grad)
    if kind == 'step':
        trainer = state['trainer']
        squares = trainer.step(state['ids'], uniforms=state['uniforms'])
        out = dict(squares=squares, perm=trainer.routing.perm, table=trainer.master, moment=trainer.grid_optimizer.m,
                   decoder=trainer.decoder.params, decoder_gradient=trainer.decoder.grad)
        if trainer.gate is not None:
            out.update(gate=trainer.gate.params, gate_gradient=trainer.gate.grad)
        return out
    if kind == 'native':
        native = state['native']
        with torch.cuda.stream(native.stream):
            ids = stratified_ids(native.uniforms, native.shape)[:native.n]
            loss = native.optimizer.train_batch(ids)
            model = native.model
            out = dict(loss=loss, squares=native.optimizer.squares[:native.n], grid=model.grid,
                       decoder=model.decoder.params)
            if model.gate is not None:
                out['gate'] = model.gate.params
            return out
    if kind == 'live':
        scores = DeviceScores(state['shape'], resolution=state['resolution'])
        pixels = state['image'].shape[0]
        rgb = []
        for begin in range(0, pixels, LIVE_BATCH):
            end = min(begin + LIVE_BATCH, pixels)
            rgb.append(state['model'](state['xy'][begin:end]))
            scores.add(rgb[-1], state['image'][begin:end], begin)
        return dict(rgb=rgb, totals=scores.totals)
    if kind == 'score':
        metrics, scores = score_image(state['grid'], state['decoder'].half, state['image'], state['shape'],
                                      state['regions'], tile=state['tile'])
        means = scores.totals / torch.from_numpy(scores.counts).cuda()
        return dict(mse=metrics['mse'], totals=scores.totals, tiles=topk_tiles(means, state['top']))
    if state['policy'] == 'rank':
        selected, record = select_mean_rank(state['scores'], state['resolution'], state['cap'])
        return dict(selected=selected, nodes=record['closure_nodes'])
    selected, nodes, iterations = select_device(state['scores'], state['resolution'], state['cap'])
    return dict(selected=selected, nodes=nodes, iterations=iterations)


# ---------------------------------------------------------------------------------------------
# What a pass cannot do without, and how far another correct implementation may be off
# ---------------------------------------------------------------------------------------------
def _head_flops(width, levels, router):
    decoder = 2 * (64 * width + 64 * 64 + 16 * 64)
    return decoder + (2 * (32 * width + 32 * _align16(levels)) if router else 0)


def _grid_size(case):
    """Parameters and features per level of a native or live case's grid."""
    _, dims, caps = _model_config(case['layout'], 0, False, case.get('log2_table', 19))
    return sum(c * d for c, d in zip(caps, dims)), dims


def work(case):
    kind = case['kind']
    if kind == 'encode':
        n, width, size = case['n'], case['levels'] * case['features'], 2 if case['half'] else 4
        params = _table_entries(_encoding(case['levels'], case['features'], case['log2_table'])) * case['features']
        touched = min(params, 4 * n * width)
        return dict(bytes=n * (8 + 2 * width * size) + touched * size + params * 4,
                    flops=n * (20 * case['levels'] + 16 * width))
    if kind == 'query':
        resolutions, caps, _, _ = LAYOUTS[case['layout']]
        dims = _dims(case['layout'])
        params, width, n = sum(c * d for c, d in zip(caps, dims)), sum(dims), case['n']
        return dict(bytes=n * (8 + 4 * width + len(dims)) + min(params, 4 * n * width) * 4 + params * 4,
                    flops=n * (20 * len(dims) + 16 * width))
    if kind == 'step':
        params = _table_entries(_encoding(16, 2, case['log2_table'])) * 2 * case['regions_x'] * case['regions_y']
        n = case['n']
        # ids, target bytes, squared errors and permutation; the optimizer reads master, moments and
        # age and writes them and the fp16 copy
        return dict(bytes=n * (8 + 3 + 4 + 4) + params * 34,
                    flops=n * (3 * _head_flops(32, 16, case['router']) + 20 * 16 + 16 * 32))
    if kind == 'native':
        params, dims = _grid_size(case)
        n, width = case['n'], sum(dims)
        touched = min(params, 4 * n * width)
        heads = _head_flops(_align16(width), len(dims), case['router'])
        return dict(bytes=BATCH * 8 + n * (8 + 3 + 4) + touched * 32,
                    flops=n * (3 * heads + 20 * len(dims) + 16 * width))
    if kind == 'live':
        n = case['height'] * case['width']
        params, dims = _grid_size(case)
        heads = _head_flops(_align16(sum(dims)), len(dims), case['router'])
        return dict(bytes=n * (8 + 12 + 3) + 4 * min(params, 4 * n * sum(dims)) + 8 * case['resolution'] ** 2,
                    flops=n * (heads + 20 * len(dims) + 8 * sum(dims)))
    if kind == 'score':
        n = case['height'] * case['width']
        params = _table_entries(_encoding(16, 2, case['log2_table'])) * 2 * case['regions_x'] * case['regions_y']
        return dict(bytes=3 * n + 2 * params, flops=n * (_head_flops(32, 16, False) + 20 * 16 + 8 * 32))
    n = case['resolution'] ** 2
    return dict(bytes=8 * n + 2 * n, flops=0)


def tolerance(case):
    """About four times the distance of each path from exact(): fp16 feature chains 4e-4, fp32 chains
    and sums 5e-8, RGB of the fp16 heads 7e-4 and cell totals of a few of its pixels 4e-5, fp16
    upstreams and the gradients formed from them 1e-2 (their small values lie among fp16's
    subnormals), which the first Adam steps carry into the weights' signs."""
    kind = case['kind']
    if kind == 'encode':
        return dict(rel=1.6e-3, max=0.03) if case['half'] else dict(rel=1e-6, max=1e-4)
    if kind == 'query':
        return dict(rel=1.6e-3, max=0.03)
    if kind in ('step', 'native'):
        return dict(rel=0.03, max=0.9)
    if kind == 'live':
        return dict(rel=3e-3, max=0.05)
    if kind == 'score':
        return dict(rel=1e-5, max=1e-4, differ=0.01)
    return 'exact'


# ---------------------------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------------------------
def _cells(xy, scale):
    """Cell and fraction of the fp32 geometry fma(scale, x, 0.5) the format defines."""
    position = (xy.double() * scale + 0.5).float().double()
    corner = position.floor()
    return corner.long(), position - corner


def _corner_weights(frac):
    fx, fy = frac[:, 0], frac[:, 1]
    return [(1 - fx) * (1 - fy), fx * (1 - fy), (1 - fx) * fy, fx * fy]


def _hash_corners(xy, level):
    cell, frac = _cells(xy, float(level.scale))
    index = []
    for dy in (0, 1):
        for dx in (0, 1):
            x, y = cell[:, 0] + dx, cell[:, 1] + dy
            raw = (x ^ ((y * 2654435761) & 0xffffffff)) if level.hashed else x + y * level.resolution
            index.append((raw & 0xffffffff) % level.size + level.offset)
    return index, _corner_weights(frac)


def _hash_encode(xy, table, levels, base=None):
    """Features of table [entries, F]; base: first entry of each coordinate's own table."""
    out = []
    for level in levels:
        index, weight = _hash_corners(xy, level)
        out.append(sum(w[:, None] * table[i if base is None else i + base].double() for i, w in zip(index, weight)))
    return torch.cat(out, dim=1)


def _hash_scatter(gradient, xy, upstream, levels, base=None):
    features = gradient.shape[1]
    for l, level in enumerate(levels):
        index, weight = _hash_corners(xy, level)
        u = upstream[:, l * features:(l + 1) * features].double()
        for i, w in zip(index, weight):
            gradient.index_add_(0, i if base is None else i + base, w[:, None] * u)


class _Planes:
    """The layout's planes as dense node tables, from the supports alone."""

    def __init__(self, layout, grid):
        resolutions, caps, _, _ = LAYOUTS[layout]
        self.resolutions, self.dims = resolutions, _dims(layout)
        self.nodes, self.points, self.starts, self.visible = [], [], [], []
        start = 0
        for r, cap, dim, support in zip(resolutions, caps, self.dims, _supports(layout)):
            points = (r * r + 7) // 8 * 8
            cells = torch.nonzero(support).flatten()
            self.nodes.append(torch.unique(torch.cat([cells, cells + 1, cells + r, cells + r + 1]) % points).cuda())
            self.points.append(points)
            self.starts.append(start)
            self.visible.append(support.cuda())
            start += cap * dim
        self.total = start
        self.tables = []
        for nodes, points, start, dim in zip(self.nodes, self.points, self.starts, self.dims):
            table = torch.zeros((points, dim), dtype=torch.float64, device='cuda')
            if grid is not None:
                table[nodes] = grid[start:start + nodes.numel() * dim].half().double().reshape(-1, dim)
            self.tables.append(table)

    def corners(self, xy, level):
        r = self.resolutions[level]
        cell, frac = _cells(xy, float(r - 1))
        cell = cell.clamp(0, r - 1)
        cell = cell[:, 0] + cell[:, 1] * r
        index = [(cell + dx + dy * r) % self.points[level] for dy in (0, 1) for dx in (0, 1)]
        return cell, index, _corner_weights(frac)

    def encode(self, xy):
        features, visible = [], []
        for level, table in enumerate(self.tables):
            cell, index, weight = self.corners(xy, level)
            seen = self.visible[level][cell]
            visible.append(seen)
            features.append(sum(w[:, None] * table[i] for i, w in zip(index, weight)) * seen[:, None])
        return torch.cat(features, dim=1), torch.stack(visible, dim=1)

    def gradient(self, xy, upstream):
        total, column = torch.zeros(self.total, dtype=torch.float64, device='cuda'), 0
        for level, dim in enumerate(self.dims):
            cell, index, weight = self.corners(xy, level)
            u = upstream[:, column:column + dim].double() * self.visible[level][cell][:, None]
            dense = torch.zeros((self.points[level], dim), dtype=torch.float64, device='cuda')
            for i, w in zip(index, weight):
                dense.index_add_(0, i, w[:, None] * u)
            nodes, start = self.nodes[level], self.starts[level]
            total[start:start + nodes.numel() * dim] = dense[nodes].reshape(-1)
            column += dim
        return total


def _weights(half, shapes):
    parts, at = [], 0
    for rows, cols in shapes:
        parts.append(half[at:at + rows * cols].double().reshape(rows, cols).requires_grad_())
        at += rows * cols
    return parts


def _heads(decoder, gate, dims):
    """The decoder's and the gate's fp16 weights in 64 bits, and the network on raw features."""
    width = decoder.width
    dw = _weights(decoder.params.half(), ((64, width), (64, 64), (16, 64)))
    gw = _weights(gate.params.half(), ((32, width), (_align16(len(dims)), 32))) if gate is not None else []
    level_of = torch.tensor([l for l, d in enumerate(dims) for _ in range(d)], device='cuda')

    def network(raw, visible=None):
        x = torch.nn.functional.pad(raw, (0, width - raw.shape[1]), value=1.0)
        if gw:
            s = torch.sigmoid(((x @ gw[0].T).relu() @ gw[1].T)[:, :len(dims)])
            if visible is not None:
                s = s * visible
            x = torch.cat([x[:, :len(level_of)] * s[:, level_of], x[:, len(level_of):]], dim=1)
        return ((x @ dw[0].T).relu() @ dw[1].T).relu() @ dw[2].T

    return network, dw, gw


def _flat(parts, scale):
    return torch.cat([p.grad.reshape(-1) for p in parts]) * scale


def _tile_starts(size, regions):
    return torch.tensor([(r * size + regions - 1) // regions for r in range(regions + 1)], device='cuda')


def _locate(ids, width, height, regions_x, regions_y):
    """Tile and local fp32 coordinate of pixel ids."""
    x, y = ids % width, torch.clamp(ids // width, max=height - 1)
    local = []
    tiles = []
    for p, size, regions in ((x, width, regions_x), (y, height, regions_y)):
        starts = _tile_starts(size, regions)
        tile = torch.searchsorted(starts, p, right=True) - 1
        extent = (starts[tile + 1] - starts[tile] - 1).float()
        local.append((p - starts[tile]).float() * (1.0 / extent))
        tiles.append(tile)
    return tiles[1] * regions_x + tiles[0], torch.stack(local, dim=1)


def _stratified(uniforms, height, width):
    side = int(round(math.sqrt(uniforms.shape[0])))
    j = torch.arange(uniforms.shape[0], device='cuda')
    place = lambda u, s, size: ((u / side + s.float() / side) * size).long().clamp(0, size - 1)
    return place(uniforms[:, 0], j % side, width) + place(uniforms[:, 1], j // side, height) * width


ROWS = 1 << 20           # rows handled at once


def _exact_step(state, case):
    trainer, n = state['trainer'], case['n']
    width, height, rx, ry = case['side_x'], case['side_y'], case['regions_x'], case['regions_y']
    ids = state['ids'] if state['ids'] is not None else _stratified(state['uniforms'], height, width)
    tile, local = _locate(ids, width, height, rx, ry)
    perm = torch.argsort(tile, stable=True)
    levels, entries = trainer.grid.levels, trainer.grid.expert_params // 2
    table = trainer.grid.table.reshape(-1, 2)
    network, dw, gw = _heads(trainer.decoder, trainer.gate, [2] * 16)
    rgb = trainer.rgb.reshape(-1, 3)
    squares, gradient = [], torch.zeros(table.shape, dtype=torch.float64, device='cuda')
    for at in range(0, n, ROWS):
        rows = perm[at:at + ROWS]
        xy, base = local[rows], tile[rows] * entries
        raw = _hash_encode(xy, table, levels, base).requires_grad_()
        with torch.enable_grad():
            d = network(raw)[:, :3] - rgb[ids[rows]].double() / 255
            (d.square().sum() / (3 * n)).backward()
        squares.append(d.detach().square().sum(dim=1) / 3)
        _hash_scatter(gradient, xy, raw.grad, levels, base)
    # the moment after one step is a tenth of the gradient; the updated weights have no value of their
    # own here: the first step of Adam moves each by the sign of its gradient
    out = dict(squares=torch.cat(squares), perm=None, table=None, moment=gradient.reshape(-1) * 0.1, decoder=None,
               decoder_gradient=_flat(dw, 16384.0))
    if trainer.gate is not None:
        out.update(gate=None, gate_gradient=_flat(gw, 16384.0))
    return out


def _exact_native(state, case):
    native, n = state['native'], case['n']
    model, (height, width) = native.model, native.shape
    ids = _stratified(native.uniforms, height, width)[:n]
    xy = torch.stack([(ids % width).float() * (1.0 / torch.tensor(width - 1.0)).item(),
                      (ids // width).float() * (1.0 / torch.tensor(height - 1.0)).item()], dim=1)
    if case['layout'] == 'hash':
        levels, _ = grid_levels(_model_config('hash', 0, False, case['log2_table'])[0]['hash_encoding'])
        raw, visible, dims = _hash_encode(xy, model.grid.half().reshape(-1, 2), levels), None, [2] * 16
    else:
        planes = _Planes(case['layout'], model.grid)
        (raw, visible), dims = planes.encode(xy), planes.dims
    network, _, _ = _heads(model.decoder, model.gate, dims)
    with torch.no_grad():
        d = network(raw, visible)[:, :3] - native.image.reshape(-1, 3)[ids].double() / 255
    squares = d.square().sum(dim=1) / 3
    out = dict(loss=squares.mean(), squares=squares, grid=None, decoder=None)   # Adam's first step: signs
    if case['router']:
        out['gate'] = None
    return out


def _exact_live(state, case):
    model, (height, width) = state['model'], state['shape']
    planes = _Planes(case['layout'], model.grid) if case['layout'] != 'hash' else None
    network, _, _ = _heads(model.decoder, model.gate, planes.dims if planes else [2] * 16)
    rgb, totals = [], torch.zeros(case['resolution'] ** 2, dtype=torch.float64, device='cuda')
    for begin in range(0, height * width, LIVE_BATCH):
        xy = state['xy'][begin:begin + LIVE_BATCH]
        if planes:
            raw, visible = planes.encode(xy)
        else:
            raw, visible = _hash_encode(xy, model.grid.half().reshape(-1, 2), model.levels), None
        with torch.no_grad():
            out = network(raw, visible)[:, :3]
        rgb.append(out)
        cell, _ = _cells(xy, float(case['resolution'] - 1))
        cell = cell.clamp(max=case['resolution'] - 1)
        term = (out - state['image'][begin:begin + LIVE_BATCH].double() / 255).square().sum(dim=1) / 3
        totals.index_add_(0, cell[:, 0] + cell[:, 1] * case['resolution'], term)
    return dict(rgb=rgb, totals=totals)


def _exact_score(state, case):
    height, width = state['shape']
    grid, side = state['grid'], -(-width // case['tile'])
    network, _, _ = _heads(state['decoder'], None, [2] * 16)
    totals = torch.zeros(side * side, dtype=torch.float64, device='cuda')
    for begin in range(0, height * width, ROWS):
        ids = torch.arange(begin, min(begin + ROWS, height * width), device='cuda')
        tile, local = _locate(ids, width, height, *state['regions'])
        raw = _hash_encode(local, grid.table.reshape(-1, 2), grid.levels, tile * (grid.expert_params // 2))
        with torch.no_grad():
            term = (network(raw)[:, :3] - state['image'][ids].double() / 255).square().sum(dim=1) / 3
        totals.index_add_(0, (ids // width // case['tile']) * side + ids % width // case['tile'], term)
    return dict(mse=totals.sum() / (height * width), totals=totals, tiles=None)


def exact(case, seed):
    kind = case['kind']
    if kind == 'select':
        return None
    state = prepare(case, seed)
    if kind == 'encode':
        module, xy, upstream = state['module'], state['xy'], state['upstream']
        table = module.params.detach().to(module.dtype).reshape(-1, module.features)
        gradient = torch.zeros(table.shape, dtype=torch.float64, device='cuda')
        features = []
        for at in range(0, case['n'], ROWS):
            features.append(_hash_encode(xy[at:at + ROWS], table, module.levels))
            _hash_scatter(gradient, xy[at:at + ROWS], upstream[at:at + ROWS], module.levels)
        return dict(features=torch.cat(features), gradient=gradient.reshape(-1))
    if kind == 'query':
        planes = _Planes(case['layout'], state['planes'].grid.detach())
        features, _ = planes.encode(state['xy'])
        return dict(features=features, visible=None, gradient=planes.gradient(state['xy'], state['upstream']))
    return dict(step=_exact_step, native=_exact_native, live=_exact_live, score=_exact_score)[kind](state, case)
