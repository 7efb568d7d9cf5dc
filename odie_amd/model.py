"""Packed xy planes: the on-demand representation's storage layout, its encode as a torch
autograd op on this library's kernels, and the model built on them.

Storage (the format of odie/model.py:37-118, which checkpoints and the native runtime read):
level l keeps only the closure of its selected cells -- every corner c, c+1, c+R, c+R+1 of a
selected cell, wrapped into the align8(R^2) node universe -- packed into a capacity of
`plane_node_caps[l]` rows of F_l features.  A level whose closure is its whole universe is
addressed directly; any other through a presence bitmap (64 nodes per uint64 word, LSB first)
and an int32 exclusive prefix count per word.  One int32 descriptor row per level, columns in
the order DESCRIPTOR_COLUMNS, tells the kernels where everything is.

Building a layout is host bookkeeping at initialization and at each plane activation; queries
run on the GPU (odie_packed_forward / odie_packed_backward).
"""
import numpy as np
import torch

from . import _lib

COORDINATE_VERSION = 'unit-endpoints-native-fmaf-half-cell-align8-modulo-v1'
LAYOUT_VERSION = 'packed-xy-only-native-closure-v1'
ADDRESSING_VERSION = 'node-bitmap64-exclusive-prefix32-v1'
INT32_MAX = 2 ** 31 - 1
DESCRIPTOR_COLUMNS = ('resolution', 'points', 'plane_offset', 'node_word_offset', 'bitmap_byte_offset', 'features',
                      'feature_offset', 'direct')
CORNERS = (0, 1)          # x offsets of a cell's corners; y offsets are the same rows of R nodes


def align8(value):
    return -(-int(value) // 8) * 8


def gate_coarse_levels(config):
    """K, the leading levels whose gate is fixed at one; it must equal coarse_levels and stay
    within the declared levels (odie/model.py:25-30)."""
    levels = int(config['n_levels'])
    coarse = int(config['coarse_levels'])
    k = int(config.get('gate_coarse_levels_K', coarse))
    if k != coarse or k < 0 or k > levels:
        raise ValueError('Gate K must agree with coarse_levels and remain within declared level count')
    return k


def plane_closure(support, resolution):
    """Sorted unique closure nodes (CPU int64 tensor) of a flat bool support of R^2 cells."""
    mask = np.asarray(torch.as_tensor(support).cpu().numpy(), dtype=bool)
    cells = np.flatnonzero(mask).astype(np.int64)
    steps = np.array([dx + dy * resolution for dy in CORNERS for dx in CORNERS], dtype=np.int64)
    corners = (cells[:, None] + steps[None, :]).reshape(-1) % align8(resolution * resolution)
    return torch.from_numpy(np.unique(corners))


def make_node_index(nodes, points):
    """(uint64 presence bitmap, int32 exclusive per-word prefix) of sorted unique nodes."""
    if not isinstance(points, int) or points <= 0 or points > INT32_MAX:
        raise ValueError('Native node universe must fit positive int32 addressing')
    if nodes.device.type != 'cpu' or nodes.dtype != torch.int64 or nodes.ndim != 1:
        raise ValueError('Nodes must be a flat CPU int64 tensor')
    values = nodes.numpy()
    if values.size and (values[0] < 0 or values[-1] >= points or bool((np.diff(values) <= 0).any())):
        raise ValueError('Nodes must be sorted, unique and inside the native universe')
    words = (points + 63) // 64
    present = np.zeros(words * 64, dtype=np.uint8)
    present[values] = 1
    packed = np.packbits(present.reshape(words, 64), axis=1, bitorder='little')
    bitmap = packed.view('<u8').reshape(words).copy()
    counts = present.reshape(words, 64).sum(1, dtype=np.int64)
    prefix = (np.cumsum(counts) - counts).astype(np.int32)
    return torch.from_numpy(bitmap.view(np.int64)).view(torch.uint64), torch.from_numpy(prefix)


def _cell_bitmap(support, points):
    """LSB-first visibility bits of the R^2 cells, padded to the node universe."""
    padded = np.zeros(points, dtype=np.uint8)
    padded[:support.numel()] = support.numpy()
    return torch.from_numpy(np.packbits(padded.reshape(-1, 8), axis=1, bitorder='little').reshape(-1))


def _check_request(config, supports, plane_dims, plane_node_caps):
    levels = int(config['n_levels'])
    lengths = {len(config['resolutions']), len(supports), len(plane_dims), len(plane_node_caps)}
    if lengths != {levels} or any(f not in (1, 2, 4) for f in plane_dims):
        raise ValueError('Require aligned level descriptors and F1/F2/F4 features')
    if config['representation'] != 'xy_planes':
        raise ValueError('XY-only representation is required')
    gate_coarse_levels(config)
    if (config['gate_topology'], config['gate_position']) != ('shared', 'feature'):
        raise ValueError('Preserve the shared feature gate')


class _Layout:
    """Running offsets and the per-level pieces of one layout, filled level by level."""

    def __init__(self, full_prefix):
        self.full_prefix = full_prefix
        self.rows, self.levels, self.supports = [], [], []
        self.words, self.prefixes, self.cells = [], [], []
        self.params = self.columns = self.word_count = self.cell_bytes = 0

    def add(self, level, resolution, support, dim, cap):
        if support.device.type != 'cpu' or support.dtype != torch.bool or tuple(support.shape) != (resolution ** 2,):
            raise ValueError('Support must be a flat CPU bool R^2 tensor')
        if level < self.full_prefix and not bool(support.all()):
            raise ValueError('Declared initial full-cover supports must remain full')
        support = support.clone()
        points = align8(resolution ** 2)
        nodes = plane_closure(support, resolution)
        if cap % 8 or not nodes.numel() <= cap <= points:
            raise ValueError('Aligned node capacity must contain the complete interpolation closure')
        if points > INT32_MAX or self.params + cap * dim > INT32_MAX:
            raise ValueError('Native points and packed offsets must fit int32 addressing')
        direct = nodes.numel() == points
        word_offset, words = -1, 0
        if not direct:
            bitmap, prefix = make_node_index(nodes, points)
            word_offset, words = self.word_count, bitmap.numel()
            self.words.append(bitmap)
            self.prefixes.append(prefix)
            self.word_count += words
        cells = _cell_bitmap(support, points)
        self.rows.append((resolution, points, self.params, word_offset, self.cell_bytes, dim, self.columns,
                          int(direct)))
        # the per-level record the reference writes into its storage statistics
        self.levels.append(dict(level=level, resolution=resolution, plane_dim=dim,
                                allowed_cells=int(support.sum()), plane_retained_nodes=nodes.numel(),
                                plane_node_capacity=cap, plane_unused_slots=cap - nodes.numel(),
                                native_plane_points=points, plane_offset=self.params,
                                feature_offset=self.columns, nodes=nodes, node_index_words=words,
                                direct_node_access=direct))
        self.cells.append(cells)
        self.supports.append(support)
        self.params += cap * dim
        self.columns += dim
        self.cell_bytes += cells.numel()

    def result(self):
        def joined(parts, dtype):
            return torch.cat(parts) if parts else torch.empty(0, dtype=dtype)
        return {'descriptors': torch.tensor(self.rows, dtype=torch.int32),
                'node_bitmap': joined(self.words, torch.uint64), 'node_prefix': joined(self.prefixes, torch.int32),
                'bitmap': torch.cat(self.cells), 'levels': self.levels, 'supports': self.supports,
                'params': self.params, 'input_width': self.columns}


def make_layout(config, supports, plane_dims, plane_node_caps):
    """Descriptors, addressing buffers and per-level records of the packed planes
    (odie/model.py:64-118)."""
    _check_request(config, supports, plane_dims, plane_node_caps)
    layout = _Layout(int(config['initial_active_prefix']))
    for level, args in enumerate(zip(config['resolutions'], supports, plane_dims, plane_node_caps)):
        layout.add(level, *args)
    return layout.result()


def _nonempty(tensor):
    """A device buffer is never empty: the kernels take a pointer even when a level needs none."""
    return tensor if tensor.numel() else torch.zeros(1, dtype=tensor.dtype, device=tensor.device)


def packed_forward(coordinates, grid, descriptors, node_bitmap, node_prefix, bitmap, width):
    """(features fp16 [N, width], visibility bool [N, L]) -- odie/packed_kernels.cu:107-125."""
    if coordinates.dtype != torch.float32 or coordinates.ndim != 2 or coordinates.shape[1] != 2:
        raise ValueError('coordinates must be CUDA contiguous FP32 Nx2')
    if grid.dtype != torch.float32 or grid.ndim != 1:
        raise ValueError('grid must be flat CUDA FP32')
    coordinates, grid = coordinates.contiguous(), grid.contiguous()
    n, levels = coordinates.shape[0], descriptors.shape[0]
    features = torch.empty((n, width), dtype=torch.float16, device=coordinates.device)
    visibility = torch.empty((n, levels), dtype=torch.bool, device=coordinates.device)
    _lib.check(_lib.library().odie_packed_forward(
        coordinates.data_ptr(), n, grid.data_ptr(), grid.numel(), descriptors.data_ptr(), levels,
        _nonempty(node_bitmap).data_ptr(), _nonempty(node_prefix).data_ptr(), bitmap.data_ptr(), width,
        features.data_ptr(), visibility.data_ptr(), _lib.stream_of(coordinates)))
    return features, visibility


def packed_backward(coordinates, upstream, descriptors, node_bitmap, node_prefix, bitmap, parameter_count):
    """fp32 gradient [parameter_count] -- odie/packed_kernels.cu:127-145."""
    if upstream.dtype != torch.float16 or upstream.ndim != 2 or upstream.shape[0] != coordinates.shape[0]:
        raise ValueError('upstream must be CUDA contiguous FP16 NxF')
    upstream = upstream.contiguous()
    gradient = torch.empty(parameter_count, dtype=torch.float32, device=coordinates.device)
    lib = _lib.library()
    need = max(int(lib.odie_packed_backward_workspace(coordinates.shape[0], upstream.shape[1])), 0)
    scratch = _lib.optional_bytes(need, coordinates.device)   # without it: the pass that needs none
    need = need if scratch is not None else 0
    _lib.check(lib.odie_packed_backward_scratch(
        coordinates.data_ptr(), coordinates.shape[0], upstream.data_ptr(), upstream.shape[1],
        descriptors.data_ptr(), descriptors.shape[0], _nonempty(node_bitmap).data_ptr(),
        _nonempty(node_prefix).data_ptr(), bitmap.data_ptr(), gradient.data_ptr(), parameter_count,
        _lib.ptr(scratch), need, _lib.stream_of(coordinates)))
    return gradient


class PackedQuery(torch.autograd.Function):
    """Same contract as odie/model.py:137-151: features and visibility forward, the fp32 grid
    gradient backward."""

    @staticmethod
    def forward(ctx, coordinates, grid, descriptors, node_bitmap, node_prefix, bitmap, width):
        features, visible = packed_forward(coordinates, grid, descriptors, node_bitmap, node_prefix, bitmap, width)
        ctx.save_for_backward(coordinates, descriptors, node_bitmap, node_prefix, bitmap)
        ctx.param_count = grid.numel()
        ctx.mark_non_differentiable(visible)
        ctx.set_materialize_grads(False)   # no zeros [N, L] for the visibility's absent gradient
        return features, visible

    @staticmethod
    def backward(ctx, feature_gradient, visibility_gradient):
        coordinates, descriptors, node_bitmap, node_prefix, bitmap = ctx.saved_tensors
        if feature_gradient is None:
            zeros = torch.zeros(ctx.param_count, dtype=torch.float32, device=coordinates.device)
            return None, zeros, None, None, None, None, None
        gradient = packed_backward(coordinates, feature_gradient.contiguous(), descriptors, node_bitmap,
                                   node_prefix, bitmap, ctx.param_count)
        return None, gradient, None, None, None, None, None


def plane_seed(seed, level):
    """Seed of level l's feature draws (odie/model.py:211-212)."""
    return (seed + 1000003 * (level + 1) + 104729 * 3) % (2 ** 31)


def _check_query(coordinates):
    if coordinates.dtype != torch.float32 or coordinates.ndim != 2 or coordinates.shape[1] != 2 \
            or coordinates.requires_grad:
        raise ValueError('Coordinates must be FP32 Nx2, without coordinate gradients')


class PackedPlanes:
    """The packed planes of PackedXYPlanes without its heads: fp32 master `grid` in packed
    storage, the layout's addressing buffers on the device, the active prefix, and the
    activation of the next plane's support (odie/model.py:154-262).

    Plane values are inputs of the path: a plane's native nodes draw N(0, feature_init_std) from
    the counter PRNG of odie_amd.synth under the level's seed, max(2, F) values per node of
    which the first F are kept, so a plane is initialized exactly once and identically on every
    machine.
    """

    def __init__(self, config, supports, plane_dims, plane_node_caps, device='cuda'):
        self.config = dict(config)
        self.plane_dims, self.plane_node_caps = list(plane_dims), list(plane_node_caps)
        self.n_levels = int(self.config['n_levels'])
        self.device = torch.device(device)
        self._install(make_layout(self.config, supports, plane_dims, plane_node_caps))
        self.input_width = self.layout['input_width']
        self.grid = torch.zeros(self.layout['params'], dtype=torch.float32, device=self.device)
        self.initialized_planes = [False] * self.n_levels
        for level, item in enumerate(self.layout['levels']):
            if item['nodes'].numel():
                self._initialize_plane(level)
        self.active_prefix = int(self.config.get('initial_active_prefix', self.n_levels))

    def _install(self, layout):
        self.layout, self.supports = layout, layout['supports']
        for name in ('descriptors', 'node_bitmap', 'node_prefix', 'bitmap'):
            setattr(self, name, _nonempty(layout[name]).to(self.device))

    @torch.no_grad()
    def _initialize_plane(self, level):
        from . import synth
        if self.initialized_planes[level]:
            raise RuntimeError('Each plane must be initialized exactly once')
        item = self.layout['levels'][level]
        draws = max(2, item['plane_dim'])
        values = synth.normal(plane_seed(int(self.config['seed']), level), 'plane',
                              item['native_plane_points'] * draws).reshape(-1, draws)
        chosen = values[item['nodes'].numpy(), :item['plane_dim']] * float(self.config['feature_init_std'])
        start = item['plane_offset']
        flat = torch.from_numpy(chosen.astype(np.float32).reshape(-1))
        self.grid[start:start + flat.numel()].copy_(flat)
        self.initialized_planes[level] = True

    @torch.no_grad()
    def activate_support(self, level, support):
        """Open the next plane with `support`, keeping the packed storage and every offset
        (odie/model.py:226-257); returns the reference's activation record."""
        if level != self.active_prefix or not 2 <= level < self.n_levels:
            raise ValueError('Select the next unopened plane before advancing the prefix')
        if self.initialized_planes[level] or bool(self.supports[level].any()):
            raise RuntimeError('An opened support cannot be replaced or initialized again')
        resolution = self.config['resolutions'][level]
        if support.device.type != 'cpu' or support.dtype != torch.bool or support.shape != (resolution ** 2,):
            raise ValueError('New support must be a flat CPU bool R^2 tensor')
        selected = plane_closure(support, resolution).numel()
        if not 0 < selected <= self.plane_node_caps[level]:
            raise ValueError('New support requires a nonempty complete closure within its cap')
        storage = self.grid.data_ptr()
        supports = [s if l != level else support.clone() for l, s in enumerate(self.supports)]
        self._install(make_layout(self.config, supports, self.plane_dims, self.plane_node_caps))
        self._initialize_plane(level)
        if self.grid.data_ptr() != storage:
            raise AssertionError('Packed storage changed during plane activation')
        points = self.layout['levels'][level]['native_plane_points']
        return {'level': level, 'initialized_once': True, 'grid_storage_unchanged': True,
                'original_dense_f2_seed': plane_seed(int(self.config['seed']), level),
                'native_dense_draw_shape': [points, max(2, self.plane_dims[level])], 'selected_nodes': selected}

    def set_active_prefix(self, prefix):
        if not isinstance(prefix, int) or not 2 <= prefix <= self.n_levels:
            raise ValueError('Active prefix must be an integer between 2 and declared level count')
        self.active_prefix = prefix

    def query_features(self, coordinates):
        """(features fp16 [N, input_width], visibility bool [N, L]) through PackedQuery."""
        _check_query(coordinates)
        return PackedQuery.apply(coordinates.contiguous(), self.grid, self.descriptors, self.node_bitmap,
                                 self.node_prefix, self.bitmap, self.input_width)


# seeds of the two heads (odie/model.py:191-193)
GATE_SEED, DECODER_SEED = 2000003, 4000037


def make_heads(config, plane_dims, router_enabled, coarse, device):
    """(gate or None, decoder) for rows of the levels' features padded to align16 columns, seeded
    as the reference seeds its heads."""
    from .decoder import Decoder
    from .gate import Gate
    width = (sum(plane_dims) + 15) // 16 * 16
    if width > 80:
        raise ValueError('the heads take at most 80 feature columns')
    seed = int(config['seed'])
    gate = (Gate(seed=(seed + GATE_SEED) % 2 ** 31, coarse=coarse,
                 activation=config.get('router_output_activation', 'sigmoid'), device=device, features=plane_dims)
            if router_enabled else None)
    return gate, Decoder(seed=(seed + DECODER_SEED) % 2 ** 31, device=device, width=width)


def heads_match(config, gate, decoder):
    """The head sizes equal the configuration's gate_parameters / decoder_parameters."""
    gate_size = gate.params.numel() if gate is not None else 0
    return gate_size == config['gate_parameters'] and decoder.params.numel() == config['decoder_parameters']


def decode_rows(raw, gate, decoder, visible=None, columns=None):
    """The heads on raw features [N, sum F] fp16: columns padded with ones to the decoder's
    width, gated per level when there is a gate, decoded; RGB fp32 [N, 3].  Rows already of the
    decoder's width are read as they are; of those, the columns past `columns` count as ones."""
    if raw.ndim != 2:
        raise ValueError('decoder input must be CUDA fp16 [n, %d]' % decoder.width)
    if raw.shape[1] != decoder.width or raw.dtype != torch.float16 or raw.data_ptr() % 16:
        rows = torch.ones((raw.shape[0], decoder.width), dtype=torch.float16, device=raw.device)
        rows[:, :raw.shape[1]] = raw
        raw = rows
    if raw.dtype != torch.float16 or not raw.is_cuda or (gate is not None and gate.width != decoder.width):
        raise ValueError('decoder input must be CUDA fp16 [n, %d]' % decoder.width)
    raw = raw.contiguous()
    decoder.sync_weights()
    if gate is not None:
        gate.sync_weights()
    rgb = torch.empty((raw.shape[0], 3), dtype=torch.float32, device=raw.device)
    _lib.check(_lib.library().odie_heads_forward(
        raw.data_ptr(), raw.shape[0], decoder.width, decoder.width if columns is None else columns,
        gate.levels if gate is not None else 0, gate._table if gate is not None else None,
        _lib.ptr(gate.half) if gate is not None else None, _lib.ptr(visible),
        gate.coarse if gate is not None else 0, int(gate.softplus) if gate is not None else 0,
        decoder.half.data_ptr(), rgb.data_ptr(), _lib.stream_of(raw)))
    return rgb


def head_storage(grid_params, gate, decoder):
    """The parameter and byte counts both models report (odie/model.py:281-314,
    odie/hash_grid.py:64-80): fp16 payload, fp32 masters and Adam moments of grid and heads."""
    gate_params = gate.params.numel() if gate is not None else 0
    decoder_params = decoder.params.numel()
    total = grid_params + gate_params + decoder_params
    return {'actual_params': total, 'grid_params': grid_params, 'head_params': gate_params + decoder_params,
            'gate_params': gate_params, 'decoder_params': decoder_params}, \
        {'fp16_parameter_payload_bytes': 2 * total, 'fp32_master_bytes': 4 * total, 'adam_moment_bytes': 8 * total}


class PackedXYPlanes(PackedPlanes):
    """The on-demand model (odie/model.py:154-314): packed planes of F1/F2/F4 levels (2..20 of
    them, at most 80 feature columns) with the router gate and the decoder (Gate / Decoder, fp32
    masters in `params`).  forward(coordinates) is the reference's evaluation path
    (odie/model.py:266-279) -- query, zero the levels past the active prefix, gate by level with
    visibility, decode, first 3 outputs as fp32 -- run without autograd; training goes through
    NativeOptimizer."""

    def __init__(self, config, supports, plane_dims, plane_node_caps, axis_mode='none', kernel_a=0.,
                 kernel_omega=1.5 * np.pi, device='cuda'):
        if axis_mode != 'none' or kernel_a != 0.:
            raise ValueError('No axis branches or non-linear interpolation kernel in this ablation')
        super().__init__(config, supports, plane_dims, plane_node_caps, device=device)
        self.router_enabled = bool(config.get('router_enabled', True))
        self.gate_coarse_levels_K = gate_coarse_levels(config)
        self.gate, self.decoder = make_heads(config, plane_dims, self.router_enabled, self.gate_coarse_levels_K,
                                             device)
        if not heads_match(config, self.gate, self.decoder):
            raise RuntimeError('Unexpected TCNN head allocation for the configured input width')
        self.feature_levels = torch.tensor([l for l, f in enumerate(plane_dims) for _ in range(f)],
                                           dtype=torch.int64, device=self.device)

    def forward(self, coordinates):
        with torch.no_grad():
            _check_query(coordinates)
            coordinates = coordinates.contiguous()
            n, width = coordinates.shape[0], self.decoder.width
            if self.input_width > width:
                raise ValueError('the planes have %d features, the decoder %d inputs' % (self.input_width, width))
            raw = torch.empty((n, width), dtype=torch.float16, device=coordinates.device)
            visible = torch.empty((n, self.n_levels), dtype=torch.uint8, device=coordinates.device)
            if self.grid.dtype != torch.float32 or self.grid.ndim != 1:
                raise ValueError('grid must be flat CUDA FP32')
            grid = self.grid.contiguous()
            _lib.check(_lib.library().odie_packed_forward_rows(
                coordinates.data_ptr(), n, grid.data_ptr(), grid.numel(), self.descriptors.data_ptr(), self.n_levels,
                self.node_bitmap.data_ptr(), self.node_prefix.data_ptr(), self.bitmap.data_ptr(), width,
                self.active_prefix, raw.data_ptr(), visible.data_ptr(), _lib.stream_of(coordinates)))
            return decode_rows(raw, self.gate, self.decoder, visible=visible)

    __call__ = forward

    def storage_stats(self):
        counts, bytes_ = head_storage(self.grid.numel(), self.gate, self.decoder)
        size = {name: getattr(self, name).numel() * getattr(self, name).element_size()
                for name in ('node_bitmap', 'node_prefix', 'bitmap', 'descriptors')}
        index = size['node_bitmap'] + size['node_prefix']
        flags = self.n_levels + 2 * self.input_width      # a bool per level, an fp16 per feature column
        lookup = 8 * self.input_width                      # the int64 feature -> level index
        stats = dict(counts, router_enabled=self.router_enabled, axis_params=0, plane_params=counts['grid_params'],
                     plane_caps=self.plane_node_caps, **bytes_,
                     full_gradient_bytes=4 * counts['actual_params'], index_bytes=index,
                     node_bitmap_bytes=size['node_bitmap'], node_prefix_bytes=size['node_prefix'],
                     bitmap_bytes=size['bitmap'], descriptor_bytes=size['descriptors'],
                     runtime_index_bytes=index + size['bitmap'] + size['descriptors'] + lookup + flags,
                     active_flag_bytes=flags, input_width=self.input_width,
                     native_input_padding=(self.input_width + 15) // 16 * 16, axis_mode='none',
                     active_layers_from_update1=int(self.config.get('initial_active_prefix', 2)),
                     active_prefix=self.active_prefix, gate_coarse_levels_K=self.gate_coarse_levels_K,
                     full_cover_coarse_layers=self.config.get('full_cover_coarse_layers', [0, 1]),
                     plane_dims=self.plane_dims, coordinate_version=COORDINATE_VERSION,
                     layout_version=LAYOUT_VERSION, addressing_version=ADDRESSING_VERSION,
                     query_cuda_launches=1, backward_cuda_launches=1,
                     forward_precision='P01 FP32 geometry and FP16 interpolation chain',
                     gradient_precision='FP16 feature gradient, FP32 interpolation weights and atomicAdd')
        stats['levels'] = [{key: value for key, value in item.items() if key != 'nodes'}
                           for item in self.layout['levels']]
        return stats


def build_model(config, supports, plane_dims, plane_node_caps, **kwargs):
    """The model of config['representation'] (odie/model.py:318-321)."""
    if config['representation'] == 'hash_grid':
        from .hash_grid import HashGrid
        return HashGrid(config, supports, plane_dims, plane_node_caps)
    return PackedXYPlanes(config, supports, plane_dims, plane_node_caps, **kwargs)
