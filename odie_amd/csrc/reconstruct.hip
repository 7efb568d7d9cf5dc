// Fused reconstruction of an image through the multi-expert hash-grid model: for every pixel
// of a raster range, its expert tile and tile coordinate (the router's convention), the 16-level
// fp16 encode from that expert's table and the decoder MLP, in one kernel, so the features never
// reach memory.  The streamed full-image inference the residual pass scores
// (odie/evaluation.py:12-36, odie/gpu_residual.py:130-179: prediction = model(coordinates(ids))
// for ids in raster order).
//
// One wave per tile of 32 consecutive pixels.  Lane (g, s) encodes pixel s's levels
// 8*kt + 4*g + j (kt = 0, 1; j = 0..3): exactly the features 16*kt + 8*g + e that the decoder's
// first MFMA takes from that lane as its B operand, so the encode feeds the MLP in registers.
// Every value is computed with the arithmetic of odie_grid_forward (fp16 table, fp16 FMA chain,
// half2_level) and odie_mlp_forward (forward_tile): the same bits as those two entry points on
// the routed coordinates.
#include "grid.h"
#include "mlp.h"
#include "residual.h"
#include "tiles.h"
#include "../../include/odie_amd.h"

namespace odie {
namespace {

constexpr int kLevels = 16;
constexpr int kReconBlock = kMlpBlock;
constexpr int kReconWaves = kReconBlock / 64;

struct ReconArgs {
    int64_t begin;
    int64_t n;
    uint32_t width;
    Divisor by_width;      // id / width with one multiply-high
    uint32_t height;
    int regions_x;
    int regions_y;
    int experts;
    const int32_t* slots;      // table slot of each tile, < 0: no expert (null: slot = tile)
    const uint32_t* table;     // fp16 pairs
    int64_t expert_pairs;      // pairs per expert
    const uint16_t* weights;
    float* prediction;         // [n][3] or null
    uint16_t* features;        // [n][32] or null
    uint16_t* output;          // [n][16] or null
    uint32_t hashed_steps;     // bit 4*kt + j: both levels of that step are hashed (FAST)
    DevLevel level[kLevels];
};

// A level as the fast encode reads it: row term y * factor, then x + term (dense) or x ^ term
// (hashed), reduced into [0, size).
struct FastLevel {
    float scale;
    uint32_t factor;    // dense: resolution; hashed: the 24 bits of the prime that the mask keeps
    uint32_t size;
    uint32_t mask;      // size - 1 for power-of-two sizes, else all ones
    uint32_t hash_mask; // all ones when hashed, else 0
    uint32_t bytes;     // of the table before the level
    uint32_t unused[2];
};

// Per-block copies of the decoder's forward weights, the tile bounds and the level descriptors
// (read from LDS, the descriptors stay out of the scalar registers the unrolled levels would
// otherwise spill).
__device__ inline void stage_model(const ReconArgs& a, const TileBounds& bounds, _Float16* w, TileBounds& tb,
                                   DevLevel* levels, FastLevel* fast) {
    stage_forward_weights<2>(a.weights, w);
    constexpr int kLevelWords = kLevels * static_cast<int>(sizeof(DevLevel) / 4);
    static_assert(kLevelWords <= kReconBlock, "one thread per descriptor word");
    if (static_cast<int>(threadIdx.x) < kLevelWords)
        reinterpret_cast<uint32_t*>(levels)[threadIdx.x] = reinterpret_cast<const uint32_t*>(a.level)[threadIdx.x];
    if (static_cast<int>(threadIdx.x) < kLevels) {
        const DevLevel lv = a.level[threadIdx.x];
        fast[threadIdx.x] = FastLevel{lv.scale, lv.hashed ? lv.prime : lv.res, lv.size, lv.mask ? lv.mask : ~0u,
                                      lv.hashed ? ~0u : 0u, lv.offset * 4u, {0u, 0u}};
    }
    for (int j = threadIdx.x; j <= kMaxTiles; j += kReconBlock) {
        tb.x0[j] = bounds.x0[j];
        tb.y0[j] = bounds.y0[j];
        if (j < kMaxTiles) {
            tb.rx[j] = bounds.rx[j];
            tb.ry[j] = bounds.ry[j];
        }
    }
    if (threadIdx.x == 0) {
        tb.sx = bounds.sx;
        tb.sy = bounds.sy;
    }
    __syncthreads();
}

// The tile of the pixel a lane last located: neighbouring pixels mostly share it, and the two
// divisions' worth of exact products that tile_of takes are then left out.
struct TileCache {
    int32_t x_lo = 0, x_hi = 0, y_lo = 0, y_hi = 0;   // its pixels: x_lo <= x < x_hi, y_lo <= y < y_hi
    float rx = 0.0f, ry = 0.0f;
    int slot = -1;
    __device__ void locate(const ReconArgs& a, const TileBounds& tb, uint32_t x, uint32_t y) {
        const int xi = static_cast<int>(x), yi = static_cast<int>(y);
        if (xi >= x_lo && xi < x_hi && yi >= y_lo && yi < y_hi) return;
        const int tx = tile_of(a.regions_x, a.width, tb.sx, x), ty = tile_of(a.regions_y, a.height, tb.sy, y);
        x_lo = tb.x0[tx];
        x_hi = tb.x0[tx + 1];
        y_lo = tb.y0[ty];
        y_hi = tb.y0[ty + 1];
        rx = tb.rx[tx];
        ry = tb.ry[ty];
        const int t = ty * a.regions_x + tx;
        slot = a.slots ? a.slots[t] : t;
        if (slot >= a.experts) slot = -1;
    }
};

// The fast encode of lane (g, s)'s eight levels (FAST: model_args' fast_levels holds): the same
// arithmetic on the same values as grid_corners and half2_level, in fewer instructions.  The
// scoring kernels are bound by VALU issue (682 vector instructions per 32 pixels before, of them
// about 70 per level), so: the tile is looked up only when the pixel leaves it; the row term is one
// 24-bit product for dense and hashed levels alike; steps whose two levels (one per lane group)
// are both hashed take xor and mask alone, the others a branch-free mixture; coordinates are >= 0, so
// the conversion truncates to the cell and v_fract is the fraction; addresses are 32-bit offsets
// from the table; and the gathers are
// issued before the first is used.  493 vector instructions per 32 pixels with the residual's quotients
// by constants: 8192^2 pixels 3.0 -> 2.5 ms a pass (scoring kernel 2.75 -> 2.2).
__device__ inline void encode_fast(const ReconArgs& a, const FastLevel* levels, const TileCache& tile, uint32_t x,
                                   uint32_t y, bool real, int g, uint32_t pairs[2][4]) {
    const float u = static_cast<float>(static_cast<int>(x) - tile.x_lo) * tile.rx;
    const float v = static_cast<float>(static_cast<int>(y) - tile.y_lo) * tile.ry;
    const uint32_t base = real ? static_cast<uint32_t>(tile.slot) * static_cast<uint32_t>(a.expert_pairs * 4) : 0u;
    uint32_t entry[8][4];
    float fx[8], fy[8];
#pragma unroll
    for (int step = 0; step < 8; ++step) {
        const FastLevel lv = levels[8 * (step / 4) + 4 * g + step % 4];
        const float px = __builtin_fmaf(lv.scale, u, 0.5f), py = __builtin_fmaf(lv.scale, v, 0.5f);
        const uint32_t gx = static_cast<uint32_t>(px), gy = static_cast<uint32_t>(py);
        fx[step] = __builtin_amdgcn_fractf(px);
        fy[step] = __builtin_amdgcn_fractf(py);
        const uint32_t t0 = __umul24(gy, lv.factor), t1 = t0 + lv.factor;
        uint32_t idx[4];
        if ((a.hashed_steps >> step) & 1u) {
            idx[0] = (gx ^ t0) & lv.mask;
            idx[1] = ((gx + 1u) ^ t0) & lv.mask;
            idx[2] = (gx ^ t1) & lv.mask;
            idx[3] = ((gx + 1u) ^ t1) & lv.mask;
        } else {
            // x ^ t = x + t - 2 (x & t); a dense index is below 2 size, so the smaller of idx and
            // idx - size (unsigned) is the reduced one
            const uint32_t h0 = t0 & lv.hash_mask, h1 = t1 & lv.hash_mask;
            idx[0] = gx + t0 - 2u * (gx & h0);
            idx[1] = gx + 1u + t0 - 2u * ((gx + 1u) & h0);
            idx[2] = gx + t1 - 2u * (gx & h1);
            idx[3] = gx + 1u + t1 - 2u * ((gx + 1u) & h1);
#pragma unroll
            for (int k = 0; k < 4; ++k) idx[k] = min(idx[k], idx[k] - lv.size) & lv.mask;
        }
        const uint32_t at = base + lv.bytes;
#pragma unroll
        for (int k = 0; k < 4; ++k)
            entry[step][k] = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(a.table) + (at + 4u * idx[k]));
    }
#pragma unroll
    for (int step = 0; step < 8; ++step) {
        const float gx = 1.0f - fx[step], gy = 1.0f - fy[step];
        const float wk[4] = {gx * gy, fx[step] * gy, gx * fy[step], fx[step] * fy[step]};
        pairs[step / 4][step % 4] = real ? half2_level(entry[step], wk) : 0u;
    }
}

__device__ inline void decode(const _Float16* w, int g, int s, const uint32_t pairs[2][4], half8& out) {
    half8 xb[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
        xb[kt] = __builtin_bit_cast(half8, u32x4{pairs[kt][0], pairs[kt][1], pairs[kt][2], pairs[kt][3]});
    half8 h1[4], h2[4];
    f32x16 acc3;
    forward_tile<2>(w, g, s, xb, h1, h2, acc3);
    out = round8(acc3, 0);
}

// The wave's 32 pixels (pixel s of lane (g, s) is `id`, `valid` when it is real): the encode of
// lane (g, s)'s eight levels (pairs) and the decoder output rows of lane group g (out).
template <bool FAST>
__device__ inline void predict(const ReconArgs& a, const TileBounds& tb, const DevLevel* levels, const FastLevel* fast,
                               const _Float16* w, TileCache& tile, uint32_t x, uint32_t y, bool valid, int g, int s,
                               uint32_t pairs[2][4], half8& out) {
    tile.locate(a, tb, x, y);
    const bool real = valid && tile.slot >= 0;
    if constexpr (FAST) {
        encode_fast(a, fast, tile, x, y, real, g, pairs);
    } else {
        const float u = static_cast<float>(x - static_cast<uint32_t>(tile.x_lo)) * tile.rx;
        const float v = static_cast<float>(y - static_cast<uint32_t>(tile.y_lo)) * tile.ry;
        const uint32_t* table = a.table + (real ? static_cast<int64_t>(tile.slot) * a.expert_pairs : 0);
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                // lane group g encodes level 8kt + 4g + j
                const DevLevel lv = levels[8 * kt + 4 * g + j];
                uint32_t idx[4];
                float wk[4];
                grid_corners(lv, u, v, idx, wk);
                uint32_t e[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) e[k] = real ? table[lv.offset + idx[k]] : 0u;
                pairs[kt][j] = real ? half2_level(e, wk) : 0u;
            }
        }
    }
    decode(w, g, s, pairs, out);
}

// Output rows 0..2 (the RGB prediction) are elements 0..2 of lane group 0.
__device__ inline void rgb_of(const half8& out, float& r, float& gr, float& b) {
    const u32x4 bits = __builtin_bit_cast(u32x4, out);   // element 2i in the low half of dword i
    r = __half2float(bits_to_half(static_cast<uint16_t>(bits.x & 0xffffu)));
    gr = __half2float(bits_to_half(static_cast<uint16_t>(bits.x >> 16)));
    b = __half2float(bits_to_half(static_cast<uint16_t>(bits.y & 0xffffu)));
}

template <bool FAST> __global__ __launch_bounds__(kReconBlock) void reconstruct_kernel(ReconArgs a, TileBounds bounds) {
    __shared__ _Float16 w[kForwardHalfs];
    __shared__ TileBounds tb;
    __shared__ DevLevel levels[kLevels];
    __shared__ __attribute__((aligned(16))) FastLevel fast[kLevels];
    stage_model(a, bounds, w, tb, levels, fast);
    TileCache tile;
    const int lane = threadIdx.x % 64, g = lane / 32, s = lane % 32;
    const int64_t tiles = (a.n + 31) / 32;
    const int64_t waves = static_cast<int64_t>(gridDim.x) * kReconWaves;
    for (int64_t chunk = static_cast<int64_t>(blockIdx.x) * kReconWaves + threadIdx.x / 64; chunk < tiles;
         chunk += waves) {
        const int64_t row = chunk * 32 + s;
        const bool valid = row < a.n;
        uint32_t pairs[2][4];
        half8 out;
        const uint32_t id = static_cast<uint32_t>(a.begin + (valid ? row : 0));
        uint32_t y = divide(id, a.by_width);
        const uint32_t x = id - y * a.width;
        if (y >= a.height) y = a.height - 1;
        predict<FAST>(a, tb, levels, fast, w, tile, x, y, valid, g, s, pairs, out);
        if (!valid) continue;
        if (a.features) {
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
                *reinterpret_cast<uint4*>(a.features + row * 32 + 16 * kt + 8 * g) =
                    make_uint4(pairs[kt][0], pairs[kt][1], pairs[kt][2], pairs[kt][3]);
        }
        if (a.output) {
            const u32x4 bits = __builtin_bit_cast(u32x4, out);
            uint16_t* p = a.output + row * 16;
            *reinterpret_cast<uint2*>(p + 4 * g) = make_uint2(bits.x, bits.y);
            *reinterpret_cast<uint2*>(p + 8 + 4 * g) = make_uint2(bits.z, bits.w);
        }
        if (a.prediction && g == 0) {
            float* p = a.prediction + row * 3;
            rgb_of(out, p[0], p[1], p[2]);
        }
    }
}

struct ScoreArgs {
    const uint8_t* target;   // RGB8 [H*W][3]
    int resolution;
    const int32_t* xb;       // cell column / row bounds [R+1]
    const int32_t* yb;
    double* totals;          // fp64 [R*R], continued
    double* squares;         // fp64 [R*R] or null: sum of (p - byte*(1/255))^2 over the cell's channels
};

__device__ inline double lane_double(double value, int lane) {
    const uint64_t bits = __double_as_longlong(value);
    const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(bits), lane);
    const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(bits >> 32), lane);
    return __longlong_as_double((static_cast<uint64_t>(hi) << 32) | lo);
}

struct CellRange {
    int x0, y0, width;
    int64_t pixels;
};

__device__ inline CellRange cell_range(const ReconArgs& a, const ScoreArgs& sc, int64_t cell) {
    const int cx = static_cast<int>(cell % sc.resolution), cy = static_cast<int>(cell / sc.resolution);
    CellRange c;
    c.x0 = max(sc.xb[cx], 0);
    c.y0 = max(sc.yb[cy], 0);
    c.width = min(sc.xb[cx + 1], static_cast<int>(a.width)) - c.x0;
    const int rows = min(sc.yb[cy + 1], static_cast<int>(a.height)) - c.y0;
    c.pixels = c.width > 0 && rows > 0 ? static_cast<int64_t>(c.width) * rows : 0;
    return c;
}

// The residual term (residual_term, the streamed pass's arithmetic) of the wave's pixel s in lane
// group 0, 0 in the other lanes; adds the pixel's squared errors to `squares`.
template <bool FAST>
__device__ inline double pixel_residual(const ReconArgs& a, const ScoreArgs& sc, const TileBounds& tb,
                                        const DevLevel* levels, const FastLevel* fast, const _Float16* w,
                                        TileCache& tile, uint32_t x, uint32_t y, bool valid, int g, int s,
                                        double& squares) {
    uint32_t pairs[2][4];
    half8 out;
    predict<FAST>(a, tb, levels, fast, w, tile, x, y, valid, g, s, pairs, out);
    if (g != 0 || !valid) return 0.0;
    const uint32_t id = y * a.width + x;
    const float inv255 = 1.0f / 255.0f;
    float p0, p1, p2;
    rgb_of(out, p0, p1, p2);
    const uint8_t* px = sc.target + 3ull * id;
    const uint8_t b0 = px[0], b1 = px[1], b2 = px[2];
    const float e0 = p0 - static_cast<float>(b0) * inv255, e1 = p1 - static_cast<float>(b1) * inv255,
                e2 = p2 - static_cast<float>(b2) * inv255;
    squares += static_cast<double>(e0 * e0);
    squares += static_cast<double>(e1 * e1);
    squares += static_cast<double>(e2 * e2);
    if (a.prediction) {
        float* p = a.prediction + 3ull * id;
        p[0] = p0;
        p[1] = p1;
        p[2] = p2;
    }
    return residual_term(p0, p1, p2, byte_target(b0), byte_target(b1), byte_target(b2));
}

__device__ inline double wave_sum(double value) {
    for (int step = 32; step; step >>= 1) value += __shfl_xor(value, step);
    return value;
}

// Walks a cell's pixels in raster order, 32 every `step` pixels from `first`: lane s's pixel, kept as
// (column, row) so that a step costs no division.
struct CellWalk {
    int column, row, column_step, row_step;
    __device__ CellWalk(const CellRange& c, int first, int step)
        : column(first % c.width), row(first / c.width), column_step(step % c.width), row_step(step / c.width) {}
    __device__ uint32_t x(const CellRange& c, bool valid) const { return static_cast<uint32_t>(c.x0 + (valid ? column : 0)); }
    __device__ uint32_t y(const CellRange& c, bool valid) const { return static_cast<uint32_t>(c.y0 + (valid ? row : 0)); }
    __device__ void next(const CellRange& c) {
        column += column_step;
        row += row_step;
        if (column >= c.width) {
            column -= c.width;
            ++row;
        }
    }
};

// Small cells: one wave per residual cell, its pixels in raster order 32 at a time (across row ends,
// so that narrow cells fill the wave), each term folded into the cell total in order -- the
// reference's sequential fp64 sum bit for bit, with no prediction in memory.
template <bool FAST> __global__ __launch_bounds__(kReconBlock) void score_cells_kernel(ReconArgs a, TileBounds bounds, ScoreArgs sc) {
    __shared__ _Float16 w[kForwardHalfs];
    __shared__ TileBounds tb;
    __shared__ DevLevel levels[kLevels];
    __shared__ __attribute__((aligned(16))) FastLevel fast[kLevels];
    stage_model(a, bounds, w, tb, levels, fast);
    TileCache tile;
    const int lane = threadIdx.x % 64, g = lane / 32, s = lane % 32;
    const int64_t cells = static_cast<int64_t>(sc.resolution) * sc.resolution;
    for (int64_t cell = static_cast<int64_t>(blockIdx.x) * kReconWaves + threadIdx.x / 64; cell < cells;
         cell += static_cast<int64_t>(gridDim.x) * kReconWaves) {
        const CellRange c = cell_range(a, sc, cell);
        double sum = sc.totals[cell], squares = 0.0;
        if (c.pixels > 0) {
            CellWalk at(c, s, 32);
            for (int64_t k = 0; k < c.pixels; k += 32, at.next(c)) {
                const int count = static_cast<int>(c.pixels - k < 32 ? c.pixels - k : 32);
                const bool valid = s < count;
                const double term = pixel_residual<FAST>(a, sc, tb, levels, fast, w, tile, at.x(c, valid),
                                                         at.y(c, valid), valid, g, s, squares);
                for (int j = 0; j < count; ++j) sum = sum + lane_double(term, j);
            }
        }
        squares = wave_sum(squares);
        if (lane == 0) {
            sc.totals[cell] = sum;
            if (sc.squares) sc.squares[cell] = squares;
        }
    }
}

// Large cells: WAVES waves predict one cell's pixels, 32 each at a time, into one of two LDS buffers
// of terms, and a wave of their own folds the previous buffer in order meanwhile.  The fold is a
// chain of dependent fp64 adds; with a wave per cell it was part of every wave's instruction stream
// (two readlanes and an add per pixel), and a 32 x 32 grid of cells left one wave per SIMD, with
// nothing to hide the gathers and the decoder's chain behind.  8192^2 pixels in 1024 cells: 11.1 ms
// a wave per cell, 3.0 with four waves, 2.2 with the fast encode and seven waves (two workgroups per
// CU, so that 1024 cells are two full rounds; four waves and one step between barriers 2.6, eleven
// waves 2.5 - 2.7).  Now bound by VALU issue (1.7 ms of it) and the gathers' address path (TA busy
// 73%).  Up to a cell per CU: fifteen waves, one workgroup per CU.
//
// Where the lines lie, us by one wave / seven waves a cell: 1024^2 pixels in cells of 24^2 84/130, 31^2
// 130/76, 32^2 (1024 cells) 118/69, 64^2 437/74; 4096^2 in 16^2 702/2154, 31^2 721/838, 32^2 (16384
// cells) 671/833, 40^2 (10609) 734/987, 48^2 (7396) 779/763, 64^2 724/654, 128^2 1788/573; 8192^2 in 32^2
// 2504/3272, 64^2 (16384) 2556/2503, 256^2 7084/2131.  So small cells need many pixels to be worth a
// workgroup, and where there are enough cells to fill the chip with waves of one, four times as many.
// Fifteen / seven waves: 4096^2 in 256 cells 566/744, 196 833/1063, 64 2185/2935, 1 143.1/191.3 ms; 8192^2
// in 256 2148/2901, 1024 2193/2130; 1024^2 in 256 65/74, 484 98/74.
constexpr int64_t kLargeCell = 1024;   // pixels per cell from which a cell gets several waves
constexpr int64_t kManyCells = 8192;   // more cells: from 4 kLargeCell on
constexpr int kScoreSteps = 4;         // 32 pixels per wave, this many times between two barriers

template <bool FAST, int WAVES>
__global__ __launch_bounds__((WAVES + 1) * 64) void score_large_cells_kernel(ReconArgs a, TileBounds bounds, ScoreArgs sc) {
    constexpr int kScoreWaves = WAVES, kScoreStep = kScoreWaves * 32, kScoreRound = kScoreStep * kScoreSteps;
    __shared__ _Float16 w[kForwardHalfs];
    __shared__ TileBounds tb;
    __shared__ DevLevel levels[kLevels];
    __shared__ __attribute__((aligned(16))) double terms[2][kScoreRound];
    __shared__ double squares_of[kScoreWaves];
    __shared__ __attribute__((aligned(16))) FastLevel fast[kLevels];
    stage_model(a, bounds, w, tb, levels, fast);
    TileCache tile;
    const int lane = threadIdx.x % 64, g = lane / 32, s = lane % 32, wave = threadIdx.x / 64;
    const int64_t cells = static_cast<int64_t>(sc.resolution) * sc.resolution;
    for (int64_t cell = blockIdx.x; cell < cells; cell += gridDim.x) {
        const CellRange c = cell_range(a, sc, cell);
        const int64_t rounds = (c.pixels + kScoreRound - 1) / kScoreRound;
        double sum = sc.totals[cell], squares = 0.0;
        if (wave < kScoreWaves) {
            if (c.pixels > 0) {
                CellWalk at(c, wave * 32 + s, kScoreStep);
                for (int64_t round = 0; round < rounds; ++round) {
                    const int64_t left = c.pixels - round * kScoreRound - wave * 32;
                    for (int step = 0; step < kScoreSteps && left > step * kScoreStep; ++step, at.next(c)) {
                        const bool valid = left > step * kScoreStep + s;
                        const double term = pixel_residual<FAST>(a, sc, tb, levels, fast, w, tile, at.x(c, valid),
                                                                 at.y(c, valid), valid, g, s, squares);
                        if (g == 0) terms[round & 1][step * kScoreStep + wave * 32 + s] = term;
                    }
                    __syncthreads();
                }
            }
            squares = wave_sum(squares);
            if (lane == 0) squares_of[wave] = squares;
        } else {
            for (int64_t round = 0; round < rounds; ++round) {
                __syncthreads();   // the round's terms are written; the next round goes to the other buffer
                const double* t = terms[round & 1];
                const int64_t left = c.pixels - round * kScoreRound;
                if (left >= kScoreRound) {
                    for (int j = 0; j < kScoreRound; j += 16) {
                        double run[16];
#pragma unroll
                        for (int q = 0; q < 16; ++q) run[q] = t[j + q];
#pragma unroll
                        for (int q = 0; q < 16; ++q) sum = sum + run[q];
                    }
                } else {
                    for (int j = 0; j < static_cast<int>(left); ++j) sum = sum + t[j];
                }
            }
            if (lane == 0) sc.totals[cell] = sum;
        }
        __syncthreads();
        if (threadIdx.x == 0 && sc.squares) {
            double total = squares_of[0];
            for (int q = 1; q < kScoreWaves; ++q) total += squares_of[q];
            sc.squares[cell] = total;
        }
        __syncthreads();
    }
}

}  // namespace
}  // namespace odie

using namespace odie;

// Validates the model arguments shared by both entry points and fills a (everything but the
// pixel range and the outputs).  Returns 0 or -1 with the error set.
static int model_args(const char* what, int width, int height, int regions_x, int regions_y, const int32_t* slots,
                      int experts, const uint16_t* table, int64_t expert_params, const odie_grid_level* levels,
                      int n_levels, const uint16_t* weights, ReconArgs& a, TileBounds& bounds, bool& fast) {
    const std::string w(what);
    if (regions_x < 1 || regions_y < 1 || regions_x > kMaxTiles || regions_y > kMaxTiles)
        return fail(w + ": regions per axis must be within 1..64");
    if (width < 2 * regions_x || height < 2 * regions_y)
        return fail(w + ": every tile needs at least two pixels per axis");
    if (static_cast<uint64_t>(width) * static_cast<uint64_t>(height) > (uint64_t{1} << 32))
        return fail(w + ": images are limited to 2^32 pixels");
    if (n_levels != kLevels) return fail(w + ": the fused decoder takes 16 levels x 2 features");
    if (experts < 1) return fail(w + ": experts must be >= 1");
    if (!levels) return fail(w + ": levels is null");
    uint64_t entries = 0;
    if (make_dev_levels(what, levels, n_levels, a.level, entries)) return -1;
    if (expert_params < static_cast<int64_t>(entries) * 2 || expert_params % 2)
        return fail(w + ": expert_params must be even and hold the levels' table");
    if (!table || !weights) return fail(w + ": null pointer");
    if (reinterpret_cast<uintptr_t>(table) % 4) return fail(w + ": table must be 4-byte aligned");
    a.width = static_cast<uint32_t>(width);
    a.by_width = make_divisor(a.width);
    a.height = static_cast<uint32_t>(height);
    a.regions_x = regions_x;
    a.regions_y = regions_y;
    a.experts = experts;
    a.slots = slots;
    a.table = reinterpret_cast<const uint32_t*>(table);
    a.expert_pairs = expert_params / 2;
    a.weights = weights;
    make_tile_bounds(width, height, regions_x, regions_y, bounds);
    // The fast encode: 24-bit row terms, indices reduced by one subtraction or a mask, byte offsets
    // of 32 bits.  Anything else (never a layout of hash_grid_layout below 2^24 entries and 4 GB)
    // takes the general geometry.
    fast = static_cast<int64_t>(experts) * expert_params * 2 < (int64_t{1} << 32);
    for (int l = 0; l < kLevels; ++l) {
        const DevLevel& lv = a.level[l];
        const bool hashed = lv.hashed && lv.mask && lv.mask < (1u << 24);
        const bool dense = !lv.hashed && lv.res >= 2 && lv.res < (1u << 12) &&
                           static_cast<uint64_t>(lv.res) * lv.res <= lv.size;
        // the cells of u <= 1 are at most scale + 0.5 (rounded up once): below the resolution
        fast = fast && (hashed || dense) && lv.scale >= 0.0f && lv.scale <= static_cast<float>(lv.res - 1) &&
               lv.res < (1u << 22);
    }
    a.hashed_steps = 0;
    for (int step = 0; step < 8; ++step) {
        const int l = 8 * (step / 4) + step % 4;
        if (a.level[l].hashed && a.level[l + 4].hashed) a.hashed_steps |= 1u << step;
    }
    return 0;
}

ODIE_API int odie_reconstruct(int64_t begin, int64_t n, int width, int height, int regions_x, int regions_y,
                              const int32_t* slots, int experts, const uint16_t* table, int64_t expert_params,
                              const odie_grid_level* levels, int n_levels, const uint16_t* weights, float* prediction,
                              uint16_t* features, uint16_t* output, uint64_t stream) {
    if (n < 0 || begin < 0) return fail("odie_reconstruct: begin and n must be nonnegative");
    ReconArgs a{};
    TileBounds bounds;
    bool fast = false;
    if (model_args("odie_reconstruct", width, height, regions_x, regions_y, slots, experts, table, expert_params,
                   levels, n_levels, weights, a, bounds, fast))
        return -1;
    if (static_cast<uint64_t>(begin) + static_cast<uint64_t>(n) > static_cast<uint64_t>(width) * height)
        return fail("odie_reconstruct: the pixel range runs past the image");
    if (n == 0) return 0;
    if (!prediction && !features && !output) return fail("odie_reconstruct: no output");
    if ((features && reinterpret_cast<uintptr_t>(features) % 16) || (output && reinterpret_cast<uintptr_t>(output) % 8))
        return fail("odie_reconstruct: features must be 16-byte and output 8-byte aligned");
    a.begin = begin;
    a.n = n;
    a.prediction = prediction;
    a.features = features;
    a.output = output;
    const int64_t tiles = (n + 31) / 32;
    int64_t blocks = (tiles + kReconWaves - 1) / kReconWaves;
    if (blocks > 4096) blocks = 4096;
    const hipStream_t st = as_stream(stream);
    if (fast) reconstruct_kernel<true><<<static_cast<uint32_t>(blocks), kReconBlock, 0, st>>>(a, bounds);
    else reconstruct_kernel<false><<<static_cast<uint32_t>(blocks), kReconBlock, 0, st>>>(a, bounds);
    return check_launch("odie_reconstruct");
}

ODIE_API int odie_reconstruct_scores(int width, int height, int regions_x, int regions_y, const int32_t* slots,
                                     int experts, const uint16_t* table, int64_t expert_params,
                                     const odie_grid_level* levels, int n_levels, const uint16_t* weights,
                                     const uint8_t* target, int resolution, const int32_t* xb, const int32_t* yb,
                                     double* totals, double* squares, float* prediction, uint64_t stream) {
    ReconArgs a{};
    TileBounds bounds;
    bool fast = false;
    if (model_args("odie_reconstruct_scores", width, height, regions_x, regions_y, slots, experts, table,
                   expert_params, levels, n_levels, weights, a, bounds, fast))
        return -1;
    if (resolution < 1 || resolution > 65536) return fail("odie_reconstruct_scores: resolution must be within 1..65536");
    if (!target || !xb || !yb || !totals) return fail("odie_reconstruct_scores: null pointer");
    a.prediction = prediction;
    ScoreArgs sc{target, resolution, xb, yb, totals, squares};
    const int64_t cells = static_cast<int64_t>(resolution) * resolution;
    const hipStream_t st = as_stream(stream);
    const int64_t large = cells > kManyCells ? 4 * kLargeCell : kLargeCell;
    if (static_cast<int64_t>(width) * height / cells >= large) {
        const uint32_t grid = static_cast<uint32_t>(cells < 65536 ? cells : 65536);
        const bool few = cells <= kCus;
        if (fast && few) score_large_cells_kernel<true, 15><<<grid, 1024, 0, st>>>(a, bounds, sc);
        else if (fast) score_large_cells_kernel<true, 7><<<grid, 512, 0, st>>>(a, bounds, sc);
        else if (few) score_large_cells_kernel<false, 15><<<grid, 1024, 0, st>>>(a, bounds, sc);
        else score_large_cells_kernel<false, 7><<<grid, 512, 0, st>>>(a, bounds, sc);
    } else {
        int64_t blocks = (cells + kReconWaves - 1) / kReconWaves;
        if (blocks > 65536) blocks = 65536;
        const uint32_t grid = static_cast<uint32_t>(blocks);
        if (fast) score_cells_kernel<true><<<grid, kReconBlock, 0, st>>>(a, bounds, sc);
        else score_cells_kernel<false><<<grid, kReconBlock, 0, st>>>(a, bounds, sc);
    }
    return check_launch("odie_reconstruct_scores");
}
