// Router gate (router_enabled): a width -> 32 -> G fp16 MLP (ReLU hidden layer, no bias, no output
// activation; TCNN FullyFusedMLP at odie/native/runtime.cu:151-162,185, odie/hash_grid.py:28-30)
// gives one logit per level (G = align16(levels) outputs, odie/native/runtime.cu:17), s = 1 for the
// first K levels and sigmoid / softplus of the logit above, and every level's features are scaled
// by fp16(s * visible) -- parallel_gate and parallel_gate_back of odie/native/runtime.cu:64-92,
// with hash_router_gradient (:99-103) forming the grid's upstream.
//
//   gate_forward:  raw x [n][width] fp16 -> weighted [n][width] fp16 (the decoder input; columns
//                  past the levels' features are 1), s [n][L] fp32
//   gate_backward: raw x, value = fp16(dL/dweighted / 128) [n][width] (odie_mlp_train's dz), s ->
//                  upstream [n][width] = fp16(direct + fp16(dL/draw_gate / 128)),
//                  dWgate fp32 [32*width + 32*G] (loss scale 16384)
//
// Gate weights: fp16 [32*width + 32*G] = Wg1 [32][width] | Wg2 [G][32], row-major [out][in]
// (odie/config.py:176: width*32 + 32*align16(levels)).  Level l owns columns
// [offset_l, offset_l + F_l) of a row, F_l in {1, 2, 4}, offsets the running sum of F in level
// order (the descriptor's output feature offset, odie/model.py:100-101).
//
// One wave per tile of 32 samples, v_mfma_f32_32x32x16_f16 with samples as columns (the layout
// scheme and helpers of mlp.h).  Lane (g, s) holds columns 16kt + 8g + e of sample s (B operand of
// layer 1) and the logits of levels 8(v/4) + 4g + v%4 (the layer-2 accumulator).  Where every level
// has two columns (the last one or two), those are the levels of the lane's own columns, and the
// gating and its derivative stay in registers (PAIRED).  Otherwise the per-level weights
// fp16(s * visible) and the per-column products value * x pass through a per-wave LDS table indexed
// by (sample, level) or (sample, column), so a level's columns may sit in any lanes.  The input
// gradient uses Wg1^T with its rows in the columns' lane order, so its accumulator lands in the
// layout of x.
//
// Measured at 16 levels of two features (bound by latency with few waves in flight, then by the rows'
// traffic): backward of 300,007 rows 69 -> 25 us (tables out of LDS, 256 -> 512 workgroups; 768 and
// 1024 workgroups equal or slower with their partials' reduction), 65536 rows 20.5 -> 11.4 us; forward
// 26 -> 19 us (values and visibility in 16- and 4-byte accesses, no transposed weights staged, at
// most 768 workgroups; 8192 before: each staged the weights for a tile per wave) and 12.1 -> 8 us.
// The evaluation's gate, decoder and outputs in one pass (heads_kernel): 50 us per 2^20 rows, where the two
// kernels took 84 + 34 us and the tensor operations around them about 200 us.
#include <cstring>
#include <string>

#include "mlp.h"
#include "../../include/odie_amd.h"

namespace odie {
namespace {

constexpr int kGateHid = 32;
constexpr int kMaxWidth = 80;              // align16(20 levels x 4 features)
constexpr int kMaxGateLevels = 32;
constexpr int kGateBlock = 256;
constexpr int kGateWaves = kGateBlock / 64;
constexpr int kS = 40;                      // LDS row stride (halfs) of 32-wide rows
constexpr int kTStride = 40;                // transposition rows: 32 samples + pad

// Operand layouts of the gate for width 16 * KT and G = 16 * GT outputs (halfs).
template <int KT, int GT> struct GateShape {
    static constexpr int kIn = 16 * KT, kG = 16 * GT;
    static constexpr int kBlocks = (KT + 1) / 2;           // 32-row blocks of the input gradient
    static constexpr int kG1 = kGateHid * kIn, kParams = kG1 + kG * kGateHid;
    static constexpr int kSIn = kIn + 8;
    static constexpr int kA1 = 0;                           // Wg1 [32][in], A operand of layer 1
    static constexpr int kA2 = kA1 + 32 * kSIn;             // Wg2 [G][slot(32)]
    static constexpr int kT2 = kA2 + kG * kS;               // Wg2^T [32][slot(G)], dHg = Wg2^T da
    static constexpr int kT1 = kT2 + 32 * kS;               // Wg1^T [blocks*32][slot(32)] in lane order
    static constexpr int kWeightHalfs = kT1 + kBlocks * 32 * kS, kForwardHalfs = kT2;
    static constexpr int kTRows = kG + 2 * kGateHid + kIn;      // da G, hg 32, dhg 32, x in
    static constexpr int kWaveHalfs = kTRows * kTStride;
    static constexpr int kTableHalfs = 32 * kMaxGateLevels; // level weights [32 samples][32 levels]
    static_assert(kTableHalfs + 32 * kIn <= kWaveHalfs, "the level and product tables share a wave's buffer");
};

// Orders this wave's LDS writes before its lanes read what other lanes wrote.
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Levels of the rows, passed by value to the kernels and copied to LDS there.
struct LevelTable {
    uint8_t level_of[kMaxWidth];       // level of column c (0xff: a padding column)
    uint8_t offset[kMaxGateLevels];    // first column of level l
    uint8_t features[kMaxGateLevels];  // columns of level l
};

struct GateArgs {
    const uint16_t* raw;       // [n][width]
    const uint16_t* value;     // [n][width] (backward)
    const uint8_t* visible;    // [n][L] or null (all visible)
    const uint16_t* weights;   // [32*width + 32*G]
    float* sigmoid;            // [n][L]
    uint16_t* out;             // weighted [n][width] (forward) / upstream [n][width] (backward)
    float* partials;           // [blocks][32*width + 32*G] (backward)
    int64_t n;
    int levels;                // L
    int quads;                 // rows of L values keep 16- (sigmoid) and 4-byte (visible) alignment
    int coarse;                // levels < coarse are not gated (s = 1, no gate gradient)
    int softplus;
    LevelTable table;
};

// Rows whose levels have two features each but the last, which may have one: the logits a lane gets
// from the second layer are those of the levels whose columns it holds (element e of K step kt is a
// column of level 8kt + 4g + e/2, logit 4kt + e/2), so nothing passes through LDS.
bool paired_rows(const LevelTable& t, int width, int levels) {
    for (int l = 0; l < levels; ++l)
        if (t.offset[l] != 2 * l || (t.features[l] != 2 && !(t.features[l] == 1 && l + 1 == levels))) return false;
    return width / 16 <= 2 * ((levels + 15) / 16);
}

struct SharedTable {
    uint8_t level_of[kMaxWidth];
    uint8_t offset[kMaxGateLevels];
    uint8_t features[kMaxGateLevels];
};

// The gate's weights into LDS in their operand layouts (BACKWARD: the transposed ones too).
template <int KT, int GT, bool BACKWARD> __device__ void stage_gate(const GateArgs& a, _Float16* w, SharedTable& t) {
    using S = GateShape<KT, GT>;
    for (int i = threadIdx.x; BACKWARD && i < S::kBlocks * 32 * kS; i += kGateBlock) w[S::kT1 + i] = 0;   // rows past width
    for (int i = threadIdx.x; i < kMaxWidth; i += kGateBlock) t.level_of[i] = a.table.level_of[i];
    for (int i = threadIdx.x; i < kMaxGateLevels; i += kGateBlock) {
        t.offset[i] = a.table.offset[i];
        t.features[i] = a.table.features[i];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < S::kParams; i += kGateBlock) {
        const _Float16 v = __builtin_bit_cast(_Float16, a.weights[i]);
        if (i < S::kG1) {
            const int r = i / S::kIn, c = i % S::kIn;     // Wg1[hidden r][input c]
            w[S::kA1 + r * S::kSIn + c] = v;
            // Wg1^T: block c / 32, row slot_of(c % 32) (the lane order of column c), column = hidden in slot order
            if (BACKWARD) w[S::kT1 + (32 * (c / 32) + slot_of(c % 32)) * kS + slot_of(r)] = v;
        } else {
            const int j = i - S::kG1, o = j / kGateHid, c = j % kGateHid;   // Wg2[level o][hidden c]
            w[S::kA2 + o * kS + slot_of(c)] = v;
            if (BACKWARD) w[S::kT2 + c * kS + slot_of(o)] = v;
        }
    }
}

template <int KT> __device__ inline void load_rows(const uint16_t* base, int64_t row, bool valid, int g, half8 v[KT]) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
        v[kt] = valid ? *reinterpret_cast<const half8*>(base + row * (16 * KT) + kt * 16 + 8 * g) : half8{};
}
template <int KT> __device__ inline void store_rows(uint16_t* base, int64_t row, int g, const half8 v[KT]) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) *reinterpret_cast<half8*>(base + row * (16 * KT) + kt * 16 + 8 * g) = v[kt];
}

// Hidden layer and logits of one tile: hg (B operand form), logits for this lane's levels
// (element v: level 8(v/4) + 4g + v%4, v < 8 GT), rounded to fp16 as the network's output.
template <int KT, int GT>
__device__ inline void gate_layers(const _Float16* w, int g, int s, const half8 x[KT], half8 hg[2], half8 z[GT]) {
    using S = GateShape<KT, GT>;
    f32x16 acc{};
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) acc = mfma(lds8(w + S::kA1 + s * S::kSIn + kt * 16 + 8 * g), x[kt], acc);
    hg[0] = relu8(round8(acc, 0));
    hg[1] = relu8(round8(acc, 8));
    f32x16 lg{};
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const half8 a = s < S::kG ? lds8(w + S::kA2 + s * kS + 16 * t + 8 * g) : half8{};
        lg = mfma(a, hg[t], lg);
    }
#pragma unroll
    for (int t = 0; t < GT; ++t) z[t] = round8(lg, 8 * t);
}

__device__ inline int level_of_element(int v, int g) { return 8 * (v / 4) + 4 * g + v % 4; }

// s of level l from its fp16 logit (odie/native/runtime.cu:72).
__device__ inline float gate_value(float z, int level, const GateArgs& a) {
    if (level < a.coarse) return 1.0f;
    if (a.softplus) return z > 20.0f ? z : log1pf(expf(z));
    return 1.0f / (1.0f + expf(-z));
}

// A lane's four consecutive levels 8q + 4g .. + 3 of a row of L values: one load or store where rows
// of L values keep the alignment (L a multiple of 4), else one by one; levels past L are 0.
__device__ inline void visible4(const GateArgs& a, int64_t row, bool valid, int first, float out[4]) {
    if (!valid || first >= a.levels) {
        out[0] = out[1] = out[2] = out[3] = 0.0f;
    } else if (!a.visible) {
#pragma unroll
        for (int j = 0; j < 4; ++j) out[j] = first + j < a.levels ? 1.0f : 0.0f;
    } else if (a.quads) {
        const uint32_t word = *reinterpret_cast<const uint32_t*>(a.visible + row * a.levels + first);
#pragma unroll
        for (int j = 0; j < 4; ++j) out[j] = static_cast<float>((word >> (8 * j)) & 0xffu);
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) out[j] = first + j < a.levels ? static_cast<float>(a.visible[row * a.levels + first + j]) : 0.0f;
    }
}
__device__ inline void load4(const GateArgs& a, int64_t row, bool valid, int first, float out[4]) {
    if (!valid || first >= a.levels) {
        out[0] = out[1] = out[2] = out[3] = 0.0f;
    } else if (a.quads) {
        const float4 v = *reinterpret_cast<const float4*>(a.sigmoid + row * a.levels + first);
        out[0] = v.x, out[1] = v.y, out[2] = v.z, out[3] = v.w;
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) out[j] = first + j < a.levels ? a.sigmoid[row * a.levels + first + j] : 0.0f;
    }
}
__device__ inline void store4(const GateArgs& a, int64_t row, int first, const float v[4]) {
    if (first >= a.levels) return;
    if (a.quads) {
        *reinterpret_cast<float4*>(a.sigmoid + row * a.levels + first) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (first + j < a.levels) a.sigmoid[row * a.levels + first + j] = v[j];
    }
}

// The gate on a tile's rows x (in place): s of the lane's levels (sv), then x times fp16(s * visible).
// weight_of: this sample's level weights in the wave's LDS table (not used when PAIRED).
template <int KT, int GT, bool PAIRED>
__device__ inline void gate_rows(const GateArgs& a, const _Float16* w, const SharedTable& table, _Float16* weight_of,
                                 int64_t row, bool valid, int g, int s, half8 x[KT], float sv[8 * GT]) {
    half8 hg[2], z[GT];
    gate_layers<KT, GT>(w, g, s, x, hg, z);
    _Float16 weight[8 * GT];
#pragma unroll
    for (int q = 0; q < 2 * GT; ++q) {
        float vis[4];
        visible4(a, row, valid, 8 * q + 4 * g, vis);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int v = 4 * q + j, level = 8 * q + 4 * g + j;
            sv[v] = gate_value(static_cast<float>(z[v / 8][v % 8]), level, a);
            weight[v] = static_cast<_Float16>(sv[v] * vis[j]);
            if (!PAIRED && level < a.levels) weight_of[level] = weight[v];
        }
    }
    if constexpr (PAIRED) {
        const int columns = table.offset[a.levels - 1] + table.features[a.levels - 1];
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int e = 0; e < 8; ++e)
                x[kt][e] = 16 * kt + 8 * g + e < columns ? x[kt][e] * weight[4 * kt + e / 2] : static_cast<_Float16>(1.0f);
    } else {
        wave_sync();
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int level = table.level_of[16 * kt + 8 * g + e];
                x[kt][e] = level != 0xff ? x[kt][e] * weight_of[level] : static_cast<_Float16>(1.0f);
            }
        wave_sync();
    }
}

template <int KT, int GT, bool PAIRED> __global__ __launch_bounds__(kGateBlock) void gate_forward_kernel(GateArgs a) {
    using S = GateShape<KT, GT>;
    __shared__ __attribute__((aligned(16))) _Float16 w[S::kForwardHalfs];
    __shared__ SharedTable table;
    __shared__ __attribute__((aligned(16))) _Float16 scratch[PAIRED ? 8 : kGateWaves * S::kTableHalfs];
    stage_gate<KT, GT, false>(a, w, table);
    __syncthreads();
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64, g = lane / 32, s = lane % 32;
    _Float16* weight_of = PAIRED ? scratch : scratch + wave * S::kTableHalfs + s * kMaxGateLevels;   // this sample's
    const int64_t tiles = (a.n + 31) / 32;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kGateWaves;
    for (int64_t tile = static_cast<int64_t>(blockIdx.x) * kGateWaves + wave; tile < tiles; tile += stride) {
        const int64_t row = tile * 32 + s;
        const bool valid = row < a.n;
        half8 x[KT];
        float sv[8 * GT];
        load_rows<KT>(a.raw, row, valid, g, x);
        gate_rows<KT, GT, PAIRED>(a, w, table, weight_of, row, valid, g, s, x, sv);
        if (!valid) continue;
#pragma unroll
        for (int q = 0; q < 2 * GT; ++q) store4(a, row, 8 * q + 4 * g, sv + 4 * q);
        store_rows<KT>(a.out, row, g, x);
    }
}

template <int KT, int GT, bool PAIRED> __global__ __launch_bounds__(kGateBlock) void gate_backward_kernel(GateArgs a) {
    using S = GateShape<KT, GT>;
    __shared__ _Float16 w[S::kWeightHalfs];
    __shared__ SharedTable table;
    __shared__ __attribute__((aligned(16))) _Float16 transposed[kGateWaves * S::kWaveHalfs];
    stage_gate<KT, GT, true>(a, w, table);
    __syncthreads();
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64, g = lane / 32, s = lane % 32;
    _Float16* T = transposed + wave * S::kWaveHalfs;
    // the level weights and the column products of this wave's samples share the wave's rows
    _Float16* weight_of = T + s * kMaxGateLevels;
    _Float16* product_of = T + S::kTableHalfs + s * S::kIn;
    f32x16 g1[S::kBlocks], g2{};
#pragma unroll
    for (int b = 0; b < S::kBlocks; ++b) g1[b] = f32x16{};
    const int64_t tiles = (a.n + 31) / 32;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kGateWaves;
    const _Float16 half128 = static_cast<_Float16>(128.0f);
    for (int64_t tile = static_cast<int64_t>(blockIdx.x) * kGateWaves + wave; tile < tiles; tile += stride) {
        const int64_t row = tile * 32 + s;
        const bool valid = row < a.n;
        half8 x[KT], value[KT], hg[2], z[GT];
        load_rows<KT>(a.raw, row, valid, g, x);
        load_rows<KT>(a.value, row, valid, g, value);
        gate_layers<KT, GT>(w, g, s, x, hg, z);
        // parallel_gate_back (odie/native/runtime.cu:77-91): products value * raw per column,
        // weights fp16(s * visible) per level
        float sv[8 * GT], vis[8 * GT];
        _Float16 weight[8 * GT];
#pragma unroll
        for (int q = 0; q < 2 * GT; ++q) {
            load4(a, row, valid, 8 * q + 4 * g, sv + 4 * q);
            visible4(a, row, valid, 8 * q + 4 * g, vis + 4 * q);
        }
#pragma unroll
        for (int v = 0; v < 8 * GT; ++v) weight[v] = static_cast<_Float16>(sv[v] * vis[v]);
        if constexpr (!PAIRED) {
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                for (int e = 0; e < 8; ++e) product_of[16 * kt + 8 * g + e] = value[kt][e] * x[kt][e];
#pragma unroll
            for (int v = 0; v < 8 * GT; ++v)
                if (level_of_element(v, g) < a.levels) weight_of[level_of_element(v, g)] = weight[v];
            wave_sync();
        }
        half8 da[GT];
#pragma unroll
        for (int v = 0; v < 8 * GT; ++v) {
            const int level = level_of_element(v, g);
            _Float16 out = static_cast<_Float16>(0.0f);
            if (level < a.levels) {
                // the level's products summed in column order, one fp16 rounding per addition
                _Float16 reduced = static_cast<_Float16>(0.0f);
                if constexpr (PAIRED) {
                    if (v / 4 < KT) {
                        const int kt = v / 4, e = 2 * (v % 4);
                        reduced = reduced + value[kt][e] * x[kt][e];
                        if (table.features[level] == 2) reduced = reduced + value[kt][e + 1] * x[kt][e + 1];
                    }
                } else {
                    const int first = table.offset[level], count = table.features[level];
                    for (int c = 0; c < count; ++c) reduced = reduced + product_of[first + c];
                }
                const float incoming = static_cast<float>(reduced) * vis[v];
                float derivative = 0.0f;
                if (level >= a.coarse)
                    derivative = a.softplus ? incoming * -expm1f(-sv[v]) : incoming * (1.0f - sv[v]) * sv[v];
                out = static_cast<_Float16>(derivative) * half128;
            }
            da[v / 8][v % 8] = out;
        }
        half8 direct[KT];
        if constexpr (PAIRED) {
            const int columns = table.offset[a.levels - 1] + table.features[a.levels - 1];
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    direct[kt][e] = 16 * kt + 8 * g + e < columns ? value[kt][e] * weight[4 * kt + e / 2]
                                                                   : static_cast<_Float16>(0.0f);
        } else {
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int level = table.level_of[16 * kt + 8 * g + e];
                    direct[kt][e] = level != 0xff ? value[kt][e] * weight_of[level] : static_cast<_Float16>(0.0f);
                }
            wave_sync();   // the tables are dead; the rows below reuse their space
        }
        // gate MLP backward: dHg = relu'(hg) * (Wg2^T da); d(raw) = Wg1^T dHg
        half8 dhg[2];
        {
            f32x16 acc{};
#pragma unroll
            for (int t = 0; t < GT; ++t) acc = mfma(lds8(w + S::kT2 + s * kS + 16 * t + 8 * g), da[t], acc);
            dhg[0] = mask8(round8(acc, 0), hg[0]);
            dhg[1] = mask8(round8(acc, 8), hg[1]);
        }
        // hash_router_gradient (odie/native/runtime.cu:99-103): direct + fp16(dr / 128); block b
        // of the input gradient holds K steps 2b, 2b + 1 of the row in x's lane layout
        const half8 scale = (half8)(static_cast<_Float16>(0.0078125f));
        half8 up[KT];
#pragma unroll
        for (int b = 0; b < S::kBlocks; ++b) {
            f32x16 acc{};
#pragma unroll
            for (int t = 0; t < 2; ++t) acc = mfma(lds8(w + S::kT1 + (32 * b + s) * kS + 16 * t + 8 * g), dhg[t], acc);
#pragma unroll
            for (int q = 0; q < 2; ++q)
                if (2 * b + q < KT) up[2 * b + q] = direct[2 * b + q] + round8(acc, 8 * q) * scale;
        }
        if (valid) store_rows<KT>(a.out, row, g, up);
        // weight gradients over this tile's samples: dWg2 = sum da (x) hg, dWg1 = sum dhg (x) x;
        // rows 0..G-1 da, G.. hg, G+32.. dhg, G+64.. x (feature-major, samples contiguous)
#pragma unroll
        for (int v = 0; v < 8 * GT; ++v) T[level_of_element(v, g) * kTStride + s] = da[v / 8][v % 8];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                T[(S::kG + feature_of(t, g, e)) * kTStride + s] = hg[t][e];
                T[(S::kG + 32 + feature_of(t, g, e)) * kTStride + s] = dhg[t][e];
            }
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int e = 0; e < 8; ++e) T[(S::kG + 64 + 16 * kt + 8 * g + e) * kTStride + s] = x[kt][e];
        wave_sync();
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
            const half8 ada = s < S::kG ? lds8(T + s * kTStride + kt * 16 + 8 * g) : half8{};
            g2 = mfma(ada, lds8(T + (S::kG + s) * kTStride + kt * 16 + 8 * g), g2);
            const half8 adh = lds8(T + (S::kG + 32 + s) * kTStride + kt * 16 + 8 * g);
#pragma unroll
            for (int b = 0; b < S::kBlocks; ++b) {
                const half8 bx = 32 * b + s < S::kIn ? lds8(T + (S::kG + 64 + 32 * b + s) * kTStride + kt * 16 + 8 * g)
                                                     : half8{};
                g1[b] = mfma(adh, bx, g1[b]);
            }
        }
        wave_sync();
    }
    // reduce the waves' gradients in a fixed order through LDS, then write this workgroup's partial
    __syncthreads();
    float* sum = reinterpret_cast<float*>(transposed);
    for (int turn = 0; turn < kGateWaves; ++turn) {
        if (wave == turn) {
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int r = 8 * (v / 4) + 4 * g + v % 4;
#pragma unroll
                for (int b = 0; b < S::kBlocks; ++b)
                    if (32 * b + s < S::kIn) {
                        float* p1 = sum + r * S::kIn + 32 * b + s;     // dWg1[hidden r][input 32b + s]
                        *p1 = turn ? *p1 + g1[b][v] : g1[b][v];
                    }
                if (r < S::kG) {
                    float* p2 = sum + S::kG1 + r * kGateHid + s;          // dWg2[level r][hidden s]
                    *p2 = turn ? *p2 + g2[v] : g2[v];
                }
            }
        }
        __syncthreads();
    }
    for (int i = threadIdx.x; i < S::kParams; i += kGateBlock)
        a.partials[static_cast<int64_t>(blockIdx.x) * S::kParams + i] = sum[i];
}

// dweights[p] = sum over workgroups of partials[b][p] in a fixed order: eight lane groups of a
// 256-thread block take the workgroups b = q, q+8, q+16, ... (q = group), eight loads in flight
// per step, and the group sums are added in group order.
constexpr int kReduceParams = 32, kReduceGroups = 256 / kReduceParams;
__global__ __launch_bounds__(256) void gate_reduce_kernel(const float* partials, int blocks, int params,
                                                          float* dweights) {
    __shared__ float group_sum[kReduceGroups][kReduceParams];
    const int local = threadIdx.x % kReduceParams, q = threadIdx.x / kReduceParams;
    const int p = blockIdx.x * kReduceParams + local;
    float total = 0.0f;
    if (p < params) {
        int b = q;
        for (; b + 7 * kReduceGroups < blocks; b += 8 * kReduceGroups) {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = partials[static_cast<int64_t>(b + kReduceGroups * j) * params + p];
#pragma unroll
            for (int j = 0; j < 8; ++j) total += v[j];
        }
        for (; b < blocks; b += kReduceGroups) total += partials[static_cast<int64_t>(b) * params + p];
    }
    group_sum[q][local] = total;
    __syncthreads();
    if (q == 0 && p < params) {
        float sum = group_sum[0][local];
        for (int j = 1; j < kReduceGroups; ++j) sum += group_sum[j][local];
        dweights[p] = sum;
    }
}

constexpr int kGateBlocks = 512, kForwardBlocks = 768;

int gate_blocks(int64_t n) {
    const int64_t tiles = (n + 31) / 32;
    const int64_t blocks = (tiles + kGateWaves - 1) / kGateWaves;
    return static_cast<int>(blocks < kGateBlocks ? (blocks < 1 ? 1 : blocks) : kGateBlocks);
}

// Validates the shape and fills the level table; returns the parameter count or -1.
int64_t gate_shape(const std::string& w, int64_t n, int width, int levels, const int32_t* features, int coarse,
                   const void* raw, const void* weights, LevelTable& table) {
    if (n < 0 || n >= (int64_t{1} << 31)) return fail(w + ": n must be within [0, 2^31)");
    if (width < 16 || width > kMaxWidth || width % 16) return fail(w + ": width must be 16, 32, 48, 64 or 80");
    if (levels < 1 || levels > kMaxGateLevels) return fail(w + ": levels must be within [1, 32]");
    if (coarse < 0 || coarse > levels) return fail(w + ": coarse levels must be within [0, levels]");
    if (!weights || (n && !raw)) return fail(w + ": null pointer");
    if (reinterpret_cast<uintptr_t>(raw) % 16) return fail(w + ": rows must be 16-byte aligned");
    std::memset(&table, 0xff, sizeof(table.level_of));
    int offset = 0;
    for (int l = 0; l < levels; ++l) {
        const int f = features ? features[l] : 2;
        if (f != 1 && f != 2 && f != 4) return fail(w + ": features per level must be 1, 2 or 4");
        if (offset + f > width) return fail(w + ": the levels' features exceed the row width");
        table.offset[l] = static_cast<uint8_t>(offset);
        table.features[l] = static_cast<uint8_t>(f);
        for (int c = 0; c < f; ++c) table.level_of[offset + c] = static_cast<uint8_t>(l);
        offset += f;
    }
    for (int l = levels; l < kMaxGateLevels; ++l) table.offset[l] = table.features[l] = 0;
    if ((offset + 15) / 16 * 16 != width) return fail(w + ": width must be align16 of the levels' features");
    const int g = (levels + 15) / 16 * 16;
    return int64_t{32} * width + int64_t{32} * g;
}

#define ODIE_GATE_CASE(KERNEL, KT, GT, paired, blocks, stream, args)                            \
    case (KT) * 4 + (GT):                                                                        \
        if (paired) KERNEL<KT, GT, (KT) <= 2 * (GT)><<<blocks, kGateBlock, 0, stream>>>(args);   \
        else KERNEL<KT, GT, false><<<blocks, kGateBlock, 0, stream>>>(args);                     \
        break

#define ODIE_GATE_SWITCH(KERNEL, kt, gt, paired, blocks, stream, args)      \
    switch ((kt) * 4 + (gt)) {                                              \
        ODIE_GATE_CASE(KERNEL, 1, 1, paired, blocks, stream, args);         \
        ODIE_GATE_CASE(KERNEL, 1, 2, paired, blocks, stream, args);         \
        ODIE_GATE_CASE(KERNEL, 2, 1, paired, blocks, stream, args);         \
        ODIE_GATE_CASE(KERNEL, 2, 2, paired, blocks, stream, args);         \
        ODIE_GATE_CASE(KERNEL, 3, 1, paired, blocks, stream, args);         \
        ODIE_GATE_CASE(KERNEL, 3, 2, paired, blocks, stream, args);         \
        ODIE_GATE_CASE(KERNEL, 4, 1, paired, blocks, stream, args);         \
        ODIE_GATE_CASE(KERNEL, 4, 2, paired, blocks, stream, args);         \
        ODIE_GATE_CASE(KERNEL, 5, 1, paired, blocks, stream, args);         \
        default: KERNEL<5, 2, false><<<blocks, kGateBlock, 0, stream>>>(args); break; \
    }

// The evaluation's heads on feature rows in one pass (odie/model.py:266-279): the gate on the rows in
// registers, then the decoder, whose first layer takes its operand in the lane layout the rows were
// loaded in, and the first three outputs as fp32 -- the bits of odie_gate_forward and
// odie_mlp_forward, without the weighted rows, the gate values and the 16 outputs in memory.
struct HeadsArgs {
    GateArgs gate;             // raw: the rows; visible, weights, table as the gate reads them
    const uint16_t* decoder;   // fp16 [64*width + 5120]
    float* rgb;                // [n][3]
    int columns;               // columns past these are 1
};

template <int KT, int GT, bool GATE, bool PAIRED> __global__ __launch_bounds__(kGateBlock) void heads_kernel(HeadsArgs a) {
    using S = GateShape<KT, GT>;
    __shared__ __attribute__((aligned(16))) _Float16 decoder[Shape<KT>::kForwardHalfs];
    __shared__ __attribute__((aligned(16))) _Float16 w[GATE ? S::kForwardHalfs : 8];
    __shared__ SharedTable table;
    __shared__ __attribute__((aligned(16))) _Float16 scratch[GATE && !PAIRED ? kGateWaves * S::kTableHalfs : 8];
    static_assert(kGateBlock == kMlpBlock, "both stagings stride by their block");
    stage_forward_weights<KT>(a.decoder, decoder);
    if constexpr (GATE) stage_gate<KT, GT, false>(a.gate, w, table);
    __syncthreads();
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64, g = lane / 32, s = lane % 32;
    _Float16* weight_of = GATE && !PAIRED ? scratch + wave * S::kTableHalfs + s * kMaxGateLevels : scratch;
    const int64_t tiles = (a.gate.n + 31) / 32;
    const int64_t stride = static_cast<int64_t>(gridDim.x) * kGateWaves;
    for (int64_t tile = static_cast<int64_t>(blockIdx.x) * kGateWaves + wave; tile < tiles; tile += stride) {
        const int64_t row = tile * 32 + s;
        const bool valid = row < a.gate.n;
        half8 x[KT];
        load_rows<KT>(a.gate.raw, row, valid, g, x);
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (16 * kt + 8 * g + e >= a.columns) x[kt][e] = static_cast<_Float16>(1.0f);
        if constexpr (GATE) {
            float sv[8 * GT];
            gate_rows<KT, GT, PAIRED>(a.gate, w, table, weight_of, row, valid, g, s, x, sv);
        }
        half8 h1[4], h2[4];
        f32x16 acc3;
        forward_tile<KT>(decoder, g, s, x, h1, h2, acc3);
        const half8 out = round8(acc3, 0);
        if (valid && g == 0) {
            float* rgb = a.rgb + row * 3;
            rgb[0] = static_cast<float>(out[0]);
            rgb[1] = static_cast<float>(out[1]);
            rgb[2] = static_cast<float>(out[2]);
        }
    }
}

template <int KT> void launch_heads(const HeadsArgs& a, bool gate, bool wide, bool paired, uint32_t blocks, hipStream_t s) {
    if (!gate) heads_kernel<KT, 1, false, false><<<blocks, kGateBlock, 0, s>>>(a);
    else if (!wide && paired && KT <= 2) heads_kernel<KT, 1, true, KT <= 2><<<blocks, kGateBlock, 0, s>>>(a);
    else if (!wide) heads_kernel<KT, 1, true, false><<<blocks, kGateBlock, 0, s>>>(a);
    else if (paired && KT <= 4) heads_kernel<KT, 2, true, KT <= 4><<<blocks, kGateBlock, 0, s>>>(a);
    else heads_kernel<KT, 2, true, false><<<blocks, kGateBlock, 0, s>>>(a);
}

// Rows of L values at 16-byte (sigmoid) and 4-byte (visible) steps.
int quad_rows(const GateArgs& a) {
    return a.levels % 4 == 0 && reinterpret_cast<uintptr_t>(a.sigmoid) % 16 == 0 &&
           reinterpret_cast<uintptr_t>(a.visible) % 4 == 0;
}

}  // namespace
}  // namespace odie

using namespace odie;

ODIE_API int odie_gate_forward(const uint16_t* raw, int64_t n, int width, int levels, const int32_t* features,
                               const uint16_t* weights, const uint8_t* visible, int coarse, int softplus,
                               uint16_t* weighted, float* sigmoid, uint64_t stream) {
    GateArgs a{};
    if (gate_shape("odie_gate_forward", n, width, levels, features, coarse, raw, weights, a.table) < 0) return -1;
    if (n == 0) return 0;
    if (!weighted || !sigmoid) return fail("odie_gate_forward: null pointer");
    if (reinterpret_cast<uintptr_t>(weighted) % 16) return fail("odie_gate_forward: rows must be 16-byte aligned");
    a.raw = raw;
    a.visible = visible;
    a.weights = weights;
    a.sigmoid = sigmoid;
    a.out = weighted;
    a.n = n;
    a.levels = levels;
    a.coarse = coarse;
    a.softplus = softplus ? 1 : 0;
    // up to the workgroups the chip holds at once: more would each stage the weights for one tile per wave
    const int64_t tiles = (n + 31) / 32;
    int64_t forward_blocks = (tiles + kGateWaves - 1) / kGateWaves;
    forward_blocks = forward_blocks < 1 ? 1 : (forward_blocks > kForwardBlocks ? kForwardBlocks : forward_blocks);
    const uint32_t blocks = static_cast<uint32_t>(forward_blocks);
    const hipStream_t s = as_stream(stream);
    a.quads = quad_rows(a);
    const bool paired = paired_rows(a.table, width, levels);
    ODIE_GATE_SWITCH(gate_forward_kernel, width / 16, (levels + 15) / 16, paired, blocks, s, a);
    return check_launch("odie_gate_forward");
}

ODIE_API int odie_gate_backward(const uint16_t* raw, const uint16_t* value, int64_t n, int width, int levels,
                                const int32_t* features, const uint16_t* weights, const uint8_t* visible,
                                const float* sigmoid, int coarse, int softplus, uint16_t* upstream, float* dweights,
                                uint64_t stream) {
    GateArgs a{};
    const int64_t params = gate_shape("odie_gate_backward", n, width, levels, features, coarse, raw, weights, a.table);
    if (params < 0) return -1;
    if (!dweights) return fail("odie_gate_backward: null pointer");
    const hipStream_t s = as_stream(stream);
    if (n == 0) return launch_fill_zero(dweights, params, s);
    if (!value || !sigmoid || !upstream) return fail("odie_gate_backward: null pointer");
    if (reinterpret_cast<uintptr_t>(value) % 16 || reinterpret_cast<uintptr_t>(upstream) % 16)
        return fail("odie_gate_backward: rows must be 16-byte aligned");
    const int blocks = gate_blocks(n);
    float* partials = static_cast<float*>(workspace(static_cast<size_t>(blocks) * params * 4, s));
    if (!partials) return -1;
    a.raw = raw;
    a.value = value;
    a.visible = visible;
    a.weights = weights;
    a.sigmoid = const_cast<float*>(sigmoid);
    a.out = upstream;
    a.partials = partials;
    a.n = n;
    a.levels = levels;
    a.coarse = coarse;
    a.softplus = softplus ? 1 : 0;
    a.quads = quad_rows(a);
    const bool paired = paired_rows(a.table, width, levels);
    ODIE_GATE_SWITCH(gate_backward_kernel, width / 16, (levels + 15) / 16, paired, static_cast<uint32_t>(blocks), s, a);
    if (check_launch("odie_gate_backward")) return -1;
    gate_reduce_kernel<<<static_cast<uint32_t>((params + kReduceParams - 1) / kReduceParams), 256, 0, s>>>(
        partials, blocks, static_cast<int>(params), dweights);
    return check_launch("odie_gate_backward reduce");
}

ODIE_API int odie_heads_forward(const uint16_t* rows, int64_t n, int width, int columns, int levels,
                                const int32_t* features, const uint16_t* gate_weights, const uint8_t* visible,
                                int coarse, int softplus, const uint16_t* decoder_weights, float* rgb,
                                uint64_t stream) {
    HeadsArgs a{};
    if (gate_weights) {
        if (gate_shape("odie_heads_forward", n, width, levels, features, coarse, rows, gate_weights, a.gate.table) < 0)
            return -1;
    } else {
        if (n < 0 || n >= (int64_t{1} << 31)) return fail("odie_heads_forward: n must be within [0, 2^31)");
        if (width < 16 || width > kMaxWidth || width % 16)
            return fail("odie_heads_forward: width must be 16, 32, 48, 64 or 80");
    }
    if (columns < 0 || columns > width) return fail("odie_heads_forward: columns must be within [0, width]");
    if (n == 0) return 0;
    if (!rows || !decoder_weights || !rgb) return fail("odie_heads_forward: null pointer");
    if (reinterpret_cast<uintptr_t>(rows) % 16) return fail("odie_heads_forward: rows must be 16-byte aligned");
    a.gate.raw = rows;
    a.gate.visible = visible;
    a.gate.weights = gate_weights;
    a.gate.n = n;
    a.gate.levels = levels;
    a.gate.coarse = coarse;
    a.gate.softplus = softplus ? 1 : 0;
    a.gate.quads = quad_rows(a.gate);
    a.decoder = decoder_weights;
    a.rgb = rgb;
    a.columns = columns;
    const bool gate = gate_weights != nullptr, wide = levels > 16;
    const bool paired = gate && paired_rows(a.gate.table, width, levels);
    const int64_t tiles = (n + 31) / 32;
    const int64_t most = (tiles + kGateWaves - 1) / kGateWaves;
    const uint32_t blocks = static_cast<uint32_t>(most < kForwardBlocks ? most : kForwardBlocks);
    const hipStream_t s = as_stream(stream);
    switch (width / 16) {
        case 1: launch_heads<1>(a, gate, wide, paired, blocks, s); break;
        case 2: launch_heads<2>(a, gate, wide, paired, blocks, s); break;
        case 3: launch_heads<3>(a, gate, wide, paired, blocks, s); break;
        case 4: launch_heads<4>(a, gate, wide, paired, blocks, s); break;
        default: launch_heads<5>(a, gate, wide, paired, blocks, s); break;
    }
    return check_launch("odie_heads_forward");
}
