// Per-source INT8 quantization and packed16 byte permutation for gfx950 (wave64).
//
// quantize: rows of features % 4 == 0 (16-byte aligned) use 16-byte loads of 4-feature groups and one
// dword store per 4 quantized bytes: quantizeRowsFit for F <= 256 (one group per lane, several rows
// per thread held in registers, X read once), quantizeRowsLong above; other widths (5 <= F <= 2048) of more
// than a few thousand rows go through LDS a tile of rows at a time (quantizeTile), the rest one wave per row
// (quantizeRows). The row's |x| maximum is reduced across its lanes with shuffles, and every element is
// divided by the scale with the IEEE-correct FP32 divide and rounded half-to-even. Results are bit-identical
// to reference src/format/int8_quantize.cu:4-25.
//
// pack: one thread per 16-byte tile; four v_perm_b32 byte shuffles turn q[0..15] into
// [q0,q8,q1,q9,...,q7,q15] (reference src/format/pack_int8.cu:6-15). Unaligned buffers use a
// byte-pair kernel with the same result.
//
// quantize + pack fused (no counterpart in the reference): the quantize kernels with `Packed` set
// write the packed layout directly, so q is never written and read back. In the vector kernels the
// four lanes of a 16-feature tile swap their quantized dwords with two quad-permute DPP moves and
// assemble their output dword with one v_perm_b32; the scalar kernel stores each byte at its packed
// position.
#include "format/int8_features.h"
#include "hip_support.h"

#include <hip/hip_runtime.h>

#include <cstddef>
#include <stdexcept>

namespace {

constexpr unsigned kWave = 64;
constexpr unsigned kRowsPerBlock = 4;

// Byte offset of feature j of a row in the packed16 layout: within each 16-feature tile, feature k
// goes to byte 2k (k < 8) or 2(k - 8) + 1.
__device__ __forceinline__ unsigned packedOffset(unsigned j) {
    const unsigned k = j & 15u;
    return (j & ~15u) + (k < 8 ? 2 * k : 2 * (k - 8) + 1);
}

template <bool Packed>
__global__ __launch_bounds__(kWave* kRowsPerBlock) void quantizeRows(
    const float* __restrict__ x, std::int8_t* __restrict__ q, float* __restrict__ scale,
    unsigned sources, unsigned features) {
    const unsigned lane = threadIdx.x & (kWave - 1);
    const std::size_t row = std::size_t(blockIdx.x) * kRowsPerBlock + (threadIdx.x / kWave);
    if (row >= sources) return;
    const float* xr = x + std::size_t(row) * features;
    float m = 0.0f;
    for (unsigned j = lane; j < features; j += kWave) m = fmaxf(m, fabsf(xr[j]));
#pragma unroll
    for (unsigned offset = kWave / 2; offset > 0; offset >>= 1) m = fmaxf(m, __shfl_xor(m, offset));
    const float s = m == 0.0f ? 1.0f : m / 127.0f;
    if (lane == 0) scale[row] = s;
    std::int8_t* qr = q + std::size_t(row) * features;
    for (unsigned j = lane; j < features; j += kWave) {
        const int v = __float2int_rn(xr[j] / s);
        qr[Packed ? packedOffset(j) : j] = std::int8_t(v < -127 ? -127 : (v > 127 ? 127 : v));
    }
}

// Vector paths for features % 4 == 0 with 16-byte aligned rows. Same arithmetic as quantizeRows
// (IEEE divide, round half to even, clamp).
__device__ __forceinline__ int quantizeOne(float v, float s) {
    const int r = __float2int_rn(v / s);
    return r < -127 ? -127 : (r > 127 ? 127 : r);
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned quantizeGroup(f32x4 v, float s) {
    return (unsigned(quantizeOne(v.x, s)) & 0xFFu) | (unsigned(quantizeOne(v.y, s)) & 0xFFu) << 8 |
           (unsigned(quantizeOne(v.z, s)) & 0xFFu) << 16 | (unsigned(quantizeOne(v.w, s)) & 0xFFu) << 24;
}

// The packed16 dword of lane `lane` from the quantized dwords of its 16-feature tile, held by the
// tile's four lanes (w0..w3 = features 0-3, 4-7, 8-11, 12-15): output dword i is bytes
// [q(2i), q(2i+8), q(2i+1), q(2i+9)], i.e. two bytes of w(i/2) and two of w(i/2 + 2). All four lanes
// of the tile must execute this together.
__device__ __forceinline__ unsigned packDword(unsigned qd, unsigned lane) {
    const unsigned lo = unsigned(__builtin_amdgcn_mov_dpp(int(qd), 0x50, 0xF, 0xF, false)); // quad [0,0,1,1]
    const unsigned hi = unsigned(__builtin_amdgcn_mov_dpp(int(qd), 0xFA, 0xF, 0xF, false)); // quad [2,2,3,3]
    // v_perm_b32 selectors: bytes 0-3 pick from the second operand, 4-7 from the first.
    return __builtin_amdgcn_perm(hi, lo, (lane & 1u) ? 0x07030602u : 0x05010400u);
}

__device__ __forceinline__ float absMax(f32x4 v) {
    return fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
}

// Rows of at most 64 groups of 4 features (F <= 256): `Lanes` (a power of two >= groups) lanes per
// row, each holding one group; a thread handles kQuantRows rows kRowsPerPass apart, issuing all of
// its 16-byte loads before the reductions, so a wave keeps 4 KiB of X in flight and reads X once.
// X is streamed with nontemporal loads and q with nontemporal stores (neither is re-read here).
constexpr unsigned kQuantRows = 4;

template <unsigned Lanes, bool Packed>
__global__ __launch_bounds__(256) void quantizeRowsFit(const f32x4* __restrict__ x,
                                                        unsigned* __restrict__ q,
                                                        float* __restrict__ scale,
                                                        unsigned sources, unsigned groups) {
    constexpr unsigned kRowsPerPass = 256 / Lanes;
    const unsigned lane = threadIdx.x & (Lanes - 1);
    const std::size_t row0 = std::size_t(blockIdx.x) * kRowsPerPass * kQuantRows + threadIdx.x / Lanes;
    f32x4 v[kQuantRows];
    float m[kQuantRows];
#pragma unroll
    for (unsigned r = 0; r < kQuantRows; ++r) {
        const std::size_t row = row0 + r * kRowsPerPass;
        const bool live = row < sources && lane < groups;
        v[r] = __builtin_nontemporal_load(x + (live ? row * groups + lane : 0));
        if (!live) v[r] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        m[r] = absMax(v[r]);
    }
#pragma unroll
    for (unsigned offset = Lanes / 2; offset > 0; offset >>= 1)
#pragma unroll
        for (unsigned r = 0; r < kQuantRows; ++r) m[r] = fmaxf(m[r], __shfl_xor(m[r], offset));
#pragma unroll
    for (unsigned r = 0; r < kQuantRows; ++r) {
        const std::size_t row = row0 + r * kRowsPerPass;
        if (row >= sources) break;
        const float s = m[r] == 0.0f ? 1.0f : m[r] / 127.0f;
        if (lane == 0) scale[row] = s;
        unsigned qd = quantizeGroup(v[r], s);
        if constexpr (Packed) qd = packDword(qd, lane); // the row's tiles are whole lane quads
        if (lane < groups) __builtin_nontemporal_store(qd, q + row * groups + lane);
    }
}

// Rows of more than 64 groups: one wave per row, looping over the groups twice (maximum, then
// quantize; the second read of the row hits L2).
template <bool Packed>
__global__ __launch_bounds__(256) void quantizeRowsLong(const f32x4* __restrict__ x,
                                                         unsigned* __restrict__ q,
                                                         float* __restrict__ scale,
                                                         unsigned sources, unsigned groups) {
    const unsigned lane = threadIdx.x & (kWave - 1);
    const std::size_t row = (std::size_t(blockIdx.x) * 256 + threadIdx.x) / kWave;
    if (row >= sources) return;
    const f32x4* xr = x + row * groups;
    float m = 0.0f;
    for (unsigned j = lane; j < groups; j += kWave) m = fmaxf(m, absMax(xr[j]));
#pragma unroll
    for (unsigned offset = kWave / 2; offset > 0; offset >>= 1) m = fmaxf(m, __shfl_xor(m, offset));
    const float s = m == 0.0f ? 1.0f : m / 127.0f;
    if (lane == 0) scale[row] = s;
    unsigned* qr = q + row * groups;
    for (unsigned j = lane; j < groups; j += kWave) {
        unsigned qd = quantizeGroup(xr[j], s);
        if constexpr (Packed) qd = packDword(qd, lane); // groups % 4 == 0: whole quads
        qr[j] = qd;
    }
}

// Rows of any width 5 <= F <= kTileFeatures whose X is 16-byte aligned, in tiles of kRows rows (a power
// of two, at least 4, so that every tile starts 16-byte aligned in X and 4-byte aligned in q). A row of
// a width that is not a multiple of 4 is not 16-byte aligned, but a tile is one contiguous stretch: it
// is copied to LDS with 16-byte loads, the row maxima are taken there (256 / rows threads each), and q is
// written four bytes at a time across the row ends. Bound by HBM: 300,007 x 50 (75 MB) in 49.9 us with
// one wave per row and 4-byte loads, 18.6 us with tiles (50,001 x 602: 48.8 -> 37.6; 1,000,003 x 5: 155 ->
// 8.4).
constexpr unsigned kTileFeatures = 2048, kTileFloats = 4096;

__global__ __launch_bounds__(256) void quantizeTile(const float* __restrict__ x,
                                                     std::int8_t* __restrict__ q,
                                                     float* __restrict__ scale, unsigned sources,
                                                     unsigned features, unsigned rows,
                                                     unsigned rowMagic) {
    extern __shared__ __align__(16) float tile[]; // [rows x features], then the rows' scales + 1
    const unsigned t = threadIdx.x;
    const std::size_t row0 = std::size_t(blockIdx.x) * rows;
    const unsigned live = unsigned(min(std::size_t(rows), sources - row0));
    const unsigned n = live * features, quads = n / 4;
    float* rowScale = tile + rows * features;
    const float* xt = x + row0 * features;
    for (unsigned i = t; i < quads; i += 256)
        reinterpret_cast<f32x4*>(tile)[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(xt) + i);
    for (unsigned i = 4 * quads + t; i < n; i += 256) tile[i] = xt[i];
    __syncthreads();
    const unsigned perRow = 256 / rows, row = t / perRow;
    float m = 0.0f;
    if (row < live)
        for (unsigned j = t % perRow; j < features; j += perRow)
            m = fmaxf(m, fabsf(tile[row * features + j]));
    for (unsigned offset = perRow / 2; offset > 0; offset >>= 1) m = fmaxf(m, __shfl_xor(m, offset));
    if (t % perRow == 0 && row < live) {
        const float s = m == 0.0f ? 1.0f : m / 127.0f;
        scale[row0 + row] = s;
        rowScale[row] = s;
    }
    if (t == 0) rowScale[live] = 1.0f; // read beside the last row's, never used
    __syncthreads();
    std::int8_t* qt = q + row0 * features;
    // floor(e / features) is the high word of e x rowMagic (floor(2^32 / features) + 1): e < 2^16 here.
    for (unsigned i = t; i < quads; i += 256) {
        const f32x4 v = reinterpret_cast<const f32x4*>(tile)[i];
        const unsigned r = __umulhi(4 * i, rowMagic), left = (r + 1) * features - 4 * i;
        const float s0 = rowScale[r], s1 = rowScale[r + 1];
        unsigned qd = 0;
#pragma unroll
        for (unsigned j = 0; j < 4; ++j)
            qd |= (unsigned(quantizeOne(v[j], j < left ? s0 : s1)) & 0xFFu) << (8 * j);
        __builtin_nontemporal_store(qd, reinterpret_cast<unsigned*>(qt) + i);
    }
    for (unsigned i = 4 * quads + t; i < n; i += 256)
        qt[i] = std::int8_t(quantizeOne(tile[i], rowScale[__umulhi(i, rowMagic)]));
}

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// One thread per 16-byte tile; q is read once and packed written once, so both use nontemporal
// access (measured on c3: 6.5 TB/s against 6.0 with the default policy).
__global__ __launch_bounds__(256) void packTiles(const u32x4* __restrict__ q,
                                                 u32x4* __restrict__ out, std::size_t tiles) {
    const std::size_t t = std::size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= tiles) return;
    const u32x4 w = __builtin_nontemporal_load(q + t);
    // v_perm_b32 selectors: bytes 0-3 pick from the second operand, 4-7 from the first.
    u32x4 r;
    r.x = __builtin_amdgcn_perm(w.z, w.x, 0x05010400u); // q0  q8  q1  q9
    r.y = __builtin_amdgcn_perm(w.z, w.x, 0x07030602u); // q2  q10 q3  q11
    r.z = __builtin_amdgcn_perm(w.w, w.y, 0x05010400u); // q4  q12 q5  q13
    r.w = __builtin_amdgcn_perm(w.w, w.y, 0x07030602u); // q6  q14 q7  q15
    __builtin_nontemporal_store(r, out + t);
}

__global__ __launch_bounds__(256) void packPairs(const std::uint8_t* __restrict__ q,
                                                 unsigned short* __restrict__ out,
                                                 std::size_t pairs) {
    const std::size_t p = std::size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (p >= pairs) return;
    const std::size_t o = (p >> 3) * 16 + (p & 7);
    out[p] = static_cast<unsigned short>(q[o] | (unsigned(q[o + 8]) << 8));
}

} // namespace

namespace {

// The quantize kernels for one call: the vector kernels for 16-byte aligned rows of features % 4 ==
// 0 with a 4-byte aligned output, the tile kernel for other widths of such buffers (at F < 5 four
// features can span more than two rows; above 2,048 a tile does not fit LDS beside others) unless they have
// few rows, the scalar kernel otherwise. `Packed` writes the packed16 layout (features % 16 == 0, checked by
// the caller).

// Whether one wave per row beats tiles. The chip holds 8,192 such waves at once, whose rows then take one
// memory latency and no barrier; a tile has two barriers, and few rows make few tiles. Well above that the waves
// come in rounds, narrow rows leave most lanes idle and wide ones loop. Device time in us, wave per row /
// tiles: F = 13: 4,096 rows 2.4 / 2.8, 8,192 3.0 / 2.8; 33: 10,007 3.4 / 3.6, 12,288 3.7 / 3.3; 50: 4,096 2.4 /
// 3.3, 16,384 4.3 / 3.9; 127: 12,500 4.7 / 5.0, 16,384 5.4 / 5.3; 201: 4,096 3.4 / 3.9, 12,500 5.9 / 6.3, 20,011 7.9 / 7.7; 257:
// 12,288 7.4 / 6.8; 511: 2,048 4.4 / 4.0, 6,144 5.4 / 5.9, 10,007 8.6 / 8.6; 599: 8,192 9.4 / 8.4; 767: 1,024
// 5.4 / 4.1.
bool fewRows(std::uint32_t sources, std::uint32_t features) {
    if (features >= 320) return features < 544 && sources > 2048 && sources <= 8192;
    if (features < 48 || features >= 256) return sources <= (features < 32 ? 7168u : 10240u);
    return sources <= (features < 96 ? 12288u : 14336u);
}

template <bool Packed>
void launchQuantize(const float* x, std::int8_t* out, float* scale, std::uint32_t sources,
                    std::uint32_t features, hipStream_t stream) {
    const bool aligned = reinterpret_cast<std::uintptr_t>(x) % 16 == 0 &&
                         reinterpret_cast<std::uintptr_t>(out) % 4 == 0;
    if (!Packed && aligned && features % 4 != 0 && features >= 5 && features <= kTileFeatures &&
        !fewRows(sources, features)) {
        // Tiles of up to 16 KB, and small enough for a block per CU where there are few rows, or two or four,
        // since one block alone waits through its copy and its barriers (one, two, four: 16,384 x 50 4.7, 3.9,
        // 4.0 us; 16,384 x 127 6.2, 6.2, 5.3; narrow rows have too little work for that: 16,384 x 13 2.5,
        // 2.9, 3.3).
        const unsigned minBlocks = features < 48 ? 256u : features < 96 ? 512u : 1024u;
        unsigned rows = 256;
        while (rows > 4 && (rows * features > kTileFloats || sources / rows < minBlocks)) rows /= 2;
        const unsigned blocks = unsigned((std::size_t(sources) + rows - 1) / rows);
        const std::size_t lds = (std::size_t(rows) * features + rows + 1) * sizeof(float);
        const unsigned magic = unsigned((std::uint64_t(1) << 32) / features) + 1;
        hipLaunchKernelGGL(quantizeTile, dim3(blocks), dim3(256), lds, stream, x, out, scale, sources,
                           features, rows, magic);
    } else if (aligned && features % 4 == 0) {
        const unsigned groups = features / 4;
        const auto* xv = reinterpret_cast<const f32x4*>(x);
        auto* qv = reinterpret_cast<unsigned*>(out);
        if (groups > kWave) {
            const unsigned blocks = unsigned((std::size_t(sources) * kWave + 255) / 256);
            hipLaunchKernelGGL(quantizeRowsLong<Packed>, dim3(blocks), dim3(256), 0, stream, xv, qv,
                               scale, sources, groups);
        } else {
            unsigned lanes = 1;
            while (lanes < groups) lanes *= 2;
            const std::size_t rowsPerBlock = std::size_t(256 / lanes) * kQuantRows;
            const unsigned blocks = unsigned((sources + rowsPerBlock - 1) / rowsPerBlock);
            switch (lanes) {
#define TCC_QUANT_CASE(L)                                                                          \
    case L:                                                                                        \
        hipLaunchKernelGGL((quantizeRowsFit<L, Packed>), dim3(blocks), dim3(256), 0, stream, xv,   \
                           qv, scale, sources, groups);                                            \
        break;
                TCC_QUANT_CASE(1) TCC_QUANT_CASE(2) TCC_QUANT_CASE(4) TCC_QUANT_CASE(8)
                TCC_QUANT_CASE(16) TCC_QUANT_CASE(32) TCC_QUANT_CASE(64)
#undef TCC_QUANT_CASE
            }
        }
    } else {
        const unsigned blocks = unsigned((std::size_t(sources) + kRowsPerBlock - 1) / kRowsPerBlock);
        hipLaunchKernelGGL(quantizeRows<Packed>, dim3(blocks), dim3(kWave * kRowsPerBlock), 0,
                           stream, x, out, scale, sources, features);
    }
    checkHip(hipGetLastError());
}

} // namespace

void quantizeFeaturesInt8(const float* x, std::int8_t* q, float* scale, std::uint32_t sources,
                          std::uint32_t features, hipStream_t stream) {
    // A zero-sized grid is a launch error, reported like the runtime would (std::runtime_error).
    if (!sources || !features) throw std::runtime_error("quantize: invalid configuration argument");
    // A null buffer would fault the GPU; rejected before any launch (the reference does not check).
    if (!x || !q || !scale) throw std::invalid_argument("quantize: null device buffer");
    launchQuantize<false>(x, q, scale, sources, features, stream);
}

void quantizePackFeaturesInt8(const float* x, std::int8_t* packed, float* scale,
                              std::uint32_t sources, std::uint32_t features, hipStream_t stream) {
    if (!sources || !features) throw std::runtime_error("quantize: invalid configuration argument");
    if (features % 16) throw std::invalid_argument("packed16 needs features % 16 == 0");
    if (!x || !packed || !scale) throw std::invalid_argument("quantize-pack: null device buffer");
    launchQuantize<true>(x, packed, scale, sources, features, stream);
}

void packFeaturesInt8x16(const std::int8_t* q, std::int8_t* packed, std::uint32_t sources,
                         std::uint32_t features, hipStream_t stream) {
    if (!sources || !features) throw std::runtime_error("pack: invalid configuration argument");
    if (features % 16) throw std::invalid_argument("packed16 needs features % 16 == 0");
    if (!q || !packed) throw std::invalid_argument("pack: null device buffer");
    const std::size_t bytes = std::size_t(sources) * features;
    const bool aligned = (reinterpret_cast<std::uintptr_t>(q) % 16 == 0) &&
                         (reinterpret_cast<std::uintptr_t>(packed) % 16 == 0);
    if (aligned) {
        const std::size_t tiles = bytes / 16;
        const std::size_t blocks = (tiles + 255) / 256;
        hipLaunchKernelGGL(packTiles, dim3(unsigned(blocks)), dim3(256), 0, stream,
                           reinterpret_cast<const u32x4*>(q), reinterpret_cast<u32x4*>(packed),
                           tiles);
    } else {
        const std::size_t pairs = bytes / 2;
        const std::size_t blocks = (pairs + 255) / 256;
        hipLaunchKernelGGL(packPairs, dim3(unsigned(blocks)), dim3(256), 0, stream,
                           reinterpret_cast<const std::uint8_t*>(q),
                           reinterpret_cast<unsigned short*>(packed), pairs);
    }
    checkHip(hipGetLastError());
}
