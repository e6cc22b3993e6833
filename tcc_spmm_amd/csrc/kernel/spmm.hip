// Fused INT8-dequantization SpMM for MI355X (gfx950, wave64): Y = A x tf32(dequant(X)).
//
// Work decomposition
//   One workgroup per task (one Sw32Task: <= 384 panels of one 32-row SW), one wavefront on large
//   plans; each XCD walks a contiguous range of the task list (xcdTask), balanced by panels when skewed,
//   the range's last 512 tasks longest size class first (tailTask).
//   The wave walks the task's panels once, in order, and accumulates all 32 rows x F features of
//   the SW, two panels at a time: four v_mfma_f32_32x32x16_f16 per pair and 128-feature slice (one per
//   32-feature block; M = features, N = the 32 rows, K = the pair's 16 slots) into 4 x 16 FP32
//   accumulators per slice. F256 runs both slices in the same wave, so the A side of a pair is loaded
//   and built once. Plans with few tasks for the chip take two, four or eight waves per task instead
//   (taskWaves), each walking its share of the pairs; the write-back adds their accumulators (writeTask).
//
// Operands of one pair (walkPairs; the 64-bit-addressed instances build the same ones in walkPanels)
//   A (features x slots): the 8 slot rows of each panel's X slice are gathered with one 16-byte load per
//   lane (lane L: 16-byte tile L & 7 of slot L >> 3) into LDS as [slot][128 bytes]. Lane l then reads
//   dword l & 31 of slots 4h..4h+3 (h = l >> 5): byte b of that dword is block b's feature for M index
//   l & 31, so each lane dequantizes 16 bytes (4 slots x 4 blocks) a panel, with the four slots' scale
//   mantissas read from LDS as one 16-byte broadcast.
//   B (slots x rows): an LDS table of f16 A values; lane l reads row l & 31, slots 4h..4h+3 of both
//   panels. Rows of row groups a panel's bucket does not touch hold 0.
//   Each operand takes its four values from the first panel and then four from the second.
//   D: lane l holds row l & 31 and, per block, M indices 8i + 4h + j (register 4i + j).
//
// Exact TF32 products in f16. With the slot's scale written s = m * 2^e (m in [0.5, 1)),
// x_hat = tf32(fp32(q * s)) = tf32(fp32(q * m)) * 2^e exactly whenever s is normal, and
// x~ = tf32(fp32(q * m)) lies in [0.5, 127]: eleven significant bits. The factor 2^e moves into B:
// a' = tf32(a) * 2^(e + kShift), also eleven bits, exact in f16 when in f16's normal range (kShift
// keeps the usual A values there). A takes x~ * 2^-kXShift (kXShift = kShift + 1), which stays in
// [2^-12, 2^-4): still eleven bits in f16's normal range. The MFMA thus sums exact products
// a' * x~ * 2^-kXShift = tf32(a) * x_hat / 2 in FP32, so any accumulation order reproduces the
// reference's products, and the task doubles its accumulators at the end (exact). The accumulators
// hold Y / 2, never a scaled-up Y, so no sum overflows where the reference's stays finite. TF32
// rounding (ties away from zero) is "add 0x1000 to the FP32 pattern, truncate", and the truncation is
// the round-toward-zero f16 conversion. A panel whose a' leaves f16's normal range (or whose scale
// is subnormal) takes an FP32 path with the same products: v_mfma_f32_32x32x2_f32 on tf32(a) / 2 and
// the TF32 features. (Halving a value below 2^-125 rounds it, an error far below the tolerance.)
//
// The walk is a software pipeline over pairs: metadata two pairs ahead, A values, scales and X one,
// the X rows as loads to LDS. F128 runs four waves per SIMD (128 registers each, accumulators included),
// F256 two.
//
// Split SWs (reference src/kernel/spmm_kernel.cuh:228-282): a split task stores its row groups of
// `task.mask` as 8-row partial tiles [tile][8][F]; one lane then publishes them with one agent-scope
// release fence and takes, per slice, a relaxed wrapping ticket on counters[sw * (F/128) + slice] with
// limit chunks - 1, so the counter returns to zero by itself; the task whose ticket is chunks - 1, after
// an acquire fence, merges all partial tiles of the SW's slice in partialIds order starting from 0.0f
// and writes Y. No float atomics, no spin-waits.
#include "spmm.h"
#include "hip_support.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <mutex>
#include <stdexcept>
#include <string>
#include <type_traits>
#include <utility>

// A 4-byte load from a structured buffer (address = base + index x stride + offsets, range-checked
// by index): the LLVM intrinsic behind the raw-buffer builtins, declared by its name since clang
// has no builtin for the structured form.
__device__ float structLoadF32(__amdgpu_buffer_rsrc_t rsrc, int index, int voffset, int soffset, int aux)
    __asm("llvm.amdgcn.struct.ptr.buffer.load.f32");

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef __fp16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr unsigned kWave = 64;
constexpr unsigned kSlice = 128;
constexpr unsigned kNoPartial = 0xFFFFFFFFu;
constexpr int kShift = 10;
constexpr int kXShift = kShift + 1;
// Buffer cache policy of the A stream (sourceIds, sourceMetadata, values): the default. The
// nontemporal hint (2) was measured to raise L2 misses of the gathered X rows by about 1.5 GB per
// c3 F128 launch.
constexpr int kNt = 0;

// TF32 rounding from its definition: keep 10 explicit mantissa bits, round to nearest with ties
// away from zero (adding half an ulp to the sign-magnitude encoding), carry into the exponent.
// Operands here are always finite (the format rejects non-finite A values; X is finite INT8 times a
// finite scale).
__device__ __forceinline__ float roundTf32(float v) {
    return __uint_as_float((__float_as_uint(v) + 0x1000u) & 0xFFFFE000u);
}

// f(0), ..., f(N - 1), the index a constant.
template <class F, unsigned... I>
__device__ __forceinline__ void forEachIndex(std::integer_sequence<unsigned, I...>, F f) {
    (f(std::integral_constant<unsigned, I>{}), ...);
}
template <unsigned N, class F>
__device__ __forceinline__ void forEachIndex(F f) {
    forEachIndex(std::make_integer_sequence<unsigned, N>{}, f);
}

struct KernelArgs {
    Sw32DeviceView m;
    const std::int8_t* packedX;
    const float* scales;
    float* y;
    float* partials;
    unsigned* counters;
    unsigned rows, cols;
    unsigned resident; // the whole grid runs at once (launch): tasks in list order
    unsigned vec4; // y and partials are 16-byte aligned: stores and merge loads of 16 bytes
#ifdef TCC_SPMM_TIMELINE
    unsigned long long* stamps; // measurement build only: [taskCount][4], see TaskClock
#endif
};

// sw32BucketOrder (include/format/sw32.h) packed four bits per bucket slot: slot t's row-group mask
// is nibble t of this constant.
constexpr std::uint64_t kBucketGroups = 0xFEDCBA9765384210ull;

// ------------------------------------------------------------------------------------------------
// Memory access of one task. Narrow (the packed X slice and the scales addressable with 32-bit
// byte offsets, the usual case): buffer loads. sourceIds, sourceMetadata and values use a per-task
// base (offsets stay below 1 MiB); scales and X use buffers sized from `cols`, so the padding
// sentinel source UINT32_MAX lands out of range and reads 0 without a clamp, and an absent A entry
// reads 0 through an out-of-range offset. Wide: 64-bit global loads with clamped indices.
// Wide with 2-byte tiles: the same, for a packed X that is u16- but not 16-byte aligned (the
// reference's own requirement, include/format/int8_features.cuh:11-13): each 16-byte tile is read
// as eight naturally aligned u16 loads, which never touch a byte outside the tile.

struct Meta {        // one panel
    unsigned id;     // lane L: source of slot L & 7
    unsigned mask;   // lane L: row mask of slot L & 7
    unsigned base;   // lane L: value base of slot L & 7
};

// Lane L's value of v from lane srcLane (LDS crossbar, no memory access).
__device__ __forceinline__ unsigned lanePermute(unsigned v, unsigned srcLane) {
    return unsigned(__builtin_amdgcn_ds_bpermute(int(srcLane * 4), int(v)));
}

// Metadata of panels q and q + 1 loaded together: lane L holds slot L & 7 of panel
// q + ((L >> 3) & 1), lanes 16..63 repeating lanes 0..15.
struct MetaPair {
    unsigned id, mask, base;
};

// Addressing modes of the X and A-stream loads, chosen per launch on the host.
enum : unsigned { kBuffer = 0, kGlobal = 1, kGlobalU16 = 2 };

template <unsigned Addr>
struct Loader;

template <>
struct Loader<kBuffer> {
    static constexpr bool kWide = false;
    __amdgpu_buffer_rsrc_t ids, meta, scales, x, vals;
    const float* values; // of the whole matrix
    unsigned first;     // the wave's first panel: panel offsets are relative to it
    unsigned vbase;     // value base of the wave's first slot, the smallest of the wave
    unsigned xShift;    // log2(features)

    __device__ Loader(const KernelArgs& a, unsigned begin, unsigned end, unsigned features)
        : values(a.m.values), first(begin), vbase(0), xShift(features == 256 ? 8u : 7u) {
        const std::size_t slot0 = std::size_t(begin) * 8;
        // Sized to the panels [begin, end): a pair's second panel past the end reads 0 (source 0, no
        // entries) without a clamp.
        ids = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned*>(a.m.sourceIds + slot0), 0,
                                                (end - begin) * 32u, 0x00020000);
        meta = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<std::uint64_t*>(a.m.sourceMetadata + slot0), 0, (end - begin) * 64u, 0x00020000);
        rebase(0);
        scales = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.scales), 4, a.cols, 0x00020000);
        x = __builtin_amdgcn_make_buffer_rsrc(const_cast<std::int8_t*>(a.packedX), 0,
                                              a.cols << xShift, 0x00020000);
    }
    // Addresses the values from value base `base` on.
    __device__ void rebase(unsigned base) {
        vbase = base;
        vals = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(values + base), 4, 0x7FFFFFF0,
                                                 0x00020000);
    }
    // Before the first value loads; `m` is the metadata of the wave's first panel. Value bases grow in
    // slot order (reference src/format/sw32.cpp:131-138) and every panel starts with a real slot, so
    // that panel's first slot (lane 0) has the smallest base. It comes with the metadata the walk loads
    // anyway; a load of its own would be one more dependent load before the first panel.
    __device__ void startTask(const Meta& m) { rebase(__builtin_amdgcn_readfirstlane(m.base)); }
    // Panel `panel`, clamped to `last` (the offset is scalar).
    __device__ Meta meta8(unsigned panel, unsigned last, unsigned lane) const {
        const int off = int((min(panel, last) - first) * 32u);
        const auto md = __builtin_amdgcn_raw_buffer_load_b64(meta, (lane & 7) * 8, 2 * off, kNt);
        return {__builtin_amdgcn_raw_buffer_load_b32(ids, (lane & 7) * 4, off, kNt), md[0], md[1]};
    }
    // Panels q (clamped to `last`) and q + 1: one load per array for both. The range check counts the
    // scalar offset.
    __device__ MetaPair meta2(unsigned q, unsigned last, unsigned lane) const {
        const int off = int((min(q, last) - first) * 32u);
        const auto md = __builtin_amdgcn_raw_buffer_load_b64(meta, (lane & 15) * 8, 2 * off, kNt);
        return {__builtin_amdgcn_raw_buffer_load_b32(ids, (lane & 15) * 4, off, kNt), md[0], md[1]};
    }
    // scales and values are structured buffers of 4-byte records, addressed by index (no shift) and
    // range-checked by index: an index past the records reads 0.
    __device__ float scale(unsigned src) const { return structLoadF32(scales, int(src), 0, 0, 0); }
    // values[idx] when `present`, else 0.
    __device__ float value(unsigned idx, bool present) const {
        return structLoadF32(vals, int(present ? idx - vbase : 0xFFFFFFFFu), 0, 0, kNt);
    }
    // 16-byte tile `lane & 7` of slice k of the packed X row of `src`. The slice offset goes in the
    // scalar offset, so both slices of a row share one per-lane offset (one VALU instruction fewer
    // per F256 panel).
    __device__ u32x4 tile(unsigned src, unsigned lane, unsigned k) const {
        return __builtin_amdgcn_raw_buffer_load_b128(x, (src << xShift) + 16 * (lane & 7), kSlice * k, 0);
    }
};

template <unsigned Addr>
struct Loader {
    static_assert(Addr == kGlobal || Addr == kGlobalU16, "64-bit addressing modes");
    static constexpr bool kWide = true;
    const KernelArgs* a;
    // Uniform bases, so that a load takes a scalar base and a 32-bit lane offset.
    const unsigned* ids;       // of the wave's first panel
    const std::uint64_t* meta;
    const float* vals;         // from value base vbase on
    unsigned first, vbase, features; // first, vbase: as in the buffer loader

    __device__ Loader(const KernelArgs& args, unsigned begin, unsigned, unsigned f)
        : a(&args), ids(args.m.sourceIds + std::size_t(begin) * 8),
          meta(args.m.sourceMetadata + std::size_t(begin) * 8), vals(args.m.values), first(begin),
          vbase(0), features(f) {}
    __device__ void startTask(const Meta& m) {
        vbase = __builtin_amdgcn_readfirstlane(m.base);
        vals = a->m.values + vbase;
    }
    // Panel `panel`, clamped to `last`.
    __device__ Meta meta8(unsigned panel, unsigned last, unsigned lane) const {
        const unsigned s = (min(panel, last) - first) * 8 + (lane & 7);
        const std::uint64_t md = __builtin_nontemporal_load(meta + s);
        return {__builtin_nontemporal_load(ids + s), unsigned(md), unsigned(md >> 32)};
    }
    __device__ float scale(unsigned src) const { return a->scales[min(src, a->cols - 1)]; }
    // values[idx] when `present`, else some value (absent entries are masked by Stage::bits).
    __device__ float value(unsigned idx, bool present) const {
        return __builtin_nontemporal_load(vals + (present ? idx - vbase : 0u));
    }
    __device__ u32x4 tile(unsigned src, unsigned lane, unsigned k) const {
        const std::int8_t* p =
            a->packedX + std::size_t(min(src, a->cols - 1)) * features + 16 * (lane & 7) + kSlice * k;
        if constexpr (Addr == kGlobalU16) {
            const unsigned short* h = reinterpret_cast<const unsigned short*>(p);
            u32x4 t;
#pragma unroll
            for (unsigned i = 0; i < 4; ++i) t[i] = unsigned(h[2 * i]) | (unsigned(h[2 * i + 1]) << 16);
            return t;
        } else {
            return *reinterpret_cast<const u32x4*>(p);
        }
    }
};

// One panel of walkPanels or of the FP32 pass, ready to compute. Panel kinds: exclusive (a bucket of one
// row group g, known per panel from the bucket bounds; walkPanels only) and shared (a bucket of several row
// groups, `groups`, or any panel taken as one).
struct Stage {
    float scale;   // lane L: scale of slot L & 7
    float v[4];    // lane L: raw A value of (slot L & 7, row 8g + (L >> 3)); v[0] when exclusive
    unsigned bits; // bit g: that entry is present (wide loader only; narrow reads 0 instead)
    u32x4 x[2];    // 16-byte tile L & 7 of the X row of slot L >> 3, per slice of the wave
};

// Loads one panel (exclusive: lane L's row bit in the slot masks, 1 << (8g + (L >> 3)), in `rowBit`;
// shared: row groups `groups`), with the X tiles of the wave's S slices.
template <bool Shared, unsigned S, class Ld>
__device__ __forceinline__ void loadStage(const Ld& ld, const Meta& m, unsigned rowBit,
                                          unsigned groups, unsigned lane, Stage& s) {
    // Padding slots (source UINT32_MAX, metadata 0) have an empty row mask; their scale and X tile
    // read 0 (narrow) or a clamped row (wide), multiplied by A entries that are all 0.
    s.scale = ld.scale(m.id);
    s.bits = 0;
    constexpr unsigned kCount = Shared ? 4 : 1;
#pragma unroll
    for (unsigned j = 0; j < kCount; ++j) {
        const unsigned at = Shared ? 1u << (j * 8 + (lane >> 3)) : rowBit;
        const bool present = (m.mask & at) != 0 && (!Shared || ((groups >> j) & 1u));
        // The k-th set row bit of a slot owns values[base + k].
        const unsigned idx = m.base + __popc(m.mask & (at - 1u));
        s.v[j] = ld.value(idx, present);
        if constexpr (Ld::kWide) s.bits |= unsigned(present) << j;
    }
    // Lane L gathers slot L >> 3's row, whose source lane L >> 3 holds: a cross-lane permute instead
    // of a second sourceIds load (one vector memory instruction fewer per panel, 2% at c3 F128).
    const unsigned gather = lanePermute(m.id, lane >> 3);
#pragma unroll
    for (unsigned k = 0; k < S; ++k) s.x[k] = ld.tile(gather, lane, k);
}

// ------------------------------------------------------------------------------------------------
// Compute

// Block B of the lane's four slots: byte B of d0..d3 (slots 4h + 0..3) sign-extended to FP32 by
// SDWA conversions, then multiplied by the slots' scale mantissas (plain multiplies: a DPP operand
// would cost about twice the issue time of each multiply).
template <unsigned B>
__device__ __forceinline__ void scaleBlock(unsigned d0, unsigned d1, unsigned d2, unsigned d3,
                                           const f32x4& mant, float (&q)[4]) {
    const unsigned d[4] = {d0, d1, d2, d3};
#pragma unroll
    for (unsigned i = 0; i < 4; ++i)
        q[i] = float(static_cast<signed char>(d[i] >> (8 * B))) * mant[i];
}

// TF32-round two values and pack them as f16 (round toward zero after adding half an ulp). Both
// half-ulp additions are one 64-bit add on the pair's patterns: no carry crosses from the low value
// into the high one, since a finite FP32 pattern plus 0x1000 stays below 2^32 (only patterns at or
// above 0xFFFFF000, negative NaNs, would carry). One v_lshl_add_u64 instead of two v_add_u32.
__device__ __forceinline__ f16x2 roundPack(float a, float b) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    const unsigned long long both =
        __builtin_bit_cast(unsigned long long, f32x2{a, b}) + 0x0000100000001000ull;
    const f32x2 r = __builtin_bit_cast(f32x2, both);
    return __builtin_amdgcn_cvt_pkrtz(r[0], r[1]);
}

// LDS handoff between the lanes of one wave: a wave's LDS operations execute in order, so only the
// compiler has to be kept from moving memory accesses across this point.
__device__ __forceinline__ void waveSync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct Lds {
    _Float16* table16; // a' (f16 path), two areas (tableEntry)
    float* table32;    // [32 rows][8 slots] tf32(a) / 2 (FP32 path)
    u32x4* xtile;      // X rows: xTile, or the ring of walkPairs
    float* mant;       // [2 areas][8 slots] scale mantissas of a panel
    unsigned short* redo; // [384]: offsets (from the wave's first panel) of the panels that need
                          // the FP32 path, in the order found (a task has <= 384 panels)
};

// Entry j of a stage as tf32(a) (0 when absent).
template <bool Wide>
__device__ __forceinline__ float stageTf32(const Stage& s, unsigned j) {
    return (Wide && !((s.bits >> j) & 1u)) ? 0.0f : roundTf32(s.v[j]); // tf32(0) = 0
}

// m * 2^-kXShift for a scale s = m * 2^e (m in [0.5, 1)): the sign and mantissa bits of s under the
// biased exponent 126 - kXShift. One v_and_or_b32 (as cheap as a v_frexp_mant); a VOP3 takes no
// literal and one scalar operand on gfx950, so the caller keeps the mask 0x807FFFFF in a VGPR
// (`keep`) and the exponent bits come from an SGPR.
__device__ __forceinline__ float shiftedMantissa(float s, unsigned keep) {
    unsigned r;
    asm("v_and_or_b32 %0, %1, %2, %3"
        : "=v"(r)
        : "v"(__float_as_uint(s)), "v"(keep), "s"(unsigned(126 - kXShift) << 23));
    return __uint_as_float(r);
}

// The lane's row and half of the MFMA operands, m = lane & 31 and h = lane >> 5, computed once per
// task (opaquely, so that the register allocator keeps them rather than recomputing them per panel).
struct LaneMh {
    unsigned m, h;
};

// Lanes whose value is a normal f16 (class bits 3 and 8: -normal, +normal), as a wave mask. The
// comparison writes the mask straight into an SGPR pair; through the class builtin the compiler
// moved the result through a VGPR and compared it again.
__device__ __forceinline__ std::uint64_t normalF16(_Float16 v) {
    std::uint64_t mask;
    asm("v_cmp_class_f16_e64 %0, %1, %2" : "=s"(mask) : "v"(v), "s"(0x108u));
    return mask;
}

__device__ __forceinline__ f16x8 join(f16x4 lo, f16x4 hi) {
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

// A panel is computed in two parts. Its operands are written to LDS area 0 or 1 (stagePanel, or for a
// pair at once walkPairs): the f16 A table, the X tiles and the scale mantissas. They are read back, the
// X blocks dequantized and multiplied, over one area (one v_mfma_f32_32x32x8_f16 per 32-feature block) or
// both (one v_mfma_f32_32x32x16_f16 per block, K = the 16 slots of two panels: lane half h holds
// k = 8h + j, j < 4 area 0's slot 4h + j and j >= 4 area 1's slot 4h + j - 4, in both operands, so
// each MFMA adds both panels' products). Pairs take half the MFMAs, and half the matrix-core time.
//
// Table layout: [32 rows][2 halves][2 areas][4 slots], so that the entries of row m and slots
// 4h .. 4h + 3 are 8 contiguous bytes per area and 16 for both, from f16 index 8 (2m + h) on. Here: the
// entry of slot L & 7 of row 8g + (L >> 3) of row group g.
__device__ __forceinline__ unsigned tableEntry(unsigned g, unsigned lane, unsigned area) {
    const unsigned row = 8 * g + (lane >> 3), slot = lane & 7;
    return ((row * 2 + (slot >> 2)) * 2 + area) * 4 + (slot & 3);
}

// X tiles in LDS of walkPanels and the FP32 pass: [8 slots][2 S blocks][128 bytes], block S * area +
// slice. Returns the 16-byte index of the first tile of (slot, block).
template <unsigned S>
__device__ __forceinline__ unsigned xTile(unsigned slot, unsigned block) {
    return (slot * 2 * S + block) * 8;
}

// Writes panel `s` to LDS area `area`. Per lane: slot lane & 7, row lane >> 3 of each row group; an
// exclusive panel writes only its own row group, whose table entry of this lane is `entry` (the
// other groups' entries hold 0). Returns whether every entry of the panel has an exact f16 a'
// (wave-uniform); if not, its table is all zero, so the panel contributes nothing here.
template <bool Shared, unsigned S>
__device__ __forceinline__ bool stagePanel(const Stage& s, unsigned lane, const Lds& lds, unsigned area,
                                           unsigned entry, unsigned keep) {
    // 2^(e + kShift) for the slot's scale s = m * 2^e (m in [0.5, 1)): its exponent bits alone are
    // 2^(e - 1). A zero or subnormal scale gives 0 and an infinite or NaN one inf, so that every
    // nonzero entry of such a slot fails the check below and the panel takes the FP32 path (the
    // mantissa trick needs a normal scale; there q x inf is inf or NaN, as in the reference).
    const float pow2 = __builtin_amdgcn_ldexpf(__uint_as_float(__float_as_uint(s.scale) & 0x7F800000u),
                                               kShift + 1);
    std::uint64_t inexact = 0; // lanes with an entry that has no exact f16 a'
    constexpr unsigned kCount = Shared ? 4 : 1;
    _Float16 ap[kCount];
#pragma unroll
    for (unsigned j = 0; j < kCount; ++j) {
        const float at = stageTf32<true>(s, j);
        // a' = at x pow2 has at most eleven significant bits, so it is exact in f16 exactly when
        // its conversion is a normal f16: [2^-14, 65504]; larger values (inf included) convert to
        // inf, smaller ones to subnormals or zero. (A product that lands in that range is a normal
        // FP32 value, so the multiply itself was exact.) Masks of comparisons combine as scalar
        // operations.
        ap[j] = static_cast<_Float16>(at * pow2);
        const std::uint64_t nonzero = __builtin_amdgcn_ballot_w64(at != 0.0f);
        inexact |= nonzero & ~normalF16(ap[j]);
    }
    // A panel without exact f16 operands still runs its MFMAs (straight-line accumulators), on an
    // all-zero table; the FP32 pass adds it later.
    const bool useF16 = inexact == 0;
#pragma unroll
    for (unsigned j = 0; j < kCount; ++j)
        lds.table16[Shared ? tableEntry(j, lane, area) : entry] =
            useF16 ? ap[j] : static_cast<_Float16>(0.0f);
#pragma unroll
    for (unsigned k = 0; k < S; ++k) lds.xtile[xTile<S>(lane >> 3, S * area + k) + (lane & 7)] = s.x[k];
    // Lane L holds slot L & 7's scale; lanes of half h read the mantissas of slots 4h .. 4h + 3,
    // stored as m * 2^-kXShift. For a scale that is not normal the bits are not that, but such a
    // panel's table is all zero (pow2 above) and the FP32 pass computes it.
    lds.mant[8 * area + (lane & 7)] = shiftedMantissa(s.scale, keep);
    return useF16;
}

// Dequantized block B (bytes B of the lane's four X dwords) of one area, as f16 x~ * 2^-kXShift.
template <unsigned B>
__device__ __forceinline__ f16x4 dequantBlock(const unsigned (&d)[4], const f32x4& mant) {
    float q[4];
    scaleBlock<B>(d[0], d[1], d[2], d[3], mant, q);
    return __builtin_bit_cast(
        f16x4, __builtin_shufflevector(roundPack(q[0], q[1]), roundPack(q[2], q[3]), 0, 1, 2, 3));
}

// A lane's operands of one panel (Areas == 1) or of a pair of panels (2), read back from LDS: the X dwords
// of its four slots, their mantissas, and its row's A entries.
template <unsigned S, unsigned Areas>
struct Operands {
    unsigned d[Areas][S][4];
    f32x4 mant[Areas];
    std::conditional_t<Areas == 1, f16x4, f16x8> b;
};

// The MFMAs of one panel or of a pair. The S x 4 blocks are dequantized one ahead of their MFMAs: block
// i + 1's conversions run between block i's last pack and its MFMA, so the MFMA's operand was written
// a dozen VALU instructions before it is read and needs no wait states.
template <unsigned S, unsigned Areas>
__device__ __forceinline__ void multiply(const Operands<S, Areas>& o, f32x16 (&acc)[4 * S]) {
    using I0 = std::integral_constant<unsigned, 0>;
    using I1 = std::integral_constant<unsigned, 1>;
    using I2 = std::integral_constant<unsigned, 2>;
    using I3 = std::integral_constant<unsigned, 3>;
    auto op = [&](auto blk, unsigned k) {
        constexpr unsigned B = decltype(blk)::value;
        if constexpr (Areas == 2)
            return join(dequantBlock<B>(o.d[0][k], o.mant[0]), dequantBlock<B>(o.d[1][k], o.mant[1]));
        else
            return dequantBlock<B>(o.d[0][k], o.mant[0]);
    };
    auto mfma = [&](unsigned t, auto x) {
        if constexpr (Areas == 2)
            acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x, o.b, acc[t], 0, 0, 0);
        else
            acc[t] = __builtin_amdgcn_mfma_f32_32x32x8f16(x, o.b, acc[t], 0, 0, 0);
    };
    auto av = op(I0{}, 0);
#pragma unroll
    for (unsigned k = 0; k < S; ++k) {
        auto nx = op(I1{}, k);
        mfma(4 * k + 0, av);
        av = op(I2{}, k);
        mfma(4 * k + 1, nx);
        nx = op(I3{}, k);
        mfma(4 * k + 2, av);
        if (k + 1 < S) av = op(I0{}, k + 1);
        mfma(4 * k + 3, nx);
    }
}

// Reads the operands of area First, or of both areas (Areas == 2), and multiplies.
template <unsigned S, unsigned Areas, unsigned First = 0>
__device__ __forceinline__ void crunch(const Lds& lds, f32x16 (&acc)[4 * S], LaneMh mh) {
    waveSync();
    const unsigned m = mh.m, h = mh.h;
    Operands<S, Areas> o;
#pragma unroll
    for (unsigned r = 0; r < Areas; ++r) {
        o.mant[r] = reinterpret_cast<const f32x4*>(lds.mant + 8 * (First + r))[h];
#pragma unroll
        for (unsigned k = 0; k < S; ++k) {
            const unsigned* xw = reinterpret_cast<const unsigned*>(lds.xtile) + m;
#pragma unroll
            for (unsigned i = 0; i < 4; ++i) o.d[r][k][i] = xw[4 * xTile<S>(4 * h + i, S * (First + r) + k)];
        }
    }
    if constexpr (Areas == 2)
        o.b = reinterpret_cast<const f16x8*>(lds.table16)[m * 2 + h];
    else
        o.b = reinterpret_cast<const f16x4*>(lds.table16)[(m * 2 + h) * 2 + First];
    multiply<S, Areas>(o, acc);
    waveSync();
}

// A shared-kind panel with exact FP32 operands (v_mfma_f32_32x32x2_f32): K = 2 steps over slot
// pairs (2j, 2j + 1), lane half h taking slot 2j + h, whose scale comes from lane 2j + h. The
// products are tf32(a) / 2 * x_hat, on the accumulators' Y / 2 scale.
template <bool Wide, unsigned S>
__device__ __forceinline__ void computePanelF32(const Stage& s, unsigned groups, unsigned lane,
                                                const Lds& lds, f32x16 (&acc)[4 * S]) {
#pragma unroll
    for (unsigned g = 0; g < 4; ++g)
        lds.table32[64 * g + lane] = ((groups >> g) & 1u) ? 0.5f * stageTf32<Wide>(s, g) : 0.0f;
#pragma unroll
    for (unsigned k = 0; k < S; ++k) lds.xtile[xTile<S>(lane >> 3, k) + (lane & 7)] = s.x[k];
    waveSync();
    const unsigned m = lane & 31, h = lane >> 5;
#pragma unroll
    for (unsigned j = 0; j < 4; ++j) {
        const unsigned slot = 2 * j + h;
        const float sc =
            __int_as_float(__builtin_amdgcn_ds_bpermute(int(slot * 4), __float_as_int(s.scale)));
        const float b = lds.table32[m * 8 + slot];
#pragma unroll
        for (unsigned k = 0; k < S; ++k) {
            const unsigned d = (reinterpret_cast<const unsigned*>(lds.xtile) + m)[4 * xTile<S>(slot, k)];
#pragma unroll
            for (unsigned blk = 0; blk < 4; ++blk) {
                const float x = roundTf32(float(int(d << (24 - 8 * blk)) >> 24) * sc);
                acc[4 * k + blk] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, b, acc[4 * k + blk], 0, 0, 0);
            }
        }
    }
    waveSync();
}

// ------------------------------------------------------------------------------------------------
// Panel walk

// Ends of the exclusive buckets of row groups 0..2 (group 3's is the end of the walk), and the first and
// the end of the first shared bucket: loaded together, before the walk.
struct GroupBounds {
    unsigned b0, b1, b2, shared, sharedEnd;
    __device__ unsigned end(unsigned g) const {
        return g == 0 ? b0 : g == 1 ? b1 : g == 2 ? b2 : 0xFFFFFFFFu;
    }
    // Row group of panel p (the ends do not decrease).
    __device__ unsigned of(unsigned p) const {
        return unsigned(p >= b0) + unsigned(p >= b1) + unsigned(p >= b2);
    }
    // Row groups of a mixed walk's first panel p, the only one of it that may be exclusive.
    template <class Cursor>
    __device__ unsigned firstGroups(Cursor& bucket, unsigned p) const {
        return p < shared ? 1u << of(p) : bucket.groups(p);
    }
};

// Row groups of the panels of one task from the first shared one on, walked in increasing panel order
// (bucket slot t covers [bucketOffsets[t], bucketOffsets[t + 1]) of the SW). `groups(p)` must be asked
// for non-decreasing p. A load for each bucket passed (empty ones too), which the wave waits for with every
// load in flight; none for the first bucket.
struct BucketCursor {
    const unsigned* offsets; // bucketOffsets of the SW (17 entries)
    unsigned t, end;         // current bucket slot and its end panel

    __device__ BucketCursor(const unsigned* bucketOffsets, const GroupBounds& b)
        : offsets(bucketOffsets), t(5), end(b.sharedEnd) {}
    __device__ unsigned groups(unsigned p) {
        while (p >= end) {
            ++t;
            end = offsets[t + 1];
        }
        return unsigned(kBucketGroups >> (4 * t)) & 15u;
    }
};

// Row groups of panel p found from scratch (the FP32 path visits few panels).
__device__ __forceinline__ unsigned groupsOf(const unsigned* offsets, unsigned p) {
    unsigned t = 1;
    while (p >= offsets[t + 1]) ++t;
    return unsigned(kBucketGroups >> (4 * t)) & 15u;
}

struct TaskWalk {
    const unsigned* offsets; // bucketOffsets of the SW
    unsigned begin, end;     // the task's panels
    unsigned lane;
    Lds lds;
    unsigned redoCount;      // entries in lds.redo
    unsigned keep;           // 0x807FFFFF in a VGPR, for shiftedMantissa
    LaneMh mh;
};

// Queues panel `panel` for the FP32 pass when `redo` (wave-uniform) is set. The branch is taken only
// for panels whose operands do not fit f16, so the common path costs one scalar branch; the queue
// length lives in a scalar register.
__device__ __forceinline__ void flagRedo(TaskWalk& w, unsigned panel, bool redo) {
    if (__builtin_expect(redo, 0)) { // wave-uniform and rare
        if (w.lane == 0) w.lds.redo[w.redoCount] = static_cast<unsigned short>(panel - w.begin);
        ++w.redoCount;
    }
}

// Row group of the exclusive panels of one task, walked in increasing panel order. Wave-uniform, in
// scalar registers: a panel inside the current bucket costs one compare and an untaken branch.
struct GroupCursor {
    unsigned g, end;
    __device__ void advance(const GroupBounds& b, unsigned p) {
        g = b.of(p);
        end = b.end(g);
    }
};

// The panels [lo, hi) of the 64-bit-addressed instances, all exclusive or of any kind (Shared), in the
// pairs and with the products of walkPairs, one panel's loads and table entries at a time. `first` is
// panel lo's metadata if lo is the wave's first panel (loaded by the caller beside the bucket bounds, one
// dependent load earlier). Stage data two panels ahead, metadata four: three stage buffers rotate, at the
// step of panel i holding panels i, i + 1 and (loaded there) i + 2. Loads past the end repeat the last
// panel and are never computed.
template <bool Shared, unsigned S, class Ld>
__device__ __forceinline__ void walkPanels(Ld& ld, TaskWalk& w, const GroupBounds& bounds,
                                           unsigned lo, unsigned hi, Meta first,
                                           f32x16 (&acc)[4 * S]) {
    if (lo >= hi) return;
    const unsigned n = hi - lo, lane = w.lane, last = w.end - 1;
    // The loads' side of a bucket change: to be called before the loads of panel p, for increasing p.
    // Returns a shared panel's row groups.
    BucketCursor bucket(w.offsets, bounds);
    GroupCursor loads{0, 0};
    const unsigned bit0 = 1u << (lane >> 3);
    unsigned rowBit = 0;
    auto enter = [&](unsigned p) __attribute__((always_inline)) {
        if constexpr (Shared) return bucket.groups(min(p, last));
        if (__builtin_expect(p >= loads.end, 0)) {
            loads.advance(bounds, p);
            rowBit = bit0 << (8 * loads.g);
        }
        return 0u;
    };
    // The table's side: an area's table holds one row group at a time, the other groups' entries 0.
    GroupCursor staged[2] = {{0, 0}, {0, 0}};
    unsigned entry[2] = {tableEntry(0, lane, 0), tableEntry(0, lane, 1)};
    if constexpr (!Shared) {
#pragma unroll
        for (unsigned i = 0; i < 4; ++i)
            reinterpret_cast<f16x2*>(w.lds.table16)[64 * i + lane] = f16x2{0, 0};
    }
    auto stage = [&](const Stage& st, unsigned p, auto area) __attribute__((always_inline)) {
        constexpr unsigned A = decltype(area)::value;
        if constexpr (!Shared) {
            if (__builtin_expect(p >= staged[A].end, 0)) {
                w.lds.table16[entry[A]] = static_cast<_Float16>(0.0f);
                staged[A].advance(bounds, p);
                entry[A] = tableEntry(staged[A].g, lane, A);
            }
        }
        flagRedo(w, p, !stagePanel<Shared, S>(st, lane, w.lds, A, entry[A], w.keep));
    };
    auto computePair = [&]() __attribute__((always_inline)) {
        if constexpr (Shared && S == 1) { // as walkPairs
            crunch<S, 1, 0>(w.lds, acc, w.mh);
            crunch<S, 1, 1>(w.lds, acc, w.mh);
        } else {
            crunch<S, 2>(w.lds, acc, w.mh);
        }
    };
    using Area0 = std::integral_constant<unsigned, 0>;
    using Area1 = std::integral_constant<unsigned, 1>;
    if (lo != w.begin) first = ld.meta8(lo, lo, lane);
    const Meta next = ld.meta8(lo + 1, last, lane);
    // The steps expect m1's loads to be older than m2's (waits are counted in issue order).
    Meta m1 = ld.meta8(lo + 2, last, lane);
    __builtin_amdgcn_sched_barrier(0);
    Meta m2 = ld.meta8(lo + 3, last, lane);
    __builtin_amdgcn_sched_barrier(0);
    if (lo == w.begin) ld.startTask(first);
    Stage sa, sb, sc;
    {
        const unsigned g0 = Shared ? bounds.firstGroups(bucket, lo) : enter(lo);
        loadStage<Shared, S>(ld, first, rowBit, g0, lane, sa);
        const unsigned g1 = enter(lo + 1);
        loadStage<Shared, S>(ld, next, rowBit, g1, lane, sb);
    }
    auto step = [&](auto area, Stage& cur, Stage& ahead, unsigned panel) __attribute__((always_inline)) {
        const unsigned g = enter(panel + 2);
        loadStage<Shared, S>(ld, m1, rowBit, g, lane, ahead);
        m1 = m2;
        m2 = ld.meta8(panel + 4, last, lane);
        __builtin_amdgcn_sched_barrier(0);
        stage(cur, panel, area);
        if constexpr (decltype(area)::value == 1) computePair();
    };
    // Panels in pairs, in a loop unrolled by six (the period of both the pairs and the stage rotation),
    // then the r < 6 panels left: their pairs by the same steps and a last panel with an empty one.
    const unsigned sixes = n / 6, r = n - 6 * sixes;
    unsigned i = lo;
#pragma unroll 1
    for (unsigned k = 0; k < sixes; ++k, i += 6) {
        step(Area0{}, sa, sc, i);
        step(Area1{}, sb, sa, i + 1);
        step(Area0{}, sc, sb, i + 2);
        step(Area1{}, sa, sc, i + 3);
        step(Area0{}, sb, sa, i + 4);
        step(Area1{}, sc, sb, i + 5);
    }
    if (r >= 2) {
        step(Area0{}, sa, sc, i);
        step(Area1{}, sb, sa, i + 1);
    }
    if (r >= 4) {
        step(Area0{}, sc, sb, i + 2);
        step(Area1{}, sa, sc, i + 3);
    }
    if (r & 1) {
        const Stage odd = r == 1 ? sa : r == 3 ? sc : sb;
        stage(odd, hi - 1, Area0{});
        stagePanel<Shared, S>(Stage{}, lane, w.lds, 1, entry[1], w.keep);
        computePair();
    }
}

// ------------------------------------------------------------------------------------------------
// Panel walk of the buffer-addressed instances: two panels at a time, with the same products as
// walkPanels.
//
// Bound by VALU issue wherever the gathers do not run at the memory system's request rate, so the
// instructions per panel decide. A pair's 16 slots fill a 16-lane row: lane L holds slot L & 7 of
// panel (L >> 3) & 1 in its metadata, scale, A values (rows (L >> 4) + 4j of the row group, j = 0, 1)
// and table entries, so nothing is moved between lanes to separate the panels; the scale's work is done
// once per pair; and the pair is one v_mfma_f32_32x32x16_f16 per 32-feature block. X goes straight from
// memory to LDS (16 bytes per lane), so rows in flight take no registers and F128's pairs fit its 128.
// Against one panel at a time at F128 and pairs staged panel by panel at F256, X through registers, the two
// builds timed in turn (us; other sessions differ by a few percent): 100K rows F128 74.5 -> 65.2, 262K power
// law F128 221 -> 213, F256 361 -> 355, 2.45M rows F128 2,872 -> 2,802, F256 4,884 -> 4,761. Loads to LDS
// alone, with the rest as before, gained nothing (F128 +0.1 to +4%): with the chip full the depth of the
// gathers is not what bounds them.
//
// LDS of a wave: a ring of two pairs' X rows, [panel & 3][slice][8 slots][128 bytes] as the loads deliver
// them (lane L: 16 bytes at 16 L); the A table [32 rows][2 halves][2 panels][4 slots]; the mantissas
// [2 panels][8 slots].
//
// The compiler orders every LDS access it knows of after the last load to LDS, which would empty the
// pipeline at each pair. So the accesses of the loop (table entries, mantissas and operands) are written
// out below, and the wait in front of the operand reads is counted by hand: the loop issues its vector
// memory instructions in a fixed order (the scheduling barriers keep it), a pair's X last, and the
// kYounger of the next pair follow before it is read. Where a shared walk passes a bucket's end, the loads of
// the next buckets' bounds come in between, and waiting for them empties the pipeline. The build checks the
// count on every path of the compiled kernels.

__device__ __forceinline__ unsigned ldsAddress(const void* p) {
    return unsigned(reinterpret_cast<std::uintptr_t>(
        (const __attribute__((address_space(3))) void*)p));
}

// Row groups of the pairs of an exclusive walk, in scalar registers: a pair inside one bucket costs a
// compare and an untaken branch.
struct PairCursor {
    unsigned g = 0, second = 0; // row groups of the pair's panels
    unsigned limit = 0;         // pairs whose second panel lies before it need no update
    __device__ bool changes(unsigned p) const { return __builtin_expect(p + 1 >= limit, 0); }
    __device__ void update(const GroupBounds& b, unsigned p) {
        g = b.of(p);
        second = b.of(p + 1);
        limit = second == g ? b.end(g) : 0u;
    }
};

// The lane's LDS byte addresses: its X dwords in ring slot 0, and its mantissas.
struct LaneLds {
    unsigned x, tableRead, mantWrite, mantRead;
};

// Waits until at most Younger vector memory instructions are outstanding, then reads a pair's operands
// (X from LDS address x).
template <unsigned S, unsigned Younger>
__device__ __forceinline__ void readPair(Operands<S, 2>& o, const LaneLds& at, unsigned x) {
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    auto put = [&](unsigned r, unsigned k, u32x2 lo, u32x2 hi) {
        o.d[r][k][0] = lo[0];
        o.d[r][k][1] = lo[1];
        o.d[r][k][2] = hi[0];
        o.d[r][k][3] = hi[1];
    };
    u32x2 a, b;
    if constexpr (S == 1) { // one address: the second panel's rows lie past the reach of two-address reads
        asm volatile("s_waitcnt vmcnt(%12)\n\t"
                     "ds_read2_b32 %0, %9 offset1:32\n\t"
                     "ds_read2_b32 %1, %9 offset0:64 offset1:96\n\t"
                     "ds_read_b32 %2, %9 offset:1024\n\t"
                     "ds_read_b32 %3, %9 offset:1152\n\t"
                     "ds_read_b32 %4, %9 offset:1280\n\t"
                     "ds_read_b32 %5, %9 offset:1408\n\t"
                     "ds_read_b128 %6, %10\n\t"
                     "ds_read_b128 %7, %10 offset:32\n\t"
                     "ds_read_b128 %8, %11\n\t"
                     "s_waitcnt lgkmcnt(0)"
                     : "=&v"(a), "=&v"(b), "=&v"(o.d[1][0][0]), "=&v"(o.d[1][0][1]),
                       "=&v"(o.d[1][0][2]), "=&v"(o.d[1][0][3]), "=&v"(o.mant[0]),
                       "=&v"(o.mant[1]), "=&v"(o.b)
                     : "v"(x), "v"(at.mantRead), "v"(at.tableRead), "n"(Younger)
                     : "memory");
        put(0, 0, a, b);
    } else {
        u32x2 c, d, e, f, g, h;
        const unsigned x0b = x + 1024, x1 = x + 2048, x1b = x + 3072;
        asm volatile("s_waitcnt vmcnt(%17)\n\t"
                     "ds_read2_b32 %0, %11 offset1:32\n\t"
                     "ds_read2_b32 %1, %11 offset0:64 offset1:96\n\t"
                     "ds_read2_b32 %2, %13 offset1:32\n\t"
                     "ds_read2_b32 %3, %13 offset0:64 offset1:96\n\t"
                     "ds_read_b128 %8, %15\n\t"
                     "ds_read_b128 %9, %15 offset:32\n\t"
                     "ds_read_b128 %10, %16\n\t"
                     "ds_read2_b32 %4, %12 offset1:32\n\t"
                     "ds_read2_b32 %5, %12 offset0:64 offset1:96\n\t"
                     "ds_read2_b32 %6, %14 offset1:32\n\t"
                     "ds_read2_b32 %7, %14 offset0:64 offset1:96\n\t"
                     "s_waitcnt lgkmcnt(0)"
                     : "=&v"(a), "=&v"(b), "=&v"(c), "=&v"(d), "=&v"(e), "=&v"(f), "=&v"(g), "=&v"(h),
                       "=&v"(o.mant[0]), "=&v"(o.mant[1]), "=&v"(o.b)
                     : "v"(x), "v"(x0b), "v"(x1), "v"(x1b), "v"(at.mantRead), "v"(at.tableRead),
                       "n"(Younger)
                     : "memory");
        put(0, 0, a, b);
        put(1, 0, c, d);
        put(0, 1, e, f);
        put(1, 1, g, h);
    }
}

// The same for panel A of a pair alone, at F128.
template <unsigned A, unsigned Younger>
__device__ __forceinline__ void readPanel(Operands<1, 1>& o, const LaneLds& at, unsigned x) {
    asm volatile("s_waitcnt vmcnt(%9)\n\t"
                 "ds_read_b32 %0, %6 offset:%10\n\t"
                 "ds_read_b32 %1, %6 offset:%10+128\n\t"
                 "ds_read_b32 %2, %6 offset:%10+256\n\t"
                 "ds_read_b32 %3, %6 offset:%10+384\n\t"
                 "ds_read_b128 %4, %7 offset:%11\n\t"
                 "ds_read_b64 %5, %8 offset:%12\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(o.d[0][0][0]), "=&v"(o.d[0][0][1]), "=&v"(o.d[0][0][2]), "=&v"(o.d[0][0][3]),
                   "=&v"(o.mant[0]), "=&v"(o.b)
                 : "v"(x), "v"(at.mantRead), "v"(at.tableRead), "n"(Younger), "n"(1024 * A),
                   "n"(32 * A), "n"(8 * A)
                 : "memory");
}

// Table entry offsets in bytes: pass j (rows + 4j) and row group g of a lane's entry.
constexpr unsigned kPassBytes = 128, kGroupBytes = 256;

__device__ __forceinline__ void writeEntry(unsigned address, unsigned offset, _Float16 v) {
    asm volatile("ds_write_b16 %0, %1 offset:%2" ::"v"(address), "v"(v), "n"(offset) : "memory");
}

// The lane's source in each panel of a pair (slot L >> 3), from the pair's sources. Asked for ahead of the
// pair's other loads, so that their addresses are computed while the permutes are on their way.
struct PairSources {
    unsigned id[2];
    __device__ PairSources(unsigned ids, unsigned lane)
        : id{lanePermute(ids, lane >> 3), lanePermute(ids, (lane >> 3) + 8)} {}
};

// The sources of the pair at panel p, out of range for panels past the wave's end (whose metadata reads as
// source 0's): their scales read 0 whatever the caller's scales[0], and the wave does not wait at its end
// for rows it has no use for.
__device__ __forceinline__ unsigned sourcesBefore(const TaskWalk& w, unsigned ids, unsigned p) {
    if (__builtin_expect(p + 1 >= w.end, 0))
        ids |= p >= w.end || (w.lane & 8) != 0 ? 0xFFFFFFFFu : 0u;
    return ids;
}

// Issues a pair's X rows, to ring slots 2 (k & 1) and 2 (k & 1) + 1.
template <unsigned S>
__device__ __forceinline__ void gatherPair(const Loader<kBuffer>& ld, const TaskWalk& w,
                                           const PairSources& from, unsigned k) {
    unsigned row[2];
#pragma unroll
    for (unsigned a = 0; a < 2; ++a) row[a] = (from.id[a] << ld.xShift) + 16 * (w.lane & 7);
    char* slot = reinterpret_cast<char*>(w.lds.xtile) + (k & 1u) * 2 * S * 1024;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (unsigned a = 0; a < 2; ++a)
#pragma unroll
        for (unsigned s = 0; s < S; ++s)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                ld.x, (__attribute__((address_space(3))) void*)(slot + 1024 * (S * a + s)), 16, row[a],
                kSlice * s, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
}

// flagRedo for the pairs, `queue` the LDS address of w.lds.redo: as a store the compiler knows, it waited for
// every load in flight, the next pair's rows among them (12,501 tasks whose panels all take the FP32 path:
// F128 419 -> 412 us, F256 854 -> 842).
__device__ __forceinline__ void queueRedo(TaskWalk& w, unsigned queue, unsigned panel, bool redo) {
    if (__builtin_expect(redo, 0)) {
        asm volatile("ds_write_b16 %0, %1" ::"v"(queue + 2 * w.redoCount), "v"(panel - w.begin) : "memory");
        ++w.redoCount;
    }
}

template <unsigned Offset>
__device__ __forceinline__ void clearWord(unsigned address) {
    asm volatile("ds_write_b32 %0, %1 offset:%2" ::"v"(address), "v"(0u), "n"(Offset) : "memory");
}

// What one pair's step leaves for the next: the next pair's scales (lane L: slot L & 7 of panel
// (L >> 3) & 1) and the metadata of the pair after it. The next pair's X is on its way.
struct PairPipe {
    MetaPair ahead;
    float scale;
};

// The pairs [k0, k1) of a wave's panels [begin, end), all exclusive or of any kind (Shared). `cur` is
// the metadata of pair k0.
template <bool Shared, unsigned S>
__device__ __forceinline__ void walkPairs(Loader<kBuffer>& ld, TaskWalk& w, const GroupBounds& bounds,
                                          unsigned k0, unsigned k1,
                                          const MetaPair& cur, PairPipe& pipe, f32x16 (&acc)[4 * S]) {
    constexpr unsigned kValues = Shared ? 8 : 2; // A values of a lane per pair: [row group][pass]
    const unsigned lane = w.lane, last = w.end - 1;
    const bool second = (lane & 8) != 0; // the lane's panel of a pair
    const unsigned bit0 = 1u << (lane >> 4);
    const unsigned table = ldsAddress(w.lds.table16) +
                           2 * (((lane >> 4) * 2 + ((lane & 7) >> 2)) * 8 + (second ? 4 : 0) + (lane & 3));
    const LaneLds at{ldsAddress(w.lds.xtile) + 4 * w.mh.m + 512 * w.mh.h,
                     ldsAddress(w.lds.table16) + 16 * (2 * w.mh.m + w.mh.h),
                     ldsAddress(w.lds.mant) + 4 * (lane & 15), ldsAddress(w.lds.mant) + 16 * w.mh.h};

    const unsigned redo = ldsAddress(w.lds.redo);

    // A pair's A values. Exclusive: `bits` is the lane's row bit of pass 0.
    PairCursor loads;
    BucketCursor bucket(w.offsets, bounds);
    unsigned bits = 0;
    auto loadValues = [&](const MetaPair& m, unsigned p, float (&v)[kValues], auto first)
        __attribute__((always_inline)) {
        unsigned present = m.mask;
        if constexpr (Shared) {
            // Only the row groups of the panel's bucket.
            auto bytes = [](unsigned g) {
                return (g & 1u) * 0xFFu | (g & 2u) * 0x7F80u | (g & 4u) * 0x3FC000u | (g & 8u) * 0x1FE00000u;
            };
            const unsigned g0 = bytes(decltype(first)::value ? bounds.firstGroups(bucket, p)
                                                             : bucket.groups(min(p, last)));
            const unsigned g1 = bytes(bucket.groups(min(p + 1, last)));
            present &= second ? g1 : g0;
        } else if (loads.changes(p)) {
            loads.update(bounds, p);
            const unsigned g0 = loads.g, g1 = loads.second;
            bits = bit0 << (8 * (second ? g1 : g0));
        }
#pragma unroll
        for (unsigned j = 0; j < kValues; ++j) {
            const unsigned bit = Shared ? bit0 << (4 * j) : bits << (4 * j);
            v[j] = ld.value(m.base + __popc(m.mask & (bit - 1u)), (present & bit) != 0);
        }
    };
    constexpr unsigned kYounger = 3 + kValues + 2 * S; // metadata (2), scales, values, X

    // The table holds one row group per panel, the other groups' entries 0.
    PairCursor staged;
    unsigned entry = table;
    if constexpr (!Shared) {
        const unsigned words = ldsAddress(w.lds.table16) + 4 * lane;
        clearWord<0>(words);
        clearWord<256>(words);
        clearWord<512>(words);
        clearWord<768>(words);
    }
    auto stage = [&](const float (&v)[kValues], float scale, unsigned p) __attribute__((always_inline)) {
        if (!Shared && staged.changes(p)) {
            writeEntry(entry, 0, 0);
            writeEntry(entry, kPassBytes, 0);
            staged.update(bounds, p);
            const unsigned g0 = staged.g, g1 = staged.second;
            entry = table + kGroupBytes * (second ? g1 : g0);
        }
        // stagePanel explains the scale factor and the exactness check.
        const float pow2 = __builtin_amdgcn_ldexpf(
            __uint_as_float(__float_as_uint(scale) & 0x7F800000u), kShift + 1);
        std::uint64_t inexact = 0;
        forEachIndex<kValues>([&](auto c) __attribute__((always_inline)) {
            constexpr unsigned j = decltype(c)::value;
            const float a = roundTf32(v[j]);
            const _Float16 e = static_cast<_Float16>(a * pow2);
            inexact |= __builtin_amdgcn_ballot_w64(a != 0.0f) & ~normalF16(e);
            writeEntry(entry, kPassBytes * j, e);
        });
        asm volatile("ds_write_b32 %0, %1" ::"v"(at.mantWrite), "v"(shiftedMantissa(scale, w.keep))
                     : "memory");
        if (__builtin_expect(inexact != 0, 0)) { // the FP32 pass adds these panels: all-zero tables here
            constexpr std::uint64_t kFirst = 0x00FF00FF00FF00FFull;
            const bool bad0 = (inexact & kFirst) != 0, bad1 = (inexact & ~kFirst) != 0;
            if (second ? bad1 : bad0)
                forEachIndex<kValues>([&](auto c) __attribute__((always_inline)) {
                    writeEntry(entry, kPassBytes * decltype(c)::value, 0);
                });
            queueRedo(w, redo, p, bad0);
            queueRedo(w, redo, p + 1, bad1);
        }
    };

    float v[kValues];
    loadValues(cur, w.begin + 2 * k0, v, std::true_type{});
    // Where the loop begins in its 32-byte fetch line decides 2-4% where one wave per SIMD waits for each pair
    // in turn (2,009 power-law tasks of four waves, F128, by begin: 0 35.6 us, 8 35.4, 16 35.1, 24 35.1, 28
    // 36.1; F256, 752 tasks, 16 45.7, 28 47.3). Fixed here, so that it does not change with the code in front.
    asm volatile(".p2align 5\n\ts_nop 0\n\ts_nop 0\n\ts_nop 0\n\ts_nop 0");
#pragma unroll 1
    for (unsigned k = k0; k < k1; ++k) {
        const unsigned p = w.begin + 2 * k;
        // The next pair's loads, and the metadata of the one after it.
        const unsigned id = sourcesBefore(w, pipe.ahead.id, p + 2);
        const PairSources from(id, lane);
        __builtin_amdgcn_sched_barrier(0);
        const MetaPair next = ld.meta2(p + 4, last, lane);
        const float scaleAhead = ld.scale(id);
        float vn[kValues];
        loadValues(pipe.ahead, p + 2, vn, std::false_type{});
        gatherPair<S>(ld, w, from, k + 1);
        stage(v, pipe.scale, p);
        const unsigned x = at.x + (k & 1u) * 2 * S * 1024;
        if constexpr (Shared && S == 1) { // eight values a lane in flight: no registers for a pair's operands
            Operands<1, 1> o;
            readPanel<0, kYounger>(o, at, x);
            multiply<1, 1>(o, acc);
            readPanel<1, kYounger>(o, at, x);
            multiply<1, 1>(o, acc);
        } else {
            Operands<S, 2> o;
            readPair<S, kYounger>(o, at, x);
            multiply<S, 2>(o, acc);
        }
#pragma unroll
        for (unsigned j = 0; j < kValues; ++j) v[j] = vn[j];
        pipe.scale = scaleAhead;
        pipe.ahead = next;
    }
}

// A wave's panels, pair by pair from its first: exclusive pairs, then (from the pair that holds the first
// shared panel) pairs of any kind. The pipeline runs through: the first shared pair's X, scales and
// successor's metadata are loaded by the last exclusive step.
template <unsigned S>
__device__ __forceinline__ void walkAllPairs(Loader<kBuffer>& ld, TaskWalk& w, const GroupBounds& bounds,
                                             unsigned exclusive, const MetaPair& first,
                                             f32x16 (&acc)[4 * S]) {
    const unsigned pairs = (w.end - w.begin + 1) / 2;
    PairPipe pipe;
    pipe.ahead = ld.meta2(w.begin + 2, w.end - 1, w.lane);
    __builtin_amdgcn_sched_barrier(0);
    ld.startTask({first.id, first.mask, first.base});
    const unsigned ids = sourcesBefore(w, first.id, w.begin);
    pipe.scale = ld.scale(ids);
    gatherPair<S>(ld, w, PairSources(ids, w.lane), 0);
    if (exclusive) walkPairs<false, S>(ld, w, bounds, 0, exclusive, first, pipe, acc);
    if (exclusive < pairs) {
        const MetaPair cur = exclusive ? ld.meta2(w.begin + 2 * exclusive, w.end - 1, w.lane) : first;
        walkPairs<true, S>(ld, w, bounds, exclusive, pairs, cur, pipe, acc);
    }
    // The loads past the end have to land before their ring slots hold anything else.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

template <unsigned S, class Ld>
__device__ __forceinline__ void walkTask(Ld& ld, const unsigned* offsets, unsigned begin,
                                         unsigned end, unsigned lane, const Lds& lds,
                                         f32x16 (&acc)[4 * S]) {
    if (begin >= end) return;
    const auto first = [&] {
        if constexpr (Ld::kWide)
            return ld.meta8(begin, begin, lane);
        else
            return ld.meta2(begin, end - 1, lane);
    }();
    // An opaque definition keeps the mask in one VGPR for the whole walk instead of a
    // rematerialised literal per use.
    unsigned keep;
    asm("v_mov_b32 %0, 0x807fffff" : "=v"(keep));
    LaneMh mh;
    // %0 is written before %2 is read again: early-clobber, so it never shares the input's register.
    asm("v_and_b32 %0, 31, %2\n\tv_lshrrev_b32 %1, 5, %2" : "=&v"(mh.m), "=v"(mh.h) : "v"(lane));
    TaskWalk w{offsets, begin, end, lane, lds, 0u, keep, mh};
    const GroupBounds bounds{offsets[2], offsets[3], offsets[4], offsets[5], offsets[6]};
    // Exclusive pairs; from the pair with the first shared panel on, pairs of any kind.
    const unsigned pairs = (end - begin + 1) / 2;
    const unsigned exclusive = bounds.shared >= end ? pairs : (max(bounds.shared, begin) - begin) / 2;
    if constexpr (Ld::kWide) {
        const unsigned split = min(begin + 2 * exclusive, end);
        walkPanels<false, S>(ld, w, bounds, begin, split, first, acc);
        walkPanels<true, S>(ld, w, bounds, split, end, first, acc);
    } else {
        walkAllPairs<S>(ld, w, bounds, exclusive, first, acc);
    }
    waveSync();
#pragma unroll 1
    for (unsigned i = 0; i < w.redoCount; ++i) {
        const unsigned panel = begin + __builtin_amdgcn_readfirstlane(lds.redo[i]);
        const unsigned groups = groupsOf(offsets, panel);
        Stage st;
        loadStage<true, S>(ld, ld.meta8(panel, panel, lane), 0u, groups, lane, st);
        // The X rows are asked for before anything waits for the values: left to the scheduler, the table's
        // entries came first, one more memory latency a panel (12,501 tasks with every panel here, F128 465 ->
        // 419 us, F256 948 -> 854).
        __builtin_amdgcn_sched_barrier(0);
        computePanelF32<Ld::kWide, S>(st, groups, lane, lds, acc);
    }
}

// Four consecutive floats of Y or of the partial tiles. Vec4: one 16-byte access (the buffer's
// base is 16-byte aligned, which every row offset keeps); otherwise four dword accesses, for a base
// that is only float-aligned (the reference stores single floats, src/kernel/spmm_kernel.cuh:
// 236-245, so it accepts one).
template <bool Vec4>
__device__ __forceinline__ void store4(float* p, const f32x4& v, bool nontemporal) {
    if constexpr (Vec4) {
        if (nontemporal)
            __builtin_nontemporal_store(v, reinterpret_cast<f32x4*>(p));
        else
            *reinterpret_cast<f32x4*>(p) = v;
    } else {
#pragma unroll
        for (unsigned t = 0; t < 4; ++t) {
            if (nontemporal)
                __builtin_nontemporal_store(v[t], p + t);
            else
                p[t] = v[t];
        }
    }
}
template <bool Vec4>
__device__ __forceinline__ f32x4 load4(const float* p) {
    if constexpr (Vec4) return *reinterpret_cast<const f32x4*>(p);
    else return f32x4{p[0], p[1], p[2], p[3]};
}

// Quad q (four consecutive features) of part i of the accumulators of one slice: per part the lane
// holds the 16 features 16 (2i + h) .. + 15 of its row (lane & 31), block b / register 4i + j
// holding feature 2j + (b >> 1) + 8 (b & 1) of them.
template <unsigned I, unsigned Q>
__device__ __forceinline__ f32x4 partQuad(const f32x16 (&acc)[4]) {
    f32x4 v;
#pragma unroll
    for (unsigned t = 0; t < 4; ++t) {
        const unsigned o = 4 * Q + t;
        const unsigned hiHalf = o >= 8 ? 1u : 0u;
        const unsigned rem = o - 8 * hiHalf;
        v[t] = acc[(rem & 1u) * 2 + hiHalf][4 * I + (rem >> 1)];
    }
    return v;
}

// Workgroup -> task. Workgroups are dispatched to the 8 XCDs round-robin by id, and XCD x walks
// one contiguous range of the task list, so neighbouring SWs share source rows of X in its L2. The
// ranges hold equal task counts unless that leaves some XCD more than 3% above the mean panel
// count (hub SWs cut into many 384-panel tasks); then the ranges hold equal panel counts, each
// boundary moved at most a quarter of a share (T / 32 tasks) from its equal-count place. The grid
// carries half a share (ceil(T / 16)) of spare workgroups per XCD, enough for the longest range
// this allows; workgroups past their XCD's range exit. Task begins never decrease along the list,
// so the panel-balanced boundaries are searches over them (panelBound), the same for every
// workgroup of an XCD.
constexpr unsigned kSpareDiv = 16; // spare workgroups per XCD: ceil(T / 16), half a share

__host__ __device__ inline unsigned spareWorkgroups(unsigned tasks) {
    return (tasks + kSpareDiv - 1) / kSpareDiv;
}

__device__ __forceinline__ unsigned equalBound(unsigned tasks, unsigned x) {
    const unsigned q = tasks >> 3, r = tasks & 7u;
    return x * q + min(x, r);
}

// The tail window: the last kTailWindow tasks of an XCD's range run longest size class first
// (panels >= 288, >= 192, >= 96, the rest; list order within a class), so that the launch does not
// end on a few long tasks started last. The window spans about the SWs an XCD holds resident at its
// end anyway, so the order inside it leaves the L2 sharing of the in-order walk in place.
constexpr unsigned kTailWindow = 512;

// Whether a task of p panels is in size class c (1..3) or above.
__device__ __forceinline__ unsigned sizeClass(unsigned p, unsigned c) {
    return c == 1 ? p >= 96 : c == 2 ? p >= 192 : p >= 288;
}

// Task at position r (r < n <= kTailWindow) of the window [w0, w0 + n) in size-class order. One
// wave, all lanes active; every wave computes the same permutation of the window. The sizes of the
// window's tasks are loaded once (lane L: tasks L, L + 64, ...; all loads in flight together); per 64
// tasks three compares give the wave masks of the tasks of at least 96, 192 and 288 panels, and
// counting and picking are scalar work on those (two bits per task in a register and a ballot per
// class took 3-4 us instead of about 2, half of it VALU work beside the other waves').
__device__ __forceinline__ unsigned tailTask(const Sw32Task* tasks, unsigned w0, unsigned n,
                                             unsigned r, unsigned lane) {
    constexpr unsigned kChunks = kTailWindow / kWave;
    unsigned panels[kChunks];
#pragma unroll
    for (unsigned ch = 0; ch < kChunks; ++ch) {
        const Sw32Task& t = tasks[w0 + min(ch * kWave + lane, n - 1)];
        panels[ch] = t.end - t.begin;
    }
    std::uint64_t atLeast[kChunks][4]; // class c or above: c = 0 any task of the window
    unsigned counts[4] = {0, 0, 0, 0};
#pragma unroll
    for (unsigned ch = 0; ch < kChunks; ++ch) {
        const unsigned in = n > ch * kWave ? min(n - ch * kWave, kWave) : 0u;
        atLeast[ch][0] = in == kWave ? ~std::uint64_t(0) : (std::uint64_t(1) << in) - 1;
#pragma unroll
        for (unsigned c = 1; c < 4; ++c)
            atLeast[ch][c] = __builtin_amdgcn_ballot_w64(sizeClass(panels[ch], c)) & atLeast[ch][0];
#pragma unroll
        for (unsigned c = 0; c < 4; ++c) counts[c] += unsigned(__builtin_popcountll(atLeast[ch][c]));
    }
    // counts[c]: tasks of class c or above; position r is in the highest class whose count exceeds it.
    const unsigned c = r < counts[3] ? 3u : r < counts[2] ? 2u : r < counts[1] ? 1u : 0u;
    unsigned k = r - (c == 3 ? 0u : c == 2 ? counts[3] : c == 1 ? counts[2] : counts[1]);
#pragma unroll
    for (unsigned ch = 0; ch < kChunks; ++ch) {
        const std::uint64_t mask = c == 3   ? atLeast[ch][3]
                                   : c == 2 ? atLeast[ch][2] & ~atLeast[ch][3]
                                   : c == 1 ? atLeast[ch][1] & ~atLeast[ch][2]
                                            : atLeast[ch][0] & ~atLeast[ch][1];
        const unsigned count = unsigned(__builtin_popcountll(mask));
        if (k < count) {
            const unsigned below = __builtin_amdgcn_mbcnt_hi(unsigned(mask >> 32),
                                                             __builtin_amdgcn_mbcnt_lo(unsigned(mask), 0u));
            const std::uint64_t hit = __builtin_amdgcn_ballot_w64(below == k) & mask;
            return w0 + ch * kWave + unsigned(__builtin_ctzll(hit));
        }
        k -= count;
    }
    return w0 + r; // not reached: the window holds n tasks
}

// Search for the boundary of a panel-balanced range: the first task of [l, r) that begins at or past
// `target`, or r. Each step probes 64 evenly spaced tasks with one load (load(), apart from the
// step that uses it, so that several searches' loads and other loads are in flight together) and
// keeps the stretch between the last probe below the target and the first one at or past it: two
// steps for the ranges of plans of up to 65,536 tasks. All bounds are wave-uniform.
struct BoundSearch {
    unsigned l, r, probed;
    __device__ unsigned stride() const { return (r - l + kWave - 1) / kWave; }
    __device__ bool done() const { return l >= r; }
    __device__ void load(const Sw32Task* tasks, unsigned lane) {
        if (!done()) probed = tasks[min(l + lane * stride(), r - 1)].begin;
    }
    __device__ void step(unsigned target, unsigned lane) {
        if (done()) return;
        const unsigned s = stride();
        const std::uint64_t at =
            __builtin_amdgcn_ballot_w64(l + lane * s >= r || probed >= target);
        const unsigned first = at ? unsigned(__builtin_ctzll(at)) : kWave;
        const unsigned nr = first < kWave ? min(l + first * s, r) : r;
        if (first) l += (first - 1) * s + 1;
        r = nr;
    }
};

// Returns false when the workgroup has no task.
__device__ __forceinline__ bool xcdTask(const KernelArgs& a, unsigned bid, unsigned& task) {
    const Sw32Task* tasks = a.m.tasks;
    const unsigned count = a.m.taskCount, x = bid & 7u, j = bid >> 3;
    const unsigned lane = threadIdx.x & (kWave - 1);
    unsigned lo = equalBound(count, x), hi = equalBound(count, x + 1);
    // Every workgroup starts at once (launch): neither the order nor the balance decides anything, and
    // finding them takes about 2 us of dependent loads (313 tasks of 8 waves, F128: 18.3 -> 16.2 us).
    if (a.resident) {
        task = lo + j;
        return task < hi;
    }
    // Boundary k (0 < k < 8) of the balanced ranges lies within `reach` tasks of the equal-count one.
    const unsigned reach = spareWorkgroups(count) / 2;
    auto search = [&](unsigned k) {
        const unsigned eq = equalBound(count, k);
        const bool fixed = k == 0 || k == 8;
        return BoundSearch{fixed ? eq : eq > reach ? eq - reach : 0u, fixed ? eq : eq + reach, 0u};
    };
    BoundSearch left = search(x), right = search(x + 1);
    left.load(tasks, lane); // in flight beside the loads of the range check
    right.load(tasks, lane);
    auto beginOf = [&](unsigned t) { return t < count ? tasks[t].begin : tasks[count - 1].end; };
    unsigned first[9];
    unsigned maxPanels = 0;
#pragma unroll
    for (unsigned k = 0; k <= 8; ++k) first[k] = beginOf(equalBound(count, k));
#pragma unroll
    for (unsigned k = 0; k < 8; ++k) maxPanels = max(maxPanels, first[k + 1] - first[k]);
    const std::uint64_t panels = first[8] - first[0];
    if (std::uint64_t(maxPanels) * 8 * 100 > panels * 103) {
        const unsigned targetLeft = first[0] + unsigned(panels * x / 8);
        const unsigned targetRight = first[0] + unsigned(panels * (x + 1) / 8);
        left.step(targetLeft, lane);
        right.step(targetRight, lane);
        while (!left.done() || !right.done()) {
            left.load(tasks, lane);
            right.load(tasks, lane);
            left.step(targetLeft, lane);
            right.step(targetRight, lane);
        }
        lo = left.l;
        hi = right.l;
    }
    task = lo + j;
    if (task >= hi) return false;
    const unsigned n = min(hi - lo, kTailWindow), w0 = hi - n;
    if (task >= w0) task = tailTask(tasks, w0, n, task - w0, lane);
    return true;
}

// Merge of slice k of a split SW by the task that took its last ticket (reference
// src/kernel/spmm_kernel.cuh:250-282): Y = the SW's partial tiles summed in partialIds order,
// starting from 0.0f, one row group (8 rows x 128 columns) at a time. Lane L sums the four 16-byte
// column blocks (L & 7) + 8j, j < 4, of row L >> 3. The group's tile ids are loaded once (one per
// lane, broadcast by readlane), and the loads of kMergeBatch tiles are issued before they are added
// in order, so a merge of many chunks waits for one load latency per batch, not per tile. Per element
// the additions run in partialIds order whatever the batch, so Y is bitwise the same for any batch.
// The task's waves take the row groups in turn.
template <unsigned Features, bool Vec4>
__device__ __forceinline__ void mergeSlice(const KernelArgs& a, const Sw32Task& task, unsigned k,
                                           unsigned wave, unsigned waves, unsigned lane) {
    constexpr unsigned kMergeBatch = 4;
    const unsigned sw = task.sw;
    const unsigned mrow = lane >> 3, mcol = k * kSlice + (lane & 7) * 4;
#pragma unroll 1
    for (unsigned g = wave; g < 4; g += waves) {
        const Sw32ReduceRange red = a.m.reductions[task.reduceFirst + g];
        const unsigned row0 = sw * 32 + g * 8;
        if (row0 >= a.rows) continue;
        f32x4 sum[4];
#pragma unroll
        for (unsigned j = 0; j < 4; ++j) sum[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        auto tileRow = [&](unsigned id) {
            return a.partials + (std::size_t(id) * 8 + mrow) * Features + mcol;
        };
#pragma unroll 1
        for (unsigned base = red.begin; base < red.end; base += kWave) {
            const unsigned items = min(red.end - base, kWave);
            const unsigned ids = a.m.partialIds[base + min(lane, items - 1)];
            unsigned i = 0;
#pragma unroll 1
            for (; i + kMergeBatch <= items; i += kMergeBatch) {
                f32x4 v[kMergeBatch][4];
#pragma unroll
                for (unsigned u = 0; u < kMergeBatch; ++u) {
                    const float* src = tileRow(__builtin_amdgcn_readlane(ids, i + u));
#pragma unroll
                    for (unsigned j = 0; j < 4; ++j) v[u][j] = load4<Vec4>(src + 32 * j);
                }
#pragma unroll
                for (unsigned u = 0; u < kMergeBatch; ++u)
#pragma unroll
                    for (unsigned j = 0; j < 4; ++j) sum[j] += v[u][j];
            }
#pragma unroll 1
            for (; i < items; ++i) {
                const float* src = tileRow(__builtin_amdgcn_readlane(ids, i));
#pragma unroll
                for (unsigned j = 0; j < 4; ++j) sum[j] += load4<Vec4>(src + 32 * j);
            }
        }
        if (row0 + mrow < a.rows) {
            float* yr = a.y + std::size_t(row0 + mrow) * Features + mcol;
#pragma unroll
            for (unsigned j = 0; j < 4; ++j) store4<Vec4>(yr + 32 * j, sum[j], false);
        }
    }
}

// LDS of one wave's walk.
template <unsigned S>
struct WaveLds {
    alignas(16) u32x4 xtile[4 * 64 * S]; // walkPairs: a ring of two pairs; walkPanels: one pair
    alignas(16) _Float16 table16[512];
    alignas(16) float mant[16];
    alignas(16) unsigned short redo[384];
};

// The write-back of a task: the doubled sum of its waves, one or two parts (32 features each, 16 per lane
// half) at a time. Every wave puts its part into LDS; then each (part, row group) of the round is one
// wave's: lane L adds piece L & 7 (four features) of row 8g + (L >> 3) over the waves in order and
// stores it, eight lanes to a 128-byte line of a row. `store(k, g, r, column, v)` stores four
// features from `column` of slice k, row r of row group g. A single wave goes the same way, for the
// stores: straight from the accumulators each instruction wrote 16 bytes of 64 different lines, and
// a line of Y took eight of them (2.45M rows: F128 2,954 -> 2,854 us, F256 4,967 -> 4,851; 1M rows with
// 64 hub rows, F256: 1,909 -> 1,774 us).
//
// LDS: [wave][part of the round][piece 0..7][33 x 16 bytes]: piece 2q + h of row r at index r, 33 so
// that the eight pieces of a row fall into different banks.
constexpr unsigned kPiece = 33, kPart = 8 * kPiece;
constexpr unsigned kRoundParts = 2;

template <unsigned Waves>
__device__ __forceinline__ void taskSync() {
    if constexpr (Waves > 1)
        __syncthreads();
    else
        waveSync();
}

template <unsigned S, unsigned Waves, class Store>
__device__ __forceinline__ void writeTask(const f32x16 (&acc)[4 * S], f32x4* mem, unsigned wave,
                                          unsigned lane, Store store) {
    constexpr unsigned kParts = kRoundParts;
    const unsigned row = lane & 31, h = lane >> 5;
    forEachIndex<4 * S / kParts>([&](auto round) __attribute__((always_inline)) {
        constexpr unsigned kFirst = decltype(round)::value * kParts;
        taskSync<Waves>(); // the walks' LDS, or the last round's, is no longer read
        f32x4* mine = mem + wave * kParts * kPart;
        forEachIndex<kParts * 4>([&](auto c) __attribute__((always_inline)) {
            constexpr unsigned P = decltype(c)::value / 4, Q = decltype(c)::value % 4;
            constexpr unsigned K = (kFirst + P) / 4, I = (kFirst + P) % 4;
            const auto& slice = *reinterpret_cast<const f32x16(*)[4]>(&acc[4 * K]);
            mine[P * kPart + (2 * Q + h) * kPiece + row] = partQuad<I, Q>(slice);
        });
        taskSync<Waves>();
        constexpr unsigned kMine = Waves >= 4 * kParts ? 1 : 4 * kParts / Waves; // stretches of this wave
        constexpr unsigned kBatch = kMine < 4 ? kMine : 4; // LDS reads in flight
        const unsigned r = lane >> 3, piece = lane & 7;
        const f32x4* from = mem + ((piece & 3) * 2 + (piece >> 2)) * kPiece + r;
#pragma unroll
        for (unsigned b = 0; b < kMine; b += kBatch) {
            f32x4 sum[kBatch];
#pragma unroll
            for (unsigned u = 0; u < kBatch; ++u) {
                const unsigned o = wave + (b + u) * Waves, part = o >> 2, g = o & 3;
                sum[u] = from[part * kPart + 8 * g];
#pragma unroll
                for (unsigned v = 1; v < Waves; ++v) sum[u] += from[(v * kParts + part) * kPart + 8 * g];
            }
#pragma unroll
            for (unsigned u = 0; u < kBatch; ++u) {
                const unsigned o = wave + (b + u) * Waves, g = o & 3;
                const unsigned at = kFirst + (o >> 2); // slice at / 4, features 32 (at % 4) .. + 31
                store(at >> 2, g, r, 32 * (at & 3) + 4 * piece, sum[u] * 2.0f); // Y / 2 to Y, exact
            }
        }
    });
}

// One task over all S = Features / 128 slices of its SW, by `Waves` waves of one workgroup:
// wave w walks the w-th equal share of the task's panels (its own LDS tables, the same walk as a whole
// task), and their sum, in wave order, is written by all of them (writeTask). A task then takes about
// 1/waves of the time, which shortens launches whose longest tasks set the time (few tasks per wave
// slot).
template <unsigned Features, unsigned Addr, unsigned Waves = 1>
__device__ __forceinline__ void runTask(const KernelArgs& a, unsigned taskIndex) {
    constexpr unsigned S = Features / kSlice;
    constexpr std::size_t kWalkBytes = sizeof(WaveLds<S>) * Waves;
    constexpr std::size_t kWriteBytes = std::size_t(Waves) * kRoundParts * kPart * 16;
    __shared__ __align__(16) unsigned char shared[kWalkBytes > kWriteBytes ? kWalkBytes : kWriteBytes];
    __shared__ unsigned lastFlag[S];
    const unsigned wave = Waves == 1 ? 0u : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned lane = Waves == 1 ? threadIdx.x : threadIdx.x & 63u;
    const Sw32Task task = a.m.tasks[taskIndex];
    const unsigned sw = task.sw;
    unsigned lo = task.begin, hi = task.end;
    if constexpr (Waves > 1) {
        const unsigned pairs = (hi - lo + 1) / 2; // whole pairs, except the last one of an odd task
        lo = task.begin + 2 * (pairs * wave / Waves);
        hi = min(task.end, task.begin + 2 * (pairs * (wave + 1) / Waves));
    }
    Loader<Addr> ld(a, lo, hi, Features);
    WaveLds<S>& mem = reinterpret_cast<WaveLds<S>*>(shared)[wave];
    // The FP32 path's table lies behind the one panel of X it uses, after the walk.
    const Lds lds{mem.table16, reinterpret_cast<float*>(mem.xtile + 128 * S), mem.xtile, mem.mant,
                  mem.redo};

    f32x16 acc[4 * S];
#pragma unroll
    for (unsigned b = 0; b < 4 * S; ++b) acc[b] = f32x16{};
    walkTask<S>(ld, a.m.bucketOffsets + std::size_t(sw) * 17, lo, hi, lane, lds, acc);
    // The last MFMAs' results are not interlocked against the moves that read them, and the compiler
    // has padded a path into this point with fewer wait states than the 18 they need.
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 15\n\ts_nop 1");
    __builtin_amdgcn_sched_barrier(0);

    // Write-back. An unsplit task stores its rows of Y (nontemporal: nothing reads them again in this
    // launch); a split task stores the row groups of task.mask as 8-row partial tiles.
    const bool split = task.partial != kNoPartial;
    writeTask<S, Waves>(
        acc, reinterpret_cast<f32x4*>(shared), wave, lane,
        [&](unsigned k, unsigned g, unsigned r, unsigned column, const f32x4& v) {
            float* dst;
            if (!split) {
                const unsigned row = sw * 32 + 8 * g + r;
                if (row >= a.rows) return;
                dst = a.y + std::size_t(row) * Features;
            } else {
                if (!((task.mask >> g) & 1u)) return;
                const std::size_t tile = task.partial + __popc(task.mask & ((1u << g) - 1u));
                dst = a.partials + (tile * 8 + r) * Features;
            }
            if (a.vec4)
                store4<true>(dst + k * kSlice + column, v, !split);
            else
                store4<false>(dst + k * kSlice + column, v, !split);
        });
    if (!split) return;

    // Completion tickets, one per slice: the release fence at agent scope publishes this task's
    // partial tiles before its tickets, and the acquire fence of the last arriver makes every other
    // task's tiles visible (the XCD L2s are not coherent with each other, so the release writes back
    // and the acquire invalidates). One release for all slices, and an acquire only where tiles are
    // read: both work on the whole L2 of the XCD. With several waves, each one's stores have reached
    // that L2 (vmcnt 0) before the barrier in front of the release.
    if constexpr (Waves > 1) __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0)
    taskSync<Waves>();
    if (wave == 0 && lane == 0) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
#pragma unroll
        for (unsigned k = 0; k < S; ++k) {
            unsigned* counter = a.counters + std::size_t(sw) * S + k;
            const unsigned ticket =
                __builtin_amdgcn_atomic_inc32(counter, task.chunks - 1, __ATOMIC_RELAXED, "agent");
            lastFlag[k] = ticket == task.chunks - 1;
        }
    }
    taskSync<Waves>();
#pragma unroll 1
    for (unsigned k = 0; k < S; ++k) {
        if (!lastFlag[k]) continue;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        if (a.vec4)
            mergeSlice<Features, true>(a, task, k, wave, Waves, lane);
        else
            mergeSlice<Features, false>(a, task, k, wave, Waves, lane);
    }
}

// Per-task timeline for the measurement build (compiled with TCC_SPMM_TIMELINE by
// model/timeline.py; the library build leaves this empty and the kernels unchanged). Lane 0 of each
// workgroup stores, for its task: the workgroup's start, the time its task was found, its end
// (s_memrealtime, a 100 MHz counter) and its XCC id << 32 | workgroup id, with vector stores.
struct TaskClock {
#ifdef TCC_SPMM_TIMELINE
    unsigned long long start = __builtin_amdgcn_s_memrealtime(), found = 0;
    __device__ void mapped() { found = __builtin_amdgcn_s_memrealtime(); }
    __device__ void done(const KernelArgs& a, unsigned task) const {
        const unsigned long long end = __builtin_amdgcn_s_memrealtime();
        if (threadIdx.x == 0 && a.stamps) {
            const unsigned long long xcc = __builtin_amdgcn_s_getreg((3 << 11) | 20); // HW_REG_XCC_ID
            unsigned long long* out = a.stamps + 4 * std::size_t(task);
            out[0] = start;
            out[1] = found;
            out[2] = end;
            out[3] = xcc << 32 | blockIdx.x;
        }
    }
#else
    __device__ void mapped() {}
    __device__ void done(const KernelArgs&, unsigned) const {}
#endif
};

// Waves per SIMD of an instance, which its registers have to allow. The launch's wave slots follow it: with
// four for the 64-bit F128 instances, plans that took all of their slots were held to leave some free and went
// without an order (2,855 power-law tasks 141 -> 124 us; 2,813 uniform ones 35.1 -> 36.4).
constexpr unsigned wavesPerSimd(unsigned features, unsigned addr) {
    return features == 256 ? 2 : addr == kBuffer ? 4 : 3;
}

// F128: four waves per SIMD; the 64 accumulators live in ordinary VGPRs and the kernel fits 128
// registers. The 64-bit-addressed instances hold a pair's operands and their stages in registers and run
// three (2.45M rows through the 64-bit instance: 3,188 us as one panel at a time and four waves, 3,179).
template <unsigned Addr, unsigned Waves = 1>
__global__ __launch_bounds__(kWave * Waves) __attribute__((amdgpu_waves_per_eu(wavesPerSimd(128, Addr), 8))) void
spmmInt8Kernel128(KernelArgs a) {
    TaskClock clock;
    unsigned task;
    if (xcdTask(a, blockIdx.x, task)) {
        clock.mapped();
        runTask<128, Addr, Waves>(a, task);
        clock.done(a, task);
    }
}

// F256: both 128-feature slices of a task in one wave (128 accumulator registers, two waves per
// SIMD). The task's A stream, scales and A table are read and built once for both slices; measured
// on c3 this moves 18% fewer bytes (33.1 GB against 40.5 GB) and runs 8.6% faster than one wave
// per (task, slice).
template <unsigned Addr, unsigned Waves = 1>
__global__ __launch_bounds__(kWave * Waves) __attribute__((amdgpu_waves_per_eu(wavesPerSimd(256, Addr), 8))) void
spmmInt8Kernel256(KernelArgs a) {
    TaskClock clock;
    unsigned task;
    if (xcdTask(a, blockIdx.x, task)) {
        clock.mapped();
        runTask<256, Addr, Waves>(a, task);
        clock.done(a, task);
    }
}

constexpr int kMaxDevices = 64;

// Launch choices forced by setSpmmLaunchOverrides or, initially, the environment (read once).
std::once_flag overridesRead;
std::atomic<unsigned> forcedWaves{0}; // 0: chosen per launch
std::atomic<bool> forcedWide{false};

bool isTaskForm(std::uint32_t waves) { return waves == 1 || waves == 2 || waves == 4 || waves == 8; }

void readOverridesOnce() {
    std::call_once(overridesRead, [] {
        if (const char* w = std::getenv("TCC_SPMM_TASK_WAVES")) {
            const unsigned waves = w[0] && !w[1] ? unsigned(w[0] - '0') : 0u;
            if (!isTaskForm(waves))
                std::fprintf(stderr, "tcc_spmm: TCC_SPMM_TASK_WAVES=%s is not 1, 2, 4 or 8; one wave "
                                     "per task\n", w);
            forcedWaves.store(isTaskForm(waves) ? waves : 1u);
        }
        if (std::getenv("TCC_SPMM_FORCE_WIDE")) forcedWide.store(true);
    });
}

// Compute units of the current device, queried once per device (0 when unknown).
std::atomic<int> deviceCuCount[kMaxDevices];

int currentDeviceCus() {
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) return 0;
    int cus = deviceCuCount[device].load(std::memory_order_relaxed);
    if (cus == 0 &&
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess)
        deviceCuCount[device].store(cus, std::memory_order_relaxed);
    return cus;
}

// Wave slots of the current device: CUs x 4 SIMDs x the instance's waves per SIMD (0 when unknown).
std::uint64_t waveSlots(unsigned features, unsigned addr) {
    const int cus = currentDeviceCus();
    return cus <= 0 ? 0 : std::uint64_t(cus) * 4 * wavesPerSimd(features, addr);
}

// Waves per task. Few tasks for the chip: as many waves as keep the chip's slots in use, since the
// longest tasks, not the bandwidth, set the launch time. Measured on MI355X (us; 256 CUs, 4,096 wave slots at
// F128 and 2,048 at F256). short: all tasks of 33 panels; equal: all of 130; skewed: power-law rows with
// communities, 89 panels in the mean and 384 in the longest (SWs split into several tasks):
//
//   tasks, about        250    500    750  1,000  1,500  2,050  3,150  4,150  6,300 12,600
//   F128 1 wave  short    16.2   16.7   17.4   18.2   20.7   21.3   31.2   35.5   55.5    121
//                equal    38.9   41.4   43.1   44.9   52.8   54.2   87.3   96.6    157    338
//                skewed   96.1    102    103    105    118    128    117    121    167    296
//   F128 2 waves short    11.1   11.8   12.5   14.2   17.5   21.3   32.2   38.8   55.4    127
//                equal    23.3   27.9   28.8   31.6   43.8   50.2   78.5    100    149    338
//                skewed   54.9   60.5   66.2   67.2   59.0   63.7   69.3   83.3    120    268
//   F128 4 waves short     8.6   10.1   12.0   16.1   22.2   25.8   36.4   44.9   62.2    135
//                equal    16.2   19.5   24.3   30.5   41.5   52.5   78.5    103    153    343
//                skewed   35.4   37.6   39.6   37.7   39.7   50.3   71.5   89.4    130    293
//   F128 8 waves short     8.0   10.6   18.4   22.2   30.5   37.8   55.2   70.1    100    194
//                equal    13.3   18.6   30.4   36.3   50.9   66.5    106    135    196    410
//                skewed   26.4   28.0   30.0   38.0   54.5   68.0    100    126    189    401
//   F256 1 wave  short    22.2   23.4   23.8   24.4   30.0   34.0   59.5   66.7    106    227
//                equal    53.4   56.9   58.5   59.9   81.5   87.0    160    176    303    623
//                skewed    131    146    146    147    150    153    161    165    255    448
//   F256 2 waves short    15.2   18.1   18.6   22.0   36.2   39.6   60.1   75.3    113    235
//                equal    32.2   42.3   43.9   48.8   87.7   93.8    151    192    291    608
//                skewed   74.0   90.9    102   81.4   83.6   85.9    119    152    235    459
//   F256 4 waves short    11.5   16.8   25.0   28.1   38.1   47.8   71.3   90.0    132    262
//                equal    21.6   30.5   44.0   53.4   75.9   99.8    156    196    308    609
//                skewed   46.1   47.6   47.4   52.5   73.1   92.5    137    170    273    546
//   F256 8 waves short    11.3   24.0   33.7   43.5   61.9   80.3    123    159    231    445
//                equal    18.9   39.2   57.4   76.0    113    150    235    296    434    817
//                skewed   36.2   41.7   58.7   73.7    113    145    215    276    428    842
//
// The lines: 8 waves while every wave has a slot (slots / 8 tasks), 4 up to 5/8 slots; then 2 up to 8 tasks
// per slot at F128 and 3 at F256, where one wave per task has longer walks and fewer fills. The host knows how
// many tasks there are, not how long they are: short ones would take fewer waves from 1,000 tasks (F128) and
// 500 (F256) on (750 at F256: 18.6 us with two, 25.0 as chosen), but skewed ones lose more by that than short
// ones gain (47.4 with four, 102 with two), and equal ones lie between.
unsigned taskWaves(unsigned taskCount, unsigned features, std::uint64_t slots) {
    if (const unsigned forced = forcedWaves.load()) return forced;
    if (!slots) return 1;
    const std::uint64_t tasks = taskCount;
    if (8 * tasks <= slots) return 8;
    if (8 * tasks <= 5 * slots) return 4;
    return tasks <= (features == 128 ? 8 : 3) * slots ? 2u : 1u;
}

template <unsigned Features>
void launch(KernelArgs args, hipStream_t stream) {
    // Buffer addressing needs the packed X and the scales within 32-bit byte offsets, with room for
    // the padding sentinel to land out of range, and 16-byte aligned X tiles. A packed X that is
    // only u16-aligned takes the 64-bit instance with 2-byte tile loads. setSpmmLaunchOverrides
    // can select the 64-bit instance for any size (used by the tests).
    const bool misaligned = reinterpret_cast<std::uintptr_t>(args.packedX) % 16 != 0;
    const bool wide = std::uint64_t(args.cols) * Features > 0xFFFFFF00ull || forcedWide.load();
    const unsigned addr = misaligned ? kGlobalU16 : wide ? kGlobal : kBuffer;
    const std::uint64_t slots = waveSlots(Features, addr);
    const unsigned waves = addr == kBuffer ? taskWaves(args.m.taskCount, Features, slots) : 1u;
    // Plans whose workgroups all start at once take their tasks in list order (xcdTask). A quarter of the
    // slots stays free, since with the slots nearly full the order does matter: three skewed plans of 450
    // tasks of eight waves ran 8-14% slower without it, and of 1,000 unsplit tasks of four waves 6-14%. Eight
    // waves of unsplit tasks (none at the 384-panel limit) are short enough to take every slot:
    // 438-500 tasks, F128, uniform 11.8 -> 9.4 us, power-law 14.8 -> 12.1 and 20.9 -> 20.6, rows sorted by
    // degree 35.4 -> 34.3; 512 tasks (all slots) 11.9 -> 9.5, but power-law 16.6 -> 17.1; 250 tasks, F256,
    // 11.7 -> 10.1 to 24.5 -> 23.3.
    const bool unsplit = args.m.taskCount <= (args.rows + 31) / 32;
    args.resident = 4 * std::uint64_t(args.m.taskCount) * waves <= (unsplit && waves == 8 ? 4 : 3) * slots;
    const dim3 grid(args.resident ? args.m.taskCount
                                  : args.m.taskCount + 8 * spareWorkgroups(args.m.taskCount));
    auto go = [&](auto kernel, unsigned n) {
        hipLaunchKernelGGL(kernel, grid, dim3(n * kWave), 0, stream, args);
    };
    if constexpr (Features == 256) {
        if (addr == kGlobalU16)
            go(spmmInt8Kernel256<kGlobalU16>, 1);
        else if (addr == kGlobal)
            go(spmmInt8Kernel256<kGlobal>, 1);
        else if (waves == 8)
            go(spmmInt8Kernel256<kBuffer, 8>, 8);
        else if (waves == 4)
            go(spmmInt8Kernel256<kBuffer, 4>, 4);
        else if (waves == 2)
            go(spmmInt8Kernel256<kBuffer, 2>, 2);
        else
            go(spmmInt8Kernel256<kBuffer>, 1);
    } else {
        if (addr == kGlobalU16)
            go(spmmInt8Kernel128<kGlobalU16>, 1);
        else if (addr == kGlobal)
            go(spmmInt8Kernel128<kGlobal>, 1);
        else if (waves == 8)
            go(spmmInt8Kernel128<kBuffer, 8>, 8);
        else if (waves == 4)
            go(spmmInt8Kernel128<kBuffer, 4>, 4);
        else if (waves == 2)
            go(spmmInt8Kernel128<kBuffer, 2>, 2);
        else
            go(spmmInt8Kernel128<kBuffer>, 1);
    }
}

} // namespace

namespace {

// Checks shared by both entry points, before anything is launched. Null buffers would fault the GPU
// and are rejected (the reference does not check). Of the view, only the arrays every plan has are
// required (tasks, and bucketOffsets with 17 entries per SW): a plan without panels has empty
// sourceIds, sourceMetadata and values, which may be null. The workspace may be null (a plan
// without split SWs), and its size is the caller's contract.
void checkLaunchArguments(const Sw32DeviceView& matrix, const std::int8_t* packedX,
                          const float* scales, const float* output) {
    if (!matrix.taskCount)
        throw std::runtime_error("launchSpmmInt8: invalid configuration argument (no tasks)");
    if (matrix.taskCount > 0x7FFFFFFFu)
        throw std::invalid_argument("launchSpmmInt8: too many tasks for one launch");
    if (!packedX || !scales || !output)
        throw std::invalid_argument("launchSpmmInt8: null packedX, scales or output");
    if (!matrix.tasks || !matrix.bucketOffsets)
        throw std::invalid_argument("launchSpmmInt8: device view with null tasks or bucketOffsets");
    // The packed features are read as u16 pairs at least (reference include/format/int8_features.cuh:
    // 11-13 states u16 alignment); an odd address cannot be.
    if (reinterpret_cast<std::uintptr_t>(packedX) % 2)
        throw std::invalid_argument("launchSpmmInt8: packedX must be u16-aligned");
    // Y is written as floats (16 bytes per lane when Y and the partials are 16-byte aligned, one
    // float per store otherwise), so a float-aligned base is accepted, as in the reference.
    if (reinterpret_cast<std::uintptr_t>(output) % alignof(float))
        throw std::invalid_argument("launchSpmmInt8: output must be float-aligned");
}

} // namespace

#ifdef TCC_SPMM_TIMELINE
// Measurement build only: the stamp buffer of the last launch, grown as needed, and its read-back.
namespace {
unsigned long long* gStamps = nullptr;
std::uint32_t gStampTasks = 0, gStampCapacity = 0;

unsigned long long* timelineStamps(std::uint32_t tasks) {
    if (tasks > gStampCapacity) {
        if (gStamps) checkHip(hipFree(gStamps));
        checkHip(hipMalloc(&gStamps, std::size_t(tasks) * 32));
        gStampCapacity = tasks;
    }
    gStampTasks = tasks;
    return gStamps;
}
} // namespace

extern "C" int tcc_timeline_stamps(unsigned long long* host, std::uint32_t tasks) {
    if (!gStamps || tasks != gStampTasks || hipDeviceSynchronize() != hipSuccess) return 1;
    return hipMemcpy(host, gStamps, std::size_t(tasks) * 32, hipMemcpyDeviceToHost) == hipSuccess ? 0 : 2;
}
#endif

void launchSpmmInt8(Sw32DeviceView matrix, const std::int8_t* packedX, const float* scales,
                    float* output, std::uint32_t rows, std::uint32_t cols, std::uint32_t features,
                    SpmmWorkspace workspace, hipStream_t stream) {
    if (features != 128 && features != 256)
        throw std::invalid_argument("feature dimension must be 128 or 256");
    checkLaunchArguments(matrix, packedX, scales, output);
    readOverridesOnce();
    if (reinterpret_cast<std::uintptr_t>(workspace.partials) % alignof(float))
        throw std::invalid_argument("launchSpmmInt8: workspace.partials must be float-aligned");
    // Y and the partial tiles move 16 bytes per lane when both bases allow it (any hipMalloc'd
    // buffer and any whole-row offset into one does), else one float per access; Y is bitwise
    // the same either way.
    const bool vec4 = (reinterpret_cast<std::uintptr_t>(output) |
                       reinterpret_cast<std::uintptr_t>(workspace.partials)) % 16 == 0;
    KernelArgs args{matrix, packedX, scales, output, workspace.partials, workspace.counters,
                    rows,   cols,    0u, unsigned(vec4)};
#ifdef TCC_SPMM_TIMELINE
    args.stamps = timelineStamps(matrix.taskCount);
#endif
    if (features == 128)
        launch<128>(args, stream);
    else
        launch<256>(args, stream);
    checkHip(hipGetLastError());
}

void setSpmmLaunchOverrides(std::uint32_t taskWaves, bool forceWide) {
    if (taskWaves && !isTaskForm(taskWaves))
        throw std::invalid_argument("setSpmmLaunchOverrides: taskWaves must be 0, 1, 2, 4 or 8");
    readOverridesOnce(); // so that a later first launch keeps these rather than the environment's
    forcedWaves.store(taskWaves);
    forcedWide.store(forceWide);
}

// ------------------------------------------------------------------------------------------------
// Allocation-free entry point (no counterpart in the reference): the split-SW workspace lives in a
// library-owned device array instead of caller buffers. Layout: completion counters
// [ceil(rows/32)][F/128] from offset 0, then the partial tiles [K][8][F] from the next 256-byte
// boundary. Every GPU the library runs on holds its own copy for the life of the process.

static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {

std::mutex scratchLock;
void* scratchAddress[kMaxDevices]; // device address of `scratch` per device, found once

// The address of the current device's `scratch`. In host code the array's name is only a stand-in
// for the symbol, never a device pointer, so the address is looked up once per device (with that
// device current) and reused.
void* deviceScratch() {
    int device = 0;
    checkHip(hipGetDevice(&device));
    if (device < 0 || device >= kMaxDevices)
        throw std::runtime_error("launchSpmmInt8NoAlloc: device index out of range");
    std::lock_guard<std::mutex> guard(scratchLock);
    if (!scratchAddress[device]) {
        void* address = nullptr;
        checkHip(hipGetSymbolAddress(&address, HIP_SYMBOL(scratch)));
        scratchAddress[device] = address;
    }
    return scratchAddress[device];
}

// Zero `count` words: a kernel rather than hipMemsetAsync, so the entry point can be captured into
// a HIP graph.
__global__ __launch_bounds__(256) void clearWords(unsigned* words, unsigned count) {
    for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < count; i += gridDim.x * 256) words[i] = 0;
}

} // namespace

void launchSpmmInt8NoAlloc(Sw32DeviceView matrix, const std::int8_t* packedX, const float* scales,
                           float* output, std::uint32_t rows, std::uint32_t cols,
                           std::uint32_t features, std::uint32_t partialCount, hipStream_t stream) {
    if (features != 128 && features != 256)
        throw std::invalid_argument("feature dimension must be 128 or 256");
    checkLaunchArguments(matrix, packedX, scales, output);
    SpmmWorkspace workspace;
    if (partialCount) {
        const std::uint64_t counters = (std::uint64_t(rows) + 31) / 32 * (features / 128);
        const std::uint64_t counterBytes = (counters * 4 + 255) / 256 * 256;
        const std::uint64_t partialBytes = std::uint64_t(partialCount) * 8 * features * 4;
        if (counterBytes + partialBytes > kNoAllocScratchBytes)
            throw std::invalid_argument(
                "launchSpmmInt8NoAlloc: the plan's " + std::to_string(partialCount) +
                " partial tiles at F=" + std::to_string(features) + " need " +
                std::to_string(counterBytes + partialBytes) + " bytes of scratch, more than its " +
                std::to_string(kNoAllocScratchBytes) + "; use launchSpmmInt8 with a workspace");
        unsigned char* base = static_cast<unsigned char*>(deviceScratch());
        workspace.counters = reinterpret_cast<std::uint32_t*>(base);
        workspace.partials = reinterpret_cast<float*>(base + counterBytes);
        // The counters must start at zero; a previous call leaves them at zero unless it failed.
        const unsigned blocks = unsigned(std::min<std::uint64_t>((counters + 255) / 256, 1024));
        hipLaunchKernelGGL(clearWords, dim3(blocks), dim3(256), 0, stream, workspace.counters,
                           unsigned(counters));
        checkHip(hipGetLastError());
    }
    launchSpmmInt8(matrix, packedX, scales, output, rows, cols, features, workspace, stream);
}
