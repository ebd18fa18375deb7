// Device-side helpers shared by the gfx950 LSSO kernels: bit-exact BF16/FP16
// conversions, MFMA operand types and the bounded complement.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace lsso_hip {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
// Operand of __builtin_amdgcn_ds_read_tr16_b64_v4i16: 16 lanes read 4 rows x 16
// columns of 16-bit values (lane i: 4 columns of row i / 4), and lane i receives
// the 4 rows of column i.
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 LdsS16x4;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// 1 - 2^-23: the one-ULP interior scale of the complement
// (reference lsso/ball/reference.py:464, csrc/ball/common.cuh:23).
constexpr float kInteriorScale = 1.0f - 0x1.0p-23f;
// log(e - 1), rounded to float32 as torch adds the Python double to a
// float32 tensor (reference lsso/ball/reference.py:13, 493).
constexpr float kSoftplusOneOffset = 0.541324854612918f;

__device__ __forceinline__ float bf16_lo(uint32_t packed) {
    return __uint_as_float(packed << 16);
}
__device__ __forceinline__ float bf16_hi(uint32_t packed) {
    return __uint_as_float(packed & 0xffff0000u);
}
__device__ __forceinline__ float bf16_bits_to_float(uint16_t bits) {
    return __uint_as_float(static_cast<uint32_t>(bits) << 16);
}
__device__ __forceinline__ float f16_lo(uint32_t packed) {
    return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(packed & 0xffffu)));
}
__device__ __forceinline__ float f16_hi(uint32_t packed) {
    return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(packed >> 16)));
}
__device__ __forceinline__ float f16_bits_to_float(uint16_t bits) {
    return static_cast<float>(__builtin_bit_cast(_Float16, bits));
}

// LDS ordering between lanes of one wave: its LDS instructions execute in
// issue order, so only the compiler must be kept from reordering.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The value unchanged, but opaque to the optimizer: lane-dependent offsets
// computed from it stay next to their use inside a loop instead of being
// hoisted out of it and held in registers across the whole loop.
__device__ __forceinline__ int opaque_int(int value) {
    asm volatile("" : "+v"(value));
    return value;
}

// Workgroups are dealt to the eight XCDs of an MI355X round robin (workgroup
// i runs on XCD i % 8, each XCD with its own L2).  A kernel whose
// neighbouring work items read the same rows calls this to renumber its
// workgroups so that consecutive logical blocks run on one XCD, one after
// the other: logical block xcd * (n / 8) + k is physical block 8 k + xcd.
// Blocks past the last whole round of eight keep their index.
__device__ __forceinline__ int64_t xcd_local_block(int64_t physical, int64_t blocks) {
    const int64_t per_xcd = blocks / 8;
    if (physical >= per_xcd * 8) {
        return physical;
    }
    return (physical % 8) * per_xcd + physical / 8;
}

// Raw buffer access.  An access past a buffer's num_records bytes does not
// touch memory: loads return zero and stores are dropped.  Tile loops use
// this instead of branches around their edge accesses, so every memory
// instruction issues unconditionally and the compiler's wait counts stay
// exact (a conditional access makes the waits before later uses
// conservative, which serializes a software pipeline).
typedef __amdgpu_buffer_rsrc_t BufferRsrc;
constexpr int kBufferConfig = 0x00020000;         // gfx9 raw buffer, 32-bit data format
constexpr uint32_t kOutOfRange = 0x80000000u;     // an offset past every buffer here

__device__ __forceinline__ BufferRsrc make_buffer(const void* base, int64_t bytes) {
    const int records = bytes < 0 ? 0 : (bytes > 0x7fffffff ? 0x7fffffff : static_cast<int>(bytes));
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, records, kBufferConfig);
}
__device__ __forceinline__ u32x4 buffer_load16(BufferRsrc buffer, uint32_t offset) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(buffer, offset, 0, 0));
}
__device__ __forceinline__ uint32_t buffer_load_byte(BufferRsrc buffer, uint32_t offset) {
    return __builtin_amdgcn_raw_buffer_load_b8(buffer, offset, 0, 0);
}
__device__ __forceinline__ void buffer_store16(u32x4 value, BufferRsrc buffer, uint32_t offset) {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(__attribute__((ext_vector_type(4))) unsigned int, value),
                                           buffer, offset, 0, 0);
}
__device__ __forceinline__ void buffer_store_f32(float value, BufferRsrc buffer, uint32_t offset) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(value), buffer, offset, 0, 0);
}
// Streaming forms: the cache-policy operand 2 sets the instruction's `nt`
// bit, so the lines are kept in the caches as streaming (first to be
// evicted).  Used for the bulk token tensors a kernel touches once, so
// that they do not push out what is reused (weights, phase tables,
// partials, records, and the second head group's read of an x tile).  The
// store adds `sc1` (operand 16): a streaming write of 1 GiB with `nt` alone
// runs about 5% slower than a plain one, with `nt` and `sc1` as fast.
__device__ __forceinline__ u32x4 buffer_load16_stream(BufferRsrc buffer, uint32_t offset) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(buffer, offset, 0, 2));
}
__device__ __forceinline__ void buffer_store16_stream(u32x4 value, BufferRsrc buffer, uint32_t offset) {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(__attribute__((ext_vector_type(4))) unsigned int, value),
                                           buffer, offset, 0, 2 | 16);
}

// Pieces of rows that are not whole 16-byte pieces (odd lengths, strides or
// bases).  A piece is one 16-byte access at an address aligned to its elements
// only: it starts early enough to end within its row, so that it never leaves
// the matrix, and is moved down by the elements it started early, which brings
// zeros in past the row's end.  Element by element, a piece took eight loads,
// eight registers in flight and eight conditional addresses.
__device__ __forceinline__ u32x4 load16_unaligned(const void* at) {
    u32x4 v;
    __builtin_memcpy(&v, at, sizeof(v));
    return v;
}
__device__ __forceinline__ void store16_unaligned(void* at, const u32x4& v) {
    __builtin_memcpy(at, &v, sizeof(v));
}
// First element of the access to elements k .. k + N - 1 of a row of `cols` >= N.
template <int N, typename I>
__device__ __forceinline__ I piece_start(I k, I cols) {
    return k < cols - N ? k : cols - N;
}
__device__ __forceinline__ u32x4 drop_dwords(const u32x4& v, uint32_t count) {   // zeros from 4 on
    u32x4 out = (count & 2) != 0 ? (u32x4){v[2], v[3], 0u, 0u} : v;
    out = (count & 1) != 0 ? (u32x4){out[1], out[2], out[3], 0u} : out;
    return count < 4 ? out : (u32x4){0u, 0u, 0u, 0u};
}
// 16-bit elements k .. k + 7 from the access at piece_start<8>(k, cols).
template <typename I>
__device__ __forceinline__ u32x4 align_piece16(const u32x4& raw, I k, I cols) {
    const I start = piece_start<8>(k, cols);
    const uint32_t early = k - start < 8 ? static_cast<uint32_t>(k - start) : 8u;
    const u32x4 v = drop_dwords(raw, early >> 1);
    const u32x4 odd = {(v[0] >> 16) | (v[1] << 16), (v[1] >> 16) | (v[2] << 16), (v[2] >> 16) | (v[3] << 16), v[3] >> 16};
    return (early & 1) != 0 ? odd : v;
}
// 16-bit elements k .. k + 7 of a row of `cols` < 8, which holds no whole piece.
__device__ __forceinline__ u32x4 load_short_piece(const uint16_t* row, int k, int cols) {
    u32x4 out = {0u, 0u, 0u, 0u};
    if (k == 0) {
        for (int i = 0; i < cols; ++i) {
            const uint32_t bits = static_cast<uint32_t>(row[i]) << (16 * (i & 1));
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                out[p] |= p == i / 2 ? bits : 0u;
            }
        }
    }
    return out;
}
// 32-bit elements k .. k + 3 from the access at piece_start<4>(k, cols).
template <typename I>
__device__ __forceinline__ u32x4 align_piece32(const u32x4& raw, I k, I cols) {
    const I start = piece_start<4>(k, cols);
    return drop_dwords(raw, k - start < 4 ? static_cast<uint32_t>(k - start) : 4u);
}

// Round two floats to BF16 (round to nearest even, v_cvt_pk_bf16_f32) and
// pack them, first value in the low half.
__device__ __forceinline__ uint32_t pack_bf16(float low, float high) {
    const bf16x2 value = __builtin_convertvector((f32x2){low, high}, bf16x2);
    return __builtin_bit_cast(uint32_t, value);
}
__device__ __forceinline__ uint16_t to_bf16_bits(float value) {
    return static_cast<uint16_t>(pack_bf16(value, 0.0f) & 0xffffu);
}
__device__ __forceinline__ uint16_t to_f16_bits(float value) {
    return __builtin_bit_cast(uint16_t, static_cast<_Float16>(value));
}
__device__ __forceinline__ uint32_t pack_f16(float low, float high) {
    return static_cast<uint32_t>(to_f16_bits(low)) |
           (static_cast<uint32_t>(to_f16_bits(high)) << 16);
}

// Split two floats into BF16 high parts and BF16 residuals so that
// hi + lo carries ~16 mantissa bits; products of split operands accumulated
// as hi*hi + hi*lo + lo*hi reproduce FP32 products to ~2^-17 relative.
__device__ __forceinline__ void split_bf16(float a, float b, uint32_t& hi, uint32_t& lo) {
    hi = pack_bf16(a, b);
    lo = pack_bf16(a - bf16_lo(hi), b - bf16_hi(hi));
}

__device__ __forceinline__ f32x4 mfma16x16x32(const u32x4& a, const u32x4& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
        __builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16x16x16(const u32x2& a, const u32x2& b, const f32x4& c) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
        __builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma32x32x16(const u32x4& a, const u32x4& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(
        __builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// eta = (1 - 2^-23) tanh(raw) through the sign-split logistic identity
// (reference lsso/ball/reference.py:450-471).
__device__ __forceinline__ float bounded_complement(float raw) {
    const bool positive = raw >= 0.0f;
    const float exponent = positive ? expf(-2.0f * raw) : expf(2.0f * raw);
    const float numerator = positive ? 1.0f - exponent : exponent - 1.0f;
    return kInteriorScale * (numerator / (1.0f + exponent));
}

// d eta / d raw of bounded_complement (reference csrc/ball/common.cuh:30-34).
__device__ __forceinline__ float bounded_complement_derivative(float raw) {
    const float exponent = raw >= 0.0f ? expf(-2.0f * raw) : expf(2.0f * raw);
    const float denominator = 1.0f + exponent;
    return kInteriorScale * 4.0f * exponent / (denominator * denominator);
}

// torch.nn.functional.softplus with beta=1, threshold=20.
__device__ __forceinline__ float softplus_one(float raw) {
    const float shifted = raw + kSoftplusOneOffset;
    return shifted > 20.0f ? shifted : log1pf(expf(shifted));
}

// Rotate one (even, odd) relation pair by an FP16 (cos, sin) phase.  The
// BF16 x FP16 products are exact in FP32, so the one rounding of each sum
// matches the reference's FP32 rotation (reference.py:719-723).
__device__ __forceinline__ void rotate_pair(uint32_t relation_pair, uint32_t phase,
                                            float& even_out, float& odd_out) {
    const float even = bf16_lo(relation_pair);
    const float odd = bf16_hi(relation_pair);
    const float cosine = f16_lo(phase);
    const float sine = f16_hi(phase);
    even_out = even * cosine - odd * sine;
    odd_out = even * sine + odd * cosine;
}

// Apply operand layout: the rank dimension is the MFMA K index.  Ranks that
// are multiples of 32 use K32 steps (16x16x32; lane group g holds ranks
// base + 8g .. +7), the others K16 steps (16x16x16; ranks base + 4g .. +3).
// One accumulation chain never mixes the two MFMA shapes: a 16x16x32 result
// consumed as SrcC of a 16x16x16 produced wrong accumulators on gfx950 with
// this toolchain.  Per lane the M' operand holds, per step, the hi values
// followed by the lo values.
template <int R>
struct ApplyLayout {
    static constexpr bool kWide = (R % 32) == 0;
    static constexpr int kSteps32 = kWide ? R / 32 : 0;
    static constexpr int kSteps16 = kWide ? 0 : R / 16;
    static constexpr int kLaneValues = R / 4;          // per hi or lo part
    static constexpr int kLaneHalfs = 2 * kLaneValues;  // bf16 per lane per block
    __device__ static constexpr int rank32(int s, int g, int i) { return 32 * s + 8 * g + i; }
    __device__ static constexpr int rank16(int s, int g, int i) { return 16 * s + 4 * g + i; }
    // offsets (in bf16) of the hi part of a step inside a lane record
    __device__ static constexpr int offset32(int s) { return 16 * s; }
    __device__ static constexpr int offset16(int s) { return 8 * s; }
};

// Resident BF16 rows of an FP32 weight [N, K] for y^T = W x^T on
// v_mfma_f32_32x32x16_bf16: NB x 32 rows of which lane i holds row i % 32 at
// columns 16 ks + 8 (i / 32) + 0..7, RNE-rounded, zero past K.  Coalesced: 8
// lanes read one row's 32 columns (one 128-byte line) per 16-byte load, the
// BF16 values pass through `scratch` (kWeightScratch bf16 of LDS of this wave's
// own, so no barrier) and come back in the lane layout.  row_offset(nb, r) is
// the byte offset of row r of block nb in the raw buffer, or kOutOfRange.
// WHOLE: rows of whole 4-column pieces (K a multiple of 4); else K is at least
// 4 and the last piece of a row is read from 4 columns before its end.  A
// buffer access of several dwords needs dword alignment only, so any FP32
// weight will do.  A persistent kernel cannot start its first tile before its
// weights are in registers.  Read by the lanes that keep them (row n at 16
// bytes per lane, one K step at a time), every load touches 32 lines for a
// quarter of their bytes and waits for the one before; with eight steps in
// flight instead, the lines of all waves no longer fit the L1 and are fetched
// four times (the training step at 262,144 tokens 4% slower).  Four 2-step
// pieces are in flight here; the scheduling barriers keep the FP32 staging of
// the whole slice from being live at once.  With it the layer call at 64 x
// 1,024 x 256 (rank 32) takes 84 us instead of 92, at 64 x 4,096 212 instead of
// 221.
constexpr int kWeightPitch = 40;                      // bf16 per row of 32: 16 rows' 16-byte reads cover all banks
constexpr int kWeightScratch = 32 * kWeightPitch;     // bf16 per wave
constexpr int kWeightRing = 4;
template <bool WHOLE, int NB, int KSTEPS, typename RowOffset>
__device__ __forceinline__ void load_weight_rows(u32x4 (&wreg)[NB][KSTEPS], BufferRsrc buffer, RowOffset row_offset,
                                                 int64_t K, int lane, uint16_t* scratch) {
    static_assert(KSTEPS % 2 == 0, "a piece is two K steps");
    constexpr int kPieces = KSTEPS / 2;
    constexpr int kTotal = NB * kPieces;
    constexpr int kRing = kTotal < kWeightRing ? kTotal : kWeightRing;
    const int row8 = lane >> 3;
    const uint32_t k_lane = 4 * (lane & 7);
    const uint32_t k_end = static_cast<uint32_t>(K);
    uint32_t offset[NB][4];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            offset[nb][j] = row_offset(nb, 8 * j + row8);
        }
    }
    u32x4 raw[kRing][4];
    const auto start = [&](uint32_t k0) { return WHOLE ? k0 : piece_start<4>(k0, k_end); };
    auto issue = [&](int i) {
        const uint32_t k0 = 32 * (i % kPieces) + k_lane;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t row = offset[i / kPieces][j];
            raw[i % kRing][j] =
                buffer_load16(buffer, k0 < k_end && row != kOutOfRange ? row + 4 * start(k0) : kOutOfRange);
        }
    };
#pragma unroll
    for (int i = 0; i < kRing; ++i) {
        issue(i);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kTotal; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const u32x4 piece = raw[i % kRing][j];
            const f32x4 v = __builtin_bit_cast(
                f32x4, WHOLE ? piece : align_piece32<uint32_t>(piece, 32 * (i % kPieces) + k_lane, k_end));
            const u32x2 packed = {pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
            *reinterpret_cast<u32x2*>(scratch + (8 * j + row8) * kWeightPitch + k_lane) = packed;
        }
        if (i + kRing < kTotal) {
            issue(i + kRing);
        }
        // Written and read by different lanes of the wave.
        wave_lds_order();
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            wreg[i / kPieces][2 * (i % kPieces) + s] = *reinterpret_cast<const u32x4*>(
                scratch + (lane & 31) * kWeightPitch + 16 * s + 8 * (lane >> 5));
        }
        wave_lds_order();   // the next piece's writes follow these reads
        __builtin_amdgcn_sched_barrier(0);
    }
}

// load_weight_rows of rows n0 .. n0 + 31 (n0 wave-uniform; rows past N are
// zeros); whole: K is a multiple of 4.
template <int KSTEPS>
__device__ __forceinline__ void load_weight_slice(u32x4 (&wreg)[1][KSTEPS], const float* weight,
                                                  int64_t N, int64_t K, int64_t n0, int lane, bool whole,
                                                  uint16_t* scratch) {
    const int64_t rows = N - n0 < 32 ? N - n0 : 32;
    const BufferRsrc buffer = make_buffer(weight + (n0 < N ? n0 : 0) * K, 4 * rows * K);
    const auto row_offset = [&](int, int r) { return static_cast<uint32_t>(4 * r * K); };
    if (whole) {   // uniform
        load_weight_rows<true, 1, KSTEPS>(wreg, buffer, row_offset, K, lane, scratch);
    } else {
        load_weight_rows<false, 1, KSTEPS>(wreg, buffer, row_offset, K, lane, scratch);
    }
}

}  // namespace lsso_hip
