// gfx950 biased projection y = cast(bf16(x) bf16(W)^T + b).
//
// Contract (reference lsso/ball/reference.py:20-75, 170-203, 347-408): BF16
// multiplicands (x rounded to BF16 with round-to-nearest-even, W likewise),
// FP32 accumulation, FP32 bias added to the accumulator, one final FP16 or
// BF16 store; FP16 output never rounds through BF16.
//
// Schedule: persistent workgroups of 8 waves.  Each wave keeps a 32-column
// slice of W (BF16, K padded to 16) in registers for the whole launch, so the
// weights are read once per workgroup.  64-row x tiles (32-row once K > 384,
// where W takes 128 or 160 of a wave's 256 registers) are staged through a
// double-buffered LDS tile (converted to BF16 once) and shared by the
// workgroup's waves.
// The MFMA computes y^T = W x^T on v_mfma_f32_32x32x16_bf16; in that form a
// lane's accumulators are 4 runs of 4 consecutive output features of one
// row.  The rounded tile is staged in LDS and written back in 16-byte pieces
// of whole row segments (scattered 8-byte writes cost half the store rate).
//
// Bound: HBM, by the latency of the tile loads.  A tile's products take about
// 1 us, a load under traffic 2 to 4, so one tile in flight (32 KB per CU) ran
// the loop at the latency's pace.  Two tiles are in flight in registers (one at
// K > 512) while a third is multiplied, and a piece is converted and its
// registers reloaded between two MFMAs, so the conversions hide under them.
// Up to K = 640 a wave holds all of K: at K > 384 the former form shared a
// 32-column slice between two waves, half of K each, and read x twice for
// 256 outputs.  Before and now (us): 262,144 x 256 -> 256 68 / 57, x 512 -> 256
// 142 / 98, 131,072 x 640 -> 256 79 / 55, x 256 -> 640 84 / 68, x 384 -> 768
// 111 / 97.
//
// Rows, strides, bases and outputs that are not whole aligned 16-byte pieces
// run the same loop (a second instantiation) on pieces aligned to their
// elements.  Element by element (eight loads and eight addresses a piece beside
// the resident W) that form spilled 25 to 187 registers, and one odd operand
// put all of them on it.  Element loads with W shared by two waves from K =
// 385, the former element loads, these pieces (us, 65,536 rows): 256 -> 260
// 55 / 68 / 34, 300 -> 300 185 / 228 / 41, 640 -> 260 75 / 209 / 53, 256 -> 256
// at an odd stride 38 / 46 / 20; K-streaming, 16,384 rows: 768 -> 1,001 88 /
// 276 / 58, 1,001 -> 768 307 / 222 / 61.

#include "lsso_device.h"
#include "lsso_internal.h"
#include "lsso_hip.h"

namespace lsso_hip {

constexpr int kXcds = 8;   // accelerator complex dies of an MI355X
constexpr int kStreamRowsHost = 128;   // tile of the K-streaming tier
constexpr int kStreamColsHost = 128;

// Rows per x tile: 64, or 32 once K exceeds 384.
template <int KSTEPS>
constexpr int linear_tile_rows_k() { return KSTEPS <= 24 ? 64 : 32; }

// Waves per workgroup: eight, two per SIMD at up to 256 registers each, of
// which a wave's 32-column W slice takes 4 per K step (160 at K = 640).
constexpr int kLinearWaves = 8;

// Instruction classes of __builtin_amdgcn_sched_group_barrier.
constexpr int kSchedValu = 0x2;
constexpr int kSchedMfma = 0x8;
constexpr int kSchedDsRead = 0x100;
constexpr int kSchedDsWrite = 0x200;

// Tier 0 is the K-streaming kernel (any in_features above 640).
int linear_tile_rows(int k_steps) { return k_steps == 0 ? kStreamRowsHost : (k_steps <= 24 ? 64 : 32); }
int linear_columns_per_group(int k_steps) {
    return k_steps == 0 ? kStreamColsHost : kLinearWaves * 32;
}

int linear_k_tier(int64_t in_features) {
    if (in_features <= 64) return 4;
    if (in_features <= 128) return 8;
    if (in_features <= 192) return 12;
    if (in_features <= 256) return 16;
    if (in_features <= 384) return 24;
    if (in_features <= 512) return 32;
    if (in_features <= 640) return 40;
    return 0;   // K-streaming tier
}

// BF16 bits of a 16-byte piece of x as loaded.
template <int XT>
__device__ __forceinline__ u32x4 to_bf16_piece(const u32x4& raw) {
    u32x4 out = raw;
    if constexpr (XT == LSSO_HIP_F16) {
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            out[p] = pack_bf16(f16_lo(raw[p]), f16_hi(raw[p]));
        }
    }
    return out;
}

// Weight rows of fewer than 8 elements, element by element.
template <int KSTEPS>
__device__ __forceinline__ void load_short_weights(u32x4 (&wreg)[1][KSTEPS], const float* weight, int64_t N, int K,
                                                   int64_t n, int lane) {
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) {
        wreg[0][ks] = (u32x4){0u, 0u, 0u, 0u};
    }
    if (lane < 32 && n < N) {
        for (int i = 0; i < K; ++i) {
            const uint32_t bits = static_cast<uint32_t>(to_bf16_bits(weight[n * K + i])) << (16 * (i & 1));
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                wreg[0][0][p] |= p == i / 2 ? bits : 0u;
            }
        }
    }
}

// A 16-byte piece of an output row at column n, of which the row may hold
// fewer than eight elements.
__device__ __forceinline__ void store_piece(uint16_t* row, int64_t n, int64_t N, const u32x4& v) {
    if (n + 8 <= N) {
        store16_unaligned(row + n, v);
    } else {
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            if (n + r < N) {
                row[n + r] = static_cast<uint16_t>(v[r >> 1] >> (16 * (r & 1)));
            }
        }
    }
}

// VEC: whole 16-byte pieces of x and y (a.vector); else pieces aligned to their
// elements (x) and stores of whole or part pieces (y).
template <int KSTEPS, int XT, int YT, bool VEC>
__global__ __launch_bounds__(kLinearWaves * 64) void linear_kernel(LinearArgs a) {
    constexpr int kWaves = kLinearWaves;
    constexpr int kTileRows = linear_tile_rows_k<KSTEPS>();
    constexpr int MB = kTileRows / 32;                  // 32-row MFMA blocks per tile
    constexpr int kGroupColumns = kWaves * 32;
    constexpr int KP = 16 * KSTEPS + 8;                  // LDS row pitch (bf16)
    constexpr int kChunksPerRow = 2 * KSTEPS;           // 8-element chunks
    constexpr int kThreads = kWaves * 64;
    constexpr int kChunksPerThread = kTileRows * kChunksPerRow / kThreads;
    static_assert(kTileRows * kChunksPerRow % kThreads == 0, "tile split");
    __shared__ __attribute__((aligned(16))) uint16_t s_x[2][kTileRows * KP];
    __shared__ __attribute__((aligned(16))) float s_bias[kGroupColumns];
    constexpr int YP = kGroupColumns + 8;                 // staged output row pitch
    constexpr int kStoreChunks = kTileRows * kGroupColumns / 8 / kThreads;
    static_assert(kTileRows * kGroupColumns / 8 % kThreads == 0, "store split");
    __shared__ __attribute__((aligned(16))) uint16_t s_y[kTileRows * YP];
    // Row flags of the tile being multiplied and of the next one.
    __shared__ int s_keep[2][kTileRows];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // scalar: the weight buffer below is
    const int half = lane >> 5;
    // Workgroups are dealt to the eight XCDs round-robin by block index.  When
    // the grid allows, the column groups of one row tile are given to blocks
    // of the same XCD, so the second read of each x tile hits that XCD's L2.
    int64_t cg, group_index;
    if (gridDim.x % (kXcds * a.column_groups) == 0) {
        const int64_t xcd = blockIdx.x % kXcds;
        const int64_t slot = blockIdx.x / kXcds;
        cg = slot % a.column_groups;
        group_index = (slot / a.column_groups) * kXcds + xcd;
    } else {
        cg = blockIdx.x % a.column_groups;
        group_index = blockIdx.x / a.column_groups;
    }
    const int64_t group_count = gridDim.x / a.column_groups;
    const int slice = wave;
    const int64_t n0 = cg * kGroupColumns + slice * 32;
    const int64_t K = a.in_features;
    const int64_t N = a.out_features;

    u32x4 wreg[1][KSTEPS];
    // The output stage (or, where it is too small, the second x tile) is not
    // written before the first tile's products.
    constexpr bool kStageHolds = kTileRows * YP >= kWaves * kWeightScratch;
    static_assert(kStageHolds || kTileRows * KP >= kWaves * kWeightScratch, "weight scratch");
    // Rows too short for a piece: only where they would be the lowest tier's.
    const bool short_rows = !VEC && KSTEPS == 4 && K < 8;   // uniform
    if (short_rows) {
        load_short_weights<KSTEPS>(wreg, a.weight, N, static_cast<int>(K), n0 + (lane & 31), lane);
    } else {
        load_weight_slice<KSTEPS>(wreg, a.weight, N, K, n0, lane, VEC || K % 4 == 0,
                                  (kStageHolds ? s_y : s_x[1]) + wave * kWeightScratch);
    }
    for (int c = tid; c < kGroupColumns; c += kThreads) {
        const int64_t n = cg * kGroupColumns + c;
        s_bias[c] = (a.bias != nullptr && n < N) ? a.bias[n] : 0.0f;
    }

    // One tile of x in flight: 16-byte pieces as loaded and the row's mask byte.  Row flags travel with their x: thread r <
    // kTileRows reads the byte of row r through a raw buffer over the tile's
    // valid rows (rows past the matrix, and every row when there is no mask,
    // read as zero without an access).
    struct Stage {
        u32x4 x[kChunksPerThread];
        uint32_t mask;
        int64_t rows;
    };
    const uint16_t* x = static_cast<const uint16_t*>(a.x);
    constexpr bool kWholeRows = kThreads % kChunksPerRow == 0;
    const int piece_k = 8 * (tid % kChunksPerRow);
    const uint32_t piece0 = piece_k < K ? 2u * static_cast<uint32_t>(tid / kChunksPerRow * static_cast<int>(a.x_stride) + piece_k)
                                        : kOutOfRange;
    const uint32_t piece_step = piece_k < K ? 2u * static_cast<uint32_t>(kThreads / kChunksPerRow) *
                                                  static_cast<uint32_t>(a.x_stride) : 0u;
    auto load_chunk = [&](Stage& stage, int64_t t, BufferRsrc buffer, int c) {
        // Without VEC, a piece's place is worked out where it is used.
        const int chunk = VEC ? tid + c * kThreads : opaque_int(tid + c * kThreads);
        const int rr = chunk / kChunksPerRow;
        const int k0 = 8 * (chunk - rr * kChunksPerRow);
        if constexpr (VEC) {
            // Rows past the matrix end the buffer; columns past K get an
            // offset beyond it.  Where the workgroup covers whole rows, a
            // thread keeps its column and one offset serves all its pieces.
            if constexpr (kWholeRows) {
                stage.x[c] = buffer_load16(buffer, piece0 + c * piece_step);
            } else {
                const int rr_c = opaque_int(rr);
                stage.x[c] = buffer_load16(
                    buffer, k0 < K ? 2u * static_cast<uint32_t>(rr_c * static_cast<int>(a.x_stride) + k0) : kOutOfRange);
            }
        } else {
            // Rows past the matrix read its last row: their outputs are not stored.
            const int64_t row = t * kTileRows + rr < a.rows ? t * kTileRows + rr : a.rows - 1;
            const uint16_t* at = x + row * a.x_stride;
            const int cols = static_cast<int>(K);
            stage.x[c] = short_rows ? load_short_piece(at, k0, cols) : load16_unaligned(at + piece_start<8>(k0, cols));
        }
    };
    auto tile_buffer = [&](int64_t t) {
        return make_buffer(x + t * kTileRows * a.x_stride, 2 * (a.rows - t * kTileRows) * a.x_stride);
    };
    auto load_flags = [&](Stage& stage, int64_t t) {
        stage.rows = a.rows - t * kTileRows;
        const BufferRsrc mask = make_buffer(a.row_mask != nullptr ? a.row_mask + t * kTileRows : nullptr,
                                            a.row_mask != nullptr ? stage.rows : 0);
        stage.mask = buffer_load_byte(mask, static_cast<uint32_t>(tid));
    };
    auto load_stage = [&](Stage& stage, int64_t t) {
        const BufferRsrc buffer = tile_buffer(t);
#pragma unroll
        for (int c = 0; c < kChunksPerThread; ++c) {
            load_chunk(stage, t, buffer, c);
        }
        load_flags(stage, t);
    };
    auto write_chunk = [&](const Stage& stage, int buf, int c) {
        const int chunk = VEC ? tid + c * kThreads : opaque_int(tid + c * kThreads);
        const int rr = chunk / kChunksPerRow;
        const int cc = chunk - rr * kChunksPerRow;
        const u32x4 piece = VEC || short_rows ? stage.x[c] : align_piece16(stage.x[c], 8 * cc, static_cast<int>(K));
        *reinterpret_cast<u32x4*>(&s_x[buf][rr * KP + 8 * cc]) = to_bf16_piece<XT>(piece);
    };
    auto write_flags = [&](const Stage& stage, int buf) {
        if (tid < kTileRows) {
            s_keep[buf][tid] = tid < stage.rows && (a.row_mask == nullptr || stage.mask != 0);
        }
    };

    // One tile from LDS buffer `buf`.  `stage` holds the next tile of this
    // workgroup, loaded two tiles ago (one where the registers hold a single
    // stage): between the MFMAs its pieces are converted into the other buffer,
    // and each piece's registers take their piece of the tile `ahead`.  Memory
    // operations complete in issue order as far as the wait counter is
    // concerned and nothing here is conditional, so each wait covers that one
    // stage only: the stage behind it and the y stores stay in flight.
    auto step = [&](int buf, int64_t tile, Stage& stage, int64_t ahead) {
        bool keep[MB];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            keep[mb] = s_keep[buf][mb * 32 + (lane & 31)] != 0;
        }
        // The FP32 bias is the accumulators' starting value: element 4 qd + e
        // is feature slice * 32 + 8 qd + 4 half + e of the group.
        f32x16 acc[MB];
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
            const f32x4 bias = *reinterpret_cast<const f32x4*>(&s_bias[slice * 32 + 8 * qd + 4 * half]);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    acc[mb][4 * qd + e] = bias[e];
                }
            }
        }
        // Operand reads run one group of two K steps ahead of the MFMAs, so
        // at most eight x fragments are live next to the resident W slice.
        constexpr int kGroup = 2;
        constexpr int kGroups = KSTEPS / kGroup;
        u32x4 xb[2][kGroup][MB];
        auto read_group = [&](int slot, int k_base) {
#pragma unroll
            for (int ks = 0; ks < kGroup; ++ks) {
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) {
                    xb[slot][ks][mb] = *reinterpret_cast<const u32x4*>(
                        &s_x[buf][(mb * 32 + (lane & 31)) * KP + 16 * (k_base + ks) + 8 * half]);
                }
            }
        };
        const BufferRsrc buffer = tile_buffer(ahead);
        read_group(0, 0);
#pragma unroll
        for (int g = 0; g < kGroups; ++g) {
            const int slot = g & 1;
            if (g + 1 < kGroups) {
                read_group(slot ^ 1, kGroup * (g + 1));
            }
#pragma unroll
            for (int ks = 0; ks < kGroup; ++ks) {
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) {
                    acc[mb] = mfma32x32x16(wreg[0][kGroup * g + ks], xb[slot][ks][mb], acc[mb]);
                }
            }
            // This group's share of the next tile's pieces.
#pragma unroll
            for (int c = 0; c < kChunksPerThread; ++c) {
                if (c * kGroups / kChunksPerThread == g) {
                    write_chunk(stage, buf ^ 1, c);
                    load_chunk(stage, ahead, buffer, c);
                }
            }
            __builtin_amdgcn_sched_group_barrier(kSchedDsRead, kGroup * MB, 0);
#pragma unroll
            for (int i = 0; i < kGroup * MB; ++i) {
                __builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 0);
                __builtin_amdgcn_sched_group_barrier(kSchedValu, 6, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        write_flags(stage, buf ^ 1);
        load_flags(stage, ahead);
        // y^T block: lane holds row m = lane%32 of the 32-row block and
        // features n0 + 8 q + 4 half + r for q, r in 0..3.  The tile is
        // rounded and staged in LDS, then written back row by row so that
        // each store instruction covers whole contiguous row segments.
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            const int mr = mb * 32 + (lane & 31);
            if (__ballot(keep[mb]) != ~0ull) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    acc[mb][i] = keep[mb] ? acc[mb][i] : 0.0f;
                }
            }
#pragma unroll
            for (int qd = 0; qd < 4; ++qd) {
                const int c = slice * 32 + 8 * qd + 4 * half;
                const float v0 = acc[mb][4 * qd + 0];
                const float v1 = acc[mb][4 * qd + 1];
                const float v2 = acc[mb][4 * qd + 2];
                const float v3 = acc[mb][4 * qd + 3];
                u32x2 packed;
                if constexpr (YT == LSSO_HIP_BF16) {
                    packed.x = pack_bf16(v0, v1);
                    packed.y = pack_bf16(v2, v3);
                } else {
                    packed.x = pack_f16(v0, v1);
                    packed.y = pack_f16(v2, v3);
                }
                *reinterpret_cast<u32x2*>(&s_y[mr * YP + c]) = packed;
            }
        }
        __syncthreads();
        const int64_t col0 = cg * kGroupColumns;
        if constexpr (VEC) {
            // 16-byte pieces through a raw buffer over the tile's valid rows:
            // pieces past the matrix are dropped without a branch.
            const int64_t tile_rows = a.rows - tile * kTileRows < kTileRows ? a.rows - tile * kTileRows : kTileRows;
            const BufferRsrc ybuf = make_buffer(static_cast<uint16_t*>(a.y) + tile * kTileRows * N, 2 * tile_rows * N);
#pragma unroll
            for (int i = 0; i < kStoreChunks; ++i) {
                const int chunk = tid + i * kThreads;
                const int mr = chunk / (kGroupColumns / 8);
                const int c8 = 8 * (chunk - mr * (kGroupColumns / 8));
                const int64_t n = col0 + c8;
                buffer_store16(*reinterpret_cast<const u32x4*>(&s_y[mr * YP + c8]), ybuf,
                               n < N ? 2u * static_cast<uint32_t>(mr * N + n) : kOutOfRange);
            }
        } else {
#pragma unroll
            for (int i = 0; i < kStoreChunks; ++i) {
                const int chunk = tid + i * kThreads;
                const int mr = chunk / (kGroupColumns / 8);
                const int c8 = 8 * (chunk - mr * (kGroupColumns / 8));
                const int64_t m = tile * kTileRows + mr;
                const int64_t n = col0 + c8;
                if (m < a.rows && n < N) {
                    store_piece(static_cast<uint16_t*>(a.y) + m * N, n, N,
                                *reinterpret_cast<const u32x4*>(&s_y[mr * YP + c8]));
                }
            }
        }
        __syncthreads();
    };

    int64_t tile = group_index;
    if (tile >= a.tiles) {
        return;
    }
    // Stages of x in flight: two where the registers hold them beside W and,
    // without VEC, the pieces' places.
    constexpr int kSets = KSTEPS == 40 || (!VEC && KSTEPS == 24) ? 1 : 2;
    constexpr int kAhead = kSets + 1;
    Stage sets[kSets];
    load_stage(sets[0], tile);
    if constexpr (kSets == 2) {
        load_stage(sets[1], tile + group_count);
    }
#pragma unroll
    for (int c = 0; c < kChunksPerThread; ++c) {
        write_chunk(sets[0], 0, c);
    }
    write_flags(sets[0], 0);
    load_stage(sets[0], tile + kSets * group_count);
    __syncthreads();
    for (;;) {
        step(0, tile, sets[kSets - 1], tile + kAhead * group_count);
        tile += group_count;
        if (tile >= a.tiles) {
            break;
        }
        step(1, tile, sets[0], tile + kAhead * group_count);
        tile += group_count;
        if (tile >= a.tiles) {
            break;
        }
    }
}

// ---------------------------------------------------------------------------
// K-streaming tier (in_features > 640): the W rows no longer fit the waves'
// registers, so both operands stream through LDS.  A workgroup of four waves
// computes a 128-row x 128-column output tile; each wave a 64 x 64 quarter
// (2 x 2 blocks of v_mfma_f32_32x32x16_bf16 on y^T = W x^T).  The K order is
// one FP32 chain per output, ascending.  Row tiles sharing x are dealt to one
// XCD.
//
// Bound: the matrix cores and LDS (a stage's fragments and writes take about
// 1.5 times its MFMA cycles), where enough workgroups share a CU to cover each
// other's prologue and epilogue.  K is taken in stages of 32: two stages of
// loads are in flight in registers while a third is multiplied, and the next
// stage's conversions (W FP32 to BF16, x FP16 to BF16, round to nearest even)
// and LDS writes run between its MFMAs.  The output tile is staged in the
// operands' LDS, which leaves 40 KB per workgroup and three workgroups per CU;
// the former kernel (64-wide stages, one in flight, 107 KB) had one.  (FP16 x
// keeps two: at three, its conversions spill inside the loop, and a scratch
// load there waits for the loads in flight.)  Before and now (us, graph launch
// included): 12,608 x 768 -> 1,344 91 / 56, 8,192 x 768 -> 1,344 57 / 36, x 1,344
// -> 768 59 / 36, x 768 -> 768 38 / 26.
constexpr int kStreamRows = 128;
constexpr int kStreamCols = 128;
constexpr int kStreamK = 32;
constexpr int kStreamThreads = 256;

// VEC: whole 16-byte pieces of x, W and y; else pieces aligned to their
// elements (rows here are longer than a piece).
template <int XT, int YT, bool VEC>
__global__ __launch_bounds__(kStreamThreads, VEC && XT == LSSO_HIP_BF16 ? 3 : 2) void linear_stream_kernel(LinearArgs a) {
    constexpr int KP = kStreamK + 8;                 // LDS row pitch (bf16): 16 rows' 16-byte reads cover all banks
    constexpr int YP = kStreamCols + 8;
    constexpr int kXPieces = kStreamRows * kStreamK / 8 / kStreamThreads;   // 16-byte pieces per thread and stage
    constexpr int kWPieces = kStreamCols * kStreamK / 4 / kStreamThreads;
    constexpr int kXRows = kStreamThreads / (kStreamK / 8);   // rows between a thread's pieces
    constexpr int kWRows = kStreamThreads / (kStreamK / 4);
    constexpr int kOperand = kStreamRows * KP;
    static_assert(kStreamRows == kStreamCols && kStreamRows * YP <= 4 * kOperand, "the output tile fits the operands'");
    // Two buffers of (x, W); afterwards the output tile.
    __shared__ __attribute__((aligned(16))) uint16_t s_t[4 * kOperand];
    __shared__ __attribute__((aligned(16))) float s_bias[kStreamCols];
    __shared__ int s_keep[kStreamRows];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5;
    const int64_t M = a.rows;
    const int64_t N = a.out_features;
    const int64_t K = a.in_features;
    const int64_t tiles_n = a.column_groups;
    // Block b runs on XCD b % 8; the column tiles of one row tile share it.
    const int64_t xcd = blockIdx.x % kXcds;
    const int64_t slot = blockIdx.x / kXcds;
    const int64_t mt = (slot / tiles_n) * kXcds + xcd;
    const int64_t nt = slot % tiles_n;
    if (mt >= a.tiles) {
        return;
    }
    const int64_t m0 = mt * kStreamRows;
    const int64_t n0 = nt * kStreamCols;

    struct Stage {
        u32x4 x[kXPieces];
        u32x4 w[kWPieces];
    };
    const uint16_t* x = static_cast<const uint16_t*>(a.x) + m0 * a.x_stride;
    const float* w = a.weight + n0 * K;
    const int x_row = tid / (kStreamK / 8);
    const int x_k = 8 * (tid % (kStreamK / 8));
    const int w_row = tid / (kStreamK / 4);
    const int w_k = 4 * (tid % (kStreamK / 4));
    const uint32_t x_at = 2u * static_cast<uint32_t>(x_row * static_cast<int>(a.x_stride) + x_k);
    const uint32_t w_at = 4u * static_cast<uint32_t>(w_row * static_cast<int>(K) + w_k);
    const uint32_t x_step = 2u * static_cast<uint32_t>(kXRows * static_cast<int>(a.x_stride));
    const uint32_t w_step = 4u * static_cast<uint32_t>(kWRows * static_cast<int>(K));
    auto load = [&](Stage& stage, int64_t k0) {
        if constexpr (VEC) {
            // Rows past the matrices end the buffers; columns past K get an
            // offset beyond them.
            const BufferRsrc xb = make_buffer(x + k0, 2 * ((M - m0) * a.x_stride - k0));
            const BufferRsrc wb = make_buffer(w + k0, 4 * ((N - n0) * K - k0));
            const uint32_t xo = k0 + x_k < K ? x_at : kOutOfRange;
            const uint32_t wo = k0 + w_k < K ? w_at : kOutOfRange;
#pragma unroll
            for (int i = 0; i < kXPieces; ++i) {
                stage.x[i] = buffer_load16(xb, xo + i * x_step);
            }
#pragma unroll
            for (int i = 0; i < kWPieces; ++i) {
                stage.w[i] = buffer_load16(wb, wo + i * w_step);
            }
        } else {
            // Rows past the matrices read their last ones: what they feed is
            // not stored.
#pragma unroll
            for (int i = 0; i < kXPieces; ++i) {
                const int64_t r = m0 + x_row + kXRows * i < M ? x_row + kXRows * i : M - 1 - m0;
                stage.x[i] = load16_unaligned(x + r * a.x_stride + piece_start<8>(k0 + x_k, K));
            }
#pragma unroll
            for (int i = 0; i < kWPieces; ++i) {
                const int64_t r = n0 + w_row + kWRows * i < N ? w_row + kWRows * i : N - 1 - n0;
                stage.w[i] = load16_unaligned(w + r * K + piece_start<4>(k0 + w_k, K));
            }
        }
    };
    // The stage at column k0 into buffer `buf`.
    auto commit = [&](const Stage& stage, int buf, int64_t k0) {
        uint16_t* s_x = s_t + 2 * buf * kOperand;
        uint16_t* s_w = s_x + kOperand;
#pragma unroll
        for (int i = 0; i < kXPieces; ++i) {
            const u32x4 piece = VEC ? stage.x[i] : align_piece16(stage.x[i], k0 + x_k, K);
            *reinterpret_cast<u32x4*>(s_x + (x_row + kXRows * i) * KP + x_k) = to_bf16_piece<XT>(piece);
        }
#pragma unroll
        for (int i = 0; i < kWPieces; ++i) {
            const u32x4 piece = VEC ? stage.w[i] : align_piece32(stage.w[i], k0 + w_k, K);
            const f32x4 v = __builtin_bit_cast(f32x4, piece);
            const u32x2 packed = {pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
            *reinterpret_cast<u32x2*>(s_w + (w_row + kWRows * i) * KP + w_k) = packed;
        }
    };

    const int wn = 64 * (wave & 1);    // this wave's columns and rows of the tile
    const int wm = 64 * (wave >> 1);
    f32x16 acc[2][2];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                acc[nb][mb][e] = 0.0f;
            }
        }
    }
    const int fragment = (lane & 31) * KP + 8 * half;
    auto step = [&](int buf, Stage& stage, int64_t ahead) {
        const uint16_t* xt = s_t + 2 * buf * kOperand + wm * KP + fragment;
        const uint16_t* wt = s_t + (2 * buf + 1) * kOperand + wn * KP + fragment;
        u32x4 wf[2][2];
        u32x4 xf[2][2];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                wf[kk][b] = *reinterpret_cast<const u32x4*>(wt + 32 * b * KP + 16 * kk);
                xf[kk][b] = *reinterpret_cast<const u32x4*>(xt + 32 * b * KP + 16 * kk);
            }
        }
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            if (kk == 1) {
                commit(stage, buf ^ 1, ahead - 2 * kStreamK);
                load(stage, ahead);
            }
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) {
#pragma unroll
                for (int mb = 0; mb < 2; ++mb) {
                    acc[nb][mb] = mfma32x32x16(wf[kk][nb], xf[kk][mb], acc[nb][mb]);
                }
            }
        }
        __builtin_amdgcn_sched_group_barrier(kSchedDsRead, 4, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            __builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 0);
            __builtin_amdgcn_sched_group_barrier(kSchedDsRead, 1, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            __builtin_amdgcn_sched_group_barrier(kSchedValu, 8, 0);
            __builtin_amdgcn_sched_group_barrier(kSchedDsWrite, 2, 0);
            __builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 0);
        }
        __syncthreads();
    };
    Stage even;
    Stage odd;
    load(even, 0);
    load(odd, kStreamK);
    for (int c = tid; c < kStreamCols; c += kStreamThreads) {
        const int64_t n = n0 + c;
        s_bias[c] = (a.bias != nullptr && n < N) ? a.bias[n] : 0.0f;
    }
    for (int r = tid; r < kStreamRows; r += kStreamThreads) {
        const int64_t m = m0 + r;
        s_keep[r] = m < M && (a.row_mask == nullptr || a.row_mask[m] != 0);
    }
    commit(even, 0, 0);
    load(even, 2 * kStreamK);
    __syncthreads();
    // An odd last stage is followed by one of zeros: a second exit from the
    // loop would make it carry copies of the accumulators.
    for (int64_t k0 = 0; k0 < K; k0 += 2 * kStreamK) {
        step(0, odd, k0 + 3 * kStreamK);
        step(1, even, k0 + 4 * kStreamK);
    }

    // Epilogue: bias, row mask, one rounding; the tile goes out through LDS
    // as 16-byte pieces of whole row segments.  Lane (half, m) of block
    // (nb, mb) holds row m of the 32-row block and features 8 q + 4 half + r.
    uint16_t* s_y = s_t;
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) {
            const int mr = wm + mb * 32 + (lane & 31);
            const bool keep = s_keep[mr] != 0;
#pragma unroll
            for (int qd = 0; qd < 4; ++qd) {
                const int c = wn + nb * 32 + 8 * qd + 4 * half;
                const f32x4 bias = *reinterpret_cast<const f32x4*>(&s_bias[c]);
                const float v0 = keep ? acc[nb][mb][4 * qd + 0] + bias[0] : 0.0f;
                const float v1 = keep ? acc[nb][mb][4 * qd + 1] + bias[1] : 0.0f;
                const float v2 = keep ? acc[nb][mb][4 * qd + 2] + bias[2] : 0.0f;
                const float v3 = keep ? acc[nb][mb][4 * qd + 3] + bias[3] : 0.0f;
                u32x2 packed;
                if constexpr (YT == LSSO_HIP_BF16) {
                    packed.x = pack_bf16(v0, v1);
                    packed.y = pack_bf16(v2, v3);
                } else {
                    packed.x = pack_f16(v0, v1);
                    packed.y = pack_f16(v2, v3);
                }
                *reinterpret_cast<u32x2*>(&s_y[mr * YP + c]) = packed;
            }
        }
    }
    __syncthreads();
    constexpr int kStorePieces = kStreamRows * kStreamCols / 8 / kStreamThreads;
#pragma unroll
    for (int i = 0; i < kStorePieces; ++i) {
        const int piece = tid + i * kStreamThreads;
        const int mr = piece / (kStreamCols / 8);
        const int c8 = 8 * (piece - mr * (kStreamCols / 8));
        const int64_t m = m0 + mr;
        const int64_t n = n0 + c8;
        if (m < M && n < N) {
            const u32x4 v = *reinterpret_cast<const u32x4*>(&s_y[mr * YP + c8]);
            uint16_t* row = static_cast<uint16_t*>(a.y) + m * N;
            if (VEC) {
                *reinterpret_cast<u32x4*>(row + n) = v;
            } else {
                store_piece(row, n, N, v);
            }
        }
    }
}

template <int KSTEPS, bool VEC>
static hipError_t launch_linear_kv(const LinearArgs& a, int x_dtype, int y_dtype, dim3 grid,
                                   hipStream_t stream) {
    const dim3 block(kLinearWaves * 64);
    if (x_dtype == LSSO_HIP_F16) {
        if (y_dtype == LSSO_HIP_F16) {
            dispatch(linear_kernel<KSTEPS, LSSO_HIP_F16, LSSO_HIP_F16, VEC>, grid, block, stream, a);
        } else {
            dispatch(linear_kernel<KSTEPS, LSSO_HIP_F16, LSSO_HIP_BF16, VEC>, grid, block, stream, a);
        }
    } else {
        if (y_dtype == LSSO_HIP_F16) {
            dispatch(linear_kernel<KSTEPS, LSSO_HIP_BF16, LSSO_HIP_F16, VEC>, grid, block, stream, a);
        } else {
            dispatch(linear_kernel<KSTEPS, LSSO_HIP_BF16, LSSO_HIP_BF16, VEC>, grid, block, stream, a);
        }
    }
    return hipGetLastError();
}

template <int KSTEPS>
static hipError_t launch_linear_k(const LinearArgs& a, int x_dtype, int y_dtype, dim3 grid,
                                  hipStream_t stream) {
    // The vector form's 32-bit offsets reach one tile's rows.
    const bool vec = a.vector && a.x_stride < (1 << 23) && a.out_features < (1 << 23);
    return vec ? launch_linear_kv<KSTEPS, true>(a, x_dtype, y_dtype, grid, stream)
                      : launch_linear_kv<KSTEPS, false>(a, x_dtype, y_dtype, grid, stream);
}

hipError_t launch_linear(const LinearArgs& a, int k_steps, int x_dtype, int y_dtype,
                         int grid_groups, hipStream_t stream) {
    if (k_steps == 0) {
        // One block per output tile; row tiles rounded up to whole XCD rounds.
        static_assert(kStreamRows == kStreamRowsHost && kStreamCols == kStreamColsHost, "tile");
        const int64_t rounds = (a.tiles + kXcds - 1) / kXcds;
        const dim3 grid(static_cast<unsigned>(rounds * kXcds * a.column_groups));
        const dim3 block(kStreamThreads);
        // The vector form's 32-bit offsets reach one tile's rows.
        const bool vec = a.vector && a.x_stride < (1 << 23) && a.in_features < (1 << 22);
        const auto run = [&](auto kernel) { dispatch(kernel, grid, block, stream, a); };
        if (x_dtype == LSSO_HIP_F16) {
            if (y_dtype == LSSO_HIP_F16) {
                vec ? run(linear_stream_kernel<LSSO_HIP_F16, LSSO_HIP_F16, true>)
                    : run(linear_stream_kernel<LSSO_HIP_F16, LSSO_HIP_F16, false>);
            } else {
                vec ? run(linear_stream_kernel<LSSO_HIP_F16, LSSO_HIP_BF16, true>)
                    : run(linear_stream_kernel<LSSO_HIP_F16, LSSO_HIP_BF16, false>);
            }
        } else {
            if (y_dtype == LSSO_HIP_F16) {
                vec ? run(linear_stream_kernel<LSSO_HIP_BF16, LSSO_HIP_F16, true>)
                    : run(linear_stream_kernel<LSSO_HIP_BF16, LSSO_HIP_F16, false>);
            } else {
                vec ? run(linear_stream_kernel<LSSO_HIP_BF16, LSSO_HIP_BF16, true>)
                    : run(linear_stream_kernel<LSSO_HIP_BF16, LSSO_HIP_BF16, false>);
            }
        }
        return hipGetLastError();
    }
    const dim3 grid(static_cast<unsigned>(grid_groups * a.column_groups));
    switch (k_steps) {
        case 4: return launch_linear_k<4>(a, x_dtype, y_dtype, grid, stream);
        case 8: return launch_linear_k<8>(a, x_dtype, y_dtype, grid, stream);
        case 12: return launch_linear_k<12>(a, x_dtype, y_dtype, grid, stream);
        case 16: return launch_linear_k<16>(a, x_dtype, y_dtype, grid, stream);
        case 24: return launch_linear_k<24>(a, x_dtype, y_dtype, grid, stream);
        case 32: return launch_linear_k<32>(a, x_dtype, y_dtype, grid, stream);
        case 40: return launch_linear_k<40>(a, x_dtype, y_dtype, grid, stream);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace lsso_hip
