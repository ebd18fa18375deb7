// gfx950 weight (and bias) gradient of the biased projection
// (reference lsso/ball/reference.py:205-247):
//   grad_weight[n][k] = sum over rows m of bf16(g[m][n]) * bf16(x[m][k])   (FP32)
//   grad_bias[n]      = sum over rows m of g[m][n]                          (FP32)
// with rows that the row mask excludes counting as zero.
//
// The contraction runs over rows, the strided dimension of both row-major
// operands, while an MFMA fragment needs 8 rows of one column.  The operands
// stay row-major in LDS, as they come from HBM, and ds_read_b64_tr_b16 turns
// them on the way into registers: 16 lanes read 4 rows x 16 columns and lane
// i receives its column's 4 rows, so two such reads are one fragment of
// v_mfma_f32_32x32x16_bf16 (A = g^T, B = x, K = rows).
//
// Bound: HBM (g and x once) plus the FP32 partials; at 262,144 x (512, 256)
// that is 403 MB and 2 x 67 MB.  What sets the form is how often the operands
// pass from L2 to the CUs, how many loads are in flight, and how much of the
// conversion work hides under the MFMAs:
// - A workgroup of eight waves owns a 256 (n) x 256 (k) output tile (128
//   accumulation registers per wave) of a large product, so g is read K / 256
//   times and x N / 256 times; a small product takes 128 x 128 tiles.
// - 32-row stages, each thread moving 16-byte pieces; two stages of loads are
//   in flight in registers while a third is multiplied from LDS (two
//   buffers).  FP16 operands are rounded to BF16 (the reference's operands)
//   between the registers and LDS.
// - A stage is one basic block in which the next stage's conversions and LDS
//   writes are scheduled between the MFMAs: the two waves of a SIMD run in
//   step, so work not interleaved within a wave does not overlap at all
//   (126 us with the conversions before the products, 101 between them).
// - The LDS pitch of 32 bf16 past the tile puts the 4 rows that a half wave
//   reads on disjoint quarters of the 64 banks.
// The former kernel (128 x 128 tiles of four waves, 8 x 8 blocks transposed in
// registers with byte permutes, one stage in flight) took, with the column
// sums, 181 us at 262,144 x (512, 256), 96 at 262,144 x (256, 256), 112 at
// 131,072 x (640, 256) and 98 at 8,192 x (1,344, 768); this one 116, 66, 85
// and 44 (4.6-5.7 TB/s of operands and partials at the first two).
//
// Operands that are not whole aligned 16-byte pieces run the same loop and
// tiles on pieces aligned to their elements; element loads remain for rows of
// fewer than 8 elements.  Former kernel, this one with element loads, with
// these pieces (us): 65,537 x (521, 263) 276 / 295 / 74, 65,536 x (228, 100) 54 /
// 70 / 26, 16,000 x (772, 772) 280 / 226 / 55.
//
// A split writes FP32 partials [split][n][k]; column_sum_kernel adds the
// splits in a fixed order, so the result is deterministic.  The bias sums are
// taken from the g pieces (in g's own precision, as the reference sums g) by
// the k-tile-0 workgroups.  The workgroups of one row split are dealt to one
// XCD, so that the re-reads of g and x by the neighbouring tiles hit that
// XCD's L2.

#include "lsso_device.h"
#include "lsso_internal.h"
#include "lsso_hip.h"

#include <algorithm>
#include <cmath>

namespace lsso_hip {

namespace {

constexpr int kWgRows = 32;             // rows per stage (two MFMA K steps)
constexpr int kWgSteps = kWgRows / 16;
constexpr int kWgThreads = 512;         // eight waves: four along n, two along k

// Output tile of a workgroup: NB x KB blocks of 32 x 32 per wave.
template <int NB>
struct WgTile {
    static constexpr int kNB = NB;
    static constexpr int kKB = 2 * NB;
    static constexpr int kEdge = 4 * 32 * NB;            // n and k
    static constexpr int kPitch = kEdge + 32;            // row-major LDS pitch (bf16): 64 bytes past a multiple of 256
    static constexpr int kPieces = kEdge / 8;            // 16-byte pieces per row
    static constexpr int kRowLanes = kWgThreads / kPieces;
    static constexpr int kPasses = kWgRows / kRowLanes;  // pieces per thread, operand and stage
    static constexpr int kSlotsPerXcd = 32 * (NB == 1 ? 2 : 1);   // resident workgroups (by registers), 32 CUs
};
using WgLarge = WgTile<2>;   // 256 x 256
using WgSmall = WgTile<1>;   // 128 x 128
constexpr int kWgXcds = 8;

// Instruction classes of __builtin_amdgcn_sched_group_barrier.
constexpr int kSchedValu = 0x2;
constexpr int kSchedMfma = 0x8;
constexpr int kSchedDsRead = 0x100;
constexpr int kSchedDsWrite = 0x200;

template <int T>
__device__ __forceinline__ float bits_to_float(uint32_t bits) {
    if constexpr (T == LSSO_HIP_BF16) {
        return bf16_bits_to_float(static_cast<uint16_t>(bits));
    } else {
        return f16_bits_to_float(static_cast<uint16_t>(bits));
    }
}

template <int T>
__device__ __forceinline__ u32x4 to_bf16_piece(const u32x4& raw) {
    if constexpr (T == LSSO_HIP_BF16) {
        return raw;
    } else {
        u32x4 v;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            v[p] = pack_bf16(f16_lo(raw[p]), f16_hi(raw[p]));
        }
        return v;
    }
}

// How the operands' pieces are loaded.
constexpr int kWgWhole = 0;      // rows of whole aligned 16-byte pieces
constexpr int kWgPieces = 1;     // pieces aligned to their elements
constexpr int kWgElements = 2;   // element loads: rows of fewer than 8 elements

// One operand's pieces of a stage as loaded: columns c .. c + 7 of rows row_lane
// + kRowLanes * i, zero past the rows (end) and the columns except for
// kWgPieces, whose pieces finish_piece moves to their columns and zeroes.
// kWgWhole: raw-buffer loads whose buffer ends with the split's last row.
template <typename Tile, int FORM>
__device__ __forceinline__ void load_pieces(u32x4 (&out)[Tile::kPasses], const uint16_t* base, int64_t row,
                                            int64_t end, int64_t stride, int64_t c, int64_t cols, int row_lane) {
    if constexpr (FORM == kWgWhole) {
        const BufferRsrc buffer = make_buffer(base + row * stride, (end - row) * stride * 2);
        const uint32_t offset = c < cols ? static_cast<uint32_t>((row_lane * stride + c) * 2) : kOutOfRange;
        const uint32_t step = c < cols ? static_cast<uint32_t>(Tile::kRowLanes * stride * 2) : 0u;
#pragma unroll
        for (int i = 0; i < Tile::kPasses; ++i) {
            out[i] = buffer_load16(buffer, offset + i * step);
        }
    } else if constexpr (FORM == kWgPieces) {
#pragma unroll
        for (int i = 0; i < Tile::kPasses; ++i) {
            const int64_t m = row + row_lane + Tile::kRowLanes * i;
            out[i] = load16_unaligned(base + (m < end ? m : end - 1) * stride + piece_start<8>(c, cols));
        }
    } else {
#pragma unroll
        for (int i = 0; i < Tile::kPasses; ++i) {
            const int64_t m = row + row_lane + Tile::kRowLanes * i;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const uint32_t lo = (m < end && c + 2 * p < cols) ? base[m * stride + c + 2 * p] : 0u;
                const uint32_t hi = (m < end && c + 2 * p + 1 < cols) ? base[m * stride + c + 2 * p + 1] : 0u;
                out[i][p] = lo | (hi << 16);
            }
        }
    }
}
template <int FORM>
__device__ __forceinline__ u32x4 finish_piece(const u32x4& raw, bool live, int64_t c, int64_t cols) {
    if constexpr (FORM != kWgPieces) {
        return raw;
    }
    return live ? align_piece16(raw, c, cols) : (u32x4){0u, 0u, 0u, 0u};
}

template <typename Tile>
struct WgStage {
    u32x4 g[Tile::kPasses];
    u32x4 x[Tile::kPasses];
    uint32_t keep[Tile::kPasses];
};

}  // namespace

// MASK: a.row_mask is set; SUMS: a.bias_partials is set.  Both are template
// choices so that a stage is one basic block: the conversions, LDS writes and
// loads of the next stages are then scheduled between the MFMAs of this one.
template <typename Tile, int GT, int XT, int FORM, bool MASK, bool SUMS>
__global__ __launch_bounds__(kWgThreads) void weight_grad_kernel(WeightGradArgs a) {
    // Row-major stage buffers: s_t[buf][operand][row * Tile::kPitch + column].
    __shared__ __attribute__((aligned(16))) uint16_t s_t[2][2][kWgRows * Tile::kPitch];
    __shared__ float s_sum[Tile::kRowLanes][Tile::kEdge];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5;
    const int64_t tiles = a.tiles_n * a.tiles_k;
    int64_t tile;
    int64_t split;
    if (a.dealt) {
        // Row splits dealt round-robin over the XCDs, each XCD walking all
        // output tiles of its splits.
        const int64_t xcd = blockIdx.x % kWgXcds;
        const int64_t slot = blockIdx.x / kWgXcds;
        tile = slot % tiles;
        split = (slot / tiles) * kWgXcds + xcd;
        if (split >= a.splits) {
            return;
        }
    } else {
        tile = blockIdx.x % tiles;
        split = blockIdx.x / tiles;
    }
    const int64_t nt = tile / a.tiles_k;
    const int64_t kt = tile - nt * a.tiles_k;
    const int64_t n0 = nt * Tile::kEdge;
    const int64_t k0 = kt * Tile::kEdge;
    const int64_t N = a.out_features;
    const int64_t K = a.in_features;
    const int64_t r0 = split * a.rows_per_split;
    const int64_t r1 = r0 + a.rows_per_split < a.rows ? r0 + a.rows_per_split : a.rows;

    const int row_lane = tid / Tile::kPieces;
    const int piece = tid % Tile::kPieces;
    const uint16_t* g = static_cast<const uint16_t*>(a.g);
    const uint16_t* x = static_cast<const uint16_t*>(a.x);

    float colsum[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        colsum[e] = 0.0f;
    }
    auto load = [&](WgStage<Tile>& stage, int64_t row) {
        load_pieces<Tile, FORM>(stage.g, g, row, r1, a.g_stride, n0 + 8 * piece, N, row_lane);
        load_pieces<Tile, FORM>(stage.x, x, row, r1, a.x_stride, k0 + 8 * piece, K, row_lane);
        if constexpr (MASK) {
            const BufferRsrc mask = make_buffer(a.row_mask + row, r1 - row);
#pragma unroll
            for (int i = 0; i < Tile::kPasses; ++i) {
                stage.keep[i] = buffer_load_byte(mask, row_lane + Tile::kRowLanes * i);
            }
        }
    };
    auto commit = [&](WgStage<Tile>& stage, int buf, int64_t row) {
#pragma unroll
        for (int i = 0; i < Tile::kPasses; ++i) {
            const bool live = row + row_lane + Tile::kRowLanes * i < r1;
            stage.g[i] = finish_piece<FORM>(stage.g[i], live, n0 + 8 * piece, N);
            stage.x[i] = finish_piece<FORM>(stage.x[i], live, k0 + 8 * piece, K);
            if constexpr (MASK) {
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    stage.g[i][p] = stage.keep[i] != 0 ? stage.g[i][p] : 0u;
                    stage.x[i][p] = stage.keep[i] != 0 ? stage.x[i][p] : 0u;
                }
            }
            if constexpr (SUMS) {
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    colsum[2 * p] += bits_to_float<GT>(stage.g[i][p] & 0xffffu);
                    colsum[2 * p + 1] += bits_to_float<GT>(stage.g[i][p] >> 16);
                }
            }
            const int at = (row_lane + Tile::kRowLanes * i) * Tile::kPitch + 8 * piece;
            *reinterpret_cast<u32x4*>(s_t[buf][0] + at) = to_bf16_piece<GT>(stage.g[i]);
            *reinterpret_cast<u32x4*>(s_t[buf][1] + at) = to_bf16_piece<XT>(stage.x[i]);
        }
    };

    constexpr int NB = Tile::kNB;
    constexpr int KB = Tile::kKB;
    const int wn = 32 * NB * (wave & 3);    // this wave's quarter (n) and half (k) of the output tile
    const int wk = 32 * KB * (wave >> 2);
    f32x16 acc[NB][KB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                acc[nb][kb][e] = 0.0f;
            }
        }
    }
    // This lane's 8 bytes of a transposed read: row (lane % 16) / 4 of the 4
    // rows (8 rows further for the upper half wave: the K order of the
    // fragments), 4 columns of its 16-column group.
    const int fragment = ((lane & 15) / 4 + 8 * half) * Tile::kPitch + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    auto read_fragment = [&](const uint16_t* base) {
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsS16x4*)(base));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsS16x4*)(base + 4 * Tile::kPitch));
        const u32x2 l = __builtin_bit_cast(u32x2, lo);
        const u32x2 h = __builtin_bit_cast(u32x2, hi);
        return (u32x4){l[0], l[1], h[0], h[1]};
    };
    // One stage: the products of LDS buffer `buf`, and between them the next
    // stage's pieces (`stage`, loaded two steps ago) into the other buffer and
    // the loads of the stage three ahead into the registers they leave.
    // Waves whose block lies past N or K multiply zeros (LDS holds zeros past
    // the columns) rather than branch.
    auto step = [&](int buf, WgStage<Tile>& stage, int64_t next_row) {
        const uint16_t* gt = s_t[buf][0] + fragment + wn;
        const uint16_t* xt = s_t[buf][1] + fragment + wk;
        u32x4 af[kWgSteps][NB];
        u32x4 bf[kWgSteps][KB];
#pragma unroll
        for (int kk = 0; kk < kWgSteps; ++kk) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                af[kk][b] = read_fragment(gt + 16 * kk * Tile::kPitch + 32 * b);
            }
#pragma unroll
            for (int b = 0; b < KB; ++b) {
                bf[kk][b] = read_fragment(xt + 16 * kk * Tile::kPitch + 32 * b);
            }
        }
#pragma unroll
        for (int kk = 0; kk < kWgSteps; ++kk) {
            if (kk == kWgSteps - 1) {
                commit(stage, buf ^ 1, next_row - 2 * kWgRows);
                load(stage, next_row);
            }
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    acc[nb][kb] = mfma32x32x16(af[kk][nb], bf[kk][kb], acc[nb][kb]);
                }
            }
        }
        // The order of the block: the first K step's fragments, its MFMAs with
        // the second's fragment reads between them, then the second's MFMAs
        // with the next stage's conversions and LDS writes between them.
        constexpr int kReads = 2 * (NB + KB);
        constexpr int kProducts = NB * KB;
        constexpr int kPerProduct = kReads / kProducts + (kReads % kProducts != 0);
        __builtin_amdgcn_sched_group_barrier(kSchedDsRead, kReads, 0);
#pragma unroll
        for (int i = 0; i < kProducts; ++i) {
            __builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 0);
            __builtin_amdgcn_sched_group_barrier(kSchedDsRead, kPerProduct, 0);
        }
#pragma unroll
        for (int i = 0; i < kProducts; ++i) {
            __builtin_amdgcn_sched_group_barrier(kSchedValu, 8, 0);
            __builtin_amdgcn_sched_group_barrier(kSchedDsWrite, 1, 0);
            __builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 0);
        }
        __syncthreads();
    };
    // Stages past the split load zeros without an access; an odd last one is
    // multiplied all the same (a branch around it would make the loop carry
    // copies of the registers in flight, and wait for them).
    WgStage<Tile> even;
    WgStage<Tile> odd;
    load(even, r0);
    load(odd, r0 + kWgRows);
    commit(even, 0, r0);
    load(even, r0 + 2 * kWgRows);
    __syncthreads();
    for (int64_t row = r0; row < r1; row += 2 * kWgRows) {
        step(0, odd, row + 3 * kWgRows);
        step(1, even, row + 4 * kWgRows);
    }

    // Partials: lane (half, j) of block (nb, kb) holds column k = j and rows
    // n = 8 q + 4 half + e of the block, for accumulator entry 4 q + e.
    float* out = a.partials + split * N * K;
    {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
                const int64_t nb0 = n0 + wn + 32 * nb;
                const int64_t kb0 = k0 + wk + 32 * kb;
                const bool whole = nb0 + 32 <= N && kb0 + 32 <= K;   // uniform
                const int64_t k = kb0 + (lane & 31);
                float* block = out + (nb0 + 4 * half) * K + k;
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int64_t n = 8 * (e / 4) + (e % 4);
                    if (whole || (nb0 + 4 * half + n < N && k < K)) {
                        block[n * K] = acc[nb][kb][e];
                    }
                }
            }
        }
    }
    if (SUMS && kt == 0) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            s_sum[row_lane][8 * piece + e] = colsum[e];
        }
        __syncthreads();
        if (tid < Tile::kEdge) {
            float total = 0.0f;
#pragma unroll
            for (int r = 0; r < Tile::kRowLanes; ++r) {
                total += s_sum[r][tid];
            }
            if (n0 + tid < N) {
                a.bias_partials[split * N + n0 + tid] = total;
            }
        }
    }
}

template <typename Tile>
static int64_t wg_tiles(int64_t in_features, int64_t out_features) {
    return ((out_features + Tile::kEdge - 1) / Tile::kEdge) * ((in_features + Tile::kEdge - 1) / Tile::kEdge);
}

// The output tile.  The large tile moves half the operand bytes between L2 and
// the CUs per product but writes four times the partials per workgroup and
// leaves short row ranges with fewer, longer chains, so it takes a long
// product; a shorter one where the small tiles leave an XCD's workgroups idle
// (36 tiles at 768 x 768: one split of 64 slots, so little over half) or are too
// many to be dealt to the XCDs.  Measured with the column sums and without a
// bias, large over small tile, at 5 / 8.5 / 12 / 20 / 50e9 multiply-adds:
// outputs of 512 x 512 1.17 / 1.15 / 1.06 / 0.95 / 0.83, 1,344 x 768 1.11 / 1.00
// / 0.96 / 0.88 / 0.78, 768 x 768 1.05 / 0.90 / 0.83 / 0.71 / 0.61, 640 x 256
// 1.17 / 1.12 / 1.05 / 0.99 / 0.94.  A single tile per split (256 x 256: 1.19 /
// 1.24 / 1.13 / 1.17 / 1.01) and outputs that half fill large tiles (384 x 384
// 1.18 / 1.17 / 1.16 / 1.16 / 1.06, 228 x 100 1.20 throughout, 64 x 64 about 1.9)
// never gain from it.
static bool weight_grad_large(int64_t rows, int64_t in_features, int64_t out_features) {
    const int64_t large = wg_tiles<WgLarge>(in_features, out_features);
    const int64_t small = wg_tiles<WgSmall>(in_features, out_features);
    const int64_t slots = WgSmall::kSlotsPerXcd;
    if (large < 2 || 8 * large >= 3 * small) {   // padded at least 1.5 times as far
        return false;
    }
    const double share = small <= slots ? static_cast<double>(slots / small * small) / slots : 0.75;
    return static_cast<double>(rows) * in_features * out_features >= 1.2e10 * share;
}

// Row splits.  More splits put more CUs on the product (its time falls as 1 /
// splits) but write and read again splits x N x K floats: with a workgroup's
// matrix rate p and the memory rate m the sum of 2 M N K / (splits tiles p)
// and 8 splits N K / m is least at splits = sqrt(M m / (4 tiles p)); m = 5
// TB/s, p = 2 TFLOP/s (a workgroup of a short problem is latency-bound).  Up
// to one XCD's resident workgroups in output tiles, the splits are a multiple
// of the eight XCDs, at least 16 (two 32-row stages already take longer than
// their sum saves), bounded so that all workgroups of an XCD (its splits x the
// output tiles) are resident at once: one more, nearly empty round would take
// as long as the first.  Beyond, as many splits as keep the device's CUs busy
// in one round, not dealt to the XCDs.
void plan_weight_grad(int64_t rows, int64_t in_features, int64_t out_features, int64_t* splits,
                      int64_t* rows_per_split) {
    const bool large = weight_grad_large(rows, in_features, out_features);
    const int64_t slots = large ? WgLarge::kSlotsPerXcd : WgSmall::kSlotsPerXcd;
    const int64_t tiles = large ? wg_tiles<WgLarge>(in_features, out_features)
                                : wg_tiles<WgSmall>(in_features, out_features);
    const int64_t stages = (rows + kWgRows - 1) / kWgRows;
    int64_t want;
    if (tiles <= slots) {
        const double best = std::sqrt(static_cast<double>(rows) * 5.0 / (4.0 * 2.0 * static_cast<double>(tiles)));
        const int64_t per_xcd = std::max<int64_t>(2, static_cast<int64_t>(best / kWgXcds + 0.5));
        want = kWgXcds * std::min(per_xcd, slots / tiles);
    } else {
        want = std::max<int64_t>(1, kWgXcds * slots / tiles);
    }
    if (want > stages) want = stages;
    if (want < 1) want = 1;
    const int64_t per = (rows + want - 1) / want;
    *rows_per_split = ((per + kWgRows - 1) / kWgRows) * kWgRows;
    *splits = rows == 0 ? 0 : (rows + *rows_per_split - 1) / *rows_per_split;
}

template <typename Tile, int GT, int XT, int FORM>
static void launch_wg(const WeightGradArgs& a, dim3 grid, hipStream_t stream) {
    const auto run = [&](auto kernel) { kernel<<<grid, kWgThreads, 0, stream>>>(a); };
    if (a.row_mask != nullptr) {
        a.bias_partials != nullptr ? run(weight_grad_kernel<Tile, GT, XT, FORM, true, true>)
                                   : run(weight_grad_kernel<Tile, GT, XT, FORM, true, false>);
    } else {
        a.bias_partials != nullptr ? run(weight_grad_kernel<Tile, GT, XT, FORM, false, true>)
                                   : run(weight_grad_kernel<Tile, GT, XT, FORM, false, false>);
    }
}

template <int GT, int XT>
static void launch_wg(const WeightGradArgs& a, dim3 grid, hipStream_t stream) {
    if (a.vec) {
        a.large ? launch_wg<WgLarge, GT, XT, kWgWhole>(a, grid, stream)
                : launch_wg<WgSmall, GT, XT, kWgWhole>(a, grid, stream);
    } else if (a.in_features >= 8 && a.out_features >= 8) {
        a.large ? launch_wg<WgLarge, GT, XT, kWgPieces>(a, grid, stream)
                : launch_wg<WgSmall, GT, XT, kWgPieces>(a, grid, stream);
    } else {
        launch_wg<WgSmall, GT, XT, kWgElements>(a, grid, stream);   // never large
    }
}

hipError_t launch_weight_grad(const WeightGradArgs& args, int g_dtype, int x_dtype, hipStream_t stream) {
    if (args.splits == 0) {
        return hipSuccess;
    }
    WeightGradArgs a = args;
    // The raw buffers' 32-bit offsets reach one stage's rows.
    a.vec = a.vec && a.g_stride < (1 << 24) && a.x_stride < (1 << 24);
    a.large = weight_grad_large(a.rows, a.in_features, a.out_features);
    const int64_t edge = a.large ? WgLarge::kEdge : WgSmall::kEdge;
    a.tiles_n = (a.out_features + edge - 1) / edge;
    a.tiles_k = (a.in_features + edge - 1) / edge;
    const int64_t tiles = a.tiles_n * a.tiles_k;
    a.dealt = a.splits > 1 && tiles <= (a.large ? WgLarge::kSlotsPerXcd : WgSmall::kSlotsPerXcd);
    const int64_t rounds = (a.splits + kWgXcds - 1) / kWgXcds;
    const dim3 grid(static_cast<unsigned>(a.dealt ? rounds * kWgXcds * tiles : a.splits * tiles));
    if (g_dtype == LSSO_HIP_F16) {
        if (x_dtype == LSSO_HIP_F16) {
            launch_wg<LSSO_HIP_F16, LSSO_HIP_F16>(a, grid, stream);
        } else {
            launch_wg<LSSO_HIP_F16, LSSO_HIP_BF16>(a, grid, stream);
        }
    } else {
        if (x_dtype == LSSO_HIP_F16) {
            launch_wg<LSSO_HIP_BF16, LSSO_HIP_F16>(a, grid, stream);
        } else {
            launch_wg<LSSO_HIP_BF16, LSSO_HIP_BF16>(a, grid, stream);
        }
    }
    return hipGetLastError();
}

}  // namespace lsso_hip
