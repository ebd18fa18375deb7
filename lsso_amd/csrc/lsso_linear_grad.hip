// gfx950 upstream-gradient pass of the biased projection's backward
// (reference lsso/ball/reference.py:205-247).
//
// The reference rounds the upstream gradient to BF16 for the weight-gradient
// GEMM and sums it in FP32 over all rows for the bias gradient.  One pass over
// g does both: every (row, 8-column chunk) is read once, rounded to BF16 and
// written (when a BF16 copy is asked for), and added to per-thread FP32
// column sums.  Rows excluded by the row mask count as zero.
//
// Schedule: blockIdx.y is a slab of `cw` 8-column chunks; blockIdx.x is a
// split of consecutive rows.  Thread t takes chunk t % cw and every
// (256 / cw)-th row of the split, eight rows' loads in flight.  The row lanes
// of a chunk are combined in LDS in lane order and the split writes one FP32
// partial per column; column_sum_kernel adds the splits in a fixed order, so
// the sums are deterministic.

#include "lsso_device.h"
#include "lsso_internal.h"
#include "lsso_hip.h"

namespace lsso_hip {

constexpr int kGradThreads = 256;
constexpr int kGradRowsInFlight = 8;

template <int GT>
__device__ __forceinline__ float grad_bits_to_float(uint16_t bits) {
    if constexpr (GT == LSSO_HIP_BF16) {
        return bf16_bits_to_float(bits);
    } else {
        return f16_bits_to_float(bits);
    }
}

template <int GT, bool VEC>
__global__ __launch_bounds__(kGradThreads) void grad_columns_kernel(GradColumnsArgs a) {
    const int t = threadIdx.x;
    const int cw = a.chunks_per_slab;
    const int row_lanes = kGradThreads / cw;
    const int row_lane = t / cw;
    const int64_t col0 = (static_cast<int64_t>(blockIdx.y) * cw + (t - row_lane * cw)) * 8;
    const bool col_live = col0 < a.cols;
    const int64_t r0 = static_cast<int64_t>(blockIdx.x) * a.rows_per_split;
    const int64_t r1 = r0 + a.rows_per_split < a.rows ? r0 + a.rows_per_split : a.rows;
    const uint16_t* g = static_cast<const uint16_t*>(a.g);

    float acc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        acc[i] = 0.0f;
    }
    for (int64_t base = r0 + row_lane; base < r1; base += static_cast<int64_t>(row_lanes) * kGradRowsInFlight) {
        float v[kGradRowsInFlight][8];
        bool live[kGradRowsInFlight];
        bool keep[kGradRowsInFlight];
#pragma unroll
        for (int u = 0; u < kGradRowsInFlight; ++u) {
            const int64_t row = base + static_cast<int64_t>(u) * row_lanes;
            live[u] = row < r1 && col_live;
            const int64_t safe_row = live[u] ? row : r0;
            keep[u] = live[u] && (a.row_mask == nullptr || a.row_mask[safe_row] != 0);
            const uint16_t* src = g + safe_row * a.g_stride;
            if constexpr (VEC) {
                const u32x4 raw = *reinterpret_cast<const u32x4*>(src + (col_live ? col0 : 0));
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    if constexpr (GT == LSSO_HIP_BF16) {
                        v[u][2 * p] = bf16_lo(raw[p]);
                        v[u][2 * p + 1] = bf16_hi(raw[p]);
                    } else {
                        v[u][2 * p] = f16_lo(raw[p]);
                        v[u][2 * p + 1] = f16_hi(raw[p]);
                    }
                }
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const bool in = col_live && col0 + i < a.cols;
                    v[u][i] = grad_bits_to_float<GT>(src[in ? col0 + i : 0]);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < kGradRowsInFlight; ++u) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                v[u][i] = keep[u] ? v[u][i] : 0.0f;
                acc[i] += v[u][i];
            }
            if (a.g_bf16 != nullptr && live[u]) {
                const int64_t row = base + static_cast<int64_t>(u) * row_lanes;
                uint16_t* dst = a.g_bf16 + row * a.cols + col0;
                if constexpr (VEC) {
                    u32x4 packed;
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        packed[p] = pack_bf16(v[u][2 * p], v[u][2 * p + 1]);
                    }
                    *reinterpret_cast<u32x4*>(dst) = packed;
                } else {
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        if (col0 + i < a.cols) {
                            dst[i] = to_bf16_bits(v[u][i]);
                        }
                    }
                }
            }
        }
    }
    if (a.partials == nullptr) {
        return;
    }
    // Row lanes of each column, combined in lane order.
    __shared__ float s_sum[kGradThreads * 8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        s_sum[t * 8 + i] = acc[i];
    }
    __syncthreads();
    for (int idx = t; idx < cw * 8; idx += kGradThreads) {
        const int64_t column = static_cast<int64_t>(blockIdx.y) * cw * 8 + idx;
        float total = 0.0f;
        for (int lane = 0; lane < row_lanes; ++lane) {
            total += s_sum[lane * cw * 8 + idx];
        }
        if (column < a.cols) {
            a.partials[static_cast<int64_t>(blockIdx.x) * a.cols + column] = total;
        }
    }
}

// out[c] = sum over splits s of partials[s][c], in a fixed order: a thread
// takes one piece (four columns, one 16-byte load; one column where the rows
// are not whole pieces) of every `lanes`-th split with eight loads in flight,
// then the lanes of a piece are added in lane order.  The lanes per piece (a
// power of two up to 32) are the fewest that give the device its threads:
// few columns over many splits need many lanes, and a wide weight over eight
// splits needs one (with eight fixed lanes of sixteen loads each, 1,344 x
// 768 columns over 8 splits ran at 1 TB/s).  One launch can serve two such
// sums over the same splits (a weight gradient and its bias): the first
// `blocks` workgroups take the first, the rest the second.
constexpr int kSumLoads = 8;
constexpr int kSumMaxLanes = 32;
constexpr int64_t kSumThreads = 256 * 512;   // threads that keep the memory busy: two per SIMD lane

struct ColumnSum {
    const float* partials;
    int64_t cols;
    float* out;
    int lanes;
};

template <int V>
struct SumPiece {
    float v[V];
};
template <int V>
__device__ __forceinline__ SumPiece<V> load_sum_piece(const float* at) {
    SumPiece<V> p;
    if constexpr (V == 4) {
        const f32x4 raw = *reinterpret_cast<const f32x4*>(at);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            p.v[e] = raw[e];
        }
    } else {
        p.v[0] = *at;
    }
    return p;
}

template <int V>
__global__ __launch_bounds__(kGradThreads) void column_sum_kernel(ColumnSum first, ColumnSum second, int64_t splits,
                                                                  int64_t blocks) {
    __shared__ float s_acc[kGradThreads][V];
    int64_t block = blockIdx.x;
    ColumnSum a = first;
    if (block >= blocks) {   // uniform over the workgroup
        block -= blocks;
        a = second;
    }
    const int pieces = kGradThreads / a.lanes;   // of this workgroup
    const int piece = threadIdx.x % pieces;
    const int lane = threadIdx.x / pieces;
    const int64_t column = (block * pieces + piece) * V;
    const bool live = column < a.cols;
    const float* base = a.partials + (live ? column : 0);
    float acc[V];
#pragma unroll
    for (int e = 0; e < V; ++e) {
        acc[e] = 0.0f;
    }
    for (int64_t s0 = lane; s0 < splits; s0 += a.lanes * kSumLoads) {
        SumPiece<V> v[kSumLoads];
#pragma unroll
        for (int u = 0; u < kSumLoads; ++u) {
            const int64_t s = s0 + u * a.lanes;
            v[u] = load_sum_piece<V>(base + (s < splits ? s : s0) * a.cols);
        }
#pragma unroll
        for (int u = 0; u < kSumLoads; ++u) {
            if (s0 + u * a.lanes < splits) {
#pragma unroll
                for (int e = 0; e < V; ++e) {
                    acc[e] += v[u].v[e];
                }
            }
        }
    }
    if (a.lanes > 1) {   // uniform
#pragma unroll
        for (int e = 0; e < V; ++e) {
            s_acc[threadIdx.x][e] = acc[e];
        }
        __syncthreads();
        if (lane != 0) {
            return;
        }
        for (int l = 1; l < a.lanes; ++l) {
#pragma unroll
            for (int e = 0; e < V; ++e) {
                acc[e] += s_acc[l * pieces + piece][e];
            }
        }
    }
    if (live) {
#pragma unroll
        for (int e = 0; e < V; ++e) {
            a.out[column + e] = acc[e];
        }
    }
}

hipError_t launch_column_sum(const float* partials, int64_t splits, int64_t cols, float* out,
                             hipStream_t stream) {
    return launch_column_sums(partials, cols, out, nullptr, 0, nullptr, splits, stream);
}

hipError_t launch_column_sums(const float* partials, int64_t cols, float* out, const float* partials2,
                              int64_t cols2, float* out2, int64_t splits, hipStream_t stream) {
    const auto whole = [](const float* base, int64_t n) {
        return n % 4 == 0 && reinterpret_cast<uintptr_t>(base) % 16 == 0;
    };
    const int v = whole(partials, cols) && (cols2 == 0 || whole(partials2, cols2)) ? 4 : 1;
    const auto plan = [&](const float* base, int64_t n, float* to, int64_t* blocks) {
        const int64_t pieces = (n + v - 1) / v;
        int lanes = 1;
        while (lanes < kSumMaxLanes && lanes < splits && pieces * lanes < kSumThreads) {
            lanes *= 2;
        }
        const int64_t per_block = kGradThreads / lanes;
        *blocks = (pieces + per_block - 1) / per_block;
        return ColumnSum{base, n, to, lanes};
    };
    int64_t blocks = 0;
    int64_t blocks2 = 0;
    const ColumnSum first = plan(partials, cols, out, &blocks);
    const ColumnSum second = plan(partials2, cols2, out2, &blocks2);
    const dim3 grid(static_cast<unsigned>(blocks + blocks2));
    if (v == 4) {
        column_sum_kernel<4><<<grid, kGradThreads, 0, stream>>>(first, second, splits, blocks);
    } else {
        column_sum_kernel<1><<<grid, kGradThreads, 0, stream>>>(first, second, splits, blocks);
    }
    return hipGetLastError();
}

hipError_t launch_grad_columns(const GradColumnsArgs& a, int g_dtype, bool vec, int64_t splits,
                               int64_t slabs, float* column_sums, hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>(splits), static_cast<unsigned>(slabs));
    if (splits == 0) {
        // No rows: the column sums are zero.
    } else if (g_dtype == LSSO_HIP_BF16) {
        if (vec) {
            grad_columns_kernel<LSSO_HIP_BF16, true><<<grid, kGradThreads, 0, stream>>>(a);
        } else {
            grad_columns_kernel<LSSO_HIP_BF16, false><<<grid, kGradThreads, 0, stream>>>(a);
        }
    } else {
        if (vec) {
            grad_columns_kernel<LSSO_HIP_F16, true><<<grid, kGradThreads, 0, stream>>>(a);
        } else {
            grad_columns_kernel<LSSO_HIP_F16, false><<<grid, kGradThreads, 0, stream>>>(a);
        }
    }
    hipError_t error = hipGetLastError();
    if (error != hipSuccess || column_sums == nullptr) {
        return error;
    }
    return launch_column_sum(a.partials, splits, a.cols, column_sums, stream);
}

// Transposed weights of the projections' value gradients (dX = dY W reads W
// by output feature).  32 x 32 tiles through LDS, both of a layer's weights in
// one launch: two tensor copies before took 3.2-6.8 us each and their host time.
constexpr int kTransposeTile = 32;

struct TransposeArgs {
    const float* in;
    int64_t rows, cols;
    float* out;
    int64_t tiles_c, tiles;
};

__global__ __launch_bounds__(kGradThreads) void transpose2_kernel(TransposeArgs first, TransposeArgs second) {
    __shared__ float s_tile[kTransposeTile][kTransposeTile + 1];
    int64_t tile = blockIdx.x;
    TransposeArgs a = first;
    if (tile >= first.tiles) {   // uniform over the workgroup
        tile -= first.tiles;
        a = second;
    }
    const int64_t r0 = tile / a.tiles_c * kTransposeTile;
    const int64_t c0 = tile % a.tiles_c * kTransposeTile;
    const int c = threadIdx.x % kTransposeTile;
    const int r = threadIdx.x / kTransposeTile;
    constexpr int kRows = kGradThreads / kTransposeTile;
#pragma unroll
    for (int i = 0; i < kTransposeTile; i += kRows) {
        if (r0 + r + i < a.rows && c0 + c < a.cols) {
            s_tile[r + i][c] = a.in[(r0 + r + i) * a.cols + c0 + c];
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kTransposeTile; i += kRows) {
        if (c0 + r + i < a.cols && r0 + c < a.rows) {
            a.out[(c0 + r + i) * a.rows + r0 + c] = s_tile[c][r + i];
        }
    }
}

hipError_t launch_transpose2(const float* in1, int64_t rows1, int64_t cols1, float* out1, const float* in2,
                             int64_t rows2, int64_t cols2, float* out2, hipStream_t stream) {
    const auto plan = [](const float* in, int64_t rows, int64_t cols, float* out) {
        const int64_t tiles_r = (rows + kTransposeTile - 1) / kTransposeTile;
        const int64_t tiles_c = (cols + kTransposeTile - 1) / kTransposeTile;
        return TransposeArgs{in, rows, cols, out, tiles_c, tiles_r * tiles_c};
    };
    const TransposeArgs first = plan(in1, rows1, cols1, out1);
    const TransposeArgs second = plan(in2, rows2, cols2, out2);
    if (first.tiles + second.tiles == 0) {
        return hipSuccess;
    }
    const dim3 grid(static_cast<unsigned>(first.tiles + second.tiles));
    transpose2_kernel<<<grid, kGradThreads, 0, stream>>>(first, second);
    return hipGetLastError();
}

}  // namespace lsso_hip
