// Token geometry of a masked or explicitly positioned batch: centred FP32
// positions and valid counts from the caller's boolean mask and position ids
// (reference lsso/ball/model.py:163-243, 364-370) in one launch.
//
// A sample's positions are taken relative to its first valid token, in the
// ids' own type (so integer ids beyond 2^24 and FP64 ids keep their
// differences), and the mean over its valid tokens is subtracted; excluded
// tokens get 0.  As separate tensor operations this is about twenty launches
// of 2-10 us (mask counts, argmax, gather, conversions, products, sums,
// selects): 40 us of kernels and 90 us of host time before the layer's own
// first launch at 8 x 513 tokens, 95 us of kernels at 32 x 4,096.  In this
// form the whole masked layer call takes 71 us instead of 161 (8 x 513, rank
// 32) and 354 instead of 437 (32 x 4,096, rank 64, ids per sample); an image
// with a shared float grid (1 x 197) 61 instead of 71.
//
// Bound: latency.  One workgroup per sample walks its row in up to three
// passes (first valid token and count; sum of differences; write), each
// thread with kTokens independent loads in flight; the row (mask byte and id)
// is read from HBM once and from L2 after that.  Sums are FP64: exact for
// integer ids, and independent of how the row is split over the threads.

#include "lsso_device.h"
#include "lsso_internal.h"

namespace lsso_hip {

namespace {

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / 64;
constexpr int kTokens = 4;   // tokens per thread and pass step, kThreads apart

// Differences in the ids' own type, then the type the mean is taken in: FP64
// for FP64 ids, FP32 otherwise (integer differences are exact before the
// cast; reference model.py:208-216).
__device__ __forceinline__ float position_difference(int64_t p, int64_t anchor) {
    return static_cast<float>(static_cast<int64_t>(static_cast<uint64_t>(p) - static_cast<uint64_t>(anchor)));
}
__device__ __forceinline__ float position_difference(float p, float anchor) { return p - anchor; }
__device__ __forceinline__ double position_difference(double p, double anchor) { return p - anchor; }

__device__ __forceinline__ int wave_sum(int v) {
    for (int s = 32; s > 0; s >>= 1) v += __shfl_xor(v, s);
    return v;
}
__device__ __forceinline__ int wave_min(int v) {
    for (int s = 32; s > 0; s >>= 1) { const int o = __shfl_xor(v, s); v = o < v ? o : v; }
    return v;
}
__device__ __forceinline__ double wave_sum(double v) {
    for (int s = 32; s > 0; s >>= 1) v += __shfl_xor(v, s);
    return v;
}

// T: the ids' load type; P: the type they are held in (int64_t for integers).
template <typename T, typename P, bool IDS, bool MASK>
__global__ __launch_bounds__(kThreads) void geometry_kernel(GeometryArgs a) {
    using D = decltype(position_difference(P{}, P{}));
    __shared__ int first_part[kWaves];
    __shared__ int count_part[kWaves];
    __shared__ double sum_part[kWaves];
    const int64_t b = blockIdx.x;
    const int length = static_cast<int>(a.length);
    const int wave = threadIdx.x >> 6;
    const T* ids = static_cast<const T*>(a.positions) + (IDS ? b * a.position_batch_stride : 0);
    const uint8_t* mask = MASK ? a.mask + b * a.length : nullptr;
    const auto id = [&](int t) -> P {
        if constexpr (IDS) {
            return static_cast<P>(ids[t * a.position_token_stride]);
        } else {
            return static_cast<P>(t);
        }
    };

    int first = 0;
    int count = length;
    if constexpr (MASK) {
        int my_first = length;
        int my_count = 0;
        for (int base = threadIdx.x; base < length; base += kThreads * kTokens) {
#pragma unroll
            for (int k = 0; k < kTokens; ++k) {
                const int t = base + k * kThreads;
                if (t < length && mask[t] != 0) {
                    my_first = t < my_first ? t : my_first;
                    ++my_count;
                }
            }
        }
        my_first = wave_min(my_first);
        my_count = wave_sum(my_count);
        if ((threadIdx.x & 63) == 0) {
            first_part[wave] = my_first;
            count_part[wave] = my_count;
        }
        __syncthreads();
        first = length;
        count = 0;
        for (int w = 0; w < kWaves; ++w) {
            first = first_part[w] < first ? first_part[w] : first;
            count += count_part[w];
        }
        // Without a valid token the anchor does not matter: every output is 0.
        first = first < length ? first : 0;
        if (threadIdx.x == 0) {
            a.counts[b] = count > 0 ? static_cast<float>(count) : 1.0f;
        }
    }

    const P anchor = id(first);
    double sum = 0.0;
    for (int base = threadIdx.x; base < length; base += kThreads * kTokens) {
#pragma unroll
        for (int k = 0; k < kTokens; ++k) {
            const int t = base + k * kThreads;
            if (t < length && (!MASK || mask[t] != 0)) {
                sum += static_cast<double>(position_difference(id(t), anchor));
            }
        }
    }
    sum = wave_sum(sum);
    if ((threadIdx.x & 63) == 0) {
        sum_part[wave] = sum;
    }
    __syncthreads();
    sum = 0.0;
    for (int w = 0; w < kWaves; ++w) {
        sum += sum_part[w];
    }
    const D mean = static_cast<D>(sum / static_cast<double>(count > 0 ? count : 1));
    float* out = a.centered + b * a.length;
    for (int base = threadIdx.x; base < length; base += kThreads * kTokens) {
#pragma unroll
        for (int k = 0; k < kTokens; ++k) {
            const int t = base + k * kThreads;
            if (t < length) {
                const bool keep = !MASK || mask[t] != 0;
                out[t] = keep ? static_cast<float>(position_difference(id(t), anchor) - mean) : 0.0f;
            }
        }
    }
}

template <typename T, typename P, bool IDS>
void launch(const GeometryArgs& a, hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>(a.rows));
    if (a.mask != nullptr) {
        dispatch(geometry_kernel<T, P, IDS, true>, grid, kThreads, stream, a);
    } else {
        dispatch(geometry_kernel<T, P, IDS, false>, grid, kThreads, stream, a);
    }
}

}  // namespace

hipError_t launch_geometry(const GeometryArgs& a, int position_type, hipStream_t stream) {
    switch (position_type) {
        case 0: launch<int32_t, int64_t, false>(a, stream); break;
        case 1: launch<int32_t, int64_t, true>(a, stream); break;
        case 2: launch<int64_t, int64_t, true>(a, stream); break;
        case 3: launch<float, float, true>(a, stream); break;
        case 4: launch<double, double, true>(a, stream); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace lsso_hip
