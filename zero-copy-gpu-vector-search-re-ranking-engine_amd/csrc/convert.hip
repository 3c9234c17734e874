// Index-side conversions (src/cuda/convert.cu:17-53, 55-93), the per-row int8 quantizer of the
// per-vector mode, and the on-device synthetic generator.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.hpp"
#include "rescore.hpp"

namespace zcgvs_hip {

namespace {

constexpr int kConvertThreads = 256;
constexpr std::size_t kMaxConvertBlocks = 65535;
constexpr int kConvertUnroll = 4;  // 16-byte loads in flight per lane of the elementwise conversions

unsigned convertBlocks(std::size_t count) {
    return static_cast<unsigned>(
        std::max<std::size_t>(1, std::min(kMaxConvertBlocks, (count + kConvertThreads - 1) / kConvertThreads)));
}

// Blocks of the vector conversions (convertElements).
unsigned vectorBlocks(std::size_t count) {
    const std::size_t per_block = static_cast<std::size_t>(kConvertThreads) * 4 * kConvertUnroll;
    return static_cast<unsigned>(std::max<std::size_t>(1, std::min(kMaxConvertBlocks, (count + per_block - 1) / per_block)));
}

// Every conversion below is bound by HBM: 4 bytes read per component and its stored size written.
// Loads are 16 bytes a lane (whole kilobytes a wavefront) and several are in flight per lane; the
// source is read once, so the loads carry the non-temporal hint. Measured at 500,000 x 768 against a
// streaming copy's 5.35 TB/s (element by element before -> now): float16 528 -> 399 us, matrix-scale
// int8 480 -> 323 us, per-row int8 789 -> 337 us (5.7 TB/s), sign bits 5200 -> 307 us.
typedef float f32x4 __attribute__((ext_vector_type(4)));

// dst[i] = convert(src[i]) for groups of 4 elements; `vectors` groups, then the elements past the
// last whole group one by one. src and dst are aligned to their 4-element groups.
template <typename Out, typename Convert>
__device__ __forceinline__ void convertElements(const float* __restrict__ src, Out* __restrict__ dst,
                                                std::size_t count, Convert&& convert) {
    typedef Out out4 __attribute__((ext_vector_type(4)));
    const std::size_t vectors = count / 4;
    const std::size_t block_vectors = static_cast<std::size_t>(blockDim.x) * kConvertUnroll;
    const f32x4* from = reinterpret_cast<const f32x4*>(src);
    out4* to = reinterpret_cast<out4*>(dst);
    for (std::size_t base = static_cast<std::size_t>(blockIdx.x) * block_vectors; base < vectors;
         base += static_cast<std::size_t>(gridDim.x) * block_vectors) {
        f32x4 v[kConvertUnroll];
#pragma unroll
        for (int u = 0; u < kConvertUnroll; ++u) {
            const std::size_t i = base + static_cast<std::size_t>(u) * blockDim.x + threadIdx.x;
            if (i < vectors) {
                v[u] = __builtin_nontemporal_load(from + i);
            }
        }
#pragma unroll
        for (int u = 0; u < kConvertUnroll; ++u) {
            const std::size_t i = base + static_cast<std::size_t>(u) * blockDim.x + threadIdx.x;
            if (i < vectors) {
                out4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    o[e] = convert(v[u][e]);
                }
                to[i] = o;
            }
        }
    }
    const std::size_t tail = vectors * 4 + threadIdx.x;
    if (blockIdx.x == 0 && threadIdx.x < 4 && tail < count) {
        dst[tail] = convert(src[tail]);
    }
}

// As above for buffers that are not aligned to 4 elements: one element a lane.
template <typename Out, typename Convert>
__device__ __forceinline__ void convertUnaligned(const float* __restrict__ src, Out* __restrict__ dst,
                                                 std::size_t count, Convert&& convert) {
    const std::size_t stride = static_cast<std::size_t>(gridDim.x) * blockDim.x;
    for (std::size_t i = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < count; i += stride) {
        dst[i] = convert(src[i]);
    }
}

template <bool kAligned>
__global__ __launch_bounds__(kConvertThreads) void convertF32ToF16Kernel(const float* __restrict__ src,
                                                                         _Float16* __restrict__ dst,
                                                                         std::size_t count) {
    const auto convert = [](float x) { return static_cast<_Float16>(x); };  // round to nearest even
    if constexpr (kAligned) {
        convertElements(src, dst, count, convert);
    } else {
        convertUnaligned(src, dst, count, convert);
    }
}

// q = clamp(rint(x * inverse_scale), -127, 127): round half to even, like nearbyint in
// tests/cpp/cpu_reference.hpp:51-62.
__device__ __forceinline__ signed char quantize(float x, float inverse_scale) {
    const float scaled = rintf(x * inverse_scale);
    return static_cast<signed char>(fminf(fmaxf(scaled, -127.0f), 127.0f));
}

template <bool kAligned>
__global__ __launch_bounds__(kConvertThreads) void convertF32ToI8Kernel(const float* __restrict__ src,
                                                                        signed char* __restrict__ dst,
                                                                        std::size_t count, float inverse_scale) {
    const auto convert = [inverse_scale](float x) { return quantize(x, inverse_scale); };
    if constexpr (kAligned) {
        convertElements(src, dst, count, convert);
    } else {
        convertUnaligned(src, dst, count, convert);
    }
}

// Word w of a row: bit b set iff x[32w + b] >= 0 (so -0.0 sets it and NaN does not); dimensions
// past dim stay zero. A wavefront reads 64 consecutive components of a row at a time (a piece),
// whose signs one ballot turns into two words, kPackPieces pieces per step with their loads in
// flight together; lanes 2u and 2u + 1 then store the words of piece u.
constexpr int kPackPieces = 16;

__global__ __launch_bounds__(kConvertThreads) void packBinaryKernel(const float* __restrict__ src,
                                                                    std::uint32_t* __restrict__ dst, long long pieces,
                                                                    int pieces_per_row, int dim, int words) {
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const long long waves = static_cast<long long>(gridDim.x) * (kConvertThreads / kWave);
    const long long first = static_cast<long long>(blockIdx.x) * (kConvertThreads / kWave) + wave;
    for (long long step = first * kPackPieces; step < pieces; step += waves * kPackPieces) {
        // piece p of row r holds components 64 p .. 64 p + 63 (fewer in a row's last piece)
        long long row = step / pieces_per_row;
        int piece = static_cast<int>(step - row * pieces_per_row);
        float x[kPackPieces];
        long long word_at = 0;  // this lane's word: dst[word_at] while word_ok
        bool word_ok = false;
#pragma unroll
        for (int u = 0; u < kPackPieces; ++u) {
            const int j = piece * kWave + lane;
            x[u] = -1.0f;
            if (step + u < pieces && j < dim) {
                x[u] = __builtin_nontemporal_load(src + static_cast<std::size_t>(row) * dim + j);
            }
            if ((lane >> 1) == u) {
                const int word = 2 * piece + (lane & 1);
                word_at = row * words + word;
                word_ok = step + u < pieces && word < words;
            }
            if (++piece == pieces_per_row) {
                piece = 0;
                ++row;
            }
        }
        std::uint32_t bits = 0u;
#pragma unroll
        for (int u = 0; u < kPackPieces; ++u) {
            const unsigned long long signs = __ballot(x[u] >= 0.0f);
            if ((lane >> 1) == u) {
                bits = static_cast<std::uint32_t>((lane & 1) != 0 ? signs >> 32 : signs);
            }
        }
        if (word_ok) {
            dst[word_at] = bits;
        }
    }
}

// Per-row scale s = max|x| / 127 (1 for an all-zero row), then the quantizer above with the
// reciprocal 1/s. A row is read once, by kLanes lanes that keep it in registers between the
// maximum and the quantization: kVectors groups of 4 components a lane (whole 16-byte groups; the
// caller checks dim % 4 and the alignment). Rows of up to 256 components take 16 lanes, up to 512
// 32, so a wavefront's loads stay whole kilobytes.
template <int kLanes, int kVectors>
__global__ __launch_bounds__(kConvertThreads) void quantizeRowsKernel(const float* __restrict__ src, int rows, int dim,
                                                                      std::int8_t* __restrict__ dst,
                                                                      float* __restrict__ scales) {
    typedef signed char i8x4 __attribute__((ext_vector_type(4)));
    const int lane = threadIdx.x & (kLanes - 1);
    const long long row = static_cast<long long>(blockIdx.x) * (kConvertThreads / kLanes) + threadIdx.x / kLanes;
    if (row >= rows) {
        return;  // (a whole row's lanes)
    }
    const int vectors = dim / 4;
    const f32x4* values = reinterpret_cast<const f32x4*>(src + static_cast<std::size_t>(row) * dim);
    f32x4 x[kVectors];
#pragma unroll
    for (int i = 0; i < kVectors; ++i) {
        const int c = i * kLanes + lane;
        x[i] = c < vectors ? __builtin_nontemporal_load(values + c) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    float peak = 0.0f;
#pragma unroll
    for (int i = 0; i < kVectors; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            peak = fmaxf(peak, fabsf(x[i][e]));
        }
    }
#pragma unroll
    for (int offset = kLanes / 2; offset > 0; offset >>= 1) {
        peak = fmaxf(peak, waveXor(peak, offset));
    }
    const float scale = peak > 0.0f ? peak / 127.0f : 1.0f;
    const float inverse = 1.0f / scale;
    i8x4* out = reinterpret_cast<i8x4*>(dst + static_cast<std::size_t>(row) * dim);
#pragma unroll
    for (int i = 0; i < kVectors; ++i) {
        const int c = i * kLanes + lane;
        if (c < vectors) {
            i8x4 codes;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                codes[e] = quantize(x[i][e], inverse);
            }
            out[c] = codes;
        }
    }
    if (lane == 0) {
        scales[row] = scale;
    }
}

// The same for any dim and alignment, one wavefront per row: rows of up to 64 * kKept components
// stay in registers, wider ones are read again for the quantization.
constexpr int kKept = 16;

__global__ __launch_bounds__(kConvertThreads) void quantizeAnyRowsKernel(const float* __restrict__ src, int rows,
                                                                         int dim, std::int8_t* __restrict__ dst,
                                                                         float* __restrict__ scales) {
    const int lane = threadIdx.x & (kWave - 1);
    const long long row = static_cast<long long>(blockIdx.x) * (blockDim.x / kWave) + threadIdx.x / kWave;
    if (row >= rows) {
        return;
    }
    const float* values = src + static_cast<std::size_t>(row) * dim;
    float x[kKept];
    float peak = 0.0f;
#pragma unroll
    for (int i = 0; i < kKept; ++i) {
        const int j = i * kWave + lane;
        x[i] = j < dim ? values[j] : 0.0f;
        peak = fmaxf(peak, fabsf(x[i]));
    }
    for (int j = kKept * kWave + lane; j < dim; j += kWave) {
        peak = fmaxf(peak, fabsf(values[j]));
    }
#pragma unroll
    for (int offset = kWave / 2; offset > 0; offset >>= 1) {
        peak = fmaxf(peak, waveXor(peak, offset));
    }
    const float scale = peak > 0.0f ? peak / 127.0f : 1.0f;
    const float inverse = 1.0f / scale;
    std::int8_t* out = dst + static_cast<std::size_t>(row) * dim;
#pragma unroll
    for (int i = 0; i < kKept; ++i) {
        const int j = i * kWave + lane;
        if (j < dim) {
            out[j] = quantize(x[i], inverse);
        }
    }
    for (int j = kKept * kWave + lane; j < dim; j += kWave) {
        out[j] = quantize(values[j], inverse);
    }
    if (lane == 0) {
        scales[row] = scale;
    }
}

template <int kLanes>
void launchQuantizeVectors(const float* src, int rows, int dim, std::int8_t* dst, float* scales, hipStream_t stream) {
    constexpr int kRows = kConvertThreads / kLanes;
    const unsigned blocks = static_cast<unsigned>((static_cast<long long>(rows) + kRows - 1) / kRows);
    switch ((dim / 4 + kLanes - 1) / kLanes) {
        case 1: quantizeRowsKernel<kLanes, 1><<<blocks, kConvertThreads, 0, stream>>>(src, rows, dim, dst, scales); break;
        case 2: quantizeRowsKernel<kLanes, 2><<<blocks, kConvertThreads, 0, stream>>>(src, rows, dim, dst, scales); break;
        case 3: quantizeRowsKernel<kLanes, 3><<<blocks, kConvertThreads, 0, stream>>>(src, rows, dim, dst, scales); break;
        default: quantizeRowsKernel<kLanes, 4><<<blocks, kConvertThreads, 0, stream>>>(src, rows, dim, dst, scales); break;
    }
}

// ---- synthetic data ------------------------------------------------------------------------
__device__ __forceinline__ std::uint64_t splitmix64(std::uint64_t x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

// Uniform double in (0, 1) from the top 53 bits.
__device__ __forceinline__ double unitOpen(std::uint64_t bits) {
    return (static_cast<double>(bits >> 11) + 0.5) * (1.0 / 9007199254740992.0);
}

// One wavefront per row: element pair p of row r comes from splitmix64 of
// (seed, r, p); Box-Muller in double; rounded to float; the row is divided by its float32 norm
// (squares summed by the wavefront's tree reduction).
__global__ __launch_bounds__(256) void generateKernel(float* __restrict__ out, long long rows,
                                                      int dim, std::uint64_t seed,
                                                      long long row_offset) {
    const int lane = threadIdx.x & (kWave - 1);
    const long long local = static_cast<long long>(blockIdx.x) * (blockDim.x / kWave) + threadIdx.x / kWave;
    if (local >= rows) {
        return;
    }
    const std::uint64_t row = static_cast<std::uint64_t>(local + row_offset);
    const std::uint64_t row_seed = splitmix64(seed ^ splitmix64(row));
    float* values = out + static_cast<std::size_t>(local) * dim;
    const int pairs = (dim + 1) / 2;
    float sum = 0.0f;
    for (int p = lane; p < pairs; p += kWave) {
        const std::uint64_t a = splitmix64(row_seed + 2ull * static_cast<std::uint64_t>(p));
        const std::uint64_t b = splitmix64(row_seed + 2ull * static_cast<std::uint64_t>(p) + 1ull);
        const double radius = sqrt(-2.0 * log(unitOpen(a)));
        const double angle = 6.283185307179586 * unitOpen(b);
        const float x0 = static_cast<float>(radius * cos(angle));
        const float x1 = static_cast<float>(radius * sin(angle));
        values[2 * p] = x0;
        sum = fmaf(x0, x0, sum);
        if (2 * p + 1 < dim) {
            values[2 * p + 1] = x1;
            sum = fmaf(x1, x1, sum);
        }
    }
#pragma unroll
    for (int offset = kWave / 2; offset > 0; offset >>= 1) {
        sum += waveXor(sum, offset);
    }
    const float norm = sqrtf(sum);
    if (norm > 0.0f) {
        for (int j = lane; j < dim; j += kWave) {
            values[j] = values[j] / norm;
        }
    }
}

}  // namespace

int launchQuantizeRows(const float* src, int rows, int dim, std::int8_t* dst, float* scales,
                       hipStream_t stream) {
    const bool vectors = dim % 4 == 0 && aligned16(src) && (reinterpret_cast<std::uintptr_t>(dst) & 3u) == 0;
    if (vectors && dim <= 256) {
        launchQuantizeVectors<16>(src, rows, dim, dst, scales, stream);
    } else if (vectors && dim <= 512) {
        launchQuantizeVectors<32>(src, rows, dim, dst, scales, stream);
    } else if (vectors && dim <= 1024) {
        launchQuantizeVectors<64>(src, rows, dim, dst, scales, stream);
    } else {
        const unsigned blocks = static_cast<unsigned>((static_cast<long long>(rows) + 3) / 4);
        quantizeAnyRowsKernel<<<blocks, kConvertThreads, 0, stream>>>(src, rows, dim, dst, scales);
    }
    ZCGVS_LAUNCH_CHECK("quantize rows");
    return ZCGVS_OK;
}

}  // namespace zcgvs_hip

using namespace zcgvs_hip;

extern "C" {

int zcgvs_launch_convert_f32_to_f16(const float* d_src, void* d_dst_half, std::size_t count,
                                    zcgvs_stream_t stream) {
    if (count == 0) {
        return clearError();
    }
    if (d_src == nullptr || d_dst_half == nullptr) {
        return setError(ZCGVS_ERR_INVALID_ARGUMENT, "zcgvs convert: null device pointer");
    }
    _Float16* dst = static_cast<_Float16*>(d_dst_half);
    if (aligned16(d_src) && (reinterpret_cast<std::uintptr_t>(dst) & 7u) == 0) {
        convertF32ToF16Kernel<true><<<vectorBlocks(count), kConvertThreads, 0, toStream(stream)>>>(d_src, dst, count);
    } else {
        convertF32ToF16Kernel<false><<<convertBlocks(count), kConvertThreads, 0, toStream(stream)>>>(d_src, dst, count);
    }
    ZCGVS_LAUNCH_CHECK("convert f16");
    return clearError();
}

int zcgvs_launch_convert_f32_to_i8(const float* d_src, void* d_dst_int8, std::size_t count,
                                   float scale, zcgvs_stream_t stream) {
    if (count == 0) {
        return clearError();
    }
    if (d_src == nullptr || d_dst_int8 == nullptr) {
        return setError(ZCGVS_ERR_INVALID_ARGUMENT, "zcgvs convert: null device pointer");
    }
    const float inverse_scale = (scale > 0.0f) ? (1.0f / scale) : 0.0f;
    signed char* dst = static_cast<signed char*>(d_dst_int8);
    if (aligned16(d_src) && (reinterpret_cast<std::uintptr_t>(dst) & 3u) == 0) {
        convertF32ToI8Kernel<true><<<vectorBlocks(count), kConvertThreads, 0, toStream(stream)>>>(d_src, dst, count,
                                                                                                inverse_scale);
    } else {
        convertF32ToI8Kernel<false><<<convertBlocks(count), kConvertThreads, 0, toStream(stream)>>>(d_src, dst, count,
                                                                                                 inverse_scale);
    }
    ZCGVS_LAUNCH_CHECK("convert i8");
    return clearError();
}

int zcgvs_launch_pack_binary(const float* d_src, void* d_dst_words, int rows, int dim,
                             zcgvs_stream_t stream) {
    if (rows <= 0 || dim <= 0) {
        return clearError();
    }
    if (d_src == nullptr || d_dst_words == nullptr) {
        return setError(ZCGVS_ERR_INVALID_ARGUMENT, "zcgvs pack: null device pointer");
    }
    const int words = static_cast<int>(binaryWords(dim));
    const int pieces_per_row = (dim + kWave - 1) / kWave;
    const long long pieces = static_cast<long long>(rows) * pieces_per_row;
    constexpr long long kBlockPieces = kPackPieces * (kConvertThreads / kWave);
    const unsigned blocks = static_cast<unsigned>(
        std::min<long long>(kMaxConvertBlocks, (pieces + kBlockPieces - 1) / kBlockPieces));
    packBinaryKernel<<<blocks, kConvertThreads, 0, toStream(stream)>>>(d_src, static_cast<std::uint32_t*>(d_dst_words),
                                                                       pieces, pieces_per_row, dim, words);
    ZCGVS_LAUNCH_CHECK("pack binary");
    return clearError();
}

int zcgvs_launch_quantize_rows_i8(const float* d_src, int rows, int dim, std::int8_t* d_dst,
                                  float* d_scales, zcgvs_stream_t stream) {
    if (rows <= 0 || dim <= 0) {
        return clearError();
    }
    if (d_src == nullptr || d_dst == nullptr || d_scales == nullptr) {
        return setError(ZCGVS_ERR_INVALID_ARGUMENT, "zcgvs quantize: null device pointer");
    }
    const int status = launchQuantizeRows(d_src, rows, dim, d_dst, d_scales, toStream(stream));
    return status == ZCGVS_OK ? clearError() : status;
}

int zcgvs_generate_normalized(float* d_out, std::int64_t rows, int dim, std::uint64_t seed,
                              std::int64_t row_offset, zcgvs_stream_t stream) {
    if (rows <= 0 || dim <= 0) {
        return clearError();
    }
    if (d_out == nullptr) {
        return setError(ZCGVS_ERR_INVALID_ARGUMENT, "zcgvs generate: null device pointer");
    }
    const long long blocks = (rows + 3) / 4;
    if (blocks > 0x7FFFFFFFLL) {
        return setError(ZCGVS_ERR_INVALID_ARGUMENT, "zcgvs generate: too many rows per call");
    }
    generateKernel<<<static_cast<unsigned>(blocks), 256, 0, toStream(stream)>>>(
        d_out, rows, dim, seed, row_offset);
    ZCGVS_LAUNCH_CHECK("generate");
    return clearError();
}

}  // extern "C"
