// Host side of the filter scan (filter.hpp) and the kernels that prepare a search for it: the
// query operands, the scale of float32 rows, and the row list of an allow-mask.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "filter.hpp"
#include "select.hpp"

namespace zcgvs_hip {

template <int kKind, bool kWide>
int launchFilterKind(const ScanArgs& scan, const FilterArgs& args, const PhaseArgs& phase, const EmitArgs& emit,
                     int workgroups, hipStream_t stream);

namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr int kPrepareThreads = 256;
constexpr int kPrepareSplit = 4;     // workgroups per query group
constexpr int kUnitRows = 16;       // float32 rows sampled for the row unit
constexpr int kListRowsPerThread = 16;
constexpr int kListThreads = 256;
constexpr int kListRows = kListThreads * kListRowsPerThread;  // mask bytes per workgroup

int stepsPerPiece(int kind) { return kind == ZCGVS_DTYPE_F32 ? 2 : kind == ZCGVS_DTYPE_I8 ? 8 : 4; }

// Component that element e of lane group h holds in step s of a row, -1 for none: the scan's
// reading order (filter_kernel.hpp).
__device__ __forceinline__ int componentOf(int dtype, int dim, int s, int h, int e) {
    const int elems = dtype == ZCGVS_DTYPE_F32 ? 4 : dtype == ZCGVS_DTYPE_F16 ? 8 : 16;
    const int per_piece = dtype == ZCGVS_DTYPE_F32 ? 2 : dtype == ZCGVS_DTYPE_F16 ? 4 : 8;
    const int piece = s / per_piece;
    const int in_piece = s - piece * per_piece;
    int j, at;  // load of the piece, element of its chunk
    if (dtype == ZCGVS_DTYPE_F32) {
        j = 2 * in_piece + e / 4;
        at = e & 3;
    } else if (dtype == ZCGVS_DTYPE_F16) {
        j = in_piece;
        at = e;
    } else {
        j = in_piece / 2;
        at = 8 * (in_piece & 1) + e;
    }
    const int chunk = 16 * piece + 4 * j + h;
    const int whole = dim / elems;
    if (chunk < whole) {
        return chunk * elems + at;
    }
    // the partial chunk is read as the row's last `elems` components; the ones the chunk before
    // holds already are left out
    const int rest = dim - whole * elems;
    return chunk == whole && at >= elems - rest ? dim - elems + at : -1;
}

// Exponent e of the power of two that brings `peak` into [2^(top - 1), 2^top) (0 for a peak that is
// zero or not finite).
__device__ __forceinline__ int exponentBelow(float peak, int top) {
    if (!(peak > 0.0f) || !(peak <= 3.402823466e+38f)) {
        return 0;
    }
    int e = 0;
    frexpf(peak, &e);  // peak = m * 2^e, m in [0.5, 1)
    return min(126, max(-126, top - e));
}

// Block (g, part): query group g's constants (part 0 writes them) and its share of the group's
// operands. Block (0, 0) also clears the row list's count; with float32 rows, the blocks past the
// groups find the row unit: the power of two that brings the largest component of a sample of rows
// to [1, 2), which leaves a factor of 2^15 to float16's largest value, 2^14 to its smallest normal
// one and 2^24 to its smallest. (A smaller component loses up to that last one, which the bound's
// absolute part counts. A row that leaves the range at the top has no bound and is scored exactly
// for every query, kOperandNorm2, hence the middle: components 2^9 times the sample's, all that a
// peak near 2^7 allows, are met where rows' lengths vary.)
__global__ __launch_bounds__(kPrepareThreads) void filterPrepareKernel(ScanArgs scan, FilterArgs args) {
    const int t = threadIdx.x;
    const int dim = scan.dim;
    if (static_cast<int>(blockIdx.x) == args.groups) {
        if (blockIdx.y != 0) {
            return;
        }
        __shared__ float lds_peak[kPrepareThreads / kWave];
        const long long rows = min(static_cast<long long>(kUnitRows), scan.doc_count);
        const float* corpus = static_cast<const float*>(scan.corpus);
        float peak = 0.0f;
        // one wavefront per row, a 64-component stretch of each (at a place that moves along)
        const int lane = t & (kWave - 1);
#pragma unroll 4
        for (int r = t / kWave; r < rows; r += kPrepareThreads / kWave) {
            const long long row = r * (scan.doc_count / rows);
            const int at = (r * kWave + lane) % dim;
            const float x = fabsf(corpus[static_cast<std::size_t>(row) * dim + at]);
            peak = x <= 3.402823466e+38f ? fmaxf(peak, x) : peak;
        }
#pragma unroll
        for (int m = kWave / 2; m > 0; m >>= 1) {
            peak = fmaxf(peak, waveXor(peak, m));
        }
        if (lane == 0) {
            lds_peak[t / kWave] = peak;
        }
        __syncthreads();
        if (t == 0) {
            for (int w = 1; w < kPrepareThreads / kWave; ++w) {
                peak = fmaxf(peak, lds_peak[w]);
            }
            *args.row_unit = ldexpf(1.0f, -exponentBelow(peak, 1));
        }
        return;
    }
    __shared__ float lds_scale[kFilterGroup];
    const int group = blockIdx.x;
    if (group == 0 && blockIdx.y == 0 && t == 0 && args.list_count != nullptr) {
        *args.list_count = 0u;
    }
    {
        // 16 threads per query
        const int q = group * kFilterGroup + t / 16;
        const float* src = static_cast<const float*>(scan.queries) + static_cast<std::size_t>(min(q, scan.batch - 1)) * dim;
        float peak = 0.0f;
        float norm2 = 0.0f;
        bool finite = true;
#pragma unroll 8
        for (int j = t & 15; j < dim; j += 16) {
            const float x = src[j];
            peak = fmaxf(peak, fabsf(x));
            finite = finite && fabsf(x) <= 3.402823466e+38f;
            norm2 = fmaf(x, x, norm2);
        }
#pragma unroll
        for (int m = 1; m < 16; m <<= 1) {
            peak = fmaxf(peak, waveXor(peak, m));
            norm2 += waveXor(norm2, m);
            finite = (waveXor(finite ? 1 : 0, m) != 0) && finite;
        }
        if ((t & 15) == 0) {
            const float scale = finite ? ldexpf(1.0f, exponentBelow(peak, 15)) : 1.0f;
            lds_scale[t / 16] = scale;
            if (blockIdx.y == 0) {
                FilterQuery out;
                out.scale = scale;
                out.norm2 = norm2;
                // (within these bounds no square, product or scaled threshold leaves float32's range
                // unnoticed; an all-zero query is in them)
                out.usable = finite && (peak == 0.0f || (peak > 1e-17f && peak < 1e17f)) ? 1.0f : 0.0f;
                out.zero = finite && peak == 0.0f && scan.metric != ZCGVS_METRIC_L2 && scan.lexical == nullptr ? 1.0f : 0.0f;
                args.queries[group * kFilterGroup + t / 16] = out;
            }
        }
    }
    __syncthreads();
    v8h* out = reinterpret_cast<v8h*>(args.operands) + static_cast<std::size_t>(group) * args.steps * kWave;
    for (int item = static_cast<int>(blockIdx.y) * kPrepareThreads + t; item < args.steps * kWave;
         item += kPrepareSplit * kPrepareThreads) {
        const int step = item / kWave;
        const int lane = item & (kWave - 1);
        const int q = group * kFilterGroup + (lane & 15);
        const float* src = static_cast<const float*>(scan.queries) + static_cast<std::size_t>(min(q, scan.batch - 1)) * dim;
        const float scale = lds_scale[lane & 15];
        v8h value;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int c = componentOf(scan.dtype, dim, step, lane >> 4, e);
            const float x = src[max(c, 0)];
            value[e] = static_cast<_Float16>(c >= 0 && q < scan.batch ? x * scale : 0.0f);
        }
        out[item] = value;
    }
}

// A certain threshold per query from the sketch: a lower edge below the width-th best slot score,
// one block per query. The slot scores' ordered bits are counted in 2048 bins over their range,
// and the threshold is the lower edge of the bin where the count from the top reaches `width` (at
// most 1/2048 of the range below that slot's score: an exact selection of it takes three passes
// for nothing). With fewer slots than that holding a score, the threshold lets every row pass that
// a selection in which only row numbers decide would take. Also clears the flagged list.
constexpr int kThresholdThreads = 512;
constexpr int kThresholdBins = 2048;
constexpr int kThresholdSlots = kMaxSketchSlots / kThresholdThreads;

__global__ __launch_bounds__(kThresholdThreads) void filterThresholdKernel(FilterArgs args, long long rows,
                                                                           const float* __restrict__ sketch, int slots,
                                                                           int batch, int width,
                                                                           std::uint64_t* __restrict__ tau,
                                                                           std::uint64_t* __restrict__ tau_safe,
                                                                           std::uint32_t* __restrict__ flag_count) {
    constexpr int kWaves = kThresholdThreads / kWave;
    constexpr int kBinsPerThread = kThresholdBins / kThresholdThreads;
    __shared__ std::uint32_t lds_bins[kThresholdBins];
    __shared__ std::uint32_t lds_low[kWaves], lds_high[kWaves], lds_sums[kWaves];
    const int q = blockIdx.x;
    const int t = threadIdx.x;
    // (with an allow-mask, only if the merge's sweep finds its rows among the first 8192 or so, about 70 us: of
    // a few rows let through, the scan scores every pair sooner)
    const float zero = args.queries[q].zero;
    auto leftOut = [&]() {
        return zero != 0.0f &&
               (args.list_count == nullptr || rows * width <= 8192LL * static_cast<long long>(*args.list_count));
    };
    std::uint32_t v[kThresholdSlots];  // ordered bits; 0: no score
    std::uint32_t low = 0xFFFFFFFFu;
    std::uint32_t high = 0u;
#pragma unroll
    for (int r = 0; r < kThresholdSlots; ++r) {
        const int s = r * kThresholdThreads + t;
        const float x = s < slots ? sketch[static_cast<std::size_t>(s) * batch + q] : -INFINITY;
        v[r] = x > -INFINITY ? orderedBits(x) : 0u;
        low = v[r] != 0u ? min(low, v[r]) : low;
        high = max(high, v[r]);
    }
#pragma unroll
    for (int b = 0; b < kBinsPerThread; ++b) {
        lds_bins[b * kThresholdThreads + t] = 0u;
    }
    if (q == 0 && t == 0) {
        *flag_count = 0u;
    }
#pragma unroll
    for (int m = kWave / 2; m > 0; m >>= 1) {
        low = min(low, waveXor(low, m));
        high = max(high, waveXor(high, m));
    }
    if ((t & (kWave - 1)) == 0) {
        lds_low[t / kWave] = low;
        lds_high[t / kWave] = high;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        low = min(low, lds_low[w]);
        high = max(high, lds_high[w]);
    }
    // bins of 2^shift: the smallest for which the range fits them
    const std::uint32_t range = high >= low ? high - low : 0u;
    const int shift = max(0, 32 - __clz(static_cast<int>(range)) - 11);
#pragma unroll
    for (int r = 0; r < kThresholdSlots; ++r) {
        if (v[r] != 0u) {
            atomicAdd(&lds_bins[(v[r] - low) >> shift], 1u);
        }
    }
    __syncthreads();
    // thread t owns the t-th bins counted from the top
    std::uint32_t own[kBinsPerThread];
    std::uint32_t sum = 0u;
#pragma unroll
    for (int b = 0; b < kBinsPerThread; ++b) {
        own[b] = lds_bins[kThresholdBins - 1 - kBinsPerThread * t - b];
        sum += own[b];
    }
    std::uint32_t total;
    std::uint32_t above = blockInclusiveSum<kThresholdThreads>(sum, lds_sums, &total) - sum;
    const std::uint32_t need = static_cast<std::uint32_t>(width);
#pragma unroll
    for (int b = 0; b < kBinsPerThread; ++b) {
        if (above < need && above + own[b] >= need) {
            const std::uint32_t edge =
                low + (static_cast<std::uint32_t>(kThresholdBins - 1 - kBinsPerThread * t - b) << shift);
            const std::uint64_t key = leftOut() ? kFilterNoKey : static_cast<std::uint64_t>(edge) << 32;
            tau[q] = key;
            tau_safe[q] = key;
        }
        above += own[b];
    }
    if (t == 0 && total < need) {
        // rows 0 to width - 1 alone are width keys at or above this one
        const std::uint64_t key = leftOut() ? kFilterNoKey : makeKey(__uint_as_float(0x7FC00000u), need - 1u) - 1ull;
        tau[q] = key;
        tau_safe[q] = key;
    }
}

// Per-vector int8: the operands are the queries' codes as they lie, chunk 16 piece + 4 j + h (step 4
// piece + j) of a row's reading order at lane group h; the constants are the query scales.
__global__ __launch_bounds__(kPrepareThreads) void filterPrepareCodesKernel(ScanArgs scan, FilterArgs args) {
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    const int t = threadIdx.x;
    const int group = blockIdx.x;
    const int chunks = scan.dim / 16;
    if (group == 0 && blockIdx.y == 0 && t == 0 && args.list_count != nullptr) {
        *args.list_count = 0u;
    }
    if (blockIdx.y == 0) {
        // 16 threads per query
        const int q = group * kFilterGroup + t / 16;
        const std::uint8_t* src = static_cast<const std::uint8_t*>(scan.queries) + static_cast<std::size_t>(min(q, scan.batch - 1)) * scan.dim;
        std::uint32_t any = 0u;
#pragma unroll 4
        for (int c = t & 15; c < chunks; c += 16) {
            const u32x4 codes = *reinterpret_cast<const u32x4*>(src + 16 * c);
            any |= codes[0] | codes[1] | codes[2] | codes[3];
        }
#pragma unroll
        for (int m = 1; m < 16; m <<= 1) {
            any |= waveXor(any, m);
        }
        if ((t & 15) == 0) {
            FilterQuery out = {};
            out.scale = q < scan.batch ? scan.query_scales[q] : 0.0f;
            out.usable = 1.0f;
            out.zero = any == 0u ? 1.0f : 0.0f;
            args.queries[q] = out;
        }
    }
    u32x4* dst = reinterpret_cast<u32x4*>(args.operands) + static_cast<std::size_t>(group) * args.steps * kWave;
    for (int item = static_cast<int>(blockIdx.y) * kPrepareThreads + t; item < args.steps * kWave;
         item += kPrepareSplit * kPrepareThreads) {
        const int step = item / kWave;
        const int lane = item & (kWave - 1);
        const int q = group * kFilterGroup + (lane & 15);
        const int chunk = 4 * step + (lane >> 4);
        u32x4 codes = {0u, 0u, 0u, 0u};
        if (q < scan.batch && chunk < chunks) {
            codes = *reinterpret_cast<const u32x4*>(static_cast<const std::uint8_t*>(scan.queries) +
                                                    static_cast<std::size_t>(q) * scan.dim + 16 * chunk);
        }
        dst[item] = codes;
    }
}

// The rows an allow-mask lets through, in no order across workgroups, 4096 mask bytes each, and the
// masked ones of the first keep_masked rows (filterMaskedRows) with kMaskedRow set.
__global__ __launch_bounds__(kListThreads) void filterListKernel(const std::uint8_t* __restrict__ mask, long long rows,
                                                                 long long keep_masked, std::uint32_t* __restrict__ list,
                                                                 std::uint32_t* __restrict__ count) {
    __shared__ std::uint32_t lds_scan[kListThreads / kWave];
    __shared__ std::uint32_t lds_first;
    const int t = threadIdx.x;
    const long long first = static_cast<long long>(blockIdx.x) * kListRows + t * kListRowsPerThread;
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4), aligned(1)));
    std::uint32_t bits = 0u;  // rows of this thread that are listed
    std::uint32_t allowed = 0u;
    if (first + kListRowsPerThread <= rows) {
        const u32x4 words = *reinterpret_cast<const u32x4*>(mask + first);
#pragma unroll
        for (int i = 0; i < kListRowsPerThread; ++i) {
            allowed |= ((words[i / 4] >> (8 * (i & 3))) & 0xFFu) != 0u ? 1u << i : 0u;
        }
        bits = 0xFFFFu;
    } else {
        for (int i = 0; i < kListRowsPerThread; ++i) {
            if (first + i < rows) {
                bits |= 1u << i;
                allowed |= mask[first + i] != 0 ? 1u << i : 0u;
            }
        }
    }
    if (first + kListRowsPerThread > keep_masked) {
        std::uint32_t kept = 0u;
        for (int i = 0; i < kListRowsPerThread; ++i) {
            kept |= first + i < keep_masked ? 1u << i : 0u;
        }
        bits &= allowed | kept;
    }
    std::uint32_t total = 0u;
    const std::uint32_t own = static_cast<std::uint32_t>(__popc(bits));
    const std::uint32_t before = blockInclusiveSum<kListThreads>(own, lds_scan, &total) - own;
    if (t == 0) {
        lds_first = atomicAdd(count, total);
    }
    __syncthreads();
    std::uint32_t at = lds_first + before;
    while (bits != 0u) {
        const int i = __ffs(bits) - 1;
        bits &= bits - 1u;
        const std::uint32_t row = static_cast<std::uint32_t>(first + i);
        list[at++] = (allowed >> i) & 1u ? row : row | 0x80000000u;
    }
}

}  // namespace

FilterShape filterShape(const ScanArgs& scan, int width) {
    FilterShape shape;
    const int kind = filterKind(scan);
    if (kind == ZCGVS_DTYPE_BINARY) {
        return shape;
    }
    const std::size_t bytes = rowBytes(scan.dtype, scan.dim);
    // rows of one chunk to 4 KB (the exact scores' lane groups), the corpus 16-byte aligned as the
    // other scans need it; an int8 scale whose products stay in range
    if (bytes < 16 || bytes > 4096 || !aligned16(scan.corpus) || scan.batch < 1) {
        return shape;
    }
    if (kind == kFilterPerVector && (bytes % 16 != 0 || bytes > 1024)) {
        return shape;
    }
    // Hybrid searches: float rows, a weight under which a higher dense score never lowers the fused
    // one, and no mask (a masked row's fused score depends on its lexical one).
    if (scan.lexical != nullptr && ((kind != ZCGVS_DTYPE_F32 && kind != ZCGVS_DTYPE_F16) || scan.mask != nullptr ||
                                    !(scan.dense_weight >= 0.0f && scan.dense_weight <= 1.0f))) {
        return shape;
    }
    if (kind == ZCGVS_DTYPE_I8 && !(scan.scale > 1e-15f && scan.scale < 1e15f)) {
        return shape;
    }
    const int slots = kFilterSketchSlots * deviceComputeUnits();
    if (slots > kMaxSketchSlots || width > slots / 4) {
        return shape;  // (too few sketch slots for this many keys)
    }
    shape.steps = static_cast<int>((bytes + 255) / 256) * stepsPerPiece(kind);
    const int most = std::min<int>(kFilterMaxGroups, static_cast<int>(kFilterOperandBytes / 1024) / shape.steps);
    if (most < 1) {
        return shape;
    }
    const int groups = (scan.batch + kFilterGroup - 1) / kFilterGroup;
    // the instantiated group counts: 1, 2, 4 and 8
    constexpr int kCounts[] = {1, 2, 4, 8};
    int largest = 1;
    for (const int c : kCounts) {
        largest = c <= (scan.lexical != nullptr ? std::min(most, 2) : most) ? c : largest;
    }
    int launches = (groups + largest - 1) / largest;
    const int even = (groups + launches - 1) / launches;  // as even a split as the counts allow
    for (const int c : kCounts) {
        if (c >= even && shape.groups_per_launch == 0) {
            shape.groups_per_launch = c;
        }
    }
    shape.tile_rows =
        1 << filterTileLog2(scan.doc_count,
                            kFilterBlockRows * filterBlocks(filterSlots(static_cast<int>((bytes + 255) / 256)),
                                                            shape.groups_per_launch, scan.lexical != nullptr),
                            deviceComputeUnits() * kFilterWaves,
                            8LL * scan.batch * width > scan.doc_count ? 0 : 4);  // (about two pairs per key are scored)
    launches = (groups + shape.groups_per_launch - 1) / shape.groups_per_launch;
    shape.groups = launches * shape.groups_per_launch;
    shape.supported = true;
    return shape;
}

int launchFilterPrepare(const ScanArgs& scan, const FilterArgs& args, hipStream_t stream) {
    const bool f32 = scan.dtype == ZCGVS_DTYPE_F32;
    const dim3 grid(static_cast<unsigned>(args.groups + (f32 ? 1 : 0)), kPrepareSplit);
    if (filterKind(scan) == kFilterPerVector) {
        filterPrepareCodesKernel<<<grid, kPrepareThreads, 0, stream>>>(scan, args);
    } else {
        filterPrepareKernel<<<grid, kPrepareThreads, 0, stream>>>(scan, args);
    }
    ZCGVS_LAUNCH_CHECK("filter prepare");
    if (args.list != nullptr) {
        const unsigned blocks = static_cast<unsigned>((scan.doc_count + kListRows - 1) / kListRows);
        const long long keep = filterMaskedRows(scan.doc_count, args.width);
        filterListKernel<<<blocks, kListThreads, 0, stream>>>(scan.mask, scan.doc_count, keep, args.list, args.list_count);
        ZCGVS_LAUNCH_CHECK("filter row list");
    }
    return ZCGVS_OK;
}

int launchFilterThreshold(const FilterArgs& args, long long rows, const float* sketch, int slots, int batch,
                          std::uint64_t* tau, std::uint64_t* tau_safe, std::uint32_t* flag_count, hipStream_t stream) {
    if (slots < 1 || slots > kMaxSketchSlots || args.width < 1) {
        return setError(ZCGVS_ERR_RUNTIME, "zcgvs filter: sketch shape out of range");
    }
    filterThresholdKernel<<<batch, kThresholdThreads, 0, stream>>>(args, rows, sketch, slots, batch, args.width, tau, tau_safe,
                                                                   flag_count);
    ZCGVS_LAUNCH_CHECK("filter threshold");
    return ZCGVS_OK;
}

int launchFilterScan(const ScanArgs& scan, const FilterArgs& args, const PhaseArgs& phase, const EmitArgs& emit,
                     int workgroups, hipStream_t stream) {
    const bool wide = rowBytes(scan.dtype, scan.dim) > 2 * 256;
    switch (filterKind(scan)) {
        case kFilterPerVector:
            return wide ? launchFilterKind<kFilterPerVector, true>(scan, args, phase, emit, workgroups, stream)
                        : launchFilterKind<kFilterPerVector, false>(scan, args, phase, emit, workgroups, stream);
        case ZCGVS_DTYPE_F32:
            return wide ? launchFilterKind<ZCGVS_DTYPE_F32, true>(scan, args, phase, emit, workgroups, stream)
                        : launchFilterKind<ZCGVS_DTYPE_F32, false>(scan, args, phase, emit, workgroups, stream);
        case ZCGVS_DTYPE_F16:
            return wide ? launchFilterKind<ZCGVS_DTYPE_F16, true>(scan, args, phase, emit, workgroups, stream)
                        : launchFilterKind<ZCGVS_DTYPE_F16, false>(scan, args, phase, emit, workgroups, stream);
        case ZCGVS_DTYPE_I8:
            return wide ? launchFilterKind<ZCGVS_DTYPE_I8, true>(scan, args, phase, emit, workgroups, stream)
                        : launchFilterKind<ZCGVS_DTYPE_I8, false>(scan, args, phase, emit, workgroups, stream);
        default:
            return setError(ZCGVS_ERR_INVALID_ARGUMENT, "zcgvs: filter scan does not take this shape");
    }
}

}  // namespace zcgvs_hip
