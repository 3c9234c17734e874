// The filter scan's kernel (filter.hpp); filter_{f32,f16,i8,i8i8}_{narrow,wide}.hip instantiate it for
// their row type and width.
//
// Work split. One workgroup of 8 wavefronts per compute unit. The launch's query operands (up to
// 8 groups of 16 queries) lie in LDS for the whole launch; every wavefront streams rows of its own
// straight into registers, so no barrier runs in the loop (but for the cuts of a crowded search). A
// wavefront's tile is kBlocks blocks of 16 rows (fewer of them where few rows are to be shared by all
// wavefronts, filterTileLog2), of which it keeps kPieces pieces of 256 bytes of
// every row in flight (whole rows up to 1 KB), four 16-byte loads a lane, block and piece: as it
// consumes a load it starts the same one of the next tile. That is 8 to 16 KB of consecutive
// memory per wavefront, read at about one time; registers take rows at any alignment, which is why rows of no
// whole 16-byte chunks come this way too.
//
// A load instruction reads 8 lanes of 16 bytes per row, whole 128-byte lines, and goes through 2 KB of
// LDS per wavefront into the matrix core's layout (16 rows side by side); loads in that layout
// touch 16 lines of 16 bytes each per quarter-wavefront and stream half as fast.
//
// What bounds it: HBM. Measured (kernel alone; the VALU scan it replaces took 17 to 6 times as long for
// the whole search, the bf16 split scan 1.2): 1M x 768 float16, 32 queries, k = 100 279 us (5.5 of
// the 7.07 TB/s a streaming read reaches), 1M x 384 float32, 64 queries 48 and 238 us in two launches (5.4),
// 500,009 x 256 float32 L2 90 us (5.7), 400,009 x 300 float16 52 us (4.6), 300,000 allowed rows of 1M x 384
// float16 43 us (5.4), 1M x 384 int8, 8 queries 80 us (4.8: it also converts its codes to halves; 94 while the
// exact scores held all of a query's chunks and spilled registers). A ring of more registers (6 and 8
// pieces) made the compiler spill: 297-310 us for the first; tiles of 64 rows a piece at a time 577 us.
//
// MFMA layout (16x16x32 f16): the queries are the first operand (lane l supplies query l % 16 and 8
// dimensions), the rows the second (row l % 16, the same 8 dimensions), so a lane's results belong
// to one row (l % 16), queries 4 (l / 16) + i, and row properties (norm, mask) stay in their lane.
// Lane group h = l / 16 loads chunk 16 g + 4 j + h of piece g (j < 4). The products may sum the
// dimensions in any order, so float32 rows pair chunks j and j + 1 into one operand.
//
// A row's last chunk may be partial: it is then read as the row's last 16 bytes and the bytes that
// repeat earlier ones are cleared; chunks past it re-read it and are cleared whole. No load leaves
// its row.
#pragma once

#include <hip/hip_runtime.h>

#include "filter.hpp"
#include "scan_core.hpp"
#include "select.hpp"

namespace zcgvs_hip {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef unsigned int v4uAny __attribute__((ext_vector_type(4), aligned(1)));
typedef float v4fAny __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kFilterThreads = kFilterWaves * kWave;
constexpr int kPieceBytes = 256;
constexpr int kPieceLoads = 4;  // 16-byte chunks of a piece per lane
constexpr std::uint32_t kMaskedRow = 0x80000000u;
constexpr std::uint32_t kNoRow = 0xFFFFFFFFu;
constexpr int kParkSlots = 160;  // pairs a wavefront parks

template <int kKind>
struct FilterKind {
    static constexpr bool kInteger = kKind == kFilterPerVector;
    static constexpr int kDtype = kInteger ? ZCGVS_DTYPE_I8 : kKind;
    // products of 32 components (64 of int8 by int8) per piece
    static constexpr int kSteps = kKind == ZCGVS_DTYPE_F32 ? 2 : kKind == ZCGVS_DTYPE_I8 ? 8 : 4;
};
template <bool kInteger>
struct FilterSums {
    typedef v4f type;
};
template <>
struct FilterSums<true> {
    typedef v4i type;
};

// Square of float16's largest value. The conversion of a float32 row rounds toward zero, so a
// component beyond that value becomes it, not infinity, and the row's approximate scores say
// nothing. Its squared norm in operand units (a float32 sum of non-negative terms, at least any one
// of them) then reaches this: such a row is unbounded.
constexpr float kOperandNorm2 = 65504.0f * 65504.0f;

// Relative error of an approximate dot product, in units of |q| |x|: operand rounding (float16
// queries to nearest, 2^-11; float32 rows toward zero, another 2^-10), float32 accumulation over
// `steps` products of 32 (each taken at 2^-21, four times a rounding of every addition inside),
// and the exact score's own rounding. For rows that are not unbounded.
__host__ __device__ inline float filterRelative(int kind, int steps) {
    const float operands = kind == ZCGVS_DTYPE_F32 ? 1.48e-3f : 4.95e-4f;
    return operands + 4.8e-7f * static_cast<float>(steps) + 3.1e-5f;
}

// (Through a pointer to global memory: a flat load counts as an LDS operation as well, and every
// operand read would wait for the rows in flight.)
template <bool kOnce>
__device__ __forceinline__ v4u loadRowChunk(const std::uint8_t* p) {
    typedef const __attribute__((address_space(1))) v4uAny* GlobalChunk;
    const GlobalChunk at = (GlobalChunk)(reinterpret_cast<std::uintptr_t>(p));
    if constexpr (kOnce) {
        return __builtin_nontemporal_load(at);
    } else {
        return *at;
    }
}

// Words of a chunk with its first `skip` bytes cleared (skip >= 16: all).
__device__ __forceinline__ v4u keepFrom(v4u v, int skip) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const int s = skip - 4 * w;
        v[w] = s <= 0 ? v[w] : s >= 4 ? 0u : v[w] & (0xFFFFFFFFu << (8 * s));
    }
    return v;
}

// A term of an L2 distance: the decoded value is rounded before the difference is, as in the VALU scan
// (a compiler left to itself subtracts the int8 product unrounded here).
__device__ __forceinline__ float l2Difference(float q, float x) {
#pragma clang fp contract(off)
    return q - x;
}

// The exact score of `row` (allowed) for query q, by the L lanes of a group, as the VALU scan
// computes it: lane g of the group takes chunks g, g + L, ... in turn, groupSum adds the lanes.
template <int kKind, int L>
__device__ __forceinline__ float exactScoreLanes(const ScanArgs& scan, std::uint32_t row, int q, int lane) {
    using Traits = ChunkTraits<kKind>;
    constexpr int E = Traits::kElems;
    constexpr int kPer = 8;
    const int dim = scan.dim;
    const int row_bytes = static_cast<int>(rowBytes(kKind, dim));
    const int chunks = row_bytes / 16;
    const std::uint8_t* base = static_cast<const std::uint8_t*>(scan.corpus) + static_cast<std::size_t>(row) * row_bytes;
    const float* query = static_cast<const float*>(scan.queries) + static_cast<std::size_t>(q) * dim;
    const bool l2 = scan.metric == ZCGVS_METRIC_L2;
    // (every load of a turn without a branch, so that all are in flight together; the opaque copy keeps
    // their addresses from being computed, and kept in memory, outside the caller's loop. int8 takes two
    // turns: a chunk's 16 query values fill the registers)
    constexpr int kTurn = kKind == ZCGVS_DTYPE_I8 ? kPer / 2 : kPer;
    int group = lane % L;
    asm volatile("" : "+v"(group));
    float acc = 0.0f;
#pragma unroll 1
    for (int first = 0; first < kPer && first * L < chunks; first += kTurn) {
        v4u raw[kTurn];
#pragma unroll
        for (int t = 0; t < kTurn; ++t) {
            if ((first + t) * L < chunks) {  // (uniform)
                raw[t] = loadRowChunk<false>(base + min(group + (first + t) * L, chunks - 1) * 16);
            }
        }
        float qe[kTurn][E];
#pragma unroll
        for (int t = 0; t < kTurn; ++t) {
            if ((first + t) * L < chunks) {  // (uniform)
                const float* qv = query + min((group + (first + t) * L) * E, dim - E);
#pragma unroll
                for (int e = 0; e < E; e += 4) {
                    const v4f part = *reinterpret_cast<const v4fAny*>(qv + e);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        qe[t][e + i] = part[i];
                    }
                }
            }
        }
#pragma unroll
        for (int t = 0; t < kTurn; ++t) {
            if (group + (first + t) * L < chunks) {
                float v[E];
                Traits::decode(make_uint4(raw[t][0], raw[t][1], raw[t][2], raw[t][3]), scan.scale, v);
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const float d = l2 ? l2Difference(qe[t][e], v[e]) : v[e];
                    acc = fmaf(l2 ? d : qe[t][e], d, acc);
                }
            }
        }
    }
    const float total = groupSum<L>(acc);
    return l2 ? -total : total;
}

// The same for rows of no whole 16-byte chunks, by a whole wavefront, as the launchers' scalar
// scan computes it.
template <int kKind>
__device__ __forceinline__ float exactScoreStrided(const ScanArgs& scan, std::uint32_t row, int q, int lane) {
    const int dim = scan.dim;
    const std::uint8_t* values = static_cast<const std::uint8_t*>(scan.corpus) + static_cast<std::size_t>(row) * rowBytes(kKind, dim);
    const float* query = static_cast<const float*>(scan.queries) + static_cast<std::size_t>(q) * dim;
    const bool l2 = scan.metric == ZCGVS_METRIC_L2;
    float acc = 0.0f;
#pragma unroll 4
    for (int j = lane; j < dim; j += kWave) {
        const float x = loadScalar<kKind>(values, j, scan.scale);
        const float d = l2 ? l2Difference(query[j], x) : x;
        acc = fmaf(l2 ? d : query[j], d, acc);
    }
    const float total = groupSum<kWave>(acc);
    return l2 ? -total : total;
}

// The exact per-vector int8 score, (float)(integer dot) * (query scale * row scale).
template <int L>
__device__ __forceinline__ float exactScorePerVector(const ScanArgs& scan, std::uint32_t row, int q, int lane) {
    constexpr int kPer = 8;
    const int dim = scan.dim;
    const int chunks = dim / 16;
    const std::uint8_t* codes = static_cast<const std::uint8_t*>(scan.corpus) + static_cast<std::size_t>(row) * dim;
    const std::uint8_t* query = static_cast<const std::uint8_t*>(scan.queries) + static_cast<std::size_t>(q) * dim;
    const float scale = scan.row_scales[row];
    int group = lane % L;
    asm volatile("" : "+v"(group));
    v4u raw[kPer], qe[kPer];
#pragma unroll
    for (int t = 0; t < kPer; ++t) {
        if (t * L < chunks) {  // (uniform)
            const int at = min(group + t * L, chunks - 1) * 16;
            raw[t] = loadRowChunk<false>(codes + at);
            qe[t] = loadRowChunk<false>(query + at);
        }
    }
    int acc = 0;
#pragma unroll
    for (int t = 0; t < kPer; ++t) {
        if (group + t * L < chunks) {
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                acc = __builtin_amdgcn_sdot4(static_cast<int>(raw[t][w]), static_cast<int>(qe[t][w]), acc, false);
            }
        }
    }
    const float combined = scan.query_scales[q] * scale;
    return static_cast<float>(groupSum<L>(acc)) * combined;
}

template <int kKind>
__device__ __forceinline__ float exactScore(const ScanArgs& scan, std::uint32_t row, int q, int lane, int lanes) {
    if constexpr (kKind == kFilterPerVector) {
        return lanes == 8 ? exactScorePerVector<8>(scan, row, q, lane) : exactScorePerVector<32>(scan, row, q, lane);
    } else
    switch (lanes) {  // (uniform)
        case 8: return exactScoreLanes<kKind, 8>(scan, row, q, lane);
        case 16: return exactScoreLanes<kKind, 16>(scan, row, q, lane);
        case 32: return exactScoreLanes<kKind, 32>(scan, row, q, lane);
        default: return exactScoreStrided<kKind>(scan, row, q, lane);
    }
}

// A sketch phase (phase.sketch) scores one block of 16 rows per tile and keeps the best lower
// bound of each query per wavefront.
// With kLex, a hybrid search: the bounds go through the fusion with the lexical scores, which is
// monotone in the dense score, rounding included.
template <int kKind, int kPieces, int kBlocks, int kGroups, bool kLex>
__global__ __launch_bounds__(kFilterThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void filterScanKernel(ScanArgs scan, FilterArgs args, PhaseArgs phase, EmitArgs emit, int q_offset, int q_count,
                      int lanes_per_row) {
    constexpr int kSteps = FilterKind<kKind>::kSteps;
    constexpr int kQueries = kGroups * kFilterGroup;
    constexpr bool kF32 = kKind == ZCGVS_DTYPE_F32;
    constexpr bool kF16 = kKind == ZCGVS_DTYPE_F16;
    constexpr bool kInteger = FilterKind<kKind>::kInteger;
    constexpr int kDtype = FilterKind<kKind>::kDtype;
    typedef typename FilterSums<kInteger>::type Sums;

    __shared__ __attribute__((aligned(16))) std::uint8_t lds_operands[kFilterOperandBytes];
    __shared__ __attribute__((aligned(16))) float lds_slope[kQueries];  // threshold = slope * row term + base
    __shared__ __attribute__((aligned(16))) float lds_base[kQueries];
    __shared__ __attribute__((aligned(16))) float lds_gain[kQueries];   // sketch: bound = gain * acc + that
    __shared__ __attribute__((aligned(16))) float lds_floor[kLex ? kQueries : 4];    // hybrid: the threshold,
    __shared__ __attribute__((aligned(16))) float lds_inverse[kLex ? kQueries : 4];  // 1 / largest lexical score
    __shared__ std::uint64_t lds_tau[kQueries];
    __shared__ std::uint32_t lds_count[kQueries];
    __shared__ std::uint64_t lds_lowest[kQueries];  // the lowest of the first `width` keys appended
    __shared__ std::uint32_t lds_placed[kQueries];  // how many of those it covers
    __shared__ std::uint32_t lds_asked[2];  // a wavefront asks for a cut of the segments (in turns)
    __shared__ __attribute__((aligned(16))) std::uint8_t lds_stage[kFilterWaves][kFilterBlockRows * kPieceBytes / 2];
    __shared__ uint2 lds_park[kFilterWaves][kParkSlots];

    const bool sketch = phase.sketch != 0;
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int r16 = lane & 15;
    const int h = lane >> 4;
    const int dim = scan.dim;
    const int row_bytes = static_cast<int>(rowBytes(kDtype, dim));
    const int rounds = (row_bytes + kPieces * kPieceBytes - 1) / (kPieces * kPieceBytes);
    const int steps = args.steps;
    const bool l2 = scan.metric == ZCGVS_METRIC_L2;
    const std::uint8_t* corpus = static_cast<const std::uint8_t*>(scan.corpus);
    const std::uint32_t* list = args.list;
    const long long rows = list != nullptr ? static_cast<long long>(*args.list_count) : scan.doc_count;

    // ---- tiles ----
    const long long row_blocks = (rows + kFilterBlockRows - 1) / kFilterBlockRows;
    // (a short row list: smaller tiles, as filterTileLog2 makes them where the host knows the rows)
    const int tile_log2 = list != nullptr ? filterTileLog2(rows, kBlocks * kFilterBlockRows, gridDim.x * kFilterWaves, 0)
                                          : args.tile_log2;
    long long tiles = list != nullptr ? (rows + (1LL << tile_log2) - 1) >> tile_log2 : phase.items;
    long long stride = 1;  // sketch: one block of every `stride`
    if (sketch) {
        // (with a row list the host knows only an upper bound of the rows: the stride that visits
        // about as many blocks as planned)
        stride = list != nullptr ? max(1LL, (row_blocks + phase.items - 1) / phase.items) : phase.stride;
        tiles = (row_blocks + stride - 1) / stride;
    }
    const long long waves = static_cast<long long>(gridDim.x) * kFilterWaves;
    const long long first_tile = static_cast<long long>(wave) * gridDim.x + blockIdx.x;
    long long tile = first_tile;

    // Place of threshold tile t among the corpus's (the list's) tiles.
    auto tileAt = [&](long long t) __attribute__((always_inline)) -> long long {
        return list != nullptr ? t : phaseBlock(t, phase.stride, phase.skip);
    };
    // Entry (row number, kMaskedRow with it for a masked one) of place `local` of tile t.
    auto entryOf = [&](long long t, int local) __attribute__((always_inline)) -> std::uint32_t {
        const long long at = (sketch ? t * stride * kFilterBlockRows : tileAt(t) << tile_log2) + local;
        std::uint32_t entry = kNoRow;
        if (at < rows && local < (sketch ? kFilterBlockRows : 1 << tile_log2)) {
            entry = list != nullptr ? list[at] : static_cast<std::uint32_t>(at);
        }
        return entry;
    };
    // The rows this lane reads: places 16 b + 8 i + lane / 8 (no row: the corpus's first, whose
    // lines all such lanes share; never used for a result).
    auto readRows = [&](long long t, std::uint32_t (&row)[kBlocks][2]) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < kBlocks; ++b) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const std::uint32_t entry = t < tiles ? entryOf(t, kFilterBlockRows * b + 8 * i + (lane >> 3)) : kNoRow;
                row[b][i] = entry == kNoRow ? 0u : entry & ~kMaskedRow;
            }
        }
    };
    const int last_chunk = row_bytes - 16;
    // Rows of whole 128-byte lines are read with the non-temporal hint (256 -> 293 us without it at
    // 1M x 384 float32); others share lines between loads, and the hint fetches those twice (65 ->
    // 92 us with it at 400,000 x 300 float16).
    const bool whole_lines = row_bytes % 128 == 0;
    v4u ring[kPieces][kBlocks][2][2];
    // Refills half `half` of slot p with that of piece `piece`: chunk 8 half + lane % 8 of the rows.
    auto issue = [&](const std::uint32_t (&row)[kBlocks][2], int p, int piece, int half) __attribute__((always_inline)) {
        const int off = min(piece * kPieceBytes + 128 * half + 16 * (lane & 7), last_chunk);
        const std::uint8_t* at[kBlocks][2];
#pragma unroll
        for (int b = 0; b < kBlocks; ++b) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                at[b][i] = corpus + (static_cast<std::uint64_t>(row[b][i]) * static_cast<std::uint32_t>(row_bytes) +
                                     static_cast<std::uint32_t>(off));
                if (p == kPieces - 1 && piece * kPieceBytes + 128 * half >= row_bytes) {
                    at[b][i] = corpus;  // nothing of the row is there: one line for all (but as many loads in
                                        // flight, which the waits count)
                }
            }
        }
        if (whole_lines) {
#pragma unroll
            for (int b = 0; b < kBlocks; ++b) {
                ring[p][b][half][0] = loadRowChunk<true>(at[b][0]);
                ring[p][b][half][1] = loadRowChunk<true>(at[b][1]);
            }
        } else {
#pragma unroll
            for (int b = 0; b < kBlocks; ++b) {
                ring[p][b][half][0] = loadRowChunk<false>(at[b][0]);
                ring[p][b][half][1] = loadRowChunk<false>(at[b][1]);
            }
        }
    };
    auto issueTile = [&](const std::uint32_t (&row)[kBlocks][2]) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < kPieces; ++p) {
            issue(row, p, p, 0);
            issue(row, p, p, 1);
        }
    };

    // the first tile's rows are on their way while the operands are
    std::uint32_t row[kBlocks][2];
    readRows(tile, row);
    issueTile(row);

    // ---- the launch's operands: groups q_offset / 16 .. + kGroups ----
    {
        const v4u* src = reinterpret_cast<const v4u*>(args.operands) +
                         static_cast<std::size_t>(q_offset / kFilterGroup) * steps * kWave;
        v4u* dst = reinterpret_cast<v4u*>(lds_operands);
        const int words = kGroups * steps * kWave;
#pragma unroll 6
        for (int i = tid; i < words; i += kFilterThreads) {
            dst[i] = src[i];
        }
    }
    const float unit = kF32 ? *args.row_unit : kF16 || kInteger ? 1.0f : scan.scale;  // stored value = unit * operand
    const float inverse_unit = kF32 ? 1.0f / unit : 1.0f;                 // (float32: a power of two)
    const float relative = filterRelative(kKind, steps);
    // Absolute part, in operand units per |q|: float32 rows below float16's smallest normal lose up
    // to 2^-24 a component; products of float16 subnormals may be dropped from the norm.
    const float root_dim = sqrtf(static_cast<float>(dim));
    const float floor_abs = kF32 ? root_dim * 5.97e-8f : kF16 ? root_dim * 6.2e-5f * relative : 0.0f;
    const float norm_abs = unit * unit * static_cast<float>(dim) * 3.8e-9f;
    // The constants of query i and, in a threshold phase, its threshold `tau` (those are written again
    // when a cut raises it).
    auto setQuery = [&](int i, std::uint64_t tau) __attribute__((always_inline)) {
        const bool valid = i < q_count && (sketch || tau != kFilterNoKey);
        const FilterQuery query = args.queries[q_offset + i];
        const float qnorm = sqrtf(query.norm2) * 1.00001f;
        // (a score, and every partial sum of one, is bounded by the norms: where that is beyond float32,
        // an exact sum may overflow on its way to a value the approximation has in range)
        const float reach = kF32 ? 65504.0f * unit : 0.0f;  // of a row that is not unbounded
        const bool usable = query.usable != 0.0f && (l2 ? (qnorm + reach) * (qnorm + reach) : qnorm * reach) < 1e38f;
        bool gated = false;
        const float floor_score = keyFloor(tau, &gated);
        lds_tau[i] = tau;
        if constexpr (kInteger) {
            // score = acc * (query scale * row scale), compared with the threshold's itself
            lds_gain[i] = valid ? query.scale : __uint_as_float(0x7FC00000u);
            lds_slope[i] = query.scale;
            lds_base[i] = !valid ? INFINITY : gated && floor_score > kMaskedScore ? floor_score : -INFINITY;
        } else if (kLex || sketch) {
            // a bound of the score (hybrid: of its dense part; an upper one in a threshold phase) =
            // gain * acc + slope * row term + base
            const float side = sketch ? -1.0f : 1.0f;
            float gain = unit / query.scale;
            float slope = side * relative * qnorm * unit;
            float base = side * qnorm * unit * floor_abs;
            if (l2) {
                gain *= 2.0f;
                slope = -(1.0f - side * 2.0f * relative) * unit * unit;
                base = 2.0f * (base + side * norm_abs) - (1.0f - side * 2.0f * relative) * query.norm2;
            }
            // (NaN: no bound, which drops a sketch's row and keeps a threshold phase's)
            lds_gain[i] = (valid || !sketch) && usable ? gain : __uint_as_float(0x7FC00000u);
            lds_slope[i] = slope;
            lds_base[i] = base;
            if constexpr (kLex) {
                lds_floor[i] = !valid ? INFINITY : gated ? floor_score : -INFINITY;
                const float peak = valid ? scan.lexical_max[q_offset + i] : 0.0f;
                lds_inverse[i] = peak > 0.0f ? 1.0f / peak : 0.0f;
            }
        } else {
            // a pair survives unless acc < slope * row term + base
            const float to_acc = query.scale / unit;  // dot product -> accumulator
            float slope = -relative * qnorm * query.scale;
            float base = to_acc * floor_score - qnorm * query.scale * floor_abs;
            if (l2) {
                slope = 0.5f * (1.0f - 2.0f * relative) * unit * query.scale;
                base = to_acc * (0.5f * (floor_score + (1.0f - 2.0f * relative) * query.norm2) - qnorm * unit * floor_abs -
                                 norm_abs);
            }
            const bool filter = gated && usable && fabsf(base) < 3.0e38f && fabsf(slope) < 3.0e38f &&
                                floor_score > kMaskedScore;
            lds_slope[i] = valid && filter ? slope : 0.0f;
            // (a query past the batch takes no pair: nothing but NaN fails acc < inf, and those
            // pairs are dropped by its threshold key)
            lds_base[i] = !valid ? INFINITY : filter ? base : -INFINITY;
        }
    };
    for (int i = tid; i < kQueries; i += kFilterThreads) {
        lds_count[i] = 0u;
        lds_lowest[i] = ~0ull;
        lds_placed[i] = 0u;
        setQuery(i, i < q_count && !sketch ? emit.tau[q_offset + i] : kFilterNoKey);
    }
    if (tid < 2) {
        lds_asked[tid] = 0u;
    }
    __syncthreads();

    Sums acc[kBlocks][kGroups];
    float norm[kBlocks];
    int norm_codes[kBlocks];
    // Consumes slot p (piece `piece`) half by half and refills it with piece `next_piece` of the rows
    // `next_row`. A half goes through the wavefront's 2 KB of LDS, which turns the loads' layout (8
    // lanes per row, whole 128-byte lines) into the matrix core's (16 rows side by side); slot c ^
    // (row / 2 % 8) of a row's 128 bytes keeps both sides free of bank conflicts. One wavefront's LDS
    // operations run in order, so neither side waits for more than its data.
    std::uint8_t* stage = lds_stage[wave];
    const int write_at = (lane >> 3) * 128 + (((lane & 7) ^ ((lane >> 4) & 3)) * 16);
    auto multiplyPiece = [&](int p, int piece, const std::uint32_t (&next_row)[kBlocks][2],
                             int next_piece) __attribute__((always_inline)) {
        // (a piece past the end of a row of several rounds is cleared whole: any operands do)
        const v8h* operands = reinterpret_cast<const v8h*>(lds_operands) +
                              static_cast<std::size_t>(min(piece * kSteps, steps - kSteps)) * kWave + lane;
        const int group_stride = steps * kWave;
        auto product = [&](int step, const v8h (&x)[kBlocks]) __attribute__((always_inline)) {
#pragma unroll
            for (int g = 0; g < kGroups; ++g) {
                const v8h q = operands[g * group_stride + step * kWave];
#pragma unroll
                for (int b = 0; b < kBlocks; ++b) {
                    if constexpr (kInteger) {
                        acc[b][g] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(v4i, q),
                                                                          __builtin_bit_cast(v4i, x[b]), acc[b][g], 0, 0, 0);
                    } else {
                        acc[b][g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(q, x[b], acc[b][g], 0, 0, 0);
                    }
                }
            }
        };
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int half_at = piece * kPieceBytes + half * (kPieceBytes / 2);
            const bool clip = half_at + kPieceBytes / 2 > row_bytes;  // (uniform)
            if (p == kPieces - 1 && half_at >= row_bytes) {  // (a row's last slot may be half or wholly empty)
                issue(next_row, p, next_piece, half);
                continue;
            }
            v4u chunk[kBlocks][2];  // chunks 8 half + 4 i + h of this lane's row
#pragma unroll
            for (int b = 0; b < kBlocks; ++b) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    v4u raw = ring[p][b][half][i];
                    if (clip) {  // bytes that repeat earlier ones
                        raw = keepFrom(raw, min(16, max(0, half_at + 16 * (lane & 7) - last_chunk)));
                    }
                    // (row 8 i + lane / 8: its swizzle has the bit 8 i / 2 = 4 i on top of the lane's)
                    *reinterpret_cast<v4u*>(stage + i * 1024 + (write_at ^ (64 * i))) = raw;
                }
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    chunk[b][i] = *reinterpret_cast<const v4u*>(stage + r16 * 128 + (((4 * i + h) ^ (r16 >> 1)) * 16));
                }
            }
            issue(next_row, p, next_piece, half);
            if constexpr (kF32) {
                v8h x[kBlocks];
#pragma unroll
                for (int b = 0; b < kBlocks; ++b) {
                    v4u halves;
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        float f[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            f[e] = __uint_as_float(chunk[b][i][e]) * inverse_unit;
                            norm[b] = fmaf(f[e], f[e], norm[b]);
                        }
                        halves[2 * i] = __builtin_bit_cast(unsigned int, __builtin_amdgcn_cvt_pkrtz(f[0], f[1]));
                        halves[2 * i + 1] = __builtin_bit_cast(unsigned int, __builtin_amdgcn_cvt_pkrtz(f[2], f[3]));
                    }
                    x[b] = __builtin_bit_cast(v8h, halves);
                }
                product(half, x);
            } else if constexpr (kF16 || kInteger) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    v8h x[kBlocks];
#pragma unroll
                    for (int b = 0; b < kBlocks; ++b) {
                        x[b] = __builtin_bit_cast(v8h, chunk[b][i]);
#pragma unroll
                        for (int w = 0; w < (kInteger ? 0 : 4); ++w) {
                            const unsigned int word = chunk[b][i][w];  // (a value of its own: a bit cast of the
                            const v2h pair = __builtin_bit_cast(v2h, word);  // element yields element 0)
                            norm[b] = __builtin_amdgcn_fdot2(pair, pair, norm[b], false);
                        }
                    }
                    product(2 * half + i, x);
                }
            } else {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
#pragma unroll
                    for (int b = 0; b < kBlocks; ++b) {
#pragma unroll
                        for (int w = 0; w < 4; ++w) {
                            norm_codes[b] = __builtin_amdgcn_sdot4(static_cast<int>(chunk[b][i][w]), static_cast<int>(chunk[b][i][w]),
                                                                   norm_codes[b], false);
                        }
                    }
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        v8h x[kBlocks];
#pragma unroll
                        for (int b = 0; b < kBlocks; ++b) {
                            // code c as the half 1024 + (c + 128) (its byte under 0x64), less 1152
                            v4u halves;
#pragma unroll
                            for (int w = 0; w < 2; ++w) {
                                const unsigned int biased = chunk[b][i][2 * s + w] ^ 0x80808080u;
                                const v2h offset = {static_cast<_Float16>(-1152.0f), static_cast<_Float16>(-1152.0f)};
                                const v2h lo =
                                    __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, biased, 0x04010400u)) + offset;
                                const v2h hi =
                                    __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, biased, 0x04030402u)) + offset;
                                halves[2 * w] = __builtin_bit_cast(unsigned int, lo);
                                halves[2 * w + 1] = __builtin_bit_cast(unsigned int, hi);
                            }
                            x[b] = __builtin_bit_cast(v8h, halves);
                        }
                        product(4 * half + 2 * i + s, x);
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // ---- cuts ----
    // A workgroup's segment of a query holds more keys than are selected, and a full one is cut to its
    // `width` best, the last of which becomes the workgroup's threshold: no row whose key is lower can
    // be selected any more. So rows that tie, or come close, by the thousand do not overflow the segments,
    // after which the exact fallback would sweep the corpus at one compute unit's rate (1M rows, 30% of
    // them copies of the row that 4 queries seek: float16 x 768, 32 queries 41.9 ms, now 0.83; per-vector
    // int8, 16 queries 14.5, now 0.26; rows within 2% of 16 topics, float16 42.3, now 1.98).
    // A cut is made by all wavefronts together, each for queries of its own: one that finds a segment
    // full asks for it and waits; the others look once a tile (and between the exact scores) and, when
    // done with their rows, wait until all are.
    const std::uint32_t capacity = 1u << emit.seg_log2;
    const std::uint32_t width = static_cast<std::uint32_t>(args.width);
    const bool cuts = capacity > width;  // (not with the segments that a test makes too small)
    std::uint32_t turn = 0u;             // cuts made: the same in all wavefronts between two barriers
    auto askedForCut = [&]() __attribute__((always_inline)) -> std::uint32_t {
        return __hip_atomic_load(&lds_asked[turn & 1u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    auto segmentOf = [&](int q) __attribute__((always_inline)) -> std::uint64_t* {
        return emit.seg + ((static_cast<std::size_t>(blockIdx.x) * scan.batch + q_offset + q) << emit.seg_log2);
    };
    // Query q's full segment, by one wavefront, which holds its keys in registers and finds the width-th
    // best of them bit by bit.
    auto cutSegment = [&](int q) __attribute__((always_inline)) {
        std::uint64_t* seg = segmentOf(q);
        std::uint64_t key[kFilterSegmentKeys / kWave];
#pragma unroll
        for (int r = 0; r < kFilterSegmentKeys / kWave; ++r) {
            // (past the compute unit's cache: the other wavefronts' stores have reached the next one)
            key[r] = static_cast<std::uint32_t>(r * kWave) < capacity
                         ? __hip_atomic_load(seg + r * kWave + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                         : 0ull;
        }
        std::uint64_t cut = 0ull;
#pragma unroll 1
        for (int bit = 63; bit >= 0; --bit) {
            const std::uint64_t candidate = cut | 1ull << bit;
            std::uint32_t above = 0u;
#pragma unroll
            for (int r = 0; r < kFilterSegmentKeys / kWave; ++r) {
                if (static_cast<std::uint32_t>(r * kWave) < capacity) {  // (uniform)
                    above += static_cast<std::uint32_t>(__popcll(__ballot(key[r] >= candidate)));
                }
            }
            cut = above >= width ? candidate : cut;
        }
        std::uint32_t kept = 0u;
#pragma unroll
        for (int r = 0; r < kFilterSegmentKeys / kWave; ++r) {
            if (static_cast<std::uint32_t>(r * kWave) < capacity) {
                const unsigned long long take = __ballot(key[r] >= cut);
                const std::uint32_t below = __builtin_amdgcn_mbcnt_hi(
                    static_cast<std::uint32_t>(take >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<std::uint32_t>(take), 0u));
                if (key[r] >= cut) {
                    seg[kept + below] = key[r];
                }
                kept += static_cast<std::uint32_t>(__popcll(take));
            }
        }
        if (lane == 0) {
            lds_count[q] = width;
            setQuery(q, cut);
        }
    };
    // By every wavefront: waits for all of them and, if one asked, cuts the full segments. False: none
    // asked, so all are done with their rows.
    auto waitForCut = [&](bool ask) __attribute__((always_inline)) -> bool {
        if (ask) {
            __hip_atomic_store(&lds_asked[turn & 1u], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        __syncthreads();
        if (__builtin_amdgcn_readfirstlane(askedForCut()) == 0u) {
            return false;  // (without a wait for the rows read past the last tile: 1 us of every launch)
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's keys have left the compute unit
        __syncthreads();
#pragma unroll 1
        for (int q = wave; q < q_count; q += kFilterWaves) {
            if (__builtin_amdgcn_readfirstlane(lds_count[q]) >= capacity) {
                cutSegment(q);
            }
        }
        // (nobody reads the other turn's word between the barriers before and after)
        if (tid == 0) {
            __hip_atomic_store(&lds_asked[(turn + 1u) & 1u], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        ++turn;
        __syncthreads();
        return true;
    };

    // ---- exact scores, a row per group of lanes_per_row lanes ----
    // The key of a pair (row as listed, query of the launch), on every lane of the group.
    auto keyOfPair = [&](std::uint32_t listed, int q) __attribute__((always_inline)) -> std::uint64_t {
        const std::uint32_t row = listed & ~kMaskedRow;
        const int query = min(q_offset + q, scan.batch - 1);  // (a query past the batch parks NaN pairs only)
        float score = exactScore<kKind>(scan, row, query, lane, lanes_per_row);
        if constexpr (kLex) {
            score = fuseHybrid(score, scan.lexical[static_cast<std::size_t>(query) * scan.doc_count + row], scan.dense_weight,
                               lds_inverse[q]);
        }
        if (args.infinite_as_nan != 0 && scan.batch - query / 128 * 128 >= 32 && fabsf(score) == INFINITY) {
            score = __uint_as_float(0x7FC00000u);
        }
        return makeKey((listed & kMaskedRow) != 0u ? kMaskedScore : score, row);
    };
    const int per_round = kWave / lanes_per_row;

    float best[kGroups * 4];  // sketch
#pragma unroll
    for (int i = 0; i < kGroups * 4; ++i) {
        best[i] = -INFINITY;
    }
    std::uint32_t parked = 0u;  // pairs that wait for their exact score (uniform)
    // The stream runs until its surviving pairs fill the wavefront's park, which is then scored with
    // the stream's registers free; a tile whose pairs do not fit (or would not even an empty park) is
    // streamed again (scored whole) after it.
    bool crowded = false;
    while (true) {
        while (tile < tiles) {
            const long long next = tile + waves;
            std::uint32_t id[kBlocks];  // this lane's rows in the results
            float row_scale[kBlocks];
            v4f lexical[kLex ? kBlocks : 1][kLex ? kGroups : 1];
            std::uint32_t next_row[kBlocks][2];
            readRows(next, next_row);
#pragma unroll
            for (int b = 0; b < kBlocks; ++b) {
                id[b] = entryOf(tile, kFilterBlockRows * b + r16);
                if constexpr (kLex) {
                    // (a row or query that does not exist re-reads the first row's, the last query's)
                    const std::size_t at = id[b] == kNoRow ? 0u : id[b];
#pragma unroll
                    for (int g = 0; g < kGroups; ++g) {
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int q = min(q_offset + kFilterGroup * g + 4 * h + i, scan.batch - 1);
                            lexical[b][g][i] = scan.lexical[static_cast<std::size_t>(q) * scan.doc_count + at];
                        }
                    }
                }
                row_scale[b] = kInteger ? scan.row_scales[id[b] == kNoRow ? 0u : id[b] & ~kMaskedRow] : 0.0f;
                norm[b] = 0.0f;
                norm_codes[b] = 0;
#pragma unroll
                for (int g = 0; g < kGroups; ++g) {
                    acc[b][g] = Sums{0, 0, 0, 0};
                }
            }
            for (int round = 0; round < rounds; ++round) {
                const bool last = round + 1 == rounds;
                std::uint32_t refill_row[kBlocks][2];
#pragma unroll
                for (int b = 0; b < kBlocks; ++b) {
                    refill_row[b][0] = last ? next_row[b][0] : row[b][0];
                    refill_row[b][1] = last ? next_row[b][1] : row[b][1];
                }
                const int refill_piece = last ? 0 : (round + 1) * kPieces;
#pragma unroll
                for (int p = 0; p < kPieces; ++p) {
                    multiplyPiece(p, round * kPieces + p, refill_row, refill_piece + p);
                }
            }

            // ---- the tile's scores (the thresholds are read again for every tile: kept, they would
            //      take the accumulators' registers) ----
            asm volatile("" ::: "memory");
            const std::uint32_t asked = askedForCut();
            float term[kBlocks];
            bool live[kBlocks], masked[kBlocks];
#pragma unroll
            for (int b = 0; b < kBlocks; ++b) {
                if constexpr (kInteger) {
                    term[b] = row_scale[b];
                } else {
                    float n2 = kF32 || kF16 ? norm[b] : static_cast<float>(norm_codes[b]);
                    n2 += waveXor(n2, 16);
                    n2 += waveXor(n2, 32);
                    term[b] = l2 ? n2 : sqrtf(n2) * 1.00001f;
                    if constexpr (kF32) {
                        // an unbounded row: every bound is NaN, which no sketch takes and every
                        // threshold lets through
                        term[b] = n2 < kOperandNorm2 ? term[b] : __uint_as_float(0x7FC00000u);
                    }
                }
                live[b] = id[b] != kNoRow;
                masked[b] = list != nullptr && (id[b] & kMaskedRow) != 0u;
            }
            // Whether the pair of block b's row and query 16 g + 4 h + i can reach the query's threshold.
            // (A masked row does where every row does; a NaN survives.) `tie`: its score is no better than
            // the threshold's, so that the row numbers decide.
            auto survives = [&](int b, int g, int i, const v4f& slope, const v4f& offset,
                                bool& tie) __attribute__((always_inline)) -> bool {
                if constexpr (kLex) {
                    const int q = kFilterGroup * g + 4 * h + i;
                    const float bound = fmaf(lds_gain[q], acc[b][g][i], fmaf(slope[i], term[b], offset[i]));
                    const float fused = fuseHybrid(bound, lexical[b][g][i], scan.dense_weight, lds_inverse[q]);
                    tie = fused == lds_floor[q] && fused > -INFINITY;
                    return !(fused < lds_floor[q]);
                } else if constexpr (kInteger) {
                    const float score = static_cast<float>(acc[b][g][i]) * (slope[i] * term[b]);
                    tie = !masked[b] && score == offset[i] && score > -INFINITY;
                    return masked[b] ? offset[i] == -INFINITY : !(score < offset[i]);
                } else {
                    const float sum = masked[b] ? -INFINITY : acc[b][g][i];
                    const float edge = fmaf(slope[i], masked[b] ? 0.0f : term[b], offset[i]);
                    tie = false;
                    return !(sum < edge);
                }
            };
            if (sketch) {
#pragma unroll
                for (int g = 0; g < kGroups; ++g) {
                    const v4f gain = *reinterpret_cast<const v4f*>(&lds_gain[kFilterGroup * g + 4 * h]);
                    const v4f slope = *reinterpret_cast<const v4f*>(&lds_slope[kFilterGroup * g + 4 * h]);
                    const v4f offset = *reinterpret_cast<const v4f*>(&lds_base[kFilterGroup * g + 4 * h]);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        float bound;
                        if constexpr (kInteger) {
                            bound = static_cast<float>(acc[0][g][i]) * (gain[i] * term[0]);
                        } else {
                            bound = fmaf(gain[i], acc[0][g][i], fmaf(slope[i], term[0], offset[i]));
                        }
                        if constexpr (kLex) {
                            bound = fuseHybrid(bound, lexical[0][g][i], scan.dense_weight,
                                               lds_inverse[kFilterGroup * g + 4 * h + i]);
                        }
                        // (an infinite or NaN bound is none)
                        best[4 * g + i] = live[0] && !masked[0] && bound < 3.0e38f ? fmaxf(best[4 * g + i], bound) : best[4 * g + i];
                    }
                }
            } else {
                bool any = false;
#pragma unroll
                for (int g = 0; g < kGroups; ++g) {
                    const v4f slope = *reinterpret_cast<const v4f*>(&lds_slope[kFilterGroup * g + 4 * h]);
                    const v4f offset = *reinterpret_cast<const v4f*>(&lds_base[kFilterGroup * g + 4 * h]);
#pragma unroll
                    for (int b = 0; b < kBlocks; ++b) {
                        bool here = false;
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            bool tie;
                            here |= survives(b, g, i, slope, offset, tie);
                        }
                        any |= here && live[b];
                    }
                }
                if (__any(any)) {
                    // bit 4 b + i of survivors[g]: block b's row and query 16 g + 4 h + i (the opaque copies
                    // keep the thresholds above from being kept for here)
#pragma unroll
                    for (int b = 0; b < kBlocks; ++b) {
                        asm volatile("" : "+v"(term[b]));
                    }
                    std::uint32_t survivors[kGroups];
#pragma unroll
                    for (int g = 0; g < kGroups; ++g) {
                        const v4f slope = *reinterpret_cast<const v4f*>(&lds_slope[kFilterGroup * g + 4 * h]);
                        const v4f offset = *reinterpret_cast<const v4f*>(&lds_base[kFilterGroup * g + 4 * h]);
                        survivors[g] = 0u;
                        std::uint32_t ties = 0u;
#pragma unroll
                        for (int b = 0; b < kBlocks; ++b) {
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                bool tie;
                                if (live[b] && survives(b, g, i, slope, offset, tie)) {
                                    survivors[g] |= 1u << (4 * b + i);
                                    ties |= tie ? 1u << (4 * b + i) : 0u;
                                }
                            }
                        }
                        while ((kLex || kInteger) && __any(ties != 0u)) {
                            if (ties != 0u) {
                                const int bit = __ffs(ties) - 1;
                                ties &= ties - 1u;
                                std::uint32_t tied = id[0];
#pragma unroll
                                for (int b = 1; b < kBlocks; ++b) {
                                    tied = (bit >> 2) == b ? id[b] : tied;
                                }
                                const std::uint64_t tau = lds_tau[kFilterGroup * g + 4 * h + (bit & 3)];
                                if (makeKey(keyScore(tau), tied) <= tau) {
                                    survivors[g] &= ~(1u << bit);
                                }
                            }
                        }
                    }
                    int own = 0;
#pragma unroll
                    for (int g = 0; g < kGroups; ++g) {
                        own += __popc(survivors[g]);
                    }
                    const std::uint32_t found = __builtin_amdgcn_readlane(waveInclusiveSum(static_cast<std::uint32_t>(own)), kWave - 1);
                    if (parked + found > static_cast<std::uint32_t>(kParkSlots)) {
                        crowded = found > static_cast<std::uint32_t>(kParkSlots);
                        break;
                    }
#pragma unroll 1
                    for (int g = 0; g < kGroups; ++g) {
                        std::uint32_t word = survivors[0];
#pragma unroll
                        for (int other = 1; other < kGroups; ++other) {
                            word = g == other ? survivors[other] : word;  // (registers have no index)
                        }
                        while (__any(word != 0u)) {
                            const bool mine = word != 0u;
                            const unsigned long long who = __ballot(mine);
                            if (mine) {
                                const int bit = __ffs(word) - 1;
                                word &= word - 1u;
                                std::uint32_t row = id[0];
#pragma unroll
                                for (int b = 1; b < kBlocks; ++b) {
                                    row = (bit >> 2) == b ? id[b] : row;
                                }
                                const std::uint32_t below = __builtin_amdgcn_mbcnt_hi(
                                    static_cast<std::uint32_t>(who >> 32),
                                    __builtin_amdgcn_mbcnt_lo(static_cast<std::uint32_t>(who), 0u));
                                lds_park[wave][parked + below] =
                                    make_uint2(row, static_cast<std::uint32_t>(kFilterGroup * g + 4 * h + (bit & 3)));
                            }
                            parked += static_cast<std::uint32_t>(__popcll(who));
                        }
                    }
                }
            }
            tile = next;
#pragma unroll
            for (int b = 0; b < kBlocks; ++b) {
                row[b][0] = next_row[b][0];
                row[b][1] = next_row[b][1];
            }
            if (__builtin_amdgcn_readfirstlane(asked) != 0u) {
                break;
            }
        }
        if (sketch) {
            break;  // (no keys)
        }
        // The exact scores of the parked pairs and, of a crowded tile, of every pair (its rows from the list
        // or the tile's place). A key that finds its segment full waits for a cut.
        const std::uint32_t total = parked + (crowded ? static_cast<std::uint32_t>(q_count) << tile_log2 : 0u);
        const long long tile_row = tileAt(tile) << tile_log2;  // (not used past the last tile)
        tile += crowded ? waves : 0;
        const bool done = tile >= tiles;
        std::uint32_t first = 0u;
        std::uint64_t key = 0ull;
        int q = 0;
        bool waits = false;
        bool over = false;
#pragma unroll 1
        while (true) {
            if (first < total && !__any(waits)) {
                const std::uint32_t e = first + static_cast<std::uint32_t>(lane / lanes_per_row);
                const uint2 pair = lds_park[wave][min(e, max(parked, 1u) - 1u)];  // (the last one's again past them)
                std::uint32_t listed = pair.x;
                q = static_cast<int>(pair.y);
                waits = e < total;
                if (crowded && e >= parked) {
                    const std::uint32_t at = min(e, total - 1u) - parked;
                    const long long place = tile_row + (at & ((1u << tile_log2) - 1u));
                    waits = waits && place < rows;
                    listed = static_cast<std::uint32_t>(min(place, rows - 1));
                    listed = list != nullptr ? list[listed] : listed;
                    q = static_cast<int>(at >> tile_log2);
                }
                key = keyOfPair(listed, q);
                waits = waits && lane % lanes_per_row == 0;
                first += static_cast<std::uint32_t>(per_round);
            }
            waits = waits && key > lds_tau[q];
            if (waits) {
                const std::uint32_t slot = atomicAdd(&lds_count[q], 1u);
                if (slot < capacity) {
                    segmentOf(q)[slot] = key;
                }
                // The workgroup's first `width` keys of a query are a threshold as a cut's are: the last of
                // them to be covered raises it, which spares the merge keys.
                if (slot < width) {
                    atomicMin(&lds_lowest[q], key);
                    if (atomicAdd(&lds_placed[q], 1u) + 1u == width) {
                        lds_tau[q] = max(lds_tau[q], lds_lowest[q]);
                    }
                }
                waits = slot >= capacity && cuts;
            }
            const bool ask = __any(waits);
            if (!ask && first < total) {
                continue;
            }
            if (!ask && !done && __builtin_amdgcn_readfirstlane(askedForCut()) == 0u) {
                break;
            }
            // (a cut leaves room for capacity - width keys, or a threshold above the ones that wait)
            if (!waitForCut(ask)) {
                over = true;
                break;
            }
        }
        parked = 0u;
        crowded = false;
        if (over) {
            break;
        }
        readRows(tile, row);  // (past the last tile too: with a branch the ring would be kept across all this)
        issueTile(row);
    }
    if (sketch) {
        // One slot per wavefront, the best over its 16 row lanes; with fewer blocks than half the slots, as
        // many slots per block (2, 4, 8 or 16, its rows dealt out to them) as there are.
        int split = 0;
        while (split < 4 && tiles << (split + 1) <= waves) {
            ++split;
        }
        // (the usual single slot first: its shuffles, of all queries side by side, end every sketch)
        auto storeBest = [&](int lanes, std::size_t slot, bool owns) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < kGroups * 4; ++i) {
                float v = best[i];
#pragma unroll
                for (int x = 1; x < kFilterBlockRows; x <<= 1) {
                    const float other = waveXor(v, x);
                    v = x < lanes ? fmaxf(v, other) : v;
                }
                const int q = kFilterGroup * (i / 4) + 4 * h + (i & 3);
                if (owns && q < q_count) {
                    emit.sketch[slot * scan.batch + q_offset + q] = v;
                }
            }
        };
        if (split == 0) {
            storeBest(kFilterBlockRows, static_cast<std::size_t>(first_tile), r16 == 0);
        } else {
            const int lanes = kFilterBlockRows >> split;
            const bool has_block = first_tile < tiles;
            storeBest(lanes, static_cast<std::size_t>(has_block ? (first_tile << split) + r16 / lanes : first_tile),
                      has_block ? r16 % lanes == 0 : r16 == 0 && first_tile >= tiles << split);
        }
    } else {
        for (int i = tid; i < q_count; i += kFilterThreads) {
            emit.seg_count[static_cast<std::size_t>(blockIdx.x) * scan.batch + q_offset + i] = lds_count[i];
        }
    }
}

template <int kKind, int kPieces>
int launchFilterPieces(const ScanArgs& scan, const FilterArgs& args, const PhaseArgs& phase, const EmitArgs& emit,
                       int workgroups, hipStream_t stream) {
    constexpr int kDtype = FilterKind<kKind>::kDtype;
    const int chunks = static_cast<int>((rowBytes(kDtype, scan.dim) + 15) / 16);
    // The lane groups of the VALU scan (a row of fewer chunks leaves lanes of its 8 at zero, which
    // changes no sum), or a wavefront per row.
    const int lanes = rowBytes(kDtype, scan.dim) % 16 != 0 ? kWave
                      : lanesPerRow(chunks, 8, 8) < 8     ? 8
                                                          : lanesPerRow(chunks, 8, 8);
    const dim3 grid(static_cast<unsigned>(workgroups));
    const int per_launch = args.groups_per_launch * kFilterGroup;
    for (int q0 = 0; q0 < scan.batch; q0 += per_launch) {
        const int count = scan.batch - q0 < per_launch ? scan.batch - q0 : per_launch;
        if constexpr (kKind == ZCGVS_DTYPE_F32 || kKind == ZCGVS_DTYPE_F16) {
            if (scan.lexical != nullptr) {
                if (args.groups_per_launch == 1) {
                    filterScanKernel<kKind, kPieces, filterBlocks(kPieces, 1, true), 1, true>
                    <<<grid, kFilterThreads, 0, stream>>>(scan, args, phase, emit, q0, count, lanes);
                } else {
                    filterScanKernel<kKind, kPieces, filterBlocks(kPieces, 2, true), 2, true>
                    <<<grid, kFilterThreads, 0, stream>>>(scan, args, phase, emit, q0, count, lanes);
                }
                ZCGVS_LAUNCH_CHECK("filter scan");
                continue;
            }
        }
        switch (args.groups_per_launch) {
            case 1:
                filterScanKernel<kKind, kPieces, filterBlocks(kPieces, 1), 1, false>
                    <<<grid, kFilterThreads, 0, stream>>>(scan, args, phase, emit, q0, count, lanes);
                break;
            case 2:
                filterScanKernel<kKind, kPieces, filterBlocks(kPieces, 2), 2, false>
                    <<<grid, kFilterThreads, 0, stream>>>(scan, args, phase, emit, q0, count, lanes);
                break;
            case 4:
                filterScanKernel<kKind, kPieces, filterBlocks(kPieces, 4), 4, false>
                    <<<grid, kFilterThreads, 0, stream>>>(scan, args, phase, emit, q0, count, lanes);
                break;
            default:
                filterScanKernel<kKind, kPieces, filterBlocks(kPieces, 8), 8, false>
                    <<<grid, kFilterThreads, 0, stream>>>(scan, args, phase, emit, q0, count, lanes);
                break;
        }
        ZCGVS_LAUNCH_CHECK("filter scan");
    }
    return ZCGVS_OK;
}

}  // namespace

// The filter scan of rows of one or two pieces (kWide clear) or more; filterSlots(pieces) of them
// are in flight.
template <int kKind, bool kWide>
int launchFilterKind(const ScanArgs& scan, const FilterArgs& args, const PhaseArgs& phase, const EmitArgs& emit,
                     int workgroups, hipStream_t stream) {
    const int slots = filterSlots(static_cast<int>((rowBytes(FilterKind<kKind>::kDtype, scan.dim) + kPieceBytes - 1) / kPieceBytes));
    if constexpr (kWide) {
        return slots == 3 ? launchFilterPieces<kKind, 3>(scan, args, phase, emit, workgroups, stream)
                          : launchFilterPieces<kKind, 4>(scan, args, phase, emit, workgroups, stream);
    } else {
        return slots == 1 ? launchFilterPieces<kKind, 1>(scan, args, phase, emit, workgroups, stream)
                          : launchFilterPieces<kKind, 2>(scan, args, phase, emit, workgroups, stream);
    }
}

}  // namespace zcgvs_hip
