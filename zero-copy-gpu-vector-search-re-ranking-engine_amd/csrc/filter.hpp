// Filter scan (filter_scan.hip): float32, float16 and matrix-scale int8 corpora of any row width,
// cosine, dot or L2, with or without an allow-mask, against a batch of float32 queries; and
// per-vector int8 corpora against int8 queries.
//
// Each (row, query) pair first gets an approximate score from the matrix cores, rounded to
// float16 operands, with a bound on its distance from the exact score; only pairs whose
// approximation plus bound reaches the query's threshold are scored exactly, as the VALU scan
// scores them (scan_core.hpp), and only exact scores become keys. So the results are those of the VALU
// scan bit for bit, and the approximation decides nothing but how many pairs are scored twice. Where that
// is most of them (rows closer to each other than the bound, about 0.15% of |q| |x| for float32 and 0.05%
// for the others; a query that is NaN) it costs: 1M rows within 2% of 16 topics, float32 x 384, 64 queries 0.34 ->
// 1.4 ms (the split scan 0.45), float16 x 768, 32 queries 0.34 -> 2.0 (the VALU scan 5.5).
#pragma once

#include "common.hpp"
#include "fused.hpp"

namespace zcgvs_hip {

constexpr int kFilterPerVector = 4;  // scan kind beside the zcgvs_dtype ones: per-vector int8
inline int filterKind(const ScanArgs& scan) {
    return scan.dtype == ZCGVS_DTYPE_I8 && scan.row_scales != nullptr ? kFilterPerVector : scan.dtype;
}

// Queries are prepared per 16 (a query group): float16 matrix-core operands and FilterQuery
// constants. Rows are read in 256-byte pieces, kFilterSteps(kind) 32-dimension products each.
constexpr int kFilterGroup = 16;
constexpr int kFilterMaxGroups = 8;                  // query groups per launch
constexpr int kFilterWaves = 8;                      // wavefronts per workgroup
constexpr std::size_t kFilterOperandBytes = 128 * 1024;  // LDS of a launch's query operands
constexpr int kFilterSketchSlots = kFilterWaves;     // sketch slots per workgroup
constexpr int kFilterBlockRows = 16;                 // rows of a sketch phase's work item
constexpr int kFilterSegmentKeys = 1024;             // most keys of a candidate segment

// 256-byte pieces of a row kept in flight: whole rows of up to 4 pieces, wider ones in rounds of 3
// or 4.
constexpr int filterSlots(int pieces) {
    return pieces <= 4 ? pieces : pieces == 5 || pieces == 6 || pieces == 9 ? 3 : 4;
}

// 16-row blocks of a wavefront's tile, which make it 8 to 16 KB in flight. (Fewer where the sums, or
// a hybrid search's lexical scores, would take the registers.)
constexpr int filterBlocks(int slots, int groups, bool lexical = false) {
    const bool few = groups <= 2 && !lexical;
    return slots == 1 ? (few ? 4 : 2) : slots == 2 && few ? 2 : 1;
}

struct FilterQuery {
    float scale;  // the power of two the operands were multiplied by; per-vector int8: the query's scale
    float norm2;  // sum q_j^2
    float usable; // 0: not finite or out of range, every pair is scored exactly
    // 1: all zero, under a metric by which every finite row then scores 0, so that the row numbers decide
    // (a batch padded to its size, say). The scan takes no pair of such a query (unless a mask lets few
    // rows through); the last merge, which
    // finds too few keys, sweeps the rows from the first on until enough score 0 (recover.hip). In the
    // scan every row would reach its threshold: 1M x 384 float32, 64 queries, 32 of them zero 14.0 ms,
    // now 0.34; with one 25.9, now 0.35.
    float zero;
};
// Threshold of a query that the scan leaves out.
constexpr std::uint64_t kFilterNoKey = ~0ull;

struct FilterArgs {
    std::uint8_t* operands = nullptr;  // [groups][steps][64 lanes][16 bytes]
    FilterQuery* queries = nullptr;    // [groups * 16]
    float* row_unit = nullptr;         // one float: stored value = unit * operand value (float32 rows)
    std::uint32_t* list = nullptr;     // allow-mask: row numbers to scan (bit 31: a masked row), or null
    std::uint32_t* list_count = nullptr;
    int steps = 0;                     // 32-dimension steps of a row, whole pieces
    int groups = 0;                    // query groups prepared (launches * groups per launch)
    int groups_per_launch = 0;
    int width = 0;                     // keys selected per query
    int tile_log2 = 0;                 // log2 of FilterShape::tile_rows
    // Launches of 32 to 128 queries over float32 rows of 256 or 384 components take NaN for an
    // infinite score, as the split scan (fused_mfma_split.hip) does.
    int infinite_as_nan = 0;
};

// How a search of this shape runs, or supported = false.
struct FilterShape {
    bool supported = false;
    int steps = 0;
    int groups = 0;
    int groups_per_launch = 0;
    int tile_rows = 0;  // rows of a threshold phase's work item
};
// log2 of the rows of a wavefront's tile: `most` (the kernel's blocks), or with fewer rows than those
// fill of `waves` wavefronts the smallest number, from 2^least on, that covers them, so that the pairs to
// score exactly are shared by all. (A tile of less than 16 rows costs what 16 do: it pays where many of its
// pairs are scored, as of the few rows that a mask may let through. 4,674 x 509 float32, 94 queries, k = 1 in
// tiles of 16 rows 65 us, of 4 rows 70; 3,000 x 922, 100 queries, k = 50 269 and, of 2 rows, 137.)
__host__ __device__ inline int filterTileLog2(long long rows, int most, int waves, int least) {
    int log2 = least;
    while (1 << log2 < most && static_cast<long long>(waves) << log2 < rows) {
        ++log2;
    }
    return log2;
}
FilterShape filterShape(const ScanArgs& scan, int width);
inline std::size_t filterOperandBytes(const FilterShape& shape) {
    return static_cast<std::size_t>(shape.groups) * shape.steps * 1024;
}
// Entries of the row list: every row, and room for a whole tile.
inline std::size_t filterListEntries(long long rows) { return static_cast<std::size_t>(rows) + 64; }

// A search with fewer allowed rows than it selects also returns masked rows, the lowest ones. All of
// those lie among the first 2 * width rows (fewer than width of them are allowed), whose masked ones
// the row list holds too. (Masked rows past these can be selected only in the place of allowed rows
// that score -inf or NaN, which the last merge sees to: MergeInputs::masked_from.)
inline long long filterMaskedRows(long long rows, int width) { return rows < 2LL * width ? rows : 2LL * width; }

// The query operands, the row unit and, with a mask, the row list.
int launchFilterPrepare(const ScanArgs& scan, const FilterArgs& args, hipStream_t stream);
// After a sketch phase: tau[q] (and tau_safe[q]), a key below the width-th best of query q's rows.
int launchFilterThreshold(const FilterArgs& args, long long rows, const float* sketch, int slots, int batch,
                          std::uint64_t* tau, std::uint64_t* tau_safe, std::uint32_t* flag_count, hipStream_t stream);
// A sketch phase (emit.sketch: the best certain lower bound of every slot's rows; items of 16 rows)
// or a threshold phase (items of tile_rows rows; over every listed row when there is a row list).
int launchFilterScan(const ScanArgs& scan, const FilterArgs& args, const PhaseArgs& phase, const EmitArgs& emit,
                     int workgroups, hipStream_t stream);

}  // namespace zcgvs_hip
