// Work split of the twiddle-table kernels and the points it needs (host logic).
// A thread makes a run of consecutive words and reaches the first of them by
// one point product for each bit of the run's number: a workgroup's eight bits
// always, the bits above them while any is set.
#pragma once
#include <stdint.h>

namespace vx {

constexpr uint32_t TABLE_THREADS_LOG = 8;
constexpr uint32_t TABLE_THREADS = 1u << TABLE_THREADS_LOG;
constexpr uint32_t TABLE_RUN_LOG = 4;   // with inverses, and in the NTT tables
constexpr uint32_t SOURCE_RUN_LOG = 2;  // sources alone: a shorter chain
constexpr uint32_t NTT_LOG_MAX = 31;    // the whole circle group

// Line layer l of a transform takes step^(2^(2l+1)) for bit 0 of a word's index
// (the circle layer step^1), so its threads read squares 2l + 1 and on, a whole
// workgroup's bits of them however short the layer is.
constexpr uint32_t line_layer_shift(uint32_t l) { return 2 * l + 1; }
constexpr uint32_t NTT_TABLE_SQUARES = line_layer_shift(NTT_LOG_MAX - 2) + TABLE_RUN_LOG + TABLE_THREADS_LOG;

}  // namespace vx
