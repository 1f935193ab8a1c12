// The recorded first levels of the fused coarse cycle (solver2d.cpp).
#pragma once

#include <array>
#include <string>

namespace cedar {
namespace hip {

// First level of the fused coarse cycle by device, word size, smoothing, extents, levels, batch and
// right-hand sides per operator: the recorded one (record < 0; -1 if none), or records `record`.  One
// table per process, guarded by a mutex, emptied when it holds 1024 entries and by
// fused_start_clear.  fused_start_report: its entries as JSON objects, comma-separated.
using fused_start_key = std::array<int, 10>;
int fused_start(const fused_start_key &key, int record);
void fused_start_clear();
std::string fused_start_report();

}  // namespace hip
}  // namespace cedar
