// host_hip.h -- what the checks read and set of the stand-in in host_hip.cpp.
#pragma once
#include <atomic>
#include <cstddef>

namespace host_hip {
extern std::atomic<long> pinned_bytes;      // pinned host memory held
extern std::atomic<int> branches;           // most parallel branches of a capture so far
extern std::atomic<int> captures;           // captures begun
extern std::atomic<int> step_us;            // time of a launch or copy
extern std::atomic<size_t> device_bytes;    // device memory reported as free

// What the stand-in's winner kernel writes to a mode's map for a pixel whose
// views sum to v (view i with weight i + 1); the integer and sub-pixel maps
// take v itself.
inline int map_value(int v, int mode) { return 7 * v + 1000 * mode; }
}  // namespace host_hip
