// The test side of fake_hip.cpp.
#pragma once
#include <hip/hip_runtime_api.h>

#include <string>
#include <vector>

namespace fake {
extern std::vector<std::string> launched;   // kernels in launch order ("graph": a captured graph, "set": an asynchronous memset)
extern std::string fail_next;               // the next launch of a kernel with this in its name fails
extern void (*on_graph_launch)();
extern void (*on_copy)(void* dst, const void* src, size_t bytes, int kind);   // after the copy
}
