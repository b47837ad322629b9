// Knobs and counters of the stand-in of the HIP runtime (runtime_stand_in.cpp).
#pragma once

#include <cstddef>
#include <functional>
#include <map>
#include <string>
#include <vector>

namespace stand_in {
extern size_t limit;             // bytes of device memory
extern size_t live, peak;        // allocated bytes now and at most
extern long syncs;               // hipStreamSynchronize calls
extern std::string fail_launch;  // the next launch of a kernel whose name contains it fails, once
extern void* capturing;          // a stream that is being captured
extern std::map<std::string, long> launches;
// called at each launch that is to succeed or fail: the kernel's name, its grid's y and its arguments
extern std::function<void(const std::string&, unsigned, void**)> on_launch;
long launched(const std::string& part);  // launches of the kernels whose names contain part
std::vector<std::string> kernels(const std::string& part);  // the library's kernels whose names contain part
}  // namespace stand_in
