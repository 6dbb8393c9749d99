// hip_stub.hpp - what a program linked against hip_stub.cpp sees of the HIP
// host calls it stands in for: device memory is malloc, a kernel launch runs
// nothing and is handed to stub::on_launch.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <functional>
#include <map>
#include <set>
#include <string>

namespace stub {

struct Launch {
    std::string kernel;  // demangled
    dim3 grid, block;
    hipStream_t stream;
    void** args;  // the kernel's arguments, valid during the call
    template <typename T>
    T arg(int i) const { return *static_cast<T*>(args[i]); }
};

extern std::function<void(const Launch&)> on_launch;
extern std::function<void(hipStream_t)> on_synchronize;  // before hipStreamSynchronize returns
extern std::set<hipStream_t> capturing;                  // streams under capture
bool allocated(const void* p);  // p lies in device memory that has not been freed
std::map<const char*, size_t> allocations();

}  // namespace stub
