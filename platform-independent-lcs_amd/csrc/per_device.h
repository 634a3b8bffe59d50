// Set-up that a process makes once for every device it uses.
#pragma once
#include <hip/hip_runtime.h>

#include <map>
#include <mutex>

// Kernel attributes belong to the device that is current when they are set, so
// a flag per process would leave a second device's kernels without theirs.
class PerDevice {
    std::mutex mu;
    std::map<int, int> status;

public:
    // set()'s result for the calling thread's device; set() runs the first time.
    template <typename Set>
    int once(Set set)
    {
        int device = 0;
        if (hipGetDevice(&device) != hipSuccess) return -5;
        const std::lock_guard<std::mutex> lock(mu);
        const auto it = status.find(device);
        if (it != status.end()) return it->second;
        return status[device] = set();
    }
};
