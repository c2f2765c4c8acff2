// Transfers between host arrays and device buffers (host code; no device types).
#pragma once
#include <cstddef>
#include <vector>

namespace p4a {

struct HostCopy {
    double* dev;
    double* host;
    size_t n;         // doubles
    const void* buf;  // the device allocation that dev lies in
};

// f(device pointer, byte offset in the staging, bytes) once per run of adjacent arrays of one allocation.  Two
// allocations may lie side by side; a copy over the end of one is not joined to the next, since the runtime may refuse it.
template <class F>
void for_runs(const std::vector<HostCopy>& x, F&& f) {
    size_t off = 0;
    for (size_t i = 0; i < x.size();) {
        size_t j = i + 1, n = x[i].n;
        while (j < x.size() && x[j].buf == x[i].buf && x[j].dev == x[j - 1].dev + x[j - 1].n) n += x[j++].n;
        f(x[i].dev, off, n * sizeof(double));
        off += n * sizeof(double);
        i = j;
    }
}

}  // namespace p4a
