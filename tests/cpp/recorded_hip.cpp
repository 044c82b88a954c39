// Stands in for the calls of the HIP runtime by which a library launches kernels: nothing is launched, and a launch that asks for more
// than 64 KB of dynamic LDS is counted, as refused where its kernel was not allowed that much on the device that is current.
#include <cstddef>
#include <map>
#include <utility>

struct Dim3 {
    unsigned x, y, z;
};

namespace {
int device = 0, large = 0, refused = 0;
std::map<std::pair<int, const void*>, int> allowed;
Dim3 grid, block;
size_t lds;
void* stream;
}  // namespace

extern "C" {
void recorded_set_device(int d) { device = d; }
int recorded_large() { return large; }
int recorded_refused() { return refused; }

int hipGetDevice(int* d) { return *d = device, 0; }
int hipGetLastError() { return 0; }
int hipFuncSetAttribute(const void* kernel, int attribute, int value) {
    if (attribute == 8) allowed[{device, kernel}] = value;        // hipFuncAttributeMaxDynamicSharedMemorySize
    return 0;
}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t l, void* s) { return grid = g, block = b, lds = l, stream = s, 0; }
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* l, void** s) { return *g = grid, *b = block, *l = lds, *s = stream, 0; }
int hipLaunchKernel(const void* kernel, Dim3, Dim3, void**, size_t bytes, void*) {
    if (bytes > 65536) {
        ++large;
        const auto it = allowed.find({device, kernel});
        if (it == allowed.end() || it->second < (int)bytes) ++refused;
    }
    return 0;
}
}
