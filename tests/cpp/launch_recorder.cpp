// Stand-ins for the HIP runtime's entry points that libtvdcn_hip.so calls. Loaded ahead of it (RTLD_GLOBAL) in a
// process of its own, they record the launches of a call on the host: no device is touched and no kernel runs.
// An empty grid is refused and a grid whose x extent times its block is not below 2^32 threads too, as by HIP.
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {

struct Dim3 {
    uint32_t x, y, z;
};
struct Launch {
    std::string name;
    Dim3 grid, block;
    size_t shared;
};
struct Config {
    Dim3 grid, block;
    size_t shared;
    void *stream;
};

constexpr int kSuccess = 0, kInvalidConfiguration = 9;
std::map<const void *, std::string> &names() {
    static std::map<const void *, std::string> m;
    return m;
}
std::vector<Launch> &launches() {
    static std::vector<Launch> v;
    return v;
}
Config config;
int last_error = kSuccess;
char scratch[256];

}  // namespace

extern "C" {

void **__hipRegisterFatBinary(const void *) {
    static void *handle = nullptr;
    return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *) {
    names()[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shared, void *stream) {
    config = {grid, block, shared, stream};
    return kSuccess;
}
int __hipPopCallConfiguration(Dim3 *grid, Dim3 *block, size_t *shared, void **stream) {
    *grid = config.grid, *block = config.block, *shared = config.shared, *stream = config.stream;
    return kSuccess;
}
int hipLaunchKernel(const void *f, Dim3 grid, Dim3 block, void **, size_t shared, void *) {
    launches().push_back({names()[f], grid, block, shared});
    const uint64_t threads = (uint64_t)grid.x * block.x;
    last_error = threads == 0 || grid.y == 0 || grid.z == 0 || threads > UINT32_MAX ? kInvalidConfiguration : kSuccess;
    return last_error;
}
int hipGetLastError() {
    const int e = last_error;
    last_error = kSuccess;
    return e;
}
const char *hipGetErrorString(int) { return "invalid configuration argument"; }
int hipGetDevice(int *device) { return *device = 0, kSuccess; }
int hipFuncSetAttribute(const void *, int, int) { return kSuccess; }
int hipGetSymbolAddress(void **p, const void *) { return *p = scratch, kSuccess; }
int hipEventCreate(void **) { return 1; }
int hipEventRecord(void *, void *) { return 1; }
int hipEventSynchronize(void *) { return 1; }
int hipEventElapsedTime(float *, void *, void *) { return 1; }

int recorded_launches() { return (int)launches().size(); }
const char *recorded_name(int i) { return launches()[i].name.c_str(); }
void recorded_shape(int i, uint32_t *v) {
    const Launch &l = launches()[i];
    const uint32_t w[7] = {l.grid.x, l.grid.y, l.grid.z, l.block.x, l.block.y, l.block.z, (uint32_t)l.shared};
    std::memcpy(v, w, sizeof(w));
}
void recorded_clear() { launches().clear(); }

}  // extern "C"
