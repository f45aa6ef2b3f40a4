// A HIP runtime that launches nothing: it records the kernel launches and
// function attributes of a library loaded after it (RTLD_GLOBAL), so that a
// test without a GPU sees which kernel and launch shape a call takes and on
// which device each attribute was set. Pointers are never followed.
#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <string>

#include <cxxabi.h>

namespace {

struct Dim3 {
    std::uint32_t x, y, z;
};

struct Config {
    Dim3 grid, block;
    std::size_t shared;
    void* stream;
};

thread_local int current_device = 0;
thread_local Config config;

std::map<const void*, std::string>& names() {
    static std::map<const void*, std::string> m;
    return m;
}

std::string& events() {
    static std::string text;
    return text;
}

std::string name_of(const void* f) {
    const auto it = names().find(f);
    if (it == names().end()) return "?";
    int status = 0;
    char* plain = abi::__cxa_demangle(it->second.c_str(), nullptr, nullptr, &status);
    std::string name = status == 0 ? plain : it->second;
    std::free(plain);
    const auto anonymous = name.find("(anonymous namespace)::");
    if (anonymous != std::string::npos) name = name.substr(anonymous + 23);
    return name.substr(0, name.find('('));
}

}  // namespace

extern "C" {

void recorder_device(int device) { current_device = device; }

// The events since the last call, one per line: "set|name|device|value" or "launch|name|device|blocks|threads|bytes".
const char* recorder_take() {
    static std::string taken;
    taken.swap(events());
    events().clear();
    return taken.c_str();
}

// The names of all registered kernels, one per line.
const char* recorder_kernels() {
    static std::string text;
    text.clear();
    for (const auto& [host, name] : names()) text += name_of(host) + "\n";
    return text.c_str();
}

void** __hipRegisterFatBinary(const void*) {
    static void* modules = nullptr;
    return &modules;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, std::size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* device, unsigned, void*, void*, void*, void*, int*) {
    names()[host] = device;
}

int __hipPushCallConfiguration(Dim3 grid, Dim3 block, std::size_t shared, void* stream) {
    config = {grid, block, shared, stream};
    return 0;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, std::size_t* shared, void** stream) {
    *grid = config.grid;
    *block = config.block;
    *shared = config.shared;
    *stream = config.stream;
    return 0;
}

int hipLaunchKernel(const void* f, Dim3 grid, Dim3 block, void**, std::size_t shared, void*) {
    const unsigned long long blocks = 1ull * grid.x * grid.y * grid.z, threads = 1ull * block.x * block.y * block.z;
    events() += "launch|" + name_of(f) + "|" + std::to_string(current_device) + "|" + std::to_string(blocks) + "|" +
                std::to_string(threads) + "|" + std::to_string(shared) + "\n";
    return 0;
}
int hipFuncSetAttribute(const void* f, int, int value) {
    events() += "set|" + name_of(f) + "|" + std::to_string(current_device) + "|" + std::to_string(value) + "\n";
    return 0;
}

int hipGetDevice(int* device) {
    *device = current_device;
    return 0;
}
int hipDeviceGetAttribute(int* value, int, int) {
    *value = 256;  // compute units of an MI355X
    return 0;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* blocks, const void*, int, std::size_t) {
    *blocks = 2;
    return 0;
}
int hipGetLastError() { return 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipStreamIsCapturing(void*, int* status) {
    *status = 0;
    return 0;
}

}  // extern "C"
