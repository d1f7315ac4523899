// Stands before the HIP runtime's hipLaunchKernel in a process that loads this library first (globally):
// launches of the kernel whose name contains refuse_name are handed on with a null function, which the
// runtime refuses on the host (an invalid device function, recorded as the thread's last error) -- what a
// launch that does not fit the device leaves behind.
#include <dlfcn.h>
#include <atomic>
#include <cstdint>
#include <cstdlib>
#include <cstring>

namespace {
struct Dim3 {
    uint32_t x, y, z;
};
typedef int (*Launch)(const void*, Dim3, Dim3, void**, size_t, void*);
typedef const char* (*Name)(const void*, void*);
char g_name[256] = "";
std::atomic<int> g_refused{0};

void* runtime(const char* symbol) {
    static void* lib = dlopen("libamdhip64.so.7", RTLD_LAZY);
    void* f = lib ? dlsym(lib, symbol) : nullptr;
    if (!f) std::abort();
    return f;
}
}  // namespace

extern "C" {
void refuse_name(const char* name) { std::strncpy(g_name, name, sizeof(g_name) - 1); }
int refused() { return g_refused.exchange(0); }

int hipLaunchKernel(const void* f, Dim3 grid, Dim3 block, void** args, size_t shmem, void* stream) {
    static const Launch launch = reinterpret_cast<Launch>(runtime("hipLaunchKernel"));
    static const Name name = reinterpret_cast<Name>(runtime("hipKernelNameRefByPtr"));
    const char* n = g_name[0] ? name(f, stream) : nullptr;
    if (n && std::strstr(n, g_name)) {
        ++g_refused;
        f = nullptr;
    }
    return launch(f, grid, block, args, shmem, stream);
}
}
