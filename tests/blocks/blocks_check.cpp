// CPU check of the library's device memory (process_amd/csrc/psx_host.cpp):
// the HIP calls that allocate, free and synchronise are this program's own, a
// device of 1 GiB that counts bytes, and the library is the built one.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

#include "psx_internal.h"

#define CHECK(c)                                                        \
    do {                                                                \
        if (!(c)) {                                                     \
            std::printf("FAIL %s:%d: %s\n", __FILE__, __LINE__, #c);    \
            std::exit(1);                                               \
        }                                                               \
    } while (0)

namespace {

constexpr size_t MIB = size_t(1) << 20, DEVICE = 1024 * MIB;
std::map<void*, size_t> live;
size_t used = 0;
hipError_t last = hipSuccess, sync_result = hipSuccess;

hipError_t ret(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}

}  // namespace

extern "C" {
hipError_t hipGetDeviceCount(int* n) { *n = 1; return ret(hipSuccess); }
hipError_t hipSetDevice(int) { return ret(hipSuccess); }
hipError_t hipGetDevice(int* d) { *d = 0; return ret(hipSuccess); }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    return ret(hipSuccess);
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)1; return ret(hipSuccess); }
hipError_t hipStreamSynchronize(hipStream_t) { return ret(hipSuccess); }
hipError_t hipStreamDestroy(hipStream_t) { return ret(hipSuccess); }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)1; return ret(hipSuccess); }
hipError_t hipEventDestroy(hipEvent_t) { return ret(hipSuccess); }
hipError_t hipGetSymbolAddress(void** p, const void*) { *p = &used; return ret(hipSuccess); }
hipError_t hipDeviceSynchronize() { return ret(sync_result); }
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipMalloc(void** p, size_t n) {
    if (used + n > DEVICE) return ret(hipErrorOutOfMemory);
    *p = std::malloc(1);
    live[*p] = n;
    used += n;
    return ret(hipSuccess);
}
hipError_t hipFree(void* p) {
    if (!p) return ret(hipSuccess);
    CHECK(live.count(p));
    used -= live[p];
    live.erase(p);
    std::free(p);
    return ret(hipSuccess);
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
    *f = DEVICE - used;
    *t = DEVICE;
    return ret(hipSuccess);
}
}

// Tables of n MiB each, freed: their blocks are idle.
static void idle_blocks(size_t n, size_t blocks) {
    std::vector<std::shared_ptr<dbuf>> held;
    for (size_t k = 0; k < blocks; ++k) held.push_back(psx_block(n * MIB));
}

// A caller's buffer takes the memory of idle blocks.
static void alloc(psx_ctx* ctx) {
    idle_blocks(256, 3);
    CHECK(used == 768 * MIB);
    void* p = nullptr;
    CHECK(psx_dev_alloc(ctx, 800 * MIB, &p) == PSX_OK && p);
    CHECK(used == 800 * MIB && last == hipSuccess);
    void* q = nullptr;
    CHECK(psx_dev_alloc(ctx, 300 * MIB, &q) == PSX_ENOMEM_DEVICE);
    psx_dev_free(ctx, p);
    CHECK(used == 0);
}

// Trimming a context gives the device's idle blocks back, and nothing that is in use.
static void trim(psx_ctx* ctx) {
    const std::shared_ptr<dbuf> held = psx_block(64 * MIB);
    idle_blocks(128, 2);
    CHECK(used == 320 * MIB);
    CHECK(psx_ctx_trim(ctx) == PSX_OK);
    CHECK(used == 64 * MIB);
}

// The free memory reported is the device's: idle blocks are not free to others.
static void info(psx_ctx* ctx) {
    uint64_t f = 0, t = 0;
    idle_blocks(256, 2);
    CHECK(psx_ctx_mem_info(ctx, &f, &t) == PSX_OK && f == 512 * MIB && t == DEVICE);
    CHECK(psx_ctx_trim(ctx) == PSX_OK);
    CHECK(psx_ctx_mem_info(ctx, &f, &t) == PSX_OK && f == DEVICE);
}

// A table freed while the device cannot be synchronised (another stream is being captured) is freed at once, and leaves
// no error for the next launch's check.
static void capture(psx_ctx*) {
    sync_result = hipErrorStreamCaptureUnsupported;
    idle_blocks(128, 2);
    sync_result = hipSuccess;
    CHECK(used == 0 && last == hipSuccess);
}

int main(int argc, char** argv) {
    psx_ctx* ctx = nullptr;
    CHECK(psx_ctx_create(0, &ctx) == PSX_OK);
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "alloc") alloc(ctx);
    else if (what == "trim") trim(ctx);
    else if (what == "info") info(ctx);
    else if (what == "capture") capture(ctx);
    else return 2;
    psx_ctx_destroy(ctx);
    CHECK(used == 0 && live.empty());
    std::puts("blocks ok");
    return 0;
}
