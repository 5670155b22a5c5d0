// Runs the C API over a stand-in for the HIP runtime: device memory is address ranges that nothing
// touches, and a launch is recorded instead of run.  The program's own hip* functions take precedence
// over libamdhip64's for libac_hip.so, so no device is needed and none is used.
//
// Commands, one a line on stdin; every answer is a line "rc <code> <seconds>", then one line per launch,
// "<kernel> <grid x> <grid y> <block x> <LDS bytes> <strips> <rows>", then "end" (strips and rows of a
// strip: of the batch kernels that take them as arguments, else 0):
//   legacy <precision> <config> <type> <w> <h>      achip_pass_config (config -1: ACHIP_AUTO)
//   layers <type> <w> <h>                           achip_pass_layers
//   net8 <blocks> <precision> <type> <w> <h>        achip_pass8_precision
//   art <channels> <blocks> <type> <w> <h>          achip_pass_net
//   fsr <channels> <blocks> <type> <w> <h>          achip_pass_net
//   batch <precision> <config> <n> <w> <h>          achip_pass_batch, u8, n images of w x h
//   batch_layers <n> <w> <h>                        achip_pass_batch_layers, the same
//   images <precision> <w> <h> <w> <h> ...          achip_pass_batch, u8, images of these sizes
//   images_layers <w> <h> <w> <h> ...               achip_pass_batch_layers, the same
//   tune <precision> <w> <h> <us of each configuration>   achip_autotune, u8, with these times
//   fail <k>                                        launch k (from 0) of the next command fails
#ifndef __HIP_PLATFORM_AMD__
#define __HIP_PLATFORM_AMD__ 1
#endif
#include <hip/hip_runtime_api.h>

#include <chrono>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <iostream>
#include <map>
#include <sstream>
#include <string>
#include <vector>

#include "achip.h"

namespace {

struct Launch {
    std::string name;
    dim3 grid, block;
    size_t lds;
    int strips, rows;
};

std::map<const void*, std::string>& names()
{
    static std::map<const void*, std::string> m;
    return m;
}
std::vector<Launch> launches;
long fail_at = -1, count = 0;
hipError_t last = hipSuccess;
std::map<uintptr_t, size_t> memory;
uintptr_t next_address = uintptr_t(1) << 40;
dim3 call_grid, call_block;
size_t call_lds = 0;
std::vector<float> tune_us;
int records = 0;

uintptr_t allocate(size_t bytes)
{
    const uintptr_t p = next_address;
    next_address += (bytes + 4095) / 4096 * 4096 + 4096;
    memory[p] = bytes;
    return p;
}

} // namespace

extern "C" {

void** __hipRegisterFatBinary(const void*)
{
    static void* module;
    return &module;
}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
    names()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t)
{
    call_grid = grid;
    call_block = block;
    call_lds = lds;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream)
{
    *grid = call_grid;
    *block = call_block;
    *lds = call_lds;
    *stream = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t)
{
    const std::string& name = names()[f];
    const bool queue = name.find("acnet_stream16_batch") != std::string::npos;   // desc, n, total, counter, 3 weights, rows
    const bool layers = name.find("conv8_rows_batch") != std::string::npos;      // desc, n, total, out, from_m1, Rows8
    launches.push_back({ name, grid, block, lds, queue || layers ? *static_cast<int*>(args[2]) : 0,
                         queue    ? *static_cast<int*>(args[7])
                         : layers ? *reinterpret_cast<int*>(static_cast<char*>(args[5]) + 64)   // after 7 pointers and longs, W, H
                                  : 0 });
    const bool empty = !grid.x || !grid.y || !grid.z || !block.x;
    // a dimension of the grid holds fewer than 2^32 threads, a workgroup at most 1024, a CU 160 KB of LDS
    const bool large = uint64_t(grid.x) * block.x > UINT32_MAX || uint64_t(grid.y) * block.y > UINT32_MAX || block.x > 1024 ||
                       lds > 160 * 1024;
    if (count++ == fail_at || empty || large) {
        last = hipErrorInvalidConfiguration;
        return last;
    }
    return hipSuccess;
}
hipError_t hipGetLastError()
{
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "recorded"; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 2; return hipSuccess; }
hipError_t hipMalloc(void** p, size_t bytes) { *p = reinterpret_cast<void*>(allocate(bytes)); return hipSuccess; }
hipError_t hipFree(void* p) { memory.erase(reinterpret_cast<uintptr_t>(p)); return hipSuccess; }
hipError_t hipMemcpy(void*, const void*, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*)
{
    std::memset(a, 0, sizeof(*a));
    a->type = hipMemoryTypeDevice;
    return hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t* base, size_t* size, hipDeviceptr_t p)
{
    auto it = memory.upper_bound(reinterpret_cast<uintptr_t>(p));
    if (it == memory.begin()) return hipErrorInvalidValue;
    --it;
    *base = reinterpret_cast<hipDeviceptr_t>(it->first);
    *size = it->second;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = nullptr; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t)
{
    *ms = tune_us.empty() ? 1.0f : tune_us[records++ % tune_us.size()];
    return hipSuccess;
}

} // extern "C"

namespace {

int size_of(int type) { return type & 0xff; }

struct Image {
    void *src, *dst;
    long ss, ds;
    Image(int type, long w, long h) : ss(w * size_of(type)), ds(2 * w * size_of(type))
    {
        src = reinterpret_cast<void*>(allocate(static_cast<size_t>(ss) * h));
        dst = reinterpret_cast<void*>(allocate(static_cast<size_t>(ds) * 2 * h));
    }
};

int run(const std::string& what, std::istringstream& in)
{
    static const std::vector<float> zeros(1 << 20, 0.0f);
    const float* z = zeros.data();
    ACHipNet* net = nullptr;
    int type = 1, w = 0, h = 0, rc = -1;
    if (what == "legacy") {
        int precision = 0, config = 0;
        in >> precision >> config >> type >> w >> h;
        if (achip_net_create(0, z, z, &net)) return -1000;
        const Image im(type, w, h);
        rc = achip_pass_config(net, precision, config, im.src, im.ss, type, w, h, im.dst, im.ds, type, nullptr);
    } else if (what == "layers") {
        in >> type >> w >> h;
        if (achip_net_create(0, z, z, &net)) return -1000;
        const Image im(type, w, h);
        const size_t need = achip_pass8_workspace_bytes(w, h);
        rc = achip_pass_layers(net, im.src, im.ss, type, w, h, im.dst, im.ds, type, reinterpret_cast<void*>(allocate(need)), need, nullptr);
    } else if (what == "net8") {
        int blocks = 0, precision = 0;
        in >> blocks >> precision >> type >> w >> h;
        if (achip_net8_create(0, blocks, z, z, z, &net)) return -1000;
        const Image im(type, w, h);
        const size_t need = achip_pass8_workspace_bytes(w, h);
        rc = achip_pass8_precision(net, precision, im.src, im.ss, type, w, h, im.dst, im.ds, type, reinterpret_cast<void*>(allocate(need)),
                                   need, nullptr);
    } else if (what == "art" || what == "fsr") {
        int channels = 0, blocks = 0;
        in >> channels >> blocks >> type >> w >> h;
        if (what == "art" ? achip_net_artcnn_create(0, channels, blocks, z, z, &net)
                          : achip_net_fsrcnnx_create(0, channels, blocks, z, z, z, &net))
            return -1000;
        const Image im(type, w, h);
        const size_t need = achip_net_workspace_bytes(net, w, h);
        rc = achip_pass_net(net, im.src, im.ss, type, w, h, im.dst, im.ds, type, reinterpret_cast<void*>(allocate(need)), need, nullptr);
    } else if (what == "batch" || what == "batch_layers" || what == "images" || what == "images_layers") {
        const bool queue = what == "batch" || what == "images", same = what == "batch" || what == "batch_layers";
        int precision = 0, config = 0, n = 0;
        if (queue) in >> precision;
        if (what == "batch") in >> config;
        if (same) in >> n >> w >> h;
        if (achip_net_create(0, z, z, &net)) return -1000;
        std::vector<ACHipImage> images;
        while (same ? static_cast<int>(images.size()) < n : static_cast<bool>(in >> w >> h)) {
            const Image im(type, w, h);
            images.push_back({ im.src, im.ss, im.dst, im.ds, w, h });
        }
        n = static_cast<int>(images.size());
        const size_t need = queue ? achip_batch_workspace_bytes(n) : achip_pass_batch_layers_bytes(images.data(), n);
        void* ws = reinterpret_cast<void*>(allocate(need));
        rc = queue ? achip_pass_batch(net, precision, config, type, type, images.data(), n, ws, need, nullptr)
                   : achip_pass_batch_layers(net, type, type, images.data(), n, ws, need, nullptr);
    } else if (what == "tune") {
        int precision = 0, best = 0;
        in >> precision >> w >> h;
        tune_us.clear();
        records = 0;
        for (float us = 0; in >> us;) tune_us.push_back(us);
        if (achip_net_create(0, z, z, &net)) return -1000;
        rc = achip_autotune(net, precision, type, type, w, h, &best, nullptr);
        if (rc == 0) rc = best;
    }
    achip_net_destroy(net);
    return rc;
}

} // namespace

int main()
{
    std::string line;
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        std::string what;
        in >> what;
        if (what == "fail") {
            in >> fail_at;
            continue;
        }
        launches.clear();
        count = 0;
        const auto t0 = std::chrono::steady_clock::now();
        const int rc = run(what, in);
        const double s = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
        fail_at = -1;
        last = hipSuccess;
        memory.clear();
        std::printf("rc %d %.6f\n", rc, s);
        for (const Launch& l : launches)
            std::printf("%s %u %u %u %zu %d %d\n", l.name.c_str(), l.grid.x, l.grid.y, l.block.x, l.lds, l.strips, l.rows);
        std::printf("end\n");
    }
    return 0;
}
