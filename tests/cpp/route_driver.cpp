// Runs libtv_hip.so's host side on a recorded HIP runtime, without a GPU: which kernels a call
// launches on which grid, and what it does to its workspace (allocations, frees, waits).
//
// The executable itself defines the HIP entry points the library imports; they come before
// libamdhip64.so's in the symbol lookup, so nothing reaches the real runtime.  The device it plays
// has 256 CUs and holds 512 threads of any kernel per CU.  Allocations are made-up addresses.
//
// Lines of standard input (operand strides in elements; pointers are made up, 256-byte aligned plus
// `mis` bytes):
//   gemm|noalloc|gemv dtype_a dtype_b dtype_c batch M N K sa_b sa_m sa_k sb_b sb_k sb_n sc_b sc_m sc_n stream act bias mis_a mis_b mis_c
//   capture 0|1        streams are (not) under capture from here on
//   fail N             the next N allocations fail
// For each call it prints the runtime's events in order, then "rc CODE":
//   launch KERNEL GRID BLOCK STREAM | malloc ID BYTES | malloc-failed BYTES | free ID | sync STREAM
// and "illegal ..." for what a stream under capture forbids.
#include <cxxabi.h>
#include <dlfcn.h>
#include <stdint.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <iostream>
#include <map>
#include <sstream>
#include <string>
#include <utility>

#include "tensorvia_hip.h"

namespace {
struct Dim3 {
    uint32_t x, y, z;
};
std::map<const void*, std::string> g_kernels;
std::map<void*, int> g_live;
int g_ids = 0, g_fail = 0, g_capture = 0;
uintptr_t g_next = (uintptr_t)1 << 44;
Dim3 g_grid, g_block;
size_t g_shmem;
void* g_stream;
int g_error = 0;

std::string demangled(const char* name) {
    std::string m = name; // spell the 16-bit types in a form that every demangler knows
    for (const auto& [from, to] : {std::pair<std::string, std::string>{"DF16b", "u6__bf16"}, {"DF16_", "u8_Float16"}})
        for (size_t at; (at = m.find(from)) != std::string::npos;) m.replace(at, from.size(), to);
    int status = 0;
    char* s = abi::__cxa_demangle(m.c_str(), nullptr, nullptr, &status);
    std::string r = status == 0 && s ? s : name;
    free(s);
    for (const char* drop : {"tvk::", "tiny::", "simt::", "f64::", "void ", " "}) // "gemm_ms_kernel<GemmCfg<...>,4,false>(GemmDesc,...)"
        for (size_t at; (at = r.find(drop)) != std::string::npos;) r.erase(at, std::strlen(drop));
    return r.substr(0, r.find('('));
}
void forbidden_under_capture(const char* what) {
    if (g_capture) std::printf("illegal %s under capture\n", what);
}
} // namespace

extern "C" {
void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* device, unsigned, void*, void*, void*, void*, int*) {
    g_kernels[host] = demangled(device);
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shmem, void* stream) {
    g_grid = grid, g_block = block, g_shmem = shmem, g_stream = stream;
    return 0;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* shmem, void** stream) {
    *grid = g_grid, *block = g_block, *shmem = g_shmem, *stream = g_stream;
    return 0;
}
int hipLaunchKernel(const void* f, Dim3 grid, Dim3 block, void**, size_t, void* stream) {
    // The runtime refuses a grid dimension of 2^32 threads or more.
    const bool ok = (uint64_t)grid.x * block.x <= 0xFFFFFFFFu && grid.x > 0;
    const std::string name = g_kernels.count(f) ? g_kernels[f] : "?";
    std::printf("%s %s %u %u %lu\n", ok ? "launch" : "launch-refused", name.c_str(), grid.x, block.x, (unsigned long)(uintptr_t)stream);
    if (!ok) g_error = 9; // hipErrorInvalidConfiguration
    return g_error;
}
int hipGetLastError() {
    const int e = g_error;
    g_error = 0;
    return e;
}
const char* hipGetErrorString(int) { return "error"; }
int hipGetDevice(int* dev) {
    *dev = 0;
    return 0;
}
int hipDeviceGetAttribute(int* v, int, int) {
    *v = 256; // the library asks for the CU count only
    return 0;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int threads, size_t) {
    *n = 512 / threads;
    return 0;
}
int hipMalloc(void** p, size_t bytes) {
    forbidden_under_capture("allocation");
    if (g_fail > 0 || bytes >= ((size_t)1 << 50)) {
        if (g_fail > 0) --g_fail;
        std::printf("malloc-failed %zu\n", bytes);
        return g_error = 2;
    }
    *p = (void*)g_next;
    g_next += (bytes + 255) / 256 * 256;
    g_live[*p] = ++g_ids;
    std::printf("malloc %d %zu\n", g_ids, bytes);
    return 0;
}
int hipFree(void* p) {
    forbidden_under_capture("free");
    std::printf("free %d\n", g_live.count(p) ? g_live[p] : -1);
    g_live.erase(p);
    return 0;
}
int hipStreamSynchronize(void* stream) {
    forbidden_under_capture("wait");
    std::printf("sync %lu\n", (unsigned long)(uintptr_t)stream);
    return 0;
}
int hipStreamIsCapturing(void*, int* status) {
    *status = g_capture; // hipStreamCaptureStatusActive = 1
    return 0;
}
int hipGetSymbolAddress(void** p, const void*) {
    *p = (void*)((uintptr_t)1 << 40);
    return 0;
}
int hipMemcpyAsync(void*, const void*, size_t, int, void*) { return 0; }
}

int main(int argc, char** argv) {
    if (argc != 2) return 2;
    void* lib = dlopen(argv[1], RTLD_NOW);
    if (!lib) {
        std::fprintf(stderr, "%s\n", dlerror());
        return 2;
    }
    using Gemm = int (*)(const tv_gemm_args*, void*);
    using GemmEx = int (*)(const tv_gemm_args*, const tv_epilogue*, void*);
    const Gemm gemm = (Gemm)dlsym(lib, "tv_hip_gemm"), noalloc = (Gemm)dlsym(lib, "tv_hip_gemm_noalloc"),
               gemv = (Gemm)dlsym(lib, "tv_hip_gemv");
    const GemmEx gemm_ex = (GemmEx)dlsym(lib, "tv_hip_gemm_ex");
    std::string line;
    while (std::getline(std::cin, line)) {
        std::istringstream in(line);
        std::string cmd;
        in >> cmd;
        if (cmd == "capture") in >> g_capture;
        else if (cmd == "fail") in >> g_fail;
        else if (cmd == "gemm" || cmd == "noalloc" || cmd == "gemv") {
            tv_gemm_args a;
            std::memset(&a, 0, sizeof(a));
            unsigned long stream = 0, mis[3] = {0, 0, 0};
            int act = 0, bias = 0;
            in >> a.dtype_a >> a.dtype_b >> a.dtype_c >> a.batch >> a.M >> a.N >> a.K >> a.sa_b >> a.sa_m >> a.sa_k >> a.sb_b >>
                a.sb_k >> a.sb_n >> a.sc_b >> a.sc_m >> a.sc_n >> stream >> act >> bias >> mis[0] >> mis[1] >> mis[2];
            if (!in) return 2;
            a.A = (const void*)(((uintptr_t)1 << 45) + mis[0]);
            a.B = (const void*)(((uintptr_t)2 << 45) + mis[1]);
            a.C = (void*)(((uintptr_t)3 << 45) + mis[2]);
            tv_epilogue ep;
            std::memset(&ep, 0, sizeof(ep));
            ep.act = act;
            if (bias) ep.bias = (const void*)((uintptr_t)5 << 45), ep.sbias_n = 1;
            int rc;
            if (cmd == "noalloc") rc = noalloc(&a, (void*)stream);
            else if (cmd == "gemv") rc = gemv(&a, (void*)stream);
            else rc = act || bias ? gemm_ex(&a, &ep, (void*)stream) : gemm(&a, (void*)stream);
            std::printf("rc %d\n", rc);
        } else return 2;
    }
    return 0;
}
