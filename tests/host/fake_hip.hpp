// A recording stand-in for the HIP runtime: the executable that includes this
// defines the HIP calls the library makes, so the library's host code runs
// without a GPU and what it allocates, launches and orders can be checked.
// Device memory is an address range that nothing reads or writes.
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <vector>

#include "ltx_args.h"
#include "ltx_block.h"

namespace fake {

struct Op {
    std::string what;  // "launch", "record", "wait", "malloc", "free", "sync", "copy2d"
    std::string name;  // launch: the kernel
    hipStream_t stream = nullptr;
    hipEvent_t event = nullptr;
    uint64_t addr = 0, bytes = 0;
    LtxSplit3Args split{};
    LtxGemmF3Args f3{};
    LtxGemmArgs gemm{};
    LtxAttnArgs attn{};
    LtxVtPadArgs vt{};
    std::map<hipStream_t, uint64_t> clock;  // launch: what of each stream precedes it, itself included
};

inline std::vector<Op> log;
inline std::map<hipStream_t, std::map<hipStream_t, uint64_t>> streams;  // each stream's clock
inline std::map<hipEvent_t, std::map<hipStream_t, uint64_t>> events;    // and each event's, as recorded
inline std::map<uint64_t, uint64_t> mem;   // live allocations
inline uint64_t next_addr = 1ull << 40, in_use = 0, limit = ~0ull;
inline std::set<hipStream_t> capturing;    // streams being captured, in global mode
inline hipStreamCaptureMode thread_mode = hipStreamCaptureModeGlobal;
inline bool broken_capture = false;        // a call that a capture forbids was made
inline std::string fail_launch;            // a launch of this kernel fails
inline uint64_t handles = 0x1000;

// what a capture in global mode forbids to threads that have not opted out
inline hipError_t forbidden() {
    if (capturing.empty() || thread_mode == hipStreamCaptureModeRelaxed) return hipSuccess;
    broken_capture = true;
    return hipErrorStreamCaptureUnsupported;
}
inline bool inside(uint64_t p, uint64_t n) {
    auto it = mem.upper_bound(p);
    if (it == mem.begin()) return false;
    --it;
    return p >= it->first && p + n <= it->first + it->second;
}
// a is done before b starts
inline bool before(const Op& a, const Op& b) {
    auto it = b.clock.find(a.stream);
    return it != b.clock.end() && it->second >= a.clock.at(a.stream) && &a != &b;
}
inline bool inside(const void* p, uint64_t n) { return inside((uint64_t)p, n); }

}  // namespace fake

extern "C" {

hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {  // (a macro: the versioned symbol)
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "fake error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
    if (hipError_t e = fake::forbidden()) return e;
    if (fake::in_use + n > fake::limit) return hipErrorOutOfMemory;
    *p = (void*)fake::next_addr;
    fake::mem[fake::next_addr] = n;
    fake::in_use += n;
    fake::Op o{"malloc"};
    o.addr = fake::next_addr;
    o.bytes = n;
    fake::log.push_back(o);
    fake::next_addr += (n + 0xffffff) & ~0xffffffull;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (hipError_t e = fake::forbidden()) return e;
    auto it = fake::mem.find((uint64_t)p);
    if (it == fake::mem.end()) return hipErrorInvalidValue;
    fake::Op o{"free"};
    o.addr = it->first;
    o.bytes = it->second;
    fake::log.push_back(o);
    fake::in_use -= it->second;
    fake::mem.erase(it);
    return hipSuccess;
}
hipError_t hipMemcpy(void*, const void*, size_t, hipMemcpyKind) { return fake::forbidden(); }
hipError_t hipMemcpy2D(void*, size_t, const void*, size_t, size_t, size_t, hipMemcpyKind) {
    fake::log.push_back({"copy2d"});
    return fake::forbidden();
}
hipError_t hipMemset(void*, int, size_t) { return fake::forbidden(); }
hipError_t hipDeviceSynchronize() {
    fake::log.push_back({"sync"});
    if (fake::capturing.empty()) return hipSuccess;
    fake::broken_capture = true;  // also for a thread that has opted out
    return hipErrorStreamCaptureUnsupported;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    fake::log.push_back({"sync"});
    return fake::capturing.count(s) ? hipErrorStreamCaptureUnsupported : hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    *p = (void*)(fake::next_addr);
    fake::mem[fake::next_addr] = LTX_NOALLOC_SCRATCH_BYTES;
    fake::next_addr += 1ull << 30;
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return *e = (hipEvent_t)(fake::handles += 16), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    fake::Op o{"record"};
    o.event = e;
    o.stream = s;
    fake::log.push_back(o);
    fake::events[e] = fake::streams[s];
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    fake::Op o{"wait"};
    o.event = e;
    o.stream = s;
    fake::log.push_back(o);
    for (auto& [stream, n] : fake::events[e]) fake::streams[s][stream] = std::max(fake::streams[s][stream], n);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    return *s = (hipStream_t)(fake::handles += 16), hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
    *st = fake::capturing.count(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) {
    std::swap(*m, fake::thread_mode);
    return hipSuccess;
}
hipError_t hipModuleLoadData(hipModule_t* m, const void*) {
    return *m = (hipModule_t)(fake::handles += 16), hipSuccess;
}
hipError_t hipModuleUnload(hipModule_t) { return hipSuccess; }
hipError_t hipModuleGetFunction(hipFunction_t* f, hipModule_t, const char* name) {
    return *f = (hipFunction_t)strdup(name), hipSuccess;
}
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned,
                                 hipStream_t s, void** params, void**) {
    fake::Op o{"launch"};
    o.name = (const char*)f;
    o.stream = s;
    if (o.name == fake::fail_launch) return hipErrorUnknown;
    fake::streams[s][s]++;
    o.clock = fake::streams[s];
    auto is = [&](const char* prefix) { return o.name.rfind(prefix, 0) == 0; };
    if (is("ltx_split3")) o.split = *(LtxSplit3Args*)params[0];
    if (is("ltx_gemm_f3_")) o.f3 = *(LtxGemmF3Args*)params[0];
    if (is("ltx_gemm_x4") || is("ltx_gemm_s4") || is("ltx_gemm_q8") || is("ltx_gemm_w16") || is("ltx_gemm_reduce"))
        o.gemm = *(LtxGemmArgs*)params[0];
    if (is("ltx_attn") && o.name != "ltx_attn_f32") o.attn = *(LtxAttnArgs*)params[0];
    if (is("ltx_vt_")) o.vt = *(LtxVtPadArgs*)params[0];
    fake::log.push_back(o);
    return hipSuccess;
}
}
