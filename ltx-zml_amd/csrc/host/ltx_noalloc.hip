// ltx_op_linear_q8_noalloc: the isolated int8 GEMM with its scratch in a
// static device array instead of memory the context allocates, for callers
// that may not allocate device memory (code under HIP graph capture, serving
// loops, harnesses that forbid hipMalloc).
//
// `scratch` is one file-scope array per GPU (the code object holding it is
// loaded on each device the library runs on, and stays until the process
// ends). Its host-side name is only a stand-in: the device address comes from
// hipGetSymbolAddress, resolved once per device with that device current
// (ltx_init), and only that address is handed to kernels.
//
// Compiled by hipcc as a host object (with the array's gfx950 code object
// embedded and registered when the library loads); the kernels that use the
// scratch live in the library's own code objects and take its address as an
// argument.
#include <hip/hip_runtime.h>

#include <mutex>

#include "ltx_internal.hpp"

static __device__ __align__(256) unsigned char scratch[LTX_NOALLOC_SCRATCH_BYTES];
// Mode F32's planes and partial sums, an array of their own: its calls use none
// of the above and may overlap calls that do.
static __device__ __align__(256) unsigned char planes[LTX_NOALLOC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_mu;
struct Device {
    void* scratch = nullptr;
    void* planes = nullptr;
    // the last use of planes: calls of every context and thread follow each other
    std::mutex mu;
    hipEvent_t ev = nullptr;
    bool used = false;
} g_dev[kMaxDevices];

// One call's use of the planes, ordered behind the last one and recorded when
// the scope ends. Not for a call that is being captured: nothing here could
// order its replays.
struct PlanesUse {
    Device* d = nullptr;
    std::unique_lock<std::mutex> lk;
    hipStream_t st;
    explicit PlanesUse(hipStream_t stream) : st(stream) {}
    void* take(Device& dev) {
        if (ltx::is_capturing(st)) return nullptr;
        lk = std::unique_lock<std::mutex>(dev.mu);
        if (dev.used) HIPC(hipStreamWaitEvent(st, dev.ev, 0));
        d = &dev;
        return dev.planes;
    }
    ~PlanesUse() {
        if (!d) return;
        if (hipEventRecord(d->ev, st) == hipSuccess)
            d->used = true;
        else
            (void)hipStreamSynchronize(st);  // nothing to wait for later
    }
};
}  // namespace

namespace ltx {

void noalloc_setup(int device) {
    std::lock_guard<std::mutex> lk(g_mu);
    if (device < 0 || device >= kMaxDevices) throw Error("noalloc: device index beyond the supported 64");
    Device& d = g_dev[device];
    if (d.ev) return;
    void *p = nullptr, *q = nullptr;
    HIPC(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    HIPC(hipGetSymbolAddress(&q, HIP_SYMBOL(planes)));
    if (!p || !q) throw Error("noalloc: hipGetSymbolAddress returned no address for the scratch array");
    HIPC(hipEventCreateWithFlags(&d.ev, hipEventDisableTiming));
    d.scratch = p;
    d.planes = q;
}

void* noalloc_scratch(int device) {
    std::lock_guard<std::mutex> lk(g_mu);
    return device >= 0 && device < kMaxDevices ? g_dev[device].scratch : nullptr;
}

}  // namespace ltx

extern "C" int ltx_op_linear_q8_noalloc(ltx_ctx* c, const void* a, const int8_t* q, const void* scales, int scale_f16,
                                        const float* bias, void* y, int out_f32, int M, int N, int K, int gelu,
                                        int mode, void* stream) {
    LTX_GUARD(c, {
        if (!c) throw ltx::Error("NULL context");
        ltx::check_linear_q8(M, N, K, mode);
        ltx::LinearScratch sc{};
        if (ltx::linear_q8_needs_scratch(c, N, K, mode)) {
            // weights as bytes q + 128, then the scale words, then (where
            // ltx_op_linear_q8 runs the four-wave kernel) the weights
            // dequantised to the operand type, each 256-byte aligned
            auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
            const size_t nq = al((size_t)N * K), np = al((size_t)N * (K / LTX_GROUP) * 4);
            const size_t nw = ltx::x4_shape(c, mode, M, N, K, K) ? (size_t)N * K * 2 : 0;
            if (nq + np + nw > LTX_NOALLOC_SCRATCH_BYTES)
                throw ltx::Error(std::string("ltx_op_linear_q8_noalloc: ") +
                                 (nw ? "N * K + 4 N K / 128 + 2 N K bytes (the 16-bit weight copy of the "
                                       "four-wave GEMM, from 4,096 rows)"
                                     : "N * K + 4 N K / 128 bytes") +
                                 " exceed the " + std::to_string(LTX_NOALLOC_SCRATCH_BYTES) + "-byte scratch");
            char* base = (char*)ltx::noalloc_scratch(c->device);
            if (!base) throw ltx::Error("ltx_op_linear_q8_noalloc: scratch not set up on this device");
            sc.q = (uint32_t*)base;
            sc.pairs = (uint32_t*)(base + nq);
            sc.w16 = nw ? base + nq + np : nullptr;
        }
        char* base = (char*)ltx::noalloc_scratch(c->device);
        HIPC(hipSetDevice(c->device));
        PlanesUse use((hipStream_t)stream);
        if (mode == LTX_MODE_F32 && ltx::f3_shape(c, M, N, K)) {
            // the planes of as many rows of A as fit, with their partial sums;
            // at least 128: a split has at most 256 tiles x slices of 64 KB,
            // and K is at most 32,768
            const int rows = ltx::f3_rows(c, M, N, K, LTX_NOALLOC_SCRATCH_BYTES);
            if (!base) throw ltx::Error("ltx_op_linear_q8_noalloc: scratch not set up on this device");
            if (!rows) throw ltx::Error("ltx_op_linear_q8_noalloc: scratch too small for 128 rows");  // (cannot happen)
            if ((sc.planes = use.take(g_dev[c->device]))) {
                sc.plane_rows = rows;
                sc.part = ltx::f3_part_bytes(c, M, N, K) ? (char*)sc.planes + ltx::f3_planes_bytes(rows, K) : nullptr;
            }
        }
        if (const size_t part = ltx::linear_packed(a, q, scales, scale_f16, bias, y, K) ? ltx::linear_part_bytes(c, M, N, K, mode) : 0) {
            // beside the scale words; the room of the bytes q + 128 is free
            // (packed operands). At most 64 MiB: 256 tiles x slices of 256 KB
            const size_t np = ((size_t)N * (K / LTX_GROUP) * 4 + 255) & ~(size_t)255;
            if (np + part > LTX_NOALLOC_SCRATCH_BYTES)
                throw ltx::Error("ltx_op_linear_q8_noalloc: scratch too small for the partial sums");  // (cannot happen)
            sc.pairs = (uint32_t*)base;
            sc.part = base + np;
        }
        ltx::linear_q8(c, a, q, scales, scale_f16, bias, y, out_f32, M, N, K, gelu, mode, sc, (hipStream_t)stream);
    })
}
