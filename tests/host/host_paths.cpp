// The library's host code on the recording HIP stand-in: one check per
// command, run by tests/test_host_paths.py. A failed check says what it saw
// and ends the program with status 1.
#include "fake_hip.hpp"
#include "ltx_internal.hpp"

#define CHECK(cond, ...)                                  \
    do {                                                  \
        if (!(cond)) {                                    \
            std::printf("line %d: %s: ", __LINE__, #cond); \
            std::printf(__VA_ARGS__);                     \
            std::printf("\n");                            \
            std::exit(1);                                 \
        }                                                 \
    } while (0)

static ltx_ctx* make_ctx() {
    ltx_ctx* c = nullptr;
    CHECK(ltx_init(0, &c), "%s", ltx_last_error(nullptr));
    return c;
}

// weights of a block, resident as the recipe keeps them (addresses only)
static void fill(ltx_block_weights& w, bool q8) {
    auto proj = [&](LtxProj& p, int N, int K, bool q) {
        p.N = N;
        p.K = K;
        p.q8 = q;
        p.qflip = q;
        p.scale_f16 = 1;
        for (ltx::DevBuf* b : {&p.q, &p.s, &p.s2, &p.w_bf16, &p.w_f16, &p.bias}) b->alloc(256);
    };
    proj(w.qkv1, 3 * LTX_D, LTX_D, q8);
    proj(w.o1, LTX_D, LTX_D, q8);
    proj(w.q2, LTX_D, LTX_D, q8);
    proj(w.kv2, 2 * LTX_D, LTX_D, q8);
    proj(w.o2, LTX_D, LTX_D, q8);
    proj(w.f1, LTX_FF, LTX_D, q8);
    proj(w.f2, LTX_D, LTX_FF, q8);
    proj(w.g1, LTX_H, LTX_D, false);
    proj(w.g2, LTX_H, LTX_D, false);
    for (ltx::DevBuf* b : {&w.qn1, &w.kn1, &w.qn2, &w.kn2, &w.sst, &w.psst}) b->alloc(256);
}

static float* const X = (float*)(1ull << 36);  // a caller's tensors: aligned addresses
static float* ptr(int i) { return X + ((size_t)i << 30); }

static void forward(ltx_ctx* c, const ltx_block_weights& w, int T, int S, int mode, hipStream_t st = nullptr) {
    CHECK(ltx_block_forward(c, &w, ptr(0), ptr(1), 3, (int32_t*)ptr(2), ptr(3), S, ptr(4), ptr(5), ptr(6), T, ptr(7), mode,
                            st),
          "T=%d S=%d: %s", T, S, ltx_last_error(c));
}

// Mode F32: what is split into planes fits the room the workspace has for them,
// and is split only for a GEMM that reads it.
static void f32_planes(int T, int S) {
    ltx_ctx* c = make_ctx();
    ltx_block_weights w;
    fill(w, true);
    forward(c, w, T, S, LTX_MODE_F32);
    const fake::Op* split = nullptr;
    int used = 0, splits = 0;
    for (const fake::Op& o : fake::log) {
        if (o.name == "ltx_split3") {
            CHECK(!split || used, "planes of %zu values that no GEMM read", split->split.n);
            split = &o;
            used = 0;
            splits++;
            for (uint16_t* p : {o.split.p0, o.split.p1, o.split.p2})
                CHECK((uint64_t)p >= (uint64_t)c->ws.p && (uint64_t)p + 2 * o.split.n <= (uint64_t)c->ws.p + c->ws.bytes,
                      "a plane of %zu values ends %.3f GB past the workspace", o.split.n,
                      ((double)(uint64_t)p + 2.0 * o.split.n - (double)(uint64_t)c->ws.p - c->ws.bytes) / 1e9);
        }
        if (o.name.rfind("ltx_gemm_f3_", 0) == 0) {
            CHECK(split && o.f3.g.a == split->split.p0 && (size_t)o.f3.g.M * o.f3.g.K == split->split.n,
                  "a GEMM of %d x %d on other planes", o.f3.g.M, o.f3.g.K);
            used++;
        }
    }
    CHECK(!split || used, "planes that no GEMM read");
    std::printf("%d splits\n", splits);
}

int main(int argc, char** argv) {
    const std::string cmd = argc > 1 ? argv[1] : "";
    auto arg = [&](int i) { return argc > i ? std::atoi(argv[i]) : 0; };
    if (cmd == "f32_planes")
        f32_planes(arg(2), arg(3));
    else
        CHECK(false, "unknown command %s", cmd.c_str());
    std::printf("ok\n");
    std::fflush(stdout);
    std::_Exit(0);  // (the library's own teardown belongs to the real runtime)
}
