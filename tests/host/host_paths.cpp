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

static bool linear(ltx_ctx* c, int M, int N, int K, int mode, hipStream_t st, bool noalloc = false, int scale_f16 = 1) {
    auto f = noalloc ? ltx_op_linear_q8_noalloc : ltx_op_linear_q8;
    return f(c, ptr(0), (const int8_t*)ptr(1), ptr(2), scale_f16, nullptr, ptr(3), mode == LTX_MODE_F32, M, N, K, 0, mode,
             st);
}
static bool attention(ltx_ctx* c, int lq, int lkv, hipStream_t st, size_t k_off = 0) {
    return ltx_op_attention(c, ptr(0), (char*)ptr(1) + k_off, ptr(2), nullptr, ptr(3), lq, lkv, LTX_MODE_F16, st);
}

// The uses of one shared scratch follow each other, whatever the stream's
// handle (the per-thread stream has one handle for all threads, and a destroyed
// stream's may come back): between two uses lies a record behind the first and a
// wait for it before the second. A call that fails half-way counts as a use.
// `scratch` names the kernels that write it, `call` makes one call on a stream.
template <class Call>
static void scratch_order(const char* scratch, const char* reader, Call call) {
    const hipStream_t s1 = (hipStream_t)0x10, s2 = (hipStream_t)0x20;
    CHECK(call(s1), "%s", ltx_last_error(nullptr));
    fake::log.clear();
    int n = 0;
    auto uses = [&]() {  // checks the calls logged so far
        hipEvent_t behind = nullptr;  // recorded behind the last use, and waited for
        bool recorded = false, waited = false;
        n = 0;
        for (const fake::Op& o : fake::log) {
            if (o.what == "record") behind = o.event, recorded = true, waited = false;
            if (o.what == "wait" && recorded && o.event == behind) waited = true;
            if (o.what == "launch" && o.name.rfind(scratch, 0) == 0) {
                CHECK(!n || (recorded && waited), "use %d: %s%s", n + 1, recorded ? "recorded " : "not recorded ",
                      waited ? "waited" : "not waited");
                recorded = waited = false;
                n++;
            }
        }
    };
    for (hipStream_t s : {s1, s1, s2, s1}) CHECK(call(s), "%s", ltx_last_error(nullptr));
    uses();
    CHECK(n == 4, "%d uses", n);
    fake::fail_launch = reader;
    CHECK(!call(s1), "a failed launch went unnoticed");
    fake::fail_launch.clear();
    CHECK(call(s2), "%s", ltx_last_error(nullptr));
    uses();
    CHECK(n == 6, "%d uses", n);
}

static int launches(const std::string& prefix) {
    int n = 0;
    for (const fake::Op& o : fake::log) n += o.what == "launch" && o.name.rfind(prefix, 0) == 0;
    return n;
}

// The scratch grows for a call beside a stream that is being captured in global
// mode: the call runs as it always does and the capture stays whole.
static void scratch_capture() {
    ltx_ctx* c = make_ctx();
    const hipStream_t s1 = (hipStream_t)0x10, other = (hipStream_t)0x20;
    CHECK(attention(c, 2970, 70, s1) && linear(c, 200, 256, 256, LTX_MODE_F32, s1), "%s", ltx_last_error(c));
    fake::capturing.insert(other);
    fake::log.clear();
    CHECK(attention(c, 2970, 2970, s1), "attention: %s", ltx_last_error(c));
    CHECK(launches("ltx_vt_pad") == 1, "%d paddings", launches("ltx_vt_pad"));
    CHECK(linear(c, 8000, 4096, 4096, LTX_MODE_F32, s1), "linear: %s", ltx_last_error(c));
    CHECK(launches("ltx_split3") == 1, "%d splits", launches("ltx_split3"));
    CHECK(!fake::broken_capture, "the other stream's capture is broken");
    CHECK(fake::thread_mode == hipStreamCaptureModeGlobal, "the thread's capture mode is changed");
}

// No memory for scratch: the calls run on the kernels that need none, and take
// the scratch again when there is memory.
static void scratch_memory() {
    ltx_ctx* c = make_ctx();
    const hipStream_t s1 = (hipStream_t)0x10;
    CHECK(attention(c, 2970, 70, s1), "%s", ltx_last_error(c));
    fake::limit = fake::in_use + (1 << 20);
    fake::log.clear();
    CHECK(attention(c, 2970, 2970, s1), "attention: %s", ltx_last_error(c));
    CHECK(launches("ltx_attn_f16_w8") == 1 && !launches("ltx_vt_pad"), "not the any-length kernel");
    CHECK(linear(c, 2000, 4096, 4096, LTX_MODE_F32, s1), "linear: %s", ltx_last_error(c));
    CHECK(launches("ltx_gemm_f32") == 1 && !launches("ltx_split3"), "not the f32 MFMA kernel");
    fake::limit = ~0ull;
    CHECK(attention(c, 2970, 2970, s1) && launches("ltx_vt_pad") == 1, "%s", ltx_last_error(c));
}

// Mode F32's planes stay below 512 MiB: larger operands go in passes of whole
// 128-row tiles, each on planes and partial sums inside the scratch, and
// together all of the rows with one split of K.
static void planes_bound(int M, int N, int K, bool noalloc) {
    ltx_ctx* c = make_ctx();
    fake::log.clear();
    CHECK(linear(c, M, N, K, LTX_MODE_F32, nullptr, noalloc), "%s", ltx_last_error(c));
    CHECK(c->op_scratch.buf.bytes <= (512u << 20), "%zu bytes kept", c->op_scratch.buf.bytes);
    size_t row = 0;
    const fake::Op* split = nullptr;
    int ks = 0;
    for (const fake::Op& o : fake::log) {
        if (o.name == "ltx_split3") {
            split = &o;
            CHECK(o.split.x == ptr(0) + row * K, "a pass starts elsewhere than at row %zu", row);
            for (uint16_t* p : {o.split.p0, o.split.p1, o.split.p2})
                CHECK(fake::inside(p, 2 * o.split.n), "planes of %zu values outside the scratch", o.split.n);
        }
        if (o.name.rfind("ltx_gemm_f3_", 0) == 0) {
            const LtxGemmArgs& g = o.f3.g;
            CHECK(split && g.a == split->split.p0 && o.f3.a2 == split->split.p2, "not the planes just split");
            CHECK((size_t)g.M * K == split->split.n && g.out == (char*)ptr(3) + row * N * 4, "not the rows just split");
            CHECK(!ks || g.ksplit == ks, "split of K %d, then %d", ks, g.ksplit);
            ks = g.ksplit;
            if (ks > 1)
                CHECK(g.part >= (const float*)((const char*)split->split.p2 + 2 * split->split.n) &&
                          fake::inside(g.part, (size_t)ks * g.M * N * 4),
                      "partial sums outside the scratch");
            row += g.M;
            CHECK(row == (size_t)M || g.M % 128 == 0, "a pass of %d rows", g.M);
            split = nullptr;
        }
    }
    CHECK(row == (size_t)M, "%zu of %d rows", row, M);
    std::printf("%d passes, %zu bytes\n", launches("ltx_split3"), c->op_scratch.buf.bytes);
}

// Mode F32 without allocations: eager calls follow each other, whatever their
// stream and context, and use none of the scratch that the 16-bit modes share;
// a captured call, whose replays may overlap anything, uses no scratch at all.
static void noalloc_f32() {
    ltx_ctx *c1 = make_ctx(), *c2 = make_ctx();
    const hipStream_t cap = (hipStream_t)0x30;
    int i = 0;
    scratch_order("ltx_split3", "ltx_gemm_f3_i8f16_store",
                  [&](hipStream_t st) { return linear(i++ % 2 ? c1 : c2, 1000, 4096, 512, LTX_MODE_F32, st, true); });
    uint64_t lo = ~0ull, hi = 0;
    for (const fake::Op& o : fake::log)
        if (o.name == "ltx_split3") lo = std::min(lo, (uint64_t)o.split.p0), hi = std::max(hi, (uint64_t)o.split.p2);
    const uint64_t s = (uint64_t)ltx::noalloc_scratch(0);
    CHECK(s && (hi < s || lo >= s + LTX_NOALLOC_SCRATCH_BYTES), "planes in the shared scratch");
    fake::capturing.insert(cap);
    fake::log.clear();
    CHECK(linear(c1, 1000, 4096, 512, LTX_MODE_F32, cap, true), "%s", ltx_last_error(c1));
    CHECK(launches("") == 1 && launches("ltx_gemm_f32") == 1, "%d launches", launches(""));
    for (const fake::Op& o : fake::log) CHECK(o.what == "launch", "%s in a capture", o.what.c_str());
}

// The stages of V at ragged token counts: addresses of the workspace, like all
// others. The first question after an eager forward may wait for it and fill them
// (allocating nothing, and beside a capture on another stream); from then on, and
// in a captured forward, they are filled between the GEMM that forms V and the
// end of the forward, and asking does nothing.
static void stage_v(int T, int S, int mode, bool captured) {
    ltx_ctx* c = make_ctx();
    ltx_block_weights w;
    fill(w, mode != LTX_MODE_BF16);
    w.f16_max = 1.0f;
    const hipStream_t st = (hipStream_t)0x10, other = (hipStream_t)0x20;
    void* first[2] = {};
    if (captured) {
        forward(c, w, T, S, mode, st);  // (sizes the workspace)
        fake::capturing.insert(st);
    }
    for (int pass = 0; pass < 2; pass++) {
        fake::log.clear();
        forward(c, w, T, S, mode, st);
        const std::vector<fake::Op> ops = fake::log;
        const bool asking = !captured && !pass;
        fake::capturing.insert(other);
        fake::log.clear();
        for (int i = 0; i < 2; i++) {
            const int n = i ? S : T;
            void* p = nullptr;
            uint64_t bytes = 0;
            CHECK(ltx_block_stage(c, i ? LTX_ST_V2 : LTX_ST_V1, &p, &bytes), "%s", ltx_last_error(c));
            for (const fake::Op& o : fake::log)
                CHECK(asking && (o.what == "sync" || o.what == "wait" || (o.name == "ltx_vt_unpad" && o.stream == c->side)),
                      "%s %s on asking for stage V%d", o.what.c_str(), o.name.c_str(), i + 1);
            CHECK(bytes == (uint64_t)n * LTX_D * 2, "%zu bytes", (size_t)bytes);
            CHECK((uint64_t)p >= (uint64_t)c->ws.p && (uint64_t)p + bytes <= (uint64_t)c->ws.p + c->ws.bytes,
                  "stage V%d outside the workspace", i + 1);
            if (!first[i]) first[i] = p;
            CHECK(p == first[i], "stage V%d moved", i + 1);
            // the attention over n keys reads V at v; p is v itself or filled from it
            const fake::Op *attn = nullptr, *copy = nullptr, *gemm = nullptr;
            for (const fake::Op& o : ops)
                if (o.name.rfind("ltx_attn", 0) == 0 && (!attn || i)) attn = &o;
            for (const fake::Op& o : ops) {
                if (o.name == "ltx_vt_unpad" && o.vt.y == p) copy = &o;
                if (o.gemm.out2 == attn->attn.vt && o.gemm.out2) gemm = &o;
            }
            CHECK(gemm, "no GEMM forms V%d", i + 1);
            CHECK(fake::before(*gemm, *attn), "the attention does not wait for V%d", i + 1);
            if (asking) {
                if (p != attn->attn.vt) {
                    int fills = 0;
                    for (const fake::Op& o : fake::log)
                        if (o.name == "ltx_vt_unpad" && o.vt.y == p) {
                            fills++;
                            CHECK(fake::before(*gemm, o), "stage V%d is filled before V is formed", i + 1);
                        }
                    CHECK(!copy && fills == 1 && fake::log.back().what == "sync", "stage V%d filled %d times", i + 1,
                          fills);
                }
            } else if (p != attn->attn.vt) {
                CHECK(copy && copy->vt.v == attn->attn.vt && copy->vt.n == n && copy->vt.ld == attn->attn.v_rs,
                      "nothing fills stage V%d", i + 1);
                CHECK(fake::before(*gemm, *copy), "stage V%d is filled before V is formed", i + 1);
                CHECK(fake::before(*copy, ops.back()), "the forward does not wait for stage V%d", i + 1);
            } else {
                CHECK(n == attn->attn.v_rs, "stage V%d has padded rows", i + 1);
            }
        }
        CHECK(!fake::broken_capture, "a capture is broken");
        fake::capturing.erase(other);
    }
}

// After one call of a shape, calls of that shape on the same stream allocate
// nothing, whatever the alignment of their operands: a program that warms up and
// then captures.
static void linear_warmed() {
    for (int mode : {LTX_MODE_F16, LTX_MODE_BF16}) {
        ltx_ctx* c = make_ctx();
        CHECK(linear(c, 300, 4096, 4096, mode, nullptr), "%s", ltx_last_error(c));
        const hipStream_t cap = (hipStream_t)0x30;
        fake::capturing.insert(cap);
        CHECK(ltx_op_linear_q8(c, ptr(0), (const int8_t*)ptr(1) + 4, ptr(2), 1, nullptr, ptr(3), 0, 300, 4096, 4096, 0, mode,
                               cap),
              "%s", ltx_last_error(c));
        CHECK(!fake::broken_capture, "the capture is broken");
        fake::capturing.clear();
    }
}

// A mode F32 forward whose planes find no memory, or no room in a workspace that a
// graph holds, runs on the f32 MFMA kernel; with room again, on the planes.
static void f32_workspace() {
    for (bool pinned : {false, true}) {
        ltx_ctx* c = make_ctx();
        ltx_block_weights w;
        fill(w, true);
        const int T = 20000;
        // what the forward took before its GEMMs had planes: 13 tensors of T x 4,096,
        // the FFN's hidden values, the gate logits and the context's, with some air
        const uint64_t plain = (uint64_t)T * (13 * LTX_D + LTX_FF + 64) * 4 + (64 << 20);
        if (pinned) {
            c->ws.alloc(plain);
            c->ws_pins = 1;
        } else {
            fake::limit = fake::in_use + plain;
        }
        fake::log.clear();
        forward(c, w, T, 128, LTX_MODE_F32);
        CHECK(!launches("ltx_split3") && launches("ltx_gemm_f32"), "planes without room");
        fake::limit = ~0ull;
        c->ws_pins = 0;
        fake::log.clear();
        forward(c, w, T, 128, LTX_MODE_F32);
        CHECK(launches("ltx_split3") && !launches("ltx_gemm_f32"), "no planes with room");
    }
}

int main(int argc, char** argv) {
    const std::string cmd = argc > 1 ? argv[1] : "";
    auto arg = [&](int i) { return argc > i ? std::atoi(argv[i]) : 0; };
    if (cmd == "f32_planes")
        f32_planes(arg(2), arg(3));
    else if (cmd == "scratch_order_planes") {
        ltx_ctx* c = make_ctx();
        scratch_order("ltx_split3", "ltx_gemm_f3_i8f16_store",
                      [&](hipStream_t st) { return linear(c, 1000, 4096, 512, LTX_MODE_F32, st); });
    } else if (cmd == "scratch_order_vt") {
        ltx_ctx* c = make_ctx();
        scratch_order("ltx_vt_pad", "ltx_attn_f16_pp_uq", [&](hipStream_t st) { return attention(c, 2970, 2970, st); });
    } else if (cmd == "scratch_capture")
        scratch_capture();
    else if (cmd == "scratch_memory")
        scratch_memory();
    else if (cmd == "planes_bound")
        planes_bound(arg(2), arg(3), arg(4), false);
    else if (cmd == "noalloc_f32")
        noalloc_f32();
    else if (cmd == "planes_bound_noalloc")
        planes_bound(arg(2), arg(3), arg(4), true);
    else if (cmd == "attn_misaligned") {
        ltx_ctx* c = make_ctx();
        for (size_t off : {2, 8}) {
            fake::log.clear();
            CHECK(attention(c, 2970, 2970, nullptr, off), "%s", ltx_last_error(c));
            CHECK(launches("") == 1 && launches("ltx_attn_f16_w8") == 1, "K %zu bytes past alignment: %s", off,
                  fake::log[0].name.c_str());
        }
    } else if (cmd == "linear_warmed")
        linear_warmed();
    else if (cmd == "f32_workspace")
        f32_workspace();
    else if (cmd == "stage_v")
        stage_v(arg(2), arg(3), arg(4), arg(5));
    else if (cmd == "attn_padded") {  // prints whether V^T is padded, for pairs lq lkv
        ltx_ctx* c = make_ctx();
        for (int i = 2; i + 1 < argc; i += 2) {
            fake::log.clear();
            CHECK(attention(c, arg(i), arg(i + 1), nullptr), "%s", ltx_last_error(c));
            std::printf("%d ", launches("ltx_vt_pad"));
        }
    } else if (cmd == "tile_rows") {  // prints whether tiles of 192 rows run, for quadruples M N K scale_f16
        ltx_ctx* c = make_ctx();
        for (int i = 2; i + 3 < argc; i += 4) {
            fake::log.clear();
            CHECK(linear(c, arg(i), arg(i + 1), arg(i + 2), LTX_MODE_BF16, nullptr, false, arg(i + 3)), "%s",
                  ltx_last_error(c));
            int h = 0;
            for (const fake::Op& o : fake::log) h += o.name.find("_h192") != std::string::npos;
            std::printf("%d ", h);
        }
    } else
        CHECK(false, "unknown command %s", cmd.c_str());
    std::printf("ok\n");
    std::fflush(stdout);
    std::_Exit(0);  // (the library's own teardown belongs to the real runtime)
}
