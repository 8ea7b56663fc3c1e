// What the library's host code does when something goes wrong, on a runtime that only pretends (fake_hip.h): one case per
// run, named on the command line, with a GGUF file of a small model where one is needed.  Prints what fails; 0: nothing did.
// And which kernels a call enqueues ("routes").
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <string>
#include <utility>
#include <vector>

#include "../../include/wick_gguf.h"
#include "../../include/wick_rocm.h"
#include "../../include/wick_rocm_lfm2.h"
#include "fake_hip.h"

namespace {

int failures = 0;
std::atomic<long> memory_left{-1};  // allocations until the one that fails (in the library and in libstdc++ alike); < 0: none does

#define CHECK(cond, ...)                                   \
    do {                                                   \
        if (!(cond)) {                                     \
            failures++;                                    \
            std::printf("line %d: %s: ", __LINE__, #cond); \
            std::printf(__VA_ARGS__);                      \
            std::printf("\n");                             \
        }                                                  \
    } while (0)

struct Ctx {
    wick_rocm_ctx* c = nullptr;
    Ctx() {
        if (wick_rocm_ctx_create(0, &c) != WICK_ROCM_OK) std::abort();
    }
    ~Ctx() { wick_rocm_ctx_destroy(c); }
    operator wick_rocm_ctx*() const { return c; }
};

// wick_rocm_upload / wick_rocm_download of a range that does not lie in its allocation, or of no device memory at all.
void ranges() {
    Ctx ctx;
    constexpr size_t kSize = 8192;
    void* d = nullptr;
    CHECK(wick_rocm_buffer_alloc(ctx, kSize, &d) == WICK_ROCM_OK, "alloc");
    char* const dev = static_cast<char*>(d);
    std::vector<char> host(16u << 20, 1), back(16u << 20);
    for (size_t off : {0, 16, 4096})
        for (size_t n : {size_t{8208}, size_t{65536}, size_t{5u << 20}}) {  // past the end by one piece; one slot; many slots
            CHECK(wick_rocm_upload(ctx, dev + off, host.data(), n) < 0, "%zu bytes at %zu", n, off);
            CHECK(wick_rocm_download(ctx, back.data(), dev + off, n) < 0, "%zu bytes at %zu", n, off);
        }
    CHECK(fake_hip::pending() == 0, "%zu", fake_hip::pending());
    // not device memory: whatever the runtime makes of it, no kernel of ours gets the address
    const long before = fake_hip::launches;
    alignas(16) static char plain[4096];
    wick_rocm_upload(ctx, plain, host.data(), sizeof plain);
    wick_rocm_download(ctx, back.data(), plain, sizeof plain);
    CHECK(fake_hip::launches == before, "%ld launches", fake_hip::launches - before);
    CHECK(fake_hip::out_of_range == 0, "%ld accesses", fake_hip::out_of_range);
    // and a range inside, up to its last byte, is copied
    for (size_t off : {0, 16, 4096}) {
        for (size_t i = 0; i < kSize; i++) host[i] = (char)(i * 7 + off);
        CHECK(wick_rocm_upload(ctx, dev + off, host.data(), kSize - off) == WICK_ROCM_OK, "at %zu", off);
        CHECK(wick_rocm_download(ctx, back.data(), dev + off, kSize - off) == WICK_ROCM_OK, "at %zu", off);
        CHECK(std::memcmp(host.data(), back.data(), kSize - off) == 0, "at %zu", off);
    }
    wick_rocm_buffer_free(ctx, d);
}

struct Gguf {
    wick_gguf* g = nullptr;
    explicit Gguf(const char* path) {
        if (wick_gguf_open(path, &g) != 0) std::abort();
    }
    ~Gguf() { wick_gguf_close(g); }
};

struct Model {
    wick_rocm_ctx* ctx;
    wick_rocm_lfm2* m = nullptr;
    Model(wick_rocm_ctx* c, const char* path, uint32_t context = 64) : ctx(c) {
        Gguf g(path);
        if (wick_rocm_lfm2_load(c, g.g, context, &m) != WICK_ROCM_OK) std::abort();
    }
    ~Model() { wick_rocm_lfm2_free(ctx, m); }
    operator wick_rocm_lfm2*() const { return m; }
};

// A copy of several pieces whose second, third, .. piece fails: nothing may be on its way in the staging memory (or in the
// caller's) when the call returns, since the next copy fills it again.
void copies(const char* path) {
    Ctx ctx;
    Model m(ctx, path);
    constexpr uint32_t kPos = 40;
    std::vector<unsigned char> in(wick_rocm_lfm2_state_bytes(m, kPos)), out(in.size());
    for (size_t i = 0; i < in.size(); i++) in[i] = (unsigned char)(i * 13 + 1);
    const auto restore = [&] { return wick_rocm_lfm2_restore_state(ctx, m, kPos, in.data(), in.size()); };
    const auto snapshot = [&] { return wick_rocm_lfm2_snapshot_state(ctx, m, kPos, out.data(), out.size()); };
    for (bool pinned : {true, false}) {  // without pinned memory the pieces are the runtime's copies, of the caller's memory
        if (!pinned) {
            fake_hip::fail_pinned(true);
            wick_rocm_ctx* other = nullptr;  // (this context has its staging memory; the model's copies on another one)
            CHECK(wick_rocm_ctx_create(0, &other) == WICK_ROCM_OK, "context");
            std::swap(ctx.c, other);
            wick_rocm_ctx_destroy(other);
            m.ctx = ctx;
        }
        for (long n = 1; n <= 6; n++)  // two conv states, two layers' keys and values
            for (bool up : {true, false}) {
                (pinned ? fake_hip::fail_launch : fake_hip::fail_copy)(n);
                CHECK((up ? restore() : snapshot()) < 0, "piece %ld, up %d, pinned %d", n, up, pinned);
                CHECK(fake_hip::pending() == 0, "%zu on their way behind piece %ld, up %d, pinned %d", fake_hip::pending(), n, up, pinned);
            }
        CHECK(restore() == WICK_ROCM_OK && snapshot() == WICK_ROCM_OK, "pinned %d", pinned);
        CHECK(in == out, "pinned %d", pinned);
    }
    fake_hip::fail_pinned(false);
    // and one of many slots, dealt out to several threads
    void* d = nullptr;
    std::vector<char> host(27u << 20, 3);
    CHECK(wick_rocm_buffer_alloc(ctx, host.size(), &d) == WICK_ROCM_OK, "alloc");
    for (long n : {1, 2, 5, 14}) {
        fake_hip::fail_launch(n);
        CHECK(wick_rocm_upload(ctx, d, host.data(), host.size()) < 0 && fake_hip::pending() == 0, "up, chunk %ld", n);
        fake_hip::fail_launch(n);
        CHECK(wick_rocm_download(ctx, host.data(), d, host.size()) < 0 && fake_hip::pending() == 0, "down, chunk %ld", n);
    }
    wick_rocm_buffer_free(ctx, d);
}

// A prompt whose n-th launch fails: its first kernel reads the tokens from the model's pinned copy, which the next prompt
// overwrites, so nothing may be pending when the call returns.
void prompts(const char* path) {
    Ctx ctx;
    Model m(ctx, path);
    uint32_t tokens[20];
    for (uint32_t i = 0; i < 20; i++) tokens[i] = i;
    const auto prompt = [&] { return wick_rocm_lfm2_forward_prefill(ctx, m, tokens, 20, 0, nullptr); };
    CHECK(prompt() == WICK_ROCM_OK, "prompt");
    const long before = fake_hip::launches;
    CHECK(prompt() == WICK_ROCM_OK, "prompt");
    const long launches = fake_hip::launches - before;
    CHECK(launches > 20, "%ld launches", launches);
    for (long n = 1; n <= launches; n++) {
        fake_hip::fail_launch(n);
        CHECK(prompt() < 0, "launch %ld", n);
        CHECK(fake_hip::pending() == 0, "%zu pending behind launch %ld", fake_hip::pending(), n);
        wick_rocm_sync(ctx);
    }
    CHECK(prompt() == WICK_ROCM_OK, "prompt");
}

// Every allocation of every call fails once: the call answers with an error (or does without), nothing is thrown through the C
// entry point, nothing is left on the device, and the same call then works.
template <typename F>
void every_allocation(const char* what, F&& call) {
    for (long n = 0;; n++) {
        if (n > 100000) {
            CHECK(false, "%s", what);
            return;
        }
        const size_t before = fake_hip::allocations();
        bool threw = false;
        int rc = 0;
        memory_left = n;
        try {
            rc = call();
        } catch (...) {
            threw = true;
        }
        const bool failed = memory_left < 0;
        memory_left = -1;
        CHECK(!threw, "%s: an exception at allocation %ld", what, n);
        CHECK(fake_hip::pending() == 0 && (rc == 0 || fake_hip::allocations() == before), "%s: allocation %ld", what, n);
        if (threw) return;  // (its locks may be held)
        if (!failed) {
            CHECK(rc == 0 && n > 0, "%s: %d after %ld allocations", what, rc, n);
            return;
        }
    }
}

void memory(const char* path) {
    std::vector<char> host(27u << 20, 3);
    std::vector<unsigned char> file(1u << 22);
    FILE* f = std::fopen(path, "rb");
    file.resize(std::fread(file.data(), 1, file.size(), f));
    std::fclose(f);
    every_allocation("context", [] {
        wick_rocm_ctx* c = nullptr;
        const int rc = wick_rocm_ctx_create(0, &c);
        wick_rocm_ctx_destroy(c);
        return rc;
    });
    Ctx ctx;
    Gguf gguf(path);
    const auto opened = [](int rc, wick_gguf* g) {
        wick_gguf_close(g);
        return rc;
    };
    every_allocation("gguf file", [&] {
        wick_gguf* g = nullptr;
        const int rc = wick_gguf_open(path, &g);
        return opened(rc, g);
    });
    every_allocation("gguf bytes", [&] {
        wick_gguf* g = nullptr;
        const int rc = wick_gguf_from_bytes(file.data(), file.size(), &g);
        return opened(rc, g);
    });
    every_allocation("load", [&] {
        wick_rocm_lfm2* m = nullptr;
        const int rc = wick_rocm_lfm2_load(ctx, gguf.g, 64, &m);
        if (m) wick_rocm_lfm2_free(ctx, m);
        return rc;
    });
    every_allocation("weight", [&] {
        wick_rocm_weight* w = nullptr;
        const int rc = wick_rocm_weight_from_gguf(ctx, gguf.g, "blk.0.ffn_down.weight", &w);
        if (w) wick_rocm_weight_free(ctx, w);
        return rc;
    });
    void* d = nullptr;
    CHECK(wick_rocm_buffer_alloc(ctx, host.size(), &d) == WICK_ROCM_OK, "alloc");
    every_allocation("upload", [&] { return wick_rocm_upload(ctx, d, host.data(), host.size()); });
    every_allocation("refused upload", [&] { return wick_rocm_upload(ctx, d, host.data(), host.size() + 16) < 0 ? 0 : -1; });
    Model m(ctx, path);
    constexpr uint32_t kPos = 40;
    std::vector<unsigned char> state(wick_rocm_lfm2_state_bytes(m, kPos), 1);
    uint32_t tokens[20] = {}, picks[4];
    every_allocation("restore", [&] { return wick_rocm_lfm2_restore_state(ctx, m, kPos, state.data(), state.size()); });
    every_allocation("snapshot", [&] { return wick_rocm_lfm2_snapshot_state(ctx, m, kPos, state.data(), state.size()); });
    every_allocation("shift", [&] { return wick_rocm_lfm2_shift_kv(ctx, m, kPos, 8, 10); });
    every_allocation("greedy", [&] {
        const int rc = wick_rocm_lfm2_generate_greedy(ctx, m, 1, 5, 4, picks);
        if (rc) wick_rocm_sync(ctx);  // (steps may be under way: they touch the model's own memory only)
        return rc;
    });
    Model fresh(ctx, path);  // (its prompt buffers are still to be made)
    memory_left = 0;
    CHECK(wick_rocm_lfm2_forward_prefill(ctx, fresh, tokens, 20, 0, nullptr) < 0, "prompt");
    memory_left = -1;
    CHECK(wick_rocm_lfm2_forward_prefill(ctx, fresh, tokens, 20, 0, nullptr) == WICK_ROCM_OK, "prompt");
    CHECK(wick_rocm_lfm2_forward_prefill(ctx, m, tokens, 20, 0, nullptr) == WICK_ROCM_OK, "prompt");
    every_allocation("timing", [&] {
        double ms[4];
        uint64_t launches[4];
        if (int rc = wick_rocm_kernel_timing_begin(ctx)) return rc;
        const int rc = wick_rocm_lfm2_forward_prefill(ctx, m, tokens, 20, 0, nullptr), end = wick_rocm_kernel_timing_end(ctx, ms, launches, 4);
        return rc ? rc : end;
    });
    wick_rocm_buffer_free(ctx, d);
}

// A model on the second GPU, called from a thread whose current one is the first: every launch of every call goes to the model's.
void devices(const char* path) {
    wick_rocm_ctx *first = nullptr, *ctx = nullptr;
    CHECK(wick_rocm_ctx_create(1, &ctx) == WICK_ROCM_OK && wick_rocm_ctx_create(0, &first) == WICK_ROCM_OK, "contexts");
    Gguf g(path);
    wick_rocm_lfm2* m = nullptr;
    CHECK(wick_rocm_lfm2_load(ctx, g.g, 64, &m) == WICK_ROCM_OK, "load");
    wick_rocm_lfm2_config cfg;
    wick_rocm_lfm2_get_config(m, &cfg);
    std::vector<float> logits(cfg.vocab_size), frame(3 * cfg.hidden_size);
    std::vector<unsigned char> state(wick_rocm_lfm2_state_bytes(m, 20));
    uint32_t tokens[20] = {}, picks[4], consumed;
    const auto each = [&](const char* what, auto&& call) {
        wick_rocm_sync(first);  // makes the first GPU current, as work of the caller's on it does
        fake_hip::other_device = 0;
        const int rc = call();
        CHECK(rc == WICK_ROCM_OK && fake_hip::other_device == 0, "%s: %d, %ld launches beside the model's GPU", what, rc, fake_hip::other_device);
    };
    for (int replay : {0, 1}) {
        wick_rocm_lfm2_set_graph_replay(m, replay);
        each("reset", [&] { return wick_rocm_lfm2_reset(ctx, m); });
        each("step", [&] { return wick_rocm_lfm2_forward(ctx, m, 1, 0, logits.data()); });
        each("prompt", [&] { return wick_rocm_lfm2_forward_prefill(ctx, m, tokens, 20, 0, logits.data()); });
        each("short prompt", [&] { return wick_rocm_lfm2_forward_prefill(ctx, m, tokens, 2, 0, logits.data()); });
        each("chunked prompt", [&] { return wick_rocm_lfm2_forward_prefill_chunked(ctx, m, tokens, 20, 0, 7, nullptr, &consumed, logits.data()); });
        each("embedded prompt", [&] { return wick_rocm_lfm2_forward_prefill_from_embeddings(ctx, m, frame.data(), 3, 0, logits.data()); });
        each("short embedded prompt", [&] { return wick_rocm_lfm2_forward_prefill_from_embeddings(ctx, m, frame.data(), 1, 0, logits.data()); });
        each("greedy", [&] { return wick_rocm_lfm2_generate_greedy(ctx, m, 1, 5, 4, picks); });
        each("greedy step", [&] { return wick_rocm_lfm2_forward_greedy(ctx, m, 1, 5, picks); });
        each("embedded step", [&] { return wick_rocm_lfm2_forward_from_embedding(ctx, m, frame.data(), 5, logits.data()); });
        each("hidden state", [&] { return wick_rocm_lfm2_forward_embedding(ctx, m, 1, 5, frame.data()); });
        each("hidden state of a frame", [&] { return wick_rocm_lfm2_forward_hidden_from_embedding(ctx, m, frame.data(), 5, frame.data()); });
        each("snapshot", [&] { return wick_rocm_lfm2_snapshot_state(ctx, m, 20, state.data(), state.size()); });
        each("restore", [&] { return wick_rocm_lfm2_restore_state(ctx, m, 20, state.data(), state.size()); });
        each("shift in place", [&] { return wick_rocm_lfm2_shift_kv(ctx, m, 20, 2, 6); });
        each("staged shift", [&] { return wick_rocm_lfm2_shift_kv(ctx, m, 40, 2, 1); });
    }
    wick_rocm_lfm2_free(ctx, m);
    wick_rocm_ctx_destroy(ctx), wick_rocm_ctx_destroy(first);
}

// The kernels of each call, a line a kernel behind a line with the call itself: "norm rows dim", "gemm m n k splits" (splits: most shares of K),
// "residual m n k", "gate_up m n k", "prompt file n".
void routes(int count, char** calls) {
    Ctx ctx;
    void* d = nullptr;  // (no kernel runs: one buffer is every operand)
    CHECK(wick_rocm_buffer_alloc(ctx, 4096, &d) == WICK_ROCM_OK, "alloc");
    const auto f = static_cast<float*>(d);
    const auto q = static_cast<int8_t*>(d);
    for (int i = 0; i < count; i++) {
        char kind[16] = "", path[512] = "";
        unsigned a[4] = {};
        int rc = -1;
        const auto weight = [&](uint32_t m, uint32_t k) {
            wick_rocm_weight* w = nullptr;
            const std::vector<char> blocks((size_t)m * k / 32 * 18);
            CHECK(wick_rocm_weight_upload(ctx, blocks.data(), blocks.size(), 2, m, k, &w) == WICK_ROCM_OK, "%s: weight", calls[i]);
            fake_hip::kernels();
            return w;
        };
        if (std::sscanf(calls[i], "prompt %511s %u", path, a) == 2) {
            Model m(ctx, path, a[0] > 64 ? a[0] : 64);
            const std::vector<uint32_t> tokens(a[0]);
            fake_hip::kernels();
            fake_hip::out_of_range = 0;  // (of the calls below: their buffer is no size)
            rc = wick_rocm_lfm2_forward_prefill(ctx, m, tokens.data(), a[0], 0, nullptr);
            CHECK(fake_hip::out_of_range == 0, "%s: %ld outputs", calls[i], fake_hip::out_of_range);
        } else if (std::sscanf(calls[i], "%15s %u %u %u %u", kind, a, a + 1, a + 2, a + 3) >= 3) {
            if (!std::strcmp(kind, "norm")) {
                rc = wick_rocm_rmsnorm_quantize_q8_0(ctx, f, f, a[0], a[1], a[1], 1e-5f, q, f);
            } else {
                wick_rocm_weight *const w = weight(a[0], a[2]), *const up = weight(a[0], a[2]);
                wick_rocm_set_gemm_max_k_splits(ctx, a[3]);
                if (!std::strcmp(kind, "gemm")) rc = wick_rocm_gemm_q8(ctx, w, q, f, a[1], f, a[0], WICK_ROCM_LAYOUT_TOKEN_MAJOR, 0);
                if (!std::strcmp(kind, "residual")) rc = wick_rocm_gemm_q8_residual_rmsnorm_quantize(ctx, w, q, f, a[1], f, a[0], f, 1e-5f, q, f);
                if (!std::strcmp(kind, "gate_up")) rc = wick_rocm_ffn_gate_up_silu_quantize_q8(ctx, w, up, q, f, a[1], q, f);
                wick_rocm_weight_free(ctx, w), wick_rocm_weight_free(ctx, up);
            }
        }
        CHECK(rc == WICK_ROCM_OK, "%s: %d", calls[i], rc);
        std::printf("%s\n", calls[i]);
        for (const std::string& name : fake_hip::kernels()) std::printf("\t%s\n", name.c_str());
    }
    wick_rocm_buffer_free(ctx, d);
}

}  // namespace

void* operator new(size_t n) {
    if (fake_hip::inside == 0 && memory_left >= 0 && memory_left-- == 0) throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void* operator new(size_t n, const std::nothrow_t&) noexcept {
    try {
        return operator new(n);
    } catch (...) {
        return nullptr;
    }
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

int main(int argc, char** argv) {
    const char* name = argc > 1 ? argv[1] : "";
    if (!std::strcmp(name, "ranges")) ranges();
    else if (!std::strcmp(name, "copies") && argc > 2) copies(argv[2]);
    else if (!std::strcmp(name, "prompts") && argc > 2) prompts(argv[2]);
    else if (!std::strcmp(name, "memory") && argc > 2) memory(argv[2]);
    else if (!std::strcmp(name, "devices") && argc > 2) devices(argv[2]);
    else if (!std::strcmp(name, "routes")) routes(argc - 2, argv + 2);
    else CHECK(false, "no case '%s'", name);
    return failures ? 1 : 0;
}
