// The host half of the library (ft_runtime.cpp, ft_step.cpp) over a HIP runtime made of host memory, in which an
// allocation can be refused: what a program on a GPU cannot bring about without filling the machine. "Device" memory
// is malloc'd and tracked, so a kernel's reads can be checked against what is live. Prints one line per failed check.
#include "ft_common.h"

#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
#include <set>

struct ft_segment {
    float *w, *g, *m, *v;
    uint32_t n;
};

static std::map<char*, size_t> g_device;
static std::set<void*> g_pinned;
static hipError_t g_last = hipSuccess;
static bool g_refuse_pinned = false, g_refuse_device = false;
static int g_device_grants = -1;  // device allocations still granted, -1: all
static long g_news_left = -1;   // operator new throws when this reaches 0
static int g_failures = 0, g_copies = 0;

static void expect(bool ok, const char* what) {
    if (ok) return;
    printf("FAILED: %s (%s)\n", what, ft_last_error());
    g_failures++;
}

static bool live(const void* p, size_t bytes) {
    auto it = g_device.upper_bound((char*)p);
    if (it == g_device.begin()) return false;
    --it;
    return (char*)p + bytes <= it->first + it->second;
}

void* operator new(size_t n) {
    if (g_news_left >= 0 && g_news_left-- == 0) throw std::bad_alloc();
    void* p = malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

static hipError_t fail(hipError_t e) { return g_last = e; }   // stays until hipGetLastError takes it

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    if (g_refuse_device || g_device_grants == 0) return fail(hipErrorOutOfMemory);
    if (g_device_grants > 0) g_device_grants--;
    *p = malloc(n);
    const long news = g_news_left;
    g_news_left = -1;   // the bookkeeping here is not the library's
    g_device[(char*)*p] = n;
    g_news_left = news;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (p && !g_device.erase((char*)p)) return fail(hipErrorInvalidValue);
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (g_refuse_pinned) return fail(hipErrorOutOfMemory);
    *p = malloc(n);
    const long news = g_news_left;
    g_news_left = -1;
    g_pinned.insert(*p);
    g_news_left = news;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    g_pinned.erase(p);
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) {
    if (k == hipMemcpyDeviceToHost) g_copies++;
    if (!live(k == hipMemcpyDeviceToHost ? s : d, n)) return fail(hipErrorInvalidValue);
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    memset(p, 0, sizeof(*p));
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = nullptr, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError(void) {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "refused"; }

// Numbers that differ from buffer to buffer in place of zeros, so that a gradient read from the wrong place shows.
int ft_zero(ft_context*, void* p, size_t bytes) {
    static float next = 1.0f;
    for (size_t i = 0; i < bytes / 4; i++) ((float*)p)[i] = next++;
    return FT_OK;
}
}

int ft_internal_noalloc_init(int) { return FT_OK; }

int ft_internal_multi_copy(ft_context*, const ft_segment* segs, size_t nseg) {
    if (!live(segs, nseg * sizeof(ft_segment))) {
        expect(false, "a kernel reads a segment table that is not there");
        return FT_OK;
    }
    for (size_t i = 0; i < nseg; i++) {
        if (live(segs[i].g, segs[i].n * 4)) memcpy(segs[i].w, segs[i].g, segs[i].n * 4);
        else expect(false, "a kernel reads memory that was freed");
    }
    FT_LAUNCH_CHECK();
    return FT_OK;
}

static ft_context* ctx;
static ft_model* model;
static const char* kLinear[2] = {"model.layers.0.self_attn.q_proj", "model.layers.0.mlp.down_proj"};

static int set_lora(const char* name, size_t in, size_t out, size_t rank) {
    std::vector<float> a(in * rank, 0.5f), b(rank * out, 0.25f);
    return ft_model_set_lora(model, name, a.data(), b.data(), rank, 8.0f);
}

// All gradients at once against one read each.
static void check_grads(const char* what, size_t want_total) {
    size_t count = 0, total = 0, numel = 0;
    expect(ft_model_param_count(model, &count) == FT_OK, what);
    std::vector<float> each;
    for (size_t i = 0; i < count; i++) {
        expect(ft_model_param_info(model, i, nullptr, &numel) == FT_OK, what);
        std::vector<float> one(numel);
        expect(ft_model_read_grad(model, i, one.data()) == FT_OK, what);
        each.insert(each.end(), one.begin(), one.end());
        total += numel;
    }
    expect(total == want_total, what);
    std::vector<float> all(total + 1, -1.0f);
    expect(ft_model_read_grads(model, all.data()) == FT_OK, what);
    expect(memcmp(all.data(), each.data(), total * 4) == 0 && all[total] == -1.0f, what);
    expect(hipGetLastError() == hipSuccess, "an error is left for the next launch check");
}

int main(int argc, char** argv) {
    const std::string scenario = argc > 1 ? argv[1] : "";
    ft_model_config cfg{};
    cfg.vocab_size = 64;
    cfg.hidden_size = 128;
    cfg.intermediate_size = 2048;
    cfg.num_hidden_layers = 1;
    cfg.num_attention_heads = 2;
    cfg.num_key_value_heads = 2;
    expect(ft_context_create(0, &ctx) == FT_OK, "context");
    expect(ft_model_create(ctx, &cfg, &model) == FT_OK, "model");
    // 4 tensors; 32 x 2048 values are 16 pieces of 4096
    expect(set_lora(kLinear[0], 128, 128, 4) == FT_OK && set_lora(kLinear[1], 2048, 128, 32) == FT_OK, "adapters");
    const size_t total = 4 * (128 + 128) + 32 * (2048 + 128);
    if (scenario == "whole") {
        check_grads("gathered", total);
        check_grads("gathered again", total);
        expect(set_lora(kLinear[0], 128, 128, 8) == FT_OK, "another rank");
        check_grads("after another rank", total + 4 * (128 + 128));
    } else if (scenario == "no_host_memory_for_the_list") {
        // each of the call's allocations on the host fails in turn; the call after it succeeds
        std::vector<float> all(total);
        size_t count = 0;
        expect(ft_model_param_count(model, &count) == FT_OK, "count");
        int refused = 0;
        for (long k = 0; k < 64; k++) {
            g_news_left = k;
            const int rc = ft_model_read_grads(model, all.data());
            g_news_left = -1;
            if (rc == FT_OK) break;
            refused++;
        }
        expect(refused > 0, "no allocation was refused");
        check_grads("after the refusals", total);
        expect(g_pinned.size() <= 1, "pinned arrays were lost");
    } else if (scenario == "no_pinned_memory" || scenario == "no_device_memory") {
        // the gradients still come, tensor by tensor, and all at once again when there is memory
        g_refuse_pinned = scenario == "no_pinned_memory";
        g_refuse_device = !g_refuse_pinned;
        check_grads("refused", total);
        expect(g_copies == 8, "one copy per tensor, twice");
        g_refuse_pinned = g_refuse_device = false;
        check_grads("with memory again", total);
        expect(g_copies == 12, "gathered");
    } else if (scenario == "no_memory_for_another_rank") {
        // each allocation of the new factors is refused in turn (ft_alloc asks twice): the adapter stays what it was
        check_grads("before", total);
        for (int granted = 0; granted < 4; granted++) {
            g_device_grants = granted;
            expect(set_lora(kLinear[0], 128, 128, 8) == FT_ERR_OOM, "refused");
            g_device_grants = -1;
            expect(ft_pool_trim(ctx) == FT_OK, "trim");
            check_grads("after a refusal", total);
        }
        expect(set_lora(kLinear[0], 128, 128, 8) == FT_OK, "another rank");
        check_grads("after another rank", total + 4 * (128 + 128));
    } else {
        printf("no such scenario\n");
        return 2;
    }
    ft_model_destroy(model);
    expect(g_pinned.empty(), "pinned memory outlives the model");
    ft_context_destroy(ctx);
    // (a buffer that ft_alloc cannot note down for want of host memory is the process's until it ends)
    if (scenario != "no_host_memory_for_the_list") expect(g_device.empty(), "device memory outlives the context");
    if (!g_failures) printf("ok\n");
    return g_failures ? 1 : 0;
}
