// What the host code enqueues and allocates, on the CPU: the library's host source over stand-ins for the HIP runtime that record
// launches (kernel, grid, arguments) and allocations.  Device pointers are numbers here; nothing follows them.
//
//   host_routes [check]     prints "ok" or what does not hold; exit status 0 or 1
#define GLLMQ_EMBED(NAME) extern "C" const unsigned char gllmq_co_##NAME[1] = { 0 };
#include "../../gllm_amd/csrc/gllmq_host.cpp"

#include <array>
#include <functional>
#include <map>
#include <set>

extern "C" int gq_noalloc_init(gllmq_ctx *, int) { return GLLMQ_OK; }

namespace fake {

struct Launch {
    std::string kernel;
    uint32_t grid;
    std::vector<uint8_t> args;
    gq::MmfwParams wide() const
    {
        gq::MmfwParams P;
        if (args.size() != sizeof P) abort();
        std::memcpy(static_cast<void *>(&P), args.data(), sizeof P);
        return P;
    }
};

std::set<std::string> names;
std::vector<Launch> launches;
std::map<void *, size_t> live; // device allocations
size_t allocations = 0, frees = 0;
uintptr_t next_address = uintptr_t(1) << 40;
bool capturing = false;
size_t refuse_from = SIZE_MAX; // allocations of as many bytes are refused

hipError_t record(hipFunction_t f, uint32_t grid, void **extra)
{
    size_t size = 0;
    const uint8_t *args = nullptr;
    for (int i = 0; extra[i] != HIP_LAUNCH_PARAM_END; i += 2) {
        if (extra[i] == HIP_LAUNCH_PARAM_BUFFER_POINTER) args = static_cast<const uint8_t *>(extra[i + 1]);
        if (extra[i] == HIP_LAUNCH_PARAM_BUFFER_SIZE) size = *static_cast<const size_t *>(extra[i + 1]);
    }
    launches.push_back({ *reinterpret_cast<const std::string *>(f), grid, std::vector<uint8_t>(args, args + size) });
    return hipSuccess;
}

} // namespace fake

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) // (the header's macro gives it its versioned name)
{
    std::memset(static_cast<void *>(p), 0, sizeof *p);
    p->multiProcessorCount = 256;
    std::strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t size)
{
    if (size >= fake::refuse_from) return hipErrorOutOfMemory;
    *p = reinterpret_cast<void *>(fake::next_address);
    fake::next_address += (size + 4095) / 4096 * 4096;
    fake::live[*p] = size;
    ++fake::allocations;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    if (p && !fake::live.erase(p)) abort();
    fake::frees += p != nullptr;
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t size, unsigned)
{
    *p = std::calloc(1, size);
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemset(void *, int, size_t) { return hipSuccess; }
hipError_t hipMemcpy(void *, const void *, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *, unsigned) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *, unsigned) { return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s)
{
    *s = fake::capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipModuleLoadData(hipModule_t *m, const void *)
{
    static int any;
    *m = reinterpret_cast<hipModule_t>(&any);
    return hipSuccess;
}
hipError_t hipModuleUnload(hipModule_t) { return hipSuccess; }
hipError_t hipModuleGetFunction(hipFunction_t *f, hipModule_t, const char *name)
{
    *f = reinterpret_cast<hipFunction_t>(const_cast<std::string *>(&*fake::names.insert(name).first));
    return hipSuccess;
}
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned gx, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, hipStream_t, void **, void **extra)
{
    return fake::record(f, gx, extra);
}
hipError_t hipExtModuleLaunchKernel(hipFunction_t f, uint32_t gx, uint32_t, uint32_t, uint32_t bx, uint32_t, uint32_t, size_t, hipStream_t, void **, void **extra,
                                    hipEvent_t, hipEvent_t, uint32_t)
{
    return fake::record(f, gx / bx, extra);
}
}

namespace {

int failures = 0;
#define EXPECT(what, ...)                                   \
    do {                                                    \
        if (!(what) && ++failures <= 10) {                  \
            std::printf("%s:%d: " #what ": ", __func__, __LINE__); \
            std::printf(__VA_ARGS__);                       \
            std::printf("\n");                              \
        }                                                   \
    } while (0)

struct Context {
    gllmq_ctx *ctx = nullptr;
    Context() { gllmq_init(&ctx, 0); }
    ~Context() { gllmq_destroy(ctx); }
    operator gllmq_ctx *() const { return ctx; }
};

// addresses of a caller's own buffers, far from each other
void *at(int i) { return reinterpret_cast<void *>((uintptr_t(1) << 44) + (uintptr_t(i) << 36)); }

int ffn(gllmq_ctx *ctx, uint32_t gate_up, uint32_t down, size_t m, size_t hidden, size_t ffn, int elem = GLLMQ_ELEM_F32, void *stream = nullptr)
{
    fake::launches.clear();
    return gllmq_ffn_swiglu_elem(ctx, at(1), at(2), ffn * gllmq_row_bytes(gate_up, hidden), gate_up, at(3), hidden * gllmq_row_bytes(down, ffn), down, at(4), at(5),
                                 m, hidden, ffn, 0, elem, 0, stream);
}

int matmul(gllmq_ctx *ctx, uint32_t dtype, size_t m, size_t n, size_t k, int elem, void *x, void *y, int mode = GLLMQ_ACT_F32_SPLIT, void *stream = nullptr)
{
    fake::launches.clear();
    const size_t bytes = n * gllmq_row_bytes(dtype, k);
    if (elem != GLLMQ_ELEM_F32) return gllmq_quantized_matmul_elem(ctx, at(1), bytes, x, y, dtype, m, n, k, elem, stream);
    return gllmq_quantized_matmul_ex(ctx, at(1), bytes, static_cast<const float *>(x), static_cast<float *>(y), dtype, m, n, k, mode, stream);
}

int batch(gllmq_ctx *ctx, uint32_t dtype, size_t m, const std::vector<size_t> &n, size_t k, int elem)
{
    fake::launches.clear();
    const uint32_t flags = elem == GLLMQ_ELEM_F16 ? GLLMQ_DESC_ELEM_F16 : elem == GLLMQ_ELEM_BF16 ? GLLMQ_DESC_ELEM_BF16 : 0u;
    std::vector<gllmq_matmul_desc> descs;
    for (size_t i = 0; i < n.size(); ++i)
        descs.push_back({ at(10 + static_cast<int>(i)), n[i] * gllmq_row_bytes(dtype, k), static_cast<const float *>(at(4)), static_cast<float *>(at(20 + static_cast<int>(i))), dtype, flags, m, n[i], k });
    return gllmq_quantized_matmul_batch(ctx, descs.data(), descs.size(), nullptr);
}

// experts' matrices in one stack a role
int moe(gllmq_ctx *ctx, uint32_t gate_up, uint32_t down, size_t tokens, size_t top_k, size_t hidden, size_t ffn, size_t experts, int elem = GLLMQ_ELEM_F32, int flags = 0)
{
    fake::launches.clear();
    const size_t one = ffn * gllmq_row_bytes(gate_up, hidden), dn = hidden * gllmq_row_bytes(down, ffn);
    uint8_t *const w = static_cast<uint8_t *>(at(1));
    return gllmq_moe_matvec_elem(ctx, w, (2 * experts - 1) * one, 2 * one, w + one, (2 * experts - 1) * one, 2 * one, gate_up, at(3), experts * dn, dn, down, at(4), at(5), tokens, hidden,
                                 ffn, experts, top_k, static_cast<const uint32_t *>(at(6)), static_cast<const float *>(at(7)), static_cast<const uint32_t *>(at(8)), 0, elem, flags, nullptr);
}
// ... its products were the GEMM's
bool moe_gemm()
{
    for (const fake::Launch &l : fake::launches)
        if (l.kernel.find("gq_moe_mmf_") == 0) return true;
    return false;
}

// the wide GEMM among the launches, if it is there
const fake::Launch *wide_launch()
{
    for (const fake::Launch &l : fake::launches)
        if (l.kernel.find("gq_mmf_") == 0 && l.kernel.find("_w") != std::string::npos) return &l;
    return nullptr;
}
bool makes_own_images(const fake::Launch &l) { return l.kernel.find("_own") != std::string::npos; }

size_t launched(const char *kernel)
{
    size_t n = 0;
    for (const fake::Launch &l : fake::launches) n += l.kernel == kernel;
    return n;
}

constexpr uint32_t kMixes[5][2] = { { T_Q4_K, T_Q6_K }, { T_Q5_K, T_Q6_K }, { T_Q6_K, T_Q6_K }, { T_Q8_0, T_Q8_0 }, { T_Q4_K, T_Q4_K } };
constexpr size_t kLayers[5][2] = { { 4096, 14336 }, { 2048, 5632 }, { 1024, 2816 }, { 5120, 13824 }, { 2304, 6912 } };

// The header's promise: what is reserved for, or grown by, one call serves every call of as many or fewer rows, so that a graph
// captured behind it keeps the scratch it holds.
void ffn_scratch_stays()
{
    for (const auto &mix : kMixes)
        for (const auto &layer : kLayers)
            for (size_t most : { 16u, 32u, 64u, 100u, 128u, 512u })
                for (bool reserved : { false, true }) {
                    Context ctx;
                    if (reserved) EXPECT(gllmq_reserve_ffn(ctx, mix[0], mix[1], most, layer[0], layer[1], nullptr) == GLLMQ_OK, "%s", gllmq_last_error(ctx));
                    else EXPECT(ffn(ctx, mix[0], mix[1], most, layer[0], layer[1]) == GLLMQ_OK, "%s", gllmq_last_error(ctx));
                    const size_t before = fake::allocations, freed = fake::frees;
                    for (size_t m = most; m >= 9; m = m > 40 ? m * 7 / 8 : m - 3) {
                        for (int elem : { GLLMQ_ELEM_F32, GLLMQ_ELEM_BF16 }) {
                            EXPECT(ffn(ctx, mix[0], mix[1], m, layer[0], layer[1], elem) == GLLMQ_OK, "%s", gllmq_last_error(ctx));
                            EXPECT(fake::allocations == before && fake::frees == freed, "formats %u/%u, %zu x %zu: %zu rows grow the scratch of %zu", mix[0], mix[1],
                                   layer[0], layer[1], m, most);
                        }
                        EXPECT(gllmq_reserve_ffn(ctx, mix[0], mix[1], m, layer[0], layer[1], nullptr) == GLLMQ_OK && fake::allocations == before,
                               "formats %u/%u, %zu x %zu: reserving %zu rows grows the scratch of %zu", mix[0], mix[1], layer[0], layer[1], m, most);
                        fake::capturing = true;
                        EXPECT(ffn(ctx, mix[0], mix[1], m, layer[0], layer[1]) == GLLMQ_OK, "captured: %s", gllmq_last_error(ctx));
                        fake::capturing = false;
                    }
                }
}

// Gate's and up's sums of K slices are left to the down projection's preparation where both fit the scratch as it is, and added up
// by a launch of their own where they do not.
void ffn_slices_are_left_where_there_is_room()
{
    Context ctx;
    EXPECT(ffn(ctx, T_Q4_K, T_Q6_K, 32, 4096, 14336) == GLLMQ_OK, "%s", gllmq_last_error(ctx));
    EXPECT(launched("gq_mmf_reduce") == 2, "%zu", launched("gq_mmf_reduce"));
    EXPECT(ffn(ctx, T_Q4_K, T_Q6_K, 16, 4096, 14336) == GLLMQ_OK, "%s", gllmq_last_error(ctx));
    EXPECT(launched("gq_mmf_reduce") == 1, "%zu", launched("gq_mmf_reduce"));
    Context larger;
    EXPECT(ffn(larger, T_Q4_K, T_Q6_K, 64, 4096, 14336) == GLLMQ_OK && ffn(larger, T_Q4_K, T_Q6_K, 32, 4096, 14336) == GLLMQ_OK, "%s", gllmq_last_error(larger));
    EXPECT(launched("gq_mmf_reduce") == 1, "%zu", launched("gq_mmf_reduce"));
}

// Outputs over the activations: workgroups that make their images themselves would read rows that others have stored over.  They
// may only where the outputs are stored by the launch that adds up slices.
void outputs_over_the_activations()
{
    Context ctx;
    size_t apart = 0, in_place = 0;
    for (const auto &f : kFormats)
        for (size_t k : { 256u, 512u, 768u, 1024u, 2048u, 4096u })
            for (size_t m : { 33u, 64u, 100u, 512u, 2048u })
                for (int elem : { GLLMQ_ELEM_F32, GLLMQ_ELEM_BF16 })
                    for (intptr_t shift : { intptr_t(-1), intptr_t(0), intptr_t(1) }) { // y from before x's end, x itself, x's last bytes
                        const size_t e = elem == GLLMQ_ELEM_F32 ? 4 : 2, size = m * k * e;
                        uint8_t *const x = static_cast<uint8_t *>(at(4)) + size;
                        EXPECT(matmul(ctx, f.dtype, m, k, k, elem, x, x + size) == GLLMQ_OK, "%s", gllmq_last_error(ctx));
                        const fake::Launch *l = wide_launch();
                        EXPECT(l, "no wide launch");
                        apart += l && makes_own_images(*l) && l->wide().ksplit == 1;
                        EXPECT(matmul(ctx, f.dtype, m, k, k, elem, x, x + shift * static_cast<intptr_t>(size - 4)) == GLLMQ_OK, "%s", gllmq_last_error(ctx));
                        l = wide_launch();
                        EXPECT(l && (!makes_own_images(*l) || l->wide().ksplit > 1), "dtype %u, %zu rows of %zu in place: %s", f.dtype, m, k, l ? l->kernel.c_str() : "");
                        in_place += l && makes_own_images(*l);
                    }
    EXPECT(apart > 20 && in_place > 20, "%zu and %zu calls make their images", apart, in_place);
}

// Several weight tiles per workgroup: the calls of test_runs_of_weight_tiles (test_gpu_gemm_wide.py) take them, odd numbers of blocks among
// them, and so do prompts by themselves; nothing that the kernel cannot do takes them.
void runs_of_weight_tiles()
{
    for (uint32_t dtype : { T_Q4_K, T_Q5_K })
        for (uint32_t tiles : { 2u, 3u, 4u })
            for (uint32_t run : { 2u, 3u, 16u }) {
                Context ctx;
                gllmq_set_option(ctx, "mmfw_mt", tiles);
                gllmq_set_option(ctx, "mmfw_ksplit", 1);
                gllmq_set_option(ctx, "mmfw_run", run);
                const size_t shapes[3][2] = { { 65, 1024 }, { 130, 1536 - 64 }, { 200, 1280 } };
                for (const auto &s : shapes) {
                    EXPECT(batch(ctx, dtype, s[0], { 513, 256, 300 }, s[1], GLLMQ_ELEM_BF16) == GLLMQ_OK, "%s", gllmq_last_error(ctx));
                    const fake::Launch *l = wide_launch();
                    EXPECT(l && l->wide().segs == 3 && l->wide().run_tiles == std::min(run, 6u), "K of %zu, three matrices", s[1]);
                    EXPECT(matmul(ctx, dtype, s[0], 513, s[1], GLLMQ_ELEM_BF16, at(4), at(5)) == GLLMQ_OK, "%s", gllmq_last_error(ctx));
                    l = wide_launch();
                    EXPECT(l && l->wide().run_tiles == std::min(run, 3u) && l->wide().n_runs == (3 + run - 1) / run, "K of %zu", s[1]);
                }
            }
    Context ctx;
    for (const auto &f : kFormats)
        for (size_t k : { 512u, 768u, 1024u, 1280u, 2304u, 4096u, 6912u, 8960u, 11008u })
            for (int elem : { GLLMQ_ELEM_F32, GLLMQ_ELEM_BF16 }) {
                EXPECT(matmul(ctx, f.dtype, 2048, 28672, k, elem, at(4), at(5)) == GLLMQ_OK, "%s", gllmq_last_error(ctx));
                const fake::Launch *l = wide_launch();
                const bool can = k >= 1024 && elem != GLLMQ_ELEM_F32 && (f.dtype == T_Q4_K || f.dtype == T_Q5_K);
                EXPECT(l && (l->wide().run_tiles > 1) == can, "dtype %u, K of %zu, element type %d: %u tiles", f.dtype, k, elem, l ? l->wide().run_tiles : 0u);
            }
}

// The calls of test_images_made_by_the_workgroup (test_gpu_gemm_wide.py) make their images exactly where the blocks fit, single ones and
// batches, and with the switch never.
void own_images()
{
    const uint32_t most[4][2] = { { 4, 3 }, { 4, 3 }, { 4, 3 }, { 4, 2 } }; // blocks of a slice [format][one plane, two]
    const uint32_t slices_blocks[9][2] = { { 1, 1 }, { 1, 2 }, { 1, 3 }, { 1, 4 }, { 1, 5 }, { 2, 2 }, { 2, 3 }, { 3, 3 }, { 3, 4 } };
    for (const auto &f : kFormats)
        for (int elem : { GLLMQ_ELEM_F32, GLLMQ_ELEM_F16, GLLMQ_ELEM_BF16 })
            for (const auto &sb : slices_blocks)
                for (bool on : { true, false }) {
                    Context ctx;
                    gllmq_set_option(ctx, "mmfw_mt", 1);
                    gllmq_set_option(ctx, "mmfw_ksplit", sb[0]);
                    gllmq_set_option(ctx, "mmfw_min_m", 9);
                    gllmq_set_option(ctx, "mmfw_own", on);
                    const size_t k = 256 * sb[0] * sb[1] - (sb[0] > 1 && sb[1] > 1 ? 256 : 0);
                    const bool fits = sb[1] <= most[mmf_format(f.dtype)][elem == GLLMQ_ELEM_F32];
                    for (size_t m : { 33u, 9u, 64u })
                        for (bool group : { false, true }) {
                            EXPECT((group ? batch(ctx, f.dtype, m, { 64, 1 }, k, elem) : matmul(ctx, f.dtype, m, 257, k, elem, at(4), at(5))) == GLLMQ_OK, "%s", gllmq_last_error(ctx));
                            const fake::Launch *l = wide_launch();
                            EXPECT(l && makes_own_images(*l) == (on && fits) && l->wide().ksplit == sb[0] && l->wide().blocks_per_split == sb[1],
                                   "dtype %u, element type %d, %u slices of %u, %zu rows: %s", f.dtype, elem, sb[0], sb[1], m, l ? l->kernel.c_str() : "no wide launch");
                        }
                }
}

// A call of 16-bit elements is the f32 call on the widened activations, rounded, bit for bit: up to eight rows it multiplies with the f32 call's
// kernel over as many workgroups, in the form that reads such elements or between launches that convert.
void elements_take_the_f32_kernels()
{
    Context ctx;
    const auto multiplies = [&](uint32_t dtype, size_t m, size_t n, size_t k, int elem) {
        EXPECT(matmul(ctx, dtype, m, n, k, elem, at(4), at(5)) == GLLMQ_OK, "%s", gllmq_last_error(ctx));
        std::string all;
        for (const fake::Launch &l : fake::launches) {
            std::string name = l.kernel;
            if (name.find("prep") != std::string::npos || name == "gq_convert_elem") continue; // (images are of the same bits wherever they are made)
            for (const char *form : { "_e16", "_hi", "_own" })
                if (const size_t p = name.find(form); p != std::string::npos) name.erase(p, std::strlen(form));
            all += name + " " + std::to_string(l.grid) + " ";
        }
        return all;
    };
    for (const auto &f : kFormats)
        for (size_t m = 1; m <= 8; ++m)
            for (size_t n : { 1u, 777u, 1024u, 1280u, 2048u, 3073u, 3500u, 4096u, 5120u, 8192u, 14336u, 128256u })
                for (size_t k : { 256u, 1024u, 2880u, 4096u, 4864u, 5120u, 7936u, 8192u, 9216u, 9728u, 9984u, 11008u, 14336u, 16384u }) {
                    const std::string f32 = multiplies(f.dtype, m, n, k, GLLMQ_ELEM_F32), bf16 = multiplies(f.dtype, m, n, k, GLLMQ_ELEM_BF16);
                    EXPECT(f32 == bf16, "dtype %u, %zu rows, %zu x %zu: %s, not %s", f.dtype, m, n, k, bf16.c_str(), f32.c_str());
                }
}

// Experts' calls of 16-bit elements, with and without accumulation, take the f32 call's form, and so its bits, on both sides of every line
// between the GEMM and the jobs.
void elements_take_the_f32_experts()
{
    Context ctx;
    size_t gemms = 0, jobs = 0;
    for (const auto &mix : kMixes)
        for (size_t experts : { 8u, 16u, 60u, 128u, 160u })
            for (size_t top_k : { 2u, 8u })
                for (const auto &layer : std::vector<std::vector<size_t>>{ { 1024, 512 }, { 1280, 768 }, { 2048, 1024 }, { 4096, 1536 }, { 4096, 2048 }, { 5120, 1536 }, { 4096, 14336 } })
                    for (size_t pairs = experts; pairs <= 16 * experts && pairs <= 4096; pairs += std::max(experts, top_k)) {
                        const size_t tokens = pairs / top_k;
                        if (tokens == 0) continue;
                        EXPECT(moe(ctx, mix[0], mix[1], tokens, top_k, layer[0], layer[1], experts) == GLLMQ_OK, "%s", gllmq_last_error(ctx));
                        const bool f32 = moe_gemm();
                        (f32 ? gemms : jobs)++;
                        for (int elem : { GLLMQ_ELEM_F32, GLLMQ_ELEM_F16, GLLMQ_ELEM_BF16 })
                            for (int flags : { 0, int(GLLMQ_OUT_ACCUMULATE) }) {
                                EXPECT(moe(ctx, mix[0], mix[1], tokens, top_k, layer[0], layer[1], experts, elem, flags) == GLLMQ_OK, "%s", gllmq_last_error(ctx));
                                EXPECT(moe_gemm() == f32, "formats %u/%u, %zu tokens, top %zu of %zu experts of %zu x %zu, element type %d, flags %d: GEMM %d, f32 %d", mix[0], mix[1], tokens,
                                       top_k, experts, layer[0], layer[1], elem, flags, !f32, f32);
                            }
                    }
    EXPECT(gemms > 200 && jobs > 200, "%zu calls on the GEMM, %zu on the jobs", gemms, jobs);
}

// A layer that is an eighth larger, in any direction, has its line between the jobs and the GEMM where the layer itself has it, to a pair an
// expert (where the GEMM's workgroups go round the device as often, by which its time is estimated).
void experts_line_has_no_edges()
{
    Context ctx;
    const auto line = [&](const uint32_t *mix, size_t hidden, size_t ffn, size_t experts) {
        size_t per = 1;
        for (; per < 16; ++per) {
            EXPECT(moe(ctx, mix[0], mix[1], per * experts / 2, 2, hidden, ffn, experts) == GLLMQ_OK, "%s", gllmq_last_error(ctx));
            if (moe_gemm()) break;
        }
        return per;
    };
    const auto rounds = [](size_t rows, size_t experts) { return ((rows + 255) / 256 * experts + 255) / 256; };
    const auto full = [](size_t ffn, size_t experts) { return (2 * ffn + 255) / 256 * experts >= 512; };
    size_t compared = 0, below = 0;
    for (const auto &mix : kMixes)
        for (size_t hidden : { 1024u, 2048u, 2560u, 4096u, 5120u, 7168u })
            for (size_t ffn : { 512u, 1024u, 1792u, 2048u, 4096u, 8192u })
                for (size_t experts : { 8u, 16u, 32u, 64u, 128u, 256u })
                    for (int way = 0; way < 3; ++way) {
                        const size_t h = hidden + (way == 0 ? hidden / 8 : 0), f = ffn + (way == 1 ? ffn / 8 : 0), e = experts + (way == 2 ? experts / 8 : 0);
                        if (rounds(2 * ffn, experts) != rounds(2 * f, e) || rounds(hidden, experts) != rounds(h, e) || full(ffn, experts) != full(f, e)) continue;
                        const size_t at = line(mix, hidden, ffn, experts), larger = line(mix, h, f, e);
                        if (std::min(at, larger) > 8) continue; // (few small experts: a pair is little of the jobs' time)
                        EXPECT(at <= larger + 1 && larger <= at + 1, "formats %u/%u: %zu experts of %zu x %zu from %zu pairs on, %zu of %zu x %zu from %zu", mix[0], mix[1], experts, hidden, ffn,
                               at, e, h, f, larger);
                        ++compared;
                        below += at < 8;
                    }
    EXPECT(compared > 200 && below > 100, "%zu layers, %zu below eight pairs", compared, below);
}

// f32 layers of few pairs an expert as they were timed in both forms: the GEMM is not taken where it is slower by 8 % and more.
void experts_take_the_faster_form()
{
    struct Timed { uint32_t gate_up, down; size_t tokens, top_k, hidden, ffn, experts; double jobs, gemm; };
    const Timed layers[] = {
        { T_Q4_K, T_Q6_K, 36, 2, 3840, 2048, 16, 91.4, 104.5 }, { T_Q4_K, T_Q6_K, 210, 2, 3840, 768, 64, 154.1, 171.5 }, { T_Q5_K, T_Q6_K, 40, 2, 3072, 1792, 16, 86.3, 94.8 },
        { T_Q4_K, T_Q6_K, 42, 2, 3072, 1536, 16, 76.7, 83.9 },  { T_Q5_K, T_Q6_K, 114, 2, 2560, 1536, 32, 130.4, 141.3 },
    };
    Context ctx;
    for (const Timed &l : layers) {
        EXPECT(moe(ctx, l.gate_up, l.down, l.tokens, l.top_k, l.hidden, l.ffn, l.experts) == GLLMQ_OK, "%s", gllmq_last_error(ctx));
        EXPECT(!moe_gemm(), "formats %u/%u, %zu experts of %zu x %zu, %zu tokens: GEMM %.1f us, jobs %.1f", l.gate_up, l.down, l.experts, l.hidden, l.ffn, l.tokens, l.gemm, l.jobs);
    }
}

// Every kernel that ends in the greedy token is some output matrix's.
void token_kernels_are_reached()
{
    Context ctx;
    std::set<std::string> reached, unreached;
    for (const auto &f : kFormats)
        for (size_t n : { 6145u, 12000u, 32000u, 128256u })
            for (size_t k = 256; k <= 16384; k += 256) {
                fake::launches.clear();
                EXPECT(gllmq_lm_head_argmax(ctx, at(1), n * gllmq_row_bytes(f.dtype, k), static_cast<const float *>(at(4)), f.dtype, n, k, static_cast<float *>(at(5)),
                                            static_cast<uint32_t *>(at(6)), static_cast<float *>(at(7)), nullptr) == GLLMQ_OK, "%s", gllmq_last_error(ctx));
                for (const fake::Launch &l : fake::launches) reached.insert(l.kernel);
            }
    for (const std::string &name : fake::names)
        if (name.find("_token") != std::string::npos && !reached.count(name)) unreached.insert(name);
    for (const std::string &name : unreached) EXPECT(false, "%s", name.c_str());
    EXPECT(reached.count("gq_mm8s_q8_0_p1_e4_token"), "no streamed token");
}

// The workgroups of four waves are the option's, and by themselves some calls' and not others'; workgroups cover all weight rows in either form.
void experts_workgroups_by_option()
{
    size_t with[3] = {}, without[3] = {};
    for (int option = 0; option < 3; ++option) {
        Context ctx;
        gllmq_set_option(ctx, "moe_wide_min", 1);
        gllmq_set_option(ctx, "moe_wide_few", option);
        for (const auto &mix : kMixes)
            for (const auto &layer : std::vector<std::vector<size_t>>{ { 512, 384 }, { 768, 520 }, { 288, 352 }, { 4096, 1536 }, { 4096, 2048 } })
                for (size_t experts : { 8u, 12u, 64u, 128u })
                    for (size_t per : { 8u, 32u, 64u, 110u })
                        for (int elem : { GLLMQ_ELEM_F32, GLLMQ_ELEM_BF16 }) {
                            EXPECT(moe(ctx, mix[0], mix[1], per * experts / 2, 2, layer[0], layer[1], experts, elem) == GLLMQ_OK && moe_gemm(), "%s", gllmq_last_error(ctx));
                            for (const fake::Launch &l : fake::launches) {
                                if (l.kernel.find("gq_moe_mmf_") != 0) continue;
                                const bool few = l.kernel.find("_few") != std::string::npos;
                                (few ? with : without)[option]++;
                                uint32_t tiles = 0;
                                for (uint32_t i = 0; i < l.wide().segs; ++i) {
                                    EXPECT(l.wide().seg[i].tile0 == tiles, "%s", l.kernel.c_str());
                                    tiles += (l.wide().seg[i].n + (few ? 127 : 255)) / (few ? 128 : 256);
                                }
                                EXPECT(l.wide().n_tiles == tiles && l.grid == (l.wide().max_jobs + 7) / 8 * 8 * tiles, "%s: %u workgroups, %u tiles", l.kernel.c_str(), l.grid, l.wide().n_tiles);
                            }
                        }
    }
    EXPECT(with[0] == 0 && without[2] == 0 && with[1] > 100 && without[1] > 100, "%zu, %zu and %zu of four waves, %zu, %zu and %zu of eight", with[0], with[1], with[2], without[0],
           without[1], without[2]);
}

// What is reserved for experts is what the calls of so many pairs need, in any formats and over any number of experts, and no more; a
// captured call of as many or fewer pairs finds it.
void experts_scratch_is_reserved()
{
    const auto held = [](const gllmq_ctx *) {
        size_t bytes = 0;
        for (const auto &b : fake::live) bytes += b.second;
        return bytes;
    };
    std::vector<std::array<uint32_t, 2>> mixes;
    for (const auto &gu : kFormats)
        for (const auto &dn : kFormats) mixes.push_back({ gu.dtype, dn.dtype });
    for (const auto &layer : std::vector<std::vector<size_t>>{ { 1024, 512 }, { 2048, 1024 }, { 4096, 1536 }, { 4096, 14336 }, { 5120, 13824 }, { 7168, 2048 } })
        for (const auto &call : std::vector<std::vector<size_t>>{ { 1, 8 }, { 16, 2 }, { 16, 8 }, { 64, 2 }, { 128, 4 }, { 100, 6 } }) {
            const size_t tokens = call[0], top_k = call[1], pairs = tokens * top_k;
            Context used, reserved;
            const size_t nothing = held(used);
            std::vector<size_t> counts;
            for (size_t e = 1; e <= pairs; e += 1 + e / 24) counts.push_back(e);
            for (size_t e = 8; e <= pairs; e += 8) counts.push_back(e);
            counts.push_back(pairs);
            for (size_t experts : counts)
                for (const auto &mix : mixes) EXPECT(moe(used, mix[0], mix[1], tokens, top_k, layer[0], layer[1], experts) == GLLMQ_OK, "%s", gllmq_last_error(used));
            const size_t needed = held(used) - nothing;
            EXPECT(gllmq_reserve_moe(reserved, tokens, top_k, layer[0], layer[1], nullptr) == GLLMQ_OK, "%s", gllmq_last_error(reserved));
            const size_t taken = held(reserved) - nothing - needed;
            // (a count of experts between the tried ones may take it: 4 % more at most)
            EXPECT(taken >= needed && taken <= needed + needed / 25, "%zu tokens, top %zu, %zu x %zu: %zu bytes, calls need %zu", tokens, top_k, layer[0], layer[1], taken, needed);
            fake::capturing = true;
            for (size_t t = tokens; t > 0; t = t * 3 / 4)
                for (size_t experts : counts)
                    for (const auto &mix : mixes)
                        EXPECT(moe(reserved, mix[0], mix[1], t, top_k, layer[0], layer[1], experts) == GLLMQ_OK, "%zu tokens behind %zu: %s", t, tokens, gllmq_last_error(reserved));
            fake::capturing = false;
        }
}

// Few pairs an expert, whose jobs need less scratch than the GEMM: where that is not to be had the call goes on the jobs, of any element type, and
// what is reserved is what there is room for.  With eight pairs (Q8_0: four) the GEMM or an error, as the reservation is for.
void experts_without_room_take_the_jobs()
{
    struct Layer { uint32_t gate_up, down; size_t few, many, top_k, hidden, ffn, experts; };
    for (const Layer &l : { Layer{ T_Q4_K, T_Q4_K, 27, 200, 2, 4096, 2048, 8 }, Layer{ T_Q8_0, T_Q8_0, 24, 200, 2, 4096, 2048, 16 }, Layer{ T_Q5_K, T_Q6_K, 56, 200, 2, 2560, 1024, 16 } })
        for (int elem : { GLLMQ_ELEM_F32, GLLMQ_ELEM_BF16 }) {
            Context ctx;
            EXPECT(moe(ctx, l.gate_up, l.down, l.few, l.top_k, l.hidden, l.ffn, l.experts, elem) == GLLMQ_OK && moe_gemm(), "%u: %s", l.gate_up, gllmq_last_error(ctx));
            size_t gemm = 0;
            for (const auto &b : fake::live) gemm = std::max(gemm, b.second); // (the largest: of the call)
            EXPECT(moe(ctx, l.gate_up, l.down, l.few, l.top_k, l.hidden, l.ffn, l.experts) == GLLMQ_OK && moe_gemm(), "%s", gllmq_last_error(ctx));
            for (const auto &b : fake::live) EXPECT(b.second <= gemm, "the f32 call grows what element type %d took", elem);
            Context small;
            gllmq_set_option(small, "moe_wide", 0);
            EXPECT(moe(small, l.gate_up, l.down, l.few, l.top_k, l.hidden, l.ffn, l.experts, elem) == GLLMQ_OK && !moe_gemm(), "%s", gllmq_last_error(small));
            gllmq_set_option(small, "moe_wide", 1);
            const std::map<void *, size_t> before = fake::live;
            fake::capturing = true;
            EXPECT(moe(small, l.gate_up, l.down, l.few, l.top_k, l.hidden, l.ffn, l.experts, elem) == GLLMQ_OK && !moe_gemm(), "captured: %s", gllmq_last_error(small));
            fake::capturing = false;
            EXPECT(fake::live == before, "captured: allocations");
            fake::refuse_from = gemm;
            Context refused;
            EXPECT(moe(refused, l.gate_up, l.down, l.few, l.top_k, l.hidden, l.ffn, l.experts, elem) == GLLMQ_OK && !moe_gemm(), "refused: %s", gllmq_last_error(refused));
            EXPECT(moe(refused, l.gate_up, l.down, l.many, l.top_k, l.hidden, l.ffn, l.experts, elem) != GLLMQ_OK, "%u: many pairs", l.gate_up);
            fake::refuse_from = SIZE_MAX;
            Context all, less;
            size_t most = 0, held = 0;
            const std::map<void *, size_t> there = fake::live;
            EXPECT(gllmq_reserve_moe(all, l.few, l.top_k, l.hidden, l.ffn, nullptr) == GLLMQ_OK, "%s", gllmq_last_error(all));
            for (const auto &b : fake::live)
                if (!there.count(b.first)) most = std::max(most, b.second);
            fake::refuse_from = most;
            const std::map<void *, size_t> then = fake::live;
            EXPECT(gllmq_reserve_moe(less, l.few, l.top_k, l.hidden, l.ffn, nullptr) == GLLMQ_OK, "refused: %s", gllmq_last_error(less));
            fake::refuse_from = SIZE_MAX;
            for (const auto &b : fake::live)
                if (!then.count(b.first)) held = std::max(held, b.second);
            EXPECT(held > 0 && held < most, "%zu of %zu bytes", held, most);
        }
}

// Scratch that a captured call has used stays, whatever eager calls of more rows, and calls on many other streams, do afterwards;
// what no graph can hold is given back as it is outgrown, and everything with the context.
void scratch_of_graphs_stays()
{
    const auto elsewhere = [](int i) { return reinterpret_cast<void *>(uintptr_t(i + 1) << 8); };
    for (int call = 0; call < 5; ++call)
        for (bool captured : { true, false }) {
            const size_t before = fake::live.size();
            {
                Context ctx;
                const size_t n = call == 3 ? 1000 : 4096;
                const auto run = [&](size_t m, void *stream) {
                    int rc = 0;
                    if (call == 0) rc = matmul(ctx, T_Q6_K, m, n, 4096, GLLMQ_ELEM_F32, at(4), at(5), GLLMQ_ACT_F32_SPLIT, stream); // GEMM
                    else if (call == 1) rc = ffn(ctx, T_Q4_K, T_Q6_K, m, 1024, 2816, GLLMQ_ELEM_BF16, stream);
                    else if (call == 2) rc = ffn(ctx, T_Q4_K, T_Q6_K, std::min<size_t>(m, 16) / 4, 1024, 2816, GLLMQ_ELEM_F32, stream); // (four rows at most)
                    else if (call == 3) rc = matmul(ctx, T_Q8_0, m == 16 ? 4 : 8, m == 16 ? n : 4 * n, 1024, GLLMQ_ELEM_BF16, at(4), at(5), GLLMQ_ACT_F32_SPLIT, stream); // converted
                    else rc = gllmq_argmax(ctx, static_cast<const float *>(at(4)), 1, 128256, 128256, static_cast<uint32_t *>(at(5)), nullptr, stream);
                    EXPECT(rc == GLLMQ_OK, "call %d: %s", call, gllmq_last_error(ctx));
                };
                const std::map<void *, size_t> first = fake::live;
                run(16, elsewhere(0));
                std::map<void *, size_t> held = fake::live;
                for (const auto &b : first) held.erase(b.first);
                EXPECT(!held.empty(), "call %d", call);
                fake::capturing = captured;
                run(16, elsewhere(0));
                fake::capturing = false;
                for (size_t m : { 64u, 512u, 2048u }) run(m, elsewhere(0));
                if (call != 2 && call != 4) EXPECT(fake::live.size() == first.size() + held.size() + captured + (call == 1 && captured), "call %d: %zu allocations", call, fake::live.size() - first.size());
                for (int other = 1; other <= 40; ++other) run(16, elsewhere(other));
                size_t there = 0;
                for (const auto &b : held) there += fake::live.count(b.first);
                EXPECT(captured ? there == held.size() : there == 0, "call %d%s: %zu of %zu buffers are there", call, captured ? ", captured" : "", there, held.size());
            }
            EXPECT(fake::live.size() == before, "call %d: %zu allocations left", call, fake::live.size() - before);
        }
}

// A prompt's decoded weights take as much scratch as the call's matrices need: other formats allocate nothing for them, a call that cannot
// have it goes without, and a reservation is enough for a captured call to have it.
void decoded_weights_scratch()
{
    const auto held = [] {
        size_t bytes = 0;
        for (const auto &b : fake::live) bytes += b.second;
        return bytes;
    };
    const auto decodes = [] { return launched("gq_mmfx_decode_q6k"); };
    for (const auto &f : kFormats)
        for (size_t m : { 1023u, 1024u, 2048u })
            for (const auto &s : std::vector<std::vector<size_t>>{ { 100, 1024 }, { 4096, 4096 }, { 4096, 14336 }, { 14336, 4096 }, { 28672, 4096 }, { 128256, 2048 } }) {
                size_t total[2], need = std::min<size_t>((s[0] + 31) / 32 * (s[1] / 256) * gq::MmfxRecord::bytes, size_t(128) << 20);
                for (int decoded = 0; decoded < 2; ++decoded) {
                    Context ctx;
                    if (!decoded) gllmq_set_option(ctx, "mmfx_min_m", 0);
                    for (int elem : { GLLMQ_ELEM_F32, GLLMQ_ELEM_BF16 }) {
                        EXPECT(matmul(ctx, f.dtype, m, s[0], s[1], elem, at(4), at(5)) == GLLMQ_OK, "%s", gllmq_last_error(ctx));
                        EXPECT((decodes() > 0) == (decoded && f.dtype == T_Q6_K && m >= 1024 && s[0] > 100), "dtype %u, %zu rows, %zu x %zu: %zu", f.dtype, m, s[0], s[1], decodes());
                    }
                    total[decoded] = held();
                }
                EXPECT(total[1] >= total[0] && total[1] - total[0] <= (f.dtype == T_Q6_K && m >= 1024 ? need : 0), "dtype %u, %zu rows, %zu x %zu: %zu bytes more, the weights need %zu",
                       f.dtype, m, s[0], s[1], total[1] - total[0], need);
            }
    // a down projection behind sums that gate and up leave, which the scratch cannot grow around: room for it is made ahead of them
    for (const auto &s : std::vector<std::vector<size_t>>{ { 1024, 8192, 1024 }, { 1536, 4096, 1024 }, { 3000, 5120, 512 } }) {
        Context ctx;
        EXPECT(ffn(ctx, T_Q4_K, T_Q6_K, s[0], s[1], s[2]) == GLLMQ_OK && launched("gq_mmf_reduce") == 0 && decodes() == 1, "%zu rows, %zu x %zu: %zu", s[0], s[1], s[2], decodes());
        fake::refuse_from = 1;
        EXPECT(ffn(ctx, T_Q4_K, T_Q6_K, s[0], s[1], s[2]) == GLLMQ_OK && decodes() == 1, "%s", gllmq_last_error(ctx));
        fake::refuse_from = SIZE_MAX;
    }
    for (bool reserved : { false, true }) {
        Context ctx;
        // no room: the weights as they are, in the scratch that there was
        EXPECT(matmul(ctx, T_Q6_K, 1024, 4096, 4096, GLLMQ_ELEM_F32, at(4), at(5)) == GLLMQ_OK && decodes() == 1, "%s", gllmq_last_error(ctx));
        fake::refuse_from = size_t(100) << 20;
        const size_t before = held(), frees = fake::frees;
        EXPECT(matmul(ctx, T_Q6_K, 1024, 14336, 4096, GLLMQ_ELEM_F32, at(4), at(5)) == GLLMQ_OK && decodes() == 0 && wide_launch(), "%s", gllmq_last_error(ctx));
        EXPECT(gllmq_reserve_matmul(ctx, T_Q6_K, 1024, 14336, 4096, nullptr) == GLLMQ_OK, "%s", gllmq_last_error(ctx));
        EXPECT(matmul(ctx, T_Q6_K, 1024, 4096, 4096, GLLMQ_ELEM_F32, at(4), at(5)) == GLLMQ_OK && decodes() == 1 && held() == before && fake::frees == frees, "%zu bytes", held());
        fake::refuse_from = SIZE_MAX;
        // captured: with what there is
        fake::capturing = true;
        EXPECT(matmul(ctx, T_Q6_K, 1024, 14336, 4096, GLLMQ_ELEM_F32, at(4), at(5)) == GLLMQ_OK && decodes() == 0, "%s", gllmq_last_error(ctx));
        EXPECT(matmul(ctx, T_Q6_K, 1024, 4096, 4096, GLLMQ_ELEM_F32, at(4), at(5)) == GLLMQ_OK && decodes() == 1, "%s", gllmq_last_error(ctx));
        fake::capturing = false;
        const std::map<void *, size_t> captured = fake::live;
        for (size_t m : { 1024u, 1500u, 2048u })
            for (int elem : { GLLMQ_ELEM_F32, GLLMQ_ELEM_BF16 }) {
                if (reserved) EXPECT(gllmq_reserve_ffn(ctx, T_Q6_K, T_Q6_K, m, 4096, 7000 / 256 * 256, nullptr) == GLLMQ_OK, "%s", gllmq_last_error(ctx));
                else EXPECT(ffn(ctx, T_Q6_K, T_Q6_K, m, 4096, 7000 / 256 * 256, elem) == GLLMQ_OK && decodes() == 3, "%zu: %s", decodes(), gllmq_last_error(ctx));
                for (const auto &b : captured) EXPECT(fake::live.count(b.first), "%zu bytes that a graph holds are gone", b.second);
                const size_t allocations = fake::allocations;
                fake::capturing = true;
                EXPECT(ffn(ctx, T_Q6_K, T_Q6_K, m, 4096, 7000 / 256 * 256, GLLMQ_ELEM_BF16) == GLLMQ_OK && decodes() == 3 && fake::allocations == allocations, "%zu: %s", decodes(), gllmq_last_error(ctx));
                fake::capturing = false;
            }
    }
}

const std::map<std::string, std::function<void()>> kChecks = {
    { "decoded_weights_scratch", decoded_weights_scratch },
    { "scratch_of_graphs_stays", scratch_of_graphs_stays },
    { "elements_take_the_f32_kernels", elements_take_the_f32_kernels },
    { "elements_take_the_f32_experts", elements_take_the_f32_experts },
    { "experts_workgroups_by_option", experts_workgroups_by_option },
    { "token_kernels_are_reached", token_kernels_are_reached },
    { "experts_line_has_no_edges", experts_line_has_no_edges },
    { "experts_take_the_faster_form", experts_take_the_faster_form },
    { "experts_scratch_is_reserved", experts_scratch_is_reserved },
    { "experts_without_room_take_the_jobs", experts_without_room_take_the_jobs },
    { "runs_of_weight_tiles", runs_of_weight_tiles },
    { "outputs_over_the_activations", outputs_over_the_activations },
    { "own_images", own_images },
    { "ffn_scratch_stays", ffn_scratch_stays },
    { "ffn_slices_are_left_where_there_is_room", ffn_slices_are_left_where_there_is_room },
};

} // namespace

int main(int argc, char **argv)
{
    if (argc > 1 && !kChecks.count(argv[1])) {
        std::printf("no check %s\n", argv[1]);
        return 1;
    }
    for (const auto &check : kChecks)
        if (argc < 2 || check.first == argv[1]) check.second();
    if (failures) std::printf("%d failures\n", failures);
    else std::printf("ok\n");
    return failures ? 1 : 0;
}
