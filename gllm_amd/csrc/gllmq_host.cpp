// Host side of libgllm_hip_quant.so: the C ABI of include/gllm_hip_quant.h over the
// embedded gfx950 code objects.  Kernels are launched with hipModuleLaunchKernel on the
// caller's stream, the driver-style convention the reference's HIP backend uses
// (src/compat/hip_backend.rs:211-238), except that the module is loaded and every
// function resolved once per context instead of once per launch.
#include "gllm_hip_quant.h"
#include "gq_host_internal.h"
#include "gq_params.h"

#include <hip/hip_runtime_api.h>
#include <hip/hip_ext.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <type_traits>
#include <unordered_map>
#include <unordered_set>
#include <vector>

// The code objects built from the kernels_*.hip translation units, placed in .rodata by the
// assembler (GLLMQ_HSACO_DIR is the build directory).  A test of this file without a GPU has its own stand-ins.
#ifndef GLLMQ_EMBED
#define GLLMQ_EMBED(NAME)                                                              \
    __asm__(".section .rodata\n"                                                       \
            ".balign 4096\n"                                                           \
            ".global gllmq_co_" #NAME "\n"                                             \
            "gllmq_co_" #NAME ":\n"                                                    \
            ".incbin \"" GLLMQ_HSACO_DIR "/kernels_" #NAME ".hsaco\"\n"                 \
            ".byte 0\n"                                                                \
            ".previous\n");                                                            \
    extern "C" const unsigned char gllmq_co_##NAME[];
#endif
GLLMQ_EMBED(codec)
GLLMQ_EMBED(mm8)
GLLMQ_EMBED(mm8s)
GLLMQ_EMBED(mm8s_q8_0)
GLLMQ_EMBED(mm8c)
GLLMQ_EMBED(mm8_q6k_q8_0)
GLLMQ_EMBED(mmf)
GLLMQ_EMBED(mmfs)
GLLMQ_EMBED(mmfw)
GLLMQ_EMBED(moe)

namespace {

constexpr uint32_t T_Q8_0 = GLLMQ_TYPE_Q8_0, T_Q4_K = GLLMQ_TYPE_Q4_K, T_Q5_K = GLLMQ_TYPE_Q5_K,
                   T_Q6_K = GLLMQ_TYPE_Q6_K;

struct Format {
    uint32_t dtype;
    size_t block_size, block_bytes;
    size_t group_bytes; // bytes of 256 elements
    size_t w_align;
    const char *tag;
};

const Format kFormats[] = {
    { T_Q8_0, 32, 34, 272, 2, "q8_0" },
    { T_Q4_K, 256, 144, 144, 16, "q4k" },
    { T_Q5_K, 256, 176, 176, 16, "q5k" },
    { T_Q6_K, 256, 210, 210, 2, "q6k" },
};
constexpr int kNumFormats = 4;

const Format *find_format(uint32_t dtype)
{
    for (const Format &f : kFormats)
        if (f.dtype == dtype) return &f;
    return nullptr;
}

int format_index(uint32_t dtype)
{
    for (int i = 0; i < kNumFormats; ++i)
        if (kFormats[i].dtype == dtype) return i;
    return -1;
}

using gq::ArgmaxParams;
using gq::GatherParams;
using gq::GemvParams;
using gq::Mm8Params;
using gq::MmfParams;
using gq::MmfPrepParams;
using gq::MmfReduceParams;
using gq::Mm8ChainEntry;
using gq::Mm8ChainParams;
using gq::MoeActParams;
using gq::MoeCombineParams;
using gq::MoeGemvParams;
using gq::MoeJob;
using gq::MoeJob8;
using gq::MoeMm8Params;
using gq::MoePlanParams;

// Bytes of one block's activation image and of the GEMM's LDS, by 32-row activation tiles (1 or
// 2) and format (0 = Q4_K, 1 = Q5_K, 2 = Q6_K).
uint32_t mmf_image_bytes(uint32_t mt) { return mt == 1 ? gq::MmfLds<1>::image : gq::MmfLds<2>::image; }
uint32_t mmf_lds_bytes(uint32_t mt, int fmt)
{
    static const uint32_t kTotal[2][4] = {
        { gq::MmfLds<1, 0>::total, gq::MmfLds<1, 1>::total, gq::MmfLds<1, 2>::total, gq::MmfLds<1, 3>::total },
        { gq::MmfLds<2, 0>::total, gq::MmfLds<2, 1>::total, gq::MmfLds<2, 2>::total, gq::MmfLds<2, 3>::total },
    };
    return kTotal[mt - 1][fmt];
}

uint32_t mmfw_lds_bytes(int fmt, int planes, uint32_t mt)
{
#define GQ_ROW(F, PL) { gq::mmfw_lds<F, PL, 1>(), gq::mmfw_lds<F, PL, 2>(), gq::mmfw_lds<F, PL, 3>(), gq::mmfw_lds<F, PL, 4>() }
    static const uint32_t kTotal[4][2][4] = { { GQ_ROW(0, 1), GQ_ROW(0, 2) }, { GQ_ROW(1, 1), GQ_ROW(1, 2) },
                                              { GQ_ROW(2, 1), GQ_ROW(2, 2) }, { GQ_ROW(3, 1), GQ_ROW(3, 2) } };
#undef GQ_ROW
    return kTotal[fmt][planes - 1][mt - 1];
}

// ... over experts' jobs (`few`: in workgroups of four waves)
uint32_t mmfw_grouped_lds(int fmt, int planes, bool few)
{
#define GQ_ROW(F, PL) { gq::mmfw_grouped_lds<F, PL, gq::MMFW_EXPERTS>(), gq::mmfw_grouped_lds<F, PL, gq::MMFW_EXPERTS_FEW>() }
    static const uint32_t kTotal[4][2][2] = { { GQ_ROW(0, 1), GQ_ROW(0, 2) }, { GQ_ROW(1, 1), GQ_ROW(1, 2) },
                                              { GQ_ROW(2, 1), GQ_ROW(2, 2) }, { GQ_ROW(3, 1), GQ_ROW(3, 2) } };
#undef GQ_ROW
    return kTotal[fmt][planes - 1][few ? 1 : 0];
}

// ... with decoded weights (Q6_K, from two tiles on)
uint32_t mmfx_lds_bytes(int planes, uint32_t mt)
{
    static const uint32_t kTotal[2][3] = { { gq::MmfxShape<1, 2>::total, gq::MmfxShape<1, 3>::total, gq::MmfxShape<1, 4>::total },
                                           { gq::MmfxShape<2, 2>::total, gq::MmfxShape<2, 3>::total, gq::MmfxShape<2, 4>::total } };
    return kTotal[planes - 1][mt - 2];
}

// ... where a workgroup makes its images itself: blocks of K that its slice may have, LDS
uint32_t mmfw_own_blocks(int fmt, int planes)
{
    static const uint32_t kBlocks[4][2] = { { gq::mmfw_own_blocks<0, 1>(), gq::mmfw_own_blocks<0, 2>() }, { gq::mmfw_own_blocks<1, 1>(), gq::mmfw_own_blocks<1, 2>() },
                                            { gq::mmfw_own_blocks<2, 1>(), gq::mmfw_own_blocks<2, 2>() }, { gq::mmfw_own_blocks<3, 1>(), gq::mmfw_own_blocks<3, 2>() } };
    return kBlocks[fmt][planes - 1];
}
uint32_t mmfw_own_lds(int fmt, int planes)
{
    static const uint32_t kTotal[4][2] = { { gq::mmfw_own_lds<0, 1>(), gq::mmfw_own_lds<0, 2>() }, { gq::mmfw_own_lds<1, 1>(), gq::mmfw_own_lds<1, 2>() },
                                           { gq::mmfw_own_lds<2, 1>(), gq::mmfw_own_lds<2, 2>() }, { gq::mmfw_own_lds<3, 1>(), gq::mmfw_own_lds<3, 2>() } };
    return kTotal[fmt][planes - 1];
}

// Formats of the int8 matrix-core kernels, in the order of the kernel tables below.
// (the grouped MoE kernels exist for the first MM8_MOE_KINDS of them)
enum Mm8Kind { MM8_Q4K = 0, MM8_Q6K = 1, MM8_Q5K = 2, MM8_Q8_0 = 3, MM8_KINDS = 4, MM8_MOE_KINDS = 3 };
int mm8_kind(uint32_t dtype)
{
    return dtype == T_Q4_K ? MM8_Q4K : dtype == T_Q6_K ? MM8_Q6K : dtype == T_Q5_K ? MM8_Q5K : dtype == T_Q8_0 ? MM8_Q8_0 : -1;
}

// Bytes of LDS the int8 matrix-core kernels need: Q4_K and Q5_K keep 8 sub-block sums per
// block, Q6_K and Q8_0 none, and the weight stage of a wave differs by format.
uint32_t mm8_lds_bytes(uint32_t groups, uint32_t m, uint32_t pairs, int kind = MM8_Q4K)
{
    const uint32_t stage = kind == MM8_Q6K ? gq::MM8Q6_STAGE_BYTES : kind == MM8_Q8_0 ? gq::MM8Q8_STAGE_BYTES
                         : kind == MM8_Q5K ? gq::Mm8Format<1>::STAGE : gq::Mm8Format<0>::STAGE;
    return gq::mm8_lds_layout(groups, m, pairs, kind == MM8_Q6K || kind == MM8_Q8_0 ? 0u : 8u, stage).total;
}

} // namespace

// Device memory beyond the inputs and outputs that the kernels of one call may use.  Every stream
// a context is used on gets its own set, so calls on different streams never share scratch and
// calls on one stream are ordered by the stream itself.
struct Scratch {
    hipStream_t stream = nullptr;
    uint64_t last_use = 0;
    bool fixed = false;          // carved from a block of fixed size: a call that needs more fails
    // K split of the int8 kernels: slice sums, and arrival counters that every launch leaves at 0
    float *mm8_part = nullptr;   // [MM8_SPLIT_PART_FLOATS]
    uint32_t *mm8_arrive = nullptr; // [MM8_SPLIT_MAX_LISTS]
    uint64_t *argmax_keys = nullptr; // [ARGMAX_MAX_ROWS][ARGMAX_MAX_PARTS]
    void *base = nullptr;        // the allocation that holds the three above
    void *mmf = nullptr;         // GEMM: activation images, then partial sums of K-split workgroups or decoded weights
    size_t mmf_bytes = 0;
    void *ffn = nullptr;         // gllmq_ffn_swiglu: gated activations, then gate/up results
    size_t ffn_bytes = 0;
    void *moe = nullptr;         // gllmq_moe_matvec: pair tables, jobs, intermediate activations
    size_t moe_bytes = 0;
    void *elem = nullptr;        // 16-bit activations and outputs as f32, for the kernels that do not convert themselves
    size_t elem_bytes = 0;
    void *box = nullptr;         // the chained launch's mailbox [kChainBoxPairs] of 64-bit words, zero when allocated
    std::vector<void *> in_graph; // the allocations there were when a call that uses scratch was last captured: a graph may hold them
};

constexpr size_t kScratchArriveBytes = 4096; // MM8_SPLIT_MAX_LISTS words, padded; the chain kernel's counters behind them
constexpr size_t kLmHeadTicketAt = 600;      // the lm_head launch's count of finished workgroups
constexpr size_t kScratchKeysBytes = sizeof(uint64_t) * gq::ARGMAX_MAX_ROWS * gq::ARGMAX_MAX_PARTS;
constexpr size_t kScratchPartBytes = sizeof(float) * gq::MM8_SPLIT_PART_FLOATS;
constexpr size_t kScratchFixedBytes = kScratchArriveBytes + kScratchKeysBytes + kScratchPartBytes;
constexpr size_t kMaxScratchSlots = 16;

// The greedy token behind a one-row matmul's outputs `y` (gllmq_lm_head_argmax).
struct TokenChoice {
    const float *y;
    size_t n;
    uint64_t *keys;
    uint32_t *ticket, *token;
    float *value;
    bool made; // the launch makes it
};

// Weights that a host-slice call uploaded, kept for the next call with the same slice
// (the reference keeps its uploaded weight blob the same way, src/compat/hip_backend.rs:141-156).
struct CachedWeights {
    const void *host = nullptr;
    size_t bytes = 0;
    void *dev = nullptr;
    uint64_t last_use = 0;
};

struct gllmq_ctx {
    int device = 0;
    hipModule_t modules[10] = {}; // one per embedded code object
    hipFunction_t dequant[kNumFormats][2] = {}; // [format][0 = scalar stores, 1 = float4 stores]
    hipFunction_t gather[kNumFormats][2] = {};  // quantized embedding lookup [format][0 = scalar stores, 1 = float4 stores]
    hipFunction_t gather_e16[kNumFormats][3] = {}; // the same into rows of a 16-bit element type [format][0 = scalar stores, 1 = 8-byte stores, 2 = 16-byte stores]
    hipFunction_t finish_elem = nullptr;        // f32 result in scratch -> output of any element type, plain or added to it
    // gated form of the int8 kernels (gate and up rows in one launch, act(gate) * up out):
    // [0 = Q4_K, 1 = Q5_K][pairs 1,2,4][early steps 1,2,4] and the register-operand variants
    hipFunction_t mm8_glu[2][3][3] = {};
    hipFunction_t mm8_gated_p4[MM8_KINDS] = {}; // five to eight rows of gated activations (a down projection's), by Mm8Kind
    hipFunction_t mm8_glu_areg[2][2][3][2] = {};
    hipFunction_t glu_act = nullptr;            // act(gate) * up as a kernel of its own
    hipFunction_t argmax_part = nullptr, argmax_final = nullptr;
    hipFunction_t dequant_wave = nullptr;       // Q4_K with 16-byte aligned blocks and outputs: one block per wave
    hipFunction_t dequant_wave_q5k = nullptr;   // the same for Q5_K
    hipFunction_t gemv[kNumFormats][2] = {};    // [format][m - 1], f32 multiply-add flavour
    hipFunction_t gemv_i8[kNumFormats][2] = {}; // [format][m - 1], integer-dot flavour (default)
    // call_mutex held: launches are only counted and the last kernel noted, nothing is enqueued
    // (gllmq_lm_head_argmax asks which kernel the one-row matmul of its shape would get)
    bool probe = false;
    uint32_t probe_launches = 0;
    hipFunction_t probe_fn = nullptr;
    hipFunction_t gemv_i8_argmax[kNumFormats] = {}; // one row, ending in the candidates of the greedy token choice
    // int8 matrix-core kernels [Mm8Kind][pairs 1,2,4][early steps 1,2,4], and the same with
    // register-resident activation operands [Mm8Kind][pairs 1,2][early][passes per tile - 1]
    hipFunction_t mm8[MM8_KINDS][3][3] = {};
    hipFunction_t mm8_areg[MM8_KINDS][2][3][2] = {};
    // streamed form (loader waves + arithmetic waves) [0 = Q4_K, 1 = Q5_K, 2 = Q6_K, 3 = Q8_0][variant]: register
    // operands p1_e1, p1_e2, p2_e4, then LDS operands p1_e2, p2_e4, p4_e4
    hipFunction_t mm8s[4][7] = {};
    hipFunction_t mm8s_token[4][3] = {};        // one row, ending in the greedy token choice [format as above][p1_e1_a, p1_e2, p1_e4]
    bool use_mm8s = true;                       // "mm8s" = 0: the fetch-and-compute kernels throughout
    bool batch_overlap = true;                  // "batch_overlap" = 0: the kernels of a batch run strictly one after the other
    bool mm8s_all = false;                      // "mm8s_all" = 1: the streamed form wherever it fits, also where another was timed faster
    bool mm8_small_to_gemv = true;              // "mm8_small_to_gemv" = 0: one Q4_K row over few weight rows stays on the matrix-core kernels
    bool mm8s_areg = true;                      // "mm8s_areg" = 0: the streamed kernels never keep the digit planes in registers
    uint32_t mm8s_depth = 0;                    // "mm8s_depth": items a loader keeps unconfirmed, 0 = by item size
    uint32_t mm8s_min_rows = 8;                 // "mm8s_min_rows": fewest weight rows per CU that take the streamed form
    hipFunction_t moe_mm8_glu_fn[3][2] = {};    // gated gate/up kernels [Mm8Kind (Q4_K and Q5_K only)][passes per tile - 1]
    hipFunction_t mmf_q4k[4][2][2] = {};        // f16 matrix-core GEMM [0 = Q4_K, 1 = Q5_K, 2 = Q6_K, 3 = Q8_0][32-row activation tiles - 1][bf16 mode]
    hipFunction_t mmfw[4][4][2] = {};           // the GEMM for more rows [format as above][32-row activation tiles - 1][0 = hi and lo plane, 1 = hi only]
    hipFunction_t moe_mmf[4][2] = {};           // the same over experts' rows [format][plane]
    hipFunction_t moe_mmf_few[4][2] = {};       // ... in workgroups of four waves
    hipFunction_t mmfw_own[4][2] = {};          // ... of one tile, which prepares the activations itself [format][0 = hi and lo plane, 1 = hi only]
    hipFunction_t mmfx_decode = nullptr;        // Q6_K weights to matrix-core operands, for prompts
    hipFunction_t mmfx[gq::MMFW_MAX_MT - 1][2] = {}; // ... and their GEMM [tiles - 2][0 = hi and lo plane, 1 = hi only]
    uint32_t mmfx_min_m = 1024;                 // "mmfx_min_m": from how many activation rows on (0: never)
    bool use_mmfw_own = true;                   // "mmfw_own" = 0: always a launch that prepares them
    hipFunction_t mmfw_prep[2] = {};            // its activation images [hi and lo plane, hi only]
    hipFunction_t mmfw_prep_e16 = nullptr;      // ... from 16-bit elements
    bool use_mmfw = true;                       // "mmfw" = 0: 64-row passes of the other forms
    uint32_t mmfw_min_m = 33;                   // "mmfw_min_m": fewest activation rows that take it
    bool batch_group = true;                    // "batch_group": independent entries over the same rows as one GEMM
    uint32_t mmfw_small_min_m = 9;              // "mmfw_small_min_m": ... where the streamed GEMMs do not take the call
    uint32_t mmfw_mt = 0, mmfw_ksplit = 0;      // "mmfw_mt", "mmfw_ksplit": activation tiles per workgroup, slices of K (0 = by the shape)
    uint32_t mmfw_run = 0;                      // "mmfw_run": weight tiles per workgroup, one after the other, where the kernel can (0 = by the shape)
    hipFunction_t mmfs[2][2] = {};              // its streamed form [0 = Q4_K, 1 = Q5_K][bf16 mode]
    hipFunction_t mmfr[2][2] = {};              // the streamed form whose waves prepare their own activations (9 to 16 rows) [0 = Q4_K, 1 = Q5_K][f32, 16-bit]
    bool use_mmfr = true;                       // "mmfr" = 0: never
    uint32_t mmfr_min_rows = 8;                 // "mmfr_min_rows": fewest weight rows per CU that take it
    hipFunction_t mm8c[3][2][2] = {};           // chains of streamed matmuls in one launch [0 = Q4_K, 1 = Q5_K, 2 = Q8_0][some entry in pairs of blocks][some entry waits for the one before it]
    bool chain_dependent = false;               // "chain_dependent" = 1: an entry that reads the output of the one before it stays in the chained launch (measured slower than a launch of its own)
    uint32_t chain_epoch = 1;                   // epochs handed to chained entries so far (see Mm8ChainParams::box)
    bool use_chain = true;                      // "chain" = 0: every entry of a batch is a launch of its own
    uint32_t chain_min_rows = 1;                // "chain_min_rows": fewest weight rows in a CU's share of an entry that joins a chain
    uint32_t chain_spin_limit = 1u << 20;       // "chain_spin_limit": polls of a dependency counter before a workgroup gives up
    uint32_t *chain_error = nullptr;            // host memory the device can write: set when such a wait ran out
    bool mmfs_all = false;                      // "mmfs_all" = 1: the streamed GEMM wherever it fits, also where the other form was timed faster
    bool use_mmfs = true;                       // "mmfs" = 0: the three-launch GEMM throughout
    uint32_t mmfs_min_rows = 8;                 // "mmfs_min_rows": fewest weight rows per CU that take the streamed GEMM
    hipFunction_t mmf_prep_lanes = nullptr;     // the images of the streamed form
    hipFunction_t mmf_prep[2] = {};             // its activation preparation [32-row activation tiles - 1]
    hipFunction_t mmf_reduce = nullptr;         // and the in-order sum of its K-split partial results
    hipFunction_t moe_plan = nullptr, moe_plan_wide = nullptr, moe_plan_few = nullptr, moe_act = nullptr, moe_combine = nullptr, moe_combine_v4 = nullptr, moe_route = nullptr;
    hipFunction_t moe_gemv[kNumFormats] = {};
    hipFunction_t moe_mm8_fn[MM8_KINDS][2] = {}; // grouped int8 matrix-core kernels [Mm8Kind][passes per tile - 1]
    hipFunction_t moe_mm8_q6k_rows = nullptr;   // Q6_K rows of at most 8 blocks: a wave per 32-row tile
    hipFunction_t moe_mm8s_fn[MM8_MOE_KINDS][2] = {}; // the grouped kernels in the streamed form [Mm8Kind][plain, gated]
    uint32_t *identity_rows = nullptr;          // device: 0..7, the activation rows of an ungathered matmul

    // Kernel-family choices (gllmq_set_option).  The defaults are the measured best; the tests
    // switch them to reach every kernel family through the public entry points.
    bool gemv_f32 = false;                      // "gemv_f32": the f32 multiply-add GEMV instead of the integer-dot one
    bool use_mm8 = true;                        // "mm8" = 0: no int8 matrix-core kernels
    bool use_mmf = true;                        // "mmf" = 0: more than 8 rows run 8-row passes
    bool ffn_fused = true;                      // "ffn_fused" = 0: gllmq_ffn_swiglu never uses the gated kernels
    // Fewest activation rows that send a format to the int8 matrix-core kernel (below, the GEMV
    // kernels are as fast or faster); 1 = always, 0 = never.
    uint32_t mm8_q6k_min_m = 3, mm8_q5k_min_m = 2, mm8_q8_0_min_m = 3;
    // Fewest rows the GEMM takes when the 8-row kernel would need more than one pass over the
    // weights (long rows: the prepared activations of all rows do not fit the LDS of a CU); 0 = never.
    uint32_t mmf_small_min_m = 3;
    uint32_t mm8_ksplit_max = 8;                // "mm8_ksplit": most slices of the K split (0 or 1 = never split)
    bool moe_mm8 = true;                        // "moe_mm8" = 0: expert rows stay on the GEMV kernels
    bool moe_mm8_q6k = true;                    // "moe_mm8_q6k" = 0: Q6_K expert rows stay there
    bool moe_glu = true;                        // "moe_glu" = 0: gate/up results to memory, activation as a kernel of its own
    uint32_t moe_slices = 0;                    // "moe_slices": workgroups that share a job's row tiles (0 = by the number of pairs and experts)
    bool moe_mm8_rows = true;                   // "moe_mm8_rows" = 0: no wave-per-tile kernel for short Q6_K rows
    uint32_t moe_streamed = 1;                  // "moe_streamed": the grouped kernels in the streamed form: 0 never, 1 while experts see few tokens each, 2 always
    bool moe_wide = true;                       // "moe_wide" = 0: experts with many tokens stay on the eight-token jobs
    bool moe_wide_cost = true;                  // ... and only where it is estimated to be ahead (off once "moe_wide_min" is set)
    uint32_t moe_wide_few = 1;                  // "moe_wide_few" = 0 / 2: its workgroups of four waves never / always
    uint32_t moe_wide_min = 2;                  // "moe_wide_min": fewest pairs per expert (on average) that take the GEMM
    uint32_t moe_depth = 0;                     // "moe_depth": items a loader of the streamed grouped kernels keeps unconfirmed (0 = as the dense launches)

    // One lock over every enqueue on this context: calls from several threads take turns on the
    // host (the kernels they enqueue overlap as their streams allow).
    // State of gllmq_quantized_matmul_batch while it enqueues (see launch2d).
    struct Overlap {
        bool on = false;                 // inside a batch
        bool entry_first = false;        // the next launch is the first of its entry
        bool group_open = false;         // a launch of this batch has been enqueued
        bool group_uses_scratch = false; // a kernel that may still be running uses the scratch
    } overlap;
    std::recursive_mutex call_mutex;
    std::vector<Scratch> scratch;               // one set per stream the context has been used on
    std::vector<void *> kept;                   // scratch that was given up while a graph may hold it
    Scratch *call_scratch = nullptr;            // the set of the call being enqueued, until it has been looked at for a capture (call_mutex held)
    uint64_t use_counter = 0;
    std::vector<CachedWeights> weights;         // host-slice calls: uploaded weights by (pointer, length)
    size_t weights_cache_limit = size_t(64) << 30; // bytes kept before the least recently used goes
    uint64_t weight_uploads = 0;                // how many host-to-device weight copies the cache has done
    std::unordered_map<hipFunction_t, std::string> kernel_names;
    hipFunction_t last_kernel = nullptr;
    int num_cus = 256;
    uint32_t gemv_waves = 2048; // waves a GEMV launch aims to put on the device
    bool lm_head_fused = true;  // lm_head_argmax: candidates from the GEMV's own workgroups
    uint32_t call_elem = 0;     // element type of x and y of the matmul being enqueued (call_mutex held); 0 = f32
    // activations of the matmul being enqueued that are a gated product: x[r][i] = act(x[r][i]) * x[r][i + call_glu_off],
    // rows call_ldx elements apart (the input of a feed-forward block's down projection); 0 = plain
    uint32_t call_glu = 0, call_glu_off = 0, call_ldx = 0;
    TokenChoice *call_token = nullptr; // the one-row matmul being enqueued ends in the greedy token where its kernel can
    bool ffn_glu_load = true;   // "ffn_glu_load" = 0: the gate activation always runs as a kernel of its own
    hipFunction_t mm8s_gated[2][6] = {};        // streamed gate/up kernels with act(g) * u at the end of a tile pair [Q4_K, Q5_K][p1_e1_a, p1_e2_a, p2_e4_a, p1_e2, p2_e4, p1_e4]
    bool ffn_streamed = true;                   // "ffn_streamed" = 0: gllmq_ffn_swiglu never uses them
    hipFunction_t mm8s_e16[4][6] = {};          // streamed kernels over 16-bit activations and outputs [format][p1_e1_a, p1_e2_a, p2_e4_a, p1_e2, p2_e4, p1_e4]
    hipFunction_t mm8s_glu[4][4] = {};          // streamed kernels that take gated activations [format][p1_e2, p2_e4, p1_e4, p4_e4]
    // streamed kernels whose items are pairs of blocks of a tile of at most 16 weight rows (one
    // activation row) [format][p1_e1_a, p1_e2_a, p1_e2, p1_e4, p1_e2 and p1_e4 over gated activations,
    // the first four over a 16-bit element type]
    hipFunction_t mm8s_fold[4][10] = {};
    // streamed kernels whose workgroups share a row range and take a slice of K each (two to four
    // activation rows over few weight rows) [format][p1_e4, p2_e4][plain, gated activations]
    hipFunction_t mm8s_split[4][2][2] = {};
    hipFunction_t mm8s_group[4][2][3] = {};     // several matrices over the same rows [format, not Q6_K][f32, 16-bit][p1_e1_a, p1_e2_a, p2_e4_a]
    bool mm8s_q8_0 = true;                      // "mm8s_q8_0" = 0: Q8_0 never takes the streamed form
    bool mm8s_split_on = true;                  // "mm8s_split" = 0: such shapes stay on the fetch-and-compute form
    bool mm8s_fold_on = true;                   // "mm8s_fold" = 0: such tiles go block by block, half of the matrix-core columns idle
    hipFunction_t gemv_i8_glu[kNumFormats][2] = {};
    hipFunction_t gemv_i8_e16[kNumFormats][2] = {}; // the integer-dot GEMV over 16-bit activations and outputs
    bool elem_fused = true;     // "elem_fused" = 0: 16-bit elements always through conversion launches
    hipFunction_t convert_elem = nullptr;
    // Weight prefetch beside the dependent launches of a batch (touch.hip.inc).  Launches that
    // take part are numbered per context; a kernel of `announces` raises *progress to its number
    // when it starts, and the prefetch launch, on a stream of the context's own, reads the weights
    // of launch s while launch s - 1 runs.
    bool prefetch = false;                      // "prefetch" = 1: on (measured slower: the prefetch shares every CU's memory pipeline with the launch it runs beside)
    uint32_t prefetch_wgs = 0;                  // "prefetch_wgs": workgroups of the prefetch launch (0 = one per CU)
    uint32_t prefetch_threads = 64;             // "prefetch_threads": threads of each (64 .. 256)
    uint32_t prefetch_timeout_us = 200;         // "prefetch_timeout_us": longest wait for the launch before an entry's
    uint32_t prefetch_flags = 0;                // "prefetch_flags": TouchParams::flags
    bool prefetch_announce = true;              // "prefetch_announce" = 0: the launches stay silent (for measurements)
    uint32_t prefetch_min_kib = 4096;           // "prefetch_min_kib": smallest weight matrix worth a prefetch
    hipFunction_t touch = nullptr;
    hipStream_t side_stream = nullptr;
    hipEvent_t side_event = nullptr;
    unsigned long long *progress = nullptr;     // device
    unsigned long long launch_seq = 0;          // number of the last launch that was given one
    unsigned long long call_seq = 0;            // number the launch being enqueued announces itself under (0: none)
    std::unordered_set<hipFunction_t> announces;
    std::mutex err_mutex;
    std::string err;
};

namespace {

int fail(gllmq_ctx *ctx, int code, const char *fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    if (ctx) {
        std::lock_guard<std::mutex> g(ctx->err_mutex);
        ctx->err = buf;
    }
    return code;
}

} // namespace

extern "C" int gq_ctx_set_error(gllmq_ctx *ctx, int status, const char *message)
{
    return fail(ctx, status, "%s", message ? message : "");
}

extern "C" int gq_ctx_device(const gllmq_ctx *ctx) { return ctx ? ctx->device : -1; }

namespace {

#define GLLMQ_HIP(ctx, call)                                                                  \
    do {                                                                                      \
        hipError_t e_ = (call);                                                               \
        if (e_ != hipSuccess)                                                                 \
            return fail(ctx, GLLMQ_ERR_HIP, "%s failed: %s", #call, hipGetErrorString(e_));   \
    } while (0)

int get_function(gllmq_ctx *ctx, hipFunction_t *f, const char *name)
{
    hipError_t e = hipErrorNotFound;
    for (hipModule_t mod : ctx->modules) {
        if (!mod) continue;
        e = hipModuleGetFunction(f, mod, name);
        if (e == hipSuccess) break;
        (void)hipGetLastError();
    }
    if (e != hipSuccess)
        return fail(ctx, GLLMQ_ERR_HIP, "kernel %s missing from the code objects: %s", name,
                    hipGetErrorString(e));
    ctx->kernel_names[*f] = name;
    return GLLMQ_OK;
}

bool stream_is_capturing(void *stream)
{
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(static_cast<hipStream_t>(stream), &st) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return st != hipStreamCaptureStatusNone;
}

void carve_fixed(Scratch &S, void *base)
{
    uint8_t *b = static_cast<uint8_t *>(base);
    S.mm8_arrive = reinterpret_cast<uint32_t *>(b);
    S.argmax_keys = reinterpret_cast<uint64_t *>(b + kScratchArriveBytes);
    S.mm8_part = reinterpret_cast<float *>(b + kScratchArriveBytes + kScratchKeysBytes);
}

// Gives an allocation of a scratch set back.  What a graph may hold stays until the context goes: graphs are replayed when their
// owner likes, and the context does not learn of their end.  That is one set of allocations per capture at most.
void drop_scratch(gllmq_ctx *ctx, const Scratch &S, void *p)
{
    if (!p) return;
    if (std::find(S.in_graph.begin(), S.in_graph.end(), p) != S.in_graph.end()) ctx->kept.push_back(p);
    else (void)hipFree(p);
}

void free_scratch(gllmq_ctx *ctx, Scratch &S)
{
    if (S.fixed) return;
    for (void *p : { S.base, S.mmf, S.ffn, S.moe, S.elem, S.box }) drop_scratch(ctx, S, p);
    S = Scratch{};
}

// A launch of the current call uses its scratch set: where the stream is being captured, a graph will hold it.  Once a call, and only
// for calls that use scratch (the question takes 50 ns).
void note_scratch_use(gllmq_ctx *ctx, void *stream)
{
    Scratch *S = ctx->call_scratch;
    ctx->call_scratch = nullptr;
    if (S && stream_is_capturing(stream)) S->in_graph = { S->base, S->mmf, S->ffn, S->moe, S->elem, S->box };
}

// The scratch set of `stream` on this context (call_mutex held).  A stream the context has not
// seen gets a new set; beyond kMaxScratchSlots streams the least recently used set is given up
// after the device has drained.  Allocating is not possible while `stream` is being captured.
int acquire_scratch(gllmq_ctx *ctx, void *stream, Scratch **out)
{
    ++ctx->use_counter;
    for (Scratch &S : ctx->scratch)
        if (S.stream == static_cast<hipStream_t>(stream)) {
            S.last_use = ctx->use_counter;
            *out = ctx->call_scratch = &S;
            return GLLMQ_OK;
        }
    if (stream_is_capturing(stream))
        return fail(ctx, GLLMQ_ERR_INVALID,
                    "the context has no scratch for this stream yet and cannot allocate it during stream capture: "
                    "call gllmq_reserve (or run the call once) on this stream before capturing");
    GLLMQ_HIP(ctx, hipSetDevice(ctx->device));
    if (ctx->scratch.size() >= kMaxScratchSlots) {
        size_t lru = 0;
        for (size_t i = 1; i < ctx->scratch.size(); ++i)
            if (ctx->scratch[i].last_use < ctx->scratch[lru].last_use) lru = i;
        GLLMQ_HIP(ctx, hipDeviceSynchronize()); // its stream may be gone: wait for everything
        free_scratch(ctx, ctx->scratch[lru]);
        ctx->scratch.erase(ctx->scratch.begin() + static_cast<long>(lru));
    }
    Scratch S;
    S.stream = static_cast<hipStream_t>(stream);
    S.last_use = ctx->use_counter;
    GLLMQ_HIP(ctx, hipMalloc(&S.base, kScratchFixedBytes));
    hipError_t e = hipMemset(S.base, 0, kScratchArriveBytes);
    if (e != hipSuccess) {
        (void)hipFree(S.base);
        return fail(ctx, GLLMQ_ERR_HIP, "scratch: %s", hipGetErrorString(e));
    }
    carve_fixed(S, S.base);
    ctx->scratch.push_back(S);
    *out = ctx->call_scratch = &ctx->scratch.back();
    return GLLMQ_OK;
}

// Makes *buf, one of S's, hold at least `need` bytes for the call being enqueued.  Growing waits for the stream's earlier work (which may
// still use the old buffer; other streams have their own scratch), so it cannot happen while the
// stream is being captured, and never happens for a set of fixed size.
int grow_scratch(gllmq_ctx *ctx, const Scratch &S, void **buf, size_t *have, size_t need, void *stream, const char *what)
{
    if (ctx->probe) return GLLMQ_OK; // (a dry run of the dispatch allocates nothing)
    if (*have >= need) {
        note_scratch_use(ctx, stream);
        return GLLMQ_OK;
    }
    if (S.fixed)
        return fail(ctx, GLLMQ_ERR_BAD_SHAPE, "%s needs %zu bytes of scratch, the fixed scratch of this entry point has %zu",
                    what, need, *have);
    if (stream_is_capturing(stream))
        return fail(ctx, GLLMQ_ERR_INVALID,
                    "%s needs %zu bytes of scratch (the stream has %zu) and cannot allocate during stream capture: "
                    "call gllmq_reserve (or run the shape once) on this stream before capturing", what, need, *have);
    GLLMQ_HIP(ctx, hipSetDevice(ctx->device));
    if (*buf) {
        GLLMQ_HIP(ctx, hipStreamSynchronize(static_cast<hipStream_t>(stream)));
        drop_scratch(ctx, S, *buf);
        *buf = nullptr;
        *have = 0;
    }
    GLLMQ_HIP(ctx, hipMalloc(buf, need));
    *have = need;
    return GLLMQ_OK;
}

// `uses_scratch`: the kernel reads or writes the stream's scratch.
// Inside a batch of independent matmuls (ctx->overlap.on) the first launch of an entry is enqueued
// without the order that a stream otherwise imposes on its kernels, so that it may start while
// the kernels of earlier entries are still running (the gap between two kernels and the first and
// last microsecond of each, when few CUs stream, are what a decode layer's matmuls lose most to).
// Everything else is an ordinary launch, which starts after all earlier work of the stream has
// finished, unordered launches included.  Two kernels that use the scratch never overlap.
int launch2d(gllmq_ctx *ctx, hipFunction_t f, uint32_t grid_x, uint32_t grid_y, uint32_t block, uint32_t lds,
             void *stream, void *params, size_t params_size, bool uses_scratch = false)
{
    if (ctx->probe) {
        ++ctx->probe_launches;
        ctx->probe_fn = f;
        return GLLMQ_OK;
    }
    if (uses_scratch) note_scratch_use(ctx, stream);
    void *config[] = { HIP_LAUNCH_PARAM_BUFFER_POINTER, params, HIP_LAUNCH_PARAM_BUFFER_SIZE,
                       &params_size, HIP_LAUNCH_PARAM_END };
    gllmq_ctx::Overlap &ov = ctx->overlap;
    // (the launch without order takes the launch's size in threads as 32-bit numbers)
    const bool unordered = ov.on && ov.entry_first && ov.group_open && !(uses_scratch && ov.group_uses_scratch) &&
                           static_cast<uint64_t>(grid_x) * block <= 0xFFFFFFFFull;
    if (unordered) {
        GLLMQ_HIP(ctx, hipExtModuleLaunchKernel(f, grid_x * block, grid_y, 1, block, 1, 1, lds, static_cast<hipStream_t>(stream),
                                                nullptr, config, nullptr, nullptr, hipExtAnyOrderLaunch));
    } else {
        GLLMQ_HIP(ctx, hipModuleLaunchKernel(f, grid_x, grid_y, 1, block, 1, 1, lds, static_cast<hipStream_t>(stream),
                                             nullptr, config));
        ov.group_uses_scratch = false; // it waits for everything before it
    }
    ov.group_open = true;
    ov.entry_first = false;
    ov.group_uses_scratch = ov.group_uses_scratch || uses_scratch;
    ctx->last_kernel = f;
    return GLLMQ_OK;
}

int launch(gllmq_ctx *ctx, hipFunction_t f, uint32_t grid, uint32_t block, uint32_t lds, void *stream,
           void *params, size_t params_size, bool uses_scratch = false)
{
    return launch2d(ctx, f, grid, 1, block, lds, stream, params, params_size, uses_scratch);
}

bool aligned(const void *p, size_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

// Element `index` of activations or outputs whose element type is that of the call being enqueued
// (pointers are typed for the f32 case).
template <class T>
T *elem_at(uint32_t elem, T *base, size_t index)
{
    typedef typename std::conditional<std::is_const<T>::value, const uint8_t, uint8_t>::type Byte;
    return reinterpret_cast<T *>(reinterpret_cast<Byte *>(base) + index * (elem ? 2u : 4u));
}
template <class T>
T *elem_at(const gllmq_ctx *ctx, T *base, size_t index) { return elem_at(ctx->call_elem, base, index); }

// Elements between activation rows of the matmul being enqueued: k unless the caller says otherwise.
uint32_t row_stride_x(const gllmq_ctx *ctx, size_t k) { return ctx->call_ldx ? ctx->call_ldx : static_cast<uint32_t>(k); }

// What a kernel family answers when it would take the shape but cannot read gated activations:
// the caller then applies the gate in a launch of its own.
constexpr int kNeedPlainActivations = -2;

// Gated activations are read as aligned float4 from both factors.
bool glu_vector_ok(const gllmq_ctx *ctx) { return ctx->call_glu_off % 4u == 0u && ctx->call_ldx % 4u == 0u; }

// Shape-dependent fields of a GEMV launch over at most 64 groups (16384 elements) of K and
// m <= 2: how a row is split over lanes and waves, rows per workgroup, LDS.  `target_waves`
// is the number of waves the launch aims to put on the device.
struct GemvPlan {
    GemvParams P;
    uint32_t grid, threads, lds;
};

GemvPlan plan_gemv(const gllmq_ctx *ctx, uint32_t m, uint32_t n, uint32_t k, size_t row_bytes, uint32_t target_waves)
{
    GemvPlan L{};
    GemvParams &P = L.P;
    P.n = n;
    P.k = k;
    P.groups = (k + 255u) / 256u;
    P.row_bytes = static_cast<uint32_t>(row_bytes);
    const uint32_t parts = 4 * P.groups;
    if (parts >= 64) {
        P.ks = (parts + 63) / 64;
        P.rps = 1;
    } else {
        P.ks = 1;
        P.rps = 64 / parts;
    }
    const uint32_t rgs = std::max(1u, 4u / P.ks);
    const uint32_t nwaves = P.ks * rgs;
    const uint32_t row_steps = (n + P.rps - 1) / P.rps;
    uint32_t wgs = std::max(1u, target_waves / nwaves);
    wgs = std::min(wgs, (row_steps + rgs - 1) / rgs);
    uint32_t steps_per_wg = (row_steps + wgs * rgs - 1) / (wgs * rgs);
    P.rows_per_wg = steps_per_wg * rgs * P.rps;
    // partial sums of a K-split row meet in LDS: keep them within 8 KiB
    const uint32_t max_rows = 8192u / (4u * P.ks * m);
    if (P.ks > 1 && P.rows_per_wg > max_rows) P.rows_per_wg = std::max(rgs, max_rows / rgs * rgs);
    L.grid = (n + P.rows_per_wg - 1) / P.rows_per_wg;
    L.threads = 64 * nwaves;
    // integer-dot flavour: per part and activation row 48 plane words + 1 scale + 4 sums
    P.prep_words = ctx->gemv_f32 ? 0u : 53u * m * parts;
    L.lds = P.prep_words * 4u + (P.ks > 1 ? P.rows_per_wg * P.ks * m * 4u : 0u);
    return L;
}

int launch_gemv(gllmq_ctx *ctx, const Format &f, const uint8_t *w, size_t row_bytes, const float *x,
                float *y, uint32_t m, uint32_t n, uint32_t k, uint32_t ldx, uint32_t ldy, bool accumulate,
                bool act_bf16, void *stream)
{
    GemvPlan L = plan_gemv(ctx, m, n, k, row_bytes, ctx->gemv_waves);
    GemvParams &P = L.P;
    P.w = w;
    P.x = x;
    P.y = y;
    P.ldx = ldx;
    P.ldy = ldy;
    P.x_vec = aligned(x, 16) && (m == 1 || ldx % (ctx->call_elem ? 8 : 4) == 0);
    P.accumulate = accumulate ? 1u : 0u;
    P.act_bf16 = act_bf16 ? 1u : 0u;
    P.elem = ctx->call_elem;
    P.glu = ctx->call_glu;
    P.glu_off = ctx->call_glu_off;
    const int fi = format_index(f.dtype);
    hipFunction_t fn = ctx->gemv_f32 ? ctx->gemv[fi][m - 1]
                     : ctx->call_glu ? ctx->gemv_i8_glu[fi][m - 1]
                     : ctx->call_elem ? ctx->gemv_i8_e16[fi][m - 1]
                                      : ctx->gemv_i8[fi][m - 1];
    return launch(ctx, fn, L.grid, L.threads, L.lds, stream, &P, sizeof P);
}

int check_matmul_args(gllmq_ctx *ctx, const Format *f, const void *w, size_t w_bytes, const float *x,
                      float *y, uint32_t dtype, size_t m, size_t n, size_t k)
{
    if (!f)
        return fail(ctx, GLLMQ_ERR_UNIMPLEMENTED,
                    "quantized_matmul: ggml dtype %u is not covered (supported: Q8_0=8, Q4_K=12, Q5_K=13, Q6_K=14)",
                    dtype);
    if (m == 0 || n == 0) return GLLMQ_OK;
    if (!w || !x || !y) return fail(ctx, GLLMQ_ERR_INVALID, "quantized_matmul: NULL device pointer");
    if (k == 0) return fail(ctx, GLLMQ_ERR_BAD_SHAPE, "quantized_matmul: k = 0");
    if (n > 0x7FFFFFFFu || k > 0x7FFFFFFFu || m > 0x7FFFFFFFu)
        return fail(ctx, GLLMQ_ERR_BAD_SHAPE, "quantized_matmul: dimension exceeds 2^31-1");
    const size_t rb = gllmq_row_bytes(dtype, k);
    // the kernels address a workgroup's rows with 32-bit byte offsets from the first of them
    if (rb > (size_t(1) << 26))
        return fail(ctx, GLLMQ_ERR_BAD_SHAPE, "quantized_matmul: rows of %zu bytes (k=%zu) exceed the supported 64 MiB", rb, k);
    if (w_bytes < n * rb)
        return fail(ctx, GLLMQ_ERR_BAD_SHAPE,
                    "quantized_matmul: weight buffer has %zu bytes, n=%zu rows of k=%zu need %zu", w_bytes, n, k,
                    n * rb);
    if (!aligned(w, f->w_align) || (rb % f->w_align) != 0)
        return fail(ctx, GLLMQ_ERR_BAD_ALIGNMENT, "quantized_matmul: weights of %s must be %zu-byte aligned",
                    f->tag, f->w_align);
    if (!aligned(x, 4) || !aligned(y, 4))
        return fail(ctx, GLLMQ_ERR_BAD_ALIGNMENT, "quantized_matmul: activations and outputs must be 4-byte aligned");
    return -1; // go on
}

// Q4_K and Q5_K with up to 8 rows in the streamed form (mm8s.hip.inc): taken when the weight rows
// give every CU at least one 32-row tile, one pass over the weights serves all activation rows and
// the LDS ring holds enough items.  Returns -1 when the shape is not for it.
// `w2` != null selects the gated form: `w` holds the n gate rows, `w2` the n up rows, and
// y = act(gate . x) * (up . x) (Q4_K and Q5_K, up to four activation rows).
// `S` != null lets few weight rows under two to four rows of long activations share a row range
// among workgroups, a slice of K each (the sums meet in S->mm8_part).
int run_mm8s(gllmq_ctx *ctx, const Format &f, const uint8_t *w, const float *x, float *y, size_t m, size_t n, size_t k,
             bool act_bf16, void *stream, const uint8_t *w2 = nullptr, bool glu_relu = false, Scratch *S = nullptr,
             gq::Mm8sGroupParams *group = nullptr)
{
    const int kind = mm8_kind(f.dtype);
    const bool glu = w2 != nullptr;
    if (glu && ((kind != MM8_Q4K && kind != MM8_Q5K) || m > 4 || ctx->call_glu || ctx->call_elem)) return -1;
    if (!ctx->use_mm8 || !ctx->use_mm8s || (kind != MM8_Q4K && kind != MM8_Q5K && kind != MM8_Q6K && kind != MM8_Q8_0) || m == 0 || m > 8) return -1;
    if (kind == MM8_Q5K && ctx->mm8_q5k_min_m == 0) return -1;
    if (kind == MM8_Q6K && ctx->mm8_q6k_min_m == 0) return -1;
    // Q8_0: an item is a group of 8 blocks, so rows of whole groups only
    if (kind == MM8_Q8_0 && (ctx->mm8_q8_0_min_m == 0 || !ctx->mm8s_q8_0 || k % 256 != 0)) return -1;
    const int sfmt = kind == MM8_Q8_0 ? 3 : kind == MM8_Q6K ? 2 : kind == MM8_Q5K ? 1 : 0;
    const uint32_t pieces = sfmt == 3 ? gq::Mm8sFormat<3>::PIECES : sfmt == 2 ? gq::Mm8sFormat<2>::PIECES : sfmt == 1 ? gq::Mm8sFormat<1>::PIECES : gq::Mm8sFormat<0>::PIECES;
    const uint32_t subs = sfmt >= 2 ? 0u : 8u, zeros = sfmt == 2 ? gq::Mm8sFormat<2>::ZEROS : 0u;
    if (!aligned(x, 16) || k % 8 != 0) return -1;
    const uint32_t cus = static_cast<uint32_t>(ctx->num_cus);
    const uint32_t groups = static_cast<uint32_t>((k + 255) / 256), tiles = static_cast<uint32_t>((n + 31) / 32);
    // Every CU gets its share of the rows, as tiles of equal height; with fewer than 32 rows per CU
    // the tiles are lower than the 32 rows the matrix cores multiply, which costs nothing here (the
    // stream bounds the kernel).  Below `mm8s_min_rows` rows per CU the K split of the other form,
    // which keeps whole tiles and shares their blocks between CUs, is left to do it.
    // (two rows and more: from 4 rows per CU, where the K split of the other form and the GEMV are
    // behind: 2 x 4096 -> 1024 Q4_K 5.1-5.4 against 5.9-6.1 and 5.5-5.7 us)
    // (one row, in pairs of blocks: likewise from 4 rows per CU, 8192 -> 1536 Q4_K 5.8 against 7.3 us,
    // 14336 -> 1024 6.8 against 9.1, Q6_K 8.7 against 11.8)
    const bool may_fold = ctx->mm8s_fold_on && m == 1 && !glu;
    const uint32_t min_rows = (m >= 2 || may_fold) ? std::min(ctx->mm8s_min_rows, 4u) : ctx->mm8s_min_rows;
    if (n < static_cast<size_t>(min_rows) * cus) return -1;
    const uint32_t mm = static_cast<uint32_t>(m), pi = mm <= 2 ? 0u : (mm <= 4 ? 1u : 2u), pairs = 1u << pi;
    // K split: two to four activation rows of at least 32 blocks over 32-row tiles for at most half
    // of the CUs.  Every workgroup prepares the activations it multiplies, so whole rows of K per
    // workgroup cost rows x K of preparation in each (and four rows of 14336 do not fit the LDS);
    // `ksplit` workgroups share a tile and take a slice of at least 16 blocks each.
    uint32_t ksplit = 1;
    // (three and four rows of Q6_K: over fewer rows than that, 14336 -> 2048 14.9-15.3 against 17.0-18.5 us for the fetch-and-compute form,
    // 8192 -> 1024 10.3 against 12.1; 14336 -> 4096 18.9-19.3 against 19.9-20.4)
    if (S && ctx->mm8s_split_on && !glu && mm >= 2 && mm <= 4 &&
        (kind != MM8_Q6K || mm == 2 || (tiles * 2u < cus && groups < 64) || ctx->mm8s_all) &&
        groups >= 32 && tiles * 2u <= cus && tiles <= gq::MM8_SPLIT_MAX_LISTS)
        ksplit = std::min(cus / tiles, groups / 16u);
    // Slices of at least 8 blocks where those of 16 are for fewer than three quarters of the CUs (us, here and in brackets in the fetch-and-compute
    // form; three rows 9216 -> 2048 Q4_K 10.5 (13.2), Q5_K 10.9 (13.9), Q6_K 11.2 (15.3), Q8_0 11.8 (17.4), 14336 -> 1024 11.6 (13.5), 12.0 (14.1),
    // 12.3 (15.5), 12.7 (17.2)), below 64 blocks (16384 -> 1024 Q4_K 12.3 (10.7), Q8_0 13.4 (13.1)).  Q4_K and Q5_K: where the other form's slices are
    // of three passes of 8 blocks and not of two, whose operands it keeps in registers (11008 -> 1280 10.7 (10.3)).  Two rows: from where the
    // GEMV, which reads 16-bit elements itself, is not the other form.
    if (ksplit > 1 && groups < 64 && ksplit * tiles * 4u < cus * 3u && (mm > 2 || groups > 38) &&
        (kind == MM8_Q6K || kind == MM8_Q8_0 || (groups + 7u) / 8u % 2u == 1u))
        ksplit = std::min(cus / tiles, groups / 8u);
    while (ksplit > 1 && static_cast<size_t>(ksplit) * mm * n > gq::MM8_SPLIT_PART_FLOATS) --ksplit;
    // (slices for fewer than three quarters of the CUs leave too many of them idle: Q8_0 8192 -> 1024
    // at two rows 10.9 against 9.6 us for the GEMV; Q6_K at three rows 10.3 against 12.1)
    if (ksplit > 1 && !ctx->mm8s_all && (kind != MM8_Q6K || (mm == 2 && groups <= 38)) && ksplit * tiles * 4u < cus * 3u) ksplit = 1;
    // slices are of f32 activations: 16-bit ones are widened first, so that their call is of the f32 call's bits
    if (ksplit > 1 && ctx->call_elem) return kNeedPlainActivations;
    const bool split = ksplit > 1;
    const uint32_t kslice = (groups + ksplit - 1u) / ksplit, lds_groups = split ? kslice : groups; // blocks a workgroup prepares
    uint32_t rows_per_wg = split ? 32u : static_cast<uint32_t>((n + cus - 1) / cus);
    uint32_t grid = static_cast<uint32_t>((n + rows_per_wg - 1) / rows_per_wg);
    if (group) { // a workgroup's rows are of one matrix: the smallest share for which a workgroup per CU is enough
        for (;; ++rows_per_wg) {
            grid = 0;
            for (uint32_t i = 0; i < group->segs; ++i) {
                group->seg[i].first_wg = grid;
                grid += (group->seg[i].n + rows_per_wg - 1u) / rows_per_wg;
            }
            if (grid <= cus) break;
        }
    }
    const uint32_t wg_tiles = (rows_per_wg + 31u) / 32u, tile_rows = (rows_per_wg + wg_tiles - 1u) / wg_tiles;
    // One activation row over tiles of at most 16 weight rows: an item is a pair of blocks of the
    // tile, so that all 32 columns of the matrix cores carry weights (14336 -> 4096 is bound by the
    // arithmetic, not by the stream, when half of them idle).
    const bool fold = may_fold && tile_rows <= 16 && groups > 8; // (up to 8 blocks there is nothing to pair: a block per wave)
    if (may_fold && !fold && n < static_cast<size_t>(ctx->mm8s_min_rows) * cus) return -1;
    const uint32_t ipt = fold ? gq::mm8s_fold_pairs(groups) : lds_groups; // items per tile
    const uint32_t item_bytes = (fold ? 2u : 1u) * tile_rows * pieces * 16u; // a row of an item in LDS: its 16-byte pieces side by side
    const uint32_t fixed = gq::mm8s_lds_layout(lds_groups, mm, pairs, item_bytes, 0, subs, glu, zeros).total;
    const uint32_t items = (glu ? 2u : 1u) * wg_tiles * ipt; // (gated: a gate tile and an up tile per tile of rows)
    uint32_t slots = std::min(items, (160u * 1024u - std::min(fixed, 160u * 1024u)) / item_bytes);
    if (slots < items) slots -= slots % gq::MM8S_LOADERS; // a reused ring is a whole number of rounds of the loaders
    // Items a loader keeps unconfirmed.  One or two activation rows: one item (the wave requests an
    // item, waits for the one before it and confirms that: an arithmetic wave sees an item as soon
    // as it is there; with more outstanding the stream got no faster and the items later: one row
    // 4096 -> 4096 5.30 against 5.95 us, 4096 -> 14336 8.46 against 8.56, 4096 -> 128256 53.5
    // against 55.4, two rows of Q6_K 4096 -> 14336 12.7 against 13.4).  Three and four rows, whose
    // arithmetic per item is longer, keep about MM8S_DEPTH_BYTES worth of items on their way
    // (three rows 4096 -> 6144: 6.6 against 6.9 us with one), fewer when a reused ring is too short.
    // Pairs of Q4_K or Q5_K blocks of a long row (4.5 and 5.5 KiB an item, its 32 pieces a whole row
    // or eight blocks apart) come in late enough for two: 14336 -> 4096 Q4_K 9.1 against 10.1 us,
    // Q5_K 11.0 against 11.5 (Q6_K pairs, 6.6 KiB: 13.6 against 13.3; whole blocks of 24 rows,
    // 4096 -> 6144: 5.46 against 5.41).
    uint32_t depth = pi == 0 ? ((fold && item_bytes < 6144u) ? 2u : 1u)
                             : std::min(gq::MM8S_MAX_DEPTH, std::max(2u, (gq::MM8S_DEPTH_BYTES + item_bytes / 2u) / item_bytes));
    if (ctx->mm8s_depth) depth = std::min(gq::MM8S_MAX_DEPTH, ctx->mm8s_depth);
    while (depth > (split ? 1u : 2u) && slots < items && slots < gq::mm8s_min_slots(depth)) --depth;
    if (slots < items && slots < gq::mm8s_min_slots(depth)) return -1;
    const bool areg = ipt <= 16 && pi <= 1 && ctx->mm8s_areg && !(fold && ctx->call_glu) && !split;
    // Where the other kernels were timed faster (rows of 14336 and of 4096 elements over 4096 to
    // 128256 weight rows): several activation rows of long weight rows, whose preparation every
    // workgroup repeats in full (Q4_K 2 x 14336 -> 4096: 13.0 against 12.2 us).
    // Five to eight activation rows lead over at most 32 weight rows per CU or rows of at most 8
    // blocks (Q4_K 6 x 4096 -> 6144: 9.9 against 10.2 us, 8 x 2048 -> 14336: 10.6 against 12.0; 6 x
    // 4096 -> 14336: 15.0 against 14.3, 6 x 4096 -> 28672: 24.7 against 21.6), Q6_K over at most 32
    // weight rows per CU (5 x 4096 -> 4096: 11.7 against 12.0; 5 x 2048 -> 14336: 13.6 against 12.9).
    const bool few_rows = n <= static_cast<size_t>(32) * cus;
    if (!ctx->mm8s_all) {
        if (pi == 2 && !(few_rows || (groups <= 8 && kind != MM8_Q6K))) return -1;
        if (mm >= 2 && groups > 16 && !split && !(kind == MM8_Q6K && pi < 2)) return -1;
        // Tiles of fewer than 16 weight rows block by block, the matrix cores mostly idle, lose to
        // the K split of the other form for long rows (Q4_K 8192 -> 2048: 7.6 against 8.6 us) and
        // to the integer-dot GEMV for one row of Q5_K (4096 -> 2048: 4.8-5.2 against 5.6).  In
        // pairs of blocks they lead (8192 -> 2048: Q4_K 5.8 against 7.5, Q5_K 5.8 against 6.8;
        // 14336 -> 2048 Q4_K 7.1 against 9.9; Q5_K 4096 -> 2048 4.5 against 4.7).
        if (!fold && kind != MM8_Q6K && groups > 16 && rows_per_wg < 16) return -1;
        if (!fold && kind == MM8_Q5K && mm == 1 && n < static_cast<size_t>(12) * cus) return -1;
        // Q6_K: two to four rows everywhere (us, here and in brackets in the other forms: two rows 5120 -> 4096 7.5 (11.7), -> 28672 25 (38), 14336 ->
        // 6144 20 (26); three 5120 -> 6144 10.7 (13.5), four 4096 -> 14336 14.0 (17.0)).  One row: in pairs of blocks from 20 blocks on; from 40 on at
        // all heights; of 17 to 39 blocks over more than 24 weight rows per CU (5120 -> 8192 9.3 (12.2), 4864 -> 32000 25 (35)); up to 16 blocks
        // (3072 -> 1024 5.0 (5.4-6.2), -> 8192 6.4 (7.6), 2048 -> 14336 7.7 (8.4)), the shortest to 16 weight rows per CU and block (2048 -> 32000
        // 12.2 (13.0), 128256 42 (40); 1024 -> 14336 5.9 (6.5), 28672 8.9 (8.7)).  A wave of the GEMV takes 4096 elements of K, and where all its lanes
        // are at work it is ahead: rows of 4096, rows of 8192 over more than 56 weight rows per CU (14336 20.3 (21.8), 128256 153 (145)), and over more
        // than 64 also rows that fill all but a part of a block of it (3968 -> 8192 7.0 (7.6), 32000 22.7 (22.3), 64000 44.6 (40.8); 8064 -> 16384
        // 22.3 (23.9), 64000 82 (78)).  Rows of 14 and 15 blocks stay here, also where it is ahead (3584 -> 128256 74.1 (69.2)): its activations have a
        // bit less and its offset comes off in f32, for nearly twice the error (3584 normal activations 1.6e-7, 2.9e-7).
        if (kind == MM8_Q6K && mm == 1 && groups < 40 && !(fold && groups >= 20)) {
            const size_t rows = (n + cus - 1) / cus;
            const size_t most = k % 4096 == 0 ? (groups == 16 ? 0u : 56u) : groups % 16 == 0 ? 64u : groups <= 8 ? 16u * groups : SIZE_MAX;
            if (rows > most || (groups > 16 && rows <= 24)) return -1;
        }
        // Q8_0, two rows over at most 8 weight rows per CU: its GEMV stays ahead (4096 -> 1024: 5.9 against 7.1 us)
        if (kind == MM8_Q8_0 && mm == 2 && n <= static_cast<size_t>(8) * cus) return -1;
        // one short row over at most 4 weight rows per CU: the integer-dot GEMV stays ahead
        // (4096 -> 1024: Q4_K 4.6 against 5.0 us, Q5_K 4.9 against 5.0; 8192 -> 1024 Q4_K: 6.3 against 5.9 here)
        // (Q6_K leads here, 3072 -> 1024: 4.9-5.1 against 5.4-6.2)
        if (mm == 1 && rows_per_wg <= 4 && groups <= 16 && kind != MM8_Q6K) return -1;
    }
    const uint32_t steps = (((groups + 7u) / 8u + 1u) / 2u) * mm; // preparation steps per wave
    int variant;
    if (areg) variant = pi == 1 ? 2 : (steps <= 1 ? 0 : 1);
    else variant = (pi == 0 && steps > 2) ? 6 : 3 + static_cast<int>(pi);
    hipFunction_t fn = ctx->mm8s[sfmt][variant];
    if (split) {
        if (ctx->call_glu && !glu_vector_ok(ctx)) return kNeedPlainActivations;
        fn = ctx->mm8s_split[sfmt][pi][ctx->call_glu ? 1 : 0];
    } else if (fold) {
        // variants 0, 1 (registers), 3, 6 (LDS) of one activation row
        const int fv = variant <= 1 ? variant : variant == 3 ? 2 : 3;
        if (ctx->call_glu) {
            if (!glu_vector_ok(ctx)) return kNeedPlainActivations;
            fn = ctx->mm8s_fold[sfmt][fv + 2];
        } else {
            fn = ctx->mm8s_fold[sfmt][ctx->call_elem ? fv + 6 : fv];
        }
    } else if (glu) {
        const int gv = variant <= 4 ? variant : variant == 6 ? 5 : -1; // no gated build of p4_e4
        if (gv < 0) return -1;
        fn = ctx->mm8s_gated[sfmt][gv];
    } else if (ctx->call_glu) {
        const int gv = variant == 3 ? 0 : variant == 4 ? 1 : variant == 6 ? 2 : variant == 5 ? 3 : -1; // (the rest keep their planes in registers: rows of at most 4096 elements, not a down projection's)
        if (gv < 0 || !glu_vector_ok(ctx)) return kNeedPlainActivations;
        fn = ctx->mm8s_glu[sfmt][gv];
    } else if (ctx->call_elem) {
        const int ev = variant <= 4 ? variant : variant == 6 ? 5 : -1; // no 16-bit build of p4_e4
        if (ev < 0) return kNeedPlainActivations;
        fn = ctx->mm8s_e16[sfmt][ev];
    }
    Mm8Params P{};
    P.glu = ctx->call_glu;
    P.glu_off = ctx->call_glu_off;
    P.w = w;
    P.w2 = w2;
    P.glu_relu = glu_relu ? 1u : 0u;
    P.x = x;
    P.y = y;
    P.n = static_cast<uint32_t>(n);
    P.k = static_cast<uint32_t>(k);
    P.groups = groups;
    P.row_bytes = static_cast<uint32_t>(gllmq_row_bytes(f.dtype, k));
    P.m = mm;
    P.ldx = row_stride_x(ctx, k);
    P.ldy = static_cast<uint32_t>(n);
    P.tiles = tiles;
    P.grid = grid;
    P.act_bf16 = act_bf16 ? 1u : 0u;
    P.elem = ctx->call_elem;
    P.xrows = ctx->identity_rows;
    P.rows_per_wg = rows_per_wg;
    P.tile_rows = tile_rows;
    P.ring_slots = slots;
    P.wg_tiles = wg_tiles;
    P.last_wg_rows = P.n - (grid - 1u) * rows_per_wg;
    P.last_wg_tiles = (P.last_wg_rows + tile_rows - 1u) / tile_rows;
    const gq::Mm8sLds L = gq::mm8s_lds_layout(lds_groups, mm, pairs, item_bytes, slots, subs, glu, zeros);
    P.lds_ctrl = L.ctrl;
    P.lds_ring = L.ring;
    P.depth = depth;
    P.progress = ctx->call_seq && ctx->prefetch_announce ? ctx->progress : nullptr;
    P.progress_seq = ctx->call_seq;
    const uint32_t lds = L.total;
    if (group) {
        if (split || fold || !areg || variant > 2 || sfmt == 2 || act_bf16) return -1;
        group->p = P;
        return launch(ctx, ctx->mm8s_group[sfmt][ctx->call_elem ? 1 : 0][variant], grid, (gq::MM8S_CWAVES + gq::MM8S_LOADERS) * 64, lds, stream, group, sizeof *group, false);
    }
    if (split) {
        P.ksplit = ksplit;
        P.kslice_groups = kslice;
        P.part = S->mm8_part;
        P.arrive = S->mm8_arrive;
    }
    if (TokenChoice *c = ctx->call_token; c && c->y == y && c->n == n && mm == 1 && !split && !fold && !glu && !ctx->call_glu && !ctx->call_elem &&
                                          grid <= gq::ARGMAX_MAX_PARTS * gq::ARGMAX_MAX_ROWS && (variant == 0 || variant == 3 || variant == 6)) {
        // (register operands are of at most 16 blocks, which one row prepares in one step: never p1_e2_a)
        gq::Mm8sTokenParams T{ P, c->keys, c->ticket, c->token, c->value };
        c->made = true;
        return launch(ctx, ctx->mm8s_token[sfmt][variant / 3], grid, (gq::MM8S_CWAVES + gq::MM8S_LOADERS) * 64, lds, stream, &T, sizeof T, true);
    }
    return launch(ctx, fn, grid * ksplit, (gq::MM8S_CWAVES + gq::MM8S_LOADERS) * 64, lds, stream, &P, sizeof P, split);
}

// Q4_K, Q5_K and Q6_K on the int8 matrix cores, activation rows in passes of at most 8 (a pass keeps
// its rows' digit planes in LDS and reads the weights once).  Returns -1 when the shape does
// not fit the kernel (LDS for the prepared activations, alignment), so that the caller
// takes the GEMV kernels.
// `w2` != null selects the gated form: `w` holds the n gate rows, `w2` the n up rows, and
// y = act(gate . x) * (up . x) (Q4_K and Q5_K, one pass only).
int run_mm8(gllmq_ctx *ctx, Scratch &S, const Format &f, const uint8_t *w, const float *x, float *y, size_t m, size_t n,
            size_t k, bool act_bf16, void *stream, bool one_pass_only = false, const uint8_t *w2 = nullptr,
            bool glu_relu = false)
{
    const int kind = mm8_kind(f.dtype);
    if (!ctx->use_mm8 || kind < 0) return -1;
    const bool glu = w2 != nullptr;
    if (glu && kind != MM8_Q4K && kind != MM8_Q5K) return -1;
    if (glu) one_pass_only = true;
    // The row thresholds below say where the GEMV kernels are as fast; that holds while a GEMV
    // workgroup's prepared activations (848 bytes per row and 256 elements) leave room for
    // several workgroups per CU.  Two rows of more than 9728 elements do not (one workgroup of
    // four waves per CU: 35 against 25 us for Q6_K 14336 -> 4096), so they come here.
    const bool gemv_cramped = 848u * m * ((k + 255) / 256) > 64u * 1024u;
    // One row of 40 blocks and more over few weight rows (a down projection): the K split below
    // gives every CU a slice, and the Q5_K and Q6_K kernels here then beat the GEMV, which walks
    // such a row with three or four waves (11008 -> 4096: Q6_K 15.5 against 17.6 us, Q5_K 13.2
    // against 16.6; 14336 -> 4096: 17.5 against 17.7 and 14.5 against 15.5).
    const bool long_single = m == 1 && (k + 255) / 256 >= 40 && ctx->mm8_ksplit_max > 1 &&
                             ((n + 31) / 32) * 2 <= static_cast<size_t>(ctx->num_cus);
    if (kind == MM8_Q6K && (ctx->mm8_q6k_min_m == 0 || (m < ctx->mm8_q6k_min_m && !gemv_cramped && !long_single))) return -1;
    if (kind == MM8_Q5K && !glu && (ctx->mm8_q5k_min_m == 0 || (m < ctx->mm8_q5k_min_m && !long_single))) return -1;
    if (kind == MM8_Q8_0 && (ctx->mm8_q8_0_min_m == 0 || (m < ctx->mm8_q8_0_min_m && !gemv_cramped))) return -1;
    if (kind == MM8_Q8_0 && k < 256) return -1; // its fetch window is one whole group of 8 blocks
    // One row of Q4_K over at most 4 weight rows per CU: a workgroup's prologue and the meeting of
    // the K slices outweigh what the matrix cores save, the integer-dot GEMV is ahead
    // (4096 -> 1024: 4.5-4.7 against 5.1-5.3 us, 8192 -> 1024: 6.2-6.3 against 7.4, 14336 -> 512: 8.4 against 9.4).
    if (kind == MM8_Q4K && m == 1 && !glu && ctx->mm8_small_to_gemv && n <= static_cast<size_t>(4) * static_cast<size_t>(ctx->num_cus)) return -1;
    if (!aligned(x, 16) || k % 8 != 0) return -1; // the kernel loads activations as aligned vectors
    const uint32_t groups = static_cast<uint32_t>((k + 255) / 256);
    // K split: with tiles for at most half of the CUs, 2..8 workgroups share each tile and take
    // a slice of K each (whole passes of 8 blocks); the slices meet inside the launch.  The
    // meeting costs about 2 us, so a slice keeps at least two passes, unless only a shorter slice
    // lets the prepared activations of all rows fit the LDS (one pass over the weights then beats
    // the alternatives by more than that).
    const uint32_t tiles = static_cast<uint32_t>((n + 31) / 32), ppt_row = (groups + 7u) / 8u;
    auto pairs_for = [](uint32_t rows) { return rows <= 2 ? 1u : (rows <= 4 ? 2u : 4u); };
    const uint32_t m_pass = static_cast<uint32_t>(std::min<size_t>(m, 8));
    uint32_t ksplit = 1, slice_passes = ppt_row;
    if (!glu && ctx->mm8_ksplit_max > 1 && ppt_row >= 2 && (kind != MM8_Q8_0 || k % 256 == 0)) {
        auto fits = [&](uint32_t slices) {
            const uint32_t passes = (ppt_row + slices - 1) / slices;
            return mm8_lds_bytes(std::min(groups, passes * 8u), m_pass, pairs_for(m_pass), kind) <= 160u * 1024u;
        };
        const uint32_t most = std::min(ppt_row, ctx->mm8_ksplit_max);
        uint32_t want = 1;
        if (tiles * 2u <= static_cast<uint32_t>(ctx->num_cus))
            want = std::max(1u, std::min({ static_cast<uint32_t>(ctx->num_cus) / tiles, ppt_row / 2u, most }));
        while (want < most && !fits(want)) ++want;
        // more workgroups than CUs run in rounds: whole rounds beat one and a half
        const uint32_t cus = static_cast<uint32_t>(ctx->num_cus);
        if (want > 1 && want * tiles > cus && tiles <= cus)
            for (uint32_t w2 = want; w2 <= most; ++w2)
                if ((w2 * tiles) % cus == 0) { want = w2; break; }
        if (fits(want)) {
            slice_passes = (ppt_row + want - 1) / want;
            ksplit = (ppt_row + slice_passes - 1) / slice_passes; // every slice gets at least one pass
        }
        if (static_cast<size_t>(ksplit) * m_pass * n > gq::MM8_SPLIT_PART_FLOATS) ksplit = 1;
        if (ksplit == 1) slice_passes = ppt_row;
    }
    const uint32_t lds_groups = ksplit > 1 ? std::min(groups, slice_passes * 8u) : groups;
    // Rows per pass: as many as the prepared activations leave room for in the 160 KiB of LDS.
    uint32_t rows_per_pass = m_pass;
    while (rows_per_pass > 0 && mm8_lds_bytes(lds_groups, rows_per_pass, pairs_for(rows_per_pass), kind) > 160u * 1024u)
        --rows_per_pass;
    if (rows_per_pass == 0) return -1;
    if (one_pass_only && rows_per_pass < m) return -1;
    if (ctx->call_elem) return kNeedPlainActivations; // these kernels read and write f32
    // gated activations (a feed-forward block's down projection): passes of five to eight rows have a kernel for them
    if (ctx->call_glu) {
        const size_t last_pass = m - ((m - 1) / rows_per_pass) * rows_per_pass;
        if (glu || rows_per_pass < 5 || last_pass < 5 || !glu_vector_ok(ctx) || !ctx->mm8_gated_p4[kind]) return kNeedPlainActivations;
    }
    for (size_t m0 = 0; m0 < m; m0 += rows_per_pass) {
        const uint32_t mm = static_cast<uint32_t>(std::min<size_t>(rows_per_pass, m - m0));
        const int pi = mm <= 2 ? 0 : (mm <= 4 ? 1 : 2);
        const uint32_t pairs = 1u << pi;
        const uint32_t lds = mm8_lds_bytes(lds_groups, mm, pairs, kind);
        Mm8Params P{};
        P.ksplit = ksplit;
        P.kslice_groups = slice_passes * 8u;
        P.part = S.mm8_part;
        P.arrive = S.mm8_arrive;
        P.w2 = w2;
        P.glu_relu = glu_relu ? 1u : 0u;
        P.glu = ctx->call_glu;
        P.glu_off = ctx->call_glu_off;
        P.w = w;
        P.x = x + m0 * row_stride_x(ctx, k);
        P.y = y + m0 * n;
        P.n = static_cast<uint32_t>(n);
        P.k = static_cast<uint32_t>(k);
        P.groups = groups;
        P.row_bytes = static_cast<uint32_t>(gllmq_row_bytes(f.dtype, k));
        P.m = mm;
        P.ldx = row_stride_x(ctx, k);
        P.ldy = static_cast<uint32_t>(n);
        P.tiles = (P.n + 31u) / 32u;
        P.act_bf16 = act_bf16 ? 1u : 0u;
        P.xrows = ctx->identity_rows;
        // preparation steps per wave: two 256-element blocks per step
        const uint32_t ppt = slice_passes, steps = ((ppt + 1u) / 2u) * mm;
        int ei = steps <= 1 ? 0 : (steps <= 2 ? 1 : 2);
        while (ei < 2 && !ctx->mm8[kind][pi][ei]) ++ei; // not every (pairs, early) pair is built
        const int gi = kind == MM8_Q5K ? 1 : 0;
        uint32_t grid = std::min<uint32_t>(P.tiles, std::max(1u, static_cast<uint32_t>(ctx->num_cus) / ksplit));
        if (ksplit > 1) grid = std::min(grid, gq::MM8_SPLIT_MAX_LISTS);
        P.grid = grid; // workgroups per slice: launch index = tile list * ksplit + slice
        hipFunction_t fn = glu ? ctx->mm8_glu[gi][pi][ei] : ctx->mm8[kind][pi][ei];
        // The register-resident variants are compiled for a fixed number of passes per tile and
        // take a tile's pass from the item's position in the register ring; a last K slice with
        // fewer passes than the others would break that, so such a split runs the LDS variants.
        const bool even_slices = ksplit == 1 || ppt_row % slice_passes == 0;
        if (pi <= 1 && ppt <= 2 && even_slices)
            fn = glu ? ctx->mm8_glu_areg[gi][pi][ei][ppt - 1] : ctx->mm8_areg[kind][pi][ei][ppt - 1];
        if (ctx->call_glu) fn = ctx->mm8_gated_p4[kind]; // (pi == 2: checked above)
        int rc = launch(ctx, fn, grid * ksplit, 512, lds, stream, &P, sizeof P, ksplit > 1);
        if (rc != GLLMQ_OK) return rc;
    }
    return GLLMQ_OK;
}

constexpr uint32_t kMmfMaxRowTiles = 16384;

// Launch shape of the GEMM for one matmul, and the scratch it needs.
struct MmfPlan {
    uint32_t groups, row_tiles, ksplit, bps;
    size_t img_bytes, need;
};

MmfPlan plan_mmf(const gllmq_ctx *ctx, size_t m, size_t n, size_t k)
{
    MmfPlan L{};
    L.groups = static_cast<uint32_t>((k + 255) / 256);
    L.row_tiles = static_cast<uint32_t>((n + 255) / 256);
    uint32_t ksplit = std::max(1u, static_cast<uint32_t>(ctx->num_cus) / std::max(1u, L.row_tiles));
    ksplit = std::min(ksplit, L.groups);
    L.bps = (L.groups + ksplit - 1) / ksplit;
    L.ksplit = (L.groups + L.bps - 1) / L.bps; // every workgroup gets at least one block
    const size_t rows = std::min<size_t>(m, 64);
    // scratch: the activation images of one pass, then the partial sums
    L.img_bytes = static_cast<size_t>(L.groups) * mmf_image_bytes(rows <= 32 ? 1u : 2u);
    L.need = L.img_bytes + (L.ksplit > 1 ? static_cast<size_t>(L.ksplit) * rows * n * 4 : 0);
    return L;
}

int run_mmf(gllmq_ctx *ctx, Scratch &S, const Format &f, const uint8_t *w, const float *x, float *y, size_t m, size_t n,
            size_t k, bool act_bf16, void *stream, size_t min_m = 9)
{
    if (!ctx->use_mmf || m < min_m) return -1;
    const int fmt = f.dtype == T_Q8_0 ? 3 : f.dtype == T_Q6_K ? 2 : f.dtype == T_Q5_K ? 1 : 0;
    if (fmt == 3 && k < 256) return -1; // the Q8_0 fetch window is one whole group of 8 blocks
    if (!aligned(x, 16) || k % 4 != 0) return -1; // activation rows are loaded as aligned float4
    if (ctx->call_glu && !glu_vector_ok(ctx)) return kNeedPlainActivations;
    const MmfPlan L = plan_mmf(ctx, m, n, k);
    const uint32_t groups = L.groups, row_tiles = L.row_tiles, ksplit = L.ksplit, bps = L.bps;
    if (row_tiles > kMmfMaxRowTiles) return -1;
    // the GEMM kernels address weight rows with 32-bit byte offsets from the start of the matrix
    if (n * gllmq_row_bytes(f.dtype, k) > 0xFFFFFFFFull) return -1;
    const size_t rows_per_pass = 64, img_bytes = L.img_bytes;
    int grc = grow_scratch(ctx, S, &S.mmf, &S.mmf_bytes, L.need, stream, "quantized_matmul (GEMM)");
    if (grc != GLLMQ_OK) return grc;
    for (size_t m0 = 0; m0 < m; m0 += rows_per_pass) {
        const uint32_t mm = static_cast<uint32_t>(std::min(rows_per_pass, m - m0));
        const uint32_t mt = mm <= 32 ? 1u : 2u;
        MmfParams P{};
        P.w = w;
        P.elem = ctx->call_elem;
        P.ldx = row_stride_x(ctx, k);
        P.x = elem_at(ctx, x, m0 * P.ldx);
        P.y = elem_at(ctx, y, m0 * n);
        P.ximg = static_cast<uint8_t *>(S.mmf);
        P.partial = reinterpret_cast<float *>(static_cast<uint8_t *>(S.mmf) + img_bytes);
        P.n = static_cast<uint32_t>(n);
        P.k = static_cast<uint32_t>(k);
        P.groups = groups;
        P.row_bytes = static_cast<uint32_t>(gllmq_row_bytes(f.dtype, k));
        P.m = mm;
        P.ldy = static_cast<uint32_t>(n);
        P.row_tiles = row_tiles;
        P.ksplit = ksplit;
        P.blocks_per_split = bps;
        P.act_bf16 = act_bf16 ? 1u : 0u;
        MmfPrepParams Q{ P.x, P.ximg, mm, P.k, P.ldx, P.act_bf16, P.elem, ctx->call_glu, ctx->call_glu_off };
        int rc = launch2d(ctx, ctx->mmf_prep[mt - 1], groups, 16, 64, 0, stream, &Q, sizeof Q, true);
        if (rc != GLLMQ_OK) return rc;
        rc = launch(ctx, ctx->mmf_q4k[fmt][mt - 1][act_bf16 ? 1 : 0], row_tiles * ksplit, 512, mmf_lds_bytes(mt, fmt), stream,
                    &P, sizeof P, true);
        if (rc == GLLMQ_OK && ksplit > 1) {
            MmfReduceParams R{};
            R.seg[0] = gq::MmfReduceSeg{ P.partial, P.y, P.n, 0u };
            R.segs = 1;
            R.m = mm;
            R.ksplit = ksplit;
            R.elem = P.elem;
            const uint64_t quads = (static_cast<uint64_t>(mm) * n + 3) / 4;
            rc = launch(ctx, ctx->mmf_reduce, static_cast<uint32_t>((quads + 255) / 256), 256, 0, stream, &R, sizeof R, true);
        }
        if (rc != GLLMQ_OK) return rc;
    }
    return GLLMQ_OK;
}

// Whether [a, a + an) and [b, b + bn) share a byte.
bool ranges_meet(const void *a, size_t an, const void *b, size_t bn)
{
    const uintptr_t a0 = reinterpret_cast<uintptr_t>(a), b0 = reinterpret_cast<uintptr_t>(b);
    return a0 < b0 + bn && b0 < a0 + an;
}

// One weight matrix of a GEMM launch.
struct MmfwMatrix {
    const uint8_t *w;
    float *y;
    size_t n;
};

// Launch geometry of the GEMM for more rows (mmfw.hip.inc), for matrices of n[0 .. count) rows that
// share their activations, and the scratch it needs.  ok = false: not for it.
struct MmfwPlan {
    bool ok = false;
    uint32_t groups = 0, planes = 2, mt = 1, n_tiles = 0, ksplit = 1, bps = 0, band = 4;
    uint32_t run = 0; // blocks whose sums are taken in one run; 0: all of a slice's
    uint32_t run_tiles = 1; // weight tiles that a workgroup multiplies one after the other
    size_t n_sum = 0; // weight rows of all matrices
    size_t rows = 0; // activation rows per pass (all of them, unless the images would pass 1 GiB or the scratch has no room: mmfw_fit)
    size_t img_bytes = 0, inv_bytes = 0, part_bytes = 0;
    size_t need() const { return img_bytes + inv_bytes + part_bytes; }
};

int mmf_format(uint32_t dtype) { return dtype == T_Q8_0 ? 3 : dtype == T_Q6_K ? 2 : dtype == T_Q5_K ? 1 : 0; }

// Whether a workgroup may take several weight tiles one after the other (mmfw_may_run): all of K, long enough for requests to reach
// into the next tile only.
bool mmfw_run_ok(int fmt, int planes, uint32_t mt, uint32_t groups, uint32_t ksplit)
{
    return ksplit == 1 && groups >= 4 && gq::mmfw_may_run(fmt, planes, static_cast<int>(mt), false);
}

uint32_t mmfw_inv_ld(size_t rows) { return static_cast<uint32_t>((rows + 31) / 32 * 32); }

void mmfw_size(MmfwPlan &L, size_t rows)
{
    L.rows = rows;
    const size_t image = L.planes == 2 ? gq::MmfwImage<2>::bytes : gq::MmfwImage<1>::bytes;
    L.img_bytes = (rows + 31) / 32 * L.groups * image;
    // (a workgroup fetches the inverse scales of its rows as one KiB)
    L.inv_bytes = (static_cast<size_t>(L.groups) * mmfw_inv_ld(rows) * 4 + 1024 + 255) & ~size_t(255);
    L.part_bytes = L.ksplit > 1 ? static_cast<size_t>(L.ksplit) * rows * L.n_sum * 4 : 0;
}

constexpr size_t kMmfwMaxImages = size_t(1) << 30;

// Fewer rows per pass, until the pass needs `limit` bytes at most (false: one row of tiles needs more).  Tiles and slices stay
// what they are, so the results do.
bool mmfw_shrink(MmfwPlan &L, size_t limit)
{
    const size_t step = 32u * L.mt;
    while ((L.img_bytes > kMmfwMaxImages || L.need() > limit) && L.rows > step)
        mmfw_size(L, std::max(step, (L.rows / 2 + step - 1) / step * step));
    return L.img_bytes < 0xFFFFFFFFull && L.need() <= limit;
}

// Most bytes that the sums of K slices take; a plan has no more slices than that allows.  32 MiB cost 3000 plans of 9 to 2048
// rows 0.6 % in the mean by the cost model, 16 MiB 1.3 %, 64 MiB 0.5 %.
size_t mmfw_most_slices(const gllmq_ctx *ctx, size_t m) { return static_cast<size_t>(ctx->num_cus) * 1024u * (m <= 32 ? 32u : 128u); }

// Decoded weights (mmfx.hip.inc): bytes, and the most that a call has of them at a time; a matrix beyond that goes in slabs of its rows.
constexpr size_t kMmfxMaxBytes = size_t(128) << 20;
size_t mmfx_bytes(size_t n, uint32_t groups) { return (n + 31) / 32 * groups * gq::MmfxRecord::bytes; }

// Scratch that any call of up to `m` rows of `k` elements fits, in one pass, and from 33 rows on any call of more rows in passes:
// what is grown for one call or reserved serves every other one of as many rows, whatever its weight rows, matrices, slices
// and element type.  (The one-launch GEMM of 9 to 16 rows has sums of 64 bytes per weight row and 2048 of K: beyond 2^28 weights they
// may be more than this.)
size_t mmfw_reserve(const gllmq_ctx *ctx, size_t m, size_t k)
{
    const size_t groups = (k + 255) / 256, tiles = m <= 32 ? 1 : std::max<size_t>((m + 31) / 32, gq::MMFW_MAX_MT);
    return std::min(tiles * groups * gq::MmfwImage<2>::bytes, kMmfwMaxImages) + ((groups * tiles * 128 + 1024 + 255) & ~size_t(255)) + mmfw_most_slices(ctx, m);
}

// Additions one after the other, in the mean over the blocks, when `blocks` of them are added up in runs of `run`
// (0: in one), and `slices` of such sums.
double mmfw_chain(uint32_t blocks, uint32_t run, uint32_t slices)
{
    const double slice = slices > 1u ? 0.5 * (slices + 1u) : 0.0;
    if (run == 0u || run >= blocks) return 0.5 * (blocks + 1u) + slice;
    return 0.5 * (run + 1u) + 0.5 * ((blocks + run - 1u) / run + 1u) + slice;
}

// Q6_K and Q8_0: blocks of a run, such that no output's additions form a longer chain than in the form of 64-row passes,
// whose slices of K are short because it has few workgroups otherwise.  Error against 64 bits, 2048 f32 rows of 4096 x 14336:
// Q6_K 1.64e-7 in one run, 1.18e-7 in runs of eight, 1.23e-7 in that form; Q8_0 1.64e-7, 1.19e-7, 1.23e-7.  It takes
// registers that four row tiles do not have: 571 -> 657 us, 535 -> 626.  Q4_K and Q5_K, whose blocks themselves cost more,
// stay below that form without (2.27e-7 against 2.33e-7).
// `bar`: that form's shortest chain over the launch's matrices (mmfw_chain_bar).
uint32_t mmfw_run(uint32_t bps, uint32_t ksplit, double bar)
{
    if (mmfw_chain(bps, 0, ksplit) <= bar) return 0;
    uint32_t run = 2;
    for (uint32_t r = 4; r <= 16; r *= 2) // the longest that is short enough, else the best
        if (mmfw_chain(bps, r, ksplit) <= std::max(bar, mmfw_chain(bps, run, ksplit))) run = r;
    return run;
}
double mmfw_chain_bar(const gllmq_ctx *ctx, int fmt, const size_t *n, int count, size_t k)
{
    double bar = 1e300;
    for (int i = 0; i < count && fmt >= 2; ++i) {
        const MmfPlan O = plan_mmf(ctx, 64, n[i], k);
        bar = std::min(bar, mmfw_chain(O.bps, 0, O.ksplit));
    }
    return bar;
}

// Sizes the plan's passes for the scratch that there is, where no more can be had: a capture cannot allocate, and a block of fixed
// size does not grow.  False: not even the smallest pass fits.
bool mmfw_fit(const gllmq_ctx *ctx, const Scratch &S, MmfwPlan &L, void *stream)
{
    if (L.need() <= S.mmf_bytes || ctx->probe || !(S.fixed || stream_is_capturing(stream))) return true;
    return mmfw_shrink(L, S.mmf_bytes);
}

MmfwPlan plan_mmfw(const gllmq_ctx *ctx, uint32_t dtype, size_t m, const size_t *n, int count, size_t k, bool hi_only)
{
    MmfwPlan L;
    const int fmt = mmf_format(dtype);
    size_t &n_sum = L.n_sum, tiles = 0;
    for (int i = 0; i < count; ++i) {
        n_sum += n[i];
        tiles += (n[i] + gq::MMFW_TILE_ROWS - 1) / gq::MMFW_TILE_ROWS;
    }
    if (!ctx->use_mmf || !ctx->use_mmfw || m == 0 || n_sum == 0 || tiles > 0xFFFFFFu) return L;
    if (fmt == 3 && k < 256) return L; // the Q8_0 window is one whole group of 8 blocks
    if (static_cast<uint64_t>(gllmq_row_bytes(dtype, k)) * gq::MMFW_TILE_ROWS > 0xFFFFFFFFull) return L;
    L.groups = static_cast<uint32_t>((k + 255) / 256);
    L.planes = hi_only ? 1u : 2u;
    L.n_tiles = static_cast<uint32_t>(tiles);
    const uint32_t row_tiles = static_cast<uint32_t>((m + 31) / 32);
    // Activation tiles per workgroup and slices of K by a cost model (us): a block of K takes a workgroup what the table says, or
    // the weights' way from memory where that is longer; a workgroup starts and ends in `start`; the slices of K meet
    // through memory.  The numbers are fitted to what they decide: 135 000 calls of 6852 shapes (9 to 2048 rows, 512 to 28672 x 1024
    // to 14336, all formats, f32 and bf16; every number of tiles and up to 20 slices) were timed, half of the shapes
    // searched for the numbers whose choices are shortest, the other half kept to check: choices 0.50 % longer than the best
    // one in the mean, 1.43 % with block times measured one by one before (1.5 to 2.7 us for one tile).  So they are no times of a block: Q8_0
    // in one tile has more for one plane than for two.  They were fitted ahead of workgroups that make their images (MmfwOwn); `prepare_us` is later.
    // Slices and runs decide the order of the sums, tiles do not; so a call of 16-bit elements has the slices of the f32 call
    // whose bits it has to give: those with which the two together are shortest.  (3000 plans of 9 to 2048 rows by the
    // model, against slices of their own: 0.5 % longer in the mean, one in a hundred by more than a tenth.)
    const double cus = ctx->num_cus;
    const double w_us = find_format(dtype)->group_bytes * 256.0 * cus / 5.85e6; // 5.85 TB/s over all CUs
    static const double block_us[4][2][gq::MMFW_MAX_MT] = { // [Q4_K, Q5_K, Q6_K, Q8_0][one plane, two][tiles - 1]
        { { 1.65, 2.07, 2.88, 3.96 }, { 1.50, 2.98, 4.69, 5.95 } },
        { { 1.76, 2.11, 2.95, 3.13 }, { 1.92, 2.98, 4.03, 5.36 } },
        { { 2.70, 3.80, 5.41, 7.22 }, { 2.97, 4.70, 7.05, 9.40 } },
        { { 3.45, 3.46, 4.16, 6.34 }, { 2.21, 5.04, 6.30, 7.98 } },
    };
    const double crowd_us = fmt == 0 ? 0.4 : 0.0; // more per block with every CU busy
    // A launch that prepares the activations, where workgroups do not do it themselves.  It takes 3 to 4 us, but costs of that and more
    // make slices too short where the numbers above are off: 300 shapes of 9 to 200 rows, against choices without it: 1.5 us 0.21 % shorter in
    // the mean, the worst 1.8 % longer (65 x 8317 x 3840 Q6_K 39.8 us, 39.7, but 42.5 from 3 us on), the best 23 % shorter (37 x 7136 x 1056
    // Q8_0 19.3, 15.1).  900 other shapes: no cost 0.17 % longer in the mean, the worst 29 %; 2.5 to 4.5 us level with 1.5.
    // Calls that cannot do without the launch (gated activations, ones rounded to bf16) have the same plan: counted for those, it trades few
    // slices of one row tile for about twice as many of two, one plan in eighty.  40 such shapes of 33 to 118 rows, whole feed-forward
    // blocks 0.4 % shorter in the mean (2.8 shorter to 4.3 longer), rounded matmuls 2.4 % longer (3.2 shorter to 12.3 longer).
    const double prepare_us = 1.5;
    const double start = 5.64, bar = mmfw_chain_bar(ctx, fmt, n, count, k);
    double best = 1e300;
    for (uint32_t ks = 1; ks <= std::min(L.groups, 32u); ++ks) {
        const uint32_t bps = (L.groups + ks - 1) / ks;
        if ((L.groups + bps - 1) / bps != ks) continue; // every slice has a block
        if (ctx->mmfw_ksplit && ks != std::min(ctx->mmfw_ksplit, L.groups)) continue;
        const size_t slices = ks > 1 ? static_cast<size_t>(ks) * n_sum * 4 : 0;
        if (slices * m > mmfw_most_slices(ctx, m) && !ctx->mmfw_ksplit) continue;
        const double meet = ks > 1 ? 0.64 + 2.2 * ks * static_cast<double>(m) * static_cast<double>(n_sum) / 1.0e6 : 0.0;
        const uint32_t run = mmfw_run(bps, ks, bar);
        double of[2] = { 1e300, 1e300 }; // one plane, two
        uint32_t of_mt[2] = { 0, 0 }, of_run[2] = { 1, 1 };
        for (uint32_t mt = 1; mt <= static_cast<uint32_t>(gq::MMFW_MAX_MT); ++mt) {
            if (ctx->mmfw_mt ? mt != ctx->mmfw_mt : (mt > row_tiles)) continue;
            if (run && !gq::mmfw_runs(static_cast<int>(mt)) && !ctx->mmfw_mt) continue;
            const uint64_t m_tiles = (row_tiles + mt - 1) / mt, items = m_tiles * tiles * ks;
            if (m_tiles * tiles > 0x7FFFFFFu) continue;
            // no plan that the fixed scratch cannot take in passes of one row of tiles (the call through it has the same one)
            if (static_cast<size_t>(L.groups) * mt * (gq::MmfwImage<2>::bytes + 128u) + 2048u + slices * std::min<size_t>(m, 32u * mt) >
                GLLMQ_NOALLOC_SCRATCH_BYTES - kScratchFixedBytes)
                continue;
            const double busy = std::min(1.0, static_cast<double>(items) / cus);
            for (int pl = 0; pl < 2; ++pl) {
                const double tile = bps * (std::max(block_us[fmt][pl][mt - 1], w_us * busy) + crowd_us * busy);
                // (runs of weight tiles only where they save rounds)
                const uint32_t most = mmfw_run_ok(fmt, pl + 1, mt, L.groups, ks) ? static_cast<uint32_t>(std::min<uint64_t>(16, (items + static_cast<uint64_t>(cus) - 1) / static_cast<uint64_t>(cus))) : 1u;
                for (uint32_t in_row = 1; in_row <= most; ++in_row) {
                    const double prepare = mt == 1 && bps <= mmfw_own_blocks(fmt, pl + 1) ? 0.0 : prepare_us;
                    const double us = std::ceil(static_cast<double>(m_tiles * ((tiles + in_row - 1) / in_row) * ks) / cus) * (in_row * tile + start) + meet + prepare;
                    if (us < of[pl]) {
                        of[pl] = us;
                        of_mt[pl] = mt;
                        of_run[pl] = in_row;
                    }
                }
            }
        }
        if (of[0] + of[1] < best) {
            best = of[0] + of[1];
            L.mt = of_mt[L.planes - 1];
            L.run_tiles = of_run[L.planes - 1];
            L.ksplit = ks;
            L.bps = bps;
            L.run = run;
        }
    }
    if (best == 1e300) return L;
    const uint32_t m_tiles = (row_tiles + L.mt - 1) / L.mt;
    L.band = std::min(m_tiles, 4u);
    mmfw_size(L, m);
    L.ok = mmfw_shrink(L, SIZE_MAX);
    return L;
}

// Whether workgroups prepare their activations themselves (MmfwOwn): one row tile, slices short enough for the images to stay in
// LDS, rows that sixteen-byte loads take piece by piece.  Where it can be done it is ahead, by 0.8 to
// 4.5 us of 13 to 30, by format and length of the slices (MmfwOwn).
bool mmfw_takes_own(const gllmq_ctx *ctx, const MmfwPlan &L, int fmt, size_t m, size_t k, size_t ldx, size_t x_bytes)
{
    return ctx->use_mmfw_own && L.mt == 1 && L.bps <= mmfw_own_blocks(fmt, static_cast<int>(L.planes)) && k * x_bytes % 16 == 0 && ldx * x_bytes % 16 == 0 &&
           m * ldx * x_bytes <= 0xFFFFFFFFull;
}

// Makes one of the stream's buffers hold `need` bytes if they can be had: not under capture, and where the allocation is refused it stays what it is.
void grow_if_possible(gllmq_ctx *ctx, const Scratch &S, void **have, size_t *have_bytes, size_t need, void *stream)
{
    if (*have_bytes >= need || S.fixed || ctx->probe || stream_is_capturing(stream)) return;
    void *buf = nullptr;
    if (hipSetDevice(ctx->device) != hipSuccess || hipMalloc(&buf, need) != hipSuccess) {
        (void)hipGetLastError();
        return;
    }
    if (*have && hipStreamSynchronize(static_cast<hipStream_t>(stream)) != hipSuccess) { // (earlier work's error, which the next launch reports)
        (void)hipFree(buf);
        return;
    }
    drop_scratch(ctx, S, *have);
    *have = buf;
    *have_bytes = need;
}

// ... the GEMM's, where decoded weights are to go, the call's own matrices' (`need` depends on them).  Without, the call has the same bits.
void grow_for_decoded(gllmq_ctx *ctx, Scratch &S, size_t need, void *stream) { grow_if_possible(ctx, S, &S.mmf, &S.mmf_bytes, need, stream); }

// ... enough for any call of up to `m` rows and `n` weight rows in up to MMFW_MAX_SEGS matrices
size_t mmfx_reserve(const gllmq_ctx *ctx, uint32_t dtype, size_t m, size_t n, size_t k)
{
    if (mmf_format(dtype) != 2 || !ctx->use_mmf || !ctx->use_mmfw || !ctx->mmfx_min_m || m < ctx->mmfx_min_m) return 0;
    return mmfw_reserve(ctx, m, k) - mmfw_most_slices(ctx, m) + 256 +
           std::min(mmfx_bytes(n + 32u * (gq::MMFW_MAX_SEGS - 1), static_cast<uint32_t>((k + 255) / 256)), kMmfxMaxBytes);
}

// How a GEMM over many activation rows of Q6_K decodes its weights first.  mt = 0: it does not.
struct MmfxPlan {
    uint32_t mt = 0;
    size_t slab_rows = 0; // weight rows decoded at a time (several matrices: all of them)
    size_t bytes = 0;     // of a slab
};

// From 1024 rows on: decoding costs 0.5 us per million weights, the GEMM then takes a fifth less.  us, decoding and GEMM, and without (f32, 4096 x
// 14336): 2048 rows 30 + 520, 625; 1024 rows 30 + 262, 313; 14336 x 4096: 1000 rows 30 + 275, 323, 512 rows 30 + 139, 164; one plane, 2048 rows of
// 4096 x 4096 9 + 108, 142.
MmfxPlan plan_mmfx(const gllmq_ctx *ctx, const MmfwPlan &L, int fmt, const size_t *n, int count, size_t m)
{
    MmfxPlan X;
    if (fmt != 2 || L.ksplit != 1 || !ctx->mmfx_min_m || m < ctx->mmfx_min_m || ctx->mmfw_mt == 1) return X;
    if (count == 1) {
        X.slab_rows = std::min(n[0], kMmfxMaxBytes / mmfx_bytes(32, L.groups) * 32 / gq::MMFW_TILE_ROWS * gq::MMFW_TILE_ROWS);
        X.bytes = mmfx_bytes(X.slab_rows, L.groups);
    } else {
        for (int i = 0; i < count; ++i) X.bytes += mmfx_bytes(n[i], L.groups);
        X.slab_rows = X.bytes <= kMmfxMaxBytes ? L.n_sum : 0;
    }
    if (X.slab_rows == 0) return X;
    // Tiles by rounds of workgroups; us per block of K as timed (14336 x 4096, 4096 x 14336).  They do not touch the order of the sums.
    static const double block_us[2][gq::MMFW_MAX_MT - 1] = { { 3.3, 4.4, 6.4 }, { 4.6, 6.3, 8.4 } }; // [one plane, two][tiles - 2]
    const uint32_t row_tiles = static_cast<uint32_t>((std::min(L.rows, m) + 31) / 32);
    double best = 1e300;
    for (uint32_t mt = 2; mt <= static_cast<uint32_t>(gq::MMFW_MAX_MT); ++mt) {
        if (ctx->mmfw_mt ? mt != ctx->mmfw_mt : (L.run && !gq::mmfw_runs(static_cast<int>(mt)))) continue;
        const double rounds = std::ceil(static_cast<double>((row_tiles + mt - 1) / mt) * L.n_tiles / ctx->num_cus);
        const double us = rounds * (L.groups * block_us[L.planes - 1][mt - 2] + 5.6);
        if (us < best) {
            best = us;
            X.mt = mt;
        }
    }
    return X;
}

// The sums of K slices of a feed-forward block's gate and up rows, left in the scratch for the preparation of the down
// projection, which adds them up while it applies the gate: a launch less, and the sums' way to memory and back.
struct MmfwSlices {
    size_t next_need = 0;    // scratch that the down projection needs,
    size_t next_reserve = 0; // and that it grows the scratch to
    size_t next_decoded = 0; // bytes of its decoded weights, which it cannot grow the scratch for with the sums there
    const float *at = nullptr;
    uint32_t slices = 0;     // 0: none were left
    size_t used = 0;         // bytes of the scratch in use
};

// The images of activation rows (mmfw.hip.inc).  16-bit elements have one plane and a launch of their own.
int launch_mmfw_prep(gllmq_ctx *ctx, gq::MmfwPrepParams &Q, bool hi_only, uint32_t row_tiles, void *stream)
{
    const bool e16 = Q.elem != 0 && !Q.glu;
    return launch2d(ctx, e16 ? ctx->mmfw_prep_e16 : ctx->mmfw_prep[hi_only ? 1 : 0], Q.groups, row_tiles, (e16 ? gq::MMFW_PREP16_WAVES : gq::MMFW_PREP_WAVES) * 64, 0,
                    stream, &Q, sizeof Q, true);
}

// The GEMM over `count` matrices of one format and K that share their activations: one launch that
// prepares the activation images (not where workgroups do: mmfw_takes_own), one that multiplies, and one that adds the slices of K where
// there are any.  Returns -1 for what it does not take.
// `elem_x`, `elem_y`: element types of the activations and of the outputs.
// `leave`: the sums of slices may stay where they are (where both calls fit the scratch in one pass each; it is not grown for that: what
// it is grown to depends on rows and K alone, so that no call of as many or fewer rows frees what a graph holds); `take`: the
// activations are such sums.
int run_mmfw(gllmq_ctx *ctx, Scratch &S, const Format &f, const MmfwMatrix *mats, int count, const float *x, uint32_t elem_x,
             uint32_t elem_y, size_t m, size_t k, bool act_bf16, void *stream, size_t min_m, MmfwSlices *leave = nullptr, const MmfwSlices *take = nullptr)
{
    if (!ctx->use_mmf || !ctx->use_mmfw || m < min_m) return -1;
    if (!aligned(x, 16) || k % 4 != 0) return -1; // activation rows are loaded as aligned float4
    if (ctx->call_glu && !glu_vector_ok(ctx)) return kNeedPlainActivations;
    size_t n[gq::MMFW_MAX_SEGS];
    for (int i = 0; i < count; ++i) n[i] = mats[i].n;
    const bool hi_only = act_bf16 || (elem_x && !ctx->call_glu);
    MmfwPlan L = plan_mmfw(ctx, f.dtype, m, n, count, k, hi_only);
    if (!L.ok || (!take && !mmfw_fit(ctx, S, L, stream))) return -1;
    if (S.fixed && plan_mmf(ctx, m, n[0], k).need > S.mmf_bytes) return -1; // beyond what that entry point takes, in passes or not
    int rc = GLLMQ_OK;
    const bool may_leave = leave && L.ksplit > 1 && L.rows >= m;
    const size_t used = (L.need() + 255) & ~size_t(255);
    size_t reserve = std::max(L.need(), mmfw_reserve(ctx, m, k));
    if (may_leave) reserve = std::max(reserve, leave->next_reserve);
    const int fmt = mmf_format(f.dtype);
    MmfxPlan X = plan_mmfx(ctx, L, fmt, n, count, m);
    const size_t decoded_at = (take ? take->used : 0) + used;
    if (X.mt && !take) grow_for_decoded(ctx, S, std::max(reserve, decoded_at + X.bytes), stream);
    if (may_leave && leave->next_decoded) grow_for_decoded(ctx, S, std::max(reserve, used + ((leave->next_need + 255) & ~size_t(255)) + leave->next_decoded), stream);
    if (!take && S.mmf_bytes < reserve && !S.fixed && !stream_is_capturing(stream)) rc = grow_scratch(ctx, S, &S.mmf, &S.mmf_bytes, reserve, stream, "quantized_matmul (GEMM)");
    if (rc != GLLMQ_OK) return rc;
    if (decoded_at + X.bytes > S.mmf_bytes && !ctx->probe) X.mt = 0;
    const bool leaves = may_leave && used + leave->next_need <= S.mmf_bytes;
    uint8_t *scratch = static_cast<uint8_t *>(S.mmf) + (take ? take->used : 0);
    const uint32_t ldx = row_stride_x(ctx, k);
    const size_t x_bytes = elem_x ? 2 : 4;
    bool own = mmfw_takes_own(ctx, L, fmt, m, k, ldx, x_bytes) && !take && !ctx->call_glu && !act_bf16;
    // outputs over the activations: what one workgroup stores another may still have to read
    for (int i = 0; i < count && L.ksplit == 1; ++i) own = own && !ranges_meet(mats[i].y, m * mats[i].n * (elem_y ? 2 : 4), x, m * ldx * x_bytes);
    if (X.mt) own = false;
    uint8_t *decoded = static_cast<uint8_t *>(S.mmf) + decoded_at;
    const bool slabs = X.mt && count == 1 && X.slab_rows < n[0];
    const uint32_t mt = X.mt ? X.mt : L.mt;
    auto decode = [&](int i, size_t row0, size_t rows, size_t at) -> int {
        const uint32_t row_bytes = static_cast<uint32_t>(gllmq_row_bytes(f.dtype, k));
        gq::MmfxDecodeParams D{ mats[i].w + row0 * row_bytes, decoded + at, static_cast<uint32_t>(rows), L.groups, row_bytes };
        return launch2d(ctx, ctx->mmfx_decode, (L.groups + gq::MMFX_DECODE_WAVES - 1) / gq::MMFX_DECODE_WAVES, static_cast<uint32_t>((rows + 31) / 32),
                        gq::MMFX_DECODE_WAVES * 64, 0, stream, &D, sizeof D, true);
    };
    if (X.mt && !slabs) {
        size_t at = 0;
        for (int i = 0; i < count && rc == GLLMQ_OK; ++i) {
            rc = decode(i, 0, n[i], at);
            at += mmfx_bytes(n[i], L.groups);
        }
        if (rc != GLLMQ_OK) return rc;
    }
    for (size_t m0 = 0; m0 < m; m0 += L.rows) {
        const uint32_t mm = static_cast<uint32_t>(std::min(L.rows, m - m0));
        gq::MmfwPrepParams Q{};
        Q.x = elem_at(elem_x, x, m0 * ldx);
        Q.ximg = scratch;
        Q.inv = reinterpret_cast<float *>(scratch + L.img_bytes);
        Q.m = mm;
        Q.k = static_cast<uint32_t>(k);
        Q.ldx = ldx;
        Q.groups = L.groups;
        Q.inv_ld = mmfw_inv_ld(L.rows);
        Q.act_bf16 = act_bf16 ? 1u : 0u;
        Q.elem = ctx->call_glu ? 0u : elem_x;
        Q.natural = fmt == 2 ? 1u : 0u; // a sub-block of Q6_K is one K step
        Q.lo_first = gq::mmfw_lo_first(fmt, static_cast<int>(L.planes), static_cast<int>(L.mt)) ? 1u : 0u;
        Q.glu = ctx->call_glu;
        Q.glu_off = ctx->call_glu_off;
        if (take) {
            Q.slices = take->slices;
            Q.slice_ld = static_cast<uint32_t>(m * k);
        }
        const uint32_t row_tiles = (mm + 31u) / 32u;
        if (!own) rc = launch_mmfw_prep(ctx, Q, hi_only, row_tiles, stream);
        if (rc != GLLMQ_OK) return rc;
        gq::MmfwParams P{};
        P.ximg = scratch;
        P.inv = Q.inv;
        if (own) {
            P.x = reinterpret_cast<const uint8_t *>(Q.x);
            P.x_row_bytes = static_cast<uint32_t>(ldx * x_bytes);
            P.x_elem = Q.elem;
        }
        P.segs = static_cast<uint32_t>(count);
        P.groups = L.groups;
        P.row_bytes = static_cast<uint32_t>(gllmq_row_bytes(f.dtype, k));
        P.m = mm;
        P.k = Q.k;
        P.row_tiles = row_tiles;
        P.inv_ld = Q.inv_ld;
        P.m_tiles = (row_tiles + mt - 1u) / mt;
        P.n_tiles = L.n_tiles;
        P.ksplit = L.ksplit;
        P.blocks_per_split = L.bps;
        P.run_mask = L.run ? L.run - 1u : ~0u;
        P.run_tiles = std::min(mmfw_run_ok(fmt, hi_only ? 1 : 2, L.mt, L.groups, L.ksplit) ? std::max(1u, ctx->mmfw_run ? ctx->mmfw_run : L.run_tiles) : 1u, P.n_tiles);
        P.n_runs = (P.n_tiles + P.run_tiles - 1u) / P.run_tiles;
        P.items = P.m_tiles * P.n_runs * L.ksplit;
        P.band = std::min(L.band, P.m_tiles);
        P.elem = elem_y;
        float *part = reinterpret_cast<float *>(scratch + L.img_bytes + L.inv_bytes);
        uint32_t tile0 = 0;
        for (int i = 0; i < count; ++i) {
            gq::MmfwSeg &G = P.seg[i];
            G.w = mats[i].w;
            G.y = elem_at(elem_y, mats[i].y, m0 * mats[i].n);
            G.partial = part;
            G.n = static_cast<uint32_t>(mats[i].n);
            G.tile0 = tile0;
            tile0 += (G.n + gq::MMFW_TILE_ROWS - 1u) / gq::MMFW_TILE_ROWS;
            part += static_cast<size_t>(L.ksplit) * mm * G.n;
        }
        if (X.mt) {
            size_t at = 0;
            for (int i = 0; i < count; ++i) {
                P.seg[i].w = decoded + at;
                at += mmfx_bytes(n[i], L.groups);
            }
            for (size_t row0 = 0; row0 < L.n_sum; row0 += X.slab_rows) {
                if (slabs) { // weight tile 0 of the launch is tile row0 / 256 of the matrix
                    const size_t rows = std::min(X.slab_rows, n[0] - row0);
                    const uint32_t first = static_cast<uint32_t>(row0 / gq::MMFW_TILE_ROWS);
                    rc = decode(0, row0, rows, 0);
                    if (rc != GLLMQ_OK) return rc;
                    P.seg[0].first_record_row = static_cast<uint32_t>(row0 / 32);
                    P.seg[0].tile0 = 0u - first;
                    P.n_tiles = P.n_runs = static_cast<uint32_t>((rows + gq::MMFW_TILE_ROWS - 1) / gq::MMFW_TILE_ROWS);
                    P.items = P.m_tiles * P.n_runs;
                }
                rc = launch(ctx, ctx->mmfx[mt - 2][hi_only ? 1 : 0], (P.items + 7u) / 8u * 8u, gq::MMFW_WAVES * 64, mmfx_lds_bytes(hi_only ? 1 : 2, mt), stream, &P, sizeof P, true);
                if (rc != GLLMQ_OK) return rc;
            }
            continue;
        }
        rc = launch(ctx, own ? ctx->mmfw_own[fmt][hi_only ? 1 : 0] : ctx->mmfw[fmt][L.mt - 1][hi_only ? 1 : 0], (P.items + 7u) / 8u * 8u, gq::MMFW_WAVES * 64,
                    own ? mmfw_own_lds(fmt, hi_only ? 1 : 2) : mmfw_lds_bytes(fmt, hi_only ? 1 : 2, L.mt), stream, &P, sizeof P, true);
        if (leaves) {
            leave->at = P.seg[0].partial;
            leave->slices = L.ksplit;
            leave->used = used;
        } else if (rc == GLLMQ_OK && L.ksplit > 1) {
            gq::MmfReduceParams R{};
            uint32_t wgs = 0;
            for (int i = 0; i < count; ++i) {
                R.seg[i] = gq::MmfReduceSeg{ P.seg[i].partial, P.seg[i].y, P.seg[i].n, wgs };
                wgs += static_cast<uint32_t>((static_cast<uint64_t>(mm) * P.seg[i].n + 1023) / 1024);
            }
            R.segs = P.segs;
            R.m = mm;
            R.ksplit = L.ksplit;
            R.elem = P.elem;
            rc = launch(ctx, ctx->mmf_reduce, wgs, 256, 0, stream, &R, sizeof R, true);
        }
        if (rc != GLLMQ_OK) return rc;
    }
    return GLLMQ_OK;
}

// Launch geometry of the streamed GEMM (mmfs.hip.inc) for one matmul; ok = false when the shape is
// left to the three-launch form.
struct MmfsPlan {
    bool ok = false;
    uint32_t groups = 0, ksplit = 1, rows_per_wg = 0, grid = 0, wg_tiles = 0, tile_rows = 0, slots = 0, depth = 2,
             lds_ctrl = 0, lds_ring = 0, lds = 0;
    size_t img_bytes = 0, need = 0; // scratch: one image per block of K (32 activation rows per launch), then the slice sums
};

MmfsPlan plan_mmfs(const gllmq_ctx *ctx, const Format &f, size_t m, size_t n, size_t k)
{
    MmfsPlan L;
    const int fmt = f.dtype == T_Q5_K ? 1 : f.dtype == T_Q4_K ? 0 : -1;
    if (!ctx->use_mmf || !ctx->use_mmfs || fmt < 0 || m == 0 || n == 0) return L;
    const uint32_t cus = static_cast<uint32_t>(ctx->num_cus);
    if (n < static_cast<size_t>(ctx->mmfs_min_rows) * cus) return L;
    // Timed against the three-launch form at 16 and 32 rows: ahead on matrices of up to 6144 x 4096
    // (32 rows: 13.2 against 22.0 us at 4096 x 4096, 15.5 against 19.2 at 6144 x 4096: two launches
    // instead of three, no pass over partial sums in a launch of its own), behind from 14336 x 4096
    // on (24.6 against 23.9 us; 38.1 against 34.0 at 28672 x 4096; 31.8 against 26.7 at 4096 x 14336):
    // one arithmetic wave per SIMD does not hide its own dependent instructions once the stream
    // is long enough to matter.
    if (!ctx->mmfs_all && n * k > (40ull << 20)) return L;
    L.groups = static_cast<uint32_t>((k + 255) / 256);
    // a workgroup multiplies four blocks of K (one per arithmetic wave); the row ranges are as many
    // as give every CU a workgroup
    L.ksplit = (L.groups + gq::MMFS_CWAVES - 1u) / gq::MMFS_CWAVES;
    const uint32_t ranges = std::max(1u, cus / L.ksplit);
    L.rows_per_wg = static_cast<uint32_t>((n + ranges - 1) / ranges);
    L.grid = static_cast<uint32_t>((n + L.rows_per_wg - 1) / L.rows_per_wg);
    // the loader's 32-bit offsets stay inside a workgroup's rows
    if (static_cast<size_t>(L.rows_per_wg) * gllmq_row_bytes(f.dtype, k) > 0xFFFFFFFFull) return L;
    L.wg_tiles = (L.rows_per_wg + 31u) / 32u;
    L.tile_rows = (L.rows_per_wg + L.wg_tiles - 1u) / L.wg_tiles; // equal heights, <= 32
    if (L.ksplit > 1 && L.grid > kScratchArriveBytes / 4u) return L; // one arrival counter per row range
    const uint32_t pieces = fmt == 1 ? gq::Mm8sFormat<1>::PIECES : gq::Mm8sFormat<0>::PIECES;
    const uint32_t item_bytes = L.tile_rows * pieces * 16u;
    L.lds_ctrl = 0;
    L.lds_ring = (static_cast<uint32_t>(sizeof(gq::Mm8sCtrl)) + gq::MMFS_RED_BUFS * gq::MMFS_CWAVES * 4096u + 1023u) & ~1023u;
    const uint32_t items = L.wg_tiles * gq::MMFS_CWAVES;
    L.slots = std::min(items, (160u * 1024u - L.lds_ring) / item_bytes);
    if (L.slots < items) L.slots -= L.slots % gq::MMFS_LOADERS; // a reused ring is a whole number of rounds of the loaders
    L.depth = ctx->mm8s_depth ? std::min(gq::MM8S_MAX_DEPTH, ctx->mm8s_depth) : 1u; // as for the one-row kernels (12.7 against 12.8 us at 32 x 4096 x 4096, 10.5 against 10.8 at 2048 x 2048)
    while (L.depth > 2u && L.slots < items && L.slots < gq::mm8s_min_slots(L.depth)) --L.depth;
    if (L.slots < items && L.slots < gq::mm8s_min_slots(L.depth)) return L;
    L.lds = L.lds_ring + L.slots * item_bytes;
    L.img_bytes = static_cast<size_t>(L.groups) * gq::MmfLanes::image;
    L.need = L.img_bytes + (L.ksplit > 1 ? static_cast<size_t>(L.ksplit) * L.grid * L.wg_tiles * 4096u : 0u);
    L.ok = true;
    return L;
}

// Q4_K and Q5_K, more than 8 activation rows, from `mmfs_min_rows` weight rows per CU up: the
// streamed GEMM, 32 activation rows per launch (a preparation launch for their images, then the
// GEMM, which leaves y complete).  Returns -1 when the shape is left to run_mmf.
int run_mmfs(gllmq_ctx *ctx, Scratch &S, const Format &f, const uint8_t *w, const float *x, float *y, size_t m, size_t n,
             size_t k, bool act_bf16, void *stream, size_t min_m = 9)
{
    if (m < min_m) return -1;
    if (!aligned(x, 16) || k % 4 != 0) return -1; // activation rows are loaded as aligned float4
    const MmfsPlan L = plan_mmfs(ctx, f, m, n, k);
    if (!L.ok) return -1;
    if (ctx->call_glu && !glu_vector_ok(ctx)) return kNeedPlainActivations;
    int grc = grow_scratch(ctx, S, &S.mmf, &S.mmf_bytes, L.need, stream, "quantized_matmul (GEMM)");
    if (grc != GLLMQ_OK) return grc;
    const int fmt = f.dtype == T_Q5_K ? 1 : 0;
    for (size_t m0 = 0; m0 < m; m0 += 32) {
        const uint32_t mm = static_cast<uint32_t>(std::min<size_t>(32, m - m0));
        MmfPrepParams Q{ elem_at(ctx, x, m0 * row_stride_x(ctx, k)), static_cast<uint8_t *>(S.mmf), mm, static_cast<uint32_t>(k),
                         row_stride_x(ctx, k), act_bf16 ? 1u : 0u, ctx->call_elem, ctx->call_glu, ctx->call_glu_off };
        int rc = launch2d(ctx, ctx->mmf_prep_lanes, L.groups, 16, 64, 0, stream, &Q, sizeof Q, true);
        if (rc != GLLMQ_OK) return rc;
        Mm8Params P{};
        P.w = w;
        P.x = static_cast<const float *>(S.mmf); // the images
        P.y = elem_at(ctx, y, m0 * n);
        P.elem = ctx->call_elem;
        P.n = static_cast<uint32_t>(n);
        P.k = static_cast<uint32_t>(k);
        P.groups = L.groups;
        P.row_bytes = static_cast<uint32_t>(gllmq_row_bytes(f.dtype, k));
        P.m = mm;
        P.ldx = static_cast<uint32_t>(k);
        P.ldy = static_cast<uint32_t>(n);
        P.grid = L.grid;
        P.ksplit = L.ksplit;
        P.kslice_groups = gq::MMFS_CWAVES;
        P.part = reinterpret_cast<float *>(static_cast<uint8_t *>(S.mmf) + L.img_bytes);
        P.arrive = S.mm8_arrive;
        P.rows_per_wg = L.rows_per_wg;
        P.tile_rows = L.tile_rows;
        P.ring_slots = L.slots;
        P.wg_tiles = L.wg_tiles;
        P.last_wg_rows = P.n - (L.grid - 1u) * L.rows_per_wg;
        P.last_wg_tiles = (P.last_wg_rows + L.tile_rows - 1u) / L.tile_rows;
        P.lds_ctrl = L.lds_ctrl;
        P.lds_ring = L.lds_ring;
        P.depth = L.depth;
        rc = launch(ctx, ctx->mmfs[fmt][act_bf16 ? 1 : 0], L.grid * L.ksplit, (gq::MMFS_CWAVES + gq::MMFS_LOADERS) * 64, L.lds,
                    stream, &P, sizeof P, true);
        if (rc != GLLMQ_OK) return rc;
    }
    return GLLMQ_OK;
}

// Q4_K and Q5_K, 9 to 16 rows of plain activations, from `mmfr_min_rows` weight rows per CU up: the
// streamed GEMM whose arithmetic waves prepare their own activations (mmfr.hip.inc), one launch and
// nothing else.  A workgroup multiplies a slice of K of eight blocks (a block per arithmetic wave);
// the slices of a row range meet through the scratch.  Returns -1 for what it does not take.
int run_mmfr(gllmq_ctx *ctx, Scratch &S, const Format &f, const uint8_t *w, const float *x, float *y, size_t m, size_t n,
             size_t k, bool act_bf16, void *stream, size_t min_m = 9)
{
    const int fmt = f.dtype == T_Q5_K ? 1 : f.dtype == T_Q4_K ? 0 : -1;
    // (17 rows and more: two ways of sharing a block between two waves were built and timed slower than the three-launch form)
    if (!ctx->use_mmf || !ctx->use_mmfr || fmt < 0 || m < min_m || m > 16 || n == 0) return -1;
    if (act_bf16 || ctx->call_glu) return -1; // plain activations
    const uint32_t ldx = row_stride_x(ctx, k);
    if (!aligned(x, 16) || k % 4 != 0 || ldx % 4 != 0) return -1; // activation rows are loaded as aligned float4
    const uint32_t cus = static_cast<uint32_t>(ctx->num_cus);
    if (n < static_cast<size_t>(ctx->mmfr_min_rows) * cus) return -1;
    const uint32_t groups = static_cast<uint32_t>((k + 255) / 256);
    const uint32_t pieces = fmt == 1 ? gq::Mm8sFormat<1>::PIECES : gq::Mm8sFormat<0>::PIECES;
    const uint32_t sb = gq::MMFR_CWAVES; // blocks of a slice
    const uint32_t ksplit = (groups + sb - 1u) / sb;
    const uint32_t ranges = std::max(1u, cus / ksplit);
    const uint32_t rows_per_wg = static_cast<uint32_t>((n + ranges - 1) / ranges);
    const uint32_t grid = static_cast<uint32_t>((n + rows_per_wg - 1) / rows_per_wg);
    // the loader's 32-bit offsets stay inside a workgroup's rows
    if (static_cast<size_t>(rows_per_wg) * gllmq_row_bytes(f.dtype, k) > 0xFFFFFFFFull) return -1;
    const uint32_t wg_tiles = (rows_per_wg + 31u) / 32u;
    const uint32_t tile_rows = (rows_per_wg + wg_tiles - 1u) / wg_tiles; // equal heights, <= 32
    if (ksplit > 1 && grid > kScratchArriveBytes / 4u) return -1;       // one arrival counter per row range
    const uint32_t item_bytes = tile_rows * pieces * 16u;
    const uint32_t lds_ring = (static_cast<uint32_t>(sizeof(gq::Mm8sCtrl)) + gq::MMFR_RED_BUFS * gq::MMFR_CWAVES * gq::MMFR_RED_WAVE + 1023u) & ~1023u;
    const uint32_t items = wg_tiles * sb;
    uint32_t slots = std::min(items, (160u * 1024u - lds_ring) / item_bytes);
    if (slots < items) slots -= slots % gq::MMFR_LOADERS; // a reused ring is a whole number of rounds of the loaders
    uint32_t depth = ctx->mm8s_depth ? std::min(gq::MM8S_MAX_DEPTH, ctx->mm8s_depth) : 1u;
    while (depth > 2u && slots < items && slots < gq::mm8s_min_slots(depth)) --depth;
    // (the waves of a tile's blocks run side by side: a ring shorter than two tiles' items would let a loader wait for a wave that waits for it)
    if (slots < items && (slots < gq::mm8s_min_slots(depth) || slots < 2u * sb)) return -1;
    const size_t part_bytes = ksplit > 1 ? static_cast<size_t>(ksplit) * grid * wg_tiles * 2048u : 0u;
    if (part_bytes) {
        int grc = grow_scratch(ctx, S, &S.mmf, &S.mmf_bytes, part_bytes, stream, "quantized_matmul (GEMM)");
        if (grc != GLLMQ_OK) return grc;
    }
    Mm8Params P{};
    P.w = w;
    P.x = x;
    P.y = y;
    P.n = static_cast<uint32_t>(n);
    P.k = static_cast<uint32_t>(k);
    P.groups = groups;
    P.row_bytes = static_cast<uint32_t>(gllmq_row_bytes(f.dtype, k));
    P.m = static_cast<uint32_t>(m);
    P.ldx = ldx;
    P.ldy = static_cast<uint32_t>(n);
    P.grid = grid;
    P.ksplit = ksplit;
    P.kslice_groups = sb;
    P.part = static_cast<float *>(S.mmf);
    P.arrive = S.mm8_arrive;
    P.rows_per_wg = rows_per_wg;
    P.tile_rows = tile_rows;
    P.ring_slots = slots;
    P.wg_tiles = wg_tiles;
    P.last_wg_rows = P.n - (grid - 1u) * rows_per_wg;
    P.last_wg_tiles = (P.last_wg_rows + tile_rows - 1u) / tile_rows;
    P.lds_ctrl = 0;
    P.lds_ring = lds_ring;
    P.depth = depth;
    P.elem = ctx->call_elem;
    return launch(ctx, ctx->mmfr[fmt][ctx->call_elem ? 1 : 0], grid * ksplit, (gq::MMFR_CWAVES + gq::MMFR_LOADERS) * 64, lds_ring + slots * item_bytes, stream, &P,
                  sizeof P, ksplit > 1);
}

// A chain of batch entries for one launch of mm8c.hip.inc: consecutive matmuls of one format
// (Q4_K or Q5_K), one K <= 4096 and one activation row count <= 2 that the streamed kernels
// would take one by one.  chain_length() says how many entries from `descs` on form one (0 or 1:
// none); run_chain() launches it.
bool chain_entry_ok(const gllmq_ctx *ctx, const gllmq_matmul_desc &d, const gllmq_matmul_desc &first)
{
    const Format *f = find_format(d.ggml_dtype);
    if (!f || (f->dtype != T_Q4_K && f->dtype != T_Q5_K && f->dtype != T_Q8_0)) return false;
    if (f->dtype == T_Q5_K && ctx->mm8_q5k_min_m == 0) return false;
    if (f->dtype == T_Q8_0 && (ctx->mm8_q8_0_min_m == 0 || !ctx->mm8s_q8_0 || d.k % 256 != 0)) return false; // whole groups of 8 blocks
    if (d.ggml_dtype != first.ggml_dtype || d.m != first.m || d.k != first.k) return false;
    if (d.m == 0 || d.m > 2 || d.k == 0 || d.k % 8 != 0 || (d.k + 255) / 256 > 16 || d.n > 0x7FFFFFFFu) return false;
    if (!d.w_dev || !d.x_dev || !d.y_dev || !aligned(d.x_dev, 16) || !aligned(d.y_dev, 4) || !aligned(d.w_dev, f->w_align)) return false;
    const size_t rb = gllmq_row_bytes(d.ggml_dtype, d.k);
    if (rb % f->w_align != 0 || d.w_bytes < d.n * rb) return false;
    const size_t cus = static_cast<size_t>(ctx->num_cus);
    return d.n > 0 && (d.n + cus - 1) / cus >= ctx->chain_min_rows; // rows of the largest share
}

constexpr size_t kChainBoxPairs = size_t(1) << 19; // 64-bit words of the mailbox (4 MiB per stream that runs such chains)

// Whether entry `d`, flagged as starting after `prev`, reads (part of) prev's output and nothing
// else, so that it can take its activations from what prev posts: one activation row anywhere
// inside prev's output row, or all rows of an output whose rows are exactly as long as d's.
bool chain_reads_previous(const gllmq_matmul_desc &d, const gllmq_matmul_desc &prev)
{
    const uintptr_t x = reinterpret_cast<uintptr_t>(d.x_dev), y = reinterpret_cast<uintptr_t>(prev.y_dev);
    if (x < y || (x - y) % 4 != 0) return false;
    const size_t at = (x - y) / 4;
    if (d.m == 1) return at + d.k <= prev.n; // (the chain's entries share m)
    return at == 0 && d.k == prev.n;
}

size_t chain_length(const gllmq_ctx *ctx, const gllmq_matmul_desc *descs, size_t count)
{
    if (!ctx->use_chain || !ctx->use_mm8 || !ctx->use_mm8s || count < 2) return 0;
    size_t len = 0, posted = 0; // entries so far, and the mailbox places their posting entries take
    while (len < count && len < gq::MM8C_MAX_ENTRIES && !(descs[len].flags & ~1u) && chain_entry_ok(ctx, descs[len], descs[0])) {
        const gllmq_matmul_desc &d = descs[len];
        const size_t xb = d.m * d.k * 4, yb = d.m * d.n * 4;
        const bool reads_prev = len > 0 && (d.flags & 1u) && ctx->chain_dependent && chain_reads_previous(d, descs[len - 1]) &&
                                posted + descs[len - 1].m * descs[len - 1].n <= kChainBoxPairs;
        // An entry that starts after the one before it and does not simply read its output begins a
        // launch of its own: the launch boundary is the one wait that covers every case.
        if (len > 0 && (d.flags & 1u) && !reads_prev) break;
        // Workgroups run through the entries at their own pace: nothing an entry writes may be
        // anything another entry of the launch reads from memory or writes.
        bool clash = false;
        for (size_t j = 0; j < len && !clash; ++j) {
            const gllmq_matmul_desc &o = descs[j];
            const bool o_reads_prev = j > 0 && (o.flags & 1u); // (then it reads the mailbox, not memory)
            clash = ranges_meet(d.y_dev, yb, o.y_dev, o.m * o.n * 4) || (!o_reads_prev && ranges_meet(d.y_dev, yb, o.x_dev, o.m * o.k * 4)) ||
                    (!reads_prev && ranges_meet(d.x_dev, xb, o.y_dev, o.m * o.n * 4));
        }
        if (clash || ranges_meet(d.y_dev, yb, d.x_dev, xb)) break;
        if (reads_prev) posted += descs[len - 1].m * descs[len - 1].n;
        ++len;
    }
    return len;
}

int run_chain(gllmq_ctx *ctx, Scratch &S, const gllmq_matmul_desc *descs, size_t len, void *stream)
{
    const Format &f = *find_format(descs[0].ggml_dtype);
    const int fmt = f.dtype == T_Q8_0 ? 2 : f.dtype == T_Q5_K ? 1 : 0;
    const uint32_t cus = static_cast<uint32_t>(ctx->num_cus);
    const size_t k = descs[0].k;
    Mm8ChainParams P{};
    P.count = static_cast<uint32_t>(len);
    P.k = static_cast<uint32_t>(k);
    P.groups = static_cast<uint32_t>((k + 255) / 256);
    P.row_bytes = static_cast<uint32_t>(gllmq_row_bytes(f.dtype, k));
    P.m = static_cast<uint32_t>(descs[0].m);
    P.ldx = P.k;
    P.act_bf16 = 0;
    const uint32_t pieces = fmt == 2 ? gq::Mm8sFormat<3>::PIECES : fmt == 1 ? gq::Mm8sFormat<1>::PIECES : gq::Mm8sFormat<0>::PIECES;
    P.slot_bytes = 32u * pieces * 16u; // a slot holds an item of any entry: 32 rows of one block
    // LDS: the preparation's planes, sums and scales; the counters; the partial sums; the ring
    const gq::Mm8Lds prep = gq::mm8_lds_layout(P.groups, P.m, 1u, fmt == 2 ? 0u : 8u, 0u);
    P.lds_ctrl = (prep.red + 15u) & ~15u;
    const uint32_t red = P.lds_ctrl + static_cast<uint32_t>(sizeof(gq::Mm8sCtrl)) + gq::MM8C_MAX_SLOTS * 4u;
    P.lds_ring = (red + gq::MM8C_RED_BUFS * gq::MM8C_CWAVES * 64u * 4u + 1023u) & ~1023u;
    P.depth = ctx->mm8s_depth ? std::min(gq::MM8S_MAX_DEPTH, ctx->mm8s_depth) : 0u; // 0: by the entry's items, see the loader
    if (P.lds_ring >= 160u * 1024u) return -1;
    uint32_t slots = std::min(gq::MM8C_MAX_SLOTS, (160u * 1024u - P.lds_ring) / P.slot_bytes);
    slots -= slots % gq::MM8C_LOADERS;
    if (slots < gq::mm8s_min_slots(std::max(2u, P.depth))) return -1;
    P.ring_slots = slots;
    P.spin_limit = ctx->chain_spin_limit;
    P.epoch0 = ctx->chain_epoch;
    P.error = ctx->chain_error;
    P.progress = ctx->call_seq ? ctx->progress : nullptr;
    P.progress_seq = ctx->call_seq;
    uint32_t launched = 0, box_used = 0;
    for (size_t i = 0; i < len; ++i) {
        const gllmq_matmul_desc &d = descs[i];
        Mm8ChainEntry &E = P.e[i];
        E.w = static_cast<const uint8_t *>(d.w_dev);
        E.x = static_cast<const float *>(d.x_dev);
        E.y = static_cast<float *>(d.y_dev);
        E.n = static_cast<uint32_t>(d.n);
        E.ldy = E.n;
        E.rows_per_wg = (E.n + cus - 1u) / cus;
        E.grid = (E.n + E.rows_per_wg - 1u) / E.rows_per_wg;
        E.wg_tiles = (E.rows_per_wg + 31u) / 32u;
        E.tile_rows = (E.rows_per_wg + E.wg_tiles - 1u) / E.wg_tiles;
        E.last_wg_rows = E.n - (E.grid - 1u) * E.rows_per_wg;
        E.last_wg_tiles = (E.last_wg_rows + E.tile_rows - 1u) / E.tile_rows;
        E.flags = i > 0 ? (d.flags & 1u) : 0u; // the chain's first entry is ordered by the stream
        if (i > 0 && E.flags) { // (chain_length() has checked that it reads the output of the entry before and that the places fit)
            Mm8ChainEntry &B = P.e[i - 1];
            B.flags |= 2u;
            B.box_at = box_used;
            box_used += P.m * B.n;
            E.x_at = B.box_at + static_cast<uint32_t>((static_cast<const float *>(d.x_dev) - static_cast<const float *>(descs[i - 1].y_dev)));
            E.x_ld = B.n;
        }
        // one activation row over tiles of at most 16 weight rows: in pairs of blocks, as run_mm8s() would
        if (ctx->mm8s_fold_on && P.m == 1 && E.tile_rows <= 16 && P.groups > 8) E.flags |= 4u;
        launched = std::max(launched, E.grid);
    }
    bool waits = false, folds = false;
    for (size_t i = 0; i < len; ++i) {
        waits = waits || (P.e[i].flags & 3u) != 0u;
        folds = folds || (P.e[i].flags & 4u) != 0u;
    }
    if (waits) {
        if (box_used > kChainBoxPairs) return -1;
        if (!S.box) {
            // first chain of this kind on the stream: the mailbox, all zero (epochs start at 1).  Not
            // during a capture and not from a block of fixed size: the entries then take a launch each.
            if (S.fixed || stream_is_capturing(stream)) return -1;
            GLLMQ_HIP(ctx, hipSetDevice(ctx->device));
            GLLMQ_HIP(ctx, hipMalloc(&S.box, kChainBoxPairs * 8));
            GLLMQ_HIP(ctx, hipMemset(S.box, 0, kChainBoxPairs * 8));
        }
        P.box = static_cast<unsigned long long *>(S.box);
        ctx->chain_epoch += static_cast<uint32_t>(len);
    }
    P.launched = launched;
    return launch(ctx, ctx->mm8c[fmt][folds ? 1 : 0][waits ? 1 : 0], launched, (gq::MM8C_CWAVES + gq::MM8C_LOADERS) * 64, P.lds_ring + slots * P.slot_bytes,
                  stream, &P, sizeof P, true);
}

int run_gemv(gllmq_ctx *ctx, const Format &f, const uint8_t *w, const float *x, float *y, size_t m, size_t n,
             size_t k, bool act_bf16, void *stream)
{
    const size_t rb = gllmq_row_bytes(f.dtype, k);
    constexpr size_t kChunk = 16384; // elements of K one launch covers (four waves of 4096)
    if (ctx->call_glu && ctx->gemv_f32) return kNeedPlainActivations;
    const uint32_t ldx = row_stride_x(ctx, k);
    // 16-bit elements are read as aligned vectors only
    if (ctx->call_elem && !(aligned(x, 16) && k % 64 == 0 && ldx % 8 == 0)) return kNeedPlainActivations;
    for (size_t m0 = 0; m0 < m; m0 += 2) {
        const uint32_t mm = static_cast<uint32_t>(std::min<size_t>(2, m - m0));
        for (size_t k0 = 0; k0 < k; k0 += kChunk) {
            const size_t kk = std::min(kChunk, k - k0);
            int rc = launch_gemv(ctx, f, w + (k0 / 256) * f.group_bytes, rb, elem_at(ctx, x, m0 * ldx + k0), elem_at(ctx, y, m0 * n), mm,
                                 static_cast<uint32_t>(n), static_cast<uint32_t>(kk), ldx,
                                 static_cast<uint32_t>(n), k0 != 0, act_bf16, stream);
            if (rc != GLLMQ_OK) return rc;
        }
    }
    return GLLMQ_OK;
}

// Whether 5 to 8 activation rows are more than the int8 kernels take in a pass (up to eight of Q4_K, seven of Q5_K and six
// of Q6_K and Q8_0); beyond it they read the weights twice, and the wide GEMM is ahead from some size on.
bool mmfw_takes_few(const gllmq_ctx *ctx, uint32_t dtype, size_t m)
{
    const size_t pass = dtype == T_Q4_K ? 8 : dtype == T_Q5_K ? 7 : 6;
    return ctx->mmfw_small_min_m <= 9 && m >= 5 && m > pass;
}

// One quantized matmul on validated arguments: the kernel family by format, rows and shape.
int dispatch_matmul(gllmq_ctx *ctx, Scratch &S, const Format &f, const uint8_t *w, const float *x, float *y, size_t m,
                    size_t n, size_t k, bool bf16, void *stream)
{
    int rc = -1;
    if (!ctx->mmfs_all) {
        const MmfwMatrix one{ w, y, n };
        rc = run_mmfw(ctx, S, f, &one, 1, x, ctx->call_elem, ctx->call_elem, m, k, bf16, stream, ctx->mmfw_min_m);
        if (rc >= 0 || rc == kNeedPlainActivations) return rc;
    }
    rc = run_mmfr(ctx, S, f, w, x, y, m, n, k, bf16, stream);
    if (rc >= 0) return rc;
    rc = run_mmfs(ctx, S, f, w, x, y, m, n, k, bf16, stream);
    if (rc >= 0 || rc == kNeedPlainActivations) return rc;
    // 9 to 32 rows of what the streamed GEMMs leave: row tiles of the GEMM for more rows.  us per call with weights that are
    // not in the caches, f32 and bf16, against run_mmf's in brackets.  32 rows: Q6_K 13824 x 5120 35.0, 31.1 (41.3, 39.9),
    // 4096 x 4096 18.4, 17.6 (23.6, 23.9); Q8_0 14336 x 4096 30.8, 25.4 (35.3, 35.5); Q4_K 13824 x 5120 28.4, 24.6 (28.9,
    // 27.9), 14336 x 4096 26.1, 21.2 (24.0, 23.3).  It is not ahead everywhere: of Q4_K and Q5_K with 17 to 32 rows f32 calls
    // of k = 4096 are 5 to 9 % behind (28672 x 4096 36.3 (34.7), 40.1 (38.3)) where bf16 calls are as much ahead (30.3 (33.5),
    // 33.4 (36.9)); both take one kernel, so that they share their bits.
    // Five to eight rows beyond a pass of the int8 kernels: from 10240 elements a row and 40 M weights on.  f32, us per call, here and in
    // brackets there (eight rows of Q5_K, seven of Q6_K and of Q8_0): 4096 x 10240 19.7 (21.9), 22.6 (24.9), 26.6 (26.1); 4096 x 11520 20.7 (26.1), 24.5
    // (29.8), 27.8 (31.8); 14336 x 14336 56.8 (67.0), 66.3 (86.4), 68.2 (96.2); below, 2390 x 11520 17.1 (18.9), 22.8 (20.4), 21.5 (20.9); 4096 x 6144 15.2
    // (16.1), 18.9 (18.6), 17.4 (18.9); 8192 x 8192 26.2 (24.6), 29.6 (29.1), 31.0 (31.4); 28672 x 8192 61.7 (58.8), 73.5 (79.0), 74.9 (90.2); 28672 x 4096
    // 36.2 (32.4), 43.0 (41.7), 43.3 (46.8).  16-bit calls gain more (8192 x 8192 21.3 (28.8), 25.9 (33.0), 24.1 (35.3)), but share the f32 call's bits
    // and so its kernel.  In a pass: Q8_0 six rows of 4096 x 14336 31.2 (26.4).
    if (!ctx->mmfs_all && (m >= ctx->mmfw_small_min_m || (!bf16 && k >= 10240 && n * k >= (40ull << 20) && mmfw_takes_few(ctx, f.dtype, m)))) {
        const MmfwMatrix one{ w, y, n };
        rc = run_mmfw(ctx, S, f, &one, 1, x, ctx->call_elem, ctx->call_elem, m, k, bf16, stream, 5);
        if (rc >= 0 || rc == kNeedPlainActivations) return rc;
    }
    rc = run_mmf(ctx, S, f, w, x, y, m, n, k, bf16, stream);
    if (rc >= 0 || rc == kNeedPlainActivations) return rc;
    // up to 8 rows: the int8 kernels when one pass over the weights does it, else the GEMM
    rc = run_mm8s(ctx, f, w, x, y, m, n, k, bf16, stream, nullptr, false, &S);
    if (rc >= 0 || rc == kNeedPlainActivations) return rc;
    rc = run_mm8(ctx, S, f, w, x, y, m, n, k, bf16, stream, true);
    if (rc >= 0 || rc == kNeedPlainActivations) return rc;
    if (ctx->mmf_small_min_m > 0) {
        rc = run_mmf(ctx, S, f, w, x, y, m, n, k, bf16, stream, ctx->mmf_small_min_m);
        if (rc >= 0 || rc == kNeedPlainActivations) return rc;
    }
    rc = run_mm8(ctx, S, f, w, x, y, m, n, k, bf16, stream);
    if (rc >= 0 || rc == kNeedPlainActivations) return rc;
    return run_gemv(ctx, f, w, x, y, m, n, k, bf16, stream);
}

size_t ffn_h_bytes(size_t m, size_t ffn) { return ((m * ffn * sizeof(float)) + 255) & ~size_t(255); }
size_t ffn_scratch_bytes(size_t m, size_t ffn) { return ffn_h_bytes(m, ffn) + m * 2 * ffn * sizeof(float); }

// Which kernel the dispatch gives a matmul: the dispatch itself, run with launches and allocations
// switched off (ctx->probe), so that the answer cannot drift from what a call does.  `fn` is the
// kernel when the call is exactly one launch, else null; `launches` counts them.
struct DispatchChoice {
    hipFunction_t fn = nullptr;
    uint32_t launches = 0;
};

template <class Call>
DispatchChoice dispatch_choice(gllmq_ctx *ctx, Call &&call)
{
    ctx->probe = true;
    ctx->probe_launches = 0;
    ctx->probe_fn = nullptr;
    const int rc = call();
    ctx->probe = false;
    DispatchChoice c;
    c.launches = rc == GLLMQ_OK ? ctx->probe_launches : 0u;
    c.fn = c.launches == 1u ? ctx->probe_fn : nullptr;
    return c;
}

// One validated quantized matmul with the scratch of `S` (call_mutex held).
int matmul_on_scratch(gllmq_ctx *ctx, Scratch &S, const void *w, size_t w_bytes, const float *x, float *y, uint32_t dtype,
                      size_t m, size_t n, size_t k, int act_mode, void *stream)
{
    const Format *f = find_format(dtype);
    int rc = check_matmul_args(ctx, f, w, w_bytes, x, y, dtype, m, n, k);
    if (rc >= 0) return rc;
    if (act_mode != GLLMQ_ACT_F32_SPLIT && act_mode != GLLMQ_ACT_BF16)
        return fail(ctx, GLLMQ_ERR_INVALID, "quantized_matmul: unknown activation mode %d", act_mode);
    const bool bf16 = act_mode == GLLMQ_ACT_BF16;
    if (bf16 && ctx->gemv_f32)
        return fail(ctx, GLLMQ_ERR_UNIMPLEMENTED, "quantized_matmul: bf16 activations are not built for the f32 GEMV flavour");
    return dispatch_matmul(ctx, S, *f, static_cast<const uint8_t *>(w), x, y, m, n, k, bf16, stream);
}

} // namespace

extern "C" {

const char *gllmq_version(void) { return "gllm_hip_quant 0.1 (gfx950)"; }

const char *gllmq_status_string(int status)
{
    switch (status) {
    case GLLMQ_OK: return "ok";
    case GLLMQ_ERR_UNIMPLEMENTED: return "unimplemented";
    case GLLMQ_ERR_BAD_SHAPE: return "bad shape";
    case GLLMQ_ERR_BAD_ALIGNMENT: return "bad alignment";
    case GLLMQ_ERR_HIP: return "hip error";
    case GLLMQ_ERR_INVALID: return "invalid argument";
    default: return "unknown status";
    }
}

size_t gllmq_block_size(uint32_t dtype)
{
    const Format *f = find_format(dtype);
    return f ? f->block_size : 0;
}

size_t gllmq_block_bytes(uint32_t dtype)
{
    const Format *f = find_format(dtype);
    return f ? f->block_bytes : 0;
}

size_t gllmq_row_bytes(uint32_t dtype, size_t k)
{
    const Format *f = find_format(dtype);
    return f ? (k + f->block_size - 1) / f->block_size * f->block_bytes : 0;
}

int gllmq_init(gllmq_ctx **out, int device)
{
    if (!out) return GLLMQ_ERR_INVALID;
    *out = nullptr;
    gllmq_ctx *ctx = new gllmq_ctx;
    ctx->device = device;
    hipError_t e = hipSetDevice(device);
    if (e == hipSuccess) e = hipFree(nullptr); // force context creation
    if (e != hipSuccess) {
        fprintf(stderr, "gllmq_init: device %d: %s\n", device, hipGetErrorString(e));
        delete ctx;
        return GLLMQ_ERR_HIP;
    }
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) == hipSuccess) {
        ctx->num_cus = prop.multiProcessorCount;
        if (strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
            fprintf(stderr, "gllmq_init: device %d is %s; this library holds gfx950 code only\n", device,
                    prop.gcnArchName);
            delete ctx;
            return GLLMQ_ERR_UNIMPLEMENTED;
        }
    }
    const unsigned char *const images[10] = { gllmq_co_codec, gllmq_co_mm8, gllmq_co_mm8s, gllmq_co_mm8s_q8_0, gllmq_co_mm8c,
                                             gllmq_co_mm8_q6k_q8_0, gllmq_co_mmf, gllmq_co_mmfs, gllmq_co_mmfw, gllmq_co_moe };
    for (int i = 0; i < 10; ++i) {
        e = hipModuleLoadData(&ctx->modules[i], images[i]);
        if (e != hipSuccess) {
            fprintf(stderr, "gllmq_init: hipModuleLoadData: %s\n", hipGetErrorString(e));
            for (hipModule_t mod : ctx->modules)
                if (mod) (void)hipModuleUnload(mod);
            delete ctx;
            return GLLMQ_ERR_HIP;
        }
    }
    int rc = GLLMQ_OK;
    char name[64];
    for (int i = 0; i < kNumFormats && rc == GLLMQ_OK; ++i) {
        snprintf(name, sizeof name, "gq_dequant_%s_v1", kFormats[i].tag);
        rc = get_function(ctx, &ctx->dequant[i][0], name);
        if (rc != GLLMQ_OK) break;
        snprintf(name, sizeof name, "gq_dequant_%s_v4", kFormats[i].tag);
        rc = get_function(ctx, &ctx->dequant[i][1], name);
        if (rc != GLLMQ_OK) break;
        snprintf(name, sizeof name, "gq_gather_%s_v1", kFormats[i].tag);
        rc = get_function(ctx, &ctx->gather[i][0], name);
        if (rc != GLLMQ_OK) break;
        snprintf(name, sizeof name, "gq_gather_%s_v4", kFormats[i].tag);
        rc = get_function(ctx, &ctx->gather[i][1], name);
        if (rc != GLLMQ_OK) break;
        snprintf(name, sizeof name, "gq_gather_%s_e16_v1", kFormats[i].tag);
        rc = get_function(ctx, &ctx->gather_e16[i][0], name);
        if (rc != GLLMQ_OK) break;
        snprintf(name, sizeof name, "gq_gather_%s_e16_v4", kFormats[i].tag);
        rc = get_function(ctx, &ctx->gather_e16[i][1], name);
        if (rc != GLLMQ_OK) break;
        snprintf(name, sizeof name, "gq_gather_%s_e16_v8", kFormats[i].tag);
        rc = get_function(ctx, &ctx->gather_e16[i][2], name);
        for (int m = 1; m <= 2 && rc == GLLMQ_OK; ++m) {
            snprintf(name, sizeof name, "gq_gemv_%s_m%d", kFormats[i].tag, m);
            rc = get_function(ctx, &ctx->gemv[i][m - 1], name);
            if (rc != GLLMQ_OK) break;
            snprintf(name, sizeof name, "gq_gemv_i8_%s_m%d", kFormats[i].tag, m);
            rc = get_function(ctx, &ctx->gemv_i8[i][m - 1], name);
            if (rc != GLLMQ_OK) break;
            snprintf(name, sizeof name, "gq_gemv_i8_%s_m%d_glu", kFormats[i].tag, m);
            rc = get_function(ctx, &ctx->gemv_i8_glu[i][m - 1], name);
            if (rc != GLLMQ_OK) break;
            snprintf(name, sizeof name, "gq_gemv_i8_%s_m%d_e16", kFormats[i].tag, m);
            rc = get_function(ctx, &ctx->gemv_i8_e16[i][m - 1], name);
        }
        if (rc != GLLMQ_OK) break;
        snprintf(name, sizeof name, "gq_gemv_i8_%s_m1_argmax", kFormats[i].tag);
        rc = get_function(ctx, &ctx->gemv_i8_argmax[i], name);
    }
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_route, "gq_moe_route");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->convert_elem, "gq_convert_elem");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->mmf_prep[0], "gq_mmf_prep_t1");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->mmf_prep[1], "gq_mmf_prep_t2");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->mmf_prep_lanes, "gq_mmf_prep_lanes");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->mmf_reduce, "gq_mmf_reduce");
    for (int q = 0; q < 4 && rc == GLLMQ_OK; ++q)
        for (int t = 0; t < 2 && rc == GLLMQ_OK; ++t)
            for (int b = 0; b < 2 && rc == GLLMQ_OK; ++b) {
                snprintf(name, sizeof name, "gq_mmf_%s_t%d%s", q == 3 ? "q8_0" : q == 2 ? "q6k" : q == 1 ? "q5k" : "q4k", t + 1, b ? "_bf16" : "");
                rc = get_function(ctx, &ctx->mmf_q4k[q][t][b], name);
            }
    static const char *const kMm8c[3][2] = { { "gq_mm8c_q4k", "gq_mm8c_q4k_f" }, { "gq_mm8c_q5k", "gq_mm8c_q5k_f" }, { "gq_mm8c_q8_0", "gq_mm8c_q8_0_f" } };
    for (int q = 0; q < 3 && rc == GLLMQ_OK; ++q)
        for (int v = 0; v < 2 && rc == GLLMQ_OK; ++v)
            for (int d = 0; d < 2 && rc == GLLMQ_OK; ++d) {
                snprintf(name, sizeof name, "%s%s", kMm8c[q][v], d ? "_d" : "");
                rc = get_function(ctx, &ctx->mm8c[q][v][d], name);
            }
    for (int q = 0; q < 2 && rc == GLLMQ_OK; ++q)
        for (int b = 0; b < 2 && rc == GLLMQ_OK; ++b) {
            snprintf(name, sizeof name, "gq_mmfs_%s%s", q ? "q5k" : "q4k", b ? "_bf16" : "");
            rc = get_function(ctx, &ctx->mmfs[q][b], name);
        }
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->mmfw_prep[0], "gq_mmfw_prep");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->mmfw_prep[1], "gq_mmfw_prep_hi");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->mmfw_prep_e16, "gq_mmfw_prep_e16");
    for (int q = 0; q < 4 && rc == GLLMQ_OK; ++q)
        for (int t = 0; t < gq::MMFW_MAX_MT && rc == GLLMQ_OK; ++t)
            for (int b = 0; b < 2 && rc == GLLMQ_OK; ++b) {
                snprintf(name, sizeof name, "gq_mmf_%s_w%d%s", q == 3 ? "q8_0" : q == 2 ? "q6k" : q == 1 ? "q5k" : "q4k", t + 1, b ? "_hi" : "");
                rc = get_function(ctx, &ctx->mmfw[q][t][b], name);
            }
    for (int q = 0; q < 4 && rc == GLLMQ_OK; ++q)
        for (int b = 0; b < 2 && rc == GLLMQ_OK; ++b) {
            snprintf(name, sizeof name, "gq_mmf_%s_w1_own%s", q == 3 ? "q8_0" : q == 2 ? "q6k" : q == 1 ? "q5k" : "q4k", b ? "_hi" : "");
            rc = get_function(ctx, &ctx->mmfw_own[q][b], name);
        }
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->mmfx_decode, "gq_mmfx_decode_q6k");
    for (int t = 2; t <= gq::MMFW_MAX_MT && rc == GLLMQ_OK; ++t)
        for (int b = 0; b < 2 && rc == GLLMQ_OK; ++b) {
            snprintf(name, sizeof name, "gq_mmf_q6k_w%d%s_dec", t, b ? "_hi" : "");
            rc = get_function(ctx, &ctx->mmfx[t - 2][b], name);
        }
    for (int q = 0; q < 4 && rc == GLLMQ_OK; ++q)
        for (int b = 0; b < 2 && rc == GLLMQ_OK; ++b) {
            snprintf(name, sizeof name, "gq_moe_mmf_%s%s", q == 3 ? "q8_0" : q == 2 ? "q6k" : q == 1 ? "q5k" : "q4k", b ? "_hi" : "");
            rc = get_function(ctx, &ctx->moe_mmf[q][b], name);
            if (rc != GLLMQ_OK) break;
            strncat(name, "_few", sizeof name - strlen(name) - 1);
            rc = get_function(ctx, &ctx->moe_mmf_few[q][b], name);
        }
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->mmfr[0][0], "gq_mmfr_q4k");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->mmfr[0][1], "gq_mmfr_q4k_e16");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->mmfr[1][0], "gq_mmfr_q5k");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->mmfr[1][1], "gq_mmfr_q5k_e16");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_plan, "gq_moe_plan");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_plan_wide, "gq_moe_plan_wide");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_plan_few, "gq_moe_plan_few");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_act, "gq_moe_act");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_combine, "gq_moe_combine");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_combine_v4, "gq_moe_combine_v4");
    for (int i = 0; i < kNumFormats && rc == GLLMQ_OK; ++i) {
        snprintf(name, sizeof name, "gq_moe_gemv_%s", kFormats[i].tag);
        rc = get_function(ctx, &ctx->moe_gemv[i], name);
    }
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_mm8_fn[0][0], "gq_moe_mm8_q4k_a1");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_mm8_fn[0][1], "gq_moe_mm8_q4k_a2");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_mm8_fn[1][0], "gq_moe_mm8_q6k_a1");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_mm8_fn[1][1], "gq_moe_mm8_q6k_a2");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_mm8_fn[2][0], "gq_moe_mm8_q5k_a1");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_mm8_fn[2][1], "gq_moe_mm8_q5k_a2");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_mm8_q6k_rows, "gq_moe_mm8_q6k_rows");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_mm8s_fn[MM8_Q4K][0], "gq_moe_mm8s_q4k");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_mm8s_fn[MM8_Q5K][0], "gq_moe_mm8s_q5k");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_mm8s_fn[MM8_Q6K][0], "gq_moe_mm8s_q6k");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_mm8s_fn[MM8_Q4K][1], "gq_moe_mm8s_glu_q4k");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_mm8s_fn[MM8_Q5K][1], "gq_moe_mm8s_glu_q5k");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_mm8_glu_fn[MM8_Q4K][0], "gq_moe_mm8_glu_q4k_a1");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_mm8_glu_fn[MM8_Q4K][1], "gq_moe_mm8_glu_q4k_a2");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_mm8_glu_fn[MM8_Q5K][0], "gq_moe_mm8_glu_q5k_a1");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->moe_mm8_glu_fn[MM8_Q5K][1], "gq_moe_mm8_glu_q5k_a2");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->dequant_wave, "gq_dequant_q4k_wave");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->dequant_wave_q5k, "gq_dequant_q5k_wave");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->argmax_part, "gq_argmax_part");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->argmax_final, "gq_argmax_final");
    if (rc == GLLMQ_OK) {
        static const uint32_t kRows[8] = { 0, 1, 2, 3, 4, 5, 6, 7 };
        hipError_t he = hipMalloc(reinterpret_cast<void **>(&ctx->identity_rows), sizeof kRows);
        if (he == hipSuccess) he = hipMemcpy(ctx->identity_rows, kRows, sizeof kRows, hipMemcpyHostToDevice);
        if (he != hipSuccess) rc = fail(ctx, GLLMQ_ERR_HIP, "row table: %s", hipGetErrorString(he));
    }
    if (rc == GLLMQ_OK) {
        hipError_t he = hipHostMalloc(reinterpret_cast<void **>(&ctx->chain_error), sizeof(uint32_t), hipHostMallocDefault);
        if (he == hipSuccess) *ctx->chain_error = 0u;
        else rc = fail(ctx, GLLMQ_ERR_HIP, "error word: %s", hipGetErrorString(he));
    }
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->touch, "gq_touch");
    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->finish_elem, "gq_finish_elem");
    if (rc == GLLMQ_OK) {
        hipError_t he = hipMalloc(reinterpret_cast<void **>(&ctx->progress), 256);
        if (he == hipSuccess) he = hipMemset(ctx->progress, 0, 256);
        if (he == hipSuccess) he = hipStreamCreateWithFlags(&ctx->side_stream, hipStreamNonBlocking);
        if (he == hipSuccess) he = hipEventCreateWithFlags(&ctx->side_event, hipEventDisableTiming);
        if (he != hipSuccess) rc = fail(ctx, GLLMQ_ERR_HIP, "prefetch stream: %s", hipGetErrorString(he));
    }
    {
        static const struct { int pi, ei; const char *tag; } kMm8[] = {
            { 0, 0, "p1_e1" }, { 0, 1, "p1_e2" }, { 0, 2, "p1_e4" }, { 1, 1, "p2_e2" }, { 1, 2, "p2_e4" }, { 2, 2, "p4_e4" },
        };
        static const char *const kMm8Format[MM8_KINDS] = { "q4k", "q6k", "q5k", "q8_0" };
        for (int q = 0; q < MM8_KINDS; ++q)
            for (const auto &k : kMm8) {
                snprintf(name, sizeof name, "gq_mm8_%s_%s", kMm8Format[q], k.tag);
                if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->mm8[q][k.pi][k.ei], name);
                for (int a = 1; a <= 2 && k.pi <= 1 && rc == GLLMQ_OK; ++a) {
                    snprintf(name, sizeof name, "gq_mm8_%s_%s_a%d", kMm8Format[q], k.tag, a);
                    rc = get_function(ctx, &ctx->mm8_areg[q][k.pi][k.ei][a - 1], name);
                }
                if (k.pi == 2) {
                    snprintf(name, sizeof name, "gq_mm8_%s_%s_g", kMm8Format[q], k.tag);
                    if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->mm8_gated_p4[q], name);
                }
                if (q != MM8_Q4K && q != MM8_Q5K) continue;
                const int gi = q == MM8_Q5K ? 1 : 0;
                snprintf(name, sizeof name, "gq_mm8_glu_%s_%s", kMm8Format[q], k.tag);
                if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->mm8_glu[gi][k.pi][k.ei], name);
                for (int a = 1; a <= 2 && k.pi <= 1 && rc == GLLMQ_OK; ++a) {
                    snprintf(name, sizeof name, "gq_mm8_glu_%s_%s_a%d", kMm8Format[q], k.tag, a);
                    rc = get_function(ctx, &ctx->mm8_glu_areg[gi][k.pi][k.ei][a - 1], name);
                }
            }
        if (rc == GLLMQ_OK) rc = get_function(ctx, &ctx->glu_act, "gq_glu_act");
        static const char *const kMm8sFormat[4] = { "q4k", "q5k", "q6k", "q8_0" };
        static const char *const kMm8s[7] = { "p1_e1_a", "p1_e2_a", "p2_e4_a", "p1_e2", "p2_e4", "p4_e4", "p1_e4" };
        for (int q = 0; q < 4; ++q)
            for (int v = 0; v < 7 && rc == GLLMQ_OK; ++v) {
                snprintf(name, sizeof name, "gq_mm8s_%s_%s", kMm8sFormat[q], kMm8s[v]);
                rc = get_function(ctx, &ctx->mm8s[q][v], name);
            }
        static const char *const kMm8sToken[3] = { "p1_e1_a", "p1_e2", "p1_e4" };
        for (int q = 0; q < 4; ++q)
            for (int v = 0; v < 3 && rc == GLLMQ_OK; ++v) {
                snprintf(name, sizeof name, "gq_mm8s_%s_%s_token", kMm8sFormat[q], kMm8sToken[v]);
                rc = get_function(ctx, &ctx->mm8s_token[q][v], name);
            }
        static const char *const kMm8sGated[6] = { "p1_e1_a", "p1_e2_a", "p2_e4_a", "p1_e2", "p2_e4", "p1_e4" };
        for (int q = 0; q < 2; ++q)
            for (int v = 0; v < 6 && rc == GLLMQ_OK; ++v) {
                snprintf(name, sizeof name, "gq_mm8s_%s_%s_glu", q ? "q5k" : "q4k", kMm8sGated[v]);
                rc = get_function(ctx, &ctx->mm8s_gated[q][v], name);
            }
        static const char *const kMm8sE16[6] = { "p1_e1_a", "p1_e2_a", "p2_e4_a", "p1_e2", "p2_e4", "p1_e4" };
        for (int q = 0; q < 4; ++q)
            for (int v = 0; v < 6 && rc == GLLMQ_OK; ++v) {
                snprintf(name, sizeof name, "gq_mm8s_%s_%s_e16", kMm8sFormat[q], kMm8sE16[v]);
                rc = get_function(ctx, &ctx->mm8s_e16[q][v], name);
            }
        static const char *const kMm8sFold[10] = { "p1_e1_a_f", "p1_e2_a_f", "p1_e2_f", "p1_e4_f", "p1_e2_g_f", "p1_e4_g_f",
                                                   "p1_e1_a_f_e16", "p1_e2_a_f_e16", "p1_e2_f_e16", "p1_e4_f_e16" };
        for (int q = 0; q < 4; ++q)
            for (int v = 0; v < 10 && rc == GLLMQ_OK; ++v) {
                snprintf(name, sizeof name, "gq_mm8s_%s_%s", kMm8sFormat[q], kMm8sFold[v]);
                rc = get_function(ctx, &ctx->mm8s_fold[q][v], name);
            }
        for (int q = 0; q < 4; ++q)
            for (int v = 0; v < 4 && rc == GLLMQ_OK; ++v) {
                snprintf(name, sizeof name, "gq_mm8s_%s_p%d_e4%s_s", kMm8sFormat[q], 1 + (v & 1), (v & 2) ? "_g" : "");
                rc = get_function(ctx, &ctx->mm8s_split[q][v & 1][v >> 1], name);
            }
        for (int q = 0; q < 4; ++q)
            for (int v = 0; v < 6 && rc == GLLMQ_OK && q != 2; ++v) {
                static const char *const kGroup[3] = { "p1_e1_a", "p1_e2_a", "p2_e4_a" };
                snprintf(name, sizeof name, "gq_mm8s_%s_%s%s_q", kMm8sFormat[q], kGroup[v % 3], v >= 3 ? "_e16" : "");
                rc = get_function(ctx, &ctx->mm8s_group[q][v / 3][v % 3], name);
            }
        static const char *const kMm8sGlu[4] = { "p1_e2_g", "p2_e4_g", "p1_e4_g", "p4_e4_g" };
        for (int q = 0; q < 4; ++q)
            for (int v = 0; v < 4 && rc == GLLMQ_OK; ++v) {
                snprintf(name, sizeof name, "gq_mm8s_%s_%s", kMm8sFormat[q], kMm8sGlu[v]);
                rc = get_function(ctx, &ctx->mm8s_glu[q][v], name);
            }
    }
    if (rc == GLLMQ_OK) {
        // the kernels that say when they start (the streamed forms and their chain)
        auto add = [&](hipFunction_t f) { if (f) ctx->announces.insert(f); };
        for (auto &q : ctx->mm8s) for (hipFunction_t f : q) add(f);
        for (auto &q : ctx->mm8s_gated) for (hipFunction_t f : q) add(f);
        for (auto &q : ctx->mm8s_group) for (auto &e : q) for (hipFunction_t f : e) add(f);
        for (auto &q : ctx->mm8s_e16) for (hipFunction_t f : q) add(f);
        for (auto &q : ctx->mm8s_glu) for (hipFunction_t f : q) add(f);
        for (auto &q : ctx->mm8s_fold) for (hipFunction_t f : q) add(f);
        for (auto &q : ctx->mm8s_split) for (auto &r : q) for (hipFunction_t f : r) add(f);
        for (auto &q : ctx->mm8c) for (auto &v : q) for (hipFunction_t f : v) add(f);
    }
    // the scratch array of the entry point that allocates nothing: found (and thereby placed on
    // this device) now, while allocating is allowed
    if (rc == GLLMQ_OK) rc = gq_noalloc_init(ctx, device);
    if (rc != GLLMQ_OK) {
        fprintf(stderr, "gllmq_init: %s\n", ctx->err.c_str());
        for (hipModule_t mod : ctx->modules)
            if (mod) (void)hipModuleUnload(mod);
        delete ctx;
        return rc;
    }
    ctx->gemv_waves = static_cast<uint32_t>(ctx->num_cus) * 8u;
    *out = ctx;
    return GLLMQ_OK;
}

void gllmq_destroy(gllmq_ctx *ctx)
{
    if (!ctx) return;
    for (Scratch &S : ctx->scratch) free_scratch(ctx, S);
    for (void *p : ctx->kept) (void)hipFree(p);
    for (CachedWeights &W : ctx->weights)
        if (W.dev) (void)hipFree(W.dev);
    if (ctx->identity_rows) (void)hipFree(ctx->identity_rows);
    if (ctx->chain_error) (void)hipHostFree(ctx->chain_error);
    if (ctx->side_stream) {
        (void)hipStreamSynchronize(ctx->side_stream);
        (void)hipStreamDestroy(ctx->side_stream);
    }
    if (ctx->side_event) (void)hipEventDestroy(ctx->side_event);
    if (ctx->progress) (void)hipFree(ctx->progress);
    for (hipModule_t mod : ctx->modules)
        if (mod) (void)hipModuleUnload(mod);
    delete ctx;
}

const char *gllmq_last_error(const gllmq_ctx *ctx)
{
    if (!ctx) return "NULL context";
    // a copy per calling thread: another thread's failing call may replace the context's string
    static thread_local std::string copy;
    {
        std::lock_guard<std::mutex> g(const_cast<gllmq_ctx *>(ctx)->err_mutex);
        copy = ctx->err;
    }
    return copy.c_str();
}

int gllmq_set_option(gllmq_ctx *ctx, const char *name, long value)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    if (!name) return fail(ctx, GLLMQ_ERR_INVALID, "set_option: NULL name");
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    const std::string n(name);
    const uint32_t u = static_cast<uint32_t>(std::max(0l, value));
    if (n == "gemv_f32") ctx->gemv_f32 = value != 0;
    else if (n == "mm8") ctx->use_mm8 = value != 0;
    else if (n == "mmf") ctx->use_mmf = value != 0;
    else if (n == "mm8s") ctx->use_mm8s = value != 0;
    else if (n == "mmfs") ctx->use_mmfs = value != 0;
    else if (n == "mmfr") ctx->use_mmfr = value != 0;
    else if (n == "mmfw") ctx->use_mmfw = value != 0;
    else if (n == "mmfw_min_m") ctx->mmfw_min_m = std::max(1u, u);
    else if (n == "batch_group") ctx->batch_group = value != 0;
    else if (n == "mmfw_small_min_m") ctx->mmfw_small_min_m = std::max(1u, u);
    else if (n == "mmfw_mt") ctx->mmfw_mt = std::min(u, static_cast<uint32_t>(gq::MMFW_MAX_MT));
    else if (n == "mmfw_ksplit") ctx->mmfw_ksplit = u;
    else if (n == "mmfw_run") ctx->mmfw_run = u;
    else if (n == "mmfw_own") ctx->use_mmfw_own = value != 0;
    else if (n == "mmfx_min_m") ctx->mmfx_min_m = static_cast<uint32_t>(std::max(0L, value));
    else if (n == "mmfr_min_rows") ctx->mmfr_min_rows = std::max(1u, u);
    else if (n == "chain") ctx->use_chain = value != 0;
    else if (n == "chain_dependent") ctx->chain_dependent = value != 0;
    else if (n == "chain_spin_limit") ctx->chain_spin_limit = u;
    else if (n == "chain_min_rows") ctx->chain_min_rows = std::max(1u, u);
    else if (n == "lm_head_fused") ctx->lm_head_fused = value != 0;
    else if (n == "elem_fused") ctx->elem_fused = value != 0;
    else if (n == "ffn_glu_load") ctx->ffn_glu_load = value != 0;
    else if (n == "ffn_streamed") ctx->ffn_streamed = value != 0;
    else if (n == "mmfs_all") ctx->mmfs_all = value != 0;
    else if (n == "mmfs_min_rows") ctx->mmfs_min_rows = std::max(1u, u);
    else if (n == "batch_overlap") ctx->batch_overlap = value != 0;
    else if (n == "mm8s_all") ctx->mm8s_all = value != 0;
    else if (n == "mm8s_depth") ctx->mm8s_depth = u;
    else if (n == "mm8s_areg") ctx->mm8s_areg = value != 0;
    else if (n == "mm8s_fold") ctx->mm8s_fold_on = value != 0;
    else if (n == "mm8s_split") ctx->mm8s_split_on = value != 0;
    else if (n == "mm8s_q8_0") ctx->mm8s_q8_0 = value != 0;
    else if (n == "mm8_small_to_gemv") ctx->mm8_small_to_gemv = value != 0;
    else if (n == "mm8s_min_rows") ctx->mm8s_min_rows = std::max(1u, u);
    else if (n == "ffn_fused") ctx->ffn_fused = value != 0;
    else if (n == "mmf_small_min_m") ctx->mmf_small_min_m = u;
    else if (n == "mm8_ksplit") ctx->mm8_ksplit_max = u;
    else if (n == "mm8_q6k_min_m") ctx->mm8_q6k_min_m = u;
    else if (n == "mm8_q5k_min_m") ctx->mm8_q5k_min_m = u;
    else if (n == "mm8_q8_0_min_m") ctx->mm8_q8_0_min_m = u;
    else if (n == "moe_mm8") ctx->moe_mm8 = value != 0;
    else if (n == "moe_mm8_q6k") ctx->moe_mm8_q6k = value != 0;
    else if (n == "moe_mm8_rows") ctx->moe_mm8_rows = value != 0;
    else if (n == "moe_glu") ctx->moe_glu = value != 0;
    else if (n == "moe_streamed") ctx->moe_streamed = u;
    else if (n == "moe_wide") ctx->moe_wide = value != 0;
    else if (n == "moe_wide_few") ctx->moe_wide_few = u;
    else if (n == "moe_wide_min") {
        ctx->moe_wide_min = std::max(1u, u);
        ctx->moe_wide_cost = false;
    }
    else if (n == "moe_depth") ctx->moe_depth = u;
    else if (n == "moe_slices") ctx->moe_slices = u;
    else if (n == "prefetch") ctx->prefetch = value != 0;
    else if (n == "prefetch_wgs") ctx->prefetch_wgs = u;
    else if (n == "prefetch_threads") ctx->prefetch_threads = std::min(256u, std::max(64u, u & ~63u));
    else if (n == "prefetch_timeout_us") ctx->prefetch_timeout_us = u;
    else if (n == "prefetch_flags") ctx->prefetch_flags = u;
    else if (n == "prefetch_announce") ctx->prefetch_announce = value != 0;
    else if (n == "prefetch_min_kib") ctx->prefetch_min_kib = u;
    else if (n == "weights_cache_mib") ctx->weights_cache_limit = static_cast<size_t>(u) << 20;
    else return fail(ctx, GLLMQ_ERR_INVALID, "set_option: unknown option %s", name);
    return GLLMQ_OK;
}

const char *gllmq_last_kernel_name(const gllmq_ctx *ctx)
{
    if (!ctx || !ctx->last_kernel) return "";
    const auto it = ctx->kernel_names.find(ctx->last_kernel);
    return it == ctx->kernel_names.end() ? "" : it->second.c_str();
}

int gllmq_dequantize(gllmq_ctx *ctx, const void *blocks, size_t n_bytes, float *out, size_t n_out,
                     uint32_t dtype, void *stream)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    const Format *f = find_format(dtype);
    if (!f)
        return fail(ctx, GLLMQ_ERR_UNIMPLEMENTED,
                    "dequantize: ggml dtype %u is not covered (supported: Q8_0=8, Q4_K=12, Q5_K=13, Q6_K=14)", dtype);
    const size_t nb = std::min(n_bytes / f->block_bytes, n_out / f->block_size);
    if (nb == 0) return GLLMQ_OK;
    if (!blocks || !out) return fail(ctx, GLLMQ_ERR_INVALID, "dequantize: NULL device pointer");
    if (!aligned(out, 4)) return fail(ctx, GLLMQ_ERR_BAD_ALIGNMENT, "dequantize: output must be 4-byte aligned");
    uint64_t n_quads = static_cast<uint64_t>(nb) * (f->block_size / 4);
    const int vec = aligned(out, 16) ? 1 : 0;
    const uint64_t want = (n_quads + 255) / 256;
    const uint32_t grid = static_cast<uint32_t>(std::min<uint64_t>(want, static_cast<uint64_t>(ctx->num_cus) * 64));
    struct { const void *b; float *o; uint64_t n; } args = { blocks, out, n_quads };
    hipFunction_t fn = ctx->dequant[format_index(dtype)][vec];
    if (vec && aligned(blocks, 16) && dtype == T_Q4_K) fn = ctx->dequant_wave;
    if (vec && aligned(blocks, 16) && dtype == T_Q5_K) fn = ctx->dequant_wave_q5k;
    return launch(ctx, fn, grid, 256, 0, stream, &args, sizeof args);
}

int gllmq_quant_gather(gllmq_ctx *ctx, const void *table, size_t table_bytes, uint32_t dtype, size_t vocab,
                       size_t hidden, const uint32_t *ids, size_t count, float scale, float *out, void *stream)
{
    return gllmq_quant_gather_elem(ctx, table, table_bytes, dtype, vocab, hidden, ids, count, scale, out, GLLMQ_ELEM_F32, stream);
}

int gllmq_quant_gather_elem(gllmq_ctx *ctx, const void *table, size_t table_bytes, uint32_t dtype, size_t vocab,
                            size_t hidden, const uint32_t *ids, size_t count, float scale, void *out, int elem, void *stream)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    if (elem != GLLMQ_ELEM_F32 && elem != GLLMQ_ELEM_F16 && elem != GLLMQ_ELEM_BF16)
        return fail(ctx, GLLMQ_ERR_INVALID, "quant_gather: unknown element type %d", elem);
    const bool e16 = elem != GLLMQ_ELEM_F32;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    const Format *f = find_format(dtype);
    if (!f)
        return fail(ctx, GLLMQ_ERR_UNIMPLEMENTED,
                    "quant_gather: ggml dtype %u is not covered (supported: Q8_0=8, Q4_K=12, Q5_K=13, Q6_K=14)", dtype);
    if (count == 0 || hidden == 0) return GLLMQ_OK;
    if (!table || !ids || !out) return fail(ctx, GLLMQ_ERR_INVALID, "quant_gather: NULL device pointer");
    if (hidden % 4 != 0) return fail(ctx, GLLMQ_ERR_BAD_SHAPE, "quant_gather: hidden = %zu is not a multiple of 4", hidden);
    if (vocab > 0xFFFFFFFFu || hidden > 0x7FFFFFFFu || count > 0x7FFFFFFFu)
        return fail(ctx, GLLMQ_ERR_BAD_SHAPE, "quant_gather: dimension exceeds its 32-bit range");
    const size_t rb = gllmq_row_bytes(dtype, hidden);
    if (table_bytes < vocab * rb)
        return fail(ctx, GLLMQ_ERR_BAD_SHAPE, "quant_gather: table has %zu bytes, %zu rows of %zu elements need %zu",
                    table_bytes, vocab, hidden, vocab * rb);
    if (!aligned(ids, 4) || !aligned(out, e16 ? 2 : 4))
        return fail(ctx, GLLMQ_ERR_BAD_ALIGNMENT, "quant_gather: ids must be 4-byte aligned, the output aligned to its element");
    GatherParams P{};
    P.table = static_cast<const uint8_t *>(table);
    P.ids = ids;
    P.out = static_cast<float *>(out);
    P.vocab = static_cast<uint32_t>(vocab);
    P.hidden = static_cast<uint32_t>(hidden);
    P.row_bytes = static_cast<uint32_t>(rb);
    P.quads_per_row = static_cast<uint32_t>(hidden / 4);
    P.count = static_cast<uint32_t>(count);
    P.scale = scale;
    P.elem = static_cast<uint32_t>(elem);
    // hidden is a multiple of 4, so every row is as aligned as the first; of 8: 16-bit rows go in 16-byte stores
    const int vec = e16 && aligned(out, 16) && hidden % 8 == 0 ? 2 : aligned(out, e16 ? 8 : 16) ? 1 : 0;
    // As many rows per workgroup as let all of them be on the chip at once (eight workgroups of 256 threads a CU).
    const uint32_t runs = vec == 2 ? P.quads_per_row / 2u : P.quads_per_row, across = (runs + 255u) / 256u, round = 8u * static_cast<uint32_t>(ctx->num_cus);
    P.rows = static_cast<uint32_t>(std::min<uint64_t>(gq::GATHER_ROWS, (static_cast<uint64_t>(across) * count + round - 1) / round));
    const size_t groups = (count + P.rows - 1) / P.rows;
    return launch2d(ctx, (e16 ? ctx->gather_e16[format_index(dtype)] : ctx->gather[format_index(dtype)])[vec], across,
                    static_cast<uint32_t>(std::min<size_t>(groups, 65535)), 256, 0, stream, &P, sizeof P);
}

int gllmq_argmax(gllmq_ctx *ctx, const float *logits, size_t rows, size_t n, size_t ld, uint32_t *token, float *value,
                 void *stream)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    if (rows == 0) return GLLMQ_OK;
    if ((!logits && n > 0) || !token) return fail(ctx, GLLMQ_ERR_INVALID, "argmax: NULL device pointer");
    if (n > 0xFFFFFFFEu || ld > 0xFFFFFFFFu || rows > 0x7FFFFFFFu || ld < n)
        return fail(ctx, GLLMQ_ERR_BAD_SHAPE, "argmax: n = %zu, ld = %zu, rows = %zu out of range", n, ld, rows);
    if (!aligned(logits, 4) || !aligned(token, 4) || (value && !aligned(value, 4)))
        return fail(ctx, GLLMQ_ERR_BAD_ALIGNMENT, "argmax: buffers must be 4-byte aligned");
    Scratch *S = nullptr;
    int src = acquire_scratch(ctx, stream, &S);
    if (src != GLLMQ_OK) return src;
    ArgmaxParams P{};
    P.keys = S->argmax_keys;
    P.n = static_cast<uint32_t>(n);
    P.ld = static_cast<uint32_t>(ld);
    P.parts = static_cast<uint32_t>(std::min<size_t>(gq::ARGMAX_MAX_PARTS, std::max<size_t>(1, (n + 4095) / 4096)));
    P.chunk = static_cast<uint32_t>((n + P.parts - 1) / P.parts);
    for (size_t r0 = 0; r0 < rows; r0 += gq::ARGMAX_MAX_ROWS) {
        const uint32_t rr = static_cast<uint32_t>(std::min<size_t>(gq::ARGMAX_MAX_ROWS, rows - r0));
        P.logits = logits + r0 * ld;
        P.token = token + r0;
        P.value = value ? value + r0 : nullptr;
        int rc = launch2d(ctx, ctx->argmax_part, P.parts, rr, 256, 0, stream, &P, sizeof P, P.parts > 1);
        if (rc == GLLMQ_OK && P.parts > 1) rc = launch(ctx, ctx->argmax_final, rr, 256, 0, stream, &P, sizeof P, true);
        if (rc != GLLMQ_OK) return rc;
    }
    return GLLMQ_OK;
}

int gllmq_lm_head_argmax(gllmq_ctx *ctx, const void *w, size_t w_bytes, const float *x, uint32_t dtype, size_t n, size_t k,
                         float *logits, uint32_t *token, float *value, void *stream)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    if (!token) return fail(ctx, GLLMQ_ERR_INVALID, "lm_head_argmax: NULL token pointer");
    if (!aligned(token, 4) || (value && !aligned(value, 4)))
        return fail(ctx, GLLMQ_ERR_BAD_ALIGNMENT, "lm_head_argmax: buffers must be 4-byte aligned");
    if (n == 0) return fail(ctx, GLLMQ_ERR_BAD_SHAPE, "lm_head_argmax: n = 0");
    const Format *f = find_format(dtype);
    // checked as the one-row matmul it is; without a logits buffer the activations stand in for it
    int rc = check_matmul_args(ctx, f, w, w_bytes, x, logits ? logits : const_cast<float *>(x), dtype, 1, n, k);
    if (rc >= 0) return rc;
    Scratch *S = nullptr;
    rc = acquire_scratch(ctx, stream, &S);
    if (rc != GLLMQ_OK) return rc;
    // The matvec whose workgroups leave their best candidate behind; the workgroup that
    // finishes last picks among the candidates.  The one-row GEMV of Q6_K and
    // Q8_0 (the types of GGUF output matrices) where one launch covers K: with a logits buffer where the GEMV is
    // the kernel gllmq_quantized_matmul gives the shape anyway (dispatch_choice() asks the dispatch
    // itself), so that the logits are that call's bit for bit; without one, always.  With a logits buffer, of any
    // format, the streamed kernel where that is the one the shape gets (run_mm8s sees the choice that is wanted).
    const size_t rb = gllmq_row_bytes(dtype, k);
    const bool gemv_type = dtype == 14u || dtype == 8u;
    bool gemv_anyway = true;
    if (ctx->lm_head_fused && gemv_type && !ctx->gemv_f32 && k <= 16384 && logits) {
        const DispatchChoice c = dispatch_choice(ctx, [&] {
            return dispatch_matmul(ctx, *S, *f, static_cast<const uint8_t *>(w), x, logits, 1, n, k, false, stream);
        });
        gemv_anyway = c.fn != nullptr && c.fn == ctx->gemv_i8[format_index(dtype)][0];
    }
    if (ctx->lm_head_fused && gemv_type && !ctx->gemv_f32 && k <= 16384 && gemv_anyway) {
        GemvPlan L = plan_gemv(ctx, 1, static_cast<uint32_t>(n), static_cast<uint32_t>(k), rb, ctx->gemv_waves);
        if (L.grid <= gq::ARGMAX_MAX_PARTS * gq::ARGMAX_MAX_ROWS) {
            GemvParams &P = L.P;
            P.w = static_cast<const uint8_t *>(w);
            P.x = x;
            P.y = logits;
            P.ldx = static_cast<uint32_t>(k);
            P.ldy = static_cast<uint32_t>(n);
            P.x_vec = aligned(x, 16);
            P.keys = S->argmax_keys;
            P.ticket = S->mm8_arrive + kLmHeadTicketAt;
            P.token = token;
            P.value = value;
            return launch(ctx, ctx->gemv_i8_argmax[format_index(dtype)], L.grid, L.threads, L.lds, stream, &P, sizeof P, true);
        }
    }
    if (!logits)
        return fail(ctx, GLLMQ_ERR_UNIMPLEMENTED,
                    "lm_head_argmax: this matrix (ggml dtype %u, k = %zu) goes through the matmul and the token choice one "
                    "after the other, which needs a logits buffer of n floats", dtype, k);
    TokenChoice choice{ logits, n, S->argmax_keys, S->mm8_arrive + kLmHeadTicketAt, token, value, false };
    if (ctx->lm_head_fused) ctx->call_token = &choice;
    rc = dispatch_matmul(ctx, *S, *f, static_cast<const uint8_t *>(w), x, logits, 1, n, k, false, stream);
    ctx->call_token = nullptr;
    if (rc != GLLMQ_OK || choice.made) return rc;
    return gllmq_argmax(ctx, logits, 1, n, n, token, value, stream);
}

int gllmq_quantized_matmul_ex(gllmq_ctx *ctx, const void *w, size_t w_bytes, const float *x, float *y,
                              uint32_t dtype, size_t m, size_t n, size_t k, int act_mode, void *stream)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    Scratch *S = nullptr;
    int rc = acquire_scratch(ctx, stream, &S);
    if (rc != GLLMQ_OK) return rc;
    return matmul_on_scratch(ctx, *S, w, w_bytes, x, y, dtype, m, n, k, act_mode, stream);
}

namespace {

int convert_elems(gllmq_ctx *ctx, const void *src, void *dst, size_t count, uint32_t elem, bool widen, void *stream)
{
    gq::ConvertParams C{};
    C.src = src;
    C.dst = dst;
    C.count = count;
    C.elem = elem;
    C.widen = widen ? 1u : 0u;
    const uint32_t grid = static_cast<uint32_t>(std::min<size_t>((count + 255) / 256, 4096));
    return launch(ctx, ctx->convert_elem, std::max(1u, grid), 256, 0, stream, &C, sizeof C, true);
}

size_t elem_scratch_bytes(size_t m, size_t n, size_t k) { return ((m * k * 4 + 255) & ~size_t(255)) + m * n * 4; }

// Whether the kernels convert 16-bit elements in their own loads and stores: all but the GEMV when
// it covers K in several launches (which add up in y), and its f32 flavour.
bool elem_in_kernel(const gllmq_ctx *ctx, size_t m, size_t k)
{
    (void)m;
    return ctx->elem_fused && !ctx->gemv_f32 && k <= 16384;
}

} // namespace

namespace {

// One validated quantized matmul over 16-bit activations and outputs with the scratch of `S`
// (call_mutex held); elem is GLLMQ_ELEM_F16 or GLLMQ_ELEM_BF16.
int matmul_elem_on_scratch(gllmq_ctx *ctx, Scratch &S, const void *w, size_t w_bytes, const void *x, void *y, uint32_t dtype,
                           size_t m, size_t n, size_t k, int elem, void *stream)
{
    const Format *f = find_format(dtype);
    int rc = check_matmul_args(ctx, f, w, w_bytes, static_cast<const float *>(x), static_cast<float *>(y), dtype, m, n, k);
    if (rc >= 0) return rc;
    if (elem_in_kernel(ctx, m, k)) {
        ctx->call_elem = static_cast<uint32_t>(elem);
        rc = dispatch_matmul(ctx, S, *f, static_cast<const uint8_t *>(w), static_cast<const float *>(x),
                             static_cast<float *>(y), m, n, k, false, stream);
        ctx->call_elem = 0;
        if (rc != kNeedPlainActivations) return rc; // else: the kernel for this shape reads f32 only
    }
    rc = grow_scratch(ctx, S, &S.elem, &S.elem_bytes, elem_scratch_bytes(m, n, k), stream, "quantized_matmul_elem");
    if (rc != GLLMQ_OK) return rc;
    float *xf = static_cast<float *>(S.elem);
    float *yf = reinterpret_cast<float *>(static_cast<uint8_t *>(S.elem) + ((m * k * 4 + 255) & ~size_t(255)));
    rc = convert_elems(ctx, x, xf, m * k, static_cast<uint32_t>(elem), true, stream);
    if (rc == GLLMQ_OK) rc = dispatch_matmul(ctx, S, *f, static_cast<const uint8_t *>(w), xf, yf, m, n, k, false, stream);
    if (rc == GLLMQ_OK) rc = convert_elems(ctx, yf, y, m * n, static_cast<uint32_t>(elem), false, stream);
    return rc;
}

} // namespace

int gllmq_quantized_matmul_elem(gllmq_ctx *ctx, const void *w, size_t w_bytes, const void *x, void *y, uint32_t dtype,
                                size_t m, size_t n, size_t k, int elem, void *stream)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    if (elem == GLLMQ_ELEM_F32)
        return gllmq_quantized_matmul_ex(ctx, w, w_bytes, static_cast<const float *>(x), static_cast<float *>(y), dtype, m, n,
                                         k, GLLMQ_ACT_F32_SPLIT, stream);
    if (elem != GLLMQ_ELEM_F16 && elem != GLLMQ_ELEM_BF16)
        return fail(ctx, GLLMQ_ERR_INVALID, "quantized_matmul_elem: unknown element type %d", elem);
    Scratch *S = nullptr;
    int rc = acquire_scratch(ctx, stream, &S);
    if (rc != GLLMQ_OK) return rc;
    return matmul_elem_on_scratch(ctx, *S, w, w_bytes, x, y, dtype, m, n, k, elem, stream);
}

int gllmq_reserve_matmul_elem(gllmq_ctx *ctx, uint32_t dtype, size_t m, size_t n, size_t k, int elem, void *stream)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    int rc = gllmq_reserve_matmul(ctx, dtype, m, n, k, stream);
    // (which kernel takes the shape also depends on the pointers' alignment: room for the widened copies either way)
    if (rc != GLLMQ_OK || elem == GLLMQ_ELEM_F32 || m == 0 || n == 0 || k == 0) return rc;
    Scratch *S = nullptr;
    rc = acquire_scratch(ctx, stream, &S);
    if (rc != GLLMQ_OK) return rc;
    return grow_scratch(ctx, *S, &S->elem, &S->elem_bytes, elem_scratch_bytes(m, n, k), stream, "reserve_matmul_elem");
}

namespace {

// The feed-forward block (call_mutex held).  x and out are of type `elem`; where the kernels of the
// shape take f32 only, kNeedPlainActivations comes back and nothing has been enqueued.
int ffn_on_stream(gllmq_ctx *ctx, const void *gate_w, const void *up_w, size_t gate_up_bytes_each, uint32_t dtype_gate_up,
                  const void *down_w, size_t down_bytes, uint32_t dtype_down, const float *x, float *out, uint32_t elem, size_t m,
                  size_t hidden, size_t ffn, int relu_gate, void *stream)
{
    const Format *fg = find_format(dtype_gate_up), *fd = find_format(dtype_down);
    if (!fg || !fd)
        return fail(ctx, GLLMQ_ERR_UNIMPLEMENTED,
                    "ffn_swiglu: ggml dtype %u / %u is not covered (supported: Q8_0=8, Q4_K=12, Q5_K=13, Q6_K=14)",
                    dtype_gate_up, dtype_down);
    if (m == 0 || hidden == 0) return GLLMQ_OK;
    if (ffn == 0) return fail(ctx, GLLMQ_ERR_BAD_SHAPE, "ffn_swiglu: ffn = 0");
    if (!up_w) return fail(ctx, GLLMQ_ERR_INVALID, "ffn_swiglu: NULL device pointer");
    // the three matrices are checked as the matmuls they are (the intermediate buffers stand in
    // for the activations that are not the caller's)
    int rc = check_matmul_args(ctx, fg, gate_w, gate_up_bytes_each, x, out, dtype_gate_up, m, ffn, hidden);
    if (rc >= 0) return rc;
    rc = check_matmul_args(ctx, fg, up_w, gate_up_bytes_each, x, out, dtype_gate_up, m, ffn, hidden);
    if (rc >= 0) return rc;
    rc = check_matmul_args(ctx, fd, down_w, down_bytes, x, out, dtype_down, m, hidden, ffn);
    if (rc >= 0) return rc;
    if (ffn > 0x7FFFFFFFu / 2u) return fail(ctx, GLLMQ_ERR_BAD_SHAPE, "ffn_swiglu: ffn exceeds 2^30-1");

    // scratch: h [m][ffn], then gate/up results [m][2 ffn] for the form with three steps
    const size_t h_bytes = ffn_h_bytes(m, ffn);
    const size_t need = ffn_scratch_bytes(m, ffn);
    Scratch *Sp = nullptr;
    rc = acquire_scratch(ctx, stream, &Sp);
    if (rc != GLLMQ_OK) return rc;
    Scratch &S = *Sp;
    rc = grow_scratch(ctx, S, &S.ffn, &S.ffn_bytes, need, stream, "ffn_swiglu");
    if (rc != GLLMQ_OK) return rc;
    float *h = static_cast<float *>(S.ffn);
    float *gu = reinterpret_cast<float *>(static_cast<uint8_t *>(S.ffn) + h_bytes);
    const uint8_t *gw = static_cast<const uint8_t *>(gate_w), *uw = static_cast<const uint8_t *>(up_w);

    // Prompts and larger batches: gate and up share their activation images and run as one launch; the
    // down projection's images are prepared from the two results.
    const size_t gate_up_n[2] = { ffn, ffn };
    // 5 to 8 rows, from 64 M gate and up weights on and whatever the element type (16-bit results are the f32 block's, rounded).
    // us per call, int8 and GEMM, f32: Q5_K with Q6_K down eight rows 2 x 2048 x 5632 29.2, 32.5, 2 x 3072 x 8192 36.5, 42.5, 2 x 4096 x
    // 8192 54.9, 47.8, 2 x 4096 x 14336 80, 65; Q6_K seven rows 49.1, 44.3 (3072 x 8192), 58.1, 51.0 (4096 x 8192), 89, 72 (4096 x 14336); Q8_0 50.5,
    // 49.1, 60.0, 53.4, 96, 74.  16-bit blocks of fewer rows are ahead on the int8 kernels with conversions (Q4_K with Q6_K
    // down 2 x 4096 x 14336, five bf16 rows 48.5, 56.2), of eight no more (60.4, 56.5).
    const bool wide = m >= std::max(5u, std::min(ctx->mmfw_min_m, ctx->mmfw_small_min_m)) ||
                      (ctx->ffn_fused && 2 * ffn * hidden >= (64ull << 20) && mmfw_takes_few(ctx, dtype_gate_up, m)); // ("ffn_fused" off: up to 8 rows in separate steps)
    auto fits = [&](MmfwPlan L) { return L.ok && mmfw_fit(ctx, S, L, stream); };
    MmfwPlan down_plan;
    if (wide && !ctx->mmfs_all && ffn % 4 == 0 && m * ffn <= 0xFFFFFFFFull) down_plan = plan_mmfw(ctx, dtype_down, m, &hidden, 1, ffn, false);
    if (fits(down_plan) && fits(plan_mmfw(ctx, dtype_gate_up, m, gate_up_n, 2, hidden, elem != 0))) {
        const MmfwMatrix gate_up[2] = { { gw, gu, ffn }, { uw, gu + m * ffn, ffn } };
        MmfwSlices sums;
        sums.next_need = down_plan.need();
        sums.next_reserve = std::max(down_plan.need(), mmfw_reserve(ctx, m, ffn));
        sums.next_decoded = plan_mmfx(ctx, down_plan, mmf_format(dtype_down), &hidden, 1, m).bytes;
        rc = run_mmfw(ctx, S, *fg, gate_up, 2, x, elem, 0, m, hidden, false, stream, 5, ctx->ffn_glu_load && down_plan.rows >= m ? &sums : nullptr);
        if (rc > 0) return rc;
        if (rc == GLLMQ_OK) {
            const MmfwMatrix down{ static_cast<const uint8_t *>(down_w), out, hidden };
            if (ctx->ffn_glu_load) {
                ctx->call_glu = relu_gate ? 2u : 1u;
                ctx->call_glu_off = static_cast<uint32_t>(m * ffn);
                ctx->call_ldx = static_cast<uint32_t>(ffn);
                if (sums.slices) { // [gate, up][slice][m][ffn]
                    ctx->call_glu_off = static_cast<uint32_t>(sums.slices * m * ffn);
                    rc = run_mmfw(ctx, S, *fd, &down, 1, sums.at, 0, elem, m, ffn, false, stream, 5, nullptr, &sums);
                } else {
                    rc = run_mmfw(ctx, S, *fd, &down, 1, gu, 0, elem, m, ffn, false, stream, 5);
                }
                ctx->call_glu = ctx->call_glu_off = ctx->call_ldx = 0;
            } else {
                gq::GluActParams A{};
                A.h = h;
                A.g = gu;
                A.u = gu + m * ffn;
                A.m = static_cast<uint32_t>(m);
                A.ffn = A.ld = static_cast<uint32_t>(ffn);
                A.relu_gate = relu_gate ? 1u : 0u;
                rc = launch2d(ctx, ctx->glu_act, static_cast<uint32_t>((ffn + 255) / 256),
                              static_cast<uint32_t>(std::min<size_t>(m, 65535)), 256, 0, stream, &A, sizeof A);
                if (rc == GLLMQ_OK) rc = run_mmfw(ctx, S, *fd, &down, 1, h, 0, elem, m, ffn, false, stream, 5);
            }
            return rc >= 0 ? rc : fail(ctx, GLLMQ_ERR_BAD_SHAPE, "ffn_swiglu: the down projection has no kernel for this shape");
        }
    }
    if (elem) return kNeedPlainActivations;
    // gate and up in one launch with the activation in its epilogue (Q4_K / Q5_K, up to 8 rows)
    rc = -1;
    if (ctx->ffn_fused && ctx->ffn_streamed && m <= 4) rc = run_mm8s(ctx, *fg, gw, x, h, m, ffn, hidden, false, stream, uw, relu_gate != 0);
    if (rc < 0 && ctx->ffn_fused && m <= 8) rc = run_mm8(ctx, S, *fg, gw, x, h, m, ffn, hidden, false, stream, true, uw, relu_gate != 0);
    if (rc > 0) return rc;
    if (rc < 0) {
        // three steps: the two products (one matmul when the up rows follow the gate rows in
        // memory), the activation, the down projection
        const size_t rb = gllmq_row_bytes(dtype_gate_up, hidden);
        const bool stacked = uw == gw + ffn * rb;
        gq::GluActParams A{};
        A.h = h;
        A.m = static_cast<uint32_t>(m);
        A.ffn = static_cast<uint32_t>(ffn);
        A.relu_gate = relu_gate ? 1u : 0u;
        if (stacked) {
            rc = dispatch_matmul(ctx, S, *fg, gw, x, gu, m, 2 * ffn, hidden, false, stream);
            A.g = gu;
            A.u = gu + ffn;
            A.ld = static_cast<uint32_t>(2 * ffn);
        } else {
            rc = dispatch_matmul(ctx, S, *fg, gw, x, gu, m, ffn, hidden, false, stream);
            if (rc == GLLMQ_OK) rc = dispatch_matmul(ctx, S, *fg, uw, x, gu + m * ffn, m, ffn, hidden, false, stream);
            A.g = gu;
            A.u = gu + m * ffn;
            A.ld = static_cast<uint32_t>(ffn);
        }
        if (rc != GLLMQ_OK) return rc;
        // the down projection reads act(gate) * up straight from the two results where its kernel
        // can; else the activation runs as a launch of its own and writes h
        const size_t up_off = static_cast<size_t>(A.u - A.g);
        if (ctx->ffn_glu_load && up_off <= 0xFFFFFFFFu) {
            ctx->call_glu = relu_gate ? 2u : 1u;
            ctx->call_glu_off = static_cast<uint32_t>(up_off);
            ctx->call_ldx = A.ld;
            rc = dispatch_matmul(ctx, S, *fd, static_cast<const uint8_t *>(down_w), gu, out, m, hidden, ffn, false, stream);
            ctx->call_glu = ctx->call_glu_off = ctx->call_ldx = 0;
            if (rc != kNeedPlainActivations) return rc;
        }
        rc = launch2d(ctx, ctx->glu_act, static_cast<uint32_t>((ffn + 255) / 256),
                      static_cast<uint32_t>(std::min<size_t>(m, 65535)), 256, 0, stream, &A, sizeof A);
        if (rc != GLLMQ_OK) return rc;
    }
    return dispatch_matmul(ctx, S, *fd, static_cast<const uint8_t *>(down_w), h, out, m, hidden, ffn, false, stream);
}

} // namespace

int gllmq_ffn_swiglu(gllmq_ctx *ctx, const void *gate_w, const void *up_w, size_t gate_up_bytes_each, uint32_t dtype_gate_up,
                     const void *down_w, size_t down_bytes, uint32_t dtype_down, const float *x, float *out, size_t m,
                     size_t hidden, size_t ffn, int relu_gate, void *stream)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    return ffn_on_stream(ctx, gate_w, up_w, gate_up_bytes_each, dtype_gate_up, down_w, down_bytes, dtype_down, x, out, 0, m, hidden, ffn,
                         relu_gate, stream);
}

namespace {

// What the element-type forms of the feed-forward block and of the expert matvec have in common:
// activations of a 16-bit type are widened into the stream's scratch (exact), the f32 entry point
// runs on them, and unless the result can go straight to `out` (f32, nothing to add) it goes to
// scratch too and one small launch writes out = round(result) or out = round(out + result).
struct ElemStage {
    const float *x = nullptr; // what the f32 entry point reads
    float *result = nullptr;  // where it writes
    bool finish = false;
};

int elem_stage_begin(gllmq_ctx *ctx, const void *x, void *out, size_t count, int elem, int flags, void *stream, const char *what,
                     ElemStage *st)
{
    if (elem != GLLMQ_ELEM_F32 && elem != GLLMQ_ELEM_F16 && elem != GLLMQ_ELEM_BF16)
        return fail(ctx, GLLMQ_ERR_INVALID, "%s: unknown element type %d", what, elem);
    if (flags & ~GLLMQ_OUT_ACCUMULATE) return fail(ctx, GLLMQ_ERR_INVALID, "%s: unknown flag bits 0x%x", what, flags);
    st->x = static_cast<const float *>(x);
    st->result = static_cast<float *>(out);
    st->finish = elem != GLLMQ_ELEM_F32 || (flags & GLLMQ_OUT_ACCUMULATE);
    if (!st->finish || count == 0) return GLLMQ_OK;
    if (!x || !out) return fail(ctx, GLLMQ_ERR_INVALID, "%s: NULL device pointer", what);
    if (!aligned(x, 2) || !aligned(out, 2)) return fail(ctx, GLLMQ_ERR_BAD_ALIGNMENT, "%s: x and out must be aligned to their element", what);
    Scratch *S = nullptr;
    int rc = acquire_scratch(ctx, stream, &S);
    if (rc != GLLMQ_OK) return rc;
    const size_t each = (count * 4 + 255) & ~size_t(255);
    rc = grow_scratch(ctx, *S, &S->elem, &S->elem_bytes, 2 * each, stream, what);
    if (rc != GLLMQ_OK) return rc;
    st->result = reinterpret_cast<float *>(static_cast<uint8_t *>(S->elem) + each);
    if (elem != GLLMQ_ELEM_F32) {
        float *xf = static_cast<float *>(S->elem);
        rc = convert_elems(ctx, x, xf, count, static_cast<uint32_t>(elem), true, stream);
        st->x = xf;
    }
    return rc;
}

int elem_stage_end(gllmq_ctx *ctx, const ElemStage &st, void *out, size_t count, int elem, int flags, void *stream)
{
    if (!st.finish || count == 0) return GLLMQ_OK;
    gq::ConvertParams C{};
    C.src = st.result;
    C.dst = out;
    C.count = count;
    C.elem = static_cast<uint32_t>(elem);
    C.accumulate = (flags & GLLMQ_OUT_ACCUMULATE) ? 1u : 0u;
    const uint32_t grid = static_cast<uint32_t>(std::min<size_t>((count + 255) / 256, 4096));
    return launch(ctx, ctx->finish_elem, std::max(1u, grid), 256, 0, stream, &C, sizeof C, true);
}

} // namespace

int gllmq_ffn_swiglu_elem(gllmq_ctx *ctx, const void *gate_w, const void *up_w, size_t gate_up_bytes_each, uint32_t dtype_gate_up,
                          const void *down_w, size_t down_bytes, uint32_t dtype_down, const void *x, void *out, size_t m,
                          size_t hidden, size_t ffn, int relu_gate, int elem, int flags, void *stream)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    int rc = kNeedPlainActivations;
    if ((elem == GLLMQ_ELEM_F16 || elem == GLLMQ_ELEM_BF16) && flags == 0 && ctx->elem_fused && aligned(x, 16) && aligned(out, 4))
        rc = ffn_on_stream(ctx, gate_w, up_w, gate_up_bytes_each, dtype_gate_up, down_w, down_bytes, dtype_down,
                           static_cast<const float *>(x), static_cast<float *>(out), static_cast<uint32_t>(elem), m, hidden, ffn, relu_gate, stream);
    if (rc != kNeedPlainActivations) return rc;
    ElemStage st;
    rc = elem_stage_begin(ctx, x, out, m * hidden, elem, flags, stream, "ffn_swiglu", &st);
    if (rc != GLLMQ_OK) return rc;
    rc = gllmq_ffn_swiglu(ctx, gate_w, up_w, gate_up_bytes_each, dtype_gate_up, down_w, down_bytes, dtype_down, st.x, st.result, m,
                          hidden, ffn, relu_gate, stream);
    if (rc != GLLMQ_OK) return rc;
    return elem_stage_end(ctx, st, out, m * hidden, elem, flags, stream);
}

namespace {
int moe_on_stream(gllmq_ctx *ctx, const void *gate, size_t gate_bytes, size_t gate_expert_stride, const void *up,
                  size_t up_bytes, size_t up_expert_stride, uint32_t dtype_gu, const void *down, size_t down_bytes,
                  size_t down_expert_stride, uint32_t dtype_dn, const float *x, float *out, uint32_t elem, size_t tokens,
                  size_t hidden, size_t ffn, size_t experts, size_t top_k, const uint32_t *route_expert,
                  const float *route_weight, const uint32_t *route_len, int relu_gate, void *stream);
}

int gllmq_moe_matvec_elem(gllmq_ctx *ctx, const void *gate, size_t gate_bytes, size_t gate_expert_stride, const void *up,
                          size_t up_bytes, size_t up_expert_stride, uint32_t dtype_gu, const void *down, size_t down_bytes,
                          size_t down_expert_stride, uint32_t dtype_dn, const void *x, void *out, size_t tokens, size_t hidden,
                          size_t ffn, size_t experts, size_t top_k, const uint32_t *route_expert, const float *route_weight,
                          const uint32_t *route_len, int relu_gate, int elem, int flags, void *stream)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    int rc = kNeedPlainActivations;
    if ((elem == GLLMQ_ELEM_F16 || elem == GLLMQ_ELEM_BF16) && flags == 0 && ctx->elem_fused && aligned(x, 16) && aligned(out, 4))
        rc = moe_on_stream(ctx, gate, gate_bytes, gate_expert_stride, up, up_bytes, up_expert_stride, dtype_gu, down, down_bytes,
                           down_expert_stride, dtype_dn, static_cast<const float *>(x), static_cast<float *>(out), static_cast<uint32_t>(elem),
                           tokens, hidden, ffn, experts, top_k, route_expert, route_weight, route_len, relu_gate, stream);
    if (rc != kNeedPlainActivations) return rc;
    ElemStage st;
    rc = elem_stage_begin(ctx, x, out, tokens * hidden, elem, flags, stream, "moe_matvec", &st);
    if (rc != GLLMQ_OK) return rc;
    rc = gllmq_moe_matvec(ctx, gate, gate_bytes, gate_expert_stride, up, up_bytes, up_expert_stride, dtype_gu, down, down_bytes,
                          down_expert_stride, dtype_dn, st.x, st.result, tokens, hidden, ffn, experts, top_k, route_expert,
                          route_weight, route_len, relu_gate, stream);
    if (rc != GLLMQ_OK) return rc;
    return elem_stage_end(ctx, st, out, tokens * hidden, elem, flags, stream);
}

int gllmq_quantized_matmul(gllmq_ctx *ctx, const void *w, size_t w_bytes, const float *x, float *y,
                           uint32_t dtype, size_t m, size_t n, size_t k, void *stream)
{
    return gllmq_quantized_matmul_ex(ctx, w, w_bytes, x, y, dtype, m, n, k, GLLMQ_ACT_F32_SPLIT, stream);
}

namespace {

// One launch (or chained launch) of a batch, as gllmq_quantized_matmul_batch will enqueue it.
struct BatchUnit {
    size_t first, len;
    bool ordered;   // starts after everything before it
    bool announces; // its kernel says when it starts
    unsigned long long seq;
};

int batch_entry(gllmq_ctx *ctx, Scratch &S, const gllmq_matmul_desc &d, void *stream)
{
    constexpr uint32_t kElemBits = GLLMQ_DESC_ELEM_F16 | GLLMQ_DESC_ELEM_BF16;
    if (d.flags & kElemBits)
        return matmul_elem_on_scratch(ctx, S, d.w_dev, d.w_bytes, d.x_dev, d.y_dev, d.ggml_dtype, d.m, d.n, d.k,
                                      (d.flags & GLLMQ_DESC_ELEM_F16) ? GLLMQ_ELEM_F16 : GLLMQ_ELEM_BF16, stream);
    return matmul_on_scratch(ctx, S, d.w_dev, d.w_bytes, d.x_dev, d.y_dev, d.ggml_dtype, d.m, d.n, d.k, GLLMQ_ACT_F32_SPLIT, stream);
}

// Entries from `descs` on that one launch can multiply: independent matmuls of one format over the same
// activation rows (a layer's Q, K and V projections), five and more for the GEMM (4096 + 1024 + 1024 rows of 4096 Q4_K,
// f32, five rows 18 us against 28 one by one), up to four for the streamed kernels.  0 or 1: none.
size_t group_length(const gllmq_ctx *ctx, const gllmq_matmul_desc *descs, size_t count)
{
    constexpr uint32_t kElemBits = GLLMQ_DESC_ELEM_F16 | GLLMQ_DESC_ELEM_BF16;
    const gllmq_matmul_desc &first = descs[0];
    const uint32_t elem = first.flags & kElemBits;
    if (count < 2 || !ctx->batch_group || first.m == 0 || (first.m <= 4 && !ctx->use_chain) || // (option "chain" off: a streamed launch per entry)
        (first.m > 4 && (ctx->mmfs_all || (first.m < std::min(ctx->mmfw_min_m, ctx->mmfw_small_min_m) && ctx->mmfw_small_min_m > 9))) || first.k == 0 || !first.x_dev || elem == kElemBits || (elem && !elem_in_kernel(ctx, first.m, first.k)))
        return 0;
    const size_t e = elem ? 2 : 4;
    size_t len = 0;
    while (len < count && len < static_cast<size_t>(gq::MMFW_MAX_SEGS)) {
        const gllmq_matmul_desc &d = descs[len];
        const uint32_t known = elem | (len == 0 ? static_cast<uint32_t>(GLLMQ_DESC_AFTER_PREVIOUS) : 0u);
        if ((d.flags & ~known) || (d.flags & kElemBits) != elem || d.ggml_dtype != first.ggml_dtype || d.m != first.m || d.k != first.k ||
            d.x_dev != first.x_dev || d.n == 0 || !d.y_dev || d.m > 0x7FFFFFFFu || d.n > 0x7FFFFFFFu || d.k > 0x7FFFFFFFu)
            break;
        bool apart = !ranges_meet(d.y_dev, d.m * d.n * e, d.x_dev, d.m * d.k * e);
        for (size_t i = 0; i < len; ++i) apart = apart && !ranges_meet(d.y_dev, d.m * d.n * e, descs[i].y_dev, descs[i].m * descs[i].n * e);
        if (!apart) break;
        ++len;
    }
    return len;
}

// The group as one launch.  -1: its entries go through the dispatch one by one (which also reports what is wrong with them).
int run_group(gllmq_ctx *ctx, Scratch &S, const gllmq_matmul_desc *descs, size_t len, void *stream)
{
    const gllmq_matmul_desc &first = descs[0];
    const Format *f = find_format(first.ggml_dtype);
    if (!f) return -1;
    MmfwMatrix mats[gq::MMFW_MAX_SEGS];
    size_t n[gq::MMFW_MAX_SEGS];
    const size_t rb = gllmq_row_bytes(first.ggml_dtype, first.k);
    for (size_t i = 0; i < len; ++i) {
        const gllmq_matmul_desc &d = descs[i];
        if (!d.w_dev || rb > (size_t(1) << 26) || d.w_bytes < d.n * rb || !aligned(d.w_dev, f->w_align) || rb % f->w_align != 0 || !aligned(d.y_dev, 4))
            return -1;
        mats[i] = MmfwMatrix{ static_cast<const uint8_t *>(d.w_dev), d.y_dev, d.n };
        n[i] = d.n;
    }
    const uint32_t elem = (first.flags & GLLMQ_DESC_ELEM_F16) ? GLLMQ_ELEM_F16 : (first.flags & GLLMQ_DESC_ELEM_BF16) ? GLLMQ_ELEM_BF16 : 0u;
    // Lines by measurement, us per call, one by one and here, two and three matrices over the same rows.
    if (first.m <= 4) { // rows of up to 4096 elements, any number of weight rows: f32, one row, Q4_K 2 x 14336 x 4096 12.5, 11.9 (a chain before), 2 x 28672 26.1, 24.4, Q8_0 25.0, 24.3, 47.5, 46.2; four rows Q4_K 17.9, 13.5, 29.4, 27.1
        gq::Mm8sGroupParams G{};
        G.segs = static_cast<uint32_t>(len);
        size_t rows = 0;
        for (size_t i = 0; i < len; ++i) {
            G.seg[i] = gq::Mm8sSeg{ mats[i].w, mats[i].y, static_cast<uint32_t>(n[i]), 0u };
            rows += n[i];
        }
        if (rows > 0x7FFFFFFFu || !ctx->use_mm8 || !ctx->use_mm8s) return -1;
        ctx->call_elem = elem;
        const int rc = run_mm8s(ctx, *f, G.seg[0].w, first.x_dev, first.y_dev, first.m, rows, first.k, false, stream, nullptr, false, nullptr, &G);
        ctx->call_elem = 0;
        // Rows of more than 4096 elements, which these kernels leave: the GEMM from three rows on, 16 bits from two.  us per
        // call, one by one in brackets, 5120 + 1024 + 1024 rows of 5120: Q4_K three f32 rows 17.7 (28.7), two bf16 16.5 (34.1), Q8_0
        // 24.7 (41.2), 23.1 (34.3); 8192 + 2 x 1024 rows of 8192 Q4_K 28.7 (32.6), 27.0 (39.1), but two f32 rows 28.5 (27.2).
        if (rc >= 0 || first.k <= 4096 || first.m < (elem ? 2u : 3u) || ctx->mmfw_small_min_m > 9) return rc;
    }
    size_t n_sum = 0;
    for (size_t i = 0; i < len; ++i) n_sum += n[i];
    // The GEMM.  Up to eight rows it takes up to 72 and 48 weight tiles, beyond which its few slices of K leave the int8 kernels ahead: three f32
    // rows Q4_K 3 x 6144 x 6144 35.1, 32.7, 3 x 8192 x 8192 42.6, 52.1, 2 x 14336 x 4352 27.7, 35.1; five rows 3 x 4096 x 4096 28.1, 21.8, 2 x 8192 x 4096 19.2,
    // 23.7 (Q6_K 28.6, 29.0), 2 x 28672 x 4096 42.8, 51.2.
    if (first.m <= 8 && n_sum > (first.m <= 4 ? 72u : 48u) * gq::MMFW_TILE_ROWS) return -1;
    // Nine to sixteen rows of Q4_K and Q5_K, which have a one-launch kernel alone: up to 128 M weights.  Nine f32 rows 2 x 14336 x 4096 33.5, 33.3 and 35.8, 37.3
    // (sixteen of Q4_K 37.6, 34.4); 2 x 14336 x 8192 47.2, 54.6 and 51.3, 62.1; 2 x 28672 x 4096 46.5, 52.0 and 50.7, 58.1.
    if (first.m >= 9 && first.m <= 16 && (first.ggml_dtype == T_Q4_K || first.ggml_dtype == T_Q5_K) && n_sum * first.k > (128ull << 20)) return -1;
    return run_mmfw(ctx, S, *f, mats, static_cast<int>(len), first.x_dev, elem, elem, first.m, first.k, false, stream, 2);
}

// The launches a batch will make, and which of them get their weights prefetched: an ordered
// launch whose kernel and whose predecessor's kernel both say when they start (the predecessor's
// start is the prefetch's cue, its own start tells a late prefetch to give up).  Nothing is
// enqueued here: single entries go through the dispatch in counting mode.
void plan_prefetch(gllmq_ctx *ctx, Scratch &S, const gllmq_matmul_desc *descs, size_t count, void *stream,
                   std::vector<BatchUnit> &units, std::vector<gq::TouchEntry> &touch)
{
    constexpr uint32_t kKnown = GLLMQ_DESC_AFTER_PREVIOUS | GLLMQ_DESC_ELEM_F16 | GLLMQ_DESC_ELEM_BF16;
    size_t alone = 0; // as in gllmq_quantized_matmul_batch, whose launches these are
    for (size_t i = 0; i < count;) {
        BatchUnit u{ i, 1, true, false, 0 };
        const size_t chain = chain_length(ctx, descs + i, count - i);
        const size_t group = i < alone && chain < 2 ? 0 : group_length(ctx, descs + i, chain >= 2 ? chain : count - i);
        const bool starts_anywhere = !(descs[i].flags & GLLMQ_DESC_AFTER_PREVIOUS) && i > 0 && ctx->batch_overlap;
        DispatchChoice c{};
        if (group >= 2 && (chain < 2 || group == chain)) c = dispatch_choice(ctx, [&] { return run_group(ctx, S, descs + i, group, stream); });
        if (c.launches) { // several matrices over the same rows: one number, that of the launch
            u.len = group;
            u.ordered = !starts_anywhere;
            u.announces = c.fn != nullptr && ctx->announces.count(c.fn) != 0;
        } else if (chain >= 2) {
            u.len = chain;
            u.announces = true;
        } else {
            if (group >= 2) alone = i + group;
            if (!(descs[i].flags & ~kKnown)) {
                u.ordered = !starts_anywhere;
                c = dispatch_choice(ctx, [&] { return batch_entry(ctx, S, descs[i], stream); });
                u.announces = c.fn != nullptr && ctx->announces.count(c.fn) != 0;
            }
        }
        u.seq = ++ctx->launch_seq;
        units.push_back(u);
        i += u.len;
    }
    for (size_t j = 1; j < units.size(); ++j) {
        const BatchUnit &u = units[j];
        const gllmq_matmul_desc &d = descs[u.first]; // (of a chain: its first matrix; the chain's own stream carries on from there)
        if (!u.ordered || !u.announces || !units[j - 1].announces || !d.w_dev) continue;
        const size_t bytes = std::min(d.w_bytes, d.n * gllmq_row_bytes(d.ggml_dtype, d.k));
        if (bytes < (static_cast<size_t>(ctx->prefetch_min_kib) << 10)) continue;
        touch.push_back(gq::TouchEntry{ static_cast<const uint8_t *>(d.w_dev), bytes, u.seq });
    }
}

int launch_prefetch(gllmq_ctx *ctx, const std::vector<gq::TouchEntry> &touch)
{
    const uint32_t wgs = ctx->prefetch_wgs ? ctx->prefetch_wgs : static_cast<uint32_t>(ctx->num_cus);
    for (size_t at = 0; at < touch.size(); at += gq::TOUCH_MAX_ENTRIES) {
        gq::TouchParams T{};
        T.progress = ctx->progress;
        T.sink = nullptr;
        T.count = static_cast<uint32_t>(std::min<size_t>(gq::TOUCH_MAX_ENTRIES, touch.size() - at));
        T.timeout_ticks = ctx->prefetch_timeout_us * 100u; // wall_clock64() counts at 100 MHz
        T.flags = ctx->prefetch_flags;
        for (uint32_t i = 0; i < T.count; ++i) T.e[i] = touch[at + i];
        size_t size = sizeof T;
        void *config[] = { HIP_LAUNCH_PARAM_BUFFER_POINTER, &T, HIP_LAUNCH_PARAM_BUFFER_SIZE, &size, HIP_LAUNCH_PARAM_END };
        GLLMQ_HIP(ctx, hipModuleLaunchKernel(ctx->touch, wgs, 1, 1, ctx->prefetch_threads, 1, 1, 0, ctx->side_stream, nullptr, config));
    }
    return GLLMQ_OK;
}

} // namespace

int gllmq_quantized_matmul_batch(gllmq_ctx *ctx, const gllmq_matmul_desc *descs, size_t count, void *stream)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    if (count && !descs) return fail(ctx, GLLMQ_ERR_INVALID, "quantized_matmul_batch: NULL descriptor list");
    Scratch *S = nullptr;
    int rc = acquire_scratch(ctx, stream, &S);
    if (rc != GLLMQ_OK) return rc;
    // (a stream that is being captured gets ordinary launches throughout: what a capture makes of a
    // launch without order is not something to rely on; the graph's replays then run the batch's
    // kernels one after the other)
    const bool capturing = stream_is_capturing(stream);
    const bool overlap_on = ctx->batch_overlap && !capturing;
    ctx->overlap = gllmq_ctx::Overlap{};
    ctx->overlap.on = overlap_on;
    if (*ctx->chain_error) { // a chain launched earlier gave up waiting for a counter: its results are not to be trusted
        *ctx->chain_error = 0u;
        return fail(ctx, GLLMQ_ERR_HIP, "quantized_matmul_batch: an earlier chained launch timed out waiting for the entry before "
                                        "(option chain_spin_limit; is the device shared?): its outputs are invalid");
    }
    // The prefetch launch goes first, on the context's own stream (never into a capture: it is not
    // part of the caller's stream).
    std::vector<BatchUnit> units;
    std::vector<gq::TouchEntry> touch;
    if (ctx->prefetch && count >= 2 && !capturing) plan_prefetch(ctx, *S, descs, count, stream, units, touch);
    if (!touch.empty()) {
        rc = launch_prefetch(ctx, touch);
        if (rc != GLLMQ_OK) return rc;
    }
    size_t unit = 0, alone = 0; // `alone`: entries before this one are of a group that no launch takes
    for (size_t i = 0; i < count && rc == GLLMQ_OK; ++i) {
        const gllmq_matmul_desc &d = descs[i];
        while (unit < units.size() && units[unit].first < i) ++unit;
        const bool planned = !touch.empty() && unit < units.size() && units[unit].first == i && units[unit].announces;
        ctx->call_seq = planned ? units[unit].seq : 0ull;
        // consecutive one-row matmuls of one kind run as one launch whose weight stream never stops
        const size_t chain = chain_length(ctx, descs + i, count - i);
        if (chain >= 2) {
            int crc = -1;
            if (chain <= static_cast<size_t>(gq::MMFW_MAX_SEGS) && group_length(ctx, descs + i, chain) == chain) { // Q, K and V, or gate and up
                ctx->overlap.entry_first = !(d.flags & GLLMQ_DESC_AFTER_PREVIOUS);
                crc = run_group(ctx, *S, descs + i, chain, stream);
                ctx->overlap.entry_first = false;
            }
            if (crc < 0) crc = run_chain(ctx, *S, descs + i, chain, stream);
            if (crc >= 0) {
                rc = crc;
                ctx->overlap = gllmq_ctx::Overlap{};
                ctx->overlap.on = overlap_on;
                i += chain - 1;
                continue;
            }
        }
        const size_t group = chain >= 2 || i < alone ? 0 : group_length(ctx, descs + i, count - i);
        if (group >= 2) {
            ctx->overlap.entry_first = !(d.flags & GLLMQ_DESC_AFTER_PREVIOUS);
            const int grc = run_group(ctx, *S, descs + i, group, stream);
            if (grc >= 0) {
                rc = grc;
                i += group - 1;
                continue;
            }
            alone = i + group;
        }
        constexpr uint32_t kElemBits = GLLMQ_DESC_ELEM_F16 | GLLMQ_DESC_ELEM_BF16;
        if ((d.flags & ~(static_cast<uint32_t>(GLLMQ_DESC_AFTER_PREVIOUS) | kElemBits)) || (d.flags & kElemBits) == kElemBits) {
            rc = fail(ctx, GLLMQ_ERR_INVALID, "quantized_matmul_batch: unknown flag bits 0x%x in entry %zu", d.flags, i);
            break;
        }
        // an entry that depends on the ones before it starts a new group: its first launch is an
        // ordinary one
        ctx->overlap.entry_first = !(d.flags & GLLMQ_DESC_AFTER_PREVIOUS);
        rc = batch_entry(ctx, *S, d, stream);
    }
    ctx->call_seq = 0;
    ctx->overlap = gllmq_ctx::Overlap{};
    if (!touch.empty()) {
        // The caller's stream ends behind the prefetch: whoever waits for the stream may free the
        // weights, which the prefetch must then be through with.
        hipError_t e = hipEventRecord(ctx->side_event, ctx->side_stream);
        if (e == hipSuccess) e = hipStreamWaitEvent(static_cast<hipStream_t>(stream), ctx->side_event, 0);
        if (e != hipSuccess && rc == GLLMQ_OK) rc = fail(ctx, GLLMQ_ERR_HIP, "prefetch: %s", hipGetErrorString(e));
    }
    return rc;
}

int gllmq_chain_status(gllmq_ctx *ctx)
{
    if (!ctx || !ctx->chain_error) return 0;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    const uint32_t raised = *static_cast<volatile uint32_t *>(ctx->chain_error);
    *ctx->chain_error = 0u;
    return raised ? 1 : 0;
}

int gllmq_moe_route(gllmq_ctx *ctx, const float *logits, size_t tokens, size_t experts, size_t top_k,
                    float capacity_factor, uint32_t *route_expert, float *route_weight, uint32_t *route_len,
                    uint32_t *route_pos, uint32_t *expert_counts, uint32_t *overflow, void *stream)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    if (tokens == 0) return GLLMQ_OK;
    if (!logits || !route_expert || !route_weight || !route_len)
        return fail(ctx, GLLMQ_ERR_INVALID, "moe_route: NULL device pointer");
    if (experts == 0 || top_k == 0) return fail(ctx, GLLMQ_ERR_BAD_SHAPE, "moe_route: experts and top_k must be positive");
    if (experts > gq::ROUTE_MAX_EXPERTS || top_k > gq::ROUTE_MAX_TOP_K || tokens > 0x7FFFFFFFu / top_k)
        return fail(ctx, GLLMQ_ERR_UNIMPLEMENTED, "moe_route: experts = %zu (max %u), top_k = %zu (max %u) or tokens = %zu is beyond this build",
                    experts, gq::ROUTE_MAX_EXPERTS, top_k, gq::ROUTE_MAX_TOP_K, tokens);
    if (!aligned(logits, 4) || !aligned(route_expert, 4) || !aligned(route_weight, 4) || !aligned(route_len, 4))
        return fail(ctx, GLLMQ_ERR_BAD_ALIGNMENT, "moe_route: buffers must be 4-byte aligned");
    gq::MoeRouteParams P{};
    P.logits = logits;
    P.route_expert = route_expert;
    P.route_weight = route_weight;
    P.route_len = route_len;
    P.route_pos = route_pos;
    P.expert_counts = expert_counts;
    P.overflow = overflow;
    P.tokens = static_cast<uint32_t>(tokens);
    P.experts = static_cast<uint32_t>(experts);
    P.top_k = static_cast<uint32_t>(top_k);
    // ExpertRouteConfig::expert_capacity (src/moe/routing.rs:53-61): the same f32 arithmetic
    float cap = std::ceil(capacity_factor * static_cast<float>(tokens) / static_cast<float>(experts));
    if (!(cap >= 0.0f)) cap = 0.0f; // negative or NaN
    if (cap > 1.0e9f) cap = 1.0e9f;
    P.capacity = static_cast<uint32_t>(cap);
    const uint32_t lds = static_cast<uint32_t>(((gq::ROUTE_WAVES + 1) * experts + 4) * 4);
    // A token chooses an expert once, so with room for every token in every expert nothing is dropped and the choices
    // stand as phase 1 leaves them; phase 2 would only count.  (16 tokens of 128 experts: 7.7 us against 19.4; 512: 8
    // against 24.)
    const bool no_drop = P.capacity >= P.tokens && !route_pos && !expert_counts;
    if (tokens <= gq::ROUTE_FUSED_MAX_TOKENS && !no_drop) {
        P.phases = 3u;
        return launch(ctx, ctx->moe_route, 1, gq::ROUTE_THREADS, lds, stream, &P, sizeof P);
    }
    P.phases = 1u;
    const uint32_t grid = static_cast<uint32_t>(std::min<size_t>((tokens + gq::ROUTE_WAVES - 1) / gq::ROUTE_WAVES,
                                                                 static_cast<size_t>(ctx->num_cus) * 4));
    int rc = launch(ctx, ctx->moe_route, grid, gq::ROUTE_THREADS, lds, stream, &P, sizeof P);
    if (rc != GLLMQ_OK || no_drop) return rc;
    P.phases = 2u;
    return launch(ctx, ctx->moe_route, 1, gq::ROUTE_THREADS, lds, stream, &P, sizeof P);
}

namespace {

// Carve-up of the MoE workspace (256-byte aligned pieces).
struct MoeWorkspace {
    size_t src, pos, jobs, jobs8, cnt, gu, h, o, total;
};

MoeWorkspace moe_workspace(size_t pairs, size_t hidden, size_t ffn)
{
    auto up256 = [](size_t v) { return (v + 255) & ~static_cast<size_t>(255); };
    MoeWorkspace W{};
    size_t off = 0;
    W.src = off; off = up256(off + pairs * 4);
    W.pos = off; off = up256(off + pairs * 4);
    W.jobs = off; off = up256(off + pairs * sizeof(MoeJob));
    W.jobs8 = off; off = up256(off + pairs * sizeof(MoeJob8));
    W.cnt = off; off = up256(off + 4 * 4);
    W.gu = off; off = up256(off + pairs * 2 * ffn * 4);
    W.h = off; off = up256(off + pairs * ffn * 4);
    W.o = off; off = up256(off + pairs * hidden * 4);
    W.total = off;
    return W;
}

// The weighted sum of each token's routes.
int launch_moe_combine(gllmq_ctx *ctx, MoeCombineParams C, void *stream)
{
    // Four columns a thread from 128 tokens on (512 tokens 15.0 us, 13.0; with 64 there are too few threads for it, 4.2, 4.3).  o is on a
    // boundary of 256 bytes and hidden a multiple of 4 (moe_matvec refuses others), so o's rows are on one of 16.
    const uint32_t per = C.tokens >= 128u ? 4u : 1u;
    return launch2d(ctx, per == 4u ? ctx->moe_combine_v4 : ctx->moe_combine, (C.hidden + 256u * per - 1u) / (256u * per), C.tokens, 256, 0, stream, &C, sizeof C);
}

// Sorts the routed pairs by expert and writes the job tables that `P` points to.
int launch_moe_plan(gllmq_ctx *ctx, MoePlanParams &P, const uint32_t *route_expert, const uint32_t *route_len, size_t tokens,
                    size_t top_k, size_t experts, void *stream)
{
    P.route_expert = route_expert;
    P.route_len = route_len;
    P.tokens = static_cast<uint32_t>(tokens);
    P.top_k = static_cast<uint32_t>(top_k);
    P.top_k_inverse = 0xFFFFFFFFu / P.top_k;
    P.experts = static_cast<uint32_t>(experts);
    P.pairs = static_cast<uint32_t>(tokens * top_k);
    if (P.pairs <= gq::MOE_PLAN_FEW) { // (from 256 pairs on the two take the same time)
        const uint32_t padded = (P.pairs + 63u) & ~63u;
        const uint32_t threads = std::max(padded, std::min(gq::MOE_PLAN_FEW_THREADS, (P.experts + 63u) & ~63u));
        P.experts_per_thread = (P.experts + threads - 1u) / threads;
        return launch(ctx, ctx->moe_plan_few, 1, threads, (2u * P.experts + 2u * padded + 16u) * 4u, stream, &P, sizeof P);
    }
    // a wave per 64 pairs up to 16, as far as their counts (a word per expert each) fit the LDS; no
    // fewer than four, which share the rest of the work
    uint32_t waves = std::min<uint32_t>(gq::MOE_PLAN_THREADS / 64, std::max(4u, (P.pairs + 63u) / 64u));
    while (waves > 4u && (waves + 4u) * P.experts * 4u > 128u * 1024u) waves /= 2u;
    const uint64_t words = static_cast<uint64_t>(waves + 4u) * P.experts + 64u, with_pairs = words + 2ull * P.pairs;
    P.in_lds = with_pairs * 4u <= 128u * 1024u ? 1u : 0u;
    P.experts_per_thread = (P.experts + waves * 64u - 1u) / (waves * 64u);
    return launch(ctx, P.tiles ? ctx->moe_plan_wide : ctx->moe_plan, 1, waves * 64u, static_cast<uint32_t>(P.in_lds ? with_pairs : words) * 4u, stream, &P, sizeof P);
}

// ---- Many tokens per expert (prompts): the GEMM of mmfw.hip.inc over the experts' own rows
struct MoeWidePlan {
    uint32_t max_tiles, max_jobs;
    size_t src, pos, token, tiles, jobs, cnt, gu, o, img, inv, total;
};

MoeWidePlan plan_moe_wide(size_t pairs, size_t hidden, size_t ffn, size_t experts, bool hi_only)
{
    auto up256 = [](size_t v) { return (v + 255) & ~static_cast<size_t>(255); };
    MoeWidePlan W{};
    const size_t hit = std::min(experts, pairs);
    W.max_tiles = static_cast<uint32_t>(pairs / 32 + hit);
    W.max_jobs = static_cast<uint32_t>(pairs / (32 * gq::MMFW_MAX_MT) + hit);
    const size_t gh = (hidden + 255) / 256, gf = (ffn + 255) / 256;
    size_t off = 0;
    W.src = off; off = up256(off + pairs * 4);
    W.pos = off; off = up256(off + pairs * 4);
    W.token = off; off = up256(off + pairs * 4);
    W.tiles = off; off = up256(off + W.max_tiles * sizeof(gq::MoeTile));
    W.jobs = off; off = up256(off + W.max_jobs * sizeof(gq::MoeWideJob));
    W.cnt = off; off = up256(off + 4 * 4);
    W.gu = off; off = up256(off + 2 * pairs * ffn * 4);
    W.o = off; off = up256(off + pairs * hidden * 4);
    W.img = off; off = up256(off + W.max_tiles * std::max(gh * (hi_only ? gq::MmfwImage<1>::bytes : gq::MmfwImage<2>::bytes), gf * gq::MmfwImage<2>::bytes));
    W.inv = off; off = up256(off + std::max(gh, gf) * W.max_tiles * 128 + 1024);
    W.total = off;
    return W;
}

constexpr size_t kMoeMaxExperts = 4096; // of a call

// Few pairs an expert: the GEMM takes the call only where there is scratch for it (run_moe_wide).
bool moe_few_pairs(uint32_t dtype_gu, uint32_t dtype_dn, size_t experts, size_t pairs) { return pairs < (dtype_gu == T_Q8_0 || dtype_dn == T_Q8_0 ? 4u : 8u) * experts; }

// Whether the GEMM is ahead of jobs of eight tokens (of Q8_0, whose other form is the GEMV, of those).
// Without the element type: the two forms round differently, and a call of 16-bit elements gives the bits of the f32 call.  A call that has it
// ahead has it so with more pairs too (moe_wide_reserve).
bool moe_wide_ahead(const gllmq_ctx *ctx, uint32_t dtype_gu, uint32_t dtype_dn, size_t hidden, size_t ffn, size_t experts, size_t pairs)
{
    const bool q8 = dtype_gu == T_Q8_0 || dtype_dn == T_Q8_0;
    if (pairs < (q8 ? (ctx->moe_wide_min + 1) / 2 : ctx->moe_wide_min) * experts) return false;
    if ((dtype_gu == T_Q8_0 && hidden < 256) || (dtype_dn == T_Q8_0 && ffn < 256)) return false; // the Q8_0 window is a whole group
    if (ctx->moe_wide_cost) {
        // Few experts, or small ones, do not fill the device with one workgroup per 256 weight rows and all of K, which the
        // int8 kernels do; those take time with every pair.  Estimates in us of an f32 call, fitted to 410 drawn layers in both forms (8 to 128 experts of 1024
        // to 4096 x 512 to 2048, 1.2 to 14 pairs an expert; within 8 and 14 %).  GEMM: a block of K 0.3 (Q5_K 0.6, Q6_K 1.1, Q8_0 1.6), 2 more with every
        // CU busy and 0.6 for the second plane of gate and up, 4 for a workgroup's start and end, 22 for the launches beside the two.  The others: 31,
        // the weights at 12 TB/s (whose pairs' time holds the rest of theirs), the products at 59 TFLOP/s (Q5_K 54, Q8_0 18).  A tenth in favour of
        // the other form.  Below 8 pairs an expert (Q8_0: 4) calls of fewer than 32 pairs stay there (8 experts of 1024 x 512, 18 pairs: GEMM 31, jobs 27),
        // and K-quants whose gate and up fill the device twice (128 experts of 3584 x 512 Q5_K, 6 pairs an expert 223, 196; of 4096 x 1792 Q4_K, 4 pairs 604, 486);
        // from two thirds of the CUs on 15 % in favour of the other form (16 experts of 3840 x 2048 Q4_K, 72 pairs, GEMM 104.5, jobs 91.4).
        // By this 400 of 2303 other layers of that range with eight pairs (four) and more go to the GEMM that the estimate before left to the other form, f32
        // 30 % shorter in the mean, and 411 of 5082 with fewer, 24 %, seven of them slower by 2 to 6 %; of larger layers (to 384 experts,
        // 8192 and 14336) 74 of 865, 50 %, and 48 of 1017, 37 %, one slower by 1 %.  A call of 16-bit elements has more of the GEMM (one plane of gate and up; the jobs'
        // rows are converted) and follows the f32 call: by an estimate of its own bf16 calls were 5 % shorter in the mean, and not the f32 call's results rounded.
        const size_t cus_whole = static_cast<size_t>(ctx->num_cus), gu_wgs = (2 * ffn + 255) / 256 * std::min(experts, pairs);
        const bool few = moe_few_pairs(dtype_gu, dtype_dn, experts, pairs);
        if (few && (pairs < 32 || (!q8 && gu_wgs >= 2 * cus_whole))) return false;
        const double e = static_cast<double>(std::min(experts, pairs)), cus = ctx->num_cus;
        auto launch_us = [&](uint32_t dtype, size_t rows, size_t k, double planes) {
            const double wgs = std::ceil(rows / 256.0) * e;
            const double block = (dtype == T_Q8_0 ? 1.6 : dtype == T_Q6_K ? 1.1 : dtype == T_Q5_K ? 0.6 : 0.3) + 2.0 * std::min(1.0, wgs / cus) + planes;
            return std::ceil(wgs / cus) * (static_cast<double>((k + 255) / 256) * block + 4.0);
        };
        const double wide = 22.0 + launch_us(dtype_gu, 2 * ffn, hidden, 0.6) + launch_us(dtype_dn, hidden, ffn, 0.0);
        const double bytes = e * (2.0 * ffn * gllmq_row_bytes(dtype_gu, hidden) + static_cast<double>(hidden) * gllmq_row_bytes(dtype_dn, ffn));
        const double rate = q8 ? 18e6 : dtype_gu == T_Q5_K || dtype_dn == T_Q5_K ? 54e6 : 59e6;
        if ((few && !q8 && 3 * gu_wgs >= 2 * cus_whole ? 1.15 : 1.1) * wide > 31.0 + bytes / 12e6 + 6.0 * pairs * static_cast<double>(hidden) * ffn / rate) return false;
    }
    return true;
}

bool takes_moe_wide(const gllmq_ctx *ctx, uint32_t dtype_gu, uint32_t dtype_dn, const void *x, size_t hidden, size_t ffn, size_t experts, size_t pairs)
{
    if (!ctx->moe_wide || !ctx->use_mmf || !ctx->use_mmfw || ctx->moe_streamed == 2 || !moe_wide_ahead(ctx, dtype_gu, dtype_dn, hidden, ffn, experts, pairs)) return false;
    const size_t tiles = pairs / 32 + std::min(experts, pairs), groups = std::max((hidden + 255) / 256, (ffn + 255) / 256);
    return aligned(x, 16) && pairs * ffn <= 0xFFFFFFFFull && tiles * groups * gq::MmfwImage<2>::bytes <= 0xFFFFFFFFull;
}

// Scratch for any call of that many pairs or fewer: the GEMM takes the more the more experts, so that of the most, in any formats, which take it
// (`few`: with few pairs too).
size_t moe_wide_reserve(const gllmq_ctx *ctx, size_t pairs, size_t hidden, size_t ffn, bool few)
{
    for (size_t experts = std::min<size_t>(kMoeMaxExperts, pairs / ((ctx->moe_wide_min + 1) / 2)); experts > 0; --experts)
        for (const Format &gu : kFormats)
            for (const Format &dn : kFormats)
                if (moe_wide_ahead(ctx, gu.dtype, dn.dtype, hidden, ffn, experts, pairs) && (few || !moe_few_pairs(gu.dtype, dn.dtype, experts, pairs))) return plan_moe_wide(pairs, hidden, ffn, experts, false).total;
    return 0;
}

// Whether a launch over experts takes the workgroups of four waves (MMFW_EXPERTS_FEW); wgs: workgroups of eight waves it would have
// at one job an expert.  170 drawn layers (8 to 128 experts of 1024 to 4096 x 512 to 2048, 6 to 512 pairs an expert), change of the call by one
// launch's form: more than one workgroup a CU, up to 40 pairs an expert -2.1 % in the mean (128 experts of 4096 x 1536, top 8 of 256 tokens 496 us,
// 473; Q5_K of two planes -0.2 %, single ones +6; above 40 pairs, jobs of three tiles and more, -0.6 and +7).  At most half a workgroup a CU, where
// it fills the device: -2.9 % up to 40 pairs, with two planes -5.4 % up to 100 (8 experts of 4096 x 2048, 100 pairs each 160, 135), with one +1.9.
// Between them the eight waves have a CU to themselves either way: +0.3 %.  By this rule 115 of the 170 calls change, 4 % shorter in the mean.
// Uneven routing, by which single experts have jobs of four tiles in two passes: 3995 calls whose experts' logits are spread by 0.7 and 1.4, 2.7 to 5.4 % shorter in
// the mean by format, 13 longer by 5 to 7 %, nine of them Q8_0.
bool moe_wide_few(const gllmq_ctx *ctx, int fmt, int planes, size_t wgs, size_t pairs, size_t experts)
{
    if (ctx->moe_wide_few != 1) return ctx->moe_wide_few == 2;
    const size_t cus = ctx->num_cus;
    if (2 * wgs <= cus) return pairs <= (planes == 2 ? 100u : 40u) * experts;
    return wgs > cus && pairs <= 40 * experts && !(fmt == 1 && planes == 2);
}

// With few pairs an expert, of which the jobs take less scratch: kNoRoomForGemm, nothing enqueued, where that cannot be had (captured behind a
// smaller reservation, or refused).
constexpr int kNoRoomForGemm = -3;
int run_moe_wide(gllmq_ctx *ctx, const Format &fg, const void *gate, size_t gate_stride, const void *up, size_t up_stride, const Format &fd,
                 const void *down, size_t down_stride, const float *x, float *out, uint32_t elem, size_t tokens, size_t hidden, size_t ffn,
                 size_t experts, size_t top_k, const uint32_t *route_expert, const float *route_weight, const uint32_t *route_len,
                 int relu_gate, void *stream)
{
    const size_t pairs = tokens * top_k;
    const bool hi_only = elem != 0;
    const MoeWidePlan W = plan_moe_wide(pairs, hidden, ffn, experts, hi_only);
    Scratch *Sp = nullptr;
    int rc = acquire_scratch(ctx, stream, &Sp);
    if (rc != GLLMQ_OK) return rc;
    if (moe_few_pairs(fg.dtype, fd.dtype, experts, pairs)) {
        const size_t f32_total = plan_moe_wide(pairs, hidden, ffn, experts, false).total; // (a 16-bit call in the f32 call's form)
        grow_if_possible(ctx, *Sp, &Sp->moe, &Sp->moe_bytes, f32_total, stream);
        if (Sp->moe_bytes < f32_total) return kNoRoomForGemm;
    }
    rc = grow_scratch(ctx, *Sp, &Sp->moe, &Sp->moe_bytes, W.total, stream, "moe_matvec");
    if (rc != GLLMQ_OK) return rc;
    uint8_t *ws = static_cast<uint8_t *>(Sp->moe);
    uint32_t *token = reinterpret_cast<uint32_t *>(ws + W.token), *counters = reinterpret_cast<uint32_t *>(ws + W.cnt);
    float *gu = reinterpret_cast<float *>(ws + W.gu), *o = reinterpret_cast<float *>(ws + W.o);
    MoePlanParams plan{};
    plan.pair_src = reinterpret_cast<uint32_t *>(ws + W.src);
    plan.pair_pos = reinterpret_cast<uint32_t *>(ws + W.pos);
    plan.tiles = reinterpret_cast<gq::MoeTile *>(ws + W.tiles);
    plan.wide = reinterpret_cast<gq::MoeWideJob *>(ws + W.jobs);
    plan.token = token;
    plan.counters = counters;
    static_assert(32u * gq::MMFW_MAX_MT == 1u << 7, "rows of a job");
    plan.job_shift = 7u;
    rc = launch_moe_plan(ctx, plan, route_expert, route_len, tokens, top_k, experts, stream);
    if (rc != GLLMQ_OK) return rc;

    // the images of the tiles' rows, then every job's products with its expert's matrices
    auto multiply = [&](const Format &f, const MmfwMatrix *mats, const size_t *strides, int count, size_t k, bool hi, gq::MmfwPrepParams &Q) -> int {
        const int fmt = mmf_format(f.dtype);
        Q.ximg = ws + W.img;
        Q.inv = reinterpret_cast<float *>(ws + W.inv);
        Q.m = static_cast<uint32_t>(pairs);
        Q.k = static_cast<uint32_t>(k);
        Q.groups = static_cast<uint32_t>((k + 255) / 256);
        Q.inv_ld = W.max_tiles * 32u;
        Q.tiles = plan.tiles;
        Q.counters = counters;
        Q.natural = fmt == 2 ? 1u : 0u;
        int r = launch_mmfw_prep(ctx, Q, hi, W.max_tiles, stream);
        if (r != GLLMQ_OK) return r;
        gq::MmfwParams P{};
        P.ximg = Q.ximg;
        P.inv = Q.inv;
        P.segs = static_cast<uint32_t>(count);
        P.groups = Q.groups;
        P.row_bytes = static_cast<uint32_t>(gllmq_row_bytes(f.dtype, k));
        P.m = Q.m;
        P.k = Q.k;
        P.inv_ld = Q.inv_ld;
        P.ksplit = 1;
        P.blocks_per_split = Q.groups;
        P.jobs = plan.wide;
        P.counters = counters;
        size_t wgs = 0;
        for (int i = 0; i < count; ++i) wgs += (mats[i].n + gq::MMFW_TILE_ROWS - 1) / gq::MMFW_TILE_ROWS;
        const bool few = moe_wide_few(ctx, fmt, hi ? 1 : 2, wgs * std::min(experts, pairs), pairs, experts);
        const uint32_t waves = gq::mmfw_waves(few ? gq::MMFW_EXPERTS_FEW : gq::MMFW_EXPERTS), tile_rows = 32 * waves;
        for (int i = 0; i < count; ++i) {
            P.seg[i].w = mats[i].w;
            P.seg[i].y = mats[i].y;
            P.seg[i].n = static_cast<uint32_t>(mats[i].n);
            P.seg[i].tile0 = P.n_tiles;
            P.seg[i].expert_stride = strides[i];
            P.n_tiles += static_cast<uint32_t>((mats[i].n + tile_rows - 1) / tile_rows);
        }
        P.max_jobs = W.max_jobs;
        P.run_tiles = 1;
        P.n_runs = P.n_tiles;
        return launch(ctx, (few ? ctx->moe_mmf_few : ctx->moe_mmf)[fmt][hi ? 1 : 0], (W.max_jobs + 7u) / 8u * 8u * P.n_runs, waves * 64,
                      mmfw_grouped_lds(fmt, hi ? 1 : 2, few), stream, &P, sizeof P, true);
    };
    {
        gq::MmfwPrepParams Q{};
        Q.x = x;
        Q.ldx = static_cast<uint32_t>(hidden);
        Q.elem = elem;
        Q.row_of = token;
        const MmfwMatrix mats[2] = { { static_cast<const uint8_t *>(gate), gu, ffn }, { static_cast<const uint8_t *>(up), gu + pairs * ffn, ffn } };
        const size_t strides[2] = { gate_stride, up_stride };
        rc = multiply(fg, mats, strides, 2, hidden, hi_only, Q);
        if (rc != GLLMQ_OK) return rc;
    }
    {
        gq::MmfwPrepParams Q{};
        Q.x = gu;
        Q.ldx = static_cast<uint32_t>(ffn);
        Q.glu = relu_gate ? 2u : 1u;
        Q.glu_off = static_cast<uint32_t>(pairs * ffn);
        const MmfwMatrix mats[1] = { { static_cast<const uint8_t *>(down), o, hidden } };
        const size_t strides[1] = { down_stride };
        rc = multiply(fd, mats, strides, 1, ffn, false, Q);
        if (rc != GLLMQ_OK) return rc;
    }
    MoeCombineParams C{ o, route_weight, route_len, plan.pair_pos, out, static_cast<uint32_t>(tokens), static_cast<uint32_t>(top_k),
                        static_cast<uint32_t>(hidden), elem };
    return launch_moe_combine(ctx, C, stream);
}

// The expert matvec (call_mutex held).  x and out are of type `elem`; where the kernels of the shape take
// f32 only, kNeedPlainActivations comes back and nothing has been enqueued.
int moe_on_stream(gllmq_ctx *ctx, const void *gate, size_t gate_bytes, size_t gate_expert_stride, const void *up,
                  size_t up_bytes, size_t up_expert_stride, uint32_t dtype_gu, const void *down, size_t down_bytes,
                  size_t down_expert_stride, uint32_t dtype_dn, const float *x, float *out, uint32_t elem, size_t tokens,
                  size_t hidden, size_t ffn, size_t experts, size_t top_k, const uint32_t *route_expert,
                  const float *route_weight, const uint32_t *route_len, int relu_gate, void *stream)
{
    const Format *fg = find_format(dtype_gu), *fd = find_format(dtype_dn);
    if (!fg || !fd)
        return fail(ctx, GLLMQ_ERR_UNIMPLEMENTED,
                    "moe_matvec: ggml dtype %u / %u is not covered (supported: Q8_0=8, Q4_K=12, Q5_K=13, Q6_K=14)",
                    dtype_gu, dtype_dn);
    if (tokens == 0 || hidden == 0) return GLLMQ_OK;
    if (!gate || !up || !down || !x || !out || !route_expert || !route_weight || !route_len)
        return fail(ctx, GLLMQ_ERR_INVALID, "moe_matvec: NULL device pointer");
    if (ffn == 0 || experts == 0 || top_k == 0)
        return fail(ctx, GLLMQ_ERR_BAD_SHAPE, "moe_matvec: ffn, experts and top_k must be positive");
    const size_t pairs = tokens * top_k;
    // The plan kernel keeps the pair list and three words per expert in LDS, and a launch
    // covers at most 16384 elements of K.
    if (pairs > 16384 || experts > kMoeMaxExperts)
        return fail(ctx, GLLMQ_ERR_UNIMPLEMENTED,
                    "moe_matvec: tokens*top_k = %zu (max 16384) or experts = %zu (max 4096) is beyond this build", pairs,
                    experts);
    if (hidden > 16384 || ffn > 16384)
        return fail(ctx, GLLMQ_ERR_UNIMPLEMENTED, "moe_matvec: hidden = %zu / ffn = %zu beyond 16384 is not built",
                    hidden, ffn);
    if (hidden % 4 != 0 || ffn % 4 != 0)
        return fail(ctx, GLLMQ_ERR_BAD_SHAPE, "moe_matvec: hidden and ffn must be multiples of 4");
    const size_t rb_gu = gllmq_row_bytes(dtype_gu, hidden), rb_dn = gllmq_row_bytes(dtype_dn, ffn);
    // every expert's matrix must lie inside its buffer
    const size_t gu_each = ffn * rb_gu, dn_each = hidden * rb_dn;
    auto inside = [&](size_t bytes, size_t stride, size_t each) {
        return stride >= each && bytes >= each && (experts - 1) <= (bytes - each) / stride;
    };
    if (!inside(gate_bytes, gate_expert_stride, gu_each) || !inside(up_bytes, up_expert_stride, gu_each) ||
        !inside(down_bytes, down_expert_stride, dn_each))
        return fail(ctx, GLLMQ_ERR_BAD_SHAPE,
                    "moe_matvec: %zu experts of %zu (gate, up) / %zu (down) bytes at strides %zu / %zu / %zu do not fit buffers of "
                    "%zu / %zu / %zu bytes", experts, gu_each, dn_each, gate_expert_stride, up_expert_stride, down_expert_stride,
                    gate_bytes, up_bytes, down_bytes);
    if (!aligned(gate, fg->w_align) || !aligned(up, fg->w_align) || rb_gu % fg->w_align != 0 ||
        gate_expert_stride % fg->w_align != 0 || up_expert_stride % fg->w_align != 0 || !aligned(down, fd->w_align) ||
        rb_dn % fd->w_align != 0 || down_expert_stride % fd->w_align != 0)
        return fail(ctx, GLLMQ_ERR_BAD_ALIGNMENT, "moe_matvec: expert weights or strides miss the alignment of their format");
    if (!aligned(x, 16) || !aligned(out, 4))
        return fail(ctx, GLLMQ_ERR_BAD_ALIGNMENT, "moe_matvec: x must be 16-byte and out 4-byte aligned");

    int rc = kNoRoomForGemm;
    if (takes_moe_wide(ctx, dtype_gu, dtype_dn, x, hidden, ffn, experts, pairs))
        rc = run_moe_wide(ctx, *fg, gate, gate_expert_stride, up, up_expert_stride, *fd, down, down_expert_stride, x, out, elem, tokens,
                          hidden, ffn, experts, top_k, route_expert, route_weight, route_len, relu_gate, stream);
    if (rc != kNoRoomForGemm) return rc;
    if (elem) return kNeedPlainActivations;
    const MoeWorkspace W = moe_workspace(pairs, hidden, ffn);
    Scratch *Sp = nullptr;
    rc = acquire_scratch(ctx, stream, &Sp);
    if (rc != GLLMQ_OK) return rc;
    rc = grow_scratch(ctx, *Sp, &Sp->moe, &Sp->moe_bytes, W.total, stream, "moe_matvec");
    if (rc != GLLMQ_OK) return rc;
    uint8_t *ws = static_cast<uint8_t *>(Sp->moe);
    uint32_t *pair_src = reinterpret_cast<uint32_t *>(ws + W.src);
    uint32_t *pair_pos = reinterpret_cast<uint32_t *>(ws + W.pos);
    MoeJob *jobs = reinterpret_cast<MoeJob *>(ws + W.jobs);
    MoeJob8 *jobs8 = reinterpret_cast<MoeJob8 *>(ws + W.jobs8);
    uint32_t *counters = reinterpret_cast<uint32_t *>(ws + W.cnt);
    float *gu = reinterpret_cast<float *>(ws + W.gu);
    float *h = reinterpret_cast<float *>(ws + W.h);
    float *o = reinterpret_cast<float *>(ws + W.o);

    // The streamed grouped kernels take up to four tokens per job (their ring shares the LDS with the
    // tokens' digit planes), the others up to eight.  An expert with more tokens is read once per
    // job, so the streamed form is for calls whose experts see few tokens each (at most two on
    // average: decode batches); with more, jobs of eight read the weights half as often.
    const bool streamed_jobs = ctx->use_mm8s && (ctx->moe_streamed == 2 || (ctx->moe_streamed == 1 && pairs <= 2 * experts));
    const uint32_t job_shift = streamed_jobs ? 2u : 3u;
    {
        MoePlanParams P{};
        P.pair_src = pair_src;
        P.pair_pos = pair_pos;
        P.jobs = jobs;
        P.jobs8 = jobs8;
        P.counters = counters;
        P.job_shift = job_shift;
        rc = launch_moe_plan(ctx, P, route_expert, route_len, tokens, top_k, experts, stream);
        if (rc != GLLMQ_OK) return rc;
    }
    // Waves per job: the device takes about 8 waves per CU of these kernels; the jobs that
    // exist (at most `pairs`, typically one per routed expert) share them.
    const uint32_t job_waves = std::max<uint32_t>(16u, 4u * ctx->gemv_waves / static_cast<uint32_t>(pairs));
    // n rows of k elements per expert, experts `stride` bytes apart; the results of a pair go to
    // yout + its sorted position * y_stride.
    auto grouped = [&](const Format &f, const void *w, size_t stride, size_t rb, uint32_t n, uint32_t k, const float *xin,
                       bool x_by_token, float *yout, uint32_t y_stride) -> int {
        GemvPlan L = plan_gemv(ctx, 2, n, k, rb, job_waves);
        MoeGemvParams Q{};
        Q.g = L.P;
        Q.g.w = static_cast<const uint8_t *>(w);
        Q.g.x = xin;
        Q.g.y = yout;
        Q.g.x_vec = 1;
        Q.g.accumulate = 0;
        Q.jobs = jobs;
        Q.counters = counters;
        Q.expert_stride = stride;
        Q.wgs_per_job = L.grid;
        Q.x_by_token = x_by_token ? 1u : 0u;
        Q.x_stride = k;
        Q.y_stride = y_stride;
        const uint64_t grid = static_cast<uint64_t>(L.grid) * pairs;
        if (grid > 0x7FFFFFFFull) return fail(ctx, GLLMQ_ERR_BAD_SHAPE, "moe_matvec: launch grid too large");
        return launch(ctx, ctx->moe_gemv[format_index(f.dtype)], static_cast<uint32_t>(grid), L.threads, L.lds, stream,
                      &Q, sizeof Q);
    };
    // Q4_K, Q5_K and Q6_K with rows of at most 16 blocks go to the int8 matrix cores, every token
    // of an expert (up to eight per job) in one pass over its weights.  `by_token`: the activation
    // rows are x[token] (gate/up), else rows by sorted position (down).
    // `up_w` != null: the gated form, n gate rows per expert at `wbase` and n up rows at `up_w`,
    // and yout receives act(gate . x) * (up . x)
    auto grouped_mm8 = [&](const Format &f, const void *wbase, size_t stride, size_t rb, uint32_t n, uint32_t k,
                           const float *xin, bool by_token, float *yout, uint32_t y_stride, const void *up_w = nullptr,
                           size_t up_stride = 0) -> int {
        const bool glu = up_w != nullptr;
        const int kind = mm8_kind(f.dtype);
        const bool q6k = kind == MM8_Q6K;
        const uint32_t groups = (k + 255u) / 256u;
        MoeMm8Params Q{};
        Q.g.w = static_cast<const uint8_t *>(wbase);
        Q.g.x = xin;
        Q.g.y = yout;
        Q.g.n = n;
        Q.g.k = k;
        Q.g.groups = groups;
        Q.g.row_bytes = static_cast<uint32_t>(rb);
        Q.g.ldx = k;
        Q.g.tiles = (n + 31u) / 32u;
        Q.jobs = jobs8;
        Q.counters = counters;
        Q.expert_stride = stride;
        Q.up = static_cast<const uint8_t *>(up_w);
        Q.up_stride = up_stride;
        Q.y_stride = y_stride;
        Q.g.glu_relu = relu_gate ? 1u : 0u;
        Q.rows = by_token ? nullptr : ctx->identity_rows;
        // upper bound of the jobs: one per expert hit, plus one per eight (four) further pairs
        const uint64_t max_jobs = std::min<uint64_t>(pairs, experts + (pairs >> job_shift));
        uint32_t slices = std::max<uint32_t>(1u, (3u * static_cast<uint32_t>(ctx->num_cus)) / (2u * static_cast<uint32_t>(std::min<uint64_t>(pairs, experts))));
        if (ctx->moe_slices) slices = ctx->moe_slices;
        const uint32_t ppt = (groups + 7u) / 8u;
        hipFunction_t fn = glu ? ctx->moe_mm8_glu_fn[kind][ppt - 1] : ctx->moe_mm8_fn[kind][ppt - 1];
        uint32_t units = Q.g.tiles; // what the slices of a job share: tiles, or groups of eight tiles
        if (q6k && groups <= 8 && ctx->moe_mm8_rows) {
            fn = ctx->moe_mm8_q6k_rows;
            units = (Q.g.tiles + 7u) / 8u;
        }
        // The streamed form (loader waves and arithmetic waves, a workgroup per CU): the kernel cuts the
        // tiles of all jobs into one run per workgroup and works the ring out per job; it must exist for
        // two and for four rows over a run of any length.
        if (streamed_jobs && ctx->moe_mm8s_fn[kind][glu ? 1 : 0] && aligned(xin, 16) && max_jobs * Q.g.tiles < 0x7FFFFFFFull) {
            const uint32_t sfmt = kind == MM8_Q6K ? 2u : kind == MM8_Q5K ? 1u : 0u;
            const uint32_t pieces = sfmt == 2 ? gq::Mm8sFormat<2>::PIECES : sfmt == 1 ? gq::Mm8sFormat<1>::PIECES : gq::Mm8sFormat<0>::PIECES;
            const uint32_t subs = sfmt == 2 ? 0u : 8u, zeros = sfmt == 2 ? gq::Mm8sFormat<2>::ZEROS : 0u, item_bytes = 32u * pieces * 16u, lds_bytes = 160u * 1024u;
            const uint32_t items = (glu ? 2u : 1u) * Q.g.tiles * groups; // the longest piece: all tiles of a job
            gq::Mm8sLds L2, L4;
            uint32_t slots, depth;
            if (gq::mm8s_ring(groups, 2, item_bytes, items, subs, glu, zeros, lds_bytes, ctx->moe_depth, L2, slots, depth) &&
                gq::mm8s_ring(groups, 4, item_bytes, items, subs, glu, zeros, lds_bytes, ctx->moe_depth, L4, slots, depth)) {
                Q.slices = 1;
                Q.g.tile_rows = 32;
                Q.g.lds_ring = lds_bytes; // the kernel carves it up per job
                Q.g.depth = ctx->moe_depth;
                const uint64_t wgs = std::min<uint64_t>(static_cast<uint64_t>(ctx->num_cus), max_jobs * Q.g.tiles);
                return launch(ctx, ctx->moe_mm8s_fn[kind][glu ? 1 : 0], static_cast<uint32_t>(wgs),
                              (gq::MM8S_CWAVES + gq::MM8S_LOADERS) * 64, lds_bytes, stream, &Q, sizeof Q);
            }
        }
        slices = std::min(slices, units);
        Q.slices = slices;
        return launch(ctx, fn, static_cast<uint32_t>(max_jobs * slices), 512, mm8_lds_bytes(groups, 8, 4, kind), stream,
                      &Q, sizeof Q);
    };
    auto fits_mm8 = [&](const Format &f, size_t k, bool glu = false) {
        const uint32_t groups = static_cast<uint32_t>((k + 255) / 256);
        const int kind = mm8_kind(f.dtype);
        if (glu && !(ctx->moe_glu && (kind == MM8_Q4K || kind == MM8_Q5K))) return false;
        if (!(ctx->use_mm8 && ctx->moe_mm8) || kind < 0 || kind >= MM8_MOE_KINDS || groups > 16 || k % 8 != 0) return false;
        if (kind == MM8_Q6K && !ctx->moe_mm8_q6k) return false;
        return mm8_lds_bytes(groups, 8, 4, kind) <= 160u * 1024u;
    };
    const uint32_t F = static_cast<uint32_t>(ffn), H = static_cast<uint32_t>(hidden);
    const bool gated = fits_mm8(*fg, hidden, true); // gate, up and the activation in one launch
    if (gated) {
        rc = grouped_mm8(*fg, gate, gate_expert_stride, rb_gu, F, H, x, true, h, F, up, up_expert_stride);
    } else {
        // an expert's up rows right behind its gate rows, both under one stride: one matrix of
        // 2 * ffn rows; otherwise the two halves of gu[pair][2 ffn] come from a launch each
        const bool stacked = static_cast<const uint8_t *>(up) == static_cast<const uint8_t *>(gate) + gu_each &&
                             up_expert_stride == gate_expert_stride;
        const bool mm8 = fits_mm8(*fg, hidden);
        for (int half = 0; half < (stacked ? 1 : 2) && rc == GLLMQ_OK; ++half) {
            const void *wb = half ? up : gate;
            const size_t st = half ? up_expert_stride : gate_expert_stride;
            const uint32_t rows = stacked ? 2u * F : F;
            if (mm8) rc = grouped_mm8(*fg, wb, st, rb_gu, rows, H, x, true, gu + half * ffn, 2u * F);
            else rc = grouped(*fg, wb, st, rb_gu, rows, H, x, true, gu + half * ffn, 2u * F);
        }
    }
    if (rc != GLLMQ_OK) return rc;
    if (!gated) {
        MoeActParams P{ gu, h, counters, F, relu_gate ? 1u : 0u };
        rc = launch2d(ctx, ctx->moe_act, (F + 255u) / 256u, static_cast<uint32_t>(pairs), 256, 0, stream, &P, sizeof P);
        if (rc != GLLMQ_OK) return rc;
    }
    if (fits_mm8(*fd, ffn)) rc = grouped_mm8(*fd, down, down_expert_stride, rb_dn, H, F, h, false, o, H);
    else rc = grouped(*fd, down, down_expert_stride, rb_dn, H, F, h, false, o, H);
    if (rc != GLLMQ_OK) return rc;
    MoeCombineParams C{ o, route_weight, route_len, pair_pos, out, static_cast<uint32_t>(tokens),
                        static_cast<uint32_t>(top_k), H, 0 };
    return launch_moe_combine(ctx, C, stream);
}

} // namespace

int gllmq_moe_matvec(gllmq_ctx *ctx, const void *gate, size_t gate_bytes, size_t gate_expert_stride, const void *up,
                     size_t up_bytes, size_t up_expert_stride, uint32_t dtype_gu, const void *down, size_t down_bytes,
                     size_t down_expert_stride, uint32_t dtype_dn, const float *x, float *out, size_t tokens,
                     size_t hidden, size_t ffn, size_t experts, size_t top_k, const uint32_t *route_expert,
                     const float *route_weight, const uint32_t *route_len, int relu_gate, void *stream)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    return moe_on_stream(ctx, gate, gate_bytes, gate_expert_stride, up, up_bytes, up_expert_stride, dtype_gu, down, down_bytes,
                         down_expert_stride, dtype_dn, x, out, 0, tokens, hidden, ffn, experts, top_k, route_expert, route_weight, route_len,
                         relu_gate, stream);
}

int gq_quantized_matmul_on_block(gllmq_ctx *ctx, const void *w, size_t w_bytes, const float *x, float *y, uint32_t dtype,
                                 size_t m, size_t n, size_t k, void *block, size_t block_bytes, void *stream)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    if (!block || block_bytes < kScratchFixedBytes || !aligned(block, 256))
        return fail(ctx, GLLMQ_ERR_INVALID, "quantized_matmul: scratch block missing, misaligned or under %zu bytes", kScratchFixedBytes);
    static_assert(kScratchArriveBytes == GQ_BLOCK_ZEROED_BYTES, "the arrival counters are the zeroed head of the block");
    Scratch S;
    ctx->call_scratch = nullptr; // (the block is the caller's)
    S.stream = static_cast<hipStream_t>(stream);
    S.fixed = true;
    carve_fixed(S, block);
    S.mmf = static_cast<uint8_t *>(block) + kScratchFixedBytes;
    S.mmf_bytes = block_bytes - kScratchFixedBytes;
    return matmul_on_scratch(ctx, S, w, w_bytes, x, y, dtype, m, n, k, GLLMQ_ACT_F32_SPLIT, stream);
}

namespace {

// Device copy of a host weight slice, uploaded on first sight and kept (call_mutex held).  The key is
// the slice itself (address and length): the reference treats weights as immutable once loaded
// and keeps its uploaded blob by length alone (src/compat/hip_backend.rs:141-156).
int cached_weights(gllmq_ctx *ctx, const void *host, size_t bytes, void **dev)
{
    ++ctx->use_counter;
    for (CachedWeights &W : ctx->weights)
        if (W.host == host && W.bytes == bytes) {
            W.last_use = ctx->use_counter;
            *dev = W.dev;
            return GLLMQ_OK;
        }
    GLLMQ_HIP(ctx, hipSetDevice(ctx->device));
    // make room: least recently used first
    size_t held = 0;
    for (const CachedWeights &W : ctx->weights) held += W.bytes;
    while (!ctx->weights.empty() && held + bytes > ctx->weights_cache_limit) {
        size_t lru = 0;
        for (size_t i = 1; i < ctx->weights.size(); ++i)
            if (ctx->weights[i].last_use < ctx->weights[lru].last_use) lru = i;
        GLLMQ_HIP(ctx, hipDeviceSynchronize());
        (void)hipFree(ctx->weights[lru].dev);
        held -= ctx->weights[lru].bytes;
        ctx->weights.erase(ctx->weights.begin() + static_cast<long>(lru));
    }
    CachedWeights W;
    W.host = host;
    W.bytes = bytes;
    W.last_use = ctx->use_counter;
    GLLMQ_HIP(ctx, hipMalloc(&W.dev, bytes));
    hipError_t e = hipMemcpy(W.dev, host, bytes, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        (void)hipFree(W.dev);
        return fail(ctx, GLLMQ_ERR_HIP, "weight upload: %s", hipGetErrorString(e));
    }
    ++ctx->weight_uploads;
    ctx->weights.push_back(W);
    *dev = W.dev;
    return GLLMQ_OK;
}

} // namespace

void gllmq_weights_forget(gllmq_ctx *ctx, const void *host)
{
    if (!ctx) return;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    for (size_t i = 0; i < ctx->weights.size();) {
        if (host == nullptr || ctx->weights[i].host == host) {
            (void)hipDeviceSynchronize();
            (void)hipFree(ctx->weights[i].dev);
            ctx->weights.erase(ctx->weights.begin() + static_cast<long>(i));
        } else {
            ++i;
        }
    }
}

uint64_t gllmq_weight_uploads(const gllmq_ctx *ctx) { return ctx ? ctx->weight_uploads : 0; }

int gllmq_reserve_matmul(gllmq_ctx *ctx, uint32_t dtype, size_t m, size_t n, size_t k, void *stream)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    if (!find_format(dtype))
        return fail(ctx, GLLMQ_ERR_UNIMPLEMENTED, "reserve_matmul: ggml dtype %u is not covered", dtype);
    Scratch *S = nullptr;
    int rc = acquire_scratch(ctx, stream, &S);
    if (rc != GLLMQ_OK || m == 0 || n == 0 || k == 0) return rc;
    // the GEMM is the only matmul kernel family whose scratch depends on the shape; it may take
    // any call of 3 rows and more, and a batch's matrices over the same two
    if (m < 2) return GLLMQ_OK;
    // (any form of it: which one runs also depends on the activation pointer's alignment)
    size_t need = plan_mmf(ctx, m, n, k).need;
    if (ctx->use_mmf && ctx->use_mmfw) need = std::max(need, mmfw_reserve(ctx, m, k));
    const MmfsPlan Ls = plan_mmfs(ctx, *find_format(dtype), m, n, k);
    if (Ls.ok) need = std::max(need, Ls.need);
    if (const size_t decoded = mmfx_reserve(ctx, dtype, m, n, k)) grow_for_decoded(ctx, *S, std::max(need, decoded), stream); // (refused: calls go without)
    return grow_scratch(ctx, *S, &S->mmf, &S->mmf_bytes, need, stream, "reserve_matmul");
}

int gllmq_reserve_ffn(gllmq_ctx *ctx, uint32_t dtype_gate_up, uint32_t dtype_down, size_t m, size_t hidden, size_t ffn,
                      void *stream)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    int rc = gllmq_reserve_matmul(ctx, dtype_gate_up, m, 2 * ffn, hidden, stream);
    if (rc == GLLMQ_OK) rc = gllmq_reserve_matmul(ctx, dtype_down, m, hidden, ffn, stream);
    if (rc != GLLMQ_OK || m == 0 || hidden == 0 || ffn == 0) return rc;
    Scratch *S = nullptr;
    rc = acquire_scratch(ctx, stream, &S);
    if (rc != GLLMQ_OK) return rc;
    return grow_scratch(ctx, *S, &S->ffn, &S->ffn_bytes, ffn_scratch_bytes(m, ffn), stream, "reserve_ffn");
}

int gllmq_reserve_moe(gllmq_ctx *ctx, size_t tokens, size_t top_k, size_t hidden, size_t ffn, void *stream)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    Scratch *S = nullptr;
    int rc = acquire_scratch(ctx, stream, &S);
    if (rc != GLLMQ_OK || tokens == 0 || top_k == 0) return rc;
    const size_t pairs = tokens * top_k;
    grow_if_possible(ctx, *S, &S->moe, &S->moe_bytes, moe_wide_reserve(ctx, pairs, hidden, ffn, true), stream); // (refused: those calls go without)
    const size_t need = std::max(moe_workspace(pairs, hidden, ffn).total, moe_wide_reserve(ctx, pairs, hidden, ffn, false));
    return grow_scratch(ctx, *S, &S->moe, &S->moe_bytes, need, stream, "reserve_moe");
}

int gllmq_dequantize_host(gllmq_ctx *ctx, const void *blocks, size_t n_bytes, float *out, size_t n_out,
                          uint32_t dtype)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    const Format *f = find_format(dtype);
    if (!f) return gllmq_dequantize(ctx, blocks, n_bytes, out, n_out, dtype, nullptr);
    const size_t nb = std::min(n_bytes / f->block_bytes, n_out / f->block_size);
    if (nb == 0) return GLLMQ_OK;
    void *d_in = nullptr, *d_out = nullptr;
    int rc = cached_weights(ctx, blocks, nb * f->block_bytes, &d_in);
    if (rc != GLLMQ_OK) return rc;
    hipError_t e = hipMalloc(&d_out, nb * f->block_size * sizeof(float));
    if (e != hipSuccess) rc = fail(ctx, GLLMQ_ERR_HIP, "hipMalloc: %s", hipGetErrorString(e));
    if (rc == GLLMQ_OK)
        rc = gllmq_dequantize(ctx, d_in, nb * f->block_bytes, static_cast<float *>(d_out), nb * f->block_size,
                              dtype, nullptr);
    if (rc == GLLMQ_OK &&
        (e = hipMemcpy(out, d_out, nb * f->block_size * sizeof(float), hipMemcpyDeviceToHost)) != hipSuccess)
        rc = fail(ctx, GLLMQ_ERR_HIP, "hipMemcpy D2H: %s", hipGetErrorString(e));
    (void)hipFree(d_out);
    return rc;
}

int gllmq_quant_gather_host(gllmq_ctx *ctx, const void *table, size_t table_bytes, uint32_t dtype, size_t vocab,
                            size_t hidden, const uint32_t *ids, size_t count, float scale, float *out)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    const Format *f = find_format(dtype);
    if (!f || count == 0 || hidden == 0 || !table || !ids || !out || hidden % 4 != 0 ||
        table_bytes < vocab * gllmq_row_bytes(dtype, hidden)) // the device entry point reports these
        return gllmq_quant_gather(ctx, table, table_bytes, dtype, vocab, hidden, ids, count, scale, out, nullptr);
    for (size_t i = 0; i < count; ++i)
        if (ids[i] >= vocab)
            return fail(ctx, GLLMQ_ERR_BAD_SHAPE, "quant_gather: id %u at position %zu is outside the %zu-row table",
                        ids[i], i, vocab);
    const size_t tb = vocab * gllmq_row_bytes(dtype, hidden);
    void *d_t = nullptr, *d_i = nullptr, *d_o = nullptr;
    int rc = cached_weights(ctx, table, tb, &d_t);
    if (rc != GLLMQ_OK) return rc;
    hipError_t e = hipMalloc(&d_i, count * sizeof(uint32_t));
    if (e == hipSuccess) e = hipMalloc(&d_o, count * hidden * sizeof(float));
    if (e == hipSuccess) e = hipMemcpy(d_i, ids, count * sizeof(uint32_t), hipMemcpyHostToDevice);
    rc = e == hipSuccess ? GLLMQ_OK : fail(ctx, GLLMQ_ERR_HIP, "quant_gather: %s", hipGetErrorString(e));
    if (rc == GLLMQ_OK)
        rc = gllmq_quant_gather(ctx, d_t, tb, dtype, vocab, hidden, static_cast<const uint32_t *>(d_i), count, scale,
                                static_cast<float *>(d_o), nullptr);
    if (rc == GLLMQ_OK && (e = hipMemcpy(out, d_o, count * hidden * sizeof(float), hipMemcpyDeviceToHost)) != hipSuccess)
        rc = fail(ctx, GLLMQ_ERR_HIP, "hipMemcpy D2H: %s", hipGetErrorString(e));
    (void)hipFree(d_i);
    (void)hipFree(d_o);
    return rc;
}

int gllmq_quantized_matmul_host(gllmq_ctx *ctx, const void *w, size_t w_bytes, const float *x, float *y,
                                uint32_t dtype, size_t m, size_t n, size_t k)
{
    if (!ctx) return GLLMQ_ERR_INVALID;
    std::lock_guard<std::recursive_mutex> call(ctx->call_mutex);
    const Format *f = find_format(dtype);
    if (!f) return gllmq_quantized_matmul(ctx, w, w_bytes, x, y, dtype, m, n, k, nullptr);
    if (m == 0 || n == 0) return GLLMQ_OK;
    if (!w || !x || !y) return fail(ctx, GLLMQ_ERR_INVALID, "quantized_matmul: NULL pointer");
    const size_t need = n * gllmq_row_bytes(dtype, k);
    if (w_bytes < need)
        return fail(ctx, GLLMQ_ERR_BAD_SHAPE, "quantized_matmul: weight buffer has %zu bytes, need %zu", w_bytes, need);
    void *d_w = nullptr, *d_x = nullptr, *d_y = nullptr;
    int rc = cached_weights(ctx, w, need, &d_w);
    if (rc != GLLMQ_OK) return rc;
    hipError_t e;
    if ((e = hipMalloc(&d_x, m * k * sizeof(float))) != hipSuccess || (e = hipMalloc(&d_y, m * n * sizeof(float))) != hipSuccess)
        rc = fail(ctx, GLLMQ_ERR_HIP, "hipMalloc: %s", hipGetErrorString(e));
    if (rc == GLLMQ_OK && (e = hipMemcpy(d_x, x, m * k * sizeof(float), hipMemcpyHostToDevice)) != hipSuccess)
        rc = fail(ctx, GLLMQ_ERR_HIP, "hipMemcpy H2D: %s", hipGetErrorString(e));
    if (rc == GLLMQ_OK)
        rc = gllmq_quantized_matmul(ctx, d_w, need, static_cast<const float *>(d_x), static_cast<float *>(d_y),
                                    dtype, m, n, k, nullptr);
    if (rc == GLLMQ_OK && (e = hipMemcpy(y, d_y, m * n * sizeof(float), hipMemcpyDeviceToHost)) != hipSuccess)
        rc = fail(ctx, GLLMQ_ERR_HIP, "hipMemcpy D2H: %s", hipGetErrorString(e));
    (void)hipFree(d_x);
    (void)hipFree(d_y);
    return rc;
}

} // extern "C"
