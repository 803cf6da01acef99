// Chunks above the 512-token slab: one MoE layer over up to 32,768 tokens
// in a single pass, so that every active expert's weights are streamed once
// per 128 routed rows instead of once per 16.  The reference prefills in
// slabs of at most 512 tokens (include/q38/cuda_moe_prefill.h:14, the V1
// plan); this path keeps the V1 plan's packed order (expert-major, stable
// in route index, q38_moe_prefill.cu:192-262) and per-route arithmetic, so
// every route's weighted_mid and route_output row and every token's output
// are bit-identical to the slab path's, and changes only the task height
// (128 rows) and how the plan is built (three launches instead of one
// workgroup).
//
// Plan: (1) per-chunk expert histograms, (2) one workgroup scans them into
// expert offsets, per-chunk bases and 128-row tasks, (3) one wave per chunk
// assigns stable positions with an LDS table of equal-id lane masks.
//
// Weights are read with ordinary (cached) loads, unlike the slab kernels'
// non-temporal streams: a hot expert's 128-row tasks run side by side and
// share its weights through L2.
//
// GEMMs: W4 in groups of 32 runs the int8 contract on fp16 MFMA, every other
// grouped format on 32x32 int8 MFMA, W8 per-channel down on 16x16 int8 MFMA,
// all with up to 128 rows of a task per weight fragment.
#include "q38m_device.h"
#include "q38m_internal.h"
#include "q38m_select.h"

namespace q38m {
namespace {

constexpr uint32_t kWideRows = Q38M_WIDE_TASK_ROWS;
constexpr uint32_t kRowTiles = kWideRows / 16u;
constexpr uint32_t kCountSlots = kExperts + 1u;  // slot 512 counts invalid ids

// The contract's SwiGLU gate, silu(g) = g / (1 + exp(-g)), for every bf16 g:
// entry h holds the fp32 word of silu(bits h << 16).  The gate enters SwiGLU
// rounded to bf16 (q38_moe_prefill.cu:449-461), so silu depends on g's 16
// bits only; the table is written at build time by q38m_silu_gen.c (the
// contract's exp and one IEEE division, equal to swiglu_fold's evaluation
// for every g), and one gather replaces ~40 VALU instructions per element
// in the compute-bound gate/up epilogue.  256 KiB, read through L2.
__device__ const uint32_t kSiluTable[65536] = {
#include "q38m_silu_table.inc"
};

// ---- plan -------------------------------------------------------------------

template <uint32_t kChunkRoutes>
__global__ __launch_bounds__(256) void wide_count_kernel(const int32_t* __restrict__ ids,
                                                         uint32_t routes,
                                                         uint32_t* __restrict__ chunk_counts) {
    __shared__ uint32_t hist[kCountSlots];
    for (uint32_t i = threadIdx.x; i < kCountSlots; i += 256u) hist[i] = 0u;
    __syncthreads();
    const uint32_t begin = blockIdx.x * kChunkRoutes;
    const uint32_t end = min(begin + kChunkRoutes, routes);
    for (uint32_t a = begin + threadIdx.x; a < end; a += 256u) {
        const int32_t id = ids[a];
        const bool valid = id >= 0 && id < static_cast<int32_t>(kExperts);
        atomicAdd(&hist[valid ? static_cast<uint32_t>(id) : kExperts], 1u);
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < kCountSlots; i += 256u)
        chunk_counts[static_cast<size_t>(blockIdx.x) * kCountSlots + i] = hist[i];
}

// One workgroup of 512 threads, thread e = expert e.  Turns the per-chunk
// counts into per-chunk bases within each expert's segment (in place) and
// writes the plan's counts, offsets, task offsets, tasks and header.
constexpr uint32_t kMaxChunks = (Q38M_WIDE_MAX_TOKENS * kTopK + kWideChunkRoutes - 1u) /
                                kWideChunkRoutes;

__global__ __launch_bounds__(512) void wide_scan_kernel(uint32_t* __restrict__ chunk_counts,
                                                        uint32_t chunks, uint32_t tokens,
                                                        q38m_route_plan_v1 plan,
                                                        uint32_t max_tasks) {
    __shared__ uint32_t wave_totals[2][8];
    __shared__ uint32_t wave_active[8];
    __shared__ uint32_t offsets[kExperts + 1u];
    __shared__ uint32_t task_offsets[kExperts + 1u];
    __shared__ uint32_t invalid;
    const uint32_t e = threadIdx.x;
    const uint32_t tid = e;
    const uint32_t lane = e & 63u;
    const uint32_t wave = e >> 6;
    const uint32_t routes = tokens * kTopK;

    // 1. running count of expert e over the chunks, in chunk order; each
    // chunk's slot becomes the expert's count in the chunks before it.
    // Batches of 32 chunks, the next batch's loads issued before this
    // batch's sums (two batches in flight), unconditionally (a chunk past
    // the last re-reads the last one and adds nothing), so no branch sits
    // between a load and the wait for it.  (One batch at a time: ~9.5 us at
    // 160 chunks, a round trip each.)
    constexpr uint32_t kBatch = 32;
    auto load_batch = [&](uint32_t c0, uint32_t (&v)[kBatch]) {
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j)
            v[j] = chunk_counts[static_cast<size_t>(min(c0 + j, chunks - 1u)) * kCountSlots + e];
    };
    uint32_t count = 0;
    uint32_t va[kBatch], vb[kBatch];
    load_batch(0u, va);
    for (uint32_t c0 = 0; c0 < chunks; c0 += 2u * kBatch) {
        load_batch(c0 + kBatch, vb);
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) {
            const bool live = c0 + j < chunks;
            if (live) chunk_counts[static_cast<size_t>(c0 + j) * kCountSlots + e] = count;
            count += live ? va[j] : 0u;
        }
        if (c0 + kBatch >= chunks) break;  // uniform
        load_batch(c0 + 2u * kBatch, va);
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) {
            const bool live = c0 + kBatch + j < chunks;
            if (live) chunk_counts[static_cast<size_t>(c0 + kBatch + j) * kCountSlots + e] = count;
            count += live ? vb[j] : 0u;
        }
    }
    // invalid ids: wave 0 sums slot 512 of every chunk (at most 160, three
    // unconditional loads per lane, one round trip)
    static_assert(kMaxChunks <= 192u, "three invalid-slot loads per lane");
    if (wave == 0u) {
        uint32_t bad[3];
#pragma unroll
        for (uint32_t j = 0; j < 3u; ++j)
            bad[j] = chunk_counts[static_cast<size_t>(min(lane + 64u * j, chunks - 1u)) *
                                      kCountSlots + kExperts];
        uint32_t sum = 0;
#pragma unroll
        for (uint32_t j = 0; j < 3u; ++j) sum += lane + 64u * j < chunks ? bad[j] : 0u;
        sum = wave_inclusive_sum(sum);
        if (lane == 63u) invalid = sum;
    }
    const uint32_t tasks = (count + kWideRows - 1u) / kWideRows;

    // 2. exclusive scans of counts and task counts over experts
    {
        plan.expert_counts[e] = static_cast<uint16_t>(count);
        const uint32_t inc_count = wave_inclusive_sum(count);
        const uint32_t inc_tasks = wave_inclusive_sum(tasks);
        const uint64_t active = __ballot(count != 0u);
        if (lane == 63u) {
            wave_totals[0][wave] = inc_count;
            wave_totals[1][wave] = inc_tasks;
        }
        if (lane == 0u) wave_active[wave] = __popcll(active);
        // inclusive values kept for after the barrier
        offsets[e] = inc_count;
        task_offsets[e] = inc_tasks;
    }
    __syncthreads();
    {
        uint32_t prefix_count = 0, prefix_tasks = 0;
#pragma unroll
        for (uint32_t w = 0; w < 8u; ++w) {
            prefix_count += w < wave ? wave_totals[0][w] : 0u;
            prefix_tasks += w < wave ? wave_totals[1][w] : 0u;
        }
        const uint32_t offset = prefix_count + offsets[e] - count;
        const uint32_t task_offset = prefix_tasks + task_offsets[e] - tasks;
        plan.expert_offsets[e] = offset;
        plan.expert_task_offsets[e] = task_offset;
        if (e == kExperts - 1u) {
            plan.expert_offsets[kExperts] = prefix_count + offsets[e];
            plan.expert_task_offsets[kExperts] = prefix_tasks + task_offsets[e];
        }
        // every read of offsets[] above precedes the writes below (one
        // thread reads and writes only its own slot)
        offsets[e] = offset;
        task_offsets[e] = task_offset;
        if (e == kExperts - 1u) {
            offsets[kExperts] = offset + count;
            task_offsets[kExperts] = task_offset + tasks;
        }
    }
    __syncthreads();
    const uint32_t total = offsets[kExperts];
    const uint32_t task_total = task_offsets[kExperts];

    // 3. tasks: 128-row tiles of each expert's segment, zero past the count.
    // Spread over the threads (a Zipf-hot expert has hundreds of tasks, and
    // one thread per expert took ~12 us at 32,768 tokens): task t's expert
    // is the last e with task_offsets[e] <= t, by binary search in LDS.
    uint2* task_words = reinterpret_cast<uint2*>(plan.tasks);
    for (uint32_t t = tid; t < max_tasks; t += 512u) {
        uint2 word = make_uint2(0u, 0u);
        if (t < task_total) {
            uint32_t lo = 0u, hi = kExperts - 1u;  // task_offsets[lo] <= t < task_offsets[lo + 1]
            while (lo < hi) {
                const uint32_t mid = (lo + hi + 1u) >> 1;
                if (task_offsets[mid] <= t) lo = mid; else hi = mid - 1u;
            }
            const uint32_t tile = t - task_offsets[lo];
            const uint32_t remaining = (offsets[lo + 1u] - offsets[lo]) - tile * kWideRows;
            const uint32_t rows = remaining < kWideRows ? remaining : kWideRows;
            word = make_uint2(offsets[lo] + tile * kWideRows, lo | (rows << 16));
        }
        task_words[t] = word;
    }
    // packed positions no valid route fills hold their own index
    for (uint32_t p = total + tid; p < routes; p += 512u) plan.packed_assignment[p] = p;

    if (tid == 0u) {
        uint32_t active_experts = 0;
        for (uint32_t w = 0; w < 8u; ++w) active_experts += wave_active[w];
        uint32_t status = Q38M_PLAN_OK;
        if (invalid != 0u)
            status = Q38M_PLAN_INVALID_EXPERT;
        else if (total != routes || task_total > max_tasks)
            status = Q38M_PLAN_INVALID_SHAPE;
        q38m_route_plan_header_v1* h = plan.header;
        h->magic = Q38M_ROUTE_PLAN_MAGIC_V1;
        h->version = Q38M_ROUTE_PLAN_VERSION_WIDE;
        h->tokens = tokens;
        h->routes = routes;
        h->active_experts = active_experts;
        h->task_count = task_total;
        h->status = status;
        h->flags = 0u;
        h->route_hash = 0u;
        h->plan_hash = 0u;
        h->reserved0 = 0u;
        h->reserved1 = 0u;
    }
}

// One wave per chunk walks its routes 64 at a time in route order, from
// the expert offsets plus the chunk's bases within each segment.  Lanes
// with equal ids find each other through an LDS table of lane masks (each
// lane ORs its bit into its id's slot, reads the slot back, clears it; one
// wave's LDS operations execute in order); the stable position is the
// chunk's running base for the id plus the equal lanes below.
template <uint32_t kChunkRoutes>
__global__ __launch_bounds__(64) void wide_scatter_kernel(const int32_t* __restrict__ ids,
                                                          uint32_t routes,
                                                          const uint32_t* __restrict__ bases,
                                                          q38m_route_plan_v1 plan) {
    __shared__ uint32_t running[kExperts];
    __shared__ unsigned long long table[kCountSlots];
    const uint32_t lane = threadIdx.x;
    const uint32_t* base = bases + static_cast<size_t>(blockIdx.x) * kCountSlots;
    const uint32_t begin = blockIdx.x * kChunkRoutes;
    const uint32_t end = min(begin + kChunkRoutes, routes);
    // every load of the chunk is issued before the first use: the segment
    // bases and the chunk's ids (clamped to its last route, unused past it)
    constexpr uint32_t kPerLane = kExperts / 64u, kSteps = kChunkRoutes / 64u;
    static_assert(kExperts % 64u == 0u && kChunkRoutes % 64u == 0u, "whole waves");
    uint32_t offset[kPerLane], chunk_base[kPerLane];
    int32_t idv[kSteps];
#pragma unroll
    for (uint32_t k = 0; k < kPerLane; ++k) {
        offset[k] = plan.expert_offsets[lane + 64u * k];
        chunk_base[k] = base[lane + 64u * k];
    }
#pragma unroll
    for (uint32_t j = 0; j < kSteps; ++j) idv[j] = ids[min(begin + 64u * j + lane, end - 1u)];
#pragma unroll
    for (uint32_t k = 0; k < kPerLane; ++k) running[lane + 64u * k] = offset[k] + chunk_base[k];
    for (uint32_t i = lane; i < kCountSlots; i += 64u) table[i] = 0ull;
    __syncthreads();
    const uint64_t below_mask = (1ull << lane) - 1ull;
#pragma unroll
    for (uint32_t j = 0; j < kSteps; ++j) {
        const uint32_t a = begin + 64u * j + lane;
        if (begin + 64u * j >= end) break;  // uniform
        const bool in = a < end;
        const int32_t id = in ? idv[j] : -1;
        const bool valid = in && id >= 0 && id < static_cast<int32_t>(kExperts);
        const uint32_t slot = valid ? static_cast<uint32_t>(id) : kExperts;
        atomicOr(&table[slot], 1ull << lane);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const unsigned long long equal = table[slot];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        table[slot] = 0ull;
        const uint32_t below = __popcll(equal & below_mask);
        const uint32_t run = valid ? running[valid ? slot : 0u] : 0u;
        if (valid && below == 0u) running[slot] = run + __popcll(equal);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (valid) {
            const uint32_t position = run + below;
            plan.packed_assignment[position] = a;
            plan.assignment_to_packed[a] = position;
        } else if (in) {
            plan.assignment_to_packed[a] = a;
        }
    }
}

// ---- workgroup placement -----------------------------------------------------

// The grouped GEMMs below run on one-dimensional grids of (task, slice)
// pairs, `slices` slices of the output channels per task slot.  The
// dispatcher hands workgroups to the 8 XCDs round-robin by id, and each XCD
// has its own L2; a task's slices next to each other on one XCD read the
// same rows, and an expert's neighbouring tasks the same weights, from one
// L2.  Two maps:
// - up to kBlockedSlots task slots, and in every wide_i8_kernel, XCD x gets the
//   blocks of kTaskBlock consecutive tasks x, x + 8, x + 16, ...  The map needs
//   no word of the plan, so a workgroup's first read is its task record;
//   slots past the plan's tasks hold zero records.
// - above, the kernels of groups of 32 and of W8 per-channel down give each
//   XCD a contiguous eighth of the plan's tasks.
// Contiguous eighths differ by 10-30 % in rows for 1,500 to 6,000 tokens, blocks
// by less, but where the hot experts lie decides a single call: of eight
// orders of popularity each gained or lost up to 10 %.  Means over them, step
// in us as eighths / blocks, W4/W8: Zipf 0.8, 600 tokens 226 / 230, 1,500 348 / 338,
// 2,500 465 / 448, 4,096 610 / 608, 8,192 982 / 958, 16,384 1,688 / 1,669; Zipf 1.1,
// 1,500 273 / 269, 4,096 507 / 510, 8,192 872 / 864.  32,768 tokens (four orders):
// uniform 3,024 / 3,087, Zipf 0.8 3,081 / 3,088, W4 in both 3,353 / 3,338: the
// second map is kept for the first of these.  wide_i8_kernel at 32,768
// tokens, W4 groups of 128, 2.73 / 2.67 ms.
struct Placement {
    uint32_t task, slice;
};

constexpr uint32_t kXcds = 8;
constexpr uint32_t kTaskBlock = 4;
constexpr uint32_t kBlockedSlots = 2048;

// the task slots a launch covers
struct TaskSlots {
    const q38m_task_v1* tasks;
    const uint32_t* live;  // the plan's task count for contiguous eighths, null for blocks
    uint32_t count;
};

__host__ __device__ constexpr uint32_t placed_workgroups(uint32_t task_slots, uint32_t slices) {
    constexpr uint32_t kRound = kXcds * kTaskBlock;
    return (task_slots + kRound - 1u) / kRound * kRound * slices;
}

__device__ inline bool place_on_xcds(const TaskSlots& t, uint32_t slices, Placement& at) {
    const uint32_t xcd = blockIdx.x % kXcds, j = blockIdx.x / kXcds;
    if (t.live != nullptr) {
        const uint32_t pairs = min(*t.live, t.count) * slices;
        const uint32_t per = pairs / kXcds, extra = pairs % kXcds;
        if (j >= per + (xcd < extra ? 1u : 0u)) return false;
        const uint32_t pair = xcd * per + min(xcd, extra) + j;
        at.task = pair / slices;
        at.slice = pair % slices;
        return true;
    }
    const uint32_t within = j % (kTaskBlock * slices);
    at.task = (j / (kTaskBlock * slices) * kXcds + xcd) * kTaskBlock + within / slices;
    at.slice = within % slices;
    return at.task < t.count;
}

// ---- gate/up ----------------------------------------------------------------

// ---- gate/up, W4 groups of 32, on fp16 MFMA --------------------------------
//
// The int8 values of both operands (activations in [-127, 127], W4 nibbles
// as 16 * w in [-128, 112]) are exact in fp16, their products (< 2^14) and
// every partial sum of a 32-wide group (< 2^19) exact in fp32, so
// v_mfma_f32_16x16x32_f16 returns (float)(16 * acc_g) itself -- the value
// an int8 MFMA path recovers with one extra VALU op per accumulator element
// and group.  The chain step is then a single v_fma_f32, and the MFMA runs
// at the same 16 cycles as v_mfma_i32_16x16x32_i8.
//
// fp16 images.  Weights (MFMA16 W4 word: byte i = k_i | k_{4+i} << 4): a
// nibble u' = w + 8 (offset binary: the nibble's top bit inverted) placed
// under the exponent bits of 1024 (0x6400) is the fp16 1024 + 16 u' (nibble
// in bits 4-7) or 1024 + u' (bits 0-3), exact; one v_pk_add_f16 of -1152 or
// -1032 leaves 16 w or w.  One v_bitop3_b32 forms two such values from a
// word (or the word shifted right by 8): per bit, field bits pass (sign bit
// inverted), exponent bits are set, the rest cleared.  A lane's eight K
// values come out as (4, 6) and (5, 7) times 16, (0, 2) and (1, 3) times 1;
// the activations are staged in the same K order with the (0, 2), (1, 3)
// pairs times 16 (one v_cvt_f16_i16 per sign-extended byte, one v_pk_mul_f16
// per pair), so every product is 16 a w, as on the int8 path.  A dot
// product does not depend on the order of its K terms, only on A and B
// agreeing; every value and product here is an integer below 2^14.
__device__ __forceinline__ uint32_t pk_add_f16(uint32_t v, float c) {
    typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
    const _Float16 h = static_cast<_Float16>(c);
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2_t, v) + h2_t{h, h});
}
__device__ __forceinline__ uint32_t pk_times16_f16(uint32_t v) {
    typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
    const _Float16 h = static_cast<_Float16>(16.0f);
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2_t, v) * h2_t{h, h});
}

// one MFMA16 W4 word -> fp16 K order (4, 6)x16, (5, 7)x16, (0, 2), (1, 3)
__device__ __forceinline__ uint4 w4_to_f16x16(uint32_t d) {
    // bitop3 truth table (index = S0*4 + S1*2 + S2): out = S0 where S1 & !S2,
    // !S0 where S1 & S2, 1 where !S1 & S2, 0 elsewhere
    constexpr uint32_t kTable = 0x6A;
    constexpr uint32_t kHiField = 0x00F000F0u, kHiConst = 0x64806480u;
    constexpr uint32_t kLoField = 0x000F000Fu, kLoConst = 0x64086408u;
    const uint32_t t = d >> 8;
    return make_uint4(
        pk_add_f16(__builtin_amdgcn_bitop3_b32(d, kHiField, kHiConst, kTable), -1152.0f),
        pk_add_f16(__builtin_amdgcn_bitop3_b32(t, kHiField, kHiConst, kTable), -1152.0f),
        pk_add_f16(__builtin_amdgcn_bitop3_b32(d, kLoField, kLoConst, kTable), -1032.0f),
        pk_add_f16(__builtin_amdgcn_bitop3_b32(t, kLoField, kLoConst, kTable), -1032.0f));
}

// bytes 0 and 2 (or 1 and 3) of v as signed integers -> two fp16 (exact):
// v_cvt_f16_i16 with a sign-extended byte source selected by SDWA, the
// second conversion writing the high half and keeping the low one
__device__ __forceinline__ uint32_t sbytes02_to_f16(uint32_t v) {
    uint32_t r;
    asm("v_cvt_f16_i16_sdwa %0, sext(%1) dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:BYTE_0\n\t"
        "v_cvt_f16_i16_sdwa %0, sext(%1) dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:BYTE_2"
        : "=&v"(r)
        : "v"(v));
    return r;
}
__device__ __forceinline__ uint32_t sbytes13_to_f16(uint32_t v) {
    uint32_t r;
    asm("v_cvt_f16_i16_sdwa %0, sext(%1) dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:BYTE_1\n\t"
        "v_cvt_f16_i16_sdwa %0, sext(%1) dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:BYTE_3"
        : "=&v"(r)
        : "v"(v));
    return r;
}

// eight int8 (k 0-3 in lo, 4-7 in hi) -> fp16 in the order and scaling of
// w4_to_f16x16's partners: (4, 6), (5, 7), 16 (0, 2), 16 (1, 3)
__device__ __forceinline__ uint4 i8_to_f16(uint32_t lo, uint32_t hi) {
    return make_uint4(sbytes02_to_f16(hi), sbytes13_to_f16(hi),
                      pk_times16_f16(sbytes02_to_f16(lo)), pk_times16_f16(sbytes13_to_f16(lo)));
}

// Staging swizzle of the fp16 A image: in fragment (group j, row tile t)
// the slot of row r (0..15) in 16-byte chunk c (0..3) is c*16 + (r ^ f(s)),
// s = (c >> 1) + 2j, f = {0, 6, 10, 12}.  A staging store instruction writes
// four rows x the four chunk pairs of a 64-column step: unswizzled, its
// eight- and sixteen-lane groups land on two and four bank groups (2- and
// 4-way conflicts); with f every group hits distinct banks, and the MFMA
// reads (one chunk, sixteen rows) stay conflict-free.
__device__ __forceinline__ uint32_t a_swizzle(uint32_t s) { return (0xCA60u >> (4u * s)) & 15u; }

__device__ __forceinline__ v4f mfma_f16_16x16x32(uint4 a, uint4 b, v4f c) {
    typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, a),
                                                  __builtin_bit_cast(h8_t, b), c, 0, 0, 0);
}

// A workgroup of 8 waves covers 8 gate/up channel pairs (128 + 128
// channels) of one task; wave p owns pair p for all of the task's row tiles
// (1, 2, 4 or 8 of 16 rows, a compile-time choice per task), so each weight
// fragment, converted once per wave, feeds up to 8 MFMAs.  The workgroup
// stages half a quad (64 columns of K, two scale groups) at a time into a
// double-buffered LDS image of 26 KB: the task's rows as fp16 MFMA
// fragments, its 16 weight tiles and their scale words; every thread loads
// one 16-byte row piece, two 8-byte weight pieces and (half of them) one
// scale word a step ahead and converts the row piece when it stores it.
// The barrier between steps waits for LDS operations only.  Two workgroups
// share a CU (8 waves each at 4 waves per SIMD), so one's barriers,
// prologue and epilogue overlap the other's MFMAs.  fp16 scales carry
// 16 * y (exact: far from the subnormal range), bf16 scales take s / 16.
template <uint32_t H, uint32_t I, bool kBf16>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4)))
void gate_up_w4g32_f16_kernel(const uint4* __restrict__ w, const uint16_t* __restrict__ s,
                              const int8_t* __restrict__ xq, const float* __restrict__ xs,
                              const uint32_t* __restrict__ packed,
                              const float* __restrict__ route_weights,
                              TaskSlots slots, uint16_t* __restrict__ mid) {
    constexpr uint32_t kHalves = H / 64u;  // staging steps
    constexpr uint32_t kTilesAll = 2u * I / 16u;
    constexpr uint32_t kWgTiles = 16u;  // 8 pairs
    static_assert(kHalves % 2u == 0u, "steps run in pairs of LDS buffers");
    // per buffer: A [K step j][row tile][lane] fp16 fragments (16 B), the
    // workgroup's 16 weight tiles [tile][K step j][lane] (one word: eight
    // nibbles) and their scale words [tile][channel] (two groups)
    __shared__ __align__(16) uint4 a_lds[2][2u * kRowTiles * 64u];
    __shared__ __align__(16) uint32_t w_lds[2][kWgTiles * 2u * 64u];
    __shared__ __align__(16) uint32_t s_lds[2][kWgTiles * 16u];
    __shared__ float2 row_info[kWideRows];  // (token scale, route weight)

    Placement at;
    if (!place_on_xcds(slots, I / 16u / 8u, at)) return;
    const TaskRecord task = read_task(slots.tasks, at.task);
    const uint32_t rows = task.rows;
    if (rows == 0u) return;
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u;
    const uint32_t pr = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t n = lane & 15u, qh = lane >> 4;
    const uint32_t e = task.expert;
    const uint32_t p0 = task.begin;
    const uint32_t tiles = __builtin_amdgcn_readfirstlane((rows + 15u) / 16u);

    // staging: row piece (row tid/4, 16-byte chunk tid%4 of the step's 64
    // bytes), weight pieces (tiles tid/64 and 8 + tid/64, lane tid%64: the
    // step's two words of the quad's four), scale piece (tile, channel) =
    // tid for tid < 256 (the step's two group words of the quad's four)
    const uint32_t sr = tid >> 2, sch = tid & 3u;
    const bool alive = sr < rows;
    const uint32_t assignment = alive ? checked(packed[p0 + sr], Q38M_WIDE_MAX_TOKENS * kTopK, kCheckToken) : 0u;
    if (sch == 0u && alive)
        row_info[sr] = make_float2(xs[assignment / kTopK], route_weights[assignment]);
    const uint4* a_src =
        reinterpret_cast<const uint4*>(xq + static_cast<size_t>(assignment / kTopK) * H) + sch;
    const uint32_t a_at = ((sch >> 1) * kRowTiles + (sr >> 4)) * 64u + (sch & 1u) * 32u +
                          ((sr & 15u) ^ a_swizzle(sch));
    const size_t slot0 = static_cast<size_t>(e) * (H / 128u) * kTilesAll + at.slice * kWgTiles;
    const uint2* w_src = reinterpret_cast<const uint2*>(w + slot0 * 64u + tid);
    // threads past the scale piece re-read thread tid % 256's word and
    // store the same value to the same LDS word
    const uint32_t s_at = tid % (kWgTiles * 16u);
    const uint32_t* s_src =
        reinterpret_cast<const uint32_t*>(s) + slot0 * 32u + 2u * s_at;
    struct Stage {
        uint4 a;
        uint2 w0, w1;
        uint32_t s;
    };
    // step h: quad h/2, words 2(h%2), 2(h%2)+1 of each weight piece and
    // scale record.  Every thread issues the same loads unconditionally (a
    // row past the task reads token 0's row, whose products land in rows
    // that are never stored), so the wait before each LDS store covers
    // exactly that step's loads and nothing waits on a prefetch early.
    auto load_stage = [&](uint32_t h) __attribute__((always_inline)) {
        Stage st;
        st.a = a_src[h * 4u];
        const uint2* wq = w_src + (static_cast<size_t>(h >> 1) * kTilesAll * 64u) * 2u + (h & 1u);
        st.w0 = wq[0];
        st.w1 = wq[8u * 64u * 2u];
        st.s = s_src[static_cast<size_t>(h >> 1) * kTilesAll * 32u + (h & 1u)];
        return st;
    };
    auto store_stage = [&](const Stage& st, uint32_t buffer) __attribute__((always_inline)) {
        a_lds[buffer][a_at] = i8_to_f16(st.a.x, st.a.y);
        a_lds[buffer][a_at + 16u] = i8_to_f16(st.a.z, st.a.w);
        const uint32_t w_at = (tid >> 6) * 128u + lane;
        w_lds[buffer][w_at] = st.w0.x;
        w_lds[buffer][w_at + 64u] = st.w0.y;
        w_lds[buffer][w_at + 8u * 128u] = st.w1.x;
        w_lds[buffer][w_at + 8u * 128u + 64u] = st.w1.y;
        s_lds[buffer][s_at] = st.s;
    };

    float y[kRowTiles][2][4];
#pragma unroll
    for (uint32_t t = 0; t < kRowTiles; ++t)
#pragma unroll
        for (uint32_t u = 0; u < 2u; ++u)
#pragma unroll
            for (uint32_t i = 0; i < 4u; ++i) y[t][u][i] = 0.0f;
    const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};

    // One step for kNt row tiles: per K step (= scale group) the pair's two
    // weight fragments are converted once; chain k = (row tile, gate/up),
    // tile t+1's A fragment read one chain ahead, each chain's fma step
    // issued after the next chain's MFMA.
    auto multiply = [&](auto ntiles, uint32_t buffer) __attribute__((always_inline)) {
        constexpr uint32_t kNt = decltype(ntiles)::value;
        constexpr uint32_t kChains = 2u * kNt * 2u;
        // lane l reads row l%16 of chunk l/16, through the staging swizzle
        const uint4* abuf0 = a_lds[buffer] + ((lane & 48u) | ((lane & 15u) ^ a_swizzle(lane >> 5)));
        const uint4* abuf1 = a_lds[buffer] + ((lane & 48u) | ((lane & 15u) ^ a_swizzle((lane >> 5) + 2u)));
        const uint32_t* srow = s_lds[buffer] + (2u * pr) * 16u + n;  // up: + 16 words
        // the step's scale words (gate, up; two groups each), read before
        // the first MFMA instead of one LDS round trip per group
        const uint32_t sword[2] = {srow[0], srow[16u]};
        const uint32_t* wrow = w_lds[buffer] + (2u * pr) * 128u + lane;  // up: + 128
        uint4 fa[2];
        uint4 bf[2];
        float sc[2];
        v4f d[2];
        auto issue = [&](uint32_t k) __attribute__((always_inline)) {
            const uint32_t m = k / 2u, u = k & 1u;
            const uint32_t j = m / kNt, t = m % kNt;
            if (u == 0u) {
                if (t == 0u) {
                    bf[0] = w4_to_f16x16(wrow[j * 64u]);
                    bf[1] = w4_to_f16x16(wrow[128u + j * 64u]);
                }
                if (m + 1u < 2u * kNt) {
                    const uint32_t jn = (m + 1u) / kNt, tn = (m + 1u) % kNt;
                    fa[(m + 1u) & 1u] = (jn == 0u ? abuf0 : abuf1)[(jn * kRowTiles + tn) * 64u];
                }
            }
            d[k & 1u] = mfma_f16_16x16x32(fa[m & 1u], bf[u], zero);
        };
        auto step = [&](uint32_t k) __attribute__((always_inline)) {
            const uint32_t m = k / 2u, u = k & 1u;
            const uint32_t j = m / kNt, t = m % kNt;
            if (t == 0u) {
                const uint32_t word = (sword[u] >> (16u * j)) & 0xFFFFu;
                sc[u] = kBf16 ? bf16_to_f32(word) * 0.0625f : f16_to_f32(word);
                asm volatile("" : "+v"(sc[u]));  // a plain v_fma_f32, not v_fma_mix
            }
#pragma unroll
            for (uint32_t i = 0; i < 4u; ++i)
                y[t][u][i] = __builtin_fmaf(d[k & 1u][i], sc[u], y[t][u][i]);
            // keep the step between the MFMAs it follows and precedes
            asm volatile("" : "+v"(y[t][u][0]), "+v"(y[t][u][1]), "+v"(y[t][u][2]),
                         "+v"(y[t][u][3]));
        };
        fa[0] = abuf0[0];
#pragma unroll
        for (uint32_t k = 0; k <= kChains; ++k) {
            if (k < kChains) issue(k);
            __builtin_amdgcn_sched_barrier(0);
            if (k > 0u) step(k - 1u);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto lds_barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    // step h: loaded at the start of step h-1, stored at its end into LDS
    // buffer h%2, multiplied during step h; the loop is instantiated per
    // row-tile count, every instance passing the same barriers
    {
        const Stage first = load_stage(0);
        store_stage(first, 0u);
    }
    __syncthreads();
    auto k_loop = [&](auto ntiles) __attribute__((always_inline)) {
#pragma unroll 1
        for (uint32_t h = 0; h < kHalves; h += 2u) {
            Stage next = load_stage(h + 1u);
            __builtin_amdgcn_sched_barrier(0);
            multiply(ntiles, 0u);
            store_stage(next, 1u);
            lds_barrier();
            // the last pair's second load repeats step h + 1 into buffer 0,
            // which nothing reads after it (unconditional, so the loads stay
            // ahead of the multiply instead of sinking into a branch)
            next = load_stage(h + 2u < kHalves ? h + 2u : h + 1u);
            __builtin_amdgcn_sched_barrier(0);
            multiply(ntiles, 1u);
            store_stage(next, 0u);
            lds_barrier();
        }
    };
    if (tiles > 4u)
        k_loop(std::integral_constant<uint32_t, 8>{});
    else if (tiles > 2u)
        k_loop(std::integral_constant<uint32_t, 4>{});
    else if (tiles > 1u)
        k_loop(std::integral_constant<uint32_t, 2>{});
    else
        k_loop(std::integral_constant<uint32_t, 1>{});

    // SwiGLU (swiglu_fold's rounding sequence with silu(g) from the table,
    // NaN written as 0x7fc0 like swiglu_fold):
    // D lane (qh, n) holds rows 4qh + i of each tile, channel n.  Four
    // tiles' gathers are in flight before their first store.
    const uint32_t channel = (at.slice * 8u + pr) * 16u + n;
    const float unscale = kBf16 ? 1.0f : 0.0625f;
    constexpr uint32_t kBatch = 4u;
#pragma unroll
    for (uint32_t t0 = 0; t0 < kRowTiles; t0 += kBatch) {
        if (16u * t0 >= rows) break;
        uint32_t silu_word[kBatch][4];
        float up_value[kBatch][4];
#pragma unroll
        for (uint32_t b = 0; b < kBatch; ++b)
#pragma unroll
            for (uint32_t i = 0; i < 4u; ++i) {
                const uint32_t r = 16u * (t0 + b) + 4u * qh + i;
                const float st = row_info[r < rows ? r : 0u].x;
                const float yg = (y[t0 + b][0][i] * unscale) * st;
                up_value[b][i] = bf16_round((y[t0 + b][1][i] * unscale) * st);
                silu_word[b][i] = kSiluTable[f32_to_bf16(yg)];
            }
#pragma unroll
        for (uint32_t b = 0; b < kBatch; ++b)
#pragma unroll
            for (uint32_t i = 0; i < 4u; ++i) {
                const uint32_t r = 16u * (t0 + b) + 4u * qh + i;
                if (r >= rows) continue;
                const float h = bf16_round(__uint_as_float(silu_word[b][i]) * up_value[b][i]);
                mid[static_cast<size_t>(p0 + r) * I + channel] = static_cast<uint16_t>(
                    bf16_canonical_nan(f32_to_bf16(h * row_info[r].y)));
            }
    }
}

// ---- down -------------------------------------------------------------------

// The route outputs of a chunk (fp32 [R][H], 2.68 GB for a config-5 layer)
// are written once here and read once by the combine, far more than the
// L2s hold: stored with ordinary stores they are allocated in L2 and evict
// the expert weights and mid rows that an expert's later tasks re-read
// (the W8 down kernel fetched 1.44x its unique bytes), so they are stored
// non-temporally.
__device__ __forceinline__ void store_route_output(float* p, float v) {
    __builtin_nontemporal_store(v, p);
}

// Down, W8 per output channel, over a task of up to 128 rows: the mid rows
// (contiguous in packed order) are staged once into LDS as [K block][row
// tile][lane] 16-byte MFMA fragments.  Each wave owns kTilesPerWave
// 16-channel output tiles and walks K in the outer loop: a K block's kRows
// A fragments are read from LDS once and multiplied into every owned tile
// (v_mfma_i32_16x16x64_i8), with the tiles' weight fragments two K blocks
// ahead.  One A fragment is live at a time (row by row): holding all kRows
// of them took the kernel to 256 VGPRs with spills (1.07 ms vs 1.00 ms on
// a config-5 layer).  kRows (8, 4, 2 or 1 row tiles) is picked per task from its row
// count.  o = ((float)acc * ws[e][c]) * sm[r], as the slab kernel.
template <uint32_t H, uint32_t I, uint32_t kTilesPerWave, uint32_t kRows, bool kBf16>
__device__ __forceinline__ void down_w8_wide_rows(const uint4* __restrict__ wt,
                                                  const uint16_t* __restrict__ ws_expert,
                                                  const uint4* a_lds, const float* row_scale,
                                                  uint32_t rows, uint32_t p0, uint32_t tile0,
                                                  float* __restrict__ out) {
    constexpr uint32_t kBlocks = I / 64u;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t n = lane & 15u;
    const uint32_t q = lane >> 4;
    const v4i zero = {0, 0, 0, 0};
    v4i acc[kTilesPerWave][kRows];
#pragma unroll
    for (uint32_t t = 0; t < kTilesPerWave; ++t)
#pragma unroll
        for (uint32_t r = 0; r < kRows; ++r) acc[t][r] = zero;
    // tile t's K block kb: wt[(t * kBlocks + kb) * 64]
    uint4 wq[3][kTilesPerWave];
    auto load_w = [&](uint32_t kb, uint4 (&dst)[kTilesPerWave]) {
        const uint32_t k = kb < kBlocks ? kb : kBlocks - 1u;
#pragma unroll
        for (uint32_t t = 0; t < kTilesPerWave; ++t) dst[t] = wt[(t * kBlocks + k) * 64u];
    };
    load_w(0, wq[0]);
    load_w(1, wq[1]);
#pragma unroll
    for (uint32_t kb = 0; kb < kBlocks; ++kb) {
        load_w(kb + 2u, wq[(kb + 2u) % 3u]);
#pragma unroll
        for (uint32_t r = 0; r < kRows; ++r) {
            const v4i a = as_v4i(a_lds[(kb * kRowTiles + r) * 64u + lane]);
#pragma unroll
            for (uint32_t t = 0; t < kTilesPerWave; ++t)
                acc[t][r] = mfma_i8_16x16x64(a, as_v4i(wq[kb % 3u][t]), acc[t][r]);
        }
    }
    // the tiles' scales of channel 16*(tile0+t)+n, read after the K loop
    // (fewer live VGPRs)
    float ws[kTilesPerWave];
#pragma unroll
    for (uint32_t t = 0; t < kTilesPerWave; ++t) {
        const uint32_t word = ws_expert[(tile0 + t) * 16u + n];
        ws[t] = kBf16 ? bf16_to_f32(word) : f16_to_f32(word);
    }
    // a row's kTilesPerWave adjacent 16-channel pieces go out in consecutive
    // stores, so its 64*kTilesPerWave bytes meet in L2 as whole lines
#pragma unroll
    for (uint32_t r = 0; r < kRows; ++r)
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) {
            const uint32_t row = 16u * r + 4u * q + i;
            if (row >= rows) continue;
            const float sm = row_scale[row];
            float* dst = out + static_cast<size_t>(p0 + row) * H + tile0 * 16u + n;
#pragma unroll
            for (uint32_t t = 0; t < kTilesPerWave; ++t)
                store_route_output(dst + 16u * t, (static_cast<float>(acc[t][r][i]) * ws[t]) * sm);
        }
}

template <uint32_t H, uint32_t I, uint32_t kWaves, uint32_t kTilesPerWave, bool kBf16>
__global__ __launch_bounds__(kWaves * 64) void down_w8_wide_kernel(
    const uint4* __restrict__ w, const uint16_t* __restrict__ s,
    const int8_t* __restrict__ mq, const float* __restrict__ ms,
    TaskSlots slots, float* __restrict__ out) {
    constexpr uint32_t kBlocks = I / 64u;
    constexpr uint32_t kTiles = H / 16u;
    constexpr uint32_t kThreads = kWaves * 64u;
    constexpr uint32_t kPieces = kWideRows * (I / 16u);
    static_assert(kPieces % kThreads == 0u, "whole pieces per thread");
    __shared__ uint4 a_lds[kBlocks * kRowTiles * 64u];
    __shared__ float row_scale[kWideRows];

    Placement at;
    if (!place_on_xcds(slots, H / 16u / (kWaves * kTilesPerWave), at)) return;
    const TaskRecord task = read_task(slots.tasks, at.task);
    const uint32_t rows = task.rows;
    if (rows == 0u) return;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t e = task.expert;
    const uint32_t p0 = task.begin;
    const uint32_t tile0 = (at.slice * kWaves + wave) * kTilesPerWave;
    const uint4* wt = w + static_cast<size_t>(e * kTiles + tile0) * kBlocks * 64u + lane;
    const uint32_t tiles = (rows + 15u) / 16u;  // uniform per workgroup

    // Piece i: row r = i / (I/16), 16-byte piece c: K block c/4, lane group
    // c%4.  Every load is issued before the first store (rows past the task
    // re-read its first row and stage zeros), so staging is one round trip.
    constexpr uint32_t kPer = kPieces / kThreads;
    uint4 v[kPer];
#pragma unroll
    for (uint32_t u = 0; u < kPer; ++u) {
        const uint32_t i = threadIdx.x + u * kThreads;
        const uint32_t r = i / (I / 16u), c = i % (I / 16u);
        v[u] = reinterpret_cast<const uint4*>(mq + static_cast<size_t>(p0 + (r < rows ? r : 0u)) *
                                                       I)[c];
    }
#pragma unroll
    for (uint32_t u = 0; u < kPer; ++u) {
        const uint32_t i = threadIdx.x + u * kThreads;
        const uint32_t r = i / (I / 16u), c = i % (I / 16u);
        if (r < 16u * tiles)
            a_lds[((c >> 2) * kRowTiles + r / 16u) * 64u + (c & 3u) * 16u + r % 16u] =
                r < rows ? v[u] : make_uint4(0u, 0u, 0u, 0u);
    }
    if (threadIdx.x < kWideRows)
        row_scale[threadIdx.x] = threadIdx.x < rows ? ms[p0 + threadIdx.x] : 0.0f;
    __syncthreads();

    const uint16_t* ws_expert = s + static_cast<size_t>(e) * H;
    auto run = [&](auto row_tiles) {
        down_w8_wide_rows<H, I, kTilesPerWave, decltype(row_tiles)::value, kBf16>(
            wt, ws_expert, a_lds, row_scale, rows, p0, tile0, out);
    };
    if (tiles > 4u)
        run(std::integral_constant<uint32_t, 8>{});
    else if (tiles > 2u)
        run(std::integral_constant<uint32_t, 4>{});
    else if (tiles == 2u)
        run(std::integral_constant<uint32_t, 2>{});
    else
        run(std::integral_constant<uint32_t, 1>{});
}

// Down, W4 groups of 32, on fp16 MFMA (see the gate/up kernel above for
// why the products are exact): a workgroup of 8 waves covers 16 output
// tiles of one task, two adjacent tiles per wave over all of the task's row
// tiles, so a row's 128-byte output line leaves one wave in two
// consecutive stores.  The mid rows are staged 64 columns at a time as fp16
// fragments in a double-buffered LDS image (16 KB per buffer); each wave
// streams its two tiles' weights and scale words one step ahead from
// global memory and converts each weight fragment once for all row tiles.
// The chain is the int8 kernel's: y = fmaf((float)acc_g, s_g / 16, y) in
// group order, then y * s_row.
template <uint32_t H, uint32_t I, bool kBf16>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4)))
void down_w4g32_f16_kernel(const uint4* __restrict__ w, const uint16_t* __restrict__ s,
                           const int8_t* __restrict__ mq, const float* __restrict__ ms,
                           TaskSlots slots, float* __restrict__ out) {
    constexpr uint32_t kSteps = I / 64u;
    constexpr uint32_t kTiles = H / 16u;
    static_assert(kSteps % 2u == 0u, "steps run in pairs of LDS buffers");
    __shared__ __align__(16) uint4 a_lds[2][2u * kRowTiles * 64u];
    __shared__ float row_scale[kWideRows];

    Placement at;
    if (!place_on_xcds(slots, H / 16u / 16u, at)) return;
    const TaskRecord task = read_task(slots.tasks, at.task);
    const uint32_t rows = task.rows;
    if (rows == 0u) return;
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t n = lane & 15u, qh = lane >> 4;
    const uint32_t e = task.expert;
    const uint32_t p0 = task.begin;
    const uint32_t tiles = __builtin_amdgcn_readfirstlane((rows + 15u) / 16u);

    // staging: row piece (row tid/4, 16-byte chunk tid%4 of the step's 64
    // bytes); the task's mid rows are contiguous
    const uint32_t sr = tid >> 2, sch = tid & 3u;
    const bool alive = sr < rows;
    const uint4* a_src =
        reinterpret_cast<const uint4*>(mq + static_cast<size_t>(p0 + (alive ? sr : 0u)) * I) + sch;
    const uint32_t a_at = ((sch >> 1) * kRowTiles + (sr >> 4)) * 64u + (sch & 1u) * 32u + (sr & 15u);
    if (tid < kWideRows) row_scale[tid] = tid < rows ? ms[p0 + tid] : 0.0f;
    auto load_a = [&](uint32_t h) __attribute__((always_inline)) {
        return alive ? a_src[h * 4u] : make_uint4(0u, 0u, 0u, 0u);
    };
    auto store_a = [&](const uint4& v, uint32_t buffer) __attribute__((always_inline)) {
        a_lds[buffer][a_at] = i8_to_f16(v.x, v.y);
        a_lds[buffer][a_at + 16u] = i8_to_f16(v.z, v.w);
    };

    // this wave's tiles tile0, tile0 + 1; quad-major layout: quad kq of tile
    // t is unit kq * kTiles + t of the expert, four K steps (one word each)
    // per lane and four scale words per channel; step h takes words
    // 2(h%2), 2(h%2)+1 of quad h/2
    const uint32_t tile0 = (at.slice * 8u + wave) * 2u;
    const size_t unit0 = static_cast<size_t>(e) * (I / 128u) * kTiles + tile0;
    const uint2* wsrc = reinterpret_cast<const uint2*>(w + unit0 * 64u + lane);
    const uint32_t* ssrc = reinterpret_cast<const uint32_t*>(s + (unit0 * 16u + n) * 4u);
    struct Step {
        uint2 w0, w1;
        uint32_t s0, s1;
    };
    auto load_w = [&](uint32_t h) __attribute__((always_inline)) {
        const size_t unit = static_cast<size_t>(h >> 1) * kTiles;
        Step st;
        st.w0 = wsrc[unit * 128u + (h & 1u)];
        st.w1 = wsrc[(unit + 1u) * 128u + (h & 1u)];
        st.s0 = ssrc[unit * 32u + (h & 1u)];
        st.s1 = ssrc[(unit + 1u) * 32u + (h & 1u)];
        return st;
    };

    float y[kRowTiles][2][4];
#pragma unroll
    for (uint32_t t = 0; t < kRowTiles; ++t)
#pragma unroll
        for (uint32_t u = 0; u < 2u; ++u)
#pragma unroll
            for (uint32_t i = 0; i < 4u; ++i) y[t][u][i] = 0.0f;
    const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};

    // one step (two groups) for kNt row tiles; chain k = (group j, row tile
    // t, tile u) as in the gate/up kernel
    auto multiply = [&](auto ntiles, uint32_t buffer, const Step& ws)
                        __attribute__((always_inline)) {
        constexpr uint32_t kNt = decltype(ntiles)::value;
        constexpr uint32_t kChains = 2u * kNt * 2u;
        const uint4* abuf = a_lds[buffer] + lane;
        const uint32_t wj[2][2] = {{ws.w0.x, ws.w0.y}, {ws.w1.x, ws.w1.y}};
        const uint32_t sj[2] = {ws.s0, ws.s1};
        uint4 fa[2];
        uint4 bf[2];
        float sc[2];
        v4f d[2];
        auto issue = [&](uint32_t k) __attribute__((always_inline)) {
            const uint32_t m = k / 2u, u = k & 1u;
            const uint32_t j = m / kNt, t = m % kNt;
            if (u == 0u) {
                if (t == 0u) {
                    bf[0] = w4_to_f16x16(wj[0][j]);
                    bf[1] = w4_to_f16x16(wj[1][j]);
                }
                if (m + 1u < 2u * kNt) {
                    const uint32_t jn = (m + 1u) / kNt, tn = (m + 1u) % kNt;
                    fa[(m + 1u) & 1u] = abuf[(jn * kRowTiles + tn) * 64u];
                }
            }
            d[k & 1u] = mfma_f16_16x16x32(fa[m & 1u], bf[u], zero);
        };
        auto step = [&](uint32_t k) __attribute__((always_inline)) {
            const uint32_t m = k / 2u, u = k & 1u;
            const uint32_t j = m / kNt, t = m % kNt;
            if (t == 0u) {
                const uint32_t word = j ? sj[u] >> 16 : sj[u] & 0xffffu;
                sc[u] = (kBf16 ? bf16_to_f32(word) : f16_to_f32(word)) * 0.0625f;
                asm volatile("" : "+v"(sc[u]));
            }
#pragma unroll
            for (uint32_t i = 0; i < 4u; ++i)
                y[t][u][i] = __builtin_fmaf(d[k & 1u][i], sc[u], y[t][u][i]);
            asm volatile("" : "+v"(y[t][u][0]), "+v"(y[t][u][1]), "+v"(y[t][u][2]),
                         "+v"(y[t][u][3]));
        };
        fa[0] = abuf[0];
#pragma unroll
        for (uint32_t k = 0; k <= kChains; ++k) {
            if (k < kChains) issue(k);
            __builtin_amdgcn_sched_barrier(0);
            if (k > 0u) step(k - 1u);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto lds_barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    store_a(load_a(0), 0u);
    Step cur = load_w(0);
    __syncthreads();
    auto k_loop = [&](auto ntiles) __attribute__((always_inline)) {
#pragma unroll 1
        for (uint32_t h = 0; h < kSteps; h += 2u) {
            uint4 a_next = load_a(h + 1u);
            Step nxt = load_w(h + 1u);
            __builtin_amdgcn_sched_barrier(0);
            multiply(ntiles, 0u, cur);
            store_a(a_next, 1u);
            lds_barrier();
            cur = nxt;
            if (h + 2u < kSteps) {
                a_next = load_a(h + 2u);
                nxt = load_w(h + 2u);
            }
            __builtin_amdgcn_sched_barrier(0);
            multiply(ntiles, 1u, cur);
            if (h + 2u < kSteps) store_a(a_next, 0u);
            lds_barrier();
            cur = nxt;
        }
    };
    if (tiles > 4u)
        k_loop(std::integral_constant<uint32_t, 8>{});
    else if (tiles > 2u)
        k_loop(std::integral_constant<uint32_t, 4>{});
    else if (tiles > 1u)
        k_loop(std::integral_constant<uint32_t, 2>{});
    else
        k_loop(std::integral_constant<uint32_t, 1>{});

    const uint32_t channel = tile0 * 16u + n;
#pragma unroll
    for (uint32_t t = 0; t < kRowTiles; ++t) {
        if (16u * t >= rows) break;
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) {
            const uint32_t row = 16u * t + 4u * qh + i;
            if (row >= rows) continue;
            float* dst = out + static_cast<size_t>(p0 + row) * H + channel;
            store_route_output(dst, y[t][0][i] * row_scale[row]);
            store_route_output(dst + 16, y[t][1][i] * row_scale[row]);
        }
    }
}

// ---- gate/up and down on 32x32 int8 MFMA ------------------------------------
//
// Every chunk format whose scale groups are at least 64 columns wide (W4 in
// groups of 64 or 128, W8 in groups of 64 or 128, W8 per channel for
// gate/up) runs one kernel.  A workgroup of four waves covers eight adjacent
// weight slots (128 output channels) and 64 rows of one task; wave w owns
// slots 2w and 2w + 1 -- the gate and the up tile of a channel pair, or two
// adjacent output tiles of down -- as the 32 columns of
// v_mfma_i32_32x32x32_i8, over one or two 32-row tiles.  Per 128-column step
// the workgroup stages its int8 rows in a double-buffered 8 KB LDS image;
// a wave's weights go straight to its registers, one to three steps ahead.
//
// What bounds it: the matrix cores and the VALU overlap only in part.  Three
// waves per SIMD of independent v_mfma_i32_32x32x32_i8 and v_fma_f32 take, per
// MFMA, 13.7 ns alone; with four v_fma_f32 (5.1 ns alone) 14.6, with eight (9.5)
// 18.5, sixteen (19.4) 28.1, 32 (38.2) 45.4: from eight on about two thirds of the
// MFMA's time come on top of the VALU's.  So both are kept few (here 13 to 21
// VALU instructions per MFMA; 6,001 tokens in W4 groups of 128: MFMA busy 25 %,
// VALU issue 50 %).  The 32x32 form does twice the work of the 16x16x32 form
// per matrix cycle.  The
// group chain is two VALU instructions per element: the MFMA accumulator
// starts from the bits of 1.5 * 2^23, so its result read as a float is
// 12582912 + acc exactly (|acc| < 2^22: 16 w a over 128 columns stays below
// 2.1e6), one v_add_f32 recovers (float)acc -- v_cvt_f32_i32 runs at half
// rate -- and one v_fma_f32 continues y = fmaf((float)acc_g, s_g, y) in group
// order.  W4 nibbles sit in the high half of their byte (16 w), so their
// scale is s / 16, exact.  Measured against the 16x16 kernels it replaces
// (128-row tasks, 16 waves): W4 groups of 128 at 6,001 tokens gate/up 411 ->
// 300 us and down 300 -> 208 us (down's 491 MB of route outputs alone: 97 us);
// W8 groups of 128 at 1,500 tokens 285 -> 190 and 136 -> 110 us, at 8,192
// tokens 751 -> 501 and 424 -> 334 us.  64 rows per workgroup at three waves
// per SIMD run as fast as 128 rows at two (W8 181 / 113 us, W4 330 / 250);
// rows resident in LDS over all of K with one workgroup per CU take 384-469
// us for the W4 gate/up, non-temporal weights 337 us.
//
// A image: row r's 16-byte chunk c (0..7 of the step's 128 columns) is at
// slot c * 64 + (r ^ c): the staging stores (eight chunks of a row by eight
// neighbouring lanes) and the fragment reads (one chunk, 32 rows) both fall
// in distinct banks.  MFMA j of a step takes chunks 2j and 2j + 1, lane
// (h, r) row r of chunk 2j + h; the weights' lane (h, c) brings column c's
// same 16 values: words j of lanes (2h, n) and (2h + 1, n) of a W4 quad, or
// the 16 bytes of lane q = 2 (j % 2) + h of a W8 64-column block j / 2.
constexpr uint32_t kI8Rows = 64;  // rows per workgroup

template <uint32_t kBits, uint32_t kGroup, bool kGateUp>
struct WideI8 {
    static constexpr uint32_t kK = kGateUp ? kHidden : kInter;
    static constexpr uint32_t kSlots = kGateUp ? 2u * kInter / 16u : kHidden / 16u;
    static constexpr uint32_t kSteps = kK / 128u;
    static constexpr uint32_t kSlices = kSlots / 8u;  // workgroups per 64 rows of a task
    static constexpr uint32_t kHalves = kWideRows / kI8Rows;
    static constexpr bool kPerChannel = kGroup == 0u;
    static constexpr uint32_t kGroups = kGroup == 64u ? 2u : 1u;  // chain steps per 128 columns
    static constexpr uint32_t kMfma = 4u / kGroups;               // MFMAs per chain step
    static constexpr uint32_t kLoads = kBits == 4u ? 2u : 4u;     // 16-byte weight loads per step
};

template <uint32_t kBits, uint32_t kGroup, bool kBf16, bool kGateUp>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
void wide_i8_kernel(const uint4* __restrict__ w, const uint16_t* __restrict__ s,
                    const int8_t* __restrict__ rows_q, const float* __restrict__ row_scales,
                    const uint32_t* __restrict__ packed, const float* __restrict__ route_weights,
                    TaskSlots slots, void* __restrict__ out) {
    using F = WideI8<kBits, kGroup, kGateUp>;
    constexpr uint32_t kK = F::kK, kSlots = F::kSlots, kSteps = F::kSteps;
    static_assert(kSteps % 2u == 0u, "steps run in pairs of LDS buffers");
    static_assert(kBits == 8u || kGroup != 0u, "W4 is always grouped");
    __shared__ u32x4 a_lds[2][8u * kI8Rows];
    __shared__ float2 row_info[kI8Rows];  // (row scale, route weight)

    Placement at;
    if (!place_on_xcds(slots, F::kSlices * F::kHalves, at)) return;
    const TaskRecord task = read_task(slots.tasks, at.task);
    // this workgroup's rows of the task: 64 from row 64 * half
    const uint32_t half = at.slice / F::kSlices;
    const uint32_t slice = at.slice % F::kSlices;
    if (task.rows <= kI8Rows * half) return;
    const uint32_t rows = min(task.rows - kI8Rows * half, kI8Rows);
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t c = lane & 31u, h = lane >> 5, n = lane & 15u;
    const uint32_t e = task.expert;
    const uint32_t p0 = task.begin + kI8Rows * half;
    const uint32_t slot0 = slice * 8u + 2u * wave;
    const uint32_t slot = slot0 + (c >> 4);

    // staging: pieces u = 0, 1, row tid/8 + 32u, 16-byte chunk tid%8; a row
    // past the task reads a row that exists, and its products land in rows
    // that are never stored
    const uint32_t sch = tid & 7u;
    uint32_t a_off[2];
#pragma unroll
    for (uint32_t u = 0; u < 2u; ++u) {
        const uint32_t r = (tid >> 3) + 32u * u;
        if constexpr (kGateUp) {
            uint32_t token = 0u;
            if (r < rows) {
                const uint32_t a = checked(packed[p0 + r], Q38M_WIDE_MAX_TOKENS * kTopK, kCheckToken);
                token = a / kTopK;
                if (sch == 0u) row_info[r] = make_float2(row_scales[token], route_weights[a]);
            }
            a_off[u] = token * kK + sch * 16u;
        } else {
            a_off[u] = (p0 + (r < rows ? r : 0u)) * kK + sch * 16u;
            if (sch == 0u && r < rows) row_info[r] = make_float2(row_scales[p0 + r], 0.0f);
        }
    }
    const uint32_t a_at = sch * kI8Rows + ((tid >> 3) ^ sch);

    // the wave's weights: see the layouts in q38m.h
    const uint4* w_step;  // uniform, advanced per step
    uint32_t w_off;       // the lane's 16-byte piece of load 0
    constexpr uint32_t kWStep = kBits == 4u ? kSlots * 64u : kGateUp ? 2u * kSlots * 64u : 128u;
    if constexpr (kBits == 4u) {
        w_step = w + static_cast<size_t>(e) * kSteps * kSlots * 64u;
        w_off = slot * 64u + 32u * h + n;
    } else if constexpr (kGateUp) {
        w_step = w + static_cast<size_t>(e) * (kK / 64u) * kSlots * 64u;
        w_off = slot * 64u + 16u * h + n;
    } else {
        w_step = w + static_cast<size_t>(e) * (kK / 64u) * kSlots * 64u;
        w_off = slot * (kK / 64u) * 64u + 16u * h + n;
    }
    const uint16_t* s_base;  // the lane's scale words of step 0
    constexpr uint32_t kSStep =
        kBits == 4u ? kSlots * 16u * F::kGroups : F::kPerChannel ? 0u : F::kGroups;
    if constexpr (kBits == 4u) {
        s_base = s + ((static_cast<size_t>(e) * kSteps * kSlots + slot) * 16u + n) * F::kGroups;
    } else {
        const uint32_t row = kGateUp ? (c >> 4) * kInter + (slot0 >> 1) * 16u + n : slot * 16u + n;
        const uint32_t per_row = F::kPerChannel ? 1u : kK / 128u * F::kGroups;
        s_base = s + (static_cast<size_t>(e) * kSlots * 16u + row) * per_row;
    }
    struct Weights {
        u32x4 v[F::kLoads];
        uint32_t s;
    };
    auto load_weights = [&](uint32_t step) __attribute__((always_inline)) {
        Weights x;
        const u32x4* p = reinterpret_cast<const u32x4*>(w_step) + static_cast<size_t>(step) * kWStep;
#pragma unroll
        for (uint32_t j = 0; j < F::kLoads; ++j) {
            constexpr uint32_t kBlock = kGateUp ? kSlots * 64u : 64u;  // W8: the next 64 columns
            x.v[j] = p[w_off + (kBits == 4u ? 16u * j : (j >> 1) * kBlock + (j & 1u) * 32u)];
        }
        const uint16_t* q = s_base + static_cast<size_t>(step) * kSStep;
        if constexpr (F::kGroups == 2u) x.s = *reinterpret_cast<const uint32_t*>(q);
        else x.s = *q;
        return x;
    };

    v16i bias;
#pragma unroll
    for (uint32_t i = 0; i < 16u; ++i) bias[i] = F::kPerChannel ? 0 : 0x4B400000;
    if constexpr (!F::kPerChannel) asm volatile("" : "+v"(bias));  // one register block
    float unbias;  // -12582912.0f in a scalar register (no literal per use)
    asm volatile("s_mov_b32 %0, 0xcb400000" : "=s"(unbias));
    auto lds_barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    auto run = [&](auto row_tiles) __attribute__((always_inline)) {
        constexpr uint32_t kNt = decltype(row_tiles)::value;
        float y[kNt][16];  // grouped: the fp32 chain
        v16i acc[F::kPerChannel ? kNt : 1];
#pragma unroll
        for (uint32_t t = 0; t < kNt; ++t)
#pragma unroll
            for (uint32_t i = 0; i < 16u; ++i) y[t][i] = 0.0f;
        if constexpr (F::kPerChannel) {
#pragma unroll
            for (uint32_t t = 0; t < kNt; ++t) acc[t] = bias;
        }
        struct Rows {
            u32x4 v[kNt];
        };
        auto load_rows = [&](uint32_t step) __attribute__((always_inline)) {
            Rows x;
            const int8_t* p = rows_q + step * 128u;
#pragma unroll
            for (uint32_t u = 0; u < kNt; ++u) x.v[u] = *reinterpret_cast<const u32x4*>(p + a_off[u]);
            return x;
        };
        auto store_rows = [&](const Rows& x, uint32_t buffer) __attribute__((always_inline)) {
#pragma unroll
            for (uint32_t u = 0; u < kNt; ++u) a_lds[buffer][a_at + 32u * u] = x.v[u];
        };
        // weights in flight: one step (two row tiles) or three (one tile,
        // whose steps are short against the memory latency); W4 sets are
        // unpacked at the start of their step and refilled at once
        constexpr uint32_t kRing = kBits == 4u ? (kNt == 1u ? 4u : 1u) : (kNt == 1u ? 4u : 2u);
        Weights ring[kRing];
        Rows ahead;
        auto clamped = [](uint32_t k) { return k < kSteps ? k : kSteps - 1u; };

        // step k on LDS buffer j4 % 2 (j4 = k % 4, a compile-time constant)
        auto step = [&](uint32_t k, auto jc) __attribute__((always_inline)) {
            constexpr uint32_t j4 = decltype(jc)::value;
            constexpr uint32_t buffer = j4 & 1u;
            ahead = load_rows(clamped(k + 1u));
            if constexpr (kBits == 8u) ring[(j4 + kRing - 1u) % kRing] = load_weights(clamped(k + kRing - 1u));
            const Weights& x = ring[j4 % kRing];
            v4i b[4];
            float sc[F::kGroups];
            if constexpr (kBits == 4u) {
                const uint32_t lo[4] = {x.v[0].x, x.v[0].y, x.v[0].z, x.v[0].w};
                const uint32_t hi[4] = {x.v[1].x, x.v[1].y, x.v[1].z, x.v[1].w};
#pragma unroll
                for (uint32_t j = 0; j < 4u; ++j) {
                    b[j].x = static_cast<int>((lo[j] << 4) & 0xf0f0f0f0u);
                    b[j].y = static_cast<int>(lo[j] & 0xf0f0f0f0u);
                    b[j].z = static_cast<int>((hi[j] << 4) & 0xf0f0f0f0u);
                    b[j].w = static_cast<int>(hi[j] & 0xf0f0f0f0u);
                }
            } else {
#pragma unroll
                for (uint32_t j = 0; j < 4u; ++j) b[j] = __builtin_bit_cast(v4i, x.v[j]);
            }
#pragma unroll
            for (uint32_t g = 0; g < F::kGroups; ++g) {
                const uint32_t word = (x.s >> (16u * g)) & 0xffffu;
                sc[g] = (kBf16 ? bf16_to_f32(word) : f16_to_f32(word)) * (kBits == 4u ? 0.0625f : 1.0f);
                asm volatile("" : "+v"(sc[g]));  // a plain v_fma_f32, not v_fma_mix
            }
            if constexpr (kBits == 4u) {
                __builtin_amdgcn_sched_barrier(0);
                ring[j4 % kRing] = load_weights(clamped(k + kRing));
            }
            __builtin_amdgcn_sched_barrier(0);
            const u32x4* image = a_lds[buffer] + h * kI8Rows;
            auto fragment = [&](uint32_t t, uint32_t j) __attribute__((always_inline)) {
                return __builtin_bit_cast(v4i, image[2u * j * kI8Rows + 32u * t + (c ^ (2u * j + h))]);
            };
            // kBatch fragments at a time: MFMA batch q of tile t is MFMAs
            // kBatch q .. kBatch q + kBatch - 1, the next batch's fragments
            // requested behind it
            constexpr uint32_t kBatch = kGateUp ? F::kMfma : 2u;
            constexpr uint32_t kBatches = 4u / kBatch;
            v4i fa[kBatch];
#pragma unroll
            for (uint32_t i = 0; i < kBatch; ++i) fa[i] = fragment(0u, i);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (uint32_t t = 0; t < kNt; ++t) {
                v16i& d = acc[F::kPerChannel ? t : 0u];
#pragma unroll
                for (uint32_t q = 0; q < kBatches; ++q) {
#pragma unroll
                    for (uint32_t i = 0; i < kBatch; ++i) {
                        const uint32_t j = q * kBatch + i;
                        d = mfma_i8_32x32x32(fa[i], b[j], !F::kPerChannel && j % F::kMfma == 0u ? bias : d);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    const uint32_t next = t * kBatches + q + 1u;
                    if (next < kNt * kBatches) {
#pragma unroll
                        for (uint32_t i = 0; i < kBatch; ++i)
                            fa[i] = fragment(next / kBatches, next % kBatches * kBatch + i);
                    }
                    if constexpr (!F::kPerChannel) {
                        if ((q + 1u) * kBatch % F::kMfma == 0u) {
                            const uint32_t g = ((q + 1u) * kBatch - 1u) / F::kMfma;
#pragma unroll
                            for (uint32_t i = 0; i < 16u; ++i)
                                y[t][i] = __builtin_fmaf(__int_as_float(d[i]) + unbias, sc[g], y[t][i]);
#pragma unroll
                            for (uint32_t i = 0; i < 16u; i += 4u)
                                asm volatile("" : "+v"(y[t][i]), "+v"(y[t][i + 1u]), "+v"(y[t][i + 2u]),
                                             "+v"(y[t][i + 3u]));
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            store_rows(ahead, buffer ^ 1u);
            lds_barrier();
        };
        // before step 0: its rows in buffer 0, the first steps' weights in
        // flight; loads past the end repeat the last step's, unread
        static_assert(kSteps % 4u == 0u, "the loop covers four ring slots");
#pragma unroll
        for (uint32_t j = 0; j + (kBits == 8u ? 1u : 0u) < kRing; ++j) ring[j] = load_weights(j);
        ahead = load_rows(0u);
        store_rows(ahead, 0u);
        __syncthreads();
#pragma unroll 1
        for (uint32_t k = 0; k < kSteps; k += 4u) {
            step(k, std::integral_constant<uint32_t, 0>{});
            step(k + 1u, std::integral_constant<uint32_t, 1>{});
            step(k + 2u, std::integral_constant<uint32_t, 2>{});
            step(k + 3u, std::integral_constant<uint32_t, 3>{});
        }
        if constexpr (F::kPerChannel) {
            const float scale = kBf16 ? bf16_to_f32(ring[0].s) : f16_to_f32(ring[0].s);
#pragma unroll
            for (uint32_t t = 0; t < kNt; ++t)
#pragma unroll
                for (uint32_t i = 0; i < 16u; ++i) y[t][i] = static_cast<float>(acc[t][i]) * scale;
        }

        // D lane (h, c): column c, rows 8 (i/4) + 4h + i%4 of each tile
        if constexpr (kGateUp) {
            // lanes 0-15 of a half hold a channel's gate values, lanes 16-31
            // its up values: exchanging two elements' halves leaves every
            // lane one element's gate and up
            uint16_t* mid = static_cast<uint16_t*>(out);
            const uint32_t channel = (slot0 >> 1) * 16u + n;
            const uint32_t odd = (lane >> 4) & 1u;
#pragma unroll
            for (uint32_t t = 0; t < kNt; ++t) {
                uint32_t silu_word[8];
                float up_value[8];
#pragma unroll
                for (uint32_t i = 0; i < 16u; i += 2u) {
                    const uint32_t r = 32u * t + 8u * (i / 4u) + 4u * h + i % 4u + odd;
                    const auto pair = __builtin_amdgcn_permlane16_swap(
                        __float_as_uint(y[t][i]), __float_as_uint(y[t][i + 1u]), false, false);
                    const float st = row_info[r < rows ? r : 0u].x;
                    up_value[i / 2u] = bf16_round(__uint_as_float(pair[1]) * st);
                    silu_word[i / 2u] = kSiluTable[f32_to_bf16(__uint_as_float(pair[0]) * st)];
                }
#pragma unroll
                for (uint32_t i = 0; i < 16u; i += 2u) {
                    const uint32_t r = 32u * t + 8u * (i / 4u) + 4u * h + i % 4u + odd;
                    if (r >= rows) continue;
                    const float hv = bf16_round(__uint_as_float(silu_word[i / 2u]) * up_value[i / 2u]);
                    mid[static_cast<size_t>(p0 + r) * kInter + channel] = static_cast<uint16_t>(
                        bf16_canonical_nan(f32_to_bf16(hv * row_info[r].y)));
                }
            }
        } else {
            float* route = static_cast<float*>(out) + slot0 * 16u + c;
#pragma unroll
            for (uint32_t t = 0; t < kNt; ++t)
#pragma unroll
                for (uint32_t i = 0; i < 16u; ++i) {
                    const uint32_t r = 32u * t + 8u * (i / 4u) + 4u * h + i % 4u;
                    if (r >= rows) continue;
                    store_route_output(route + static_cast<size_t>(p0 + r) * kHidden,
                                       y[t][i] * row_info[r].x);
                }
        }
    };
    if (rows > 32u)
        run(std::integral_constant<uint32_t, 2>{});
    else
        run(std::integral_constant<uint32_t, 1>{});
}

}  // namespace

uint32_t wide_chunks(uint32_t tokens) {
    return (routes_v1(tokens) + kWideChunkRoutes - 1u) / kWideChunkRoutes;
}

namespace {

template <uint32_t kChunkRoutes>
hipError_t build_wide_plan(const int32_t* ids, uint32_t tokens, const q38m_route_plan_v1& plan,
                           uint32_t* chunk_counts, hipStream_t stream) {
    const uint32_t routes = routes_v1(tokens);
    const uint32_t chunks = (routes + kChunkRoutes - 1u) / kChunkRoutes;
    wide_count_kernel<kChunkRoutes><<<chunks, 256, 0, stream>>>(ids, routes, chunk_counts);
    wide_scan_kernel<<<1, 512, 0, stream>>>(chunk_counts, chunks, tokens, plan,
                                            max_tasks_wide(tokens));
    wide_scatter_kernel<kChunkRoutes><<<chunks, 64, 0, stream>>>(ids, routes, chunk_counts, plan);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_build_wide_plan(const int32_t* ids, uint32_t tokens,
                                  const q38m_route_plan_v1& plan, uint32_t* chunk_counts,
                                  hipStream_t stream) {
    return build_wide_plan<kWideChunkRoutes>(ids, tokens, plan, chunk_counts, stream);
}

// The step's plan cuts the routes into shorter chunks where there are few of
// them.  The scatter kernel walks a chunk in serial rounds of 64 routes, so
// its time is the chunk's length (2048 routes: 9.2 us at any token count,
// 1024: 5.8-6.4, 512: 3.6); the scan reads two batches of 32 chunk counts at
// once and takes a round trip more for each further batch (15 us at 160
// chunks), hence the shortest chunk that leaves at most 64.  Step with
// 2048-route chunks -> this rule: 600 tokens 240.5 -> 234.4 us, 1,500 tokens
// W8 g128 343.0 -> 338.5 us, 4,096 tokens W4/W8 512.0 -> 507.6 us; 6,001
// tokens within the runs' difference.
hipError_t launch_step_wide_plan(const int32_t* ids, uint32_t tokens,
                                 const q38m_route_plan_v1& plan, uint32_t* chunk_counts,
                                 hipStream_t stream) {
    constexpr uint32_t kChunks = 64;
    const uint32_t routes = routes_v1(tokens);
    if (routes <= kChunks * 512u)
        return build_wide_plan<512>(ids, tokens, plan, chunk_counts, stream);
    if (routes <= kChunks * 1024u)
        return build_wide_plan<1024>(ids, tokens, plan, chunk_counts, stream);
    return build_wide_plan<2048>(ids, tokens, plan, chunk_counts, stream);
}

namespace {

template <uint32_t kBits, uint32_t kGroup, bool kBf16>
void launch_gate_up_i8(const q38m_expert_weights_v1& w, const int8_t* xq, const float* xs,
                       const uint32_t* packed, const float* route_weights, const TaskSlots& t,
                       uint16_t* mid, hipStream_t stream) {
    using F = WideI8<kBits, kGroup, true>;
    const uint32_t grid = placed_workgroups(t.count, F::kSlices * F::kHalves);
    wide_i8_kernel<kBits, kGroup, kBf16, true><<<grid, 256, 0, stream>>>(
        static_cast<const uint4*>(w.data), static_cast<const uint16_t*>(w.scales), xq, xs, packed,
        route_weights, TaskSlots{t.tasks, nullptr, t.count}, mid);
}

template <uint32_t kBits, uint32_t kGroup, bool kBf16>
void launch_down_i8(const q38m_expert_weights_v1& w, const int8_t* mid_q, const float* mid_s,
                    const TaskSlots& t, float* route_output, hipStream_t stream) {
    using F = WideI8<kBits, kGroup, false>;
    const uint32_t grid = placed_workgroups(t.count, F::kSlices * F::kHalves);
    wide_i8_kernel<kBits, kGroup, kBf16, false><<<grid, 256, 0, stream>>>(
        static_cast<const uint4*>(w.data), static_cast<const uint16_t*>(w.scales), mid_q, mid_s,
        nullptr, nullptr, TaskSlots{t.tasks, nullptr, t.count}, route_output);
}

template <bool kBf16>
hipError_t launch_gate_up_wide_dtype(const q38m_expert_weights_v1& w, const int8_t* xq,
                                     const float* xs, const uint32_t* packed,
                                     const float* route_weights, const TaskSlots& t,
                                     uint16_t* mid, hipStream_t stream) {
    const uint32_t key = (w.format == Q38M_FORMAT_W8_SYM ? 8000u : 4000u) + w.group_size;
    switch (key) {
        case 4032u: {
            // fp16 MFMA form: 8 channel pairs (256 rows of gate/up) per workgroup
            const uint32_t grid = placed_workgroups(t.count, kInter / 16u / 8u);
            gate_up_w4g32_f16_kernel<kHidden, kInter, kBf16><<<grid, 512, 0, stream>>>(
                static_cast<const uint4*>(w.data), static_cast<const uint16_t*>(w.scales), xq, xs,
                packed, route_weights, t, mid);
            break;
        }
        case 4064u: launch_gate_up_i8<4, 64, kBf16>(w, xq, xs, packed, route_weights, t, mid, stream); break;
        case 4128u: launch_gate_up_i8<4, 128, kBf16>(w, xq, xs, packed, route_weights, t, mid, stream); break;
        case 8000u: launch_gate_up_i8<8, 0, kBf16>(w, xq, xs, packed, route_weights, t, mid, stream); break;
        case 8064u: launch_gate_up_i8<8, 64, kBf16>(w, xq, xs, packed, route_weights, t, mid, stream); break;
        case 8128u: launch_gate_up_i8<8, 128, kBf16>(w, xq, xs, packed, route_weights, t, mid, stream); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <bool kBf16>
hipError_t launch_down_wide_dtype(const q38m_expert_weights_v1& w, const int8_t* mid_q,
                                  const float* mid_s, const TaskSlots& t, float* out,
                                  hipStream_t stream) {
    const uint32_t key = (w.format == Q38M_FORMAT_W8_SYM ? 8000u : 4000u) + w.group_size;
    switch (key) {
        case 4032u: {
            // fp16 MFMA form: 16 output tiles per 8-wave workgroup
            const uint32_t grid = placed_workgroups(t.count, kHidden / 16u / 16u);
            down_w4g32_f16_kernel<kHidden, kInter, kBf16><<<grid, 512, 0, stream>>>(
                static_cast<const uint4*>(w.data), static_cast<const uint16_t*>(w.scales), mid_q,
                mid_s, t, out);
            break;
        }
        case 4064u: launch_down_i8<4, 64, kBf16>(w, mid_q, mid_s, t, out, stream); break;
        case 4128u: launch_down_i8<4, 128, kBf16>(w, mid_q, mid_s, t, out, stream); break;
        case 8000u: {
            // per channel: four tiles per wave
            constexpr uint32_t kWaves = 8, kTilesPerWave = 4;
            const uint32_t grid = placed_workgroups(t.count, kHidden / 16u / (kWaves * kTilesPerWave));
            down_w8_wide_kernel<kHidden, kInter, kWaves, kTilesPerWave, kBf16>
                <<<grid, kWaves * 64u, 0, stream>>>(static_cast<const uint4*>(w.data),
                                                    static_cast<const uint16_t*>(w.scales), mid_q,
                                                    mid_s, t, out);
            break;
        }
        case 8064u: launch_down_i8<8, 64, kBf16>(w, mid_q, mid_s, t, out, stream); break;
        case 8128u: launch_down_i8<8, 128, kBf16>(w, mid_q, mid_s, t, out, stream); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_gate_up_wide(const q38m_expert_weights_v1& w, const int8_t* xq, const float* xs,
                               const uint32_t* packed, const float* route_weights,
                               const q38m_task_v1* tasks, const uint32_t* live_tasks,
                               uint32_t task_count, uint16_t* weighted_mid,
                               hipStream_t stream) {
    const TaskSlots t{tasks, task_count > kBlockedSlots ? live_tasks : nullptr, task_count};
    return w.scale_dtype == Q38M_SCALE_BF16
               ? launch_gate_up_wide_dtype<true>(w, xq, xs, packed, route_weights, t,
                                                 weighted_mid, stream)
               : launch_gate_up_wide_dtype<false>(w, xq, xs, packed, route_weights, t,
                                                  weighted_mid, stream);
}

hipError_t launch_down_wide(const q38m_expert_weights_v1& w, const int8_t* mid_q,
                            const float* mid_s, const q38m_task_v1* tasks,
                            const uint32_t* live_tasks, uint32_t task_count,
                            float* route_output, hipStream_t stream) {
    const TaskSlots t{tasks, task_count > kBlockedSlots ? live_tasks : nullptr, task_count};
    return w.scale_dtype == Q38M_SCALE_BF16
               ? launch_down_wide_dtype<true>(w, mid_q, mid_s, t, route_output, stream)
               : launch_down_wide_dtype<false>(w, mid_q, mid_s, t, route_output, stream);
}

}  // namespace q38m
