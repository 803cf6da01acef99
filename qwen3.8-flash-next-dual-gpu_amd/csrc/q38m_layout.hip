// Device weight layout conversion (the load-time re-tiling of
// cuda/cuda_weights.cu:229-285, for this build's MFMA16 layout),
// deterministic synthetic data, and kernel-level self checks.
#include "q38m_device.h"
#include "q38m_internal.h"
#include "q38m_select.h"

#include <type_traits>

namespace q38m {
namespace {

// Slot -> row tile of the quad-major W4 layouts: identity, or, paired, tile
// s/2 of the first half and tile s/2 of the second half alternating.
__device__ __forceinline__ uint32_t slot_tile(uint32_t slot, uint32_t row_tiles, bool paired) {
    return paired ? (slot >> 1) + (slot & 1u) * (row_tiles >> 1) : slot;
}

// W4 row-major [E][R][K/2] -> MFMA16 [E][K/128][slot][64][4 dwords], data and
// scale words.  Output dword (e, kq, slot, lane=(q,n), j) covers row
// 16*tile(slot)+n, group g=4kq+j, k0 = 32g+8q: byte i = nib(k0+i) |
// nib(k0+4+i) << 4; the source dword at k0/2 holds nibbles k0..k0+7 in order.
// Scales [E][R][K/g] -> [E][K/128][slot][16][128/g] (g = 32, 64, 128:
// kPerQuad = 4, 2, 1 words per row and quad).
//
// What bounds it is memory: a workgroup moves one row tile of up to 16 quads
// through LDS, so that it reads whole row pieces (1 KB) and writes whole slots
// (1 KB); reading each output's four dwords straight from the 16 rows took
// 49.8 us for 64 experts of gate/up (134 MB) and a second launch for their
// scales 16 us, this kernel 23.4 us.  LDS row n starts 4 banks after row n-1,
// which puts the 64 lanes' gather (n rows, q) on distinct banks.
constexpr uint32_t kRepackQuads = 16;

template <uint32_t kPerQuad>
__global__ __launch_bounds__(256) void repack_w4_kernel(const uint4* __restrict__ src,
                                                        uint4* __restrict__ dst,
                                                        const uint16_t* __restrict__ src_scales,
                                                        uint16_t* __restrict__ dst_scales,
                                                        uint32_t rows, uint32_t cols, bool paired) {
    constexpr uint32_t kPitch = kRepackQuads * 16u + 4u;  // dwords
    __shared__ __align__(16) uint32_t tile[16u * kPitch];
    const uint32_t quads = cols / 128u, row_tiles = rows / 16u;
    const uint32_t slot = blockIdx.x % row_tiles;
    const uint64_t e = blockIdx.x / row_tiles;
    const uint32_t kq0 = blockIdx.y * kRepackQuads;
    const uint32_t here = min(quads - kq0, kRepackQuads);  // quads of this workgroup
    const uint32_t row0 = slot_tile(slot, row_tiles, paired) * 16u;
    const uint32_t pieces = here * 4u;  // 16-byte pieces of a row here
    for (uint32_t i = threadIdx.x; i < 16u * pieces; i += 256u) {
        const uint32_t n = i / pieces, c = i % pieces;
        const uint4 v = src[(e * rows + row0 + n) * (cols / 32u) + kq0 * 4u + c];
        *reinterpret_cast<uint4*>(&tile[n * kPitch + 4u * c]) = v;
    }
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63u, n = lane & 15u, q = lane >> 4;
    for (uint32_t k = threadIdx.x >> 6; k < here; k += 4u) {
        uint32_t out[4];
#pragma unroll
        for (uint32_t j = 0; j < 4u; ++j) {
            const uint32_t c = tile[n * kPitch + 16u * k + 4u * j + q];
            uint32_t lo = (c & 0xffu) | ((c & 0xff00u) << 8);          // nibbles 0-1, 2-3
            uint32_t hi = ((c >> 16) & 0xffu) | ((c >> 24) << 16);     // nibbles 4-5, 6-7
            lo = (lo | (lo << 4)) & 0x0f0f0f0fu;
            hi = (hi | (hi << 4)) & 0x0f0f0f0fu;
            out[j] = lo | (hi << 4);
        }
        dst[((e * quads + kq0 + k) * row_tiles + slot) * 64u + lane] =
            make_uint4(out[0], out[1], out[2], out[3]);
    }
    for (uint32_t i = threadIdx.x; i < 16u * here; i += 256u) {
        const uint32_t k = i / 16u, r = i % 16u;
        const uint64_t from = ((e * rows + row0 + r) * quads + kq0 + k) * kPerQuad;
        const uint64_t to = (((e * quads + kq0 + k) * row_tiles + slot) * 16u + r) * kPerQuad;
#pragma unroll
        for (uint32_t j = 0; j < kPerQuad; ++j) dst_scales[to + j] = src_scales[from + j];
    }
}

// W8 row-major [E][R][K] -> MFMA16 [E][R/16][K/64][64][16 B]; lane (q,n)
// holds row 16rt+n, columns 64kb+16q .. +15.
__global__ void repack_w8_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst,
                                 uint32_t rows, uint32_t cols, uint64_t total,
                                 const uint16_t* __restrict__ src_scales,
                                 uint16_t* __restrict__ dst_scales, uint64_t scales) {
    const uint64_t o = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (o >= total) {
        // the workgroups past the data copy the scales (artifact order kept)
        const uint64_t i = o - (total + blockDim.x - 1u) / blockDim.x * blockDim.x;
        if (o >= (total + blockDim.x - 1u) / blockDim.x * blockDim.x && i < scales)
            dst_scales[i] = src_scales[i];
        return;
    }
    const uint32_t blocks = cols / 64u;
    const uint32_t row_tiles = rows / 16u;
    const uint32_t lane = static_cast<uint32_t>(o & 63u);
    const uint64_t block = o >> 6;
    const uint32_t kb = static_cast<uint32_t>(block % blocks);
    const uint64_t tmp = block / blocks;
    const uint32_t rt = static_cast<uint32_t>(tmp % row_tiles);
    const uint64_t e = tmp / row_tiles;
    const uint32_t n = lane & 15u, q = lane >> 4;
    dst[o] = src[((e * rows + rt * 16u + n) * cols + kb * 64u + q * 16u) / 16u];
}

// W8 gate/up row-major [E][R][K] -> paired K-block-major MFMA16
// [E][K/64][slot][64][16 B]: for block kb every slot (1 KiB) is adjacent,
// slot s holding row tile s/2 + (s%2)*R/32 (the gate tile of channel block
// p next to its up tile), lane (q,n) row 16t+n, columns 64kb+16q .. +15.
__global__ void repack_w8_paired_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst,
                                        uint32_t rows, uint32_t cols, uint64_t total,
                                        const uint16_t* __restrict__ src_scales,
                                        uint16_t* __restrict__ dst_scales, uint64_t scales) {
    const uint64_t o = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (o >= total) {
        // the workgroups past the data copy the scales (artifact order kept)
        const uint64_t i = o - (total + blockDim.x - 1u) / blockDim.x * blockDim.x;
        if (o >= (total + blockDim.x - 1u) / blockDim.x * blockDim.x && i < scales)
            dst_scales[i] = src_scales[i];
        return;
    }
    const uint32_t blocks = cols / 64u;
    const uint32_t row_tiles = rows / 16u;
    const uint32_t lane = static_cast<uint32_t>(o & 63u);
    const uint64_t unit = o >> 6;
    const uint32_t slot = static_cast<uint32_t>(unit % row_tiles);
    const uint64_t tmp = unit / row_tiles;
    const uint32_t kb = static_cast<uint32_t>(tmp % blocks);
    const uint64_t e = tmp / blocks;
    const uint32_t n = lane & 15u, q = lane >> 4;
    const uint32_t row = slot_tile(slot, row_tiles, true) * 16u + n;
    dst[o] = src[((e * rows + row) * cols + kb * 64u + q * 16u) / 16u];
}

// ---------------------------------------------------------------------------
// Weight quantiser (tools/q38_artifact_compiler.py:193-253, quantize_groupwise):
// per group s = max|w| / qmax (qmax 7 for W4, 127 for W8), s == 0 -> 1,
// q = clamp(rint(w / s), +-qmax); W4 packs column 2i in the low nibble.
// Scales are stored as fp16 (round to nearest even, subnormals kept) or,
// as the reference does (f32_to_bf16_rne, :232), as RNE bf16; q always
// comes from the fp32 s.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t f32_to_f16_bits(float v) {
    return static_cast<uint32_t>(__builtin_bit_cast(uint16_t, static_cast<_Float16>(v)));
}

// The integers of eight bf16 values (four words) of a group with scale s,
// r = RN(1/s), in the low kBits bits of each byte of (even values, odd
// values).  Scales in [2^-120, FLT_MAX] take no division per value: one
// Markstein correction step rounds like it (tests/weight_quotient_check.c walks
// every bf16 pair of the lowest, middle and largest binades of maxima, between
// which powers of two scale exactly), and adding 1.5 * 2^23 rounds to the integer
// in the low bits; a NaN quotient clamps to -qmax on both paths.  (With
// an IEEE division and a half-rate conversion per value the kernels moved
// 3.5-4.4 TB/s, now 5.9-6.2.)
template <uint32_t kBits>
__device__ __forceinline__ uint2 quant_weights(const uint32_t (&w)[4], float s, float r, bool fast) {
    constexpr float kMax = kBits == 4u ? 7.0f : 127.0f;
    uint32_t bits[8];
#pragma unroll
    for (uint32_t i = 0; i < 8u; ++i) {
        const float x = __uint_as_float(i & 1u ? w[i / 2u] & 0xffff0000u : w[i / 2u] << 16);
        float quotient;
        if (fast) {  // uniform
            const float q0 = x * r;
            quotient = __builtin_fmaf(__builtin_fmaf(-q0, s, x), r, q0);
        } else {
            quotient = __builtin_rintf(x / s);
        }
        bits[i] = __float_as_uint(fminf(fmaxf(quotient, -kMax), kMax) + 12582912.0f);
    }
    // byte 0 of four words: v_perm selectors 0 and 4 pick the two operands'
    auto bytes = [](uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
        const uint32_t lo = __builtin_amdgcn_perm(b, a, 0x0c0c0400u);
        const uint32_t hi = __builtin_amdgcn_perm(d, c, 0x04000c0cu);
        return lo | hi;
    };
    return make_uint2(bytes(bits[0], bits[2], bits[4], bits[6]),
                      bytes(bits[1], bits[3], bits[5], bits[7]));
}

// eight W4 values: one byte per pair, the even column in the low nibble
__device__ __forceinline__ uint32_t pack_w4(uint2 v) {
    return (v.x & 0x0f0f0f0fu) | ((v.y & 0x0f0f0f0fu) << 4);
}
// eight W8 values in column order
__device__ __forceinline__ uint2 pack_w8(uint2 v) {
    return make_uint2(__builtin_amdgcn_perm(v.y, v.x, 0x05010400u),
                      __builtin_amdgcn_perm(v.y, v.x, 0x07030602u));
}

__device__ __forceinline__ float absmax8(const uint32_t (&w)[4]) {
    float amax = 0.0f;
#pragma unroll
    for (uint32_t i = 0; i < 4u; ++i) {
        amax = fmaxf(amax, fabsf(__uint_as_float(w[i] << 16)));
        amax = fmaxf(amax, fabsf(__uint_as_float(w[i] & 0xffff0000u)));
    }
    return amax;
}

// s = amax / qmax, 0 -> 1, and whether every lane's scale takes the fast path
struct WeightScale {
    float s, r;
    bool fast;
};
template <uint32_t kBits>
__device__ __forceinline__ WeightScale weight_scale(float amax) {
    float s = amax / (kBits == 4u ? 7.0f : 127.0f);
    if (s == 0.0f) s = 1.0f;
    return WeightScale{s, 1.0f / s, __all(s >= 0x1p-120f && s <= 0x1.fffffep+127f) != 0};
}
__device__ __forceinline__ uint16_t scale_word(float s, bool bf16) {
    return static_cast<uint16_t>(bf16 ? f32_to_bf16(s) : f32_to_f16_bits(s));
}

// Groups of kGroup columns (contiguous in memory): kGroup/8 neighbouring lanes
// per group, 8 values a lane, kVec pieces per thread 256 lanes apart, so every
// load and store instruction covers whole lines (one thread per group read 64
// bytes a lane; 64 experts of gate/up in W4 groups of 32, 343 MB: 77.1 us, now
// 55.3).
// The absmax crosses the group's lanes by DPP inside a row of 16, or the wave
// for whole rows of 512 columns (W8 per output channel; 64 experts of down, 202
// MB: 58.6 us with a wave per row and two passes over it, now 33.8).
template <uint32_t kBits, uint32_t kGroup>
__global__ __launch_bounds__(256) void quantize_weights_group_kernel(
    const uint4* __restrict__ src, uint64_t vectors, uint8_t* __restrict__ data,
    uint16_t* __restrict__ scales, bool scale_bf16) {
    constexpr uint32_t kVec = 4, kLanes = kGroup / 8u;
    const uint64_t v0 = static_cast<uint64_t>(blockIdx.x) * (kVec * 256u) + threadIdx.x;
    uint4 v[kVec];
#pragma unroll
    for (uint32_t i = 0; i < kVec; ++i) {
        const uint64_t at = v0 + i * 256u;
        v[i] = load_stream(src + (at < vectors ? at : vectors - 1u));
    }
#pragma unroll
    for (uint32_t i = 0; i < kVec; ++i) {
        const uint64_t at = v0 + i * 256u;
        const uint32_t w[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
        auto across = [](float x, auto control) {
            return fmaxf(x, __int_as_float(__builtin_amdgcn_mov_dpp(
                                __float_as_int(x), decltype(control)::value, 0xf, 0xf, false)));
        };
        float amax = absmax8(w);
        if constexpr (kLanes == 64u) {
            amax = wave_max_f32(amax);
        } else {
            amax = across(amax, std::integral_constant<int, 0xB1>{});  // quad_perm [1,0,3,2]
            amax = across(amax, std::integral_constant<int, 0x4E>{});  // quad_perm [2,3,0,1]
            if constexpr (kLanes >= 8u) amax = across(amax, std::integral_constant<int, 0x141>{});   // row_half_mirror
            if constexpr (kLanes >= 16u) amax = across(amax, std::integral_constant<int, 0x140>{});  // row_mirror
        }
        const WeightScale ws = weight_scale<kBits>(amax);
        const uint2 q = quant_weights<kBits>(w, ws.s, ws.r, ws.fast);
        if (at >= vectors) continue;
        if (at % kLanes == 0u) scales[at / kLanes] = scale_word(ws.s, scale_bf16);
        if constexpr (kBits == 4u)
            reinterpret_cast<uint32_t*>(data)[at] = pack_w4(q);
        else
            reinterpret_cast<uint2*>(data)[at] = pack_w8(q);
    }
}

// W8 per output channel, rows of 512 kChunks columns: one wave per row, its
// values in registers between the absmax and the quotients.
template <uint32_t kChunks>
__global__ __launch_bounds__(256) void quantize_weights_row_w8_kernel(
    const uint4* __restrict__ src, uint64_t rows, uint8_t* __restrict__ data,
    uint16_t* __restrict__ scales, bool scale_bf16) {
    const uint64_t row = static_cast<uint64_t>(blockIdx.x) * 4u + (threadIdx.x >> 6);
    if (row >= rows) return;  // uniform per wave
    const uint32_t lane = threadIdx.x & 63u;
    uint4 v[kChunks];
#pragma unroll
    for (uint32_t c = 0; c < kChunks; ++c)
        v[c] = load_stream(src + row * (64u * kChunks) + 64u * c + lane);
    float amax = 0.0f;
#pragma unroll
    for (uint32_t c = 0; c < kChunks; ++c) {
        const uint32_t w[4] = {v[c].x, v[c].y, v[c].z, v[c].w};
        amax = fmaxf(amax, absmax8(w));
    }
    const WeightScale ws = weight_scale<8u>(wave_max_f32(amax));
    if (lane == 0u) scales[row] = scale_word(ws.s, scale_bf16);
#pragma unroll
    for (uint32_t c = 0; c < kChunks; ++c) {
        const uint32_t w[4] = {v[c].x, v[c].y, v[c].z, v[c].w};
        reinterpret_cast<uint2*>(data)[row * (64u * kChunks) + 64u * c + lane] =
            pack_w8(quant_weights<8u>(w, ws.s, ws.r, ws.fast));
    }
}

// W8 per output channel, other widths (columns % 512 == 0): one wave per row,
// two passes.
__global__ __launch_bounds__(256) void quantize_weights_wide_row_w8_kernel(
    const uint4* __restrict__ src, uint64_t rows, uint32_t cols, uint8_t* __restrict__ data,
    uint16_t* __restrict__ scales, bool scale_bf16) {
    const uint64_t row = static_cast<uint64_t>(blockIdx.x) * 4u + (threadIdx.x >> 6);
    if (row >= rows) return;
    const uint32_t lane = threadIdx.x & 63u;
    const uint4* r = src + row * (cols / 8u);
    float amax = 0.0f;
    for (uint32_t c = lane; c < cols / 8u; c += 64u) {
        const uint4 v = r[c];
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        amax = fmaxf(amax, absmax8(w));
    }
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) amax = fmaxf(amax, __shfl_xor(amax, offset, 64));
    const WeightScale ws = weight_scale<8u>(amax);
    if (lane == 0u) scales[row] = scale_word(ws.s, scale_bf16);
    uint2* out = reinterpret_cast<uint2*>(data) + row * (cols / 8u);
    for (uint32_t c = lane; c < cols / 8u; c += 64u) {
        const uint4 v = r[c];
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        out[c] = pack_w8(quant_weights<8u>(w, ws.s, ws.r, ws.fast));
    }
}

// Synthetic data, one element (or one packed W4 byte) per thread, grid-
// stride so any count fits the grid.
__global__ void synth_kernel(uint32_t kind, uint64_t base, uint64_t count, float sigma,
                             int32_t lo, int32_t hi, const float* __restrict__ bias,
                             uint32_t bias_len, void* __restrict__ out) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < count;
         i += stride) {
        switch (kind) {
            case Q38M_SYNTH_NORMAL_F32: {
                float v = normal_at(base, i) * sigma;
                if (bias) v = v + bias[i % bias_len];
                static_cast<float*>(out)[i] = v;
                break;
            }
            case Q38M_SYNTH_NORMAL_BF16:
                static_cast<uint16_t*>(out)[i] =
                    static_cast<uint16_t>(f32_to_bf16(normal_at(base, i) * sigma));
                break;
            case Q38M_SYNTH_ABS_NORMAL_F16:
                static_cast<uint16_t*>(out)[i] =
                    static_cast<uint16_t>(f32_to_f16(fabsf(normal_at(base, i) * sigma)));
                break;
            case Q38M_SYNTH_UNIFORM_W4: {
                const int low = uniform_at(base, 2u * i, lo, hi);
                const int high = uniform_at(base, 2u * i + 1u, lo, hi);
                static_cast<uint8_t*>(out)[i] = static_cast<uint8_t>(
                    (static_cast<uint32_t>(low) & 0xfu) | ((static_cast<uint32_t>(high) & 0xfu) << 4));
                break;
            }
            case Q38M_SYNTH_UNIFORM_I8:
                static_cast<int8_t*>(out)[i] = static_cast<int8_t>(uniform_at(base, i, lo, hi));
                break;
            default:
                break;
        }
    }
}

inline uint32_t blocks_for(uint64_t total, uint32_t threads) {
    return static_cast<uint32_t>((total + threads - 1u) / threads);
}

}  // namespace

hipError_t launch_repack(const q38m_expert_weights_v1& src,
                         const q38m_expert_weights_v1& dst, hipStream_t stream) {
    const uint64_t elements = static_cast<uint64_t>(src.experts) * src.rows * src.columns;
    if (src.format == Q38M_FORMAT_W4_SYM) {
        const bool paired = dst.layout == Q38M_LAYOUT_MFMA16_PAIRED;
        const dim3 grid(static_cast<uint32_t>(static_cast<uint64_t>(src.experts) * (src.rows / 16u)),
                        (src.columns / 128u + kRepackQuads - 1u) / kRepackQuads);
        const uint4* from = static_cast<const uint4*>(src.data);
        uint4* to = static_cast<uint4*>(const_cast<void*>(dst.data));
        const uint16_t* from_scales = static_cast<const uint16_t*>(src.scales);
        uint16_t* to_scales = static_cast<uint16_t*>(const_cast<void*>(dst.scales));
#define Q38M_REPACK(per_quad)                                                                  \
    repack_w4_kernel<per_quad><<<grid, 256, 0, stream>>>(from, to, from_scales, to_scales,     \
                                                         src.rows, src.columns, paired)
        if (src.group_size == 32u) Q38M_REPACK(4u);
        else if (src.group_size == 64u) Q38M_REPACK(2u);
        else Q38M_REPACK(1u);
#undef Q38M_REPACK
    } else {
        const uint64_t vectors = elements / 16u;
        // W8 scales keep the artifact order (per channel or [E][R][K/g])
        const uint64_t scales = src.group_size ? elements / src.group_size
                                               : static_cast<uint64_t>(src.experts) * src.rows;
        // (no columns: an empty grid, refused by the launch)
        const uint32_t grid = vectors ? blocks_for(vectors, 256) + blocks_for(scales, 256) : 0u;
        auto* kernel = dst.layout == Q38M_LAYOUT_MFMA16_PAIRED ? repack_w8_paired_kernel
                                                               : repack_w8_kernel;
        kernel<<<grid, 256, 0, stream>>>(
            static_cast<const uint4*>(src.data), static_cast<uint4*>(const_cast<void*>(dst.data)),
            src.rows, src.columns, vectors, static_cast<const uint16_t*>(src.scales),
            static_cast<uint16_t*>(const_cast<void*>(dst.scales)), scales);
    }
    return hipGetLastError();
}

hipError_t launch_quantize_weights(const uint16_t* src, const q38m_expert_weights_v1& dst,
                                  hipStream_t stream) {
    const uint64_t rows = static_cast<uint64_t>(dst.experts) * dst.rows;
    uint8_t* data = static_cast<uint8_t*>(const_cast<void*>(dst.data));
    uint16_t* scales = static_cast<uint16_t*>(const_cast<void*>(dst.scales));
    const uint4* s4 = reinterpret_cast<const uint4*>(src);
    const uint32_t g = dst.group_size;
    const bool w4 = dst.format == Q38M_FORMAT_W4_SYM;
    const bool bf16 = dst.scale_dtype == Q38M_SCALE_BF16;
    if (g == 0u) {
        if (dst.columns == 512u)
            quantize_weights_group_kernel<8u, 512u>
                <<<blocks_for(rows * 64u, 1024), 256, 0, stream>>>(s4, rows * 64u, data, scales, bf16);
        else if (dst.columns == 2048u)
            quantize_weights_row_w8_kernel<4>
                <<<blocks_for(rows, 4), 256, 0, stream>>>(s4, rows, data, scales, bf16);
        else
            quantize_weights_wide_row_w8_kernel<<<blocks_for(rows, 4), 256, 0, stream>>>(
                s4, rows, dst.columns, data, scales, bf16);
        return hipGetLastError();
    }
    const uint64_t vectors = rows * dst.columns / 8u;
    const uint32_t grid = blocks_for(vectors, 1024);
#define Q38M_QUANT(BITS, G)                                                                    \
    quantize_weights_group_kernel<BITS, G><<<grid, 256, 0, stream>>>(s4, vectors, data, scales, \
                                                                     bf16)
    if (w4 && g == 32u) Q38M_QUANT(4u, 32u);
    else if (w4 && g == 64u) Q38M_QUANT(4u, 64u);
    else if (w4) Q38M_QUANT(4u, 128u);
    else if (g == 32u) Q38M_QUANT(8u, 32u);
    else if (g == 64u) Q38M_QUANT(8u, 64u);
    else Q38M_QUANT(8u, 128u);
#undef Q38M_QUANT
    return hipGetLastError();
}

hipError_t launch_synth(uint32_t kind, uint64_t seed, uint64_t tag, uint64_t count,
                        float sigma, int32_t lo, int32_t hi, const float* bias,
                        uint32_t bias_len, void* out, hipStream_t stream) {
    const uint64_t items = kind == Q38M_SYNTH_UNIFORM_W4 ? count / 2u : count;
    const uint32_t blocks = static_cast<uint32_t>(
        items / 256u + 1u < 65536u ? items / 256u + 1u : 65536u);
    synth_kernel<<<blocks, 256, 0, stream>>>(kind, stream_base_host(seed, tag), items, sigma, lo,
                                             hi, bias, bias_len, out);
    return hipGetLastError();
}

}  // namespace q38m
