// tq4_rms.hip -- the vllm-ascend RMS + threshold codec (TurboQuantCodec<4>)
// and the baseline writer that applies it, on gfx950.
//
// Reference semantics (paths relative to the reference checkout):
//   codec      kernels/ops/turboquant/baseline/common/turboquant_codec_950.h
//                ApplyPi = signs, FWHT (strides 1..n/2, a+b | a-b), x inv_sqrt_len, signs  :115-151
//                scale = sqrt(sum y^2) * inv_sqrt_len + 1e-20                               :186-197
//                level = #{i : y * (-1/scale) + t_i has its sign bit set}                    :199-231
//                byte = (even level + 16 * odd level) - 128 as int8                         :234-248
//                dequantize: byte + 128 -> even / odd level -> centroid                     :251-285
//   writer     kernels/ops/turboquant/baseline/turboquant_paged_attention.cpp:98-246
//                (per token: every (plane, kv head) vector; rows at slot*H*(d/2) + h*(d/2);
//                 the slot's scale record [K scales, V scales, zeros to a multiple of 8];
//                 tokens with a slot outside [0, num_blocks * block_size) write nothing)
//   thresholds / centroids: codec_950.h:43-51,
//                tests/npu/bench/bench_turboquant_reshape_and_cache.cpp:55-61
//
// MI355X design: a vector is spread over 16 lanes of one wave row, d/16
// consecutive channels per lane (one 16-byte load of BF16 at d = 128), in the
// row lane order of the TQ4 writers (row_lane). The FWHT runs in registers
// below d/16 and as DPP-fed fused butterflies above (row_fmac_stage, same a+b
// / a-b bits); the sum of squares is a sequential per-lane sum and a 4-step
// tree over logical lanes. The level is one comparison: bins a quarter wide
// hold at most one threshold each (level_of). A row's d/2 packed bytes leave
// as one coalesced run (d/32 bytes per lane).
// Built with -ffp-contract=off: every FP32 operation is the one written, so the
// bits are those of the C oracle's restatement.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tq4_device.hpp"
#include "tq4_internal.hpp"

namespace tq4 {
namespace {

constexpr int kRmsThreads = 256;
constexpr int kRowLanes = 16;
constexpr float kRmsEps = 1e-20f;

// The positive thresholds t_8 .. t_14 (codec_950.h:45-49); t_7 = 0 and
// t_{14-i} = -t_i.
constexpr float kPos[7] = {0.2582216646707196f, 0.5224037090113789f, 0.7995497875097155f,
                           1.0992858269170722f, 1.4371387916845330f, 1.8435318062766393f,
                           2.4008033987632817f};
// The 16 centroids, level order (bench_turboquant_reshape_and_cache.cpp:55-61).
constexpr float kCentroids[16] = {
    -2.7325895709951710f, -2.0690172265313920f, -1.6180463860218863f, -1.2562311973471796f,
    -0.9423404564869651f, -0.6567591185324659f, -0.3880482994902919f, -0.1283950298511473f,
    0.1283950298511473f,  0.3880482994902919f,  0.6567591185324659f,  0.9423404564869651f,
    1.2562311973471796f,  1.6180463860218863f,  2.0690172265313920f,  2.7325895709951710f};

// sqrt(x) rounded to nearest even for x >= 0: v_sqrt_f32 is faithful (within
// one ulp), so the neighbour whose residual sign says the root lies beyond
// the midpoint replaces it; x below 2^-96 is scaled by 2^32 first (and the
// root back by 2^-16) so the residuals stay normal.
__device__ __forceinline__ float sqrt_rn(float x)
{
    const bool tiny = x < 0x1.0p-96f;
    const float xs = tiny ? x * 0x1.0p+32f : x;
    float s = __builtin_amdgcn_sqrtf(xs);
    const float dn = __uint_as_float(__float_as_uint(s) - 1u);
    const float up = __uint_as_float(__float_as_uint(s) + 1u);
    const float r_dn = __builtin_fmaf(-dn, s, xs);
    const float r_up = __builtin_fmaf(-up, s, xs);
    s = r_dn <= 0.0f ? dn : s;
    s = r_up > 0.0f ? up : s;
    // zero and +inf pass through unchanged (their neighbours are not roots)
    s = (xs == 0.0f || xs == __builtin_inff()) ? __builtin_amdgcn_sqrtf(xs) : s;
    return tiny ? s * 0x1.0p-16f : s;
}

// The level search by bins a quarter wide over the signed line: bin 0 is below
// -2.5, bin i = 1 .. 20 is [(i - 11)/4, (i - 10)/4), bin 21 is [2.5, inf]. The
// 15 thresholds lie more than a quarter apart and, but for t_7 = 0 (the first
// point of its bin), away from the bins' ends, so a bin holds at most one:
// #{i : t_i < z} = below + (inside < z) of z's bin, `below` counting the
// thresholds under the bin and `inside` its own (+inf when it has none).
struct LevelBin {
    float inside;
    uint32_t below;
};
constexpr int kLevelBins = 22;
constexpr float kInf = __builtin_inff();
constexpr LevelBin kBins[kLevelBins] = {
    {kInf, 0},     {-kPos[6], 0}, {kInf, 1},     {-kPos[5], 1}, {kInf, 2},     {-kPos[4], 2},
    {-kPos[3], 3}, {-kPos[2], 4}, {-kPos[1], 5}, {-kPos[0], 6}, {kInf, 7},     {0.0f, 7},
    {kPos[0], 8},  {kPos[1], 9},  {kPos[2], 10}, {kPos[3], 11}, {kPos[4], 12}, {kInf, 13},
    {kPos[5], 13}, {kInf, 14},    {kPos[6], 14}, {kInf, 15}};
static_assert((int)(kPos[0] * 4) == 1 && (int)(kPos[1] * 4) == 2 && (int)(kPos[2] * 4) == 3 &&
                  (int)(kPos[3] * 4) == 4 && (int)(kPos[4] * 4) == 5 &&
                  (int)(kPos[5] * 4) == 7 && (int)(kPos[6] * 4) == 9,
              "each threshold sits in the bin the table gives it");
static_assert(kPos[0] * 4 != 1 && kPos[1] * 4 != 2 && kPos[2] * 4 != 3 && kPos[3] * 4 != 4 &&
                  kPos[4] * 4 != 5 && kPos[5] * 4 != 7 && kPos[6] * 4 != 9,
              "no threshold but 0 on a bin boundary");

// The codec's level of z = y * (1/scale): #{i : t_i < z} (NaN -> 0). lut:
// kBins staged in LDS. The bin is the truncated 4z + 11, held within the table
// before the conversion (v_med3 of a NaN is the smaller bound); where that sum's rounding crosses a bin's end, no threshold
// lies between z and the end, so both bins give the same count.
__device__ __forceinline__ uint32_t level_of(float z, const LevelBin* lut)
{
    // 8 bytes an entry: the byte offset is the truncated 32z + 88, its low
    // bits dropped
    const uint32_t u = (uint32_t)__builtin_amdgcn_fmed3f(__builtin_fmaf(z, 32.0f, 88.0f), 0.0f,
                                                         (float)(8 * kLevelBins - 1));
    const LevelBin e = *(const LevelBin*)((const char*)lut + (u & ~7u));
    return e.below + (e.inside < z ? 1u : 0u);
}

// Sixteen (token, kv head) items per workgroup, both planes of an item on its
// 16 lanes: the two rows share the index arithmetic, the slot, the signs and
// the scale's square root and division. Bound by the vector ALU: the codec's
// arithmetic is about 240 instructions a row against 330 bytes of traffic at
// d = 128. 4096 BF16 tokens x 8 heads of 128, launches in a row from a graph:
// 11.4 us with one row a lane and bins of |z| (17 instructions a level), 9.1 with
// two rows and signed bins (6 and an LDS read), 8.2 with the shared scale and a
// multiplier for item / H; 1024 tokens 5.2 -> 4.4, 16384 35.8 -> 23.5 us (3.6
// TB/s). (Eager calls over fewer buffers, 4096 tokens: 10.4 -> 7.7.)
template <int D, int IN_BF16>
__global__ __launch_bounds__(kRmsThreads) void rms_writer(
    const uint16_t* __restrict__ key, const uint16_t* __restrict__ value,
    int8_t* __restrict__ key_cache, int8_t* __restrict__ value_cache,
    float* __restrict__ scale_cache, const int32_t* __restrict__ slots,
    const float* __restrict__ pi_signs, uint32_t tokens, uint32_t H, uint32_t h_magic,
    uint32_t h_shift, uint64_t slot_count, float inv_sqrt_len)
{
    constexpr int CPL = D / kRowLanes;
    const int lane = threadIdx.x & (kRowLanes - 1);
    const int l = row_lane(lane);  // logical lane: channels l*CPL ..
    // the level search's bins, staged before any lane leaves
    __shared__ LevelBin lut[kLevelBins];
    if (threadIdx.x < kLevelBins) lut[threadIdx.x] = kBins[threadIdx.x];
    __syncthreads();
    const uint64_t item = (uint64_t)blockIdx.x * (kRmsThreads / kRowLanes) + threadIdx.x / kRowLanes;
    const uint64_t items = (uint64_t)tokens * H;
    if (item >= items) return;
    // item / H by the launch's multiplier when every item is below 2^31 (a
    // uniform branch)
    const uint32_t t = items <= 0x7fffffffull
                           ? (uint32_t)(((uint64_t)(uint32_t)item * h_magic) >> h_shift)
                           : (uint32_t)(item / H);
    const uint32_t h = (uint32_t)(item - (uint64_t)t * H);
    const int32_t slot = slots[t];
    // the rows' channels l*CPL .. +CPL, and the signs
    uint32_t raw[2][CPL / 2];
    __builtin_memcpy(raw[0], key + item * D + l * CPL, CPL * 2);
    __builtin_memcpy(raw[1], value + item * D + l * CPL, CPL * 2);
    float sg[CPL];
#pragma unroll
    for (int j = 0; j < CPL; ++j) sg[j] = pi_signs[l * CPL + j];
    if (slot < 0 || (uint64_t)slot >= slot_count) return;  // a pad token or a slot past the pool

    // ApplyPi: signs, FWHT at strides 1 .. D/2, x inv_sqrt_len, signs (products:
    // any float is taken). The FWHT's cross-lane stages run on sign-tracked
    // values (row_fmac_stage): v holds sigma * y afterwards, sigma = row_sigma(l)
    float v[2][CPL];
#pragma unroll
    for (int j = 0; j < CPL; j += 2) {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const uint32_t w = raw[r][j / 2];
            if constexpr (IN_BF16) {
                v[r][j] = __uint_as_float(w << 16) * sg[j];
                v[r][j + 1] = __uint_as_float(w & 0xffff0000u) * sg[j + 1];
            } else {
                v[r][j] = (float)__builtin_bit_cast(_Float16, (uint16_t)w) * sg[j];
                v[r][j + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16)) * sg[j + 1];
            }
        }
    }
#pragma unroll
    for (int s = 1; s < D; s <<= 1) {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            if (s < CPL) {
#pragma unroll
                for (int j = 0; j < CPL; ++j) {
                    if (j & s) continue;
                    const float a = v[r][j];
                    const float b = v[r][j + s];
                    v[r][j] = b + a;
                    v[r][j + s] = a - b;
                }
            } else {
                const int k = __builtin_ctz(s / CPL);
                row_fmac_stage<CPL>(v[r], ((l >> k) & 1) ? -1.0f : 1.0f, k);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 2; ++r) {
#pragma unroll
        for (int j = 0; j < CPL; ++j) v[r][j] = (v[r][j] * inv_sqrt_len) * sg[j];
    }

    // scale = sqrt(sum y^2) * inv_sqrt_len + eps: per-lane sequential sum, then
    // the tree over logical lanes l ^ 1, l ^ 2, l ^ 4, l ^ 8 ((sigma y)^2 is
    // y^2 exactly). Even lanes then finish the key row, odd lanes the value row.
    float ss[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        ss[r] = v[r][0] * v[r][0];
#pragma unroll
        for (int j = 1; j < CPL; ++j) ss[r] = ss[r] + v[r][j] * v[r][j];
#pragma unroll
        for (int k = 0; k < 4; ++k) row_add1(ss[r], k);
    }
    const float scale = sqrt_rn((lane & 1) ? ss[1] : ss[0]) * inv_sqrt_len + kRmsEps;
    const uint32_t ssf = (2u * H + 7u) / 8u * 8u;
    float* rec = scale_cache + (uint64_t)slot * ssf;
    if (lane < 2) rec[lane * H + h] = scale;
    // sigma rides on the reciprocal: (sigma y) * (sigma r) rounds as y * r
    const int rcp = __float_as_int(__fdiv_rn(1.0f, scale));
    const float sigma = row_sigma(l);
    const float rcps[2] = {
        sigma * __int_as_float(__builtin_amdgcn_mov_dpp(rcp, 0xA0, 0xf, 0xf, true)),   // lanes 0,0,2,2
        sigma * __int_as_float(__builtin_amdgcn_mov_dpp(rcp, 0xF5, 0xf, 0xf, true))};  // lanes 1,1,3,3
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        // levels, packed (even | odd << 4) ^ 0x80 -- the -128 bias of the int8 byte
        uint32_t pk[CPL / 8 > 0 ? CPL / 8 : 1] = {};
#pragma unroll
        for (int j = 0; j < CPL; ++j) pk[j / 8] |= level_of(v[r][j] * rcps[r], lut) << (4 * (j % 8));
        int8_t* dst = (r == 0 ? key_cache : value_cache) + ((uint64_t)slot * H + h) * (D / 2) +
                      l * (CPL / 2);
        if constexpr (CPL == 4) {
            *(uint16_t*)dst = (uint16_t)(pk[0] ^ 0x8080u);
        } else if constexpr (CPL == 8) {
            *(uint32_t*)dst = pk[0] ^ 0x80808080u;
        } else {
            *(uint2*)dst = make_uint2(pk[0] ^ 0x80808080u, pk[1] ^ 0x80808080u);
        }
    }
    // the slot's scale record ends in at most 7 zeros, head 0's to write
    if (h == 0 && lane > 0 && 2u * H + lane - 1u < ssf) rec[2u * H + lane - 1u] = 0.0f;
}

// Dequantize4Bit: four packed bytes -> eight centroids per lane, grid-stride.
__global__ __launch_bounds__(kRmsThreads) void rms_dequant(const uint32_t* __restrict__ packed,
                                                           float4* __restrict__ out,
                                                           uint64_t words)
{
    __shared__ float cent[16];
    if (threadIdx.x < 16) cent[threadIdx.x] = kCentroids[threadIdx.x];
    __syncthreads();
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < words;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t w = packed[i] ^ 0x80808080u;
        float f[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) f[k] = cent[(w >> (4 * k)) & 15u];
        out[2 * i] = make_float4(f[0], f[1], f[2], f[3]);
        out[2 * i + 1] = make_float4(f[4], f[5], f[6], f[7]);
    }
}

__global__ void rms_dequant_tail(const uint8_t* __restrict__ packed, float* __restrict__ out,
                                 uint64_t first, uint64_t bytes)
{
    const uint64_t j = first + threadIdx.x;
    if (j >= bytes) return;
    const uint32_t v = packed[j] ^ 0x80u;
    out[2 * j] = kCentroids[v & 15u];
    out[2 * j + 1] = kCentroids[v >> 4];
}

template <int D>
hipError_t launch_rms_writer_t(hipStream_t stream, int in_bf16, const uint16_t* key,
                               const uint16_t* value, int8_t* kc, int8_t* vc, float* sc,
                               const int32_t* slots, const float* signs, uint32_t tokens,
                               uint32_t H, uint64_t slot_count, float isl)
{
    const uint64_t items = (uint64_t)tokens * H;
    const uint32_t blocks = (uint32_t)((items + kRmsThreads / kRowLanes - 1) / (kRmsThreads / kRowLanes));
    // n / H for n < 2^31: (n * magic) >> shift, magic = floor(2^shift / H) + 1
    // with 2^(shift - 31) the power of two at or above H
    uint32_t shift = 31;
    while (shift < 63 && (1ull << (shift - 31)) < H) ++shift;
    const uint32_t magic = H == 1 ? 0x80000000u : (uint32_t)((1ull << shift) / H + 1);
    if (in_bf16)
        hipLaunchKernelGGL((rms_writer<D, 1>), dim3(blocks), dim3(kRmsThreads), 0, stream, key,
                           value, kc, vc, sc, slots, signs, tokens, H, magic, shift, slot_count, isl);
    else
        hipLaunchKernelGGL((rms_writer<D, 0>), dim3(blocks), dim3(kRmsThreads), 0, stream, key,
                           value, kc, vc, sc, slots, signs, tokens, H, magic, shift, slot_count, isl);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_rms_writer(hipStream_t stream, int in_bf16, const uint16_t* key,
                             const uint16_t* value, int8_t* key_cache, int8_t* value_cache,
                             float* scale_cache, const int32_t* slots, const float* pi_signs,
                             uint32_t tokens, uint32_t H, uint32_t D, uint64_t slot_count,
                             float inv_sqrt_len)
{
    if (tokens == 0) return hipSuccess;
    switch (D) {
        case 64: return launch_rms_writer_t<64>(stream, in_bf16, key, value, key_cache, value_cache,
                                                scale_cache, slots, pi_signs, tokens, H, slot_count,
                                                inv_sqrt_len);
        case 128: return launch_rms_writer_t<128>(stream, in_bf16, key, value, key_cache,
                                                  value_cache, scale_cache, slots, pi_signs, tokens,
                                                  H, slot_count, inv_sqrt_len);
        case 256: return launch_rms_writer_t<256>(stream, in_bf16, key, value, key_cache,
                                                  value_cache, scale_cache, slots, pi_signs, tokens,
                                                  H, slot_count, inv_sqrt_len);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_rms_dequantize(hipStream_t stream, const int8_t* packed, float* out,
                                 uint64_t bytes)
{
    const uint64_t words = bytes / 4;
    if (words) {
        uint64_t blocks = (words + kRmsThreads - 1) / kRmsThreads;
        if (blocks > 2048) blocks = 2048;
        hipLaunchKernelGGL(rms_dequant, dim3((uint32_t)blocks), dim3(kRmsThreads), 0, stream,
                           (const uint32_t*)packed, (float4*)out, words);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (bytes % 4) {
        hipLaunchKernelGGL(rms_dequant_tail, dim3(1), dim3(4), 0, stream, (const uint8_t*)packed,
                           out, words * 4, bytes);
        return hipGetLastError();
    }
    return hipSuccess;
}

}  // namespace tq4
