// tq4_writer.hip -- reshape_and_cache for the TQ4 cache on gfx950.
//
// Three kernels:
//   strip_writer          aligned 16-token strips (the reference's A8/BF16 prefill
//                         writers, turboquant_reshape_and_cache_{a8,bf16}.cpp)
//   scatter_writer        requests of several tokens at arbitrary slots, in chunks
//                         of 16 tokens, nibble-exact merges into the value strips
//                         (turboquant_reshape_scatter_aiv.cpp:598-731)
//   scatter_token_writer  the same, one token to a request
//
// Work decomposition of the strip writer (MI355X): one 256-lane workgroup owns one strip of one
// head, both planes: two panels of 16 rows x d channels, one row of each per
// 16-lane group (two independent row jobs per lane). A row lives on 16
// lanes with CPL = d/16 consecutive channels per lane, so the 16-point
// Hadamard stages below CPL are in-register and the rest are lane exchanges
// inside the row; a strip's 16 rows are the workgroup's 16 row groups.
// Activations load as one contiguous vector per lane (coalesced: a strip of
// a head is 16 rows of d elements, row stride H*d). Key rows store as one
// contiguous word per lane (token-major); the value strip is transposed
// through LDS and stored as d*8 contiguous bytes (channel-major).
//
// Bit-exactness: the rotation is adds and subtracts in the fixed stage order
// of the reference's Ingress cascade (rotate_butterfly_oracle.hpp:44-48), the
// scale is a power of two taken from the exponent field, y * 2^(2-e) is exact
// (ldexp), and the one rounding is v_rndne. This translation unit is built
// with -ffp-contract=off.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tq4_device.hpp"
#include "tq4_internal.hpp"

namespace tq4 {
namespace {

constexpr int kWriterThreads = 256;  // 16 rows x 16 lanes

// Input element loads: CPL consecutive channels of one row.
template <int CPL>
__device__ __forceinline__ void load_row(const int8_t* src, float (&x)[CPL])
{
#pragma unroll
    for (int j = 0; j < CPL; ++j) x[j] = (float)src[j];
}

template <int CPL>
__device__ __forceinline__ void load_row(const uint16_t* src, float (&x)[CPL])
{
#pragma unroll
    for (int j = 0; j < CPL; ++j) x[j] = bf16_to_f32(src[j]);
}

// Signs for the lane's CPL channels: pi_signs when given (CPL consecutive
// floats, vector loads), else the first column of the reference's rotation
// tables (T[0][g][c0][0] = sign[g*32+c0]). The source is chosen once per
// launch (a uniform branch), never per channel.
template <int CPL>
__device__ __forceinline__ void load_signs(const float* pi_signs, const void* tables,
                                           int tables_bf16, int c0, float (&sign)[CPL])
{
    if (pi_signs != nullptr) {
        const float* src = pi_signs + c0;
        if constexpr (CPL % 4 == 0) {
#pragma unroll
            for (int j = 0; j < CPL; j += 4) {
                const float4 v = *(const float4*)(src + j);
                sign[j] = v.x;
                sign[j + 1] = v.y;
                sign[j + 2] = v.z;
                sign[j + 3] = v.w;
            }
        } else {
#pragma unroll
            for (int j = 0; j < CPL; ++j) sign[j] = src[j];
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
        const int c = c0 + j;
        if (tables_bf16) {
            const uint16_t raw = ((const uint16_t*)tables)[(size_t)c * 32];
            sign[j] = (raw & 0x8000u) ? -1.0f : 1.0f;
        } else {
            const int8_t raw = ((const int8_t*)tables)[(size_t)c * 32];
            sign[j] = raw < 0 ? -1.0f : 1.0f;
        }
    }
}

// ------------------------------------------------------------ strip writer
// The strip writer's row order and arithmetic, tuned for the VALU issue rate
// (with two waves per SIMD the writer's rotation, quantisation and packing
// are issue-bound, four cycles per wave64 instruction):
//
// * Lane order and butterflies: the row lane order of tq4_device.hpp
//   (row_lane), where every cross-lane stride is one DPP pattern, and the
//   sign-tracked butterfly (row_fmac_stage): one DPP-fed v_fmac_f32 per
//   element and stage.
// * Quantiser. t = fma(y, 2^(2-e), kQMagic) with kQMagic = 1.5 * 2^23 + 8:
//   y * 2^(2-e) is exact and |y * 2^(2-e)| < 8, so the one rounding of the
//   sum is the round-to-nearest-even of y * 2^(2-e) (kQMagic is even: ties
//   keep their parity), and t = kQMagic + n exactly; min(t, kQMagic + 7) is
//   the clamp at 7. Bits 0..3 of t then hold n + 8 and bits 4..7 are zero,
//   so codes pack with one shift-or per pair and byte permutes, and the
//   packed word is XORed with 0x8...8 to give the two's-complement nibbles.
//   Non-finite inputs saturate: +inf and NaN give 7, -inf gives -8.
// * One barrier: the slot vote and the value-strip transpose share it. The
//   slot loads go out first, ahead of the rows they do not depend on, so
//   their round trip is the rows' round trip.

constexpr float kQMagic = 12582920.0f;     // 1.5 * 2^23 + 8
constexpr float kQMagicTop = 12582927.0f;  // kQMagic + 7

// One butterfly stage over the writer's two rows (key, value), l being this
// lane's logical lane: in registers below CPL, else row_fmac_stage on the
// sign-tracked values.
template <int CPL>
__device__ __forceinline__ void writer_butterfly(float (&v)[2][CPL], int stride, int l)
{
    if (stride < CPL) {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                if (j & stride) continue;
                const float a = v[r][j];
                const float b = v[r][j + stride];
                v[r][j] = b + a;
                v[r][j + stride] = a - b;
            }
        }
    } else {
        const int k = __builtin_ctz(stride / CPL);
        const float c = ((l >> k) & 1) ? -1.0f : 1.0f;
        row_fmac_stage<CPL>(v[0], c, k);
        row_fmac_stage<CPL>(v[1], c, k);
    }
}

// Rotate both rows (strides 1..16, the sign diagonal, 32..D/2). The results
// are held as sigma * v with sigma = (-1)^popcount(l) (row_sigma).
template <int D, int CPL>
__device__ __forceinline__ void writer_rotate(float (&v)[2][CPL], const float (&sign)[CPL], int l)
{
#pragma unroll
    for (int s = 1; s < 32 && s < D; s <<= 1) writer_butterfly<CPL>(v, s, l);
#pragma unroll
    for (int r = 0; r < 2; ++r) {
#pragma unroll
        for (int j = 0; j < CPL; ++j) v[r][j] *= sign[j];
    }
#pragma unroll
    for (int s = 32; s < D; s <<= 1) writer_butterfly<CPL>(v, s, l);
}

// Each row's absmax over its 16 lanes, starting from `floor` (1.0 for the
// prefill policy, 0 for the exact one).
template <int CPL>
__device__ __forceinline__ void writer_absmax(const float (&v)[2][CPL], float floor, float (&a)[2])
{
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        a[r] = floor;
#pragma unroll
        for (int j = 0; j < CPL; ++j) a[r] = fmaxf(a[r], fabsf(v[r][j]));
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) row_max2(a[0], a[1], k);
}

// Rotate both rows, take each row's absmax (prefill policy: floored at 1.0)
// and quantise: t[r][j] receives kQMagic + code as bits; scale[r] is the
// row's stored scale.
template <int D, int CPL>
__device__ __forceinline__ void writer_rotate_quantise(float (&v)[2][CPL], const float (&sign)[CPL],
                                                       int l, float inv_sqrt_len,
                                                       uint32_t (&t)[2][CPL], float (&scale)[2])
{
    writer_rotate<D, CPL>(v, sign, l);
    float a[2];
    writer_absmax<CPL>(v, 1.0f, a);
    // the stored values are sigma * v: the quantiser's exact power of two
    // carries sigma
    const float sigma = row_sigma(l);
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        // a >= 1 (the prefill floor; NaN never wins fmaxf): the exponent
        // field alone, 0 .. 128 (128: infinity); 2^(2-e) is a normal float
        const int e = (int)(__float_as_uint(a[r]) >> 23) - 127;
        const float p2 = sigma * ldexpf(1.0f, 2 - e);
#pragma unroll
        for (int j = 0; j < CPL; ++j)
            t[r][j] = __float_as_uint(fminf(__builtin_fmaf(v[r][j], p2, kQMagic), kQMagicTop));
        scale[r] = ldexpf(1.0f, e - 2) * inv_sqrt_len;
    }
}

// Eight codes (t[k] bits 0..3 = code + 8, bits 4..7 zero) as one word of
// signed nibbles, code k at bits 4k.
__device__ __forceinline__ uint32_t pack8(const uint32_t* t)
{
    const uint32_t p01 = (t[1] << 4) | t[0];
    const uint32_t p23 = (t[3] << 4) | t[2];
    const uint32_t p45 = (t[5] << 4) | t[4];
    const uint32_t p67 = (t[7] << 4) | t[6];
    const uint32_t lo = __builtin_amdgcn_perm(p23, p01, 0x0C0C0400u);  // p01.b0, p23.b0
    const uint32_t hi = __builtin_amdgcn_perm(p67, p45, 0x0C0C0400u);
    return __builtin_amdgcn_perm(hi, lo, 0x05040100u) ^ 0x88888888u;
}

// Four codes as 16 bits of signed nibbles.
__device__ __forceinline__ uint32_t pack4(const uint32_t* t)
{
    const uint32_t p01 = (t[1] << 4) | t[0];
    const uint32_t p23 = (t[3] << 4) | t[2];
    return (__builtin_amdgcn_perm(p23, p01, 0x0C0C0400u) ^ 0x8888u) & 0xffffu;
}

// Word w (channel w / 2, token half w % 2) of a strip's value words from the
// transpose buffer: that channel's codes of tokens 8 * half .. + 7, one nibble
// of each of 8 consecutive buffer words (two 16-byte reads).
__device__ __forceinline__ uint32_t strip_word(const uint32_t (*lds_t)[20], int w)
{
    const int channel = w >> 1, half = w & 1;
    const uint32_t* src = &lds_t[channel >> 3][8 * half];
    const uint4 a = *(const uint4*)src;
    const uint4 b = *(const uint4*)(src + 4);
    const uint32_t sh = 4u * (uint32_t)(channel & 7);
    const uint32_t n[8] = {__builtin_amdgcn_ubfe(a.x, sh, 4), __builtin_amdgcn_ubfe(a.y, sh, 4),
                           __builtin_amdgcn_ubfe(a.z, sh, 4), __builtin_amdgcn_ubfe(a.w, sh, 4),
                           __builtin_amdgcn_ubfe(b.x, sh, 4), __builtin_amdgcn_ubfe(b.y, sh, 4),
                           __builtin_amdgcn_ubfe(b.z, sh, 4), __builtin_amdgcn_ubfe(b.w, sh, 4)};
    const uint32_t p01 = (n[1] << 4) | n[0];
    const uint32_t p23 = (n[3] << 4) | n[2];
    const uint32_t p45 = (n[5] << 4) | n[4];
    const uint32_t p67 = (n[7] << 4) | n[6];
    const uint32_t lo = __builtin_amdgcn_perm(p23, p01, 0x0C0C0400u);
    const uint32_t hi = __builtin_amdgcn_perm(p67, p45, 0x0C0C0400u);
    return __builtin_amdgcn_perm(hi, lo, 0x05040100u);
}

// grid = (strips, H): a workgroup owns one strip of one head, both planes;
// every lane runs two row jobs (key, value), whose loads go out together
// with the slot loads before the first rotation.
template <int D, typename In>
__global__ __launch_bounds__(kWriterThreads) void strip_writer(
    const In* __restrict__ key, const In* __restrict__ value, int8_t* __restrict__ key_cache,
    int8_t* __restrict__ value_cache, float* __restrict__ scale_cache,
    const int32_t* __restrict__ slots, const float* __restrict__ pi_signs,
    const void* __restrict__ tables, int tables_bf16, uint32_t H, uint32_t S, uint32_t P,
    float inv_sqrt_len)
{
    constexpr int CPL = D / 16;
    constexpr int TS = 20;  // token stride of the transpose buffer, in words
    // [channel / 8][token, padded to TS] words of 8 channel codes; 20-word
    // rows put the 64 lanes of a wave (16 lanes x 4 tokens) on distinct banks
    __shared__ __align__(16) uint32_t lds_t[D / 8][TS];
    __shared__ __align__(16) int ok_w[kWriterThreads / 64];  // per-wave slot checks

    const uint32_t strip = blockIdx.x, head = blockIdx.y;
    const int tid = threadIdx.x;
    const int row = tid >> 4;                 // token within the strip
    const int l = row_lane(tid & 15);      // logical lane: channels l*CPL ..

    // slots first, then the rows and the signs: one round trip for all
    const int32_t slot0 = slots[(size_t)strip * kStrip];
    const int32_t mine = slots[(size_t)strip * kStrip + row];
    float v[2][CPL], sign[CPL];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const In* src = (j == 0 ? key : value) +
                        ((size_t)((size_t)strip * kStrip + row) * H + head) * D + l * CPL;
        load_row<CPL>(src, v[j]);
    }
    load_signs<CPL>(pi_signs, tables, tables_bf16, l * CPL, sign);

    uint32_t t[2][CPL];
    float scale[2];
    writer_rotate_quantise<D, CPL>(v, sign, l, inv_sqrt_len, t, scale);

    // Slot contract for this strip: consecutive, strip-aligned, in range.
    // Each wave votes; the vote is read behind the transpose's barrier.
    const bool ok = slot0 >= 0 && (slot0 % kStrip) == 0 && mine == slot0 + row &&
                    (uint32_t)slot0 / S < P;
    static_assert(kWriterThreads == 256, "four wave votes");
    const int wv = __all(ok);
    if ((tid & 63) == 0) ok_w[tid >> 6] = wv;
    // value codes into the transpose buffer: one word of 8 channels per store
    // (at d = 64 two lanes share a word, 16 bits each)
    if constexpr (CPL >= 8) {
#pragma unroll
        for (int k = 0; k < CPL / 8; ++k) lds_t[l * (CPL / 8) + k][row] = pack8(&t[1][8 * k]);
    } else {
        ((uint16_t*)&lds_t[l >> 1][row])[l & 1] = (uint16_t)pack4(t[1]);
    }
    lds_barrier();
    {
        const int4 w4 = *(const int4*)ok_w;
        if (!(w4.x & w4.y & w4.z & w4.w)) return;
    }
    const uint32_t page = (uint32_t)slot0 / S;
    const uint32_t tip = (uint32_t)slot0 % S + (uint32_t)row;
    const size_t head_base = ((size_t)page * H + head) * S;  // in tokens
    if ((tid & 15) == 0) {
        scale_cache[((size_t)page * H + head) * S + tip] = scale[0];
        scale_cache[(((size_t)P + page) * H + head) * S + tip] = scale[1];
    }
    int8_t* kdst = key_cache + (head_base + tip) * (D / 2) + l * (CPL / 2);
    if constexpr (CPL == 16)
        *(uint2*)kdst = make_uint2(pack8(t[0]), pack8(&t[0][8]));
    else if constexpr (CPL == 8)
        *(uint32_t*)kdst = pack8(t[0]);
    else
        *(uint16_t*)kdst = (uint16_t)pack4(t[0]);
    // the value strip leaves as d*8 contiguous bytes: output word (channel,
    // half) holds that channel's codes of tokens 8*half .. +7, one nibble
    // from each of 8 consecutive buffer words (two 16-byte reads)
    uint32_t* strip_words =
        (uint32_t*)(value_cache + (head_base + (tip & ~(uint32_t)15)) * (D / 2));
    for (int w = tid; w < D * 2; w += kWriterThreads) {
        strip_words[w] = strip_word(lds_t, w);
    }
}

// ----------------------------------------------------------- scatter writer
// Requests of several tokens (cu_seqlens). The reference walks a (request,
// head) item's tokens in order, run by run; here a request is cut into
// chunks of 16 tokens that workgroups take independently, with the same bytes
// as that walk for any slots:
//   * Chunk c holds tokens 16c - a .. 16c - a + 15, a the first slot's place
//     in its strip, so a request written at consecutive positions has one
//     strip to a chunk, wherever it begins.
//   * A chunk whose valid tokens sit at consecutive slots of one strip that no
//     other token of the request touches is written at once (scatter_chunk):
//     the strip writer's arithmetic and transpose, the value strip's words
//     merged under the mask of the columns written (whole words are stored
//     without a read).
//   * To know that no other token touches the strip, a chunk of a request of
//     up to 8192 tokens reads the request's slots under its rows' loads (32 KB
//     a chunk there, from the caches). That grows with the square of the length,
//     so of longer requests a workgroup searches the chunks of its run together,
//     16 to a pass over the slots (scatter_search); a request of one chunk
//     needs no search.
//   * Any other chunk goes token by token (scatter_tokens): a strip belongs to
//     the chunk that holds its first token, which writes all of its tokens in
//     token order; the other chunks skip them. So one workgroup at a time
//     merges into a strip, and of two tokens with one slot the later wins. It
//     reads the request's slots once a token, so a fully shuffled request
//     costs the square of its length (8192 tokens x 8 heads: 1.0 ms; 18.4 ms
//     item by item).
// A workgroup takes a run of (chunk, head) pairs: the slots are read once for
// the heads of a chunk, and the next head's rows are in flight under the
// current head's arithmetic.
// 8 ragged chunks of 17..2048 tokens (8256 tokens, 8 heads of 128):
// 790 us a (request, head) item at a time, 16.8 us in chunks; bound there by
// the vector ALU (about 310 instructions a wave, chunk and head) and by the
// two loads in turn that a chunk begins with (slots, rows). One request of
// 32768 / 131072 tokens, 8 heads of 128: 66 / 465 us with a search a chunk,
// 56 / 230 together (64 requests of 2048: 169). Requests of one token, 8 heads
// (1 head): 256 of them 9.5 (5.2) us, 1024 22.9 (8.2), 4096 77 (23.5); item by
// item 9.3 (4.6), 27.9 (6.2) and 98 (15.7): there the one head's workgroups
// wait for the chunk count that a workgroup to an item does without.

// One lane's CPL consecutive BF16 channels as loaded (any alignment).
template <int CPL>
struct RawRow {
    uint32_t w[CPL / 2];
};

template <int CPL>
__device__ __forceinline__ void load_raw(const uint16_t* src, RawRow<CPL>& r)
{
    __builtin_memcpy(r.w, src, CPL * 2);
}

template <int CPL>
__device__ __forceinline__ void unpack_raw(const RawRow<CPL>& r, float (&v)[CPL])
{
#pragma unroll
    for (int i = 0; i < CPL / 2; ++i) {
        v[2 * i] = __uint_as_float(r.w[i] << 16);
        v[2 * i + 1] = __uint_as_float(r.w[i] & 0xffff0000u);
    }
}

// Exact policy on both rows (held as sigma * v, absmax a): t as the strip
// writer's (kQMagic + code as bits). Rows with an absmax below 2^-100, zero or
// infinite (their power of two is not a normal float, or the row has its own
// rule: zero rows store codes 0 and scale 1, -inf stores code 0) take the
// written-out form behind a wave vote.
template <int CPL>
__device__ __forceinline__ void quantise_exact(const float (&v)[2][CPL], const float (&a)[2],
                                               float sigma, float inv_sqrt_len,
                                               uint32_t (&t)[2][CPL], float (&scale)[2])
{
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const uint32_t field = __float_as_uint(a[r]) >> 23;  // a >= 0
        const float p2 = sigma * __uint_as_float((256u - field) << 23);  // 2^(2-e)
#pragma unroll
        for (int j = 0; j < CPL; ++j)
            t[r][j] = __float_as_uint(fminf(__builtin_fmaf(v[r][j], p2, kQMagic), kQMagicTop));
        scale[r] = __uint_as_float((field - 2u) << 23) * inv_sqrt_len;
    }
    const bool odd0 = !(a[0] >= 0x1p-100f && a[0] < INFINITY);
    const bool odd1 = !(a[1] >= 0x1p-100f && a[1] < INFINITY);
    if (__builtin_expect(__any(odd0 || odd1), 0)) {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            if (!(r == 0 ? odd0 : odd1)) continue;
            const bool zero = a[r] == 0.0f;
            const int e = zero ? 2 : exponent_of(a[r]);
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const float y = fminf(rintf(ldexpf(sigma * v[r][j], 2 - e)), 7.0f);
                const uint32_t q = zero ? 0u : (uint32_t)(int)y & 0xfu;
                t[r][j] = 0x4B400000u | (q ^ 8u);
            }
            scale[r] = zero ? 1.0f : ldexpf(1.0f, e - 2) * inv_sqrt_len;
        }
    }
}

// The nibble mask of 8 columns (bit i -> nibble i).
__device__ __forceinline__ uint32_t nibble_mask(uint32_t b)
{
    uint32_t x = (b | (b << 12)) & 0x000F000Fu;
    x = (x | (x << 6)) & 0x03030303u;
    x = (x | (x << 3)) & 0x11111111u;
    return x * 15u;
}

template <int CPL>
__device__ __forceinline__ void store_key_word(int8_t* dst, const uint32_t (&t)[CPL])
{
    if constexpr (CPL == 16)
        *(uint2*)dst = make_uint2(pack8(t), pack8(&t[8]));
    else if constexpr (CPL == 8)
        *(uint32_t*)dst = pack8(t);
    else
        *(uint16_t*)dst = (uint16_t)pack4(t);
}

// Workgroups of the launch: as many as the registers keep resident on 256
// CUs (four waves a SIMD, three at d = 256), so one generation takes it all.
// 8 requests of 17..2048 tokens: 512 / 768 / 1024 / 2048 workgroups 18.7 /
// 17.6 / 18.2 / 20.2 us; one of 8000 tokens 17.4 / 20.1 / 16.2 / 20.2 us
// (1024 at 16.8 and 15.5 since the requests' lengths and places are staged).
template <int D>
constexpr uint32_t kScatterGrid = D == 256 ? 768 : 1024;
constexpr uint32_t kScatterPlan = 1024;  // requests whose chunk prefix is staged on chip

// The search for other tokens in the strips of a run's chunks (scatter_search).
constexpr uint32_t kGroup = kWriterThreads / kStrip;  // chunks to a pass: a slot a thread
constexpr uint32_t kTable = kWriterThreads;           // their strips, open-addressed
constexpr int32_t kNoStrip = 0x7fffffff;              // above every slot / 16
// Longer requests are searched by runs: a pass of its own costs more than the
// search under the rows' loads until the run has several chunks (8 heads: 8192
// tokens 20.9 us a chunk at a time, 21.5 together; 32768 66 / 56).
constexpr uint32_t kSearchFrom = 8192;
constexpr uint32_t kSearchRun = 256;  // chunks of a run searched together at most
struct SearchShared {
    int32_t table[kTable];
    uint32_t owner[kTable];
    uint32_t clash;
    uint8_t found[kSearchRun];  // the run's chunks (modulo its size) with a clash
};

struct ScatterArgs {
    const uint16_t *key, *value;
    int8_t *key_cache, *value_cache;
    float* scale_cache;
    const int32_t* slots;
    uint32_t H, S, P;
    float inv_sqrt_len;
};

__device__ __forceinline__ bool slot_in_pool(int32_t slot, uint32_t S, uint32_t P)
{
    return slot >= 0 && (uint64_t)(uint32_t)slot < (uint64_t)S * P;
}

// Tokens first .. first + 15 (of the request's n at t0) one at a time, heads
// [h0, h1): each strip whose first token of the request lies here, with all
// of its tokens in token order. Every thread of the workgroup runs it (it has
// barriers); a 16-lane group takes a head, so one lane makes all merges of a
// strip word, in order.
template <int D>
__device__ __forceinline__ void scatter_tokens(const ScatterArgs& p, uint32_t t0, uint32_t n,
                                               int64_t first, uint32_t h0, uint32_t h1,
                                               const float (&sign)[D / 16])
{
    constexpr int CPL = D / 16;
    const int tid = threadIdx.x;
    const int l = row_lane(tid & 15);
    const float sigma = row_sigma(l);
    for (int i = 0; i < kStrip; ++i) {
        const int64_t at = first + i;
        if (at < 0 || at >= (int64_t)n) continue;
        const uint32_t i0 = (uint32_t)at;
        const int32_t slot0 = p.slots[t0 + i0];
        if (!slot_in_pool(slot0, p.S, p.P)) continue;
        const int32_t strip = slot0 >> 4;
        int seen = 0;  // an earlier token of the request in this strip
        const int32_t* sl = p.slots + t0;
        for (uint32_t u = tid; u < i0; u += 4 * kWriterThreads) {
#pragma unroll
            for (int k = 0; k < 4; ++k) seen |= (sl[min(u + k * kWriterThreads, i0 - 1)] >> 4) == strip;
        }
        if (__syncthreads_or(seen)) continue;
        for (uint32_t base = i0; base < n; base += 4 * 64) {
            uint64_t in[4];  // four loads in flight
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t u = base + 64 * k + (tid & 63);
                in[k] = __ballot((sl[min(u, n - 1)] >> 4) == strip && u < n);
            }
#pragma unroll 1
            for (int k = 0; k < 4; ++k) {
                uint64_t m = k == 0 ? in[0] : k == 1 ? in[1] : k == 2 ? in[2] : in[3];
                for (; m != 0; m &= m - 1) {
                    const uint32_t token = t0 + base + 64 * k + (uint32_t)__builtin_ctzll(m);
                    const uint32_t slot = (uint32_t)p.slots[token];
                    const uint32_t page = slot / p.S, tip = slot % p.S, col = tip % kStrip;
                    for (uint32_t h = h0 + (tid >> 4); h < h1; h += kWriterThreads / 16) {
                        const size_t src = ((size_t)token * p.H + h) * D + l * CPL;
                        RawRow<CPL> rk, rv;
                        load_raw<CPL>(p.key + src, rk);
                        load_raw<CPL>(p.value + src, rv);
                        float v[2][CPL], a[2], sc[2];
                        unpack_raw<CPL>(rk, v[0]);
                        unpack_raw<CPL>(rv, v[1]);
                        writer_rotate<D, CPL>(v, sign, l);
                        writer_absmax<CPL>(v, 0.0f, a);
                        uint32_t t[2][CPL];
                        quantise_exact<CPL>(v, a, sigma, p.inv_sqrt_len, t, sc);
                        const size_t row = ((size_t)page * p.H + h) * p.S + tip;
                        if ((tid & 15) == 0) {
                            p.scale_cache[row] = sc[0];
                            p.scale_cache[(size_t)p.P * p.H * p.S + row] = sc[1];
                        }
                        store_key_word<CPL>(p.key_cache + row * (D / 2) + l * (CPL / 2), t[0]);
                        uint32_t* words = (uint32_t*)(p.value_cache + (row - col) * (D / 2)) +
                                          2 * l * CPL + (col >> 3);
                        const uint32_t sh = 4u * (col & 7u);
#pragma unroll
                        for (int j = 0; j < CPL; ++j)
                            words[2 * j] = (words[2 * j] & ~(0xfu << sh)) |
                                           (((t[1][j] ^ 8u) & 0xfu) << sh);
                    }
                }
            }
        }
    }
}

// Which of the chunks c .. c + m - 1 (m <= kGroup) of a request (n tokens at
// t0, the first at place a of its strip) share a strip with a token outside
// them, into found[v ..]: their strips go into a table, and every slot of the
// request is looked up in it, once for all of them. A chunk with several strips
// stays out of the table (scatter_chunk finds it).
__device__ __forceinline__ void scatter_search(const ScatterArgs& p, SearchShared& s, uint32_t t0,
                                               uint32_t n, uint32_t a, uint32_t c, uint32_t v,
                                               uint32_t m)
{
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // nothing derived from it is held for long
    const int row = tid >> 4, j16 = tid & 15;
    const int64_t at = (int64_t)c * kStrip - a + tid;
    const int32_t slot =
        (uint32_t)row < m && at >= 0 && at < (int64_t)n ? p.slots[t0 + (uint32_t)at] : -1;
    s.table[tid] = kNoStrip;
    if (tid == 0) s.clash = 0;
    lds_barrier();
    const bool ok = slot_in_pool(slot, p.S, p.P);
    const int sh = tid & 48;
    const uint32_t vmask = (uint32_t)(__ballot(ok) >> sh) & 0xffffu;
    const int32_t strip = __shfl(slot, sh + (vmask != 0 ? __builtin_ctz(vmask) : 0), 64) >> 4;
    const bool several = ((uint32_t)(__ballot(ok && (slot >> 4) != strip) >> sh) & 0xffffu) != 0;
    if (j16 == 0 && vmask != 0 && !several) {
        for (uint32_t x = (uint32_t)strip % kTable;; x = (x + 1) % kTable) {
            const int32_t was = atomicCAS(&s.table[x], kNoStrip, strip);
            if (was == kNoStrip) s.owner[x] = (uint32_t)row;
            if (was == strip) atomicOr(&s.clash, 1u << row);  // another chunk's as well
            if (was == kNoStrip || was == strip) break;       // at most kGroup of kTable are taken
        }
    }
    lds_barrier();
    const int32_t* sl = p.slots + t0;
    uint32_t hit = 0;
    for (uint64_t ub = 0; ub < n; ub += 8 * kWriterThreads) {  // eight loads in flight a thread
        int32_t st[8], e[8];
#pragma unroll
        for (int k = 0; k < 8; ++k)
            st[k] = sl[min((uint32_t)ub + k * kWriterThreads + tid, n - 1)] >> 4;
#pragma unroll
        for (int k = 0; k < 8; ++k) e[k] = s.table[(uint32_t)st[k] % kTable];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            uint32_t x = (uint32_t)st[k] % kTable;
            while (e[k] != kNoStrip && e[k] != st[k]) {
                x = (x + 1) % kTable;
                e[k] = s.table[x];
            }
            if (e[k] == st[k]) {
                const uint32_t u = min((uint32_t)ub + k * kWriterThreads + tid, n - 1);
                if (((u + a) >> 4) != c + s.owner[x]) hit |= 1u << s.owner[x];
            }
        }
    }
    if (hit != 0) atomicOr(&s.clash, hit);
    lds_barrier();
    if ((uint32_t)tid < m) s.found[(v + tid) % kSearchRun] = (uint8_t)((s.clash >> tid) & 1u);
    lds_barrier();
}

// One chunk of 16 tokens (first .. first + 15 of the request's n at t0), heads
// [h0, h1). searched: no token outside the chunk touches its strip (known
// already). False: nothing is written, the chunk goes token by token.
template <int D>
__device__ __forceinline__ bool scatter_chunk(const ScatterArgs& p, uint32_t t0, uint32_t n,
                                              int64_t first, bool searched, uint32_t h0,
                                              uint32_t h1, const float (&sign)[D / 16],
                                              uint32_t (*lds_t)[D / 8][20], int* clash_w)
{
    constexpr int CPL = D / 16;
    const int tid = threadIdx.x;
    const int row = tid >> 4;
    const int l = row_lane(tid & 15);
    const float sigma = row_sigma(l);

    // the first head's rows, and lane j of every 16 the slot of token j
    const int64_t at = first + row;
    const uint32_t tok = t0 + (uint32_t)(at < 0 ? 0 : at < (int64_t)n ? at : (int64_t)n - 1);
    const size_t src0 = ((size_t)tok * p.H + h0) * D + l * CPL;
    RawRow<CPL> rk, rv;
    load_raw<CPL>(p.key + src0, rk);
    load_raw<CPL>(p.value + src0, rv);
    const int j16 = tid & 15;
    const int64_t aj = first + j16;
    const int32_t slot_j = aj >= 0 && aj < (int64_t)n ? p.slots[t0 + (uint32_t)aj] : -1;
    const bool valid_j = slot_in_pool(slot_j, p.S, p.P);
    const uint32_t vmask = (uint32_t)__ballot(valid_j) & 0xffffu;  // the same in every wave
    if (vmask == 0) return true;
    // regular: every valid token j at slot base + j, all in one strip
    const int lead = __builtin_ctz(vmask);
    const int32_t base = __builtin_amdgcn_readlane(slot_j, lead) - lead;
    const int32_t strip = (base + lead) >> 4;
    const bool odd = valid_j && (slot_j - j16 != base || (slot_j >> 4) != strip);
    const bool regular = __ballot(odd) == 0;
    // does another token of the request touch the strip?
    int clash = !regular;
    if (regular && !searched) {
        // eight loads in flight a thread (past the end: the last token again)
        const int32_t* sl = p.slots + t0;
        const uint32_t f = (uint32_t)first;  // mod 2^32, as the distance below
        for (uint32_t u0 = tid; u0 < n; u0 += 8 * kWriterThreads) {
            int32_t s[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) s[k] = sl[min(u0 + k * kWriterThreads, n - 1)];
#pragma unroll
            for (int k = 0; k < 8; ++k)
                clash |= (s[k] >> 4) == strip &&
                         min(u0 + k * kWriterThreads, n - 1) - f >= (uint32_t)kStrip;
        }
    }
    const int wc = __any(clash);
    if ((tid & 63) == 0) clash_w[tid >> 6] = wc;

    const int shift = base - strip * kStrip;           // column of token j: j + shift
    const uint32_t cmask = shift >= 0 ? vmask << shift : vmask >> -shift;  // columns written
    const uint32_t m0 = nibble_mask(cmask & 0xffu), m1 = nibble_mask((cmask >> 8) & 0xffu);
    const bool whole = (cmask & 0xffffu) == 0xffffu;
    const uint32_t page = (uint32_t)(base + lead) / p.S;
    const uint32_t strip_tip = (uint32_t)strip * kStrip - page * p.S;
    const bool mine = (vmask >> row) & 1u;
    const uint32_t col = (uint32_t)(row + shift) & 15u;
    const size_t plane = (size_t)p.P * p.H * p.S;
    constexpr int NW = (2 * D + kWriterThreads - 1) / kWriterThreads;  // strip words a thread

    for (uint32_t h = h0, it = 0; h < h1; ++h, ++it) {
        const size_t srow = ((size_t)page * p.H + h) * p.S + strip_tip;  // the strip's first row
        uint32_t* words = (uint32_t*)(p.value_cache + srow * (D / 2));
        float v[2][CPL];
        unpack_raw<CPL>(rk, v[0]);
        unpack_raw<CPL>(rv, v[1]);
        if (h + 1 < h1) {
            const size_t src = src0 + (size_t)(it + 1) * D;
            load_raw<CPL>(p.key + src, rk);
            load_raw<CPL>(p.value + src, rv);
        }
        uint32_t old[NW];
        if (!whole) {
#pragma unroll
            for (int k = 0; k < NW; ++k)
                old[k] = tid + k * kWriterThreads < 2 * D ? words[tid + k * kWriterThreads] : 0u;
        }
        writer_rotate<D, CPL>(v, sign, l);
        float a[2], sc[2];
        writer_absmax<CPL>(v, 0.0f, a);
        uint32_t t[2][CPL];
        quantise_exact<CPL>(v, a, sigma, p.inv_sqrt_len, t, sc);
        uint32_t(*buf)[20] = lds_t[it & 1];
        if (mine) {
            if constexpr (CPL >= 8) {
#pragma unroll
                for (int k = 0; k < CPL / 8; ++k) buf[l * (CPL / 8) + k][col] = pack8(&t[1][8 * k]);
            } else {
                ((uint16_t*)&buf[l >> 1][col])[l & 1] = (uint16_t)pack4(t[1]);
            }
        }
        // one barrier a head: the buffer written two heads on is read before
        // the barrier in between
        lds_barrier();
        if (it == 0) {
            const int4 c4 = *(const int4*)clash_w;
            if (c4.x | c4.y | c4.z | c4.w) return false;
        }
        if (mine) {
            const size_t r = srow + col;
            if ((tid & 15) == 0) {
                p.scale_cache[r] = sc[0];
                p.scale_cache[plane + r] = sc[1];
            }
            store_key_word<CPL>(p.key_cache + r * (D / 2) + l * (CPL / 2), t[0]);
        }
#pragma unroll
        for (int k = 0; k < NW; ++k) {
            const int w = tid + k * kWriterThreads;
            const uint32_t m = (w & 1) ? m1 : m0;
            if (w < 2 * D && m != 0) {
                const uint32_t bits = strip_word(buf, w);
                words[w] = whole ? bits : (old[k] & ~m) | (bits & m);
            }
        }
    }
    return true;
}

// The inclusive prefix sum over a wave: four shifts within the rows of 16
// lanes, then each row's last lane added to the next rows.
__device__ __forceinline__ uint32_t wave_prefix(uint32_t v)
{
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);  // row_shr 1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);  // row_shr 2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);  // row_shr 4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);  // row_shr 8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);  // row_bcast 15
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);  // row_bcast 31
    return v;
}

// The lengths are on the device only, so the grid is fixed: every workgroup
// counts the requests' chunks (blocks of 64 requests to the waves in turn, a
// prefix over each in LDS and one over the blocks) and takes an equal run of the
// (chunk, head) pairs.
template <int D>
__global__ __launch_bounds__(kWriterThreads, D == 256 ? 3 : 4) void scatter_writer(
    ScatterArgs p, const float* __restrict__ pi_signs, const int32_t* __restrict__ cu_seqlens,
    int32_t* __restrict__ probe, uint32_t probe_grid, uint32_t num_requests, uint32_t item_begin,
    uint32_t item_count)
{
    constexpr int CPL = D / 16;
    __shared__ __align__(16) uint32_t lds_t[2][D / 8][20];
    __shared__ __align__(16) int clash_w[kWriterThreads / 64];
    __shared__ SearchShared search;
    // the requests: inclusive prefix of their chunks within their 64, first
    // token, length, and the first token's place in its strip; read once here,
    // so a chunk does not begin with two more dependent loads
    __shared__ uint32_t chunks[kScatterPlan], starts[kScatterPlan], counts[kScatterPlan];
    __shared__ uint8_t places[kScatterPlan];
    __shared__ uint32_t sums[kScatterPlan / 64];
    const int tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    if (probe != nullptr && blockIdx.x == 0 && tid < 32) {
        const int32_t fields[4] = {0, (int32_t)probe_grid, 1, (int32_t)item_count};
        probe[tid] = fields[tid >> 3];
    }
    const uint64_t item_end = (uint64_t)item_begin + item_count;
    const uint32_t r0 = item_begin / p.H;
    const uint32_t r1 = (uint32_t)min((uint64_t)num_requests, (item_end + p.H - 1) / p.H);
    if (r1 <= r0) return;
    float sign[CPL];
    load_signs<CPL>(pi_signs, nullptr, 0, row_lane(tid & 15) * CPL, sign);

    for (uint64_t rb = r0; rb < r1; rb += kScatterPlan) {
        const uint32_t nr = (uint32_t)min((uint64_t)kScatterPlan, r1 - rb);
        const int32_t* cu = cu_seqlens + rb;
#pragma unroll 1
        for (uint32_t b = wave; 64 * b < nr; b += kWriterThreads / 64) {
            const uint32_t i = min(64 * b + lane, nr - 1);
            const uint32_t t0 = (uint32_t)cu[i], t1 = (uint32_t)cu[i + 1];
            const uint32_t n = 64 * b + lane < nr && t1 > t0 ? t1 - t0 : 0u;
            const int32_t s0 = n > 0 ? p.slots[t0] : 0;
            const uint32_t place = s0 >= 0 ? (uint32_t)s0 % kStrip : 0u;
            const uint32_t v = wave_prefix(n > 0 ? (n + place + 15u) >> 4 : 0u);
            if (lane == 63) sums[b] = v;
            chunks[64 * b + lane] = v;
            starts[64 * b + lane] = t0;
            counts[64 * b + lane] = n;
            places[64 * b + lane] = (uint8_t)place;
        }
        lds_barrier();
        // lane b: the chunks up to and with block b of 64 requests
        const uint32_t blocks = wave_prefix(64u * lane < nr ? sums[lane] : 0u);
        auto before = [&](uint32_t b) -> uint32_t {
            return b > 0 ? __builtin_amdgcn_readlane(blocks, b - 1) : 0u;
        };
        // the prefix up to and with request i
        auto upto = [&](uint32_t i) -> uint32_t {
            return __builtin_amdgcn_readfirstlane(chunks[i]) + before(i / 64);
        };
        // an equal run of (chunk, head) pairs to every workgroup
        const uint32_t total = __builtin_amdgcn_readlane(blocks, 63);
        const uint64_t pairs = (uint64_t)total * p.H;
        const uint64_t per = (pairs + kScatterGrid<D> - 1) / kScatterGrid<D>;
        const uint64_t at = per * blockIdx.x;
        uint32_t v = pairs <= 0xffffffffull ? (uint32_t)at / p.H : (uint32_t)(at / p.H);
        uint32_t h = (uint32_t)(at - (uint64_t)v * p.H);
        uint32_t i = 0;  // the first request whose prefix passes v
        if (at < pairs) {
            const uint32_t b = (uint32_t)__builtin_ctzll(__ballot(blocks > v));
            i = 64 * b + (uint32_t)__builtin_ctzll(__ballot(chunks[64 * b + lane] + before(b) > v));
        }
        // (a workgroup's run is far below 2^32: its rows are in memory)
        uint32_t left = at < pairs ? (uint32_t)min(per, pairs - at) : 0u;
        uint32_t known = 0;  // the run's chunks before this one are searched
        if (__builtin_expect(left > p.H - h &&
                                 __builtin_amdgcn_readfirstlane(counts[i]) > kSearchFrom,
                             0)) {
            const uint32_t begin = i > 0 ? upto(i - 1) : 0u;
            known = min(min(upto(i), v + kSearchRun), v + (left + h + p.H - 1) / p.H);
            for (uint32_t x = v; x < known; x += kGroup)
                scatter_search(p, search, __builtin_amdgcn_readfirstlane(starts[i]),
                               __builtin_amdgcn_readfirstlane(counts[i]),
                               __builtin_amdgcn_readfirstlane((uint32_t)places[i]), x - begin, x,
                               min(kGroup, known - x));
        }
        while (left > 0) {
            const uint32_t take = min(left, p.H - h);
            const uint32_t c = v - (i > 0 ? upto(i - 1) : 0u);
            const uint64_t item0 = (rb + i) * p.H;  // the request's heads inside the window
            const uint32_t h0 = (uint32_t)(max(item0 + h, (uint64_t)item_begin) - item0);
            const uint32_t h1 = (uint32_t)(min(item0 + h + take, item_end) - item0);
            const uint32_t t0 = __builtin_amdgcn_readfirstlane(starts[i]);
            const uint32_t n = __builtin_amdgcn_readfirstlane(counts[i]);
            const uint32_t place = __builtin_amdgcn_readfirstlane((uint32_t)places[i]);
            const int64_t first = (int64_t)c * kStrip - place;
            if ((int32_t)(h1 - h0) > 0) {
                if ((v < known && __builtin_amdgcn_readfirstlane(search.found[v % kSearchRun])) ||
                    !scatter_chunk<D>(p, t0, n, first, v < known || n + place <= kStrip, h0, h1,
                                      sign, lds_t, clash_w))
                    scatter_tokens<D>(p, t0, n, first, h0, h1, sign);
            }
            lds_barrier();  // the next chunk writes clash_w and the first buffer again
            left -= take;
            h = 0;
            ++v;
            while (left > 0 && upto(i) <= v) ++i;
        }
        lds_barrier();
    }
}

// One-token requests (cu_seqlens NULL: the decode step's writer). A 16-lane
// row group takes one (token, kv head) item, sixteen items per workgroup;
// each lane rotates and quantises its channels of both planes. The value
// strip's column is merged in registers: a lane reads the 2 CPL consecutive
// strip words of its channels (channel c's 16 tokens are words 2c and
// 2c + 1), replaces its nibble in each and writes the words back. A strip
// has one owner per launch (the writer's contract), so writing back the
// words read is safe. The rows' loads go out with the slot's; the strip's
// load follows the slot.
template <int D>
__global__ __launch_bounds__(kWriterThreads) void scatter_token_writer(
    const uint16_t* __restrict__ key, const uint16_t* __restrict__ value,
    int8_t* __restrict__ key_cache, int8_t* __restrict__ value_cache,
    float* __restrict__ scale_cache, const int32_t* __restrict__ slots,
    const float* __restrict__ pi_signs, int32_t* __restrict__ probe, uint32_t probe_grid,
    uint32_t num_requests, uint32_t H, uint32_t S, uint32_t P, uint32_t item_begin,
    uint32_t item_count, float inv_sqrt_len)
{
    constexpr int CPL = D / 16;
    constexpr int NW = 2 * CPL;  // strip words of a lane's channels
    const int tid = threadIdx.x;
    const int grp = tid >> 4;
    const int l = row_lane(tid & 15);  // logical lane: channels l*CPL ..

    if (probe != nullptr && blockIdx.x == 0 && tid < 32) {
        const int32_t fields[4] = {0, (int32_t)probe_grid, 1, (int32_t)item_count};
        probe[tid] = fields[tid >> 3];
    }

    float sign[CPL];
    load_signs<CPL>(pi_signs, nullptr, 0, l * CPL, sign);
    const float sigma = row_sigma(l);
    auto one = [&](uint32_t request, uint32_t head) {
        if (request >= num_requests) return;
        // The rows do not depend on the slot: their loads go out with its
        // load. A pad or out-of-pool slot reads page 0's strip and stores
        // nothing (so no load waits behind a branch).
        const size_t src_off = ((size_t)request * H + head) * D + l * CPL;
        const int32_t slot = slots[request];
        float v[2][CPL];
        load_row<CPL>(key + src_off, v[0]);
        load_row<CPL>(value + src_off, v[1]);
        const uint32_t page_raw = (uint32_t)slot / S;
        const bool ok = slot >= 0 && page_raw < P;
        const uint32_t page = ok ? page_raw : 0u;
        const uint32_t tip = ok ? (uint32_t)slot - page_raw * S : 0u;
        const uint32_t col = tip % kStrip;
        const size_t head_base = ((size_t)page * H + head) * S;
        uint4* strip = (uint4*)(value_cache + (head_base + (tip - col)) * (D / 2)) + l * (NW / 4);
        uint32_t w[NW];
#pragma unroll
        for (int i = 0; i < NW / 4; ++i) {
            const uint4 u = strip[i];
            w[4 * i] = u.x;
            w[4 * i + 1] = u.y;
            w[4 * i + 2] = u.z;
            w[4 * i + 3] = u.w;
        }
        // exact policy: absmax as is; a zero row (every element +-0 or
        // NaN) stores codes 0 and scale 1.0
        writer_rotate<D, CPL>(v, sign, l);
        float a[2];
        writer_absmax<CPL>(v, 0.0f, a);
        int e[2];
        float sc[2];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            e[r] = a[r] == 0.0f ? 2 : exponent_of(a[r]);
            sc[r] = a[r] == 0.0f ? 1.0f : ldexpf(1.0f, e[r] - 2) * inv_sqrt_len;
        }
        // y = v * 2^(2-e) by ldexp (e may be as low as -149), then the
        // magic-number rounding with sigma folded into the multiplier: keys
        // with kQMagic (code + 8 in bits 0..3, packed), values with
        // kQMagic - 8 (the two's-complement nibble in bits 0..3, spliced)
        uint32_t tk[CPL], tv[CPL];
#pragma unroll
        for (int j = 0; j < CPL; ++j) {
            const float yk = a[0] == 0.0f ? 0.0f : ldexpf(v[0][j], 2 - e[0]);
            const float yv = a[1] == 0.0f ? 0.0f : ldexpf(v[1][j], 2 - e[1]);
            tk[j] = __float_as_uint(fminf(__builtin_fmaf(yk, sigma, kQMagic), kQMagicTop));
            tv[j] = __float_as_uint(
                fminf(__builtin_fmaf(yv, sigma, kQMagic - 8.0f), kQMagicTop - 8.0f));
        }
        if (!ok) return;
        if ((tid & 15) == 0) {
            scale_cache[((size_t)page * H + head) * S + tip] = sc[0];
            scale_cache[(((size_t)P + page) * H + head) * S + tip] = sc[1];
        }
        int8_t* kdst = key_cache + (head_base + tip) * (D / 2) + l * (CPL / 2);
        if constexpr (CPL == 16)
            *(uint2*)kdst = make_uint2(pack8(tk), pack8(&tk[8]));
        else if constexpr (CPL == 8)
            *(uint32_t*)kdst = pack8(tk);
        else
            *(uint16_t*)kdst = (uint16_t)pack4(tk);
        // the column's nibble in word 2j (tokens 0..7) or 2j + 1 (8..15):
        // both words take a bit-field insert, one under an empty mask (no
        // register array indexed by a lane value)
        const uint32_t sh = 4u * (col & 7u);
        const uint32_t m1 = (col >> 3) ? 0xfu << sh : 0u, m0 = (0xfu << sh) ^ m1;
#pragma unroll
        for (int j = 0; j < CPL; ++j) {
            const uint32_t y = tv[j] << sh;
            w[2 * j] = (w[2 * j] & ~m0) | (y & m0);
            w[2 * j + 1] = (w[2 * j + 1] & ~m1) | (y & m1);
        }
#pragma unroll
        for (int i = 0; i < NW / 4; ++i)
            strip[i] = make_uint4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
    };
    const uint64_t item_end = (uint64_t)item_begin + item_count;
    const uint32_t stride = gridDim.x * 16u;  // at most 4096 * 16
    if (item_end + stride <= 0xffffffffull) {
        // 32-bit item arithmetic: no item, nor the step past the last one,
        // reaches 2^32
        for (uint32_t item = item_begin + blockIdx.x * 16u + (uint32_t)grp;
             item < (uint32_t)item_end; item += stride)
            one(item / H, item % H);
    } else {
        for (uint64_t item = (uint64_t)item_begin + (uint64_t)blockIdx.x * 16u + (uint32_t)grp;
             item < item_end; item += (uint64_t)gridDim.x * 16u)
            one((uint32_t)(item / H), (uint32_t)(item % H));
    }
}

}  // namespace

// ------------------------------------------------------------- launchers
template <int D, typename In>
static hipError_t launch_strip_writer_t(hipStream_t stream, const In* key, const In* value,
                                        int8_t* key_cache, int8_t* value_cache, float* scale_cache,
                                        const int32_t* slots, const float* pi_signs,
                                        const void* tables, int tables_bf16, uint32_t strips,
                                        uint32_t H, uint32_t S, uint32_t P, float inv_sqrt_len)
{
    // One head per workgroup (two row jobs per lane) measured faster than
    // two (four jobs): with one wave per SIMD nothing hides the rotation's
    // dependent lane exchanges.
    if (strips == 0 || H == 0) return hipSuccess;
    if (H > 65535u) return hipErrorInvalidValue;
    hipLaunchKernelGGL((strip_writer<D, In>), dim3(strips, H), dim3(kWriterThreads), 0, stream,
                       key, value, key_cache, value_cache, scale_cache, slots, pi_signs, tables,
                       tables_bf16, H, S, P, inv_sqrt_len);
    return hipGetLastError();
}

hipError_t launch_strip_writer(hipStream_t stream, int in_bf16, const void* key,
                               const void* value, int8_t* key_cache, int8_t* value_cache,
                               float* scale_cache, const int32_t* slots, const float* pi_signs,
                               const void* tables, uint32_t strips, uint32_t H, uint32_t D,
                               uint32_t S, uint32_t P, float inv_sqrt_len)
{
#define TQ4_STRIP_CASE(DD)                                                                        \
    if (D == DD) {                                                                                \
        if (in_bf16)                                                                              \
            return launch_strip_writer_t<DD, uint16_t>(                                           \
                stream, (const uint16_t*)key, (const uint16_t*)value, key_cache, value_cache,     \
                scale_cache, slots, pi_signs, tables, 1, strips, H, S, P, inv_sqrt_len);          \
        return launch_strip_writer_t<DD, int8_t>(stream, (const int8_t*)key, (const int8_t*)value, \
                                                 key_cache, value_cache, scale_cache, slots,      \
                                                 pi_signs, tables, 0, strips, H, S, P,            \
                                                 inv_sqrt_len);                                   \
    }
    TQ4_STRIP_CASE(64)
    TQ4_STRIP_CASE(128)
    TQ4_STRIP_CASE(256)
#undef TQ4_STRIP_CASE
    return hipErrorInvalidValue;
}

hipError_t launch_scatter_writer(hipStream_t stream, uint32_t grid, const uint16_t* key,
                                 const uint16_t* value, int8_t* key_cache, int8_t* value_cache,
                                 float* scale_cache, const int32_t* slots, const float* pi_signs,
                                 const int32_t* cu_seqlens, int32_t* probe, uint32_t num_requests,
                                 uint32_t H, uint32_t D, uint32_t S, uint32_t P,
                                 uint32_t item_begin, uint32_t item_count, float inv_sqrt_len)
{
    // one-token requests: sixteen items per workgroup, a grid covering them
    // (at most 4096 workgroups, striding beyond); `grid` is still what the
    // launch probe reports
    const uint64_t groups = ((uint64_t)item_count + 15) / 16;
    const uint32_t tgrid = (uint32_t)(groups < 4096 ? groups : 4096);
    const ScatterArgs args{key, value, key_cache, value_cache, scale_cache, slots, H, S, P,
                           inv_sqrt_len};
#define TQ4_SCATTER_CASE(DD)                                                                      \
    if (D == DD) {                                                                                \
        if (cu_seqlens == nullptr)                                                                \
            hipLaunchKernelGGL((scatter_token_writer<DD>), dim3(tgrid), dim3(kWriterThreads), 0, \
                               stream, key, value, key_cache, value_cache, scale_cache, slots,    \
                               pi_signs, probe, grid, num_requests, H, S, P, item_begin,          \
                               item_count, inv_sqrt_len);                                         \
        else                                                                                      \
            hipLaunchKernelGGL((scatter_writer<DD>), dim3(kScatterGrid<DD>), dim3(kWriterThreads), 0, \
                               stream, args, pi_signs, cu_seqlens, probe, grid, num_requests,     \
                               item_begin, item_count);                                           \
        return hipGetLastError();                                                                 \
    }
    TQ4_SCATTER_CASE(64)
    TQ4_SCATTER_CASE(128)
    TQ4_SCATTER_CASE(256)
#undef TQ4_SCATTER_CASE
    return hipErrorInvalidValue;
}

}  // namespace tq4
