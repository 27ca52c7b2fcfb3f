// Prefill attention at head width 64 on binary16 matrix cores, f32-exact
// operands split in halves.
//
// Flash-style causal GQA for many (token, query head) pairs.  A block of
// kWaves waves serves one key/value head and kRows query rows: `tile_tokens`
// consecutive tokens times the group's query heads (row r is token t0 + r /
// group, query head r % group of the key/value head); each wave owns 16 rows.
// Key and value rows stream through LDS in kKeys-key tiles that every row of
// the block shares.
//
// Exactness plan.  Every operand is a power of two times hi + lo binary16
// halves: a query row by its own largest magnitude, a key tile by the tile's,
// a value tile by the largest seen so far (the output accumulators are
// rescaled when it grows), probabilities by 2^7 (they stay below 2^8).  The
// largest magnitude sits below 2^15, so a value keeps 22 bits down to 2^-18 of it and an absolute
// error of 2^-40 of it below that.  Products are exact in f32; lo * lo, below
// 2^-22 of each term, is dropped.  Scores, the softmax and all sums are f32.
// Where a key or value of a block's range is infinite, or a wave's query is not
// finite, the rows are computed again on v_mfma_f32_16x16x4_f32 from the f32
// values, so infinities act as in f32 arithmetic (NaN does in both halves).  A
// key the causal mask hides gets probability zero; a non-finite value row later
// in the same tile still reaches the earlier rows (0 * NaN), where the
// reference skips it (attention_convolution.rs:90-170).
//
// Per tile, S^T = K Q^T leaves row j of a wave in lane column j: lane 16q + j
// holds the scores of keys 16c + 4q + r in register r of column block c.  The
// running maximum, the exponent sum and the output rescale stay in the row's
// own four lanes.  The output accumulates as O^T = V^T P^T, whose B operand of
// 32 keys is the lane's own probabilities of two column blocks; V^T is staged
// in that key order.
//
// LDS holds each operand in 16-byte chunks, [16-row tile][chunk][row], so a
// wave's operand read is one contiguous KB; the row index is swizzled to spread
// the staging writes over the banks.
//
// Bound.  Per wave and tile 48 MFMAs (768 cycles) against about 290 vector
// instructions of softmax and splitting, the two overlapping across the four
// waves of a SIMD; the causal triangle leaves 2.4 of them busy on average.
// 2048 tokens, 32 / 8 heads: 101 us per call with the cache append, against 227
// for the fp32 matrix cores this replaces (128 MFMAs of 32 cycles per tile);
// error against 64-bit sums 2.6e-7 (before: 4.0e-7).  One 16-wave block per CU
// whose halves take tiles in turn measured 104 us.
#include <algorithm>

#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace mfh {
namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v2f __attribute__((ext_vector_type(2)));

constexpr int kWaves = 8;  // of 16 rows each
constexpr uint32_t kThreads = 64 * kWaves;
constexpr uint32_t kRows = 16 * kWaves;
constexpr uint32_t kKeys = 64;
constexpr uint32_t kDim = 64;
constexpr uint32_t kPlane = kKeys * kDim * 2;  // one half of one operand tile
constexpr int kTop = 15;                       // scaled magnitudes stay below 2^kTop
constexpr int kSlack = 8;                      // p stays below 2^kSlack
constexpr int kMinExponent = -90;              // smaller values keep this scale

// Byte offset of row `row`'s 16-byte chunk `chunk` (of 8) in a plane.
__device__ __forceinline__ uint32_t key_at(uint32_t row, uint32_t chunk)
{
    return (row >> 4) * 2048 + chunk * 256 + (((row & 15) ^ ((chunk & 1) << 3)) << 4);
}
__device__ __forceinline__ uint32_t value_at(uint32_t dim, uint32_t chunk)
{
    return (dim >> 4) * 2048 + chunk * 256 + (((dim & 15) ^ ((dim >> 4) & 1)) << 4);
}

__device__ __forceinline__ uint32_t magnitude(float x)
{
    return __builtin_bit_cast(uint32_t, x) & 0x7fffffffu;
}

constexpr uint32_t kInfBits = 0x7f800000u;

// The exponent e with every magnitude pattern up to `bits` (finite) below 2^e.
__device__ __forceinline__ int exponent_of(uint32_t bits)
{
    const int e = int(bits >> 23) - 126;
    return e < kMinExponent ? kMinExponent : e;
}

// 2^e, -126 <= e <= 127.
__device__ __forceinline__ float power_of_two(int e)
{
    return __builtin_bit_cast(float, uint32_t(e + 127) << 23);
}

__device__ __forceinline__ uint32_t larger(uint32_t a, uint32_t b) { return a > b ? a : b; }

// max(a, |b|, |c|); NaN operands are ignored.
__device__ __forceinline__ float max3_abs(float a, float b, float c)
{
    float r;
    asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// Maximum over the wave of a magnitude's bits: DPP within the 16-lane rows,
// then row swaps.
__device__ __forceinline__ uint32_t wave_max_bits(float m)
{
    uint32_t v = __float_as_uint(m);
    v = larger(v, uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0xB1, 0xF, 0xF, true)));   // xor 1
    v = larger(v, uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0x4E, 0xF, 0xF, true)));   // xor 2
    v = larger(v, uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0x141, 0xF, 0xF, true)));  // half mirror
    v = larger(v, uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0x140, 0xF, 0xF, true)));  // mirror
    const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = larger(a[0], a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return larger(b[0], b[1]);
}

// Maximum and sum over a row's four lanes (q = 0..3).
__device__ __forceinline__ float quad_max(float v)
{
    const uint32_t x = __builtin_bit_cast(uint32_t, v);
    const auto a = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const uint32_t y = __builtin_bit_cast(uint32_t, v);
    const auto b = __builtin_amdgcn_permlane32_swap(y, y, false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float quad_sum(float v)
{
    const uint32_t x = __builtin_bit_cast(uint32_t, v);
    const auto a = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const uint32_t y = __builtin_bit_cast(uint32_t, v);
    const auto b = __builtin_amdgcn_permlane32_swap(y, y, false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// hi + lo of x * scale.  (Adding zero keeps both on the mixed-precision FMA,
// which rounds straight to binary16.)
template <int N, typename F, typename H>
__device__ __forceinline__ void split(const F &x, float scale, H &hi, H &lo)
{
#pragma unroll
    for (int i = 0; i < N; ++i) {
        hi[i] = _Float16(fmaf(x[i], scale, 0.0f));
        lo[i] = _Float16(fmaf(x[i], scale, -float(hi[i])));
    }
}

__global__ __launch_bounds__(kThreads, 4) void gqa_flash_split_kernel(
    float *__restrict__ out, const float *__restrict__ query, const float *__restrict__ key_cache,
    const float *__restrict__ value_cache, GqaShape g, uint32_t tile_tokens, uint32_t token_tiles,
    bool paired, uint32_t ranges, uint32_t range_tiles, float *__restrict__ records)
{
    __shared__ __align__(1024) uint8_t lds[2][4 * kPlane];  // K hi, K lo, V^T hi, V^T lo
    __shared__ uint32_t wave_bits[2][2][kWaves];

    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t q = lane >> 4, j = lane & 15;
    const uint32_t kv_heads = g.key_value_heads, group = g.group;
    const uint32_t kv_head = blockIdx.x % kv_heads;
    const uint32_t range = blockIdx.x / kv_heads % ranges, nth = blockIdx.x / kv_heads / ranges;
    // Longest token tiles (most keys) first; where the whole grid is resident,
    // its second half runs shortest first, beside the first half's long ones.
    const uint32_t half = (token_tiles + 1) / 2;
    const uint32_t tile = paired && nth >= half ? nth - half : token_tiles - 1 - nth;
    const uint32_t start = uint32_t(g.initial_len), tokens = uint32_t(g.tokens);
    const uint32_t t0 = tile * tile_tokens;
    const uint32_t t_end = t0 + tile_tokens < tokens ? t0 + tile_tokens : tokens;
    const uint32_t k_end = start + t_end;  // keys [0, k_end) reach some row
    const size_t kv_width = size_t(kv_heads) * kDim;
    const float *const keys = key_cache + kv_head * kDim;
    const float *const values = value_cache + kv_head * kDim;

    // The lane's row.  Rows past the tile (or past the last token) compute
    // over every staged key and store nothing.
    const uint32_t row = 16 * wave + j;
    const uint32_t token = t0 + row / group;
    const uint32_t head = kv_head * group + row % group;
    const bool valid = row < tile_tokens * group && token < tokens;
    const uint32_t last = valid ? start + token : k_end - 1;  // last visible key
    const uint32_t wave_first = start + t0 + 16 * wave / group;         // smallest `last`
    const uint32_t wave_last = start + t0 + (16 * wave + 15) / group;  // largest stored `last`
    const float *const q_row = query + (size_t(valid ? token : 0) * g.query_heads + head) * kDim;

    // Q^T operand: dimensions 32s + 8q + e of the row at step s.
    v8h qh[2], ql[2];
    float row_scale;  // of the scores: 1 / sqrt(d), log2(e) and the row's power of two
    bool q_bad;
    constexpr float kLog2e = 1.44269504088896341f;
    {
        float f[2][8];
        uint32_t bits = 0;
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const v4f v = valid ? *reinterpret_cast<const v4f *>(q_row + 32 * s + 8 * q + 4 * h)
                                    : v4f{0, 0, 0, 0};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    f[s][4 * h + e] = v[e];
                    bits = larger(bits, magnitude(v[e]));
                }
            }
        bits = larger(bits, __shfl_xor(bits, 16, 64));
        bits = larger(bits, __shfl_xor(bits, 32, 64));
        q_bad = __any(bits >= kInfBits);
        const int e = bits >= kInfBits ? 0 : exponent_of(bits);
#pragma unroll
        for (int s = 0; s < 2; ++s)
            split<8>(f[s], power_of_two(kTop - e), qh[s], ql[s]);
        row_scale = g.scale * kLog2e * power_of_two(e - kTop);
    }

    // Staging: a thread loads chunk `tid % 8` of key `tid / 8`, and dimensions
    // 2b, 2b + 1 of keys 4a..4a + 3.
    const uint32_t k_key = tid / 8, k_chunk = tid % 8;
    const uint32_t v_quad = tid / 32, v_pair = tid % 32;
    v4f kr[2];
    v2f vr[4];
    // Rows past the end repeat the last one: the mask hides their scores, and
    // as values they meet probability zero.
    const uint32_t row_bytes = uint32_t(kv_width) * 4;
    auto stage_load = [&](uint32_t n) {
        const uint32_t k0 = n * kKeys, most = k_end - 1 - k0;
        const char *const kt = reinterpret_cast<const char *>(keys + k0 * kv_width);
        const char *const vt = reinterpret_cast<const char *>(values + k0 * kv_width);
        const uint32_t k_off = min(k_key, most) * row_bytes + 32 * k_chunk;
        kr[0] = *reinterpret_cast<const v4f *>(kt + k_off);
        kr[1] = *reinterpret_cast<const v4f *>(kt + k_off + 16);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            vr[i] = *reinterpret_cast<const v2f *>(
                vt + min(4 * v_quad + i, most) * row_bytes + 8 * v_pair);
    };

    // What a staged tile's halves are scaled by.
    struct Scales {
        int v_exp = kMinExponent;  // values: 2^(kTop - v_exp), growing with the tiles
        float k_unit = 1.0f;       // keys: their power of two
        bool bad = false;          // an infinity: nothing is staged
    };
    auto publish = [&](uint32_t slot, float a, float b) {
        const uint32_t a_bits = wave_max_bits(a), b_bits = wave_max_bits(b);
        if (lane == 0) {
            wave_bits[slot][0][wave] = a_bits;
            wave_bits[slot][1][wave] = b_bits;
        }
    };
    auto block_max = [&](uint32_t slot, uint32_t which) {
        uint32_t v = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w)
            v = larger(v, wave_bits[slot][which][w]);
        return uint32_t(__builtin_amdgcn_readfirstlane(int(v)));
    };
    // The loaded tile's largest magnitudes (before the barrier) ...
    auto stage_max = [&](uint32_t slot) {
        float km = 0.0f, vm = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            km = max3_abs(km, kr[i / 2][2 * (i % 2)], kr[i / 2][2 * (i % 2) + 1]);
            vm = max3_abs(vm, vr[i][0], vr[i][1]);
        }
        publish(slot, km, vm);
    };
    // ... and its halves (after it).
    auto stage_store = [&](uint32_t slot, Scales &t) {
        const uint32_t k_bits = block_max(slot, 0), v_bits = block_max(slot, 1);
        t.bad = larger(k_bits, v_bits) >= kInfBits;
        if (t.bad)
            return;
        const int ve = exponent_of(v_bits);
        t.v_exp = ve > t.v_exp ? ve : t.v_exp;
        const int ke = exponent_of(k_bits);
        t.k_unit = power_of_two(ke - kTop);
        const float ks = power_of_two(kTop - ke), vs = power_of_two(kTop - t.v_exp);
        uint8_t *const k_hi = lds[slot], *const v_hi = k_hi + 2 * kPlane;
        v8h hi, lo;
        float f[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            f[i] = kr[i / 4][i % 4];
        split<8>(f, ks, hi, lo);
        *reinterpret_cast<v8h *>(k_hi + key_at(k_key, k_chunk)) = hi;
        *reinterpret_cast<v8h *>(k_hi + kPlane + key_at(k_key, k_chunk)) = lo;
        // Keys 4a..4a + 3 of 32-key step t are the low (a % 8 < 4) or high
        // half of the chunk of lane block a % 4.
        const uint32_t chunk = v_quad / 8 * 4 + v_quad % 4, high = v_quad % 8 / 4 * 8;
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            const float x[4] = {vr[0][d], vr[1][d], vr[2][d], vr[3][d]};
            v4h vh, vl;
            split<4>(x, vs, vh, vl);
            const uint32_t at = value_at(2 * v_pair + d, chunk) + high;
            *reinterpret_cast<v4h *>(v_hi + at) = vh;
            *reinterpret_cast<v4h *>(v_hi + kPlane + at) = vl;
        }
    };

    v4f o[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
        o[u] = v4f{0, 0, 0, 0};
    int o_exp = kMinExponent;  // the value scale of the wave's accumulators
    float m = -__builtin_inff(), l = 0.0f;  // m in log2 units
    // The block's key tiles.
    const uint32_t tiles = (k_end + kKeys - 1) / kKeys;
    const uint32_t begin = range * range_tiles;
    const uint32_t end = begin + range_tiles < tiles ? begin + range_tiles : tiles;
    Scales next;
    if (begin < end) {
        stage_load(begin);
        stage_max(begin & 1);
        __syncthreads();
        stage_store(begin & 1, next);
        if (begin + 1 < end)
            stage_load(begin + 1);
    }
    // Per tile one barrier: behind it the tile's halves are complete and the
    // buffer of the tile before is free, so the next tile (in registers since
    // the last one) is split into it and the one after requested while this one
    // is multiplied.
    for (uint32_t n = begin; n < end; ++n) {
        const uint32_t k0 = n * kKeys;
        const Scales cur = next;
        const uint8_t *const k_hi = lds[n & 1], *const v_hi = k_hi + 2 * kPlane;
        if (n + 1 < end)
            stage_max((n + 1) & 1);
        __syncthreads();
        if (cur.bad)
            break;
        if (n + 1 < end)
            stage_store((n + 1) & 1, next);
        if (n + 2 < end)
            stage_load(n + 2);
        if (k0 <= wave_last && !q_bad) {
            // S^T = K Q^T.
            v4f s[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                v4f acc = {0, 0, 0, 0};
#pragma unroll
                for (int st = 0; st < 2; ++st) {
                    const uint32_t at = key_at(16 * c + j, 4 * st + q);
                    const v8h kh = *reinterpret_cast<const v8h *>(k_hi + at);
                    const v8h kl = *reinterpret_cast<const v8h *>(k_hi + kPlane + at);
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(kl, qh[st], acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh, ql[st], acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh, qh[st], acc, 0, 0, 0);
                }
                s[c] = acc;
            }
            const float unit = fminf(fmaxf(row_scale * cur.k_unit, __FLT_MIN__), __FLT_MAX__);
            // Causal mask, online softmax over the row's four lanes.
            if (k0 + kKeys - 1 > wave_first || k0 + kKeys > k_end) {
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (k0 + 16 * c + 4 * q + r > last)
                            s[c][r] = -__builtin_inff();
            }
            // The reference m of the exponents follows the running maximum
            // only when that has grown by more than 2^kSlack, so most tiles
            // leave the accumulators alone; p stays below 2^kSlack.
            float mx = s[0][0];
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int r = c == 0 ? 1 : 0; r < 4; ++r)
                    mx = fmaxf(mx, s[c][r]);
            mx = quad_max(mx) * unit;
            const int shrink = o_exp - cur.v_exp;
            if (__any(mx > m + kSlack) || shrink != 0) {
                // A row without a visible key so far keeps m = -inf, l = 0.
                const float m_new = fmaxf(m, mx);
                const float alpha =
                    m_new == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(m - m_new);
                m = m_new;
                l *= alpha;
                const float rescale = alpha * (shrink < -126 ? 0.0f : power_of_two(shrink));
                o_exp = cur.v_exp;
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    o[u] *= rescale;
            }
            const float m_ref = m == -__builtin_inff() ? 0.0f : m;
            v8h ph[2], pl[2];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                float p[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    p[r] = __builtin_amdgcn_exp2f(fmaf(s[c][r], unit, -m_ref));
                    l += p[r];
                    s[c][r] = p[r];
                }
                v4h hi, lo;
                split<4>(p, power_of_two(kTop - kSlack), hi, lo);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    ph[c / 2][4 * (c % 2) + r] = hi[r];
                    pl[c / 2][4 * (c % 2) + r] = lo[r];
                }
            }
            // O^T += V^T P^T.
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int st = 0; st < 2; ++st) {
                    const uint32_t at = value_at(16 * u + j, 4 * st + q);
                    const v8h vh = *reinterpret_cast<const v8h *>(v_hi + at);
                    const v8h vl = *reinterpret_cast<const v8h *>(v_hi + kPlane + at);
                    o[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vl, ph[st], o[u], 0, 0, 0);
                    o[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh, pl[st], o[u], 0, 0, 0);
                    o[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh, ph[st], o[u], 0, 0, 0);
                }
        }
    }
    // The accumulators carry the scales of p and of the values.
    float unscale = power_of_two(o_exp - 2 * kTop + kSlack);
    if (next.bad || q_bad) {
        // An infinity among the range's keys or values, or a non-finite query
        // of this wave: the rows over again in f32, straight from memory.
        unscale = 1.0f;
        m = -__builtin_inff();
        l = 0.0f;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            o[u] = v4f{0, 0, 0, 0};
        const float unit = g.scale * kLog2e;
#pragma unroll 1
        for (uint32_t k0 = begin * kKeys; k0 < end * kKeys && k0 <= wave_last; k0 += 16) {
            // 16 keys: scores of key 4q + r, operand key j.
            v4f s = {0, 0, 0, 0};
            const float *const kp = keys + size_t(min(k0 + j, k_end - 1)) * kv_width + 4 * q;
#pragma unroll 1
            for (uint32_t at = 0; at < kDim; at += 16) {
                const v4f kk = *reinterpret_cast<const v4f *>(kp + at);
                const v4f qq = *reinterpret_cast<const v4f *>(q_row + 4 * q + at);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    s = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[e], qq[e], s, 0, 0, 0);
            }
            float mx = -__builtin_inff();
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s[r] = k0 + 4 * q + r > last ? -__builtin_inff() : s[r] * unit;
                mx = fmaxf(mx, s[r]);
            }
            const float m_new = fmaxf(m, quad_max(mx));
            const float m_ref = m_new == -__builtin_inff() ? 0.0f : m_new;
            const float alpha = __builtin_amdgcn_exp2f(m - m_ref);
            m = m_new;
            l *= alpha;
#pragma unroll
            for (int u = 0; u < 4; ++u)
                o[u] *= alpha;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float p = __builtin_amdgcn_exp2f(s[r] - m_ref);
                l += p;
                const float *const vp =
                    values + size_t(min(k0 + 4 * q + r, k_end - 1)) * kv_width + j;
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    o[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(vp[16 * u], p, o[u], 0, 0, 0);
            }
        }
    }
    l = quad_sum(l);  // each lane holds its own keys' share
    if (!valid)
        return;
    const size_t pair = size_t(token) * g.query_heads + head;
    if (ranges > 1) {
        // The range's record: maximum, exponent sum, unnormalised output.
        float *const rec = records + (pair * ranges + range) * (kDim + 2);
        if (q == 0) {
            rec[0] = m;
            rec[1] = l;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                rec[2 + 16 * u + 4 * q + e] = o[u][e] * unscale;
        return;
    }
    float *const o_row = out + pair * kDim;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        v4f r;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            r[e] = o[u][e] / l * unscale;
        *reinterpret_cast<v4f *>(o_row + 16 * u + 4 * q) = r;
    }
}

// One wave per (token, query head), lane = dimension: the ranges' records
// merged at their largest maximum.  A range without a visible key stores
// l = 0 and is skipped.
__global__ __launch_bounds__(256) void gqa_flash_merge_kernel(float *__restrict__ out,
                                                              const float *__restrict__ records,
                                                              uint32_t ranges, uint32_t pairs)
{
    const uint32_t pair = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (pair >= pairs)
        return;
    const float *const rec = records + size_t(pair) * ranges * (kDim + 2);
    float m = -__builtin_inff();
    for (uint32_t r = 0; r < ranges; ++r)
        if (rec[r * (kDim + 2) + 1] != 0.0f)
            m = fmaxf(m, rec[r * (kDim + 2)]);
    float l = 0.0f, o = 0.0f;
    for (uint32_t r = 0; r < ranges; ++r) {
        const float *const at = rec + r * (kDim + 2);
        if (at[1] == 0.0f)
            continue;
        const float w = __builtin_amdgcn_exp2f(at[0] - m);
        l = fmaf(at[1], w, l);
        o = fmaf(at[2 + lane], w, o);
    }
    out[size_t(pair) * kDim + lane] = o / l;
}

struct Grid {
    uint32_t tile_tokens, token_tiles, ranges, range_tiles;
};

// Blocks the CUs hold at once, two each (128 registers, 64 KB of LDS).
constexpr uint32_t kResident = 512;

// A launch that leaves most CUs idle cuts its keys into ranges of at least four
// tiles, whose records a second launch merges: 64 tokens over 2000 keys (32 / 8
// heads) 112 -> 24 us, 1024 over 1024 (16 / 4) 111 -> 57.  Fuller launches lose
// by the records' traffic (2048 tokens 101 unsplit, 141 in two ranges).
// Of a served call: at least one token, so at least one block.
Grid grid_of(const GqaShape &g, bool records)
{
    Grid d;
    d.tile_tokens = kRows / g.group;
    d.token_tiles = uint32_t((g.tokens + d.tile_tokens - 1) / d.tile_tokens);
    d.ranges = 1;
    d.range_tiles = uint32_t((g.initial_len + g.tokens + kKeys - 1) / kKeys);
    const uint32_t blocks = d.token_tiles * g.key_value_heads;
    if (records && blocks <= kResident / 2) {
        const uint32_t most = std::min(kResident / blocks, d.range_tiles / 4);
        if (most > 1) {
            d.range_tiles = (d.range_tiles + most - 1) / most;
            d.ranges = uint32_t((g.initial_len + g.tokens + kKeys * d.range_tiles - 1) /
                                (kKeys * d.range_tiles));
        }
    }
    return d;
}

}  // namespace

bool gqa_flash_split_served(const GqaShape &g)
{
    return g.tokens >= 1 && g.head_dim == kDim && g.group >= 1 && g.group <= kRows &&
           g.key_value_heads <= 65536 && g.initial_len + g.tokens < (uint64_t(1) << 31);
}

size_t gqa_flash_records_bytes(const GqaShape &g)
{
    const Grid d = grid_of(g, true);
    return d.ranges > 1 ? size_t(g.tokens) * g.query_heads * d.ranges * (kDim + 2) * sizeof(float)
                        : 0;
}

void launch_gqa_flash_split(hipStream_t stream, float *out, const float *query,
                            const float *key_cache, const float *value_cache, const GqaShape &g,
                            float *records)
{
    const Grid d = grid_of(g, records != nullptr);
    gqa_flash_split_kernel<<<d.token_tiles * d.ranges * g.key_value_heads, kThreads, 0,
                             stream>>>(out, query, key_cache, value_cache, g, d.tile_tokens,
                                       d.token_tiles, d.token_tiles * g.key_value_heads <= kResident && d.ranges == 1,
                             d.ranges, d.range_tiles, records);
    if (d.ranges > 1) {
        const uint32_t pairs = uint32_t(g.tokens) * g.query_heads;
        gqa_flash_merge_kernel<<<(pairs + 3) / 4, 256, 0, stream>>>(out, records, d.ranges, pairs);
    }
}

}  // namespace mfh
