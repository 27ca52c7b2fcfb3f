// Prefill attention at head width 64 on bfloat16 matrix cores, f32 operands split
// in three parts.
//
// Flash-style causal GQA for many (token, query head) pairs.  A block serves one
// key/value head and kRows query rows: `tile_tokens` consecutive tokens times the
// group's query heads (row r is token t0 + r / group, query head r % group of the
// key/value head).  Its one or two teams of kWaves waves, 16 rows each, take the
// kKeys-key tiles in turn, each through LDS tiles of its own that every row of the
// team shares, and the first team adds the second's rows to its own in the end.
//
// Exactness plan.  Every query, key, value and probability is the sum of three
// bfloat16 parts that hold all 24 bits (bfloat16 has the exponents of f32, so no
// scale is shared between elements).  Of the nine products of parts the three
// below 2^-23 of a term are left out; products are exact in f32.  Scores, the
// softmax and all sums are f32, and a tile's share of the output is summed by
// itself before it is added.  Where the largest of eight staged values is past
// 2^60 (an infinity, or one whose parts or products could overflow) or below 2^-100
// (whose parts are subnormal), or eight of a wave's query are, the rows are
// computed again on v_mfma_f32_16x16x4_f32 from the f32 values (NaN acts alike in
// both).  A key the causal mask hides gets probability zero; a non-finite value row
// later in the same tile still reaches the earlier rows (0 * NaN), where the
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
// wave's operand read is one contiguous KB; the row index is swizzled so that the
// staging writes of 16 (keys) and 32 (values) lanes fall on distinct banks.
//
// Bound.  Per wave and tile 96 MFMAs (1536 cycles) and about 350 vector
// instructions (1400 cycles) of softmax and splitting, which hardly overlap: they
// take 80 % of the time.  2048 tokens, 32 / 8 heads: 117 us per call with the cache
// append, 227 on the fp32 matrix cores (128 MFMAs of 32 cycles per tile), 100 on
// binary16 hi + lo halves with shared scales, which lost small values beside large
// ones; error against 64-bit sums 1.8e-7 (fp32 matrix cores 4.0e-7, halves 2.6e-7;
// summing the tiles in one chain 3.2e-7).  One team of eight waves per block, two
// blocks per CU, measured 136 us (the causal triangle leaves a CU one long block);
// two teams of four waves with 32 rows each 126.
#include <algorithm>

#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace mfh {
namespace {

typedef __bf16 v8b __attribute__((ext_vector_type(8)));
typedef __bf16 v2b __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));

constexpr int kWaves = 8;  // per team, of 16 rows each
constexpr uint32_t kThreads = 64 * kWaves;  // per team
constexpr uint32_t kRows = 16 * kWaves;
constexpr uint32_t kKeys = 64;
constexpr uint32_t kDim = 64;
constexpr int kParts = 3;                      // bfloat16 parts of an operand
constexpr uint32_t kPlane = kKeys * kDim * 2;  // one part of one operand tile
constexpr int kSlack = 8;                      // p stays below 2^kSlack
// Magnitudes whose parts are normal and whose products are finite.
constexpr float kSmallest = 0x1p-100f, kLargest = 0x1p60f;

// Byte offset of row `row`'s 16-byte chunk `chunk` (of 8) in a plane.
__device__ __forceinline__ uint32_t key_at(uint32_t row, uint32_t chunk)
{
    return (row >> 4) * 2048 + chunk * 256 + (((row & 15) ^ (2 * chunk)) << 4);
}
__device__ __forceinline__ uint32_t value_at(uint32_t dim, uint32_t chunk)
{
    return (dim >> 4) * 2048 + chunk * 256 + (((dim & 15) ^ ((dim >> 4) & 1)) << 4);
}

// max(a, |b|, |c|); NaN operands are ignored.
__device__ __forceinline__ float max3_abs(float a, float b, float c)
{
    float r;
    asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// Whether x's largest magnitude is neither zero nor in the range of the parts.
template <int N, typename F>
__device__ __forceinline__ bool out_of_range(const F &x)
{
    static_assert(N % 2 == 0, "pairs");
    float most = 0.0f;
#pragma unroll
    for (int i = 0; i < N; i += 2)
        most = max3_abs(most, x[i], x[i + 1]);
    return most > kLargest || (most < kSmallest && most != 0.0f);
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

// x[0..N) as N / 2 dwords of bfloat16 pairs in each of three parts: every part is
// the nearest bfloat16 of what the ones before it left, and the three hold all 24
// bits.
template <int N, typename F, typename P>
__device__ __forceinline__ void split(const F &x, P &hi, P &mid, P &lo)
{
    auto nearest = [](float a, float b) {
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{a, b}, v2b));
    };
    auto first = [](uint32_t pair) { return __uint_as_float(pair << 16); };
    auto second = [](uint32_t pair) { return __uint_as_float(pair & 0xffff0000u); };
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
        float a = x[2 * i], b = x[2 * i + 1];
        hi[i] = nearest(a, b);
        a -= first(hi[i]);
        b -= second(hi[i]);
        mid[i] = nearest(a, b);
        a -= first(mid[i]);
        b -= second(mid[i]);
        lo[i] = nearest(a, b);
    }
}

// c + a b without the products below 2^-24 of a term, smallest first.
struct Parts {
    v4u hi, mid, lo;
};
__device__ __forceinline__ v4f multiply_add(const v4u &a, const v4u &b, const v4f &c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8b, a),
                                                   __builtin_bit_cast(v8b, b), c, 0, 0, 0);
}
__device__ __forceinline__ v4f multiply_add(const Parts &a, const Parts &b, v4f c)
{
    c = multiply_add(a.lo, b.hi, c);
    c = multiply_add(a.hi, b.lo, c);
    c = multiply_add(a.mid, b.mid, c);
    c = multiply_add(a.mid, b.hi, c);
    c = multiply_add(a.hi, b.mid, c);
    return multiply_add(a.hi, b.hi, c);
}

template <int TEAMS>
__global__ __launch_bounds__(TEAMS * kThreads, 4) void gqa_flash_split_kernel(
    float *__restrict__ out, const float *__restrict__ query, const float *__restrict__ key_cache,
    const float *__restrict__ value_cache, GqaShape g, uint32_t tile_tokens, uint32_t token_tiles,
    uint32_t ranges, uint32_t range_tiles, float *__restrict__ records)
{
    // Per team the parts of a key tile and of a transposed value tile; in the end
    // the second team's accumulators.
    constexpr uint32_t kTile = kParts * kPlane;
    __shared__ __align__(1024) uint8_t lds[TEAMS][2 * kTile];
    // The parts of the rows' queries, [part][step].
    __shared__ __align__(1024) v4u q_lds[kParts][2][kThreads];
    __shared__ uint32_t any_bad;
    if (threadIdx.x == 0)
        any_bad = 0;

    const uint32_t tid = threadIdx.x % kThreads, lane = tid & 63;
    const uint32_t team = __builtin_amdgcn_readfirstlane(threadIdx.x / kThreads);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint8_t *const k_lds = lds[team], *const v_lds = k_lds + kTile;
    const uint32_t q = lane >> 4, j = lane & 15;
    const uint32_t kv_heads = g.key_value_heads, group = g.group;
    const uint32_t kv_head = blockIdx.x % kv_heads;
    const uint32_t range = blockIdx.x / kv_heads % ranges;
    // Longest token tiles (most keys) first: a CU that is done takes a shorter one.
    const uint32_t tile = token_tiles - 1 - blockIdx.x / kv_heads / ranges;
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
    // The last visible key, less the lane's first one of 16.
    const int reach = int(valid ? start + token : k_end - 1) - int(4 * q);
    const uint32_t wave_first = start + t0 + 16 * wave / group;         // smallest last key
    const uint32_t wave_last = start + t0 + (16 * wave + 15) / group;  // largest stored one
    const float *const q_row = query + (size_t(valid ? token : 0) * g.query_heads + head) * kDim;

    // Q^T operand: dimensions 32s + 8q + e of the row at step s.
    bool q_bad = false;  // of the wave
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        float f[8];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const v4f v = valid ? *reinterpret_cast<const v4f *>(q_row + 32 * s + 8 * q + 4 * h)
                                : v4f{0, 0, 0, 0};
#pragma unroll
            for (int e = 0; e < 4; ++e)
                f[4 * h + e] = v[e];
        }
        q_bad |= __any(out_of_range<8>(f));
        if (team == 0) {
            Parts p;
            split<8>(f, p.hi, p.mid, p.lo);
            q_lds[0][s][tid] = p.hi;
            q_lds[1][s][tid] = p.mid;
            q_lds[2][s][tid] = p.lo;
        }
    }
    constexpr float kLog2e = 1.44269504088896341f;
    const float unit = g.scale * kLog2e;

    // Staging: a thread loads chunk `tid % 8` of key `tid / 8`, and dimensions
    // 2b, 2b + 1 of keys 4a..4a + 3.  Those keys are the low (a % 8 < 4) or high
    // half of the chunk of lane block a % 4 at 32-key step a / 8; a wave stores both
    // halves of one chunk.
    const uint32_t k_key = tid / 8, k_chunk = tid % 8;
    const uint32_t v_high = (tid >> 4) & 1, v_pair = (tid & 15) | ((tid >> 5) & 1) << 4;
    const uint32_t v_key = 4 * (wave / 4 * 8 + v_high * 4 + wave % 4);
    v4f kr[2];
    v2f vr[4];
    // Rows past the end repeat the last one: the mask hides their scores, and
    // as values they meet probability zero.
    const uint32_t row_bytes = uint32_t(kv_width) * 4;
    const uint32_t k_row = k_key * row_bytes, v_row = v_key * row_bytes;
    auto load_keys = [&](uint32_t n) {
        const uint32_t k0 = n * kKeys, most = min(k_end - 1 - k0, kKeys - 1) * row_bytes;
        const char *const kt = reinterpret_cast<const char *>(keys + k0 * kv_width);
        const uint32_t at = min(k_row, most) + 32 * k_chunk;
        kr[0] = *reinterpret_cast<const v4f *>(kt + at);
        kr[1] = *reinterpret_cast<const v4f *>(kt + at + 16);
    };
    auto load_values = [&](uint32_t n) {
        const uint32_t k0 = n * kKeys, most = min(k_end - 1 - k0, kKeys - 1) * row_bytes;
        const char *const vt = reinterpret_cast<const char *>(values + k0 * kv_width);
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            const uint32_t at = min(v_row + i * row_bytes, most) + 8 * v_pair;
            vr[i] = *reinterpret_cast<const v2f *>(vt + at);
        }
    };
    bool bad = false;  // a value out of the parts' range was staged
    auto store_keys = [&] {
        float f[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            f[i] = kr[i / 4][i % 4];
        bad |= out_of_range<8>(f);
        Parts p;
        split<8>(f, p.hi, p.mid, p.lo);
        uint8_t *const at = k_lds + key_at(k_key, k_chunk);
        *reinterpret_cast<v4u *>(at) = p.hi;
        *reinterpret_cast<v4u *>(at + kPlane) = p.mid;
        *reinterpret_cast<v4u *>(at + 2 * kPlane) = p.lo;
    };
    auto store_values = [&] {
        const float all[8] = {vr[0][0], vr[0][1], vr[1][0], vr[1][1],
                              vr[2][0], vr[2][1], vr[3][0], vr[3][1]};
        bad |= out_of_range<8>(all);
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            const float x[4] = {vr[0][d], vr[1][d], vr[2][d], vr[3][d]};
            v2u hi, mid, lo;
            split<4>(x, hi, mid, lo);
            uint8_t *const at = v_lds + value_at(2 * v_pair + d, wave) + 8 * v_high;
            *reinterpret_cast<v2u *>(at) = hi;
            *reinterpret_cast<v2u *>(at + kPlane) = mid;
            *reinterpret_cast<v2u *>(at + 2 * kPlane) = lo;
        }
    };
    auto parts_at = [](const uint8_t *plane) {
        return Parts{*reinterpret_cast<const v4u *>(plane),
                     *reinterpret_cast<const v4u *>(plane + kPlane),
                     *reinterpret_cast<const v4u *>(plane + 2 * kPlane)};
    };

    v4f o[4];
    float m, l;  // m in log2 units
    auto clear = [&] {
        m = -__builtin_inff();
        l = 0.0f;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            o[u] = v4f{0, 0, 0, 0};
    };
    clear();
    // The block's key tiles.
    const uint32_t tiles = (k_end + kKeys - 1) / kKeys;
    const uint32_t begin = range * range_tiles;
    const uint32_t end = begin + range_tiles < tiles ? begin + range_tiles : tiles;
    if (begin + team < end) {
        load_keys(begin + team);
        load_values(begin + team);
        store_keys();
    }
    // The teams take the key tiles in turn.  Per tile two barriers: behind the first
    // the tile's keys are complete and the values of the tile before are free, behind
    // the second the tile's values are complete and its keys are free.  The values
    // (the next keys) to store there were requested half a tile earlier.
    for (uint32_t first = begin; first < end; first += TEAMS) {
        const uint32_t n = first + team, next = n + TEAMS;
        const uint32_t k0 = n * kKeys;
        const bool active = n < end && k0 <= wave_last && !q_bad;
        __syncthreads();
        if (n < end)
            store_values();
        if (next < end)
            load_keys(next);
        v4f s[4];
        if (active) {
            // S^T = K Q^T.
#pragma unroll
            for (int c = 0; c < 4; ++c)
                s[c] = v4f{0, 0, 0, 0};
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                const Parts qp = {q_lds[0][st][tid], q_lds[1][st][tid], q_lds[2][st][tid]};
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    s[c] = multiply_add(parts_at(k_lds + key_at(16 * c + j, 4 * st + q)), qp,
                                        s[c]);
            }
        }
        __syncthreads();
        if (next < end) {
            store_keys();
            load_values(next);
        }
        if (active) {
            // Causal mask, online softmax over the row's four lanes.
            if (k0 + kKeys - 1 > wave_first || k0 + kKeys > k_end) {
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (int(k0 + 16 * c + r) > reach)
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
            if (__any(mx > m + kSlack)) {
                // A row without a visible key so far keeps m = -inf, l = 0.
                const float m_new = fmaxf(m, mx);
                const float alpha =
                    m_new == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(m - m_new);
                m = m_new;
                l *= alpha;
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    o[u] *= alpha;
            }
            const float m_ref = m == -__builtin_inff() ? 0.0f : m;
            Parts p[2];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                v2u hi, mid, lo;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    s[c][r] = __builtin_amdgcn_exp2f(fmaf(s[c][r], unit, -m_ref));
                    l += s[c][r];
                }
                split<4>(s[c], hi, mid, lo);
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    p[c / 2].hi[2 * (c % 2) + r] = hi[r];
                    p[c / 2].mid[2 * (c % 2) + r] = mid[r];
                    p[c / 2].lo[2 * (c % 2) + r] = lo[r];
                }
            }
            // O^T += V^T P^T, the tile's sums added whole.
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                v4f sum = {0, 0, 0, 0};
#pragma unroll
                for (int st = 0; st < 2; ++st)
                    sum = multiply_add(parts_at(v_lds + value_at(16 * u + j, 4 * st + q)), p[st],
                                       sum);
                o[u] += sum;
            }
        }
    }
    if (bad)
        any_bad = 1;
    __syncthreads();  // and the tiles are free
    if (any_bad || q_bad) {
        // A key or value of the range, or a query of this wave, that the parts do
        // not serve: the rows over again in f32, straight from memory.
        clear();
#pragma unroll 1
        for (uint32_t k0 = begin * kKeys + 16 * team; k0 < end * kKeys && k0 <= wave_last;
             k0 += 16 * TEAMS) {
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
                s[r] = int(k0 + r) > reach ? -__builtin_inff() : s[r] * unit;
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
    if constexpr (TEAMS == 2) {
        // The second team hands its rows to the first.
        static_assert(kThreads * (4 * 16 + 2 * 4) <= sizeof(lds), "the teams' exchange");
        v4f *const o_lds = reinterpret_cast<v4f *>(lds[0]) + tid;
        float *const ml_lds = reinterpret_cast<float *>(lds[0] + 4 * 16 * kThreads) + tid;
        if (team != 0) {
#pragma unroll
            for (int u = 0; u < 4; ++u)
                o_lds[u * kThreads] = o[u];
            ml_lds[0] = m;
            ml_lds[kThreads] = l;
        }
        __syncthreads();
        if (team != 0)
            return;
        const float m_other = ml_lds[0], m_new = fmaxf(m, m_other);
        const float m_ref = m_new == -__builtin_inff() ? 0.0f : m_new;
        const float w = __builtin_amdgcn_exp2f(m - m_ref);
        const float w_other = __builtin_amdgcn_exp2f(m_other - m_ref);
        m = m_new;
        l = l * w + ml_lds[kThreads] * w_other;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            o[u] = o[u] * w + o_lds[u * kThreads] * w_other;
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
                rec[2 + 16 * u + 4 * q + e] = o[u][e];
        return;
    }
    float *const o_row = out + pair * kDim;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        v4f r;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            r[e] = o[u][e] / l;
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

// Key tiles per block up to which one team, without the exchange, is faster (us, two
// teams and one: 40 tokens of 32 / 8 heads 10.6, 9.2, 128 tokens 12.7, 12.2; at four
// tiles 200 tokens of 16 / 8 16.2, 16.8).
constexpr uint32_t kOneTeam = 2;

// Blocks the CUs hold at once: one each.
constexpr uint32_t kResident = 256;

// A launch that leaves half of the CUs idle cuts its keys into ranges of at least
// four tiles, whose records a second launch merges: 64 tokens over 2000 keys (32 / 8
// heads) 87 -> 26 us, 1024 over 1024 (16 / 4) 89 -> 63, 256 over 512 (32 / 8) 37 ->
// 23.  Fuller launches lose by the records' traffic (700 over 300, 32 / 8, 49
// unsplit, 61 in two ranges; 2048 tokens 119, 173).
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
    const uint32_t blocks = d.token_tiles * d.ranges * g.key_value_heads;
    if (d.range_tiles <= kOneTeam)
        gqa_flash_split_kernel<1><<<blocks, kThreads, 0, stream>>>(
            out, query, key_cache, value_cache, g, d.tile_tokens, d.token_tiles, d.ranges,
            d.range_tiles, records);
    else
        gqa_flash_split_kernel<2><<<blocks, 2 * kThreads, 0, stream>>>(
            out, query, key_cache, value_cache, g, d.tile_tokens, d.token_tiles, d.ranges,
            d.range_tiles, records);
    if (d.ranges > 1) {
        const uint32_t pairs = uint32_t(g.tokens) * g.query_heads;
        gqa_flash_merge_kernel<<<(pairs + 3) / 4, 256, 0, stream>>>(out, records, d.ranges, pairs);
    }
}

}  // namespace mfh
