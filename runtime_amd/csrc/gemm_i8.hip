// Matrix-core prefill GEMM for packed INT8 weights (m > 8) on the integer MFMA.
//
// out[m, n] = sum_g scale[n, g] * sum_{k in g} x[m, k] * code[n, k], the
// reference's group-then-scale order (kernels-simd/src/lib.rs:54,205).
//
// Exactness plan.
// - i8_split_kernel writes each 128-group of a row as whole multiples, up to
//   8355711 (0x7f7f7f), of one unit (the group's largest magnitude over that),
//   in three signed 8-bit digits: every value is within half a unit.
// - v_mfma_i32_16x16x64_i8 multiplies digits and codes exactly.  The highest
//   digit's sums, shifted by eight bits, start the middle digit's (below 2^30);
//   the group's sum is that times 256 plus the lowest digit's, in f32, and one
//   FMA adds it times unit * scale.
// - A group with a non-finite value gets a NaN unit, so the row's outputs are NaN.
// - A unit times a scale stays normal for group maxima from 2^-40 on (and f32
//   scales of 2^-60 to 2^22).  Elsewhere the range plan of digits.hpp applies: the
//   unit is rounded up to 14 bits, its code is those and its exponent, and the
//   second pass multiplies mantissas and adds exponents.
//
// Bound and split.  Integer MFMAs run at twice the binary16 rate, so three
// digits cost 1.5 binary16 passes where hi + lo halves cost two, and the codes
// are the operand as they are stored: no decode.  The price is the epilogue, 24
// vector instructions per six MFMAs.
//
// Operands, tiling and grid mapping are those of the ternary kernel
// (gemm_mx.hip): the weights straight from the decode GEMV's repacked tiles, the
// digits through LDS in records of (128-group, 16 rows), blocks of four waves
// along n, 16 TI rows x 16 TJ columns each.
#include <algorithm>
#include <type_traits>

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "digits.hpp"
#include "kernels.hpp"

namespace mfh {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kDigits = 3;
constexpr float kLargest = 8355711.0f;  // 0x7f7f7f
constexpr int kSmall = -40;             // a group below 2^kSmall stores a unit code
constexpr uint32_t kCodeMask = 0x3ff;   // mantissa bits a coded unit leaves out
constexpr int kCodeBias = 200;          // of its exponent, -172..-63
// One digit's operands of 16 rows x 128 k: two 64-wide ksteps of 16 bytes per
// lane.
constexpr uint32_t kDigitBytes = 2 * 64 * 16;
constexpr uint32_t kUnitsAt = kDigits * kDigitBytes;  // 16 f32: the rows' units
constexpr uint32_t kRecord = kUnitsAt + 64;
// Records a block may read past the last row tile of the last group.
constexpr uint32_t kMaxRowTiles = 2;

// One wave per (group, 16-row tile).  Lane 16q + i holds row i, k = 16q + 0..15 of
// both ksteps, the lane's bytes of a repacked INT8 tile.
__global__ __launch_bounds__(kThreads) void i8_split_kernel(const float *__restrict__ x,
                                                            uint32_t m, uint32_t k,
                                                            uint32_t row_tiles, uint32_t records,
                                                            uint8_t *__restrict__ dst)
{
    const uint32_t record = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
    if (record >= records)
        return;
    const uint32_t lane = threadIdx.x & 63, i = lane & 15, q = lane >> 4;
    const uint32_t group = record / row_tiles, row = record % row_tiles * 16 + i;
    float v[32];
    // Rows past m are zeros (their outputs are never stored).
    const float *src = x + size_t(row < m ? row : 0) * k + group * 128 + 16 * q;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const float4 f = *reinterpret_cast<const float4 *>(src + (u / 4) * 64 + 4 * (u % 4));
        v[4 * u] = f.x;
        v[4 * u + 1] = f.y;
        v[4 * u + 2] = f.z;
        v[4 * u + 3] = f.w;
    }
    // A non-finite value makes the group's maximum +inf.
    float mx = 0.0f;
#pragma unroll
    for (int t = 0; t < 32; ++t) {
        if (row >= m)
            v[t] = 0.0f;
        mx = fmaxf(mx, isfinite(v[t]) ? fabsf(v[t]) : __builtin_inff());
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const bool bad = !isfinite(mx);
    int e = 0;
    if (mx > 0.0f && !bad)
        mx = frexpf(mx, &e);
    float units = mx > 0.0f && !bad ? kLargest / mx : 0.0f;  // per 2^e
    const bool small = units > 0.0f && e <= kSmall;
    uint32_t code = 0;
    if (__builtin_expect(__any(small), 0)) {
        // 1 / units, in [2^-24, 2^-22], rounded up to 14 bits.
        const uint32_t up = (__float_as_uint(1.0f / units) + kCodeMask) & ~kCodeMask;
        const int exponent = int(up >> 23) - 127 + e + kCodeBias;  // 28..137
        if (small) {
            units = 1.0f / __uint_as_float(up);
            code = uint32_t(exponent) << 13 | ((up & 0x7fffffu) >> 10);
        }
    }
    uint8_t *out = dst + size_t(record) * kRecord + 16 * lane;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        v4u digit[kDigits];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            unsigned d2 = 0, d1 = 0, d0 = 0;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const float y = bad ? 0.0f : ldexpf(v[16 * half + 4 * w + t], -e) * units;
                int whole = int(rintf(fminf(fmaxf(y, -kLargest), kLargest)));
                const int low = int8_t(whole);
                whole = (whole - low) >> 8;
                const int mid = int8_t(whole);
                const int high = (whole - mid) >> 8;
                d0 |= unsigned(low & 255) << (8 * t);
                d1 |= unsigned(mid & 255) << (8 * t);
                d2 |= unsigned(high & 255) << (8 * t);
            }
            digit[0][w] = d2;
            digit[1][w] = d1;
            digit[2][w] = d0;
        }
#pragma unroll
        for (int d = 0; d < kDigits; ++d)
            *reinterpret_cast<v4u *>(out + d * kDigitBytes + 1024 * half) = digit[d];
    }
    if (q == 0)
        *reinterpret_cast<float *>(dst + size_t(record) * kRecord + kUnitsAt + 4 * i) =
            bad || code ? nan_of(code) : units > 0.0f ? ldexpf(1.0f / units, e) : 0.0f;
}

struct I8Args {
    const uint8_t *x;          // digit records [group][row tile]
    const uint8_t *wtiles[2];  // repacked codes per stream
    const void *scales[2];     // tiled scales per stream: [tile][groups_pad][16]
    float *out[2];
    float *partial;            // split-K: [chunk][stream][m][n] raw sums
    uint32_t m, n;
    uint32_t row_tiles;        // 16-row record tiles
    uint32_t n_tiles;          // 16-row tiles of each repacked stream
    uint32_t tile_vecs;        // 16-byte lane loads per tile (of 64 lanes)
    uint32_t groups_pad;       // tiled scale groups per tile
    uint32_t tiles_n, tiles;   // output block tiles along n, and in all
    uint32_t chunks, chunk_groups;
};

template <int S, Epilogue E, bool HALF, int TI, int TJ>
__global__ __launch_bounds__(kThreads, 3) void gemm_i8_kernel(I8Args g)
{
    constexpr int TJS = TJ / S;                       // column tiles per stream per wave
    constexpr uint32_t BNS = 4 * 16 * TJS;            // block columns per stream
    constexpr uint32_t UNITS = TI * kRecord / 16;     // 16-byte units of a stage
    __shared__ __align__(1024) uint8_t stage[2][TI * kRecord];

    const uint32_t blocks = g.tiles * g.chunks;
    uint32_t block = blockIdx.x;
    if (blocks % 8 == 0)
        block = (blockIdx.x % 8) * (blocks / 8) + blockIdx.x / 8;
    const uint32_t chunk = block / g.tiles, tile = block % g.tiles;
    const uint32_t mt0 = (tile / g.tiles_n) * TI, n0 = (tile % g.tiles_n) * BNS;
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t li = lane & 15, lq = lane >> 4;
    const uint32_t g_begin = chunk * g.chunk_groups, g_end = g_begin + g.chunk_groups;

    const uint32_t lds0 = uint32_t(reinterpret_cast<uintptr_t>(
        (__attribute__((address_space(3))) uint8_t *)&stage[0][0]));
    const uint8_t *x_src = g.x + size_t(mt0) * kRecord;
    const size_t x_step = size_t(g.row_tiles) * kRecord;
    auto fetch = [&](uint32_t grp, uint32_t buf) {
        const uint8_t *src = x_src + grp * x_step;
#pragma unroll
        for (uint32_t r = 0; r * kThreads < UNITS; ++r)
            if ((r + 1) * kThreads <= UNITS || r * kThreads + tid < UNITS)
                copy_to_lds(src + r * kThreads * 16, 16 * tid,
                            lds0 + buf * (TI * kRecord) + (r * kThreads + wave * 64) * 16);
    };

    // Wave-uniform tile addresses.
    const char *wptr[TJ], *sptr[TJ];
#pragma unroll
    for (int jt = 0; jt < TJ; ++jt) {
        const int st = jt / TJS;
        const uint32_t t = n0 / 16 + wave * TJS + jt % TJS;
        // Tiles past n read tile 0 (their columns are never stored).
        const size_t live = t < g.n_tiles ? t : 0;
        wptr[jt] = reinterpret_cast<const char *>(g.wtiles[st]) + live * g.tile_vecs * 16;
        sptr[jt] = static_cast<const char *>(g.scales[st]) +
                   live * g.groups_pad * 16 * (HALF ? 2 : 4);
    }
    // A uniform address plus a 32-bit lane offset, both opaque: otherwise the
    // offsets are widened outside the loop and every load adds 64 bits per lane.
    typedef const __attribute__((address_space(1))) char *Global;
    auto at = [](const char *base, size_t offset, uint32_t lane_offset) {
        Global p = Global(base + offset);
        asm volatile("" : "+s"(p), "+v"(lane_offset));
        return p + lane_offset;
    };
    typedef typename std::conditional<HALF, unsigned short, float>::type Scale;
    // Weight operands and scales, one register set per group parity.
    v4i wts[2][TJ][2];
    Scale scale[2][TJ];
    auto load_weights = [&](uint32_t grp, v4i (&dst)[TJ][2]) {
#pragma unroll
        for (int jt = 0; jt < TJ; ++jt)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                dst[jt][h] = *reinterpret_cast<const __attribute__((address_space(1))) v4i *>(
                    at(wptr[jt], size_t(grp) * 2048 + 1024 * h, lane * 16));
    };
    auto load_scales = [&](uint32_t grp, Scale (&dst)[TJ]) {
#pragma unroll
        for (int jt = 0; jt < TJ; ++jt)
            dst[jt] = *reinterpret_cast<const __attribute__((address_space(1))) Scale *>(
                at(sptr[jt], size_t(grp) * 16 * sizeof(Scale), li * sizeof(Scale)));
    };

    v4f total[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int jt = 0; jt < TJ; ++jt)
            total[i][jt] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

    struct Frag {
        v4i digit[kDigits][2];
        v4f unit;
    };
    auto read_frag = [&](uint32_t buf, int i, Frag &f) {
        const uint8_t *rec = &stage[buf][i * kRecord];
        f.unit = *reinterpret_cast<const v4f *>(rec + kUnitsAt + 16 * lq);
#pragma unroll
        for (int d = 0; d < kDigits; ++d)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                f.digit[d][h] = *reinterpret_cast<const v4i *>(rec + d * kDigitBytes + 1024 * h +
                                                               16 * lane);
    };

    fetch(g_begin, 0);
    load_weights(g_begin, wts[0]);
    load_scales(g_begin, scale[0]);
    uint32_t odd_scale = 0;  // f32 scales: set by one outside the first pass's range
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    __syncthreads();

    // One group; its parity within the run picks the LDS buffer and the register
    // sets, so the main loop takes two groups per iteration and moves nothing.
    auto step = [&](uint32_t grp, auto parity) {
        constexpr int odd = decltype(parity)::value;
        // The next group's loads, in flight behind this one's products (the last
        // group loads its own again).
        const uint32_t next = grp + 1 < g_end ? grp + 1 : grp;
        if (grp + 1 < g_end)
            fetch(grp + 1, odd ^ 1);
        load_weights(next, wts[odd ^ 1]);
        load_scales(next, scale[odd ^ 1]);
        float gsc[TJ];
#pragma unroll
        for (int jt = 0; jt < TJ; ++jt) {
            if constexpr (HALF) {
                gsc[jt] = __half2float(__ushort_as_half(scale[odd][jt]));
            } else {
                gsc[jt] = scale[odd][jt];
                odd_scale |= gsc[jt] != 0.0f && !(fabsf(gsc[jt]) >= 0x1p-60f &&
                                                  fabsf(gsc[jt]) <= 0x1p22f);
            }
        }
        Frag f[2];
        read_frag(odd, 0, f[0]);
        // Row tile i's products run while tile i + 1's operands are read.
#pragma unroll
        for (int i = 0; i < TI; ++i) {
            __builtin_amdgcn_sched_barrier(0);
            if (i + 1 < TI)
                read_frag(odd, i + 1, f[(i + 1) & 1]);
            const Frag &a = f[i & 1];
            v4i high[TJ], low[TJ];
            auto product = [&](int d, int h, int jt, const v4i &c) {
                return __builtin_amdgcn_mfma_i32_16x16x64_i8(a.digit[d][h], wts[odd][jt][h], c, 0, 0,
                                                             0);
            };
#pragma unroll
            for (int jt = 0; jt < TJ; ++jt)
                high[jt] = product(0, 1, jt, product(0, 0, jt, v4i{0, 0, 0, 0}));
#pragma unroll
            for (int jt = 0; jt < TJ; ++jt)
                low[jt] = product(2, 1, jt, product(2, 0, jt, v4i{0, 0, 0, 0}));
#pragma unroll
            for (int jt = 0; jt < TJ; ++jt)
                high[jt] = product(1, 1, jt, product(1, 0, jt, high[jt] << 8));
#pragma unroll
            for (int jt = 0; jt < TJ; ++jt)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    total[i][jt][r] = fmaf(fmaf(float(high[jt][r]), 256.0f, float(low[jt][r])),
                                           a.unit[r] * gsc[jt], total[i][jt][r]);
        }
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the next stage is in LDS
        __syncthreads();
    };
    uint32_t grp = g_begin;
    for (; grp + 1 < g_end; grp += 2) {
        step(grp, std::integral_constant<int, 0>{});
        step(grp + 1, std::integral_constant<int, 1>{});
    }
    if (grp < g_end)
        step(grp, std::integral_constant<int, 0>{});

    // NaN totals (of rows that exist: the records past the last are no rows).
    float nan = 0.0f;
#pragma unroll
    for (int i = 0; i < TI; ++i)
        if (mt0 + i < g.row_tiles) {
#pragma unroll
            for (int jt = 0; jt < TJ; ++jt)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    nan += total[i][jt][r];
        }
    if (__builtin_expect(__any(nan != nan || odd_scale), 0)) {
        // A tile at a time, straight from memory.
#pragma unroll 1
        for (uint32_t tile = 0; tile < uint32_t(TI * TJ); ++tile) {
            if (mt0 + tile / TJ >= g.row_tiles)
                break;
            const uint32_t st = tile % TJ / TJS, t = n0 / 16 + wave * TJS + tile % TJS;
            const size_t live = t < g.n_tiles ? t : 0;
            const char *const w_tile =
                reinterpret_cast<const char *>(g.wtiles[st]) + live * g.tile_vecs * 16;
            const char *const s_tile = static_cast<const char *>(g.scales[st]) +
                                       live * g.groups_pad * 16 * (HALF ? 2 : 4);
            v4f sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
            for (uint32_t gr = g_begin; gr < g_end; ++gr) {
                const uint8_t *rec = x_src + gr * x_step + tile / TJ * kRecord;
                const char *w = w_tile + size_t(gr) * 2048 + 16 * lane;
                const char *sp = s_tile + (size_t(gr) * 16 + li) * sizeof(Scale);
                float gs;
                if constexpr (HALF)
                    gs = __half2float(*reinterpret_cast<const __half *>(sp));
                else
                    gs = *reinterpret_cast<const float *>(sp);
                int gs_exp = 0;
                const float gs_frac = frexpf(gs, &gs_exp);
                v4i digit[kDigits];
#pragma unroll
                for (int d = 0; d < kDigits; ++d) {
                    digit[d] = v4i{0, 0, 0, 0};
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        digit[d] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                            *reinterpret_cast<const v4i *>(rec + d * kDigitBytes + 1024 * h +
                                                           16 * lane),
                            *reinterpret_cast<const v4i *>(w + 1024 * h), digit[d], 0, 0, 0);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float whole = fmaf(float((digit[0][r] << 8) + digit[1][r]), 256.0f,
                                             float(digit[2][r]));
                    const uint32_t unit =
                        reinterpret_cast<const uint32_t *>(rec + kUnitsAt)[4 * lq + r];
                    int exp = 0;
                    float frac = frexpf(__uint_as_float(unit), &exp);
                    if (is_code(unit)) {
                        exp = int((unit >> 13) & 511) - kCodeBias;
                        frac = __uint_as_float(0x3f800000u | (unit & 0x1fffu) << 10);
                    }
                    sum[r] += ldexpf(whole * (frac * gs_frac), exp + gs_exp);
                }
            }
#pragma unroll
            for (int i = 0; i < TI; ++i)
#pragma unroll
                for (int jt = 0; jt < TJ; ++jt)
                    if (tile == uint32_t(i * TJ + jt))
                        total[i][jt] = sum;
        }
    }

#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t mm = (mt0 + i) * 16 + lq * 4 + r;
            if (mm >= g.m)
                continue;
#pragma unroll
            for (int tt = 0; tt < TJS; ++tt) {
                const uint32_t nn = n0 + (wave * TJS + tt) * 16 + li;
                if (nn >= g.n)
                    continue;
                const size_t o = size_t(mm) * g.n + nn;
                if (g.chunks > 1) {
                    const size_t plane = size_t(g.m) * g.n;
#pragma unroll
                    for (int st = 0; st < S; ++st)
                        g.partial[(size_t(chunk) * S + st) * plane + o] =
                            total[i][st * TJS + tt][r];
                    continue;
                }
                if constexpr (E == Epilogue::SwigluPair) {
                    g.out[0][o] = silu_mul(total[i][tt][r], total[i][(S - 1) * TJS + tt][r]);
                } else {
                    g.out[0][o] = total[i][tt][r];
                    if constexpr (E == Epilogue::Pair)
                        g.out[1][o] = total[i][(S - 1) * TJS + tt][r];
                }
            }
        }
}

struct Plan {
    uint32_t ti, tj;  // 16-row and 16-column tiles per wave
    uint32_t tiles_n, tiles, chunks;
};

// The largest wave tile that still gives the launch enough blocks (400; a pair
// that asked for 1000 took smaller tiles: M = 100 x 8192 x 2048 43 us against 29.5,
// M = 300 x 4608 x 1024 30.4 against 23.8), and for a launch of one-tile waves still
// short of blocks K runs of at least four groups.  us per call, before (two binary16
// passes) -> now: M = 2048 x 2048 x 8192 184 -> 160, 1024 x 2048 x 2048 36.6 ->
// 26.6, 128 x 2048 x 1024 15.0 -> 10.3, 16 x 8192 x 2048 16.5 -> 11.8; gate/up pairs
// with SwiGLU M = 346 x 2560 x 1024 24.4 -> 19.1, 100 x 8192 x 2048 33.6 -> 29.5.
// Four column tiles per wave (two waves per SIMD instead of four) took 344 against
// 324 us on the pair M = 2048 x 8192 x 2048.  Error against 64-bit sums 5.3e-7 ->
// 2.7e-7 (2048 x 8192 x 2048).
//
// Weights of 2^24 values and more are read once per 16 TI rows from beyond the L2s:
// there 100 blocks are enough (M = 128 x 8192 x 8192 82 us with small tiles, 53 with
// large ones, 57 on the halves; 64 x 8192 x 4096 30, 23, 25; pairs 128 x 4096 x 4096
// 46, 32, 34; the other way only 48 x 16384 x 2048 21, 23, 24).
Plan plan_of(const PackedCall &call)
{
    const uint32_t s = call.epilogue == Epilogue::Single ? 1 : 2;
    const uint32_t groups = call.k / 128, row_tiles = (call.m + 15) / 16;
    auto with = [&](uint32_t ti, uint32_t tj) {
        Plan p{ti, tj, 0, 0, 1};
        p.tiles_n = (call.n + 64 * tj / s - 1) / (64 * tj / s);
        p.tiles = p.tiles_n * ((row_tiles + ti - 1) / ti);
        return p;
    };
    const uint32_t enough = uint64_t(call.n) * call.k * s >= 1u << 24 ? 100 : 400;
    Plan p = with(2, 2);
    if (p.tiles < enough)
        p = with(1, 2);
    if (s == 1 && p.tiles < enough) {
        const Plan one = with(1, 1);
        if (groups < 32 || p.tiles < 200)
            p = one;
    }
    for (uint32_t c = 2; c <= groups / 4; ++c)
        if (groups % c == 0 && groups - groups / c >= 8 && p.tiles * c <= 512)
            p.chunks = c;
    return p;
}

template <int S, Epilogue E, bool HALF>
void launch_plan(hipStream_t stream, const I8Args &args, const Plan &p)
{
    const unsigned grid = p.tiles * p.chunks;
#define I8_CASE(TI, TJ)                                                                          \
    if (p.ti == TI && p.tj == TJ)                                                                \
        return gemm_i8_kernel<S, E, HALF, TI, TJ><<<grid, kThreads, 0, stream>>>(args);
    I8_CASE(2, 2)
    I8_CASE(1, 2)
    if constexpr (S == 1)
        I8_CASE(1, 1)
#undef I8_CASE
}

template <bool HALF>
void launch_half(hipStream_t stream, const PackedCall &call, const I8Args &args, const Plan &p)
{
    switch (call.epilogue) {
    case Epilogue::Single: return launch_plan<1, Epilogue::Single, HALF>(stream, args, p);
    case Epilogue::Pair: return launch_plan<2, Epilogue::Pair, HALF>(stream, args, p);
    case Epilogue::SwigluPair: return launch_plan<2, Epilogue::SwigluPair, HALF>(stream, args, p);
    }
}

size_t records_bytes(const PackedCall &call)
{
    return (size_t((call.m + 15) / 16) * (call.k / 128) + kMaxRowTiles - 1) * kRecord;
}

}  // namespace

// The binary16-halves kernel keeps the launches that fill the device with its
// 64-row tiles over wide outputs, where both take the same time within 5 % (us,
// halves and here: M = 1024 x 8192 x 2048 86.8, 89.9; 2048 x 8192 x 2048 171, 173;
// 2048 x 4096 x 8192 334, 337; 512 x 8192 x 2048 50.0, 48.0; at its edge 1024 x 4096
// x 2048 48.0, 43.6).  Outside, here is faster: 2048 x 2048 x 2048 51.7, 44.7 (as many
// blocks, fewer columns), 2048 x 2048 x 8192 184, 160, 512 x 4096 x 8192 98, 89, 256
// x 6144 x 2048 31.9, 25.8, 128 x 4096 x 2048 24.8, 17.5; K = 8192 at 48-96 rows is the
// closest (96 x 4096 x 8192 32.7, 34.3).
bool gemm_i8_served(const PackedCall &call)
{
    const uint32_t columns = call.epilogue == Epilogue::Single ? 128 : 64;
    const uint64_t blocks =
        uint64_t((call.m + 31) / 32) * ((uint64_t(call.n) + columns - 1) / columns);
    return call.format == Format::Int8 && !call.single_half && !call.halves &&
           (call.n < 4096 || blocks < 1024);
}

size_t gemm_i8_scratch_bytes(const PackedCall &call)
{
    const Plan p = plan_of(call);
    const int s = call.epilogue == Epilogue::Single ? 1 : 2;
    return records_bytes(call) +
           (p.chunks > 1 ? size_t(p.chunks) * s * call.m * call.n * sizeof(float) : 0);
}

void launch_gemm_i8(hipStream_t stream, const PackedCall &call, void *scratch)
{
    const Plan p = plan_of(call);
    const uint32_t groups = call.k / 128, row_tiles = (call.m + 15) / 16;
    uint8_t *records = static_cast<uint8_t *>(scratch);
    const uint32_t count = groups * row_tiles;
    i8_split_kernel<<<(count + kThreads / 64 - 1) / (kThreads / 64), kThreads, 0, stream>>>(
        call.x, call.m, call.k, row_tiles, count, records);
    I8Args args{};
    args.x = records;
    args.wtiles[0] = call.a.tiles;
    args.wtiles[1] = call.b.tiles;
    args.scales[0] = call.a.tiled_scales;
    args.scales[1] = call.b.tiled_scales;
    args.out[0] = call.out_a;
    args.out[1] = call.out_b;
    args.partial = reinterpret_cast<float *>(records + records_bytes(call));
    args.m = call.m;
    args.n = call.n;
    args.row_tiles = row_tiles;
    args.n_tiles = (call.n + 63) / 64 * 4;
    args.tile_vecs = call.k / 64 * 64;
    args.groups_pad = groups;
    args.tiles_n = p.tiles_n;
    args.tiles = p.tiles;
    args.chunks = p.chunks;
    args.chunk_groups = groups / p.chunks;
    const bool half =
        call.a.tiled_half && (call.epilogue == Epilogue::Single || call.b.tiled_half);
    if (half)
        launch_half<true>(stream, call, args, p);
    else
        launch_half<false>(stream, call, args, p);
    if (p.chunks > 1)
        launch_splitk_reduce(stream, call.epilogue, call.out_a, call.out_b, args.partial,
                             size_t(call.m) * call.n, p.chunks);
}

}  // namespace mfh
