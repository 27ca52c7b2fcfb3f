// Matrix-core prefill GEMM for packed ternary weights (m > 8) on the
// block-scaled FP6 x FP4 MFMA.
//
// out[m, n] = sum_g scale[n, g] * sum_{k in g} x[m, k] * (code[n, k] - 1),
// the reference's group-then-scale order (kernels-simd/src/lib.rs:54,205).
//
// Exactness plan.
// - mx_split_kernel cuts every run of 32 activations of a row (the k of one
//   MFMA lane) into five FP6 (E2M3) digits under one power of two: with every
//   |x| of the run below 2^e, x = 2^(e-2) * sum_d 2^(-5d) * q_d, each q_d the
//   nearest FP6 value of what the digits before it left.  What five digits
//   leave is at most 2^-25 of 2^e.
// - The weight code itself is the FP4 (E2M1) operand: the bit patterns 0..3
//   are 0, 0.5, 1 and 1.5, so code / 2 needs no conversion, only the 2-bit
//   fields spread to nibbles.  The factor 2 sits in the weight operand's
//   block scale, and the levels' -1 enters as the accumulator's start value,
//   minus the row's sum over the group.
// - v_mfma_scale_f32_16x16x128_f8f6f4 multiplies exactly, applies both block
//   scales and accumulates in f32; a 128-group is five of them, the largest
//   digit first, which cancels the start value at once.  The epilogue adds
//   group_sum * scale in f32 (one FMA).
// - A row with a non-finite value gets NaN start values, so all of its
//   outputs are NaN, as with a NaN or infinity in every dot.
// - These are sums of true magnitudes (small ones keep their precision: the
//   accumulators hold subnormals).  A group of a row with a run past 2^100 is
//   written times 2^-64 and takes the range plan of digits.hpp: its start value is
//   a code, and the second pass multiplies by signed levels, which need none.
//
// Bound and split.  FP6 x FP4 runs at four times the binary16 rate (measured
// 8.2 against 2.27 PFLOP/s with eight waves per CU), so five passes cost 1.25
// binary16 passes where hi + lo halves cost two, and the weights need no
// decode to halves.  us per call, halves -> digits: M = 2048 x 8192 x 2048 160 ->
// 107, 2048 x 2048 x 8192 174 -> 117, 512 x 8192 x 2048 50 -> 31, 128 x 4608 x 1024
// 19.9 -> 10.4.  The matrix pipe is busy 46 % of the first; vector work hardly
// overlaps these MFMAs (four FMAs beside one take its slot from 20 to 32 cycles),
// so the inner loop keeps to 68 vector instructions per 40 MFMAs (118 before it
// took two groups per iteration: 111 us).  Loading two groups ahead over three
// LDS buffers needs a second register set and leaves two waves per SIMD: 117 us.
//
// Operands.  The weights are read from the decode GEMV's repacked tiles (16
// rows x K per tile, one 16-byte load per lane covering 256 k) straight into
// registers.  The activation digits are staged through LDS, double buffered:
// mx_split_kernel writes one kRecord-byte record per (128-group, 16 rows)
// holding the MFMA operand of every digit in lane order, the row sums and
// the block exponents, and a block's records of a group are one contiguous
// run that global_load_lds copies without passing through registers.
//
// Tiling.  A block is four waves along n; a wave owns 16 TI rows x 16 TJ
// columns (TJ / S of each of S weight streams).  At least three waves share a
// SIMD, so one wave's loads and epilogue run beside another's MFMAs.
//
// Grid mapping.  Workgroups are dealt round-robin to the 8 XCDs; block b
// computes tile (b % 8) * (tiles / 8) + b / 8, so each XCD's L2 holds a
// contiguous run of tiles: neighbouring n-tiles of the same m rows.
#include <algorithm>
#include <type_traits>

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "digits.hpp"
#include "kernels.hpp"

namespace mfh {
namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef unsigned v6u __attribute__((ext_vector_type(6)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v32f __attribute__((ext_vector_type(32)));

constexpr int kThreads = 256;
constexpr int kDigits = 5;
constexpr int kDigitBits = 5;  // each digit's scale against the one before
// One digit's operand of 16 rows x 128 k: 24 bytes per lane, the first 16 of
// every lane, then the last 8 (both reads conflict-free).
constexpr uint32_t kDigitBytes = 64 * 24;
constexpr uint32_t kSumsAt = kDigits * kDigitBytes;  // 16 f32: -(row sum)
constexpr uint32_t kExpsAt = kSumsAt + 64;           // 64 bytes: block scales
constexpr uint32_t kRecord = kExpsAt + 64;
// A row's group with a run past 2^kLargeRun is written times 2^-kShift.
constexpr int kLargeRun = 100, kShift = 64;
constexpr uint32_t kShifted = 1;  // its start value's code
// Records a block may read past the last row tile of the last group.
constexpr uint32_t kMaxRowTiles = 2;

// One wave per (group, 16-row tile).  Lane 16q + i holds row i, k = 16q + 0..15
// and 64 + 16q + 0..15 of the group: the 32 k of lane block q of a repacked
// ternary tile.  Bound by memory at size (2048 x 8192 values, 131 MB read and
// written: 22-27 us, 4.9-6 TB/s), by its own latency at 128 x 1024 (4.6 us).
__global__ __launch_bounds__(kThreads) void mx_split_kernel(const float *__restrict__ x,
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
    float mx = 0.0f;
    bool bad = false;
#pragma unroll
    for (int t = 0; t < 32; ++t) {
        if (row >= m)
            v[t] = 0.0f;
        mx = fmaxf(mx, fabsf(v[t]));
        bad |= !isfinite(v[t]);
    }
    int e = 0;
    if (mx > 0.0f && !bad)
        frexpf(mx, &e);  // |x| < 2^e
    int shift = 0;
    const unsigned long long large = __ballot(e > kLargeRun);
    if (__builtin_expect(large != 0, 0))
        shift = (large >> i) & 0x0001000100010001ull ? kShift : 0;
    e = max(e, shift - 124);
    // Operand slots 2t and 2t + 1 take even[t] and odd[t].  Slot order of the
    // weight nibbles: k = 0, 2, .., 14, 1, 3, .., 15 of each run of 16.
    v16f even, odd;
    double sum = 0.0;
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        const int at = 16 * (t / 8) + 4 * (t % 4) + (t / 4) % 2;
        even[t] = bad ? 0.0f : ldexpf(v[at], 2 - e);  // |.| < 4
        odd[t] = bad ? 0.0f : ldexpf(v[at + 2], 2 - e);
        sum += double(even[t]);
        sum += double(odd[t]);
    }
    uint8_t *out = dst + size_t(record) * kRecord;
#pragma unroll
    for (int d = 0; d < kDigits; ++d) {
        const float scale = 1.0f / float(1u << (kDigitBits * d));
        const v6u digit = __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(even, odd, scale);
        *reinterpret_cast<v4u *>(out + d * kDigitBytes + 16 * lane) =
            v4u{digit[0], digit[1], digit[2], digit[3]};
        *reinterpret_cast<v2u *>(out + d * kDigitBytes + 1024 + 8 * lane) = v2u{digit[4], digit[5]};
        const v32f taken = __builtin_amdgcn_cvt_scalef32_pk32_f32_fp6(digit, scale);
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            even[t] -= taken[2 * t];
            odd[t] -= taken[2 * t + 1];
        }
    }
    // The digits' sum is what the products see: leave the remainder out.
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        sum -= double(even[t]);
        sum -= double(odd[t]);
    }
    sum = ldexp(sum, e - 2);
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    const unsigned long long any_bad = __ballot(bad);
    const bool row_bad = (any_bad >> i) & 0x0001000100010001ull;
    out[kExpsAt + lane] = uint8_t(127 + e - 2 - shift);
    if (q == 0)
        reinterpret_cast<float *>(out + kSumsAt)[i] =
            row_bad ? nan_of(0) : shift ? nan_of(kShifted) : float(-sum);
}

struct MxArgs {
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
__global__ __launch_bounds__(kThreads, 3) void gemm_mx_kernel(MxArgs g)
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
    v4u raw[TJ];
    auto load_weights = [&](uint32_t grp) {
#pragma unroll
        for (int jt = 0; jt < TJ; ++jt)
            raw[jt] = *reinterpret_cast<const __attribute__((address_space(1))) v4u *>(
                at(wptr[jt], size_t(grp / 2) * 1024, lane * 16));
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
        v4u lo[kDigits];
        v2u hi[kDigits];
        v4f start;
        int exps;
    };
    // The 8-byte parts keep an address register per digit: with one base the
    // compiler pairs two digits' reads and moves the halves apart again.
    uint32_t hi_at[kDigits];
    auto read_frag = [&](uint32_t buf, int i, Frag &f) {
        const uint8_t *rec = &stage[buf][i * kRecord];
        f.start = *reinterpret_cast<const v4f *>(rec + kSumsAt + 16 * lq);
        f.exps = rec[kExpsAt + lane];
#pragma unroll
        for (int d = 0; d < kDigits; ++d) {
            f.lo[d] = *reinterpret_cast<const v4u *>(rec + d * kDigitBytes + 16 * lane);
            f.hi[d] = *reinterpret_cast<const __attribute__((address_space(3))) v2u *>(
                hi_at[d] + i * kRecord);
        }
    };

    fetch(g_begin, g_begin & 1);
    load_weights(g_begin);
    Scale scale[2][TJ];
    load_scales(g_begin, scale[0]);
    load_scales(g_begin, scale[1]);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    __syncthreads();

    // One group; its parity picks the half of the weight load, the LDS buffer
    // and the scale registers, so the main loop takes two groups per iteration
    // and moves nothing between registers.
    auto step = [&](uint32_t grp, auto parity) {
        constexpr int odd = decltype(parity)::value;
        // The group's weight operands, then the next group's loads, in flight
        // behind this one's products (the last group loads its own again).
        v8i b[TJ];
#pragma unroll
        for (int jt = 0; jt < TJ; ++jt) {
            b[jt] = v8i{};
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const unsigned w = raw[jt][2 * odd + t] ^ 0x80808080u;  // canonical codes
                b[jt][2 * t] = int(w & 0x33333333u);                    // fields 0, 2
                b[jt][2 * t + 1] = int((w >> 2) & 0x33333333u);         // fields 1, 3
            }
        }
        const uint32_t next = grp + 1 < g_end ? grp + 1 : grp;
        if (grp + 1 < g_end)
            fetch(grp + 1, odd ^ 1);
        load_scales(next, scale[odd ^ 1]);
        if (odd)
            load_weights(next);
        float gsc[TJ];
#pragma unroll
        for (int jt = 0; jt < TJ; ++jt) {
            if constexpr (HALF)
                gsc[jt] = __half2float(__ushort_as_half(scale[odd][jt]));
            else
                gsc[jt] = scale[odd][jt];
        }
#pragma unroll
        for (int d = 0; d < kDigits; ++d) {
            hi_at[d] = lds0 + odd * (TI * kRecord) + d * kDigitBytes + 1024 + 8 * lane;
            asm volatile("" : "+v"(hi_at[d]));
        }
        Frag f[2];
        v4f acc[2][TJ];
        auto add_group = [&](int i) {
#pragma unroll
            for (int jt = 0; jt < TJ; ++jt)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    total[i][jt][r] = fmaf(acc[i & 1][jt][r], gsc[jt], total[i][jt][r]);
        };
        read_frag(odd, 0, f[0]);
        // Row tile i's products run while tile i + 1's operands are read and
        // tile i - 1's group sums are added.
#pragma unroll
        for (int i = 0; i < TI; ++i) {
            __builtin_amdgcn_sched_barrier(0);
            if (i + 1 < TI)
                read_frag(odd, i + 1, f[(i + 1) & 1]);
            const Frag &a = f[i & 1];
#pragma unroll
            for (int d = 0; d < kDigits; ++d) {
                const v8i ad = {int(a.lo[d][0]), int(a.lo[d][1]), int(a.lo[d][2]), int(a.lo[d][3]),
                                int(a.hi[d][0]), int(a.hi[d][1]), 0, 0};
#pragma unroll
                for (int jt = 0; jt < TJ; ++jt)
                    acc[i & 1][jt] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                        ad, b[jt], d == 0 ? a.start : acc[i & 1][jt], 2, 4, 0, a.exps, 0,
                        128 - kDigitBits * d);
            }
            if (i > 0)
                add_group(i - 1);
            // Operand reads two at a time between the products.
            if (i + 1 < TI) {
#pragma unroll
                for (int u = 0; u < 6; ++u) {
                    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, 3, 0);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        add_group(TI - 1);
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the next stage is in LDS
        __syncthreads();
    };
    uint32_t grp = g_begin;
    if (grp & 1)
        step(grp++, std::integral_constant<int, 1>{});
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
    if (__builtin_expect(__any(nan != nan), 0)) {
        // A tile at a time, straight from memory, on signed levels.
        const uint32_t at = cold_lane(), ci = at & 15, cq = at >> 4;
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
                const v2u codes = *reinterpret_cast<const v2u *>(
                    w_tile + size_t(gr / 2) * 1024 + 16 * at + 8 * (gr & 1));
                v8i level = {};
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const unsigned w = ((codes[t / 2] ^ 0x80808080u) >> (2 * (t & 1))) &
                                       0x33333333u;
                    // Nibbles 0..3 to the FP4 values -0.5, 0, 0.5 and 1.
                    const unsigned zero = ~(w | w >> 1) & 0x11111111u;
                    level[t] = int((w - (zero ^ 0x11111111u)) | zero * 9);
                }
                v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
                for (int d = kDigits - 1; d >= 0; --d) {
                    const v4u lo =
                        *reinterpret_cast<const v4u *>(rec + d * kDigitBytes + 16 * at);
                    const v2u hi = *reinterpret_cast<const v2u *>(rec + d * kDigitBytes +
                                                                  1024 + 8 * at);
                    const v8i ad = {int(lo[0]), int(lo[1]), int(lo[2]), int(lo[3]),
                                    int(hi[0]), int(hi[1]), 0, 0};
                    acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                        ad, level, acc, 2, 4, 0, int(rec[kExpsAt + at]), 0,
                        128 - kDigitBits * d);
                }
                const char *sp = s_tile + (size_t(gr) * 16 + ci) * sizeof(Scale);
                float gs;
                if constexpr (HALF)
                    gs = __half2float(*reinterpret_cast<const __half *>(sp));
                else
                    gs = *reinterpret_cast<const float *>(sp);
                int gs_exp = 0;
                const float gs_frac = frexpf(gs, &gs_exp);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t start =
                        reinterpret_cast<const uint32_t *>(rec + kSumsAt)[4 * cq + r];
                    if (start == kNanBits)
                        sum[r] = nan_of(0);
                    const int back = start == (kNanBits | kShifted) ? kShift : 0;
                    sum[r] += ldexpf(acc[r] * gs_frac, gs_exp + back);
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

// The largest wave tile that still gives the launch enough blocks: larger
// tiles read each operand for more products, more blocks hide each other's
// loads.  Enough is 400 blocks for a single product and 1000 for a pair
// (us per call, larger / smaller tile: M = 2048 x 8192 x 2048 109-114 (2 x 4)
// / 127 (2 x 2), 2048 x 2048 x 8192 120-127 / 131; M = 256 x 8192 x 2048 24.4 (256
// blocks) / 22.0 (512); M = 346 x 2560 x 1024 13.1 (220) / 11.3 (440); M = 128 x
// 4608 x 1024 pair 13.5 (576) / 12.0 (1152)).  Four row tiles per wave (two waves
// per SIMD instead of three), tried before the loop took two groups per iteration,
// measured 109 against 103 us on the first shape and 136 against 110 on the second.
//
// A launch of one-tile waves that is still short of blocks splits K into runs
// of at least four groups, up to 512 blocks, where that saves eight groups
// of each block's chain, which pays for the second launch that adds the runs
// (M = 64 x 2048 x 2048 12.7 -> 12.0, M = 128 x 1024 x 4608 21 -> 14.2; M =
// 128 x 1024 x 1024 unsplit 9.7 against 10.5).  At 32 groups or more two runs
// over one-by-two tiles beat one over one-by-one tiles (M = 256 x 2048 x 8192
// 33 -> 27.4).
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
    const uint32_t enough = s == 1 ? 400 : 1000;
    Plan p = with(2, 4);
    if (p.tiles < enough)
        p = with(2, 2);
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
void launch_plan(hipStream_t stream, const MxArgs &args, const Plan &p)
{
    const unsigned grid = p.tiles * p.chunks;
#define MX_CASE(TI, TJ)                                                                          \
    if (p.ti == TI && p.tj == TJ)                                                                \
        return gemm_mx_kernel<S, E, HALF, TI, TJ><<<grid, kThreads, 0, stream>>>(args);
    MX_CASE(2, 4)
    MX_CASE(2, 2)
    MX_CASE(1, 2)
    if constexpr (S == 1)
        MX_CASE(1, 1)
#undef MX_CASE
}

template <bool HALF>
void launch_half(hipStream_t stream, const PackedCall &call, const MxArgs &args, const Plan &p)
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

bool gemm_mx_served(const PackedCall &call)
{
    return call.format == Format::Ternary && !call.single_half;
}

size_t gemm_mx_scratch_bytes(const PackedCall &call)
{
    const Plan p = plan_of(call);
    const int s = call.epilogue == Epilogue::Single ? 1 : 2;
    return records_bytes(call) +
           (p.chunks > 1 ? size_t(p.chunks) * s * call.m * call.n * sizeof(float) : 0);
}

void launch_gemm_mx(hipStream_t stream, const PackedCall &call, void *scratch)
{
    const Plan p = plan_of(call);
    const uint32_t groups = call.k / 128, row_tiles = (call.m + 15) / 16;
    uint8_t *records = static_cast<uint8_t *>(scratch);
    const uint32_t count = groups * row_tiles;
    mx_split_kernel<<<(count + kThreads / 64 - 1) / (kThreads / 64), kThreads, 0, stream>>>(
        call.x, call.m, call.k, row_tiles, count, records);
    const uint32_t k_pad = (call.k + 255) / 256 * 256;
    MxArgs args{};
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
    args.tile_vecs = k_pad / 256 * 64;
    args.groups_pad = k_pad / 128;
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
