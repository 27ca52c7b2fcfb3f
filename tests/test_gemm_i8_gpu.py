"""The INT8 prefill GEMM on integer digits (runtime_amd/csrc/gemm_i8.hip) at the
edges of its tiles, K runs and number range, against 64-bit sums.

Bound.  An activation is within half a unit of its digits, a unit being its
128-group's largest magnitude over 8355711, and its scaling rounds by 2 * 2^-24
of itself; digit sums are exact.  Per group the middle digits' sum, the group's
sum and unit * scale round by 2^-24 of |x| |w| summed over the group, at most
three each, and the totals by 2^-24 of all of it per group.  So an output is
within sum_g sum_k (0.51 unit + 2^-22 |x_k| + (groups + 6) 2^-24 |x_k|) |w_k|.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from runtime_amd import convert
from runtime_amd.backend import ExecutorError, HipBackend, Limits
from tests.test_packed_gpu import make_weights, run_linear, say, upload_weights
from tests.test_resources_gpu import MIB, total

pytestmark = pytest.mark.gpu


def check(got, x, codes, scales, floor=0.0):
    groups = scales.shape[1]
    w = codes.view(np.int8).astype(np.float64) * np.repeat(scales.astype(np.float64), 128, axis=1)
    x = x.astype(np.float64)
    want = x @ w.T
    unit = np.abs(x).reshape(x.shape[0], groups, 128).max(axis=2) / 8355711.0
    off = 0.51 * np.repeat(unit, 128, axis=1) + np.abs(x) * (2.0 ** -22 + (groups + 6) * 2.0 ** -24)
    bound = off @ np.abs(w).T + floor
    diff = np.abs(got.astype(np.float64) - want)
    assert np.all(diff <= bound), f"max over bound {np.max(diff / np.maximum(bound, 1e-300)):.3g}"


# Row tiles around 16 and 32 rows, column tiles around 64, 128 and 256, one group,
# K runs of odd length (9 and 11 groups), and launches of 1 x 1 and 2 x 2 wave tiles
# (1 x 2: test_wave_tiles).
SHAPES = [(9, 16, 128), (15, 63, 256), (16, 65, 384), (17, 129, 640), (31, 257, 1280),
          (33, 1000, 3456), (20, 70, 2816), (48, 512, 8192), (200, 1100, 4096), (130, 4608, 1024),
          (400, 4100, 256), (1025, 3300, 128), (2048, 2049, 384)]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_edges(backend, m, n, k):
    say("i8 gemm", m, n, k)
    codes, scales = make_weights(n, k, "int8", 0x5EED0800 + n + k)
    x = convert.normal((m, k), 0xAC70800 + m)
    check(run_linear(backend, x, codes, scales), x, codes, scales)


# (rows, columns, width, streams): 1 x 2 wave tiles (enough blocks, long K), 2 x 2
# ones in K runs (weights of more than 2^24 values), a pair's.
TILES = [(330, 2500, 256, 1), (300, 1300, 4096, 1), (100, 4100, 4224, 1), (300, 2600, 256, 2),
         (120, 2050, 4224, 2)]


@pytest.mark.parametrize("m,n,k,streams", TILES)
def test_wave_tiles(backend, m, n, k, streams):
    say("i8 wave tiles", m, n, k, streams)
    weights = [make_weights(n, k, "int8", 0x5EED08A0 + n + k + i) for i in range(streams)]
    x = convert.normal((m, k), 0xAC70800 + m)
    if streams == 1:
        check(run_linear(backend, x, *weights[0]), x, *weights[0])
        return
    bufs = [upload_weights(backend, *w) for w in weights]
    xb = backend.upload_f32(x.shape, x)
    outs = [backend.allocate_f32((m, n)) for _ in range(3)]
    backend.packed_linear_pair(*outs[:2], xb, *bufs[0], *bufs[1])
    backend.packed_swiglu_pair(outs[2], xb, *bufs[0], *bufs[1])
    a, b, fused = (backend.read(out) for out in outs)
    check(a, x, *weights[0])
    check(b, x, *weights[1])
    np.testing.assert_allclose(fused, oracle.swiglu(a, b), rtol=2e-6, atol=1e-30)


@pytest.mark.parametrize("m,n,k", [(9, 40, 384), (70, 300, 1024), (300, 2600, 256)])
def test_pairs(backend, m, n, k):
    say("i8 pair", m, n, k)
    ca, sa = make_weights(n, k, "int8", 0x5EED0810 + n)
    cb, sb = make_weights(n, k, "int8", 0x5EED0811 + n)
    x = convert.normal((m, k), 0xAC70810 + m)
    ga, gsa = upload_weights(backend, ca, sa)
    gb, gsb = upload_weights(backend, cb, sb)
    xb = backend.upload_f32(x.shape, x)
    out_a, out_b, fused = (backend.allocate_f32((m, n)) for _ in range(3))
    backend.packed_linear_pair(out_a, out_b, xb, ga, gsa, gb, gsb)
    backend.packed_swiglu_pair(fused, xb, ga, gsa, gb, gsb)
    a, b = backend.read(out_a), backend.read(out_b)
    check(a, x, ca, sa)
    check(b, x, cb, sb)
    np.testing.assert_allclose(backend.read(fused), oracle.swiglu(a, b), rtol=2e-6, atol=1e-30)


@pytest.mark.parametrize("case", ["zeros", "tiny", "large", "spikes", "ramp", "extreme"])
def test_number_range(backend, case):
    say("i8 range", case)
    m, n, k = 40, 200, 512
    codes, scales = make_weights(n, k, "int8", 0x5EED0820)
    x = convert.normal((m, k), 0xAC70820)
    if case == "zeros":
        x[:, 100:300] = 0.0
        x[7] = 0.0
    elif case == "tiny":
        x *= np.float32(2.0 ** -90)
    elif case == "large":
        x *= np.float32(2.0 ** 90)
    elif case == "spikes":
        x[:, ::61] *= np.float32(4096.0)
    elif case == "ramp":
        x *= np.exp2(np.linspace(-40, 40, k)).astype(np.float32)
    else:  # every digit and code at its largest: the integer sums' range
        codes = np.where(np.arange(k) % 256 < 128, 127, -127).astype(np.int8)
        codes = np.tile(codes, (n, 1)).view(np.uint8)
        x = np.full((m, k), 3.0, np.float32)
        x[1::2] *= -1
        x[2] = np.where(np.arange(k) % 2, 1.0, -1.0)
    got = run_linear(backend, x, codes, scales)
    check(got, x, codes, scales)
    if case == "zeros":
        assert not got[7].any()


# Launches of 1 x 1, 1 x 2 (32 groups or more), 2 x 2 wave tiles, of K runs, and
# a pair's; the last column of the block is ragged in each.
SMALL_SHAPES = [(40, 200, 512), (300, 1300, 4096), (1030, 3300, 256), (20, 70, 2816)]


@pytest.mark.parametrize("m,n,k", SMALL_SHAPES)
@pytest.mark.parametrize("power", [-41, -104, -116, -120])
def test_small_values(backend, power, m, n, k):
    """Activations whose digit units, or units times scales, are below f32's
    normal range: every row, then single rows and groups between ordinary ones.
    A group's sum may itself be subnormal and round at 2^-149."""
    say("i8 small", power, m, n, k)
    floor = k // 128 * 2.0 ** -149
    codes, scales = make_weights(n, k, "int8", 0x5EED0860)
    x = convert.normal((m, k), 0xAC70860)
    small = x * np.float32(2.0 ** power)
    check(run_linear(backend, small, codes, scales), small, codes, scales, floor)
    mixed = x.copy()
    mixed[3::7] = small[3::7]
    mixed[5, 128:256] = small[5, 128:256]
    mixed[m - 1, :128] = small[m - 1, :128]
    check(run_linear(backend, mixed, codes, scales), mixed, codes, scales, floor)


def test_small_values_in_pairs(backend):
    say("i8 small pair")
    m, n, k = 70, 300, 1024
    (ca, sa), (cb, sb) = (make_weights(n, k, "int8", 0x5EED0870 + i) for i in range(2))
    x = convert.normal((m, k), 0xAC70870) * np.float32(2.0 ** -112)
    x[::3] *= np.float32(2.0 ** 112)
    a, b = upload_weights(backend, ca, sa), upload_weights(backend, cb, sb)
    xb = backend.upload_f32(x.shape, x)
    out_a, out_b = (backend.allocate_f32((m, n)) for _ in range(2))
    backend.packed_linear_pair(out_a, out_b, xb, *a, *b)
    check(backend.read(out_a), x, ca, sa, k // 128 * 2.0 ** -149)
    check(backend.read(out_b), x, cb, sb, k // 128 * 2.0 ** -149)


@pytest.mark.parametrize("x_power,scale_power", [(0, -116), (-60, -55), (60, -118), (-30, 80),
                                                 (-100, 60)])
def test_f32_scales_far_from_one(backend, x_power, scale_power):
    say("i8 f32 scale range", x_power, scale_power)
    m, n, k = 35, 200, 640
    rng = np.random.default_rng(0x5EED0880)
    codes = rng.integers(-127, 128, (n, k), dtype=np.int8).view(np.uint8)
    scales = rng.uniform(0.01, 0.03, (n, k // 128)).astype(np.float32)
    scales[1::2] *= np.float32(2.0 ** scale_power)
    x = convert.normal((m, k), 0xAC70880) * np.float32(2.0 ** x_power)
    check(run_linear(backend, x, codes, scales), x, codes, scales, k // 128 * 2.0 ** -149)


def test_f32_scales(backend):
    say("i8 f32 scales")
    m, n, k = 35, 100, 640
    rng = np.random.default_rng(0x5EED0830)
    codes = rng.integers(-127, 128, (n, k), dtype=np.int8).view(np.uint8)
    scales = rng.uniform(0.01, 0.03, (n, k // 128)).astype(np.float32)  # not binary16 values
    x = convert.normal((m, k), 0xAC70830)
    check(run_linear(backend, x, codes, scales), x, codes, scales)


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_non_finite_rows(backend, value):
    say("i8 non-finite", value)
    m, n, k = 50, 130, 768
    codes, scales = make_weights(n, k, "int8", 0x5EED0840)
    x = convert.normal((m, k), 0xAC70840)
    hit = [(0, 0), (17, 127), (18, 128 + 79), (49, k - 1)]
    for row, column in hit:
        x[row, column] = value
    got = run_linear(backend, x, codes, scales)
    bad = np.zeros(m, dtype=bool)
    bad[[row for row, _ in hit]] = True
    assert np.isnan(got[bad]).all()
    check(got[~bad], x[~bad], codes, scales)


@pytest.mark.parametrize("room,runs", [(3 * MIB + 16384, True), (MIB // 2, False)])
def test_scratch_limit(room, runs):
    """The digit records round nine rows up to sixteen, so 3 MiB of room holds the
    binary16-halves plan's scratch but not theirs: the product still runs.  Less
    room than that refuses, before anything is written."""
    say("i8 scratch limit", room)
    m, n, k = 9, 16, 65536
    codes, scales = make_weights(n, k, "int8", 0x5EED0850)
    x = convert.normal((m, k), 0xAC70850)
    sentinel = np.full((m, n), 5.0, np.float32)
    limit = 48 * MIB
    be = HipBackend(0, limits=Limits(max_total_bytes=limit))
    try:
        cb, sb = upload_weights(be, codes, scales)
        xb = be.upload_f32(x.shape, x)
        out = be.upload_f32(sentinel.shape, sentinel)
        be.prepare_packed(cb, sb)
        fill = []
        while True:
            want = limit - total(be.resource_report()) - room
            if want < 1024:
                break
            size = 1 << (want.bit_length() - 1) if want > MIB else want // 256 * 256
            fill.append(be.allocate_f32_classified((size // 4,), 1))
        if runs:
            be.packed_linear(out, xb, cb, sb)
            check(be.read(out), x, codes, scales)
        else:
            with pytest.raises(ExecutorError) as e:
                be.packed_linear(out, xb, cb, sb)
            assert e.value.variant == "ResourceLimit"
            assert np.array_equal(be.read(out), sentinel)
    finally:
        be.close()
