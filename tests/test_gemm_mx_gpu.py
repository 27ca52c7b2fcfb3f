"""The ternary prefill GEMM on block-scaled digits (runtime_amd/csrc/gemm_mx.hip)
at the edges of its tiles, K runs and number range, against 64-bit sums.

Bound.  With A = sum_k |x_k| * scale * (|level_k| + 1) of one output: five FP6
digits leave at most 2^-25 of a run's power of two, below 2^-24 of the run's
largest |x|; a 128-group is one rounded start value and five accumulations of
exact products, each rounded (or, inside one MFMA, aligned) at 2^-23 of a
magnitude of at most A's share of the group; the totals add one rounding of
2^-24 * A per group.  Together below (8 + groups / 2) * 2^-23 * A.
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


def reference(x, codes, scales):
    """(64-bit products, the bound's A) of each output."""
    n, groups = scales.shape
    level = np.stack([(codes >> s) & 3 for s in (0, 2, 4, 6)], axis=2).reshape(n, -1) - 1.0
    scale = np.repeat(scales.astype(np.float64), 128, axis=1)
    x = x.astype(np.float64)
    return x @ (level * scale).T, np.abs(x) @ ((np.abs(level) + 1.0) * np.abs(scale)).T


def check(got, x, codes, scales, floor=0.0):
    want, size = reference(x, codes, scales)
    bound = (8 + scales.shape[1] / 2) * 2.0 ** -23 * size + floor
    diff = np.abs(got.astype(np.float64) - want)
    assert np.all(diff <= bound), f"max over bound {np.max(diff / np.maximum(bound, 1e-300)):.3g}"


# One to two row tiles around 16 and 32 rows, column tiles around 64, 128 and
# 256, one group, K runs that start inside a 256-wide tile load (3456 and 2816
# split into runs of 9 and 11 groups), and launches of 1 x 1, 2 x 2 and 2 x 4 wave
# tiles (1 x 2: test_wave_tiles).
SHAPES = [(9, 16, 128), (15, 63, 256), (16, 65, 384), (17, 129, 640), (31, 257, 1280),
          (33, 1000, 3456), (20, 70, 2816), (48, 512, 8192), (200, 1100, 4096), (130, 4608, 1024),
          (400, 4100, 256), (1025, 3300, 128), (2048, 2049, 384)]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_edges(backend, m, n, k):
    say("mx gemm", m, n, k)
    codes, scales = make_weights(n, k, "ternary", 0x5EED0700 + n + k)
    x = convert.normal((m, k), 0xAC70700 + m)
    check(run_linear(backend, x, codes, scales), x, codes, scales)


# (rows, columns, width, streams): 1 x 2 wave tiles (enough blocks, long K) and a
# pair's 2 x 2 and 2 x 4 ones.
TILES = [(330, 2500, 256, 1), (300, 1300, 4096, 1), (1030, 2050, 256, 2), (1030, 4100, 384, 2)]


@pytest.mark.parametrize("m,n,k,streams", TILES)
def test_wave_tiles(backend, m, n, k, streams):
    say("mx wave tiles", m, n, k, streams)
    weights = [make_weights(n, k, "ternary", 0x5EED07A0 + n + k + i) for i in range(streams)]
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
    say("mx pair", m, n, k)
    ca, sa = make_weights(n, k, "ternary", 0x5EED0710 + n)
    cb, sb = make_weights(n, k, "ternary", 0x5EED0711 + n)
    x = convert.normal((m, k), 0xAC70710 + m)
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


@pytest.mark.parametrize("case", ["zeros", "tiny", "large", "spikes", "ramp"])
def test_number_range(backend, case):
    say("mx range", case)
    m, n, k = 40, 200, 512
    codes, scales = make_weights(n, k, "ternary", 0x5EED0720)
    x = convert.normal((m, k), 0xAC70720)
    if case == "zeros":
        x[:, 100:300] = 0.0
        x[7] = 0.0
    elif case == "tiny":
        x *= np.float32(2.0 ** -100)
    elif case == "large":
        x *= np.float32(2.0 ** 100)
    elif case == "spikes":
        x[:, ::61] *= np.float32(4096.0)
    else:
        x *= np.exp2(np.linspace(-40, 40, k)).astype(np.float32)
    got = run_linear(backend, x, codes, scales)
    check(got, x, codes, scales)
    if case == "zeros":
        assert not got[7].any()


# Launches of 1 x 1, 1 x 2 (32 groups or more), 2 x 2 and 2 x 4 wave tiles, and of
# K runs, the odd one starting inside a 256-wide tile load; the last column of
# the block is ragged in each.
RANGE_SHAPES = [(40, 200, 512), (300, 1300, 4096), (1030, 1700, 256), (1025, 3300, 384),
                (20, 70, 2816)]


@pytest.mark.parametrize("m,n,k", RANGE_SHAPES)
@pytest.mark.parametrize("power", [-61, -100, -116, -120, 99, 121, 124])
def test_values_at_the_ends_of_the_range(backend, power, m, n, k):
    """All rows, then single rows and groups between ordinary ones.  The large
    ones meet sparse levels and small scales: group sums (of |x| and of 2 |x|)
    that overflow f32 where the products of every output stay finite."""
    say("mx range ends", power, m, n, k)
    codes, scales = make_weights(n, k, "ternary", 0x5EED0760)
    floor = k // 128 * 2.0 ** -149  # a group's sum may itself be subnormal
    if power > 0:
        rng = np.random.default_rng(0x5EED0761)
        level = np.where(rng.random((n, k)) < 0.05, rng.integers(0, 3, (n, k)), 1)
        codes = np.zeros((n, k // 4), np.uint8)
        for i in range(4):
            codes |= (level[:, i::4] << (2 * i)).astype(np.uint8)
    x = convert.normal((m, k), 0xAC70760)
    if power > 0:
        x = np.abs(x)
    far = x * np.float32(2.0 ** power)
    assert np.isfinite(far).all()
    check(run_linear(backend, far, codes, scales), far, codes, scales, floor)
    mixed = x.copy()
    mixed[3::7] = far[3::7]
    mixed[5, 128:256] = far[5, 128:256]
    mixed[m - 1, :128] = far[m - 1, :128]
    mixed[6, 100:140] = far[6, 100:140]
    check(run_linear(backend, mixed, codes, scales), mixed, codes, scales, floor)


@pytest.mark.parametrize("power", [-112, 124])
def test_ends_of_the_range_in_pairs(backend, power):
    say("mx range pair", power)
    m, n, k = 70, 300, 1024
    (ca, sa), (cb, sb) = (make_weights(n, k, "ternary", 0x5EED0770 + i) for i in range(2))
    x = convert.normal((m, k), 0xAC70770)
    x[::3] *= np.float32(2.0 ** power)
    a, b = upload_weights(backend, ca, sa), upload_weights(backend, cb, sb)
    xb = backend.upload_f32(x.shape, x)
    out_a, out_b = (backend.allocate_f32((m, n)) for _ in range(2))
    backend.packed_linear_pair(out_a, out_b, xb, *a, *b)
    check(backend.read(out_a), x, ca, sa, k // 128 * 2.0 ** -149)
    check(backend.read(out_b), x, cb, sb, k // 128 * 2.0 ** -149)


def test_reserved_code_and_f32_scales(backend):
    say("mx reserved code")
    m, n, k = 35, 100, 640
    rng = np.random.default_rng(0x5EED0730)
    codes = rng.integers(0, 256, (n, k // 4), dtype=np.uint8)  # code 3 is level +2
    scales = rng.uniform(0.01, 0.03, (n, k // 128)).astype(np.float32)  # not binary16 values
    x = convert.normal((m, k), 0xAC70730)
    check(run_linear(backend, x, codes, scales), x, codes, scales)
    x[::2] *= np.float32(2.0 ** -110)
    check(run_linear(backend, x, codes, scales), x, codes, scales)


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_non_finite_rows(backend, value):
    say("mx non-finite", value)
    m, n, k = 50, 130, 768
    codes, scales = make_weights(n, k, "ternary", 0x5EED0740)
    x = convert.normal((m, k), 0xAC70740)
    hit = [(0, 0), (17, 127), (18, 128 + 79), (49, k - 1)]
    for row, column in hit:
        x[row, column] = value
    got = run_linear(backend, x, codes, scales)
    bad = np.zeros(m, dtype=bool)
    bad[[row for row, _ in hit]] = True
    assert np.isnan(got[bad]).all()
    check(got[~bad], x[~bad], codes, scales)


@pytest.mark.parametrize("room,runs", [(MIB + 16384, True), (MIB // 2, False)])
def test_scratch_limit(room, runs):
    """The digit records round nine rows up to sixteen, so 1 MiB of room holds
    the binary16-halves plan's scratch but not theirs: the product still runs.
    Less room than that refuses, before anything is written."""
    say("mx scratch limit", room)
    m, n, k = 9, 64, 16384
    codes, scales = make_weights(n, k, "ternary", 0x5EED0750)
    x = convert.normal((m, k), 0xAC70750)
    sentinel = np.full((m, n), 5.0, np.float32)
    limit = 32 * MIB
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
        left = limit - total(be.resource_report())
        assert room <= left < room + 1024
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


@pytest.mark.parametrize("m,n,room,runs", [(9, 64, MIB + 16384, True), (17, 16, 1400000, True),
                                           (33, 16, 2700000, True), (33, 16, 2200000, False)])
def test_scratch_limit_in_pieces(m, n, room, runs):
    """A budget that holds the binary16-halves plan's scratch but not the digit
    records of all rows: pieces of the rows run where their records fit (17 rows as
    16 + 1, 33 as 32 + 1), and what does not (9 rows) takes no memory; less than
    the halves plan's need refuses."""
    say("mx scratch pieces", m, room)
    k = 16384
    codes, scales = make_weights(n, k, "ternary", 0x5EED0780)
    x = convert.normal((m, k), 0xAC70780)
    limit = 64 * MIB
    be = HipBackend(0, limits=Limits(max_total_bytes=limit))
    try:
        cb, sb = upload_weights(be, codes, scales)
        xb = be.upload_f32(x.shape, x)
        out, out_b = be.allocate_f32((m, n)), be.allocate_f32((m, n))
        be.prepare_packed(cb, sb)
        fill = []
        while (want := limit - total(be.resource_report()) - room) >= 1024:
            size = 1 << (want.bit_length() - 1) if want > MIB else want // 256 * 256
            fill.append(be.allocate_f32_classified((size // 4,), 1))
        left = limit - total(be.resource_report())
        assert room <= left < room + 1024
        if not runs:
            with pytest.raises(ExecutorError) as e:
                be.packed_linear(out, xb, cb, sb)
            assert e.value.variant == "ResourceLimit"
            return
        be.packed_linear(out, xb, cb, sb)
        taken = left - (limit - total(be.resource_report()))
        assert taken == 0 if m == 9 else 0 < taken <= room
        check(be.read(out), x, codes, scales)
        if m == 17:  # the pair's halves fit the same block
            be.packed_linear_pair(out, out_b, xb, cb, sb, cb, sb)
            assert np.array_equal(be.read(out), be.read(out_b))
            check(be.read(out), x, codes, scales)
    finally:
        be.close()
