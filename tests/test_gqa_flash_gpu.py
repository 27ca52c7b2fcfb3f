"""The 64-wide prefill attention on split bfloat16 operands
(runtime_amd/csrc/gqa_flash.hip) at the edges of its tiles and key ranges, over
the number range, and with infinities and NaN, against 64-bit softmax.

Bound.  With s = sum_d |q_d k_d| / 8 of a (row, key) pair: the parts drop at most
2 * 2^-24 of each product and twelve f32 accumulations round by 2^-24 of at most s
each, so a score is off by at most d = 2^-20 s.  Probabilities then move by a
factor within 2 d (both in the exponent and in the sum), plus 2^-20 for exponent,
parts and sums.
"""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from runtime_amd import hiptime
from runtime_amd.backend import CacheLength, GqaSpec, HipBackend, Limits
from tests.test_dense_gpu import rng_f32, run_gqa, say, up
from tests.test_resources_gpu import MIB, total

pytestmark = pytest.mark.gpu
D = 64


def reference(q, k, v, start, qh, kvh):
    """(64-bit outputs, bound) per (token, head, dimension)."""
    tokens, total = q.shape[0], k.shape[0]
    q = q.astype(np.float64).reshape(tokens, qh, D)
    k = k.astype(np.float64).reshape(total, kvh, D)
    v = v.astype(np.float64).reshape(total, kvh, D)
    want, bound = np.empty_like(q), np.empty_like(q)
    hidden = np.arange(total)[None, :] > start + np.arange(tokens)[:, None]
    for h in range(qh):
        qq, kk, vv = q[:, h], k[:, h // (qh // kvh)], v[:, h // (qh // kvh)]
        score = np.where(hidden, -np.inf, qq @ kk.T / 8.0)
        p = np.exp(score - score.max(axis=1, keepdims=True))
        p /= p.sum(axis=1, keepdims=True)
        off = 2.0 ** -20 * (np.abs(qq) @ np.abs(kk).T) / 8.0
        off = np.where(hidden, 0.0, off).max(axis=1, keepdims=True)
        want[:, h] = p @ vv
        bound[:, h] = (2 * off + 2.0 ** -20) * (p @ np.abs(vv))
    return want.reshape(tokens, -1), bound.reshape(tokens, -1)


def operands(seed, tokens, start, qh, kvh):
    cap = start + tokens
    return (rng_f32(seed, (tokens, qh * D)), rng_f32(seed + 1, (tokens, kvh * D)),
            rng_f32(seed + 2, (tokens, kvh * D)), rng_f32(seed + 3, (cap, kvh * D)),
            rng_f32(seed + 4, (cap, kvh * D)))


def check(backend, q, k, v, kc, vc, start, qh, kvh):
    out, _, _, _ = run_gqa(backend, q, k, v, kc, vc, start, qh, kvh, D)
    want, bound = reference(q, np.concatenate([kc[:start], k]), np.concatenate([vc[:start], v]),
                            start, qh, kvh)
    diff = np.abs(out.astype(np.float64) - want)
    assert np.all(diff <= bound), f"max over bound {np.max(diff / bound):.3g}"


# (tokens, start, query heads, kv heads): 128-row blocks of 128, 64, 42 (group
# of three), 32 and 1 tokens with ragged last ones, 64-key tiles ending one key
# before, at and one past an edge, and key ranges (short launches over long
# caches), the last with a single key and with rows that see none of it.
CASES = [(129, 0, 8, 8), (513, 0, 2, 1), (350, 5, 6, 2), (63, 0, 32, 8), (64, 0, 32, 8),
         (65, 0, 32, 8), (33, 0, 128, 1), (32, 992, 32, 8), (40, 985, 32, 8), (64, 2000, 32, 8),
         (300, 1000, 32, 16), (90, 2047, 16, 4), (1024, 0, 4, 1)]


@pytest.mark.parametrize("tokens,start,qh,kvh", CASES)
def test_edges(backend, tokens, start, qh, kvh):
    say("flash", tokens, start, qh, kvh)
    check(backend, *operands(9000 + tokens + start, tokens, start, qh, kvh), start, qh, kvh)


@pytest.mark.parametrize("case", ["sharp", "tiny", "huge", "channels", "growing", "zero"])
def test_number_range(backend, case):
    say("flash range", case)
    tokens, start, qh, kvh = 160, 100, 16, 4
    q, k, v, kc, vc = operands(9100, tokens, start, qh, kvh)
    if case == "sharp":  # one key takes nearly all of a row
        q *= np.float32(40)
    elif case == "tiny":
        for a in (q, k, kc, v, vc):
            a *= np.float32(2.0 ** -60)
    elif case == "huge":
        for a in (k, kc, v, vc):
            a *= np.float32(2.0 ** 60)
        q *= np.float32(2.0 ** -58)
    elif case == "channels":  # dimensions of very different size
        gain = np.exp2(np.linspace(-12, 12, D)).astype(np.float32)
        for a in (v, vc):
            a *= np.tile(gain, kvh)
    elif case == "growing":  # the value scale grows from tile to tile
        steps = np.exp2(np.arange(start + tokens) // 16).astype(np.float32)
        vc[:start] *= steps[:start, None]
        v *= steps[start:, None]
    else:
        for a in (q, k, kc, v, vc):
            a[:] = 0
    check(backend, q, k, v, kc, vc, start, qh, kvh)


@pytest.mark.parametrize("start", [0, 100, 2000])
@pytest.mark.parametrize("case", ["component", "elements", "later row", "large then small",
                                  "2^-120", "2^100", "2^-105 among ones"])
def test_values_of_very_different_size(backend, case, start):
    """Every output keeps its own relative error, whatever stands beside its
    operands in a tile."""
    say("flash spread", case, start)
    tokens, qh, kvh = 160, 16, 4
    q, k, v, kc, vc = operands(9150 + start, tokens, start, qh, kvh)
    rng = np.random.default_rng(9160 + start)
    if case == "component":  # dimensions far below the largest
        gain = np.exp2(-np.arange(D) / 2).astype(np.float32)
        for a in (v, vc):
            a *= np.tile(gain, kvh)
    elif case == "elements":
        for a in (v, vc):
            a *= np.exp2(rng.uniform(-40, 40, a.shape)).astype(np.float32)
        for a in (k, kc):
            a *= np.exp2(rng.uniform(-40, 2, a.shape)).astype(np.float32)
    elif case == "later row":  # a key that the rows before it must not see
        v[70] *= np.float32(2.0 ** 45)
        k[70] *= np.float32(2.0 ** 45)
        q[70:] = 0  # (scores past 2^45 differ by more than any softmax resolves)
    elif case == "large then small":
        for a in (vc, v):
            a[:max(start, 64) // 2] *= np.float32(2.0 ** 40)
        q *= np.float32(4)
    elif case == "2^-120":
        v *= np.float32(2.0 ** -120)
        vc *= np.float32(2.0 ** -120)
    elif case == "2^100":
        v *= np.float32(2.0 ** 100)
        vc *= np.float32(2.0 ** 100)
        k *= np.float32(2.0 ** 70)
        kc *= np.float32(2.0 ** 70)
        q *= np.float32(2.0 ** -70)
    else:
        v[::3] *= np.float32(2.0 ** -105)
        k[::5] *= np.float32(2.0 ** -105)
    check(backend, q, k, v, kc, vc, start, qh, kvh)


def test_minus_infinity_score_drops_its_key(backend):
    """Keys at -inf under positive queries score -inf: probability zero."""
    say("flash -inf key")
    tokens, qh, kvh = 150, 16, 8
    q, k, v, kc, vc = operands(9200, tokens, 0, qh, kvh)
    q = np.abs(q) + np.float32(0.01)
    k[70] = -np.inf
    out, _, _, _ = run_gqa(backend, q, k, v, kc, vc, 0, qh, kvh, D)
    keep = np.arange(tokens) != 70
    for row in (69, 70, 71, 149):
        seen = keep[:row + 1]
        want, bound = reference(q[row:row + 1], k[:row + 1][seen], v[:row + 1][seen],
                                int(seen.sum()) - 1, qh, kvh)
        assert np.all(np.abs(out[row] - want[0]) <= bound[0])


@pytest.mark.parametrize("what", ["key", "value", "query", "query-inf"])
def test_non_finite_operands(backend, what):
    say("flash non-finite", what)
    tokens, qh, kvh = 200, 16, 8
    q, k, v, kc, vc = operands(9300, tokens, 0, qh, kvh)
    clean, _, _, _ = run_gqa(backend, q, k, v, kc, vc, 0, qh, kvh, D)
    if what == "key":
        k[130, 5] = np.nan
    elif what == "value":
        v[130, 5] = np.inf
    elif what == "query":
        q[130, 5] = np.nan
    else:
        q[130, 5] = np.inf
    out, _, _, _ = run_gqa(backend, q, k, v, kc, vc, 0, qh, kvh, D)
    out, clean = out.reshape(tokens, qh, D), clean.reshape(tokens, qh, D)
    if what == "key":  # both query heads of key/value head 0, every row that sees it
        assert np.isnan(out[130:, :2]).all()
        np.testing.assert_allclose(out[:128], clean[:128], rtol=1e-4, atol=1e-5)
        np.testing.assert_allclose(out[:, 2:], clean[:, 2:], rtol=1e-4, atol=1e-5)
    elif what == "value":
        assert np.isposinf(out[130:, :2, 5]).all()
        others = [d for d in range(D) if d != 5]
        np.testing.assert_allclose(out[:, :2][:, :, others], clean[:, :2][:, :, others], rtol=1e-4,
                                   atol=1e-5)
        np.testing.assert_allclose(out[:, 2:], clean[:, 2:], rtol=1e-4, atol=1e-5)
    else:
        assert not np.isfinite(out[130, 0]).any()
        out[130, 0] = clean[130, 0]
        np.testing.assert_allclose(out, clean, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("group", [4, 128])
@pytest.mark.parametrize("prefix", [0, 64, 100])
def test_no_tokens(backend, prefix, group):
    """A call without tokens returns, and leaves caches and length alone."""
    say("flash no tokens", prefix, group)
    q, k, v, kc, vc = (a[:rows] for a, rows in zip(operands(9400, 128, 0, group, 1),
                                                   (0, 0, 0, 128, 128)))
    out, keys, values, length = run_gqa(backend, q, k, v, kc, vc, prefix, group, 1, D)
    assert out.shape == (0, group * D) and length == prefix
    assert np.array_equal(keys, kc) and np.array_equal(values, vc)


@pytest.mark.parametrize("room", [24 * MIB, 2 * MIB])
def test_key_ranges_leave_the_budget_alone(room):
    """The key ranges' records (17 MB here) are memory the call does without:
    with room for them, an allocation that takes that room afterwards succeeds;
    without, the call runs, evicts no idle block and takes nothing."""
    say("flash records", room)
    tokens, start, qh, kvh = 1024, 1024, 16, 4
    q, k, v, kc, vc = operands(9500, tokens, start, qh, kvh)
    limit = 96 * MIB
    be = HipBackend(0, limits=Limits(max_total_bytes=limit))
    try:
        bufs = [up(be, a) for a in (q, k, v, kc, vc)]
        out = be.allocate_f32(q.shape)
        idle = be.allocate_f32((MIB // 4,))
        held = []
        while (want := limit - total(be.resource_report()) - room) >= MIB:
            held.append(be.allocate_f32(((1 << (want.bit_length() - 1)) // 4,)))
        idle.release()
        before = total(be.resource_report())
        assert room <= limit - before < room + MIB
        for _ in range(2):
            be.causal_gqa(out, *bufs, CacheLength(start), GqaSpec(qh, kvh, D))
            after = total(be.resource_report())
            assert after > before if room > 17 * MIB else after == before
        be.allocate_f32((1 << (room.bit_length() - 3),)).release()
        for buf in held:  # room for the readback
            buf.release()
        want, bound = reference(q, np.concatenate([kc[:start], k]),
                                np.concatenate([vc[:start], v]), start, qh, kvh)
        assert np.all(np.abs(be.read(out).astype(np.float64) - want) <= bound)
    finally:
        be.close()


def test_capture_keeps_no_pool_block(backend):
    """A captured call writes nothing but its output and caches when the graph
    runs, whatever the pool's idle blocks hold by then."""
    say("flash capture")
    tokens, start, qh, kvh = 1024, 1024, 16, 4
    q, k, v, kc, vc = operands(9600, tokens, start, qh, kvh)
    want, bound = reference(q, np.concatenate([kc[:start], k]), np.concatenate([vc[:start], v]),
                            start, qh, kvh)
    bufs, out = [up(backend, a) for a in (q, k, v, kc, vc)], backend.allocate_f32(q.shape)
    zeros = up(backend, np.zeros_like(q))

    def call():
        backend.causal_gqa(out, *bufs, CacheLength(start), GqaSpec(qh, kvh, D))

    call()  # leaves its records' block idle
    backend.synchronize()
    hip, stream = hiptime.hip(), ctypes.c_void_p(backend.stream())
    graph, program = ctypes.c_void_p(), ctypes.c_void_p()
    hiptime.check(hip.hipStreamBeginCapture(stream, 0), "begin capture")
    try:
        call()
    finally:
        hiptime.check(hip.hipStreamEndCapture(stream, ctypes.byref(graph)), "end capture")
    hiptime.check(hip.hipGraphInstantiate(ctypes.byref(program), graph, None, None,
                                          ctypes.c_size_t(0)), "instantiate")
    sentinel = np.full((tokens * qh * 2 * (D + 2),), 7.0, np.float32)  # takes that block
    other = up(backend, sentinel)
    for _ in range(3):
        backend.copy(out, zeros)
        hiptime.check(hip.hipGraphLaunch(program, stream), "launch")
        backend.synchronize()
        assert np.all(np.abs(backend.read(out).astype(np.float64) - want) <= bound)
        assert np.array_equal(backend.read(other), sentinel)
    hiptime.check(hip.hipGraphExecDestroy(program), "destroy")
    hiptime.check(hip.hipGraphDestroy(graph), "destroy")
