"""float32 attention whose products run as six products of bf16 parts (csrc/attention_f32.hip), and a mask's set tiles in equal shares
(csrc/attention_balance.hpp): the edges of tiles, query blocks and shares, and values that have no parts, against float64."""
import math

import numpy as np
import pytest

from anygpu_amd import synth
from helpers import scaled_rel_err
from test_gpu_parity import dev, host

pytestmark = pytest.mark.gpu

# A product of two floats as six products of their parts is off by 2^-24 at most, fp32 sums of some thousand of them by 1e-6 of the terms' norm; the
# softcap's tanh from exp2 and a reciprocal by 2e-6 of the cap.
TOL = 1e-5


def attend64(q, k, v, alpha, softcap=0.0, hidden=None, bias=None):
    """softmax(softcap(alpha q k^T) + bias) v in float64; rows without a visible key: zeros"""
    k, v = (np.repeat(t, q.shape[0] // t.shape[0], axis=0).astype(np.float64) for t in (k, v))
    s = (q.astype(np.float64) @ k.transpose(0, 2, 1)) * alpha
    if softcap:
        s = softcap * np.tanh(s / softcap)
    if bias is not None:
        s = s + bias
    if hidden is not None:
        s[:, hidden] = -np.inf
    top = s.max(axis=-1, keepdims=True)
    p = np.exp(s - np.where(np.isfinite(top), top, 0.0))
    total = p.sum(axis=-1, keepdims=True)
    return np.where(total > 0, p / np.where(total > 0, total, 1.0), 0.0) @ v


def hidden_keys(n_q, n_k, causal, window):
    at = np.arange(n_q)[:, None] + n_k - n_q
    key = np.arange(n_k)[None, :]
    hidden = np.zeros((n_q, n_k), dtype=bool)
    if causal:
        hidden |= key > at
    if window:
        hidden |= key <= at - window
    return hidden


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("heads,kv,n_q,n_k,softcap,causal,window", [
    (2, 2, 65, 350, 0.0, True, 0), (2, 2, 130, 349, 0.0, False, 0), (4, 2, 129, 352, 0.0, False, 0), (2, 1, 129, 383, 30.0, True, 100), (3, 3, 300, 1025, 0.0, True, 0),
    (2, 2, 400, 400, 0.0, True, 33), (2, 2, 500, 353, 0.0, True, 0), (1, 1, 1000, 1000, 50.0, True, 256), (40, 8, 1100, 1100, 0.0, True, 0),
    (40, 8, 900, 900, 0.0, True, 40), (2, 2, 700, 700, 30.0, True, 600)])
def test_attention_f32_in_bf16_parts(ops, d, heads, kv, n_q, n_k, softcap, causal, window):
    q, k, v = (synth.normal(s + n_q, (1, h, n, d)) for s, h, n in ((1, heads, n_q), (2, kv, n_k), (3, kv, n_k)))
    alpha = d ** -0.5
    got = host(ops.sdp_attention_fwd(dev(q), dev(k), dev(v), alpha, softcap=softcap, causal=causal, window=window, decode=False))[0]
    want = attend64(q[0], k[0], v[0], alpha, softcap, hidden_keys(n_q, n_k, causal, window))
    assert scaled_rel_err(got, want, 1.0) <= TOL
    assert not got[want.any(axis=-1) == 0].any()


@pytest.mark.parametrize("d,heads", [(64, 24), (128, 10), (256, 3)])
def test_attention_f32_in_bf16_parts_of_like_mantissas(ops, monkeypatch, d, heads):
    # products that all leave out what they can with one sign: no further from float64 than on the fp32 instruction, to a seventh
    n = 800
    rng = np.random.default_rng(d)

    def alike():
        exponent_and_sign = rng.integers(126, 129, (heads, n, d)) << 23 | rng.integers(0, 2, (heads, n, d)) << 31
        return (exponent_and_sign | 0x00FFFF).astype(np.uint32).view(np.float32)
    q, k, v = alike(), alike(), alike()
    args = [dev(t[None]) for t in (q, k, v)]
    mask = np.zeros((1, 1, n, n), dtype=np.float32)
    want = attend64(q, k, v, d ** -0.5)

    def err(y):
        return np.linalg.norm(host(y)[0] - want) / np.linalg.norm(want)
    rules, masked = err(ops.sdp_attention_fwd(*args, d ** -0.5, decode=False)), err(ops.sdp_attention_masked_scaled_fwd(*args, dev(mask), d ** -0.5))
    monkeypatch.setenv("ANYGPU_ATTN_MASK_MAP_FROM", str(1 << 60))
    plain = err(ops.sdp_attention_masked_scaled_fwd(*args, dev(mask), d ** -0.5))
    assert max(rules, masked) <= 1.15 * plain


@pytest.mark.parametrize("d,heads", [(64, 24), (128, 10), (256, 3)])
@pytest.mark.parametrize("masked", [False, True])
def test_attention_f32_in_bf16_parts_of_small_operands(ops, d, heads, masked):
    # floats below 2^-110 have parts below the smallest bf16: blocks that hold one keep the precision of float32 all the same (fp32 sums: 1e-6), and
    # the other heads keep their bits.  Normal floats all of them: magnitudes from one to two times a power of two.
    n = 800
    q, k, v = (synth.normal(s, (heads, n, d)) for s in (1, 2, 3))
    k, v = (np.sign(t) * (1 + np.abs(t) % 1) for t in (k, v))
    mask = np.zeros((1, 1, n, n), dtype=np.float32)

    def run(*qkv):
        args = [dev(t.astype(np.float32)[None]) for t in qkv]
        return host(ops.sdp_attention_masked_scaled_fwd(*args, dev(mask), d ** -0.5) if masked else ops.sdp_attention_fwd(*args, d ** -0.5, decode=False))[0]

    def small(t, exponent):
        t = t.copy()
        t[0] = np.ldexp(t[0], exponent)
        return t.astype(np.float32)
    base, want = run(q, k, v), attend64(q[:1].astype(np.float32), k[:1].astype(np.float32), v[:1].astype(np.float32), d ** -0.5)
    for exponent in (-110, -112, -118, -125):
        for at, got in ((exponent, run(q, k, small(v, exponent))), (0, run(small(q, -exponent), small(k, exponent), v)), (0, run(small(q, exponent), small(k, -exponent), v))):
            assert np.array_equal(got[1:], base[1:])
            got = np.ldexp(got[0].astype(np.float64), -at)
            if at == 0 or exponent > -118:
                assert np.linalg.norm(got - want) <= 2e-6 * np.linalg.norm(want), exponent
            else:
                # (results here are floats below the smallest normal one: half a step of 2^-149 each)
                assert np.all(np.abs(got - want) <= 1e-5 * np.abs(want).max() + 2.0 ** (-150 - at)), exponent


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("masked", [False, True])
def test_attention_f32_in_bf16_parts_of_values_without_parts(ops, d, masked):
    # an infinity or a NaN reaches the queries that see its key, in the column it stands in, and no other block of queries; the largest floats
    # and floats near the smallest one have parts like all others
    import torch
    heads, n = (26, 800) if masked else (30, 800)
    q, k, v = (synth.normal(s, (1, heads, n, d)) for s in (1, 2, 3))
    alpha = d ** -0.5

    def run(q, k, v):
        if not masked:
            return host(ops.sdp_attention_fwd(dev(q), dev(k), dev(v), alpha, causal=True, decode=False))[0]
        mask = np.where(hidden_keys(n, n, True, 0), -np.inf, 0.0).astype(np.float32).reshape(1, 1, n, n)
        return host(ops.sdp_attention_masked_scaled_fwd(dev(q), dev(k), dev(v), dev(mask), alpha))[0]
    base = run(q, k, v)
    w = v.copy()
    w[0, 0, 300, 5], w[0, 1, 700, 7] = math.inf, math.nan
    got = run(q, k, w)
    assert np.array_equal(got[2:], base[2:])
    assert np.all(got[0, 300:, 5] == math.inf) and np.all(np.isnan(got[1, 700:, 7]))
    for h, key, col in ((0, 300, 5), (1, 700, 7)):
        rest = np.delete(got[h], col, axis=1)
        assert scaled_rel_err(rest, np.delete(base[h], col, axis=1), 1.0) <= TOL
        assert np.isfinite(got[h, :key // 128 * 128, col]).all()
    kk = k.copy()
    kk[0, 0, 500, 0], kk[0, 1, 256] = math.nan, 0.0
    kk[0, 1, 256, 3] = -math.inf * np.sign(q[0, 1, 790, 3])
    got = run(q, kk, v)
    assert np.array_equal(got[2:], base[2:])
    assert np.all(np.isnan(got[0, 500:])) and np.isfinite(got[0, :384]).all()
    assert np.isfinite(got[1, 790]).all()                                # the key's score is -inf there: no weight
    # scores of order one from tiny queries and large keys; a large result (floats from 2^-110 on have all of their parts)
    got = run((q * np.float32(2.0 ** -105)), (k * np.float32(2.0 ** 105)), (v * np.float32(2.0 ** 100)))
    assert scaled_rel_err(got * 2.0 ** -100, base, 1.0) <= TOL


@pytest.mark.parametrize("d,block", [(64, 64), (128, 64), (256, 128)])
@pytest.mark.parametrize("heads,window", [(2, 0), (2, 200), (50, 0), (50, 200)])
def test_attention_f32_value_that_is_not_finite_reaches_its_query_block(ops, d, block, heads, window):
    # the queries that see its key, and of those that the rules hide it from at most the rest of a block of 64 (head dimension 256: 128): the blocks of the fp32 instruction
    n, key = 800, 485
    q, k, v = (synth.normal(s, (1, heads, n, d)) for s in (1, 2, 3))
    v[0, 0, key, 5], v[0, 1, key] = math.nan, math.inf
    got = host(ops.sdp_attention_fwd(dev(q), dev(k), dev(v), d ** -0.5, causal=True, window=window, decode=False))[0]
    # (a block walks whole tiles: its last query that sees a key of the tile of 32 that holds this one, its first likewise)
    tile = key // 32 * 32
    first, last = tile // block * block, n if window == 0 else min(n, (tile + 31 + window - 1) // block * block + block)
    for h, cols in ((0, [5]), (1, range(d))):
        assert not np.isfinite(got[h][key:key + window or n, cols]).any()
        assert np.isfinite(got[h][:first]).all() and np.isfinite(got[h][last:]).all()
        assert np.isfinite(np.delete(got[h], cols, axis=1)).all()
    assert np.isfinite(got[2:]).all()


@pytest.mark.parametrize("heads,n_q,n_k,d,kind", [
    (1, 800, 801, 256, "causal"), (2, 1000, 600, 256, "bias"), (3, 780, 1300, 256, "blind blocks"), (1, 130, 5003, 256, "window"), (7, 775, 775, 256, "nothing"),
    (25, 900, 773, 128, "blind blocks"), (1, 300, 520, 256, "bias"), (9, 830, 1001, 128, "window"), (26, 790, 790, 64, "window"), (24, 1000, 700, 64, "bias"), (300, 800, 800, 256, "window"), (40, 770, 800, 128, "causal")])
def test_attention_f32_mask_tensor_in_equal_shares(ops, monkeypatch, heads, n_q, n_k, d, kind):
    # shares that end inside query blocks, at their ends, and that hold several; query blocks and heads without a set tile; more query blocks
    # than shares are made for (300 heads); against float64 and, where shares are made, against the launch without a map
    rng = np.random.default_rng(n_q)
    q, k, v = (synth.normal(s, (1, heads, n, d)) for s, n in ((1, n_q), (2, n_k), (3, n_k)))
    if kind in ("causal", "window"):
        mask = np.where(hidden_keys(n_q, n_k, True, 100 if kind == "window" else 0), -np.inf, 0.0)
    elif kind == "nothing":
        mask = np.full((n_q, n_k), -np.inf)
        mask[n_q - 1, n_k - 1] = 1.0
    else:
        mask = rng.normal(0.0, 2.0, (n_q, n_k))
        if kind == "blind blocks":
            mask[128:256] = -np.inf
            mask[n_q - 70:] = np.finfo(np.float32).min           # the lowest float hides as well
            mask[300:600, 64:n_k - 40] = -np.inf
    mask = mask.astype(np.float32)
    alpha = d ** -0.5
    args = [dev(t) for t in (q, k, v, mask.reshape(1, 1, n_q, n_k))]
    got = host(ops.sdp_attention_masked_scaled_fwd(*args, alpha))[0]
    again = host(ops.sdp_attention_masked_scaled_fwd(*args, alpha))[0]
    assert np.array_equal(got, again)
    bias = np.where(mask < -3e38, -np.inf, mask).astype(np.float64)
    some = [0, heads - 1] if heads > 8 else range(heads)
    want = attend64(q[0, some], k[0, some], v[0, some], alpha, bias=bias)
    assert scaled_rel_err(got[some], want, 1.0) <= TOL
    assert not got[:, ~np.isfinite(bias).any(axis=1)].any()
    monkeypatch.setenv("ANYGPU_ATTN_MASK_MAP_FROM", str(1 << 60))
    whole = host(ops.sdp_attention_masked_scaled_fwd(*args, alpha))[0]
    assert scaled_rel_err(got, whole, 1.0) <= TOL


def test_attention_f32_equal_shares_replayed_from_a_graph(ops):
    # with a caller's workspace that holds the map and the partial results every replay gives the eager call's bits, a new mask and new queries each
    # time; without one the captured call makes no map, and agrees to rounding
    import torch
    h, n, d = 2, 900, 256
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    q, k, v = (torch.empty(1, h, n, d, device="cuda").normal_(generator=gen) for _ in range(3))
    mask = torch.empty(1, 1, n, n, device="cuda")
    workspace = torch.empty(160 << 20, dtype=torch.uint8, device="cuda")
    stream = torch.cuda.Stream()
    graphs = []
    for ws in (workspace, None):
        with torch.cuda.stream(stream):
            ops.set_workspace(ws, stream)
            mask.normal_(generator=gen)
            ops.sdp_attention_masked_scaled_fwd(q, k, v, mask, 0.0625)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out = ops.sdp_attention_masked_scaled_fwd(q, k, v, mask, 0.0625)
        graphs.append((graph, out))
        for turn in range(4):
            q.normal_(generator=gen)
            mask.normal_(generator=gen)
            mask[..., (turn + 1) * 200:] = -math.inf
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            eager = ops.sdp_attention_masked_scaled_fwd(q, k, v, mask, 0.0625)
            torch.cuda.synchronize()
            if ws is not None:
                assert torch.equal(out, eager), turn
            else:
                assert float((out - eager).abs().max()) <= TOL, turn
    ops.set_workspace(None, stream)
