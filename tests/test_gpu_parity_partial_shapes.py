"""GPU parity of the kernels that take part of a wider operator's shapes (few rows, small products, 32 queries per wave, key ranges in
parts), at the sizes where such a kernel can go wrong, against the oracle or exact integers."""
import math

import numpy as np
import pytest

from anygpu_amd import synth
from helpers import exact_int_product, scaled_rel_err
from test_gpu_parity import ATTN_D256_CASES, TOL_F16_GEMM, TOL_F16_ROWOPS, TOL_F32, dev, hide_key_stripes, host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("m,steps,n", [(1, 36, 2304), (2, 16, 300), (3, 17, 1), (8, 36, 9216), (8, 23, 2305), (5, 31, 5003), (4, 16, 7001), (7, 18, 8193),
                                       (9, 16, 257), (16, 36, 2048), (12, 19, 4099), (16, 17, 6000), (8, 144, 130)])
def test_mm_few_rows_k_cut_over_waves(ops, oracle, dtype, m, steps, n):
    # up to 16 rows against k-contiguous weights, K in steps of 128 bytes from 16 of them on (two for each of eight waves), blocks of 1 to
    # 32 columns that end past N, operands and results inside wider buffers.  Small integers: the sums are exact in both types (below 2048).
    import torch
    from anygpu_amd import capi
    np_dt, t_dt = (np.float16, torch.float16) if dtype == "f16" else (np.float32, torch.float32)
    pad, k = (8, 64 * steps) if dtype == "f16" else (4, 32 * steps)
    a, bt, b2t = (synth.integers(s, shape, -2, 2).astype(np_dt) for s, shape in ((m + 1, (m, k)), (n + 2, (n, k)), (n + 3, (n, k))))
    want = exact_int_product(a, np.ascontiguousarray(bt.T))
    assert np.max(np.abs(want)) < 2048
    abuf, bbuf = torch.full((m, k + pad), 9.0, dtype=t_dt, device="cuda"), torch.full((n, k + 2 * pad), 9.0, dtype=t_dt, device="cuda")
    abuf[:, :k], bbuf[:, :k] = dev(a), dev(bt)
    cbuf = torch.full((m + 1, n + 3), -7.0, dtype=t_dt, device="cuda")
    ops.tensor_mm(abuf[:, :k], bbuf[:, :k], out=cbuf[:m, :n], b_layout=capi.B_COL_MAJOR)
    got = host(cbuf).astype(np.int64)
    assert np.array_equal(got[:m, :n], want)
    assert np.all(got[m:, :] == -7) and np.all(got[:, n:] == -7)
    bias = synth.integers(3, (n,), -9, 9).astype(np_dt)
    assert np.array_equal(host(ops.tensor_gemm(dev(a), dev(bt), dev(bias), b_layout=capi.B_COL_MAJOR)).astype(np.int64), want + bias.astype(np.int64))
    # the epilogues on sums of size O(1) (a power of two keeps them exact): half an ulp of the result's type, and 1e-6 of the
    # arguments for the fp32 tanh (tanh_for_half: 4e-5 of the result)
    scale = 2.0 ** -6
    half_ulp = 2.0 ** -11 if dtype == "f16" else 2.0 ** -24
    s1, s2 = want * scale, exact_int_product(a, np.ascontiguousarray(b2t.T)) * scale
    got = host(ops.tensor_gemma_linear_softcap(dev((a * scale).astype(np_dt)).reshape(1, m, k), dev(bt), 30.0)).astype(np.float64).reshape(m, n)
    capped = 30.0 * np.tanh(s1 / 30.0)
    assert np.all(np.abs(got - capped) <= (half_ulp + (4.4e-5 if dtype == "f16" else 0.0)) * np.abs(capped) + 30.0 * 1e-6)
    got = host(ops.mlp_gemma2_fused_upproj(dev((a * scale).astype(np_dt)), dev(bt), dev(b2t), b_layout=capi.B_COL_MAJOR)).astype(np.float64)
    gated = 0.5 * s1 * (1.0 + np.tanh(math.sqrt(2.0 / math.pi) * (s1 + 0.044715 * s1 ** 3))) * s2
    assert np.all(np.abs(got - gated) <= half_ulp * np.abs(gated) + 1e-6 * np.abs(s1 * s2) + 2.0 ** -24)


@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("m", [3, 8, 16])
def test_mm_few_rows_k_cut_over_waves_nan_and_infinities(ops, dtype, m):
    # a NaN or an infinity reaches the row (left operand) or column (weights) that it belongs to and no other, in either half of a step's
    # chunks and in the shares of different waves; +inf and -inf that meet in a sum give NaN
    import torch
    from anygpu_amd import capi
    t_dt, k, n = (torch.float16, 64 * 19, 300) if dtype == "f16" else (torch.float32, 32 * 19, 300)
    a, w = (torch.from_numpy(synth.integers(s, shape, -2, 2)).to(t_dt) for s, shape in ((5, (m, k)), (6, (n, k))))
    a[1, 3] = math.nan
    a[2, k - 1], w[:, k - 1] = math.inf, 1.0
    w[7, k // 2 + 9], a[:, k // 2 + 9] = math.nan, 2.0
    w[9, 17], w[9, k - 40], a[:, 17], a[:, k - 40] = math.inf, -math.inf, 1.0, 1.0
    w[299, 40], a[:, 40] = -math.inf, 1.0
    want = a.double() @ w.double().t().contiguous()
    got = host(ops.tensor_mm(dev(a.numpy()), dev(w.numpy()), b_layout=capi.B_COL_MAJOR)).astype(np.float64)
    assert np.array_equal(got, want.numpy(), equal_nan=True)
    assert 0 < np.isnan(got).sum() < got.size // 2


@pytest.mark.parametrize("m,n,k", [(17, 31, 1), (3, 33, 31), (33, 32, 32), (32, 95, 63), (64, 64, 128), (65, 70, 129), (31, 100, 256),
                                   (40, 33, 385), (128, 128, 768), (97, 130, 1533), (700, 701, 333)])
@pytest.mark.parametrize("layout", ["kn", "nk"])
def test_gemm_f32_small_products(ops, oracle, m, n, k, layout):
    # 32 x 32 tiles with K cut over four waves in steps of 32: edges of tiles, one step, fewer steps than waves, the rest of K in
    # each wave's turn, padded rows at odd pitches and element alignment.  Integer-valued: every order of summation is
    # exact.  The buffers behind the operands hold NaN: nothing of them may reach a sum, and what lies between the rows of C stays.
    import torch
    from anygpu_amd import capi
    a = synth.integers(91, (m, k), -8, 8)
    b = synth.integers(92, (k, n), -8, 8)
    bias = synth.integers(93, (n,), -8, 8)
    want = exact_int_product(a, b)
    b_store = b if layout == "kn" else np.ascontiguousarray(b.T)
    lay = capi.B_ROW_MAJOR if layout == "kn" else capi.B_COL_MAJOR

    def padded(x, extra, shift):
        buf = torch.full((x.shape[0] * (x.shape[1] + extra) + shift,), float("nan"), device="cuda")
        view = buf[shift:].view(x.shape[0], x.shape[1] + extra)[:, :x.shape[1]]
        view.copy_(dev(x))
        return view

    for extra, shift in ((0, 0), (3, 1)):
        out = padded(np.zeros((m, n), np.float32), extra, shift)
        got = host(ops.tensor_mm(padded(a, extra, shift), padded(b_store, extra, shift), out=out, b_layout=lay))
        assert np.array_equal(got.astype(np.int64), want)
        if extra:
            assert bool(torch.isnan(out._base[shift:].view(m, n + extra)[:, n:]).all())
    got = host(ops.tensor_gemm(dev(a), dev(b_store), dev(bias), b_layout=lay))
    assert np.array_equal(got.astype(np.int64), want + bias.astype(np.int64))


def test_sdp_attention_f32_mask_tensor_blocks_in_parts_that_fill_the_rounds(ops, oracle, monkeypatch):
    # head dimension 256 with fewer blocks than CUs (16 heads x 12 blocks of 128 queries; 66 key tiles): four parts, whose results take 101 MB,
    # more than the workspace holds to begin with, which grows.  Against a caller's workspace of 64 MB, which has room for two parts,
    # and one that only has room for the map (whole blocks), and one head against the oracle
    import torch
    heads, n_q, n_k, d = 16, 1500, 2090, 256
    q = synth.normal(81, (1, heads, n_q, d))
    k = synth.normal(82, (1, heads, n_k, d))
    v = synth.normal(83, (1, heads, n_k, d))
    alpha = float(d) ** -0.5
    rng = np.random.default_rng(84)
    mask = rng.normal(0.0, 1.0, (n_q, n_k)).astype(np.float32)
    hide_key_stripes(mask, rng)
    mask4 = mask.reshape(1, 1, n_q, n_k)
    dq, dk, dv, dm = dev(q), dev(k), dev(v), dev(mask4)
    monkeypatch.setenv("ANYGPU_ATTN_MASK_MAP_FROM", "0")
    got = [host(ops.sdp_attention_masked_scaled_fwd(dq, dk, dv, dm, alpha))]
    for size in (1 << 26, 1 << 17):
        workspace = torch.empty(size, dtype=torch.uint8, device="cuda")
        ops.set_workspace(workspace)
        try:
            got.append(host(ops.sdp_attention_masked_scaled_fwd(dq, dk, dv, dm, alpha)))
        finally:
            torch.cuda.synchronize()
            ops.set_workspace(None)
    assert all(np.isfinite(y).all() for y in got)
    for i, j in ((0, 1), (0, 2), (1, 2)):
        assert scaled_rel_err(got[i], got[j], 1.0) <= 1e-5
        assert not np.array_equal(got[i], got[j]), "the three runs were expected to sum in different orders"
    want = oracle.sdp_attention_masked_scaled_fwd(q[:, 3:4], k[:, 3:4], v[:, 3:4], mask4, alpha, threads=8)
    assert scaled_rel_err(got[0][:, 3:4], want, 1.0) <= TOL_F32


# head dimensions 64 and 128 run 32 queries per wave, four waves and 128 queries per block, tiles of 64 keys, where there are more query
# blocks than CUs (here: 66 copies of four heads), 16 rows per block or, with a single tile of keys, 16 queries per wave in eight waves where there are few: one query and
# the edges of a wave's and a block's queries, tiles of one key, one short of whole and whole, queries of a wave that see
# nothing, and the first and last tile of a window that only some waves of a block see
@pytest.mark.parametrize("copies", [1, 66])
@pytest.mark.parametrize("n_q,n_k,causal,window", [(1, 65, True, 0), (31, 64, True, 0), (33, 63, False, 0), (127, 129, True, 0), (128, 128, True, 0),
                                                    (129, 257, True, 70), (160, 100, True, 0), (300, 321, False, 64), (257, 600, True, 1)])
@pytest.mark.parametrize("d,cap,alpha", [(64, 0.0, 0.125), (128, 0.0, -0.0884), (64, 30.0, 0.0), (128, 50.0, 0.0884)])
def test_sdp_attention_fused_kernel_32_queries_per_wave(ops, oracle, n_q, n_k, causal, window, d, cap, alpha, copies):
    heads, kv_heads = 4, 2
    if window and copies > 1:
        copies *= 2                                              # (under a window from one and a half blocks per CU on)
    q = synth.normal(1 + n_q, (1, heads, n_q, d)).astype(np.float16)
    k = synth.normal(2 + n_k, (1, kv_heads, n_k, d)).astype(np.float16) * np.float16(4.0)        # (scores of tens: the running maximum moves)
    v = synth.normal(3 + d, (1, kv_heads, n_k, d)).astype(np.float16)
    got = host(ops.sdp_attention_fwd(*(dev(t).repeat(copies, 1, 1, 1) for t in (q, k, v)), alpha, softcap=cap, causal=causal, window=window,
                                     decode=False)).astype(np.float32)
    want = oracle.sdp_attention_rules(*(oracle.cvt_f16_to_f32(t)[0] for t in (q, k, v)), alpha=alpha, softcap=cap,
                                      causal=causal, window=window, q_per_kv=heads // kv_heads, threads=8)
    blind = ~np.isfinite(want).all(axis=-1)                      # queries without a visible key: zeros
    assert not got[0][blind].any()
    assert np.isfinite(got).all()
    assert np.array_equal(got, np.broadcast_to(got[:1], got.shape))
    # p rounded to fp16 (2^-11 each, weights that sum to 1) and the result's own rounding, values of up to about 4
    assert scaled_rel_err(got[0][~blind], want[~blind], 1.0) <= TOL_F16_ROWOPS * 2


# the same kernel's walk over two tiles at a time: waves that see one to seven tiles, odd and even in number, whose first and last ones lie
# before, on and behind those of the block's other waves, the last tile whole, of one key and one short
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("n_q,n_k,causal,window", [(128, 192, True, 0), (128, 193, True, 65), (100, 319, True, 130), (130, 385, True, 200), (60, 447, False, 0),
                                                    (256, 256, True, 33), (129, 448, True, 64), (97, 384, False, 90)])
def test_sdp_attention_32_queries_per_wave_tiles_in_pairs(ops, oracle, n_q, n_k, causal, window, d):
    copies, heads = 132, 4
    q, k, v = (synth.normal(80 + i, (1, heads, n, d)).astype(np.float16) for i, n in enumerate((n_q, n_k, n_k)))
    got = host(ops.sdp_attention_fwd(*(dev(t).repeat(copies, 1, 1, 1) for t in (q, k, v)), d ** -0.5, causal=causal, window=window,
                                     decode=False)).astype(np.float32)
    want = oracle.sdp_attention_rules(*(oracle.cvt_f16_to_f32(t)[0] for t in (q, k, v)), alpha=d ** -0.5, softcap=0.0,
                                      causal=causal, window=window, q_per_kv=1, threads=8)
    blind = ~np.isfinite(want).all(axis=-1)                      # queries without a visible key: zeros
    assert not got[0][blind].any() and np.isfinite(got).all()
    assert np.array_equal(got, np.broadcast_to(got[:1], got.shape))
    # p rounded to fp16 (2^-11 each, weights that sum to 1) and the result's own rounding, values of up to about 4
    assert scaled_rel_err(got[0][~blind], want[~blind], 1.0) <= TOL_F16_ROWOPS * 2


# blocks of enough tiles that the scores of one run beside the softmax of the one before (those above take them in turn): the first query block of a causal launch with
# waves of one and two tiles, ranges that begin and end within and between blocks, odd and even numbers of tiles
@pytest.mark.parametrize("d,cap", [(64, 0.0), (128, 0.0), (64, 30.0), (128, 30.0)])
@pytest.mark.parametrize("n_q,n_k,causal,window", [(1000, 1000, True, 0), (897, 960, True, 0), (1100, 1161, True, 600), (130, 641, False, 0), (97, 577, True, 0), (385, 1025, False, 520)])
def test_sdp_attention_32_queries_per_wave_tiles_overlapped(ops, oracle, n_q, n_k, causal, window, d, cap):
    copies, heads = 66, 4
    q, k, v = (synth.normal(80 + i, (1, heads, n, d)).astype(np.float16) for i, n in enumerate((n_q, n_k, n_k)))
    k *= np.float16(2.0)
    got = host(ops.sdp_attention_fwd(*(dev(t).repeat(copies, 1, 1, 1) for t in (q, k, v)), d ** -0.5, softcap=cap, causal=causal, window=window,
                                     decode=False)).astype(np.float32)
    want = oracle.sdp_attention_rules(*(oracle.cvt_f16_to_f32(t)[0] for t in (q, k, v)), alpha=d ** -0.5, softcap=cap,
                                      causal=causal, window=window, q_per_kv=1, threads=8)
    assert np.isfinite(want).all() and np.isfinite(got).all()
    assert np.array_equal(got, np.broadcast_to(got[:1], got.shape))
    # p rounded to fp16 (2^-11 each, weights that sum to 1) and the result's own rounding, values of up to about 4
    assert scaled_rel_err(got[0], want, 1.0) <= TOL_F16_ROWOPS * 2


# a window over a long cache: blocks of two or three tiles, products and softmax in turn, in parts of the range that the window leaves mostly empty, and whole without a workspace for them
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("cap", [0.0, 30.0])
def test_sdp_attention_32_queries_per_wave_short_window_in_parts(ops, oracle, d, cap):
    import torch
    copies, heads, n_q, n_k, window = (40 if d == 64 else 65), 4, 200, 6000, 100        # one and a quarter and two rounds of blocks, cut into three and two parts
    q, k, v = (synth.normal(80 + i, (1, heads, n, d)).astype(np.float16) for i, n in enumerate((n_q, n_k, n_k)))
    args = [dev(t).repeat(copies, 1, 1, 1) for t in (q, k, v)]

    def run(workspace_bytes):
        workspace = torch.empty((workspace_bytes,), dtype=torch.uint8, device="cuda")
        ops.set_workspace(workspace)
        try:
            return host(ops.sdp_attention_fwd(*args, d ** -0.5, softcap=cap, causal=True, window=window, decode=False)).astype(np.float32)
        finally:
            torch.cuda.synchronize()
            ops.set_workspace(None)
    parts, whole = run(160 << 20), run(256)
    assert not np.array_equal(parts, whole), "the launch was expected to take parts of the key range"
    want = oracle.sdp_attention_rules(*(oracle.cvt_f16_to_f32(t)[0] for t in (q, k, v)), alpha=d ** -0.5, softcap=cap, causal=True, window=window, q_per_kv=1, threads=8)
    for got in (parts, whole):
        assert np.isfinite(got).all() and np.array_equal(got, np.broadcast_to(got[:1], got.shape))
        assert scaled_rel_err(got[0], want, 1.0) <= TOL_F16_ROWOPS * 2


# the same kernel where the second round of blocks is dispatched backwards: 56 to 66 blocks per XCD (55.5 are just too few), with padding at the end of a head and of the launch
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("copies,heads,kv_heads,n,causal", [(7, 4, 2, 1930, True), (40, 4, 2, 300, True), (37, 4, 2, 300, True), (31, 5, 1, 260, True), (64, 4, 4, 200, False), (33, 4, 2, 510, True)])
def test_sdp_attention_32_queries_per_wave_second_round_backwards(ops, oracle, copies, heads, kv_heads, n, causal, d):
    q, k, v = (synth.normal(s + n, (1, h, n, d)).astype(np.float16) for s, h in ((1, heads), (2, kv_heads), (3, kv_heads)))
    got = host(ops.sdp_attention_fwd(*(dev(t).repeat(copies, 1, 1, 1) for t in (q, k, v)), d ** -0.5, causal=causal)).astype(np.float32)
    want = oracle.sdp_attention_rules(*(oracle.cvt_f16_to_f32(t)[0] for t in (q, k, v)), alpha=d ** -0.5, softcap=0.0, causal=causal, window=0, q_per_kv=heads // kv_heads, threads=8)
    assert np.array_equal(got, np.broadcast_to(got[:1], got.shape))
    assert scaled_rel_err(got[0], want, 1.0) <= TOL_F16_ROWOPS * 2


# launches of few query blocks: 16 rows per block, the tiles of 32 keys shared out among eight waves (up to a block per CU) or four (more, at 64 and 128: most of the copies; copies of few keys, and at 64
# and 128 a single tile of 64 keys, run on the kernels of 128 queries per block).
# Rows and keys on both sides of 16 and 32, as many tiles as waves and one more, blocks whose window starts behind the first tile,
# queries that see nothing, and generation steps whose rows of several heads and queries share a block
@pytest.mark.parametrize("copies", [1, 40])
@pytest.mark.parametrize("heads,kv_heads,n_q,n_k,causal,window", [(4, 2, 17, 17, True, 0), (4, 1, 16, 31, False, 0), (2, 2, 33, 32, True, 0), (4, 4, 40, 257, True, 0),
                                                                   (4, 2, 31, 288, False, 0), (4, 2, 100, 129, True, 33), (2, 1, 70, 600, False, 64), (4, 2, 60, 40, True, 0),
                                                                   (4, 2, 80, 150, True, 1), (6, 2, 5, 300, True, 0), (8, 4, 1, 256, True, 0), (4, 4, 4, 319, True, 100),
                                                                   (12, 4, 3, 290, False, 0), (40, 2, 1, 260, True, 0),
                                                                   (4, 2, 130, 97, True, 0), (4, 4, 33, 65, True, 0), (3, 1, 16, 95, False, 0)])
@pytest.mark.parametrize("d,cap,alpha", [(64, 0.0, 0.125), (128, 30.0, -0.0884), (256, 0.0, 0.0625), (256, 50.0, 0.0625)])
def test_sdp_attention_few_rows_keys_over_waves(ops, oracle, heads, kv_heads, n_q, n_k, causal, window, d, cap, alpha, copies):
    q = synth.normal(1 + n_q, (1, heads, n_q, d)).astype(np.float16)
    k = synth.normal(2 + n_k, (1, kv_heads, n_k, d)).astype(np.float16) * np.float16(4.0)        # (scores of tens: the running maximum moves)
    v = synth.normal(3 + d, (1, kv_heads, n_k, d)).astype(np.float16)
    got = host(ops.sdp_attention_fwd(*(dev(t).repeat(copies, 1, 1, 1) for t in (q, k, v)), alpha, softcap=cap, causal=causal, window=window)).astype(np.float32)
    want = oracle.sdp_attention_rules(*(oracle.cvt_f16_to_f32(t)[0] for t in (q, k, v)), alpha=alpha, softcap=cap,
                                      causal=causal, window=window, q_per_kv=heads // kv_heads, threads=8)
    blind = ~np.isfinite(want).all(axis=-1)                      # queries without a visible key: zeros
    assert not got[0][blind].any() and np.isfinite(got).all()
    assert np.array_equal(got, np.broadcast_to(got[:1], got.shape))
    # p rounded to fp16 (2^-11 each, weights that sum to 1) and the result's own rounding, values of up to about 4
    assert scaled_rel_err(got[0][~blind], want[~blind], 1.0) <= TOL_F16_ROWOPS * 2


@pytest.mark.parametrize("n_q", [1, 40])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_sdp_attention_few_rows_nan_infinities_and_large_scores(ops, n_q, d):
    # a NaN in a query reaches its row, a NaN in the last key every row that sees it; among scores of 10^9 the largest one's row of v,
    # bit for bit, whichever wave has it; strangers around the keys are never read
    import torch
    heads, n = 4, 288
    q, k, v = (synth.normal(70 + i, (heads, m, d)).astype(np.float16) for i, m in enumerate((n_q, n, n)))
    q[1, n_q // 2, 3] = np.nan
    k[2, n - 1, 0] = np.nan
    got = host(ops.sdp_attention_fwd(*(dev(t) for t in (q, k, v)), d ** -0.5, causal=True))
    seen = np.zeros((heads, n_q), dtype=bool)
    seen[1, n_q // 2] = seen[2, n_q - 1] = True
    assert np.array_equal(np.isnan(got).all(-1), seen) and np.array_equal(np.isnan(got).any(-1), seen)
    order = np.random.default_rng(6).permutation(n)
    q = torch.full((1, heads, n_q, d), 10000.0, dtype=torch.half, device="cuda")
    pool = torch.full((n + 64, d), math.nan, dtype=torch.half, device="cuda")
    pool[32:32 + n] = dev((10000.0 - 16.0 * order)[:, None].repeat(d, axis=1).astype(np.float16))
    v = synth.normal(9, (1, 1, n, d)).astype(np.float16)
    got = host(ops.sdp_attention_fwd(q, pool[32:32 + n].view(1, 1, n, d), dev(v), 1.0))
    assert np.array_equal(got, np.broadcast_to(v[0, 0, int(np.argmin(order))], got.shape))


# the same in float32 (tiles of 16 keys): fp32 sums of up to 300 products and weights
@pytest.mark.parametrize("copies", [1, 40])
@pytest.mark.parametrize("heads,kv_heads,n_q,n_k,causal,window", [(4, 2, 17, 17, True, 0), (4, 1, 16, 15, False, 0), (2, 2, 33, 16, True, 0), (4, 4, 40, 129, True, 0),
                                                                   (4, 2, 31, 128, False, 0), (4, 2, 100, 145, True, 33), (2, 1, 70, 300, False, 64), (4, 2, 60, 40, True, 0),
                                                                   (4, 2, 80, 150, True, 1), (4, 4, 1, 31, True, 0)])
@pytest.mark.parametrize("d,cap,alpha", [(64, 0.0, 0.125), (128, 30.0, -0.0884), (256, 0.0, 0.0625), (256, 50.0, 0.0625)])
def test_sdp_attention_f32_few_rows_keys_over_waves(ops, oracle, heads, kv_heads, n_q, n_k, causal, window, d, cap, alpha, copies):
    q, k, v = (synth.normal(s + n, (1, h, n, d)) for s, h, n in ((1, heads, n_q), (2, kv_heads, n_k), (3, kv_heads, n_k)))
    got = host(ops.sdp_attention_fwd(*(dev(t).repeat(copies, 1, 1, 1) for t in (q, k, v)), alpha, softcap=cap, causal=causal, window=window, decode=False))
    want = oracle.sdp_attention_rules(q[0], k[0], v[0], alpha=alpha, softcap=cap, causal=causal, window=window, q_per_kv=heads // kv_heads, threads=8)
    blind = ~np.isfinite(want).all(axis=-1)                      # queries without a visible key: zeros
    assert not got[0][blind].any() and np.isfinite(got).all()
    assert np.array_equal(got, np.broadcast_to(got[:1], got.shape))
    assert scaled_rel_err(got[0][~blind], want[~blind], 1.0) <= TOL_F32


# the long query blocks of a causal launch: at head dimension 256 those beyond their share in two halves of their keys (2100 keys), half of the longest ones where the second round of blocks does
# not fit (3108 and 3332 under a window), none (2048 under a window, 1100, 1339; 2111 has fewer blocks than CUs), at 64 and 128 up to one and a third block per CU; in float32 some; sequence
# ends inside and on a block and a tile
@pytest.mark.parametrize("dtype,copies,heads,kv_heads,n,window,d", [("f16", 4, 4, 2, 2100, 0, 256), ("f16", 8, 4, 2, 2048, 1024, 256), ("f16", 8, 4, 2, 1100, 0, 256), ("f16", 5, 3, 1, 2111, 1500, 256), ("f16", 4, 4, 2, 3108, 1024, 256), ("f16", 4, 4, 1, 3332, 1536, 256),
                                                                    ("f32", 2, 4, 4, 2100, 0, 256), ("f32", 8, 4, 1, 1339, 0, 256), ("f32", 4, 4, 2, 1536, 1000, 256),
                                                                    ("f16", 4, 4, 2, 2600, 0, 128), ("f16", 4, 4, 2, 2600, 0, 64), ("f16", 4, 4, 2, 2688, 0, 128)])
def test_sdp_attention_causal_blocks_partly_in_halves(ops, oracle, dtype, copies, heads, kv_heads, n, window, d):
    half, alpha = dtype == "f16", d ** -0.5
    q, k, v = (synth.normal(s + n, (1, h, n, d)).astype(np.float16 if half else np.float32) for s, h in ((1, heads), (2, kv_heads), (3, kv_heads)))
    got = host(ops.sdp_attention_fwd(*(dev(t).repeat(copies, 1, 1, 1) for t in (q, k, v)), alpha, softcap=50.0, causal=True, window=window)).astype(np.float32)
    want = oracle.sdp_attention_rules(*(oracle.cvt_f16_to_f32(t)[0] if half else t[0] for t in (q, k, v)), alpha=alpha, softcap=50.0, causal=True, window=window,
                                      q_per_kv=heads // kv_heads, threads=8)
    assert np.array_equal(got, np.broadcast_to(got[:1], got.shape))
    assert scaled_rel_err(got[0], want, 1.0) <= (TOL_F16_ROWOPS * 2 if half else TOL_F32)


# and with a mask tensor: rows and tiles that it hides altogether, values of either sign, the type's lowest, keys that end inside a tile
@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("heads,n_q,n_k", [(3, 1, 1), (2, 17, 15), (4, 33, 32), (2, 40, 257), (150, 30, 100), (3, 100, 131), (2, 16, 300)])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_sdp_attention_mask_tensor_few_rows_keys_over_waves(ops, oracle, heads, n_q, n_k, d, dtype):
    ndt = np.float16 if dtype == "f16" else np.float32
    q, k, v = (synth.normal(s + n, (1, heads, n, d)).astype(ndt) for s, n in ((1, n_q), (2, n_k), (3, n_k)))
    mask = synth.normal(7, (n_q, n_k)).astype(ndt)
    if n_q > 2:
        mask[:, n_k // 2:] = np.where(synth.normal(8, (n_q, n_k - n_k // 2)) > 0, -np.inf, mask[:, n_k // 2:])
        mask[n_q // 3, :] = -np.inf                              # sees nothing: zeros
        mask[n_q - 1, :] = np.finfo(ndt).min if dtype == "f16" else -1e30
        mask[1, :n_k - 1] = -np.inf
        mask[1, n_k - 1] = 0.0
    if n_k > 64:
        mask[:, 32:64] = -np.inf
    got = host(ops.sdp_attention_masked_scaled_fwd(*(dev(t) for t in (q, k, v)), dev(mask).reshape(1, 1, n_q, n_k), d ** -0.5)).astype(np.float32)
    wide = [oracle.cvt_f16_to_f32(t) if dtype == "f16" else t for t in (q, k, v, mask)]
    want = oracle.sdp_attention_masked_scaled_fwd(*(t[:, :3] for t in wide[:3]), wide[3].reshape(1, 1, n_q, n_k), d ** -0.5, threads=8)
    seen = np.isfinite(wide[3]).any(axis=-1)
    assert not got[:, :, ~seen].any() and np.isfinite(got).all()
    tol = TOL_F16_ROWOPS * 2 if dtype == "f16" else TOL_F32
    assert scaled_rel_err(got[:, :3][:, :, seen], want[:, :, seen], 1.0) <= tol


# head dimensions 64 and 128, half a block of 128 queries to one for each CU and fewer than ten tiles: 16 queries per wave in eight waves
@pytest.mark.parametrize("copies,n_q,n_k,causal,window", [(35, 31, 64, True, 0), (35, 127, 129, True, 0), (35, 128, 128, True, 0), (35, 113, 63, False, 0), (30, 129, 257, True, 70), (30, 160, 100, True, 0),
                                                           (14, 300, 321, False, 64), (16, 257, 600, True, 1), (30, 130, 513, True, 0)])
@pytest.mark.parametrize("d,cap,alpha", [(64, 0.0, 0.125), (128, 0.0, -0.0884), (64, 30.0, 0.125), (128, 50.0, 0.0884)])
def test_sdp_attention_16_queries_per_wave(ops, oracle, copies, n_q, n_k, causal, window, d, cap, alpha):
    heads, kv_heads = 4, 2
    q = synth.normal(1 + n_q, (1, heads, n_q, d)).astype(np.float16)
    k = synth.normal(2 + n_k, (1, kv_heads, n_k, d)).astype(np.float16) * np.float16(4.0)        # (scores of tens: the running maximum moves)
    v = synth.normal(3 + d, (1, kv_heads, n_k, d)).astype(np.float16)
    got = host(ops.sdp_attention_fwd(*(dev(t).repeat(copies, 1, 1, 1) for t in (q, k, v)), alpha, softcap=cap, causal=causal, window=window, decode=False)).astype(np.float32)
    want = oracle.sdp_attention_rules(*(oracle.cvt_f16_to_f32(t)[0] for t in (q, k, v)), alpha=alpha, softcap=cap, causal=causal, window=window, q_per_kv=heads // kv_heads, threads=8)
    blind = ~np.isfinite(want).all(axis=-1)                      # queries without a visible key: zeros
    assert not got[0][blind].any() and np.isfinite(got).all()
    assert np.array_equal(got, np.broadcast_to(got[:1], got.shape))
    assert scaled_rel_err(got[0][~blind], want[~blind], 1.0) <= TOL_F16_ROWOPS * 2


# head dimension 256 with so many heads that blocks of 128 queries take the launch, whose scores of a tile run beside the softmax of the one before: the shapes of one and two tiles, short last
# tiles, windows and queries that see nothing that few heads run on 16 rows per block
@pytest.mark.parametrize("case", [case for case in ATTN_D256_CASES if case[3] < 1500] + [(2, 2, 129, 3000, 256, 0.0625, 0.0, True, 1800)])
def test_sdp_attention_head_dim_256_many_heads(ops, oracle, case):
    heads, kv_heads, n_q, n_k, d, alpha, cap, causal, window = case
    copies = 1030 // (heads * ((n_q + 15) // 16)) + 1 if n_k < 1500 else 1
    q, k, v = (synth.normal(s + n, (1, h, n, d)).astype(np.float16) for s, h, n in ((1, heads, n_q), (2, kv_heads, n_k), (3, kv_heads, n_k)))
    got = host(ops.sdp_attention_fwd(*(dev(t).repeat(copies, 1, 1, 1) for t in (q, k, v)), alpha, softcap=cap, causal=causal, window=window, decode=False)).astype(np.float32)
    want = oracle.sdp_attention_rules(*(oracle.cvt_f16_to_f32(t)[0] for t in (q, k, v)), alpha=alpha, softcap=cap, causal=causal, window=window, q_per_kv=heads // kv_heads, threads=8)
    blind = ~np.isfinite(want).all(axis=-1)                      # queries without a visible key: zeros
    assert not got[0][blind].any() and np.isfinite(got).all()
    assert np.array_equal(got, np.broadcast_to(got[:1], got.shape))
    assert scaled_rel_err(got[0][~blind], want[~blind], 1.0) <= TOL_F16_ROWOPS * 2


# alpha 0 without a softcap: the mean of the visible values, on every kernel (16 rows per block, 16 and 32 queries per wave, head dimension 256, float32 in either form), and nothing of the hidden ones
@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("heads,n", [(4, 100), (60, 300), (160, 130), (512, 200), (300, 700)])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_sdp_attention_alpha_zero(ops, heads, n, d, dtype):
    import torch
    q, k, v = (dev(synth.normal(s, (1, 4, n, d)).astype(np.float16 if dtype == "f16" else np.float32)).repeat(1, heads // 4, 1, 1) for s in (1, 2, 3))
    got = host(ops.sdp_attention_fwd(q, k, v, 0.0, causal=True, window=90)).astype(np.float64)
    sums = np.cumsum(np.concatenate([np.zeros((4, 1, d)), host(v[0, :4]).astype(np.float64)], axis=1), axis=1)
    at = np.arange(1, n + 1)
    lo = np.maximum(at - 90, 0)
    want = (sums[:, at] - sums[:, lo]) / (at - lo)[None, :, None]
    assert scaled_rel_err(got[0, :4], want, 1.0) <= (2.0 ** -10 if dtype == "f16" else TOL_F32)
    assert np.array_equal(got[0].reshape(-1, 4, n, d), np.broadcast_to(got[:, :4], (heads // 4, 4, n, d)))


# a mask tensor with softcap (logits capped before the mask is added) and grouped heads, which only the C entry points take: 16 rows per block with eight waves and with four, 128 queries per block
@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("heads,q_per_kv,n_q,n_k", [(4, 2, 40, 257), (6, 3, 17, 130), (160, 4, 40, 300), (8, 8, 100, 90), (200, 2, 100, 200)])
@pytest.mark.parametrize("d,cap,alpha", [(64, 30.0, 0.3), (128, 0.0, 0.0884), (128, 50.0, 0.2), (256, 30.0, 0.2), (256, 0.0, 0.0625)])
def test_sdp_attention_mask_tensor_softcap_and_grouped_heads(ops, heads, q_per_kv, n_q, n_k, d, cap, alpha, dtype):
    import torch
    from anygpu_amd import capi
    from test_gpu_attention_f32_parts import attend64
    ndt = np.float16 if dtype == "f16" else np.float32
    q, k, v = (synth.normal(s + n, (h, n, d)).astype(ndt) for s, h, n in ((1, heads, n_q), (2, heads // q_per_kv, n_k), (3, heads // q_per_kv, n_k)))
    mask = synth.normal(7, (n_q, n_k), std=2.0).astype(ndt)
    mask[synth.normal(8, (n_q, n_k)) > 0.5] = -np.inf
    mask[:, 64:96] = -np.inf
    mask[n_q // 2] = -np.inf                                     # sees nothing: zeros
    dq, dk, dv, dm = (dev(t) for t in (q, k, v, mask))
    y = torch.full_like(dq, 9.0)
    fn = getattr(capi.load(), f"anygpu_sdp_attention_fwd_masked_{dtype}")
    assert fn(dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), dm.data_ptr(), y.data_ptr(), heads, q_per_kv, n_q, n_k, d, n_k, alpha, cap, None) == capi.ANYGPU_OK
    got, bias = host(y).astype(np.float64), mask.astype(np.float64)
    some = sorted({0, 1, heads // 2, heads - 1})
    want = np.stack([attend64(q[h:h + 1], k[h // q_per_kv:h // q_per_kv + 1], v[h // q_per_kv:h // q_per_kv + 1], alpha, cap, bias=bias)[0] for h in some])
    assert not got[:, n_q // 2].any() and np.isfinite(got).all()
    # (float32: logits of up to about 20 carry the hardware exponential's 2^-22 of themselves into the weights)
    assert scaled_rel_err(got[some], want, 1.0) <= (TOL_F16_ROWOPS * 2 if dtype == "f16" else TOL_F32)


# what a mask tensor hides from all queries of a wave (whole tiles of 64 keys) takes no part in their results, whatever it holds: the tail of a padded cache,
# a stretch within, and one that the first sixteen queries see and the others do not; 16 rows per block with eight waves (3 heads) and four (100),
# 128 queries per block (700)
@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("heads", [3, 100, 700])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_sdp_attention_mask_tensor_hidden_tiles_hold_anything(ops, heads, d, dtype):
    ndt = np.float16 if dtype == "f16" else np.float32
    n_q, n_k = 40, 300
    q, k, v = (synth.normal(s + n, (1, heads, n, d)).astype(ndt) for s, n in ((1, n_q), (2, n_k), (3, n_k)))
    mask = synth.normal(7, (n_q, n_k)).astype(ndt)
    mask[:, 128:192] = -np.inf
    mask[:, 256:] = -np.inf
    mask[16:, 64:128] = np.finfo(ndt).min if dtype == "f32" else -np.inf
    run = lambda kk, vv: host(ops.sdp_attention_masked_scaled_fwd(dev(q), dev(kk), dev(vv), dev(mask).reshape(1, 1, n_q, n_k), d ** -0.5))
    clean = run(k, v)
    assert np.isfinite(clean).all()
    for value in (np.nan, np.inf):
        kk, vv = k.copy(), v.copy()
        kk[:, :, 128:192] = vv[:, :, 128:192] = value
        kk[:, :, 257::3] = vv[:, :, 256:] = value
        assert np.array_equal(run(kk, vv), clean)
        kk[:, :, 70] = vv[:, :, 64:128] = value
        got = run(kk, vv)
        assert np.array_equal(got[:, :, 16:], clean[:, :, 16:]) and not np.isfinite(got[:, :, :16]).any()


# keys and values that end inside a tile (one key over whole tiles of 32 and 16, one short, in between), with NaN in memory in front of the first and behind the last
# of them, and in place of the head in the middle: no result takes any of it
@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("n_k", [33, 129, 143, 257, 273, 287])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_sdp_attention_few_rows_nothing_behind_the_last_key(ops, n_k, d, dtype):
    import torch
    ndt, tdt = (np.float16, torch.float16) if dtype == "f16" else (np.float32, torch.float32)
    for n_q in (40, 1):
        q, k, v = (dev(synth.normal(s + n, (1, 3, n, d)).astype(ndt)) for s, n in ((1, n_q), (2, n_k), (3, n_k)))
        mask = dev(synth.normal(7, (1, 1, n_q, n_k)).astype(ndt))

        def among_nan(t):
            pool = torch.full((3 * n_k + 128, d), math.nan, dtype=tdt, device="cuda")
            view = pool[64:64 + 3 * n_k].view(1, 3, n_k, d)
            view.copy_(t)
            view[:, 1] = math.nan
            return view
        for run in (lambda kk, vv: ops.sdp_attention_fwd(q, kk, vv, d ** -0.5), lambda kk, vv: ops.sdp_attention_fwd(q, kk, vv, d ** -0.5, causal=True, window=50),
                    lambda kk, vv: ops.sdp_attention_fwd(q, kk, vv, d ** -0.5, decode=False), lambda kk, vv: ops.sdp_attention_masked_scaled_fwd(q, kk, vv, mask, d ** -0.5)):
            clean, got = host(run(k, v)), host(run(among_nan(k), among_nan(v)))
            assert np.isfinite(clean).all() and np.array_equal(got[:, ::2], clean[:, ::2])


# the note of a mask's hidden tiles (always / never) in launches of so many heads that blocks of 128 queries (float32 at 64 and 128: 64) take them: masks below the
# sizes that get one by default, ragged last tiles and blocks, queries that see nothing, mask rows at an odd pitch; and the launches of few query blocks, which have none while
# the variable is not set
@pytest.mark.parametrize("dtype,d,heads,n_q,n_k,kind", [("f16", 64, 70, 300, 333, "slide"), ("f16", 64, 140, 130, 1500, "stripes"), ("f16", 128, 48, 300, 300, "blind rows"), ("f16", 128, 96, 130, 700, "odd stride"),
                                                        ("f16", 256, 26, 300, 301, "slide"), ("f16", 256, 30, 130, 1030, "stripes"), ("f32", 64, 120, 300, 333, "slide"), ("f32", 64, 64, 200, 2100, "stripes"),
                                                        ("f32", 128, 80, 300, 300, "blind rows"), ("f32", 128, 40, 200, 1500, "odd stride"), ("f32", 256, 24, 300, 301, "slide"), ("f32", 256, 4, 150, 1100, "stripes")])
def test_sdp_attention_mask_tensor_with_and_without_note(ops, oracle, monkeypatch, dtype, d, heads, n_q, n_k, kind):
    import torch
    from anygpu_amd import capi
    half, alpha = dtype == "f16", d ** -0.5
    q, k, v = (synth.normal(s + n, (heads, n, d)).astype(np.float16 if half else np.float32) for s, n in ((1, n_q), (2, n_k), (3, n_k)))
    if kind == "slide":
        mask = oracle.slide_mask(oracle.causal_mask(n_q, n_k, diag=n_k - n_q), n_k // 3)
    else:
        rng = np.random.default_rng(n_q * 1000 + n_k)
        mask = rng.normal(0.0, 2.0, (n_q, n_k)).astype(np.float32)
        hide_key_stripes(mask, rng)
        if kind == "blind rows":
            mask[[5, n_q // 2]] = -np.inf
    with np.errstate(over="ignore"):
        mask = np.ascontiguousarray(mask).astype(q.dtype)
    pitch = n_k + (3 if kind == "odd stride" else 0)
    rows = torch.full((n_q * pitch + 1,), float("nan"), dtype=torch.float16 if half else torch.float32, device="cuda")[1:].view(n_q, pitch)
    rows[:, :n_k] = dev(mask)
    fn = getattr(capi.load(), f"anygpu_sdp_attention_fwd_masked_{dtype}")

    def run(count, env):
        if env is None:
            monkeypatch.delenv("ANYGPU_ATTN_MASK_MAP_FROM", raising=False)
        else:
            monkeypatch.setenv("ANYGPU_ATTN_MASK_MAP_FROM", env)
        args = [dev(t[:count]) for t in (q, k, v)]
        y = torch.empty_like(args[0])
        assert fn(*(t.data_ptr() for t in args), rows.data_ptr(), y.data_ptr(), count, 1, n_q, n_k, d, pitch, alpha, 0.0, None) == capi.ANYGPU_OK
        return host(y).astype(np.float32)
    tol = TOL_F16_ROWOPS * 2 if half else TOL_F32
    always, never = run(heads, "0"), run(heads, str(1 << 60))
    assert scaled_rel_err(always, never, 1.0) <= (TOL_F16_ROWOPS if half else 1e-5)
    some = [0, heads // 2, heads - 1]
    wide = [(oracle.cvt_f16_to_f32(t) if half else t) for t in (q[some], k[some], v[some], mask)]
    seen = np.isfinite(wide[3]).any(axis=-1)
    with np.errstate(invalid="ignore", over="ignore"):
        want = oracle.sdp_attention_masked_scaled_fwd(*(t[None] for t in wide[:3]), wide[3].reshape(1, 1, n_q, n_k), alpha, threads=8)[0]
    for got in (always[some], never[some]):
        assert not got[:, ~seen].any() and np.isfinite(got).all()
        assert scaled_rel_err(got[:, seen], want[:, seen], 1.0) <= tol
    if n_k < 500:
        few = [run(2, env) for env in (None, "0", str(1 << 60))]
        assert scaled_rel_err(few[1], few[2], 1.0) <= (TOL_F16_ROWOPS if half else 1e-5) and not np.array_equal(few[0], few[1])
        for got in few:
            assert not got[:, ~seen].any() and scaled_rel_err(got[0][seen], want[0][seen], 1.0) <= tol


# The next tests reach the kernel with 32 queries per wave by more than one query block per CU (512 heads), or by few blocks with so
# many key tiles that each goes out in parts.  Scores are set by the first component of q and k alone.

def _scores_operands(heads, n_q, k0, d, q0=None):
    import torch
    q = torch.zeros((1, heads, n_q, d), dtype=torch.half, device="cuda")
    q[..., 0] = 1.0 if q0 is None else dev(q0.astype(np.float16))
    k = torch.zeros((1, 1, len(k0), d), dtype=torch.half, device="cuda")
    k[0, 0, :, 0] = dev(k0.astype(np.float16))
    return q, k


def _softmax_product(scores, v):
    w = np.exp(scores - scores.max(axis=-1, keepdims=True))
    return (w @ v) / w.sum(axis=-1, keepdims=True)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("first", [True, False])
def test_sdp_attention_32_queries_per_wave_small_weights_keep_their_bits(ops, d, first):
    # one key with the largest score among keys whose weights are 2^-15 ... 2^-24 of it: as halves below 1 these would be denormal.
    # The small weights come into the result rounded to 11 bits each (2^-11), as does the result (2^-11)
    import torch
    for n, b in ((1000, 17), (4096, 15), (4096, 17), (4096, 20), (4096, 24)):
        k0 = np.full((n,), -b * math.log(2.0))
        at = 0 if first else n - 1
        k0[at] = 0.0
        q, k = _scores_operands(512, 40, k0, d)
        v = torch.ones((1, 1, n, d), dtype=torch.half, device="cuda")
        v[:, :, at] = 0.0
        small = (n - 1) * math.exp(float(np.float16(k0[n // 2])))
        got = host(ops.sdp_attention_fwd(q, k, v, 1.0)).astype(np.float64)
        assert np.abs(got / (small / (1.0 + small)) - 1.0).max() <= 2.0 ** -10 + 1e-5
    # and into the sum in 32 bits: 65535 of 2^-23.6 each, which halves would round by a quarter
    n, b = 65536, 23.6
    k0 = np.full((n,), -b * math.log(2.0))
    k0[0 if first else n - 1] = 0.0
    q, k = _scores_operands(512, 40, k0, d)
    v = torch.zeros((1, 1, n, d), dtype=torch.half, device="cuda")
    v[:, :, 0 if first else n - 1] = 1.0
    small = (n - 1) * math.exp(float(np.float16(k0[n // 2])))
    got = host(ops.sdp_attention_fwd(q, k, v, 1.0)).astype(np.float64)
    assert np.abs(got * (1.0 + small) - 1.0).max() <= 2.0 ** -11 + 1e-5


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("step", [0.3, 7.9, 8.1, 15.0, -8.1])
def test_sdp_attention_32_queries_per_wave_moving_maximum(ops, d, step):
    # the largest score of a tile of 64 keys is 2^step times that of the tile before, for one query of each wave; the other queries see
    # the steps a hundredth as high.  Whole blocks (512 heads), and 32 heads x 40 queries over 20000 keys in parts, where
    # the steps come round every seven tiles.  Weights and result rounded to 11 bits, |v| <= 1
    rng = np.random.default_rng(5)
    q0 = np.where(np.arange(40) % 32 == 5, 1.0, 0.01)
    for heads, n in ((512, 7 * 64 - 3), (32, 20000)):
        k0 = ((np.arange(n) // 64) % 7 * step + rng.uniform(-1.0, 0.0, n)) * math.log(2.0)
        q, k = _scores_operands(heads, 40, k0, d, q0)
        v = rng.uniform(-1.0, 1.0, (n, d)).astype(np.float16)
        got = host(ops.sdp_attention_fwd(q, k, dev(v).reshape(1, 1, n, d), 1.0, decode=False)).astype(np.float64)
        want = _softmax_product(np.float16(q0).astype(np.float64)[:, None] * np.float16(k0).astype(np.float64)[None, :], v.astype(np.float64))
        assert np.abs(got[0] - want).max() <= 2.0 ** -10


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("alpha", [1.0, -1.0])
@pytest.mark.parametrize("heads", [4, 120, 512])
def test_sdp_attention_scores_beyond_the_mantissa(ops, d, alpha, heads):
    # scores of 10^9 and more, whose rounding as a float is larger than the halves' range of exponents: still the row of the key
    # with the largest score, bit for bit (16 rows per block with few heads, 16 queries per wave with 120, 32 with 512)
    import torch
    n = 300
    order = np.random.default_rng(6).permutation(n)
    q = torch.full((1, heads, 130, d), 10000.0, dtype=torch.half, device="cuda")
    k = dev((alpha * (10000.0 - 16.0 * order))[:, None].repeat(d, axis=1).astype(np.float16)).reshape(1, 1, n, d)
    v = synth.normal(9, (1, 1, n, d)).astype(np.float16)
    got = host(ops.sdp_attention_fwd(q, k, dev(v), alpha))
    assert np.array_equal(got, np.broadcast_to(v[0, 0, int(np.argmin(order))], got.shape))


@pytest.mark.parametrize("n", [200, 900])                        # a tile's products and softmax in turn, and overlapped
@pytest.mark.parametrize("d", [64, 128])
def test_sdp_attention_32_queries_per_wave_nan_and_infinities(ops, d, n):
    # a NaN in a query reaches its row; a NaN in a key, or a score of +inf, the rows that see the key; a score of -inf hides it
    import torch
    copies, heads = 64, 8
    q, k, v = (synth.normal(70 + i, (heads, n, d)).astype(np.float16) for i in range(3))
    q[1, 37, 3] = np.nan
    k[2, 150, 0] = np.nan
    k[3, 100, 5] = np.inf
    q[4, 11, 7] = -np.inf
    alpha = d ** -0.5
    got = host(ops.sdp_attention_fwd(*(dev(t).reshape(1, heads, n, d).repeat(copies, 1, 1, 1) for t in (q, k, v)), alpha, causal=True))
    assert np.array_equal(got, np.broadcast_to(got[:1], got.shape), equal_nan=True)
    s = torch.from_numpy(q).double() @ torch.from_numpy(k).double().transpose(1, 2).contiguous() * alpha
    s = s.masked_fill(torch.ones(n, n, dtype=torch.bool).triu(1), -math.inf)
    want = (torch.softmax(s, -1) @ torch.from_numpy(v).double()).numpy()
    assert np.array_equal(np.isnan(got[0]), np.isnan(want))
    assert 0 < np.isnan(want).any(-1).sum() < heads * n // 2
    seen = ~np.isnan(want)
    assert scaled_rel_err(got[0].astype(np.float64)[seen], want[seen], 1.0) <= TOL_F16_ROWOPS * 2


# head dimensions 64 and 128 with 32 queries per wave: the longest blocks in two halves of their key range (causal, 320 blocks; window, 288
# blocks; long ranges, 448 blocks) and all blocks in parts of a long range (32 blocks x 313 tiles), and 256 blocks with 16 queries per
# wave in halves: against whole blocks, which a workspace without room gives, and the oracle
@pytest.mark.parametrize("heads,kv_heads,n_q,n_k,d,causal,window", [(10, 5, 4086, 4086, 128, True, 0), (9, 3, 4086, 4086, 64, True, 1024),
                                                                     (7, 7, 8182, 8182, 64, True, 0), (16, 2, 200, 20000, 64, True, 0),
                                                                     (32, 4, 70, 20000, 128, True, 0), (8, 8, 4086, 4086, 64, True, 0)])
def test_sdp_attention_key_parts_agree_with_whole_blocks(ops, oracle, heads, kv_heads, n_q, n_k, d, causal, window):
    import torch
    q = synth.normal(31, (heads, n_q, d)).astype(np.float16)
    k = synth.normal(32, (kv_heads, n_k, d)).astype(np.float16) * np.float16(2.0)
    v = synth.normal(33, (kv_heads, n_k, d)).astype(np.float16)
    alpha = d ** -0.5
    run = lambda: host(ops.sdp_attention_fwd(dev(q), dev(k), dev(v), alpha, causal=causal, window=window, decode=False)).astype(np.float32)
    parts = run()
    tiny = torch.empty((64,), device="cuda")
    ops.set_workspace(tiny)
    try:
        whole = run()
    finally:
        torch.cuda.synchronize()
        ops.set_workspace(None)
    assert not np.array_equal(parts, whole), "the launch was expected to take parts of the key range"
    idx = np.array(sorted({0, 31, 63, n_q // 2, n_q - 130, n_q - 70, n_q - 1} & set(range(n_q))), dtype=np.int64)
    want = oracle.sdp_attention_rules(*(oracle.cvt_f16_to_f32(t) for t in (q, k, v)), alpha=alpha, softcap=0.0, causal=causal, window=window,
                                      q_per_kv=heads // kv_heads, query_index=idx, threads=8)
    for got in (parts, whole):
        assert np.isfinite(got).all()
        assert scaled_rel_err(got[:, idx, :], want, 1.0) <= TOL_F16_ROWOPS * 2
    assert scaled_rel_err(parts, whole, 1.0) <= 2e-3


def test_sdp_attention_decode_takes_the_least_workspace(ops):
    # 32 key / value heads x 5001 keys: 32 splits of 160 keys by the query, 27 of 192 in the least workspace (fp16), which stays
    # enough.  Where the library's scratch of 8 MB holds the 27 splits only (8 rows x 256: 7.1 MB against 8.5), the query is theirs too,
    # and with 28 heads and a window of 4096 the finer cut has the fewer splits.  The scratch always gives the bits of a workspace
    # of the queried size.
    import torch
    from anygpu_amd import capi
    lib = capi.load()
    for kv, per, d, n_k, window, query, coarse in ((32, 4, 128, 5001, 0, 32, 27), (32, 8, 256, 5001, 0, 27, 27), (28, 2, 256, 4128, 4096, 32, 33)):
        rng = torch.Generator(device="cuda")
        rng.manual_seed(7)
        q = torch.randn((kv * per, 1, d), device="cuda", generator=rng).half()
        k, v = (torch.randn((kv, n_k, d), device="cuda", generator=rng).half() for _ in range(2))
        shape = (kv * per, per, 1, n_k, d)
        need, least = (kv * splits * per * (d + 2) * 4 for splits in (query, min(query, coarse)))
        assert lib.anygpu_sdp_attention_decode_workspace_bytes(*shape, 1, window) == need
        rest = (*shape, d ** -0.5, 0.0, 1, window, torch.cuda.current_stream().cuda_stream)
        ptrs = (q.data_ptr(), k.data_ptr(), v.data_ptr())
        outs = []
        for size in (need, need + 4096, least):
            ws = torch.empty(size, dtype=torch.uint8, device="cuda")
            outs.append(torch.empty_like(q))
            assert lib.anygpu_sdp_attention_decode_f16(*ptrs, outs[-1].data_ptr(), ws.data_ptr(), size, *rest) == 0
        assert lib.anygpu_sdp_attention_decode_f16(*ptrs, outs[-1].data_ptr(), ws.data_ptr(), least - 1, *rest) == capi.ANYGPU_ERR_BAD_SHAPE
        outs.append(torch.empty_like(q))
        assert lib.anygpu_sdp_attention_decode_f16_static(*ptrs, outs[-1].data_ptr(), *rest) == 0
        assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[3])
        seen = slice(n_k - window, n_k) if window else slice(0, n_k)
        s = (q.float().view(kv, per, d) @ k.float()[:, seen].transpose(1, 2).contiguous()) * d ** -0.5
        want = host((torch.softmax(s, -1) @ v.float()[:, seen]).view(kv * per, 1, d))
        for out in outs:
            assert scaled_rel_err(host(out), want, float(np.abs(want).mean())) <= TOL_F16_GEMM


def test_sdp_attention_decode_under_a_window_of_whole_tiles(ops, oracle):
    # batch 7, 8 / 4 heads, window 4096, 4128 keys: the queried workspace is below that of the cut in tiles of 64
    q, k, v = (synth.normal(60 + i, (7, h, n, 256)).astype(np.float16) for i, (h, n) in enumerate(((8, 1), (4, 4128), (4, 4128))))
    got = host(ops.sdp_attention_fwd(dev(q), dev(k), dev(v), 0.0625, softcap=50.0, causal=True, window=4096)).astype(np.float32)
    for b in (0, 6):
        want = oracle.sdp_attention_rules(*(oracle.cvt_f16_to_f32(np.ascontiguousarray(t[b])) for t in (q, k, v)), alpha=0.0625, softcap=50.0,
                                          causal=True, window=4096, q_per_kv=2, threads=8)
        assert scaled_rel_err(got[b], want, 1.0) <= TOL_F16_ROWOPS * 2


@pytest.mark.parametrize("m,n,k", [(130, 72, 64), (200, 1000, 128), (300, 2056, 192), (256, 2048, 320), (2000, 4072, 320), (2048, 4096, 320),
                                   (4090, 4072, 320), (4096, 4096, 320)])
def test_upproj_and_bias_f16_row_major_weights_in_whole_slabs(ops, m, n, k):
    # [K, N] weights, K in whole slabs of 64: one and two matrices in 128 x 128, 256 x 128 and 256 x 256 tiles, whole and ending past M and N.
    # Small integers times a power of two: the sums are exact; bounds as in test_mm_few_rows_k_cut_over_waves
    a, w1, w2 = (synth.integers(s, shape, -2, 2).astype(np.float16) for s, shape in ((m, (m, k)), (n + 2, (k, n)), (n + 3, (k, n))))
    bias = synth.integers(3, (n,), -9, 9).astype(np.float16)
    s1 = exact_int_product(a, w1)
    assert np.array_equal(host(ops.tensor_gemm(dev(a), dev(w1), dev(bias))).astype(np.int64), s1 + bias.astype(np.int64))
    scale = 2.0 ** -6
    s1, s2 = s1 * scale, exact_int_product(a, w2) * scale
    got = host(ops.mlp_gemma2_fused_upproj(dev((a * scale).astype(np.float16)), dev(w1), dev(w2))).astype(np.float64)
    gated = 0.5 * s1 * (1.0 + np.tanh(math.sqrt(2.0 / math.pi) * (s1 + 0.044715 * s1 ** 3))) * s2
    # (the half epilogue's tanh: 4.4e-5 of the gate's factor)
    assert np.all(np.abs(got - gated) <= 2.0 ** -11 * np.abs(gated) + 5e-5 * np.abs(s1 * s2) + 2.0 ** -24)


@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("rows,cols,pad,off,window", [(64, 1, 0, 0, 0), (70, 7, 0, 3, 0), (65, 8, 1, 5, 0), (64, 63, 2, 1, 0), (80, 505, 0, 7, 100), (64, 512, 3, 2, 0),
                                                      (3, 65, 0, 1, 0), (5, 449, 5, 63, 0), (9, 1473, 0, 0, 1000), (7, 1537, 1, 33, 0), (5, 3009, 0, 9, 2049),
                                                      (6, 3073, 3, 62, 0), (9, 4097, 0, 1, 4096), (4, 8129, 0, 31, 0), (3, 16321, 7, 2, 0), (300, 16385, 0, 0, 4096),
                                                      (260, 32705, 1, 3, 0)])
def test_softmax_rows_of_any_width_and_start(ops, oracle, dtype, rows, cols, pad, off, window):
    # rows that start at any element and share their first and last 16 bytes with other rows: what lies between the rows (NaN here) reaches
    # no result, and nothing is stored there; x and y start at different places of the same 16 bytes, lines apart
    import torch
    np_dt, t_dt = (np.float16, torch.float16) if dtype == "f16" else (np.float32, torch.float32)
    epv, pitch = 16 // np.dtype(np_dt).itemsize, cols + pad
    x = synth.normal(cols + rows, (rows, cols), std=8.0).astype(np_dt)
    xbuf, ybuf = torch.full((off + rows * pitch + 64,), math.nan, dtype=t_dt, device="cuda"), torch.full((off + 3 * epv + rows * pitch + 64,), -7.0, dtype=t_dt, device="cuda")
    xv, yv = torch.as_strided(xbuf, (rows, cols), (pitch, 1), off), torch.as_strided(ybuf, (rows, cols), (pitch, 1), off + 3 * epv)
    xv.copy_(dev(x))
    kw = dict(alpha=0.5, softcap=20.0 if off % 2 else 0.0, causal=window > 0, window=window, q_len=rows, diag=cols - rows)
    ops.tensor_softmax(xv, out=yv, **kw)
    got = host(yv).astype(np.float64)
    want = oracle.attention_softmax(oracle.cvt_f16_to_f32(x) if dtype == "f16" else x, **kw).reshape(rows, cols).astype(np.float64)
    tol = TOL_F16_ROWOPS if dtype == "f16" else TOL_F32
    assert np.max(np.abs(got - want) / (want + want.max(axis=1, keepdims=True))) <= tol
    assert np.all(got[want == 0] == 0)
    yv.fill_(-7.0)
    assert bool((ybuf == -7.0).all())


@pytest.mark.parametrize("dtype,rows,cols,off", [("f16", 256, 32712, 0), ("f16", 300, 32760, 0), ("f32", 256, 16356, 0), ("f32", 300, 16380, 0), ("f16", 256, 32768, 8), ("f32", 256, 16384, 4)])
@pytest.mark.parametrize("window", [0, 16000])
def test_softmax_aligned_rows_that_just_fill_a_block(ops, oracle, dtype, rows, cols, off, window):
    # 4089 to 4096 vectors of 16 bytes in rows that start inside a line: more than the block of 512 threads counts, as many as 256 hold
    import torch
    np_dt, t_dt = (np.float16, torch.float16) if dtype == "f16" else (np.float32, torch.float32)
    x = synth.normal(cols + rows, (rows, cols), std=8.0).astype(np_dt)
    xbuf, ybuf = (torch.full((off + rows * cols + 64,), -7.0, dtype=t_dt, device="cuda") for _ in range(2))
    xv, yv = (torch.as_strided(buf, (rows, cols), (cols, 1), off) for buf in (xbuf, ybuf))
    xv.copy_(dev(x))
    kw = dict(alpha=0.5, softcap=20.0, causal=window > 0, window=window, q_len=rows, diag=cols - rows)
    ops.tensor_softmax(xv, out=yv, **kw)
    got = host(yv).astype(np.float64)
    want = oracle.attention_softmax(oracle.cvt_f16_to_f32(x) if dtype == "f16" else x, **kw).reshape(rows, cols).astype(np.float64)
    tol = TOL_F16_ROWOPS if dtype == "f16" else TOL_F32
    assert np.max(np.abs(got - want) / (want + want.max(axis=1, keepdims=True))) <= tol
    assert np.all(got[want == 0] == 0)
    yv.fill_(-7.0)
    assert bool((ybuf == -7.0).all())


@pytest.mark.parametrize("softcap", [50.0, 64.0, 65.0, 1e5, -1e5])
@pytest.mark.parametrize("cols", [500, 1001, 12000])
def test_softmax_f16_softcap_of_any_size(ops, softcap, cols):
    # the logit keeps its precision however far the cap lies beyond the scores.  One rounding to half (2^-11, 2^-25 below the smallest normal half), the logit to
    # 1.5e-7 of a cap of up to 64 or of a score of up to 32, some roundings of the fp32 sum and of exp2 (1e-6 each)
    x = synth.normal(cols, (64, cols), std=4.0).astype(np.float16)
    got = host(ops.tensor_softmax(dev(x), softcap=softcap)).astype(np.float64)
    z = softcap * np.tanh(x.astype(np.float64) / softcap)
    want = np.exp(z - z.max(axis=1, keepdims=True))
    want /= want.sum(axis=1, keepdims=True)
    assert np.all(np.abs(got - want) <= (2.0 ** -11 + 1.5e-5) * want + 2.0 ** -25)


@pytest.mark.parametrize("layout", ["kn", "nk"])
@pytest.mark.parametrize("m,n,k,shift", [(3, 1, 1, 0), (1, 333, 211, 1), (5, 33, 31, 0), (32, 32, 32, 1), (33, 31, 33, 0), (64, 65, 127, 1), (31, 97, 129, 3),
                                         (100, 40, 160, 1), (70, 130, 161, 2), (45, 300, 543, 0), (200, 129, 1000, 1), (17, 50, 1502, 2), (2, 1001, 700, 0)])
def test_mm_f16_small_products_as_they_lie(ops, m, n, k, layout, shift):
    # 32 x 32 tiles and steps of 32 of K from before to behind their ends, none to a dozen steps per wave; operands `shift` halves into wider buffers of
    # NaN, so that rows start at odd halves and at words that are no multiple of 16 bytes, the result likewise.  Small integers: exact.
    import torch
    from anygpu_amd import capi
    lay = capi.B_ROW_MAJOR if layout == "kn" else capi.B_COL_MAJOR
    a, b = (synth.integers(s + m, shape, -2, 2).astype(np.float16) for s, shape in ((1, (m, k)), (2, (k, n))))
    want = exact_int_product(a, b)
    assert np.max(np.abs(want)) < 2000
    w = b if layout == "kn" else np.ascontiguousarray(b.T)

    def inside(x):
        buf = torch.full((x.shape[0], x.shape[1] + 5), math.nan, dtype=torch.float16, device="cuda")
        view = buf[:, shift:shift + x.shape[1]]
        view.copy_(dev(x))
        return view
    av, wv = inside(a), inside(w)
    out = torch.full((m + 1, n + 4), -7.0, dtype=torch.float16, device="cuda")
    ops.tensor_mm(av, wv, out=out[:m, shift:shift + n], b_layout=lay)
    got = host(out).astype(np.int64)
    assert np.array_equal(got[:m, shift:shift + n], want)
    assert np.all(got[m:] == -7) and np.all(got[:, :shift] == -7) and np.all(got[:, shift + n:] == -7)
    bias = synth.integers(3, (n,), -9, 9).astype(np.float16)
    assert np.array_equal(host(ops.tensor_gemm(dev(a), dev(w), dev(bias), b_layout=lay)).astype(np.int64), want + bias.astype(np.int64))
    if layout == "nk":
        # half an ulp of the result, 4.4e-5 of it for the fp16 tanh
        scale = 2.0 ** -6
        got = host(ops.tensor_gemma_linear_softcap(dev((a * scale).astype(np.float16)).reshape(1, m, k), dev(w), 30.0)).astype(np.float64).reshape(m, n)
        capped = 30.0 * np.tanh(want * scale / 30.0)
        assert np.all(np.abs(got - capped) <= (2.0 ** -11 + 4.4e-5) * np.abs(capped) + 30.0 * 1e-6)
    # a NaN or an infinity reaches its row or column and no other
    av[0, k - 1], wv[(k // 2, n - 1) if layout == "kn" else (n - 1, k // 2)] = math.nan, math.inf
    got = host(ops.tensor_mm(av, wv, b_layout=lay)).astype(np.float64)
    assert np.all(np.isnan(got[0])) and not np.isfinite(got[1:, n - 1]).any()
    assert np.array_equal(got[1:, :n - 1], want[1:, :n - 1])


# convolution over rows of any length as one run of vectors (256 vectors and more, off their boundaries or in tiles mostly empty): every remainder of
# a row's end in a vector, rows that end with a block and one sample on, a single row, a last vector that is not whole; what
# the row before holds (here NaN and infinities at its end) never reaches a row
@pytest.mark.parametrize("dtype,b,d,s,width", [("f16", 1, 1, 2049, 4), ("f16", 3, 5, 2055, 4), ("f16", 2, 3, 4093, 3), ("f16", 1, 3, 4095, 4), ("f16", 2, 2, 4097, 2), ("f16", 3, 3, 4099, 1),
                                               ("f16", 2, 7, 2042, 4), ("f16", 1, 5, 4168, 4), ("f16", 2, 3, 8190, 4), ("f32", 1, 1, 1021, 4), ("f32", 3, 5, 1026, 4),
                                               ("f32", 2, 3, 2047, 3), ("f32", 2, 7, 2049, 2), ("f32", 1, 3, 2108, 4), ("f32", 2, 2, 1023, 1)])
def test_conv1d_rows_as_one_run_of_vectors(ops, oracle, dtype, b, d, s, width):
    ndt = np.float16 if dtype == "f16" else np.float32
    x = synth.normal(s, (b, d, s)).astype(ndt)
    w, bias = synth.normal(1, (d, width), std=0.5).astype(ndt), synth.normal(2, (d,), std=0.1).astype(ndt)
    wide = [oracle.cvt_f16_to_f32(t) if dtype == "f16" else t for t in (x, w, bias)]
    want = oracle.tensor_causal_conv1d(*wide, threads=4)
    got = host(ops.tensor_causal_conv1d(dev(x), dev(w), dev(bias))).astype(np.float32)
    assert scaled_rel_err(got, want, 1.0) <= (TOL_F16_ROWOPS if dtype == "f16" else TOL_F32)
    x[0, 0, -3:] = np.array([np.nan, np.inf, np.nan])
    again = host(ops.tensor_causal_conv1d(dev(x), dev(w), dev(bias))).astype(np.float32)
    rows = again.reshape(b * d, s)
    assert np.array_equal(rows[1:], got.reshape(b * d, s)[1:]) and np.array_equal(rows[0, :-3], got[0, 0, :-3]) and np.isnan(rows[0, -3:]).any()


# one channel, where every row has the same taps: batches of two to sixteen rows, whose row number is no channel's, off the vectors' boundaries and with a nearly empty
# last tile, taps and bias as slices of buffers that hold NaN everywhere else
@pytest.mark.parametrize("dtype,b,s,width", [("f16", 2, 2049, 4), ("f16", 3, 4095, 2), ("f16", 4, 2049, 4), ("f16", 9, 4259, 3), ("f16", 16, 4168, 4), ("f16", 4, 4168, 1),
                                             ("f32", 2, 1025, 4), ("f32", 4, 1025, 4), ("f32", 9, 2049, 2), ("f32", 16, 2108, 4)])
def test_conv1d_rows_as_one_run_of_vectors_one_channel(ops, oracle, dtype, b, s, width):
    import torch
    ndt = np.float16 if dtype == "f16" else np.float32
    x = synth.normal(s, (b, 1, s)).astype(ndt)
    w, bias = synth.normal(1, (1, width), std=0.5).astype(ndt), synth.normal(2, (1,), std=0.1).astype(ndt)
    wide = [oracle.cvt_f16_to_f32(t) if dtype == "f16" else t for t in (x, w, bias)]
    want = oracle.tensor_causal_conv1d(*wide, threads=4)
    pool = torch.full((256,), math.nan, dtype=torch.float16 if dtype == "f16" else torch.float32, device="cuda")
    pool[64:64 + width], pool[160] = dev(w[0]), float(bias[0])
    got = host(ops.tensor_causal_conv1d(dev(x), pool[64:64 + width].view(1, width), pool[160:161])).astype(np.float32)
    assert scaled_rel_err(got, want, 1.0) <= (TOL_F16_ROWOPS if dtype == "f16" else TOL_F32)
