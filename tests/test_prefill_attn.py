"""GPU parity: prefill flash attention over a Q8_0 cache vs the f64 oracle.

Template: crates/sg-gpu/tests/parity_attn.rs (prefill cases, q0 in {0, 200},
causal and sliding, oracle attention_head with t0 = 0 or the window start,
parity_attn.rs:688-784) and BASELINE config 4 (4096 queries, 32 q / 16 kv
heads, hd 128, causal and sliding-1024).  The oracle attends the exactly
dequantized K/V in f64; the kernel rounds K, V, q and P to f16 (as the
reference's f16 PV path does: 2^-12 relative each), which leaves up to ~1e-3
absolute on queries that see only a few keys of magnitude ~2.  The bar is
1e-3 relative to the output scale: normwise max|err|/max|want| <= 1e-3, and
elementwise |err| <= 2e-3*|want| + 1e-3*max|want| (the reference's own
prefill tolerance was 1e-2).
"""
import numpy as np
import pytest
import torch

from _util import assert_close, dev, empty, host, rel_err

pytestmark = pytest.mark.gpu

HD = 128


def _case(oracle, seed, n_slots, n_kv, n_tok, n_q, qscale=1.0):
    rng = oracle.Rng(seed)
    k = rng.f32_vec(n_slots * n_kv * HD)
    v = rng.f32_vec(n_slots * n_kv * HD)
    ks, kq = oracle.quant_q8_0(k)
    vs, vq = oracle.quant_q8_0(v)
    q = rng.f32_vec(n_tok * n_q * HD) * np.float32(qscale)
    return q, kq, ks, vq, vs, oracle.dequant_q8_0(ks, kq), oracle.dequant_q8_0(vs, vq)


def _run(ctx, q, kq, ks, vq, vs, n_tok, q0, n_q, n_kv, window, scale):
    out = empty(n_tok * n_q * HD, torch.float32)
    ctx.attn_prefill_q8(dev(q), dev(kq), dev(ks), dev(vq), dev(vs), n_tok, q0, n_q, n_kv, out,
                        window=window, scale=scale)
    torch.cuda.synchronize()
    return host(out).reshape(n_tok, n_q, HD)


def _want_rows(oracle, q, kd, vd, rows, q0, n_q, n_kv, window, scale):
    out = np.empty((len(rows), n_q, HD), np.float32)
    for r, i in enumerate(rows):
        p = q0 + i
        t0 = max(0, p + 1 - window) if window else 0
        for h in range(n_q):
            out[r, h] = oracle.attention_head(q, kd, vd, i, h, n_q, n_kv, HD, scale, t0, p)
    return out


def _check(got, want, what):
    top = float(np.abs(want).max())
    assert_close(got, want, 2e-3, 1e-3 * top, what)
    assert rel_err(got, want) <= 1e-3, (what, rel_err(got, want))


@pytest.mark.parametrize("n_tok,q0,window,n_q,n_kv", [
    (1, 0, 0, 32, 16), (37, 0, 0, 32, 16), (128, 0, 0, 32, 16), (300, 0, 0, 32, 16),
    (130, 200, 0, 32, 16), (200, 0, 64, 32, 16), (150, 100, 64, 8, 8), (257, 31, 100, 4, 2)])
def test_attn_prefill_matches_oracle(ctx, oracle, n_tok, q0, window, n_q, n_kv):
    print(f"prefill attn n_tok={n_tok} q0={q0} window={window} heads={n_q}/{n_kv}", flush=True)
    scale = 1.0 / np.sqrt(HD)
    q, kq, ks, vq, vs, kd, vd = _case(oracle, 0xF1A5 + n_tok + q0 + window, q0 + n_tok, n_kv,
                                      n_tok, n_q)
    got = _run(ctx, q, kq, ks, vq, vs, n_tok, q0, n_q, n_kv, window, scale)
    rows = list(range(n_tok))
    want = _want_rows(oracle, q, kd, vd, rows, q0, n_q, n_kv, window, scale)
    _check(got, want, f"prefill n_tok={n_tok} q0={q0} w={window}")


@pytest.mark.parametrize("window", [0, 1024])
def test_attn_prefill_config4_sampled(ctx, oracle, window):
    """BASELINE config 4 prefill: 4096 queries, 32 q / 16 kv, causal and
    sliding-1024; sampled query rows (all heads) against the oracle."""
    n_tok, n_q, n_kv = 4096, 32, 16
    print(f"prefill attn config 4 window={window}", flush=True)
    scale = 1.0 / np.sqrt(HD)
    q, kq, ks, vq, vs, kd, vd = _case(oracle, 0xC0F4 + window, n_tok, n_kv, n_tok, n_q)
    got = _run(ctx, q, kq, ks, vq, vs, n_tok, 0, n_q, n_kv, window, scale)
    rows = [0, 1, 63, 127, 128, 1023, 1024, 1025, 2047, 3000, 4094, 4095]
    want = _want_rows(oracle, q, kd, vd, rows, 0, n_q, n_kv, window, scale)
    _check(got[rows], want, f"config 4 w={window}")
    assert np.isfinite(got).all()


def test_attn_prefill_kats(ctx, oracle):
    """reference.rs:572-596: identical keys -> each query's output is the
    mean of the values it sees; window 2 -> mean of the last two values."""
    n_tok, n_q, n_kv = 40, 2, 1
    k = np.zeros(n_tok * HD, np.float32)
    v = np.tile(np.arange(n_tok, dtype=np.float32)[:, None] * 0.25, (1, HD)).reshape(-1)
    ks, kq = oracle.quant_q8_0(k)
    vs, vq = oracle.quant_q8_0(v)
    q = np.ones(n_tok * n_q * HD, np.float32)
    vd = oracle.dequant_q8_0(vs, vq).reshape(n_tok, HD)[:, 0].astype(np.float64)
    for window in (0, 2):
        got = _run(ctx, q, kq, ks, vq, vs, n_tok, 0, n_q, n_kv, window, 0.1)
        for i in range(n_tok):
            lo = max(0, i + 1 - window) if window else 0
            want = vd[lo:i + 1].mean()
            assert np.allclose(got[i], want, rtol=2e-3, atol=1e-3), (window, i)


def test_attn_prefill_is_bit_deterministic(ctx, oracle):
    n_tok, n_q, n_kv = 300, 8, 4
    q, kq, ks, vq, vs, _, _ = _case(oracle, 0xDE7, n_tok, n_kv, n_tok, n_q)
    a = _run(ctx, q, kq, ks, vq, vs, n_tok, 0, n_q, n_kv, 0, 0.1)
    b = _run(ctx, q, kq, ks, vq, vs, n_tok, 0, n_q, n_kv, 0, 0.1)
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("hd,n_tok,q0,window,n_q,n_kv", [
    (256, 1, 0, 0, 32, 16), (256, 300, 0, 0, 32, 16), (256, 150, 77, 64, 32, 16),
    (256, 200, 0, 100, 4, 2), (512, 1, 0, 0, 32, 4), (512, 130, 0, 0, 32, 4),
    (512, 100, 41, 0, 32, 4), (512, 70, 5, 33, 8, 1)])
def test_attn_prefill_wide_head_dims_match_oracle(ctx, oracle, hd, n_tok, q0, window, n_q, n_kv):
    """head_dim 256 / 512 (the released checkpoint's sliding and global
    layers: 32 q heads over 16 kv heads of 256, or over 4 kv heads of 512),
    every row and head against the f64 oracle at the same bar."""
    print(f"prefill attn hd={hd} n_tok={n_tok} q0={q0} window={window} heads={n_q}/{n_kv}",
          flush=True)
    rng = oracle.Rng(0xD1DE + hd + n_tok + q0 + window)
    n_slots = q0 + n_tok
    k = rng.f32_vec(n_slots * n_kv * hd)
    v = rng.f32_vec(n_slots * n_kv * hd)
    ks, kq = oracle.quant_q8_0(k)
    vs, vq = oracle.quant_q8_0(v)
    q = rng.f32_vec(n_tok * n_q * hd)
    kd, vd = oracle.dequant_q8_0(ks, kq), oracle.dequant_q8_0(vs, vq)
    scale = 1.0 / np.sqrt(hd)
    out = empty(n_tok * n_q * hd, torch.float32)
    ctx.attn_prefill_q8(dev(q), dev(kq), dev(ks), dev(vq), dev(vs), n_tok, q0, n_q, n_kv, out,
                        window=window, scale=scale, head_dim=hd)
    torch.cuda.synchronize()
    got = host(out).reshape(n_tok, n_q, hd)
    want = np.empty_like(got)
    for i in range(n_tok):
        p = q0 + i
        t0 = max(0, p + 1 - window) if window else 0
        for h in range(n_q):
            want[i, h] = oracle.attention_head(q, kd, vd, i, h, n_q, n_kv, hd, scale, t0, p)
    _check(got, want, f"prefill hd={hd} n_tok={n_tok} q0={q0} w={window}")


@pytest.mark.parametrize("hd,n_tok,q0,window", [
    (256, 33, 0, 0), (256, 65, 0, 32), (256, 130, 100, 40), (256, 129, 63, 0), (256, 20, 500, 0),
    (512, 64, 0, 0), (512, 70, 260, 0), (512, 33, 288, 0), (512, 40, 300, 33), (512, 16, 500, 100),
    (512, 2, 319, 0)])
@pytest.mark.parametrize("grow", [1.0, 4.0])
def test_attn_prefill_wide_tile_edges(ctx, oracle, hd, n_tok, q0, window, grow):
    """head_dim 256 / 512 around the key tiles (64 / 32 keys), the query tiles
    and the switch of kernels at few keys, windows that leave whole key parts
    of a tile masked; with grow > 1 the keys' magnitude rises by that factor
    over the last third, so that reference maxima move inside the loop.  The
    rounding of q to f16 moves a score by up to 2^-11 of its size, so the bar
    of _check scales with the scores."""
    n_q, n_kv = 4, 2
    print(f"prefill edges hd={hd} n_tok={n_tok} q0={q0} window={window} grow={grow}", flush=True)
    rng = oracle.Rng(0xED9E + hd + n_tok + q0 + window)
    n_slots = q0 + n_tok
    k = rng.f32_vec(n_slots * n_kv * hd).reshape(n_slots, -1)
    k[2 * n_slots // 3:] *= np.float32(grow)
    v = rng.f32_vec(n_slots * n_kv * hd)
    ks, kq = oracle.quant_q8_0(k.reshape(-1))
    vs, vq = oracle.quant_q8_0(v)
    q = rng.f32_vec(n_tok * n_q * hd) * np.float32(2.0)
    kd, vd = oracle.dequant_q8_0(ks, kq), oracle.dequant_q8_0(vs, vq)
    scale = 1.0 / np.sqrt(hd)
    buf = torch.full((n_tok * n_q * hd + 512,), float("nan"), dtype=torch.float32, device="cuda")
    out = buf[256:-256]
    ctx.attn_prefill_q8(dev(q), dev(kq), dev(ks), dev(vq), dev(vs), n_tok, q0, n_q, n_kv, out,
                        window=window, scale=scale, head_dim=hd)
    torch.cuda.synchronize()
    all_ = host(buf)
    assert np.isnan(all_[:256]).all() and np.isnan(all_[-256:]).all()
    got = all_[256:-256].reshape(n_tok, n_q, hd)
    want = np.empty_like(got)
    for i in range(n_tok):
        p = q0 + i
        t0 = max(0, p + 1 - window) if window else 0
        for h in range(n_q):
            want[i, h] = oracle.attention_head(q, kd, vd, i, h, n_q, n_kv, hd, scale, t0, p)
    f = 2.0 * grow
    assert_close(got, want, f * 2e-3, f * 1e-3 * float(np.abs(want).max()), "prefill edges")
    assert rel_err(got, want) <= f * 1e-3


@pytest.mark.parametrize("hd,n_kv", [(256, 2), (512, 1)])
def test_attn_prefill_denominator_keeps_small_probabilities(ctx, oracle, hd, n_kv):
    """A dominating first key (weight 1, V = 127/128) before some 4000 keys of weight
    2^-25.3 each (V = 0): P is rounded to f16, where they are zero, but the
    denominator is the fp32 sum of the unrounded P, so the output is
    V / (1 + n·2^-25.3), 1e-4 below V.  Bar 2e-5: the running fp32 sum may lose
    half an ulp of 1 per 32 keys (125 · 6e-8), and a weight off by q's f16
    rounding (25.3 · 2^-12 of its exponent) moves the result by 4e-7; K and V
    are f16 numbers."""
    n_q, n_tok, q0 = 2 * n_kv, 40, 4000
    n_slots = q0 + n_tok
    gap = 25.3 * np.log(2.0)  # between the first key's score and the others'
    scale = 1.0 / np.sqrt(hd)
    print(f"prefill denominator hd={hd}", flush=True)
    k = np.zeros((n_slots, n_kv, hd), np.float32)
    k[0] = 127.0 / 64.0  # 127 quants of 2^-6
    q = np.full((n_tok, n_q, hd), gap / (hd * scale * k[0, 0, 0]), np.float32)
    v = np.zeros_like(k)
    v[0] = 127.0 / 128.0
    ks, kq = oracle.quant_q8_0(k.reshape(-1))
    vs, vq = oracle.quant_q8_0(v.reshape(-1))
    out = empty(n_tok * n_q * hd, torch.float32)
    ctx.attn_prefill_q8(dev(q.reshape(-1)), dev(kq), dev(ks), dev(vq), dev(vs), n_tok, q0, n_q, n_kv,
                        out, scale=scale, head_dim=hd)
    torch.cuda.synchronize()
    got = host(out).reshape(n_tok, -1).astype(np.float64)
    assert oracle.dequant_q8_0(ks, kq)[0] == k[0, 0, 0] and oracle.dequant_q8_0(vs, vq)[0] == v[0, 0, 0]
    # besides the first, query i sees q0 + i keys
    want = v[0, 0, 0] / (1.0 + np.exp(-gap) * np.arange(q0, q0 + n_tok))
    assert np.abs(got / want[:, None] - 1.0).max() <= 2e-5


@pytest.mark.parametrize("hd,q0,short,long_", [
    (256, 0, 20, 150), (256, 0, 32, 33), (256, 0, 90, 97), (256, 0, 128, 160), (512, 0, 60, 600), (512, 60, 20, 470), (512, 0, 512, 513)])
@pytest.mark.parametrize("grow", [1.0, 4.0])
def test_attn_prefill_rows_do_not_depend_on_the_chunk(ctx, oracle, hd, q0, short, long_, grow):
    """Few keys take another kernel than many: the rows that a short and a long
    chunk share have the same bits, also where the references move."""
    n_q, n_kv = 4, 2
    print(f"prefill chunks hd={hd} q0={q0} {short}/{long_} grow={grow}", flush=True)
    rng = oracle.Rng(0xB175 + hd + q0 + long_)
    k = rng.f32_vec((q0 + long_) * n_kv * hd).reshape(q0 + long_, -1)
    k[(q0 + short) // 3:] *= np.float32(grow)
    ks, kq = oracle.quant_q8_0(k.reshape(-1))
    vs, vq = oracle.quant_q8_0(rng.f32_vec(k.size))
    q = rng.f32_vec(long_ * n_q * hd) * np.float32(2.0)
    got = []
    for n in (short, long_):
        out = empty(n * n_q * hd, torch.float32)
        ctx.attn_prefill_q8(dev(q[:n * n_q * hd]), dev(kq), dev(ks), dev(vq), dev(vs), n, q0, n_q, n_kv,
                            out, scale=1.0 / np.sqrt(hd), head_dim=hd)
        torch.cuda.synchronize()
        got.append(host(out, np.uint32).reshape(n, -1)[:short])
    assert np.array_equal(got[0], got[1])
