"""GPU parity: S>1 causal attention (fp16 MFMA flash kernel) against the CPU
oracle on the same seeded inputs, through the C ABI.

mia_attention_batch follows attention_batch (mistral/mistral_ane_prefill.h:
207-275) over the ring as it stands; mia_attention_step equals S sequential
decode steps (mistral/speculative.h:92-101), also on a wrapped ring."""

import numpy as np
import pytest

import _data as D
import _gpu as G
import _oracle as O

pytestmark = pytest.mark.gpu

TH = O.theta_inv(D.THETA, D.HD)


def _oracle_prefill(kc, vc, Q, K, V, M, start, S):
    """Reference batched prefill on an unwrapped ring: apply_rope_batch,
    kv_write_batch, attention_batch (mistral_ane_prefill.h:746-755)."""
    Qr, Kr = Q.copy(), K.copy()
    O.load().ora_apply_rope_batch(Qr.ctypes.data, Kr.ctypes.data, start, TH.ctypes.data, 32, 8,
                                  128, S)
    O.kv_write_batch(kc, vc, Kr, V, 8, 128, M, start, S)
    return Qr, O.attention_batch_parallel(Qr, kc, vc, 32, 8, 128, M, start, S)


def test_prefill_chunk_after_cache():
    # 512 new tokens appended after 1536 cached positions (2048 total).
    G.say("attention_step prefill S=512 start=1536 M=4096")
    g = D.rng(40)
    M, start, S = 4096, 1536, 512
    kc, vc = D.ring(g, M, filled=start)
    Q, K, V = D.normal(g, (S, 4096)), D.normal(g, (S, 1024)), D.normal(g, (S, 1024))
    out, kc_g, vc_g = G.attention_step(kc, vc, Q, K, V, TH, M, start, S)
    kc_o, vc_o = kc.copy(), vc.copy()
    Qr, ref = _oracle_prefill(kc_o, vc_o, Q, K, V, M, start, S)
    D.check_close(out, ref, what="prefill S=512")
    pos = np.arange(start, start + S)
    D.check_ring(kc_g, kc_o, vc_g, vc_o, pos % M, K, pos, TH, "prefill ring")
    # the literal attention_batch over the written ring gives the same answer
    G.say("attention_batch prefill S=512 start=1536 M=4096")
    out_b = G.attention_batch(Qr, kc_o, vc_o, M, start, S)
    D.check_close(out_b, ref, what="attention_batch S=512")


@pytest.mark.parametrize("start,S", [(0, 2), (0, 3), (5, 7), (0, 8), (100, 9), (0, 33), (3, 64),
                                     (250, 100)])
def test_attention_batch_shapes(start, S):
    G.say(f"attention_batch start={start} S={S}")
    g = D.rng(50 + start + S)
    M = 512
    kc, vc = D.ring(g, M, filled=start + S)
    Q = D.normal(g, (S, 4096))
    out = G.attention_batch(Q, kc, vc, M, start, S)
    ref = O.attention_batch(Q, kc, vc, 32, 8, 128, M, start, S)
    D.check_close(out, ref, what=f"start={start} S={S}")


@pytest.mark.parametrize("start,S", [(16, 16), (17, 40), (15, 50), (100, 9), (1536, 200), (27, 5),
                                     (28, 8), (40, 3), (24, 5), (2000, 48)])
def test_attention_batch_slots_past_range_unread(start, S):
    # Every ring slot from start + S on holds fp16 NaN: a key range whose
    # last tile is partial must neither read those slots nor let them reach
    # the output (0 x NaN in P.V).  The cases put the range end on and off
    # the 32-key tile grid, with ranges of exactly one tile (16 + 16,
    # 27 + 5), a last tile of 1..31 keys, 32- and 64-row tiles, and starts
    # that take the per-lane load path (15, 24) and the uniform one.
    G.say(f"attention_batch NaN past the range start={start} S={S}")
    g = D.rng(70 + start + S)
    M = 4096
    kc, vc = D.ring(g, M, filled=start + S)
    kc[start + S:] = 0x7E00
    vc[start + S:] = 0x7E00
    Q = D.normal(g, (S, 4096))
    out = G.attention_batch(Q, kc, vc, M, start, S)
    assert np.isfinite(out).all(), f"non-finite output start={start} S={S}"
    ref = O.attention_batch(Q, kc, vc, 32, 8, 128, M, start, S)
    D.check_close(out, ref, what=f"NaN past range start={start} S={S}")


@pytest.mark.parametrize("sigma", [2.0, 4.0, 6.0])
def test_attention_batch_large_scores(sigma):
    # Q ~ sigma N(0,1) fp32 and K ~ sigma N(0,1) fp16: scores of order
    # sigma^2 (in units of 1/sqrt(128)), as attention sinks reach.  Q rounded
    # to fp16 alone errs by ~2^-12 |q||k| per score, which breaks the
    # tolerance from sigma = 2 on (max_abs 2.8e-3 measured); the kernel's
    # hi + lo split keeps ~3e-4 at sigma = 6.
    G.say(f"attention_batch large scores sigma={sigma}")
    g = D.rng(int(60 + 10 * sigma))
    M, start, S = 4096, 1536, 64
    kc = np.zeros((M, 1024), np.uint16)
    vc = np.zeros((M, 1024), np.uint16)
    kc[:start + S] = (sigma * g.standard_normal((start + S, 1024))).astype(np.float16).view(np.uint16)
    vc[:start + S] = g.standard_normal((start + S, 1024)).astype(np.float16).view(np.uint16)
    Q = (sigma * g.standard_normal((S, 4096))).astype(np.float32)
    out = G.attention_batch(Q, kc, vc, M, start, S)
    ref = O.attention_batch(Q, kc, vc, 32, 8, 128, M, start, S)
    D.check_close(out, ref, what=f"large scores sigma={sigma}")


@pytest.mark.parametrize("M,start,S", [(300, 1000, 8), (64, 200, 5), (128, 100, 40),
                                       (2048, 2000, 64)])
def test_verify_step_wrapped_small(M, start, S):
    G.say(f"attention_step wrapped M={M} start={start} S={S}")
    g = D.rng(M + start + S)
    kc, vc = D.ring(g, M)
    Q, K, V = D.normal(g, (S, 4096)), D.normal(g, (S, 1024)), D.normal(g, (S, 1024))
    out, kc_g, vc_g = G.attention_step(kc, vc, Q, K, V, TH, M, start, S)
    kc_o, vc_o = kc.copy(), vc.copy()
    ref = O.verify_steps(kc_o, vc_o, Q, K, V, start, S, TH, 32, 8, 128, M)
    D.check_close(out, ref, what=f"verify M={M} start={start} S={S}")
    pos = np.arange(start, start + S)
    D.check_ring(kc_g, kc_o, vc_g, vc_o, pos % M, K, pos, TH, "verify ring")


@pytest.mark.parametrize("start", [70000, 66536])
def test_verify_step_wrapped_65536_ring(start):
    # 65536-slot ring already wrapped; S=8 drafts at start..start+7 (slots
    # 4464.. for 70000, slots 1000.. for 66536).
    G.say(f"attention_step verify M=65536 start={start} S=8")
    g = D.rng(start)
    M, S = 65536, 8
    kc, vc = D.ring(g, M)
    Q, K, V = D.normal(g, (S, 4096)), D.normal(g, (S, 1024)), D.normal(g, (S, 1024))
    out, kc_g, vc_g = G.attention_step(kc, vc, Q, K, V, TH, M, start, S)
    kc_o, vc_o = kc.copy(), vc.copy()
    ref = O.verify_steps(kc_o, vc_o, Q, K, V, start, S, TH, 32, 8, 128, M)
    D.check_close(out, ref, what=f"verify 65536 start={start}")
    pos = np.arange(start, start + S)
    D.check_ring(kc_g, kc_o, vc_g, vc_o, pos % M, K, pos, TH, "verify ring")


def test_verify_causal_among_drafts_index_revealing():
    # Drafts carry keys aligned with every query (in the lowest-frequency RoPE
    # pair, so the alignment survives rotation) and V = their position id; old
    # ring entries have zero keys.  Query t must average exactly drafts 0..t:
    # any future draft leaking in, or an evicted entry resurfacing, moves it.
    G.say("attention_step index-revealing drafts M=40 start=100 S=8")
    M, start, S = 40, 100, 8
    kc = np.zeros((M, 1024), np.uint16)
    vc = np.zeros((M, 1024), np.uint16)
    vc[:] = D.to_f16_bits(np.full(1024, -500.0, np.float32))
    Q = np.zeros((S, 4096), np.float32)
    K = np.zeros((S, 1024), np.float32)
    Q.reshape(S, 32, 128)[:, :, 126] = 40.0
    K.reshape(S, 8, 128)[:, :, 126] = 40.0
    ids = np.arange(start, start + S)
    V = np.zeros((S, 1024), np.float32)
    V[:, 0::2] = (ids // 64)[:, None]
    V[:, 1::2] = (ids % 64)[:, None]
    out, _, _ = G.attention_step(kc, vc, Q, K, V, TH, M, start, S)
    out = out.reshape(S, 32, 128)
    for t in range(S):
        sel = ids[: t + 1]
        assert np.allclose(out[t, :, 0::2], (sel // 64).mean(), atol=2e-2), t
        assert np.allclose(out[t, :, 1::2], (sel % 64).mean(), atol=2e-2), t


def _peaked_large_v(g, M, filled, sigma=2.0, vscale=8.0):
    """Ring with K ~ sigma N(0,1) (scores ~ sigma^2 N(0,1) in units of
    1/sqrt(128): a handful of keys carry each row's weight) and V ~ vscale
    N(0,1) (|v| up to ~5 vscale)."""
    kc = np.zeros((M, 1024), np.uint16)
    vc = np.zeros((M, 1024), np.uint16)
    n = min(filled, M)
    kc[:n] = D.to_f16_bits(sigma * D.normal(g, (n, 1024)))
    vc[:n] = D.to_f16_bits(vscale * D.normal(g, (n, 1024)))
    return kc, vc


def _batch_f64(Q, kc, vc, start, S):
    """float64 causal attention of queries start..start+S-1 over an unwrapped
    ring (slot = position), Q already rotated."""
    n = start + S
    Kf = D.f16_bits_to_f32(kc[:n]).astype(np.float64).reshape(n, 8, 128)
    Vf = D.f16_bits_to_f32(vc[:n]).astype(np.float64).reshape(n, 8, 128)
    Qh = Q.astype(np.float64).reshape(S, 32, 128)
    future = np.arange(n)[None, :] > (start + np.arange(S))[:, None]
    out = np.empty((S, 32, 128))
    for h in range(32):
        s = Qh[:, h] @ Kf[:, h // 4].T / np.sqrt(128.0)
        s[future] = -np.inf
        s -= s.max(axis=1, keepdims=True)
        p = np.exp(s)
        out[:, h] = (p / p.sum(axis=1, keepdims=True)) @ Vf[:, h // 4]
    return out.reshape(S, 4096)


def _check_vs_exact_and_oracle(out, exact, ref, what):
    """The stated bar against the exact (float64) attention; against the
    oracle, the bar plus the oracle's own distance from the exact result
    (the reference's fp32 sums of scores near 20 natural-log units and of
    |v| ~ 40 values err by up to ~3e-3 themselves)."""
    D.check_close(out, exact, what=what + " vs float64")
    slack = np.abs(np.asarray(ref, np.float64) - exact)
    err = np.abs(np.asarray(out, np.float64) - ref)
    assert np.all(err <= D.ATOL + slack), f"{what}: vs oracle {float((err - slack).max()):.3e}"


@pytest.mark.parametrize("start,S", [(1536, 512), (1536, 64), (100, 9)])
def test_attention_batch_peaked_large_v(start, S):
    # Peaked rows over values of magnitude up to ~40: an fp16 P would err
    # by up to 2^-11 |v| per output (2e-2 here); P carried as hi + lo keeps
    # the output within the stated tolerance at any |v|.
    G.say(f"attention_batch peaked rows, V ~ 8 N(0,1): start={start} S={S}")
    g = D.rng(90 + S)
    M = 4096
    kc, vc = _peaked_large_v(g, M, start + S)
    Q = (2.0 * D.normal(g, (S, 4096))).astype(np.float32)
    out = G.attention_batch(Q, kc, vc, M, start, S)
    ref = O.attention_batch_parallel(Q, kc, vc, 32, 8, 128, M, start, S)
    exact = _batch_f64(Q, kc, vc, start, S)
    assert np.abs(exact).max() > 16.0  # the case reaches the large values
    _check_vs_exact_and_oracle(out, exact, ref, f"peaked large V start={start} S={S}")


def test_verify_step_65536_peaked_large_v():
    # The wrapped 65536-slot ring of the verify workload (drafts at 70000..)
    # with peaked rows and V ~ 8 N(0,1): the key range is split over
    # workgroups here, so the split merge is covered at large |v| too.
    G.say("attention_step verify M=65536 start=70000 S=8, peaked rows, V ~ 8 N(0,1)")
    g = D.rng(7)
    M, start, S = 65536, 70000, 8
    kc, vc = _peaked_large_v(g, M, M)
    Q = (2.0 * D.normal(g, (S, 4096))).astype(np.float32)
    K = (2.0 * D.normal(g, (S, 1024))).astype(np.float32)
    V = (8.0 * D.normal(g, (S, 1024))).astype(np.float32)
    out, kc_g, vc_g = G.attention_step(kc, vc, Q, K, V, TH, M, start, S)
    kc_o, vc_o = kc.copy(), vc.copy()
    ref = O.verify_steps(kc_o, vc_o, Q, K, V, start, S, TH, 32, 8, 128, M)
    pos = np.arange(start, start + S)
    D.check_ring(kc_g, kc_o, vc_g, vc_o, pos % M, K, pos, TH, "verify ring")
    # exact: token t over the ring with drafts 0..t written (sequential
    # verify), q and the drafts' keys as the oracle rotated them
    Qr = Q.copy()
    O.load().ora_apply_rope_batch(Qr.ctypes.data, None, start, TH.ctypes.data, 32, 8, 128, S)
    exact = np.empty((S, 4096))
    rk, rv = kc.copy(), vc.copy()
    for t in range(S):
        rk[(start + t) % M] = kc_o[(start + t) % M]
        rv[(start + t) % M] = vc_o[(start + t) % M]
        exact[t] = D.gqa_decode_f64(Qr[t], rk, rv, 32, 8, 128, M, start + t)
    assert np.abs(exact).max() > 16.0
    _check_vs_exact_and_oracle(out, exact, ref, "verify 65536 peaked large V")


@pytest.mark.parametrize("M,start,S,peaks", [
    (4096, 1536, 64, (33, 700, 1599)),   # 64-row tiles: second tile, mid-range, the last key
    (4096, 0, 70, (31, 32, 69)),         # rows whose waves have no keys in their first tile
    (4096, 500, 8, (64, 507)),           # 32-row tiles
    (300, 1000, 40, (5, 250)),           # wrapped windows (slots): rows that start mid-tile
    (300, 1000, 8, (5, 104, 250)),
    (4096, 1500, 300, (131, 160, 1000, 1799)),  # 64-row tiles, split by wave: second tile to the last
    (4096, 0, 270, (100, 128, 129, 269)),       # rows whose waves have one tile, or none
    (2048, 2500, 320, (1, 1000, 2047)),         # a wrapped ring
])
def test_attention_batch_peaks_raise_the_reference(M, start, S, peaks):
    # A few keys 16 times as large: scores reach +-70 log2 units, so rows
    # raise their softmax reference at those tiles (and only some rows of a
    # wave do).  Against float64, with V ~ 8 N(0,1): what was summed before a
    # peak must be scaled with it, at the precision of the other rows.
    G.say(f"attention_batch peaks M={M} start={start} S={S} at {peaks}")
    g = D.rng(300 + S + M)
    kc, vc = _peaked_large_v(g, M, start + S, sigma=1.0)
    for p in peaks:
        kc[p] = D.to_f16_bits(16.0 * D.f16_bits_to_f32(kc[p]))
    Q = D.normal(g, (S, 4096))
    out = G.attention_batch(Q, kc, vc, M, start, S)
    exact = np.empty((S, 4096))
    for t in range(S):  # the ring as it stands holds the positions up to start + S - 1
        n = min(start + t + 1, M)
        exact[t] = D.gqa_decode_f64(Q[t], kc[:n], vc[:n], 32, 8, 128, n, n - 1)
    D.check_close(out, exact, what=f"peaks M={M} start={start} S={S}")


@pytest.mark.parametrize("M,start,S", [
    (8192, 0, 1), (8192, 0, 17), (8192, 30, 2),   # row tiles with fewer keys than a tile
    (24, 100, 5),                                 # a ring smaller than a tile
    (300, 290, 40),                               # a chunk that wraps: windows of 291 .. 300 slots
    (300, 1000, 70), (1024, 5000, 16),            # wrapped, whole ring; split over workgroups
    (4096, 900, 16), (4096, 505, 8),              # the shortest ranges that are split
])
def test_attention_batch_ring_in_slot_order(M, start, S):
    # Attention over the ring as it stands walks slots 0 .. min(pos, M - 1);
    # slots no window reaches hold NaN and must not be read into a product.
    G.say(f"attention_batch slot order M={M} start={start} S={S}")
    g = D.rng(M + start + S)
    filled = min(start + S, M)
    kc, vc = D.ring(g, M, filled=filled)
    kc[filled:], vc[filled:] = 0x7E00, 0x7E00
    Q = D.normal(g, (S, 4096))
    out = G.attention_batch(Q, kc, vc, M, start, S)
    exact = np.empty((S, 4096))
    for t in range(S):
        n = min(start + t + 1, M)
        exact[t] = D.gqa_decode_f64(Q[t], kc[:n], vc[:n], 32, 8, 128, n, n - 1)
    D.check_close(out, exact, what=f"slot order M={M} start={start} S={S}")


@pytest.mark.parametrize("M,start,S", [
    (8192, 0, 9), (8192, 1008, 16), (8192, 1009, 16),  # 8-token tiles; the merge as its own launch
    (8192, 1260, 20), (8192, 1261, 20),                # one split, two splits
    (8192, 7000, 17), (700, 3000, 33),                 # eight splits; a wrapped ring in one
    (4096, 1300, 128), (4096, 1300, 129),              # two splits of every tile, none
    (2048, 700, 256), (2048, 700, 257),                # 8-token tiles fill the device; 16-token tiles
])
def test_attention_batch_tiles_and_splits(M, start, S):
    # Where the row tile, the split of the keys and its merge change; twice (the merge's counters
    # are back at rest).
    G.say(f"attention_batch tiles and splits M={M} start={start} S={S}")
    g = D.rng(7 * M + start + S)
    filled = min(start + S, M)
    kc, vc = D.ring(g, M, filled=filled, spike_every=256)
    kc[filled:], vc[filled:] = 0x7E00, 0x7E00
    Q = D.normal(g, (S, 4096))
    rows = range(S) if S < 20 else sorted({0, 1, 7, 8, S // 2, S - 2, S - 1})
    for turn in range(2):
        out = G.attention_batch(Q, kc, vc, M, start, S)
        assert np.all(np.isfinite(out))
        for t in rows:
            n = min(start + t + 1, M)
            exact = D.gqa_decode_f64(Q[t], kc[:n], vc[:n], 32, 8, 128, n, n - 1)
            D.check_close(out[t], exact, what=f"turn={turn} M={M} start={start} S={S} t={t}")


@pytest.mark.parametrize("M,start,S,peaks", [
    (600, 580, 40, (300, 577)),            # 64-row tiles with staged rows: the window's middle and end
    (600, 1500, 33, (1000, 1200, 1499)),   # a wrapped window, split over workgroups or whole
    (300, 2000, 70, (1800, 1999)),
])
def test_attention_step_peaks_next_to_staged_rows(M, start, S, peaks):
    # The reference-raising path with per-lane key addresses (ring and staging
    # buffer): a chunk that does not fit the ring beside its window, a few of
    # the cached keys and one new key 16 times as large.
    G.say(f"attention_step peaks M={M} start={start} S={S} at {peaks}")
    g = D.rng(500 + S + M)
    kc, vc = _peaked_large_v(g, M, M, sigma=1.0)
    for p in peaks:
        kc[p % M] = D.to_f16_bits(16.0 * D.f16_bits_to_f32(kc[p % M]))
    Q, K, V = D.normal(g, (S, 4096)), D.normal(g, (S, 1024)), D.normal(g, (S, 1024))
    K[S // 2] *= 16.0
    # kn, vn: the rings as the library left them, whose new fp16 rows the queries attended
    out, kn, vn = G.attention_step(kc, vc, Q, K, V, TH, M, start, S)
    exact = np.empty((S, 4096))
    for t in range(S):
        kc[(start + t) % M], vc[(start + t) % M] = kn[(start + t) % M], vn[(start + t) % M]
        q = D.rope_f64(Q[t], start + t, TH, 32, 128)
        exact[t] = D.gqa_decode_f64(q, kc, vc, 32, 8, 128, M, start + t)
    D.check_close(out, exact, what=f"step peaks M={M} start={start} S={S}")
