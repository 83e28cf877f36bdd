"""GPU: calls that share row tiles between tokens (mia_attention_positions,
mia_attention_chunk, unstaged steps) on several streams, from several threads
and in HIP graphs: each stream has its own work area, and the counts by which
the splits of a tile find the last one start anew in every launch."""

import ctypes
import threading

import numpy as np
import pytest

import _data as D
import _gpu as G
import _oracle as O
from anetransformers_amd import DeviceBuffer as DB
from anetransformers_amd import check
from test_gpu_positions import _call_ms
from test_zz_no_alloc import _hip

pytestmark = pytest.mark.gpu

TH = O.theta_inv(D.THETA, D.HD)
M = 8192


class Call:
    """One entry point on its own ring and inputs, rows at start .. start + S - 1 (n_kv kv heads)."""

    def __init__(self, op, start, S, seed, n_kv=8, M=M):
        self.op, self.start, self.S, self.n_kv, self.M = op, start, S, n_kv, M
        g = D.rng(seed)
        kv, dim = n_kv * 128, n_kv * 512
        self.kc, self.vc = D.ring(g, M, kv_dim=kv, filled=start)
        self.Q = D.normal(g, (S, dim))
        self.K, self.V = D.normal(g, (S, kv)), D.normal(g, (S, kv))
        self.dev = [DB.from_array(a) for a in (self.kc, self.vc, self.Q, self.K, self.V, TH)]
        self.pos = DB.from_array(np.arange(start, start + S, dtype=np.int32))
        if op in ("positions", "batch"):  # the ring as it stands: the tokens' rows are in it
            for dev, host in zip(self.dev, (self.kc, self.vc)):
                host[start:start + S] = D.to_f16_bits(D.normal(g, (S, kv)))
                dev.upload(host)

    def __call__(self, out, stream):
        kc, vc, Q, K, V, th = (d.ptr for d in self.dev)
        lib, heads, S = G.lib(), 4 * self.n_kv, self.S
        if self.op == "positions":
            rc = lib.mia_attention_positions(Q, out.ptr, kc, vc, self.pos.ptr, heads, self.n_kv,
                                             128, self.M, S, stream)
        elif self.op == "batch":
            rc = lib.mia_attention_batch(Q, out.ptr, kc, vc, heads, self.n_kv, 128, self.M, self.start, S,
                                         stream)
        elif self.op == "chunk":
            rc = lib.mia_attention_chunk(Q, K, V, self.pos.ptr, th, kc, vc, out.ptr, heads,
                                         self.n_kv, 128, self.M, S, stream)
        else:
            rc = lib.mia_attention_step(Q, K, V, th, kc, vc, out.ptr, heads, self.n_kv, 128, self.M,
                                        self.start, S, stream)
        check(rc, self.op)

    def buffer(self):
        return DB.from_array(np.full((self.S, self.Q.shape[1]), np.nan, np.float32))

    def rows(self, out):
        return out.download(self.Q.shape, np.float32)

    def alone(self):
        out = self.buffer()
        self(out, None)
        check(G.lib().mia_stream_sync(None), "sync")
        return self.rows(out)


def _stream():
    s = ctypes.c_void_p()
    check(G.lib().mia_stream_create(ctypes.byref(s)), "stream")
    return s


@pytest.mark.parametrize("op", ["positions", "chunk"])
def test_overlapping_streams(op):
    # Two threads, a stream each, 60 calls without a wait in between: other
    # numbers of tokens, of splits and of tiles, so that neither partials nor
    # counts of one fit the other.  Bit for bit what each call gives alone.
    G.say(f"two streams of attention_{op}")
    calls = [Call(op, 7000, 32, 70), Call(op, 2600, 56, 71)]
    want = [c.alone() for c in calls]
    streams = [_stream(), _stream()]
    outs = [[c.buffer() for _ in range(60)] for c in calls]
    failed = []

    def run(i):
        try:
            for o in outs[i]:
                calls[i](o, streams[i])
            check(G.lib().mia_stream_sync(streams[i]), "sync")
        except Exception as e:
            failed.append(e)

    threads = [threading.Thread(target=run, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed
    for i, c in enumerate(calls):
        for n, o in enumerate(outs[i]):
            assert np.array_equal(c.rows(o), want[i]), f"stream {i} call {n}"
        G.lib().mia_stream_destroy(streams[i])


def test_more_streams_than_areas():
    # Streams without an area take the kernels that need none; a destroyed
    # stream's area goes to the next.
    G.say("attention_positions on twelve streams")
    c = Call("positions", 7000, 40, 72)
    want = c.alone()
    exact = np.stack([D.gqa_decode_f64(c.Q[t], c.kc, c.vc, 32, 8, 128, M, c.start + t)
                      for t in range(c.S)])
    streams = [_stream() for _ in range(12)]
    outs = [c.buffer() for _ in streams]
    for o, s in zip(outs, streams):
        c(o, s)
    for o, s in zip(outs, streams):
        check(G.lib().mia_stream_sync(s), "sync")
        D.check_close(c.rows(o), exact, what="one of twelve streams")
    same = [np.array_equal(c.rows(o), want) for o in outs]
    assert same[0] and not same[-1]  # (the two kernels round differently here)
    for s in streams:
        check(G.lib().mia_stream_destroy(s), "destroy")
    s, o = _stream(), c.buffer()
    c(o, s)
    check(G.lib().mia_stream_sync(s), "sync")
    assert np.array_equal(c.rows(o), want)
    check(G.lib().mia_stream_destroy(s), "destroy")


@pytest.mark.parametrize("op", ["positions", "batch", "chunk", "step"])
def test_first_call_of_a_stream_captured(op):
    # The first call on a stream is captured in global mode (no allocation, no
    # synchronisation), then replayed between eager calls of the same stream
    # with other splits: each leaves its counts behind, of later launches than
    # the captured one, and every replay and every eager call is right.
    G.say(f"attention_{op} captured as a stream's first call")
    lib, hip = G.lib(), _hip()
    c, other = Call(op, 5000, 40, 73), Call(op, 1400, 40, 74)
    want, want_other = c.alone(), other.alone()
    stream, out, out_other = _stream(), c.buffer(), other.buffer()
    graph, gexec = ctypes.c_void_p(), ctypes.c_void_p()
    try:
        assert hip.hipStreamBeginCapture(stream, 0) == 0
        try:
            c(out, stream)
        finally:
            end = hip.hipStreamEndCapture(stream, ctypes.byref(graph))
        assert end == 0, f"capture ended with hipError {end}"
        assert hip.hipGraphInstantiate(ctypes.byref(gexec), graph, None, None, 0) == 0
        for rep in range(4):
            out.zero()
            out_other.zero()
            check(lib.mia_device_sync(), "sync")
            assert hip.hipGraphLaunch(gexec, stream) == 0
            check(lib.mia_stream_sync(stream), "sync")
            assert np.array_equal(c.rows(out), want), f"replay {rep}"
            other(out_other, stream)
            check(lib.mia_stream_sync(stream), "sync")
            assert np.array_equal(other.rows(out_other), want_other), f"eager call {rep}"
    finally:
        if gexec.value:
            hip.hipGraphExecDestroy(gexec)
        if graph.value:
            hip.hipGraphDestroy(graph)
        lib.mia_stream_destroy(stream)


@pytest.mark.parametrize("n_kv,S", [(2, 33), (4, 20), (1, 70), (2, 500)])
@pytest.mark.parametrize("op", ["positions", "step"])
def test_fewer_kv_heads(op, n_kv, S):
    # a rank that owns some of the heads: other numbers of tiles and splits
    G.say(f"attention_{op} n_kv={n_kv} S={S}")
    c = Call(op, 3000, S, 75 + n_kv, n_kv)
    got = c.alone()
    kc, vc = (d.download(a.shape, np.uint16) for d, a in zip(c.dev, (c.kc, c.vc)))
    Q = c.Q.copy()
    if op == "step":
        for t in range(S):
            O.apply_rope(Q[t], c.K[t].copy(), c.start + t, TH, 4 * n_kv, n_kv, 128)
    for t in sorted({0, 1, 7, 8, S // 2, S - 2, S - 1}):
        exact = D.gqa_decode_f64(Q[t], kc, vc, 4 * n_kv, n_kv, 128, M, c.start + t)
        D.check_close(got[t], exact, what=f"{op} n_kv={n_kv} S={S} t={t}")


@pytest.mark.parametrize("n_kv,S,M,keys", [
    (1, 17, 4096, 900), (1, 17, 4096, 901),      # short windows: tiles that share keys at any count
    (8, 16, 4096, 1024), (8, 16, 4096, 1025),    # 16 tiles
    (8, 24, 8192, 4800), (8, 24, 8192, 4801),    # 24 tiles
    (8, 80, 16384, 9216), (8, 80, 16384, 9217),
    (8, 128, 16384, 12288), (8, 128, 16384, 12289),
])
def test_batch_where_the_kernel_changes(n_kv, S, M, keys):
    G.say(f"attention_batch n_kv={n_kv} S={S} keys={keys}")
    c = Call("batch", keys - S, S, 80, n_kv, M)
    got = c.alone()
    for t in sorted({0, 7, 8, S - 2, S - 1}):
        exact = D.gqa_decode_f64(c.Q[t], c.kc, c.vc, 4 * n_kv, n_kv, 128, M, c.start + t)
        D.check_close(got[t], exact, what=f"n_kv={n_kv} S={S} keys={keys} t={t}")


def test_long_windows_of_few_rows_use_the_device():
    # 17 tokens of one kv head: three row tiles.  With eight ranges of keys a tile
    # the step took 4.3 times as long after 64K keys as after 4K; split over the
    # device it takes 1.6 times as long.
    G.say("attention_batch n_kv=1 S=17, 4K and 64K keys")
    ms = []
    for keys in (4096, 65536):
        c = Call("batch", keys - 17, 17, 81, 1, keys)
        out = c.buffer()
        ms.append(min(_call_ms(lambda: c(out, None), 20) for _ in range(3)))
    print(f"{ms[0] * 1e3:.1f} us, {ms[1] * 1e3:.1f} us", flush=True)
    assert ms[1] < 2.7 * ms[0]


@pytest.mark.parametrize("n_kv,S,M,keys", [
    (1, 32, 4096, 3000), (1, 33, 4096, 3000), (2, 16, 4096, 3000), (2, 17, 4096, 3000),
    (8, 32, 1024, 1024), (8, 32, 1025, 1025), (8, 31, 1024, 1024),
])
@pytest.mark.parametrize("op", ["positions", "chunk"])
def test_positions_where_the_kernel_changes(op, n_kv, S, M, keys):
    G.say(f"attention_{op} n_kv={n_kv} S={S} M={M}")
    c = Call(op, keys - S, S, 82, n_kv, M)
    got = c.alone()
    kc, vc = (d.download(a.shape, np.uint16) for d, a in zip(c.dev, (c.kc, c.vc)))
    Q = c.Q.copy()
    if op == "chunk":
        for t in range(S):
            O.apply_rope(Q[t], c.K[t].copy(), c.start + t, TH, 4 * n_kv, n_kv, 128)
    for t in sorted({0, 7, 8, S - 2, S - 1}):
        exact = D.gqa_decode_f64(Q[t], kc, vc, 4 * n_kv, n_kv, 128, M, c.start + t)
        D.check_close(got[t], exact, what=f"{op} n_kv={n_kv} S={S} M={M} t={t}")


def test_few_rows_of_a_long_ring_use_the_device():
    # 16 tokens of one kv head on a 64K ring: two row tiles, at most eight ranges
    # of keys each, took 1.7 times as long as the decode kernel's 256 workgroups.
    G.say("attention_positions n_kv=1, 16 tokens and 8 on a 64K ring")
    ms = []
    for S in (8, 16):
        c = Call("positions", 65536 - S, S, 83, 1, 65536)
        out = c.buffer()
        ms.append(min(_call_ms(lambda: c(out, None), 20) for _ in range(3)))
    print(f"{ms[0] * 1e3:.1f} us, {ms[1] * 1e3:.1f} us", flush=True)
    assert ms[1] < 1.9 * ms[0]
