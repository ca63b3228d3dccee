"""The prompt-chunk attention kernel over bf16 caches: tile edges, splits of the cache, their workspace."""
import numpy as np
import pytest

from tests.util import rel_err, rel_err_rows

pytestmark = pytest.mark.gpu

# The query and the probabilities enter as two bf16 parts: 2^-17 of an operand each, on scores of a few units.
TOL = 1e-4


def _inputs(oracle, Hq, Hkv, d, T, L0, seed):
    rng = np.random.default_rng(seed)
    k, v = (oracle.bf16_to_f32(oracle.f32_to_bf16(rng.standard_normal((L0 + T, Hkv * d)).astype(np.float32))) for _ in range(2))
    q = rng.standard_normal((T, Hq * d)).astype(np.float32)
    return q, rng.standard_normal((T, Hq * d)).astype(np.float32), k, v


def _ctx(mfa, Hq, Hkv, d, cap):
    from moeflux_amd import Config
    return mfa.Ctx(Config(num_layers=1, full_attn_interval=1, num_attn_heads=Hq, num_kv_heads=Hkv, head_dim=d,
                          kv_capacity=cap, kv_dtype=1))


# Rows of a workgroup are 128 or 64, of a wave 32, blocks 32 positions, chunks of K 64; long caches are split.
@pytest.mark.parametrize("Hq,Hkv,d,T,L0", [
    (8, 2, 128, 8, 0), (8, 2, 128, 9, 23), (4, 1, 64, 31, 1), (4, 1, 256, 33, 31),     # a row either side of a tile
    (16, 1, 128, 2, 62), (16, 1, 256, 3, 61), (6, 2, 64, 65, 64),                      # positions either side of a chunk of K
    (32, 4, 128, 40, 2500), (16, 2, 256, 50, 1990), (16, 2, 64, 40, 5000), (4, 1, 64, 70, 1900),   # splits
    (16, 2, 256, 130, 600), (3, 3, 128, 129, 4000), (24, 1, 256, 11, 2303),                             # two wave sets; few rows
])
def test_chunk_against_the_oracle(mfa, oracle, Hq, Hkv, d, T, L0):
    q, g, k, v = _inputs(oracle, Hq, Hkv, d, T, L0, T + L0)
    ref = oracle.prefill_attn(T, L0, Hq, Hkv, d, q, g, k, v).reshape(T, Hq * d)
    with _ctx(mfa, Hq, Hkv, d, L0 + T) as c:
        if L0:
            c.kv_import(0, k[:L0], v[:L0])
        out = c.prefill_attn(0, q, g, k[L0:], v[L0:])
        # once more over a workspace of NaN: a split whose positions a tile cannot see leaves its part unwritten
        c.memory_seq_rm(L0)
        if L0:
            c.kv_import(0, k[:L0], v[:L0])
        assert c.lib.mfa_debug_fill_workspace(c.h, 0x7FC00000) == 0
        again = c.prefill_attn(0, q, g, k[L0:], v[L0:])
    assert rel_err(out, ref) <= TOL
    assert rel_err_rows(out, ref, d) <= 5 * TOL
    assert np.array_equal(out, again)


def test_chunk_split_with_peaked_scores(mfa, oracle):
    """Scores of +-130: the running maximum rises by far more than the lazy rescaling's 2^8, in some splits only."""
    Hq, Hkv, d, T, L0 = 16, 2, 256, 50, 1990
    q, g, k, v = _inputs(oracle, Hq, Hkv, d, T, L0, 3)
    q *= 8.0
    k[::97] *= 4.0
    ref = oracle.prefill_attn(T, L0, Hq, Hkv, d, q, g, k, v).reshape(T, Hq * d)
    with _ctx(mfa, Hq, Hkv, d, L0 + T) as c:
        c.kv_import(0, k[:L0], v[:L0])
        out = c.prefill_attn(0, q, g, k[L0:], v[L0:])
    # a score s carries up to 2^-17 |s| from the query's two parts: 1e-3 of a probability at |s| = 130
    assert rel_err(out, ref) <= 2e-3


@pytest.mark.parametrize("Hq,Hkv,d,T,L0", [(16, 2, 256, 203, 3001), (32, 4, 128, 128, 4000), (16, 2, 64, 40, 5000)])
def test_chunk_split_of_nothing_but_nan(mfa, oracle, Hq, Hkv, d, T, L0):
    """The first n keys of a kv head are NaN, for every n that a split of the cache may end at: the rows of its query heads
    are NaN, as in the token loop, and the other heads' are what they were."""
    q, g, k, v = _inputs(oracle, Hq, Hkv, d, T, L0, 5)
    ref = oracle.prefill_attn(T, L0, Hq, Hkv, d, q, g, k, v).reshape(T, Hkv, -1)
    with _ctx(mfa, Hq, Hkv, d, L0 + T) as c:
        for n in range(32, 1600, 32):
            bad = k.copy()
            bad[:n, :d] = np.nan
            c.memory_clear()
            c.kv_import(0, bad[:L0], v[:L0])
            out = c.prefill_attn(0, q, g, bad[L0:], v[L0:]).reshape(T, Hkv, -1)
            assert np.isnan(out[:, 0]).all(), n
            assert rel_err(out[:, 1:], ref[:, 1:]) <= TOL


@pytest.mark.parametrize("Hq,Hkv,d,T,L0,rotary", [
    (32, 4, 128, 70, 0, 32), (16, 2, 256, 70, 41, 64), (32, 4, 128, 40, 2500, 32), (16, 2, 256, 50, 1990, 64),
    (16, 2, 256, 50, 1990, 32), (8, 2, 64, 70, 41, 16),     # not a quarter of the head, head_dim 64: a prologue of its own
    (6, 3, 128, 77, 10, 32),
])
def test_raw_projections_against_the_separate_prologue(mfa, oracle, Hq, Hkv, d, T, L0, rotary):
    """The chunk kernel's own norm and rotation of the query against the prologue launch, the decode kernel (a forced
    split count) and the prologue's cache rows; and with the result written over the projection, which sends the call
    down the prologue's path too."""
    from moeflux_amd.hip import DeviceArray
    rng = np.random.default_rng(T + L0 + d)
    norm = [oracle.f32_to_bf16(1.0 + 0.3 * rng.standard_normal(d)) for _ in range(2)]
    qp = rng.standard_normal((T, Hq * 2 * d)).astype(np.float32)
    k, v = (rng.standard_normal((L0 + T, Hkv * d)).astype(np.float32) for _ in range(2))

    def run(how):
        with _ctx(mfa, Hq, Hkv, d, L0 + T) as c:
            c.set_rope(1.0e7, rotary)
            c.set_full_weights(0, *norm)
            if L0:
                c.kv_import(0, k[:L0], v[:L0])
            if how == "decode":
                c.set_num_splits(1)
            if how == "in place":
                dq, dk, dv = (DeviceArray.from_host(x) for x in (qp, k[L0:], v[L0:]))
                assert c.lib.mfa_prefill_full_attn_dev(c.h, 0, L0, T, dq.ptr, dk.ptr, dv.ptr, dq.ptr) == 0
                c.sync()
                out = dq.to_host().reshape(-1)[:T * Hq * d].reshape(T, Hq * d)
            else:
                out = c.prefill_full_attn(0, L0, qp, k[L0:], v[L0:])
            return out, c.kv_export(0)

    out, cache = run("raw")
    for how in ("decode", "in place"):
        other, other_cache = run(how)
        assert rel_err(out, other) <= TOL, how
        assert all(np.array_equal(a, b) for a, b in zip(cache, other_cache)), how


def test_chunk_and_short_decode_in_a_captured_graph(mfa, oracle):
    """Captured on a context that has no chunk workspace yet (the plan then needs none), replayed between eager calls: a
    chunk whose eager plan splits the cache, and a decode call that draws tickets."""
    import ctypes as C

    from moeflux_amd.hip import DeviceArray, rt
    Hq, Hkv, d, T, L0, short = 16, 2, 256, 50, 1990, 515
    q, g, k, v = _inputs(oracle, Hq, Hkv, d, T, L0, 9)
    with _ctx(mfa, Hq, Hkv, d, L0 + T) as e:
        e.kv_import(0, k[:L0], v[:L0])
        want = e.prefill_attn(0, q, g, k[L0:], v[L0:])
        e.memory_clear()
        e.kv_import(0, k[:short], v[:short])
        want_short = e.sdpa_decode(0, q[0], g[0])
    dq, dg, dk, dv = (DeviceArray.from_host(x) for x in (q, g, k[L0:], v[L0:]))
    for what in ("chunk", "decode"):
        n = L0 if what == "chunk" else short
        with _ctx(mfa, Hq, Hkv, d, L0 + T) as c:
            c.kv_import(0, k[:n], v[:n])
            out = DeviceArray((T, Hq * d), zero=True)
            stream, graph, run = C.c_void_p(c.lib.mfa_stream(c.h)), C.c_void_p(), C.c_void_p()
            assert rt().hipStreamBeginCapture(stream, C.c_int(2)) == 0   # relaxed: other streams are not held up
            if what == "chunk":
                rc = c.lib.mfa_prefill_attn_dev(c.h, 0, T, dq.ptr, dg.ptr, dk.ptr, dv.ptr, out.ptr)
            else:
                rc = c.lib.mfa_sdpa_decode_dev(c.h, 0, dq.ptr, dg.ptr, out.ptr)
            assert rt().hipStreamEndCapture(stream, C.byref(graph)) == 0 and rc == 0
            assert rt().hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
            for _ in range(3):
                assert rt().hipGraphLaunch(run, stream) == 0
                c.sync()
                got = out.to_host()
                if what == "chunk":
                    assert rel_err(got, want) <= TOL
                else:
                    assert np.array_equal(got[0], want_short)
                    assert np.array_equal(c.sdpa_decode(0, q[0], g[0]), want_short)   # eager work in between
            assert rt().hipGraphExecDestroy(run) == 0 and rt().hipGraphDestroy(graph) == 0


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("route", [1, 2001, 4001, 2003, 4003])
def test_every_form_against_the_oracle(mfa, oracle, route, d):
    """16-row groups, and both shapes of the 32x32-tile kernel on the whole cache and on three splits of it, a row either
    side of their tiles and of a block; from a normed query and from raw projections (rows of the oracle's prologue over
    the cache as exported)."""
    theta = 1.0e7
    for Hq, Hkv, T, L0 in [(8, 2, 8, 0), (4, 1, 31, 1), (4, 1, 33, 31), (16, 1, 3, 61), (6, 2, 65, 64), (3, 3, 129, 290), (24, 1, 11, 95)]:
        q, g, k, v = _inputs(oracle, Hq, Hkv, d, T, L0, T + L0)
        qp = np.stack([q.reshape(T, Hq, d), g.reshape(T, Hq, d)], 2).reshape(T, Hq * 2 * d)
        rng = np.random.default_rng(T)
        norm = [oracle.f32_to_bf16(1.0 + 0.3 * rng.standard_normal(d)) for _ in range(2)]
        with _ctx(mfa, Hq, Hkv, d, L0 + T) as c:
            c.set_full_weights(0, *norm)
            c.set_rope(theta, d // 4)
            assert c.lib.mfa_debug_set_chunk_route(c.h, route) == 0
            for raw in (False, True):
                c.memory_clear()
                if L0:
                    c.kv_import(0, k[:L0], v[:L0])
                c.lib.mfa_debug_fill_workspace(c.h, 0x7FC00000)
                out = c.prefill_full_attn(0, L0, qp, k[L0:], v[L0:]) if raw else c.prefill_attn(0, q, g, k[L0:], v[L0:])
                kc, vc = c.kv_export(0)
                qr = q
                if raw:
                    qr = np.stack([oracle.attn_prologue(L0 + t, Hq, Hkv, d, d // 4, theta, 1e-6, *norm, qp[t], k[L0 + t], v[L0 + t])[0]
                                   for t in range(T)])
                ref = oracle.prefill_attn(T, L0, Hq, Hkv, d, qr, g, kc, vc).reshape(T, Hq * d)
                assert rel_err(out, ref) <= TOL, (Hq, Hkv, T, L0, raw)
                assert rel_err_rows(out, ref, d) <= 5 * TOL, (Hq, Hkv, T, L0, raw)


class _Graph:
    """What `call` puts on a context's stream, captured (relaxed: other streams are not held up)."""

    def __init__(self, c, call):
        import ctypes as C

        from moeflux_amd.hip import rt
        self.c, self.rt, self.stream, self.graph, self.run = c, rt(), C.c_void_p(c.lib.mfa_stream(c.h)), C.c_void_p(), C.c_void_p()
        assert self.rt.hipStreamBeginCapture(self.stream, C.c_int(2)) == 0
        rc = call()
        end = self.rt.hipStreamEndCapture(self.stream, C.byref(self.graph))
        assert rc == 0, c.lib.mfa_last_error_string()
        assert end == 0
        assert self.rt.hipGraphInstantiate(C.byref(self.run), self.graph, None, None, C.c_size_t(0)) == 0

    def __call__(self):
        assert self.rt.hipGraphLaunch(self.run, self.stream) == 0
        self.c.sync()

    def close(self):
        assert self.rt.hipGraphExecDestroy(self.run) == 0 and self.rt.hipGraphDestroy(self.graph) == 0


@pytest.mark.parametrize("few", [0, 40])
@pytest.mark.parametrize("first", ["over the projection", "apart"])
def test_both_routes_of_a_raw_chunk_share_their_scratch(mfa, oracle, first, few):
    """A chunk whose result lies over its projection (a prologue of its own) captured behind one of as many tokens whose
    result lies apart (query normed in the attention launch), and the other way round, on scratch that the capture makes or
    (after a chunk of few tokens) grows; then the first route again, eagerly, and replays."""
    from moeflux_amd.hip import H2D, DeviceArray, rt
    Hq, Hkv, d, T = 16, 2, 256, 300
    rng = np.random.default_rng(4)
    norm = [oracle.f32_to_bf16(1.0 + 0.3 * rng.standard_normal(d)) for _ in range(2)]
    qp = rng.standard_normal((T, Hq * 2 * d)).astype(np.float32)
    k, v = (rng.standard_normal((T, Hkv * d)).astype(np.float32) for _ in range(2))
    dk, dv = (DeviceArray.from_host(x) for x in (k, v))
    with _ctx(mfa, Hq, Hkv, d, T) as c:
        c.set_full_weights(0, *norm)
        want = c.prefill_full_attn(0, 0, qp, k, v)
        bufs = {"apart": (DeviceArray.from_host(qp), DeviceArray((T, Hq * d), zero=True)), "over the projection": (DeviceArray.from_host(qp),) * 2}

        def call(where, n=T):
            q, out = bufs[where]
            return c.lib.mfa_prefill_full_attn_dev(c.h, 0, 0, n, q.ptr, dk.ptr, dv.ptr, out.ptr)

        def check(where):
            assert rel_err(bufs[where][1].to_host().reshape(-1)[:T * Hq * d].reshape(T, Hq * d), want) <= TOL
            assert rt().hipMemcpy(bufs[where][0].ptr, qp.ctypes.data, qp.nbytes, H2D) == 0

        second = next(w for w in bufs if w != first)
    with _ctx(mfa, Hq, Hkv, d, T) as c:   # its scratch is of its own first chunk
        c.set_full_weights(0, *norm)
        if few:
            assert call(second, few) == 0
            c.sync()
            assert rt().hipMemcpy(bufs[second][0].ptr, qp.ctypes.data, qp.nbytes, H2D) == 0
            c.memory_clear()
        assert call(first) == 0
        c.sync()
        check(first)
        c.memory_clear()
        graph = _Graph(c, lambda: call(second))
        for _ in range(3):
            graph()
            check(second)
            c.memory_clear()
            assert call(first) == 0
            c.sync()
            check(first)
        graph.close()


@pytest.mark.parametrize("long", [8000, 0])
def test_a_capture_takes_a_route_whose_memory_is_there(mfa, oracle, long):
    """A chunk of few rows behind 2137 positions is the split-K kernel's, whose workspace grows with the tokens: captured
    on a context that has not made room for it (the chunk before, behind another length, took another kernel, or none was
    before), it takes a route that needs none."""
    from moeflux_amd.hip import DeviceArray
    Hq, Hkv, d, T, L0 = 16, 1, 64, 145, 2137
    q, g, k, v = _inputs(oracle, Hq, Hkv, d, T, max(L0, long), 7)
    ref = oracle.prefill_attn(T, L0, Hq, Hkv, d, q, g, k[:L0 + T], v[:L0 + T]).reshape(T, Hq * d)
    dq, dg, dk, dv = (DeviceArray.from_host(x) for x in (q, g, k[L0:L0 + T], v[L0:L0 + T]))
    out = DeviceArray((T, Hq * d), zero=True)
    with _ctx(mfa, Hq, Hkv, d, max(L0, long) + T) as c:
        assert c.lib.mfa_debug_chunk_route(1, Hq, Hkv, d, T, L0 + T, 256, 0) == 0
        assert c.lib.mfa_debug_chunk_route(1, Hq, Hkv, d, T, 8000 + T, 256, 0) > 1

        def call():
            return c.lib.mfa_prefill_attn_dev(c.h, 0, T, dq.ptr, dg.ptr, dk.ptr, dv.ptr, out.ptr)

        if long:
            c.kv_import(0, k[:long], v[:long])
            assert call() == 0
            c.sync()
            c.memory_clear()
        c.kv_import(0, k[:L0], v[:L0])
        graph = _Graph(c, call)
        for _ in range(3):
            graph()
            assert rel_err(out.to_host(), ref) <= TOL
            c.memory_seq_rm(L0)
            assert call() == 0      # eagerly: the split-K kernel, which makes its room
            c.sync()
            assert rel_err(out.to_host(), ref) <= TOL
            c.memory_seq_rm(L0)
        graph.close()


def test_first_split_chunk_beside_another_streams_capture(mfa, oracle):
    """A context's first split chunk allocates its workspace: while another stream is being captured in the mode that
    holds up the whole process (hipStreamCaptureModeGlobal), neither the chunk nor that capture fails."""
    import ctypes as C

    from moeflux_amd.hip import rt
    Hq, Hkv, d, T, L0 = 16, 2, 256, 50, 1990
    q, g, k, v = _inputs(oracle, Hq, Hkv, d, T, L0, 9)
    ref = oracle.prefill_attn(T, L0, Hq, Hkv, d, q, g, k, v).reshape(T, Hq * d)
    from moeflux_amd.hip import DeviceArray
    dq, dg, dk, dv = (DeviceArray.from_host(x) for x in (q, g, k[L0:], v[L0:]))
    out = DeviceArray((T, Hq * d), zero=True)
    other, graph = C.c_void_p(), C.c_void_p()
    assert rt().hipStreamCreateWithFlags(C.byref(other), C.c_uint(1)) == 0
    with _ctx(mfa, Hq, Hkv, d, L0 + T) as c:
        c.kv_import(0, k[:L0], v[:L0])
        assert c.lib.mfa_debug_chunk_route(1, Hq, Hkv, d, T, L0 + T, 256, 0) % 1000 > 1
        assert rt().hipStreamBeginCapture(other, C.c_int(0)) == 0
        rc = c.lib.mfa_prefill_attn_dev(c.h, 0, T, dq.ptr, dg.ptr, dk.ptr, dv.ptr, out.ptr)
        end = rt().hipStreamEndCapture(other, C.byref(graph))
        assert rc == 0, c.lib.mfa_last_error_string()
        assert end == 0
        c.sync()
        assert rel_err(out.to_host(), ref) <= TOL
    assert rt().hipGraphDestroy(graph) == 0 and rt().hipStreamDestroy(other) == 0
