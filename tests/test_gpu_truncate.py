"""Truncation over all layers at once: what is kept, what is zeroed, and layers of different lengths."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("lens,p0,p1", [((130, 130, 130), 37, -1), ((130, 130, 130), 0, 64), ((70, 129, 129), 65, -1), ((1, 96, 31), 31, 90),
                                        ((64, 64, 64), 63, -1), ((130, 0, 20), 16, -1)])
def test_truncate_keeps_the_head_and_zeroes_the_rest(mfa, oracle, bf16, lens, p0, p1):
    """Positions either side of a unit, a block and a chunk of the tiles: lengths, rows up to the new length as they were, and
    attention once a position is appended there (that the rows behind are zero: the next test)."""
    from moeflux_amd import Config
    Hq, Hkv, d, cap = 4, 2, 64, 200
    rng = np.random.default_rng(sum(lens) + p0)
    k, v = (rng.standard_normal((3, cap, Hkv * d)).astype(np.float32) for _ in range(2))
    if bf16:
        k, v = (oracle.bf16_to_f32(oracle.f32_to_bf16(a)) for a in (k, v))
    q, g = (rng.standard_normal(Hq * d).astype(np.float32) for _ in range(2))
    with mfa.Ctx(Config(num_layers=3, full_attn_interval=1, num_attn_heads=Hq, num_kv_heads=Hkv, head_dim=d, kv_capacity=cap,
                        kv_dtype=1 if bf16 else 0)) as c:
        for i, n in enumerate(lens):
            if n:
                c.kv_import(i, k[i, :n], v[i, :n])
        c.memory_seq_rm(p0, p1)
        for i, n in enumerate(lens):
            end = n if p1 < 0 else min(p1, n)
            keep = min(p0, end)
            assert c.kv_len(i) == keep
            if keep:
                ke, ve = c.kv_export(i)
                assert np.array_equal(ke, k[i, :keep]) and np.array_equal(ve, v[i, :keep])
            # the block of the next position holds zeros behind it: an attention over it is that of a fresh cache
            c.kv_append(i, k[i, keep], v[i, keep])
            out = c.sdpa_decode(i, q, g)
            assert np.isfinite(out).all()
            kk, vv = k[i, :keep + 1], v[i, :keep + 1]
            ref = oracle.sdpa(keep + 1, Hq, Hkv, d, q, g, kk, vv)
            assert np.abs(out - ref).max() <= 1e-4 * np.abs(ref).max()
        c.memory_clear()
        assert all(c.kv_len(i) == 0 for i in range(3))


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_dropped_rows_are_zero_and_no_others(mfa, oracle, d, bf16):
    """The planes themselves after a truncation, in three layers of one or several lengths: zero from the new length on, the
    rows before it as they were, and the rows of a layer that keeps more untouched (p1 ends the dropped range)."""
    from moeflux_amd import Config
    Hkv, cap = 2, 200
    rng = np.random.default_rng(d)
    k, v = (1.0 + rng.random((3, cap, Hkv * d)).astype(np.float32) for _ in range(2))   # no zero among them
    if bf16:
        k, v = (oracle.bf16_to_f32(oracle.f32_to_bf16(a)) for a in (k, v))
    for lens, p0, p1 in [((200, 200, 200), 0, -1), ((130, 130, 130), 37, -1), ((70, 129, 129), 65, -1), ((1, 96, 31), 31, 90),
                         ((64, 64, 64), 63, -1), ((130, 0, 20), 16, -1), ((200, 200, 199), 199, -1), ((100, 160, 160), 4, 128),
                         ((97, 97, 97), 19, -1), ((33, 33, 97), 32, -1)]:
        with mfa.Ctx(Config(num_layers=3, full_attn_interval=1, num_attn_heads=4, num_kv_heads=Hkv, head_dim=d, kv_capacity=cap,
                            kv_dtype=1 if bf16 else 0)) as c:
            for i, n in enumerate(lens):
                if n:
                    c.kv_import(i, k[i, :n], v[i, :n])
            c.memory_seq_rm(p0, p1)
            for i, n in enumerate(lens):
                keep = min(p0, n if p1 < 0 else min(p1, n))
                got = [np.full((cap, Hkv * d), np.nan, np.float32) for _ in range(2)]
                assert c.lib.mfa_debug_kv_export(c.h, i, cap, *(g.ctypes.data for g in got)) == 0
                for g, x in zip(got, (k, v)):
                    assert np.array_equal(g[:keep], x[i, :keep]), (lens, p0, p1, i)
                    assert not g[keep:].any(), (lens, p0, p1, i, np.argwhere(g[keep:])[:3])
