"""GPU parity of the Gated-DeltaNet path against the CPU oracle, through the C ABI."""
import numpy as np
import pytest

from tests.util import TOL_F32, GdnCase, idx, rel_err

pytestmark = pytest.mark.gpu


def _ctx(mfa, case, num_layers=1):
    from moeflux_amd import Config
    c = mfa.Ctx(Config(num_layers=num_layers, full_attn_interval=num_layers + 1,
                       linear_num_k_heads=case.Hk, linear_num_v_heads=case.Hv,
                       linear_key_dim=case.dk, linear_value_dim=case.dv,
                       conv_kernel_size=case.K, rms_norm_eps=case.eps))
    for l in range(num_layers):
        c.set_linear_weights(l, case.conv_w, case.a_log, case.dt_bias, case.norm_w)
    return c


@pytest.mark.parametrize("Hk,Hv,dk,dv", [(16, 32, 128, 128), (16, 64, 128, 128), (2, 2, 128, 128),
                                          (4, 8, 64, 64), (1, 3, 128, 128)])
def test_gdn_step_matches_oracle(mfa, Hk, Hv, dk, dv):
    case = GdnCase(5 + Hv, Hk, Hv, dk, dv, T=6)
    ref_out, ref_conv, ref_ssm = case.oracle()
    with _ctx(mfa, case) as c:
        c.linear_state_import(0, case.conv_state, case.ssm_state)
        for t in range(case.T):
            out = c.gdn_step(0, case.qkv[t], case.z[t], case.alpha[t], case.beta[t])
            assert rel_err(out, ref_out[t]) <= TOL_F32, f"step {t}"
        conv, ssm = c.linear_state_export(0)
    assert np.array_equal(conv.reshape(-1), ref_conv)  # the history is copied, never computed
    assert rel_err(ssm, ref_ssm) <= TOL_F32


def test_config2_from_zero_state_and_prefill(mfa):
    """The 16 / 32-head, dk = dv = 128 step shape with A_log = dt_bias = 0 and unit norm weight; the
    chunk call equals the token loop."""
    case = GdnCase(0xC0FFEE + 2, 16, 32, 128, 128, T=9, zero_state=True, plain=True)
    ref_out, ref_conv, ref_ssm = case.oracle()
    with _ctx(mfa, case, num_layers=2) as c:
        out = c.prefill_gdn(1, case.qkv, case.z, case.alpha, case.beta)
        conv, ssm = c.linear_state_export(1)
        conv0, ssm0 = c.linear_state_export(0)
    assert rel_err(out, ref_out) <= TOL_F32
    assert np.array_equal(conv.reshape(-1), ref_conv)
    assert rel_err(ssm, ref_ssm) <= TOL_F32
    assert not conv0.any() and not ssm0.any()  # the other layer is untouched


def test_gdn_kernel_hooks(mfa, oracle):
    """The five reference kernels one at a time (inputs of tests/diff_oracle.rs:2091-2260)."""
    Hk, Hv, dk, dv, K = 16, 32, 128, 128, 4
    case = GdnCase(3, Hk, Hv, dk, dv)
    C = case.C
    state = (np.sin(0.013 * idx(3 * C)) * 0.4 + 0.02).astype(np.float32)
    x = (np.cos(0.019 * idx(C)) * 0.5 - 0.1).astype(np.float32)
    out, rolled = mfa.conv1d_step(state, x, case.conv_w, C, K)
    assert rel_err(out, oracle.conv1d_step(state, x, case.conv_w, C, K)) <= TOL_F32
    assert np.array_equal(rolled, oracle.conv_state_shift(state, x, C, K))

    q = (np.sin(0.011 * idx(Hk * dk)) * 0.4 + 0.05).astype(np.float32)
    k = (np.cos(0.019 * idx(Hk * dk)) * 0.5 - 0.1).astype(np.float32)
    v = (np.sin(0.023 * idx(Hv * dv)) * 0.6 + 0.02).astype(np.float32)
    qn, kn = mfa.rms_norm_qk(Hk, dk, q, k)
    qr, kr = oracle.rms_norm_qk(Hk, dk, q, k)
    assert rel_err(qn, qr) <= TOL_F32 and rel_err(kn, kr) <= TOL_F32

    xb = (np.sin(0.011 * idx(128)) * 0.6 + 0.05).astype(np.float32)
    zb = (np.cos(0.017 * idx(128)) * 1.2 - 0.1).astype(np.float32)
    assert rel_err(mfa.rms_norm_bare_cpu(xb, 1e-6), oracle.rms_norm_bare(xb, 1e-6)) <= TOL_F32
    assert rel_err(mfa.rms_norm_gated_cpu(xb, zb, case.norm_w, 1e-6),
                   oracle.rms_norm_gated(xb, zb, case.norm_w, 1e-6)) <= TOL_F32

    alpha = (np.sin(0.013 * idx(Hv)) * 0.3).astype(np.float32)
    beta = (np.cos(0.017 * idx(Hv)) * 0.5).astype(np.float32)
    g, b = mfa.compute_decay_beta(alpha, beta, case.a_log, case.dt_bias)
    gr, br = oracle.decay_beta(alpha, beta, case.a_log, case.dt_bias)
    assert rel_err(g, gr) <= TOL_F32 and rel_err(b, br) <= TOL_F32

    s1, o1 = mfa.gated_delta_net_step(Hv, Hk, dk, dv, gr, br, qr, kr, v, case.ssm_state)
    s2, o2 = oracle.delta_net_step(Hv, Hk, dk, dv, gr, br, qr, kr, v, case.ssm_state)
    assert rel_err(o1, o2) <= TOL_F32 and rel_err(s1, s2) <= TOL_F32

    zero = np.zeros_like(case.ssm_state)  # the reference's test starts from a zero state
    s1, o1 = mfa.gated_delta_recurrence_cpu(case.a_log, case.dt_bias, alpha, beta, qr, kr, v, Hv,
                                            Hk, dk, dv, zero)
    s2, o2 = oracle.gated_delta_recurrence(case.a_log, case.dt_bias, alpha, beta, qr, kr, v, Hv,
                                           Hk, dk, dv, zero)
    assert rel_err(o1, o2) <= TOL_F32 and rel_err(s1, s2) <= TOL_F32

    z = case.z[0]
    y1 = mfa.gated_rms_norm(Hv, dv, 1e-6, o2, z, case.norm_w)
    y2 = np.concatenate([oracle.rms_norm_gated(o2[h * dv:(h + 1) * dv], z[h * dv:(h + 1) * dv],
                                               case.norm_w, 1e-6) for h in range(Hv)])
    assert rel_err(y1, y2) <= TOL_F32


@pytest.mark.parametrize("T", [2, 3, 4, 5, 37, 47, 48, 64, 65, 100, 200])
def test_chunk_equals_token_loop(mfa, T):
    """The chunk kernels do, token for token, the operations of the single-step kernel
    (riir/mod.rs:1196-1214: a prompt is a loop of steps) and differ from it only in f32
    rounding: below 48 tokens in how a state row's dot products are grouped over lanes, from
    48 tokens on by the blocked form of the recurrence.  The conv history is copied and must
    be identical.  T below, at and above the conv width exercises the history ring on both
    sides of the chunk boundary; 47/48 and 64/65 the switch of algorithm and a block edge."""
    case = GdnCase(40 + T, 4, 8, 128, 128, T=T)
    with _ctx(mfa, case, num_layers=2) as c:
        for layer in (0, 1):
            c.linear_state_import(layer, case.conv_state, case.ssm_state)
        chunk = c.prefill_gdn(0, case.qkv, case.z, case.alpha, case.beta)
        loop = np.stack([c.gdn_step(1, case.qkv[t], case.z[t], case.alpha[t], case.beta[t])
                         for t in range(T)])
        s0, s1 = c.linear_state_export(0), c.linear_state_export(1)
        # a further single step continues correctly from the chunk's ring and state
        extra = GdnCase(99, 4, 8, 128, 128, T=1)
        n0 = c.gdn_step(0, extra.qkv[0], extra.z[0], extra.alpha[0], extra.beta[0])
        n1 = c.gdn_step(1, extra.qkv[0], extra.z[0], extra.alpha[0], extra.beta[0])
    tol = 2e-6 if T < 48 else TOL_F32
    assert rel_err(chunk, loop) <= tol
    assert np.array_equal(s0[0], s1[0]) and rel_err(s0[1], s1[1]) <= tol
    assert rel_err(n0, n1) <= tol
    ref_out, ref_conv, ref_ssm = case.oracle()
    assert rel_err(chunk, ref_out) <= TOL_F32
    assert np.array_equal(s0[0].reshape(-1), ref_conv) and rel_err(s0[1], ref_ssm) <= TOL_F32


@pytest.mark.parametrize("T", [50, 64, 129])
def test_chunk_blocked_form_dk64(mfa, T):
    """Chunks of 48 tokens and more take the blocked form (64-token blocks on the matrix
    cores); here at the 64-wide head shape, from a non-zero state, with a ragged last block."""
    case = GdnCase(70 + T, 2, 4, 64, 64, T=T)
    ref_out, ref_conv, ref_ssm = case.oracle()
    with _ctx(mfa, case) as c:
        c.linear_state_import(0, case.conv_state, case.ssm_state)
        out = c.prefill_gdn(0, case.qkv, case.z, case.alpha, case.beta)
        conv, ssm = c.linear_state_export(0)
    assert rel_err(out, ref_out) <= TOL_F32
    assert np.array_equal(conv.reshape(-1), ref_conv)
    assert rel_err(ssm, ref_ssm) <= TOL_F32


def test_config4_gdn_chunk_of_512_from_zero_state(mfa):
    """The DeltaNet half of the 512-token prompt chunk: 512 tokens of the 16 / 32-head step shape from a zero state,
    against 512 sequential oracle steps; outputs and the final state."""
    case = GdnCase(0xC0FFEE + 4, 16, 32, 128, 128, T=512, zero_state=True)
    ref_out, ref_conv, ref_ssm = case.oracle()
    with _ctx(mfa, case) as c:
        out = c.prefill_gdn(0, case.qkv, case.z, case.alpha, case.beta)
        conv, ssm = c.linear_state_export(0)
    assert rel_err(out, ref_out) <= TOL_F32
    worst = max(rel_err(out[t], ref_out[t]) for t in range(0, 512, 37))
    assert worst <= 5e-5
    assert np.array_equal(conv.reshape(-1), ref_conv)
    assert rel_err(ssm, ref_ssm) <= TOL_F32


def _same_tokens(c):
    c.qkv[:] = c.qkv[0]


def _same_tokens_beta_one(c):
    c.qkv[:] = c.qkv[0]
    c.beta[:] = 20.0
    c.alpha[:] = -20.0


def _drift(c):
    d = np.random.default_rng(1).standard_normal(c.qkv.shape).astype(np.float32) * 0.02
    c.qkv[:] = c.qkv[0] + np.cumsum(d, axis=0)


def _strong_decay(c):
    c.alpha[:] = 8.0
    c.a_log[:] = 1.5


def _big(c):
    c.qkv *= 30.0


@pytest.mark.parametrize("mutate", [_same_tokens, _same_tokens_beta_one, _drift, _strong_decay, _big],
                         ids=["identical-tokens", "identical-tokens-beta1-g1", "drifting-tokens", "strong-decay",
                              "inputs-x30"])
def test_blocked_form_on_hard_inputs(mfa, mutate):
    """The blocked form inverts I + A per 64-token block, A built from key-key products: keys that
    repeat or drift slowly make A dense with entries near beta, gates at their extremes stretch the
    decay factors (e^{L_C} underflows under strong decay).  Same criterion as everywhere."""
    case = GdnCase(5, 2, 4, 128, 128, T=256)
    mutate(case)
    ref_out, ref_conv, ref_ssm = case.oracle()
    with _ctx(mfa, case) as c:
        c.linear_state_import(0, case.conv_state, case.ssm_state)
        out = c.prefill_gdn(0, case.qkv, case.z, case.alpha, case.beta)
        conv, ssm = c.linear_state_export(0)
    assert np.isfinite(out).all()
    assert rel_err(out, ref_out) <= TOL_F32 and rel_err(ssm, ref_ssm) <= TOL_F32
    assert np.array_equal(conv.reshape(-1), ref_conv)


def _run(mfa, case, state=None):
    """(out [T, Hv, dv], conv history, state [Hv dv, dk]) of the chunk call."""
    with _ctx(mfa, case) as c:
        c.linear_state_import(0, case.conv_state, case.ssm_state if state is None else state)
        out = c.prefill_gdn(0, case.qkv, case.z, case.alpha, case.beta)
        conv, ssm = c.linear_state_export(0)
    return out.reshape(case.T, case.Hv, case.dv), conv.reshape(-1), ssm.reshape(case.Hv * case.dv, case.dk)


def _own_scale_err(a, b, row_len):
    """Worst max|a_row - b_row| / max|b_row| over the rows, however small a row is; rows of zeros have to be zeros."""
    a, b = (np.asarray(x, np.float64).reshape(-1, row_len) for x in (a, b))
    top = np.abs(b).max(axis=1)
    assert not a[top == 0].any()
    return float((np.abs(a - b).max(axis=1)[top > 0] / top[top > 0]).max())


@pytest.mark.parametrize("dk,Hk,Hv,K,T", [(128, 2, 4, 4, 48), (128, 1, 3, 3, 65), (64, 2, 2, 4, 128), (64, 1, 4, 2, 200)])
def test_blocked_form_keeps_each_row_of_the_state_to_its_own_scale(mfa, dk, Hk, Hv, K, T):
    """A row of the state and of the values is independent of the others, so each is held to TOL_F32 of its own largest
    value: rows from 2^-60 to 2^60 side by side, one of 2^-100 (the smallest whose three bf16 parts are all exact is 2^-102),
    one of 2^80 and a row of zeros with no input.  A row that holds NaN or
    infinity changes no bit of any other row of the state and leaves the other heads' outputs as they were."""
    case = GdnCase(900 + T, Hk, Hv, dk, dk, K=K, T=T)
    rng = np.random.default_rng(T)
    scale = np.exp2(rng.integers(-60, 61, Hv * dk)).astype(np.float32)
    scale[1], scale[dk + 17], scale[2 * dk - 1] = 0.0, 2.0 ** -100, 2.0 ** 80
    v0 = 2 * Hk * dk                      # SiLU is linear for the small rows and the identity for the large ones
    case.qkv[:, v0:] = np.abs(case.qkv[:, v0:]) * scale
    case.conv_w = case.conv_w.copy()
    case.conv_w.reshape(case.C, K)[v0:] &= 0x7fff
    case.conv_state = np.abs(case.conv_state)
    case.conv_state.reshape(K - 1, case.C)[:, v0:] *= scale
    case.ssm_state = (case.ssm_state.reshape(Hv * dk, dk) * scale[:, None]).reshape(-1)
    _, ref_conv, ref_ssm = case.oracle()

    out, conv, ssm = _run(mfa, case)
    assert np.array_equal(conv, ref_conv)
    assert np.isfinite(ssm).all() and not ssm[1].any()
    assert _own_scale_err(ssm, ref_ssm, dk) <= TOL_F32
    for bad in (np.nan, np.inf):
        state = case.ssm_state.copy()
        row = dk + 5                      # a row of head 1
        state[row * dk + 7] = bad
        out2, _, ssm2 = _run(mfa, case, state)
        rows = np.arange(Hv * dk) != row
        assert not np.isfinite(ssm2[row]).all()
        assert np.array_equal(ssm2[rows], ssm[rows])
        heads = np.arange(Hv) != 1
        assert np.array_equal(out2[:, heads], out[:, heads])


@pytest.mark.parametrize("dk,Hk,Hv,K,at", [(128, 2, 4, 4, 40), (128, 1, 3, 3, 27), (64, 2, 2, 4, 124)])
@pytest.mark.parametrize("part", ["q", "k", "v"])
@pytest.mark.parametrize("factor", [1e8, 1e13, np.inf, np.nan])
def test_blocked_form_earlier_tokens_do_not_see_later_ones(mfa, dk, Hk, Hv, K, at, part, factor):
    """One token whose q, k or v is 1e8 or 1e13 times the others', infinite or NaN, in the first block and late in the
    second: what comes before it is the same bits.  (A product of 16 x 16 tiles multiplies the tokens ahead of a tile's
    last by zeros, so a token that is not finite may reach the others of its own 16.)  A token's q is no other's business."""
    case = GdnCase(500 + at + dk + K, Hk, Hv, dk, dk, K=K, T=150)
    clean, _, _ = _run(mfa, case)
    first = {"q": 0, "k": Hk * dk, "v": 2 * Hk * dk}[part]
    last = {"q": Hk * dk, "k": 2 * Hk * dk, "v": case.C}[part]
    case.qkv[at, first:last] *= np.float32(factor)
    out, _, ssm = _run(mfa, case)
    before = at if np.isfinite(factor) else at // 16 * 16
    assert np.array_equal(out[:before], clean[:before])
    if part == "q":
        assert np.array_equal(out[at + K:], clean[at + K:])
    if np.isfinite(factor):
        ref_out, _, ref_ssm = case.oracle()
        assert rel_err(out, ref_out) <= TOL_F32 and rel_err(ssm, ref_ssm) <= TOL_F32
    else:
        assert not np.isfinite(out[at]).all(axis=1).any()


@pytest.mark.parametrize("dk,K,T", [(128, 4, 64), (128, 3, 64), (64, 4, 130), (128, 4, 256)])
@pytest.mark.parametrize("logit", [-8.0, -16.0, -20.0, -40.0, -60.0])
def test_blocked_form_of_barely_open_gates(mfa, dk, K, T, logit):
    """beta of 3e-4 down to 9e-27 into an empty state under a decay of 0.99: T diag(beta) and W are as small as beta, and
    state and outputs are held to their own size."""
    case = GdnCase(11, 2, 4, dk, dk, K=K, T=T, zero_state=True, plain=True)
    case.alpha[:] = -4.6
    case.beta[:] = logit
    ref_out, _, ref_ssm = case.oracle()
    out, _, ssm = _run(mfa, case)
    assert _own_scale_err(ssm, ref_ssm, dk) <= TOL_F32
    assert _own_scale_err(out, ref_out, dk) <= TOL_F32


@pytest.mark.parametrize("dk,K,T,alpha", [(128, 4, 64, -0.846), (128, 3, 65, 0.0), (64, 4, 130, -0.846), (128, 4, 200, -0.846)])
def test_blocked_form_of_a_state_that_only_decays(mfa, dk, K, T, alpha):
    """No values at all, beta = 0.5 and a decay of 0.7 or 0.5 a token: what is left of the state after the chunk, 1e-10 to 1e-32
    of what it was, and the outputs read from it on the way keep their precision.  The decay, the same for every token, is
    rounded by up to 2^-24 in the oracle and its logarithm as much here: T 2^-23 beside the usual bar."""
    tol = TOL_F32 + T * 2.0 ** -23
    case = GdnCase(12, 2, 4, dk, dk, K=K, T=T, plain=True)
    v0 = 4 * dk
    case.qkv[:, v0:] = 0.0
    case.conv_state.reshape(K - 1, case.C)[:, v0:] = 0.0
    case.alpha[:] = alpha
    case.beta[:] = 0.0
    ref_out, _, ref_ssm = case.oracle()
    out, _, ssm = _run(mfa, case)
    assert _own_scale_err(ssm, ref_ssm, dk) <= tol
    assert _own_scale_err(out, ref_out, dk) <= tol


@pytest.mark.parametrize("dk,K,T", [(128, 4, 64), (128, 3, 65), (64, 4, 130), (128, 4, 200)])
def test_blocked_form_of_tokens_and_channels_of_every_size(mfa, dk, K, T):
    """Values whose size changes by up to 2^24 from token to token under a decay of 0.5, and key channels of 2^-30 to 1: outputs
    are held to their own row's size, the state's columns (a key channel each) to theirs.  The decay's logarithm runs up to
    -45 in a block, in six additions that round by up to 2^-19 each, and a factor is e to the difference of two such sums:
    2.3e-5 beside the usual bar."""
    tol = TOL_F32 + 12 * 2.0 ** -19
    case = GdnCase(13 + T, 2, 4, dk, dk, K=K, T=T, plain=True)
    rng = np.random.default_rng(T)
    v0, k0 = 4 * dk, 2 * dk
    case.qkv[:, v0:] *= np.exp2(rng.integers(-12, 13, T)).astype(np.float32)[:, None]
    case.alpha[:] = 0.0
    col = np.exp2(rng.integers(-30, 1, 2 * dk)).astype(np.float32)
    case.qkv[:, k0:v0] *= col
    case.conv_state.reshape(K - 1, case.C)[:, k0:v0] *= col
    state = case.ssm_state.reshape(2, 2, dk, dk)
    state *= col.reshape(2, 1, 1, dk)
    ref_out, _, ref_ssm = case.oracle()
    out, _, ssm = _run(mfa, case)
    cols = lambda s: s.reshape(4, dk, dk).transpose(0, 2, 1)  # noqa: E731
    assert _own_scale_err(cols(ssm), cols(ref_ssm), dk) <= tol
    assert _own_scale_err(out, ref_out, dk) <= tol


def test_chunk_at_the_a17b_head_counts(mfa):
    """16 key heads, 64 value heads (variants.rs:396-397), a ragged 130-token chunk."""
    case = GdnCase(6, 16, 64, 128, 128, T=130)
    ref_out, ref_conv, ref_ssm = case.oracle()
    with _ctx(mfa, case) as c:
        c.linear_state_import(0, case.conv_state, case.ssm_state)
        out = c.prefill_gdn(0, case.qkv, case.z, case.alpha, case.beta)
        _, ssm = c.linear_state_export(0)
    assert rel_err(out, ref_out) <= TOL_F32 and rel_err(ssm, ref_ssm) <= TOL_F32


@pytest.mark.parametrize("K", [4, 3])
@pytest.mark.parametrize("T", [256, 257, 385])
def test_blocked_form_at_and_past_a_workgroup_per_cu(mfa, K, T):
    """64 heads of 128 channels: four blocks are a workgroup of the block precompute per CU, from five on a CU has more than
    one; with the conv inside it (width 4) and ahead of it."""
    case = GdnCase(60 + T + K, 16, 64, 128, 128, K=K, T=T)
    ref_out, ref_conv, ref_ssm = case.oracle()
    with _ctx(mfa, case) as c:
        c.linear_state_import(0, case.conv_state, case.ssm_state)
        out = c.prefill_gdn(0, case.qkv, case.z, case.alpha, case.beta)
        conv, ssm = c.linear_state_export(0)
    assert rel_err(out, ref_out) <= TOL_F32 and rel_err(ssm, ref_ssm) <= TOL_F32
    assert np.array_equal(conv.reshape(-1), ref_conv)


def test_prompt_longer_than_one_segment(mfa):
    """A prompt of more than 4096 tokens goes through the chunk kernels in 4096-token segments; the
    ring and the state carry from one segment to the next as they do between calls."""
    case = GdnCase(8, 2, 4, 64, 64, T=4096 + 70)
    ref_out, ref_conv, ref_ssm = case.oracle()
    with _ctx(mfa, case) as c:
        c.linear_state_import(0, case.conv_state, case.ssm_state)
        out = c.prefill_gdn(0, case.qkv, case.z, case.alpha, case.beta)
        conv, ssm = c.linear_state_export(0)
    assert rel_err(out, ref_out) <= TOL_F32 and rel_err(ssm, ref_ssm) <= TOL_F32
    assert rel_err(out[4090:], ref_out[4090:]) <= 5e-5
    assert np.array_equal(conv.reshape(-1), ref_conv)


def test_random_shapes_and_conv_widths(mfa):
    """Seeded random head counts, both head widths, conv widths 2 to 8 and chunk lengths on either
    side of the switch to the blocked form: a chunk after a few single steps, against the oracle's
    sequential steps; outputs, the conv history (bit for bit) and the recurrent state."""
    rng = np.random.default_rng(77)
    shapes = [(128, 2, 4, 8, 5, 70), (64, 1, 2, 2, 0, 130), (128, 1, 1, 5, 9, 48), (64, 2, 8, 8, 17, 64)]
    for _ in range(14):
        Hk = int(rng.choice([1, 2, 4]))
        K = int(rng.choice([2, 3, 4, 5, 8]))
        shapes.append((int(rng.choice([64, 128])), Hk, Hk * int(rng.choice([1, 2, 4])), K, int(rng.integers(0, 2 * K)),
                       int(rng.choice([1, 2, 7, 40, 48, 63, 64, 65, 130]))))
    for case_no, (dk, Hk, Hv, K, pre, T) in enumerate(shapes):
        case = GdnCase(500 + case_no, Hk, Hv, dk, dk, K=K, T=pre + T)
        ref_out, ref_conv, ref_ssm = case.oracle()
        with _ctx(mfa, case) as c:
            c.linear_state_import(0, case.conv_state, case.ssm_state)
            outs = [c.gdn_step(0, case.qkv[t], case.z[t], case.alpha[t], case.beta[t]) for t in range(pre)]
            outs.extend(c.prefill_gdn(0, case.qkv[pre:], case.z[pre:], case.alpha[pre:], case.beta[pre:]))
            conv, ssm = c.linear_state_export(0)
        what = (case_no, Hk, Hv, dk, K, pre, T)
        assert rel_err(np.stack(outs), ref_out) <= TOL_F32, what
        assert np.array_equal(conv.reshape(-1), ref_conv), what
        assert rel_err(ssm, ref_ssm) <= TOL_F32, what
