"""The work a user of this framework has it do, as cases that can be timed and compared.

A case is a dict of plain values.  `kind` names the path through the public entry points:

  step         one generated token through the full-attention layers of a stack, from the raw projections
               (per-head norms, rotation, cache append, attention, gate)
  decode       the attention core alone for one token: query already normed and rotated, cache already appended
  gdn_step     one generated token through the DeltaNet layers of a stack
  sweep        one token through every layer of a hybrid stack, all inputs handed over at once
  prompt_attn  a chunk of prompt tokens through full-attention layers, from an empty cache or behind a context
  prompt_gdn   a chunk of prompt tokens through DeltaNet layers, and the first generated token after it
  latent       one token of a latent-attention layer (multi-head latent attention, folded)
  proj         the 4-bit projections either side of a full-attention layer's core (q, k, v in one call, then o)

Shapes are those of bench.py, the tests and the variants they cite: 32 or 16 query heads over 2 kv heads of 256
channels, 32 over 4 of 128; 16 key heads with 32 or 64 value heads of 128 channels; 128 heads over a latent cache of
512 + 64; hidden width 4096.  Every layer has a cache, a state, weights and inputs of its own, as in a model.
"""
import ctypes as C
import math

import torch

from moeflux_amd import Config, Ctx, ffi

ROLLBACK = 256   # tokens generated behind a prompt before the cache is taken back to it


def listed():
    return [
        # The smallest call there is: a token early in a conversation, one layer; latency and launches.
        dict(name="step_short", kind="step", hq=16, hkv=2, d=256, bf16=True, length=515, layers=1),
        # Ordinary generation behind a long document.
        dict(name="step_32k", kind="step", hq=32, hkv=2, d=256, bf16=True, length=32768, layers=4),
        # The attention core over f32 caches of a mid-length conversation.
        dict(name="decode_f32_4k", kind="decode", hq=32, hkv=4, d=128, bf16=False, length=4096, layers=8),
        # The longest contexts, at a length that fills no unit of the cache.
        dict(name="decode_131k", kind="decode", hq=32, hkv=2, d=256, bf16=True, length=131009, layers=1),
        # A token through DeltaNet layers that depend on each other: one launch chain per layer.
        dict(name="gdn_step", kind="gdn_step", hk=16, hv=32, layers=9),
        # A token over the whole 48-layer stack with every layer's inputs known (independent sequences).
        dict(name="sweep_48", kind="sweep", hq=32, hkv=2, d=256, bf16=True, hk=16, hv=32, length=8192, layers=48),
        # A new prompt: memory cleared, one 512-token chunk through each layer.
        dict(name="prompt_attn_512", kind="prompt_attn", hq=32, hkv=4, d=128, bf16=True, length=0, tokens=512, layers=8),
        # A ragged chunk of a new turn behind a conversation, the wide heads.
        dict(name="prompt_attn_turn", kind="prompt_attn", hq=16, hkv=2, d=256, bf16=True, length=3001, tokens=203, layers=4),
        # A chunk of a very long prompt: the largest matrix work of the framework.
        dict(name="prompt_attn_behind_32k", kind="prompt_attn", hq=32, hkv=4, d=128, bf16=True, length=32768, tokens=512,
             layers=1),
        # The same 512-token chunk for the DeltaNet layers of the stack.
        dict(name="prompt_gdn_512", kind="prompt_gdn", hk=16, hv=32, tokens=512, layers=6),
        # A latent-attention layer with a long context.
        dict(name="latent_32k", kind="latent", heads=128, length=32768, layers=2),
        # The projections of a token, from weights re-ordered at load time.
        dict(name="proj_tiled", kind="proj", hidden=4096, hq=32, hkv=2, d=256, tiled=True, layers=4),
    ]


def _spread(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi], odd ones among them."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "decode", "gdn_step", "sweep", "prompt_attn", "prompt_gdn", "latent", "proj"])
    c = dict(kind=kind)
    if kind in ("step", "decode", "sweep", "prompt_attn"):
        c["hq"], c["hkv"], c["d"] = rng.choice([(32, 2, 256), (16, 2, 256), (32, 4, 128)])
        c["bf16"] = rng.random() < 0.75
    if kind in ("gdn_step", "sweep", "prompt_gdn"):
        c["hk"], c["hv"] = 16, rng.choice([32, 64])
    if kind in ("step", "decode"):
        c["length"] = _spread(rng, 1, 65536)
        c["layers"] = rng.randint(1, 4)
    elif kind == "gdn_step":
        c["layers"] = rng.randint(1, 12)
    elif kind == "sweep":
        c["layers"] = 4 * rng.randint(2, 12)
        c["length"] = _spread(rng, 64, 4096)
    elif kind == "prompt_attn":
        c["tokens"] = _spread(rng, 2, 2048)
        # the context a chunk of this size may have behind it at the cost of the largest listed case (an f32 cache: at
        # the f32 matrix rate, a sixteenth of the bf16 one, of which the bf16 path spends four)
        most = int((2.7e11 if c["bf16"] else 6.7e10) / (4 * c["hq"] * c["d"] * c["tokens"])) - c["tokens"]
        c["length"] = rng.choice([0, _spread(rng, 1, min(16384, most))]) if most > 1 else 0
        c["layers"] = 1 if c["tokens"] * (c["tokens"] + c["length"]) > 1_000_000 else rng.randint(1, 4)
    elif kind == "prompt_gdn":
        c["tokens"] = _spread(rng, 2, 4200)
        c["layers"] = 1 if c["tokens"] > 1000 else rng.randint(1, 4)
    elif kind == "latent":
        c["heads"] = rng.choice([16, 64, 128])
        c["length"] = _spread(rng, 64, 32768)
        c["layers"] = rng.randint(1, 2)
    else:
        c["hidden"] = 64 * _spread(rng, 16, 112)
        c["hq"], c["hkv"], c["d"] = rng.choice([(32, 2, 256), (16, 2, 256), (32, 4, 128)])
        c["tiled"] = rng.random() < 0.5
        c["layers"] = rng.randint(1, 4)
    return c


# ---- what a program has in hand before the call -----------------------------------------------------------------

class _State:
    """A context (closed with the state), device inputs and outputs, and the calls' arguments."""

    def __init__(self, case, seed):
        self.case, self.lib = case, ffi.load()
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)
        self.keep = []

    def randn(self, *shape, scale=1.0):
        t = torch.randn(shape, device="cuda", generator=self.gen) * scale
        self.keep.append(t)
        return t

    def empty(self, *shape):
        t = torch.zeros(shape, device="cuda")
        self.keep.append(t)
        return t


def _bits(t):
    """bf16 bit patterns of a float tensor, on the host."""
    return t.to(torch.bfloat16).view(torch.int16).cpu().numpy().view("uint16")


def _check(rc):
    if rc != 0:
        raise RuntimeError(ffi.last_error())


def _attention_layer(s):
    """Norm weights [2, d] (bf16) of a full-attention layer and the keys and values its cache holds, [2, length, hkv * d]
    in the cache's type (None where it is empty): keys of unit variance per channel, as a per-head norm leaves them, and
    values of unit variance."""
    c = s.case
    norm = (1.0 + 0.1 * torch.randn(2, c["d"], device="cuda", generator=s.gen)).to(torch.bfloat16)
    if not c["length"]:
        return norm, None
    kv = torch.randn(2, c["length"], c["hkv"] * c["d"], device="cuda", generator=s.gen)
    return norm, kv.to(torch.bfloat16) if c["bf16"] else kv


def _attention(s, layers, length, capacity, interval=1):
    """A context of `layers` layers whose full-attention caches hold `length` positions."""
    c = s.case
    lin = {} if interval == 1 else dict(linear_num_k_heads=c["hk"], linear_num_v_heads=c["hv"])
    s.ctx = Ctx(Config(num_layers=layers, full_attn_interval=interval, num_attn_heads=c["hq"], num_kv_heads=c["hkv"],
                       head_dim=c["d"], kv_capacity=capacity, kv_dtype=ffi.KV_BF16 if c["bf16"] else ffi.KV_F32, **lin))
    for layer in range(layers):
        if (layer + 1) % interval:
            continue
        norm, kv = _attention_layer(s)
        norm = _bits(norm)
        s.ctx.set_full_weights(layer, norm[0], norm[1])
        if length:
            kv = _bits(kv) if c["bf16"] else kv.cpu().numpy()
            s.ctx.kv_import(layer, kv[0], kv[1])


def _deltanet_layer(s):
    """conv weights, A_log, dt bias, norm weights, conv history and recurrent state of a DeltaNet layer."""
    hv, conv = s.case["hv"], (2 * s.case["hk"] + s.case["hv"]) * 128
    rnd = lambda *n: torch.randn(*n, device="cuda", generator=s.gen)  # noqa: E731
    bf = torch.bfloat16
    return ((0.5 * rnd(conv, 4)).to(bf), 0.5 * rnd(hv), (0.5 * rnd(hv)).to(bf), (1.0 + 0.2 * rnd(128)).to(bf),
            rnd(3, conv), 0.02 * rnd(hv * 128 * 128))


def _deltanet(s, layers):
    """Weights and states of the DeltaNet layers `layers` of the state's context."""
    for layer in layers:
        conv_w, a_log, dt_bias, norm, history, state = _deltanet_layer(s)
        s.ctx.set_linear_weights(layer, _bits(conv_w), a_log.cpu().numpy(), _bits(dt_bias), _bits(norm))
        s.ctx.linear_state_import(layer, history.cpu().numpy(), state.cpu().numpy())


def _deltanet_inputs(s, layers, tokens):
    hv, n = s.case["hv"], layers * tokens
    return (s.randn(n, (2 * s.case["hk"] + hv) * 128), s.randn(n, hv * 128), s.randn(n, hv), s.randn(n, hv), s.empty(n, hv * 128))


def _weights(s, out_dim, in_dim):
    """4-bit weights: nibbles of all values, group scales and biases (bf16) that give weights of about 1 / sqrt(in_dim)."""
    w = torch.randint(-2 ** 31, 2 ** 31, (out_dim, in_dim // 8), device="cuda", generator=s.gen, dtype=torch.int64).to(torch.int32)
    scale = 0.2 / math.sqrt(in_dim) * (0.5 + torch.rand(out_dim, in_dim // 64, device="cuda", generator=s.gen))
    return w, scale.to(torch.bfloat16), (-7.5 * scale).to(torch.bfloat16)


def _projection(s, out_dim, in_dim, x, out):
    """A spec of one 4-bit product."""
    w, scale, bias = _weights(s, out_dim, in_dim)
    if s.case["tiled"]:
        t = torch.empty(int(s.lib.mfa_matvec_tiled_words(out_dim, in_dim)), device="cuda", dtype=torch.int32)
        _check(s.lib.mfa_matvec_tile_weights_dev(s.ctx.h, out_dim, in_dim, w.data_ptr(), scale.data_ptr(), bias.data_ptr(),
                                                 t.data_ptr()))
        s.ctx.sync()
        s.keep.append(t)
        return ffi.mfa_matvec_spec(t.data_ptr(), None, None, x.data_ptr(), out.data_ptr(), out_dim, in_dim)
    s.keep += [w, scale, bias]
    return ffi.mfa_matvec_spec(w.data_ptr(), scale.data_ptr(), bias.data_ptr(), x.data_ptr(), out.data_ptr(), out_dim, in_dim)


def _plain_ctx():
    """A context for the calls that need its stream and workspace only."""
    return Ctx(Config(num_layers=1, full_attn_interval=1, num_attn_heads=8, num_kv_heads=2, head_dim=64, kv_capacity=4))


def prepare(case, seed):
    s = _State(case, seed)
    kind, n = case["kind"], case["layers"]
    if kind in ("step", "decode", "prompt_attn"):
        qd, kd = case["hq"] * case["d"], case["hkv"] * case["d"]
        t = case.get("tokens", 1)
        room = {"step": ROLLBACK, "decode": 0, "prompt_attn": t}[kind]
        _attention(s, n, case["length"], case["length"] + room)
        if kind == "decode":
            s.q, s.gate = s.randn(n, qd), s.randn(n, qd)
            s.out = s.empty(n, qd)
            s.args = [(s.ctx.h, i, s.q[i].data_ptr(), s.gate[i].data_ptr(), s.out[i].data_ptr()) for i in range(n)]
        else:
            s.qp, s.k, s.v = s.randn(n, t, 2 * qd), s.randn(n, t, kd), s.randn(n, t, kd)
            s.out = s.empty(n, t, qd)
            s.args = [(s.qp[i].data_ptr(), s.k[i].data_ptr(), s.v[i].data_ptr(), s.out[i].data_ptr()) for i in range(n)]
            s.pos = case["length"]
    elif kind in ("gdn_step", "prompt_gdn"):
        s.ctx = Ctx(Config(num_layers=n, full_attn_interval=n + 1, linear_num_k_heads=case["hk"], linear_num_v_heads=case["hv"]))
        _deltanet(s, range(n))
        s.inputs = _deltanet_inputs(s, n, case.get("tokens", 1))
        s.args = _per_layer(s.inputs, n)
        if kind == "prompt_gdn":
            s.first = _deltanet_inputs(s, n, 1)
            s.first_args = _per_layer(s.first, n)
    elif kind == "sweep":
        full = n // 4
        _attention(s, n, case["length"], case["length"], interval=4)
        _deltanet(s, [i for i in range(n) if (i + 1) % 4])
        s.q, s.gate, s.out = s.randn(full, case["hq"] * case["d"]), s.randn(full, case["hq"] * case["d"]), s.empty(full, case["hq"] * case["d"])
        s.inputs = _deltanet_inputs(s, n - full, 1)
        s.args = (s.ctx.h, s.q.data_ptr(), s.gate.data_ptr(), s.out.data_ptr()) + tuple(t.data_ptr() for t in s.inputs)
    elif kind == "latent":
        s.ctx = _plain_ctx()
        h, length = case["heads"], case["length"]
        s.q, s.qe = s.randn(n, h, 512), s.randn(n, h, 64)
        s.latent, s.rope = s.randn(n, length, 512), s.randn(n, length, 64)
        s.out = s.empty(n, h, 512)
        s.args = [(s.ctx.h, h, 512, 64, length, 1.0 / math.sqrt(576.0), s.q[i].data_ptr(), s.qe[i].data_ptr(), s.latent[i].data_ptr(),
                   s.rope[i].data_ptr(), s.out[i].data_ptr()) for i in range(n)]
    else:
        s.ctx = _plain_ctx()
        s.args, s.out = [], []
        qd, kd, hidden = case["hq"] * case["d"], case["hkv"] * case["d"], case["hidden"]
        for _ in range(n):
            x, core = s.randn(hidden), s.randn(qd)
            outs = [s.empty(m) for m in (2 * qd, kd, kd, hidden)]
            s.out.append(outs)
            qkv = (ffi.mfa_matvec_spec * 3)(*[_projection(s, o.numel(), hidden, x, o) for o in outs[:3]])
            o = (ffi.mfa_matvec_spec * 1)(_projection(s, hidden, qd, core, outs[3]))
            s.keep += [qkv, o]
            s.args += [(s.ctx.h, 3, C.byref(qkv)), (s.ctx.h, 1, C.byref(o))]
    torch.cuda.synchronize()
    return s


def _per_layer(tensors, n):
    """data pointers of each layer's slice of [layers * tokens, ...] tensors."""
    return [tuple(t[i * (t.shape[0] // n)].data_ptr() for t in tensors) for i in range(n)]


# ---- one pass -----------------------------------------------------------------------------------------------------

def run(s):
    lib, kind = s.lib, s.case["kind"]
    if kind == "step":
        # the positions of a token: one on from the last; after ROLLBACK tokens the conversation is taken back to its prompt
        if s.pos == s.case["length"] + ROLLBACK:
            s.pos = s.case["length"]
            s.ctx.memory_seq_rm(s.pos)
        for layer, (qp, k, v, out) in enumerate(s.args):
            _check(lib.mfa_full_attn_step_dev(s.ctx.h, layer, s.pos, qp, k, v, out))
        s.pos += 1
        return s.out
    if kind == "decode":
        for a in s.args:
            _check(lib.mfa_sdpa_decode_dev(*a))
        return s.out
    if kind == "gdn_step":
        for layer, a in enumerate(s.args):
            _check(lib.mfa_gdn_step_dev(s.ctx.h, layer, *a))
        return s.inputs[4]
    if kind == "sweep":
        _check(lib.mfa_token_sweep_dev(*s.args))
        return s.out, s.inputs[4]
    if kind == "prompt_attn":
        if s.case["length"]:
            s.ctx.memory_seq_rm(s.case["length"])
        else:
            s.ctx.memory_clear()
        for layer, (qp, k, v, out) in enumerate(s.args):
            _check(lib.mfa_prefill_full_attn_dev(s.ctx.h, layer, s.pos, s.case["tokens"], qp, k, v, out))
        return s.out
    if kind == "prompt_gdn":
        # the layers go on from the state they hold; the first generated token shows what the chunk left in it
        for layer, a in enumerate(s.args):
            _check(lib.mfa_prefill_gdn_dev(s.ctx.h, layer, s.case["tokens"], *a))
        for layer, a in enumerate(s.first_args):
            _check(lib.mfa_gdn_step_dev(s.ctx.h, layer, *a))
        return s.inputs[4], s.first[4]
    if kind == "latent":
        for a in s.args:
            _check(lib.mfa_mla_sdpa_folded_dev(*a))
        return s.out
    call = lib.mfa_dequant_matvec_4bit_tiled_dev if s.case["tiled"] else lib.mfa_dequant_matvec_4bit_dev
    for a in s.args:
        _check(call(*a))
    return s.out


# ---- the same outputs in 64 bits ------------------------------------------------------------------------------------
# The inputs are drawn again, in prepare's order.  A cache holds keys and values in its own type, so appended rows are
# rounded to it here too; all else is float64.

def _rotate(x, pos):
    """Rotation of the first quarter of the channels of [tokens, heads, d] at positions pos (base 1e7)."""
    half = x.shape[2] // 8
    angle = pos.double()[:, None] * 1e7 ** (-torch.arange(half, device="cuda", dtype=torch.float64) / half)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]
    a, b = x[..., :half], x[..., half:2 * half]
    return torch.cat([a * cos - b * sin, b * cos + a * sin, x[..., 2 * half:]], 2)


def _rms(x, eps=1e-6):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _attend(q, k, v, gate, length):
    """Causal attention of tokens [t, hq, d] at positions length .. over keys and values [length + t, hkv, d]."""
    t, hq, d = q.shape
    hpk, out = hq // k.shape[1], torch.empty_like(q)
    hidden = torch.arange(k.shape[0], device="cuda")[None, :] > length + torch.arange(t, device="cuda")[:, None]
    for h in range(hq):
        scores = q[:, h] @ k[:, h // hpk].T / math.sqrt(d)
        out[:, h] = scores.masked_fill_(hidden, -math.inf).softmax(1) @ v[:, h // hpk]
    return (out * gate.sigmoid()).reshape(t, hq * d)


def _exact_layers(s, cached, qp, k, v):
    """Attention layers from the raw projections: [layers, tokens, hq * d]."""
    c, kept = s.case, torch.bfloat16 if s.case["bf16"] else torch.float32
    t, outs = qp.shape[1], []
    for layer, (norm, kv) in enumerate(cached):
        pos, norm = c["length"] + torch.arange(t, device="cuda"), norm.double()
        split = qp[layer].double().view(t, c["hq"], 2, c["d"])
        q = _rotate(_rms(split[:, :, 0]) * norm[0], pos)
        rows = (_rotate(_rms(k[layer].double().view(t, c["hkv"], c["d"])) * norm[1], pos), v[layer].view(t, c["hkv"], c["d"]))
        keys, values = (torch.cat(([kv[i].double().view(-1, c["hkv"], c["d"])] if kv is not None else []) + [r.to(kept).double()])
                        for i, r in enumerate(rows))
        outs.append(_attend(q, keys, values, split[:, :, 1], c["length"]))
    return torch.stack(outs)


def _exact_deltanet(s, layers, *chunks):
    """Chunks of inputs, one after the other, through DeltaNet layers `layers` = [_deltanet_layer(s), ...] together:
    outputs [layers * tokens, hv * 128] of each chunk."""
    n, hk, hv = len(layers), s.case["hk"], s.case["hv"]
    conv_w, a_log, dt_bias, norm, history, state = (torch.stack([x[i].double() for x in layers]) for i in range(6))
    state, outs = state.view(n, hv, 128, 128), []   # [layer, head, value channel, key channel]
    for qkv, z, alpha, beta, _ in chunks:
        t = qkv.shape[0] // n
        seen = torch.cat([history, qkv.double().view(n, t, -1)], 1)
        history = seen[:, -3:]
        y = sum(seen[:, i:i + t] * conv_w[:, None, :, i] for i in range(4))
        y = y * y.sigmoid()
        q, k = (_rms(y[..., i * hk * 128:(i + 1) * hk * 128].view(n, t, hk, 128)).repeat_interleave(hv // hk, 2) for i in range(2))
        q, k, v = q / 128.0, k / math.sqrt(128.0), y[..., 2 * hk * 128:].view(n, t, hv, 128)
        keep = (-a_log.exp()[:, None] * torch.log1p((alpha.double().view(n, t, hv) + dt_bias[:, None]).exp())).exp()
        rate = beta.double().view(n, t, hv).sigmoid()
        o = torch.empty_like(v)
        for i in range(t):
            state = state * keep[:, i, :, None, None]
            off = rate[:, i, :, None] * (v[:, i] - (state * k[:, i, :, None]).sum(-1))
            state = state + off[..., None] * k[:, i, :, None]
            o[:, i] = (state * q[:, i, :, None]).sum(-1)
        z = z.double().view(n, t, hv, 128)
        outs.append((_rms(o) * norm[:, None, None] * z * z.sigmoid()).reshape(n * t, hv * 128))
    return outs


def _exact_weights(s, out_dim, in_dim):
    w, scale, bias = _weights(s, out_dim, in_dim)
    nibbles = torch.stack([(w >> (4 * i)) & 15 for i in range(8)], -1).view(out_dim, in_dim // 64, 64)
    return (nibbles.double() * scale.double()[..., None] + bias.double()[..., None]).view(out_dim, in_dim)


def exact(case, seed):
    s = _State(case, seed)
    kind, n = case["kind"], case["layers"]
    if kind in ("step", "decode", "prompt_attn"):
        qd, kd, t = case["hq"] * case["d"], case["hkv"] * case["d"], case.get("tokens", 1)
        cached = [_attention_layer(s) for _ in range(n)]
        if kind != "decode":
            return _exact_layers(s, cached, s.randn(n, t, 2 * qd), s.randn(n, t, kd), s.randn(n, t, kd))
        return _exact_decode(s, cached, s.randn(n, qd), s.randn(n, qd))
    if kind in ("gdn_step", "prompt_gdn"):
        layers = [_deltanet_layer(s) for _ in range(n)]
        chunks = [_deltanet_inputs(s, n, case.get("tokens", 1))]
        if kind == "gdn_step":
            return _exact_deltanet(s, layers, *chunks)[0]
        return tuple(_exact_deltanet(s, layers, *chunks, _deltanet_inputs(s, n, 1)))
    if kind == "sweep":
        full, qd = n // 4, case["hq"] * case["d"]
        cached = [_attention_layer(s) for _ in range(full)]
        layers = [_deltanet_layer(s) for _ in range(n - full)]
        out = _exact_decode(s, cached, s.randn(full, qd), s.randn(full, qd))
        return out, _exact_deltanet(s, layers, _deltanet_inputs(s, n - full, 1))[0]
    if kind == "latent":
        h, length = case["heads"], case["length"]
        q, qe, latent, rope = s.randn(n, h, 512), s.randn(n, h, 64), s.randn(n, length, 512), s.randn(n, length, 64)
        return torch.stack([((q[i].double() @ latent[i].double().T + qe[i].double() @ rope[i].double().T) / math.sqrt(576.0))
                            .softmax(1) @ latent[i].double() for i in range(n)])
    qd, kd, hidden, out = case["hq"] * case["d"], case["hkv"] * case["d"], case["hidden"], []
    for _ in range(n):
        x, core = s.randn(hidden), s.randn(qd)
        out.append([_exact_weights(s, m, hidden) @ x.double() for m in (2 * qd, kd, kd)] + [_exact_weights(s, hidden, qd) @ core.double()])
    return out


def _exact_decode(s, cached, q, gate):
    c = s.case
    heads = lambda x, n: x.double().view(-1, n, c["d"])  # noqa: E731
    return torch.cat([_attend(heads(q[i], c["hq"]), heads(kv[0], c["hkv"]), heads(kv[1], c["hkv"]), heads(gate[i], c["hq"]),
                              c["length"] - 1) for i, (_, kv) in enumerate(cached)])


# ---- what a pass cannot do without ---------------------------------------------------------------------------------

def _deltanet_work(hk, hv, tokens):
    """Inputs, outputs, weights and state (in and out) of one DeltaNet layer, and the delta rule's operations."""
    conv = 2 * hk * 128 + hv * 128
    bytes_ = 4 * tokens * (conv + 2 * hv * 128 + 2 * hv) + 2 * 4 * hv * 128 * 128 + 2 * 4 * conv + 8 * conv
    return bytes_, 7 * 128 * 128 * hv * tokens + 8 * conv * tokens


def work(case):
    kind, n = case["kind"], case["layers"]
    b = f = 0
    if kind in ("step", "decode", "sweep", "prompt_attn"):
        es, t, length = 2 if case["bf16"] else 4, case.get("tokens", 1), case["length"]
        qd, kd = case["hq"] * case["d"], case["hkv"] * case["d"]
        io = 4 * t * 3 * qd + (0 if kind in ("decode", "sweep") else t * 2 * kd * (4 + es))
        # tokens of a step or a prompt see themselves and what was before them
        seen = t * length + (t * (t + 1) // 2 if kind in ("step", "prompt_attn") else 0)
        full = n // 4 if kind == "sweep" else n
        b += full * (io + 2 * length * kd * es)
        f += full * 4 * qd * seen
    if kind in ("gdn_step", "sweep", "prompt_gdn"):
        lin = n - n // 4 if kind == "sweep" else n
        lb, lf = _deltanet_work(case["hk"], case["hv"], case.get("tokens", 1))
        b, f = b + lin * lb, f + lin * lf
        if kind == "prompt_gdn":
            lb, lf = _deltanet_work(case["hk"], case["hv"], 1)
            b, f = b + lin * lb, f + lin * lf
    if kind == "latent":
        h, length = case["heads"], case["length"]
        b = n * 4 * (length * 576 + h * (576 + 512))
        f = n * 2 * h * length * (576 + 512)
    if kind == "proj":
        qd, kd, hidden = case["hq"] * case["d"], case["hkv"] * case["d"], case["hidden"]
        weights = (2 * qd + 2 * kd) * hidden + hidden * qd
        b = n * (weights // 2 + weights // 16 + 4 * (2 * hidden + 3 * qd + 2 * kd))
        f = n * 2 * weights
    return {"bytes": b, "flops": f}


def tolerance(case):
    """Largest relative error of another correct implementation at the same precision: about four times what these paths
    show against a float64 computation of the same case.  Over bf16 caches the query and the probabilities enter as two
    bf16 parts (3e-6; 4e-6 for the latent cache, whose every operand does), over f32 caches sums are f32 (5e-7), the
    delta rule's as well (7e-7; 3e-7 for the projections).  Where q and k are rotated, the rounding of the frequency table moves the angle by
    6e-8 of itself (1e-5 at position 3000, 1e-4 at 32768), and a key that rounds to the neighbouring bf16 value moves
    single results by 2e-3."""
    kind = case["kind"]
    if kind in ("step", "prompt_attn"):
        far = case["length"] + case.get("tokens", ROLLBACK) > 4096
        return {"rel": 3e-4 if far else 6e-5, "max": 8e-3 if case["bf16"] else 2e-3}
    if kind == "decode":
        return {"rel": 1.5e-5 if case["bf16"] else 2e-6}
    if kind == "sweep":
        return {"rel": 1.5e-5 if case["bf16"] else 3e-6}
    if kind in ("gdn_step", "prompt_gdn"):
        return {"rel": 3e-6, "max": 4e-4}
    return {"rel": 1.8e-5 if kind == "latent" else 1.5e-6}
