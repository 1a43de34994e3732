"""Performance cases of the Qwen3 decode kernels on one MI355X: the blocks a decoder built on this
library calls for every token (attention block, MLP block, LM head and token pick), the
many-row elementwise sweeps, and whole decodes through ``model.Decoder``.

Sizes are those of the benchmark's configurations (Qwen3-0.6B, 1.7B and 4B widths, 8192-position
histories, 4096-row sweeps) and of the parity tests (head_dim 64 and 256, wide and ragged rows,
small vocabularies). ``draw`` spreads over the same ranges. All inputs come from the seed through
torch's generators: N(0, 0.02) matrices, 1 + N(0, 0.1) norm weights, N(0, 1) activations and caches.
"""
import importlib.util
import math
import sys
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parents[1]
EPS, THETA = 1e-6, 1e6
BF16, F64 = torch.bfloat16, torch.float64

WIDTHS = {
    "0.6B": dict(hidden=1024, inter=3072, layers=28, heads=16, kv_heads=8, head_dim=128, vocab=151936),
    "1.7B": dict(hidden=2048, inter=6144, layers=28, heads=16, kv_heads=8, head_dim=128, vocab=151936),
    "4B": dict(hidden=2560, inter=9728, layers=36, heads=32, kv_heads=8, head_dim=128, vocab=151936),
}
# a configuration without a specialised step (its layers run as single launches in a hipGraph)
OTHER = dict(hidden=512, inter=1024, layers=12, heads=8, kv_heads=4, vocab=3000)


def _package():
    if "llm_inference_amd" not in sys.modules:
        home = ROOT / "llm-inference_amd"
        spec = importlib.util.spec_from_file_location(
            "llm_inference_amd", home / "__init__.py", submodule_search_locations=[str(home)])
        module = importlib.util.module_from_spec(spec)
        sys.modules["llm_inference_amd"] = module
        spec.loader.exec_module(module)
    return sys.modules["llm_inference_amd"]


def listed():
    w06, w4 = WIDTHS["0.6B"], WIDTHS["4B"]
    return [
        # the smallest call: the head of a small model (the parity tests' widths), greedy
        dict(name="head_small", kind="head", hidden=256, vocab=1000, pick="argmax", temperature=1.0),
        # the end of every token of a sampled chat at 0.6B: final norm, LM head, temperature draw
        dict(name="head_sample", kind="head", hidden=1024, vocab=151936, pick="sample", temperature=0.8),
        # one layer's attention block early in a conversation (short prompt + 256 tokens) at 0.6B
        dict(name="attn_short", kind="attn", form="separate", hidden=1024, heads=16, kv_heads=8,
             head_dim=128, pos=260, max_seq=4096),
        # the same at 4B deep into a long document
        dict(name="attn_long", kind="attn", form="separate", hidden=2560, heads=32, kv_heads=8,
             head_dim=128, pos=8300, max_seq=8448),
        # a small-head model, ragged position, the form with the rotation inside the scores pass
        dict(name="attn_d64", kind="attn", form="fused", hidden=512, heads=8, kv_heads=4,
             head_dim=64, pos=12345, max_seq=16640),
        # one layer's MLP block at 4B
        dict(name="mlp_4B", kind="mlp", form="fused", hidden=2560, inter=9728),
        # many-row sweeps (a prompt's rows at 4B widths): RMSNorm, QK-norm + RoPE, SwiGLU
        dict(name="norm_rows", kind="norm", rows=4096, dim=2560),
        dict(name="norm_wide", kind="norm", rows=1000, dim=9000),
        dict(name="rope_rows", kind="rope", rows=4096, heads=32, kv_heads=8, head_dim=128, first=0),
        dict(name="swiglu_rows", kind="swiglu", rows=4096, inter=9728),
        # whole decodes: the headline (5-token prompt, 256 greedy tokens at 0.6B) ...
        dict(name="decode_greedy", kind="decode", **w06, history=0, prompt=5, steps=256,
             pick="argmax", temperature=1.0, max_seq=512),
        # ... and a sampled continuation of a long document at 4B, token by token
        dict(name="decode_sampled", kind="decode", **w4, history=8192, prompt=2, steps=14,
             pick="sample", temperature=0.8, max_seq=8448),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["head", "attn", "attn", "mlp", "norm", "rope", "swiglu", "decode"])
    if kind == "head":
        return dict(kind=kind, hidden=8 * _log(rng, 32, 320), vocab=_log(rng, 1000, 151936),
                    pick=rng.choice(["argmax", "sample"]), temperature=round(rng.uniform(0.3, 1.5), 3))
    if kind == "attn":
        head_dim = rng.choice([64, 128, 128, 128, 256])
        kv_heads = rng.choice([1, 2, 4, 8])
        heads = kv_heads * rng.choice([1, 2, 4, 8])
        pos = _log(rng, 1, 16000)
        return dict(kind=kind, form=rng.choice(["separate", "fused"]), hidden=8 * _log(rng, 32, 320),
                    heads=heads, kv_heads=kv_heads, head_dim=head_dim, pos=pos,
                    max_seq=pos + _log(rng, 1, 8192))
    if kind == "mlp":
        return dict(kind=kind, form=rng.choice(["separate", "fused"]), hidden=8 * _log(rng, 32, 640),
                    inter=8 * _log(rng, 64, 1728))
    if kind == "norm":
        dim = _log(rng, 64, 12288)
        return dict(kind=kind, rows=_log(rng, 1, 4096), dim=dim if rng.random() < 0.4 else (dim + 7) // 8 * 8)
    if kind == "rope":
        kv_heads = rng.choice([1, 2, 4, 8])
        return dict(kind=kind, rows=_log(rng, 1, 4096), heads=kv_heads * rng.choice([1, 2, 4]),
                    kv_heads=kv_heads, head_dim=rng.choice([64, 128, 128, 256]), first=rng.randint(0, 4096))
    if kind == "swiglu":
        return dict(kind=kind, rows=_log(rng, 1, 4096), inter=_log(rng, 512, 9728))
    size = rng.choice(["0.6B", "0.6B", "1.7B", "4B", "other"])
    if size == "other":
        widths = dict(OTHER, head_dim=rng.choice([64, 128, 256]))
        history, prompt, steps = rng.choice([0, _log(rng, 16, 12000)]), rng.randint(1, 8), rng.randint(8, 64)
    else:
        widths = WIDTHS[size]
        history = rng.choice([0, _log(rng, 16, 8192)])
        prompt, steps = rng.randint(1, 8), rng.randint(4, {"0.6B": 96, "1.7B": 40, "4B": 16}[size])
    return dict(kind="decode", **widths, history=history, prompt=prompt, steps=steps,
                pick=rng.choice(["argmax", "sample"]), temperature=round(rng.uniform(0.3, 1.5), 3),
                max_seq=history + prompt + steps + rng.randint(1, 500))


# ---------------------------------------------------------------- inputs

class Inputs:
    """Seeded device tensors, in the order they are asked for."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape, std=1.0, mean=0.0):
        t = torch.randn(*shape, generator=self.g, device="cuda", dtype=BF16)
        if std != 1.0:
            t.mul_(std)
        return t.add_(mean) if mean else t

    def weight(self, rows, cols):
        return self.normal(rows, cols, std=0.02)

    def gamma(self, dim):
        return self.normal(dim, std=0.1, mean=1.0)


def _layer_tensors(c, put):
    """put(name, shape, is_gamma) for one decode configuration's weights, in checkpoint order."""
    H, I, D = c["hidden"], c["inter"], c["head_dim"]
    qd, kvd = c["heads"] * D, c["kv_heads"] * D
    put("model.embed_tokens.weight", (c["vocab"], H), False)
    for layer in range(c["layers"]):
        p = f"model.layers.{layer}."
        put(p + "input_layernorm.weight", (H,), True)
        put(p + "self_attn.q_proj.weight", (qd, H), False)
        put(p + "self_attn.k_proj.weight", (kvd, H), False)
        put(p + "self_attn.v_proj.weight", (kvd, H), False)
        put(p + "self_attn.q_norm.weight", (D,), True)
        put(p + "self_attn.k_norm.weight", (D,), True)
        put(p + "self_attn.o_proj.weight", (H, qd), False)
        put(p + "post_attention_layernorm.weight", (H,), True)
        put(p + "mlp.gate_proj.weight", (I, H), False)
        put(p + "mlp.up_proj.weight", (I, H), False)
        put(p + "mlp.down_proj.weight", (H, I), False)
    put("model.norm.weight", (H,), True)


def _make(c, seed):
    """A case's inputs: what a program holds before the call."""
    r = Inputs(seed)
    kind = c["kind"]
    if kind == "head":
        u = float(torch.rand(1, generator=torch.Generator().manual_seed(int(seed))))
        return dict(x=r.normal(c["hidden"]), gamma=r.gamma(c["hidden"]),
                    w=r.weight(c["vocab"], c["hidden"]), coin=u)
    if kind == "attn":
        H, D = c["hidden"], c["head_dim"]
        qd, kvd = c["heads"] * D, c["kv_heads"] * D
        return dict(x=r.normal(H), gamma=r.gamma(H), wq=r.weight(qd, H), wk=r.weight(kvd, H),
                    wv=r.weight(kvd, H), wo=r.weight(H, qd), qn=r.gamma(D), kn=r.gamma(D),
                    kc=r.normal(c["max_seq"], kvd), vc=r.normal(c["max_seq"], kvd))
    if kind == "mlp":
        H, I = c["hidden"], c["inter"]
        return dict(x=r.normal(H), gamma=r.gamma(H), wg=r.weight(I, H), wu=r.weight(I, H),
                    wd=r.weight(H, I))
    if kind == "norm":
        return dict(x=r.normal(c["rows"], c["dim"]), gamma=r.gamma(c["dim"]))
    if kind == "rope":
        D, T = c["head_dim"], c["rows"]
        qd, kvd = c["heads"] * D, c["kv_heads"] * D
        return dict(q=r.normal(T, qd), k=r.normal(T, kvd), v=r.normal(T, kvd), qn=r.gamma(D),
                    kn=r.gamma(D))
    if kind == "swiglu":
        return dict(gate=r.normal(c["rows"], c["inter"]), up=r.normal(c["rows"], c["inter"]))
    host = np.random.default_rng(int(seed))
    return dict(tokens=[int(t) for t in host.integers(0, c["vocab"], c["prompt"])],
                coins=[float(v) for v in host.random(c["steps"])], r=r)


class _DeviceArray:
    """A bf16 array of a decoder's run state or weights, for torch.as_tensor (as raw int16). The
    tensor's storage keeps this object, and with it the decoder that owns the memory."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr="<i2", data=(ptr, False),
                                             version=2, strides=None)


def _view(owner, ptr, shape):
    return torch.as_tensor(_DeviceArray(owner, ptr, shape), device="cuda").view(BF16)


def prepare(case, seed):
    pkg = _package()
    pkg.lib()
    c, kind = dict(case), case["kind"]
    s = _make(c, seed)
    s["c"] = c

    def empty(*shape):
        return torch.empty(*shape, device="cuda", dtype=BF16)

    if kind == "head":
        s.update(logits=empty(c["vocab"]), token=torch.zeros(1, device="cuda", dtype=torch.int32))
    elif kind == "attn":
        D = c["head_dim"]
        qd, kvd = c["heads"] * D, c["kv_heads"] * D
        floats = pkg.attention_workspace_floats(c["heads"], D, c["max_seq"])
        s.update(q=empty(qd), k=empty(kvd), v=empty(kvd), out=empty(qd),
                 att=torch.empty(floats, device="cuda", dtype=torch.float32),
                 pos=torch.tensor([c["pos"]], device="cuda", dtype=torch.int32))
    elif kind == "mlp":
        s.update(act=empty(c["inter"]), normed=empty(c["hidden"]))
    elif kind == "norm":
        s.update(out=empty(c["rows"], c["dim"]))
    elif kind == "rope":
        slots, kvd = c["first"] + c["rows"], c["kv_heads"] * c["head_dim"]
        s.update(kc=torch.zeros(slots, kvd, device="cuda", dtype=BF16),
                 vc=torch.zeros(slots, kvd, device="cuda", dtype=BF16),
                 positions=torch.arange(c["first"], slots, device="cuda", dtype=torch.int32))
    elif kind == "swiglu":
        s.update(act=empty(c["rows"], c["inter"]))
    else:
        from llm_inference_amd import model
        cfg = model.make_config(c["hidden"], c["inter"], c["layers"], c["heads"], c["kv_heads"],
                                head_dim=c["head_dim"], vocab_size=c["vocab"],
                                max_seq_len=c["max_seq"], rms_norm_eps=EPS, rope_theta=THETA)
        dec = model.Decoder(cfg, ("synth", int(seed), 0.02, 0.1), max_seq=c["max_seq"])
        tensors, r = dec.tensors(), s.pop("r")

        def put(name, shape, is_gamma):
            t = r.gamma(*shape) if is_gamma else r.weight(*shape)
            _view(dec, tensors[name][0], shape).copy_(t)

        _layer_tensors(c, put)
        shape = (c["layers"], c["max_seq"], c["kv_heads"] * c["head_dim"])
        s["key_cache"] = _view(dec, dec.s.key_cache, shape)
        s["value_cache"] = _view(dec, dec.s.value_cache, shape)
        for layer in range(c["layers"] if c["history"] else 0):
            for cache in (s["key_cache"], s["value_cache"]):
                cache[layer, :c["history"]] = r.normal(c["history"], shape[2])
        torch.cuda.synchronize()
        dec.capture_graph()
        s["dec"] = dec
    return s


# ---------------------------------------------------------------- one pass

def run(s):
    pkg, c = _package(), s["c"]
    kind = c["kind"]
    if kind == "head":
        pkg.rmsnorm_gemv_forward(s["logits"], s["w"], s["x"], s["gamma"], EPS, c["vocab"], c["hidden"])
        if c["pick"] == "argmax":
            pkg.argmax_forward(s["token"], s["logits"], c["vocab"])
        else:
            pkg.sample_forward(s["token"], s["logits"], c["vocab"], 1.0 / c["temperature"], s["coin"])
        return dict(logits=s["logits"], token=s["token"])
    if kind == "attn":
        H, D, hq, hkv = c["hidden"], c["head_dim"], c["heads"], c["kv_heads"]
        scale = 1.0 / math.sqrt(D)
        pkg.rmsnorm_qkv_forward(s["q"], s["k"], s["v"], s["wq"], s["wk"], s["wv"], s["x"], s["gamma"],
                                EPS, hq * D, hkv * D, H)
        if c["form"] == "separate":
            pkg.qk_norm_rope_forward(s["q"], s["k"], s["v"], s["qn"], s["kn"], s["kc"], s["vc"],
                                     s["pos"], hq, hkv, D, EPS, THETA)
            pkg.attention_forward(s["out"], s["q"], s["kc"], s["vc"], s["att"], hq, hkv, D, s["pos"],
                                  c["max_seq"], scale)
        else:
            pkg.qk_norm_rope_attention_forward(s["out"], s["q"], s["k"], s["v"], s["qn"], s["kn"],
                                               s["kc"], s["vc"], s["att"], s["pos"], hq, hkv, D, EPS,
                                               THETA, c["max_seq"], scale)
        pkg.gemv_residual_forward(s["x"], s["wo"], s["out"], H, hq * D)
        return dict(out=s["out"], x=s["x"], key_cache=s["kc"], value_cache=s["vc"])
    if kind == "mlp":
        H, I = c["hidden"], c["inter"]
        if c["form"] == "fused":
            pkg.rmsnorm_gate_up_forward(s["act"], s["wg"], s["wu"], s["x"], s["gamma"], EPS, I, H)
        else:
            pkg.rmsnorm_forward(s["normed"], s["x"], s["gamma"], 1, H, EPS)
            pkg.gate_up_forward(s["act"], s["wg"], s["wu"], s["normed"], I, H)
        pkg.gemv_residual_forward(s["x"], s["wd"], s["act"], H, I)
        return dict(act=s["act"], x=s["x"])
    if kind == "norm":
        pkg.rmsnorm_forward(s["out"], s["x"], s["gamma"], c["rows"], c["dim"], EPS)
        return s["out"]
    if kind == "rope":
        pkg.qk_norm_rope_rows(s["q"], s["k"], s["v"], s["qn"], s["kn"], s["kc"], s["vc"],
                              s["positions"], c["rows"], c["heads"], c["kv_heads"], c["head_dim"],
                              EPS, THETA)
        return dict(q=s["q"], k=s["k"], key_cache=s["kc"], value_cache=s["vc"])
    if kind == "swiglu":
        pkg.swiglu_forward(s["act"], s["gate"], s["up"], c["rows"] * c["inter"])
        return s["act"]
    dec, pos = s["dec"], c["history"]
    for token in s["tokens"]:  # the prompt, one position at a time
        dec.forward(token, pos)
        pos += 1
    prompt_logits = _bits(dec.logits())
    if c["pick"] == "argmax":
        tokens = [dec.sample_argmax()]
        tokens += dec.generate_greedy(tokens[0], pos, c["steps"])
    else:
        tokens = []
        for coin in s["coins"]:
            tokens.append(dec.sample_temperature(c["temperature"], coin))
            dec.forward(tokens[-1], pos)
            pos += 1
    return dict(prompt_logits=prompt_logits, tokens=torch.tensor(tokens), logits=_bits(dec.logits()),
                key_cache=s["key_cache"], value_cache=s["value_cache"])


def _bits(raw):
    return torch.from_numpy(raw.view(np.int16)).view(BF16)


# ---------------------------------------------------------------- what a pass cannot do without

def work(c):
    kind = c["kind"]
    if kind == "head":
        n = c["vocab"] * c["hidden"]
        return dict(bytes=2.0 * (n + 2 * c["hidden"] + c["vocab"]), flops=2.0 * n)
    if kind == "attn":
        qd, kvd = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
        n = c["hidden"] * (2 * qd + 2 * kvd)
        kv = 2 * (c["pos"] + 1) * kvd
        return dict(bytes=2.0 * (n + kv + 3 * c["hidden"] + qd),
                    flops=2.0 * n + 4.0 * (c["pos"] + 1) * qd)
    if kind == "mlp":
        n = 3 * c["hidden"] * c["inter"]
        return dict(bytes=2.0 * (n + 3 * c["hidden"] + c["inter"]), flops=2.0 * n)
    if kind == "norm":
        n = c["rows"] * c["dim"]
        return dict(bytes=2.0 * (2 * n + c["dim"]), flops=4.0 * n)
    if kind == "rope":
        q, kv = c["rows"] * c["heads"] * c["head_dim"], c["rows"] * c["kv_heads"] * c["head_dim"]
        return dict(bytes=2.0 * (2 * q + 5 * kv), flops=10.0 * (q + kv))
    if kind == "swiglu":
        n = c["rows"] * c["inter"]
        return dict(bytes=6.0 * n, flops=5.0 * n)
    qd, kvd = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    per_layer = c["hidden"] * (2 * qd + 2 * kvd + 3 * c["inter"])
    n = c["layers"] * per_layer + c["vocab"] * c["hidden"]
    tokens = c["prompt"] + c["steps"]
    reach = tokens * c["history"] + tokens * (tokens + 1) / 2
    return dict(bytes=2.0 * tokens * n + 4.0 * c["layers"] * kvd * reach,
                flops=2.0 * tokens * n + 4.0 * c["layers"] * qd * reach)


def tolerance(c):
    """About four times what bf16 rounding alone leaves against 64 bits (measured: head 0.0027, attn
    0.0071, mlp 0.0045, norm and swiglu 0.0024, rope 0.0034, a whole model 0.016-0.06). The token of
    a pick and the tokens of a decode must be the same."""
    return dict(rel={"head": 0.011, "attn": 0.028, "mlp": 0.018, "norm": 0.0095, "rope": 0.0135,
                     "swiglu": 0.0095, "decode": 0.03}[c["kind"]])


# ---------------------------------------------------------------- the same in 64 bits

def _rms(x, gamma):
    x = x.to(F64)
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * gamma.to(F64)


def _rope(x, positions):
    """x [tokens, heads, D] rotated at the positions."""
    D = x.shape[-1]
    freq = THETA ** (-torch.arange(0, D, 2, device=x.device, dtype=F64) / D)
    angle = positions.to(F64)[:, None] * freq[None, :]
    cos, sin = angle.cos()[:, None, :], angle.sin()[:, None, :]
    a, b = x[..., :D // 2], x[..., D // 2:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _attend(q, keys, values, pos):
    """One query [heads, D] over rows 0..pos of [slots, kv_heads, D] caches."""
    rep = q.shape[0] // keys.shape[1]
    out = torch.empty_like(q)
    for h in range(q.shape[0]):
        k, v = keys[:pos + 1, h // rep], values[:pos + 1, h // rep]
        p = torch.softmax(k @ q[h] / math.sqrt(q.shape[1]), 0)
        out[h] = p @ v
    return out


def exact(case, seed):
    c, kind = dict(case), case["kind"]
    s = _make(c, seed)
    if kind == "head":
        x = _rms(s["x"], s["gamma"])
        return dict(logits=torch.cat([w.to(F64) @ x for w in s["w"].split(8192)]), token=None)
    if kind == "attn":
        D = c["head_dim"]
        x = _rms(s["x"], s["gamma"])
        at = torch.tensor([c["pos"]], device="cuda")
        q = _rope(_rms((s["wq"].to(F64) @ x).view(1, -1, D), s["qn"]), at)[0]
        k = _rope(_rms((s["wk"].to(F64) @ x).view(1, -1, D), s["kn"]), at)[0]
        kc, vc = s["kc"].to(F64), s["vc"].to(F64)
        kc[c["pos"]], vc[c["pos"]] = k.reshape(-1), s["wv"].to(F64) @ x
        out = _attend(q, kc.view(c["max_seq"], -1, D), vc.view(c["max_seq"], -1, D), c["pos"]).reshape(-1)
        return dict(out=out, x=s["x"].to(F64) + s["wo"].to(F64) @ out, key_cache=kc, value_cache=vc)
    if kind == "mlp":
        x = _rms(s["x"], s["gamma"])
        act = torch.nn.functional.silu(s["wg"].to(F64) @ x) * (s["wu"].to(F64) @ x)
        return dict(act=act, x=s["x"].to(F64) + s["wd"].to(F64) @ act)
    if kind == "norm":
        return _rms(s["x"], s["gamma"])
    if kind == "rope":
        D, T = c["head_dim"], c["rows"]
        at = torch.arange(c["first"], c["first"] + T, device="cuda")
        q = _rope(_rms(s["q"].view(T, -1, D), s["qn"]), at).reshape(T, -1)
        k = _rope(_rms(s["k"].view(T, -1, D), s["kn"]), at).reshape(T, -1)
        pad = torch.zeros(c["first"], k.shape[1], device="cuda", dtype=F64)
        return dict(q=q, k=k, key_cache=torch.cat([pad, k]), value_cache=torch.cat([pad, s["v"].to(F64)]))
    if kind == "swiglu":
        return torch.nn.functional.silu(s["gate"].to(F64)) * s["up"].to(F64)
    # a decode: the logits after the prompt (later tokens follow from picks among near ties)
    w, r, D, T = {}, s["r"], c["head_dim"], c["prompt"]

    def put(name, shape, is_gamma):
        w[name] = r.gamma(*shape) if is_gamma else r.weight(*shape)

    _layer_tensors(c, put)
    embed = w["model.embed_tokens.weight"]
    x = embed[torch.tensor(s["tokens"], device="cuda")].to(F64)
    at = torch.arange(c["history"], c["history"] + T, device="cuda")
    for layer in range(c["layers"]):
        p = f"model.layers.{layer}."

        def linear(v, name):
            return v @ w[p + name].to(F64).T

        past = [r.normal(c["history"], c["kv_heads"] * D).to(F64) for _ in range(2)] if c["history"] else None
        h = _rms(x, w[p + "input_layernorm.weight"])
        q = _rope(_rms(linear(h, "self_attn.q_proj.weight").view(T, -1, D), w[p + "self_attn.q_norm.weight"]), at)
        k = _rope(_rms(linear(h, "self_attn.k_proj.weight").view(T, -1, D), w[p + "self_attn.k_norm.weight"]), at)
        v = linear(h, "self_attn.v_proj.weight").view(T, -1, D)
        if past:
            k = torch.cat([past[0].view(-1, c["kv_heads"], D), k])
            v = torch.cat([past[1].view(-1, c["kv_heads"], D), v])
        out = torch.stack([_attend(q[t], k, v, c["history"] + t).reshape(-1) for t in range(T)])
        x = x + linear(out, "self_attn.o_proj.weight")
        h = _rms(x, w[p + "post_attention_layernorm.weight"])
        act = torch.nn.functional.silu(linear(h, "mlp.gate_proj.weight")) * linear(h, "mlp.up_proj.weight")
        x = x + linear(act, "mlp.down_proj.weight")
    last = _rms(x[-1], w["model.norm.weight"])
    logits = torch.cat([rows.to(F64) @ last for rows in embed.split(8192)])
    return dict(prompt_logits=logits, tokens=None, logits=None, key_cache=None, value_cache=None)
