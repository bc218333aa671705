"""The work this library is measured on, through its public entry points.

The sizes are those of the Qwen3.5-35B-A3B mixer stack that the tests and the
benchmark use: hidden 2048, 16 key and 32 value heads of 128 in a GatedDeltaNet
layer, 16 query and 2 key/value heads of 256 in an attention layer, a 248,320
row vocabulary, 4-bit weights in groups of 64, bf16 activations and f32 states.
Drawn cases also take the smaller head counts that the tests run.

Every case has a "kind":

  decode         one token for each sequence of a batch through the fused
                 GatedDeltaNet step of several layers (gdn_decode[_gated])
  recurrent      the recurrence alone on prepared q, k, v, g, beta
  prefill        packed prompts through the chunked GatedDeltaNet core
  layer_decode   whole layers (both 4-bit projections) on one token a sequence
  layer_prefill  a whole layer on packed prompts
  attn_decode    attention layers, one token a sequence on long KV caches
  attn_prefill   an attention layer on new tokens behind cached ones
  linear         one 4-bit linear layer (lm_head, the projections)
  exec_decode    the executor's decode step over the hybrid stack
  exec_prefill   the executor's batched prefill over the hybrid stack
"""
import math
import os
import sys

import torch

sys.path.insert(1, os.path.join(os.getcwd(), "qwen-mlx_amd"))

import gdn_amd  # noqa: E402

DEV = "cuda:0"
BF = torch.bfloat16
F64 = torch.float64
HIDDEN, DH, KCONV = 2048, 128, 4
HQ, HKV, HD, THETA, ROT = 16, 2, 256, 1.0e7, 64
NQ, NKV = HQ * 2 * HD, HKV * HD
EPS = 1e-6
VOCAB = 248320


def listed():
    return [
        # one user's token through a stack of GatedDeltaNet layers: 16 work
        # items a launch, so launches and latency are what count
        dict(name="decode_b1", kind="decode", batch=1, slots=8, layers=20, hk=16, hv=32,
             gated=True),
        # a full serving batch on scattered slots of a larger pool (the
        # benchmark's step); the states of 4 layers do not fit the caches
        dict(name="decode_b64", kind="decode", batch=64, slots=96, layers=4, hk=16, hv=32,
             gated=False),
        # the reference's recurrence kernel with its own interface, an odd
        # number of tokens
        dict(name="recurrent_b4_t37", kind="recurrent", batch=4, steps=37, hk=16, hv=32),
        # the benchmark's long-context prefill, every CU busy
        dict(name="prefill_8x16384", kind="prefill", lens="16384," * 7 + "16384", hk=16, hv=32),
        # a small serving batch through whole layers, weights from HBM
        dict(name="layer_decode_b8", kind="layer_decode", batch=8, layers=16),
        # four ragged prompts admitted together
        dict(name="layer_prefill_ragged", kind="layer_prefill", lens="128,512,1000,2048"),
        # one long prompt
        dict(name="layer_prefill_16384", kind="layer_prefill", lens="16384"),
        # a serving batch at 2K-6K contexts
        dict(name="attn_decode_b64", kind="attn_decode", batch=64, lo=2048, hi=6144, layers=3),
        # a 2048-token chunk of a prompt behind 2048 cached tokens
        dict(name="attn_prefill_2048", kind="attn_prefill", cached=2048, lens="2048"),
        # the vocabulary projection of a full batch
        dict(name="lm_head_b64", kind="linear", m=64, k=HIDDEN, n=VOCAB),
        # a serving engine's step over three periods of the stack (an attention
        # layer at every fourth position), lm_head, greedy pick; the model's 40
        # layers would carry one layer's rounding through all the others
        dict(name="exec_decode_b16", kind="exec_decode", batch=16, prompt=256, layers=12),
        # three prompts admitted in one pass, two periods of the stack
        dict(name="exec_prefill_ragged", kind="exec_prefill", lens="37,512,1200", layers=8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_lens(rng, most, count):
    total = _log(rng, 17, most)
    n = min(rng.randint(1, count), total)
    cuts = sorted(rng.sample(range(1, total), n - 1)) if n > 1 else []
    return ",".join(str(b - a) for a, b in zip([0] + cuts, cuts + [total]))


def draw(rng):
    kind = rng.choice(["decode", "recurrent", "prefill", "layer_decode", "layer_prefill",
                       "attn_decode", "attn_prefill", "linear", "exec_decode", "exec_prefill"])
    hk, hv = rng.choice([(16, 32), (16, 32), (4, 16), (2, 8), (4, 4)])
    if kind == "decode":
        b = _log(rng, 1, 64)
        return dict(kind=kind, batch=b, slots=b + rng.randint(0, 32), layers=rng.randint(2, 4),
                    hk=hk, hv=hv, gated=rng.random() < 0.5)
    if kind == "recurrent":
        return dict(kind=kind, batch=_log(rng, 1, 16), steps=_log(rng, 1, 200), hk=hk, hv=hv)
    if kind == "prefill":
        return dict(kind=kind, lens=_draw_lens(rng, 65536, 8), hk=hk, hv=hv)
    if kind == "layer_decode":
        return dict(kind=kind, batch=_log(rng, 1, 64), layers=8)
    if kind == "layer_prefill":
        return dict(kind=kind, lens=_draw_lens(rng, 16384, 6))
    if kind == "attn_decode":
        hi = _log(rng, 64, 6144)
        return dict(kind=kind, batch=_log(rng, 1, 64), lo=max(1, hi // 3), hi=hi, layers=2)
    if kind == "attn_prefill":
        return dict(kind=kind, cached=rng.choice([0, _log(rng, 1, 4096)]),
                    lens=_draw_lens(rng, 4096, 3))
    if kind == "linear":
        k, n = rng.choice([(2048, 12352), (4096, 2048), (2048, 9216), (2048, VOCAB), (1024, 4096),
                           (512, 2064)])
        return dict(kind=kind, m=_log(rng, 1, 64 if n == VOCAB else 8192), k=k, n=n)
    if kind == "exec_decode":
        return dict(kind=kind, batch=_log(rng, 1, 64), prompt=rng.randint(8, 64), layers=8)
    return dict(kind=kind, lens=_draw_lens(rng, 4096, 6), layers=4)


# ------------------------------------------------------------------ inputs --

def _lens(case):
    return [int(x) for x in case["lens"].split(",")]


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _n(g, *shape, std=1.0, dtype=BF):
    return torch.empty(shape, device=DEV, dtype=torch.float32).normal_(0, std, generator=g).to(dtype)


def _u(g, lo, hi, *shape):
    return torch.empty(shape, device=DEV, dtype=torch.float32).uniform_(lo, hi, generator=g)


def _conv_dim(hk, hv):
    return 2 * hk * DH + hv * DH


def _gdn_params(g, hk, hv):
    return dict(A_log=_u(g, 0.0, math.log(16.0), hv), dt_bias=_n(g, hv, std=0.1, dtype=torch.float32),
                conv_w=_n(g, _conv_dim(hk, hv), KCONV, std=0.25),
                norm_w=(1 + 0.1 * _n(g, DH, dtype=torch.float32)).to(BF))


def _gdn_state(g, n, hk, hv):
    return (_n(g, n, hv, DH, DH, std=0.01, dtype=torch.float32),
            _n(g, n, KCONV - 1, _conv_dim(hk, hv)))


def _w4(g, n, k, std=0.03):
    """A 4-bit weight in MLX's storage: words, scales, biases."""
    w = torch.randint(-2 ** 31, 2 ** 31, (n, k // 8), device=DEV, dtype=torch.int32, generator=g)
    s = (_u(g, 0.5, 1.5, n, k // 64) * (std / 4.8)).to(BF)
    b = (-7.5 * s.float() * _u(g, 0.9, 1.1, n, k // 64)).to(BF)
    return w, s, b


def _scattered(g, slots, n):
    return torch.randperm(slots, device=DEV, generator=g)[:n].to(torch.int32)


def _mixer_gdn(g):
    d = _conv_dim(16, 32)
    p = _gdn_params(g, 16, 32)
    p["in_parts"] = [_w4(g, n, HIDDEN) for n in (d, 32 * DH, 32, 32)]
    p["out"] = _w4(g, HIDDEN, 32 * DH)
    return p


def _mixer_attn(g):
    return dict(qkv=_w4(g, NQ + 2 * NKV, HIDDEN), o=_w4(g, HIDDEN, HQ * HD),
                qn=(1 + 0.1 * _n(g, HD, dtype=torch.float32)).to(BF),
                kn=(1 + 0.1 * _n(g, HD, dtype=torch.float32)).to(BF))


def _is_attn(i):
    return i % 4 == 3


def _inputs(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    i = {}
    if kind == "decode":
        hk, hv, b = case["hk"], case["hv"], case["batch"]
        i["ids"] = _scattered(g, case["slots"], b)
        i["layers"] = []
        for _ in range(case["layers"]):
            p = _gdn_params(g, hk, hv)
            p["state"], p["conv"] = _gdn_state(g, b, hk, hv)
            p["x"] = _n(g, b, _conv_dim(hk, hv) + (hv * DH if case["gated"] else 0))
            p["ab"] = _n(g, b, 2 * hv)
            i["layers"].append(p)
    elif kind == "recurrent":
        hk, hv, b, t = case["hk"], case["hv"], case["batch"], case["steps"]
        i["ids"] = _scattered(g, b + 2, b)
        i["state"], i["conv"] = _gdn_state(g, b, hk, hv)
        unit = lambda x: x / x.norm(dim=-1, keepdim=True)  # noqa: E731
        i["q"] = (unit(_n(g, b, t, hk, DH, dtype=torch.float32)) / math.sqrt(DH)).to(BF)
        i["k"] = unit(_n(g, b, t, hk, DH, dtype=torch.float32)).to(BF)
        i["v"] = _n(g, b, t, hv, DH)
        p = _gdn_params(g, hk, hv)
        a = _n(g, b, t, hv, dtype=torch.float32)
        i["g"] = torch.exp(-torch.exp(p["A_log"]) * torch.nn.functional.softplus(a + p["dt_bias"]))
        i["beta"] = torch.sigmoid(_n(g, b, t, hv, dtype=torch.float32)).to(BF)
    elif kind in ("prefill", "layer_prefill"):
        lens = _lens(case)
        hk, hv = case.get("hk", 16), case.get("hv", 32)
        t, n = sum(lens), len(lens)
        i["ids"] = _scattered(g, n + 1, n)
        cu = [0]
        for x in lens:
            cu.append(cu[-1] + x)
        i["cu"] = torch.tensor(cu, device=DEV, dtype=torch.int32)
        if kind == "prefill":
            i.update(_gdn_params(g, hk, hv))
            i["x"] = _n(g, t, _conv_dim(hk, hv))
            i["ab"] = _n(g, t, 2 * hv)
        else:
            i.update(_mixer_gdn(g))
            i["x"] = _n(g, t, HIDDEN)
    elif kind == "layer_decode":
        b = case["batch"]
        i["ids"] = _scattered(g, b + 8, b)
        i["layers"] = []
        for _ in range(case["layers"]):
            p = _mixer_gdn(g)
            p["state"], p["conv"] = _gdn_state(g, b, 16, 32)
            p["x"] = _n(g, b, HIDDEN)
            i["layers"].append(p)
    elif kind in ("attn_decode", "attn_prefill"):
        if kind == "attn_decode":
            n = case["batch"]
            i["cached"] = torch.randint(case["lo"], case["hi"] + 1, (n,), device=DEV,
                                        generator=g).tolist()
            i["new"] = [1] * n
        else:
            i["new"] = _lens(case)
            i["cached"] = [case["cached"]] * len(i["new"])
        i["layers"] = []
        for _ in range(case.get("layers", 1)):
            p = _mixer_attn_norms(g)
            p["ck"] = _n(g, sum(i["cached"]), NKV)
            p["cv"] = _n(g, sum(i["cached"]), NKV)
            p["q"] = _n(g, sum(i["new"]), NQ)
            p["k"] = _n(g, sum(i["new"]), NKV)
            p["v"] = _n(g, sum(i["new"]), NKV)
            i["layers"].append(p)
    elif kind == "linear":
        i["w"] = _w4(g, case["n"], case["k"])
        i["x"] = _n(g, case["m"], case["k"])
    else:
        i["layers"] = [_mixer_attn(g) if _is_attn(l) else _mixer_gdn(g)
                       for l in range(case["layers"])]
        i["in_norm"] = [(1 + 0.1 * _n(g, HIDDEN, dtype=torch.float32)).to(BF) for _ in i["layers"]]
        i["final_norm"] = (1 + 0.1 * _n(g, HIDDEN, dtype=torch.float32)).to(BF)
        i["embed"] = _n(g, VOCAB, HIDDEN)
        i["head"] = _w4(g, VOCAB, HIDDEN)
        if kind == "exec_decode":
            # prompts of slightly different lengths, so that positions differ
            lens = [max(1, case["prompt"] - 3 * (s % 5)) for s in range(case["batch"])]
            i["tokens"] = torch.randint(0, VOCAB, (case["batch"],), device=DEV,
                                        generator=g).tolist()
        else:
            lens = _lens(case)
        i["prompts"] = [torch.randint(0, VOCAB, (x,), device=DEV, generator=g).tolist()
                        for x in lens]
    return i


def _mixer_attn_norms(g):
    return dict(qn=(1 + 0.1 * _n(g, HD, dtype=torch.float32)).to(BF),
                kn=(1 + 0.1 * _n(g, HD, dtype=torch.float32)).to(BF))


# ------------------------------------------------------------ prepare / run --

def _out(*shape):
    return torch.empty(shape, device=DEV, dtype=BF)


def _qlinear(k, parts):
    return gdn_amd.QLinear(k, parts)


def _layer(pool, l, p):
    return gdn_amd.Layer(pool, l, _qlinear(HIDDEN, p["in_parts"]), _qlinear(32 * DH, [p["out"]]),
                         p["A_log"], p["dt_bias"], p["conv_w"], p["norm_w"], EPS)


class _Owned:
    """A view of library memory that keeps the object which owns it alive: the
    pool's and the executor's own views end with them."""

    def __init__(self, t, owner):
        self.__cuda_array_interface__ = dict(
            shape=tuple(t.shape), typestr={torch.float32: "<f4", torch.int16: "<i2"}[t.dtype],
            data=(t.data_ptr(), False), version=3, strides=None)
        self.owner = owner


def _owned(t, owner):
    return torch.as_tensor(_Owned(t, owner), device=DEV)


def _views(pool, layer):
    state, conv = (_owned(t, pool) for t in pool.layer_views(layer))
    return state, conv.view(BF)


def prepare(case, seed):
    i = _inputs(case, seed)
    kind = case["kind"]
    s = dict(kind=kind, i=i)
    if kind == "decode":
        pool = gdn_amd.Pool(case["layers"], case["slots"], case["hk"], case["hv"])
        s["outs"] = []
        for l, p in enumerate(i["layers"]):
            pool.write(l, i["ids"], p.pop("state"), p.pop("conv"))
            s["outs"].append((_out(case["batch"], case["hv"], DH),) + _views(pool, l))
        s.update(pool=pool, gated=case["gated"])
    elif kind == "recurrent":
        pool = gdn_amd.Pool(1, case["batch"] + 2, case["hk"], case["hv"])
        pool.write(0, i["ids"], i["state"], i["conv"])
        s.update(pool=pool, y=_out(case["batch"], case["steps"], case["hv"], DH),
                 state=_views(pool, 0)[0])
    elif kind == "prefill":
        t = i["x"].shape[0]
        pool = gdn_amd.Pool(1, len(i["ids"]) + 1, case["hk"], case["hv"])
        s.update(pool=pool, t=t, y=_out(t, case["hv"], DH), views=_views(pool, 0))
    elif kind == "layer_prefill":
        t = i["x"].shape[0]
        pool = gdn_amd.Pool(1, len(i["ids"]) + 1)
        pool.reserve(t)
        s.update(pool=pool, t=t, y=_out(t, HIDDEN), views=_views(pool, 0), layer=_layer(pool, 0, i))
    elif kind == "layer_decode":
        b = case["batch"]
        pool = gdn_amd.Pool(case["layers"], b + 8)
        pool.reserve(b)
        s["layers"], s["outs"] = [], []
        for l, p in enumerate(i["layers"]):
            pool.write(l, i["ids"], p.pop("state"), p.pop("conv"))
            s["layers"].append(_layer(pool, l, p))
            s["outs"].append((_out(b, HIDDEN),) + _views(pool, l))
        s["pool"] = pool
    elif kind in ("attn_decode", "attn_prefill"):
        _prepare_attn(case, i, s)
    elif kind == "linear":
        s.update(w=_qlinear(case["k"], [i["w"]]), y=_out(case["m"], case["n"]))
    else:
        _prepare_exec(case, i, s)
    return s


def _prepare_attn(case, i, s):
    """The KV cache with the cached tokens in it, in steps of up to 2048."""
    n, most = len(i["new"]), 4096
    pages = [(c + w + 63) // 64 for c, w in zip(i["cached"], i["new"])]
    kv = gdn_amd.KVCache(len(i["layers"]), n, sum(pages), max(pages), HQ, HKV,
                         max_step_tokens=max(most, sum(i["new"])))
    q = _n(_gen(0), most, NQ)
    o = _out(most, HQ * HD)
    step = 2048
    base = 0
    for slot, c in enumerate(i["cached"]):
        for a in range(0, c, step):
            m = min(step, c - a)
            kv.step([slot], [m])
            for l, p in enumerate(i["layers"]):
                rows = slice(base + a, base + a + m)
                kv.forward(l, q[:m], p["ck"][rows], p["cv"][rows], p["qn"], p["kn"], EPS, THETA, ROT,
                           o[:m])
        base += c
    kv.step(list(range(n)), i["new"])
    s.update(kv=kv, outs=[_out(sum(i["new"]), HQ * HD) for _ in i["layers"]])


def _prepare_exec(case, i, s):
    most = sum(len(p) for p in i["prompts"])
    batch = len(i["prompts"])
    ngdn = sum(not _is_attn(l) for l in range(case["layers"]))
    pool = gdn_amd.Pool(ngdn, batch)
    # room for thousands of decode steps behind the prompts
    # (a slot has to hold the executor's longest prompt, here the whole pass)
    pages = (most + 63) // 64 + (128 if case["kind"] == "exec_decode" else 0)
    kv = gdn_amd.KVCache(max(1, case["layers"] - ngdn), batch, batch * pages, pages, HQ, HKV,
                         max_step_tokens=max(most, batch))
    layers, attn = [], []
    for l, p in enumerate(i["layers"]):
        if _is_attn(l):
            attn.append((l, _qlinear(HIDDEN, [p["qkv"]]), _qlinear(HQ * HD, [p["o"]]), p["qn"],
                         p["kn"]))
        else:
            layers.append(_layer(pool, len(layers), p))
    ex = gdn_amd.Executor(pool, layers, i["in_norm"], i["final_norm"], i["embed"],
                          _qlinear(HIDDEN, [i["head"]]), EPS, max_batch=batch, max_prompt=most,
                          attn_layers=attn, kv=kv, rope_theta=THETA, rotary_dim=ROT)
    s.update(ex=ex, pool=pool, kv=kv, ids=list(range(batch)))
    if case["kind"] == "exec_decode":
        ex.prefill_batch(s["ids"], i["prompts"])


def run(s):
    i, kind = s["i"], s["kind"]
    if kind == "decode":
        for l, (p, o) in enumerate(zip(i["layers"], s["outs"])):
            if s["gated"]:
                s["pool"].decode_gated(l, i["ids"], p["x"], p["ab"], p["A_log"], p["dt_bias"],
                                       p["conv_w"], p["norm_w"], EPS, o[0])
            else:
                s["pool"].decode(l, i["ids"], p["x"], p["ab"], p["A_log"], p["dt_bias"],
                                 p["conv_w"], o[0])
        return s["outs"]
    if kind == "recurrent":
        s["pool"].recurrent(0, i["ids"], i["q"], i["k"], i["v"], i["g"], i["beta"], s["y"])
        return [s["y"], s["state"]]
    if kind == "prefill":
        # fresh prompts: their slots start from zero states
        s["pool"].zero(0, i["ids"])
        s["pool"].prefill(0, i["ids"], i["cu"], s["t"], i["x"], i["ab"], i["A_log"], i["dt_bias"],
                          i["conv_w"], s["y"])
        return [s["y"], *s["views"]]
    if kind == "layer_prefill":
        s["pool"].zero(0, i["ids"])
        s["layer"].prefill(i["ids"], i["cu"], s["t"], i["x"], s["y"])
        return [s["y"], *s["views"]]
    if kind == "layer_decode":
        for layer, p, o in zip(s["layers"], i["layers"], s["outs"]):
            layer.decode(i["ids"], p["x"], o[0])
        return s["outs"]
    if kind in ("attn_decode", "attn_prefill"):
        # the planned step's layers; a repeated pass writes the same keys and
        # values to the same positions
        for l, (p, o) in enumerate(zip(i["layers"], s["outs"])):
            s["kv"].forward(l, p["q"], p["k"], p["v"], p["qn"], p["kn"], EPS, THETA, ROT, o)
        return s["outs"]
    if kind == "linear":
        s["w"].forward(i["x"], s["y"])
        return s["y"]
    if kind == "exec_decode":
        s["ex"].decode_batch(s["ids"], i["tokens"])
    else:
        s["ex"].prefill_batch(s["ids"], i["prompts"])
    return _owned(s["ex"].logits(), s["ex"]).view(BF)


# ------------------------------------------------------------------- work --

def _core_work(tokens, seqs, hk, hv, zgate=False):
    """One GatedDeltaNet core call: states read and written once a sequence,
    the recurrence's 7 d^2 operations a token and value head."""
    d = _conv_dim(hk, hv)
    state = hv * DH * DH * 4 + (KCONV - 1) * d * 2
    return (2 * seqs * state + tokens * (d + 2 * hv + hv * DH * (2 if zgate else 1)) * 2 +
            d * KCONV * 2, tokens * hv * 7 * DH * DH)


def _lin_work(m, k, n):
    return n * k // 2 + n * k // 16 + 2 * m * (k + n), 2 * m * k * n


def _attn_work(cached, new):
    b = f = 0
    for c, w in zip(cached, new):
        b += 2 * ((c + w) * 2 * NKV + w * (2 * NKV + NQ + HQ * HD))
        f += 4 * HQ * HD * (w * c + w * (w + 1) // 2)
    return b, f


def _layer_work(tokens, seqs):
    """A layer's own inputs, outputs, weights and states: what passes between
    its parts need not reach memory."""
    state = 32 * DH * DH * 4 + (KCONV - 1) * _conv_dim(16, 32) * 2
    n = _conv_dim(16, 32) + 32 * DH + 64
    return (2 * seqs * state + (n * HIDDEN + HIDDEN * 32 * DH) * 9 // 16 + 4 * tokens * HIDDEN,
            tokens * (2 * n * HIDDEN + 2 * HIDDEN * 32 * DH + 32 * 7 * DH * DH))


def work(case):
    kind = case["kind"]
    if kind == "decode":
        b, f = _core_work(case["batch"], case["batch"], case["hk"], case["hv"], case["gated"])
        return dict(bytes=case["layers"] * b, flops=case["layers"] * f)
    if kind == "recurrent":
        hk, hv, n = case["hk"], case["hv"], case["batch"] * case["steps"]
        return dict(bytes=2 * case["batch"] * hv * DH * DH * 4 +
                    n * (2 * hk * DH * 2 + 2 * hv * DH * 2 + 6 * hv), flops=n * hv * 7 * DH * DH)
    if kind == "prefill":
        b, f = _core_work(sum(_lens(case)), len(_lens(case)), case["hk"], case["hv"])
    elif kind == "layer_prefill":
        b, f = _layer_work(sum(_lens(case)), len(_lens(case)))
    elif kind == "layer_decode":
        b, f = _layer_work(case["batch"], case["batch"])
        b, f = b * case["layers"], f * case["layers"]
    elif kind == "attn_decode":
        mean = (case["lo"] + case["hi"]) // 2
        b, f = _attn_work([mean] * case["batch"], [1] * case["batch"])
        b, f = b * case["layers"], f * case["layers"]
    elif kind == "attn_prefill":
        b, f = _attn_work([case["cached"]] * len(_lens(case)), _lens(case))
    elif kind == "linear":
        b, f = _lin_work(case["m"], case["k"], case["n"])
    else:
        if kind == "exec_decode":
            cached, new = [case["prompt"]] * case["batch"], [1] * case["batch"]
        else:
            new = _lens(case)
            cached = [0] * len(new)
        t, n = sum(new), len(new)
        b, f = _lin_work(n, HIDDEN, VOCAB)
        for l in range(case["layers"]):
            if _is_attn(l):
                parts = [_attn_work(cached, new), _lin_work(t, HIDDEN, NQ + 2 * NKV),
                         _lin_work(t, HQ * HD, HIDDEN)]
                b += sum(c + w for c, w in zip(cached, new)) * 4 * NKV
                b += (HIDDEN * (NQ + 2 * NKV) + HIDDEN * HQ * HD) * 9 // 16
                f += sum(p[1] for p in parts)
            else:
                lb, lf = _layer_work(t, n)
                b, f = b + lb - 4 * t * HIDDEN, f + lf
    return dict(bytes=b, flops=f)


# --------------------------------------------------------------- tolerance --

def tolerance(case):
    """Two correct implementations differ by the order of f32 sums and by where
    a bf16 rounding falls; each figure is about four times the distance to the
    64-bit result that a pass of that kind shows."""
    return dict(rel=_REL[case["kind"]])


_REL = dict(decode=2.5e-2, recurrent=7e-3, prefill=2.5e-2, layer_decode=3.5e-2,
            layer_prefill=3.5e-2, attn_decode=2e-2, attn_prefill=2e-2, linear=7e-3,
            exec_decode=0.15, exec_prefill=0.15)


# ------------------------------------------------------------------- exact --

def _pool_order(state, ids, slots, hk, hv):
    """[n, Hv, Dv, Dk] states as the pool holds them: all slots, idle ones zero,
    4-row pieces of the key heads interleaved."""
    n, r = state.shape[0], hv // hk
    x = state.reshape(n, hk, r * DH // 4, 4 * DH).transpose(1, 2).reshape(n, -1)
    out = torch.zeros(slots, x.shape[1], dtype=state.dtype, device=DEV)
    out[ids.long()] = x
    return out


def _slot_rows(conv, ids, slots):
    out = torch.zeros((slots,) + conv.shape[1:], dtype=conv.dtype, device=DEV)
    out[ids.long()] = conv
    return out


def _f(t):
    return t.to(F64)


def _scan(q, k, v, g, beta, state):
    """The gated delta rule over [n, T, heads, ...] in 64 bits; q, k by value head."""
    n, t, hv = v.shape[:3]
    y = torch.empty(n, t, hv, DH, dtype=F64, device=DEV)
    s = state.reshape(n * hv, DH, DH).clone()
    for j in range(t):
        kj, qj = k[:, j].reshape(n * hv, DH, 1), q[:, j].reshape(n * hv, DH, 1)
        s *= g[:, j].reshape(n * hv, 1, 1)
        d = (v[:, j].reshape(n * hv, DH, 1) - torch.bmm(s, kj)) * beta[:, j].reshape(n * hv, 1, 1)
        s.baddbmm_(d, kj.reshape(n * hv, 1, DH))
        y[:, j] = torch.bmm(s, qj).reshape(n, hv, DH)
    return y, s.reshape(n, hv, DH, DH)


def _core_exact(x, ab, p, state, conv, lens, hk, hv):
    """Conv, silu, q/k norm, gates and recurrence of packed tokens. Sequences
    are padded to the longest with tokens that leave the state alone."""
    n, t, d = len(lens), max(lens), _conv_dim(hk, hv)
    xp = torch.zeros(n, t, d, dtype=F64, device=DEV)
    abp = torch.zeros(n, t, 2 * hv, dtype=F64, device=DEV)
    live = torch.zeros(n, t, 1, dtype=F64, device=DEV)
    a = 0
    for j, m in enumerate(lens):
        xp[j, :m], abp[j, :m], live[j, :m] = _f(x[a:a + m]), _f(ab[a:a + m]), 1.0
        a += m
    full = torch.cat([_f(conv), xp], 1)
    del xp
    tail = torch.stack([full[j, m:m + KCONV - 1] for j, m in enumerate(lens)])
    w = _f(p["conv_w"])
    c = sum(full[:, j:j + t] * w[:, j] for j in range(KCONV))
    del full
    c = c * torch.sigmoid(c)
    q, k, v = c.split([hk * DH, hk * DH, hv * DH], -1)
    norm = lambda z: z * torch.rsqrt((z * z).mean(-1, keepdim=True) + EPS)  # noqa: E731
    rep = hv // hk
    q = norm(q.reshape(n, t, hk, DH)).repeat_interleave(rep, 2) / DH
    # the key weight is the bf16 value of 128^-0.5
    k = norm(k.reshape(n, t, hk, DH)).repeat_interleave(rep, 2) * 0.08837890625
    beta = torch.sigmoid(abp[..., :hv]) * live
    g = torch.exp(-torch.exp(_f(p["A_log"])) *
                  torch.nn.functional.softplus(abp[..., hv:] + _f(p["dt_bias"])) * live)
    y, s = _scan(q, k, v.reshape(n, t, hv, DH), g, beta, _f(state))
    return torch.cat([y[j, :m] for j, m in enumerate(lens)]), s, tail


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * _f(w)


def _gate_exact(y, z, w):
    return torch.nn.functional.silu(z) * _rms(y, w)


def _deq(parts):
    out = []
    for w, s, b in parts:
        q = (w.unsqueeze(-1) >> (4 * torch.arange(8, device=DEV, dtype=torch.int32))) & 15
        n = w.shape[0]
        out.append((q.reshape(n, -1, 64) * _f(s).unsqueeze(-1) + _f(b).unsqueeze(-1)).reshape(n, -1))
    return torch.cat(out)


def _lin_exact(x, parts):
    """Columns in slices, so that the 64-bit weights stay small."""
    x = _f(x)
    return torch.cat([x @ _deq([tuple(t[a:a + 16384] for t in p)]).t()
                      for p in parts for a in range(0, p[0].shape[0], 16384)], 1)


def _layer_exact(x, p, state, conv, lens):
    hk, hv, d = 16, 32, _conv_dim(16, 32)
    proj = _lin_exact(x, p["in_parts"])
    y, s, tail = _core_exact(proj[:, :d], proj[:, d + hv * DH:], p, state, conv, lens, hk, hv)
    z = proj[:, d:d + hv * DH].reshape(-1, hv, DH)
    return _lin_exact(_gate_exact(y, z, p["norm_w"]).reshape(-1, hv * DH), [p["out"]]), s, tail


def _rope(x, pos):
    h = ROT // 2
    ang = pos.to(F64)[:, None, None] * THETA ** (-torch.arange(h, device=DEV, dtype=F64) / h)
    a, b = x[..., :h], x[..., h:ROT]
    return torch.cat([a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos(), x[..., ROT:]],
                     -1)


def _attn_exact(q, k, v, ck, cv, p, cached, new):
    outs, a, c = [], 0, 0
    for n0, m in zip(cached, new):
        pos = torch.arange(n0 + m, device=DEV)
        qg = _f(q[a:a + m]).reshape(m, HQ, 2, HD)
        kk = torch.cat([_f(ck[c:c + n0]), _f(k[a:a + m])]).reshape(-1, HKV, HD)
        vv = torch.cat([_f(cv[c:c + n0]), _f(v[a:a + m])]).reshape(-1, HKV, HD)
        qr, kr = _rope(_rms(qg[:, :, 0], p["qn"]), pos[n0:]), _rope(_rms(kk, p["kn"]), pos)
        o = torch.empty(m, HQ, HD, dtype=F64, device=DEV)
        mask = pos[None, :] > pos[n0:, None]
        for h in range(HQ):
            s = qr[:, h] @ kr[:, h // (HQ // HKV)].t() / math.sqrt(HD)
            o[:, h] = torch.softmax(s.masked_fill_(mask, -math.inf), -1) @ vv[:, h // (HQ // HKV)]
        outs.append((o * torch.sigmoid(qg[:, :, 1])).reshape(m, -1))
        a, c = a + m, c + n0
    return torch.cat(outs)


def _stack_exact(i, seqs):
    """The executor's stack on whole sequences: the last token's logits of each."""
    lens = [len(t) for t in seqs]
    h = _f(i["embed"][torch.tensor([x for t in seqs for x in t], device=DEV)])
    zero_s = torch.zeros(len(lens), 32, DH, DH, dtype=F64, device=DEV)
    zero_c = torch.zeros(len(lens), KCONV - 1, _conv_dim(16, 32), dtype=F64, device=DEV)
    for l, p in enumerate(i["layers"]):
        x = _rms(h, i["in_norm"][l])
        if _is_attn(l):
            q, k, v = _lin_exact(x, [p["qkv"]]).split([NQ, NKV, NKV], 1)
            none = torch.zeros(0, NKV, dtype=F64, device=DEV)
            h = h + _lin_exact(_attn_exact(q, k, v, none, none, p, [0] * len(lens), lens), [p["o"]])
        else:
            h = h + _layer_exact(x, p, zero_s, zero_c, lens)[0]
    last = torch.tensor(lens, device=DEV).cumsum(0) - 1
    return _lin_exact(_rms(h[last], i["final_norm"]), [i["head"]])


def exact(case, seed):
    i = _inputs(case, seed)
    kind = case["kind"]
    if kind == "decode":
        hk, hv, b, outs = case["hk"], case["hv"], case["batch"], []
        for p in i["layers"]:
            d = _conv_dim(hk, hv)
            y, s, tail = _core_exact(p["x"][:, :d], p["ab"], p, p["state"], p["conv"], [1] * b, hk,
                                     hv)
            if case["gated"]:
                y = _gate_exact(y, _f(p["x"][:, d:]).reshape(b, hv, DH), p["norm_w"])
            outs.append((y, _pool_order(s, i["ids"], case["slots"], hk, hv),
                         _slot_rows(tail, i["ids"], case["slots"])))
        return outs
    if kind == "recurrent":
        rep = case["hv"] // case["hk"]
        y, s = _scan(_f(i["q"]).repeat_interleave(rep, 2), _f(i["k"]).repeat_interleave(rep, 2),
                     _f(i["v"]), _f(i["g"]), _f(i["beta"]), _f(i["state"]))
        return [y, _pool_order(s, i["ids"], case["batch"] + 2, case["hk"], case["hv"])]
    if kind in ("prefill", "layer_prefill"):
        lens = _lens(case)
        hk, hv = case.get("hk", 16), case.get("hv", 32)
        s0 = torch.zeros(len(lens), hv, DH, DH, dtype=F64, device=DEV)
        c0 = torch.zeros(len(lens), KCONV - 1, _conv_dim(hk, hv), dtype=F64, device=DEV)
        if kind == "prefill":
            y, s, tail = _core_exact(i["x"], i["ab"], i, s0, c0, lens, hk, hv)
        else:
            y, s, tail = _layer_exact(i["x"], i, s0, c0, lens)
        n = len(lens) + 1
        return [y, _pool_order(s, i["ids"], n, hk, hv), _slot_rows(tail, i["ids"], n)]
    if kind == "layer_decode":
        outs = []
        for p in i["layers"]:
            y, s, tail = _layer_exact(p["x"], p, p["state"], p["conv"], [1] * case["batch"])
            outs.append((y, _pool_order(s, i["ids"], case["batch"] + 8, 16, 32),
                         _slot_rows(tail, i["ids"], case["batch"] + 8)))
        return outs
    if kind in ("attn_decode", "attn_prefill"):
        return [_attn_exact(p["q"], p["k"], p["v"], p["ck"], p["cv"], p, i["cached"], i["new"])
                for p in i["layers"]]
    if kind == "linear":
        return _lin_exact(i["x"], [i["w"]])
    if kind == "exec_decode":
        return _stack_exact(i, [p + [t] for p, t in zip(i["prompts"], i["tokens"])])
    return _stack_exact(i, i["prompts"])
