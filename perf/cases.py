"""The calls that a program using this library spends its time in, with their real sizes.

GPT-OSS decodes one token at a time, serves small batches of concurrent requests and prefills
prompts: each is the mixture-of-experts block of every layer, over device buffers on one stream.
Around it stand the LM head of each generated token, the per-expert host call of programs that
route by themselves, and the Beaver-triple generator of the MPC layers.

Layers hold weights of a checkpoint's kind: MXFP4 nibbles uniform, block scales 2^-10 .. 2^-6 (a
weight of about 0.015, so that gate and up of a unit-variance input are of order one, as behind an
RMSNorm), router weights N(0, 0.02), biases N(0, 0.01).
"""
import ctypes
import math

import numpy as np
import torch

import silentotithrandousha_amd as pkg

GPT_OSS_20B = dict(H=2880, I=2880, E=32, k=4)
GPT_OSS_120B = dict(H=2880, I=2880, E=128, k=4)
VOCAB = 201088
E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)
SCALE_LO, SCALE_HI = 117, 121  # E8M0: 2^(s - 127)
CLAMP = 7.0
EPS = 1e-5
FIELD = (1 << 31) - 1


def _layer(name, T, layers=1, norm=False, quant=False, **shape):
    return dict(name=name, op="layer", T=T, layers=layers, norm=norm, quant=quant, **shape)


def listed():
    return [
        # one token of one request: every layer streams four experts, several layers so that the
        # weights come from HBM and not from a cache
        _layer("decode1_20b", 1, layers=8, **GPT_OSS_20B),
        # the same with the post-attention norm and the residual, over 128 experts
        _layer("block1_120b", 1, layers=4, norm=True, **GPT_OSS_120B),
        # a handful of concurrent requests (an odd count): most experts have one or two tokens
        _layer("batch7_20b", 7, layers=2, norm=True, **GPT_OSS_20B),
        # a serving batch on the large model: one or two tokens an expert
        _layer("batch48_120b", 48, **GPT_OSS_120B),
        # a serving batch on the small model: eight tokens an expert
        _layer("batch64_20b", 64, **GPT_OSS_20B),
        # a short prompt, odd, on a model of other dimensions
        _layer("prompt333_2048", 333, norm=True, H=2048, I=1536, E=16, k=2),
        # prefill of a long prompt on either model
        _layer("prefill4096_20b", 4096, **GPT_OSS_20B),
        _layer("prefill2048_120b", 2048, **GPT_OSS_120B),
        # prefill with the opt-in MXFP6 activations
        _layer("prefill1000_20b_mxfp6", 1000, quant=True, **GPT_OSS_20B),
        # a program that routes by itself: the experts of a token in two layers, host arrays
        dict(name="experts_host", op="expert", H=2880, I=2880, layers=2, k=4),
        # the logits of one generated token, from the checkpoint's bf16 rows
        dict(name="lm_head_bf16", op="lm_head", H=2880, V=VOCAB, bf16=True),
        # triples for the MPC layers, every party's share
        dict(name="beaver_5_1", op="beaver", n=5, t=1, count=5_000_001, party=-1),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.random()
    if kind < 0.70:
        which = rng.random()
        if which < 0.45:
            shape, top = dict(GPT_OSS_20B), 4096
        elif which < 0.75:
            shape, top = dict(GPT_OSS_120B), 2048
        else:
            E = rng.choice((8, 16, 32, 64))
            shape = dict(H=32 * rng.randint(16, 96), I=32 * rng.randint(16, 96), E=E, k=rng.choice((1, 2, 4)))
            top = 2048
        T = _log_int(rng, 1, top)
        return dict(op="layer", T=T, layers=rng.choice((2, 4, 8)) if T == 1 else 1, norm=rng.random() < 0.5,
                    quant=T >= 64 and rng.random() < 0.2, **shape)
    if kind < 0.80:
        return dict(op="expert", H=2880, I=2880, layers=rng.randint(1, 4), k=rng.randint(1, 4))
    if kind < 0.90:
        bf16 = rng.random() < 0.7
        return dict(op="lm_head", H=8 * rng.randint(64, 360), V=_log_int(rng, 10_000, VOCAB if bf16 else 50_000), bf16=bf16)
    n, t = rng.choice(((3, 1), (4, 1), (5, 1), (5, 2), (7, 2), (7, 3)))
    return dict(op="beaver", n=n, t=t, count=_log_int(rng, 1_000, 20_000_000 // n), party=rng.choice((-1, 0, n - 1)))


# ---------------------------------------------------------------- inputs, from the seed alone


class _Buf:
    """A torch tensor as the library takes device buffers."""

    def __init__(self, t):
        self.t, self.ptr = t, t.data_ptr()


_stream = None


def _on():
    """The stream that every call of the program is enqueued on."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream.cuda_stream


def _gen(seed, *tags):
    g = torch.Generator(device="cuda")
    s = int(seed) * 1_000_003
    for t in tags:
        s = (s * 1009 + t + 17) % (1 << 62)
    return g.manual_seed(s)


def _layer_tensors(case, seed, layer, E):
    """One layer's checkpoint tensors on the GPU."""
    H, I = case["H"], case["I"]
    g = _gen(seed, 1, layer)

    def u8(lo, hi, *shape):
        return torch.randint(lo, hi + 1, shape, dtype=torch.uint8, device="cuda", generator=g)

    def f32(sigma, *shape):
        return torch.randn(shape, device="cuda", generator=g).mul_(sigma)

    return dict(gu_blocks=u8(0, 255, E, 2 * I, H // 32, 16), gu_scales=u8(SCALE_LO, SCALE_HI, E, 2 * I, H // 32),
                gu_bias=f32(0.01, E, 2 * I).bfloat16().float(),
                d_blocks=u8(0, 255, E, H, I // 32, 16), d_scales=u8(SCALE_LO, SCALE_HI, E, H, I // 32),
                d_bias=f32(0.01, E, H).bfloat16().float(),
                router_w=f32(0.02, E, H).bfloat16(), gamma=f32(0.1, H).add_(1.0).bfloat16().float())


_KEYS = ("gu_blocks", "gu_scales", "gu_bias", "d_blocks", "d_scales", "d_bias")


def _load_layer(d, i, w, E, router=True, norm=False):
    torch.cuda.synchronize()
    L = pkg.lib()
    if L.moe_preload_layer_device(d.ctx, i, E, *[ctypes.c_void_p(w[n].data_ptr()) for n in _KEYS], None):
        raise RuntimeError(L.moe_last_error().decode())
    if router:
        rw = w["router_w"].view(torch.int16).cpu().numpy().view(np.uint16)
        rb = np.zeros(E, np.float32)
        if L.moe_preload_router(d.ctx, i, E, rw.ctypes.data, rb.ctypes.data):
            raise RuntimeError(L.moe_last_error().decode())
    if norm:
        d.preload_norm(i, w["gamma"].cpu().numpy(), EPS)
    d.synchronize()


def _hidden(case, seed, layer):
    return torch.randn((case["T"], case["H"]), device="cuda", generator=_gen(seed, 2, layer))


def _expert_inputs(case, seed):
    rng = np.random.default_rng([seed, 3])
    return rng.standard_normal((case["layers"], case["H"])).astype(np.float32)


def _lm_weights(case, seed):
    w = torch.randn((case["V"], case["H"]), device="cuda", generator=_gen(seed, 4)).mul_(0.02)
    return w.bfloat16() if case["bf16"] else w


def _lm_input(case, seed):
    return torch.randn(case["H"], device="cuda", generator=_gen(seed, 5))


def prepare(case, seed):
    op = case["op"]
    if op == "layer":
        d = pkg.GpuMoeDispatcher(case["H"], case["I"], CLAMP)
        if case["quant"]:
            d.set_act_quant(1)
        for i in range(case["layers"]):
            _load_layer(d, i, _layer_tensors(case, seed, i, case["E"]), case["E"], norm=case["norm"])
        xs = [_Buf(_hidden(case, seed, i)) for i in range(case["layers"])]
        ys = [_Buf(torch.empty_like(x.t)) for x in xs]
        return dict(op=op, d=d, xs=xs, ys=ys, T=case["T"], k=case["k"],
                    call=d.block_forward_device if case["norm"] else d.layer_forward_device)
    if op == "expert":
        d = pkg.GpuMoeDispatcher(case["H"], case["I"], CLAMP)
        for i in range(case["layers"]):
            _load_layer(d, i, _layer_tensors(case, seed, i, case["k"]), case["k"], router=False)
        return dict(op=op, d=d, xs=_expert_inputs(case, seed), k=case["k"])
    if op == "lm_head":
        d = pkg.GpuMoeDispatcher(case["H"], 32, CLAMP)
        w = _lm_weights(case, seed)
        torch.cuda.synchronize()
        if case["bf16"]:
            d.init_lm_head_bf16_device(w.data_ptr(), case["V"])
        else:
            d.init_lm_head(w.cpu().numpy(), case["V"])
        d.synchronize()
        return dict(op=op, d=d, x=_Buf(_lm_input(case, seed)), y=_Buf(torch.empty(case["V"], device="cuda")), V=case["V"])
    g = pkg.GpuTripleGen32(case["n"], case["t"])
    seeds = torch.randint(0, 1 << 31, (g.num_rounds(case["count"]),), device="cuda", generator=_gen(seed, 6), dtype=torch.int64)
    shape = (case["n"], case["count"]) if case["party"] < 0 else (case["count"],)
    outs = [_Buf(torch.empty(shape, dtype=torch.int32, device="cuda")) for _ in range(3)]
    return dict(op=op, g=g, seeds=_Buf(seeds.to(torch.int32)), outs=outs, count=case["count"], party=case["party"])


def run(state):
    op = state["op"]
    if op == "layer":
        s = _on()
        for i, (x, y) in enumerate(zip(state["xs"], state["ys"])):
            state["call"](i, x, state["T"], state["k"], y, s)
        return [y.t for y in state["ys"]]
    if op == "expert":
        return [state["d"].dispatch_expert_preloaded(x, i, e) for i, x in enumerate(state["xs"]) for e in range(state["k"])]
    if op == "lm_head":
        state["d"].dispatch_lm_head_device(state["x"], state["V"], state["y"], _on())
        return state["y"].t
    state["g"].generate_device(state["party"], state["count"], state["seeds"], *state["outs"], _on())
    return [o.t for o in state["outs"]]


# ---------------------------------------------------------------- what a pass cannot do without


def _expert_size(H, I):
    """Bytes of one expert: nibbles, a scale per 32 values, f32 biases."""
    return 3 * H * I * 17 // 32 + 4 * (2 * I + H)


def work(case):
    op = case["op"]
    if op == "layer":
        H, I, E, k, T = (case[n] for n in "HIEkT")
        active = E * (1.0 - (1.0 - k / E) ** T)  # experts that T tokens are expected to choose
        one_bytes = active * _expert_size(H, I) + 2 * E * H + 8 * T * H
        one_flops = 2 * T * (3 * k * H * I + E * H)
        return {"bytes": case["layers"] * one_bytes, "flops": case["layers"] * one_flops}
    if op == "expert":
        n = case["layers"] * case["k"]
        return {"bytes": n * (_expert_size(case["H"], case["I"]) + 8 * case["H"]), "flops": 6 * n * case["H"] * case["I"]}
    if op == "lm_head":
        w = case["V"] * case["H"]
        return {"bytes": w * (2 if case["bf16"] else 4) + 4 * (case["V"] + case["H"]), "flops": 2 * w}
    spr = case["n"] - 2 * case["t"]
    parties = case["n"] if case["party"] < 0 else 1
    return {"bytes": 12 * case["count"] * parties + 4 * -(-case["count"] // spr), "flops": 0}


def tolerance(case):
    """About four times what the path differs from the 64-bit results by: the grouped GEMM's
    activations (exact to 2^-13 of a block's maximum) 7e-5, the single token's 2e-5, the
    per-expert call's 4e-6, 32-bit sums 1.4e-7."""
    op = case["op"]
    if op == "beaver":
        return "exact"
    if op == "lm_head":
        return {"rel": 1e-6}
    if op == "expert":
        return {"rel": 2e-5}
    if case["quant"]:
        return {"rel": 3e-4}
    return {"rel": 1e-4 if case["T"] == 1 else 3e-4}


# ---------------------------------------------------------------- the same in 64 bits


def _dequant(blocks, scales):
    """[rows, nb, 16] nibble pairs and [rows, nb] scales to f64 [rows, 32 nb]."""
    lut = torch.tensor(E2M1 + tuple(-v for v in E2M1), dtype=torch.float64, device="cuda")
    b = blocks.to(torch.int64)
    v = torch.stack((lut[b & 15], lut[b >> 4]), dim=-1).flatten(-2)
    v = v * torch.exp2(scales.to(torch.float64) - 127.0).unsqueeze(-1)
    return v.flatten(-2)


def _mxfp6(v):
    """v [.., 32 n] quantised per 32 values to E2M3 with a power-of-two scale, to nearest even."""
    b = v.unflatten(-1, (-1, 32))
    amax = b.abs().amax(-1, keepdim=True)
    _, e = torch.frexp(amax)  # amax = f 2^e, f in [1/2, 1)
    scale = torch.where(amax > 0, torch.exp2(e.to(b.dtype) - 3.0), torch.ones_like(amax))
    u = b / scale
    _, ue = torch.frexp(u.abs().clamp(min=1.0))
    step = torch.exp2(ue.to(b.dtype) - 4.0)
    u = (torch.round(u / step) * step).clamp(-7.5, 7.5)
    return (u * scale).flatten(-2)


def _ffn(x, w, e, quant):
    gu = x @ _dequant(w["gu_blocks"][e], w["gu_scales"][e]).T + w["gu_bias"][e].double()
    gate, up = gu[:, 0::2].clamp(max=CLAMP), gu[:, 1::2].clamp(-CLAMP, CLAMP)
    h = (up + 1.0) * gate * torch.sigmoid(1.702 * gate)
    if quant:
        h = _mxfp6(h)
    y = h @ _dequant(w["d_blocks"][e], w["d_scales"][e]).T + w["d_bias"][e].double()
    return y.clamp(-65504.0, 65504.0)


def _exact_layer(case, seed, i):
    w, x = _layer_tensors(case, seed, i, case["E"]), _hidden(case, seed, i).double()
    n = x
    if case["norm"]:
        n = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w["gamma"].double()
    top, idx = torch.topk(n @ w["router_w"].double().T, case["k"], dim=-1)
    p = torch.softmax(top, dim=-1)
    m = _mxfp6(n) if case["quant"] else n
    y = torch.zeros_like(x)
    for e in idx.unique().tolist():
        t, slot = (idx == e).nonzero(as_tuple=True)
        y.index_add_(0, t, _ffn(m[t], w, e, case["quant"]) * p[t, slot].unsqueeze(-1))
    return x + y if case["norm"] else y


def exact(case, seed):
    op = case["op"]
    if op == "layer":
        return [_exact_layer(case, seed, i) for i in range(case["layers"])]
    if op == "expert":
        out = []
        for i, x in enumerate(_expert_inputs(case, seed)):
            w = _layer_tensors(case, seed, i, case["k"])
            x = torch.from_numpy(x).cuda().double().unsqueeze(0)
            out += [_ffn(x, w, e, False)[0].cpu().numpy() for e in range(case["k"])]
        return out
    if op == "lm_head":
        w, x = _lm_weights(case, seed), _lm_input(case, seed).double()
        return torch.cat([c.double() @ x for c in w.split(16384)])
    return None  # whole numbers of a field: they are the same or they are wrong
