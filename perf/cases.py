"""What a program built on this package has the GPU do, as measurable cases.

Each case is one building block of a served model (an MLP, a QKV stage, an
attention layer, a routed-expert layer, one whole pi05 prediction), called
through the package's public entry points. Programs of this kind capture their
launch-bound loops into HIP graphs, as ``Pi05Forward.capture`` does, so blocks of
up to 1024 tokens run as one captured graph of a few layers with weights of
their own; larger blocks and the ``nn.Linear`` drop-in run eagerly.

``exact`` states the same computation in 64 bits. Quantizing a projection's
operands to E4M3 is part of what these blocks compute, so it is kept there, with
the recipe's own scale (max(amax, 1e-12) * fl32(1/448)); intermediate results
that the kernels store in 16 bits are not rounded.
"""
import math

import torch

from instinctflash_amd import kernels as ifx
from instinctflash_amd.kernels.attention import SplitWorkspace, split_count
from instinctflash_amd.kernels.fp8 import quantize_weight
from instinctflash_amd.kernels.wan import wan_rope_tables
from instinctflash_amd.modules import Gfx950FP8Linear
from instinctflash_amd.pi05_forward import Pi05Dims, Pi05Forward, random_pi05

F32, F64, BF16, F16 = torch.float32, torch.float64, torch.bfloat16, torch.float16
DTYPES = {"bf16": BF16, "fp16": F16}
INV448 = 1.0 / 448.0


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # GR00T-style action head: 16 action tokens through a DiT stack's MLPs, every layer's
        # weights streamed from HBM. The smallest calls: launches and latency count.
        dict(name="head_mlp", kind="mlp", M=16, D=1536, FF=6144, act="gelu_tanh", gate=False, layers=16),
        # SigLIP vision tower MLP of three 256-patch views: FF = 4304 is no multiple of the
        # 128-byte K step.
        dict(name="vision_mlp", kind="mlp", M=768, D=1152, FF=4304, act="gelu_tanh", gate=False, layers=4),
        # PaliGemma prefix MLP of pi05: 768 image rows and 48 prompt rows, GeGLU.
        dict(name="prefix_mlp", kind="mlp", M=816, D=2048, FF=16384, act="geglu", gate=False, layers=2),
        # Wan-style video DiT block FFN over 8192 latent tokens with adaLN-gated residual.
        dict(name="video_mlp", kind="mlp", M=8192, D=3072, FF=14336, act="gelu_tanh", gate=True, layers=1),
        # Qwen2.5-style decoder QKV stage of a VLA prefill: pre-norm, projection with bias, M-RoPE
        # and KV-cache store (16 query / 2 KV heads).
        dict(name="decoder_qkv", kind="qkv", M=1024, D=2048, HQ=16, HKV=2, HD=128, layers=4),
        # Wan DiT QKV stage: adaLN pre-norm, raw projection, full-width q/k norm, 3-D rotary, KV pools.
        dict(name="video_qkv", kind="wan", M=8192, H=24, HD=128, layers=1),
        # pi05 expert attention: 50 action tokens over an 866-row cache in 18 layers, writing the
        # output projection's E4M3 operand.
        dict(name="chunk_attention", kind="attention", B=1, Tq=50, Tk=866, HQ=8, HKV=1, HD=256, dtype="fp16",
             causal=False, fp8=True, layers=18),
        # Wan DiT self-attention over one 8192-token latent clip.
        dict(name="video_attention", kind="attention", B=1, Tq=8192, Tk=8192, HQ=24, HKV=24, HD=128, dtype="bf16",
             causal=False, fp8=False, layers=1),
        # Routed-expert layer of a VLA action expert: pre-norm with the router, dense gate|up over 32
        # concatenated experts and the shared one, routed SwiGLU, down.
        dict(name="moe_layer", kind="moe", M=51, D=768, experts=32, group=512, shared=704, top_k=4, layers=4),
        # An engine written against the unfused kernel seam (raw gemm, then a consumer), with an odd
        # number of prompt tokens.
        dict(name="seam_mlp", kind="seam", M=333, D=2048, FF=11008, act="silu", layers=2),
        # nn.Linear drop-in with per-tensor activation scales, called eagerly.
        dict(name="module_linear", kind="module", M=50, K=1024, N=4096, bias=True),
        # One whole pi05 prediction: three views, 48 prompt tokens, 50 actions, 10 flow steps.
        dict(name="pi05_chunk", kind="pi05", views=3, prompt=48, chunk=50, steps=10),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _layers(M):
    return 8 if M <= 64 else 2 if M <= 1024 else 1


MAX_MLP = 8192 * 3072 * 14336
MAX_ATTENTION = 24 * 128 * 8192 * 8192


def draw(rng):
    kind = rng.choice(["mlp", "mlp", "mlp", "qkv", "wan", "attention", "attention", "moe", "seam", "module", "pi05"])
    if kind in ("mlp", "seam"):
        M = _log_int(rng, 1, 8192)
        D, FF = 16 * _log_int(rng, 32, 256), 16 * _log_int(rng, 64, 1024)
        while M * D * FF > MAX_MLP:
            M //= 2
        if kind == "seam":
            return dict(kind=kind, M=M, D=D, FF=FF, act=rng.choice(["gelu_tanh", "silu"]), layers=_layers(M))
        act = rng.choice(["gelu_tanh", "geglu", "swiglu"])
        return dict(kind=kind, M=M, D=D, FF=FF, act=act, gate=act == "gelu_tanh" and rng.random() < 0.5,
                    layers=_layers(M))
    if kind == "qkv":
        M = _log_int(rng, 1, 4096)
        HQ, HKV = rng.choice([(8, 1), (16, 2), (16, 16), (28, 4), (32, 8)])
        return dict(kind=kind, M=M, D=16 * _log_int(rng, 48, 224), HQ=HQ, HKV=HKV, HD=rng.choice([64, 128]),
                    layers=_layers(M))
    if kind == "wan":
        M = _log_int(rng, 64, 8192)
        return dict(kind=kind, M=M, H=rng.choice([12, 16, 24]), HD=128, layers=_layers(M))
    if kind == "attention":
        HQ, HKV, HD = rng.choice([(8, 1, 256), (16, 2, 128), (16, 16, 72), (24, 24, 128), (28, 4, 128), (16, 16, 64)])
        if rng.random() < 0.4:
            # an action chunk over its prefix cache, with the E4M3 output row
            Tq = rng.randint(8, 64)
            return dict(kind=kind, B=1, Tq=Tq, Tk=Tq + rng.randint(128, 2048), HQ=HQ, HKV=HKV, HD=HD, dtype="fp16",
                        causal=False, fp8=True, layers=8)
        T, B = _log_int(rng, 64, 8192), rng.choice([1, 1, 2, 3])
        while B * HQ * HD * T * T > MAX_ATTENTION:
            T //= 2
        return dict(kind=kind, B=B, Tq=T, Tk=T, HQ=HQ, HKV=HKV, HD=HD, dtype=rng.choice(["bf16", "fp16"]),
                    causal=B == 1 and rng.random() < 0.4, fp8=False, layers=_layers(B * T))
    if kind == "moe":
        M = _log_int(rng, 1, 512)
        return dict(kind=kind, M=M, D=128 * rng.randint(4, 16), experts=rng.choice([8, 16, 32]),
                    group=rng.choice([256, 512]), shared=64 * rng.randint(2, 16), top_k=rng.choice([2, 4]),
                    layers=_layers(M))
    if kind == "module":
        return dict(kind=kind, M=_log_int(rng, 1, 4096), K=16 * _log_int(rng, 32, 512), N=16 * _log_int(rng, 32, 512),
                    bias=rng.random() < 0.5)
    return dict(kind=kind, views=rng.randint(1, 3), prompt=rng.randint(1, 48), chunk=rng.randint(10, 50),
                steps=rng.randint(4, 10))


# ---------------------------------------------------------------------------
# inputs, made on the GPU from the seed alone
# ---------------------------------------------------------------------------

class _Random:
    def __init__(self, seed):
        self.dev = torch.device("cuda", torch.cuda.current_device())
        self.g = torch.Generator(device=self.dev).manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=F32):
        return torch.randn(*shape, generator=self.g, device=self.dev).mul_(std).to(dtype)

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, generator=self.g, device=self.dev).mul_(hi - lo).add_(lo)


def _mlp_inputs(c, r):
    """Activations of unit scale with a few outlier channels (Qwen2.5-style), weights N(0, 0.02)."""
    rows = 2 * c["FF"] if c["act"] in ("geglu", "swiglu", "silu") or c["kind"] == "seam" else c["FF"]
    x = r.normal(c["M"], c["D"])
    x[:, torch.randperm(c["D"], generator=r.g, device=r.dev)[:4]] *= 10.0
    t = dict(x=x.to(BF16), up=r.normal(rows, c["D"], std=0.02), down=r.normal(c["D"], c["FF"], std=0.02),
             residual=r.normal(c["M"], c["D"], dtype=BF16))
    if c.get("gate"):
        t["gate"] = r.uniform(c["D"]).to(BF16)
    if c["kind"] == "seam":
        t.update(hidden=x, norm1=r.uniform(c["D"], lo=0.5, hi=1.5), norm2=r.uniform(c["D"], lo=0.5, hi=1.5))
    return t


def _qkv_inputs(c, r):
    n = (c["HQ"] + 2 * c["HKV"]) * c["HD"]
    return dict(hidden=r.normal(c["M"], c["D"]), norm=r.uniform(c["D"], lo=0.5, hi=1.5),
                w=r.normal(n, c["D"], std=0.02), bias=r.normal(n, std=0.1),
                inv_freq=torch.tensor([1e6 ** (-2.0 * i / c["HD"]) for i in range(c["HD"] // 2)], device=r.dev),
                sections=(torch.arange(c["HD"] // 2, device=r.dev) % 3).int(),
                pos=torch.stack([torch.arange(c["M"], device=r.dev) + 5 * s for s in range(3)], 1).float())


def _wan_inputs(c, r):
    D = c["H"] * c["HD"]
    side = 32
    t = torch.arange(c["M"], device=r.dev)
    inv_freq, sections = wan_rope_tables(c["HD"], device=r.dev)
    return dict(hidden=r.normal(c["M"], D), scale=r.normal(D, std=0.1), shift=r.normal(D, std=0.1),
                w=r.normal(3 * D, D, std=0.02), bias=r.normal(3 * D, std=0.1),
                q_norm=r.uniform(D, lo=0.5, hi=1.5), k_norm=r.uniform(D, lo=0.5, hi=1.5),
                pos=torch.stack([t // (side * side), t // side % side, t % side], 1).float(),
                inv_freq=inv_freq, sections=sections,
                slots=torch.randperm(c["M"], generator=r.g, device=r.dev).int())


def _attention_inputs(c, r):
    dt = DTYPES[c["dtype"]]
    return dict(q=r.normal(c["B"], c["Tq"], c["HQ"], c["HD"], std=1.5, dtype=dt),
                k=r.normal(c["B"], c["Tk"], c["HKV"], c["HD"], dtype=dt),
                v=r.normal(c["B"], c["Tk"], c["HKV"], c["HD"], dtype=dt))


def _moe_inputs(c, r):
    F = c["experts"] * c["group"] + c["shared"]
    return dict(hidden=r.normal(c["M"], c["D"]), scale=r.normal(c["D"], std=0.1), shift=r.normal(c["D"], std=0.1),
                router=r.normal(c["experts"], c["D"], std=0.05), e_bias=r.normal(c["experts"], std=0.01),
                up=r.normal(2 * F, c["D"], std=0.02), down=r.normal(c["D"], F, std=0.02),
                residual=r.normal(c["M"], c["D"], dtype=BF16))


def _module_inputs(c, r):
    t = dict(x=r.normal(c["M"], c["K"], dtype=BF16), w=r.normal(c["N"], c["K"], std=0.02, dtype=BF16))
    if c["bias"]:
        t["bias"] = r.normal(c["N"], std=0.1, dtype=BF16)
    return t


def _pi05_dims(c):
    return Pi05Dims(views=c["views"], max_prompt=48, chunk=c["chunk"], steps=c["steps"])


def _pi05_inputs(c, r):
    d = _pi05_dims(c)
    return dict(images=r.uniform(d.views, 3, 224, 224, lo=-1.0), prompt=r.normal(c["prompt"], d.lm_d),
                noise=r.normal(d.chunk, d.action))


INPUTS = {"mlp": _mlp_inputs, "seam": _mlp_inputs, "qkv": _qkv_inputs, "wan": _wan_inputs,
          "attention": _attention_inputs, "moe": _moe_inputs, "module": _module_inputs, "pi05": _pi05_inputs}


def _inputs(c, seed):
    """Every layer's inputs; layers differ in weights and activations alike."""
    r = _Random(seed)
    return [INPUTS[c["kind"]](c, r) for _ in range(c.get("layers", 1))]


# ---------------------------------------------------------------------------
# the program: weights and buffers once, then one call per pass
# ---------------------------------------------------------------------------

def _empty(shape, dtype, dev):
    return torch.empty(shape, dtype=dtype, device=dev)


def _op(M, K, dev):
    """The E4M3 operand of a projection and its token scales."""
    return _empty((M, K), ifx.E4M3, dev), _empty((M,), F32, dev)


def _make_mlp(c, t, dev):
    M, D, FF = c["M"], c["D"], c["FF"]
    up, down = quantize_weight(t["up"]), quantize_weight(t["down"])
    if c["act"] != "gelu_tanh":
        up = ifx.pack_glu(up)
    h, out = _empty((M, FF), BF16, dev), _empty((M, D), BF16, dev)
    if M <= 64:  # decode and action-head sizes: the tile layout of both operands
        up, down, quant = ifx.pack_skinny(up), ifx.pack_skinny(down), ifx.quant_rows_tiled
        (q1, s1), (q2, s2) = quant(t["x"]), quant(h.zero_())
    else:
        quant, (q1, s1), (q2, s2) = ifx.quant_rows, _op(M, D, dev), _op(M, FF, dev)

    def call():
        quant(t["x"], q1, s1)
        ifx.linear(q1, s1, up, out=h, act=c["act"])
        quant(h, q2, s2)
        return ifx.linear(q2, s2, down, out=out, residual=t["residual"], gate=t.get("gate"))
    return call


def _make_seam(c, t, dev):
    M, D, FF = c["M"], c["D"], c["FF"]
    up, down = quantize_weight(t["up"]), quantize_weight(t["down"])
    stream = _empty((M, D), F32, dev)
    q1, s1 = _op(M, D, dev)
    q2, s2 = _op(M, FF, dev)
    q3, s3 = _op(M, D, dev)
    gu, y = _empty((M, 2 * FF), BF16, dev), _empty((M, D), BF16, dev)
    act = ifx.SILU if c["act"] == "silu" else ifx.GELU_TANH

    def call():
        stream.copy_(t["hidden"])
        ifx.residual_norm_quant(stream, weight=t["norm1"], q=q1, q_scale=s1, write_res=False)
        ifx.gemm(q1, up, gu)
        ifx.gated_act_quant(gu, q2, s2, row=s1, col=up.scale, act=act)
        ifx.gemm(q2, down, y)
        ifx.residual_norm_quant(stream, delta=y, delta_row=s2, delta_col=down.scale, weight=t["norm2"], q=q3,
                                q_scale=s3)
        return [stream, q3.view(torch.uint8), s3]
    return call


def _make_qkv(c, t, dev):
    M, HQ, HKV, HD = c["M"], c["HQ"], c["HKV"], c["HD"]
    w = quantize_weight(t["w"], t["bias"])
    q8, s = _op(M, c["D"], dev)
    raw = _empty((M, (HQ + 2 * HKV) * HD), BF16, dev)
    q = _empty((M, HQ, HD), BF16, dev)
    k, v = torch.zeros(M + 64, HKV, HD, dtype=BF16, device=dev), torch.zeros(M + 64, HKV, HD, dtype=BF16, device=dev)

    def call():
        ifx.residual_norm_quant(t["hidden"], weight=t["norm"], q=q8, q_scale=s, write_res=False)
        ifx.linear(q8, s, w, out=raw)
        ifx.qkv_split(raw, q, k, v, heads_q=HQ, heads_kv=HKV, head_dim=HD, inv_freq=t["inv_freq"], pos=t["pos"],
                      sections=t["sections"], kv_base=64)
        return [q, k, v]
    return call


def _make_wan(c, t, dev):
    M, D = c["M"], c["H"] * c["HD"]
    w = quantize_weight(t["w"])
    q8, s = _op(M, D, dev)
    raw, q = _empty((M, 3 * D), BF16, dev), _empty((M, D), BF16, dev)
    k, v = _empty((1, M, D), BF16, dev), _empty((1, M, D), BF16, dev)

    def call():
        ifx.residual_norm_quant(t["hidden"], layernorm=True, mod_scale=t["scale"], mod_shift=t["shift"], q=q8,
                                q_scale=s, write_res=False)
        ifx.gemm(q8, w, raw)
        ifx.wan_qkv(raw, q, heads=c["H"], head_dim=c["HD"], tokens=M, k_pool=k, v_pool=v, slots=t["slots"], row=s,
                    col=w.scale, bias=t["bias"], q_norm=t["q_norm"], k_norm=t["k_norm"], pos=t["pos"],
                    sections=t["sections"], inv_freq=t["inv_freq"])
        return [q, k, v]
    return call


def _make_attention(c, t, dev):
    B, Tq, Tk, HQ, HKV, HD = (c[n] for n in ("B", "Tq", "Tk", "HQ", "HKV", "HD"))
    if c["fp8"]:
        split = SplitWorkspace(B, Tq, HQ, HKV, HD, max(2, split_count(B, Tq, HQ, HKV, Tk)), dev)
        q8, s = _op(Tq, HQ * HD, dev)

        def call():
            ifx.attention(t["q"], t["k"], t["v"], split=split, q8=q8, q8_scale=s)
            return [q8, s]
        return call
    out = _empty((B, Tq, HQ, HD), DTYPES[c["dtype"]], dev)
    return lambda: ifx.attention(t["q"], t["k"], t["v"], out=out, causal=c["causal"])


def _make_moe(c, t, dev):
    M, D, E = c["M"], c["D"], c["experts"]
    F = E * c["group"] + c["shared"]
    up, down = quantize_weight(t["up"]), quantize_weight(t["down"])
    q1, s1 = _op(M, D, dev)
    q2, s2 = _op(M, F, dev)
    gu, out, route = _empty((M, 2 * F), BF16, dev), _empty((M, D), BF16, dev), _empty((M, E), F32, dev)

    def call():
        ifx.residual_norm_quant(t["hidden"], mod_scale=t["scale"], mod_shift=t["shift"], q=q1, q_scale=s1,
                                write_res=False, router=(t["router"], t["e_bias"], route, c["top_k"], 4.0))
        ifx.gemm(q1, up, gu)
        ifx.moe_act_quant(gu, q2, s2, route, row=s1, col=up.scale, experts=E, group=c["group"],
                          n_routed=E * c["group"])
        ifx.linear(q2, s2, down, out=out, residual=t["residual"])
        return [out, route]
    return call


def _make_module(c, t, dev):
    lin = torch.nn.Linear(c["K"], c["N"], bias=c["bias"], device=dev, dtype=BF16)
    with torch.no_grad():
        lin.weight.copy_(t["w"])
        if c["bias"]:
            lin.bias.copy_(t["bias"])
    module = Gfx950FP8Linear(lin)
    return lambda: module(t["x"])


MAKE = {"mlp": _make_mlp, "seam": _make_seam, "qkv": _make_qkv, "wan": _make_wan, "attention": _make_attention,
        "moe": _make_moe, "module": _make_module}


def prepare(case, seed):
    inputs = _inputs(case, seed)
    dev = torch.device("cuda", torch.cuda.current_device())
    if case["kind"] == "pi05":
        model = Pi05Forward(random_pi05(_pi05_dims(case), dev, seed=seed), dev)
        model.set_inputs(**{"images": inputs[0]["images"], "prompt_rows": inputs[0]["prompt"],
                            "noise": inputs[0]["noise"]})
        return dict(graph=model.capture(), outputs=model.actions, keep=model)
    calls = [MAKE[case["kind"]](case, t, dev) for t in inputs]
    tokens = case["B"] * case["Tq"] if case["kind"] == "attention" else case["M"]
    if case["kind"] == "module" or tokens > 1024:
        return dict(calls=calls)

    def layers():
        return [call() for call in calls]
    side = torch.cuda.Stream(dev)
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side):
        layers()
    torch.cuda.current_stream(dev).wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        outputs = layers()
    return dict(graph=graph, outputs=outputs, keep=(calls, side))


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["outputs"]
    return [call() for call in state["calls"]]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    c, kind = case, case["kind"]
    if kind in ("mlp", "seam"):
        M, D, FF = c["M"], c["D"], c["FF"]
        rows = FF if c["act"] == "gelu_tanh" and kind == "mlp" else 2 * FF
        weights, act = (rows + FF) * D, 6 * M * D if kind == "mlp" else 9 * M * D
        flops = 2 * M * D * (rows + FF)
    elif kind in ("qkv", "wan"):
        D = c["D"] if kind == "qkv" else c["H"] * c["HD"]
        n = (c["HQ"] + 2 * c["HKV"]) * c["HD"] if kind == "qkv" else 3 * D
        weights, act, flops = n * D, c["M"] * (4 * D + 2 * n), 2 * c["M"] * n * D
    elif kind == "attention":
        q = c["B"] * c["Tq"] * c["HQ"] * c["HD"]
        weights, act = 0, q * (3 if c["fp8"] else 4) + 4 * c["B"] * c["Tk"] * c["HKV"] * c["HD"]
        flops = 4 * q * c["Tk"] / (2 if c["causal"] else 1)
    elif kind == "moe":
        F = c["experts"] * c["group"] + c["shared"]
        weights, act = 3 * F * c["D"] + 4 * c["experts"] * c["D"], 8 * c["M"] * c["D"] + 4 * c["M"] * c["experts"]
        flops = 6 * c["M"] * F * c["D"]
    elif kind == "module":
        weights, act, flops = c["N"] * c["K"], 2 * c["M"] * (c["K"] + c["N"]), 2 * c["M"] * c["N"] * c["K"]
    else:
        return _pi05_work(c)
    layers = c.get("layers", 1)
    return {"bytes": layers * (weights + act), "flops": layers * flops}


def _pi05_work(c):
    d = _pi05_dims(c)
    ctx, S = d.heads * d.head_dim, d.image_rows + c["prompt"]
    vision = 4 * d.vis_d * d.vis_d + 2 * d.vis_d * d.vis_ff
    prefix = d.qkv_n * d.lm_d + ctx * d.lm_d + 3 * d.lm_d * d.lm_ff
    expert = d.qkv_n * d.ex_d + ctx * d.ex_d + 3 * d.ex_d * d.ex_ff
    last = d.qkv_n * d.lm_d  # the prefix's last layer only feeds the expert's cache
    params = d.vision_layers * vision + d.vis_d * d.lm_d + (d.prefix_layers - 1) * prefix + last + \
        d.expert_layers * expert
    flops = 2 * d.image_rows * (d.vision_layers * vision + d.vis_d * d.lm_d)
    flops += 4 * d.vision_layers * d.image_rows * d.patches * d.vis_d
    flops += 2 * S * ((d.prefix_layers - 1) * prefix + last) + 4 * (d.prefix_layers - 1) * S * S * ctx
    flops += d.steps * d.expert_layers * (2 * d.chunk * expert + 4 * d.chunk * (S + d.chunk) * ctx)
    act = 4 * d.views * 3 * 224 * 224 + 4 * c["prompt"] * d.lm_d + 8 * d.chunk * d.action
    return {"bytes": params + act, "flops": flops}


# A projection's operands are E4M3 and results are stored in bf16: another order of sums
# moves a stored value by a bf16 step and, ahead of a quantizer, an operand by an E4M3 step.
TOLERANCE = {
    "mlp": {"rel": 1e-2, "max": 0.2},
    "seam": {"rel": 1e-2, "max": 0.2, "differ": 0.01},
    "qkv": {"rel": 1e-2, "max": 0.2},
    "wan": {"rel": 1e-2, "max": 0.2},
    "attention": {"rel": 1e-2, "max": 0.1},
    "moe": {"rel": 1e-2, "max": 0.2},
    "module": {"rel": 1e-2, "max": 0.1},
    # a change of one operand code travels through 63 layers and ten flow steps
    "pi05": {"rel": 2e-2, "max": 0.2},
}


def tolerance(case):
    if case["kind"] == "attention" and case["fp8"]:
        # outputs are E4M3 codes: a partial sum's last bit moves a code at a tie by a whole step (1/8)
        return {"rel": 2e-2, "max": 0.3}
    return TOLERANCE[case["kind"]]


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _scale(amax):
    return (amax.to(F32).clamp_min(1e-12) * torch.tensor(INV448, dtype=F32)).double()


def _codes(x, s):
    return (x / s).clamp(-448.0, 448.0).to(F32).to(ifx.E4M3).double()


def _fp8(x):
    """A matrix as its E4M3 rows carry it: codes times the row's scale."""
    s = _scale(x.double().abs().amax(dim=1))[:, None]
    return _codes(x.double(), s) * s


def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))


def _silu(x):
    return x * torch.sigmoid(x)


def _rms(x, eps=1e-6):
    return x * torch.rsqrt(x.square().mean(dim=1, keepdim=True) + eps)


def _layer_norm(x, eps=1e-6):
    x = x - x.mean(dim=1, keepdim=True)
    return x * torch.rsqrt(x.square().mean(dim=1, keepdim=True) + eps)


def _glu(c, gu):
    F = gu.shape[1] // 2
    act = _silu if c["act"] in ("swiglu", "silu") else _gelu
    return act(gu[:, :F]) * gu[:, F:]


def _softmax_attention(q, k, v, scale, causal=False):
    """q [Tq, H, D] over k / v [Tk, Hkv, D], one head and 2048 query rows at a time."""
    group = q.shape[1] // k.shape[1]
    out = torch.empty(q.shape, dtype=F64, device=q.device)
    for h in range(q.shape[1]):
        kh, vh = k[:, h // group].double(), v[:, h // group].double()
        for t in range(0, q.shape[0], 2048):
            a = (q[t:t + 2048, h].double() @ kh.t()) * scale
            if causal:
                rows = torch.arange(t, t + a.shape[0], device=q.device)[:, None]
                a.masked_fill_(torch.arange(a.shape[1], device=q.device) > rows, -math.inf)
            out[t:t + 2048, h] = a.softmax(dim=1) @ vh
    return out


def _angles(t):
    # the angle is a 32-bit product in these models; its sine and cosine are exact here
    return (t["pos"][:, t["sections"].long()] * t["inv_freq"]).double()


def _rotate_halves(x, ang):
    half = x.shape[-1] // 2
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]
    lo, hi = x[..., :half], x[..., half:]
    return torch.cat([lo * cos - hi * sin, hi * cos + lo * sin], dim=-1)


def _rotate_pairs(x, ang):
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]
    even, odd = x[..., 0::2], x[..., 1::2]
    return torch.stack([even * cos - odd * sin, odd * cos + even * sin], dim=-1).flatten(-2)


def _exact_mlp(c, t):
    up = _fp8(t["x"]) @ _fp8(t["up"]).t()
    y = _fp8(_gelu(up) if c["act"] == "gelu_tanh" else _glu(c, up)) @ _fp8(t["down"]).t()
    if "gate" in t:
        y = y * t["gate"].double()
    return y + t["residual"].double()


def _exact_seam(c, t):
    x = t["hidden"].double()
    h = _glu(c, _fp8(_rms(x) * t["norm1"].double()) @ _fp8(t["up"]).t())
    x = x + _fp8(h) @ _fp8(t["down"]).t()
    s = _scale((_rms(x) * t["norm2"].double()).abs().amax(dim=1))
    return [x, None, s]


def _exact_qkv(c, t):
    M, HQ, HKV, HD = c["M"], c["HQ"], c["HKV"], c["HD"]
    raw = _fp8(_rms(t["hidden"].double()) * t["norm"].double()) @ _fp8(t["w"]).t() + t["bias"].double()
    heads, ang = raw.view(M, HQ + 2 * HKV, HD), _angles(t)

    def cache(x):
        return torch.cat([torch.zeros(64, HKV, HD, dtype=F64, device=x.device), x])
    return [_rotate_halves(heads[:, :HQ], ang), cache(_rotate_halves(heads[:, HQ:HQ + HKV], ang)),
            cache(heads[:, HQ + HKV:])]


def _exact_wan(c, t):
    M, H, HD = c["M"], c["H"], c["HD"]
    D = H * HD
    x = _layer_norm(t["hidden"].double()) * (1.0 + t["scale"].double()) + t["shift"].double()
    raw = _fp8(x) @ _fp8(t["w"]).t() + t["bias"].double()
    ang = _angles(t)

    def rotated(x, norm):
        return _rotate_pairs((_rms(x) * norm.double()).view(M, H, HD), ang).reshape(M, D)

    def pool(x):
        out = torch.empty(1, M, D, dtype=F64, device=x.device)
        out[0, t["slots"].long()] = x
        return out
    return [rotated(raw[:, :D], t["q_norm"]), pool(rotated(raw[:, D:2 * D], t["k_norm"])), pool(raw[:, 2 * D:])]


def _exact_attention(c, t):
    out = torch.stack([_softmax_attention(t["q"][b], t["k"][b], t["v"][b], c["HD"] ** -0.5, c["causal"])
                       for b in range(c["B"])])
    if not c["fp8"]:
        return out
    rows = out.view(c["Tq"], -1)
    s = _scale(rows.abs().amax(dim=1))
    return [_codes(rows, s[:, None]), s]


def _exact_moe(c, t):
    E, M = c["experts"], c["M"]
    y = _rms(t["hidden"].double()) * (1.0 + t["scale"].double()) + t["shift"].double()
    score = torch.sigmoid(y @ t["router"].double().t())
    chosen = (score + t["e_bias"].double()).topk(c["top_k"], dim=1).indices
    route = torch.zeros_like(score).scatter_(1, chosen, score.gather(1, chosen))
    route = 4.0 * route / route.sum(dim=1, keepdim=True)
    gu = _fp8(y) @ _fp8(t["up"]).t()
    F = gu.shape[1] // 2
    weight = torch.ones(M, F, dtype=F64, device=gu.device)
    weight[:, :E * c["group"]] = route.repeat_interleave(c["group"], dim=1)
    out = _fp8(_silu(gu[:, :F]) * gu[:, F:] * weight) @ _fp8(t["down"]).t()
    return [out + t["residual"].double(), route]


def _exact_module(c, t):
    def tensor(x):
        s = _scale(x.double().abs().amax())
        return _codes(x.double(), s) * s
    y = tensor(t["x"]) @ tensor(t["w"]).t()
    return y + t["bias"].double() if c["bias"] else y


def _exact_pi05(c, inputs, seed):
    dev = inputs["images"].device
    d = _pi05_dims(c)
    p = random_pi05(d, dev, seed=seed, keep_plain=True)  # its weights, as drawn and quantized

    def lin(x, name):
        w = p.plain[name]
        y = _fp8(x) @ (w.w.double() * w.scale.double()[:, None]).t()
        return y if w.bias is None else y + w.bias.double()

    def norm(x, affine):
        return _layer_norm(x) * affine[0].double() + affine[1].double()

    def geglu(gu):
        return _glu(dict(act="geglu"), gu)
    T, n, HD = d.image_rows, c["prompt"], d.head_dim
    pix = inputs["images"].view(d.views, 3, 16, 14, 16, 14).permute(0, 2, 4, 3, 5, 1).reshape(T, 588)
    x = pix.half().double() @ p.patch_w.double() + p.patch_b.double()
    x = (x.view(d.views, d.patches, d.vis_d) + p.pos_emb.double()).view(T, d.vis_d)
    for i, blk in enumerate(p.vision):
        qkv = lin(norm(x, blk.ln1), f"v{i}.qkv").view(d.views, d.patches, 3, d.vis_heads, d.vis_hd)
        ctx = torch.cat([_softmax_attention(v[:, 0], v[:, 1], v[:, 2], d.vis_hd ** -0.5) for v in qkv])
        x = x + lin(ctx.view(T, d.vis_d), f"v{i}.o")
        x = x + lin(_gelu(lin(norm(x, blk.ln2), f"v{i}.fc1")), f"v{i}.fc2")
    x = torch.cat([lin(norm(x, p.post_ln), "projector"), inputs["prompt"].double()])
    S, A = T + n, d.chunk
    inv = torch.tensor([10000.0 ** (-2.0 * i / HD) for i in range(HD // 2)], device=dev)
    ang = (torch.arange(S + A, device=dev).float()[:, None] * inv).double()
    keys, values = [], []
    for i, blk in enumerate(p.prefix):
        qkv = lin(_rms(x), f"p{i}.qkv").view(S, d.heads + 2, HD)
        keys.append(_rotate_halves(qkv[:, d.heads:d.heads + 1], ang[:S]))
        values.append(qkv[:, d.heads + 1:])
        if blk.o is None:
            break
        ctx = _softmax_attention(_rotate_halves(qkv[:, :d.heads], ang[:S]), keys[i], values[i], HD ** -0.5)
        x = x + lin(ctx.view(S, -1), f"p{i}.o")
        x = x + lin(geglu(lin(_rms(x), f"p{i}.gate_up")), f"p{i}.down")
    act = inputs["noise"].double()
    for step in range(d.steps):
        ma, mf = p.mod_attn[step].double(), p.mod_ffn[step].double()
        x = act @ p.action_in[0].double() + p.action_in[1].double()
        for i in range(d.expert_layers):
            qkv = lin(_rms(x) * (1.0 + ma[i, 0]) + ma[i, 1], f"e{i}.qkv").view(A, d.heads + 2, HD)
            k = torch.cat([keys[i], _rotate_halves(qkv[:, d.heads:d.heads + 1], ang[S:])])
            v = torch.cat([values[i], qkv[:, d.heads + 1:]])
            ctx = _softmax_attention(_rotate_halves(qkv[:, :d.heads], ang[S:]), k, v, HD ** -0.5)
            x = x + lin(ctx.view(A, -1), f"e{i}.o") * ma[i, 2]
            h = geglu(lin(_rms(x) * (1.0 + mf[i, 0]) + mf[i, 1], f"e{i}.gate_up"))
            x = x + lin(h, f"e{i}.down") * mf[i, 2]
        out = _rms(x) * (1.0 + p.mod_final[step, 0].double()) + p.mod_final[step, 1].double()
        act = act - (out @ p.action_out[0].double() + p.action_out[1].double()) / d.steps
    return act


EXACT = {"mlp": _exact_mlp, "seam": _exact_seam, "qkv": _exact_qkv, "wan": _exact_wan, "attention": _exact_attention,
         "moe": _exact_moe, "module": _exact_module}


def exact(case, seed):
    inputs = _inputs(case, seed)
    if case["kind"] == "pi05":
        return _exact_pi05(case, inputs[0], seed)
    return [EXACT[case["kind"]](case, t) for t in inputs]
