"""The workloads that this library's speed is judged on: what a program that runs
MLX 4-bit models has it compute, through the package's public entry points.

A case is a dict of plain values.  Its "work" names one of these paths:

    linear   one projection, fp16 in: matmul_q4 (fp16 out), matmul_q4_fast (the
             M > 1 kernels), or matmul_q4_fast_f32 (fp32 out)
    layer    the five calls of a decoder layer over M rows (a prompt, or M
             sequences decoded together): input norm, q|k|v, o + residual +
             norm, gate/up with SiLU, down + residual + the next layer's norm;
             the attention output is an input (attention is the caller's)
    geglu    a text encoder's feed-forward: the GELU pair, then the fp32-out projection
    dit      a diffusion transformer's feed-forward: up + bias + GELU-tanh,
             then down + bias; bf16 or fp32 activations
    proj     one diffusion-transformer projection + bias, fp32 out
    decode   one greedy token through a whole model, replayed as a HIP graph
    sample   top-p sampling of one token from a vocabulary of logits

Weights are random 4-bit codes with scales |N(0, 0.02)| and biases -8 * scale,
activations N(0, 1): the distributions of the benchmark and the tests.
"""
import math
from types import SimpleNamespace

import torch

from __graft_entry__ import load_package

EPS = 1e-5

# (hidden, intermediate, q rows, q|k|v rows) of decoder layers
LAYERS = ((3072, 8192, 3072, 5120), (2048, 8192, 2048, 3072), (4096, 14336, 4096, 6144))


def listed():
    return [
        # The smallest call: one token through one square projection, where launch and
        # host latency are most of the time.
        dict(name="linear_m1", work="linear", entry="plain", M=1, N=3072, K=3072, g=64),
        # Interactive chat: one token through a 3B decoder, the loop a generation spends
        # its time in.  All 4-bit weights are read once.
        dict(name="decode_token", work="decode", layers=28, shape=0, vocab=128256, g=64),
        # The end of every sampled token.
        dict(name="sample_token", work="sample", vocab=128256, half=True, spread=3.0, seen=700,
             temperature=0.7, top_p=0.9, penalty=1.1),
        # Eight sequences decoded together, or the last few tokens of a chunked prompt.
        dict(name="layer_m8", work="layer", shape=0, M=8, g=64),
        # A short chat turn with a checkpoint of the finest group size.
        dict(name="layer_m96_g32", work="layer", shape=0, M=96, g=32),
        # An ordinary prompt; prompts have no round lengths.
        dict(name="layer_m333", work="layer", shape=0, M=333, g=64),
        # The benchmark's prompt of 750 tokens.
        dict(name="layer_m750", work="layer", shape=0, M=750, g=64),
        # The text encoder of a video pipeline at its padded length of 128 tokens.
        dict(name="geglu_m128", work="geglu", M=128, K=4096, F=10240, g=64),
        # The video model's feed-forward at 16 x 16 x 24 latent patches, bf16 activations.
        dict(name="dit_m6144_bf16", work="dit", M=6144, K=2048, F=8192, g=64, x="bf16"),
        # The same block on a small clip of odd size, from fp32 activations and a checkpoint
        # of the coarsest group size.
        dict(name="dit_m1537_f32_g128", work="dit", M=1537, K=2048, F=8192, g=128, x="f32"),
        # The video model's output projection to 128 latent channels.
        dict(name="proj_n128_f32", work="proj", M=6144, K=2048, N=128, g=64, x="f32"),
        # Logits of every row of a prompt (scoring a text): the largest product.
        dict(name="linear_m750_vocab", work="linear", entry="fast", M=750, N=128256, K=3072, g=64),
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "layer", "layer", "layer", "geglu", "dit", "dit", "proj",
                       "decode", "sample"))
    g = rng.choice((64, 64, 64, 32, 128))
    if kind == "linear":
        case = dict(work=kind, entry=rng.choice(("plain", "fast", "f32")), M=_log_int(rng, 1, 2048),
                    N=_log_int(rng, 256, 16384), K=g * _log_int(rng, 512 // g, 12288 // g), g=g)
    elif kind == "layer":
        case = dict(work=kind, shape=rng.randrange(len(LAYERS)), M=_log_int(rng, 2, 1500), g=g)
    elif kind == "geglu":
        case = dict(work=kind, M=_log_int(rng, 8, 512), K=4096, F=10240, g=g)
    elif kind == "dit":
        case = dict(work=kind, M=_log_int(rng, 256, 6144), K=2048, F=8192, g=g,
                    x=rng.choice(("bf16", "f32")))
    elif kind == "proj":
        case = dict(work=kind, M=_log_int(rng, 64, 6144), K=rng.choice((128, 2048, 4096)),
                    N=rng.choice((128, 256, 2048, 4096)), g=g, x=rng.choice(("bf16", "f32")))
    elif kind == "decode":
        case = dict(work=kind, layers=_log_int(rng, 2, 16), shape=rng.randrange(len(LAYERS)),
                    vocab=_log_int(rng, 32000, 128256), g=g)
    else:
        case = dict(work=kind, vocab=_log_int(rng, 2000, 128256), half=rng.random() < 0.5,
                    spread=rng.choice((0.01, 1.0, 3.0, 6.0)), seen=_log_int(rng, 1, 4000),
                    temperature=round(rng.uniform(0.5, 1.2), 2),
                    top_p=rng.choice((0.8, 0.9, 0.95, 1.0)), penalty=rng.choice((1.0, 1.1)))
    flops = work(case)["flops"]
    most = 4.2e11 if g == 64 else 2.4e11   # no drawn case takes longer than the largest listed one
    if flops > most:
        case["M"] = int(case["M"] * most / flops)
    return case


# ---- inputs ----

def _generator(seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return gen


def _normal(gen, *shape, dtype=torch.float16):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32).to(dtype)


def _weight(gen, N, K, g):
    """A random 4-bit weight of N rows in the checkpoint layout."""
    codes = torch.randint(-2**31, 2**31, (N, K // 8), generator=gen, device="cuda",
                          dtype=torch.int64).to(torch.int32)
    scales = (torch.randn(N, K // g, generator=gen, device="cuda") * 0.02).abs().half()
    return load_package().Q4Weight(codes, scales, scales * -8.0, K, g)


def _norm_weight(gen, K):
    return 1.0 + 0.1 * torch.randn(K, generator=gen, device="cuda")


def _inputs(case, seed):
    """The tensors a program has in hand before the call."""
    gen = _generator(seed)
    s = SimpleNamespace(case=case)
    work, g = case["work"], case.get("g", 64)
    if work == "linear":
        s.x = _normal(gen, case["M"], case["K"])
        s.w = _weight(gen, case["N"], case["K"], g)
    elif work == "layer":
        H, F, q, qkv = LAYERS[case["shape"]]
        s.h = _normal(gen, case["M"], H)
        s.attn = _normal(gen, case["M"], q)
        s.qkv, s.o = _weight(gen, qkv, H, g), _weight(gen, H, q, g)
        s.gate, s.up, s.down = _weight(gen, F, H, g), _weight(gen, F, H, g), _weight(gen, H, F, g)
        s.norms = [_norm_weight(gen, H) for _ in range(3)]
    elif work == "geglu":
        s.x = _normal(gen, case["M"], case["K"])
        s.gate, s.up = _weight(gen, case["F"], case["K"], g), _weight(gen, case["F"], case["K"], g)
        s.down = _weight(gen, case["K"], case["F"], g)
    elif work in ("dit", "proj"):
        s.x = _normal(gen, case["M"], case["K"], dtype=_DTYPES[case["x"]])
        if work == "dit":
            s.up, s.down = _weight(gen, case["F"], case["K"], g), _weight(gen, case["K"], case["F"], g)
            s.up_bias, s.down_bias = (_normal(gen, n, dtype=torch.float32)
                                      for n in (case["F"], case["K"]))
        else:
            s.w = _weight(gen, case["N"], case["K"], g)
            s.bias = _normal(gen, case["N"], dtype=torch.float32)
    elif work == "decode":
        H, F, q, qkv = LAYERS[case["shape"]]
        # residual writers (o, down) scaled down as training leaves them: the stream's size
        # then stays of the order of the embedding's through the depth
        def small(N, K, by):
            w = _weight(gen, N, K, g)
            w.scales.mul_(by)
            w.biases.mul_(by)
            return w
        embed = _weight(gen, case["vocab"], H, g)
        layers = [SimpleNamespace(qkv_proj=_weight(gen, qkv, H, g), o_proj=small(H, q, 0.02),
                                  gate_proj=small(F, H, 0.2), up_proj=small(F, H, 0.2),
                                  down_proj=small(H, F, 0.02), input_norm_weight=_norm_weight(gen, H),
                                  post_norm_weight=_norm_weight(gen, H))
                  for _ in range(case["layers"])]
        config = SimpleNamespace(hidden_size=H, intermediate_size=F, num_attention_heads=q // 128,
                                 num_key_value_heads=(qkv - q) // 256, head_dim=128,
                                 vocab_size=case["vocab"], rms_norm_eps=EPS)
        s.model = SimpleNamespace(config=config, embed_tokens=embed, lm_head=embed, layers=layers,
                                  norm_weight=_norm_weight(gen, H))
        s.token = torch.randint(0, case["vocab"], (1,), generator=gen, device="cuda",
                                dtype=torch.int32)
    else:
        dtype = torch.float16 if case["half"] else torch.float32
        s.logits = (torch.randn(case["vocab"], generator=gen, device="cuda") * case["spread"]).to(dtype)
        s.seen = torch.randint(0, case["vocab"], (case["seen"],), generator=gen, device="cuda",
                               dtype=torch.int32)
        s.u = float(torch.rand(1, generator=torch.Generator().manual_seed(seed)))
    return s


_DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def prepare(case, seed):
    load_package()
    s = _inputs(case, seed)
    if case["work"] == "decode":
        from swiftltx_amd.decode import DecodeStep
        torch.cuda.current_stream().synchronize()
        s.step = DecodeStep(s.model, stream=torch.cuda.Stream())
        s.step.capture()
        s.step.stream.synchronize()
    return s


def run(s):
    lib, case = load_package(), s.case
    work, M = case["work"], case.get("M", 1)
    if work == "linear":
        f = {"plain": lib.matmul_q4, "fast": lib.matmul_q4_fast, "f32": lib.matmul_q4_fast_f32}
        return f[case["entry"]](s.x, s.w.weight, s.w.scales, s.w.biases, M, case["K"], case["N"],
                                case["g"])
    if work == "layer":
        H, F, q, qkv = LAYERS[case["shape"]]
        normed = lib.rms_norm(s.h, s.norms[0], EPS, M, H)
        qkv_rows = lib.linear(normed, s.qkv, M, H, qkv, fast=True)
        res, normed = lib.matmul_q4_residual_rms_norm(s.attn, s.o, s.h, s.norms[1], EPS, M, H, False)
        act = lib.matmul_q4_silu_mul(normed, s.gate, s.up, M, H, F)
        out, next_normed = lib.matmul_q4_residual_rms_norm(act, s.down, res, s.norms[2], EPS, M, H,
                                                           True)
        return {"qkv": qkv_rows, "res": res, "normed": normed, "act": act, "out": out,
                "next_normed": next_normed}
    if work == "geglu":
        act = lib.matmul_q4_geglu(s.x, s.gate, s.up, M, case["K"], case["F"])
        return lib.matmul_q4_fast_f32(act, s.down.weight, s.down.scales, s.down.biases, M, case["F"],
                                      case["K"], case["g"])
    if work == "dit":
        act = lib.matmul_q4_ex(s.x, s.up, M, case["F"], out_dtype=s.x.dtype, bias=s.up_bias,
                               epilogue=lib.SLTX_EPI_GELU_TANH)
        return lib.matmul_q4_ex(act, s.down, M, case["K"], out_dtype=s.x.dtype, bias=s.down_bias)
    if work == "proj":
        return lib.matmul_q4_ex(s.x, s.w, M, case["N"], bias=s.bias)
    if work == "decode":
        s.step.token.copy_(s.token)
        s.step.replay()
        return s.step.logits
    return lib.sample(s.logits, case["temperature"], case["top_p"], case["penalty"], s.seen, s.u)


# ---- what a pass cannot do without ----

def _set(N, K, g):
    return N * K // 2 + 4 * N * (K // g)


def work(case):
    work, M, g = case["work"], case.get("M", 1), case.get("g", 64)
    if work == "linear":
        N, K = case["N"], case["K"]
        out = 4 if case["entry"] == "f32" else 2
        return {"bytes": _set(N, K, g) + 2 * M * K + out * M * N, "flops": 2 * M * N * K}
    if work == "layer":
        H, F, q, qkv = LAYERS[case["shape"]]
        sets = _set(qkv, H, g) + _set(H, q, g) + 2 * _set(F, H, g) + _set(H, F, g)
        # in: h and the attention output; out: the six results
        return {"bytes": sets + 12 * H + 2 * M * (H + q + qkv + F + 4 * H),
                "flops": 2 * M * (qkv * H + H * q + 3 * F * H)}
    if work == "geglu":
        K, F = case["K"], case["F"]
        return {"bytes": 2 * _set(F, K, g) + _set(K, F, g) + 6 * M * K, "flops": 6 * M * K * F}
    if work == "dit":
        K, F, each = case["K"], case["F"], 2 if case["x"] == "bf16" else 4
        return {"bytes": _set(F, K, g) + _set(K, F, g) + 4 * (F + K) + 2 * each * M * K,
                "flops": 4 * M * K * F}
    if work == "proj":
        K, N, each = case["K"], case["N"], 2 if case["x"] == "bf16" else 4
        return {"bytes": _set(N, K, g) + 4 * N + each * M * K + 4 * M * N, "flops": 2 * M * N * K}
    if work == "decode":
        H, F, q, qkv = LAYERS[case["shape"]]
        sets = _set(qkv, H, g) + _set(H, q, g) + 2 * _set(F, H, g) + _set(H, F, g) + 8 * H
        L, V = case["layers"], case["vocab"]
        return {"bytes": L * sets + _set(V, H, g) + 4 * H + 2 * V,
                "flops": 2 * L * (qkv * H + H * q + 3 * F * H) + 2 * V * H}
    return {"bytes": case["vocab"] * (2 if case["half"] else 4) + 4 * case["seen"], "flops": 0}


def tolerance(case):
    work = case["work"]
    if work == "sample":
        return "exact"   # a token id; its sums are exact whatever their order
    # Four times what the outputs were off by against 64 bits, where fp16 rounds weights,
    # activations and results once each (bf16 eight times as coarse).
    if work == "layer":
        return {"rel": 3e-3}
    if case.get("x") == "bf16":
        return {"rel": 8e-3}
    if work == "dit":
        return {"rel": 4e-4}   # mostly the common part of the GELU outputs: roundings cancel
    return {"rel": 1.5e-3}


# ---- the same in 64 bits ----

def _dequant(w, rows=slice(None)):
    words = w.weight[rows].to(torch.int64)
    q = torch.stack([(words >> (4 * i)) & 15 for i in range(8)], dim=-1).flatten(1).double()
    s, b = (t[rows].double().repeat_interleave(w.group_size, dim=1) for t in (w.scales, w.biases))
    return q.mul_(s).add_(b)


def _mm(x, w):
    """x . W^T, some rows of W at a time."""
    return torch.cat([x @ _dequant(w, slice(n, n + 16384)).t() for n in range(0, w.N, 16384)], dim=1)


def _rms(v, weight):
    return v * torch.rsqrt((v * v).mean(-1, keepdim=True) + EPS) * weight.double()


def _silu(v):
    return v * torch.sigmoid(v)


def _gelu(v):
    return 0.5 * v * (1 + torch.tanh((0.7978845608 * (v + 0.044715 * v ** 3)).clamp(-10, 10)))


def exact(case, seed):
    work = case["work"]
    if work == "sample":
        return None   # a token id
    s = _inputs(case, seed)
    if work == "linear":
        return _mm(s.x.double(), s.w)
    if work == "layer":
        h = s.h.double()
        qkv = _mm(_rms(h, s.norms[0]), s.qkv)
        res = h + _mm(s.attn.double(), s.o)
        normed = _rms(res, s.norms[1])
        act = _silu(_mm(normed, s.gate)) * _mm(normed, s.up)
        out = res + _mm(act, s.down)
        return {"qkv": qkv, "res": res, "normed": normed, "act": act, "out": out,
                "next_normed": _rms(out, s.norms[2])}
    if work == "geglu":
        x = s.x.double()
        return _mm(_gelu(_mm(x, s.gate)) * _mm(x, s.up), s.down)
    if work == "dit":
        act = _gelu(_mm(s.x.double(), s.up) + s.up_bias.double())
        return _mm(act, s.down) + s.down_bias.double()
    if work == "proj":
        return _mm(s.x.double(), s.w) + s.bias.double()
    m = s.model
    q = LAYERS[case["shape"]][2]
    h = _dequant(m.embed_tokens, s.token.long())
    for w in m.layers:
        attn = _mm(_rms(h, w.input_norm_weight), w.qkv_proj)[:, :q]   # the stand-in: the q rows
        res = h + _mm(attn, w.o_proj)
        n = _rms(res, w.post_norm_weight)
        h = res + _mm(_silu(_mm(n, w.gate_proj)) * _mm(n, w.up_proj), w.down_proj)
    return _mm(_rms(h, m.norm_weight), m.lm_head)
