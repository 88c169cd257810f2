"""The performance cases of this framework: what its users have it do, over the
real range of sizes, types and batch widths.

  gemv     one matrix times one token (hip_gemv): every projection of a decode step
           that is issued on its own, any of the 17 GGUF types
  gemm     one matrix times n tokens (hip_gemm): a batch of sequences decoding
           together, or the tokens of a prompt
  mmq81    the same in ggml's Q8_1 arithmetic (hip_gemm_q8_1_mmq), bit-exact
  dequant  a whole tensor decoded to f32 (hip_dequant)
  attn     RoPE, K/V append and attention of one decode step for n_seq sequences
           (hip_attention_step_batched)
  moe      a routed mixture-of-experts FFN for a batch of tokens (MoeStep)
  step     a whole decode step of a Llama-3-8B-shaped Q4_K_M model, replayed from a
           captured graph as a serving loop does (ForwardStep, BatchStep)

Sizes are those of the benchmark configurations: hidden 4096, FFN 14336, vocabulary
128256, 32 heads on 8 K/V heads of 128, 8 experts of which 2 per token.
"""
import ctypes as C
import math
import re
from pathlib import Path

import numpy as np
import torch

from saient_quartz_amd import GGML_TYPES, lib, type_size
from saient_quartz_amd.api import check
from saient_quartz_amd.decode import BatchStep, ForwardStep, ModelConfig, MoeStep

TYPE = {name: t for t, (name, _, _) in GGML_TYPES.items()}
HIDDEN, KV, FFN, VOCAB, HEADS, HEADS_KV, HEAD_DIM = 4096, 1024, 14336, 128256, 32, 8, 128
EXPERTS, TOP_K = 8, 2
THETA = 500000.0


# ---------------------------------------------------------------- cases

def listed():
    return [
        # the smallest projection of a layer (attn_v), one token: launch and latency
        dict(name="gemv_v_q6k", kind="gemv", type="Q6_K", out=KV, inp=HIDDEN),
        # the FFN up projection, one token: the headline GEMV
        dict(name="gemv_up_q4k", kind="gemv", type="Q4_K", out=FFN, inp=HIDDEN),
        # the FFN down projection of a model in a 32-element block type
        dict(name="gemv_down_q5_0", kind="gemv", type="Q5_0", out=HIDDEN, inp=FFN),
        # one token of one sequence in the middle of a conversation
        dict(name="step_n1", kind="step", n=1, pos=511),
        # 16 sequences decoding together
        dict(name="step_n16", kind="step", n=16, pos=511),
        # 16 sequences through an attention projection stored in 8 bits
        dict(name="gemm_q_q8_0_n16", kind="gemm", type="Q8_0", out=HIDDEN, inp=HIDDEN, n=16),
        # a short prompt through the down projection, an odd number of tokens
        dict(name="gemm_down_q6k_n77", kind="gemm", type="Q6_K", out=HIDDEN, inp=FFN, n=77),
        # a chunk of a long prompt through the up projection
        dict(name="gemm_up_q4k_n512", kind="gemm", type="Q4_K", out=FFN, inp=HIDDEN, n=512),
        # a prompt in ggml's own rounding, one row tile of it
        dict(name="mmq81_q_q4k_n128", kind="mmq81", type="Q4_K", out=HIDDEN, inp=HIDDEN, n=128),
        # the expert FFN of a batch of 64 tokens, routed on the device
        dict(name="moe_iq3s_n64", kind="moe", type="IQ3_S", n=64),
        # the attention of 16 sequences well into their context
        dict(name="attn_16x2047", kind="attn", n=16, pos=2047),
        # a tensor decoded to f32 for a consumer that has no quantised kernel
        dict(name="dequant_q6k", kind="dequant", type="Q6_K", out=FFN, inp=HIDDEN),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mat(rng, t, most=FFN * HIDDEN):
    """Rows x columns of a matrix of type t: the columns a whole number of blocks."""
    qk = GGML_TYPES[TYPE[t]][1]
    unit = 256 if qk == 256 or rng.random() < 0.7 else 32
    inp = rng.choice([HIDDEN, FFN]) if rng.random() < 0.3 else unit * max(1, _log(rng, 512, FFN) // unit)
    out = _log(rng, 256, max(256, min(VOCAB, most // inp)))
    return out, inp


def draw(rng):
    kind = rng.choice(["gemv"] * 5 + ["gemm"] * 5 + ["mmq81", "dequant", "attn", "moe", "step"])
    if kind == "gemv":
        # the types of the decode path as often as all the others together
        t = rng.choice(["Q4_K", "Q5_K", "Q6_K", "Q8_0"]) if rng.random() < 0.5 else rng.choice(sorted(TYPE))
        out, inp = _mat(rng, t)
        return dict(kind=kind, type=t, out=out, inp=inp)
    if kind == "gemm":
        t = rng.choice(["Q4_K", "Q4_K", "Q5_K", "Q6_K", "Q8_0", "Q4_0", "Q5_0", "IQ3_S", "IQ2_XXS"])
        n = _log(rng, 2, 512)
        out, inp = _mat(rng, t)
        return dict(kind=kind, type=t, out=out, inp=inp, n=n)
    if kind == "mmq81":
        t = rng.choice(["Q4_K", "Q6_K"])
        out, inp = _mat(rng, t, HIDDEN * HIDDEN)
        return dict(kind=kind, type=t, out=out, inp=256 * (inp // 256), n=_log(rng, 2, 128))
    if kind == "dequant":
        t = rng.choice(sorted(TYPE))
        out, inp = _mat(rng, t)
        return dict(kind=kind, type=t, out=out, inp=inp)
    if kind == "attn":
        return dict(kind=kind, n=_log(rng, 1, 32), pos=_log(rng, 1, 2047) - 1)
    if kind == "moe":
        return dict(kind=kind, type=rng.choice(["IQ3_S", "IQ2_XXS", "Q4_K"]), n=_log(rng, 1, 64))
    return dict(kind=kind, n=_log(rng, 1, 16), pos=_log(rng, 1, 1000) - 1)


# ---------------------------------------------------------------- inputs

# Per type: the byte offsets of the f16 scale, the offset of the f16 minimum and the
# multiple of the scale it takes (the mean of the quants it is subtracted for, so that
# weights average zero), and the standard deviation of a weight at scale 1.
_FIELDS = {
    "Q4_0": (0, None, 0, 4.7), "Q4_1": (0, 2, -7.5, 4.6), "Q5_0": (0, None, 0, 9.3), "Q5_1": (0, 2, -15.5, 9.2),
    "Q8_0": (0, None, 0, 73.0), "IQ4_NL": (0, None, 0, 67.0), "Q2_K": (80, 82, 1.5, 14.0), "Q4_K": (0, 2, 7.5, 256.0),
    "Q5_K": (0, 2, 15.5, 511.0), "Q6_K": (208, None, 0, 690.0), "IQ2_XXS": (0, None, 0, 50.0),
    "IQ2_XS": (0, None, 0, 50.0), "IQ2_S": (0, None, 0, 50.0), "IQ3_S": (0, None, 0, 150.0),
}


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * (seed + 1))
    return g


def weights(t, out, inp, g, std=None):
    """GGUF rows of type t as a checkpoint holds them: random quants, scales for
    weights of standard deviation `std` (1 / sqrt(inp) by default)."""
    std = std or 1.0 / math.sqrt(inp)
    n = out * inp
    if t in ("F32", "F16", "BF16"):
        w = torch.randn(n, device="cuda", generator=g).mul_(std)
        return w.to({"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[t]).view(torch.uint8)
    _, qk, bb = GGML_TYPES[TYPE[t]]
    nb = n // qk
    blk = torch.randint(0, 256, (nb, bb), dtype=torch.uint8, device="cuda", generator=g)
    if t == "Q8_0":
        q = torch.randint(-127, 128, (nb, 32), dtype=torch.int8, device="cuda", generator=g)
        blk[:, 2:34] = q.view(torch.uint8)
    if t == "Q6_K":
        sc = torch.randint(-64, 64, (nb, 16), dtype=torch.int8, device="cuda", generator=g)
        blk[:, 192:208] = sc.view(torch.uint8)
    off, off_min, mean, unit = _FIELDS[t]
    d = torch.rand(nb, device="cuda", generator=g).mul_(0.8).add_(0.6).mul_(std / unit).half()
    blk[:, off:off + 2] = d.view(torch.uint8).view(nb, 2)
    if off_min is not None:
        m = d.float().mul(mean).half()
        blk[:, off_min:off_min + 2] = m.view(torch.uint8).view(nb, 2)
    return blk.reshape(-1)


def _tokens(n, dim, g):
    """Activations: normal, with a few channels much larger than the rest."""
    x = torch.randn(n, dim, device="cuda", generator=g)
    x[:, 7::509] *= 8.0
    return x


def _step_inputs(case, seed):
    cfg, g = ModelConfig(max_seq=1024), _gen(seed)
    names = {12: "Q4_K", 14: "Q6_K"}
    w = {name: [] for name, _, _ in cfg.mats()}
    for _ in range(cfg.layers):
        for name, o, i in cfg.mats():
            w[name].append(weights(names[cfg.type_of(name)], o, i, g))
    w["head"] = weights("Q6_K", cfg.vocab, cfg.hidden, g)
    w["embed"] = weights("Q4_K", cfg.vocab, cfg.hidden, g, std=1.0)

    def norm():
        return 1.0 + 0.1 * torch.randn(cfg.hidden, device="cuda", generator=g)

    w["attn_norm"] = [norm() for _ in range(cfg.layers)]
    w["ffn_norm"] = [norm() for _ in range(cfg.layers)]
    w["out_norm"] = norm()
    n, kvd = case["n"], cfg.n_kv * cfg.head_dim
    kv = []
    for _ in range(cfg.layers):
        pair = []
        for _ in range(2):
            c = torch.zeros(n, cfg.max_seq, kvd, device="cuda")
            c[:, :case["pos"]] = torch.randn(n, case["pos"], kvd, device="cuda", generator=g)
            pair.append(c)
        kv.append(pair)
    tokens = torch.randint(0, cfg.vocab, (n,), device="cuda", generator=g).tolist()
    return cfg, w, kv, tokens


def _attn_inputs(case, seed):
    g, n, rows = _gen(seed), case["n"], case["pos"] + 1
    t = {name: torch.randn(n, d, device="cuda", generator=g) for name, d in (("q", HIDDEN), ("k", KV), ("v", KV))}
    t["kc"] = torch.randn(n, rows, KV, device="cuda", generator=g)
    t["vc"] = torch.randn(n, rows, KV, device="cuda", generator=g)
    return t


def _moe_inputs(case, seed):
    g, t = _gen(seed), case["type"]
    w = {}
    for name, o, i in (("gate", FFN, HIDDEN), ("up", FFN, HIDDEN), ("down", HIDDEN, FFN)):
        w[name] = torch.cat([weights(t, o, i, g) for _ in range(EXPERTS)])
    w["router"] = torch.randn(EXPERTS, HIDDEN, device="cuda", generator=g) / math.sqrt(HIDDEN)
    return w, torch.randn(case["n"], HIDDEN, device="cuda", generator=g)


def prepare(case, seed):
    kind, L = case["kind"], lib()
    if kind in ("gemv", "gemm", "mmq81"):
        g, t, out, inp, n = _gen(seed), case["type"], case["out"], case["inp"], case.get("n", 1)
        w, x = weights(t, out, inp, g), _tokens(n, inp, g)
        y = torch.empty(n, out, device="cuda")
        stream = torch.cuda.current_stream().cuda_stream
        args = [TYPE[t], w.data_ptr(), x.data_ptr(), y.data_ptr(), inp, out]
        if kind == "gemv":
            call = ("hip_gemv_async", L.hip_gemv_async, args + [stream])
        elif kind == "gemm":
            call = ("hip_gemm_async", L.hip_gemm_async, args + [n, stream])
        else:
            call = ("hip_gemm_q8_1_mmq_async", L.hip_gemm_q8_1_mmq_async, args + [n, 0, 0, stream])
        return dict(call=call, out=y, keep=(w, x))
    if kind == "dequant":
        w = weights(case["type"], case["out"], case["inp"], _gen(seed))
        y = torch.empty(case["out"], case["inp"], device="cuda")
        call = ("hip_dequant_async", L.hip_dequant_async,
                [TYPE[case["type"]], w.data_ptr(), y.data_ptr(), y.numel(), torch.cuda.current_stream().cuda_stream])
        return dict(call=call, out=y, keep=(w,))
    if kind == "attn":
        t, n, rows = _attn_inputs(case, seed), case["n"], case["pos"] + 1
        out = torch.empty(n, HIDDEN, device="cuda")
        call = ("hip_attention_step_batched_async", L.hip_attention_step_batched_async,
                [out.data_ptr(), t["q"].data_ptr(), t["k"].data_ptr(), t["v"].data_ptr(), t["kc"].data_ptr(),
                 t["vc"].data_ptr(), None, n, rows * KV, HEADS, HEADS_KV, HEAD_DIM, KV, case["pos"], THETA, 1.0, 0, 0,
                 1.0 / math.sqrt(HEAD_DIM), torch.cuda.current_stream().cuda_stream])
        return dict(call=call, out={"out": out, "k": t["kc"][:, -1], "v": t["vc"][:, -1]}, keep=t)
    if kind == "moe":
        w, x = _moe_inputs(case, seed)
        t = TYPE[case["type"]]
        step = MoeStep((t, t, t), w["gate"], w["up"], w["down"], w["router"], EXPERTS, TOP_K, HIDDEN, FFN, case["n"])
        return dict(moe=step, x=x, n=case["n"], out=torch.empty(case["n"], HIDDEN, device="cuda"))
    cfg, w, kv, tokens = _step_inputs(case, seed)
    if case["n"] == 1:
        step = ForwardStep(cfg, w)
        step.set_state(tokens[0], case["pos"])
    else:
        step = BatchStep(cfg, w, case["n"])
        step.set_state(tokens, case["pos"])
    for l in range(cfg.layers):
        step.kc[l].copy_(kv[l][0].reshape(-1))
        step.vc[l].copy_(kv[l][1].reshape(-1))
    torch.cuda.synchronize()
    return dict(step=step, graph=_Graph(step),
                out={"logits": step.logits.view(-1, cfg.vocab), "hidden": step.hidden.view(-1, cfg.hidden)})


class _Graph:
    """One decode step recorded through the C ABI, as a serving loop records it once
    and replays it per token.  The token and the position are read on the device."""

    def __init__(self, step):
        self.L = lib()
        stream, self.exec = C.c_void_p(), C.c_void_p()
        check("hip_stream_create", self.L.hip_stream_create(C.byref(stream)))
        check("hip_graph_begin", self.L.hip_graph_begin(stream))
        step.issue(dev=True, stream=stream.value)
        check("hip_graph_end", self.L.hip_graph_end(stream, C.byref(self.exec)))
        self.L.hip_stream_destroy(stream)
        self.on = torch.cuda.current_stream().cuda_stream

    def launch(self):
        check("hip_graph_launch", self.L.hip_graph_launch(self.exec, self.on))

    def __del__(self):
        self.L.hip_graph_destroy(self.exec)


def run(state):
    if "call" in state:
        name, fn, args = state["call"]
        check(name, fn(*args))
    elif "moe" in state:
        state["moe"].issue(state["x"], state["out"], state["n"])
    else:
        state["graph"].launch()
    return state["out"]


# ---------------------------------------------------------------- what a pass needs

def work(case):
    kind, n = case["kind"], case.get("n", 1)
    if kind in ("gemv", "gemm", "mmq81"):
        out, inp = case["out"], case["inp"]
        return dict(bytes=type_size(TYPE[case["type"]], out * inp) + 4 * n * (inp + out), flops=2 * n * out * inp)
    if kind == "dequant":
        e = case["out"] * case["inp"]
        return dict(bytes=type_size(TYPE[case["type"]], e) + 4 * e, flops=2 * e)
    if kind == "attn":
        rows = case["pos"] + 1
        return dict(bytes=4 * n * (2 * rows * KV + 2 * KV + 2 * HIDDEN), flops=4 * n * rows * HIDDEN)
    if kind == "moe":
        per = FFN * HIDDEN
        used = EXPERTS if n * TOP_K >= 3 * EXPERTS else min(EXPERTS, max(TOP_K, n))
        return dict(bytes=3 * used * type_size(TYPE[case["type"]], per) + 8 * n * HIDDEN + 4 * EXPERTS * HIDDEN,
                    flops=6 * n * TOP_K * per)
    cfg = ModelConfig(max_seq=1024)
    params = cfg.layers * sum(o * i for _, o, i in cfg.mats()) + cfg.vocab * cfg.hidden
    rows = case["pos"] + 1
    return dict(bytes=cfg.weight_bytes() + 8 * n * cfg.layers * rows * KV + 4 * n * cfg.vocab,
                flops=2 * n * params + 4 * n * cfg.layers * rows * HIDDEN)


def tolerance(case):
    kind = case["kind"]
    if kind in ("mmq81", "dequant"):
        return "exact"  # both promise the reference's bits
    # about four times the error against 64 bits that 32-bit arithmetic shows
    if kind == "step":
        return {"rel": 1e-5}  # 32 layers after each other: 2.3e-6 seen
    if kind == "attn":
        return {"rel": 7e-5}  # the RoPE angle in 32 bits: 1.8e-5 seen at position 2047
    return {"rel": 5e-6}  # 1e-6 seen


# ---------------------------------------------------------------- 64-bit results

def _f16(b, o):
    return b[:, o:o + 2].contiguous().view(torch.float16).double()


def _grid(name):
    """A codebook of the IQ formats as float64 rows (tables that the formats define)."""
    import saient_quartz_amd
    txt = (Path(saient_quartz_amd.__file__).parent / "csrc" / "iq_grids.h").read_text()
    body = re.search(r"#define QH_%s_GRID_VALUES \\\n(.*?)\n\n" % name, txt, re.S).group(1)
    width = 4 if name == "IQ3S" else 8
    raw = b"".join(int(v, 16).to_bytes(8, "little")[:width] for v in re.findall(r"0x[0-9a-fA-F]+", body))
    return torch.from_numpy(np.frombuffer(raw, np.int8).reshape(-1, width).astype(np.float64)).cuda()


def _pm(signs):
    """Sign bytes -> (..., 8) of +1 / -1, bit j for element j."""
    return 1.0 - 2.0 * ((signs[..., None] >> torch.arange(8, device="cuda")) & 1).double()


def _ksigns(i):
    p = i ^ (i >> 4)
    p = p ^ (p >> 2)
    return i | (((p ^ (p >> 1)) & 1) << 7)


def _k4(b):
    """The eight 6-bit scales and minimums of Q4_K / Q5_K."""
    s = b[:, 4:16].int()
    lo, mid, hi = s[:, 0:4], s[:, 4:8], s[:, 8:12]
    return (torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1).double(),
            torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1).double())


def _decode(t, data):
    """Flat GGUF bytes -> float64 values, from the formats' definitions."""
    if t in ("F32", "F16", "BF16"):
        return data.view({"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[t]).double()
    b = data.view(-1, GGML_TYPES[TYPE[t]][2])
    nb = b.shape[0]
    off, off_min, _, _ = _FIELDS[t]
    d = _f16(b, off)
    if t == "Q8_0":
        return (d * b[:, 2:34].contiguous().view(torch.int8).double()).reshape(-1)
    if t in ("Q4_0", "Q4_1", "Q5_0", "Q5_1", "IQ4_NL"):
        qs = b[:, -16:].int()
        q = torch.cat([qs & 15, qs >> 4], 1)
        if t in ("Q5_0", "Q5_1"):
            o = 2 if t == "Q5_0" else 4
            qh = b[:, o:o + 4].contiguous().view(torch.int32)
            q = q | (((qh >> torch.arange(32, device="cuda")) & 1) << 4)
        if t == "IQ4_NL":
            tab = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]
            return (d * torch.tensor(tab, device="cuda").double()[q.long()]).reshape(-1)
        v = d * (q.double() - {"Q4_0": 8.0, "Q5_0": 16.0}.get(t, 0.0))
        return (v + _f16(b, off_min) if off_min is not None else v).reshape(-1)
    if t in ("Q4_K", "Q5_K"):
        s, m = _k4(b)
        qs = b[:, -128:].int().view(nb, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).view(nb, 8, 32)
        if t == "Q5_K":
            bit = torch.arange(8, device="cuda")[None, :, None]
            q = q | (((b[:, 16:48].int()[:, None, :] >> bit) & 1) << 4)
        return ((d * s)[:, :, None] * q.double() - (_f16(b, off_min) * m)[:, :, None]).reshape(-1)
    if t == "Q6_K":
        ql, qh = b[:, :128].int().view(nb, 2, 2, 32), b[:, 128:192].int().view(nb, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2)
        high = (qh >> (2 * torch.arange(4, device="cuda"))[None, None, :, None]) & 3
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        return ((d * sc)[:, :, None] * ((low | (high << 4)).double() - 32).view(nb, 16, 16)).reshape(-1)
    if t == "Q2_K":
        sc = b[:, :16].int()
        q = (b[:, 16:80].int().view(nb, 2, 1, 32) >> (2 * torch.arange(4, device="cuda"))[None, None, :, None]) & 3
        s, m = d * (sc & 15).double(), _f16(b, off_min) * (sc >> 4).double()
        return (s[:, :, None] * q.double().view(nb, 16, 16) - m[:, :, None]).reshape(-1)
    l = torch.arange(4, device="cuda")
    if t == "IQ2_XXS":
        q = b[:, 2:].int().view(nb, 8, 8)
        a = q[:, :, 4].long() | (q[:, :, 5].long() << 8) | (q[:, :, 6].long() << 16) | (q[:, :, 7].long() << 24)
        v = _grid("IQ2XXS")[q[:, :, :4].long()] * _pm(_ksigns((a[:, :, None] >> (7 * l)) & 127))
        return ((d * (0.5 + (a >> 28).double()) * 0.25)[:, :, None, None] * v).reshape(-1)
    if t in ("IQ2_XS", "IQ2_S"):
        sc = b[:, -8:].int()
        s = d[:, :, None] * (0.5 + torch.stack([sc & 15, sc & 15, sc >> 4, sc >> 4], 2).double()) * 0.25
        if t == "IQ2_XS":
            q = b[:, 2:66].contiguous().view(torch.int16).view(nb, 8, 4).long() & 0xFFFF
            v = _grid("IQ2XS")[q & 511] * _pm(_ksigns(q >> 9))
        else:
            i = b[:, 2:34].long().view(nb, 8, 4) | ((b[:, 66:74].long()[:, :, None] << (8 - 2 * l)) & 0x300)
            v = _grid("IQ2S")[i] * _pm(b[:, 34:66].long().view(nb, 8, 4))
        return (s[..., None] * v).reshape(-1)
    sc = b[:, 106:110].int()  # IQ3_S
    s = d * (1.0 + 2.0 * torch.stack([sc & 15, sc >> 4], 2).view(nb, 8).double())
    q, qh = b[:, 2:66].long().view(nb, 8, 4, 2), b[:, 66:74].long()[:, :, None]
    i = q | torch.stack([(qh << (8 - 2 * l)) & 256, (qh << (7 - 2 * l)) & 256], 3)
    v = _grid("IQ3S")[i].view(nb, 8, 4, 8) * _pm(b[:, 74:106].long().view(nb, 8, 4))
    return (s[:, :, None, None] * v).reshape(-1)


def _times(x, t, data, out, inp):
    """x (n, inp) float64 times the matrix, a slab of rows at a time."""
    rows = max(1, (1 << 26) // inp)
    size = type_size(TYPE[t], inp)
    return torch.cat([x @ _decode(t, data[r * size:min(out, r + rows) * size]).view(-1, inp).T.contiguous()
                      for r in range(0, out, rows)], 1)


def _rope(x, pos, heads):
    x = x.view(x.shape[0], heads, HEAD_DIM // 2, 2)
    i = torch.arange(HEAD_DIM // 2, device="cuda", dtype=torch.float64)
    a = pos * THETA ** (-2.0 * i / HEAD_DIM)
    c, s = torch.cos(a), torch.sin(a)
    return torch.stack([x[..., 0] * c - x[..., 1] * s, x[..., 0] * s + x[..., 1] * c], -1).view(x.shape[0], -1)


def _attend(q, k, v, kc, vc, pos):
    """One attention step in float64 -> (out, rotated k); kc, vc: (n, rows, KV) before row pos."""
    n, group = q.shape[0], HEADS // HEADS_KV
    q, k = _rope(q, pos, HEADS), _rope(k, pos, HEADS_KV)
    out = torch.empty(n, HEADS, HEAD_DIM, device="cuda", dtype=torch.float64)
    for z in range(n):
        kz = torch.cat([kc[z, :pos].double(), k[z:z + 1]]).view(pos + 1, HEADS_KV, HEAD_DIM)
        vz = torch.cat([vc[z, :pos].double(), v[z:z + 1]]).view(pos + 1, HEADS_KV, HEAD_DIM)
        for h in range(HEADS):
            s = (kz[:, h // group] @ q[z].view(HEADS, HEAD_DIM)[h]) / math.sqrt(HEAD_DIM)
            out[z, h] = torch.softmax(s, 0) @ vz[:, h // group]
    return out.view(n, -1), k


def _norm(x, w):
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + 1e-5) * w.double()


def exact(case, seed):
    kind = case["kind"]
    if kind == "mmq81":
        return None  # the rounding is what the path is defined by: there is no 64-bit value
    if kind in ("gemv", "gemm"):
        g, t, out, inp, n = _gen(seed), case["type"], case["out"], case["inp"], case.get("n", 1)
        w, x = weights(t, out, inp, g), _tokens(n, inp, g)
        return _times(x.double(), t, w, out, inp)
    if kind == "dequant":
        return _decode(case["type"], weights(case["type"], case["out"], case["inp"], _gen(seed))).view(case["out"], -1)
    if kind == "attn":
        t = _attn_inputs(case, seed)
        out, k = _attend(t["q"].double(), t["k"].double(), t["v"].double(), t["kc"], t["vc"], case["pos"])
        return {"out": out, "k": k, "v": t["v"].double()}
    if kind == "moe":
        w, x = _moe_inputs(case, seed)
        x, t = x.double(), case["type"]
        per = type_size(TYPE[t], FFN * HIDDEN)
        top, ids = torch.topk(x @ w["router"].double().T, TOP_K, 1)
        share = torch.softmax(top, 1)
        out = torch.zeros_like(x)
        for e in range(EXPERTS):
            tok, j = torch.nonzero(ids == e, as_tuple=True)
            if len(tok) == 0:
                continue
            part = {m: w[m][e * per:(e + 1) * per] for m in ("gate", "up", "down")}
            gate = _times(x[tok], t, part["gate"], FFN, HIDDEN)
            act = gate * torch.sigmoid(gate) * _times(x[tok], t, part["up"], FFN, HIDDEN)
            out.index_add_(0, tok, share[tok, j][:, None] * _times(act, t, part["down"], HIDDEN, FFN))
        return out
    cfg, w, kv, tokens = _step_inputs(case, seed)
    row = type_size(cfg.type_of("embed"), cfg.hidden)
    x = torch.stack([_decode("Q4_K", w["embed"][t * row:(t + 1) * row]) for t in tokens])
    names = {12: "Q4_K", 14: "Q6_K"}
    size = {m: (o, i) for m, o, i in cfg.mats()}
    for l in range(cfg.layers):
        def mul(name, v, l=l):
            return _times(v, names[cfg.type_of(name)], w[name][l], *size[name])

        xn = _norm(x, w["attn_norm"][l])
        y = {m: mul(m, xn) for m in ("q", "k", "v")}
        att, _ = _attend(y["q"], y["k"], y["v"], kv[l][0], kv[l][1], case["pos"])
        x = x + mul("o", att)
        xn = _norm(x, w["ffn_norm"][l])
        gate = mul("gate", xn)
        x = x + mul("down", gate * torch.sigmoid(gate) * mul("up", xn))
    return {"logits": _times(_norm(x, w["out_norm"]), "Q6_K", w["head"], cfg.vocab, cfg.hidden), "hidden": x}
