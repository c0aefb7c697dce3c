"""The work a user of this framework has it do, as timed cases: LoRA training steps of the repository's model
configurations, and the single operations those steps are built from, through the public entry points (``Gpu`` and
``PeftModel``, i.e. the C ABI of ``include/hos_hip.h``).

Kinds (``case["kind"]``):
  step   a short run of optimizer steps on one resident batch, then the adapters and the last gradients are read back
  linear a frozen quantized projection, forward or input gradient, at a precision mode, with or without the fused
         rank-r LoRA term
  lora   the gradient products of one LoRA branch (u, dA, dB)
  attn   causal GQA attention, forward and backward
  ce     softmax cross-entropy over the vocabulary, loss and logit gradient
  block  the elementwise part of a layer: RMSNorm forward and backward, SwiGLU forward and backward

Inputs are made on the device from the seed alone. Quantized weights are ~N(0, 0.02) values packed into GGUF blocks
here (block layouts: src/gguf.rs:354-477), so the reference results below need nothing of the library.
"""
import dataclasses
import itertools
import math

import numpy as np
import torch

from hos_amd import Gpu, synth
from hos_amd.hip_be import GGML_F32, GGML_Q4_K, GGML_Q6_K, GGML_Q8_0
from hos_amd.peft import PeftModel

TYPES = {"F32": GGML_F32, "Q8_0": GGML_Q8_0, "Q4_K": GGML_Q4_K, "Q6_K": GGML_Q6_K}
DEV = "cuda:0"
F64 = torch.float64


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # Fine-tuning runs. The repository's smallest configuration (one short sequence: launches and latency), its
        # benchmark configuration, and its mixture-of-experts architecture at full layer width, two layers of it.
        {"name": "step_smollm2_1x128", "kind": "step", "model": "smollm2-135m", "layers": 30, "B": 1, "T": 128,
         "steps": 32},
        {"name": "step_qwen_4x512", "kind": "step", "model": "qwen2.5-0.5b", "layers": 24, "B": 4, "T": 512,
         "steps": 16},
        {"name": "step_olmoe2_4x512", "kind": "step", "model": "olmoe", "layers": 2, "B": 4, "T": 512, "steps": 4},
        # Projections. A short sequence through a narrow layer (the smallest call).
        {"name": "fwd_q8_1536x576_t128", "kind": "linear", "dx": False, "type": "Q8_0", "rows": 1536, "cols": 576,
         "t": 128, "passes": 5, "rank": 0},
        # The gate (or up) projection of a 1B model over the benchmark's 8 x 1024 tokens with its adapter fused, at the
        # precision the training step uses.
        {"name": "fwd_q4k_8192x2048_t8192_r32", "kind": "linear", "dx": False, "type": "Q4_K", "rows": 8192,
         "cols": 2048, "t": 8192, "passes": 5, "rank": 32},
        # The isolated input-gradient GEMM of the benchmark, 4096 cubed in one fp16 pass.
        {"name": "dx_q4k_4096cubed_p1", "kind": "linear", "dx": True, "type": "Q4_K", "rows": 4096, "cols": 4096,
         "t": 4096, "passes": 1, "rank": 0},
        # The down projection's input gradient over a ragged batch (999 tokens), weights in the 6-bit encoding, at the
        # precision the training step uses.
        {"name": "dx_q6k_2048x8192_t999_p3", "kind": "linear", "dx": True, "type": "Q6_K", "rows": 2048,
         "cols": 8192, "t": 999, "passes": 3, "rank": 0},
        # One LoRA branch's gradients on the benchmark's shapes.
        {"name": "lora_4096_r16", "kind": "lora", "rows": 4096, "in": 4096, "out": 4096, "rank": 16},
        # Attention of a 1B model at the benchmark's batch, and head size 128 with a ragged sequence length.
        {"name": "attn_8x1024_h32kv8_d64", "kind": "attn", "B": 8, "T": 1024, "nh": 32, "nkv": 8, "hd": 64},
        {"name": "attn_3x333_h16kv16_d128", "kind": "attn", "B": 3, "T": 333, "nh": 16, "nkv": 16, "hd": 128},
        # The loss over the largest vocabulary of the configurations.
        {"name": "ce_2048x151936", "kind": "ce", "rows": 2048, "V": 151936},
        # The elementwise part of a layer at the benchmark's batch.
        {"name": "block_2048_d896_f4864", "kind": "block", "rows": 2048, "d": 896, "F": 4864},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "linear", "linear", "linear", "lora", "attn", "ce", "block"])
    if kind == "step":
        model = rng.choice(["smollm2-135m", "qwen2.5-0.5b", "llama3.2-1b", "olmoe"])
        most = {"smollm2-135m": 30, "qwen2.5-0.5b": 24, "llama3.2-1b": 4, "olmoe": 2}[model]
        B = rng.randint(1, 4)
        return {"kind": "step", "model": model, "layers": rng.randint(1, most), "B": B, "T": _log(rng, 32, 512),
                "steps": rng.randint(4, 16)}
    if kind == "linear":
        ty = rng.choice(["Q8_0", "Q4_K", "Q6_K", "F32"])
        unit = 256 if ty in ("Q4_K", "Q6_K") else 32
        rows, cols = 32 * _log(rng, 4, 304), unit * _log(rng, max(1, 256 // unit), 8192 // unit)
        t = min(_log(rng, 16, 8192), int(1.4e11 / (rows * cols)))
        return {"kind": "linear", "dx": rng.random() < 0.5, "type": ty, "rows": rows, "cols": cols, "t": t,
                "passes": rng.choice([1, 3, 5]), "rank": rng.choice([0, 0, 16, 32])}
    if kind == "lora":
        return {"kind": "lora", "rows": _log(rng, 64, 4096), "in": 64 * _log(rng, 9, 128),
                "out": 64 * _log(rng, 2, 128), "rank": rng.choice([8, 16, 32])}
    if kind == "attn":
        nh, nkv, hd = rng.choice([(9, 3, 64), (14, 2, 64), (32, 8, 64), (16, 16, 128)])
        return {"kind": "attn", "B": rng.randint(1, 8), "T": _log(rng, 32, 1024), "nh": nh, "nkv": nkv, "hd": hd}
    if kind == "ce":
        return {"kind": "ce", "rows": _log(rng, 32, 2048), "V": _log(rng, 2000, 151936)}
    d, F = rng.choice([(576, 1536), (896, 4864), (2048, 8192), (2048, 1024)])
    return {"kind": "block", "rows": _log(rng, 32, 4096), "d": d, "F": F}


# ---------------------------------------------------------------- inputs
_gpu = None
_keys = itertools.count(0x1000)


def gpu():
    """The program's one device context."""
    global _gpu
    if _gpu is None:
        _gpu = Gpu(0)
    return _gpu


def _gen(seed, salt):
    g = torch.Generator(DEV)
    g.manual_seed(seed * 1009 + salt)
    return g


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32).mul_(std)


def _f16_bytes(x):
    """f16 values [n] as little-endian byte pairs [n, 2]."""
    return x.to(torch.float16).reshape(-1, 1).view(torch.uint8)


def pack(w, ty):
    """GGUF bytes (uint8, on the device) of an f32 matrix."""
    if ty == GGML_F32:
        return w.contiguous().view(torch.uint8).reshape(-1)
    if ty == GGML_Q8_0:
        b = w.reshape(-1, 32)
        d = (b.abs().amax(1) / 127).to(torch.float16)
        q = (b / d.float().clamp_min(1e-8)[:, None]).round_().clamp_(-127, 127).to(torch.int8)
        return torch.cat([_f16_bytes(d), q.view(torch.uint8)], 1).reshape(-1)
    if ty == GGML_Q4_K:
        b = w.reshape(-1, 8, 32)
        lo, hi = b.amin(2).clamp_max(0), b.amax(2)
        sc, mn = (hi - lo) / 15, -lo
        d, dm = (sc.amax(1) / 63).to(torch.float16), (mn.amax(1) / 63).to(torch.float16)
        s6 = (sc / d.float().clamp_min(1e-8)[:, None]).round().clamp(0, 63)
        m6 = (mn / dm.float().clamp_min(1e-8)[:, None]).round().clamp(0, 63)
        step = (d.float()[:, None] * s6).clamp_min(1e-12)[..., None]
        q = ((b + (dm.float()[:, None] * m6)[..., None]) / step).round_().clamp_(0, 15).to(torch.uint8)
        s, m = s6.to(torch.uint8), m6.to(torch.uint8)
        packed = torch.cat([s[:, :4] | (s[:, 4:] >> 4) << 6, m[:, :4] | (m[:, 4:] >> 4) << 6,
                            (s[:, 4:] & 15) | (m[:, 4:] & 15) << 4], 1)
        q = q.reshape(-1, 4, 2, 32)
        qs = (q[:, :, 0] | q[:, :, 1] << 4).reshape(-1, 128)
        return torch.cat([_f16_bytes(d), _f16_bytes(dm), packed, qs], 1).reshape(-1)
    b = w.reshape(-1, 16, 16)  # Q6_K
    sc = b.abs().amax(2) / 31
    d = (sc.amax(1) / 127).to(torch.float16)
    s8 = (sc / d.float().clamp_min(1e-10)[:, None]).round().clamp(1, 127)
    q = (b / (d.float()[:, None] * s8).clamp_min(1e-12)[..., None]).round_().clamp_(-32, 31)
    q = (q + 32).to(torch.uint8).reshape(-1, 2, 4, 32)
    ql = torch.cat([q[:, :, 0] & 15 | (q[:, :, 2] & 15) << 4, q[:, :, 1] & 15 | (q[:, :, 3] & 15) << 4], 2)
    qh = q[:, :, 0] >> 4 | (q[:, :, 1] >> 4) << 2 | (q[:, :, 2] >> 4) << 4 | (q[:, :, 3] >> 4) << 6
    return torch.cat([ql.reshape(-1, 128), qh.reshape(-1, 64), s8.to(torch.int8).view(torch.uint8),
                      _f16_bytes(d)], 1).reshape(-1)


def unpack(raw, ty, rows, cols):
    """The matrix that GGUF bytes stand for, in 64 bits (on the device)."""
    if ty == GGML_F32:
        return raw.view(torch.float32).reshape(rows, cols).to(F64)

    def f16(b):
        return b.contiguous().view(torch.float16).to(F64)
    if ty == GGML_Q8_0:
        b = raw.reshape(-1, 34)
        return (f16(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).to(F64)).reshape(rows, cols)
    if ty == GGML_Q4_K:
        b = raw.reshape(-1, 144)
        p = b[:, 4:16]
        s = torch.cat([p[:, :4] & 63, (p[:, 8:] & 15) | (p[:, :4] >> 6) << 4], 1).to(F64)
        m = torch.cat([p[:, 4:8] & 63, p[:, 8:] >> 4 | (p[:, 4:8] >> 6) << 4], 1).to(F64)
        qs = b[:, 16:].reshape(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).to(F64)
        return ((f16(b[:, :2]) * s)[..., None] * q - (f16(b[:, 2:4]) * m)[..., None]).reshape(rows, cols)
    b = raw.reshape(-1, 210)
    ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 32)
    q = torch.stack([ql[:, :, 0] & 15 | (qh & 3) << 4, ql[:, :, 1] & 15 | (qh >> 2 & 3) << 4,
                     ql[:, :, 0] >> 4 | (qh >> 4 & 3) << 4, ql[:, :, 1] >> 4 | (qh >> 6) << 4], 2)
    q = q.reshape(-1, 16, 16).to(F64) - 32
    s = b[:, 192:208].contiguous().view(torch.int8).to(F64) * f16(b[:, 208:])
    return (s[..., None] * q).reshape(rows, cols)


class Weight:
    """A quantized weight uploaded under a key of its own, evicted with its last user."""

    def __init__(self, raw, ty, rows, cols):
        self.key = next(_keys)
        gpu().upload_quant(self.key, raw.cpu().numpy(), ty, rows, cols)

    def __del__(self):
        gpu().evict(self.key)


def _linear_inputs(case, seed):
    g = _gen(seed, 1)
    ty, rows, cols, t, r = TYPES[case["type"]], case["rows"], case["cols"], case["t"], case["rank"]
    raw = pack(_randn(g, rows, cols, std=0.02), ty)
    # normalized activations forward, small gradients backward
    x = _randn(g, t, rows if case["dx"] else cols, std=1e-2 if case["dx"] else 1.0)
    u = _randn(g, t, r, std=1e-3 if case["dx"] else 0.6) if r else None
    f = _randn(g, r, cols if case["dx"] else rows, std=0.02) if r else None
    return raw, x, u, f


def _step_config(case):
    return dataclasses.replace(synth.CONFIGS[case["model"]], n_layers=case["layers"], batch=case["B"], seq=case["T"])


def _step_inputs(case, seed):
    """(config, name -> (bytes on the device, type, rows, cols), adapters, ids, targets)"""
    cfg = _step_config(case)
    g = _gen(seed, 2)
    tensors = {}
    for name, rows, cols, kind in synth.tensor_list(cfg):
        if kind == "norm":
            ty, w = GGML_F32, 1.0 + 0.1 * _randn(g, rows, cols)
        elif kind in ("bias", "router"):
            ty, w = GGML_F32, _randn(g, rows, cols, std=0.02)
        else:
            ty = synth.storage_type(cfg.head_quant if kind == "head" else cfg.quant, cols)
            w = _randn(g, rows, cols, std=0.02)
        tensors[name] = (pack(w, ty), ty, rows, cols)
    # an adapter taken up again: B is no longer zero
    lora = {}
    for layer in range(cfg.n_layers):
        for t in cfg.lora_targets:
            i, o = cfg.target_dims(t)
            lora[layer, t] = (_randn(g, i, cfg.lora_rank, std=0.02), _randn(g, cfg.lora_rank, o, std=0.02))
    ids = torch.randint(0, cfg.vocab, (case["B"], case["T"] + 1), generator=g, device=DEV, dtype=torch.int32)
    return cfg, tensors, lora, ids[:, :-1].contiguous(), ids[:, 1:].contiguous()


def _attn_inputs(case, seed):
    g = _gen(seed, 3)
    B, T, nh, nkv, hd = (case[k] for k in ("B", "T", "nh", "nkv", "hd"))
    return _randn(g, B * T, (nh + 2 * nkv) * hd), _randn(g, B * T, nh * hd, std=1e-2)


def _ce_inputs(case, seed):
    g = _gen(seed, 4)
    logits = _randn(g, case["rows"], case["V"], std=1.5)
    tg = torch.randint(0, case["V"], (case["rows"],), generator=g, device=DEV, dtype=torch.int32)
    return logits, tg


def _lora_inputs(case, seed):
    g = _gen(seed, 5)
    m, i, o, r = case["rows"], case["in"], case["out"], case["rank"]
    return _randn(g, m, i), _randn(g, m, o, std=1e-2), _randn(g, i, r, std=0.02), _randn(g, r, o, std=0.02)


def _block_inputs(case, seed):
    g = _gen(seed, 6)
    m, d, F = case["rows"], case["d"], case["F"]
    return (_randn(g, m, d), 1.0 + 0.1 * _randn(g, d), _randn(g, m, d, std=1e-2), _randn(g, m, 2 * F),
            _randn(g, m, F, std=1e-2))


EPS = 1e-6
LR = 1e-4
SCALE = 2.0


class Linear:
    def __init__(self, case, seed):
        self.case = case
        raw, self.x, self.u, self.f = _linear_inputs(case, seed)
        self.w = Weight(raw, TYPES[case["type"]], case["rows"], case["cols"])
        self.out = torch.empty(case["t"], case["cols"] if case["dx"] else case["rows"], device=DEV)
        gpu().set_gemm_passes(case["passes"])

    def run(self):
        c = self.case
        if c["rank"]:
            gpu().op_async("qgemm_lora_dev", int(c["dx"]), self.w.key, self.x.data_ptr(), c["t"], self.u.data_ptr(),
                           c["rank"], self.f.data_ptr(), self.f.shape[1], 1, c["rank"], SCALE, self.out.data_ptr())
        else:
            gpu().op_async("qgemm_dx_dev" if c["dx"] else "qgemm_fwd_dev", self.w.key, self.x.data_ptr(), c["t"],
                           self.out.data_ptr())
        return self.out


class Lora:
    def __init__(self, case, seed):
        self.case = case
        self.x, self.dy, self.A, self.B = _lora_inputs(case, seed)
        self.u = torch.empty(case["rows"], case["rank"], device=DEV)
        self.dA, self.dB = torch.empty_like(self.A), torch.empty_like(self.B)

    def run(self):
        c = self.case
        gpu().op_async("lora", self.x.data_ptr(), self.dy.data_ptr(), c["rows"], c["in"], c["out"], c["rank"],
                       self.A.data_ptr(), self.B.data_ptr(), SCALE, None, self.u.data_ptr(), self.dA.data_ptr(),
                       self.dB.data_ptr(), None)
        return self.u, self.dA, self.dB


class Attn:
    def __init__(self, case, seed):
        self.case = case
        self.qkv, self.do = _attn_inputs(case, seed)
        self.o, self.dqkv = torch.empty_like(self.do), torch.empty_like(self.qkv)
        self.lse = torch.empty(case["B"], case["nh"], case["T"], device=DEV)

    def run(self):
        B, T, nh, nkv, hd = (self.case[k] for k in ("B", "T", "nh", "nkv", "hd"))
        ld, kc, vc = (nh + 2 * nkv) * hd, nh * hd, (nh + nkv) * hd
        g = gpu()
        g.op_async("attention_fwd", self.qkv.data_ptr(), ld, kc, vc, B, T, nh, nkv, hd, self.o.data_ptr(), nh * hd,
                   self.lse.data_ptr())
        g.op_async("attention_bwd", self.qkv.data_ptr(), ld, kc, vc, self.o.data_ptr(), self.do.data_ptr(), nh * hd,
                   self.lse.data_ptr(), B, T, nh, nkv, hd, self.dqkv.data_ptr(), ld)
        return self.o, self.lse, self.dqkv


class CrossEntropy:
    def __init__(self, case, seed):
        self.case = case
        self.logits, self.tg = _ce_inputs(case, seed)
        self.loss, self.dl = torch.empty(case["rows"], device=DEV), torch.empty_like(self.logits)

    def run(self):
        c = self.case
        gpu().op_async("cross_entropy", self.logits.data_ptr(), c["rows"], c["V"], self.tg.data_ptr(),
                       1.0 / c["rows"], self.loss.data_ptr(), self.dl.data_ptr())
        return self.loss, self.dl


class Block:
    def __init__(self, case, seed):
        self.case = case
        self.x, self.w, self.g, self.gu, self.dh = _block_inputs(case, seed)
        self.y, self.gx = torch.empty_like(self.x), torch.empty_like(self.x)
        self.inv = torch.empty(case["rows"], device=DEV)
        self.h, self.dgu = torch.empty_like(self.dh), torch.empty_like(self.gu)

    def run(self):
        m, d, F = (self.case[k] for k in ("rows", "d", "F"))
        g = gpu()
        g.op_async("rmsnorm_fwd", self.x.data_ptr(), self.w.data_ptr(), m, d, EPS, self.y.data_ptr(),
                   self.inv.data_ptr())
        g.op_async("swiglu_fwd", self.gu.data_ptr(), m, F, self.h.data_ptr())
        g.op_async("swiglu_bwd", self.gu.data_ptr(), self.dh.data_ptr(), m, F, self.dgu.data_ptr())
        g.op_async("rmsnorm_bwd", self.g.data_ptr(), self.x.data_ptr(), self.inv.data_ptr(), self.w.data_ptr(), m, d,
                   self.gx.data_ptr())
        return self.y, self.inv, self.h, self.dgu, self.gx


class Step:
    """A model with a resident batch. A pass is a few optimizer steps; then the loss of the last one, the adapters and
    its gradients are read (stacked over the layers, per target), as a program does at a checkpoint."""

    def __init__(self, case, seed):
        self.case = case
        self.cfg, tensors, lora, self.ids, self.tg = _step_inputs(case, seed)
        self.pm = PeftModel(gpu(), self.cfg)
        for name, (raw, ty, rows, cols) in tensors.items():
            self.pm.set_tensor(name, raw.cpu().numpy(), ty, rows, cols)
        for (layer, t), (A, B) in lora.items():
            self.pm.set_lora(layer, t, A.cpu().numpy(), B.cpu().numpy())
        self.loss = torch.empty(1, device=DEV)

    def run(self):
        c, cfg = self.case, self.cfg
        for _ in range(c["steps"]):
            self.pm.step_dev(self.ids.data_ptr(), self.tg.data_ptr(), c["B"], c["T"], LR, 0.0, self.loss.data_ptr())
        gpu().synchronize()
        out = {"loss": float(self.loss)}
        for t in cfg.lora_targets:
            factors = [self.pm.get_lora(layer, t) for layer in range(cfg.n_layers)]
            grads = [self.pm.get_lora_grad(layer, t) for layer in range(cfg.n_layers)]
            out[t] = [np.stack(z) for z in (*zip(*factors), *zip(*grads))]
        return out


KINDS = {"step": Step, "linear": Linear, "lora": Lora, "attn": Attn, "ce": CrossEntropy, "block": Block}


def prepare(case, seed):
    s = KINDS[case["kind"]](case, seed)
    torch.cuda.synchronize()  # the library has a stream of its own: the inputs are there before its first call
    return s


def run(state):
    return state.run()


# ---------------------------------------------------------------- what a pass cannot do without
def _gguf_bytes(ty, n):
    return {GGML_F32: 4, GGML_Q8_0: 34 / 32, GGML_Q4_K: 144 / 256, GGML_Q6_K: 210 / 256}[ty] * n


def work(case):
    k = case["kind"]
    if k == "linear":
        t, n = case["t"], case["rows"] * case["cols"]
        r = case["rank"]
        width = case["rows"] + case["cols"]
        return {"bytes": 4.0 * t * (width + r) + 4.0 * r * (case["cols"] if case["dx"] else case["rows"]) +
                _gguf_bytes(TYPES[case["type"]], n),
                "flops": 2.0 * t * n + 2.0 * t * r * (case["cols"] if case["dx"] else case["rows"])}
    if k == "lora":
        m, w, r = case["rows"], case["in"] + case["out"], case["rank"]
        return {"bytes": 4.0 * (m * w + 2 * r * w + m * r), "flops": 2.0 * 2.0 * m * r * w}
    if k == "attn":
        m, hd = case["B"] * case["T"], case["hd"]
        nh, nkv = case["nh"], case["nkv"]
        # forward: read q, k, v, write o and lse; backward: read them, o and do, write dq, dk, dv
        pairs = case["B"] * nh * case["T"] * (case["T"] + 1) / 2
        return {"bytes": 4.0 * m * (3 * (nh + 2 * nkv) * hd + 3 * nh * hd + 2 * nh), "flops": 2.0 * pairs * hd * 7}
    if k == "ce":
        return {"bytes": 8.0 * case["rows"] * case["V"], "flops": 0}
    if k == "block":
        m, d, F = case["rows"], case["d"], case["F"]
        return {"bytes": 4.0 * m * (2 * d + 3 * F + 5 * F + 3 * d), "flops": 0}
    cfg = _step_config(case)
    tok = case["B"] * case["T"]
    flops = synth.algorithmic_flops_per_token(cfg, case["T"]) * tok
    nbytes = sum(_gguf_bytes(GGML_F32 if kind in ("norm", "bias", "router") else
                             synth.storage_type(cfg.head_quant if kind == "head" else cfg.quant, cols), rows * cols)
                 for _, rows, cols, kind in synth.tensor_list(cfg))
    p_lora = cfg.n_layers * sum(cfg.lora_rank * sum(cfg.target_dims(t)) for t in cfg.lora_targets)
    # every weight once forward and once backward; parameters, gradients and both moments of the adapters
    return {"bytes": case["steps"] * (2 * nbytes + 28.0 * p_lora), "flops": case["steps"] * flops}


def tolerance(case):
    """About four times the largest distance from exact() over the listed and some drawn cases (in parentheses)."""
    k = case["kind"]
    if k == "linear":
        # one pass rounds both operands to fp16 (2.9e-4); three, or integer codes, carry them to ~22 bits (9.1e-7)
        return {"rel": 1.2e-3} if case["passes"] == 1 else {"rel": 4e-6}
    if k == "lora":
        return {"rel": 1.2e-6}  # (3.0e-7)
    if k == "attn":
        return {"rel": 3e-5}  # bf16 hi/lo products, ~2^-16 each (7.2e-6)
    if k in ("ce", "block"):
        return {"rel": 3e-7}  # (6.9e-8)
    # "max": AdamW makes a sign out of a rounding where a gradient is near zero, so single values of the adapters can
    # be off by 2 lr a step
    if synth.CONFIGS[case["model"]].n_experts:
        return {"rel": 0.03, "max": 0.9}  # a selection near a tie goes either way, a token's gradients with it (9.8e-3)
    return {"rel": 8e-4, "max": 0.9}  # (2.0e-4)


# ---------------------------------------------------------------- the same in 64 bits
def exact(case, seed):
    with torch.no_grad():
        return {"step": _exact_step, "linear": _exact_linear, "lora": _exact_lora, "attn": _exact_attn,
                "ce": _exact_ce, "block": _exact_block}[case["kind"]](case, seed)


def _exact_linear(case, seed):
    raw, x, u, f = _linear_inputs(case, seed)
    w = unpack(raw, TYPES[case["type"]], case["rows"], case["cols"])
    y = x.to(F64) @ (w if case["dx"] else w.T)
    return y if u is None else y + SCALE * (u.to(F64) @ f.to(F64))


def _exact_lora(case, seed):
    x, dy, A, B = (v.to(F64) for v in _lora_inputs(case, seed))
    u, du = x @ A, SCALE * (dy @ B.T)
    return u, x.T @ du, SCALE * (u.T @ dy)


def _heads(x, B, T, n, hd):
    return x.reshape(B, T, n, hd).transpose(1, 2).reshape(B * n, T, hd).contiguous()


def _exact_attn(case, seed):
    B, T, nh, nkv, hd = (case[k] for k in ("B", "T", "nh", "nkv", "hd"))
    qkv, do = (v.to(F64) for v in _attn_inputs(case, seed))
    gr, qd, kvd = nh // nkv, nh * hd, nkv * hd
    o, lse, dqkv = torch.empty_like(do), torch.empty(B, nh, T, device=DEV, dtype=F64), torch.zeros_like(qkv)
    mask = torch.ones(T, T, device=DEV, dtype=torch.bool).triu(1)
    for b in range(B):
        rows = slice(b * T, (b + 1) * T)
        for h in range(nh):
            cq, ck, cv = (slice(c, c + hd) for c in (h * hd, qd + h // gr * hd, qd + kvd + h // gr * hd))
            q, k, v, g = qkv[rows, cq], qkv[rows, ck], qkv[rows, cv], do[rows, cq]
            s = (q @ k.T / math.sqrt(hd)).masked_fill_(mask, -math.inf)
            lse[b, h] = s.logsumexp(1)
            p = torch.exp(s - lse[b, h][:, None])
            o[rows, cq] = p @ v
            dp = g @ v.T
            ds = p * (dp - (dp * p).sum(1, keepdim=True)) / math.sqrt(hd)
            dqkv[rows, cq] = ds @ k
            dqkv[rows, ck] += ds.T @ q
            dqkv[rows, cv] += p.T @ g
    return o, lse, dqkv


def _exact_ce(case, seed):
    logits, tg = _ce_inputs(case, seed)
    rows = torch.arange(case["rows"], device=DEV)
    p = torch.softmax(logits.to(F64), 1)
    loss = -torch.log(p[rows, tg.long()].clamp_min(1e-12))
    p[rows, tg.long()] -= 1
    return loss, p.mul_(1.0 / case["rows"])


def _exact_block(case, seed):
    x, w, g, gu, dh = (v.to(F64) for v in _block_inputs(case, seed))
    inv = 1 / torch.sqrt(x.square().mean(1) + EPS)
    xn = x * inv[:, None]
    gw = g * w
    gx = inv[:, None] * (gw - xn * (gw * xn).mean(1, keepdim=True))
    a, b = gu[:, :case["F"]], gu[:, case["F"]:]
    s = torch.sigmoid(a)
    dgu = torch.cat([dh * b * s * (1 + a * (1 - s)), dh * a * s], 1)
    return xn * w, inv, a * s * b, dgu, gx


def _rope(x, cs, sn, neox):
    """x [B, T, n, hd] rotated by the angles' cos / sin [T, hd/2]."""
    h = x.shape[-1] // 2
    cs, sn = cs[None, :, None], sn[None, :, None]
    if neox:
        a, b = x[..., :h], x[..., h:]
        return torch.cat([a * cs - b * sn, a * sn + b * cs], -1)
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * cs - b * sn, a * sn + b * cs], -1).flatten(-2)


def _exact_step(case, seed):
    if _step_config(case).n_experts:
        return None  # the selection of experts is no continuous function: near a tie, 64 bits select others
    cfg, tensors, lora, ids, tg = _step_inputs(case, seed)
    B, T, L = case["B"], case["T"], cfg.n_layers
    nh, nkv, hd, s = cfg.n_heads, cfg.n_kv_heads, cfg.head_dim, cfg.lora_alpha / cfg.lora_rank
    W = {n: unpack(raw, ty, r, c) for n, (raw, ty, r, c) in tensors.items()}
    P = {k: [v.to(F64).requires_grad_() for v in ab] for k, ab in lora.items()}
    flat = [v for ab in P.values() for v in ab]
    m1, v1 = [torch.zeros_like(v) for v in flat], [torch.zeros_like(v) for v in flat]
    f32 = np.float32  # the rotation angles are f32 by definition of the op (src/tensor.rs:2769-2778)
    freq = (f32(1) / np.power(f32(cfg.rope_base), f32(2) * np.arange(hd // 2, dtype=f32) / f32(hd))).astype(f32)
    ang = torch.from_numpy(np.arange(T, dtype=f32)[:, None] * freq).to(DEV, F64)
    cs, sn = ang.cos(), ang.sin()
    mask = torch.ones(T, T, device=DEV, dtype=torch.bool).triu(1)

    def norm(x, w):
        return x / torch.sqrt(x.square().mean(-1, keepdim=True) + cfg.rms_eps) * w

    def proj(layer, t, leaf, x):
        y = x @ W[f"blk.{layer}.{leaf}.weight"].T
        if (layer, t) in P:
            A, Bf = P[layer, t]
            y = y + s * (x @ A @ Bf)
        return y

    def block(layer, x):
        p = f"blk.{layer}."
        xn = norm(x, W[p + "attn_norm.weight"])
        q, k, v = (proj(layer, t, "attn_" + t, xn) for t in "qkv")
        if cfg.attn_bias:
            q, k, v = q + W[p + "attn_q.bias"], k + W[p + "attn_k.bias"], v + W[p + "attn_v.bias"]
        q, k = (_rope(z.reshape(B, T, n, hd), cs, sn, cfg.rope_neox) for z, n in ((q, nh), (k, nkv)))
        k, v = (z.reshape(B, T, nkv, hd).repeat_interleave(nh // nkv, 2) for z in (k, v))
        q, k, v = (_heads(z, B, T, nh, hd) for z in (q, k, v))
        a = torch.softmax((torch.bmm(q, k.transpose(1, 2).contiguous()) / math.sqrt(hd))
                          .masked_fill(mask, -math.inf), 2)
        o = torch.bmm(a, v).reshape(B, nh, T, hd).transpose(1, 2).reshape(B * T, nh * hd)
        x = x + proj(layer, "o", "attn_output", o)
        xn = norm(x, W[p + "ffn_norm.weight"])
        h = torch.nn.functional.silu(proj(layer, "gate", "ffn_gate", xn)) * proj(layer, "up", "ffn_up", xn)
        return x + proj(layer, "down", "ffn_down", h)

    head = W.get("output.weight", W["token_embd.weight"])
    for step in range(1, case["steps"] + 1):
        with torch.enable_grad():
            x = W["token_embd.weight"][ids.reshape(-1).long()]
            for layer in range(L):
                x = block(layer, x)
            z = norm(x, W["output_norm.weight"]) @ head.T
            loss = torch.nn.functional.cross_entropy(z, tg.reshape(-1).long())
            grads = torch.autograd.grad(loss, flat)
        for v, gr, m, q in zip(flat, grads, m1, v1):
            m.mul_(0.9).add_(gr, alpha=0.1)
            q.mul_(0.95).addcmul_(gr, gr, value=0.05)
            v.sub_(LR * (m / (1 - 0.9 ** step)) / (torch.sqrt(q / (1 - 0.95 ** step)) + 1e-8))
        del z, x
    G = {k: grads[2 * i:2 * i + 2] for i, k in enumerate(P)}
    out = {"loss": float(loss)}
    for t in cfg.lora_targets:
        out[t] = [torch.stack([D[layer, t][i].detach() for layer in range(L)]) for D in (P, G) for i in (0, 1)]
    return out

