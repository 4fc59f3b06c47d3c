"""The work this framework is measured on: the blocks of the forward pass and three whole calls.

Every case runs through the public entry points, as a program that serves a GGUF model calls them:
the C ABI's entries for single blocks (axon_hip.call), axon_hip.Model for whole passes. Sizes are
those of the benchmark's models (synth.CONFIGS) and of its kernel sweep; drawn cases spread over
the ranges between and around them, odd sizes among them.

Kinds, and what in real use each stands for:
  mlp      the feed-forward block of one layer: RMSNorm and Q8_0 quantization of the residual rows,
           gate|up with SiLU * up, down added to the residual stream.
  proj     one weight matrix through its kernel-table entry (matmul_<type>[_q8][_rows]): attention
           projections, down matrices, models stored in F16 / BF16 / F32.
  attn     one layer's attention over cached keys and values: the rows of a ragged decode batch, or
           a chunk of a prompt behind its earlier positions.
  head     the Q6_K output matrix over its upload-time planar copy, and the greedy ids of its rows.
  sample   the top-k candidates of every row of a batch's logits.
  decode   greedy generation of one sequence on the Llama-3.2-1B-shaped Q4_0 model.
  batch    decode steps of a ragged batch of sequences on it.
  prefill  a prompt into an empty cache on it, in chunks of 512, with its last row's logits.
"""
from __future__ import annotations

import ctypes as C
import math
import random
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "axon-infer_amd"))

import axon_hip as H  # noqa: E402
import synth  # noqa: E402

TYPES = {"f32": H.F32, "f16": H.F16, "bf16": H.BF16, "q4_0": H.Q4_0, "q4_1": H.Q4_1, "q8_0": H.Q8_0, "q6_k": H.Q6_K}
BITS = {"f32": 32, "f16": 16, "bf16": 16, "q4_0": 4.5, "q4_1": 5, "q8_0": 8.5, "q6_k": 210 / 32}
HEAD_DIM = 64
EPS = 1e-5
SPEC = synth.LLAMA32_1B
MAX_CTX = 2304   # positions of a sequence's cache: the benchmark's contexts and some decode steps
CHUNK = 512      # prompt tokens per pass
HEADS = ((9, 3), (32, 4), (32, 8), (14, 2))  # query heads / KV heads of the benchmark's models


def listed():
    return [
        # The smallest block: one decode row of SmolLM2-135M's feed-forward, two launches.
        {"name": "mlp-1x576-q8_0", "kind": "mlp", "type": "q8_0", "rows": 1, "n_embd": 576, "n_ff": 1536},
        # A batch of 17 sequences in decode (one more than a tile of 16) on the 1B shape.
        {"name": "mlp-17x2048-q4_0", "kind": "mlp", "type": "q4_0", "rows": 17, "n_embd": 2048, "n_ff": 8192},
        # A full prompt chunk on the 1B shape: most of prefill's time.
        {"name": "mlp-512x2048-q4_0", "kind": "mlp", "type": "q4_0", "rows": 512, "n_embd": 2048, "n_ff": 8192},
        # gate|up-sized Q4_1 projection of a prompt chunk (published Q4_0 files hold some Q4_1 tensors).
        {"name": "proj-512-q4_1", "kind": "proj", "type": "q4_1", "rows": 512, "n_out": 5632, "n_in": 2048},
        # A model stored in F16: a batch of 16 rows through one square projection.
        {"name": "proj-16-f16", "kind": "proj", "type": "f16", "rows": 16, "n_out": 2048, "n_in": 2048},
        # The ragged decode batch of the benchmark: 32 sequences, contexts U[64, 2048].
        {"name": "attn-ragged-32", "kind": "attn", "rows": 32, "past": -1, "lo": 64, "hi": 2048, "n_head": 32,
         "n_kv": 8, "f16": False},
        # The second 512-token chunk of a prompt.
        {"name": "attn-prefill-512", "kind": "attn", "rows": 512, "past": 512, "lo": 0, "hi": 0, "n_head": 32,
         "n_kv": 8, "f16": False},
        # The output matrix for the ragged batch, and its greedy ids.
        {"name": "head-32x128256", "kind": "head", "rows": 32, "n_vocab": 128256, "n_embd": 2048},
        # Stochastic sampling of 64 sequences on the Qwen2.5 vocabulary, top-k 40.
        {"name": "sample-64x151936", "kind": "sample", "rows": 64, "n_vocab": 151936, "k": 40},
        # The headline: batch-1 greedy decode behind a 512-token prompt.
        {"name": "decode-b1", "kind": "decode", "ctx": 512, "steps": 16},
        # Eight steps of the 32-sequence ragged batch.
        {"name": "batch-ragged-32", "kind": "batch", "rows": 32, "lo": 64, "hi": 2048, "steps": 8},
        # A 512-token prompt.
        {"name": "prefill-512", "kind": "prefill", "tokens": 512},
    ]


def _log(rng: random.Random, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(("mlp", "mlp", "proj", "proj", "attn", "attn", "head", "sample", "decode", "batch", "prefill"))
    if kind == "mlp":
        return {"kind": kind, "type": rng.choice(("q4_0", "q4_0", "q8_0", "q4_1")), "rows": _log(rng, 1, 512),
                "n_embd": 64 * _log(rng, 9, 32), "n_ff": 32 * _log(rng, 48, 256)}
    if kind == "proj":
        t = rng.choice(("q4_0", "q4_1", "q8_0", "q6_k", "f16", "bf16", "f32"))
        unit = 256 if t == "q6_k" else 32
        n_in = unit * _log(rng, 512 // unit, 8192 // unit)
        rows = _log(rng, 1, 512 if t in ("q4_0", "q4_1", "q8_0") else 64)
        # Wide and deep at once costs more than any listed case: the product of the sizes is bounded.
        cap = (1 << 33) if t in ("q4_0", "q4_1", "q8_0") else (1 << 29)
        n_out = min(_log(rng, 300, 16384), max(300, cap // (rows * n_in)))
        return {"kind": kind, "type": t, "rows": rows, "n_out": n_out, "n_in": n_in}
    if kind == "attn":
        n_head, n_kv = rng.choice(HEADS)
        f16 = rng.random() < 0.5
        if rng.random() < 0.5:
            hi = _log(rng, 64, 2048)
            return {"kind": kind, "rows": _log(rng, 1, 64), "past": -1, "lo": rng.randint(1, hi), "hi": hi,
                    "n_head": n_head, "n_kv": n_kv, "f16": f16}
        return {"kind": kind, "rows": _log(rng, 33, 512), "past": rng.choice((0, rng.randint(1, 1024))), "lo": 0,
                "hi": 0, "n_head": n_head, "n_kv": n_kv, "f16": f16}
    if kind == "head":
        return {"kind": kind, "rows": _log(rng, 1, 64), "n_vocab": _log(rng, 4000, 128256),
                "n_embd": 256 * rng.randint(2, 8)}
    if kind == "sample":
        return {"kind": kind, "rows": _log(rng, 1, 64), "n_vocab": _log(rng, 4000, 151936), "k": _log(rng, 1, 256)}
    if kind == "decode":
        return {"kind": kind, "ctx": _log(rng, 32, 2048), "steps": rng.randint(4, 32)}
    if kind == "batch":
        return {"kind": kind, "rows": _log(rng, 2, 32), "lo": 64, "hi": _log(rng, 128, 2048), "steps": rng.randint(2, 8)}
    return {"kind": kind, "tokens": _log(rng, 33, 2048)}


# ---------------------------------------------------------------------------------------------
# Inputs: made on the GPU from the seed, the same for prepare() and exact()

def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(shape, gen, std=1.0, mean=0.0) -> torch.Tensor:
    return torch.randn(shape, generator=gen, device="cuda") * std + mean


def _round_away(v: torch.Tensor) -> torch.Tensor:
    t = torch.trunc(v)
    return t + torch.where((v - t).abs() >= 0.5, torch.sign(v), torch.zeros_like(v))


def _inverse(d: torch.Tensor) -> torch.Tensor:
    return torch.where(d != 0, 1.0 / torch.where(d != 0, d, torch.ones_like(d)), torch.zeros_like(d))


def _half_bytes(d: torch.Tensor) -> torch.Tensor:
    return d.to(torch.float16).contiguous().view(torch.uint8).reshape(d.shape[0], 2)


def _blocks(x: torch.Tensor, kind: str, values: bool = False):
    """x [rows, n] as GGUF blocks (uint8 [rows, bytes]) and, with values, the values that the blocks
    hold in 64 bits. The quantizers are those that synth.py writes models with."""
    rows, n = x.shape
    if kind in ("f32", "f16", "bf16"):
        w = x.to({"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[kind]).contiguous()
        return w.view(torch.uint8), w.double() if values else None
    if kind == "q6_k":
        b = x.reshape(-1, 16, 16)
        s = b.abs().amax(2) / 31
        d = (s.amax(1) / 127).to(torch.float16)
        df = d.float()[:, None]
        sc = torch.round(s * _inverse(df)).clamp(-128, 127)
        step = (df * sc)[:, :, None]
        q = (torch.round(b * _inverse(step)).clamp(-32, 31) + 32).to(torch.uint8).reshape(-1, 2, 4, 32)
        ql = torch.cat([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2)
        qh = (q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)
        out = torch.cat([ql.reshape(-1, 128), qh.reshape(-1, 64), sc.to(torch.int8).view(torch.uint8), _half_bytes(d)], 1)
        v = (step.double() * (q.reshape(-1, 16, 16).double() - 32)).reshape(rows, n) if values else None
        return out.reshape(rows, -1).contiguous(), v
    b = x.reshape(-1, 32)
    if kind == "q8_0":
        d = b.abs().amax(1) / 127
        q = _round_away(b * _inverse(d)[:, None])
        out = torch.cat([_half_bytes(d), q.to(torch.int8).view(torch.uint8)], 1)
        v = d.half().double()[:, None] * q.double() if values else None
    else:
        if kind == "q4_0":
            mx = b.gather(1, b.abs().argmax(1, keepdim=True))[:, 0]
            d = mx / -8
            q = torch.trunc(b * _inverse(d)[:, None] + 8.5).clamp(0, 15)
            head = _half_bytes(d)
            v = d.half().double()[:, None] * (q.double() - 8) if values else None
        else:
            lo = b.amin(1)
            d = (b.amax(1) - lo) / 15
            q = torch.trunc((b - lo[:, None]) * _inverse(d)[:, None] + 0.5).clamp(0, 15)
            head = torch.cat([_half_bytes(d), _half_bytes(lo)], 1)
            v = d.half().double()[:, None] * q.double() + lo.half().double()[:, None] if values else None
        u = q.to(torch.uint8)
        out = torch.cat([head, u[:, :16] | (u[:, 16:] << 4)], 1)
    return out.reshape(rows, -1).contiguous(), v.reshape(rows, n) if values else None


def _weights(gen, n_out, n_in, kind, values=False):
    return _blocks(_normal((n_out, n_in), gen, 0.02), kind, values)


def _mlp_inputs(case, seed, values=False):
    g = _generator(seed)
    d, ff, t = case["n_embd"], case["n_ff"], case["type"]
    x = _normal((case["rows"], d), g)
    norm = _normal((d,), g, 0.01, 1.0)
    return x, norm, _weights(g, ff, d, t, values), _weights(g, ff, d, t, values), _weights(g, d, ff, t, values)


def _proj_inputs(case, seed, values=False):
    g = _generator(seed)
    w = _weights(g, case["n_out"], case["n_in"], case["type"], values)
    return w, _normal((case["rows"], case["n_in"]), g)


def _attn_lengths(case, seed):
    """Visible positions per row, and the cache rows of each sequence."""
    r = random.Random(seed)
    if case["past"] >= 0:
        return [case["past"] + i + 1 for i in range(case["rows"])], [case["past"] + case["rows"]]
    n = [r.randint(case["lo"], case["hi"]) for _ in range(case["rows"])]
    return n, n


def _attn_inputs(case, seed):
    """q [rows][heads * dim], and one pool of [K rows, V rows] per sequence."""
    g = _generator(seed)
    q = _normal((case["rows"], case["n_head"] * HEAD_DIM), g)
    _, seqs = _attn_lengths(case, seed)
    kv = _normal((2 * sum(seqs), case["n_kv"] * HEAD_DIM), g)
    return q, kv.half() if case["f16"] else kv


def _head_inputs(case, seed, values=False):
    g = _generator(seed)
    return _weights(g, case["n_vocab"], case["n_embd"], "q6_k", values), _normal((case["rows"], case["n_embd"]), g)


def _sample_inputs(case, seed):
    return _normal((case["rows"], case["n_vocab"]), _generator(seed), 3.0)


# ---------------------------------------------------------------------------------------------
# Preparation

def _p(t) -> C.c_void_p:
    return C.c_void_p(t.data_ptr())


def _empty(*shape, dtype=torch.float32) -> torch.Tensor:
    return torch.zeros(shape, dtype=dtype, device="cuda")


class _Calls:
    """The entry calls of one pass, with what their pointers point at."""

    def __init__(self, outputs, keep):
        self.calls, self.outputs, self.keep = [], outputs, keep

    def add(self, name, *args):
        """args as axon_hip.call takes them; an argument record goes by its address and is kept."""
        self.keep += tuple(a for a in args if isinstance(a, C.Structure))
        self.calls.append((name, [C.c_void_p(C.addressof(a)) if isinstance(a, C.Structure) else a for a in args]))

    def run(self):
        for name, args in self.calls:
            H.call(name, *args)
        return self.outputs


def _fused(t, n_rows, n_in, ws, outs, in_mode, out_mode, ys, **more):
    a = H.MatvecFusedArgs()
    a.type, a.n_seg, a.n_rows, a.n_in, a.in_mode, a.out_mode = t, len(ws), n_rows, n_in, in_mode, out_mode
    for i, (w, n) in enumerate(zip(ws, outs)):
        a.w[i], a.n_out[i] = w.data_ptr(), n
    for i, (y, n) in enumerate(ys):
        a.y[i], a.y_stride[i] = y.data_ptr(), n
    for k, v in more.items():
        setattr(a, k, v)
    return a


def _prepare_mlp(case, seed):
    x, norm, (wg, _), (wu, _), (wd, _) = _mlp_inputs(case, seed)
    n, d, ff, t = case["rows"], case["n_embd"], case["n_ff"], TYPES[case["type"]]
    y = x.clone()                                     # the residual stream that down adds to
    act = _empty(n, ff // 32 * 34, dtype=torch.uint8)  # Q8_0 blocks of SiLU(gate) * up
    xq = _empty(n, d // 32 * 34, dtype=torch.uint8)
    gate, up = _empty(n, ff), _empty(n, ff)
    s = _Calls({"act": act, "y": y}, (x, norm, wg, wu, wd, xq, gate, up))
    lib = H.lib()
    if n <= 4 and lib.axon_hip_matvec_fused_supported(t, 2, C.c_size_t(n), C.c_size_t(d), 1) == 1 \
            and lib.axon_hip_matvec_fused_supported(t, 0, C.c_size_t(n), C.c_size_t(ff), 0) == 1:
        a = _fused(t, n, d, (wg, wu), (ff, ff), 2, 2, [(gate, ff)], x=x.data_ptr(), x_stride=d,
                   norm_w=norm.data_ptr(), eps=EPS, outq=act.data_ptr())
        torch.cuda.synchronize()
        fits = lib.axon_hip_matvec_fused(C.byref(a)) == 0
        if not fits:  # the blocks of the product need whole blocks per workgroup: a launch of their own
            a.outq = None
        s.add("matvec_fused", a)
        if not fits:
            s.add("quantize_rows_q8_0", _p(gate), _p(act), ff, n, ff)
        b = _fused(t, n, ff, (wd,), (d,), 0, 1, [(y, d)], xq=act.data_ptr())
        s.add("matvec_fused", b)
        return s
    s.add("rmsnorm_rows", _p(x), _p(norm), None, _p(xq), d, n, float(EPS))
    if n > 64 or ff >= 4096:
        s.add("matmul_q8_swiglu", C.c_int(t), _p(xq), n, d, _p(wg), _p(wu), ff, None, _p(act))
    else:
        ws, ys, no = (C.c_void_p * 2)(_p(wg), _p(wu)), (C.c_void_p * 2)(_p(gate), _p(up)), (C.c_size_t * 2)(ff, ff)
        s.add("matmul_q8_fused", C.c_int(t), _p(xq), n, d, 2, ws, ys, no, no, C.c_int(0))
        s.add("silu_mul_rows", _p(gate), _p(up), None, _p(act), ff, n)
    s.add("matmul_q8_fused", C.c_int(t), _p(act), n, ff, 1, (C.c_void_p * 1)(_p(wd)), (C.c_void_p * 1)(_p(y)),
          (C.c_size_t * 1)(d), (C.c_size_t * 1)(d), C.c_int(1))
    return s


def _prepare_proj(case, seed):
    (w, _), x = _proj_inputs(case, seed)
    n, n_out, n_in, t = case["rows"], case["n_out"], case["n_in"], case["type"]
    y = _empty(n, n_out)
    q8 = t in ("q4_0", "q4_1", "q8_0")
    a = _blocks(x, "q8_0")[0] if q8 else x.contiguous()
    s = _Calls(y, (w, a))
    name = "matmul_" + t + ("_q8" if q8 else "")
    if n == 1:
        s.add(name, _p(w), _p(a), _p(y), n_out, n_in)
    else:
        s.add(name + "_rows", _p(w), _p(a), _p(y), n, n_out, n_in, n_out)
    return s


def _prepare_attn(case, seed):
    q, kv = _attn_inputs(case, seed)
    vis, seqs = _attn_lengths(case, seed)
    n, n_head, n_kv = case["rows"], case["n_head"], case["n_kv"]
    row = n_kv * HEAD_DIM
    starts, at = [], 0
    for m in seqs:
        starts.append(at)
        at += 2 * m * row
    seq_of = range(n) if case["past"] < 0 else [0] * n
    k_off = torch.tensor([starts[i] for i in seq_of], dtype=torch.int64, device="cuda")
    v_off = torch.tensor([starts[i] + seqs[i] * row for i in seq_of], dtype=torch.int64, device="cuda")
    n_vis = torch.tensor(vis, dtype=torch.int32, device="cuda")
    out, outq = _empty(n, n_head * HEAD_DIM), _empty(n, n_head * HEAD_DIM // 32 * 34, dtype=torch.uint8)
    a = H.AttentionRowsArgs()
    a.q, a.out, a.q_stride, a.out_stride = q.data_ptr(), out.data_ptr(), n_head * HEAD_DIM, n_head * HEAD_DIM
    a.kv, a.k_off, a.v_off, a.n_vis = kv.data_ptr(), k_off.data_ptr(), v_off.data_ptr(), n_vis.data_ptr()
    a.n_head, a.n_kv, a.head_dim, a.scale, a.f16 = n_head, n_kv, HEAD_DIM, HEAD_DIM ** -0.5, int(case["f16"])
    a.max_vis, a.outq = max(vis), outq.data_ptr()
    scratch = _empty(max(1, H.lib().axon_hip_attention_scratch_floats(C.byref(a), C.c_size_t(n))))
    a.scratch = scratch.data_ptr()
    s = _Calls({"out": out, "blocks": outq}, (q, kv, k_off, v_off, n_vis, scratch))
    s.add("attention_rows", a, n)
    return s


def _prepare_head(case, seed):
    (w, _), x = _head_inputs(case, seed)
    n, v, d = case["rows"], case["n_vocab"], case["n_embd"]
    lib = H.lib()
    lib.axon_hip_q6k_planar_bytes.restype = C.c_size_t
    lib.axon_hip_argmax_scratch_words.restype = C.c_size_t
    planar = _empty(lib.axon_hip_q6k_planar_bytes(C.c_size_t(v), C.c_size_t(d)), dtype=torch.uint8)
    torch.cuda.synchronize()
    H.call("q6k_repack", _p(w), v, d, _p(planar))  # once, as at a model's upload
    H.synchronize()
    y, ids = _empty(n, v), _empty(n, dtype=torch.int32)
    keys = _empty(lib.axon_hip_argmax_scratch_words(C.c_size_t(n)), dtype=torch.int64)
    s = _Calls({"logits": y, "ids": ids}, (planar, x, keys))
    s.add("matmul_q6_k_planar", _p(planar), _p(x), _p(y), n, v, d, v)
    s.add("argmax_rows", _p(y), v, n, v, _p(keys), _p(ids))
    return s


def _prepare_sample(case, seed):
    x = _sample_inputs(case, seed)
    n, v, k = case["rows"], case["n_vocab"], case["k"]
    logit, ids = _empty(n, k), _empty(n, k, dtype=torch.int32)
    s = _Calls({"logit": logit, "id": ids}, (x,))
    s.add("topk_rows", _p(x), v, n, v, k, _p(logit), _p(ids))
    return s


_models = {}


def _model() -> H.Model:
    """The served model: one handle per process, its weights read once from the GGUF file that
    synth.py writes (about 45 s the first time on a machine)."""
    if "m" not in _models:
        _models["m"] = H.Model(synth.cached_model(SPEC), max_seq=CHUNK, max_ctx=MAX_CTX, max_batch=32, max_caches=208)
    return _models["m"]


class _Sequences:
    """Sequences in progress: their caches hold prompts, prefilled through the model."""

    def __init__(self, case, lengths, seed):
        self.case, self.lengths, self.model = case, lengths, _model()
        r = np.random.default_rng(seed)
        self.prompts = [r.integers(0, SPEC.n_vocab, n + 1).astype(np.int32) for n in lengths]
        self.caches = [self.model.new_cache() for _ in lengths]
        self.next = np.array([p[-1] for p in self.prompts], np.int32)

    def __del__(self):
        for c in self.caches:
            self.model.free_cache(c)

    def prefill(self):
        logits = None
        for c, p, n in zip(self.caches, self.prompts, self.lengths):
            for at in range(0, n, CHUNK):
                last = at + CHUNK >= n
                logits = self.model.forward_mixed(c, p[at:min(n, at + CHUNK)], [], [], logits=last)
        return logits

    def run(self):
        case, m = self.case, self.model
        if case["kind"] == "prefill":
            m.truncate(self.caches[0], 0)
            return self.prefill()
        for c, n in zip(self.caches, self.lengths):
            m.truncate(c, n)
        if case["kind"] == "decode":
            ids = m.generate_greedy(self.caches[0], int(self.next[0]), case["steps"] - 1)
            return {"ids": ids, "logits": m.forward_prefill(self.caches[0], ids[-1:])}
        tokens, ids = self.next, []
        for _ in range(case["steps"] - 1):
            m.forward_batch(self.caches, tokens, logits=False)
            tokens = m.greedy(len(tokens))
            ids.append(tokens)
        return {"ids": ids, "logits": m.forward_batch(self.caches, tokens)}


def _prepare_model(case, seed):
    if case["kind"] == "prefill":
        return _Sequences(case, [case["tokens"]], seed)
    if case["kind"] == "decode":
        s = _Sequences(case, [case["ctx"]], seed)
    else:
        r = random.Random(seed)
        s = _Sequences(case, [r.randint(case["lo"], case["hi"]) for _ in range(case["rows"])], seed)
    s.prefill()
    return s


def prepare(case, seed):
    H.init(0)
    kind = case["kind"]
    if kind in ("decode", "batch", "prefill"):
        return _prepare_model(case, seed)
    return {"mlp": _prepare_mlp, "proj": _prepare_proj, "attn": _prepare_attn, "head": _prepare_head,
            "sample": _prepare_sample}[kind](case, seed)


def run(state):
    return state.run()


# ---------------------------------------------------------------------------------------------
# What a pass cannot do without, and how exactly it is known

def _layer_bytes(rows_kv: int) -> int:
    """One pass over the model's layers with rows_kv cached positions read."""
    d, ff, kv = SPEC.n_embd, SPEC.n_ff, SPEC.n_head_kv * HEAD_DIM
    return int(SPEC.n_layer * ((2 * d * d + 2 * d * kv + 3 * d * ff) * BITS["q4_0"] / 8 + rows_kv * 2 * kv * 4))


def _layer_flops(rows: int, positions: int) -> int:
    """rows through every layer's matrices, positions (row, position) pairs through its attention."""
    d, ff, kv = SPEC.n_embd, SPEC.n_ff, SPEC.n_head_kv * HEAD_DIM
    return SPEC.n_layer * (2 * rows * (2 * d * d + 2 * d * kv + 3 * d * ff) + 4 * positions * d)


_HEAD_BYTES = int(SPEC.n_vocab * SPEC.n_embd * BITS["q6_k"] / 8)
_HEAD_FLOPS = 2 * SPEC.n_vocab * SPEC.n_embd


def work(case):
    kind = case["kind"]
    if kind == "mlp":
        n, d, ff = case["rows"], case["n_embd"], case["n_ff"]
        return {"bytes": 3 * d * ff * BITS[case["type"]] / 8 + n * (3 * d * 4 + ff // 32 * 34), "flops": 6 * n * d * ff}
    if kind == "proj":
        n, o, i = case["rows"], case["n_out"], case["n_in"]
        x = i // 32 * 34 if case["type"] in ("q4_0", "q4_1", "q8_0") else 4 * i
        return {"bytes": o * i * BITS[case["type"]] / 8 + n * (x + 4 * o), "flops": 2 * n * o * i}
    if kind == "attn":
        n, d, kv = case["rows"], case["n_head"] * HEAD_DIM, case["n_kv"] * HEAD_DIM
        if case["past"] >= 0:
            read, pairs = case["past"] + n, sum(case["past"] + i + 1 for i in range(n))
        else:
            read = pairs = n * (case["lo"] + case["hi"]) // 2
        return {"bytes": 2 * read * kv * (2 if case["f16"] else 4) + n * d * 9, "flops": 4 * pairs * d}
    if kind == "head":
        n, v, d = case["rows"], case["n_vocab"], case["n_embd"]
        return {"bytes": v * d * BITS["q6_k"] / 8 + n * 4 * (d + v), "flops": 2 * n * v * d}
    if kind == "sample":
        return {"bytes": case["rows"] * (case["n_vocab"] * 4 + 8 * case["k"]), "flops": 0}
    if kind == "decode":
        n, ctx = case["steps"], case["ctx"]
        pos = n * ctx + n * (n + 1) // 2
        return {"bytes": n * (_layer_bytes(0) + _HEAD_BYTES) + _layer_bytes(pos) - _layer_bytes(0),
                "flops": _layer_flops(n, pos) + n * _HEAD_FLOPS}
    if kind == "batch":
        n, r = case["steps"], case["rows"]
        pos = n * r * ((case["lo"] + case["hi"]) // 2)
        return {"bytes": n * (_layer_bytes(0) + _HEAD_BYTES) + _layer_bytes(pos) - _layer_bytes(0),
                "flops": _layer_flops(n * r, pos) + n * r * _HEAD_FLOPS}
    n = case["tokens"]
    chunks = -(-n // CHUNK)
    return {"bytes": chunks * _layer_bytes(0) + _layer_bytes(n) - _layer_bytes(0) + _HEAD_BYTES,
            "flops": _layer_flops(n, n * (n + 1) // 2) + _HEAD_FLOPS}


def tolerance(case):
    """Single blocks: sums of 32-bit floats in another order. The blocks that a kernel quantizes, the
    ids and the candidates are whole values and stay the same. Whole calls: a rounding in one layer
    can move a value of the next Q8_0 quantization by one step (1/127 of its block's largest)."""
    kind = case["kind"]
    if kind in ("decode", "batch", "prefill"):
        return {"rel": 1e-2, "max": 0.1}
    if kind == "sample":
        return "exact"
    return {"rel": 1e-5}


# ---------------------------------------------------------------------------------------------
# The same outputs in 64 bits, in plain torch

def _quantized(x: torch.Tensor) -> torch.Tensor:
    """The values of x's Q8_0 blocks, quantized from 64 bits."""
    b = x.reshape(-1, 32)
    d = b.abs().amax(1) / 127
    q = _round_away(b * _inverse(d)[:, None])
    return (d.half().double()[:, None] * q).reshape(x.shape)


def _exact_attn(case, seed):
    q, kv = _attn_inputs(case, seed)
    vis, seqs = _attn_lengths(case, seed)
    n, n_head, n_kv = case["rows"], case["n_head"], case["n_kv"]
    group = n_head // n_kv
    scale = float(np.float32(HEAD_DIM ** -0.5))
    out, at = torch.empty((n, n_head, HEAD_DIM), dtype=torch.float64, device="cuda"), 0
    for i, m in enumerate(seqs):
        k = kv[at:at + m].double().reshape(m, n_kv, HEAD_DIM)
        v = kv[at + m:at + 2 * m].double().reshape(m, n_kv, HEAD_DIM)
        at += 2 * m
        rows = range(n) if case["past"] >= 0 else range(i, i + 1)
        qs = q[rows.start:rows.stop].double().reshape(len(rows), n_head, HEAD_DIM)
        seen = torch.arange(m, device="cuda")[None, :] < torch.tensor([vis[r] for r in rows], device="cuda")[:, None]
        for h in range(n_head):
            s = torch.mm(qs[:, h], k[:, h // group].t().contiguous()) * scale
            p = torch.softmax(s.masked_fill(~seen, -math.inf), 1)
            out[rows.start:rows.stop, h] = torch.mm(p, v[:, h // group].contiguous())
    return {"out": out.reshape(n, -1), "blocks": None}


def exact(case, seed):
    kind = case["kind"]
    if kind == "mlp":
        x, norm, (_, wg), (_, wu), (_, wd) = _mlp_inputs(case, seed, True)
        xd = x.double()
        h = xd * torch.rsqrt(xd.square().mean(1, keepdim=True) + float(np.float32(EPS))) * norm.double()
        hq = _quantized(h)
        a = torch.nn.functional.silu(hq @ wg.t().contiguous()) * (hq @ wu.t().contiguous())
        return {"act": None, "y": xd + _quantized(a) @ wd.t().contiguous()}
    if kind == "proj":
        (_, w), x = _proj_inputs(case, seed, True)
        xd = _blocks(x, "q8_0", True)[1] if case["type"] in ("q4_0", "q4_1", "q8_0") else x.double()
        return xd @ w.t().contiguous()
    if kind == "attn":
        return _exact_attn(case, seed)
    if kind == "head":
        (_, w), x = _head_inputs(case, seed, True)
        y = x.double() @ w.t().contiguous()
        return {"logits": y, "ids": y.argmax(1)}
    if kind == "sample":
        v, i = torch.sort(_sample_inputs(case, seed).double(), dim=1, descending=True, stable=True)
        return {"logit": v[:, :case["k"]].contiguous(), "id": i[:, :case["k"]].contiguous()}
    # A whole model's values in 64 bits would take other roundings at every activation quantization:
    # no value of its logits is closer than the tolerance.
    return None
