"""Performance cases: the work a program has this library do, through its public entry points, with float64 answers to
compare against.

Kinds of case:
- "matvec"   zl_mat_gemv_noalloc: one quantised matrix times 1..16 rows of activations, on the caller's stream;
- "decode"   HipModel.forward: one token at position `prefix` of a model with that many cached positions;
- "verify"   HipModel.forward_batch(..., logits="all"): the k + 1 rows of a speculative verification pass;
- "prompt"   prefill_tokens: `tokens` prompt tokens after `prefix` cached ones, in chunks of max_batch, last logits;
- "speculate" generate_speculative: a whole call after a cached prompt, with the sampler on the device.
The model kinds build a few layers of the shapes in zerollm_amd.synth (random weights made from the seed), so that each
layer's work and its rounding can be told apart; the output head of those has the 2048 ids of the tiny test models.
"""
import ctypes as C
import math

import numpy as np
import torch

from zerollm_amd import _lib, gguf, synth
from zerollm_amd import model as M
from zerollm_amd.generate import prefill_tokens
from zerollm_amd.sampler import HipSampler
from zerollm_amd.speculative import generate_speculative

DEV = "cuda"
TYPES = {"q8_0": gguf.Q8_0, "q4_0": gguf.Q4_0, "q5_0": gguf.Q5_0, "q4_k": gguf.Q4_K, "q5_k": gguf.Q5_K, "q6_k": gguf.Q6_K,
         "f16": gguf.F16}
VOCAB = 2048      # ids of the layer cases' heads
PROMPT = 512      # cached prompt of the whole calls (the benchmark's)

# the shapes of zerollm_amd.synth: arguments of build_spec (llama: the adjacent-pair rotation, no head norms)
DENSE = {
    "qwen3-8b": dict(arch="qwen3", n_embd=4096, n_head=32, n_head_kv=8, head_dim=128, n_ff=12288, types=synth.Q4_K_M),
    "qwen3-0.6b": dict(arch="qwen3", n_embd=1024, n_head=16, n_head_kv=8, head_dim=128, n_ff=3072,
                       types=synth.all_type(gguf.Q8_0)),
    "tiny": dict(arch="qwen3", n_embd=512, n_head=8, n_head_kv=4, head_dim=64, n_ff=1536, types=synth.all_type(gguf.Q8_0)),
    "tiny-llama": dict(arch="llama", n_embd=512, n_head=8, n_head_kv=4, head_dim=64, n_ff=1536, types=synth.Q4_K_M),
}


def listed():
    return [
        # the smallest matrix of the 0.6B draft (attn_k, attn_v) for the two tokens it is fed after a fully accepted
        # cycle: launch latency
        {"name": "matvec_q8_1024_m2", "kind": "matvec", "type": "q8_0", "rows": 1024, "cols": 1024, "tokens": 2},
        # attn_q / attn_output of the 8B target at the verify width of k = 4
        {"name": "matvec_q4k_4096_m5", "kind": "matvec", "type": "q4_k", "rows": 4096, "cols": 4096, "tokens": 5},
        # the hybrid's attn_qkv for a full default batch of prompt tokens
        {"name": "matvec_q5k_8192_m16", "kind": "matvec", "type": "q5_k", "rows": 8192, "cols": 2560, "tokens": 16},
        # the 8B target's output head for one token of plain decoding: the largest matrix
        {"name": "matvec_q6k_head_m1", "kind": "matvec", "type": "q6_k", "rows": 151936, "cols": 4096, "tokens": 1},
        # plain decoding / drafting at an ordinary length, default (f32) KV cache
        {"name": "decode_0.6b", "kind": "decode", "shape": "qwen3-0.6b", "layers": 8, "prefix": 700, "tokens": 1,
         "ctx": 1024, "max_batch": 64, "kv": "f32"},
        # the target's verification pass of k = 4 at an ordinary length
        {"name": "verify_8b", "kind": "verify", "shape": "qwen3-8b", "layers": 2, "prefix": 601, "tokens": 5,
         "ctx": 1024, "max_batch": 64, "kv": "f16"},
        # a prompt of an ordinary, odd length from nothing, in 64-token chunks
        {"name": "prompt_8b", "kind": "prompt", "shape": "qwen3-8b", "layers": 2, "prefix": 0, "tokens": 509,
         "ctx": 1024, "max_batch": 64, "kv": "f16"},
        # drafting deep into a long conversation, the cache as large as the models' trained context
        {"name": "decode_0.6b_16k", "kind": "decode", "shape": "qwen3-0.6b", "layers": 4, "prefix": 16384, "tokens": 1,
         "ctx": 32768, "max_batch": 64, "kv": "f16"},
        # verifying k = 8 drafts there, the cache sized for the call (the benchmark's long workload)
        {"name": "verify_8b_16k", "kind": "verify", "shape": "qwen3-8b", "layers": 2, "prefix": 16384, "tokens": 9,
         "ctx": 16658, "max_batch": 64, "kv": "f16"},
        # the next turn of a long conversation: a few chunks of new prompt over a long cached prefix
        {"name": "prompt_8b_12k", "kind": "prompt", "shape": "qwen3-8b", "layers": 2, "prefix": 12000, "tokens": 256,
         "ctx": 16384, "max_batch": 64, "kv": "f16"},
        # the hybrid target's cycle: rollback mark, verification pass, rollback (three DeltaNet layers, one attention)
        {"name": "verify_hybrid", "kind": "verify", "shape": "qwen35-4b", "layers": 4, "prefix": 2048, "tokens": 5,
         "ctx": 4096, "max_batch": 64, "kv": "f16"},
        # a whole call: the full pair, sampled, drafts accepted and rejected
        {"name": "speculate_8b", "kind": "speculate", "target_layers": 36, "draft_layers": 28, "k": 4, "tokens": 24,
         "temperature": 0.7},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    r = rng.random()
    if r < 0.45:
        t = rng.choice(["q8_0", "q4_k", "q4_k", "q6_k", "q6_k", "q5_k", "q4_0", "q5_0", "f16"])
        step = 256 if t in ("q4_k", "q5_k", "q6_k") else 32
        # (rows and columns of one matrix whose split sums the entry point's fixed work space holds)
        band = rng.random()
        if band < 0.6:
            rows, cols = _log(rng, 64, 4096), _log(rng, 256, 12288)
        elif band < 0.85:
            rows, cols = _log(rng, 4097, 16384), _log(rng, 256, 2048)
        else:
            rows, cols = _log(rng, 16448, 151936), _log(rng, 512, 4096)
        cols = max(step, cols // step * step)
        return {"kind": "matvec", "type": t, "rows": rows, "cols": cols, "tokens": rng.choice([1, 1, 2, 3, 4, 5, 5, 7, 9, 11, 16])}
    kv = rng.choice(["f16", "f16", "f32"])
    mb = rng.choice([16, 64, 64])
    if r < 0.53:
        n, p = rng.randint(2, 9), _log(rng, 64, 3000)
        return {"kind": "verify", "shape": "qwen35-4b", "layers": 4, "prefix": p, "tokens": n, "ctx": _ctx(rng, p + n),
                "max_batch": mb, "kv": kv}
    if r < 0.58:
        return {"kind": "speculate", "target_layers": rng.randint(2, 8), "draft_layers": rng.randint(1, 6), "k": rng.randint(1, 8),
                "tokens": rng.randint(9, 40), "temperature": rng.choice([0.0, 0.7, 1.0])}
    shape = rng.choice(["qwen3-8b", "qwen3-8b", "qwen3-0.6b", "qwen3-0.6b", "tiny", "tiny-llama"])
    layers = rng.randint(1, 2 if shape == "qwen3-8b" else 4)
    kind = rng.choice(["decode", "verify", "prompt"])
    p = _log(rng, 16, 16384)
    n = 1 if kind == "decode" else rng.randint(2, 9) if kind == "verify" else _log(rng, 10, 300)
    return {"kind": kind, "shape": shape, "layers": layers, "prefix": p, "tokens": n, "ctx": _ctx(rng, p + n), "max_batch": mb, "kv": kv}


def _ctx(rng, n):
    """A cache sized for the call, or the next power of two."""
    return n + 16 + rng.randint(0, 200) if rng.random() < 0.5 else max(1024, 1 << (n + 15).bit_length())


# ---------------------------------------------------------------------------------------------- inputs
def _spec(case, seed):
    if case["shape"] == "qwen35-4b":
        return synth.build_qwen35_spec(2560, case["layers"], 16, 4, 256, 64, 9216, VOCAB, 262144, synth.QWEN35_Q4_K_M, seed,
                                       layer_type=synth._qwen35_4b_layer_type)
    return synth.build_spec(n_layer=case["layers"], vocab=VOCAB, ctx_train=32768, seed=seed, **DENSE[case["shape"]])


def _ids(case, seed):
    ids = synth.seeded_ids(case["prefix"] + case["tokens"], 1000 + seed, VOCAB)
    return ids[:case["prefix"]], ids[case["prefix"]:]


def _bytes_of(t):
    return t.view(torch.uint8)


def _raw(case, seed):
    """The matrix as a file holds it: [rows, blocks, bytes] uint8 on the GPU, values of about N(0, 0.02)."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    t, rows, cols = case["type"], case["rows"], case["cols"]

    def normal(shape, mean, std, lo, hi):
        return torch.empty(shape, device=DEV).normal_(mean, std, generator=g).round_().clamp_(lo, hi).to(torch.int16)

    def half(shape, scale):
        return (scale * (0.8 + 0.4 * torch.rand(shape, device=DEV, generator=g))).half()

    if t == "f16":
        return _bytes_of(torch.empty((rows, 1, cols), device=DEV).normal_(0, 0.02, generator=g).half())
    if t in ("q8_0", "q4_0", "q5_0"):
        nb = cols // 32
        d = _bytes_of(half((rows, nb, 1), 0.02 / {"q8_0": 42.0, "q4_0": 2.7, "q5_0": 5.3}[t]))
        if t == "q8_0":
            return torch.cat([d, _bytes_of(normal((rows, nb, 32), 0, 42, -127, 127).to(torch.int8))], 2)
        if t == "q4_0":
            v = normal((rows, nb, 32), 8, 2.7, 0, 15)
            return torch.cat([d, (v[..., :16] | (v[..., 16:] << 4)).to(torch.uint8)], 2)
        v = normal((rows, nb, 32), 16, 5.3, 0, 31)
        h = (v >> 4).reshape(rows, nb, 4, 8)
        hb = (h << torch.arange(8, device=DEV, dtype=torch.int16)).sum(-1).to(torch.uint8)
        return torch.cat([d, hb, ((v[..., :16] & 15) | ((v[..., 16:] & 15) << 4)).to(torch.uint8)], 2)
    nb = cols // 256
    if t == "q6_k":
        v = normal((rows, nb, 2, 4, 32), 32, 10, 0, 63)  # [half][quarter][value]
        ql = torch.cat([(v[..., 0, :] & 15) | ((v[..., 2, :] & 15) << 4), (v[..., 1, :] & 15) | ((v[..., 3, :] & 15) << 4)], -1)
        qh = (v[..., 0, :] >> 4) | ((v[..., 1, :] >> 4) << 2) | ((v[..., 2, :] >> 4) << 4) | ((v[..., 3, :] >> 4) << 6)
        sc = normal((rows, nb, 16), 0, 60, -128, 127).to(torch.int8)
        return torch.cat([ql.reshape(rows, nb, 128).to(torch.uint8), qh.reshape(rows, nb, 64).to(torch.uint8), _bytes_of(sc),
                          _bytes_of(half((rows, nb, 1), 0.02 / 600))], 2)
    five = t == "q5_k"
    top = 31 if five else 15
    v = normal((rows, nb, 8, 32), top / 2, top / 5.5, 0, top)
    sc, mn = normal((rows, nb, 8), 40, 10, 1, 63), normal((rows, nb, 8), 40, 10, 1, 63)
    s = torch.cat([(sc[..., :4]) | ((sc[..., 4:] >> 4) << 6), mn[..., :4] | ((mn[..., 4:] >> 4) << 6),
                   (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)], -1).to(torch.uint8)
    step = 0.02 * 5.5 / top / 40
    parts = [_bytes_of(half((rows, nb, 1), step)), _bytes_of(half((rows, nb, 1), step * top / 2)), s]
    if five:
        parts.append((((v >> 4) & 1) << torch.arange(8, device=DEV, dtype=torch.int16)[:, None]).sum(2).to(torch.uint8))
    q = v & 15
    parts.append((q[..., 0::2, :] | (q[..., 1::2, :] << 4)).reshape(rows, nb, 128).to(torch.uint8))
    return torch.cat(parts, 2)


def _rows(case, seed):
    """Normed activations: N(0, 1) with a few large channels, as the inputs of projections have."""
    g = torch.Generator(device=DEV).manual_seed(seed + 7919)
    x = torch.empty((case["tokens"], case["cols"]), device=DEV).normal_(0, 1, generator=g)
    return x * torch.empty((1, case["cols"]), device=DEV).normal_(0, 0.7, generator=g).exp()


_streams = []


def _stream():
    """One stream for every call of the entry point (its calls share a work space, so they must not overlap)."""
    if not _streams:
        _streams.append(torch.cuda.Stream())
    return _streams[0]


class _State:
    """What a program keeps: handles that are released with it."""

    def __init__(self, **kw):
        self.mat, self.models, self.sampler = None, [], None
        self.__dict__.update(kw)

    def __del__(self):
        for m in self.models:
            m.close()
        if self.sampler is not None:
            self.sampler.close()
        if self.mat is not None:
            _lib.call("zl_mat_free", self.mat)


def prepare(case, seed):
    M.init(0)
    if case["kind"] == "matvec":
        raw = _raw(case, seed).cpu().numpy()
        h = C.c_void_p()
        _lib.call("zl_mat_upload", TYPES[case["type"]], raw.ctypes.data_as(C.c_void_p), case["rows"], case["cols"], C.byref(h))
        s = _State(case=case, mat=h, x=_rows(case, seed), y=torch.empty((case["tokens"], case["rows"]), device=DEV))
        s.stream = C.c_void_p(_stream().cuda_stream)
        s.xp, s.yp = C.c_void_p(s.x.data_ptr()), C.c_void_p(s.y.data_ptr())
        torch.cuda.synchronize()
        return s
    if case["kind"] == "speculate":
        t, d = _pair(case, seed)
        ctx = PROMPT + case["tokens"] + 2 * (case["k"] + 1)
        models = [synth.build_on_device(x, ctx=ctx, kv="f16", max_batch=64) for x in (t, d)]
        prompt = synth.seeded_ids(PROMPT, 2024 + seed, t.vocab)
        for m in models:
            prefill_tokens(m, prompt[:-1], want_logits=False)
        smp = HipSampler(temperature=case["temperature"], top_k=40, top_p=0.9, seed=1234, argmax=case["temperature"] == 0)
        row = np.empty(t.vocab, np.float32)
        return _State(case=case, models=models, sampler=smp, prompt=prompt, row=row)
    spec = _spec(case, seed)
    prefix, new = _ids(case, seed)
    m = synth.build_on_device(spec, ctx=case["ctx"], kv=case["kv"], max_batch=case["max_batch"])
    prefill_tokens(m, prefix, want_logits=False)
    return _State(case=case, models=[m], ids=prefix + new, new=new, prefix=len(prefix))


def run(state):
    case = state.case
    if case["kind"] == "matvec":
        _lib.call("zl_mat_gemv_noalloc", state.mat, state.xp, case["tokens"], state.yp, state.stream)
        return state.y
    if case["kind"] == "speculate":
        t, d = state.models
        state.sampler.rng_state = 1234
        out = list(generate_speculative(t, d, state.prompt, k=case["k"], max_tokens=case["tokens"], sample=state.sampler))
        _lib.call("zl_model_logits", t._h, 0, 1, _lib.ptr(state.row, C.c_float))
        return {"tokens": np.array(out, np.int64), "logits": state.row}
    m = state.models[0]
    if case["shape"] == "qwen35-4b":
        # the cycle a speculative loop runs on a hybrid target; nothing accepted, so the state can be run again
        m.mark_rollback()
        rows = m.forward_batch(state.new, logits="all")
        m.truncate(state.prefix)
        return rows
    m.truncate(state.prefix)
    if case["kind"] == "decode":
        return m.forward(state.new[0])
    if case["kind"] == "verify":
        return m.forward_batch(state.new, logits="all")
    return prefill_tokens(m, state.ids, start=state.prefix)[0]


def _pair(case, seed):
    """The benchmark's agreeing pair (zerollm_amd.synth.qwen3_8b_close_pair) with so many layers, of this seed."""
    t, d = synth.qwen3_8b_close_pair(seed=seed, draft_seed=seed + 1)
    for s, n in ((t, case["target_layers"]), (d, case["draft_layers"])):
        s.n_layer = n
        s.tensors = [x for x in s.tensors if not x.name.startswith("blk.") or int(x.name.split(".")[1]) < n]
    return t, d


# ---------------------------------------------------------------------------------------------- what a pass needs
def work(case):
    if case["kind"] == "matvec":
        r, c, n = case["rows"], case["cols"], case["tokens"]
        return {"bytes": r * gguf.row_size(TYPES[case["type"]], c) + 4 * n * (r + c), "flops": 2 * r * c * n}
    if case["kind"] == "speculate":
        # at least tokens / (k + 1) cycles, each k draft passes and one target pass
        t, d = _pair(case, 1)
        cyc = math.ceil(case["tokens"] / (case["k"] + 1))
        kv = sum(4 * s.n_layer * s.n_head_kv * s.head_dim * PROMPT * w for s, w in ((t, 1), (d, case["k"])))
        wt, wd = (sum(x.rows * x.cols for x in s.tensors if x.rows > 1 and x.name != "token_embd.weight") for s in (t, d))
        return {"bytes": cyc * (t.weight_bytes + case["k"] * d.weight_bytes + kv), "flops": 2 * cyc * ((case["k"] + 1) * wt + case["k"] * wd)}
    s = _spec(case, 1)
    n, p = case["tokens"], case["prefix"]
    kvb = 4 if case["kv"] == "f32" else 2
    n_att = s.n_layer if not s.hybrid else sum((l + 1) % s.interval == 0 for l in range(s.n_layer))
    head = s.weight_bytes - sum(x.nbytes for x in s.tensors if x.rows > 1 and x.name.startswith("blk."))
    rows = 1 if case["kind"] == "prompt" else n
    weights = sum(x.rows * x.cols for x in s.tensors if x.name.startswith("blk.") and x.rows > 1 and x.type != gguf.F32)
    nbytes = sum(x.nbytes for x in s.tensors if x.rows > 1 and x.name.startswith("blk.")) + head + 4 * rows * s.vocab
    nbytes += 2 * n_att * s.n_head_kv * s.head_dim * (p + 2 * n) * kvb
    flops = 2 * n * weights + 2 * rows * s.vocab * s.n_embd + 4 * n_att * s.n_head * s.head_dim * n * (p + n // 2)
    if s.hybrid:  # the recurrent state read, written and captured after every token; its rank-1 updates
        rec = (s.n_layer - n_att) * s.dt_rank * s.d_state * s.d_state
        nbytes += 4 * rec * (2 + n)
        flops += 8 * rec * n
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["kind"] == "matvec":
        # float64 sums rounded once to float32: 2.5e-8 from the exact products, half an ulp
        return {"rel": 1e-7, "max": 4e-6}
    # One float32 rounding that moves one int8 code in a layer moves codes in every product after it, until all of the
    # products' quantisation noise (0.7 % each) is another draw: attention sums in another order (float64 chunks for the
    # float32 chain) change the logits of 1..4 layers by 0.4..1.5 %, largest single logit 8 % of their r.m.s., and both
    # are 0.4..1.8 % from the float64 pass. Two layers of the largest shape at most, so that this bound says something.
    tol = {"rel": 0.03, "max": 0.3}
    # (a call's tokens are drawn by seeded uniforms from distributions whose logits move this much)
    return dict(tol, differ=0.01) if case["kind"] == "speculate" else tol


# ---------------------------------------------------------------------------------------------- float64 answers
def _dequant(ty, raw, rows, cols):
    """The matrix's values as float64 [rows, cols] from its blocks (uint8, on the GPU)."""
    def f16(b):
        return b.contiguous().view(torch.float16).double()

    if ty == gguf.F32:
        return raw.view(torch.float32).reshape(rows, cols).double()
    if ty == gguf.F16:
        return f16(raw.reshape(rows, cols * 2))
    size = gguf.row_size(ty, 256) if ty in (gguf.Q4_K, gguf.Q5_K, gguf.Q6_K) else gguf.row_size(ty, 32)
    o = raw.reshape(rows, -1, size)
    nb = o.shape[1]
    if ty == gguf.Q8_0:
        return (f16(o[..., :2]) * o[..., 2:].contiguous().view(torch.int8).double()).reshape(rows, cols)
    if ty == gguf.Q4_0:
        q = o[..., 2:]
        return (f16(o[..., :2]) * (torch.cat([q & 15, q >> 4], -1).double() - 8)).reshape(rows, cols)
    bits = torch.arange(8, device=raw.device, dtype=torch.uint8)
    if ty == gguf.Q5_0:
        h = ((o[..., 2:6, None] >> bits) & 1).reshape(rows, nb, 32)
        q = o[..., 6:]
        return (f16(o[..., :2]) * ((torch.cat([q & 15, q >> 4], -1) | (h << 4)).double() - 16)).reshape(rows, cols)
    if ty == gguf.Q6_K:
        ql, qh, sc = o[..., :128].reshape(rows, nb, 2, 64), o[..., 128:192].reshape(rows, nb, 2, 32), o[..., 192:208]
        lo = torch.stack([ql[..., :32] & 15, ql[..., 32:] & 15, ql[..., :32] >> 4, ql[..., 32:] >> 4], 3)
        hi = torch.stack([(qh >> (2 * i)) & 3 for i in range(4)], 3)
        q = ((lo | (hi << 4)).double() - 32).reshape(rows, nb, 16, 16)
        return (q * sc.contiguous().view(torch.int8).double()[..., None] * f16(o[..., 208:210])[..., None]).reshape(rows, cols)
    s = o[..., 4:16]
    sc = torch.cat([s[..., :4] & 63, (s[..., 8:] & 15) | ((s[..., :4] >> 6) << 4)], -1).double()
    mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1).double()
    q = o[..., -128:].reshape(rows, nb, 4, 32)
    q = torch.stack([q & 15, q >> 4], 3).reshape(rows, nb, 8, 32)
    if ty == gguf.Q5_K:
        q = q | (((o[..., 16:48][..., None, :] >> bits[:, None]) & 1) << 4)
    w = q.double() * (f16(o[..., :2]) * sc)[..., None] - (f16(o[..., 2:4]) * mn)[..., None]
    return w.reshape(rows, cols)


def _quantised(x):
    """Activations as the products see them: 32-value blocks of int8 codes and a float32 scale."""
    b = x.double().reshape(x.shape[0], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127
    v = b * torch.where(d > 0, 1 / d, torch.zeros_like(d))
    q = torch.where(v < 0, -torch.floor(-v + 0.5), torch.floor(v + 0.5))
    return (q * d.float().double()).reshape(x.shape)


def _f32(x):
    return x.float().double()


class _Exact:
    """The pass in float64. Values are rounded where a layer stores them: float32 activations, the cache's type, int8
    codes and the float32 recurrent state."""

    def __init__(self, case, seed):
        self.case, self.s = case, _spec(case, seed)
        self.t = {t.name: t for t in self.s.tensors}

    def w(self, name):
        t = self.t[name]
        raw = torch.from_numpy(synth.tensor_bytes(t, use_device=True)).to(DEV)
        return _dequant(t.type, raw, t.rows, t.cols)

    def mv(self, name, x):
        return _f32((x if self.t[name].type == gguf.F32 else _quantised(x)) @ self.w(name).T)

    def norm(self, x, w):
        return _f32(x / torch.sqrt((x * x).mean(-1, keepdim=True) + self.s.rms_eps) * w)

    def rope(self, v, pos):
        n = self.s.n_rot or self.s.head_dim
        half = n // 2
        f = float(self.s.rope_base) ** (-2.0 * torch.arange(half, device=DEV, dtype=torch.float64) / n)
        a = pos.double()[:, None, None] * f
        c, s = _f32(torch.cos(a)), _f32(torch.sin(a))
        out = v.clone()
        i0, i1 = (slice(0, n, 2), slice(1, n, 2)) if self.s.arch == "llama" else (slice(0, half), slice(half, n))
        out[..., i0] = v[..., i0] * c - v[..., i1] * s
        out[..., i1] = v[..., i0] * s + v[..., i1] * c
        return _f32(out)

    def attention(self, p, h, first):
        """Rows `first`.. of the layer's attention output (every row's keys and values are formed)."""
        s = self.s
        T, G, D = h.shape[0], s.n_head // s.n_head_kv, s.head_dim
        q = self.mv(p + "attn_q.weight", h[first:]).reshape(T - first, s.n_head, -1)
        q, gate = q[..., :D], q[..., D:]
        k = self.mv(p + "attn_k.weight", h).reshape(T, s.n_head_kv, D)
        v = self.mv(p + "attn_v.weight", h).reshape(T, s.n_head_kv, D)
        if s.arch != "llama":
            q, k = self.norm(q, self.w(p + "attn_q_norm.weight")[0]), self.norm(k, self.w(p + "attn_k_norm.weight")[0])
        pos = torch.arange(T, device=DEV)
        q, k = self.rope(q, pos[first:]), self.rope(k, pos)
        if self.case["kv"] == "f16":
            k, v = k.half().double(), v.half().double()
        out = torch.empty(T - first, s.n_head, D, device=DEV, dtype=torch.float64)
        for a in range(first, T, 512):
            b = min(T, a + 512)
            for kh in range(s.n_head_kv):
                qq = q[a - first:b - first, kh * G:(kh + 1) * G].transpose(0, 1).reshape(-1, D)
                sc = ((qq @ k[:b, kh].T) / math.sqrt(D)).reshape(G, b - a, b)
                sc.masked_fill_(pos[:b] > pos[a:b, None], -math.inf)
                o = (torch.softmax(sc, -1).reshape(-1, b) @ v[:b, kh]).reshape(G, b - a, D)
                out[a - first:b - first, kh * G:(kh + 1) * G] = o.transpose(0, 1)
        out = _f32(out)
        if gate.shape[-1]:
            out = _f32(out * torch.sigmoid(gate))
        return self.mv(p + "attn_output.weight", out.reshape(T - first, -1))

    def delta(self, p, h):
        s = self.s
        T, D, nk, nv = h.shape[0], s.d_state, s.n_group, s.dt_rank
        u = self.mv(p + "attn_qkv.weight", h)
        z = self.mv(p + "attn_gate.weight", h).reshape(T, nv, D)
        beta = torch.sigmoid(self.mv(p + "ssm_beta.weight", h))
        al = self.mv(p + "ssm_alpha.weight", h) + self.w(p + "ssm_dt.bias")[0]
        decay = torch.exp(torch.where(al > 20, al, torch.log1p(torch.exp(al))) * self.w(p + "ssm_a")[0])
        cw = self.w(p + "ssm_conv1d.weight")
        pad = torch.cat([torch.zeros(s.conv_k - 1, u.shape[1], device=DEV, dtype=torch.float64), u])
        acc = sum(cw[:, i] * pad[i:i + T] for i in range(s.conv_k))
        u = _f32(acc * torch.sigmoid(acc))

        def l2(v, scale):
            return _f32(v * (scale / torch.sqrt((v * v).sum(-1, keepdim=True) + s.rms_eps)))

        head = torch.arange(nv, device=DEV) % nk
        q = l2(u[:, :nk * D].reshape(T, nk, D), 1 / math.sqrt(D))[:, head]
        k = l2(u[:, nk * D:2 * nk * D].reshape(T, nk, D), 1.0)[:, head]
        v = u[:, 2 * nk * D:].reshape(T, nv, D)
        S = torch.zeros(nv, D, D, device=DEV, dtype=torch.float64)
        o = torch.empty(T, nv, D, device=DEV, dtype=torch.float64)
        for t in range(T):
            S = S * decay[t][:, None, None]
            d = (v[t] - torch.bmm(S, k[t][:, :, None])[..., 0]) * beta[t][:, None]
            S = S.float().double() + d[:, :, None] * k[t][:, None, :]
            o[t] = torch.bmm(S, q[t][:, :, None])[..., 0]
            S = S.float().double()
        o = _f32(o)
        o = _f32(o / torch.sqrt((o * o).mean(-1, keepdim=True) + s.rms_eps) * self.w(p + "ssm_norm.weight")[0] * (z * torch.sigmoid(z)))
        return self.mv(p + "ssm_out.weight", o.reshape(T, -1))

    def logits(self, ids, rows):
        """Logits of the last `rows` positions of ids."""
        s = self.s
        x = _f32(self.w("token_embd.weight"))[torch.tensor(ids, device=DEV)]
        for l in range(s.n_layer):
            p, last = f"blk.{l}.", l == s.n_layer - 1
            first = len(ids) - rows if last else 0
            h = self.norm(x, self.w(p + "attn_norm.weight")[0])
            if s.hybrid and (l + 1) % s.interval:
                x = _f32(x + self.delta(p, h))[first:]
            else:
                x = _f32(x[first:] + self.attention(p, h, first))
            h = self.norm(x, self.w(p + ("post_attention_norm.weight" if s.hybrid else "ffn_norm.weight"))[0])
            g, u = self.mv(p + "ffn_gate.weight", h), self.mv(p + "ffn_up.weight", h)
            x = _f32(x + self.mv(p + "ffn_down.weight", _f32(g * torch.sigmoid(g) * u)))
        x = self.norm(x, self.w("output_norm.weight")[0])
        return self.mv("output.weight" if "output.weight" in self.t else "token_embd.weight", x)


def exact(case, seed):
    if case["kind"] == "matvec":
        x = _rows(case, seed)
        w = _dequant(TYPES[case["type"]], _raw(case, seed), case["rows"], case["cols"])
        return (x.double() if case["type"] == "f16" else _quantised(x)) @ w.T
    if case["kind"] == "speculate":
        return None  # a pass of all the layers for every token of the prompt and the answer: minutes
    prefix, new = _ids(case, seed)
    out = _Exact(case, seed).logits(prefix + new, 1 if case["kind"] == "prompt" else len(new))
    return out.cpu().numpy() if case["kind"] == "verify" else out[0].cpu().numpy()
