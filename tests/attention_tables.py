"""A one-layer float32 model whose queries, keys and values are written down per token id, and its attention in float64.

Token id j has the embedding e_j; attn_q, attn_k and attn_v hold a table row per id, attn_output copies the heads' outputs
into embedding dimensions of their own, the feed-forward part is zero and the head is the identity, so the logits of a row
are its attention output up to the row's norm: o_i = logits[IDS + i] / logits[id]. Queries and keys live in the last 16
dimensions of a head, which the rotation leaves as they are (frequencies below 1e-22)."""
import numpy as np

from zerollm_amd import gguf, synth
from zerollm_amd import model as M

IDS, LIVE, HEADS = 128, 16, 2


class Tables:
    """q[id][head], k[id] (LIVE values each) and v[id] (head_dim values), one KV head for HEADS query heads."""

    def __init__(self, head_dim, seed):
        rng = np.random.default_rng(seed)
        self.hd = head_dim
        self.q = rng.standard_normal((IDS, HEADS, LIVE)).astype(np.float16).astype(np.float64)
        self.k = rng.standard_normal((IDS, LIVE)).astype(np.float16).astype(np.float64)
        self.v = rng.standard_normal((IDS, head_dim)).astype(np.float16).astype(np.float64)

    def load(self, monkeypatch, path, **kw):
        hd, d = self.hd, IDS + HEADS * self.hd
        spec = synth.build_spec("llama", d, 1, HEADS, 1, hd, 32, d, 1 << 18, synth.all_type(gguf.F32), 1)
        spec.rope_base = 1e30
        x = 1.0 / np.sqrt(1.0 / d + spec.rms_eps)  # the normed embedding's one value
        w = {t.name: np.zeros((t.rows, t.cols), np.float32) for t in spec.tensors}
        for n in ("output_norm", "blk.0.attn_norm", "blk.0.ffn_norm"):
            w[n + ".weight"][:] = 1
        w["token_embd.weight"][:] = np.eye(d)
        w["output.weight"][:] = np.eye(d)
        for h in range(HEADS):
            w["blk.0.attn_q.weight"][(h + 1) * hd - LIVE:(h + 1) * hd, :IDS] = self.q[:, h].T / x
        w["blk.0.attn_k.weight"][hd - LIVE:, :IDS] = self.k.T / x
        w["blk.0.attn_v.weight"][:, :IDS] = self.v.T / x
        w["blk.0.attn_output.weight"][IDS:] = np.eye(HEADS * hd)
        monkeypatch.setattr(synth, "tensor_bytes", lambda t, use_device=False: w[t.name].view(np.uint8).reshape(-1))
        synth.write_gguf(path, spec)
        return M.HipModel.load(path, max_batch=64, logits_batch=64, **kw)

    def outputs(self, logits, ids):
        """The attention outputs [rows][HEADS hd] that rows of logits hold."""
        own = logits[np.arange(len(ids)), ids].astype(np.float64)
        return logits[:, IDS:].astype(np.float64) / own[:, None]

    def exact(self, ids, rows):
        """The outputs of positions `rows` (softmax over the whole row, float64; keys and values as an f16 cache holds them)."""
        with np.errstate(all="ignore"):
            k, v = (t[ids].astype(np.float16).astype(np.float64) for t in (self.k, self.v))
            out = np.empty((len(rows), HEADS * self.hd))
            for i, r in enumerate(rows):
                for h in range(HEADS):
                    s = (k[:r + 1] * self.q[ids[r], h]).sum(1) / np.sqrt(self.hd)
                    p = np.exp(s - s.max())
                    out[i, h * self.hd:(h + 1) * self.hd] = ((p / p.sum())[:, None] * v[:r + 1]).sum(0)
        return out
