"""A synthetic attention-only decoder and its GPU backend for the engine.

This is the harness that drives the paged KV path the way rvllm's forward
does (src/model.rs:600-644 per layer; the CUDA backend's forward_sample,
src/cuda/engine.rs:339-404): token embedding, then per layer the Q/K/V
projection (one fused QKV GEMM), attention prep with the K/V append
(rvkv_attn_prep_qkv),
attention straight over the paged cache (rvkv_paged_prefill for a prefill
item, rvkv_paged_decode_planned under a per-forward decode plan for a decode
batch) and the output projection with
a residual add; then tied-embedding logits and the greedy pick on the GPU
(rvkv_argmax). The MLP, norms and real checkpoints are outside the KV path
and left out: the weights are seeded random. The projections are plain
library GEMMs (torch on the GPU); every KV-path step is this library's HIP
code.

Sampling is greedy only (the GPU argmax), like the reference's CUDA
backend fast path for SamplingParams::GREEDY (src/cuda/engine.rs:96-125).
"""
from __future__ import annotations

import ctypes
import math
from dataclasses import dataclass
from itertools import chain
from types import SimpleNamespace
from typing import Dict, List

import numpy as np
import torch

from . import _lib
from ._lib import check
from .kv_storage import HipDecodePlan, HipKvStorage
from .rope import rope_cos_sin


@dataclass
class AttnModelConfig:
    vocab: int = 1024
    hidden: int = 256
    n_layers: int = 2
    n_heads: int = 8
    n_kv_heads: int = 2
    head_dim: int = 64
    qkv_bias: bool = False
    qk_norm: bool = False
    rope_theta: float = 10000.0
    eps: float = 1e-6
    context_length: int = 4096
    window: int = 0
    seed: int = 1234


def init_weights(cfg: AttnModelConfig) -> Dict[str, np.ndarray]:
    """Seeded f32 weights (host). Projections are scaled so q/k/v and the
    attention output keep unit-order magnitudes."""
    rng = np.random.default_rng(cfg.seed)
    D, H, KV, hd = cfg.hidden, cfg.n_heads, cfg.n_kv_heads, cfg.head_dim
    f = lambda *s, scale=1.0: (rng.standard_normal(s) * scale).astype(
        np.float32)
    w = {"embed": f(cfg.vocab, D)}
    for l in range(cfg.n_layers):
        w[f"wq{l}"] = f(D, H * hd, scale=1 / math.sqrt(D))
        w[f"wk{l}"] = f(D, KV * hd, scale=1 / math.sqrt(D))
        w[f"wv{l}"] = f(D, KV * hd, scale=1 / math.sqrt(D))
        w[f"wo{l}"] = f(H * hd, D, scale=1 / math.sqrt(H * hd))
        if cfg.qkv_bias:
            w[f"bq{l}"] = f(H * hd, scale=0.5)
            w[f"bk{l}"] = f(KV * hd, scale=0.5)
            w[f"bv{l}"] = f(KV * hd, scale=0.5)
        if cfg.qk_norm:
            w[f"qn{l}"] = (1.0 + f(hd, scale=0.2)).astype(np.float32)
            w[f"kn{l}"] = (1.0 + f(hd, scale=0.2)).astype(np.float32)
    return w


def logit_scale(cfg: AttnModelConfig) -> float:
    return 1.0 / math.sqrt(cfg.hidden)


def padded_tables(items) -> np.ndarray:
    """[batch, max_blocks] u32 block tables, padded with each row's last
    block (GatherPlan's padding, src/kv_storage.rs:50-75)."""
    rows = [list(it.read_blocks) or [0] for it in items]
    n = np.array([len(r) for r in rows])
    flat = np.fromiter(chain.from_iterable(rows), np.uint32, int(n.sum()))
    col = np.minimum(np.arange(n.max()), n[:, None] - 1)
    return flat[col + (np.cumsum(n) - n)[:, None]]


class HipBackend:
    """Engine backend (forward_sample / release / copy_blocks) on one GPU."""

    def __init__(self, cfg: AttnModelConfig, weights: Dict[str, np.ndarray],
                 num_blocks: int, block_size: int, device: str = "cuda"):
        self.cfg = cfg
        self.config = SimpleNamespace(context_length=cfg.context_length)
        self.dev = torch.device(device)
        self.w = {k: torch.from_numpy(v).to(self.dev) for k, v in
                  weights.items()}
        # One fused QKV projection per layer (Q heads, then K, then V),
        # consumed in place by rvkv_attn_prep_qkv.
        for l in range(cfg.n_layers):
            self.w[f"wqkv{l}"] = torch.cat(
                [self.w[f"wq{l}"], self.w[f"wk{l}"], self.w[f"wv{l}"]],
                dim=1).contiguous()
            if cfg.qkv_bias:
                self.w[f"bqkv{l}"] = torch.cat(
                    [self.w[f"bq{l}"], self.w[f"bk{l}"], self.w[f"bv{l}"]])
        self.st = HipKvStorage(cfg.n_layers, num_blocks, block_size,
                               cfg.n_kv_heads, cfg.head_dim)
        self._L = _lib.load()
        self.last_logits = None
        self.forwards = 0
        self._plans = {}
        # Pinned staging of a forward's index arrays, one copy a forward (nine
        # pageable copies, each waited for, took 0.16 ms of a decode forward
        # and 0.86 ms of a prompt's); _sent: that copy is done.
        self._stage = torch.empty(0, dtype=torch.int32)
        self._sent = torch.cuda.Event()
        # RoPE rows of every position the model takes, on the GPU; a forward
        # gathers its own (computing 1700 rows' angles on the host took 0.9 ms
        # a forward). 2^17 positions take 0.2-0.3 s here, once.
        self._rope = self._rope_rows(np.arange(min(cfg.context_length,
                                                   1 << 17)))

    def _rope_rows(self, pos) -> tuple:
        """cos and sin of the positions' angles, on the GPU."""
        return tuple(torch.from_numpy(a).to(self.dev) for a in
                     rope_cos_sin(self.cfg.rope_theta, self.cfg.head_dim,
                                  pos))

    def _send(self, arrays) -> List[torch.Tensor]:
        """The arrays as int32 device tensors, in one copy (each starts on
        a 256-byte boundary)."""
        at, n = [], 0
        for a in arrays:
            at.append(n)
            n += -(-a.size // 64) * 64
        self._sent.synchronize()  # the staging of the last forward is free
        if self._stage.numel() < n:
            self._stage = torch.empty(2 * n, dtype=torch.int32,
                                      pin_memory=True)
        host = self._stage.numpy()
        for a, i in zip(arrays, at):
            host[i:i + a.size] = a.reshape(-1)
        dev = torch.empty(n, dtype=torch.int32, device=self.dev)
        dev.copy_(self._stage[:n], non_blocking=True)
        self._sent.record()
        return [dev[i:i + a.size].view(a.shape) for a, i in zip(arrays, at)]

    def _u32(self, a) -> torch.Tensor:
        arr = np.ascontiguousarray(np.asarray(a, np.uint32)).view(np.int32)
        return torch.from_numpy(arr.copy()).to(self.dev)

    def release(self, seq_id: int) -> None:
        pass  # the KV path keeps no per-sequence device state

    def copy_blocks(self, src, dst) -> None:
        self.st.copy_blocks(self._u32(src), self._u32(dst))

    def forward_sample(self, items, last_only: bool, samplers) -> List[int]:
        c, w, st = self.cfg, self.w, self.st
        H, KV, hd = c.n_heads, c.n_kv_heads, c.head_dim
        n_new = np.array([len(it.tokens) for it in items])
        first = np.array([it.position_offset for it in items], np.int64)
        rows, last = int(n_new.sum()), np.cumsum(n_new) - 1
        toks = np.fromiter(chain.from_iterable(it.tokens for it in items),
                           np.int64, rows)
        # row r of item i: first[i] + r - (row the item starts at)
        pos = np.arange(rows) + np.repeat(first - (last + 1 - n_new), n_new)
        slots = np.fromiter(
            chain.from_iterable(chain.from_iterable(
                it.write_positions for it in items)),
            np.uint32).reshape(-1, 2)
        rope = None
        if rows and int(pos.max()) >= self._rope[0].shape[0]:
            rope = self._rope_rows(pos)  # (past the table: these rows alone)
        toks, pos, sb, so, tables, offs, reads, last = self._send(
            [toks, pos, slots[:, 0], slots[:, 1], padded_tables(items),
             first, np.array([it.read_num_tokens for it in items], np.int64),
             last])
        cos, sin = rope or (t.index_select(0, pos) for t in self._rope)
        x = w["embed"][toks]
        scale = 1.0 / math.sqrt(hd)
        decode = not last_only and bool((n_new == 1).all())
        if decode:
            # One decode plan per forward, shared by every layer (rvllm's
            # GatherPlan); kept per batch size and updated in place.
            lens = [it.read_num_tokens for it in items]
            plan = self._plans.get(len(items))
            if plan is None:
                plan = HipDecodePlan(st, lens, H, window=c.window)
                self._plans[len(items)] = plan
            else:
                plan.update(lens)
        for l in range(c.n_layers):
            qkv = x @ w[f"wqkv{l}"]
            qr = st.attn_prep_qkv(l, qkv, H, cos, sin, sb, so,
                                  bias=w.get(f"bqkv{l}"),
                                  q_norm=w.get(f"qn{l}"),
                                  k_norm=w.get(f"kn{l}"), eps=c.eps)
            if decode:
                att = st.paged_decode_planned(l, plan, qr, tables, reads,
                                              scale=scale)
            else:
                att = torch.empty_like(qr)
                r0 = 0
                for i, it in enumerate(items):  # one prefill item at a time
                    n = len(it.tokens)
                    # (its own blocks: by the batch's width a short prompt
                    # would be taken for a chunk behind a long context)
                    w_i = max(1, len(it.read_blocks))
                    st.paged_prefill(l, qr[r0:r0 + n].view(1, n, H, hd),
                                     tables[i:i + 1, :w_i], offs[i:i + 1],
                                     reads[i:i + 1],
                                     out=att[r0:r0 + n].view(1, n, H, hd),
                                     scale=scale, window=c.window)
                    r0 += n
            x = x + att.view(rows, H * hd) @ w[f"wo{l}"]
        xs = x[last]
        logits = (xs @ w["embed"].T) * logit_scale(c)
        logits = logits.contiguous()
        ids = torch.empty(len(items), dtype=torch.int32, device=self.dev)
        check(self._L.rvkv_argmax(ctypes.c_void_p(logits.data_ptr()),
                                  len(items), c.vocab,
                                  ctypes.c_void_p(ids.data_ptr()),
                                  ctypes.c_void_p(st.stream.cuda_stream)))
        self.last_logits = logits
        self.forwards += 1
        return ids.cpu().numpy().view(np.uint32).tolist()
