"""Batched server-side sampling (the last stage samples; only token ids leave it).

Reference: ``StageConnectionHandler._sample_token`` samples one row per request in
Python (reference src/rpc_handler.py:327-403) with defaults temperature 0.8 / top_p 0.9 /
top_k 0 in the handler (:71-73) and repetition penalty 1.5 (:164); the CLI sends
temperature 1.0 / top_p 0.92 / top_k 50 (src/main.py:806-809).  Here all rows of a step are
sampled by one HIP kernel launch with per-row parameters (``ops.sample``).
"""
from __future__ import annotations

import dataclasses
import hashlib
from typing import List, Optional, Sequence

import numpy as np
import torch

from .. import ops

RECENT = 50  # reference: generated_tokens[-50:] (src/rpc_handler.py:348; src/rpc_transport.py:797)


@dataclasses.dataclass
class SamplingParams:
    temperature: float = 0.8
    top_p: float = 0.9
    top_k: int = 0
    repetition_penalty: float = 1.5

    @classmethod
    def from_metadata(cls, md: dict) -> "SamplingParams":
        return cls(float(md.get("temperature", 0.8)), float(md.get("top_p", 0.9)), int(md.get("top_k", 0)),
                   float(md.get("repetition_penalty", 1.5)))


def session_seed(session_id: str, step: int, base_seed: int = 0) -> int:
    h = hashlib.blake2b(f"{base_seed}:{session_id}:{step}".encode(), digest_size=8).digest()
    return int.from_bytes(h, "little") & 0x7FFFFFFFFFFFFFFF


class BatchSampler:
    """Samples the rows of a step; token ids [rows] on the logits' device, in the order of its current stream.

    The rows' parameters, histories and seeds go to the device as one copy from pinned memory, which two calls use in turn, and
    a call does not wait for its tokens.  With five copies, the one from pageable memory waiting for the step's kernels, and a
    wait at the end, 64 rows of a 7B model's last 4 blocks took 779 us a step, and 637 with this alone, where steps follow each
    other unread.  A server reads each step's tokens: 738 us instead of 806, the kernels' changes of that time among them."""

    ROW = 2 + 3 + 2 + RECENT  # 32-bit words of a row: seed; temperature, top p, penalty; top k, history's length; history

    def __init__(self, device, max_rows: int = 256):
        self.device = torch.device(device)
        self.max_rows = max_rows
        pin = self.device.type == "cuda"
        self._host = [torch.empty(self.ROW * max_rows, dtype=torch.int32, pin_memory=pin) for _ in range(2)]
        self._done = [None, None]  # the calls that used them: (stream, event)
        self._turn = 0
        self._ws: Optional[torch.Tensor] = None

    def __call__(self, logits: torch.Tensor, params: Sequence[SamplingParams], histories: Sequence[Sequence[int]],
                 seeds: Sequence[int]) -> torch.Tensor:
        R, V = logits.shape
        assert R == len(params) == len(histories) == len(seeds)
        if R == 0:
            return torch.empty(0, dtype=torch.long, device=logits.device)
        if all(p.temperature <= 0 for p in params):
            return ops.argmax(logits)
        if R > self.max_rows:
            return torch.cat([self(logits[i:i + self.max_rows], params[i:i + self.max_rows],
                                   histories[i:i + self.max_rows], seeds[i:i + self.max_rows])
                              for i in range(0, R, self.max_rows)])
        dev = logits.device
        cuda = dev.type == "cuda"
        if cuda and torch.cuda.is_current_stream_capturing():
            raise RuntimeError("sampling reads its rows' parameters from the host: it cannot be captured")
        last, self._turn = self._done[self._turn], self._turn ^ 1
        if self._done[self._turn] is not None:
            self._done[self._turn][1].synchronize()
        host = self._host[self._turn][: self.ROW * R]
        words = host.numpy()
        words[: 2 * R].view(np.int64)[:] = [int(s) & 0x7FFFFFFFFFFFFFFF for s in seeds]
        f = words[2 * R:5 * R].view(np.float32).reshape(3, R)
        f[0] = [p.temperature for p in params]
        f[1] = [p.top_p for p in params]
        f[2] = [p.repetition_penalty for p in params]
        ii = words[5 * R:7 * R].reshape(2, R)
        ii[0] = [p.top_k for p in params]
        rec = words[7 * R:].reshape(R, RECENT)
        rec[:] = 0
        for r, h in enumerate(histories):
            h = list(h)[-RECENT:]
            ii[1, r] = len(h)
            if h:
                rec[r, : len(h)] = h
        d = host.to(dev, non_blocking=True)
        fd, idv = d[2 * R:5 * R].view(torch.float32).view(3, R), d[5 * R:7 * R].view(2, R)
        ws = None
        if cuda:
            stream = torch.cuda.current_stream(dev)
            if self._ws is None or self._ws.device != dev or self._ws.numel() < R * V:
                self._ws = torch.empty(self.max_rows * V, dtype=torch.float32, device=dev)
            ws = self._ws
            if last is not None and last[0] != stream:  # the workspace is the other stream's until its call has run
                stream.wait_event(last[1])
                ws.record_stream(stream)
        out = ops.sample(logits, fd[0], fd[1], idv[0], fd[2], d[7 * R:].view(R, RECENT), idv[1], d[: 2 * R].view(torch.int64),
                         workspace=ws)
        if cuda:
            event = torch.cuda.Event()
            event.record(stream)
            self._done[self._turn] = (stream, event)
        return out
