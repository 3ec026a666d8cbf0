"""The GSPO reward on the device: strict identity of every call against its window's label.

Reference: scripts/gspo.py:86-89 (strict_identity), 446 (the reward of a rollout), scripts/train.py:170-188
(ref_errors, the edlib NW path's error positions), scripts/evaluate.py:30 (EMPTY_MAX). The reference runs
edlib on the host, one call after another; here one kernel scores every call of a rollout at once
(vk_strict_identity: the edit-distance DP as a systolic array, 256 label rows per wavefront).

The alignment path behind the error positions: at every cell the first optimal predecessor in the order
diagonal, deletion, insertion. edlib's own traceback order is not available here; the edit distance, and
the reward whenever every label base is scored, do not depend on the path.
"""

from typing import List, Optional, Sequence

import numpy as np
import torch

from . import _lib
from ._lib import call, ptr, require_device
from .tokenizer import EOS, N_SPECIAL

MAX_CALL = 8192  # the longest call vk_strict_identity takes
EMPTY_MAX = 4  # scripts/evaluate.py:30: a window without DNA scores 1 for a call of at most this many bases


def _pack(strings: Sequence[bytes], device):
    lens = [len(s) for s in strings]
    off = np.zeros(len(strings), dtype=np.int64)
    if len(strings) > 1:
        off[1:] = np.cumsum(lens[:-1])
    data = np.frombuffer(b"".join(strings), dtype=np.uint8) if sum(lens) else np.zeros(1, np.uint8)
    return (torch.from_numpy(data.copy()).to(device), torch.from_numpy(off).to(device),
            torch.tensor(lens, dtype=torch.int32).to(device), max(lens) if lens else 0)


def _upload(arrays, device):
    """Host arrays as device tensors of one upload (8-byte aligned slices of one buffer)."""
    sizes = [-(-a.nbytes // 8) * 8 for a in arrays]
    host = np.zeros(max(sum(sizes), 8), dtype=np.uint8)
    o = 0
    spans = []
    for a, n in zip(arrays, sizes):
        host[o:o + a.nbytes] = a.reshape(-1).view(np.uint8)
        spans.append((o, a.nbytes, getattr(torch, a.dtype.name)))
        o += n
    dev = torch.from_numpy(host).to(device)
    return [dev[o:o + n].view(dt) for o, n, dt in spans]


def _run(call_data, call_off, call_len, max_call, refs: Sequence[str], scored: Sequence[np.ndarray], ref_of_call,
         device, empty_max):
    ref_b = [r.encode() for r in refs]
    sc = [np.asarray(s, dtype=bool).astype(np.uint8) for s in scored]
    assert all(len(s) == len(r) for s, r in zip(sc, ref_b)), "strict_identity: a scored mask per label base"
    lens = np.array([len(r) for r in ref_b], dtype=np.int32)
    off = np.concatenate([[0], np.cumsum(lens[:-1], dtype=np.int64)])[:len(lens)].astype(np.int64)
    data = np.frombuffer(b"".join(ref_b) or b"\0", dtype=np.uint8)
    mask = np.concatenate([*sc, np.zeros(0 if lens.sum() else 1, np.uint8)])
    ref_off, ref_len, roc, ref_data, sc_data = _upload([off, lens, np.asarray(ref_of_call, dtype=np.int32), data, mask],
                                                       device)
    n = call_len.shape[0]
    reward = torch.empty(n, dtype=torch.float32, device=device)
    dist = torch.empty(n, dtype=torch.int32, device=device)
    errs = torch.empty(n, dtype=torch.int32, device=device)
    call("vk_strict_identity", ptr(call_data), ptr(call_off), ptr(call_len), ptr(ref_data), ptr(ref_off),
         ptr(ref_len), ptr(sc_data), ptr(roc), n, len(refs), int(lens.max()) if len(lens) else 0, max_call,
         float(empty_max), ptr(reward), ptr(dist), ptr(errs), _lib.stream_handle())
    return {"reward": reward, "edit_distance": dist, "scored_errors": errs}


def strict_identity(calls: Sequence[str], labels: Sequence[str], scored: Sequence[np.ndarray],
                    ref_of_call: Optional[Sequence[int]] = None, device="cuda", empty_max=EMPTY_MAX):
    """Strict identity of calls[c] against labels[ref_of_call[c]] (default: labels[c]) with scored[r] the bool
    mask of label r's counted bases; returns device tensors {reward fp32, edit_distance, scored_errors} [len(calls)].
    Reference: scripts/gspo.py:86-89."""
    require_device(torch.empty(0, device=device), "strict_identity")
    ref_of_call = list(range(len(calls))) if ref_of_call is None else list(ref_of_call)
    data, off, lens, max_call = _pack([c.encode() for c in calls], device)
    return _run(data, off, lens, max_call, labels, scored, ref_of_call, device, empty_max)


def gspo_rewards(calls: List[str], labels: List[str], weights: List[np.ndarray], G: int, device="cuda"):
    """The rollout's reward [windows, G] (scripts/gspo.py:446): call i against label i // G, scored where the
    label's weight is positive. float64 host array, as the reference's."""
    res = strict_identity(calls, labels, [np.asarray(w) > 0 for w in weights], [i // G for i in range(len(calls))],
                          device)
    return res["reward"].double().cpu().numpy().reshape(-1, G)


def _bases(tokens: torch.Tensor, tokenizer):
    """The base strings of output tokens [N, T] on the device (vk_tokens_to_bases): rows [N, T k] uint8 and their
    lengths [N] int32. No host synchronisation."""
    require_device(tokens, "output tokens to bases")
    N, T = tokens.shape
    V, k = tokenizer.vocab_size, tokenizer.k
    strings = [b"" if t < N_SPECIAL else tokenizer.strings[t].encode() for t in range(V)]
    host = b"".join(s.ljust(k, b"\0") + bytes([len(s)]) for s in strings)
    table = torch.from_numpy(np.frombuffer(host, dtype=np.uint8).copy()).to(tokens.device)
    tokens = tokens.long().contiguous()
    rows = torch.empty(N, T * k, dtype=torch.uint8, device=tokens.device)
    lens = torch.empty(N, dtype=torch.int32, device=tokens.device)
    call("vk_tokens_to_bases", ptr(tokens), N, T, ptr(table), V, k, EOS, ptr(rows), ptr(lens), _lib.stream_handle())
    return rows, lens


def calls_from_tokens(tokens: torch.Tensor, tokenizer):
    """Device base strings of the engine's output tokens [N, T] (int64): the tokenizer's decode on the device
    (stops at the first EOS, skips PAD and BOS; a token writes its k-mer or tail). Returns (bytes [total] uint8,
    offsets [N] int64, lengths [N] int32, max length). Host tokens are decoded on the host."""
    if not tokens.is_cuda:
        ids = tokens.clamp(0, tokenizer.vocab_size - 1).tolist()
        return _pack([tokenizer.decode(r).encode() for r in ids], tokens.device)
    rows, lens = _bases(tokens, tokenizer)
    offsets = torch.cumsum(lens.long(), 0) - lens
    out = rows[torch.arange(rows.shape[1], device=rows.device) < lens[:, None]]
    if out.numel() == 0:
        out = torch.zeros(1, dtype=torch.uint8, device=rows.device)
    return out, offsets, lens, int(lens.max()) if lens.numel() else 0


def gspo_rewards_from_tokens(tokens: torch.Tensor, tokenizer, labels: List[str], weights: List[np.ndarray], G: int,
                             empty_max=EMPTY_MAX):
    """The rollout's rewards straight from the engine's device output (no host decode): tokens [windows * G, T];
    returns the device dict of strict_identity (reward [windows * G] fp32)."""
    rows, lens = _bases(tokens, tokenizer)
    N, width = rows.shape
    # rows longer than the kernel's longest call: only then the lengths are read back
    longest = width if width <= MAX_CALL else int(lens.max())
    off = torch.arange(N, device=rows.device) * width
    return _run(rows, off, lens, longest, labels, [np.asarray(w) > 0 for w in weights], np.arange(N) // G,
                tokens.device, empty_max)
