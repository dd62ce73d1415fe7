"""Token-shift mixing and the decayed linear-attention recurrence ("wkv") on per-sequence
state slots -> csrc/kernels/wkv.hip.

State per sequence slot and layer: ``S`` fp32 [slots, heads, dk, dv] and ``prev`` fp32 [slots,
width] (the previous token's layer input).  A sequence whose first row of a step is position 0
starts from zeros whatever the slot held, so freed slots are reused without clearing.

Batch layout: sequence ``s`` owns rows ``[cu[s], cu[s+1])`` of the step (``cu`` None: row ``s``,
a pure decode step); ``slots[s]`` is its state slot (< 0: padding row, skipped).
"""

from __future__ import annotations

from typing import Optional

import torch

from ._dispatch import check, lib, ptr, require, stream, use_hip, workspace


CHUNK = 64                 # tokens per chunk of the chunk-parallel form (wkv.hip WC)
CHUNK_DIM = 64             # ... and its widest head


def chunk_rows(nseq: int, heads: int) -> int:
    """Rows from which a sequence takes the chunk-parallel form.  The token-by-token kernel costs
    0.5 us a token whatever the batch, until its workgroups share CUs; the other form about 23 us
    for its launches and then work per chunk: 1.7 us per sequence at 32 heads, so that a step of
    many sequences needs longer ones.  MI355X, 32 heads, token by token / chunks: 1 x 32 rows 21 /
    20 us, 1 x 64 35 / 22, 16 x 32 25 / 36, 64 x 8 29 / 95, 1 x 4096 2091 / 100."""
    return 48 + min(64, nseq * heads // 32)


def chunk_rows_beside(nseq: int, heads: int) -> int:
    """Rows from which the shorter sequences of a step go along where the chunk-parallel form is launched for a long
    one: they then cost a chunk each, but no more tokens after one another.  MI355X, a sequence of 500 rows and so many
    shorter ones, token by token / along: 40 heads, 3 of 8 43 / 36 us, 3 of 48 64 / 43, 15 of 8 49 / 63, 15 of 24 59 / 64,
    15 of 48 74 / 67, 63 of 48 147 / 160; 16 heads, 15 of 8 33 / 32, 15 of 24 41 / 34, 63 of 24 55 / 72, 63 of 48 75 / 82;
    51 to 102 rows, 11 sequences of 40 heads 84 / 54."""
    return max(1, nseq * heads // 20)


def takes_chunks(rows: int, nseq: int, split: int, longest: int = 0) -> bool:
    """Whether the chunk-parallel form is launched beside the token-by-token one, each of which takes
    its own sequences.  Where the caller does not know the ``longest`` sequence's rows, only the device
    does: the three launches cost 10 to 13 us when they take nothing (MI355X, 32 heads, without / with
    them: 8 x 24 rows 18 / 28 us, 64 x 48 82 / 95), a long sequence left to the other form 0.5 us a row
    (16 sequences, one of 160 rows 93 / 45, of 256 146 / 47).  So they are made where rows enough for a
    long sequence are there and it is likely -- 24 rows a sequence: 16 sequences of 20 but one of 96 take
    57 / 51 -- or would cost some fifty us if it were one, 160 rows beside one for every sequence."""
    if split <= 0 or longest:
        return 0 < split <= longest
    return rows - nseq + 1 >= split and (rows >= 24 * nseq or rows - nseq >= 160)


def chunk_split(rows: int, nseq: int, heads: int, longest: int = 0) -> int:
    """Rows from which the sequences of a step take the chunk-parallel form, 0: it is not launched.  Shorter ones go
    along beside a long one.  Where the ``longest`` sequence's rows are not given there may be none, and the launches were
    made for nothing: then they do if the average is some 20 rows above what goes along.  MI355X, token by token (with
    those launches 5 to 6 us more) / in chunks: 32 heads, 8 of 24 18 / 28 us, 16 of 32 25 / 36, 8 of 50 31 / 32; 16 heads, 16 of
    20 16 / 28, 16 of 20 to 40 27 / 33, 8 of 50 30 / 24.  (The device could look for a long one: 1 us in each such step.)"""
    split = chunk_rows(nseq, heads)
    if not takes_chunks(rows, nseq, split, longest):
        return 0
    if nseq == 1:
        return 1                           # (whatever part of the rows it owns)
    least = min(split, chunk_rows_beside(nseq, heads))
    return least if longest or rows // nseq >= min(split, least + 20) else split


def _seq_bounds(cu: Optional[torch.Tensor], nseq: int):
    if cu is None:
        return [(s, s + 1) for s in range(nseq)]
    c = cu.tolist()
    return [(c[s], c[s + 1]) for s in range(nseq)]


def token_shift_mix(x: torch.Tensor, mu: torch.Tensor, prev_state: torch.Tensor,
                    slots: torch.Tensor, cu: Optional[torch.Tensor], nseq: int,
                    positions: torch.Tensor, out_dtype: torch.dtype) -> torch.Tensor:
    """x fp32 [T, W]; mu [NS, W] -> [NS, T, W] in out_dtype:  x_t + (x_{t-1} - x_t) * mu_s, with
    x_{-1} read from the sequence's slot (zeros at position 0).  Does not update the slot."""
    T, W = x.shape
    NS = mu.shape[0]
    if not use_hip(x):
        prev = torch.zeros_like(x)
        for s, (lo, hi) in enumerate(_seq_bounds(cu, nseq)):
            if hi <= lo or int(slots[s]) < 0:
                continue
            prev[lo + 1:hi] = x[lo:hi - 1]
            if int(positions[lo]) > 0:
                prev[lo] = prev_state[int(slots[s])]
        return (x[None] + (prev - x)[None] * mu.float()[:, None, :]).to(out_dtype)
    require(x.dtype == torch.float32 and x.is_contiguous() and prev_state.dtype == torch.float32
            and prev_state.is_contiguous() and mu.is_contiguous() and mu.dtype == out_dtype,
            "token_shift_mix: layout")
    require(slots.dtype == torch.int32 and positions.dtype == torch.int32 and
            (cu is None or cu.dtype == torch.int32), "token_shift_mix: int32 metadata")
    out = torch.empty(NS, T, W, dtype=out_dtype, device=x.device)
    check(lib().eia_token_shift_mix(ptr(x), ptr(mu), NS, ptr(prev_state), ptr(slots), ptr(cu),
                                    nseq, ptr(positions), ptr(out), out.stride(0), T, W,
                                    1 if out_dtype == torch.bfloat16 else 0, stream(x)),
          "token_shift_mix")
    return out


def wkv_scan(r: torch.Tensor, k: torch.Tensor, v: torch.Tensor, g: torch.Tensor,
             dec: torch.Tensor, w0: torch.Tensor, u: torch.Tensor, norm_w: torch.Tensor,
             S: torch.Tensor, prev_state: torch.Tensor, x: torch.Tensor, slots: torch.Tensor,
             cu: Optional[torch.Tensor], nseq: int, positions: torch.Tensor,
             seq_lens: Optional[torch.Tensor], eps: float, heads: int,
             longest: int = 0) -> torch.Tensor:
    """r, k, v, g [T, H*D] (same row stride), dec fp32 [T, H*D] (decay pre-activation without
    w0) -> y [T, H*D].  Per head and token, in fp32:
        w = exp(-exp(dec + w0));  o = (S + diag(u) k v^T)^T r;  S <- diag(w) S + k v^T
        y = o / rms(o) * norm_w * silu(g)
    S is read from / written to the sequence's slot; prev_state[slot] <- x[last row].
    ``longest``: rows of the longest sequence, where they are known on the host."""
    T, HD = r.shape
    D = HD // heads
    if not use_hip(r):
        y = torch.zeros(T, HD, dtype=torch.float32)
        rf, kf, vf, gf = (t.float().view(T, heads, D) for t in (r, k, v, g))
        w = torch.exp(-torch.exp(dec.float() + w0.float())).view(T, heads, D)
        uf = u.float().view(heads, D)
        for s, (lo, hi) in enumerate(_seq_bounds(cu, nseq)):
            sl = int(slots[s])
            if hi <= lo or sl < 0:
                continue
            st = torch.zeros(heads, D, D) if int(positions[lo]) == 0 else S[sl].clone()
            for t in range(lo, hi):
                kv = kf[t][:, :, None] * vf[t][:, None, :]
                o = torch.einsum("hi,hij->hj", rf[t], st + uf[:, :, None] * kv)
                st = w[t][:, :, None] * st + kv
                o = o / torch.sqrt((o * o).mean(-1, keepdim=True) + eps)
                y[t] = o.reshape(-1)
            S[sl] = st
            prev_state[sl] = x[hi - 1]
        return (y * norm_w.float() * torch.nn.functional.silu(gf.reshape(T, HD))).to(r.dtype)
    bf = r.dtype == torch.bfloat16
    require(bf or r.dtype == torch.float32, "wkv_scan: bf16 or fp32")
    ld = r.stride(0)
    for t in (r, k, v, g):
        require(t.dtype == r.dtype and t.stride(1) == 1 and t.stride(0) == ld and
                t.shape == r.shape, "wkv_scan: r/k/v/g layout")
    require(dec.dtype == torch.float32 and dec.stride(1) == 1 and dec.shape == r.shape, "dec fp32")
    require(S.dtype == torch.float32 and S.is_contiguous() and S.shape[1:] == (heads, D, D), "S")
    require(prev_state.dtype == torch.float32 and prev_state.is_contiguous() and
            x.dtype == torch.float32 and x.is_contiguous(), "prev / x fp32")
    require(slots.dtype == torch.int32 and positions.dtype == torch.int32, "int32 metadata")
    for t in (w0, u, norm_w):
        require(t.dtype == r.dtype and t.is_contiguous() and t.numel() == HD, "per-channel params")
    y = torch.empty(T, HD, dtype=r.dtype, device=r.device)
    args = (ptr(r), ptr(k), ptr(v), ptr(g), ld, ptr(dec), dec.stride(0), ptr(w0), ptr(u),
            ptr(norm_w), ptr(S), ptr(prev_state), ptr(x), x.shape[1], ptr(slots), ptr(cu),
            ptr(positions), ptr(seq_lens), ptr(y), y.stride(0), float(eps), nseq)
    split = chunk_split(T, nseq, heads, longest) if cu is not None and D <= CHUNK_DIM else 0
    if split != 1:
        check(lib().eia_wkv_scan(*args, heads, D, split, 1 if bf else 0, stream(r)), "wkv_scan")
    if split:
        n = T // CHUNK + nseq
        ws, (U, L) = workspace(r.device, 4 * n * heads * CHUNK_DIM * CHUNK_DIM, 4 * n * heads * CHUNK_DIM)
        check(lib().eia_wkv_scan_chunked(*args, T, heads, D, split, U, L,
                                         1 if bf else 0, stream(r)), "wkv_scan_chunked")
    return y
