"""Linear-attention recurrences with one decay number per head and token, or one per key channel
and token, on per-sequence state slots -> csrc/kernels/linear_scan.hip.

Per head a matrix state S [dk, dv] (fp32, slot-resident) that every token scales and adds an
outer product to; the token's output reads the updated state:

    S_t = a_t S_(t-1) + b_t k_t v_t^T,        o_t = S_t^T q_t

* ``mode="decay"`` (retention): a_t = decay[h], b_t = 1.
* ``mode="exp_gates"`` (matrix memory with exponential gating): per head two gate
  pre-activations x_i, x_f per token; i = cap tanh(x_i / cap), f = logsigmoid(cap tanh(x_f /
  cap)) (cap 0: i = x_i, f = logsigmoid(x_f)); a running maximum m_t = max(f + m_(t-1), i) (m starts at 0) keeps the exponentials
  bounded: a_t = exp(f + m_(t-1) - m_t), b_t = exp(i - m_t); a normaliser n_t = a_t n_(t-1) +
  b_t k_t divides the output, o_t / (max(|n_t . q_t|, exp(-m_t)) + 1e-6).
* ``mode="channel"`` (gated linear attention): the row also holds ``rank`` columns of a low-rank
  branch; z = A2 lo + bias per head and key channel (fp32), a_t = sigmoid(z)^(1/tau) -- a vector
  that scales the state's rows channel by channel -- and b_t = 1.

q and k may be rotated by the token's position on their first ``rot_dims`` entries and are then
scaled; every head's output is divided by its root mean square, multiplied by an optional weight,
by silu or sigmoid of the gate columns and by ``out_scale``.

A sequence whose first row of the step is position 0 starts from the initial state whatever its
slot held, so freed slots are reused without clearing.  Batch layout: sequence ``s`` owns rows
``[cu[s], cu[s+1])`` of the step (``cu`` None: row ``s``, a pure decode step); ``slots[s]`` is its
state slot (< 0: padding row, skipped).

Prompt portions run a chunk-parallel form on the GPU (``chunk_plan``): the step's rows are cut
into chunks of 128 tokens (with a decay per key channel 64, or 32 where keys are wider than 64), every
chunk's own contribution to the state is formed in parallel, a short scan over a sequence's chunks
yields the state before each chunk, and the outputs of all chunks are formed in parallel from that
state and the chunk's own tokens.  Decode steps (also inside captured graphs) run a kernel of their
own for heads up to 128 wide.  The token-by-token kernel serves wider heads, prompt portions too short
for chunks or inside a captured graph, and value widths that four does not divide.
"""

from __future__ import annotations

import dataclasses
import math
import os
from typing import Optional

import torch

from ._dispatch import check, lib, ptr, require, stream, use_hip, workspace


@dataclasses.dataclass
class ScanSpec:
    """Constants of one recurrent layer (device tensors are fp32)."""
    heads: int
    dim: int                        # dk
    vdim: int                       # dv
    mode: str                       # "decay" | "exp_gates" | "channel"
    decay: Optional[torch.Tensor] = None        # [H] fp32 ("decay")
    cap: float = 0.0                            # gate soft cap ("exp_gates")
    inv_freq: Optional[torch.Tensor] = None     # [rot_dims / 2] fp32
    rot_dims: int = 0
    rot_half: bool = True
    qscale: float = 1.0
    kscale: float = 1.0
    gate_act: str = "silu"          # "silu" | "sigmoid"
    out_scale: float = 1.0
    eps: float = 0.0
    # "channel": A2 transposed [rank, H*dk] and its bias [H*dk] (fp32, device), tau
    a2t: Optional[torch.Tensor] = None
    a2b: Optional[torch.Tensor] = None
    tau: float = 1.0
    norm_shared: bool = False       # the weight after the head norm is [dv], shared by the heads


class ScanState:
    """Per-sequence slots of one recurrent layer: S fp32 [slots, H, dk, dv]; with exponential
    gates also the normaliser n [slots, H, dk] and the running maximum m [slots, H]."""

    __slots__ = ("S", "n", "m")

    def __init__(self, S: torch.Tensor, n: Optional[torch.Tensor] = None,
                 m: Optional[torch.Tensor] = None):
        self.S, self.n, self.m = S, n, m

    @classmethod
    def allocate(cls, num_slots: int, spec: ScanSpec, device):
        z = lambda *shape: torch.zeros(*shape, dtype=torch.float32, device=device)
        n = max(1, num_slots)
        if spec.mode == "exp_gates":
            return cls(z(n, spec.heads, spec.dim, spec.vdim), z(n, spec.heads, spec.dim),
                       z(n, spec.heads))
        return cls(z(n, spec.heads, spec.dim, spec.vdim))

    @staticmethod
    def slot_bytes(spec: ScanSpec) -> int:
        per = spec.heads * spec.dim * spec.vdim
        if spec.mode == "exp_gates":
            per += spec.heads * (spec.dim + 1)
        return 4 * per


CHUNK = 32                 # tokens per chunk with a decay per key channel (linear_scan.hip LC)
HEAD_CHUNK = 128           # ... with one decay per head and token (LK)
KEY_CHUNK64, KEY_DIM64 = 64, 64     # ... with a decay per key channel and narrow keys (GC), its widest dk
CHUNK_MAX_DIM = 128        # ... and its largest dk / dv
CHUNK_MIN_ROWS = 48        # a sequence with at least this many rows in the step selects it
# tests and measurements: take the chunk-parallel form whenever a plan is handed over
FORCE_CHUNKED = os.environ.get("EIA_SCAN_FORCE_CHUNKED", "0") == "1"


# (decays 0 / exponential gates 1 / a decay per channel 2, wider than 64): us per token of the token-by-token form; us for
# the launches, per row and head, per sequence and head of the chunk-parallel one (fitted to the figures behind).
# Sequences x rows, token by token / chunks, us:
RATES = {
    (0, False): (0.52, 24, 0.00034, 0.015),   # 32 x 64: 1x64 33 / 27, 16x64 36 / 43, 16x128 78 / 55, 64x64 107 / 126
    (0, True): (0.90, 36, 0.0012, 0.10),      # 16 x 128, rotated: 1x48 44 / 36, 16x64 67 / 82, 16x128 120 / 101, 64x64 241 / 209
    (1, False): (0.85, 25, 0.0003, 0.025),    # 32 x 64: 1x48 38 / 32, 16x48 43 / 47, 16x64 53 / 48, 64x64 166 / 115
    (1, True): (1.30, 31, 0.0010, 0.065),     # 16 x 128: 1x48 65 / 32, 16x48 70 / 61, 16x128 166 / 74, 64x64 339 / 159
    (2, False): (0.70, 30, 0.00059, 0.019),   # 32 x 32 x 64: 1x48 34 / 32, 16x64 50 / 59, 16x128 97 / 78, 64x64 130 / 146
    (2, True): (1.00, 32, 0.0017, 0.0),       # 16 x 64 x 128: 1x48 54 / 36, 16x64 72 / 60, 16x128 142 / 71, 64x64 281 / 141
}


class ChunkPlan:
    """A step's rows cut into chunks for the chunk-parallel forms: ``n`` chunks over sequences of
    ``lens`` rows from row ``row0`` on; ``rows`` the step's row count, ``longest`` the longest
    sequence's.  Forms that do not find their chunks themselves read two lists on the device, made
    when first asked for: ``chunks`` int32 [n, 4] (sequence, first row, tokens, 0) and ``seq_first``
    int32 [nseq + 1] (first chunk of every sequence)."""

    __slots__ = ("lens", "device", "chunk", "row0", "n", "rows", "nseq", "longest", "_lists")

    def __init__(self, lens, device, chunk: int, row0: int = 0):
        self.lens, self.device, self.chunk, self.row0 = list(lens), device, chunk, row0
        self.n = sum(-(-k // chunk) for k in self.lens)
        self.rows, self.nseq, self.longest = row0 + sum(self.lens), len(self.lens), max(self.lens)
        self._lists = None

    def lists(self):
        """(chunks, seq_first)."""
        if self._lists is None:
            chunks, first, row = [], [0], self.row0
            for s, n in enumerate(self.lens):
                for lo in range(0, n, self.chunk):
                    chunks += [s, row + lo, min(self.chunk, n - lo), 0]
                row += n
                first.append(len(chunks) // 4)
            i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=self.device)
            self._lists = i32(chunks).view(-1, 4), i32(first)
        return self._lists

    @property
    def chunks(self) -> torch.Tensor:
        return self.lists()[0]

    @property
    def seq_first(self) -> torch.Tensor:
        return self.lists()[1]

    def pays(self, heads: int, dim: int, cus: int = 256, channel: bool = False,
             key_dim: int = 0, exp_gates: bool = False) -> bool:
        """Whether the chunk-parallel form beats the token-by-token one for a layer of ``heads``
        heads up to ``dim`` wide.  The latter walks the longest sequence, so many us a token, while its
        workgroups, one per (sequence, head), do not share CUs.  The former costs so many us for its
        launches and for a head so many per row and per sequence."""
        wide = dim > 64
        if channel and key_dim > KEY_DIM64:
            serial = self.longest * (0.85 if wide else 0.5) * -(-self.nseq * heads // cus)
            return self.rows * heads * (0.0072 if wide else 0.0052) < serial
        token, launches, row, seq = RATES[(2 if channel else 1 if exp_gates else 0, wide)]
        busy = self.nseq * heads / (cus if wide else 2.7 * cus)
        return (launches + heads * (row * self.rows + seq * self.nseq) <
                token * self.longest * max(1.0, busy))


def chunk_plan(host_lens, device, chunk: int = CHUNK, min_rows: int = CHUNK_MIN_ROWS,
               row0: int = 0) -> Optional["ChunkPlan"]:
    """The chunk plan of a step whose sequences own ``host_lens`` rows each (batch order, from row
    ``row0`` on), or None when no sequence is long enough for the chunk-parallel form to pay."""
    if not host_lens or max(host_lens) < min_rows:
        return None
    return ChunkPlan(host_lens, device, chunk, row0)


def _seq_bounds(cu: Optional[torch.Tensor], nseq: int):
    if cu is None:
        return [(s, s + 1) for s in range(nseq)]
    c = cu.tolist()
    return [(c[s], c[s + 1]) for s in range(nseq)]


def _rotate(v: torch.Tensor, pos: torch.Tensor, spec: ScanSpec) -> torch.Tensor:
    """v fp32 [T, H, D]; pos [T]."""
    rd = spec.rot_dims
    if not rd:
        return v
    ang = pos.float()[:, None] * spec.inv_freq.float()[None, :rd // 2]       # [T, rd/2]
    cs, sn = torch.cos(ang)[:, None, :], torch.sin(ang)[:, None, :]
    out = v.clone()
    if spec.rot_half:
        a, b = v[..., :rd // 2], v[..., rd // 2:rd]
        out[..., :rd // 2], out[..., rd // 2:rd] = a * cs - b * sn, b * cs + a * sn
    else:
        a, b = v[..., 0:rd:2], v[..., 1:rd:2]
        out[..., 0:rd:2], out[..., 1:rd:2] = a * cs - b * sn, b * cs + a * sn
    return out


def linear_scan(fused: torch.Tensor, q_off: int, k_off: int, v_off: int, g_off: int,
                spec: ScanSpec, state: ScanState, slots: torch.Tensor,
                cu: Optional[torch.Tensor], nseq: int, positions: torch.Tensor,
                seq_lens: Optional[torch.Tensor] = None, norm_w: Optional[torch.Tensor] = None,
                i_off: int = 0, f_off: int = 0, out: Optional[torch.Tensor] = None,
                plan: Optional[ChunkPlan] = None, lo_off: int = 0) -> torch.Tensor:
    """fused [T, *]: rows of one fused projection holding q [H*dk], k [H*dk], v [H*dv], the gate
    [H*dv] (and, with exponential gates, the H input-gate and H forget-gate pre-activations) at
    the given column offsets -> y [T, H*dv] in fused's dtype (``out``: a view to write into).
    ``norm_w`` [H*dv] (or [dv], ``spec.norm_shared``): weight after the head RMS norm.
    ``lo_off``: first column of the low-rank decay branch ("channel").  Updates the sequences' slots.
    ``plan``: the step's ``chunk_plan`` -- the GPU then runs the chunk-parallel form (heads up to
    128 wide, outside graph capture)."""
    T = fused.shape[0]
    H, D, Dv = spec.heads, spec.dim, spec.vdim
    exp_gates = spec.mode == "exp_gates"
    channel = spec.mode == "channel"
    R = spec.a2t.shape[0] if channel else 0
    if out is None:
        out = torch.empty(T, H * Dv, dtype=fused.dtype, device=fused.device)
    require(out.shape == (T, H * Dv) and out.dtype == fused.dtype and out.stride(1) == 1,
            "linear_scan: out layout")
    if not use_hip(fused):
        f = fused.float()
        q = _rotate(f[:, q_off:q_off + H * D].reshape(T, H, D), positions[:T], spec) * spec.qscale
        k = _rotate(f[:, k_off:k_off + H * D].reshape(T, H, D), positions[:T], spec) * spec.kscale
        v = f[:, v_off:v_off + H * Dv].reshape(T, H, Dv)
        g = f[:, g_off:g_off + H * Dv]
        y = torch.zeros(T, H, Dv)
        if exp_gates:
            soft = (lambda z: spec.cap * torch.tanh(z / spec.cap)) if spec.cap > 0 else \
                (lambda z: z)
            gi = soft(f[:, i_off:i_off + H])
            gf = torch.nn.functional.logsigmoid(soft(f[:, f_off:f_off + H]))
        if channel:
            z = f[:, lo_off:lo_off + R] @ spec.a2t.float()
            z = z + spec.a2b.float() if spec.a2b is not None else z
            al = torch.exp(torch.nn.functional.logsigmoid(z) / spec.tau).reshape(T, H, D)
        for s, (lo, hi) in enumerate(_seq_bounds(cu, nseq)):
            sl = int(slots[s])
            if hi <= lo or sl < 0:
                continue
            fresh = int(positions[lo]) == 0
            S = torch.zeros(H, D, Dv) if fresh else state.S[sl].clone()
            if exp_gates:
                n = torch.zeros(H, D) if fresh else state.n[sl].clone()
                m = torch.zeros(H) if fresh else state.m[sl].clone()
            for t in range(lo, hi):
                kv = k[t][:, :, None] * v[t][:, None, :]
                if exp_gates:
                    m_new = torch.maximum(gf[t] + m, gi[t])
                    a, b = torch.exp(gf[t] + m - m_new), torch.exp(gi[t] - m_new)
                    S = a[:, None, None] * S + b[:, None, None] * kv
                    n = a[:, None] * n + b[:, None] * k[t]
                    m = m_new
                    den = torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-m)) + 1e-6
                    o = torch.einsum("hi,hij->hj", q[t], S) / den[:, None]
                else:
                    S = (al[t][:, :, None] if channel else spec.decay.float()[:, None, None]) * S + kv
                    o = torch.einsum("hi,hij->hj", q[t], S)
                y[t] = o / torch.sqrt((o * o).mean(-1, keepdim=True) + spec.eps)
            state.S[sl] = S
            if exp_gates:
                state.n[sl], state.m[sl] = n, m
        if norm_w is not None:
            y = y * (norm_w.float() if spec.norm_shared else norm_w.float().reshape(H, Dv))
        y = y.reshape(T, H * Dv)
        y = y * (torch.nn.functional.silu(g) if spec.gate_act == "silu" else torch.sigmoid(g))
        out.copy_((y * spec.out_scale).to(out.dtype))
        return out
    bf = fused.dtype == torch.bfloat16
    require(bf or fused.dtype == torch.float32, "linear_scan: bf16 or fp32")
    require(fused.stride(1) == 1 and max(q_off + H * D, k_off + H * D, v_off + H * Dv,
                                         g_off + H * Dv) <= fused.shape[1],
            "linear_scan: columns outside the row")
    require(spec.mode in ("decay", "exp_gates", "channel") and spec.gate_act in ("silu", "sigmoid"),
            "linear_scan: mode")
    require(state.S.dtype == torch.float32 and state.S.is_contiguous() and
            state.S.shape[1:] == (H, D, Dv), "linear_scan: state layout")
    if exp_gates:
        require(max(i_off, f_off) + H <= fused.shape[1] and state.n is not None and
                state.m is not None and state.n.is_contiguous() and state.m.is_contiguous() and
                spec.cap >= 0, "linear_scan: gates")
    elif channel:
        require(lo_off + R <= fused.shape[1] and spec.tau > 0 and
                spec.a2t.shape == (R, H * D) and spec.a2t.is_contiguous() and all(
                    t is None or (t.dtype == torch.float32 and t.is_cuda)
                    for t in (spec.a2t, spec.a2b)) and
                (spec.a2b is None or spec.a2b.numel() == H * D), "linear_scan: channel decays")
    else:
        require(spec.decay is not None and spec.decay.dtype == torch.float32 and
                spec.decay.is_cuda and spec.decay.numel() == H, "linear_scan: decay per head")
    require(spec.rot_dims == 0 or (spec.inv_freq is not None and spec.inv_freq.is_cuda and
                                   spec.inv_freq.dtype == torch.float32 and
                                   spec.inv_freq.numel() >= spec.rot_dims // 2 and
                                   spec.rot_dims <= D and spec.rot_dims % 2 == 0),
            "linear_scan: rotation")
    require(slots.dtype == torch.int32 and positions.dtype == torch.int32 and
            (cu is None or cu.dtype == torch.int32), "linear_scan: int32 metadata")
    require(norm_w is None or (norm_w.dtype == fused.dtype and norm_w.is_contiguous() and
                               norm_w.numel() == (Dv if spec.norm_shared else H * Dv)),
            "linear_scan: norm weight")
    mode = {"decay": 0, "exp_gates": 1, "channel": 2}[spec.mode]
    chan = (lo_off, R, ptr(spec.a2t), ptr(spec.a2b), 1.0 / float(spec.tau),
            0 if spec.norm_shared else Dv)
    if (plan is not None and plan.n and max(D, Dv) <= CHUNK_MAX_DIM and cu is not None
            and plan.rows == T and
            (FORCE_CHUNKED or plan.pays(H, max(D, Dv), channel=channel, key_dim=D, exp_gates=exp_gates))
            and not torch.cuda.is_current_stream_capturing()):
        dev = fused.device
        act = 0 if spec.gate_act == "silu" else 1
        if channel and D <= KEY_DIM64:
            n, W = T // KEY_CHUNK64 + nseq, -(-Dv // 64) * 64
            ws, (U, L, l, rot) = workspace(dev, 4 * n * H * KEY_DIM64 * W, 4 * n * H * KEY_DIM64, 4 * T * H * D,
                                           4 * T * spec.rot_dims)
            check(lib().eia_linear_scan_channels64(
                ptr(fused), fused.stride(0), q_off, k_off, v_off, g_off, ptr(spec.inv_freq),
                spec.rot_dims, 1 if spec.rot_half else 0, float(spec.qscale), float(spec.kscale),
                float(spec.out_scale), ptr(norm_w), ptr(state.S), ptr(slots), ptr(cu),
                ptr(positions), ptr(out), out.stride(0), float(spec.eps), nseq, T, H, D, Dv, act,
                chan[-1], *chan[:-1], U, L, l, rot if spec.rot_dims else None, 1 if bf else 0,
                stream(fused)), "linear_scan_channels64")
            return out
        if channel:
            ws, (wsS, wsG, cA) = workspace(dev, 4 * plan.n * H * D * Dv, 4 * plan.n * H * D, 4 * T * H * D)
            check(lib().eia_linear_scan_channels(
                ptr(fused), fused.stride(0), q_off, k_off, v_off, g_off, ptr(spec.inv_freq),
                spec.rot_dims, 1 if spec.rot_half else 0, float(spec.qscale), float(spec.kscale),
                float(spec.out_scale), ptr(norm_w), ptr(state.S), ptr(slots), ptr(cu),
                ptr(positions), ptr(out), out.stride(0), float(spec.eps), nseq, H, D, Dv, act,
                chan[-1], ptr(plan.chunks), ptr(plan.seq_first), plan.n, wsS, wsG,
                *chan[:-1], cA, 1 if bf else 0, stream(fused)), "linear_scan_channels")
            return out
        # (these chunks are longer than the plan's and found on the device)
        n, up16 = T // HEAD_CHUNK + nseq, lambda v: -(-v // 16) * 16
        ws, (U, G, m0, rot) = workspace(dev, 4 * n * H * up16(D) * (up16(Dv) + (4 if exp_gates else 0)),
                                        8 * n * H, 4 * n * H, 4 * T * spec.rot_dims)
        check(lib().eia_linear_scan_chunked(
            ptr(fused), fused.stride(0), q_off, k_off, v_off, g_off, i_off, f_off,
            ptr(spec.decay), ptr(spec.inv_freq), spec.rot_dims, 1 if spec.rot_half else 0,
            float(spec.qscale), float(spec.kscale), float(spec.cap), float(spec.out_scale),
            ptr(norm_w), ptr(state.S), ptr(state.n), ptr(state.m), ptr(slots), ptr(cu),
            ptr(positions), ptr(out), out.stride(0), float(spec.eps), nseq, T, H, D, Dv, mode, act,
            chan[-1], U, G, m0 if exp_gates else None, rot if spec.rot_dims else None, 1 if bf else 0,
            stream(fused)), "linear_scan_chunked")
        return out
    check(lib().eia_linear_scan(
        ptr(fused), fused.stride(0), q_off, k_off, v_off, g_off, i_off, f_off, ptr(spec.decay),
        ptr(spec.inv_freq), spec.rot_dims, 1 if spec.rot_half else 0, float(spec.qscale),
        float(spec.kscale), float(spec.cap), float(spec.out_scale), ptr(norm_w), ptr(state.S),
        ptr(state.n), ptr(state.m), ptr(slots), ptr(cu), ptr(positions), ptr(seq_lens), ptr(out),
        out.stride(0), float(spec.eps), nseq, H, D, Dv, mode,
        0 if spec.gate_act == "silu" else 1, *chan, 1 if bf else 0, stream(fused)), "linear_scan")
    return out
