// Linear-attention recurrences with one decay number per head and token (modes 0, 1) or per key
// channel and token (mode 2) on per-sequence state slots: a matrix state S [dk, dv] per head that
// every token scales and adds an outer product to,
//
//   S_t = a_t S_(t-1) + b_t k_t v_t^T,      o_t = S_t^T q_t        (the token sees itself)
//
// mode 0 (fixed decay, "retention"):  a_t = decay[h], b_t = 1.
// mode 1 (exponential gates with a running maximum, "matrix memory"): per head two gate
//   pre-activations x_i, x_f ride in the token's row;
//     i = cap tanh(x_i / cap),  f = logsigmoid(cap tanh(x_f / cap))   (cap 0: no cap),
//     m_t = max(f + m_(t-1), i),
//     a_t = exp(f + m_(t-1) - m_t),  b_t = exp(i - m_t),  n_t = a_t n_(t-1) + b_t k_t,
//     o_t <- o_t / (max(|n_t . q_t|, exp(-m_t)) + 1e-6);       m starts at 0, S and n at zero.
// mode 2 (a decay per key channel, "gated linear attention"): the row holds a low-rank branch of
//   R columns; z = A2 lo + bias per channel (fp32), a_t = sigmoid(z)^(1/tau) = exp(logsigmoid(z) /
//   tau) scales the state's ROWS (row i belongs to key channel i), b_t = 1.
// All: q and k may be rotated by the token's position on their first rot_dims entries (pairs
// (i, i + rot_dims/2) or (2i, 2i+1)), then scaled (qscale, kscale); each head's o is divided by
// its root mean square, multiplied by an optional weight and by silu or sigmoid of the gate
// columns, and by out_scale.
//
// q, k, v, the gate and the gate pre-activations are column ranges of one fused projection row
// per token (type T: bf16 or float).  Decays, gates, exponentials, the state, the normaliser and
// the head norm are fp32, as is mode 2's last decay product.  A sequence whose first row of the
// step is position 0 starts from the initial state whatever its slot held, so slots are reused
// without clearing.
// Batch layout: sequence s owns rows [cu[s], cu[s+1]) (cu == nullptr: row s).
#include <type_traits>

#include "eia_chunks.h"

struct ScanArgs {
  const void* x; long ld;                   // fused rows [rows, *]
  int q_off, k_off, v_off, g_off, i_off, f_off;
  const float* decay;                       // [H] (mode 0)
  const float* inv_freq; int rot_dims, rot_half;
  float qscale, kscale, cap, out_scale;
  const void* norm_w;                       // [H * Dv] or null
  float* S; float* N; float* M;             // [slots, H, D, Dv], [slots, H, D], [slots, H]
  const int* slots; const int* cu; const int* positions; const int* seq_lens;
  void* y; long ldy;                        // [rows, >= H * Dv]
  float eps;
  int H, D, Dv, mode, gate_act;
  // mode 2: low-rank columns, A2 transposed [R, H * D], bias [H * D], 1 / tau
  int lo_off, R; const float* a2t; const float* a2b; float inv_tau;
  int norm_h;                               // columns of norm_w per head: 0: [Dv] shared by heads
};

EIA_DEV float ls_logsigmoid(float z) { return -(log1pf(expf(-fabsf(z))) + fmaxf(-z, 0.f)); }

// log decay of channel j of head h for one row (mode 2)
template <typename T>
EIA_DEV float ls_chan_log(const ScanArgs& a, const T* xr, int h, int j) {
  const float* w = a.a2t + (long)h * a.D + j;
  float z = a.a2b ? a.a2b[(long)h * a.D + j] : 0.f;
#pragma unroll 8
  for (int r = 0; r < a.R; ++r) z += ld_f32<T>(xr, a.lo_off + r) * w[(long)r * a.H * a.D];
  return ls_logsigmoid(z) * a.inv_tau;
}

// One workgroup per (sequence, head), 4 x max(64, DMAX) threads: thread (qt, j) owns rows
// [qt DMAX/4, (qt+1) DMAX/4) of column j of S in registers and walks the sequence's tokens in
// order.  Tokens are staged TC at a time: q, k (rotated, scaled), v and the gate of TC tokens go
// to LDS, the gate recurrence of the chunk runs (its transcendentals in parallel over the
// tokens, the running maximum serially in one thread), then the state recurrence runs TC steps on
// LDS broadcasts leaving four partial outputs per token and column, which are summed, divided,
// normed and gated.  CH: a decay per key channel (mode 2), staged beside k.  NRM: the normaliser n
// rides along (every thread of a quarter keeps the quarter's rows of n; column 0 reports n . q).
template <typename T, int DMAX, bool NRM, bool CH>
__global__ void __launch_bounds__(4 * (DMAX < 64 ? 64 : DMAX))
linear_scan_kernel(ScanArgs a) {
  constexpr int DP = DMAX < 64 ? 64 : DMAX;          // threads per quarter
  constexpr int DQ = DMAX / 4;                       // dk rows per thread
  constexpr int TC = DMAX <= 64 ? 16 : DMAX <= 128 ? 8 : 4;
  constexpr int NWV = DP / 64;
  __shared__ __align__(16) float sq[TC][DMAX], sk[TC][DMAX];
  __shared__ float sv[TC][DMAX], sg[TC][DMAX], po[TC][4][DP];
  __shared__ __align__(16) float sal[CH ? TC : 1][CH ? DMAX : 1];
  __shared__ float sa[TC], sb[TC], se[TC], gi[TC], gf[TC], pn[TC][4];
  __shared__ float red[4][NWV];
  __shared__ float m_run;
  const int s = blockIdx.x, h = blockIdx.y, D = a.D, Dv = a.Dv;
  const int qt = threadIdx.x / DP, j = threadIdx.x % DP;
  const int slot = a.slots[s];
  if (slot < 0 || (a.seq_lens && a.seq_lens[s] <= 0)) return;
  const int lo = a.cu ? a.cu[s] : s, hi = a.cu ? a.cu[s + 1] : s + 1;
  if (hi <= lo) return;
  const bool fresh = a.positions[lo] == 0;
  const bool col = j < Dv;                           // this thread owns a state column
  const bool chan = j < D;                           // ... and stages a q / k channel
  float* Sg = a.S + ((long)slot * a.H + h) * D * Dv;
  float* Ng = NRM ? a.N + ((long)slot * a.H + h) * D : nullptr;
  const int i0 = qt * DQ;
  float S[DQ], Nn[NRM ? DQ : 1];
#pragma unroll
  for (int i = 0; i < DQ; ++i) {
    S[i] = (!fresh && i0 + i < D && col) ? Sg[(long)(i0 + i) * Dv + j] : 0.f;
    if constexpr (NRM) Nn[i] = (!fresh && i0 + i < D) ? Ng[i0 + i] : 0.f;
  }
  if (threadIdx.x == 0) m_run = (NRM && !fresh) ? a.M[(long)slot * a.H + h] : 0.f;
  const float dec = a.mode == 0 ? a.decay[h] : 1.f;
  const T* X = static_cast<const T*>(a.x);
  const T* NW = static_cast<const T*>(a.norm_w);
  T* Y = static_cast<T*>(a.y);
  const float nw = (NW && col) ? ld_f32<T>(NW, (long)h * a.norm_h + j) : 1.f;
  const float inv_dv = 1.0f / (float)Dv;
  // rotation of channel j: partner channel, the pair's frequency and the sign of the cross term
  const int hd = a.rot_dims >> 1;
  const bool rot = chan && j < a.rot_dims;
  int jp = j;
  float freq = 0.f, sgn = 0.f;
  if (rot) {
    const bool second = a.rot_half ? j >= hd : (j & 1);
    const int pi = a.rot_half ? (second ? j - hd : j) : (j >> 1);
    jp = a.rot_half ? (second ? j - hd : j + hd) : (j ^ 1);
    freq = a.inv_freq[pi];
    sgn = second ? 1.f : -1.f;
  }
  const long qc = a.q_off + (long)h * D, kc = a.k_off + (long)h * D;
  const long vc = a.v_off + (long)h * Dv, gc = a.g_off + (long)h * Dv;
  for (int base = lo; base < hi; base += TC) {
    const int nt = min(TC, hi - base);
    __syncthreads();                       // the previous chunk's LDS reads are done
    if (j < DMAX) {
#pragma unroll
      for (int tt = 0; tt < TC / 4; ++tt) {            // quarter qt stages tokens qt, qt + 4, ...
        const int t = tt * 4 + qt;
        if (t < nt) {
          const T* xr = X + (long)(base + t) * a.ld;
          float q = 0.f, k = 0.f, v = 0.f, g = 0.f;
          if (chan) {
            q = ld_f32<T>(xr, qc + j);
            k = ld_f32<T>(xr, kc + j);
            if (rot) {
              float sn, cs;
              sincosf((float)a.positions[base + t] * freq, &sn, &cs);
              q = q * cs + sgn * ld_f32<T>(xr, qc + jp) * sn;
              k = k * cs + sgn * ld_f32<T>(xr, kc + jp) * sn;
            }
            q *= a.qscale;
            k *= a.kscale;
          }
          if (col) {
            v = ld_f32<T>(xr, vc + j);
            g = ld_f32<T>(xr, gc + j);
          }
          sq[t][j] = q;
          sk[t][j] = k;
          if constexpr (CH) sal[t][j] = chan ? expf(ls_chan_log<T>(a, xr, h, j)) : 1.f;
          sv[t][j] = v;
          sg[t][j] = g;
        }
      }
    }
    if constexpr (NRM) {
      if (threadIdx.x < nt) {                          // log gates of the chunk's tokens
        const T* xr = X + (long)(base + threadIdx.x) * a.ld;
        const float xi = ld_f32<T>(xr, a.i_off + h), xf = ld_f32<T>(xr, a.f_off + h);
        gi[threadIdx.x] = a.cap > 0.f ? a.cap * tanhf(xi / a.cap) : xi;
        gf[threadIdx.x] = ls_logsigmoid(a.cap > 0.f ? a.cap * tanhf(xf / a.cap) : xf);
      }
      __syncthreads();
      if (threadIdx.x == 0) {                          // the running maximum, token by token
        float m = m_run;
        for (int t = 0; t < nt; ++t) {
          const float fm = gf[t] + m;
          m = fmaxf(fm, gi[t]);
          sa[t] = fm;                                  // f + m_(t-1)
          se[t] = m;
        }
        m_run = m;
      }
      __syncthreads();
      if (threadIdx.x < nt) {
        const float m = se[threadIdx.x];
        sa[threadIdx.x] = expf(sa[threadIdx.x] - m);
        sb[threadIdx.x] = expf(gi[threadIdx.x] - m);
        se[threadIdx.x] = expf(-m);
      }
    }
    __syncthreads();
    for (int t = 0; t < nt; ++t) {
      const float v = sv[t][j < DMAX ? j : 0];
      const float at = NRM ? sa[t] : dec, bt = NRM ? sb[t] : 1.f;
      float o = 0.f, nq = 0.f;
#pragma unroll
      for (int i = 0; i < DQ; ++i) {
        const float bk = bt * sk[t][i0 + i];
        S[i] = (CH ? sal[t][i0 + i] : at) * S[i] + bk * v;
        o += sq[t][i0 + i] * S[i];
        if constexpr (NRM) {
          Nn[i] = at * Nn[i] + bk;
          nq += sq[t][i0 + i] * Nn[i];
        }
      }
      po[t][qt][j] = o;
      if (NRM && j == 0) pn[t][qt] = nq;
    }
    __syncthreads();
    // quarter qt finishes tokens qt, qt + 4, ...: sum of the partials, normaliser, head RMS norm,
    // weight, gate
#pragma unroll
    for (int tt = 0; tt < TC / 4; ++tt) {
      const int t = tt * 4 + qt;
      const bool ok = t < nt && col;
      float o = ok ? po[t][0][j] + po[t][1][j] + po[t][2][j] + po[t][3][j] : 0.f;
      if constexpr (NRM) {
        if (t < nt) {
          const float nq = pn[t][0] + pn[t][1] + pn[t][2] + pn[t][3];
          o = o / (fmaxf(fabsf(nq), se[t]) + 1e-6f);
        }
      }
      float ss = wave_sum(o * o);
      if (NWV > 1) {
        __syncthreads();
        if ((j & 63) == 0) red[qt][j >> 6] = ss;
        __syncthreads();
        ss = 0.f;
#pragma unroll
        for (int x = 0; x < NWV; ++x) ss += red[qt][x];
      }
      if (ok) {
        const float g = sg[t][j];
        const float sig = 1.0f / (1.0f + expf(-g));
        const float gate = a.gate_act == 0 ? g * sig : sig;
        st_f32<T>(Y, (long)(base + t) * a.ldy + (long)h * Dv + j,
                  o / sqrtf(ss * inv_dv + a.eps) * nw * gate * a.out_scale);
      }
    }
  }
  if (col) {
#pragma unroll
    for (int i = 0; i < DQ; ++i)
      if (i0 + i < D) Sg[(long)(i0 + i) * Dv + j] = S[i];
  }
  if constexpr (NRM) {
    if (j == 0) {
#pragma unroll
      for (int i = 0; i < DQ; ++i)
        if (i0 + i < D) Ng[i0 + i] = Nn[i];
    }
    __syncthreads();
    if (threadIdx.x == 0) a.M[(long)slot * a.H + h] = m_run;
  }
}

// Decode rows (one token per sequence, dk and dv up to 128): one workgroup per (row, head).  The state
// is requested first, 16 bytes per access, and everything else -- q, k, v, the gates or the decays,
// each by threads of its own -- is formed while it is on its way; it is scaled, used and stored from the
// registers that it arrives in.  Thread (rg, cg) holds rows rg, rg + RG, ... of columns 4 cg ..
//
// Bound by the state's traffic (64 rows, 16 heads of 128 x 128, exponential gates: 22 us for 134 MB on an
// MI355X) and, at a few rows, by one round of dependent loads (6 us).  The kernel above, made to walk
// tokens, took 61 and 15 us: 4-byte state accesses, the gates and decays in a chain of their own behind
// barriers, and with dk < dv half of its threads without rows.
template <typename T, int DM, int W, bool NRM, bool CH>       // dk <= DM, dv <= W
__global__ void __launch_bounds__(256)
linear_decode_kernel(ScanArgs a) {
  constexpr int CG = W / 4, RG = 256 / CG, NR = DM / RG;
  __shared__ float sq[DM], sk[DM], sal[CH ? DM : 1];
  __shared__ __align__(16) float sv[W], po[RG][W];
  __shared__ float sgate[3], red[4], rn[4];
  const int s = blockIdx.x, h = blockIdx.y, D = a.D, Dv = a.Dv, tid = threadIdx.x;
  const int slot = a.slots[s];
  if (slot < 0 || (a.seq_lens && a.seq_lens[s] <= 0)) return;
  const bool fresh = a.positions[s] == 0;
  const int cg = tid % CG, rg = tid / CG, c0 = min(4 * cg, Dv - 4);     // (Dv % 4 == 0)
  float* Sg = a.S + ((long)slot * a.H + h) * D * Dv;
  f32x4 S[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i)
    S[i] = *reinterpret_cast<const f32x4*>(Sg + (long)min(rg + RG * i, D - 1) * Dv + c0);
  const T* xr = static_cast<const T*>(a.x) + (long)s * a.ld;
  const bool chan = tid < D, col = tid < Dv;
  float n = 0.f, q = 0.f, k = 0.f;
  if (tid < DM) {
    if (chan) {
      if (NRM && !fresh) n = a.N[((long)slot * a.H + h) * D + tid];
      const long qc = a.q_off + (long)h * D, kc = a.k_off + (long)h * D;
      q = ld_f32<T>(xr, qc + tid);
      k = ld_f32<T>(xr, kc + tid);
      if (tid < a.rot_dims) {
        const int hd = a.rot_dims >> 1;
        const bool second = a.rot_half ? tid >= hd : (tid & 1);
        const int pi = a.rot_half ? (second ? tid - hd : tid) : (tid >> 1);
        const int jp = a.rot_half ? (second ? tid - hd : tid + hd) : (tid ^ 1);
        const float sgn = second ? 1.f : -1.f;
        float sn, cs;
        sincosf((float)a.positions[s] * a.inv_freq[pi], &sn, &cs);
        q = q * cs + sgn * ld_f32<T>(xr, qc + jp) * sn;
        k = k * cs + sgn * ld_f32<T>(xr, kc + jp) * sn;
      }
      q *= a.qscale;
      k *= a.kscale;
    }
    sq[tid] = q;
    sk[tid] = k;
  }
  if (tid < W) sv[tid] = col ? ld_f32<T>(xr, a.v_off + (long)h * Dv + tid) : 0.f;
  if constexpr (CH) {
    const int j = tid - 128;
    if (j >= 0 && j < DM) sal[j] = j < D ? expf(ls_chan_log<T>(a, xr, h, j)) : 1.f;
  } else if (NRM && tid == 255) {
    const float xi = ld_f32<T>(xr, a.i_off + h), xf = ld_f32<T>(xr, a.f_off + h);
    const float gi = a.cap > 0.f ? a.cap * tanhf(xi / a.cap) : xi;
    const float gf = ls_logsigmoid(a.cap > 0.f ? a.cap * tanhf(xf / a.cap) : xf);
    const float fm = gf + (fresh ? 0.f : a.M[(long)slot * a.H + h]), m = fmaxf(fm, gi);
    sgate[0] = expf(fm - m);
    sgate[1] = expf(gi - m);
    sgate[2] = expf(-m);
    a.M[(long)slot * a.H + h] = m;
  }
  const float g = (tid < W && col) ? ld_f32<T>(xr, a.g_off + (long)h * Dv + tid) : 0.f;
  const T* NW = static_cast<const T*>(a.norm_w);
  const float nw = (NW && tid < W && col) ? ld_f32<T>(NW, (long)h * a.norm_h + tid) : 1.f;
  __syncthreads();
  const float at = NRM ? sgate[0] : CH ? 1.f : a.decay[h], bt = NRM ? sgate[1] : 1.f;
  if constexpr (NRM) {
    n = at * n + bt * k;
    if (chan) a.N[((long)slot * a.H + h) * D + tid] = n;
    const float nq = wave_sum(chan ? q * n : 0.f);
    if ((tid & 63) == 0) rn[tid >> 6] = nq;
  }
  const f32x4 v = *reinterpret_cast<const f32x4*>(&sv[c0]);
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int r = rg + RG * i;
    if (r < D) {
      const f32x4 z = fresh ? f32x4{0.f, 0.f, 0.f, 0.f} : S[i];
      const f32x4 u = (CH ? sal[r] : at) * z + (bt * sk[r]) * v;
      o += sq[r] * u;
      if (4 * cg < Dv) *reinterpret_cast<f32x4*>(Sg + (long)r * Dv + c0) = u;
    }
  }
  if (4 * cg < Dv) *reinterpret_cast<f32x4*>(&po[rg][4 * cg]) = o;
  __syncthreads();
  float y = 0.f;
  if (tid < W && col) {
#pragma unroll
    for (int x = 0; x < RG; ++x) y += po[x][tid];
    if constexpr (NRM) y = y / (fmaxf(fabsf(rn[0] + rn[1] + rn[2] + rn[3]), sgate[2]) + 1e-6f);
  }
  const float ss = wave_sum(y * y);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  if (tid < W && col) {
    const float sig = 1.0f / (1.0f + expf(-g));
    const float all = W == 64 ? red[0] : red[0] + red[1];
    st_f32<T>(static_cast<T*>(a.y), (long)s * a.ldy + (long)h * Dv + tid,
              y / sqrtf(all * (1.0f / (float)Dv) + a.eps) * nw * (a.gate_act == 0 ? g * sig : sig) *
                  a.out_scale);
  }
}

template <typename T>
static void linear_decode(const ScanArgs& a, int nseq, hipStream_t st) {
  const dim3 grid(nseq, a.H), block(256);
#define LD_GO(DM, W, N, C) \
  hipLaunchKernelGGL((linear_decode_kernel<T, DM, W, N, C>), grid, block, 0, st, a)
#define LD_MODES(DM, W)                                                                             \
  do {                                                                                              \
    if (a.mode == 1) LD_GO(DM, W, true, false);                                                     \
    else if (a.mode == 2) LD_GO(DM, W, false, true);                                                \
    else LD_GO(DM, W, false, false);                                                                \
  } while (0)
  if (a.D <= 64) { if (a.Dv <= 64) LD_MODES(64, 64); else LD_MODES(64, 128); }
  else { if (a.Dv <= 64) LD_MODES(128, 64); else LD_MODES(128, 128); }
#undef LD_MODES
#undef LD_GO
}

// x: fused rows (bf16 when is_bf16, else fp32) holding the q [H*D], k [H*D], v [H*Dv] and gate
// [H*Dv] columns at the given offsets (mode 1: also the H input-gate and H forget-gate
// pre-activations at i_off / f_off); y [rows, >= H*Dv] of the same type.
EIA_API int eia_linear_scan(const void* x, long ld, int q_off, int k_off, int v_off, int g_off,
                            int i_off, int f_off, const float* decay, const float* inv_freq,
                            int rot_dims, int rot_half, float qscale, float kscale, float cap,
                            float out_scale, const void* norm_w, float* S, float* N, float* M,
                            const int* slots, const int* cu, const int* positions,
                            const int* seq_lens, void* y, long ldy, float eps, int nseq, int H,
                            int D, int Dv, int mode, int gate_act, int lo_off, int R,
                            const float* a2t, const float* a2b, float inv_tau, int norm_h,
                            int is_bf16, hipStream_t st) {
  if (nseq < 0 || H < 1 || D < 1 || Dv < 1 || !x || !y || !S || !slots || !positions ||
      mode < 0 || mode > 2 || (mode == 2 && (R < 1 || !a2t)) || (mode == 0 && !decay) ||
      (mode == 1 && (!N || !M || cap < 0.f)) ||
      rot_dims < 0 || rot_dims > D || (rot_dims & 1) || (rot_dims && !inv_freq) ||
      (gate_act != 0 && gate_act != 1))
    return EIA_BAD_SHAPE;
  const int dm = D > Dv ? D : Dv;
  if (dm > 256) return EIA_UNSUPPORTED;
  if (nseq == 0) return EIA_OK;
  ScanArgs a{x, ld, q_off, k_off, v_off, g_off, i_off, f_off, decay, inv_freq, rot_dims, rot_half,
             qscale, kscale, cap, out_scale, norm_w, S, N, M, slots, cu, positions, seq_lens, y,
             ldy, eps, H, D, Dv, mode, gate_act, lo_off, R, a2t, a2b, inv_tau, norm_h};
  if (!cu && D <= 128 && Dv <= 128 && Dv % 4 == 0 && reinterpret_cast<uintptr_t>(S) % 16 == 0) {
    if (is_bf16) linear_decode<bf16_t>(a, nseq, st); else linear_decode<float>(a, nseq, st);
    EIA_LAUNCH_CHECK();
  }
  dim3 grid(nseq, H);
#define LS_LAUNCH(TT, DM, NR, CHN)                                                                  \
  hipLaunchKernelGGL((linear_scan_kernel<TT, DM, NR, CHN>), grid, dim3(4 * (DM < 64 ? 64 : DM)), 0, \
                     st, a)
#define LS_SIZES(TT, NR, CHN)                        \
  do {                                               \
    if (dm <= 32) LS_LAUNCH(TT, 32, NR, CHN);        \
    else if (dm <= 64) LS_LAUNCH(TT, 64, NR, CHN);   \
    else if (dm <= 128) LS_LAUNCH(TT, 128, NR, CHN); \
    else LS_LAUNCH(TT, 256, NR, CHN);                \
  } while (0)
#define LS_MODES(TT)                                 \
  do {                                               \
    if (mode == 1) LS_SIZES(TT, true, false);        \
    else if (mode == 2) LS_SIZES(TT, false, true);   \
    else LS_SIZES(TT, false, false);                 \
  } while (0)
  if (is_bf16) LS_MODES(bf16_t); else LS_MODES(float);
#undef LS_MODES
#undef LS_SIZES
#undef LS_LAUNCH
  EIA_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------------------------
// Chunk-parallel form for prompt portions, one decay per head and token (modes 0 and 1), dk, dv <=
// 128.  The token-by-token kernel above walks a sequence with one workgroup per head; here a
// sequence's rows are cut into chunks of LK tokens and, with l_t = log2 a_t, m_t = log2 b_t,
//
//   U   = sum_s 2^(m_s + sum_(x>s) l_x) k_s v_s^T                         (1) per chunk, in parallel
//   S' = 2^(sum_x l_x) S + U                                              (2) a sequence's chunks in order
//   o_t = 2^(sum_(x<=t) l_x) S^T q_t
//         + sum_(s<=t) 2^(m_s + sum_(s<x<=t) l_x) (q_t . k_s) v_s         (3) per chunk, in parallel
//
// (the normaliser n is one more state column, n_t . q_t the row sum of the same weights).  Sums of l
// run over 16-token blocks and over whole blocks, inside a block over just the tokens between: every
// exponent is a sum of what it covers, so it is <= 0 and keeps its precision.  (Differences of two running
// sums inside a block: 9.9e-7 instead of 1.8e-7 against 64 bits, fp32 gates that close hard.)  Angles of rotated heads
// come from a table.  Chunks are found on the device (eia_chunks.h).
//
// The running maximum of mode 1 is a scan over pairs (sum of f, maximum behind it).  (1) forms U relative to the maximum
// of the chunk's own gates and leaves the chunk's pair, (2) walks the pairs beside the states and brings both to the
// carried maximum, (3) forms its gates again from the maximum before its chunk.  (A pass of its own for the gates of all
// rows, one workgroup per sequence and head, was bound by the latency of reads a projected row apart: 11 us and a launch,
// where the gates now cost (1) 5 us and (3) nothing.  The op below 124.5 -> 111.9 us; S against 64 bits, four shapes,
// 1.53e-7 .. 1.75e-7 -> 1.29e-7 .. 1.58e-7.)
//
// Rows of bf16: all products take bf16 operands, fp32 factors as the sum of three (split3).  Values, and
// unrotated keys and queries, are exact as they are, so most products are three of 16x16x32 at 3/16 of the matrix
// cycles that fp32 products took, and none is less precise: S against 64 bits 0.98e-7 .. 2.4e-7 where fp32
// products left 1.45e-7 .. 2.6e-7 (fewer roundings of the sums).  Rows of fp32, and chunks in which a sum is not
// finite, which the parts of a split cannot follow, take fp32 products (ls_state_fp32, ls_out_fp32).
//
// 128-token chunks: the states between chunks are the larger part of the memory
// traffic (4 passes over chunks x H x dk x dv floats), and halving their number costs less than the
// longer sums inside a chunk add.
// Four prompts of 1000 .. 2000 tokens (6688 rows), 16 heads of 128, mode 1, bf16 take 34 + 21 +
// 54 us on an MI355X ((1), (2), (3)); in fp32 products (1) and (3) took 57 + 103 us.  Bound by the
// workspace and the rows, which (1), (2) and (3) move at 3.4, 5.5 and 3.6 TB/s, and by the steps of
// a workgroup, which reads, splits and multiplies in turn: half of (3)'s wave cycles wait, and vector instructions
// fill 0.4 of the others.  All heads of a chunk run side by side in (1) and (3), so
// that whole rows are read together, and (3) asks for its queries before it waits for the gates: 135 -> 129 us for the
// op; three rotated prompts of up to 2700 tokens 188 -> 178, five of up to 1100 of 32 heads of 64 78 -> 77.  What the
// normaliser, the norm and the gate read is asked for at once (four rounds behind each other: 129 -> 124 us, 178 -> 177,
// 77 -> 76).  (3) asks for unrotated keys and values before the last products of the state, and forms what is one number
// a token in one lane of the sixteen that hold it (61.4 -> 57.0 us; the op, eight heads, 4000 tokens 47.0 -> 45.3, four
// rotated prompts of up to 2000 173 -> 168).  Asking for the gates before the last products spills: 64 us.  (1) asks for unrotated rows a half ahead, the first before it waits for the gates (33.2 -> 30.0 us, before it
// formed the gates itself).
constexpr int LK = 128;                     // tokens per chunk
constexpr float LS_LOG2E = 1.4426950408889634f;

struct KChunkArgs {
  float* U;                                 // [numbers, H, DP, UW]: contribution, then state before
  float* G;                                 // [numbers, H]: sums of l; mode 1: [.., 2] a chunk's pair (f, m)
  float* m0;                                // [numbers, H]: the running maximum before the chunk (mode 1)
  float* la;                                // [rows, H * D]: log2 a (mode 2)
  float2* rot;                              // [rows, rot_dims / 2]: cos, sin
  int nseq, rows, DP, VP, UW;               // UW: VP, and in mode 1 four more (the normaliser, 0, 0, 0)
};

// The chunk of number x; false where there is none or the sequence is skipped.
EIA_DEV bool ls_chunk(const ScanArgs& a, int nseq, int x, int& s, int& row0, int& n) {
  return chunk_of<LK>(a.cu, nseq, x, s, row0, n) && a.slots[s] >= 0;
}

// Angles of the rotated channels, shared by all heads and by the q and k of (1) and (3).
__global__ void __launch_bounds__(256)
ls_angles_kernel(ScanArgs a, KChunkArgs c) {
  const int hd = a.rot_dims >> 1;
  const long u = (long)blockIdx.x * 256 + threadIdx.x;
  if (u >= (long)c.rows * hd) return;
  float sn, cs;
  sincosf((float)a.positions[u / hd] * a.inv_freq[u % hd], &sn, &cs);
  c.rot[u] = make_float2(cs, sn);
}

// Eight channels i .. i + 7 (i % 8 == 0) of a q or k head of one row, rotated, not scaled; zero past
// D.  VEC: 16-byte loads (D, the rotated channels and every offset are multiples of eight).
template <typename T, bool VEC, bool ROT>
EIA_DEV void ls_head8(const ScanArgs& a, const KChunkArgs& c, long row, long off, int i, float (&v)[8]) {
  const T* x = static_cast<const T*>(a.x) + row * a.ld + off;
  auto get = [&](int j, float (&o)[8]) {
    if constexpr (VEC) {
      alignas(16) T t[8];
      const f32x4* p = reinterpret_cast<const f32x4*>(x + (j < a.D ? j : 0));
#pragma unroll
      for (int e = 0; e < (int)(sizeof(T) / 2); ++e) *reinterpret_cast<f32x4*>(&t[e * 16 / sizeof(T)]) = p[e];
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = j < a.D ? (float)t[e] : 0.f;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = j + e < a.D ? (float)x[j + e] : 0.f;
    }
  };
  get(i, v);
  if constexpr (ROT) {
    const int rd = a.rot_dims, hd = rd >> 1;
    const float2* r = c.rot + row * hd;
    if (i >= rd) return;
    if (a.rot_half) {
      if (VEC) {
        const bool second = i >= hd;
        const int j = second ? i - hd : i;
        float p[8];
        get(second ? j : j + hd, p);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = v[e] * r[j + e].x + (second ? p[e] : -p[e]) * r[j + e].y;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int ch = i + e;
          if (ch < rd) {
            const bool second = ch >= hd;
            const int j = second ? ch - hd : ch;
            const float p = (float)x[second ? j : j + hd];
            v[e] = v[e] * r[j].x + (second ? p : -p) * r[j].y;
          }
        }
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        if (VEC || i + e < rd) {
          const float2 cs = r[(i + e) >> 1];
          const float u = v[e], w = v[e + 1];
          v[e] = u * cs.x - w * cs.y;
          v[e + 1] = w * cs.x + u * cs.y;
        }
      }
    }
  }
}

// Places in LDS tiles [tokens][MX] where four tokens' runs of sixteen channels meet: the key rows of (3),
// in units of 16 / sizeof(KT) entries; fp32 rows lie as tile_at has them.
template <int MX, typename KT> EIA_DEV int ls_kat(int t, int i) {
  if constexpr (sizeof(KT) == 4) return tile_at<MX>(t, i);
  else return t * MX + (i ^ (MX == 128 ? (t & 15) << 3 : ((t >> 1) & 7) << 3));
}
// value rows: four tokens' runs meet as rows 4 g + e
template <int MX> EIA_DEV int ls_vat(int t, int i) { return t * MX + (i ^ (((t >> 2) & 1) * (MX / 2))); }

// Four value columns of a staged row as fp32.
template <typename T> EIA_DEV f32x4 ls_v4(const T* p) {
  if constexpr (sizeof(T) == 4) return *reinterpret_cast<const f32x4*>(p);
  else {
    const bf16x4 v = *reinterpret_cast<const bf16x4*>(p);
    return f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
  }
}

// Tokens t0 .. t0 + N - 1 of the chunk's values to LDS, zero past the chunk and past Dv.
template <typename T, bool VEC, int MX, int N, int NT>
EIA_DEV void ls_stage_v(const ScanArgs& a, int row0, int n, int h, int t0, T* sv) {
  constexpr int E = VEC ? 16 / (int)sizeof(T) : 1;
  const T* X = static_cast<const T*>(a.x) + a.v_off + (long)h * a.Dv;
#pragma unroll
  for (int u = threadIdx.x; u < N * MX / E; u += NT) {
    const int t = u / (MX / E), i = E * (u % (MX / E));
    const bool ok = t0 + t < n && i < a.Dv;
    const T* p = X + (long)(row0 + (ok ? t0 + t : 0)) * a.ld + (ok ? i : 0);
    if constexpr (VEC) {
      const f32x4 z = {0.f, 0.f, 0.f, 0.f};
      const f32x4 v = *reinterpret_cast<const f32x4*>(p);
      *reinterpret_cast<f32x4*>(sv + ls_vat<MX>(t, i)) = ok ? v : z;
    } else {
      sv[ls_vat<MX>(t, i)] = ok ? *p : (T)0.f;
    }
  }
}

// What the logs of the chunk's token threadIdx.x are formed from (threads 0 .. LK - 1): the decay or the two gate
// pre-activations of the token and, for the second wave, of the token 64 before it.
struct LsGates {
  unsigned xi[2], xf[2];                    // as they lie in memory: a conversion here would wait for them
  float decay;
};
template <typename T> EIA_DEV LsGates ls_log_load(const ScanArgs& a, int row0, int n, int h) {
  using Bits = typename std::conditional<sizeof(T) == 2, unsigned short, unsigned>::type;
  LsGates g = {};
  const int t = threadIdx.x;
  if (a.mode == 0) {
    g.decay = a.decay[h];
  } else if (__builtin_amdgcn_readfirstlane(t) < LK) {
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      const Bits* x = static_cast<const Bits*>(a.x) + (long)(row0 + min(y ? t & 63 : t, n - 1)) * a.ld + h;
      g.xi[y] = x[a.i_off];
      g.xf[y] = x[a.f_off];
    }
  }
  return g;
}
// Mode 1: log decay l and log weight b of the token, m the running maximum with it, from the maximum m0 before the
// chunk (-inf: none, what lies before the chunk weighs nothing).  m_t = max(f_t + m_(t-1), i_t) is a scan over pairs
// (sum of f, maximum behind it).  -> the pair up to and with the token.
template <typename T>
EIA_DEV float2 ls_log_gates(const ScanArgs& a, int n, LsGates g, float m0, float& l, float& b, float& m) {
  const int t = threadIdx.x, lane = t & 63;
  asm volatile("" : "+v"(g.xi[0]), "+v"(g.xi[1]), "+v"(g.xf[0]), "+v"(g.xf[1]));     // (keeps the conversions here)
  auto value = [](unsigned u) { return __uint_as_float(sizeof(T) == 2 ? u << 16 : u); };
  auto soft = [&](float x) { return a.cap > 0.f ? a.cap * tanhf(x / a.cap) : x; };
  auto join = [](float2 p, float2 q) { return make_float2(p.x + q.x, fmaxf(p.y + q.x, q.y)); };
  auto scan = [&](float2 q) {               // inclusive over the lanes
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const float2 up = make_float2(__shfl_up(q.x, o, 64), __shfl_up(q.y, o, 64));
      if (lane >= o) q = join(up, q);
    }
    return q;
  };
  // a token that forgets everything and adds nothing (f = i = -inf), or whose f is no number, leaves none, in the state
  // as in its outputs
  auto shut = [](float f, float i) { return !(f > -INFINITY) && !(f == -INFINITY && i > -INFINITY); };
  auto pair = [&](float f, float i) { return make_float2(shut(f, i) ? __builtin_nanf("") : f, i); };
  const float2 none = make_float2(0.f, -INFINITY);
  const float gi = soft(value(g.xi[0])), gf = ls_logsigmoid(soft(value(g.xf[0])));
  float2 first = none;                      // of the 64 tokens before the second wave's
  if (t >= 64) {
    first = scan(lane < n ? pair(ls_logsigmoid(soft(value(g.xf[1]))), soft(value(g.xi[1]))) : none);
    first = make_float2(__shfl(first.x, 63, 64), __shfl(first.y, 63, 64));
  }
  const float2 p = join(first, scan(t < n ? pair(gf, gi) : none));
  m = fmaxf(m0 + p.x, p.y);
  const float up = __shfl_up(m, 1, 64), before = lane ? up : fmaxf(m0 + first.x, first.y);
  // (not gf + before - m: where nothing new is met the maximum moves with the decays, and the roundings of its
  // steps would add up.  S against 64 bits 2.5e-7 instead of 1.6e-7)
  const float fm = pair(gf, gi).x + before;
  l = t >= n || before == -INFINITY || fm >= gi ? 0.f : fm - gi;
  b = t >= n ? 0.f : shut(gf, gi) ? __builtin_nanf("") : m > -INFINITY ? gi - m : gi;      // (gi: -inf or no number)
  return p;
}
// Sums of l over 16-token blocks: pre up to and with a token, suf behind it, tot of whole blocks;
// mb: log2 b, sl: l, mx: m (mode 1).  Threads 0 .. LK - 1.  pair: where mode 1's pair of the chunk goes, or null.
template <typename T>
EIA_DEV void ls_chunk_logs(const ScanArgs& a, int n, const LsGates& g, float m0, float* pre, float* suf, float* tot,
                           float* mb, float* sl, float* mx, float2* pair) {
  const int t = threadIdx.x;
  if (t >= LK) return;
  float l, b = 0.f;
  if (a.mode == 0) {
    l = t < n ? logf(g.decay) : 0.f;
  } else {
    const float2 p = ls_log_gates<T>(a, n, g, m0, l, b, mx[t]);
    if (pair && t == LK - 1) *pair = p;
  }
  l *= LS_LOG2E;
  b *= LS_LOG2E;
  l = l < -150.f ? -150.f : l;                         // (2^-150 is zero; what is no number stays so)
  sl[t] = l;
  float p = l, s = l;
  const int t16 = t & 15;
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) {
    const float up = __shfl_up(p, o, 16), dn = __shfl_down(s, o, 16);
    if (t16 >= o) p += up;
    if (t16 + o < 16) s += dn;
  }
  const float after = __shfl_down(s, 1, 16);
  pre[t] = p;
  suf[t] = t16 == 15 ? 0.f : after;
  mb[t] = b;
  if (t16 == 15) tot[t >> 4] = p;
}

// Sums of l over the tokens s < x <= t of one 16-token block, for the lane's query t = lane % 16 and keys
// s = 4 (lane / 16) + i: the rest of the key's four, the fours between, the query's four up to it.
EIA_DEV f32x4 ls_inside(const float* l, int lane) {
  const f32x4* four = reinterpret_cast<const f32x4*>(l);
  const int g4 = lane >> 4, f4 = lane >> 2 & 3, t4 = lane & 3;
  const f32x4 kf = four[g4], qf = four[f4], f1 = four[1], f2 = four[2];
  float up = qf[0];
#pragma unroll
  for (int j = 1; j < 4; ++j) up += j <= t4 ? qf[j] : 0.f;
  if (g4 < 1 && f4 > 1) up += f1[0] + f1[1] + f1[2] + f1[3];
  if (g4 < 2 && f4 > 2) up += f2[0] + f2[1] + f2[2] + f2[3];
  const int last = g4 == f4 ? t4 : 3;
  f32x4 e;
  float rest = g4 < f4 ? up : 0.f;
#pragma unroll
  for (int j = 3; j >= 0; --j) {
    e[j] = rest;
    rest += j <= last ? kf[j] : 0.f;
  }
  return e;
}

// What (1) and (3) share of a chunk: its rows and the sums of l in LDS.
struct LsChunk {
  int row0, n, h;
  const float *pre, *suf, *mb, *tot, *sl;
};

// The weight of token tk's key in what the chunk adds to the state, 0 past the chunk.
EIA_DEV float ls_key_weight(const ScanArgs& a, const LsChunk& k, int tk) {
  float e = k.mb[tk] + k.suf[tk];
  for (int b = (tk >> 4) + 1; b < LK / 16; ++b) e += k.tot[b];
  return tk < k.n ? a.kscale * __builtin_amdgcn_exp2f(e) : 0.f;
}
// The weighted key of token tk, channels i .. i + 7: what it adds to the state after the chunk.
template <typename T, bool VEC, bool ROT>
EIA_DEV void ls_weighted_key(const ScanArgs& a, const KChunkArgs& c, const LsChunk& k, int tk, int i, float (&v)[8]) {
  ls_head8<T, VEC, ROT>(a, c, k.row0 + min(tk, k.n - 1), a.k_off + (long)k.h * a.D, i, v);
  const float wt = ls_key_weight(a, k, tk);
#pragma unroll
  for (int x = 0; x < 8; ++x) v[x] = tk < k.n ? v[x] * wt : 0.f;
}

// U in fp32 products: wave w forms rows 16 w ..  Tokens come in two halves of 64.  A lane of a product over
// tokens holds columns 64 x + 4 (lane % 16) + j in tile 4 x + j, here and in (3).
template <typename T, bool VEC, bool ROT, int MX>
EIA_DEV void ls_state_fp32(const ScanArgs& a, const KChunkArgs& c, const LsChunk& k, long at, unsigned char* lds) {
  float* sk = reinterpret_cast<float*>(lds);
  T* sv = reinterpret_cast<T*>(sk + 64 * MX);
  const int row0 = k.row0, n = k.n, h = k.h, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int l16 = lane & 15, g4 = lane >> 4;
  f32x4 acc[MX / 16];
  float un = 0.f;                                      // normaliser row 16 w + l16
#pragma unroll
  for (int j = 0; j < MX / 16; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int half = 0; half < 2; ++half) {
    const int t0 = 64 * half;
    if (t0 >= n) break;
    __syncthreads();                                   // logs are there; the first half was read
    ls_stage_v<T, VEC, MX, 64, 512>(a, row0, n, h, t0, sv);
#pragma unroll
    for (int u = threadIdx.x; u < 64 * MX / 8; u += 512) {
      const int t = u / (MX / 8), i = 8 * (u % (MX / 8)), tk = t0 + t;
      float v[8];
      ls_weighted_key<T, VEC, ROT>(a, c, k, tk, i, v);
#pragma unroll
      for (int x = 0; x < 8; x += 4)
        *reinterpret_cast<f32x4*>(sk + tile_at<MX>(t, i + x)) = f32x4{v[x], v[x + 1], v[x + 2], v[x + 3]};
    }
    __syncthreads();
    if (16 * w >= c.DP) continue;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      if (t0 + 16 * b >= n) break;
      f32x4 ka, vb[MX / 16];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int t = 16 * b + 4 * g4 + e;
        ka[e] = sk[tile_at<MX>(t, 16 * w + l16)];
#pragma unroll
        for (int x = 0; x < MX / 64; ++x) {
          const f32x4 v = ls_v4<T>(sv + ls_vat<MX>(t, 64 * x + 4 * l16));
#pragma unroll
          for (int j = 0; j < 4; ++j) vb[4 * x + j][e] = v[j];
        }
      }
#pragma unroll
      for (int j = 0; j < MX / 16; ++j) acc[j] = mfma_f32_k16(ka, vb[j], acc[j]);
      un += ka[0] + ka[1] + ka[2] + ka[3];
    }
  }
  if (16 * w >= c.DP) return;
  float* U = c.U + (at * c.DP + 16 * w + 4 * g4) * c.UW;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int x = 0; x < MX / 64; ++x)
      if (64 * x + 4 * l16 < c.VP)
        *reinterpret_cast<f32x4*>(U + (long)i * c.UW + 64 * x + 4 * l16) =
            f32x4{acc[4 * x][i], acc[4 * x + 1][i], acc[4 * x + 2][i], acc[4 * x + 3][i]};
  }
  if (a.mode == 1) {
    un += __shfl_xor(un, 16, 64);
    un += __shfl_xor(un, 32, 64);
    if (g4 == 0)
      *reinterpret_cast<f32x4*>(c.U + (at * c.DP + 16 * w + l16) * c.UW + c.VP) = f32x4{un, 0.f, 0.f, 0.f};
  }
}

// U in bf16 products, for bf16 rows: the values are operands as they are, the weighted keys in three parts
// (split3).  Wave (cw, dw) forms MX / 4 rows and MX / 2 columns, U transposed in its registers; the
// normaliser is the product with ones.  Rows of an LDS tile are 32 bytes more than a multiple of the banks
// apart, so that the transposing reads of eight rows meet all of them.  false: something was not finite
// (uniform over the workgroup; nothing was written).
template <bool VEC, bool ROT, int MX, typename Logs>
EIA_DEV bool ls_state_bf16(const ScanArgs& a, const KChunkArgs& c, const LsChunk& k, long at, unsigned char* lds,
                           Logs&& logs) {
  constexpr int PITCH = MX + 16, PLANE = 64 * PITCH, NA = MX / 32, NB = MX / 64, NU = 64 * MX / 8 / 512;
  constexpr bool AHEAD = VEC && !ROT;                  // a half's rows are on their way during what stands before it
  bf16_t* sk = reinterpret_cast<bf16_t*>(lds);         // [3][64][PITCH]
  bf16_t* sv = sk + 3 * PLANE;                         // [64][PITCH]
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, g4 = lane >> 4, c0 = MX / 4 * (w & 3), d0 = MX / 2 * (w >> 2);
  const bool live = c0 < c.DP, norm = a.mode == 1 && d0 == 0;
  const bf16_t* X = static_cast<const bf16_t*>(a.x) + a.v_off + (long)k.h * a.Dv;
  const int ut = threadIdx.x / (MX / 8), ui = 8 * (threadIdx.x % (MX / 8));        // a thread's first token, its channels
  constexpr int UT = 512 / (MX / 8);
  bf16x8 kr[NU], vr[NU];
  auto fetch = [&](int t0) {
    const bf16_t* xk = static_cast<const bf16_t*>(a.x) + a.k_off + (long)k.h * a.D + (ui < a.D ? ui : 0);
    const bf16_t* xv = X + (ui < a.Dv ? ui : 0);
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const long r = (long)(k.row0 + min(t0 + ut + UT * u, k.n - 1)) * a.ld;
      kr[u] = *reinterpret_cast<const bf16x8*>(xk + r);
      vr[u] = *reinterpret_cast<const bf16x8*>(xv + r);
    }
  };
  if constexpr (AHEAD) fetch(0);
  logs();
  bf16x8 ones;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = (bf16_t)1.f;
  f32x4 acc[NA][NB], un[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    un[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NA; ++i) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  for (int t0 = 0; t0 < k.n; t0 += 64) {
    __syncthreads();                                   // logs are there; the first half was read
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int t = ut + UT * u;
      const bool ok = t0 + t < k.n && ui < a.Dv;
      bf16x8 v;
      float kw[8];
      if constexpr (AHEAD) {
        const bool in = t0 + t < k.n && ui < a.D;
        const float wt = ls_key_weight(a, k, t0 + t);
#pragma unroll
        for (int e = 0; e < 8; ++e) kw[e] = in ? (float)kr[u][e] * wt : 0.f;
        v = vr[u];
        if (!ok) v = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
      } else {
        const bf16_t* p = X + (long)(k.row0 + (ok ? t0 + t : 0)) * a.ld + (ok ? ui : 0);
        if constexpr (VEC) {
          v = *reinterpret_cast<const bf16x8*>(p);
          if (!ok) v = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = ok && ui + e < a.Dv ? p[e] : (bf16_t)0.f;
        }
        ls_weighted_key<bf16_t, VEC, ROT>(a, c, k, t0 + t, ui, kw);
      }
      *reinterpret_cast<bf16x8*>(sv + t * PITCH + ui) = v;
      bf16x8 part[3];
      split3(kw, part);
#pragma unroll
      for (int p3 = 0; p3 < 3; ++p3) *reinterpret_cast<bf16x8*>(sk + p3 * PLANE + t * PITCH + ui) = part[p3];
    }
    if constexpr (AHEAD) {
      if (t0 + 64 < k.n) fetch(t0 + 64);
    }
    __syncthreads();
    if (!live) continue;
#pragma unroll
    for (int b = 0; b < 64; b += 32) {
      if (t0 + b >= k.n) break;
      const int at0 = (b + 4 * g4 + (l16 >> 2)) * PITCH + 4 * (l16 & 3);
      bf16x8 kf[3][NB];
#pragma unroll
      for (int p3 = 0; p3 < 3; ++p3)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const bf16_t* q = sk + p3 * PLANE + at0 + c0 + 16 * j;
          kf[p3][j] = lds_columns(q, q + 16 * PITCH);
        }
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        const bf16_t* q = sv + at0 + d0 + 16 * i;
        const bf16x8 vf = lds_columns(q, q + 16 * PITCH);
#pragma unroll
        for (int p3 = 2; p3 >= 0; --p3)
#pragma unroll
          for (int j = 0; j < NB; ++j) acc[i][j] = mfma_bf16_k32(vf, kf[p3][j], acc[i][j]);
      }
      if (norm) {
#pragma unroll
        for (int p3 = 2; p3 >= 0; --p3)
#pragma unroll
          for (int j = 0; j < NB; ++j) un[j] = mfma_bf16_k32(ones, kf[p3][j], un[j]);
      }
    }
  }
  mfma_settle(un);
#pragma unroll
  for (int i = 0; i < NA; ++i) mfma_settle(acc[i]);
  bool bad = false;
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    bad |= !(fabsf(un[j][0]) < INFINITY);
#pragma unroll
    for (int i = 0; i < NA; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) bad |= !(fabsf(acc[i][j][e]) < INFINITY);
  }
  if (__syncthreads_or(bad)) return false;
  if (!live) return true;
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    if (c0 + 16 * j >= c.DP) break;
    float* U = c.U + (at * c.DP + c0 + 16 * j + l16) * c.UW;
#pragma unroll
    for (int i = 0; i < NA; ++i)
      if (d0 + 16 * i < c.VP) *reinterpret_cast<f32x4*>(U + d0 + 16 * i + 4 * g4) = acc[i][j];
    if (norm && g4 == 0) *reinterpret_cast<f32x4*>(U + c.VP) = f32x4{un[j][0], 0.f, 0.f, 0.f};
  }
  return true;
}

// (1) Eight waves, two workgroups on a CU: 128 registers a lane.  Rotated bf16 rows of any alignment need 204 and
// spilled 122 of them; they take a CU to themselves: four prompts of up to 2000 tokens, 16 heads of 128, 371 -> 355
// us.  (fp32 rows, rotated: aligned 274 us with 128 registers, 289 with the 130 they would like; unaligned, where
// 128 spill 9, 492 and 516.)
template <typename T, bool VEC, bool ROT, int MX>
__global__ void __launch_bounds__(512, sizeof(T) == 2 && ROT && !VEC && MX == 128 ? 2 : 4)
ls_chunk_state_kernel(ScanArgs a, KChunkArgs c) {
  constexpr bool BF = sizeof(T) == 2;
  constexpr int FP32 = 64 * MX * (4 + (int)sizeof(T)), SPLIT = BF ? 4 * 64 * (MX + 16) * 2 : 0;
  __shared__ __align__(16) unsigned char tiles[FP32 > SPLIT ? FP32 : SPLIT];
  __shared__ float pre[LK], suf[LK], mb[LK], tot[LK / 16], sl[LK], mx[LK];
  int s, row0, n;
  if (!ls_chunk(a, c.nseq, chunk_number(), s, row0, n)) return;
  const int h = blockIdx.x;
  const LsGates g = ls_log_load<T>(a, row0, n, h);
  const long at = (long)chunk_number() * a.H + h;
  const LsChunk k{row0, n, h, pre, suf, mb, tot, sl};
  auto logs = [&] {
    ls_chunk_logs<T>(a, n, g, -INFINITY, pre, suf, tot, mb, sl, mx, reinterpret_cast<float2*>(c.G) + at);
  };
  if constexpr (BF) {
    if (!ls_state_bf16<VEC, ROT, MX>(a, c, k, at, tiles, logs)) ls_state_fp32<T, VEC, ROT, MX>(a, c, k, at, tiles);
  } else {
    logs();
    ls_state_fp32<T, VEC, ROT, MX>(a, c, k, at, tiles);
  }
  if (a.mode == 0 && threadIdx.x == 0) {
    float sum = 0.f;
    for (int b = 0; b < LK / 16; ++b) sum += tot[b];
    c.G[at] = sum;
  }
}

// (2) Four columns of a state row per thread; the slot receives the state after the last chunk.
__global__ void __launch_bounds__(256)
ls_chunk_scan_kernel(ScanArgs a, KChunkArgs c) {
  const int s = blockIdx.x, h = blockIdx.y;
  const int slot = a.slots[s], lo = a.cu[s], hi = a.cu[s + 1];
  const int u4 = blockIdx.z * 256 + threadIdx.x, q = c.UW / 4, i = u4 / q, j = 4 * (u4 % q);
  if (slot < 0 || hi <= lo || i >= c.DP) return;
  const long x0 = lo / LK + s;
  const int nc = (hi - lo + LK - 1) / LK;
  const bool norm = j >= c.VP;                         // the normaliser's columns
  const int nj = norm ? 1 : a.Dv;
  float* Sg = norm ? a.N + ((long)slot * a.H + h) * a.D + i
                   : a.S + (((long)slot * a.H + h) * a.D + i) * a.Dv + j;
  const int j0 = norm ? 0 : j;
  f32x4 S = {0.f, 0.f, 0.f, 0.f};
  if (a.positions[lo] != 0 && i < a.D) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (j0 + k < nj) S[k] = Sg[k];
  }
  const long us = (long)a.H * c.DP * c.UW;
  float* U = c.U + (x0 * a.H + h) * c.DP * c.UW + (long)i * c.UW + j;
  if (a.mode == 0) {
    chunk_walk(U, us, c.G + x0 * a.H + h, a.H, nc, S);
  } else {                                             // U stands relative to the chunk's own maximum
    const float2* G = reinterpret_cast<const float2*>(c.G) + x0 * a.H + h;
    float* m0 = c.m0 + x0 * a.H + h;                   // ((3) leaves the slot's new maximum: others here still read it)
    float m = a.positions[lo] == 0 ? 0.f : a.M[(long)slot * a.H + h];
    chunk_walk_with<float2>(U, us, nc, S, [&](int x) { return G[(long)x * a.H]; }, [&](int x, float2 p, f32x4 u) {
      if (u4 == 0) m0[(long)x * a.H] = m;
      const float mn = fmaxf(m + p.x, p.y);
      S = S * __builtin_amdgcn_exp2f((m + p.x - mn) * LS_LOG2E) + u * __builtin_amdgcn_exp2f((p.y - mn) * LS_LOG2E);
      m = mn;
    });
  }
  if (i < a.D) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (j0 + k < nj) Sg[k] = S[k];
  }
}

// (3) Eight waves; a wave forms the outputs of 16 tokens.  A later block meets more keys: waves i
// and i + 4, which share a SIMD, take blocks that add up to the same work.
//
// Sums of a wave's queries in fp32 products (o: query 4 (lane / 16) + i, columns as above; rs: this lane's
// part of the row sum of query lane % 16).
template <typename T, bool VEC, bool ROT, int MX>
EIA_DEV void ls_out_fp32(const ScanArgs& a, const KChunkArgs& c, const LsChunk& k, bool state, unsigned char* tiles,
                         float* sn, f32x4 (&o)[MX / 16], float& rs) {
  // unrotated bf16 keys and queries meet as they are; else both are fp32
  constexpr bool BF = sizeof(T) == 2 && !ROT;
  using KT = typename std::conditional<BF, T, float>::type;
  constexpr bool PRE = BF && VEC;            // keys fetched while the state is used
  float* sS = reinterpret_cast<float*>(tiles);         // [MX][MX] the state, then keys and values
  KT* sk = reinterpret_cast<KT*>(tiles);
  T* sv = reinterpret_cast<T*>(sk + LK * MX);
  const int row0 = k.row0, n = k.n, h = k.h, D = a.D;
  const float *pre = k.pre, *suf = k.suf, *mb = k.mb, *tot = k.tot, *sl = k.sl;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int w = wv < 4 ? wv : 11 - wv, l16 = lane & 15, g4 = lane >> 4, t0 = 16 * w;
  if (state) {                                         // straight to LDS, 1 KB per access
    const float* S = c.U + ((long)chunk_number() * a.H + h) * c.DP * c.UW;
#pragma unroll
    for (int u = 0; u < MX * MX / 256 / 8; ++u) {
      const int at = 256 * (8 * u + wv), r = (at + 4 * lane) / MX, d = (at + 4 * lane) % MX;
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(S + (long)min(r, c.DP - 1) * c.UW +
                                                          (d < c.VP ? d : 0)),
          (__attribute__((address_space(3))) void*)(sS + __builtin_amdgcn_readfirstlane(at)), 16, 0, 0);
    }
    if (a.mode == 1 && threadIdx.x < MX)
      sn[threadIdx.x] = S[(long)min((int)threadIdx.x, c.DP - 1) * c.UW + c.VP];
  }
  // this lane's query: channels 32 x + 8 g4 + e
  const int tq = t0 + l16;
  typedef KT KT8 __attribute__((ext_vector_type(8)));
  KT8 qf[MX / 32];
#pragma unroll
  for (int x = 0; x < MX / 32; ++x) {
    float v[8];
    ls_head8<T, VEC, ROT>(a, c, row0 + min(tq, n - 1), a.q_off + (long)h * D, 32 * x + 8 * g4, v);
#pragma unroll
    for (int e = 0; e < 8; ++e) qf[x][e] = (KT)v[e];
  }
  constexpr int NU = LK * MX / 8 / 512;                // units of 8 channels per thread
  f32x4 kp[PRE ? NU : 1];                              // (the values too: 84 bytes spilled, 109 us)
  const T* X0 = static_cast<const T*>(a.x) + (long)row0 * a.ld;
  if constexpr (PRE) {
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int at = threadIdx.x + 512 * u, t = min(at / (MX / 8), n - 1), i = 8 * (at % (MX / 8));
      const T* r = X0 + (long)t * a.ld;
      kp[u] = *reinterpret_cast<const f32x4*>(r + a.k_off + (long)h * D + (i < D ? i : 0));
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
#pragma unroll
  for (int j = 0; j < MX / 16; ++j) o[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  rs = 0.f;
  const float pq = pre[tq];
  if (state && t0 < n) {
    float front = 0.f;                                 // l of the blocks before the query's
    for (int b = 0; b < w; ++b) front += tot[b];
    const float eq = a.qscale * __builtin_amdgcn_exp2f(pq + front);
#pragma unroll
    for (int x = 0; x < MX / 32; ++x)
#pragma unroll
      for (int e = 0; e < 8; e += 4) {
        const int i = 32 * x + 8 * g4 + e;
        if (32 * x >= c.DP) break;
        const f32x4 qa = f32x4{(float)qf[x][e], (float)qf[x][e + 1], (float)qf[x][e + 2],
                               (float)qf[x][e + 3]} * eq;
#pragma unroll
        for (int y = 0; y < 4; ++y) {
          if (a.mode == 1) rs += qa[y] * sn[i + y];
#pragma unroll
          for (int z = 0; z < MX / 64; ++z) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(sS + (i + y) * MX + 64 * z + 4 * l16);
#pragma unroll
            for (int j = 0; j < 4; ++j)
              o[4 * z + j] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[y], v[j], o[4 * z + j], 0, 0, 0);
          }
        }
      }
  }
  __syncthreads();                                     // the state was read
  if constexpr (PRE) {
    ls_stage_v<T, VEC, MX, LK, 512>(a, row0, n, h, 0, sv);
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int at = threadIdx.x + 512 * u, t = at / (MX / 8), i = 8 * (at % (MX / 8));
      *reinterpret_cast<f32x4*>(sk + ls_kat<MX, KT>(t, i)) = t < n && i < D ? kp[u] : zero;
    }
  } else {
    ls_stage_v<T, VEC, MX, LK, 512>(a, row0, n, h, 0, sv);
#pragma unroll
    for (int u = threadIdx.x; u < LK * MX / 8; u += 512) {
      const int t = u / (MX / 8), i = 8 * (u % (MX / 8));
      float v[8];
      ls_head8<T, VEC, ROT>(a, c, row0 + min(t, n - 1), a.k_off + (long)h * a.D, i, v);
      if constexpr (BF) {
        bf16x8 b;
#pragma unroll
        for (int e = 0; e < 8; ++e) b[e] = t < n ? (bf16_t)v[e] : (bf16_t)0.f;
        *reinterpret_cast<bf16x8*>(sk + ls_kat<MX, KT>(t, i)) = b;
      } else {
#pragma unroll
        for (int x = 0; x < 8; x += 4)
          *reinterpret_cast<f32x4*>(sk + ls_kat<MX, KT>(t, i + x)) =
              t < n ? f32x4{v[x], v[x + 1], v[x + 2], v[x + 3]} : f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
  }
  __syncthreads();
  if (t0 >= n) return;
  const float qk = a.qscale * a.kscale;
  float back = 0.f;                                    // l from the end of block b to the query's
  for (int b = w; b >= 0; --b) {
    // weights are formed transposed, keys x queries: their registers are the A operand of P v
    f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < MX / 32; ++x) {
      if constexpr (BF) {
        const bf16x8 kb = *reinterpret_cast<const bf16x8*>(sk + ls_kat<MX, KT>(16 * b + l16, 32 * x + 8 * g4));
        p = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kb, qf[x], p, 0, 0, 0);
      } else {
#pragma unroll
        for (int e = 0; e < 8; e += 4)
          p = mfma_f32_k16(*reinterpret_cast<const f32x4*>(sk + ls_kat<MX, KT>(16 * b + l16, 32 * x + 8 * g4 + e)),
                           f32x4{qf[x][e], qf[x][e + 1], qf[x][e + 2], qf[x][e + 3]}, p);
      }
    }
    f32x4 e;
    if (b == w) e = ls_inside(sl + t0, lane);
    else e = *reinterpret_cast<const f32x4*>(suf + 16 * b + 4 * g4) + (pq + back);
    e += *reinterpret_cast<const f32x4*>(mb + 16 * b + 4 * g4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[i] = 16 * b + 4 * g4 + i <= tq ? p[i] * qk * __builtin_amdgcn_exp2f(e[i]) : 0.f;
      rs += p[i];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int x = 0; x < MX / 64; ++x) {
        const f32x4 v = ls_v4<T>(sv + ls_vat<MX>(16 * b + 4 * g4 + e, 64 * x + 4 * l16));
#pragma unroll
        for (int j = 0; j < 4; ++j)
          o[4 * x + j] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[e], v[j], o[4 * x + j], 0, 0, 0);
      }
    if (b < w) back += tot[b];
  }
}

// The same sums in bf16 products, for bf16 rows: rotated queries and keys, the state and the weights P are
// three parts (split3), all others operands as they are.  The state goes through LDS in halves of 64 rows,
// split where it is written.  Tile 4 x + j of the sums takes columns 64 x + 4 l + j, which lie together in
// LDS, so that the transposing reads find them.  false: something was not finite (uniform).
template <bool VEC, bool ROT, int MX> struct LsOutTiles {
  static constexpr int NQ = ROT ? 3 : 1, PITCH = MX + 16, SPLANE = 64 * PITCH, KPLANE = LK * MX;
  static constexpr int S = 3 * SPLANE * 2, KV = (NQ * KPLANE + LK * PITCH) * 2, BYTES = S > KV ? S : KV;
};
// Sixteen columns from 16 u on of row r to the places of their tiles.
template <int MX> EIA_DEV int ls_col16(int u) { return 64 * (u >> 2) + 4 * (u & 3); }

template <bool VEC, bool ROT, int MX, typename Logs>
EIA_DEV bool ls_out_bf16(const ScanArgs& a, const KChunkArgs& c, const LsChunk& k, bool state, unsigned char* tiles,
                         const float* sn, f32x4 (&o)[MX / 16], float& rs, Logs&& logs) {
  using L = LsOutTiles<VEC, ROT, MX>;
  constexpr int NQ = L::NQ, PITCH = L::PITCH, NX = MX / 32;
  bf16_t* sS = reinterpret_cast<bf16_t*>(tiles);       // [3][64][PITCH], then keys and values
  bf16_t* sk = sS;                                     // [NQ][LK][MX]
  bf16_t* sv = sk + NQ * L::KPLANE;                    // [LK][PITCH]
  const int row0 = k.row0, n = k.n, h = k.h, D = a.D;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int w = wv < 4 ? wv : 11 - wv, l16 = lane & 15, g4 = lane >> 4, t0 = 16 * w, tq = t0 + l16;
  const bf16_t* X0 = static_cast<const bf16_t*>(a.x) + (long)row0 * a.ld;
  // rows 64 x + r of the state, columns 16 u ..: one unit per thread and half
  const int su = threadIdx.x % (MX / 16), sr = threadIdx.x / (MX / 16);
  f32x4 sf[4];
  auto fetch = [&](int x) {
    if (!state || sr >= 64) return;
    const float* S = c.U + (((long)chunk_number() * a.H + h) * c.DP + min(64 * x + sr, c.DP - 1)) * c.UW +
                     (16 * su < c.VP ? 16 * su : 0);
#pragma unroll
    for (int e = 0; e < 4; ++e) sf[e] = *reinterpret_cast<const f32x4*>(S + 4 * e);
  };
  bf16x8 qf[NQ][NX];                                   // this lane's query: channels 32 x + 8 g4 + e
  auto queries = [&](bool use) {                       // use: q . n, else nothing but qf
    float z = 0.f;
#pragma unroll
    for (int x = 0; x < NX; ++x) {
      float v[8];
      ls_head8<bf16_t, VEC, ROT>(a, c, row0 + min(tq, n - 1), a.q_off + (long)h * D, 32 * x + 8 * g4, v);
      if constexpr (ROT) {
        bf16x8 part[3];
        split3(v, part);
#pragma unroll
        for (int p = 0; p < 3; ++p) qf[p][x] = part[p];
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) qf[0][x][e] = (bf16_t)v[e];
      }
      if (use) {
#pragma unroll
        for (int e = 0; e < 8; ++e) z += v[e] * sn[32 * x + 8 * g4 + e];
      }
    }
    return z;
  };
  const bool norm = a.mode == 1 && state;
  if constexpr (!ROT) queries(false);                  // (asked for before the state and the logs are waited for)
  fetch(0);
  logs();
  __syncthreads();
  float nq = 0.f;
  if constexpr (ROT) {
    nq = queries(norm);
  } else if (norm) {
#pragma unroll
    for (int x = 0; x < NX; ++x)
#pragma unroll
      for (int e = 0; e < 8; ++e) nq += (float)qf[0][x][e] * sn[32 * x + 8 * g4 + e];
  }
#pragma unroll
  for (int j = 0; j < MX / 16; ++j) o[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  rs = 0.f;
  auto dot = [&](const bf16x8 (&x)[NQ], const bf16x8 (&y)[3], f32x4 z) {       // y in three parts
    if constexpr (NQ == 3) {
      z = mfma_bf16_k32(x[0], y[2], z);
      z = mfma_bf16_k32(x[2], y[0], z);
      z = mfma_bf16_k32(x[1], y[1], z);
      z = mfma_bf16_k32(x[0], y[1], z);
      z = mfma_bf16_k32(x[1], y[0], z);
    } else {
      z = mfma_bf16_k32(x[0], y[2], z);
      z = mfma_bf16_k32(x[0], y[1], z);
    }
    return mfma_bf16_k32(x[0], y[0], z);
  };
  const float pq = k.pre[tq];
  // keys and values of unrotated rows are on their way during the last products of the state
  constexpr bool AHEAD = VEC && !ROT;
  constexpr int NV = LK * MX / 16 / 512, NK = 2 * NV, UT = 512 / (MX / 8);
  const int vt = threadIdx.x / (MX / 16), vu = threadIdx.x % (MX / 16);          // a thread's first value row, its columns
  const int kt = threadIdx.x / (MX / 8), ki = 8 * (threadIdx.x % (MX / 8));
  bf16x8 vr[AHEAD ? NV : 1][2], kr[AHEAD ? NK : 1];
  auto ahead = [&] {
    if constexpr (AHEAD) {
      const bf16_t* xv = X0 + a.v_off + (long)h * a.Dv;
      const bf16_t* xk = X0 + a.k_off + (long)h * D + (ki < D ? ki : 0);
#pragma unroll
      for (int u = 0; u < NV; ++u) {
        const bf16_t* p = xv + (long)min(vt + 2 * UT * u, n - 1) * a.ld;
        vr[u][0] = *reinterpret_cast<const bf16x8*>(p + (16 * vu < a.Dv ? 16 * vu : 0));
        vr[u][1] = *reinterpret_cast<const bf16x8*>(p + (16 * vu + 8 < a.Dv ? 16 * vu + 8 : 0));
      }
#pragma unroll
      for (int u = 0; u < NK; ++u) kr[u] = *reinterpret_cast<const bf16x8*>(xk + (long)min(kt + UT * u, n - 1) * a.ld);
    }
  };
  if (!state) ahead();
  if (state) {
#pragma unroll
    for (int x = 0; x < MX / 64; ++x) {
      if (x) __syncthreads();                          // the half before was read
      if (sr < 64) {
        const int at = sr * PITCH + (ls_col16<MX>(su) ^ (MX == 128 ? (sr & 8) << 3 : 0));
        const bool ok = 64 * x + sr < c.DP;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          bf16x2 lo[3], hi[3];
          split3(ok ? sf[0][j] : 0.f, ok ? sf[1][j] : 0.f, lo[0], lo[1], lo[2]);
          split3(ok ? sf[2][j] : 0.f, ok ? sf[3][j] : 0.f, hi[0], hi[1], hi[2]);
#pragma unroll
          for (int p = 0; p < 3; ++p)
            *reinterpret_cast<bf16x4*>(sS + p * L::SPLANE + at + 16 * j) = bf16x4{lo[p][0], lo[p][1], hi[p][0], hi[p][1]};
        }
      }
      if (x + 1 < MX / 64) fetch(x + 1);               // (on its way during these products)
      else ahead();
      __syncthreads();
      if (t0 >= n) continue;
#pragma unroll
      for (int y = 0; y < 2; ++y) {
        if (64 * x + 32 * y >= c.DP) break;
        bf16x8 qx[NQ];
#pragma unroll
        for (int p = 0; p < NQ; ++p) qx[p] = qf[p][2 * x + y];
        // (rows 8 apart meet the other half of the banks)
        const int r = (32 * y + 8 * g4 + (l16 >> 2)) * PITCH, turn = MX == 128 ? (g4 & 1) << 6 : 0;
#pragma unroll
        for (int j = 0; j < MX / 16; ++j) {
          bf16x8 sp[3];
#pragma unroll
          for (int p = 0; p < 3; ++p) {
            const bf16_t* q = sS + p * L::SPLANE + r + ((16 * j + 4 * (l16 & 3)) ^ turn);
            sp[p] = lds_columns(q, q + 4 * PITCH);
          }
          o[j] = dot(qx, sp, o[j]);
        }
      }
    }
    float front = 0.f;                                 // l of the blocks before the query's
    for (int b = 0; b < w; ++b) front += k.tot[b];
    const float eq = a.qscale * __builtin_amdgcn_exp2f(pq + front);
    rs = nq * eq;
    f32x4 er;
#pragma unroll
    for (int i = 0; i < 4; ++i) er[i] = __shfl(eq, 4 * g4 + i, 64);
    mfma_settle(o);
#pragma unroll
    for (int j = 0; j < MX / 16; ++j) o[j] *= er;
    __syncthreads();                                   // the state was read
  }
#pragma unroll
  for (int u = 0; u < NV; ++u) {                       // values: sixteen columns of a row
    const int t = vt + 2 * UT * u;
    bf16x8 v0, v1;
    if constexpr (VEC) {
      const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
      if constexpr (AHEAD) {
        v0 = vr[u][0];
        v1 = vr[u][1];
      } else {
        const bf16_t* p = X0 + (long)min(t, n - 1) * a.ld + a.v_off + (long)h * a.Dv;
        v0 = *reinterpret_cast<const bf16x8*>(p + (16 * vu < a.Dv ? 16 * vu : 0));
        v1 = *reinterpret_cast<const bf16x8*>(p + (16 * vu + 8 < a.Dv ? 16 * vu + 8 : 0));
      }
      if (t >= n || 16 * vu >= a.Dv) v0 = zero;
      if (t >= n || 16 * vu + 8 >= a.Dv) v1 = zero;
    } else {
      const bf16_t* p = X0 + (long)min(t, n - 1) * a.ld + a.v_off + (long)h * a.Dv;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        v0[e] = t < n && 16 * vu + e < a.Dv ? p[16 * vu + e] : (bf16_t)0.f;
        v1[e] = t < n && 16 * vu + 8 + e < a.Dv ? p[16 * vu + 8 + e] : (bf16_t)0.f;
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *reinterpret_cast<bf16x4*>(sv + t * PITCH + ls_col16<MX>(vu) + 16 * j) = bf16x4{v0[j], v0[4 + j], v1[j], v1[4 + j]};
  }
#pragma unroll
  for (int u = 0; u < NK; ++u) {
    const int t = kt + UT * u;
    if constexpr (AHEAD) {
      if (t >= n || ki >= D) kr[u] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
      *reinterpret_cast<bf16x8*>(sk + ls_kat<MX, bf16_t>(t, ki)) = kr[u];
    } else {
      float v[8];
      ls_head8<bf16_t, VEC, ROT>(a, c, row0 + min(t, n - 1), a.k_off + (long)h * D, ki, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = t < n ? v[e] : 0.f;
      if constexpr (ROT) {
        bf16x8 part[3];
        split3(v, part);
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<bf16x8*>(sk + p * L::KPLANE + ls_kat<MX, bf16_t>(t, ki)) = part[p];
      } else {
        bf16x8 b;
#pragma unroll
        for (int e = 0; e < 8; ++e) b[e] = (bf16_t)v[e];
        *reinterpret_cast<bf16x8*>(sk + ls_kat<MX, bf16_t>(t, ki)) = b;
      }
    }
  }
  __syncthreads();
  bool bad = false;
  if (t0 < n) {
    const float qk = a.qscale * a.kscale;
    float back = 0.f;                                  // l from the end of block b to the query's
    // weights of block b, transposed (keys x queries): their registers are an operand of P v
    auto weights = [&](int b) {
      f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int x = 0; x < NX; ++x) {
        bf16x8 kb[NQ], qx[NQ];
#pragma unroll
        for (int y = 0; y < NQ; ++y) {
          kb[y] = *reinterpret_cast<const bf16x8*>(sk + y * L::KPLANE + ls_kat<MX, bf16_t>(16 * b + l16, 32 * x + 8 * g4));
          qx[y] = qf[y][x];
        }
        if constexpr (ROT) p = dot(kb, qx, p);
        else p = mfma_bf16_k32(kb[0], qx[0], p);
      }
      f32x4 e;
      if (b == w) e = ls_inside(k.sl + t0, lane);
      else e = *reinterpret_cast<const f32x4*>(k.suf + 16 * b + 4 * g4) + (pq + back);
      e += *reinterpret_cast<const f32x4*>(k.mb + 16 * b + 4 * g4);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[i] = 16 * b + 4 * g4 + i <= tq ? p[i] * qk * __builtin_amdgcn_exp2f(e[i]) : 0.f;
        rs += p[i];
      }
      if (b < w) back += k.tot[b];
      return p;
    };
    for (int b = w; b >= 0; b -= 2) {                  // two blocks of keys to a product
      const f32x4 p0 = weights(b), p1 = b ? weights(b - 1) : f32x4{0.f, 0.f, 0.f, 0.f};
      const float p8[8] = {p0[0], p0[1], p0[2], p0[3], p1[0], p1[1], p1[2], p1[3]};
      bf16x8 pp[3];
      split3(p8, pp);
      const bf16_t* v0 = sv + (16 * b + 4 * g4 + (l16 >> 2)) * PITCH + 4 * (l16 & 3);
      const bf16_t* v1 = v0 - (b ? 16 * PITCH : 0);
#pragma unroll
      for (int j = 0; j < MX / 16; ++j) {
        const bf16x8 vf = lds_columns(v0 + 16 * j, v1 + 16 * j);
#pragma unroll
        for (int p = 2; p >= 0; --p) o[j] = mfma_bf16_k32(pp[p], vf, o[j]);
      }
    }
    mfma_settle(o);
#pragma unroll
    for (int j = 0; j < MX / 16; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) bad |= !(fabsf(o[j][i]) < INFINITY);
  }
  return !__syncthreads_or(bad);
}

// Two workgroups on a CU where the LDS holds two: 128 registers a lane, of which aligned, unrotated heads of 128 spill 7.
// One with all registers: four gated prompts of up to 2000 tokens, 16 heads, the op 123 -> 150 us.  Heads of 64, unrotated:
// three, 80 registers (82, and two, without the bound: five prompts of up to 1100 tokens, 32 heads, 76 -> 82 us).
template <typename T, bool VEC, bool ROT, int MX>
__global__ void __launch_bounds__(512, sizeof(T) == 2 && VEC && !ROT && MX == 64 ? 6 : 4)
ls_chunk_out_kernel(ScanArgs a, KChunkArgs c) {
  constexpr bool BF = sizeof(T) == 2;
  constexpr int KV = LK * MX * ((BF && !ROT ? 2 : 4) + (int)sizeof(T)), FP32 = KV > MX * MX * 4 ? KV : MX * MX * 4;
  constexpr int SPLIT = BF ? LsOutTiles<VEC, ROT, MX>::BYTES : 0;
  __shared__ __align__(16) unsigned char tiles[FP32 > SPLIT ? FP32 : SPLIT];
  __shared__ __align__(16) float pre[LK], suf[LK], mb[LK], sl[LK], tot[LK / 16], mx[LK], sn[MX];
  int s, row0, n;
  if (!ls_chunk(a, c.nseq, chunk_number(), s, row0, n)) return;
  const int h = blockIdx.x, lane = threadIdx.x & 63, wv = threadIdx.x >> 6, Dv = a.Dv;
  const int w = wv < 4 ? wv : 11 - wv, l16 = lane & 15, g4 = lane >> 4, t0 = 16 * w;
  const long at = (long)chunk_number() * a.H + h;
  const LsGates g = ls_log_load<T>(a, row0, n, h);
  const float m0 = a.mode == 1 ? c.m0[at] : 0.f;
  const bool state = row0 != a.cu[s] || a.positions[a.cu[s]] != 0;   // (else a fresh sequence: S = 0)
  float sv = 0.f;                                      // (stored with the logs: a store here would wait for it)
  if (a.mode == 1 && __builtin_amdgcn_readfirstlane(threadIdx.x) < MX)
    sv = c.U[(at * c.DP + min((int)threadIdx.x, c.DP - 1)) * c.UW + c.VP];
  const LsChunk k{row0, n, h, pre, suf, mb, tot, sl};
  auto logs = [&] {
    ls_chunk_logs<T>(a, n, g, m0, pre, suf, tot, mb, sl, mx, nullptr);
    if (threadIdx.x < MX) sn[threadIdx.x] = sv;
  };
  f32x4 o[MX / 16];
  float rs;
  if constexpr (BF) {
    if (!ls_out_bf16<VEC, ROT, MX>(a, c, k, state, tiles, sn, o, rs, logs))
      ls_out_fp32<T, VEC, ROT, MX>(a, c, k, state, tiles, sn, o, rs);
  } else {
    logs();
    __syncthreads();
    ls_out_fp32<T, VEC, ROT, MX>(a, c, k, state, tiles, sn, o, rs);
  }
  if (a.mode == 1 && threadIdx.x == n - 1 && row0 + n == a.cu[s + 1]) a.M[(long)a.slots[s] * a.H + h] = mx[n - 1];
  if (t0 >= n) return;
  const T* X = static_cast<const T*>(a.x);
  const T* NW = static_cast<const T*>(a.norm_w);
  T* Y = static_cast<T*>(a.y);
  typedef T T4 __attribute__((ext_vector_type(4)));
  // what a lane's four tokens need besides, asked for together
  T4 gt[4][MX / 64], nw[MX / 64];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const T* gp = X + (row0 + min(t0 + 4 * g4 + i, n - 1)) * a.ld + a.g_off + (long)h * Dv;
#pragma unroll
    for (int x = 0; x < MX / 64; ++x) {
      const int d = 64 * x + 4 * l16;
      if constexpr (VEC) gt[i][x] = *reinterpret_cast<const T4*>(gp + (d < Dv ? d : 0));
      else {
#pragma unroll
        for (int j = 0; j < 4; ++j) gt[i][x][j] = gp[min(d + j, Dv - 1)];
      }
    }
  }
  if (NW) {
#pragma unroll
    for (int x = 0; x < MX / 64; ++x)
#pragma unroll
      for (int j = 0; j < 4; ++j) nw[x][j] = NW[(long)h * a.norm_h + min(64 * x + 4 * l16 + j, Dv - 1)];
  } else {
#pragma unroll
    for (int x = 0; x < MX / 64; ++x) nw[x] = T4{(T)1.f, (T)1.f, (T)1.f, (T)1.f};
  }
  // normaliser, head RMS norm, weight, gate.  What is one number a token is formed by one lane of the sixteen that
  // hold it.
  float ss[4], den = 1.f;
  if (a.mode == 1) {
    rs += __shfl_xor(rs, 16, 64);                      // n_t . q_t of query l16
    rs += __shfl_xor(rs, 32, 64);
    den = 1.0f / (fmaxf(fabsf(rs), expf(-mx[min(t0 + l16, n - 1)])) + 1e-6f);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float di = a.mode == 1 ? __shfl(den, 4 * g4 + i, 64) : 1.f;
    ss[i] = 0.f;
#pragma unroll
    for (int j = 0; j < MX / 16; ++j) {
      const bool col = 64 * (j >> 2) + 4 * l16 + (j & 3) < Dv;
      o[j][i] = col ? o[j][i] * di : 0.f;              // (padded columns read column 0 of S)
      ss[i] += o[j][i] * o[j][i];
    }
    ss[i] = row16_sum(ss[i]);
  }
  const float lo = l16 & 1 ? ss[1] : ss[0], hi = l16 & 1 ? ss[3] : ss[2];
  const float mine = a.out_scale / sqrtf((l16 & 2 ? hi : lo) / (float)Dv + a.eps);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = t0 + 4 * g4 + i;
    const float inv = __shfl(mine, 16 * g4 + i, 64);
    if (t >= n) continue;
#pragma unroll
    for (int x = 0; x < MX / 64; ++x) {
      const int d = 64 * x + 4 * l16;
      if (d >= Dv) continue;
      T* yp = Y + (row0 + t) * a.ldy + (long)h * Dv + d;
      T4 y4;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float g = (float)gt[i][x][j];
        const float sig = sizeof(T) == 2 ? __builtin_amdgcn_rcpf(1.0f + __expf(-g)) : 1.0f / (1.0f + expf(-g));
        y4[j] = (T)(o[4 * x + j][i] * inv * (float)nw[x][j] * (a.gate_act == 0 ? g * sig : sig));
      }
      if constexpr (VEC) *reinterpret_cast<T4*>(yp) = y4;
      else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (d + j < Dv) yp[j] = y4[j];
      }
    }
  }
}

template <typename T, bool VEC, bool ROT, int MX>
static void ls_chunked(const ScanArgs& a, const KChunkArgs& c, hipStream_t st) {
  const dim3 gc = chunk_grid(c.rows / LK + c.nseq, a.H), gs(c.nseq, a.H);
  const dim3 gz(c.nseq, a.H, (c.DP * c.UW / 4 + 255) / 256);
  if (ROT) {
    const long u = (long)c.rows * (a.rot_dims >> 1);
    hipLaunchKernelGGL(ls_angles_kernel, dim3((unsigned)((u + 255) / 256)), dim3(256), 0, st, a, c);
  }
  hipLaunchKernelGGL((ls_chunk_state_kernel<T, VEC, ROT, MX>), gc, dim3(512), 0, st, a, c);
  hipLaunchKernelGGL(ls_chunk_scan_kernel, gz, dim3(256), 0, st, a, c);
  hipLaunchKernelGGL((ls_chunk_out_kernel<T, VEC, ROT, MX>), gc, dim3(512), 0, st, a, c);
}

template <typename T>
static void ls_chunked_forms(const ScanArgs& a, const KChunkArgs& c, hipStream_t st) {
  constexpr int A = 16 / (int)sizeof(T), W = 8;        // elements in 16 bytes; channels of a unit
  const int rot8 = a.rot_dims ? (a.rot_half ? a.rot_dims / 2 : a.rot_dims) : 0;
  const bool vec = (reinterpret_cast<uintptr_t>(a.x) | reinterpret_cast<uintptr_t>(a.y)) % 16 == 0 &&
                   (a.ld | a.ldy | a.q_off | a.k_off | a.v_off | a.g_off) % A == 0 && a.D % W == 0 &&
                   a.Dv % W == 0 && rot8 % W == 0;
  const bool wide = a.D > 64 || a.Dv > 64, rot = a.rot_dims > 0;
#define LS_GO(V, R) \
  do { if (wide) ls_chunked<T, V, R, 128>(a, c, st); else ls_chunked<T, V, R, 64>(a, c, st); } while (0)
  if (vec) { if (rot) LS_GO(true, true); else LS_GO(true, false); }
  else { if (rot) LS_GO(false, true); else LS_GO(false, false); }
#undef LS_GO
}

// Modes 0 and 1 for steps with prompt portions (cu given; rows: at least cu[nseq]): fp32 workspaces
// U [rows / 128 + nseq, H, DP, UW] and G [rows / 128 + nseq, H, 1 + mode] with DP and VP = dk and dv rounded up
// to 16, UW = VP + 4 mode; m0 [rows / 128 + nseq, H] (mode 1); rot [rows, rot_dims] (rotated heads).
EIA_API int eia_linear_scan_chunked(const void* x, long ld, int q_off, int k_off, int v_off, int g_off,
                                    int i_off, int f_off, const float* decay, const float* inv_freq,
                                    int rot_dims, int rot_half, float qscale, float kscale, float cap,
                                    float out_scale, const void* norm_w, float* S, float* N, float* M,
                                    const int* slots, const int* cu, const int* positions, void* y,
                                    long ldy, float eps, int nseq, int rows, int H, int D, int Dv,
                                    int mode, int gate_act, int norm_h, float* U, float* G, float* m0,
                                    float* rot, int is_bf16, hipStream_t st) {
  if (nseq < 0 || rows < 0 || H < 1 || D < 1 || Dv < 1 || !x || !y || !S || !slots || !cu ||
      !positions || !U || !G || (mode != 0 && mode != 1) || (mode == 0 && !decay) ||
      (mode == 1 && (!N || !M || cap < 0.f || !m0)) || rot_dims < 0 || rot_dims > D ||
      (rot_dims & 1) || (rot_dims && (!inv_freq || !rot)) || (gate_act != 0 && gate_act != 1))
    return EIA_BAD_SHAPE;
  if (D > 128 || Dv > 128 || H > 65535) return EIA_UNSUPPORTED;
  if (nseq == 0 || rows == 0) return EIA_OK;
  ScanArgs a{x, ld, q_off, k_off, v_off, g_off, i_off, f_off, decay, inv_freq, rot_dims, rot_half,
             qscale, kscale, cap, out_scale, norm_w, S, N, M, slots, cu, positions, nullptr, y,
             ldy, eps, H, D, Dv, mode, gate_act, 0, 0, nullptr, nullptr, 1.f, norm_h};
  const int DP = (D + 15) / 16 * 16, VP = (Dv + 15) / 16 * 16;
  KChunkArgs c{U, G, m0, nullptr, reinterpret_cast<float2*>(rot), nseq, rows, DP, VP, VP + 4 * mode};
  if (is_bf16) ls_chunked_forms<bf16_t>(a, c, st); else ls_chunked_forms<float>(a, c, st);
  EIA_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------------------------
// Chunk-parallel form of mode 2 (a decay per key channel), dk, dv <= 128: a step's rows are cut into
// chunks of LC tokens (never across sequences) and, with A_t the running sum of log a inside a chunk,
// a vector over the key channels,
//
//   U_c   = sum_s (exp(A_end - A_s) k_s) v_s^T              (1) per chunk, in parallel
//   S_c+1 = diag(exp(A_end)) S_c + U_c                      (2) a short scan over a sequence's chunks
//   o_t   = S_c^T (exp(A_t) q_t) + sum_(s<=t) (q_t exp(A_t - A_s) . k_s) v_s       (3) per chunk
//
// Every exponent is <= 0.  All of it fp32 FMA.
constexpr int LC = 32;                      // tokens per chunk
constexpr int LD = 128;                     // largest dk / dv of this form
constexpr int LP = LD + 4;                  // LDS row pitch: 16-byte rows that rotate the banks

struct ChunkArgs {
  const int* chunks;                        // [nchunk, 4]: sequence, first row, tokens, unused
  const int* seq_first;                     // [nseq + 1]: first chunk of every sequence
  float* wsS; float* wsG;                   // [nchunk, H, D, Dv], [nchunk, H, D]
  float* cA;                                // [rows, H * D] running log decays of a chunk
};

// (A') running log decays per key channel inside every chunk, thread = channel.
template <typename T>
__global__ void __launch_bounds__(128)
ls_chan_decay_kernel(ScanArgs a, ChunkArgs c) {
  const int ch = blockIdx.x, h = blockIdx.y, j = threadIdx.x;
  const int s = c.chunks[4 * ch], row0 = c.chunks[4 * ch + 1], n = c.chunks[4 * ch + 2];
  if (a.slots[s] < 0 || j >= a.D) return;
  const T* X = static_cast<const T*>(a.x);
  float A = 0.f;
  for (int t = 0; t < n; ++t) {
    A += ls_chan_log<T>(a, X + (long)(row0 + t) * a.ld, h, j);
    c.cA[((long)(row0 + t) * a.H + h) * a.D + j] = A;
  }
  c.wsG[((long)ch * a.H + h) * a.D + j] = A;
}

// Stages rotated, scaled q or k rows ([LC][LD], zero beyond n tokens / D channels).
template <typename T>
EIA_DEV void ls_stage_rot(const ScanArgs& a, const T* X, int row0, int n, long off, float scale,
                          float (*dst)[LP]) {
  const int hd = a.rot_dims >> 1;
  for (int idx = threadIdx.x; idx < LC * LD; idx += blockDim.x) {
    const int t = idx / LD, j = idx % LD;
    float v = 0.f;
    if (t < n && j < a.D) {
      const T* xr = X + (long)(row0 + t) * a.ld;
      v = ld_f32<T>(xr, off + j);
      if (j < a.rot_dims) {
        const bool second = a.rot_half ? j >= hd : (j & 1);
        const int pi = a.rot_half ? (second ? j - hd : j) : (j >> 1);
        const int jp = a.rot_half ? (second ? j - hd : j + hd) : (j ^ 1);
        float sn, cs;
        sincosf((float)a.positions[row0 + t] * a.inv_freq[pi], &sn, &cs);
        v = v * cs + (second ? 1.f : -1.f) * ld_f32<T>(xr, off + jp) * sn;
      }
      v *= scale;
    }
    dst[t][j] = v;
  }
}

// (1) a chunk's own contribution to the state.  Thread (r, j): rows
// [64 r, 64 r + 64) of column j.
template <typename T>
__global__ void __launch_bounds__(256)
ls_chan_state_kernel(ScanArgs a, ChunkArgs c) {
  __shared__ __align__(16) float sk[LC][LP], sv[LC][LD];
  const int ch = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int s = c.chunks[4 * ch], row0 = c.chunks[4 * ch + 1], n = c.chunks[4 * ch + 2];
  if (a.slots[s] < 0) return;
  const int D = a.D, Dv = a.Dv;
  const T* X = static_cast<const T*>(a.x);
  ls_stage_rot<T>(a, X, row0, n, a.k_off + (long)h * D, a.kscale, sk);
  for (int idx = tid; idx < LC * LD; idx += 256) {
    const int t = idx / LD, j = idx % LD;
    sv[t][j] = (t < n && j < Dv) ? ld_f32<T>(X + (long)(row0 + t) * a.ld, a.v_off + (long)h * Dv + j)
                                 : 0.f;
  }
  __syncthreads();
  for (int idx = tid; idx < LC * LD; idx += 256) {     // k_s <- w_s k_s
    const int t = idx / LD, j = idx % LD;
    if (t < n && j < D)
      sk[t][j] *= expf(c.wsG[((long)ch * a.H + h) * D + j] -
                       c.cA[((long)(row0 + t) * a.H + h) * D + j]);
  }
  __syncthreads();
  const int r = tid >> 7, j = tid & 127;
  float acc[64];
#pragma unroll
  for (int i = 0; i < 64; ++i) acc[i] = 0.f;
  for (int t = 0; t < n; ++t) {
    const float v = sv[t][j];
#pragma unroll
    for (int i = 0; i < 64; ++i) acc[i] += sk[t][64 * r + i] * v;
  }
  float* U = c.wsS + ((long)ch * a.H + h) * D * Dv;
  if (j < Dv) {
#pragma unroll
    for (int i = 0; i < 64; ++i)
      if (64 * r + i < D) U[(long)(64 * r + i) * Dv + j] = acc[i];
  }
}

// (2) the scan over a sequence's chunks, element by element: the workspace entry of a chunk turns
// from its own contribution into the state BEFORE the chunk; the slot receives the final state.
__global__ void __launch_bounds__(256)
ls_chan_scan_kernel(ScanArgs a, ChunkArgs c) {
  const int s = blockIdx.x, h = blockIdx.y;
  const int slot = a.slots[s];
  if (slot < 0) return;
  const int c0 = c.seq_first[s], c1 = c.seq_first[s + 1];
  if (c1 <= c0) return;
  const int lo = a.cu ? a.cu[s] : s;
  const bool fresh = a.positions[lo] == 0;
  const long n_el = (long)a.D * a.Dv;
  const long e = (long)blockIdx.z * 256 + threadIdx.x;
  if (e < n_el) {
    float* Sg = a.S + ((long)slot * a.H + h) * n_el;
    const int ei = (int)(e / a.Dv);                    // state row (key channel)
    float S = fresh ? 0.f : Sg[e];
    for (int ch = c0; ch < c1; ++ch) {
      float* w = c.wsS + ((long)ch * a.H + h) * n_el + e;
      const float U = *w;
      *w = S;
      S = expf(c.wsG[((long)ch * a.H + h) * a.D + ei]) * S + U;
    }
    Sg[e] = S;
  }
}

// (3) a chunk's outputs from the state before it and its own tokens.  Thread (r, j): tokens
// r, r + 2, ... of column j.
// The pair weights sum q_t k_u exp(A_t - A_u) over the channels.  A
// chunk is four blocks of eight tokens; pairs inside a block form their exponents one by one,
// pairs of different blocks factor them through the block edges (E_b: A just before block b),
//   exp(A_t - A_u) = exp(A_t - E_tb) exp(E_tb - E_(ub+1)) exp(E_(ub+1) - A_u),
// so every exponent stays <= 0 whatever the decays.
template <typename T>
__global__ void __launch_bounds__(256)
ls_chan_out_kernel(ScanArgs a, ChunkArgs c) {
  __shared__ __align__(16) float sq[LC][LP], sk[LC][LP], sv[LC][LD];
  __shared__ float P[LC][LC + 1];
  __shared__ float red[LC][2];
  __shared__ __align__(16) float sC[LC][LP];           // running log decays per channel
  __shared__ __align__(16) float sE[3][LP];            // products over whole blocks
  const int ch = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int s = c.chunks[4 * ch], row0 = c.chunks[4 * ch + 1], n = c.chunks[4 * ch + 2];
  if (a.slots[s] < 0) return;
  const int D = a.D, Dv = a.Dv;
  const T* X = static_cast<const T*>(a.x);
  ls_stage_rot<T>(a, X, row0, n, a.q_off + (long)h * D, a.qscale, sq);
  ls_stage_rot<T>(a, X, row0, n, a.k_off + (long)h * D, a.kscale, sk);
  for (int idx = tid; idx < LC * LD; idx += 256) {
    const int t = idx / LD, j = idx % LD;
    sv[t][j] = (t < n && j < Dv) ? ld_f32<T>(X + (long)(row0 + t) * a.ld, a.v_off + (long)h * Dv + j)
                                 : 0.f;
  }
  for (int idx = tid; idx < LC * LD; idx += 256) {
    const int t = idx / LD, j = idx % LD;            // (past the chunk's end: the last token's)
    sC[t][j] = j < D ? c.cA[((long)(row0 + min(t, n - 1)) * a.H + h) * D + j] : 0.f;
  }
  __syncthreads();
  // pairs inside a block of eight
  for (int idx = tid; idx < LC * 8; idx += 256) {
    const int t = idx >> 3, u = (t & ~7) + (idx & 7);
    float p = 0.f;
    if (u <= t && t < n) {
      const f32x4* qa = reinterpret_cast<const f32x4*>(sq[t]);
      const f32x4* ka = reinterpret_cast<const f32x4*>(sk[u]);
      const f32x4* At = reinterpret_cast<const f32x4*>(sC[t]);
      const f32x4* Au = reinterpret_cast<const f32x4*>(sC[u]);
#pragma unroll 4
      for (int i = 0; i < (D + 3) / 4; ++i) {
        const f32x4 x = qa[i] * ka[i], d = At[i] - Au[i];
        p += x[0] * __expf(d[0]) + x[1] * __expf(d[1]) + x[2] * __expf(d[2]) + x[3] * __expf(d[3]);
      }
    }
    P[t][u] = p;
  }
  __syncthreads();
  // q_t <- q_t exp(A_t - E_tb), k_u <- k_u exp(E_(ub+1) - A_u); block products for the carry
  for (int idx = tid; idx < LC * LD; idx += 256) {
    const int t = idx / LD, j = idx % LD, b = t >> 3;
    const float A = sC[t][j];
    sq[t][j] *= expf(A - (b ? sC[8 * b - 1][j] : 0.f));
    sk[t][j] *= expf(sC[8 * b + 7][j] - A);
    if (t < 3) sE[t][j] = expf(sC[8 * t + 15][j] - sC[8 * t + 7][j]);   // over block t + 1
  }
  __syncthreads();
  // pairs of different blocks: (t, u) with ub < tb, over the blocks between them
  for (int idx = tid; idx < LC * LC; idx += 256) {
    const int t = idx / LC, u = idx % LC, tb = t >> 3, ub = u >> 3;
    if (ub == tb) continue;
    float p = 0.f;
    if (ub < tb && t < n) {
      const f32x4* qa = reinterpret_cast<const f32x4*>(sq[t]);
      const f32x4* ka = reinterpret_cast<const f32x4*>(sk[u]);
      const f32x4* e0 = reinterpret_cast<const f32x4*>(sE[ub]);        // block ub + 1
      const f32x4* e1 = reinterpret_cast<const f32x4*>(sE[ub < 1 ? 1 : ub]);   // block ub + 2
#pragma unroll 4
      for (int i = 0; i < (D + 3) / 4; ++i) {
        f32x4 x = qa[i] * ka[i];
        if (tb - ub > 1) x *= e0[i];
        if (tb - ub > 2) x *= e1[i];
        p += x[0] + x[1] + x[2] + x[3];
      }
    }
    P[t][u] = p;
  }
  __syncthreads();
  // the carry reads q_t exp(A_t)
  for (int idx = tid; idx < (LC - 8) * LD; idx += 256) {
    const int t = 8 + idx / LD, j = idx % LD;
    sq[t][j] *= expf(sC[8 * (t >> 3) - 1][j]);
  }
  __syncthreads();
  const int r = tid >> 7, j = tid & 127;
  const float* Sb = c.wsS + ((long)ch * a.H + h) * D * Dv;      // the state before the chunk
  float own[LC / 2], carry[LC / 2];
#pragma unroll
  for (int tt = 0; tt < LC / 2; ++tt) { own[tt] = 0.f; carry[tt] = 0.f; }
  if (j < Dv) {
    for (int i = 0; i < D; ++i) {
      const float sv_ = Sb[(long)i * Dv + j];
#pragma unroll
      for (int tt = 0; tt < LC / 2; ++tt) carry[tt] += sq[2 * tt + r][i] * sv_;
    }
    for (int u = 0; u < n; ++u) {
      const float v = sv[u][j];
#pragma unroll
      for (int tt = 0; tt < LC / 2; ++tt) own[tt] += P[2 * tt + r][u] * v;
    }
  }
  const T* NW = static_cast<const T*>(a.norm_w);
  const float nw = (NW && j < Dv) ? ld_f32<T>(NW, (long)h * a.norm_h + j) : 1.f;
  T* Y = static_cast<T*>(a.y);
  const float inv_dv = 1.0f / (float)Dv;
#pragma unroll
  for (int tt = 0; tt < LC / 2; ++tt) {
    const int t = 2 * tt + r;
    const float o = (j < Dv && t < n) ? own[tt] + carry[tt] : 0.f;
    const float ss = wave_sum(o * o);
    if ((tid & 63) == 0) red[t][(tid >> 6) & 1] = ss;
    own[tt] = o;
  }
  __syncthreads();
#pragma unroll
  for (int tt = 0; tt < LC / 2; ++tt) {
    const int t = 2 * tt + r;
    if (t < n && j < Dv) {
      const float g = ld_f32<T>(X + (long)(row0 + t) * a.ld, a.g_off + (long)h * Dv + j);
      const float sig = 1.0f / (1.0f + expf(-g));
      const float gate = a.gate_act == 0 ? g * sig : sig;
      st_f32<T>(Y, (long)(row0 + t) * a.ldy + (long)h * Dv + j,
                own[tt] / sqrtf((red[t][0] + red[t][1]) * inv_dv + a.eps) * nw * gate * a.out_scale);
    }
  }
}

// Mode 2 with the step's chunk list (chunks int32 [nchunk, 4]: sequence, first row, tokens (1 .. 32),
// 0; seq_first int32 [nseq + 1]) and fp32 workspaces wsS [nchunk, H, D, Dv], wsG [nchunk, H, D], cA
// [rows, H * D].
EIA_API int eia_linear_scan_channels(const void* x, long ld, int q_off, int k_off, int v_off,
                                     int g_off, const float* inv_freq, int rot_dims, int rot_half,
                                     float qscale, float kscale, float out_scale,
                                     const void* norm_w, float* S, const int* slots, const int* cu,
                                     const int* positions, void* y, long ldy, float eps, int nseq,
                                     int H, int D, int Dv, int gate_act, int norm_h,
                                     const int* chunks, const int* seq_first, int nchunk, float* wsS,
                                     float* wsG, int lo_off, int R, const float* a2t,
                                     const float* a2b, float inv_tau, float* cA, int is_bf16,
                                     hipStream_t st) {
  if (nseq < 0 || nchunk < 0 || H < 1 || D < 1 || Dv < 1 || !x || !y || !S || !slots || !positions ||
      !chunks || !seq_first || !wsS || !wsG || R < 1 || !a2t || !cA || rot_dims < 0 ||
      rot_dims > D || (rot_dims & 1) || (rot_dims && !inv_freq) ||
      (gate_act != 0 && gate_act != 1))
    return EIA_BAD_SHAPE;
  if (D > LD || Dv > LD) return EIA_UNSUPPORTED;
  if (nseq == 0 || nchunk == 0) return EIA_OK;
  ScanArgs a{x, ld, q_off, k_off, v_off, g_off, 0, 0, nullptr, inv_freq, rot_dims, rot_half,
             qscale, kscale, 0.f, out_scale, norm_w, S, nullptr, nullptr, slots, cu, positions,
             nullptr, y, ldy, eps, H, D, Dv, 2, gate_act, lo_off, R, a2t, a2b, inv_tau, norm_h};
  ChunkArgs c{chunks, seq_first, wsS, wsG, cA};
  const dim3 gc(nchunk, H), gz(nseq, H, (D * Dv + 255) / 256);
#define LS_CHUNKED(TT)                                                              \
  do {                                                                              \
    hipLaunchKernelGGL((ls_chan_decay_kernel<TT>), gc, dim3(128), 0, st, a, c);     \
    hipLaunchKernelGGL((ls_chan_state_kernel<TT>), gc, dim3(256), 0, st, a, c);     \
    hipLaunchKernelGGL(ls_chan_scan_kernel, gz, dim3(256), 0, st, a, c);            \
    hipLaunchKernelGGL((ls_chan_out_kernel<TT>), gc, dim3(256), 0, st, a, c);       \
  } while (0)
  if (is_bf16) LS_CHUNKED(bf16_t); else LS_CHUNKED(float);
#undef LS_CHUNKED
  EIA_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------------------------
// Mode 2 for dk <= 64 on matrix cores: the chunks of GC tokens and the block edges of wkv.hip's
// chunk-parallel form, with the token itself among its keys,
//
//   U   = sum_s 2^(sum_(s<x) l_x) k_s v_s^T                            (1) per chunk, in parallel
//   S' = 2^(sum_x l_x) S + U                                           (2) a sequence's chunks in order
//   o_t = (q_t 2^(sum_(x<=t) l_x)) S + sum_(s<=t) P_ts v_s
//   P_ts = sum_channels q_t k_s 2^(sum_(s<x<=t) l_x)                   (3) per chunk, in parallel
//
// where l_x = log2 a_x per key channel, formed by a pass of its own for all rows and heads (its
// low-rank product and logarithms are the same for (1) and (3)).  Exponents are sums of the l_x that they
// cover; pairs of different 8-token blocks meet through the edges of the blocks between them, for those
// inside a block see eia_chunks.h.  Products are fp32 matrix-core products.  Bound by instruction issue
// (exponentials, operand rows through LDS), as there.
// Four prompts of 556 to 977 tokens, 16 heads of 64 x 128, bf16: 21 + 21 + 11 + 45 us on an MI355X (l, (1),
// (2), (3)); in the 32-token chunks of vector FMAs above, of 490 to 977, 38 + 71 + 21 + 235 us, which remain for keys
// wider than 64.
constexpr int GC = 64;                      // tokens per chunk
constexpr int GD = 64;                      // widest key head

EIA_DEV bool gl_chunk(const ScanArgs& a, int nseq, int x, int& s, int& row0, int& n) {
  return chunk_of<GC>(a.cu, nseq, x, s, row0, n) && a.slots[s] >= 0;
}

// l of all rows: thread = channel of one head and 16 rows.
template <typename T>
__global__ void __launch_bounds__(256)
gl_logs_kernel(ScanArgs a, KChunkArgs c) {
  constexpr int RB = 32;
  __shared__ float lo[64][RB + 1];
  const int h = blockIdx.y, j = threadIdx.x & 63, g = threadIdx.x >> 6, r0 = blockIdx.x * 64;
  const long HD = (long)a.H * a.D, hc = (long)h * a.D + min(j, a.D - 1);
  const T* X = static_cast<const T*>(a.x) + a.lo_off;
  float z[16];
  const float b = a.a2b ? a.a2b[hc] : 0.f;
#pragma unroll
  for (int t = 0; t < 16; ++t) z[t] = b;
  for (int k0 = 0; k0 < a.R; k0 += RB) {
    const int kn = min(RB, a.R - k0);
    __syncthreads();
    for (int u = threadIdx.x; u < 64 * kn; u += 256) {
      const int t = u / kn, k = u % kn;
      lo[t][k] = ld_f32<T>(X + (long)min(r0 + t, c.rows - 1) * a.ld, k0 + k);
    }
    __syncthreads();
#pragma unroll 8
    for (int k = 0; k < kn; ++k) {
      const float w = a.a2t[(k0 + k) * HD + hc];
#pragma unroll
      for (int t = 0; t < 16; ++t) z[t] += lo[16 * g + t][k] * w;
    }
  }
  if (j >= a.D) return;
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const int r = r0 + 16 * g + t;
    if (r < c.rows) c.la[r * HD + hc] = ls_logsigmoid(z[t]) * a.inv_tau * LS_LOG2E;
  }
}

// l of channel i, tokens t0 .. t0 + 15 of the chunk (0 past its end and past D).
EIA_DEV void gl_decays(const ScanArgs& a, const KChunkArgs& c, int h, int row0, int n, int t0, int i,
                       float (&l)[16]) {
  const float* p = c.la + (long)h * a.D + min(i, a.D - 1);
#pragma unroll
  for (int t = 0; t < 16; ++t) l[t] = p[(long)(row0 + min(t0 + t, n - 1)) * a.H * a.D];
  __builtin_amdgcn_sched_barrier(0);                   // all of them, and the rows before them, are asked for first
#pragma unroll
  for (int t = 0; t < 16; ++t) l[t] = (i < a.D && t0 + t < n) ? l[t] : 0.f;
}

// A chunk's [GC][GD] tile of q or k, rotated and scaled, on its way to LDS.
template <typename T, bool VEC, bool ROT>
struct GlTile {
  float v[2][8];
  EIA_DEV void load(const ScanArgs& a, const KChunkArgs& c, int row0, int n, long off) {
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const int u = threadIdx.x + 256 * x;
      ls_head8<T, VEC, ROT>(a, c, row0 + min(u >> 3, n - 1), off, 8 * (u & 7), v[x]);
    }
  }
  EIA_DEV void store(float* tile, int n, float scale) const {
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const int u = threadIdx.x + 256 * x, t = u >> 3, i = 8 * (u & 7);
#pragma unroll
      for (int e = 0; e < 8; e += 4) {
        f32x4 f = f32x4{v[x][e], v[x][e + 1], v[x][e + 2], v[x][e + 3]} * scale;
        asm volatile("" : "+v"(f));                    // (else some rows are asked for behind the choice, and waited for)
        *reinterpret_cast<f32x4*>(tile + tile_at<GD>(t, i + e)) = t < n ? f : f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
  }
};

// ... and of v, GC x 64 NV, zero past the chunk and past Dv.
template <typename T, bool VEC, int NV>
struct GlValues {
  static constexpr int E = VEC ? 16 / (int)sizeof(T) : 1, W = 64 * NV, N = GC * W / (256 * E);
  alignas(16) T v[N][E];
  EIA_DEV void load(const ScanArgs& a, int row0, int n, int h) {
    const T* X = static_cast<const T*>(a.x) + a.v_off + (long)h * a.Dv;
#pragma unroll
    for (int x = 0; x < N; ++x) {
      const int u = threadIdx.x + 256 * x, t = u / (W / E), i = E * (u % (W / E));
      const T* p = X + (long)(row0 + min(t, n - 1)) * a.ld + (i < a.Dv ? i : 0);
      if constexpr (VEC) *reinterpret_cast<f32x4*>(v[x]) = *reinterpret_cast<const f32x4*>(p);
      else v[x][0] = *p;
    }
  }
  EIA_DEV void store(float* tile, int n, int Dv) const {
    typedef __attribute__((ext_vector_type(4))) int i32x4;
#pragma unroll
    for (int x = 0; x < N; ++x) {
      const int u = threadIdx.x + 256 * x, t = u / (W / E), i = E * (u % (W / E));
      const int keep = t < n && i < Dv ? -1 : 0;
      if constexpr (VEC && sizeof(T) == 2) {
        const i32x4 q = *reinterpret_cast<const i32x4*>(v[x]) & keep;
#pragma unroll
        for (int e = 0; e < 4; e += 2)
          *reinterpret_cast<i32x4*>(tile + tile_at<W>(t, i + 2 * e)) =
              i32x4{q[e] << 16, q[e] & (int)0xffff0000, q[e + 1] << 16, q[e + 1] & (int)0xffff0000};
      } else if constexpr (VEC) {
        *reinterpret_cast<i32x4*>(tile + tile_at<W>(t, i)) = *reinterpret_cast<const i32x4*>(v[x]) & keep;
      } else {
        tile[tile_at<W>(t, i)] = __int_as_float(__float_as_int((float)v[x][0]) & keep);
      }
    }
  }
};

// (1) Wave w forms rows 16 w .. of U [GD][64 NV].  A lane holds value columns 64 z + 4 (lane % 16) + j
// in its tile 4 z + j, here and in (3).
template <typename T, bool VEC, bool ROT, int NV>
__global__ void __launch_bounds__(256)
gl_state_kernel(ScanArgs a, KChunkArgs c) {
  constexpr int W = 64 * NV;
  __shared__ __align__(16) float sk[GC * GD], sv[GC * W];
  __shared__ float stot[4][GD];
  int s, row0, n;
  if (!gl_chunk(a, c.nseq, chunk_number(), s, row0, n)) return;
  const int h = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int l16 = lane & 15, g4 = lane >> 4;
  GlTile<T, VEC, ROT> tk;
  GlValues<T, VEC, NV> tv;
  tk.load(a, c, row0, n, a.k_off + (long)h * a.D);
  tv.load(a, row0, n, h);
  float l[16];
  gl_decays(a, c, h, row0, n, 16 * w, lane, l);
  float tot = 0.f;
#pragma unroll
  for (int t = 0; t < 16; ++t) tot += l[t];
  stot[w][lane] = tot;
  tk.store(sk, n, a.kscale);
  tv.store(sv, n, a.Dv);
  __syncthreads();
  float after = 0.f;                                   // sum of l from the next token on
  for (int b = 3; b > w; --b) after += stot[b][lane];
#pragma unroll
  for (int t = 15; t >= 0; --t) {
    sk[tile_at<GD>(16 * w + t, lane)] *= __builtin_amdgcn_exp2f(after);
    after += l[t];
  }
  const long at = (long)chunk_number() * a.H + h;
  if (w == 0) c.G[at * GD + lane] = after;
  __syncthreads();
  f32x4 acc[4 * NV];
#pragma unroll
  for (int j = 0; j < 4 * NV; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    if (16 * b >= n) break;
    f32x4 ka, vb[4 * NV];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t = 16 * b + 4 * g4 + e;
      ka[e] = sk[tile_at<GD>(t, 16 * w + l16)];
#pragma unroll
      for (int z = 0; z < NV; ++z) {
        const f32x4 x = tile_get<W>(sv, t, 64 * z + 4 * l16);
#pragma unroll
        for (int j = 0; j < 4; ++j) vb[4 * z + j][e] = x[j];
      }
    }
#pragma unroll
    for (int j = 0; j < 4 * NV; ++j) acc[j] = mfma_f32_k16(ka, vb[j], acc[j]);
  }
  float* U = c.U + at * GD * W + (long)(16 * w + 4 * g4) * W + 4 * l16;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int z = 0; z < NV; ++z)
      *reinterpret_cast<f32x4*>(U + i * W + 64 * z) =
          f32x4{acc[4 * z][i], acc[4 * z + 1][i], acc[4 * z + 2][i], acc[4 * z + 3][i]};
}

// (2) Four columns of a state row per thread; the slot receives the state after the last chunk.
template <int NV>
__global__ void __launch_bounds__(256)
gl_scan_kernel(ScanArgs a, KChunkArgs c) {
  constexpr int W = 64 * NV;
  const int s = chunk_number(), h = blockIdx.x % a.H;
  if (s >= c.nseq) return;
  const int slot = a.slots[s], lo = a.cu[s], hi = a.cu[s + 1];
  if (slot < 0 || hi <= lo) return;
  const int e = 4 * (blockIdx.x / a.H * 256 + threadIdx.x), i = e / W, j = e % W, D = a.D, Dv = a.Dv;
  const long x0 = lo / GC + s;
  const int nc = (hi - lo + GC - 1) / GC;
  float* Sg = a.S + ((long)slot * a.H + h) * D * Dv + (long)i * Dv + j;
  f32x4 S = {0.f, 0.f, 0.f, 0.f};
  if (a.positions[lo] != 0 && i < D) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (j + k < Dv) S[k] = Sg[k];
  }
  float* U = c.U + (x0 * a.H + h) * GD * W + e;
  const float* L = c.G + (x0 * a.H + h) * GD + i;
  chunk_walk(U, (long)a.H * GD * W, L, (long)a.H * GD, nc, S);
  if (i < D) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (j + k < Dv) Sg[k] = S[k];
  }
}

// (3) Wave w forms the outputs of tokens 16 w .. (which wave takes which rotates with the chunk).  The
// running sums of l share their LDS with the values, which move in after them.
// WIDE: gate, weight and output rows can be taken four at a time.
template <typename T, bool VEC, bool WIDE, bool ROT, int NV>
__global__ void __launch_bounds__(256, 2)
gl_out_kernel(ScanArgs a, KChunkArgs c) {
  constexpr int W = 64 * NV;
  __shared__ __align__(16) float sq[GC * GD], sk[GC * GD], sAv[GC * W];
  __shared__ __align__(16) float se[8][GD];            // decays over whole 8-token blocks
  int s, row0, n;
  if (!gl_chunk(a, c.nseq, chunk_number(), s, row0, n)) return;
  const int h = blockIdx.x, lane = threadIdx.x & 63, w = ((threadIdx.x >> 6) + blockIdx.y) & 3;
  const int Dv = a.Dv, l16 = lane & 15, g4 = lane >> 4, t0 = 16 * w;
  GlTile<T, VEC, ROT> tq, tk;
  GlValues<T, VEC, NV> tv;
  tq.load(a, c, row0, n, a.q_off + (long)h * a.D);
  tk.load(a, c, row0, n, a.k_off + (long)h * a.D);
  float l[16];
  gl_decays(a, c, h, row0, n, t0, lane, l);
  tv.load(a, row0, n, h);                              // (before the decays: eight prompts of 300 tokens 57.1 -> 58.1 us)
  tq.store(sq, n, a.qscale);
  tk.store(sk, n, a.kscale);
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    float tot = 0.f;
#pragma unroll
    for (int t = 8 * b; t < 8 * b + 8; ++t) tot += l[t];
    se[2 * w + b][lane] = __builtin_amdgcn_exp2f(tot);
  }
  block_edges<true>(l, sAv, t0, lane);
  __syncthreads();
  f32x4 p = {0.f, 0.f, 0.f, 0.f};                      // weights inside the wave's 8-token blocks
  if (t0 < n) {
    float b = 0.f;                                     // q . k of token t0 + l16
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
      const int d = 16 * g4 + i;
      const f32x4 x = tile_get<GD>(sq, t0 + l16, d) * tile_get<GD>(sk, t0 + l16, d);
      b += x[0] + x[1] + x[2] + x[3];
    }
    b += __shfl_xor(b, 16, 64);
    b += __shfl_xor(b, 32, 64);
    p = block_weights<true>(sq, sk, sAv, l, b, t0, lane);
  }
  __syncthreads();
  // q_t <- q_t 2^(block start .. t], k_s <- k_s 2^(s .. block end), 8-token blocks; v moves in
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    float pre = 0.f, suf = 0.f;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      pre += l[8 * b + t];
      sq[tile_at<GD>(t0 + 8 * b + t, lane)] *= __builtin_amdgcn_exp2f(pre);
      sk[tile_at<GD>(t0 + 8 * b + 7 - t, lane)] *= __builtin_amdgcn_exp2f(suf);
      suf += l[8 * b + 7 - t];
    }
  }
  tv.store(sAv, n, Dv);
  __syncthreads();
  if (t0 >= n) return;
  f32x4 rt[4], o[4 * NV], pq = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int i = 16 * b + 4 * g4;
    rt[b] = tile_get<GD>(sq, t0 + l16, i);
    pq = mfma_f32_k16(tile_get<GD>(sk, t0 + l16, i), rt[b], pq);
    if (l16 >= 8) rt[b] *= *reinterpret_cast<const f32x4*>(&se[2 * w][i]);
  }
#pragma unroll
  for (int j = 0; j < 4 * NV; ++j) o[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // (weights are formed transposed, keys x queries: their registers are the A operand of P v)
  if (l16 >= 8 && g4 < 2) p += pq;                     // second 8 queries, first 8 keys
  // the first quarter of the state is on its way during the weights' products, the next during those of the one before
  const float* S = c.U + ((long)chunk_number() * a.H + h) * GD * W + (long)4 * g4 * W + 4 * l16;
  f32x4 sq4[2][NV][4];
  auto ask = [&](int x) {
#pragma unroll
    for (int z = 0; z < NV; ++z)
#pragma unroll
      for (int e = 0; e < 4; ++e) sq4[x & 1][z][e] = *reinterpret_cast<const f32x4*>(S + (16 * x + e) * W + 64 * z);
  };
  ask(0);
  for (int b = w;;) {
    f32x4 vb[4 * NV];
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int z = 0; z < NV; ++z) {
        const f32x4 x = tile_get<W>(sAv, 16 * b + 4 * g4 + e, 64 * z + 4 * l16);
#pragma unroll
        for (int j = 0; j < 4; ++j) vb[4 * z + j][e] = x[j];
      }
#pragma unroll
    for (int j = 0; j < 4 * NV; ++j) o[j] = mfma_f32_k16(p, vb[j], o[j]);
    if (--b < 0) break;
    p = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < 4; ++x) {                      // keys of block b; rt: from its end on
      const int i = 16 * x + 4 * g4;
      const f32x4 e1 = *reinterpret_cast<const f32x4*>(&se[2 * b + 1][i]);
      f32x4 kk = tile_get<GD>(sk, 16 * b + l16, i);
      if (l16 < 8) kk *= e1;
      p = mfma_f32_k16(kk, rt[x], p);
      rt[x] *= e1 * *reinterpret_cast<const f32x4*>(&se[2 * b][i]);
    }
  }
  // the gates and the norm's weight are on their way during the last products
  typedef T T4 __attribute__((ext_vector_type(4)));
  T4 gv[4][NV], nw[NV];
  {
    const T* G = static_cast<const T*>(a.x) + a.g_off + (long)h * Dv;
    const T* NW = static_cast<const T*>(a.norm_w) + (a.norm_w ? (long)h * a.norm_h : 0);
#pragma unroll
    for (int z = 0; z < NV; ++z) {
      const int d = 64 * z + 4 * l16;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const T* q = G + (row0 + min(t0 + 4 * g4 + i, n - 1)) * a.ld;
        if constexpr (WIDE) {
          gv[i][z] = *reinterpret_cast<const T4*>(q + min(d, Dv - 4));
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) gv[i][z][j] = q[min(d + j, Dv - 1)];
        }
      }
    }
    if (a.norm_w) {
#pragma unroll
      for (int z = 0; z < NV; ++z) {
        const int d = 64 * z + 4 * l16;
        if constexpr (WIDE) {
          nw[z] = *reinterpret_cast<const T4*>(NW + min(d, Dv - 4));
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) nw[z][j] = NW[min(d + j, Dv - 1)];
        }
      }
    } else {
#pragma unroll
      for (int z = 0; z < NV; ++z) nw[z] = T4{(T)1.f, (T)1.f, (T)1.f, (T)1.f};
    }
  }
  if (row0 != a.cu[s] || a.positions[a.cu[s]] != 0) {  // (a fresh sequence's first chunk: S = 0)
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      if (x < 3) ask(x + 1);
#pragma unroll
      for (int z = 0; z < NV; ++z) {
        f32x4 sb[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int j = 0; j < 4; ++j) sb[j][e] = sq4[x & 1][z][e][j];
#pragma unroll
        for (int j = 0; j < 4; ++j) o[4 * z + j] = mfma_f32_k16(rt[x], sb[j], o[4 * z + j]);
      }
    }
  }
  mfma_settle(o);
  T4 yv[4][NV];
#pragma unroll
  for (int i = 0; i < 4; ++i) {                        // head RMS norm (zeros past Dv), weight, gate
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 4 * NV; ++j) ss += o[j][i] * o[j][i];
    const float inv = a.out_scale / sqrtf(row16_sum(ss) / (float)Dv + a.eps);
#pragma unroll
    for (int z = 0; z < NV; ++z) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float g = (float)gv[i][z][j];
        const float sig = sizeof(T) == 2 ? __builtin_amdgcn_rcpf(1.0f + __expf(-g)) : 1.0f / (1.0f + expf(-g));
        yv[i][z][j] = (T)(o[4 * z + j][i] * inv * (float)nw[z][j] * (a.gate_act == 0 ? g * sig : sig));
      }
      asm volatile("" : "+v"(yv[i][z]));               // (formed before the branches of the stores)
    }
  }
  T* Y = static_cast<T*>(a.y) + (long)(row0 + t0 + 4 * g4) * a.ldy + (long)h * Dv;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (t0 + 4 * g4 + i >= n) break;
#pragma unroll
    for (int z = 0; z < NV; ++z) {
      const int d = 64 * z + 4 * l16;
      if constexpr (WIDE) {
        if (d < Dv) *reinterpret_cast<T4*>(Y + i * a.ldy + d) = yv[i][z];
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (d + j < Dv) Y[i * a.ldy + d + j] = yv[i][z][j];
      }
    }
  }
}

template <typename T, bool VEC, bool WIDE, bool ROT, int NV>
static void gl_launch(const ScanArgs& a, const KChunkArgs& c, hipStream_t st) {
  const dim3 gc = chunk_grid(c.rows / GC + c.nseq, a.H), gs = chunk_grid(c.nseq, a.H * (GD * 64 * NV / 1024));
  hipLaunchKernelGGL((gl_logs_kernel<T>), dim3((c.rows + 63) / 64, a.H), dim3(256), 0, st, a, c);
  if (ROT) {
    const long u = (long)c.rows * (a.rot_dims >> 1);
    hipLaunchKernelGGL(ls_angles_kernel, dim3((unsigned)((u + 255) / 256)), dim3(256), 0, st, a, c);
  }
  hipLaunchKernelGGL((gl_state_kernel<T, VEC, ROT, NV>), gc, dim3(256), 0, st, a, c);
  hipLaunchKernelGGL((gl_scan_kernel<NV>), gs, dim3(256), 0, st, a, c);
  hipLaunchKernelGGL((gl_out_kernel<T, VEC, WIDE, ROT, NV>), gc, dim3(256), 0, st, a, c);
}

template <typename T>
static void gl_forms(const ScanArgs& a, const KChunkArgs& c, hipStream_t st) {
  constexpr int A = 16 / (int)sizeof(T);               // elements in 16 bytes
  // rows of q, k and v move by 16 bytes, gates, weights and outputs four at a time, each where they lie so: one flag for
  // both took three prompts of up to 1000 tokens, 16 heads of 64 x 128, with weights off 8 bytes from 81 to 93 us
  const uintptr_t io = reinterpret_cast<uintptr_t>(a.x) | reinterpret_cast<uintptr_t>(a.y) | reinterpret_cast<uintptr_t>(a.norm_w);
  const bool four = io % (4 * sizeof(T)) == 0 && (a.ld | a.ldy | a.g_off | a.Dv | a.norm_h) % 4 == 0;
  const int rot8 = a.rot_dims ? (a.rot_half ? a.rot_dims / 2 : a.rot_dims) : 0;
  const bool vec = reinterpret_cast<uintptr_t>(a.x) % 16 == 0 &&
                   (a.ld | a.q_off | a.k_off | a.v_off) % A == 0 && a.D % 8 == 0 && a.Dv % 8 == 0 &&
                   rot8 % 8 == 0;
  const bool wide = a.Dv > 64, rot = a.rot_dims > 0;
#define GL_ROT(V, F, NV) do { if (rot) gl_launch<T, V, F, true, NV>(a, c, st); else gl_launch<T, V, F, false, NV>(a, c, st); } while (0)
#define GL_GO(V, F) do { if (wide) GL_ROT(V, F, 2); else GL_ROT(V, F, 1); } while (0)
  if (vec) { if (four) GL_GO(true, true); else GL_GO(true, false); }
  else { if (four) GL_GO(false, true); else GL_GO(false, false); }
#undef GL_ROT
#undef GL_GO
}

// As eia_linear_scan_channels for D <= 64, Dv <= 128, chunks found on the device (rows: at least
// cu[nseq]): fp32 workspaces U [rows / 64 + nseq, H, 64, Dv rounded up to 64], L [rows / 64 + nseq, H,
// 64], l [rows, H, D] and, with rotated heads, rot [rows, rot_dims].
EIA_API int eia_linear_scan_channels64(const void* x, long ld, int q_off, int k_off, int v_off, int g_off,
                                       const float* inv_freq, int rot_dims, int rot_half, float qscale,
                                       float kscale, float out_scale, const void* norm_w, float* S,
                                       const int* slots, const int* cu, const int* positions, void* y,
                                       long ldy, float eps, int nseq, int rows, int H, int D, int Dv,
                                       int gate_act, int norm_h, int lo_off, int R, const float* a2t,
                                       const float* a2b, float inv_tau, float* U, float* L, float* l,
                                       float* rot, int is_bf16, hipStream_t st) {
  if (nseq < 0 || rows < 0 || H < 1 || D < 1 || Dv < 1 || !x || !y || !S || !slots || !cu ||
      !positions || !U || !L || !l || R < 1 || !a2t || rot_dims < 0 || rot_dims > D ||
      (rot_dims & 1) || (rot_dims && (!inv_freq || !rot)) || (gate_act != 0 && gate_act != 1))
    return EIA_BAD_SHAPE;
  if (D > GD || Dv > 128 || H > 65535) return EIA_UNSUPPORTED;
  if (nseq == 0 || rows == 0) return EIA_OK;
  ScanArgs a{x, ld, q_off, k_off, v_off, g_off, 0, 0, nullptr, inv_freq, rot_dims, rot_half,
             qscale, kscale, 0.f, out_scale, norm_w, S, nullptr, nullptr, slots, cu, positions,
             nullptr, y, ldy, eps, H, D, Dv, 2, gate_act, lo_off, R, a2t, a2b, inv_tau, norm_h};
  KChunkArgs c{U, L, nullptr, l, reinterpret_cast<float2*>(rot), nseq, rows, GD, Dv, Dv};
  if (is_bf16) gl_forms<bf16_t>(a, c, st); else gl_forms<float>(a, c, st);
  EIA_LAUNCH_CHECK();
}
