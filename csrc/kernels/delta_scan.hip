// Gated delta rule on per-sequence state slots: a matrix state S [dk, dv] per head whose answer to
// the key moves towards the value by the step size,
//
//   S <- a_t S_(t-1);   u_t = b_t (v_t - S^T k_t);   S_t = S + k_t u_t^T;   o_t = S_t^T q_t
//
// with one decay a_t = exp(la_t), la_t = -exp(A_log[h]) softplus(x_a + dt_bias[h]), and one step size
// b_t = sigmoid(x_b) per head and token.  q and k [G heads] and v [H heads] are projections that pass
// a short causal convolution over time and silu; q and k are made unit vectors per head,
// x / sqrt(sum x^2 + 1e-6), q is then scaled; head h reads q / k head h / (H / G).  Each head's o is
// divided by its root mean square, multiplied by a weight shared by the heads, by silu of its gate
// columns and by out_scale.
//
// q, k, v, la and b arrive as the fp32 rows that delta_prep.hip leaves.  Everything here is fp32, the
// matrix products included (v_mfma_f32_16x16x4_f32 in the chunk-parallel form).
//
// A sequence whose first row of the step is position 0 starts from zeros whatever its slot held, so
// slots are reused without clearing.  Batch layout: sequence s owns rows [cu[s], cu[s+1])
// (cu == nullptr: row s).
#include "eia_common.h"

EIA_DEV float dl_silu(float z) { return z / (1.0f + expf(-z)); }

// ---------------------------------------------------------------------------------------------
struct DeltaArgs {
  const float* q; const float* k; const float* v; const float* la; const float* beta;
  int H, G, D, Dv, DP, VP;
  const void* g; long ldg; const void* norm_w; float out_scale, eps;
  float* S; const int* slots; const int* cu; const int* positions; const int* seq_lens;
  void* y; long ldy;
};

// Token by token: one workgroup of 256 threads per (sequence, head).  Thread (rg, cg) owns rows
// rg, rg + RG, ... and columns 4 cg .. of S in registers (CGP = 2^LG column groups, RG = 256 / CGP row
// groups).  Per token one pass over the registers forms S^T k and S^T q of the state BEFORE the
// token; with them and k . q, u = b (v - a S^T k) and o = a S^T q + (k . q) u, so the update needs no
// second reduction (the four waves' partial sums of odd and even tokens alternate between two LDS
// buffers: one barrier per token).  Tokens are staged DS_TC at a time, (k, q) pairs zero past D.
// vec: 16-byte accesses to the state.
constexpr int DS_TC = 8;

template <typename T, int LG, int RPT>
__global__ void __launch_bounds__(256)
delta_scan_kernel(DeltaArgs a, int vec) {
  constexpr int CGP = 1 << LG, RG = 256 >> LG, CW = 4 * CGP, RW = RG * RPT;
  __shared__ __align__(16) float2 skq[DS_TC][RW];
  __shared__ __align__(16) float sv[DS_TC][CW], so[DS_TC][CW], sp[2][4][2][CW];
  __shared__ float dot[DS_TC], sa[DS_TC], sb[DS_TC];
  const int s = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int slot = a.slots[s];
  if (slot < 0 || (a.seq_lens && a.seq_lens[s] <= 0)) return;
  const int lo = a.cu ? a.cu[s] : s, hi = a.cu ? a.cu[s + 1] : s + 1;
  if (hi <= lo) return;
  const int H = a.H, G = a.G, D = a.D, Dv = a.Dv, DP = a.DP, VP = a.VP, kh = h / (H / G);
  const int cg = tid & (CGP - 1), rg = tid >> LG, c0 = 4 * cg;
  float* Sg = a.S + ((long)slot * H + h) * D * Dv;
  const bool fresh = a.positions[lo] == 0;
  f32x4 S[RPT];
#pragma unroll
  for (int ii = 0; ii < RPT; ++ii) {
    const int i = rg + RG * ii;
    S[ii] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (fresh || i >= D || c0 >= Dv) continue;
    if (vec) {
      S[ii] = *reinterpret_cast<const f32x4*>(Sg + (long)i * Dv + c0);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c0 + e < Dv) S[ii][e] = Sg[(long)i * Dv + c0 + e];
    }
  }
  const T* NW = static_cast<const T*>(a.norm_w);
  const T* GT = static_cast<const T*>(a.g);
  T* Y = static_cast<T*>(a.y);
  const int lane = tid & 63, wave = tid >> 6;
  for (int base = lo; base < hi; base += DS_TC) {
    const int nt = min(DS_TC, hi - base);
    __syncthreads();                                   // the previous tokens' LDS reads are done
    for (int idx = tid; idx < nt * RW; idx += 256) {
      const int t = idx / RW, d = idx % RW;
      const long r = ((long)(base + t) * G + kh) * DP + min(d, DP - 1);
      skq[t][d] = d < D ? make_float2(a.k[r], a.q[r]) : make_float2(0.f, 0.f);
    }
    for (int idx = tid; idx < nt * CW; idx += 256) {
      const int t = idx / CW, d = idx % CW;
      sv[t][d] = d < Dv ? a.v[((long)(base + t) * H + h) * VP + d] : 0.f;
    }
    if (tid < nt) {
      sa[tid] = expf(a.la[(long)(base + tid) * H + h]);
      sb[tid] = a.beta[(long)(base + tid) * H + h];
    }
    __syncthreads();
    for (int t = wave; t < nt; t += 4) {               // k . q
      float v = 0.f;
      for (int d = lane; d < RW; d += 64) v += skq[t][d].x * skq[t][d].y;
      v = wave_sum(v);
      if (lane == 0) dot[t] = v;
    }
    for (int t = 0; t < nt; ++t) {
      f32x4 ak = {0.f, 0.f, 0.f, 0.f}, aq = ak;
      float kr[RPT <= 16 ? RPT : 1];
#pragma unroll
      for (int ii = 0; ii < RPT; ++ii) {
        const float2 kq = skq[t][rg + RG * ii];
        if constexpr (RPT <= 16) kr[ii] = kq.x;
        ak += S[ii] * kq.x;
        aq += S[ii] * kq.y;
      }
#pragma unroll
      for (int o = CGP; o < 64; o <<= 1) {             // row groups inside the wave
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          ak[e] += __shfl_xor(ak[e], o, 64);
          aq[e] += __shfl_xor(aq[e], o, 64);
        }
      }
      if (lane < CGP) {
        *reinterpret_cast<f32x4*>(&sp[t & 1][wave][0][c0]) = ak;
        *reinterpret_cast<f32x4*>(&sp[t & 1][wave][1][c0]) = aq;
      }
      __syncthreads();
      f32x4 pk[4], pq[4];
#pragma unroll
      for (int z = 0; z < 4; ++z) {
        pk[z] = *reinterpret_cast<const f32x4*>(&sp[t & 1][z][0][c0]);
        pq[z] = *reinterpret_cast<const f32x4*>(&sp[t & 1][z][1][c0]);
      }
      const float at = sa[t];
      const f32x4 u = (*reinterpret_cast<const f32x4*>(&sv[t][c0]) -
                       (pk[0] + pk[1] + pk[2] + pk[3]) * at) * sb[t];
      if (rg == 0)
        *reinterpret_cast<f32x4*>(&so[t][c0]) = (pq[0] + pq[1] + pq[2] + pq[3]) * at + u * dot[t];
#pragma unroll
      for (int ii = 0; ii < RPT; ++ii)
        S[ii] = S[ii] * at + u * (RPT <= 16 ? kr[RPT <= 16 ? ii : 0] : skq[t][rg + RG * ii].x);
    }
    __syncthreads();
    for (int t = wave; t < nt; t += 4) {               // head RMS norm, weight, gate
      float ss = 0.f;
      for (int d = lane; d < Dv; d += 64) ss += so[t][d] * so[t][d];
      const float inv = a.out_scale / sqrtf(wave_sum(ss) / (float)Dv + a.eps);
      for (int d = lane; d < Dv; d += 64)
        st_f32<T>(Y + (long)(base + t) * a.ldy, (long)h * Dv + d,
                  so[t][d] * inv * ld_f32<T>(NW, d) *
                      dl_silu(ld_f32<T>(GT + (long)(base + t) * a.ldg, (long)h * Dv + d)));
    }
  }
#pragma unroll
  for (int ii = 0; ii < RPT; ++ii) {
    const int i = rg + RG * ii;
    if (i >= D || c0 >= Dv) continue;
    if (vec) {
      *reinterpret_cast<f32x4*>(Sg + (long)i * Dv + c0) = S[ii];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c0 + e < Dv) Sg[(long)i * Dv + c0 + e] = S[ii][e];
    }
  }
}

static bool delta_args_ok(const DeltaArgs& a, int nseq) {
  return nseq >= 0 && a.H >= 1 && a.G >= 1 && a.H % a.G == 0 && a.D >= 1 && a.Dv >= 1 &&
         a.DP >= a.D && a.VP >= a.Dv && a.q && a.k && a.v && a.la && a.beta && a.g && a.norm_w &&
         a.S && a.slots && a.positions && a.y;
}

template <typename T>
static int delta_step(const DeltaArgs& a, int nseq, hipStream_t st) {
  if (a.D > 256 || a.Dv > 256) return EIA_UNSUPPORTED;
  const int vec = a.Dv % 4 == 0 && reinterpret_cast<uintptr_t>(a.S) % 16 == 0;
  const dim3 grid(nseq, a.H);
#define DS_GO(LG, R) \
  hipLaunchKernelGGL((delta_scan_kernel<T, LG, R>), grid, dim3(256), 0, st, a, vec)
#define DS_ROWS(LG, R)                                                                \
  do {                                                                                \
    if (a.D <= 64) DS_GO(LG, R); else if (a.D <= 128) DS_GO(LG, 2 * R);               \
    else DS_GO(LG, 4 * R);                                                            \
  } while (0)
  if (a.Dv <= 64) DS_ROWS(4, 4); else if (a.Dv <= 128) DS_ROWS(5, 8); else DS_ROWS(6, 16);
#undef DS_ROWS
#undef DS_GO
  EIA_LAUNCH_CHECK();
}

// q, k [rows, G, DP], v [rows, H, VP] (fp32, zero past D / Dv), la, beta [rows, H]: the rows that
// eia_delta_prep leaves; g [rows, >= H * Dv], norm_w [Dv] and y [rows, >= H * Dv] are bf16 when
// is_bf16, else fp32; S fp32 [slots, H, D, Dv].
EIA_API int eia_delta_scan(const float* q, const float* k, const float* v, const float* la,
                           const float* beta, int H, int G, int D, int Dv, int DP, int VP,
                           const void* g, long ldg, const void* norm_w, float out_scale, float eps,
                           float* S, const int* slots, const int* cu, const int* positions,
                           const int* seq_lens, void* y, long ldy, int nseq, int is_bf16,
                           hipStream_t st) {
  DeltaArgs a{q, k, v, la, beta, H, G, D, Dv, DP, VP, g, ldg, norm_w, out_scale, eps, S, slots, cu,
              positions, seq_lens, y, ldy};
  if (!delta_args_ok(a, nseq)) return EIA_BAD_SHAPE;
  if (nseq == 0) return EIA_OK;
  return is_bf16 ? delta_step<bf16_t>(a, nseq, st) : delta_step<float>(a, nseq, st);
}

// ---------------------------------------------------------------------------------------------
// Chunk-parallel form for prompt portions (dk, dv <= 128).  A step's rows are cut into chunks of DC
// tokens (never across sequences).  With A_t the running sum of la inside a chunk and S the state
// before it, the chunk's updates solve a unit lower triangular system,
//
//   u_t + sum_(s<t) L_ts u_s = b_t v_t - b_t exp(A_t) S^T k_t,    L_ts = b_t exp(A_t - A_s) k_t . k_s
//
// whose right side is linear in S:  with T = (I + L)^-1,  u = X - Y S,  X = T diag(b) V,
// Y = T diag(b exp(A)) K.
//   (1) T, X, Y of every chunk, in parallel (T by 16-token blocks, diagonal inverses first)
//   (2) a sequence's chunks in order, in parallel over heads and slices of the state's columns:
//       u = X - Y S (replaces X), S <- exp(A_end) S + sum_t exp(A_end - A_t) k_t u_t^T
//   (3) outputs of every chunk, in parallel:
//       o_t = exp(A_t) S^T q_t + sum_(s<=t) exp(A_t - A_s) (q_t . k_s) u_s
// Every exponent is <= 0.  All products are fp32 matrix-core products (16x16x4): an accumulator's
// registers (row 4 (lane / 16) + i, column lane % 16) are, step i, the B operand of a product over
// its rows; an A operand's lane holds four consecutive k of row lane % 16.
//
// Layout.  With row-major workspaces most operands were 4-byte accesses, and issuing them took longer
// than the products.  So everything that passes between the kernels lies as the lanes of the next
// product take it, 16 bytes per lane and 1 KB per access: a fragment [64 lanes][4].  The row and
// column order inside a head is free as long as all products agree, and is chosen so that rows of q, k and v are
// read 8 or 16 bytes at a time: tile j of a group of 64 holds entries 64 g + 4 x + j; its column r is
// x = r, its row r (dk only) x = 4 (r % 4) + r / 4, the order in which an A operand's rows are read.
//   Y  [chunk, H, 4 token tiles, DP tiles]   A operand, rows tokens
//   X  [chunk, H, 4 token tiles, VP tiles]   B operand, rows tokens (u after the scan)
//   Kt [chunk, G, DP tiles, 4 token tiles]   A operand, rows dk
//   S  [chunk, H, DP tiles, VP tiles]        B operand, rows dk
// with DP and VP rounded up to 64.  MI355X, 16 heads of 128 x 128, three prompts of 750 to 1500
// tokens: 48 + 77 + 83 us (row-major: 87 + 138 + 129), of which the products alone are 14 + 46 + 26.
constexpr int DC = 64;                      // tokens per chunk
constexpr int DL = DC + 4;                  // LDS row pitch of the triangular blocks

struct DeltaChunkArgs {
  const int* chunks;                        // [nchunk, 4]: sequence, first row, tokens, unused
  const int* seq_first;                     // [nseq + 1]: first chunk of every sequence
  float* Y; float* X; float* Kt; float* wsS;   // fragments, as above (wsS: the state before each chunk)
  float* cA;                                // [nchunk, H, DC] running sums of la, constant past the end
  int ncg;                                  // groups of 64 state columns
  int vec;                                  // out, gate and weight rows can be taken 4 at a time
};

EIA_DEV f32x4 mm(f32x4 a, f32x4 b, f32x4 c) { return mfma_f32_k16(a, b, c); }
EIA_DEV int dl_row(int r) { return 4 * (r & 3) + (r >> 2); }
EIA_DEV f32x4 frag(const float* p, long tile, int lane) {
  return *reinterpret_cast<const f32x4*>(p + tile * 256 + 4 * lane);
}
EIA_DEV void put_frag(float* p, long tile, int lane, f32x4 v) {
  *reinterpret_cast<f32x4*>(p + tile * 256 + 4 * lane) = v;
}

// (1) one workgroup per (chunk, head).  K is staged in LDS: the triangle takes it by rows, Y by
// columns.  Y and X are made in units of 32 columns, 8-byte reads; a wave has at most one unit of
// each, and the rows of v for its unit are on their way from the start.
template <int NDG>                                     // groups of 64 dk
__global__ void __launch_bounds__(256)
delta_chunk_solve_kernel(DeltaArgs a, DeltaChunkArgs c) {
  constexpr int KP = 64 * NDG + 4;
  __shared__ __align__(16) float ks[DC][KP];
  __shared__ __align__(16) float Ls[DC][DL];           // -L, then T
  __shared__ float sA[DC], sb[DC];
  const int ch = blockIdx.y, h = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int s = c.chunks[4 * ch], row0 = c.chunks[4 * ch + 1], n = c.chunks[4 * ch + 2];
  if (a.slots[s] < 0) return;
  const int H = a.H, G = a.G, DP = a.DP, VP = a.VP, kh = h / (H / G);
  const int g4 = lane >> 4, l16 = lane & 15;
  const long ldk = (long)G * DP, ldv = (long)H * VP;
  const float* K = a.k + (long)row0 * ldk + (long)kh * DP;
  f32x4 kst[4 * NDG];
#pragma unroll
  for (int i = 0; i < 4 * NDG; ++i) {
    const int e = tid + 256 * i, r = e / (16 * NDG), d = 4 * (e % (16 * NDG));
    kst[i] = *reinterpret_cast<const f32x4*>(K + min(r, n - 1) * ldk + min(d, DP - 4));
  }
  const int xu = wave >= 2 * NDG ? wave - 2 * NDG : wave + 4 - 2 * NDG;     // this wave's unit of X
  const bool hasx = xu < 2 * c.ncg;
  float2 vf[4][4];
  if (hasx) {
    const int col = min(64 * (xu >> 1) + 4 * l16 + 2 * (xu & 1), VP - 2);   // past VP: unused columns
    const float* V = a.v + (long)row0 * ldv + (long)h * VP + col;
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        vf[k][i] = *reinterpret_cast<const float2*>(V + min(16 * k + 4 * g4 + i, n - 1) * ldv);
  }
  if (wave == 0) {                                     // running sums of the log decays
    float la = lane < n ? a.la[(long)(row0 + lane) * H + h] : 0.f;
    const float b = lane < n ? a.beta[(long)(row0 + lane) * H + h] : 0.f;
#pragma unroll
    for (int o = 1; o < DC; o <<= 1) {
      const float up = __shfl_up(la, o, 64);
      if (lane >= o) la += up;
    }
    sA[lane] = la;
    sb[lane] = b;
    c.cA[((long)ch * H + h) * DC + lane] = la;
  }
#pragma unroll
  for (int i = 0; i < 4 * NDG; ++i) {
    const int e = tid + 256 * i, r = e / (16 * NDG), d = 4 * (e % (16 * NDG));
    *reinterpret_cast<f32x4*>(&ks[r][d]) = d < DP ? kst[i] : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  __syncthreads();
  // the ten blocks of -L, two or three per wave: block p is row tile t, column tile u
  for (int p = wave; p < 10; p += 4) {
    const int t = p >= 6 ? 3 : p >= 3 ? 2 : p >= 1 ? 1 : 0, u = p - t * (t + 1) / 2;
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int b = 0; b < 4 * NDG; ++b)
      acc[b & 1] = mm(*reinterpret_cast<const f32x4*>(&ks[16 * t + l16][16 * b + 4 * g4]),
                      *reinterpret_cast<const f32x4*>(&ks[16 * u + l16][16 * b + 4 * g4]), acc[b & 1]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int tr = 16 * t + 4 * g4 + i, tc = 16 * u + l16;
      const float z = acc[0][i] + acc[1][i];
      Ls[tr][tc] = tc < tr ? -sb[tr] * expf(sA[tr] - sA[tc]) * z : 0.f;
    }
  }
  __syncthreads();
  {                                                    // column l16 of the wave's diagonal inverse
    float x[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float v = r == l16 ? 1.f : 0.f;
#pragma unroll
      for (int u = 0; u < r; ++u) v += Ls[16 * wave + r][16 * wave + u] * x[u];
      x[r] = v;
    }
    if (lane < 16) {                                   // after every lane's reads: one wave, in order
#pragma unroll
      for (int r = 0; r < 16; ++r) Ls[16 * wave + r][16 * wave + l16] = x[r];
    }
  }
  __syncthreads();
  // block column `wave` of T:  T_ij = T_ii sum_(j<=k<i) (-L_ik) T_kj
  f32x4 tc[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) tc[0][e] = Ls[16 * wave + 4 * g4 + e][16 * wave + l16];
#pragma unroll
  for (int i = 1; i < 4; ++i)
    if (wave + i < 4) {
      f32x4 r = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < i; ++k)
        r = mm(*reinterpret_cast<const f32x4*>(&Ls[16 * (wave + i) + l16][16 * (wave + k) + 4 * g4]),
               tc[k], r);
      tc[i] = mm(*reinterpret_cast<const f32x4*>(&Ls[16 * (wave + i) + l16][16 * (wave + i) + 4 * g4]),
                 r, f32x4{0.f, 0.f, 0.f, 0.f});
    }
  __syncthreads();
#pragma unroll
  for (int i = 1; i < 4; ++i)
    if (wave + i < 4) {
#pragma unroll
      for (int e = 0; e < 4; ++e) Ls[16 * (wave + i) + 4 * g4 + e][16 * wave + l16] = tc[i][e];
    }
  __syncthreads();
  f32x4 tf[4][4];                                      // row l16 of token tile i, tokens 16 k + 4 g4 ..
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int k = 0; k <= i; ++k)
      tf[i][k] = *reinterpret_cast<const f32x4*>(&Ls[16 * i + l16][16 * k + 4 * g4]);
  const long blk = ((long)ch * H + h) * 4;
  if (wave < 2 * NDG) {                                // Y^T = (diag(b exp A) K)^T T^T
    f32x4 o[2][4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      f32x4 kt[2], fs;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = 16 * k + 4 * g4 + i;
        const float f = sb[t] * expf(sA[t]);
        const int d = 64 * (wave >> 1) + 4 * dl_row(l16) + 2 * (wave & 1);
        const float2 z = *reinterpret_cast<const float2*>(&ks[t][d]);
        kt[0][i] = z.x;
        kt[1][i] = z.y;
        fs[i] = f;
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (h == kh * (H / G))
          put_frag(c.Kt, (((long)ch * G + kh) * (4 * NDG) + 2 * wave + j) * 4 + k, lane, kt[j]);
        kt[j] *= fs;
      }
#pragma unroll
      for (int i = k; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          o[j][i] = mm(kt[j], tf[i][k], k ? o[j][i] : f32x4{0.f, 0.f, 0.f, 0.f});
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        put_frag(c.Y, (blk + i) * (4 * NDG) + 2 * wave + j, lane, o[j][i]);
  }
  if (hasx) {                                          // X = T diag(b) V
    f32x4 o[2][4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      f32x4 vt[2];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float f = sb[16 * k + 4 * g4 + i];
        vt[0][i] = vf[k][i].x * f;
        vt[1][i] = vf[k][i].y * f;
      }
#pragma unroll
      for (int i = k; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          o[j][i] = mm(tf[i][k], vt[j], k ? o[j][i] : f32x4{0.f, 0.f, 0.f, 0.f});
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        put_frag(c.X, (blk + i) * (4 * c.ncg) + 2 * xu + j, lane, o[j][i]);
  }
}

// (2) one workgroup per (sequence, head, tile of 16 state columns).  Wave w owns tokens 16 w .. of u and
// NDG row tiles of the state; u and S pass between the waves through LDS.  The next chunk's operands
// are fetched between this one's products: issued in one go they held every wave up for 2800 to 6100
// cycles of the 9400 that a chunk took, 5800 now.  Two tiles per workgroup halve the reads but leave
// a quarter of the CUs idle here: 93 us instead of 77.
template <int NDG>
__global__ void __launch_bounds__(256)
delta_chunk_scan_kernel(DeltaArgs a, DeltaChunkArgs c) {
  constexpr int NB = 4 * NDG;                          // row tiles
  __shared__ __align__(16) f32x4 Ss[NB][64];
  __shared__ __align__(16) f32x4 Us[4][64];
  const int s = blockIdx.x, h = blockIdx.y, ct = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63, g4 = lane >> 4, l16 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int slot = a.slots[s];
  if (slot < 0) return;
  const int c0 = c.seq_first[s], c1 = c.seq_first[s + 1];
  if (c1 <= c0) return;
  const int H = a.H, G = a.G, D = a.D, Dv = a.Dv, kh = h / (H / G), nct = 4 * c.ncg;
  const bool fresh = a.positions[c.chunks[4 * c0 + 1]] == 0;
  const int tile0 = NDG * wave;                        // tiles tile0 .. + NDG - 1, one group's
  const int d0 = 64 * (tile0 >> 2) + (tile0 & 3);      // entries d0 + 4 x + o
  const int col = 64 * (ct >> 2) + 4 * l16 + (ct & 3);
  float* Sg = a.S + ((long)slot * H + h) * D * Dv;
  f32x4 S[NDG];
#pragma unroll
  for (int o = 0; o < NDG; ++o) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = d0 + 4 * (4 * i + g4) + o;
      S[o][i] = (!fresh && r < D && col < Dv) ? Sg[(long)r * Dv + col] : 0.f;
    }
    Ss[tile0 + o][lane] = S[o];
  }
  struct Op { f32x4 y[NB], x, k[NDG][4], ca; float ga; };
  auto load = [&](int ch, Op& p) {
    const long hb = (long)ch * H + h, gb = (long)ch * G + kh;
    p.ca = *reinterpret_cast<const f32x4*>(c.cA + hb * DC + 16 * wave + 4 * g4);
    p.ga = c.cA[hb * DC + DC - 1];
#pragma unroll
    for (int b = 0; b < NB; ++b) p.y[b] = frag(c.Y, (hb * 4 + wave) * NB + b, lane);
    p.x = frag(c.X, (hb * 4 + wave) * nct + ct, lane);
#pragma unroll
    for (int o = 0; o < NDG; ++o)
#pragma unroll
      for (int t = 0; t < 4; ++t) p.k[o][t] = frag(c.Kt, (gb * NB + tile0 + o) * 4 + t, lane);
  };
  auto step = [&](int ch, const Op& p) {
    const long hb = (long)ch * H + h;
#pragma unroll
    for (int o = 0; o < NDG; ++o)                      // the state before the chunk, for the outputs
      put_frag(c.wsS, (hb * NB + tile0 + o) * nct + ct, lane, S[o]);
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b & 1] = mm(p.y[b], Ss[b][lane], acc[b & 1]);
    f32x4 us = p.x - acc[0] - acc[1];
    put_frag(c.X, (hb * 4 + wave) * nct + ct, lane, us);
#pragma unroll
    for (int i = 0; i < 4; ++i) us[i] *= expf(p.ga - p.ca[i]);
    Us[wave][lane] = us;
#pragma unroll
    for (int i = 0; i < NB + 4 * NDG + 3; ++i) {       // one load per product
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
    __syncthreads();
    const float eg = expf(p.ga);
#pragma unroll
    for (int o = 0; o < NDG; ++o) {
      f32x4 v[2] = {S[o] * eg, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) v[tt & 1] = mm(p.k[o][tt], Us[tt][lane], v[tt & 1]);
      S[o] = v[0] + v[1];
      Ss[tile0 + o][lane] = S[o];
    }
    __syncthreads();
  };
  Op p0, p1;
  load(c0, p0);
  __syncthreads();
  for (int ch = c0; ch < c1; ch += 2) {
    load(min(ch + 1, c1 - 1), p1);
    step(ch, p0);
    if (ch + 1 >= c1) break;
    load(min(ch + 2, c1 - 1), p0);
    step(ch + 1, p1);
  }
#pragma unroll
  for (int o = 0; o < NDG; ++o)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = d0 + 4 * (4 * i + g4) + o;
      if (r < D && col < Dv) Sg[(long)r * Dv + col] = S[o][i];
    }
}

// (3) one workgroup per (chunk, head).  A wave owns one query tile and 64 columns; the waves of the same
// queries share the weights P through LDS, key tiles in turn.  The state is read once, straight to LDS,
// while the weights are formed.  Bound by the reads of a round of workgroups, which all come at its start.
template <typename T, int NDG, int NCG>
__global__ void __launch_bounds__(256 * NCG)
delta_chunk_out_kernel(DeltaArgs a, DeltaChunkArgs c) {
  constexpr int NB = 4 * NDG, NCT = 4 * NCG;
  __shared__ __align__(16) f32x4 Ss[NB * NCT][64];
  __shared__ __align__(16) f32x4 Ps[10][64];
  __shared__ float red[NCG][DC];
  const int ch = blockIdx.y, h = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int s = c.chunks[4 * ch], row0 = c.chunks[4 * ch + 1], n = c.chunks[4 * ch + 2];
  if (a.slots[s] < 0) return;
  const int H = a.H, G = a.G, Dv = a.Dv, DP = a.DP, kh = h / (H / G);
  const int g4 = lane >> 4, l16 = lane & 15, cg = wave % NCG, qt = wave / NCG;
  const long ldk = (long)G * DP, hb = (long)ch * H + h;
  // entries 64 g + 4 (4 i + g4) + j of a row, i = 0 .. 3: the k of tile j's fragment
  auto rows = [&](const float* base, int tile, f32x4 (&f)[NDG][4]) {
    const float* p = base + (long)(row0 + min(16 * tile + l16, n - 1)) * ldk + (long)kh * DP;
#pragma unroll
    for (int g = 0; g < NDG; ++g)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x4 z = *reinterpret_cast<const f32x4*>(p + min(64 * g + 16 * i + 4 * g4, DP - 4));
#pragma unroll
        for (int j = 0; j < 4; ++j) f[g][j][i] = z[j];
      }
  };
  f32x4 qf[NDG][4], kf[NDG][4];
  rows(a.q, qt, qf);
  rows(a.k, cg, kf);
  const float* cA = c.cA + hb * DC;
  const int tq = 16 * qt + l16;
  const float aq = cA[tq];
  const f32x4 ar = *reinterpret_cast<const f32x4*>(cA + 16 * qt + 4 * g4);
  f32x4 ak = *reinterpret_cast<const f32x4*>(cA + 16 * cg + 4 * g4);
  // the state goes to LDS while the weights are formed; nothing reads LDS until it is there
#pragma unroll
  for (int t = 0; t < NB; ++t) {
    const int tile = wave + 4 * NCG * t;
    __builtin_amdgcn_global_load_lds(
        (const __attribute__((address_space(1))) void*)(c.wsS + (hb * NB * NCT + tile) * 256 + 4 * lane),
        (__attribute__((address_space(3))) void*)&Ss[tile][0], 16, 0, 0);
  }
  if (DP & 63) {                                       // entries past DP are not the row's
#pragma unroll
    for (int g = 0; g < NDG; ++g)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (64 * g + 16 * i + 4 * g4 >= DP) {
#pragma unroll
          for (int j = 0; j < 4; ++j) qf[g][j][i] = 0.f;
        }
  }
  // P^T = K Q^T: its registers are the A operand of P u
  for (int kt = cg; kt <= qt; kt += NCG) {
    if (kt != cg) {
      rows(a.k, kt, kf);
      ak = *reinterpret_cast<const f32x4*>(cA + 16 * kt + 4 * g4);
    }
    f32x4 p[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int b = 0; b < NB; ++b) p[b & 1] = mm(kf[b >> 2][b & 3], qf[b >> 2][b & 3], p[b & 1]);
    f32x4 w;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int tk = 16 * kt + 4 * g4 + i;
      w[i] = tk <= tq && tk < n ? (p[0][i] + p[1][i]) * expf(aq - ak[i]) : 0.f;
    }
    Ps[qt * (qt + 1) / 2 + kt][lane] = w;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  f32x4 z[4], o[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) z[j] = frag(c.X, hb * 4 * NCT + 4 * cg + j, lane);
#pragma unroll
  for (int j = 0; j < 4; ++j) o[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      o[j] = mm(qf[b >> 2][b & 3], Ss[b * NCT + 4 * cg + j][lane], o[j]);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float e = expf(ar[i]);
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j][i] *= e;
  }
  for (int kt = 0; kt <= qt; ++kt) {
    f32x4 zn[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) zn[j] = frag(c.X, (hb * 4 + min(kt + 1, qt)) * NCT + 4 * cg + j, lane);
    const f32x4 w = Ps[qt * (qt + 1) / 2 + kt][lane];
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = mm(w, z[j], o[j]);
#pragma unroll
    for (int j = 0; j < 4; ++j) z[j] = zn[j];
  }
  // head RMS norm, weight, gate
  const int col = 64 * cg + 4 * l16;
  float ss[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float z = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) z += col + j < Dv ? o[j][i] * o[j][i] : 0.f;
    z += __shfl_xor(z, 1, 64);
    z += __shfl_xor(z, 2, 64);
    z += __shfl_xor(z, 4, 64);
    z += __shfl_xor(z, 8, 64);
    ss[i] = z;
    if (NCG == 2 && l16 == 0) red[cg][16 * qt + 4 * g4 + i] = z;
  }
  if (NCG == 2) __syncthreads();
  const T* NW = static_cast<const T*>(a.norm_w);
  const T* GT = static_cast<const T*>(a.g);
  T* Yo = static_cast<T*>(a.y);
  if (col >= Dv) return;
  float nw[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) nw[j] = ld_f32<T>(NW, min(col + j, Dv - 1)) * a.out_scale;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int tr = 16 * qt + 4 * g4 + i;
    if (tr >= n) continue;
    const float sq = NCG == 2 ? ss[i] + red[NCG - 1 - cg][tr] : ss[i];
    const float inv = 1.0f / sqrtf(sq / (float)Dv + a.eps);
    const long r = row0 + tr;
    const T* gp = GT + r * a.ldg + (long)h * Dv + col;
    T* yp = Yo + r * a.ldy + (long)h * Dv + col;
    if (c.vec) {
      typedef T T4 __attribute__((ext_vector_type(4)));
      const T4 gz = *reinterpret_cast<const T4*>(gp);
      T4 yz;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const T gj = gz[j];
        T v;
        st_f32<T>(&v, 0, o[j][i] * inv * nw[j] * dl_silu(ld_f32<T>(&gj, 0)));
        yz[j] = v;
      }
      *reinterpret_cast<T4*>(yp) = yz;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (col + j < Dv) st_f32<T>(yp, j, o[j][i] * inv * nw[j] * dl_silu(ld_f32<T>(gp, j)));
    }
  }
}

// As eia_delta_scan for sequences whose chunk list is given (chunks int32 [nchunk, 4]: sequence,
// first row, tokens (1 .. 64), 0; seq_first int32 [nseq + 1], indexed by sequence), with fp32
// workspaces Y [nchunk, H, 64, DQ], X [nchunk, H, 64, VQ], Kt [nchunk, G, DQ, 64], wsS [nchunk, H, DQ,
// VQ], cA [nchunk, H, 64], 16-byte aligned; DP and VP multiples of 16, at most 128, DQ and VQ the
// same rounded up to 64.
EIA_API int eia_delta_scan_chunked(const float* q, const float* k, const float* v, const float* la,
                                   const float* beta, int H, int G, int D, int Dv, int DP, int VP,
                                   const void* g, long ldg, const void* norm_w, float out_scale,
                                   float eps, float* S, const int* slots, const int* positions,
                                   void* y, long ldy, int nseq, const int* chunks,
                                   const int* seq_first, int nchunk, float* Y, float* X, float* Kt,
                                   float* wsS, float* cA, int is_bf16, hipStream_t st) {
  DeltaArgs a{q, k, v, la, beta, H, G, D, Dv, DP, VP, g, ldg, norm_w, out_scale, eps, S, slots,
              nullptr, positions, nullptr, y, ldy};
  if (!delta_args_ok(a, nseq) || nchunk < 0 || !chunks || !seq_first || !Y || !X || !Kt || !wsS || !cA ||
      DP % 16 || VP % 16)
    return EIA_BAD_SHAPE;
  if (DP > 128 || VP > 128) return EIA_UNSUPPORTED;
  if (nseq == 0 || nchunk == 0) return EIA_OK;
  const int ndg = (DP + 63) / 64, ncg = (VP + 63) / 64, es = is_bf16 ? 2 : 4;
  const bool vec = Dv % 4 == 0 && ldy % 4 == 0 && ldg % 4 == 0 &&
                   (reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(g)) % (4 * es) == 0;
  DeltaChunkArgs c{chunks, seq_first, Y, X, Kt, wsS, cA, ncg, vec};
  const dim3 gc(H, nchunk), b(256);
#define DO_GO(TT, A, B) \
  hipLaunchKernelGGL((delta_chunk_out_kernel<TT, A, B>), gc, dim3(256 * B), 0, st, a, c)
#define DO_DIMS(A, B)                                                                              \
  do {                                                                                             \
    hipLaunchKernelGGL(delta_chunk_solve_kernel<A>, gc, b, 0, st, a, c);                           \
    hipLaunchKernelGGL(delta_chunk_scan_kernel<A>, dim3(nseq, H, 4 * ncg), b, 0, st, a, c);        \
    if (is_bf16) DO_GO(bf16_t, A, B); else DO_GO(float, A, B);                                     \
  } while (0)
  if (ndg == 2) { if (ncg == 2) DO_DIMS(2, 2); else DO_DIMS(2, 1); }
  else { if (ncg == 2) DO_DIMS(1, 2); else DO_DIMS(1, 1); }
#undef DO_DIMS
#undef DO_GO
  EIA_LAUNCH_CHECK();
}
