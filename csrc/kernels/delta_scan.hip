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
// q, k, v, la and b arrive as the fp32 rows that delta_prep.hip leaves.  Everything here keeps fp32; matrix
// products are fp32 ones or take fp32 factors as sums of bf16 parts.
//
// A sequence whose first row of the step is position 0 starts from zeros whatever its slot held, so
// slots are reused without clearing.  Batch layout: sequence s owns rows [cu[s], cu[s+1])
// (cu == nullptr: row s).
#include <type_traits>
#include "eia_common.h"
#include "eia_delta_plan.h"

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
//   (1) T, X, Y and P_ts = exp(A_t - A_s) (q_t . k_s), s <= t, of every chunk, in parallel (T by 16-token
//       blocks, diagonal inverses first)
//   (2) a sequence's chunks in order, in parallel over heads and slices of the state's columns:
//       u = X - Y S,  o_t = exp(A_t) S^T q_t + sum_s P_ts u_s,  S <- exp(A_end) S + sum_t exp(A_end - A_t) k_t u_t^T
//   (3) norm, weight and gate of all outputs, in parallel
// Every exponent is <= 0.
//
// Layout.  Everything that passes between the kernels lies as the lanes of the next product take it, 16 bytes
// per lane and 1 KB per access.  A product over 32 rows (16x16x32) takes two tiles of 16, entry e of a
// lane from row 4 (lane / 16) + e % 4 of tile e / 4: two accumulators are an operand as they are, and so are rows
// of q 16 bytes at a time.
// Factors of the scan's products are three bf16 parts each (split3, six products for one: 6/16 of the
// matrix cycles of fp32 ones, and no less precise), made once where they are formed:
//   Y  [chunk, H, 4 token tiles, DP / 32, 3 parts]    A operand, rows tokens
//   Kt [chunk, G, DP / 16 tiles, 2, 3 parts]          A operand, rows dk
//   Qt [chunk, G, 4 token tiles, DP / 32, 3 parts]    A operand, rows tokens
//   P  [chunk, H, 6 blocks, 3 parts]                  A operand, rows queries: blocks of 32 keys that queries
//                                                     of a 16-token tile see, tiles in order (1, 1, 2, 2)
//   X  [chunk, H, 4 token tiles, VP / 16 tiles]       fp32, B operand, rows tokens
//   O  [chunk, 64, H, VP]                             fp32, outputs before their norm
// with DP rounded up to 64 and VP to 32; tile j of 32 columns holds columns 2 x + j.
// MI355X, 16 heads of 128 x 128 on 8, three prompts of 750 to 1500 tokens: 50 + 69 + 15 us
// ((1), (2), (3)).  Before, with fp32 products and the states between chunks and u in memory for a kernel that formed
// the outputs, 48 + 77 + 83 (the op: 197 -> 147).  S against 64 bits: 1.2e-7 .. 1.5e-7 where fp32 products left 1.3e-7 .. 1.6e-7.
// (1) and (3) are bound by their writes and reads (3.1, 4.4 TB/s), (2) by the chain of its chunks: 6000 cycles
// each, of which matrix products take 2700 of a SIMD's.
constexpr int DC = 64;                      // tokens per chunk
constexpr int DL = DC + 4;                  // LDS row pitch of the triangular blocks

struct DeltaChunkArgs {
  const int* chunks;                        // [nchunk, 4]: sequence, first row, tokens, unused
  const int* seq_first;                     // [nseq + 1]: first chunk of every sequence
  bf16_t *Y, *Kt, *Qt, *P; float *X, *O;    // as above
  float* cA;                                // [nchunk, H, 2, DC] exp(A_t), exp(A_end - A_t); A constant past the end
  int ncu, nseq;                            // units of 32 state columns
  int whole, parts;                         // the workgroups of (1): dn_solve
  DeltaSpread spread;                       // the workgroups of (2) over the XCDs
};

EIA_DEV f32x4 mm(f32x4 a, f32x4 b, f32x4 c) { return mfma_f32_k16(a, b, c); }
EIA_DEV f32x4 frag(const float* p, long tile, int lane) {
  return *reinterpret_cast<const f32x4*>(p + tile * 256 + 4 * lane);
}
EIA_DEV void put_frag(float* p, long tile, int lane, f32x4 v) {
  *reinterpret_cast<f32x4*>(p + tile * 256 + 4 * lane) = v;
}
struct Parts { bf16x8 p[3]; };
// split3 of eight numbers whose parts' sum is the number whatever it is: one that is not finite is its first
// part, one that rounds out of bf16 is cut instead.
EIA_DEV void split_whole(const float (&v)[8], Parts& f) {
  split3(v, f.p);
  float z = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) z += (float)f.p[2][e];
  if (__any(!(fabsf(z) < INFINITY))) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float h = (float)(bf16_t)v[e];
      if (fabsf(h) == INFINITY) h = __uint_as_float(__float_as_uint(v[e]) & 0xffff0000u);
      float r = v[e] - h;
      if (!(fabsf(r) < INFINITY)) r = 0.f;
      const bf16_t m = (bf16_t)r;
      f.p[0][e] = (bf16_t)h;
      f.p[1][e] = m;
      f.p[2][e] = (bf16_t)(r - (float)m);
    }
  }
}
// split3 with a cut first part: any finite number, in parts that are finite.  (Y and P that are not finite reach
// all columns alike, so that it does not matter which such number they become.)
EIA_DEV void split_cut(const float (&v)[8], Parts& f) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float h = __uint_as_float(__float_as_uint(v[e]) & 0xffff0000u), r = v[e] - h;
    const bf16_t m = (bf16_t)r;
    f.p[0][e] = (bf16_t)h;
    f.p[1][e] = m;
    f.p[2][e] = (bf16_t)(r - (float)m);
  }
}
EIA_DEV void put_parts(bf16_t* p, long block, int lane, f32x4 lo, f32x4 hi) {
  const float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  Parts f;
  split_cut(v, f);
#pragma unroll
  for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x8*>(p + ((block * 3 + i) * 64 + lane) * 8) = f.p[i];
}
EIA_DEV Parts parts(const bf16_t* p, long block, int lane) {
  Parts f;
#pragma unroll
  for (int i = 0; i < 3; ++i) f.p[i] = *reinterpret_cast<const bf16x8*>(p + ((block * 3 + i) * 64 + lane) * 8);
  return f;
}
EIA_DEV f32x4 whole(const Parts& f, int half) {        // of a tile of the two
  f32x4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    v[e] = ((float)f.p[0][4 * half + e] + (float)f.p[1][4 * half + e]) + (float)f.p[2][4 * half + e];
  return v;
}
// The six largest products of parts.  What is left out (m l, l m, l l) is below 2^-24 of the product where both numbers
// were split by rounding (m up to 2^-8 of the number, l up to 2^-17), below 2^-23 where one was cut (split_cut:
// 2^-7, 2^-16): about the one rounding of an fp32 product.
template <int N> EIA_DEV void mm6(const Parts& a, const Parts (&b)[N], f32x4 (&c)[N]) {
  constexpr int pa[6] = {0, 2, 1, 0, 1, 0}, pb[6] = {2, 0, 1, 1, 0, 0};
#pragma unroll
  for (int x = 0; x < 6; ++x)
#pragma unroll
    for (int j = 0; j < N; ++j) c[j] = mfma_bf16_k32(a.p[pa[x]], b[j].p[pb[x]], c[j]);
}
template <int N> EIA_DEV void mm6(const Parts (&a)[N], const Parts& b, f32x4 (&c)[N]) {
  constexpr int pa[6] = {0, 2, 1, 0, 1, 0}, pb[6] = {2, 0, 1, 1, 0, 0};
#pragma unroll
  for (int x = 0; x < 6; ++x)
#pragma unroll
    for (int j = 0; j < N; ++j) c[j] = mfma_bf16_k32(a[j].p[pa[x]], b.p[pb[x]], c[j]);
}
// A tile's four numbers per lane to their half of an operand in LDS.
EIA_DEV void put_half(bf16_t* lds, int half, int lane, f32x4 v) {
  bf16x2 a[3], b[3];
  split3(v[0], v[1], a[0], a[1], a[2]);
  split3(v[2], v[3], b[0], b[1], b[2]);
#pragma unroll
  for (int i = 0; i < 3; ++i)
    *reinterpret_cast<bf16x4*>(lds + (i * 64 + lane) * 8 + 4 * half) = bf16x4{a[i][0], a[i][1], b[i][0], b[i][1]};
}
EIA_DEV bool all_finite(f32x4 v) {
  bool ok = true;
#pragma unroll
  for (int e = 0; e < 4; ++e) ok &= fabsf(v[e]) < INFINITY;
  return ok;
}

// (1) one workgroup per (chunk, key head, part of its heads: dn_solve), those heads in turn.  K is staged in LDS in parts: the triangle and P
// take it by rows, Y and Kt by columns (transposing reads).  Waves 0 .. 3 form the triangle, its inverse and Y,
// a token tile each; waves 4 .. 7 meanwhile P, and then X in units of 32 columns.  k . k and q . k are
// formed once for all heads.  X takes fp32 products: a value that is not finite stays in its column and out
// of earlier tiles.  (Products of 32 tokens would carry it over: an operand's half that a tile does not meet is
// zero.)
constexpr int DHB = 8;                                 // heads whose sums of la are formed at a time
template <int NDG>                                     // groups of 64 dk
__global__ void __launch_bounds__(512, 4)
delta_chunk_solve_kernel(DeltaArgs a, DeltaChunkArgs c) {
  constexpr int KP = 64 * NDG + 8, PLANE = DC * KP, NK = 2 * NDG;
  __shared__ __align__(16) bf16_t ks[3 * PLANE];
  __shared__ __align__(16) float Ls[DC][DL];           // -L, then T
  __shared__ __align__(16) float sAs[DHB][DC], sbs[DHB][DC], sfs[DHB][DC];
  const DeltaSolveWg wg = dn_solve_place(blockIdx.x, a.G, c.whole, c.parts);
  const int ch = wg.chunk, kh = wg.kh, part = wg.part, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), w = wave & 3;
  const int row0 = c.chunks[4 * ch + 1], n = c.chunks[4 * ch + 2], slot = a.slots[c.chunks[4 * ch]];
  const int H = a.H, G = a.G, DP = a.DP, VP = a.VP, rep = H / G;
  const int x0 = dn_first_head(rep, wg.parts, part), nh = dn_first_head(rep, wg.parts, part + 1) - x0, h0 = kh * rep + x0;
  const int g4 = lane >> 4, l16 = lane & 15;
  const long ldk = (long)G * DP, ldv = (long)H * VP;
  const float* K = a.k + (long)row0 * ldk + (long)kh * DP;
  float kst[NDG][8];
#pragma unroll
  for (int i = 0; i < NDG; ++i) {
    const int e = tid + 512 * i, r = e / (8 * NDG), d = 8 * (e % (8 * NDG));
    const float* p = K + min(r, n - 1) * ldk + min(d, DP - 8);
#pragma unroll
    for (int x = 0; x < 8; x += 4) *reinterpret_cast<f32x4*>(&kst[i][x]) = *reinterpret_cast<const f32x4*>(p + x);
  }
  f32x4 q[2 * NK];
  if (wave >= 4) {                                     // q rows of tile w
    const float* Q = a.q + (long)row0 * ldk + (long)kh * DP + min(16 * w + l16, n - 1) * ldk;
#pragma unroll
    for (int b = 0; b < 2 * NK; ++b) q[b] = *reinterpret_cast<const f32x4*>(Q + min(16 * b + 4 * g4, DP - 4));
  }
#pragma unroll
  for (int i = 0; i < NDG; ++i) {
    const int e = tid + 512 * i, r = e / (8 * NDG), d = 8 * (e % (8 * NDG));
    if (d >= DP) {
#pragma unroll
      for (int x = 0; x < 8; ++x) kst[i][x] = 0.f;
    }
    Parts f;
    split_whole(kst[i], f);
#pragma unroll
    for (int p = 0; p < 3; ++p) *reinterpret_cast<bf16x8*>(ks + p * PLANE + r * KP + d) = f.p[p];
  }
  if (slot < 0) return;                                // (whole workgroup; the rows did not wait for it)
  __syncthreads();
  auto k_rows = [&](int t, int b) {                    // 32 dk of a token tile's rows, in order
    Parts f;
#pragma unroll
    for (int p = 0; p < 3; ++p) f.p[p] = *reinterpret_cast<const bf16x8*>(ks + p * PLANE + (16 * t + l16) * KP + 32 * b + 8 * g4);
    return f;
  };
  auto k_columns = [&](int x, int b) {                 // dk tile x, tokens of 32 as two tiles' rows
    Parts f;
    const bf16_t* p0 = ks + (32 * b + 4 * g4 + (l16 >> 2)) * KP + 16 * x + 4 * (l16 & 3);
#pragma unroll
    for (int p = 0; p < 3; ++p) f.p[p] = lds_columns(p0 + p * PLANE, p0 + p * PLANE + 16 * KP);
    return f;
  };
  // the ten blocks of k . k, two or three per wave: block p is row tile t, column tile u; q . k of a wave's
  // tile (keys by queries)
  f32x4 raw[4][1];
  auto block_of = [](int p, int& t, int& u) {
    t = p >= 6 ? 3 : p >= 3 ? 2 : p >= 1 ? 1 : 0;
    u = p - t * (t + 1) / 2;
  };
  auto weights = [&](auto tile) {                      // (the tile's number is a constant: no branches)
    constexpr int W = decltype(tile)::value;
#pragma unroll
    for (int b = 0; b < NK; ++b) {
      // (q comes as rows 4 g4 .. of two dk tiles; the keys' 32 dk are read the same way)
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = 32 * b + 16 * (e >> 2) + 4 * g4 < DP ? q[2 * b + (e >> 2)][e & 3] : 0.f;
      Parts y[1];
      split_cut(v, y[0]);
      if (part == 0) {
#pragma unroll
        for (int p = 0; p < 3; ++p)
          *reinterpret_cast<bf16x8*>(c.Qt + ((((((long)ch * G + kh) * 4 + W) * NK + b) * 3 + p) * 64 + lane) * 8) = y[0].p[p];
      }
#pragma unroll
      for (int u = 0; u <= W; ++u) {
        Parts f;
        const bf16_t* p0 = ks + (16 * u + l16) * KP + 32 * b + 4 * g4;
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          const bf16x4 lo = *reinterpret_cast<const bf16x4*>(p0 + p * PLANE);
          const bf16x4 hi = *reinterpret_cast<const bf16x4*>(p0 + p * PLANE + 16);
          f.p[p] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
        mm6(f, y, raw[u]);
      }
    }
  };
#pragma unroll
  for (int u = 0; u < 4; ++u) raw[u][0] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (wave < 4) {
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      int t, u;
      block_of(min(wave + 4 * x, 9), t, u);
#pragma unroll
      for (int b = 0; b < NK; ++b) {
        const Parts y[1] = {k_rows(u, b)};
        mm6(k_rows(t, b), y, raw[x]);
      }
    }
  } else if (w == 0) {
    weights(std::integral_constant<int, 0>());
  } else if (w == 1) {
    weights(std::integral_constant<int, 1>());
  } else if (w == 2) {
    weights(std::integral_constant<int, 2>());
  } else {
    weights(std::integral_constant<int, 3>());
  }
  mfma_settle(raw[0][0], raw[1][0]);
  mfma_settle(raw[2][0], raw[3][0]);
  if (part == 0 && wave < 4 * NDG) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const Parts f = k_columns(wave, b);
#pragma unroll
      for (int p = 0; p < 3; ++p)
        *reinterpret_cast<bf16x8*>(c.Kt + ((((((long)ch * G + kh) * (4 * NDG) + wave) * 2 + b) * 3 + p) * 64 + lane) * 8) = f.p[p];
    }
  }
  int here = lane;
  for (int x = 0; x < nh; ++x) {
    asm volatile("" : "+v"(here));                     // (addresses are formed anew: kept for the next head they spill)
    const int lane = here, g4 = lane >> 4, l16 = lane & 15, h = h0 + x;
    const long hb = (long)ch * H + h;
    const float *sA = sAs[x % DHB], *sb = sbs[x % DHB], *sf = sfs[x % DHB];
    const bool hasx = wave >= 4 && w < c.ncu;
    float2 vf[4][4];
    if (hasx) {
      const int col = min(32 * w + 2 * l16, VP - 2);   // past VP: unused columns
      const float* V = a.v + (long)row0 * ldv + (long)h * VP + col;
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          vf[k][i] = *reinterpret_cast<const float2*>(V + min(16 * k + 4 * g4 + i, n - 1) * ldv);
    }
    __syncthreads();                                   // the head before has been read
    if (x % DHB == 0) {
      if (x + wave < nh) {                             // running sums of the log decays
        const int hx = h + wave;
        const long hbx = (long)ch * H + hx;
        float la = lane < n ? a.la[(long)(row0 + lane) * H + hx] : 0.f;
        const float b = lane < n ? a.beta[(long)(row0 + lane) * H + hx] : 0.f;
#pragma unroll
        for (int o = 1; o < DC; o <<= 1) {
          const float up = __shfl_up(la, o, 64);
          if (lane >= o) la += up;
        }
        const float e = expf(la);
        sAs[wave][lane] = la;
        sbs[wave][lane] = b;
        sfs[wave][lane] = b * e;
        c.cA[hbx * 2 * DC + lane] = e;
        c.cA[(hbx * 2 + 1) * DC + lane] = expf(__shfl(la, DC - 1, 64) - la);
      }
      __syncthreads();
    }
    if (wave < 4) {                                    // -L
#pragma unroll
      for (int y = 0; y < 3; ++y)
        if (wave + 4 * y < 10) {
          int t, u;
          block_of(wave + 4 * y, t, u);
          const int tc = 16 * u + l16, t0 = 16 * t + 4 * g4;
          const f32x4 at = *reinterpret_cast<const f32x4*>(sA + t0), bt = *reinterpret_cast<const f32x4*>(sb + t0);
          const float ac = sA[tc];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float z = -bt[i] * expf(at[i] - ac) * raw[y][0][i];
            Ls[t0 + i][tc] = tc < t0 + i ? z : 0.f;
          }
        }
    }
    __syncthreads();
    if (wave < 4) {                                    // column l16 of the wave's diagonal inverse
      float z[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float v = r == l16 ? 1.f : 0.f;
#pragma unroll
        for (int u = 0; u < r; ++u) v += Ls[16 * wave + r][16 * wave + u] * z[u];
        z[r] = v;
      }
      if (lane < 16) {                                 // after every lane's reads: one wave, in order
#pragma unroll
        for (int r = 0; r < 16; ++r) Ls[16 * wave + r][16 * wave + l16] = z[r];
      }
    } else {                                           // P
      const int tq = 16 * w + l16;
      const float aq = sA[tq];
      f32x4 p[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const f32x4 ak = *reinterpret_cast<const f32x4*>(sA + 16 * u + 4 * g4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int tk = 16 * u + 4 * g4 + i;
          const float z = raw[u][0][i] * expf(aq - ak[i]);
          p[u][i] = tk <= tq && tk < n ? z : 0.f;
        }
      }
      const long first = hb * 6 + (w < 2 ? w : 2 * w - 2);
      put_parts(c.P, first, lane, p[0], p[1]);
      if (w >= 2) put_parts(c.P, first + 1, lane, p[2], p[3]);
    }
    __syncthreads();
    // block column `wave` of T:  T_ij = T_ii sum_(j<=k<i) (-L_ik) T_kj
    f32x4 tc[4];
    if (wave < 4) {
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
          mfma_settle(tc[i]);
        }
    }
    __syncthreads();
    if (wave < 4) {
#pragma unroll
      for (int i = 1; i < 4; ++i)
        if (wave + i < 4) {
#pragma unroll
          for (int e = 0; e < 4; ++e) Ls[16 * (wave + i) + 4 * g4 + e][16 * wave + l16] = tc[i][e];
        }
    }
    __syncthreads();
    if (wave < 4) {                                      // Y^T = K^T (T diag(b exp A))^T, token tile w
      Parts tp[2][1];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        float v[8];
#pragma unroll
        for (int y = 0; y < 2; ++y) {
          const int at = 32 * b + 16 * y + 4 * g4;
          const f32x4 f = *reinterpret_cast<const f32x4*>(&Ls[16 * w + l16][at]) * *reinterpret_cast<const f32x4*>(&sf[at]);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[4 * y + e] = 2 * b + y <= w ? f[e] : 0.f;
        }
        split_cut(v, tp[b][0]);
      }
#pragma unroll
      for (int d = 0; d < NK; ++d) {
        f32x4 o[2][1];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          o[j][0] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int b = 0; b < 2; ++b)
            if (2 * b <= w) {
              Parts f = k_columns(2 * d + j, b);
              if (2 * b == w) {                          // (the tile's own 16 tokens alone)
#pragma unroll
                for (int p = 0; p < 3; ++p)
#pragma unroll
                  for (int e = 4; e < 8; ++e) f.p[p][e] = (bf16_t)0.f;
              }
              mm6(f, tp[b], o[j]);
            }
        }
        mfma_settle(o[0][0], o[1][0]);
        put_parts(c.Y, (hb * 4 + w) * NK + d, lane, o[0][0], o[1][0]);
      }
    } else if (hasx) {                                   // X = T diag(b) V
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
        for (int i = k; i < 4; ++i) {
          const f32x4 t = *reinterpret_cast<const f32x4*>(&Ls[16 * i + l16][16 * k + 4 * g4]);
#pragma unroll
          for (int j = 0; j < 2; ++j)
            o[j][i] = mm(t, vt[j], k ? o[j][i] : f32x4{0.f, 0.f, 0.f, 0.f});
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          put_frag(c.X, (hb * 4 + i) * (2 * c.ncu) + 2 * w + j, lane, o[j][i]);
    }
  }
}

// (2) one workgroup per (sequence, head, 16 NC state columns).  Waves 0 .. 3 carry the state: wave w owns
// tokens 16 w .. of u and NDG row tiles of S.  Waves 4 .. 7, a half step behind, form the outputs of
// their 16 tokens from the same S and u while the first four wait for each other, so that neither goes to memory.
// u and S pass between the waves through LDS, in parts; a chunk has two steps, u and then S.
// An operand of the next chunk is requested where this chunk's has been used, a whole chunk ahead.
// S, u and the outputs are carried times 2^24, so that the third part of a number as small as 2^-126 is still one (parts
// of those of 2^-105, unscaled, left an error of 1.1e-6 in S, fp32 products 2.5e-7).
// 32 columns halve the reads per product, which a workgroup of 16 columns is bound by; 16 give twice the
// workgroups: dn_columns.  A sum that is not finite, which parts cannot follow, sends the workgroup through
// delta_scan_fp32: fp32 products from the start.
constexpr float DN_UP = 0x1p24f;
template <int NDG, int NC> struct ScanTiles {
  static constexpr int OP = 3 * 64 * 8;                // one operand, in bf16 numbers
  static constexpr int S = 2 * NDG * NC * OP, U = 2 * NC * OP;
  static constexpr int TOTAL = 2 * S + 2 * U;          // S twice, u weighted and not
};
// What the waves of (2) share: a group of tiles' state columns is ct0 .. ct0 + NC - 1.
struct ScanAt {
  int h, kh, ct0, c0, c1, last, wave, lane;
  bool fresh;
  float* Sg;
  EIA_DEV int rows(int ch) const { return ch + 1 < c1 ? DC : last; }
};

// (f: a power of two that S is multiplied by on its way)
template <int NDG, int NC>
EIA_DEV void scan_state(const DeltaArgs& a, const ScanAt& k, f32x4 (&S)[NDG][NC], bool put, float f) {
  const int g4 = k.lane >> 4, l16 = k.lane & 15, tile0 = NDG * (k.wave & 3);
#pragma unroll
  for (int o = 0; o < NDG; ++o)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 16 * (tile0 + o) + 4 * g4 + i;
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        const int ct = k.ct0 + j, col = 32 * (ct >> 1) + 2 * l16 + (ct & 1);
        const bool in = r < a.D && col < a.Dv;
        if (put) {
          if (in) k.Sg[(long)r * a.Dv + col] = S[o][j][i] * f;
        } else {
          S[o][j][i] = in && !k.fresh ? k.Sg[(long)r * a.Dv + col] : 0.f;
        }
      }
    }
  if (!put) {                                          // (beside its load each product would wait for it)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int o = 0; o < NDG; ++o)
#pragma unroll
      for (int j = 0; j < NC; ++j) S[o][j] *= f;
  }
}
template <int NC>
EIA_DEV void scan_put_out(const DeltaArgs& a, const DeltaChunkArgs& c, const ScanAt& k, int ch, const f32x4 (&o)[NC], float f) {
  const int g4 = k.lane >> 4, l16 = k.lane & 15, n = k.rows(ch), VQ = 32 * c.ncu;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = 16 * (k.wave & 3) + 4 * g4 + i;
    float* p = c.O + (((long)ch * DC + t) * a.H + k.h) * VQ + 32 * (k.ct0 >> 1) + 2 * l16 + (k.ct0 & 1);
    if (t < n) {
      if constexpr (NC == 2) *reinterpret_cast<float2*>(p) = float2{o[0][i] * f, o[1][i] * f};
      else *p = o[0][i] * f;
    }
  }
}
template <int NDG, int NC>
EIA_DEV void delta_scan_fp32(const DeltaArgs& a, const DeltaChunkArgs& c, const ScanAt& k, bf16_t* lds) {
  constexpr int NB = 4 * NDG;
  f32x4* Ss = reinterpret_cast<f32x4*>(lds);           // [NB][NC][64]
  f32x4* Us = Ss + NB * NC * 64;                       // [2][4][NC][64]: weighted, not
  const int lane = k.lane, g4 = lane >> 4, w = k.wave & 3, nct = 2 * c.ncu;
  const bool carry = k.wave < 4;
  f32x4 S[NDG][NC];
  if (carry) {
    scan_state<NDG, NC>(a, k, S, false, 1.f);
#pragma unroll
    for (int o = 0; o < NDG; ++o)
#pragma unroll
      for (int j = 0; j < NC; ++j) Ss[((NDG * w + o) * NC + j) * 64 + lane] = S[o][j];
  }
  __syncthreads();
  for (int ch = k.c0; ch < k.c1; ++ch) {
    const long hb = (long)ch * a.H + k.h, gb = (long)ch * a.G + k.kh;
    const float* cA = c.cA + hb * 2 * DC;
    const f32x4 ea = *reinterpret_cast<const f32x4*>(cA + 16 * w + 4 * g4);
    const f32x4 ew = *reinterpret_cast<const f32x4*>(cA + DC + 16 * w + 4 * g4);
    const float eg = cA[DC - 1];
    f32x4 o[NC];
#pragma unroll
    for (int j = 0; j < NC; ++j) o[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const f32x4 f = carry ? whole(parts(c.Y, (hb * 4 + w) * (2 * NDG) + (b >> 1), lane), b & 1)
                            : whole(parts(c.Qt, (gb * 4 + w) * (2 * NDG) + (b >> 1), lane), b & 1);
#pragma unroll
      for (int j = 0; j < NC; ++j) o[j] = mm(f, Ss[(b * NC + j) * 64 + lane], o[j]);
    }
    if constexpr (NC == 2) mfma_settle(o[0], o[1]);
    else mfma_settle(o[0]);
    if (carry) {
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        const f32x4 u = frag(c.X, (hb * 4 + w) * nct + k.ct0 + j, lane) - o[j];
        Us[((4 + w) * NC + j) * 64 + lane] = u;
        Us[(w * NC + j) * 64 + lane] = u * ew;
      }
    } else {
#pragma unroll
      for (int j = 0; j < NC; ++j) o[j] *= ea;
    }
    __syncthreads();
    if (carry) {
#pragma unroll
      for (int x = 0; x < NDG; ++x) {
#pragma unroll
        for (int j = 0; j < NC; ++j) S[x][j] *= eg;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const f32x4 f = whole(parts(c.Kt, (gb * NB + NDG * w + x) * 2 + (t >> 1), lane), t & 1);
#pragma unroll
          for (int j = 0; j < NC; ++j) S[x][j] = mm(f, Us[(t * NC + j) * 64 + lane], S[x][j]);
        }
#pragma unroll
        for (int j = 0; j < NC; ++j) Ss[((NDG * w + x) * NC + j) * 64 + lane] = S[x][j];
      }
    } else {
      for (int t = 0; t <= w; ++t) {
        const f32x4 f = whole(parts(c.P, hb * 6 + (w < 2 ? w : 2 * w - 2 + (t >> 1)), lane), t & 1);
#pragma unroll
        for (int j = 0; j < NC; ++j) o[j] = mm(f, Us[((4 + t) * NC + j) * 64 + lane], o[j]);
        if constexpr (NC == 2) mfma_settle(o[0], o[1]);
        else mfma_settle(o[0]);
      }
      scan_put_out<NC>(a, c, k, ch, o, 1.f);
    }
    __syncthreads();
  }
  if (carry) scan_state<NDG, NC>(a, k, S, true, 1.f);
}

template <int NDG, int NC>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
delta_chunk_scan_kernel(DeltaArgs a, DeltaChunkArgs c) {
  constexpr int NB = 4 * NDG, NK = 2 * NDG;            // row tiles; pairs of them
  using L = ScanTiles<NDG, NC>;
  __shared__ __align__(16) bf16_t lds[L::TOTAL];
  const int tid = threadIdx.x, lane = tid & 63, g4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), w = wave & 3;
  // the column groups of a head meet the same Y and P, the heads of a key head the same Kt and Qt (dn_spread)
  const int nct = 2 * c.ncu, ncg = nct / NC, rep = a.H / a.G;
  const DeltaWg wg = dn_place(blockIdx.x, c.spread);
  const int kv = wg.kv, in = wg.in;
  if (kv >= c.nseq * a.G || in >= c.spread.per_kv) return;
  const int s = kv / a.G, h = kv % a.G * rep + in / ncg, slot = a.slots[s];
  if (slot < 0) return;
  const int c0 = c.seq_first[s], c1 = c.seq_first[s + 1];
  if (c1 <= c0) return;
  const ScanAt k{h, kv % a.G, in % ncg * NC, c0, c1, c.chunks[4 * c1 - 2], wave, lane,
                 a.positions[c.chunks[4 * c0 + 1]] == 0, a.S + ((long)slot * a.H + h) * a.D * a.Dv};
  auto Ss = [&](int buf, int kb, int j) { return lds + buf * L::S + (kb * NC + j) * L::OP; };
  auto Us = [&](int raw, int kb, int j) { return lds + 2 * L::S + raw * L::U + (kb * NC + j) * L::OP; };
  auto operands = [&](const bf16_t* p, Parts (&f)[NC]) {
#pragma unroll
    for (int j = 0; j < NC; ++j) f[j] = parts(p + j * L::OP, 0, lane);
  };
  // stands between reads of LDS and products that do not need them: left alone, the compiler moves each read
  // to the product that it is for
  auto in_order = [] { __builtin_amdgcn_sched_barrier(0); };
  bool bad = false;
  f32x4 S[NDG][NC];
  if (wave < 4) {
    const int tile0 = NDG * w;
    auto put_state = [&](int buf) {
#pragma unroll
      for (int o = 0; o < NDG; ++o)
#pragma unroll
        for (int j = 0; j < NC; ++j) put_half(Ss(buf, (tile0 + o) >> 1, j), (tile0 + o) & 1, lane, S[o][j]);
    };
    Parts y[NK], kt[NDG][2];
    f32x4 x[NC], ew;
    float eg;
    auto load_y = [&](int ch, int b) { y[b] = parts(c.Y, (((long)ch * a.H + h) * 4 + w) * NK + b, lane); };
    auto load_k = [&](int ch, int o, int b) {
      kt[o][b] = parts(c.Kt, (((long)ch * a.G + k.kh) * NB + tile0 + o) * 2 + b, lane);
    };
    auto load_x = [&](int ch) {
      const long hb = (long)ch * a.H + h;
      ew = *reinterpret_cast<const f32x4*>(c.cA + (hb * 2 + 1) * DC + 16 * w + 4 * g4);
      eg = c.cA[hb * 2 * DC + DC - 1];
#pragma unroll
      for (int j = 0; j < NC; ++j) x[j] = frag(c.X, (hb * 4 + w) * nct + k.ct0 + j, lane);
    };
#pragma unroll
    for (int b = 0; b < NK; ++b) load_y(c0, b);
    load_x(c0);
#pragma unroll
    for (int o = 0; o < NDG; ++o)
#pragma unroll
      for (int b = 0; b < 2; ++b) load_k(c0, o, b);
    scan_state<NDG, NC>(a, k, S, false, DN_UP);
    put_state(0);
    __syncthreads();
    for (int ch = c0; ch < c1; ++ch) {
      const int buf = (ch - c0) & 1, nx = min(ch + 1, c1 - 1);
      f32x4 acc[2][NC];
#pragma unroll
      for (int j = 0; j < NC; ++j) acc[0][j] = acc[1][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      Parts f[2][NC];
      operands(Ss(buf, 0, 0), f[0]);
#pragma unroll
      for (int b = 0; b < NK; ++b) {
        if (b + 1 < NK) operands(Ss(buf, b + 1, 0), f[(b + 1) & 1]);
        in_order();
        mm6(y[b], f[b & 1], acc[b & 1]);
        load_y(nx, b);
        in_order();
      }
      f32x4 u[NC];
      const float decay = eg;
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        u[j] = x[j] * DN_UP - acc[0][j] - acc[1][j];
        put_half(Us(0, w >> 1, j), w & 1, lane, u[j] * ew);
      }
      load_x(nx);
      __syncthreads();
      operands(Us(0, 0, 0), f[0]);
      operands(Us(0, 1, 0), f[1]);
      in_order();
#pragma unroll
      for (int o = 0; o < NDG; ++o)
#pragma unroll
        for (int j = 0; j < NC; ++j) S[o][j] *= decay;
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int o = 0; o < NDG; ++o) {
          mm6(kt[o][b], f[b], S[o]);
          load_k(nx, o, b);
        }
#pragma unroll
      for (int j = 0; j < NC; ++j) put_half(Us(1, w >> 1, j), w & 1, lane, u[j]);
      put_state(buf ^ 1);
      __syncthreads();
    }
#pragma unroll
    for (int o = 0; o < NDG; ++o)
#pragma unroll
      for (int j = 0; j < NC; ++j) bad |= !all_finite(S[o][j]);
  } else {
    f32x4 ea, o[NC];
    Parts p[2], q[NK];
    const int blocks = w < 2 ? 1 : 2, first = w < 2 ? w : 2 * w - 2;
    auto load_q = [&](int ch) {
#pragma unroll
      for (int b = 0; b < NK; ++b) q[b] = parts(c.Qt, (((long)ch * a.G + k.kh) * 4 + w) * NK + b, lane);
      ea = *reinterpret_cast<const f32x4*>(c.cA + ((long)ch * a.H + h) * 2 * DC + 16 * w + 4 * g4);
    };
    auto load_p = [&](int ch) {
#pragma unroll
      for (int b = 0; b < 2; ++b)
        if (b < blocks) p[b] = parts(c.P, ((long)ch * a.H + h) * 6 + first + b, lane);
    };
    auto finish = [&](int ch) {                        // P u, and out with it
      Parts f[2][NC];
#pragma unroll
      for (int b = 0; b < 2; ++b)
        if (b < blocks) operands(Us(1, b, 0), f[b]);
#pragma unroll
      for (int b = 0; b < 2; ++b)
        if (b < blocks) mm6(p[b], f[b], o);
      if constexpr (NC == 2) mfma_settle(o[0], o[1]);
      else mfma_settle(o[0]);
#pragma unroll
      for (int j = 0; j < NC; ++j) bad |= !all_finite(o[j]);
      scan_put_out<NC>(a, c, k, ch, o, 1.f / DN_UP);
    };
    load_q(c0);
    __syncthreads();
    for (int ch = c0; ch < c1; ++ch) {
      const int buf = (ch - c0) & 1;
      if (ch > c0) finish(ch - 1);
      load_p(ch);
      __syncthreads();
      f32x4 acc[2][NC];
#pragma unroll
      for (int j = 0; j < NC; ++j) acc[0][j] = acc[1][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      Parts f[2][NC];
      operands(Ss(buf, 0, 0), f[0]);
#pragma unroll
      for (int b = 0; b < NK; ++b) {
        if (b + 1 < NK) operands(Ss(buf, b + 1, 0), f[(b + 1) & 1]);
        in_order();
        mm6(q[b], f[b & 1], acc[b & 1]);
        in_order();
      }
#pragma unroll
      for (int j = 0; j < NC; ++j) o[j] = (acc[0][j] + acc[1][j]) * ea;
      load_q(min(ch + 1, c1 - 1));
      __syncthreads();
    }
    finish(c1 - 1);
  }
  if (__syncthreads_or(bad)) {
    delta_scan_fp32<NDG, NC>(a, c, k, lds);
    return;
  }
  if (wave < 4) scan_state<NDG, NC>(a, k, S, true, 1.f / DN_UP);
}

// (3) Norm, weight and gate of the outputs: LN lanes per token and head, two heads each; the heads come first in the
// grid, so that those of a key head run on the XCD that formed them where G is eight.  Bound by memory.  (Four heads, chunks
// first: three prompts of 155 tokens, 8 heads 32.9 -> 30.8 us, three of up to 1500, 16 heads 146.0 -> 145.2.)  All five
// reads of a thread are in flight together (the second head's behind the first one's gate: the op 128.6 us instead of 125,
// both with the instructions' own reciprocals).  Root and silu are formed with divisions and expf also of bf16 outputs:
// with v_rsq, v_rcp and __expf the op takes 128.0 instead of 130.6 us, but of gates below -87.3 v_rcp leaves zero.
constexpr int DN_HEADS = 2;
template <typename T, int LN, bool VEC>
__global__ void __launch_bounds__(256)
delta_chunk_norm_kernel(DeltaArgs a, DeltaChunkArgs c) {
  constexpr int NH = DN_HEADS;
  typedef T T4 __attribute__((ext_vector_type(4)));
  const int ch = blockIdx.y, sub = threadIdx.x % LN, t = blockIdx.z * (256 / LN) + threadIdx.x / LN;
  // no branch before the store: the outputs are asked for beside the chunk, the gates beside its slot
  const int row0 = c.chunks[4 * ch + 1], n = c.chunks[4 * ch + 2], slot = a.slots[c.chunks[4 * ch]];
  const int col = 4 * sub, Dv = a.Dv, VQ = 32 * c.ncu;
  const long r = row0 + min(t, n - 1);
  f32x4 o[NH];
  T4 gv[NH], nw;
  const T *GT = static_cast<const T*>(a.g) + r * a.ldg, *NW = static_cast<const T*>(a.norm_w);
  auto four = [&](const T* p) {
    if constexpr (VEC) return *reinterpret_cast<const T4*>(p + min(col, Dv - 4));
    T4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = p[min(col + j, Dv - 1)];
    return v;
  };
#pragma unroll
  for (int x = 0; x < NH; ++x) {
    const int h = min((int)blockIdx.x * NH + x, a.H - 1);
    o[x] = *reinterpret_cast<const f32x4*>(c.O + (((long)ch * DC + t) * a.H + h) * VQ + min(col, VQ - 4));
    gv[x] = four(GT + (long)h * Dv);
  }
  nw = four(NW);
  T4 v[NH];
#pragma unroll
  for (int x = 0; x < NH; ++x) {
    float sq = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) sq += col + j < Dv ? o[x][j] * o[x][j] : 0.f;
#pragma unroll
    for (int b = 1; b < LN; b <<= 1) sq += __shfl_xor(sq, b, 64);
    const float inv = 1.0f / sqrtf(sq / (float)Dv + a.eps);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      v[x][j] = (T)(o[x][j] * inv * ((float)nw[j] * a.out_scale) * dl_silu((float)gv[x][j]));
    asm volatile("" : "+v"(v[x]));                     // (formed here: else the gates are asked for behind the branch)
  }
  if (slot < 0 || t >= n || col >= Dv) return;
#pragma unroll
  for (int x = 0; x < NH; ++x) {
    const int h = (int)blockIdx.x * NH + x;
    if (h >= a.H) break;
    T* yp = static_cast<T*>(a.y) + r * a.ldy + (long)h * Dv + col;
    if constexpr (VEC) {
      *reinterpret_cast<T4*>(yp) = v[x];
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (col + j < Dv) yp[j] = v[x][j];
    }
  }
}

// State columns per workgroup of (2), in tiles of 16, for nunit workgroups of 32 columns: 16 while that leaves
// no CU (256) with two workgroups, 32 beyond.  Heads of 128, the whole op in us with 16 / 32 columns: 64
// workgroups of 32 (one prompt of 4096 tokens, 16 heads) 186 / 216, 128 (two of 1500) 105 / 113, 192 (three)
// 146 / 130, 256 (four of 1024) 123 / 108, 1024 (sixteen of 256) 145 / 119; heads of 64: 128 54 / 57, 192 128 / 118.
static int dn_columns(int nunit) { return nunit > 128 ? 2 : 1; }

// As eia_delta_scan for sequences whose chunk list is given (chunks int32 [nchunk, 4]: sequence,
// first row, tokens (64, of a sequence's last chunk 1 .. 64), 0; seq_first int32 [nseq + 1], indexed by sequence), with workspaces,
// 16-byte aligned: bf16 Y [nchunk, H, 64, DQ, 3], Kt and Qt [nchunk, G, DQ, 64, 3], P [nchunk, H, 6, 3, 512], fp32
// X [nchunk, H, 64, VQ], O [nchunk, 64, H, VQ], cA [nchunk, H, 2, 64]; DP and VP multiples of 16, at most
// 128; DQ: DP rounded up to 64, VQ: VP rounded up to 32.
EIA_API int eia_delta_scan_chunked(const float* q, const float* k, const float* v, const float* la,
                                   const float* beta, int H, int G, int D, int Dv, int DP, int VP,
                                   const void* g, long ldg, const void* norm_w, float out_scale,
                                   float eps, float* S, const int* slots, const int* positions,
                                   void* y, long ldy, int nseq, const int* chunks,
                                   const int* seq_first, int nchunk, void* Y, void* Kt, void* Qt, void* P,
                                   float* X, float* O, float* cA, int is_bf16, hipStream_t st) {
  DeltaArgs a{q, k, v, la, beta, H, G, D, Dv, DP, VP, g, ldg, norm_w, out_scale, eps, S, slots,
              nullptr, positions, nullptr, y, ldy};
  if (!delta_args_ok(a, nseq) || nchunk < 0 || !chunks || !seq_first || !Y || !X || !Kt || !Qt || !P || !O || !cA ||
      DP % 16 || VP % 16)
    return EIA_BAD_SHAPE;
  if (DP > 128 || VP > 128) return EIA_UNSUPPORTED;
  if (nseq == 0 || nchunk == 0) return EIA_OK;
  const int ndg = (DP + 63) / 64, ncu = (VP + 31) / 32, es = is_bf16 ? 2 : 4;
  const bool vec = Dv % 4 == 0 && ldy % 4 == 0 && ldg % 4 == 0 &&
                   (reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(g) |
                    reinterpret_cast<uintptr_t>(norm_w)) % (4 * es) == 0;
  const DeltaSolve solve = dn_solve(G, nchunk, H / G);
  DeltaChunkArgs c{chunks, seq_first, static_cast<bf16_t*>(Y), static_cast<bf16_t*>(Kt), static_cast<bf16_t*>(Qt),
                   static_cast<bf16_t*>(P), X, O, cA, ncu, nseq, solve.whole, solve.parts, {}};
  const dim3 gc((unsigned)solve.blocks), b(256);
  const int nc = dn_columns(nseq * H * ncu);
  c.spread = dn_spread(G, 2 * ncu / nc * (H / G));
  const int grid = dn_grid(nseq * G, c.spread);
#define DO_SCAN(A, C) \
  hipLaunchKernelGGL((delta_chunk_scan_kernel<A, C>), dim3(grid), dim3(512), 0, st, a, c)
#define DO_DIMS(A)                                                                                 \
  do {                                                                                             \
    hipLaunchKernelGGL(delta_chunk_solve_kernel<A>, gc, dim3(512), 0, st, a, c);                           \
    if (nc == 2) DO_SCAN(A, 2); else DO_SCAN(A, 1);                                                \
  } while (0)
#define DO_NORM_V(TT, LN, V)                                                                       \
  hipLaunchKernelGGL((delta_chunk_norm_kernel<TT, LN, V>), dim3((H + DN_HEADS - 1) / DN_HEADS, nchunk, DC * LN / 256), b, 0, st, a, c)
#define DO_NORM(TT, LN) do { if (vec) DO_NORM_V(TT, LN, true); else DO_NORM_V(TT, LN, false); } while (0)
  if (ndg == 2) DO_DIMS(2); else DO_DIMS(1);
  if (is_bf16) { if (VP > 64) DO_NORM(bf16_t, 32); else DO_NORM(bf16_t, 16); }
  else { if (VP > 64) DO_NORM(float, 32); else DO_NORM(float, 16); }
#undef DO_NORM
#undef DO_NORM_V
#undef DO_DIMS
#undef DO_SCAN
  EIA_LAUNCH_CHECK();
}
