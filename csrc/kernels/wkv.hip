// Linear-attention recurrence with per-channel data-dependent decay (RWKV-style "wkv" mixing)
// on per-sequence state slots.
//
// State of a sequence and layer: S [heads, dk, dv] fp32 and the previous token's layer input
// prev [width] fp32.  A sequence whose first scheduled position is 0 starts from zeros whatever
// its slot held before, so slots are reused without clearing.
//
//   eia_token_shift_mix : mix_s[t] = x[t] + (x[t-1] - x[t]) * mu_s  for NS streams (x[-1] from
//                         the slot; zeros at position 0)
//   eia_wkv_scan        : w = exp(-exp(dec + w0));  o = (S + diag(u) k v^T)^T r;
//                         S = diag(w) S + k v^T;  y = o / rms(o) * norm_w * silu(g)
//                         and prev <- x[last token of the step]
//
// Batch layout: sequence s owns rows [cu[s], cu[s+1]) (cu == nullptr: row s).  All recurrence
// math is fp32; activations are bf16 or fp32 (template T).
#include "eia_chunks.h"

EIA_DEV int find_seq(const int* cu, int nseq, int row) {
  int lo = 0, hi = nseq - 1;               // largest s with cu[s] <= row
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (cu[mid] <= row) lo = mid; else hi = mid - 1;
  }
  return lo;
}

template <typename T>
__global__ void __launch_bounds__(256)
token_shift_mix_kernel(const float* __restrict__ x, const T* __restrict__ mu, int NS,
                       const float* __restrict__ prev_state, const int* __restrict__ slots,
                       const int* __restrict__ cu, int nseq, const int* __restrict__ positions,
                       T* __restrict__ out, long out_ss, int W) {
  const int row = blockIdx.x;
  const int s = cu ? find_seq(cu, nseq, row) : row;
  const int first = cu ? cu[s] : row;
  const float* cur = x + (long)row * W;
  const float* prv = nullptr;
  if (row > first) prv = cur - W;
  else if (positions[row] > 0 && slots[s] >= 0) prv = prev_state + (long)slots[s] * W;
  for (int c = threadIdx.x; c < W; c += blockDim.x) {
    const float a = cur[c];
    const float d = (prv ? prv[c] : 0.f) - a;
    for (int k = 0; k < NS; ++k)
      st_f32<T>(out + (long)k * out_ss + (long)row * W, c, a + d * ld_f32<T>(mu, (long)k * W + c));
  }
}

// x fp32 [rows, W]; mu [NS, W]; out [NS, rows, W] (stream stride out_ss elements).
EIA_API int eia_token_shift_mix(const float* x, const void* mu, int NS, const float* prev_state,
                                const int* slots, const int* cu, int nseq, const int* positions,
                                void* out, long out_ss, int rows, int W, int is_bf16,
                                hipStream_t st) {
  if (rows < 0 || W < 1 || NS < 1 || nseq < 1) return EIA_BAD_SHAPE;
  if (rows == 0) return EIA_OK;
  if (is_bf16)
    hipLaunchKernelGGL((token_shift_mix_kernel<bf16_t>), dim3(rows), dim3(256), 0, st, x,
                       (const bf16_t*)mu, NS, prev_state, slots, cu, nseq, positions,
                       (bf16_t*)out, out_ss, W);
  else
    hipLaunchKernelGGL((token_shift_mix_kernel<float>), dim3(rows), dim3(256), 0, st, x,
                       (const float*)mu, NS, prev_state, slots, cu, nseq, positions, (float*)out,
                       out_ss, W);
  EIA_LAUNCH_CHECK();
}

struct WkvArgs {
  const void *r, *k, *v, *g; long ld;       // [rows, H*D] each, row stride ld
  const float* dec; long ld_dec;            // [rows, H*D] fp32 decay pre-activation (without w0)
  const void *w0, *u, *norm_w;              // [H*D] each
  float* S;                                 // [slots, H, D, D]
  float* prev; const float* x; int W;       // prev [slots, W]; x fp32 [rows, W]
  const int* slots; const int* cu; const int* positions; const int* seq_lens;
  void* y; long ldy;                        // [rows, H*D]
  float eps; int H, D;
  int split;                                // rows from which a sequence takes the chunk-parallel form (0: never)
};

// One workgroup per (sequence, head), 4 x max(64, DMAX) threads: thread (q, j) owns rows
// [q DMAX/4, (q+1) DMAX/4) of column j of S in registers and walks the sequence's tokens in
// order.  Tokens are staged TC at a time: r, k, decay, v and the gate of TC tokens go to LDS
// (coalesced over the channels; channels >= D hold zeros so the dk loops run branch-free), the
// recurrence runs TC steps on LDS broadcasts leaving four partial outputs per token and column,
// and the partials are then summed, RMS-normed per head, weighted and gated -- so a token costs
// a quarter pass over dk per thread instead of a global-memory round trip.
template <typename T, int DMAX, bool SPLIT>
__global__ void __launch_bounds__(4 * (DMAX < 64 ? 64 : DMAX))
wkv_scan_kernel(WkvArgs a) {
  constexpr int DP = DMAX < 64 ? 64 : DMAX;          // threads per quarter
  constexpr int DQ = DMAX / 4;                       // dk rows per thread
  constexpr int TC = DMAX <= 64 ? 16 : DMAX <= 128 ? 8 : 4;
  constexpr int NWV = DP / 64;                       // waves per quarter
  __shared__ __align__(16) float sr[TC][DMAX], sk[TC][DMAX], sw[TC][DMAX], su[DMAX];
  __shared__ float sv[TC][DMAX], sg[TC][DMAX], po[TC][4][DP];
  __shared__ float red[4][NWV];
  const int s = blockIdx.x, h = blockIdx.y, D = a.D;
  const int q = threadIdx.x / DP, j = threadIdx.x % DP;
  const int slot = a.slots[s];
  if (slot < 0 || (a.seq_lens && a.seq_lens[s] <= 0)) return;
  const int lo = a.cu ? a.cu[s] : s, hi = a.cu ? a.cu[s + 1] : s + 1;
  if (hi <= lo || (SPLIT && hi - lo >= a.split)) return;
  const bool fresh = a.positions[lo] == 0;
  const bool live = j < D, mine = j < DMAX;
  float* Sg = a.S + ((long)slot * a.H + h) * D * D;
  const int i0 = q * DQ;
  float S[DQ];
#pragma unroll
  for (int i = 0; i < DQ; ++i)
    S[i] = (!fresh && i0 + i < D && live) ? Sg[(long)(i0 + i) * D + j] : 0.f;
  const long hc = (long)h * D;
  if (q == 0 && mine) su[j] = live ? ld_f32<T>(static_cast<const T*>(a.u), hc + j) : 0.f;
  const float w0 = live ? ld_f32<T>(static_cast<const T*>(a.w0), hc + j) : 0.f;
  const float nw = live ? ld_f32<T>(static_cast<const T*>(a.norm_w), hc + j) : 0.f;
  const T* R = static_cast<const T*>(a.r);
  const T* K = static_cast<const T*>(a.k);
  const T* V = static_cast<const T*>(a.v);
  const T* G = static_cast<const T*>(a.g);
  T* Y = static_cast<T*>(a.y);
  const float inv_d = 1.0f / (float)D;
  for (int base = lo; base < hi; base += TC) {
    const int nt = min(TC, hi - base);
    __syncthreads();                       // the previous chunk's LDS reads are done
    if (mine) {
#pragma unroll
      for (int tt = 0; tt < TC / 4; ++tt) {            // quarter q stages tokens q, q + 4, ...
        const int t = tt * 4 + q;
        if (t < nt) {
          const long row = base + t;
          float r = 0.f, k = 0.f, w = 0.f, v = 0.f, g = 0.f;
          if (live) {
            r = ld_f32<T>(R, row * a.ld + hc + j);
            k = ld_f32<T>(K, row * a.ld + hc + j);
            w = expf(-expf(a.dec[row * a.ld_dec + hc + j] + w0));
            v = ld_f32<T>(V, row * a.ld + hc + j);
            g = ld_f32<T>(G, row * a.ld + hc + j);
          }
          sr[t][j] = r;
          sk[t][j] = k;
          sw[t][j] = w;
          sv[t][j] = v;
          sg[t][j] = g;
        }
      }
    }
    __syncthreads();
    for (int t = 0; t < nt; ++t) {
      const float v = mine ? sv[t][j] : 0.f;
      float o = 0.f;
#pragma unroll
      for (int i = 0; i < DQ; ++i) {
        const float kv = sk[t][i0 + i] * v;
        o += sr[t][i0 + i] * (S[i] + su[i0 + i] * kv);
        S[i] = sw[t][i0 + i] * S[i] + kv;
      }
      po[t][q][j] = o;
    }
    __syncthreads();
    // quarter q finishes tokens q, q + 4, ...: sum of the partials, head RMS norm, weight, gate
#pragma unroll
    for (int tt = 0; tt < TC / 4; ++tt) {
      const int t = tt * 4 + q;
      const bool ok = t < nt && live;
      const float o = ok ? po[t][0][j] + po[t][1][j] + po[t][2][j] + po[t][3][j] : 0.f;
      float ss = wave_sum(o * o);
      if (NWV > 1) {
        __syncthreads();
        if ((j & 63) == 0) red[q][j >> 6] = ss;
        __syncthreads();
        ss = 0.f;
#pragma unroll
        for (int x = 0; x < NWV; ++x) ss += red[q][x];
      }
      if (ok) {
        const float g = sg[t][j];
        const float gate = g / (1.0f + expf(-g));
        st_f32<T>(Y, (long)(base + t) * a.ldy + hc + j, o / sqrtf(ss * inv_d + a.eps) * nw * gate);
      }
    }
  }
  if (live) {
#pragma unroll
    for (int i = 0; i < DQ; ++i)
      if (i0 + i < D) Sg[(long)(i0 + i) * D + j] = S[i];
  }
  if (h == 0) {
    const float* last = a.x + (long)(hi - 1) * a.W;
    float* p = a.prev + (long)slot * a.W;
    for (int c = threadIdx.x; c < a.W; c += blockDim.x) p[c] = last[c];
  }
}

// split > 0: sequences of that many rows or more are left out (eia_wkv_scan_chunked takes them).
EIA_API int eia_wkv_scan(const void* r, const void* k, const void* v, const void* g, long ld,
                         const float* dec, long ld_dec, const void* w0, const void* u,
                         const void* norm_w, float* S, float* prev, const float* x, int W,
                         const int* slots, const int* cu, const int* positions,
                         const int* seq_lens, void* y, long ldy, float eps, int nseq, int H, int D,
                         int split, int is_bf16, hipStream_t st) {
  if (nseq < 0 || H < 1 || D < 1 || W < 1 || split < 0) return EIA_BAD_SHAPE;
  if (D > 256) return EIA_UNSUPPORTED;
  if (nseq == 0) return EIA_OK;
  WkvArgs a{r, k, v, g, ld, dec, ld_dec, w0, u, norm_w, S, prev, x, W, slots, cu, positions,
            seq_lens, y, ldy, eps, H, D, split};
  dim3 grid(nseq, H);
#define WKV_LAUNCH(TT, DM)                                                                 \
  do {                                                                                     \
    const dim3 block(4 * (DM < 64 ? 64 : DM));                                             \
    if (split) hipLaunchKernelGGL((wkv_scan_kernel<TT, DM, true>), grid, block, 0, st, a); \
    else hipLaunchKernelGGL((wkv_scan_kernel<TT, DM, false>), grid, block, 0, st, a);      \
  } while (0)
  if (is_bf16) {
    if (D <= 32) WKV_LAUNCH(bf16_t, 32);
    else if (D <= 64) WKV_LAUNCH(bf16_t, 64);
    else if (D <= 128) WKV_LAUNCH(bf16_t, 128);
    else WKV_LAUNCH(bf16_t, 256);
  } else {
    if (D <= 32) WKV_LAUNCH(float, 32);
    else if (D <= 64) WKV_LAUNCH(float, 64);
    else if (D <= 128) WKV_LAUNCH(float, 128);
    else WKV_LAUNCH(float, 256);
  }
#undef WKV_LAUNCH
  EIA_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------------------------
// Chunk-parallel form for prompt portions (D <= 64).  The kernel above walks a sequence with one
// workgroup per head (0.5 us a token); here a sequence's rows are cut into chunks of WC tokens and,
// with l_t = log2 w_t = -exp(dec_t + w0) / ln 2 per channel, S the state before a chunk and sums over the
// chunk's tokens,
//
//   U   = sum_s 2^(sum_(s<x) l_x) k_s v_s^T                            (1) per chunk, in parallel
//   S' = 2^(sum_x l_x) S + U                                           (2) a sequence's chunks in order
//   o_t = (r_t 2^(sum_(x<t) l_x)) S + sum_(s<t) P_ts v_s + (r_t . u . k_t) v_t
//   P_ts = sum_channels r_t k_s 2^(sum_(s<x<t) l_x)                    (3) per chunk, in parallel
//
// All products are fp32 matrix-core products.  Exponents are sums of the l_x that they cover, never
// differences, so they are <= 0 and keep their precision behind tokens that forget almost everything; a
// pair of tokens meets through the edges of the 8-token blocks between them,
//   P_ts = (r_t 2^(block start .. t)) . (whole blocks between) . (k_s 2^(s .. block end)),
// inside a block see eia_chunks.h.  (With differences of a running sum over eight tokens, l cut at -40: 8e-7
// instead of 1.2e-7 against 64 bits where every second token forgets, in the same time.)
//
// Bound by instruction issue (exponentials, conversions, fp32 products; 31 us of vector and 15 us of
// matrix issue in (3)), not by memory: one 4096-token prompt, 32 heads of 64, bf16 takes 98 us on an
// MI355X (25 + 17 + 62 in a trace), 2091 us token by token.  All that a workgroup reads is asked for before
// it waits for any: with a row of r, u and half the decays behind branches and conversions, the state at
// its products and a wait for each stored row 105 us (27 + 15 + 64).
constexpr int WC = 64;                      // tokens per chunk
constexpr int WD = 64;                      // widest head

struct WkvChunkArgs {
  float* U;                                 // [numbers, H, WD, WD]: contribution, then state before
  float* L;                                 // [numbers, H, WD]: sums of l
  int nseq;
};

// The chunk of number x; false where there is none or the sequence is skipped.
EIA_DEV bool wkv_chunk(const WkvArgs& a, int nseq, int x, int& s, int& row0, int& n) {
  return chunk_of<WC>(a.cu, nseq, x, s, row0, n) && a.cu[s + 1] - a.cu[s] >= a.split && a.slots[s] >= 0 &&
         (!a.seq_lens || a.seq_lens[s] > 0);
}

// A chunk's [WC][WD] tile of r, k or v on its way to LDS, zero past the chunk and past D: requested
// by load, stored as fp32 by store.  VEC: 16-byte loads (D == WD, rows on 16-byte addresses).
template <typename T, bool VEC>
struct WkvTile {
  typedef __attribute__((ext_vector_type(4))) int i32x4;
  static constexpr int E = VEC ? 16 / sizeof(T) : 1, N = WC * WD / (256 * E);
  alignas(16) T v[N][E];
  EIA_DEV void load(const void* src, long ld, long hc, int row0, int n, int D) {
#pragma unroll
    for (int x = 0; x < N; ++x) {
      const int u = threadIdx.x + 256 * x, t = u / (WD / E), i = E * (u % (WD / E));
      const T* p = static_cast<const T*>(src) + (row0 + min(t, n - 1)) * ld + hc + (VEC ? i : min(i, D - 1));
      if constexpr (VEC) *reinterpret_cast<f32x4*>(v[x]) = *reinterpret_cast<const f32x4*>(p);
      else v[x][0] = *p;
    }
  }
  // (what lies past the chunk is masked away: behind a branch the compiler would ask for some of it only there, and wait)
  EIA_DEV void store(float* tile, int n, int D) const {
#pragma unroll
    for (int x = 0; x < N; ++x) {
      const int u = threadIdx.x + 256 * x, t = u / (WD / E), i = E * (u % (WD / E));
      const int keep = t < n && (VEC || i < D) ? -1 : 0;
      if constexpr (VEC && sizeof(T) == 2) {
        const i32x4 q = *reinterpret_cast<const i32x4*>(v[x]) & keep;
#pragma unroll
        for (int e = 0; e < 4; e += 2)
          *reinterpret_cast<i32x4*>(tile + tile_at<WD>(t, i + 2 * e)) =
              i32x4{q[e] << 16, q[e] & (int)0xffff0000, q[e + 1] << 16, q[e + 1] & (int)0xffff0000};
      } else if constexpr (VEC) {
        *reinterpret_cast<i32x4*>(tile + tile_at<WD>(t, i)) = *reinterpret_cast<const i32x4*>(v[x]) & keep;
      } else {
        tile[tile_at<WD>(t, i)] = __int_as_float(__float_as_int((float)v[x][0]) & keep);
      }
    }
  }
  // Whether one of this thread's values is infinite or no number.
  EIA_DEV bool wild() const {
    float z = 0.f;
#pragma unroll
    for (int x = 0; x < N; ++x)
#pragma unroll
      for (int e = 0; e < E; ++e) z += 0.f * (float)v[x][e];
    return z != 0.f;
  }
};

// Base-2 log decays of channel i, tokens t0 .. t0 + 15 (0 past the chunk and past D): a weight then
// costs one v_exp_f32.
// ask: requests of the caller that go out behind the decays' own.  HOLD: nothing is waited for before all of them are out;
// else the compiler chooses.
template <typename T, bool HOLD, typename Ask>
EIA_DEV void wkv_decays(const WkvArgs& a, long hc, int row0, int n, int t0, int i, float (&l)[16], Ask&& ask) {
  const int ic = min(i, a.D - 1);
  const float w0 = ld_f32<T>(static_cast<const T*>(a.w0), hc + ic);
#pragma unroll
  for (int t = 0; t < 16; ++t) l[t] = a.dec[(long)(row0 + min(t0 + t, n - 1)) * a.ld_dec + hc + ic];
  ask();
  if constexpr (HOLD) __builtin_amdgcn_sched_barrier(0);                   // (else the second half of them behind the first's exponentials)
#pragma unroll
  for (int t = 0; t < 16; ++t)
    l[t] = (i < a.D && t0 + t < n) ? -1.4426950408889634f * expf(l[t] + w0) : 0.f;
}

// (1) Wave w forms rows 16 w .. of U.  A lane of a product over tokens holds value columns
// 4 (lane % 16) + j in its j-th tile, here and in (3): U, S and v move in 16-byte units.
template <typename T, bool VEC>
__global__ void __launch_bounds__(256)
wkv_chunk_state_kernel(WkvArgs a, WkvChunkArgs c) {
  __shared__ __align__(16) float sk[WC * WD], sv[WC * WD];
  __shared__ float stot[4][WD];
  int s, row0, n;
  if (!wkv_chunk(a, c.nseq, chunk_number(), s, row0, n)) return;
  const int h = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int l16 = lane & 15, g4 = lane >> 4;
  const long hc = (long)h * a.D;
  WkvTile<T, VEC> tk, tv;
  float l[16];
  auto rows = [&] {
    tk.load(a.k, a.ld, hc, row0, n, a.D);
    tv.load(a.v, a.ld, hc, row0, n, a.D);
  };
  // (rows by elements: 32 registers more, and two workgroups a CU, where they come behind the decays)
  if constexpr (!VEC) rows();
  wkv_decays<T, VEC>(a, hc, row0, n, 16 * w, lane, l, [&] { if constexpr (VEC) rows(); });
  float tot = 0.f;
#pragma unroll
  for (int t = 0; t < 16; ++t) tot += l[t];
  stot[w][lane] = tot;
  tk.store(sk, n, a.D);
  tv.store(sv, n, a.D);
  __syncthreads();
  float after = 0.f;                                   // sum of l from the next token on
  for (int b = 3; b > w; --b) after += stot[b][lane];
#pragma unroll
  for (int t = 15; t >= 0; --t) {
    sk[tile_at<WD>(16 * w + t, lane)] *= __builtin_amdgcn_exp2f(after);
    after += l[t];
  }
  const long at = (long)chunk_number() * a.H + h;
  if (w == 0) c.L[at * WD + lane] = after;
  __syncthreads();
  f32x4 acc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    if (16 * b >= n) break;
    f32x4 ka, vb[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t = 16 * b + 4 * g4 + e;
      ka[e] = sk[tile_at<WD>(t, 16 * w + l16)];
      const f32x4 x = tile_get<WD>(sv, t, 4 * l16);
#pragma unroll
      for (int j = 0; j < 4; ++j) vb[j][e] = x[j];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = mfma_f32_k16(ka, vb[j], acc[j]);
  }
  float* U = c.U + at * WD * WD + (long)(16 * w + 4 * g4) * WD + 4 * l16;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    *reinterpret_cast<f32x4*>(U + i * WD) = f32x4{acc[0][i], acc[1][i], acc[2][i], acc[3][i]};
}

// (2) Four columns of a state row per thread; the slot receives the state after the last chunk.
__global__ void __launch_bounds__(256)
wkv_chunk_scan_kernel(WkvArgs a, WkvChunkArgs c) {
  const int s = chunk_number(), h = blockIdx.x % a.H;
  if (s >= c.nseq) return;
  const int slot = a.slots[s], lo = a.cu[s], hi = a.cu[s + 1];
  if (slot < 0 || hi - lo < a.split || (a.seq_lens && a.seq_lens[s] <= 0)) return;
  const int e = 4 * (blockIdx.x / a.H * 256 + threadIdx.x), i = e / WD, j = e % WD, D = a.D;
  const long x0 = lo / WC + s;
  const int nc = (hi - lo + WC - 1) / WC;
  float* Sg = a.S + ((long)slot * a.H + h) * D * D + (long)i * D + j;
  f32x4 S = {0.f, 0.f, 0.f, 0.f};
  if (a.positions[lo] != 0 && i < D) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (j + k < D) S[k] = Sg[k];
  }
  float* U = c.U + (x0 * a.H + h) * WD * WD + e;
  const float* L = c.L + (x0 * a.H + h) * WD + i;
  chunk_walk(U, (long)a.H * WD * WD, L, (long)a.H * WD, nc, S);
  if (i < D) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (j + k < D) Sg[k] = S[k];
  }
  if (h == 0) {                                        // the last token's layer input
    const float* last = a.x + (long)(hi - 1) * a.W;
    float* p = a.prev + (long)slot * a.W;
    for (int k = e / 4; k < a.W; k += WD * WD / 4) p[k] = last[k];
  }
}

// (3) Wave w forms the outputs of tokens 16 w .. (later tokens meet more keys: which wave takes them
// rotates with the chunk, so that no SIMD gets all of them).  50 KiB of LDS: three workgroups per CU.
// WIDE: gate, weight and output rows can be taken four at a time.
template <typename T, bool VEC, bool WIDE>
__global__ void __launch_bounds__(256, 3)
wkv_chunk_out_kernel(WkvArgs a, WkvChunkArgs c) {
  __shared__ __align__(16) float sr[WC * WD], sk[WC * WD], sAv[WC * WD];
  __shared__ __align__(16) float se[8][WD], su[WD];    // decays over whole 8-token blocks; u
  __shared__ int swild;                                // a value of the chunk is not finite
  int s, row0, n;
  if (!wkv_chunk(a, c.nseq, chunk_number(), s, row0, n)) return;
  const int h = blockIdx.x, lane = threadIdx.x & 63, w = ((threadIdx.x >> 6) + blockIdx.y) & 3;
  const int D = a.D, l16 = lane & 15, g4 = lane >> 4, t0 = 16 * w;
  const long hc = (long)h * D;
  WkvTile<T, VEC> tr, tk, tv;
  const T u = static_cast<const T*>(a.u)[hc + min(lane, D - 1)];
  if constexpr (VEC) __builtin_amdgcn_sched_barrier(0);
  float l[16];
  wkv_decays<T, VEC>(a, hc, row0, n, t0, lane, l, [&] {
    tr.load(a.r, a.ld, hc, row0, n, D);
    tk.load(a.k, a.ld, hc, row0, n, D);
    tv.load(a.v, a.ld, hc, row0, n, D);
  });
  tr.store(sr, n, D);
  tk.store(sk, n, D);
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    float tot = 0.f;
#pragma unroll
    for (int t = 8 * b; t < 8 * b + 8; ++t) tot += l[t];
    se[2 * w + b][lane] = __builtin_amdgcn_exp2f(tot);
  }
  block_edges<false>(l, sAv, t0, lane);
  su[lane] = lane < D ? (float)u : 0.f;                // (from every wave: no load behind a branch)
  if (threadIdx.x == 0) swild = 0;
  __syncthreads();
  f32x4 p = {0.f, 0.f, 0.f, 0.f};                      // weights inside the wave's 8-token blocks
  if (t0 < n) {
    float b = 0.f;                                     // r . u . k of token t0 + l16
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
      const int d = 16 * g4 + i;
      const f32x4 x = tile_get<WD>(sr, t0 + l16, d) * tile_get<WD>(sk, t0 + l16, d) *
                      *reinterpret_cast<const f32x4*>(&su[d]);
      b += x[0] + x[1] + x[2] + x[3];
    }
    b += __shfl_xor(b, 16, 64);
    b += __shfl_xor(b, 32, 64);
    p = block_weights<false>(sr, sk, sAv, l, b, t0, lane);
  }
  __syncthreads();
  // r_t <- r_t 2^(block start .. t), k_s <- k_s 2^(s .. block end), 8-token blocks; v moves in
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    float pre = 0.f, suf = 0.f;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      sr[tile_at<WD>(t0 + 8 * b + t, lane)] *= __builtin_amdgcn_exp2f(pre);
      pre += l[8 * b + t];
      sk[tile_at<WD>(t0 + 8 * b + 7 - t, lane)] *= __builtin_amdgcn_exp2f(suf);
      suf += l[8 * b + 7 - t];
    }
  }
  tv.store(sAv, n, D);
  if (tv.wild()) swild = 1;
  __syncthreads();
  if (t0 >= n) return;
  f32x4 rt[4], o[4], pq = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int i = 16 * b + 4 * g4;
    rt[b] = tile_get<WD>(sr, t0 + l16, i);
    pq = mfma_f32_k16(tile_get<WD>(sk, t0 + l16, i), rt[b], pq);
    if (l16 >= 8) rt[b] *= *reinterpret_cast<const f32x4*>(&se[2 * w][i]);
    o[b] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // (weights are formed transposed, keys x queries: their registers are the A operand of P v)
  if (l16 >= 8 && g4 < 2) p += pq;                     // second 8 queries, first 8 keys
  const bool wild = swild;
  // the first half of the state is on its way during the weights' products, the rest during its own
  const float* S = c.U + ((long)chunk_number() * a.H + h) * WD * WD + (long)4 * g4 * WD + 4 * l16;
  f32x4 sq[2][2][4];
  auto ask = [&](int half) {
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int e = 0; e < 4; ++e) sq[half][x][e] = *reinterpret_cast<const f32x4*>(S + (16 * (2 * half + x) + e) * WD);
  };
  ask(0);
  for (int b = w;;) {
    if (wild && b == w) {
      // key by key: in the product a later token's value times a weight of zero would be no number
#pragma unroll 1
      for (int k4 = 0; k4 < 4; ++k4)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const f32x4 x = tile_get<WD>(sAv, t0 + 4 * k4 + e, 4 * l16);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float pt = __shfl(p[e], 16 * k4 + 4 * g4 + i, 64);
            if (4 * k4 + e > 4 * g4 + i) continue;
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j][i] += pt * x[j];
          }
        }
    } else {
      f32x4 vb[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const f32x4 x = tile_get<WD>(sAv, 16 * b + 4 * g4 + e, 4 * l16);
#pragma unroll
        for (int j = 0; j < 4; ++j) vb[j][e] = x[j];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = mfma_f32_k16(p, vb[j], o[j]);
    }
    if (--b < 0) break;
    p = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < 4; ++x) {                      // keys of block b; rt: from its end on
      const int i = 16 * x + 4 * g4;
      const f32x4 e1 = *reinterpret_cast<const f32x4*>(&se[2 * b + 1][i]);
      f32x4 kk = tile_get<WD>(sk, 16 * b + l16, i);
      if (l16 < 8) kk *= e1;
      p = mfma_f32_k16(kk, rt[x], p);
      rt[x] *= e1 * *reinterpret_cast<const f32x4*>(&se[2 * b][i]);
    }
  }
  ask(1);
  // the gates and the norm's weight are on their way during the last products
  typedef T T4 __attribute__((ext_vector_type(4)));
  T4 gv[4], nw;
  {
    const T* G = static_cast<const T*>(a.g) + hc;
    const T* NW = static_cast<const T*>(a.norm_w) + hc;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const T* q = G + (long)(row0 + min(t0 + 4 * g4 + i, n - 1)) * a.ld;
      if constexpr (WIDE) {
        gv[i] = *reinterpret_cast<const T4*>(q + 4 * l16);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) gv[i][j] = q[min(4 * l16 + j, D - 1)];
      }
    }
    if constexpr (WIDE) {
      nw = *reinterpret_cast<const T4*>(NW + 4 * l16);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) nw[j] = NW[min(4 * l16 + j, D - 1)];
    }
  }
  if (row0 != a.cu[s] || a.positions[a.cu[s]] != 0) {  // (a fresh sequence's first chunk: S = 0)
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      f32x4 sb[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < 4; ++j) sb[j][e] = sq[x >> 1][x & 1][e][j];
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = mfma_f32_k16(rt[x], sb[j], o[j]);
    }
  }
  mfma_settle(o);
  T4 yv[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {                        // head RMS norm (zeros past D), weight, gate
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) ss += o[j][i] * o[j][i];
    const float inv = 1.0f / sqrtf(row16_sum(ss) / (float)D + a.eps);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float g = (float)gv[i][j];
      yv[i][j] = (T)(o[j][i] * inv * (float)nw[j] *
                     (sizeof(T) == 2 ? g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)) : g / (1.0f + expf(-g))));
    }
    // formed here: behind the branches below, each row's gate would be waited for, and the store before it with it
    asm volatile("" : "+v"(yv[i]));
  }
  T* Y = static_cast<T*>(a.y) + (long)(row0 + t0 + 4 * g4) * a.ldy + hc + 4 * l16;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (t0 + 4 * g4 + i >= n) break;
    if constexpr (WIDE) {
      *reinterpret_cast<T4*>(Y + i * a.ldy) = yv[i];
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (4 * l16 + j < D) Y[i * a.ldy + j] = yv[i][j];
    }
  }
}

template <typename T, bool VEC, bool WIDE>
static void wkv_chunked(const WkvArgs& a, const WkvChunkArgs& c, int rows, hipStream_t st) {
  const dim3 gc = chunk_grid(rows / WC + c.nseq, a.H), gs = chunk_grid(c.nseq, a.H * (WD * WD / 1024));
  hipLaunchKernelGGL((wkv_chunk_state_kernel<T, VEC>), gc, dim3(256), 0, st, a, c);
  hipLaunchKernelGGL(wkv_chunk_scan_kernel, gs, dim3(256), 0, st, a, c);
  hipLaunchKernelGGL((wkv_chunk_out_kernel<T, VEC, WIDE>), gc, dim3(256), 0, st, a, c);
}

// As eia_wkv_scan for D <= 64 with cu given, for the sequences of split rows or more; rows: cu[nseq] at most; workspaces U
// [rows / 64 + nseq, H, 64, 64] and L [rows / 64 + nseq, H, 64] fp32.
EIA_API int eia_wkv_scan_chunked(const void* r, const void* k, const void* v, const void* g,
                                 long ld, const float* dec, long ld_dec, const void* w0,
                                 const void* u, const void* norm_w, float* S, float* prev,
                                 const float* x, int W, const int* slots, const int* cu,
                                 const int* positions, const int* seq_lens, void* y, long ldy,
                                 float eps, int nseq, int rows, int H, int D, int split, float* U,
                                 float* L, int is_bf16, hipStream_t st) {
  if (nseq < 0 || rows < 0 || H < 1 || D < 1 || W < 1 || split < 1 || !cu || !U || !L)
    return EIA_BAD_SHAPE;
  if (D > WD || H > 65535) return EIA_UNSUPPORTED;
  if (nseq == 0 || rows == 0) return EIA_OK;
  WkvArgs a{r, k, v, g, ld, dec, ld_dec, w0, u, norm_w, S, prev, x, W, slots, cu, positions,
            seq_lens, y, ldy, eps, H, D, split};
  const WkvChunkArgs c{U, L, nseq};
  // rows of r, k and v by 16 bytes, gates, weights and outputs four at a time, each where they lie so: one flag for both
  // took a prompt of 4096 tokens, 32 heads of 64, with weights off 8 bytes from 101 to 108 us
  const int es = is_bf16 ? 2 : 4;
  const uintptr_t any = (uintptr_t)r | (uintptr_t)k | (uintptr_t)v | (uintptr_t)(ld * es);
  const uintptr_t io = (uintptr_t)g | (uintptr_t)y | (uintptr_t)norm_w | (uintptr_t)(ld * es) | (uintptr_t)(ldy * es);
  const bool vec = D == WD && any % 16 == 0, wide = D == WD && io % (4 * es) == 0;
#define WKV_GO(T)                                                                                   \
  do {                                                                                              \
    if (vec && wide) wkv_chunked<T, true, true>(a, c, rows, st);                                    \
    else if (vec) wkv_chunked<T, true, false>(a, c, rows, st);                                      \
    else if (wide) wkv_chunked<T, false, true>(a, c, rows, st);                                     \
    else wkv_chunked<T, false, false>(a, c, rows, st);                                              \
  } while (0)
  if (is_bf16) WKV_GO(bf16_t); else WKV_GO(float);
#undef WKV_GO
  EIA_LAUNCH_CHECK();
}
