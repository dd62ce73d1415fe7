// Windowed attention over prompt portions (bf16), for layers without head mixing or a distance term:
// the caches, masks, weights and epilogues of window_attention.hip, on v_mfma_f32_32x32x16_bf16 with
// keys and values shared through LDS.
//
// A workgroup of four waves owns HPW heads of one kv head (4, 2 or 1: as many as divide the group) and
// 128 / HPW queries of one sequence; wave w takes head w % HPW and 32 queries, so that a 64-key tile
// of K and V^T staged once in LDS feeds 128 (query, head) rows.  (The 16-query form in
// window_attention.hip reads every operand of every head from the caches: 64 bytes of operand loads
// per matrix instruction and lane, which bound it at 77 .. 127 TFLOP/s.)
//
// Per wave and tile: S^T[key, q] = K Q^T with Q^T in registers; a lane owns one query column, so the
// softmax is lane-local but for one exchange with lane ^ 32; key rows are fed with bits 2 and 3 of
// their number swapped, which makes a lane's accumulators eight consecutive keys, the operand of
// O^T += V^T P^T.  The weights stay fp32: they enter the second product as a bf16 high part plus a
// bf16 remainder, and the normaliser sums the fp32 values.  The running maximum moves only when a
// tile exceeds it by 2^8.  Tile i + 1 is fetched into registers before tile i is multiplied and
// written to the other LDS buffer behind it; one barrier per tile.  Rows are padded by 16 bytes, so
// that the sixteen rows of an operand read lie on different banks.  The page of a tile is looked up a tile
// before its fetch, and keys are read four fragments ahead of their products.
//
// Four ragged prompts of up to 2048 tokens, 16 heads of 128 on 4, window 1024, soft-capped: 65 us on an
// MI355X (249 us in the 16-query form); one 4096-token causal prompt, 8 heads on 2: 65 + 9 us in
// parts (459 us).  With the page looked up by the fetch, each read in front of its product and no priorities 72 and 75 +
// 12 us (parts of 13 tiles; 70 + 12 with both): of a tile's 5600 cycles (two workgroups on a CU) the fetch took 1100.  What bounds it now is issue: 1540 cycles of
// matrix products and 1800 (soft-capped 3300) of vector instructions a tile and wave, two waves on a SIMD.
// Tiles straight to LDS (128 registers' worth of staging less, but one more wait at a time) were no faster, nor were equal
// shares of all tiles over the workgroups, where beginning a row block costs more than the evenness gives.
#include "eia_flash.h"

namespace {

constexpr int WF_KEYS = 64;                 // keys per tile
constexpr int WF_ROWS = 128;                // (query, head) rows per workgroup

struct FlashArgs {
  const bf16_t* q; long ldq;                // [rows, H * P * D]
  const bf16_t* kc; const bf16_t* vc;       // [blocks, bs, G * P * D], [blocks, G * Dv, bs]
  const int* bt; int ldbt;
  const int* positions; const int* cu; const int* work;
  const float* mult; const float* bias; const float* sink; const float* lam;
  const bf16_t* gate; long ldg;
  bf16_t* out; long ldo;
  int H, G, D, Dv, bs, window, keep, gate_heads, hpw;
  float cap, eps, post;
  int per, nparts, items;                   // tiles of a part, parts the workspace has room for, work items
  float* part;
};

// What the lanes of a workgroup work on; qn <= 0: nothing.
struct WfRows {
  int s, h, qn;                             // sequence, this wave's head, queries of the workgroup
  bool live, mine;                          // the wave has a query; so has the lane
  long row;                                 // the lane's query (the last one where it has none)
  int p_last, w_first, w_last;              // last position of the workgroup; of the wave
  // tiles: those of the kept first tokens that lie before the window's (nkeep), then the window's
  // from key lo on
  int lo, nkeep, ntile;
};
template <bool SPLIT> EIA_DEV WfRows wf_rows(const FlashArgs& a, int w, int r32) {
  WfRows r;
  const int item = SPLIT ? min((int)blockIdx.y, a.items - 1) : blockIdx.y;         // (with parts the grid is padded)
  r.s = a.work[2 * item];
  const int q0 = a.work[2 * item + 1], qbeg = a.cu[r.s], qlen = a.cu[r.s + 1] - qbeg;
  r.qn = !SPLIT || item == (int)blockIdx.y ? min(WF_ROWS / a.hpw, qlen - q0) : 0;
  r.h = blockIdx.x * a.hpw + w % a.hpw;
  if (r.qn <= 0) return r;
  const int wq0 = q0 + 32 * (w / a.hpw);
  r.live = wq0 < qlen;
  r.mine = wq0 + r32 < qlen;
  r.row = qbeg + min(wq0 + r32, qlen - 1);
  const int p_first = a.positions[qbeg + q0];
  r.p_last = a.positions[qbeg + q0 + r.qn - 1];
  r.w_first = a.positions[qbeg + min(wq0, qlen - 1)];
  r.w_last = a.positions[qbeg + min(wq0 + 31, qlen - 1)];
  const int lo_min = a.window > 0 ? max(0, p_first - a.window + 1) : 0;
  r.lo = lo_min & ~(WF_KEYS - 1);
  r.nkeep = min((min(a.keep, lo_min) + WF_KEYS - 1) / WF_KEYS, r.lo / WF_KEYS);
  r.ntile = r.nkeep + (r.p_last - r.lo) / WF_KEYS + 1;
  return r;
}

// The place of wave w of P maps for part z of the workgroup's rows: 4 NDV + 1 units of 64 lanes x 4 floats.
template <int P, int NDV>
EIA_DEV float* wf_part(const FlashArgs& a, int z, int w) {
  const long wg = (long)blockIdx.y * gridDim.x + blockIdx.x;
  return a.part + ((wg * a.nparts + z) * 4 * P + w) * (4 * NDV + 1) * 256;
}

// Column tile dt of the part at x joins the lane's sums.
template <bool SIG, int NDV>
EIA_DEV void wf_join(const float* x, int dt, float& m, float& lsum, f32x16_t (&o)[1]) {
  const f32x4 ml = *reinterpret_cast<const f32x4*>(x + 4 * NDV * 256);
  float w0 = 1.f, w1 = 1.f;
  if constexpr (!SIG) {
    const float mn = fmaxf(m, ml[0]);
    w0 = __builtin_amdgcn_exp2f(m - mn);
    w1 = __builtin_amdgcn_exp2f(ml[0] - mn);
    m = mn;
  }
  lsum = SIG ? 1.f : lsum * w0 + ml[1] * w1;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(x + (4 * dt + i) * 256);
#pragma unroll
    for (int e = 0; e < 4; ++e) o[0][4 * i + e] = o[0][4 * i + e] * w0 + v[e] * w1;
  }
}

// From a lane's sums to its outputs: columns c0 + 32 dt + 8 j + 4 hh + i of its query.
template <int P, int NDV>
EIA_DEV void wf_finish(const FlashArgs& a, const WfRows& rw, int hh, const f32x16_t (&o)[NDV], float lsum,
                       int c0 = 0) {
  const int Dv = a.Dv, h = rw.h;
  const long row = rw.row;
  float inv = a.post / lsum;
  if constexpr (P == 2) {                   // root mean square of the head (columns past Dv are zero)
    float ss = 0.f;
#pragma unroll
    for (int dt = 0; dt < NDV; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) ss += o[dt][i] * o[dt][i];
    inv = a.post / sqrtf(flash_pair_sum(ss) / (float)Dv + a.eps);
  } else if (a.gate && a.gate_heads) {
    inv *= 1.0f / (1.0f + __expf(-bf2f(a.gate[row * a.ldg + h])));
  }
  if (!rw.mine) return;
  bf16_t* op = a.out + row * a.ldo + (long)h * Dv + 4 * hh;
#pragma unroll
  for (int dt = 0; dt < NDV; ++dt)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = c0 + 32 * dt + 8 * j;
      if (c >= Dv) continue;                // (Dv % 16 == 0)
      bf16x4 o4;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float v = o[dt][4 * j + i] * inv;
        if (P == 1 && a.gate && !a.gate_heads)
          v *= 1.0f / (1.0f + __expf(-bf2f(a.gate[row * a.ldg + (long)h * Dv + 4 * hh + c + i])));
        o4[i] = f2bf(v);
      }
      *reinterpret_cast<bf16x4*>(op + c) = o4;
    }
}

// P: score maps per head (2: a differential pair).  ND: 16-channel steps of a map (D <= 16 ND), NDV:
// 32-column tiles of the values (Dv <= 32 NDV).  SIG: sigmoid weights, not normalised.
// With P == 2 there are eight waves, four for each map of the same rows; the first four finish them.
// SPLIT: a row block of more than a.per tiles is cut over grid.z, the parts meet in
// window_flash_merge_kernel.
template <int P, int ND, int NDV, bool SIG, bool SPLIT>
__global__ void __launch_bounds__(256 * P, 2)
window_flash_kernel(FlashArgs a) {
  constexpr int NT = 256 * P;
  constexpr int KW = P * 16 * ND, KS = KW + 8, VS = WF_KEYS + 8;
  constexpr int KBUF = WF_KEYS * KS, BUF = KBUF + 32 * NDV * VS;
  constexpr int NKU = WF_KEYS * KW / 8 / NT, NVU = 32 * NDV * WF_KEYS / 8 / NT;   // 16-byte units per thread
  __shared__ __align__(16) bf16_t wf_lds[2 * BUF];
  static_assert(P == 1 || sizeof(wf_lds) >= 4 * 4 * 64 * 16 * NDV, "room to hand rows over");
  const int tid = threadIdx.x, lane = tid & 63, grp = tid >> 8, w = (tid >> 6) & 3;
  const int r32 = lane & 31, hh = lane >> 5, map = P == 2 ? grp : 0;
  const WfRows rw = wf_rows<SPLIT>(a, w, r32);
  if (rw.qn <= 0) return;                               // (whole workgroup)
  const int D = a.D, Dv = a.Dv, bs = a.bs, kvh = blockIdx.x * a.hpw / (a.H / a.G), h = rw.h;
  const long row = rw.row;
  const int qpos = a.positions[row], p_last = rw.p_last, w_first = rw.w_first, w_last = rw.w_last;
  const bool live = rw.live;
  const int lo = rw.lo, nkeep = rw.nkeep;
  const int parts = SPLIT ? min(a.nparts, (rw.ntile + a.per - 1) / a.per) : 1;
  if (SPLIT && (int)blockIdx.z >= parts) return;        // (whole workgroup)
  // (equal parts)
  const int it0 = SPLIT ? rw.ntile * blockIdx.z / parts : 0;
  const int it1 = SPLIT ? rw.ntile * (blockIdx.z + 1) / parts : rw.ntile;
  auto tile_key = [&](int it) { return it < nkeep ? it * WF_KEYS : lo + (it - nkeep) * WF_KEYS; };

  bf16x8 qf[ND];
  const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int t = 0; t < ND; ++t) {
    const int d = 16 * t + 8 * hh;
    const bf16x8 v = *reinterpret_cast<const bf16x8*>(a.q + row * a.ldq + (long)(h * P + map) * D + (d < D ? d : 0));
    qf[t] = d < D ? v : zero8;
  }
  // base-2 scores are raw * ml (a negative multiplier changes the sign of the query instead, so that
  // the largest raw score is the largest score); soft-capped, cap + 2 cap x with x = -1 / (exp(2 raw / cap) + 1)
  float ml = a.mult[h * P + map] * FLASH_LOG2E;
  if (ml < 0.f) {
    ml = -ml;
#pragma unroll
    for (int t = 0; t < ND; ++t) qf[t] = -qf[t];
  }
  const float capl = a.cap * FLASH_LOG2E, icap = a.cap > 0.f ? 2.f * ml / a.cap : 0.f;
  const float sc = a.cap > 0.f ? 2.f * capl : fmaxf(ml, 1e-30f), shift = a.cap > 0.f ? capl : 0.f;

  const int* bt = a.bt + (long)rw.s * a.ldbt;
  const long vpage = (long)a.G * Dv * bs;
  const int krow = a.G * P * D;
  const bool whole = D == 16 * ND && Dv == 32 * NDV;    // no channel and no column to be zeroed
  unsigned koff[NKU], voff[NVU];
#pragma unroll
  for (int i = 0; i < NKU; ++i) {
    const int u = tid + NT * i, m = u % (KW / 8) / (2 * ND), d = 8 * (u % (KW / 8) % (2 * ND));
    koff[i] = u / (KW / 8) * krow + m * D + (d < D ? d : 0);
  }
#pragma unroll
  for (int i = 0; i < NVU; ++i) {
    const int u = tid + NT * i, c = u >> 3;
    voff[i] = (c < Dv ? c : 0) * bs + 8 * (u & 7);
  }
  // the page of a tile is looked up a tile ahead of its fetch: the fetch would wait for it
  int off = 0, at = 0, page = 0;                        // the next fetch: token in its page, page's place, page
  auto look = [&](int it) {
    if (it == it0 || it == nkeep) {
      at = tile_key(it) / bs;
      off = tile_key(it) - at * bs;
    } else {
      off += WF_KEYS;
      if (off == bs) off = 0, ++at;
    }
    page = bt[at];
  };
  bf16x8 kst[NKU], vst[NVU];
  // (nothing may look at the values before stash: the loads are in flight during a whole tile)
  auto fetch = [&] {
    const long pg = __builtin_amdgcn_readfirstlane(page);
    const bf16_t* kp = a.kc + (pg * bs + off) * krow + (long)kvh * P * D;
    const bf16_t* vp = a.vc + pg * vpage + (long)kvh * Dv * bs + off;
#pragma unroll
    for (int i = 0; i < NKU; ++i) kst[i] = *reinterpret_cast<const bf16x8*>(kp + koff[i]);
#pragma unroll
    for (int i = 0; i < NVU; ++i) vst[i] = *reinterpret_cast<const bf16x8*>(vp + voff[i]);
  };
  auto stash = [&](int buf, int kb) {
    bf16_t* kl = wf_lds + buf * BUF;
    if (!whole) {
#pragma unroll
      for (int i = 0; i < NKU; ++i)
        if (8 * ((tid + NT * i) % (KW / 8) % (2 * ND)) >= D) kst[i] = zero8;
#pragma unroll
      for (int i = 0; i < NVU; ++i)
        if ((tid + NT * i) >> 3 >= Dv) vst[i] = zero8;
    }
#pragma unroll
    for (int i = 0; i < NKU; ++i) {
      const int u = tid + NT * i;
      *reinterpret_cast<bf16x8*>(kl + u / (KW / 8) * KS + 8 * (u % (KW / 8))) = kst[i];
    }
    if (kb + WF_KEYS > p_last + 1) {        // (slots behind the last key may hold anything: 0 x inf)
#pragma unroll
      for (int i = 0; i < NVU; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (kb + 8 * ((tid + NT * i) & 7) + e > p_last) vst[i][e] = (bf16_t)0.f;
    }
#pragma unroll
    for (int i = 0; i < NVU; ++i) {
      const int u = tid + NT * i;
      *reinterpret_cast<bf16x8*>(kl + KBUF + (u >> 3) * VS + 8 * (u & 7)) = vst[i];
    }
  };

  f32x16_t oacc[NDV];
#pragma unroll
  for (int dt = 0; dt < NDV; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[dt][i] = 0.f;
  const bool snk = !SIG && a.sink && it0 == 0;
  // (never below -1e30: a sink that weighs nothing must not make the maximum -inf, which a tile of
  // which the lane sees no key would keep, and -inf - -inf is no number)
  const float sinkl = snk ? a.sink[h * P + map] * FLASH_LOG2E : 0.f;
  float m_run = snk ? fmaxf(sinkl, -1e30f) : -1e30f;
  float l_run = snk && hh == 0 ? __builtin_amdgcn_exp2f(sinkl - m_run) : 0.f;
  const float bl = (SIG && a.bias ? a.bias[h] * FLASH_LOG2E : 0.f) + shift;
  const int krow0 = (r32 & ~12) | ((r32 & 4) << 1) | ((r32 & 8) >> 1);

  auto compute = [&](int buf, int kb) {
    const bf16_t* kf0 = wf_lds + buf * BUF + krow0 * KS + map * 16 * ND + 8 * hh;
    const bf16_t* vf0 = wf_lds + buf * BUF + KBUF + r32 * VS + 8 * hh;
    // reads of LDS go four fragments ahead of the products, kept there by the barriers to the scheduler:
    // left alone, each is moved to its product, which then waits for it
    constexpr int NF = 2 * ND;
    f32x16_t sacc[2];
    bf16x8 kf[2][4];
    auto keys = [&](int b) {
#pragma unroll
      for (int x = 0; x < 4; ++x)
        kf[b & 1][x] = *reinterpret_cast<const bf16x8*>(kf0 + 32 * KS * (x & 1) + 16 * (2 * b + (x >> 1)));
    };
    // matrix products go first, the second ones before all: else the two waves of a SIMD wait for the same unit in
    // turn.  (Heads of 64, whose exponentials take longer than their products, lose 5 % by it.)
    constexpr bool PRIO = NDV > 2;
    if (PRIO) __builtin_amdgcn_s_setprio(1);
    keys(0);
#pragma unroll
    for (int b = 0; b < NF / 4; ++b) {
      if (b + 1 < NF / 4) keys(b + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int sh = x & 1, t = 2 * b + (x >> 1);
        sacc[sh] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[b & 1][x], qf[t], t == 0 ? f32x16_t{} : sacc[sh], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    mfma_settle(sacc[0], sacc[1]);
    if (PRIO) __builtin_amdgcn_s_setprio(0);
    // element i of half sh is key kb + 32 sh + 16 (i >> 3) + 8 hh + (i & 7)
    if (a.cap > 0.f) {
#pragma unroll
      for (int sh = 0; sh < 2; ++sh)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          sacc[sh][i] = __builtin_amdgcn_rcpf(-1.f - __builtin_amdgcn_exp2f(sacc[sh][i] * icap));
    }
    // every query of the wave sees every key of the tile?
    if (kb + WF_KEYS - 1 > w_first ||
        (a.window > 0 && w_last - kb >= a.window && kb + WF_KEYS > a.keep)) {
      const int d0 = qpos - kb - 8 * hh;
      const int win = a.window > 0 ? a.window : 0x7fffffff, kp = a.keep - kb - 8 * hh;
#pragma unroll
      for (int sh = 0; sh < 2; ++sh)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int j = 32 * sh + 16 * (i >> 3) + (i & 7);
          sacc[sh][i] = d0 >= j && (d0 - j < win || j < kp) ? sacc[sh][i] : -INFINITY;
        }
    }
    float muse = 0.f;
    if constexpr (!SIG) {
      float mx4[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        mx4[c] = sacc[c >> 1][8 * (c & 1)];
#pragma unroll
        for (int j = 1; j < 8; ++j) mx4[c] = fmaxf(mx4[c], sacc[c >> 1][8 * (c & 1) + j]);
      }
      const float mt = flash_pair_max(fmaxf(fmaxf(mx4[0], mx4[1]), fmaxf(mx4[2], mx4[3]))) * sc + shift;
      const bool grow = mt > m_run + FLASH_DEFER;
      if (__any(grow)) {
        const float m_new = grow ? mt : m_run;
        const float alpha = grow ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.f;
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int dt = 0; dt < NDV; ++dt) oacc[dt] *= alpha;
      }
      muse = m_run - shift;
    }
    if (PRIO) __builtin_amdgcn_s_setprio(2);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      bf16x8 ph, pl;
      float ps = 0.f;
#pragma unroll
      for (int j = 0; j < 8; j += 2) {
        float p[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const float x = sacc[ks >> 1][8 * (ks & 1) + j + e];
          if constexpr (SIG) p[e] = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(fmaf(-x, sc, -bl)));
          else p[e] = __builtin_amdgcn_exp2f(fmaf(x, sc, -muse));
        }
        ps += p[0] + p[1];
        flash_split(p[0], p[1], j, ph, pl);
      }
      l_run += ps;
      bf16x8 vf[NDV];
#pragma unroll
      for (int dt = 0; dt < NDV; ++dt) {
        vf[dt] = *reinterpret_cast<const bf16x8*>(vf0 + 32 * VS * dt + 16 * ks);
        oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[dt], ph, oacc[dt], 0, 0, 0);
      }
#pragma unroll
      for (int dt = 0; dt < NDV; ++dt)
        oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[dt], pl, oacc[dt], 0, 0, 0);
    }
    if (PRIO) __builtin_amdgcn_s_setprio(0);
  };

  look(it0);
  fetch();
  if (it0 + 1 < it1) look(it0 + 1);
  stash(0, tile_key(it0));
  __syncthreads();
  for (int it = it0; it < it1; ++it) {
    const int kb = tile_key(it);
    const bool more = it + 1 < it1;
    if (more) {
      fetch();
      if (it + 2 < it1) look(it + 2);
    }
    // does any query of the wave see a key of the tile?
    if (live && kb <= w_last && (a.window <= 0 || w_first - (kb + WF_KEYS - 1) < a.window || kb < a.keep))
      compute((it - it0) & 1, kb);
    if (more) stash((it - it0 + 1) & 1, tile_key(it + 1));
    __syncthreads();
  }
  float lsum = SIG ? 1.f : flash_pair_sum(l_run);
  if (SPLIT && parts > 1) {
    float* x = wf_part<P, NDV>(a, blockIdx.z, 4 * map + w) + 4 * lane;
#pragma unroll
    for (int dt = 0; dt < NDV; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<f32x4*>(x + (4 * dt + i) * 256) =
            f32x4{oacc[dt][4 * i], oacc[dt][4 * i + 1], oacc[dt][4 * i + 2], oacc[dt][4 * i + 3]};
    *reinterpret_cast<f32x4*>(x + 4 * NDV * 256) = f32x4{m_run, lsum, 0.f, 0.f};
    return;
  }
  if constexpr (P == 2) {                               // a1 - lam a2
    float* x = reinterpret_cast<float*>(wf_lds) + (w * 16 * NDV) * 64 + lane;
    if (grp == 1) {
      const float w1 = -a.lam[0] / lsum;
#pragma unroll
      for (int dt = 0; dt < NDV; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) x[(16 * dt + i) * 64] = oacc[dt][i] * w1;
    }
    __syncthreads();
    if (grp == 1) return;
    const float w0 = 1.f / lsum;
    lsum = 1.f;
#pragma unroll
    for (int dt = 0; dt < NDV; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) oacc[dt][i] = oacc[dt][i] * w0 + x[(16 * dt + i) * 64];
  }
  wf_finish<P, NDV>(a, rw, hh, oacc, lsum);
}

// The parts of a row block put together: the rows, lanes and registers of the kernel above, a workgroup
// for each 32 columns.  Bound by the parts' traffic and by the dependent reads in front of it: 256 row blocks of
// up to 5 parts x 69 KB, 44 MB in all, take 12.4 us (of up to 3 parts 8.4); with one workgroup for all columns of a row block (one
// wave per SIMD, part after part) 16.4 us.
template <int NDV, bool SIG>
__global__ void __launch_bounds__(256)
window_flash_merge_kernel(FlashArgs a) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, dt = blockIdx.z;
  const WfRows rw = wf_rows<true>(a, w, lane & 31);
  const int parts = min(a.nparts, (rw.ntile + a.per - 1) / a.per);
  if (rw.qn <= 0 || parts <= 1 || !rw.live) return;
  float m = -INFINITY, lsum = 0.f;
  f32x16_t oacc[1];
#pragma unroll
  for (int i = 0; i < 16; ++i) oacc[0][i] = 0.f;
#pragma unroll 2
  for (int z = 0; z < parts; ++z) wf_join<SIG, NDV>(wf_part<1, NDV>(a, z, w) + 4 * lane, dt, m, lsum, oacc);
  wf_finish<1, 1>(a, rw, lane >> 5, oacc, lsum, 32 * dt);
}

// The parts of a differential pair, 32 rows a workgroup: a wave for each map and 32 columns, as above; the second
// map's waves hand theirs over, and the root mean square of the difference meets in LDS.  (One wave a map with all
// columns: 2 parts of 46 row blocks of 128 columns 44 us with the products, this way 36; uncut 49.)
template <int NDV>
__global__ void __launch_bounds__(128 * NDV)
window_flash_merge_pair_kernel(FlashArgs a) {
  __shared__ float other[NDV][16][64], sq[NDV][64];
  const int lane = threadIdx.x & 63, dt = (threadIdx.x >> 6) % NDV, map = threadIdx.x / (64 * NDV), w = blockIdx.z;
  const WfRows rw = wf_rows<true>(a, w, lane & 31);
  const int parts = min(a.nparts, (rw.ntile + a.per - 1) / a.per);
  if (rw.qn <= 0 || parts <= 1 || !rw.live) return;     // (whole workgroup)
  float m = -INFINITY, lsum = 0.f, ss = 0.f;
  f32x16_t o[1];
#pragma unroll
  for (int i = 0; i < 16; ++i) o[0][i] = 0.f;
#pragma unroll 2
  for (int z = 0; z < parts; ++z)
    wf_join<false, NDV>(wf_part<2, NDV>(a, z, 4 * map + w) + 4 * lane, dt, m, lsum, o);
  const float f = map ? -a.lam[0] / lsum : 1.f / lsum;
  if (map) {
#pragma unroll
    for (int i = 0; i < 16; ++i) other[dt][i][lane] = o[0][i] * f;
  }
  __syncthreads();
  if (!map) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      o[0][i] = o[0][i] * f + other[dt][i][lane];
      ss += o[0][i] * o[0][i];
    }
    sq[dt][lane] = flash_pair_sum(ss);
  }
  __syncthreads();
  if (map) return;
  ss = 0.f;
#pragma unroll
  for (int t = 0; t < NDV; ++t) ss += sq[t][lane];
  wf_finish<1, 1>(a, rw, lane >> 5, o, sqrtf(ss / (float)a.Dv + a.eps), 32 * dt);
}

template <int P, int ND, int NDV, bool SIG, bool SPLIT>
static void wf_launch(const FlashArgs& a, int n_items, int parts, hipStream_t st) {
  // With parts the grid is padded to whole rounds of the XCDs, so that the parts of a row block and their merge share
  // one (us without / with: 725 tokens behind 1900, window 1024, 8 heads of 128 26.9 / 24.0, of pairs 31.3 / 28.4; 2500
  // tokens 43.1 / 41.0).
  const int x = a.H / a.hpw, pad = SPLIT ? (x % 8 == 0 ? 1 : x % 4 == 0 ? 2 : x % 2 == 0 ? 4 : 8) : 1;
  n_items = (n_items + pad - 1) / pad * pad;
  hipLaunchKernelGGL((window_flash_kernel<P, ND, NDV, SIG, SPLIT>), dim3(x, n_items, parts), dim3(256 * P), 0, st, a);
  if constexpr (SPLIT && P == 2)
    hipLaunchKernelGGL((window_flash_merge_pair_kernel<NDV>), dim3(x, n_items, 4), dim3(128 * NDV), 0,
                       st, a);
  else if constexpr (SPLIT)
    hipLaunchKernelGGL((window_flash_merge_kernel<NDV, SIG>), dim3(x, n_items, NDV), dim3(256), 0, st, a);
}

template <int P, int ND, int NDV, bool SIG>
static void wf_go(const FlashArgs& a, int n_items, int parts, hipStream_t st) {
  if (parts > 1)
    wf_launch<P, ND, NDV, SIG, true>(a, n_items, parts, st);
  else
    wf_launch<P, ND, NDV, SIG, false>(a, n_items, 1, st);
}

}  // namespace

// 32-column tiles of a wave's part in the workspace: those of the kernel that takes the shape, whatever Dv needs.
EIA_API int eia_window_flash_columns(int P, int D, int Dv) {
  return P == 2 ? 4 : D <= 64 && Dv <= 64 ? 2 : D <= 64 ? 4 : D <= 96 && Dv <= 96 ? 3 : 4;
}

// Queries per work item of eia_window_flash, 0 where it does not take the shape.
EIA_API int eia_window_flash_queries(int H, int G, int P, int D, int Dv, int bs) {
  if (G < 1 || H < 1 || H % G || (P != 1 && P != 2) || D < 8 || D % 8 || Dv < 16 || Dv % 16 ||
      D > (P == 2 ? 64 : 128) || Dv > 128 || bs < 64 || bs % 64)
    return 0;
  const int rep = H / G;
  return WF_ROWS / (rep % 4 == 0 ? 4 : rep % 2 == 0 ? 2 : 1);
}

// Prompt portions of window attention without head mixing or slopes; the arguments are those of
// eia_window_attn_mfma, work holds blocks of eia_window_flash_queries queries.  nparts > 1:
// row blocks of more than per 64-key tiles are cut into parts of at most that many (nparts * per
// tiles cover the longest), which meet in part [n_items * H / hpw, nparts, 4 P, 4 eia_window_flash_columns + 1,
// 256] fp32, hpw = 128 / queries.
EIA_API int eia_window_flash(const void* q, long ldq, const void* kc, const void* vc, const int* bt,
                             int ldbt, const int* positions, const int* cu, const int* work,
                             int n_items, const float* mult, const void* gate, long ldg, void* out,
                             long ldo, int H, int G, int P, int D, int Dv, int bs, int window,
                             int keep, const float* lam, float eps, float post, int wmode,
                             const float* bias, const float* sink, float cap, int gate_heads,
                             int nparts, int per, float* part, hipStream_t st) {
  if (n_items < 0 || keep < 0 || cap < 0.f || !q || !kc || !vc || !bt || !positions || !cu || !work ||
      !mult || !out || (P == 2) != (lam != nullptr) || (P == 2 && gate) ||
      (wmode != 0 && wmode != 1) || (wmode == 1 && (P != 1 || sink)) || ldq % 8 || ldo % 4 ||
      nparts < 1 || (nparts > 1 && (per < 1 || !part)))
    return EIA_BAD_SHAPE;
  const int qb = eia_window_flash_queries(H, G, P, D, Dv, bs);
  if (!qb) return EIA_UNSUPPORTED;
  if (n_items == 0) return EIA_OK;
  FlashArgs a{(const bf16_t*)q, ldq, (const bf16_t*)kc, (const bf16_t*)vc, bt, ldbt, positions, cu,
              work, mult, bias, sink, lam, (const bf16_t*)gate, ldg, (bf16_t*)out, ldo, H, G, D, Dv,
              bs, window, keep, gate_heads, WF_ROWS / qb, cap, eps, post, per, nparts, n_items, part};
  const int cols = eia_window_flash_columns(P, D, Dv);
#define WF_SIZES(SG)                                                    \
  do {                                                                  \
    if (cols == 2) wf_go<1, 4, 2, SG>(a, n_items, nparts, st);          \
    else if (cols == 3) wf_go<1, 6, 3, SG>(a, n_items, nparts, st);     \
    else if (D <= 64) wf_go<1, 4, 4, SG>(a, n_items, nparts, st);       \
    else wf_go<1, 8, 4, SG>(a, n_items, nparts, st);                    \
  } while (0)
  if (P == 2) wf_go<2, 4, 4, false>(a, n_items, nparts, st);
  else if (wmode == 1) WF_SIZES(true);
  else WF_SIZES(false);
#undef WF_SIZES
  EIA_LAUNCH_CHECK();
}
