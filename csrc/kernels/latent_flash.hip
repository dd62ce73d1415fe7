// Latent attention (absorbed form, bf16) over prompt portions: every head reads the same cache rows
// [latent c (R) | rotated key part (rd)], scores over R + rd entries, values = the first R.
//
// A workgroup of four waves owns 128 (query, head) rows -- 128 / HB queries of HB = min(H, 16) heads --
// and a wave 32 of them, on v_mfma_f32_32x32x16_bf16.  KT cache rows are staged in LDS once, as they
// are: the first product reads them row by row (S^T = C Q^T, a lane owns one query row; rows of C are
// fed with bits 2 and 3 of their number swapped, so that a lane's accumulators are eight consecutive
// keys), the second as columns through the transposing LDS read (O^T += C^T P^T), so there is no second
// copy.  (Before, a 16-row wave read every operand for itself and 32-key tiles went through LDS twice,
// the second time as 2-byte transposed stores.)  Softmax as in window_flash.hip: fp32 weights as a
// bf16 high part plus a remainder, normaliser over the fp32 values, deferred rescale.  Rows of an LDS
// tile are an odd number of 16-byte units apart, so that sixteen rows lie on different banks.
//
// MI355X, one 4096-token causal prompt: 8 heads, R 128 + 32: 71 + 9 us in parts; 8 heads, R 256 + 64: 202 us; 16
// heads, R 512 + 64: 915, with a window of 1024 488.  With the page of a tile looked up by its fetch, every read of LDS in
// front of its product, no priorities and parts in more than one round 82 + 12, 299, 1100 and 573 us.
// A wave's registers hold the sums of 32 rows over 256 columns beside its queries only alone on its
// SIMD; at R 512 two waves share the rows and form the same scores (one wave alone spilled 1.3 KB a
// lane and took 1847 us at the window of 1024).
#include "eia_flash.h"

namespace {

// (query, head) rows per workgroup.  CS: waves that share 32 rows, each with a part of the latent
// columns: the sums of 32 rows over 512 columns do not fit beside their queries in one wave's
// registers, so two waves form the same scores.
constexpr int lf_nrows(int CS) { return 128 / CS; }

struct LatentFlashArgs {
  const bf16_t* qa; long qa_st, qa_sh;      // [rows, H, R]
  const bf16_t* qr; long qr_st, qr_sh;      // [rows, H, rd], not yet rotated
  const float* inv_freq; int rot_dims, rot_half; float rot_amp;
  const bf16_t* cache; long cache_row;
  const int* bt; int ldbt;
  const int* positions; const int* cu; const int* work;
  const bf16_t* gate; long gate_st;
  bf16_t* out; long out_st, out_sh;
  const float* sink;
  float scale;
  int H, R, rd, bs, HB, window;
  int per, nparts, items;                   // tiles of a part, parts the workspace has room for, work items
  float* part;
};

// What the lanes of a workgroup work on; ntok <= 0: nothing.
struct LfRows {
  int s, ntok, row0, h;                     // sequence, queries, first row; the lane's head
  bool live, mine;                          // the wave has a row; so has the lane
  long row;                                 // the lane's query (the first one where it has none)
  int p_last, w_first, w_last;              // last position of the workgroup; of the wave's rows
  int lo, ntile;                            // first key, tiles
};
template <int KT, int CS, bool SPLIT> EIA_DEV LfRows lf_rows(const LatentFlashArgs& a, int w, int r32) {
  LfRows r;
  const int item = SPLIT ? min((int)blockIdx.x, a.items - 1) : blockIdx.x;         // (with parts the grid is padded)
  r.s = a.work[2 * item];
  const int q0 = a.work[2 * item + 1], qbeg = a.cu[r.s], qlen = a.cu[r.s + 1] - qbeg;
  r.ntok = !SPLIT || item == (int)blockIdx.x ? min(lf_nrows(CS) / a.HB, qlen - q0) : 0;
  if (r.ntok <= 0) return r;
  r.row0 = qbeg + q0;
  const int b = w / CS, m = 32 * b + r32, t = m / a.HB, t0 = 32 * b / a.HB, t1 = (32 * b + 31) / a.HB;
  r.h = blockIdx.y * a.HB + m - t * a.HB;
  r.live = t0 < r.ntok;
  r.mine = t < r.ntok && r.h < a.H;
  r.row = r.row0 + (r.mine ? t : 0);
  const int p_first = a.positions[r.row0];
  r.p_last = a.positions[r.row0 + r.ntok - 1];
  r.w_first = a.positions[r.row0 + min(t0, r.ntok - 1)];
  r.w_last = a.positions[r.row0 + min(t1, r.ntok - 1)];
  r.lo = a.window > 0 ? max(0, p_first - a.window + 1) & ~(KT - 1) : 0;
  r.ntile = (r.p_last - r.lo) / KT + 1;
  return r;
}

// Wave w's place for part z of the workgroup's rows: 4 NDV + 1 units of 64 lanes x 4 floats.
EIA_DEV float* lf_part(const LatentFlashArgs& a, int z, int w, int ndv) {
  const long wg = (long)blockIdx.x * gridDim.y + blockIdx.y;
  return a.part + ((wg * a.nparts + z) * 4 + w) * (4 * ndv + 1) * 256;
}

// From a lane's sums to its outputs: columns c0 + 32 dt + 8 j + 4 hh + i of its row.
template <int NDV>
EIA_DEV void lf_finish(const LatentFlashArgs& a, const LfRows& rw, int hh, int c0,
                       const f32x16_t (&o)[NDV], float m, float lsum) {
  if (!rw.mine) return;
  if (a.sink) lsum += __builtin_amdgcn_exp2f(a.sink[rw.h] * FLASH_LOG2E - m);
  float f = 1.0f / lsum;
  if (a.gate) f *= 1.0f / (1.0f + expf(-bf2f(a.gate[rw.row * a.gate_st + rw.h])));
  bf16_t* op = a.out + rw.row * a.out_st + (long)rw.h * a.out_sh + 4 * hh;
#pragma unroll
  for (int dt = 0; dt < NDV; ++dt)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = c0 + 32 * dt + 8 * j;
      if (c >= a.R) continue;               // (R % 8 == 0)
      bf16x4 o4;
#pragma unroll
      for (int i = 0; i < 4; ++i) o4[i] = f2bf(o[dt][4 * j + i] * f);
      *reinterpret_cast<bf16x4*>(op + c) = o4;
    }
}

// NK: 16-entry steps of a cache row (R + rd <= 16 NK), NDV: 32-column tiles of a wave's part of the
// latent (R <= 32 NDV CS), KT: keys per tile, WPS: waves per SIMD that the registers are cut for.
template <int NK, int NDV, int KT, int WPS, int CS, bool SPLIT>
__global__ void __launch_bounds__(256, WPS)
latent_flash_kernel(LatentFlashArgs a) {
  constexpr int KS = 16 * NK + 8, BUF = KT * KS;        // (2 NK + 1 units of 16 bytes per row)
  constexpr int NU = KT * 2 * NK / 256;                 // 16-byte units of a tile per thread
  constexpr int SH = KT / 32, VB = 4;
  static_assert(NDV % VB == 0, "whole groups");
  static_assert(KT * 2 * NK % 256 == 0, "whole units");
  extern __shared__ __align__(16) bf16_t lf_lds[];      // 2 * BUF + 64
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r32 = lane & 31, hh = lane >> 5;
  const LfRows rw = lf_rows<KT, CS, SPLIT>(a, w, r32);
  if (rw.ntok <= 0) return;                             // (whole workgroup)
  const int parts = SPLIT ? min(a.nparts, (rw.ntile + a.per - 1) / a.per) : 1;
  if (SPLIT && (int)blockIdx.z >= parts) return;        // (whole workgroup)
  const int it0 = SPLIT ? rw.ntile * blockIdx.z / parts : 0;      // (equal parts)
  const int it1 = SPLIT ? rw.ntile * (blockIdx.z + 1) / parts : rw.ntile;
  const int R = a.R, Dk = R + a.rd, bs = a.bs;
  const int qpos = rw.mine ? a.positions[rw.row] : -1;

  // the rotary query parts of the workgroup's rows, rotated once into LDS: a thread takes whole pairs
  bf16_t* qrs = lf_lds;                                 // [rows][rd]
  {
    const int hp = a.rot_dims >> 1, npass = a.rd - a.rot_dims;
    for (int e = tid; e < lf_nrows(CS) * hp; e += 256) {
      const int m = e / hp, i = e - m * hp, t = m / a.HB, h = blockIdx.y * a.HB + m - t * a.HB;
      if (t < rw.ntok && h < a.H) {
        const bf16_t* src = a.qr + (long)(rw.row0 + t) * a.qr_st + (long)h * a.qr_sh;
        const int ia = a.rot_half ? i : 2 * i, ib = a.rot_half ? i + hp : 2 * i + 1;
        const float u = bf2f(src[ia]), v = bf2f(src[ib]);
        float sn, cs;
        sincosf((float)a.positions[rw.row0 + t] * a.inv_freq[i], &sn, &cs);
        sn *= a.rot_amp;
        cs *= a.rot_amp;
        qrs[m * a.rd + ia] = f2bf(u * cs - v * sn);
        qrs[m * a.rd + ib] = f2bf(v * cs + u * sn);
      }
    }
    for (int e = tid; e < lf_nrows(CS) * npass; e += 256) {  // entries past rot_dims pass unchanged
      const int m = e / npass, d = a.rot_dims + e - m * npass, t = m / a.HB, h = blockIdx.y * a.HB + m - t * a.HB;
      if (t < rw.ntok && h < a.H)
        qrs[m * a.rd + d] = a.qr[(long)(rw.row0 + t) * a.qr_st + (long)h * a.qr_sh + d];
    }
    __syncthreads();
  }
  const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  bf16x8 qf[NK];
  {
    // R % 8 == 0: a lane's eight entries lie wholly in the absorbed or wholly in the rotary part
    const bf16_t* qa = a.qa + rw.row * a.qa_st + (long)(rw.mine ? rw.h : 0) * a.qa_sh;
    const bool vec = ((reinterpret_cast<uintptr_t>(a.qa) | (uintptr_t)(a.qa_st * 2) | (uintptr_t)(a.qa_sh * 2)) & 15) == 0;
#pragma unroll
    for (int t = 0; t < NK; ++t) {
      const int d = 16 * t + 8 * hh;
      bf16x8 v = zero8;
      if (rw.mine && d < Dk) {
        if (d >= R) {
          v = *reinterpret_cast<const bf16x8*>(qrs + (32 * (w / CS) + r32) * a.rd + (d - R));
        } else if (vec) {
          v = *reinterpret_cast<const bf16x8*>(qa + d);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = qa[d + e];
        }
      }
      qf[t] = v;
    }
  }
  __syncthreads();                                      // the rotary parts make room for tiles

  const int* bt = a.bt + (long)rw.s * a.ldbt;
  const bool paged = bs % KT == 0;                      // a tile lies in one page
  bf16x8 kst[NU];
  // (nothing may look at the values before stash: the loads are in flight during a whole tile)
  // the page of a tile is looked up a tile ahead of its fetch: the fetch would wait for it
  int off = 0, at = 0, page = 0;                        // the next fetch: token in its page, page's place, page
  auto look = [&](int it) {
    if (!paged) return;
    if (it == it0) {
      at = (rw.lo + it * KT) / bs;
      off = rw.lo + it * KT - at * bs;
    } else {
      off += KT;
      if (off == bs) off = 0, ++at;
    }
    page = bt[at];
  };
  auto fetch = [&](int kb) {
    const long base = paged ? (long)__builtin_amdgcn_readfirstlane(page) * bs + off : 0;
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = tid + 256 * i, j = u / (2 * NK), d = 8 * (u % (2 * NK));
      const int kp = min(kb + j, rw.p_last);
      const long slot = paged ? base + j : (long)bt[kp / bs] * bs + kp % bs;
      kst[i] = *reinterpret_cast<const bf16x8*>(a.cache + slot * a.cache_row + (d < Dk ? d : 0));
    }
  };
  auto stash = [&](int buf, int kb) {       // (slots behind the last key may hold anything: 0 x inf)
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = tid + 256 * i, j = u / (2 * NK), d = 8 * (u % (2 * NK));
      *reinterpret_cast<bf16x8*>(lf_lds + buf * BUF + j * KS + d) = d < Dk && kb + j <= rw.p_last ? kst[i] : zero8;
    }
  };

  f32x16_t oacc[NDV];
#pragma unroll
  for (int dt = 0; dt < NDV; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[dt][i] = 0.f;
  float m_run = -1e30f, l_run = 0.f;
  const float sc = fabsf(a.scale) * FLASH_LOG2E;
  if (a.scale < 0.f) {                      // (the largest raw score is then the largest score)
#pragma unroll
    for (int t = 0; t < NK; ++t) qf[t] = -qf[t];
  }
  const int krow0 = (r32 & ~12) | ((r32 & 4) << 1) | ((r32 & 8) >> 1);
  // transposing read: lane l of sixteen addresses row l / 4, entries 4 (l % 4), and receives column l
  const int l16 = lane & 15, vrow = 8 * hh + (l16 >> 2), c0 = 32 * NDV * (w % CS);
  const int vcol = c0 + 16 * ((lane >> 4) & 1) + 4 * (l16 & 3);

  auto compute = [&](int buf, int kb) {
    const bf16_t* kf0 = lf_lds + buf * BUF + krow0 * KS + 8 * hh;
    // reads of LDS go AH fragments ahead of the products, kept there by the barriers to the scheduler: left alone,
    // each is moved to its product, which then waits for it
    // (R 512, whose registers are short: 16 heads, 4096 tokens 915 us with one ahead, 980 with two, 1100 with four)
    constexpr int AH = NK >= 36 && NDV == 8 ? 1 : 4, NF = SH * NK;
    static_assert(NF % AH == 0, "whole groups");
    f32x16_t sacc[SH];
    bf16x8 kf[2][AH];
    auto keys = [&](int b) {
#pragma unroll
      for (int x = 0; x < AH; ++x) {
        const int f = AH * b + x;
        kf[b & 1][x] = *reinterpret_cast<const bf16x8*>(kf0 + 32 * KS * (f % SH) + 16 * (f / SH));
      }
    };
    // matrix products go first, the second ones before all: else the two waves of a SIMD wait for the same unit in turn.
    // (Not in whole row blocks of R 128, whose waves are rarely at the same place: two prompts of up to 3743 tokens,
    // 8 heads 130 us with priorities, 122 without, in halves 109 and 113.)
    constexpr bool PRIO = SPLIT || NK > 10;
    if (PRIO) __builtin_amdgcn_s_setprio(1);
    keys(0);
#pragma unroll
    for (int b = 0; b < NF / AH; ++b) {
      if (b + 1 < NF / AH) keys(b + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < AH; ++x) {
        const int f = AH * b + x, sh = f % SH, t = f / SH;
        sacc[sh] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[b & 1][x], qf[t], t == 0 ? f32x16_t{} : sacc[sh], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (PRIO) __builtin_amdgcn_s_setprio(0);
    // element i of half sh is key kb + 32 sh + 16 (i >> 3) + 8 hh + (i & 7); scores of the wave's
    // first products are read here, in line with them
#pragma unroll
    for (int sh = 0; sh < SH; ++sh)
#pragma unroll
      for (int i = 0; i < 16; ++i) sacc[sh][i] *= sc;
    if (kb + KT - 1 > rw.w_first || (a.window > 0 && rw.w_last - kb >= a.window)) {
      const int d0 = qpos - kb - 8 * hh, win = a.window > 0 ? a.window : 0x7fffffff;
#pragma unroll
      for (int sh = 0; sh < SH; ++sh)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int j = 32 * sh + 16 * (i >> 3) + (i & 7);
          sacc[sh][i] = d0 >= j && d0 - j < win ? sacc[sh][i] : -INFINITY;
        }
    }
    float mx[2 * SH];
#pragma unroll
    for (int c = 0; c < 2 * SH; ++c) {
      mx[c] = sacc[c >> 1][8 * (c & 1)];
#pragma unroll
      for (int j = 1; j < 8; ++j) mx[c] = fmaxf(mx[c], sacc[c >> 1][8 * (c & 1) + j]);
    }
#pragma unroll
    for (int c = 1; c < 2 * SH; ++c) mx[0] = fmaxf(mx[0], mx[c]);
    const float mt = flash_pair_max(mx[0]);
    const bool grow = mt > m_run + FLASH_DEFER;
    if (__any(grow)) {
      const float m_new = grow ? mt : m_run;
      const float alpha = grow ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.f;
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < NDV; ++dt) oacc[dt] *= alpha;
    }
    if (PRIO) __builtin_amdgcn_s_setprio(2);
#pragma unroll
    for (int ks = 0; ks < 2 * SH; ++ks) {
      bf16x8 ph, pl;
      float ps = 0.f;
#pragma unroll
      for (int j = 0; j < 8; j += 2) {
        const float p0 = __builtin_amdgcn_exp2f(sacc[ks >> 1][8 * (ks & 1) + j] - m_run);
        const float p1 = __builtin_amdgcn_exp2f(sacc[ks >> 1][8 * (ks & 1) + j + 1] - m_run);
        ps += p0 + p1;
        flash_split(p0, p1, j, ph, pl);
      }
      l_run += ps;
      const bf16_t* v0 = lf_lds + buf * BUF + (16 * ks + vrow) * KS + vcol;
      bf16x8 vf[VB];
#pragma unroll
      for (int d0 = 0; d0 < NDV; d0 += VB) {
#pragma unroll
        for (int x = 0; x < VB; ++x) {
          vf[x] = lds_columns(v0 + 32 * (d0 + x), v0 + 32 * (d0 + x) + 4 * KS);
          oacc[d0 + x] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[x], ph, oacc[d0 + x], 0, 0, 0);
        }
#pragma unroll
        for (int x = 0; x < VB; ++x)
          oacc[d0 + x] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[x], pl, oacc[d0 + x], 0, 0, 0);
      }
    }
    if (PRIO) __builtin_amdgcn_s_setprio(0);
  };

  look(it0);
  fetch(rw.lo + it0 * KT);
  if (it0 + 1 < it1) look(it0 + 1);
  stash(0, rw.lo + it0 * KT);
  __syncthreads();
  for (int it = it0; it < it1; ++it) {
    const int kb = rw.lo + it * KT;
    const bool more = it + 1 < it1;
    if (more) {
      fetch(kb + KT);
      if (it + 2 < it1) look(it + 2);
    }
    // does any row of the wave see a key of the tile?
    if (rw.live && kb <= rw.w_last && (a.window <= 0 || rw.w_first - (kb + KT - 1) < a.window))
      compute((it - it0) & 1, kb);
    if (more) stash((it - it0 + 1) & 1, kb + KT);
    __syncthreads();
  }
  const float lsum = flash_pair_sum(l_run);
  if (SPLIT && parts > 1) {
    float* x = lf_part(a, blockIdx.z, w, NDV) + 4 * lane;
#pragma unroll
    for (int dt = 0; dt < NDV; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<f32x4*>(x + (4 * dt + i) * 256) =
            f32x4{oacc[dt][4 * i], oacc[dt][4 * i + 1], oacc[dt][4 * i + 2], oacc[dt][4 * i + 3]};
    *reinterpret_cast<f32x4*>(x + 4 * NDV * 256) = f32x4{m_run, lsum, 0.f, 0.f};
    return;
  }
  lf_finish<NDV>(a, rw, hh, c0, oacc, m_run, lsum);
}

// The parts of a row block put together: the rows, lanes and registers of the kernel above, a workgroup
// for each 32 columns of every wave's part (one for all of them, one wave per SIMD that reads part after part:
// 16.4 instead of 12.2 us for 256 row blocks of up to 5 parts x 69 KB; of up to 3 parts 8.2).
template <int NDV, int KT, int CS>
__global__ void __launch_bounds__(256)
latent_flash_merge_kernel(LatentFlashArgs a) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, dt = blockIdx.z;
  const LfRows rw = lf_rows<KT, CS, true>(a, w, lane & 31);
  if (rw.ntok <= 0) return;
  const int parts = min(a.nparts, (rw.ntile + a.per - 1) / a.per);
  if (parts <= 1 || !rw.live) return;
  float m = -INFINITY, lsum = 0.f;
  f32x16_t oacc[1];
#pragma unroll
  for (int i = 0; i < 16; ++i) oacc[0][i] = 0.f;
#pragma unroll 2
  for (int z = 0; z < parts; ++z) {
    const float* x = lf_part(a, z, w, NDV) + 4 * lane;
    const f32x4 ml = *reinterpret_cast<const f32x4*>(x + 4 * NDV * 256);
    const float mn = fmaxf(m, ml[0]);
    const float w0 = __builtin_amdgcn_exp2f(m - mn), w1 = __builtin_amdgcn_exp2f(ml[0] - mn);
    m = mn;
    lsum = lsum * w0 + ml[1] * w1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(x + (4 * dt + i) * 256);
#pragma unroll
      for (int e = 0; e < 4; ++e) oacc[0][4 * i + e] = oacc[0][4 * i + e] * w0 + v[e] * w1;
    }
  }
  lf_finish<1>(a, rw, lane >> 5, 32 * (NDV * (w % CS) + dt), oacc, m, lsum);
}

template <int NK, int NDV, int KT, int WPS, int CS, bool SPLIT>
static void lf_launch(const LatentFlashArgs& a, dim3 grid, hipStream_t st) {
  constexpr int TILES = 2 * (2 * KT * (16 * NK + 8) + 64);
  const int need = lf_nrows(CS) * a.rd * 2, bytes = need > TILES ? need : TILES;
  auto* f = &latent_flash_kernel<NK, NDV, KT, WPS, CS, SPLIT>;
  if (bytes > 64 * 1024)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(f), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  hipLaunchKernelGGL(f, grid, dim3(256), bytes, st, a);
  if (SPLIT)
    hipLaunchKernelGGL((latent_flash_merge_kernel<NDV, KT, CS>), dim3(grid.x, grid.y, NDV), dim3(256), 0, st, a);
}

}  // namespace

static int lf_split(int R, int rd) { return R <= 256 && R + rd <= 320 ? 1 : 2; }

// Queries per work item: a workgroup's rows are those of min(H, 16) heads.
EIA_API int eia_latent_flash_queries(int H, int R, int rd) {
  return H < 1 || R < 1 || rd < 0 ? 0 : lf_nrows(lf_split(R, rd)) / (H < 16 ? H : 16);
}
// Keys per tile (what parts are counted in) and 32-column tiles of a wave's part in the workspace.
EIA_API int eia_latent_flash_keys(int R, int rd) { return lf_split(R, rd) == 1 ? 64 : 32; }
EIA_API int eia_latent_flash_columns(int R, int rd) {
  return (R <= 128 && R + rd <= 160) || (R <= 256 && R + rd > 320) ? 4 : 8;
}

// Prompt portions: the arguments are those of eia_latent_attn_mfma, work holds blocks of
// eia_latent_flash_queries queries.  nparts > 1: row blocks of more than per tiles are cut into parts
// of at most that many (nparts * per tiles cover the longest), which meet in part [n_items *
// ceil(H / 16), nparts, 4, 4 eia_latent_flash_columns + 1, 256] fp32.
EIA_API int eia_latent_flash(const void* qa, long qa_st, long qa_sh, const void* qr, long qr_st,
                             long qr_sh, const float* inv_freq, int rot_dims, const void* cache,
                             long cache_row, const int* bt, int ldbt, const int* cu, const int* work,
                             int n_items, const int* positions, const void* gate, long gate_st,
                             void* out, long out_st, long out_sh, float scale, int H, int R, int rd,
                             int bs, int window, const float* sink, int rot_half, float rot_amp,
                             int nparts, int per, float* part, hipStream_t st) {
  if (H < 1 || R < 1 || rd < 0 || bs < 1 || rot_dims > rd || (rot_dims & 1) || cache_row < R + rd ||
      !qa || !cache || !bt || !cu || !work || !positions || !out || n_items < 0 || nparts < 1 ||
      (nparts > 1 && (per < 1 || !part)))
    return EIA_BAD_SHAPE;
  const int Dk = R + rd;
  // 16-byte units must not straddle the latent / rotary boundary or the row end
  if ((R & 7) || (Dk & 7) || (cache_row & 7) || Dk > 640 || R > 512 || out_sh % 4 || out_st % 4)
    return EIA_UNSUPPORTED;
  if (n_items == 0) return EIA_OK;
  const int HB = H < 16 ? H : 16;
  LatentFlashArgs a{(const bf16_t*)qa, qa_st, qa_sh, (const bf16_t*)qr, qr_st, qr_sh, inv_freq,
                    rot_dims, rot_half, rot_amp, (const bf16_t*)cache, cache_row, bt, ldbt, positions,
                    cu, work, (const bf16_t*)gate, gate_st, (bf16_t*)out, out_st, out_sh, sink, scale,
                    H, R, rd, bs, HB, window, per, nparts, n_items, part};
  // With parts the grid is padded to whole rounds of the XCDs, so that the parts of a row block and their merge share
  // one (us without / with, window 1024: 1000 tokens behind 1900, 8 heads of 128 + 32 31.7 / 26.3; 300 behind 1000, 16 of
  // 256 + 32 42.2 / 38.4).
  const int y = (H + HB - 1) / HB, pad = nparts == 1 || y % 8 == 0 ? 1 : y % 4 == 0 ? 2 : y % 2 == 0 ? 4 : 8;
  const dim3 grid((n_items + pad - 1) / pad * pad, y, nparts);
#define LF_GO(NK, NDV, KT, WPS, CS)                                       \
  do {                                                                    \
    if (nparts > 1) lf_launch<NK, NDV, KT, WPS, CS, true>(a, grid, st);   \
    else lf_launch<NK, NDV, KT, WPS, CS, false>(a, grid, st);             \
  } while (0)
  if (R <= 128 && Dk <= 160) LF_GO(10, 4, 64, 2, 1);
  else if (R <= 256 && Dk <= 288) LF_GO(18, 8, 64, 1, 1);
  else if (R <= 256 && Dk <= 320) LF_GO(20, 8, 64, 1, 1);
  else if (R <= 256) LF_GO(40, 4, 32, 1, 2);
  else if (Dk <= 576) LF_GO(36, 8, 32, 1, 2);
  else LF_GO(40, 8, 32, 1, 2);
#undef LF_GO
  EIA_LAUNCH_CHECK();
}
