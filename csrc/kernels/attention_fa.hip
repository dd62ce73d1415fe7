// K2 (long prompts): paged flash-attention prefill on v_mfma_f32_32x32x16_bf16, D = 128.
//
// Work split: a workgroup of 8 waves owns HPW query heads of one KV group -- 4, 2 or 1, as many as
// divide the group -- and 256 / HPW queries of one sequence (wave w: head HPW*hg + w % HPW, queries
// q0 + 32*(w / HPW) + [0, 32)), so every 64-key K/V tile staged in LDS feeds 256 query rows.
// One 4096-token causal prompt, 40 heads on 8 (one head per workgroup): 225 us on an MI355X, 16 on 8
// (two): 143 us, against 749 and 381 us in the 16-query register form (attention.hip), which reads
// every K/V unit once per head and 48 or 96 queries; equal below about 100 tokens.  These groups keep
// that form's exact running maximum and normalise by the weights as rounded, which keeps their error
// against 64 bits (1.94e-3 to 1.93e-3; deferred and unrounded, as with four heads, 2.0e-3 and 205 us).
//
// Per wave and tile (swapped products, guide §3 "An accumulator tile as the next MFMA's
// operand"):
//   S^T[key, q] = K Q^T   : A = K rows from LDS, B = Q^T fragments held in registers,
//                           2 x 8 MFMAs (two 32-key halves x 8 k-steps of 16 dims)
//   O^T[d, q]  += V^T P^T : A = V^T rows from LDS, B = P^T taken straight from the S^T
//                           accumulators (no LDS round trip, no lane movement), 4 x 4 MFMAs
// Each lane owns ONE query column q = lane & 31 of S^T and O^T, so the online softmax (max,
// exp2, running sum, O rescale) is lane-local but for one xor-32 shuffle per tile.
// Key order: accumulator element j of lane half h in k-step s is S^T row 16s+8(j>>2)+4h+(j&3);
// feeding K row pi(R) (bits 2 and 3 of R swapped) into A-row R makes that element the
// PHYSICAL key 16s + 8h + j, so the V^T operand of the same k-step is 8 consecutive keys --
// one 16-B LDS read per lane.
//
// LDS (70 KiB): two buffers of [K 64 x (128+8) | V^T 128 x (64+8)] bf16.  One 16-B
// pad per row makes every ds_read_b128 group conflict-free (K slot = (row + chunk) mod 16,
// V^T slot = (9 d + chunk) mod 16; a 16-lane read group touches rows distinct mod 16 under pi)
// AND keeps a lane's fragment addresses one base register plus immediate offsets (an XOR
// swizzle costs VALU address math on every read).  Tile i+1 is fetched to registers before
// tile i is multiplied and written to the other buffer after it; one barrier per tile.
// Softmax: deferred rescale (the running max moves only when a column's tile max exceeds it by
// more than 2^8, guide T13), row max combined across the two lane halves by permlane32_swap.
// Measured variants (profiles/prefill_attn_fa_r2.log): 4-wave workgroups (two per CU), other
// MFMA / exp orders: all within 3 %; a software pipeline holding two tiles' S (QK(i+1) beside
// the exp work of tile i) and two 32-query sub-blocks per wave (one wave per SIMD) both exceed
// the register file and spill.  Round 4 (profiles/prefill_attn_fa_r4.md): raw v_exp_f32, a
// branch-free mask, tree max / sum chains and dwordx4 output stores
// (65x128: 135 -> 174 TFLOP/s); fetching K/V two tiles ahead (+24 VGPRs) was slower at 1x8192
// (800 vs 757 us) -- the one-tile-ahead fetch is not the bound there -- and a software
// pipeline computing S of tile i+1 beside the exponentials of tile i (three LDS buffers, two S
// register sets, 256 VGPRs) ran at 0.81x, and running the two wave halves half a tile apart
// (two raw barriers per tile, the younger half one slot behind, so one wave of each SIMD is in
// its softmax while the other is in P.V) at 0.92-0.94x (profiles/prefill_attn_fa_r4.md).
// Pages looked up a tile ahead, LDS fragments read ahead of their products and matrix products first (a priority
// per phase instead of one for the younger half of the waves): 32 heads on 8, 1 x 8192 582 -> 543 us, 1 x 2048 72 -> 65,
// 40 heads 1 x 4096 232 -> 219, the same bits.  A tile and wave takes 1020 cycles of matrix products and about 1500
// of vector instructions, two waves on a SIMD.
//
// Launches of fewer workgroups than CUs wait for their longest one (a tile of 64 keys takes 1.65 us): there blocks
// are cut along the keys (CUT; attention.py fa_parts says where), parts hand over fp32 sums as their lanes hold
// them, and a second kernel puts them together.  32 heads on 8, 100 tokens behind 2000: 58.9 -> 20.6 us, 1000 behind
// 2000 80.8 -> 59.4, 1 x 1000 31.6 -> 25; 16 on 4, 500 behind 1000 44.1 -> 21.6, 1 x 4000 109 -> 94; error against 64
// bits 2.35e-3 -> 2.29e-3.  Uncut launches run as before (1 x 8192 522, 4 x 300 14.6).
#include "eia_common.h"

namespace {

typedef __attribute__((ext_vector_type(16))) float f32x16_t;

constexpr int FD = 128;        // head dim
constexpr int FKB = 64;        // keys per tile
constexpr int FROWS = 256;     // (query, head) rows per workgroup
constexpr int FTHREADS = 512;  // 8 waves
constexpr int KS = FD + 8;           // K row stride (elements)
constexpr int VS = FKB + 8;          // V^T row stride (elements)
constexpr int KBUF = FKB * KS, BUF = KBUF + FD * VS;
constexpr float DEFER_LOG2 = 8.f;
    // rescale only when the max grows by > 2^8

EIA_DEV int perm_row(int R) { return (R & ~12) | ((R & 4) << 1) | ((R & 8) >> 1); }
EIA_DEV float pair_max(float v) {    // max with lane l ^ 32
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
EIA_DEV float pair_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// The key tiles of a query block: from key lo on (64-aligned), n of them.
struct KeyTiles { int lo, n; };

EIA_DEV int first_key(int qa, int sliding_window, int chunk_size) {
  int lo = 0;
  if (sliding_window > 0) lo = max(lo, qa - sliding_window + 1);
  if (chunk_size > 0) lo = max(lo, (qa / chunk_size) * chunk_size);
  return lo;
}

EIA_DEV KeyTiles key_tiles(int q0, int queries, int qlen, int L, int causal, int sliding_window, int chunk_size) {
  const int ctx = L - qlen, qlast = min(q0 + queries, qlen) - 1;
  const int hi = causal ? min(L, ctx + qlast + 1) : L;
  const int lo = first_key(ctx + q0, sliding_window, chunk_size) & ~(FKB - 1);
  return {lo, (hi - lo + FKB - 1) / FKB};
}

// Where the keys of query blocks are cut: at most `per` tiles a part, `most` parts a block.  A wave's part of
// O^T lies in o as its lanes hold it ([part][16 registers of four][64 lanes]), maxima and sums of its 32
// queries in ml.
// apart: the parts of a block do not stand together in the grid, whose slowest places they are.
struct KeyParts {
  float* o; float2* ml;
  int per, most, apart;
};

EIA_DEV int parts_of(int tiles, const KeyParts& cut) { return max(1, min((tiles + cut.per - 1) / cut.per, cut.most)); }

// Output rows of a wave, one 32-dim tile: lane (q, h) holds d = 8 j + 4 h + [0, 4) of it, the two lane halves of
// a query own alternating 8-B pieces.  One permlane32_swap per dword pairs pieces j / j+1 so each lane
// stores 16 contiguous bytes: dwordx4 stores instead of dwordx2.
// Both lanes of a swap pair hold the same query, so they are valid (or exited) together.
EIA_DEV void put_rows(bf16_t* op, const f32x16_t& o, float inv) {
  uint2 pk[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    bf16x4 o4;
#pragma unroll
    for (int r = 0; r < 4; ++r) o4[r] = f2bf(o[4 * j + r] * inv);
    pk[j] = __builtin_bit_cast(uint2, o4);
  }
#pragma unroll
  for (int j = 0; j < 4; j += 2) {
    const auto rx = __builtin_amdgcn_permlane32_swap(pk[j].x, pk[j + 1].x, false, false);
    const auto ry = __builtin_amdgcn_permlane32_swap(pk[j].y, pk[j + 1].y, false, false);
    *reinterpret_cast<uint4*>(op + 8 * j) = make_uint4(rx[0], ry[0], rx[1], ry[1]);
  }
}

template <int HPW, bool CUT>
__global__ void __launch_bounds__(FTHREADS, 1)
paged_prefill_fa_kernel(const bf16_t* __restrict__ q, long q_stride, bf16_t* __restrict__ out,
                        long out_stride, const bf16_t* __restrict__ kc,
                        const bf16_t* __restrict__ vc, const int* __restrict__ block_tables,
                        int bt_stride, const int* __restrict__ seq_lens,
                        const int* __restrict__ cu_q, const int* __restrict__ work,
                        float scale_log2, int Hq, int Hkv, int bs, int causal, int sliding_window,
                        int chunk_size, KeyParts cut) {
  __shared__ __align__(16) bf16_t lds[2 * BUF];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int r32 = lane & 31, h = lane >> 5;
  // grid (head groups, work items): the heads of one query block are dispatched together and
  // the work list is latest-block-first, so the dispatch order is longest-first over the
  // whole grid (causal blocks grow with their position), not per head
  const int item = CUT && !cut.apart ? blockIdx.z : blockIdx.y, part = cut.apart ? blockIdx.z : blockIdx.y;
  const int s = work[2 * item], q0 = work[2 * item + 1];
  constexpr int FQB = FROWS / HPW;
  const int G = Hq / Hkv, NHG = G / HPW;
  const int kvh = blockIdx.x / NHG, hg = blockIdx.x % NHG;
  const int hq = kvh * G + hg * HPW + w % HPW;
  const int qsub = w / HPW;
  const int qbeg = cu_q[s], qlen = cu_q[s + 1] - qbeg;
  if (q0 >= qlen) return;                                  // workgroup-uniform
  const int L = seq_lens[s], ctx = L - qlen;
  const bool window = sliding_window > 0 || chunk_size > 0;
  // this lane's query column
  const int qi = q0 + 32 * qsub + r32;
  const bool qvalid = qi < qlen;
  const int qe = min(qi, qlen - 1);
  const long tok = qbeg + qe;
  const int qa = ctx + qe;
  const int q_lo = first_key(qa, sliding_window, chunk_size);
  // Q^T fragments (B operand): k-step t = dims [16t, 16t+16), lane half h holds 16t+8h..+8
  bf16x8 qf[FD / 16];
  {
    const bf16_t* qp = q + tok * q_stride + (long)hq * FD + 8 * h;
#pragma unroll
    for (int t = 0; t < FD / 16; ++t) qf[t] = *reinterpret_cast<const bf16x8*>(qp + 16 * t);
  }

  // workgroup key range: key_tiles written out, through which the compiler took another layout of the loop in uncut launches
  // (28 heads on 4, ten prompts of 109 behind 1837 93.4 -> 94.2 us, twenty of 64 behind 1800 136.1 -> 137.9)
  const int qlast = min(q0 + FQB, qlen) - 1;
  const int hi = causal ? min(L, ctx + qlast + 1) : L;
  int lo = first_key(ctx + q0, sliding_window, chunk_size) & ~(FKB - 1);
  int ntile = (hi - lo + FKB - 1) / FKB, parts = 1;
  if constexpr (CUT) {
    parts = parts_of(ntile, cut);
    const int each = (ntile + parts - 1) / parts;
    if (part >= parts) return;
    lo += FKB * each * part;
    ntile = min(each, ntile - each * part);
  }
  // this wave's key range
  const int wq0 = q0 + 32 * qsub;                          // wave's first query
  const bool wave_live = wq0 < qlen;
  const int wq1 = min(wq0 + 32, qlen) - 1;                 // wave's last valid query
  const int w_hi = !wave_live ? 0 : (causal ? min(L, ctx + wq1 + 1) : L);
  const int w_lo = wave_live ? first_key(ctx + wq0, sliding_window, chunk_size) : 0;      // no query of the wave sees below

  const int* bt = block_tables + (long)s * bt_stride;
  // the page of a tile is looked up a tile ahead of its fetch: the fetch would wait for it
  int o = lo % bs, at = lo / bs, page = ntile > 0 ? bt[at] : 0;          // the next fetch: token in its page, page
  auto look = [&] {
    o += FKB;
    if (o == bs) o = 0, ++at;
    page = bt[at];
  };
  auto fetch = [&](bf16x8 (&st)[4]) {
    const long base = ((long)__builtin_amdgcn_readfirstlane(page) * Hkv + kvh) * (long)bs * FD;
    const bf16_t* kp = kc + base + (long)o * FD;          // 64 rows x 128, contiguous
    const bf16_t* vp = vc + base + o;                     // 128 rows x 64 keys, row stride bs
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int id = tid + FTHREADS * i;
      st[i] = *reinterpret_cast<const bf16x8*>(kp + 8 * id);
      st[2 + i] = *reinterpret_cast<const bf16x8*>(vp + (long)(id >> 3) * bs + 8 * (id & 7));
    }
  };
  auto stash = [&](int buf, const bf16x8 (&st)[4]) {
    bf16_t* kl = lds + buf * BUF;
    bf16_t* vl = kl + KBUF;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int id = tid + FTHREADS * i;
      *reinterpret_cast<bf16x8*>(kl + (id >> 4) * KS + 8 * (id & 15)) = st[i];
      *reinterpret_cast<bf16x8*>(vl + (id >> 3) * VS + 8 * (id & 7)) = st[2 + i];
    }
  };

  f32x16_t oacc[FD / 32];
#pragma unroll
  for (int dt = 0; dt < FD / 32; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[dt][i] = 0.f;
  float m_run = (-INFINITY), l_run = 0.f;
  const int krow0 = perm_row(r32);

  auto compute = [&](int buf, int kb) {
    // lane fragment bases: K row pi(lane) (+32 rows for the second half), chunk h; V^T row
    // lane (+32 rows per d-tile), chunk h -- every read below is base + immediate
    const bf16_t* kf0 = lds + buf * BUF + krow0 * KS + 8 * h;
    const bf16_t* vf0 = lds + buf * BUF + KBUF + r32 * VS + 8 * h;
    f32x16_t sacc[2];
    // reads of LDS go four fragments ahead of the products, kept there by the barriers to the scheduler:
    // left alone, each is moved to its product, which then waits for it
    bf16x8 kf[2][4];
    auto keys = [&](int b) {
#pragma unroll
      for (int x = 0; x < 4; ++x)
        kf[b & 1][x] = *reinterpret_cast<const bf16x8*>(kf0 + 32 * KS * (x & 1) + 16 * (2 * b + (x >> 1)));
    };
    // matrix products go first, the second ones before all: else the two waves of a SIMD wait for the same unit in turn
    __builtin_amdgcn_s_setprio(1);
    keys(0);
#pragma unroll
    for (int b = 0; b < FD / 32; ++b) {
      if (b + 1 < FD / 32) keys(b + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int sh = x & 1, t = 2 * b + (x >> 1);
        sacc[sh] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[b & 1][x], qf[t], t == 0 ? f32x16_t{} : sacc[sh], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_setprio(0);
    // element i of half sh is key kb + 32 sh + 16 (i >> 3) + 8 h + (i & 7)
    const bool whole = !window && kb + FKB <= L && (!causal || kb + FKB - 1 <= ctx + wq0);
    mfma_settle(sacc[0], sacc[1]);
    if (!whole) {
      // key kp is visible iff q_lo <= kp <= kmax: one unsigned compare per score, no branches
      const int kmax = causal ? min(L - 1, qa) : L - 1;
      const unsigned lim = (unsigned)(kmax - q_lo);
      const int d0 = kb + 8 * h - q_lo;
#pragma unroll
      for (int sh = 0; sh < 2; ++sh)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const unsigned dk = (unsigned)(d0 + 32 * sh + 16 * (i >> 3) + (i & 7));
          sacc[sh][i] = dk <= lim ? sacc[sh][i] : (-INFINITY);
        }
    }
    // four independent max3 chains instead of one 16-deep dependent chain
    float mx4[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      mx4[c] = sacc[c >> 1][8 * (c & 1)];
#pragma unroll
      for (int j = 1; j < 8; ++j) mx4[c] = fmaxf(mx4[c], sacc[c >> 1][8 * (c & 1) + j]);
    }
    const float mx = fmaxf(fmaxf(mx4[0], mx4[1]), fmaxf(mx4[2], mx4[3]));
    const float mt = pair_max(mx) * scale_log2;
    const bool grow = mt > m_run + (HPW == 4 ? DEFER_LOG2 : 0.f);
    if (__any(grow)) {                                     // wave-uniform
      const float m_new = grow ? mt : m_run;
      const float alpha = grow ? exp2f(m_run - m_new) : 1.f;
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < FD / 32; ++dt) oacc[dt] *= alpha;
    }
    const float muse = m_run == (-INFINITY) ? 0.f : m_run;
    // row sums as four independent chains.  V^T fragments and exponentials of a k-step stand beside the
    // products of the one before.
    bf16x8 pb[4];
    float ps4[4] = {0.f, 0.f, 0.f, 0.f};
    auto expk = [&](int ks) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float p = __builtin_amdgcn_exp2f(fmaf(sacc[ks >> 1][8 * (ks & 1) + j], scale_log2, -muse));
        pb[ks][j] = f2bf(p);
        ps4[ks] += HPW == 4 ? p : bf2f(pb[ks][j]);
      }
    };
    bf16x8 vf[2][4];
    auto values = [&](int ks) {
#pragma unroll
      for (int dt = 0; dt < FD / 32; ++dt) vf[ks & 1][dt] = *reinterpret_cast<const bf16x8*>(vf0 + 32 * VS * dt + 16 * ks);
    };
    auto pv = [&](int ks) {
#pragma unroll
      for (int dt = 0; dt < FD / 32; ++dt) oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[ks & 1][dt], pb[ks], oacc[dt], 0, 0, 0);
    };
    __builtin_amdgcn_s_setprio(2);
    values(0);
    __builtin_amdgcn_sched_barrier(0);
    expk(0);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (ks < 3) {
        values(ks + 1);
        expk(ks + 1);
      }
      pv(ks);
      __builtin_amdgcn_sched_barrier(0);
    }
    l_run += (ps4[0] + ps4[1]) + (ps4[2] + ps4[3]);
    __builtin_amdgcn_s_setprio(0);
  };

  bf16x8 st[4];
  if (ntile > 0) {
    fetch(st);
    if (ntile > 1) look();
    stash(0, st);
  }
  __syncthreads();
  for (int it = 0; it < ntile; ++it) {
    const int kb = lo + FKB * it;
    const bool more = it + 1 < ntile;
    if (more) {
      fetch(st);
      if (it + 2 < ntile) look();
    }
    // wave-uniform: does any of this wave's queries see a key of the tile?
    if (kb < w_hi && kb + FKB > w_lo) compute(it & 1, kb);
    if (more) stash((it + 1) & 1, st);
    __syncthreads();
  }

  const float lt = pair_sum(l_run);
  if (CUT && parts > 1) {
    if (!wave_live) return;
    const long at = (((long)item * cut.most + part) * gridDim.x + blockIdx.x) * (FTHREADS / 64) + w;
    f32x4* po = reinterpret_cast<f32x4*>(cut.o) + at * (FD / 8 * 64) + lane;
#pragma unroll
    for (int dt = 0; dt < FD / 32; ++dt)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        po[(4 * dt + j) * 64] = f32x4{oacc[dt][4 * j], oacc[dt][4 * j + 1], oacc[dt][4 * j + 2], oacc[dt][4 * j + 3]};
    if (h == 0) cut.ml[at * 32 + r32] = make_float2(m_run, lt);
    return;
  }
  if (!qvalid) return;
  const float inv = lt > 0.f ? 1.f / lt : 0.f;
  bf16_t* op = out + tok * out_stride + (long)hq * FD + 8 * h;
#pragma unroll
  for (int dt = 0; dt < FD / 32; ++dt) put_rows(op + 32 * dt, oacc[dt], inv);
}

// A workgroup puts the parts of one wave's 32 queries together, wave dt 32 dims of them; the head group comes
// first in both grids, so where there are a multiple of eight the parts are read on the XCD that wrote them.
template <int HPW>
__global__ void __launch_bounds__(256)
paged_prefill_fa_merge_kernel(bf16_t* __restrict__ out, long out_stride, const int* __restrict__ seq_lens,
                              const int* __restrict__ cu_q, const int* __restrict__ work, int Hq, int Hkv,
                              int causal, int sliding_window, int chunk_size, KeyParts cut) {
  constexpr int FQB = FROWS / HPW, NP = 4;
  const int item = blockIdx.z, w = blockIdx.y, lane = threadIdx.x & 63, dt = threadIdx.x >> 6;
  const int r32 = lane & 31, h = lane >> 5;
  const int s = work[2 * item], q0 = work[2 * item + 1];
  const int qbeg = cu_q[s], qlen = cu_q[s + 1] - qbeg;
  if (q0 + 32 * (w / HPW) >= qlen) return;
  const KeyTiles kt = key_tiles(q0, FQB, qlen, seq_lens[s], causal, sliding_window, chunk_size);
  const int parts = parts_of(kt.n, cut);
  if (parts == 1) return;
  const long step = (long)gridDim.x * (FTHREADS / 64);
  const long at = ((long)item * cut.most * gridDim.x + blockIdx.x) * (FTHREADS / 64) + w;
  const f32x4* po = reinterpret_cast<const f32x4*>(cut.o) + at * (FD / 8 * 64) + dt * 4 * 64 + lane;
  const float2* ml = cut.ml + at * 32 + r32;
  f32x16_t o;
#pragma unroll
  for (int i = 0; i < 16; ++i) o[i] = 0.f;
  float m = (-INFINITY), l = 0.f;
  for (int p0 = 0; p0 < parts; p0 += NP) {
    float2 x[NP];
    f32x4 v[NP][4];
#pragma unroll
    for (int k = 0; k < NP; ++k) {                         // (a part past the last: the last one again, weight 0)
      const long p = min(p0 + k, parts - 1) * step;
      x[k] = ml[p * 32];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[k][j] = po[p * (FD / 8 * 64) + j * 64];
    }
    float mx = m;
#pragma unroll
    for (int k = 0; k < NP; ++k) mx = fmaxf(mx, x[k].x);
    const float ref = mx == (-INFINITY) ? 0.f : mx, old = __builtin_amdgcn_exp2f(m - ref);
    m = mx;
    l *= old;
    o *= old;
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      if (p0 + k >= parts) break;
      const float c = __builtin_amdgcn_exp2f(x[k].x - ref);
      l += c * x[k].y;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[4 * j + i] += c * v[k][j][i];
    }
  }
  const int qi = q0 + 32 * (w / HPW) + r32;
  if (qi >= qlen) return;
  const int G = Hq / Hkv, NHG = G / HPW;
  const int hq = blockIdx.x / NHG * G + blockIdx.x % NHG * HPW + w % HPW;
  put_rows(out + (long)(qbeg + qi) * out_stride + (long)hq * FD + 8 * h + 32 * dt, o, l > 0.f ? 1.f / l : 0.f);
}

}  // namespace

// work = [seq, first query] pairs with blocks of 256 / HPW queries (attention.prefill_query_block);
// grid (Hkv * G / HPW, n_work).  Requires D = 128, block size % 64 == 0.
// parts > 1: blocks of more than `per` key tiles are cut into up to `parts` parts; ws holds
// n_work * parts * (Hq / HPW) * 256 * (128 + 2) floats.  (Longer ones than parts * per get longer parts.)
EIA_API int eia_paged_prefill_fa(const void* q, long q_stride, void* out, long out_stride,
                                 const void* k_cache, const void* v_cache,
                                 const int* block_tables, int bt_stride, const int* seq_lens,
                                 const int* cu_q, const int* work, int n_work, float scale, int Hq,
                                 int Hkv, int D, int bs, int causal, int sliding_window,
                                 int chunk_size, int parts, int per, float* ws, hipStream_t st) {
  if (Hkv <= 0 || Hq % Hkv != 0) return EIA_BAD_SHAPE;
  if (D != FD || bs % FKB != 0 || out_stride % 8 != 0) return EIA_UNSUPPORTED;   // (16-B output stores)
  if (n_work == 0) return EIA_OK;
  const int G = Hq / Hkv, hpw = G % 4 == 0 ? 4 : G % 2 == 0 ? 2 : 1;
  if (parts > 1 && (per < 1 || !ws || n_work > 65535 || parts > 65535)) return EIA_BAD_SHAPE;
  // Workgroups go to XCDs, and to the parts of one, in turn.  Where an even number of parts stand together, the first parts
  // of all blocks, of which there are most, meet in some places, and launches of several rounds wait for those: 1350
  // launches of 4 to 256 blocks, in all numbers of parts, apart against together beyond 256 parts: even numbers 0.88 to
  // 0.97 of the time, odd ones 0.98.  16 heads on 4, 3754 tokens 118 -> 95 us, two of 1639 55.7 -> 47.7; 28 on 4, two of 766
  // 37.6 -> 35.5.  In one round those that stand together read fewer keys on an XCD: 4 on 1, 2023 tokens 27.9 -> 24.9.
  const int groups = Hq / hpw;
  KeyParts cut{nullptr, nullptr, per, parts, parts > 1 && (long)n_work * groups * parts > 256};
  if (parts > 1) {
    cut.o = ws;
    cut.ml = reinterpret_cast<float2*>(ws + (long)n_work * parts * groups * FROWS * FD);
  }
#define FA_GO(HPW)                                                                                  \
  do {                                                                                              \
    const float sl = scale * 1.4426950408889634f;                                                   \
    const dim3 grid = cut.apart ? dim3(groups, n_work, parts) : parts > 1 ? dim3(groups, parts, n_work) : dim3(groups, n_work);   \
    auto* f = parts > 1 ? paged_prefill_fa_kernel<HPW, true> : paged_prefill_fa_kernel<HPW, false>; \
    hipLaunchKernelGGL(f, grid, dim3(FTHREADS), 0, st, (const bf16_t*)q, q_stride, (bf16_t*)out,    \
                       out_stride, (const bf16_t*)k_cache, (const bf16_t*)v_cache, block_tables,    \
                       bt_stride, seq_lens, cu_q, work, sl, Hq, Hkv, bs, causal, sliding_window,    \
                       chunk_size, cut);                                                            \
    if (parts > 1)                                                                                  \
      hipLaunchKernelGGL(paged_prefill_fa_merge_kernel<HPW>, dim3(Hq / HPW, FTHREADS / 64, n_work), \
                         dim3(256), 0, st, (bf16_t*)out, out_stride, seq_lens, cu_q, work, Hq, Hkv, \
                         causal, sliding_window, chunk_size, cut);                                  \
  } while (0)
  if (hpw == 4) FA_GO(4); else if (hpw == 2) FA_GO(2); else FA_GO(1);
#undef FA_GO
  EIA_LAUNCH_CHECK();
}
