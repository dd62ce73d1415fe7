// K9 (prefill-sized MoE): grouped GEMM over device-side expert slices on v_mfma_f32_32x32x16_bf16.
//
//   out[p][:] = X[row(p)][:] . W_e^T          (p in expert e's slice [offs[e], offs[e+1]))
//   SwiGLU form: W_e = [gate; up] (2I rows), out[p][c] = silu(g_c) * u_c, I columns
//
// The expert slices come from eia_moe_align on the device, so nothing here is known to the
// host: the grid is an upper bound on the tiles ((ceil(rows / tile) + experts) M tiles), every
// workgroup maps blockIdx.x to (expert, M tile, N tile) by a wave-wide scan of the per-expert tile
// counts, and surplus workgroups exit.  No host synchronisation, no per-expert launches, and
// the same launch is valid inside a HIP graph.
//
// Tile 64 MU (M) x 64 NU (N) x 64 (K), four waves of 32 MU x 32 NU (MFMA tiles of 32 x 32).  Operand
// roles are swapped (A = W rows, B = X^T) so a lane ends up with one output ROW and runs of 4 consecutive
// columns -> 8-B stores; in the SwiGLU form the first half of a wave's N sub-tiles are gate rows and the
// others the matching up rows, so silu(g) * u is formed in registers.  A slice's 64-row units are shared
// evenly among as few M tiles as MAXMU allows, MU of each on the device; the host picks (NU, MAXMU)
// by the mean rows per expert (grouped_form).
//
// Tiles go from memory straight to LDS (16 bytes per lane; X rows gathered through row_idx): two K
// steps of X and three of W, the next accesses spread between the products.  A step's first
// fragments are read, behind the barrier, before the products of the last quarter of the step before.
// The accesses are inline asm: behind the compiler's own, which it takes for ones that may end out of
// order, every read of LDS is waited for at once.  Row r keeps its 16-byte chunk c at c ^ (r / 2 % 8):
// fragment reads of 16 rows meet all 64 banks.  An XCD takes a contiguous share of the tiles, ordered by
// expert, N tile, M tile, so that it reads the weights of its own experts only, and a weight tile once for
// all M tiles.
//
// The products of 128 x 128 tiles need as many cycles as their bytes take through a CU's 64-byte path from
// L2, and a larger tile fewer bytes; without any access the products run at the rate of a large library
// product (1180 TFLOP/s).  MI355X, us, cold weights, gate_up + down, 128 x 128 tiles in one form / now:
//   16 experts of 2048 x 1024, 128 rows each 48 + 27 / 38 + 23; 256: 65 + 41 / 47 + 30; 400: 80 + 50 / 61 + 39
//   8 of 1024 x 512, 340 rows: 14.8 + 10.9 / 12.0 + 9.5; 1024: 34 + 24 / 25 + 18.5
//   8 of 4096 x 14336, 122 rows: 442 + 305 / 376 + 234 (2.8 GB of weights: 550); 256: 717 + 416 / 568 + 297
#include "eia_common.h"
#include "eia_moe_tiles.h"
#include <math.h>

namespace {

typedef __attribute__((ext_vector_type(16))) float f32x16_t;

constexpr int BK = 64;
constexpr int UNIT = 64 * BK;                      // elements of 64 rows of one K step
constexpr int XS = 2, WS = 3;                      // K steps of X and of W in LDS

EIA_DEV float silu_f(float x) { return __fdividef(x, 1.f + __expf(-x)); }

struct GroupedArgs {
  const bf16_t* X; long ldx; const int* row_idx; const bf16_t* W; long w_estride; const int* offs;
  int E, I, K, NT; bf16_t* out; long ldo; int relu2;
};

// One tile: MU x 64 rows from row m0 of the slice [rb, rb + rows) of expert weights We, N tile n_tile.
template <bool SWIGLU, int MU, int NU, int MAXMU, bool FRONT>
EIA_DEV void grouped_tile(const GroupedArgs& a, bf16_t* lds, const bf16_t* We, int rb, int rows, int m0,
                          int n_tile) {
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r32 = lane & 31, h = lane >> 5;
  // Access i of a step stands behind product i * RATE, with FRONT before all products.  Small tiles wait for memory rather than for the
  // access path: 8 experts of 4096 x 14336, 64 rows, gate_up 346 us (RATE 2: 366, 8 of 1024 x 512, 512 rows
  // 19.6 against 17.7); a step of large ones with all accesses in front stalls its first products.
  constexpr int RATE = MU == 1 || MU * NU <= 4 ? 1 : 2;
  static_assert((2 * (MU + NU) - 1) * RATE < 4 * MU * NU, "");
  bf16_t* xlds = lds;
  bf16_t* wlds = lds + XS * MAXMU * UNIT;
  // 1 KB accesses of 8 rows, 32 rows apart for the waves' turns: lane -> row lane / 8, LDS chunk lane % 8
  const bf16_t* xsrc[2 * MU];
  const bf16_t* wsrc[2 * NU];
#pragma unroll
  for (int i = 0; i < 2 * MU; ++i) {
    const int r = 32 * i + 8 * w + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    const int p = rb + min(m0 + r, rows - 1);              // rows past the slice clamp
    const long xr = a.row_idx != nullptr ? a.row_idx[p] : p;
    xsrc[i] = a.X + xr * a.ldx + 8 * c;
  }
#pragma unroll
  for (int i = 0; i < 2 * NU; ++i) {
    const int r = 32 * i + 8 * w + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    int wr;
    if (SWIGLU) wr = i < NU ? n_tile * 32 * NU + r : a.I + n_tile * 32 * NU + (r - 32 * NU);
    else wr = n_tile * 64 * NU + r;
    wsrc[i] = We + (long)wr * a.K + 8 * c;
  }
  const int nk = a.K / BK;
  auto put = [&](const bf16_t* src, bf16_t* dst) { glds16(src, lds_offset(dst)); };
  auto fetch_x = [&](int i, int kt, int slot) {
    put(xsrc[i] + kt * BK, xlds + slot * MAXMU * UNIT + (32 * i + 8 * w) * BK);
  };
  auto fetch_w = [&](int i, int kt, int slot) {
    put(wsrc[i] + kt * BK, wlds + slot * NU * UNIT + (32 * i + 8 * w) * BK);
  };
  auto all_x = [&](int kt, int slot) {
#pragma unroll
    for (int i = 0; i < 2 * MU; ++i) fetch_x(i, kt, slot);
  };
  auto all_w = [&](int kt, int slot) {
#pragma unroll
    for (int i = 0; i < 2 * NU; ++i) fetch_w(i, kt, slot);
  };

  // wave (wm, wn): rows [32 MU wm, + 32 MU) of the X tile; W tile rows of N sub-tile nt: plain
  // 32 (NU wn + nt); SwiGLU: the first NU / 2 sub-tiles gate, the others the same columns of up
  const int wm = w & 1, wn = w >> 1;
  int wrow[NU];
#pragma unroll
  for (int nt = 0; nt < NU; ++nt)
    wrow[nt] = SWIGLU ? (nt < NU / 2 ? 0 : 32 * NU) + 32 * (NU / 2 * wn + nt % (NU / 2))
                      : 32 * (NU * wn + nt);
  f32x16_t acc[NU][MU];                                    // [nt][mt]: C^T (rows n, cols m)
#pragma unroll
  for (int i = 0; i < NU; ++i)
#pragma unroll
    for (int j = 0; j < MU; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  bf16x8 wf[2][NU], xf[2][MU];
  auto frags = [&](int kk, int xs, int ws) {
    const int c = 8 * ((2 * kk + h) ^ ((r32 >> 1) & 7));
    const bf16_t* wl = wlds + ws * NU * UNIT + r32 * BK + c;
    const bf16_t* xl = xlds + xs * MAXMU * UNIT + (32 * MU * wm + r32) * BK + c;
#pragma unroll
    for (int nt = 0; nt < NU; ++nt)
      wf[kk & 1][nt] = *reinterpret_cast<const bf16x8*>(wl + wrow[nt] * BK);
#pragma unroll
    for (int mt = 0; mt < MU; ++mt)
      xf[kk & 1][mt] = *reinterpret_cast<const bf16x8*>(xl + 32 * mt * BK);
  };
  // all but the newest step of W is in LDS, and every wave's reads are done
  auto arrive = [&](bool newer) {
    if (newer) {
      if constexpr (NU == 2) asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    }
    __builtin_amdgcn_s_barrier();                          // (__syncthreads would wait for all of them)
    asm volatile("" ::: "memory");
  };

  all_x(0, 0);
  all_w(0, 0);
  if (nk > 1) all_w(1, 1);
  arrive(nk > 1);
  if (nk > 1) all_x(1, 1);
  if (nk > 2) all_w(2, 2);
  // quarter kk of a step's products, its fragments in registers; between them accesses to
  // X(xk) and then W(wk); `from`: products of the step before these
  auto products = [&](int kk, int from, bool fx, int xk, int xslot, bool fw, int wk, int wslot) {
#pragma unroll
    for (int j = 0; j < NU * MU; ++j) {
      const int nt = j / MU, mt = j % MU, at = from + j, i = at / RATE;
      acc[nt][mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[kk & 1][nt], xf[kk & 1][mt], acc[nt][mt], 0,
                                                            0, 0);
      if (at % RATE == 0) {
        if (i < 2 * MU) {
          if (fx) fetch_x(i, xk, xslot);
        } else if (i < 2 * MU + 2 * NU) {
          if (fw) fetch_w(i - 2 * MU, wk, wslot);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  frags(0, 0, 0);
#pragma unroll
  for (int kk = 0; kk < 3; ++kk) {
    frags(kk + 1, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    products(kk, 0, false, 0, 0, false, 0, 0);
  }
  // from step kt to kt + 1: X(kt + 2) goes where X(kt) was, W(kt + 3) where W(kt) was
  int ws = 0;
  auto advance = [&](int kt, auto fx, auto fw) {
    const int xs = kt & 1, wn1 = ws + 1 < WS ? ws + 1 : 0;
    arrive(fx);
    if constexpr (FRONT) {
      if (fx) all_x(kt + 2, xs);
      if (fw) all_w(kt + 3, ws);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      frags(q, xs ^ 1, wn1);
      __builtin_amdgcn_sched_barrier(0);                   // the next fragments before these products
      products((q + 3) & 3, q * NU * MU, fx && !FRONT, kt + 2, xs, fw && !FRONT, kt + 3, ws);
    }
    ws = wn1;
  };
  struct Yes { constexpr operator bool() const { return true; } };
  struct No { constexpr operator bool() const { return false; } };
  int kt = 0;
  for (; kt + 3 < nk; ++kt) advance(kt, Yes{}, Yes{});
  if (kt + 2 < nk) advance(kt++, Yes{}, No{});
  if (kt + 1 < nk) advance(kt++, No{}, No{});
  products(3, 0, false, 0, 0, false, 0, 0);

  // lane: output row m = 32 MU wm + 32 mt + r32; registers 4j..4j+3 = columns 8j + 4h + 0..3 of
  // the N sub-tile
#pragma unroll
  for (int mt = 0; mt < MU; ++mt) {
    const int m = m0 + 32 * MU * wm + 32 * mt + r32;
    if (m >= rows) continue;
    bf16_t* op = a.out + (long)(rb + m) * a.ldo;
#pragma unroll
    for (int nt = 0; nt < (SWIGLU ? NU / 2 : NU); ++nt) {
      const int c0 = n_tile * (SWIGLU ? 32 : 64) * NU + wrow[nt];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        bf16x4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float x = acc[nt][mt][4 * j + r];
          if (SWIGLU) x = silu_f(x) * acc[nt + NU / 2][mt][4 * j + r];
          else if (a.relu2) { x = fmaxf(x, 0.f); x *= x; } // ungated experts: squared ReLU
          v[r] = f2bf(x);
        }
        *reinterpret_cast<bf16x4*>(op + c0 + 8 * j + 4 * h) = v;
      }
    }
  }
}

template <bool SWIGLU, int NU, int MAXMU, int OCC, bool FRONT>
__global__ void __launch_bounds__(256, OCC)
moe_grouped_mfma_kernel(GroupedArgs a) {
  __shared__ __align__(16) bf16_t lds[(XS * MAXMU + WS * NU) * UNIT];
  const int lane = threadIdx.x & 63, E = a.E, NT = a.NT;
  // blockIdx.x -> tile -> (expert, N tile, M tile); every wave for itself, a lane for each of 64 experts.  The first 64
  // come last, so that their slices, read once, serve the search as well (read anew, and the tile's expert by itself
  // once more, three trips to the L2 and twelve more shuffles stood before the first load)
  int lo = 0, hi = 0, nt = 0, incl = 0;                    // the expert's rows, its M tiles, those up to and with it
  auto slices = [&](int e0) {
    const int e = e0 + lane;
    lo = a.offs[min(e, E)];
    hi = a.offs[min(e + 1, E)];
    nt = e < E ? moe_slice_tiles(hi - lo, MAXMU) : 0;
    incl = nt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(incl, o, 64);
      if (lane >= o) incl += v;
    }
  };
  int total = 0;
  for (int e0 = (E - 1) & ~63; e0 >= 0; e0 -= 64) {
    slices(e0);
    total += __builtin_amdgcn_readlane(incl, 63);
  }
  total *= NT;
  const int share = (total + 7) / 8, at = blockIdx.x >> 3;
  const int tile = (blockIdx.x & 7) * share + at;
  if (at >= share || tile >= total) return;                // surplus workgroup (uniform)
  int ex = 0, n_tile = 0, m_tile = 0, m_tiles = 1, rb = 0, rows = 0;
  for (int e0 = 0, base = 0; e0 < E; e0 += 64) {
    if (e0) slices(e0);
    const int q = tile - (base + incl - nt) * NT;
    const unsigned long long hit = __ballot(q >= 0 && q < nt * NT);
    if (hit) {
      const int src = __ffsll(hit) - 1, qe = __builtin_amdgcn_readlane(q, src);
      m_tiles = __builtin_amdgcn_readlane(nt, src);
      rb = __builtin_amdgcn_readlane(lo, src);
      rows = __builtin_amdgcn_readlane(hi, src) - rb;
      ex = e0 + src;
      n_tile = qe / m_tiles;
      m_tile = qe - n_tile * m_tiles;
      break;
    }
    base += __builtin_amdgcn_readlane(incl, 63);
  }
  ex = __builtin_amdgcn_readfirstlane(ex);
  n_tile = __builtin_amdgcn_readfirstlane(n_tile);
  m_tile = __builtin_amdgcn_readfirstlane(m_tile);
  m_tiles = __builtin_amdgcn_readfirstlane(m_tiles);
  rb = __builtin_amdgcn_readfirstlane(rb);
  rows = __builtin_amdgcn_readfirstlane(rows);
  const bf16_t* We = a.W + (long)ex * a.w_estride;
  // Where weights come first (FRONT), tiles of 64 rows fall behind ones of 128 in long K loops: the op with 8 experts
  // of 4096 x 14336, 50 and 55 rows an expert: shares 578 and 573 us, whole tiles 555 and 557; not in short ones: 16
  // of 2048 x 1024, 50 rows 60.8 and 63.8.
  const MoeTile m = moe_slice_tile(rows, m_tiles, m_tile, FRONT && a.K > 2048, MAXMU);
#define GG_TILE(M)                                                                            \
  case M:                                                                                     \
    if constexpr (M <= MAXMU) grouped_tile<SWIGLU, M, NU, MAXMU, FRONT>(a, lds, We, rb, rows, 64 * m.lo, n_tile); \
    break
  switch (m.mu) { GG_TILE(1); GG_TILE(2); GG_TILE(3); GG_TILE(4); GG_TILE(5); }
#undef GG_TILE
}

// Which form multiplies `avg` rows per expert: 0: up to 128 x 128, two workgroups per CU; 1: up to 320 x
// 128, one; 2: up to 256 x 256, one.  Large tiles read less but may leave CUs idle or a second round nearly
// empty, so the estimate counts rounds over 256 CUs, with the tiles of slices 1.8 deviations of
// a random routing shorter and longer than the mean.  A K step of a tile costs its products (0.06 per 64
// x 64), its reads (0.03 per 64 rows) and a constant; fitted to 76 measured shapes (2 to 64 experts, 32 to
// 1024 rows), where its choice is within 1 % of the best form in the mean and 12 % at worst (always form 0:
// 9 % in the mean, always form 1: 7 %).  Wide tiles of up to a unit and a half of rows never won.  Up to 104 rows, where
// hardly a slice needs more than form 0's two units, they are left out too where form 0 just fills the chip, two
// workgroups on every CU, whose overlap the estimate does not see.  The op with 100 rows an expert without / with wide tiles,
// us: 512 tiles of form 0, 64 experts of 1024 x 512 70 / 75, 32 of 1024 x 1024 66 / 68, 16 of 1024 x 2048 65 / 67, 8 of
// 4096 x 4096 197 / 206; 384, 32 of 2048 x 768 94 / 90, 8 of 2048 x 3072 (97 rows) 100 / 91; 1024, 8 of 3072 x 8192
// 286 / 278; 1792, 8 of 4096 x 14336 604 / 588.  With 120 rows 64 of 1024 x 512 95 / 81, 32 of 1024 x 1024 84 / 79.
static int grouped_form(float avg, int E, int N, int K) {
  constexpr int MM[3] = {2, 5, 4}, NU[3] = {2, 2, 4};
  const int tiles0 = E * (N / 128);
  const bool fills = avg <= 104.f && tiles0 > 384 && tiles0 <= 512;
  int best = 0;
  float least = 0.f;
  for (int f = 0; f < 3; ++f) {
    if (f == 2 && (N % 256 != 0 || avg <= 96.f || fills)) continue;
    float tiles = 0.f, work = 0.f, longest = 0.f;
    for (int z = -1; z <= 1; ++z) {
      const float units = ceilf(fmaxf(1.f, floorf(avg + 1.8f * z * sqrtf(avg))) / 64.f);
      const float mt = ceilf(units / MM[f]), mu = units / mt;
      auto step = [&](float m) { return 0.06f * m * NU[f] + 0.03f * (m + NU[f]) + (f == 0 ? 0.1f : 0.15f); };
      tiles += mt / 3.f;
      work += mt / 3.f * step(mu);
      longest = fmaxf(longest, step(ceilf(mu)));
    }
    const float rounds = tiles * E * (N / (64 * NU[f])) / 256.f;
    const float t = fmaxf(longest, (rounds < 4.f ? ceilf(rounds) : rounds + 0.5f) * work / tiles) * K;
    if (f == 0 || t < least) { best = f; least = t; }
  }
  return best;
}

}  // namespace

// Grouped expert GEMM over the device-side expert slices of eia_moe_align.
//   X [*, K] (ldx), rows gathered through row_idx (nullptr: identity); W [E][N][K] (expert
//   stride N*K); out [rows_total][ldo] in sorted order.
//   swiglu 1: N = 2I ([gate; up]), out has I columns; 0: out has N columns; 2: N columns with
//   a squared-ReLU epilogue (ungated experts' up projection).
//   max_rows: host upper bound of offs[E] (T * top_k) -- sizes the grid.
EIA_API int eia_moe_grouped_gemm(const void* X, long ldx, const int* row_idx, const void* W, int N,
                                 int K, int E, const int* offs, int max_rows, int swiglu, void* out,
                                 long ldo, hipStream_t st) {
  if (E < 1 || K % BK != 0 || (ldx % 8) || (ldo % 4) ||
      (reinterpret_cast<uintptr_t>(X) | reinterpret_cast<uintptr_t>(W)) % 16)
    return EIA_BAD_SHAPE;
  const int relu2 = swiglu == 2;
  if (relu2) swiglu = 0;
  if (swiglu ? (N % 2 != 0 || (N / 2) % 64 != 0) : (N % 128 != 0)) return EIA_BAD_SHAPE;
  if (max_rows <= 0) return EIA_OK;
  const int form = grouped_form((float)max_rows / E, E, N, K);
  // Up to 128 rows an expert, its weights take longer from memory than its products: the sooner a step asks, the
  // better, while beyond it holds the products up.  The op, spread / in front, us, cold weights: 8 experts of 4096 x
  // 14336, 64 rows 558 / 545; 16 of 2048 x 1024, 112 rows 70.6 / 69.8; 8 of 1024 x 512, 512 rows (form 0) 44.5 / 47.7.
  const bool front = max_rows <= 128L * E;
#define GG_GO(SW, NU, MM, OCC, FRONT)                                                               \
  do {                                                                                              \
    const int nt = N / (64 * NU);                                                                   \
    GroupedArgs a{(const bf16_t*)X, ldx, row_idx, (const bf16_t*)W, (long)N * K, offs, E, N / 2, K, \
                  nt, (bf16_t*)out, ldo, relu2};                                                    \
    const dim3 grid((unsigned)((((max_rows + 64 * MM - 1) / (64 * MM) + E) * (long)nt + 7) / 8 * 8)); \
    hipLaunchKernelGGL((moe_grouped_mfma_kernel<SW, NU, MM, OCC, FRONT>), grid, dim3(256), 0, st, a);      \
  } while (0)
#define GG_FORM(SW) \
  do {                                                                                              \
    if (form == 0 && front) GG_GO(SW, 2, 2, 2, true);                                               \
    else if (form == 0) GG_GO(SW, 2, 2, 2, false);                                                  \
    else if (form == 1) GG_GO(SW, 2, 5, 1, false);                                                  \
    else GG_GO(SW, 4, 4, 1, false);                                                                 \
  } while (0)
  if (swiglu) GG_FORM(true); else GG_FORM(false);
#undef GG_FORM
#undef GG_GO
  EIA_LAUNCH_CHECK();
}
