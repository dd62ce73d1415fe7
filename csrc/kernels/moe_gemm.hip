// K9 (prefill-sized MoE): grouped GEMM over device-side expert slices on v_mfma_f32_32x32x16_bf16.
//
//   out[p][:] = X[row(p)][:] . W_e^T          (p in expert e's slice [offs[e], offs[e+1]))
//   SwiGLU form: W_e = [gate; up] (2I rows), out[p][c] = silu(g_c) * u_c, I columns
//
// The expert slices come from eia_moe_align on the device, so nothing here is known to the
// host: the grid is an upper bound on the tiles ((ceil(rows / 128) + experts) M tiles), every
// workgroup maps blockIdx.x to (expert, M tile, N tile) by a wave-wide scan of the per-expert tile
// counts, and surplus workgroups exit.  No host synchronisation, no per-expert launches, and
// the same launch is valid inside a HIP graph.
//
// Tile 128 (M) x 128 (N) x 64 (K), 4 waves each owning 64 x 64 (2 x 2 MFMA tiles of 32 x 32).
// Operand roles are swapped (A = W rows, B = X^T) so a lane ends up with one output ROW and
// runs of 4 consecutive columns -> 8-B stores; in the SwiGLU form a wave's two N sub-tiles are
// the gate rows and the matching up rows, so silu(g) * u is formed in registers.
//
// Tiles go from memory straight to LDS (16 bytes per lane; X rows gathered through row_idx), 16 KB
// pieces in the order W0 X0 W1 X1 ... through a ring of five: two are multiplied while three are on
// their way, one K step ahead for X, which its N tiles find in L2, two for W.  Two workgroups fill the
// LDS of a CU.  Row r keeps its 16-byte chunk c at c ^ (r / 2 % 8): fragment reads of 16 rows meet all
// 64 banks.  An XCD takes a contiguous share of the tiles, ordered by expert, N tile, M tile, so that it reads
// the weights of its own experts only, and a weight tile once for all M tiles.
//
// Bound by the reads from L2 (1 MB per tile at K 2048; alone 47 us below, the products alone 46), which
// the products only partly cover, and by rounding up to whole tiles (640 on 512 places).  MI355X, 4096
// rows over 16 experts, K 2048, I 1024: 69 us, down projection (K 1024, N 2048) 39 us (staged through
// registers one step ahead, M tiles spread over the XCDs: 78 and 45); 16384 rows: 174 us.  Weights
// straight to registers 79 us (32-byte reads), 256-wide tiles 75 us (320 on 256 places).
#include "eia_common.h"

namespace {

typedef __attribute__((ext_vector_type(16))) float f32x16_t;

constexpr int BM = 128, BN = 128, BK = 64;
constexpr int PIECE = 128 * BK;                    // elements of one operand's K step
constexpr int RING = 5;
constexpr int GG_LDS_BYTES = RING * PIECE * 2;     // half of a CU's LDS

EIA_DEV float silu_f(float x) { return __fdividef(x, 1.f + __expf(-x)); }

template <bool SWIGLU>
__global__ void __launch_bounds__(256, 2)
moe_grouped_mfma_kernel(const bf16_t* __restrict__ X, long ldx, const int* __restrict__ row_idx,
                        const bf16_t* __restrict__ W, long w_estride, const int* __restrict__ offs,
                        int E, int I, int K, int NT, bf16_t* __restrict__ out, long ldo, int relu2) {
  extern __shared__ __align__(16) bf16_t lds[];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r32 = lane & 31, h = lane >> 5;

  // blockIdx.x -> tile -> (expert, N tile, first row of its M tile); every wave for itself
  int total = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int e = e0 + lane;
    int nt = e < E ? (offs[e + 1] - offs[e] + BM - 1) / BM : 0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) nt += __shfl_xor(nt, o, 64);
    total += nt;
  }
  total *= NT;
  const int share = (total + 7) / 8, at = blockIdx.x >> 3;
  const int tile = (blockIdx.x & 7) * share + at;
  if (at >= share || tile >= total) return;                // surplus workgroup (uniform)
  int ex = 0, n_tile = 0, m_tile = 0;
  for (int e0 = 0, base = 0; e0 < E; e0 += 64) {
    const int e = e0 + lane;
    const int nt = e < E ? (offs[e + 1] - offs[e] + BM - 1) / BM : 0;
    int incl = nt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(incl, o, 64);
      if (lane >= o) incl += v;
    }
    const int q = tile - (base + incl - nt) * NT;
    const unsigned long long hit = __ballot(q >= 0 && q < nt * NT);
    if (hit) {
      const int src = __ffsll(hit) - 1, qe = __shfl(q, src, 64), ne = __shfl(nt, src, 64);
      ex = e0 + src;
      n_tile = qe / ne;
      m_tile = qe - n_tile * ne;
      break;
    }
    base += __shfl(incl, 63, 64);
  }
  ex = __builtin_amdgcn_readfirstlane(ex);
  n_tile = __builtin_amdgcn_readfirstlane(n_tile);
  const int m0 = __builtin_amdgcn_readfirstlane(m_tile) * BM;
  const int rb = offs[ex], rows = offs[ex + 1] - rb;
  const bf16_t* We = W + (long)ex * w_estride;

  // a piece is 16 accesses of 1 KB (8 rows), four per wave: lane -> row lane / 8, LDS chunk lane % 8
  const bf16_t* xsrc[4];
  const bf16_t* wsrc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 32 * w + 8 * i + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    const int p = rb + min(m0 + r, rows - 1);              // rows past the slice clamp
    const long xr = row_idx != nullptr ? row_idx[p] : p;
    xsrc[i] = X + xr * ldx + 8 * c;
    int wr;
    if (SWIGLU) wr = r < 64 ? n_tile * 64 + r : I + n_tile * 64 + (r - 64);
    else wr = n_tile * BN + r;
    wsrc[i] = We + (long)wr * K + 8 * c;
  }
  const int nk = K / BK;
  auto fetch = [&](const bf16_t* const (&src)[4], int kt, int slot) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(src[i] + kt * BK),
          (__attribute__((address_space(3))) void*)(lds + slot * PIECE + (32 * w + 8 * i) * BK), 16, 0,
          0);
  };

  // wave (wm, wn): rows [64 wm, +64) of the X tile; W tile rows of N sub-tile nt:
  // plain 64 wn + 32 nt, SwiGLU 64 nt + 32 wn (nt 0 = gate, 1 = up, same output columns)
  const int wm = w & 1, wn = w >> 1;
  int wrow[2];
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) wrow[nt] = SWIGLU ? 64 * nt + 32 * wn : 64 * wn + 32 * nt;
  f32x16_t acc[2][2];                                      // [nt][mt]: C^T (rows n, cols m)
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;

  fetch(wsrc, 0, 0);
  fetch(xsrc, 0, 1);
  if (nk > 1) fetch(wsrc, 1, 2);
  int s0 = 0;                                              // slot of step kt's W
  const bool live = m0 + 64 * wm < rows;                   // this wave has output rows
  for (int kt = 0; kt < nk; ++kt) {
    // step kt is in LDS (W of step kt + 1 may not be), and step kt - 1 has been read
    if (kt + 1 < nk) asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();                          // (__syncthreads would wait for all pieces)
    asm volatile("" ::: "memory");
    const int s1 = s0 + 1 < RING ? s0 + 1 : 0, s3 = s0 + 3 < RING ? s0 + 3 : s0 + 3 - RING;
    const int s4 = s0 + 4 < RING ? s0 + 4 : s0 + 4 - RING;
    if (kt + 1 < nk) fetch(xsrc, kt + 1, s3);
    if (kt + 2 < nk) fetch(wsrc, kt + 2, s4);
    if (live) {
      const bf16_t* wl = lds + s0 * PIECE + r32 * BK;
      const bf16_t* xl = lds + s1 * PIECE + (64 * wm + r32) * BK;
      bf16x8 wf[2][2], xf[2][2];
      auto frags = [&](int kk) {
        const int c = 8 * ((2 * kk + h) ^ ((r32 >> 1) & 7));
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          wf[kk & 1][nt] = *reinterpret_cast<const bf16x8*>(wl + wrow[nt] * BK + c);
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
          xf[kk & 1][mt] = *reinterpret_cast<const bf16x8*>(xl + 32 * mt * BK + c);
      };
      frags(0);
#pragma unroll
      for (int kk = 0; kk < BK / 16; ++kk) {
        if (kk + 1 < BK / 16) frags(kk + 1);
        __builtin_amdgcn_sched_barrier(0);                 // the next fragments before these products
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
          for (int mt = 0; mt < 2; ++mt)
            acc[nt][mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[kk & 1][nt], xf[kk & 1][mt],
                                                                  acc[nt][mt], 0, 0, 0);
      }
    }
    s0 = s0 + 2 < RING ? s0 + 2 : s0 + 2 - RING;
  }

  // lane: output row m = 64 wm + 32 mt + r32; registers 4j..4j+3 = columns 8j + 4h + 0..3 of
  // the N sub-tile
#pragma unroll
  for (int mt = 0; mt < 2; ++mt) {
    const int m = m0 + 64 * wm + 32 * mt + r32;
    if (m >= rows) continue;
    bf16_t* op = out + (long)(rb + m) * ldo;
    if (SWIGLU) {
      const int c0 = n_tile * 64 + 32 * wn;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        bf16x4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          v[r] = f2bf(silu_f(acc[0][mt][4 * j + r]) * acc[1][mt][4 * j + r]);
        *reinterpret_cast<bf16x4*>(op + c0 + 8 * j + 4 * h) = v;
      }
    } else {
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        const int c0 = n_tile * BN + wrow[nt];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          bf16x4 v;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float x = acc[nt][mt][4 * j + r];
            if (relu2) { x = fmaxf(x, 0.f); x *= x; }     // ungated experts: squared ReLU
            v[r] = f2bf(x);
          }
          *reinterpret_cast<bf16x4*>(op + c0 + 8 * j + 4 * h) = v;
        }
      }
    }
  }
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
  if (swiglu ? (N % 2 != 0 || (N / 2) % 64 != 0) : (N % BN != 0)) return EIA_BAD_SHAPE;
  if (max_rows <= 0) return EIA_OK;
  const int nt = N / BN;
  const dim3 grid((unsigned)((((max_rows + BM - 1) / BM + E) * (long)nt + 7) / 8 * 8));
#define GG_GO(SW)                                                                                   \
  do {                                                                                              \
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(moe_grouped_mfma_kernel<SW>),           \
                              hipFuncAttributeMaxDynamicSharedMemorySize, GG_LDS_BYTES);            \
    hipLaunchKernelGGL(moe_grouped_mfma_kernel<SW>, grid, dim3(256), GG_LDS_BYTES, st,              \
                       (const bf16_t*)X, ldx, row_idx, (const bf16_t*)W, (long)N * K, offs, E,      \
                       N / 2, K, nt, (bf16_t*)out, ldo, relu2);                                     \
  } while (0)
  if (swiglu) GG_GO(true); else GG_GO(false);
#undef GG_GO
  EIA_LAUNCH_CHECK();
}
