// Latent (low-rank KV) attention over a paged latent cache.
//
// Cache row of one token: [ c (kv_rank, RMS-normed latent) | k_rot (rot_dim, rotated key part
// shared by all heads) ].  With the key up-projection absorbed into the query,
//   q_abs[h] = W_uk[h]^T q_nope[h]                       (a batched GEMM, done by the caller)
//   score[h][j] = (q_abs[h] . c_j + rot(q_rot[h]) . k_rot_j) * scale
//   lat[h] = sum_j softmax(score[h])_j c_j                (value up-projection by the caller)
// every head reads the SAME cache rows, so a workgroup stages a key tile in LDS once and uses it
// for all (query, head) rows it owns.  Options: a sliding window (position i sees j with
// 0 <= i - j < window), a per-head sink (the softmax denominator also holds exp(sink[h]), which
// has no key and no value and is not scaled), and the pair layout of the rotation ((2i, 2i+1) or
// (i, i + rot_dims/2)) with a common factor on cos and sin.  Scores, softmax weights and the
// accumulators are fp32; activations are bf16 or fp32 (template T).
//
//   eia_latent_prep : RMS-norm of the query latent, RMS-norm of c, rotation of k_rot, cache write
//   eia_latent_attn : rotation of q_rot, tiled online-softmax attention, sigmoid head gate
#include "eia_flash.h"

// Entry d (< rot_dims) of a vector after the rotation by position pos: src holds the unrotated
// vector; pairs are (2i, 2i+1), or (i, i + rot_dims/2) when half; cos and sin are times amp.
template <typename T>
EIA_DEV float lat_rotated(const T* src, int d, int rot_dims, bool half, float amp, float pos,
                          const float* __restrict__ inv_freq) {
  const int hd = rot_dims >> 1;
  const int i = half ? (d < hd ? d : d - hd) : (d >> 1);
  const bool second = half ? d >= hd : (d & 1);
  float sn, cs;
  sincosf(pos * inv_freq[i], &sn, &cs);
  sn *= amp;
  cs *= amp;
  const float u = ld_f32<T>(src, half ? i : 2 * i), w = ld_f32<T>(src, half ? i + hd : 2 * i + 1);
  return second ? (w * cs + u * sn) : (u * cs - w * sn);
}

// ------------------------------------------------------------------------------------------ prep
// fused [T, ld]: columns [q_off, q_off+q_rank) query latent, [c_off, c_off+R) KV latent,
// [kr_off, kr_off+rd) shared rotary key part.  q_rank == 0: no query latent; cache == nullptr:
// no KV part (a layer that reads another layer's cache).
template <typename T>
__global__ void __launch_bounds__(128)
latent_prep_kernel(const T* __restrict__ fused, long ld, int q_off, int q_rank,
                   const T* __restrict__ wq, T* __restrict__ cq, long ldcq, int c_off, int R,
                   const T* __restrict__ wc, int kr_off, int rd, int rot_dims,
                   const float* __restrict__ inv_freq, const int* __restrict__ positions,
                   const int* __restrict__ slot_mapping, T* __restrict__ cache, long cache_row,
                   float eps, int rot_half, float rot_amp) {
  __shared__ float scratch[2];
  const long t = blockIdx.x;
  const T* row = fused + t * ld;
  if (q_rank > 0) {
    float ss = 0.f;
    for (int c = threadIdx.x; c < q_rank; c += blockDim.x) {
      const float v = ld_f32<T>(row, q_off + c);
      ss += v * v;
    }
    const float inv = 1.0f / sqrtf(block_sum(ss, scratch) / (float)q_rank + eps);
    for (int c = threadIdx.x; c < q_rank; c += blockDim.x)
      st_f32<T>(cq + t * ldcq, c, ld_f32<T>(row, q_off + c) * inv * ld_f32<T>(wq, c));
  }
  if (cache == nullptr) return;
  const int slot = slot_mapping[t];
  if (slot < 0) return;                       // uniform per workgroup
  T* dst = cache + (long)slot * cache_row;
  float ss = 0.f;
  for (int c = threadIdx.x; c < R; c += blockDim.x) {
    const float v = ld_f32<T>(row, c_off + c);
    ss += v * v;
  }
  const float inv = 1.0f / sqrtf(block_sum(ss, scratch) / (float)R + eps);
  for (int c = threadIdx.x; c < R; c += blockDim.x)
    st_f32<T>(dst, c, ld_f32<T>(row, c_off + c) * inv * ld_f32<T>(wc, c));
  const float pos = (float)positions[t];
  for (int d = threadIdx.x; d < rd; d += blockDim.x) {
    const float v = d < rot_dims
        ? lat_rotated<T>(row + kr_off, d, rot_dims, rot_half != 0, rot_amp, pos, inv_freq)
        : ld_f32<T>(row, kr_off + d);
    st_f32<T>(dst, R + d, v);
  }
}

EIA_API int eia_latent_prep(const void* fused, long ld, int q_off, int q_rank, const void* wq,
                            void* cq, long ldcq, int c_off, int R, const void* wc, int kr_off,
                            int rd, int rot_dims, const float* inv_freq, const int* positions,
                            const int* slot_mapping, void* cache, long cache_row, float eps,
                            int rot_half, float rot_amp, int T_, int is_bf16, hipStream_t st) {
  if (T_ < 0 || q_rank < 0 || (cache && (R < 1 || rd < 0 || rot_dims > rd || (rot_dims & 1))))
    return EIA_BAD_SHAPE;
  if (T_ == 0) return EIA_OK;
  if (is_bf16)
    hipLaunchKernelGGL((latent_prep_kernel<bf16_t>), dim3(T_), dim3(128), 0, st,
                       (const bf16_t*)fused, ld, q_off, q_rank, (const bf16_t*)wq, (bf16_t*)cq,
                       ldcq, c_off, R, (const bf16_t*)wc, kr_off, rd, rot_dims, inv_freq, positions,
                       slot_mapping, (bf16_t*)cache, cache_row, eps, rot_half, rot_amp);
  else
    hipLaunchKernelGGL((latent_prep_kernel<float>), dim3(T_), dim3(128), 0, st,
                       (const float*)fused, ld, q_off, q_rank, (const float*)wq, (float*)cq, ldcq,
                       c_off, R, (const float*)wc, kr_off, rd, rot_dims, inv_freq, positions,
                       slot_mapping, (float*)cache, cache_row, eps, rot_half, rot_amp);
  EIA_LAUNCH_CHECK();
}

// ------------------------------------------------------------------------------------- attention
constexpr int LAT_UNIT = 64;       // keys per tile of the decode form, cut at multiples of it

// Tiles of a decode row, and of each of the key partitions that it uses out of the launch's: the fewest that leave the
// longest one as short; where a tile takes less than its partition's place in the merge (R up to 256), two tiles each beyond
// 32 partitions (eight rows at 4000 tokens, 256 + 32: 15.7 us in 63, 14.8 in 32).
struct LatTiles { int n, per; };
EIA_DEV LatTiles lat_tiles(int nparts, int kmin, int kmax, int R) {
  const int n = (kmax - kmin + LAT_UNIT - 1) / LAT_UNIT;
  const int most = R <= 256 && n < 2 * nparts ? min(nparts, 32) : nparts;
  return {n, (n + most - 1) / most};
}

#define LAT_ACC_MAX 32     // fp32 accumulators per thread: QB * HB * R <= 256 * LAT_ACC_MAX

struct LatentAttnArgs {
  const void* qa; long qa_st, qa_sh;        // absorbed queries (t, h, r)
  const void* qr; long qr_st, qr_sh;        // rotary query part, not yet rotated (t, h, d)
  const float* inv_freq; int rot_dims;
  const void* cache; long cache_row;        // rows of R + rd
  const int* block_table; int bt_stride;
  const int* seq_lens;                      // nullable: rows with 0 are padding
  const int* cu_q;                          // nullable: one query per sequence (decode)
  const int* work; int n_work;              // nullable with cu_q == nullptr: item = sequence
  const int* positions;                     // per query row
  const void* gate; long gate_st;           // nullable: sigmoid(gate[t][h]) scales head h
  void* out; long out_st, out_sh;           // (t, h, r)
  float scale; int H, R, rd, bs, QB, HB, KC, ldk;
  int window;                               // > 0: position i sees j with 0 <= i - j < window
  const float* sink;                        // nullable [H]: exp(sink[h]) joins the denominator
  int rot_half; float rot_amp;              // pair layout and cos / sin factor of the rotation
  // MFMA decode only: the keys of a row split over grid.z partitions; each writes its
  // unnormalised accumulators and (running max in log2 units, sum) for the merge kernel
  int nparts; float* part_acc; float* part_ml;
};

template <typename T>
__global__ void __launch_bounds__(256)
latent_attn_kernel(LatentAttnArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int Dk = a.R + a.rd, M = a.QB * a.HB, KC = a.KC, ldk = a.ldk;
  float* qs = reinterpret_cast<float*>(smem);            // [M][Dk]
  float* ps = qs + (long)M * Dk;                         // [M][KC]
  float* mrow = ps + (long)M * KC;                       // [M]
  float* lrow = mrow + M;                                // [M]
  float* arow = lrow + M;                                // [M]
  T* kt = reinterpret_cast<T*>(arow + M);                // [KC][ldk]

  int seq, row0, ntok;
  if (a.cu_q) {
    seq = a.work[2 * blockIdx.x];
    const int q0 = a.work[2 * blockIdx.x + 1];
    const int lo = a.cu_q[seq], hi = a.cu_q[seq + 1];
    row0 = lo + q0;
    ntok = min(a.QB, hi - row0);
  } else {
    seq = blockIdx.x;
    row0 = seq;
    ntok = 1;
  }
  if (ntok <= 0 || (a.seq_lens && a.seq_lens[seq] <= 0)) return;
  const int h0 = blockIdx.y * a.HB;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const T* qa = static_cast<const T*>(a.qa);
  const T* qr = static_cast<const T*>(a.qr);
  const T* cache = static_cast<const T*>(a.cache);
  const int* bt = a.block_table + (long)seq * a.bt_stride;

  // queries -> LDS (rotated, pre-scaled); rows of absent tokens / heads are zero
  for (int e = tid; e < M * Dk; e += 256) {
    const int m = e / Dk, d = e - m * Dk;
    const int t = m / a.HB, h = h0 + (m - t * a.HB);
    float v = 0.f;
    if (t < ntok && h < a.H) {
      const long row = row0 + t;
      if (d < a.R) {
        v = ld_f32<T>(qa, row * a.qa_st + h * a.qa_sh + d);
      } else {
        const int dd = d - a.R;
        const T* src = qr + row * a.qr_st + h * a.qr_sh;
        v = dd < a.rot_dims
            ? lat_rotated<T>(src, dd, a.rot_dims, a.rot_half != 0, a.rot_amp,
                             (float)a.positions[row], a.inv_freq)
            : ld_f32<T>(src, dd);
      }
      v *= a.scale;
    }
    qs[e] = v;
  }
  for (int m = tid; m < M; m += 256) {
    mrow[m] = -INFINITY;
    lrow[m] = 0.f;
    arow[m] = 1.f;
  }
  float acc[LAT_ACC_MAX];
#pragma unroll
  for (int i = 0; i < LAT_ACC_MAX; ++i) acc[i] = 0.f;
  const int nacc = (M * a.R + 255) >> 8;
  const int kmax = a.positions[row0 + ntok - 1] + 1;     // keys kmin..kmax-1 are visible to the tile
  const int kmin = a.window > 0 ? max(0, a.positions[row0] - a.window + 1) : 0;
  __syncthreads();

  for (int k0 = kmin; k0 < kmax; k0 += KC) {
    // key tile -> LDS
    for (int e = tid; e < KC * Dk; e += 256) {
      const int j = e / Dk, d = e - j * Dk;
      const int kp = k0 + j;
      T v = (T)0.f;
      if (kp < kmax) {
        const long slot = (long)bt[kp / a.bs] * a.bs + (kp % a.bs);
        v = cache[slot * a.cache_row + d];
      }
      kt[j * ldk + d] = v;
    }
    __syncthreads();
    // scores: consecutive lanes take consecutive keys of one query row
    for (int e = tid; e < M * KC; e += 256) {
      const int m = e / KC, j = e - m * KC;
      const int t = m / a.HB;
      const int kp = k0 + j;
      float s = -INFINITY;
      if (t < ntok && kp <= a.positions[row0 + t] &&
          (a.window <= 0 || a.positions[row0 + t] - kp < a.window)) {
        const float* q = qs + (long)m * Dk;
        const T* k = kt + (long)j * ldk;
        s = 0.f;
        for (int d = 0; d < Dk; ++d) s += q[d] * ld_f32<T>(k, d);
      }
      ps[e] = s;
    }
    __syncthreads();
    // online softmax per row: one wave per row, lanes over the tile's keys
    for (int m = wave; m < M; m += 4) {
      float tmax = -INFINITY;
      for (int j = lane; j < KC; j += 64) tmax = fmaxf(tmax, ps[m * KC + j]);
      tmax = wave_max(tmax);
      const float mold = mrow[m];
      const float mnew = fmaxf(mold, tmax);
      float psum = 0.f;
      for (int j = lane; j < KC; j += 64) {
        const float s = ps[m * KC + j];
        const float p = (s == -INFINITY) ? 0.f : expf(s - mnew);
        ps[m * KC + j] = p;
        psum += p;
      }
      psum = wave_sum(psum);
      if (lane == 0) {
        const float al = (mold == -INFINITY) ? ((mnew == -INFINITY) ? 1.f : 0.f) : expf(mold - mnew);
        arow[m] = al;
        lrow[m] = lrow[m] * al + psum;
        mrow[m] = mnew;
      }
    }
    __syncthreads();
    // accumulate the latent part of the keys
#pragma unroll
    for (int i = 0; i < LAT_ACC_MAX; ++i) {
      if (i < nacc) {
        const int e = tid + (i << 8);
        const int m = e / a.R, r = e - m * a.R;
        if (m < M) {
          float v = acc[i] * arow[m];
          const float* p = ps + (long)m * KC;
          for (int j = 0; j < KC; ++j) v += p[j] * ld_f32<T>(kt, (long)j * ldk + r);
          acc[i] = v;
        }
      }
    }
    __syncthreads();
  }

  T* out = static_cast<T*>(a.out);
  const T* gate = static_cast<const T*>(a.gate);
#pragma unroll
  for (int i = 0; i < LAT_ACC_MAX; ++i) {
    if (i < nacc) {
      const int e = tid + (i << 8);
      const int m = e / a.R, r = e - m * a.R;
      if (m < M) {
        const int t = m / a.HB, h = h0 + (m - t * a.HB);
        if (t < ntok && h < a.H) {
          const long row = row0 + t;
          float l = lrow[m];
          if (a.sink) l += expf(a.sink[h] - mrow[m]);
          float v = acc[i] / l;
          if (gate) v *= 1.0f / (1.0f + expf(-ld_f32<T>(gate, row * a.gate_st + h)));
          st_f32<T>(out, row * a.out_st + h * a.out_sh + r, v);
        }
      }
    }
  }
}

// n_items: sequences (cu_q == nullptr, one query row per sequence) or work items (seq, first
// query) of QB queries each.  Heads are processed HB at a time (grid.y).
EIA_API int eia_latent_attn(const void* qa, long qa_st, long qa_sh, const void* qr, long qr_st,
                            long qr_sh, const float* inv_freq, int rot_dims, const void* cache,
                            long cache_row, const int* block_table, int bt_stride,
                            const int* seq_lens, const int* cu_q, const int* work, int n_items,
                            const int* positions, const void* gate, long gate_st, void* out,
                            long out_st, long out_sh, float scale, int H, int R, int rd, int bs,
                            int QB, int window, const float* sink, int rot_half, float rot_amp,
                            int is_bf16, hipStream_t st) {
  if (H < 1 || R < 1 || rd < 0 || bs < 1 || QB < 1 || rot_dims > rd || (rot_dims & 1) ||
      cache_row < R + rd || (cu_q && !work))
    return EIA_BAD_SHAPE;
  if (n_items <= 0) return EIA_OK;
  int HB = H < 16 ? H : 16;
  while (HB > 1 && (long)QB * HB * R > 256L * LAT_ACC_MAX) HB = (HB + 1) / 2;
  if ((long)QB * HB * R > 256L * LAT_ACC_MAX) return EIA_UNSUPPORTED;
  const int Dk = R + rd, M = QB * HB;
  const int esz = is_bf16 ? 2 : 4;
  // key-tile row stride: an odd number of 32-bit words, so lanes reading one column of
  // consecutive rows hit distinct LDS banks
  int ldk = Dk;
  if (is_bf16) { ldk += ldk & 1; if (((ldk / 2) & 1) == 0) ldk += 2; }
  else if ((ldk & 1) == 0) ldk += 1;
  int KC = 64;
  size_t lds = 0;
  for (;; KC >>= 1) {
    lds = ((size_t)M * Dk + (size_t)M * KC + 3 * (size_t)M) * 4 + (size_t)KC * ldk * esz;
    if (lds <= 96 * 1024 || KC == 8) break;
  }
  if (lds > 150 * 1024) return EIA_UNSUPPORTED;
  LatentAttnArgs a{qa, qa_st, qa_sh, qr, qr_st, qr_sh, inv_freq, rot_dims, cache, cache_row,
                   block_table, bt_stride, seq_lens, cu_q, work, n_items, positions, gate, gate_st,
                   out, out_st, out_sh, scale, H, R, rd, bs, QB, HB, KC, ldk, window, sink, rot_half,
                   rot_amp, 1, nullptr, nullptr};
  dim3 grid(n_items, (H + HB - 1) / HB);
  if (is_bf16) {
    if (lds > 48 * 1024)
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&latent_attn_kernel<bf16_t>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL((latent_attn_kernel<bf16_t>), grid, dim3(256), lds, st, a);
  } else {
    if (lds > 48 * 1024)
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&latent_attn_kernel<float>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL((latent_attn_kernel<float>), grid, dim3(256), lds, st, a);
  }
  EIA_LAUNCH_CHECK();
}

// ------------------------------------------------------------------------- decode rows, MFMA (bf16)
// One workgroup of NW waves per (decode row, 16 heads, key partition), v_mfma_f32_16x16x32_bf16.
// 64 cache rows at a time are staged in LDS as they are; wave w forms the scores of keys 16 (w % 4) .. + 15
// (S^T: keys x heads), with eight waves over half of the entries each, the waves exchange them through LDS, every wave
// forms the softmax weights of all 64 keys and takes its share of the latent columns in O^T += C^T P^T, whose operand
// comes from the same rows through the transposing LDS read.  Rows that leave a CU to one workgroup (R + rd > 288) take
// eight waves: half of a tile's chain for each (48 rows of 16 heads, 512 + 64, below: 27.6 -> 25.9 us with the merge, 13 rows
// 19.0 -> 16.3, 100 rows at 2500 tokens, no window 79.3 -> 75.6, 30 rows of 64 heads at 4000 109 -> 103).  Weights stay fp32: a bf16 high part plus a bf16
// remainder (two products), and the normaliser sums the fp32 weights.  The next rows are in flight
// during the products, the first ones during the rotation of the queries.
//
// Bound by latency: a row's 64-key tiles are a chain of cache loads and two barriers, and the launch
// lasts as long as the longest partition.  MI355X, 48 rows at up to 4096 tokens, window 1024, 16
// heads, R 512 + 64: 19.8 + 4.0 us in five partitions, 6 of them before the first tile is there and 2.6 a tile (pages read beside
// the position, not behind it: 25.9 -> 25.8; queries and angles asked for before the first rows, not behind them and two
// barriers: 24.5 -> 23.9); 200 rows at up to 2500 tokens, no window, with
// 16 heads 153 -> 134 us and with 64 heads 499 -> 437 us since a tile's page is known before its fetch and
// its LDS reads are asked for before the first product; R 128 + 32 with 64 heads 120 -> 115 us, R 256 + 64
// 292 -> 292 us.  (Two tiles of cache loads in flight, in registers: 27 us instead of 24; the reads held in
// front by barriers to the scheduler and two chains of products: 25 us.  32-key units that went through LDS
// twice, the second time as transposed 2-byte stores, with the scores formed by every wave and sixteen
// partitions: 91 + 21 us.)
constexpr int lat_bufs(int NK) { return NK <= 18 ? 2 : 1; }       // tiles that fit 160 KB of LDS

// NK: 32-entry steps of a cache row; NCW: column tiles of a wave; NW: waves, four or eight.
template <int NK, int NCW, int NW>
__global__ void __launch_bounds__(64 * NW)
latent_decode_kernel(LatentAttnArgs a) {
  constexpr int NB = lat_bufs(NK), KT = LAT_UNIT;
  constexpr int KS = 32 * NK + 8;                       // 4 NK + 1 units of 16 bytes per row
  constexpr int SP = KT + 4;                            // pitch of the exchanged scores
  constexpr int NT = 64 * NW, NH = NW / 4, NS = NK / NH, NU = KT * 4 * NK / NT;    // steps of a wave; 16-byte units of a thread
  static_assert(NK % NH == 0 && KT * 4 * NK % NT == 0, "whole shares");
  // (static: more than 64 KB of dynamic LDS takes a call to the runtime for each launch)
  __shared__ __align__(16) bf16_t tiles[NB * KT * KS];
  __shared__ __align__(16) float sS[NH * 16 * SP];      // the exchanged scores
  __shared__ float2 rot[16 * NK];                       // [rot_dims / 2], rot_dims <= 32 NK
  int row = blockIdx.x, z = blockIdx.z;
  if (row >= a.n_work) {                                // beside the rows: the partitions that their own places do not hold
    const int others = a.nparts - gridDim.z, at = row - a.n_work + (gridDim.x - a.n_work) * z;
    if (others <= 0) return;
    row = at / others;
    z = gridDim.z + at - row * others;
  }
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int l16 = lane & 15, g4 = lane >> 4;
  if (row >= a.n_work || (a.seq_lens && a.seq_lens[row] <= 0)) return;
  const int qpos = a.positions[row], kmax = qpos + 1;
  const int wlo = a.window > 0 ? max(0, kmax - a.window) : 0, kmin = wlo & ~(KT - 1);
  const LatTiles tl = lat_tiles(a.nparts, kmin, kmax, a.R);
  if (z * tl.per >= tl.n) return;                       // (whole workgroup)
  const int k_begin = kmin + z * tl.per * KT, k_end = min(kmax, k_begin + tl.per * KT);
  const int R = a.R, Dk = R + a.rd, bs = a.bs, h0 = blockIdx.y * a.HB, nh = min(a.HB, a.H - h0);
  const bf16_t* cache = static_cast<const bf16_t*>(a.cache);
  const int* bt = a.block_table + (long)row * a.bt_stride;
  const bool paged = bs % KT == 0;                      // a tile lies in one page
  const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  bf16x8 kst[NU];
  // the page of a tile is looked up a tile ahead of its fetch: the fetch would wait for it
  int off = 0, at = 0, page = 0;                        // the next fetch: token in its page, page's place, page
  auto look = [&](int k0) {
    if (!paged || k0 >= k_end) return;
    if (k0 == k_begin) {
      at = k0 / bs;
      off = k0 - at * bs;
    } else {
      off += KT;
      if (off == bs) off = 0, ++at;
    }
    page = bt[at];
  };
  // (nothing may look at the values before stash)
  auto fetch = [&](int k0) {
    const long base = paged ? (long)__builtin_amdgcn_readfirstlane(page) * bs + off : 0;
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = tid + NT * i, j = u / (4 * NK), d = 8 * (u % (4 * NK));
      const int kp = min(k0 + j, kmax - 1);
      const long slot = paged ? base + j : (long)bt[kp / bs] * bs + kp % bs;
      kst[i] = *reinterpret_cast<const bf16x8*>(cache + slot * a.cache_row + (d < Dk ? d : 0));
    }
  };
  auto stash = [&](int buf, int k0) {       // (slots behind the last key may hold anything: 0 x inf)
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = tid + NT * i, j = u / (4 * NK), d = 8 * (u % (4 * NK));
      *reinterpret_cast<bf16x8*>(tiles + (buf * KT + j) * KS + d) = d < Dk && k0 + j < k_end ? kst[i] : zero8;
    }
  };
  look(k_begin);
  // What the queries are formed from is asked for before the first rows, of whose arrival nothing then waits, where a
  // workgroup has a CU to itself.  Others wait less for their rows than they lose to the longer start: 57 rows of 64
  // heads, 256 + 32, window 1024 31.5 -> 32.6 us, of 32 heads, 128 + 32 17.6 -> 19.1.
  constexpr bool AHEAD = NW == 8;
  const int hp = a.rot_dims >> 1, npass = a.rd - a.rot_dims;
  const bf16_t* qrb = static_cast<const bf16_t*>(a.qr) + (long)row * a.qr_st + (long)h0 * a.qr_sh;
  auto pair = [&](int e, int& m, int& ia, int& ib) {    // pair e of the rotary parts: head, places
    m = e / hp;
    const int i = e - m * hp;
    ia = a.rot_half ? i : 2 * i;
    ib = a.rot_half ? i + hp : 2 * i + 1;
    return i;
  };
  float turn = 0.f;
  unsigned pu = 0, pv = 0;                              // (as they lie in memory: a conversion here would wait for them)
  if constexpr (AHEAD) {
    turn = tid < hp ? a.inv_freq[tid] : 0.f;
    if (tid < nh * hp) {
      int m, ia, ib;
      pair(tid, m, ia, ib);
      const unsigned short* src = reinterpret_cast<const unsigned short*>(qrb) + (long)m * a.qr_sh;
      pu = src[ia];
      pv = src[ib];
    }
  }
  const bool ok = l16 < nh;                             // this lane's head
  const int h = h0 + (ok ? l16 : 0);
  const int kg = w & 3, s0 = NS * (w >> 2);             // the wave's keys of a tile, and steps of their rows
  bf16x8 qf[NS];
  // R % 8 == 0 and rd % 8 == 0: a lane's eight entries lie wholly in one of the two parts
  const bf16_t* qa = static_cast<const bf16_t*>(a.qa) + (long)row * a.qa_st + (long)h * a.qa_sh;
  const bool vec = ((reinterpret_cast<uintptr_t>(a.qa) | (uintptr_t)(a.qa_st * 2) | (uintptr_t)(a.qa_sh * 2)) & 15) == 0;
  auto query = [&](int d) {
    if (vec) return *reinterpret_cast<const bf16x8*>(qa + d);
    bf16x8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = qa[d + e];
    return v;
  };
  if constexpr (AHEAD) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int d = 32 * (s0 + s) + 8 * g4;
      qf[s] = query(d < R ? d : 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  fetch(k_begin);
  look(k_begin + KT);

  // the rotary query parts, rotated once into LDS: the heads of a row turn by the same angles
  for (int i = tid; i < hp; i += NT) {
    float sn, cs;
    sincosf((float)qpos * (AHEAD && i == tid ? turn : a.inv_freq[i]), &sn, &cs);
    rot[i] = make_float2(cs * a.rot_amp, sn * a.rot_amp);
  }
  __syncthreads();
  bf16_t* qrs = tiles;                                  // [16][rd]
  if constexpr (AHEAD) asm volatile("" : "+v"(pu), "+v"(pv));
  for (int e = tid; e < nh * hp; e += NT) {
    int m, ia, ib;
    const int i = pair(e, m, ia, ib);
    const bf16_t* src = qrb + (long)m * a.qr_sh;
    const float u = AHEAD && e == tid ? __uint_as_float(pu << 16) : bf2f(src[ia]);
    const float v = AHEAD && e == tid ? __uint_as_float(pv << 16) : bf2f(src[ib]);
    const float2 cs = rot[i];
    qrs[m * a.rd + ia] = f2bf(u * cs.x - v * cs.y);
    qrs[m * a.rd + ib] = f2bf(v * cs.x + u * cs.y);
  }
  for (int e = tid; e < nh * npass; e += NT) {         // entries past rot_dims pass unchanged
    const int m = e / npass, d = a.rot_dims + e - m * npass;
    qrs[m * a.rd + d] = qrb[(long)m * a.qr_sh + d];
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int d = 32 * (s0 + s) + 8 * g4;
    if constexpr (AHEAD) {
      if (!ok || d >= Dk) qf[s] = zero8;
      else if (d >= R) qf[s] = *reinterpret_cast<const bf16x8*>(qrs + l16 * a.rd + (d - R));
    } else {
      bf16x8 v = zero8;
      if (ok && d < Dk) {
        v = d >= R ? *reinterpret_cast<const bf16x8*>(qrs + l16 * a.rd + (d - R)) : query(d);
      }
      qf[s] = v;
    }
  }
  __syncthreads();                                      // the rotary parts make room for tiles
  stash(0, k_begin);
  f32x4 acc[NCW];
#pragma unroll
  for (int i = 0; i < NCW; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float mrun = -INFINITY, lrun = 0.f;
  const float scale_log2 = a.scale * 1.4426950408889634f;
  // transposing read: lane l of sixteen addresses row l / 4, entries 4 (l % 4), and receives column l
  const int c0 = 16 * NCW * w, vrow = 8 * g4 + (l16 >> 2), vcol = c0 + 4 * (l16 & 3);
  for (int k0 = k_begin, buf = 0; k0 < k_end; k0 += KT, buf ^= NB - 1) {
    const bf16_t* t = tiles + buf * KT * KS;
    __syncthreads();
    if (k0 + KT < k_end) {
      fetch(k0 + KT);
      look(k0 + 2 * KT);
    }
    f32x4 sc = {0.f, 0.f, 0.f, 0.f};
    bf16x8 kf[NS];                                      // (all asked for before the first product)
#pragma unroll
    for (int s = 0; s < NS; ++s) kf[s] = *reinterpret_cast<const bf16x8*>(t + (16 * kg + l16) * KS + 32 * (s0 + s) + 8 * g4);
#pragma unroll
    for (int s = 0; s < NS; ++s) sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[s], qf[s], sc, 0, 0, 0);
    *reinterpret_cast<f32x4*>(sS + (16 * (w >> 2) + l16) * SP + 16 * kg + 4 * g4) = sc * scale_log2;
    __syncthreads();
    // head l16, keys 32 x + 8 g4 + e
    float v[2][8];
    float mloc = -INFINITY;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int e = 0; e < 8; e += 4) {
        f32x4 q = *reinterpret_cast<const f32x4*>(sS + l16 * SP + 32 * x + 8 * g4 + e);
        if constexpr (NH == 2) q += *reinterpret_cast<const f32x4*>(sS + (16 + l16) * SP + 32 * x + 8 * g4 + e);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = k0 + 32 * x + 8 * g4 + e + i;
          v[x][e + i] = key >= wlo && key < k_end ? q[i] : -INFINITY;
          mloc = fmaxf(mloc, v[x][e + i]);
        }
      }
    mloc = column_max(mloc);
    const float mnew = fmaxf(mrun, mloc), muse = mnew == -INFINITY ? 0.f : mnew;
    const float alpha = exp2f(mrun - muse);             // mrun = -inf: 0 (nothing summed yet)
    bf16x8 ph[2], pl[2];
    float psum = 0.f;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const float p0 = exp2f(v[x][e] - muse), p1 = exp2f(v[x][e + 1] - muse);
        psum += p0 + p1;
        flash_split(p0, p1, e, ph[x], pl[x]);
      }
    psum = column_sum(psum);
    lrun = lrun * alpha + psum;
    mrun = mnew;
#pragma unroll
    for (int i = 0; i < NCW; ++i) acc[i] *= alpha;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int i = 0; i < NCW; ++i) {
        const bf16_t* p = t + (32 * x + vrow) * KS + vcol + 16 * i;
        const bf16x8 vf = lds_columns(p, p + 4 * KS);
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, ph[x], acc[i], 0, 0, 0);
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pl[x], acc[i], 0, 0, 0);
      }
    if (k0 + KT < k_end) {
      if (NB == 1) __syncthreads();                     // the tile was read
      stash(buf ^ (NB - 1), k0 + KT);
    }
  }
  if (!ok) return;
  // the lane holds columns c0 + 16 i + 4 g4 .. + 3 of its head (R % 8 == 0)
  if (tl.per < tl.n) {
    const long pr = ((long)row * a.H + h) * a.nparts + z;
#pragma unroll
    for (int i = 0; i < NCW; ++i) {
      const int c = c0 + 16 * i + 4 * g4;
      if (c < R) *reinterpret_cast<f32x4*>(a.part_acc + pr * R + c) = acc[i];
    }
    if (g4 == 0 && w == 0) {
      a.part_ml[2 * pr] = mrun;
      a.part_ml[2 * pr + 1] = lrun;
    }
    return;
  }
  if (a.sink) lrun += exp2f(a.sink[h] * 1.4426950408889634f - mrun);
  float f = 1.0f / lrun;
  if (a.gate) f *= 1.0f / (1.0f + expf(-bf2f(static_cast<const bf16_t*>(a.gate)[row * a.gate_st + h])));
  bf16_t* out = static_cast<bf16_t*>(a.out) + row * a.out_st + (long)h * a.out_sh;
#pragma unroll
  for (int i = 0; i < NCW; ++i) {
    const int c = c0 + 16 * i + 4 * g4;
    if (c >= R) continue;
    bf16x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = f2bf(acc[i][e] * f);
    *reinterpret_cast<bf16x4*>(out + c) = o;
  }
}

// Merge of the decode partitions: out = sum_p acc_p 2^(m_p - M) / sum_p l_p 2^(m_p - M), times
// the head gate.  One workgroup per (row, head); lane p first turns partition p's (max, sum) into
// its weight, then the threads sum four latent columns each over the partitions (nparts <= 64).
// Rows whose context is too short for two partitions were finished by the
// attention kernel itself.  Bound by latency: the partials of up to eight partitions are asked for together with the
// weights' inputs (48 rows of 16 heads, R 512, five partitions: 4.8 -> 4.0 us), sixteen at a time where there are many more
// (four at a time: 4000 tokens, 16 heads, one row in 63 partitions, both launches: 28.7 us instead of 19.3).
constexpr int LM_P = 8;
__global__ void __launch_bounds__(128)
latent_merge_kernel(const float* __restrict__ part_acc, const float* __restrict__ part_ml,
                    int nparts, const int* __restrict__ seq_lens, const int* __restrict__ positions,
                    int window, const bf16_t* __restrict__ gate, long gate_st,
                    const float* __restrict__ sink, bf16_t* __restrict__ out, long out_st,
                    long out_sh, int n_items, int H, int R) {
  const int row = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63;
  if (row >= n_items) return;
  const int kmax = positions[row] + 1, len = (seq_lens ? seq_lens : positions)[row];
  if (seq_lens && len <= 0) return;
  const int kmin = window > 0 ? max(0, kmax - window) & ~(LAT_UNIT - 1) : 0;
  const LatTiles tl = lat_tiles(nparts, kmin, kmax, R);
  if (tl.per >= tl.n) return;
  const int np = (tl.n + tl.per - 1) / tl.per;
  const long pr = ((long)row * H + h) * nparts;
  const float mp = lane < np ? part_ml[2 * (pr + lane)] : -INFINITY;
  const float lp = lane < np ? part_ml[2 * (pr + lane) + 1] : 0.f;
  const float gv = gate ? bf2f(gate[row * gate_st + h]) : 0.f, sk = sink ? sink[h] : 0.f;
  // (R % 8 == 0, R <= 512: one unit of four columns per thread; past R: the last one, unused)
  const int c = min(4 * (int)threadIdx.x, R - 4);
  f32x4 x[LM_P];
#pragma unroll
  for (int p = 0; p < LM_P; ++p)                        // (past the last one: the last one, unused)
    x[p] = *reinterpret_cast<const f32x4*>(part_acc + (pr + min(p, np - 1)) * R + c);
  const float M = wave_max(mp);
  const float wp = (mp == -INFINITY) ? 0.f : exp2f(mp - M);
  float L = wave_sum(lp * wp);
  if (sink && M != -INFINITY) L += exp2f(sk * 1.4426950408889634f - M);
  float f = L > 0.f ? 1.0f / L : 0.f;
  if (gate) f *= 1.0f / (1.0f + expf(-gv));
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  int p = 0;
  auto join = [&](const f32x4& part) {
    v += part * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wp), p));
    ++p;
  };
#pragma unroll
  for (int i = 0; i < LM_P; ++i)
    if (i < np) join(x[i]);
  while (np - p > LM_P) {
    f32x4 y[2 * LM_P];
#pragma unroll
    for (int i = 0; i < 2 * LM_P; ++i) y[i] = *reinterpret_cast<const f32x4*>(part_acc + (pr + min(p + i, np - 1)) * R + c);
    const int n = min(2 * LM_P, np - p);
#pragma unroll
    for (int i = 0; i < 2 * LM_P; ++i)
      if (i < n) join(y[i]);
  }
#pragma unroll 4
  while (p < np) join(*reinterpret_cast<const f32x4*>(part_acc + (pr + p) * R + c));
  if (4 * (int)threadIdx.x >= R) return;
  bf16x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = f2bf(v[e] * f);
  *reinterpret_cast<bf16x4*>(out + row * out_st + h * out_sh + c) = o;
}

// Decode rows (one query each); prompt portions: latent_flash.hip.
EIA_API int eia_latent_attn_mfma(const void* qa, long qa_st, long qa_sh, const void* qr,
                                 long qr_st, long qr_sh, const float* inv_freq, int rot_dims,
                                 const void* cache, long cache_row, const int* block_table,
                                 int bt_stride, const int* seq_lens, int n_items,
                                 const int* positions, const void* gate, long gate_st, void* out,
                                 long out_st, long out_sh, float scale, int H, int R, int rd, int bs,
                                 int window, const float* sink, int rot_half, float rot_amp,
                                 int nparts, float* part_acc, float* part_ml, hipStream_t st) {
  if (H < 1 || R < 1 || rd < 0 || bs < 1 || rot_dims > rd || (rot_dims & 1) || cache_row < R + rd)
    return EIA_BAD_SHAPE;
  const int Dk = R + rd;
  // 16-byte chunks must not straddle the latent / rotary boundary or the row end
  if ((R & 7) || (Dk & 7) || (cache_row & 7) || Dk > 640 || R > 512 || out_sh % 4 || out_st % 4)
    return EIA_UNSUPPORTED;
  if (n_items <= 0) return EIA_OK;
  const int HB = H < 16 ? H : 16;
  if (nparts < 1 || nparts > 64 || (nparts > 1 && (!part_acc || !part_ml))) return EIA_BAD_SHAPE;
  LatentAttnArgs a{qa, qa_st, qa_sh, qr, qr_st, qr_sh, inv_freq, rot_dims, cache, cache_row,
                   block_table, bt_stride, seq_lens, nullptr, nullptr, n_items, positions, gate,
                   gate_st, out, out_st, out_sh, scale, H, R, rd, bs, 1, HB, 0, 0, window, sink,
                   rot_half, rot_amp, nparts, part_acc, part_ml};
  // Workgroup b runs on XCD b % 8, and partials that meet on the XCD that wrote them come from its L2: so with partitions
  // the grid is padded to whole rounds of the XCDs, a row and its merge on one.  Where a row has more partitions than its
  // share of that XCD's CUs (one workgroup of wide rows each, two of others), the last ones, which only long contexts
  // use, go to the XCDs with fewer rows, as the workgroups beside the rows there; where these are too few, no row is padded.
  // us, unpadded / a row on one XCD only / so, R 512 + 64, no window: one row of 16 heads at 1500 tokens 18.8 / 14.6 / 13.8, at
  // 32768 51 / 64 / 42, of 64 heads at 4000 33 / 34 / 25, at 32768 55 / 193 / 45; 20 rows of 64 heads at 4000 71 / 101 / 73.
  const int y = (H + HB - 1) / HB, per = (n_items + 7) / 8;
  const int home = min(nparts, max(1, (Dk <= 288 ? 64 : 32) / y / per));
  const bool pad = nparts > 1 && (nparts - home) * n_items <= (8 * per - n_items) * home;
  const int rows = pad ? 8 * per : n_items;
  const dim3 grid(rows, y, pad ? home : nparts);
#define LAT_DECODE(NK, NCW, NW) hipLaunchKernelGGL((latent_decode_kernel<NK, NCW, NW>), grid, dim3(64 * NW), 0, st, a)
  if (Dk <= 160 && R <= 128) LAT_DECODE(5, 2, 4);
  else if (Dk <= 288 && R <= 256) LAT_DECODE(9, 4, 4);
  else if (Dk <= 320 && R <= 256) LAT_DECODE(10, 2, 8);
  else if (Dk <= 576) LAT_DECODE(18, 4, 8);
  else LAT_DECODE(20, 4, 8);
#undef LAT_DECODE
  if (nparts > 1)
    hipLaunchKernelGGL(latent_merge_kernel, dim3(rows, H), dim3(128), 0, st, part_acc, part_ml,
                       nparts, seq_lens, positions, window, static_cast<const bf16_t*>(gate),
                       gate_st, sink, static_cast<bf16_t*>(out), out_st, out_sh, n_items, H, R);
  EIA_LAUNCH_CHECK();
}
