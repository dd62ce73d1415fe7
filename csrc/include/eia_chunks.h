// Shared by the chunk-parallel recurrences (wkv.hip, linear_scan.hip): chunks that are found on the
// device, the walk over a sequence's chunks, and tiles and weights of chunks with a decay per key channel.
#pragma once
#include "eia_common.h"

// Chunks of C tokens are numbered without a list from the host: sequence s owns the numbers from
// cu[s] / C + s on, at least as many as it has chunks; numbers past its last chunk do nothing.
// The chunk of number x: sequence, first row and tokens; false where there is none.
template <int C>
EIA_DEV bool chunk_of(const int* cu, int nseq, int x, int& s, int& row0, int& n) {
  int lo = 0, hi = nseq - 1;                // largest s with cu[s] / C + s <= x
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (cu[mid] / C + mid <= x) lo = mid; else hi = mid - 1;
  }
  s = lo;
  if (x < cu[s] / C + s) return false;      // (rows before the first sequence)
  row0 = cu[s] + (x - cu[s] / C - s) * C;
  n = min(C, cu[s + 1] - row0);
  return n > 0;
}

// Grids of a workgroup per (head, chunk): all heads of a chunk run side by side, so that the rows they share a
// part of each come in whole; and where eight divides the heads, a head's state stays in the L2 of one XCD between
// the passes (workgroup b runs on XCD b % 8; a grid of a workgroup per sequence takes parts x heads as its heads).
// wkv, two prompts of 571 tokens, 32 heads: 47 -> 39 us, eleven of 196, 16 heads: 44 -> 41, sixteen of 433, 40 heads:
// 178 -> 173; with (1) alone chunk by chunk, one of 4096, 32 heads 105.8, of 1000, 16 heads 27.8, heads first 104.2 and
// 25.8; a decay per channel, four of 977, 16 heads: 109.9 -> 108.0.
// chunk_number: the workgroup's chunk or sequence (past the last one: none).
constexpr int CHUNKS_Y = 32768;
inline dim3 chunk_grid(int chunks, int H) {
  return dim3(H, chunks < CHUNKS_Y ? chunks : CHUNKS_Y, (chunks + CHUNKS_Y - 1) / CHUNKS_Y);
}
EIA_DEV int chunk_number() { return blockIdx.z * CHUNKS_Y + blockIdx.y; }

// Four columns of a state row over a sequence's nc chunks, us apart: U of a chunk, its own contribution, turns into
// the state S before it; step(x, l, u) then takes S past chunk x, with u what U held and l what load(x) gave.  A
// group's contributions are requested while the previous group is summed.
constexpr int CHUNKS_AHEAD = 8;             // chunks whose contributions are in flight
template <typename L, typename Load, typename Step>
EIA_DEV void chunk_walk_with(float* U, long us, int nc, const f32x4& S, Load&& load, Step&& step) {
  f32x4 u[CHUNKS_AHEAD];
  L d[CHUNKS_AHEAD];
  auto fetch = [&](int b, f32x4 (&u)[CHUNKS_AHEAD], L (&d)[CHUNKS_AHEAD]) {
#pragma unroll
    for (int k = 0; k < CHUNKS_AHEAD; ++k) {
      const int x = min(b + k, nc - 1);
      u[k] = *reinterpret_cast<const f32x4*>(U + x * us);
      d[k] = load(x);
    }
  };
  fetch(0, u, d);
  for (int b = 0; b < nc; b += CHUNKS_AHEAD) {
    f32x4 un[CHUNKS_AHEAD];
    L dn[CHUNKS_AHEAD];
    fetch(b + CHUNKS_AHEAD, un, dn);
#pragma unroll
    for (int k = 0; k < CHUNKS_AHEAD; ++k) {
      if (b + k < nc) {
        *reinterpret_cast<f32x4*>(U + (b + k) * us) = S;
        step(b + k, d[k], u[k]);
      }
    }
#pragma unroll
    for (int k = 0; k < CHUNKS_AHEAD; ++k) {
      u[k] = un[k];
      d[k] = dn[k];
    }
  }
}
// The same where the step is a decay; l: its log2, ls apart.
EIA_DEV void chunk_walk(float* U, long us, const float* l, long ls, int nc, f32x4& S) {
  chunk_walk_with<float>(U, us, nc, S, [&](int x) { return l[x * ls]; },
                         [&](int, float d, f32x4 u) { S = S * __builtin_amdgcn_exp2f(d) + u; });
}

// Place of (token, channel) in an fp32 LDS tile [tokens][W]: the 16-byte units of a row are turned by the
// token, so that sixteen tokens' units of one channel group lie on different banks.
template <int W> EIA_DEV int tile_at(int t, int i) { return t * W + (i ^ ((t & 15) << 2)); }
template <int W> EIA_DEV f32x4 tile_get(const float* tile, int t, int i) {       // channels i .. i + 3, i % 4 == 0
  return *reinterpret_cast<const f32x4*>(tile + tile_at<W>(t, i));
}

// Weights inside the 8-token blocks of a wave's tokens t0 .. t0 + 15, 64 channels,
//   P_ts = sum_channels q_t k_s 2^(sum of l_x over the tokens x between),    s < t,
// between: s < x < t, or s < x <= t with SELF.  Every exponent is a sum of the l_x that it covers, never a
// difference of longer sums, so it is <= 0 and keeps its precision behind tokens that forget almost
// everything: through the edge between a block's fours for tokens of both, token by token inside a four.
//
// block_edges leaves the sums up to that edge in tile E (rows of tokens; l: this lane's channel, every
// token of the wave); rows of q, k and E have to be there before block_weights, which uses E up.
template <bool SELF>
EIA_DEV void block_edges(const float (&l)[16], float* E, int t0, int lane) {
#pragma unroll
  for (int b = 0; b < 16; b += 8) {
    float suf = 0.f, pre = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      E[tile_at<64>(t0 + b + 3 - t, lane)] = suf;
      suf += l[b + 3 - t];
      if (SELF) pre += l[b + 4 + t];
      E[tile_at<64>(t0 + b + 4 + t, lane)] = pre;
      if (!SELF) pre += l[b + 4 + t];
    }
  }
}
// -> the operand of P v that a lane holds: query t0 + lane % 16, keys t0 + 4 (lane / 16) + i, with the
// query's weight for itself (own, of query lane % 16) and zero for what is not in its block before it.
template <bool SELF>
EIA_DEV f32x4 block_weights(const float* q, const float* k, float* E, const float (&l)[16], float own,
                            int t0, int lane) {
  // lane: a pair and half of the channels
  const int pr = lane & 31, c0 = lane & 32;
  float v4 = 0.f, v8 = 0.f;
  {                                         // t in the second four of its eight, s in the first
    const int s8 = t0 + 8 * (pr >> 4) + (pr & 3), t8 = t0 + 8 * (pr >> 4) + 4 + (pr >> 2 & 3);
#pragma unroll 4
    for (int i = c0; i < c0 + 32; i += 4) {
      const f32x4 y = tile_get<64>(q, t8, i) * tile_get<64>(k, s8, i);
      const f32x4 d = tile_get<64>(E, t8, i) + tile_get<64>(E, s8, i);
#pragma unroll
      for (int e = 0; e < 4; ++e) v8 += y[e] * __builtin_amdgcn_exp2f(d[e]);
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int t = 0; t < 16; ++t)              // the wave's own rows: l of the tokens that lie between
    if ((t & 3) && (SELF || (t & 3) < 3)) E[tile_at<64>(t0 + t, lane)] = l[t];
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  if (pr < 24) {                            // s < t in the same four
    const int x = pr % 6, t = x >= 3 ? 3 : x >= 1 ? 2 : 1, s = x - t * (t - 1) / 2, r = t0 + 4 * (pr / 6);
    const int end = SELF ? t : t - 1;       // tokens s + 1 .. end lie between
    const bool b1 = s < 1 && end >= 1, b2 = s < 2 && end >= 2, b3 = end >= 3;
#pragma unroll 4
    for (int i = c0; i < c0 + 32; i += 4) {
      const f32x4 y = tile_get<64>(q, r + t, i) * tile_get<64>(k, r + s, i);
      const f32x4 d1 = tile_get<64>(E, r + 1, i), d2 = tile_get<64>(E, r + 2, i);
      f32x4 d3 = {0.f, 0.f, 0.f, 0.f};
      if (SELF) d3 = tile_get<64>(E, r + 3, i);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v4 += y[e] * __builtin_amdgcn_exp2f((b1 ? d1[e] : 0.f) + (b2 ? d2[e] : 0.f) + (SELF && b3 ? d3[e] : 0.f));
    }
  }
  v4 += __shfl_xor(v4, 32, 64);
  v8 += __shfl_xor(v8, 32, 64);
  const float v = lane < 32 ? v8 : v4;
  // to the lanes that hold them as an operand
  const int l16 = lane & 15, g4 = lane >> 4, f4 = l16 >> 2, t4 = l16 & 3;      // the query's four, its place there
  const int from = g4 == f4 ? 32 + 6 * f4 + (t4 * (t4 - 1) >> 1) : 16 * (f4 >> 1) + 4 * t4;
  f32x4 p;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float x = __shfl(v, from + i, 64);
    if (g4 == f4) p[i] = i == t4 ? own : i < t4 ? x : 0.f;
    else p[i] = (f4 & 1) && g4 == f4 - 1 ? x : 0.f;
  }
  return p;
}
