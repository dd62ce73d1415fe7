// How the chunk-parallel delta rule (delta_scan.hip) spreads its workgroups; plain C++, so that host code can
// include it.
#pragma once
#ifdef __HIPCC__
#define EIA_DELTA_HD __host__ __device__ __forceinline__
#else
#define EIA_DELTA_HD inline
#endif

// Workgroups of the solve that share the rep heads of a key head: heads are halved among more of them while all
// nwg (chunks x key heads) times that have a place (512: two per CU).  Each of them stages and multiplies K; in
// turn a head costs 7 us.  MI355X, the whole op in us with 1 / 2 / 4 / 8: 16 heads of 128 on 2, one prompt of 64
// tokens (nwg 2) 74 / 51 / 40 / 33, of 500 (16) 104 / 80 / 67 / 61, three of 1500 (112) 146 / 125 / 125 / 131; 32 on
// 4, three of 1500 (224) 248 / 241 / 253 / 272; 16 on 8, one of 1000 (128) 65 / 60, of 2048 (256) 100 / 98, of 4096
// (512) 179 / 189.
inline int dn_parts(long nwg, int rep) {
  int parts = 1;
  for (int heads = rep / 2; heads >= 1; heads /= 2) {
    const int more = (rep + heads - 1) / heads;
    if (nwg * more > 512) break;
    parts = more;
  }
  return parts;
}
// First head of part `part` of a key head's rep heads (part == parts: the end).
EIA_DELTA_HD int dn_first_head(int rep, int parts, int part) { return rep * part / parts; }
