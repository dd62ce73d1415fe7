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
// Beyond 512 the chunks that fill whole rounds of 512 keep a key head's heads together, and those of the last round are
// spread as above: 66 chunks of 16 heads of 128 on 8, 528 workgroups, the solve 58.5 -> 51.5 us on an MI355X.  The whole
// op against one without the spread, 8, 16 and 32 heads: 8 to 104 workgroups in the last round 3 to 7 % faster, more of them
// the same (1 %, as runs differ).
struct DeltaSolve {
  int whole, parts;                                    // chunks whose heads stay together; parts of a key head of the others
  long blocks;                                         // workgroups
};
inline DeltaSolve dn_solve(int G, int nchunk, int rep) {
  const long nwg = (long)G * nchunk;
  const int whole = nwg > 512 ? (int)(nwg / 512 * 512 / G) : 0;
  const int parts = whole < nchunk ? dn_parts((long)G * (nchunk - whole), rep) : 1;
  return {whole, parts, (long)G * whole + (long)G * (nchunk - whole) * parts};
}
struct DeltaSolveWg {
  int chunk, kh, parts, part;
};
EIA_DELTA_HD DeltaSolveWg dn_solve_place(long block, int G, int whole, int parts) {
  const long rest = block - (long)whole * G;
  if (rest < 0) return {(int)(block / G), (int)(block % G), 1, 0};
  const int u = (int)(rest % (G * parts));
  return {whole + (int)(rest / (G * parts)), u / parts, parts, u % parts};
}
// First head of part `part` of a key head's rep heads (part == parts: the end).
EIA_DELTA_HD int dn_first_head(int rep, int parts, int part) { return rep * part / parts; }

// Workgroups of the scan: the per_kv ones of a (sequence, key head) meet the same keys and queries, and lie on as few
// XCDs (workgroup b runs on XCD b % 8) as leave all eight of them the same share: 8 / G where G key heads divide
// eight, then the XCD that solved a head also scans it; one where eight divides G; two for others.  MI355X, the
// whole op in us on 1 / 2 / 4 / 8, heads of 128: 8 on 1, one prompt of 3000 tokens 217 / 125 / 120 / 120; 16 on 2, 200
// tokens 47 / 38 / 35 / 33, 1500 130 / 83 / 81 / 81, five of 700 103 / 103 / 91 / 92; 32 on 4, three of 1500 246 / 210 /
// 214 / 217; 8 on 4, 500 tokens 46 / 40 / 44 / 45; 16 on 8, 1000 60 / 60 / 61 / 63; 12 on 3, 1000 61 / 59 / 59 / 59; 10 on
// 5, 1000 58 / 57 / 58 / 60.
struct DeltaSpread {
  int per_kv, shift, each;                             // 2^shift XCDs, `each` workgroups on one
};
inline DeltaSpread dn_spread(int G, int per_kv) {
  const int shift = G % 8 == 0 ? 0 : G == 1 ? 3 : G == 2 ? 2 : 1;
  return {per_kv, shift, (per_kv + (1 << shift) - 1) >> shift};
}
inline int dn_grid(int kvs, const DeltaSpread& x) { return (int)((((long)kvs << x.shift) + 7) / 8 * 8 * x.each); }
struct DeltaWg {
  int kv, in;                                          // in >= per_kv or kv >= kvs: surplus
};
EIA_DELTA_HD DeltaWg dn_place(int block, const DeltaSpread& x) {
  const int slot = block >> 3, row = slot / x.each, unit = 8 * row + (block & 7);
  return {unit >> x.shift, (unit & ((1 << x.shift) - 1)) * x.each + slot - row * x.each};
}
