// Which GEMM a call's EXL3 linears over M rows take: the many-row one (Exl3GemmRowsKernel) or the
// few-row path (split-K GEMM and output transform), both with the same bits.  Host code only.
#pragma once

#include <algorithm>

namespace cx {

constexpr int kRowsMaxBlocks = 8;  // 16-row blocks of an entry of the many-row GEMM

// One linear of a call: A and ncp its k-tiles and column pairs, S the few-row path's K segments.
struct RowsShape {
  int A, ncp, S, k2, cb;
};

// Workgroups of a linear of `entries` row entries in the many-row GEMM: entry e's column blocks on XCD e % 8
// (ids go to the XCDs round-robin), so its activation rows are fetched into one L2; with fewer than 16
// entries in plain order.
constexpr int RowsJobGroups(int entries, int ncp) { return (entries < 16 ? entries : (entries + 7) / 8 * 8) * (ncp / 4); }

// Returns the 16-row blocks per entry of the cheapest many-row form, 0 for the few-row path, by their
// estimated times in us.  Both estimates: a fixed part, the traffic beside the weights, and per launch
// (the linears of one rate and codebook) the steps of its workgroups.
//   Few rows: waves of A / (8 S) steps (32 k) for each 64 rows, 256 workgroups a round.
//   Many rows: a step of a wave decodes one column pair (p below: by rate and codebook) and multiplies n row
//   blocks; up to 256 workgroups run one per CU, further ones two per CU, 512 a round.
// Fitted to 4,356 calls in both forms (1-8 bpw, three codebooks, 18 shapes and groups, 65-4,096 rows): 97% of
// the few-row times are met within 15%, 94% of the many-row ones within 10%.  The chosen form is on average 0.3%
// above the best of all nine; 11 of the calls are more than 3%, none more than 6.1% above the few-row path.
// Few rows / many rows measured: 2048 -> 4096 128 rows 22.7 / 24.7 (3inst 8 bpw 23.4 / 36.6), 512 rows
// 56.5 / 33.9 (57 / 46), 2,048 rows 181 / 64; 2048 -> 512 1,024 rows 26.3 / 26.9 (26.5 / 39.3).
inline int RowsBlocks(const RowsShape* jobs, int n_jobs, int M) {
  if (M <= 64) return 0;
  const int blocks = (M + 15) / 16;
  const double m = 1e-6 * M;
  double few = 9.2, many[kRowsMaxBlocks + 1] = {};
  for (int j = 0; j < n_jobs; ++j) {
    const double in = m * 16.0 * jobs[j].A, out = m * 32.0 * jobs[j].ncp;
    few += 0.98 * in + 5.9 * out * jobs[j].S;
    many[0] += 1.08 * in + 0.76 * out + 0.68 * out * (jobs[j].S - 1);
  }
  for (int n = 1; n <= kRowsMaxBlocks; ++n) many[n] = 7.2 + many[0];
  for (int j = 0; j < n_jobs; ++j) {
    const int k2 = jobs[j].k2, cb = jobs[j].cb;  // the launch of the linears like j, at the first of them
    const auto like = [&](int i) { return jobs[i].k2 == k2 && jobs[i].cb == cb; };
    bool seen = false;
    for (int i = 0; i < j; ++i) seen = seen || like(i);
    if (seen) continue;
    double wgs = 0, work = 0, longest = 0;
    for (int i = j; i < n_jobs; ++i) {
      if (!like(i)) continue;
      const double w = (double)jobs[i].ncp * jobs[i].S * ((M + 63) / 64), steps = jobs[i].A / (8.0 * jobs[i].S) + 2.0;
      wgs += w;
      work += w * steps;
      longest = std::max(longest, steps);
    }
    few += 0.24 * longest + 0.25 * (work / wgs) * (double)((long)(wgs + 255) / 256);
    const double p = cb == 2 ? 0.205 + 0.0043 * k2 : (cb == 1 ? 0.305 : 0.336) + 0.0038 * k2;
    for (int n = 1; n <= std::min(kRowsMaxBlocks, blocks); ++n) {
      const int entries = (blocks + n - 1) / n;
      long groups = 0;
      double full = 0, full_max = 0, lone_max = 0;
      for (int i = j; i < n_jobs; ++i) {
        if (!like(i)) continue;
        const int g = RowsJobGroups(entries, jobs[i].ncp);
        const double steps = jobs[i].A / 2, f = steps * (1.5 * p + 0.016 * n) + 0.51 * n;
        groups += g;
        full += g * f;
        full_max = std::max(full_max, f);
        lone_max = std::max(lone_max, steps * (p + 0.0215 * n) + 0.47 * n);
      }
      const long rest = groups % 512;
      many[n] += (double)(groups / 512) * (full / groups) + (rest == 0 ? 0 : rest <= 256 ? lone_max : full_max);
    }
  }
  int best = 0;
  for (int n = 1; n <= std::min(kRowsMaxBlocks, blocks); ++n)
    if (many[n] < (best ? many[best] : 0.97 * few)) best = n;
  return best;
}

}  // namespace cx
