// CPU check of the grouped GEMM tile schedule (csrc/gemm_sched.hpp), built with
// the host compiler alone by tests/test_gemm_schedule.py. Prints "OK" or the
// first failing case and exits non-zero.
//   1. Every tile of a launch is run by exactly one workgroup, whatever the
//      tile count, grid size and chunk size.
//      The same for launches of one tile per workgroup, whose balanced chunk also leaves no
//      XCD with more rounds than an even deal.
//   2. The launcher's grid keeps every workgroup within the LDS row table,
//      for any row table size, group sizes, M and CU count, at the kernel's
//      real tile count (which the launcher bounds from above).
//   3. A group's tile order (panels of M tiles) maps its local tile indices
//      onto its (N tile, M tile) pairs one to one.
//   4. The even split of a group's 32-row blocks over its M tiles covers the blocks in
//      order, at most a tile's worth each, up to the most rows an operand of 4 GiB has.
#include <cstdio>
#include <cstdlib>
#include <algorithm>
#include <random>
#include <vector>

#include "../deepseek-v2-lite-cuda_amd/csrc/gemm_sched.hpp"

using namespace dsk;

static int fail(const char* what, long long a, long long b, long long c) {
  std::printf("FAIL %s (%lld, %lld, %lld)\n", what, a, b, c);
  return 1;
}

int main() {
  // 1. coverage: each tile exactly once
  std::vector<int> seen;
  for (int chunk : {1, 7, 11, 16, 22, 33, 64}) {
    for (int nwg = 8; nwg <= 512; nwg += (chunk == kTileChunk ? 8 : 24)) {
      for (int total = 0; total <= 3000; total += (total < 300 ? 1 : 37)) {
        seen.assign(total, 0);
        long long sum = 0;
        for (int x = 0; x < kXcds; ++x) {
          const int xt = sched_xcd_tiles(total, x, chunk);
          for (int slot = 0; slot < nwg / kXcds; ++slot) {
            const int n = sched_slot_tiles(xt, slot, nwg / kXcds);
            sum += n;
            for (int t = 0; t < n; ++t) {
              const int w = sched_tile_index(x, slot, t, nwg / kXcds, chunk);
              if (w < 0 || w >= total) return fail("tile index out of range", nwg, total, w);
              if (seen[w]++) return fail("tile run twice", nwg, total, w);
            }
          }
        }
        if (sum != total) return fail("tiles lost", nwg, total, sum);
      }
    }
  }
  // 1b. one tile per workgroup, on the grid and balanced chunk of the medium-problem launcher
  for (int cus : {8, 80, 256, 304}) {
    for (int tiles = 1; tiles <= 20000; tiles += (tiles < 1200 ? 1 : 173)) {
      const int chunk = sched_balanced_chunk(tiles, cus);
      if (chunk < 1 || chunk > kTileChunk) return fail("chunk out of range", cus, tiles, chunk);
      const long long even = ((tiles + kXcds - 1) / kXcds + cus / kXcds - 1) / (cus / kXcds);
      // the kernel's tile count may be below the launcher's bound
      for (int total : {tiles, tiles - tiles / 3, tiles / 2}) {
        const long long nwg = sched_single_workgroups(tiles, chunk);
        if (nwg % kXcds || nwg < tiles) return fail("one-tile grid", cus, tiles, nwg);
        seen.assign(total, 0);
        long long sum = 0;
        for (long long i = 0; i < nwg; ++i) {
          const int w = sched_tile_index((int)(i & 7), (int)(i >> 3), 0, 1, chunk);
          if (w < 0) return fail("one-tile index out of range", cus, tiles, w);
          if (w >= total) continue;
          if (seen[w]++) return fail("one-tile launch runs a tile twice", cus, tiles, w);
          ++sum;
        }
        if (sum != total) return fail("one-tile launch loses tiles", cus, tiles, sum);
      }
      for (int x = 0; x < kXcds; ++x)
        if (sched_xcd_tiles(tiles, x, chunk) > even * (cus / kXcds))
          return fail("uneven deal", cus, tiles, x);
    }
  }
  // 2. the launcher's grid respects the row table at the real tile count
  std::mt19937 rng(1234);
  const int BM = 256;
  for (int cus : {8, 80, 256, 304}) {
    for (int rt = 1; rt <= 64; rt = rt < 8 ? rt + 1 : rt * 2) {
      for (int iter = 0; iter < 400; ++iter) {
        const int G = 1 + rng() % 128;
        const int nt = 1 + rng() % 24;
        const int M = rng() % 40000;
        // random group sizes summing to M (the kernel clamps offsets into [0, M])
        std::vector<int> cut(G - 1);
        for (int& c : cut) c = M ? rng() % (M + 1) : 0;
        std::sort(cut.begin(), cut.end());
        long long total = 0;
        int prev = 0;
        for (int g = 0; g < G; ++g) {
          const int end = g + 1 < G ? cut[g] : M;
          total += (long long)((end - prev + BM - 1) / BM) * nt;
          prev = end;
        }
        const long long upper = ((long long)(M + BM - 1) / BM + G) * nt;
        if (total > upper) return fail("tile count above the launcher's bound", M, G, total);
        const int chunk = sched_chunk((int)(rng() % 5), nt, (int)upper, cus);  // 0: balanced
        const long long nwg = sched_persistent_workgroups(upper, cus, rt, chunk);
        if (nwg % kXcds || nwg < kXcds) return fail("grid not a multiple of 8", upper, cus, nwg);
        if (sched_max_tiles((int)total, (int)nwg, chunk) > rt)
          return fail("workgroup beyond the row table", total, nwg, rt);
        if (sched_max_tiles((int)upper, (int)nwg, chunk) > rt)
          return fail("bound beyond the row table", upper, nwg, rt);
        // every tile exactly once on that grid and chunk
        seen.assign(total, 0);
        for (int i = 0; i < nwg; ++i) {
          const int per = (int)nwg / kXcds, x = i & 7, slot = i >> 3;
          const int n = sched_slot_tiles(sched_xcd_tiles((int)total, x, chunk), slot, per);
          for (int t = 0; t < n; ++t) {
            const int w = sched_tile_index(x, slot, t, per, chunk);
            if (w < 0 || w >= total) return fail("persistent tile index", total, nwg, w);
            if (seen[w]++) return fail("persistent launch runs a tile twice", total, nwg, w);
          }
        }
        if (std::count(seen.begin(), seen.end(), 1) != total)
          return fail("persistent launch loses tiles", total, nwg, chunk);
      }
    }
  }
  // 3. the panel order inside a group is a bijection
  for (int mt = 1; mt <= 4 * kPanelM + 3; ++mt) {
    for (int nc = 1; nc <= 24; ++nc) {
      seen.assign(mt * nc, 0);
      for (int l = 0; l < mt * nc; ++l) {
        int nt = -1, mi = -1;
        sched_group_tile(l, mt, nc, &nt, &mi);
        if (nt < 0 || nt >= nc || mi < 0 || mi >= mt) return fail("group tile out of range", mt, nc, l);
        if (seen[mi * nc + nt]++) return fail("group tile run twice", mt, nc, l);
      }
    }
  }
  // 4. the row split, against the same in 64 bits
  for (int tm : {2, 4, 8}) {
    for (long long rows = 1; rows <= 33554432; rows += rows < 5000 ? 1 : rows / 3 + 17) {
      const int nblk = (int)((rows + 31) / 32), mt = (int)((rows + 32 * tm - 1) / (32 * tm));
      const int step = mt > 20000 ? 61 : 1;
      for (int mi = 0; mi <= mt; mi += mi + step <= mt || mi == mt ? step : mt - mi) {
        const int b = sched_tile_block(mi, mt, nblk, tm);
        if (b != (long long)mi * nblk / mt) return fail("row split", rows, tm, mi);
        if (mi < mt) {
          const int n = sched_tile_block(mi + 1, mt, nblk, tm) - b;
          if (n < 1 || n > tm) return fail("blocks of a tile", rows, tm, mi);
        }
      }
      if (sched_tile_block(mt, mt, nblk, tm) != nblk) return fail("row split end", rows, tm, mt);
      if (rows <= kMidMaxRows && (long long)mt * nblk > INT32_MAX)
        return fail("split of the medium-problem kernel", rows, tm, mt);
    }
  }
  std::printf("OK\n");
  return 0;
}
