// How the kernels of the statequant layout split a matrix's V columns over
// workgroups. Host rules only, plain C++: tests/test_column_tiles_cpu.py compiles
// this header by itself.
#pragma once

#include <stdint.h>

namespace ck {
namespace qs {

constexpr int kGroups = 32;  // column groups per workgroup (one half-wave)

// How a workgroup's threads are laid over a tile's columns and the K-slices.
//  kTileFull: 32 groups of 4 columns.
//  kTileAny: G <= 40 (K = 256, whose 16 slices would take 640 threads and spill:
//    32) groups of 4 columns, G and the number of threads (S * G
//    rounded up to whole waves) set per launch, so a head of any V >= 4 wastes
//    only the last wave's rest.
//  kTileOne: 32 single columns, for V < 4 and where the others' lane offsets do
//    not reach: 2^32 elements (KP V) with 32-bit ones, 2^30 columns otherwise.
// The tiles of a matrix are of equal width (a multiple of 4) and the last one has
// at least 4 columns, so its last thread can take the 4 that end with V, sharing
// some with its neighbour in the same workgroup; the threads past S * G repeat the
// last one's work. What is computed twice has the same value from the same
// inputs, and every input of a workgroup is read before it stores (a barrier
// lies between), which in-place use needs. Columns shared by two workgroups would
// break that: one could read what the other has stored.
enum TileForm : int { kTileFull, kTileAny, kTileOne };

constexpr int max_groups(int KP) { return KP <= 128 ? 40 : 32; }

struct ColTiles {
  int nvt, width;   // tiles and columns per tile (the last one: what is left)
  int groups;       // column groups per tile
  uint32_t inv;     // ceil(2^16 / groups): t / groups = t * inv >> 16 for t < 1024
  TileForm form;
};

// Whether tiles of 32 whole groups are the better split of a V that is a multiple
// of 4, the last tile's idle lanes notwithstanding. fp32_rows: the rows' largest
// elements are fp32. Steps, us, full / any:
//  * V > 160: two or more tiles either way, and of 33 or more groups one takes a
//    fifth wave that is nearly empty (HV=8, K=128, V=516, B=63: int8 43.7 / 56.9,
//    fp16 51.7 / 62.9; V=192, B=170: int8 32.4 / 35.2).
//  * 96 < V < 128: four waves either way (K=256, V=100, B=163: int8 39.5 / 46.0);
//    V = 96 is three waves of any (HV=32, K=128, B=40: fp32 step 20.3 / 22.3, fp32
//    residual 31.8 / 32.8; fp16 21.4 / 20.3, fp8 17.3 / 15.9).
//  * 128 < V <= 160: two tiles of four waves against one of five (K <= 128). From
//    K = 128 that is better with the smaller rows only (V=132, B=248: int8 42.1 /
//    47.5, fp32 step 62.9 / 44.4; K=64, B=496: int8 43.5 / 33.8).
// The ingest holds fewer registers, so its fifth wave costs nothing (K=128, V=132:
// any in 0.79 of full's time, 260 0.98, 516 1.00).
inline bool full_tiles(int V, int KP, bool fp32_rows, bool ingest) {
  const int rest = V % (kGroups * 4);
  if (rest == 0) return true;
  if (V % 4 != 0) return false;
  if (ingest) return rest >= 96;
  return V > 160 || rest > 96 || (rest == 96 && fp32_rows) || (V > 128 && KP >= 128 && !fp32_rows);
}

// ingest: the column ingest, whose lane offsets have 64 bits (a step's: 32).
inline ColTiles col_tiles(int V, int KP, bool fp32_rows, bool ingest) {
  const bool reach = ingest ? V <= 1 << 30 : (int64_t)KP * V < (int64_t)1 << 32;
  const int cpt = V >= 4 && reach ? 4 : 1;
  const int all = (V + cpt - 1) / cpt;  // column groups
  const bool full = full_tiles(V, KP, fp32_rows, ingest);
  const bool any = cpt == 4 && !full;
  int groups = kGroups;
  int nvt = (all + groups - 1) / groups;
  // the fewest tiles, of as many groups as that needs; fewer where that leaves the
  // last tile one group of fewer than 4 columns (V = 6241: 40 tiles of 40 groups)
  for (int most = any ? max_groups(KP) : 0; most > 0; --most) {
    nvt = (all + most - 1) / most;
    groups = (all + nvt - 1) / nvt;
    if (V - (nvt - 1) * groups * 4 >= 4) break;
  }
  return ColTiles{nvt, groups * cpt, groups, (65536u + groups - 1) / groups,
                  cpt == 1 ? kTileOne : full ? kTileFull : kTileAny};
}

// Whether the column ingest is faster with one thread per column than with a
// workgroup per matrix: many matrices, each too small for one. A workgroup costs
// about 0.5 ns (KP = 16) to 5 ns (256) of the chip's time however few columns it
// has; a column's thread K row accesses one after another, 0.4 us each, and lines
// that its neighbours use only while they stay in L2. us, workgroups / threads:
//  * M: [1, 1] 64 matrices 2.4 / 2.2, 4096 3.9 / 2.4, 262144 108 / 2.9; [8, 4] 4096
//    4.5 / 4.1; [16, 3] 4096 4.6 / 6.8, 32768 20.8 / 8.3; [128, 1] 4096 13.7 / 62,
//    32768 80 / 63.
//  * K <= 16: 65535 of [8, 32] 32 / 28, 262144 of it 126 / 151, of [16, 12] 118 / 89,
//    of [16, 16] 129 / 140.
//  * K <= 32: 65535 of [32, 6] 50 / 44, 262144 of [32, 8] 193 / 163, [32, 12] 206 / 242.
//  * above: 65535 of [64, 3] 91 / 63, [100, 4] 143 / 93, [128, 3] 158 / 129, [128, 5]
//    157 / 175; 262144 of [64, 1] 351 / 529.
inline bool few_columns(int64_t M, int K, int V) {
  if (K > 2 && M < (K <= 16 ? 512 * K : 16384)) return false;
  if (K <= 16) return K * (int64_t)V <= (M <= 1 << 17 ? 256 : 224);
  if (K <= 32) return V <= 8;
  return V <= 4 && M <= 1 << 17;
}

// Threads of a workgroup with S slices.
inline int tile_threads(const ColTiles& t, int S) { return (t.groups * S + 63) / 64 * 64; }

// K padded to KP = max(16, next_pow2(K)) (K <= 256)
inline int padded_k(int K) {
  int kp = 16;
  while (kp < K) kp *= 2;
  return kp;
}

inline bool valid_k(int K) { return K >= 1 && K <= 256; }

}  // namespace qs
}  // namespace ck
