// How a call of the fp8 GEMM is cut into tiles: plain C++, so that the CPU tests
// compile it as it stands.
#pragma once

#include <algorithm>

#ifdef __HIPCC__
#define QH_HD __host__ __device__ __forceinline__
#else
#define QH_HD inline
#endif

namespace qh {

namespace gemm {
constexpr int BM = 256;     // tile tokens
constexpr int BR = 256;     // tile weight rows
constexpr int BK = 128;     // K block: one MFMA, one scale block
constexpr int GROUP_M = 4;  // tile rows per column sweep (see launch_gemm)
enum { kStoreBf16 = 0, kSiluQuant = 1, kQkvRope = 2 };
}  // namespace gemm

// Tile t of tiles_m x tiles_n in tile order: group_m tile rows per column sweep.
QH_HD void tile_at(int t, int group_m, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int in_group = group_m * tiles_n;
  const int first_m = (t / in_group) * group_m;
  const int gsize = tiles_m - first_m < group_m ? tiles_m - first_m : group_m;
  tm = first_m + (t % in_group) % gsize;
  tn = (t % in_group) / gsize;
}

namespace gemm_small {

constexpr int MAX_NK = 256;  // K blocks whose weight scales a small tiling's LDS rows hold

// A tiling's cost model: tiles in rounds of one per CU, `fixed` us plus per K
// block `first` us for the first round and `more` us for each further one
// (shorter where two workgroups share a CU, longer where a full chip runs at a
// lower clock). Fitted over the Qwen3-4B and Qwen3-32B projections at 1 to
// 40,000 tokens (248 sizes, every tiling timed at each, one MI355X).
struct Tiling {
  int rows, tokens;
  float fixed, first, more;
};
constexpr Tiling kLarge[3] = {{256, 256, 2.7f, 1.288f, 1.784f},    // kStoreBf16
                              {256, 256, 0.0f, 1.726f, 1.822f},    // kSiluQuant
                              {256, 256, 11.9f, 1.214f, 1.975f}};  // kQkvRope
constexpr int kTilings[3] = {7, 4, 5};
constexpr Tiling kSmall[3][7] = {
    {{32, 16, 4.1f, 0.104f, 0.132f},
     {64, 16, 2.6f, 0.161f, 0.162f},
     {64, 32, 2.8f, 0.186f, 0.193f},
     {64, 64, 2.4f, 0.245f, 0.268f},
     {128, 64, 0.5f, 0.408f, 0.326f},
     {128, 128, 3.1f, 0.498f, 0.629f},
     {256, 128, 2.6f, 0.767f, 1.001f}},
    {{256, 16, 0.f, 0.704f, 0.568f},
     {256, 32, 0.f, 0.797f, 0.682f},
     {256, 64, 0.f, 0.900f, 0.780f},
     {256, 128, 0.f, 1.155f, 1.125f}},
    {{128, 16, 4.3f, 0.236f, 0.249f},
     {128, 32, 4.1f, 0.278f, 0.256f},
     {128, 64, 5.5f, 0.314f, 0.469f},
     {128, 128, 7.5f, 0.430f, 0.771f},
     {256, 128, 10.2f, 0.672f, 1.249f}}};

// How a chunk is tiled: the first `large` 256 x 256 tiles, in tile order, as
// such, the rest, if any, on tiling `small` (an index into kSmall[epi]).
struct Plan {
  int large, small;
};

static int all_tiles(int M, int N) {
  return ((M + gemm::BM - 1) / gemm::BM) * (N / gemm::BR);
}

// The 256 x 256 tiles of a call from tile `from` on, cut into pieces of a
// tiling. A tile of the last tile row has pieces only where it has tokens, and
// the launch holds those and no others. Workgroups are dealt to XCDs and shader
// engines in turn, whatever they do: with the pieces of no tokens among them some
// engines got more live ones than they have CUs, and a round that the cost model
// counts once took two. Times against 256 x 256 tiles alone, with those pieces
// -> without: gate_up at 2,840 tokens 1.10 -> 0.96, at 7,271 1.05 -> 0.99,
// Qwen3-32B's at 277 tokens 1.17 -> 0.88, qkv at 6,747 1.12 -> 0.97.
struct Pieces {
  int from, tiles_n, tiles_m;
  int first_m, gsize;   // the last group of tile rows: its first row, its rows
  int cm, cn, cm_last;  // pieces of a tile along tokens and rows; along tokens in the last row

  QH_HD Pieces(int from_, int M, int N, int tokens, int rows) {
    from = from_;
    tiles_m = (M + gemm::BM - 1) / gemm::BM;
    tiles_n = N / gemm::BR;
    first_m = (tiles_m - 1) / gemm::GROUP_M * gemm::GROUP_M;
    gsize = tiles_m - first_m;
    cm = gemm::BM / tokens;
    cn = gemm::BR / rows;
    cm_last = (M - (tiles_m - 1) * gemm::BM + tokens - 1) / tokens;
  }
  // pieces ahead of the last group, and of a column of it
  QH_HD int ahead() const { return max0(first_m * tiles_n - from) * cm * cn; }
  QH_HD int column() const { return ((gsize - 1) * cm + cm_last) * cn; }
  // tiles of the last group ahead of `from`: whole columns, then tiles that are
  // not in the last row
  QH_HD int skipped() const { return max0(from - first_m * tiles_n); }
  QH_HD long count() const {
    return (long)max0(first_m * tiles_n - from) * cm * cn +
           (long)(tiles_n - skipped() / gsize) * column() - skipped() % gsize * cm * cn;
  }
  // piece t in tile order: row tm and column tn of a matrix of pieces
  QH_HD void at(int t, int& tm, int& tn) const {
    int p;  // piece of the tile
    if (t < ahead()) {
      tile_at(from + t / (cm * cn), gemm::GROUP_M, tiles_m, tiles_n, tm, tn);
      p = t % (cm * cn);
    } else {
      t += skipped() % gsize * cm * cn - ahead();
      tn = skipped() / gsize + t / column();
      t %= column();
      const bool whole = t < (gsize - 1) * cm * cn;
      tm = whole ? first_m + t / (cm * cn) : tiles_m - 1;
      p = whole ? t % (cm * cn) : t - (gsize - 1) * cm * cn;
      if (!whole) {
        tm = tm * cm + p % cm_last;
        tn = tn * cn + p / cm_last;
        return;
      }
    }
    tm = tm * cm + p % cm;
    tn = tn * cn + p / cm;
  }

 private:
  static QH_HD int max0(int x) { return x > 0 ? x : 0; }
};

// The plan with the lowest cost, the small tilings' taken 10 % up (so that no
// size of the fit runs slower than on 256 x 256 tiles alone; without it eight
// did, by up to 9 %). With one tiling for all tokens the choice costs 0.02 %
// on average and 2 % at most against the best measured one. Against 256 x 256
// tiles alone (us, Qwen3-4B):
//   tokens   qkv           o             gate_up       down
//        1   32.9 ->  8.5  42.6 ->  6.6  32.7 -> 12.3  94.0 -> 11.6
//       64   33.3 ->  9.0  42.6 ->  7.9  32.4 -> 14.4  94.0 -> 14.2
//      256   35.4 -> 11.9  43.3 -> 10.6  33.0 -> 22.0  95.8 -> 21.2
//     1024   37.1 -> 25.8  44.1 -> 20.8  69.6 -> 57.7  96.0 -> 43.0
//     2048   40.1          44.0 -> 29.7   109 ->  103  96.1 -> 62.2
// Where the last round of 256 x 256 tiles would leave most of the chip idle,
// its tiles are cut into small ones in a second launch, which costs 8 us here
// (its start, and a first round on cold LDS; with 4 two sizes ran up to 4 %
// slower than unsplit). Tiles and not whole tile rows: gate_up has 76 tiles a
// row. Measured (us, 256 x 256 tiles alone -> so): gate_up at 1,157 tokens, 380
// tiles on 256 CUs, 71.7 -> 66.2, at 900 68 -> 56; o at 7,200 tokens, 290 tiles,
// 98 -> 75; down 218 -> 160, at 14,000 343 -> 293; qkv at 3,000 76 -> 58;
// Qwen3-32B at 4,000 tokens o 189 -> 151, down 565 -> 441. A split saves less of
// a longer call: gate_up's of both models take 0.89 of the unsplit time on
// average behind one or two whole rounds, 0.93 behind 3 to 5, 0.97 behind 6 to 11,
// 0.99 behind 12 to 49 and 1.00 past that, where a call's runs differ by 1 to 2 %
// (to 131,072 tokens; the constants are fitted to 40,000).
static Plan choose(int epi, int M, int N, int K, int cus) {
  const int all = all_tiles(M, N);
  const int nk = K / gemm::BK;
  if (nk >= MAX_NK) return {all, 0};  // the scale rows in LDS hold fewer blocks
  auto cost = [&](const Tiling& t, long tiles) {
    const long rounds = (tiles + cus - 1) / cus;
    return t.fixed + (float)nk * (t.first + t.more * (float)(rounds - 1));
  };
  Plan best = {all, 0};
  float least = cost(kLarge[epi], all);
  auto with_small = [&](int large) {
    const float ahead = large > 0 ? cost(kLarge[epi], large) + 8.f : 0.f;
    for (int i = 0; i < kTilings[epi]; ++i) {
      const Tiling& t = kSmall[epi][i];
      const float c = ahead + 1.10f * cost(t, Pieces(large, M, N, t.tokens, t.rows).count());
      if (c < least) {
        least = c;
        best = {large, i};
      }
    }
  };
  with_small(0);
  // whole rounds of 256 x 256 tiles, all but the last one or two (gate_up: the
  // last; one more round in small tiles, 128 tokens at best, measured 1 % slower
  // than unsplit at 6,000 tokens and never best)
  const int rounds = all / cus;
  for (int r = rounds; r >= 1 && r >= rounds - (epi == gemm::kSiluQuant ? 0 : 1); --r) {
    // qkv past two rounds stays whole. The line was drawn when its small tilings'
    // epilogue was longer and whole tile rows were cut (the split measured -3 to
    // +5 %). With the present ones it would gain where the last round is short:
    // -4 to -12 % up to 0.4 of a round, -1.4 to +1.4 % above (130 sizes of 3 to 25
    // rounds, both models; 11,462 tokens 201 -> 189 us, Qwen3-32B's 6,523 346 -> 304).
    if (epi == gemm::kQkvRope && r > 2) continue;
    if (r * cus < all) with_small(r * cus);
  }
  return best;
}

}  // namespace gemm_small
}  // namespace qh
