// Host-side (CPU) algorithms of the hot path; see host_algos.cpp.
#pragma once
#include <algorithm>
#include <cstdint>
#include <string>
#include <vector>

namespace laamd {

int topo_sort2(int n, int base, const int *ai, const int *aj, bool upper,
               int *iperm, int *prefix);
void split_ldu(int n, int base, const int *ai, const int *aj, const double *av,
               int *Lai, int *Laj, double *Lav, double *D, int *Uai, int *Uaj,
               double *Uav, int64_t *lnnz, int64_t *unnz);
void split_triangle(int n, int base, const int *ai, const int *aj,
                    const double *av, bool upper, int *Tai, int *Taj,
                    double *Tav, int64_t *tnnz);
void rowwise_sqrt_norm(int n, int base, const int *ai, const double *av, double *d);
void dtad(int n, int base, const int *ai, const int *aj, double *av, const double *d);
bool diagonal(int n, int base, const int *ai, const int *aj, const double *av,
              int *diagpos, double *diag);
void transpose(int rows, int cols, int base, const int *ai, const int *aj,
               const double *av, int *ti, int *tj, double *tv);
void permute(int n, int base, const int *ai, const int *aj, const double *av,
             const int *iperm, const int *perm, int *pai, int *paj,
             double *pav);
// RCM, bit-exact with the reference's SerialCM: with a team of host threads
// (nthreads <= 0: LAAMD_HOST_THREADS, else the hardware's, at most 16) for
// structurally symmetric patterns, serially otherwise
void rcm(int n, int base, const int *ai, const int *aj, int *iperm, int *perm,
         int nthreads = 0);
void rcm_serial(int n, int base, const int *ai, const int *aj, int *iperm, int *perm);
bool pattern_symmetric(int n, int base, const int *ai, const int *aj);
void iluk_symbolic(int n, int base, const int *ai, const int *aj, int level,
                   std::vector<int> &fai, std::vector<int> &faj,
                   std::vector<int> &first_upper);
bool iluk_numeric(int n, int base, const int *ai, const int *aj,
                  const double *av, const int *fai, const int *faj,
                  const int *first_upper, double *fav);
void icc_symbolic(int n, int base, const int *ai, const int *aj,
                  const int *diag_pos, int lvl, std::vector<int> &icc_ai,
                  std::vector<int> &icc_aj);
bool icc_numeric(int n, int base, const int *ai, const int *aj, const double *av,
                 const int *diag_pos, double omega, const int *icc_ai,
                 const int *icc_aj, double *icc_av);
bool ick_numeric(int n, int base, const int *ai, const int *aj, const double *av,
                 const int *diag_pos, double shift, const int *icc_ai,
                 const int *icc_aj, double *icc_av);

// Tiled schedule of the sync-free triangular solve (tiling.cpp): rows cut
// into tiles of a grid the pattern is recognised as, each tile's rows in
// (level, index) order in groups of at most `lanes` / rlanes rows of one
// level. Rows of up to kTileMaxEntries entries take one lane; longer rows,
// up to kTileRowLanes * kTileMaxEntries, take kTileRowLanes lanes.
constexpr int kTileMaxEntries = 8;  // entries per lane
constexpr int kTileRowLanes = 4;    // lanes of a long row
constexpr int kTileWindow = 16;     // groups a tile keeps its results for
struct TileLayout {
  int nparts = 0, ngroups = 0;
  int rlanes = 1;  // lanes per row (a row's entries are split in order)
  int m_max = 0;   // rows of the largest tile
  int h_max = 0;   // most values one tile reads from other tiles
  int maxe = 0;    // entries per lane slot (2, 4 or kTileMaxEntries)
  int tau = 0;     // tile edge in grid steps
  double remote_frac = 0;  // entries read from another tile
  // most rows of one group that other tiles read; those rows come first in
  // their group
  int shared_max = 0;
  std::vector<int> part_gptr;  // tile p: groups [part_gptr[p], part_gptr[p+1])
  std::vector<int> grp_row;    // group g: row positions [grp_row[g], grp_row[g+1])
  std::vector<int> tperm;      // row position -> row
  // per row position, rlanes slots of maxe entries: >= 0 an LDS slot of
  // the tile's own earlier rows ((group % kTileWindow) * lanes + rlanes *
  // row in group; the slot kTileWindow * lanes reads 0 and pads short
  // rows), < 0 the halo slot -(code+1); tsrc: the entry's index in the
  // row-order triangle (-1: pad)
  std::vector<int> tcode, tsrc;
  // group g's first reads from other tiles: [rf_ptr[g], rf_ptr[g+1]) of
  // (rf_col: the row, rf_slot: its halo slot, rf_grp, rf_pos: the
  // group that solves it and its place there)
  std::vector<int> rf_ptr, rf_col, rf_slot, rf_grp, rf_pos;
};
// ai/aj: 0-based strict triangle in row order; level: each row's level.
// False (with the reason) when no tiling applies.
bool build_tile_layout(int n, const int *ai, const int *aj, const int *level, int lanes,
                       int max_parts, int max_rows, int max_halo, TileLayout &out,
                       std::string &why);

// Tiled solve (sptrsv.hip): groups whose rows sit in registers, which is one
// block of its I/O wavefronts.
constexpr int kTileDepth = 8;
// The I/O wavefronts touch a block's records kTileAhead blocks ahead of the
// solver, if the records between the two, over the tiles that are active at
// a time (groups / levels), stay within kTileTouchBytes: with more, lines are
// displaced before they are used and the touches only add traffic. A lower
// triangle with / without touches: 512^2 FP64 (0.5 MB) 158 / 169 us, 27-point
// 24^3 FP64 (2.0 MB) 75 / 79 us, 7-point 128^3 FP32 (7.1 MB) 118 / 126 us,
// 100^3 FP64 (7.4 MB) 99 / 106 us; 160^3 FP64 (16 MB) 493 / 422 us, 27-point
// 112^3 FP32 (14 MB) 329 / 313 us, 96^3 FP64 (19 MB) 359 / 301 us. The line is
// a compromise: 27-point FP64 already loses at 6-7 MB (56^3 186 / 178 us, 1250
// x 22 x 22 394 / 320 us), 7-point 128^3 FP64 still gains at 11 MB (126 / 134
// us). Three blocks ahead: 2-4% slower than four.
constexpr int kTileAhead = 4;
constexpr int64_t kTileTouchBytes = 8 << 20;
inline bool tile_touch(int64_t groups, int64_t levels, int64_t record_bytes) {
  const int64_t active = groups / levels + 1;
  return active * kTileAhead * kTileDepth * record_bytes <= kTileTouchBytes;
}

// Device factorisation (numeric.hip).
// One sync-free launch, or one launch per level? The first gives every row as
// many lanes as the longest one needs and keeps about 4096 wavefronts in
// flight, 0.049 ns per row and lane, and a level costs it 1.4-4 us; the second
// pays about 14 us a level and 0.25 ns a row with 0.28 ns an elimination. So
// levels decide, except where few of them hold very many rows that are much
// shorter than the longest. One launch / one per level, ILU(0) of a random
// graph with n rows of mean degree d: n = 500K, d = 4 (17 levels, 32 lanes)
// 821 / 675 us, d = 8 (26 levels, 32 lanes) 857 / 1164 us; n = 2M, d = 2 (12
// levels, 16 lanes) 1.58 / 1.21 ms, d = 4 (32 lanes) 3.06 / 1.87 ms. 128^3
// 7-point cells by colour (2 levels, 8 lanes) 0.91 / 2.00 ms; 1M rows of a
// diagonal and one of 60 entries (64 lanes) 2.93 / 0.35 ms.
inline bool factor_one_launch(int64_t rows, int64_t levels, int lanes, int64_t eliminations) {
  const double one = 4000.0 * levels + 0.049 * rows * lanes;
  const double per_level = 14000.0 * levels + 0.25 * rows + 0.28 * eliminations;
  return one <= per_level;
}
// Workgroups of the one launch: kFacAhead levels of chunks at a time (clamped
// to 64 .. 1024), so that the pattern work of later rows is done while they
// wait. 27-point ILU(1) on 48^3 with 1 / 2 / 4 / 8 / 16 levels ahead (8
// wavefronts): 8.3 / 6.1 / 3.4 / 2.3 / 2.2 ms; 72^3 IC(0) with 4 / 8 / 32: 490
// / 465 / 573 us (more pollers)
constexpr int64_t kFacAhead = 12;
inline int factor_workgroups(int64_t chunks, int64_t levels) {
  return static_cast<int>(
      std::min<int64_t>(chunks, std::clamp<int64_t>(kFacAhead * chunks / levels, 64, 1024)));
}

// seeded generators (gen.cpp)
struct SplitMix64 {
  uint64_t s;
  explicit SplitMix64(uint64_t seed) : s(seed) {}
  uint64_t next() {
    uint64_t z = (s += 0x9E3779B97F4A7C15ULL);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
  }
  // uniform in [0,1) with 53 random bits
  double uniform() { return (next() >> 11) * (1.0 / 9007199254740992.0); }
};

}  // namespace laamd
