// Subdomain factors in frontal form: a nested dissection order of each
// subdomain, its fronts (dense column panels over the rows their subtrees
// touch), and the work lists of the solve.  Host part of the set-up; the
// kernels are in doug_fronts.hip.
#pragma once
#include <cstdint>
#include <vector>

#include "doug_setup.hpp"

namespace doug {

constexpr int kFrontCols = 64;    // columns of a front at most
constexpr int kFrontWavesMax = 16;  // wavefronts of the solve's workgroup: 8 or 16
constexpr int kFrontGroupsMax = 8;  // workgroups that share a subdomain's subtrees
// column groups per unit of the solve, FP32 and FP64: 64 rows of them are 8 KB
constexpr int kFrontUnitGroups32 = 8, kFrontUnitGroups64 = 4;

// One front: columns at positions c0 .. c0+k-1 of the elimination order and
// m boundary rows (later positions, ascending).  Its panel holds, for the
// assembled and factored pivot block L L^T, D = inv(L) in rows 0..k-1 and
// C = L_RS inv(L) in rows k..k+m-1, so that a forward step is
// [y; -du] = panel * f and a backward step x = panel^T [y; -x_R].
// Panel layout: groups of four columns; group g keeps rows 4g.. of the
// panel's H = k + m rows (the pivot block is lower triangular), each row's
// four entries in one 16-byte piece (FP32) or in two pieces of two columns,
// the second after the first one's rows (FP64).
struct Front {
  int32_t pan;    // first element of the panel, from the subdomain's base
  int32_t row0;   // first of the front's k + m row records
  int32_t sch;    // first element of its m x m update matrix (set-up)
  int32_t child[2];  // fronts whose updates it takes, or -1
  uint16_t c0, k, m;
  uint16_t u;     // solve: work index of its update vector
};

// elements of a panel, a multiple of 16; a front without columns (a merge of
// two children) keeps one group of zeros
constexpr int64_t front_panel_elems(int64_t k, int64_t m) {
  const int64_t ng = k > 0 ? (k + 3) / 4 : 1, h = k + m;
  return (4 * (ng * h - 2 * ng * (ng - 1)) + 15) / 16 * 16;
}

// Everything a subdomain's structure determines; subdomains of the same
// local graph share one.
//
// Work vector of a solve (of even length): positions 0..n-1, then usz entries:
// entry n stays zero, update vectors follow; in the backward pass the same entries hold
// the solution at the positions from top0 on (entry n + p - top0).
// Row records: rpos, the position of each of the k + m rows; src, the work
// indices of up to two children's update entries for the row (low and high
// half, n where there is none).
// Work lists: each wavefront of the solve walks its own list of units, one
// list forward and one backward.  A unit is 64 rows (one chunk) of up to
// `ug` column groups of one front.  Every list has an even length.
struct alignas(16) FrontUnit {
  int32_t pan, row0;   // the front's panel and first row record
  uint16_t h, k, c0, u;  // rows, columns, first position, update vector
  uint8_t g0, g1;      // column groups [g0, g1)
  uint8_t chunk;       // rows 64 chunk ..
  uint8_t flags;       // FU_*
  uint16_t nbar;       // workgroup barriers behind this unit
  uint16_t pad0;
  int32_t pad1, pad2;
};
enum {
  FU_FIRST = 1,   // the front's first unit on this wavefront
  FU_BEGIN = 2,   // forward: first unit of its rows; backward: of its columns
  FU_END = 4,     // ... and the last
  FU_WHOLE = 8    // forward: the wavefront has all rows of the front
};  // no flag: nothing is kept, barriers only

struct FrontPattern {
  int n = 0, top0 = 0, usz = 0;
  bool mirrored = false;  // edges were added in reverse: its subdomains' own structures may differ
  int64_t elems = 0;   // panel elements
  int64_t schur = 0;   // set-up work elements
  std::vector<int32_t> order;      // position -> index in the subdomain's list
  std::vector<uint16_t> colfront;  // front of each position
  std::vector<Front> fronts;       // children before parents
  std::vector<uint16_t> rpos;
  std::vector<uint32_t> src;
  std::vector<int32_t> hptr;       // fronts by height: hlist[hptr[h]..hptr[h+1])
  std::vector<uint16_t> hlist;
  std::vector<FrontUnit> units_f, units_b;   // wavefront w: units[list[w] .. list[w + 1])
  std::vector<int32_t> list_f, list_b;
  // With several groups the lists above hold the apex only; workgroup g takes
  // subtrees, their bottom fronts at the positions [gpos[g], gpos[g + 1]) and
  // top ones at [gtop[g], gtop[g + 1]), its wavefront w list nw g + w of these.
  // uidx: the work indices of the updates that the apex takes from them, group
  // by group.
  int groups = 1;
  std::vector<FrontUnit> bunits_f, bunits_b;
  std::vector<int32_t> blist_f, blist_b, gpos, gtop, uoff;
  std::vector<uint16_t> uidx;
  int work() const { return n + usz; }
};

// Element of a panel of H rows that holds (row, col), row >= col; `dbl`: the
// FP64 layout.
inline int64_t front_elem(int H, int row, int col, bool dbl) {
  const int64_t g = col / 4, j = col % 4;
  const int64_t base = 4 * (g * H - 2 * g * (g - 1));
  if (!dbl) return base + 4 * (row - 4 * g) + j;
  return base + (j / 2) * 2 * (H - 4 * g) + 2 * (row - 4 * g) + j % 2;
}
// Panel element of the pair of positions lo <= hi (lo's front holds hi).
int64_t front_entry(const FrontPattern& p, int lo, int hi, bool dbl);

// Patterns of all subdomains (blocks of `inds`, structure of A restricted to
// each): pat[b] is subdomain b's pattern in `patterns`, out its blocks in
// elimination order.  False, with nothing usable, when some subdomain's
// structure exceeds the format (work indices of 16 bits, `max_work` entries
// of work vector, panel offsets of 31 bits).  nw wavefronts per workgroup,
// `groups` workgroups for the subtrees, ug column groups per unit.  With
// `chosen`, half as many workgroups for all, a quarter and so on down to one
// where `groups` do not fit: the dissections, nearly all of the work, serve
// each try.
bool build_front_patterns(const Csr& A, const std::vector<int>& starts, const std::vector<int>& inds,
                          int64_t max_work, int nw, int groups, int ug,
                          std::vector<FrontPattern>& patterns, std::vector<int>& pat,
                          std::vector<int>& out, int* chosen = nullptr);

}  // namespace doug
