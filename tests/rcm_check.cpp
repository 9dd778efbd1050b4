// block_rcm: blocks that are said to share a local graph come out as when each
// is ordered by itself, whatever the numbering and the thread count.
#include "doug_setup.hpp"

#include <algorithm>
#include <cstdio>

using namespace doug;

int main() {
  // a grid whose boxes of two shapes repeat, numbered in strides so that a
  // block's numbers lie far apart, and single nodes in between
  const int nx = 24, ny = 20, n = nx * ny;
  std::vector<int> to((size_t)n);
  for (int i = 0; i < n; i++) to[i] = (int)((int64_t)i * 77 % n);
  Csr A;
  A.nrows = A.ncols = n;
  std::vector<std::vector<int>> row((size_t)n);
  auto edge = [&](int a, int b) {
    row[to[a]].push_back(to[b]);
    row[to[b]].push_back(to[a]);
  };
  for (int x = 0; x < nx; x++)
    for (int y = 0; y < ny; y++) {
      row[to[x * ny + y]].push_back(to[x * ny + y]);
      if (x + 1 < nx) edge(x * ny + y, (x + 1) * ny + y);
      if (y + 1 < ny) edge(x * ny + y, x * ny + y + 1);
    }
  A.ptr.assign(1, 0);
  for (auto& r : row) {
    A.col.insert(A.col.end(), r.begin(), r.end());
    A.ptr.push_back((int)A.col.size());
  }
  A.val.assign(A.col.size(), 1.0);
  std::vector<int> starts{0}, inds, same;
  for (int shape = 0; shape < 2; shape++)
    for (int x = 0; x + 4 <= nx; x += 4)
      for (int y = 0; y + 4 <= ny; y += 4) {
        for (int a = 0; a < 4; a++)
          for (int b = 0; b < (shape ? 3 : 4); b++) inds.push_back(to[(x + a) * ny + y + b]);
        starts.push_back((int)inds.size());
        same.push_back(shape ? 7 : 2);
        if ((x + y) % 3 == 0) {  // a node by itself, ordered for itself
          inds.push_back(to[x * ny + y]);
          starts.push_back((int)inds.size());
          same.push_back(-1);
        }
      }
  // entries of a row come in one order for all blocks: sorted by the grid's
  // own numbers, so that equal boxes have equal local graphs entry by entry
  std::vector<int> from((size_t)n);
  for (int i = 0; i < n; i++) from[to[i]] = i;
  for (int i = 0; i < n; i++)
    std::sort(A.col.begin() + A.ptr[i], A.col.begin() + A.ptr[i + 1], [&](int a, int b) { return from[a] < from[b]; });
  std::vector<int> each;
  set_setup_thread_cap(1);
  block_rcm(A, starts, inds, each);
  int bad = 0;
  for (int threads : {1, 2, 5})
    for (bool share : {false, true}) {
      std::vector<int> out;
      set_setup_thread_cap(threads);
      block_rcm(A, starts, inds, out, share ? &same : nullptr);
      if (out != each) {
        printf("%d threads, shared %d: another order\n", threads, (int)share);
        bad++;
      }
    }
  for (size_t b = 0; b + 1 < starts.size(); b++) {  // each block a permutation of its input
    std::vector<int> a(inds.begin() + starts[b], inds.begin() + starts[b + 1]);
    std::vector<int> c(each.begin() + starts[b], each.begin() + starts[b + 1]);
    std::sort(a.begin(), a.end());
    std::sort(c.begin(), c.end());
    bad += a != c;
  }
  return bad;
}
