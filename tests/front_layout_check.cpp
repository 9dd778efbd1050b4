// Layout of the frontal patterns that the kernels rely on, on odd and even
// boxes: prints what fails, returns the number of failures.
#include "doug_fronts.hpp"

#include <cstdio>

using namespace doug;

namespace {

// the grid graph of a box, both triangles and the diagonal
Csr box(int nx, int ny, int nz) {
  Csr A;
  A.nrows = A.ncols = nx * ny * nz;
  A.ptr.assign(1, 0);
  auto id = [&](int x, int y, int z) { return (x * ny + y) * nz + z; };
  for (int x = 0; x < nx; x++)
    for (int y = 0; y < ny; y++)
      for (int z = 0; z < nz; z++) {
        if (x > 0) A.col.push_back(id(x - 1, y, z));
        if (y > 0) A.col.push_back(id(x, y - 1, z));
        if (z > 0) A.col.push_back(id(x, y, z - 1));
        A.col.push_back(id(x, y, z));
        if (z + 1 < nz) A.col.push_back(id(x, y, z + 1));
        if (y + 1 < ny) A.col.push_back(id(x, y + 1, z));
        if (x + 1 < nx) A.col.push_back(id(x + 1, y, z));
        A.ptr.push_back((int)A.col.size());
      }
  A.val.assign(A.col.size(), 1.0);
  return A;
}

}  // namespace

int main() {
  int bad = 0;
  for (int ug : {kFrontUnitGroups32, kFrontUnitGroups64})
    for (int groups : {1, 2, 4, 8})
      for (int e = 1; e <= 18; e++)
        for (int dims : {2, 3}) {
          const int s = dims == 2 ? 3 * e : e;
          const Csr A = dims == 2 ? box(s, s + 1, 1) : box(s, s, s);
          std::vector<int> starts{0, A.nrows}, inds((size_t)A.nrows), out, pat;
          for (int i = 0; i < A.nrows; i++) inds[i] = i;
          std::vector<FrontPattern> p;
          if (!build_front_patterns(A, starts, inds, 65534, groups > 1 ? 16 : 8, groups, ug, p, pat, out)) continue;
          // what follows the work vector is read in 16-byte pieces (FP64)
          if (p[0].work() % 2 != 0) {
            printf("box %d, %d groups: work vector of %d entries\n", s, groups, p[0].work());
            bad++;
          }
        }
  return bad;
}
