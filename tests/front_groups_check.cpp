// build_front_patterns with a choice of workgroups: it takes the largest count
// that fits every subdomain, with the patterns that this count gives when asked
// for outright, and refuses where none fits; and its patterns do not depend on
// the matrix's numbering.  Returns the number of failures.
#include "doug_fronts.hpp"

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <string>

using namespace doug;

namespace {

// boxes side by side without coupling, the grid graph of each
Csr boxes(const std::vector<std::vector<int>>& dims, std::vector<int>& starts) {
  Csr A;
  A.ptr.assign(1, 0);
  starts.assign(1, 0);
  for (const std::vector<int>& d : dims) {
    const int base = starts.back();
    auto id = [&](int x, int y, int z) { return base + (x * d[1] + y) * d[2] + z; };
    for (int x = 0; x < d[0]; x++)
      for (int y = 0; y < d[1]; y++)
        for (int z = 0; z < d[2]; z++) {
          for (int a = -1; a <= 1; a += 2) {
            if (x + a >= 0 && x + a < d[0]) A.col.push_back(id(x + a, y, z));
            if (y + a >= 0 && y + a < d[1]) A.col.push_back(id(x, y + a, z));
            if (z + a >= 0 && z + a < d[2]) A.col.push_back(id(x, y, z + a));
          }
          A.col.push_back(id(x, y, z));
          A.ptr.push_back((int)A.col.size());
        }
    starts.push_back(base + d[0] * d[1] * d[2]);
  }
  A.nrows = A.ncols = starts.back();
  A.val.assign(A.col.size(), 1.0);
  return A;
}

template <typename V>
void append(std::string& s, const V& v) {
  s.append(reinterpret_cast<const char*>(v.data()), v.size() * sizeof(v[0]));
  s += '|';
}

// everything a subdomain's set-up and solve read
std::string bytes(const FrontPattern& p) {
  std::string s = std::to_string(p.n) + ' ' + std::to_string(p.top0) + ' ' + std::to_string(p.usz) + ' ' +
                  std::to_string(p.elems) + ' ' + std::to_string(p.schur) + ' ' + std::to_string(p.groups);
  for (const Front& f : p.fronts)
    for (int v : {f.pan, f.row0, f.sch, f.child[0], f.child[1], (int)f.c0, (int)f.k, (int)f.m, (int)f.u})
      s += ' ' + std::to_string(v);
  append(s, p.order), append(s, p.colfront), append(s, p.rpos), append(s, p.src), append(s, p.hptr), append(s, p.hlist);
  for (auto* units : {&p.units_f, &p.units_b, &p.bunits_f, &p.bunits_b})
    for (const FrontUnit& u : *units)
      for (int v : {u.pan, u.row0, (int)u.h, (int)u.k, (int)u.c0, (int)u.u, (int)u.g0, (int)u.g1, (int)u.chunk,
                    (int)u.flags, (int)u.nbar})
        s += ' ' + std::to_string(v);
  append(s, p.list_f), append(s, p.list_b), append(s, p.blist_f), append(s, p.blist_b), append(s, p.gpos);
  append(s, p.gtop), append(s, p.uoff), append(s, p.uidx);
  return s;
}

}  // namespace

int main() {
  int bad = 0;
  for (int ug : {kFrontUnitGroups32, kFrontUnitGroups64}) {
    std::vector<int> starts;
    const Csr A = boxes({{9, 9, 9}, {40, 31, 1}, {12, 12, 12}, {9, 9, 9}, {1, 1, 1}}, starts);
    std::vector<int> inds((size_t)A.nrows);
    for (int i = 0; i < A.nrows; i++) inds[i] = i;
    // work vectors of each count where nothing is refused
    int work[4], limits[10], nl = 0;
    for (int e = 0; e < 4; e++) {
      std::vector<FrontPattern> p;
      std::vector<int> pat, out;
      if (!build_front_patterns(A, starts, inds, 65534, 16, 1 << e, ug, p, pat, out)) return 1;
      work[e] = 0;
      for (const FrontPattern& q : p) work[e] = std::max(work[e], q.work());
      limits[nl++] = work[e];
      limits[nl++] = work[e] - 1;
    }
    limits[nl++] = 65534;
    limits[nl++] = A.nrows / 4;
    for (int l = 0; l < nl; l++)
      for (int most : {1, 2, 4, 8}) {
        int expect = 0, chosen = -1;
        for (int e = 0; e < 4; e++)
          if (1 << e <= most && work[e] <= limits[l]) expect = 1 << e;
        std::vector<FrontPattern> p, q;
        std::vector<int> pat, out, pat2, out2;
        const bool ok = build_front_patterns(A, starts, inds, limits[l], 16, most, ug, p, pat, out, &chosen);
        if (ok != (expect > 0) || (ok && chosen != expect)) {
          printf("limit %d, at most %d: %d groups, expected %d\n", limits[l], most, ok ? chosen : 0, expect);
          bad++;
          continue;
        }
        if (!ok) continue;
        if (!build_front_patterns(A, starts, inds, limits[l], 16, expect, ug, q, pat2, out2)) return 1;
        bool same = out == out2;
        for (size_t b = 0; b < pat.size(); b++) same = same && bytes(p[pat[b]]) == bytes(q[pat2[b]]);
        if (!same) {
          printf("limit %d, at most %d: other patterns than %d groups asked for outright\n", limits[l], most, expect);
          bad++;
        }
      }
  }
  // other numbers for the nodes, in reverse and scattered over four times as
  // many rows, leave the local graphs and so the patterns as they are
  {
    std::vector<int> starts;
    const Csr A = boxes({{7, 8, 9}, {1, 1, 1}, {30, 21, 1}, {7, 8, 9}, {2, 3, 4}}, starts);
    const int n = A.nrows;
    std::vector<int> inds((size_t)n);
    for (int i = 0; i < n; i++) inds[i] = i;
    for (int way = 0; way < 2; way++) {
      Csr B;
      B.nrows = B.ncols = 4 * n;
      std::vector<int> to((size_t)n), from((size_t)(4 * n), -1);
      for (int i = 0; i < n; i++) to[i] = way == 0 ? 4 * n - 1 - i : (int)((int64_t)i * 1031 % n) * 4 + 3;
      for (int i = 0; i < n; i++) from[to[i]] = i;
      B.ptr.assign(1, 0);
      for (int i = 0; i < 4 * n; i++) {
        if (from[i] >= 0)
          for (int e = A.ptr[from[i]]; e < A.ptr[from[i] + 1]; e++) B.col.push_back(to[A.col[e]]);
        else  // rows of no subdomain, with neighbours in several
          for (int c = 0; c < 3; c++) B.col.push_back((i + c) % (4 * n));
        B.ptr.push_back((int)B.col.size());
      }
      B.val.assign(B.col.size(), 1.0);
      std::vector<FrontPattern> p, q;
      std::vector<int> pat, out, pat2, out2;
      if (!build_front_patterns(A, starts, inds, 65534, 16, 2, 8, p, pat, out) ||
          !build_front_patterns(B, starts, to, 65534, 16, 2, 8, q, pat2, out2))
        return 1;
      bool same = true;
      for (int i = 0; i < n; i++) same = same && to[out[i]] == out2[i];
      for (size_t b = 0; b < pat.size(); b++) same = same && bytes(p[pat[b]]) == bytes(q[pat2[b]]);
      if (!same) {
        printf("numbering %d: other patterns\n", way);
        bad++;
      }
    }
  }
  return bad;
}
