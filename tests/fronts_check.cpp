// Frontal subdomain patterns run on the CPU: the factorisation front by front
// and the solve by its wavefronts' lists, against the known solution.
// Graphs at the edges of the format; both panel layouts; the wavefronts taken
// in both orders, with every entry that is read before it is written a NaN.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>

#include "doug_fronts.hpp"

using namespace doug;
using std::vector;
typedef vector<vector<std::pair<int, double>>> Rows;

static Csr finish(const Rows& rows) {  // diagonally dominant
  Csr A;
  A.nrows = A.ncols = (int)rows.size();
  A.ptr.push_back(0);
  for (int i = 0; i < A.nrows; i++) {
    double d = 0.1;
    for (auto& e : rows[i]) {
      A.col.push_back(e.first);
      A.val.push_back(e.second);
      d -= e.second;
    }
    A.col.push_back(i);
    A.val.push_back(d);
    A.ptr.push_back((int)A.col.size());
  }
  return A;
}

static Csr grid(int nx, int ny, int nz) {
  Rows rows((size_t)nx * ny * nz);
  auto id = [&](int x, int y, int z) { return (x * ny + y) * nz + z; };
  for (int x = 0; x < nx; x++)
    for (int y = 0; y < ny; y++)
      for (int z = 0; z < nz; z++)
        for (int d = 0; d < 3; d++) {
          const int a = x + (d == 0), b = y + (d == 1), c = z + (d == 2);
          if (a >= nx || b >= ny || c >= nz) continue;
          rows[id(x, y, z)].push_back({id(a, b, c), -1.0});
          rows[id(a, b, c)].push_back({id(x, y, z), -1.0});
        }
  return finish(rows);
}

// `deg` random neighbours near each node in its own one of `parts` components;
// with `hub`, node 0 touches every other one
static Csr scattered(int n, int deg, int parts, bool hub) {
  std::mt19937 r(n + deg);
  Rows rows((size_t)n);
  auto link = [&](int i, int j) {
    if (i == j || j < 0 || j >= n) return;
    for (auto& e : rows[i])
      if (e.first == j) return;
    const double v = -1.0 - (double)(r() % 100) / 100.0;
    rows[i].push_back({j, v});
    rows[j].push_back({i, v});
  };
  for (int i = 0; i < n; i++)
    for (int d = 0; d < deg; d++) {
      const int j = (int)((i + r() % std::max(2, n / 20)) % n);
      link(i, j - j % parts + i % parts);
    }
  for (int i = 1; hub && i < n; i++) link(0, i);
  return finish(rows);
}

struct Run {
  const FrontPattern& p;
  vector<double> pan, sch;
  bool dbl;

  int64_t at(const Front& f, int r, int c) const { return f.pan + front_elem(f.k + f.m, r, c, dbl); }

  bool factor(const Csr& A, const vector<int>& pos) {
    pan.assign((size_t)p.elems, 0.0);
    sch.assign((size_t)p.schur, NAN);
    for (int i = 0; i < A.nrows; i++)
      for (int e = A.ptr[i]; e < A.ptr[i + 1]; e++) {
        const int a = pos[i], b = pos[A.col[e]];
        if (b <= a) pan.at((size_t)front_entry(p, b, a, dbl)) = A.val[e];
      }
    for (size_t h = 0; h + 1 < p.hptr.size(); h++)
      for (int i = p.hptr[h]; i < p.hptr[h + 1]; i++) {
        const Front& f = p.fronts[p.hlist[i]];
        const int k = f.k, m = f.m, H = k + m;
        vector<double> X((size_t)H * H, 0.0), D((size_t)k * k, 0.0);
        for (int r = 0; r < H; r++)
          for (int c = 0; c <= std::min(r, k - 1); c++) X[(size_t)r * H + c] = pan.at((size_t)at(f, r, c));
        for (int b = 0; b < 2; b++) {
          if (f.child[b] < 0) continue;
          const Front& q = p.fronts[f.child[b]];
          vector<int> row((size_t)H, -1);
          int found = 0;
          for (int r = 0; r < H; r++) {
            const uint32_t s = p.src[f.row0 + r];
            const int x = (int)(b == 0 ? s & 0xffffu : s >> 16);
            if (x == p.n) continue;
            row[r] = x - q.u;
            found++;
            if (p.rpos[f.row0 + r] != p.rpos[q.row0 + q.k + row[r]]) return false;
          }
          if (found != q.m) return false;  // every row of the child goes somewhere
          for (int r = 0; r < H; r++)
            for (int c = 0; c <= r; c++)
              if (row[r] >= 0 && row[c] >= 0) X[(size_t)r * H + c] += sch.at((size_t)(q.sch + (int64_t)row[r] * q.m + row[c]));
        }
        for (int c = 0; c < k; c++) {
          const double d = std::sqrt(X[(size_t)c * H + c]);
          if (!(d > 0)) return false;
          for (int r = c; r < H; r++) X[(size_t)r * H + c] /= d;
          for (int q = c + 1; q < H; q++)
            for (int r = q; r < H; r++) X[(size_t)r * H + q] -= X[(size_t)r * H + c] * X[(size_t)q * H + c];
        }
        for (int c = 0; c < k; c++)
          for (int r = c; r < k; r++) {
            double s = r == c ? 1.0 : 0.0;
            for (int j = c; j < r; j++) s -= X[(size_t)r * H + j] * D[j * k + c];
            D[r * k + c] = s / X[(size_t)r * H + r];
          }
        for (int r = 0; r < H; r++)
          for (int c = 0; c < (k + 3) / 4 * 4 && c < 4 * (std::min(r, k - 1) / 4 + 1); c++) {
            double s = 0;
            if (r < k)
              s = c <= r ? D[r * k + c] : 0.0;
            else if (c < k)
              for (int j = c; j < k; j++) s += X[(size_t)r * H + j] * D[j * k + c];
            pan.at((size_t)at(f, r, c)) = s;
          }
        for (int r = 0; r < m; r++)
          for (int c = 0; c <= r; c++)
            sch.at((size_t)(f.sch + (int64_t)r * m + c)) = X[(size_t)(k + r) * H + k + c];
      }
    return true;
  }

  // One pass; a wavefront runs to its next barrier before the next one starts.
  void pass(bool fwd, bool reversed, vector<double>& L) const {
    if (p.groups == 1) return walk(fwd, reversed, fwd ? p.units_f : p.units_b, fwd ? p.list_f : p.list_b, L);
    const vector<double> in = L;
    const int n = p.n, nw = (int)p.blist_f.size() / p.groups, apex0 = p.gtop.back();
    auto slot = [&](int q) { return (size_t)(q < p.top0 || fwd ? q : n + q - p.top0); };
    // each group has a work vector of its own: its positions and, backward,
    // the apex's solution; forward it leaves its y and its updates for the apex
    auto subtrees = [&]() {
      const vector<int32_t>& list = fwd ? p.blist_f : p.blist_b;
      for (int g = 0; g < p.groups; g++) {
        vector<double> own(L.size(), NAN);
        for (int q = p.gpos[g]; q < p.gpos[g + 1]; q++) own[q] = in[q];
        for (int q = p.gtop[g]; q < p.gtop[g + 1]; q++) own[q] = in[q];
        if (fwd) own[n] = 0;
        for (int q = apex0; !fwd && q < n; q++) own[slot(q)] = L[slot(q)];
        walk(fwd, reversed, fwd ? p.bunits_f : p.bunits_b,
             vector<int32_t>(list.begin() + g * nw, list.begin() + (g + 1) * nw + 1), own);
        for (int q = p.gpos[g]; q < p.gpos[g + 1]; q++) L[slot(q)] = own[slot(q)];
        for (int q = p.gtop[g]; q < p.gtop[g + 1]; q++) L[slot(q)] = own[slot(q)];
        for (int q = p.uoff[g]; fwd && q < p.uoff[g + 1]; q++) L[p.uidx[q]] = own[p.uidx[q]];
      }
    };
    if (fwd) subtrees();
    walk(fwd, reversed, fwd ? p.units_f : p.units_b, fwd ? p.list_f : p.list_b, L);
    if (!fwd) subtrees();
  }
  void walk(bool fwd, bool reversed, const vector<FrontUnit>& units, const vector<int32_t>& list,
            vector<double>& L) const {
    const int nw = (int)list.size() - 1, n = p.n;
    vector<int> next(list.begin(), list.end() - 1), owed((size_t)nw, 0);
    vector<vector<double>> f((size_t)nw, vector<double>(64, 0.0)), acc(f), y0(f);
    vector<vector<std::pair<int, double>>> late((size_t)nw);
    auto slot = [&](int q) { return (size_t)(q < p.top0 ? q : n + q - p.top0); };
    for (bool busy = true; busy;) {
      busy = false;
      for (int v = 0; v < nw; v++) {
        const int w = reversed ? nw - 1 - v : v;
        while (owed[w] == 0 && next[w] < list[w + 1]) {
          const FrontUnit& u = units[next[w]++];
          const int k = u.k, h = u.h;
          auto entry = [&](int r, int c) { return pan.at((size_t)(u.pan + front_elem(h, r, c, dbl))); };
          auto sums = [&](int r) {
            const uint32_t s = p.src[u.row0 + r];
            return L.at(s & 0xffffu) + L.at(s >> 16);
          };
          auto value = [&](int r) {
            return r < k ? L.at((size_t)(u.c0 + r)) : r < h ? -L.at(slot(p.rpos[u.row0 + r])) : 0.0;
          };
          if (fwd && (u.flags & FU_FIRST))
            for (int c = 0; c < 64; c++) f[w][c] = c < k ? L.at((size_t)(u.c0 + c)) + sums(c) : 0.0;
          if (!fwd && (u.flags & FU_FIRST))
            for (int r = 0; r < 64; r++) y0[w][r] = value(r);
          if (u.flags & FU_BEGIN) acc[w].assign(64, 0.0);
          for (int l = 0; l < 64; l++) {
            const int r = 64 * u.chunk + l;
            const double x = fwd || r >= h ? 0.0 : u.chunk == 0 ? y0[w][l] : value(r);
            for (int c = 4 * u.g0; r < h && c < 4 * u.g1; c++)
              if (r >= c / 4 * 4) {
                if (fwd)
                  acc[w][l] += entry(r, c) * f[w][c];
                else
                  acc[w][c - 4 * u.g0] += entry(r, c) * x;
              }
          }
          if (u.flags & FU_END)
            for (int l = 0; l < 64; l++) {
              const int r = 64 * u.chunk + l, c = 4 * u.g0 + l;
              if (!fwd) {
                if (c < k && c < 4 * u.g1) L.at(slot(u.c0 + c)) = acc[w][l];
              } else if (r < k) {
                if (u.flags & FU_WHOLE)
                  L.at((size_t)(u.c0 + r)) = acc[w][l];
                else
                  late[w].push_back({u.c0 + r, acc[w][l]});
              } else if (r < h) {
                L.at((size_t)(u.u + r - k)) = sums(r) - acc[w][l];
              }
            }
          owed[w] = u.nbar;
        }
        busy = busy || owed[w] > 0 || next[w] < list[w + 1];
      }
      for (int w = 0; w < nw; w++) {
        for (auto& x : late[w]) L.at((size_t)x.first) = x.second;
        late[w].clear();
        if (owed[w] > 0) owed[w]--;
      }
    }
  }
};

static int check(const char* name, const Csr& A, int nw, int groups, int ug) {
  const int n = A.nrows;
  vector<int> starts{0, n}, inds((size_t)n), pat, out, pos((size_t)n);
  for (int i = 0; i < n; i++) inds[i] = i;
  vector<FrontPattern> P;
  if (!build_front_patterns(A, starts, inds, 65535, nw, groups, ug, P, pat, out)) {
    printf("%s: refused\n", name);
    return 1;
  }
  for (int q = 0; q < n; q++) pos[out[q]] = q;
  const FrontPattern& p = P[0];
  if (groups > 1) {  // the groups' positions follow one another, and each lists only its own fronts
    if (p.gpos.front() != 0 || p.gpos.back() != p.top0 || p.gtop.front() != p.top0) return 1;
    for (int w = 0; w < nw * groups; w++)
      for (int i = p.blist_f[w]; i < p.blist_f[w + 1]; i++) {
        const FrontUnit& u = p.bunits_f[i];
        const vector<int32_t>& range = u.c0 < p.top0 ? p.gpos : p.gtop;
        if (u.flags && (u.c0 < range[w / nw] || u.c0 + u.k > range[w / nw + 1])) {
          printf("%s: a front outside its group\n", name);
          return 1;
        }
      }
  }
  for (bool dbl : {true, false}) {
    Run run{p, {}, {}, dbl};
    if (!run.factor(A, pos)) {
      printf("%s: factor\n", name);
      return 1;
    }
    for (bool reversed : {false, true}) {
      vector<double> x((size_t)n), L((size_t)p.work(), NAN);
      for (int i = 0; i < n; i++) x[i] = std::sin(1.0 + i);
      for (int q = 0; q < n; q++) {
        L[q] = 0;
        for (int e = A.ptr[out[q]]; e < A.ptr[out[q] + 1]; e++) L[q] += A.val[e] * x[A.col[e]];
      }
      L[n] = 0;
      run.pass(true, reversed, L);
      for (int q = p.top0; q < n; q++) L[(size_t)(n + q - p.top0)] = NAN;
      run.pass(false, reversed, L);
      double err = 0, norm = 0;
      for (int q = 0; q < n; q++) {
        const double d = L[(size_t)(q < p.top0 ? q : n + q - p.top0)] - x[out[q]];
        err += d * d;
        norm += x[out[q]] * x[out[q]];
      }
      // condition at most 2 max_i a_ii / 0.1 (diagonal dominance by 0.1)
      double dmax = 0;
      for (int i = 0; i < n; i++)
        for (int e = A.ptr[i]; e < A.ptr[i + 1]; e++)
          if (A.col[e] == i) dmax = std::max(dmax, A.val[e]);
      const double bound = 2.3e-16 * n * 20.0 * dmax;
      if (!(std::sqrt(err / norm) <= bound)) {
        printf("%s nw %d groups %d ug %d dbl %d reversed %d: error %g, bound %g\n", name, nw, groups, ug, dbl, reversed,
               std::sqrt(err / norm), bound);
        return 1;
      }
    }
  }
  return 0;
}

int main() {
  int bad = 0;
  for (int cfg = 0; cfg < 9; cfg++) {
    const int nw = cfg == 0 || cfg == 2 ? 8 : 16, ug = cfg == 0 || cfg > 5 ? 8 : 4, groups = cfg < 3 ? 1 : 1 << (cfg < 6 ? cfg - 2 : cfg - 5);
    bad |= check("one node", grid(1, 1, 1), nw, groups, ug);
    bad |= check("two nodes", grid(1, 1, 2), nw, groups, ug);
    bad |= check("line of 33", grid(33, 1, 1), nw, groups, ug);
    bad |= check("line of 1000", grid(1000, 1, 1), nw, groups, ug);
    bad |= check("4 x 4 x 4", grid(4, 4, 4), nw, groups, ug);
    bad |= check("5 x 7 x 9", grid(5, 7, 9), nw, groups, ug);
    bad |= check("14 x 14 x 14", grid(14, 14, 14), nw, groups, ug);
    bad |= check("66 x 66", grid(66, 66, 1), nw, groups, ug);
    bad |= check("2 x 70 x 30", grid(2, 70, 30), nw, groups, ug);
    bad |= check("scattered", scattered(700, 3, 1, false), nw, groups, ug);
    bad |= check("seven components", scattered(900, 2, 7, false), nw, groups, ug);
    bad |= check("many components", scattered(600, 1, 200, false), nw, groups, ug);
    bad |= check("hub", scattered(800, 1, 5, true), nw, groups, ug);
    bad |= check("dense", scattered(200, 150, 1, true), nw, groups, ug);
  }
  // refused, not truncated, where the work vector does not fit
  {
    const Csr A = grid(14, 14, 14);
    vector<int> starts{0, A.nrows}, inds((size_t)A.nrows), pat, out;
    for (int i = 0; i < A.nrows; i++) inds[i] = i;
    vector<FrontPattern> P;
    if (build_front_patterns(A, starts, inds, A.nrows + 10, 8, 1, 8, P, pat, out)) {
      printf("a work vector too long was accepted\n");
      bad = 1;
    }
  }
  printf(bad ? "FAILED\n" : "OK\n");
  return bad;
}
