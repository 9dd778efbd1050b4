// Nested dissection, fronts and solve schedule of the subdomain factors
// (doug_fronts.hpp).  Separators are levels of a breadth-first search from a
// pseudo-peripheral node (A. George, J. Liu, Computer Solution of Large
// Sparse Positive Definite Systems, 1981, ch. 8), which needs no coordinates;
// a part of at most kLeaf nodes becomes one dense front.  Independent of the
// thread count: a subdomain's pattern depends on its local graph alone.
#include "doug_fronts.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>
#include <unordered_map>

namespace doug {

namespace {

constexpr int kLeaf = 32;

struct Graph {
  std::vector<int> ptr, adj;
  int n() const { return (int)ptr.size() - 1; }
};

uint64_t mix(uint64_t x) {
  x ^= x >> 31;
  x *= 0x9e3779b97f4a7c15ull;
  x ^= x >> 29;
  x *= 0xd1342543de82ef95ull;
  return x ^ (x >> 32);
}

// A node of the dissection tree: its own nodes (a separator, or a leaf part)
// and up to two subtrees.
struct Part {
  int first, count;  // slice of Dissector::listed
  int child[2];
};

struct Dissector {
  const Graph& g;
  std::vector<int> verts, tmp, lab, mark, bfs, lev, listed, comp;
  std::vector<Part> parts;
  int stamp = 0, nlab = 0;

  explicit Dissector(const Graph& g_) : g(g_) {
    const int n = g.n();
    verts.resize((size_t)n);
    tmp.resize((size_t)n);
    for (int v = 0; v < n; v++) verts[v] = v;
    lab.assign((size_t)n, 0);
    mark.assign((size_t)n, 0);
    bfs.resize((size_t)n + 1);
    listed.reserve((size_t)n);
  }

  // breadth-first order from root inside part `id`; lev holds the starts of
  // its levels and the end.  What is found loses its label until the end: one
  // array to look up for each edge (a mark beside the label, without branches,
  // took 1.4 times as long).
  int search(int root, int id) {
    ++stamp;
    int* q = bfs.data();
    int* lb = lab.data();
    const int* ptr = g.ptr.data();
    const int* adj = g.adj.data();
    q[0] = root;
    lb[root] = -2;
    int b = 0, top = 1;
    lev.clear();
    lev.push_back(0);
    while (true) {
      const int e = top;
      for (int k = b; k < e; k++) {
        const int v = q[k];
        for (int p = ptr[v]; p < ptr[v + 1]; p++) {
          const int u = adj[p];
          if (lb[u] == id) {
            lb[u] = -2;
            q[top++] = u;
          }
        }
      }
      lev.push_back(e);
      if (top == e) break;
      b = e;
    }
    for (int k = 0; k < top; k++) {
      lb[q[k]] = id;
      mark[q[k]] = stamp;
    }
    return top;
  }

  int leaf(int b, int e) {
    std::sort(verts.begin() + b, verts.begin() + e);
    Part p{(int)listed.size(), e - b, {-1, -1}};
    listed.insert(listed.end(), verts.begin() + b, verts.begin() + e);
    parts.push_back(p);
    return (int)parts.size() - 1;
  }

  // verts[b, e), all labelled `id`.  With `known`, the first `known` of them
  // are what search(verts[b], id) finds, in its order, and lev holds its levels.
  int run(int b, int e, int id, int known = 0) {
    const int n = e - b;
    if (n <= kLeaf) return leaf(b, e);
    int reached = known;
    if (known > 0) {
      ++stamp;
      std::copy(verts.begin() + b, verts.begin() + b + known, bfs.begin());
      for (int k = 0; k < known; k++) mark[bfs[k]] = stamp;
    } else {
      reached = search(verts[b], id);
    }
    int na = 0, nb = 0, nc = n;  // nc: nodes of the component to cut
    int near = 0;                // nodes before the separator
    std::vector<int> sep, rest;
    comp.clear();
    if (reached < n) {
      // several components: cut the largest if it holds most of the nodes,
      // the others go to the lighter side; else share them out
      const int first = stamp;
      int big = verts[b];
      nc = reached;
      comp.push_back(reached);
      rest.assign(bfs.begin(), bfs.begin() + reached);
      for (int k = b; k < e; k++)
        if (mark[verts[k]] < first) {
          const int r = search(verts[k], id);
          if (r > nc) nc = r, big = verts[k];
          comp.push_back(r);
          rest.insert(rest.end(), bfs.begin(), bfs.begin() + r);
        }
      if (2 * nc > n && nc > kLeaf) {
        reached = search(big, id);
        const int s = stamp;
        size_t at = 0, to = 0, kept = 0;
        for (int r : comp) {
          if (mark[rest[at]] != s) {
            std::copy(rest.begin() + at, rest.begin() + at + r, rest.begin() + to);
            to += r;
            comp[kept++] = r;
          }
          at += r;
        }
        rest.resize(to);
        comp.resize(kept);
      } else {
        nc = 0;
      }
    }
    if (nc > 0) {
      // from a low-degree node of the last level; once more while it grows
      int nl = (int)lev.size();
      for (int round = 0; round < 3; round++) {
        int cand = -1, deg = 0;
        for (int k = lev[lev.size() - 2]; k < reached; k++) {
          const int v = bfs[k], d = g.ptr[v + 1] - g.ptr[v];
          if (cand < 0 || d < deg || (d == deg && v < cand)) cand = v, deg = d;
        }
        search(cand, id);
        if ((int)lev.size() <= nl) break;
        nl = (int)lev.size();
      }
      const int levels = (int)lev.size() - 1;
      if (levels < 3) return leaf(b, e);
      // the smallest level, weighted by the sides' imbalance, that leaves each
      // side at least 27 % of the nodes; else the level at the middle
      int best = -1;
      int64_t score = 0;
      for (int k = 1; k + 1 < levels; k++) {
        const int64_t a = lev[k], c = nc - lev[k + 1], s = lev[k + 1] - lev[k];
        if (100 * std::min(a, c) < 27 * (int64_t)nc) continue;
        const int64_t sc = s * (2 * nc + (a > c ? a - c : c - a));
        if (best < 0 || sc < score) best = k, score = sc;
      }
      if (best < 0) {
        best = 1;
        while (best + 2 < levels && lev[best + 1] < nc / 2) best++;
      }
      // level `best` without its nodes that touch only the nearer side
      const int l0 = lev[best], l1 = lev[best + 1];
      for (int k = l1; k < nc; k++) tmp[nb++] = bfs[k];
      ++stamp;
      for (int k = 0; k < nb; k++) mark[tmp[k]] = stamp;
      for (int k = 0; k < l0; k++) verts[b + na++] = bfs[k];
      for (int k = l0; k < l1; k++) {
        const int v = bfs[k];
        bool far = false;
        for (int p = g.ptr[v]; p < g.ptr[v + 1] && !far; p++) far = mark[g.adj[p]] == stamp;
        if (far)
          sep.push_back(v);
        else
          verts[b + na++] = v;
      }
      for (int v : sep) lab[v] = -1;
      // the nearer side's own search from the same root goes over the same
      // levels, the last one without the separator
      near = na;
      lev.resize((size_t)best + 1);
      if (near > l0) lev.push_back(near);
    }
    {  // the components that were not cut: the next one to the lighter side
      size_t at = 0;
      for (int r : comp) {
        if (na <= nb) {
          std::copy(rest.begin() + at, rest.begin() + at + r, verts.begin() + b + na);
          na += r;
        } else {
          std::copy(rest.begin() + at, rest.begin() + at + r, tmp.begin() + nb);
          nb += r;
        }
        at += r;
      }
      std::copy(tmp.begin(), tmp.begin() + nb, verts.begin() + b + na);
    }
    const int ia = ++nlab, ib = ++nlab;
    for (int k = b; k < b + na; k++) lab[verts[k]] = ia;
    for (int k = b + na; k < b + na + nb; k++) lab[verts[k]] = ib;
    const int mid = b + na, end = mid + nb;
    const int ca = run(b, mid, ia, near), cb = nb > 0 ? run(mid, end, ib) : -1;
    std::sort(sep.begin(), sep.end());
    Part p{(int)listed.size(), (int)sep.size(), {ca, cb}};
    listed.insert(listed.end(), sep.begin(), sep.end());
    parts.push_back(p);
    return (int)parts.size() - 1;
  }
};

// First-fit space for update vectors and matrices.
struct Space {
  std::vector<std::pair<int64_t, int64_t>> hole;  // [first, last)
  int64_t top = 0;
  int64_t take(int64_t n) {
    if (n == 0) return 0;
    for (size_t k = 0; k < hole.size(); k++)
      if (hole[k].second - hole[k].first >= n) {
        const int64_t at = hole[k].first;
        hole[k].first += n;
        if (hole[k].first == hole[k].second) hole.erase(hole.begin() + k);
        return at;
      }
    if (!hole.empty() && hole.back().second == top) {  // grow the last hole
      const int64_t at = hole.back().first;
      hole.pop_back();
      top = at + n;
      return at;
    }
    const int64_t at = top;
    top += n;
    return at;
  }
  void give(int64_t at, int64_t n) {
    if (n == 0) return;
    auto it = std::lower_bound(hole.begin(), hole.end(), std::make_pair(at, at));
    it = hole.insert(it, {at, at + n});
    if (it + 1 != hole.end() && it->second == (it + 1)->first) {
      it->second = (it + 1)->second;
      it = hole.erase(it + 1) - 1;
    }
    if (it != hole.begin() && (it - 1)->second == it->first) {
      (it - 1)->second = it->second;
      hole.erase(it);
    }
  }
};

// cost of a front in the solve: its units (a unit costs what its loads do,
// filled or not)
int64_t front_cost(const Front& f, int ug) {
  return (int64_t)((f.k + f.m + 63) / 64) * std::max(1, (f.k + 4 * ug - 1) / (4 * ug));
}

// A share of a front: 64-row chunks (forward) or column groups (backward).
struct Item {
  int front, first, count;
};

// Items phase by phase and wavefront by wavefront.
struct ItemLists {
  int nw;
  std::vector<std::vector<Item>> cell;
  std::vector<Item>& at(size_t phase, int w) {
    if (cell.size() < (phase + 1) * nw) cell.resize((phase + 1) * nw);
    return cell[phase * nw + (size_t)w];
  }
  // each wavefront's units, a barrier behind each phase, appended
  void flatten(const std::vector<Front>& F, int ug, bool fwd, std::vector<FrontUnit>& units,
               std::vector<int32_t>& list) const {
    if (list.empty()) list.push_back(0);
    const size_t phases = cell.size() / nw;
    for (int w = 0; w < nw; w++) {
      const size_t first = units.size();
      auto barrier = [&]() {
        if (units.size() == first) {
          FrontUnit u{};
          u.h = F[0].k + F[0].m;
          u.g1 = 1;
          units.push_back(u);
        }
        units.back().nbar++;
      };
      for (size_t p = 0; p < phases; p++) {
        for (const Item& it : cell[p * nw + w]) {
          const Front& f = F[it.front];
          const int h = f.k + f.m, nch = (h + 63) / 64, ng = f.k > 0 ? (f.k + 3) / 4 : 1;
          FrontUnit u{};
          u.pan = f.pan;
          u.row0 = f.row0;
          u.h = (uint16_t)h;
          u.k = f.k;
          u.c0 = f.c0;
          u.u = f.u;
          bool start = true;
          auto put = [&](int chunk, int g0, int g1, bool begin, bool end) {
            u.chunk = (uint8_t)chunk;
            u.g0 = (uint8_t)g0;
            u.g1 = (uint8_t)g1;
            u.flags = (start ? FU_FIRST : 0) | (begin ? FU_BEGIN : 0) | (end ? FU_END : 0) |
                      (fwd && it.count == nch ? FU_WHOLE : 0);
            start = false;
            units.push_back(u);
          };
          if (fwd) {
            for (int c = it.first; c < it.first + it.count; c++)
              for (int g = 0; g < ng; g += ug) put(c, g, std::min(ng, g + ug), g == 0, g + ug >= ng);
          } else {
            const int hi = it.first + it.count;
            for (int g = it.first; g < hi; g += ug)
              for (int c = 0; c < nch; c++) put(c, g, std::min(hi, g + ug), c == 0, c + 1 == nch);
          }
        }
        barrier();
      }
      if ((units.size() - first) % 2 == 1) {  // the kernel takes two a turn
        FrontUnit u = units.back();
        u.flags = 0;
        u.nbar = 0;
        units.push_back(u);
      }
      list.push_back((int32_t)units.size());
    }
  }
};

// The fronts of a graph in postorder and their boundary rows (in postorder
// positions), whatever the work vector and the number of workgroups.
struct Tree {
  std::vector<int> listed;  // position -> node
  std::vector<Front> fronts;
  std::vector<int> parent;
  std::vector<uint16_t> rows;  // front f's: rptr[f] ..
  std::vector<int> rptr;
};

// False where a front or the graph exceeds the format.
bool make_tree(const Graph& g, Tree& T) {
  const int n = g.n();
  if (n > 65535) return false;
  Dissector D(g);
  D.run(0, n, 0);
  // fronts in postorder, at most kFrontCols columns each: a longer separator
  // becomes a chain, cut into equal pieces
  std::vector<int> part_front(D.parts.size(), -1);  // last front of each part
  std::vector<int>& parent = T.parent;
  std::vector<Front>& F = T.fronts;
  for (size_t q = 0; q < D.parts.size(); q++) {
    const Part& p = D.parts[q];
    int kid[2] = {-1, -1}, nk = 0;
    for (int c : p.child)
      if (c >= 0 && part_front[c] >= 0) kid[nk++] = part_front[c];
    const int pieces = std::max(1, (p.count + kFrontCols - 1) / kFrontCols);
    for (int s = 0; s < pieces; s++) {
      const int b = (int)((int64_t)p.count * s / pieces), e = (int)((int64_t)p.count * (s + 1) / pieces);
      Front f{};
      f.c0 = (uint16_t)(p.first + b);
      f.k = (uint16_t)(e - b);
      f.child[0] = s == 0 ? kid[0] : (int)F.size() - 1;
      f.child[1] = s == 0 ? kid[1] : -1;
      for (int c : f.child)
        if (c >= 0) parent[c] = (int)F.size();
      F.push_back(f);
      parent.push_back(-1);
    }
    part_front[q] = (int)F.size() - 1;
  }
  const int nf = (int)F.size();
  if (nf > 65535) return false;
  // boundary rows in postorder positions: the children's and the columns'
  // later neighbours, as bit sets
  std::vector<int> pos((size_t)n);
  for (int p = 0; p < n; p++) pos[D.listed[p]] = p;
  const int words = (n + 63) / 64;
  std::vector<uint16_t>& rows = T.rows;
  std::vector<int>& rptr = T.rptr;
  rptr.assign(1, 0);
  std::vector<uint64_t> bits((size_t)words);
  for (int f = 0; f < nf; f++) {
    const int c0 = F[f].c0, c1 = c0 + F[f].k;
    std::fill(bits.begin() + c0 / 64, bits.end(), 0);
    for (int c : F[f].child)
      if (c >= 0) {
        for (int i = rptr[c]; i < rptr[c + 1]; i++) bits[rows[i] >> 6] |= 1ull << (rows[i] & 63);
      }
    for (int p = c0; p < c1; p++) {
      const int v = D.listed[p];
      for (int e = g.ptr[v]; e < g.ptr[v + 1]; e++) {
        const int r = pos[g.adj[e]];
        if (r >= c1) bits[r >> 6] |= 1ull << (r & 63);
      }
    }
    for (int w = c1 / 64; w < words; w++) {
      uint64_t x = bits[w];
      if (w == c1 / 64) x &= ~0ull << (c1 & 63);
      for (; x; x &= x - 1) rows.push_back((uint16_t)(64 * w + __builtin_ctzll(x)));
    }
    const int m = (int)rows.size() - rptr[f];
    rptr.push_back((int)rows.size());
    if ((int)F[f].k + m > 64 * 250) return false;
    F[f].m = (uint16_t)m;
  }
  T.listed.swap(D.listed);
  return true;
}

// The pattern of `groups` workgroups of nw wavefronts; false where its work
// vector or panels do not fit.
bool make_pattern(const Tree& T, int64_t max_work, int nw, int groups, int ug, FrontPattern& P) {
  P = FrontPattern{};
  const int n = (int)T.listed.size(), nwb = nw * groups;  // nwb wavefronts for the bottom subtrees
  P.n = n;
  P.groups = groups;
  P.fronts = T.fronts;
  std::vector<Front>& F = P.fronts;
  const int nf = (int)F.size();
  const std::vector<int>& parent = T.parent;
  std::vector<int64_t> cost((size_t)nf);
  for (int f = 0; f < nf; f++) {
    cost[f] = front_cost(F[f], ug);
    for (int c : F[f].child)
      if (c >= 0) cost[f] += cost[c];
  }
  auto heavier = [&](int a, int b) { return cost[a] != cost[b] ? cost[a] > cost[b] : a < b; };
  // Cuts the subtrees at `roots` until `ways` shares differ by less than
  // num / den of their mean, or `most` subtrees: share[f] of each that is left,
  // cut[f] = mark of the fronts above them.
  auto cut_up = [&](std::vector<int>& roots, int ways, int num, int den, int most, std::vector<char>& cut,
                    std::vector<int>& share) {
    while (true) {
      std::sort(roots.begin(), roots.end(), heavier);
      int64_t load[kFrontWavesMax] = {}, sum = 0;
      for (int f : roots) {
        int w = 0;
        for (int q = 1; q < ways; q++)
          if (load[q] < load[w]) w = q;
        load[w] += cost[f];
        share[f] = w;
        sum += cost[f];
      }
      const int64_t worst = *std::max_element(load, load + ways);
      if (roots.empty() || den * ways * worst <= num * sum || (int)roots.size() >= most) break;
      const int f = roots.front();
      if (F[f].child[0] < 0 && F[f].child[1] < 0) break;  // a leaf is the heaviest
      cut[f] = 1;
      roots.erase(roots.begin());
      for (int c : F[f].child)
        if (c >= 0) roots.push_back(c);
    }
  };
  // groups: whole subtrees each; the apex above them is the last workgroup's
  std::vector<int> group((size_t)nf, 0), wave((size_t)nf, 0);
  std::vector<char> apex((size_t)nf, 0), top((size_t)nf, 0), is_root((size_t)nf, 0);
  std::vector<int> all_roots;
  for (int f = 0; f < nf; f++)
    if (parent[f] < 0) all_roots.push_back(f);
  if (groups > 1) cut_up(all_roots, groups, 12, 10, 4 * groups, apex, group);
  std::vector<std::vector<int>> roots((size_t)groups);
  for (int f : all_roots) roots[group[f]].push_back(f);
  for (int f = nf - 1; f >= 0; f--)
    if (!apex[f] && parent[f] >= 0 && !apex[parent[f]]) group[f] = group[parent[f]];
  // in a group: bottom subtrees, one wavefront each; what is above them goes
  // level by level
  for (auto& r : roots) {
    cut_up(r, nw, 11, 10, 6 * nw, top, wave);
    for (int f : r) is_root[f] = 1;
  }
  // new numbering: the groups' bottom subtrees in postorder, then their top
  // fronts by level, then the apex by level
  std::vector<int> seq, height((size_t)nf, 0), level((size_t)nf, -1);
  for (int f = nf - 1; f >= 0; f--)  // a bottom front runs with its subtree's root
    if (!apex[f] && !top[f] && !is_root[f]) wave[f] = wave[parent[f]];
  std::vector<int> levels((size_t)groups + 1, 0);  // of each group, of the apex
  for (int f = 0; f < nf; f++) {
    const bool up = top[f] || apex[f];
    if (up) level[f] = 0;
    for (int c : F[f].child)
      if (c >= 0) {
        height[f] = std::max(height[f], height[c] + 1);
        if (up && (top[c] || apex[c]) && apex[f] == apex[c]) level[f] = std::max(level[f], level[c] + 1);
      }
    int& l = levels[apex[f] ? groups : group[f]];
    if (up) l = std::max(l, level[f] + 1);
  }
  std::vector<int> first_of(2 * (size_t)groups + 2, 0);  // fronts: bottoms of group g, tops of group g, apex, end
  for (int q = 0; q < groups; q++) {
    first_of[q] = (int)seq.size();
    for (int f = 0; f < nf; f++)
      if (!apex[f] && !top[f] && group[f] == q) seq.push_back(f);
  }
  const int nbottom = (int)seq.size();
  for (int q = 0; q < groups; q++) {
    first_of[groups + q] = (int)seq.size();
    for (int l = 0; l < levels[q]; l++)
      for (int f = 0; f < nf; f++)
        if (top[f] && group[f] == q && level[f] == l) seq.push_back(f);
  }
  first_of[2 * groups] = (int)seq.size();
  for (int l = 0; l < levels[groups]; l++)
    for (int f = 0; f < nf; f++)
      if (apex[f] && level[f] == l) seq.push_back(f);
  first_of[2 * groups + 1] = nf;
  std::vector<int> newid((size_t)nf), newpos((size_t)n);
  P.order.resize((size_t)n);
  P.colfront.resize((size_t)n);
  {
    int at = 0;
    for (int q = 0; q < nf; q++) {
      const Front& f = F[seq[q]];
      newid[seq[q]] = q;
      if (q == nbottom) P.top0 = at;
      for (int c = 0; c < f.k; c++) {
        newpos[f.c0 + c] = at;
        P.colfront[at] = (uint16_t)q;
        P.order[at++] = T.listed[f.c0 + c];
      }
    }
    if (nbottom == nf) P.top0 = n;
  }
  std::vector<Front> G((size_t)nf);
  P.rpos.reserve(T.rows.size() + (size_t)n);
  std::vector<int> lv((size_t)nf), wv((size_t)nf), hv((size_t)nf);
  int at = 0;
  int64_t elems = 0, recs = 0;
  for (int q = 0; q < nf; q++) {
    const int o = seq[q];
    Front f = F[o];
    f.c0 = (uint16_t)at;
    at += f.k;
    for (int& c : f.child) c = c >= 0 ? newid[c] : -1;
    f.pan = (int32_t)elems;
    f.row0 = (int32_t)recs;
    elems += front_panel_elems(f.k, f.m);
    recs += f.k + f.m;
    if (elems > INT32_MAX || recs > INT32_MAX) return false;
    // ancestors keep their relative order, so the rows stay ascending
    for (int c = 0; c < f.k; c++) P.rpos.push_back((uint16_t)(f.c0 + c));
    for (int r = T.rptr[o]; r < T.rptr[o + 1]; r++) P.rpos.push_back((uint16_t)newpos[T.rows[r]]);
    lv[q] = level[o];
    wv[q] = group[o] * nw + wave[o];
    hv[q] = height[o];
    G[q] = f;
  }
  F.swap(G);
  P.elems = elems;
  // update vectors: each wavefront's bottom fronts use a space of their own,
  // one after the other; the top levels share what is free by then
  std::vector<int64_t> u((size_t)nf, 0);
  Space space;
  space.take(1);  // the zero entry
  {
    Space own[kFrontWavesMax * kFrontGroupsMax];
    for (int q = 0; q < nbottom; q++) {
      Space& s = own[wv[q]];
      u[q] = s.take(F[q].m);
      for (int c : F[q].child)
        if (c >= 0) s.give(u[c], F[c].m);
    }
    for (int w = 0; w < nwb; w++) {
      const int64_t b = space.top;
      space.top += own[w].top;
      for (auto& h : own[w].hole) space.give(b + h.first, h.second - h.first);
      for (int q = 0; q < nbottom; q++)
        if (wv[q] == w) u[q] += b;
    }
    for (int q = nbottom; q < nf;) {
      int e = q;
      while (e < nf && lv[e] == lv[q]) e++;  // (of two groups, too)
      for (int f = q; f < e; f++) u[f] = space.take(F[f].m);
      for (int f = q; f < e; f++)
        for (int c : F[f].child)
          if (c >= 0) space.give(u[c], F[c].m);
      q = e;
    }
  }
  P.usz = (int)std::max<int64_t>(space.top, n - P.top0 + 1);
  P.usz += (n + P.usz) % 2;  // what lies behind the work vector in LDS is read in 16-byte pieces
  if ((int64_t)n + P.usz > std::min<int64_t>(max_work, 65535)) return false;
  for (int q = 0; q < nf; q++) F[q].u = (uint16_t)(n + u[q]);
  // row records
  P.src.resize((size_t)recs);
  for (int q = 0; q < nf; q++) {
    const Front& f = F[q];
    const uint16_t* rp = P.rpos.data() + f.row0;
    uint32_t* sr = P.src.data() + f.row0;
    const int h = f.k + f.m;
    for (int r = 0; r < h; r++) sr[r] = (uint32_t)n | (uint32_t)n << 16;
    for (int b = 0; b < 2; b++) {
      const int c = f.child[b];
      if (c < 0) continue;
      const uint16_t* rc = P.rpos.data() + F[c].row0 + F[c].k;
      int r = 0;
      for (int j = 0; j < F[c].m; j++) {  // both ascending
        while (rp[r] != rc[j]) r++;
        const uint32_t idx = (uint32_t)F[c].u + (uint32_t)j;
        sr[r] = b == 0 ? (sr[r] & 0xffff0000u) | idx : (sr[r] & 0xffffu) | idx << 16;
      }
    }
  }
  // update matrices of the factorisation, freed once the parent's height is done
  int heights = 0;
  for (int q = 0; q < nf; q++) heights = std::max(heights, hv[q] + 1);
  P.hptr.assign((size_t)heights + 1, 0);
  for (int q = 0; q < nf; q++) P.hptr[hv[q] + 1]++;
  for (int h = 0; h < heights; h++) P.hptr[h + 1] += P.hptr[h];
  P.hlist.resize((size_t)nf);
  {
    std::vector<int> fill(P.hptr.begin(), P.hptr.end() - 1);
    for (int q = 0; q < nf; q++) P.hlist[fill[hv[q]]++] = (uint16_t)q;
    Space sp;
    for (int h = 0; h < heights; h++) {
      for (int i = P.hptr[h]; i < P.hptr[h + 1]; i++) {
        const Front& f = F[P.hlist[i]];
        const int64_t o = sp.take((int64_t)f.m * f.m);
        if (o + (int64_t)f.m * f.m > INT32_MAX) return false;
        F[P.hlist[i]].sch = (int32_t)o;
      }
      for (int i = P.hptr[h]; i < P.hptr[h + 1]; i++)
        for (int c : F[P.hlist[i]].child)
          if (c >= 0) sp.give(F[c].sch, (int64_t)F[c].m * F[c].m);
    }
    P.schur = sp.top;
  }
  // work lists
  auto rows_of = [&](int f) { return (F[f].k + F[f].m + 63) / 64; };
  auto put = [&](ItemLists& l, size_t phase, int w, int f, int first, int count) {
    if (count > 0) l.at(phase, w).push_back(Item{f, first, count});
  };
  // the fronts [from, to), one level after the other from phase `first` on,
  // backward the other way round from phase 0
  auto put_levels = [&](ItemLists& fw, ItemLists& bw, int from, int to, size_t first, int count) {
    for (int q = from; q < to;) {
      int e = q;
      while (e < to && lv[e] == lv[q]) e++;
      const size_t pf = (size_t)lv[q] + first, pb = (size_t)(count - 1 - lv[q]);
      std::vector<int> byw;
      for (int f = q; f < e; f++) byw.push_back(f);
      std::sort(byw.begin(), byw.end(), [&](int a, int b) {
        const int64_t x = front_cost(F[a], ug), y = front_cost(F[b], ug);
        return x != y ? x > y : a < b;
      });
      fw.at(pf, 0);
      bw.at(pb, 0);
      if (e - q >= nw) {  // whole fronts, heaviest first to the least loaded
        int64_t load[kFrontWavesMax] = {};
        for (int f : byw) {
          int w = 0;
          for (int x = 1; x < nw; x++)
            if (load[x] < load[w]) w = x;
          load[w] += front_cost(F[f], ug);
          put(fw, pf, w, f, 0, rows_of(f));
          put(bw, pb, w, f, 0, (F[f].k + 3) / 4);
        }
      } else {  // each front split over its share of the wavefronts
        int w0 = 0;
        const int cnt = e - q;
        for (int i = 0; i < cnt; i++) {
          const int share = nw / cnt + (i < nw % cnt ? 1 : 0), f = byw[i];
          const int nc = rows_of(f), ng = (F[f].k + 3) / 4;
          for (int x = 0; x < share; x++) {
            const int b = nc * x / share, c = nc * (x + 1) / share, gb = ng * x / share, gc = ng * (x + 1) / share;
            put(fw, pf, w0 + x, f, b, c - b);
            put(bw, pb, w0 + x, f, gb, gc - gb);
          }
          w0 += share;
        }
      }
      q = e;
    }
  };
  for (int g = 0; g < groups; g++) {
    ItemLists fw{nw, {}}, bw{nw, {}};
    for (int q = first_of[g]; q < (g + 1 < groups ? first_of[g + 1] : nbottom); q++)
      put(fw, 0, wv[q] - g * nw, q, 0, rows_of(q));
    put_levels(fw, bw, first_of[groups + g], first_of[groups + g + 1], 1, levels[g]);
    for (int q = (g + 1 < groups ? first_of[g + 1] : nbottom) - 1; q >= first_of[g]; q--)
      put(bw, (size_t)levels[g], wv[q] - g * nw, q, 0, (F[q].k + 3) / 4);
    fw.at((size_t)levels[g], 0);
    bw.at((size_t)levels[g], 0);
    fw.flatten(F, ug, true, groups > 1 ? P.bunits_f : P.units_f, groups > 1 ? P.blist_f : P.list_f);
    bw.flatten(F, ug, false, groups > 1 ? P.bunits_b : P.units_b, groups > 1 ? P.blist_b : P.list_b);
  }
  if (groups > 1) {
    ItemLists fw{nw, {}}, bw{nw, {}};
    put_levels(fw, bw, first_of[2 * groups], nf, 0, levels[groups]);
    fw.flatten(F, ug, true, P.units_f, P.list_f);
    bw.flatten(F, ug, false, P.units_b, P.list_b);
    auto position = [&](int q) { return q < nf ? (int)F[q].c0 : n; };
    for (int q = 0; q <= groups; q++) {
      P.gpos.push_back(q < groups ? position(first_of[q]) : P.top0);
      P.gtop.push_back(position(first_of[groups + q]));
    }
    P.uoff.assign(1, 0);
    for (int g = 0; g < groups; g++) {
      for (int q = first_of[2 * groups]; q < nf; q++)
        for (int c : F[q].child)
          if (c >= 0 && c < first_of[2 * groups] && wv[c] / nw == g)
            for (int r = 0; r < F[c].m; r++) P.uidx.push_back((uint16_t)(F[c].u + r));
      P.uoff.push_back((int32_t)P.uidx.size());
    }
  }
  return true;
}

// Local graph of block [s0, s0 + s): neighbours inside the block, without
// self loops, symmetric (reverse edges are added where the matrix lacks
// them, and `mirrored` is set); returns a hash of it.  `floc` is scratch, -1 between calls: it spans
// the block's numbers alone, which for a box of a grid is a small part of the
// matrix's (a whole array per thread costs more page faults than work).
uint64_t local_graph(const Csr& A, const int* inds, int s, std::vector<int>& floc, Graph& g, bool& mirrored) {
  const int first = s > 0 ? *std::min_element(inds, inds + s) : 0;
  const int span = s > 0 ? *std::max_element(inds, inds + s) - first + 1 : 0;  // floc[span]: outside
  if (floc.size() <= (size_t)span) floc.assign((size_t)span + 1, -1);
  for (int li = 0; li < s; li++) floc[inds[li] - first] = li;
  g.ptr.assign((size_t)s + 1, 0);
  size_t cap = 0;
  for (int li = 0; li < s; li++) cap += (size_t)(A.ptr[inds[li] + 1] - A.ptr[inds[li]]);
  g.adj.resize(cap + 1);
  int* adj = g.adj.data();
  const int* col = A.col.data();
  int top = 0;
  uint64_t fwd = 0, rev = 0, hash = (uint64_t)s;
  for (int li = 0; li < s; li++) {
    const int gi = inds[li], b = top;
    for (int p = A.ptr[gi]; p < A.ptr[gi + 1]; p++) {
      const int lj = floc[std::min((unsigned)(col[p] - first), (unsigned)span)];
      adj[top] = lj;
      top += (lj >= 0) & (lj != li);
    }
    g.ptr[li + 1] = top;
    for (int k = b; k < top; k++) {
      const uint64_t a = (uint64_t)li << 32 | (uint32_t)adj[k], c = (uint64_t)adj[k] << 32 | (uint32_t)li;
      const uint64_t m = mix(a);
      fwd += m;
      rev += mix(c);
      hash = (hash ^ m) * 0x9e3779b97f4a7c15ull;
    }
  }
  for (int li = 0; li < s; li++) floc[inds[li] - first] = -1;
  g.adj.resize((size_t)top);
  mirrored = fwd != rev;
  if (mirrored) {  // unsymmetric structure: every edge in both directions
    Graph t;
    t.ptr.assign((size_t)s + 1, 0);
    for (int v = 0; v < s; v++)
      for (int p = g.ptr[v]; p < g.ptr[v + 1]; p++) {
        t.ptr[v + 1]++;
        t.ptr[g.adj[p] + 1]++;
      }
    for (int v = 0; v < s; v++) t.ptr[v + 1] += t.ptr[v];
    t.adj.resize((size_t)t.ptr[s]);
    std::vector<int> fill(t.ptr.begin(), t.ptr.end() - 1);
    for (int v = 0; v < s; v++)
      for (int p = g.ptr[v]; p < g.ptr[v + 1]; p++) {
        t.adj[fill[v]++] = g.adj[p];
        t.adj[fill[g.adj[p]]++] = v;
      }
    g.ptr.swap(t.ptr);
    g.adj.swap(t.adj);
  }
  return hash;
}

}  // namespace

int64_t front_entry(const FrontPattern& p, int lo, int hi, bool dbl) {
  const Front& f = p.fronts[p.colfront[lo]];
  const uint16_t* rp = p.rpos.data() + f.row0;
  const int h = f.k + f.m;
  const int row = hi < f.c0 + f.k ? hi - f.c0 : (int)(std::lower_bound(rp + f.k, rp + h, (uint16_t)hi) - rp);
  return f.pan + front_elem(h, row, lo - f.c0, dbl);
}

bool build_front_patterns(const Csr& A, const std::vector<int>& starts, const std::vector<int>& inds,
                          int64_t max_work, int nw, int groups, int ug,
                          std::vector<FrontPattern>& patterns, std::vector<int>& pat,
                          std::vector<int>& out, int* chosen) {
  const int nb = (int)starts.size() - 1, least = chosen ? 1 : groups;
  pat.assign((size_t)nb, -1);
  out.resize(inds.size());
  // the first block of a graph makes the pattern, the others of the same
  // graph (compared entry by entry) share it
  struct Known {
    Graph g;
    bool mirrored;
    Tree t;
    FrontPattern p;
  };
  std::vector<std::unique_ptr<Known>> known;
  std::unordered_map<uint64_t, std::vector<int>> by_hash;
  std::mutex mu;
  bool ok = true;
  int limit = groups;  // workgroups that suit every pattern so far
  const int nth = std::max(1, std::min(setup_threads(), nb));
  // f on every thread; next() deals out the numbers below `count`, one at a time
  // (another thread of the set-up may keep a core busy for part of it)
  auto parallel = [&](int count, auto&& f) {
    std::atomic<int> taken{0};
    auto next = [&]() { return std::min(taken++, count); };
    std::vector<std::thread> th;
    for (int t = 0; t < nth; t++) th.emplace_back([&]() { f(next); });
    for (auto& x : th) x.join();
  };
  parallel(nb, [&](auto&& next) {
    std::vector<int> floc;
    Graph g;
    for (int b = next(); b < nb; b = next()) {
      const int s0 = starts[b], s = starts[b + 1] - s0;
      bool mirrored;
      const uint64_t h = local_graph(A, inds.data() + s0, s, floc, g, mirrored);
      Known* mine = nullptr;
      int count = 0;
      for (size_t seen = 0; pat[b] < 0; seen++) {  // the graphs of this hash one by one, compared outside the lock
        const Known* like = nullptr;
        int at = 0;
        {
          std::lock_guard<std::mutex> lk(mu);
          if (!ok) return;
          std::vector<int>& all = by_hash[h];
          if (seen < all.size()) {
            at = all[seen];
            like = known[at].get();
          } else {
            pat[b] = (int)known.size();
            all.push_back(pat[b]);
            known.emplace_back(new Known{std::move(g), mirrored, {}, {}});
            mine = known.back().get();
            count = limit;
          }
        }
        if (like && like->mirrored == mirrored && like->g.ptr == g.ptr && like->g.adj == g.adj) pat[b] = at;
      }
      if (!mine) continue;
      bool fits = make_tree(mine->g, mine->t);
      while (fits && !(fits = make_pattern(mine->t, max_work, nw, count, ug, mine->p)) && count > least)
        fits = true, count /= 2;
      if (count == least) mine->t = Tree{};  // nothing smaller will be asked for
      std::lock_guard<std::mutex> lk(mu);
      ok = ok && fits;
      limit = std::min(limit, count);
    }
  });
  // the others follow the one that takes the fewest workgroups
  for (; ok; limit /= 2) {
    const int count = (int)known.size();
    std::atomic<bool> fits{true};
    parallel(count, [&](auto&& next) {
      for (int k = next(); k < count && fits; k = next())
        if (known[k]->p.groups != limit && !make_pattern(known[k]->t, max_work, nw, limit, ug, known[k]->p)) fits = false;
    });
    if (fits) break;
    ok = limit > least;
  }
  if (!ok) return false;
  if (chosen) *chosen = limit;
  patterns.clear();
  for (auto& k : known) {
    patterns.push_back(std::move(k->p));
    patterns.back().mirrored = k->mirrored;
  }
  parallel(nb, [&](auto&& next) {
    for (int b = next(); b < nb; b = next()) {
      const std::vector<int32_t>& o = patterns[pat[b]].order;
      for (size_t p = 0; p < o.size(); p++) out[starts[b] + p] = inds[starts[b] + o[p]];
    }
  });
  return true;
}

}  // namespace doug
