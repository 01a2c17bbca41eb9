// sx_tree_plan.cpp -- host side of the dissection solve: the element tree,
// its classes, the cut into levels and the kernels' tables (sx_tree.h).
#include <algorithm>
#include <cmath>
#include <map>
#include <utility>
#include <vector>

#include "sx_internal.h"
#include "sx_tree.h"

namespace sx {
namespace {

struct Node {
  int l = -1, r = -1, depth = 0, elem = -1, cls = -1;
  std::vector<int> bnd;                    // boundary nodes, canonical order
  int nelim = 0;                           // nodes eliminated right here
};

struct Builder {
  const sx_mesh* m;
  std::vector<Node> node;
  std::vector<double> cx, cy;
  std::vector<int> left;                   // node -> elements of it not yet inside
  std::vector<int> total, stamp, pos;
  int tick = 0, maxdepth = 0;
  int pin = -1;                            // the unknown a singular mode drops
  std::map<std::vector<int>, int> keys;
  std::vector<int> rep;                    // class -> a node of it

  int next () const { return m->next; }
  int gid (int e, int i) const { return m->btog[(size_t) e * m->next + i]; }

  // the unknowns shared by two sets of elements
  int interface (const std::vector<int>& a, const std::vector<int>& b)
  {
    tick += 2;
    int n = 0;
    for (int e : a)
      for (int i = 0; i < next (); i++) {
        const int g = gid (e, i);
        if (g < m->nsolve) stamp[g] = tick;
      }
    for (int e : b)
      for (int i = 0; i < next (); i++) {
        const int g = gid (e, i);
        if (g < m->nsolve && stamp[g] == tick) { stamp[g] = tick + 1; n++; }
      }
    return n;
  }

  // the halves of `el` across one coordinate: cut where the element centres
  // jump, as near the middle as there is a jump
  bool cut (const std::vector<int>& el, const std::vector<double>& c, std::vector<int>& a,
            std::vector<int>& b) const
  {
    std::vector<double> v;
    for (int e : el) v.push_back (c[e]);
    std::sort (v.begin (), v.end ());
    const int n = (int) v.size ();
    const double tol = 1e-9 * std::max (1.0, std::max (std::fabs (v.front ()), std::fabs (v.back ())))
                       + 1e-6 * (v.back () - v.front ()) / n;
    int best = 0;
    for (int p = 1; p < n; p++)
      if (v[p] - v[p - 1] > tol && (!best || std::abs (2 * p - n) < std::abs (2 * best - n))) best = p;
    if (!best || 4 * best < n || 4 * (n - best) < n) return false;
    const double at = 0.5 * (v[best] + v[best - 1]);
    a.clear ();
    b.clear ();
    for (int e : el) (c[e] < at ? a : b).push_back (e);
    return true;
  }

  int make (const std::vector<int>& el, int depth)
  {
    const int id = (int) node.size ();
    node.emplace_back ();
    node[id].depth = depth;
    maxdepth = std::max (maxdepth, depth);
    if (el.size () == 1) {
      const int e = el[0];
      std::vector<int> key {-1, m->cls[e]}, bnd;
      for (int i = 0; i < next (); i++) {
        const int g = gid (e, i);
        key.push_back (g >= m->nsolve ? 0 : g == pin ? 2 : 1);
        if (g < m->nsolve) bnd.push_back (g);
      }
      node[id].elem = e;
      // (a node only this element holds is eliminated by the first front)
      node[id].bnd = bnd;
      classify (id, key);
      return id;
    }
    std::vector<int> a, b, a2, b2;
    const bool hx = cut (el, cx, a, b), hy = cut (el, cy, a2, b2);
    if (!hx && !hy) {
      a.assign (el.begin (), el.begin () + el.size () / 2);
      b.assign (el.begin () + el.size () / 2, el.end ());
    } else if (!hx || (hy && interface (a2, b2) < interface (a, b))) {
      a.swap (a2);
      b.swap (b2);
    }
    const int l = make (a, depth + 1), r = make (b, depth + 1);
    node[id].l = l;
    node[id].r = r;
    // union of the halves' boundaries; a node all of whose elements are
    // inside is eliminated here
    tick += 2;
    std::vector<int> key {node[l].cls, node[r].cls}, uni = node[l].bnd;
    for (size_t i = 0; i < uni.size (); i++) { stamp[uni[i]] = tick; pos[uni[i]] = (int) i; }
    for (int g : node[r].bnd) {
      if (stamp[g] == tick) {
        key.push_back (pos[g]);
      } else {
        key.push_back (-1);
        uni.push_back (g);
      }
    }
    // elements inside that hold g: counted once per leaf on the way up
    std::vector<int> bnd;
    for (int e : el)
      for (int i = 0; i < next (); i++) {
        const int g = gid (e, i);
        if (g < m->nsolve) left[g]++;
      }
    for (int g : uni) {
      const bool in = left[g] == total[g] && (g != pin || depth == 0);
      key.push_back (in ? (g == pin ? 3 : 1) : (g == pin ? 2 : 0));
      if (in) node[id].nelim++;
      else bnd.push_back (g);
    }
    for (int e : el)
      for (int i = 0; i < next (); i++) {
        const int g = gid (e, i);
        if (g < m->nsolve) left[g] = 0;
      }
    node[id].bnd.swap (bnd);
    classify (id, key);
    return id;
  }

  void classify (int id, const std::vector<int>& key)
  {
    auto it = keys.find (key);
    if (it == keys.end ()) {
      it = keys.emplace (key, (int) rep.size ()).first;
      rep.push_back (id);
    }
    node[id].cls = it->second;
  }

  // nodes eliminated in the subtree of id above depth c
  int elim_to (int id, int c) const
  {
    const Node& n = node[id];
    if (n.depth >= c || n.elem >= 0) return 0;
    return n.nelim + elim_to (n.l, c) + elim_to (n.r, c);
  }
  // the parts of the front at id when the next cut is at depth c
  void parts (int id, int c, std::vector<int>& out) const
  {
    const Node& n = node[id];
    if (n.depth >= c || n.elem >= 0) { out.push_back (id); return; }
    parts (n.l, c, out);
    parts (n.r, c, out);
  }
};

// Columns a tile may hold: 16, fewer where the column operand of K rows
// would not fit the LDS bound
int tile_fronts (int K, int nr)
{
  int nf = 16 / nr;
  while (nf > 1 && sizeof (double) * (size_t) K * ((nf * nr) | 1) > TREE_LDS_MAX) nf--;
  return nf;
}

// How a tile's row blocks go to workgroups.  With workgroups to spare
// (WG_FILL, three a CU) one takes every block of a tile, four at a time, so
// the columns are gathered once; with few tiles the blocks are dealt out
// and the k steps of a block split over wavefronts, as far as each still
// keeps its part of the operator in flight at once.  In a batch (tiles of
// many sizes in one launch) four blocks a workgroup, k split from 24 pairs:
// 309 us for 64 uneven problems, 380 with whole tiles, 324 with eight blocks.
constexpr int WG_FILL = 768;
void split_rows (int blocks, int pairs, long long tiles, bool batch, int* nrb, int* kw)
{
  if (batch) {
    *kw = pairs <= 24 ? 1 : pairs <= 48 ? 2 : 4;
    *nrb = 4 / *kw;
    return;
  }
  const int quads = (blocks + 3) / 4;
  if (tiles * quads >= WG_FILL) {
    const int parts = (int) std::min<long long> ((WG_FILL + tiles - 1) / tiles, quads);
    *kw = 1;
    *nrb = 4 * ((quads + parts - 1) / parts);
    return;
  }
  *kw = pairs <= 10 ? 1 : pairs <= 24 ? 2 : 4;
  *nrb = 4 / *kw;
}

// Time of a level (both directions, two right-hand sides per mode), us; the
// cuts are chosen by it.  src: its fronts have fronts among their parts.
// Up to TREE_FEW_MODES modes (and TREE_FEW_OPERATORS element classes times
// modes: on a mesh graded both ways each front is a class and a tile of its
// own) most workgroups are resident at once and a level costs its launches
// (4.5 us each measured) and the bytes of its operators, once from memory
// (4 TB/s) and once per tile of columns from the L2s (12 TB/s).  share:
// solves side by side share the launches.
// With more the workgroups queue: that of a small front is a chain of
// load rounds, and its place on a CU, not the bytes, bounds a level of many
// modes or many classes (cuts chosen by bytes alone took up to 1.9x the
// solve of these or of the band at 128 to 256 modes).  The terms, a launch
// with one workgroup's chain, every workgroup, operators, gathers and
// stores, are the fit to 2,400 traced launches (4x4 to 32x32 elements, N_P 4
// to 12, uniform and graded): a solve within 16 % for nine tenths of them.
// (The fit is no better than the bytes up to 32 modes: it cut the 16x16
// N_P=10 problem into 3 levels instead of 4, 152 us instead of 145.)
constexpr int TREE_FEW_OPERATORS = 4096;
struct LevelClass { int k, b, count; };
double direction_us (const std::vector<LevelClass>& cl, int nmodes, bool down, bool src)
{
  long long tiles = 0;
  for (const LevelClass& c : cl) {
    const int nf = tile_fronts (c.k + c.b, 2);
    tiles += (c.count + nf - 1) / nf;
  }
  double wg = 0.0, bytes = 0.0, in = 0.0, out = 0.0, turns = 0.0;
  int kmax = 0;
  for (const LevelClass& c : cl) {
    const int nf = tile_fronts (c.k + c.b, 2), nt = (c.count + nf - 1) / nf;
    const int K = down ? c.k + c.b : c.k, rows = down ? c.k : c.b;
    const int blocks = (rows + 15) / 16, pairs = (K + 7) / 8;
    if (!blocks) continue;
    kmax = std::max (kmax, K);
    int nrb, kw;
    split_rows (blocks, pairs, tiles * nmodes, false, &nrb, &kw);
    const int per = (blocks + nrb - 1) / nrb;            // workgroups of a tile
    wg += (double) nt * per;
    bytes += 1024.0 * nt * blocks * pairs;
    in += 2.0 * c.count * per * K;
    out += 2.0 * c.count * rows;
    turns += (double) nt * per * ((nrb + 4 / kw - 1) / (4 / kw)) * ((pairs + kw - 1) / kw);
  }
  if (wg == 0.0) return 0.0;
  const double chain = down ? 3.8 + 0.032 * turns / wg + 9.4e-4 * kmax + 1.5e-3 * in / wg
                           : 2.6 + 0.26 * turns / wg + 2.3e-3 * kmax + 7.6e-4 * in / wg;
  const double each = down ? 4.0e-3 * wg + 1.7e-7 * bytes + (src ? 6.4e-6 : 3.4e-6) * out
                           : 4.4e-3 * wg + 2.3e-7 * bytes + (src ? 1.4e-6 * in + 2.8e-5 * out : 5.0e-6 * out);
  return chain + nmodes * each;
}

double level_us (const std::vector<LevelClass>& cl, int nmodes, int share, bool many, bool root,
                 bool src)
{
  if (many)
    return direction_us (cl, nmodes, true, src) + (root ? 0.0 : direction_us (cl, nmodes, false, src));
  double us = (root ? 4.5 : 9.0) / share;
  for (const LevelClass& c : cl) {
    const int K = c.k + c.b, nf = tile_fronts (K, 2);
    const double bytes = 8.0 * nmodes * ((double) c.k * K + (double) c.k * c.b);
    us += bytes / 4.0e6 + bytes * ((c.count + nf - 1) / nf) / 12.0e6;
    // one wavefront's chain of k-step rounds, each a memory latency
    us += 1e-3 * K / share;
  }
  return us;
}

}  // namespace

bool tree_plan (const sx_mesh* m, int nmodes, int share, TreePlan& P)
{
  if (m->nsolve < 1) return false;
  Builder B;
  B.m = m;
  // (a mode is singular only with no essential node; the fronts that hold
  // its dropped unknown are then classes of their own)
  if (m->nglobal == m->nsolve) B.pin = m->nsolve - 1;
  const int next = m->next, npnp = m->npnp;
  B.stamp.assign (m->nglobal, 0);
  B.pos.assign (m->nglobal, 0);
  B.left.assign (m->nglobal, 0);
  B.total.assign (m->nglobal, 0);
  for (int e = 0; e < m->nel; e++) {
    B.tick++;
    for (int i = 0; i < next; i++) {
      const int g = B.gid (e, i);
      if (g >= m->nsolve) continue;
      if (B.stamp[g] == B.tick) return false;
      B.stamp[g] = B.tick;
      B.total[g]++;
    }
    double x = 0.0, y = 0.0;
    for (int i = 0; i < npnp; i++) {
      x += m->hx[(size_t) e * npnp + i];
      y += m->hy[(size_t) e * npnp + i];
    }
    B.cx.push_back (x / npnp);
    B.cy.push_back (y / npnp);
  }
  for (int g = 0; g < m->nsolve; g++)
    if (!B.total[g]) return false;
  std::vector<int> all (m->nel);
  for (int e = 0; e < m->nel; e++) all[e] = e;
  // canonical element order: rows of equal y, then x
  std::stable_sort (all.begin (), all.end (), [&] (int a, int b) {
    return B.cy[a] < B.cy[b] - 1e-9 * (1.0 + std::fabs (B.cy[b]));
  });
  const int root = B.make (all, 0);

  // -- cut the binary tree into levels: the cheapest chain of depths
  // 0 = d0 < d1 < ... (a level's fronts are the tree nodes at its depth)
  const int nd = B.maxdepth + 1;
  std::vector<std::vector<int>> at (nd + 1);
  for (int i = 0; i < (int) B.node.size (); i++)
    if (B.node[i].elem < 0 || i == root) at[B.node[i].depth].push_back (i);
  auto bnd_dim = [&] (int id) { return (int) B.node[id].bnd.size (); };
  const int last = std::max (nd - 1, 1);         // elements lie at depth <= nd - 1
  const bool many = share == 1 && (nmodes > TREE_FEW_MODES ||
                                   (long long) nmodes * m->nclass > TREE_FEW_OPERATORS);
  auto cost = [&] (int a, int c) {
    std::map<int, int> count;
    for (int id : at[a]) count[B.node[id].cls]++;
    std::vector<LevelClass> cl;
    for (auto& kv : count) {
      const int id = B.rep[kv.first];
      // the representative may sit at another depth: same subtree, shifted
      const int k = B.node[id].elem >= 0 ? bnd_dim (id)
                                         : B.elim_to (id, c - a + B.node[id].depth);
      const int b = B.node[id].elem >= 0 ? 0 : bnd_dim (id);
      if (sizeof (double) * (size_t) (k + b) * 7 > TREE_LDS_MAX || k + b > 4096) return 1e30;
      cl.push_back ({k, b, kv.second});
    }
    return level_us (cl, nmodes, share, many, a == 0, c < last);
  };
  std::vector<double> best (nd + 1, 1e30);
  std::vector<int> from (nd + 1, -1);
  best[0] = 0.0;
  for (int c = 1; c <= last; c++)
    for (int a = 0; a < c; a++) {
      if (best[a] >= 1e30) continue;
      const double v = best[a] + cost (a, c);
      if (v < best[c]) { best[c] = v; from[c] = a; }
    }
  if (best[last] >= 1e30) return false;
  P.est_us = best[last];
  std::vector<int> cuts;
  for (int c = last; c > 0; c = from[c]) cuts.push_back (from[c]);
  std::reverse (cuts.begin (), cuts.end ());     // depths of the levels
  const int nl = (int) cuts.size ();
  cuts.push_back (last);

  // -- fronts per level, sorted by class
  P.nsolve = m->nsolve;
  std::vector<int> front_of (B.node.size (), -1);     // tree node -> front
  std::vector<int> fnode;                             // front -> tree node
  std::vector<int> fcls;                              // front -> plan class
  std::vector<int> lev_of;
  std::vector<std::vector<int>> fk, fb;               // a front's node lists
  P.lev.resize (nl);
  std::vector<std::vector<int>> level_fronts (nl);
  for (int j = 0; j < nl; j++) {
    std::vector<int> ids = at[cuts[j]];
    std::stable_sort (ids.begin (), ids.end (),
                      [&] (int a, int b) { return B.node[a].cls < B.node[b].cls; });
    P.lev[j].cls0 = (int) P.cls.size ();
    int prev = -1;
    for (int id : ids) {
      if (B.node[id].cls != prev) {
        prev = B.node[id].cls;
        P.cls.emplace_back ();
        P.lev[j].ncls++;
      }
      front_of[id] = (int) fnode.size ();
      level_fronts[j].push_back ((int) fnode.size ());
      fnode.push_back (id);
      fcls.push_back ((int) P.cls.size () - 1);
      lev_of.push_back (j);
    }
  }
  const int nf = (int) fnode.size ();
  fk.resize (nf);
  fb.resize (nf);
  std::vector<int> offk (nf), offb (nf), offn (nf);
  std::vector<std::vector<int>> pt (nf);
  size_t ok = 0, ob = 0, on = 0;
  for (int f = 0; f < nf; f++) {
    const int id = fnode[f], c = cuts[lev_of[f] + 1];
    B.parts (id, c, pt[f]);
    B.tick += 2;
    std::vector<int> uni;
    for (int p : pt[f])
      for (int g : B.node[p].bnd)
        if (B.stamp[g] != B.tick) { B.stamp[g] = B.tick; uni.push_back (g); }
    if (B.node[id].elem >= 0) {
      fk[f] = uni;
    } else {
      for (int g : B.node[id].bnd) B.stamp[g] = B.tick + 1;
      for (int g : uni) (B.stamp[g] == B.tick + 1 ? fb[f] : fk[f]).push_back (g);
    }
    if (f && fb[f].empty ()) return false;       // a component of its own
    offk[f] = (int) ok;
    offb[f] = (int) ob;
    offn[f] = (int) on;
    ok += fk[f].size ();
    ob += fb[f].size ();
    on += fk[f].size () + fb[f].size ();
  }
  if ((int) ok != m->nsolve) return false;       // every unknown in one front
  // -- classes: dimensions, parts, maps
  std::vector<char> seen (P.cls.size (), 0);
  std::vector<int> local (m->nglobal, -1);
  for (int f = 0; f < nf; f++) {
    TreeClass& C = P.cls[fcls[f]];
    const int k = (int) fk[f].size (), b = (int) fb[f].size ();
    if (seen[fcls[f]]) {
      if (C.k != k || C.b != b || C.nch != (int) pt[f].size ()) return false;
      continue;
    }
    seen[fcls[f]] = 1;
    C.k = k;
    C.b = b;
    C.ch0 = (int) P.child.size ();
    C.nch = (int) pt[f].size ();
    C.mfp = (k + 7) / 8;
    C.mbp = (k + b + 7) / 8;
    for (int p : pt[f]) {
      TreeChild ch;
      ch.front = B.node[p].elem < 0;
      ch.map0 = (int) P.map.size ();
      if (ch.front) {
        ch.cls = fcls[front_of[p]];
        const std::vector<int>& pb = fb[front_of[p]];
        for (size_t i = 0; i < pb.size (); i++) local[pb[i]] = (int) i;
      } else {
        const int e = B.node[p].elem;
        ch.cls = m->cls[e];
        for (int i = 0; i < next; i++)
          if (B.gid (e, i) < m->nsolve) local[B.gid (e, i)] = i;
      }
      for (const std::vector<int>* v : {&fk[f], &fb[f]})
        for (int g : *v) P.map.push_back (local[g]);
      if (ch.front) for (int g : fb[front_of[p]]) local[g] = -1;
      else for (int i = 0; i < next; i++) local[B.gid (B.node[p].elem, i)] = -1;
      P.child.push_back (ch);
    }
    for (int i = 0; i < k + b; i++)
      if ((i < k ? fk[f][i] : fb[f][i - k]) == B.pin) C.pin = i;
  }
  // -- node tables, and the parents' slots the boundary contributions go to
  P.perm.resize (m->nsolve);
  for (int f = 0; f < nf; f++) {
    for (size_t i = 0; i < fk[f].size (); i++) P.perm[fk[f][i]] = offk[f] + (int) i;
    P.gk.insert (P.gk.end (), fk[f].begin (), fk[f].end ());
    P.gb.insert (P.gb.end (), fb[f].begin (), fb[f].end ());
  }
  std::vector<int> held (on, 0);               // parts that hold an unknown so far
  std::vector<std::pair<int, int>> to (ob);    // boundary node -> (parent's unknown, slot)
  int W = 1;
  for (int f = 0; f < nf; f++) {
    for (size_t i = 0; i < fk[f].size (); i++) local[fk[f][i]] = offn[f] + (int) i;
    for (size_t i = 0; i < fb[f].size (); i++)
      local[fb[f][i]] = offn[f] + (int) (fk[f].size () + i);
    for (int p : pt[f]) {
      if (B.node[p].elem >= 0) continue;
      P.lev[lev_of[f]].src = 1;
      const int cf = front_of[p];
      for (size_t i = 0; i < fb[cf].size (); i++) {
        const int u = local[fb[cf][i]];
        to[offb[cf] + i] = {u, held[u]++};
        W = std::max (W, held[u]);
      }
    }
  }
  if (W > 8) return false;
  P.W = W <= 4 ? 4 : 8;
  P.slots = on * P.W;
  if (P.slots >= ((size_t) 1 << 31)) return false;
  for (auto& t : to) P.tgt.push_back (t.first * P.W + t.second);
  // -- level sizes, operator offsets, work items
  for (int j = 0; j < nl; j++) {
    TreeLevel& L = P.lev[j];
    for (int c = L.cls0; c < L.cls0 + L.ncls; c++) {
      TreeClass& C = P.cls[c];
      const int n = C.k + C.b;
      C.foff = L.fsize;
      L.fsize += (size_t) n * n;
      L.kmax = std::max (L.kmax, C.k);
      L.nmax = std::max (L.nmax, n);
      C.mf = P.ops;
      P.ops += (size_t) ((C.b + 15) / 16) * C.mfp * 128;
      C.mb = P.ops;
      P.ops += (size_t) ((C.k + 15) / 16) * C.mbp * 128;
    }
    for (int q = 0; q < 3; q++) {
      const int nr = 2 * (q + 1);
      for (int dir = 0; dir < 2; dir++) {            // 0 forward, 1 backward
        (dir ? L.it_b : L.it_f)[q] = (int) P.item.size ();
        size_t lds = 0;
        const std::vector<int>& fr = level_fronts[j];
        std::vector<std::pair<size_t, size_t>> tile;
        for (size_t i0 = 0, i1; i0 < fr.size (); i0 = i1) {
          const TreeClass& C = P.cls[fcls[fr[i0]]];
          const int cap = tile_fronts (C.k + C.b, nr);
          for (i1 = i0; i1 < fr.size () && fcls[fr[i1]] == fcls[fr[i0]] && (int) (i1 - i0) < cap;) i1++;
          tile.push_back ({i0, i1});
        }
        for (auto& t : tile) {
          const int f = fr[t.first], n = (int) (t.second - t.first);
          const TreeClass& C = P.cls[fcls[f]];
          const int K = dir && j ? C.k + C.b : C.k, rows = dir ? C.k : C.b;
          int nrb, kw;
          split_rows ((rows + 15) / 16, (K + 7) / 8, (long long) tile.size () * nmodes, share > 1, &nrb,
                      &kw);
          for (int rb = 0; 16 * rb < rows; rb += nrb)
            P.item.push_back ({C.k, C.b, n, rb, std::min (nrb, (rows + 15) / 16 - rb), kw, L.src,
                               offk[f], offb[f], offn[f], (long long) (dir ? C.mb : C.mf)});
          // the column operand, k rows padded to whole pairs of steps, and
          // the partial tiles of split k ranges
          lds = std::max (lds, sizeof (double) * ((size_t) (K + 7) / 8 * 8 * ((n * nr) | 1) +
                                                  (kw > 1 ? 4 * 256 : 0)));
        }
        (dir ? L.nit_b : L.nit_f)[q] = (int) P.item.size () - (dir ? L.it_b : L.it_f)[q];
        (dir ? L.lds_b : L.lds_f)[q] = lds;
      }
    }
  }
  return true;
}

}  // namespace sx
