// sx_tree.h -- plan of the condensed systems' dissection solve: the elements
// of a mesh split recursively into halves, the binary tree cut into a few
// levels of fronts, and the tables the kernels of sx_tree.hip read.
//
// A front is a connected set of elements.  Its unknowns are the nodes it
// eliminates (k of them: shared by its parts, touching no element outside)
// followed by its boundary (b nodes shared with elements outside).  Fronts
// whose parts have the same matrices and fit together alike form a class:
// they share one factor per Fourier mode, as elements of one geometry share
// their condensed matrices.
#pragma once
#include <cstddef>
#include <vector>

struct sx_mesh;

namespace sx {

struct TreeClass {
  int k = 0, b = 0;            // eliminated and boundary unknowns
  int ch0 = 0, nch = 0;        // its parts in TreePlan::child
  int pin = -1;                // unknown nsolve-1 (dropped in a singular mode) or -1
  int mfp = 0, mbp = 0;        // k-step pairs of the forward / backward operator
  size_t foff = 0;             // front matrix in its level's buffer (doubles per mode)
  size_t mf = 0, mb = 0;       // forward / backward operator (doubles per mode)
};

// One part of a class: an element (cls: its class, matrix next x next) or a
// front of the next level (cls: class index in the plan, its trailing b x b
// block); map0: its table in TreePlan::map, front unknown -> part row or -1.
struct TreeChild { int front = 0, cls = 0, map0 = 0; };

struct TreeLevel {
  int cls0 = 0, ncls = 0;      // classes
  int src = 0;                 // its fronts have fronts among their parts
  int kmax = 0, nmax = 0;      // largest k and k + b of a class
  size_t fsize = 0;            // doubles per mode of its front matrices
  // work items per number of right-hand sides per mode (2, 4, 6: index nr/2-1)
  int it_f[3] = {}, nit_f[3] = {}, it_b[3] = {}, nit_b[3] = {};
  size_t lds_f[3] = {}, lds_b[3] = {};
};

// A workgroup's share of a level: nf consecutive fronts of one class (their
// right-hand sides are the columns), the 16-row blocks [rb0, rb0 + nrb) of
// the operator, the k steps of a block split over kw wavefronts.  Everything
// the kernel addresses by is here, so its loads depend on this one.
struct TreeItem {
  int k, b, nf, rb0, nrb, kw, src;
  int offk, offb, offn;        // of the first front; front j of the tile: + j k, + j b, + j (k + b)
  long long op;                // the class's operator (doubles per mode)
};

struct TreePlan {
  std::vector<TreeLevel> lev;      // lev[0]: the root
  std::vector<TreeClass> cls;
  std::vector<TreeChild> child;
  std::vector<int> map;
  // fronts, sorted by level and class: eliminated nodes at offk, boundary
  // at offb of the node tables.  Position offk + i is also where the
  // right-hand side of that node lies (perm: node -> position).  A front
  // leaves its boundary contributions in its parent's slots (tgt): W slots
  // for each of the parent's unknowns, one per part that holds it, so the
  // parent adds W neighbouring values; slots no part fills stay zero.
  std::vector<int> gk, gb;         // global node numbers
  std::vector<int> tgt;            // per boundary node of a front
  std::vector<int> perm;
  size_t slots = 0;
  std::vector<TreeItem> item;
  int W = 4;                       // 4 or 8
  int nsolve = 0;                  // unknowns (= gk.size())
  size_t ops = 0;                  // operator doubles per mode
  double est_us = 0.0;             // the cost the level cuts were chosen by
};

constexpr size_t TREE_LDS_MAX = 96 * 1024;   // a workgroup's column operand
constexpr int TREE_FEW_MODES = 32;           // all workgroups of a level resident at once

// false when the mesh does not suit it (an element holding one node twice,
// a node no element holds, operators past the size bound).  share: solves
// of this size that run side by side (a batch): a level's launches cost a
// share-th each, so more and smaller levels pay.
bool tree_plan (const sx_mesh* m, int nmodes, int share, TreePlan& P);

}  // namespace sx
