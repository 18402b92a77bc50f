// Host-side check of the 4-state walks' schedule (netrax_amd/csrc/
// schedule.cpp): the depth-first op order and the LDS slots of both walks,
// replayed for one network, whole and cut into launches.
//
// Input (stdin): n_nodes n_tips root n_edges n_retic, then n_edges edge
// parents, n_edges edge children, n_retic first and n_retic second parent
// edges, then pairs "slots pieces" until end of input.
// Output: one line per pair, "ok <counts>" or "error <what>" lines, then
// "rows <depth-first> <by level>", the fewest CLV rows a cut order needs.
#include <algorithm>
#include <cstdio>
#include <iostream>
#include <string>
#include <vector>

#include "../netrax_amd/csrc/schedule.hpp"

using namespace nrx;

static int errors = 0;
static void fail(const std::string &what) {
  if (errors++ < 20) std::printf("error %s\n", what.c_str());
}

static std::vector<DevOp> make_ops(const Dag &dag, const std::vector<int> &order) {
  std::vector<DevOp> ops;
  for (int s : order) {
    DevOp op{};
    op.out = s;
    op.nk = dag.var[s].nkids;
    for (int k = 0; k < 2; ++k) {
      op.kid[k] = k < op.nk ? dag.var[s].kid[k] : NO_CHILD;
      op.edge[k] = k < op.nk ? dag.var[s].edge[k] : 0;
    }
    op.root = -1;
    ops.push_back(op);
  }
  return ops;
}

static void check(const Dag &dag, const std::vector<int> &order, int n_slots, int pieces) {
  const int nv = static_cast<int>(dag.var.size()), n = static_cast<int>(order.size());
  std::vector<DevOp> fwd = make_ops(dag, order);
  std::vector<int> back, uses(nv, 0);
  for (int i = n - 1; i >= 0; --i) back.push_back(i);
  set_adjoint_flags(fwd, back, nv);
  std::vector<DevOp> rev = fwd;
  std::vector<int> cut;
  for (int j = 0; j <= pieces; ++j) cut.push_back(static_cast<int>(static_cast<long>(n) * j / pieces));
  for (int j = 0; j < pieces; ++j) {
    assign_forward_slots(fwd.data() + cut[j], cut[j + 1] - cut[j], n_slots);
    assign_reverse_slots(rev.data() + cut[j], cut[j + 1] - cut[j], n_slots);
  }
  int slot_reads = 0, handoffs = 0;
  std::vector<int> made(nv, -1);
  for (int j = 0; j < pieces; ++j) {
    std::vector<int> held(n_slots, -1);
    for (int i = cut[j]; i < cut[j + 1]; ++i) {
      const DevOp &op = fwd[i];
      for (int k = 0; k < op.nk; ++k) {
        const int kid = op.kid[k];
        if (kid < 0) continue;
        ++uses[kid];
        if (made[kid] < 0) fail("child after its parent");
        if (op.flags & (k == 0 ? OP_PASS_KID0 : OP_PASS_KID1)) {
          ++slot_reads;
          if (walk_slot(op, k) >= n_slots || held[walk_slot(op, k)] != kid) fail("slot holds another CLV");
        } else {
          if (made[kid] >= cut[j] && made[kid] == i - 1) fail("CLV loaded before it is stored");
          if (!(op.flags & (k == 0 ? OP_LOAD0 : OP_LOAD1))) fail("CLV not loaded");
        }
      }
      if (made[op.out] >= 0) fail("variant twice");
      made[op.out] = i;
      if (op.flags & OP_A_PASS) held[walk_slot(op, 2)] = op.out;
    }
  }
  // reverse: deliveries made to a row, where they lie, and when the last was made
  std::vector<int> got(nv, 0), last(nv, n + 1);
  for (int j = pieces - 1; j >= 0; --j) {
    std::vector<int> held(n_slots, -1);
    for (int i = cut[j + 1] - 1; i >= cut[j]; --i) {
      const DevOp &op = rev[i];
      if (((op.flags & OP_HAS_CONSUMERS) != 0) != (uses[op.out] > 0)) fail("OP_HAS_CONSUMERS");
      if (got[op.out] != uses[op.out]) fail("adjoint read before its deliveries");
      if (op.flags & OP_A_PASS) {
        const int q = walk_slot(op, 2);
        if (q >= n_slots || held[q] != op.out) fail("adjoint not in its slot");
        held[q] = -1;
      } else if (uses[op.out] && last[op.out] == i + 1 && last[op.out] < cut[j + 1] && !(op.flags & OP_A_LATE)) {
        fail("adjoint loaded before its last delivery");
      }
      for (int k = 0; k < op.nk; ++k) {
        const int kid = op.kid[k];
        if (kid < 0) continue;
        const bool first = (op.flags & (k == 0 ? OP_FIRST_KID0 : OP_FIRST_KID1)) != 0;
        if (first != (got[kid] == 0)) fail("first delivery");
        if (op.flags & (k == 0 ? OP_PASS_KID0 : OP_PASS_KID1)) {
          const int q = walk_slot(op, k);
          ++handoffs;
          if (q >= n_slots || held[q] != (first ? -1 : kid)) fail("delivery to another row's slot");
          held[q] = kid;
          if (op.flags & (k == 0 ? OP_ACC0 : OP_ACC1)) fail("slot delivery reads HBM");
        } else {
          if (std::find(held.begin(), held.end(), kid) != held.end()) fail("row in a slot and in HBM");
          if (((op.flags & (k == 0 ? OP_ACC0 : OP_ACC1)) != 0) == first) fail("accumulated delivery");
          last[kid] = i;
        }
        ++got[kid];
      }
    }
    for (int q = 0; q < n_slots; ++q)
      if (held[q] >= 0) fail("slot still held at the end of a launch");
  }
  if (!errors) std::printf("ok slot_reads %d handoffs %d\n", slot_reads, handoffs);
}

// Fewest rows over the ways a memory budget may cut `order` into segments of
// about equal op counts at the ends of `chunk`s.
static int fewest_rows(const Dag &dag, const std::vector<int> &order, const std::vector<int> &chunk_end) {
  const int nv = static_cast<int>(dag.var.size()), nch = static_cast<int>(chunk_end.size());
  const long total = static_cast<long>(order.size());
  int best = nv;
  for (int K = 2; K <= nch; ++K) {
    std::vector<int> seg_of(nv, -1), last(nv, -1);
    int seg = 0, ncut = 1;
    for (int c = 0, i = 0; c < nch; ++c) {
      for (; i < chunk_end[c]; ++i) {
        seg_of[order[i]] = seg;
        for (int k = 0; k < dag.var[order[i]].nkids; ++k)
          if (dag.var[order[i]].kid[k] >= 0) last[dag.var[order[i]].kid[k]] = seg;
      }
      if (ncut < K && c + 1 < nch && static_cast<long>(chunk_end[c]) * K >= static_cast<long>(ncut) * total) {
        ++ncut;
        ++seg;
      }
    }
    std::vector<int> inner(seg + 1, 0);
    int boundary = 0;
    for (int s : order) last[s] > seg_of[s] ? ++boundary : ++inner[seg_of[s]];
    best = std::min(best, boundary + *std::max_element(inner.begin(), inner.end()));
  }
  return best;
}

int main() {
  int nn, nt, root, ne, nr;
  if (!(std::cin >> nn >> nt >> root >> ne >> nr)) return 2;
  std::vector<int32_t> ep(ne), ec(ne), rf(nr), rs(nr);
  for (auto *v : {&ep, &ec, &rf, &rs})
    for (auto &x : *v) std::cin >> x;
  nrx_network_desc net{};
  net.n_nodes = nn;
  net.n_tips = nt;
  net.root = root;
  net.n_edges = ne;
  net.n_retic = nr;
  net.edge_parent = ep.data();
  net.edge_child = ec.data();
  net.retic_first_edge = rf.data();
  net.retic_second_edge = rs.data();
  const Dag dag = compile_dag(net);
  std::vector<int> roots;
  for (const auto &c : dag.classes)
    if (std::find(roots.begin(), roots.end(), c.dtroot_slot) == roots.end()) roots.push_back(c.dtroot_slot);
  const std::vector<int> order = depth_first_order(dag, roots);
  for (int r : roots)
    if (std::find(order.begin(), order.end(), r) == order.end()) fail("root variant missing");
  int n_slots, pieces;
  while (std::cin >> n_slots >> pieces) check(dag, order, n_slots, std::min<int>(pieces, order.size()));
  std::vector<int> ends, by_level = order, level_ends;
  for (size_t i = 0; i < order.size(); ++i) ends.push_back(static_cast<int>(i) + 1);
  std::stable_sort(by_level.begin(), by_level.end(), [&](int a, int b) {
    return dag.var[a].level != dag.var[b].level ? dag.var[a].level < dag.var[b].level : a < b;
  });
  for (size_t i = 0; i < by_level.size(); ++i)
    if (i + 1 == by_level.size() || dag.var[by_level[i]].level != dag.var[by_level[i + 1]].level)
      level_ends.push_back(static_cast<int>(i) + 1);
  std::printf("rows %d %d\n", fewest_rows(dag, order, ends), fewest_rows(dag, by_level, level_ends));
  return errors ? 1 : 0;
}
