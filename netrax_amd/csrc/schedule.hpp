// Schedules of the op DAG: the depth-first order of the walks, the flags the
// reverse walk reads and the LDS slots; and the level runs and groups of
// independent ops (split_level_runs, set_acc_early, set_pass_slots,
// build_batched_order), which no pass of the engine takes and
// tests/schedule_check.cpp replays.  Host code only, no HIP calls, so the
// schedules can be built and checked without a GPU.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

#include "engine.hpp"

namespace nrx {

// OP_HAS_CONSUMERS / OP_FIRST_KID* for ops walked by the adjoint in the
// order `adj_order` (indices into ops).
void set_adjoint_flags(std::vector<DevOp> &ops, const std::vector<int> &adj_order, int nv);

// Plain form: splits every level chunk into runs of ops that share no child
// (first fit, in op order) and reorders the chunk's ops so that each run is
// contiguous.  The ops of a run can deliver their adjoints concurrently;
// runs are returned as op ranges, per chunk in order, with run_begin[c]
// the first run of chunk c (size chunks + 1).
void split_level_runs(std::vector<DevOp> &ops, const std::vector<LevelChunk> &chunks, std::vector<LevelChunk> &runs,
                      std::vector<int> &run_begin);

// Walks: every variant the roots need, children first, each
// root's subtrees depth first and the child that needs more rows at once
// before the other, so that few rows are held at a time.
std::vector<int> depth_first_order(const Dag &dag, const std::vector<int> &root_slots);

// LDS slots of the forward walk over ops[0, n) (OP_PASS_KID*: the child is
// read from the slot its op left it in; OP_A_PASS: the op leaves its CLV in
// a slot), of which the wave has n_slots (2 to WALK_SLOTS).  Rows are the
// numbers in the ops; a child no slot holds is read from HBM (OP_LOAD*), one
// op early.
void assign_forward_slots(DevOp *ops, int n, int n_slots);

// LDS slots and load flags (OP_PASS_*, OP_A_PASS, OP_A_LATE, OP_ACC*)
// of the reverse walk over ops[n - 1] .. ops[0]; the adjoint flags
// (set_adjoint_flags) hold for the whole sweep, of which the ops may be a part.
// An op's own adjoint, where HBM holds it, is read one op early unless
// OP_A_LATE.
void assign_reverse_slots(DevOp *ops, int n, int n_slots);

constexpr int CUS = 256, LDS_PER_CU = 160 * 1024, LDS_PER_GROUP = 64 * 1024;
constexpr int LDS_PIECE = 1280;  // LDS is given out in pieces of this

// LDS slots per wave of a walk of `groups` workgroups, of which a CU's
// registers hold at most `most_per_cu`: as many as let the workgroups that a CU
// gets be resident together.  lds(n): a workgroup's dynamic LDS with n slots;
// fixed: what its kernel declares besides.
template <typename Lds>
int walk_slots(int64_t groups, Lds &&lds, int most_per_cu = 12, size_t fixed = 0) {
  const int per_cu = static_cast<int>(std::min<int64_t>(most_per_cu, (groups + CUS - 1) / CUS));
  const size_t most = std::min<size_t>(LDS_PER_CU / per_cu / LDS_PIECE * LDS_PIECE - fixed, LDS_PER_GROUP);
  int n = 2;
  while (n < WALK_SLOTS && lds(n + 1) <= most) ++n;
  return n;
}

// LDS slots of the 20-state walks over `sites` padded sites.
struct AaSlots {
  int fwd, adj;
};
AaSlots aa_walk_slots(int C, bool fp32, int64_t sites);

// OP_ACC_EARLY* for the FP32 reverse sweep (groups backwards).
void set_acc_early(std::vector<DevOp> &ops, const std::vector<int32_t> &group_begin, int nv);

// OP_PASS_* / OP_A_PASS for the FP32 4-state reverse sweep with n_slots
// per-thread LDS slots (at most PASS_SLOTS).
void set_pass_slots(std::vector<DevOp> &ops, const std::vector<int32_t> &group_begin, int nv, int n_slots);

// The FP32 op order: depth-first post-order from the root CLVs, then groups
// of up to `group` mutually independent ops (greedy list schedule, lowest
// post-order index first, preferring ops that do not consume the group
// before).  proto[v] is the op computing variant v.  Sets the adjoint
// flags, OP_GROUP_INDEP and OP_ACC_EARLY*; pass slots are left to
// set_pass_slots.
void build_batched_order(const Dag &dag, const std::vector<int> &root_slots, const std::vector<DevOp> &proto,
                         int group, std::vector<DevOp> &ops, std::vector<int32_t> &group_begin);

}  // namespace nrx
