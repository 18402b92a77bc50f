// Internal structures of the MI355X network-likelihood engine.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "../../include/netrax_gpu.h"

namespace nrx {

// Sites of every partition are padded to a multiple of this tile, so that a
// wave's sites are of one partition.
constexpr int TILE = 64;
constexpr int MAX_CATS = 8;

// 20-state data (matrix cores): a wave holds one category of 16 sites, and
// each (partition, edge, category) has tables of P and P^T in the order of the
// matrix instructions' operands.
constexpr int AA_STATES = 20;
constexpr int AA_TILE = 32;  // tile_sites of a kernel shape's name
constexpr int AA_MAT = AA_STATES * AA_STATES;
constexpr int AA_MATS = 2 * AA_MAT;
constexpr int AA_SITES = 16;                 // sites of a wave
constexpr int AA_ROW = AA_SITES * AA_STATES;  // a wave's row: one category of its sites

// ---------------------------------------------------------------- model
struct EigenModel {
  int S = 0;
  std::vector<double> eval;   // [S]
  std::vector<double> V;      // [S][S]  P = V diag(exp(eval r t)) Vinv
  std::vector<double> Vinv;   // [S][S]
  std::vector<double> freqs;  // [S]
};

std::vector<double> gamma_mean_rates(double alpha, int ncat);
void build_model(int S, const double *subst, const double *freqs, EigenModel &m);

// ---------------------------------------------------------------- op DAG
// Child code: >= 0 is a variant slot, < 0 is tip (-code - 1).
constexpr int32_t NO_CHILD = INT32_MIN;
inline int32_t tip_code(int tip) { return -tip - 1; }
inline bool is_tip_code(int32_t c) { return c < 0 && c != NO_CHILD; }
inline int tip_of(int32_t c) { return -c - 1; }

struct Variant {
  int node = -1;
  int nkids = 0;
  int32_t kid[2] = {NO_CHILD, NO_CHILD};
  int32_t edge[2] = {-1, -1};
  int level = 0;
};

struct RootClass {
  std::vector<uint32_t> configs;  // member configurations
  int dtroot_slot = -1;           // variant at the displayed-tree root
  std::vector<uint64_t> edges;    // alive edge set (bitset over edges)
};

struct Dag {
  int n_retic = 0;
  std::vector<Variant> var;
  std::vector<RootClass> classes;
};

// Enumerates the 2^r displayed-tree configurations and deduplicates CLVs
// by (node, alive subtree).  Throws std::invalid_argument on bad input.
Dag compile_dag(const nrx_network_desc &net);

// ---------------------------------------------------------------- device
// One CLV op.  The forward pass computes CLV `out` from its children; the
// adjoint pass (push form) reads the adjoint of `out` and delivers the
// back-propagated vectors to the children.
struct DevOp {
  int32_t out;
  int32_t nk;
  int32_t kid[2];    // child codes
  int32_t edge[2];   // edge to each child
  int32_t root;      // index of the root-CLV site sum this op feeds, or -1
  int32_t flags;     // OP_HAS_CONSUMERS | OP_FIRST_KID0 | OP_FIRST_KID1
  int32_t gslot[2];  // gradient-partial row of (this op, child k)
  int32_t slots;     // LDS slots of the uses 0, 1 (children) and 2 (own row), see walk_slot
  int32_t pad;
};
inline __host__ __device__ int walk_slot(const DevOp &op, int u) { return (op.slots >> (8 * u)) & 255; }
constexpr int32_t OP_HAS_CONSUMERS = 1;  // adjoint of `out` was accumulated by consumers
constexpr int32_t OP_FIRST_KID0 = 2;     // first consumer of kid[0] in adjoint order
constexpr int32_t OP_FIRST_KID1 = 4;
// A row that a walk hands over in an LDS slot of the wave (DevOp::slots) instead
// of HBM.  Forward: OP_A_PASS, the op leaves its CLV in slot walk_slot(op, 2);
// OP_PASS_KIDk, child k is read from slot walk_slot(op, k).  Reverse:
// OP_PASS_KIDk, child k's adjoint is delivered to slot walk_slot(op, k) (written
// by the first delivery, added to by later ones); OP_A_PASS, the op's own
// adjoint is in slot walk_slot(op, 2).
constexpr int32_t OP_PASS_KID0 = 64;
constexpr int32_t OP_PASS_KID1 = 128;
constexpr int32_t OP_A_PASS = 256;
// reverse: the op's own adjoint lies in HBM and the op before it in the sweep
// delivered to it last, so it is read after that delivery instead of one op
// ahead
constexpr int32_t OP_A_LATE = 512;
// reverse: child k's adjoint lies in HBM and holds deliveries
constexpr int32_t OP_ACC0 = 1024;
constexpr int32_t OP_ACC1 = 2048;
// forward: child k's CLV is read from HBM
constexpr int32_t OP_LOAD0 = 1 << 21;
constexpr int32_t OP_LOAD1 = 1 << 22;
constexpr int WALK_SLOTS = 32;  // LDS slots of a wave, at most
// Of the order in groups of independent ops that no kernel walks any more
// (build_batched_order, set_acc_early and set_pass_slots in schedule.hpp):
// the first op of a group that consumes no CLV of the group before it; child
// k's adjoint holds deliveries of earlier groups only; slots in the flags,
// where OP_PASS_* and OP_A_PASS stand for those.
constexpr int32_t OP_GROUP_INDEP = 8;
constexpr int32_t OP_ACC_EARLY0 = 16;
constexpr int32_t OP_ACC_EARLY1 = 32;
constexpr int PASS_SLOTS = 5;
constexpr int PASS_SHIFT = 12;  // slot of use u (0, 1: children, 2: own) in bits 12 + 3u
constexpr int32_t PASS_BITS = 0x1FF << PASS_SHIFT;
inline __host__ __device__ int pass_slot(int32_t flags, int u) { return (flags >> (PASS_SHIFT + 3 * u)) & 7; }

// The ops [op_begin, op_end): one op of the walk (where a memory budget may cut it).
struct LevelChunk {
  int level, op_begin, op_end;
};

// One step of a root-to-branch path: the op (its output slot), the child
// the path continues into and the other child (NO_CHILD for a one-child
// op), with their edges; children are slots or tip codes as in DevOp.
struct PathStep {
  int32_t out, child, sib;
  int32_t edge_child, edge_sib;
  int32_t nk;
};
// P blocks of a path's first PATH_STAGED_STEPS steps are staged in LDS by
// the path kernels (4 states)
constexpr int PATH_STAGED_STEPS = 24;
inline size_t path_lds_bytes(int S, int C, int max_steps) {
  return S == 4 ? sizeof(double) * 2 * C * S * S * static_cast<size_t>(std::min(max_steps, PATH_STAGED_STEPS)) : 0;
}

// Device-side Newton-Raphson of one branch length (nrx_optimize_branches):
// the safeguarded iteration's state, and per displayed-tree class what the
// derivative mixture needs.
struct NewtonState {
  double x, a, b;      // current length and the bracket of the maximiser
  double x0, lo, hi, tol;
  double d1, d2;       // last derivatives
  double lnl_old, lnl_new;
  int32_t n_paths, done, iters, accepted;
  int32_t max_iters, pad;
};
struct DerivClassDev {
  double logprob;
  int32_t use;   // passes min_tree_logprob
  int32_t has;   // its alive edges contain the branch
  int32_t path;  // sumtable row, or -1
  int32_t pad;
};

struct DevClass {
  double logprob;
  int32_t root_index;
  int32_t use;
};

// Everything a kernel needs about the site axis and the models.
struct DevLayout {
  int64_t n_sites_pad;   // sites over all partitions, tile padded
  int32_t n_tiles;
  int32_t n_parts;
  int32_t n_edges;
  int32_t S;
  int32_t C;
};

// Device view of one FP32-form engine, read by the walks; a 4-state launch has a
// table of (network, wave) work items, so it scores one network or a batch.
struct NetDesc {
  DevLayout L;
  int32_t n_root;
  int32_t n_uses;  // gradient rows
  // op lists (forward and reverse) and LDS slots per wave
  const DevOp *ops_fwd, *ops_adj;
  int32_t n_fwd, n_adj, fwd_slots, adj_slots;
  double *seed;      // root seed factors [root][site]
  const float *PfT;  // transposes of Pf's matrices
  float *clv;
  int32_t *scl;
  float *adj;
  int32_t *adj_exp;
  const uint8_t *tips;
  const float *Pf;
  const float *Qf;
  const float *Pa;  // 20-state data: operand tables [part][edge][C][P, P^T][AA_MAT]
  const int32_t *tile_part;
  const double *freqs;
  const double *weights;
  const double *beta;
  double *root_partials;
  double *grad_partials;
};

struct WorkItem {
  int32_t net;
  int32_t tile;  // the wave's sites, in the launch's blocks per wave
};

// Per-network parameters of the small kernels when a batch is scored.
struct SmallDesc {
  DevLayout L;
  // P matrices
  const double *V, *Vinv, *ev, *rates, *host_brlen;  // lengths: pinned host memory
  double *brlen;
  double *P;
  float *Pf, *PfT;
  // reductions and mixture
  int32_t n_root, nc, R, n_uses;
  const int32_t *part_tile_begin;
  const DevClass *classes;
  const double *class_dlogprob;
  double *root_partials, *root_sums, *grad_partials, *use_sums, *beta;
  const int32_t *edge_use_begin, *edge_use_list;
  double *res;
  int32_t rl_total, rl_per_part, rl_root_logl, rl_tree_logl, rl_alpha, rl_dbrlen,
      rl_part_dbrlen, rl_dprob;
  int32_t pw;           // root partials per 64-site tile
  int32_t gwpt, pad[2];  // gradient partials per 64-site tile: the launch's waves
};

struct Engine;

// Batch launchers (kernels.hip): one launch per kernel for n networks.
void launch_pmatrices_multi(hipStream_t s, const SmallDesc *d, int n, int max_elems);
void launch_root_reduce_multi(hipStream_t s, const SmallDesc *d, int n, int max_rows);
void launch_mixture_multi(hipStream_t s, const SmallDesc *d, int n, int variant);
void launch_grad_reduce_multi(hipStream_t s, const SmallDesc *d, int n, int max_uses, int max_parts, int max_edges);
void launch_gather_results(hipStream_t s, const SmallDesc *d, int n, const int64_t *offsets,
                           double *out, int max_size);
// blocks: 64-row blocks per wave (1 or 2); slots: LDS slots, as every network's descriptor has them
void launch_forward_persistent_multi(hipStream_t stream, int C, int blocks, const NetDesc *nets, const WorkItem *work,
                                     int n_work, int slots);
void launch_adjoint_persistent_multi(hipStream_t stream, int C, int blocks, const NetDesc *nets, const WorkItem *work,
                                     int n_work, int slots);

// Dynamic LDS of the 4-state walks: the reverse walk's ring of gradient sums
// on their way to HBM, and n_slots rows with their scaler words or exponents.
constexpr int GRAD_RING = 128;
// Slices of a partition's waves that a gradient row is summed in.
constexpr int GRAD_SLICES = 32;
constexpr size_t forward_walk_lds(int nq, int n_slots) { return static_cast<size_t>(n_slots) * (nq * 512 + 256); }
constexpr size_t adjoint_walk_lds(int nq, int n_slots) {
  return sizeof(double) * GRAD_RING + static_cast<size_t>(n_slots) * nq * 512;
}
// (20 states: a wave per category of 16 sites)
constexpr size_t forward_walk_lds_aa(int C, int n_slots) {
  return static_cast<size_t>(n_slots) * C * (sizeof(double) * AA_ROW + 4 * AA_SITES);
}
// (what the forward kernels declare besides: the cells that the categories' waves trade)
constexpr size_t forward_fixed_lds_aa(int C) { return C > 1 ? 2 * C * (4 + 8 * AA_SITES) : 0; }
constexpr size_t forward_fixed_lds_aa32(int C) { return C > 1 ? 2 * C * (4 + 8) * AA_SITES : 0; }
constexpr size_t adjoint_walk_lds_aa(int n_slots) {
  return sizeof(double) * (GRAD_RING + static_cast<size_t>(n_slots) * AA_ROW);
}
constexpr size_t forward_lds_aa32(int C, int n_slots) {
  return static_cast<size_t>(n_slots) * C * 4 * (AA_ROW + AA_SITES);
}
constexpr size_t adjoint_lds_aa32(int n_slots) {
  return sizeof(double) * GRAD_RING + forward_lds_aa32(1, n_slots);
}
constexpr size_t forward_lds32(int C, int blocks, int n_slots) {
  return static_cast<size_t>(n_slots) * blocks * (1024 + 256 / C);
}
constexpr size_t adjoint_lds32(int C, int blocks, int n_slots) {
  return sizeof(double) * GRAD_RING + forward_lds32(C, blocks, n_slots);
}

// Kernel launchers (kernels.hip)
void launch_pmatrices(Engine &e);
// FP64: ops in an order with children first, with their LDS slots
// assigned (assign_forward_slots); root site sums and seed factors included
void launch_forward_walk(Engine &e, const DevOp *ops, int n_ops);
// host: pinned memory that the results go to as well, or null
void launch_mixture(Engine &e, int variant, int partials_per_tile, double *host);
// FP64: the ops backwards (slots from assign_reverse_slots); model: for the
// model gradient's sums per use (in the adjoint rows) and root (d_mg_r; 4 states)
void launch_adjoint_walk(Engine &e, const DevOp *ops, int n_ops, bool model);
void launch_grad_reduce(Engine &e, double *host);
// nets: a descriptor other than the engine's own (its invalid ops only)
void launch_forward_persistent(Engine &e, const NetDesc *nets = nullptr);
void launch_adjoint_persistent(Engine &e);
void launch_forward_mfma(Engine &e, const NetDesc *nets = nullptr);
void launch_adjoint_mfma(Engine &e);
void launch_sumtables(Engine &e, int n_paths, int max_steps);
// FP64 4-state: from the walk's sums per partition dJ/dQ [16], dJ/drates [C]
// and the frequencies' direct share [4] into out; the others are workspaces:
// g_sum [uses][P][slices][64 or 128], r_sum [roots][P][slices][4], edge_out [P][E][16 + C]
void launch_model_grad(Engine &e, double *g_sum, double *r_sum, double *edge_out, double *out, int n_slice);
// Newton-Raphson of a branch length on the device: `rounds` rounds of
// (evaluate the sumtables at the state's length, reduce, Newton step; no-ops
// once the state is done or has taken its max_iters steps), then the
// evaluation at the current length and the acceptance check.  The number
// of paths and every length come from the device state, so the sequence is
// captured once and replayed per branch (and again while not done).
void enqueue_newton(Engine &e, int variant, int mode, int rounds, int max_paths, NewtonState *st,
                    const DerivClassDev *cls, const double *base_logl);
// allocation-free branch derivatives: a fixed device array of this many
// bytes per GPU holds every scratch buffer of nrx_brlen_derivatives_noalloc
constexpr size_t NOALLOC_SCRATCH_BYTES = size_t(16) << 20;
void *noalloc_scratch();  // its device address on the current device
// max_steps: the longest path's step count (sizes the staged P in LDS)
void launch_deriv_fused(Engine &e, const PathStep *steps, const int32_t *path_begin, int n_paths, int max_steps,
                        double brlen, double *partials, double *sums);
void launch_sumtable_eval(Engine &e, int n_paths, double brlen);

struct HipCheck {
  static void check(hipError_t err, const char *what);
};
#define NRX_HIP(x) ::nrx::HipCheck::check((x), #x)

}  // namespace nrx
