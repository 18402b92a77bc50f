// Engine state shared by the host orchestration (engine.cpp) and the
// kernel launchers (kernels.hip).
#pragma once

#include <memory>
#include <vector>

#include "engine.hpp"

struct nrx_engine {};

namespace nrx {

struct DevBuf {
  void *p = nullptr;
  size_t bytes = 0;
  DevBuf() = default;
  DevBuf(const DevBuf &) = delete;
  DevBuf &operator=(const DevBuf &) = delete;
  ~DevBuf() { release(); }
  void alloc(size_t n) {
    if (n <= bytes && p) return;
    release();
    if (n == 0) n = 16;
    NRX_HIP(hipMalloc(&p, n));
    bytes = n;
  }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
  }
  template <typename T>
  T *as() const {
    return static_cast<T *>(p);
  }
};

struct PartInfo {
  int n_sites = 0;        // patterns
  int64_t site_off = 0;   // first padded site
  int tile_begin = 0, tile_end = 0;
  bool model_set = false;
  EigenModel model;
  std::vector<double> rates;  // [C]
  std::vector<double> subst;  // exchangeabilities as given
  double alpha = 0.0;         // Gamma shape of the rates; NaN after nrx_set_category_rates
};

// Result block offsets (doubles) inside the device/host result buffers.
struct ResultLayout {
  int total, per_part, root_logl, tree_logl, alpha, dbrlen, part_dbrlen, dprob, size;
};

struct Engine : nrx_engine {
  nrx_options opt{};
  int N = 0, E = 0, R = 0, T = 0, root = 0;
  std::vector<int32_t> edge_parent, edge_child, retic_first, retic_second;
  int P = 0, S = 0, C = 0;
  std::vector<PartInfo> parts;
  DevLayout L{};
  Dag dag;

  // host parameters
  std::vector<double> brlen;  // clamped
  std::vector<double> probs;  // first-parent probabilities
  std::vector<double> class_logprob, class_dlogprob;  // [nc], [nc][R]
  std::vector<char> class_use;

  // schedule (rebuilt when the set of used classes changes)
  std::vector<char> needed;                 // [n_var]
  std::vector<std::vector<int>> level_ops;  // variant slots per level (needed only)
  std::vector<int> root_slots;              // distinct displayed-tree-root CLVs
  std::vector<int> class_root_index;        // [nc]
  // ops in the depth-first order of the walks, with their LDS slots in the two
  // lists the walks read
  std::vector<DevOp> ops_all, ops_fwd, ops_adj;
  std::vector<LevelChunk> chunks;
  std::vector<int32_t> edge_use_begin, edge_use_list;  // gradient rows per edge
  int n_uses = 0;
  int pw = 1;   // branch derivatives: site-sum partials per tile (one per wave)
  int rpw = 1;  // root site-sum partials per tile
  // walks: granules per wave (FP64, 4 states), and LDS slots per wave
  int walk_nq = 4, fwd_slots = 4, adj_slots = 4;
  int walk_blocks = 1;  // 64-row blocks per wave (FP32)
  int gwpt = 1;  // gradient partials [wave][row]: waves per tile
  // hand-offs in LDS of the batches that this engine is in (nrx_stats)
  std::vector<std::weak_ptr<const int>> batch_handoffs;
  // FP32 form shape (nrx_autotune / nrx_set_tuning): for the first, see
  // walk_blocks_of (4 states); the others are part of a shape's name only.
  int tune_group = 4;
  int tune_tile = TILE;
  int tune_lanes = 1;
  int schedule_version = 0;  // bumped by every schedule rebuild

  // branch derivatives: sumtables of one branch for every displayed tree
  // containing it (valid while nothing but that branch's length changes)
  bool deriv_valid = false;
  int deriv_edge = -1;
  std::vector<int> deriv_class;       // used classes whose alive edges contain the edge
  std::vector<int> deriv_path;        // per such class: sumtable row, or -1 (edge above the root)
  int deriv_n_paths = 0;
  std::vector<double> deriv_base_logl;  // [P][nc] tree lnLs when the sumtables were built
  DevBuf d_steps, d_path_begin, d_st, d_st_partials, d_st_sums;
  // device Newton-Raphson: state, class table, tree lnLs; its captured
  // sequence, valid while the sumtable buffers keep their addresses
  DevBuf d_nr_state, d_nr_cls;
  // model gradient (FP64, 4 states): its reverse walk's granules per wave (as
  // many as make a wave's part of an adjoint row hold an op's sums), waves per
  // tile, LDS slots and op list (of schedule model_version, where the shape is
  // not the gradient's); the sums per root, and what is made of the sums
  int model_nq() const { return C == 8 ? 4 : walk_nq < 2 ? 2 : walk_nq; }
  int model_wpt() const { return TILE * C / (16 * model_nq()); }
  int model_slots = 0, model_version = -1;
  DevBuf d_ops_model, d_use_row;  // use_row: adjoint row and child of each use
  DevBuf d_mg_r, d_mg_sums;
  // Memory budget of the FP64 form: with n_seg > 1 the CLV, adjoint and
  // scaler rows live in n_phys physical rows.  The ops are cut into
  // n_seg segments; a CLV consumed in a later segment than its own keeps a
  // fixed row (the boundary rows), the others share the rows of a pool that
  // each segment reuses.  The forward pass runs the segments in order; the
  // reverse sweep recomputes a segment's pooled CLVs before its adjoint.
  uint64_t mem_budget = 0;  // bytes of CLV + adjoint + scaler rows, 0 = all resident
  struct BudgetPlan {
    int n_seg = 0;  // 0 or 1: every CLV resident
    int n_phys = 0, n_boundary = 0;
    std::vector<int> seg_chunk;         // [n_seg + 1] chunk ranges of the segments
    std::vector<int> rec_begin;         // [n_chunks + 1] ranges of ops_rec per chunk
  } bp;
  DevBuf d_ops_b, d_ops_b_adj, d_ops_rec;
  hipGraphExec_t nr_graph = nullptr;
  int nr_graph_key[4] = {-1, -1, -1, -1};  // variant, mode, max_iters, paths
  const void *nr_graph_bufs[3] = {nullptr, nullptr, nullptr};
  NewtonState *h_nr_state = nullptr;  // pinned
  char *h_stage = nullptr;             // pinned staging for per-branch uploads
  size_t h_stage_bytes = 0, h_stage_off = 0;
  std::vector<double> h_st_sums;

  // dirty tracking
  bool model_dirty = true;
  std::vector<char> edge_dirty;  // P needs recompute
  std::vector<char> clv_dirty;   // [n_var]
  bool probs_dirty = true;
  bool cache_valid = false;
  int cache_variant = -1;
  double cached_total = 0.0;
  std::vector<double> cached_per_part;

  // device memory
  hipStream_t stream = nullptr;
  DevBuf d_tips, d_weights, d_tile_part, d_part_tile_begin;
  DevBuf d_V, d_Vinv, d_eval, d_rates, d_freqs, d_brlen;
  DevBuf d_P, d_Pf, d_PfT;
  DevBuf d_clv, d_scl, d_adj, d_adj_exp, d_Qf;
  DevBuf d_PA;  // 20-state FP64 form: P and P^T in operand order
  DevBuf d_Pa;  // 20-state FP32 form: likewise
  DevBuf d_ops_dirty, d_Qd;
  DevBuf d_ops_fwd, d_ops_adj;  // the walks' op lists
  // FP32 form, incremental evaluation: the invalid ops and their descriptor
  DevBuf d_ops_inc, d_netdesc_inc;
  DevBuf d_edge_use_begin, d_edge_use_list;
  DevBuf d_netdesc, d_work;  // FP32 form: this engine's NetDesc and (0, tile) work table
  DevBuf d_classes, d_class_dlogprob;
  DevBuf d_root_partials, d_beta, d_grad_partials, d_root_sums, d_use_sums;
  DevBuf d_site_seed;  // plain form: adjoint seed factor w / (C Ltilde) [root][site]
  DevBuf d_result;
  double *h_result = nullptr;  // pinned
  double *h_result_dev = nullptr;  // its device address
  // branch lengths as the P kernels read them: pinned, with its device address;
  // in flight from a launch to the next wait for the stream
  double *h_brlen = nullptr, *h_brlen_dev = nullptr;
  bool brlen_in_flight = false;
  ResultLayout rl{};
  size_t clv_elems_per_slot = 0;  // n_sites_pad * C * S

  // FP32 form: instantiated graphs of one evaluation, [variant][gradient],
  // valid for schedule `graph_version`
  hipGraphExec_t graph_exec[2][2][2] = {};  // [variant][gradient][P matrices updated in the graph]
  int graph_version = -1;

  // timing
  hipEvent_t ev_begin = nullptr, ev_end = nullptr;
  // event pairs around pruning (kind 0) and adjoint (kind 1) launches
  std::vector<hipEvent_t> ev_k[2];
  int n_k[2] = {0, 0};
  nrx_timing last_timing{};

  ~Engine();
};

}  // namespace nrx
