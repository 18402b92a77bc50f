// HIP kernels of the network-likelihood engine (gfx950).
//
// Data layout in HBM (one engine):
//   CLV arena   one row of S values per (variant, site, category): FP64 in the
//               order of row_offset, FP32 in the lane order of the walks
//               (Rows; Row20f)
//   scalers     int32 [n_variants][n_sites_pad], words as the walks describe
//   adjoints    as the CLVs
//   tips        uint8 (S <= 8) or uint32 (S = 20) state masks [n_tips][n_sites_pad]
//   P           real  [n_parts][n_edges][C][S][S], 20 states also in operand order
// Forward and reverse passes are walks of one wave (20 states forward: one per
// category) through the whole op list; the path kernels of the branch
// derivatives work on tiles of TILE = 64 sites with TILE * C threads.
#include <cfloat>
#include <cmath>
#include <map>
#include <mutex>
#include <stdexcept>
#include <type_traits>

#include "engine_state.hpp"

namespace nrx {

void HipCheck::check(hipError_t err, const char *what) {
  if (err != hipSuccess)
    throw std::runtime_error(std::string("HIP error ") + hipGetErrorString(err) + " in " + what);
}

namespace {

// libpll's per-site scaling constants (PLL_SCALE_THRESHOLD = 2^-256,
// PLL_SCALE_FACTOR = 2^256): a site is rescaled when all its entries are
// below the threshold; the scaler counts rescalings.
constexpr double SCALE_THRESHOLD = 0x1p-256;
constexpr double SCALE_FACTOR = 0x1p256;
constexpr double LOG_SCALE_THRESHOLD = -256.0 * 0.69314718055994530941723212145818;

template <int S>
struct TipType {
  using type = uint8_t;
};
template <>
struct TipType<20> {
  using type = uint32_t;
};

// Dynamic LDS is one untyped buffer per kernel (all extern __shared__
// declarations of a translation unit must agree on the type).
template <typename T>
__device__ __forceinline__ T *dyn_lds() {
  extern __shared__ double lds_dyn[];
  return reinterpret_cast<T *>(lds_dyn);
}

// Pointers read from a device-side descriptor table are generic (flat)
// pointers to the compiler; kernels that walk such tables retype them as
// global-memory pointers so CLV traffic uses global (not flat) loads and
// stores with scalar base addresses.
// (The host pass of this file never runs these kernels and has no address
// spaces, so the qualifier exists in the device pass only.)
#ifdef __HIP_DEVICE_COMPILE__
#define GAS __attribute__((address_space(1)))
#define CAS __attribute__((address_space(4)))
#else
#define GAS
#define CAS
#endif
template <typename T>
__device__ __forceinline__ GAS T *to_global(T *p) {
  return (GAS T *)p;
}
// Op tables never change during a launch: read through
// the constant address space they are fetched with scalar loads, whatever
// stores the kernel makes in between.
template <typename T>
__device__ __forceinline__ const CAS T *to_constant(const T *p) {
  return (const CAS T *)p;
}

// A thread's word in one slot of a per-slot arena (CLVs, adjoints,
// scalers, tip rows): the slot's base address is the same for the whole
// wave (scalar arithmetic) and the thread's offset into every slot is one
// fixed 32-bit byte offset, so each access is a scalar base plus that
// offset, with no per-lane 64-bit address arithmetic.
template <typename T>
__device__ __forceinline__ T *at(T *slot_base, uint32_t byte_off) {
  using B = typename std::conditional<std::is_const<T>::value, const char, char>::type;
  return reinterpret_cast<T *>(reinterpret_cast<B *>(slot_base) + byte_off);
}
#ifdef __HIP_DEVICE_COMPILE__
template <typename T>
__device__ __forceinline__ GAS T *at(GAS T *slot_base, uint32_t byte_off) {
  using B = typename std::conditional<std::is_const<T>::value, const char, char>::type;
  return reinterpret_cast<GAS T *>(reinterpret_cast<GAS B *>(slot_base) + byte_off);
}
#endif

// Cross-lane moves by DPP (a VALU operand modifier, no LDS round trip).
// Controls: quad_perm(p0, p1, p2, p3) = p0 | p1 << 2 | p2 << 4 | p3 << 6
// within each group of 4 lanes; row_shr:n = 0x110 + n shifts up by n lanes
// within each row of 16.  Lanes whose source lies outside the row read 0.
constexpr int DPP_XOR1 = 0xB1;  // quad_perm(1, 0, 3, 2): lane ^ 1
constexpr int DPP_XOR2 = 0x4E;  // quad_perm(2, 3, 0, 1): lane ^ 2
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}
// value of lane `off` apart within the C adjacent lanes of a site
template <int OFF, typename T>
__device__ __forceinline__ T lane_xor(T v) {
  if constexpr (OFF == 1)
    return dpp<DPP_XOR1>(v);
  else if constexpr (OFF == 2)
    return dpp<DPP_XOR2>(v);
  else
    return __shfl_xor(v, OFF);
}

template <int C>
__device__ __forceinline__ double cat_max(double m) {
  if constexpr (C > 1) m = fmax(m, lane_xor<1>(m));
  if constexpr (C > 2) m = fmax(m, lane_xor<2>(m));
  if constexpr (C > 4) m = fmax(m, lane_xor<4>(m));
  return m;
}
template <int C>
__device__ __forceinline__ double cat_sum(double m) {
  if constexpr (C > 1) m += lane_xor<1>(m);
  if constexpr (C > 2) m += lane_xor<2>(m);
  if constexpr (C > 4) m += lane_xor<4>(m);
  return m;
}

// Waits until every vector-memory load this wave issued has returned
// (s_waitcnt vmcnt(0); expcnt and lgkmcnt left unconstrained).  Placed after
// a load phase whose loads depend on runtime conditions, it leaves every
// path with no pending load, so the compiler needs no conservative waits
// before the next phase's loads.
__device__ __forceinline__ void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0F70); }

__device__ __forceinline__ double readlane(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Sum over the 64 lanes of a wave, in a fixed order (deterministic); the
// result is the same in every lane.  Row sums by four row_shr steps (lane
// 15 of each row of 16 ends with its row's sum S_r), then row_bcast:15
// (0x142: each row adds lane 15 of the row before it; lane 31 = S0 + S1,
// lane 63 = S2 + S3) and row_bcast:31 (0x143: rows 2 and 3 add lane 31), so
// lane 63 ends with the total: one lane read instead of four.
__device__ __forceinline__ double wave_sum(double v) {
  v += dpp<0x111>(v);
  v += dpp<0x112>(v);
  v += dpp<0x114>(v);
  v += dpp<0x118>(v);
  v += dpp<0x142>(v);
  v += dpp<0x143>(v);
  return readlane(v, 63);
}

// Sum over the 64 lanes, in every lane.
__device__ __forceinline__ double lane_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// Sums that carry their rounding errors along (Knuth's two-sum): the trees'
// log-likelihoods, large and nearly equal, are compared by their exponentials.
struct Exact {
  double s = 0.0, e = 0.0;
  __device__ __forceinline__ void add(double v) {
    const double t = s + v, b = t - s;
    e += (s - (t - b)) + (v - b);
    s = t;
  }
  // over the 64 lanes, in every lane
  __device__ __forceinline__ double lanes() {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const double v = __shfl_xor(s, off), w = __shfl_xor(e, off);
      add(v);
      e += w;
    }
    return value();
  }
  __device__ __forceinline__ double value() const { return fabs(s) < INFINITY ? s + e : s; }
};
// over the 256 threads, in thread 0
__device__ __forceinline__ double block_sum_exact(Exact x) {
  __shared__ double sh[4];
  const double v = x.lanes();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  Exact sum;
  for (int i = 0; i < 4; ++i) sum.add(sh[i]);
  return sum.value();
}

// Deterministic workgroup sum; result valid in thread 0.
template <int NT>
__device__ __forceinline__ double block_sum(double v, double *sh) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) sh[w] = v;
  __syncthreads();
  double r = 0.0;
  if (threadIdx.x == 0) {
#pragma unroll
    for (int i = 0; i < NT / 64; ++i) r += sh[i];
  }
  __syncthreads();
  return r;
}

// FP64 rows: S states of one (site, category), in the lane order of the
// matrix instructions, so that an access of the walks is one 512-byte span:
//   4 states   granules of 64 doubles (see k_forward_walk): [state 4][block
//              4][site 4], a block being one category of 4 sites.  A granule
//              holds all categories of 16 / C sites (8 categories: half the
//              categories of 4 sites, two granules in turn).
//   20 states  [16-site block][category][state 20][site 16]
// Sumtables of 4 states have the same order, of 20 states they are kept in
// pairs: [64 sites][category][pair 10][site 64][2].
// A row kept whole (32 or 160 bytes) would make every access of a wave touch
// the lines of all its 64 rows and use 16 bytes of each.
constexpr int PAIR_STRIDE = 128;  // doubles between a row's state pairs
constexpr int STATE_STRIDE = 16;  // doubles between a CLV row's entries
template <int S, int C>
__device__ __forceinline__ size_t row_offset(int64_t site, int c) {
  if constexpr (S != 4) {
    return static_cast<size_t>(((site >> 4) * C + c) * (S * STATE_STRIDE) + (site & 15));
  } else if constexpr (C == 8) {
    return static_cast<size_t>(((site >> 2) * 2 + (c >> 2)) * 64 + (c & 3) * 4 + (site & 3));
  } else {
    constexpr int SB = 4 / C;  // 4-site groups of a granule
    const int64_t g = site >> 2;
    return static_cast<size_t>(g / SB * 64 + (c * SB + g % SB) * 4 + (site & 3));
  }
}

template <int S>
__device__ __forceinline__ void load_clv(const double *__restrict__ p, double (&x)[S]) {
#pragma unroll
  for (int i = 0; i < S; ++i) x[i] = p[i * STATE_STRIDE];
}

// a sumtable row of (site, category)
template <int S, int C>
__device__ __forceinline__ size_t st_offset(int64_t site, int c) {
  if constexpr (S == 4)
    return row_offset<S, C>(site, c);
  else
    return static_cast<size_t>(((site >> 6) * C + c) * (S / 2 * PAIR_STRIDE) + (site & 63) * 2);
}
template <int S>
__device__ __forceinline__ void load_st(const double *__restrict__ p, double (&x)[S]) {
  if constexpr (S == 4) {
    load_clv<S>(p, x);
  } else {
#pragma unroll
    for (int i = 0; i < S / 2; ++i) {
      const double2 v = *reinterpret_cast<const double2 *>(p + i * PAIR_STRIDE);
      x[2 * i] = v.x;
      x[2 * i + 1] = v.y;
    }
  }
}
template <int S>
__device__ __forceinline__ void store_st(double *__restrict__ p, const double (&x)[S]) {
#pragma unroll
  for (int i = 0; i < S; ++i) p[S == 4 ? i * STATE_STRIDE : i / 2 * PAIR_STRIDE + i % 2] = x[i];
}

template <int S>
__device__ __forceinline__ void tip_vec(uint32_t mask, double (&x)[S]) {
#pragma unroll
  for (int i = 0; i < S; ++i) x[i] = ((mask >> i) & 1u) ? 1.0 : 0.0;
}

// y = M x for one S x S row-major matrix.  PIECES: two rows at a time, which
// keeps a matrix of 20 states, where it is in scalar registers, from spilling
// (sumtables of 2,000 patterns, 4 categories 91 us against 108; the kernel that
// evaluates them as well has more registers in use and is 3 % faster without).
template <int S, bool PIECES>
__device__ __forceinline__ void matvec(const double *__restrict__ M, const double (&x)[S],
                                       double (&y)[S]) {
#pragma unroll
  for (int i = 0; i < S; ++i) {
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < S; ++j) s = fma(M[i * S + j], x[j], s);
    y[i] = s;
    if (PIECES && i % 2) __builtin_amdgcn_sched_barrier(0);
  }
}

// y = M^T x (PIECES: row by row of M, which adds each sum's terms in the same order)
template <int S, bool PIECES>
__device__ __forceinline__ void matvec_t(const double *__restrict__ M, const double (&x)[S],
                                         double (&y)[S]) {
  if constexpr (PIECES) {
#pragma unroll
    for (int j = 0; j < S; ++j) y[j] = 0.0;
#pragma unroll
    for (int i = 0; i < S; ++i) {
#pragma unroll
      for (int j = 0; j < S; ++j) y[j] = fma(M[i * S + j], x[i], y[j]);
      if (i % 2) __builtin_amdgcn_sched_barrier(0);
    }
  } else {
#pragma unroll
    for (int j = 0; j < S; ++j) {
      double s = 0.0;
#pragma unroll
      for (int i = 0; i < S; ++i) s = fma(M[i * S + j], x[i], s);
      y[j] = s;
    }
  }
}

// ------------------------------------------------------------- P matrices
// Place of entry (i, k) of a matrix in its operand table: per chunk of four
// columns, rows 0-15 as [column][row 16], then rows 16-19 as [column][row 4].
__device__ __forceinline__ int aa_place(int i, int k) {
  return (k >> 2) * 80 + (i < 16 ? (k & 3) * 16 + i : 64 + (k & 3) * 4 + (i & 3));
}

// The same for FP32 (see mul20 there): rows 0-15 as [lane 16 q + m][step r] of
// column 4 r + q, then [lane] of the last step, m = 4 (i & 3) + (i >> 2); then
// rows 16-19 as [4 q + row][r] and [4 q + row].
__device__ __forceinline__ int aa_place32(int i, int k) {
  const int q = k & 3, r = k >> 2;
  const int lane = i < 16 ? 16 * q + 4 * (i & 3) + (i >> 2) : 4 * q + (i - 16);
  const int base = i < 16 ? 0 : 320, lanes = i < 16 ? 64 : 16;
  return base + (r < 4 ? lane * 4 + r : 4 * lanes + lane);
}

// exp(lambda_k r_c t_e) of the matrices that a workgroup of 256 entries has a
// part in, [matrix from the first][k]: one exponential per matrix and
// eigenvalue instead of one per entry and eigenvalue.  Ends with a barrier.
constexpr int PM_EXPS = 2 * AA_STATES;  // 256 entries lie in two matrices of 20 states
__device__ __forceinline__ void stage_pm_exps(const DevLayout &L, const double *__restrict__ ev,
                                              const double *__restrict__ rates, const double *__restrict__ lengths,
                                              int64_t total, double *s_ex) {
  const int S = L.S, C = L.C, SS = S * S;
  const int64_t first = static_cast<int64_t>(blockIdx.x) * blockDim.x, m0 = first / SS;
  const int64_t m1 = (min(first + blockDim.x, total) + SS - 1) / SS;
  for (int i = threadIdx.x; i < (m1 - m0) * S; i += blockDim.x) {
    const int64_t m = m0 + i / S;
    const int64_t p = m / (static_cast<int64_t>(C) * L.n_edges);
    const double lr = ev[p * S + i % S] * rates[p * C + m % C];
    s_ex[i] = exp(lr * lengths[m / C % L.n_edges]);
  }
  __syncthreads();
}

// P_{p,e,c} = V diag(exp(lambda r_c t_e)) V^-1 (libpll's
// pll_update_prob_matrices computes the same product from the same
// eigendecomposition).
__global__ void __launch_bounds__(256)
    k_pmatrices(DevLayout L, const double *__restrict__ V,
                            const double *__restrict__ Vinv, const double *__restrict__ ev,
                            const double *__restrict__ rates, const double *__restrict__ in_brlen,
                            double *__restrict__ brlen, double *__restrict__ P, float *__restrict__ Pf,
                            float *__restrict__ PfT, double *__restrict__ PA, float *__restrict__ Pa) {
  const int S = L.S, C = L.C;
  const int64_t total = static_cast<int64_t>(L.n_parts) * L.n_edges * C * S * S;
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  // (20 states, 80 edges x 4 categories: 13.3 -> 10.9 us; four exponentials per
  // entry of 4 states cost less than the barrier)
  __shared__ double s_ex[PM_EXPS];
  const bool staged = S == AA_STATES;
  if (staged) stage_pm_exps(L, ev, rates, in_brlen, total, s_ex);
  if (idx >= total) return;
  const double *ex = s_ex + (idx / (S * S) - static_cast<int64_t>(blockIdx.x) * 256 / (S * S)) * S;
  const int j = idx % S;
  const int i = (idx / S) % S;
  const int c = (idx / (S * S)) % C;
  const int e = (idx / (S * S * C)) % L.n_edges;
  const int p = idx / (static_cast<int64_t>(S) * S * C * L.n_edges);
  const double rt = rates[p * C + c];
  const double t = in_brlen[e];
  if (brlen && p == 0 && idx % (C * S * S) == 0) brlen[e] = t;
  const double *Vp = V + static_cast<size_t>(p) * S * S;
  const double *Wp = Vinv + static_cast<size_t>(p) * S * S;
  const double *lp = ev + static_cast<size_t>(p) * S;
  double a0 = 0.0;
  for (int k = 0; k < S; ++k) a0 += Vp[i * S + k] * (staged ? ex[k] : exp(lp[k] * rt * t)) * Wp[k * S + j];
  P[idx] = a0;
  if (Pf) Pf[idx] = static_cast<float>(a0);
  if (PfT) PfT[idx - (i * S + j) + (j * S + i)] = static_cast<float>(a0);
  if (PA) {
    double *tab = PA + idx / AA_MAT * AA_MATS;
    tab[aa_place(i, j)] = a0;
    tab[AA_MAT + aa_place(j, i)] = a0;
  }
  if (Pa) {
    float *tab = Pa + idx / AA_MAT * AA_MATS;
    tab[aa_place32(i, j)] = static_cast<float>(a0);
    tab[AA_MAT + aa_place32(j, i)] = static_cast<float>(a0);
  }
}

// ----------------------------------------------------------------- mixture
// Per partition: lnL_p = log sum_t P(t) exp(lnL_{p,t}) (AVERAGE) or
// max_t log P(t) + lnL_{p,t} (BEST) over root classes whose log-probability
// passes min_interesting_tree_logprob (ImprovedLoglikelihood.cpp:521-604);
// a max-shifted FP64 log-sum-exp stands in for the reference's MPFR sum.
// Also produces the adjoint seeds beta[p][root CLV] = sum of the class
// weights d lnL_p / d lnL_{p,t}, and d lnL / d p_r.
// The inputs (root sums, class data, d log P / d p) and alpha are staged in
// LDS when they fit in MIX_LDS_DOUBLES (the usual case), so the serial loops
// over classes read LDS instead of making a memory round trip per class;
// otherwise the same code runs on the global arrays.  The arithmetic and
// its order are the same either way.
constexpr int MIX_LDS_DOUBLES = 6144;  // 48 KiB
constexpr int MIX_PARTIALS = 2048, MIX_ROWS = 16;  // see launch_mixture
__host__ __device__ inline int mixture_lds_doubles(int n_root, int nc, int R, int P) {
  return n_root * P + 2 * nc + nc * P + nc * R;
}
__device__ void mixture_body(const DevLayout &L, int n_root, int nc, int R, int variant,
                             const DevClass *__restrict__ classes,
                             const double *__restrict__ class_dlogprob,
                             const double *__restrict__ root_sums, double *__restrict__ beta,
                             double *__restrict__ res, double *__restrict__ host, const ResultLayout &rl) {
  __shared__ double per_part[64];
  // results, for the device and (unless null) straight into the host's pinned block
  auto put = [&](int i, double v) {
    res[i] = v;
    if (host) host[i] = v;
  };
  const int P = L.n_parts;  // <= 64 (checked on the host)
  const bool staged = mixture_lds_doubles(n_root, nc, R, P) <= MIX_LDS_DOUBLES;
  // class k: log-probability lp[k], root index ri[k], use flag cu[k]
  const double *rs = root_sums, *cdl = class_dlogprob;
  double *alpha = res + rl.alpha;
  double *lp = nullptr;
  int *ri = nullptr, *cu = nullptr;
  if (staged) {
    double *sm = dyn_lds<double>();
    double *s_rs = sm, *s_lp = s_rs + n_root * P, *s_ri = s_lp + nc, *s_alpha = s_ri + nc, *s_cdl = s_alpha + nc * P;
    for (int i = threadIdx.x; i < n_root * P; i += blockDim.x) s_rs[i] = root_sums[i];
    for (int i = threadIdx.x; i < nc * R; i += blockDim.x) s_cdl[i] = class_dlogprob[i];
    int *s_ri_int = reinterpret_cast<int *>(s_ri), *s_cu = s_ri_int + nc;
    for (int k = threadIdx.x; k < nc; k += blockDim.x) {
      const DevClass cl = classes[k];
      s_lp[k] = cl.logprob;
      s_ri_int[k] = cl.root_index;
      s_cu[k] = cl.use;
    }
    rs = s_rs;
    cdl = s_cdl;
    alpha = s_alpha;
    lp = s_lp;
    ri = s_ri_int;
    cu = s_cu;
    __syncthreads();
  }
  const auto logprob = [&](int k) { return staged ? lp[k] : classes[k].logprob; };
  const auto used = [&](int k) { return (staged ? cu[k] : classes[k].use) != 0; };
  const auto root_of = [&](int k) { return staged ? ri[k] : classes[k].root_index; };
  // per-(root CLV, partition) tree lnL and per-class copies
  for (int idx = threadIdx.x; idx < n_root * P; idx += blockDim.x) {
    const int r = idx / P, p = idx % P;
    put(rl.root_logl + p * n_root + r, rs[idx]);
  }
  for (int idx = threadIdx.x; idx < nc * P; idx += blockDim.x) {
    const int p = idx / nc, k = idx % nc;
    const int r = root_of(k);
    put(rl.tree_logl + p * nc + k, r >= 0 ? rs[r * P + p] : 0.0);
  }
  // a group of lanes per partition, lanes over the classes: as many lanes as
  // there are classes, at most a wave, so that many partitions with few trees
  // are done in few rounds (64 partitions, 4 trees: 6.6 us, 34 with a wave each)
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, n_waves = blockDim.x >> 6;
  int width = 64;
  while (width > 1 && width / 2 >= nc) width /= 2;
  const int member = threadIdx.x & (width - 1);
  for (int p0 = 0; p0 < P; p0 += blockDim.x / width) {
    const int p = p0 + threadIdx.x / width, n = p < P ? nc : 0;  // (every lane takes part in the exchanges)
    // best class (first maximum in class order)
    double best = -INFINITY;
    int arg = -1;
    for (int k = member; k < n; k += width) {
      const double v = used(k) ? logprob(k) + rs[root_of(k) * P + p] : -INFINITY;
      if (v > best) {
        best = v;
        arg = k;
      }
    }
    for (int off = width / 2; off > 0; off >>= 1) {
      const double v = __shfl_xor(best, off);
      const int k = __shfl_xor(arg, off);
      if (v > best || (v == best && k >= 0 && (arg < 0 || k < arg))) {
        best = v;
        arg = k;
      }
    }
    double sum = 0.0;
    for (int k = member; k < n; k += width) {
      double a = 0.0;
      if (variant == 1)
        a = k == arg ? 1.0 : 0.0;
      else if (used(k) && best > -INFINITY)
        a = exp(logprob(k) + rs[root_of(k) * P + p] - best);
      alpha[p * nc + k] = a;
      sum += a;
    }
    for (int off = width / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
    if (variant != 1)
      for (int k = member; k < n; k += width) alpha[p * nc + k] = sum > 0.0 ? alpha[p * nc + k] / sum : 0.0;
    if (member == 0 && p < P) {
      per_part[p] = variant == 1 ? best : best + log(sum);
      put(rl.per_part + p, per_part[p]);
    }
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < nc * P; idx += blockDim.x) put(rl.alpha + idx, alpha[idx]);
  for (int idx = threadIdx.x; idx < n_root * P; idx += blockDim.x) {
    const int p = idx / n_root, r = idx % n_root;
    double b = 0.0;
#pragma unroll 8
    for (int k = 0; k < nc; ++k) b += root_of(k) == r ? alpha[p * nc + k] : 0.0;
    beta[p * n_root + r] = b;
  }
  for (int r = wave; r < R; r += n_waves) {
    double g = 0.0;
    for (int idx = lane; idx < nc * P; idx += 64) g += alpha[idx] * cdl[static_cast<size_t>(idx % nc) * R + r];
    g = lane_sum(g);
    if (lane == 0) put(rl.dprob + r, g);
  }
  if (threadIdx.x == 0) {
    double tot = 0.0;
    for (int p = 0; p < P; ++p) tot += per_part[p];
    put(rl.total, tot);
  }
}

__global__ void __launch_bounds__(256)
    k_mixture(DevLayout L, int n_root, int nc, int R, int variant,
              const DevClass *__restrict__ classes, const double *__restrict__ class_dlogprob,
              double *__restrict__ root_sums, double *__restrict__ beta,
              double *__restrict__ res, double *__restrict__ host, ResultLayout rl,
              const double *__restrict__ root_partials, int pw,
              const int32_t *__restrict__ part_tile_begin) {
  if (root_partials) {
    // few partials: summed here, a wave per (root CLV, partition)
    const int P = L.n_parts, lane = threadIdx.x & 63;
    for (int i = threadIdx.x >> 6; i < n_root * P; i += blockDim.x >> 6) {
      const int p = i % P;
      const double *in = root_partials + static_cast<int64_t>(i / P) * L.n_tiles * pw;
      const int t1 = part_tile_begin[p + 1] * pw;
      Exact sum;
#pragma unroll 8
      for (int t = part_tile_begin[p] * pw + lane; t < t1; t += 64) sum.add(in[t]);
      const double s = sum.lanes();
      if (lane == 0) root_sums[i] = s;
    }
    __threadfence_block();
    __syncthreads();
  }
  mixture_body(L, n_root, nc, R, variant, classes, class_dlogprob, root_sums, beta, res, host, rl);
}

// ------------------------------------------------ 4 states, FP64 plain form
// The pruning walks on the matrix cores.  v_mfma_f64_4x4x4 multiplies four
// independent 4 x 4 blocks: A lane (l & 3, block, l >> 4) = A[row][k], B lane
// = B[k = l >> 4][col = l & 3], D lane = D[row = l >> 4][col = l & 3], block =
// (l >> 2) & 3.  With blocks = rate categories (and 4-site groups when there
// are fewer than 4 categories), rows = states and columns = sites, D has B's
// layout: a product of a CLV is itself a CLV operand, and the stored rows are
// these registers (see row_offset), one coalesced 512-byte access per 16
// rows.  P is one register per lane (a 512-byte load of all categories of an
// edge) instead of 16 LDS reads per lane, and r_c Q stays in one.
//
// One wave walks its sites through the whole op list, in depth-first order,
// and hands a CLV (forward) or an adjoint (reverse) to its consumer through
// an LDS slot of the wave; a row travels through HBM only where no slot was
// free (schedule.cpp).  Every CLV is still stored once: the reverse sweep,
// later incremental passes and the branch derivatives read it.  The loads of
// an op are issued one op ahead.
//
// NQ granules (64 (state, site, category) entries each) per wave: 4 share
// each matrix load, sum and scalar step among 16 sites at 4 categories; 2 or
// 1 spread few sites over more waves.
template <int C, int NQ>
struct Quad {
  static constexpr int SPW = 16 * NQ / C;    // sites of a wave
  static constexpr int NA = C == 8 ? 2 : 1;  // matrix registers per edge (halves of 8 categories)
  static constexpr int SB = C >= 4 ? 1 : 4 / C;  // 4-site groups of a granule
  static constexpr int NW = SPW / 4;         // 4-site tip words of a wave
  static __device__ __forceinline__ int cat(int lane, int h) { return ((lane >> 2) & 3) / SB + 4 * h; }
  static __device__ __forceinline__ constexpr int half(int q) { return C == 8 ? q & 1 : 0; }
  // first 4-site group of granule q, and a lane's site within the wave
  static __device__ __forceinline__ constexpr int group(int q) { return C == 8 ? q >> 1 : q * SB; }
  static __device__ __forceinline__ int site(int lane, int q) {
    return 4 * (group(q) + ((lane >> 2) & 3) % SB) + (lane & 3);
  }
};

__device__ __forceinline__ double mfma4(double a, double b, double c) {
  return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}

// Granule q of a tip's 0/1 vectors; lane w of `words` holds the masks of the
// wave's 4-site group w.
template <int C, int NQ>
__device__ __forceinline__ double tip_entry(uint32_t words, int q, int lane, int shift) {
  using W = Quad<C, NQ>;
  uint32_t w;
  if constexpr (W::SB == 1)
    w = __builtin_amdgcn_readlane(words, W::group(q));
  else
    w = __shfl(words, W::group(q) + ((lane >> 2) & 3) % W::SB);
  return __hiloint2double(-static_cast<int>((w >> shift) & 1u) & 0x3FF00000, 0);  // 1.0 or 0.0
}

// Sites of the wave (bit s = site s) all of whose entries' bits are set in
// the granules' lane masks.
template <int C, int NQ>
__device__ __forceinline__ uint64_t whole_sites(const uint64_t (&m)[NQ]) {
  using W = Quad<C, NQ>;
  uint64_t sites = 0;
#pragma unroll
  for (int q = 0; q < NQ; q += W::NA) {
    uint64_t t = m[q];
    if constexpr (C == 8) t &= m[q + 1];
    t &= t >> 32;
    t &= t >> 16;  // over the states
    if constexpr (C >= 4) {
      t &= t >> 8;
      t &= t >> 4;
      t &= 0xF;
    } else if constexpr (C == 2) {
      t &= t >> 8;
      t &= 0xFF;
    } else {
      t &= 0xFFFF;
    }
    sites |= t << (4 * W::group(q));
  }
  return sites;
}

// Sums over the 64 lanes of two values at once: lane 31 ends with a's total,
// lane 63 with b's (the halves of the wave trade one value each, then five
// DPP steps serve both).
__device__ __forceinline__ double pair_wave_sum(double a, double b) {
  const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
  double v = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
  v += dpp<0x111>(v);
  v += dpp<0x112>(v);
  v += dpp<0x114>(v);
  v += dpp<0x118>(v);
  v += dpp<0x142>(v);
  return v;
}

// A use of every register of x here: the wait for the loads into them goes
// here, ahead of the next op's loads, whose count a condition may change.
template <typename T, int N>
__device__ __forceinline__ void arrive(T (&x)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(x[i]));
}

// Brings a walk's P matrices (one 128-byte line each) and op list into the
// XCD's L2: the kernels before it left them in other XCDs, and every op of
// the walk would otherwise wait for its matrices' first read from memory.
// Each wave touches one 64-line piece; workgroups b, b + 8, ... share an XCD.
__device__ __forceinline__ uint32_t warm_l2(const GAS double *P, int n_mats, const DevOp *ops, int n_ops, int lane) {
  const int op_lines = (n_ops * static_cast<int>(sizeof(DevOp)) + 127) / 128;
  const int pieces = (n_mats + op_lines + 63) / 64;
  const int line = (static_cast<int>(blockIdx.x >> 3) % pieces) * 64 + lane;
  uint32_t v = 0;
  if (line < n_mats)
    v = *reinterpret_cast<const GAS uint32_t *>(P + line * 16);
  else if (line < n_mats + op_lines)
    v = *(reinterpret_cast<const GAS uint32_t *>(to_global(ops)) + (line - n_mats) * 32);
  return v;
}

// One op's descriptor in scalar registers, fetched whole: read field by
// field where it is used, every field would be a scalar load with a wait.
typedef int32_t i32x8 __attribute__((ext_vector_type(8), aligned(16)));
typedef int32_t i32x4 __attribute__((ext_vector_type(4), aligned(16)));
struct OpRegs {
  i32x8 a;
  i32x4 b;
  __device__ __forceinline__ uint32_t out() const { return a[0]; }
  __device__ __forceinline__ int nk() const { return a[1]; }
  __device__ __forceinline__ int32_t kid(int k) const { return a[2 + k]; }
  __device__ __forceinline__ uint32_t edge(int k) const { return a[4 + k]; }
  __device__ __forceinline__ int root() const { return a[6]; }
  __device__ __forceinline__ int flags() const { return a[7]; }
  __device__ __forceinline__ bool has(int f0, int f1, int k) const { return (a[7] & (k == 0 ? f0 : f1)) != 0; }
  __device__ __forceinline__ int gslot() const { return b[0]; }
  __device__ __forceinline__ int slot(int u) const { return (b[2] >> (8 * u)) & 255; }
};
static_assert(sizeof(DevOp) == 48, "OpRegs restates DevOp");
__device__ __forceinline__ OpRegs fetch_op(const CAS DevOp *ops, int t) {
  OpRegs r;
  r.a = *reinterpret_cast<const CAS i32x8 *>(ops + t);
  r.b = *reinterpret_cast<const CAS i32x4 *>(reinterpret_cast<const CAS int32_t *>(ops + t) + 8);
  return r;
}
__device__ __forceinline__ void arrive(OpRegs &r) { asm volatile("" : "+s"(r.a), "+s"(r.b)); }

// A lane's byte offset, hidden from the optimiser: it would otherwise keep
// base + offset of every buffer as a register pair across the op loop and add
// each row to that, instead of addressing with a scalar base plus the offset.
__device__ __forceinline__ uint32_t opaque(uint32_t x) {
  asm volatile("" : "+v"(x));
  return x;
}

template <int C, int NQ>
struct FwdIn4 {
  double A[2 * Quad<C, NQ>::NA];  // P of both children
  double x[2 * NQ];               // children read from HBM
  uint32_t raw[2];                // the children's scaler words, or tip mask words
};

// Scaler words: 2 x (rescalings below and at this CLV) + (rescaled here).
//
// Bound: HBM (a CLV written per op; 50 taxa, 41,345 patterns: 1.01 GB of traffic
// in 0.222 ms, 4.5 TB/s; a thread per row with P in LDS and CLVs through HBM took
// 0.311 + 0.023 ms for the root sums), or a wave's chain of ops for few sites.
template <int S, int C, int NQ>
__global__ void __launch_bounds__(64, 3)
    k_forward_walk(const DevOp *__restrict__ ops_, int n_ops, int n_slots, DevLayout L, double *__restrict__ clv_,
                   int32_t *__restrict__ scl_, const uint8_t *__restrict__ tips_, const double *__restrict__ P_,
                   const double *__restrict__ freqs, const double *__restrict__ weights,
                   const int32_t *__restrict__ tile_part, double *__restrict__ root_partials,
                   double *__restrict__ seed) {
  static_assert(S == 4, "20 states take k_forward_level_aa");
  using W = Quad<C, NQ>;
  constexpr int NA = W::NA, SPW = W::SPW;
  const CAS DevOp *ops = to_constant(ops_);
  const int lane = threadIdx.x, state = lane >> 4;
  const uint64_t n = L.n_sites_pad, row = n * (C * 4);
  const int64_t site0 = static_cast<int64_t>(blockIdx.x) * SPW;
  const int part = to_constant(tile_part)[site0 / TILE];
  double *slots = dyn_lds<double>();  // [slot][granule][lane], then the slots' scaler words
  uint32_t *slot_scl = reinterpret_cast<uint32_t *>(slots + n_slots * (NQ * 64));
  GAS double *clv = to_global(clv_) + static_cast<int64_t>(blockIdx.x) * (NQ * 64);
  GAS int32_t *scl = to_global(scl_) + site0;
  const GAS uint8_t *tips = to_global(tips_) + site0;
  const GAS double *P = to_global(P_) + static_cast<int64_t>(part) * L.n_edges * (C * 16);
  const uint32_t off = lane * 8, soff = (lane % SPW) * 4, woff = (lane % W::NW) * 4;
  const int tip_shift = 8 * (lane & 3) + state;
  uint32_t aoff[NA];
#pragma unroll
  for (int h = 0; h < NA; ++h) aoff[h] = (W::cat(lane, h) * 16 + (lane & 3) * 4 + state) * 8;
  const double w = weights[site0 + lane % SPW];
  const double pi_c = freqs[part * 4 + state] * (1.0 / C);

  auto load = [&](const OpRegs &op, FwdIn4<C, NQ> &in) {
    const uint32_t o = opaque(off);
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int h = 0; h < NA; ++h) in.A[k * NA + h] = *at(P + op.edge(k) * (C * 16), opaque(aoff[h]));
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      // a tip's mask words, or the row's scaler words (a one-child op's
      // second child stands for its first)
      const int32_t kid = k < op.nk() ? op.kid(k) : op.kid(0);
      const GAS char *tip = reinterpret_cast<const GAS char *>(tips) + static_cast<uint32_t>(~kid) * n;
      const GAS char *word = reinterpret_cast<const GAS char *>(scl) + static_cast<uint32_t>(kid) * (n * 4);
      in.raw[k] = *at(reinterpret_cast<const GAS uint32_t *>(kid < 0 ? tip : word), kid < 0 ? woff : soff);
    }
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (op.has(OP_LOAD0, OP_LOAD1, k))
#pragma unroll
        for (int q = 0; q < NQ; ++q)
          in.x[k * NQ + q] = *at(clv + static_cast<uint32_t>(op.kid(k)) * row, o + q * 512);
  };
  // y = P x of child k
  auto child = [&](const OpRegs &op, FwdIn4<C, NQ> &in, int k, double (&y)[NQ], uint32_t &count) {
    uint32_t below = in.raw[k] >> 1;
    if (op.kid(k) < 0) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) in.x[k * NQ + q] = tip_entry<C, NQ>(in.raw[k], q, lane, tip_shift);
      below = 0;
    }
    if (op.has(OP_PASS_KID0, OP_PASS_KID1, k)) {
      const int slot = op.slot(k);
#pragma unroll
      for (int q = 0; q < NQ; ++q) in.x[k * NQ + q] = slots[slot * (NQ * 64) + q * 64 + lane];
      below = slot_scl[slot * 64 + lane] >> 1;
    }
    count += below;
#pragma unroll
    for (int q = 0; q < NQ; ++q) y[q] = mfma4(in.A[k * NA + W::half(q)], in.x[k * NQ + q], 0.0);
  };
  // op t with its inputs `in`; loads those of op t + 1 and fetches op t + 2
  auto step = [&](int t, const OpRegs &op, OpRegs &ahead, OpRegs &after, FwdIn4<C, NQ> &in, FwdIn4<C, NQ> &next) {
    arrive(in.A);
    arrive(in.x);
    arrive(in.raw);
    arrive(ahead);
    __builtin_amdgcn_sched_barrier(0);
    load(ahead, next);
    after = fetch_op(ops, min(t + 2, n_ops - 1));
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t o = opaque(off);
    double v[NQ];
    uint32_t count = 0;
    child(op, in, 0, v, count);
    if (op.nk() == 2) {
      double y[NQ];
      child(op, in, 1, y, count);
#pragma unroll
      for (int q = 0; q < NQ; ++q) v[q] *= y[q];
    }
    // a site is rescaled when all its entries are below the threshold; most
    // ops have no entry there at all
    uint32_t word = count << 1;
    uint64_t small[NQ], any = 0;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      small[q] = __builtin_amdgcn_ballot_w64(v[q] < SCALE_THRESHOLD);
      any |= small[q];
    }
    if (any) {
      const uint64_t sites = whole_sites<C, NQ>(small);
#pragma unroll
      for (int q = 0; q < NQ; ++q)
        if ((sites >> W::site(lane, q)) & 1) v[q] *= SCALE_FACTOR;
      if ((sites >> (lane % SPW)) & 1) word += 3;
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) *at(clv + op.out() * row, o + q * 512) = v[q];
    *at(scl + op.out() * n, opaque(soff)) = static_cast<int32_t>(word);  // lanes of a site store the same word
    if (op.flags() & OP_A_PASS) {
      const int slot = op.slot(2);
#pragma unroll
      for (int q = 0; q < NQ; ++q) slots[slot * (NQ * 64) + q * 64 + lane] = v[q];
      slot_scl[slot * 64 + lane] = word;
    }
    if (op.root() >= 0) {
      // site likelihoods Ltilde = (1/C) sum_c pi . x: the sum over the states
      // as a product with rows pi / C (every row of D holds it), then over
      // the categories; lane l takes site l % SPW
      double t_site = 0.0;
#pragma unroll
      for (int q = 0; q < NQ; q += NA) {
        double t = mfma4(pi_c, v[q], 0.0);
        if constexpr (C == 8) t += mfma4(pi_c, v[q + 1], 0.0);
        if constexpr (C >= 4) t += dpp<0x124>(t);  // row_ror:4
        if constexpr (C >= 2) t += dpp<0x128>(t);  // row_ror:8
        if ((lane % SPW) / (4 * W::SB) == q / NA) t_site = t;
      }
      const double wk = lane < SPW ? w : 0.0;
      const double val = wk != 0.0 ? wk * (log(t_site) + static_cast<double>(word >> 1) * LOG_SCALE_THRESHOLD) : 0.0;
      const double sum = wave_sum(val);
      if (lane == 0) root_partials[static_cast<int64_t>(op.root()) * gridDim.x + blockIdx.x] = sum;
      // the adjoint's seed factor at this root and site, w / (C Ltilde)
      seed[op.root() * n + site0 + lane % SPW] = w != 0.0 ? w * (1.0 / C) / t_site : 0.0;
    }
  };
  OpRegs op0 = fetch_op(ops, 0), op1 = fetch_op(ops, min(1, n_ops - 1));
  uint32_t warm[1] = {warm_l2(P, L.n_edges * C, ops_, n_ops, lane)};
  FwdIn4<C, NQ> a;
  load(op0, a);
  arrive(warm);
  // complete before the loop, so that the waits inside it count only what the
  // step before issued (its stores need not have ended)
  arrive(a.A);
  arrive(a.x);
  arrive(a.raw);
  for (int t = 0; t < n_ops; t += 2) {
    FwdIn4<C, NQ> b, c;  // what an op does not load stays undefined: nothing is carried over
    OpRegs op2, op3;
    step(t, op0, op1, op2, a, b);
    if (t + 1 >= n_ops) break;
    step(t + 1, op1, op2, op3, b, c);
    a = c;
    op0 = op2;
    op1 = op3;
  }
}

// The factor that a displayed-tree root seeds at a site: beta w / (C Ltilde).
// A tree without weight seeds nothing, also where its likelihood is zero.
__device__ __forceinline__ double root_seed(double beta, double factor) { return beta != 0.0 ? beta * factor : 0.0; }

// Reverse pruning in push form.  For op q with children k (edge e_k, CLV
// x_k, y_k = P_k x_k) and rescale factor F = 2^256 where q was rescaled:
//   z_k      = Abar_q * F * prod_{j != k} y_j
//   Abar_k  += P_k^T z_k            (delivered to child k)
//   dJ/dt_k += z_k . (P'_k x_k),    P'_k x_k = r_c Q y_k
// where J = sum_p sum_t beta_{p,t} lnL_{p,t} and Abar is the derivative of
// J w.r.t. the *scaled* CLV values; a root CLV adds the seed
// beta * w_s * (1/C) pi_i / Ltilde_s.  The ops are walked backwards: every
// consumer of a CLV delivers before the CLV's own op runs, the first one
// writes and later ones accumulate (in the matrix instruction's C operand).
// The same lane owns an entry in every op: no atomics, no barriers,
// deterministic.
template <int C, int NQ>
struct AdjIn4 {
  double A[2 * Quad<C, NQ>::NA], AT[2 * Quad<C, NQ>::NA];  // P and P^T of both children
  double x[2 * NQ];    // inner children
  double a[NQ];        // own adjoint, where no slot holds it
  double sd[1];        // seed factor of a displayed-tree root (lane l: site l % SPW)
  uint32_t raw[2];     // tip children's mask words
  uint32_t word[1];    // own scaler word
};

// Bound: HBM (every inner child's CLV once per use; 50 taxa, 41,345 patterns:
// 1.67 GB of traffic in 0.317 ms, 5.3 TB/s, as a large copy; with P in LDS and
// every adjoint through HBM 2.99 GB in 0.648 ms).
//
// MODEL: instead of the gradient's shares, per use, the sums over the wave's
// sites of z x^T (dJ/dP), one entry per lane of a granule, and per root those of
// the frequencies' direct share, f x with f = beta w / (C Ltilde) (r_part,
// [root][wave][4]).  Both are products over sites: z and x are transposed by a
// product with the identity, which is exact, and multiplied (41,345 patterns,
// 138 ops: 0.39 ms, the gradient's walk 0.32, and 0.08 for k_model_reduce; a pass
// of its own over stored adjoints and CLVs took 0.85 ms, and storing the adjoints
// 0.10).  The sums of
// child k go to [k][NA][64] of the wave's part of the op's own adjoint row: no
// one reads that any more, it holds both (NQ >= 2 NA), and they take no memory
// of their own (a buffer for them was a quarter of the CLVs and adjoints).
template <int C, int NQ, bool MODEL>
__device__ __forceinline__ void adjoint_walk4(
    const DevOp *__restrict__ ops_, int n_ops, const DevLayout &L, const double *__restrict__ clv_,
    const int32_t *__restrict__ scl_, double *__restrict__ adj_, const uint8_t *__restrict__ tips_,
    const double *__restrict__ P_, const double *__restrict__ Qd, const double *__restrict__ freqs,
    const double *__restrict__ seed, const int32_t *__restrict__ tile_part, const double *__restrict__ beta, int n_root,
    int n_uses, double *__restrict__ grad_partials, double *__restrict__ r_part) {
  using W = Quad<C, NQ>;
  constexpr int NA = W::NA, SPW = W::SPW;
  static_assert(!MODEL || NQ >= 2 * NA);
  const CAS DevOp *ops = to_constant(ops_);
  const int lane = threadIdx.x, state = lane >> 4;
  const uint64_t n = L.n_sites_pad, row = n * (C * 4);
  const int64_t site0 = static_cast<int64_t>(blockIdx.x) * SPW;
  const int part = to_constant(tile_part)[site0 / TILE];
  double *ring = dyn_lds<double>();
  double *slots = ring + GRAD_RING;  // [slot][granule][lane]
  const GAS double *clv = to_global(clv_) + static_cast<int64_t>(blockIdx.x) * (NQ * 64);
  GAS double *adj = to_global(adj_) + static_cast<int64_t>(blockIdx.x) * (NQ * 64);
  const GAS int32_t *scl = to_global(scl_) + site0;
  const GAS uint8_t *tips = to_global(tips_) + site0;
  const GAS double *P = to_global(P_) + static_cast<int64_t>(part) * L.n_edges * (C * 16);
  GAS double *grad = to_global(grad_partials) + static_cast<int64_t>(blockIdx.x) * n_uses;
  const uint32_t off = lane * 8, soff = (lane % SPW) * 4, woff = (lane % W::NW) * 4;
  const int tip_shift = 8 * (lane & 3) + state;
  uint32_t aoff[NA], toff[NA];
  double Q[NA];
#pragma unroll
  for (int h = 0; h < NA; ++h) {
    aoff[h] = (W::cat(lane, h) * 16 + (lane & 3) * 4 + state) * 8;
    toff[h] = (W::cat(lane, h) * 16 + state * 4 + (lane & 3)) * 8;
    Q[h] = Qd[part * (C * 16) + aoff[h] / 8];
  }
  const double pi = freqs[part * 4 + state];

  auto load = [&](const OpRegs &op, AdjIn4<C, NQ> &in) {
    const uint32_t o = opaque(off);
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int h = 0; h < NA; ++h) {
        in.A[k * NA + h] = *at(P + op.edge(k) * (C * 16), opaque(aoff[h]));
        in.AT[k * NA + h] = *at(P + op.edge(k) * (C * 16), opaque(toff[h]));
      }
    in.word[0] = static_cast<uint32_t>(*at(scl + op.out() * n, opaque(soff)));
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      // (a one-child op's second child stands for its first)
      const int32_t kid = k < op.nk() ? op.kid(k) : op.kid(0);
      if (kid < 0)
        in.raw[k] = *at(reinterpret_cast<const GAS uint32_t *>(tips + static_cast<uint32_t>(~kid) * n), opaque(woff));
      else if (k < op.nk())
#pragma unroll
        for (int q = 0; q < NQ; ++q) in.x[k * NQ + q] = *at(clv + static_cast<uint32_t>(kid) * row, o + q * 512);
    }
    if ((op.flags() & (OP_HAS_CONSUMERS | OP_A_PASS | OP_A_LATE)) == OP_HAS_CONSUMERS)
#pragma unroll
      for (int q = 0; q < NQ; ++q) in.a[q] = *at(adj + op.out() * row, o + q * 512);
    if (op.root() >= 0) in.sd[0] = seed[op.root() * n + site0 + lane % SPW];
  };
  // back-propagated vectors to child k's adjoint
  auto deliver = [&](const OpRegs &op, const AdjIn4<C, NQ> &in, int k, const double (&z)[NQ], double (&b)[NQ]) {
    const bool first = op.has(OP_FIRST_KID0, OP_FIRST_KID1, k), pass = op.has(OP_PASS_KID0, OP_PASS_KID1, k);
    double *slot = slots + op.slot(k) * (NQ * 64) + lane;
    GAS double *dst = adj + static_cast<uint32_t>(op.kid(k)) * row;
    if (pass && !first) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) b[q] = slot[q * 64];
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) b[q] = mfma4(in.AT[k * NA + W::half(q)], z[q], b[q]);
    const uint32_t o = opaque(off);
    if (pass) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) slot[q * 64] = b[q];
    } else {
#pragma unroll
      for (int q = 0; q < NQ; ++q) *at(dst, o + q * 512) = b[q];
    }
  };
  auto product = [&](const OpRegs &op, AdjIn4<C, NQ> &in, int k, double (&y)[NQ]) {
    if (op.kid(k) < 0)
#pragma unroll
      for (int q = 0; q < NQ; ++q) in.x[k * NQ + q] = tip_entry<C, NQ>(in.raw[k], q, lane, tip_shift);
#pragma unroll
    for (int q = 0; q < NQ; ++q) y[q] = mfma4(in.A[k * NA + W::half(q)], in.x[k * NQ + q], 0.0);
  };
  int flushed = ops[n_ops - 1].gslot[0];  // the sweep's first gradient row
  // op t with its inputs `in`; loads those of op t - 1 and fetches op t - 2
  auto step = [&](int t, const OpRegs &op, OpRegs &ahead, OpRegs &after, AdjIn4<C, NQ> &in, AdjIn4<C, NQ> &next) {
    arrive(in.A);
    arrive(in.AT);
    arrive(in.x);
    arrive(in.a);
    arrive(in.sd);
    arrive(in.raw);
    arrive(in.word);
    arrive(ahead);
    __builtin_amdgcn_sched_barrier(0);
    // what the children's adjoints hold already, where no slot does (the
    // deliveries before this op's are stores of this wave, so in order)
    double acc[2][NQ];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) acc[k][q] = 0.0;
      if (op.has(OP_ACC0, OP_ACC1, k))
#pragma unroll
        for (int q = 0; q < NQ; ++q) acc[k][q] = *at(adj + static_cast<uint32_t>(op.kid(k)) * row, opaque(off) + q * 512);
    }
    load(ahead, next);
    after = fetch_op(ops, max(t - 2, 0));
    __builtin_amdgcn_sched_barrier(0);
    double (&a)[NQ] = in.a;
    if (op.flags() & OP_A_PASS) {
      const double *slot = slots + op.slot(2) * (NQ * 64) + lane;
#pragma unroll
      for (int q = 0; q < NQ; ++q) a[q] = slot[q * 64];
    } else if (op.flags() & OP_A_LATE) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) a[q] = *at(adj + op.out() * row, opaque(off) + q * 512);
      wait_loads();
    } else if (!(op.flags() & OP_HAS_CONSUMERS)) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) a[q] = 0.0;
    }
    if (op.root() >= 0) {
      // seed beta * w * (1/C) pi_i / Ltilde at a displayed-tree root
      const double f = root_seed(beta[part * n_root + op.root()], in.sd[0]);
      if constexpr (MODEL) {
        double r = 0.0;
#pragma unroll
        for (int q = 0; q < NQ; ++q)
          r = fma(__shfl(f, W::site(lane, q)), *at(clv + op.out() * row, off + q * 512), r);
        r += dpp<0x121>(r);  // over the 16 lanes of a state: row_ror 1, 2, 4, 8
        r += dpp<0x122>(r);
        r += dpp<0x124>(r);
        r += dpp<0x128>(r);
        if ((lane & 15) == 0) *at(to_global(r_part) + (static_cast<int64_t>(op.root()) * gridDim.x + blockIdx.x) * 4, opaque(state) * 8) = r;
      }
#pragma unroll
      for (int q = 0; q < NQ; ++q) a[q] = fma(__shfl(f, W::site(lane, q)), pi, a[q]);
    }
    const uint64_t scaled = __builtin_amdgcn_ballot_w64(lane < SPW && (in.word[0] & 1u));
    if (scaled)
#pragma unroll
      for (int q = 0; q < NQ; ++q)
        if ((scaled >> W::site(lane, q)) & 1) a[q] *= SCALE_FACTOR;
    double y[2][NQ], z[NQ], g[2] = {0.0, 0.0};
    auto use = [&](int k) {
      if constexpr (!MODEL) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) g[k] = fma(z[q], mfma4(Q[W::half(q)], y[k][q], 0.0), g[k]);
      } else {
        const uint32_t l = opaque(lane);
        const double eye = (l & 3) == l >> 4 ? 1.0 : 0.0;
        double m[NA];
#pragma unroll
        for (int h = 0; h < NA; ++h) m[h] = 0.0;
#pragma unroll
        for (int q = 0; q < NQ; ++q)
          m[W::half(q)] = mfma4(mfma4(z[q], eye, 0.0), mfma4(in.x[k * NQ + q], eye, 0.0), m[W::half(q)]);
        GAS double *dst = adj + op.out() * row + k * (NA * 64);
#pragma unroll
        for (int h = 0; h < NA; ++h) *at(dst, opaque(off) + h * 512) = m[h];
      }
      if (op.kid(k) >= 0) deliver(op, in, k, z, acc[k]);
    };
    product(op, in, 0, y[0]);
    if (op.nk() == 2) {
      product(op, in, 1, y[1]);
#pragma unroll
      for (int q = 0; q < NQ; ++q) z[q] = a[q] * y[1][q];
      use(0);
#pragma unroll
      for (int q = 0; q < NQ; ++q) z[q] = a[q] * y[0][q];
      use(1);
    } else {
#pragma unroll
      for (int q = 0; q < NQ; ++q) z[q] = a[q];
      use(0);
    }
    if constexpr (MODEL) return;
    // rows are numbered in the order of the sweep: row r waits in ring[r %
    // GRAD_RING], and 64 at a time leave as one store
    const double total = pair_wave_sum(g[0], g[1]);
    const int k = lane >> 5;
    if ((lane & 31) == 31 && k < op.nk()) ring[(op.gslot() + k) % GRAD_RING] = total;
    const int done = op.gslot() + op.nk();
    if (done - flushed >= 64) {
      grad[flushed + lane] = ring[(flushed + lane) % GRAD_RING];
      flushed += 64;
    }
    if (t == 0 && lane < done - flushed) grad[flushed + lane] = ring[(flushed + lane) % GRAD_RING];
  };
  OpRegs op0 = fetch_op(ops, n_ops - 1), op1 = fetch_op(ops, max(n_ops - 2, 0));
  uint32_t warm[1] = {warm_l2(P, L.n_edges * C, ops_, n_ops, lane)};
  AdjIn4<C, NQ> u;
  load(op0, u);
  arrive(warm);
  for (int t = n_ops - 1; t >= 0; t -= 2) {
    AdjIn4<C, NQ> v, w;  // what an op does not load stays undefined: nothing is carried over
    OpRegs op2, op3;
    step(t, op0, op1, op2, u, v);
    if (t == 0) break;
    step(t - 1, op1, op2, op3, v, w);
    u = w;
    op0 = op2;
    op1 = op3;
  }
}

template <int C, int NQ>
__global__ void __launch_bounds__(64, 3)
    k_adjoint_level(const DevOp *__restrict__ ops, int n_ops, DevLayout L, const double *__restrict__ clv,
                    const int32_t *__restrict__ scl, double *__restrict__ adj, const uint8_t *__restrict__ tips,
                    const double *__restrict__ P, const double *__restrict__ Qd, const double *__restrict__ freqs,
                    const double *__restrict__ seed, const int32_t *__restrict__ tile_part,
                    const double *__restrict__ beta, int n_root, int n_uses, double *__restrict__ grad_partials) {
  adjoint_walk4<C, NQ, false>(ops, n_ops, L, clv, scl, adj, tips, P, Qd, freqs, seed, tile_part, beta, n_root, n_uses,
                              grad_partials, nullptr);
}

template <int C, int NQ>
__global__ void __launch_bounds__(64, C == 8 ? 2 : 3)
    k_model_adjoint(const DevOp *__restrict__ ops, int n_ops, DevLayout L, const double *__restrict__ clv,
                    const int32_t *__restrict__ scl, double *__restrict__ adj, const uint8_t *__restrict__ tips,
                    const double *__restrict__ P, const double *__restrict__ Qd, const double *__restrict__ freqs,
                    const double *__restrict__ seed, const int32_t *__restrict__ tile_part,
                    const double *__restrict__ beta, int n_root, int n_uses, double *__restrict__ r_part) {
  adjoint_walk4<C, NQ, true>(ops, n_ops, L, clv, scl, adj, tips, P, Qd, freqs, seed, tile_part, beta, n_root, n_uses,
                             nullptr, r_part);
}

// ------------------------------------------------ 20 states, FP64 plain form
// The walks of the 4-state form at 20 states: a wave holds one rate category
// of 16 sites, as five chunks of 64 entries (chunk j, lane l: state 4 j +
// (l >> 4), site l & 15), which are both the columns that
// v_mfma_f64_16x16x4 takes as its B operand over four states and the rows
// that it returns; a product's rows 0-15 are five of those, its rows 16-19
// five v_mfma_f64_4x4x4 whose blocks are the four 4-site groups.  So no entry
// is padding (20 = 16 + 4 rows, 5 x 4 states summed over), a product's result
// is the next one's operand, and the stored rows are these registers.
// P comes from tables in the lane order of the A operands (k_pmatrices).
typedef double f64x4 __attribute__((ext_vector_type(4)));

struct Mat20 {
  double a[10];  // chunk j: rows 0-15 in a[2 j], rows 16-19 in a[2 j + 1]
};

// big, small: a lane's byte offsets within a chunk's two parts
__device__ __forceinline__ void load_mat(const GAS double *tab, uint32_t big, uint32_t small, Mat20 &m) {
#pragma unroll
  for (int j = 0; j < 5; ++j) {
    m.a[2 * j] = *at(tab, big + j * 640);
    m.a[2 * j + 1] = *at(tab, small + j * 640);
  }
}

// y = M x + y
__device__ __forceinline__ void mul20(const Mat20 &m, const double (&x)[5], double (&y)[5]) {
  f64x4 d = {y[0], y[1], y[2], y[3]};
#pragma unroll
  for (int j = 0; j < 5; ++j) {
    d = __builtin_amdgcn_mfma_f64_16x16x4f64(m.a[2 * j], x[j], d, 0, 0, 0);
    y[4] = mfma4(m.a[2 * j + 1], x[j], y[4]);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) y[r] = d[r];
}

__device__ __forceinline__ void zero(double (&y)[5]) {
#pragma unroll
  for (int r = 0; r < 5; ++r) y[r] = 0.0;
}

// A lane's entries of a tip's 0/1 vectors; mask: of the lane's site.
__device__ __forceinline__ void tip20(uint32_t mask, int quad, double (&x)[5]) {
#pragma unroll
  for (int r = 0; r < 5; ++r)
    x[r] = __hiloint2double(-static_cast<int>((mask >> (4 * r + quad)) & 1u) & 0x3FF00000, 0);
}

// The waves of a workgroup meet, their LDS accesses done (accesses to global
// memory stay in flight).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

struct FwdIn20 {
  Mat20 m[2];
  double x[2][5];  // children read from HBM
  uint32_t raw[2]; // the children's scaler words, or tip masks
};

// Workgroup: 16 sites, a wave per category; scaler words as in
// k_forward_walk.  Per op the waves trade which of their sites are small
// (and at a root the categories' likelihoods) through LDS, with one barrier.
// Bound: each wave's chain of ops, the matrix cores busy 27 % of the time (18,564
// patterns x 4 categories, 73 ops: 0.40 ms, 0.45 with both matrices an op ahead
// at two waves per SIMD; 0.72 in ten launches of a thread per row and category
// with P in scalar registers, whose FMAs wait for every row of it).
template <int C>
__global__ void __launch_bounds__(64 * C, 3)
    k_forward_level_aa(const DevOp *__restrict__ ops_, int n_ops, int n_slots, DevLayout L, double *__restrict__ clv_,
                      int32_t *__restrict__ scl_, const uint32_t *__restrict__ tips_, const double *__restrict__ PA_,
                      const double *__restrict__ freqs, const double *__restrict__ weights,
                      const int32_t *__restrict__ tile_part, double *__restrict__ root_partials,
                      double *__restrict__ seed) {
  __shared__ uint32_t small_sites[2][C];
  __shared__ double site_like[2][C][AA_SITES];
  static_assert(C == 1 || sizeof(small_sites) + sizeof(site_like) == forward_fixed_lds_aa(C));
  const CAS DevOp *ops = to_constant(ops_);
  const int c = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63, quad = lane >> 4, col = lane & 15;
  const uint64_t n = L.n_sites_pad, row = n * (C * AA_STATES);
  const int64_t site0 = static_cast<int64_t>(blockIdx.x) * AA_SITES;
  const int part = to_constant(tile_part)[site0 / TILE];
  // [slot][chunk][lane], then the slots' scaler words
  double *slots = dyn_lds<double>() + c * n_slots * AA_ROW;
  uint32_t *slot_scl = reinterpret_cast<uint32_t *>(dyn_lds<double>() + C * n_slots * AA_ROW) + c * n_slots * AA_SITES;
  GAS double *clv = to_global(clv_) + (static_cast<int64_t>(blockIdx.x) * C + c) * AA_ROW;
  GAS int32_t *scl = to_global(scl_) + site0;
  const GAS uint32_t *tips = to_global(tips_) + site0;
  const GAS double *PA = to_global(PA_) + (static_cast<int64_t>(part) * L.n_edges * C + c) * AA_MATS;
  const uint32_t off = lane * 8, soff = col * 4;
  const uint32_t big = lane * 8, small = 512 + (quad * 4 + (lane & 3)) * 8;

  auto load = [&](const OpRegs &op, FwdIn20 &in) {
    const uint32_t o = opaque(off), so = opaque(soff);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      // (a one-child op's second child stands for its first)
      const int32_t kid = k < op.nk() ? op.kid(k) : op.kid(0);
      const GAS char *tip = reinterpret_cast<const GAS char *>(tips) + static_cast<uint32_t>(~kid) * (n * 4);
      const GAS char *word = reinterpret_cast<const GAS char *>(scl) + static_cast<uint32_t>(kid) * (n * 4);
      in.raw[k] = *at(reinterpret_cast<const GAS uint32_t *>(kid < 0 ? tip : word), so);
      if (op.has(OP_LOAD0, OP_LOAD1, k))
#pragma unroll
        for (int r = 0; r < 5; ++r) in.x[k][r] = *at(clv + static_cast<uint32_t>(op.kid(k)) * row, o + r * 512);
    }
    load_mat(PA + static_cast<int64_t>(op.edge(0)) * (C * AA_MATS), opaque(big), opaque(small), in.m[0]);
  };
  auto child = [&](const OpRegs &op, FwdIn20 &in, int k, double (&y)[5], uint32_t &count) {
    uint32_t below = in.raw[k] >> 1;
    if (op.kid(k) < 0) {
      tip20(in.raw[k], quad, in.x[k]);
      below = 0;
    }
    if (op.has(OP_PASS_KID0, OP_PASS_KID1, k)) {
      const int slot = op.slot(k);
#pragma unroll
      for (int r = 0; r < 5; ++r) in.x[k][r] = slots[slot * AA_ROW + r * 64 + lane];
      below = slot_scl[slot * AA_SITES + col] >> 1;
    }
    count += below;
    zero(y);
    mul20(in.m[k], in.x[k], y);
  };
  auto step = [&](int t, const OpRegs &op, OpRegs &ahead, OpRegs &after, FwdIn20 &in, FwdIn20 &next) {
    arrive(in.raw);
    arrive(in.x[0]);
    arrive(in.x[1]);
    arrive(in.m[0].a);
    arrive(ahead);
    __builtin_amdgcn_sched_barrier(0);
    // (the second child's matrix comes while the first is multiplied: one op
    // ahead it would cost a third of the waves)
    load_mat(PA + static_cast<int64_t>(op.edge(1)) * (C * AA_MATS), opaque(big), opaque(small), in.m[1]);
    load(ahead, next);
    after = fetch_op(ops, min(t + 2, n_ops - 1));
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t o = opaque(off);
    double v[5];
    uint32_t count = 0;
    child(op, in, 0, v, count);
    if (op.nk() == 2) {
      double y[5];
      child(op, in, 1, y, count);
#pragma unroll
      for (int r = 0; r < 5; ++r) v[r] *= y[r];
    }
    // a site is rescaled when its entries of every category are below the
    // threshold
    double m = v[0];
#pragma unroll
    for (int r = 1; r < 5; ++r) m = fmax(m, v[r]);
    uint64_t low = __builtin_amdgcn_ballot_w64(m < SCALE_THRESHOLD);
    low &= low >> 32;
    uint32_t sites = static_cast<uint32_t>(low & (low >> 16)) & 0xFFFF;
    double like = 0.0;
    if (op.root() >= 0) {
      // site likelihoods Ltilde = (1/C) sum_c pi . x
#pragma unroll
      for (int r = 0; r < 5; ++r) like = fma(freqs[part * AA_STATES + 4 * r + quad], v[r], like);
      like += __shfl_xor(like, 16);
      like += __shfl_xor(like, 32);
    }
    if constexpr (C > 1) {
      // (two sets of cells in turn: one barrier separates a cell's readers
      // from the op after next, which writes it again)
      if (lane == 0) small_sites[t & 1][c] = sites;
      if (op.root() >= 0 && lane < AA_SITES) site_like[t & 1][c][col] = like;
      lds_barrier();
#pragma unroll
      for (int cc = 0; cc < C; ++cc) sites &= small_sites[t & 1][cc];
      if (op.root() >= 0) {
        like = 0.0;
#pragma unroll
        for (int cc = 0; cc < C; ++cc) like += site_like[t & 1][cc][col];
      }
    }
    uint32_t word = count << 1;
    const bool scaled = (sites >> col) & 1;
    if (sites) {
#pragma unroll
      for (int r = 0; r < 5; ++r)
        if (scaled) v[r] *= SCALE_FACTOR;
      if (scaled) word += 3;
    }
#pragma unroll
    for (int r = 0; r < 5; ++r) *at(clv + op.out() * row, o + r * 512) = v[r];
    // (lanes of a site and the categories' waves store the same word)
    *at(scl + op.out() * n, opaque(soff)) = static_cast<int32_t>(word);
    if (op.flags() & OP_A_PASS) {
      const int slot = op.slot(2);
#pragma unroll
      for (int r = 0; r < 5; ++r) slots[slot * AA_ROW + r * 64 + lane] = v[r];
      slot_scl[slot * AA_SITES + col] = word;
    }
    if (op.root() >= 0 && c == 0) {
      const double t_site = like * (scaled ? SCALE_FACTOR : 1.0) * (1.0 / C);
      const double w = weights[site0 + col];
      const double wk = lane < AA_SITES ? w : 0.0;
      const double val = wk != 0.0 ? wk * (log(t_site) + static_cast<double>(word >> 1) * LOG_SCALE_THRESHOLD) : 0.0;
      const double sum = wave_sum(val);
      if (lane == 0) root_partials[static_cast<int64_t>(op.root()) * gridDim.x + blockIdx.x] = sum;
      // the adjoint's seed factor at this root and site, w / (C Ltilde)
      seed[op.root() * n + site0 + col] = w != 0.0 ? w * (1.0 / C) / t_site : 0.0;
    }
  };
  OpRegs op0 = fetch_op(ops, 0), op1 = fetch_op(ops, min(1, n_ops - 1));
  FwdIn20 a;
  load(op0, a);
  for (int t = 0; t < n_ops; t += 2) {
    FwdIn20 b, d;  // what an op does not load stays undefined: nothing is carried over
    OpRegs op2, op3;
    step(t, op0, op1, op2, a, b);
    if (t + 1 >= n_ops) break;
    step(t + 1, op1, op2, op3, b, d);
    a = d;
    op0 = op2;
    op1 = op3;
  }
}

struct AdjIn20 {
  Mat20 m[2];
  double x[2][5];   // inner children
  double a[5];      // own adjoint, where no slot holds it
  uint32_t raw[2];  // tip children's masks
  uint32_t word;    // own scaler word
};

// The reverse sweep of k_adjoint_level at 20 states.  A workgroup is one wave
// (a category of 16 sites; nothing crosses the categories), categories in the
// grid's slow direction, so that waves running together read the same tables.
// Bound: as the forward walk, at two waves per SIMD, the matrix cores busy 38 %
// (18,564 patterns x 4 categories: 0.75 ms; 1.79 in 18 launches of a thread per
// row, with every adjoint through HBM).
template <int C>
__global__ void __launch_bounds__(64, 2)
    k_adjoint_level_aa(const DevOp *__restrict__ ops_, int n_ops, int n_slots, DevLayout L,
                      const double *__restrict__ clv_, const int32_t *__restrict__ scl_, double *__restrict__ adj_,
                      const uint32_t *__restrict__ tips_, const double *__restrict__ PA_,
                      const double *__restrict__ Qd, const double *__restrict__ freqs,
                      const double *__restrict__ seed, const int32_t *__restrict__ tile_part,
                      const double *__restrict__ beta, int n_root, int n_uses, double *__restrict__ grad_partials) {
  const CAS DevOp *ops = to_constant(ops_);
  const int lane = threadIdx.x, quad = lane >> 4, col = lane & 15;
  const int n_blocks = L.n_tiles * (TILE / AA_SITES);
  const int c = blockIdx.x / n_blocks, block = blockIdx.x % n_blocks;
  const uint64_t n = L.n_sites_pad, row = n * (C * AA_STATES);
  const int64_t site0 = static_cast<int64_t>(block) * AA_SITES;
  const int part = to_constant(tile_part)[site0 / TILE];
  double *ring = dyn_lds<double>();
  double *slots = ring + GRAD_RING;  // [slot][chunk][lane]
  const int64_t wave = static_cast<int64_t>(block) * C + c;
  const GAS double *clv = to_global(clv_) + wave * AA_ROW;
  GAS double *adj = to_global(adj_) + wave * AA_ROW;
  const GAS int32_t *scl = to_global(scl_) + site0;
  const GAS uint32_t *tips = to_global(tips_) + site0;
  const GAS double *PA = to_global(PA_) + (static_cast<int64_t>(part) * L.n_edges * C + c) * AA_MATS;
  GAS double *grad = to_global(grad_partials) + wave * n_uses;
  const uint32_t off = lane * 8, soff = col * 4;
  const uint32_t big = lane * 8, small = 512 + (quad * 4 + (lane & 3)) * 8;
  Mat20 Q;
#pragma unroll
  for (int j = 0; j < 5; ++j) {
    const double *Qc = Qd + (static_cast<size_t>(part) * C + c) * AA_MAT + 4 * j + quad;
    Q.a[2 * j] = Qc[col * AA_STATES];
    Q.a[2 * j + 1] = Qc[(16 + (lane & 3)) * AA_STATES];
  }

  auto load = [&](const OpRegs &op, AdjIn20 &in) {
    const uint32_t o = opaque(off), so = opaque(soff);
    in.word = static_cast<uint32_t>(*at(scl + op.out() * n, so));
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      // (a one-child op's second child stands for its first)
      const int32_t kid = k < op.nk() ? op.kid(k) : op.kid(0);
      if (kid < 0)
        in.raw[k] = *at(tips + static_cast<uint32_t>(~kid) * n, so);
      else if (k < op.nk())
#pragma unroll
        for (int r = 0; r < 5; ++r) in.x[k][r] = *at(clv + static_cast<uint32_t>(kid) * row, o + r * 512);
    }
    if ((op.flags() & (OP_HAS_CONSUMERS | OP_A_PASS | OP_A_LATE)) == OP_HAS_CONSUMERS)
#pragma unroll
      for (int r = 0; r < 5; ++r) in.a[r] = *at(adj + op.out() * row, o + r * 512);
#pragma unroll
    for (int k = 0; k < 2; ++k)
      load_mat(PA + static_cast<int64_t>(op.edge(k)) * (C * AA_MATS), opaque(big), opaque(small), in.m[k]);
  };
  int flushed = ops[n_ops - 1].gslot[0];  // the sweep's first gradient row
  auto step = [&](int t, const OpRegs &op, OpRegs &ahead, OpRegs &after, AdjIn20 &in, AdjIn20 &next) {
    arrive(in.raw);
    asm volatile("" : "+v"(in.word));
    arrive(in.x[0]);
    arrive(in.x[1]);
    arrive(in.a);
    arrive(in.m[0].a);
    arrive(in.m[1].a);
    arrive(ahead);
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t o = opaque(off);
    // the transposes of the inner children's matrices, used after the products
    Mat20 mt[2];
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (k < op.nk() && op.kid(k) >= 0)
        load_mat(PA + static_cast<int64_t>(op.edge(k)) * (C * AA_MATS) + AA_MAT, opaque(big), opaque(small), mt[k]);
    __builtin_amdgcn_sched_barrier(0);
    double (&a)[5] = in.a;
    if (op.flags() & OP_A_PASS) {
      const double *slot = slots + op.slot(2) * AA_ROW + lane;
#pragma unroll
      for (int r = 0; r < 5; ++r) a[r] = slot[r * 64];
    } else if (op.flags() & OP_A_LATE) {
#pragma unroll
      for (int r = 0; r < 5; ++r) a[r] = *at(adj + op.out() * row, o + r * 512);
    } else if (!(op.flags() & OP_HAS_CONSUMERS)) {
      zero(a);
    }
    if (op.root() >= 0) {
      // seed beta * w * (1/C) pi_i / Ltilde at a displayed-tree root
      const double f = root_seed(beta[part * n_root + op.root()], seed[op.root() * n + site0 + col]);
#pragma unroll
      for (int r = 0; r < 5; ++r) a[r] = fma(f, freqs[part * AA_STATES + 4 * r + quad], a[r]);
    }
    if (in.word & 1u)
#pragma unroll
      for (int r = 0; r < 5; ++r) a[r] *= SCALE_FACTOR;
    double y[2][5];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (k >= op.nk()) continue;
      if (op.kid(k) < 0) tip20(in.raw[k], quad, in.x[k]);
      zero(y[k]);
      mul20(in.m[k], in.x[k], y[k]);
    }
    __builtin_amdgcn_sched_barrier(0);
    load(ahead, next);  // into the registers the products freed
    after = fetch_op(ops, max(t - 2, 0));
    __builtin_amdgcn_sched_barrier(0);
    double g[2] = {0.0, 0.0};
    auto use = [&](int k, const double (&z)[5]) {
      const bool inner = op.kid(k) >= 0, pass = op.has(OP_PASS_KID0, OP_PASS_KID1, k);
      double *slot = slots + op.slot(k) * AA_ROW + lane;
      GAS double *dst = adj + static_cast<uint32_t>(op.kid(k)) * row;
      double b[5];
      zero(b);
      // what the child's adjoint holds already (the deliveries before this
      // op's are stores of this wave, so in order)
      if (op.has(OP_ACC0, OP_ACC1, k)) {
#pragma unroll
        for (int r = 0; r < 5; ++r) b[r] = *at(dst, o + r * 512);
      } else if (inner && pass && !op.has(OP_FIRST_KID0, OP_FIRST_KID1, k)) {
#pragma unroll
        for (int r = 0; r < 5; ++r) b[r] = slot[r * 64];
      }
      double q[5];
      zero(q);
      mul20(Q, y[k], q);
#pragma unroll
      for (int r = 0; r < 5; ++r) g[k] = fma(z[r], q[r], g[k]);
      if (!inner) return;
      mul20(mt[k], z, b);
      if (pass) {
#pragma unroll
        for (int r = 0; r < 5; ++r) slot[r * 64] = b[r];
      } else {
#pragma unroll
        for (int r = 0; r < 5; ++r) *at(dst, o + r * 512) = b[r];
      }
    };
    double z[5];
    if (op.nk() == 2) {
#pragma unroll
      for (int r = 0; r < 5; ++r) z[r] = a[r] * y[1][r];
      use(0, z);
#pragma unroll
      for (int r = 0; r < 5; ++r) z[r] = a[r] * y[0][r];
      use(1, z);
    } else {
      use(0, a);
    }
    // rows are numbered in the order of the sweep: row r waits in ring[r %
    // GRAD_RING], and 64 at a time leave as one store
    const double total = pair_wave_sum(g[0], g[1]);
    const int k = lane >> 5;
    if ((lane & 31) == 31 && k < op.nk()) ring[(op.gslot() + k) % GRAD_RING] = total;
    const int done = op.gslot() + op.nk();
    if (done - flushed >= 64) {
      grad[flushed + lane] = ring[(flushed + lane) % GRAD_RING];
      flushed += 64;
    }
    if (t == 0 && lane < done - flushed) grad[flushed + lane] = ring[(flushed + lane) % GRAD_RING];
  };
  OpRegs op0 = fetch_op(ops, n_ops - 1), op1 = fetch_op(ops, max(n_ops - 2, 0));
  AdjIn20 u;
  load(op0, u);
  for (int t = n_ops - 1; t >= 0; t -= 2) {
    AdjIn20 v, w;  // what an op does not load stays undefined: nothing is carried over
    OpRegs op2, op3;
    step(t, op0, op1, op2, u, v);
    if (t == 0) break;
    step(t - 1, op1, op2, op3, v, w);
    u = w;
    op0 = op2;
    op1 = op3;
  }
}

// ---------------------------------------------- model gradient (FP64)
// dJ/dP of every use from the walk's sums: per (use, partition, slice of the
// partition's waves) the sum over the slice, [use][partition][slice][nl]; the
// rows after the uses are the roots' sums r_part ([root][wave][4]) likewise.
// Use u lies at [wave][part] (wave_part doubles) of adjoint row use_row[u] / 2,
// as its child use_row[u] % 2.  A workgroup holds 256 / nl waves' entries at
// once and adds them in order.
__global__ void __launch_bounds__(256)
    k_model_reduce(const double *__restrict__ adj, size_t adj_row, int wave_part, const int32_t *__restrict__ use_row,
                   const double *__restrict__ r_part, int n_uses, int nl, int n_waves, int waves_per_tile,
                   const int32_t *__restrict__ part_tile_begin, int P, int n_slice, double *__restrict__ g_sum,
                   double *__restrict__ r_sum) {
  __shared__ double sh[256];
  const bool root = static_cast<int>(blockIdx.x) >= n_uses;
  const int row = root ? blockIdx.x - n_uses : blockIdx.x, width = root ? 4 : nl;
  const int p = blockIdx.y / n_slice, slice = blockIdx.y % n_slice;
  const int wb = part_tile_begin[p] * waves_per_tile, we = part_tile_begin[p + 1] * waves_per_tile;
  const int w0 = wb + static_cast<int>(static_cast<int64_t>(we - wb) * slice / n_slice);
  const int w1 = wb + static_cast<int>(static_cast<int64_t>(we - wb) * (slice + 1) / n_slice);
  const int i = threadIdx.x % width, lead = threadIdx.x / width, step = 256 / width;
  const int stride = root ? 4 : wave_part;
  const double *in = i + (root ? r_part + static_cast<size_t>(row) * n_waves * 4
                               : adj + static_cast<size_t>(use_row[row] >> 1) * adj_row + (use_row[row] & 1) * nl);
  double s = 0.0;
  for (int w = w0 + lead; w < w1; w += step) s += in[static_cast<size_t>(w) * stride];
  sh[threadIdx.x] = s;
  __syncthreads();
  if (lead == 0) {
    for (int j = 1; j < step; ++j) s += sh[j * width + i];
    (root ? r_sum : g_sum)[((static_cast<size_t>(row) * P + p) * n_slice + slice) * width + i] = s;
  }
}

// Per (edge, partition): G_c = sum over the edge's uses, and through P_c =
// exp(Q r_c t) = V exp(L s) V^-1 (s = r_c t) the edge's part of
//   dJ/dQ   = sum_c V^-T ((V^T G_c V^-T) o Psi) V^T,
//             Psi_kl = (e^{l_k s} - e^{l_l s}) / (l_k - l_l), s e^{l_k s} for equal eigenvalues
//   dJ/dr_c = t tr(G_c^T Q P_c)
// into out[partition][edge][16 + C] (on the host, 84,000 exponentials for 110
// edges, it took 0.6 ms).  Lane (c & 3, i, j) holds entry (i, j) of
// category c; with 8 categories the lanes take two in turn.
template <int C>
__global__ void __launch_bounds__(64)
    k_model_chain(DevLayout L, const double *__restrict__ g_sum, int n_slice,
                  const int32_t *__restrict__ edge_use_begin, const int32_t *__restrict__ edge_use_list,
                  const double *__restrict__ V_, const double *__restrict__ Vinv_, const double *__restrict__ ev_,
                  const double *__restrict__ rates, const double *__restrict__ brlen, double *__restrict__ out) {
  constexpr int NA = C == 8 ? 2 : 1, NL = 64 * NA, SB = C >= 4 ? 1 : 4 / C;
  __shared__ double raw[NL], m0[64], m1[64], sums[64];
  const int edge = blockIdx.x, p = blockIdx.y, lane = threadIdx.x;
  const int i = (lane >> 2) & 3, j = lane & 3;
  const double *V = V_ + p * 16, *W = Vinv_ + p * 16, *ev = ev_ + p * 4;
  double total[NA];
#pragma unroll
  for (int h = 0; h < NA; ++h) {
    double s = 0.0;
    for (int u = edge_use_begin[edge]; u < edge_use_begin[edge + 1]; ++u)
#pragma unroll 8
      for (int sl = 0; sl < n_slice; ++sl)
        s += g_sum[((static_cast<size_t>(edge_use_list[u]) * L.n_parts + p) * n_slice + sl) * NL + h * 64 + lane];
    raw[h * 64 + lane] = s;  // [half][row i][block][column j]
  }
  __syncthreads();
  const double t = brlen[edge];
  double *dst = out + (static_cast<size_t>(p) * L.n_edges + edge) * (16 + C);
  double dq = 0.0;
#pragma unroll
  for (int h = 0; h < NA; ++h) {
    const int c = (lane >> 4) + 4 * h, cc = min(c, C - 1), base = (lane >> 4) * 16;
    const bool mine = c < C;
    double g = 0.0;
#pragma unroll
    for (int b = 0; b < SB; ++b) g += mine ? raw[h * 64 + i * 16 + ((lane >> 4) * SB + b) % 4 * 4 + j] : 0.0;
    const double s = rates[p * C + cc] * t;
    double qp = 0.0;  // Q P_c = V L exp(L s) V^-1
#pragma unroll
    for (int k = 0; k < 4; ++k) qp = fma(V[i * 4 + k] * (ev[k] * exp(ev[k] * s)), W[k * 4 + j], qp);
    sums[lane] = g * qp;
    m0[lane] = g;
    __syncthreads();
    if ((lane & 15) == 0 && mine) {
      double tr = 0.0;
      for (int k = 0; k < 16; ++k) tr += sums[base + k];
      dst[16 + c] = t * tr;
    }
    auto product = [&](const double *src, double *to, auto &&left, bool times_left) {
      double acc = 0.0;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        acc = times_left ? fma(left(i, k), src[base + k * 4 + j], acc) : fma(src[base + i * 4 + k], left(k, j), acc);
      to[lane] = acc;
      __syncthreads();
      return acc;
    };
    product(m0, m1, [&](int a, int k) { return V[k * 4 + a]; }, true);             // V^T G
    const double hv = product(m1, m0, [&](int k, int b) { return W[b * 4 + k]; }, false);  // (V^T G) V^-T
    const double la = ev[i], lb = ev[j];
    const double psi = fabs(la - lb) > 1e-10 * fmax(1.0, fabs(la)) ? (exp(la * s) - exp(lb * s)) / (la - lb)
                                                                   : s * exp(0.5 * (la + lb) * s);
    __syncthreads();
    m0[lane] = hv * psi;
    __syncthreads();
    product(m0, m1, [&](int a, int k) { return W[k * 4 + a]; }, true);             // V^-T H
    dq += product(m1, m0, [&](int k, int b) { return V[b * 4 + k]; }, false);      // (V^-T H) V^T
    total[h] = mine ? dq : 0.0;
  }
  sums[lane] = total[NA - 1];
  __syncthreads();
  if (lane < 16) {
    double d = 0.0;
    for (int c = 0; c < (C < 4 ? C : 4); ++c) d += sums[c * 16 + lane];
    dst[lane] = d;
  }
}

// Per partition the sums over the edges and, of the roots' shares, over roots
// and slices: out[partition][16 + C + 4].  Eight groups of 32 threads take
// every eighth term.
__global__ void __launch_bounds__(256)
    k_model_total(int n_edges, int C, int n_root, int n_slice, int P, const double *__restrict__ edge_out,
                  const double *__restrict__ r_sum, double *__restrict__ out) {
  __shared__ double sh[8][32];
  const int p = blockIdx.x, i = threadIdx.x & 31, group = threadIdx.x >> 5, width = 16 + C;
  double s = 0.0;
  if (i < width) {
#pragma unroll 4
    for (int e = group; e < n_edges; e += 8) s += edge_out[(static_cast<size_t>(p) * n_edges + e) * width + i];
  } else if (i < width + 4) {
#pragma unroll 4
    for (int t = group; t < n_root * n_slice; t += 8)
      s += r_sum[((static_cast<size_t>(t / n_slice) * P + p) * n_slice + t % n_slice) * 4 + i - width];
  }
  sh[group][i] = s;
  __syncthreads();
  if (threadIdx.x < width + 4) {
    for (int g = 1; g < 8; ++g) s += sh[g][i];
    out[p * (width + 4) + i] = s;
  }
}

// ------------------------------------------------------- reductions
// out[row][p] = sum of in[row][t] over the partials t of partition p
// (partials_per_tile per tile, tiles of a partition are contiguous).  One
// workgroup per (row, partition): coalesced strided loads, fixed tree
// order, so the sums are deterministic.
__device__ void reduce_segments_body(const double *__restrict__ in, size_t row_stride, int pw,
                                     const int32_t *__restrict__ ptb, int P, int row, int p,
                                     double *__restrict__ out) {
  const double *r = in + static_cast<size_t>(row) * row_stride;
  const int t0 = ptb[p] * pw, t1 = ptb[p + 1] * pw;
  Exact sum;
  for (int t = t0 + threadIdx.x; t < t1; t += 256) sum.add(r[t]);
  const double s = block_sum_exact(sum);
  if (threadIdx.x == 0) out[static_cast<size_t>(row) * P + p] = s;
}

__global__ void __launch_bounds__(256)
    k_reduce_segments(const double *__restrict__ in, size_t row_stride, int pw,
                      const int32_t *__restrict__ part_tile_begin, int P,
                      double *__restrict__ out) {
  reduce_segments_body(in, row_stride, pw, part_tile_begin, P, blockIdx.x / P, blockIdx.x % P, out);
}

// Per gradient row and slice of a partition's waves the sum of their partials
// ([wave][row]): out[row][partition][slice].  A workgroup takes 64 rows, so
// that what it reads are whole lines (a workgroup per row read 8 bytes of each
// line: 41,345 patterns, 248 rows, with k_grad_total 16 us against 9).
__device__ void reduce_grad_body(const double *__restrict__ in, int n_uses, int waves_per_tile,
                                 const int32_t *__restrict__ ptb, int P, double *__restrict__ out) {
  __shared__ double sh[4][64];
  const int lane = threadIdx.x & 63, quarter = threadIdx.x >> 6;
  const int row = blockIdx.x * 64 + lane, p = blockIdx.y / GRAD_SLICES, slice = blockIdx.y % GRAD_SLICES;
  const int64_t wb = static_cast<int64_t>(ptb[p]) * waves_per_tile, n = static_cast<int64_t>(ptb[p + 1]) * waves_per_tile - wb;
  const int64_t w0 = wb + n * slice / GRAD_SLICES, w1 = wb + n * (slice + 1) / GRAD_SLICES;
  const bool mine = row < n_uses;
  double s = 0.0;
#pragma unroll 8
  for (int64_t w = w0 + quarter; w < w1; w += 4) s += mine ? in[w * n_uses + row] : 0.0;
  sh[quarter][lane] = s;
  __syncthreads();
  if (quarter == 0 && mine)
    out[(static_cast<int64_t>(row) * P + p) * GRAD_SLICES + slice] = s + sh[1][lane] + sh[2][lane] + sh[3][lane];
}

// part_dbrlen[p][e] = sum over the uses of edge e, dbrlen[e] = over the
// partitions too.  A workgroup per edge, a wave per partition in turn.
__device__ void grad_total_body(int n_edges, int P, const int32_t *__restrict__ edge_use_begin,
                                const int32_t *__restrict__ edge_use_list, const double *__restrict__ use_sums,
                                double *__restrict__ part_dbrlen, double *__restrict__ dbrlen,
                                double *__restrict__ host_part_dbrlen, double *__restrict__ host_dbrlen) {
  __shared__ double sh[64];  // P <= 64 (checked on the host)
  const int e = blockIdx.x, lane = threadIdx.x & 63;
  const int u0 = edge_use_begin[e], n = (edge_use_begin[e + 1] - u0) * GRAD_SLICES;
  for (int p = threadIdx.x >> 6; p < P; p += blockDim.x >> 6) {
    double s = 0.0;
    for (int i = lane; i < n; i += 64)
      s += use_sums[(static_cast<int64_t>(edge_use_list[u0 + i / GRAD_SLICES]) * P + p) * GRAD_SLICES + i % GRAD_SLICES];
    s = lane_sum(s);
    if (lane == 0) {
      sh[p] = s;
      part_dbrlen[p * n_edges + e] = s;
      if (host_part_dbrlen) host_part_dbrlen[p * n_edges + e] = s;
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double tot = 0.0;
    for (int p = 0; p < P; ++p) tot += sh[p];
    dbrlen[e] = tot;
    if (host_dbrlen) host_dbrlen[e] = tot;
  }
}

__global__ void __launch_bounds__(256)
    k_grad_total(int n_edges, int P, const int32_t *__restrict__ edge_use_begin,
                 const int32_t *__restrict__ edge_use_list, const double *__restrict__ use_sums,
                 double *__restrict__ res, double *__restrict__ host, ResultLayout rl) {
  grad_total_body(n_edges, P, edge_use_begin, edge_use_list, use_sums, res + rl.part_dbrlen, res + rl.dbrlen,
                  host ? host + rl.part_dbrlen : nullptr, host ? host + rl.dbrlen : nullptr);
}

// ==================================================== FP32 form, 4 states
// The walks of the FP64 form (k_forward_walk, k_adjoint_level) in FP32.  A
// product of 64 rows with their 4 x 4 matrices is four v_mfma_f32_4x4x1 (16
// blocks): step k takes A lane (l & 3, block l >> 2) = P[l & 3][k] and B lane
// l = x[k] of the lane's own row, and register i of D is entry i of that row,
// so a lane owns a (site, category) row in every op and its four entries stay
// in four registers.  A lane's part of P is one row of it (16 bytes), of P^T
// (back-propagation) one column, stored apart.
//
// CLVs are renormalised at every op by an exact power of two so the site
// maximum lies in [0.5, 1); the per-site exponent k (true = stored * 2^-k) is
// carried as an int32.  Site sums, the mixture and the gradient reduction
// across row blocks are FP64; inside a block of 64 rows the gradient's
// per-(site, category) shares (each of order weight / branch length) are
// summed in FP32.
constexpr double LN2 = 0.69314718055994530941723212145818;
constexpr int EXP_EMPTY = -(1 << 28);  // exponent of an all-zero adjoint
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}

// A wave's rows: NR blocks of 64 rows, a block being 64 / C sites.  Lane l
// holds site j = l & 3 of a 4-site group and one category; the categories of
// a site are 4 or 8 lanes apart in a row of 16 lanes (8 categories: in two
// rows of 16), where DPP rotations reach them.
template <int C, int NR>
struct Rows {
  static constexpr int SPB = 64 / C;    // sites of a block
  static constexpr int SPW = SPB * NR;  // sites of a wave
  static __device__ __forceinline__ int cat(int lane) {
    return C == 2 ? (lane >> 3) & 1 : (lane >> 2) & (C - 1);
  }
  static __device__ __forceinline__ int site(int lane) {  // within the block
    const int b = lane >> 2;
    const int group = C == 8 ? b >> 3 : C == 4 ? b >> 2 : C == 2 ? (b & 1) | ((b >> 2) << 1) : b;
    return 4 * group + (lane & 3);
  }
  static __device__ __forceinline__ int lane_of(int site, int c) {
    const int g = site >> 2;
    const int b = C == 8 ? g * 8 + c : C == 4 ? g * 4 + c : C == 2 ? (g & 1) | (c << 1) | ((g >> 1) << 2) : g;
    return 4 * b + (site & 3);
  }
};

// Maximum over the category lanes of a site, comparing the float bit
// patterns as signed integers: the float order for values >= 0, and every
// positive value beats every negative one, which is all a site maximum
// needs.  (fmaxf would add a NaN canonicalisation around every cross-lane
// move; the integer max takes the DPP move as an operand modifier.)
template <int C>
__device__ __forceinline__ float site_max(float m) {
  int u = __float_as_int(m);
  if constexpr (C >= 4) u = max(u, dpp_i<0x124>(u));  // row_ror:4
  if constexpr (C >= 2) u = max(u, dpp_i<0x128>(u));  // row_ror:8
  if constexpr (C == 8) {
    const auto s = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    u = max(static_cast<int>(s[0]), static_cast<int>(s[1]));
  }
  return __int_as_float(u);
}
template <int C>
__device__ __forceinline__ double site_total(double t) {
  if constexpr (C >= 4) t += dpp<0x124>(t);
  if constexpr (C >= 2) t += dpp<0x128>(t);
  if constexpr (C == 8) t += __shfl_xor(t, 16);
  return t;
}
template <int C>
__device__ __forceinline__ float site_absmax(const f32x4 &x) {
  return site_max<C>(fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3]))));
}

__device__ __forceinline__ f32x4 product4(const f32x4 &M, const f32x4 &x) {
  f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < 4; ++k) y = __builtin_amdgcn_mfma_f32_4x4x1f32(M[k], x[k], y, 0, 0, 0);
  return y;
}
__device__ __forceinline__ f32x4 tip_row(uint32_t mask) {
  f32x4 x;
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = __int_as_float(-static_cast<int>((mask >> i) & 1u) & 0x3F800000);  // 1.0f or 0.0f
  return x;
}
__device__ __forceinline__ f32x4 scale4(const f32x4 &x, int e) {
  f32x4 y;
#pragma unroll
  for (int i = 0; i < 4; ++i) y[i] = ldexpf(x[i], e);
  return y;
}

// Sums over the 64 lanes of pairs of FP32 values at once, in a fixed order: lane
// 31 of v[r] ends with the total of g[r][0], lane 63 with that of g[r][1] (see
// pair_wave_sum).  The pairs take each step in turn, so that a step need not
// wait for the one before it.
template <int NR>
__device__ __forceinline__ void pair_wave_sums_f32(const float (&g)[NR][2], float (&v)[NR]) {
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(g[r][0]), __float_as_uint(g[r][1]), false, false);
    v[r] = __uint_as_float(s[0]) + __uint_as_float(s[1]);
  }
  auto step = [&](auto control) {
#pragma unroll
    for (int r = 0; r < NR; ++r) v[r] += dpp<decltype(control)::value>(v[r]);
  };
  step(std::integral_constant<int, 0x111>{});
  step(std::integral_constant<int, 0x112>{});
  step(std::integral_constant<int, 0x114>{});
  step(std::integral_constant<int, 0x118>{});
  step(std::integral_constant<int, 0x142>{});
}

// Sum of v over the lanes of a row block that hold the lane's category (C > 1),
// in all of them.
template <int C>
__device__ __forceinline__ double block_total(double v) {
  auto add = [](double x, auto &&swap) {
    const auto lo = swap(__double2loint(x)), hi = swap(__double2hiint(x));
    return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
  };
  v += dpp<DPP_XOR1>(v);
  v += dpp<DPP_XOR2>(v);
  if constexpr (C == 2) v += dpp<0x141>(v);  // row_half_mirror: the other quad of eight lanes
  if constexpr (C <= 4) v = add(v, [](int x) { return __builtin_amdgcn_permlane16_swap(x, x, false, false); });
  return add(v, [](int x) { return __builtin_amdgcn_permlane32_swap(x, x, false, false); });
}

// x 2^ex + y 2^ey with both aligned to the larger exponent, which is
// returned.  Branch-free (one side shifts by zero): the comparison differs
// between the sites of a wave.
__device__ __forceinline__ int align_add(f32x4 &x, int ex, const f32x4 &y, int ey) {
  const int e = max(ex, ey);
  // power-of-two scales: the products are exact, as ldexp would be
  const float sx = ldexpf(1.0f, ex - e), sy = ldexpf(1.0f, ey - e);
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = fmaf(x[i], sx, y[i] * sy);
  return e;
}

__device__ __forceinline__ void arrive(f32x4 &x) { asm volatile("" : "+v"(x)); }
template <int N>
__device__ __forceinline__ void arrive(f32x4 (&x)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) arrive(x[i]);
}

// The loop of a walk over ops[0, n) (backwards: ops[n - 1] first): the inputs
// of an op are loaded one op ahead, its descriptor one op before that (loading
// two ops ahead measured the same).  `early` issues what the op must read
// after the stores of the op before it.
template <typename In, typename Load, typename Early, typename Step>
__device__ __forceinline__ void walk_ops(const CAS DevOp *ops, int n, bool backwards, Load load, Early early, Step step) {
  auto at_step = [&](int i) { return backwards ? max(n - 1 - i, 0) : min(i, n - 1); };
  OpRegs op[2] = {fetch_op(ops, at_step(0)), fetch_op(ops, at_step(1))};
  In in[2];
  load(op[0], in[0]);
  // complete before the loop, so that the waits inside it count only what the
  // step before issued (its stores need not have ended)
  in[0].arrive_all();
  for (int t = 0;; t += 2) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (t + u >= n) return;
      in[u].arrive_all();
      arrive(op[1 - u]);
      __builtin_amdgcn_sched_barrier(0);
      const OpRegs now = op[u];
      auto held = early(now);
      In next;  // what an op does not load stays undefined: nothing is carried over
      load(op[1 - u], next);
      op[u] = fetch_op(ops, at_step(t + u + 2));
      __builtin_amdgcn_sched_barrier(0);
      step(now, in[u], held);
      in[1 - u] = next;
    }
  }
}

// Scaler words: exponent k of the CLV << 9 | exponent of this op's
// renormalisation in 9 bits (-149 .. 1); k stays far below 2^22 for the
// networks the form takes.
__device__ __forceinline__ int word_k(int32_t word) { return word >> 9; }
__device__ __forceinline__ int word_step(int32_t word) { return (word << 23) >> 23; }

template <int C, int NR>
struct FwdIn32 {
  f32x4 A[2], x[2 * NR];
  uint32_t raw[2 * NR];  // the children's scaler words, or tip masks
  __device__ __forceinline__ void arrive_all() {
    arrive(A);
    arrive(x);
    arrive(raw);
  }
};

struct Nothing {};

template <int C, int NR>
__device__ __forceinline__ void forward_walk32(const NetDesc &nd, float *lds, int64_t site0) {
  using W = Rows<C, NR>;
  const int lane = threadIdx.x & 63;
  const uint64_t n = nd.L.n_sites_pad, row = n * (C * 16);  // bytes of a CLV row
  const int part = to_constant(nd.tile_part)[site0 / TILE];
  const int n_slots = nd.fwd_slots;
  f32x4 *slots = reinterpret_cast<f32x4 *>(lds);  // [slot][block][lane], then the scaler words [slot][block][site]
  int32_t *slot_scl = reinterpret_cast<int32_t *>(slots + n_slots * (NR * 64));
  const int sl = W::site(lane);
  GAS char *clv = reinterpret_cast<GAS char *>(to_global(nd.clv)) + site0 * (C * 16);
  GAS char *scl = reinterpret_cast<GAS char *>(to_global(nd.scl)) + site0 * 4;
  const GAS char *tips = reinterpret_cast<const GAS char *>(to_global(nd.tips)) + site0;
  const GAS char *P =
      reinterpret_cast<const GAS char *>(to_global(nd.Pf)) + static_cast<int64_t>(part) * nd.L.n_edges * (C * 64);
  const uint32_t off = lane * 16, soff = sl * 4, aoff = W::cat(lane) * 64 + (lane & 3) * 16;
  double w[NR], pi[4];
#pragma unroll
  for (int r = 0; r < NR; ++r) w[r] = to_global(nd.weights)[site0 + r * W::SPB + sl];
#pragma unroll
  for (int i = 0; i < 4; ++i) pi[i] = to_global(nd.freqs)[part * 4 + i];
  GAS double *root_partials = to_global(nd.root_partials) + site0 / W::SPB;  // [root][block]
  GAS double *seed = to_global(nd.seed) + site0 + sl;
  const int64_t n_blocks = static_cast<int64_t>(n) / W::SPB;

  auto load = [&](const OpRegs &op, FwdIn32<C, NR> &in) {
    const uint32_t o = opaque(off), so = opaque(soff), tip_o = opaque(sl), ao = opaque(aoff);
#pragma unroll
    for (int k = 0; k < 2; ++k) in.A[k] = *reinterpret_cast<const GAS f32x4 *>(P + op.edge(k) * (C * 64) + ao);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (op.has(OP_LOAD0, OP_LOAD1, k)) {
        const GAS char *src = clv + static_cast<uint32_t>(op.kid(k)) * row;
        const GAS char *word = scl + static_cast<uint32_t>(op.kid(k)) * (n * 4);
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          in.x[k * NR + r] = *reinterpret_cast<const GAS f32x4 *>(src + o + r * 1024);
          in.raw[k * NR + r] = *reinterpret_cast<const GAS uint32_t *>(word + so + r * (W::SPB * 4));
        }
      }
      if (k < op.nk() && op.kid(k) < 0) {
        const GAS char *tip = tips + static_cast<uint32_t>(~op.kid(k)) * n;
#pragma unroll
        for (int r = 0; r < NR; ++r)
          in.raw[k * NR + r] = *reinterpret_cast<const GAS uint8_t *>(tip + tip_o + r * W::SPB);
      }
    }
  };
  auto child = [&](const OpRegs &op, FwdIn32<C, NR> &in, int k, f32x4 (&y)[NR], int (&ks)[NR]) {
    if (op.kid(k) < 0) {
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        in.x[k * NR + r] = tip_row(in.raw[k * NR + r]);
        in.raw[k * NR + r] = 0;
      }
    }
    if (op.has(OP_PASS_KID0, OP_PASS_KID1, k)) {
      const int slot = op.slot(k);
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        in.x[k * NR + r] = slots[(slot * NR + r) * 64 + lane];
        in.raw[k * NR + r] = slot_scl[(slot * NR + r) * W::SPB + sl];
      }
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      y[r] = product4(in.A[k], in.x[k * NR + r]);
      ks[r] += word_k(static_cast<int32_t>(in.raw[k * NR + r]));
    }
  };
  auto step = [&](const OpRegs &op, FwdIn32<C, NR> &in, Nothing) {
    f32x4 v[NR];
    int word[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) word[r] = 0;
    child(op, in, 0, v, word);
    if (op.nk() == 2) {
      f32x4 y[NR];
      child(op, in, 1, y, word);
#pragma unroll
      for (int r = 0; r < NR; ++r) v[r] *= y[r];
    }
    GAS char *dst = clv + op.out() * row, *dst_scl = scl + op.out() * (n * 4);
    const uint32_t o = opaque(off), so = opaque(soff);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const float m = site_max<C>(fmaxf(fmaxf(v[r][0], v[r][1]), fmaxf(v[r][2], v[r][3])));
      const int e = m > 0.f ? __builtin_amdgcn_frexp_expf(m) : 0;
      v[r] = scale4(v[r], -e);
      word[r] = ((word[r] - e) << 9) | (e & 511);
      *reinterpret_cast<GAS f32x4 *>(dst + o + r * 1024) = v[r];
      // (the lanes of a site store the same word)
      *reinterpret_cast<GAS int32_t *>(dst_scl + so + r * (W::SPB * 4)) = word[r];
    }
    if (op.flags() & OP_A_PASS) {
      const int slot = op.slot(2);
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        slots[(slot * NR + r) * 64 + lane] = v[r];
        slot_scl[(slot * NR + r) * W::SPB + sl] = word[r];
      }
    }
    if (op.root() >= 0) {
      // (a sum per block, whatever the number of blocks of a wave: an engine
      // and a batch that it is in leave each other the same sums; category r's
      // lanes form that of block r)
      double like = 1.0, w_like = 0.0;
      int k_like = 0;
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        double t = 0.0;
#pragma unroll
        for (int i = 0; i < 4; ++i) t = fma(pi[i], static_cast<double>(v[r][i]), t);
        t = site_total<C>(t) * (1.0 / C);
        if (W::cat(lane) == r) {
          like = t;
          w_like = w[r];
          k_like = word_k(word[r]);
        }
        // the adjoint's seed factor at this root and site, w / (C Ltilde)
        seed[op.root() * static_cast<int64_t>(n) + r * W::SPB] = w[r] != 0.0 ? w[r] / (C * t) : 0.0;
      }
      const double val = w_like != 0.0 ? w_like * (log(like) - k_like * LN2) : 0.0;
      const double sum = C == 1 ? wave_sum(val) : block_total<C>(val);
      if (W::cat(lane) < NR && sl == 0) root_partials[op.root() * n_blocks + W::cat(lane)] = sum;
    }
  };
  walk_ops<FwdIn32<C, NR>>(to_constant(nd.ops_fwd), nd.n_fwd, false, load,
                              [](const OpRegs &) { return Nothing{}; }, step);
}

// Reverse sweep in push form (as k_adjoint_level).  The adjoint of every CLV
// is FP32 mantissas with a per-site exponent g: dJ/d(stored CLV) = stored *
// 2^g, renormalised at its op; contributions are aligned to the
// larger exponent before they are added, so no intermediate can overflow.
template <int C, int NR>
struct AdjIn32 {
  f32x4 A[2], AT[2], x[2 * NR], a[NR];
  double sd[NR];
  int32_t ea[NR], word[NR];
  uint32_t raw[2 * NR];  // tip masks
  __device__ __forceinline__ void arrive_all() {
    arrive(A);
    arrive(AT);
    arrive(x);
    arrive(a);
    arrive(sd);
    arrive(ea);
    arrive(word);
    arrive(raw);
  }
};
// What the children's adjoints hold already, where no slot does.
template <int NR>
struct Held32 {
  f32x4 m[2 * NR];
  int32_t e[2 * NR];
};

template <int C, int NR>
__device__ __forceinline__ void adjoint_walk32(const NetDesc &nd, float *lds, int64_t site0) {
  using W = Rows<C, NR>;
  const int lane = threadIdx.x & 63;
  const uint64_t n = nd.L.n_sites_pad, row = n * (C * 16);
  const int part = to_constant(nd.tile_part)[site0 / TILE];
  const int n_slots = nd.adj_slots;
  double *ring = reinterpret_cast<double *>(lds);
  f32x4 *slots = reinterpret_cast<f32x4 *>(ring + GRAD_RING);  // [slot][block][lane], then exponents [slot][block][site]
  int32_t *slot_e = reinterpret_cast<int32_t *>(slots + n_slots * (NR * 64));
  const int sl = W::site(lane);
  const GAS char *clv = reinterpret_cast<const GAS char *>(to_global(nd.clv)) + site0 * (C * 16);
  GAS char *adj = reinterpret_cast<GAS char *>(to_global(nd.adj)) + site0 * (C * 16);
  GAS char *adj_exp = reinterpret_cast<GAS char *>(to_global(nd.adj_exp)) + site0 * 4;
  const GAS char *scl = reinterpret_cast<const GAS char *>(to_global(nd.scl)) + site0 * 4;
  const GAS char *tips = reinterpret_cast<const GAS char *>(to_global(nd.tips)) + site0;
  const int64_t p0 = static_cast<int64_t>(part) * nd.L.n_edges * (C * 64);
  const GAS char *P = reinterpret_cast<const GAS char *>(to_global(nd.Pf)) + p0;
  const GAS char *PT = reinterpret_cast<const GAS char *>(to_global(nd.PfT)) + p0;
  const uint32_t off = lane * 16, soff = sl * 4, aoff = W::cat(lane) * 64 + (lane & 3) * 16;
  const f32x4 Q = *reinterpret_cast<const GAS f32x4 *>(reinterpret_cast<const GAS char *>(to_global(nd.Qf)) +
                                                       part * (C * 64) + aoff);
  double pi[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) pi[i] = to_global(nd.freqs)[part * 4 + i];
  const GAS double *seed = to_global(nd.seed) + site0 + sl;
  const GAS double *beta = to_global(nd.beta) + part * nd.n_root;
  GAS double *grad = to_global(nd.grad_partials) + site0 / W::SPW * nd.n_uses;
  const CAS DevOp *ops = to_constant(nd.ops_adj);
  const int n_ops = nd.n_adj;

  auto load = [&](const OpRegs &op, AdjIn32<C, NR> &in) {
    const uint32_t o = opaque(off), so = opaque(soff), tip_o = opaque(sl), ao = opaque(aoff);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      in.A[k] = *reinterpret_cast<const GAS f32x4 *>(P + op.edge(k) * (C * 64) + ao);
      in.AT[k] = *reinterpret_cast<const GAS f32x4 *>(PT + op.edge(k) * (C * 64) + ao);
    }
#pragma unroll
    for (int r = 0; r < NR; ++r)
      in.word[r] = *reinterpret_cast<const GAS int32_t *>(scl + op.out() * (n * 4) + so + r * (W::SPB * 4));
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      // (a one-child op's second child stands for its first)
      const int32_t kid = k < op.nk() ? op.kid(k) : op.kid(0);
      if (kid < 0) {
#pragma unroll
        for (int r = 0; r < NR; ++r)
          in.raw[k * NR + r] =
              *reinterpret_cast<const GAS uint8_t *>(tips + static_cast<uint32_t>(~kid) * n + tip_o + r * W::SPB);
      } else if (k < op.nk()) {
#pragma unroll
        for (int r = 0; r < NR; ++r)
          in.x[k * NR + r] = *reinterpret_cast<const GAS f32x4 *>(clv + static_cast<uint32_t>(kid) * row + o + r * 1024);
      }
    }
    if ((op.flags() & (OP_HAS_CONSUMERS | OP_A_PASS | OP_A_LATE)) == OP_HAS_CONSUMERS)
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        in.a[r] = *reinterpret_cast<const GAS f32x4 *>(adj + op.out() * row + o + r * 1024);
        in.ea[r] = *reinterpret_cast<const GAS int32_t *>(adj_exp + op.out() * (n * 4) + so + r * (W::SPB * 4));
      }
    if (op.root() >= 0)
#pragma unroll
      for (int r = 0; r < NR; ++r) in.sd[r] = seed[op.root() * static_cast<int64_t>(n) + r * W::SPB];
  };
  auto early = [&](const OpRegs &op) {
    Held32<NR> held;
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (op.has(OP_ACC0, OP_ACC1, k))
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          const uint64_t kid = static_cast<uint32_t>(op.kid(k));
          const uint32_t o = opaque(off), so = opaque(soff);
          held.m[k * NR + r] = *reinterpret_cast<const GAS f32x4 *>(adj + kid * row + o + r * 1024);
          held.e[k * NR + r] = *reinterpret_cast<const GAS int32_t *>(adj_exp + kid * (n * 4) + so + r * (W::SPB * 4));
        }
    return held;
  };
  // Delivers the vectors b (exponents ez) to child k's adjoint, adding what is
  // there already unless this is the first delivery.  The sum is left as it
  // is: mantissas between an op's factor (far above FP32's smallest) and the
  // number of deliveries; the child's op renormalises it.
  auto deliver = [&](const OpRegs &op, int k, f32x4 (&b)[NR], const int (&ez)[NR], Held32<NR> &held) {
    const bool pass = op.has(OP_PASS_KID0, OP_PASS_KID1, k);
    f32x4 *slot = slots + op.slot(k) * (NR * 64) + lane;
    int32_t *se = slot_e + op.slot(k) * (NR * W::SPB) + sl;
    int eb[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) eb[r] = ez[r];
    if (!op.has(OP_FIRST_KID0, OP_FIRST_KID1, k)) {
      if (pass)
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          held.m[k * NR + r] = slot[r * 64];
          held.e[k * NR + r] = se[r * W::SPB];
        }
#pragma unroll
      for (int r = 0; r < NR; ++r) eb[r] = align_add(b[r], eb[r], held.m[k * NR + r], held.e[k * NR + r]);
    }
    if (pass) {
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        slot[r * 64] = b[r];
        se[r * W::SPB] = eb[r];  // (the lanes of a site store the same exponent)
      }
    } else {
      const uint64_t kid = static_cast<uint32_t>(op.kid(k));
      const uint32_t o = opaque(off), so = opaque(soff);
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        *reinterpret_cast<GAS f32x4 *>(adj + kid * row + o + r * 1024) = b[r];
        *reinterpret_cast<GAS int32_t *>(adj_exp + kid * (n * 4) + so + r * (W::SPB * 4)) = eb[r];
      }
    }
  };
  int flushed = ops[n_ops - 1].gslot[0];  // the sweep's first gradient row
  const int rows_end = nd.n_uses;
  auto step = [&](const OpRegs &op, AdjIn32<C, NR> &in, Held32<NR> &held) {
    f32x4 (&a)[NR] = in.a;
    int32_t (&ez)[NR] = in.ea;
    if (op.flags() & OP_A_PASS) {
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        a[r] = slots[(op.slot(2) * NR + r) * 64 + lane];
        ez[r] = slot_e[(op.slot(2) * NR + r) * W::SPB + sl];
      }
    } else if (op.flags() & OP_A_LATE) {
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        a[r] = *reinterpret_cast<const GAS f32x4 *>(adj + op.out() * row + off + r * 1024);
        ez[r] = *reinterpret_cast<const GAS int32_t *>(adj_exp + op.out() * (n * 4) + soff + r * (W::SPB * 4));
      }
      wait_loads();
    } else if (!(op.flags() & OP_HAS_CONSUMERS)) {
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        a[r] = f32x4{0.f, 0.f, 0.f, 0.f};
        ez[r] = EXP_EMPTY;
      }
    }
    if (op.root() >= 0) {
      // seed beta * w * (1/C) pi_i / Ltilde at a displayed-tree root
      const double bt = beta[op.root()];
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        int ef = EXP_EMPTY;
        f32x4 sd = {0.f, 0.f, 0.f, 0.f};
        const double f = root_seed(bt, in.sd[r]);
        if (f != 0.0) {
          const double mf = frexp(f, &ef);
#pragma unroll
          for (int i = 0; i < 4; ++i) sd[i] = static_cast<float>(mf * pi[i]);
        }
        ez[r] = align_add(a[r], ez[r], sd, ef);
      }
    }
    // the site maximum of |a| to [0.5, 1), an all-zero adjoint to exponent
    // EXP_EMPTY (so that what it delivers cannot scale another delivery away),
    // and the exponent of z: the CLV's exponent less its children's is the
    // op's step
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const float m = site_absmax<C>(a[r]);
      const int e = __builtin_amdgcn_frexp_expf(m);  // 0 of 0
      a[r] = scale4(a[r], -e);
      ez[r] = m > 0.f ? ez[r] + e - word_step(in.word[r]) : EXP_EMPTY;
    }
    f32x4 y[2][NR];
    float g[NR][2];
#pragma unroll
    for (int r = 0; r < NR; ++r) g[r][1] = 0.f;
    auto product = [&](int k) {
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        if (op.kid(k) < 0) in.x[k * NR + r] = tip_row(in.raw[k * NR + r]);
        y[k][r] = product4(in.A[k], in.x[k * NR + r]);
      }
    };
    auto use = [&](int k, f32x4 (&z)[NR]) {
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        const f32x4 d = product4(Q, y[k][r]);
        const float gd = fmaf(z[r][3], d[3], fmaf(z[r][2], d[2], fmaf(z[r][1], d[1], z[r][0] * d[0])));
        // the site's share of dlnL/dt is O(weight / t): FP32 holds it
        g[r][k] = ldexpf(gd, ez[r]);
      }
      if (op.kid(k) >= 0) {
#pragma unroll
        for (int r = 0; r < NR; ++r) z[r] = product4(in.AT[k], z[r]);
        deliver(op, k, z, ez, held);
      }
    };
    product(0);
    f32x4 z[NR];
    if (op.nk() == 2) {
      product(1);
#pragma unroll
      for (int r = 0; r < NR; ++r) z[r] = a[r] * y[1][r];
      use(0, z);
#pragma unroll
      for (int r = 0; r < NR; ++r) z[r] = a[r] * y[0][r];
      use(1, z);
    } else {
#pragma unroll
      for (int r = 0; r < NR; ++r) z[r] = a[r];
      use(0, z);
    }
    // (rows leave as in k_adjoint_level)
    float sums[NR];
    pair_wave_sums_f32<NR>(g, sums);
    double total = sums[0];
#pragma unroll
    for (int r = 1; r < NR; ++r) total += sums[r];
    const int k = lane >> 5;
    if ((lane & 31) == 31 && k < op.nk()) ring[(op.gslot() + k) % GRAD_RING] = total;
    const int done = op.gslot() + op.nk();
    if (done - flushed >= 64) {
      grad[flushed + lane] = ring[(flushed + lane) % GRAD_RING];
      flushed += 64;
    }
    if (done == rows_end && lane < done - flushed) grad[flushed + lane] = ring[(flushed + lane) % GRAD_RING];
  };
  walk_ops<AdjIn32<C, NR>>(ops, n_ops, true, load, early, step);
}

// WG threads per workgroup: one wave, which the device places wherever a SIMD
// has room (41,345 patterns, gradient: 0.41 ms, 0.54 with four waves per
// workgroup).  G = 2: two row blocks per wave, G = 3: one (see walk_blocks).
template <int G>
constexpr int row_blocks = G == 2 ? 2 : 1;

template <int C, int G, int WG>
__global__ void __launch_bounds__(WG, 3)
    k_forward_persistent(const NetDesc *__restrict__ nets, const WorkItem *__restrict__ work) {
  static_assert(WG == 64, "a workgroup is one wave");
  const WorkItem wi = to_constant(work)[blockIdx.x];
  forward_walk32<C, row_blocks<G>>(nets[wi.net], dyn_lds<float>(),
                                   static_cast<int64_t>(wi.tile) * Rows<C, row_blocks<G>>::SPW);
}

template <int C, int G, int WG>
__global__ void __launch_bounds__(WG, 3)
    k_adjoint_persistent(const NetDesc *__restrict__ nets, const WorkItem *__restrict__ work) {
  static_assert(WG == 64, "a workgroup is one wave");
  const WorkItem wi = to_constant(work)[blockIdx.x];
  adjoint_walk32<C, row_blocks<G>>(nets[wi.net], dyn_lds<float>(),
                                   static_cast<int64_t>(wi.tile) * Rows<C, row_blocks<G>>::SPW);
}

// ==================================================== FP32 form, 20 states
// The walks of the 20-state FP64 form in FP32: a wave holds one rate category
// of 16 sites, lane l the states 4 r + q (r <= 4) of site l & 15, q = l >> 4.
// Rows 0-15 of a product are a chain of five v_mfma_f32_16x16x4, over the
// states in order; row m = 4 a + b of it is state 4 b + a, so register b of
// lane group a of its result is the next product's operand.  Rows 16-19 are
// another such chain in the forward walk (its rows 0, 4, 8, 12; the others are
// not used), 320 cycles a product in all; in the reverse walk they are five
// v_mfma_f32_4x4x1 whose blocks sum a quarter of the states each, 230 cycles.
// (Summed that way forward, lnL rounds differently, by 1e-9 of its value.)
// Rows are stored as [lane 64][4] then [lane 64].
// Tables of P and P^T in operand order come from k_pmatrices; r_c Q, the same
// for every edge, is read once per sweep.
//
// CLVs are renormalised per site as in the 4-state form (scaler words too);
// adjoint exponents are per (site, category), so the reverse walk's waves
// never meet.
struct Mat20f {
  f32x4 big, small;  // steps 0-3 of rows 0-15, of rows 16-19
  float big4, small4;
};

struct Row20f {
  f32x4 v;  // states 4 r + q
  float e;  // state 16 + q
};

__device__ __forceinline__ void arrive(Mat20f &m) {
  arrive(m.big);
  arrive(m.small);
  asm volatile("" : "+v"(m.big4), "+v"(m.small4));
}
__device__ __forceinline__ void arrive(Row20f &x) {
  arrive(x.v);
  asm volatile("" : "+v"(x.e));
}

// lane16, small16: a lane's byte offsets among the 16-byte parts
__device__ __forceinline__ void load_mat(const GAS float *tab_, uint32_t lane16, uint32_t small16, Mat20f &m) {
  const GAS char *tab = reinterpret_cast<const GAS char *>(tab_);
  m.big = *reinterpret_cast<const GAS f32x4 *>(tab + lane16);
  m.big4 = *reinterpret_cast<const GAS float *>(tab + 1024 + (lane16 >> 2));
  m.small = *reinterpret_cast<const GAS f32x4 *>(tab + 1280 + small16);
  m.small4 = *reinterpret_cast<const GAS float *>(tab + 1536 + (small16 >> 2));
}

__device__ __forceinline__ Row20f load_row(const GAS char *p, uint32_t lane16) {
  Row20f x;
  x.v = *reinterpret_cast<const GAS f32x4 *>(p + lane16);
  x.e = *reinterpret_cast<const GAS float *>(p + 1024 + (lane16 >> 2));
  return x;
}
__device__ __forceinline__ void store_row(GAS char *p, uint32_t lane16, const Row20f &x) {
  *reinterpret_cast<GAS f32x4 *>(p + lane16) = x.v;
  *reinterpret_cast<GAS float *>(p + 1024 + (lane16 >> 2)) = x.e;
}
__device__ __forceinline__ Row20f slot_row(const float *slot, int lane) {
  return Row20f{*reinterpret_cast<const f32x4 *>(slot + lane * 4), slot[256 + lane]};
}
__device__ __forceinline__ void slot_store(float *slot, int lane, const Row20f &x) {
  *reinterpret_cast<f32x4 *>(slot + lane * 4) = x.v;
  slot[256 + lane] = x.e;
}

// y = M x.  BLOCKS: rows 16-19 in blocks (lanes hold row 16 + (l & 3) of them),
// else in a chain (row 16 + (l & 15) / 4).
template <bool BLOCKS>
__device__ __forceinline__ Row20f mul20(const Mat20f &m, const Row20f &x) {
  f32x4 d = {0.f, 0.f, 0.f, 0.f}, t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int r = 0; r < 5; ++r) {
    const float xr = r < 4 ? x.v[r & 3] : x.e, big = r < 4 ? m.big[r & 3] : m.big4;
    const float low = r < 4 ? m.small[r & 3] : m.small4;
    d = __builtin_amdgcn_mfma_f32_16x16x4f32(big, xr, d, 0, 0, 0);
    t = BLOCKS ? __builtin_amdgcn_mfma_f32_4x4x1f32(low, xr, t, 0, 0, 0)
               : __builtin_amdgcn_mfma_f32_16x16x4f32(low, xr, t, 0, 0, 0);
  }
  if constexpr (!BLOCKS) return Row20f{d, t[0]};
  // t[i] of quad q: row 16 + i over q's states; quad i gets the sum over the quads
  auto add = [](auto s) { return __uint_as_float(s[0]) + __uint_as_float(s[1]); };
  const float a = add(__builtin_amdgcn_permlane32_swap(__float_as_uint(t[0]), __float_as_uint(t[2]), false, false));
  const float b = add(__builtin_amdgcn_permlane32_swap(__float_as_uint(t[1]), __float_as_uint(t[3]), false, false));
  return Row20f{d, add(__builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false))};
}

// A lane's entries of a tip's 0/1 vector; mask: of the lane's site.
__device__ __forceinline__ Row20f tip20f(uint32_t mask, int quad) {
  Row20f x;
#pragma unroll
  for (int r = 0; r < 4; ++r) x.v[r] = __int_as_float(-static_cast<int>((mask >> (4 * r + quad)) & 1u) & 0x3F800000);
  x.e = __int_as_float(-static_cast<int>((mask >> (16 + quad)) & 1u) & 0x3F800000);
  return x;
}

__device__ __forceinline__ Row20f scale_row(const Row20f &x, int e) { return Row20f{scale4(x.v, e), ldexpf(x.e, e)}; }

// Maximum over the states of a site of values >= 0 (see site_max).
__device__ __forceinline__ float quad_max(float m) {
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
  const int u = max(static_cast<int>(s[0]), static_cast<int>(s[1]));
  const auto t = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  return __int_as_float(max(static_cast<int>(t[0]), static_cast<int>(t[1])));
}

struct FwdIn20f {
  Mat20f m[2];
  Row20f x[2];      // children read from HBM
  uint32_t raw[2];  // the children's scaler words, or tip masks
  __device__ __forceinline__ void arrive_all() {
    arrive(raw);
    arrive(x[0]);
    arrive(x[1]);
    arrive(m[0]);
    arrive(m[1]);
  }
};

// Workgroup: 16 sites, a wave per category, as k_forward_level_aa.
// Bound: each wave's chain of ops, the matrix cores busy 36 % of the time, here and
// in the reverse walk (18,564 patterns x 4 categories, 73 ops: 0.24 ms; 0.35 with 32-site waves of v_mfma_f32_32x32x2, whose 12 of 32 rows
// are padding, a group of four ops at a time and every CLV through HBM).
template <int C, int G>
__global__ void __launch_bounds__(64 * C, 4)
    k_forward_mfma(const NetDesc *__restrict__ nets) {
  static_assert(G == 4, "group widths name one kernel");
  __shared__ float site_most[2][C][AA_SITES];
  __shared__ double site_like[2][C][AA_SITES];
  static_assert(C == 1 || sizeof(site_most) + sizeof(site_like) == forward_fixed_lds_aa32(C));
  const NetDesc &nd = nets[0];
  const CAS DevOp *ops = to_constant(nd.ops_fwd);
  const int n_slots = nd.fwd_slots;
  const int c = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63, quad = lane >> 4, col = lane & 15;
  const uint64_t n = nd.L.n_sites_pad, row = n * (C * AA_STATES * 4);  // bytes of a CLV
  const int64_t site0 = static_cast<int64_t>(blockIdx.x) * AA_SITES;
  const int part = to_constant(nd.tile_part)[site0 / TILE];
  // [slot][row], then the slots' scaler words
  float *slots = dyn_lds<float>() + c * n_slots * AA_ROW;
  int32_t *slot_scl = reinterpret_cast<int32_t *>(dyn_lds<float>() + C * n_slots * AA_ROW) + c * n_slots * AA_SITES;
  GAS char *clv = reinterpret_cast<GAS char *>(to_global(nd.clv) + (static_cast<int64_t>(blockIdx.x) * C + c) * AA_ROW);
  GAS char *scl = reinterpret_cast<GAS char *>(to_global(nd.scl) + site0);
  const GAS char *tips = reinterpret_cast<const GAS char *>(to_global(nd.tips)) + site0 * 4;
  const GAS float *Pa = to_global(nd.Pa) + (static_cast<int64_t>(part) * nd.L.n_edges * C + c) * AA_MATS;
  const GAS double *freqs = to_global(nd.freqs) + part * AA_STATES;
  const uint32_t off = lane * 16, soff = col * 4, small = (quad * 4 + (col >> 2)) * 16;

  auto load = [&](const OpRegs &op, FwdIn20f &in) {
    const uint32_t o = opaque(off), so = opaque(soff), sm = opaque(small);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      // (a one-child op's second child stands for its first)
      const int32_t kid = k < op.nk() ? op.kid(k) : op.kid(0);
      const GAS char *tip = tips + static_cast<uint32_t>(~kid) * (n * 4);
      const GAS char *word = scl + static_cast<uint32_t>(kid) * (n * 4);
      in.raw[k] = *reinterpret_cast<const GAS uint32_t *>((kid < 0 ? tip : word) + so);
      if (op.has(OP_LOAD0, OP_LOAD1, k)) in.x[k] = load_row(clv + static_cast<uint32_t>(op.kid(k)) * row, o);
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) load_mat(Pa + static_cast<int64_t>(op.edge(k)) * (C * AA_MATS), o, sm, in.m[k]);
  };
  auto child = [&](const OpRegs &op, FwdIn20f &in, int k, int &ks) {
    if (op.kid(k) < 0) {
      in.x[k] = tip20f(in.raw[k], quad);
      in.raw[k] = 0;
    }
    if (op.has(OP_PASS_KID0, OP_PASS_KID1, k)) {
      in.x[k] = slot_row(slots + op.slot(k) * AA_ROW, lane);
      in.raw[k] = slot_scl[op.slot(k) * AA_SITES + col];
    }
    ks += word_k(static_cast<int32_t>(in.raw[k]));
    return mul20<false>(in.m[k], in.x[k]);
  };
  int turn = 0;
  auto step = [&](const OpRegs &op, FwdIn20f &in, Nothing) {
    int ks = 0;
    Row20f v = child(op, in, 0, ks);
    if (op.nk() == 2) {
      const Row20f y = child(op, in, 1, ks);
      v.v *= y.v;
      v.e *= y.e;
    }
    // (products of values >= 0; a negative rounding error loses to any
    // positive value, see site_max)
    float m = quad_max(fmaxf(fmaxf(fmaxf(v.v[0], v.v[1]), fmaxf(v.v[2], v.v[3])), v.e));
    double like = 0.0;
    if (op.root() >= 0) {
      // site likelihoods Ltilde = (1/C) sum_c pi . x
#pragma unroll
      for (int r = 0; r < 4; ++r) like = fma(freqs[4 * r + quad], static_cast<double>(v.v[r]), like);
      like = fma(freqs[16 + quad], static_cast<double>(v.e), like);
      like += __shfl_xor(like, 16);
      like += __shfl_xor(like, 32);
    }
    if constexpr (C > 1) {
      // (two sets of cells in turn: one barrier separates a cell's readers
      // from the op after next, which writes it again)
      if (lane < AA_SITES) site_most[turn][c][col] = m;
      if (op.root() >= 0 && lane < AA_SITES) site_like[turn][c][col] = like;
      lds_barrier();
      int most = 0;
#pragma unroll
      for (int cc = 0; cc < C; ++cc) most = max(most, __float_as_int(site_most[turn][cc][col]));
      m = __int_as_float(most);
      if (op.root() >= 0) {
        like = 0.0;
#pragma unroll
        for (int cc = 0; cc < C; ++cc) like += site_like[turn][cc][col];
      }
      turn ^= 1;
    }
    const int e = m > 0.f ? __builtin_amdgcn_frexp_expf(m) : 0;
    v = scale_row(v, -e);
    const int32_t word = ((ks - e) << 9) | (e & 511);
    store_row(clv + op.out() * row, opaque(off), v);
    // (lanes of a site and the categories' waves store the same word)
    *reinterpret_cast<GAS int32_t *>(scl + op.out() * (n * 4) + opaque(soff)) = word;
    if (op.flags() & OP_A_PASS) {
      slot_store(slots + op.slot(2) * AA_ROW, lane, v);
      slot_scl[op.slot(2) * AA_SITES + col] = word;
    }
    if (op.root() >= 0 && c == 0) {
      const double t = ldexp(like, -e) * (1.0 / C), w = to_global(nd.weights)[site0 + col];
      const double val = lane < AA_SITES && w != 0.0 ? w * (log(t) - word_k(word) * LN2) : 0.0;
      const double sum = wave_sum(val);
      if (lane == 0) to_global(nd.root_partials)[op.root() * static_cast<int64_t>(gridDim.x) + blockIdx.x] = sum;
      // the adjoint's seed factor at this root and site, w / (C Ltilde)
      to_global(nd.seed)[op.root() * static_cast<int64_t>(n) + site0 + col] = w != 0.0 ? w / (C * t) : 0.0;
    }
  };
  walk_ops<FwdIn20f>(ops, nd.n_fwd, false, load, [](const OpRegs &) { return Nothing{}; }, step);
}

__device__ __forceinline__ int align_add(Row20f &x, int ex, const Row20f &y, int ey) {
  const int e = max(ex, ey);
  const float sx = ldexpf(1.0f, ex - e), sy = ldexpf(1.0f, ey - e);
#pragma unroll
  for (int i = 0; i < 4; ++i) x.v[i] = fmaf(x.v[i], sx, y.v[i] * sy);
  x.e = fmaf(x.e, sx, y.e * sy);
  return e;
}

struct AdjIn20f {
  Mat20f m[2];
  Row20f x[2], a;   // inner children; own adjoint, where no slot holds it
  double sd[1];     // seed factor of a displayed-tree root
  uint32_t raw[2];  // tip children's masks
  int32_t ea[1], word[1];
  __device__ __forceinline__ void arrive_all() {
    arrive(raw);
    arrive(ea);
    arrive(word);
    arrive(sd);
    arrive(a);
    arrive(x[0]);
    arrive(x[1]);
    arrive(m[0]);
    arrive(m[1]);
  }
};
// What the op reads while its products run: the inner children's transposed
// matrices, and what their adjoints hold already, where no slot does.
struct Held20f {
  Mat20f mt[2];
  Row20f m[2];
  int32_t e[2];
};

// The reverse sweep (as k_adjoint_persistent) of one category of 16 sites,
// categories in the grid's slow direction, so that waves running together
// read the same tables.  The sums over sites of dJ/dt are FP64.  Bound: as the
// forward walk, at three waves per SIMD (same shape: 0.40 ms; 0.69 with
// 32-site waves, products reordered through LDS).
template <int C>
__global__ void __launch_bounds__(64, 3)
    k_adjoint_mfma(const NetDesc *__restrict__ nets) {
  const NetDesc &nd = nets[0];
  const CAS DevOp *ops = to_constant(nd.ops_adj);
  const int n_ops = nd.n_adj;
  const int lane = threadIdx.x, quad = lane >> 4, col = lane & 15;
  const int n_blocks = nd.L.n_tiles * (TILE / AA_SITES);
  const int c = blockIdx.x / n_blocks, block = blockIdx.x % n_blocks;
  const uint64_t n = nd.L.n_sites_pad, row = n * (C * AA_STATES * 4);
  const int64_t site0 = static_cast<int64_t>(block) * AA_SITES;
  const int part = to_constant(nd.tile_part)[site0 / TILE];
  double *ring = dyn_lds<double>();
  float *slots = reinterpret_cast<float *>(ring + GRAD_RING);  // [slot][row], then the slots' exponents
  int32_t *slot_e = reinterpret_cast<int32_t *>(slots + nd.adj_slots * AA_ROW) + col;
  const int64_t wave = static_cast<int64_t>(block) * C + c;
  const GAS char *clv = reinterpret_cast<const GAS char *>(to_global(nd.clv) + wave * AA_ROW);
  GAS char *adj = reinterpret_cast<GAS char *>(to_global(nd.adj) + wave * AA_ROW);
  GAS char *adj_exp = reinterpret_cast<GAS char *>(to_global(nd.adj_exp) + wave * AA_SITES);  // [slot][wave][site]
  const GAS char *scl = reinterpret_cast<const GAS char *>(to_global(nd.scl) + site0);
  const GAS char *tips = reinterpret_cast<const GAS char *>(to_global(nd.tips)) + site0 * 4;
  const GAS float *Pa = to_global(nd.Pa) + (static_cast<int64_t>(part) * nd.L.n_edges * C + c) * AA_MATS;
  const GAS double *freqs = to_global(nd.freqs) + part * AA_STATES;
  const GAS double *seed = to_global(nd.seed) + site0 + col;
  const GAS double *beta = to_global(nd.beta) + part * nd.n_root;
  GAS double *grad = to_global(nd.grad_partials) + wave * nd.n_uses;
  const uint32_t off = lane * 16, soff = col * 4, small = (quad * 4 + (lane & 3)) * 16;
  Mat20f Q;
  {
    const GAS float *q = to_global(nd.Qf) + (static_cast<size_t>(part) * C + c) * AA_MAT + quad;
    const GAS float *big = q + (4 * (col & 3) + (col >> 2)) * AA_STATES, *low = q + (16 + (lane & 3)) * AA_STATES;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      Q.big[r] = big[4 * r];
      Q.small[r] = low[4 * r];
    }
    Q.big4 = big[16];
    Q.small4 = low[16];
  }

  auto load = [&](const OpRegs &op, AdjIn20f &in) {
    const uint32_t o = opaque(off), so = opaque(soff), sm = opaque(small);
    in.word[0] = *reinterpret_cast<const GAS int32_t *>(scl + op.out() * (n * 4) + so);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      // (a one-child op's second child stands for its first)
      const int32_t kid = k < op.nk() ? op.kid(k) : op.kid(0);
      if (kid < 0)
        in.raw[k] = *reinterpret_cast<const GAS uint32_t *>(tips + static_cast<uint32_t>(~kid) * (n * 4) + so);
      else if (k < op.nk())
        in.x[k] = load_row(clv + static_cast<uint32_t>(kid) * row, o);
    }
    if ((op.flags() & (OP_HAS_CONSUMERS | OP_A_PASS | OP_A_LATE)) == OP_HAS_CONSUMERS) {
      in.a = load_row(adj + op.out() * row, o);
      in.ea[0] = *reinterpret_cast<const GAS int32_t *>(adj_exp + op.out() * (n * (C * 4)) + so);
    }
    if (op.root() >= 0) in.sd[0] = seed[op.root() * static_cast<int64_t>(n)];
#pragma unroll
    for (int k = 0; k < 2; ++k) load_mat(Pa + static_cast<int64_t>(op.edge(k)) * (C * AA_MATS), o, sm, in.m[k]);
  };
  auto early = [&](const OpRegs &op) {
    Held20f held;
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (k < op.nk() && op.kid(k) >= 0)
        load_mat(Pa + static_cast<int64_t>(op.edge(k)) * (C * AA_MATS) + AA_MAT, opaque(off), opaque(small),
                 held.mt[k]);
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (op.has(OP_ACC0, OP_ACC1, k)) {
        const uint64_t kid = static_cast<uint32_t>(op.kid(k));
        held.m[k] = load_row(adj + kid * row, opaque(off));
        held.e[k] = *reinterpret_cast<const GAS int32_t *>(adj_exp + kid * (n * (C * 4)) + opaque(soff));
      }
    return held;
  };
  // Delivers b (exponent ez) to child k's adjoint (as the 4-state walk).
  auto deliver = [&](const OpRegs &op, int k, Row20f b, int ez, Held20f &held) {
    const bool pass = op.has(OP_PASS_KID0, OP_PASS_KID1, k);
    float *slot = slots + op.slot(k) * AA_ROW;
    int32_t *se = slot_e + op.slot(k) * AA_SITES;
    if (!op.has(OP_FIRST_KID0, OP_FIRST_KID1, k)) {
      if (pass) {
        held.m[k] = slot_row(slot, lane);
        held.e[k] = *se;
      }
      ez = align_add(b, ez, held.m[k], held.e[k]);
    }
    if (pass) {
      slot_store(slot, lane, b);
      *se = ez;  // (the lanes of a site store the same exponent)
    } else {
      const uint64_t kid = static_cast<uint32_t>(op.kid(k));
      store_row(adj + kid * row, opaque(off), b);
      *reinterpret_cast<GAS int32_t *>(adj_exp + kid * (n * (C * 4)) + opaque(soff)) = ez;
    }
  };
  int flushed = ops[n_ops - 1].gslot[0];  // the sweep's first gradient row
  const int rows_end = nd.n_uses;
  auto step = [&](const OpRegs &op, AdjIn20f &in, Held20f &held) {
    Row20f &a = in.a;
    int &ez = in.ea[0];
    if (op.flags() & OP_A_PASS) {
      a = slot_row(slots + op.slot(2) * AA_ROW, lane);
      ez = slot_e[op.slot(2) * AA_SITES];
    } else if (op.flags() & OP_A_LATE) {
      a = load_row(adj + op.out() * row, off);
      ez = *reinterpret_cast<const GAS int32_t *>(adj_exp + op.out() * (n * (C * 4)) + soff);
      wait_loads();
    } else if (!(op.flags() & OP_HAS_CONSUMERS)) {
      a = Row20f{{0.f, 0.f, 0.f, 0.f}, 0.f};
      ez = EXP_EMPTY;
    }
    if (op.root() >= 0) {
      // seed beta * w * (1/C) pi_i / Ltilde at a displayed-tree root
      int ef = EXP_EMPTY;
      Row20f sd = {{0.f, 0.f, 0.f, 0.f}, 0.f};
      const double f = root_seed(beta[op.root()], in.sd[0]);
      if (f != 0.0) {
        const double mf = frexp(f, &ef);
#pragma unroll
        for (int r = 0; r < 4; ++r) sd.v[r] = static_cast<float>(mf * freqs[4 * r + quad]);
        sd.e = static_cast<float>(mf * freqs[16 + quad]);
      }
      ez = align_add(a, ez, sd, ef);
    }
    // (renormalised and its exponent made z's as in the 4-state walk)
    const float m = quad_max(
        fmaxf(fmaxf(fmaxf(fabsf(a.v[0]), fabsf(a.v[1])), fmaxf(fabsf(a.v[2]), fabsf(a.v[3]))), fabsf(a.e)));
    const int e = __builtin_amdgcn_frexp_expf(m);  // 0 of 0
    a = scale_row(a, -e);
    ez = m > 0.f ? ez + e - word_step(in.word[0]) : EXP_EMPTY;
    Row20f y[2];
    double g[2] = {0.0, 0.0};
    auto product = [&](int k) {
      if (op.kid(k) < 0) in.x[k] = tip20f(in.raw[k], quad);
      y[k] = mul20<true>(in.m[k], in.x[k]);
    };
    auto use = [&](int k, const Row20f &z) {
      const Row20f d = mul20<true>(Q, y[k]);
      const float gd =
          fmaf(z.e, d.e, fmaf(z.v[3], d.v[3], fmaf(z.v[2], d.v[2], fmaf(z.v[1], d.v[1], z.v[0] * d.v[0]))));
      g[k] = ldexp(static_cast<double>(gd), ez);
      if (op.kid(k) >= 0) deliver(op, k, mul20<true>(held.mt[k], z), ez, held);
    };
    product(0);
    if (op.nk() == 2) {
      product(1);
      use(0, Row20f{a.v * y[1].v, a.e * y[1].e});
      use(1, Row20f{a.v * y[0].v, a.e * y[0].e});
    } else {
      use(0, a);
    }
    // (rows leave as in k_adjoint_level)
    const double total = pair_wave_sum(g[0], g[1]);
    const int k = lane >> 5;
    if ((lane & 31) == 31 && k < op.nk()) ring[(op.gslot() + k) % GRAD_RING] = total;
    const int done = op.gslot() + op.nk();
    if (done - flushed >= 64) {
      grad[flushed + lane] = ring[(flushed + lane) % GRAD_RING];
      flushed += 64;
    }
    if (done == rows_end && lane < done - flushed) grad[flushed + lane] = ring[(flushed + lane) % GRAD_RING];
  };
  walk_ops<AdjIn20f>(ops, n_ops, true, load, early, step);
}

// ===================================================== branch derivatives
// Sumtables of one branch e, one row per displayed tree t containing it
// (the device-side counterpart of computePartitionSumtables,
// src/likelihood/LikelihoodDerivatives.cpp:249-344).  A path adjoint walks
// from t's root CLV down to e with the seed (1/C) pi_i / Ltilde (weight 1),
// so at e the vector z = d log L_s / d (P_e x) satisfies z . (P_e x) = 1.
// In the eigenbasis of the partition's rate matrix
//   ST[s,c,k] = (z^T V)_k (V^-1 x)_k,   rho_s(b) = sum_{c,k} ST e^(lambda_k r_c b)
// and rho_s(b) = L_s(b) / L_s(b_now).  Works on either form's CLVs (T =
// double with 2^256 scaler units, or float with unit exponents) in FP64.
template <int S>
__device__ __forceinline__ void load_any(const double *p, double (&x)[S]) {
  load_clv<S>(p, x);
}
template <int S>
__device__ __forceinline__ void load_any(const float *p, double (&x)[S]) {
#pragma unroll
  for (int i = 0; i < S; ++i) x[i] = static_cast<double>(p[i]);
}

// The P blocks (child edge, sibling edge; every category) of a path's first
// n_staged steps into LDS, [step][2][C][S][S]; ends with a barrier.
template <int S, int C>
__device__ __forceinline__ void stage_path_p(double *sPp, const PathStep *__restrict__ steps, int n_staged,
                                             const double *__restrict__ P, int part, const DevLayout &L) {
  if constexpr (S == 4) {
    constexpr int ROW = C * S * S;
    for (int i = threadIdx.x; i < n_staged * 2 * ROW; i += blockDim.x) {
      const int blk = i / ROW, r = i % ROW;
      const PathStep &ps = steps[blk >> 1];
      const int edge = (blk & 1) ? ps.edge_sib : ps.edge_child;
      sPp[i] = P[(static_cast<size_t>(part) * L.n_edges + edge) * ROW + r];
    }
    __syncthreads();
  }
}

// Sumtable row of a path at (site, category): the path adjoint z walked
// from the displayed tree's root to the branch, then (z^T V)_k (V^-1 x)_k
// with x the CLV below the branch.  The steps go in batches of PB: every
// load of a batch (sibling rows, tip masks, scalers; slot 0 and tip 0 stand
// in for absent ones, so no load sits on one path of a branch) is issued
// before its arithmetic, which then only waits on LDS and registers.  A
// step's own scaler is the previous step's child scaler.  over_cats: the sum of
// a value over the categories of the thread's site.
// rescalings (FP64) or exponent (FP32) that a CLV's scaler word counts
template <int S, typename T>
__device__ __forceinline__ int scl_count(int32_t word) {
  return std::is_same<T, double>::value ? word >> 1 : word_k(word);
}
// a thread's row in a CLV slot of either form (FP32, 4 states: rows are kept whole)
template <int S, int C, typename T>
__device__ __forceinline__ size_t clv_row(int64_t site, int c) {
  if constexpr (std::is_same<T, double>::value) {
    return row_offset<S, C>(site, c);
  } else {
    static_assert(S == 4, "branch derivatives of 20 states are of the FP64 form");
    constexpr int SPB = Rows<C, 1>::SPB;
    return static_cast<size_t>(site / SPB * 64 + Rows<C, 1>::lane_of(static_cast<int>(site % SPB), c)) * 4;
  }
}

template <int S, int C, typename T, bool PIECES, typename CatSum>
__device__ __forceinline__ void path_sumtable(CatSum over_cats, const PathStep *__restrict__ steps, int b0, int b1,
                                              const double *sPp, int n_staged, const DevLayout &L,
                                              int part, int64_t site, int c, const T *__restrict__ clv,
                                              const int32_t *__restrict__ scl, int scale_unit,
                                              const typename TipType<S>::type *__restrict__ tips,
                                              const double *__restrict__ P, const double *__restrict__ V,
                                              const double *__restrict__ Vinv,
                                              const double *__restrict__ freqs, double (&st)[S]) {
  using TT = typename TipType<S>::type;
  constexpr int PB = S == 4 ? 4 : 1;
  const int64_t n = L.n_sites_pad;
  const size_t slot = static_cast<size_t>(n) * (C * S), ro = clv_row<S, C, T>(site, c);
  auto slot_of = [](int32_t x) { return x >= 0 ? x : 0; };
  auto tip_of = [](int32_t x) { return (x < 0 && x != NO_CHILD) ? -x - 1 : 0; };
  auto prow = [&](int j, int which, int edge) -> const double * {
    if (S == 4 && j < n_staged) return sPp + ((j * 2 + which) * C + c) * (S * S);
    return P + ((static_cast<size_t>(part) * L.n_edges + edge) * C + c) * (S * S);
  };
  const int32_t root = steps[b0].out, low = steps[b1 - 1].child;
  double xr[S], xc[S];
  load_any<S>(clv + static_cast<size_t>(root) * slot + ro, xr);
  int kq = scl_count<S, T>(scl[static_cast<size_t>(root) * n + site]);
  load_any<S>(clv + static_cast<size_t>(slot_of(low)) * slot + ro, xc);
  const TT tmc = tips[static_cast<size_t>(tip_of(low)) * n + site];
  double a[S];
  {
    double t = 0.0;
#pragma unroll
    for (int i = 0; i < S; ++i) t = fma(freqs[part * S + i], xr[i], t);
    t = over_cats(t) * (1.0 / C);
#pragma unroll
    for (int i = 0; i < S; ++i) a[i] = freqs[part * S + i] / (C * t);
  }
  for (int s0 = b0; s0 < b1; s0 += PB) {
    double xs[PB][S];
    int kc[PB], ks[PB];
    TT tm[PB];
#pragma unroll
    for (int u = 0; u < PB; ++u) {
      if (s0 + u < b1) {
        const PathStep &ps = steps[s0 + u];
        kc[u] = scl[static_cast<size_t>(slot_of(ps.child)) * n + site];
        ks[u] = scl[static_cast<size_t>(slot_of(ps.sib)) * n + site];
        tm[u] = tips[static_cast<size_t>(tip_of(ps.sib)) * n + site];
        load_any<S>(clv + static_cast<size_t>(slot_of(ps.sib)) * slot + ro, xs[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < PB; ++u) {
      if (s0 + u < b1) {
        const PathStep &ps = steps[s0 + u];
        const int j = s0 + u - b0;
        double y[S];
        int ksu = 0;
        if (ps.nk == 2) {
          if (ps.sib < 0)
            tip_vec<S>(tm[u], xs[u]);
          else
            ksu = scl_count<S, T>(ks[u]);
          matvec<S, PIECES>(prow(j, 1, ps.edge_sib), xs[u], y);
        } else {
#pragma unroll
          for (int i = 0; i < S; ++i) y[i] = 1.0;
        }
        const int kcu = ps.child >= 0 ? scl_count<S, T>(kc[u]) : 0;
        const double F = ldexp(1.0, scale_unit * (kq - kcu - ksu));
        double z[S];
#pragma unroll
        for (int i = 0; i < S; ++i) z[i] = a[i] * F * y[i];
        if (s0 + u + 1 < b1) {
          matvec_t<S, PIECES>(prow(j, 0, ps.edge_child), z, a);  // adjoint of the on-path child
          kq = kcu;
        } else {
          double uu[S], v[S];
          if (low < 0) tip_vec<S>(tmc, xc);
          matvec_t<S, PIECES>(V + static_cast<size_t>(part) * S * S, z, uu);  // u_k = sum_i z_i V[i][k]
          matvec<S, PIECES>(Vinv + static_cast<size_t>(part) * S * S, xc, v);  // v_k = sum_j Vinv[k][j] x_j
#pragma unroll
          for (int kk = 0; kk < S; ++kk) st[kk] = uu[kk] * v[kk];
        }
      }
    }
  }
}

// The same on the matrix cores, for 4 states in FP64 (see k_forward_walk for
// the granules): a wave walks one path for its four granules, a step being
// y = P_sib x_sib, z = a F y, a' = P_child^T z.  Bound: the siblings' rows
// through L2 (16 paths, 41,345 patterns: 68 us, 116 with a thread per row and
// P in LDS, 32 reads of it per row and step).
constexpr int PATH_BATCH = 4;  // steps whose loads are issued together
// put(q, v): a lane's entry of granule q (state lane >> 4).
template <int C, typename Put>
__device__ __forceinline__ void path_sumtable4(const PathStep *__restrict__ steps_, int n_steps, const DevLayout &L,
                                               int part, int64_t site0, const double *__restrict__ clv_,
                                               const int32_t *__restrict__ scl_, const uint8_t *__restrict__ tips_,
                                               const double *__restrict__ P_, const double *__restrict__ V,
                                               const double *__restrict__ Vinv, const double *__restrict__ freqs,
                                               Put put) {
  constexpr int NQ = 4;
  using W = Quad<C, NQ>;
  constexpr int NA = W::NA, SPW = W::SPW;
  const CAS PathStep *steps = to_constant(steps_);
  const int lane = threadIdx.x & 63, state = lane >> 4;
  const uint64_t n = L.n_sites_pad, row = n * (C * 4);
  const GAS double *clv = to_global(clv_) + site0 * (C * 4);
  const GAS int32_t *scl = to_global(scl_) + site0;
  const GAS uint8_t *tips = to_global(tips_) + site0;
  const GAS double *P = to_global(P_) + static_cast<int64_t>(part) * L.n_edges * (C * 16);
  const uint32_t off = lane * 8, soff = (lane % SPW) * 4, woff = (lane % W::NW) * 4;
  const int tip_shift = 8 * (lane & 3) + state;
  uint32_t aoff[NA], toff[NA];
#pragma unroll
  for (int h = 0; h < NA; ++h) {
    aoff[h] = (W::cat(lane, h) * 16 + (lane & 3) * 4 + state) * 8;
    toff[h] = (W::cat(lane, h) * 16 + state * 4 + (lane & 3)) * 8;
  }
  auto load_row = [&](int32_t kid, double (&x)[NQ], uint32_t &raw) {
    if (kid < 0)
      raw = *at(reinterpret_cast<const GAS uint32_t *>(tips + static_cast<uint32_t>(~kid) * n), woff);
    else
#pragma unroll
      for (int q = 0; q < NQ; ++q) x[q] = *at(clv + static_cast<uint32_t>(kid) * row, off + q * 512);
  };
  auto tip_row = [&](int32_t kid, double (&x)[NQ], uint32_t raw) {
    if (kid < 0)
#pragma unroll
      for (int q = 0; q < NQ; ++q) x[q] = tip_entry<C, NQ>(raw, q, lane, tip_shift);
  };
  const int32_t low = steps[n_steps - 1].child;
  double a[NQ], xc[NQ];
  uint32_t rawc = 0;
  load_row(steps[0].out, a, rawc);
  load_row(low, xc, rawc);
  const double pi = freqs[part * 4 + state], pi_c = pi * (1.0 / C);
  // the seed (1/C) pi_i / Ltilde at the root
#pragma unroll
  for (int q = 0; q < NQ; q += NA) {
    double t = mfma4(pi_c, a[q], 0.0);
    if constexpr (C == 8) t += mfma4(pi_c, a[q + 1], 0.0);
    if constexpr (C >= 4) t += dpp<0x124>(t);  // row_ror:4
    if constexpr (C >= 2) t += dpp<0x128>(t);  // row_ror:8
#pragma unroll
    for (int h = 0; h < NA; ++h) a[q + h] = pi / (C * t);
  }
  for (int s0 = 0; s0 < n_steps; s0 += PATH_BATCH) {
    double x[PATH_BATCH][NQ], A[PATH_BATCH][NA], AT[PATH_BATCH][NA];
    uint32_t raw[PATH_BATCH], word[PATH_BATCH];
#pragma unroll
    for (int u = 0; u < PATH_BATCH; ++u) {
      if (s0 + u >= n_steps) continue;
      const CAS PathStep &ps = steps[s0 + u];
      word[u] = *at(scl + static_cast<uint32_t>(ps.out) * n, soff);
#pragma unroll
      for (int h = 0; h < NA; ++h) AT[u][h] = *at(P + static_cast<int64_t>(ps.edge_child) * (C * 16), toff[h]);
      if (ps.nk == 2) {
        load_row(ps.sib, x[u], raw[u]);
#pragma unroll
        for (int h = 0; h < NA; ++h) A[u][h] = *at(P + static_cast<int64_t>(ps.edge_sib) * (C * 16), aoff[h]);
      }
    }
#pragma unroll
    for (int u = 0; u < PATH_BATCH; ++u) {
      if (s0 + u >= n_steps) continue;
      const CAS PathStep &ps = steps[s0 + u];
      const uint64_t scaled = __builtin_amdgcn_ballot_w64(lane < SPW && (word[u] & 1u));
      if (scaled)
#pragma unroll
        for (int q = 0; q < NQ; ++q)
          if ((scaled >> W::site(lane, q)) & 1) a[q] *= SCALE_FACTOR;
      if (ps.nk == 2) {
        tip_row(ps.sib, x[u], raw[u]);
#pragma unroll
        for (int q = 0; q < NQ; ++q) a[q] *= mfma4(A[u][W::half(q)], x[u][q], 0.0);
      }
      if (s0 + u + 1 < n_steps)
#pragma unroll
        for (int q = 0; q < NQ; ++q) a[q] = mfma4(AT[u][W::half(q)], a[q], 0.0);
    }
  }
  // st_k = (z^T V)_k (V^-1 x)_k
  tip_row(low, xc, rawc);
  const double vt = V[part * 16 + state * 4 + (lane & 3)], wi = Vinv[part * 16 + (lane & 3) * 4 + state];
#pragma unroll
  for (int q = 0; q < NQ; ++q) put(q, mfma4(vt, a[q], 0.0) * mfma4(wi, xc[q], 0.0));
}

// The (site, category) of a thread that walks a path, and sums over the
// categories of its site.  4 states: the categories of a site in adjacent lanes.
// 20 states: a wave per category, so that P is the same for a wave and read
// through scalar registers (branches of 30 taxa, 8 trees, 2,000 patterns, 4
// categories: 91 us on average, 242 with every lane reading its category's P).
template <int S, int C>
struct PathRow {
  static constexpr bool WAVES = S == AA_STATES;
  int c, site;  // site within the tile
  __device__ __forceinline__ PathRow() {
    c = C == 1 ? 0 : WAVES ? __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / TILE)) : static_cast<int>(threadIdx.x % C);
    site = WAVES ? threadIdx.x % TILE : threadIdx.x / C;
  }
  // (every thread of the workgroup takes part)
  __device__ __forceinline__ double over_cats(double v) const {
    if constexpr (!WAVES || C == 1) return cat_sum<C>(v);
    __shared__ double cats[C][TILE];
    __syncthreads();  // the sum before this one has been read
    cats[c][site] = v;
    __syncthreads();
    double s[C];
#pragma unroll
    for (int k = 0; k < C; ++k) s[k] = cats[k][site];
#pragma unroll
    for (int w = 1; w < C; w *= 2)  // (in cat_sum's order)
#pragma unroll
      for (int k = 0; k < C; k += 2 * w) s[k] += s[k + w];
    return s[0];
  }
};

template <int S, int C, typename T>
__global__ void __launch_bounds__(TILE *C)
    k_sumtables(const PathStep *__restrict__ steps, const int32_t *__restrict__ path_begin,
                int n_paths, DevLayout L, const int32_t *__restrict__ tile_part, const T *__restrict__ clv,
                const int32_t *__restrict__ scl, int scale_unit,
                const typename TipType<S>::type *__restrict__ tips,
                const double *__restrict__ P, const double *__restrict__ V,
                const double *__restrict__ Vinv, const double *__restrict__ freqs,
                double *__restrict__ st) {
  if constexpr (S == 4 && std::is_same<T, double>::value) {
    // the paths of eight tiles in turn, one tile per XCD: what they have in
    // common (siblings' rows) is read from its L2
    const int group = blockIdx.x / (8 * n_paths), r = blockIdx.x % (8 * n_paths);
    const int tile = group * 8 + r % 8, path = r / 8;
    if (tile >= L.n_tiles) return;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int64_t site0 = static_cast<int64_t>(tile) * TILE + wave * Quad<C, 4>::SPW;
    GAS double *out = to_global(st) + static_cast<int64_t>(path) * L.n_sites_pad * (C * 4) + site0 * (C * 4);
    const uint32_t off = (threadIdx.x & 63) * 8;
    path_sumtable4<C>(steps + path_begin[path], path_begin[path + 1] - path_begin[path], L, tile_part[tile], site0, clv,
                      scl, tips, P, V, Vinv, freqs, [&](int q, double v) { *at(out, off + q * 512) = v; });
    return;
  } else {
  double *sPp = dyn_lds<double>();
  const int tile = blockIdx.x;
  const int part = tile_part[tile];
  const PathRow<S, C> row;
  const int c = row.c;
  const int64_t site = static_cast<int64_t>(tile) * TILE + row.site;
  // one displayed tree's path per workgroup (grid tiles x paths): the path
  // walks are independent, and one per workgroup fills the GPU
  const int j = blockIdx.y;
  if (j >= n_paths) return;
  const int b0 = path_begin[j], b1 = path_begin[j + 1];
  const int n_staged = S == 4 ? min(b1 - b0, PATH_STAGED_STEPS) : 0;
  stage_path_p<S, C>(sPp, steps + b0, n_staged, P, part, L);
  double stv[S];
  path_sumtable<S, C, T, S == AA_STATES>([&](double v) { return row.over_cats(v); }, steps, b0, b1, sPp, n_staged, L, part, site, c,
                         clv, scl, scale_unit, tips, P, V, Vinv, freqs, stv);
  store_st<S>(st + static_cast<size_t>(j) * L.n_sites_pad * (C * S) + st_offset<S, C>(site, c), stv);
  }
}

// Per displayed tree j and wave: sums over sites of w log rho(b),
// w rho'/rho and w (rho''/rho - (rho'/rho)^2) at branch length b, from the
// sumtable row of (site, category).
template <int S, int C, typename CatSum>
__device__ __forceinline__ void sumtable_partials(CatSum over_cats, const double (&in)[S], const double (&ex)[S],
                                                  const double (&lr)[S], double w, int c, double *out3) {
  double t0 = 0.0, t1 = 0.0, t2 = 0.0;
#pragma unroll
  for (int k = 0; k < S; ++k) {
    const double q = in[k] * ex[k];
    t0 += q;
    t1 += q * lr[k];
    t2 += q * lr[k] * lr[k];
  }
  t0 = over_cats(t0);
  t1 = over_cats(t1);
  t2 = over_cats(t2);
  double v0 = 0.0, v1 = 0.0, v2 = 0.0;
  if (c == 0 && w != 0.0) {
    const double r1 = t1 / t0;
    v0 = w * log(t0);
    v1 = w * r1;
    v2 = w * (t2 / t0 - r1 * r1);
  }
  out3[0] = wave_sum(v0);
  out3[1] = wave_sum(v1);
  out3[2] = wave_sum(v2);
}

// lambda_k r_c and e^(lambda_k r_c b) of the workgroup's partition for every
// (category, state): site-independent, so computed once per workgroup (the
// exponentials would otherwise dominate the evaluation's arithmetic) and
// handed to every thread through LDS; the values are the ones each thread
// computed itself before.  Ends with a barrier.
template <int S, int C>
__device__ __forceinline__ void stage_exps(const double *__restrict__ ev, const double *__restrict__ rates, int part,
                                           double brlen, int c, double (&ex)[S], double (&lr)[S]) {
  __shared__ double s_lr[C * S], s_ex[C * S];
  for (int i = threadIdx.x; i < C * S; i += blockDim.x) {
    const double l = ev[part * S + i % S] * rates[part * C + i / S];
    s_lr[i] = l;
    s_ex[i] = exp(l * brlen);
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < S; ++k) {
    lr[k] = s_lr[c * S + k];
    ex[k] = s_ex[c * S + k];
  }
}

template <int S, int C>
__global__ void __launch_bounds__(TILE *C)
    k_sumtable_eval(const double *__restrict__ st, int n_paths, DevLayout L,
                    const int32_t *__restrict__ tile_part,
                    const double *__restrict__ ev, const double *__restrict__ rates,
                    const double *__restrict__ weights, double brlen,
                    double *__restrict__ partials) {
  if (static_cast<int>(blockIdx.y) >= n_paths) return;
  constexpr int PW = TILE * C / 64;
  const int tile = blockIdx.x;
  const int part = tile_part[tile];
  const int c = threadIdx.x % C;
  const int64_t site = static_cast<int64_t>(tile) * TILE + threadIdx.x / C;
  const int64_t n = L.n_sites_pad;
  const size_t slot = static_cast<size_t>(n) * (C * S), ro = st_offset<S, C>(site, c);
  const size_t n_wt = static_cast<size_t>(L.n_tiles) * PW;
  const int wt = tile * PW + threadIdx.x / 64;
  const double w = weights[site];
  double ex[S], lr[S];
  stage_exps<S, C>(ev, rates, part, brlen, c, ex, lr);
  // one path per workgroup (grid tiles x paths)
  for (int j = blockIdx.y; j < min(n_paths, static_cast<int>(blockIdx.y) + 1); ++j) {
    double stv[S], v[3];
    load_st<S>(st + static_cast<size_t>(j) * slot + ro, stv);
    sumtable_partials<S, C>([](double x) { return cat_sum<C>(x); }, stv, ex, lr, w, c, v);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
      for (int q = 0; q < 3; ++q) partials[(static_cast<size_t>(j) * 3 + q) * n_wt + wt] = v[q];
  }
}

// ------------------------------------- Newton-Raphson of a branch on the device
// The sumtable evaluation and its reduction at the length held in the
// device state (nothing once the iteration is done, unless `final_eval`),
// the Newton step and the acceptance check.  The step restates the
// safeguarded iteration of the host sweep (netrax_amd/optimization.py
// newton_maximise) in FP64; the mixture of the per-tree derivatives is
// computePartitionLhData's (LikelihoodDerivatives.cpp:30-188, reference
// normalisation) or the true derivative.
template <int S, int C>
__global__ void __launch_bounds__(TILE *C)
    k_sumtable_eval_nr(const double *__restrict__ st, DevLayout L, const int32_t *__restrict__ tile_part,
                       const double *__restrict__ ev, const double *__restrict__ rates,
                       const double *__restrict__ weights, const NewtonState *__restrict__ ns, int final_eval,
                       double *__restrict__ partials) {
  if (!final_eval && ns->done) return;
  constexpr int PW = TILE * C / 64;
  const int n_paths = ns->n_paths;
  if (static_cast<int>(blockIdx.y) >= n_paths) return;  // uniform: the grid covers the largest path count
  const double brlen = ns->x;
  const int tile = blockIdx.x;
  const int part = tile_part[tile];
  const int c = threadIdx.x % C;
  const int64_t site = static_cast<int64_t>(tile) * TILE + threadIdx.x / C;
  const int64_t n = L.n_sites_pad;
  const size_t slot = static_cast<size_t>(n) * (C * S), ro = st_offset<S, C>(site, c);
  const size_t n_wt = static_cast<size_t>(L.n_tiles) * PW;
  const int wt = tile * PW + threadIdx.x / 64;
  const double w = weights[site];
  double ex[S], lr[S];
  stage_exps<S, C>(ev, rates, part, brlen, c, ex, lr);
  // one path per workgroup (grid tiles x the largest path count)
  for (int j = blockIdx.y; j < min(n_paths, static_cast<int>(blockIdx.y) + 1); ++j) {
    double stv[S], v[3];
    load_st<S>(st + static_cast<size_t>(j) * slot + ro, stv);
    sumtable_partials<S, C>([](double x) { return cat_sum<C>(x); }, stv, ex, lr, w, c, v);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
      for (int q = 0; q < 3; ++q) partials[(static_cast<size_t>(j) * 3 + q) * n_wt + wt] = v[q];
  }
}

__global__ void __launch_bounds__(256)
    k_reduce_segments_nr(const double *__restrict__ in, size_t row_stride, int pw,
                         const int32_t *__restrict__ part_tile_begin, int P, const NewtonState *__restrict__ ns,
                         int final_eval, double *__restrict__ out) {
  if (!final_eval && ns->done) return;
  if (static_cast<int>(blockIdx.x) >= ns->n_paths * 3 * P) return;
  __shared__ double sh[4];
  const int row = blockIdx.x / P, p = blockIdx.x % P;
  const double *r = in + static_cast<size_t>(row) * row_stride;
  const int t0 = part_tile_begin[p] * pw, t1 = part_tile_begin[p + 1] * pw;
  double s = 0.0;
  for (int t = t0 + threadIdx.x; t < t1; t += 256) s += r[t];
  s = block_sum<256>(s, sh);
  if (threadIdx.x == 0) out[static_cast<size_t>(row) * P + p] = s;
}

// tree lnL of class k in partition p at the evaluated length
__device__ __forceinline__ double nr_tree_logl(const double *sums, const DerivClassDev &cl, const double *base,
                                               int P, int nc, int k, int p) {
  double ll = base[static_cast<size_t>(p) * nc + k];
  if (cl.has && cl.path >= 0) ll += sums[(static_cast<size_t>(cl.path) * 3 + 0) * P + p];
  return ll;
}

// The class table, the base tree lnLs and the path sums are small: the
// workgroup copies them into LDS when they fit (NR_LDS_BYTES), so the serial
// mixture below reads LDS instead of making a memory round trip per value.
constexpr int NR_LDS_BYTES = 32768;
__device__ __forceinline__ void nr_stage(const double *&sums, const DerivClassDev *&cls, const double *&base, int P,
                                         int nc, int n_paths) {
  const size_t n_cls = static_cast<size_t>(nc), n_base = static_cast<size_t>(P) * nc,
               n_sums = static_cast<size_t>(n_paths) * 3 * P;
  if (sizeof(DerivClassDev) * n_cls + sizeof(double) * (n_base + n_sums) > NR_LDS_BYTES) return;
  DerivClassDev *s_cls = dyn_lds<DerivClassDev>();
  double *s_base = reinterpret_cast<double *>(s_cls + n_cls), *s_sums = s_base + n_base;
  for (size_t i = threadIdx.x; i < n_cls; i += blockDim.x) s_cls[i] = cls[i];
  for (size_t i = threadIdx.x; i < n_base; i += blockDim.x) s_base[i] = base[i];
  for (size_t i = threadIdx.x; i < n_sums; i += blockDim.x) s_sums[i] = sums[i];
  __syncthreads();
  cls = s_cls;
  base = s_base;
  sums = s_sums;
}

// Butterfly reductions over the 64 lanes of the (one-wave) Newton kernels;
// every lane ends with the result.
__device__ __forceinline__ double nr_wave_sum(double v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  return v;
}
__device__ __forceinline__ double nr_wave_max(double v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = fmax(v, __shfl_xor(v, o));
  return v;
}
__device__ __forceinline__ int nr_wave_isum(int v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  return v;
}
__device__ __forceinline__ int nr_wave_imax(int v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = max(v, __shfl_xor(v, o));
  return v;
}

// One wave: lane l takes the classes l, l + 64, ...; the class loops of the
// mixture become wave reductions.
__global__ void __launch_bounds__(64)
    k_newton_step(const double *__restrict__ sums_g, int P, int nc,
                  const DerivClassDev *__restrict__ cls_g, const double *__restrict__ base_g,
                  int variant, int mode, NewtonState *__restrict__ ns) {
  if (ns->done) return;  // uniform: every thread reads the same flag
  const double *sums = sums_g, *base = base_g;
  const DerivClassDev *cls = cls_g;
  nr_stage(sums, cls, base, P, nc, ns->n_paths);
  const int lane = threadIdx.x;
  auto member = [&](int k) { return cls[k].use && (mode == NRX_DERIV_TRUE || cls[k].has); };
  // derivatives at ns->x, mixed per partition as the host does
  double D1 = 0.0, D2 = 0.0;
  for (int p = 0; p < P; ++p) {
    auto d1 = [&](int k) {
      return cls[k].has && cls[k].path >= 0 ? sums[(static_cast<size_t>(cls[k].path) * 3 + 1) * P + p] : 0.0;
    };
    auto d2 = [&](int k) {
      return cls[k].has && cls[k].path >= 0 ? sums[(static_cast<size_t>(cls[k].path) * 3 + 2) * P + p] : 0.0;
    };
    int cnt = 0, last = -1;
    for (int k = lane; k < nc; k += 64)
      if (member(k)) {
        ++cnt;
        last = k;
      }
    const int n_members = nr_wave_isum(cnt), only = nr_wave_imax(last);
    double pd1 = 0.0, pd2 = 0.0;
    if (n_members == 1 && mode == NRX_DERIV_REFERENCE) {
      pd1 = d1(only);  // single-tree mode
      pd2 = d2(only);
    } else if (n_members > 0) {
      if (variant == NRX_AVERAGE_DISPLAYED_TREES) {
        double m = -INFINITY;
        for (int k = lane; k < nc; k += 64)
          if (member(k)) m = fmax(m, cls[k].logprob + nr_tree_logl(sums, cls[k], base, P, nc, k, p));
        const double mx = nr_wave_max(m);
        double s0 = 0.0, s1 = 0.0, s2 = 0.0;
        for (int k = lane; k < nc; k += 64) {
          if (!member(k)) continue;
          const double wgt = exp(cls[k].logprob + nr_tree_logl(sums, cls[k], base, P, nc, k, p) - mx);
          const double a1 = d1(k);
          s0 += wgt;
          s1 += wgt * a1;
          s2 += wgt * (a1 * a1 + d2(k));
        }
        s0 = nr_wave_sum(s0);
        s1 = nr_wave_sum(s1);
        s2 = nr_wave_sum(s2);
        pd1 = s1 / s0;
        pd2 = (s2 * s0 - s1 * s1) / (s0 * s0);
      } else {
        // the first class (lowest index) with the highest score, as the
        // host's strict comparison in class order picks it
        double best = -INFINITY;
        int kb = -1;
        for (int k = lane; k < nc; k += 64) {
          if (!member(k)) continue;
          const double ll = nr_tree_logl(sums, cls[k], base, P, nc, k, p);
          // reference mode: the tree maximising tree_logl * tree_prob
          // (LikelihoodDerivatives.cpp:161-167)
          const double score = mode == NRX_DERIV_REFERENCE ? ll * exp(cls[k].logprob) : cls[k].logprob + ll;
          if (score > best) {
            best = score;
            kb = k;
          }
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
          const double ob = __shfl_xor(best, o);
          const int ok = __shfl_xor(kb, o);
          if (ok >= 0 && (kb < 0 || ob > best || (ob == best && ok < kb))) {
            best = ob;
            kb = ok;
          }
        }
        if (kb >= 0) {
          pd1 = d1(kb);
          pd2 = d2(kb);
        }
      }
    }
    D1 += pd1;
    D2 += pd2;
  }
  if (lane != 0) return;
  ns->d1 = D1;
  ns->d2 = D2;
  ns->iters += 1;
  if (ns->iters >= ns->max_iters) ns->done = 1;  // this step is the last
  // safeguarded Newton step: keep the maximiser's bracket [a, b], take the
  // Newton step when the curvature is negative and the step stays inside,
  // else grow geometrically toward a far bound or bisect
  const double x = ns->x, tol = ns->tol;
  double a = ns->a, b = ns->b;
  if (D1 > 0.0) {
    a = x;
  } else if (D1 < 0.0) {
    b = x;
  } else {
    ns->done = 1;
    return;
  }
  double nx = 0.0;
  bool ok = false;
  if (D2 < 0.0) {
    nx = x - D1 / D2;
    ok = a < nx && nx < b;
  }
  if (!ok) {
    if (D1 > 0.0 && b - x > 4.0 * (x + tol))
      nx = fmin(b, 2.0 * x + tol);
    else if (D1 < 0.0 && x - a > 4.0 * tol && x > 4.0 * a)
      nx = fmax(a, 0.5 * x);
    else
      nx = 0.5 * (a + b);
  }
  ns->a = a;
  ns->b = b;
  if (fabs(nx - x) < tol) ns->done = 1;
  ns->x = fmin(fmax(nx, ns->lo), ns->hi);
}

// network lnL at the final length vs at the start (both from the same tree
// lnLs); a worse length is given up (optimize_branch,
// BranchLengthOptimization.cpp:317-330)
__global__ void __launch_bounds__(64)
    k_newton_accept(const double *__restrict__ sums_g, int P, int nc,
                    const DerivClassDev *__restrict__ cls_g, const double *__restrict__ base_g,
                    int variant, NewtonState *__restrict__ ns) {
  const double *sums = sums_g, *base = base_g;
  const DerivClassDev *cls = cls_g;
  nr_stage(sums, cls, base, P, nc, ns->n_paths);
  const int lane = threadIdx.x;
  double l_new = 0.0, l_old = 0.0;
  for (int p = 0; p < P; ++p) {
    double mn = -INFINITY, mo = -INFINITY;
    for (int k = lane; k < nc; k += 64) {
      if (!cls[k].use) continue;
      mn = fmax(mn, cls[k].logprob + nr_tree_logl(sums, cls[k], base, P, nc, k, p));
      mo = fmax(mo, cls[k].logprob + base[static_cast<size_t>(p) * nc + k]);
    }
    mn = nr_wave_max(mn);
    mo = nr_wave_max(mo);
    if (variant == NRX_BEST_DISPLAYED_TREE) {
      l_new += mn;
      l_old += mo;
      continue;
    }
    double sn = 0.0, so = 0.0;
    for (int k = lane; k < nc; k += 64) {
      if (!cls[k].use) continue;
      sn += exp(cls[k].logprob + nr_tree_logl(sums, cls[k], base, P, nc, k, p) - mn);
      so += exp(cls[k].logprob + base[static_cast<size_t>(p) * nc + k] - mo);
    }
    l_new += mn + log(nr_wave_sum(sn));
    l_old += mo + log(nr_wave_sum(so));
  }
  if (lane != 0) return;
  ns->lnl_new = l_new;
  ns->lnl_old = l_old;
  ns->accepted = l_new >= l_old;
}

// The two kernels above in one, with no sumtable stored: each (path, site,
// category) walks its path adjoint and evaluates at b right away (the
// allocation-free variant of the branch derivatives re-walks the paths on
// every call instead of keeping sumtables).
template <int S, int C, typename T>
__global__ void __launch_bounds__(TILE *C)
    k_deriv_fused(const PathStep *__restrict__ steps, const int32_t *__restrict__ path_begin, int n_paths,
                  DevLayout L, const int32_t *__restrict__ tile_part,
                  const T *__restrict__ clv, const int32_t *__restrict__ scl, int scale_unit,
                  const typename TipType<S>::type *__restrict__ tips, const double *__restrict__ P,
                  const double *__restrict__ V, const double *__restrict__ Vinv,
                  const double *__restrict__ freqs, const double *__restrict__ ev,
                  const double *__restrict__ rates, const double *__restrict__ weights, double brlen,
                  double *__restrict__ partials) {
  constexpr int PW = TILE * C / 64;
  const int tile = blockIdx.x;
  const int part = tile_part[tile];
  const size_t n_wt = static_cast<size_t>(L.n_tiles) * PW;
  const int wt = tile * PW + threadIdx.x / 64;
  if constexpr (S == 4 && std::is_same<T, double>::value) {
    // on the matrix cores, as the sumtables; a lane's entries are of one state
    // and category (of two, with 8 categories), and the sums over the states are
    // products with ones (30 taxa, 8 trees, 20,000 patterns, 4 categories, the
    // whole call: 90 us, 107 with a thread per row)
    using W = Quad<C, 4>;
    constexpr int NA = W::NA, SPW = W::SPW;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int64_t site0 = static_cast<int64_t>(tile) * TILE + wave * SPW;
    const double w = lane < SPW ? weights[site0 + lane % SPW] : 0.0;
    double lr[NA], ex[NA];
#pragma unroll
    for (int h = 0; h < NA; ++h) {
      lr[h] = ev[part * 4 + (lane >> 4)] * rates[part * C + W::cat(lane, h)];
      ex[h] = exp(lr[h] * brlen);
    }
    for (int j = 0; j < n_paths; ++j) {
      double x[4];
      path_sumtable4<C>(steps + path_begin[j], path_begin[j + 1] - path_begin[j], L, part, site0, clv, scl, tips, P, V,
                        Vinv, freqs, [&](int q, double v) { x[q] = v; });
      double t[3] = {1.0, 0.0, 0.0};  // rho and its derivatives at site lane % SPW
#pragma unroll
      for (int q = 0; q < 4; q += NA) {
        double r[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int h = 0; h < NA; ++h) {
          double v = x[q + h] * ex[h];
#pragma unroll
          for (int d = 0; d < 3; ++d, v *= lr[h]) r[d] = mfma4(1.0, v, r[d]);
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          if constexpr (C >= 4) r[d] += dpp<0x124>(r[d]);  // row_ror:4
          if constexpr (C >= 2) r[d] += dpp<0x128>(r[d]);  // row_ror:8
          if ((lane % SPW) / (4 * W::SB) == q / NA) t[d] = r[d];
        }
      }
      const double r1 = t[1] / t[0];
      const double v[3] = {w != 0.0 ? w * log(t[0]) : 0.0, w != 0.0 ? w * r1 : 0.0,
                           w != 0.0 ? w * (t[2] / t[0] - r1 * r1) : 0.0};
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const double sum = wave_sum(v[d]);
        if (lane == 0) partials[(static_cast<size_t>(j) * 3 + d) * n_wt + wt] = sum;
      }
    }
    return;
  } else {
  const PathRow<S, C> row;
  const int c = row.c;
  const int64_t site = static_cast<int64_t>(tile) * TILE + row.site;
  const auto over_cats = [&](double v) { return row.over_cats(v); };
  const double w = weights[site];
  double ex[S], lr[S];
  stage_exps<S, C>(ev, rates, part, brlen, c, ex, lr);
  double *sPp = dyn_lds<double>();
  for (int j = 0; j < n_paths; ++j) {
    double stv[S], v[3];
    const int b0 = path_begin[j], b1 = path_begin[j + 1];
    const int n_staged = S == 4 ? min(b1 - b0, PATH_STAGED_STEPS) : 0;
    if (S == 4 && j > 0) __syncthreads();  // every lane is done with the previous path's staged P
    stage_path_p<S, C>(sPp, steps + b0, n_staged, P, part, L);
    path_sumtable<S, C, T, false>(over_cats, steps, b0, b1, sPp, n_staged, L, part, site, c, clv, scl, scale_unit, tips, P, V,
                           Vinv, freqs, stv);
    sumtable_partials<S, C>(over_cats, stv, ex, lr, w, c, v);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
      for (int q = 0; q < 3; ++q) partials[(static_cast<size_t>(j) * 3 + q) * n_wt + wt] = v[q];
  }
  }
}


// ============================================= batches of networks (FP32)
// blockIdx.y selects the network; every kernel reads that network's
// SmallDesc and does exactly what the single-network kernel does.
__global__ void __launch_bounds__(256) k_pmatrices_multi(const SmallDesc *__restrict__ descs) {
  const SmallDesc &d = descs[blockIdx.y];
  const DevLayout L = d.L;
  const int S = L.S, C = L.C;
  const int64_t total = static_cast<int64_t>(L.n_parts) * L.n_edges * C * S * S;
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const int j = idx % S;
  const int i = (idx / S) % S;
  const int c = (idx / (S * S)) % C;
  const int e = (idx / (S * S * C)) % L.n_edges;
  const int p = idx / (static_cast<int64_t>(S) * S * C * L.n_edges);
  const double rt = d.rates[p * C + c];
  const double t = d.host_brlen[e];
  if (p == 0 && idx % (C * S * S) == 0) d.brlen[e] = t;
  double a0 = 0.0;
  for (int k = 0; k < S; ++k)
    a0 += d.V[(p * S + i) * S + k] * exp(d.ev[p * S + k] * rt * t) * d.Vinv[(p * S + k) * S + j];
  d.P[idx] = a0;
  d.Pf[idx] = static_cast<float>(a0);
  d.PfT[idx - (i * S + j) + (j * S + i)] = static_cast<float>(a0);
}

__global__ void __launch_bounds__(256) k_root_reduce_multi(const SmallDesc *__restrict__ descs) {
  const SmallDesc &d = descs[blockIdx.y];
  const int P = d.L.n_parts;
  if (static_cast<int>(blockIdx.x) >= d.n_root * P) return;
  reduce_segments_body(d.root_partials, static_cast<size_t>(d.L.n_tiles) * d.pw, d.pw,
                       d.part_tile_begin, P, blockIdx.x / P, blockIdx.x % P, d.root_sums);
}

__global__ void __launch_bounds__(256)
    k_reduce_grad(const double *__restrict__ in, int n_uses, int waves_per_tile, const int32_t *__restrict__ ptb, int P,
                  double *__restrict__ out) {
  reduce_grad_body(in, n_uses, waves_per_tile, ptb, P, out);
}

__global__ void __launch_bounds__(256) k_use_reduce_multi(const SmallDesc *__restrict__ descs) {
  const SmallDesc &d = descs[blockIdx.z];
  const int P = d.L.n_parts;
  if (static_cast<int>(blockIdx.x) * 64 >= d.n_uses || static_cast<int>(blockIdx.y) >= P * GRAD_SLICES) return;
  reduce_grad_body(d.grad_partials, d.n_uses, d.gwpt, d.part_tile_begin, P, d.use_sums);
}

__global__ void __launch_bounds__(256) k_mixture_multi(const SmallDesc *__restrict__ descs,
                                                       int variant) {
  const SmallDesc &d = descs[blockIdx.x];
  ResultLayout rl{};
  rl.total = d.rl_total;
  rl.per_part = d.rl_per_part;
  rl.root_logl = d.rl_root_logl;
  rl.tree_logl = d.rl_tree_logl;
  rl.alpha = d.rl_alpha;
  rl.dbrlen = d.rl_dbrlen;
  rl.part_dbrlen = d.rl_part_dbrlen;
  rl.dprob = d.rl_dprob;
  mixture_body(d.L, d.n_root, d.nc, d.R, variant, d.classes, d.class_dlogprob, d.root_sums,
               d.beta, d.res, nullptr, rl);
}

__global__ void __launch_bounds__(256) k_grad_total_multi(const SmallDesc *__restrict__ descs) {
  const SmallDesc &d = descs[blockIdx.y];
  if (static_cast<int>(blockIdx.x) >= d.L.n_edges) return;
  grad_total_body(d.L.n_edges, d.L.n_parts, d.edge_use_begin, d.edge_use_list, d.use_sums, d.res + d.rl_part_dbrlen,
                  d.res + d.rl_dbrlen, nullptr, nullptr);
}

// Puts every network's result block next to each other into pinned host memory.
__global__ void k_gather_results(const SmallDesc *__restrict__ descs,
                                 const int64_t *__restrict__ offsets, double *__restrict__ out) {
  const SmallDesc &d = descs[blockIdx.y];
  const int64_t n = offsets[blockIdx.y + 1] - offsets[blockIdx.y];
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x)
    out[offsets[blockIdx.y] + i] = d.res[i];
}

template <typename F>
void dispatch_sc(int S, int C, F &&f) {
  // instantiated shapes: DNA (4 states) and protein (20 states) with
  // 1, 2, 4 or 8 rate categories
  auto withC = [&](auto s_tag) {
    constexpr int SS = decltype(s_tag)::value;
    switch (C) {
      case 1: f(std::integral_constant<int, SS>{}, std::integral_constant<int, 1>{}); break;
      case 2: f(std::integral_constant<int, SS>{}, std::integral_constant<int, 2>{}); break;
      case 4: f(std::integral_constant<int, SS>{}, std::integral_constant<int, 4>{}); break;
      case 8: f(std::integral_constant<int, SS>{}, std::integral_constant<int, 8>{}); break;
      default: throw std::invalid_argument("unsupported number of rate categories");
    }
  };
  if (S == 4)
    withC(std::integral_constant<int, 4>{});
  else if (S == 20)
    withC(std::integral_constant<int, 20>{});
  else
    throw std::invalid_argument("unsupported number of states");
}

}  // namespace

constexpr int64_t PM_DIRECT_WAVES = 4096;
void launch_pmatrices(Engine &e) {
  const int64_t total = static_cast<int64_t>(e.P) * e.E * e.C * e.S * e.S;
  const int nb = static_cast<int>((total + 255) / 256);
  // the kernel reads the lengths in the host's pinned memory (and leaves them
  // in d_brlen): a copy ahead of it takes 4 us and a gap.  Every wave's read
  // crosses the bus, so many waves get the copy.
  const bool direct = total <= 64 * PM_DIRECT_WAVES;
  if (!direct)
    NRX_HIP(hipMemcpyAsync(e.d_brlen.p, e.h_brlen, sizeof(double) * e.E, hipMemcpyHostToDevice, e.stream));
  hipLaunchKernelGGL(k_pmatrices, dim3(nb), dim3(256), 0, e.stream, e.L, e.d_V.as<double>(),
                     e.d_Vinv.as<double>(), e.d_eval.as<double>(), e.d_rates.as<double>(),
                     direct ? e.h_brlen_dev : e.d_brlen.as<double>(), direct ? e.d_brlen.as<double>() : nullptr,
                     e.d_P.as<double>(), e.d_Pf.as<float>(), e.d_PfT.as<float>(), e.d_PA.as<double>(),
                     e.d_Pa.as<float>());
  NRX_HIP(hipGetLastError());
}

template <typename F>
void dispatch_c(int C, F &&f) {
  switch (C) {
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    default: throw std::invalid_argument("unsupported number of rate categories");
  }
}

// Shapes of the 4-state FP64 walks: C categories, NQ granules per wave (8
// categories take granules in pairs, and 4 of them would spill registers).
template <typename F>
static void dispatch_walk(int C, int NQ, F &&f) {
  dispatch_c(C, [&](auto c) {
    constexpr int CC = decltype(c)::value;
    if constexpr (CC != 8)
      if (NQ == 4) return f(c, std::integral_constant<int, 4>{});
    if (NQ == 2) return f(c, std::integral_constant<int, 2>{});
    if constexpr (CC != 8)
      if (NQ == 1) return f(c, std::integral_constant<int, 1>{});
    throw std::logic_error("unsupported walk shape");
  });
}


void launch_forward_walk(Engine &e, const DevOp *ops, int n_ops) {
  if (n_ops == 0) return;
  const unsigned waves = static_cast<unsigned>(e.L.n_tiles) * e.rpw;
  if (e.S == AA_STATES) {
    dispatch_c(e.C, [&](auto c) {
      constexpr int C = decltype(c)::value;
      hipLaunchKernelGGL((k_forward_level_aa<C>), dim3(waves), dim3(64 * C), forward_walk_lds_aa(C, e.fwd_slots),
                         e.stream, ops, n_ops, e.fwd_slots, e.L, e.d_clv.as<double>(), e.d_scl.as<int32_t>(),
                         e.d_tips.as<uint32_t>(), e.d_PA.as<double>(), e.d_freqs.as<double>(),
                         e.d_weights.as<double>(), e.d_tile_part.as<int32_t>(), e.d_root_partials.as<double>(),
                         e.d_site_seed.as<double>());
    });
    NRX_HIP(hipGetLastError());
    return;
  }
  dispatch_walk(e.C, e.walk_nq, [&](auto c, auto nq) {
    constexpr int C = decltype(c)::value, NQ = decltype(nq)::value;
    hipLaunchKernelGGL((k_forward_walk<4, C, NQ>), dim3(waves), dim3(64), forward_walk_lds(NQ, e.fwd_slots), e.stream,
                       ops, n_ops, e.fwd_slots, e.L, e.d_clv.as<double>(), e.d_scl.as<int32_t>(),
                       e.d_tips.as<uint8_t>(), e.d_P.as<double>(), e.d_freqs.as<double>(), e.d_weights.as<double>(),
                       e.d_tile_part.as<int32_t>(), e.d_root_partials.as<double>(), e.d_site_seed.as<double>());
  });
  NRX_HIP(hipGetLastError());
}

void launch_mixture(Engine &e, int variant, int pw, double *host) {
  const int nr = static_cast<int>(e.root_slots.size());
  // few root sums of few partials are formed by the mixture's workgroup, which
  // saves a launch (4.8 us with the gap): it adds about 500 partials per us, and
  // a sum takes one of its four waves 1 us (lnL of 12 taxa: 16 sums 47 us either
  // way, 32 sums 59 us in the workgroup, 54 before it, 256 sums 96 and 42)
  const int64_t n_wt = static_cast<int64_t>(e.L.n_tiles) * pw;
  const bool fused = nr * n_wt <= MIX_PARTIALS && nr * e.P <= MIX_ROWS;
  if (!fused) {
    hipLaunchKernelGGL(k_reduce_segments, dim3(nr * e.P), dim3(256), 0, e.stream, e.d_root_partials.as<double>(),
                       static_cast<size_t>(n_wt), pw, e.d_part_tile_begin.as<int32_t>(), e.P,
                       e.d_root_sums.as<double>());
    NRX_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL(k_mixture, dim3(1), dim3(256), sizeof(double) * MIX_LDS_DOUBLES, e.stream, e.L, nr,
                     static_cast<int>(e.dag.classes.size()), e.R, variant,
                     e.d_classes.as<DevClass>(), e.d_class_dlogprob.as<double>(),
                     e.d_root_sums.as<double>(), e.d_beta.as<double>(), e.d_result.as<double>(), host, e.rl,
                     fused ? e.d_root_partials.as<double>() : nullptr, pw, e.d_part_tile_begin.as<int32_t>());
  NRX_HIP(hipGetLastError());
}

void launch_adjoint_walk(Engine &e, const DevOp *ops, int n_ops, bool model) {
  if (n_ops == 0) return;
  const unsigned waves = static_cast<unsigned>(e.L.n_tiles) * (model ? e.model_wpt() : e.rpw);
  if (e.S == AA_STATES) {
    if (model) throw std::logic_error("launch_adjoint_walk: model gradients are built for 4-state data");
    dispatch_c(e.C, [&](auto c) {
      constexpr int C = decltype(c)::value;
      hipLaunchKernelGGL((k_adjoint_level_aa<C>), dim3(waves * C), dim3(64), adjoint_walk_lds_aa(e.adj_slots), e.stream,
                         ops, n_ops, e.adj_slots, e.L, e.d_clv.as<double>(), e.d_scl.as<int32_t>(),
                         e.d_adj.as<double>(), e.d_tips.as<uint32_t>(), e.d_PA.as<double>(), e.d_Qd.as<double>(),
                         e.d_freqs.as<double>(), e.d_site_seed.as<double>(), e.d_tile_part.as<int32_t>(),
                         e.d_beta.as<double>(), static_cast<int>(e.root_slots.size()), e.n_uses,
                         e.d_grad_partials.as<double>());
    });
    NRX_HIP(hipGetLastError());
    return;
  }
  auto go = [&](auto kernel, int nq, int slots, const DevBuf &partials) {
    hipLaunchKernelGGL(kernel, dim3(waves), dim3(64), adjoint_walk_lds(nq, slots), e.stream, ops, n_ops, e.L,
                       e.d_clv.as<double>(), e.d_scl.as<int32_t>(), e.d_adj.as<double>(), e.d_tips.as<uint8_t>(),
                       e.d_P.as<double>(), e.d_Qd.as<double>(), e.d_freqs.as<double>(), e.d_site_seed.as<double>(),
                       e.d_tile_part.as<int32_t>(), e.d_beta.as<double>(), static_cast<int>(e.root_slots.size()),
                       e.n_uses, partials.as<double>());
  };
  if (model)
    dispatch_c(e.C, [&](auto c) {
      constexpr int C = decltype(c)::value;
      if (e.model_nq() == 4) return go(k_model_adjoint<C, 4>, 4, e.model_slots, e.d_mg_r);
      if constexpr (C != 8) go(k_model_adjoint<C, 2>, 2, e.model_slots, e.d_mg_r);
    });
  else
    dispatch_walk(e.C, e.walk_nq, [&](auto c, auto nq) {
      constexpr int C = decltype(c)::value, NQ = decltype(nq)::value;
      go(k_adjoint_level<C, NQ>, NQ, e.adj_slots, e.d_grad_partials);
    });
  NRX_HIP(hipGetLastError());
}

void launch_grad_reduce(Engine &e, double *host) {
  hipLaunchKernelGGL(k_reduce_grad, dim3((e.n_uses + 63) / 64, e.P * GRAD_SLICES), dim3(256), 0, e.stream,
                     e.d_grad_partials.as<double>(), e.n_uses, e.gwpt, e.d_part_tile_begin.as<int32_t>(), e.P,
                     e.d_use_sums.as<double>());
  NRX_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_grad_total, dim3(e.E), dim3(256), 0, e.stream, e.E, e.P, e.d_edge_use_begin.as<int32_t>(),
                     e.d_edge_use_list.as<int32_t>(), e.d_use_sums.as<double>(), e.d_result.as<double>(), host, e.rl);
  NRX_HIP(hipGetLastError());
}

// Shapes of the 4-state FP32 walks: C categories, one or two row blocks.
template <typename F>
static void dispatch_walk32(int C, int blocks, F &&f) {
  dispatch_c(C, [&](auto c) {
    if (blocks == 2)
      f(c, std::integral_constant<int, 2>{});
    else
      f(c, std::integral_constant<int, 3>{});
  });
}

void launch_forward_persistent(Engine &e, const NetDesc *nets) {
  launch_forward_persistent_multi(e.stream, e.C, e.walk_blocks, nets ? nets : e.d_netdesc.as<NetDesc>(),
                                  e.d_work.as<WorkItem>(), e.L.n_tiles * e.gwpt, e.fwd_slots);
}

void launch_adjoint_persistent(Engine &e) {
  launch_adjoint_persistent_multi(e.stream, e.C, e.walk_blocks, e.d_netdesc.as<NetDesc>(), e.d_work.as<WorkItem>(),
                                  e.L.n_tiles * e.gwpt, e.adj_slots);
}

void launch_forward_persistent_multi(hipStream_t stream, int C, int blocks, const NetDesc *nets, const WorkItem *work,
                                     int n_work, int slots) {
  if (n_work == 0) return;
  dispatch_walk32(C, blocks, [&](auto c, auto g) {
    hipLaunchKernelGGL((k_forward_persistent<decltype(c)::value, decltype(g)::value, 64>), dim3(n_work), dim3(64),
                       forward_lds32(C, blocks, slots), stream, nets, work);
  });
  NRX_HIP(hipGetLastError());
}

void launch_adjoint_persistent_multi(hipStream_t stream, int C, int blocks, const NetDesc *nets, const WorkItem *work,
                                     int n_work, int slots) {
  if (n_work == 0) return;
  dispatch_walk32(C, blocks, [&](auto c, auto g) {
    hipLaunchKernelGGL((k_adjoint_persistent<decltype(c)::value, decltype(g)::value, 64>), dim3(n_work), dim3(64),
                       adjoint_lds32(C, blocks, slots), stream, nets, work);
  });
  NRX_HIP(hipGetLastError());
}

void launch_forward_mfma(Engine &e, const NetDesc *nets) {
  dispatch_c(e.C, [&](auto c) {
    constexpr int C = decltype(c)::value;
    hipLaunchKernelGGL((k_forward_mfma<C, 4>), dim3(e.L.n_tiles * e.rpw), dim3(64 * C), forward_lds_aa32(C, e.fwd_slots),
                       e.stream, nets ? nets : e.d_netdesc.as<NetDesc>());
  });
  NRX_HIP(hipGetLastError());
}

void launch_adjoint_mfma(Engine &e) {
  dispatch_c(e.C, [&](auto c) {
    constexpr int C = decltype(c)::value;
    hipLaunchKernelGGL((k_adjoint_mfma<C>), dim3(e.L.n_tiles * e.rpw * C), dim3(64), adjoint_lds_aa32(e.adj_slots),
                       e.stream, e.d_netdesc.as<NetDesc>());
  });
  NRX_HIP(hipGetLastError());
}

void launch_sumtables(Engine &e, int n_paths, int max_steps) {
  if (n_paths == 0) return;
  const size_t lds = path_lds_bytes(e.S, e.C, max_steps);
  dispatch_sc(e.S, e.C, [&](auto s, auto c) {
    constexpr int S = decltype(s)::value, C = decltype(c)::value;
    using TT = typename TipType<S>::type;
    if (e.opt.precision == NRX_FP32) {
      if constexpr (S == 4)
        hipLaunchKernelGGL((k_sumtables<S, C, float>), dim3(e.L.n_tiles, n_paths), dim3(TILE * C), lds,
                           e.stream, e.d_steps.as<PathStep>(), e.d_path_begin.as<int32_t>(), n_paths,
                           e.L, e.d_tile_part.as<int32_t>(),
                           e.d_clv.as<float>(), e.d_scl.as<int32_t>(), 1, e.d_tips.as<TT>(),
                           e.d_P.as<double>(), e.d_V.as<double>(), e.d_Vinv.as<double>(),
                           e.d_freqs.as<double>(), e.d_st.as<double>());
      else
        throw std::logic_error("sumtables of 20 states are of the FP64 form");
    } else {
      // (4 states: see the kernel)
      const dim3 grid = S == 4 ? dim3((e.L.n_tiles + 7) / 8 * 8 * n_paths) : dim3(e.L.n_tiles, n_paths);
      hipLaunchKernelGGL((k_sumtables<S, C, double>), grid, dim3(TILE * C), S == 4 ? 0 : lds,
                         e.stream, e.d_steps.as<PathStep>(), e.d_path_begin.as<int32_t>(), n_paths,
                         e.L, e.d_tile_part.as<int32_t>(),
                         e.d_clv.as<double>(), e.d_scl.as<int32_t>(), 256, e.d_tips.as<TT>(),
                         e.d_P.as<double>(), e.d_V.as<double>(), e.d_Vinv.as<double>(),
                         e.d_freqs.as<double>(), e.d_st.as<double>());
    }
  });
  NRX_HIP(hipGetLastError());
}

void launch_sumtable_eval(Engine &e, int n_paths, double brlen) {
  if (n_paths == 0) return;
  dispatch_sc(e.S, e.C, [&](auto s, auto c) {
    constexpr int S = decltype(s)::value, C = decltype(c)::value;
    hipLaunchKernelGGL((k_sumtable_eval<S, C>), dim3(e.L.n_tiles, n_paths), dim3(TILE * C), 0, e.stream,
                       e.d_st.as<double>(), n_paths, e.L, e.d_tile_part.as<int32_t>(),
                       e.d_eval.as<double>(), e.d_rates.as<double>(), e.d_weights.as<double>(),
                       brlen, e.d_st_partials.as<double>());
  });
  NRX_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_reduce_segments, dim3(n_paths * 3 * e.P), dim3(256), 0, e.stream,
                     e.d_st_partials.as<double>(), static_cast<size_t>(e.L.n_tiles) * e.pw, e.pw,
                     e.d_part_tile_begin.as<int32_t>(), e.P, e.d_st_sums.as<double>());
  NRX_HIP(hipGetLastError());
}


// Scratch of the allocation-free branch derivatives (nrx_brlen_derivatives_noalloc):
// a fixed device array, one copy per GPU, whose address host code takes
// once per device from hipGetSymbolAddress (the array's name in host code
// is not a device address).
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

void *noalloc_scratch() {
  static std::mutex mu;
  static std::map<int, void *> ptr_of_device;
  int dev = 0;
  NRX_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(mu);
  const auto it = ptr_of_device.find(dev);
  if (it != ptr_of_device.end()) return it->second;
  void *ptr = nullptr;
  NRX_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
  if (!ptr) throw std::runtime_error("HIP error: no device address for the no-alloc scratch");
  ptr_of_device[dev] = ptr;
  return ptr;
}

void launch_deriv_fused(Engine &e, const PathStep *steps, const int32_t *path_begin, int n_paths, int max_steps,
                        double brlen, double *partials, double *sums) {
  if (n_paths == 0) return;
  const size_t lds = path_lds_bytes(e.S, e.C, max_steps);
  dispatch_sc(e.S, e.C, [&](auto s, auto c) {
    constexpr int S = decltype(s)::value, C = decltype(c)::value;
    using TT = typename TipType<S>::type;
    if (e.opt.precision == NRX_FP32) {
      if constexpr (S == 4)
        hipLaunchKernelGGL((k_deriv_fused<S, C, float>), dim3(e.L.n_tiles), dim3(TILE * C), lds, e.stream, steps,
                           path_begin, n_paths, e.L, e.d_tile_part.as<int32_t>(), e.d_clv.as<float>(),
                           e.d_scl.as<int32_t>(), 1, e.d_tips.as<TT>(), e.d_P.as<double>(), e.d_V.as<double>(),
                           e.d_Vinv.as<double>(), e.d_freqs.as<double>(), e.d_eval.as<double>(),
                           e.d_rates.as<double>(), e.d_weights.as<double>(), brlen, partials);
      else
        throw std::logic_error("branch derivatives of 20 states are of the FP64 form");
    } else {
      hipLaunchKernelGGL((k_deriv_fused<S, C, double>), dim3(e.L.n_tiles), dim3(TILE * C), S == 4 ? 0 : lds, e.stream,
                         steps, path_begin, n_paths, e.L, e.d_tile_part.as<int32_t>(),
                         e.d_clv.as<double>(), e.d_scl.as<int32_t>(), 256, e.d_tips.as<TT>(),
                         e.d_P.as<double>(), e.d_V.as<double>(), e.d_Vinv.as<double>(), e.d_freqs.as<double>(),
                         e.d_eval.as<double>(), e.d_rates.as<double>(), e.d_weights.as<double>(), brlen,
                         partials);
    }
  });
  NRX_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_reduce_segments, dim3(n_paths * 3 * e.P), dim3(256), 0, e.stream, partials,
                     static_cast<size_t>(e.L.n_tiles) * e.pw, e.pw, e.d_part_tile_begin.as<int32_t>(), e.P, sums);
  NRX_HIP(hipGetLastError());
}

void launch_model_grad(Engine &e, double *g_sum, double *r_sum, double *edge_out, double *out, int n_slice) {
  const int n_root = static_cast<int>(e.root_slots.size()), nl = e.C == 8 ? 128 : 64;
  hipLaunchKernelGGL(k_model_reduce, dim3(e.n_uses + n_root, e.P * n_slice), dim3(256), 0, e.stream,
                     e.d_adj.as<double>(), e.clv_elems_per_slot, e.model_nq() * 64, e.d_use_row.as<int32_t>(),
                     e.d_mg_r.as<double>(), e.n_uses, nl, e.L.n_tiles * e.model_wpt(), e.model_wpt(),
                     e.d_part_tile_begin.as<int32_t>(), e.P, n_slice, g_sum, r_sum);
  NRX_HIP(hipGetLastError());
  dispatch_c(e.C, [&](auto c) {
    constexpr int C = decltype(c)::value;
    hipLaunchKernelGGL((k_model_chain<C>), dim3(e.E, e.P), dim3(64), 0, e.stream, e.L, g_sum, n_slice,
                       e.d_edge_use_begin.as<int32_t>(), e.d_edge_use_list.as<int32_t>(), e.d_V.as<double>(),
                       e.d_Vinv.as<double>(), e.d_eval.as<double>(), e.d_rates.as<double>(), e.d_brlen.as<double>(),
                       edge_out);
  });
  NRX_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_model_total, dim3(e.P), dim3(256), 0, e.stream, e.E, e.C, n_root, n_slice, e.P, edge_out, r_sum,
                     out);
  NRX_HIP(hipGetLastError());
}

void enqueue_newton(Engine &e, int variant, int mode, int rounds, int max_paths, NewtonState *st,
                    const DerivClassDev *cls, const double *base_logl) {
  const int nc = static_cast<int>(e.dag.classes.size());
  const size_t row_stride = static_cast<size_t>(e.L.n_tiles) * e.pw;
  auto eval_reduce = [&](int final_eval) {
    dispatch_sc(e.S, e.C, [&](auto s, auto c) {
      constexpr int S = decltype(s)::value, C = decltype(c)::value;
      hipLaunchKernelGGL((k_sumtable_eval_nr<S, C>), dim3(e.L.n_tiles, max_paths), dim3(TILE * C), 0, e.stream,
                         e.d_st.as<double>(), e.L, e.d_tile_part.as<int32_t>(), e.d_eval.as<double>(),
                         e.d_rates.as<double>(), e.d_weights.as<double>(), st, final_eval,
                         e.d_st_partials.as<double>());
    });
    NRX_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_reduce_segments_nr, dim3(max_paths * 3 * e.P), dim3(256), 0, e.stream,
                       e.d_st_partials.as<double>(), row_stride, e.pw, e.d_part_tile_begin.as<int32_t>(), e.P, st,
                       final_eval, e.d_st_sums.as<double>());
    NRX_HIP(hipGetLastError());
  };
  for (int it = 0; it < rounds; ++it) {
    eval_reduce(0);
    hipLaunchKernelGGL(k_newton_step, dim3(1), dim3(64), NR_LDS_BYTES, e.stream, e.d_st_sums.as<double>(), e.P,
                       nc, cls, base_logl, variant, mode, st);
    NRX_HIP(hipGetLastError());
  }
  eval_reduce(1);
  hipLaunchKernelGGL(k_newton_accept, dim3(1), dim3(64), NR_LDS_BYTES, e.stream, e.d_st_sums.as<double>(), e.P,
                     nc, cls, base_logl, variant, st);
  NRX_HIP(hipGetLastError());
}

void launch_pmatrices_multi(hipStream_t s, const SmallDesc *d, int n, int max_elems) {
  hipLaunchKernelGGL(k_pmatrices_multi, dim3((max_elems + 255) / 256, n), dim3(256), 0, s, d);
  NRX_HIP(hipGetLastError());
}

void launch_root_reduce_multi(hipStream_t s, const SmallDesc *d, int n, int max_rows) {
  if (max_rows == 0) return;
  hipLaunchKernelGGL(k_root_reduce_multi, dim3(max_rows, n), dim3(256), 0, s, d);
  NRX_HIP(hipGetLastError());
}

void launch_mixture_multi(hipStream_t s, const SmallDesc *d, int n, int variant) {
  hipLaunchKernelGGL(k_mixture_multi, dim3(n), dim3(256), sizeof(double) * MIX_LDS_DOUBLES, s, d, variant);
  NRX_HIP(hipGetLastError());
}

void launch_grad_reduce_multi(hipStream_t s, const SmallDesc *d, int n, int max_uses, int max_parts, int max_edges) {
  if (max_uses > 0) {
    hipLaunchKernelGGL(k_use_reduce_multi, dim3((max_uses + 63) / 64, max_parts * GRAD_SLICES, n), dim3(256), 0, s, d);
    NRX_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL(k_grad_total_multi, dim3(max_edges, n), dim3(256), 0, s, d);
  NRX_HIP(hipGetLastError());
}

void launch_gather_results(hipStream_t s, const SmallDesc *d, int n, const int64_t *offsets,
                           double *out, int max_size) {
  hipLaunchKernelGGL(k_gather_results, dim3((max_size + 255) / 256, n), dim3(256), 0, s, d,
                     offsets, out);
  NRX_HIP(hipGetLastError());
}

}  // namespace nrx
