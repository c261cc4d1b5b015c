// Batched LM for small robot-3D-localization problems: one persistent launch, one wavefront per
// problem running the whole Levenberg-Marquardt loop (the state-block bookkeeping of
// LevenbergMarquardtSolver::Iterate, levenberg_marquardt_solver.tcc:138-343, with the shared
// accept / lambda logic of lm_logic.h).
//
// Structure exploited: the optimized keys are the poses of one chain, odometry factors join
// consecutive poses and matching factors touch one pose, so H is block tridiagonal with 6 x 6
// blocks. Lane i linearizes pose i (its matching factors and the odometry factor to pose i + 1,
// whose pose-(i + 1) terms are handed to lane i + 1 by a shuffle); the wavefront then solves the
// damped system by a block-tridiagonal LDL^T from both ends of the chain at once. Per state block
// and pose the linearization keeps 63 doubles: the lower diagonal block (21), H(i + 1, i) (36,
// row-major) and the rhs (6), entry by entry over the poses so that a wavefront's lanes read and
// write consecutive addresses.
#include "./batch.h"

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <mutex>
#include <type_traits>

#include "./dpp.h"
#include "./factor_traits.h"
#include "./geo.h"
#include "./lm_logic.h"
#include "./problem.h"
#include "./util.h"

namespace symhip {

namespace {

constexpr int kLin = 63;
// offsets of a pose's record: lower diagonal block, H(i + 1, i), rhs
constexpr int kRecB = 21, kRecX = 57;
constexpr int kRec = 65;  // LDS stride of a pose's record (odd: lanes on their own poses spread over the banks)
constexpr int kMaxPoses = 64;

struct BatchView {
  int64_t total_poses;
  const int32_t* pose_begin;  // [n_problems + 1] global pose index
  const int32_t* pose_soff;   // [total_poses] offset of the initial pose value in cvals
  const int32_t* match_ptr;   // [total_poses + 1]
  const int32_t* match_args;  // 3 per match: landmark, measurement, sigma offsets in cvals
  const int32_t* odo_args;    // 3 per pose: measurement, sigmas, epsilon offsets (-1: last pose)
  const double* cvals;
  double* vals;  // [3][total_poses][7]
  double* lin;   // [3][kLin][total_poses]
  double* maxd;  // [total_poses][6]
  double* vout;  // storage copy; best poses written back
  symhip_iteration_stats* recs;
  int32_t rec_stride;
  symhip_optimization_stats* stats;
  int64_t* ticks;  // [n_problems][2]
  const int32_t* order;  // workgroup -> problem (null: the identity)
};

__device__ __forceinline__ double wave_total(double v) {
  v = xor16_sum(xor32_sum(v));
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

__device__ __forceinline__ int tri(int r, int c) { return r * (r + 1) / 2 + c; }

// Relinearize state block b: lane i < n writes pose i's D, H(i + 1, i), rhs. Returns the error
// 0.5 |r|^2 of the problem (the same value in every lane). With S = float (the precision form)
// the Jacobians come from the FP32 factor bodies while the residual, and with it the cost and
// the gradient J^T r, comes from the FP64 bodies: the cost stays FP64-accurate, so LM's gain
// ratio and relative-reduction exit behave as in FP64 (FP32 residuals put a ~1e-7 floor under
// the cost, which kept LM from its early exit on some problems). The products J^T J are formed
// in FP64 from the FP32 Jacobians, so H stays positive semi-definite (FP32 sums of products
// made a near-singular H slightly indefinite: the LDL^T takes no square roots and gives a finite
// step there that need not descend, an iteration spent on its rejection).
template <typename S>
__device__ __forceinline__ double linearize(const BatchView& v, int b, int g0, int n, int lane) {
  double D[21] = {}, gv[6] = {}, Dn[21] = {}, gn[6] = {};
  double e = 0;
  int has_next = 0;
  const bool live = lane < n;
  const int g = g0 + min(lane, n - 1);
  const int64_t TP = v.total_poses;
  double* lin = v.lin + (int64_t)b * kLin * TP;  // entry k of pose g at lin[k * TP + g]
  auto put = [&](int k, double x) { (lin + k * TP)[g] = x; };
  if (live) {
    const double* pose = v.vals + (b * TP + g) * 7;
    const int32_t* oa = v.odo_args + 3 * g;
    if (oa[0] >= 0) {
      has_next = 1;
      const double* a[5] = {pose, pose + 7, v.cvals + oa[0], v.cvals + oa[1], v.cvals + oa[2]};
      S rs[6], J[6][12];
      factor_odometry<S>(a, rs, J);
      double r[6], Jd[6][12];
      if constexpr (std::is_same_v<S, double>) {
#pragma unroll
        for (int q = 0; q < 6; ++q) r[q] = rs[q];
      } else {
        factor_odometry<double>(a, r, Jd);
      }
      // sum_q J[q][i] J[q][j] over the residual rows where both columns have entries: rotation
      // columns of the first pose touch all six rows, those of the second the first three,
      // translation columns the last three (factor_odometry); the other products are zeros.
      auto dot = [&](int i, int j, int q0, int q1) {
        double h = 0;
        for (int q = q0; q < q1; ++q) h += (double)J[q][i] * (double)J[q][j];
        return h;
      };
#pragma unroll
      for (int i = 0; i < 6; ++i) {
        double ga = 0, gb = 0;
        for (int q = i < 3 ? 0 : 3; q < 6; ++q) ga += (double)J[q][i] * r[q];
        for (int q = i < 3 ? 0 : 3; q < (i < 3 ? 3 : 6); ++q) gb += (double)J[q][6 + i] * r[q];
        gv[i] = ga;
        gn[i] = gb;
        // H(i + 1, i), rows of the next pose, columns of this one: stored as it is formed
#pragma unroll
        for (int j = 0; j < 6; ++j) {
          const double hb = i < 3 ? (j < 3 ? dot(6 + i, j, 0, 3) : 0.0) : dot(6 + i, j, 3, 6);
          put(kRecB + i * 6 + j, hb);
        }
#pragma unroll
        for (int j = 0; j <= i; ++j) {
          D[tri(i, j)] = j < 3 && i < 3 ? dot(i, j, 0, 6) : dot(i, j, 3, 6);
          Dn[tri(i, j)] = i < 3 ? dot(6 + i, 6 + j, 0, 3) : (j < 3 ? 0.0 : dot(6 + i, 6 + j, 3, 6));
        }
      }
#pragma unroll
      for (int q = 0; q < 6; ++q) e += r[q] * r[q];
    } else {
#pragma unroll
      for (int k = 0; k < 36; ++k) put(kRecB + k, 0.0);
    }
  }
  // the odometry factor's pose-(i + 1) terms belong to the next lane
  const int prev = __shfl_up(has_next, 1, 64);
  const bool take = lane >= 1 && prev != 0;
#pragma unroll
  for (int k = 0; k < 21; ++k) {
    const double t = __shfl_up(Dn[k], 1, 64);
    if (take) D[k] += t;
  }
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const double t = __shfl_up(gn[k], 1, 64);
    if (take) gv[k] += t;
  }
  // The matching factors. A problem of at most 32 (16) poses gives each pose two (four) lanes,
  // lane + 32 (lane + 16, ..), which take its factors in turn. A lane takes kMatch of them at a
  // time: their offsets in one round of loads, their inputs in the next (one factor after the
  // other waits for both rounds; the compiler sinks a hand-pipelined loop's loads back to their
  // uses). Past the list's end the last factor repeats with an infinite sigma, which adds zeros. A
  // problem without poses (hand-made tables) reads row g0 in place of a row before the tables: an
  // entry of match_ptr in any case, and of the pose blocks or the linearizations behind them.
  {
    constexpr int kMatch = 4;
    const int stride = n <= 16 ? 16 : n <= 32 ? 32 : 64;
    const int parts = 64 / stride, i = lane & (stride - 1), part = lane / stride;
    const int gm = g0 + min(i, max(n, 1) - 1);
    const double* pose = v.vals + (b * TP + gm) * 7;
    const int m0 = v.match_ptr[gm], m1 = i < n ? v.match_ptr[gm + 1] : m0;
    double p[7];
#pragma unroll
    for (int k = 0; k < 7; ++k) p[k] = pose[k];
    for (int m = m0 + part; m < m1; m += kMatch * parts) {
      int32_t o[kMatch][3];
#pragma unroll
      for (int t = 0; t < kMatch; ++t)
#pragma unroll
        for (int k = 0; k < 3; ++k) o[t][k] = v.match_args[3 * min(m + t * parts, m1 - 1) + k];
      double lm[kMatch][3], meas[kMatch][3], sigma[kMatch];
#pragma unroll
      for (int t = 0; t < kMatch; ++t) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          lm[t][k] = v.cvals[o[t][0] + k];
          meas[t][k] = v.cvals[o[t][1] + k];
        }
        sigma[t] = v.cvals[o[t][2]];
      }
#pragma unroll
      for (int t = 0; t < kMatch; ++t) {
        const double sg = m + t * parts < m1 ? sigma[t] : __builtin_huge_val();
        const double* a[4] = {p, lm[t], meas[t], &sg};
        S rs[3], J[3][6];
        factor_matching<S>(a, rs, J);
        double r[3], Jd[3][6];
        if constexpr (std::is_same_v<S, double>) {
#pragma unroll
          for (int q = 0; q < 3; ++q) r[q] = rs[q];
        } else {
          factor_matching<double>(a, r, Jd);
        }
        // rotation column c has no entry in row c (a cross product's matrix)
#pragma unroll
        for (int c = 0; c < 6; ++c)
#pragma unroll
          for (int q = 0; q < 3; ++q) {
            if (q == c) continue;
            const double jc = (double)J[q][c];
            gv[c] = fma(jc, r[q], gv[c]);
#pragma unroll
            for (int d = 0; d <= c; ++d)
              if (q != d) D[tri(c, d)] = fma(jc, (double)J[q][d], D[tri(c, d)]);
          }
#pragma unroll
        for (int q = 0; q < 3; ++q) e = fma(r[q], r[q], e);
      }
    }
    // the lanes of a pose together
    if (parts > 1) {
#pragma unroll
      for (int k = 0; k < 21; ++k) D[k] = xor32_sum(D[k]);
#pragma unroll
      for (int k = 0; k < 6; ++k) gv[k] = xor32_sum(gv[k]);
    }
    if (parts > 2) {
#pragma unroll
      for (int k = 0; k < 21; ++k) D[k] = xor16_sum(D[k]);
#pragma unroll
      for (int k = 0; k < 6; ++k) gv[k] = xor16_sum(gv[k]);
    }
  }
  if (live) {
#pragma unroll
    for (int k = 0; k < 21; ++k) put(k, D[k]);
#pragma unroll
    for (int k = 0; k < 6; ++k) put(kRecX + k, gv[k]);
  }
  return 0.5 * wave_total(e);
}

__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Block-tridiagonal LDL^T of H and the two triangular solves, by the whole wavefront, from both
// ends of the chain towards its middle pose m = n / 2 (no fill: each half's elimination touches its
// own poses only, and the middle block takes an update from either side). The row of lanes 0..15
// eliminates poses 0, 1, .. m - 1, the row of lanes 16..31 poses n - 1, n - 2, .. m + 1 (one fewer
// when n is even: its first step is an identity pose), the upper two rows repeat them.
//
// Inside a row, a step's lanes hold the rows of [A_i; B; x_i^T]: six pivot rows of the pose's
// diagonal block, the six rows that its coupling block gives the next pose towards the middle, and
// the right-hand side as a thirteenth row. All of them undergo the same elimination: for column k,
// d = pivot k, l = own entry / d, and the columns after it lose l times the pivot rows' entries,
// which cross the row of lanes by row_bcast. Each non-pivot row then forms its row of the next
// pose's update, -sum_k l_k w_ck (w = l d, row c's from its lane), so the next diagonal block and
// right-hand side appear in the lanes that held the coupling block: pivot rows alternate between
// lanes 0..5 and 6..11 from step to step, and nothing moves. In the records (LDS) A's strict lower
// part is overwritten by -L, B by the coupling rows' -l, x by -D^-1 L^-1 x and then by the solution.
//
// A step's dependent chain is six reciprocals with their updates, ~0.3 us: one row of lanes
// eliminating the whole chain by Cholesky, with scalar lane reads, square roots and divisions, took
// four times as long per pose and twice the poses (4096 problems of 5-50 poses: 1.98 ms a launch,
// one wavefront per SIMD; with this and the linearization above 0.43).
//
// Columns K.. of a step whose pivot rows are in lanes kBase.. of each row of lanes and whose coupling
// rows are in lanes kCouple..: v's column K becomes the unscaled w_K, nl_K = -w_K / d_K, and acc_c
// collects sum_k nl_k w_ck with w_ck from lane kCouple + c (each column's share as soon as its nl
// is there, behind the next column's reciprocal).
template <int kBase, int kCouple, int K = 0>
__device__ __forceinline__ void eliminate(double (&v)[6], double (&nl)[6], double (&acc)[6]) {
  if constexpr (K < 6) {
    const double w = v[K];
    nl[K] = w * -refined_rcp(row_bcast<kBase + K>(w));
    row_fmac<kBase + K + 1, 5 - K>(v + K + 1, w, nl[K]);
    row_fmac<kCouple, 6>(acc, w, nl[K]);
    eliminate<kBase, kCouple, K + 1>(v, nl, acc);
  }
}
// t_c += nl(q, c) x_q for q = 5 .. 1, x_q = t of lane q (lc[q] = nl(q, own c), zero where c >= q)
template <int Q = 5>
__device__ __forceinline__ void back_columns(double& t, const double (&lc)[6]) {
  if constexpr (Q > 0) {
    t = fma(lc[Q], row_bcast<Q>(t), t);
    back_columns<Q - 1>(t, lc);
  }
}
// t += sum_r wc_r x_r, x_r from lane r (wc_r = nl of coupling row r, own column)
template <int R = 0>
__device__ __forceinline__ void back_coupling(double& t, const double (&wc)[6], double x) {
  if constexpr (R < 6) {
    t = fma(wc[R], row_bcast<R>(x), t);
    back_coupling<R + 1>(t, wc, x);
  }
}

__device__ __forceinline__ void block_tridiagonal_solve(int n, double* rec, int lane) {
  const int q = lane & 15;
  const bool second = (lane >> 4) & 1;  // the chain from the far end
  const int m = n >> 1;                    // the middle pose: m steps on the first chain,
  const int skip = m - (n - 1 - m);        // m - skip on the second
  // offsets of this lane's row in a pose's record, as a pivot row, a coupling row (row r of the
  // pose towards the middle; the second chain's block is stored transposed) or the rhs row, for the
  // two alternating lane roles; kept as row r and its role
  const int r0 = q < 6 ? q : q - 6;
  auto offset = [&](bool pivot, bool rhs, int c) {
    const int a = c <= r0 ? tri(r0, c) : tri(c, r0);
    const int b = kRecB + (second ? c * 6 + r0 : r0 * 6 + c);
    return rhs ? kRecX + c : pivot ? a : b;
  };
  const bool rhs_row = q >= 12;
  // the pose of step s on this lane's chain (clamped at the second chain's identity step)
  auto pose_of = [&](int s) { return second ? min(n - 1, n - 1 - (s - skip)) : s; };
  auto is_pivot = [&](int par) { return par == 0 ? q < 6 : q >= 6 && !rhs_row; };
  // a coupling row of the second chain is in the record of the pose before its own
  auto record = [&](int s, int par) {
    const int p = pose_of(s);
    return (!is_pivot(par) && !rhs_row && second ? max(p - 1, 0) : p) * kRec;
  };
  // Rows are read whole and written but for a pivot row's entries from its diagonal on: those go
  // to the record's padding, and all entries of lanes that have nothing to store (the repeating
  // rows of lanes, the spare lanes, the identity pose) to the spare record, without a branch.
  int off[2][6], put[2][6];
#pragma unroll
  for (int par = 0; par < 2; ++par)
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      off[par][c] = offset(is_pivot(par), rhs_row, c);
      put[par][c] = is_pivot(par) && c >= r0 ? kLin : off[par][c];
    }
  const bool writer = lane < 32 && q <= 12;
  double acc[6] = {}, cur[6], nl[6];
  auto load = [&](int s, int par) {
    const double* x = rec + record(s, par);
#pragma unroll
    for (int c = 0; c < 6; ++c) cur[c] = x[off[par][c]];
  };
  auto step = [&]<int kPar>(int s) __attribute__((always_inline)) {
    constexpr int kPivot = kPar ? 6 : 0, kCouple = kPar ? 0 : 6;
    double v[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) v[c] = cur[c] + acc[c];
    load(min(s + 1, m - 1), kPar ^ 1);  // the next step's rows (not used after the last one)
#pragma unroll
    for (int c = 0; c < 6; ++c) acc[c] = 0.0;
    eliminate<kPivot, kCouple>(v, nl, acc);
    double* x = rec + (writer && !(second && s < skip) ? record(s, kPar) : n * kRec);
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      x[put[kPar][c]] = nl[c];
      acc[c] = is_pivot(kPar) ? 0.0 : acc[c];  // these lanes take coupling rows next
    }
  };
  if (m > 0) {
    load(0, 0);
    if (second && skip > 0) {  // the identity pose: nothing couples
#pragma unroll
      for (int c = 0; c < 6; ++c) cur[c] = q < 6 && c == r0 ? 1.0 : 0.0;
    }
    for (int s = 0; s < m; s += 2) {
      step.template operator()<0>(s);
      if (s + 1 < m) step.template operator()<1>(s + 1);
    }
  }
  // The middle pose: its own block and right-hand side, plus the update of either chain.
  auto middle = [&]<int kPar>() __attribute__((always_inline)) {
    constexpr int kPivot = kPar ? 6 : 0;
    const bool row = is_pivot(kPar) || rhs_row;
    double v[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      const double x = rec[m * kRec + off[kPar][c]];
      const double mine = acc[c] + (second ? 0.0 : x);
      const double both = xor16_sum(mine);
      v[c] = row ? both : 0.0;
    }
    double unused[6] = {};
    eliminate<kPivot, 0>(v, nl, unused);
    double* x = rec + (lane < 13 && row ? m : n) * kRec;
#pragma unroll
    for (int c = 0; c < 6; ++c) x[put[kPar][c]] = nl[c];
  };
  if (m & 1) middle.template operator()<1>(); else middle.template operator()<0>();
  wave_lds_sync();  // the factor's rows are read by columns below
  // Back from the middle: x_i = L^-T (D^-1 L^-1 x_i - W^T x_next), lane c of a row holding column c.
  const int c = min(q, 5);
  int lo[6], wo[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    lo[k] = tri(k, c < k ? c : 0);
    wo[k] = kRecB + (second ? c * 6 + k : k * 6 + c);
  }
  double x = 0, lc[6], wc[6], z = 0;
  auto load_back = [&](int s) {
    const int p = s == m ? m : pose_of(s);
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      const double t = rec[p * kRec + lo[k]];
      lc[k] = c < k ? t : 0.0;
      wc[k] = s == m ? 0.0 : rec[(second ? max(p - 1, 0) : p) * kRec + wo[k]];
    }
    z = rec[p * kRec + kRecX + c];
  };
  load_back(m);
  for (int s = m; s >= 0; --s) {
    double t = -z;
    back_coupling(t, wc, x);
    double lq[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) lq[k] = lc[k];
    if (s > 0) load_back(s - 1);
    back_columns(t, lq);
    x = t;
    const int p = s == m ? m : pose_of(s);
    if (q < 6 && (s == m ? lane < 16 : lane < 32 && !(second && s < skip)))
      rec[p * kRec + kRecX + c] = x;
  }
  wave_lds_sync();
}

// LDS of a launch whose largest problem has max_poses poses (the launches that do not know it take
// kMaxPoses: four problems per CU; 50 poses: six).
constexpr uint32_t rec_bytes(int32_t max_poses) {
  return (uint32_t)((max_poses + 1) * kRec * sizeof(double));
}

// kWaves: wavefronts per SIMD the register allocation must allow (1: no spills, ~360 VGPRs; 2: as
// many more resident problems as their LDS records leave room for, at the cost of spilled
// registers); the batch autotuner picks per batch.
template <typename S, int kWaves>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kWaves)))
batch_lm_kernel(BatchView v, symhip_optimizer_params p, double eps) {
  extern __shared__ double rec[];  // a record per pose and a spare one (rec_bytes)
  const int prob = v.order ? v.order[blockIdx.x] : (int)blockIdx.x, lane = threadIdx.x;
  const int64_t t_start = wall_clock64();
  const int g0 = v.pose_begin[prob], n = v.pose_begin[prob + 1] - g0;
  const bool live = lane < n;
  const int g = g0 + min(lane, n - 1);
  const int64_t TP = v.total_poses;
  // Reset: the start Values go into the New block (block 1)
  if (live) {
    const double* src = v.cvals + v.pose_soff[g];
    double t[7];
    for (int k = 0; k < 7; ++k) t[k] = src[k];
    for (int k = 0; k < 7; ++k) v.vals[(TP + g) * 7 + k] = t[k];
  }
  // the first linearization reads the next lane's start pose (odometry), written just above
  __syncthreads();
  // the state blocks as Iterate's first step and first linearization leave them
  int init = 1, nw = 0, best = 1, fre = 2, best_index = 0;
  int status = 0, reason = 0, nrec = 0;
  bool have_max = false, done = false;
  double err[3] = {0, 0, 0};
  double lambda = p.initial_lambda, nu = p.dynamic_lambda_update_beta;
  auto record = [&](const symhip_iteration_stats& r) __attribute__((always_inline)) {
    if (lane == 0 && v.recs && nrec < v.rec_stride)
      v.recs[(int64_t)prob * v.rec_stride + nrec] = r;
    ++nrec;
  };
  // One damped step: New = Init retracted by the update. Returns this lane's share of the linear
  // error's update . (rhs - damping * update).
  auto take_step = [&]() __attribute__((always_inline)) {
    double lde = 0;
    // DampHessian (levenberg_marquardt_solver.tcc:22-54) out of place, and the staged system
    const double* lin = v.lin + (int64_t)init * kLin * TP;  // entry k of pose g at lin[k * TP + g]
    double damp[6] = {}, u[6] = {}, rhs[6] = {};
    if (live) {
      double* own = rec + lane * kRec;
      double t[kLin];
#pragma unroll
      for (int k = 0; k < kLin; ++k) t[k] = (lin + k * TP)[g];
      __builtin_amdgcn_sched_barrier(0);  // all loads in flight before the first LDS write
#pragma unroll
      for (int k = 0; k < kLin; ++k) own[k] = t[k];
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        rhs[k] = t[kRecX + k];
        const double dk = t[tri(k, k)];
        double d = 0;
        if (p.use_diagonal_damping) {
          if (p.keep_max_diagonal_damping) {
            const double md = have_max ? fmax(v.maxd[g * 6 + k], dk) : fmax(dk, p.diagonal_damping_min);
            v.maxd[g * 6 + k] = md;
            d = md * lambda;
          } else {
            d = fmax(dk, p.diagonal_damping_min) * lambda;
          }
        }
        if (p.use_unit_damping) d += lambda;
        damp[k] = d;
        // an infinite damping leaves no step; its reciprocal in the elimination would be a NaN (by
        // fmin 499 problems take 153.4 us instead of 151.3)
        const double h = dk + d;
        own[tri(k, k)] = h == __builtin_huge_val() ? DBL_MAX : h;
      }
    }
    if (p.use_diagonal_damping && p.keep_max_diagonal_damping) have_max = true;
    __syncthreads();
    block_tridiagonal_solve(n, rec, lane);
    __syncthreads();
    if (live) {
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        u[k] = -rec[lane * kRec + kRecX + k];
        lde += u[k] * (rhs[k] - damp[k] * u[k]);
      }
      // UpdateNewFromInit: New = Init retracted by the update
      const double* src = v.vals + (init * TP + g) * 7;
      double* dst = v.vals + (nw * TP + g) * 7;
      for (int k = 0; k < 7; ++k) dst[k] = src[k];
      rot3_retract_inplace(dst, u, eps);
      dst[4] += u[3];
      dst[5] += u[4];
      dst[6] += u[5];
    }
    __syncthreads();  // the records are rewritten next iteration
    return lde;
  };
  // One body for the start's linearization (iteration -1, of Init) and each step's (of New): the
  // code is fetched as it runs, a few times per launch, and a second copy of the linearization
  // costs more than the branches.
  int iteration = -1;
  while (iteration < p.iterations && !done) {
    double lde = 0;
    if (iteration >= 1) {
      const int t = init;
      init = nw;
      nw = t;
    }
    if (iteration >= 0) lde = take_step();
    const double e_new = linearize<S>(v, iteration < 0 ? init : nw, g0, n, lane);
    if (iteration < 0) {
      err[init] = e_new;
      symhip_iteration_stats r{};
      r.iteration = -1;
      r.new_error = e_new;
      r.current_lambda = lambda;
      record(r);
      if (!isfinite(e_new)) {
        status = SYMHIP_STATUS_FAILED;
        reason = SYMHIP_FAILURE_INITIAL_ERROR_NOT_FINITE;
        break;
      }
      iteration = 0;
      asm volatile("" : "+s"(iteration));  // keeps the first pass from being peeled into a copy
      continue;
    }
    err[nw] = e_new;
    lde = wave_total(lde);
    const LmDecision d = lm_decide(err[init], err[nw], err[best], lde, lambda, nu, iteration, p,
                                   0, 0.0, 0.0, 0.0, eps);
    record(d.rec);
    lambda = d.lambda;
    nu = d.nu;
    // the same in every lane: through readfirstlane the state blocks' indices stay scalar, and with
    // them the addresses of their records
    const int accept = __builtin_amdgcn_readfirstlane(d.accept);
    const int set_best = __builtin_amdgcn_readfirstlane(d.set_best);
    if (!accept) {
      const int s = nw;
      nw = init;
      init = s;
    } else {
      if (set_best) {
        if (best != nw) {
          if (best != init) fre = best;
          best = nw;
        }
        best_index = nrec - 1;
      }
      if (best == init) {
        init = fre;
        fre = best;
      }
    }
    status = __builtin_amdgcn_readfirstlane(d.status);
    reason = d.reason;
    done = status != 0;
    ++iteration;
  }
  if (!done && status == 0) status = SYMHIP_STATUS_HIT_ITERATION_LIMIT;
  if (live)
    for (int k = 0; k < 7; ++k) v.vout[v.pose_soff[g] + k] = v.vals[(best * TP + g) * 7 + k];
  if (lane == 0) {
    v.stats[prob] = symhip_optimization_stats{nrec, best_index, status, reason};
    v.ticks[2 * prob] = t_start;
    v.ticks[2 * prob + 1] = wall_clock64();
  }
}

}  // namespace

PackedBatch pack_batch(const symhip_problem_desc* descs, int32_t n_problems,
                       const symhip_optimizer_params& params) {
  SYMHIP_CHECK(descs && n_problems > 0, "batch: no problems");
  SYMHIP_CHECK(params.iterations > 0, "batch: iterations must be positive");
  SYMHIP_CHECK(!params.enable_bold_updates, "batch: bold updates are not supported");
  PackedBatch pk;
  pk.pose_begin.push_back(0);
  pk.match_ptr.push_back(0);
  for (int32_t pi = 0; pi < n_problems; ++pi) {
    HostProblem hp;
    build_host_problem(&descs[pi], hp);
    const int32_t n = (int32_t)hp.state_keys.size();
    SYMHIP_CHECK(n >= 1 && n <= kMaxPoses, "batch: each problem needs 1..64 optimized poses");
    std::vector<int32_t> pos_of(hp.n_keys, -1);
    for (int32_t i = 0; i < n; ++i) {
      SYMHIP_CHECK(hp.types[hp.state_keys[i]] == SYMHIP_TYPE_POSE3,
                   "batch: optimized keys must be Pose3");
      pos_of[hp.state_keys[i]] = i;
    }
    const int64_t base = (int64_t)pk.cvals.size();
    pk.cvals.insert(pk.cvals.end(), hp.values.begin(), hp.values.end());
    SYMHIP_CHECK(pk.cvals.size() < (size_t)INT32_MAX, "batch: storage too large");
    auto off = [&](int32_t key) { return (int32_t)(base + hp.storage_offset[key]); };
    auto constant = [&](int32_t key) {
      SYMHIP_CHECK(pos_of[key] < 0, "batch: factor constants must not be optimized");
      return off(key);
    };
    std::vector<std::vector<int32_t>> matches(n);
    std::vector<int32_t> odo(3 * (size_t)n, -1);
    for (int32_t f = 0; f < hp.n_factors; ++f) {
      const int32_t* a = hp.fargs.data() + hp.fargs_ptr[f];
      if (hp.ftype[f] == SYMHIP_FACTOR_MATCHING) {
        const int32_t i = pos_of[a[0]];
        SYMHIP_CHECK(i >= 0, "batch: matching factor on a constant pose");
        matches[i].insert(matches[i].end(), {constant(a[1]), constant(a[2]), constant(a[3])});
      } else if (hp.ftype[f] == SYMHIP_FACTOR_ODOMETRY) {
        const int32_t i = pos_of[a[0]], j = pos_of[a[1]];
        SYMHIP_CHECK(i >= 0 && j == i + 1,
                     "batch: odometry factors must join consecutive optimized poses (a, a + 1)");
        SYMHIP_CHECK(odo[3 * i] < 0, "batch: two odometry factors leave the same pose");
        odo[3 * i] = constant(a[2]);
        odo[3 * i + 1] = constant(a[3]);
        odo[3 * i + 2] = constant(a[4]);
      } else {
        throw Error("batch: only matching and odometry factors are supported");
      }
    }
    for (int32_t i = 0; i < n; ++i) {
      pk.pose_soff.push_back(off(hp.state_keys[i]));
      pk.match_args.insert(pk.match_args.end(), matches[i].begin(), matches[i].end());
      pk.match_ptr.push_back((int32_t)(pk.match_args.size() / 3));
      pk.odo_args.insert(pk.odo_args.end(), odo.begin() + 3 * i, odo.begin() + 3 * i + 3);
    }
    pk.pose_begin.push_back(pk.pose_begin.back() + n);
  }
  return pk;
}

BatchLocalization::BatchLocalization(const symhip_problem_desc* descs, int32_t n_problems,
                                     const symhip_optimizer_params& params, bool compute_f32,
                                     double epsilon)
    : n_problems_(n_problems), p_(params), f32_(compute_f32), eps_(epsilon) {
  PackedBatch pk = pack_batch(descs, n_problems, params);
  std::vector<int32_t>& pose_begin = pk.pose_begin;
  std::vector<double>& cvals = pk.cvals;
  total_poses_ = pose_begin.back();
  for (int32_t i = 0; i < n_problems; ++i)
    max_poses_ = std::max(max_poses_, pose_begin[i + 1] - pose_begin[i]);
  cvals_host_size_ = cvals.size();
  HIP_OK(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
  HIP_OK(hipEventCreate(&ev0_));
  HIP_OK(hipEventCreate(&ev1_));
  pose_begin_.upload(pose_begin, stream_);
  pose_soff_.upload(pk.pose_soff, stream_);
  match_ptr_.upload(pk.match_ptr, stream_);
  match_args_.upload(pk.match_args.empty() ? std::vector<int32_t>{0} : pk.match_args, stream_);
  odo_args_.upload(pk.odo_args, stream_);
  cvals_.upload(cvals, stream_);
  vout_.upload(cvals, stream_);
  vals_.resize((size_t)3 * total_poses_ * 7);
  lin_.resize((size_t)3 * total_poses_ * kLin);
  maxd_.resize((size_t)total_poses_ * 6);
  recs_.resize((size_t)n_problems_ * (p_.iterations + 1));
  stats_.resize(n_problems_);
  ticks_.resize(2 * (size_t)n_problems_);
  {
    std::vector<int32_t> order(n_problems_);
    for (int32_t i = 0; i < n_problems_; ++i) order[i] = i;
    std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) {
      return pose_begin[a + 1] - pose_begin[a] > pose_begin[b + 1] - pose_begin[b];
    });
    order_.upload(order, stream_);
  }
  HIP_OK(hipStreamSynchronize(stream_));
  build_graph(config_);
}

BatchLocalization::~BatchLocalization() {
  for (auto& g : graphs_)
    if (g) (void)hipGraphExecDestroy(g);
  if (ev0_) (void)hipEventDestroy(ev0_);
  if (ev1_) (void)hipEventDestroy(ev1_);
  if (stream_) (void)hipStreamDestroy(stream_);
}

// Launch configuration c: bit 0 = two wavefronts per SIMD (else one), bit 1 = problems with
// the most poses first (else in the given order).
void BatchLocalization::build_graph(int c) {
  if (graphs_[c]) return;
  BatchView v{total_poses_,      pose_begin_.get(), pose_soff_.get(), match_ptr_.get(),
              match_args_.get(), odo_args_.get(),   cvals_.get(),     vals_.get(),
              lin_.get(),        maxd_.get(),       vout_.get(),      recs_.get(),
              p_.iterations + 1, stats_.get(),      ticks_.get(),
              (c & 2) ? order_.get() : nullptr};
  hipGraph_t graph;
  HIP_OK(hipStreamBeginCapture(stream_, hipStreamCaptureModeThreadLocal));
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(n_problems_), dim3(64), rec_bytes(max_poses_), stream_, v, p_,
                       eps_);
  };
  if (f32_) {
    if (c & 1) launch(batch_lm_kernel<float, 2>); else launch(batch_lm_kernel<float, 1>);
  } else {
    if (c & 1) launch(batch_lm_kernel<double, 2>); else launch(batch_lm_kernel<double, 1>);
  }
  HIP_OK(hipStreamEndCapture(stream_, &graph));
  HIP_OK(hipGraphInstantiate(&graphs_[c], graph, nullptr, nullptr, 0));
  HIP_OK(hipGraphDestroy(graph));
}

// The autotuner: every configuration solves the batch `reps` times (the solves are complete and
// give the same results: the configurations change occupancy and order, not the arithmetic) and
// the one with the shortest launch is kept for later solves.
void BatchLocalization::tune(int reps, double* config_ms) {
  SYMHIP_CHECK(reps >= 1, "batch: tune needs reps >= 1");
  double best = 0;
  for (int c = 0; c < kConfigs; ++c) {
    build_graph(c);
    double ms = 0;
    for (int r = 0; r < reps; ++r) {
      HIP_OK(hipEventRecord(ev0_, stream_));
      HIP_OK(hipGraphLaunch(graphs_[c], stream_));
      HIP_OK(hipEventRecord(ev1_, stream_));
      HIP_OK(hipStreamSynchronize(stream_));
      float t = 0;
      HIP_OK(hipEventElapsedTime(&t, ev0_, ev1_));
      ms = r == 0 ? t : std::min<double>(ms, t);
    }
    if (config_ms) config_ms[c] = ms;
    if (c == 0 || ms < best) {
      best = ms;
      config_ = c;
    }
  }
}

void BatchLocalization::solve(double* values_out, symhip_optimization_stats* stats_out,
                              symhip_iteration_stats* iters_out, double* solve_ms,
                              double* total_ms) {
  HIP_OK(hipEventRecord(ev0_, stream_));
  HIP_OK(hipGraphLaunch(graphs_[config_], stream_));
  HIP_OK(hipEventRecord(ev1_, stream_));
  if (values_out) vout_.download(values_out, cvals_host_size_, stream_);
  if (stats_out) stats_.download(stats_out, n_problems_, stream_);
  if (iters_out) recs_.download(iters_out, recs_.size(), stream_);
  std::vector<int64_t> ticks;
  if (solve_ms) {
    ticks.resize(ticks_.size());
    ticks_.download(ticks.data(), ticks.size(), stream_);
  }
  HIP_OK(hipStreamSynchronize(stream_));
  if (total_ms) {
    float ms = 0;
    HIP_OK(hipEventElapsedTime(&ms, ev0_, ev1_));
    *total_ms = ms;
  }
  if (solve_ms) {
    int dev = 0, khz = 0;
    HIP_OK(hipGetDevice(&dev));
    HIP_OK(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
    SYMHIP_CHECK(khz > 0, "batch: wall clock rate unavailable");
    for (int32_t i = 0; i < n_problems_; ++i)
      solve_ms[i] = (double)(ticks[2 * i + 1] - ticks[2 * i]) / (double)khz;
  }
}

// ---------------------------------------------------------------------------------------------
// Allocation-free solve: the kernel's working state (three state blocks of poses and their
// linearizations, the running maximum of the diagonal and the per-problem clock stamps) lives in
// a file-scope device array instead of buffers allocated per batch. Every call on a device shares
// that device's array, so calls that overlap on one device race. Nothing in it has to start at
// zero: each launch writes every entry it later reads (state block 1 from the inputs, the
// linearizations before they are read, the maximum diagonal on its first damping).
namespace {

constexpr int64_t kPerPoseScratch = 3 * 7 + 3 * kLin + 6;  // state blocks, linearizations, max diag
constexpr int64_t kScratchDoubles =
    SYMHIP_BATCH_NOALLOC_MAX_POSES * kPerPoseScratch + 2 * SYMHIP_BATCH_NOALLOC_MAX_POSES;

static __device__ __align__(256) double scratch[kScratchDoubles];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// The address of the current device's copy of `scratch`, looked up once per device.
double* device_scratch() {
  int dev = 0;
  HIP_OK(hipGetDevice(&dev));
  SYMHIP_CHECK(dev >= 0 && dev < kMaxDevices, "batch: device index out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    HIP_OK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    SYMHIP_CHECK(p != nullptr, "batch: scratch symbol has no device address");
    g_scratch_ptr[dev] = p;
  }
  return static_cast<double*>(g_scratch_ptr[dev]);
}

__global__ void copy_storage_kernel(int64_t n, const double* __restrict__ src,
                                    double* __restrict__ dst) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

}  // namespace

void batch_solve_noalloc(const symhip_batch_tables& t, const symhip_optimizer_params& p,
                         int32_t precision, double epsilon, double* values_out,
                         symhip_optimization_stats* stats_out, symhip_iteration_stats* iters_out,
                         hipStream_t stream) {
  SYMHIP_CHECK(t.n_problems > 0 && t.total_poses >= t.n_problems && t.storage_size > 0,
               "batch_noalloc: empty or inconsistent tables");
  SYMHIP_CHECK(t.total_poses <= SYMHIP_BATCH_NOALLOC_MAX_POSES,
               "batch_noalloc: more poses than the scratch array holds "
               "(SYMHIP_BATCH_NOALLOC_MAX_POSES)");
  SYMHIP_CHECK(t.pose_begin && t.pose_soff && t.match_ptr && t.odo_args && t.values &&
                   values_out && stats_out,
               "batch_noalloc: null table or output pointer");
  SYMHIP_CHECK(p.iterations > 0, "batch: iterations must be positive");
  SYMHIP_CHECK(!p.enable_bold_updates, "batch: bold updates are not supported");
  SYMHIP_CHECK(precision == SYMHIP_PRECISION_F64 || precision == SYMHIP_PRECISION_F32_JAC,
               "batch_noalloc: unknown precision");
  const int64_t TP = t.total_poses;
  double* base = device_scratch();
  double* vals = base;
  double* lin = vals + 3 * TP * 7;
  double* maxd = lin + 3 * TP * kLin;
  int64_t* ticks = reinterpret_cast<int64_t*>(maxd + TP * 6);
  // the output storage starts as the inputs; the kernel writes each problem's best poses into it
  hipLaunchKernelGGL(copy_storage_kernel, dim3((unsigned)((t.storage_size + 255) / 256)),
                     dim3(256), 0, stream, t.storage_size, t.values, values_out);
  BatchView v{TP,          t.pose_begin, t.pose_soff, t.match_ptr,        t.match_args,
              t.odo_args,  t.values,     vals,        lin,                maxd,
              values_out,  iters_out,    p.iterations + 1, stats_out,     ticks, nullptr};
  if (precision == SYMHIP_PRECISION_F32_JAC)
    hipLaunchKernelGGL((batch_lm_kernel<float, 1>), dim3(t.n_problems), dim3(64),
                       rec_bytes(kMaxPoses), stream, v, p, epsilon);
  else
    hipLaunchKernelGGL((batch_lm_kernel<double, 1>), dim3(t.n_problems), dim3(64),
                       rec_bytes(kMaxPoses), stream, v, p, epsilon);
  HIP_OK(hipGetLastError());
}

}  // namespace symhip
