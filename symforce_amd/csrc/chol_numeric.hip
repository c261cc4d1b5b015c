// Device numeric supernodal LDL^T: assembly, per-level fused diagonal-block factorization + panel
// triangular solve, right-looking update (SYRK-like) scattered into ancestor panels, and the
// triangular solves. FP64, except the trailing updates of the mixed-precision form (FP32 matrix
// cores, set_f32_updates).
//
// The work per supernode is small (panels are at most 64 columns wide), so every kernel is
// latency-bound: the kernels are written to avoid data-dependent branches (16 elimination steps
// are unrolled over panels padded to 64 columns, the padding being an identity block) and chains of
// dependent global loads (each supernode's metadata is one descriptor, scatter targets are
// precomputed per below-row).
#include <algorithm>

#include "./chol_numeric.h"
#include "./dpp.h"
#include "./util.h"

namespace symhip {

namespace {

constexpr int kMaxCols = 64;  // supernode width cap (panels padded to this width)
// Update tile (rows). 32-row tiles on every level, with shared memory sized for them (four
// blocks per CU at 33 KB, seven with the columns staged in two halves): a level's update time is the latency of its slowest tiles, and a 64-row tile's
// product (K = 64 on the FP64 matrix cores) and 4096-entry scatter take ~15 us where four 32-row
// tiles run side by side in ~6 (measured: 1000-camera system 464 -> 388 us of updates per
// factorization, 100 000-node pose graph 460 -> 205 us).
constexpr int kTile = 32;
constexpr int kCus = 256;  // compute units of an MI355X (block-count thresholds of the launches)

// l11_off: the factored diagonal block L11 (n x n, column-major, strictly lower part used) is
// kept apart from the panel, so the row-chunk blocks of one supernode, which all read the
// unfactored A11 from the panel, never see it half overwritten.
struct SnDesc {
  int64_t panel_off, l11_off;
  int32_t ncols, ld, col_begin, rows_off;
};

// One task of a level launch: its supernode's descriptor together with the task's own indices,
// fetched in one scalar-load round trip (an index list followed by a descriptor lookup costs two
// dependent round trips at the head of every latency-bound launch).
struct SnTask {
  SnDesc d;
  int32_t s, a, b, pad;  // supernode; chunk or tile row; tile column
};

// Assembly of A + diag(damping) (damping null: of A) into the panels. The matrix's map holds the
// panel place of every entry off the diagonal, ~j for column j's diagonal entry, which takes the
// damping, and behind the nnz entries the diagonal's places by column.
//
// Panels of up to kListPanel entries: by a list of what each panel entry is assembled from (src,
// built on the device: q >= 0 is entry q of the matrix, -2 - j the diagonal entry of column j, at
// diag[j], kPanelFill neither), every entry written once, in one launch. Larger ones: zeroed, then
// the matrix scattered into them. The list is read for every panel entry, four fifths of them
// fill-in, and its dependent loads keep it at 2.9 TB/s; the second launch costs ~3 us. From
// assembly to factorization on pose graphs, list against scatter: panels of 0.85 M entries 7.6
// against 11.0 us, 3.3 M 16.4 / 19.5, 6.6 M 26.9 / 26.7, 13.3 M 51.8 / 37.0, 33 M (100 000 nodes)
// 137 / 94 (of which 44 zero 266 MB), where the list also held 133 MB against the map's 50.
constexpr int64_t kListPanel = 6 << 20;
constexpr int32_t kPanelFill = -1;
__global__ void panel_fill_kernel(int64_t size, int32_t* __restrict__ src) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < size;
       i += (int64_t)gridDim.x * blockDim.x)
    src[i] = kPanelFill;
}
__global__ void panel_list_kernel(int64_t nnz, const int64_t* __restrict__ map,
                                  int32_t* __restrict__ src) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= nnz) return;
  const int64_t p = map[i];
  if (p >= 0) src[p] = (int32_t)i;
  else src[map[nnz + ~p]] = (int32_t)(-2 - ~p);
}

__global__ void __launch_bounds__(256) assemble_list_kernel(int64_t size,
                                                            const int32_t* __restrict__ src,
                                                            const int32_t* __restrict__ diag,
                                                            const double* __restrict__ vals,
                                                            const double* __restrict__ damping,
                                                            double* __restrict__ panel) {
  const int64_t i = 2 * (blockIdx.x * (int64_t)256 + threadIdx.x);
  if (i >= size) return;
  auto value = [&](int32_t c) __attribute__((always_inline)) {
    if (c >= 0) return vals[c];
    if (c == kPanelFill) return 0.0;
    const int32_t j = -2 - c;
    const double v = vals[diag[j]];
    return damping ? v + damping[j] : v;
  };
  if (i + 1 < size) {  // the buffers' own bases and an even i: aligned pairs
    const int2 c = *reinterpret_cast<const int2*>(src + i);
    *reinterpret_cast<double2*>(panel + i) = make_double2(value(c.x), value(c.y));
  } else {
    panel[i] = value(src[i]);
  }
}

__global__ void __launch_bounds__(256) assemble_scatter_kernel(int64_t nnz,
                                                               const int64_t* __restrict__ map,
                                                               const double* __restrict__ vals,
                                                               const double* __restrict__ damping,
                                                               double* __restrict__ panel) {
  for (int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x; i < nnz; i += (int64_t)gridDim.x * 256) {
    int64_t p = map[i];
    double v = vals[i];
    if (p < 0) {
      if (damping) v += damping[~p];
      p = map[nnz + ~p];
    }
    panel[p] = v;
  }
}

// Diagonal task (s, chunk): one 512-thread block eliminates the 64 x 64 diagonal block of
// supernode s together with the chunk's 64 below rows and, with kFwd, the right-hand side as one
// more row, in a right-looking sweep of 16-column panels (the diagonal block is factored
// redundantly by every chunk of s; chunk 0 writes L11 to l11 and D), leaving L21 = A21 L11^-T D^-1
// for its rows, written back into the panel in place.
//
// The working matrix (rows 0..63 the diagonal block padded with identity, rows 64..127 the chunk's
// below rows, row 128 the right-hand side) is in LDS, Lc[column][row]; its columns past the
// current panel live in matrix-core accumulators: wave w holds rows 16w .. 16w + 15 as 16 x 16
// tiles. Per panel:
//  1. two wavefronts eliminate its 16 columns with a row per lane and no barrier inside
//     (panel_columns): X the diagonal block's rows and the right-hand side, Y the below rows, each
//     with its own copy of the pivot rows. The other waves meanwhile apply the previous panel to
//     their later tiles;
//  2. every wave applies A(i, j) -= sum_u L(i, u) w(j, u) (w = L D) to its tile of the next panel's
//     columns with four v_mfma_f64_16x16x4f64, operands read from Lc and Wt, and puts the tile
//     into Lc; the operands of its later tiles are fetched for step 1.
// X and Y are waves whose own tiles are finished: the panel's pivot rows' and those before them.
// Panels past the supernode's last column are skipped (the padding stays the identity, which its
// elimination would not change).
//
// Bound by latency: with one task per CU a launch is 5.7 k cycles of descriptor and staging loads,
// four panels (2.7 k each, the vector pipe full with the broadcasts and multiply-adds of 16 columns
// on two rows a lane; the first one 2 k more, its code being fetched), three exchanges (1.3 k) and
// 4.7 k for the right-hand side's products and the stores. Before, 4-column steps with two barriers
// each (a pivot block formed by every row's owner, 16 LDS round trips and rank-4 products): per
// launch 17.7 -> 15.8 us on the 1000-camera system, 16.8 -> 14.8 at 137 cameras, 38 -> 33 on the
// 100 000-node pose graph (8 006 leaf tasks, two per CU). Leaving a panel early after 4, 8 or 12
// columns spilled its registers; the pivot rows' entries through LDS or scalar lane reads were
// slower (see panel_columns).
constexpr int kDiagThreads = 512;
constexpr int kPanel = 16;                 // columns per panel
constexpr int kDiagRows = 2 * kMaxCols;    // diagonal block + one chunk of below rows
constexpr int kRhsRow = kDiagRows;         // the right-hand side's row
// LDS: two spare rows keep column starts off the same banks (and hold the right-hand side); two
// blocks fit a CU (75.5 KB each)
constexpr int kLcLd = kDiagRows + 2;       // Lc[col][row]
constexpr int kWtLd = kMaxCols + 2;        // Wt[u][row]: w of the panel's columns
constexpr int kWtRhs = kMaxCols;           // .. and of the right-hand side's row
constexpr int kDiagSmem = kMaxCols * kLcLd + kPanel * kWtLd + kMaxCols;

// Value of v in lane k (k wave-uniform), through two scalar lane reads: a short dependency for
// the triangular recurrences (an LDS-based shuffle costs a full LDS round trip per step).
__device__ __forceinline__ double lane_value(double v, int k) {
  const int2 u = __builtin_bit_cast(int2, v);
  return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_readlane(u.x, k),
                                              __builtin_amdgcn_readlane(u.y, k)));
}

template <int K, int J>
__device__ __forceinline__ void panel_updates(double (&s0)[kPanel], double (&s1)[kPanel], double w,
                                              double l0, double l1) {
  if constexpr (J < kPanel) {
    const double b = row_bcast<J>(w);
    s0[J] = fma(-l0, b, s0[J]);
    s1[J] = fma(-l1, b, s1[J]);
    panel_updates<K, J + 1>(s0, s1, w, l0, l1);
  }
}

// Columns K.. of a panel: s0 holds the pivot rows (row l % 16 in lane l, four copies), s1 a row per
// lane. Column K: d = its pivot, l = own entry / d, and each later column j loses l w_j, w_j the
// pivot row j's entry, which row_bcast brings from the lane's own row of 16 (a broadcast and two
// multiply-adds, ~17 cycles; by scalar lane reads, or through LDS, the panel took 3.0-4.4 k cycles
// against 2.8). s0 and s1 end as L, and every lane's s1 entry goes to put[K * kLcLd] as it is
// formed; with kX its w goes to wput[K * kWtLd] too and pivot row r's lanes keep their d in dg.
template <bool kX, int K = 0>
__device__ __forceinline__ void panel_columns(double (&s0)[kPanel], double (&s1)[kPanel],
                                              double* put, double* wput, int lr, double& dg) {
  if constexpr (K < kPanel) {
    const double w = s0[K], w1 = s1[K];
    const double dinv = refined_rcp(row_bcast<K>(w));
    if (kX) wput[K * kWtLd] = w1;
    const double l0 = w * dinv, l1 = w1 * dinv;
    panel_updates<K, K + 1>(s0, s1, w, l0, l1);
    put[K * kLcLd] = l1;
    if (kX) {
      dg = lr == K ? w : dg;
      s0[K] = l0;
    }
    // a column's instructions fill the vector pipe by themselves; mixing columns only costs registers
    __builtin_amdgcn_sched_barrier(0);
    panel_columns<kX, K + 1>(s0, s1, put, wput, lr, dg);
  }
}

// Forward solve fused into the diagonal task (kFwd): with y = P b plus the updates of every
// descendant (earlier levels), the right-hand side's row leaves the sweep as w = L11^-1 y_own,
// chunk 0 writes it to yout, and the chunk's below rows get y(row) -= L21(row, :) y_own atomically
// (siblings share ancestors). The same work as a separate forward launch per level, without the
// launch.
template <bool kFwd>
__device__ __forceinline__ void diag_body(const SnTask& tk, double* __restrict__ panel,
                                          double* __restrict__ l11,
                                          double* __restrict__ D, const int32_t* __restrict__ rows,
                                          double* __restrict__ y, double* __restrict__ yout,
                                          double* smem) {
  typedef double d4 __attribute__((ext_vector_type(4)));
  auto Lc = reinterpret_cast<double (*)[kLcLd]>(smem);
  auto Wt = reinterpret_cast<double (*)[kWtLd]>(smem + kMaxCols * kLcLd);
  double* zs = smem + kMaxCols * kLcLd + kPanel * kWtLd;  // the solved right-hand side
  const SnDesc sd = tk.d;
  const int chunk = tk.a;
  const int n = sd.ncols, ld = sd.ld, mb = ld - n;
  double* P = panel + sd.panel_off;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  // forward-solve operands, fetched up front (clamped indices, selected at use)
  double y_in = 0.0;
  int32_t y_row = 0;
  if (kFwd && wave == 0) {
    y_in = y[sd.col_begin + min(lane, n - 1)];
    y_row = rows[sd.rows_off + (mb > 0 ? n + min(chunk * kMaxCols + lane, mb - 1) : 0)];
  }
  // Stage the working matrix in Lc with coalesced loads (consecutive threads take consecutive
  // rows of one column): one unconditional load per element from a clamped valid address, then
  // a select (a guarded load is compiled as a branch that waits for each load in turn).
  constexpr int kPer = kDiagRows * kMaxCols / kDiagThreads;
  double v[kPer];
#pragma unroll
  for (int q = 0; q < kPer; ++q) {  // all loads first
    const int idx = tid + kDiagThreads * q;
    const int i = idx & (kDiagRows - 1), j = idx / kDiagRows;
    const int jc = min(j, n - 1), ic = min(i, n - 1);
    const int r = chunk * kMaxCols + i - kMaxCols;
    const int row = (i >= kMaxCols) & (mb > 0) ? n + min(r, mb - 1) : ic;
    v[q] = P[(int64_t)jc * ld + row];
  }
#pragma unroll
  for (int q = 0; q < kPer; ++q) {
    const int idx = tid + kDiagThreads * q;
    const int i = idx & (kDiagRows - 1), j = idx / kDiagRows;
    const int r = chunk * kMaxCols + i - kMaxCols;
    const int below = i >= kMaxCols;
    // below rows: inside the chunk; diagonal block: lower triangle inside n x n, identity padding
    const int keep = (below & (r < mb) & (j < n)) | (!below & (i < n) & (j < n) & (i >= j));
    const double fill = (!below & (i == j)) ? 1.0 : 0.0;
    Lc[j][i] = keep ? v[q] : fill;
  }
  if (wave == 0) {
    Lc[lane][kRhsRow] = kFwd && lane < n ? y_in : 0.0;
    zs[lane] = 0.0;
  }
  __syncthreads();
  // acc[t] holds the tile of columns 16 (p + 1 + t) .. for the current panel p, in the
  // v_mfma_f64_16x16x4f64 layout: acc[t][r] = A(16w + lane / 16 + 4r, 16 (p + 1 + t) + lane % 16).
  // A tile above the diagonal block's diagonal is never read: waves 0..3 keep columns up to 16w.
  constexpr int kTiles = kMaxCols / kPanel - 1;
  d4 acc[kTiles] = {};
  auto load_tiles = [&] {
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        acc[t][r] = Lc[kPanel * (1 + t) + lr][16 * wave + lk + 4 * r];
  };
  if (wave >= 2) load_tiles();
  // operands of the later tiles, from one panel's step 2 to the next one's step 1
  double av[4], bv[kTiles - 1][4];
#pragma unroll
  for (int h = 0; h < 4; ++h) av[h] = bv[0][h] = bv[1][h] = 0.0;
  for (int k0 = 0;; k0 += kPanel) {
    const int p = k0 / kPanel;
    const int wx = p, wy = p == 0 ? 1 : p - 1;
    // The panel's own waves run at a higher priority than the tile waves on their SIMDs: they are
    // the block's critical path.
    if (wave == wx) {
      // lanes: rows 16 .. 63 of the diagonal block, then the right-hand side; rows up to the
      // panel's pivots are finished, eliminated along and stored to the spare row
      const int row = lane < kMaxCols - kPanel ? kPanel + lane : kRhsRow;
      __builtin_amdgcn_s_setprio(2);
      double s0[kPanel], s1[kPanel], dg = 0.0;
#pragma unroll
      for (int u = 0; u < kPanel; ++u) {
        s0[u] = Lc[k0 + u][k0 + lr];
        s1[u] = Lc[k0 + u][row];
      }
      panel_columns<true>(s0, s1, &Lc[k0][row < k0 + kPanel ? kRhsRow + 1 : row],
                          &Wt[0][row == kRhsRow ? kWtRhs : row], lr, dg);
      __builtin_amdgcn_s_setprio(0);
      __syncthreads();
      if (lane < kPanel) {
        // the pivot rows, which Y has read by now: L, D on the diagonal, zeros right of it
#pragma unroll
        for (int u = 0; u < kPanel; ++u)
          Lc[k0 + u][k0 + lane] = u < lane ? s0[u] : (u == lane ? dg : 0.0);
        if (kFwd) zs[k0 + lane] = Wt[lane][kWtRhs];
      }
#pragma unroll
      for (int t = 0; t < kTiles; ++t) acc[t] = d4{};  // finished: not live across the panel
    } else if (wave == wy) {
      __builtin_amdgcn_s_setprio(2);
      double s0[kPanel], s1[kPanel], dg = 0.0;
#pragma unroll
      for (int u = 0; u < kPanel; ++u) {
        s0[u] = Lc[k0 + u][k0 + lr];
        s1[u] = Lc[k0 + u][kMaxCols + lane];
      }
      panel_columns<false>(s0, s1, &Lc[k0][kMaxCols + lane], nullptr, lr, dg);
      __builtin_amdgcn_s_setprio(0);
      __syncthreads();
#pragma unroll
      for (int t = 0; t < kTiles; ++t) acc[t] = d4{};
      if (p == 0) load_tiles();
    } else {
      if (k0 > 0) {
#pragma unroll
        for (int t = 1; t < kTiles; ++t) {
#pragma unroll
          for (int h = 0; h < 4; ++h)
            acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[h], bv[t - 1][h], acc[t], 0, 0, 0);
          acc[t - 1] = acc[t];
        }
      }
      __syncthreads();
    }
    const int kn = k0 + kPanel;  // first column still to be eliminated
    if (kn >= n) break;          // uniform
    if (wave > p) {
      // A(i, j) -= sum_u L(i, k0 + u) w(j, u): lane l feeds A(l % 16, l / 16) =
      // -L(16w + l % 16, k0 + 4h + l / 16) and B(l / 16, l % 16) = w(16c + l % 16, 4h + l / 16)
      double bn[4];
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        av[h] = -Lc[k0 + 4 * h + lk][16 * wave + lr];
        bn[h] = Wt[4 * h + lk][kn + lr];
      }
#pragma unroll
      for (int h = 0; h < 4; ++h)
        acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[h], bn[h], acc[0], 0, 0, 0);
#pragma unroll
      for (int t = 1; t < kTiles; ++t)
#pragma unroll
        for (int h = 0; h < 4; ++h)  // past the last tile: clamped, its accumulator is not used
          bv[t - 1][h] = Wt[4 * h + lk][min(kn + kPanel * t, kMaxCols - kPanel) + lr];
#pragma unroll
      for (int r = 0; r < 4; ++r) Lc[kn + lr][16 * wave + lk + 4 * r] = acc[0][r];
    } else {
#pragma unroll
      for (int h = 0; h < 4; ++h) av[h] = bv[0][h] = bv[1][h] = 0.0;
    }
    if (kFwd && wave == (p == 0 ? 0 : p - 1)) {  // a wave without tiles, X's stores aside
      // the right-hand side's later columns: y_j -= sum_u l_y w_j
      const int j = kn + lane;
      if (j < kMaxCols) {
        double t = Lc[j][kRhsRow];
#pragma unroll
        for (int u = 0; u < kPanel; ++u) t = fma(-Lc[k0 + u][kRhsRow], Wt[u][j], t);
        Lc[j][kRhsRow] = t;
      }
    }
    __syncthreads();
  }
  __syncthreads();
  if (kFwd) {
    // L21 y_own, 16 columns by each of four waves, then added up by the first
    auto part = reinterpret_cast<double (*)[kMaxCols]>(&Wt[0][0]);
    if (wave < 4) {
      double t = 0.0;
#pragma unroll
      for (int u = 0; u < kPanel; ++u) {
        const int k = kPanel * wave + u;
        t = fma(Lc[k][kMaxCols + lane], zs[k], t);
      }
      part[wave][lane] = t;
    }
    __syncthreads();
    if (wave == 0) {
      if (chunk == 0 && lane < n) yout[sd.col_begin + lane] = zs[lane];
      if (chunk * kMaxCols + lane < mb)
        unsafeAtomicAdd(&y[y_row],
                        -((part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane])));
    }
  }
  // Write back with coalesced stores: L11 (strict lower, column-major n x n) and D from chunk 0
  // (the even waves), the chunk's L21 rows into the panel (the odd ones); a wave takes every fourth
  // column. The thread index passes through an empty asm so the compiler recomputes these
  // addresses here instead of holding the load phase's across the sweep.
  int tid_w = tid;
  asm volatile("" : "+v"(tid_w));
  const int i = tid_w & (kDiagRows - 1);
  const int j0 = __builtin_amdgcn_readfirstlane(tid_w / kDiagRows);
  constexpr int kStride = kDiagThreads / kDiagRows;
  // (four columns a turn: the code is fetched for the first time here, and a fully unrolled copy of
  // all sixteen is slower for it)
  if (wave & 1) {
    const int r = chunk * kMaxCols + i - kMaxCols;
    double* dst = P + (int64_t)j0 * ld + n + r;
    const int64_t step = (int64_t)kStride * ld;
    if (r < mb) {
#pragma unroll 4
      for (int j = j0; j < n; j += kStride, dst += step) *dst = Lc[j][i];
    }
  } else if (chunk == 0) {
    double* dst = l11 + sd.l11_off + (int64_t)j0 * n + i;
    const int64_t step = (int64_t)kStride * n;
    if (i < n) {
#pragma unroll 4
      for (int j = j0; j < n; j += kStride, dst += step)
        if (i > j) *dst = Lc[j][i];
      if ((i & (kStride - 1)) == j0) D[sd.col_begin + i] = Lc[i][i];
    }
  }
}

template <bool kFwd>
__global__ void __launch_bounds__(kDiagThreads) __attribute__((amdgpu_waves_per_eu(4)))
diag_trsm_kernel(
    const SnTask* __restrict__ tasks, double* __restrict__ panel, double* __restrict__ l11,
    double* __restrict__ D, const int32_t* __restrict__ rows, double* __restrict__ y,
    double* __restrict__ yout) {
  __shared__ __attribute__((aligned(16))) double smem[kDiagSmem];
  diag_body<kFwd>(tasks[blockIdx.x], panel, l11, D, rows, y, yout, smem);
}

// Update task (s, ti, tj), one 256-thread block: U = L21 D L21^T tile (ti, tj) of KT x KT,
// scattered as -U into ancestor panels. For below-row j of the supernode, scat_col[j] is the
// panel offset of its column in the target supernode and scat_rel[j] + i indexes upd_rel for the
// target row position of below-row i >= j (i < mb). The launches use KT = kTile = 32 (the body
// also takes 64-row tiles).
//
// T = float is the mixed-precision form of the update: both row tiles are rounded to FP32 (the
// D scaling applied first, in FP64), the product runs on the FP32 matrix cores
// (v_mfma_f32_16x16x4f32, FP32 accumulation) and is scattered as FP64 like the FP64 form; the
// diagonal blocks and panels stay FP64 (diag_trsm_kernel), and the caller refines its solves
// against the FP64 matrix.
template <int KT, typename T>
__device__ __forceinline__ void update_body(const SnTask& tk, double* __restrict__ panel,
                                            const double* __restrict__ D,
                                            const int64_t* __restrict__ scat_col,
                                            const int32_t* __restrict__ scat_rel,
                                            const int32_t* __restrict__ upd_rel, double* smem) {
  static_assert(KT == 64 || KT == 32, "update tiles are 64 or 32 rows");
  constexpr bool kF64 = sizeof(T) == 8;
  constexpr int kKh = kMaxCols / 2;  // columns staged per half
  auto As = reinterpret_cast<T (*)[KT + 1]>(smem);
  auto Bs = reinterpret_cast<T (*)[KT + 1]>(reinterpret_cast<T*>(smem) + kKh * (KT + 1));
  const SnDesc sd = tk.d;
  const int ti = tk.a, tj = tk.b;
  const int n = sd.ncols, ld = sd.ld, mb = ld - n;
  const double* P = panel + sd.panel_off;
  const double* Ds = D + sd.col_begin;
  // Stage both row tiles, half the columns at a time (unconditional loads from clamped
  // addresses; an update item exists only when mb > 0). Two halves take half the shared memory
  // (17 KB: seven blocks per CU instead of four), and a supernode of at most 32 columns skips the
  // second, all-padding half (the 100 000-node pose graph's updates 206 -> 192 us per
  // factorization; the 1000-camera system's 63-column supernodes unchanged).
  auto stage = [&](int h) {
#pragma unroll
    for (int t = 0; t < kKh * KT / 256; ++t) {  // blockDim.x == 256
      const int idx = threadIdx.x + 256 * t;
      const int k = idx / KT, r = idx % KT;
      const int kk = kKh * h + k;
      const int ri = ti * KT + r, rj = tj * KT + r;
      const int kc = min(kk, n - 1);
      const double va = P[(int64_t)kc * ld + n + min(ri, mb - 1)];
      const double vb = P[(int64_t)kc * ld + n + min(rj, mb - 1)] * Ds[kc];
      As[k][r] = (kk < n && ri < mb) ? T(va) : T(0);
      Bs[k][r] = (kk < n && rj < mb) ? T(vb) : T(0);
    }
  };
  stage(0);
  // The product on the FP64 matrix cores, in 16 x 16 output blocks, K = 64 in two halves of 8
  // steps of v_mfma_f64_16x16x4f64: a 64-row tile gives wave w row block w and all four column blocks, a
  // 32-row tile gives it row block w / 2 and column block w % 2. Lane l feeds
  // A(i = l % 16, k = l / 16) = As[k][16 rb + i] and B(k, j = l % 16) = Bs[k][16 c + j] and holds
  // D(l / 16 + 4 r, l % 16) of block c in accumulator register r (FP64) or D(4 (l / 16) + r,
  // l % 16) (FP32).
  typedef T d4 __attribute__((ext_vector_type(4)));
  constexpr int NBW = KT == 64 ? 4 : 1;  // output blocks per wave
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: scalar metadata
  const int lr = lane & 15, lk = lane >> 4;
  const int rb = KT == 64 ? wave : wave >> 1, c0 = KT == 64 ? 0 : wave & 1;
  // Scatter targets, fetched while the tiles load and before the product loop (the row
  // positions depend on the metadata: two dependent loads, off the critical path here). The
  // scatter runs column by column: wave w takes tile columns w, w + 4, .. and each atomic
  // instruction covers KT consecutive rows of 64 / KT columns (a few cache lines) instead of 16
  // columns x 4 rows. Row indices are clamped into the column's update segment (rows j ..
  // mb - 1); clamped entries are masked at the scatter.
  constexpr int kCpi = 64 / KT;             // columns per scatter instruction
  constexpr int kNq = KT / 4 / kCpi;        // scatter instructions per lane
  const int srow = lane % KT, ssub = lane / KT;
  int64_t cbase[kNq];
  int32_t rel[kNq];
  {
    const int i = ti * KT + srow;
#pragma unroll
    for (int q = 0; q < kNq; ++q) {
      const int j = min(tj * KT + wave + 4 * (kCpi * q + ssub), mb - 1);
      cbase[q] = scat_col[sd.rows_off + n + j];
      const int32_t rbase = scat_rel[sd.rows_off + n + j];
      rel[q] = upd_rel[rbase + min(max(i, j), mb - 1)];
    }
  }
  __syncthreads();
  d4 acc[NBW] = {};
  for (int h = 0; h < 2; ++h) {
    if (h == 1) {
      if (n <= kKh) break;  // uniform: the second half is all padding
      __syncthreads();
      stage(1);
      __syncthreads();
    }
#pragma unroll 4
    for (int k0 = 0; k0 < kKh; k0 += 4) {
      const T av = As[k0 + lk][16 * rb + lr];
      T bv[NBW];
#pragma unroll
      for (int c = 0; c < NBW; ++c) bv[c] = Bs[k0 + lk][16 * (c0 + c) + lr];
#pragma unroll
      for (int c = 0; c < NBW; ++c) {
        if constexpr (kF64)
          acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv[c], acc[c], 0, 0, 0);
        else
          acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, bv[c], acc[c], 0, 0, 0);
      }
    }
  }
  // transpose through LDS (the tiles' space, as FP64): Tr[column][row]
  __syncthreads();
  auto Tr = reinterpret_cast<double (*)[KT + 1]>(smem);
#pragma unroll
  for (int c = 0; c < NBW; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = kF64 ? lk + 4 * r : 4 * lk + r;
      Tr[16 * (c0 + c) + lr][16 * rb + row] = double(acc[c][r]);
    }
  __syncthreads();
  const int i = ti * KT + srow;
#pragma unroll
  for (int q = 0; q < kNq; ++q) {
    const int jl = wave + 4 * (kCpi * q + ssub), j = tj * KT + jl;
    const double v = Tr[jl][srow];
    if (j < mb && i < mb && i >= j) unsafeAtomicAdd(panel + cbase[q] + rel[q], -v);
  }
}

template <int KT, typename T>
__global__ void __launch_bounds__(256) update_kernel(const SnTask* __restrict__ tasks,
                                                     double* __restrict__ panel,
                                                     const double* __restrict__ D,
                                                     const int64_t* __restrict__ scat_col,
                                                     const int32_t* __restrict__ scat_rel,
                                                     const int32_t* __restrict__ upd_rel) {
  __shared__ double smem[kMaxCols * (KT + 1)];
  update_body<KT, T>(tasks[blockIdx.x], panel, D, scat_col, scat_rel, upd_rel, smem);
}

// An entry of the backward pass's result that no block has written yet: a NaN that is never stored
// as a result (final_value).
constexpr unsigned long long kPending = ~0ull;

// y = P b; also clears the backward pass's partial sums, results and ticket.
__global__ void permute_kernel(int32_t n, const int32_t* __restrict__ perm,
                               const double* __restrict__ b, double* __restrict__ y,
                               double* __restrict__ part, unsigned long long* __restrict__ ysol,
                               int32_t* __restrict__ ticket) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    y[perm[i]] = b[i];
    part[i] = 0.0;
    ysol[i] = kPending;
  }
  if (i == 0) *ticket = 0;
}
__global__ void unpermute_kernel(int32_t n, const int32_t* __restrict__ perm,
                                 const double* __restrict__ y, double sign,
                                 double* __restrict__ x) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = sign * y[perm[i]];
}

// Stages the strictly lower part of L11 (n x n column-major at Lc, padded with zeros; unit
// diagonal implied) into LDS: Ls[i][k].
__device__ __forceinline__ void stage_l11(const double* Lc, int n, double (*Ls)[kMaxCols + 1]) {
#pragma unroll
  for (int t = 0; t < kMaxCols * kMaxCols / 256; ++t) {  // blockDim.x == 256
    const int idx = threadIdx.x + 256 * t;
    const int i = idx % kMaxCols, k = idx / kMaxCols;
    const double v = Lc[(int64_t)min(k, n - 1) * n + min(i, n - 1)];  // clamped, then masked
    Ls[i][k] = (i < n && k < n && i > k) ? v : 0.0;
  }
}

// below-rows per solve block: a backward block sums them 64 at a time (chunks of 128 beat 256 and
// 512: more, shorter blocks per level); a forward block takes one per thread
constexpr int kSolveRows = 128;
static_assert(kSolveRows % 64 == 0 && kSolveRows <= 256, "solve chunk: whole waves, one block");

// Forward, block (s, chunk): y_own = L11^-1 y_own (one wavefront, lane r holds y_r, L11 from LDS;
// every chunk block of s solves redundantly, chunk 0 writes the result to yout) and, for the
// chunk's below-rows i, y(row i) -= L21(i, :) y_own with atomics into yacc (siblings at the same
// level share ancestors). A thread takes one below-row and all 64 (padded) columns; its 64 panel
// loads are issued before the triangular solve so they overlap it. Columns past n are clamped to
// column n - 1 and multiplied by ys = 0.
__global__ void __launch_bounds__(256) fwd_kernel(const SnTask* __restrict__ tasks,
                                                  const int32_t* __restrict__ rows,
                                                  const double* __restrict__ panel,
                                                  const double* __restrict__ l11,
                                                  double* __restrict__ yacc,
                                                  double* __restrict__ yout) {
  __shared__ double Ls[kMaxCols][kMaxCols + 1];
  __shared__ double ys[kMaxCols];
  const SnTask tk = tasks[blockIdx.x];
  const int chunk = tk.a;
  const SnDesc sd = tk.d;
  const int n = sd.ncols, ld = sd.ld, mb = ld - n;
  const double* P = panel + sd.panel_off;
  const int32_t* rw = rows + sd.rows_off + n;
  const int i = chunk * kSolveRows + threadIdx.x;
  double lrow[kMaxCols];
  {
    // clamped into the panel (the diagonal block when there are no below-rows)
    const int64_t r = mb > 0 ? n + min(i, mb - 1) : 0;
#pragma unroll
    for (int k = 0; k < kMaxCols; ++k) lrow[k] = P[(int64_t)min(k, n - 1) * ld + r];
  }
  stage_l11(l11 + sd.l11_off, n, Ls);
  double yi = 0;
  if (threadIdx.x < n) yi = yacc[sd.col_begin + threadIdx.x];
  __syncthreads();
  if (threadIdx.x < 64) {
    const int r = threadIdx.x;
#pragma unroll
    for (int k = 0; k < kMaxCols; ++k) yi -= Ls[r][k] * lane_value(yi, k);
    if (chunk == 0 && r < n) yout[sd.col_begin + r] = yi;
    ys[r] = r < n ? yi : 0.0;
  }
  __syncthreads();
  if (threadIdx.x < kSolveRows && i < mb) {  // a chunk may be narrower than the block
    double acc = 0;
#pragma unroll
    for (int k = 0; k < kMaxCols; ++k) acc += lrow[k] * ys[k];
    unsafeAtomicAdd(&yacc[rw[i]], -acc);
  }
}

// Backward, block (s, chunk): part(own) += L21(chunk rows, :)^T y(chunk rows) (wave w takes
// columns w, w + 4, ..., w + 60: 16 accumulators per lane, lanes over the rows, reduced across the
// wave), added atomically into part; the last chunk block of s to finish (a per-supernode arrival
// counter, reset by that block for the next solve) then forms y_own = L11^-T (D^-1 y_own - part)
// with one wavefront (the D^-1 of the solve folded in: own entries are read by their supernode's
// blocks only). part must be zero on entry (the permutation kernel clears it). A supernode of
// one chunk (at most kSolveRows below-rows: most of a pose graph's) skips part, the atomics and
// the arrival: its block's column sums are final and go through LDS.
//
// kLean (levels with more blocks than fit two to a CU, e.g. the thousands of small leaf
// supernodes of a pose graph): L11 is held in registers instead of LDS until the block knows it
// is the last, then written over the partials' space, so the block needs 33 KB of LDS instead of
// 66 KB and four blocks fit a CU instead of two (the 100 000-node pose graph's backward solve
// 0.43 -> 0.35 ms). On levels of a few blocks the extra barrier only adds latency.
template <bool kLean>
__global__ void __launch_bounds__(256) bwd_kernel(const SnTask* __restrict__ tasks,
                                                  const int32_t* __restrict__ rows,
                                                  const double* __restrict__ panel,
                                                  const double* __restrict__ l11,
                                                  const double* __restrict__ D,
                                                  double* __restrict__ yout,
                                                  double* __restrict__ part,
                                                  int32_t* __restrict__ counter) {
  // the waves' column partials and L11; with kLean, L11 takes the partials' space at the end
  constexpr int kRed = (kMaxCols / 4) * (64 + 1);
  constexpr int kLs = kMaxCols * (kMaxCols + 1);
  static_assert(4 * kRed >= kLs, "L11 fits the partials' space");
  __shared__ double buf[4 * kRed + (kLean ? 0 : kLs)];
  auto red_all = reinterpret_cast<double (*)[kRed]>(buf);
  auto Ls = reinterpret_cast<double (*)[kMaxCols + 1]>(kLean ? buf : buf + 4 * kRed);
  __shared__ double colsum[kMaxCols];  // a single-chunk supernode's column sums
  __shared__ int last;
  const SnTask tk = tasks[blockIdx.x];
  const int s = tk.s, chunk = tk.a;
  const SnDesc sd = tk.d;
  const int n = sd.ncols, ld = sd.ld, mb = ld - n;
  const int nchunks = max(1, (mb + kSolveRows - 1) / kSolveRows);
  const double* P = panel + sd.panel_off + n;
  const int32_t* rw = rows + sd.rows_off + n;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // Every block loads L11 and y_own up front: only the last block of s uses them, but this way
  // their loads overlap the partial sums instead of following the arrival counter (y_own is
  // written by no other block of this launch).
  constexpr int kL11 = kLean ? kMaxCols * kMaxCols / 256 : 1;  // blockDim.x == 256
  double l11v[kL11];
  if constexpr (kLean) {
    const double* Lc = l11 + sd.l11_off;
#pragma unroll
    for (int t = 0; t < kL11; ++t) {
      const int idx = threadIdx.x + 256 * t;
      const int i = idx % kMaxCols, k = idx / kMaxCols;
      const double v = Lc[(int64_t)min(k, n - 1) * n + min(i, n - 1)];  // clamped, then masked
      l11v[t] = (i < n && k < n && i > k) ? v : 0.0;
    }
  } else {
    stage_l11(l11 + sd.l11_off, n, Ls);
  }
  double yown = 0;
  if (threadIdx.x < n) yown = yout[sd.col_begin + threadIdx.x] / D[sd.col_begin + threadIdx.x];
  if (mb > 0) {
    constexpr int kPer = kMaxCols / 4;
    double acc[kPer] = {};
    int64_t coff[kPer];
#pragma unroll
    for (int c = 0; c < kPer; ++c) coff[c] = (int64_t)min(wave + 4 * c, n - 1) * ld;
#pragma unroll
    for (int t = 0; t < kSolveRows / 64; ++t) {
      const int i = chunk * kSolveRows + lane + 64 * t;
      const int ic = min(i, mb - 1);
      const double yl = yout[rw[ic]];
      const double yv = i < mb ? yl : 0.0;
#pragma unroll
      for (int c = 0; c < kPer; ++c) acc[c] += P[coff[c] + ic] * yv;
    }
    // Each wave's 16 column sums across its 64 lanes, through LDS: the partials go in as
    // red[c][lane], lane l then adds 16 of column l / 4's (quarter l % 4) and two quad shuffles
    // finish. (Six rounds of 64-lane shuffles for 16 values took longer than the loads.)
    auto red = reinterpret_cast<double (*)[64 + 1]>(&red_all[wave][0]);
#pragma unroll
    for (int c = 0; c < kPer; ++c) red[c][lane] = acc[c];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int c = lane >> 2, qtr = lane & 3;
    double v = 0;
#pragma unroll
    for (int t = 0; t < 16; ++t) v += red[c][16 * qtr + t];
    v += __shfl_xor(v, 1, 64);
    v += __shfl_xor(v, 2, 64);
    const int k = wave + 4 * c;
    if (qtr == 0 && k < n) {
      if (nchunks == 1) colsum[k] = v;  // the block holds every row: the sums are final
      else unsafeAtomicAdd(&part[sd.col_begin + k], v);
    }
  }
  if (nchunks == 1) {  // uniform: no other block of s, no arrival
    __syncthreads();
  } else {
    // Every wave waits for its own atomics into part before the block arrives: a workgroup
    // barrier does not wait for the memory operations of the other waves, and an agent fence
    // in the arriving thread would cover only its own wave (and write back and invalidate the
    // L2).
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0)
      last = __hip_atomic_fetch_add(&counter[s], 1, __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT) == nchunks - 1;
    __syncthreads();
    if (!__builtin_amdgcn_readfirstlane(last)) return;  // uniform across the block
  }
  if constexpr (kLean) {  // every wave is past its partials (the barriers above)
#pragma unroll
    for (int t = 0; t < kL11; ++t) {
      const int idx = threadIdx.x + 256 * t;
      Ls[idx % kMaxCols][idx / kMaxCols] = l11v[t];
    }
    __syncthreads();
  }
  // every chunk's sums are in part: read them at agent scope (past the per-XCD L2)
  if (threadIdx.x < 64) {
    const int r = threadIdx.x;
    double yi = 0;
    if (r < n) {
      if (nchunks == 1)
        yi = mb > 0 ? yown - colsum[r] : yown;
      else
        yi = yown - __hip_atomic_load(&part[sd.col_begin + r], __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll
    for (int k = kMaxCols - 1; k >= 0; --k) yi -= Ls[k][r] * lane_value(yi, k);
    if (r < n) yout[sd.col_begin + r] = yi;
    if (r == 0 && nchunks > 1) counter[s] = 0;
  }
}

__device__ __forceinline__ unsigned long long final_value(double v) {
  return v != v ? 0x7FF8000000000000ull : (unsigned long long)__double_as_longlong(v);
}
// Waits for a result entry; the entry itself is the signal, so it costs one round trip.
__device__ __forceinline__ double wait_value(const unsigned long long* p) {
  unsigned long long v;
  while ((v = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == kPending)
    __builtin_amdgcn_s_sleep(1);
  return __longlong_as_double((long long)v);
}

// Backward over all the narrow levels at the top of the tree in one launch. A block (s, chunk) does
// what bwd_kernel's does, but has its panel rows in registers and L11 in LDS before it waits for
// the results it needs, entry by entry in ysol (written and read at agent scope). Chunk 0, whose
// rows begin with the parent's columns, is the one that forms y_own; the other chunks' rows belong
// to farther ancestors, so their sums are normally in part before chunk 0's rows are final.
//
// A level is a chain of dependent steps: results' round trip, column sums, the triangular solve of
// 64 steps, the store. With a launch per level that chain also held the launch, the descriptor,
// the panel's and L11's loads and the arrival of every chunk: 7.3 us a level on the 1000-camera
// system's 38 levels, now 3.1 (an optimizer run of ten solves 23.2 -> 21.6 ms; 137 cameras 5.94 ->
// 5.35 ms; 2503-node pose graph 2.05 -> 1.89 ms).
//
// Every wait ends: a block's task is the ticket it draws when it starts, counted back from the last
// solve task (last): from the root level down and, a supernode's chunks being listed in their order,
// with chunk 0 last in each supernode. A block waits only for tasks drawn before its own, whose
// blocks have therefore started; the earliest unfinished one waits for none.
__global__ void __launch_bounds__(256) bwd_chain_kernel(
    const SnTask* __restrict__ last, const int32_t* __restrict__ rows,
    const double* __restrict__ panel, const double* __restrict__ l11, const double* __restrict__ D,
    double* __restrict__ yout, unsigned long long* ysol, double* part, int32_t* counter,
    int32_t* ticket) {
  constexpr int kPer = kMaxCols / 4, kHalves = kSolveRows / 64;
  __shared__ double Ls[kMaxCols][kMaxCols + 1];
  __shared__ double red_all[4][kPer][64 + 1];
  __shared__ double ys[kSolveRows], colsum[kMaxCols], others[kMaxCols];
  __shared__ int drawn;
  if (threadIdx.x == 0)
    drawn = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const int t = __builtin_amdgcn_readfirstlane(drawn);
  if (t >= (int)gridDim.x) return;  // uniform; not after a permute_kernel, which resets the ticket
  const SnTask tk = last[-t];
  const int s = tk.s, chunk = tk.a;
  const SnDesc sd = tk.d;
  const int n = sd.ncols, ld = sd.ld, mb = ld - n;
  const int nchunks = max(1, (mb + kSolveRows - 1) / kSolveRows);
  const double* P = panel + sd.panel_off;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double l[kHalves][kPer];
#pragma unroll
  for (int h = 0; h < kHalves; ++h) {
    // clamped into the panel (the diagonal block when there are no below-rows)
    const int64_t r = mb > 0 ? n + min(chunk * kSolveRows + lane + 64 * h, mb - 1) : 0;
#pragma unroll
    for (int c = 0; c < kPer; ++c) l[h][c] = P[(int64_t)min(wave + 4 * c, n - 1) * ld + r];
  }
  double yown = 0;
  if (chunk == 0) {
    stage_l11(l11 + sd.l11_off, n, Ls);
    if (threadIdx.x < n) yown = yout[sd.col_begin + threadIdx.x] / D[sd.col_begin + threadIdx.x];
    if (threadIdx.x < kMaxCols) colsum[threadIdx.x] = others[threadIdx.x] = 0.0;
  }
  if (mb > 0) {
    const int i = chunk * kSolveRows + threadIdx.x;
    const int32_t row = rows[sd.rows_off + n + min(i, mb - 1)];
    __syncthreads();
    if (threadIdx.x < kSolveRows) {
      const double y = wait_value(ysol + row);
      ys[threadIdx.x] = i < mb ? y : 0.0;
    } else if (wave == 3 && chunk == 0 && nchunks > 1) {
      // the other chunks' sums: read at agent scope (past the per-XCD L2) once all have arrived
      while (__hip_atomic_load(&counter[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) !=
             nchunks - 1)
        __builtin_amdgcn_s_sleep(1);
      asm volatile("" ::: "memory");  // the sums are not read before
      if (lane < n)
        others[lane] = __hip_atomic_load(&part[sd.col_begin + lane], __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    auto red = red_all[wave];
#pragma unroll
    for (int c = 0; c < kPer; ++c) {
      double acc = 0;
#pragma unroll
      for (int h = 0; h < kHalves; ++h) acc += l[h][c] * ys[lane + 64 * h];
      red[c][lane] = acc;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int c = lane >> 2, qtr = lane & 3;
    double v = 0;
#pragma unroll
    for (int e = 0; e < 16; ++e) v += red[c][16 * qtr + e];
    v += __shfl_xor(v, 1, 64);
    v += __shfl_xor(v, 2, 64);
    const int k = wave + 4 * c;
    if (qtr == 0 && k < n) {
      if (chunk == 0) colsum[k] = v;
      else unsafeAtomicAdd(&part[sd.col_begin + k], v);
    }
    if (chunk != 0) {
      // every wave waits for its own atomics before the block arrives (as in bwd_kernel)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (threadIdx.x == 0)
        __hip_atomic_fetch_add(&counter[s], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    const int r = threadIdx.x;
    double yi = yown - (colsum[r] + others[r]);
#pragma unroll
    for (int k = kMaxCols - 1; k >= 0; --k) yi -= Ls[k][r] * lane_value(yi, k);
    if (r < n) {
      __hip_atomic_store(&ysol[sd.col_begin + r], final_value(yi), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
      yout[sd.col_begin + r] = yi;  // for the levels below and the inverse permutation
    }
    if (r == 0 && nchunks > 1) counter[s] = 0;
  }
}

// Several right-hand sides at once (covariances: every column of the identity). A block takes its
// task's panel rows for a group of kRhsGroup right-hand sides (blockIdx.y), stored one after the
// other with stride n: the panel and L11 are read once per group, each wavefront runs the
// triangular solve of one of them, and a level is one launch whatever their number. One launch pair
// per level per right-hand side left the chip to one block chain at a time: the 906 columns of a
// 151-pose covariance took 202 ms from Hessian to dense inverse, now 4.0 (analysis and transfers
// included).
constexpr int kRhsGroup = 4;

__global__ void __launch_bounds__(256) permute_many_kernel(int32_t n, int32_t nrhs,
                                                           const int32_t* __restrict__ perm,
                                                           const double* __restrict__ b,
                                                           double* __restrict__ y,
                                                           double* __restrict__ part) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  for (int32_t r = blockIdx.y; r < nrhs; r += gridDim.y) {
    y[(int64_t)r * n + perm[i]] = b[(int64_t)r * n + i];
    part[(int64_t)r * n + i] = 0.0;
  }
}
__global__ void __launch_bounds__(256) unpermute_many_kernel(int32_t n, int32_t nrhs,
                                                             const int32_t* __restrict__ perm,
                                                             const double* __restrict__ y,
                                                             double* __restrict__ x) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  for (int32_t r = blockIdx.y; r < nrhs; r += gridDim.y)
    x[(int64_t)r * n + i] = y[(int64_t)r * n + perm[i]];
}

// Forward: as fwd_kernel; wave w solves right-hand side w of the group, then thread t takes below
// row t % 128 for two of the four.
__global__ void __launch_bounds__(256) fwd_many_kernel(const SnTask* __restrict__ tasks, int32_t n_all,
                                                       int32_t nrhs,
                                                       const int32_t* __restrict__ rows,
                                                       const double* __restrict__ panel,
                                                       const double* __restrict__ l11,
                                                       double* __restrict__ yacc,
                                                       double* __restrict__ yout) {
  static_assert(kSolveRows == 128 && kRhsGroup == 4, "two halves of 128 threads, four wavefronts");
  __shared__ double Ls[kMaxCols][kMaxCols + 1];
  __shared__ double ys[kRhsGroup][kMaxCols];
  const SnTask tk = tasks[blockIdx.x];
  const int chunk = tk.a;
  const SnDesc sd = tk.d;
  const int n = sd.ncols, ld = sd.ld, mb = ld - n;
  const double* P = panel + sd.panel_off;
  const int32_t* rw = rows + sd.rows_off + n;
  const int i = chunk * kSolveRows + (threadIdx.x & (kSolveRows - 1));
  double lrow[kMaxCols];
  {
    const int64_t r = mb > 0 ? n + min(i, mb - 1) : 0;  // clamped into the panel
#pragma unroll
    for (int k = 0; k < kMaxCols; ++k) lrow[k] = P[(int64_t)min(k, n - 1) * ld + r];
  }
  stage_l11(l11 + sd.l11_off, n, Ls);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int rhs = blockIdx.y * kRhsGroup + wave;
  double yi = 0;
  if (rhs < nrhs && lane < n) yi = yacc[(int64_t)rhs * n_all + sd.col_begin + lane];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kMaxCols; ++k) yi -= Ls[lane][k] * lane_value(yi, k);
  if (chunk == 0 && rhs < nrhs && lane < n) yout[(int64_t)rhs * n_all + sd.col_begin + lane] = yi;
  ys[wave][lane] = lane < n ? yi : 0.0;
  __syncthreads();
  if (i < mb) {
    const int32_t row = rw[i];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int g = 2 * (threadIdx.x / kSolveRows) + h, q = blockIdx.y * kRhsGroup + g;
      if (q >= nrhs) break;
      double acc = 0;
#pragma unroll
      for (int k = 0; k < kMaxCols; ++k) acc += lrow[k] * ys[g][k];
      unsafeAtomicAdd(&yacc[(int64_t)q * n_all + row], -acc);
    }
  }
}

// Backward: as bwd_kernel (wave w forms the sums of columns w, w + 4, .. for the whole group); the
// last chunk block of (s, group) solves the four right-hand sides, a wavefront each.
__global__ void __launch_bounds__(256) bwd_many_kernel(const SnTask* __restrict__ tasks, int32_t n_all,
                                                       int32_t n_snodes, int32_t nrhs,
                                                       const int32_t* __restrict__ rows,
                                                       const double* __restrict__ panel,
                                                       const double* __restrict__ l11,
                                                       const double* __restrict__ D,
                                                       double* __restrict__ yout,
                                                       double* __restrict__ part,
                                                       int32_t* __restrict__ counter) {
  constexpr int kPer = kMaxCols / 4;
  __shared__ double Ls[kMaxCols][kMaxCols + 1];
  __shared__ double red_all[4][kPer][64 + 1];
  __shared__ int last;
  const SnTask tk = tasks[blockIdx.x];
  const int s = tk.s, chunk = tk.a;
  const SnDesc sd = tk.d;
  const int n = sd.ncols, ld = sd.ld, mb = ld - n;
  const int nchunks = max(1, (mb + kSolveRows - 1) / kSolveRows);
  const double* P = panel + sd.panel_off + n;
  const int32_t* rw = rows + sd.rows_off + n;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  stage_l11(l11 + sd.l11_off, n, Ls);
  const int rhs = blockIdx.y * kRhsGroup + wave;
  double yown = 0;
  if (rhs < nrhs && lane < n)
    yown = yout[(int64_t)rhs * n_all + sd.col_begin + lane] / D[sd.col_begin + lane];
  if (mb > 0) {
    double acc[kRhsGroup][kPer] = {};
#pragma unroll
    for (int t = 0; t < kSolveRows / 64; ++t) {
      const int i = chunk * kSolveRows + lane + 64 * t;
      const int ic = min(i, mb - 1);
      const int32_t row = rw[ic];
      double yv[kRhsGroup];
#pragma unroll
      for (int g = 0; g < kRhsGroup; ++g) {
        const int q = blockIdx.y * kRhsGroup + g;
        const double yl = yout[(int64_t)min(q, nrhs - 1) * n_all + row];
        yv[g] = (i < mb && q < nrhs) ? yl : 0.0;
      }
#pragma unroll
      for (int c = 0; c < kPer; ++c) {
        const double l = P[(int64_t)min(wave + 4 * c, n - 1) * ld + ic];
#pragma unroll
        for (int g = 0; g < kRhsGroup; ++g) acc[g][c] += l * yv[g];
      }
    }
    auto red = red_all[wave];
    const int c = lane >> 2, qtr = lane & 3, k = wave + 4 * c;
#pragma unroll
    for (int g = 0; g < kRhsGroup; ++g) {
#pragma unroll
      for (int e = 0; e < kPer; ++e) red[e][lane] = acc[g][e];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      double v = 0;
#pragma unroll
      for (int t = 0; t < 16; ++t) v += red[c][16 * qtr + t];
      v += __shfl_xor(v, 1, 64);
      v += __shfl_xor(v, 2, 64);
      const int q = blockIdx.y * kRhsGroup + g;
      if (qtr == 0 && k < n && q < nrhs)
        unsafeAtomicAdd(&part[(int64_t)q * n_all + sd.col_begin + k], v);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();  // the next right-hand side overwrites red
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  }
  // every wave waits for its own atomics before the block arrives (as in bwd_kernel)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  int32_t* cnt = counter + (int64_t)blockIdx.y * n_snodes + s;
  if (threadIdx.x == 0)
    last = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
           nchunks - 1;
  __syncthreads();
  if (!__builtin_amdgcn_readfirstlane(last)) return;  // uniform across the block
  if (threadIdx.x == 0) *cnt = 0;  // ready for the next solve
  if (rhs >= nrhs) return;
  double yi = 0;
  if (lane < n)
    yi = yown - (mb > 0 ? __hip_atomic_load(&part[(int64_t)rhs * n_all + sd.col_begin + lane],
                                            __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                        : 0.0);
#pragma unroll
  for (int k = kMaxCols - 1; k >= 0; --k) yi -= Ls[k][lane] * lane_value(yi, k);
  if (lane < n) yout[(int64_t)rhs * n_all + sd.col_begin + lane] = yi;
}

}  // namespace

void SupernodalLDLT::setup(const CholSymbolic& sym, const int32_t* colptr, const int32_t* rowind,
                           hipStream_t s) {
  SYMHIP_CHECK(sym.max_snode_cols <= kMaxCols, "supernode wider than the kernel tile");
  sym_ = sym;
  panel_.resize(std::max<int64_t>(1, sym.panel_size()));
  std::vector<int64_t> map;
  std::vector<int32_t> diag;
  nnz_ = 0;
  if (colptr) {
    map = chol_assembly_map(sym, colptr, rowind);
    nnz_ = colptr[sym.n];
    asm_map_.upload(map, s);
    const int64_t size = sym.panel_size();
    if (size > 0 && size <= kListPanel) {
      diag.assign(sym.n, 0);
      for (int32_t j = 0; j < sym.n; ++j)
        for (int32_t q = colptr[j]; q < colptr[j + 1]; ++q)
          if (rowind[q] == j) diag[j] = q;
      diag_pos_.upload(diag, s);
      panel_src_.resize(size);
      hipLaunchKernelGGL(panel_fill_kernel, dim3(std::min(grid_for(size, 256), 4096)), dim3(256), 0,
                         s, size, panel_src_.get());
      if (nnz_)
        hipLaunchKernelGGL(panel_list_kernel, dim3(grid_for(nnz_, 256)), dim3(256), 0, s, nnz_,
                           asm_map_.get(), panel_src_.get());
      HIP_OK(hipGetLastError());
    }
  }
  const size_t len = line_round(std::max(1, sym.n));
  vectors_.resize(5 * len);
  D_ = vectors_.get();
  y_ = D_ + len;
  yout_ = y_ + len;
  part_ = yout_ + len;
  ysol_ = reinterpret_cast<unsigned long long*>(part_ + len);
  counter_.resize(line_round(sym.n_snodes) + 1);
  fill_zero_i32(counter_.get(), counter_.size(), s);
  rows_.upload(sym.sn_rows, s);
  perm_.upload(sym.perm, s);
  upd_rel_.upload(sym.upd_rel, s);
  // supernode descriptors
  std::vector<SnDesc> desc(std::max(1, sym.n_snodes));
  int64_t l11_size = 0;
  for (int k = 0; k < sym.n_snodes; ++k) {
    const int n = sym.sn_col_begin[k + 1] - sym.sn_col_begin[k];
    desc[k] = SnDesc{sym.sn_panel_off[k], l11_size, n, sym.sn_rows_ptr[k + 1] - sym.sn_rows_ptr[k],
                     sym.sn_col_begin[k], sym.sn_rows_ptr[k]};
    l11_size += (int64_t)n * n;
  }
  l11_.resize(std::max<int64_t>(1, l11_size));
  fill_zero(l11_.get(), l11_.size(), s);
  // scatter targets per below-row
  std::vector<int64_t> scol(std::max<size_t>(1, sym.sn_rows.size()), 0);
  std::vector<int32_t> srel(std::max<size_t>(1, sym.sn_rows.size()), 0);
  for (int k = 0; k < sym.n_snodes; ++k) {
    const int n = sym.sn_col_begin[k + 1] - sym.sn_col_begin[k];
    const int q0 = sym.sn_rows_ptr[k] + n;
    for (int seg = sym.upd_ptr[k]; seg < sym.upd_ptr[k + 1]; ++seg) {
      const int t = sym.upd_target[seg];
      const int jb = sym.upd_seg_begin[seg];
      const int je = seg + 1 < sym.upd_ptr[k + 1] ? sym.upd_seg_begin[seg + 1]
                                                  : sym.sn_rows_ptr[k + 1] - q0;
      const int ldt = sym.sn_rows_ptr[t + 1] - sym.sn_rows_ptr[t];
      for (int j = jb; j < je; ++j) {
        const int col = sym.sn_rows[q0 + j] - sym.sn_col_begin[t];
        scol[q0 + j] = sym.sn_panel_off[t] + (int64_t)col * ldt;
        srel[q0 + j] = sym.upd_rel_ptr[seg] - jb;
      }
    }
  }
  scat_col_.upload(scol, s);
  scat_rel_.upload(srel, s);
  // Work lists per level
  std::vector<int32_t> snl, dt, upd, sol;
  lvl_snode_ptr_.assign(1, 0);
  lvl_solve_ptr_.assign(1, 0);
  lvl_trsm_ptr_.assign(1, 0);
  lvl_upd_ptr_.assign(1, 0);
  for (int l = 0; l < sym.n_levels; ++l) {
    for (int q = sym.level_ptr[l]; q < sym.level_ptr[l + 1]; ++q) {
      const int sn = sym.level_snodes[q];
      snl.push_back(sn);
      const int n = sym.sn_col_begin[sn + 1] - sym.sn_col_begin[sn];
      const int mb = sym.sn_rows_ptr[sn + 1] - sym.sn_rows_ptr[sn] - n;
      const int chunks = std::max(1, (mb + 63) / 64);
      for (int c = 0; c < chunks; ++c) {
        dt.push_back(sn);
        dt.push_back(c);
      }
      const int schunks = std::max(1, (mb + kSolveRows - 1) / kSolveRows);
      for (int c = 0; c < schunks; ++c) {
        sol.push_back(sn);
        sol.push_back(c);
      }
    }
    constexpr int kt = kTile;
    for (int q = sym.level_ptr[l]; q < sym.level_ptr[l + 1]; ++q) {
      const int sn = sym.level_snodes[q];
      const int n = sym.sn_col_begin[sn + 1] - sym.sn_col_begin[sn];
      const int mb = sym.sn_rows_ptr[sn + 1] - sym.sn_rows_ptr[sn] - n;
      const int T = (mb + kt - 1) / kt;
      for (int ti = 0; ti < T; ++ti)
        for (int tj = 0; tj <= ti; ++tj) {
          upd.push_back(sn);
          upd.push_back(ti);
          upd.push_back(tj);
        }
    }
    lvl_snode_ptr_.push_back((int32_t)snl.size());
    lvl_solve_ptr_.push_back((int32_t)sol.size() / 2);
    lvl_trsm_ptr_.push_back((int32_t)dt.size() / 2);
    lvl_upd_ptr_.push_back((int32_t)upd.size() / 3);
  }
  lvl_snodes_.upload(snl, s);
  auto upload_tasks = [&](const std::vector<int32_t>& items, int per, DBuf<uint8_t>& out) {
    std::vector<SnTask> t(std::max<size_t>(1, items.size() / per));
    for (size_t q = 0; q < items.size() / per; ++q) {
      const int32_t* it = &items[q * per];
      t[q] = SnTask{desc[it[0]], it[0], it[1], per > 2 ? it[2] : 0, 0};
    }
    out.resize(t.size() * sizeof(SnTask));
    HIP_OK(hipMemcpyAsync(out.get(), t.data(), t.size() * sizeof(SnTask), hipMemcpyHostToDevice, s));
  };
  upload_tasks(sol, 2, solve_tasks_);
  // Backward in one launch: the levels from the root down to the first with more blocks than are
  // resident (two to a CU). Below it a level's time is its blocks', not its chain's, and
  // bwd_kernel's lean form runs four to a CU.
  for (chain_levels_ = 0; chain_levels_ < sym.n_levels; ++chain_levels_) {
    const int l = sym.n_levels - 1 - chain_levels_;
    if (lvl_solve_ptr_[l + 1] - lvl_solve_ptr_[l] > 2 * kCus) break;
  }
  n_chain_ = lvl_solve_ptr_[sym.n_levels] - lvl_solve_ptr_[sym.n_levels - chain_levels_];
  upload_tasks(dt, 2, trsm_tasks_);
  upload_tasks(upd, 3, upd_tasks_);
  HIP_OK(hipStreamSynchronize(s));
}

void SupernodalLDLT::factorize(const double* a_values, hipStream_t s, const double* b,
                               const double* damping) {
  if (sym_.n_levels == 0) return;
  fused_ = b != nullptr;
  HIP_OK(hipGraphLaunch(cached_graph(fact_graphs_, {a_values, damping, b}, nullptr, 1.0, s, [&] {
    const int64_t size = sym_.panel_size();
    if (panel_src_.size()) {
      hipLaunchKernelGGL(assemble_list_kernel, dim3(grid_for(size, 512)), dim3(256), 0, s, size,
                         panel_src_.get(), diag_pos_.get(), a_values, damping, panel_.get());
    } else {
      fill_zero(panel_.get(), size, s);
      if (nnz_)
        hipLaunchKernelGGL(assemble_scatter_kernel, dim3(std::min(grid_for(nnz_, 256), 8192)),
                           dim3(256), 0, s, nnz_, asm_map_.get(), a_values, damping, panel_.get());
    }
    launch_factorize(b, s);
  }), s));
}

SupernodalLDLT::~SupernodalLDLT() {
  for (auto* cache : {&fact_graphs_, &solve_graphs_, &bwd_graphs_})
    for (auto& g : *cache) (void)hipGraphExecDestroy(g.exec);
}

namespace {
template <typename F>
hipGraphExec_t capture(hipStream_t s, F&& launches) {
  hipGraph_t g;
  hipGraphExec_t exec;
  HIP_OK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
  launches();
  HIP_OK(hipStreamEndCapture(s, &g));
  HIP_OK(hipGraphInstantiate(&exec, g, nullptr, nullptr, 0));
  HIP_OK(hipGraphDestroy(g));
  return exec;
}
}  // namespace

void SupernodalLDLT::factorize_assembled(hipStream_t s, const double* b) {
  if (sym_.n_levels == 0) return;
  fused_ = b != nullptr;
  HIP_OK(hipGraphLaunch(cached_graph(fact_graphs_, {nullptr, nullptr, b}, nullptr, 1.0, s,
                                     [&] { launch_factorize(b, s); }), s));
}

void SupernodalLDLT::solve(const double* b, double* x, hipStream_t s) {
  if (sym_.n == 0) return;
  HIP_OK(hipGraphLaunch(cached_graph(solve_graphs_, {nullptr, nullptr, b}, x, 1.0, s,
                                     [&] { launch_solve(b, x, s); }), s));
}

int32_t SupernodalLDLT::many_capacity(int32_t nrhs) const {
  const int64_t per = 5 * sizeof(double) * (int64_t)std::max(1, sym_.n);  // y, yout, part, b, x
  return (int32_t)std::min<int64_t>(nrhs, std::clamp<int64_t>(kManyBytes / per, kRhsGroup, 4096));
}

void SupernodalLDLT::reserve_many(int32_t nrhs, hipStream_t s) {
  const size_t need = (size_t)sym_.n * nrhs;
  const size_t cneed = (size_t)grid_for(nrhs, kRhsGroup) * sym_.n_snodes;
  HIP_OK(hipStreamSynchronize(s));  // an earlier pass may still use the smaller buffers
  for (auto* v : {&many_y_, &many_yout_, &many_part_})
    if (v->size() < need) v->resize(need);
  if (many_counter_.size() < cneed) {
    many_counter_.resize(cneed);
    fill_zero_i32(many_counter_.get(), (int64_t)cneed, s);
  }
}

void SupernodalLDLT::solve_many(const double* b, double* x, int32_t nrhs, hipStream_t s) {
  const int32_t n = sym_.n;
  if (n == 0 || nrhs <= 0) return;
  const int32_t groups = grid_for(nrhs, kRhsGroup);
  SYMHIP_CHECK(many_part_.size() >= (size_t)n * nrhs &&
                   many_counter_.size() >= (size_t)groups * sym_.n_snodes,
               "internal: solve_many without reserve_many");
  const SnTask* tasks = reinterpret_cast<const SnTask*>(solve_tasks_.get());
  const dim3 pg(grid_for(n, 256), std::min(nrhs, 65535));
  hipLaunchKernelGGL(permute_many_kernel, pg, dim3(256), 0, s, n, nrhs, perm_.get(), b,
                     many_y_.get(), many_part_.get());
  for (int l = 0; l < sym_.n_levels; ++l) {
    const int nb = lvl_solve_ptr_[l + 1] - lvl_solve_ptr_[l];
    hipLaunchKernelGGL(fwd_many_kernel, dim3(nb, groups), dim3(256), 0, s,
                       tasks + lvl_solve_ptr_[l], n, nrhs, rows_.get(), panel_.get(), l11_.get(),
                       many_y_.get(), many_yout_.get());
  }
  for (int l = sym_.n_levels - 1; l >= 0; --l) {
    const int nb = lvl_solve_ptr_[l + 1] - lvl_solve_ptr_[l];
    hipLaunchKernelGGL(bwd_many_kernel, dim3(nb, groups), dim3(256), 0, s,
                       tasks + lvl_solve_ptr_[l], n, sym_.n_snodes, nrhs, rows_.get(),
                       panel_.get(), l11_.get(), D_, many_yout_.get(), many_part_.get(),
                       many_counter_.get());
  }
  hipLaunchKernelGGL(unpermute_many_kernel, pg, dim3(256), 0, s, n, nrhs, perm_.get(),
                     many_yout_.get(), x);
  HIP_OK(hipGetLastError());
}

void SupernodalLDLT::solve_fused(double* x, hipStream_t s, bool negate) {
  if (sym_.n == 0) return;
  SYMHIP_CHECK(fused_, "solve_fused needs a factorization given the right-hand side");
  const double sign = negate ? -1.0 : 1.0;
  HIP_OK(hipGraphLaunch(cached_graph(bwd_graphs_, {}, x, sign, s,
                                     [&] { launch_backward(x, sign, s); }), s));
}

template <typename F>
hipGraphExec_t SupernodalLDLT::cached_graph(std::vector<CachedGraph>& cache, const GraphInputs& in,
                                            double* x, double sign, hipStream_t s, F&& launches) {
  for (const auto& g : cache)
    if (g.in == in && g.x == x && g.sign == sign && g.f32 == f32_updates_) return g.exec;
  if (cache.size() >= 8) {  // bound the cache; the oldest goes
    (void)hipGraphExecDestroy(cache.front().exec);
    cache.erase(cache.begin());
  }
  cache.push_back({in, x, sign, f32_updates_, capture(s, launches)});
  return cache.back().exec;
}

void SupernodalLDLT::launch_factorize(const double* b, hipStream_t s) {
  const SnTask* trsm = reinterpret_cast<const SnTask*>(trsm_tasks_.get());
  const SnTask* upd = reinterpret_cast<const SnTask*>(upd_tasks_.get());
  if (b)
    hipLaunchKernelGGL(permute_kernel, dim3(grid_for(sym_.n, 256)), dim3(256), 0, s, sym_.n,
                       perm_.get(), b, y_, part_, ysol_, ticket());
  for (int l = 0; l < sym_.n_levels; ++l) {
    const int nt = lvl_trsm_ptr_[l + 1] - lvl_trsm_ptr_[l];
    if (nt) {
      if (b)
        hipLaunchKernelGGL(diag_trsm_kernel<true>, dim3(nt), dim3(kDiagThreads), 0, s,
                           trsm + lvl_trsm_ptr_[l], panel_.get(),
                           l11_.get(), D_, rows_.get(), y_, yout_);
      else
        hipLaunchKernelGGL(diag_trsm_kernel<false>, dim3(nt), dim3(kDiagThreads), 0, s,
                           trsm + lvl_trsm_ptr_[l], panel_.get(),
                           l11_.get(), D_, nullptr, nullptr, nullptr);
    }
    const int nu = lvl_upd_ptr_[l + 1] - lvl_upd_ptr_[l];
    if (nu) {
      auto kern = f32_updates_ ? update_kernel<kTile, float> : update_kernel<kTile, double>;
      hipLaunchKernelGGL(kern, dim3(nu), dim3(256), 0, s, upd + lvl_upd_ptr_[l], panel_.get(),
                         D_, scat_col_.get(), scat_rel_.get(), upd_rel_.get());
    }
  }
  HIP_OK(hipGetLastError());
}

void SupernodalLDLT::launch_solve(const double* b, double* x, hipStream_t s) {
  const int n = sym_.n;
  const SnTask* tasks = reinterpret_cast<const SnTask*>(solve_tasks_.get());
  hipLaunchKernelGGL(permute_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, n, perm_.get(), b,
                     y_, part_, ysol_, ticket());
  for (int l = 0; l < sym_.n_levels; ++l) {
    const int nb = lvl_solve_ptr_[l + 1] - lvl_solve_ptr_[l];
    hipLaunchKernelGGL(fwd_kernel, dim3(nb), dim3(256), 0, s,
                       tasks + lvl_solve_ptr_[l], rows_.get(),
                       panel_.get(), l11_.get(), y_, yout_);
  }
  launch_backward(x, 1.0, s);
}

// The backward levels (D^-1 folded in) and the inverse permutation (times sign), from the forward
// result in yout.
void SupernodalLDLT::launch_backward(double* x, double sign, hipStream_t s) {
  const int n = sym_.n;
  const SnTask* tasks = reinterpret_cast<const SnTask*>(solve_tasks_.get());
  if (n_chain_)
    hipLaunchKernelGGL(bwd_chain_kernel, dim3(n_chain_), dim3(256), 0, s,
                       tasks + lvl_solve_ptr_[sym_.n_levels] - 1, rows_.get(), panel_.get(),
                       l11_.get(), D_, yout_, ysol_, part_, counter_.get(), ticket());
  for (int l = sym_.n_levels - 1 - chain_levels_; l >= 0; --l) {
    const int nb = lvl_solve_ptr_[l + 1] - lvl_solve_ptr_[l];
    auto kern = nb > 2 * kCus ? bwd_kernel<true> : bwd_kernel<false>;
    hipLaunchKernelGGL(kern, dim3(nb), dim3(256), 0, s, tasks + lvl_solve_ptr_[l], rows_.get(),
                       panel_.get(), l11_.get(), D_, yout_, part_, counter_.get());
  }
  hipLaunchKernelGGL(unpermute_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, n, perm_.get(), yout_,
                     sign, x);
  HIP_OK(hipGetLastError());
}

void SupernodalLDLT::factor_values(const std::vector<int32_t>& l_colptr,
                                   const std::vector<int32_t>& l_rowind, double* values,
                                   hipStream_t s) const {
  std::vector<double> panels(sym_.panel_size()), l11(l11_.size());
  panel_.download(panels.data(), panels.size(), s);
  l11_.download(l11.data(), l11.size(), s);
  HIP_OK(hipStreamSynchronize(s));
  int64_t l11_off = 0;
  for (int32_t k = 0; k < sym_.n_snodes; ++k) {
    const int32_t c0 = sym_.sn_col_begin[k], c1 = sym_.sn_col_begin[k + 1], n = c1 - c0;
    const int32_t r0 = sym_.sn_rows_ptr[k], nrows = sym_.sn_rows_ptr[k + 1] - r0;
    const int32_t* rows = sym_.sn_rows.data() + r0;
    for (int32_t j = c0; j < c1; ++j) {
      const int32_t jj = j - c0;
      for (int32_t q = l_colptr[j]; q < l_colptr[j + 1]; ++q) {
        const int32_t r = l_rowind[q];
        if (r < c1) {
          values[q] = l11[l11_off + (int64_t)jj * n + (r - c0)];
        } else {
          const int32_t* pos = std::lower_bound(rows + n, rows + nrows, r);
          SYMHIP_CHECK(pos != rows + nrows && *pos == r,
                       "factor pattern entry outside the supernodal panel");
          values[q] = panels[sym_.sn_panel_off[k] + (int64_t)jj * nrows + (pos - rows)];
        }
      }
    }
    l11_off += (int64_t)n * n;
  }
}

void SupernodalLDLT::download_factor(std::vector<double>& panels, std::vector<double>& d,
                                     hipStream_t s) const {
  panels.resize(sym_.panel_size());
  d.resize(sym_.n);
  panel_.download(panels.data(), panels.size(), s);
  if (!d.empty())
    HIP_OK(hipMemcpyAsync(d.data(), D_, d.size() * sizeof(double), hipMemcpyDeviceToHost, s));
  HIP_OK(hipStreamSynchronize(s));
}

}  // namespace symhip
