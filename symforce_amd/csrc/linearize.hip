// Batched per-factor-type linearization into the reference's hessian_lower CSC layout, in two
// atomic-free passes (the local-record pass and the gather pass described in linearize.h).
//
// FP64 atomics were the scatter form's cost: at 100 000 Pose3 nodes (115 000 between factors, 90
// hessian and rhs entries each, ~10 M atomic adds per linearization) its launch took 480 us, and
// 81 us with the atomics replaced by plain stores (timing only). The local records (720 B per
// between factor) and the gather move ~0.2 GB instead.
#include "./factor_traits.h"
#include "./linearize.h"
#include "./util.h"

namespace symhip {

namespace {

// Local outputs per factor of type FTC, in the order the pass-1 kernel writes them: for each
// linearized argument i, its rhs entries (td_i), its lower diagonal block column by column
// (td_i (td_i + 1) / 2), then its block with each earlier argument j, rows of i by columns of j
// (td_i td_j).
template <int FTC>
constexpr int local_size() {
  using F = FT<FTC>;
  int L = 0;
  for (int i = 0; i < F::NL; ++i) {
    L += F::td(i) + F::td(i) * (F::td(i) + 1) / 2;
    for (int j = 0; j < i; ++j) L += F::td(i) * F::td(j);
  }
  return L;
}

template <int FTC>
__global__ void __launch_bounds__(128) lin_local_kernel(int32_t n, const int32_t* __restrict__ arg_off,
                                                        const int32_t* __restrict__ res_off,
                                                        const double* __restrict__ values,
                                                        double* __restrict__ residual,
                                                        double* __restrict__ contrib) {
  using F = FT<FTC>;
  constexpr int L = local_size<FTC>();
  const int32_t f = blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= n) return;
  const double* a[F::NA];
#pragma unroll
  for (int k = 0; k < F::NA; ++k) a[k] = values + arg_off[k * n + f];
  double r[F::D];
  double J[F::D][F::T];
  F::template eval<double>(a, r, J);
  if (residual) {
    const int32_t ro = res_off[f];
#pragma unroll
    for (int i = 0; i < F::D; ++i) residual[ro + i] = r[i];
  }
  if (!contrib) return;
  double* out = contrib + (int64_t)f * L;
  int o = 0;
#pragma unroll
  for (int ki = 0; ki < F::NL; ++ki) {
    const int tdi = F::td(ki), fi = F::foff(ki);
#pragma unroll
    for (int c = 0; c < tdi; ++c) {
      double acc = 0;
#pragma unroll
      for (int q = 0; q < F::D; ++q) acc += J[q][fi + c] * r[q];
      out[o++] = acc;
    }
#pragma unroll
    for (int c = 0; c < tdi; ++c)
#pragma unroll
      for (int rr = c; rr < tdi; ++rr) {
        double acc = 0;
#pragma unroll
        for (int q = 0; q < F::D; ++q) acc += J[q][fi + rr] * J[q][fi + c];
        out[o++] = acc;
      }
#pragma unroll
    for (int kj = 0; kj < ki; ++kj) {
      const int tdj = F::td(kj), fj = F::foff(kj);
#pragma unroll
      for (int rr = 0; rr < tdi; ++rr)
#pragma unroll
        for (int cc = 0; cc < tdj; ++cc) {
          double acc = 0;
#pragma unroll
          for (int q = 0; q < F::D; ++q) acc += J[q][fi + rr] * J[q][fj + cc];
          out[o++] = acc;
        }
    }
  }
}

// out[e] = sum of contrib[idx[p]] over p in [ptr[e], ptr[e + 1]), for the hessian_lower entries
// e < nnz (into hval) and the rhs entries after them (into rhs), in one launch. An entry's list is
// as long as the number of factors that touch its two keys: 1 to 3 in a pose graph, but as many as
// a camera has observations on its diagonal block, and a thread that walks a thousand of them one
// dependent load pair after the other takes 370 us (20 cameras x 1000 landmarks: 74 % of the device
// time; dealing the lists by length took six LM iterations there from 7.10 to 1.93 ms). Up to
// kThreadList contributions are summed by a thread (two rounds of four loads), up to kGroupList by
// 16 lanes (at most eight such rounds, and four neighbouring lists share a wavefront), longer ones
// by a block of 256. Fixed strides and a fixed reduction tree: the sums are the same from run to
// run.
constexpr int kThreadList = 8, kGroupList = 512, kGroup = 16;

// The partial sum of every `step`-th contribution from q on, four loads in flight.
__device__ __forceinline__ double list_sum(const int32_t* __restrict__ idx,
                                           const double* __restrict__ contrib, int32_t q,
                                           int32_t end, int32_t step) {
  double acc = 0;
  const int32_t* p = idx + q;
  int32_t left = end - q;  // negative for a lane past a short list's end
  for (; left > 3 * step; left -= 4 * step, p += 4 * step) {
    const int32_t i0 = p[0], i1 = p[step], i2 = p[2 * step], i3 = p[3 * step];
    const double c0 = contrib[i0], c1 = contrib[i1], c2 = contrib[i2], c3 = contrib[i3];
    acc += c0;
    acc += c1;
    acc += c2;
    acc += c3;
  }
  for (; left > 0; left -= step, p += step) acc += contrib[*p];
  return acc;
}

__global__ void __launch_bounds__(256) gather_sum_kernel(
    int64_t nnz, int64_t n, const int32_t* __restrict__ ptr, const int32_t* __restrict__ idx,
    const int32_t* __restrict__ group, int32_t n_group, const int32_t* __restrict__ wide,
    int32_t thread_blocks, int32_t group_blocks, const double* __restrict__ contrib,
    double* __restrict__ hval, double* __restrict__ rhs) {
  auto put = [&](int64_t e, double v) {
    if (e < nnz) {
      if (hval) hval[e] = v;
    } else if (rhs) {
      rhs[e - nnz] = v;
    }
  };
  const int t = threadIdx.x;
  if ((int)blockIdx.x < thread_blocks) {
    const int64_t e = blockIdx.x * (int64_t)256 + t;
    if (e >= n) return;
    const int32_t q0 = ptr[e], q1 = ptr[e + 1];
    if (q1 - q0 <= kThreadList) put(e, list_sum(idx, contrib, q0, q1, 1));
  } else if ((int)blockIdx.x < thread_blocks + group_blocks) {
    const int32_t k = ((int)blockIdx.x - thread_blocks) * (256 / kGroup) + t / kGroup;
    const bool live = k < n_group;
    const int32_t e = live ? group[k] : 0;
    double v = live ? list_sum(idx, contrib, ptr[e] + t % kGroup, ptr[e + 1], kGroup) : 0.0;
#pragma unroll
    for (int o = kGroup / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if (live && t % kGroup == 0) put(e, v);
  } else {  // a block per list
    __shared__ double ws[4];
    const int32_t e = wide[(int)blockIdx.x - thread_blocks - group_blocks];
    double v = list_sum(idx, contrib, ptr[e] + t, ptr[e + 1], 256);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((t & 63) == 0) ws[t >> 6] = v;
    __syncthreads();
    if (t == 0) put(e, (ws[0] + ws[1]) + (ws[2] + ws[3]));
  }
}

int local_size_of(int type) {
  int L = 0;
  dispatch_factor_type(type, [&]<int C>() { L = local_size<C>(); });
  return L;
}

}  // namespace

void CscLinearizer::setup(const HostProblem& p, hipStream_t s) {
  nnz = p.nnz();
  N = p.N;
  M = p.M;
  groups_.clear();
  std::vector<std::vector<int32_t>> by_type(kNumFactorTypes);
  for (int32_t f = 0; f < p.n_factors; ++f) by_type[p.ftype[f]].push_back(f);
  std::vector<int64_t> base(p.n_factors);  // first contribution entry of each factor
  int64_t total = 0;
  for (int t = 1; t < kNumFactorTypes; ++t) {
    const auto& fs = by_type[t];
    if (fs.empty()) continue;
    const FactorSpec spec = factor_spec(t);
    const int32_t n = (int32_t)fs.size();
    const int L = local_size_of(t);
    std::vector<int32_t> ao((size_t)spec.nargs * n), ro(n);
    for (int32_t i = 0; i < n; ++i) {
      const int32_t f = fs[i];
      for (int a = 0; a < spec.nargs; ++a)
        ao[(size_t)a * n + i] = p.storage_offset[p.fargs[p.fargs_ptr[f] + a]];
      ro[i] = p.res_off[f];
      base[f] = total + (int64_t)i * L;
    }
    FactorGroup g;
    g.type = t;
    g.n = n;
    g.arg_off.upload(ao, s);
    g.res_off.upload(ro, s);
    g.contrib_off = total;
    groups_.push_back(std::move(g));
    total += (int64_t)n * L;
  }
  SYMHIP_CHECK(total < INT32_MAX && nnz + N < INT32_MAX,
               "linearization exceeds 2^31 local contributions");
  contrib_.resize(std::max<int64_t>(1, total));
  // Gather lists, replaying each factor's local layout against the reference's storage map
  // (col_starts in the order problem.cc builds it); factors in their given order.
  auto replay = [&](auto&& emit_h, auto&& emit_r) {
    for (int32_t f = 0; f < p.n_factors; ++f) {
      const FactorSpec spec = factor_spec(p.ftype[f]);
      int td[6], toff[6], nl = 0;
      for (int a = 0; a < spec.nargs; ++a) {
        if (!((spec.lin_mask >> a) & 1)) continue;
        const int32_t k = p.fargs[p.fargs_ptr[f] + a];
        td[nl] = tangent_dim(p.types[k]);
        toff[nl++] = p.tan_off[k];
      }
      const int32_t* cs = p.col_starts.data() + p.cs_ptr[f];
      int64_t o = base[f];
      for (int ki = 0; ki < nl; ++ki) {
        const int tdi = td[ki];
        if (toff[ki] < 0) {
          o += tdi + tdi * (tdi + 1) / 2;
          for (int kj = 0; kj < ki; ++kj) o += tdi * td[kj];
          continue;
        }
        for (int c = 0; c < tdi; ++c) emit_r(toff[ki] + c, o + c);
        o += tdi;
        for (int c = 0; c < tdi; ++c) {
          const int32_t start = *cs++;
          for (int rr = c; rr < tdi; ++rr) emit_h(start + rr - c, o++);
        }
        for (int kj = 0; kj < ki; ++kj) {
          const int tdj = td[kj];
          if (toff[kj] >= 0) {
            if (toff[kj] < toff[ki]) {
              // stored as columns of argument j, rows of argument i
              for (int cj = 0; cj < tdj; ++cj) {
                const int32_t start = *cs++;
                for (int rr = 0; rr < tdi; ++rr) emit_h(start + rr, o + rr * tdj + cj);
              }
            } else {
              // stored as columns of argument i, rows of argument j
              for (int ci = 0; ci < tdi; ++ci) {
                const int32_t start = *cs++;
                for (int rr = 0; rr < tdj; ++rr) emit_h(start + rr, o + ci * tdj + rr);
              }
            }
          }
          o += tdi * tdj;
        }
      }
    }
  };
  // one list per entry: hessian_lower's, then the rhs's
  const int64_t ne = nnz + N;
  std::vector<int32_t> ptr(ne + 1, 0);
  replay([&](int64_t e, int64_t) { ++ptr[e + 1]; }, [&](int64_t e, int64_t) { ++ptr[nnz + e + 1]; });
  for (int64_t e = 0; e < ne; ++e) ptr[e + 1] += ptr[e];
  std::vector<int32_t> idx(std::max(1, ptr[ne]));
  {
    std::vector<int32_t> fill(ptr.begin(), ptr.end() - 1);
    replay([&](int64_t e, int64_t q) { idx[fill[e]++] = (int32_t)q; },
           [&](int64_t e, int64_t q) { idx[fill[nnz + e]++] = (int32_t)q; });
  }
  std::vector<int32_t> group, wide;
  for (int64_t e = 0; e < ne; ++e) {
    const int32_t len = ptr[e + 1] - ptr[e];
    if (len > kGroupList) wide.push_back((int32_t)e);
    else if (len > kThreadList) group.push_back((int32_t)e);
  }
  n_group_ = (int32_t)group.size();
  n_wide_ = (int32_t)wide.size();
  ptr_.upload(ptr, s);
  idx_.upload(idx, s);
  group_.upload(group, s);
  wide_.upload(wide, s);
  HIP_OK(hipStreamSynchronize(s));
}

void CscLinearizer::run(const double* values, double* residual, double* hval, double* rhs,
                        hipStream_t s) const {
  const bool sums = hval || rhs;
  for (const FactorGroup& g : groups_) {
    const int block = 128;
    const int grid = (g.n + block - 1) / block;
    dispatch_factor_type(g.type, [&]<int C>() {
      hipLaunchKernelGGL(lin_local_kernel<C>, dim3(grid), dim3(block), 0, s, g.n,
                         g.arg_off.get(), g.res_off.get(), values, residual,
                         sums ? contrib_.get() + g.contrib_off : static_cast<double*>(nullptr));
    });
    HIP_OK(hipGetLastError());
  }
  const int64_t ne = nnz + N;
  if (sums && ne > 0) {
    const int tb = grid_for(ne, 256), gb = grid_for(n_group_, 256 / kGroup);
    hipLaunchKernelGGL(gather_sum_kernel, dim3(tb + gb + n_wide_), dim3(256), 0, s, nnz, ne,
                       ptr_.get(), idx_.get(), group_.get(), n_group_, wide_.get(), tb, gb,
                       contrib_.get(), hval, rhs);
    HIP_OK(hipGetLastError());
  }
}

}  // namespace symhip
