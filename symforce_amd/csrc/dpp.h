// Cross-lane reads inside rows of 16 lanes, and the reciprocal of the elimination sweeps.
#pragma once

#include <hip/hip_runtime.h>

namespace symhip {

// llvm.amdgcn.update.dpp on a 64-bit value (one v_mov_b64_dpp; clang's builtin takes 32-bit values
// only, two instructions and two registers apart). The compiler keeps the wait states a DPP read of
// a just-written register needs. Device code only.
__device__ double dpp_update_f64(double old, double src, int ctrl, int row_mask, int bank_mask,
                                 bool bound_ctrl) __asm("llvm.amdgcn.update.dpp.f64");

// The value lane N of this lane's row of 16 holds (row_newbcast: four rows, four values at once).
// One vector instruction and no scalar register, where v_readlane needs two instructions per value
// and gives the whole wavefront the same one. All lanes of the row must be active.
template <int N>
__device__ __forceinline__ double row_bcast(double v) {
  static_assert(N >= 0 && N < 16, "a row has 16 lanes");
  return dpp_update_f64(v, v, 0x150 + N, 0xf, 0xf, true);
}

// acc[i] += row_bcast<N0 + i>(w) * f for i < kCount (1..6): v_fmac_f64 with the broadcast as its
// first operand, one instruction each (the compiler leaves the broadcast a separate move). The
// block starts with the two wait states between a vector write of w and its DPP read, which the
// compiler does not see from outside; w and f are not written inside it.
template <int N0, int kCount>
__device__ __forceinline__ void row_fmac(double* acc, double w, double f) {
  static_assert(kCount >= 0 && kCount <= 6 && N0 >= 0 && N0 + kCount <= 16, "lanes of a row");
#define SYMHIP_FMAC(a, n) \
  "v_fmac_f64_dpp %" #a ", %[w], %[f] row_newbcast:%[" #n "] row_mask:0xf bank_mask:0xf\n\t"
  if constexpr (kCount == 1) {
    asm("s_nop 1\n\t" SYMHIP_FMAC(0, n0) : "+v"(acc[0]) : [w] "v"(w), [f] "v"(f), [n0] "n"(N0));
  } else if constexpr (kCount == 2) {
    asm("s_nop 1\n\t" SYMHIP_FMAC(0, n0) SYMHIP_FMAC(1, n1)
        : "+v"(acc[0]), "+v"(acc[1])
        : [w] "v"(w), [f] "v"(f), [n0] "n"(N0), [n1] "n"(N0 + 1));
  } else if constexpr (kCount == 3) {
    asm("s_nop 1\n\t" SYMHIP_FMAC(0, n0) SYMHIP_FMAC(1, n1) SYMHIP_FMAC(2, n2)
        : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2])
        : [w] "v"(w), [f] "v"(f), [n0] "n"(N0), [n1] "n"(N0 + 1), [n2] "n"(N0 + 2));
  } else if constexpr (kCount == 4) {
    asm("s_nop 1\n\t" SYMHIP_FMAC(0, n0) SYMHIP_FMAC(1, n1) SYMHIP_FMAC(2, n2) SYMHIP_FMAC(3, n3)
        : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3])
        : [w] "v"(w), [f] "v"(f), [n0] "n"(N0), [n1] "n"(N0 + 1), [n2] "n"(N0 + 2),
          [n3] "n"(N0 + 3));
  } else if constexpr (kCount == 5) {
    asm("s_nop 1\n\t" SYMHIP_FMAC(0, n0) SYMHIP_FMAC(1, n1) SYMHIP_FMAC(2, n2) SYMHIP_FMAC(3, n3)
            SYMHIP_FMAC(4, n4)
        : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]), "+v"(acc[4])
        : [w] "v"(w), [f] "v"(f), [n0] "n"(N0), [n1] "n"(N0 + 1), [n2] "n"(N0 + 2),
          [n3] "n"(N0 + 3), [n4] "n"(N0 + 4));
  } else if constexpr (kCount == 6) {
    asm("s_nop 1\n\t" SYMHIP_FMAC(0, n0) SYMHIP_FMAC(1, n1) SYMHIP_FMAC(2, n2) SYMHIP_FMAC(3, n3)
            SYMHIP_FMAC(4, n4) SYMHIP_FMAC(5, n5)
        : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]), "+v"(acc[4]), "+v"(acc[5])
        : [w] "v"(w), [f] "v"(f), [n0] "n"(N0), [n1] "n"(N0 + 1), [n2] "n"(N0 + 2),
          [n3] "n"(N0 + 3), [n4] "n"(N0 + 4), [n5] "n"(N0 + 5));
  }
#undef SYMHIP_FMAC
}

// x + (x of lane ^ 32) and x + (x of lane ^ 16): the half / row swaps of gfx950 put either side in
// a register of its own, vector instructions where an LDS-based shuffle takes a round trip.
__device__ __forceinline__ double xor32_sum(double x) {
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  const u2 v = __builtin_bit_cast(u2, x);
  const auto lo = __builtin_amdgcn_permlane32_swap(v.x, v.x, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(v.y, v.y, false, false);
  return __builtin_bit_cast(double, u2{lo[0], hi[0]}) + __builtin_bit_cast(double, u2{lo[1], hi[1]});
}
__device__ __forceinline__ double xor16_sum(double x) {
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  const u2 v = __builtin_bit_cast(u2, x);
  const auto lo = __builtin_amdgcn_permlane16_swap(v.x, v.x, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(v.y, v.y, false, false);
  return __builtin_bit_cast(double, u2{lo[0], hi[0]}) + __builtin_bit_cast(double, u2{lo[1], hi[1]});
}

// 1 / d by the hardware estimate (2^-24) and one third-order step, r + r (e + e^2) with e = 1 - d r:
// three dependent operations to the same last bit as two Newton steps' four (both within half an
// ulp of the exact reciprocal in 4e6 samples); the IEEE division sequence is twice as long, and
// these sit on the elimination sweeps' critical paths.
__device__ __forceinline__ double refined_rcp(double d) {
  const double r = __builtin_amdgcn_rcp(d);
  const double e = fma(-d, r, 1.0);
  return fma(r, fma(e, e, e), r);
}

}  // namespace symhip
