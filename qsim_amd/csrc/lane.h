// lane.h -- gate passes with a group per lane and no LDS: geometry, member
// addresses and the swaps between lane bits and register bits.  Used by the
// vector kernel (gate_kernels.hip) and the k = 4 MFMA kernel
// (mfma_kernels.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "internal.h"

namespace qhip {

template <int K>
__device__ __forceinline__ uint64_t MemberOffset(unsigned j,
                                                 const uint64_t* tbit) {
  uint64_t o = 0;
#pragma unroll
  for (int b = 0; b < K; ++b) o += ((j >> b) & 1) ? tbit[b] : 0;
  return o;
}

// Geometry of the lane kernels.  A wave's chunk is 2^(6+K) amplitudes.  Lane
// bit i is qubit lane[i]: the six lowest qubits, passing over controls that
// can be skipped.  Register bit j is the amplitude offset roff[j]: first,
// one per target among the lane qubits, the lowest qubits that are neither
// lane, target nor control; then the other targets, ascending.  Chunk c
// starts at c << low (the lane qubits 0 .. low - 1) with zero bits inserted
// at ins[0..nins) (every other lane qubit, register bit and control,
// ascending) OR cbits.
struct LaneGeom {
  uint64_t nchunks;
  uint64_t cbits;
  uint64_t roff[6];
  unsigned low;
  unsigned nins;
  unsigned ins[kMaxInserted];
  unsigned lane[6];
  unsigned nlow;        // targets among the lane qubits: bits lbit[0..nlow)
  unsigned lbit[6];
  unsigned cmask;       // controls among the lane bits
  unsigned cvals;
};

// This workgroup's place.  Workgroups go to the XCDs in turn; taken in order,
// an XCD's waves in flight lie eight workgroups apart in every member's run,
// and with the members at large powers of two they meet few HBM channels: 29
// qubits, complex64 k = 4, targets 19..22 2.46 ms, 23..26 1.53.  FAR: an XCD
// takes runs of 32 consecutive workgroups instead (1.60 and 1.56), where
// LaneFar says so.
template <bool FAR>
__device__ __forceinline__ uint64_t LaneBlock() {
  constexpr unsigned kRun = 32;
  const unsigned b = blockIdx.x;
  if (!FAR || gridDim.x % (8u * kRun) != 0) return b;
  const unsigned q = b / (8u * kRun), r = b % (8u * kRun);
  return kRun * (8u * q + (r & 7u)) + (r >> 3);
}

// The value of lane ^ 2^B, B < 4: cross-lane moves within rows of 16.
template <int B>
__device__ __forceinline__ unsigned PullLane(unsigned v) {
  static_assert(B < 4, "row of 16 lanes");
  // quad_perm [1,0,3,2] and [2,3,0,1]; half mirror (^ 7) after quad_perm
  // [3,2,1,0] (^ 3); rotation by 8.
  constexpr int kCtrl[4] = {0xB1, 0x4E, 0x141, 0x128};
  if (B == 2) v = __builtin_amdgcn_update_dpp(0, v, 0x1B, 0xf, 0xf, true);
  return __builtin_amdgcn_update_dpp(0, v, kCtrl[B], 0xf, 0xf, true);
}

// Swaps lane bit B of `lo` with the register bit that tells `lo` from `up`:
// the lanes of `lo` with bit B set trade places with the lanes of `up`
// without it (lane ^ 2^B).  Lane bits 5 and 4 are one instruction; the
// others move within a row, without ds_bpermute's latency and registers (28
// qubits, k = 3, 4 with 2-4 low targets: 1-3 % less).
template <int B>
__device__ __forceinline__ void TradeLanes(unsigned& lo, unsigned& up) {
  if constexpr (B == 5) {
    const auto r = __builtin_amdgcn_permlane32_swap(lo, up, false, false);
    lo = r[0];
    up = r[1];
  } else if constexpr (B == 4) {
    const auto r = __builtin_amdgcn_permlane16_swap(lo, up, false, false);
    lo = r[0];
    up = r[1];
  } else {
    const bool hi = (threadIdx.x >> B) & 1u;
    const unsigned x = PullLane<B>(hi ? lo : up);
    lo = hi ? x : lo;
    up = hi ? up : x;
  }
}
template <int B>
__device__ __forceinline__ void TradeLanes(float& lo, float& up) {
  unsigned a = __builtin_bit_cast(unsigned, lo);
  unsigned b = __builtin_bit_cast(unsigned, up);
  TradeLanes<B>(a, b);
  lo = __builtin_bit_cast(float, a);
  up = __builtin_bit_cast(float, b);
}
template <int B>
__device__ __forceinline__ void TradeLanes(double& lo, double& up) {
  uint64_t a = __builtin_bit_cast(uint64_t, lo);
  uint64_t b = __builtin_bit_cast(uint64_t, up);
  unsigned a0 = unsigned(a), a1 = unsigned(a >> 32);
  unsigned b0 = unsigned(b), b1 = unsigned(b >> 32);
  TradeLanes<B>(a0, b0);
  TradeLanes<B>(a1, b1);
  a = a0 | (uint64_t(a1) << 32);
  b = b0 | (uint64_t(b1) << 32);
  lo = __builtin_bit_cast(double, a);
  up = __builtin_bit_cast(double, b);
}

// Swaps lane bit B with register bit I of the 2^K values a lane holds.
template <int K, int I, int B, typename C>
__device__ __forceinline__ void SwapLaneBit(C (&v)[1 << K]) {
#pragma unroll
  for (int j = 0; j < (1 << K); ++j) {
    if ((j >> I) & 1) continue;
    TradeLanes<B>(v[j].x, v[j | (1 << I)].x);
    TradeLanes<B>(v[j].y, v[j | (1 << I)].y);
  }
}

template <int K, int I, typename C>
__device__ __forceinline__ void SwapLowTargets(C (&v)[1 << K],
                                               const LaneGeom& g) {
  if constexpr (I < K) {
    if (I < int(g.nlow)) {
      switch (g.lbit[I]) {
        case 0: SwapLaneBit<K, I, 0>(v); break;
        case 1: SwapLaneBit<K, I, 1>(v); break;
        case 2: SwapLaneBit<K, I, 2>(v); break;
        case 3: SwapLaneBit<K, I, 3>(v); break;
        case 4: SwapLaneBit<K, I, 4>(v); break;
        default: SwapLaneBit<K, I, 5>(v); break;
      }
      SwapLowTargets<K, I + 1>(v, g);
    }
  }
}

// Gates without targets in the lanes: k = 4 with members 4 MiB apart or more,
// and complex64 k = 2 with a control in the lanes.  Random sets of targets on
// 26-30 qubits, runs of 32 against workgroups in order: complex64 k = 4 2 %
// less on average, 38 % at most, 6 % more at worst; complex128 k = 4 3 %, 34 %,
// 8 %; complex64 k = 2 6 %, 31 %, 7 %.  With every set of k = 4 the worst is 16
// % more, and complex128 k <= 3 have 20 %.
template <typename FP, int K>
inline bool LaneFar(const LaneGeom& g) {
  if (g.nlow != 0) return false;
  if (K == 4) return g.roff[0] * 2 * sizeof(FP) >= uint64_t{1} << 22;
  return K == 2 && sizeof(FP) == 4 && g.cmask != 0;
}

// The lane kernels' geometry; false where the state is too small for it.
template <typename FP>
inline bool LaneGeometry(unsigned n, const unsigned* qs, unsigned k,
                  const unsigned* cqs, unsigned nc, uint64_t cvals,
                  LaneGeom& g) {
  constexpr unsigned kLineQubit = sizeof(FP) == 4 ? 3 : 2;
  uint64_t targets = 0, skipped = 0, kept = 0;  // kept: controls in the lanes
  uint64_t kept_bits = 0;
  g = LaneGeom{};
  for (unsigned b = 0; b < k; ++b) targets |= uint64_t{1} << qs[b];
  for (unsigned i = 0; i < nc; ++i) {
    const uint64_t bit = (cvals >> i) & 1;
    if (cqs[i] < kLineQubit) {
      kept |= uint64_t{1} << cqs[i];
      kept_bits |= bit << cqs[i];
    } else {
      skipped |= uint64_t{1} << cqs[i];
      g.cbits |= bit << cqs[i];
    }
  }
  const unsigned ns = unsigned(__builtin_popcountll(skipped));
  if (n < 6 + k + ns) return false;
  unsigned q = 0, nl = 0;
  uint64_t taken = skipped;
  for (; nl < 6; ++q) {
    if ((skipped >> q) & 1) continue;
    if ((targets >> q) & 1) g.lbit[g.nlow++] = nl;
    if ((kept >> q) & 1) {
      g.cmask |= 1u << nl;
      g.cvals |= unsigned((kept_bits >> q) & 1) << nl;
    }
    taken |= uint64_t{1} << q;
    g.lane[nl++] = q;
  }
  unsigned r = 0;
  for (unsigned o = q; r < g.nlow; ++o) {
    if (((targets | skipped) >> o) & 1) continue;
    taken |= uint64_t{1} << o;
    g.roff[r++] = uint64_t{1} << o;
  }
  for (unsigned b = g.nlow; b < k; ++b) {
    taken |= uint64_t{1} << qs[b];
    g.roff[r++] = uint64_t{1} << qs[b];
  }
  while (g.low < 6 && g.lane[g.low] == g.low) ++g.low;
  for (unsigned b = g.low; b < n; ++b)
    if ((taken >> b) & 1) g.ins[g.nins++] = b;
  g.nchunks = uint64_t{1} << (n - 6 - k - ns);
  return true;
}

}  // namespace qhip
