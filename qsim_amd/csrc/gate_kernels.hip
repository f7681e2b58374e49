// gate_kernels.hip -- k-qubit gate passes and <psi|U|psi> on gfx950.
//
// Three kernel families apply psi <- U psi on every 2^k-amplitude group
// (the operation of SimulatorCUDA::ApplyGate / ApplyControlledGate,
// lib/simulator_cuda.h:70-207; arithmetic as lib/simulator_basic.h:167-275):
//
//  * GateLaneKernel -- k <= 4, low targets or controls, states of at least
//    2^(6+k) amplitudes per control pattern.  A wave loads 2^k runs of 64
//    consecutive amplitudes; targets among the lane qubits move to register
//    bits by swaps across lanes.  No LDS, no barriers.
//  * GateRegKernel  -- all targets and controls at qubit >= 5 (not k = 4):
//    one group per work item, held in registers.
//  * GateTileKernel -- the rest (k = 5, 6 with a qubit below 5, small states,
//    far-apart k = 2 with a low control).  A workgroup stages a tile of 2^tb
//    amplitudes (the Lc lowest qubits, contiguous in memory, times the high
//    targets) in LDS with coalesced loads, applies the groups from LDS and
//    streams the tile back.
//
// The gate matrix (row-major, row/column bit j <-> qs[j]) travels by value in
// the kernel arguments when it fits in 2 KiB (scalar loads, uniform across the
// wave) and otherwise through a device buffer.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "internal.h"
#include "lane.h"
#include "reduce.h"
#include "tile.h"

namespace qhip {

namespace {

template <typename FP, int K>
struct MatVal {
  FP v[2 << (2 * K)];
  __device__ __forceinline__ FP operator()(int i) const { return v[i]; }
};

template <typename FP>
struct MatPtr {
  const FP* __restrict__ p;
  __device__ __forceinline__ FP operator()(int i) const { return p[i]; }
};

// Largest tile per element type: 64 KiB of LDS (2^13 complex64 or 2^12
// complex128).  Passes with k <= 5 use half of it unless the larger tile
// splits into fewer contiguous runs; k = 6 always uses it.
template <typename FP, int K>
constexpr unsigned TileBitsMax() {
  return sizeof(FP) == 4 ? 13u : 12u;
}

// out = U v for one group; writes row r through `store(r, value)`.
template <typename FP, int K, typename M, typename Store>
__device__ __forceinline__ void MatVec(const typename Cplx<FP>::T* v,
                                       const M& m, Store store) {
  using C = typename Cplx<FP>::T;
  constexpr int D = 1 << K;
  if constexpr (K <= 4) {
#pragma unroll
    for (int r = 0; r < D; ++r) {
      FP re = 0, im = 0;
#pragma unroll
      for (int c = 0; c < D; ++c) {
        const FP mr = m(2 * (r * D + c));
        const FP mi = m(2 * (r * D + c) + 1);
        re = fma(mr, v[c].x, re);
        re = fma(-mi, v[c].y, re);
        im = fma(mi, v[c].x, im);
        im = fma(mr, v[c].y, im);
      }
      store(r, C{re, im});
    }
  } else {
#pragma unroll 1
    for (int r = 0; r < D; ++r) {
      FP re = 0, im = 0;
#pragma unroll
      for (int c = 0; c < D; ++c) {
        const FP mr = m(2 * (r * D + c));
        const FP mi = m(2 * (r * D + c) + 1);
        re = fma(mr, v[c].x, re);
        re = fma(-mi, v[c].y, re);
        im = fma(mi, v[c].x, im);
        im = fma(mr, v[c].y, im);
      }
      store(r, C{re, im});
    }
  }
}

template <typename FP, int K, typename M>
__global__ void __launch_bounds__(256)
GateRegKernel(typename Cplx<FP>::T* __restrict__ s, GateGeom g, M m) {
  using C = typename Cplx<FP>::T;
  constexpr int D = 1 << K;
  const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
  for (uint64_t t = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
       t < g.ngroups; t += stride) {
    const uint64_t base = InsertZeros(t, g.ins, g.nins) | g.cbits;
    C v[D];
#pragma unroll
    for (int j = 0; j < D; ++j) v[j] = s[base + MemberOffset<K>(j, g.tbit)];
    MatVec<FP, K>(v, m, [&](int r, C val) {
      s[base + MemberOffset<K>(r, g.tbit)] = val;
    });
  }
}

template <int K>
__device__ __forceinline__ unsigned TileMemberOffset(unsigned j,
                                                     const unsigned* tpos) {
  unsigned o = 0;
#pragma unroll
  for (int b = 0; b < K; ++b) o |= ((j >> b) & 1u) << tpos[b];
  return o;
}

template <typename FP, int K, typename M>
__global__ void __launch_bounds__(256)
GateTileKernel(typename Cplx<FP>::T* __restrict__ s, TileGeom g, M m) {
  using C = typename Cplx<FP>::T;
  constexpr int D = 1 << K;
  extern __shared__ char lds_raw[];
  C* lds = reinterpret_cast<C*>(lds_raw);
  const unsigned T = 1u << g.tb;
  const unsigned ngroups = T >> K;
  constexpr int PER = (size_t{1} << TileBitsMax<FP, K>()) / 256;
  for (uint64_t tile = blockIdx.x; tile < g.ntiles; tile += gridDim.x) {
    const uint64_t base =
        InsertZeros(tile << g.Lc, g.outer, g.nouter) | g.cbits_high;
    TileLoad<PER>(s, base, g, lds);
    __syncthreads();
    for (unsigned gr = threadIdx.x; gr < ngroups; gr += 256) {
      unsigned tb0 = gr;
#pragma unroll
      for (int b = 0; b < K; ++b) {
        const unsigned p = g.tpos[b];
        tb0 = ((tb0 >> p) << (p + 1)) | (tb0 & ((1u << p) - 1));
      }
      if ((tb0 & g.low_cmask) != g.low_cvals) continue;
      C v[D];
#pragma unroll
      for (int j = 0; j < D; ++j)
        v[j] = lds[TileSwz(tb0 + TileMemberOffset<K>(j, g.tpos))];
      MatVec<FP, K>(v, m, [&](int r, C val) {
        lds[TileSwz(tb0 + TileMemberOffset<K>(r, g.tpos))] = val;
      });
    }
    __syncthreads();
    TileStore<PER>(s, base, g, lds);
    __syncthreads();
  }
}

// Any targets and controls, K <= 4, on states with 2^(6+K) amplitudes in the
// subspace of the skipped controls.  A wave's loads and stores are runs of
// consecutive amplitudes (64 of them unless a control is skipped below
// qubit 6); targets among the lane qubits are brought from lane bits into
// register bits, and back, by swaps across lanes, so that each lane holds
// whole groups in matrix order.  No LDS, no barriers.
//
// Bound by the HBM stream.  Complex128, 27 qubits, targets below qubit 6:
// k = 1..3 0.77-0.83 ms, k = 4 0.81-1.0 ms (the LDS tile kernel, half of
// whose threads have no group at these sizes: 1.8 and 2.3-2.5 ms); complex64,
// 28 qubits: k = 1..3 0.72-0.83 ms (0.78-0.87); 2^12 .. 2^20 amplitudes:
// 1-5 us less per pass, many short waves instead of a few large tiles.
//
// A control below kLineQubit (8 complex64 or 4 complex128 to a 64-byte
// half line) cannot skip memory: its lanes load and store too and keep
// their values; masked partial lines measured 7 % slower (28 qubits,
// control 0).  Controls above are skipped as any other high qubit.
template <typename FP, int K, bool FAR, typename M>
__global__ void __launch_bounds__(256)
GateLaneKernel(typename Cplx<FP>::T* __restrict__ s, LaneGeom g, M m) {
  using C = typename Cplx<FP>::T;
  constexpr int D = 1 << K;
  const unsigned lane = threadIdx.x & 63;
  const bool active = (lane & g.cmask) == g.cvals;
  uint64_t loff = 0;
#pragma unroll
  for (int b = 0; b < 6; ++b) loff += uint64_t((lane >> b) & 1u) << g.lane[b];
  const uint64_t stride = uint64_t(gridDim.x) * 4;
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (uint64_t c = LaneBlock<FAR>() * 4 + wave; c < g.nchunks; c += stride) {
    C* p = s + (InsertZeros(c << g.low, g.ins, g.nins) | g.cbits);
    C v[D], u[D];
#pragma unroll
    for (int j = 0; j < D; ++j) v[j] = p[MemberOffset<K>(j, g.roff) + loff];
    SwapLowTargets<K, 0>(v, g);
    MatVec<FP, K>(v, m, [&](int r, C val) {
      u[r].x = active ? val.x : v[r].x;
      u[r].y = active ? val.y : v[r].y;
    });
    SwapLowTargets<K, 0>(u, g);
#pragma unroll
    for (int j = 0; j < D; ++j) p[MemberOffset<K>(j, g.roff) + loff] = u[j];
  }
}

// <psi|U|psi>; products in FP, sums in FP64 (lib/simulator_basic.h:316-317).
template <typename C>
__device__ __forceinline__ void AddExpectation(Dbl2& acc, const C& v,
                                               const C& u) {
  // conj(v) * u
  acc.x += double(v.x * u.x + v.y * u.y);
  acc.y += double(v.x * u.y - v.y * u.x);
}

// The gate kernels' read side (GateLaneKernel): runs of 64 amplitudes, low
// targets swapped into registers; bound by the read.  LaunchExpect says where
// it beats ExpectationKernel.
template <typename FP, int K, typename M>
__global__ void __launch_bounds__(256)
ExpectationLaneKernel(const typename Cplx<FP>::T* __restrict__ s, LaneGeom g,
                      M m, Dbl2* __restrict__ partials) {
  using C = typename Cplx<FP>::T;
  constexpr int D = 1 << K;
  const unsigned lane = threadIdx.x & 63;
  const uint64_t stride = uint64_t(gridDim.x) * 4;
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  Dbl2 acc;
  for (uint64_t c = uint64_t(blockIdx.x) * 4 + wave; c < g.nchunks;
       c += stride) {
    const C* p = s + InsertZeros(c << 6, g.ins, g.nins);
    C v[D];
#pragma unroll
    for (int j = 0; j < D; ++j) v[j] = p[MemberOffset<K>(j, g.roff) + lane];
    SwapLowTargets<K, 0>(v, g);
    MatVec<FP, K>(v, m, [&](int r, C u) { AddExpectation(acc, v[r], u); });
  }
  acc = BlockSum<256>(acc);
  if (threadIdx.x == 0) partials[blockIdx.x] = acc;
}

// Any sizes, one group per work item; the members come through the caches.
template <typename FP, int K, typename M>
__global__ void __launch_bounds__(256)
ExpectationKernel(const typename Cplx<FP>::T* __restrict__ s, GateGeom g, M m,
                  Dbl2* __restrict__ partials) {
  using C = typename Cplx<FP>::T;
  constexpr int D = 1 << K;
  Dbl2 acc;
  const uint64_t stride = uint64_t(gridDim.x) * blockDim.x;
  for (uint64_t t = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
       t < g.ngroups; t += stride) {
    const uint64_t base = InsertZeros(t, g.ins, g.nins);
    C v[D];
#pragma unroll
    for (int j = 0; j < D; ++j) v[j] = s[base + MemberOffset<K>(j, g.tbit)];
    MatVec<FP, K>(v, m, [&](int r, C u) { AddExpectation(acc, v[r], u); });
  }
  acc = BlockSum<256>(acc);
  if (threadIdx.x == 0) partials[blockIdx.x] = acc;
}

// ---- host side -------------------------------------------------------------

uint64_t Deposit(uint64_t v, uint64_t mask) {
  uint64_t r = 0;
  for (unsigned i = 0; i < 64; ++i) {
    if ((mask >> i) & 1) {
      r |= (v & 1) << i;
      v >>= 1;
    }
  }
  return r;
}

int CheckQubits(unsigned n, const unsigned* qs, unsigned k, const unsigned* cqs,
                unsigned nc) {
  for (unsigned i = 0; i < k; ++i) {
    if (qs[i] >= n || (i > 0 && qs[i] <= qs[i - 1])) {
      SetError("target qubits must be ascending, distinct and < %u", n);
      return QSIM_HIP_ERR_ARG;
    }
  }
  for (unsigned i = 0; i < nc; ++i) {
    if (cqs[i] >= n || (i > 0 && cqs[i] <= cqs[i - 1])) {
      SetError("control qubits must be ascending, distinct and < %u", n);
      return QSIM_HIP_ERR_ARG;
    }
    for (unsigned j = 0; j < k; ++j) {
      if (cqs[i] == qs[j]) {
        SetError("qubit %u is both target and control", cqs[i]);
        return QSIM_HIP_ERR_ARG;
      }
    }
  }
  if (k + nc > kMaxInserted) {
    SetError("too many gate qubits (%u)", k + nc);
    return QSIM_HIP_ERR_UNSUPPORTED;
  }
  return QSIM_HIP_OK;
}

template <typename FP, int K>
constexpr bool kByValue = sizeof(FP) * (2u << (2 * K)) <= 2048;



template <typename FP, int K, typename M>
int LaunchReg(typename Cplx<FP>::T* s, const GateGeom& g, const M& m) {
  uint64_t blocks = (g.ngroups + 255) / 256;
  blocks = std::min<uint64_t>(std::max<uint64_t>(blocks, 1), uint64_t{1} << 20);
  PassTimerBegin();
  hipLaunchKernelGGL((GateRegKernel<FP, K, M>), dim3(unsigned(blocks)),
                     dim3(256), 0, Stream(), s, g, m);
  PassTimerEnd();
  QHIP_LAUNCHED("GateRegKernel");
  return QSIM_HIP_OK;
}

template <typename FP, int K, typename M>
int LaunchTile(typename Cplx<FP>::T* s, const TileGeom& g, const M& m) {
  using C = typename Cplx<FP>::T;
  size_t lds = (size_t{1} << g.tb) * sizeof(C);
  if (lds > 65536) {
    SetError("tile of %zu bytes exceeds the 64 KiB LDS budget", lds);
    return QSIM_HIP_ERR_RUNTIME;
  }
  uint64_t blocks = std::min<uint64_t>(g.ntiles, uint64_t{1} << 20);
  PassTimerBegin();
  hipLaunchKernelGGL((GateTileKernel<FP, K, M>), dim3(unsigned(blocks)),
                     dim3(256), lds, Stream(), s, g, m);
  PassTimerEnd();
  QHIP_LAUNCHED("GateTileKernel");
  return QSIM_HIP_OK;
}


template <typename FP, int K, typename M>
int LaunchLane(typename Cplx<FP>::T* s, const LaneGeom& g, const M& m) {
  const uint64_t blocks =
      std::min<uint64_t>((g.nchunks + 3) / 4, uint64_t{1} << 20);
  PassTimerBegin();
  // Only what LaneFar can answer with true.
  constexpr bool far = K == 4 || (K == 2 && sizeof(FP) == 4);
  if (far && LaneFar<FP, K>(g))
    hipLaunchKernelGGL((GateLaneKernel<FP, K, far, M>), dim3(unsigned(blocks)),
                       dim3(256), 0, Stream(), s, g, m);
  else
    hipLaunchKernelGGL((GateLaneKernel<FP, K, false, M>),
                       dim3(unsigned(blocks)), dim3(256), 0, Stream(), s, g, m);
  PassTimerEnd();
  QHIP_LAUNCHED("GateLaneKernel");
  return QSIM_HIP_OK;
}

template <typename FP, int K>
int DispatchK(typename Cplx<FP>::T* s, unsigned n, const unsigned* qs,
              const unsigned* cqs, unsigned nc, uint64_t cvals, const FP* m) {
  // Lowest qubit the pass touches decides the kernel family.
  unsigned lowest = 64;
  if (K > 0) lowest = std::min(lowest, qs[0]);
  if (nc > 0) lowest = std::min(lowest, cqs[0]);

  MatVal<FP, K> mv;
  MatPtr<FP> mp{nullptr};
  constexpr bool byval = kByValue<FP, K>;
  if constexpr (byval) {
    std::memcpy(mv.v, m, sizeof(mv.v));
  } else {
    size_t bytes = sizeof(FP) * (size_t{2} << (2 * K));
    void* d = MatrixBuffer(bytes);
    if (d == nullptr) return QSIM_HIP_ERR_OOM;
    QHIP_TRY(StageMatrix(d, m, bytes));
    mp.p = static_cast<const FP*>(d);
  }

  if constexpr (K <= 4) {
    // Nothing to bring into the lanes (no target or control below qubit 5):
    // GateRegKernel, up to k = 3.  Against the lane kernel, complex64 k = 2
    // 28 qubits, highest targets 803 us : 853, k = 3 20 qubits 8.2 : 8.9;
    // complex128 k = 3 20 qubits 12.1 : 13.8, 29 qubits 3231 : 3340; equal
    // for k = 1.  With controls, complex128 is 2-5 % better on the lanes (27
    // qubits 191-210 : 187-198), and k = 4 too (20 qubits 26 : 16).
    const bool reg = lowest >= 5 && K <= 3 && (nc == 0 || sizeof(FP) == 4);
    // complex64 k = 2 with a control below a half line and both targets from
    // qubit 14 up stays on the tile kernel, whose runs are of 2^11 amplitudes,
    // from 28 qubits: there the lane kernel takes 0.89-1.21 times its time on
    // random sets, 1.04 on average (27 qubits 0.90-1.14, 0.99; with a target
    // below 14 0.76-1.02, 0.89).  Not with controls inside the tile's run
    // that the lane kernel skips (twice the traffic).
    bool tile = K == 2 && sizeof(FP) == 4 && n >= 28 && nc > 0 &&
                cqs[0] < 3 && qs[0] >= 14;
    for (unsigned i = 0; i < nc; ++i)
      tile = tile && (cqs[i] < 3 || cqs[i] >= 13);
    LaneGeom lg;
    if (!reg && !tile && LaneGeometry<FP>(n, qs, K, cqs, nc, cvals, lg)) {
      if constexpr (byval) return LaunchLane<FP, K>(s, lg, mv);
      else return LaunchLane<FP, K>(s, lg, mp);
    }
  }

  if (lowest >= 5 || n < 5) {
    GateGeom g{};
    std::vector<unsigned> ins(qs, qs + K);
    ins.insert(ins.end(), cqs, cqs + nc);
    std::sort(ins.begin(), ins.end());
    g.nins = ins.size();
    for (unsigned i = 0; i < g.nins; ++i) g.ins[i] = ins[i];
    uint64_t cmask = 0;
    for (unsigned i = 0; i < nc; ++i) cmask |= uint64_t{1} << cqs[i];
    g.cbits = Deposit(cvals, cmask);
    for (int b = 0; b < K; ++b) g.tbit[b] = uint64_t{1} << qs[b];
    g.ngroups = uint64_t{1} << (n - K - nc);
    if constexpr (byval) return LaunchReg<FP, K>(s, g, mv);
    else return LaunchReg<FP, K>(s, g, mp);
  }

  // Tile geometry: find tb <= n, h with h = #targets >= tb - h, and enough
  // outer bits left for the high controls.  The tile is 2^h contiguous runs;
  // the larger tile (64 KiB) is taken when it leaves fewer runs, or for k = 6.
  TileGeom g{};
  auto fit = [&](unsigned TB, unsigned* hout, unsigned* lcout,
                 unsigned* tbout) {
    for (;;) {
      unsigned h = 0, Lc = TB;
      for (unsigned hh = 0; hh <= unsigned(K); ++hh) {
        if (hh > TB) break;
        unsigned lc = TB - hh;
        unsigned cnt = 0;
        for (int b = 0; b < K; ++b) cnt += qs[b] >= lc;
        if (cnt == hh) {
          h = hh;
          Lc = lc;
          break;
        }
      }
      unsigned hc = 0;
      for (unsigned i = 0; i < nc; ++i) hc += cqs[i] >= Lc;
      if (n >= TB + hc) {
        *hout = h;
        *lcout = Lc;
        *tbout = TB;
        return;
      }
      --TB;
    }
  };
  const unsigned small_tb = TileBitsMax<FP, K>() - (K >= 6 ? 0u : 1u);
  fit(std::min(small_tb, n), &g.h, &g.Lc, &g.tb);
  if (K < 6 && n > small_tb) {
    unsigned h2, lc2, tb2;
    fit(std::min(TileBitsMax<FP, K>(), n), &h2, &lc2, &tb2);
    if (h2 < g.h) {
      g.h = h2;
      g.Lc = lc2;
      g.tb = tb2;
    }
  }
  std::vector<unsigned> outer;
  unsigned hi = 0;
  for (int b = 0; b < K; ++b) {
    if (qs[b] >= g.Lc) {
      g.hbit[hi] = uint64_t{1} << qs[b];
      g.tpos[b] = g.Lc + hi;
      ++hi;
      outer.push_back(qs[b]);
    } else {
      g.tpos[b] = qs[b];
    }
  }
  uint64_t cmask_high = 0;
  unsigned low_cmask = 0;
  uint64_t cvals_high = 0, cvals_low = 0;
  {
    unsigned lo_i = 0, hi_i = 0;
    for (unsigned i = 0; i < nc; ++i) {
      uint64_t bit = (cvals >> i) & 1;
      if (cqs[i] >= g.Lc) {
        cmask_high |= uint64_t{1} << cqs[i];
        cvals_high |= bit << cqs[i];
        outer.push_back(cqs[i]);
        ++hi_i;
      } else {
        low_cmask |= 1u << cqs[i];
        cvals_low |= bit << cqs[i];
        ++lo_i;
      }
    }
    (void)lo_i;
    (void)hi_i;
  }
  std::sort(outer.begin(), outer.end());
  g.nouter = outer.size();
  for (unsigned i = 0; i < g.nouter; ++i) g.outer[i] = outer[i];
  g.cbits_high = cvals_high;
  g.low_cmask = low_cmask;
  g.low_cvals = unsigned(cvals_low);
  unsigned hc = 0;
  for (unsigned i = 0; i < nc; ++i) hc += cqs[i] >= g.Lc;
  // Every tile-local position must lie inside the tile and every amplitude
  // index inside the state; refuse to launch otherwise.
  bool ok = hi == g.h && g.tb == g.Lc + g.h && g.tb <= n && n >= g.tb + hc;
  for (int b = 0; b < K; ++b) ok = ok && g.tpos[b] < g.tb;
  for (int b = 1; b < K; ++b) ok = ok && g.tpos[b] > g.tpos[b - 1];
  if (!ok) {
    SetError("internal: inconsistent tile geometry (n=%u k=%d)", n, K);
    return QSIM_HIP_ERR_RUNTIME;
  }
  g.ntiles = uint64_t{1} << (n - g.tb - hc);
  if constexpr (byval) return LaunchTile<FP, K>(s, g, mv);
  else return LaunchTile<FP, K>(s, g, mp);
}

// Workgroups of an expectation pass: at most eight a CU of 256, or four
// (kExpectBlocksFew), which is better for ExpectationKernel and for
// complex128 k = 1 (27 qubits: 353-392 us against 372-408).
constexpr unsigned kExpectBlocks = 2048, kExpectBlocksFew = 1024;

static_assert(kExpectBlocks * sizeof(Dbl2) <= kHostResultBytes, "partials");

// Returns the number of partial sums, one per workgroup, in `partials`.
template <typename FP, int K, typename M>
unsigned LaunchExpect(const typename Cplx<FP>::T* s, unsigned n,
                  const unsigned* qs, const M& m, Dbl2* partials) {
  if constexpr (K != 2 && K <= (sizeof(FP) == 4 ? 3 : 4)) {
    // Where swapping low targets across lanes beats reading groups through the
    // caches (complex64 k = 4 is LaunchExpectationMfma's, here only with the
    // vector kernels asked for); calls on 27 qubits, lanes against groups (us):
    //   complex64   k = 1 183-197 : 225-234; k = 2 201-215 : 186-190;
    //               k = 3 215 : 237 without a target in the lanes, else
    //               245-286 : 236-245
    //   complex128  k = 1 353-392 : 359-397; k = 2 362-394 : 360-378; k = 3
    //               440 : 540 with 3 targets in the lanes, 420 : 395 with 2 (24
    //               qubits 66 : 59, 29 1621 : 1522), 391 : 392 with 1;
    //               k = 4 543 : 555 without, 593-673 : 555-629 with
    // The same choices are no more than 3 % behind on 12-30 qubits.
    constexpr bool f32 = sizeof(FP) == 4;
    LaneGeom lg;
    if (LaneGeometry<FP>(n, qs, K, nullptr, 0, 0, lg) &&
        (K < 3 || lg.nlow == (K == 3 && !f32 ? 3 : 0))) {
      const uint64_t blocks = std::min<uint64_t>(
          (lg.nchunks + 3) / 4,
          K == 1 && !f32 ? kExpectBlocksFew : kExpectBlocks);
      hipLaunchKernelGGL((ExpectationLaneKernel<FP, K, M>),
                         dim3(unsigned(blocks)), dim3(256), 0, Stream(), s, lg,
                         m, partials);
      return unsigned(blocks);
    }
  }
  GateGeom g{};
  g.nins = K;
  for (int b = 0; b < K; ++b) {
    g.ins[b] = qs[b];
    g.tbit[b] = uint64_t{1} << qs[b];
  }
  g.ngroups = uint64_t{1} << (n - K);
  const uint64_t blocks = std::max<uint64_t>(
      1, std::min<uint64_t>((g.ngroups + 255) / 256, kExpectBlocksFew));
  hipLaunchKernelGGL((ExpectationKernel<FP, K, M>), dim3(unsigned(blocks)),
                     dim3(256), 0, Stream(), s, g, m, partials);
  return unsigned(blocks);
}

template <typename FP, int K>
int DispatchExpectation(const typename Cplx<FP>::T* s, unsigned n,
                        const unsigned* qs, const FP* m, double* re,
                        double* im) {
  std::lock_guard<std::mutex> lock(ScratchLock());
  Dbl2* partials = static_cast<Dbl2*>(HostResult());
  unsigned count = 0;
  int rc = QSIM_HIP_ERR_UNSUPPORTED;
  if constexpr (K == 4 && sizeof(FP) == 4) {
    if (qsim_hip_get_gate_method() != QSIM_HIP_METHOD_VECTOR) {
      rc = LaunchExpectationMfma(s, n, qs, m, partials, kExpectBlocks, &count);
      if (rc != QSIM_HIP_OK && rc != QSIM_HIP_ERR_UNSUPPORTED) return rc;
    }
  }
  if (rc != QSIM_HIP_OK) {
    if constexpr (kByValue<FP, K>) {
      MatVal<FP, K> mv;
      std::memcpy(mv.v, m, sizeof(mv.v));
      count = LaunchExpect<FP, K>(s, n, qs, mv, partials);
    } else {
      size_t bytes = sizeof(FP) * (size_t{2} << (2 * K));
      void* d = MatrixBuffer(bytes);
      if (d == nullptr) return QSIM_HIP_ERR_OOM;
      QHIP_TRY(StageMatrix(d, m, bytes));
      MatPtr<FP> mp{static_cast<const FP*>(d)};
      count = LaunchExpect<FP, K>(s, n, qs, mp, partials);
    }
  }
  QHIP_LAUNCHED("expectation kernel");
  Dbl2 r;
  QHIP_TRY(HostTotal(count, &r));
  *re = r.x;
  *im = r.y;
  return QSIM_HIP_OK;
}

}  // namespace

template <typename FP>
int LaunchGate(typename Cplx<FP>::T* s, unsigned n, const unsigned* qs,
               unsigned k, const unsigned* cqs, unsigned nc, uint64_t cvals,
               const FP* m) {
  if (k > 6) {
    SetError("gates on %u > 6 qubits are not supported", k);
    return QSIM_HIP_ERR_UNSUPPORTED;
  }
  if (k + nc > n) {
    SetError("gate on %u qubits does not fit a %u-qubit state", k + nc, n);
    return QSIM_HIP_ERR_ARG;
  }
  QHIP_TRY(CheckQubits(n, qs, k, cqs, nc));
  if constexpr (sizeof(FP) == 8) {
    if (k >= 5 && nc == 0 &&
        qsim_hip_get_gate_method() != QSIM_HIP_METHOD_VECTOR) {
      const int rc = LaunchGateF64(s, n, qs, k, m);
      if (rc != QSIM_HIP_ERR_UNSUPPORTED) return rc;
    }
  }
  switch (k) {
    case 0: return DispatchK<FP, 0>(s, n, qs, cqs, nc, cvals, m);
    case 1: return DispatchK<FP, 1>(s, n, qs, cqs, nc, cvals, m);
    case 2: return DispatchK<FP, 2>(s, n, qs, cqs, nc, cvals, m);
    case 3: return DispatchK<FP, 3>(s, n, qs, cqs, nc, cvals, m);
    case 4: return DispatchK<FP, 4>(s, n, qs, cqs, nc, cvals, m);
    case 5: return DispatchK<FP, 5>(s, n, qs, cqs, nc, cvals, m);
    default: return DispatchK<FP, 6>(s, n, qs, cqs, nc, cvals, m);
  }
}

template <typename FP>
int LaunchExpectation(const typename Cplx<FP>::T* s, unsigned n,
                      const unsigned* qs, unsigned k, const FP* m, double* re,
                      double* im) {
  if (k == 0 || k > 6) {
    SetError("expectation values need 1..6 qubits (got %u)", k);
    return QSIM_HIP_ERR_UNSUPPORTED;
  }
  if (k > n) {
    SetError("operator on %u qubits does not fit a %u-qubit state", k, n);
    return QSIM_HIP_ERR_ARG;
  }
  QHIP_TRY(CheckQubits(n, qs, k, nullptr, 0));
  switch (k) {
    case 1: return DispatchExpectation<FP, 1>(s, n, qs, m, re, im);
    case 2: return DispatchExpectation<FP, 2>(s, n, qs, m, re, im);
    case 3: return DispatchExpectation<FP, 3>(s, n, qs, m, re, im);
    case 4: return DispatchExpectation<FP, 4>(s, n, qs, m, re, im);
    case 5: return DispatchExpectation<FP, 5>(s, n, qs, m, re, im);
    default: return DispatchExpectation<FP, 6>(s, n, qs, m, re, im);
  }
}

template int LaunchGate<float>(float2*, unsigned, const unsigned*, unsigned,
                               const unsigned*, unsigned, uint64_t,
                               const float*);
template int LaunchGate<double>(double2*, unsigned, const unsigned*, unsigned,
                                const unsigned*, unsigned, uint64_t,
                                const double*);
template int LaunchExpectation<float>(const float2*, unsigned, const unsigned*,
                                      unsigned, const float*, double*,
                                      double*);
template int LaunchExpectation<double>(const double2*, unsigned,
                                       const unsigned*, unsigned,
                                       const double*, double*, double*);

}  // namespace qhip
