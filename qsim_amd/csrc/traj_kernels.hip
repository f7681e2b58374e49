// traj_kernels.hip -- batched noisy trajectories.
//
// qsim's trajectory simulator (lib/qtrajectory.h:112-387) runs trajectories
// one after another, each gate batch as its own set of kernel launches with a
// host synchronisation at every channel whose Kraus operator depends on the
// state.  Here a whole batch -- hundreds of trajectories of uneven qubit
// counts, their states in a device pool -- runs at once.  The per-gate kernels
// are ONE launch: workgroup t owns trajectory t and walks its operation stream
// with nothing but workgroup barriers between operations.  The tiled batch is
// one launch per step of the streams, over pieces of all trajectories.  The
// operations:
//
//   gate      a fused gate (k <= 4, FP32 matrix in LDS) over all 2^(n-k)
//             groups of the trajectory's state;
//   tile pass a run of gates applied tile by tile through LDS with the
//             FP16 MFMA product of the circuit kernel's blocked passes (the
//             tiled batch; the per-gate kernels run the gates one by one);
//   channel   a channel whose draw fell past the probability bounds: FP64
//             sweeps for <psi|K^dagger K|psi> operator by operator (the
//             first also giving the norm), the choice exactly as
//             RunIteration makes it (lib/qtrajectory.h:330-370), then the
//             chosen operator applied (scaled to the normalised state where
//             the trajectory is not unitary).
//
// The Kraus operators that the bounds decide (depolarising Paulis, damping
// K0 when the draw is below its bound, any unitary operator whose
// cumulative bound covers the draw) are sampled on the host from the same
// mt19937(rep) draws and folded into the fused gates.  At the end each
// trajectory writes <Z_a Z_b> of its qubit pairs, FP64-accumulated and
// divided by the norm (the normalisation of lib/qtrajectory.h:377-383).
//
// Workgroups are dispatched in order, so the host puts the largest states and
// items first (longest-processing-time-first balancing across CUs).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <memory>
#include <atomic>
#include <cmath>
#include <cstring>
#include <mutex>
#include <new>
#include <string>
#include <system_error>
#include <thread>
#include <type_traits>
#include <unordered_map>
#include <vector>

#include "block_tile.h"
#include "internal.h"
#include "lane.h"
#include "reduce.h"

namespace qhip {

namespace {

using namespace tileop;

// Pairs per <Z_a Z_b> sweep (FP64 accumulators per thread: 32 would not fit
// beside the step's registers) and amplitudes per thread per step of a
// whole-state sweep.
template <int NT>
constexpr unsigned kPairChunk = 16;
template <int NT>
constexpr unsigned kPairRed = (kPairChunk<NT> + 1) * (NT / 64);
template <int NT>
constexpr unsigned kSweep = NT <= 512 ? 16 : 8;

// Groups [lo, hi) of a gate.
template <int NT, int K>
__device__ void ApplyGateK(float2* __restrict__ s, const qsim_hip_traj_op& o,
                           const float* lm, uint64_t lo, uint64_t hi) {
  constexpr unsigned D = 1u << K;
  unsigned q[K];
#pragma unroll
  for (int b = 0; b < K; ++b) q[b] = o.q[b];
  for (uint64_t g = lo + threadIdx.x; g < hi; g += NT) {
    uint64_t base = g;
#pragma unroll
    for (int b = 0; b < K; ++b) {
      base = ((base >> q[b]) << (q[b] + 1)) | (base & ((uint64_t{1} << q[b]) - 1));
    }
    float2 v[D];
#pragma unroll
    for (unsigned j = 0; j < D; ++j) {
      uint64_t off = 0;
#pragma unroll
      for (int b = 0; b < K; ++b) off |= uint64_t((j >> b) & 1u) << q[b];
      v[j] = s[base + off];
    }
    // Rows stay a loop for k >= 3: unrolled, the compiler would hoist the
    // whole LDS matrix (2 D^2 floats) into registers across the group loop.
#pragma unroll(K <= 2 ? D : 1)
    for (unsigned r = 0; r < D; ++r) {
      float re = 0.0f, im = 0.0f;
#pragma unroll
      for (unsigned j = 0; j < D; ++j) {
        const float mr = lm[2 * (r * D + j)], mi = lm[2 * (r * D + j) + 1];
        re = fmaf(mr, v[j].x, re);
        re = fmaf(-mi, v[j].y, re);
        im = fmaf(mr, v[j].y, im);
        im = fmaf(mi, v[j].x, im);
      }
      uint64_t off = 0;
#pragma unroll
      for (int b = 0; b < K; ++b) off |= uint64_t((r >> b) & 1u) << q[b];
      s[base + off] = float2{re, im};
    }
  }
}

// LDS scratch of the reductions: NT / 64 wave partials, then two broadcast
// slots.
template <int NT>
constexpr unsigned kRedWords = NT / 64 + 2;

template <int NT>
__device__ void ZeroState(float2* __restrict__ s, uint64_t N) {
  for (uint64_t i = threadIdx.x; i < N; i += NT) {
    s[i] = float2{i == 0 ? 1.0f : 0.0f, 0.0f};
  }
}

// Groups [lo, hi) of a fused gate, its FP32 matrix staged in LDS (lm).
template <int NT>
__device__ void TrajGate(float2* __restrict__ s, const qsim_hip_traj_op& o,
                         const float* __restrict__ mats, float* lm,
                         uint64_t lo, uint64_t hi) {
  const unsigned D = 1u << o.k;
  for (unsigned i = threadIdx.x; i < 2 * D * D; i += NT) lm[i] = mats[o.moff + i];
  __syncthreads();
  switch (o.k) {
    case 1: ApplyGateK<NT, 1>(s, o, lm, lo, hi); break;
    case 2: ApplyGateK<NT, 2>(s, o, lm, lo, hi); break;
    case 3: ApplyGateK<NT, 3>(s, o, lm, lo, hi); break;
    default: ApplyGateK<NT, 4>(s, o, lm, lo, hi); break;
  }
  __syncthreads();
}

// Most Kraus operators of a channel decided on the device, and its most
// qubits.
constexpr unsigned kMaxKraus = 16;
constexpr unsigned kMaxChannelQubits = 2;

// Scales the state by a (a sweep).
template <int NT>
__device__ void ScaleState(float2* __restrict__ s, uint64_t N, float a) {
  for (uint64_t i = threadIdx.x; i < N; i += NT) {
    const float2 v = s[i];
    s[i] = float2{v.x * a, v.y * a};
  }
}

// The 2^NQ amplitudes of group g over ascending qubits q.
template <int NQ>
__device__ __forceinline__ void LoadGroup(const float2* __restrict__ s,
                                          uint64_t g, const uint32_t* q,
                                          float2 (&v)[1 << NQ]) {
  const unsigned q0 = q[0], q1 = NQ > 1 ? q[1] : 0;
  uint64_t base = ((g >> q0) << (q0 + 1)) | (g & ((uint64_t{1} << q0) - 1));
  if (NQ > 1) {
    base = ((base >> q1) << (q1 + 1)) | (base & ((uint64_t{1} << q1) - 1));
  }
#pragma unroll
  for (unsigned j = 0; j < (1u << NQ); ++j) {
    const uint64_t off = ((j & 1u) ? uint64_t{1} << q0 : 0) |
                         ((j & 2u) ? uint64_t{1} << q1 : 0);
    v[j] = s[base + off];
  }
}

// Re v^dagger (K^dagger K) v, the matrix K^dagger K at lm.
template <int NQ>
__device__ __forceinline__ float GroupQuadratic(const float2 (&v)[1 << NQ],
                                                const float* lm) {
  constexpr unsigned D = 1u << NQ;
  float w = 0.0f;
#pragma unroll
  for (unsigned r = 0; r < D; ++r) {
    float re = 0.0f, im = 0.0f;
#pragma unroll
    for (unsigned k = 0; k < D; ++k) {
      const float mr = lm[2 * (r * D + k)], mi = lm[2 * (r * D + k) + 1];
      re += mr * v[k].x - mi * v[k].y;
      im += mr * v[k].y + mi * v[k].x;
    }
    w += v[r].x * re + v[r].y * im;
  }
  return w;
}

// A channel that the draw's bounds did not decide (header ops[oi], its
// Kraus operators at ops[oi + 1 ..]), decided as RunIteration decides it
// (lib/qtrajectory.h:330-370) and in the same order: the non-unitary
// operators one at a time, each with a sweep for <psi|K^dagger K|psi>
// (each group's value in FP32, summed in FP64) -- the first sweep also
// giving the norm where the trajectory is not unitary, so that the
// probabilities are those of the normalised state (NormalizeState,
// lib/qtrajectory.h:449-456) -- until the draw falls below the running
// sum; the chosen operator is then applied, scaled by the normalisation.
// lm: LDS of 2 x 4^NQ floats (at least one 4 x 4 complex matrix); vals:
// LDS of 2 doubles.
template <int NT, int NQ>
__device__ void TrajChannelQ(float2* __restrict__ s, unsigned n,
                             const qsim_hip_traj_op* __restrict__ ops,
                             uint64_t oi, const float* __restrict__ mats,
                             int32_t* __restrict__ dec_out, double* red,
                             float* lm, double* vals) {
  constexpr unsigned D = 1u << NQ;
  const qsim_hip_traj_op h = ops[oi];
  const unsigned M = h.k;
  const uint64_t N = uint64_t{1} << n;
  const uint64_t ngroups = N >> NQ;
  const bool normalise = h.pad & 1u;
  bool have_norm = !normalise;
  double norm = 1.0;
  double cp = h.cp, max_prob = 0.0;
  int max_index = 0, pick = -1;
  for (unsigned i = 0; i < M; ++i) {
    const qsim_hip_traj_op c = ops[oi + 1 + i];
    if (c.pad & 1u) continue;  // unitary: decided by its bound alone
    __syncthreads();           // earlier reads of lm are done
    for (unsigned e = threadIdx.x; e < 2 * D * D; e += NT)
      lm[e] = mats[c.moff2 + e];
    __syncthreads();
    double acc = 0.0, nacc = 0.0;
    for (uint64_t g = threadIdx.x; g < ngroups; g += NT) {
      float2 v[D];
      LoadGroup<NQ>(s, g, h.q, v);
      const float w = GroupQuadratic<NQ>(v, lm);
      acc += double(w);
      if (!have_norm) {
#pragma unroll
        for (unsigned j = 0; j < D; ++j)
          nacc += double(v[j].x) * v[j].x + double(v[j].y) * v[j].y;
      }
    }
    acc = BlockSum<NT>(acc, red);
    if (threadIdx.x == 0) vals[0] = acc;
    if (!have_norm) {
      nacc = BlockSum<NT>(nacc, red);
      if (threadIdx.x == 0) vals[1] = nacc;
    }
    __syncthreads();
    if (!have_norm) {
      norm = vals[1];
      have_norm = true;
    }
    // The walk, the same in every thread.
    const double prob = vals[0] / norm;
    if (prob > max_prob) {
      max_prob = prob;
      max_index = int(i);
    }
    cp += prob - c.r;
    if (h.r < cp || i == M - 1) {
      pick = h.r < cp ? int(i) : max_index;
      break;
    }
  }
  if (!have_norm) {
    // Every operator unitary: nothing chosen, the state only normalised.
    double nacc = 0.0;
    for (uint64_t i = threadIdx.x; i < N; i += NT) {
      const float2 v = s[i];
      nacc += double(v.x) * v.x + double(v.y) * v.y;
    }
    nacc = BlockSum<NT>(nacc, red);
    if (threadIdx.x == 0) vals[1] = nacc;
    __syncthreads();
    norm = vals[1];
  }
  if (threadIdx.x == 0) dec_out[h.slot] = pick;
  __syncthreads();  // every thread is done with lm and vals
  const float a = normalise ? float(1.0 / std::sqrt(norm)) : 1.0f;
  const qsim_hip_traj_op c = ops[oi + 1 + (pick >= 0 ? pick : 0)];
  if (pick < 0 || c.k == 0) {
    // Nothing applied (or the identity): the state is only normalised.
    if (normalise) ScaleState<NT>(s, N, a);
    __syncthreads();
    return;
  }
  const unsigned DK = 1u << c.k;
  for (unsigned e = threadIdx.x; e < 2 * DK * DK; e += NT)
    lm[e] = mats[c.moff + e] * a;
  __syncthreads();
  if (c.k == 1) ApplyGateK<NT, 1>(s, c, lm, 0, N >> 1);
  else ApplyGateK<NT, 2>(s, c, lm, 0, N >> 2);
  __syncthreads();
}

template <int NT>
__device__ void TrajChannel(float2* __restrict__ s, unsigned n,
                            const qsim_hip_traj_op* __restrict__ ops,
                            uint64_t oi, const float* __restrict__ mats,
                            int32_t* __restrict__ dec_out, double* red,
                            float* lm, double* vals) {
  static_assert(kMaxChannelQubits == 2, "channel sizes");
  if (ops[oi].moff2 == 1)
    TrajChannelQ<NT, 1>(s, n, ops, oi, mats, dec_out, red, lm, vals);
  else
    TrajChannelQ<NT, 2>(s, n, ops, oi, mats, dec_out, red, lm, vals);
}

// Signs (-1)^(bit a + bit b) of index i for the pairs (pa[j], pb[j]),
// j < kPC, as bit j of a mask.  The map is linear over XOR, so the sign mask
// of i = x | y (disjoint bits) is the XOR of those of x and y.
template <unsigned kPC>
__device__ __forceinline__ uint32_t PairSigns(uint64_t i,
                                              const unsigned (&pa)[kPC],
                                              const unsigned (&pb)[kPC]) {
  uint32_t m = 0;
#pragma unroll
  for (unsigned j = 0; j < kPC; ++j) {
    m |= uint32_t(((i >> pa[j]) ^ (i >> pb[j])) & 1u) << j;
  }
  return m;
}

// w[p] for a wave-uniform p: a scalar branch instead of an indexed register.
template <unsigned N>
__device__ __forceinline__ double PickUniform(const double (&w)[N],
                                              unsigned p) {
  p = unsigned(__builtin_amdgcn_readfirstlane(int(p)));
  double v = 0.0;
  // The empty asm keeps the cases apart: folded into w[p] they would put w
  // into scratch memory.
  auto take = [&](auto u) {
    v = w[decltype(u)::value];
    asm volatile("" : "+v"(v));
  };
  if constexpr (N == 16) {
    switch (p) {
      case 8: take(std::integral_constant<int, 8>{}); break;
      case 9: take(std::integral_constant<int, 9>{}); break;
      case 10: take(std::integral_constant<int, 10>{}); break;
      case 11: take(std::integral_constant<int, 11>{}); break;
      case 12: take(std::integral_constant<int, 12>{}); break;
      case 13: take(std::integral_constant<int, 13>{}); break;
      case 14: take(std::integral_constant<int, 14>{}); break;
      case 15: take(std::integral_constant<int, 15>{}); break;
    }
    if (p > 7) return v;
  }
  switch (p) {
    case 0: take(std::integral_constant<int, 0>{}); break;
    case 1: take(std::integral_constant<int, 1>{}); break;
    case 2: take(std::integral_constant<int, 2>{}); break;
    case 3: take(std::integral_constant<int, 3>{}); break;
    case 4: take(std::integral_constant<int, 4>{}); break;
    case 5: take(std::integral_constant<int, 5>{}); break;
    case 6: take(std::integral_constant<int, 6>{}); break;
    default: take(std::integral_constant<int, 7>{}); break;
  }
  return v;
}

// Sums over amplitudes [lo, hi) of |s_i|^2 (-1)^(bit a + bit b) for the
// trajectory's pairs (FP64) and of |s_i|^2: put(j, sum) for pair j,
// put(num_pairs, norm) for the norm, each in one thread; ends with a barrier.
// lo is a multiple of kS NT; red: LDS of kPairRed<NT> doubles.
template <int NT, unsigned kS, typename Put>
__device__ void PairSums(const float2* __restrict__ s,
                         const qsim_hip_traj_desc& d,
                         const uint32_t* __restrict__ pairs, uint64_t lo,
                         uint64_t hi, double* red, Put put) {
  constexpr unsigned kPC = kPairChunk<NT>;
  constexpr unsigned kLog = kS == 16 ? 4 : 3;
  static_assert(kS == 1u << kLog, "step");
  for (unsigned p0 = 0; p0 == 0 || p0 < d.num_pairs; p0 += kPC) {
    const unsigned np = std::min(kPC, d.num_pairs - p0);
    unsigned pa[kPC], pb[kPC];
    double acc[kPC];
#pragma unroll
    for (unsigned j = 0; j < kPC; ++j) {
      pa[j] = j < np ? pairs[2 * (d.pair_offset + p0 + j)] : 0;
      pb[j] = j < np ? pairs[2 * (d.pair_offset + p0 + j) + 1] : 0;
      acc[j] = 0.0;
    }
    // Element u of a step is i0 + u NT = i0 | u NT (i0's bits from
    // log2 NT to log2 (kS NT) are zero), so a pair's sign is the thread's
    // times the step's (scalar work) times the parity of u with the pair's pattern
    // over u's bits, the same for every thread.
    uint32_t su[kLog];
#pragma unroll
    for (unsigned b = 0; b < kLog; ++b) su[b] = PairSigns(uint64_t(NT) << b, pa, pb);
    double nrm = 0.0;
    const uint32_t st = PairSigns(threadIdx.x, pa, pb);
    for (uint64_t b0 = lo; b0 < hi; b0 += kS * NT) {
      const uint64_t i0 = b0 + threadIdx.x;
      const uint32_t s0 = st ^ PairSigns(b0, pa, pb);
      float2 a[kS];
#pragma unroll
      for (unsigned u = 0; u < kS; ++u) {
        const uint64_t i = i0 + u * NT;
        a[u] = i < hi ? s[i] : float2{0.0f, 0.0f};
      }
      // w[p] = sum over u of |a_u|^2 (-1)^parity(u & p): all patterns at once
      // (a Walsh-Hadamard transform), then one addition per pair and step
      // instead of one per pair and amplitude.
      double w[kS];
#pragma unroll
      for (unsigned u = 0; u < kS; ++u)
        w[u] = double(a[u].x) * a[u].x + double(a[u].y) * a[u].y;
#pragma unroll
      for (unsigned b = 0; b < kLog; ++b)
#pragma unroll
        for (unsigned u = 0; u < kS; ++u) {
          if ((u >> b) & 1u) continue;
          const double x = w[u], y = w[u | (1u << b)];
          w[u] = x + y;
          w[u | (1u << b)] = x - y;
        }
      nrm += w[0];
#pragma unroll
      for (unsigned j = 0; j < kPC; ++j) {
        unsigned p = 0;
#pragma unroll
        for (unsigned b = 0; b < kLog; ++b) p |= ((su[b] >> j) & 1u) << b;
        const double v = PickUniform(w, p);
        acc[j] += (s0 >> j) & 1u ? -v : v;
      }
    }
    // All sums with one exchange between the waves: one after the other they
    // took most of a 2^14-amplitude chunk's time.
    const unsigned wave = threadIdx.x >> 6;
#pragma unroll
    for (unsigned j = 0; j < kPC; ++j) acc[j] = WaveSum(acc[j]);
    nrm = WaveSum(nrm);
    if ((threadIdx.x & 63u) == 0) {
#pragma unroll
      for (unsigned j = 0; j < kPC; ++j) red[wave * (kPC + 1) + j] = acc[j];
      red[wave * (kPC + 1) + kPC] = nrm;
    }
    __syncthreads();
    const unsigned j = threadIdx.x;
    const bool last = p0 + kPC >= d.num_pairs;
    if (j < np || (j == kPC && last)) {
      double v = 0.0;
#pragma unroll
      for (unsigned w = 0; w < NT / 64; ++w) v += red[w * (kPC + 1) + j];
      put(j == kPC ? d.num_pairs : p0 + j, v);
    }
    __syncthreads();
  }
}

// <Z_a Z_b> = sum_i |s_i|^2 (-1)^(bit a + bit b) / sum_i |s_i|^2 for the
// trajectory's pairs, FP64-accumulated.  A non-unitary trajectory ends
// normalised (lib/qtrajectory.h:377-383): its norm goes to norm_out and the
// scaling is applied where the state is read (qsim_hip_traj_state), which
// saves a read-write sweep of every state.
template <int NT>
__device__ void TrajFinish(const float2* __restrict__ s,
                           const qsim_hip_traj_desc& d,
                           const uint32_t* __restrict__ pairs,
                           double* __restrict__ zz_out,
                           double* __restrict__ norm_out) {
  __shared__ double pair_red[kPairRed<NT>];
  __shared__ double nrm;
  PairSums<NT, kSweep<NT>>(s, d, pairs, 0, uint64_t{1} << d.num_qubits,
                           pair_red, [&](unsigned j, double v) {
                             if (j == d.num_pairs) nrm = v;
                             else zz_out[d.pair_offset + j] = v;
                           });
  __threadfence_block();
  for (unsigned j = threadIdx.x; j < d.num_pairs; j += NT)
    zz_out[d.pair_offset + j] /= nrm;
  if (threadIdx.x == 0 && (d.pad & 1u)) norm_out[blockIdx.x] = nrm;
}

// Workgroup t runs trajectory t, one sweep of the state per operation.  A
// tile-pass header is skipped: the gates of its pass follow it in the
// stream and run here one sweep each.
template <int NT>
__global__ void __launch_bounds__(NT)
TrajectoryKernel(const qsim_hip_traj_desc* __restrict__ descs,
                 const qsim_hip_traj_op* __restrict__ ops,
                 const float* __restrict__ mats,
                 const uint32_t* __restrict__ pairs, float2* __restrict__ pool,
                 double* __restrict__ zz_out, double* __restrict__ norm_out,
                 int32_t* __restrict__ dec_out) {
  __shared__ float lm[2 * 16 * 16];
  __shared__ double red[kRedWords<NT>];
  __shared__ double vals[2];
  const qsim_hip_traj_desc d = descs[blockIdx.x];
  const unsigned n = d.num_qubits;
  float2* s = pool + d.state_offset;
  ZeroState<NT>(s, uint64_t{1} << n);
  __syncthreads();
  for (uint64_t oi = d.op_begin; oi < d.op_end; ++oi) {
    const qsim_hip_traj_op o = ops[oi];
    if (o.kind == QSIM_HIP_TRAJ_GATE) {
      TrajGate<NT>(s, o, mats, lm, 0, uint64_t{1} << (n - o.k));
    } else if (o.kind == QSIM_HIP_TRAJ_CHANNEL) {
      TrajChannel<NT>(s, n, ops, oi, mats, dec_out, red, lm, vals);
      oi += o.k;  // its Kraus operators
    }
  }
  TrajFinish<NT>(s, d, pairs, zz_out, norm_out);
}

// A tile pass of a trajectory on the device: geometry, program, and the
// index of its first op record (kF16RecWords words each) in the record pool.
struct TrajTilePass {
  BlockGeom g;
  BlockProgram p;
  uint64_t rec;
};

// ---- the tiled batch: many workgroups per trajectory -----------------------
//
// The tiled batch is a sequence of launches (TrajSchedule on the host), each
// over work items of many trajectories: a run of a trajectory's tiles for a
// tile pass, a run of its amplitudes for a sweep.  A trajectory advances by
// one operation per launch, so the end of a launch is the only
// synchronisation, and a batch of a few large trajectories fills the chip as
// well as one of many small ones.
//
// One workgroup per trajectory with barriers between its operations, which
// this replaces, streamed each state at 12-15 GB/s and lasted as long as the
// largest trajectories' serial chains: 100 trajectories each of 20, 18 and
// 16 qubits, 4 passes of 5 gates: 11.1 ms, against 4.3 ms here.
// An item of a tile pass: a run of tiles, one workgroup.
struct TrajItem {
  uint64_t op;        // operation index
  uint32_t traj;
  uint32_t first;     // first tile
  uint32_t count;     // tiles
};
// A trajectory's share of a sweep launch: one workgroup per chunk.  (An item
// per chunk would hold 24 bytes per 2^14 amplitudes and gate, on the host and
// the device: 200 MB for 8000 gates on 24 qubits.)
struct TrajSweep {
  uint64_t op;        // operation index
  uint64_t part;      // partial sums of chunk 0 (channel sums, finish)
  uint32_t traj;
  uint32_t first;     // workgroup of chunk 0
  uint32_t count;     // chunks
};

// The entry of this workgroup, the last of e[0..n) whose first workgroup is
// not past it: each wave compares 64 entries at a time (two loads up to 4096
// trajectories).
__device__ __forceinline__ TrajSweep SweepOf(const TrajSweep* __restrict__ e,
                                             unsigned n) {
  const unsigned l = threadIdx.x & 63;
  unsigned lo = 0;
  while (n > 1) {
    const unsigned step = (n + 63) / 64, at = l * step;
    const bool le = at < n && e[lo + at].first <= blockIdx.x;
    const unsigned last = __builtin_popcountll(__ballot(le)) - 1;
    lo += last * step;
    n = step < n - last * step ? step : n - last * step;
  }
  return e[__builtin_amdgcn_readfirstlane(lo)];
}

// Amplitudes of a sweep chunk: 2^14, and more where a trajectory would have
// over 1024 chunks, so that the steps that add up a trajectory's chunks in one
// workgroup (TrajChannelPickKernel, TrajFinishKernel) stay short.
constexpr uint64_t kSweepChunk = uint64_t{1} << 14;
constexpr unsigned kMaxChunkBits = 10;
__host__ __device__ inline uint64_t ChunkSize(unsigned n) {
  return n > 14 + kMaxChunkBits ? uint64_t{1} << (n - kMaxChunkBits)
                                : kSweepChunk;
}
constexpr int kSweepNT = 256;
// Partial sums of a channel's chunk (ChannelSums), at most.
constexpr unsigned kChanSums = 16;
static_assert(kMaxChannelQubits == 2, "channel sums");

// A pass over tiles of up to 13 qubits, with the FP16 arithmetic of the
// circuit kernel's blocked passes (block_kernels.hip): the pass's op records
// are copied into LDS once, then every tile of the item is staged in LDS
// scaled by a power of two (TileScale), the ops run on it and it is stored
// back scaled the other way, with the next tile's loads in flight meanwhile
// (in two halves around the first ops); two workgroups a CU.  A pass's ops
// are unitary or Kraus operators (spectral norm <= 1), so the tile never
// grows.  The tile sits at LDS offset 0 (no static LDS in the kernel,
// checked on the host).  FULL: tiles of 13 qubits.
template <bool FULL>
__device__ __forceinline__ void TrajTileRun(float2* __restrict__ s,
                                            const TrajTilePass* __restrict__ tp,
                                            const uint32_t* __restrict__ recs,
                                            char* lds_raw, uint64_t first,
                                            uint64_t end) {
  constexpr int TB = 13;
  constexpr int NT = BlockShape<TB>::NT;
  constexpr int NW = BlockShape<TB>::kWaves;
  constexpr int PER = 32;
  static_assert((1 << TB) / NT == PER, "shape");
  float2* lds = reinterpret_cast<float2*>(lds_raw);
  float* slots = reinterpret_cast<float*>(lds_raw + F16Lds<TB>::kMaxOff);
  uint32_t* rec = reinterpret_cast<uint32_t*>(lds_raw + F16Lds<TB>::kRecOff);
  const BlockGeom& g = tp->g;
  const BlockProgram& p = tp->p;
  const unsigned nops = p.nops;
  const int l = threadIdx.x & 63;
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned nbatch = (1u << g.tb) >> 9;
  const unsigned nper = (1u << g.tb) / NT;
  {
    const unsigned nq = nops * unsigned(kF16RecWords / 4);
    const uint4* src =
        reinterpret_cast<const uint4*>(recs + tp->rec * kF16RecWords);
    uint4* dst = reinterpret_cast<uint4*>(rec);
    for (unsigned q = threadIdx.x; q < nq; q += NT) dst[q] = src[q];
  }
  TileIo<PER, NT, true> io;
  io.Init(g);
  float2 buf[PER];
  io.template Fetch<FULL, 15u>(
      s, InsertZeros(first << g.Lc, g.outer, g.nouter), g, buf);
  int e = TileScale<NW>(LocalMax<PER, FULL>(buf, nper), slots, p.headroom);
  io.template PutScaled<FULL>(g, buf, lds, e);
  __syncthreads();
  for (uint64_t tile = first; tile < end; ++tile) {
    const uint64_t base = InsertZeros(tile << g.Lc, g.outer, g.nouter);
    // The next tile, or this one again after the last (an in-bounds read
    // that is never used).
    const uint64_t next = tile + 1 < end ? tile + 1 : tile;
    const uint64_t nb = InsertZeros(next << g.Lc, g.outer, g.nouter);
    io.template Fetch<FULL, 3u>(s, nb, g, buf);
    for (unsigned op = 0; op < nops; ++op) {
      F16Op o;
      o.Load(rec + op * unsigned(kF16RecWords), l);
      ApplyTileOpF16(o, nbatch, wave, NW);
      __syncthreads();
      if (op == 1) io.template Fetch<FULL, 12u>(s, nb, g, buf);
    }
    if (nops == 1) io.template Fetch<FULL, 12u>(s, nb, g, buf);
    io.template StoreScaled<16, FULL>(s, base, g, lds, e);
    e = TileScale<NW>(LocalMax<PER, FULL>(buf, nper), slots, p.headroom);
    io.template PutScaled<FULL>(g, buf, lds, e);
    __syncthreads();
  }
}

template <bool FULL>
__global__ void __launch_bounds__(BlockShape<13>::NT)
__attribute__((amdgpu_waves_per_eu(2)))
TrajPass13Kernel(const qsim_hip_traj_desc* __restrict__ descs,
                 const qsim_hip_traj_op* __restrict__ ops,
                 const TrajTilePass* __restrict__ passes,
                 const uint32_t* __restrict__ recs,
                 const TrajItem* __restrict__ items,
                 float2* __restrict__ pool) {
  extern __shared__ char lds_raw[];
  const TrajItem it = items[blockIdx.x];
  TrajTileRun<FULL>(pool + descs[it.traj].state_offset,
                    passes + ops[it.op].moff, recs, lds_raw, it.first,
                    uint64_t(it.first) + it.count);
}

// Passes over 14-qubit tiles: the circuit kernel's run (BlockIoRun).
__global__ void __launch_bounds__(kIoThreads)
__attribute__((amdgpu_waves_per_eu(3, 3)))
TrajPass14Kernel(const qsim_hip_traj_desc* __restrict__ descs,
                 const qsim_hip_traj_op* __restrict__ ops,
                 const TrajTilePass* __restrict__ passes,
                 const uint32_t* __restrict__ recs,
                 const TrajItem* __restrict__ items,
                 float2* __restrict__ pool) {
  extern __shared__ char lds_raw[];
  const TrajItem it = items[blockIdx.x];
  const TrajTilePass* tp = passes + ops[it.op].moff;
  BlockIoRun(pool + descs[it.traj].state_offset, tp->g, tp->p,
             recs + tp->rec * kF16RecWords, lds_raw, it.first,
             uint64_t(it.first) + it.count, 1);
}

// Every state to |0...0>: the pool to zeros, then each first amplitude.
__global__ void __launch_bounds__(kSweepNT)
TrajZeroKernel(float2* __restrict__ pool, uint64_t size) {
  const uint64_t stride = uint64_t(gridDim.x) * kSweepNT;
  for (uint64_t i = uint64_t(blockIdx.x) * kSweepNT + threadIdx.x; i < size;
       i += stride)
    pool[i] = float2{0.0f, 0.0f};
}
__global__ void __launch_bounds__(kSweepNT)
TrajOneKernel(const qsim_hip_traj_desc* __restrict__ descs, unsigned num,
              float2* __restrict__ pool) {
  const unsigned t = blockIdx.x * kSweepNT + threadIdx.x;
  if (t < num) pool[descs[t].state_offset] = float2{1.0f, 0.0f};
}

// Groups [lo, hi) of sweep chunk `chunk` for operators on k qubits.
__device__ __forceinline__ void SweepGroups(unsigned n, unsigned k,
                                            uint64_t chunk, uint64_t& lo,
                                            uint64_t& hi) {
  const uint64_t all = uint64_t{1} << (n - k), per = ChunkSize(n) >> k;
  lo = chunk * per;
  hi = lo + per < all ? lo + per : all;
}

__global__ void __launch_bounds__(kSweepNT)
TrajGateKernel(const qsim_hip_traj_desc* __restrict__ descs,
               const qsim_hip_traj_op* __restrict__ ops,
               const float* __restrict__ mats,
               const TrajSweep* __restrict__ sweeps, unsigned num, float2* __restrict__ pool) {
  __shared__ float lm[2 * 16 * 16];
  const TrajSweep it = SweepOf(sweeps, num);
  const unsigned chunk = blockIdx.x - it.first;
  const qsim_hip_traj_op o = ops[it.op];
  const qsim_hip_traj_desc d = descs[it.traj];
  uint64_t lo, hi;
  SweepGroups(d.num_qubits, o.k, chunk, lo, hi);
  TrajGate<kSweepNT>(pool + d.state_offset, o, mats, lm, lo, hi);
}

// Partial sums P_rc = sum conj(v_r) v_c over the groups v of the channel's
// qubits, r <= c (FP64 of FP32 amplitudes): its reduced density matrix, from
// which every operator's probability and the norm follow without another
// sweep.  Order: the diagonal, then (re, im) of the pairs r < c.
template <int NQ>
__device__ void ChannelSums(const float2* __restrict__ s, unsigned n,
                            const uint32_t* q, uint64_t chunk,
                            double* __restrict__ out) {
  constexpr unsigned D = 1u << NQ;
  double acc[D * D];
#pragma unroll
  for (unsigned e = 0; e < D * D; ++e) acc[e] = 0.0;
  uint64_t lo, hi;
  SweepGroups(n, NQ, chunk, lo, hi);
  constexpr int U = NQ == 1 ? 4 : 2;  // groups in flight
  for (uint64_t g0 = lo + threadIdx.x; g0 < hi; g0 += U * kSweepNT) {
    float2 v[U][D];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint64_t g = g0 + u * kSweepNT;
      if (g < hi) {
        LoadGroup<NQ>(s, g, q, v[u]);
      } else {
#pragma unroll
        for (unsigned r = 0; r < D; ++r) v[u][r] = float2{0.0f, 0.0f};
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      unsigned e = D;
#pragma unroll
      for (unsigned r = 0; r < D; ++r) {
        const double x = v[u][r].x, y = v[u][r].y;
        acc[r] += x * x + y * y;
#pragma unroll
        for (unsigned c = r + 1; c < D; ++c) {
          const double cx = v[u][c].x, cy = v[u][c].y;
          acc[e++] += x * cx + y * cy;
          acc[e++] += x * cy - y * cx;
        }
      }
    }
  }
#pragma unroll
  for (unsigned e = 0; e < D * D; ++e) {
    const double v = BlockSum<kSweepNT>(acc[e]);
    if (threadIdx.x == 0) out[e] = v;
  }
}

// <psi|M|psi> from the sums, M = K^dagger K at m (FP32 pairs, row-major).
__device__ __forceinline__ double ChannelProb(const double* p, unsigned D,
                                              const float* __restrict__ m) {
  double prob = 0.0;
  unsigned e = D;
  for (unsigned r = 0; r < D; ++r) {
    prob += double(m[2 * (r * D + r)]) * p[r];
    for (unsigned c = r + 1; c < D; ++c, e += 2) {
      // Re(M_rc P_rc + M_cr conj(P_rc))
      prob += (double(m[2 * (r * D + c)]) + m[2 * (c * D + r)]) * p[e] -
              (double(m[2 * (r * D + c) + 1]) - m[2 * (c * D + r) + 1]) *
                  p[e + 1];
    }
  }
  return prob;
}

__global__ void __launch_bounds__(kSweepNT)
TrajChannelSumKernel(const qsim_hip_traj_desc* __restrict__ descs,
                     const qsim_hip_traj_op* __restrict__ ops,
                     const TrajSweep* __restrict__ sweeps, unsigned num,
                     const float2* __restrict__ pool,
                     double* __restrict__ parts) {
  const TrajSweep it = SweepOf(sweeps, num);
  const unsigned chunk = blockIdx.x - it.first;
  const qsim_hip_traj_desc d = descs[it.traj];
  const float2* s = pool + d.state_offset;
  double* out = parts + it.part + uint64_t(chunk) * kChanSums;
  const qsim_hip_traj_op h = ops[it.op];
  if (h.moff2 == 1)
    ChannelSums<1>(s, d.num_qubits, h.q, chunk, out);
  else
    ChannelSums<2>(s, d.num_qubits, h.q, chunk, out);
}

// A channel's choice: the operator (-1: none) and the scale that normalises
// the state.
struct TrajPick {
  int32_t op;
  float scale;
};

// The trajectory's chunk sums added up by the workgroup, then the walk of
// RunIteration (lib/qtrajectory.h:330-370) over the operators' probabilities,
// the same in every thread.
__device__ __forceinline__ TrajPick PickOperator(
    const qsim_hip_traj_op* __restrict__ ops, const float* __restrict__ mats,
    const TrajSweep& it, const double* __restrict__ parts) {
  __shared__ double sums[kChanSums];
  const qsim_hip_traj_op h = ops[it.op];
  const bool normalise = h.pad & 1u;
  const unsigned DC = 1u << h.moff2;  // states of the channel's qubits
  for (unsigned i = 0; i < DC * DC; ++i) {
    double acc = 0.0;
    for (unsigned c = threadIdx.x; c < it.count; c += kSweepNT)
      acc += parts[it.part + uint64_t(c) * kChanSums + i];
    acc = BlockSum<kSweepNT>(acc);
    if (threadIdx.x == 0) sums[i] = acc;
  }
  __syncthreads();
  double norm = 1.0;
  if (normalise) {
    norm = 0.0;
    for (unsigned r = 0; r < DC; ++r) norm += sums[r];
  }
  double cp = h.cp, max_prob = 0.0;
  int max_index = 0, pick = -1;
  for (unsigned i = 0; i < h.k; ++i) {
    const qsim_hip_traj_op c = ops[it.op + 1 + i];
    if (c.pad & 1u) continue;
    const double prob = ChannelProb(sums, DC, mats + c.moff2) / norm;
    if (prob > max_prob) {
      max_prob = prob;
      max_index = int(i);
    }
    cp += prob - c.r;
    if (h.r < cp || i == h.k - 1) {
      pick = h.r < cp ? int(i) : max_index;
      break;
    }
  }
  return TrajPick{pick, normalise ? float(1.0 / std::sqrt(norm)) : 1.0f};
}

// The choices of a launch's channels, one workgroup a trajectory, where a
// trajectory has more than kPickChunks chunks.  Picked by every workgroup of
// the apply launch, the sums read grow with the square of the chunks; a launch
// more costs 2 us.  Four channels on one qubit, picked there / here: 18 qubits
// (16 chunks) 124 / 131 us, 22 (256) 176 / 169, 24 422 / 365, 28 21.2 / 6.1
// ms; on two qubits 28 qubits 66.1 / 6.2 ms.
constexpr unsigned kPickChunks = 64;
__global__ void __launch_bounds__(kSweepNT)
TrajChannelPickKernel(const qsim_hip_traj_op* __restrict__ ops,
                      const float* __restrict__ mats,
                      const TrajSweep* __restrict__ sweeps,
                      const double* __restrict__ parts,
                      TrajPick* __restrict__ picks) {
  const TrajSweep it = sweeps[blockIdx.x];
  const TrajPick p = PickOperator(ops, mats, it, parts);
  if (threadIdx.x == 0) picks[it.traj] = p;
}

// The chosen operator (PICK: chosen here) on this workgroup's chunk.
template <bool PICK>
__global__ void __launch_bounds__(kSweepNT)
TrajChannelApplyKernel(const qsim_hip_traj_desc* __restrict__ descs,
                       const qsim_hip_traj_op* __restrict__ ops,
                       const float* __restrict__ mats,
                       const TrajSweep* __restrict__ sweeps, unsigned num,
                       float2* __restrict__ pool,
                       const double* __restrict__ parts,
                       const TrajPick* __restrict__ picks,
                       int32_t* __restrict__ dec_out) {
  __shared__ float lm[2 * 4 * 4];
  const TrajSweep it = SweepOf(sweeps, num);
  const unsigned chunk = blockIdx.x - it.first;
  const qsim_hip_traj_desc d = descs[it.traj];
  const bool normalise = ops[it.op].pad & 1u;
  const TrajPick p =
      PICK ? PickOperator(ops, mats, it, parts) : picks[it.traj];
  const int pick = p.op;
  const float a = p.scale;
  if (chunk == 0 && threadIdx.x == 0) dec_out[ops[it.op].slot] = pick;
  float2* s = pool + d.state_offset;
  const qsim_hip_traj_op c = ops[it.op + 1 + (pick >= 0 ? pick : 0)];
  uint64_t lo, hi;
  if (pick < 0 || c.k == 0) {
    // Nothing applied (or the identity): the state is only normalised.
    if (!normalise) return;
    SweepGroups(d.num_qubits, 0, chunk, lo, hi);
    for (uint64_t i = lo + threadIdx.x; i < hi; i += kSweepNT) {
      const float2 v = s[i];
      s[i] = float2{v.x * a, v.y * a};
    }
    return;
  }
  const unsigned DK = 1u << c.k;
  for (unsigned e = threadIdx.x; e < 2 * DK * DK; e += kSweepNT)
    lm[e] = mats[c.moff + e] * a;
  __syncthreads();
  SweepGroups(d.num_qubits, c.k, chunk, lo, hi);
  if (c.k == 1) ApplyGateK<kSweepNT, 1>(s, c, lm, lo, hi);
  else ApplyGateK<kSweepNT, 2>(s, c, lm, lo, hi);
}

// One step of a Walsh-Hadamard transform over the lanes of a wave: lane bit
// B's pairs become sum (bit clear) and difference (bit set).
template <int B>
__device__ __forceinline__ double LaneButterfly(double v) {
  const uint64_t w = __builtin_bit_cast(uint64_t, v);
  const unsigned l = unsigned(w), h = unsigned(w >> 32);
  const unsigned neg = ((threadIdx.x >> B) & 1u) << 31;
  auto join = [](unsigned lo, unsigned hi) {
    return __builtin_bit_cast(double, uint64_t(hi) << 32 | lo);
  };
  if constexpr (B < 4) {
    return join(PullLane<B>(l), PullLane<B>(h)) + join(l, h ^ neg);
  } else {
    // Swapped with itself: [0] holds the clear lanes' values in both, [1]
    // the set lanes'.
    unsigned l0, l1, h0, h1;
    if constexpr (B == 4) {
      const auto x = __builtin_amdgcn_permlane16_swap(l, l, false, false);
      const auto y = __builtin_amdgcn_permlane16_swap(h, h, false, false);
      l0 = x[0]; l1 = x[1]; h0 = y[0]; h1 = y[1];
    } else {
      const auto x = __builtin_amdgcn_permlane32_swap(l, l, false, false);
      const auto y = __builtin_amdgcn_permlane32_swap(h, h, false, false);
      l0 = x[0]; l1 = x[1]; h0 = y[0]; h1 = y[1];
    }
    return join(l0, h0) + join(l1, h1 ^ neg);
  }
}

// The transform over all six lane bits: lane m gets sum (-1)^|l & m| v_l.
__device__ __forceinline__ double LaneTransform(double v) {
  v = LaneButterfly<0>(v);
  v = LaneButterfly<1>(v);
  v = LaneButterfly<2>(v);
  v = LaneButterfly<3>(v);
  v = LaneButterfly<4>(v);
  return LaneButterfly<5>(v);
}

// Partial sums of a chunk: one per pair, then the norm, 2^14 amplitudes a
// round.  A pair's sum over a round is the Walsh-Hadamard coefficient of
// |s_i|^2 at (1 << a) ^ (1 << b) (the higher index bits give a sign), so the
// coefficients of at most two set bits are made once, whatever the number of
// pairs, from one read of the round.  Index bits of a round: 0-5 the lane, 6-7 the wave, 8-13 "own":
// a thread's 64 amplitudes, 16 a step.  A thread sums 1 + 6 + 15 coefficients
// over its own bits; the first 7 take a transform over the lanes, the last 15
// (two bits already) are needed at lane 0 only; the four waves are combined
// by the threads that write.  100 trajectories each of 20, 18 and 16 qubits, all
// grid pairs: 375 us, 800 us with a sum per pair (branches for the sign pattern of
// each pair and step, and the chunk read once per 16 pairs).
constexpr unsigned kChunkOwn = 6;
constexpr unsigned kChunkSums =
    64 * (1 + kChunkOwn) + kChunkOwn * (kChunkOwn - 1) / 2;
__global__ void __launch_bounds__(kSweepNT, 4)
TrajFinishSumKernel(const qsim_hip_traj_desc* __restrict__ descs,
                    const uint32_t* __restrict__ pairs,
                    const TrajSweep* __restrict__ sweeps, unsigned num,
                    const float2* __restrict__ pool,
                    double* __restrict__ parts) {
  static_assert(kSweepNT == 256 && kSweepChunk == kSweepNT << kChunkOwn,
                "chunk's index bits");
  __shared__ double red[kSweepNT / 64][kChunkSums];
  const TrajSweep it = SweepOf(sweeps, num);
  const unsigned chunk = blockIdx.x - it.first;
  const qsim_hip_traj_desc d = descs[it.traj];
  const float2* __restrict__ s = pool + d.state_offset;
  double* out = parts + it.part + uint64_t(chunk) * (d.num_pairs + 1);
  uint64_t begin, hi;
  SweepGroups(d.num_qubits, 0, chunk, begin, hi);
  auto two = [](unsigned b, unsigned c) { return c * (c - 1) / 2 + b; };
  // One round, more in the long chunks of more than 24 qubits.
  for (uint64_t lo = begin; lo < hi; lo += kSweepChunk) {
    if (lo != begin) __syncthreads();  // red is read
    double none = 0.0, one[kChunkOwn] = {}, both[15] = {};
    // Unrolled, all steps' loads would be issued first and their values spilled.
#pragma unroll 1
    for (unsigned t = 0; t < 4; ++t) {
      // The signs of the step's two bits.
      const double s4 = t & 1u ? -1.0 : 1.0, s5 = t & 2u ? -1.0 : 1.0;
      double w[16];
#pragma unroll
      for (unsigned u = 0; u < 16; ++u) {
        const uint64_t i = lo + (t * 16 + u) * kSweepNT + threadIdx.x;
        const float2 a = i < hi ? s[i] : float2{0.0f, 0.0f};
        w[u] = double(a.x) * a.x + double(a.y) * a.y;
      }
#pragma unroll
      for (unsigned b = 0; b < 4; ++b)
#pragma unroll
        for (unsigned u = 0; u < 16; ++u) {
          if ((u >> b) & 1u) continue;
          const double x = w[u], y = w[u | (1u << b)];
          w[u] = x + y;
          w[u | (1u << b)] = x - y;
        }
      none += w[0];
      one[4] = fma(s4, w[0], one[4]);
      one[5] = fma(s5, w[0], one[5]);
      both[two(4, 5)] = fma(s4 * s5, w[0], both[two(4, 5)]);
#pragma unroll
      for (unsigned b = 0; b < 4; ++b) {
        const double v = w[1u << b];
        one[b] += v;
        both[two(b, 4)] = fma(s4, v, both[two(b, 4)]);
        both[two(b, 5)] = fma(s5, v, both[two(b, 5)]);
#pragma unroll
        for (unsigned c = b + 1; c < 4; ++c)
          both[two(b, c)] += w[(1u << b) | (1u << c)];
      }
    }
    const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    red[wave][lane] = LaneTransform(none);
#pragma unroll
    for (unsigned b = 0; b < kChunkOwn; ++b)
      red[wave][64 * (1 + b) + lane] = LaneTransform(one[b]);
#pragma unroll
    for (unsigned j = 0; j < 15; ++j) {
      const double v = LaneTransform(both[j]);
      if (lane == 0) red[wave][64 * (1 + kChunkOwn) + j] = v;
    }
    __syncthreads();
    for (unsigned j = threadIdx.x; j <= d.num_pairs; j += kSweepNT) {
      uint64_t m = 0;  // at most two bits; none for the norm
      if (j < d.num_pairs)
        m = (uint64_t{1} << pairs[2 * (d.pair_offset + j)]) ^
            (uint64_t{1} << pairs[2 * (d.pair_offset + j) + 1]);
      const unsigned own = unsigned(m >> 8) & 63u, waves = unsigned(m >> 6) & 3u;
      unsigned at = unsigned(m) & 63u;
      if (own != 0) {
        const unsigned c = 31 - __builtin_clz(own), rest = own ^ (1u << c);
        at = rest == 0 ? 64 * (1 + c) + at
                       : 64 * (1 + kChunkOwn) + two(31 - __builtin_clz(rest), c);
      }
      double v = 0.0;
#pragma unroll
      for (unsigned w = 0; w < kSweepNT / 64; ++w)
        v += __builtin_popcount(w & waves) & 1 ? -red[w][at] : red[w][at];
      if (__builtin_popcountll(lo & m) & 1) v = -v;
      out[j] = lo == begin ? v : out[j] + v;
    }
  }
}

// <Z_a Z_b> and the norm of one trajectory from its chunks' sums.
__global__ void __launch_bounds__(kSweepNT)
TrajFinishKernel(const qsim_hip_traj_desc* __restrict__ descs,
                 const TrajSweep* __restrict__ sweeps,
                 const double* __restrict__ parts,
                 double* __restrict__ zz_out, double* __restrict__ norm_out) {
  __shared__ double norm_s;
  const TrajSweep it = sweeps[blockIdx.x];
  const qsim_hip_traj_desc d = descs[it.traj];
  const unsigned np = d.num_pairs;
  const double* in = parts + it.part;
  double nrm = 0.0;
  for (unsigned c = threadIdx.x; c < it.count; c += kSweepNT)
    nrm += in[uint64_t(c) * (np + 1) + np];
  nrm = BlockSum<kSweepNT>(nrm);
  if (threadIdx.x == 0) norm_s = nrm;
  __syncthreads();
  nrm = norm_s;
  if (threadIdx.x == 0 && (d.pad & 1u)) norm_out[it.traj] = nrm;
  for (unsigned j = threadIdx.x; j < np; j += kSweepNT) {
    double acc = 0.0;
#pragma unroll 4
    for (unsigned c = 0; c < it.count; ++c) acc += in[uint64_t(c) * (np + 1) + j];
    zz_out[d.pair_offset + j] = acc / nrm;
  }
}

// One launch of a tiled batch.
struct TrajLaunch {
  enum Kind { kPass14, kPass13, kPass12, kGate, kChannelSum, kChannelPick,
              kChannelApply, kChannelPickApply, kFinishSum, kFinish } kind;
  uint64_t first;   // items (passes), sweep entries (the rest)
  uint32_t count;
  uint32_t blocks;  // workgroups
  unsigned nops;    // passes: the longest program
};

// The launches of a tiled batch, and what they read.
struct TrajPlan {
  std::vector<TrajLaunch> launches;
  std::vector<TrajItem> items;
  std::vector<TrajSweep> sweeps;
  uint64_t num_parts = 1;  // partial sums
};

struct TrajBatch {
  unsigned num_traj = 0;
  uint32_t num_pairs = 0, num_decisions = 0;
  std::vector<unsigned> max_qubits;
  qsim_hip_traj_desc* descs = nullptr;
  qsim_hip_traj_op* ops = nullptr;
  float* mats = nullptr;
  uint32_t* pairs = nullptr;
  float2* pool = nullptr;
  double* zz = nullptr;
  double* norms = nullptr;  // per trajectory (device order)
  std::vector<uint8_t> normalize;
  int32_t* dec = nullptr;
  TrajTilePass* passes = nullptr;
  uint32_t* recs = nullptr;
  // The tiled batch's launches, their items and sweep entries (BuildTiled).
  bool tiled = false;
  std::vector<TrajLaunch> launches;
  TrajItem* items = nullptr;
  TrajSweep* sweeps = nullptr;
  double* parts = nullptr;
  TrajPick* picks = nullptr;  // by trajectory
  uint64_t pool_size = 0;  // amplitudes
  uint64_t num_ops = 0;
  std::vector<uint64_t> state_offset;
  std::vector<unsigned> nq;
  hipStream_t gstream = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  unsigned graph_threads = 0;
};

template <int NT>
void LaunchTraj(TrajBatch& b, hipStream_t st) {
  hipLaunchKernelGGL(TrajectoryKernel<NT>, dim3(b.num_traj), dim3(NT), 0, st,
                     b.descs, b.ops, b.mats, b.pairs, b.pool, b.zz, b.norms,
                     b.dec);
}

// The pass kernels need more than 64 KiB of dynamic LDS (allowed once per
// process, outside any stream capture) and address the tile from LDS
// offset 0, which holds only with no static LDS ahead of the dynamic block.
int TileKernelReady() {
  static std::once_flag once;
  static hipError_t attr = hipSuccess;
  static size_t static_lds = 0;
  std::call_once(once, [] {
    const struct {
      const void* fn;
      size_t lds;
    } fns[3] = {
        {reinterpret_cast<const void*>(&TrajPass13Kernel<true>),
         F16Lds<13>::Bytes(F16Lds<13>::kMaxOps)},
        {reinterpret_cast<const void*>(&TrajPass13Kernel<false>),
         F16Lds<13>::Bytes(F16Lds<13>::kMaxOps)},
        {reinterpret_cast<const void*>(&TrajPass14Kernel),
         F16Lds<14>::Bytes(F16Lds<14>::kMaxOps)}};
    for (const auto& f : fns) {
      hipFuncAttributes fa{};
      if (attr == hipSuccess) attr = hipFuncGetAttributes(&fa, f.fn);
      static_lds = std::max(static_lds, fa.sharedSizeBytes);
      if (attr == hipSuccess) {
        attr = hipFuncSetAttribute(
            f.fn, hipFuncAttributeMaxDynamicSharedMemorySize, int(f.lds));
      }
    }
  });
  QHIP_CHECK(attr);
  if (static_lds != 0) {
    SetError("tiled trajectory kernel has %zu bytes of static LDS", static_lds);
    return QSIM_HIP_ERR_RUNTIME;
  }
  return QSIM_HIP_OK;
}

// The launches of a tiled batch.  In turn: gates and channels of every
// trajectory that stands at one, until all stand at a tile pass or at their
// end; then one pass of every trajectory.  Passes are cut into items of
// about a quarter of a CU's share of the launch, largest first, so that the
// last items to run are short; an item's first load and last store are
// exposed, so it has at least four tiles where the state has.
TrajPlan TrajSchedule(const std::vector<qsim_hip_traj_desc>& d,
                      const std::vector<qsim_hip_traj_op>& ops,
                      const std::vector<TrajTilePass>& passes, unsigned cus) {
  TrajPlan plan;
  const uint32_t T = uint32_t(d.size());
  std::vector<uint64_t> at(T);
  for (uint32_t t = 0; t < T; ++t) at[t] = d[t].op_begin;
  auto chunks = [&](uint32_t t) {
    const uint64_t N = uint64_t{1} << d[t].num_qubits;
    return uint32_t(std::max<uint64_t>(1, N / ChunkSize(d[t].num_qubits)));
  };
  // A launch over the trajectories of `list`; blocks: one workgroup an entry
  // or (0) one a chunk.
  auto sweep = [&](TrajLaunch::Kind kind, std::vector<TrajSweep> list,
                   uint32_t blocks) {
    if (list.empty()) return;
    uint32_t total = 0;
    for (TrajSweep& e : list) {
      e.first = total;
      total += e.count;
    }
    plan.launches.push_back({kind, plan.sweeps.size(), uint32_t(list.size()),
                             blocks ? blocks : total, 0});
    plan.sweeps.insert(plan.sweeps.end(), list.begin(), list.end());
  };
  for (;;) {
    bool pass = false;
    std::vector<TrajSweep> gates, channels;
    uint64_t part = 0;
    for (uint32_t t = 0; t < T; ++t) {
      if (at[t] >= d[t].op_end) continue;
      const qsim_hip_traj_op& o = ops[at[t]];
      if (o.kind == QSIM_HIP_TRAJ_TILE_PASS) {
        pass = true;
        continue;
      }
      const uint32_t nc = chunks(t);
      if (o.kind == QSIM_HIP_TRAJ_GATE) {
        gates.push_back({at[t], 0, t, 0, nc});
        at[t] += 1;
      } else {
        channels.push_back({at[t], part, t, 0, nc});
        part += uint64_t(nc) * kChanSums;
        at[t] += 1 + o.k;
      }
    }
    plan.num_parts = std::max(plan.num_parts, part);
    if (!gates.empty() || !channels.empty()) {
      sweep(TrajLaunch::kGate, gates, 0);
      sweep(TrajLaunch::kChannelSum, channels, 0);
      if (std::any_of(channels.begin(), channels.end(), [](const TrajSweep& e) {
            return e.count > kPickChunks;
          })) {
        sweep(TrajLaunch::kChannelPick, channels, uint32_t(channels.size()));
        sweep(TrajLaunch::kChannelApply, channels, 0);
      } else {
        sweep(TrajLaunch::kChannelPickApply, channels, 0);
      }
      continue;
    }
    if (!pass) break;
    // The tile qubits of the pass each trajectory stands at (0: its end).
    std::vector<unsigned> tile_bits(T, 0);
    for (uint32_t t = 0; t < T; ++t) {
      if (at[t] < d[t].op_end) tile_bits[t] = passes[ops[at[t]].moff].g.tb;
    }
    for (const auto kind :
         {TrajLaunch::kPass14, TrajLaunch::kPass13, TrajLaunch::kPass12}) {
      uint64_t tiles = 0;
      unsigned nops = 0;
      auto takes = [&](uint32_t t) {
        const unsigned tb = tile_bits[t];
        return tb != 0 && kind == (tb == 14   ? TrajLaunch::kPass14
                                   : tb == 13 ? TrajLaunch::kPass13
                                              : TrajLaunch::kPass12);
      };
      std::vector<uint32_t> who;
      for (uint32_t t = 0; t < T; ++t) {
        if (!takes(t)) continue;
        who.push_back(t);
        const TrajTilePass& tp = passes[ops[at[t]].moff];
        tiles += tp.g.ntiles;
        nops = std::max(nops, tp.p.nops);
      }
      if (who.empty()) continue;
      const uint64_t slots = uint64_t(cus) * (kind == TrajLaunch::kPass14 ? 1 : 2);
      const uint64_t per = std::max<uint64_t>(4, (tiles + 4 * slots - 1) /
                                                     (4 * slots));
      std::vector<TrajItem> list;
      for (const uint32_t t : who) {
        const uint64_t nt = passes[ops[at[t]].moff].g.ntiles;
        const uint64_t parts = (nt + per - 1) / per;
        for (uint64_t i = 0; i < parts; ++i) {
          const uint64_t a = nt * i / parts, b = nt * (i + 1) / parts;
          list.push_back({at[t], t, uint32_t(a), uint32_t(b - a)});
        }
      }
      std::stable_sort(list.begin(), list.end(),
                       [](const TrajItem& x, const TrajItem& y) {
                         return x.count > y.count;
                       });
      plan.launches.push_back({kind, plan.items.size(), uint32_t(list.size()),
                               uint32_t(list.size()), nops});
      plan.items.insert(plan.items.end(), list.begin(), list.end());
      for (const uint32_t t : who) at[t] += 1 + ops[at[t]].k;
    }
  }
  uint64_t part = 0;
  std::vector<TrajSweep> ends;
  for (uint32_t t = 0; t < T; ++t) {
    const uint32_t nc = chunks(t);
    ends.push_back({0, part, t, 0, nc});
    part += uint64_t(nc) * (d[t].num_pairs + 1);
  }
  plan.num_parts = std::max(plan.num_parts, part);
  sweep(TrajLaunch::kFinishSum, ends, 0);
  sweep(TrajLaunch::kFinish, ends, T);
  return plan;
}

int LaunchTiled(TrajBatch& b, hipStream_t st) {
  const unsigned zb = unsigned(std::min<uint64_t>(
      (b.pool_size + kSweepNT - 1) / kSweepNT, uint64_t(NumCUs()) * 32));
  hipLaunchKernelGGL(TrajZeroKernel, dim3(zb), dim3(kSweepNT), 0, st, b.pool,
                     b.pool_size);
  hipLaunchKernelGGL(TrajOneKernel,
                     dim3((b.num_traj + kSweepNT - 1) / kSweepNT),
                     dim3(kSweepNT), 0, st, b.descs, b.num_traj, b.pool);
  for (const TrajLaunch& l : b.launches) {
    const TrajItem* it = b.items + l.first;
    const TrajSweep* sw = b.sweeps + l.first;
    const dim3 grid(l.blocks), nt(kSweepNT);
    switch (l.kind) {
      case TrajLaunch::kPass14:
        hipLaunchKernelGGL(TrajPass14Kernel, grid, dim3(kIoThreads),
                           F16Lds<14>::Bytes(l.nops), st, b.descs, b.ops,
                           b.passes, b.recs, it, b.pool);
        break;
      case TrajLaunch::kPass13:
        hipLaunchKernelGGL(TrajPass13Kernel<true>, grid,
                           dim3(BlockShape<13>::NT),
                           F16Lds<13>::Bytes(l.nops), st, b.descs, b.ops,
                           b.passes, b.recs, it, b.pool);
        break;
      case TrajLaunch::kPass12:
        hipLaunchKernelGGL(TrajPass13Kernel<false>, grid,
                           dim3(BlockShape<13>::NT),
                           F16Lds<13>::Bytes(l.nops), st, b.descs, b.ops,
                           b.passes, b.recs, it, b.pool);
        break;
      case TrajLaunch::kGate:
        hipLaunchKernelGGL(TrajGateKernel, grid, nt, 0, st, b.descs, b.ops,
                           b.mats, sw, l.count, b.pool);
        break;
      case TrajLaunch::kChannelSum:
        hipLaunchKernelGGL(TrajChannelSumKernel, grid, nt, 0, st, b.descs,
                           b.ops, sw, l.count, b.pool, b.parts);
        break;
      case TrajLaunch::kChannelPick:
        hipLaunchKernelGGL(TrajChannelPickKernel, grid, nt, 0, st, b.ops,
                           b.mats, sw, b.parts, b.picks);
        break;
      case TrajLaunch::kChannelApply:
        hipLaunchKernelGGL(TrajChannelApplyKernel<false>, grid, nt, 0, st,
                           b.descs, b.ops, b.mats, sw, l.count, b.pool,
                           b.parts, b.picks, b.dec);
        break;
      case TrajLaunch::kChannelPickApply:
        hipLaunchKernelGGL(TrajChannelApplyKernel<true>, grid, nt, 0, st,
                           b.descs, b.ops, b.mats, sw, l.count, b.pool,
                           b.parts, b.picks, b.dec);
        break;
      case TrajLaunch::kFinishSum:
        hipLaunchKernelGGL(TrajFinishSumKernel, grid, nt, 0, st, b.descs,
                           b.pairs, sw, l.count, b.pool, b.parts);
        break;
      case TrajLaunch::kFinish:
        hipLaunchKernelGGL(TrajFinishKernel, grid, nt, 0, st, b.descs, sw,
                           b.parts, b.zz, b.norms);
        break;
    }
  }
  QHIP_LAUNCHED("tiled trajectory batch");
  return QSIM_HIP_OK;
}

int Launch(TrajBatch& b, unsigned threads, hipStream_t st) {
  switch (threads) {
    case 256: LaunchTraj<256>(b, st); break;
    case 512: LaunchTraj<512>(b, st); break;
    case 1024: LaunchTraj<1024>(b, st); break;
    case QSIM_HIP_TRAJ_TILED:
      return LaunchTiled(b, st);
    default:
      SetError("trajectory batches run with 256, 512 or 1024 threads or "
               "tiled (%u), not %u", unsigned(QSIM_HIP_TRAJ_TILED), threads);
      return QSIM_HIP_ERR_ARG;
  }
  QHIP_LAUNCHED("TrajectoryKernel");
  return QSIM_HIP_OK;
}

// A distinct tile pass to build: the header of its first occurrence (its
// gates o[1..k] follow) and the state size.
struct TilePassJob {
  unsigned n;
  const qsim_hip_traj_op* o;
};

// Index of the tile pass whose header is o[0] among the batch's distinct
// passes, adding it if new.  Passes with the same state size, tile, gate
// qubits and matrix offsets -- most passes of the trajectories of one
// circuit, when the caller shares identical matrices as the batch planner
// does -- share one device copy.
uint32_t TilePassIndex(unsigned n, const qsim_hip_traj_op* o,
                       std::vector<TilePassJob>& jobs,
                       std::unordered_map<std::string, uint32_t>& seen) {
  std::string key;
  auto put = [&](const void* p, size_t bytes) {
    key.append(static_cast<const char*>(p), bytes);
  };
  put(&n, sizeof(n));
  put(o[0].q, 2 * sizeof(uint32_t));
  for (unsigned j = 1; j <= o[0].k; ++j) {
    put(&o[j].k, sizeof(uint32_t));
    put(o[j].q, o[j].k * sizeof(uint32_t));
    put(&o[j].moff, sizeof(uint32_t));
  }
  auto it = seen.emplace(std::move(key), uint32_t(jobs.size())).first;
  if (it->second == jobs.size()) jobs.push_back({n, o});
  return it->second;
}

// The device form of a tile pass (header and gates validated, including the
// conditions PrepareGateBlock checks): geometry, program and FP16 op
// records as the circuit kernel's blocked passes build them, from the
// gates' FP32 matrices (exact in FP64); the records go to
// rec[0 .. k kF16RecWords).
int BuildTilePass(const TilePassJob& job, const float* mats, TrajTilePass& tp,
                  uint32_t* rec) {
  const qsim_hip_traj_op* o = job.o;
  const unsigned n = job.n, nops = o[0].k;
  const uint64_t mask = uint64_t(o[0].q[0]) | (uint64_t(o[0].q[1]) << 32);
  unsigned tile[kBlockMaxBits], nt = 0;
  for (unsigned q = 0; q < n; ++q) {
    if ((mask >> q) & 1u) tile[nt++] = q;
  }
  std::vector<unsigned> ks(nops), qs(4 * size_t(nops), 0);
  std::vector<double> m64;
  std::vector<size_t> moff(nops);
  for (unsigned j = 0; j < nops; ++j) {
    const qsim_hip_traj_op& gop = o[j + 1];
    ks[j] = gop.k;
    for (unsigned b = 0; b < gop.k; ++b) qs[4 * j + b] = gop.q[b];
    moff[j] = m64.size();
    const size_t nf = size_t{2} << (2 * gop.k);
    m64.insert(m64.end(), mats + gop.moff, mats + gop.moff + nf);
  }
  std::vector<uint16_t> fb;
  const int rc = PrepareGateBlock(n, tile, nt, nops, ks.data(), qs.data(),
                                  m64.data(), moff.data(), tp.g, tp.p, fb,
                                  kBlockArithF16);
  if (rc != QSIM_HIP_OK) return rc;
  if (tp.p.arith != kBlockArithF16) {
    // Matrices that could grow the state by 2^10: not Kraus operators.
    SetError("tile pass gates grow the state by more than 2^10 (run the "
             "per-gate kernels)");
    return QSIM_HIP_ERR_UNSUPPORTED;
  }
  std::memcpy(rec, fb.data(), fb.size() * sizeof(uint16_t));
  return QSIM_HIP_OK;
}

// Builds the distinct passes, spread over a few host threads that take jobs
// from a shared counter (each pass is independent; the lane-position memo is
// shared under its lock).  A thread that cannot be started leaves its share
// to the others, and a failed host allocation in a worker becomes an error
// return instead of ending the process.
int BuildTilePasses(const std::vector<TilePassJob>& jobs, const float* mats,
                    std::vector<TrajTilePass>& passes,
                    std::vector<uint32_t>& recs) {
  constexpr size_t kRec = kF16RecWords;  // words per record
  passes.assign(jobs.size(), TrajTilePass{});
  size_t total = 0;
  for (size_t j = 0; j < jobs.size(); ++j) {
    passes[j].rec = total;
    total += jobs[j].o[0].k;
  }
  recs.assign(total * kRec, 0);
  constexpr int kHostAlloc = 1;  // worker-side marker, never returned
  std::vector<int> rc(jobs.size(), QSIM_HIP_OK);
  const unsigned hw = std::max(1u, std::thread::hardware_concurrency());
  const unsigned nw = unsigned(std::min<size_t>(
      std::min(hw, 16u), std::max<size_t>(1, jobs.size() / 64)));
  std::atomic<size_t> next{0};
  auto work = [&]() {
    for (size_t j; (j = next.fetch_add(1)) < jobs.size();) {
      try {
        rc[j] = BuildTilePass(jobs[j], mats, passes[j],
                              recs.data() + passes[j].rec * kRec);
      } catch (const std::bad_alloc&) {
        rc[j] = kHostAlloc;
      }
    }
  };
  std::vector<std::thread> pool;
  pool.reserve(nw);
  for (unsigned w = 1; w < nw; ++w) {
    try {
      pool.emplace_back(work);
    } catch (const std::system_error&) {
      break;
    }
  }
  work();
  for (auto& th : pool) th.join();
  for (size_t j = 0; j < jobs.size(); ++j) {
    if (rc[j] == kHostAlloc) {
      SetError("traj_prepare: out of host memory building tile pass %zu", j);
      return QSIM_HIP_ERR_RUNTIME;
    }
    if (rc[j] != QSIM_HIP_OK) {
      // Again on this thread, for its error message.
      return BuildTilePass(jobs[j], mats, passes[j],
                           recs.data() + passes[j].rec * kRec);
    }
  }
  return QSIM_HIP_OK;
}

__global__ void FillInt(int32_t* __restrict__ p, unsigned n, int32_t v) {
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

template <typename T>
int Upload(T** dst, const T* src, size_t count) {
  const size_t bytes = std::max<size_t>(count, 1) * sizeof(T);
  QHIP_CHECK(hipMalloc(dst, bytes));
  if (count) {
    QHIP_CHECK(hipMemcpy(*dst, src, count * sizeof(T), hipMemcpyHostToDevice));
  }
  return QSIM_HIP_OK;
}

// What a tiled run reads beside the streams.  Batches with tile passes have it
// from the start; the rest, planned for the per-gate kernels, not before they
// are first run tiled (from their streams on the device).
int BuildTiled(TrajBatch& b, const std::vector<qsim_hip_traj_desc>& d,
               const std::vector<qsim_hip_traj_op>& ops,
               const std::vector<TrajTilePass>& passes) {
  QHIP_TRY(TileKernelReady());
  TrajPlan plan = TrajSchedule(d, ops, passes, unsigned(NumCUs()));
  // A first try may have ended for want of memory.
  (void)hipFree(b.items);
  (void)hipFree(b.sweeps);
  (void)hipFree(b.parts);
  (void)hipFree(b.picks);
  b.items = nullptr;
  b.sweeps = nullptr;
  b.parts = nullptr;
  b.picks = nullptr;
  QHIP_TRY(Upload(&b.items, plan.items.data(), plan.items.size()));
  QHIP_TRY(Upload(&b.sweeps, plan.sweeps.data(), plan.sweeps.size()));
  QHIP_CHECK(hipMalloc(&b.parts, plan.num_parts * sizeof(double)));
  QHIP_CHECK(hipMalloc(&b.picks, b.num_traj * sizeof(TrajPick)));
  b.launches = std::move(plan.launches);
  b.tiled = true;
  return QSIM_HIP_OK;
}

int BuildTiledFromDevice(TrajBatch& b) {
  std::vector<qsim_hip_traj_desc> d(b.num_traj);
  std::vector<qsim_hip_traj_op> ops(b.num_ops);
  QHIP_CHECK(hipMemcpy(d.data(), b.descs, d.size() * sizeof(d[0]),
                       hipMemcpyDeviceToHost));
  if (!ops.empty()) {
    QHIP_CHECK(hipMemcpy(ops.data(), b.ops, ops.size() * sizeof(ops[0]),
                         hipMemcpyDeviceToHost));
  }
  return BuildTiled(b, d, ops, {});
}

void Release(TrajBatch* b) {
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  if (b->gstream) (void)hipStreamDestroy(b->gstream);
  (void)hipFree(b->descs);
  (void)hipFree(b->ops);
  (void)hipFree(b->mats);
  (void)hipFree(b->pairs);
  (void)hipFree(b->pool);
  (void)hipFree(b->zz);
  (void)hipFree(b->norms);
  (void)hipFree(b->dec);
  (void)hipFree(b->passes);
  (void)hipFree(b->recs);
  (void)hipFree(b->items);
  (void)hipFree(b->sweeps);
  (void)hipFree(b->parts);
  (void)hipFree(b->picks);
  delete b;
}

}  // namespace

}  // namespace qhip

using namespace qhip;

extern "C" {

static int TrajPrepare(const qsim_hip_traj_desc* trajs, unsigned num_traj,
                       const qsim_hip_traj_op* ops, uint64_t num_ops,
                       const float* matrices, uint64_t num_floats,
                       const uint32_t* pairs, uint32_t num_pairs,
                       uint32_t num_decisions, void** handle) {
  if (handle == nullptr || trajs == nullptr || num_traj == 0 ||
      (num_ops && ops == nullptr) || (num_floats && matrices == nullptr) ||
      (num_pairs && pairs == nullptr)) {
    SetError("trajectory batch: null or empty operand");
    return QSIM_HIP_ERR_ARG;
  }
  *handle = nullptr;
  QHIP_TRY(EnsureInit());
  // Validate every stream against the kernel's assumptions before anything
  // reaches the device.
  uint64_t pool = 0;
  std::vector<qsim_hip_traj_desc> d(trajs, trajs + num_traj);
  for (unsigned t = 0; t < num_traj; ++t) {
    const unsigned n = d[t].num_qubits;
    if (n < 4 || n > 34 || d[t].op_begin > d[t].op_end ||
        d[t].op_end > num_ops ||
        uint64_t(d[t].pair_offset) + d[t].num_pairs > num_pairs) {
      SetError("trajectory %u: bad size, operation range or pair range", t);
      return QSIM_HIP_ERR_ARG;
    }
    d[t].state_offset = pool;
    pool += uint64_t{1} << n;
    for (uint64_t i = d[t].op_begin; i < d[t].op_end; ++i) {
      const qsim_hip_traj_op& o = ops[i];
      bool ok;
      if (o.kind == QSIM_HIP_TRAJ_GATE) {
        ok = o.k >= 1 && o.k <= 4 &&
             uint64_t(o.moff) + (size_t{2} << (2 * o.k)) <= num_floats;
        for (unsigned b = 0; ok && b < o.k; ++b)
          ok = o.q[b] < n && (b == 0 || o.q[b] > o.q[b - 1]);
      } else if (o.kind == QSIM_HIP_TRAJ_CHANNEL) {
        // The header of a channel decision and its Kraus operators: each K
        // on qubits of the channel, K^dagger K over the channel's qubits.
        const unsigned nq = o.moff2;
        ok = o.k >= 1 && o.k <= kMaxKraus && i + o.k < d[t].op_end &&
             nq >= 1 && nq <= kMaxChannelQubits && o.slot < num_decisions;
        uint64_t cmask = 0;
        for (unsigned b = 0; ok && b < nq; ++b) {
          ok = o.q[b] < n && (b == 0 || o.q[b] > o.q[b - 1]);
          if (ok) cmask |= uint64_t{1} << o.q[b];
        }
        for (unsigned j = 1; ok && j <= o.k; ++j) {
          const qsim_hip_traj_op& c = ops[i + j];
          ok = c.kind == QSIM_HIP_TRAJ_KRAUS && c.k <= nq &&
               (c.k == 0 ||
                uint64_t(c.moff) + (size_t{2} << (2 * c.k)) <= num_floats) &&
               ((c.pad & 1u) ||
                uint64_t(c.moff2) + (size_t{2} << (2 * nq)) <= num_floats);
          for (unsigned b = 0; ok && b < c.k; ++b) {
            ok = c.q[b] < 64 && ((cmask >> c.q[b]) & 1u) &&
                 (b == 0 || c.q[b] > c.q[b - 1]);
          }
        }
        if (ok) i += o.k;  // the Kraus operators are part of the header
      } else if (o.kind == QSIM_HIP_TRAJ_TILE_PASS) {
        // The header of a pass over the gates that follow it (each checked
        // as a gate in its turn; their tile membership when the pass is
        // built).
        // The tile holds qubits 0, 1 and 2 (the contiguous low run) and
        // every qubit of the pass's gates.
        const uint64_t mask = uint64_t(o.q[0]) | (uint64_t(o.q[1]) << 32);
        const unsigned nt = unsigned(__builtin_popcountll(mask));
        // At most as many gates as the tile kernel keeps resident.
        ok = o.k >= 1 && o.k <= BlockResidentOps(nt) && i + o.k < d[t].op_end &&
             (mask >> n) == 0 && nt >= kBlockMinBits && nt <= kBlockMaxBits &&
             (mask & 7u) == 7u;
        for (unsigned j = 1; ok && j <= o.k; ++j) {
          const qsim_hip_traj_op& g = ops[i + j];
          ok = g.kind == QSIM_HIP_TRAJ_GATE && g.k >= 1 && g.k <= 4;
          for (unsigned b = 0; ok && b < g.k; ++b)
            ok = g.q[b] < 64 && ((mask >> g.q[b]) & 1u);
        }
      } else {
        ok = false;
      }
      if (!ok) {
        SetError("trajectory %u: operation %llu is malformed", t,
                 (unsigned long long)(i - d[t].op_begin));
        return QSIM_HIP_ERR_ARG;
      }
    }
    for (uint32_t p = 0; p < d[t].num_pairs; ++p) {
      const uint32_t* pp = pairs + 2 * (size_t(d[t].pair_offset) + p);
      if (pp[0] >= n || pp[1] >= n || pp[0] == pp[1]) {
        SetError("trajectory %u: bad qubit pair", t);
        return QSIM_HIP_ERR_ARG;
      }
    }
  }
  // Tile passes to their device form; the header's moff becomes the pass
  // index.
  std::vector<qsim_hip_traj_op> ov(ops, ops + num_ops);
  std::vector<TrajTilePass> passes;
  std::vector<uint32_t> recs;
  {
    std::vector<TilePassJob> jobs;
    std::unordered_map<std::string, uint32_t> seen;
    for (unsigned t = 0; t < num_traj; ++t) {
      for (uint64_t i = d[t].op_begin; i < d[t].op_end; ++i) {
        if (ov[i].kind != QSIM_HIP_TRAJ_TILE_PASS) continue;
        ov[i].moff = TilePassIndex(d[t].num_qubits, ops + i, jobs, seen);
      }
    }
    QHIP_TRY(BuildTilePasses(jobs, matrices, passes, recs));
  }
  // Released (device buffers included) on every early return or exception.
  std::unique_ptr<TrajBatch, void (*)(TrajBatch*)> b(new TrajBatch, Release);
  b->num_traj = num_traj;
  b->pool_size = pool;
  b->num_ops = num_ops;
  b->num_pairs = num_pairs;
  b->num_decisions = num_decisions;
  for (unsigned t = 0; t < num_traj; ++t) {
    b->state_offset.push_back(d[t].state_offset);
    b->nq.push_back(d[t].num_qubits);
    b->normalize.push_back(d[t].pad & 1u);
  }
  int rc = Upload(&b->descs, d.data(), d.size());
  if (rc == QSIM_HIP_OK) rc = Upload(&b->ops, ov.data(), num_ops);
  if (rc == QSIM_HIP_OK) rc = Upload(&b->passes, passes.data(), passes.size());
  if (rc == QSIM_HIP_OK) rc = Upload(&b->recs, recs.data(), recs.size());
  if (rc == QSIM_HIP_OK) rc = Upload(&b->mats, matrices, num_floats);
  if (rc == QSIM_HIP_OK) rc = Upload(&b->pairs, pairs, size_t(2) * num_pairs);
  if (rc == QSIM_HIP_OK) {
    hipError_t e = hipMalloc(&b->pool, pool * sizeof(float2));
    if (e == hipSuccess) e = hipMalloc(&b->zz, std::max<size_t>(num_pairs, 1) * 8);
    if (e == hipSuccess) e = hipMalloc(&b->norms, size_t(num_traj) * 8);
    if (e == hipSuccess)
      e = hipMalloc(&b->dec, std::max<size_t>(num_decisions, 1) * 4);
    if (e != hipSuccess) rc = HipFail(e, "trajectory batch buffers");
  }
  if (rc == QSIM_HIP_OK && !passes.empty()) rc = BuildTiled(*b, d, ov, passes);
  if (rc != QSIM_HIP_OK) return rc;
  *handle = b.release();
  return QSIM_HIP_OK;
}

// A failed host allocation (the validated copies of the streams, the tile
// passes, the batch record) becomes an error return: an exception may not
// cross the C ABI.
int qsim_hip_traj_prepare(const qsim_hip_traj_desc* trajs, unsigned num_traj,
                          const qsim_hip_traj_op* ops, uint64_t num_ops,
                          const float* matrices, uint64_t num_floats,
                          const uint32_t* pairs, uint32_t num_pairs,
                          uint32_t num_decisions, void** handle) {
  try {
    return TrajPrepare(trajs, num_traj, ops, num_ops, matrices, num_floats,
                       pairs, num_pairs, num_decisions, handle);
  } catch (const std::bad_alloc&) {
    if (handle) *handle = nullptr;
    SetError("traj_prepare: out of host memory");
    return QSIM_HIP_ERR_RUNTIME;
  }
}

int qsim_hip_traj_run(void* handle, unsigned threads, int use_graph) {
  QHIP_TRY(FlushGateQueue());
  auto* b = static_cast<TrajBatch*>(handle);
  if (b == nullptr) return QSIM_HIP_ERR_ARG;
  if (threads == QSIM_HIP_TRAJ_TILED && !b->tiled) {
    QHIP_TRY(GuardHost([&]() -> int { return BuildTiledFromDevice(*b); }));
  }
  // Undecided slots read -1 (the decision kernel writes the reached ones).
  hipLaunchKernelGGL(FillInt, dim3((b->num_decisions + 255) / 256 + 1),
                     dim3(256), 0, Stream(), b->dec, b->num_decisions, -1);
  QHIP_LAUNCHED("FillInt");
  if (!use_graph) {
    PassTimerBegin();
    QHIP_TRY(Launch(*b, threads, Stream()));
    PassTimerEnd();
    QHIP_CHECK(hipStreamSynchronize(Stream()));
    return QSIM_HIP_OK;
  }
  QHIP_CHECK(hipStreamSynchronize(Stream()));
  if (b->exec == nullptr || b->graph_threads != threads) {
    if (b->exec) (void)hipGraphExecDestroy(b->exec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    b->exec = nullptr;
    b->graph = nullptr;
    if (b->gstream == nullptr) QHIP_CHECK(hipStreamCreate(&b->gstream));
    QHIP_CHECK(hipStreamBeginCapture(b->gstream, hipStreamCaptureModeThreadLocal));
    int rc = Launch(*b, threads, b->gstream);
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(b->gstream, &g);
    if (rc != QSIM_HIP_OK) return rc;
    if (e != hipSuccess) return HipFail(e, "hipStreamEndCapture");
    b->graph = g;
    QHIP_CHECK(hipGraphInstantiate(&b->exec, g, nullptr, nullptr, 0));
    b->graph_threads = threads;
  }
  QHIP_CHECK(hipGraphLaunch(b->exec, b->gstream));
  QHIP_CHECK(hipStreamSynchronize(b->gstream));
  return QSIM_HIP_OK;
}

int qsim_hip_traj_results(void* handle, double* zz, uint32_t num_pairs,
                          int32_t* decisions, uint32_t num_decisions) {
  auto* b = static_cast<TrajBatch*>(handle);
  if (b == nullptr || num_pairs > b->num_pairs ||
      num_decisions > b->num_decisions) {
    SetError("trajectory batch: result sizes exceed the batch");
    return QSIM_HIP_ERR_ARG;
  }
  if (zz && num_pairs)
    QHIP_CHECK(hipMemcpy(zz, b->zz, num_pairs * 8ull, hipMemcpyDeviceToHost));
  if (decisions && num_decisions)
    QHIP_CHECK(hipMemcpy(decisions, b->dec, num_decisions * 4ull,
                         hipMemcpyDeviceToHost));
  return QSIM_HIP_OK;
}

int qsim_hip_traj_state(void* handle, unsigned t, float* out) {
  auto* b = static_cast<TrajBatch*>(handle);
  if (b == nullptr || t >= b->num_traj || out == nullptr) {
    SetError("trajectory batch: bad trajectory index");
    return QSIM_HIP_ERR_ARG;
  }
  const size_t count = size_t{2} << b->nq[t];
  QHIP_CHECK(hipMemcpy(out, b->pool + b->state_offset[t],
                       count * sizeof(float), hipMemcpyDeviceToHost));
  if (b->normalize[t]) {
    // The end-of-trajectory normalisation (the norm from the final sweep).
    double nrm = 0.0;
    QHIP_CHECK(hipMemcpy(&nrm, b->norms + t, sizeof(double),
                         hipMemcpyDeviceToHost));
    const float a = float(1.0 / std::sqrt(nrm));
    for (size_t i = 0; i < count; ++i) out[i] *= a;
  }
  return QSIM_HIP_OK;
}

int qsim_hip_traj_free(void* handle) {
  auto* b = static_cast<TrajBatch*>(handle);
  if (b == nullptr) return QSIM_HIP_OK;
  QHIP_CHECK(hipStreamSynchronize(Stream()));
  Release(b);
  return QSIM_HIP_OK;
}

}  // extern "C"
