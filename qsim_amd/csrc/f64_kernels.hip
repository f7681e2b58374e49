// f64_kernels.hip -- k = 5, 6 gate passes on complex128 states, on FP64 MFMA.
//
// Per 2^k-amplitude group out = U in is the real product C = A B of
// mfma_kernels.hip (A: the 2D x 2D real matrix, D = 2^k; B: one column per
// group), on v_mfma_f64_16x16x4f64 (exact FP64 fused multiply-adds, the rate
// of the vector unit, a quarter of its instructions).  Operand maps (verified
// on gfx950): a = A[l%16][4t + l/16], b = B[4t + l/16][l%16] for K step t,
// C register r of lane l = C[4r + l/16][l%16].
//
// Work split, as the complex64 set kernels of f16_kernels.hip: a set is the
// 2^10 (k = 5) or 2^11 amplitudes over the targets and the 5 lowest other
// qubits, so runs of 32 or more amplitudes whatever the targets.  A 256-thread
// workgroup copies a set to LDS; wave w computes 16-row blocks w, w + 4, ...
// (their rows of A stay in its registers for the whole pass) for every group
// of the set; the results go back to their slots and the set is copied out.
// The next set is loaded before the product, but the compiler holds it in
// scratch memory (80 / 144 bytes a lane) and waits for it there, so its latency
// is one of the phases.  Four (k = 5) or two workgroups share a CU.
//
// The vector kernels need a group per thread: 2^k amplitudes of 16 bytes in
// registers, and half (k = 5) or a quarter (k = 6) of the tile kernel's
// threads have one.  27 qubits: k = 6 1.65-1.83 ms (10.5 with high targets,
// 29-34 in tiles; the FP64 MFMA rate allows 0.95), k = 5 1.09-1.38 ms (3.4-3.7
// in tiles); the phases between a set's barriers bound both.  On 12-28 qubits
// k = 6 takes 0.03-0.20 of the vector kernels' time, k = 5 with a low target
// 0.2-0.4.  k = 5 with every
// target at qubit >= 5 stays on the vector kernel, which keeps a group per
// thread without LDS there: 0.92-1.08 ms against 1.27-1.38.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "internal.h"

namespace qhip {

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));

struct F64SetGeom {
  uint64_t nsets;
  unsigned pos[11];  // the set's qubits, ascending
  unsigned tmask;    // bit b: pos[b] is a target
};

template <int K>
struct F64Dims {
  static constexpr int D = 1 << K;
  static constexpr int kSetBits = K == 5 ? 10 : 11;
  static constexpr int kSet = 1 << kSetBits;
  static constexpr int kPerCu = K == 5 ? 4 : 2;  // workgroups
  static constexpr int RB = D / 8;        // 16-row blocks of the 2D rows
  static constexpr int RPW = RB / 4;      // row blocks of a wave
  static constexpr int KS = D / 2;        // K steps of 4 reals (2 members)
  static constexpr int G = kSet / D;      // groups of a set
  static constexpr int CB = G / 16;       // 16-group column blocks
};

// LDS slot of member m of group grp.  Members are a multiple of 16 bytes off
// the bank period apart, and the product's reads, fixed strides from a lane's
// base, are instruction offsets.
template <int K>
__device__ __forceinline__ unsigned F64Slot(unsigned m, unsigned grp) {
  return m * (F64Dims<K>::G + 1) + grp;
}

template <int K>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(F64Dims<K>::kPerCu)))
GateF64SetKernel(double2* __restrict__ s, F64SetGeom g,
                 const double* __restrict__ frag) {
  using Dm = F64Dims<K>;
  constexpr int kSet = Dm::kSet, kSetBits = Dm::kSetBits;
  constexpr int PERT = kSet / 256;  // amplitudes each thread copies
  __shared__ double2 buf[2][kSet + Dm::D];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const unsigned j = lane & 15;
  const unsigned half = (lane >> 5) & 1;   // member of a K step
  const unsigned comp = (lane >> 4) & 1;   // 0 real, 1 imaginary
  double a[Dm::RPW][Dm::KS];
#pragma unroll
  for (int i = 0; i < Dm::RPW; ++i)
#pragma unroll
    for (int t = 0; t < Dm::KS; ++t)
      a[i][t] = frag[((wave + 4 * i) * Dm::KS + t) * 64 + lane];
  // Copy map: element r of this thread is set-local amplitude t + 256 r.
  uint64_t goff[PERT];
  unsigned slot[PERT];
#pragma unroll
  for (int r = 0; r < PERT; ++r) {
    const unsigned x = threadIdx.x + 256u * r;
    uint64_t o = 0;
    unsigned m = 0, grp = 0, mi = 0, gi = 0;
#pragma unroll
    for (int b = 0; b < kSetBits; ++b) {
      const unsigned bit = (x >> b) & 1u;
      o |= uint64_t(bit) << g.pos[b];
      if ((g.tmask >> b) & 1u) {
        m |= bit << mi++;
      } else {
        grp |= bit << gi++;
      }
    }
    goff[r] = o;
    slot[r] = F64Slot<K>(m, grp);
  }
  double2 pre[PERT];
  auto fetch = [&](uint64_t set) {
    const double2* p = s + InsertZeros(set, g.pos, kSetBits);
#pragma unroll
    for (int r = 0; r < PERT; ++r) pre[r] = p[goff[r]];
  };
  auto put = [&](double2* b) {
#pragma unroll
    for (int r = 0; r < PERT; ++r) b[slot[r]] = pre[r];
  };
  uint64_t set = blockIdx.x;
  if (set < g.nsets) {
    fetch(set);
    put(buf[0]);
  }
  __syncthreads();
  int cur = 0;
  for (; set < g.nsets; set += gridDim.x) {
    const uint64_t nxt = set + gridDim.x;
    if (nxt < g.nsets) fetch(nxt);
    double* b = reinterpret_cast<double*>(buf[cur]);
    v4d c[Dm::RPW][Dm::CB];
#pragma unroll
    for (int i = 0; i < Dm::RPW; ++i)
#pragma unroll
      for (int n = 0; n < Dm::CB; ++n) c[i][n] = v4d{};
#pragma unroll
    for (int t = 0; t < Dm::KS; ++t) {
#pragma unroll
      for (int n = 0; n < Dm::CB; ++n) {
        const double x = b[2 * F64Slot<K>(2u * t + half, 16u * n + j) + comp];
#pragma unroll
        for (int i = 0; i < Dm::RPW; ++i)
          c[i][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i][t], x, c[i][n],
                                                         0, 0, 0);
      }
    }
    // Every wave has read the set before any result overwrites it.
    __syncthreads();
#pragma unroll
    for (int i = 0; i < Dm::RPW; ++i)
#pragma unroll
      for (int n = 0; n < Dm::CB; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          // Row 16 rb + 4 r + l/16: component comp of member 8 rb + 2 r + half.
          const unsigned m = 8u * (wave + 4 * i) + 2u * r + half;
          b[2 * F64Slot<K>(m, 16u * n + j) + comp] = c[i][n][r];
        }
    __syncthreads();
    double2* p = s + InsertZeros(set, g.pos, kSetBits);
#pragma unroll
    for (int r = 0; r < PERT; ++r) p[goff[r]] = buf[cur][slot[r]];
    if (nxt < g.nsets) put(buf[cur ^ 1]);
    __syncthreads();
    cur ^= 1;
  }
}

template <int K>
int LaunchK(double2* s, unsigned n, const unsigned* qs, const double* m) {
  using Dm = F64Dims<K>;
  constexpr int kSetBits = Dm::kSetBits;
  // frag[(rb KS + t) 64 + l] = A[16 rb + l%16][4 t + l/16], where
  // A[2r][2m] = A[2r+1][2m+1] = Re U[r][m], A[2r+1][2m] = -A[2r][2m+1] = Im.
  std::vector<double> f(size_t(Dm::RB) * Dm::KS * 64);
  for (int rb = 0; rb < Dm::RB; ++rb)
    for (int t = 0; t < Dm::KS; ++t)
      for (int l = 0; l < 64; ++l) {
        const int row = 16 * rb + l % 16, col = 4 * t + l / 16;
        const double* u = m + 2 * (size_t(row >> 1) * Dm::D + (col >> 1));
        f[(size_t(rb) * Dm::KS + t) * 64 + l] =
            (row & 1) == (col & 1) ? u[0] : (row & 1) ? u[1] : -u[1];
      }
  const size_t bytes = f.size() * sizeof(double);
  void* d = MatrixBuffer(bytes);
  if (d == nullptr) return QSIM_HIP_ERR_OOM;
  QHIP_TRY(StageMatrix(d, f.data(), bytes));
  F64SetGeom g{};
  uint64_t mask = 0;
  for (int b = 0; b < K; ++b) mask |= uint64_t{1} << qs[b];
  const uint64_t targets = mask;
  for (unsigned q = 0; __builtin_popcountll(mask) < kSetBits; ++q)
    mask |= uint64_t{1} << q;
  for (unsigned q = 0, i = 0; i < kSetBits; ++q) {
    if (!((mask >> q) & 1)) continue;
    if ((targets >> q) & 1) g.tmask |= 1u << i;
    g.pos[i++] = q;
  }
  g.nsets = uint64_t{1} << (n - kSetBits);
  // The resident workgroups, four rounds of them (2 and 16 measured alike).
  const uint64_t blocks =
      std::min<uint64_t>(g.nsets, uint64_t(NumCUs()) * Dm::kPerCu * 4);
  PassTimerBegin();
  hipLaunchKernelGGL(GateF64SetKernel<K>, dim3(unsigned(blocks)), dim3(256), 0,
                     Stream(), s, g, static_cast<const double*>(d));
  PassTimerEnd();
  QHIP_LAUNCHED("GateF64SetKernel");
  return QSIM_HIP_OK;
}

}  // namespace

int LaunchGateF64(double2* s, unsigned n, const unsigned* qs, unsigned k,
                  const double* m) {
  if (k == 5 && qs[0] >= 5) return QSIM_HIP_ERR_UNSUPPORTED;
  if (n < unsigned(k == 5 ? F64Dims<5>::kSetBits : F64Dims<6>::kSetBits)) {
    return QSIM_HIP_ERR_UNSUPPORTED;
  }
  return k == 5 ? LaunchK<5>(s, n, qs, m) : LaunchK<6>(s, n, qs, m);
}

}  // namespace qhip
