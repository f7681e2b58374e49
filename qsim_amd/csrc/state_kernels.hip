// state_kernels.hip -- state-space passes of the gfx950 backend: fills,
// elementwise updates, FP64 reductions, measurement and parallel sampling.
//
// Counterparts: StateSpaceCUDA (lib/statespace_cuda.h) and its kernels
// (lib/statespace_cuda_kernels.h), with the arithmetic of StateSpaceBasic
// (lib/statespace_basic.h).  The layout is interleaved complex, so the
// reference's layout conversions are no-ops here.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "internal.h"
#include "reduce.h"

namespace qhip {

namespace {

constexpr unsigned kBS = 256;

inline unsigned GridFor(uint64_t items, uint64_t cap = uint64_t{1} << 16) {
  uint64_t b = (items + kBS - 1) / kBS;
  return unsigned(std::max<uint64_t>(1, std::min(b, cap)));
}

template <typename C>
__global__ void __launch_bounds__(kBS)
FillKernel(C* __restrict__ s, uint64_t size, C v, uint64_t one_index, C one) {
  const uint64_t stride = uint64_t(gridDim.x) * kBS;
  for (uint64_t i = uint64_t(blockIdx.x) * kBS + threadIdx.x; i < size;
       i += stride)
    s[i] = i == one_index ? one : v;
}

template <typename C, typename FP>
__global__ void __launch_bounds__(kBS)
BulkSetKernel(C* __restrict__ s, uint64_t size, uint64_t mask, uint64_t bits,
              FP re, FP im, bool exclude) {
  const uint64_t stride = uint64_t(gridDim.x) * kBS;
  for (uint64_t i = uint64_t(blockIdx.x) * kBS + threadIdx.x; i < size;
       i += stride) {
    bool in = ((i & mask) == bits) != exclude;
    if (in) s[i] = C{re, im};
  }
}

template <typename C>
__global__ void __launch_bounds__(kBS)
AddKernel(const C* __restrict__ src, C* __restrict__ dst, uint64_t size) {
  const uint64_t stride = uint64_t(gridDim.x) * kBS;
  for (uint64_t i = uint64_t(blockIdx.x) * kBS + threadIdx.x; i < size;
       i += stride) {
    C a = src[i], b = dst[i];
    b.x += a.x;
    b.y += a.y;
    dst[i] = b;
  }
}

template <typename C, typename FP>
__global__ void __launch_bounds__(kBS)
ScaleKernel(C* __restrict__ s, uint64_t size, FP a) {
  const uint64_t stride = uint64_t(gridDim.x) * kBS;
  for (uint64_t i = uint64_t(blockIdx.x) * kBS + threadIdx.x; i < size;
       i += stride) {
    C v = s[i];
    v.x *= a;
    v.y *= a;
    s[i] = v;
  }
}

// Sweeps of the state load 16 bytes a thread, kFly of them in flight: norm of
// 27 qubits 173 us (6.2 TB/s) where one 8-byte load of each operand took 274.
// One 16-byte load: two complex64 amplitudes or one complex128.  Complex64
// states need only be aligned to an amplitude.
typedef float Pair64 __attribute__((ext_vector_type(4), aligned(8)));
template <typename C>
struct Unit;
template <>
struct Unit<float2> {
  static constexpr unsigned kAmps = 2;
  Pair64 v;
  __device__ __forceinline__ void Load(const float2* s, uint64_t u) {
    v = *reinterpret_cast<const Pair64*>(s + 2 * u);
  }
  __device__ __forceinline__ float2 At(int i) const {
    return i ? float2{v[2], v[3]} : float2{v[0], v[1]};
  }
  __device__ __forceinline__ void Set(int i, float2 a) {
    v[2 * i] = a.x;
    v[2 * i + 1] = a.y;
  }
  __device__ __forceinline__ void Store(float2* s, uint64_t u) const {
    *reinterpret_cast<Pair64*>(s + 2 * u) = v;
  }
};
template <>
struct Unit<double2> {
  static constexpr unsigned kAmps = 1;
  double2 v;
  __device__ __forceinline__ void Load(const double2* s, uint64_t u) {
    v = s[u];
  }
  __device__ __forceinline__ double2 At(int) const { return v; }
  __device__ __forceinline__ void Set(int, double2 a) { v = a; }
  __device__ __forceinline__ void Store(double2* s, uint64_t u) const {
    s[u] = v;
  }
};

// Loads in flight per thread of a reduction sweep.
constexpr int kFly = 4;

// Calls f(amplitude index, amplitude) over amplitudes [i0, i1) with the
// workgroup's threads, kFly 16-byte loads a thread in flight; i0 and i1 are
// multiples of a unit unless the range is a single amplitude.
template <typename C, typename F>
__device__ __forceinline__ void SweepRange(const C* __restrict__ s,
                                           uint64_t i0, uint64_t i1,
                                           uint64_t first, uint64_t step,
                                           F f) {
  constexpr unsigned kA = Unit<C>::kAmps;
  const uint64_t u1 = i1 / kA;
  uint64_t u = i0 / kA + first;
  for (; u + (kFly - 1) * step < u1; u += kFly * step) {
    Unit<C> x[kFly];
#pragma unroll
    for (int k = 0; k < kFly; ++k) x[k].Load(s, u + k * step);
#pragma unroll
    for (int k = 0; k < kFly; ++k)
#pragma unroll
      for (unsigned j = 0; j < kA; ++j) f((u + k * step) * kA + j, x[k].At(j));
  }
  for (; u < u1; u += step) {
    Unit<C> x;
    x.Load(s, u);
#pragma unroll
    for (unsigned j = 0; j < kA; ++j) f(u * kA + j, x.At(j));
  }
  if (i1 % kA != 0 && first == 0) f(i1 - 1, s[i1 - 1]);  // one amplitude
}

// The amplitudes with (i & mask) == bits, enumerated: item t is t with zero
// bits inserted at the measured qubits at or above kSkipQubit, OR cbits;
// measured qubits below it (within a 64-byte half line) are a test.
struct KeepGeom {
  uint64_t items;
  uint64_t cbits;
  uint64_t low_mask, low_bits;
  unsigned nins;
  unsigned ins[40];
};

// Norm of the kept amplitudes (FP products, FP64 sums), as partial sums.
constexpr unsigned kKeptBlocks = 1024;
template <typename C>
__global__ void __launch_bounds__(kBS)
KeptNormKernel(const C* __restrict__ s, KeepGeom g,
               double* __restrict__ part) {
  double acc = 0;
  const uint64_t stride = uint64_t(gridDim.x) * kBS;
  uint64_t t = uint64_t(blockIdx.x) * kBS + threadIdx.x;
  auto add = [&](uint64_t i, const C& v) {
    if ((i & g.low_mask) == g.low_bits) acc += double(v.x * v.x + v.y * v.y);
  };
  for (; t + 3 * stride < g.items; t += 4 * stride) {
    C v[4];
    uint64_t i[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      i[k] = InsertZeros(t + k * stride, g.ins, g.nins) | g.cbits;
      v[k] = s[i[k]];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) add(i[k], v[k]);
  }
  for (; t < g.items; t += stride) {
    const uint64_t i = InsertZeros(t, g.ins, g.nins) | g.cbits;
    add(i, s[i]);
  }
  acc = BlockSum<kBS>(acc);
  if (threadIdx.x == 0) part[blockIdx.x] = acc;
}

// Zero amplitudes outside (i & mask) == bits, scale the rest by 1/sqrt of
// their norm rounded to the element type
// (lib/statespace_cuda_kernels.h:273-285 semantics); amplitudes to be zeroed
// are not read.  Every workgroup adds up the norm's partial sums itself, so
// nothing waits on the host between the two passes.
constexpr unsigned kCollapseBlocks = 8192;
template <typename C, typename FP>
__global__ void __launch_bounds__(kBS)
CollapseKernel(C* __restrict__ s, uint64_t size, uint64_t mask, uint64_t bits,
               const double* __restrict__ part, unsigned nparts) {
  __shared__ double norm_s;
  double norm = 0;
  for (unsigned i = threadIdx.x; i < nparts; i += kBS) norm += part[i];
  norm = BlockSum<kBS>(norm);
  if (threadIdx.x == 0) norm_s = norm;
  __syncthreads();
  const FP a = FP(1.0 / sqrt(norm_s));
  constexpr unsigned kA = Unit<C>::kAmps;
  auto keep = [&](uint64_t i) { return (i & mask) == bits; };
  auto scaled = [&](const C& v) { return C{v.x * a, v.y * a}; };
  const uint64_t stride = uint64_t(gridDim.x) * kBS;
  const uint64_t first = uint64_t(blockIdx.x) * kBS + threadIdx.x;
  for (uint64_t u = first; u < size / kA; u += stride) {
    bool any = false;
#pragma unroll
    for (unsigned j = 0; j < kA; ++j) any = any || keep(u * kA + j);
    Unit<C> x;
    if (any) x.Load(s, u);
#pragma unroll
    for (unsigned j = 0; j < kA; ++j)
      x.Set(j, keep(u * kA + j) ? scaled(x.At(j)) : C{0, 0});
    x.Store(s, u);
  }
  if (size % kA != 0 && first == 0) {
    s[size - 1] = keep(size - 1) ? scaled(s[size - 1]) : C{0, 0};
  }
}

// Partial sums of |s_i|^2 over contiguous ranges of `part` amplitudes, one
// workgroup per range; FP products (lib/statespace_basic.h:237-273), FP64
// sums.  out may be host memory.
// 26 qubits: 131 us (178 with one 8-byte load a thread in flight).
constexpr int kPartsNT = 512;
template <typename C>
__global__ void __launch_bounds__(kPartsNT)
NormPartsKernel(const C* __restrict__ s, uint64_t part,
                double* __restrict__ out) {
  const uint64_t i0 = uint64_t(blockIdx.x) * part;
  double acc = 0;
  SweepRange(s, i0, i0 + part, threadIdx.x, kPartsNT,
             [&](uint64_t, const C& v) {
               acc += double(v.x * v.x + v.y * v.y);
             });
  acc = BlockSum<kPartsNT>(acc);
  if (threadIdx.x == 0) out[blockIdx.x] = acc;
}

// What sampling needs of the state, in one read of it: per sample block of
// `part` amplitudes the sum of |s_i|^2 with FP64 products
// (lib/statespace_basic.h:203-222) and the sum with FP products, whose total
// is the norm that scales the draws.  One wave per block: a draw then reads
// half a block of kSampleBlock = 1024 amplitudes on average (20000 draws of a
// 28-qubit state: 151 us with blocks of 4096).
constexpr uint64_t kSampleBlock = 1024;
template <typename C>
__global__ void __launch_bounds__(kBS)
SampleSumsKernel(const C* __restrict__ s, uint64_t part, uint64_t nblocks,
                 double* __restrict__ sums, double* __restrict__ norms) {
  const uint64_t b = uint64_t(blockIdx.x) * (kBS / 64) + (threadIdx.x >> 6);
  if (b >= nblocks) return;
  const unsigned l = threadIdx.x & 63;
  double sum = 0, norm = 0;
  SweepRange(s, b * part, (b + 1) * part, l, 64, [&](uint64_t, const C& v) {
    sum += double(v.x) * double(v.x) + double(v.y) * double(v.y);
    norm += double(v.x * v.x + v.y * v.y);
  });
  sum = WaveSum(sum);
  norm = WaveSum(norm);
  if (l == 0) {
    sums[b] = sum;
    norms[b] = norm;
  }
}

// sum conj(a_i) b_i (REAL: real part only) with FP64 accumulation
// (lib/statespace_cuda_kernels.h:181-190 via lib/util_cuda.h:101-122).  SAME:
// a is b (the norm), read once.
template <typename C, bool REAL, bool SAME>
__global__ void __launch_bounds__(kBS)
DotKernel(const C* __restrict__ a, const C* __restrict__ b, uint64_t size,
          Dbl2* __restrict__ part) {
  constexpr unsigned kA = Unit<C>::kAmps;
  Dbl2 acc;
  auto add = [&](const C& u, const C& v) {
    acc.x += double(u.x * v.x + u.y * v.y);
    if (!REAL) acc.y += double(u.x * v.y - u.y * v.x);
  };
  const uint64_t step = uint64_t(gridDim.x) * kBS;
  const uint64_t first = uint64_t(blockIdx.x) * kBS + threadIdx.x;
  if (SAME) {
    SweepRange(a, 0, size, first, step, [&](uint64_t, const C& v) { add(v, v); });
  } else {
    const uint64_t units = size / kA;
    uint64_t u = first;
    for (; u + (kFly - 1) * step < units; u += kFly * step) {
      Unit<C> x[kFly], y[kFly];
#pragma unroll
      for (int k = 0; k < kFly; ++k) {
        x[k].Load(a, u + k * step);
        y[k].Load(b, u + k * step);
      }
#pragma unroll
      for (int k = 0; k < kFly; ++k)
#pragma unroll
        for (unsigned j = 0; j < kA; ++j) add(x[k].At(j), y[k].At(j));
    }
    for (; u < units; u += step) {
      Unit<C> x, y;
      x.Load(a, u);
      y.Load(b, u);
#pragma unroll
      for (unsigned j = 0; j < kA; ++j) add(x.At(j), y.At(j));
    }
    if (size % kA != 0 && first == 0) add(a[size - 1], b[size - 1]);
  }
  acc = BlockSum<kBS>(acc);
  if (threadIdx.x == 0) part[blockIdx.x] = acc;
}

// Finds, inside amplitudes [i0, i1), the first k with r < running sum of
// |s|^2 (FP64, in index order); writes k or ~0 when the range ends first.
// One workgroup of 16 waves narrows the range 16-fold per step, each wave
// summing a contiguous sixteenth, until a wave's inclusive scan of 64
// amplitudes ends it: the range is read little more than once, in parallel.
// (One scan of the whole range, 256 amplitudes per step: 65 us for 2^16
// amplitudes.)
// A piece is entered because its sum puts r inside it, so one of its
// amplitudes is not zero.  Its parts, added in another order, may fall short
// of r by rounding: then its last part that is not zero is taken, down to its
// last such amplitude, never an index of probability zero.
template <typename C>
__global__ void __launch_bounds__(1024)
FindFirstKernel(const C* __restrict__ s, uint64_t i0, uint64_t i1, double r,
                uint64_t* __restrict__ out) {
  __shared__ double tot[16];
  __shared__ uint64_t lo_s, hi_s;
  __shared__ double before_s;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  auto prob = [&](uint64_t i) {
    const C v = s[i];
    return double(v.x * v.x + v.y * v.y);
  };
  double before = 0;  // the sum ahead of lo
  uint64_t lo = i0, hi = i1;
  bool none = false, inside = false;  // inside: a piece was entered
  while (hi - lo > 64 && !none) {
    const uint64_t piece = (hi - lo + 15) / 16;
    const uint64_t a = std::min(hi, lo + w * piece);
    const uint64_t b = std::min(hi, a + piece);
    double acc = 0;
    uint64_t i = a + l;
    for (; i + 448 < b; i += 512) {
      double p[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) p[k] = prob(i + 64 * k);
#pragma unroll
      for (int k = 0; k < 8; ++k) acc += p[k];
    }
    for (; i < b; i += 64) acc += prob(i);
    acc = WaveSum(acc);
    if (l == 0) tot[w] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
      double c = before, c_last = before;
      int k = 0, last = 16;
      while (k < 16 && !(r < c + tot[k])) {
        if (tot[k] > 0) {
          last = k;
          c_last = c;
        }
        c += tot[k++];
      }
      if (k == 16 && inside) {
        k = last;
        c = c_last;
      }
      lo_s = k < 16 ? std::min(hi, lo + k * piece) : hi;
      hi_s = k < 16 ? std::min(hi, lo + (k + 1) * piece) : hi;
      before_s = c;
    }
    __syncthreads();
    none = lo_s == hi_s;
    inside = true;
    lo = lo_s;
    hi = hi_s;
    before = before_s;
    __syncthreads();
  }
  if (w != 0) return;
  uint64_t found = ~uint64_t{0};
  if (!none) {
    const uint64_t i = lo + l;
    const double p = i < hi ? prob(i) : 0.0;
    const double incl = WaveInclusiveScan(p);
    const unsigned long long ballot = __ballot(i < hi && r < before + incl);
    const unsigned long long some = __ballot(p > 0);
    if (ballot != 0) {
      found = lo + __builtin_ctzll(ballot);
    } else if (inside && some != 0) {
      found = lo + 63 - __builtin_clzll(some);
    }
  }
  if (l == 0) out[0] = found;
}

// Exclusive scan of v over a workgroup of 256; the total in `all`.
__device__ inline double BlockExclusiveScan(double v, double& all) {
  __shared__ double wave_tot[4];
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const double incl = WaveInclusiveScan(v);
  __syncthreads();
  if (l == 63) wave_tot[w] = incl;
  __syncthreads();
  double before = 0;
  all = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (j < w) before += wave_tot[j];
    all += wave_tot[j];
  }
  return before + (incl - v);
}

// Prefix sums of the sample blocks in two levels: workgroup w scans its
// kScanSpan blocks (inner[b], from zero) and leaves their totals, the next
// launch scans the workgroups' (outer[w]) and adds up the norm.  A block's
// prefix is outer[b / kScanSpan] + inner[b].  (One workgroup that scanned
// everything took 108 us for 2^16 blocks.)
constexpr unsigned kScanSpan = 1024;
__global__ void __launch_bounds__(256)
SampleScanKernel(const double* __restrict__ sums,
                 const double* __restrict__ norms, uint64_t count,
                 double* __restrict__ inner, Dbl2* __restrict__ totals) {
  const uint64_t b0 = uint64_t(blockIdx.x) * kScanSpan + 4 * threadIdx.x;
  double v[4], sum = 0, nrm = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    v[k] = b0 + k < count ? sums[b0 + k] : 0.0;
    sum += v[k];
    nrm += b0 + k < count ? norms[b0 + k] : 0.0;
  }
  double all;
  double p = BlockExclusiveScan(sum, all);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (b0 + k < count) inner[b0 + k] = p;
    p += v[k];
  }
  nrm = BlockSum<256>(nrm);
  if (threadIdx.x == 0) totals[blockIdx.x] = Dbl2(all, nrm);
}

__global__ void __launch_bounds__(256)
SampleOuterKernel(const Dbl2* __restrict__ totals, unsigned spans,
                  double* __restrict__ outer, double* __restrict__ norm) {
  double carry = 0, nrm = 0, all;
  for (unsigned c0 = 0; c0 < spans; c0 += 256) {
    const unsigned i = c0 + threadIdx.x;
    const Dbl2 t = i < spans ? totals[i] : Dbl2();
    nrm += t.y;
    const double q = BlockExclusiveScan(t.x, all);
    if (i < spans) outer[i] = carry + q;
    carry += all;
  }
  nrm = BlockSum<256>(nrm);
  if (threadIdx.x == 0) *norm = nrm;
}

// One wave per draw: binary searches of the two prefix levels, then an
// in-order walk of the block, 512 amplitudes a step (8 consecutive ones per
// lane, FP64).  A draw that the rounding of the block sums places past its
// block continues in the next block; a draw beyond the last amplitude maps
// to size - 1 (lib/statespace_basic.h:227-229).
template <typename C>
__global__ void __launch_bounds__(64)
SampleKernel(const C* __restrict__ s, uint64_t size, uint64_t sblock,
             const double* __restrict__ inner,
             const double* __restrict__ outer, uint64_t nblocks,
             const double* __restrict__ draws, uint64_t* __restrict__ out) {
  const uint64_t d = blockIdx.x;
  const double r = draws[d];
  const int l = threadIdx.x;
  // Largest index in [lo, hi) whose prefix is <= r (or lo).
  auto search = [&](uint64_t lo, uint64_t hi, auto prefix) {
    while (hi - lo > 1) {
      const uint64_t mid = (lo + hi) / 2;
      if (prefix(mid) <= r) lo = mid;
      else hi = mid;
    }
    return lo;
  };
  const uint64_t span =
      search(0, (nblocks + kScanSpan - 1) / kScanSpan,
             [&](uint64_t i) { return outer[i]; });
  const double o = outer[span];
  const uint64_t b =
      search(span * kScanSpan, std::min(nblocks, (span + 1) * kScanSpan),
             [&](uint64_t i) { return o + inner[i]; });
  double carry = o + inner[b];
  uint64_t result = size - 1;
  // The match lies in block b, or in b + 1 when rounding of the block sums
  // moved it; the walk never goes further (a NaN state ends here too).
  const uint64_t iend = std::min(size, (b + 2) * sblock);
  for (uint64_t i0 = b * sblock; i0 < iend; i0 += 512) {
    const uint64_t i = i0 + 8 * l;
    double p[8], mine = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      p[k] = 0;
      if (i + k < iend) {
        const C v = s[i + k];
        p[k] = double(v.x) * double(v.x) + double(v.y) * double(v.y);
      }
      mine += p[k];
    }
    const double incl = WaveInclusiveScan(mine);
    double c = carry + (incl - mine);
    // The first of this lane's amplitudes that passes the draw.
    int hit = 8;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      c += p[k];
      if (hit == 8 && i + k < iend && r < c) hit = k;
    }
    const unsigned long long ballot = __ballot(hit < 8);
    if (ballot != 0) {
      const int who = __builtin_ctzll(ballot);
      result = i0 + 8 * who + __shfl(hit, who, 64);
      break;
    }
    carry += __shfl(incl, 63, 64);
  }
  if (l == 0) out[d] = result;
}

template <typename FP>
using C_t = typename Cplx<FP>::T;

// Blocks of a reduction pass, kFly 16-byte units a thread and turn: at most
// kReduceBlocks partial sums (eight workgroups a CU of 256).
constexpr unsigned kReduceBlocks = 2047;
template <typename FP>
unsigned ReduceBlocks(uint64_t size) {
  return GridFor(size / Unit<C_t<FP>>::kAmps / kFly, kReduceBlocks);
}

// Partial sums of a dot product, one per workgroup, into `part`; returns
// their number.
template <typename FP>
unsigned LaunchDot(const C_t<FP>* a, const C_t<FP>* b, uint64_t size,
                   bool real, Dbl2* part) {
  // A norm reads one state: half the workgroups (29 qubits: 709 us complex64,
  // 1396 complex128, against 737 and 1430; two states 1400 and 2776 against
  // 1383 and 2743).
  const unsigned most = real && a == b ? kReduceBlocks / 2 : kReduceBlocks;
  const dim3 blocks(std::min(ReduceBlocks<FP>(size), most)), bs(kBS);
  const hipStream_t st = Stream();
  if (real && a == b)
    hipLaunchKernelGGL((DotKernel<C_t<FP>, true, true>), blocks, bs, 0, st, a,
                       b, size, part);
  else if (real)
    hipLaunchKernelGGL((DotKernel<C_t<FP>, true, false>), blocks, bs, 0, st, a,
                       b, size, part);
  else
    hipLaunchKernelGGL((DotKernel<C_t<FP>, false, false>), blocks, bs, 0, st,
                       a, b, size, part);
  return blocks.x;
}

template <typename FP>
int Reduce(const C_t<FP>* a, const C_t<FP>* b, uint64_t size, bool real,
           double* re, double* im) {
  std::lock_guard<std::mutex> lock(ScratchLock());
  const unsigned count =
      LaunchDot<FP>(a, b, size, real, static_cast<Dbl2*>(HostResult()));
  QHIP_LAUNCHED("DotKernel");
  Dbl2 r;
  QHIP_TRY(HostTotal(count, &r));
  *re = r.x;
  if (im) *im = r.y;
  return QSIM_HIP_OK;
}

// ---- fixed scratch of the no-allocation reductions -------------------------
//
// The partial sums of DotStatic live in this array (one per device, held
// until the process ends), as (re, im) pairs.  Its name is a host-side stand-in: host code
// uses only the device address hipGetSymbolAddress gives for it
// (g_static_scratch, taken once when the library is initialised).
constexpr unsigned kStaticScratchDbl2 = 2048;
static_assert(kStaticScratchDbl2 >= kReduceBlocks + 1, "reduction scratch");
static_assert(kReduceBlocks * sizeof(Dbl2) <= kHostResultBytes, "partials");
static __device__ __align__(256) double scratch[2 * kStaticScratchDbl2];
Dbl2* g_static_scratch = nullptr;
std::mutex g_static_scratch_mu;

// Number of equal index ranges for partial norms.
unsigned NumParts(unsigned n) {
  uint64_t size = uint64_t{1} << n;
  uint64_t p = size / 1024;
  return unsigned(std::max<uint64_t>(1, std::min<uint64_t>(p, 1024)));
}

}  // namespace

// ---- entry points used by api.hip -----------------------------------------

template <typename FP>
int Fill(C_t<FP>* s, unsigned n, int what) {
  // what: 0 zeros, 1 |0>, 2 uniform
  uint64_t size = uint64_t{1} << n;
  C_t<FP> v{0, 0}, one{0, 0};
  uint64_t one_index = ~uint64_t{0};
  if (what == 1) {
    one = C_t<FP>{1, 0};
    one_index = 0;
  } else if (what == 2) {
    // lib/statespace_cuda.h:115-127: 1/sqrt(2^n) rounded to the element type.
    v = C_t<FP>{FP(1.0 / std::sqrt(double(size))), 0};
  }
  hipLaunchKernelGGL((FillKernel<C_t<FP>>), dim3(GridFor(size)), dim3(kBS), 0,
                     Stream(), s, size, v, one_index, one);
  QHIP_LAUNCHED("FillKernel");
  return QSIM_HIP_OK;
}

template <typename FP>
int BulkSet(C_t<FP>* s, unsigned n, uint64_t mask, uint64_t bits, double re,
            double im, bool exclude) {
  uint64_t size = uint64_t{1} << n;
  hipLaunchKernelGGL((BulkSetKernel<C_t<FP>, FP>), dim3(GridFor(size)),
                     dim3(kBS), 0, Stream(), s, size, mask, bits, FP(re),
                     FP(im), exclude);
  QHIP_LAUNCHED("BulkSetKernel");
  return QSIM_HIP_OK;
}

template <typename FP>
int Add(const C_t<FP>* src, C_t<FP>* dst, unsigned n) {
  uint64_t size = uint64_t{1} << n;
  hipLaunchKernelGGL((AddKernel<C_t<FP>>), dim3(GridFor(size)), dim3(kBS), 0,
                     Stream(), src, dst, size);
  QHIP_LAUNCHED("AddKernel");
  return QSIM_HIP_OK;
}

template <typename FP>
int Scale(C_t<FP>* s, unsigned n, double a) {
  uint64_t size = uint64_t{1} << n;
  hipLaunchKernelGGL((ScaleKernel<C_t<FP>, FP>), dim3(GridFor(size)),
                     dim3(kBS), 0, Stream(), s, size, FP(a));
  QHIP_LAUNCHED("ScaleKernel");
  return QSIM_HIP_OK;
}

template <typename FP>
int Dot(const C_t<FP>* a, const C_t<FP>* b, unsigned n, bool real, double* re,
        double* im) {
  return Reduce<FP>(a, b, uint64_t{1} << n, real, re, im);
}

template <typename FP>
int DotStatic(const C_t<FP>* a, const C_t<FP>* b, unsigned n, bool real,
              double* re, double* im) {
  const uint64_t size = uint64_t{1} << n;
  if (g_static_scratch == nullptr) {
    SetError("no-allocation reduction: the fixed scratch was not set up "
             "(library not initialised)");
    return QSIM_HIP_ERR_RUNTIME;
  }
  std::lock_guard<std::mutex> lock(g_static_scratch_mu);
  Dbl2* part = g_static_scratch;
  const unsigned count = LaunchDot<FP>(a, b, size, real, part + 1);
  QHIP_LAUNCHED("DotKernel");
  hipLaunchKernelGGL((FinalSumKernel<Dbl2>), dim3(1), dim3(256), 0, Stream(),
                     part + 1, count, part);
  QHIP_LAUNCHED("FinalSumKernel");
  Dbl2 r;
  QHIP_CHECK(hipMemcpyAsync(&r, part, sizeof(Dbl2), hipMemcpyDeviceToHost,
                            Stream()));
  QHIP_CHECK(hipStreamSynchronize(Stream()));
  *re = r.x;
  if (im) *im = r.y;
  return QSIM_HIP_OK;
}

int InitStaticScratch() {
  void* p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess) return HipFail(e, "hipGetSymbolAddress(scratch)");
  g_static_scratch = static_cast<Dbl2*>(p);
  return QSIM_HIP_OK;
}

unsigned PartialNormCount(unsigned n) { return NumParts(n); }

template <typename FP>
int PartialNorms(const C_t<FP>* s, unsigned n, double* out) {
  std::lock_guard<std::mutex> lock(ScratchLock());
  unsigned parts = NumParts(n);
  uint64_t part = (uint64_t{1} << n) / parts;
  double* host = static_cast<double*>(HostResult());
  hipLaunchKernelGGL((NormPartsKernel<C_t<FP>>), dim3(parts), dim3(kPartsNT), 0,
                     Stream(), s, part, host);
  QHIP_LAUNCHED("NormPartsKernel");
  QHIP_CHECK(hipStreamSynchronize(Stream()));
  std::copy(host, host + parts, out);
  return QSIM_HIP_OK;
}

template <typename FP>
int FindMeasuredBits(const C_t<FP>* s, unsigned n, unsigned m, double r,
                     uint64_t mask, uint64_t* out) {
  unsigned parts = NumParts(n);
  if (m >= parts) {
    SetError("partial-norm index %u out of range (%u)", m, parts);
    return QSIM_HIP_ERR_ARG;
  }
  std::lock_guard<std::mutex> lock(ScratchLock());
  uint64_t part = (uint64_t{1} << n) / parts;
  uint64_t* host = static_cast<uint64_t*>(HostResult());
  hipLaunchKernelGGL((FindFirstKernel<C_t<FP>>), dim3(1), dim3(1024), 0,
                     Stream(), s, uint64_t(m) * part, uint64_t(m + 1) * part, r,
                     host);
  QHIP_LAUNCHED("FindFirstKernel");
  QHIP_CHECK(hipStreamSynchronize(Stream()));
  uint64_t k = *host;
  // Past the end of the range (rounding): the last index of the range, as
  // lib/statespace_basic.h:291-294 returns.
  if (k == ~uint64_t{0}) k = uint64_t(m + 1) * part - 1;
  *out = k & mask;
  return QSIM_HIP_OK;
}

template <typename FP>
int Collapse(C_t<FP>* s, unsigned n, uint64_t mask, uint64_t bits) {
  const uint64_t size = uint64_t{1} << n;
  KeepGeom g{};
  const uint64_t skip = ~uint64_t{sizeof(FP) == 4 ? 7u : 3u};
  g.items = size;
  // Qubits from n up are zero in every index: a mask there tests bits only.
  for (unsigned q = 0; q < n; ++q) {
    if (!((mask & skip) >> q & 1)) continue;
    g.ins[g.nins++] = q;
    g.items >>= 1;
  }
  g.low_mask = mask & ~(skip & (size - 1));
  g.cbits = bits & mask & skip & (size - 1);
  // A bit wanted outside the mask matches nothing.
  g.low_bits = bits & ~(mask & skip & (size - 1));
  std::lock_guard<std::mutex> lock(ScratchLock());
  const unsigned blocks = GridFor(g.items / 4, kKeptBlocks);
  double* part =
      static_cast<double*>(DeviceScratch(sizeof(double) * kKeptBlocks));
  if (part == nullptr) return QSIM_HIP_ERR_OOM;
  hipLaunchKernelGGL((KeptNormKernel<C_t<FP>>), dim3(blocks), dim3(kBS), 0,
                     Stream(), s, g, part);
  QHIP_LAUNCHED("KeptNormKernel");
  hipLaunchKernelGGL((CollapseKernel<C_t<FP>, FP>),
                     dim3(GridFor(size / Unit<C_t<FP>>::kAmps, kCollapseBlocks)),
                     dim3(kBS), 0,
                     Stream(), s, size, mask, bits, part, blocks);
  QHIP_LAUNCHED("CollapseKernel");
  // The partial sums belong to the scratch lock's holder.
  QHIP_CHECK(hipStreamSynchronize(Stream()));
  return QSIM_HIP_OK;
}

namespace {

// Scratch of a sampling call: block sums and norms, the two prefix levels,
// then draws and results.
struct SampleScratch {
  uint64_t size, sblock, nblocks, spans;
  double *sums, *norms, *inner, *outer, *draws;
  Dbl2* totals;
  uint64_t* out;
};

int SampleLayout(unsigned n, uint64_t num, SampleScratch& c) {
  c.size = uint64_t{1} << n;
  c.sblock = std::min(c.size, kSampleBlock);
  c.nblocks = c.size / c.sblock;
  c.spans = (c.nblocks + kScanSpan - 1) / kScanSpan;
  char* base = static_cast<char*>(DeviceScratch(
      sizeof(Dbl2) * c.spans +
      sizeof(double) * (3 * c.nblocks + c.spans + 2 * num)));
  if (base == nullptr) return QSIM_HIP_ERR_OOM;
  c.totals = reinterpret_cast<Dbl2*>(base);
  c.sums = reinterpret_cast<double*>(c.totals + c.spans);
  c.norms = c.sums + c.nblocks;
  c.inner = c.norms + c.nblocks;
  c.outer = c.inner + c.nblocks;
  c.draws = c.outer + c.spans;
  c.out = reinterpret_cast<uint64_t*>(c.draws + num);
  return QSIM_HIP_OK;
}

// The state's sums, prefixes and (in *HostResult()) norm.
template <typename FP>
int SampleSums(const C_t<FP>* s, const SampleScratch& c) {
  hipLaunchKernelGGL((SampleSumsKernel<C_t<FP>>),
                     dim3(unsigned((c.nblocks + 3) / 4)), dim3(kBS), 0,
                     Stream(), s, c.sblock, c.nblocks, c.sums, c.norms);
  QHIP_LAUNCHED("SampleSumsKernel");
  hipLaunchKernelGGL(SampleScanKernel, dim3(unsigned(c.spans)), dim3(256), 0,
                     Stream(), c.sums, c.norms, c.nblocks, c.inner, c.totals);
  QHIP_LAUNCHED("SampleScanKernel");
  hipLaunchKernelGGL(SampleOuterKernel, dim3(1), dim3(256), 0, Stream(),
                     c.totals, unsigned(c.spans), c.outer,
                     static_cast<double*>(HostResult()));
  QHIP_LAUNCHED("SampleOuterKernel");
  return QSIM_HIP_OK;
}

template <typename FP>
int SampleDraws(const C_t<FP>* s, const SampleScratch& c, const double* draws,
                uint64_t num, uint64_t* out) {
  QHIP_CHECK(hipMemcpyAsync(c.draws, draws, sizeof(double) * num,
                            hipMemcpyHostToDevice, Stream()));
  hipLaunchKernelGGL((SampleKernel<C_t<FP>>), dim3(unsigned(num)), dim3(64), 0,
                     Stream(), s, c.size, c.sblock, c.inner, c.outer,
                     c.nblocks, c.draws, c.out);
  QHIP_LAUNCHED("SampleKernel");
  QHIP_CHECK(hipMemcpyAsync(out, c.out, sizeof(uint64_t) * num,
                            hipMemcpyDeviceToHost, Stream()));
  QHIP_CHECK(hipStreamSynchronize(Stream()));
  return QSIM_HIP_OK;
}

}  // namespace

template <typename FP>
int Sample(const C_t<FP>* s, unsigned n, const double* draws, uint64_t num,
           uint64_t* out) {
  if (num == 0) return QSIM_HIP_OK;
  std::lock_guard<std::mutex> lock(ScratchLock());
  SampleScratch c;
  QHIP_TRY(SampleLayout(n, num, c));
  QHIP_TRY(SampleSums<FP>(s, c));
  return SampleDraws<FP>(s, c, draws, num, out);
}

template <typename FP>
int SampleSeeded(const C_t<FP>* s, unsigned n, uint64_t num,
                 const std::function<void()>& draws, std::vector<double>& rs,
                 uint64_t* out) {
  // Beside the device's sums, with the scratch buffer held, unless they take
  // much longer (20000 draws 0.3 ms): other threads need it meanwhile.
  const bool ahead = num > (uint64_t{1} << 20);
  if (ahead) draws();
  std::lock_guard<std::mutex> lock(ScratchLock());
  SampleScratch c;
  QHIP_TRY(SampleLayout(n, num, c));
  QHIP_TRY(SampleSums<FP>(s, c));
  if (!ahead) draws();
  QHIP_CHECK(hipStreamSynchronize(Stream()));
  const double norm = *static_cast<double*>(HostResult());
  for (double& r : rs) r *= norm;
  return SampleDraws<FP>(s, c, rs.data(), num, out);
}

// out[j] = s[idx[j]]: the amplitudes of a batch of bitstrings in one pass.
template <typename C>
__global__ void __launch_bounds__(kBS)
GatherKernel(const C* __restrict__ s, const uint64_t* __restrict__ idx,
             uint64_t count, C* __restrict__ out) {
  const uint64_t stride = uint64_t(gridDim.x) * kBS;
  for (uint64_t j = uint64_t(blockIdx.x) * kBS + threadIdx.x; j < count;
       j += stride) {
    out[j] = s[idx[j]];
  }
}

// Amplitudes of `count` indices (host arrays; indices checked by the caller)
// in chunks that fit the scratch buffer: one upload, one gather launch and
// one download per chunk.
template <typename FP>
int Gather(const C_t<FP>* s, const uint64_t* idx, uint64_t count,
           C_t<FP>* out) {
  constexpr uint64_t kChunk = uint64_t{1} << 20;
  std::lock_guard<std::mutex> lock(ScratchLock());
  const uint64_t cap = std::min(count, kChunk);
  char* base = static_cast<char*>(
      DeviceScratch(cap * (sizeof(uint64_t) + sizeof(C_t<FP>))));
  if (base == nullptr) return QSIM_HIP_ERR_OOM;
  uint64_t* d_idx = reinterpret_cast<uint64_t*>(base);
  C_t<FP>* d_out = reinterpret_cast<C_t<FP>*>(d_idx + cap);
  for (uint64_t j0 = 0; j0 < count; j0 += cap) {
    const uint64_t m = std::min(cap, count - j0);
    QHIP_CHECK(hipMemcpyAsync(d_idx, idx + j0, sizeof(uint64_t) * m,
                              hipMemcpyHostToDevice, Stream()));
    hipLaunchKernelGGL((GatherKernel<C_t<FP>>), dim3(GridFor(m)), dim3(kBS), 0,
                       Stream(), s, d_idx, m, d_out);
    QHIP_LAUNCHED("GatherKernel");
    QHIP_CHECK(hipMemcpyAsync(out + j0, d_out, sizeof(C_t<FP>) * m,
                              hipMemcpyDeviceToHost, Stream()));
    QHIP_CHECK(hipStreamSynchronize(Stream()));
  }
  return QSIM_HIP_OK;
}

#define QHIP_INSTANTIATE(FP)                                                   \
  template int Fill<FP>(C_t<FP>*, unsigned, int);                              \
  template int BulkSet<FP>(C_t<FP>*, unsigned, uint64_t, uint64_t, double,     \
                           double, bool);                                      \
  template int Add<FP>(const C_t<FP>*, C_t<FP>*, unsigned);                    \
  template int Scale<FP>(C_t<FP>*, unsigned, double);                          \
  template int Dot<FP>(const C_t<FP>*, const C_t<FP>*, unsigned, bool,         \
                       double*, double*);                                      \
  template int DotStatic<FP>(const C_t<FP>*, const C_t<FP>*, unsigned, bool,   \
                             double*, double*);                                \
  template int PartialNorms<FP>(const C_t<FP>*, unsigned, double*);            \
  template int FindMeasuredBits<FP>(const C_t<FP>*, unsigned, unsigned,        \
                                    double, uint64_t, uint64_t*);              \
  template int Collapse<FP>(C_t<FP>*, unsigned, uint64_t, uint64_t);           \
  template int Sample<FP>(const C_t<FP>*, unsigned, const double*, uint64_t,   \
                          uint64_t*);                                          \
  template int SampleSeeded<FP>(const C_t<FP>*, unsigned, uint64_t,            \
                                const std::function<void()>&,                  \
                                std::vector<double>&, uint64_t*);              \
  template int Gather<FP>(const C_t<FP>*, const uint64_t*, uint64_t, C_t<FP>*);

template <typename D, typename S>
__global__ void __launch_bounds__(kBS)
ConvertKernel(D* __restrict__ dst, const S* __restrict__ src, uint64_t size) {
  const uint64_t stride = uint64_t(gridDim.x) * kBS;
  for (uint64_t i = uint64_t(blockIdx.x) * kBS + threadIdx.x; i < size;
       i += stride) {
    S v = src[i];
    dst[i] = D{decltype(dst->x)(v.x), decltype(dst->x)(v.y)};
  }
}

int Convert(void* dst, int dprec, const void* src, int sprec, unsigned n) {
  const uint64_t size = uint64_t{1} << n;
  const dim3 grid(GridFor(size));
  if (dprec == QSIM_HIP_F64 && sprec == QSIM_HIP_F32) {
    hipLaunchKernelGGL((ConvertKernel<double2, float2>), grid, dim3(kBS), 0,
                       Stream(), (double2*)dst, (const float2*)src, size);
  } else if (dprec == QSIM_HIP_F32 && sprec == QSIM_HIP_F64) {
    hipLaunchKernelGGL((ConvertKernel<float2, double2>), grid, dim3(kBS), 0,
                       Stream(), (float2*)dst, (const double2*)src, size);
  } else if (dprec == QSIM_HIP_F32) {
    hipLaunchKernelGGL((ConvertKernel<float2, float2>), grid, dim3(kBS), 0,
                       Stream(), (float2*)dst, (const float2*)src, size);
  } else {
    hipLaunchKernelGGL((ConvertKernel<double2, double2>), grid, dim3(kBS), 0,
                       Stream(), (double2*)dst, (const double2*)src, size);
  }
  QHIP_LAUNCHED("ConvertKernel");
  return QSIM_HIP_OK;
}

QHIP_INSTANTIATE(float)
QHIP_INSTANTIATE(double)

}  // namespace qhip
