// block_tile.h -- the tile machinery of blocked passes, shared by the
// circuit kernels (block_kernels.hip) and the batched trajectory kernel
// (traj_kernels.hip): kernel shapes, the op-record layouts, the MFMA
// product of one 4-qubit op over an LDS tile (FP16 with scaling, the
// default, and split-BF16), and tile staging between HBM and LDS.
//
// Each op is a 4-qubit gate on tile-local positions (smaller gates are
// padded with identity factors on the host).  The split-BF16 form is the
// product of the gate kernels (mfma_kernels.hip): the 16 x 16 complex
// matrix becomes a real 32 x 32 A operand, 32 groups side by side the B
// operand of v_mfma_f32_32x32x16_bf16; the matrix is split in three bf16
// parts, the amplitudes in two, and Al Bh + Am Bh + Ah Bl + Ah Bh is
// accumulated in FP32.  Operand maps (verified on gfx950):
// a[e] = A[l%32][8(l/32) + e], b[e] = B[8(l/32) + e][l%32],
// C register r of lane l = C[8(r/4) + 4(l/32) + r%4][l%32].
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "internal.h"
#include "tile.h"

namespace qhip {
namespace tileop {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));

// Kernel shapes by tile qubits TB: up to 13 (64 KiB tiles), two 256-thread
// workgroups per CU; 14 (128 KiB), one 512-thread workgroup per CU.  Both
// give every thread 32 tile elements and every wave 256 registers.
template <int TB>
struct BlockShape {
  static_assert(TB == 13 || TB == 14, "tile shape");
  static constexpr int NT = TB == 13 ? 256 : 512;
  static constexpr int kWaves = NT / 64;
  static constexpr size_t kTileBytes = (size_t{1} << TB) * sizeof(float2);
};
// BF16 fragment elements of one 4-qubit op: 2 K blocks x (hi, mid, lo) x 512.
constexpr size_t kOpFrag = 2 * 3 * 512;
// One op record in 32-bit words: the fragments (1536 words); the member
// tables -- LDS byte offsets, relative to a group's slot, of the members a
// lane reads (8) and writes (8), for lane half 0 then 1 (32 words); the
// group table -- LDS byte offset of lane j's group within a batch, j < 32
// (32 words); the op's five batch-bit positions (one byte each, 2 words);
// padded to 8 KiB.  The positions travel in the record so that an op reads
// them from LDS: read from the kernel arguments (bytes at a run-time index)
// they would be vector memory loads, and waiting for them would wait for
// every tile load issued before them.
constexpr int kFragWords = int(kOpFrag / 2);
constexpr int kTableWords = 32;
constexpr int kLaneWords = 32;
constexpr int kBposWord = kFragWords + kTableWords + kLaneWords;
constexpr int kOpWords = 2048;
static_assert(kBposWord + 2 <= kOpWords, "op record");
template <int TB>
constexpr size_t BlockLds() {
  return BlockShape<TB>::kTileBytes + 2 * kOpWords * sizeof(uint32_t);
}

// The tile at LDS byte offset `b`: the kernel has no static LDS, so its
// dynamic block starts at offset 0 (checked on the host before launch), and
// an address is the offset itself, with no base to add.
typedef __attribute__((address_space(3))) v2f LdsV2f;
__device__ __forceinline__ LdsV2f* LdsAt(unsigned b) {
  return reinterpret_cast<LdsV2f*>(size_t{b});
}

// Slot of amplitude a in the LDS tile of an FP16 pass: the 16-byte unit
// a / 2 with the bits of a from position 4 up folded into its low three.
// Position 0 stays where it is, so the two amplitudes of a pair are one
// aligned 16-byte LDS access: an op with position 0 among its targets reads
// and writes pairs (on MI355X 16-byte LDS reads run at ~192 B/clock per CU
// against ~118 for 8-byte ones, writes at ~75 against ~64), and so does the
// staging.  Each unit bit hashes four positions, so every other op finds
// lane positions free of bank conflicts unless its targets are one whole
// class.  Linear over GF(2).
__host__ __device__ constexpr unsigned F16Swz(unsigned a) {
  return a ^ ((((a >> 4) ^ (a >> 7) ^ (a >> 10) ^ (a >> 13)) & 7u) << 1);
}
template <bool F16>
__device__ __forceinline__ unsigned BlockSwz(unsigned a) {
  return F16 ? F16Swz(a) : TileSwz(a);
}

// One 4-qubit op over the LDS tile.  A group (the 16 amplitudes the op
// mixes) is fixed by its bits at the tile's non-target positions; the host
// splits those positions into 5 lane positions (chosen so that the 32
// groups of a batch fall into distinct LDS banks) and tb - 9 batch
// positions `bp`.  Wave `wave` (wave-uniform) of `nwaves` takes batches
// bt = wave, wave + nwaves, ...; lanes j and j + 32 serve the batch's j-th
// group.  `f` holds the op's fragments (hi, mid, lo per K block); rd / wr
// are this lane's member offsets with its group's offset already folded in
// (LDS bytes).  TileSwz is linear over GF(2) and the lane part, batch part
// and member offsets occupy disjoint bits, so a member's slot is the XOR of
// the three parts' swizzled slots: the batch part is scalar work and an
// address is one XOR (the tile sits at LDS offset 0).
template <bool F16 = false>
__device__ __forceinline__ unsigned BatchSlot(unsigned bt,
                                              const unsigned (&b)[5]) {
  unsigned pb = 0;
#pragma unroll
  for (int i = 0; i < 5; ++i) pb |= ((bt >> i) & 1u) << b[i];
  return BlockSwz<F16>(pb) * unsigned(sizeof(float2));
}

// Lane half h's 8 members of its group as bf16 (hi, lo) pairs.
__device__ __forceinline__ void SplitBf16(const v2f (&v)[8], v8bf (&bh)[2],
                                          v8bf (&bl)[2]) {
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const v2bf hi = __builtin_convertvector(v[q], v2bf);
    const v2f r = v[q] - __builtin_convertvector(hi, v2f);
    const v2bf lo = __builtin_convertvector(r, v2bf);
    bh[q >> 2][2 * (q & 3)] = hi[0];
    bh[q >> 2][2 * (q & 3) + 1] = hi[1];
    bl[q >> 2][2 * (q & 3)] = lo[0];
    bl[q >> 2][2 * (q & 3) + 1] = lo[1];
  }
}

// The op on one batch: Al Bh + Am Bh + Ah Bl + Ah Bh per K block, one
// accumulator chain.
__device__ __forceinline__ v16f MfmaChain(const v8bf (&f)[6],
                                          const v8bf (&bh)[2],
                                          const v8bf (&bl)[2]) {
  v16f c = v16f{};
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[2], bh[0], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[1], bh[0], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[0], bl[0], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[0], bh[0], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[5], bh[1], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[4], bh[1], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[3], bl[1], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[3], bh[1], c, 0, 0, 0);
  return c;
}

// Lane half h's 8 members of its group in three bf16 parts (hi, mid, lo):
// the amplitudes to about 2^-25 instead of 2^-18.
__device__ __forceinline__ void SplitBf16x3(const v2f (&v)[8], v8bf (&bh)[2],
                                            v8bf (&bm)[2], v8bf (&bl)[2]) {
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const v2bf hi = __builtin_convertvector(v[q], v2bf);
    const v2f r1 = v[q] - __builtin_convertvector(hi, v2f);
    const v2bf mid = __builtin_convertvector(r1, v2bf);
    const v2f r2 = r1 - __builtin_convertvector(mid, v2f);
    const v2bf lo = __builtin_convertvector(r2, v2bf);
    bh[q >> 2][2 * (q & 3)] = hi[0];
    bh[q >> 2][2 * (q & 3) + 1] = hi[1];
    bm[q >> 2][2 * (q & 3)] = mid[0];
    bm[q >> 2][2 * (q & 3) + 1] = mid[1];
    bl[q >> 2][2 * (q & 3)] = lo[0];
    bl[q >> 2][2 * (q & 3) + 1] = lo[1];
  }
}

// The accurate product: every term down to 2^-16 relative (Al Bh + Am Bm +
// Ah Bl + Am Bh + Ah Bm + Ah Bh per K block, smallest first), 12 MFMAs.
__device__ __forceinline__ v16f MfmaChain6(const v8bf (&f)[6],
                                           const v8bf (&bh)[2],
                                           const v8bf (&bm)[2],
                                           const v8bf (&bl)[2]) {
  v16f c = v16f{};
#pragma unroll
  for (int kb = 0; kb < 2; ++kb) {
    const v8bf& ah = f[3 * kb];
    const v8bf& am = f[3 * kb + 1];
    const v8bf& al = f[3 * kb + 2];
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, bh[kb], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(am, bm[kb], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bl[kb], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(am, bh[kb], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bm[kb], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bh[kb], c, 0, 0, 0);
  }
  return c;
}

// Lane l holds (re, im) of members 4 s + 2 h + {0, 1}.
__device__ __forceinline__ void WriteBatch(unsigned sp, const uint32_t (&wr)[8],
                                           const v16f& c) {
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      *LdsAt(sp ^ wr[2 * q + u]) = v2f{c[4 * q + 2 * u], c[4 * q + 2 * u + 1]};
    }
}

// ACCURATE: amplitudes in three parts and the 12-MFMA product (one batch at
// a time), for passes on structured states such as the first passes from a
// basis state, where the two-part split's rounding is the same for many
// amplitudes and shifts the norm coherently.
template <bool ACCURATE = false>
__device__ __forceinline__ void ApplyTileOp(const uint8_t* bp,
                                            const v8bf (&f)[6],
                                            const uint32_t (&rd)[8],
                                            const uint32_t (&wr)[8],
                                            unsigned nbatch, unsigned wave,
                                            unsigned nwaves) {
  unsigned b[5];
#pragma unroll
  for (int i = 0; i < 5; ++i)
    b[i] = unsigned(__builtin_amdgcn_readfirstlane(int(bp[i])));
  if (ACCURATE) {
    for (unsigned bt = wave; bt < nbatch; bt += nwaves) {
      const unsigned sp0 = BatchSlot(bt, b);
      v2f v0[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) v0[q] = *LdsAt(sp0 ^ rd[q]);
      v8bf bh0[2], bm0[2], bl0[2];
      SplitBf16x3(v0, bh0, bm0, bl0);
      WriteBatch(sp0, wr, MfmaChain6(f, bh0, bm0, bl0));
    }
    return;
  }
  // Two batches at a time (their groups are disjoint): batch 1's reads and
  // split overlap batch 0's MFMA chain.
  unsigned bt = wave;
  for (; bt + nwaves < nbatch; bt += 2 * nwaves) {
    const unsigned sp0 = BatchSlot(bt, b);
    const unsigned sp1 = BatchSlot(bt + nwaves, b);
    v2f v0[8], v1[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) v0[q] = *LdsAt(sp0 ^ rd[q]);
    v8bf bh0[2], bl0[2], bh1[2], bl1[2];
    SplitBf16(v0, bh0, bl0);
#pragma unroll
    for (int q = 0; q < 8; ++q) v1[q] = *LdsAt(sp1 ^ rd[q]);
    const v16f c0 = MfmaChain(f, bh0, bl0);
    SplitBf16(v1, bh1, bl1);
    const v16f c1 = MfmaChain(f, bh1, bl1);
    WriteBatch(sp0, wr, c0);
    WriteBatch(sp1, wr, c1);
  }
  if (bt < nbatch) {
    const unsigned sp0 = BatchSlot(bt, b);
    v2f v0[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) v0[q] = *LdsAt(sp0 ^ rd[q]);
    v8bf bh0[2], bl0[2];
    SplitBf16(v0, bh0, bl0);
    WriteBatch(sp0, wr, MfmaChain(f, bh0, bl0));
  }
}

// ---- FP16-with-scaling ops ---------------------------------------------
//
// The same product on v_mfma_f32_32x32x16_f16: the matrix in two fp16 parts
// (Ah + Al, 22 bits), the amplitudes in two (Bh + Bl, 22 bits) and
// Al Bh + Ah Bl + Ah Bh accumulated in FP32 (6 MFMAs per 32 groups instead
// of 8; the dropped Al Bl is 2^-22 relative).  fp16 has a 5-bit exponent,
// so the tile is scaled by a power of two when it is staged (TileScale):
// its largest real or imaginary part goes to [2^5, 2^6) / 2^headroom.  The
// ops of a pass keep the tile's norm (unitary, or contractive for headroom
// 0), so no value passes sqrt(2 * 2^14) * 2^6 < 2^14 < 65504; values below
// 2^-8 of the tile's largest keep an absolute error under 2^-30 of it.
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));

// FP16 op record, 32-bit words: the 16 x 16 complex matrix as packed
// (re, im) fp16 pairs, row r at words 16 r .. 16 r + 15 with record column
// p holding matrix column F16Col(p), hi part then lo part; the member
// tables, the group table and the batch-bit positions as in the bf16
// record; padded to a multiple of 4 words.  With that column order the 8
// members a lane reads for the B operand are the 8 members its C registers
// hold, in the same order (both: 8 kb + 4 (c / 2) + 2 h + c % 2 for
// q = 4 kb + c), so one LDS address per member serves the read and the
// write of a batch (the read and write halves of the member table are the
// same).
constexpr int kF16MatWords = 256;
constexpr int kF16TabOff = 2 * kF16MatWords;
constexpr int kF16BposOff = kF16TabOff + kTableWords + kLaneWords;
constexpr int kF16RecWords = kF16BposOff + 4;  // 580
static_assert(kF16RecWords % 4 == 0, "records are copied as uint4");

// Matrix column stored at record column p: p with bits 1 and 2 swapped.
__host__ __device__ constexpr unsigned F16Col(unsigned p) {
  return (p & 9u) | ((p & 2u) << 1) | ((p & 4u) >> 1);
}

// LDS of an FP16 blocked-pass workgroup: the tile, 16 floats for the
// per-wave maxima, then the pass's op records (all of them, loaded once per
// workgroup).  14-qubit tiles: one workgroup per CU (160 KiB); 13: two.
template <int TB>
struct F16Lds {
  static constexpr size_t kLimit = TB == 14 ? 163840 : 81920;
  static constexpr size_t kMaxOff = BlockShape<TB>::kTileBytes;
  static constexpr size_t kRecOff = kMaxOff + 64;
  static constexpr unsigned kMaxOps =
      unsigned((kLimit - kRecOff) / (kF16RecWords * sizeof(uint32_t)));
  static constexpr size_t Bytes(unsigned nops) {
    return kRecOff + size_t(nops) * kF16RecWords * sizeof(uint32_t);
  }
};

// Lane l's A fragments of the op whose record is at r (LDS): for K block
// kb, f[2 kb] = hi and f[2 kb + 1] = lo of A[l%32][16 kb + 8 (l/32) + e].
// Row l%32 = 2 i + p reads record columns 8 kb + 4 (l/32) + c, c < 4, of
// row i, and forms (Re, -Im) for p = 0 or (Im, Re) for p = 1 from the
// stored (Re, Im) pair.
__device__ __forceinline__ void LoadFragF16(const uint32_t* r, int l,
                                            v8h (&f)[4]) {
  const unsigned i = unsigned(l & 31) >> 1, hh = unsigned(l) >> 5;
  const unsigned rot = (l & 1) ? 16u : 0u;
  const uint32_t sx = (l & 1) ? 0u : 0x80000000u;
#pragma unroll
  for (int kb = 0; kb < 2; ++kb)
#pragma unroll
    for (int part = 0; part < 2; ++part) {
      const uint4 w = *reinterpret_cast<const uint4*>(
          r + part * kF16MatWords + 16 * i + 8 * kb + 4 * hh);
      uint4 x;
      x.x = __builtin_amdgcn_alignbit(w.x, w.x, rot) ^ sx;
      x.y = __builtin_amdgcn_alignbit(w.y, w.y, rot) ^ sx;
      x.z = __builtin_amdgcn_alignbit(w.z, w.z, rot) ^ sx;
      x.w = __builtin_amdgcn_alignbit(w.w, w.w, rot) ^ sx;
      f[2 * kb + part] = __builtin_bit_cast(v8h, x);
    }
}

// Lane half h's 8 members as fp16 (hi, lo) pairs: hi rounds to nearest;
// the residual v - hi is exact in FP32 and v_fma_mix{lo,hi}_f16 round it
// to fp16 straight from the fp16 half, one instruction per value.
__device__ __forceinline__ void SplitF16(const v2f (&v)[8], v8h (&bh)[2],
                                         v8h (&bl)[2]) {
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const v2h hi = __builtin_convertvector(v[q], v2h);
    uint32_t lw;
    asm("v_fma_mixlo_f16 %0, -%1, 1.0, %2 op_sel_hi:[1,0,0]"
        : "=v"(lw)
        : "v"(hi), "v"(v[q][0]));
    asm("v_fma_mixhi_f16 %0, -%1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
        : "+v"(lw)
        : "v"(hi), "v"(v[q][1]));
    const v2h lo = __builtin_bit_cast(v2h, lw);
    bh[q >> 2][2 * (q & 3)] = hi[0];
    bh[q >> 2][2 * (q & 3) + 1] = hi[1];
    bl[q >> 2][2 * (q & 3)] = lo[0];
    bl[q >> 2][2 * (q & 3) + 1] = lo[1];
  }
}

// Al Bh + Ah Bl + Ah Bh per K block, smallest first, one accumulator chain.
__device__ __forceinline__ v16f MfmaChainF16(const v8h (&f)[4],
                                             const v8h (&bh)[2],
                                             const v8h (&bl)[2]) {
  v16f c = v16f{};
#pragma unroll
  for (int kb = 0; kb < 2; ++kb) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[2 * kb + 1], bh[kb], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[2 * kb], bl[kb], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[2 * kb], bh[kb], c, 0, 0, 0);
  }
  return c;
}

// A lane's part of an FP16 op: its A fragments, its member offsets (record
// column order, so that reads and writes share them) XOR its group's slot,
// the batch-bit positions, and whether members 2 q and 2 q + 1 are the two
// amplitudes of a 16-byte unit (position 0 is a target).
struct F16Op {
  v8h f[4];
  uint32_t mo[8];
  uint32_t bw[2];
  bool pair;

  __device__ __forceinline__ void Load(const uint32_t* r, int l) {
    LoadFragF16(r, l, f);
    const uint32_t* tab = r + kF16TabOff + 16 * (l >> 5);
    const uint32_t sj = r[kF16TabOff + kTableWords + (l & 31)];
#pragma unroll
    for (int q = 0; q < 8; ++q) mo[q] = tab[q] ^ sj;
    bw[0] = r[kF16BposOff];
    bw[1] = r[kF16BposOff + 1];
  }
  // The wave-uniform part, in scalar registers.
  __device__ __forceinline__ void Uniform(unsigned (&b)[5]) {
    const unsigned w0 = unsigned(__builtin_amdgcn_readfirstlane(int(bw[0])));
    const unsigned w1 = unsigned(__builtin_amdgcn_readfirstlane(int(bw[1])));
#pragma unroll
    for (int i = 0; i < 4; ++i) b[i] = (w0 >> (8 * i)) & 255u;
    b[4] = w1 & 255u;
    pair = (w1 >> 8) & 1u;
  }
};

typedef float v4f __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4f LdsV4f;
__device__ __forceinline__ LdsV4f* LdsAt16(unsigned b) {
  return reinterpret_cast<LdsV4f*>(size_t{b});
}

template <bool PAIR>
__device__ __forceinline__ void ReadBatch(unsigned sp, const uint32_t (&mo)[8],
                                          v2f (&v)[8]) {
  if (PAIR) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const v4f x = *LdsAt16(sp ^ mo[2 * q]);
      v[2 * q] = v2f{x[0], x[1]};
      v[2 * q + 1] = v2f{x[2], x[3]};
    }
  } else {
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = *LdsAt(sp ^ mo[q]);
  }
}

// Results of a batch back to the slots its inputs came from: C registers
// (2 q, 2 q + 1) are the q-th member of the lane's list.
template <bool PAIR>
__device__ __forceinline__ void WriteBack(unsigned sp, const uint32_t (&mo)[8],
                                          const v16f& c) {
  if (PAIR) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *LdsAt16(sp ^ mo[2 * q]) =
          v4f{c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3]};
  } else {
#pragma unroll
    for (int q = 0; q < 8; ++q)
      *LdsAt(sp ^ mo[q]) = v2f{c[2 * q], c[2 * q + 1]};
  }
}

// One FP16 op over the LDS tile; batches as in ApplyTileOp, two at a time.
// SCALE: the tile in LDS is not scaled yet; what is read is multiplied by
// 2^e.
template <bool PAIR, bool SCALE>
__device__ __forceinline__ void RunOpF16(const F16Op& o,
                                         const unsigned (&b)[5],
                                         unsigned nbatch, unsigned wave,
                                         unsigned nwaves, int e) {
  auto read = [&](unsigned sp, v2f (&v)[8]) {
    ReadBatch<PAIR>(sp, o.mo, v);
    if (SCALE) {
#pragma unroll
      for (int q = 0; q < 8; ++q)
        v[q] = v2f{ldexpf(v[q][0], e), ldexpf(v[q][1], e)};
    }
  };
  unsigned bt = wave;
  for (; bt + nwaves < nbatch; bt += 2 * nwaves) {
    const unsigned sp0 = BatchSlot<true>(bt, b);
    const unsigned sp1 = BatchSlot<true>(bt + nwaves, b);
    v2f v0[8], v1[8];
    read(sp0, v0);
    v8h bh0[2], bl0[2], bh1[2], bl1[2];
    SplitF16(v0, bh0, bl0);
    read(sp1, v1);
    const v16f c0 = MfmaChainF16(o.f, bh0, bl0);
    SplitF16(v1, bh1, bl1);
    const v16f c1 = MfmaChainF16(o.f, bh1, bl1);
    WriteBack<PAIR>(sp0, o.mo, c0);
    WriteBack<PAIR>(sp1, o.mo, c1);
  }
  if (bt < nbatch) {
    const unsigned sp0 = BatchSlot<true>(bt, b);
    v2f v0[8];
    read(sp0, v0);
    v8h bh0[2], bl0[2];
    SplitF16(v0, bh0, bl0);
    WriteBack<PAIR>(sp0, o.mo, MfmaChainF16(o.f, bh0, bl0));
  }
}

template <bool SCALE = false>
__device__ __forceinline__ void ApplyTileOpF16(F16Op& o, unsigned nbatch,
                                               unsigned wave, unsigned nwaves,
                                               int e = 0) {
  unsigned b[5];
  o.Uniform(b);
  if (o.pair)
    RunOpF16<true, SCALE>(o, b, nbatch, wave, nwaves, e);
  else
    RunOpF16<false, SCALE>(o, b, nbatch, wave, nwaves, e);
}

// Largest |re| or |im| over the first `nper` of a thread's PER elements
// (FULL: all of them).
template <int PER, bool FULL>
__device__ __forceinline__ float LocalMax(const float2 (&v)[PER],
                                          unsigned nper) {
  float m = 0.0f;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    if (FULL || unsigned(i) < nper) {
      m = fmaxf(m, fmaxf(fabsf(v[i].x), fabsf(v[i].y)));
    }
  }
  return m;
}

// The scale exponent of a tile whose largest |re| or |im| is t: t goes to
// [2^5, 2^6) / 2^headroom; 0 for an all-zero (or non-finite) tile.
__device__ __forceinline__ int ScaleExponent(float t, unsigned headroom) {
  if (!(t > 0.0f) || !(t <= 3.0e38f)) return 0;
  int e;
  (void)frexpf(t, &e);  // t in [2^(e-1), 2^e)
  return 6 - int(headroom) - e;  // |e| <= 149: ldexpf takes any such shift
}

// Workgroup maximum of `m` through `slots` (one float per wave), then the
// tile's scale exponent.  Ends with a barrier before the slots are read;
// the slots are written again only after a later barrier.
template <int NWAVES>
__device__ __forceinline__ int TileScale(float m, float* slots,
                                         unsigned headroom) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) m = fmaxf(m, __shfl_xor(m, d));
  if ((threadIdx.x & 63) == 0) slots[threadIdx.x >> 6] = m;
  __syncthreads();
  float t = 0.0f;
#pragma unroll
  for (int w = 0; w < NWAVES; ++w) t = fmaxf(t, slots[w]);
  return ScaleExponent(t, headroom);
}

// Offset (in amplitudes) of tile-local high index x: x's bits deposited at
// the tile's high qubits.
__device__ __forceinline__ uint64_t DepositHigh(unsigned x, const BlockGeom& g) {
  uint64_t o = 0;
  for (unsigned b = 0; b < g.h; ++b) o += ((x >> b) & 1u) ? g.hbit[b] : 0;
  return o;
}

// The same for x's bits at tile positions first, first + 1, ... (a
// compile-time x < 2^NB, none of them in the low run), in units of 2^Lc
// amplitudes; hbit is zero past the tile's last position.
template <int NB>
__device__ __forceinline__ uint32_t HighOffset(unsigned x, unsigned first,
                                               const BlockGeom& g) {
  uint32_t o = 0;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    if ((x >> b) & 1u) o += uint32_t(g.hbit[first - g.Lc + b] >> g.Lc);
  }
  return o;
}

// Tile staging with addresses split into a per-thread part and a per-element
// part.  Element i of thread t is tile-local amplitude a = t + NT i (valid
// for i < 2^tb / NT, a wave-uniform test).  The host keeps the low run
// within the thread bits (Lc <= log2 NT), so a's low bits come from t alone
// and its high index is (t >> Lc) | (i << (log2 NT - Lc)) with disjoint
// bits: its offset is D(t >> Lc) + D(i << (log2 NT - Lc)), one add per
// element instead of a deposit loop.  The element parts are wave-uniform
// and kept in units of 2^Lc amplitudes (32 bits: no tile qubit is 32 above
// the low run).
template <int PER, int NT, bool F16>
struct TileIo {
  static_assert(NT == 256 || NT == 512, "thread bits");
  static_assert(PER <= 32, "element bits");
  static constexpr unsigned kLogNT = NT == 256 ? 8 : 9;
  uint64_t tofs;       // this thread's part
  uint32_t eofs[PER];  // the element parts >> Lc

  // LDS slot of element i: the swizzle S is linear and changes only the low
  // four bits, so S(t + NT i) = (S(t) ^ (S(NT i) & 15)) + NT i with
  // S(t) < NT: the NT i part is an instruction offset and the
  // rest takes one XOR with a constant.
  __device__ __forceinline__ unsigned Slot(int i) const {
    return (BlockSwz<F16>(threadIdx.x) ^
            (BlockSwz<F16>(NT * unsigned(i)) & 15u)) +
           NT * unsigned(i);
  }

  __device__ __forceinline__ void Init(const BlockGeom& g) {
    const unsigned t = threadIdx.x;
    tofs = (t & ((1u << g.Lc) - 1)) + DepositHigh(t >> g.Lc, g);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      eofs[i] = HighOffset<5>(unsigned(i), kLogNT, g);
    }
  }

  // Issues the loads of the tile at `base` into v (this thread's elements),
  // those of the quarters of v whose bits are set in MASK (quarter c holds
  // elements c PER/4 .. (c+1) PER/4 - 1).
  template <bool FULL, unsigned MASK>
  __device__ __forceinline__ void Fetch(const float2* __restrict__ s,
                                        uint64_t base, const BlockGeom& g,
                                        float2 (&v)[PER]) const {
    const unsigned nper = (1u << g.tb) >> kLogNT;  // elements per thread
    const float2* p = s + base + tofs;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (((MASK >> (4 * i / PER)) & 1u) && (FULL || unsigned(i) < nper)) {
        v[i] = p[uint64_t(eofs[i]) << g.Lc];
      }
    }
  }

  // Writes fetched elements to their LDS slots.
  template <bool FULL>
  __device__ __forceinline__ void Put(const BlockGeom& g,
                                      const float2 (&v)[PER],
                                      float2* lds) const {
    const unsigned nper = (1u << g.tb) >> kLogNT;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (FULL || unsigned(i) < nper) lds[Slot(i)] = v[i];
    }
  }

  // Put with every value multiplied by 2^e (exact for normal results).
  template <bool FULL>
  __device__ __forceinline__ void PutScaled(const BlockGeom& g,
                                            const float2 (&v)[PER],
                                            float2* lds, int e) const {
    const unsigned nper = (1u << g.tb) >> kLogNT;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (FULL || unsigned(i) < nper) {
        lds[Slot(i)] = float2{ldexpf(v[i].x, e), ldexpf(v[i].y, e)};
      }
    }
  }

  // Store with every value multiplied by 2^-e.
  template <int CH, bool FULL>
  __device__ __forceinline__ void StoreScaled(float2* __restrict__ s,
                                              uint64_t base,
                                              const BlockGeom& g,
                                              const float2* lds,
                                              int e) const {
    const unsigned nper = (1u << g.tb) >> kLogNT;
    float2* p = s + base + tofs;
#pragma unroll
    for (int i0 = 0; i0 < PER; i0 += CH) {
      float2 v[CH];
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        if (FULL || unsigned(i0 + i) < nper) {
          const float2 x = lds[Slot(i0 + i)];
          v[i] = float2{ldexpf(x.x, -e), ldexpf(x.y, -e)};
        }
      }
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        if (FULL || unsigned(i0 + i) < nper) p[uint64_t(eofs[i0 + i]) << g.Lc] = v[i];
      }
    }
  }

  template <int CH, bool FULL>
  __device__ __forceinline__ void Store(float2* __restrict__ s, uint64_t base,
                                        const BlockGeom& g,
                                        const float2* lds) const {
    const unsigned nper = (1u << g.tb) >> kLogNT;
    float2* p = s + base + tofs;
#pragma unroll
    for (int i0 = 0; i0 < PER; i0 += CH) {
      float2 v[CH];
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        if (FULL || unsigned(i0 + i) < nper) v[i] = lds[Slot(i0 + i)];
      }
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        if (FULL || unsigned(i0 + i) < nper) p[uint64_t(eofs[i0 + i]) << g.Lc] = v[i];
      }
    }
  }
};

// The FP16 pass over 14-qubit tiles.  One 128 KiB tile fills a CU's LDS, so
// no second workgroup can hide its HBM phases; the workgroup hides them
// itself: 8 waves run the ops and 4 waves (one per SIMD) do nothing but move
// tiles.  The IO waves hold a whole tile in registers (32 16-byte pairs a
// thread).  While the ops of a tile run they issue, share by share, the
// stores of the previous tile and, into the registers each store frees, the
// loads of the next one; a wave that stalls on a full memory queue holds up
// no op until the barrier that ends it.  Between two tiles they exchange the
// tile in LDS for the one in registers.  Shares go out with all ops but the
// last, whose time covers the last loads' latency.
//
// The tile is scaled as in GateBlockF16Kernel, but by the first op as it
// reads (the maximum is known only once the loads have arrived, and the
// exchange, which nothing overlaps, moves bits unchanged) and on the way out
// by the stores.
//
// Bound by the HBM stream up to 4 ops; the ops take as long at 5, and each
// further one 2.1 ms more (LDS reads and writes of the whole tile, the fp16
// split and the MFMA chain in sequence).  32 qubits, tiles of 4 low and 10
// random higher qubits, 1 / 3
// / 5 / 7 ops: 13.3-16.0 / 13.5-16.0 / 16.0-16.6 / 20.3-20.9 ms, against
// 16.3 / 16.0-17.5 / 18.7-20.1 / 23.2-24.2 with every wave doing both.  The
// 64 KiB shape has two workgroups a CU, which hide each other's phases, and
// keeps that structure.
constexpr unsigned kIoNT = 256;                       // 4 IO waves
constexpr unsigned kIoThreads = BlockShape<14>::NT + kIoNT;

// Pair i of IO thread t: tile-local amplitudes 2 t + 512 i and its
// successor.  Positions 9 and up are never in the low run (PrepareGateBlock),
// so i's bits are the tile's five highest qubits, h[0..4].
struct TileIoPairs {
  static constexpr int PER = (1 << 14) / (2 * kIoNT);  // 32 pairs a thread
  uint64_t tofs;  // t's part of the offset in the state, amplitudes
  uint64_t h[5];  // wave-uniform
  unsigned unit;  // t's part of the 16-byte LDS unit

  __device__ __forceinline__ void Init(const BlockGeom& g, unsigned t) {
    const unsigned a = 2 * t;
    tofs = (a & ((1u << g.Lc) - 1)) + DepositHigh(a >> g.Lc, g);
#pragma unroll
    for (int b = 0; b < 5; ++b) h[b] = g.hbit[9 - g.Lc + b];
    unit = F16Swz(a) >> 1;
  }
  // A state is aligned to an amplitude only.
  typedef float Pair __attribute__((ext_vector_type(4), aligned(8)));
  // Addresses of the four pairs 4 C .. 4 C + 3 of the tile at `base`.  The
  // thread's part is hidden from the optimiser so that the 32 addresses are
  // not kept in registers across the tile loop, where the pairs are.
  template <int C>
  __device__ __forceinline__ void At(float2* s, uint64_t base,
                                     Pair* (&q)[4]) const {
    uint64_t o = tofs;
    asm volatile("" : "+v"(o));
    uint64_t b = base;
    if (C & 1) b += h[2];
    if (C & 2) b += h[3];
    if (C & 4) b += h[4];
    float2* p = s + o;
    q[0] = reinterpret_cast<Pair*>(p + b);
    q[1] = reinterpret_cast<Pair*>(p + (b + h[0]));
    q[2] = reinterpret_cast<Pair*>(p + (b + h[1]));
    q[3] = reinterpret_cast<Pair*>(p + (b + h[0] + h[1]));
  }
  __device__ __forceinline__ unsigned Unit(int i) const {
    unsigned u = unit;
    asm volatile("" : "+v"(u));
    return (u ^ ((F16Swz(512u * unsigned(i)) & 15u) >> 1)) +
           256u * unsigned(i);
  }
};

// Maximum of a non-negative value over the wave, in lane 63.
__device__ __forceinline__ float WaveMaxTo63(float m) {
  auto step = [&](auto ctrl) {
    m = fmaxf(m, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
                     0, __builtin_bit_cast(int, m), decltype(ctrl)::value, 0xf,
                     0xf, false)));
  };
  step(std::integral_constant<int, 0x111>{});  // row_shr:1, :2, :4, :8
  step(std::integral_constant<int, 0x112>{});
  step(std::integral_constant<int, 0x114>{});
  step(std::integral_constant<int, 0x118>{});
  step(std::integral_constant<int, 0x142>{});  // row_bcast:15, :31
  step(std::integral_constant<int, 0x143>{});
  return m;
}

template <int N, typename F>
__device__ __forceinline__ void Unrolled(F&& f) {
  if constexpr (N > 0) {
    Unrolled<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

// Applies the pass to tiles first, first + stride, ... < end (at least one)
// of the state at s, with the kIoThreads threads of the workgroup.
// lds_raw: LDS offset 0, F16Lds<14>::Bytes(p.nops) bytes.
__device__ __forceinline__ void BlockIoRun(
    float2* __restrict__ s, const BlockGeom& g, const BlockProgram& p,
    const uint32_t* __restrict__ recs, char* lds_raw, uint64_t first,
    uint64_t end, uint64_t stride) {
  constexpr int NW = BlockShape<14>::kWaves;
  constexpr int PER = TileIoPairs::PER;
  constexpr int kShares = PER / 4;
  v4f* lds4 = reinterpret_cast<v4f*>(lds_raw);
  float* slots = reinterpret_cast<float*>(lds_raw + F16Lds<14>::kMaxOff);
  uint32_t* rec = reinterpret_cast<uint32_t*>(lds_raw + F16Lds<14>::kRecOff);
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // The scale exponent of the tile whose wave maxima are in slots 4 par ...
  auto scale_of = [&](unsigned par) {
    const float* m = slots + 4 * par;
    return __builtin_amdgcn_readfirstlane(ScaleExponent(
        fmaxf(fmaxf(m[0], m[1]), fmaxf(m[2], m[3])), p.headroom));
  };
  if (wave < unsigned(NW)) {
    const int l = threadIdx.x & 63;
    const unsigned nq = p.nops * unsigned(kF16RecWords / 4);
    const uint4* src = reinterpret_cast<const uint4*>(recs);
    uint4* dst = reinterpret_cast<uint4*>(rec);
    for (unsigned q = threadIdx.x; q < nq; q += 64 * NW) dst[q] = src[q];
    __syncthreads();
    unsigned par = 0;
    // An op's record is read while the op before it finishes.
    F16Op o;
    o.Load(rec, l);
    auto run_op = [&](unsigned op, auto scale, int e) {
      ApplyTileOpF16<decltype(scale)::value>(o, 32u, wave, NW, e);
      o.Load(rec + (op + 1 < p.nops ? op + 1 : 0) * unsigned(kF16RecWords), l);
      __syncthreads();
    };
    for (uint64_t tile = first; tile < end; tile += stride) {
      run_op(0, std::true_type{}, scale_of(par));
      for (unsigned op = 1; op < p.nops; ++op) run_op(op, std::false_type{}, 0);
      __syncthreads();
      par ^= 1u;
    }
    return;
  }
  const unsigned t = threadIdx.x - 64u * NW;
  TileIoPairs io;
  io.Init(g, t);
  v4f buf[PER];
  auto load = [&](auto c, uint64_t base) {
    constexpr int C = decltype(c)::value;
    TileIoPairs::Pair* q[4];
    io.At<C>(s, base, q);
#pragma unroll
    for (int i = 0; i < 4; ++i) buf[4 * C + i] = *q[i];
  };
  auto store = [&](auto c, uint64_t base, int e) {
    constexpr int C = decltype(c)::value;
    TileIoPairs::Pair* q[4];
    io.At<C>(s, base, q);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const v4f v = buf[4 * C + i];
      *q[i] = v4f{ldexpf(v.x, -e), ldexpf(v.y, -e), ldexpf(v.z, -e),
                  ldexpf(v.w, -e)};
    }
  };
  // Waits for the loads; the maximum of this wave's values to its slot.
  auto arrive = [&](unsigned par) {
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const v4f v = buf[i];
      m = fmaxf(fmaxf(m, fabsf(v.x)), fabsf(v.y));
      m = fmaxf(fmaxf(m, fabsf(v.z)), fabsf(v.w));
    }
    m = WaveMaxTo63(m);
    if ((t & 63u) == 63u) slots[4 * par + (t >> 6)] = m;
  };
  uint64_t tile = first;
  uint64_t base = InsertZeros(tile << g.Lc, g.outer, g.nouter);
  Unrolled<kShares>([&](auto c) { load(c, base); });
  arrive(0);
#pragma unroll
  for (int i = 0; i < PER; ++i) lds4[io.Unit(i)] = buf[i];
  __syncthreads();
  unsigned par = 0;
  uint64_t obase = 0;  // the finished tile in buf
  int oe = 0;
  const unsigned spread = p.nops > 1 ? p.nops - 1 : 1;
  for (bool out = false;; out = true) {
    const int e = scale_of(par);
    const bool more = tile + stride < end;
    tile += stride;
    const uint64_t nb =
        more ? InsertZeros(tile << g.Lc, g.outer, g.nouter) : 0;
    unsigned op = 0;
    Unrolled<kShares>([&](auto c) {
      constexpr unsigned C = decltype(c)::value;
      // Share C goes out with op C spread / 8.
      for (const unsigned due = C * spread / kShares; op < due; ++op)
        __syncthreads();
      if (out) store(c, obase, oe);
      if (more) load(c, nb);
    });
    for (; op + 1 < p.nops; ++op) __syncthreads();
    par ^= 1u;
    if (more) arrive(par);
    __syncthreads();
    // The exchange: every slot of the tile belongs to one thread here.  The
    // reads of one step are in flight while the step before is written.
    constexpr int ST = 2;
    v4f old[2][ST];
    auto take = [&](auto c) {
      constexpr int C = decltype(c)::value;
#pragma unroll
      for (int i = 0; i < ST; ++i) old[C & 1][i] = lds4[io.Unit(ST * C + i)];
    };
    take(std::integral_constant<int, 0>{});
    Unrolled<PER / ST>([&](auto c) {
      constexpr int C = decltype(c)::value;
      if constexpr (C + 1 < PER / ST) take(std::integral_constant<int, C + 1>{});
#pragma unroll
      for (int i = 0; i < ST; ++i) {
        if (more) lds4[io.Unit(ST * C + i)] = buf[ST * C + i];
        buf[ST * C + i] = old[C & 1][i];
      }
    });
    __syncthreads();
    obase = base;
    oe = e;
    if (!more) break;
    base = nb;
  }
  Unrolled<kShares>([&](auto c) { store(c, obase, oe); });
}

}  // namespace tileop
}  // namespace qhip
