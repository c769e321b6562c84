// FP32 products on the bfloat16 matrix cores: every FP32 operand is split into three bfloat16
// numbers, x = x0 + x1 + x2, exactly (24 significand bits in three pieces of 8, rounded to nearest;
// the method of Henry, Tang and Heinecke, "Leveraging the bfloat16 artificial intelligence datatype
// for higher-precision computations", ARITH 2019), and a product keeps the six partial products above
// 2^-24 of it,
//
//   a b  ~  a0 b2 + a2 b0 + a0 b1 + a0 b0 + a1 b0 + a1 b1        (left out: a1 b2, a2 b1, a2 b2)
//
// each exact in FP32 and accumulated in FP32 by v_mfma_f32_16x16x32_bf16.
//
// Why: the FP32 MFMA rate is 1/16 of the bfloat16 rate, so six bfloat16 MFMAs cost 6/16 of the
// FP32 MFMAs they replace.  The error is below that of v_mfma_f32_16x16x4f32: k_split3_gemm sums the six
// MFMAs of 32 k values from zero and adds them to the accumulator once, where the FP32 MFMA rounds
// the accumulator at every step.  Measured against FP64 over 1600 terms falling as exp(-k/20),
// smallest first (2-norm of the error over that of the result): 5.0e-8, FP32 MFMA 8.1e-8.
//
// Packed operands.  The split operands are laid out so that one MFMA operand of a wavefront is
// one contiguous kilobyte: block (rb, kg) of 16 rows and 32 k values holds three planes (x0, x1,
// x2) of 64 lanes x 8 bfloat16, lane l = row l % 16, k values 32 kg + 8 (l / 16) + 0..7 -- the A and
// B layout of the instruction.  Rows past the last and k values past K are zero.  A complex operand
// holds the real parts of 16 rows as one block row and the imaginary parts as the next, so both
// parts of a result land in the same lane.
//
// Infinities: an infinite x has x0 = x and x1 = x2 = 0, and its products with the pieces of the
// other operand may cancel to NaN where the FP32 product is infinite.  A result that is not
// finite is therefore formed again from the pieces' sums on the FP32 matrix cores (redo_non_finite).
#pragma once

#include "afq_internal.hpp"
#include "gemm.hpp"

namespace afq {
namespace s3 {

using gemm::f32x4;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr long kPlane = 1024;  // bytes of one plane of a block; a block (kBlock) has three

// The three pieces of eight values, each piece as one 16-byte word of a lane.
__device__ inline void split8(const float (&x)[8], u32x4 (&p)[3]) {
  bf16x8 q[3];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    __bf16 h = (__bf16)x[j];
    float hf = (float)h;
    if (!__builtin_isfinite(hf) && __builtin_isfinite(x[j])) {
      // the largest finite values round up to infinity: truncate instead
      hf = __uint_as_float(__float_as_uint(x[j]) & 0xFFFF0000u);
      h = (__bf16)hf;
    }
    // an infinite value has no remainder (a NaN stays one in x0)
    const float r = __builtin_isfinite(hf) ? x[j] - hf : 0.f;
    const __bf16 m = (__bf16)r;
    q[0][j] = h;
    q[1][j] = m;
    q[2][j] = (__bf16)(r - (float)m);
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) p[c] = __builtin_bit_cast(u32x4, q[c]);
}

// As split8, for values whose infinities need no care (an infinity gives NaN pieces).  Two values at a
// time: three packed conversions, and the rounded pieces taken back from the packed words (11
// instructions for two values).
__device__ inline void split8_finite(const float (&x)[8], bf16x8 (&q)[3]) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  u32x4 p[3];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float a = x[2 * j], b = x[2 * j + 1];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const unsigned int u =
          __builtin_bit_cast(unsigned int, __builtin_convertvector((f32x2{a, b}), bf16x2));
      p[c][j] = u;
      if (c < 2) {
        a -= __uint_as_float(u << 16);
        b -= __uint_as_float(u & 0xFFFF0000u);
      }
    }
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) q[c] = __builtin_bit_cast(bf16x8, p[c]);
}

// ---- packing ---------------------------------------------------------------------------------

// Rows of an operand: row n of the product is row src(n) of a [..][ld] tensor, or zero (src < 0).
struct RowsPlain {
  int rows;
  __device__ inline long src(long n) const { return n < rows ? n : -1; }
};
// row n is the orbital pair pairs[n] = i << 16 | k of an [N * N][ld] tensor
struct RowsPairs {
  const uint32_t* pairs;
  int rows, N;
  __device__ inline long src(long n) const {
    if (n >= rows) return -1;
    const uint32_t p = pairs[n];
    return (long)(p >> 16) * N + (p & 0xFFFFu);
  }
};
// items of n rows (a walker's or a Cholesky vector's electrons), each padded to nsp rows
struct RowsItems {
  int items, n, nsp;
  __device__ inline long src(long r) const {
    const long it = r / nsp;
    const int b = (int)(r % nsp);
    return it < items && b < n ? it * n + b : -1;
  }
};

// One wavefront per (16-row block, k group) of a complex operand X [rows][ld].  Blocks of nb rows
// form a tile: block i of tile t holds its real parts at block row (2 t) nb + i of `out` and its
// imaginary parts at (2 t + 1) nb + i.  Reads 8 (TIn float) or 16 bytes a value and writes 12: 4.3 TB/s
// from FP32 (G of 1024 walkers, N = 200, n = 40: 38 us), 1.9 TB/s from FP64, whose loads touch twice
// the lines; a copy reaches 5.
template <typename TIn, class ROWS>
__global__ void __launch_bounds__(256)
    k_pack_cplx(long blocks, int K0, int KG0, int K, int KG, const cplx<TIn>* __restrict__ X,
                long ld, ROWS rmap, int nb, char* __restrict__ out) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long q = (long)blockIdx.x * 4 + wave;
  const long rb = q / KG;
  const int kg = (int)(q % KG);
  if (rb >= blocks) return;
  const long r = rmap.src(16 * rb + (lane & 15));
  // values [0, K0) fill the first KG0 groups, [K0, K) the others
  const int k0 = 32 * kg + 8 * (lane >> 4) + (kg < KG0 ? 0 : K0 - 32 * KG0);
  const int kn = kg < KG0 ? K0 : K;
  const cplx<TIn>* x = X + max(r, 0L) * ld + k0;
  float re[8], im[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const cplx<TIn> v = (r >= 0 && k0 + j < kn) ? x[j] : cplx<TIn>{0, 0};
    re[j] = (float)v.re;
    im[j] = (float)v.im;
  }
  u32x4 p[3];
  char* o = out + (((rb / nb) * 2 * nb + rb % nb) * KG + kg) * kBlock + lane * 16;
  split8(re, p);
#pragma unroll
  for (int c = 0; c < 3; ++c) *reinterpret_cast<u32x4*>(o + c * kPlane) = p[c];
  o += (long)nb * KG * kBlock;
  split8(im, p);
#pragma unroll
  for (int c = 0; c < 3; ++c) *reinterpret_cast<u32x4*>(o + c * kPlane) = p[c];
}

// A real operand (built once per hamiltonian): one wavefront per (16-row block, k group), to the
// groups from g0 on of rows of ldg groups.  *bad is set when a value is not finite.
template <class ROWS>
__global__ void __launch_bounds__(256)
    k_pack_real(long blocks, int K, int KG, const float* __restrict__ X, long ld, ROWS rmap,
                char* __restrict__ out, int ldg, int g0, int* __restrict__ bad) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long q = (long)blockIdx.x * 4 + wave;
  const long rb = q / KG;
  const int kg = (int)(q % KG);
  if (rb >= blocks) return;
  const long r = rmap.src(16 * rb + (lane & 15));
  const int k0 = 32 * kg + 8 * (lane >> 4);
  const float* x = X + max(r, 0L) * ld + k0;
  float v[8];
  bool fin = true;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    v[j] = (r >= 0 && k0 + j < K) ? x[j] : 0.f;
    fin = fin && __builtin_isfinite(v[j]);
  }
  if (!fin) *bad = 1;
  u32x4 p[3];
  split8(v, p);
  char* o = out + (rb * ldg + g0 + kg) * kBlock + lane * 16;
#pragma unroll
  for (int c = 0; c < 3; ++c) *reinterpret_cast<u32x4*>(o + c * kPlane) = p[c];
}

// ---- C = A B^T, A complex [M][K], B real [N][K], both packed -----------------------------------

// The plain epilogues of gemm.hpp, called per element, under the interface of this kernel: a
// handle per column, then one call per element.
template <class E>
struct Plain {
  E e;
  __device__ inline int column(int n) const { return n; }
  __device__ inline void operator()(int ks, int m, int n, float re, float im) const {
    e(ks, m, n, re, im);
  }
};

// V[w][i][k] = V[w][k][i] = (ar + i ai) (re, im): column n is the orbital pair pairs[n] (the complex
// factor of gemm::EpiStoreSym, ai = 0, so an infinite part makes the other NaN there and here)
struct EpiPairs {
  c32* V;
  const uint32_t* pairs;
  int N;
  float ar, ai;
  __device__ inline uint32_t column(int n) const { return pairs[n]; }
  __device__ inline void operator()(int, int m, uint32_t p, float re, float im) const {
    const int i = (int)(p >> 16), k = (int)(p & 0xFFFFu);
    const c32 v = {ar * re - ai * im, ar * im + ai * re};
    c32* o = V + (long)m * N * N;
    o[(long)i * N + k] = v;
    o[(long)k * N + i] = v;
  }
};

// A packed operand as a buffer resource (raw 32-bit data, bounds checked): a load is one lane
// offset register, one scalar offset (block, k group) and an immediate (plane).
__device__ inline __amdgpu_buffer_rsrc_t resource(const char* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p), 0, bytes, 0x00027000);
}

template <int PLANE>
__device__ inline bf16x8 load_block(__amdgpu_buffer_rsrc_t base, uint32_t ofs, int lane16) {
  return __builtin_bit_cast(
      bf16x8, __builtin_amdgcn_raw_buffer_load_b128(base, lane16 + PLANE * (int)kPlane, (int)ofs, 0));
}

__device__ inline f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ inline f32x4 mfma_f32(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Whether any accumulator is infinite or NaN (x 0 is NaN for these, 0 for every other)
template <int RA, int CB>
__device__ inline bool any_non_finite(const f32x4 (&c)[RA][CB]) {
  f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < RA; ++i)
#pragma unroll
    for (int j = 0; j < CB; ++j) z += c[i][j] * 0.f;
  return __ballot(!((z[0] + z[1]) + (z[2] + z[3]) == 0.f)) != 0;
}

// The eight FP32 values of a lane of a block, from their pieces
__device__ inline void load_sums(float (&x)[8], __amdgpu_buffer_rsrc_t base, uint32_t ofs,
                                 int lane16) {
  const bf16x8 p = load_block<0>(base, ofs, lane16), q = load_block<1>(base, ofs, lane16),
               r = load_block<2>(base, ofs, lane16);
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = ((float)p[e] + (float)q[e]) + (float)r[e];
}

// The accumulators that are not finite (c[i][j]: block row at oa[i], block column at ob[j], the
// groups [g0, g0 + gn)) again on the FP32 matrix cores: eight v_mfma_f32_16x16x4_f32 a group, the e-th
// with the e-th k value of every lane, which leave the same elements in the same lanes.  Rows of A
// that hold a NaN are NaN throughout and need no product.  It costs about three times the tile's own
// products, or one pass over A's first pieces where a walker is NaN: vHS at N = 200, M = 1600 of 1024
// walkers takes 0.88 ms, with one infinite walker 1.5, with 100 infinite ones 3.3 and with 100 NaN ones
// 0.92.
template <int RA, int CB>
__device__ inline void redo_non_finite(f32x4 (&c)[RA][CB], __amdgpu_buffer_rsrc_t rA,
                                       const uint32_t (&oa)[RA], __amdgpu_buffer_rsrc_t rB,
                                       const uint32_t (&ob)[CB], int g0, int gn, int lane) {
  const int l16 = lane * 16, fk = lane >> 4;
  bool need = false;
#pragma unroll
  for (int i = 0; i < RA; ++i) {
    uint32_t rows = 0;  // the lane's rows with such an accumulator
#pragma unroll
    for (int j = 0; j < CB; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) rows |= !__builtin_isfinite(c[i][j][r]) ? 1u << (4 * fk + r) : 0u;
    // until each of them has shown a NaN: a dead walker's does in the first group
    for (int u = g0; u < g0 + gn && __ballot(rows != 0) != 0; ++u) {  // uniform
      const bf16x8 p = load_block<0>(rA, oa[i] + (uint32_t)(u * (int)kBlock), l16);
      bool nan = false;
#pragma unroll
      for (int e = 0; e < 8; ++e) nan = nan || p[e] != p[e];
      uint64_t q = __ballot(nan);
      q |= q >> 32;
      q |= q >> 16;
      rows &= ~(uint32_t)q;
    }
    need = need || rows != 0;
  }
  if (__ballot(need) == 0) return;  // uniform
#pragma unroll
  for (int j = 0; j < CB; ++j) {
    f32x4 t[RA];
#pragma unroll
    for (int i = 0; i < RA; ++i) t[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int u = g0; u < g0 + gn; ++u) {
      float a[8], b[8];
      load_sums(b, rB, ob[j] + (uint32_t)(u * (int)kBlock), l16);
#pragma unroll
      for (int i = 0; i < RA; ++i) {
        load_sums(a, rA, oa[i] + (uint32_t)(u * (int)kBlock), l16);
#pragma unroll
        for (int e = 0; e < 8; ++e) t[i] = mfma_f32(a[e], b[e], t[i]);
        __builtin_amdgcn_sched_barrier(0);  // (one block's loads at a time: the registers are few)
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < RA; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (!__builtin_isfinite(c[i][j][r])) c[i][j][r] = t[i][r];
  }
}

// One wavefront per tile of 16 RB rows (2 RB blocks: real and imaginary parts) x 16 CB columns,
// four wavefronts a workgroup, no LDS and no barrier: the operands stream from memory through
// L2/L1 straight into MFMA operands.  Column by column, the six partial products of a k group
// are summed from zero (2 RB independent chains of six MFMAs) and then added to the accumulators,
// so the accumulators are rounded once per 32 k values instead of six times (at 1024 x 20100 over
// 1600 terms falling as exp(-k/20): error 5.0e-8 against 8.5e-8 with all six MFMAs on the
// accumulator and 8.1e-8 with the FP32 MFMA; the additions cost 9 %).  A column's operands are
// reloaded for the next group as soon as its last product has issued, the row operands plane by
// plane during the last column, so there is no second operand buffer and the 32 x 96 tile (96
// accumulators, 120 operand registers) leaves two wavefronts per SIMD, one multiplying while the
// other waits.
// Tiles run in strips two columns wide, so the four wavefronts of a workgroup form a 2 x 2 patch
// and share both operands through L1; workgroups are renumbered so that each of the 8 XCDs takes
// a contiguous run.  REVK: k groups from the last to the first (terms that fall with k are added
// smallest first).  Split-K slices pass ks to the epilogue: ks0 slices of kchunk groups of the first
// KG0 groups, then those of the others (the two spins of vbias, whose sums stay apart).
//
// Bound by the operand feed through L2: the matrix cores are busy half of the time.  Measured in a
// walker step (1024 x 20100 outputs over 1600): 0.75 ms = 177 TFLOP/s of FP32 products, 0.46 of what six
// back-to-back MFMAs reach on this card (2.33 PFLOP/s / 6); with the FP32 MFMA 1.13 ms.  Repeated on
// fields of full amplitude it takes 0.77 to 0.93 ms.  Eight wavefronts per workgroup or a
// barrier per k group (more reuse in L1) measured 2-18 % slower.
template <int RB, int CB, bool REVK, class EPI>
__global__ void __launch_bounds__(256, 2)
    k_split3_gemm(int M, int N, int KG, int KG0, const char* __restrict__ A,
                  const char* __restrict__ B, int tm, int tn, int ksplit, int ks0, int kchunk,
                  EPI epi) {
  constexpr int RA = 2 * RB;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int fr = lane & 15, fk = lane >> 4;
  const long total = gridDim.x, xcd = blockIdx.x % 8, slot = blockIdx.x / 8;
  const long wg = xcd * (total / 8) + min(xcd, total % 8) + slot;
  const long q = wg * 4 + wave;
  if (q >= (long)tm * tn * ksplit) return;  // uniform per wavefront; no barrier in the kernel
  const int ks = (int)(q / ((long)tm * tn));
  const int t = (int)(q % ((long)tm * tn));
  const int strip = t / (2 * tm), in0 = 2 * strip, wd = min(2, tn - in0), rem = t - strip * 2 * tm;
  const int im = rem / wd, in = in0 + rem % wd;
  const int m0 = 16 * RB * im, n0 = 16 * CB * in;
  const int g0 = ks < ks0 ? ks * kchunk : KG0 + (ks - ks0) * kchunk;
  const int gn = min((ks < ks0 ? KG0 : KG) - g0, kchunk);
  const int rba = (M + 15) / 16, rbb = (N + 15) / 16;
  // blocks past the last row block read the last one; their results are never stored
  uint32_t oa[RA], ob[CB];
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    const long rb = min(RB * im + i, rba - 1);
    oa[2 * i] = (uint32_t)((2 * rb) * KG * kBlock);
    oa[2 * i + 1] = (uint32_t)((2 * rb + 1) * KG * kBlock);
  }
#pragma unroll
  for (int j = 0; j < CB; ++j) ob[j] = (uint32_t)((long)min(CB * in + j, rbb - 1) * KG * kBlock);
  f32x4 c[RA][CB];
#pragma unroll
  for (int i = 0; i < RA; ++i)
#pragma unroll
    for (int j = 0; j < CB; ++j) c[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int l16 = lane * 16;
  const auto rA = resource(A, (uint32_t)(2L * rba * KG * kBlock));
  const auto rB = resource(B, (uint32_t)((long)rbb * KG * kBlock));
  auto goff = [&](int u) {
    const int g = g0 + (REVK ? gn - 1 - u : u);
    return (uint32_t)(g * (int)kBlock);
  };
  bf16x8 a0[RA], a1[RA], a2[RA], b0[CB], b1[CB], b2[CB];
  uint32_t g = goff(0);
  auto load_b = [&](int j) {
    b0[j] = load_block<0>(rB, ob[j] + g, l16);
    b1[j] = load_block<1>(rB, ob[j] + g, l16);
    b2[j] = load_block<2>(rB, ob[j] + g, l16);
  };
  auto load_a2 = [&] {
#pragma unroll
    for (int i = 0; i < RA; ++i) a2[i] = load_block<2>(rA, oa[i] + g, l16);
  };
  auto load_a1 = [&] {
#pragma unroll
    for (int i = 0; i < RA; ++i) a1[i] = load_block<1>(rA, oa[i] + g, l16);
  };
  auto load_a0 = [&] {
#pragma unroll
    for (int i = 0; i < RA; ++i) a0[i] = load_block<0>(rA, oa[i] + g, l16);
  };
  // (in the order of the loop, so that the waits counted for its back edge hold on entry too)
#pragma unroll
  for (int j = 0; j < CB - 1; ++j) {
    load_b(j);
    __builtin_amdgcn_sched_barrier(0);
  }
  load_a2();
  __builtin_amdgcn_sched_barrier(0);
  load_a1();
  __builtin_amdgcn_sched_barrier(0);
  load_b(CB - 1);
  load_a0();
  __builtin_amdgcn_sched_barrier(0);
  for (int u = 0; u < gn; ++u) {
    g = goff(min(u + 1, gn - 1));  // the last group reloads itself
    f32x4 t[2][RA];
#pragma unroll
    for (int j = 0; j < CB; ++j) {
      f32x4(&x)[RA] = t[j & 1];
      const bool last = j == CB - 1;
#pragma unroll
      for (int i = 0; i < RA; ++i) x[i] = mfma(a2[i], b0[j], f32x4{0.f, 0.f, 0.f, 0.f});
      __builtin_amdgcn_sched_barrier(0);
      if (last) load_a2();
      if (j > 0) {  // the previous column's sums are complete by now
#pragma unroll
        for (int i = 0; i < RA; ++i) c[i][j - 1] += t[(j - 1) & 1][i];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < RA; ++i) x[i] = mfma(a1[i], b1[j], x[i]);
#pragma unroll
      for (int i = 0; i < RA; ++i) x[i] = mfma(a1[i], b0[j], x[i]);
      __builtin_amdgcn_sched_barrier(0);
      if (last) load_a1();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < RA; ++i) x[i] = mfma(a0[i], b2[j], x[i]);
#pragma unroll
      for (int i = 0; i < RA; ++i) x[i] = mfma(a0[i], b1[j], x[i]);
#pragma unroll
      for (int i = 0; i < RA; ++i) x[i] = mfma(a0[i], b0[j], x[i]);
      __builtin_amdgcn_sched_barrier(0);
      load_b(j);
      if (last) load_a0();
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < RA; ++i) c[i][CB - 1] += t[(CB - 1) & 1][i];
  }
  if (any_non_finite(c)) redo_non_finite(c, rA, oa, rB, ob, g0, gn, lane);
#pragma unroll
  for (int j = 0; j < CB; ++j) {
    const int n = n0 + 16 * j + fr;
    if (n >= N) continue;
    const auto col = epi.column(n);
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + 16 * i + 4 * fk + r;
        if (m < M) epi(ks, m, col, c[2 * i][j][r], c[2 * i + 1][j][r]);
      }
  }
}

}  // namespace s3
}  // namespace afq
