// Phi <- P1 expM(V) P1 Phi in FP32 on the bfloat16 matrix cores (propagate_impl + apply_expM,
// propagate.hpp:41-70, :241-298), one launch for both one-body products and every Taylor term.
//
// The Taylor recurrence T_k = (i/k) V T_{k-1} and both P1 products act on each column of the
// walker matrix separately, so a workgroup owns one walker and up to 40 of its columns.  The current
// term lives in LDS as the B operand of v_mfma_f32_16x16x32_bf16, split into three bfloat16 pieces
// (split3.hpp) in the order of the instruction's operand: [16-column block][32-k group][piece]
// [lane], so every read is one conflict-free 16-byte word a lane.  Each wavefront owns 16-row
// stripes of the result: it streams the matching rows of V (or P1) from memory as FP32, splits
// them in registers and multiplies, and keeps its accumulators and its part of the running sum S in
// registers.
//
// Columns.  A block of 16 columns has one LDS block for the real and one for the imaginary parts
// (a pair); the up to 8 columns past a multiple of 16 share one mixed block, real parts in its
// first 8 columns and imaginary parts in the last 8, so 40 columns take exactly 5 blocks.  With
// V = Vr + i Vi and T = Tr + i Ti a pair takes Vr Tr - Vi Ti and Vr Ti + Vi Tr; the mixed block M
// takes Vr M + Vi M' with M' = (-Ti | Tr), read from M with the lanes' columns exchanged.
//
// Stripes.  Eight wavefronts (four when N <= 64) take one stripe each, two above N = 128, dealt in
// rows of four, so the SIMDs carry equal shares; the one or two stripes past a multiple of four are
// split by column blocks over the four wavefronts of their row (N = 200: 13 stripes of 5 blocks;
// the busiest SIMD carries 17 of the 65 blocks).  Every block is summed in the same order
// whichever wavefront owns it, so neither this nor the number of columns per workgroup (a tuner
// candidate) changes a bit.
//
// V.  Up to N = 128 a stripe of V (64 registers a lane as FP32) stays in registers for all Taylor
// terms: at these sizes a k group is multiplied faster than memory answers, and a stream of V was
// bound by that latency (N = 97, n = 23, 301 walkers: 93 us).  Above, V is streamed once per term,
// one k group ahead; two stripes a wavefront read the B operand half as often as one.
//
// P1 is close to the identity, and the products of a 32-deep bfloat16 MFMA are aligned to the largest
// of each eight before they are added, which truncates the many small ones beside a diagonal
// entry.  So a diagonal entry between 1/2 and 2 enters as P1_ii - 1 (exact) and the row's own entry
// of the operand is added to the finished sum in FP32.
//
// FP32 range: the tile enters scaled by 2^-e, e the binary exponent of its largest entry, and
// leaves scaled back by 2^e.
//
// Bound by the matrix cores and by V, which is read from memory once per term (the V of the resident
// walkers does not fit the L2s): the cores are busy 45 % of the time at N = 200.  Against the same
// recurrence on FP32 MFMAs (six terms; errors against 64 bits 0.3 to 0.6 of its): N = 200, n = 40,
// 1024 walkers 1020 -> 639 us, 128 walkers 189 -> 113 us, N = 97, n = 23, 301 walkers 97 -> 75 us;
// with a complex P1 N = 24, n = 5, 64 walkers 13.4 -> 11.3 us, N = 160, n = 40, 256 walkers 192 -> 179
// us.  Above 16 columns and N = 64 the registers do not suffice: 32 to 144 bytes a lane are spilled,
// outside the k loops, and with a complex P1 up to 720.  So every size and both kinds of P1 that fit take
// this kernel.
#include <cstdlib>
#include <type_traits>

#include "ops.hpp"
#include "split3.hpp"
#include "tuner.hpp"

namespace afq {
namespace det_ops {

namespace {

using gemm::f32x4;
using s3::bf16x8;
using s3::u32x4;
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

constexpr int kMaxCols = 40;  // columns of one workgroup

// Eight consecutive k values of one row of A (complex: 64 bytes).  The loads go through a buffer
// resource of the N x N matrix: past its end (the k values past N of the last row) they return
// zero.  A 16-byte buffer load asks for 4-byte alignment only, so rows of any N take the same loads.
template <bool CPLX>
struct Raw {
  uint32_t v[CPLX ? 16 : 8];
};
template <bool CPLX>
__device__ inline void load_raw(Raw<CPLX>& r, __amdgpu_buffer_rsrc_t a, int vofs) {
#pragma unroll
  for (int j = 0; j < (CPLX ? 16 : 8); j += 4) {
    const u32x4 x =
        __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(a, vofs + 4 * j, 0, 0));
#pragma unroll
    for (int t = 0; t < 4; ++t) r.v[j + t] = x[t];
  }
}

__device__ inline void read_block(bf16x8 (&f)[3], const char* lds, int blk, int KG, int g,
                                  int lane16) {
  const char* p = lds + (blk * KG + g) * (int)s3::kBlock + lane16;
#pragma unroll
  for (int c = 0; c < 3; ++c) f[c] = *reinterpret_cast<const bf16x8*>(p + c * s3::kPlane);
}

// t += the five partial products of a b between 2^-24 and 2^-7 of it
__device__ inline f32x4 mul_small(const bf16x8 (&a)[3], const bf16x8 (&b)[3], f32x4 t) {
  t = s3::mfma(a[2], b[0], t);
  t = s3::mfma(a[0], b[2], t);
  t = s3::mfma(a[1], b[1], t);
  t = s3::mfma(a[1], b[0], t);
  return s3::mfma(a[0], b[1], t);
}

// changes the signs of the values whose bits `sign` selects
__device__ inline void flip(bf16x8 (&a)[3], uint32_t sign) {
#pragma unroll
  for (int c = 0; c < 3; ++c)
    a[c] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, a[c]) ^
                                          u32x4{sign, sign, sign, sign});
}

// the value of the lane 8 columns further (lane ^ 8)
__device__ inline float lane_xor8(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xF, 0xF, true));
}

// A wavefront's stripes (st < 0: none) and the column blocks it owns of each (bit t < P: pair t,
// bit P: the mixed block).  A slot before the last owns all of its stripe.
template <int SLOTS>
struct Share {
  int st[SLOTS];
  uint32_t mask[SLOTS];
};

template <int P, int X>
struct Blocks {
  f32x4 re[P > 0 ? P : 1], im[P > 0 ? P : 1], mx;
};
template <int P, int X, int SLOTS>
using Accs = Blocks<P, X>[SLOTS];

// The pieces of one k group of a stripe: real and imaginary parts
template <bool CPLX>
struct Pieces {
  bf16x8 r[3], i[CPLX ? 3 : 1];
};

// The rows of A that a wavefront multiplies, RES k groups in registers: all of them, or (RES = 1,
// KG > 1) one, the next one loading while it is multiplied.  UNIT (P1): diagonal entries between
// 1/2 and 2 are reduced by one; bit r of unit[s] is set when row r of stripe s is such a row.
template <bool CPLX, bool UNIT, int RES, int SLOTS>
struct Rows {
  static constexpr int E = CPLX ? 8 : 4, GB = 32 * E;  // bytes of a value, of a k group in a row
  Raw<CPLX> raw[SLOTS][RES];
  int vofs[SLOTS], dk[SLOTS];
  uint32_t unit[SLOTS];
  __amdgpu_buffer_rsrc_t a;

  __device__ inline void init(const float* A, int N, const Share<SLOTS>& sh, int fr, int fk) {
    a = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(A), 0, (uint32_t)(N * N * E),
                                          0x00027000);
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
      // (rows past the last read it; their results are stored as zero or not at all)
      const int row = min(max(sh.st[s], 0) * 16 + fr, N - 1);
      vofs[s] = (row * N + 8 * fk) * E;
      if constexpr (UNIT) {
        const float d = A[(long)row * (N + 1) * (E / 4)];
        const bool u = d >= 0.5f && d <= 2.f;
        unit[s] = (uint32_t)__ballot(u) & 0xFFFFu;
        dk[s] = u ? (row & 31) - 8 * fk : -1;  // the entry's place among the lane's eight
      }
    }
  }
  // loads every group (RES > 1) or the first one
  __device__ inline void start(int KG) {
#pragma unroll
    for (int s = 0; s < SLOTS; ++s)
#pragma unroll
      for (int g = 0; g < RES; ++g)
        if (g < KG) load_raw<CPLX>(raw[s][g], a, vofs[s] + g * GB);
  }
  __device__ inline void next(int g) {
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) load_raw<CPLX>(raw[s][0], a, vofs[s] + g * GB);
    __builtin_amdgcn_sched_barrier(0);
  }
  // the pieces of group g, held in raw[s][i].  TAIL: k values >= left are zero
  template <bool TAIL>
  __device__ inline void pieces(Pieces<CPLX>& p, int s, int i, int g, int left, int st) const {
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      x[j] = !TAIL || j < left ? __uint_as_float(raw[s][i].v[CPLX ? 2 * j : j]) : 0.f;
    if (UNIT && g == st >> 1) {  // uniform
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] -= j == dk[s] ? 1.f : 0.f;
    }
    s3::split8_finite(x, p.r);
    if constexpr (CPLX) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        x[j] = !TAIL || j < left ? __uint_as_float(raw[s][i].v[2 * j + 1]) : 0.f;
      s3::split8_finite(x, p.i);
    }
  }
};

// acc += A B over one k group (FULL: the last slot owns every block, no branches).  SUM0: the small
// partial products are summed from zero and added to the accumulator once, after the large ones
// (more accurate, 8 more registers a slot).
template <bool CPLX, int P, int X, int SLOTS, bool SUM0, bool FULL>
__device__ inline void group(const Pieces<CPLX> (&A)[SLOTS], int g, int KG,
                             const Share<SLOTS>& sh, int lane16, int lanex16, uint32_t msign,
                             const char* lds, Accs<P, X, SLOTS>& acc) {
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  auto owns = [&](int s, int t) { return FULL || s + 1 < SLOTS || (sh.mask[s] >> t & 1u); };
  // (the same order of the products in a pair and in the mixed block)
#pragma unroll
  for (int t = 0; t < P; ++t) {
    if (SLOTS == 1 && !owns(0, t)) continue;
    bf16x8 br[3], bi[3];
    read_block(br, lds, 2 * t, KG, g, lane16);
    read_block(bi, lds, 2 * t + 1, KG, g, lane16);
    f32x4 tr[SLOTS], ti[SLOTS];
#pragma unroll
    for (int s = 0; s < SLOTS; ++s)
      if (owns(s, t)) {
        f32x4 &re = acc[s].re[t], &im = acc[s].im[t];
        tr[s] = mul_small(A[s].r, br, SUM0 ? zero : re);
        ti[s] = mul_small(A[s].r, bi, SUM0 ? zero : im);
        (SUM0 ? re : tr[s]) = s3::mfma(A[s].r[0], br[0], SUM0 ? re : tr[s]);
        (SUM0 ? im : ti[s]) = s3::mfma(A[s].r[0], bi[0], SUM0 ? im : ti[s]);
      }
    if constexpr (CPLX) flip(bi, 0x80008000u);
#pragma unroll
    for (int s = 0; s < SLOTS; ++s)
      if (owns(s, t)) {
        f32x4 &re = acc[s].re[t], &im = acc[s].im[t];
        if constexpr (CPLX) {
          tr[s] = mul_small(A[s].i, bi, tr[s]);
          ti[s] = mul_small(A[s].i, br, ti[s]);
          (SUM0 ? re : tr[s]) = s3::mfma(A[s].i[0], bi[0], SUM0 ? re : tr[s]);
          (SUM0 ? im : ti[s]) = s3::mfma(A[s].i[0], br[0], SUM0 ? im : ti[s]);
        }
        re = SUM0 ? re + tr[s] : tr[s];
        im = SUM0 ? im + ti[s] : ti[s];
      }
  }
  if constexpr (X) {
    if (SLOTS == 1 && !owns(0, P)) return;
    bf16x8 b[3], c[3];
    read_block(b, lds, 2 * P, KG, g, lane16);
    if constexpr (CPLX) {
      read_block(c, lds, 2 * P, KG, g, lanex16);
      flip(c, msign);
    }
#pragma unroll
    for (int s = 0; s < SLOTS; ++s)
      if (owns(s, P)) {
        f32x4& mx = acc[s].mx;
        f32x4 t = mul_small(A[s].r, b, SUM0 ? zero : mx);
        (SUM0 ? mx : t) = s3::mfma(A[s].r[0], b[0], SUM0 ? mx : t);
        if constexpr (CPLX) {
          t = mul_small(A[s].i, c, t);
          (SUM0 ? mx : t) = s3::mfma(A[s].i[0], c[0], SUM0 ? mx : t);
        }
        mx = SUM0 ? mx + t : t;
      }
  }
}

template <int P, int X, int SLOTS>
__device__ inline void clear(Accs<P, X, SLOTS>& acc) {
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
#pragma unroll
    for (int t = 0; t < P; ++t) acc[s].re[t] = acc[s].im[t] = zero;
    acc[s].mx = zero;
  }
}

// acc = A[stripes][0:N] B (without the units of A's diagonal)
template <int P, int X, int SLOTS, bool SUM0, bool FULL, bool CPLX, bool UNIT, int RES>
__device__ inline void product(Rows<CPLX, UNIT, RES, SLOTS>& A, int N, int KG,
                               const Share<SLOTS>& sh, int fr, int fk, const char* lds,
                               Accs<P, X, SLOTS>& acc) {
  const int lane16 = (fr + 16 * fk) * 16, lanex16 = ((fr ^ 8) + 16 * fk) * 16;
  const uint32_t msign = fr < 8 ? 0x80008000u : 0u;
  clear<P, X, SLOTS>(acc);
  const int left = N - 32 * (KG - 1) - 8 * fk;  // k values of the lane in the last group
  Pieces<CPLX> p[SLOTS];
  if constexpr (RES > 1) {
#pragma unroll
    for (int g = 0; g < RES; ++g) {
      if (g >= KG) break;  // uniform
#pragma unroll
      for (int s = 0; s < SLOTS; ++s)
        A.template pieces<true>(p[s], s, g, g, g + 1 < KG ? 8 : left, sh.st[s]);
      group<CPLX, P, X, SLOTS, SUM0, FULL>(p, g, KG, sh, lane16, lanex16, msign, lds, acc);
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
    for (int g = 0; g + 1 < KG; ++g) {
      // the registers of a group are free for the next one's values once it is split
#pragma unroll
      for (int s = 0; s < SLOTS; ++s) A.template pieces<false>(p[s], s, 0, g, 8, sh.st[s]);
      A.next(g + 1);
      group<CPLX, P, X, SLOTS, SUM0, FULL>(p, g, KG, sh, lane16, lanex16, msign, lds, acc);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) A.template pieces<true>(p[s], s, 0, KG - 1, left, sh.st[s]);
    group<CPLX, P, X, SLOTS, SUM0, FULL>(p, KG - 1, KG, sh, lane16, lanex16, msign, lds, acc);
  }
}

// the same with the pieces of all groups in registers
template <int P, int X, bool FULL, int RES>
__device__ inline void product(const Pieces<true> (&A)[RES], int KG, const Share<1>& sh, int fr,
                               int fk, const char* lds, Accs<P, X, 1>& acc) {
  const int lane16 = (fr + 16 * fk) * 16, lanex16 = ((fr ^ 8) + 16 * fk) * 16;
  const uint32_t msign = fr < 8 ? 0x80008000u : 0u;
  clear<P, X, 1>(acc);
#pragma unroll
  for (int g = 0; g < RES; ++g) {
    if (g >= KG) break;  // uniform
    const Pieces<true> p[1] = {A[g]};
    group<true, P, X, 1, true, FULL>(p, g, KG, sh, lane16, lanex16, msign, lds, acc);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// four consecutive rows (k0 .. k0 + 3, a multiple of 4) of one column from LDS block blk: the pieces
// summed, which is the FP32 value they were split from
__device__ inline f32x4 read4(const char* lds, int blk, int KG, int k0, int col) {
  const char* o = lds + (blk * KG + (k0 >> 5)) * (int)s3::kBlock +
                  (((k0 >> 3) & 3) * 16 + col) * 16 + (k0 & 4) * 2;
  f32x4 v;
  bf16x4 p[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) p[c] = *reinterpret_cast<const bf16x4*>(o + c * s3::kPlane);
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = ((float)p[0][r] + (float)p[1][r]) + (float)p[2][r];
  return v;
}

// acc += x for the rows of the stripe whose bit is set in unit
__device__ inline void add_unit(f32x4& acc, const f32x4& x, uint32_t unit, int fk) {
#pragma unroll
  for (int r = 0; r < 4; ++r) acc[r] += (unit >> (4 * fk + r) & 1u) ? x[r] : 0.f;
}

// four consecutive rows (k0 .. k0 + 3, a multiple of 4) of one column into LDS block blk
__device__ inline void write4(char* lds, int blk, int KG, int k0, int col, int N, f32x4 v) {
  bf16x4 p[3];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float x = k0 + r < N ? v[r] : 0.f;
    const __bf16 h = (__bf16)x;
    const float e = x - (float)h;
    const __bf16 m = (__bf16)e;
    p[0][r] = h;
    p[1][r] = m;
    p[2][r] = (__bf16)(e - (float)m);
  }
  char* o = lds + (blk * KG + (k0 >> 5)) * (int)s3::kBlock + (((k0 >> 3) & 3) * 16 + col) * 16 +
            (k0 & 4) * 2;
#pragma unroll
  for (int c = 0; c < 3; ++c) *reinterpret_cast<bf16x4*>(o + c * s3::kPlane) = p[c];
}

template <int P, int X, int SLOTS>
__device__ inline void write_share(char* lds, int KG, int N, const Share<SLOTS>& sh, int fr,
                                   int fk, const Accs<P, X, SLOTS>& v) {
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
    const int k0 = sh.st[s] * 16 + 4 * fk;
#pragma unroll
    for (int t = 0; t < P; ++t)
      if (sh.mask[s] >> t & 1u) {
        write4(lds, 2 * t, KG, k0, fr, N, v[s].re[t]);
        write4(lds, 2 * t + 1, KG, k0, fr, N, v[s].im[t]);
      }
    if (X && (sh.mask[s] >> P & 1u)) write4(lds, 2 * P, KG, k0, fr, N, v[s].mx);
  }
}

// k groups of V and P1 that a wavefront holds in registers (1: streams them)
template <int SLOTS, int WAVES>
constexpr int kResident = SLOTS == 2 ? 1 : WAVES / 2;

// A workgroup's part of the work
struct Tile {
  const float *P1, *V;  // V: this walker's
  z64* Pw;
  int N, n, c0, c1, order, e, wave;
};

// One wavefront's recurrence (FULL: it owns every block of its last stripe); every wavefront passes
// the same barriers.  False, with the walker as it was, where a sum is not finite.
template <int P, int X, int SLOTS, int WAVES, bool P1C, bool FULL>
__device__ inline bool recur(Rows<P1C, true, kResident<SLOTS, WAVES>, SLOTS>& rp,
                             Rows<true, false, kResident<SLOTS, WAVES>, SLOTS>& rv, int KG,
                             const Tile& a, const Share<SLOTS>& sh, int& fr, int& fk,
                             uint32_t* votes, char* lds) {
  // the running sum takes the rounded term, whichever way a block is laid out
#pragma clang fp contract(off)
  constexpr int RES = kResident<SLOTS, WAVES>;
  constexpr bool SUM0 = SLOTS == 1;
  const int N = a.N, n = a.n, order = a.order, c0 = a.c0, c1 = a.c1, e = a.e;
  z64* Pw = a.Pw;
  Accs<P, X, SLOTS> acc, S;
  // T_0 = P1 Phi, S = T_0
  __syncthreads();
  product<P, X, SLOTS, SUM0, FULL>(rp, N, KG, sh, fr, fk, lds, acc);
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
    const int k0 = max(sh.st[s], 0) * 16 + 4 * fk;
#pragma unroll
    for (int t = 0; t < P; ++t) {
      add_unit(acc[s].re[t], read4(lds, 2 * t, KG, k0, fr), rp.unit[s], fk);
      add_unit(acc[s].im[t], read4(lds, 2 * t + 1, KG, k0, fr), rp.unit[s], fk);
      S[s].re[t] = acc[s].re[t];
      S[s].im[t] = acc[s].im[t];
    }
    if constexpr (X) add_unit(acc[s].mx, read4(lds, 2 * P, KG, k0, fr), rp.unit[s], fk);
    S[s].mx = acc[s].mx;
  }
  Pieces<true> vp[RES];
  if constexpr (RES == 1) {
    rv.start(KG);
  } else {
    const int left = N - 32 * (KG - 1) - 8 * fk;
#pragma unroll
    for (int g = 0; g < RES; ++g)
      if (g < KG) rv.template pieces<true>(vp[g], 0, g, g, g + 1 < KG ? 8 : left, 0);
  }
  __syncthreads();
  write_share<P, X, SLOTS>(lds, KG, N, sh, fr, fk, acc);
  __syncthreads();
  for (int k = 1;; ++k) {
    // (opaque to the compiler, which would keep every address of the loop in a register)
    asm volatile("" : "+v"(fr), "+v"(fk));
    if constexpr (RES == 1) product<P, X, SLOTS, SUM0, FULL>(rv, N, KG, sh, fr, fk, lds, acc);
    else product<P, X, FULL>(vp, KG, sh, fr, fk, lds, acc);
    // T_k = (i / k) V T_{k-1}; S += T_k
    const float f = (float)(1.0 / (double)k);
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
#pragma unroll
      for (int t = 0; t < P; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float tr = -(f * acc[s].im[t][r]), ti = f * acc[s].re[t][r];
          acc[s].re[t][r] = tr;
          acc[s].im[t][r] = ti;
          S[s].re[t][r] += tr;
          S[s].im[t][r] += ti;
        }
      if constexpr (X) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float o = lane_xor8(acc[s].mx[r]);
          const float v = fr < 8 ? -(f * o) : f * o;
          acc[s].mx[r] = v;
          S[s].mx[r] += v;
        }
      }
    }
    if (k == order) break;
    if constexpr (RES == 1) rv.start(KG);
    __syncthreads();
    write_share<P, X, SLOTS>(lds, KG, N, sh, fr, fk, acc);
    __syncthreads();
  }
  rp.start(KG);
  asm volatile("" : "+v"(fr), "+v"(fk));
  // (x 0 is 0 for every finite x)
  f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
#pragma unroll
    for (int t = 0; t < P; ++t)
      if (sh.mask[s] >> t & 1u) z += S[s].re[t] * 0.f + S[s].im[t] * 0.f;
    if (X && (sh.mask[s] >> P & 1u)) z += S[s].mx * 0.f;
  }
  const bool bad = __ballot(!((z[0] + z[1]) + (z[2] + z[3]) == 0.f)) != 0;
  if (fr + fk == 0) votes[a.wave] = bad;
  __syncthreads();
  bool any = false;
#pragma unroll
  for (int i = 0; i < WAVES; ++i) any = any || votes[i];
  if (__ballot(any) != 0) return false;  // uniform per workgroup
  write_share<P, X, SLOTS>(lds, KG, N, sh, fr, fk, S);
  __syncthreads();
  // Phi = P1 S, scaled back by 2^e
  product<P, X, SLOTS, SUM0, FULL>(rp, N, KG, sh, fr, fk, lds, acc);
  const double sb = e == 0 ? 1.0 : ldexp(1.0, e);
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
#pragma unroll
    for (int t = 0; t < P; ++t) {
      add_unit(acc[s].re[t], S[s].re[t], rp.unit[s], fk);
      add_unit(acc[s].im[t], S[s].im[t], rp.unit[s], fk);
    }
    if constexpr (X) add_unit(acc[s].mx, S[s].mx, rp.unit[s], fk);
  }
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = sh.st[s] * 16 + 4 * fk + r;
#pragma unroll
      for (int t = 0; t < P; ++t) {
        const int col = c0 + 16 * t + fr;
        if ((sh.mask[s] >> t & 1u) && row < N && col < c1)
          Pw[(long)row * n + col] =
              z64{(double)acc[s].re[t][r] * sb, (double)acc[s].im[t][r] * sb};
      }
      if constexpr (X) {
        const float im = lane_xor8(acc[s].mx[r]);
        const int col = c0 + 16 * P + fr;
        if ((sh.mask[s] >> P & 1u) && fr < 8 && row < N && col < c1)
          Pw[(long)row * n + col] = z64{(double)acc[s].mx[r] * sb, (double)im * sb};
      }
    }
  }
  return true;
}

// The workgroup's columns from plain FP32 products, for a walker whose sum came out infinite or NaN: the
// split turns an infinity into NaN.  (A NaN in V or P1, or in a column, makes NaN of all its columns,
// or of that one, in any arithmetic, without products.)  Columns by halves, so that the term, its
// successor and the running sum fit where the pieces lay.  A function of its own, called when nothing
// else is live: inlined, or with the sums kept across it, its registers cost the kernel 1 to 25 %.  One
// infinite walker of 1024 (N = 200, n = 40) takes 3.0 ms instead of 0.87, 100 of them 4.1.
template <int P, int X, int WAVES, bool P1C>
__device__ __attribute__((noinline)) void redo_plain(Tile a, int tid, uint32_t* votes, char* lds) {
#pragma clang fp contract(off)
  constexpr int NC = 16 * P + 8 * X, H = NC / 2, TH = 64 * WAVES;
  const int N = a.N;
  auto vote = [&](bool v) {
    const bool mine = __ballot(v) != 0;
    __syncthreads();
    if ((tid & 63) == 0) votes[tid >> 6] = mine;
    __syncthreads();
    bool any = false;
    for (int i = 0; i < WAVES; ++i) any = any || votes[i];
    return __ballot(any) != 0;
  };
  // a column without a NaN (a dead walker's have one in the first row)
  auto clean = [&](int rows) {
    bool any = false;
    for (int c = tid; c < a.c1 - a.c0; c += TH) {
      bool nan = false;
      for (int k = 0; k < rows; ++k) {
        const z64 v = a.Pw[(long)k * a.n + a.c0 + c];
        nan = nan || v.re != v.re || v.im != v.im;
      }
      any = any || !nan;
    }
    return any;
  };
  bool products = vote(clean(1)) && vote(clean(N));
  if (products) {
    bool nan = false;
    for (int t = tid; t < 2 * N * N; t += TH) {
      nan = nan || a.V[t] != a.V[t];
      if (P1C || t < N * N) nan = nan || a.P1[t] != a.P1[t];
    }
    products = !vote(nan);
  }
  if (!products) {
    const double nan = __builtin_nan("");
    for (int t = tid; t < N * (a.c1 - a.c0); t += TH)
      a.Pw[(long)(t / (a.c1 - a.c0)) * a.n + a.c0 + t % (a.c1 - a.c0)] = z64{nan, nan};
    return;
  }
  float2* T = reinterpret_cast<float2*>(lds);
  float2 *U = T + N * H, *S = U + N * H;
  const double sc = ldexp(1.0, -a.e), sb = ldexp(1.0, a.e);
  // element (row, c) of A T
  auto dot = [&](const float* A, auto cplx, const float2* B, int row, int c) {
    float re = 0.f, im = 0.f;
    for (int k = 0; k < N; ++k) {
      const float2 b = B[k * H + c];
      if constexpr (decltype(cplx)::value) {
        const float ar = A[2 * ((long)row * N + k)], ai = A[2 * ((long)row * N + k) + 1];
        re = fmaf(-ai, b.y, fmaf(ar, b.x, re));
        im = fmaf(ai, b.x, fmaf(ar, b.y, im));
      } else {
        const float ar = A[(long)row * N + k];
        re = fmaf(ar, b.x, re);
        im = fmaf(ar, b.y, im);
      }
    }
    return float2{re, im};
  };
  for (int h = 0; h < NC; h += H) {
    __syncthreads();
    for (int t = tid; t < N * H; t += TH) {
      const int col = a.c0 + h + t % H;
      const z64 v = col < a.c1 ? a.Pw[(long)(t / H) * a.n + col] : z64{0.0, 0.0};
      T[t] = float2{(float)(v.re * sc), (float)(v.im * sc)};
    }
    __syncthreads();
    for (int t = tid; t < N * H; t += TH)
      S[t] = U[t] = dot(a.P1, std::bool_constant<P1C>{}, T, t / H, t % H);
    for (int k = 1; k <= a.order; ++k) {
      const float f = (float)(1.0 / (double)k);
      __syncthreads();
      for (int t = tid; t < N * H; t += TH) {
        const float2 x = dot(a.V, std::true_type{}, U, t / H, t % H);
        T[t] = float2{-(f * x.y), f * x.x};
        S[t].x += T[t].x;
        S[t].y += T[t].y;
      }
      float2* const o = T;
      T = U;
      U = o;
    }
    __syncthreads();
    for (int t = tid; t < N * H; t += TH) {
      const int col = a.c0 + h + t % H;
      const float2 x = dot(a.P1, std::bool_constant<P1C>{}, S, t / H, t % H);
      if (col < a.c1) a.Pw[(long)(t / H) * a.n + col] = z64{(double)x.x * sb, (double)x.y * sb};
    }
  }
}

// P1C: complex P1.  (The last bound keeps three workgroups a CU where 168 registers allow them.)
template <int P, int X, int SLOTS, int WAVES, bool P1C>
__global__ void __launch_bounds__(64 * WAVES, WAVES == 4 && P == 1 && !P1C ? 3 : 2)
    k_prop_split(int W, int N, int n, int nchunk, int order, const float* __restrict__ P1,
                 const float* __restrict__ V, long v_bs, z64* __restrict__ Phi, long phi_bs) {
  constexpr int NC = 16 * P + 8 * X;
  extern __shared__ __align__(16) char lds[];
  __shared__ double wmx[WAVES];
  __shared__ uint32_t votes[WAVES];
  const int NS = (N + 15) / 16, KG = (N + 31) / 32;
  const long total = gridDim.x, xcd = blockIdx.x % 8, slot = blockIdx.x / 8;
  const long q = xcd * (total / 8) + min(xcd, total % 8) + slot;
  const int w = (int)(q / nchunk), ch = (int)(q % nchunk);
  // this workgroup's columns: the n columns in nchunk runs of whole 8-column groups
  const int n8 = (n + 7) / 8, c0 = 8 * (n8 * ch / nchunk), c1 = min(n, 8 * (n8 * (ch + 1) / nchunk));
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int fr = lane & 15, fk = lane >> 4;
  z64* Pw = Phi + (long)w * phi_bs;
  const float* Vw = V + 2 * (long)w * v_bs;

  // the stripes and blocks of this wavefront (rows of four stripes, the last one split)
  constexpr uint32_t ALL = (1u << (P + X)) - 1u;
  const int base = NS & ~3, rem = NS - base, quad = wave & 3;
  Share<SLOTS> sh;
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
    const int st = s * WAVES + wave;
    sh.st[s] = -1;
    sh.mask[s] = 0;
    if (st < base || (rem == 3 && st < NS)) {
      sh.st[s] = st;
      sh.mask[s] = ALL;
    } else if (st - quad == base && (rem == 1 || rem == 2)) {
      const int part = rem == 1 ? quad : quad >> 1, parts = rem == 1 ? 4 : 2;
      sh.st[s] = base + (rem == 1 ? 0 : quad & 1);
#pragma unroll
      for (int t = 0; t < P + X; ++t)
        if (t % parts == part) sh.mask[s] |= 1u << t;
    }
  }

  // the first rows of P1 and V load while the walker does
  constexpr int RES = kResident<SLOTS, WAVES>;
  Rows<P1C, true, RES, SLOTS> rp;
  Rows<true, false, RES, SLOTS> rv;
  rp.init(P1, N, sh, fr, fk);
  rv.init(Vw, N, sh, fr, fk);
  rp.start(KG);
  if constexpr (RES > 1) rv.start(KG);

  // the tile (8 rows of a column a thread and item), its binary scale, then its entries scaled,
  // split and laid out; rows past N and columns past n are zero
  constexpr int IT = (NC * SLOTS + 31) / 32;  // >= items per thread: KG <= SLOTS WAVES / 2
  const int items = NC * KG * 4;
  z64 val[IT][8];
  double mx = 0.0;
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int t = tid + i * 64 * WAVES, c = t % NC, k0 = 8 * (t / NC);
    const bool in = t < items && c0 + c < c1;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      val[i][j] = in && k0 + j < N ? Pw[(long)(k0 + j) * n + c0 + c] : z64{0.0, 0.0};
  }
#pragma unroll
  for (int i = 0; i < IT; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) mx = fmax(mx, fmax(fabs(val[i][j].re), fabs(val[i][j].im)));
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mx = fmax(mx, __shfl_xor(mx, off, 64));
  if (lane == 0) wmx[wave] = mx;
  __syncthreads();
  mx = 0.0;
#pragma unroll
  for (int i = 0; i < WAVES; ++i) mx = fmax(mx, wmx[i]);
  int e = 0;
  if (mx > 0.0 && mx <= 1.7976931348623157e308) e = __builtin_amdgcn_readfirstlane(ilogb(mx));
  const double sc = ldexp(1.0, -e);
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int t = tid + i * 64 * WAVES, c = t % NC, k0 = 8 * (t / NC);
    if (t >= items) continue;
    float re[8], im[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      re[j] = (float)(val[i][j].re * sc);
      im[j] = (float)(val[i][j].im * sc);
    }
    bf16x8 p[3];
    const bool mixed = c >= 16 * P;
    const int blk = mixed ? 2 * P : 2 * (c >> 4), col = mixed ? c - 16 * P : c & 15;
    char* o = lds + (blk * KG + (k0 >> 5)) * (int)s3::kBlock + (((k0 >> 3) & 3) * 16 + col) * 16;
    s3::split8_finite(re, p);
#pragma unroll
    for (int x = 0; x < 3; ++x) *reinterpret_cast<bf16x8*>(o + x * s3::kPlane) = p[x];
    o += mixed ? 8 * 16 : KG * (int)s3::kBlock;
    s3::split8_finite(im, p);
#pragma unroll
    for (int x = 0; x < 3; ++x) *reinterpret_cast<bf16x8*>(o + x * s3::kPlane) = p[x];
  }

  const Tile a{P1, Vw, Pw, N, n, c0, c1, order, e, wave};
  bool done;
  if (sh.mask[SLOTS - 1] == ALL)
    done = recur<P, X, SLOTS, WAVES, P1C, true>(rp, rv, KG, a, sh, fr, fk, votes, lds);
  else
    done = recur<P, X, SLOTS, WAVES, P1C, false>(rp, rv, KG, a, sh, fr, fk, votes, lds);
  if (__ballot(!done) != 0)  // uniform per workgroup
    redo_plain<P, X, WAVES, P1C>(a, 64 * wave + 16 * fk + fr, votes, lds);
}

template <int P, int X, int SLOTS, int WAVES>
void launch(hipStream_t s, const PropagateArgs& a, const float* P1, bool p1c, z64* Phi,
            int nchunk) {
  const int KG = ceil_div(a.N, 32);
  const size_t lds = (size_t)(2 * P + X) * KG * s3::kBlock;
  const float* V = reinterpret_cast<const float*>(a.V);
  auto go = [&](auto kern) {
    if (lds > 48 * 1024)
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(kern, dim3((unsigned)((long)a.W * nchunk)), dim3(64 * WAVES), lds, s, a.W,
                       a.N, a.n, nchunk, a.order, P1, V, a.v_bs, Phi, a.phi_bs);
  };
  if (p1c) go(k_prop_split<P, X, SLOTS, WAVES, true>);
  else go(k_prop_split<P, X, SLOTS, WAVES, false>);
  AFQ_LAUNCH_CHECK();
}

}  // namespace

bool propagate_split(Context& c, const PropagateArgs& a) {
  const char* m3 = std::getenv("AFQ_PROP_M3");
  const int N = a.N, n = a.n, NS = ceil_div(N, 16);
  if (a.TA != 'N' || a.order < 1 || NS > 16 || (m3 && m3[0] == '1'))
    return false;
  const bool p1c = a.P1r32 == nullptr;
  const float* P1 = p1c ? &a.P1c32->re : a.P1r32;
  // workgroups per walker: the fewest whose columns fit, and up to three more candidates (fewer
  // columns each: V is read more often, but more workgroups fill the machine)
  const int n8 = ceil_div(n, 8), lo = ceil_div(n8, kMaxCols / 8);
  int cand[4], ncand = 0;
  for (int k = lo; k <= n8 && ncand < 4; ++k)
    if (ncand == 0 || ceil_div(n8, k) < ceil_div(n8, cand[ncand - 1])) cand[ncand++] = k;
  AFQ_CHECK((long)a.W * n8 < (1L << 31), kErrShape, "grid too large");
  hipStream_t s = c.stream();
  auto run = [&](int i, z64* Phi) {
    const int k = cand[i], cols = 8 * ceil_div(n8, k);
#define AFQ_PSP(P, X)                                                                     \
  do {                                                                                    \
    if (NS <= 4) launch<P, X, 1, 4>(s, a, P1, p1c, Phi, k);                               \
    else if (NS <= 8) launch<P, X, 1, 8>(s, a, P1, p1c, Phi, k);                          \
    else launch<P, X, 2, 8>(s, a, P1, p1c, Phi, k);                                       \
  } while (0)
    if (cols <= 8) AFQ_PSP(0, 1);
    else if (cols <= 16) AFQ_PSP(1, 0);
    else if (cols <= 24) AFQ_PSP(1, 1);
    else if (cols <= 32) AFQ_PSP(2, 0);
    else AFQ_PSP(2, 1);
#undef AFQ_PSP
  };
  // (a candidate means other work with another kind of P1 or number of 8-column groups)
  tuned_on_copy(c,
                tune_key("prop_fused", sizeof(float), a.W, N, n, N) + (p1c ? ":c" : ":r") +
                    std::to_string(n8),
                ncand, a.Phi, (size_t)a.W * a.phi_bs, run);
  return true;
}

}  // namespace det_ops
}  // namespace afq
