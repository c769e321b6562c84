// Fused exchange and Coulomb contraction of the local energy (Real3IndexFactorization::energy,
// energy_impl, Real3IndexFactorization.hpp:476-590) for a real half-rotated tensor in FP32.
//
// For walker w and Cholesky vector m the n x n matrix T^m_ba = sum_k G[w][b][k] L[m][a][k] is
// formed on the matrix cores and reduced on chip to sum_ab T^m_ab T^m_ba (exchange) and
// sum_a T^m_aa (Coulomb); no T reaches memory.  A tile is two walkers x two Cholesky vectors: rows
// (walker, b) and columns (vector, a), each item padded to nsp = 8 NB >= n, so the tile is
// 16 NB x 16 NB and every (walker, vector) block lies inside it.
//   * Two wavefronts share a tile: one forms the real, the other the imaginary part of T, NB x NB
//     16 x 16 blocks each (100 accumulators at n = 40), so two wavefronts fit on a SIMD and one
//     multiplies while the other loads or reduces.
//   * The operands are packed bfloat16 pieces (split3.hpp: FP32 products as six bfloat16 MFMAs),
//     streamed from memory straight into MFMA operands; each piece's registers take the next k
//     group's values as soon as its last product has issued.
//   * The pairing T_ab T_ba crosses lanes, so the accumulators go through LDS: the columns of
//     one vector at a time, column-major ([nsp][2 nsp + 8] per tile and part), then each of the two
//     wavefronts takes one walker and adds the products in FP64 over 8 x 8 blocks of (b, a), using
//     the symmetry of the sum to visit only the blocks on and above the diagonal.  Each lane keeps
//     its own FP64 sums over all its tiles; a fixed-order wavefront reduction at the end gives one
//     exchange partial per (walker, tile run).
//   * Coulomb traces sum_a T^m_aa go to Kl[w][m] (added, so both spin blocks of a COLLINEAR
//     walker accumulate), each (w, m) owned by exactly one wavefront.
// A workgroup (four wavefronts, two tiles side by side in m) takes one walker pair and a run of
// 4 VPW Cholesky vectors; workgroups are renumbered so that each XCD processes a contiguous run
// with the walker pair fastest, so the workgroups resident on one XCD share their Cholesky vectors
// through its L2.
#include <algorithm>

#include "ops.hpp"
#include "split3.hpp"

namespace afq {

namespace {

using gemm::f32x4;
using s3::bf16x8;

constexpr int kXTiles = 2;  // tiles (pairs of wavefronts) per workgroup
constexpr int kXVpw = 4;    // tiles a pair of wavefronts takes one after the other

// LDS pitch of a column of T: the rows of both walkers plus 8, which keeps the 8 x 8 lane blocks of the
// exchange reads on distinct banks
template <int NB>
constexpr int kXPitch = 16 * NB + 8;

// What a wavefront of a tile works on
struct XTile {
  int W, ns, M, ldk, pair, cpart, lane;
  float* tre;  // LDS: real parts of the vector's columns of T, then the imaginary parts
  z64* Kl;
};

// Adds the exchange and Coulomb terms of vector 2 mt0 + mj, whose T lies in LDS.  A trace that is not
// finite is left out and noted in bit 2 vp + mj of `left`; LAST adds just those.
template <int NB, bool LAST>
__device__ inline void exx_terms(const XTile& x, int vp, int mt0, int mj, double& xr, double& xi,
                                 uint32_t& left) {
  constexpr int NSP = 8 * NB, LDC = kXPitch<NB>;
  const int xb = x.lane & 7, xa = x.lane >> 3;
  const int m = 2 * mt0 + mj, w = 2 * x.pair + x.cpart;
  if (m >= x.M || w >= x.W) return;  // uniform per wavefront
  const float* ur = x.tre + x.cpart * NSP;
  const float* ui = ur + NSP * LDC;
  // exchange: sum_ab T_ab T_ba over 8 x 8 blocks (ib, ia) of (b, a), lane (xb, xa) taking
  // b = 8 ib + xb, a = 8 ia + xa; the sum is symmetric in (a, b), so the blocks above the
  // diagonal count twice and those below are skipped
#pragma unroll
  for (int ib = 0; ib < NB; ++ib)
#pragma unroll
    for (int ia = ib; ia < NB; ++ia) {
      const int b = 8 * ib + xb, a = 8 * ia + xa;
      const double pr = ur[a * LDC + b], pi = ui[a * LDC + b];  // T_ba
      const double qr = ur[b * LDC + a], qi = ui[b * LDC + a];  // T_ab
      const double wgt = (b < x.ns && a < x.ns) ? (ia == ib ? 1.0 : 2.0) : 0.0;
      xr += wgt * (pr * qr - pi * qi);
      xi += wgt * (pr * qi + pi * qr);
    }
  // Coulomb trace of this (walker, vector)
  if (x.Kl) {
    double kr = 0.0, ki = 0.0;
    if (x.lane < x.ns) {
      kr = ur[x.lane * LDC + x.lane];
      ki = ui[x.lane * LDC + x.lane];
    }
    kr = wave_sum(kr);
    ki = wave_sum(ki);
    const bool fin = __builtin_isfinite(kr) && __builtin_isfinite(ki);  // the same in every lane
    if (!LAST && !fin) left |= 1u << (2 * vp + mj);
    if (x.lane == 0 && (LAST ? (left >> (2 * vp + mj) & 1u) != 0 : fin)) {
      z64* o = x.Kl + (long)w * x.ldk + m;
      *o = z64{o->re + kr, o->im + ki};
    }
  }
}

// The sums again for walkers whose T holds an infinity or NaN, with T from plain FP32 products: the split
// products turn an infinity into NaN (split3.hpp).  A walker with a NaN in both parts of G is NaN
// throughout either way.  One 16 x 16 block at a time: its registers must not weigh on the kernel's
// loop.  The energy of 1024 walkers (N = 200, n = 40, M = 1600) takes 10.4 ms, with 1 and 100 infinite
// ones 11.1 and 26.8, with NaN ones 10.5.
template <int NB>
__device__ inline z64 exx_redo(const XTile& x, int KG, const char* G, uint32_t gbytes,
                               const char* L, uint32_t lbytes, int tile, int mtile0, uint32_t* flags,
                               bool redo, z64 sum, uint32_t left) {
  constexpr int NSP = 8 * NB, LDC = kXPitch<NB>;
  const int l16 = x.lane * 16, fr = x.lane & 15, fk = x.lane >> 4;
  const auto rG = s3::resource(G, gbytes);
  const auto rL = s3::resource(L, lbytes);
  const uint32_t oa = (uint32_t)(((long)x.pair * 2 + x.cpart) * NB * KG * s3::kBlock);
  // the walkers with a NaN in this wavefront's part of G
  uint32_t nan = 0;
#pragma unroll 1
  for (int i = 0; i < NB; ++i)
    for (int g = 0; g < KG; ++g) {
      const bf16x8 p = s3::load_block<0>(rG, oa + (uint32_t)((i * KG + g) * (int)s3::kBlock), l16);
#pragma unroll
      for (int e = 0; e < 8; ++e) nan |= p[e] != p[e] ? (16 * i + fr < NSP ? 1u : 2u) : 0u;
    }
  const bool n0 = __ballot(nan & 1u) != 0, n1 = __ballot(nan & 2u) != 0;
  if (x.lane == 0) flags[2 * tile + x.cpart] = (n0 ? 1u : 0u) | (n1 ? 2u : 0u);
  __syncthreads();
  redo = redo && !((flags[2 * tile] & flags[2 * tile + 1]) >> x.cpart & 1u);
  __syncthreads();
  if (x.lane == 0) flags[2 * tile + x.cpart] = redo;
  __syncthreads();
  bool any = false;
#pragma unroll
  for (int i = 0; i < 2 * kXTiles; ++i) any = any || flags[i];
  if (__ballot(any) == 0) return sum;  // uniform per workgroup
  const bool own = __ballot(flags[2 * tile] || flags[2 * tile + 1]) != 0;
  double xr = 0.0, xi = 0.0;
  float* tmine = x.tre + (x.cpart ? NSP * LDC : 0);
#pragma unroll 1
  for (int v = 0; v < 2 * kXVpw; ++v) {
    const int mt0 = mtile0 + v / 2, mj = v & 1;
    __syncthreads();
#pragma unroll 1
    for (int ij = 0; ij < NB * NB && own && 2 * mt0 < x.M; ++ij) {
      const int i = ij / NB, j = ij % NB, col = 16 * j + fr - mj * NSP;
      const uint32_t ob = (uint32_t)(((long)mt0 * NB + j) * KG * s3::kBlock);
      f32x4 c = {0.f, 0.f, 0.f, 0.f};
      for (int g = 0; g < KG; ++g) {
        float a[8], b[8];
        s3::load_sums(a, rG, oa + (uint32_t)((i * KG + g) * (int)s3::kBlock), l16);
        s3::load_sums(b, rL, ob + (uint32_t)(g * (int)s3::kBlock), l16);
#pragma unroll
        for (int e = 0; e < 8; ++e) c = s3::mfma_f32(a[e], b[e], c);
      }
      if (col < 0 || col >= NSP) continue;
      // (an infinity times the zeros that pad a vector to NSP rows is NaN)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if ((16 * i + 4 * fk + r) % NSP >= x.ns || col >= x.ns) c[r] = 0.f;
      *reinterpret_cast<f32x4*>(tmine + col * LDC + 16 * i + 4 * fk) = c;
    }
    __syncthreads();
    exx_terms<NB, true>(x, v / 2, mt0, mj, xr, xi, left);
  }
  return redo ? z64{xr, xi} : sum;
}

template <int NB>
__global__ void __launch_bounds__(128 * kXTiles, 2)
    k_exx_split(int W, int ns, int KG, int M, int ldk, const char* __restrict__ G, uint32_t gbytes,
                const char* __restrict__ L, uint32_t lbytes, int npairs, z64* __restrict__ part,
                int nparts, z64* __restrict__ Kl) {
  constexpr int NSP = 8 * NB, LDC = kXPitch<NB>;
  extern __shared__ __align__(16) float smem_x[];  // [kXTiles][2][NSP * LDC]
  __shared__ uint32_t flags[2 * kXTiles];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cpart = wave & 1, tile = wave >> 1;  // real (0) or imaginary (1) part; the tile
  const long total = gridDim.x, xcd = blockIdx.x % 8, slot = blockIdx.x / 8;
  const long q = xcd * (total / 8) + min(xcd, total % 8) + slot;
  const int pair = (int)(q % npairs), chunk = (int)(q / npairs);
  const int mtiles = (M + 1) / 2;
  const auto rG = s3::resource(G, gbytes);
  const auto rL = s3::resource(L, lbytes);
  const int l16 = lane * 16;
  float* tre = smem_x + tile * 2 * NSP * LDC;
  float* tim = tre + NSP * LDC;
  float* tmine = cpart ? tim : tre;
  XTile x{W, ns, M, ldk, pair, cpart, lane, tre, Kl};
  double xr = 0.0, xi = 0.0;  // exchange of walker 2 pair + cpart
  uint32_t left = 0;          // bit 2 vp + mj: that vector's trace is left out

  for (int vp = 0; vp < kXVpw; ++vp) {
    const int mt0 = (chunk * kXTiles + tile) * kXVpw + vp;
    const bool live = mt0 < mtiles;  // uniform per pair of wavefronts
    const int mt = min(mt0, mtiles - 1);
    f32x4 c[NB][NB];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) c[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (live) {
      uint32_t oa[NB], ob[NB];
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        oa[i] = (uint32_t)((((long)pair * 2 + cpart) * NB + i) * KG * s3::kBlock);
        ob[i] = (uint32_t)(((long)mt * NB + i) * KG * s3::kBlock);
      }
      bf16x8 a0[NB], a1[NB], a2[NB], b0[NB], b1[NB], b2[NB];
      uint32_t g = 0;
#define AFQ_LD(F, PL, RES, OFS)                                                    \
  do {                                                                             \
    _Pragma("unroll") for (int i = 0; i < NB; ++i)                                 \
        F[i] = s3::load_block<PL>(RES, OFS[i] + g, l16);                           \
    __builtin_amdgcn_sched_barrier(0);                                             \
  } while (0)
#define AFQ_MM(A, B)                                                               \
  do {                                                                             \
    _Pragma("unroll") for (int i = 0; i < NB; ++i) _Pragma("unroll")               \
        for (int j = 0; j < NB; ++j) c[i][j] = s3::mfma(A[i], B[j], c[i][j]);      \
    __builtin_amdgcn_sched_barrier(0);                                             \
  } while (0)
      // (the loads in the order of the loop, so that the waits counted for its back edge hold)
      AFQ_LD(b2, 2, rL, ob);
      AFQ_LD(a2, 2, rG, oa);
      AFQ_LD(a0, 0, rG, oa);
      AFQ_LD(b0, 0, rL, ob);
      AFQ_LD(a1, 1, rG, oa);
      AFQ_LD(b1, 1, rL, ob);
      for (int u = 0; u < KG; ++u) {
        g = (uint32_t)(min(u + 1, KG - 1) * (int)s3::kBlock);  // the last group reloads itself
        AFQ_MM(a0, b2);
        AFQ_LD(b2, 2, rL, ob);
        AFQ_MM(a2, b0);
        AFQ_LD(a2, 2, rG, oa);
        AFQ_MM(a0, b1);
        AFQ_MM(a0, b0);
        AFQ_LD(a0, 0, rG, oa);
        AFQ_MM(a1, b0);
        AFQ_LD(b0, 0, rL, ob);
        AFQ_MM(a1, b1);
        AFQ_LD(a1, 1, rG, oa);
        AFQ_LD(b1, 1, rL, ob);
      }
#undef AFQ_LD
#undef AFQ_MM
    }
    // (opaque to the compiler, which would keep the reduction's LDS addresses in registers through the
    // products and spill them: 60 bytes a lane and 1.8 % of the time at n = 40)
    asm volatile("" : "+v"(x.lane));
    const int fr = x.lane & 15, fk = x.lane >> 4;
    // one Cholesky vector (tile columns mj NSP .. mj NSP + NSP - 1) at a time through LDS,
    // column-major: T[row][c] at c LDC + row, so each lane stores its four accumulator rows as
    // one 16-byte write
#pragma unroll
    for (int mj = 0; mj < 2; ++mj) {
      __syncthreads();  // the previous vector's reads are done
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int col = 16 * j + fr - mj * NSP;
        if (col < 0 || col >= NSP) continue;
#pragma unroll
        for (int i = 0; i < NB; ++i)
          *reinterpret_cast<f32x4*>(tmine + col * LDC + 16 * i + 4 * fk) = c[i][j];
      }
      __syncthreads();
      exx_terms<NB, false>(x, vp, mt0, mj, xr, xi, left);
    }
  }
  const bool redo = __ballot(!(__builtin_isfinite(xr) && __builtin_isfinite(xi))) != 0;
  if (lane == 0) flags[wave] = redo;
  __syncthreads();
  bool any = false;
#pragma unroll
  for (int i = 0; i < 2 * kXTiles; ++i) any = any || flags[i];
  if (__ballot(any) != 0) {  // uniform per workgroup
    __syncthreads();  // (the flags are read)
    const z64 r = exx_redo<NB>(x, KG, G, gbytes, L, lbytes, tile,
                               (chunk * kXTiles + tile) * kXVpw, flags, redo, z64{xr, xi}, left);
    xr = r.re;
    xi = r.im;
  }
  const double er = wave_sum(xr), ei = wave_sum(xi);
  const int w = 2 * pair + cpart;
  if (lane == 0 && w < W) part[(long)w * nparts + chunk * kXTiles + tile] = z64{er, ei};
}

// The Cholesky vectors in runs whose packed pieces the kernel's 32-bit offsets reach
template <int NB>
void launch_exx(hipStream_t s, int W, int ns, int N, int M, const char* G, const char* L,
                z64* part, int nparts, z64* Kl) {
  constexpr int kChunk = 2 * kXTiles * kXVpw;  // vectors of a workgroup
  const int npairs = ceil_div(W, 2);
  AFQ_CHECK(nparts == ceil_div(M, kChunk) * kXTiles, kErrArg, "exchange partial count");
  constexpr int NSP = 8 * NB;
  constexpr size_t lds = sizeof(float) * kXTiles * 2 * NSP * kXPitch<NB>;
  static_assert(lds <= 64 * 1024, "the default LDS limit");
  const size_t per = s3::bytes_exx_L(kChunk, ns, N);
  const int run = (int)std::min<size_t>((size_t)M, kChunk * std::max<size_t>(1, 0xFFFF0000u / per));
  for (int m0 = 0; m0 < M; m0 += run) {
    const int mc = std::min(run, M - m0), c0 = m0 / kChunk;
    const long blocks = (long)npairs * ceil_div(mc, kChunk);
    AFQ_CHECK(blocks < (1L << 31), kErrShape, "grid too large");
    hipLaunchKernelGGL((k_exx_split<NB>), dim3((unsigned)blocks), dim3(128 * kXTiles), lds, s, W,
                       ns, (int)s3::k_groups(N), mc, M, G, (uint32_t)s3::bytes_exx_G(W, ns, N),
                       L + c0 * per, (uint32_t)s3::bytes_exx_L(mc, ns, N), npairs,
                       part + c0 * kXTiles, nparts, Kl ? Kl + m0 : nullptr);
    AFQ_LAUNCH_CHECK();
  }
}

}  // namespace

int exx_fused_parts(int M) { return ceil_div(M, 2 * kXTiles * kXVpw) * kXTiles; }

void exchange_fused(hipStream_t s, int W, int ns, int N, int M, const void* G, const void* L,
                    z64* part, int nparts, z64* Kl) {
  AFQ_CHECK(ns >= 1 && ns <= 40 && s3::bytes_exx_G(W, ns, N) < (size_t)0xFFFF0000u, kErrShape,
            "fused exchange supports 1 <= n <= 40 and a packed G under 4 GiB");
  const char* g = static_cast<const char*>(G);
  const char* l = static_cast<const char*>(L);
  switch (s3::exx_nb(ns)) {
    case 1: launch_exx<1>(s, W, ns, N, M, g, l, part, nparts, Kl); break;
    case 2: launch_exx<2>(s, W, ns, N, M, g, l, part, nparts, Kl); break;
    case 3: launch_exx<3>(s, W, ns, N, M, g, l, part, nparts, Kl); break;
    case 4: launch_exx<4>(s, W, ns, N, M, g, l, part, nparts, Kl); break;
    default: launch_exx<5>(s, W, ns, N, M, g, l, part, nparts, Kl); break;
  }
}

}  // namespace afq
