// The FP32 contractions of the mixed precision on the bfloat16 matrix cores (split3.hpp): packing
// of the operands and the two products of the walker step, vHS and vbias.
#include <algorithm>

#include "split3.hpp"

namespace afq {
namespace s3 {

// Tile and K slices of a product: the fewest MFMAs on the busiest of the 1024 SIMDs, weighted by
// what a tile's MFMAs cost.  The weights are the measured times per MFMA of a full machine
// against the 32 x 96 tile (the smaller the tile, the more operand bytes per MFMA); a SIMD with a
// single wavefront has nothing to run while that one waits, which costs 15 %.  Slices keep at
// least 4 k groups and the partials' traffic is counted against them.  The rule depends on the
// shape only (measured: 128 x 20100 over 1600 takes 32 x 80, 88 us against 97 with 32 x 96 and 109
// with 32 x 64; 301 x 4753 over 487 takes 16 x 96, 25 us against 35, 32 and 28).
constexpr int kTiles = 4;
constexpr int kTileRB[kTiles] = {2, 2, 2, 1}, kTileCB[kTiles] = {6, 5, 4, 6};

static Plan plan(int M, int N, int KG0, int KG1, bool split_k) {
  constexpr double kWeight[kTiles] = {1.0, 1.05, 1.15, 1.34};
  const int KG = std::max(KG0, KG1);
  Plan best{0, 1, KG, 1};
  double tb = 1e300;
  for (int t = 0; t < kTiles; ++t) {
    const int rb = kTileRB[t], cb = kTileCB[t];
    const long tiles = (long)ceil_div(M, 16 * rb) * ceil_div(N, 16 * cb);
    const int cap = split_k ? std::max(1, std::min(KG / 4, 16)) : 1;
    for (int c = 1; c <= cap; ++c) {
      const int kc = ceil_div(KG, c);
      if (ceil_div(KG, kc) != c) continue;
      const int ks0 = ceil_div(KG0, kc), ks = ks0 + ceil_div(KG1, kc);
      if (c > 1 && ks > 16) continue;
      const long per_simd = (tiles * ks + 1023) / 1024;
      // 12 MFMAs of 16 cycles per block and k group; partials: 16 bytes per element and slice at
      // about 2 bytes a cycle and SIMD
      double x = (double)per_simd * rb * cb * kc * 12 * 16 * kWeight[t];
      if (per_simd == 1) x *= 1.15;
      if (ks > 1) x += 4000.0 + 16.0 * ks * M * (double)N / 2048.0;
      if (x < tb * 0.999) {
        tb = x;
        best = Plan{t, ks, kc, ks0};
      }
    }
  }
  return best;
}

namespace {

template <typename TIn, class ROWS>
void pack_cplx_t(hipStream_t s, long blocks, int K0, int K1, const cplx<TIn>* X, long ld,
                 const ROWS& rmap, int nb, void* out) {
  const long KG = k_groups(K0) + k_groups(K1), waves = blocks * KG;
  if (waves == 0) return;
  AFQ_CHECK((waves + 3) / 4 < (1L << 31), kErrShape, "grid too large");
  hipLaunchKernelGGL((k_pack_cplx<TIn, ROWS>), dim3((unsigned)ceil_div(waves, 4)), dim3(256), 0, s,
                     blocks, K0, (int)k_groups(K0), K0 + K1, (int)KG, X, ld, rmap, nb,
                     static_cast<char*>(out));
  AFQ_LAUNCH_CHECK();
}

template <class ROWS>
void pack_real_t(hipStream_t s, long blocks, int K, const float* X, long ld, const ROWS& rmap,
                 void* out, long ldg, long g0, int* bad) {
  const long KG = k_groups(K), waves = blocks * KG;
  if (waves == 0) return;
  AFQ_CHECK((waves + 3) / 4 < (1L << 31), kErrShape, "grid too large");
  hipLaunchKernelGGL((k_pack_real<ROWS>), dim3((unsigned)ceil_div(waves, 4)), dim3(256), 0, s,
                     blocks, K, (int)KG, X, ld, rmap, static_cast<char*>(out), (int)ldg, (int)g0,
                     bad);
  AFQ_LAUNCH_CHECK();
}

template <int RB, int CB, bool REVK, class EPI>
void launch_tile(hipStream_t s, int M, int N, int KG, int KG0, const void* A, const void* B,
                 const Plan& p, const EPI& e) {
  const int tm = ceil_div(M, 16 * RB), tn = ceil_div(N, 16 * CB);
  const long blocks = ceil_div((long)tm * tn * p.ksplit, 4);
  AFQ_CHECK(blocks < (1L << 31), kErrShape, "grid too large");
  hipLaunchKernelGGL((k_split3_gemm<RB, CB, REVK, EPI>), dim3((unsigned)blocks), dim3(256), 0, s, M,
                     N, KG, KG0, static_cast<const char*>(A), static_cast<const char*>(B), tm, tn,
                     p.ksplit, p.ks0, p.kchunk, e);
  AFQ_LAUNCH_CHECK();
}

template <bool REVK, class EPI>
void launch_planned(hipStream_t s, int M, int N, int KG, int KG0, const void* A, const void* B,
                    const Plan& p, const EPI& e) {
  switch (p.tile) {
    case 0: launch_tile<2, 6, REVK>(s, M, N, KG, KG0, A, B, p, e); break;
    case 1: launch_tile<2, 5, REVK>(s, M, N, KG, KG0, A, B, p, e); break;
    case 2: launch_tile<2, 4, REVK>(s, M, N, KG, KG0, A, B, p, e); break;
    default: launch_tile<1, 6, REVK>(s, M, N, KG, KG0, A, B, p, e); break;
  }
}

// C = epi(A B^T): one launch, or K slices whose FP32 partials (ws [ksplit][M][N]) are summed in
// slice order in FP64 before the epilogue.
template <bool REVK, class EPI>
void product_splitk(hipStream_t s, int M, int N, int KG, int KG0, const void* A, const void* B,
                    const Plan& p, const EPI& e, c32* ws) {
  if (p.ksplit == 1) {
    launch_planned<REVK>(s, M, N, KG, KG0, A, B, p, Plain<EPI>{e});
    return;
  }
  launch_planned<REVK>(s, M, N, KG, KG0, A, B, p,
                       Plain<gemm::EpiPartial<float>>{{ws, (long)M * N, N}});
  const long tot = (long)M * N;
  hipLaunchKernelGGL((gemm::kreduce_splitk<float, EPI>), dim3((unsigned)ceil_div(tot, 256)),
                     dim3(256), 0, s, 1, M, N, p.ksplit, ws, e);
  AFQ_LAUNCH_CHECK();
}

}  // namespace

void pack_cplx(hipStream_t s, int rows, int K0, int K1, const c32* X, long ld, void* out) {
  pack_cplx_t(s, row_blocks(rows), K0, K1, X, ld, RowsPlain{rows}, 1, out);
}
void pack_cplx(hipStream_t s, int rows, int K0, int K1, const z64* X, long ld, void* out) {
  pack_cplx_t(s, row_blocks(rows), K0, K1, X, ld, RowsPlain{rows}, 1, out);
}
void pack_rows(hipStream_t s, int rows, int K, const float* X, long ld, void* out, long ldg,
               long g0, int* bad) {
  pack_real_t(s, row_blocks(rows), K, X, ld, RowsPlain{rows}, out, ldg, g0, bad);
}
void pack_pairs(hipStream_t s, int rows, int K, const float* X, int N, const uint32_t* pairs,
                void* out, int* bad) {
  pack_real_t(s, row_blocks(rows), K, X, K, RowsPairs{pairs, rows, N}, out, k_groups(K), 0, bad);
}
void pack_exx_G(hipStream_t s, int W, int n, int N, const z64* G, void* out) {
  const int nb = exx_nb(n);
  pack_cplx_t(s, (long)ceil_div(W, 2) * nb, N, 0, G, N, RowsItems{W, n, 8 * nb}, nb, out);
}
void pack_exx_L(hipStream_t s, int M, int n, int N, const float* L, void* out, int* bad) {
  const int nb = exx_nb(n);
  pack_real_t(s, (long)ceil_div(M, 2) * nb, N, L, N, RowsItems{M, n, 8 * nb}, out, k_groups(N), 0,
              bad);
}

void vhs_pairs(hipStream_t s, int W, int np, int K, const void* A, const void* B,
               const uint32_t* pairs, int N, float alpha, c32* V) {
  const int KG = (int)k_groups(K);
  launch_planned<true>(s, W, np, KG, KG, A, B, plan(W, np, KG, 0, false),
                       EpiPairs{V, pairs, N, alpha, 0.f});
}

Plan vbias_plan(int W, int M, int K0, int K1) {
  return plan(W, M, (int)k_groups(K0), (int)k_groups(K1), true);
}

void vbias(hipStream_t s, int W, int M, int K0, int K1, const Plan& p, const void* A,
           const void* B, float alpha, z64* v, c32* ws) {
  const int KG0 = (int)k_groups(K0), KG = KG0 + (int)k_groups(K1);
  // the vectors in runs that the 32-bit offsets reach
  const long per = KG * kBlock;  // of 16 vectors
  const int run = 16 * (int)std::max<long>(1, 0xFFFF0000L / per);
  for (int m0 = 0; m0 < M; m0 += run) {
    const gemm::EpiStore<float, double> e{v + m0, M, 0, alpha, 0.f, 0};
    product_splitk<false>(s, W, std::min(run, M - m0), KG, KG0, A,
                          static_cast<const char*>(B) + m0 / 16 * per, p, e, ws);
  }
}

}  // namespace s3
}  // namespace afq
