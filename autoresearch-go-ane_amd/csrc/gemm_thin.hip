// Which GEMMs run as gemm_thin_kernel (gemm_thin.h), in which form, and
// their launcher.
#include "gemm_thin.h"

namespace ane {
using namespace gemm_detail;

// The reduction length from which a split K pays for its second pass.
constexpr int kThinSplitK = 8192;

// The smallest tile that still fits the 256 CUs in one round: a smaller one
// brings more CUs' loads to bear, a second round costs the whole latency
// again.  Measured on MI355X with cold weights (us; the tile gemm_pick_tile
// takes -> this kernel), K-major, fp32 store:
//   M x N x K          before   32x32   32x64   64x64, 128 KB   64x64, 64 KB of LDS
//   256 x 768 x 768      8.2     3.5     4.4        5.5             5.7
//   256 x 768 x 2048    25.0     6.4     8.1       10.4            11.2
//   256 x 2048 x 768    11.1     5.7     5.3        6.5             6.8
//   512 x 768 x 2048    25.0     9.4     7.8       10.0            10.9
//   1024 x 768 x 2048   24.1    13.0    14.1        9.9            10.9
//   2240 x 768 x 2048   25.3    22.5    23.3       18.5            15.8
//   2240 x 768 x 768     9.7    12.1    13.6       10.2             8.6
// Past 512 blocks of 64x64 (two per CU) a short K loses (1216 x 2304 x 768
// 13.6 against 14.8, 2752 x 768 x 768 10.1 against 11.7); a long one still
// gains alone (4096 x 768 x 4096 50.9 against 42.0), but not beside the
// weight-gradient stream of a training step (12.93 against 13.06 ms per B16
// step and read-back with it), and at 1536 blocks no longer at all.
ThinTile gemm_pick_thin(int M, int N, int K, int epi) {
  ThinTile t;
  if (M <= 0 || N <= 0 || K <= 0 || M % 64 || N % 64 || K % BK || !thin_epi(epi)) return t;
  const long b64 = (long)(M / 64) * (N / 64);
  if (b64 > 512) return t;
  // A very long K (dy: K = the vocabulary) is split (gemm_pick_thin_splits),
  // which brings the blocks, so the tile is the one that reads least; once
  // two splits no longer fit one round, 256x256 tiles in up to 10 splits
  // read less still.  N = 768, us, before / this kernel: K = 32000, 64 rows
  // 30.6 / 18.3, 256 rows 37.4 / 33.6, 512 rows 54.6 / 56.4, 1024 rows 76 /
  // 87; K = 8192, 256 rows 15.6 / 13.8, 1024 rows 29.9 / 24.2 (one split).
  if (K >= kThinSplitK) {
    if (b64 <= (K < 2 * kThinSplitK ? 256 : 128)) t = {64, 64, 4, 2};
    return t;
  }
  // SwiGLU pairs 32-column blocks; the residual's row sums are per 64 columns
  const bool wide = epi == EPI_SWIGLU || epi == EPI_SWIGLU_RR || epi == EPI_RESID_NORM;
  if (!wide && 4 * b64 <= 256) t = {32, 32, 4, 2};
  else if (2 * b64 <= 256) t = {32, 64, 8, 1};
  else if (b64 <= 256) t = {64, 64, 4, 2};
  else t = {64, 64, 4, 1};
  return t;
}

int gemm_pick_thin_splits(int M, int N, int K, size_t ws_cap) {
  const ThinTile t = gemm_pick_thin(M, N, K, EPI_STORE_F);
  if (!t.bm || K < kThinSplitK) return 1;
  const long tiles = (long)(M / t.bm) * (N / t.bn);
  int best = 1;
  for (int sp = 2; sp <= kMaxSplits; sp++)
    if (K % (sp * BK) == 0 && (size_t)sp * M * N <= ws_cap && tiles * sp <= 256) best = sp;
  return best;
}

bool gemm_thin_aligned(const GemmArgs& g, int epi, const EpiParams& e) {
  auto a16 = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
  if (g.a_t || g.b_t || g.grp || !a16(g.A) || !a16(g.B) || g.lda % 8 || g.ldb % 8) return false;
  if (!a16(e.C) || !a16(e.C2) || !a16(e.R) || !a16(e.X0) || e.ldc % 8 || e.ldc2 % 8) return false;
  return epi != EPI_RESID_NORM || a16(e.gain);
}

namespace {
template <int EPI>
hipError_t thin_launch(const ThinTile& t, const GemmArgs& g, const EpiParams& e, hipStream_t s) {
  const dim3 grid((g.M / t.bm) * (g.N / t.bn) * g.splits);
#define ANE_THIN(BM_, BN_, KS_, DEP_)                                                                             \
  if (t.bm == BM_ && t.bn == BN_ && t.ks == KS_ && t.dep == DEP_) {                                               \
    hipLaunchKernelGGL((gemm_thin_kernel<BM_, BN_, EPI, KS_, DEP_>), grid, dim3(64 * KS_), 0, s, g, e);           \
    return hipGetLastError();                                                                                     \
  }
  if constexpr (EPI != EPI_SWIGLU && EPI != EPI_SWIGLU_RR && EPI != EPI_RESID_NORM) ANE_THIN(32, 32, 4, 2)
  ANE_THIN(32, 64, 8, 1)
  ANE_THIN(64, 64, 4, 2)
  ANE_THIN(64, 64, 4, 1)
#undef ANE_THIN
  return hipErrorInvalidValue;
}
}  // namespace

hipError_t gemm_thin_run(const ThinTile& t, const GemmArgs& g, int epi, const EpiParams& e, hipStream_t s) {
  switch (epi) {
    case EPI_STORE_H: return thin_launch<EPI_STORE_H>(t, g, e, s);
    case EPI_STORE_F: return thin_launch<EPI_STORE_F>(t, g, e, s);
    case EPI_RESID: return thin_launch<EPI_RESID>(t, g, e, s);
    case EPI_SWIGLU: return thin_launch<EPI_SWIGLU>(t, g, e, s);
    case EPI_RELU2: return thin_launch<EPI_RELU2>(t, g, e, s);
    case EPI_SMEAR: return thin_launch<EPI_SMEAR>(t, g, e, s);
    case EPI_SWIGLU_BWD: return thin_launch<EPI_SWIGLU_BWD>(t, g, e, s);
    case EPI_RELU2_BWD: return thin_launch<EPI_RELU2_BWD>(t, g, e, s);
    case EPI_RESID_NORM: return thin_launch<EPI_RESID_NORM>(t, g, e, s);
    case EPI_STORE_H_RR: return thin_launch<EPI_STORE_H_RR>(t, g, e, s);
    case EPI_SWIGLU_RR: return thin_launch<EPI_SWIGLU_RR>(t, g, e, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace ane
