// GEMM kernel for outputs too small to fill the chip with the tiles of
// gemm_ho_kernel (a window or two of tokens: 256 x 768 is 48 blocks of 64x64).
//
// There the time is memory latency, not MFMA: a 64x64 block walks its K in
// 64-wide steps with two stages and one barrier each, so every step waits
// out a load issued one step before (K = 768, cold weights: 12 steps at
// ~1 us).  Here the waves of a block share one small output tile and split
// its K: wave w takes k-tiles w, w + KS, ..., each with an LDS ring of its
// own that only it fills (the same swizzled global_load_lds tiles) and only
// it reads, so nothing but its own loads ever holds it up: no barrier until
// the end, and KS * DEP k-tiles of the block in flight from the start.  The
// waves' partial tiles then meet in LDS, are added in wave order (so the
// result does not depend on timing) and leave through an epilogue in which
// each thread owns 4 consecutive columns: 16-byte accesses, and what the
// epilogue reads (residual, x0, saved activations) is requested before the
// main loop.
//
// K-major operands (A [M][K], B [N][K]); M % BM == 0, N % BN == 0, K % 64 == 0.
#pragma once
#include "gemm_impl.h"

namespace ane {
namespace gemm_detail {

// The epilogues the kernel has (those of the layers; the classifier's
// outputs are large enough for the other kernels).
__host__ __device__ constexpr bool thin_epi(int epi) {
  return epi == EPI_STORE_H || epi == EPI_STORE_F || epi == EPI_RESID || epi == EPI_SWIGLU || epi == EPI_RELU2 ||
         epi == EPI_SMEAR || epi == EPI_SWIGLU_BWD || epi == EPI_RELU2_BWD || epi == EPI_RESID_NORM ||
         epi == EPI_STORE_H_RR || epi == EPI_SWIGLU_RR;
}

template <int N>
__device__ __forceinline__ void wait_vm_mem() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ float4 ld_f4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ void st_h4(half_t* p, float a, float b, float c, float d) {
  half4 h;
  h[0] = (half_t)a; h[1] = (half_t)b; h[2] = (half_t)c; h[3] = (half_t)d;
  *reinterpret_cast<half4*>(p) = h;
}
__device__ __forceinline__ float4 ld_h4f(const half_t* p) {
  const half4 h = *reinterpret_cast<const half4*>(p);
  return make_float4((float)h[0], (float)h[1], (float)h[2], (float)h[3]);
}

template <int BM, int BN, int EPI, int KS, int DEP>
__global__ __launch_bounds__(64 * KS) void gemm_thin_kernel(GemmArgs g, EpiParams e) {
  constexpr int TM = BM / 32, TN = BN / 32;
  constexpr int STAGE = (BM + BN) * BK;      // halves
  constexpr int LPT = (BM + BN) / 8;         // load instructions per k-tile
  // row stride of a partial tile (floats): the pad puts rows r and r + 4 on
  // other banks, where the ring has room for it
  constexpr int SW = BM * (BN + 8) * 4 <= DEP * STAGE * 2 ? BN + 8 : BN;
  constexpr bool PAIR = EPI == EPI_SWIGLU || EPI == EPI_SWIGLU_RR;  // h1 | h3 in adjacent 32-column blocks
  constexpr int CPR = (PAIR ? BN / 2 : BN) / 4;                     // 4-column groups per row
  constexpr int NG = BM * CPR;                                      // groups of the tile
  constexpr int NE = (NG + 64 * KS - 1) / (64 * KS);                // groups per thread
  static_assert(LPT * (DEP > 1 ? DEP - 1 : 1) < 64, "vmcnt range");
  static_assert(!PAIR || BN % 64 == 0, "SwiGLU pairs 32-column blocks");
  static_assert(BM * SW * 4 <= DEP * STAGE * 2, "a wave's partial tile lies in its own ring");
  static_assert(EPI != EPI_RESID_NORM || CPR == 16, "row sums reduce over 16 lanes");
  __shared__ __attribute__((aligned(16))) half_t lds[KS * DEP * STAGE];
  __shared__ float rr_s[epi_rr(EPI) ? BM : 1];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ntiles = (g.M / BM) * (g.N / BN);
  int bid = blockIdx.x, ks = 0;
  if (g.splits > 1) {
    ks = bid / ntiles;
    bid -= ks * ntiles;
  }
  int bm, bn;
  block_tile(g.M / BM, g.N / BN, bid, bm, bn);
  const int m0 = bm * BM, n0 = bn * BN;
  const int nk = g.K / BK / g.splits;
  const half_t* A = g.A + (size_t)m0 * g.lda + (size_t)ks * nk * BK;
  const half_t* B = g.B + (size_t)n0 * g.ldb + (size_t)ks * nk * BK;
  const int nw = nk > wave ? (nk - wave + KS - 1) / KS : 0;  // this wave's k-tiles

  half_t* ring = lds + wave * (DEP * STAGE);
  const unsigned ring0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(lds_ptr_t)ring);
  // load q of a tile fills rows 8 q + lane / 8; lane's slot lane % 8 holds
  // the chunk that swz maps there
  const int c0 = (lane & 7) ^ (lane >> 3);
  const unsigned ra = (unsigned)((lane >> 3) * g.lda * 2), rb = (unsigned)((lane >> 3) * g.ldb * 2);
  auto issue = [&](int i) {
    const int kt = wave + KS * i;
    const unsigned st = ring0 + (unsigned)((i % DEP) * STAGE * 2);
#pragma unroll
    for (int q = 0; q < BM / 8; q++)
      dma16_s(A + (size_t)(q * 8) * g.lda + kt * BK, ra + (unsigned)((c0 ^ (q & 7)) * 16), st + (unsigned)(q * 1024));
#pragma unroll
    for (int q = 0; q < BN / 8; q++)
      dma16_s(B + (size_t)(q * 8) * g.ldb + kt * BK, rb + (unsigned)((c0 ^ (q & 7)) * 16),
              st + (unsigned)(BM * BK * 2 + q * 1024));
  };

  // what the epilogue reads, requested first (C may be R: each element is
  // read and written by the same thread)
  float4 p0[NE], p1[NE];
  float rrv[epi_rr(EPI) ? kRrMaxParts : 1];
  auto grp_row = [&](int u) { return (tid + 64 * KS * u) / CPR; };
  auto grp_col = [&](int u) { return (tid + 64 * KS * u) % CPR * 4; };
  auto live = [&](int u) { return NG % (64 * KS) == 0 || tid + 64 * KS * u < NG; };
  if constexpr (epi_rr(EPI)) {
#pragma unroll
    for (int p = 0; p < kRrMaxParts; p++)
      rrv[p] = tid < BM && p < e.rr_nparts ? e.rr_part[(size_t)p * e.rr_ld + m0 + tid] : 0.f;
  }
#pragma unroll
  for (int u = 0; u < NE; u++) {
    p0[u] = p1[u] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (!live(u)) continue;
    const int row = m0 + grp_row(u), col = n0 + grp_col(u);
    const size_t at = (size_t)row * e.ldc + col;
    if constexpr (EPI == EPI_STORE_F) {
      if (e.accumulate && g.splits == 1) p0[u] = ld_f4((const float*)e.C + at);
    } else if constexpr (EPI == EPI_RESID) {
      p0[u] = ld_f4(e.R + at);
      if (e.X0) p1[u] = ld_f4(e.X0 + at);
    } else if constexpr (EPI == EPI_RESID_NORM) {
      p0[u] = ld_f4(e.R + at);
      p1[u] = ld_f4(e.gain + col);
    } else if constexpr (EPI == EPI_SMEAR) {
      p0[u] = ld_f4(e.X0 + at);
      if (row % e.seq != 0) p1[u] = ld_f4(e.X0 + at - e.ldc);
    } else if constexpr (EPI == EPI_RELU2_BWD) {
      p0[u] = ld_h4f((const half_t*)e.C2 + (size_t)row * e.ldc2 + col);
    } else if constexpr (EPI == EPI_SWIGLU_BWD) {
      const half_t* h = (const half_t*)e.C2 + (size_t)row * e.ldc2 + (col >> 5) * 64 + (col & 31);
      p0[u] = ld_h4f(h);
      p1[u] = ld_h4f(h + 32);
    }
  }
  asm volatile("" ::: "memory");

#pragma unroll
  for (int i = 0; i < DEP; i++)
    if (i < nw) issue(i);

  floatx16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;
  const int frow = lane & 31, fch = lane >> 5;
  for (int i = 0; i < nw; i++) {
    // tile i is in once at most the later tiles' loads are outstanding
    const int later = min(nw - 1 - i, DEP - 1);
    if (DEP > 3 && later == 3) wait_vm_mem<LPT * (DEP > 3 ? 3 : 0)>();
    else if (DEP > 2 && later == 2) wait_vm_mem<LPT * (DEP > 2 ? 2 : 0)>();
    else if (DEP > 1 && later == 1) wait_vm_mem<LPT * (DEP > 1 ? 1 : 0)>();
    else wait_vm_mem<0>();
    const half_t* st = ring + (i % DEP) * STAGE;
    half8 fa[4][TM], fb[4][TN];
#pragma unroll
    for (int s = 0; s < 4; s++) {
#pragma unroll
      for (int a = 0; a < TM; a++) fa[s][a] = ld_h8(st + (a * 32 + frow) * BK + swz(a * 32 + frow, 2 * s + fch) * 8);
#pragma unroll
      for (int b = 0; b < TN; b++)
        fb[s][b] = ld_h8(st + (BM + b * 32 + frow) * BK + swz(b * 32 + frow, 2 * s + fch) * 8);
    }
    if (i + DEP < nw) {
      // the stage is refilled once its reads have returned
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      issue(i + DEP);
    }
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int a = 0; a < TM; a++)
#pragma unroll
        for (int b = 0; b < TN; b++)
          acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[s][a], fb[s][b], acc[a][b], 0, 0, 0);
  }

  // partial tiles, each in its wave's own ring (its reads are done)
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  constexpr int SLAB = DEP * STAGE / 2;  // floats between two waves' rings
  float* slab = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int a = 0; a < TM; a++)
#pragma unroll
    for (int b = 0; b < TN; b++)
#pragma unroll
      for (int r = 0; r < 16; r++)
        slab[wave * SLAB + (a * 32 + 8 * (r >> 2) + 4 * fch + (r & 3)) * SW + b * 32 + frow] = acc[a][b][r];
  if constexpr (epi_rr(EPI)) {
    if (tid < BM) {
      float sum = 0.f;
#pragma unroll
      for (int p = 0; p < kRrMaxParts; p++)
        if (p < e.rr_nparts) sum += rrv[p];
      rr_s[tid] = 1.0f / sqrtf(sum / (float)e.rr_dim + 1e-5f);
    }
  }
  __syncthreads();
  auto total = [&](int row, int col) {
    float4 v = ld_f4(slab + row * SW + col);
#pragma unroll
    for (int w = 1; w < KS; w++) {
      const float4 x = ld_f4(slab + w * SLAB + row * SW + col);
      v.x += x.x; v.y += x.y; v.z += x.z; v.w += x.w;
    }
    return v;
  };
  float alpha = e.alpha, beta = e.beta;
  if constexpr (EPI == EPI_RESID || EPI == EPI_SMEAR) {
    if (e.alpha_ptr) alpha = *e.alpha_ptr;
    if (e.beta_ptr) beta = *e.beta_ptr;
  }
#pragma unroll
  for (int u = 0; u < NE; u++) {
    if (!live(u)) continue;
    const int lr = grp_row(u), lc = grp_col(u), row = m0 + lr, col = n0 + lc;
    const size_t at = (size_t)row * e.ldc + col;
    if constexpr (PAIR) {
      // columns 64 q + [0, 32) are W1's, the next 32 W3's
      const int c1 = (lc >> 5) * 64 + (lc & 31);
      float4 h1 = total(lr, c1), h3 = total(lr, c1 + 32);
      if constexpr (EPI == EPI_SWIGLU_RR) {
        const float rr = rr_s[lr];
        h1.x *= rr; h1.y *= rr; h1.z *= rr; h1.w *= rr;
        h3.x *= rr; h3.y *= rr; h3.z *= rr; h3.w *= rr;
      }
      const int hc = (n0 >> 1) + lc;
      st_h4((half_t*)e.C + (size_t)row * e.ldc + hc, h1.x * sigmoid_f(h1.x) * h3.x, h1.y * sigmoid_f(h1.y) * h3.y,
            h1.z * sigmoid_f(h1.z) * h3.z, h1.w * sigmoid_f(h1.w) * h3.w);
      if (e.C2) {
        half_t* d = (half_t*)e.C2 + (size_t)row * e.ldc2 + n0 + c1;
        st_h4(d, h1.x, h1.y, h1.z, h1.w);
        st_h4(d + 32, h3.x, h3.y, h3.z, h3.w);
      }
      continue;
    }
    const float4 v = total(lr, lc);
    if constexpr (EPI == EPI_STORE_H || EPI == EPI_STORE_H_RR) {
      const float s = EPI == EPI_STORE_H_RR ? rr_s[lr] * e.scale : e.scale;
      st_h4((half_t*)e.C + at, v.x * s, v.y * s, v.z * s, v.w * s);
    } else if constexpr (EPI == EPI_STORE_F) {
      float* C = (float*)e.C + (g.splits > 1 ? (size_t)ks * g.M * g.N : 0);  // (workspace slice: ldc = N, scale 1)
      *reinterpret_cast<float4*>(C + at) = make_float4(p0[u].x + v.x * e.scale, p0[u].y + v.y * e.scale,
                                                       p0[u].z + v.z * e.scale, p0[u].w + v.w * e.scale);
    } else if constexpr (EPI == EPI_RESID) {
      const float4 o = make_float4(alpha * p0[u].x + v.x + beta * p1[u].x, alpha * p0[u].y + v.y + beta * p1[u].y,
                                   alpha * p0[u].z + v.z + beta * p1[u].z, alpha * p0[u].w + v.w + beta * p1[u].w);
      *reinterpret_cast<float4*>((float*)e.C + at) = o;
      if (e.C2) *reinterpret_cast<float4*>((float*)e.C2 + at) = o;
    } else if constexpr (EPI == EPI_RESID_NORM) {
      const float4 o = make_float4(p0[u].x + v.x, p0[u].y + v.y, p0[u].z + v.z, p0[u].w + v.w);
      *reinterpret_cast<float4*>((float*)e.C + at) = o;
      st_h4((half_t*)e.C2 + (size_t)row * e.ldc2 + col, o.x * p1[u].x, o.y * p1[u].y, o.z * p1[u].z, o.w * p1[u].w);
      // the row's 16 lanes (consecutive, 64 columns) to one sum
      float ss = o.x * o.x + o.y * o.y + o.z * o.z + o.w * o.w;
#pragma unroll
      for (int m = 1; m < 16; m <<= 1) ss += __shfl_xor(ss, m, 64);
      if ((tid & 15) == 0) e.ssq_part[(size_t)(n0 / BN) * e.ssq_ld + row] = ss;
    } else if constexpr (EPI == EPI_RELU2) {
      const float4 r = make_float4(fmaxf(v.x, 0.f), fmaxf(v.y, 0.f), fmaxf(v.z, 0.f), fmaxf(v.w, 0.f));
      st_h4((half_t*)e.C + at, r.x * r.x, r.y * r.y, r.z * r.z, r.w * r.w);
      if (e.C2) st_h4((half_t*)e.C2 + (size_t)row * e.ldc2 + col, v.x, v.y, v.z, v.w);
    } else if constexpr (EPI == EPI_RELU2_BWD) {
      const float4 h = p0[u];
      st_h4((half_t*)e.C + at, v.x * 2.f * fmaxf(h.x, 0.f), v.y * 2.f * fmaxf(h.y, 0.f), v.z * 2.f * fmaxf(h.z, 0.f),
            v.w * 2.f * fmaxf(h.w, 0.f));
    } else if constexpr (EPI == EPI_SWIGLU_BWD) {
      auto d1 = [](float dg, float h1, float h3) {
        const float sg = sigmoid_f(h1);
        return dg * h3 * (sg + h1 * sg * (1.f - sg));
      };
      const float4 h1 = p0[u], h3 = p1[u];
      half_t* d = (half_t*)e.C + (size_t)row * e.ldc + (col >> 5) * 64 + (col & 31);
      st_h4(d, d1(v.x, h1.x, h3.x), d1(v.y, h1.y, h3.y), d1(v.z, h1.z, h3.z), d1(v.w, h1.w, h3.w));
      st_h4(d + 32, v.x * h1.x * sigmoid_f(h1.x), v.y * h1.y * sigmoid_f(h1.y), v.z * h1.z * sigmoid_f(h1.z),
            v.w * h1.w * sigmoid_f(h1.w));
    } else if constexpr (EPI == EPI_SMEAR) {
      const float4 gt = make_float4(sigmoid_f(v.x), sigmoid_f(v.y), sigmoid_f(v.z), sigmoid_f(v.w));
      *reinterpret_cast<float4*>((float*)e.C + at) =
          make_float4(p0[u].x + alpha * gt.x * p1[u].x, p0[u].y + alpha * gt.y * p1[u].y,
                      p0[u].z + alpha * gt.z * p1[u].z, p0[u].w + alpha * gt.w * p1[u].w);
      if (e.C2) *reinterpret_cast<float4*>((float*)e.C2 + at) = gt;
    }
  }
}

}  // namespace gemm_detail
}  // namespace ane
