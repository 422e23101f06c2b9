// Narrow 32 x 32 GEMM tiles for grids that would leave most CUs idle, and their element-wise
// epilogue (device code and launches shared by gemm.hip and gemm_ragged.hip).
#pragma once

#include "common.hpp"
#include "gemm_tile.hpp"
#include "kernels.hpp"

namespace tt {

// Epilogue of 4 consecutive outputs n .. n + 3 of row m from their fp32 sums (the semantics of
// gemm_kernel's epilogue, element by element), for the small-shape and narrow-tile kernels.
// G lanes (aligned) share a row and hold consecutive 4-column groups of it: with ep.part_out,
// they write the partial statistics slot of their 4 G columns; with ep.ln_part, K is the row
// length of the folded LayerNorm.
// Folded-LayerNorm inputs of one thread's 4 outputs, loaded before the GEMM's K loop so their
// latency overlaps it: the row's (mean, rstd) and the 4 columns' c and b'.
struct LnPre {
  float2 rs;
  floatx4 c, b;
};

template <int MODE, int G>
__device__ __forceinline__ LnPre ln_pre4(const EpiArgs& ep, int m, int n, int K) {
  LnPre p{};
  constexpr bool ZERO_MASKED = MODE == TT_EPI_BIAS || MODE == TT_EPI_BIAS_GELU || MODE == TT_EPI_QKV;
  if (ZERO_MASKED && ep.ln_part != nullptr) {
    p.rs = combine_row_stats_group<G>(ep.ln_part + (size_t)m * ep.ln_stride, ep.ln_slots, K);
    p.c = *(const floatx4*)(ep.ln_colsum + n);
    p.b = *(const floatx4*)(ep.ln_bias + n);
  }
  return p;
}

template <int MODE, int G>
__device__ __forceinline__ void epilogue4(const EpiArgs& ep, int m, int n, const float acc[4],
                                          const LnPre& pre) {
  const bool keep = ep.valid == nullptr || ep.valid[m] != 0;
  half4 hv;
  constexpr bool ZERO_MASKED = MODE == TT_EPI_BIAS || MODE == TT_EPI_BIAS_GELU || MODE == TT_EPI_QKV;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float v;
    if (ZERO_MASKED && ep.ln_part != nullptr)
      v = fmaf(pre.rs.y, fmaf(-pre.rs.x, pre.c[e], acc[e]), pre.b[e]);
    else
      v = acc[e] + (float)ep.bias[n + e];
    if constexpr (MODE == TT_EPI_BIAS_GELU) v = gelu_erf(v);
    if constexpr (MODE == TT_EPI_QKV) v *= n < ep.d_model ? ep.q_scale : 1.f;
    hv[e] = (half)v;
  }
  if constexpr (MODE == TT_EPI_QKV) {
    const int D = ep.d_model, hd = ep.head_dim, S = ep.seq;
    const size_t plane = (size_t)ep.batch * S * D;
    const int bb = m / S, sq = m - bb * S;
    if (!keep) hv = half4{(half)0.f, (half)0.f, (half)0.f, (half)0.f};
    const int which = n / D, nn = n - which * D;
    const int hh = nn / hd, d = nn - hh * hd;  // hd % 4 == 0: the 4 outputs share a head
    if (which < 2) {
      *(half4*)(ep.y + which * plane + (((size_t)bb * ep.heads + hh) * S + sq) * hd + d) = hv;
    } else {
      const size_t ldv = (size_t)(S + 63) / 64 * 64;
      half* vt = ep.y + 2 * plane + (((size_t)bb * ep.heads + hh) * hd + d) * ldv + sq;
#pragma unroll
      for (int e = 0; e < 4; ++e) vt[(size_t)e * ldv] = hv[e];
    }
  } else {
    half* dst = ep.y + (size_t)m * ep.ldy + n;
    if constexpr (MODE == TT_EPI_RESID_MASKED || MODE == TT_EPI_MASKED_RESID) {
      const half4 rv = *(const half4*)(ep.resid + (size_t)m * ep.ldy + n);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (MODE == TT_EPI_RESID_MASKED)
          hv[e] = keep ? (half)((float)rv[e] + (float)hv[e]) : rv[e];
        else
          hv[e] = keep ? (half)((float)rv[e] + (float)hv[e]) : (half)0.f;
      }
      if (ep.part_out != nullptr) {
        float f[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = (float)hv[e];
        const float2 st = slot_stats<G, 4>(f);
        if ((threadIdx.x & (G - 1)) == 0) ep.part_out[(size_t)m * ep.ln_stride + n / (4 * G)] = st;
      }
    } else if (!keep) {
      hv = half4{(half)0.f, (half)0.f, (half)0.f, (half)0.f};
    }
    *(half4*)dst = hv;
  }
}
// Narrow-tile GEMM for grids that would leave most CUs idle (few tokens): 32 x 32 output tiles, so
// four times as many blocks as 64 x 64 tiles pull operands (each CU's streaming rate is set by the
// bytes it keeps in flight), with the K range split over the block's NW waves.  Each wave loads
// its W and X fragments straight into registers (lane l: row l % 32, 8 K values at 8 (l / 32)),
// NPF K steps ahead, and accumulates one 32 x 32 MFMA tile; the NW partial tiles are summed in
// LDS in wave order (deterministic) and the epilogue runs 4 outputs per thread on the first 256
// threads.  Long K (few blocks, each streaming many bytes) uses 8 waves with 8 steps per buffer,
// so a block keeps 128 KiB of operands in flight.
constexpr int kNarrow = 32;
//
// RAG: N (for the QKV projection each of its three parts) and K are multiples of 8 only.  A part's last
// column tile is then partial: W rows past the part are clamped to its last one and their outputs not
// stored.  K is dealt to the waves in whole 16-wide steps; 8-value chunks at or past K read as zero.
template <int MODE, int NW, int NPF, bool RAG>
__global__ __launch_bounds__(64 * NW) void gemm_narrow_kernel(const half* __restrict__ X,
                                                              const half* __restrict__ W, int M,
                                                              int N, int K, EpiArgs ep) {
  const int tiles_n = column_tiles<kNarrow, MODE, RAG>(N);
  const int tm = blockIdx.x / tiles_n, tn = blockIdx.x - tm * tiles_n;
  const int m0 = tm * kNarrow;
  int n0 = tn * kNarrow;
  [[maybe_unused]] int n_end = N;
  if constexpr (RAG && MODE == TT_EPI_QKV) {
    const int width = N / 3, per = tiles_n / 3, part = tn / per;
    n0 = part * width + (tn - part * per) * kNarrow;
    n_end = (part + 1) * width;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 31, kh = 8 * (lane >> 5);
  const half* xr = X + (size_t)min(m0 + r, M - 1) * K + kh;
  const half* wr = W + (size_t)(RAG ? min(n0 + r, n_end - 1) : n0 + r) * K + kh;
  // K steps of this wave (K % (16 NW) == 0 unless RAG, whose last waves may have fewer or none)
  int steps = K / 16 / NW;
  int kbeg = wave * steps * 16;
  if constexpr (RAG) {
    // The step count differs between waves, and MFMAs ignore the lane mask: it is made provably
    // uniform so that a wave with fewer steps branches over them.
    const int all = (K + 15) / 16, per = (all + NW - 1) / NW;
    const int first = __builtin_amdgcn_readfirstlane(wave) * per;
    kbeg = first * 16;
    steps = max(0, min(per, all - first));
  }
  // epilogue mapping (below): thread -> row ml, 4 columns nl; 8 aligned threads per row
  const int et = threadIdx.x & 255;
  const int ml = et >> 3, nl = 4 * (et & 7);
  const LnPre pre = ln_pre4<MODE, 8>(ep, min(m0 + ml, M - 1),
                                     RAG ? min(n0 + nl, n_end - 4) : n0 + nl, K);
  floatx16 acc;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = 0.f;
  half8 a[2][NPF], b[2][NPF];
  auto load = [&](int buf, int s0) {
#pragma unroll
    for (int j = 0; j < NPF; ++j) {
      const int k = kbeg + 16 * min(s0 + j, steps - 1);  // past the end: reload the last step
      if constexpr (RAG) {
        const bool in = k >= 0 && k + kh < K;  // 8 values of one row, all inside K or none
        const half8 wv = *(const half8*)(in ? wr + k : wr - kh);
        const half8 xv = *(const half8*)(in ? xr + k : xr - kh);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          a[buf][j][e] = in ? wv[e] : (half)0.f;
          b[buf][j][e] = in ? xv[e] : (half)0.f;
        }
      } else {
        a[buf][j] = *(const half8*)(wr + k);
        b[buf][j] = *(const half8*)(xr + k);
      }
    }
  };
  auto mma = [&](int buf, int s0) {
#pragma unroll
    for (int j = 0; j < NPF; ++j)
      if (s0 + j < steps) acc = mfma32x32x16(a[buf][j], b[buf][j], acc);
  };
  // Two buffers, alternated by a loop unrolled twice (register arrays need compile-time indices).
  load(0, 0);
  for (int s0 = 0; s0 < steps; s0 += 2 * NPF) {
    if (s0 + NPF < steps) load(1, s0 + NPF);
    mma(0, s0);
    if (s0 + NPF >= steps) break;
    if (s0 + 2 * NPF < steps) load(0, s0 + 2 * NPF);
    mma(1, s0 + NPF);
  }
  // acc[4g + e] = C[m0 + r][n0 + 8g + 4 (lane / 32) + e]
  __shared__ __align__(16) float part[NW][kNarrow][kNarrow];
#pragma unroll
  for (int g = 0; g < 4; ++g)
    *(floatx4*)&part[wave][r][8 * g + 4 * (lane >> 5)] =
        floatx4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
  __syncthreads();
  if (threadIdx.x >= 256 || m0 + ml >= M) return;
  float sum[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float v = part[0][ml][nl + e];
#pragma unroll
    for (int w = 1; w < NW; ++w) v += part[w][ml][nl + e];
    sum[e] = v;
  }
  if (RAG && n0 + nl >= n_end) return;
  epilogue4<MODE, 8>(ep, m0 + ml, n0 + nl, sum, pre);
}

// Long K: 8 waves (more than two 4-step buffers per wave at 4 waves).
template <bool RAG>
static bool narrow_long_k(int k) { return (RAG || k % 128 == 0) && k / 64 > 8; }

template <int MODE, bool RAG>
static int launch_narrow_mode(const half* x, const half* w, int m, int n, int k, const EpiArgs& ep,
                              hipStream_t stream) {
  const long blocks = (long)((m + kNarrow - 1) / kNarrow) * column_tiles<kNarrow, MODE, RAG>(n);
  TT_REQUIRE(blocks < (1L << 31), "linear: grid too large");
  const dim3 grid((unsigned)blocks);
  if (narrow_long_k<RAG>(k))
    hipLaunchKernelGGL((gemm_narrow_kernel<MODE, 8, 8, RAG>), grid, dim3(512), 0, stream, x, w, m, n, k, ep);
  else
    hipLaunchKernelGGL((gemm_narrow_kernel<MODE, 4, 4, RAG>), grid, dim3(256), 0, stream, x, w, m, n, k, ep);
  return launch_status("gemm_narrow_kernel");
}

}  // namespace tt
