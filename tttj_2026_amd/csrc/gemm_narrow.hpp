// Narrow 32 x 32 GEMM tiles for grids that would leave most CUs idle, and their element-wise
// epilogue (device code and launches shared by gemm.hip and gemm_ragged.hip).
#pragma once

#include "common.hpp"
#include "gemm_tile.hpp"
#include "kernels.hpp"

namespace tt {

// Epilogue of 4 consecutive outputs n .. n + 3 of row m from their fp32 sums (the semantics of
// gemm_kernel's epilogue, element by element).
// G lanes (aligned) share a row and hold consecutive 4-column groups of it: with ep.part_out,
// they write the partial statistics slot of their 4 G columns, or, in a matrix whose width 4 G does not
// divide, pairs of lanes those of 8 columns (slots are of one width); with ep.ln_part, K is the row
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
        float2* const part = ep.part_out + (size_t)m * ep.ln_stride;
        if (ep.ldy % (4 * G) != 0) {
          const float2 st = slot_stats<2, 4>(f);
          if ((threadIdx.x & 1) == 0) part[n / 8] = st;
        } else {
          const float2 st = slot_stats<G, 4>(f);
          if ((threadIdx.x & (G - 1)) == 0) part[n / (4 * G)] = st;
        }
      }
    } else if (!keep) {
      hv = half4{(half)0.f, (half)0.f, (half)0.f, (half)0.f};
    }
    *(half4*)dst = hv;
  }
}

// Narrow-tile GEMM for grids that would leave most CUs idle (few tokens): 32 x 32 output tiles, so
// four times as many blocks as 64 x 64 tiles pull operands (each CU's streaming rate is set by the
// bytes it keeps in flight), with the K range dealt to the block's NW waves in 64-wide slices.  Each wave copies
// its slices (32 X rows and 32 W rows of 128 bytes) from global memory straight into its own part of LDS, two
// slices in flight, and accumulates one 32 x 32 MFMA tile from it; no wave reads another's copies, so there is no
// barrier before the NW partial tiles are summed in wave order (deterministic).  The epilogue runs 4 outputs per
// thread on the first 256 threads.  Copies read 8 rows x 128 bytes an instruction (18 cycles of the CU's address
// unit); fragments loaded straight into registers, 32 rows x 16 bytes twice, took 64, the bound of this kernel at
// long K.  Measured on MI355X, registers -> LDS: 512 x 768 x 256 4.7 -> 4.1 us, 512 x 256 x 1024 6.2 -> 4.6,
// 21 x 320 x 1280 8.9 -> 4.7, 128 x 1024 x 4096 17.0 -> 7.6, 396 x 768 x 3072 25.3 -> 12.2 (a launch by itself ~3.5).
// Long K uses 8 waves, so that a block keeps 128 KiB of operands in flight.
//
// RAG: N (for the QKV projection each of its three parts) and K are multiples of 8 only.  A part's last
// column tile is then partial: W rows past the part are clamped to its last one and their outputs not
// stored.  8-value chunks at or past K are replaced by zeros when they are read from LDS.
//
// STAGED: X or W is not 16-byte aligned.  The copies go through registers, by plain loads, which take any
// alignment; nothing is documented for the direct copies.
constexpr int kNarrow = 32;
constexpr int kNarrowSlice = 2 * kNarrow * kBK;  // halfs: X rows 0 .. 31, W rows 32 .. 63
constexpr size_t narrow_lds_bytes(int nw) { return (size_t)nw * 2 * kNarrowSlice * sizeof(half); }

template <int MODE, int NW, bool RAG, bool STAGED = false>
__global__ __launch_bounds__(64 * NW) void gemm_narrow_kernel(const half* __restrict__ X,
                                                              const half* __restrict__ W, int M,
                                                              int N, int K, unsigned first_block,
                                                              EpiArgs ep) {
  extern __shared__ __align__(16) half lds[];
  const int tiles_n = column_tiles<kNarrow, MODE, RAG>(N);
  const int block = (int)(first_block + blockIdx.x);
  const int tm = block / tiles_n, tn = block - tm * tiles_n;
  const int m0 = tm * kNarrow;
  int n0 = tn * kNarrow;
  [[maybe_unused]] int n_end = N;
  if constexpr (RAG && MODE == TT_EPI_QKV) {
    const int width = N / 3, per = tiles_n / 3, part = tn / per;
    n0 = part * width + (tn - part * per) * kNarrow;
    n_end = (part + 1) * width;
  }
  // wave index provably uniform: MFMAs ignore the lane mask, so a wave with fewer slices must branch
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 31, hi = lane >> 5;
  half* const ring = lds + wave * (2 * kNarrowSlice);
  // Copy c fills rows 8 c .. 8 c + 7 of the slice: lane l row 8 c + l / 8, physical chunk l % 8, which holds
  // logical chunk (l % 8) ^ bits 1-3 of the row (the layout of gemm_kernel's direct copies).
  const int lrow = lane >> 3;
  const half* src[8];
  int col[2];  // the lane's first column in a slice, for even and odd copies
#pragma unroll
  for (int c = 0; c < 2; ++c) col[c] = 8 * ((lane & 7) ^ ((c << 2) | (lrow >> 1)));
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const int row = 8 * (c & 3) + lrow;
    src[c] = c < 4 ? X + (size_t)min(m0 + row, M - 1) * K
                   : W + (size_t)(RAG ? min(n0 + row, n_end - 1) : n0 + row) * K;
  }
  auto copy = [&](int s, int slot) {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int k = s * kBK + col[c & 1];
      const half* p = src[c] + (RAG && k >= K ? 0 : k);
      half* dst = ring + slot * kNarrowSlice + c * 512;
      if constexpr (STAGED) *(u32x4*)(dst + 8 * lane) = *(const u32x4_any*)p;
      else lds_copy16(p, dst);
    }
  };
  // slices wave, wave + NW, ...
  const int all = RAG ? (K + kBK - 1) / kBK : K / kBK;
  const int mine = (all - wave + NW - 1) / NW;
  // epilogue mapping (below): thread -> row ml, 4 columns nl; 8 aligned threads per row
  const int et = threadIdx.x & 255;
  const int ml = et >> 3, nl = 4 * (et & 7);
  const LnPre pre = ln_pre4<MODE, 8>(ep, min(m0 + ml, M - 1),
                                     RAG ? min(n0 + nl, n_end - 4) : n0 + nl, K);
  floatx16 acc;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = 0.f;
  if (mine > 0) copy(wave, 0);
  if (mine > 1) copy(wave + NW, 1);
  for (int j = 0; j < mine; ++j) {
    const int s = wave + NW * j;
    if (j + 1 < mine) wait_vmcnt<8>();  // this slice's copies have landed (the next one's 8 may not have)
    else wait_vmcnt<0>();
    asm volatile("" ::: "memory");
    const half* st = ring + (j & 1) * kNarrowSlice;
    half8 a[4], b[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const int pc = ((2 * kk + hi) ^ ((r >> 1) & 7)) * 8;
      b[kk] = *(const half8*)(st + r * kBK + pc);
      a[kk] = *(const half8*)(st + (kNarrow + r) * kBK + pc);
      if constexpr (RAG) {
        const bool in = s * kBK + 16 * kk + 8 * hi < K;  // 8 values of one row, all inside K or none
        const u32x4 wa = __builtin_bit_cast(u32x4, a[kk]), wb = __builtin_bit_cast(u32x4, b[kk]);
        a[kk] = __builtin_bit_cast(half8, u32x4{in ? wa[0] : 0u, in ? wa[1] : 0u, in ? wa[2] : 0u, in ? wa[3] : 0u});
        b[kk] = __builtin_bit_cast(half8, u32x4{in ? wb[0] : 0u, in ? wb[1] : 0u, in ? wb[2] : 0u, in ? wb[3] : 0u});
      }
    }
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) acc = mfma32x32x16(a[kk], b[kk], acc);
    if (j + 2 < mine) {
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the slice has been read ...
      asm volatile("" ::: "memory");
      copy(s + 2 * NW, j & 1);             // ... and its place is free
    }
  }
  // acc[4g + e] = C[m0 + r][n0 + 8g + 4 (lane / 32) + e]
  // (a wave's partial tile takes the place of its own slices)
  auto part = [&](int w) { return reinterpret_cast<float*>(lds + w * (2 * kNarrowSlice)); };
  __builtin_amdgcn_s_waitcnt(0xC07F);
  asm volatile("" ::: "memory");
#pragma unroll
  for (int g = 0; g < 4; ++g)
    *(floatx4*)(part(wave) + r * kNarrow + 8 * g + 4 * hi) =
        floatx4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
  __syncthreads();
  if (threadIdx.x >= 256 || m0 + ml >= M) return;
  float sum[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float v = part(0)[ml * kNarrow + nl + e];
#pragma unroll
    for (int w = 1; w < NW; ++w) v += part(w)[ml * kNarrow + nl + e];
    sum[e] = v;
  }
  if (RAG && n0 + nl >= n_end) return;
  epilogue4<MODE, 8>(ep, m0 + ml, n0 + nl, sum, pre);
}

// 8 waves above K = 512 (more than the two slices per wave that 4 waves hold at once).
static bool narrow_long_k(int k) { return k > 512; }

template <int MODE, int NW, bool RAG, bool STAGED>
static int launch_narrow_waves(const half* x, const half* w, int m, int n, int k, const EpiArgs& ep,
                               hipStream_t stream) {
  static std::once_flag once;
  static hipError_t attr = hipSuccess;
  std::call_once(once, [] {
    attr = hipFuncSetAttribute((const void*)gemm_narrow_kernel<MODE, NW, RAG, STAGED>,
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)narrow_lds_bytes(NW));
  });
  if (attr != hipSuccess)
    return fail(TT_ERR_HIP, "hipFuncSetAttribute(gemm_narrow): %s", hipGetErrorString(attr));
  const long blocks = (long)((m + kNarrow - 1) / kNarrow) * column_tiles<kNarrow, MODE, RAG>(n);
  TT_REQUIRE(blocks < (1L << 31), "linear: grid too large");
  launch_in_parts(blocks, 64 * NW, [&](unsigned first, unsigned part) {
    hipLaunchKernelGGL((gemm_narrow_kernel<MODE, NW, RAG, STAGED>), dim3(part), dim3(64 * NW), narrow_lds_bytes(NW),
                       stream, x, w, m, n, k, first, ep);
  });
  return launch_status("gemm_narrow_kernel");
}

template <int MODE, bool RAG, bool STAGED = false>
static int launch_narrow_mode(const half* x, const half* w, int m, int n, int k, const EpiArgs& ep,
                              hipStream_t stream) {
  return narrow_long_k(k) ? launch_narrow_waves<MODE, 8, RAG, STAGED>(x, w, m, n, k, ep, stream)
                          : launch_narrow_waves<MODE, 4, RAG, STAGED>(x, w, m, n, k, ep, stream);
}

}  // namespace tt
