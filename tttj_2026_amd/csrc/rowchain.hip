// Row-chain kernel for narrow models (d_model 32 ... 192): everything of a layer between two attentions in
// one launch.
//
// For R = 16 RT rows (tokens) of the residual stream one 512-thread block runs, with every intermediate in
// LDS,
//   [out_proj + residual, LN2, ffn_in + GELU, ffn_out + residual + block mask]   (MID)
//   then LN1 of the next layer and its QKV projection (head-major Q / K, transposed V), or the final norm,
// so a layer is two launches (attention, row chain) instead of seven, and of the activations only the
// residual stream, Q / K / V^T and the attention context travel through memory.  The values rounded to
// fp16 on the way are those of the layer-wise kernels (every op boundary), all sums are fp32.
//
// What bounds it is latency: a block is a chain of five short GEMMs and two LayerNorms.  So
//   * each of the eight waves owns 16-feature tiles (v_mfma_f32_16x16x32_f16, weights as the A operand)
//     over all R rows: the shortest MFMA chain per wave, and its B fragments (the activations, from LDS rows
//     padded by 16 bytes) are read once per GEMM and kept in registers for all of the wave's tiles;
//   * weights go from global memory (L2) straight into registers, requested at the start of the block or
//     at least one GEMM before their use; biases, gains and the like are copied to LDS at the start;
//   * the barriers wait for LDS only, not for loads in flight (lds_barrier).
// Weights are read from their fragment-order copies (launch_pack_fragments): a wave's load is 1 KiB contiguous.
// Read from the row-major matrices, 16 rows x 64 bytes per instruction, a load holds the address unit for 64
// cycles: 196 KB (all weights of D = F = 128) take 12800 cycles instead of 4300 per CU, and a 32-row tile at
// D = F = 128 took 21800 cycles, with its Q / K / V^T stored from the accumulators, instead of 15800.  Where a
// block walks several tiles (KEEP) it reads them once.
// Cycles of one 32-row tile at D = F = 128 (14600): rows and weights arriving 3700, out_proj 2400, LN2 1200, FFN
// 2600, ffn_out and its epilogue 900, LN1 1100, QKV 2300, stores 500.  64-row tiles are bound by the vector
// work of the epilogues (GELU, conversions, LayerNorm) and the fragment reads; with the weights kept they spill
// registers (15 at D 96, 51 at D 128).
// For the V part of the QKV projection the operands change places, so that a lane ends with 4 consecutive
// tokens of one feature: pieces of V^T rows without a transposing pass.
#include "common.hpp"
#include "kernels.hpp"

#include <algorithm>
#include <climits>
#include <mutex>
#include <type_traits>

namespace tt {

constexpr int kChainFC = 128;  // hidden columns per chunk: 16 per wave
constexpr int kChainThreads = 512;

// LDS: residual stream and LayerNorm output [R][D + 8], two hidden chunks [R][136], and the fp16 vectors
// bo, norm2 gain / bias, b2, norm1 gain / bias (or the final norm's), bqkv, b1.
constexpr size_t chain_hidden_halfs(int D, int rt) {  // or V^T [D][R + 8]
  return std::max((size_t)(16 * rt) * 2 * (kChainFC + 8), (size_t)D * (16 * rt + 8));
}
constexpr size_t chain_lds_bytes(int D, int rt, int F) {
  return ((size_t)(16 * rt) * 2 * (D + 8) + chain_hidden_halfs(D, rt) + 9 * D + F) * sizeof(half);
}

// KEEP (D, F <= 128): a wave's share of the weights fits its registers, and the block walks several row tiles
// with them.  Otherwise a block has one tile.
template <int D, int RT, bool MID, bool KEEP>
__global__ __launch_bounds__(kChainThreads, 2) void rowchain_kernel(ChainArgs a) {
  constexpr int R = 16 * RT;
  constexpr int KD = D / 32;              // k-steps of a K = D GEMM
  constexpr int KF = kChainFC / 32;
  constexpr int TN = D / 16;              // 16-feature tiles of a D-wide output
  constexpr int TPW = (TN + 7) / 8;       // of them per wave, at most
  constexpr int QPW = (3 * TN + 7) / 8;   // tiles of the QKV projection per wave
  constexpr int QPRE = QPW < 3 ? QPW : (KD <= 4 ? 3 : 2);  // of them requested ahead
  constexpr int LD = D + 8, LH = kChainFC + 8, LV = R + 8;
  constexpr int CH = D / 8;               // 16-byte chunks per row
  constexpr int G = CH <= 8 ? 8 : (CH <= 16 ? 16 : 32);  // lanes per row in the LayerNorms
  constexpr int NT = kChainThreads;
  extern __shared__ __align__(16) half lds[];
  half* const sx = lds;                   // residual stream [R][LD]
  half* const sn = sx + R * LD;           // LayerNorm output / attention context [R][LD]
  half* const sh0 = sn + R * LD;          // two hidden chunks [R][LH]
  half* const sv = sh0 + chain_hidden_halfs(D, RT);  // vectors
  half *const v_bo = sv, *const v_g2 = sv + D, *const v_t2 = sv + 2 * D, *const v_b2 = sv + 3 * D,
             *const v_g1 = sv + 4 * D, *const v_t1 = sv + 5 * D, *const v_qkv = sv + 6 * D,
             *const v_b1 = sv + 9 * D;
  __shared__ int s_qoff[R], s_voff[R];    // token -> offsets in the Q / K planes and V^T
  __shared__ __align__(8) uint8_t s_ok[R];  // valid token
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, g4 = lane >> 4;
  const int T = a.T, S = a.S;
  const bool last = MID && a.y != nullptr;
  const int nblocks = (int)gridDim.x - (MID ? 0 : a.info_blocks);  // blocks with row tiles
  if (!MID && (int)blockIdx.x >= nblocks) {
    // One block per sequence behind them: the mask summary the attention launches read (as
    // mask_info_kernel), beside the row tiles instead of in a launch of its own.
    const int b = blockIdx.x - nblocks;
    int end, count;
    block_mask_summary<kChainThreads / 64>(a.valid + (size_t)b * S, S, end, count);
    if (tid == 0) {
      a.info[b] = end;
      a.info[a.info_blocks + b] = count == end;
    }
    return;
  }

  // Loads the first GEMM waits for come first: the rows, then its weights, then the rest.
  constexpr int XL = (R * CH + NT - 1) / NT;
  const int ntiles = (T + R - 1) / R;
  u32x4 gx[XL], gc[MID ? XL : 1];
  auto load_rows = [&](int tile) {  // clamped: rows past T re-read the last one
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int e = min(tid + NT * i, R * CH - 1), r = e / CH, c = e - r * CH;
      const size_t o = (size_t)min(tile * R + r, T - 1) * D + 8 * c;
      if (MID) gc[i] = *(const u32x4*)(a.ctx + o);
      gx[i] = *(const u32x4*)(a.x + o);
    }
  };
  // Tile of this block in a round of gridDim.x tiles: shifted by 5 per round, so that with sequences of a
  // power-of-two number of tiles a block does not meet the same (live or padded) position every time.
  // Past the last tile: INT_MAX (later rounds lie past it too).
  auto tile_of = [&](int round) {
    if (!KEEP) return INT_MAX;
    const int g = nblocks, t = round * g + (int)((blockIdx.x + 5u * round) % (unsigned)g);
    return t < ntiles ? t : INT_MAX;
  };
  load_rows(blockIdx.x);
  // A fragments of 16 weight rows (tile nt of a matrix of K columns), k-steps [k0, k0 + n).
  auto load_w = [&](const half* W, int K, int nt, int k0, half8* f, auto n) {
    const half* p = W + ((size_t)nt * (K / 32) + k0) * 512 + 8 * lane;
#pragma unroll
    for (int kk = 0; kk < decltype(n)::value; ++kk) f[kk] = *(const half8*)(p + 512 * kk);
  };
  constexpr std::integral_constant<int, KD> kd{};
  constexpr std::integral_constant<int, KF> kf{};
  const half* const Wqkv = a.fwn;
  const half* const Wo = a.fw + 3 * D * D;
  const half* const W1 = Wo + D * D;
  const half* const W2 = W1 + (size_t)a.F * D;
  half8 wo[MID ? TPW : 1][KD], w1[KD], w2[MID ? TPW : 1][KF], wq[QPRE][KD];
  auto load_out = [&] {
#pragma unroll
    for (int j = 0; j < TPW; ++j)
      if (wave + 8 * j < TN) load_w(Wo, D, wave + 8 * j, 0, wo[j], kd);
  };
  auto load_ffn = [&] {  // of the first hidden chunk
    if (16 * wave < a.F) load_w(W1, D, wave, 0, w1, kd);
    if (a.F >= kChainFC) {
#pragma unroll
      for (int j = 0; j < TPW; ++j)
        if (wave + 8 * j < TN) load_w(W2, a.F, wave + 8 * j, 0, w2[j], kf);
    }
  };
  auto load_qkv = [&] {
#pragma unroll
    for (int j = 0; j < QPRE; ++j)
      if (wave + 8 * j < 3 * TN) load_w(Wqkv, D, wave + 8 * j, 0, wq[j], kd);
  };
  if constexpr (MID) load_out();
  else load_qkv();
  static_assert(!KEEP || QPW <= QPRE, "every weight tile of the wave has its registers");
  // vectors: 16-byte chunk c of the list above
  const int nvec = (MID ? 9 * D + a.F : 9 * D) / 8;
  for (int c = tid; c < nvec; c += NT) {
    const int seg = min(c / CH, 6), in = c - seg * CH;
    const half* src;
    if (seg < 4) {  // bo, norm2, b2
      src = MID ? a.w + (seg == 0 ? a.off[5] : seg == 1 ? a.off[6] : seg == 2 ? a.off[7] : a.off[11])
                : nullptr;
    } else if (seg < 6) {
      src = seg == 4 ? (last ? a.fin_g : a.wn + a.off[0]) : (last ? a.fin_b : a.wn + a.off[1]);
    } else if (in < 3 * CH) {
      src = last ? nullptr : a.wn + a.off[3];
    } else {
      src = a.w + a.off[9] - 3 * D;  // in counts on from bqkv
    }
    if (src != nullptr) *(u32x4*)(sv + 8 * c) = *(const u32x4*)(src + 8 * in);
  }
  const size_t qplane = (size_t)T * D;
  const u32x4 zero = {0u, 0u, 0u, 0u};

  // B fragments: all R rows of an LDS tile, K columns [0, 32 n).
  auto load_x = [&](const half* t, int ld, half8 (*f)[RT], auto n) {
#pragma unroll
    for (int kk = 0; kk < decltype(n)::value; ++kk)
#pragma unroll
      for (int i = 0; i < RT; ++i) f[kk][i] = *(const half8*)(t + (16 * i + col) * ld + 32 * kk + 8 * g4);
  };
  // MFMA chains start from the bias of their output features.
  auto init_acc = [&](floatx4 (&acc)[RT], const half* bias) {
    const half4 b = *(const half4*)bias;
#pragma unroll
    for (int i = 0; i < RT; ++i) acc[i] = floatx4{(float)b[0], (float)b[1], (float)b[2], (float)b[3]};
  };
  // Selects of whole dwords (two halfs each), and the residual sum (branch rounded to fp16 first).
  auto pick = [](bool c, half4 x, half4 y) {
    const u32x2 p = __builtin_bit_cast(u32x2, x), q = __builtin_bit_cast(u32x2, y);
    return __builtin_bit_cast(half4, u32x2{c ? p[0] : q[0], c ? p[1] : q[1]});
  };
  auto to_half = [](floatx4 v) { return half4{(half)v[0], (half)v[1], (half)v[2], (half)v[3]}; };
  auto add_resid = [](half4 x, floatx4 v) {
    half4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (half)((float)x[e] + (float)(half)v[e]);
    return o;
  };
  const half4 hzero = {(half)0.f, (half)0.f, (half)0.f, (half)0.f};
  // LayerNorm of the R rows of sx (D values each, G lanes per row); padded rows give +0.0.
  auto layer_norm = [&](const half* gamma, const half* beta, auto&& store) {
    const int c = tid & (G - 1);
    const bool in = c < CH;
    half8 g, bt;
    if (in) {
      g = *(const half8*)(gamma + 8 * c);
      bt = *(const half8*)(beta + 8 * c);
    }
    constexpr int RPP = NT / G;  // rows per pass
#pragma unroll
    for (int p = 0; p < (R + RPP - 1) / RPP; ++p) {
      const int r = p * RPP + tid / G;
      if (R % RPP != 0 && r >= R) break;
      half8 v;
      float s = 0.f;
      if (in) {
        v = *(const half8*)(sx + r * LD + 8 * c);
#pragma unroll
        for (int e = 0; e < 8; ++e) s += (float)v[e];
      }
      const float mean = seg_sum<G>(s) * (1.f / D);
      float q = 0.f;
      if (in) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float t = (float)v[e] - mean;
          q += t * t;
        }
      }
      const float rstd = rsqrtf(seg_sum<G>(q) * (1.f / D) + 1e-5f);
      if (in) {
        const bool ok = s_ok[r] != 0;
        half8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (half)(((float)v[e] - mean) * rstd * (float)g[e] + (float)bt[e]);
        const u32x4 w = __builtin_bit_cast(u32x4, o);
        store(r, c, __builtin_bit_cast(half8, u32x4{ok ? w[0] : 0u, ok ? w[1] : 0u, ok ? w[2] : 0u,
                                                    ok ? w[3] : 0u}));
      }
    }
  };
  auto to_sn = [&](int r, int c, half8 o) { *(half8*)(sn + r * LD + 8 * c) = o; };
  bool have_w = false;  // KEEP: a live tile has loaded all weights

  for (int round = 0, tile = blockIdx.x; tile < ntiles; tile = tile_of(++round)) {
  const int r0 = tile * R;
  if (KEEP && round != 0) lds_barrier();  // the previous tile's LDS is no longer read
  int any = 0;
  if (tid < R) {
    const int t = r0 + tid, tc = min(t, T - 1);
    const int ok = t < T && (a.valid == nullptr || a.valid[tc] != 0);
    const int b = tc / S, s = tc - b * S;
    s_qoff[tid] = (b * a.H * S + s) * a.hd;
    s_voff[tid] = b * D * a.ldv + s;
    s_ok[tid] = ok;
    any = ok;
  }
  if (a.valid != nullptr && !__syncthreads_or(any)) {
    // Only padded rows: Q / K / V^T get +0.0 once (the later layers keep it), the output +0.0.
    if (!MID) {
      for (int e = tid; e < R * D; e += NT) {
        const int r = e / D, n = e - r * D, hh = n >> a.hd_log2, d = n & (a.hd - 1);
        if (r0 + r >= T) break;
        const size_t o = (size_t)s_qoff[r] + (size_t)hh * S * a.hd + d;
        a.q[o] = (half)0.f;
        a.q[qplane + o] = (half)0.f;
        a.q[2 * qplane + (size_t)s_voff[r] + (size_t)n * a.ldv] = (half)0.f;
      }
    }
    if (MID && a.hid != nullptr)
      for (int e = tid; e < R * (a.F / 8); e += NT) {
        const int r = e / (a.F / 8);
        if (r0 + r < T) *(u32x4*)(a.hid + (size_t)r0 * a.F + 8 * (size_t)e) = zero;
      }
    if (last)
      for (int e = tid; e < R * CH; e += NT)
        if (r0 + e / CH < T) *(u32x4*)(a.y + (size_t)r0 * D + 8 * (size_t)e) = zero;
    if (!KEEP) return;
    if (tile_of(round + 1) < ntiles) load_rows(tile_of(round + 1));
    continue;
  }
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int e = tid + NT * i, r = e / CH, c = e - r * CH;
    if (R * CH % NT == 0 || e < R * CH) {
      if (MID) *(u32x4*)(sn + r * LD + 8 * c) = gc[i];
      *(u32x4*)(sx + r * LD + 8 * c) = gx[i];
    }
  }
  if (KEEP && tile_of(round + 1) < ntiles) load_rows(tile_of(round + 1));
  if constexpr (MID) {
    if (!have_w) load_ffn();
  }
  lds_barrier();

  bool ok_row[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) ok_row[i] = s_ok[16 * i + col] != 0;
  half8 xf[KD][RT];
  if constexpr (MID) {
    // out_proj: x += valid ? ctx Wo^T + bo : 0
    load_x(sn, LD, xf, kd);
#pragma unroll
    for (int j = 0; j < TPW; ++j) {
      if (wave + 8 * j < TN) {
        floatx4 acc[RT];
        const int n = 16 * (wave + 8 * j) + 4 * g4;
        init_acc(acc, v_bo + n);
#pragma unroll
        for (int kk = 0; kk < KD; ++kk)
#pragma unroll
          for (int i = 0; i < RT; ++i) acc[i] = mfma16x16x32(wo[j][kk], xf[kk][i], acc[i]);
#pragma unroll
        for (int i = 0; i < RT; ++i) {
          half4* px = (half4*)(sx + (16 * i + col) * LD + n);
          const half4 x = *px;
          *px = pick(ok_row[i], add_resid(x, acc[i]), x);
        }
      }
    }
    if (!last && !have_w) load_qkv();  // land during LN2 and the FFN
    lds_barrier();
    layer_norm(v_g2, v_t2, to_sn);
    lds_barrier();
    load_x(sn, LD, xf, kd);
    floatx4 acc2[TPW][RT];
#pragma unroll
    for (int j = 0; j < TPW; ++j)
      if (wave + 8 * j < TN) init_acc(acc2[j], v_b2 + 16 * (wave + 8 * j) + 4 * g4);
    for (int fc = 0; fc < a.F; fc += kChainFC) {
      half* const sh = sh0 + ((fc / kChainFC) & 1) * (R * LH);
      const int n0 = fc + 16 * wave;
      if (n0 < a.F) {
        floatx4 acc[RT];
        init_acc(acc, v_b1 + n0 + 4 * g4);
#pragma unroll
        for (int kk = 0; kk < KD; ++kk)
#pragma unroll
          for (int i = 0; i < RT; ++i) acc[i] = mfma16x16x32(w1[kk], xf[kk][i], acc[i]);
        if (!KEEP && n0 + kChainFC < a.F) load_w(W1, D, (n0 + kChainFC) / 16, 0, w1, kd);  // the next chunk's
#pragma unroll
        for (int i = 0; i < RT; ++i) {
          half4 h;
#pragma unroll
          for (int e = 0; e < 4; ++e) h[e] = (half)gelu_erf(acc[i][e]);
          *(half4*)(sh + (16 * i + col) * LH + 16 * wave + 4 * g4) = pick(ok_row[i], h, hzero);
        }
      }
      lds_barrier();
      const int kc = a.F - fc;
      if (a.hid != nullptr) {
        const int hc = min(kc, kChainFC) / 8;  // 16-byte chunks per row
        for (int e = tid; e < R * (kChainFC / 8); e += NT) {
          const int r = e / (kChainFC / 8), c = e % (kChainFC / 8);
          if (c < hc && r0 + r < T)
            *(u32x4*)(a.hid + (size_t)(r0 + r) * a.F + fc + 8 * c) = *(const u32x4*)(sh + r * LH + 8 * c);
        }
      }
      if (kc >= kChainFC) {
        half8 hx[KF][RT];
        load_x(sh, LH, hx, kf);
#pragma unroll
        for (int j = 0; j < TPW; ++j)
          if (wave + 8 * j < TN) {
#pragma unroll
            for (int kk = 0; kk < KF; ++kk)
#pragma unroll
              for (int i = 0; i < RT; ++i) acc2[j][i] = mfma16x16x32(w2[j][kk], hx[kk][i], acc2[j][i]);
            if (!KEEP && kc >= 2 * kChainFC) load_w(W2, a.F, wave + 8 * j, (fc + kChainFC) / 32, w2[j], kf);
          }
      } else {  // the last, partial chunk (a multiple of 32)
        for (int k0 = 0; k0 < kc; k0 += 32) {
          half8 hx[1][RT], wt[1];
          load_x(sh + k0, LH, hx, std::integral_constant<int, 1>{});
#pragma unroll
          for (int j = 0; j < TPW; ++j)
            if (wave + 8 * j < TN) {
              load_w(W2, a.F, wave + 8 * j, (fc + k0) / 32, wt, std::integral_constant<int, 1>{});
#pragma unroll
              for (int i = 0; i < RT; ++i) acc2[j][i] = mfma16x16x32(wt[0], hx[0][i], acc2[j][i]);
            }
        }
      }
      if (KEEP) break;
    }
    // ffn_out: x = valid ? x + h W2^T + b2 : 0
#pragma unroll
    for (int j = 0; j < TPW; ++j) {
      if (wave + 8 * j < TN) {
        const int n = 16 * (wave + 8 * j) + 4 * g4;
#pragma unroll
        for (int i = 0; i < RT; ++i) {
          half4* px = (half4*)(sx + (16 * i + col) * LD + n);
          *px = pick(ok_row[i], add_resid(*px, acc2[j][i]), hzero);
        }
      }
    }
    lds_barrier();
    if (last) {
      layer_norm(v_g1, v_t1, [&](int r, int c, half8 o) {
        if (r0 + r < T) *(half8*)(a.y + (size_t)(r0 + r) * D + 8 * c) = o;
      });
      if (!KEEP) return;
      have_w = true;
      continue;
    }
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int e = tid + NT * i, r = e / CH, c = e - r * CH;
      if (e < R * CH && r0 + r < T)
        *(u32x4*)(a.xa + (size_t)(r0 + r) * D + 8 * c) = *(const u32x4*)(sx + r * LD + 8 * c);
    }
  }

  // LN1 and the QKV projection of the next layer.
  layer_norm(v_g1, v_t1, to_sn);
  lds_barrier();
  load_x(sn, LD, xf, kd);
  lds_barrier();  // sx, sn and the hidden chunks now stage Q, K [R][LD] and V^T [D][LV]
#pragma unroll
  for (int j = 0; j < QPW; ++j) {
    const int ct = wave + 8 * j;
    if (ct >= 3 * TN) break;
    const int which = ct / TN;
    const int nn0 = 16 * (ct - which * TN);
    half8 (&wt)[KD] = wq[j % QPRE];
    floatx4 acc[RT];
    const int nn = nn0 + (which < 2 ? 4 * g4 : col);  // this lane's (first) feature
    if (which < 2) {
      init_acc(acc, v_qkv + which * D + nn);
#pragma unroll
      for (int kk = 0; kk < KD; ++kk)
#pragma unroll
        for (int i = 0; i < RT; ++i) acc[i] = mfma16x16x32(wt[kk], xf[kk][i], acc[i]);
    } else {
      const float bv = (float)v_qkv[2 * D + nn];
#pragma unroll
      for (int i = 0; i < RT; ++i) acc[i] = floatx4{bv, bv, bv, bv};
#pragma unroll
      for (int kk = 0; kk < KD; ++kk)
#pragma unroll
        for (int i = 0; i < RT; ++i) acc[i] = mfma16x16x32(xf[kk][i], wt[kk], acc[i]);
    }
    if (j + QPRE < QPW && ct + 8 * QPRE < 3 * TN) load_w(Wqkv, D, ct + 8 * QPRE, 0, wt, kd);
    if (which < 2) {
      half* const st = (which == 0 ? sx : sn) + nn;
      const float qs = which == 0 ? a.q_scale : 1.f;
#pragma unroll
      for (int i = 0; i < RT; ++i)
        *(half4*)(st + (16 * i + col) * LD) = pick(ok_row[i], to_half(acc[i] * qs), hzero);
    } else {
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const int r = 16 * i + 4 * g4;  // 4 tokens from here
        const uint32_t ok4 = *(const uint32_t*)(s_ok + r) * 0xFFu;  // bytes 0 / 1 -> 0x00 / 0xFF
        const u32x2 o = __builtin_bit_cast(u32x2, to_half(acc[i]));
        *(u32x2*)(sh0 + nn * LV + r) = u32x2{o[0] & __builtin_amdgcn_perm(0u, ok4, 0x01010000u),
                                             o[1] & __builtin_amdgcn_perm(0u, ok4, 0x03030202u)};
      }
    }
  }
  have_w = true;
  lds_barrier();
  // Q and K: a head's rows of consecutive tokens are contiguous, so chunks go out head by head.
  {
    const int cl = a.hd_log2 - 3;  // log2 of the 16-byte chunks per head row
    for (int e = tid; e < R * CH; e += NT) {
      const int c = e & ((1 << cl) - 1), r = (e >> cl) & (R - 1), hh = e / (R << cl);
      if (r0 + r < T) {
        const size_t o = (size_t)s_qoff[r] + (size_t)hh * S * a.hd + 8 * c;
        const int n = (hh << a.hd_log2) + 8 * c;
        *(u32x4*)(a.q + o) = *(const u32x4*)(sx + r * LD + n);
        *(u32x4*)(a.q + qplane + o) = *(const u32x4*)(sn + r * LD + n);
      }
    }
  }
  if (S % 8 == 0) {  // 8 aligned rows are tokens of one sequence
    for (int e = tid; e < D * (R / 8); e += NT) {
      const int f = e / (R / 8), r = 8 * (e % (R / 8));
      if (r0 + r < T)
        *(u32x4*)(a.q + 2 * qplane + (size_t)f * a.ldv + s_voff[r]) = *(const u32x4*)(sh0 + f * LV + r);
    }
  } else {
    for (int e = tid; e < D * R; e += NT) {
      const int f = e / R, r = e % R;
      if (r0 + r < T) a.q[2 * qplane + (size_t)f * a.ldv + s_voff[r]] = sh0[f * LV + r];
    }
  }
  if (!KEEP) break;
  }  // tiles
}

template <int D, int RT, bool MID, bool KEEP>
static int run_chain(const ChainArgs& a, hipStream_t stream) {
  static std::once_flag once;
  static hipError_t attr = hipSuccess;
  std::call_once(once, [] {
    attr = hipFuncSetAttribute((const void*)rowchain_kernel<D, RT, MID, KEEP>,
                               hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)chain_lds_bytes(D, RT, kChainMaxF));
  });
  if (attr != hipSuccess)
    return fail(TT_ERR_HIP, "hipFuncSetAttribute(rowchain): %s", hipGetErrorString(attr));
  int blocks = (a.T + 16 * RT - 1) / (16 * RT);
  if (KEEP) blocks = std::min(blocks, device_cus());
  if (!MID) blocks += a.info_blocks;
  hipLaunchKernelGGL((rowchain_kernel<D, RT, MID, KEEP>), dim3(blocks), dim3(kChainThreads),
                     chain_lds_bytes(D, RT, MID ? a.F : 0), stream, a);
  return launch_status("rowchain_kernel");
}

template <int D, int RT, bool KEEP>
static int run_chain_mid(const ChainArgs& a, bool mid, hipStream_t stream) {
  return mid ? run_chain<D, RT, true, KEEP>(a, stream) : run_chain<D, RT, false, KEEP>(a, stream);
}

// 64-row tiles beyond 32 rows per CU.  Measured on MI355X, forwards of two layers, 32-row -> 64-row tiles: 1024 to
// 7680 tokens 7% (D 32) to 44% (D 128) slower; 16384 tokens D 32 31.7 -> 27.2 us, D 64 37.2 -> 29.8, D 96 51.0 ->
// 50.0, D 128 with F 512 68.3 -> 67.0; 65536 tokens D 32 81.3 -> 64.9, D 64 97.4 -> 78.6 (F 256 92.1 -> 95.6),
// D 96 125.8 -> 118.7, D 128 with F 512 200.9 -> 186.4.  The line is wrong for the spilling form at D = F = 128:
// 16384 tokens 54.6 -> 57.8 us, 65536 125.8 -> 141.1.
template <int D>
static int run_chain_d(const ChainArgs& a, bool mid, hipStream_t stream) {
  const bool many = a.T > 32 * device_cus();
  if constexpr (D <= 128) {
    if (a.F <= kChainFC)
      return many ? run_chain_mid<D, 4, true>(a, mid, stream) : run_chain_mid<D, 2, true>(a, mid, stream);
  }
  if constexpr (D <= 128) {
    if (many) return run_chain_mid<D, 4, false>(a, mid, stream);
  }
  return run_chain_mid<D, 2, false>(a, mid, stream);
}

int launch_rowchain(const ChainArgs& a, int d_model, bool mid, hipStream_t stream) {
  TT_REQUIRE(a.F > 0 && a.F % 32 == 0 && a.F <= kChainMaxF && (a.hd & (a.hd - 1)) == 0 && (1 << a.hd_log2) == a.hd,
             "rowchain: bad ffn_dim %d or head_dim %d", a.F, a.hd);
  switch (d_model) {
    case 32: return run_chain_d<32>(a, mid, stream);
    case 64: return run_chain_d<64>(a, mid, stream);
    case 96: return run_chain_d<96>(a, mid, stream);
    case 128: return run_chain_d<128>(a, mid, stream);
    case 160: return run_chain_d<160>(a, mid, stream);
    case 192: return run_chain_d<192>(a, mid, stream);
    default: return fail(TT_ERR_INVALID, "rowchain: d_model %d", d_model);
  }
}

int64_t chain_fragment_halfs(int64_t D, int64_t F) {
  if (D % 32 != 0 || D > kChainMaxD || F % 32 != 0 || F > kChainMaxF) return 0;
  return 4 * D * D + 2 * F * D;
}

// Thread = 8 consecutive halfs of the fragment order.
__global__ __launch_bounds__(256) void pack_fragments_kernel(const half* __restrict__ w, int64_t stride,
                                                             int64_t o_qkv, int64_t o_out, int64_t o_in,
                                                             int64_t o_ffn, half* __restrict__ frag, int D,
                                                             int F) {
  const int64_t per = 4 * (int64_t)D * D + 2 * (int64_t)F * D;
  int64_t e = 8 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
  if (e >= per) return;
  const half* wl = w + blockIdx.y * stride;
  half* dst = frag + blockIdx.y * per + e;
  const int64_t n_qkv = 3 * (int64_t)D * D, n_out = (int64_t)D * D, n_in = (int64_t)F * D;
  const half* src;
  int K = D;
  if (e < n_qkv) {
    src = wl + o_qkv;
  } else if ((e -= n_qkv) < n_out) {
    src = wl + o_out;
  } else if ((e -= n_out) < n_in) {
    src = wl + o_in;
  } else {
    e -= n_in;
    src = wl + o_ffn;
    K = F;
  }
  const int tile = (int)(e / 512), lane = (int)(e % 512) / 8;
  const int nt = tile / (K / 32), kk = tile % (K / 32);
  *(half8*)dst = *(const half8*)(src + (size_t)(16 * nt + (lane & 15)) * K + 32 * kk + 8 * (lane >> 4));
}

int launch_pack_fragments(const half* w, int64_t stride, const int64_t* off, half* frag, int D, int F, int L,
                          hipStream_t stream) {
  const int64_t per = chain_fragment_halfs(D, F);
  if (per == 0) return TT_OK;
  hipLaunchKernelGGL(pack_fragments_kernel, dim3((unsigned)((per / 8 + 255) / 256), L), dim3(256), 0, stream,
                     w, stride, off[2], off[4], off[8], off[10], frag, D, F);
  return launch_status("pack_fragments_kernel");
}

}  // namespace tt
