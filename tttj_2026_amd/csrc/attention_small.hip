// Flash attention for head_dim 8 and 16 (the reference's D = 32 / 4-head and D = 128 / 16-head model
// shapes).
//
// block = (b, h, 128 queries), four independent waves of 32 queries (two 16-query column tiles), 64 keys
// per step.  At these widths a 32 x 32 MFMA would be mostly padding, so the 16-wide shapes are used:
//   S^T = K Q^T     v_mfma_f32_16x16x16_f16, 16 keys x 16 queries, K dim = head_dim (the lanes of the
//                   upper half are zero at head_dim 8); lane l holds query l % 16 and the 4 keys
//                   4 (l / 16) + j of each 16-key tile.
//   O^T += V^T P^T  v_mfma_f32_16x16x32_f16 over 32 keys: the B operand of lane l is its own 4 + 4
//                   probabilities of two key tiles, so the A operand takes V^T at those same keys and
//                   no value crosses lanes.
// Probabilities enter as p = hi + lo, two fp16 values in two MFMAs: 22 of fp32's 24 bits (hi is p cut to 11
// bits, lo the rest), scaled by 2^7 (in the exponent; it cancels in the division by the row sum) so that lo's
// fp16 granularity is 2^-31 of the largest p and hi still fits after the 2^8 growth the reference max allows;
// row sums add fp32 values.  The cut is below the rounding of exp2 and of the sums: where P V nearly cancels
// (values chosen so that the low bits of p are the result) the error against 64 bits is 3.1e-8 of sum p |v|
// (rms; 1.3e-7 at most), that of fp32 FMAs over single keys, which these MFMAs replaced, 3.4e-8 (1.7e-7).
// Infinite and NaN values of V, which the split cannot carry (0 inf is NaN), take a second pass with fp32
// MFMAs (v_mfma_f32_16x16x4_f32: exact products; in the place of the split they made the last shape below
// 81 -> 124 us).
// K and V^T fragments are read from global memory straight into registers, the next step's before this
// one's arithmetic (a head's K and V^T are 16-32 bytes per key and stay in the L1 / L2), so there is no
// LDS and no barrier.
// Bound by the softmax's vector work (exp, max, sum, the hi / lo split: ~12 issue slots a score; the
// MFMAs are a tenth of it).  Measured on MI355X against one query per lane with fp32 FMAs and K / V
// broadcast from LDS (bound by those LDS reads), per call: B 64, S 128, 16 heads of 8, causal 23.4 ->
// 11.6 us; B 64, S 1024 of the same 417 -> 209; B 4, S 2048, 16 heads of 16, non-causal 447 -> 88.
//
// Softmax in the exp2 domain (scale * log2(e) in Q already, or applied to the fp32 scores), against a
// reference max that moves only when a row's max grows by more than 2^8 over it.
// Masking as in attention_block.hpp: keys >= kv_end, keys > query (causal) and, for masks that
// are not right-padded prefixes, keys whose mask byte is 0 get no weight; padded query rows are
// written as +0.0.  Causal query tiles are dispatched heaviest first.
#include "attention_block.hpp"
#include "kernels.hpp"

namespace tt {

constexpr int kSmallBQ = 128;   // queries per block
constexpr int kSmallBKV = 64;   // keys per step
constexpr float kSmallExp = 7.f;  // log2 scale of the probabilities

__device__ __forceinline__ float quad_rows_max(float v) {  // max over lanes l, l ^ 16, l ^ 32, l ^ 48
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return xhalf_max(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
}

__device__ __forceinline__ float quad_rows_sum(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return xhalf_sum(__uint_as_float(r[0]) + __uint_as_float(r[1]));
}

template <int HD, bool CAUSAL>
__global__ __launch_bounds__(256) void attention_small_kernel(unsigned first_block,
                                                              const int32_t* __restrict__ info,
                                                              AttnArgs a) {
  constexpr float kLazy = 8.0f;  // log2 growth of the row max that moves the reference
  const int S = a.S, H = a.H;
  const int BH = a.B * H;
  const int nqt = (S + kSmallBQ - 1) / kSmallBQ;
  const int block = (int)(first_block + blockIdx.x);
  const int bh = block % BH;
  int qt = block / BH;
  if (CAUSAL) qt = nqt - 1 - qt;
  const int b = bh / H, h = bh - b * H;
  int kv_end = S;
  bool prefix = true;
  if (info != nullptr) {
    kv_end = info[b];
    prefix = info[a.B + b] != 0;
  } else if (a.mask != nullptr) {
    int count;
    block_mask_summary<4>(a.mask + (size_t)b * S, S, kv_end, count);
    prefix = count == kv_end;
  }
  const bool keymask = a.mask != nullptr && !prefix;
  const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
  const int qw = qt * kSmallBQ + 32 * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (qw >= S) return;
  const int ldv = round_up(S, 64);
  const half* __restrict__ Qbh = a.Q + (size_t)bh * S * HD;
  const half* __restrict__ Kbh = a.K + (size_t)bh * S * HD;
  const half* __restrict__ Vbh = a.Vt + (size_t)bh * HD * ldv;
  const uint8_t* __restrict__ mask = a.mask;
  const bool klane = 4 * g < HD;  // lanes that hold part of a head row (K and Q fragments)
  const half4 hzero = {(half)0.f, (half)0.f, (half)0.f, (half)0.f};
  // Queries at or past the last valid key are padded: no key step, zero output.
  const int wave_end = qw >= kv_end ? 0 : (CAUSAL ? min(kv_end, qw + 32) : kv_end);

  half4 qf[2];
  floatx4 o[2], sinit[2];
  float m_ref[2], l_run[2], thr[2];
  int lim[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int q = qw + 16 * t + col;
    qf[t] = hzero;
    if (klane && q < S) qf[t] = *(const half4*)(Qbh + (size_t)q * HD + 4 * g);
    o[t] = sinit[t] = floatx4{0.f, 0.f, 0.f, 0.f};
    m_ref[t] = -INFINITY;
    thr[t] = -INFINITY;
    l_run[t] = 0.f;
    lim[t] = CAUSAL ? min(kv_end, q + 1) : kv_end;
  }

  half4 kf[4], kn[4];
  half8 vf[2], vn[2];
  int mcur = 0, mnext = 0;
  // Fragments of the step at t0: key row t0 + 16 i + col, elements 4 g .. (K rows past S are clamped,
  // their scores masked); V^T feature row col at keys t0 + 32 i + 4 g .. + 3 and 16 later (keys past S,
  // the padding of V^T, read as 0).
  auto load = [&](int t0, half4 (&kk)[4], half8 (&vv)[2], int& mb) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      kk[i] = hzero;
      if (klane) kk[i] = *(const half4*)(Kbh + (size_t)min(t0 + 16 * i + col, S - 1) * HD + 4 * g);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int key = t0 + 32 * i + 4 * g;
      half4 lo = hzero, hi = hzero;
      if (col < HD) {
        const half* v = Vbh + (size_t)col * ldv + key;
        lo = *(const half4*)v;
        hi = *(const half4*)(v + 16);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        vv[i][e] = lo[e];
        vv[i][4 + e] = hi[e];
      }
    }
    if (keymask) mb = mask[(size_t)b * S + min(t0 + lane, S - 1)];
  };
  if (wave_end > 0) load(0, kf, vf, mcur);
  for (int t0 = 0; t0 < wave_end; t0 += kSmallBKV) {
    // past the last step: reload the last one (keeps the loop body free of a branch around the loads)
    const int tn = t0 + kSmallBKV < wave_end ? t0 + kSmallBKV : t0;
    load(tn, kn, vn, mnext);
    floatx4 s[2][4];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        s[t][i] = __builtin_amdgcn_mfma_f32_16x16x16f16(kf[i], qf[t], sinit[t], 0, 0, 0);
    if (!a.q_prescaled) {  // raw scores: scale them in fp32 (sinit stays 0)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const float off = m_ref[t] == -INFINITY ? 0.f : m_ref[t] - kSmallExp;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) s[t][i][j] = fmaf(s[t][i][j], a.scale_log2, -off);
      }
    }
    if (t0 + kSmallBKV > kv_end || (CAUSAL && t0 + kSmallBKV - 1 > qw) || keymask) {
      // per lane 4 bits for each key tile: keys 16 i + 4 g + j below lim, and mask bytes
      uint64_t kbits = ~0ull;
      if (keymask) kbits = __ballot(mcur != 0 && t0 + lane < S);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int n = min(max(lim[t] - t0 - (16 * i + 4 * g), 0), 4);
          const uint32_t ok = ((1u << n) - 1u) & (uint32_t)(kbits >> (16 * i + 4 * g));
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (!((ok >> j) & 1u)) s[t][i][j] = -INFINITY;
        }
    }
    if (t0 + kSmallBKV > S) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (t0 + 32 * i + 4 * g + (e & 3) + 4 * (e & 4) >= S) vf[i][e] = (half)0.f;
    }
    float mt[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      float mx = s[t][0][0];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) mx = fmaxf(mx, s[t][i][j]);
      mt[t] = quad_rows_max(mx);
    }
    if (__builtin_amdgcn_ballot_w64(mt[0] > thr[0] || mt[1] > thr[1]) != 0) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        // the new reference is the true running max; a row with no valid key so far keeps -inf
        const float mc = m_ref[t] == -INFINITY ? 0.f : m_ref[t] - kSmallExp;  // what s is relative to
        const float m_new = fmaxf(m_ref[t], mt[t] + mc);
        const bool none = m_new == -INFINITY;
        const float corr = none ? 1.f : __builtin_amdgcn_exp2f(m_ref[t] - m_new);
        const float shift = none ? 0.f : m_new - kSmallExp - mc;
        m_ref[t] = m_new;
        thr[t] = none ? -INFINITY : kSmallExp + kLazy;
        l_run[t] *= corr;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          o[t][e] *= corr;
          sinit[t][e] = (none || !a.q_prescaled) ? 0.f : kSmallExp - m_new;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) s[t][i][j] -= shift;
      }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        half8 ph, pl;
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          const float p0 = __builtin_amdgcn_exp2f(s[t][2 * i + (e >> 2)][e & 3]);
          const float p1 = __builtin_amdgcn_exp2f(s[t][2 * i + (e >> 2)][(e & 3) + 1]);
          l_run[t] += p0;
          l_run[t] += p1;
          const half2v hi = __builtin_bit_cast(half2v, __builtin_amdgcn_cvt_pkrtz(p0, p1));
          ph[e] = hi[0];
          ph[e + 1] = hi[1];
          pl[e] = (half)(p0 - (float)hi[0]);
          pl[e + 1] = (half)(p1 - (float)hi[1]);
        }
        o[t] = mfma16x16x32(vf[i], ph, o[t]);
        o[t] = mfma16x16x32(vf[i], pl, o[t]);
      }
#pragma unroll
    for (int i = 0; i < 4; ++i) kf[i] = kn[i];
    vf[0] = vn[0];
    vf[1] = vn[1];
    mcur = mnext;
  }

  // An infinite or NaN value of V leaves no finite output in its feature, whatever the weight: 0 inf and
  // inf - inf (lo's sign is not hi's) are NaN.  Such a wave starts over with fp32 products, 16 keys at a
  // time, each key tile only for the query tiles that may attend it.
  bool odd = false;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) odd |= !(fabsf(o[t][e]) < INFINITY);
  if (__builtin_amdgcn_ballot_w64(odd) != 0) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      o[t] = floatx4{0.f, 0.f, 0.f, 0.f};
      l_run[t] = 0.f;
      float m = -INFINITY;
      const int end = CAUSAL ? min(kv_end, qw + 16 * t + 16) : kv_end;
#pragma unroll 1
      for (int k0 = 0; k0 < end; k0 += 16) {
        half4 kk = hzero, vv = hzero;
        if (klane) kk = *(const half4*)(Kbh + (size_t)min(k0 + col, S - 1) * HD + 4 * g);
        if (col < HD) vv = *(const half4*)(Vbh + (size_t)col * ldv + k0 + 4 * g);
        const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
        floatx4 s = __builtin_amdgcn_mfma_f32_16x16x16f16(kk, qf[t], zero, 0, 0, 0);
        float mx = -INFINITY;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int key = k0 + 4 * g + j;
          const bool ok = key < lim[t] && (!keymask || mask[(size_t)b * S + min(key, S - 1)] != 0);
          s[j] = ok ? (a.q_prescaled ? s[j] : s[j] * a.scale_log2) : -INFINITY;
          mx = fmaxf(mx, s[j]);
        }
        const float m_new = fmaxf(m, quad_rows_max(mx));
        const bool none = m_new == -INFINITY;  // no allowed key so far
        const float corr = none ? 1.f : __builtin_amdgcn_exp2f(m - m_new);
        m = m_new;
        floatx4 acc;
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = o[t][e] *= corr;
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float p = __builtin_amdgcn_exp2f(s[j] - (none ? 0.f : m_new));
          sum += p;
          const float v = k0 + 4 * g + j < S ? (float)vv[j] : 0.f;
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(v, p, acc, 0, 0, 0);
        }
        l_run[t] = l_run[t] * corr + sum;
        if (!(none && quad_rows_sum(sum) == 0.f)) o[t] = acc;  // (before the first allowed key: nothing)
      }
    }
  }

#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const float l = quad_rows_sum(l_run[t]);
    const int q = qw + 16 * t + col;
    if (q >= S || !klane) continue;
    size_t orow = (size_t)b * S + q;
    if (a.out_row != nullptr) {  // packed context: padded tokens have no row
      const int r = a.out_row[orow];
      if (r < 0) continue;
      orow = (size_t)r;
    }
    const bool qvalid = q < kv_end && (mask == nullptr || mask[(size_t)b * S + q] != 0);
    const float inv = (qvalid && l > 0.f) ? 1.0f / l : 0.f;
    half4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = qvalid ? (half)(o[t][e] * inv) : (half)0.f;
    *(half4*)(a.ctx + orow * ((size_t)H * HD) + (size_t)h * HD + 4 * g) = v;
  }
}

int launch_attention_small(const AttnArgs& args, const int32_t* info, int head_dim, int causal,
                           hipStream_t stream) {
  TT_REQUIRE(head_dim == 8 || head_dim == 16, "attention_small: head_dim %d not in {8, 16}",
             head_dim);
  const long blocks = (long)args.B * args.H * ((args.S + kSmallBQ - 1) / kSmallBQ);
  TT_REQUIRE(blocks < (1L << 31), "attention: grid too large");
#define TT_ATT_SMALL(HD, C)                                                                             \
  launch_in_parts(blocks, 256, [&](unsigned first, unsigned n) {                                        \
    hipLaunchKernelGGL((attention_small_kernel<HD, C>), dim3(n), dim3(256), 0, stream, first, info, args); \
  })
  if (head_dim == 8) {
    if (causal) TT_ATT_SMALL(8, true); else TT_ATT_SMALL(8, false);
  } else {
    if (causal) TT_ATT_SMALL(16, true); else TT_ATT_SMALL(16, false);
  }
#undef TT_ATT_SMALL
  return launch_status("attention_small_kernel");
}

}  // namespace tt
