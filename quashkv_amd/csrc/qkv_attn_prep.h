// Shared by the decode-attention and the search translation units: the
// integer-MFMA query operands (prepare_mfma) and the Walsh coefficients of a
// symmetric codebook.
#pragma once

#include <math.h>

#include "qkv_attn_dev.h"

namespace {

using namespace qkv_attn;


template <typename T>
T* at(void* base, int64_t off) {
  return reinterpret_cast<T*>(static_cast<char*>(base) + off);
}

// Query operands for the score MFMA.  One workgroup per (b, kv head, chunk of
// 4 rows).  Row bit p of a K row (plane-major, D bits per plane) has weight W_p:
//   MSE plane r, coordinate j:  2 kg[r] q~_j
//   QJL plane,   coordinate j:  2 alpha |q~_j| S_j
// (mixed-precision rows: per-slot coefficients, see Tables).  The operand
// holds Z_p = round(W_p 2^Fq / 2^i), negated for i = 7 (a set bit masks to
// the byte value -128), where i = p % 8 is the bit's place in its byte, as
// signed base-256 digits; |Z| < 2^30.  Fq comes from the bound
// max |W| <= 2 max(kg, alpha) ||q|| (Pi is orthogonal), so no reduction over
// the rotated row stands between the rotation and the digits.
// Operand register layout: aq[(bhc * NU + u) * 64 + lane] (4 dwords), lane
// (m = 4 row + digit, g = lane / 16); byte beta of dword e <-> row bit
//   D = 128:  32 (g DPL + u / 2) + 8 beta + 4 (u % 2) + e   (NU = 2 DPL)
//   D = 64:   32 (2 u + g / 2) + 8 beta + 4 (g % 2) + e      (NU = NPL)
// i.e. the score kernel's lane group g reads row dwords g DPL .. (D = 128) or
// 2 u + g / 2 (D = 64) and masks nibble half u % 2 (D = 128) or g % 2.
// NPL planes per row: NPL - 1 MSE planes (odd bit subsets s, weight
// 2 kg[s] q~_j), then the QJL plane.  The decode rows have NPL = mbits + 1
// (mbits <= 2: the subsets are the single bits); the search index also uses
// NPL = 5 for 3-bit MSE codes (three bits and their parity).
// Thread (j, part) rotates coordinate j of all rows over one of 256 / D parts
// of k, then turns coordinate j of rows part, part + 256 / D, ... into digit
// bytes, scattered into an LDS image of the operands that is copied out whole.
template <int D, int NPL, bool FP4>
__global__ __launch_bounds__(256) void prepare_mfma(QLayers ql, int Bl, int q_dtype,
                                                    float alpha, int Hq, int Hkv, int Q, int R,
                                                    int chunks, Tables tb,
                                                    qkv_v4i* __restrict__ aq,
                                                    float* __restrict__ rowc,
                                                    float* __restrict__ qw) {
  constexpr int MB = NPL - 1;  // weighted MSE planes
  constexpr int KRB = NPL * D / 8;
  constexpr int DPL = KRB / 16;
  constexpr int NU = KRB / 8;        // score MFMAs per 16 tokens
  constexpr int NW = NU * 64 * 4;    // operand dwords per chunk
  constexpr int NPART = 256 / D;     // threads per coordinate
  constexpr int KP = D / NPART;      // k per thread in the rotation
  constexpr int RPT = kRowsM / NPART;  // rows per thread in the digit phase
  constexpr int WPP = D / 64;        // waves per part
  static_assert(D == 128 || D == 64, "64- or 128-dim rows");
  static_assert(D == 64 || KRB % 16 == 0, "128-dim rows split into 4 lane groups");
  static_assert(kRowsM == 4, "rows per chunk");
  static_assert(!FP4 || (D == 128 && NPL <= 3), "fp4 operands: the fused d = 128 decode");
  __shared__ float qs[kRowsM][D];
  __shared__ float part[NPART][kRowsM][D];
  __shared__ float nqs[kRowsM];
  __shared__ uint32_t stage[NW];
  __shared__ float red[4][RPT][3];  // [wave][row slot][sq, sw, fp4 halves]

  const int tid = threadIdx.x;
  const int G = Hq / Hkv;
  const int bhc = blockIdx.x;  // over the batch of all layers
  const int chunk = bhc % chunks;
  const int bh = bhc / chunks;
  const int hkv = bh % Hkv, bz = bh / Hkv;
  const int layer = bz / Bl, b = bz - layer * Bl;
  const void* __restrict__ q = ql.q[layer];
  const float* __restrict__ pi = ql.pi[layer];
  const float* __restrict__ signs = ql.signs[layer];
  const int r0 = chunk * kRowsM;
  const int nr = min(kRowsM, R - r0);
  // Pi staged in LDS by coalesced loads (rows padded by 4 floats: the
  // threads of a wave then read 16 rows' float4s conflict-free), then this
  // thread's part of row j from there
  extern __shared__ __align__(16) float4 pis[];  // [D][(D + 4) / 4]
  constexpr int PR4 = (D + 4) / 4;
  {
    const float4* src = reinterpret_cast<const float4*>(pi);
#pragma unroll
    for (int x = 0; x < D * D / 4 / 256; ++x) {
      const int i = tid + 256 * x, row = i / (D / 4), c4 = i - row * (D / 4);
      pis[row * PR4 + c4] = src[i];
    }
  }
  const int j = tid % D, half = tid / D;
  float qv[kRowsM * D / 256];
#pragma unroll
  for (int x = 0; x < kRowsM * D / 256; ++x) {
    const int i = tid + 256 * x;
    const int r = i / D, jj = i - r * D;
    float v = 0.f;
    if (r < nr) {
      const int row = r0 + r;
      const int g = row / Q, qi = row - g * Q;
      const int h = hkv * G + g;
      v = qkv_load(q, ((int64_t(b) * Hq + h) * Q + qi) * D + jj, q_dtype);
    }
    qv[x] = v;
  }
  const float sgn = signs[j];
#pragma unroll
  for (int x = 0; x < kRowsM * D / 256; ++x) {
    const int i = tid + 256 * x;
    qs[i / D][i % D] = qv[x];
  }
  __syncthreads();
  float4 prow[KP / 4];
#pragma unroll
  for (int k4 = 0; k4 < KP / 4; ++k4) prow[k4] = pis[j * PR4 + half * (KP / 4) + k4];
  {  // ||q_r||^2: wave w sums row w
    const int wave = tid >> 6, lane = tid & 63;
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < D / 64; ++c) {
      const float a = qs[wave][lane + 64 * c];
      ss = fmaf(a, a, ss);
    }
    ss = wave_sum_dpp(ss);
    if (lane == 0) nqs[wave] = ss;
  }
  {  // q~_j = sum_k q_k Pi[j][k], this thread's part of k for all rows
    float acc[kRowsM] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k4 = 0; k4 < KP / 4; ++k4) {
      const int k = half * KP + 4 * k4;
#pragma unroll
      for (int r = 0; r < kRowsM; ++r) {
        acc[r] = fmaf(qs[r][k], prow[k4].x, acc[r]);
        acc[r] = fmaf(qs[r][k + 1], prow[k4].y, acc[r]);
        acc[r] = fmaf(qs[r][k + 2], prow[k4].z, acc[r]);
        acc[r] = fmaf(qs[r][k + 3], prow[k4].w, acc[r]);
      }
    }
#pragma unroll
    for (int r = 0; r < kRowsM; ++r) part[half][r][j] = acc[r];
  }
  float kgmax = alpha;
#pragma unroll
  for (int r = 0; r < MB; ++r) kgmax = fmaxf(kgmax, fabsf(tb.kg[r]));
  __syncthreads();

  uint8_t* sb = reinterpret_cast<uint8_t*>(stage);
  // digit bytes of weight W at row bit p of row r
  auto put8 = [&](int p, float W, int fq, int r) {
    const int i = p & 7;
    int Z = static_cast<int>(rintf(ldexpf(W, fq - i)));
    if (i == 7) Z = -Z;
    const uint32_t dg = (static_cast<uint32_t>(Z) + 0x808080u) ^ 0x808080u;
    const int w32 = p >> 5, e = i & 3, beta = (p >> 3) & 3;
    int g, u;
    if constexpr (D == 128) {
      g = w32 / DPL;
      u = 2 * (w32 - g * DPL) + (i >> 2);
    } else {
      g = 2 * (w32 & 1) + (i >> 2);
      u = w32 >> 1;
    }
    const int base = ((u * 64 + 16 * g + 4 * r) * 4 + e) * 4 + beta;
#pragma unroll
    for (int v = 0; v < 4; ++v) sb[base + 16 * v] = static_cast<uint8_t>(dg >> (8 * v));
  };
  float csq[RPT], csw[RPT], chf[RPT];
#pragma unroll
  for (int rr = 0; rr < RPT; ++rr) {
    const int r = half + NPART * rr;
    float hf = 0.f;
    float v = 0.f;
#pragma unroll
    for (int pp = 0; pp < NPART; ++pp) v += part[pp][r][j];
    const float w = alpha * fabsf(v) * sgn;
    if (qw != nullptr && r < nr) {  // q~ and w for the VALU kernel, qw[b][hkv][row][2][D]
      float* dst = qw + (int64_t(bh) * R + r0 + r) * 2 * D;
      dst[j] = v;
      dst[D + j] = w;
    }
    const float wmax = 2.f * kgmax * sqrtf(nqs[r]);
    int ex = 0;
    if (wmax > 0.f) frexpf(wmax, &ex);  // wmax = f 2^ex, f in [0.5, 1)
    // int8 digits: the fixed-point exponent (|Z| < 2^30); fp4: the row's sigma
    const int fq = FP4 ? kf4_sigma(wmax) : wmax > 0.f ? 30 - ex : 0;
    // IP keys (the mixed-key formats run on decode_fused's own prologue)
    if constexpr (FP4) {
      csq[rr] = key_weights<MB>(tb, j, v, w, [&](int pb, float W) {
        hf += kf4_put<DPL, 4 * DPL, false>(sb, pb, W, fq, r);
      });
    } else {
      csq[rr] = v;
#pragma unroll
      for (int pl = 0; pl < MB; ++pl) put8(pl * D + j, 2.f * tb.kg[pl] * v, fq, r);
      put8(MB * D + j, 2.f * w, fq, r);
    }
    csw[rr] = w;
    chf[rr] = hf;
  }
  {  // row constants: sums over j (a wave holds 64 j of one part)
    const int wave = tid >> 6, lane = tid & 63;
#pragma unroll
    for (int rr = 0; rr < RPT; ++rr) {
      const float a = wave_sum_dpp(csq[rr]);
      const float c = wave_sum_dpp(csw[rr]);
      const float h = FP4 ? wave_sum_dpp(chf[rr]) : 0.f;
      if (lane == 0) {
        red[wave][rr][0] = a;
        red[wave][rr][1] = c;
        red[wave][rr][2] = h;
      }
    }
  }
  __syncthreads();
  uint32_t* aqw = reinterpret_cast<uint32_t*>(aq) + int64_t(bhc) * NW;
#pragma unroll
  for (int x = 0; x < NW / 256; ++x) aqw[tid + 256 * x] = stage[tid + 256 * x];
  if (tid < kRowsM) {  // row r = tid: part r % NPART (waves WPP h ..), slot r / NPART
    const int r = tid, h = r % NPART, rr = r / NPART;
    float sq = 0.f, sw = 0.f, sh = 0.f;
#pragma unroll
    for (int w = 0; w < WPP; ++w) {
      sq += red[WPP * h + w][rr][0];
      sw += red[WPP * h + w][rr][1];
      sh += red[WPP * h + w][rr][2];
    }
    const float wmax = 2.f * kgmax * sqrtf(nqs[r]);
    int ex = 0;
    if (wmax > 0.f) frexpf(wmax, &ex);
    const int fq = wmax > 0.f ? 30 - ex : 0;
    rowc[(int64_t(bhc) * kRowsM + r) * 2 + 0] = tb.kconst * sq - sw + sh;
    // fp4: the row's sigma (an integer, as a float); int8: 2^-Fq
    rowc[(int64_t(bhc) * kRowsM + r) * 2 + 1] =
        FP4 ? static_cast<float>(kf4_sigma(wmax)) : ldexpf(1.f, -fq);
  }
}

// Dynamic LDS of prepare_mfma<D, NPL> (the padded Pi), raising the kernel's
// limit past 64 KiB once where needed.
template <int D, int NPL, bool FP4>
uint32_t prep_lds() {
  constexpr uint32_t bytes = D * (D + 4) * 4;
  if constexpr (bytes > 65536) {
    static const bool raised = hipFuncSetAttribute(
        reinterpret_cast<const void*>(&prepare_mfma<D, NPL, FP4>),
        hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes)) == hipSuccess;
    (void)raised;
  }
  return bytes;
}

// Walsh coefficients of a codebook: c[code] = g_empty + sum_S g_S chi_S(code),
// chi_S(code) = prod_{k in S} (2 bit_k(code) - 1).  The plane decomposition
// used by the MFMA path needs a symmetric codebook (c[~code] == -c[code]),
// for which every even-size subset (g_empty included) has g_S = 0.
bool walsh_odd(const float* cent, int bits, float* g, float* gconst) {
  const int n = 1 << bits;
  for (int c = 0; c < n; ++c)
    if (cent[(n - 1) ^ c] != -cent[c]) return false;
  const int ns = n_odd_subsets(bits);
  double sum = 0.0;
  for (int s = 0; s < ns; ++s) {
    const uint32_t sub = odd_subset(bits, s);
    double acc = 0.0;
    for (int c = 0; c < n / 2; ++c) {  // pair code c with ~c: chi flips sign for odd S
      int par = 0;
      for (int k = 0; k < bits; ++k)
        if ((sub >> k) & 1u) par += ((c >> k) & 1) ? 0 : 1;  // count of (-1) factors
      const double chi = (par & 1) ? -1.0 : 1.0;
      acc += 2.0 * static_cast<double>(cent[c]) * chi;
    }
    g[s] = static_cast<float>(acc / n);
    sum += acc / n;
  }
  // reconstruction check
  for (int c = 0; c < n; ++c) {
    double v = 0.0;
    for (int s = 0; s < ns; ++s) {
      const uint32_t sub = odd_subset(bits, s);
      double chi = 1.0;
      for (int k = 0; k < bits; ++k)
        if ((sub >> k) & 1u) chi *= ((c >> k) & 1) ? 1.0 : -1.0;
      v += static_cast<double>(g[s]) * chi;
    }
    if (fabs(v - cent[c]) > 1e-6 * (fabs(static_cast<double>(cent[c])) + 1e-6)) return false;
  }
  *gconst = static_cast<float>(-sum);
  return true;
}

}  // namespace
