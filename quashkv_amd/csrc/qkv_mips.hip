// Maximum inner-product search over K rows (QuashIndex.search): a one-digit
// filter with rigorous bounds and exact scores of what passes it, or a full scan
// with streaming top-k; query operands from prepare_mfma.
#include <math.h>

#include <algorithm>
#include <climits>
#include <cmath>

#include "qkv_attn_prep.h"

namespace {


// ------------------------------------------------------------ MIPS search

// QuashIndex.search (quashkv/nn_search/index.py:121-163): for each query q and
// database vector x (K row + norm), score = n_x (<q~, c[code]> + alpha
// sum_j |q~_j| S_j (2 b_j - 1)), no 1/sqrt(d); then the k largest scores per
// query (descending; equal scores: lower index first).
//
// The scores are the decode kernel's integer MFMA dot products (same query
// operands from prepare_mfma), with the database row bits as the B operand.
// A workgroup (4 waves) takes 16 QC queries (QC chunks of 4 per wave) and a
// range of vectors; the 128 rows of each step are staged once in LDS and every
// wave expands them against its own query operands, held in registers.  Each
// wave keeps a sorted top-k list per query in LDS; a score enters only if it
// beats the list's k-th (a ballot finds the rare candidates).  Lists go to the
// workspace per (query, vector split) and mips_merge picks the final k.
constexpr int kMipsStep = 128;  // vectors staged per workgroup step (13.2 ms at cfg5; 64: 14.1)
constexpr int kMipsKMax = 256;

// Order-preserving float <-> uint32 map, for a device-wide running maximum
// (atomicMax on the image) of each query's k-th best score.
__device__ __forceinline__ uint32_t fkey(float f) {
  const uint32_t b = __float_as_uint(f);
  return (b & 0x80000000u) ? ~b : (b ^ 0x80000000u);
}
__device__ __forceinline__ float fkey_inv(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k ^ 0x80000000u) : ~k);
}

template <int MB, int PDW>
struct MipsCfg {
  static constexpr int NS = n_odd_subsets(MB);  // MSE planes of the virtual row
  static constexpr int NPL = NS + 1;            // + QJL plane
  static constexpr int RAWD = (MB + 1) * PDW;   // stored row dwords (PDW = d / 32)
  static constexpr int DPL = NPL;               // virtual dwords per lane group
  static constexpr int NU = 2 * DPL;            // MFMAs per 16 vectors and chunk
  static constexpr int QC = MB <= 2 ? 4 : 2;    // query chunks (of 4) per wave
};

// Rows of d < 128 (PDW = d / 32 dwords per plane) run as 128-wide rows whose
// missing plane words are zero, against queries padded with zeros.  Two
// workgroups per CU: the query operands (QC x NU x 4 registers), two groups'
// accumulators and the pipelined expansion need more than a third of the
// register file without spills.
template <int MB, int PDW>
__global__ __launch_bounds__(256, 2) void mips_scan(const qkv_v4i* __restrict__ aq,
                                                 const float* __restrict__ rowc, int M,
                                                 const uint8_t* __restrict__ kst,
                                                 const float* __restrict__ norms, int64_t N,
                                                 int nvc, int64_t vlen, int64_t n_items, int k,
                                                 float* __restrict__ cand_s,
                                                 int* __restrict__ cand_i,
                                                 uint32_t* __restrict__ gth,
                                                 const int* __restrict__ left) {
  using C = MipsCfg<MB, PDW>;
  constexpr int NU = C::NU, QC = C::QC, RAWD = C::RAWD;
  constexpr int QW = 4 * QC;                      // queries per wave
  constexpr int SD = kMipsStep * RAWD;            // row dwords per step
  constexpr int LPT = (SD + 255) / 256;           // row dwords each thread stages
  extern __shared__ __align__(16) float smem_ms[];
  uint32_t* rows = reinterpret_cast<uint32_t*>(smem_ms);           // [2][64][RAWD]
  float* nrm_s = smem_ms + 2 * kMipsStep * RAWD;                    // [2][kMipsStep]
  float* ls = nrm_s + 2 * kMipsStep;                                // [4][QW][k] scores
  int* li = reinterpret_cast<int*>(ls + 4 * QW * k);                // [4][QW][k] indices

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ln = lane & 15, lg = lane >> 4;
  const int nchunks = (M + 3) / 4;
  float* wls = ls + wave * QW * k;
  int* wli = li + wave * QW * k;
  const uint32_t* kw = reinterpret_cast<const uint32_t*>(kst);
  // this lane's virtual row dwords lg*DPL + x: up to three stored dwords
  // (offsets within a row) XORed, a zero mask where the plane word is absent
  // (d < 128) -- precomputed so the row loop has no divergent branches
  constexpr int NT = MB >= 3 ? 3 : 1;
  int voff[C::DPL][NT];
  uint32_t vmask[C::DPL][NT];
#pragma unroll
  for (int x = 0; x < C::DPL; ++x) {
    const int vv = lg * C::DPL + x, pv = vv >> 2, w = vv & 3;
    int t = 0;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      voff[x][j] = 0;
      vmask[x][j] = 0u;
    }
    if (w < PDW) {
      if (pv < C::NS) {
        const uint32_t sub = odd_subset(MB, pv);
        for (int r = 0; r < MB; ++r)
          if (((sub >> r) & 1u) && t < NT) {
            voff[x][t] = PDW * r + w;
            vmask[x][t] = 0xffffffffu;
            ++t;
          }
      } else {
        voff[x][0] = PDW * MB + w;
        vmask[x][0] = 0xffffffffu;
      }
    }
  }

  // items (query tile, vector chunk), vector-chunk major, so that a query's
  // later chunks start from the k-th best score its earlier chunks published
  // (gth); a workgroup takes items blockIdx.x, blockIdx.x + gridDim.x, ...
  // Behind the filter (left): only the query chunks it left, left[0] of them in
  // left[1 ..].
  int qtiles = static_cast<int>(n_items / nvc), nch = nchunks;
  if (left != nullptr) {
    nch = left[0];
    qtiles = (nch + 4 * QC - 1) / (4 * QC);
    n_items = int64_t(qtiles) * nvc;
  }
  for (int64_t item = blockIdx.x; item < n_items; item += gridDim.x) {
    const int vc = static_cast<int>(item / qtiles), qt = static_cast<int>(item % qtiles);
    // this wave's query chunks (nchunks: none)
    int chs[QC];
#pragma unroll
    for (int c = 0; c < QC; ++c) {
      const int i = (qt * 4 + __builtin_amdgcn_readfirstlane(wave)) * QC + c;
      chs[c] = i >= nch ? nchunks : left != nullptr ? left[1 + i] : i;
    }
    const int64_t v0 = int64_t(vc) * vlen;
    const int64_t v1 = min<int64_t>(N, v0 + vlen);

    qkv_v4i a[QC][NU];
    // theta: this chunk list's k-th score (a candidate must beat it);
    // tg: the query's device-wide bound (a candidate must reach it);
    // thr = max(the float above theta, tg): a candidate is a score >= thr
    float fq[QC], cr[QC], theta[QC], tg[QC], thr[QC];
#pragma unroll
    for (int c = 0; c < QC; ++c) {
      const int ch = min(chs[c], nchunks - 1);
#pragma unroll
      for (int u = 0; u < NU; ++u) a[c][u] = aq[(int64_t(ch) * NU + u) * 64 + lane];
      cr[c] = rowc[(int64_t(ch) * kRowsM + lg) * 2 + 0];
      fq[c] = rowc[(int64_t(ch) * kRowsM + lg) * 2 + 1];
      theta[c] = -INFINITY;
      const int qg = chs[c] * 4 + lg;
      tg[c] = qg < M ? fkey_inv(__hip_atomic_load(&gth[qg], __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT))
                     : INFINITY;
      thr[c] = fmaxf(-__FLT_MAX__, tg[c]);
    }
    for (int i = lane; i < QW * k; i += 64) {
      wls[i] = -INFINITY;
      wli[i] = -1;
    }

    // rows of step s0 staged through registers: loaded one step ahead
    uint32_t pre[LPT];
    float pn = 0.f;
    auto fetch = [&](int64_t s0) {
#pragma unroll
      for (int x = 0; x < LPT; ++x) {
        const int i = tid + 256 * x;
        const int64_t v = s0 + i / RAWD;
        pre[x] = (i < SD && v < v1) ? kw[v * RAWD + i % RAWD] : 0u;
      }
      // rows past the range score NaN, which no threshold test admits
      if (tid < kMipsStep) pn = s0 + tid < v1 ? norms[s0 + tid] : __builtin_nanf("");
    };
    auto stash = [&](int buf) {
#pragma unroll
      for (int x = 0; x < LPT; ++x)
        if (tid + 256 * x < SD) rows[buf * SD + tid + 256 * x] = pre[x];
      if (tid < kMipsStep) nrm_s[buf * kMipsStep + tid] = pn;
    };
    __syncthreads();  // the previous item's buffers are consumed
    fetch(v0);
    stash(0);
    __syncthreads();
    int buf = 0;
    for (int64_t s0 = v0; s0 < v1; s0 += kMipsStep) {
      const bool more = s0 + kMipsStep < v1;
      if (more) fetch(s0 + kMipsStep);  // in flight during this step
      const uint32_t* rb = rows + buf * kMipsStep * RAWD;
      const float* nb = nrm_s + buf * kMipsStep;
      // 16-vector groups, software-pipelined: group g + 1's row words are
      // expanded and its MFMAs issued before group g's scores and candidates,
      // so that the score arithmetic overlaps the matrix cores' work
      constexpr int NG = kMipsStep / 16;
      auto expand_mfma = [&](int g, qkv_v4i* acc) {
        // virtual row dwords lg*DPL .. : plane p < NS is the parity of the
        // code bits in odd subset p, plane NS the QJL plane
        uint32_t vd[C::DPL];
        const uint32_t* rv = rb + (g * 16 + ln) * RAWD;
#pragma unroll
        for (int x = 0; x < C::DPL; ++x) {
          uint32_t val = rv[voff[x][0]] & vmask[x][0];
#pragma unroll
          for (int j = 1; j < NT; ++j) val ^= rv[voff[x][j]] & vmask[x][j];
          vd[x] = val;
        }
#pragma unroll
        for (int u = 0; u < NU; ++u) {
          const uint32_t x = vd[u >> 1];
          const int sh = 4 * (u & 1);
          qkv_v4i bo;
          bo[0] = static_cast<int>(x & (0x01010101u << sh));
          bo[1] = static_cast<int>(x & (0x02020202u << sh));
          bo[2] = static_cast<int>(x & (0x04040404u << sh));
          bo[3] = static_cast<int>(x & (0x08080808u << sh));
#pragma unroll
          for (int c = 0; c < QC; ++c)
            acc[c] = mfma_i8(a[c][u], bo, u == 0 ? qkv_v4i{0, 0, 0, 0} : acc[c]);
        }
      };
      qkv_v4i accs[2][QC];
      expand_mfma(0, accs[0]);
      // (a group's accumulators are read after the next group's MFMAs and a
      // branch; the first and the last group take the explicit pad)
      mfma_settle();
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        if (g + 1 < NG) expand_mfma(g + 1, accs[(g + 1) & 1]);
        if (g + 1 == NG) mfma_settle();
        const qkv_v4i* acc = accs[g & 1];
        const float nv = nb[g * 16 + ln];  // NaN past the range
        float sc[QC];
#pragma unroll
        for (int c = 0; c < QC; ++c) {
          if constexpr (NU * (1 << 20) < (1 << 23)) {
            // |digit sums| < NU 2^20 < 2^23: two exact int32 halves
            // (base 256), one rounding each
            const int zlo = acc[c][0] + acc[c][1] * 256;
            const int zhi = acc[c][2] + acc[c][3] * 256;
            sc[c] = nv * fmaf(static_cast<float>(zhi), 65536.f * fq[c],
                              fmaf(static_cast<float>(zlo), fq[c], cr[c]));
          } else {
            const float z = static_cast<float>(acc[c][0]) +
                            256.f * static_cast<float>(acc[c][1]) +
                            65536.f * static_cast<float>(acc[c][2]) +
                            16777216.f * static_cast<float>(acc[c][3]);
            sc[c] = nv * fmaf(z, fq[c], cr[c]);
          }
        }
#pragma unroll
        for (int c = 0; c < QC; ++c) {
          uint64_t cand = __builtin_amdgcn_ballot_w64(sc[c] >= thr[c]);
          while (cand) {  // rare: insert in ascending lane (= index) order
            const int L = __builtin_ctzll(cand);
            cand &= cand - 1;
            const float s_new = __shfl(sc[c], L, 64);
            const int q = c * 4 + (L >> 4);  // wave-local query
            float* qs = wls + q * k;
            int* qi = wli + q * k;
            if (s_new > qs[k - 1]) {
              // position = number of entries >= s_new (they hold lower indices)
              int ge = 0;
              for (int j = lane; j < k; j += 64) ge += qs[j] >= s_new ? 1 : 0;
              ge = qkv_wave_sum(ge);
              // shift [ge, k - 1) up by one, 64-entry blocks from the top down
              // (a block reads its entries before the block below is written)
              for (int t = (k - 1) >> 6; t >= 0; --t) {
                const int j = lane + 64 * t;
                const bool mv = j > ge && j < k;
                const float sv = mv ? qs[j - 1] : 0.f;
                const int iv = mv ? qi[j - 1] : 0;
                if (mv) {
                  qs[j] = sv;
                  qi[j] = iv;
                }
              }
              if (lane == 0) {
                qs[ge] = s_new;
                qi[ge] = static_cast<int>(s0 + g * 16 + (L & 15));
              }
              const float th = qs[k - 1];
              if (lg == (L >> 4)) {
                theta[c] = th;
                thr[c] = fmaxf(nextafterf(th, INFINITY), tg[c]);
              }
            }
          }
        }
      }
      if (more) stash(buf ^ 1);
      __syncthreads();
      buf ^= 1;
    }
    // this wave's lists -> candidates [query][vector chunk][k]; a full list's
    // k-th score raises the query's device-wide bound
#pragma unroll 1
    for (int q = 0; q < QW; ++q) {
      int ch = chs[0];
#pragma unroll
      for (int c = 1; c < QC; ++c) ch = q / 4 == c ? chs[c] : ch;
      const int qg = ch * 4 + (q % 4);
      if (qg >= M) continue;
      const int64_t base = (int64_t(qg) * nvc + vc) * k;
      for (int j = lane; j < k; j += 64) {
        cand_s[base + j] = wls[q * k + j];
        cand_i[base + j] = wli[q * k + j];
      }
      if (lane == 0 && wli[q * k + k - 1] >= 0)
        atomicMax(&gth[qg], fkey(wls[q * k + k - 1]));
    }
  }
}

// Final top-k per query over its (vector split) candidate lists: k rounds of a
// wave-wide arg-max (score descending, index ascending).
__global__ __launch_bounds__(64) void mips_merge(const float* __restrict__ cand_s,
                                                 const int* __restrict__ cand_i, int nsplit,
                                                 int k, float* __restrict__ out_s,
                                                 int64_t* __restrict__ out_i,
                                                 const int* __restrict__ over, int cap) {
  extern __shared__ __align__(16) float smem_mm[];
  const int q = blockIdx.x, lane = threadIdx.x;
  if (over != nullptr && over[q] <= cap) return;
  const int n = nsplit * k;
  float* cs = smem_mm;
  int* ci = reinterpret_cast<int*>(smem_mm + n);
  for (int i = lane; i < n; i += 64) {
    cs[i] = cand_s[int64_t(q) * n + i];
    ci[i] = cand_i[int64_t(q) * n + i];
  }
  __syncthreads();
  for (int r = 0; r < k; ++r) {
    float bs = -INFINITY;
    int bi = INT_MAX, bp = -1;
    for (int i = lane; i < n; i += 64) {
      const float s = cs[i];
      const int id = ci[i];
      if (id >= 0 && (s > bs || (s == bs && id < bi))) {
        bs = s;
        bi = id;
        bp = i;
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float os = __shfl_xor(bs, o, 64);
      const int oi = __shfl_xor(bi, o, 64), op = __shfl_xor(bp, o, 64);
      if (op >= 0 && (bp < 0 || os > bs || (os == bs && oi < bi))) {
        bs = os;
        bi = oi;
        bp = op;
      }
    }
    if (lane == 0) {
      out_s[int64_t(q) * k + r] = bs;
      out_i[int64_t(q) * k + r] = bi;
      if (bp >= 0) ci[bp] = -1;
    }
    __syncthreads();
  }
}


// ------------------------------------------------------------ filtered search
//
// The full scan above spends 4 query digits on every plane bit of every vector;
// only the handful of scores near the top need them.  Here a coordinate's code
// becomes one small integer L[code] (LUT, c[code] ~ a L[code]) and its weight
// q~_j one int8 digit, the QJL bit likewise, so that
//   score / n = f I - sum_j w_j + e,   I = sum_j d_j L[code_j] + dq_j V b_j
// exactly in int32, with |e| bounded from the digits' residuals (about 0.13
// standard deviations of the scores).  So:
//   1. mips_pass<false> takes the lower bounds of every 8th 16-vector group and
//      keeps the largest one of each (stream, column): maxima of disjoint sets
//      of vectors, so mips_bound's k-th largest of them bounds the k-th best
//      score from below;
//   2. mips_pass<true> lists the vectors whose upper bound reaches that bound
//      (about 25 times k per query on N(0, 1) data): every vector of the exact top
//      k, ties included, is among them;
//   3. mips_pick scores the listed vectors with all four digits, the same
//      integers and float operations as the full scan, and takes the k best.
// A query whose list overflows (or is seen in step 1 to be about to), or whose
// weights are not finite or all zero, goes to the full scan, with its 4-query chunk;
// the scan starts from its bound of step 1.  The results are the full scan's bit for
// bit.
//
// Measured (10^6 L2-normalised N(0, 1) vectors, 10^4 queries, d = 128, 3 bits,
// top-10): 3.02 - 3.19 ms against the full scan's 13.1: pass 2 ~2.4 ms (matrix cores
// busy ~45 %; MFMA time 1.06 ms), pass 1 0.3, the exact scores 0.19.  QT = 4 / 6 / 8:
// 3.98 / 3.22 / 3.02 ms.  Other data, against the full scan alone: norms that differ
// (the float products) 8.0 ms against 13.0; 1,000 clusters of spread 0.1 - 0.5 of
// their centres' 3.2 - 3.5; 100 clusters of spread 0.05, where lists of 10,000 would
// overflow, 12.3 against 13.0; every vector 2,000 times 12.1 against 12.4, a twentieth
// of them so 6.1 against 13.1 (1 query over 10^5: 112 us against 119).  Without the
// overflows foreseen and with whole 64-query tiles sent to the full scan the last
// four were 16.8, 16.1, 16.0 ms and 163 us.
// Six bit-plane operands in place of the level bytes (one digit, band twice as
// wide, 24 MFMAs per 64 queries) left half of the lists past their cap.
//
// Bounds: int8 MFMA, d / 32 per 16 queries x 16 vectors (the full scan at 2 MSE
// bits, d = 128: 24), beside ~41 VALU instructions of expansion per 16 vectors
// and one compare per score.  A wave holds the operands of 16 QT queries in
// registers and streams 16-vector groups from L2 into registers two groups
// ahead; no barrier, so the waves drift apart and one's VALU overlaps another's
// MFMAs.
// (the HIP headers' min of 64-bit integers goes through double)
__device__ __forceinline__ int64_t imin(int64_t a, int64_t b) { return a < b ? a : b; }

constexpr int kNoI = -(1 << 30);   // no value of I (|I| < 2^22) brings it to 0
constexpr int kFiltStep = 8;       // groups per sampled group of pass 1, from
constexpr int64_t kFiltStepN = 8192;     // this many vectors (below, pass 1 takes every group)
constexpr int kFiltQueue = 64;     // candidates a wave holds in LDS before a flush
constexpr int kFiltQT = 8;         // 16-query tiles per wave, many queries
constexpr int kFiltKMax = 64;      // k up to which the filter runs
constexpr int64_t kFiltMinN = 256;  // vectors from which the filter runs

// The codebook's integer levels: c[code] = a L[code] + (at most delta), L as the
// bytes of (hi, lo); the QJL bit's byte value V = 1 << vlog, 2 qjl_scale <= a V.
struct FiltTab {
  uint32_t lo, hi;
  float a, delta;
  int lmax, vlog;
};

// Lane group g expands word g of each plane (d = 128; d = 96: group 3 has none)
// into NU = 4 operands, MSE bits 0-3 and 4-7 of each byte, then the QJL bits; at
// d = 64 word g % 2, the bits 4 (g / 2) .. + 3 of each byte, NU = 2.
template <int PDW>
struct FiltCfg {
  static constexpr int NU = PDW == 2 ? 2 : 4;
};

// Filter operands of one 16-query tile per workgroup, from q~ and w =
// alpha |q~| S (prepare_mfma's qw): 16 threads per query, d / 16 coordinates
// each.  ciu / cil: the bounds' constants in units of f, rounded outwards.  The
// slack covers the rounding of the exact path's 30-bit weights (at most 64 2^-fq
// for each of 640) and of its floats.
template <int PDW>
__global__ __launch_bounds__(256) void mips_fprep(const float* __restrict__ qw,
                                                  const float* __restrict__ rowc, int M,
                                                  FiltTab ft, uint32_t* __restrict__ af,
                                                  int* __restrict__ ciu, int* __restrict__ cil,
                                                  int* __restrict__ cnt, int cap,
                                                  float* __restrict__ unit,
                                                  int* __restrict__ left,
                                                  int* __restrict__ claimed) {
  constexpr int NU = FiltCfg<PDW>::NU, NWD = NU * 256;
  constexpr int JT = PDW * 2;  // coordinates per thread
  __shared__ uint32_t img[NWD];
  int8_t* ib = reinterpret_cast<int8_t*>(img);
  const int tid = threadIdx.x, m = tid >> 4, t16 = tid & 15;
  for (int i = tid; i < NWD; i += 256) img[i] = 0;
  if (tid < 4) claimed[blockIdx.x * 4 + tid] = 0;  // no chunk left to the full scan yet
  if (blockIdx.x == 0 && tid == 0) left[0] = 0;
  const int q = blockIdx.x * 16 + m, qc = min(q, M - 1);
  float v[JT], w[JT];
  float mx = 0.f, l1 = 0.f, sw = 0.f, aw = 0.f;
#pragma unroll
  for (int x = 0; x < JT; ++x) {
    const int j = t16 + 16 * x;
    v[x] = qw[int64_t(qc) * 256 + j];
    w[x] = qw[int64_t(qc) * 256 + 128 + j];
    mx = fmaxf(mx, fabsf(v[x]));
    l1 += fabsf(v[x]);
    sw += w[x];
    aw += fabsf(w[x]);
  }
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) {
    mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    l1 += __shfl_xor(l1, o, 64);
    sw += __shfl_xor(sw, o, 64);
    aw += __shfl_xor(aw, o, 64);
  }
  const float f = mx * ft.a / 127.f;
  const bool ok = f > 1e-30f && l1 < 1e30f && aw < 1e30f;  // false for NaN sums too
  const float rf = ok ? 1.f / f : 0.f;
  const float iv = 1.f / static_cast<float>(1 << ft.vlog);
  __syncthreads();
  float er = 0.f, eu = 0.f, el = 0.f;
  // byte of operand dword e of MFMA u, lane group g: (word wd, bit i of byte beta)
  auto byte_at = [&](int j, bool qjl) {
    const int wd = j >> 5, i = j & 7, beta = (j >> 3) & 3;
    int g, u;
    if constexpr (PDW == 2) {
      g = wd + 2 * (i >> 2);
      u = qjl ? 1 : 0;
    } else {
      g = wd;
      u = (qjl ? 2 : 0) + (i >> 2);
    }
    return ((u * 64 + m + 16 * g) * 4 + (i & 3)) * 4 + beta;
  };
  auto digit = [&](float W, int at, float& r) {
    const float d = fminf(fmaxf(rintf(W * rf), -127.f), 127.f);
    r = fmaf(-d, f, W);
    ib[at] = ok ? static_cast<int8_t>(static_cast<int>(d)) : 0;
  };
#pragma unroll
  for (int x = 0; x < JT; ++x) {
    const int j = t16 + 16 * x;
    float r;
    digit(v[x] * ft.a, byte_at(j, false), r);
    er += fabsf(r);
    digit(2.f * w[x] * iv, byte_at(j, true), r);
    eu += fmaxf(r, 0.f);
    el += fmaxf(-r, 0.f);
  }
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) {
    er += __shfl_xor(er, o, 64);
    eu += __shfl_xor(eu, o, 64);
    el += __shfl_xor(el, o, 64);
  }
  if (t16 == 0) {
    const float cr = rowc[int64_t(qc) * 2];
    const float vq = static_cast<float>(1 << ft.vlog);
    const float slack = 1.9e-6f * (2.f * ft.a * ft.lmax * l1 + 4.f * aw + fabsf(cr)) +
                        65536.f * rowc[int64_t(qc) * 2 + 1];
    const float e = er * ft.lmax + ft.delta * l1 + slack;
    const float up = (e + vq * eu - sw) * rf, low = (-e - vq * el - sw) * rf;
    // (bounds that int32 sums hold; QJL weights far past the digits give larger ones)
    const bool use = ok && fabsf(cr) < 1e30f && fabsf(up) < 1e9f && fabsf(low) < 1e9f;
    ciu[q] = use ? static_cast<int>(ceilf(up)) + 1 : 0;
    cil[q] = use ? static_cast<int>(floorf(low)) - 1 : 0;
    cnt[q] = use || q >= M ? 0 : cap + 1;  // past cap: left to the full scan
    unit[q] = f;
  }
  __syncthreads();
  for (int i = tid; i < NWD; i += 256) af[int64_t(blockIdx.x) * NWD + i] = img[i];
}

// One pass over the database.  Waves: (query tile of 16 QT, stream p of P);
// stream p takes the groups p, p + P, ... of the ng (sampled: every gstep-th)
// 16-vector groups, so that all waves sweep the database together, and with P a
// multiple of 8 a stream's waves share an XCD's L2.
//
// While a group's norms all lie within 0.1 % below nq (an L2-normalised
// database), the scores are compared as integers: COLLECT starts the
// accumulators at minus the queries' thresholds at nq, so that a set sign bit in
// every accumulator (one AND of two values each) dismisses the group, and the
// sampling pass keeps integer maxima.  Other groups take the float products.
// Such a group costs 4 QT MFMAs (512 cycles at QT = 8) and ~75 VALU
// instructions; the next group's expansion and the reductions are scheduled
// between the MFMAs (three VALU instructions fill an MFMA's 16 cycles).
template <int MB, int PDW, int QT, bool COLLECT>
__global__ __launch_bounds__(256, 2) void mips_pass(
    const qkv_v4i* __restrict__ af, const int* __restrict__ cinit, const float* __restrict__ thr,
    const uint8_t* __restrict__ kst, const float* __restrict__ norms, int64_t N, int ntile,
    int wq, int pb, int64_t ng, int gstep, int M, FiltTab ft, float* __restrict__ mxo,
    int* __restrict__ cnt, int* __restrict__ cand, int cap) {
  constexpr int NU = FiltCfg<PDW>::NU, RAWD = (MB + 1) * PDW, NP = MB + 1;
  constexpr int NI = PDW == 2 ? 4 : 8;  // bits of each byte a lane expands
  constexpr int kQ = COLLECT ? kFiltQueue + 256 * QT : 1;  // one group lists 256 QT at most
  __shared__ int qv[COLLECT ? 4 : 1][kQ];
  __shared__ uint8_t qq[COLLECT ? 4 : 1][kQ];
  __shared__ __align__(16) int cis[4][16 * QT];
  __shared__ __align__(16) float ths[COLLECT ? 4 : 1][COLLECT ? 16 * QT : 4];
  __shared__ float mxl[COLLECT ? 1 : 4][COLLECT ? 1 : 4 * QT][64];  // running maxima

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 15, lg = lane >> 4;
  const int ws = 4 / wq;  // streams per workgroup
  const int tile = (blockIdx.x / pb) * wq + wave % wq;
  const int p = (blockIdx.x % pb) * ws + wave / wq, P = pb * ws;
  if (tile >= ntile) return;  // (no barrier below: the LDS arrays are each wave's own)

  qkv_v4i a[QT][NU];
#pragma unroll
  for (int t = 0; t < QT; ++t)
#pragma unroll
    for (int u = 0; u < NU; ++u)
      a[t][u] = af[((int64_t(tile) * QT + t) * NU + u) * 64 + lane];
  if constexpr (!COLLECT) {
    for (int i = lane; i < 16 * QT; i += 64) cis[wave][i] = cinit[int64_t(tile) * 16 * QT + i];
  } else {
    // A 4-query chunk with a query left to the full scan goes there whole (the scan
    // takes it at the same cost), and so does a tile of whose chunks fewer than a
    // fifth remain: this pass costs a fifth of the scan.  (Every wave of the tile
    // decides alike, before any lists.)
    const int q0 = tile * 16 * QT;
    bool real = false, keep = false;
    if (lane < 4 * QT) {
      real = keep = q0 + 4 * lane < M;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float th = thr[q0 + 4 * lane + r];
        if (q0 + 4 * lane + r < M && th != th) keep = false;
      }
    }
    const uint64_t kept = __builtin_amdgcn_ballot_w64(keep);
    const bool few = 5 * __builtin_popcountll(kept) <
                     __builtin_popcountll(__builtin_amdgcn_ballot_w64(real));
    bool some = false;
    for (int i = lane; i < 16 * QT; i += 64) {
      float th = thr[q0 + i];
      if (few || !((kept >> (i / 4)) & 1u)) {
        if (th == th) cnt[q0 + i] = cap + 1;
        th = __builtin_nanf("");
      }
      cis[wave][i] = cinit[q0 + i];
      ths[wave][i] = th;
      some |= th == th;
    }
    if (__builtin_amdgcn_ballot_w64(some) == 0) return;
  }
  // COLLECT: minus the integer thresholds at nq; else the largest I at nq
  qkv_v4i ti[COLLECT ? QT : 1];
  int mi[COLLECT ? 1 : 4 * QT];
  float nq = -1.f;
  if constexpr (!COLLECT) {
#pragma unroll
    for (int t = 0; t < 4 * QT; ++t) mxl[wave][t][lane] = -INFINITY;
  }
  if constexpr (!COLLECT) {
#pragma unroll
    for (int t = 0; t < 4 * QT; ++t) mi[t] = kNoI;
  }

  struct Row {
    uint32_t w[NP];
    float n;
  };
  // this lane's word of each plane: 32-bit lane offsets from a wave-uniform base
  const uint32_t wo = PDW == 2 ? (lg & 1) : PDW == 3 ? min(lg, 2) : lg;
  auto load = [&](int64_t x) {
    Row r;
    const int64_t v0 = imin(x, ng - 1) * gstep * 16;
    // (the last group may be partial; no branch, which would split the schedule)
    const uint32_t left = static_cast<uint32_t>(imin(N - 1 - v0, 15));
    const uint32_t ni = min<uint32_t>(ln, left), lo = (ni * RAWD + wo) * 4;
    const uint8_t* base = kst + v0 * (RAWD * 4);
#pragma unroll
    for (int j = 0; j < NP; ++j)
      r.w[j] = *reinterpret_cast<const uint32_t*>(base + (lo + 4 * PDW * j));
    const float n = norms[v0 + ni];
    // past the end (and, among the lower bounds, a negative norm): passes no compare
    r.n = ni == static_cast<uint32_t>(ln) && (COLLECT || n >= 0.f) ? n : __builtin_nanf("");
    return r;
  };

  // the NU operands of 16 vectors: codes' levels, then QJL bits (byte value V)
  const uint32_t vmask = 0x01010101u << ft.vlog;
  auto expand = [&](const Row& row, qkv_v4i* bo) {
    uint32_t w[NP];
#pragma unroll
    for (int j = 0; j < NP; ++j) w[j] = PDW == 2 ? row.w[j] >> (4 * (lg >> 1)) : row.w[j];
    // codes of the even and of the odd bits, two bits each (their low two bits)
    uint32_t ze, zo;
    if constexpr (MB == 1) {
      ze = w[0];
      zo = w[0] >> 1;
    } else {
      ze = (w[0] & 0x55555555u) | ((w[1] << 1) & 0xaaaaaaaau);
      zo = ((w[0] >> 1) & 0x55555555u) | (w[1] & 0xaaaaaaaau);
    }
    const uint32_t y = __builtin_amdgcn_alignbit(w[MB], w[MB], 32 - ft.vlog);  // left by vlog
    constexpr uint32_t zm = MB == 1 ? 0x01010101u : 0x03030303u;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      uint32_t sel = ((i & 1 ? zo : ze) >> (i & ~1)) & zm;
      if constexpr (MB == 3)
        sel |= (i < 2 ? w[2] << (2 - i) : w[2] >> (i - 2)) & 0x04040404u;
      bo[i >> 2][i & 3] = static_cast<int>(__builtin_amdgcn_perm(ft.hi, ft.lo, sel));
      bo[NU / 2 + (i >> 2)][i & 3] = static_cast<int>(__builtin_amdgcn_alignbit(y, y, i) & vmask);
    }
  };

  int qn = 0;  // queued candidates (wave-uniform)
  bool done = false;  // every query's list is past its cap
  auto flush = [&]() {
    bool any = false;
    for (int i = lane; i < qn; i += 64) {
      const int ql = qq[wave][i];
      const int64_t q = int64_t(tile) * 16 * QT + ql;
      const int at = atomicAdd(&cnt[q], 1);
      if (at < cap) {
        cand[q * cap + at] = qv[wave][i];
      } else {  // the query goes to the full scan: take no more of it
        ths[wave][ql] = __builtin_nanf("");
        any = true;
      }
    }
    qn = 0;
    if (__builtin_amdgcn_ballot_w64(any)) {
      nq = -1.f;  // (new integer thresholds)
      bool alive = false;
      for (int i = lane; i < 16 * QT; i += 64) alive |= ths[wave][i] == ths[wave][i];
      done = __builtin_amdgcn_ballot_w64(alive) == 0;
    }
  };

  // COLLECT: minus the smallest I that may pass at norms in (0.999 nq, nq]
  auto thresholds = [&]() {
    const float rhi = 1.f / nq, rlo = rhi * 1.00101f;
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      const qkv_v4f th = *reinterpret_cast<const qkv_v4f*>(&ths[wave][16 * t + 4 * lg]);
      const qkv_v4i ci = *reinterpret_cast<const qkv_v4i*>(&cis[wave][16 * t + 4 * lg]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float x = fminf(th[r] * rhi, th[r] * rlo);
        const float y = x - fabsf(x) * 1e-6f;
        ti[t][r] = th[r] == th[r] ? ci[r] - static_cast<int>(floorf(fminf(fmaxf(y, -1e9f), 1e9f)))
                                  : kNoI;
      }
    }
  };
  // sampling: the integer maxima at nq into the float ones
  auto settle_max = [&]() {
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      const qkv_v4i ci = *reinterpret_cast<const qkv_v4i*>(&cis[wave][16 * t + 4 * lg]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (mi[4 * t + r] > kNoI) {
          const float s = static_cast<float>(mi[4 * t + r] + ci[r]) * nq;
          float& m = mxl[wave][4 * t + r][lane];
          m = fmaxf(m, s >= 0.f ? 0.998999f * s : s);
        }
        mi[4 * t + r] = kNoI;
      }
    }
  };
  auto product = [&](int t, const qkv_v4i* bo, qkv_v4i c) {
#pragma unroll
    for (int u = 0; u < NU; ++u) c = mfma_i8(a[t][u], bo[u], c);
    return c;
  };
  auto push = [&](uint64_t h, int ql, int64_t x) {
    const int nh = __builtin_popcountll(h);
    if ((h >> lane) & 1u) {
      const int at = qn + __builtin_popcountll(h & ((uint64_t(1) << lane) - 1));
      qv[wave][at] = static_cast<int>(x * 16 + ln);
      qq[wave][at] = static_cast<uint8_t>(ql + 4 * lg);
    }
    qn += nh;
  };

  // group x from its operands cur and norms nc, while row (the group P on)
  // becomes nxt and the row's registers take the load of the group 3 P on
  auto body = [&](const qkv_v4i* cur, float nc, qkv_v4i* nxt, float& nn, Row& row, int64_t x) {
    bool uni = __builtin_amdgcn_ballot_w64(nc <= nq && nc > nq * 0.999f) == ~0ull;
    if (!uni) {
      // the largest norm, its low 12 mantissa bits rounded up: the next nq
      float m = nc == nc ? nc : 0.f;
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
      const float c = __uint_as_float((__float_as_uint(m) + 0xfffu) & ~0xfffu);
      if (__builtin_amdgcn_ballot_w64(nc <= c && nc > c * 0.999f) == ~0ull && c > 1e-30f &&
          c < 1e30f) {
        if constexpr (!COLLECT) settle_max();
        nq = c;
        if constexpr (COLLECT) thresholds();
        uni = true;
      }
    }
    if (uni) {
      int m[QT];
#pragma unroll
      for (int t = 0; t < QT; t += 2) {  // two independent accumulator chains
        qkv_v4i c0 = {0, 0, 0, 0}, c1 = {0, 0, 0, 0};
        if constexpr (COLLECT) {
          c0 = ti[t];
          if (t + 1 < QT) c1 = ti[t + 1];
        }
#pragma unroll
        for (int u = 0; u < NU; ++u) {
          c0 = mfma_i8(a[t][u], cur[u], c0);
          if (t + 1 < QT) c1 = mfma_i8(a[t + 1 < QT ? t + 1 : 0][u], cur[u], c1);
        }
        if constexpr (COLLECT) {
          m[t] = c0[0] & c0[1] & c0[2] & c0[3];
          if (t + 1 < QT) m[t + 1] = c1[0] & c1[1] & c1[2] & c1[3];
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            mi[4 * t + r] = max(mi[4 * t + r], c0[r]);
            if (t + 1 < QT) mi[4 * t + 4 + r] = max(mi[4 * t + 4 + r], c1[r]);
          }
        }
      }
      expand(row, nxt);
#pragma unroll
      for (int u = 0; u < NU; ++u) asm volatile("" : "+v"(nxt[u]));  // (not sunk past the branch)
      nn = row.n;
      row = load(x + 3 * P);
#pragma unroll
      for (int i = 0; i < QT * NU; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);   // MFMA
        __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);   // VALU
      }
      if constexpr (COLLECT) {
        int all = m[0];
#pragma unroll
        for (int t = 1; t < QT; ++t) all &= m[t];
        if (__builtin_amdgcn_ballot_w64(all >= 0)) {
#pragma unroll
          for (int t = 0; t < QT; ++t) {
            if (__builtin_amdgcn_ballot_w64(m[t] >= 0) == 0) continue;
            const qkv_v4i c = product(t, cur, ti[t]);  // again: the sums were not kept
            mfma_settle();
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const uint64_t h = __builtin_amdgcn_ballot_w64(c[r] >= 0);
              if (h) push(h, 16 * t + r, x);
            }
          }
          if (qn > kFiltQueue) flush();
        }
      }
      return;
    }
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      const qkv_v4i c = product(t, cur, qkv_v4i{0, 0, 0, 0});
      const qkv_v4i ci = *reinterpret_cast<const qkv_v4i*>(&cis[wave][16 * t + 4 * lg]);
      mfma_settle();
      if constexpr (COLLECT) {
        const qkv_v4f th = *reinterpret_cast<const qkv_v4f*>(&ths[wave][16 * t + 4 * lg]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          // (the bounds hold for norms >= 0: any other vector is listed)
          const uint64_t h = __builtin_amdgcn_ballot_w64(
              static_cast<float>(c[r] + ci[r]) * nc >= th[r] || (nc < 0.f && th[r] == th[r]));
          if (h) push(h, 16 * t + r, x);
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float& m = mxl[wave][4 * t + r][lane];
          m = fmaxf(m, static_cast<float>(c[r] + ci[r]) * nc);
        }
      }
    }
    if constexpr (COLLECT) {
      if (qn > kFiltQueue) flush();
    }
    // (opaque: kept apart from the same lines above, whose place is among the MFMAs)
#pragma unroll
    for (int j = 0; j < NP; ++j) asm volatile("" : "+v"(row.w[j]));
    expand(row, nxt);
    nn = row.n;
    row = load(x + 3 * P);
  };

  qkv_v4i b0[NU], b1[NU];
  float n0, n1 = 0.f;
  Row r1 = load(p), r0 = load(int64_t(p) + P);
  expand(r1, b0);
  n0 = r1.n;
  r1 = load(int64_t(p) + 2 * P);
  for (int64_t x = p; x < ng; x += 2 * P) {
    body(b0, n0, b1, n1, r0, x);
    if (x + P < ng) body(b1, n1, b0, n0, r1, x + P);
    if (COLLECT && done) break;
  }
  if constexpr (COLLECT) {
    flush();
  } else {
    settle_max();
#pragma unroll
    for (int t = 0; t < QT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t q = (int64_t(tile) * QT + t) * 16 + 4 * lg + r;
        mxo[(q * P + p) * 16 + ln] = mxl[wave][4 * t + r][lane];
      }
  }
}

// Threshold of one query per workgroup: the k-th largest of 256 R maxima, each
// the largest of a disjoint share of the query's n stream maxima, lowered by the
// rounding of one float product.  NaN (admits nothing) for a query the filter
// does not serve: past the cap already, without k finite maxima, or with so many
// shares whose upper bound reaches the threshold (at the mean of 64 norms) that its
// list would overflow: v sampled vectors fall on c of S shares, v ~ -S ln(1 - c / S),
// and step times as many are listed.  (10^6 vectors, 2,000 copies of each, 10^4
// queries: pass 2 was 2.4 ms of 16.1, the full scan alone takes 12.4.)  In units of a
// score the threshold is where the full scan of such a query starts from (gth),
// instead of filling its lists (100 queries, 10^5 such vectors: 790 us, now 246; the
// full scan alone 570).
template <int R>
__global__ __launch_bounds__(256) void mips_bound(const float* __restrict__ mx, int n, int k,
                                                  int M, int step, const float* __restrict__ unit,
                                                  const int* __restrict__ ciu,
                                                  const int* __restrict__ cil,
                                                  const float* __restrict__ norms, int64_t N,
                                                  float* __restrict__ thr, int* __restrict__ cnt,
                                                  int cap, uint32_t* __restrict__ gth) {
  __shared__ float sh[256 * R];
  const int q = blockIdx.x, tid = threadIdx.x;
  if (q >= M || cnt[q] > cap) {
    if (tid == 0) thr[q] = __builtin_nanf("");
    return;
  }
#pragma unroll
  for (int x = 0; x < R; ++x) {
    float m = -INFINITY;
#pragma unroll 4
    for (int i = tid + 256 * x; i < n; i += 256 * R) m = fmaxf(m, mx[int64_t(q) * n + i]);
    sh[tid + 256 * x] = m;
  }
  __syncthreads();
  if (tid >= 64) return;
  float v[4 * R];
#pragma unroll
  for (int x = 0; x < 4 * R; ++x) v[x] = sh[tid + 64 * x];
  float kth = -INFINITY;
  for (int r = 0; r < k; ++r) {
    float best = v[0];
#pragma unroll
    for (int x = 1; x < 4 * R; ++x) best = fmaxf(best, v[x]);
    kth = wave_max_dpp(best);
    const uint64_t who = __builtin_amdgcn_ballot_w64(best == kth);
    if (tid == static_cast<int>(__builtin_ctzll(who))) {
      bool out = false;  // the first slot that holds it
#pragma unroll
      for (int x = 0; x < 4 * R; ++x)
        if (!out && v[x] == kth) {
          v[x] = -INFINITY;
          out = true;
        }
    }
  }
  const float t = kth - fabsf(kth) * 1.9e-6f;
  float nm = norms[tid * (N / 64)];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) nm += __shfl_xor(nm, o, 64);
  const float reach = t - static_cast<float>(ciu[q] - cil[q]) * (nm * (1.f / 64.f));
  int c = k;  // shares that reach it (the k best were taken out above)
#pragma unroll
  for (int x = 0; x < 4 * R; ++x) c += __builtin_popcountll(__builtin_amdgcn_ballot_w64(v[x] >= reach));
  if (tid == 0) {
    const bool ok = fabsf(kth) < INFINITY;  // else: left to the full scan
    const float S = 256.f * R, est = step * S * -logf(fmaxf(1.f - c / S, 1e-6f));
    const bool list = ok && est <= cap;
    thr[q] = list ? t : __builtin_nanf("");
    if (!list) cnt[q] = cap + 1;
    const float s = t * unit[q], lo = s - fabsf(s) * 2e-6f - 1e-36f;
    if (ok && fabsf(lo) < 1e38f) gth[q] = fkey(lo);
  }
}

// Exact scores of a query's listed vectors (the full scan's integers: digit
// pairs of each weight, summed over the set plane bits) and the k best of them
// (score descending, index ascending).  One query per workgroup, a thread per
// vector; the query's weights as LDS tables that all lanes read together.
template <int MB, int PDW>
__global__ __launch_bounds__(256) void mips_pick(const qkv_v4i* __restrict__ aq,
                                                 const float* __restrict__ rowc,
                                                 const uint8_t* __restrict__ kst,
                                                 const float* __restrict__ norms, int k,
                                                 const int* __restrict__ cnt,
                                                 const int* __restrict__ cand, int cap,
                                                 int* __restrict__ left, int* __restrict__ claimed,
                                                 float* __restrict__ out_s,
                                                 int64_t* __restrict__ out_i) {
  using F = MipsCfg<MB, PDW>;
  constexpr int NPL = F::NPL, NU = F::NU, DPL = F::DPL, RAWD = F::RAWD;
  constexpr int VD = NPL * PDW;  // virtual row dwords
  constexpr bool kPair = NU * (1 << 20) < (1 << 23);  // two exact halves, as the full scan
  __shared__ int tab[VD * 32][kPair ? 2 : 4];
  extern __shared__ __align__(16) float smem_mk[];  // [cap] scores, [cap] indices
  const int q = blockIdx.x, tid = threadIdx.x;
  const int n = cnt[q];
  if (n > cap) {  // the query's chunk goes to the full scan
    if (tid == 0 && atomicExch(&claimed[q / 4], 1) == 0) left[1 + atomicAdd(&left[0], 1)] = q / 4;
    return;
  }
  float* cs = smem_mk;
  int* ci = reinterpret_cast<int*>(smem_mk + cap);
  // digit v of the weight at virtual bit (plane, coordinate) from the operand image
  const int8_t* ab = reinterpret_cast<const int8_t*>(aq) + int64_t(q >> 2) * NU * 1024;
  for (int p = tid; p < VD * 32; p += 256) {
    const int pl = p / (32 * PDW), j = p - pl * 32 * PDW;
    const int w32 = pl * 4 + (j >> 5), i = p & 7, e = i & 3, beta = (p >> 3) & 3;
    const int g = w32 / DPL, u = 2 * (w32 - g * DPL) + (i >> 2);
    const int8_t* src = ab + ((u * 64 + 16 * g + 4 * (q & 3)) * 4 + e) * 4 + beta;
    const int m = i == 7 ? -128 : 1 << i;
    const int d0 = src[0], d1 = src[16], d2 = src[32], d3 = src[48];
    if constexpr (kPair) {
      tab[p][0] = m * (d0 + 256 * d1);
      tab[p][1] = m * (d2 + 256 * d3);
    } else {
      tab[p][0] = m * d0;
      tab[p][1] = m * d1;
      tab[p][2] = m * d2;
      tab[p][3] = m * d3;
    }
  }
  const float cr = rowc[int64_t(q) * 2], fq = rowc[int64_t(q) * 2 + 1];
  __syncthreads();
  for (int c = tid; c < n; c += 256) {
    const int v = cand[int64_t(q) * cap + c];
    const uint32_t* src = reinterpret_cast<const uint32_t*>(kst) + int64_t(v) * RAWD;
    int z[kPair ? 2 : 4] = {};
    // (rolled: unrolled, the tables move out of the candidate loop into registers)
#pragma unroll 1
    for (int wd = 0; wd < VD; ++wd) {
      uint32_t x;
      if constexpr (MB <= 2) {
        x = src[wd];
      } else {  // virtual planes b0, b1, b2, their parity, QJL
        x = src[wd < 3 * PDW ? wd : wd - PDW];
        if (wd >= 3 * PDW && wd < 4 * PDW) x ^= src[wd - 3 * PDW] ^ src[wd - 2 * PDW];
      }
      const int* tp = tab[wd * 32];
#pragma unroll
      for (int b = 0; b < 32; ++b) {
        const int on = -static_cast<int>((x >> b) & 1u);
#pragma unroll
        for (int h = 0; h < (kPair ? 2 : 4); ++h) z[h] += tp[b * (kPair ? 2 : 4) + h] & on;
      }
    }
    const float nv = norms[v];
    float s;
    if constexpr (kPair) {
      s = nv * fmaf(static_cast<float>(z[1]), 65536.f * fq,
                    fmaf(static_cast<float>(z[0]), fq, cr));
    } else {
      const float zz = static_cast<float>(z[0]) + 256.f * static_cast<float>(z[1]) +
                       65536.f * static_cast<float>(z[2]) + 16777216.f * static_cast<float>(z[3]);
      s = nv * fmaf(zz, fq, cr);
    }
    cs[c] = s;
    ci[c] = s > -INFINITY ? v : -1;  // (NaN and -inf are no results, as in the full scan)
  }
  __syncthreads();
  if (tid >= 64) return;
  // each lane's best of its stride; a round re-reads only the winner's stride
  float bs = -INFINITY;
  int bi = INT_MAX, bp = -1;
  auto scan = [&]() {
    bs = -INFINITY;
    bi = INT_MAX;
    bp = -1;
    for (int i = tid; i < n; i += 64) {
      const float s = cs[i];
      const int id = ci[i];
      if (id >= 0 && (s > bs || (s == bs && id < bi))) {
        bs = s;
        bi = id;
        bp = i;
      }
    }
  };
  scan();
  for (int r = 0; r < k; ++r) {
    float ms = bs;
    int mi = bi, mp = bp;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float os = __shfl_xor(ms, o, 64);
      const int oi = __shfl_xor(mi, o, 64), op = __shfl_xor(mp, o, 64);
      if (op >= 0 && (mp < 0 || os > ms || (os == ms && oi < mi))) {
        ms = os;
        mi = oi;
        mp = op;
      }
    }
    if (tid == 0) {
      out_s[int64_t(q) * k + r] = mp < 0 ? -INFINITY : ms;
      out_i[int64_t(q) * k + r] = mp < 0 ? INT_MAX : mi;
    }
    if (mp >= 0 && mp == bp) {
      ci[bp] = -1;
      scan();
    }
  }
}

}  // namespace

// ------------------------------------------------------------ MIPS search (ABI)

// Device-wide per-query bounds start at -inf.
__global__ __launch_bounds__(256) void mips_init(uint32_t* __restrict__ gth, int M) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < M) gth[i] = 0x007fffffu;  // fkey(-inf)
}

// Queries (fp32), Pi and S of a d < 128 index zero-padded to 128.
__global__ __launch_bounds__(256) void mips_pad(const void* __restrict__ q, int q_dtype, int M,
                                                int d, const float* __restrict__ pi,
                                                const float* __restrict__ signs,
                                                float* __restrict__ qp, float* __restrict__ pip,
                                                float* __restrict__ sp) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  const int64_t nq = int64_t(M) * 128;
  if (i < nq) {
    const int64_t m = i / 128;
    const int j = static_cast<int>(i - m * 128);
    qp[i] = j < d ? qkv_load(q, m * d + j, q_dtype) : 0.f;
  } else if (i < nq + 128 * 128) {
    const int64_t e = i - nq;
    const int r = static_cast<int>(e / 128), c = static_cast<int>(e % 128);
    pip[e] = (r < d && c < d) ? pi[r * d + c] : 0.f;
  } else if (i < nq + 128 * 128 + 128) {
    const int j = static_cast<int>(i - nq - 128 * 128);
    sp[j] = j < d ? signs[j] : 0.f;
  }
}

namespace {

struct MipsLayout {
  int64_t aq, rowc, cs, ci, gth, pad;
  int64_t qw, af, ciu, cil, cnt, thr, unit, left, claimed, mx, cand;  // the filter's
  int64_t total;
};

// Vector chunks per query tile: enough (query tile, chunk) items for several
// per workgroup slot (12 per CU: six per workgroup at two per CU; fewer,
// longer chunks fill fewer per-chunk top-k lists -- cfg5 14.0 ms against
// 14.4 at 24 per CU and 15.4 at 48), chunks of at least 16 steps, at most
// 256 chunks.
int mips_splits(int32_t M, int64_t N, int mbits) {
  const int qc = mbits <= 2 ? 4 : 2;
  const int64_t qtiles = (M + 16 * qc - 1) / (16 * qc);
  const int64_t want = (12 * int64_t(qkv_num_cus()) + qtiles - 1) / qtiles;
  const int64_t maxs = std::max<int64_t>(1, (N + 16 * kMipsStep - 1) / (16 * kMipsStep));
  return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>({want, maxs, 256})));
}

// How a batch of M queries runs: on the full scan, or through the filter with
// 16 qt queries per wave, wq query tiles and 4 / wq streams per workgroup, pb
// workgroups (P = 4 pb / wq streams) along the database.
struct MipsPlan {
  bool filt;
  int qt, wq, pb, P, ntile, cap, step;
};

// Listed vectors a query may have (about 25 times k on N(0, 1) data), and the queries
// per batch that this allows (64 MiB of lists).
int filt_cap(int k) { return std::max(1024, 64 * k); }
int filt_batch(int k) { return 16384 * 1024 / filt_cap(k); }

// The filter serves every k <= 64 (its bound comes from 1024 maxima at most):
// a scan's lists fill at ~0.7 ms per call whatever the size (top-10 of 10^4
// vectors for 64 queries 753 us, filtered 78; for one query 116 and 49; of 10^6
// for 10^4 queries 13.1 ms and 3.0).  One or two queries over a few hundred
// vectors are the exception, where a scan is two launches against seven (top-1 of
// 256: 24 - 29 us and 37 - 44; of 700: 34 - 45 and 38 - 44; top-3 of 400: 34 - 43
// and 40 - 46; top-10 of 256: 50 - 60 and 38 - 51).
MipsPlan mips_plan(int32_t M, int64_t N, int k) {
  MipsPlan pl{};
  const bool tiny = M <= 2 && N < 700 && N * N * k * M < 700 * 700;
  pl.filt = k <= kFiltKMax && N >= kFiltMinN && !tiny;
  if (!pl.filt) return pl;
  pl.qt = M <= 16 ? 1 : M <= 64 ? 2 : M <= 1024 ? 4 : kFiltQT;
  pl.ntile = (M + 16 * pl.qt - 1) / (16 * pl.qt);
  pl.wq = pl.ntile >= 4 ? 4 : pl.ntile >= 2 ? 2 : 1;
  pl.cap = filt_cap(k);
  const int ws = 4 / pl.wq, tg = (pl.ntile + pl.wq - 1) / pl.wq;
  const int64_t slots = 2 * int64_t(qkv_num_cus());
  pl.step = N >= kFiltStepN ? kFiltStep : 1;
  const int64_t ng1 = (N + 16 * pl.step - 1) / (16 * pl.step);  // sampled groups
  // streams: whole rounds of the chip as nearly as a multiple of 8 allows, at
  // least 4 k stream maxima, at least one sampled group each
  const int lo = std::max(8, (k + 4 * ws - 1) / (4 * ws) + 7 & ~7);
  const int hi = static_cast<int>(std::max<int64_t>(lo, std::min<int64_t>(ng1 / ws, 512)));
  double best = 0.0;
  pl.pb = lo;
  for (int pb = lo; pb <= hi; pb += 8) {
    const int64_t wg = int64_t(tg) * pb, rounds = (wg + slots - 1) / slots;
    const double eff = double(wg) / double(rounds * slots) - 0.01 * double(rounds);
    if (eff > best) {
      best = eff;
      pl.pb = pb;
    }
  }
  pl.P = pl.pb * ws;
  return pl;
}

// Integer levels of a symmetric codebook: the largest level mapped to 8 .. 100,
// the others rounded, whichever fits best; false where the QJL weights would
// need a byte value past 64 (the full scan then runs).
bool filt_table(const float* kc, int mbits, float qjl_scale, FiltTab* ft) {
  const int n = 1 << mbits;
  const float cmax = *std::max_element(kc, kc + n);  // (a caller's codebook may be in any order)
  bool found = false;
  for (int lm = 8; lm <= 100; ++lm) {
    const float a = cmax / lm;
    if (!(a > 0.f)) return false;
    int vlog = 0;
    while (vlog < 7 && a * (1 << vlog) < 2.f * fabsf(qjl_scale)) ++vlog;
    if (vlog > 6) continue;
    uint32_t tab[2] = {0, 0};
    float delta = 0.f;
    for (int c = 0; c < n; ++c) {
      const float l = rintf(kc[c] / a);
      delta = std::max(delta, fabsf(kc[c] - a * l));
      tab[c >> 2] |= (static_cast<uint32_t>(static_cast<int>(l)) & 0xffu) << (8 * (c & 3));
    }
    if (!found || delta < ft->delta) *ft = FiltTab{tab[0], tab[1], a, delta, lm, vlog};
    found = true;
  }
  return found;
}

MipsLayout mips_layout(int32_t M, int d, int mbits, int k, int nsplit, const MipsPlan& pl) {
  const int ns = n_odd_subsets(mbits);
  const int64_t nu = 2 * (ns + 1);
  const int64_t chunks = (M + kRowsM - 1) / kRowsM;
  MipsLayout w{};
  int64_t off = 0;
  auto up = [](int64_t x) { return (x + 255) / 256 * 256; };
  w.aq = off;   off += up(chunks * nu * 64 * 16);
  w.rowc = off; off += up(chunks * kRowsM * 2 * 4);
  w.cs = off;   off += up(int64_t(M) * nsplit * k * 4);
  w.ci = off;   off += up(int64_t(M) * nsplit * k * 4);
  w.gth = off;  off += up(int64_t(M) * 4);
  w.pad = off;  // d < 128: padded queries, Pi and S (fp32)
  if (d < 128) off += up((int64_t(M) * 128 + 128 * 128 + 128) * 4);
  if (pl.filt) {
    const int64_t mq = int64_t(pl.ntile) * pl.qt * 16;
    w.qw = off;   off += up(int64_t(M) * 256 * 4);
    w.af = off;   off += up(mq / 16 * nu * 64 * 16);
    w.ciu = off;  off += up(mq * 4);
    w.cil = off;  off += up(mq * 4);
    w.cnt = off;  off += up(mq * 4);
    w.thr = off;  off += up(mq * 4);
    w.unit = off; off += up(mq * 4);
    w.left = off; off += up((1 + mq / 4) * 4);  // count, then query chunks
    w.claimed = off; off += up(mq / 4 * 4);
    w.mx = off;   off += up(mq * 16 * pl.P * 4);
    w.cand = off; off += up(mq * pl.cap * 4);
  }
  w.total = off;
  return w;
}

int64_t mips_scan_smem(int d, int mbits, int k) {
  const int rawd = (mbits + 1) * (d / 32), qw = 4 * (mbits <= 2 ? 4 : 2);
  return 2 * (int64_t(kMipsStep) * rawd * 4 + kMipsStep * 4) + int64_t(4) * qw * k * 8;
}

}  // namespace

namespace {

struct MipsArgs {
  const void* q;
  int q_dtype, M, d, mbits;
  const float* pi;
  const float* signs;
  float qjl_scale;
  const uint8_t* kst;
  const float* norms;
  int64_t N;
  int k;
  float* out_s;
  int64_t* out_i;
};

template <int MB, int PDW>
int launch_scan(const MipsArgs& a, void* ws, const MipsLayout& L, int nsplit, const int* left,
                const int* over, int cap, hipStream_t s) {
  const int chunks = (a.M + kRowsM - 1) / kRowsM;
  constexpr int qc = MipsCfg<MB, PDW>::QC;
  const int64_t vlen = ((a.N + nsplit - 1) / nsplit + kMipsStep - 1) / kMipsStep * kMipsStep;
  const int64_t qtiles = (chunks + 4 * qc - 1) / (4 * qc);
  const int64_t n_items = qtiles * nsplit;
  const int64_t smem = mips_scan_smem(a.d, a.mbits, a.k);
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, mips_scan<MB, PDW>, 256,
                                                   static_cast<size_t>(smem)) != hipSuccess)
    per_cu = 0;
  per_cu = std::max(per_cu, 1);
  const dim3 grid(
      static_cast<unsigned>(std::min<int64_t>(n_items, int64_t(per_cu) * qkv_num_cus())));
  if (smem > 65536)
    QKV_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&mips_scan<MB, PDW>),
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                static_cast<int>(smem)));
  hipLaunchKernelGGL((mips_scan<MB, PDW>), grid, dim3(256), static_cast<uint32_t>(smem), s,
                     at<qkv_v4i>(ws, L.aq), at<float>(ws, L.rowc), a.M, a.kst, a.norms, a.N,
                     nsplit, vlen, n_items, a.k, at<float>(ws, L.cs), at<int>(ws, L.ci),
                     at<uint32_t>(ws, L.gth), left);
  QKV_LAUNCHED();
  const int64_t msmem = int64_t(nsplit) * a.k * 8;
  if (msmem > 65536)
    QKV_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&mips_merge),
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                static_cast<int>(std::min<int64_t>(msmem, 160 * 1024))));
  QKV_REQUIRE(msmem <= 160 * 1024, "too many candidates per query");
  hipLaunchKernelGGL(mips_merge, dim3(a.M), dim3(64), static_cast<uint32_t>(msmem), s,
                     at<float>(ws, L.cs), at<int>(ws, L.ci), nsplit, a.k, a.out_s, a.out_i, over,
                     cap);
  QKV_LAUNCHED();
  return QKV_OK;
}

template <int MB, int PDW, int QT>
int launch_passes(const MipsArgs& a, void* ws, const MipsLayout& L, const MipsPlan& pl,
                  const FiltTab& ft, hipStream_t s) {
  const int tg = (pl.ntile + pl.wq - 1) / pl.wq;
  const dim3 grid(static_cast<unsigned>(tg * pl.pb));
  const int64_t ng = (a.N + 15) / 16, ng1 = (ng + pl.step - 1) / pl.step;
  int* cnt = at<int>(ws, L.cnt);
  float* thr = at<float>(ws, L.thr);
  float* mx = at<float>(ws, L.mx);
  hipLaunchKernelGGL((mips_pass<MB, PDW, QT, false>), grid, dim3(256), 0, s,
                     at<qkv_v4i>(ws, L.af), at<int>(ws, L.cil), thr, a.kst, a.norms, a.N,
                     pl.ntile, pl.wq, pl.pb, ng1, pl.step, a.M, ft, mx, cnt, at<int>(ws, L.cand),
                     pl.cap);
  QKV_LAUNCHED();
  const unsigned mq = static_cast<unsigned>(pl.ntile * QT * 16);
  const float* unit = at<float>(ws, L.unit);
  uint32_t* gth = at<uint32_t>(ws, L.gth);
  if (a.k <= 16)
    hipLaunchKernelGGL(mips_bound<1>, dim3(mq), dim3(256), 0, s, mx, 16 * pl.P, a.k, a.M, pl.step,
                       unit, at<int>(ws, L.ciu), at<int>(ws, L.cil), a.norms, a.N, thr, cnt,
                       pl.cap, gth);
  else
    hipLaunchKernelGGL(mips_bound<4>, dim3(mq), dim3(256), 0, s, mx, 16 * pl.P, a.k, a.M, pl.step,
                       unit, at<int>(ws, L.ciu), at<int>(ws, L.cil), a.norms, a.N, thr, cnt,
                       pl.cap, gth);
  QKV_LAUNCHED();
  hipLaunchKernelGGL((mips_pass<MB, PDW, QT, true>), grid, dim3(256), 0, s,
                     at<qkv_v4i>(ws, L.af), at<int>(ws, L.ciu), thr, a.kst, a.norms, a.N,
                     pl.ntile, pl.wq, pl.pb, ng, 1, a.M, ft, mx, cnt, at<int>(ws, L.cand), pl.cap);
  QKV_LAUNCHED();
  return QKV_OK;
}

template <int MB, int PDW>
int launch_filter(const MipsArgs& a, void* ws, const MipsLayout& L, const MipsPlan& pl,
                  const FiltTab& ft, hipStream_t s) {
  int* cnt = at<int>(ws, L.cnt);
  hipLaunchKernelGGL((mips_fprep<PDW>), dim3(static_cast<unsigned>(pl.ntile * pl.qt)),
                     dim3(256), 0, s, at<float>(ws, L.qw), at<float>(ws, L.rowc), a.M, ft,
                     at<uint32_t>(ws, L.af), at<int>(ws, L.ciu), at<int>(ws, L.cil), cnt, pl.cap,
                     at<float>(ws, L.unit), at<int>(ws, L.left), at<int>(ws, L.claimed));
  QKV_LAUNCHED();
  int st;
  switch (pl.qt) {
    case 1: st = launch_passes<MB, PDW, 1>(a, ws, L, pl, ft, s); break;
    case 2: st = launch_passes<MB, PDW, 2>(a, ws, L, pl, ft, s); break;
    case 4: st = launch_passes<MB, PDW, 4>(a, ws, L, pl, ft, s); break;
    default: st = launch_passes<MB, PDW, kFiltQT>(a, ws, L, pl, ft, s); break;
  }
  if (st != QKV_OK) return st;
  hipLaunchKernelGGL((mips_pick<MB, PDW>), dim3(a.M), dim3(256),
                     static_cast<uint32_t>(pl.cap * 8), s, at<qkv_v4i>(ws, L.aq),
                     at<float>(ws, L.rowc), a.kst, a.norms, a.k, cnt, at<int>(ws, L.cand), pl.cap,
                     at<int>(ws, L.left), at<int>(ws, L.claimed), a.out_s, a.out_i);
  QKV_LAUNCHED();
  return QKV_OK;
}

int mips_batch(const MipsArgs& a, void* ws, const Tables& tb, hipStream_t s) {
  MipsPlan pl = mips_plan(a.M, a.N, a.k);
  const int nsplit = mips_splits(a.M, a.N, a.mbits);
  const MipsLayout L = mips_layout(a.M, a.d, a.mbits, a.k, nsplit, pl);
  FiltTab ft{};
  if (pl.filt) pl.filt = filt_table(tb.kc, a.mbits, a.qjl_scale, &ft);
  const int chunks = (a.M + kRowsM - 1) / kRowsM;
  hipLaunchKernelGGL(mips_init, dim3((a.M + 255) / 256), dim3(256), 0, s,
                     at<uint32_t>(ws, L.gth), a.M);
  QLayers ql{};
  ql.q[0] = a.q;
  ql.pi[0] = a.pi;
  ql.signs[0] = a.signs;
  int qdt = a.q_dtype;
  if (a.d < 128) {
    float* qp = at<float>(ws, L.pad);
    float* pip = qp + int64_t(a.M) * 128;
    float* sp = pip + 128 * 128;
    const int64_t n = int64_t(a.M) * 128 + 128 * 128 + 128;
    hipLaunchKernelGGL(mips_pad, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, s,
                       a.q, a.q_dtype, a.M, a.d, a.pi, a.signs, qp, pip, sp);
    QKV_LAUNCHED();
    ql.q[0] = qp;
    qdt = QKV_F32;
    ql.pi[0] = pip;
    ql.signs[0] = sp;
  }
  // query operands: the decode prepare kernel with one "kv head" of M rows
  float* qw = pl.filt ? at<float>(ws, L.qw) : nullptr;
#define QKV_PREP(NPLV)                                                                           \
  hipLaunchKernelGGL((prepare_mfma<128, NPLV, false>), dim3(chunks), dim3(256),                  \
                     (prep_lds<128, NPLV, false>()), s, ql, 1, qdt, a.qjl_scale, a.M, 1, 1, a.M, \
                     chunks, tb, at<qkv_v4i>(ws, L.aq), at<float>(ws, L.rowc), qw)
  if (a.mbits == 1) QKV_PREP(2);
  else if (a.mbits == 2) QKV_PREP(3);
  else QKV_PREP(5);
#undef QKV_PREP
  QKV_LAUNCHED();
  switch (a.mbits * 10 + a.d / 32) {
#define QKV_MIPS(MBV, PDWV)                                                                \
  case MBV * 10 + PDWV:                                                                    \
    if (pl.filt) {                                                                         \
      const int st = launch_filter<MBV, PDWV>(a, ws, L, pl, ft, s);                        \
      if (st != QKV_OK) return st;                                                         \
    }                                                                                      \
    return launch_scan<MBV, PDWV>(a, ws, L, nsplit, pl.filt ? at<int>(ws, L.left) : nullptr, \
                                  pl.filt ? at<int>(ws, L.cnt) : nullptr, pl.cap, s);
    QKV_MIPS(1, 2) QKV_MIPS(1, 3) QKV_MIPS(1, 4)
    QKV_MIPS(2, 2) QKV_MIPS(2, 3) QKV_MIPS(2, 4)
    QKV_MIPS(3, 2) QKV_MIPS(3, 3) QKV_MIPS(3, 4)
#undef QKV_MIPS
  }
  return QKV_E_UNSUPPORTED;
}

// Workspace of M queries: the largest batch's (batches of filt_batch where the
// filter runs; its plan depends on the batch's size).
int64_t mips_ws_bytes(int32_t M, int32_t d, int32_t mbits, int32_t k, int64_t N, int32_t* batch) {
  auto bytes = [&](int32_t m) {
    return mips_layout(m, d, mbits, k, mips_splits(m, N, mbits), mips_plan(m, N, k)).total;
  };
  *batch = M;
  const int32_t most = filt_batch(k);
  if (M <= most || !mips_plan(M, N, k).filt) return bytes(M);
  *batch = most;
  const int32_t rest = M % most;
  return std::max(bytes(most), rest > 0 ? bytes(rest) : 0);
}

}  // namespace

extern "C" int64_t qkv_mips_workspace_bytes(int32_t M, int32_t d, int32_t mbits, int32_t k,
                                            int64_t N) {
  if (M <= 0 || !qkv_d_ok(d) || mbits < 1 || mbits > 3 || k <= 0 || N <= 0) return -1;
  int32_t batch = 0;
  return mips_ws_bytes(M, d, mbits, static_cast<int>(std::min<int64_t>(k, N)), N, &batch);
}

extern "C" int qkv_mips_search(const void* queries, int32_t q_dtype, int32_t M, int32_t d,
                               int32_t mbits, const float* pi, const float* signs,
                               const float* kcent_host, float qjl_scale, const uint8_t* kstore,
                               const float* norms, int64_t N, int32_t k, float* out_scores,
                               int64_t* out_indices, void* workspace, int64_t ws_bytes,
                               void* stream) {
  QKV_REQUIRE(qkv_dtype_ok(q_dtype), "unsupported query dtype %d", q_dtype);
  QKV_REQUIRE(N > 0, "Index is empty. Call add() first.");
  QKV_REQUIRE(N < (int64_t(1) << 31), "index holds at most 2^31 - 1 vectors");
  QKV_REQUIRE(M > 0 && k > 0, "invalid shape");
  if (!qkv_d_ok(d) || mbits < 1 || mbits > 3) {
    qkv_set_error("search runs on dim 64, 96 or 128 with 2..4-bit codes (got dim %d, %d MSE "
                  "bits)", d, mbits);
    return QKV_E_UNSUPPORTED;
  }
  k = static_cast<int32_t>(std::min<int64_t>(k, N));
  if (k > kMipsKMax) {
    qkv_set_error("search returns at most %d neighbours per query (asked %d)", kMipsKMax, k);
    return QKV_E_UNSUPPORTED;
  }
  QKV_REQUIRE(queries && pi && signs && kcent_host && kstore && norms && out_scores &&
                  out_indices && workspace,
              "null pointer");
  QKV_REQUIRE(qkv_aligned(pi, 16) && qkv_aligned(kstore, 4) && qkv_aligned(workspace, 256),
              "pi 16-B, store 4-B and workspace 256-B aligned");
  Tables tb{};
  for (int i = 0; i < (1 << mbits); ++i) tb.kc[i] = kcent_host[i];
  if (!walsh_odd(kcent_host, mbits, tb.kg, &tb.kconst)) {
    qkv_set_error("search needs a symmetric key codebook");
    return QKV_E_UNSUPPORTED;
  }
  tb.mfma_ok = 1;
  int32_t batch = 0;
  const int64_t need = mips_ws_bytes(M, d, mbits, k, N, &batch);
  QKV_REQUIRE(ws_bytes >= need, "workspace too small: %lld < %lld", (long long)ws_bytes,
              (long long)need);
  const int esize = q_dtype == QKV_F32 ? 4 : 2;
  for (int32_t m0 = 0; m0 < M; m0 += batch) {
    MipsArgs a{static_cast<const char*>(queries) + int64_t(m0) * d * esize,
               q_dtype, std::min(batch, M - m0), d, mbits, pi, signs, qjl_scale, kstore, norms, N,
               k, out_scores + int64_t(m0) * k, out_indices + int64_t(m0) * k};
    const int st = mips_batch(a, workspace, tb, static_cast<hipStream_t>(stream));
    if (st != QKV_OK) return st;
  }
  return QKV_OK;
}
