// Attention of many query rows (a prompt, a chunk of one) over the compressed
// store: the decode kernels' scores and values (see qkv_attention.hip), for
// G Q >= kPrefillMinRows rows per kv head.
//
// The decode kernels serve 4 query rows per workgroup and expand every K/V bit
// again for each; at 8192 rows (Q = T = 2048, 4 query heads per kv head) that is
// 1.05 ms where the dense f16 MFMA work is ~0.1 ms.  Here a workgroup of 8 waves
// takes 128 rows (ordered query-major so that causal tiles are narrow; two waves
// per 32 rows, one per 32-token half) and steps through 64 tokens at a time: the tile's codes become f16 levels
// in LDS once, and the products run on v_mfma_f32_32x32x16_f16.
//
// Precision: every f16 pair below is hi + lo, both rounded to nearest (24 bits).
//   * q~ = q Pi^T in three f16 products (hi hi + hi lo + lo hi), kept as hi + lo per
//     row; both meet every key level and the QJL weight;
//   * key levels: hi + lo, with a scale at which the QJL weight is an f16 value.
//     Codebooks of 1 magnitude, and of 2 at d >= 96, keep one f16 each: a scale s, by
//     search over the 1024 mantissas of the first level, brings the second to 5e-7
//     (1 magnitude: the QJL weight to 1e-7); what f16 then leaves of the QJL weight
//     (~1e-4) is put back by one multiplication of the QJL term's sums;
//   * softmax weights times |v| hi + lo, value levels likewise (1 magnitude: exact).
//   Sums are fp32 MFMA accumulators.  Relative errors against 64 bits, N(0, 1) queries
//   over 512 / 1500 keys: 0.5e-6 - 1.0e-6 / 0.7e-6 - 1.2e-6 (the decode kernels 1.1e-6 /
//   1.5e-6 at d = 64 with up to 2 MSE bits, 6e-6 - 10e-6 otherwise); logits up to 100 -
//   170: 1.1e-6 - 1.8e-6 (1.2e-6 - 23e-6); logits near 0, where the fp32 sums over the
//   keys set it: 2.2e-7 - 2.6e-7 (1.8e-7 - 5.5e-7).
//
// Layout.  The score product is S^T = K Q^T (rows tokens, columns query rows),
// so a lane owns one query row (lane & 31) and 16 of the 32 tokens: the softmax
// is per lane, and the accumulator registers, packed to f16, are already the B
// operand of O^T = V^T P^T.  The same chaining turns q Pi^T into the score
// operand and O into the un-rotation's.  C row rho holds token (or coordinate)
//   perm32(rho) = 8 (rho & 3) + 4 (rho >> 4) + 2 ((rho >> 2) & 1) + ((rho >> 3) & 1)
// of its 32: the 8 values of an operand register group then are the bits 2 p and
// 2 p + 1 of the four bytes of one plane word, which byte permutes turn into f16
// levels 4 at a time.
//
// Bounds: 56 MFMAs (32 cycles each) per 32 tokens x 32 rows at d = 128 with 3-bit
// keys and values; beside them ~250 VALU instructions of softmax and ~140 of
// expansion per wave.  One workgroup per CU (LDS: two 64-token buffers); of the two
// waves on a SIMD one expands before its products and the other after.  Measured,
// Q = T = 2048, 32 query and 8 kv heads, d = 128, causal, a pass among others: 142 -
// 151 us on three cards against 1056 - 1064 us on the decode kernel (164 - 167 us with
// a wait after each; matrix cores busy 37 %); 4.4 us per 64-token step.  On the way:
// 4 waves per workgroup, two workgroups per CU 447 us; 8 waves 284; q~'s |.| parts
// kept out of loop-invariant registers (spills, whose reloads wait for the loads in
// flight) 244; the halves' phases staggered 230; two QJL products instead of three
// 160; set-up loads issued together and its tiles shared by the wave pairs 140; f16
// pairs rounded to nearest and the QJL weight mended 142.  2-bit values: hi + lo
// levels 142 - 147 us, one f16 each 133.  A second accumulator chain for the QJL
// products changed nothing.
#include <math.h>

#include <algorithm>
#include <cmath>
#include <cstring>

#include "qkv_prefill.h"

namespace {

using namespace qkv_attn;

// (the HIP headers' min / max of 64-bit integers go through double)
__device__ __forceinline__ int64_t imin(int64_t a, int64_t b) { return a < b ? a : b; }
__device__ __forceinline__ int64_t imax(int64_t a, int64_t b) { return a > b ? a : b; }

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

constexpr int kTok = 32;      // tokens per wave and step
constexpr int kStep = 64;     // tokens per workgroup and step
constexpr int kThr = 512;
constexpr int kRowsWg = 128;
constexpr float kMinNorm = 0x1p-90f;  // |v| as the softmax reference sees it
constexpr int kMinExp = -123;         // of a row's scale: its inverse stays finite
constexpr float kHead = 8.f;  // the running maximum may lag by 2^8 before a rescale

// f16 levels of a codebook: bytes of the f16 values of codes 0 .. 7 (16-level
// codebooks: of the 8 positive magnitudes), hi and lo parts.
struct Levels {
  uint32_t hl[2], hh[2];  // hi part: low bytes, high bytes
  uint32_t ll[2], lh[2];  // lo part
  float inv;              // 1 / scale
};

struct PreArgs {
  const void* q;
  int q_dtype, q_vec;  // q_vec: 16-byte aligned
  int64_t t_stride, T;
  int Hq, Hkv, Q, R, G, BH, rt, n_splits;
  const float* pi;
  const float* signs;
  float alpha;   // qjl_scale times the key levels' scale
  float ae;      // alpha / f16(alpha) - 1 (0 unless PreCfg::AE)
  float c0;      // scale log2(e) / key levels' scale
  int causal;
  int64_t split_len;
  void* out;
  int out_dtype, out_vec;
  float* part_o;
  float* part_ml;
  Levels kl, vl;
};

__host__ __device__ constexpr int perm32(int rho) {
  return 8 * (rho & 3) + 4 * (rho >> 4) + 2 * ((rho >> 2) & 1) + ((rho >> 3) & 1);
}

__device__ __forceinline__ v16f mfma_h(v4u a, v4u b, v16f c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a),
                                                __builtin_bit_cast(v8h, b), c, 0, 0, 0);
}

typedef float v2f __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t pk(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f{a, b}), v2h));
}
// x as f16 hi + lo, both rounded to nearest (24 bits, no bias), two values per dword
__device__ __forceinline__ void split2(float a, float b, uint32_t& hi, uint32_t& lo) {
  hi = pk(a, b);
  const v2h h = __builtin_bit_cast(v2h, hi);
  lo = pk(a - static_cast<float>(h[0]), b - static_cast<float>(h[1]));
}

// Codes of bits 2 p (even) and 2 p + 1 (odd) of the four bytes of NB plane
// words already shifted right by 2 p: one code per byte.
template <int NB>
__device__ __forceinline__ void codes_of(const uint32_t* t, uint32_t& e, uint32_t& o) {
  e = t[0] & 0x01010101u;
  o = (t[0] >> 1) & 0x01010101u;
  if constexpr (NB >= 2) {
    e |= (t[1] << 1) & 0x02020202u;
    o |= t[1] & 0x02020202u;
  }
  if constexpr (NB >= 3) {
    e |= (t[2] << 2) & 0x04040404u;
    o |= (t[2] << 1) & 0x04040404u;
  }
}

// Four f16 levels (dwords 2 x, 2 x + 1 of out) of the four codes in sel.
__device__ __forceinline__ void levels4(uint32_t sel, v4u t, uint32_t flip, uint32_t& d0,
                                        uint32_t& d1) {
  const uint32_t lo = __builtin_amdgcn_perm(t[1], t[0], sel);
  const uint32_t hi = __builtin_amdgcn_perm(t[3], t[2], sel) ^ flip;
  d0 = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
  d1 = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
}

// The two operand halves (hi, and lo if LO) of a unit: 8 f16 from NB plane words.
// th, tl: the level tables (low bytes of codes 0-3, 4-7, high bytes) of each half.
template <int NB, bool LO>
__device__ __forceinline__ void expand_unit(const uint32_t* w, int p, v4u th, v4u tl, v4u& hi,
                                            v4u& lo) {
  uint32_t t[NB];
#pragma unroll
  for (int k = 0; k < NB; ++k) t[k] = w[k] >> (2 * p);
  uint32_t e, o, fe = 0, fo = 0;
  codes_of<NB < 3 ? NB : 3>(t, e, o);
  if constexpr (NB == 4) {  // magnitude index and sign of a 16-level code
    const uint32_t ne = ~t[3] & 0x01010101u, no = (~t[3] >> 1) & 0x01010101u;
    e ^= (ne << 3) - ne;
    o ^= (no << 3) - no;
    fe = ne << 7;
    fo = no << 7;
  }
  uint32_t a, b;
  levels4(e, th, fe, a, b);
  hi[0] = a;
  hi[1] = b;
  levels4(o, th, fo, a, b);
  hi[2] = a;
  hi[3] = b;
  if constexpr (LO) {
    levels4(e, tl, fe, a, b);
    lo[0] = a;
    lo[1] = b;
    levels4(o, tl, fo, a, b);
    lo[2] = a;
    lo[3] = b;
  }
}

// Whether key levels keep f16 hi + lo.  At d = 64 the decode kernel's int8 scores
// are good to ~1e-6 already, and a product more costs less than at d = 128.
__host__ __device__ constexpr bool key_lo(int d, int mb) { return mb >= 3 || (mb == 2 && d == 64); }

template <int CT, int MB, int VB>
struct PreCfg {
  static constexpr int D = 32 * CT;
  static constexpr int KK = 2 * CT;                 // 16-wide k steps of a d-long sum
  static constexpr bool KLO = key_lo(32 * CT, MB), VLO = VB >= 2;
  static constexpr bool AE = MB == 2 && !KLO;       // the QJL weight's f16 error is mended
  static constexpr int KPW = (KK + 3) / 4;          // units of K and of V per thread and step
  static constexpr int SEG = KK * 1024;             // bytes of one operand image
  static constexpr int OFF_S = SEG * (KLO ? 2 : 1), OFF_V = OFF_S + SEG;
  static constexpr int OFF_N = OFF_V + SEG * (VLO ? 2 : 1);
  static constexpr int BUF = OFF_N + 512;           // scaled key norms, |v|, log2 |v| (32 each)
  static constexpr int IMG = CT * KK * 1024;        // one f16 half of Pi
  // two images per buffer (one per token half), two buffers where they fit
  static constexpr int NBUF = 4 * BUF + KK * 64 + 64 <= 160 * 1024 ? 2 : 1;
  static constexpr int MERGE = 4 * 64 * (16 * CT + 2) * 4;
  static constexpr int MAIN = 2 * NBUF * BUF;
  // beside Pi's halves, four row groups' q~ (then O) operands, hi and lo, and scales
  static constexpr int OPND = KK * 2 * 1024, EDGE = 2 * IMG + 4 * OPND + 4 * 256;
  static constexpr int BASE = MAIN > EDGE ? (MAIN > MERGE ? MAIN : MERGE)
                                          : (EDGE > MERGE ? EDGE : MERGE);
  // eps and sg (16 bytes per k step and lane half each), the four level tables
  static constexpr int CST = KK * 64 + 64;
  static constexpr int LDS = BASE + CST;
};

// Pi (scaled by 64) as f16 hi + lo A operands in LDS.  TR: of Pi^T.
// All of a thread's loads are issued before the first is converted.
template <int CT, bool TR>
__device__ __forceinline__ void stage_pi(const float* __restrict__ pi, uint8_t* img, int tid) {
  constexpr int D = 32 * CT, KK = 2 * CT, IMG = CT * KK * 1024;
  constexpr int NU = CT * KK * 64, NX = (NU + kThr - 1) / kThr;
  float x[NX][8];
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    const int u = min(tid + kThr * i, NU - 1);
    const int m = u & 31, h = (u >> 5) & 1, kk = (u >> 6) % KK, ct = (u >> 6) / KK;
    if constexpr (!TR) {  // row perm32(m) of tile ct, columns 16 kk + 8 h ..
      const float* src = pi + (32 * ct + perm32(m)) * D + 16 * kk + 8 * h;
      *reinterpret_cast<float4*>(x[i]) = *reinterpret_cast<const float4*>(src);
      *reinterpret_cast<float4*>(x[i] + 4) = *reinterpret_cast<const float4*>(src + 4);
    } else {  // column 32 ct + m, the rows that O's accumulators hold in this order
#pragma unroll
      for (int j = 0; j < 8; ++j)
        x[i][j] = pi[(16 * kk + 8 * (j >> 2) + 4 * h + (j & 3)) * D + 32 * ct + m];
    }
  }
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    const int u = min(tid + kThr * i, NU - 1);  // (the last unit: the same bytes again)
    v4u hi, lo;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t a, b;
      split2(64.f * x[i][2 * j], 64.f * x[i][2 * j + 1], a, b);
      hi[j] = a;
      lo[j] = b;
    }
    *reinterpret_cast<v4u*>(img + u * 16) = hi;
    *reinterpret_cast<v4u*>(img + IMG + u * 16) = lo;
  }
}

template <int CT, int MB, int VB, bool PAGED>
__global__ __launch_bounds__(kThr, 2) void prefill(PreArgs A, KVLayers kv) {
  using C = PreCfg<CT, MB, VB>;
  constexpr int D = C::D, KK = C::KK, KPW = C::KPW;
  extern __shared__ __align__(16) uint8_t lds[];
  // constants that the steps read from LDS instead of holding registers
  v4u* eps = reinterpret_cast<v4u*>(lds + C::BASE);  // [KK][2 halves] QJL residuals
  v4u* sgs = eps + KK * 2;                           // [KK][2 halves] -f16(alpha S)
  v4u* tabs = sgs + KK * 2;                          // key hi, lo, value hi, lo

  const int tid = threadIdx.x, lane = tid & 63;
  // waves 0-3: rows 32 wave .. of the tile over the first 32 tokens of each step,
  // waves 4-7 the same rows over the second 32 (merged at the end)
  const int wave8 = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave = wave8 & 3, th = wave8 >> 2;
  const int n = lane & 31, h = lane >> 5;
  // workgroup -> (row tile, split, sequence, kv head), long causal row tiles first
  const int bhs = A.BH * A.n_splits;
  const int id = blockIdx.x, rt = A.rt - 1 - id / bhs, rem = id % bhs;
  const int split = rem / A.BH, bh = rem % A.BH;
  const int b = bh / A.Hkv, hkv = bh - b * A.Hkv;
  const SeqRange sr = seq_range(kv, b, A.T);

  // this lane's query row, query-major: rr = qi G + g
  const int rr = min(rt * kRowsWg + wave * 32 + n, A.R - 1);
  const int qi = rr / A.G, g = rr - qi * A.G;
  const bool live = rt * kRowsWg + wave * 32 + n < A.R;

  // ---- q~ = q Pi^T as the score operand, f16 hi + lo
  uint8_t* const opnd = lds + 2 * C::IMG + wave * C::OPND + lane * 16;  // [kk][hi, lo]
  v4u qhi[KK], qlo[KK];
  float fr;  // 2^e: q~ = 2^e (qhi + qlo)
  {
    const int64_t q0 = ((int64_t(b) * A.Hq + hkv * A.G + g) * A.Q + qi) * D + 8 * h;
    float x[KK][8];
    if (A.q_vec && A.q_dtype == QKV_F32) {
      const float4* src = reinterpret_cast<const float4*>(static_cast<const float*>(A.q) + q0);
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        *reinterpret_cast<float4*>(x[kk]) = src[4 * kk];
        *reinterpret_cast<float4*>(x[kk] + 4) = src[4 * kk + 1];
      }
    } else if (A.q_vec) {
      const v4u* src = reinterpret_cast<const v4u*>(static_cast<const uint16_t*>(A.q) + q0);
      v4u raw[KK];
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) raw[kk] = src[2 * kk];
      if (A.q_dtype == QKV_BF16) {
#pragma unroll
        for (int i = 0; i < 8 * KK; ++i)
          x[i >> 3][i & 7] =
              qkv_bf16_to_f32(static_cast<uint16_t>(raw[i >> 3][(i & 7) >> 1] >> (16 * (i & 1))));
      } else {
#pragma unroll
        for (int i = 0; i < 8 * KK; ++i)
          x[i >> 3][i & 7] = static_cast<float>(__builtin_bit_cast(
              _Float16, static_cast<uint16_t>(raw[i >> 3][(i & 7) >> 1] >> (16 * (i & 1)))));
      }
    } else {  // (rolled, through LDS: unrolled it was near half of the kernel's code)
      float* const t = reinterpret_cast<float*>(lds + 2 * C::IMG + wave * C::OPND) + lane;
#pragma unroll 1
      for (int i = 0; i < 8 * KK; ++i)
        t[64 * i] = qkv_load(A.q, q0 + 16 * (i >> 3) + (i & 7), A.q_dtype);
#pragma unroll
      for (int i = 0; i < 8 * KK; ++i) x[i >> 3][i & 7] = t[64 * i];
    }
    stage_pi<CT, false>(A.pi, lds, tid);
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < 8 * KK; ++i) amax = fmaxf(amax, fabsf(x[i >> 3][i & 7]));
    amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
    int ex = 0;
    if (amax > 0.f && amax < INFINITY) frexpf(amax, &ex);
    ex = max(ex, kMinExp);
    const float up = ldexpf(1.f, 3 - ex);  // the row's largest into [4, 8)
    fr = ldexpf(1.f, ex - 3);
    v4u xh[KK], xl[KK];
#pragma unroll
    for (int i = 0; i < 4 * KK; ++i) {
      uint32_t a, c;
      split2(x[i >> 2][2 * (i & 3)] * up, x[i >> 2][2 * (i & 3) + 1] * up, a, c);
      xh[i >> 2][i & 3] = a;
      xl[i >> 2][i & 3] = c;
    }
    __syncthreads();
    // the two waves of a row group take every other tile and share them through LDS
    // (rolled: straight-line code runs once and waits on its own fetches)
#pragma unroll 1
    for (int ct = th; ct < CT; ct += 2) {
      v16f acc = {};
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        const uint8_t* src = lds + ((ct * KK + kk) * 64 + lane) * 16;
        const v4u ph = *reinterpret_cast<const v4u*>(src);
        const v4u pl = *reinterpret_cast<const v4u*>(src + C::IMG);
        acc = mfma_h(ph, xh[kk], acc);
        acc = mfma_h(ph, xl[kk], acc);
        acc = mfma_h(pl, xh[kk], acc);
      }
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        v4u hi, lo;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          uint32_t a, c;
          split2(acc[8 * ks + 2 * j] * 0.015625f, acc[8 * ks + 2 * j + 1] * 0.015625f, a, c);
          hi[j] = a;
          lo[j] = c;
        }
        *reinterpret_cast<v4u*>(opnd + (2 * ct + ks) * 2048) = hi;
        *reinterpret_cast<v4u*>(opnd + (2 * ct + ks) * 2048 + 1024) = lo;
      }
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      qhi[kk] = *reinterpret_cast<const v4u*>(opnd + kk * 2048);
      qlo[kk] = *reinterpret_cast<const v4u*>(opnd + kk * 2048 + 1024);
    }
    __syncthreads();
  }

  // QJL operand constants of this thread's K units: f16(alpha S_j), negated (a set
  // bit flips the sign back); eps: what f16 and (1 + ae) leave of them.  Signs other
  // than +-1 (more than 1e-6 of them left) take a third QJL product.
  const int w0 = (wave * KPW) >> 1;  // this thread's plane word, for K and for V
  const bool work = wave * KPW < KK;
  bool res = false;
#pragma unroll
  for (int x = 0; x < KPW; ++x) {
    const int kk = wave * KPW + x;
    if (kk < KK) {
      v4u e4, s4;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float a2[2], e2[2];
#pragma unroll
        for (int y = 0; y < 2; ++y) {
          const int jj = 2 * j + y;
          const int c = 32 * (kk >> 1) + 8 * (jj & 3) + 2 * (2 * (kk & 1) + h) + (jj >> 2);
          a2[y] = A.alpha * A.signs[c];
          const float hf = static_cast<float>(static_cast<_Float16>(a2[y]));
          e2[y] = a2[y] - fmaf(hf, A.ae, hf);
          res |= fabsf(e2[y]) > 1e-6f * fabsf(a2[y]);
          a2[y] = -hf;
        }
        s4[j] = pk(a2[0], a2[1]);
        e4[j] = pk(e2[0], e2[1]);
      }
      if (n == 0) {
        eps[kk * 2 + h] = e4;
        sgs[kk * 2 + h] = s4;
      }
    }
  }
  if (tid == 0) {
    tabs[0] = v4u{A.kl.hl[0], A.kl.hl[1], A.kl.hh[0], A.kl.hh[1]};
    tabs[1] = v4u{A.kl.ll[0], A.kl.ll[1], A.kl.lh[0], A.kl.lh[1]};
    tabs[2] = v4u{A.vl.hl[0], A.vl.hl[1], A.vl.hh[0], A.vl.hh[1]};
    tabs[3] = v4u{A.vl.ll[0], A.vl.ll[1], A.vl.lh[0], A.vl.lh[1]};
  }
  const bool third = __syncthreads_or(res);

  // ---- the split's steps; token positions relative to its first
  const int64_t s0 = split * A.split_len, s1 = imin(A.T, s0 + A.split_len);
  const int64_t t_lo = imax(sr.lo, s0) & ~int64_t(kStep - 1);
  // last key that query qx attends to, relative to t_lo
  auto limit = [&](int qx) {
    int64_t x = sr.hi - 1;
    if (A.causal) x = imin(x, sr.cpos - A.Q + qx);
    return static_cast<int>(imax(imin(x, s1 - 1) - t_lo, -1));
  };
  const int lo_rel = static_cast<int>(imin(imax(sr.lo - t_lo, 0), 1 << 30));
  const int lim = limit(qi);
  const int r_wave = rt * kRowsWg + wave * 32;
  const int wg_lim = limit((min(rt * kRowsWg + kRowsWg, A.R) - 1) / A.G);
  const int nst = wg_lim < lo_rel ? 0 : wg_lim / kStep + 1;
  // the wave's rows attend to all keys up to wave_lim, to none past wave_end
  const int wave_lim = limit(min(r_wave, A.R - 1) / A.G);
  const int wave_end = limit(min(r_wave + 31, A.R - 1) / A.G);

  // raw words of one step: this thread's K row words, V words, a norm
  struct Raw {
    uint32_t k[MB + 1], v[VB];
    float nm;
  };
  constexpr int RB = (MB + 1) * CT;  // row dwords
  const uint32_t* kst = reinterpret_cast<const uint32_t*>(kv.kst[0]);
  const uint32_t* vst = kv.vst[0];
  auto row_of = [&](int64_t t) -> int64_t {  // store row of the 32-token tile at t (-1: no page)
    if constexpr (PAGED) {
      const int pg = kv.ptab[int64_t(b) * kv.pmax + (t >> kv.plg)];
      if (pg < 0 || pg >= kv.npages) return -1;
      return ((int64_t(pg) * A.Hkv + hkv) << kv.plg) + (t & ((int64_t(1) << kv.plg) - 1));
    } else {
      return int64_t(bh) * A.t_stride + t;
    }
  };
  const uint32_t kofs = (perm32(n) * RB + w0) * 4, vofs = (32 * w0 + n) * 4;
  auto load = [&](int st) {
    Raw r;
    const int64_t t = t_lo + int64_t(min(st, nst - 1)) * kStep + kTok * th;
    const int64_t row = imax(row_of(t), 0);
    if (work) {  // (32-bit lane offsets from wave-uniform bases)
      const uint8_t* src = reinterpret_cast<const uint8_t*>(kst + row * RB);
#pragma unroll
      for (int k = 0; k <= MB; ++k)
        r.k[k] = *reinterpret_cast<const uint32_t*>(src + (kofs + 4 * CT * k));
      const uint8_t* vs = reinterpret_cast<const uint8_t*>(vst + (row >> 5) * (VB * D));
#pragma unroll
      for (int k = 0; k < VB; ++k)
        r.v[k] = *reinterpret_cast<const uint32_t*>(vs + (vofs + 4 * D * k));
    }
    r.nm = 0.f;
    // (0 outside the key range: its slots may hold anything)
    if (wave < 2 && h == 0 && t + perm32(n) >= sr.lo && t + perm32(n) < sr.hi)
      r.nm = (wave == 0 ? kv.knorm[0] : kv.vnorm[0])[row + perm32(n)];
    return r;
  };
  auto store = [&](const Raw& r, uint8_t* buf) {
    if (work) {
      const v4u t0 = tabs[0], t1 = tabs[1], t2 = tabs[2], t3 = tabs[3];
#pragma unroll
      for (int x = 0; x < KPW; ++x) {
        const int kk = wave * KPW + x;
        if (kk < KK) {
          const int p = 2 * (kk & 1) + h;
          const v4u sg = sgs[kk * 2 + h];
          v4u hi, lo;
          expand_unit<MB, C::KLO>(r.k, p, t0, t1, hi, lo);
          uint8_t* at = buf + kk * 1024 + lane * 16;
          *reinterpret_cast<v4u*>(at) = hi;
          if constexpr (C::KLO) *reinterpret_cast<v4u*>(at + C::SEG) = lo;
          const uint32_t q = r.k[MB] >> (2 * p);
          const uint32_t ye = (q << 7) & 0x80808080u, yo = (q << 6) & 0x80808080u;
          v4u s4;
          s4[0] = __builtin_amdgcn_perm(0u, ye, 0x010c000cu) ^ sg[0];
          s4[1] = __builtin_amdgcn_perm(0u, ye, 0x030c020cu) ^ sg[1];
          s4[2] = __builtin_amdgcn_perm(0u, yo, 0x010c000cu) ^ sg[2];
          s4[3] = __builtin_amdgcn_perm(0u, yo, 0x030c020cu) ^ sg[3];
          *reinterpret_cast<v4u*>(at + C::OFF_S) = s4;
          expand_unit<VB, C::VLO>(r.v, p, t2, t3, hi, lo);
          *reinterpret_cast<v4u*>(at + C::OFF_V) = hi;
          if constexpr (C::VLO) *reinterpret_cast<v4u*>(at + C::OFF_V + C::SEG) = lo;
        }
      }
    }
    float* nm = reinterpret_cast<float*>(buf + C::OFF_N);
    if (wave < 2) {
      if (h == 0) {
        // a value norm that is not finite: weight 0 times 0 where the slot is masked, a
        // reference of infinity (NaN out) for the rows that see it
        float nv = wave == 0 ? r.nm * A.c0 : r.nm;
        // log2, from 2^-90 up: a row of zero norms alone keeps finite weights
        float lg = __builtin_amdgcn_logf(fmaxf(fabsf(nv), kMinNorm));
        if (__builtin_expect(wave == 1 && !(fabsf(nv) < INFINITY), 0)) {
          nv = 0.f;
          lg = INFINITY;
        }
        nm[32 * wave + n] = nv;
        if (wave == 1) nm[64 + n] = lg;
      }
    }
  };

  v16f O[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) O[ct] = v16f{};
  float l = 0.f, mref = kMFloor;

  uint8_t* const own = lds + th * C::BUF;  // this token half's images
  if (nst > 0) {
    Raw raw = load(0);
    if constexpr (C::NBUF == 2) {
      store(raw, own);
      raw = load(1);
    }
    for (int st = 0; st < nst; ++st) {
      uint8_t* buf = own + (C::NBUF == 2 ? (st & 1) * 2 * C::BUF : 0);
      __syncthreads();
      // the next step's images: the first half's waves expand before their products,
      // the second half's after them, so that of the two waves on a SIMD (w, w + 4)
      // one has VALU work while the other has MFMAs
      auto next = [&]() {
        if (st + 1 < nst) {
          store(raw, own + ((st + 1) & 1) * 2 * C::BUF);
          raw = load(st + 2);
        }
      };
      if constexpr (C::NBUF == 2) {
        if (th == 0) next();
      } else {
        store(raw, buf);
        raw = load(st + 1);
        __syncthreads();
      }
      const int t0 = st * kStep + kTok * th;
      if (t0 <= wave_end && !(PAGED && row_of(t_lo + t0) < 0)) {
      const float* nm = reinterpret_cast<const float*>(buf + C::OFF_N);

      // scores: rows tokens, this lane's column its query row
      v16f S = {};
      const uint8_t* const at = buf + lane * 16;
      auto op = [&](int ofs, int kk) {
        return *reinterpret_cast<const v4u*>(at + ofs + kk * 1024);
      };
      // |q~| = |hi| + lo sign(hi)  (opaque: as loop invariants the two would take 64
      // registers and spill)
      auto magnitudes = [&](int kk, v4u& wh, v4u& wl) {
        asm volatile("" : "+v"(qhi[kk]));
        wh = qhi[kk] & 0x7fff7fffu;
        wl = qlo[kk] ^ (qhi[kk] & 0x80008000u);
      };
      if constexpr (C::AE) {  // the whole QJL term first, to mend its weight
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
          const v4u sa = op(C::OFF_S, kk);
          v4u wh, wl;
          magnitudes(kk, wh, wl);
          S = mfma_h(sa, wh, S);
          S = mfma_h(sa, wl, S);
        }
        // (as S (1 + ae) the schedule around it was 2.4 % slower)
#pragma unroll
        for (int r = 0; r < 16; ++r) S[r] = fmaf(S[r], A.ae, S[r]);
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
          const v4u ka = op(0, kk);
          S = mfma_h(ka, qhi[kk], S);
          S = mfma_h(ka, qlo[kk], S);
        }
      } else {
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
          const v4u ka = op(0, kk), sa = op(C::OFF_S, kk);
          v4u wh, wl;
          magnitudes(kk, wh, wl);
          S = mfma_h(ka, qhi[kk], S);
          S = mfma_h(sa, wh, S);
          S = mfma_h(ka, qlo[kk], S);
          S = mfma_h(sa, wl, S);
          if constexpr (C::KLO) S = mfma_h(op(C::SEG, kk), qhi[kk], S);
        }
      }
      if (third) {
#pragma unroll 1
        for (int kk = 0; kk < KK; ++kk) {
          const uint8_t* at = buf + kk * 1024 + lane * 16;
          const v4u sa = *reinterpret_cast<const v4u*>(at + C::OFF_S);
          // +-eps: the operand's sign relative to f16(alpha S) is the QJL bit
          v4u e4 = eps[kk * 2 + h], q4;
#pragma unroll
          for (int x = 0; x < KK; ++x)
            if (x == kk) q4 = qhi[x];
          v4u a4;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            float s2[2];
#pragma unroll
            for (int y = 0; y < 2; ++y) {
              const int jj = 2 * j + y;
              const int c = 32 * (kk >> 1) + 8 * (jj & 3) + 2 * (2 * (kk & 1) + h) + (jj >> 2);
              const uint32_t sbit = (sa[j] >> (16 * y + 15)) & 1u;
              const uint32_t rbit = __float_as_uint(A.alpha * A.signs[c]) >> 31;
              s2[y] = sbit == rbit ? 0.f : -0.f;
            }
            a4[j] = e4[j] ^ pk(s2[0], s2[1]);
          }
          S = mfma_h(a4, q4 & 0x7fff7fffu, S);
        }
      }
      // softmax of this lane's row over its 16 tokens
      float x[16];
      const bool full = t0 >= lo_rel && t0 + kTok - 1 <= wave_lim;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float nk = nm[8 * (r >> 2) + 4 * h + (r & 3)];
        x[r] = S[r] * nk;
      }
      if (!full) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int t = t0 + 8 * (r & 3) + 4 * (r >> 3) + 2 * h + ((r >> 2) & 1);
          if (t > lim || t < lo_rel) x[r] = -INFINITY;
        }
      }
      // reference: the running maximum of score + log2 |v| (not of the score alone,
      // so that the f16 weights p |v| keep their bits where a large score meets a
      // small |v|), lagging by 2^8 at most
      float xm = -INFINITY;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        xm = fmaxf(xm, fmaf(x[r], fr, nm[64 + 8 * (r >> 2) + 4 * h + (r & 3)]));
      xm = fmaxf(xm, __shfl_xor(xm, 32, 64));
      if (__builtin_amdgcn_ballot_w64(xm > mref + kHead)) {
        const float mn = fmaxf(mref, xm);
        const float f = exp2f(mref - mn);
        mref = mn;
        l *= f;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) O[ct] *= f;
      }
      const float M = mref - 6.f;
      v4u ph[2], pl[2];
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const float p0 = __builtin_amdgcn_exp2f(fmaf(x[r], fr, -M));
        const float p1 = __builtin_amdgcn_exp2f(fmaf(x[r + 1], fr, -M));
        l += p0 + p1;
        const float* nv = nm + 32 + 8 * (r >> 2) + 4 * h + (r & 3);
        uint32_t a, c;
        split2(p0 * nv[0], p1 * nv[1], a, c);
        ph[r >> 3][(r & 7) >> 1] = a;
        pl[r >> 3][(r & 7) >> 1] = c;
      }
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          const uint8_t* at = buf + C::OFF_V + (2 * ct + ks) * 1024 + lane * 16;
          const v4u va = *reinterpret_cast<const v4u*>(at);
          O[ct] = mfma_h(va, ph[ks], O[ct]);
          O[ct] = mfma_h(va, pl[ks], O[ct]);
          if constexpr (C::VLO)
            O[ct] = mfma_h(*reinterpret_cast<const v4u*>(at + C::SEG), ph[ks], O[ct]);
        }
      }
      if constexpr (C::NBUF == 2) {
        if (th == 1) next();
      }
    }
  }
  l += __shfl_xor(l, 32, 64);

  // ---- merge the token halves into waves 0-3
  float* mg = reinterpret_cast<float*>(lds) + wave * 64 * (16 * CT + 2) + lane;
  __syncthreads();
  if (th == 1) {
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int r = 0; r < 16; ++r) mg[64 * (16 * ct + r)] = O[ct][r];
    mg[64 * 16 * CT] = mref;
    mg[64 * (16 * CT + 1)] = l;
  }
  __syncthreads();
  if (th == 0) {
    const float m2 = mg[64 * 16 * CT], l2 = mg[64 * (16 * CT + 1)];
    const float mn = fmaxf(mref, m2), f1 = exp2f(mref - mn), f2 = exp2f(m2 - mn);
    mref = mn;
    l = l * f1 + l2 * f2;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int r = 0; r < 16; ++r) O[ct][r] = O[ct][r] * f1 + mg[64 * (16 * ct + r)] * f2;
  }

  // ---- partials of the split: O~ / l (rotated) and (m, l) with the weights' sum in m,
  // so that l is 1 as nearly as m's rounding allows: mref holds log2 |v|, and the raw l
  // of large norms (~64 / |v|) would meet the merge's floor of 1e-8
  if (A.n_splits > 1) {
    const int64_t row = (int64_t(split) * A.BH + bh) * A.R + int64_t(g) * A.Q + qi;
    const float e2 = mref - 6.f;
    const float m = (e2 + __builtin_amdgcn_logf(l)) * 0.69314718055994531f;
    // 2^(e2 - m log2 e), log2 e in two parts: 1 / l
    const float f =
        __builtin_amdgcn_exp2f(fmaf(-m, 1.92596299e-8f, fmaf(-m, 1.44269502f, e2)));
    const float fo = l > 0.f ? f * A.vl.inv : 0.f;
    if (live && th == 0) {
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int r = 0; r < 16; r += 4)
          *reinterpret_cast<float4*>(A.part_o + row * D + 32 * ct + 8 * (r >> 2) + 4 * h) =
              make_float4(O[ct][r] * fo, O[ct][r + 1] * fo, O[ct][r + 2] * fo, O[ct][r + 3] * fo);
      if (h == 0) {
        // (l NaN: no reference that the merge would leave out)
        A.part_ml[row * 2] = l > 0.f ? m : l == 0.f ? -INFINITY : 0.f;
        A.part_ml[row * 2 + 1] = l > 0.f ? l * f : l;
      }
    }
    return;
  }

  // ---- out = (O~ / l) Pi: operands by waves 0-3, tiles by both waves of a row group
  float* const rsc = reinterpret_cast<float*>(lds + 2 * C::IMG + 4 * C::OPND) + wave * 64 + lane;
  __syncthreads();
  stage_pi<CT, true>(A.pi, lds, tid);
  if (th == 0) {
    const float inv = l > 0.f ? A.vl.inv / l : 0.f;
    float amax = 0.f;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      O[ct] *= inv;
#pragma unroll
      for (int r = 0; r < 16; ++r) amax = fmaxf(amax, fabsf(O[ct][r]));
    }
    amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
    int ex = 0;
    if (amax > 0.f && amax < INFINITY) frexpf(amax, &ex);
    ex = max(ex, kMinExp);
    const float up = ldexpf(1.f, 3 - ex);
    *rsc = ldexpf(1.f, ex - 9);  // (Pi is scaled by 64)
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      v4u hi, lo;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t a, c;
        const int r = 8 * (kk & 1) + 2 * j;
        split2(O[kk >> 1][r] * up, O[kk >> 1][r + 1] * up, a, c);
        hi[j] = a;
        lo[j] = c;
      }
      *reinterpret_cast<v4u*>(opnd + kk * 2048) = hi;
      *reinterpret_cast<v4u*>(opnd + kk * 2048 + 1024) = lo;
    }
  }
  __syncthreads();
  const float down = *rsc;
  const int64_t qrow = (int64_t(b) * A.Hq + hkv * A.G + g) * A.Q + qi;
#pragma unroll 1
  for (int kt = th; kt < CT; kt += 2) {
    v16f acc = {};
#pragma unroll
    for (int cc = 0; cc < KK; ++cc) {
      const uint8_t* src = lds + ((kt * KK + cc) * 64 + lane) * 16;
      const v4u ph = *reinterpret_cast<const v4u*>(src);
      const v4u pl = *reinterpret_cast<const v4u*>(src + C::IMG);
      const v4u oh = *reinterpret_cast<const v4u*>(opnd + cc * 2048);
      const v4u ol = *reinterpret_cast<const v4u*>(opnd + cc * 2048 + 1024);
      acc = mfma_h(ph, oh, acc);
      acc = mfma_h(ph, ol, acc);
      acc = mfma_h(pl, oh, acc);
    }
    if (!live) continue;
    const int64_t at = qrow * D + 32 * kt + 4 * h;  // quads of 4 columns, 8 apart
    if (A.out_vec && A.out_dtype == QKV_F32) {
#pragma unroll
      for (int r = 0; r < 16; r += 4)
        *reinterpret_cast<float4*>(static_cast<float*>(A.out) + at + 2 * r) =
            make_float4(acc[r] * down, acc[r + 1] * down, acc[r + 2] * down, acc[r + 3] * down);
    } else if (A.out_vec) {
#pragma unroll
      for (int r = 0; r < 16; r += 4) {
        uint16_t u[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          u[j] = A.out_dtype == QKV_BF16
                     ? qkv_f32_to_bf16(acc[r + j] * down)
                     : __builtin_bit_cast(uint16_t, static_cast<_Float16>(acc[r + j] * down));
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(A.out) + at + 2 * r) =
            make_uint2(u[0] | uint32_t(u[1]) << 16, u[2] | uint32_t(u[3]) << 16);
      }
    } else {
#pragma unroll 1
      for (int r = 0; r < 16; ++r) {
        float v = acc[0];
#pragma unroll
        for (int y = 1; y < 16; ++y) v = y == r ? acc[y] : v;
        qkv_store(A.out, at + 2 * (r & ~3) + (r & 3), v * down, A.out_dtype);
      }
    }
  }
}

// ------------------------------------------------------------ host

float f16_round(float x) { return static_cast<float>(static_cast<_Float16>(x)); }

// Scale for the positive magnitudes mag[0 .. n) (n <= 2) and, if set, the QJL
// weight (whose error weighs qw): the first becomes an f16 value exactly, with
// the mantissa that leaves the others closest to f16 values.
float best_scale(const float* mag, int n, float alpha, float qw) {
  float best = 0.f, err = 1e30f;
  for (int m = 1024; m < 2048; ++m) {
    const float s = (m / 1024.f) / mag[0];
    float e = 0.f;
    for (int i = 0; i < n; ++i) e = std::max(e, fabsf(f16_round(mag[i] * s) / (mag[i] * s) - 1.f));
    if (alpha > 0.f) e = std::max(e, qw * fabsf(f16_round(alpha * s) / (alpha * s) - 1.f));
    if (e < err) {
      err = e;
      best = s;
    }
  }
  return best;
}

// Levels of a symmetric codebook at scale s.
void fill_levels(const float* cent, int bits, float s, Levels* lv) {
  memset(lv, 0, sizeof(*lv));
  const int n = std::min(8, 1 << bits), first = bits == 4 ? 8 : 0;
  for (int c = 0; c < n; ++c) {
    const float x = cent[first + c] * s;
    const _Float16 h = static_cast<_Float16>(x);
    const _Float16 l = static_cast<_Float16>(x - static_cast<float>(h));
    uint16_t hb, lb;
    memcpy(&hb, &h, 2);
    memcpy(&lb, &l, 2);
    const int sh = 8 * (c & 3);
    lv->hl[c >> 2] |= static_cast<uint32_t>(hb & 0xff) << sh;
    lv->hh[c >> 2] |= static_cast<uint32_t>(hb >> 8) << sh;
    lv->ll[c >> 2] |= static_cast<uint32_t>(lb & 0xff) << sh;
    lv->lh[c >> 2] |= static_cast<uint32_t>(lb >> 8) << sh;
  }
  lv->inv = 1.f / s;
}

struct PreLevels {
  Levels kl, vl;
  float ks;
  bool fits;  // levels and QJL weight inside f16's range at their scales, single levels exact
};

// Largest positive magnitude of a symmetric codebook (its upper half, in any order).
float top_level(const float* cent, int bits) {
  float top = 0.f;
  for (int c = 1 << (bits - 1); c < 1 << bits; ++c) top = std::max(top, cent[c]);
  return top;
}

// The levels of a (key, value) codebook pair: a pure function of its arguments,
// 1024 candidate scales per codebook (~10 us), kept for the last pair per thread.
const PreLevels& levels_for(int d, int kbits, int vbits, const float* kc, const float* vc,
                            float alpha) {
  struct Memo {
    int d = 0, kbits = 0, vbits = 0;
    float alpha = 0.f, kc[16], vc[16];
    PreLevels lv;
  };
  static thread_local Memo m;
  const size_t nk = sizeof(float) << kbits, nv = sizeof(float) << vbits;
  if (m.d == d && m.kbits == kbits && m.vbits == vbits && m.alpha == alpha && !memcmp(m.kc, kc, nk) &&
      !memcmp(m.vc, vc, nv))
    return m.lv;
  m.d = d;
  m.kbits = kbits;
  m.vbits = vbits;
  m.alpha = alpha;
  memcpy(m.kc, kc, nk);
  memcpy(m.vc, vc, nv);
  const float* kp = kc + (1 << (kbits - 1));
  // where the key levels keep hi + lo, their scale serves the QJL weight alone
  if (!key_lo(d, kbits)) {
    m.lv.ks = best_scale(kp, 1 << (kbits - 1), fabsf(alpha), 0.003f);
  } else {
    const float top = top_level(kc, kbits);
    const float lo = alpha != 0.f ? fabsf(alpha) : top;
    int e;
    frexpf(top, &e);
    // alpha s = 2^k exactly, the largest level in (8, 32)
    int ea;  // (the largest level and lo parts well inside f16's range)
    const float ma = frexpf(lo, &ea);
    m.lv.ks = ldexpf(1.f / ma, 4 - e);
  }
  const float vs = 16.f / top_level(vc, vbits);
  auto in_f16 = [](float x) { return x <= 32768.f; };  // (false for NaN)
  m.lv.fits = m.lv.ks > 0.f && vs > 0.f && in_f16(top_level(kc, kbits) * m.lv.ks) &&
              in_f16(fabsf(alpha) * m.lv.ks) && in_f16(top_level(vc, vbits) * vs);
  if (!key_lo(d, kbits))  // (a rare pair of magnitudes has no such scale)
    for (int c = 0; c < 1 << (kbits - 1); ++c)
      m.lv.fits &= fabsf(f16_round(kp[c] * m.lv.ks) - kp[c] * m.lv.ks) <= 2e-6f * kp[c] * m.lv.ks;
  fill_levels(kc, kbits, m.lv.ks, &m.lv.kl);
  fill_levels(vc, vbits, vs, &m.lv.vl);
  return m.lv;
}

template <int CT, int MB, int VB, bool PAGED>
int launch(const PreArgs& A, const KVLayers& kv, unsigned grid, hipStream_t s) {
  constexpr int smem = PreCfg<CT, MB, VB>::LDS;
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&prefill<CT, MB, VB, PAGED>),
      hipFuncAttributeMaxDynamicSharedMemorySize, smem);
  QKV_HIP(attr);
  hipLaunchKernelGGL((prefill<CT, MB, VB, PAGED>), dim3(grid), dim3(kThr), smem, s, A, kv);
  QKV_LAUNCHED();
  return QKV_OK;
}

bool symmetric(const float* c, int bits) {
  const int n = 1 << bits;
  for (int i = 0; i < n; ++i)
    if (!(c[n - 1 - i] == -c[i])) return false;
  for (int i = n / 2; i < n; ++i)
    if (!(c[i] > 1e-18f && c[i] < 1e18f)) return false;
  return true;
}

}  // namespace

bool qkv_prefill_ok(int d, int kbits, int vbits, const float* kcent, const float* vcent,
                    float qjl_scale) {
  if (!qkv_d_ok(d) || kbits < 1 || kbits > 3 || vbits < 1 || vbits > 4) return false;
  if (!symmetric(kcent, kbits) || !symmetric(vcent, vbits)) return false;
  // the QJL weight and the key levels within reach of one scale
  const float top = top_level(kcent, kbits), a = fabsf(qjl_scale);
  for (int c = 1 << (kbits - 1); c < 1 << kbits; ++c)
    if (!(kcent[c] > 1e-2f * top)) return false;
  return a < 1e3f * top && (a == 0.f || a > 1e-4f * top) &&
         levels_for(d, kbits, vbits, kcent, vcent, qjl_scale).fits;
}

int qkv_prefill_splits(int64_t bh, int R, int d, int64_t T) {
  const int64_t groups = bh * ((R + kRowsWg - 1) / kRowsWg);
  int64_t sp = qkv_num_cus() / groups;  // (a merge of the partials costs ~20 us)
  sp = std::min<int64_t>(sp, T / 256);
  // the partials stay within 64 MiB
  sp = std::min<int64_t>(sp, (int64_t(64) << 20) / (bh * R * d * 4));
  return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(sp, 64)));
}

int qkv_prefill(const QkvPrefillArgs& a, hipStream_t s) {
  const PreLevels& lv = levels_for(a.d, a.kbits, a.vbits, a.kcent, a.vcent, a.qjl_scale);
  PreArgs A{};
  A.q = a.q;
  A.q_dtype = a.q_dtype;
  A.q_vec = qkv_aligned(a.q, 16);
  A.t_stride = a.t_stride;
  A.T = a.T;
  A.Hq = a.Hq;
  A.Hkv = a.Hkv;
  A.Q = a.Q;
  A.G = a.Hq / a.Hkv;
  A.R = A.G * a.Q;
  A.BH = a.B * a.Hkv;
  A.rt = (A.R + kRowsWg - 1) / kRowsWg;
  A.n_splits = a.n_splits;
  A.pi = a.pi;
  A.signs = a.signs;
  A.alpha = a.qjl_scale * lv.ks;
  const float ah = f16_round(A.alpha);
  if (a.kbits == 2 && !key_lo(a.d, 2) && ah != 0.f) A.ae = A.alpha / ah - 1.f;
  A.c0 = a.scale * 1.4426950408889634f / lv.ks;
  A.causal = a.causal;
  A.split_len = ((a.T + a.n_splits - 1) / a.n_splits + 63) / 64 * 64;
  A.out = a.out;
  A.out_dtype = a.out_dtype;
  A.out_vec = qkv_aligned(a.out, 16);
  A.part_o = a.part_o;
  A.part_ml = a.part_ml;
  A.kl = lv.kl;
  A.vl = lv.vl;
  const int64_t grid = int64_t(A.rt) * A.BH * a.n_splits;
  QKV_REQUIRE(grid < (int64_t(1) << 31), "too many query rows");
  const unsigned g = static_cast<unsigned>(grid);
  const bool paged = a.kv.ptab != nullptr;
  switch (a.d / 32 * 100 + a.kbits * 10 + a.vbits) {
#define QKV_PF(CT, MB, VB)                                                       \
  case CT * 100 + MB * 10 + VB:                                                  \
    return paged ? launch<CT, MB, VB, true>(A, a.kv, g, s)                       \
                 : launch<CT, MB, VB, false>(A, a.kv, g, s);
#define QKV_PFV(CT, MB) QKV_PF(CT, MB, 1) QKV_PF(CT, MB, 2) QKV_PF(CT, MB, 3) QKV_PF(CT, MB, 4)
#define QKV_PFM(CT) QKV_PFV(CT, 1) QKV_PFV(CT, 2) QKV_PFV(CT, 3)
    QKV_PFM(2) QKV_PFM(3) QKV_PFM(4)
#undef QKV_PFM
#undef QKV_PFV
#undef QKV_PF
  }
  qkv_set_error("prefill: head_dim %d, %d / %d bits unsupported", a.d, a.kbits, a.vbits);
  return QKV_E_UNSUPPORTED;
}
