// Quantized lower bound on the canonical distance, used to skip exact
// distance gathers whose result cannot change the search state.
//
// Each vector row x gets a companion row of QC chunk groups (128 bytes, a cache
// line, each; QC = 1 up to 112 dimensions, 2 up to 240):
//   chunk 0                header {float s, float r, float lo, float hi}
//   chunks 1..(8 QC - 1)   int8 codes q (16 dimensions per chunk, zero padded)
// with x ~ s*q, a = s^2 * sum(q^2), r >= ||x - s*q||_2 (rounded up),
// lo <= a (1 - k) - r^2 (1 + k) (rounded down) and hi >= a (1 + k) -
// r^2 (1 - k) (rounded up), k = kQSlack = 2^-18. For a pair (x, y) with code
// dot product c (an exact integer),
//   Q = a_x + a_y - 2 s_x s_y c = ||s_x q_x - s_y q_y||^2,
// and the triangle inequality gives ||x - y|| >= sqrt(Q) - r_x - r_y.
//
// The canonical fp32 distance (fmaf per lane over n_lane non-negative terms,
// then the three-level octet tree) satisfies dist >= D (1 - u)^(n_lane + 5)
// - 1e-30, with D the exact squared distance, u = 2^-24 and 1e-30 an
// underflow slack, so D >= (T + eta)(1 + kappa2), kappa2 = 2 (n_lane + 8) u,
// eta = 1e-30, proves dist >= T. The fp16 distance rounds each difference and
// square to binary16 (unit 2^-11): a term t^2 becomes at least
// t^2 (1 - 3 2^-11) - 2^-24 (the absolute part covers the subnormal range),
// so for fp16 rows kappa2 = 2 (3 2^-11 + (n_lane + 8) u) and
// eta = 1e-30 + dim 2^-24.
//
// Lower test: with S >= sqrt((T + eta)(1 + kappa2)) + r_x, Q >= (S + r_y)^2
// proves dist >= T. Expanded by what belongs to which row it reads
//   (a_y - r_y^2) - 2 S r_y - 2 s_x s_y c >= S^2 - a_x,
// two fmaf and a product per candidate against one number of the querying
// row (q_lower, q_lower_proves). In fp32 with lo_y for a_y - r_y^2: a test
// that passes has S^2, 2 S r_y and r_y^2 each at most 3.1 (a_x + a_y) (the
// left side is at most 2 a_y + a_x up to rounding), so its roundings sum to
// less than 32 u (a_x + a_y); lo and the right side give up
// k (a_x + a_y) = 64 u (a_x + a_y), and 1e-30 covers underflow.
// Upper test: with 0 <= r_y <= e and e <= root - r_x, Q <= (e - r_y)^2 proves
// ||x - y|| <= root, in the same form with hi_y and e^2 lowered by k e^2 (its
// roundings are at most 8 u (e^2 + a_x + a_y)); see q_upper.
// A candidate the lower test proves would be rejected by the pool's threshold
// test, so skipping its exact distance leaves every result bit-identical.
// Rows with non-finite values, or whose scale leaves [2^-60, 2^50], get
// r = +inf and are never proved either way.
#pragma once

#include "wave.h"

namespace dance {

constexpr uint32_t kQChunks = 8;  // 16-byte chunks per chunk group
constexpr uint32_t q_chunks(int qc) { return kQChunks * (uint32_t)qc; }  // per code row
constexpr uint32_t q_max_dim(int qc) { return (q_chunks(qc) - 1u) * 16u; }  // dimensions it holds
constexpr uint32_t kQMaxDim = q_max_dim(1);
// Whether rows of this kind and width (chunks per lane) can have code rows of
// QC groups: the widths that hold 1..112 (QC = 1) or 113..240 dimensions.
constexpr bool q_width(int dt, int cpl, int qc) {
  if (dt == DANCE_U8) return false;
  if (is_f16(dt)) return qc == 1 ? cpl <= 2 : cpl >= 2 && cpl <= 4;
  return qc == 1 ? cpl <= 4 : cpl == 4 || cpl == 8;
}
constexpr float kQSlack = 0x1p-18f;

struct QBoundSet {
  const uint4* rows;  // N code rows; nullptr disables the bound
  int groups;         // chunk groups per code row (QC)
  float kappa2;       // relative rounding slack of the row type and width
  float eta;          // absolute slack (underflow; binary16 subnormals)
};

// The next fp32 value above (up) or below a finite x.
__device__ __forceinline__ float next_toward(float x, bool up) {
  if (x == 0.0f) return up ? __uint_as_float(1u) : __uint_as_float(0x80000001u);
  const uint32_t b = __float_as_uint(x);
  return __uint_as_float((x > 0.0f) == up ? b + 1u : b - 1u);
}

// One octet per row (8 rows per wave): lane sub owns code words sub, sub+8,
// sub+16, sub+24 (word w = dimensions 4w..4w+3), so every load and store of
// an octet covers contiguous bytes. Computes codes, scale and radius from the
// first `dim` elements of the row.
template <int DT, int QC>
__global__ __launch_bounds__(256) void k_quantize(RowSet rs, uint32_t N, uint32_t dim, uint4* __restrict__ out) {
  constexpr uint32_t kWords = (q_chunks(QC) - 1) * 4;  // code words
  constexpr uint32_t kPer = 4 * QC;                    // of each lane
  constexpr uint32_t kEB = DT == DANCE_F32 ? 4u : 2u;  // element bytes
  const uint32_t lane = threadIdx.x & 63u, sub = lane & 7u;
  const uint32_t row = (blockIdx.x * 256u + threadIdx.x) >> 3;
  const bool act = row < N;
  const uint8_t* rb = reinterpret_cast<const uint8_t*>(rs.rows + (size_t)(act ? row : 0u) * rs.stride16);
  const uint32_t row_bytes = rs.stride16 * 16u;
  float v[kPer][4];
#pragma unroll
  for (uint32_t k = 0; k < kPer; ++k) {
    const uint32_t w = sub + 8u * k;
    const bool in = act && w < kWords && 4u * w < dim && (4u * w + 4u) * kEB <= row_bytes;
    if constexpr (DT == DANCE_F32) {
      const uint4 c = in ? *reinterpret_cast<const uint4*>(rb + 16u * w) : make_uint4(0u, 0u, 0u, 0u);
      v[k][0] = __uint_as_float(c.x);
      v[k][1] = __uint_as_float(c.y);
      v[k][2] = __uint_as_float(c.z);
      v[k][3] = __uint_as_float(c.w);
    } else {
      const uint2 c = in ? *reinterpret_cast<const uint2*>(rb + 8u * w) : make_uint2(0u, 0u);
      v[k][0] = (float)__builtin_bit_cast(_Float16, (uint16_t)(c.x & 0xFFFFu));
      v[k][1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(c.x >> 16));
      v[k][2] = (float)__builtin_bit_cast(_Float16, (uint16_t)(c.y & 0xFFFFu));
      v[k][3] = (float)__builtin_bit_cast(_Float16, (uint16_t)(c.y >> 16));
    }
#pragma unroll
    for (uint32_t e = 0; e < 4; ++e)
      if (4u * w + e >= dim) v[k][e] = 0.0f;  // padding inside a word
  }
  float mx = 0.0f;
  int fin = 1;
#pragma unroll
  for (uint32_t k = 0; k < kPer; ++k)
#pragma unroll
    for (uint32_t e = 0; e < 4; ++e) {
      fin &= __builtin_isfinite(v[k][e]) ? 1 : 0;
      mx = fmaxf(mx, fabsf(v[k][e]));
    }
  // octet reductions (every lane of the octet ends with the result)
  mx = fmaxf(mx, __int_as_float(dpp<kDppQuadXor1>(0, __float_as_int(mx))));
  mx = fmaxf(mx, __int_as_float(dpp<kDppQuadXor2>(0, __float_as_int(mx))));
  mx = fmaxf(mx, __int_as_float(dpp<kDppHalfMirror>(0, __float_as_int(mx))));
  fin &= dpp<kDppQuadXor1>(1, fin);
  fin &= dpp<kDppQuadXor2>(1, fin);
  fin &= dpp<kDppHalfMirror>(1, fin);
  float s = mx / 127.0f;
  // all-zero rows are exact with s = 0; other scales must stay in range
  const bool usable = fin && (mx == 0.0f || (s >= 0x1p-60f && s <= 0x1p50f));
  if (!usable || mx == 0.0f) s = 0.0f;
  int A = 0;
  double err = 0.0;
  uint32_t words[kPer];
#pragma unroll
  for (uint32_t k = 0; k < kPer; ++k) {
    uint32_t word = 0u;
#pragma unroll
    for (uint32_t e = 0; e < 4; ++e) {
      int qv = 0;
      if (s > 0.0f) qv = (int)fminf(127.0f, fmaxf(-127.0f, rintf(v[k][e] / s)));
      A += qv * qv;
      const double d = (double)v[k][e] - (double)s * (double)qv;
      err = fma(d, d, err);
      word |= ((uint32_t)(qv & 0xFF)) << (8u * e);
    }
    words[k] = word;
  }
  A += dpp<kDppQuadXor1>(0, A);
  A += dpp<kDppQuadXor2>(0, A);
  A += dpp<kDppHalfMirror>(0, A);
  err += __shfl_xor(err, 1);
  err += __shfl_xor(err, 2);
  err += __shfl_xor(err, 4);
  if (!act) return;
  uint32_t* o = reinterpret_cast<uint32_t*>(out + (size_t)row * q_chunks(QC));
#pragma unroll
  for (uint32_t k = 0; k < kPer; ++k) {
    const uint32_t w = sub + 8u * k;
    if (w < kWords) o[4u + w] = words[k];
  }
  if (sub == 0) {
    float r = __builtin_inff();
    if (usable) {
      const double rd = sqrt(err) * (1.0 + 0x1p-40);
      r = (float)rd;
      if ((double)r < rd) r = __uint_as_float(__float_as_uint(r) + 1u);  // r >= 0: next float up
    }
    float lo = 0.0f, hi = 0.0f;
    if (usable) {
      const double a = (double)s * (double)s * (double)A, r2 = (double)r * (double)r, k = (double)kQSlack;
      // one fp32 step outward covers the conversion and the double roundings
      lo = next_toward((float)(a * (1.0 - k) - r2 * (1.0 + k)), false);
      hi = next_toward((float)(a * (1.0 + k) - r2 * (1.0 - k)), true);
    }
    reinterpret_cast<uint4*>(o)[0] =
        make_uint4(__float_as_uint(s), __float_as_uint(r), __float_as_uint(lo), __float_as_uint(hi));
  }
}

// The querying row's header (scalars) and code row address.
struct QSelf {
  const uint4* row;
  float s, r, lo;
};

template <int QC>
__device__ __forceinline__ void q_load_self(const QBoundSet& qb, uint32_t id, QSelf& me) {
  const uint4* p = qb.rows + (size_t)id * q_chunks(QC);
  me.row = p;
  const uint4 h = p[0];  // same address in every lane: kept as scalars
  me.s = __uint_as_float(uni_u(h.x));
  me.r = __uint_as_float(uni_u(h.y));
  me.lo = __uint_as_float(uni_u(h.z));
}

// Upper bound of sqrt((T + eta)(1 + kappa2)) + r, r the querying row's.
__device__ __forceinline__ float q_threshold(const QBoundSet& qb, float r, float T) {
  const float t = (T + qb.eta) * (1.0f + qb.kappa2);
  return (__builtin_sqrtf(t) + r) * (1.0f + kQSlack);
}

// Chunks sub, sub + 8, ... of a code row.
template <int QC>
struct QCodes {
  uint4 c[QC];
};

// The lane's chunks of the code row of candidate `id`. An inactive lane loads
// nothing and the value is left unset (as in load_row): `active` is the same
// on the 8 lanes of an octet, and callers discard the answers of inactive
// octets.
template <int QC>
__device__ __forceinline__ QCodes<QC> q_load(const QBoundSet& qb, uint32_t id, bool active, uint32_t sub) {
  QCodes<QC> b;
  const uint4* p = qb.rows + (size_t)id * q_chunks(QC);
#pragma unroll
  for (int c = 0; c < QC; ++c)
    if (active) b.c[c] = p[sub + 8u * (uint32_t)c];
  return b;
}
// The querying row's chunks, its header replaced by zeros, so that a
// candidate's header adds nothing to the dot.
template <int QC>
__device__ __forceinline__ QCodes<QC> q_codes(QCodes<QC> row, uint32_t sub) {
  if (sub == 0u) row.c[0] = make_uint4(0u, 0u, 0u, 0u);
  return row;
}

// The querying side of the lower test (see above): row header s, r, lo and S.
struct QLower {
  float m2s;  // -2 s
  float n2S;  // -2 S
  float K;    // S^2 - a (1 - k), 1e-30 added
};
__device__ __forceinline__ QLower q_lower(float s, float r, float lo, float S) {
  return QLower{-2.0f * s, -2.0f * S, __builtin_fmaf(S, S, 1e-30f) - __builtin_fmaf(r, r, lo)};
}
// Whether the bound proves dist >= T for a candidate with header s, r, lo and
// code dot c. Non-finite r or S make a NaN or -inf here, which proves nothing.
__device__ __forceinline__ bool q_lower_proves(const QLower& me, float s, float r, float lo, int c) {
  return __builtin_fmaf(me.m2s * s, (float)c, __builtin_fmaf(me.n2S, r, lo)) >= me.K;
}

// Exact integer code dot of a querying row (q_codes) and a row whose chunks an
// octet holds (q_load); every lane of the octet receives it. Must be called by
// all 64 lanes.
template <int QC>
__device__ __forceinline__ int q_octet_dot(const QCodes<QC>& code, const QCodes<QC>& b) {
  int c = 0;
#pragma unroll
  for (int k = 0; k < QC; ++k) {
    c = __builtin_amdgcn_sdot4((int)code.c[k].x, (int)b.c[k].x, c, false);
    c = __builtin_amdgcn_sdot4((int)code.c[k].y, (int)b.c[k].y, c, false);
    c = __builtin_amdgcn_sdot4((int)code.c[k].z, (int)b.c[k].z, c, false);
    c = __builtin_amdgcn_sdot4((int)code.c[k].w, (int)b.c[k].w, c, false);
  }
  c += dpp<kDppHalfMirror>(0, c);
  c += dpp<kDppQuadXor2>(0, c);
  c += dpp<kDppQuadXor1>(0, c);
  return c;
}

// Octet test for a candidate: the lanes of the octet hold its code row `b`
// (q_load); the lane with sub == 0 (which holds the header) returns whether the
// bound proves dist >= T. `code` is the querying row (q_codes). Must be called
// by all 64 lanes.
template <int QC>
__device__ __forceinline__ bool q_proves_reject(const QLower& me, const QCodes<QC>& code, const QCodes<QC>& b) {
  const int c = q_octet_dot<QC>(code, b);
  return q_lower_proves(me, __uint_as_float(b.c[0].x), __uint_as_float(b.c[0].y), __uint_as_float(b.c[0].z), c);
}

// The upper-bound side, for a pair test fl(alpha * dist) <= T0 (the online
// insert's occlusion test). The canonical distance satisfies dist <= D (1 +
// u)^(n_lane + 5) + 1e-30 <= D (1 + kappa2) + eta' by the rounding argument of
// the lower side (binary16 terms: at most t^2 (1 + 2^-11)^3 + 2^-24 each),
// with eta' <= 2 eta, and fl(alpha * dist) <= alpha dist (1 + u). So D <=
// (T0 / (alpha (1 + u)) - 2 eta) / (1 + kappa2) proves the test. q_ub_root
// returns the square root of that bound on D, rounded down (every step's
// rounding absorbed by the 2^-20 and kQSlack factors), or -1 (never proved)
// when T0 is below 1e-30 or not finite or the bound is not a positive finite
// number.
__device__ __forceinline__ float q_ub_root(const QBoundSet& qb, float T0, float alpha) {
  if (!(T0 >= 1e-30f) || !(T0 <= FLT_MAX)) return -1.0f;
  const float t = T0 / alpha * (1.0f - 0x1p-20f);
  const float t2 = (t - 2.0f * qb.eta) / (1.0f + qb.kappa2) * (1.0f - kQSlack);
  if (!(t2 > 0.0f) || !(t2 <= FLT_MAX)) return -1.0f;
  return __builtin_sqrtf(t2) * (1.0f - kQSlack);
}
// q_ub_root for rows of type DT. The binary16 distance squares each
// difference in binary16, which overflows to +inf past 65504; D <= 254^2
// keeps every term finite (a difference of at most 254 (1 + 2^-11) squares
// to below 65504), so the root is capped there for fp16 rows.
template <int DT>
__device__ __forceinline__ float q_ub_root_of(const QBoundSet& qb, float T0, float alpha) {
  const float r = q_ub_root(qb, T0, alpha);
  return is_f16(DT) ? fminf(r, 254.0f) : r;
}
// The querying side of the upper test (see above): row header s, r, hi and
// the root that ||x - y|| must not pass (negative: nothing is proved).
struct QUpper {
  float m2s;  // -2 s
  float e, e2;  // e <= root - r (-1 when not positive), 2 e
  float K;    // e^2 (1 - k) - a (1 + k) - 1e-30
};
__device__ __forceinline__ QUpper q_upper(float s, float r, float hi, float root) {
  float e = (root - r) * (1.0f - kQSlack);
  if (!(e > 0.0f)) e = -1.0f;
  return QUpper{-2.0f * s, e, 2.0f * e, e * e * (1.0f - kQSlack) - __builtin_fmaf(r, r, hi) - 1e-30f};
}
__device__ __forceinline__ bool q_upper_proves(const QUpper& me, float s, float r, float hi, int c) {
  return r <= me.e && __builtin_fmaf(me.m2s * s, (float)c, __builtin_fmaf(me.e2, r, hi)) <= me.K;
}

// Threshold of the prune's bound for a candidate at stored distance sd: a
// pair distance d >= T gives fl(alpha * d) >= fl(alpha * T) > sd, so the
// candidate survives. Returns sqrt((T + eta)(1 + kappa2)) rounded up, the
// per-candidate part of q_threshold; +inf (never skipped) for sd < 1e-30 or
// non-finite sd, where the relative slack would not cover rounding.
__device__ __forceinline__ float prune_bound_root(const QBoundSet& qb, float sd, float alpha) {
  if (!(sd >= 1e-30f) || !(sd <= FLT_MAX)) return __builtin_inff();
  const float T = sd / alpha * (1.0f + 0x1p-20f);
  const float t = (T + qb.eta) * (1.0f + qb.kappa2);
  return __builtin_sqrtf(t) * (1.0f + kQSlack);
}

// Bits 0, 8, ..., 56 of a ballot -> bits 0..7.
__device__ __forceinline__ uint32_t octet_bits(uint64_t m) {
  return (uint32_t)(((m & 0x0101010101010101ull) * 0x0102040810204080ull) >> 56);
}

}  // namespace dance
