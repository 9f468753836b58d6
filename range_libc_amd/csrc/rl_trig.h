// Single-precision sine/cosine that reproduce the host C library's sinf/cosf
// bit for bit, usable from host and device code.
//
// The reference casts rays with glibc's cosf/sinf (RangeLib.h:713-714 for
// Bresenham, RangeLib.h:931-932 for ray marching).  glibc's float routines are
// not correctly rounded: on about 0.2% of inputs with |x| <= 64 their result is
// the float on the far side of the rounding midpoint (the true value always lies within
// ~0.061 ulp of that midpoint).  A one-ulp change in a ray direction moves a
// sample across a cell edge now and then, so the GPU must reproduce glibc's
// choice exactly.
//
// Method (own derivation):
//   1. Evaluate sin/cos in double precision: Cody-Waite reduction by pi/2 with
//      a three-part constant (the first two parts carry 33 significant bits, so
//      n*P1 and n*P2 are exact for |n| < 2^20), then Taylor polynomials of
//      degree 17 (sin) and 18 (cos) on |r| <= pi/4 + eps, evaluated in Horner
//      form.  Truncation error < 1e-19, so the double result is within a few
//      ulp(double) of the true value.  Only IEEE +,-,*,/ and rint are used and
//      the file must be built with contraction off, so host and device produce
//      identical doubles.
//   2. Round to float.  If the double lies within `delta` of the midpoint
//      between the two candidate floats, consult an exception set listing
//      the inputs for which glibc returns the other candidate.  The set and
//      delta are produced by exhaustively enumerating every float x with
//      |x| <= 64 against the C library at build time (gen_trig_table.cpp),
//      stored compactly (sorted keys per 4096-value bucket) and expanded at
//      load time into a flat bitmap so that the device probes it with a
//      single load (exceptions cluster: up to ~350 per bucket).
//
// Outside |x| <= 64 the result is the double value rounded to nearest.  The C
// library (glibc 2.35) rounds the other way on 1.3% of such inputs for sinf and
// 1.3% for cosf (2.6% of inputs differ in one of the two; 2e7 samples, uniform
// over the float encodings of 64 < |x| < 1.6e6 and uniform in value over
// [64, 1000]); the result is never more than one float away while the
// reduction is exact, i.e. for |x| < 2^20 * pi/2 (about 1.6e6).  Beyond that
// n * PIO2_1 is no longer exact and the result can differ further.  Bit
// parity with the reference therefore holds for ray headings |h| <= 64.
#pragma once
#include <stdint.h>
#include <math.h>
#include <string.h>

#ifdef __HIPCC__
#define RL_HD __host__ __device__ __forceinline__
#else
#define RL_HD static inline
#endif

#pragma clang fp contract(off)

namespace rltrig {

// pi/2 = PIO2_1 + PIO2_2 + PIO2_3 (to ~2^-122)
#define RLT_PIO2_1 0x1.921fb54400000p+0
#define RLT_PIO2_2 0x1.0b4611a600000p-34
#define RLT_PIO2_3 0x1.3198a2e037073p-69
#define RLT_TWO_OVER_PI 0.6366197723675814

// Exception-table geometry: a bucket holds 4096 consecutive float encodings of
// one sign; buckets cover |x| <= 64.0f (encoding 0x42800000).
#define RLT_ABS_LIMIT 0x42800000u
#define RLT_BUCKET_SHIFT 12
#define RLT_SIGN_SHIFT 19
#define RLT_NBUCKETS (1u << 20)

struct Table {
  const uint32_t* off;   // RLT_NBUCKETS + 1 offsets into keys
  const uint16_t* keys;  // low 12 bits of |x|'s encoding, sorted per bucket
  double delta;          // probe only when |v - midpoint| / gap <= delta
};

RL_HD uint32_t f2u(float f) {
  uint32_t u;
  memcpy(&u, &f, 4);
  return u;
}
RL_HD float u2f(uint32_t u) {
  float f;
  memcpy(&f, &u, 4);
  return f;
}

// sin(r) and cos(r) in double, r = x - n pi/2 with n = rint(x * 2/pi), |r| <= pi/4
// (n = 0 subtracts zeros and leaves x).
RL_HD void sincos_reduced(double x, double* sr, double* cr, double* n_out) {
  double n = rint(x * RLT_TWO_OVER_PI);
  double r = x - n * RLT_PIO2_1;
  r = r - n * RLT_PIO2_2;
  r = r - n * RLT_PIO2_3;
  double r2 = r * r;
  // sin r = r + r^3 * P(r^2), P = -1/3! + r^2/5! - ...  (Taylor, to r^17: on
  // |r| <= pi/4 the first dropped term, r^19 / 19!, is below 1e-19)
  double ps = 2.8114572543455206e-15;
  ps = ps * r2 - 7.647163731819816e-13;
  ps = ps * r2 + 1.6059043836821613e-10;
  ps = ps * r2 - 2.505210838544172e-08;
  ps = ps * r2 + 2.7557319223985893e-06;
  ps = ps * r2 - 0.0001984126984126984;
  ps = ps * r2 + 0.008333333333333333;
  ps = ps * r2 - 0.16666666666666666;
  *sr = r + (r * r2) * ps;
  // cos r = 1 - r^2/2 + r^4 * Q(r^2), Q = 1/4! - r^2/6! + ...  (Taylor, to r^18:
  // the first dropped term, r^20 / 20!, is below 1e-20)
  double pc = -1.5619206968586225e-16;
  pc = pc * r2 + 4.779477332387385e-14;
  pc = pc * r2 - 1.1470745597729725e-11;
  pc = pc * r2 + 2.08767569878681e-09;
  pc = pc * r2 - 2.755731922398589e-07;
  pc = pc * r2 + 2.48015873015873e-05;
  pc = pc * r2 - 0.001388888888888889;
  pc = pc * r2 + 0.041666666666666664;
  *cr = (1.0 - 0.5 * r2) + (r2 * r2) * pc;
  *n_out = n;
}

// sin(x) and cos(x) in double for float x.
RL_HD void sincos_d(float xf, double* s_out, double* c_out) {
  double x = (double)xf;
  if (!(fabs(x) < 1.0e9)) {  // inf, nan, or absurdly large headings
    if (x != x || fabs(x) == INFINITY) {
      *s_out = NAN;
      *c_out = NAN;
      return;
    }
  }
  if (x == 0.0) {  // keeps the sign of a zero input: sin(-0) = -0
    *s_out = x;
    *c_out = 1.0;
    return;
  }
  double sr, cr, n;
  sincos_reduced(x, &sr, &cr, &n);
  int q = (int)(((long long)n) & 3);
  double s, c;
  if (q == 0) {
    s = sr;
    c = cr;
  } else if (q == 1) {
    s = cr;
    c = -sr;
  } else if (q == 2) {
    s = -sr;
    c = -cr;
  } else {
    s = -cr;
    c = sr;
  }
  *s_out = s;
  *c_out = c;
}

// Round v to float the way the C library does for input x: nearest unless x
// is a listed exception, in which case the far neighbour.
// `dist_out` (optional) receives |v - midpoint| / gap, 0.5 when exact.
RL_HD float neighbours(double v, float* other_out, double* dist_out) {
  float f = (float)v;
  double fd = (double)f;
  if (fd == v) {
    *other_out = f;
    *dist_out = 0.5;
    return f;
  }
  bool up = v > fd;
  uint32_t fb = f2u(f);
  uint32_t ob;
  if ((fb & 0x7fffffffu) == 0u) {
    ob = up ? 0x00000001u : 0x80000001u;
  } else if ((fb >> 31) == 0u) {
    ob = up ? fb + 1u : fb - 1u;
  } else {
    ob = up ? fb - 1u : fb + 1u;
  }
  float o = u2f(ob);
  double od = (double)o;
  double m = 0.5 * (fd + od);
  double gap = fabs(od - fd);
  *other_out = o;
  *dist_out = fabs(v - m) / gap;
  return f;
}

RL_HD bool table_has(const Table& t, float x) {
  uint32_t xb = f2u(x);
  uint32_t ab = xb & 0x7fffffffu;
  if (ab > RLT_ABS_LIMIT) return false;
  uint32_t b = (ab >> RLT_BUCKET_SHIFT) | ((xb >> 31) << RLT_SIGN_SHIFT);
  uint32_t lo = t.off[b], hi = t.off[b + 1];
  uint16_t key = (uint16_t)(ab & ((1u << RLT_BUCKET_SHIFT) - 1u));
  for (uint32_t i = lo; i < hi; ++i) {
    uint16_t k = t.keys[i];
    if (k == key) return true;
    if (k > key) break;
  }
  return false;
}

RL_HD float round_like_libc(double v, float x, const Table& t) {
  float o;
  double dist;
  float f = neighbours(v, &o, &dist);
  if (dist <= t.delta && table_has(t, x)) return o;
  return f;
}

// cosf(h) and sinf(h) as the C library computes them (bucketed table: a
// scan of sorted keys; used on the host).
RL_HD void sincosf_libc(float h, const Table& ts, const Table& tc, float* s, float* c) {
  double sd, cd;
  sincos_d(h, &sd, &cd);
  *s = round_like_libc(sd, h, ts);
  *c = round_like_libc(cd, h, tc);
}

// The same exception set as a flat bitmap: one bit per float encoding of
// each sign whose exponent field lies in [e_min, 133] (133 = exponent of
// 64.0f), so a lookup is a single byte load.  e_min is the smallest exponent
// field of any listed input.
#define RLT_EXP_MAX 133
struct Bitmap {
  const uint8_t* bits;
  int e_min;
  double delta;
};

RL_HD int bitmap_binades(int e_min) { return RLT_EXP_MAX - e_min + 1; }

RL_HD unsigned long long bitmap_bytes(int e_min) {
  return (2ull * (unsigned long long)bitmap_binades(e_min)) << 20;  // 2^23 bits per binade
}

// Bit index of x, or -1 when x is outside the covered encodings.
RL_HD long long bitmap_index(int e_min, float x) {
  uint32_t xb = f2u(x);
  uint32_t ab = xb & 0x7fffffffu;
  if (ab > RLT_ABS_LIMIT) return -1;
  int e = (int)(ab >> 23);
  if (e < e_min) return -1;
  unsigned long long slot = (unsigned long long)(xb >> 31) * (unsigned long long)bitmap_binades(e_min) +
                            (unsigned long long)(e - e_min);
  return (long long)((slot << 23) | (ab & 0x7fffffu));
}

// The float nearest to v >= 0 (or NaN), and whether to look x up: |v - midpoint| <=
// delta * gap with the float on v's other side, *other.  gap, the spacing of the
// two floats, is a power of two, and |v - midpoint| = gap / 2 - |v - f|, all exact.
// A float v is not looked up (delta is below 1/2).
RL_HD float nearest_near(double v, double delta, float* other, bool* look) {
  const float f = (float)v;
  const double fd = (double)f;
  const double e = v - fd;
  const float o = u2f(f2u(f) + (e > 0.0 ? 1u : ~0u));
  const double gap = fabs((double)o - fd);
  *other = o;
  *look = gap * 0.5 - fabs(e) <= delta * gap;
  return f;
}

// Byte of the bitmap that holds x's bit (bit x & 7 of its encoding), or byte 0 with
// *look cleared when x is not covered: bitmap_index(x) >> 3 in 32 bits.  (The
// encodings just past 64 that share its byte have no bits set.)
RL_HD uint32_t bitmap_byte(int e_min, uint32_t xb, bool* look) {
  const uint32_t lo = (uint32_t)e_min << 20;
  const uint32_t b = ((xb & 0x7fffffffu) >> 3) - lo;
  *look = *look && b <= (RLT_ABS_LIMIT >> 3) - lo;
  const uint32_t off = b + ((xb >> 31) ? (uint32_t)bitmap_binades(e_min) << 20 : 0u);
  return *look ? off : 0u;
}

// cosf(h) and sinf(h) as the C library computes them: sincos_d and round_like_libc
// without a branch.  The same double operations in the same order (a quadrant of 0
// subtracts zeros; NaN and infinities give NaN by themselves; n mod 4 is exact in
// double), the quadrant's swap by selects and its signs on the float results, as
// rounding is symmetric.  A lane of a wave takes each quadrant and nearly every
// wave has inputs to look up, so branches ran all their sides: with them 174 vector
// and 159 scalar instructions, without 127 and 78 (a kernel of
// nothing else).  Kernel times, traced: 4000 particles x 60 beams 22.1 -> 21.7 us, 100,000
// queries 24.0 -> 23.4, 20011 x 107 from pools 103.2 -> 100.6, Bresenham as before; a
// whole call's gain is within its spread.
RL_HD void sincosf_libc_bm(float h, const Bitmap& bs, const Bitmap& bc, float* s, float* c) {
  double sr, cr, n;
  sincos_reduced((double)h, &sr, &cr, &n);
  const int q = (int)(n - 4.0 * floor(n * 0.25));
  const bool odd = (q & 1) != 0;
  const double sv = odd ? cr : sr, cv = odd ? sr : cr;
  float os, oc;
  bool ls, lc;
  const float fs = nearest_near(fabs(sv), bs.delta, &os, &ls);
  const float fc = nearest_near(fabs(cv), bc.delta, &oc, &lc);
  const uint32_t xb = f2u(h);
  const uint32_t is = bitmap_byte(bs.e_min, xb, &ls), ic = bitmap_byte(bc.e_min, xb, &lc);
  // both bytes are requested before either is used (byte 0 when not looked up)
  const uint32_t ws = bs.bits[is], wc = bc.bits[ic];
  const float ms = ls && ((ws >> (xb & 7u)) & 1u) ? os : fs;
  const float mc = lc && ((wc >> (xb & 7u)) & 1u) ? oc : fc;
  const uint32_t neg_s = (sv < 0.0 ? 0x80000000u : 0u) ^ ((uint32_t)(q & 2) << 30);
  const uint32_t neg_c = (cv < 0.0 ? 0x80000000u : 0u) ^ ((uint32_t)((q + 1) & 2) << 30);
  *s = h == 0.0f ? h : u2f(f2u(ms) ^ neg_s);  // sin(-0) = -0
  *c = u2f(f2u(mc) ^ neg_c);
}

// Host-side helpers (plain host functions under hipcc).
// Smallest exponent field among the listed inputs of a bucketed table, RLT_EXP_MAX if
// there are none: the device reads a byte of the bitmap for every input.
static inline int table_min_exponent(const uint32_t* off, const uint16_t* keys) {
  int e_min = RLT_EXP_MAX;
  for (uint32_t b = 0; b < RLT_NBUCKETS; ++b)
    for (uint32_t i = off[b]; i < off[b + 1]; ++i) {
      uint32_t ab = ((b & ((1u << RLT_SIGN_SHIFT) - 1u)) << RLT_BUCKET_SHIFT) | keys[i];
      int e = (int)(ab >> 23);
      if (e < e_min) e_min = e;
      break;  // keys ascend within a bucket: the first has the smallest exponent
    }
  return e_min;
}

// Sets the bits of every listed input; `bits` holds bitmap_bytes(e_min) zeroed bytes.
static inline void table_to_bitmap(const uint32_t* off, const uint16_t* keys, int e_min, uint8_t* bits) {
  for (uint32_t b = 0; b < RLT_NBUCKETS; ++b)
    for (uint32_t i = off[b]; i < off[b + 1]; ++i) {
      uint32_t xb = (((b & ((1u << RLT_SIGN_SHIFT) - 1u)) << RLT_BUCKET_SHIFT) | keys[i]) |
                    ((b >> RLT_SIGN_SHIFT) << 31);
      long long idx = bitmap_index(e_min, u2f(xb));
      if (idx >= 0) bits[idx >> 3] |= (uint8_t)(1u << (idx & 7));
    }
}

}  // namespace rltrig
