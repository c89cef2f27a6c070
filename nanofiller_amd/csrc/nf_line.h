// nf_line.h - the line filter of the generation passes: a pair of rods whose
// infinite axes certainly stay apart cannot overlap.
//
// With p and q the centres from a common origin, u1 and u2 the directions and
// v = u1 x u2, the distance of the two lines is |w.v| / |v|, w = p - q, and
// never exceeds the segments' (Lumelsky 1985).  From the lines' moments
// m = centre x direction,
//   w.v = m1.u2 + m2.u1   and   |v|^2 = 1 - (u1.u2)^2,
// so with t = w.v / R and c = u1.u2 (moments stored over R)
//   t^2 + c^2 - 1 - slack >= 0
// drops the pair: 11 FMAs and one multiplication, no root, no quotient, and
// each rod's side depends on the rod alone.
//
// Margins.  R exceeds the cut distance by its roundings and by the FP64
// algorithm's error bound (1e-12 S^2 in the squared distance, see pair_f32).
// A pair that may be cut lies within reach, so with S = |p| + hl1 + hl2 + R
// over all pairs of the pass both centres are below S.  The error of w.v:
// w's components are each off by less than 4 ew (ew bounds the rounding of a
// shifted centre; centre, shift and origin give 2 ew per rod), together less
// than 8 ew |v|; the moments' products and sums, each below 2 S, take 4
// roundings per component and the six-term sum 6 more of values below 4 S:
// below 64 u S.  So |t| is off by less than Et = (8 ew + 64 u S) / R, which
// raises t^2 by less than 2 Et + Et^2 where |t| <= 1; c^2 and the directions'
// own norms (their squares within 4 u of 1) are off by less than 24 u.  The
// slack takes 64 u for these and the three last roundings.  Rods of another
// source may have directions less exact: with squares within dev of 1,
// |v|^2 = |u1|^2 |u2|^2 - c^2 exceeds 1 - c^2 by at most 2 dev + dev^2, and
// lengths, moments and |t| grow by less than a factor 1 + dev.
#pragma once

#include "nf_common.h"

namespace nf {

struct LineFilter {
  float scale;  // 1 / R, rounded down
  float slack;
};

struct LineSide {
  float ux, uy, uz;  // direction
  float mx, my, mz;  // moment over R
};

// R_max: largest cut distance; S: see above; dev: at most 1e-3.
NF_HD LineFilter line_filter(float R_max, float ew, float S, float dev = 0.0f) {
  S = S * (1.0f + dev);
  const float R2 = fmaf(R_max * 1.00002f, R_max, 2e-12f * S * S);
  LineFilter f;
  f.scale = recip(sqrt_up(R2)) * (1.0f - 4.0f * U32);
  const float Et = (8.0f * ew + 64.0f * U32 * S) * f.scale;
  f.slack = fmaf(Et, Et, 2.0f * Et) * (1.001f + 2.0f * dev) + 64.0f * U32 + 2.1f * dev;
  return f;
}

// (x, y, z): the centre from the common origin.
NF_HD LineSide line_side(const LineFilter& f, float x, float y, float z, const float4 D) {
  LineSide s;
  s.ux = D.x;
  s.uy = D.y;
  s.uz = D.z;
  s.mx = f.scale * fmaf(y, D.z, -(z * D.y));
  s.my = f.scale * fmaf(z, D.x, -(x * D.z));
  s.mz = f.scale * fmaf(x, D.y, -(y * D.x));
  return s;
}

// Negative when the lines may come within R; b = -1 - slack.
NF_HD float line_apart(const LineSide& p, const LineSide& q, float b) {
  const float t =
      fmaf(p.ux, q.mx, fmaf(p.uy, q.my, fmaf(p.uz, q.mz, fmaf(p.mx, q.ux, fmaf(p.my, q.uy, p.mz * q.uz)))));
  const float c = fmaf(p.ux, q.ux, fmaf(p.uy, q.uy, p.uz * q.uz));
  return fmaf(t, t, fmaf(c, c, b));
}

// A staging slot's side of the cell-pair engine's filter: its line, or, where
// every pair within reach is tested (ALL), its centre (u), the reach part rq
// (mx) and rq^2 - |centre|^2 (b).
struct SlotSide {
  LineSide l;
  float b;  // -1 - slack; a slot without a rod is apart from everything
};

// (x, y, z), hl, D: the rod's centre from the common origin, half length and
// direction; without `valid` whatever memory held, NaN included.
template <bool ALL>
NF_HD SlotSide slot_side(const LineFilter& f, float x, float y, float z, float hl, float4 D, bool valid) {
  SlotSide q;
  x = valid ? x : 0.0f;
  y = valid ? y : 0.0f;
  z = valid ? z : 0.0f;
  if (ALL) {
    const float r = valid ? (hl * 1.000001f) * 1.000006f : 0.0f;
    q.l = LineSide{x, y, z, r, 0.0f, 0.0f};
    q.b = valid ? fmaf(r, r, -fmaf(z, z, fmaf(y, y, x * x))) : -3e38f;
  } else {
    D.x = valid ? D.x : 0.0f;
    D.y = valid ? D.y : 0.0f;
    D.z = valid ? D.z : 0.0f;
    q.l = line_side(f, x, y, z, D);
    q.b = valid ? -1.0f - f.slack : 3e38f;
  }
  return q;
}

// Negative when the pair may be cut.  (f, h): the probe's line (direction,
// moment), or 2 (P - o), 2 rp and |P - o|^2 - rp^2 - slack.
template <bool ALL>
NF_HD float slot_apart(const float4 f, const float2 h, const SlotSide& q) {
  if (ALL) return h.x - fmaf(f.w, q.l.mx, fmaf(f.z, q.l.uz, fmaf(f.y, q.l.uy, fmaf(f.x, q.l.ux, q.b))));
  return line_apart(LineSide{f.x, f.y, f.z, f.w, h.x, h.y}, q.l, q.b);
}

// line_apart with the origin at the first rod's centre, whose moment is then
// zero: u1s its direction times scale, (x, y, z) the second rod's centre.
NF_HD float line_apart_from(const float3 u1s, float x, float y, float z, const float4 D1, const float4 D2, float b) {
  const float mx = fmaf(y, D2.z, -(z * D2.y)), my = fmaf(z, D2.x, -(x * D2.z)), mz = fmaf(x, D2.y, -(y * D2.x));
  const float t = fmaf(u1s.x, mx, fmaf(u1s.y, my, u1s.z * mz));
  const float c = fmaf(D1.x, D2.x, fmaf(D1.y, D2.y, D1.z * D2.z));
  return fmaf(t, t, fmaf(c, c, b));
}

}  // namespace nf
