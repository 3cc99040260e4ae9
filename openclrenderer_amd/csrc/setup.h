// setup.h — what prearrange and the raster passes form of one triangle: near
// clip, culling, the raster setup with its sample count, and the exact shortcuts
// taken where they hold beyond doubt (rows solved from the edge inequalities,
// pieces that cover nothing, triangles that face away from a light).  No lane
// of a wavefront looks at another here: tests/setup_check.cpp runs this code on
// the CPU, pixel by pixel and triangle by triangle.
#pragma once
#pragma clang fp contract(off)

#include "ocr_internal.h"
#include "walk.h"

namespace ocr {

// Setup of one cut triangle for the raster passes (kernel1 cl2.cl:5000-5046).
__device__ __forceinline__ void raster_setup(const f3 p[3], float rc, float ew, float eh, RasterTri& t,
                                             float& max_y) {
  const float xs[3] = {p[0].x, p[1].x, p[2].x}, ys[3] = {p[0].y, p[1].y, p[2].y};
  float mm[4];
  calc_min_max(xs, ys, ew, eh, mm);
  t.min_x = mm[0];
  t.min_y = mm[2];
  max_y = mm[3];
  t.w = mm[1] - mm[0];
  t.iw = rcp_cr((float)(int)t.w);   // integer-valued
  const float xp[3] = {roundf(p[0].x), roundf(p[1].x), roundf(p[2].x)};
  const float yp[3] = {roundf(p[0].y), roundf(p[1].y), roundf(p[2].y)};
  // 1 / (z / depth_far) for z in [20, 350000]: the quotient by the constant
  // is exact for every finite z >= 0, its reciprocal lies in rcp_rn's range
  auto inv_rel = [](float z) { return rcp_rn(div_rcp(z, kDepthFar, kInvDepthFar)); };
  const f3 depths = mk3(inv_rel(p[0].z), inv_rel(p[1].z), inv_rel(p[2].z));
  plane_const(depths, mk3(xp[0], xp[1], xp[2]), mk3(yp[0], yp[1], yp[2]), rc, t.A, t.B, t.C);
  // point_in_tri (cl2.cl:4798-4807), loop-invariant terms in the same order
  const float p0x = xp[0], p0y = yp[0], p1x = xp[1], p1y = yp[1], p2x = xp[2], p2y = yp[2];
  const float A = 0.5f * (-p1y * p2x + p0y * (-p1x + p2x) + p0x * (p1y - p2y) + p1x * p2y);
  const float sign = A < 0 ? -1.f : 1.f;
  t.ek[0] = (p0y * p2x - p0x * p2y) * sign;
  t.ek[1] = (p2y - p0y) * sign;
  t.ek[2] = (p0x - p2x) * sign;
  t.ek[3] = (p0x * p1y - p0y * p1x) * sign;
  t.ek[4] = (p0y - p1y) * sign;
  t.ek[5] = (p1x - p0x) * sign;
  t.ek[6] = 2.0001f * A * sign;
}

// Samples of all fragments of a cut triangle.  Fragment a visits
// q in [op*a, op*a + op] up to the first q whose row is >= max_y (q_end), so
// it holds clamp(q_end - op*a, 0, op + 1) samples; the full fragments come
// first, then at most one partial one.
__device__ __forceinline__ uint32_t triangle_samples(const RasterTri& t, float max_y, int op, uint32_t nfrag) {
  if (nfrag == 0 || !(t.w > 0.f)) return 0;
  // q_end < 2^24 (frames hold at most 16,000,000 pixels): 32-bit arithmetic
  const uint32_t q_end = (uint32_t)run_start(max_y, t.w, t.iw, t.min_y);
  const uint32_t uop = (uint32_t)op;
  uint32_t m = q_end >= uop + 1 ? (q_end - (uop + 1)) / uop + 1 : 0;
  if (m > nfrag) m = nfrag;
  uint64_t s = (uint64_t)(uop + 1) * m;
  if (m < nfrag) {
    const int64_t r = (int64_t)q_end - (int64_t)uop * m;
    s += r < 0 ? 0 : (r > (int64_t)uop + 1 ? uop + 1 : (uint64_t)r);
  }
  return s > (uint64_t)kMaxTriSamples ? kMaxTriSamples : (uint32_t)s;
}

// Culling of one projected triangle (cl2.cl:4344-4380): whether it is kept.
__device__ __forceinline__ bool piece_kept(const f3 p[3], float ew, float eh, bool two_sided) {
  bool valid = two_sided || front_facing(p[0], p[1], p[2]);
  bool cond = (p[0].x < 0 && p[1].x < 0 && p[2].x < 0) ||
              (p[0].x >= ew && p[1].x >= ew && p[2].x >= ew) ||
              (p[0].y < 0 && p[1].y < 0 && p[2].y < 0) ||
              (p[0].y >= eh && p[1].y >= eh && p[2].y >= eh);
  return valid && !cond;
}

// The reference's fragment count ceil(bbox_area / op_size) of one kept.
__device__ __forceinline__ uint32_t frag_count(const f3 p[3], float ew, float eh, int op_size, float& rconst) {
  f3 xpv = mk3(roundf(p[0].x), roundf(p[1].x), roundf(p[2].x));
  f3 ypv = mk3(roundf(p[0].y), roundf(p[1].y), roundf(p[2].y));
  rconst = rconstant(xpv, ypv);
  float xs[3] = {p[0].x, p[1].x, p[2].x}, ys[3] = {p[0].y, p[1].y, p[2].y};
  float mm[4];
  calc_min_max(xs, ys, ew, eh, mm);
  float area = (mm[1] - mm[0]) * (mm[3] - mm[2]);
  float n = ceilf(div_rcp(area, (float)op_size, 1.0f / (float)op_size));   // area >= 0, op 300 or 500
  return n > 0.f ? (uint32_t)n : 0u;
}

// full_rotate_quat's rotation into a camera or cube face (cl2.cl:700-729) and
// near clip, from world-space vertices: 0..2 triangles.
__device__ __forceinline__ int face_clip(const f3 w[3], f3 cpos, const SinCos& sc, f3 tris[2][3]) {
  f3 pr[3];
#pragma unroll
  for (int i = 0; i < 3; i++) pr[i] = rot(w[i], cpos, sc);
  return clip_near(pr[0], pr[1], pr[2], tris);
}

// Whether point_in_tri's sums are exact integers for every pixel of the box
// up to column xe and row ye: the edge terms are integer-valued (vertex
// coordinates are rounded), and with |s|, |t| and the area bound at most
// 2^23 in all their partial sums nothing rounds.  Then s > -0.0001 is s >= 0,
// and s + t < e6 is s + t <= ceil(e6) - 1.
__device__ __forceinline__ bool span_exact(const float ek[7], float xe, float ye) {
  const float bs = fmaf(fabsf(ek[2]), ye, fmaf(fabsf(ek[1]), xe, fabsf(ek[0])));
  const float bt = fmaf(fabsf(ek[5]), ye, fmaf(fabsf(ek[4]), xe, fabsf(ek[3])));
  return bs + bt <= 8388608.f && ek[6] <= 8388608.f;
}

// One cut piece: its projected vertices, raster setup (key: kKeyBoxForm or
// 0, the caller adds the key), fragments, and samples: `seen` by the
// reference, `ns` of them in the list.
struct Piece {
  f3 p[3];
  RasterTri rt;
  float rc, my;   // 1/det constant; max_y, the end row of the box
  uint32_t nf, seen, ns;
};

// Count and set up a projected triangle P.p that is kept.  A piece whose walk
// visits exactly its box gets the box form: one sample per box pixel, mapped
// without the walk's fragment arithmetic.  A piece of zero rounded area with
// exact edge sums covers no pixel (s >= 0 and t >= 0 leave no s + t < 0): it
// counts, but is not listed.  Of the 1080p, 1 M-triangle frame's 446,000
// pieces 105,000 are such, of a 1024^2 cube face's small ones in that scene
// half.
__device__ __forceinline__ void setup_piece(float ew, float eh, int op, Piece& P) {
  P.nf = frag_count(P.p, ew, eh, op, P.rc);
  if (!P.nf) return;
  raster_setup(P.p, P.rc, ew, eh, P.rt, P.my);
  // the box holds at most 16,000,000 pixels (frames and cube faces), an exact
  // product, 0 when the walk has no samples (w or rows 0); the closed forms
  // of walk_is_rect settle all but tall triangles near the top row, which
  // keep the walk's samples
  const float area = P.rt.w * (P.my - P.rt.min_y);
  const bool box = area >= 1.f && area <= (float)kMaxTriSamples &&
                   walk_is_rect_closed(P.rt.min_y, P.my, P.rt.w, P.rt.iw);
  P.rt.key = box ? kKeyBoxForm : 0u;
  P.seen = box ? (uint32_t)area : triangle_samples(P.rt, P.my, op, P.nf);
  const bool empty = P.rt.ek[6] == 0.f && span_exact(P.rt.ek, P.rt.min_x + P.rt.w, P.my);
  P.ns = empty ? 0u : P.seen;
}

// Project, cull, count and set up a clipped triangle.
__device__ __forceinline__ void cut_piece(const f3 tri[3], float fovc, float ew, float eh, bool two_sided, int op,
                                          Piece& P) {
  P.nf = P.seen = P.ns = 0u;
#pragma unroll
  for (int i = 0; i < 3; i++) P.p[i] = depth_project_clipped(tri[i], ew, eh, fovc);
  if (piece_kept(P.p, ew, eh, two_sided)) setup_piece(ew, eh, op, P);
}

// Whether setup_piece finds P.p empty beyond doubt, in a quarter of its
// instructions: its vertices round, none of them from halfway (there roundf
// and this rounding may differ), to integers of zero area in [0, 1150], where
// each of span_exact's two sums is at most 3 * 1150^2 and both together below
// 2^23 (as they are up to 1182).
__device__ __forceinline__ bool piece_empty(const f3 p[3]) {
  float x[3], y[3], off = 0.f;
#pragma unroll
  for (int i = 0; i < 3; i++) {
    x[i] = rintf(p[i].x);
    y[i] = rintf(p[i].y);
    off = max3f(off, fabsf(p[i].x - x[i]), fabsf(p[i].y - y[i]));
  }
  const float lo = fminf(min3f(x[0], x[1], x[2]), min3f(y[0], y[1], y[2]));
  const float hi = fmaxf(max3f(x[0], x[1], x[2]), max3f(y[0], y[1], y[2]));
  return off < 0.5f && lo >= 0.f && hi <= 1150.f &&
         (x[1] - x[0]) * (y[2] - y[0]) == (x[2] - x[0]) * (y[1] - y[0]);
}

// ------------------------------------------------------------------- rows
// floor(a / b) for integer-valued 0 <= a < 2^24 and b >= 1 (ib close to
// 1/b): the estimate is off by at most one, the remainder is exact.
__device__ __forceinline__ float floor_div(float a, float b, float ib) {
  float q = floorf(a * ib);
  const float r = fmaf(-q, b, a);
  q = r < 0.f ? q - 1.f : q;
  return r >= b ? q + 1.f : q;
}

// The columns dx in [lo, hi] with v + c * dx >= 0 (v, c integer-valued, |v| <
// 2^24).  floor(v / |c|) from the reciprocal estimate: below 2^20 it is off
// by at most one, which the exact remainder settles; above, it stays far
// beyond every column (widths are below 2^15), which is all that matters.
__device__ __forceinline__ void edge_span(float v, float c, float& lo, float& hi) {
  const float ac = fabsf(c);
  float q = floorf(v * __builtin_amdgcn_rcpf(ac));
  const float r = fmaf(-q, ac, v);
  q = r < 0.f ? q - 1.f : q;
  q = r >= ac ? q + 1.f : q;
  lo = c > 0.f ? fmaxf(lo, -q) : lo;
  hi = c < 0.f ? fminf(hi, q) : hi;
  hi = c == 0.f && v < 0.f ? -1.f : hi;
}

// The run [lo, hi] of a row's columns (from fx, within the given lo and hi) that
// a triangle of exact edge sums covers, empty where hi < lo: e[0..5] its edge
// terms, k = ceil(e6) - 1.
__device__ __forceinline__ void row_span(float e0, float e1, float e2, float e3, float e4, float e5, float k, float fx,
                                         float fy, float& lo, float& hi) {
  // s, t and k - s - t at the row's first column (exact)
  const float vs = fmaf(e2, fy, fmaf(e1, fx, e0));
  const float vt = fmaf(e5, fy, fmaf(e4, fx, e3));
  edge_span(vs, e1, lo, hi);
  edge_span(vt, e4, lo, hi);
  edge_span(k - vs - vt, -(e1 + e4), lo, hi);
}

// ----------------------------------------------------------------- facing
// Whether front_facing is false beyond doubt for a triangle that lies in one
// cube face of a light: nrm its normal, edge the largest component of its
// edges, rel0 its first vertex from the light, near and far the smallest and
// largest distance along the face's axis (the largest component of a vertex).
// Per 64 (triangle, face) pairs the clip, projection and set-up that this
// saves are ~400 instructions; half of all pairs face away: with the faces
// found by selects from vertices kept in registers 606 M -> 498 M vector
// instructions a pass (16 lights, 4 M triangles).
//
// With u = 2^-24, L texels a side and e = edge / near: a projected coordinate
// is (L/2) x/z + L/2 with |x| <= z, formed within 10 L u (u from the difference
// to the light, 7 u from the rotation, whose sines and cosines of right angles
// are off by up to 1.5 u, the same again through z, 4 u from quotient, fma and
// sum); coordinate differences are at most L e; so the computed cross product
// is within L^2 u (80 e + 800 u + 16 e^2) of the true one, (L/2)^2 det / (z0 z1
// z2) with det = nrm . rel0, which is formed within 48 u e^2 far^3.  The cross
// product is therefore positive (facing away) if
//   det > far^3 u (320 e + 3200 u + 112 e^2),
// here with twice that bound.  Depths inside (21, 349000) are not clipped.
__device__ __forceinline__ bool faces_away(f3 nrm, float edge, f3 rel0, float near, float far) {
  const float e = edge * __builtin_amdgcn_rcpf(near);
  const float bound = far * far * far * fmaf(e, fmaf(e, 224.f * 0x1p-24f, 640.f * 0x1p-24f), 6400.f * 0x1p-48f);
  return near > 21.f && far < 349000.f && dot(nrm, rel0) > bound;
}

}  // namespace ocr
