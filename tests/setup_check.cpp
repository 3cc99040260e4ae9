// The shortcuts of csrc/setup.h against what they stand for, both as the
// kernels are built from them (the headers compiled for the CPU, see
// host/device/hip/hip_runtime.h), with the hardware's reciprocal estimate up to
// two units in the last place off:
//   rows     row_span's run of every row, where span_exact accepts a triangle,
//            is the pixels inside_tri covers
//   facing   what faces_away drops, clip, projection and culling drop, on every
//            face
//   empty    what piece_empty drops, setup_piece finds without samples; vertices
//            on, halfway between and beside whole numbers, around 0 and 1150,
//            infinite and NaN among them
// usage: setup_check rows|facing|empty <count> <seed>
#include <stdio.h>
#include <stdlib.h>

#include "../openclrenderer_amd/csrc/setup.h"

using namespace ocr;

static uint64_t state;
static double uni() {
  state += 0x9E3779B97F4A7C15ull;
  uint64_t z = state;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return (double)((z ^ (z >> 31)) >> 11) * (1.0 / 9007199254740992.0);
}
static float in(double lo, double hi) { return (float)(lo + (hi - lo) * uni()); }
static long bad = 0;

static long rows_exact = 0, rows_pixels = 0;
static void check_rows(const f3 p[3], float W, float H) {
  RasterTri t;
  float my;
  raster_setup(p, 1.f, W, H, t, my);
  if (!(t.w >= 1.f) || !(my > t.min_y) || !span_exact(t.ek, t.min_x + t.w, my - 1.f)) return;
  rows_exact++;
  for (float y = t.min_y; y < my; y += 1.f) {
    float first = 0.f, last = -1.f;
    long n = 0;
    for (float dx = 0.f; dx < t.w; dx += 1.f)
      if (inside_tri(t.min_x + dx, y, t.ek[0], t.ek[1], t.ek[2], t.ek[3], t.ek[4], t.ek[5], t.ek[6])) {
        if (!n++) first = dx;
        last = dx;
      }
    rows_pixels += n;
    for (host_ulps = -2; host_ulps <= 2; host_ulps++) {
      float lo = 0.f, hi = t.w - 1.f;
      row_span(t.ek[0], t.ek[1], t.ek[2], t.ek[3], t.ek[4], t.ek[5], ceilf(t.ek[6]) - 1.f, t.min_x, y, lo, hi);
      const bool same = n ? lo == first && hi == last && n == (long)(hi - lo) + 1 : hi < lo;
      if (!same && bad++ < 5) printf("row %g: [%g %g] against %ld in [%g %g]\n", y, lo, hi, n, first, last);
    }
    host_ulps = 0;
  }
}
static void rows(long count) {
  const float dims[5][2] = {{64, 48}, {1920, 1080}, {3840, 2160}, {1024, 1024}, {4000, 4000}};
  const float sizes[7] = {0.6f, 1.5f, 4.f, 12.f, 60.f, 300.f, 5000.f};
  for (long i = 0; i < count; i++) {
    const float* d = dims[i % 5];
    const float size = sizes[(i / 5) % 7];
    if (size > 50.f && i % (size > 100.f ? 211 : 11)) continue;
    const float cx = in(-0.1 * d[0], 1.1 * d[0]), cy = in(-0.1 * d[1], 1.1 * d[1]);
    f3 p[3];
    for (f3& v : p) v = mk3(cx + in(-size, size), cy + in(-size, size), 1000.f);
    if (i % 3 == 0) p[1].y = p[0].y;
    if (i % 4 == 0) p[2].x = p[0].x;
    if (i % 11 == 0) p[2] = p[1];
    check_rows(p, d[0], d[1]);
  }
  for (const float* d : dims) {
    const f3 half[3] = {mk3(0, 0, 1000.f), mk3(d[0], 0, 1000.f), mk3(0, d[1], 1000.f)};
    const f3 full[3] = {mk3(-1, -1, 1000.f), mk3(2 * d[0], 0, 1000.f), mk3(0, 2 * d[1], 1000.f)};
    check_rows(half, d[0], d[1]);
    check_rows(full, d[0], d[1]);
  }
  printf("exact %ld covered %ld", rows_exact, rows_pixels);
}

static int cube_face(f3 r) {   // ret_cubeface, cl2.cl:1745-1790
  const float ax = fabsf(r.x), ay = fabsf(r.y), az = fabsf(r.z);
  if (ax >= ay && ax >= az) return r.x < 0 ? 4 : 5;
  if (ay > ax && ay >= az) return r.y < 0 ? 1 : 3;
  return az > ax && az > ay && r.z < 0 ? 2 : 0;
}
static void facing(long count) {
  const float pi = kPi, ang[6][3] = {{0, 0, 0}, {pi / 2.0f, 0, 0}, {0, pi, 0}, {3.0f * pi / 2.0f, 0, 0},
                                     {0, 3.0f * pi / 2.0f, 0}, {0, pi / 2.0f, 0}};
  SinCos face[6];
  for (int f = 0; f < 6; f++)
    for (int k = 0; k < 3; k++) {
      face[f].s[k] = (float)sin((double)ang[f][k]);
      face[f].c[k] = (float)cos((double)ang[f][k]);
    }
  long dropped = 0, culled = 0;
  for (long i = 0; i < count; i++) {
    const double spread = i % 3 ? pow(10.0, 5.0 * uni()) : 0.0;
    const f3 l = mk3(in(-spread, spread), in(-spread, spread), in(-spread, spread));
    const double d = 22.0 * pow(340000.0 / 22.0, uni()), size = d * pow(10.0, -5.0 + 4.6 * uni());
    double dir[3], t1[3], t2[3];
    for (int k = 0; k < 3; k++) {
      dir[k] = 2 * uni() - 1;
      t1[k] = 2 * uni() - 1;
      t2[k] = 2 * uni() - 1;
    }
    if (i % 4) {   // most of them nearly edge-on
      const double tilt = pow(10.0, -7.0 * uni()) * (uni() < 0.5 ? -1 : 1);
      for (int k = 0; k < 3; k++) t2[k] = dir[k] + tilt * t2[k];
    }
    f3 w[3];
    float near = 3.0e38f, far = 0.f;
    int f = -1;
    bool one = true;
    for (int v = 0; v < 3; v++) {
      const double a = 2 * uni() - 1, b = 2 * uni() - 1;
      w[v] = mk3((float)(l.x + d * dir[0] + size * (a * t1[0] + b * t2[0])),
                 (float)(l.y + d * dir[1] + size * (a * t1[1] + b * t2[1])),
                 (float)(l.z + d * dir[2] + size * (a * t1[2] + b * t2[2])));
      const f3 rel = w[v] - l;
      const float z = max3f(fabsf(rel.x), fabsf(rel.y), fabsf(rel.z));
      near = fminf(near, z);
      far = fmaxf(far, z);
      one = one && (v == 0 || cube_face(rel) == f);
      f = cube_face(rel);
    }
    if (!one) continue;
    const f3 a = w[1] - w[0], b = w[2] - w[0], c = b - a;
    const float edge = max3f(max3f(fabsf(a.x), fabsf(a.y), fabsf(a.z)), max3f(fabsf(b.x), fabsf(b.y), fabsf(b.z)),
                             max3f(fabsf(c.x), fabsf(c.y), fabsf(c.z)));
    bool drop = false;
    for (host_ulps = -2; host_ulps <= 2; host_ulps++) drop = drop || faces_away(cross(a, b), edge, w[0] - l, near, far);
    host_ulps = 0;
    dropped += drop;
    for (const float L : {8.f, 127.f, 1024.f, 4000.f}) {
      f3 tris[2][3];
      const int num = face_clip(w, l, face[f], tris);
      bool kept = false;
      for (int n = 0; n < num; n++) {
        f3 p[3];
        for (int k = 0; k < 3; k++) p[k] = depth_project_clipped(tris[n][k], L, L, L / 2.0f);
        kept = kept || front_facing(p[0], p[1], p[2]);
      }
      culled += !kept;
      if (drop && kept && bad++ < 5) printf("kept: L %g face %d size %g at %g\n", L, f, size, d);
    }
  }
  printf("dropped %ld culled %ld", dropped, culled);
}

// A coordinate near an interesting one.
static float coordinate(double centre, double size) {
  const double c = centre + (2 * uni() - 1) * size;
  switch ((int)(uni() * 8)) {
    case 0: return roundf((float)c);
    case 1: return floorf((float)c) + 0.5f;
    case 2: return nextafterf(floorf((float)c) + 0.5f, uni() < 0.5 ? -1e9f : 1e9f);
    case 3: return nextafterf(roundf((float)c), uni() < 0.5 ? -1e9f : 1e9f);
    default: return (float)c;
  }
}
static void empty(long count) {
  const double centres[8] = {0.0, 0.5, 7.0, 512.0, 1149.0, 1150.5, 1182.0, 3999.0};
  const float sides[6] = {8.f, 100.f, 1024.f, 1151.f, 1183.f, 4000.f};
  const float odd[5] = {INFINITY, -INFINITY, NAN, -0.f, 3.0e38f};
  long dropped = 0, without = 0;
  for (long i = 0; i < count; i++) {
    const double cx = centres[i % 8], cy = centres[(i / 8) % 8], size = i % 5 ? 1.5 : i % 2 ? 30.0 : 1200.0;
    f3 p[3];
    for (f3& v : p) v = mk3(coordinate(cx, size), coordinate(cy, size), in(20.0, 350000.0));
    if (i % 3 == 0) p[2] = mk3(p[1].x, p[1].y, p[2].z);
    if (i % 7 == 0) p[1].x = p[2].x = p[0].x;
    if (i % 11 == 0) p[1] = mk3(p[0].x + 3 * (p[2].x - p[0].x), p[0].y + 3 * (p[2].y - p[0].y), p[1].z);
    if (i % 97 == 0) (i % 2 ? p[i % 3].x : p[i % 3].y) = odd[(i / 97) % 5];
    const bool drop = piece_empty(p);
    dropped += drop;
    for (const float L : sides)
      for (const int op : {kOpSizeLight, kOpSize}) {
        Piece P;
        P.nf = P.seen = P.ns = 0u;
        for (int k = 0; k < 3; k++) P.p[k] = p[k];
        setup_piece(L, L, op, P);
        without += P.ns == 0u;
        if (drop && P.ns && bad++ < 5)
          printf("L %g: (%a %a) (%a %a) (%a %a) has %u samples\n", L, p[0].x, p[0].y, p[1].x, p[1].y, p[2].x, p[2].y, P.ns);
      }
  }
  printf("dropped %ld without %ld", dropped, without);
}

int main(int argc, char** argv) {
  if (argc < 4) return 2;
  const long count = atol(argv[2]);
  state = strtoull(argv[3], nullptr, 10);
  if (!strcmp(argv[1], "rows")) rows(count);
  else if (!strcmp(argv[1], "facing")) facing(count);
  else empty(count);
  printf(" mismatches %ld\n", bad);
  return bad != 0;
}
