/* The shadow prearrange drops a triangle that certainly faces away from a
 * light before it is projected (raster.hip: faces_away).  This program
 * restates that test and the culling it stands for (rotation into the cube
 * face, projection, the cross product of the projected vertices; cl2.cl:
 * 220-236, 488-494, 535-545) in the same binary32 operations, and requires
 * every triangle that is dropped to be culled, for each of the six faces,
 * with the reciprocal estimate of the device modelled up to two units in the
 * last place off.  Triangles run from far below a texel to many texels, seen
 * from every angle, most of them close to edge-on, at distances from 22 to
 * 340000, around lights at the origin and far from it.
 *
 * usage: facing_check <triangles> <seed> */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static uint64_t rs;
static double uni(void) {
    rs += 0x9E3779B97F4A7C15ull;
    uint64_t z = rs;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return (double)((z ^ (z >> 31)) >> 11) * (1.0 / 9007199254740992.0);
}
static float ulps(float v, int n) {
    int32_t b;
    memcpy(&b, &v, 4);
    b += n;
    memcpy(&v, &b, 4);
    return v;
}
typedef struct { float s[3], c[3]; } sc;
static void rot(const float* p, const float* l, const sc* q, float* r) {
    const float x = p[0] - l[0], y = p[1] - l[1], z = p[2] - l[2];
    const float inner = fmaf(q->s[2], y, q->c[2] * x);
    r[0] = fmaf(q->c[1], inner, -q->s[1] * z);
    const float t = fmaf(q->c[1], z, q->s[1] * inner), u = fmaf(q->c[2], y, -q->s[2] * x);
    r[1] = fmaf(q->s[0], t, q->c[0] * u);
    r[2] = fmaf(q->c[0], t, -q->s[0] * u);
}
static int cubeface(const float* p, const float* l) {
    const float x = p[0] - l[0], y = p[1] - l[1], z = p[2] - l[2], ax = fabsf(x), ay = fabsf(y), az = fabsf(z);
    if (ax >= ay && ax >= az) return x < 0 ? 4 : 5;
    if (ay > ax && ay >= az) return y < 0 ? 1 : 3;
    if (az > ax && az > ay && z < 0) return 2;
    return 0;
}
static float dot3(const float* a, const float* b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; }
static float max3(const float* a) { return fmaxf(fmaxf(fabsf(a[0]), fabsf(a[1])), fabsf(a[2])); }

int main(int argc, char** argv) {
    const long n = argc > 1 ? atol(argv[1]) : 1000000;
    rs = argc > 2 ? strtoull(argv[2], 0, 10) : 1;
    const float pi = 3.1415927f;
    const float ang[6][3] = {{0, 0, 0}, {pi / 2.0f, 0, 0}, {0, pi, 0}, {3.0f * pi / 2.0f, 0, 0}, {0, 3.0f * pi / 2.0f, 0}, {0, pi / 2.0f, 0}};
    sc F[6];
    for (int f = 0; f < 6; f++)
        for (int k = 0; k < 3; k++) { F[f].s[k] = (float)sin((double)ang[f][k]); F[f].c[k] = (float)cos((double)ang[f][k]); }
    long one = 0, away = 0, back = 0, bad = 0;
    const float Ls[4] = {8, 127, 1024, 4000};
    for (long i = 0; i < n; i++) {
        float l[3], w[3][3];
        const double lscale = pow(10.0, 5.0 * uni());
        for (int k = 0; k < 3; k++) l[k] = i % 3 ? (float)((uni() - 0.5) * lscale) : 0.f;
        const double d = 22.0 * pow(340000.0 / 22.0, uni()), size = d * pow(10.0, -5.0 + 4.6 * uni());
        double dir[3], c[3], t1[3], t2[3];
        for (int k = 0; k < 3; k++) dir[k] = 2 * uni() - 1;
        for (int k = 0; k < 3; k++) c[k] = l[k] + dir[k] * d;
        /* a triangle in the plane of two random directions, most of the time
           tilted so that the light lies close to that plane */
        for (int k = 0; k < 3; k++) { t1[k] = 2 * uni() - 1; t2[k] = 2 * uni() - 1; }
        if (i % 4) {
            const double tilt = pow(10.0, -7.0 * uni()) * (uni() < 0.5 ? -1 : 1);
            for (int k = 0; k < 3; k++) t2[k] = dir[k] + tilt * t2[k];
        }
        for (int v = 0; v < 3; v++) {
            const double a = 2 * uni() - 1, b = 2 * uni() - 1;
            for (int k = 0; k < 3; k++) w[v][k] = (float)(c[k] + size * (a * t1[k] + b * t2[k]));
        }
        const int f = cubeface(w[0], l);
        if (cubeface(w[1], l) != f || cubeface(w[2], l) != f) continue;
        one++;
        float a[3], b[3], e[3], rel0[3], near = 3.0e38f, far = 0.f;
        for (int k = 0; k < 3; k++) { a[k] = w[1][k] - w[0][k]; b[k] = w[2][k] - w[0][k]; }
        for (int k = 0; k < 3; k++) { e[k] = b[k] - a[k]; rel0[k] = w[0][k] - l[k]; }
        const float nrm[3] = {a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]};
        const float edge = fmaxf(fmaxf(max3(a), max3(b)), max3(e));
        for (int v = 0; v < 3; v++) {
            float r[3] = {w[v][0] - l[0], w[v][1] - l[1], w[v][2] - l[2]};
            near = fminf(near, max3(r));
            far = fmaxf(far, max3(r));
        }
        int drop = 0;
        for (int off = -2; off <= 2; off++) {
            const float ee = edge * ulps(1.0f / near, off);
            const float bound = far * far * far * fmaf(ee, fmaf(ee, 224.f * 0x1p-24f, 640.f * 0x1p-24f), 6400.f * 0x1p-48f);
            drop |= near > 21.f && far < 349000.f && dot3(nrm, rel0) > bound;
        }
        for (int li = 0; li < 4; li++) {
            const float L = Ls[li];
            float p[3][2];
            for (int v = 0; v < 3; v++) {
                float r[3];
                rot(w[v], l, &F[f], r);
                const float q = (L / 2.0f) / r[2];
                p[v][0] = fmaf(r[0], q, L / 2.f);
                p[v][1] = fmaf(r[1], q, L / 2.f);
                if (drop && !(r[2] > 20.f && r[2] <= 350000.f)) bad++;
            }
            const float ax = p[1][0] - p[0][0], ay = p[1][1] - p[0][1], bx = p[2][0] - p[0][0], by = p[2][1] - p[0][1];
            const int front = ax * by - ay * bx < 0.f;
            back += !front;
            away += drop;
            if (drop && front) {
                if (bad++ < 5) printf("bad: L %g face %d size %g at %g\n", L, f, size, d);
            }
        }
    }
    printf("in one face %ld, culled %ld, dropped %ld, %ld mismatches\n", one, back, away, bad);
    return bad ? 1 : 0;
}
