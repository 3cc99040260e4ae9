/* The raster passes draw a box-form triangle by rows when its edge functions
 * are exact integers over the box (raster.hip: span_exact, edge_span): each
 * row's covered columns are solved from the three edge inequalities instead
 * of testing every box pixel (point_in_tri, cl2.cl:4798-4807).  This program
 * restates both in the same binary32 operations and compares the covered set
 * of every row of every triangle that span_exact accepts; the hardware
 * reciprocal estimate is modelled by the correctly rounded one and by its
 * neighbours one and two units in the last place away.
 *
 * usage: span_check <triangles per shape> <seed> */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static uint64_t rs;
static uint32_t rnd(void) {
    rs += 0x9E3779B97F4A7C15ull;
    uint64_t z = rs;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return (uint32_t)((z ^ (z >> 31)) >> 32);
}
static float uni(float lo, float hi) { return lo + (hi - lo) * (float)(rnd() / 4294967296.0); }
static float clampf(float x, float lo, float hi) { return fminf(fmaxf(x, lo), hi); }
static float ulps(float v, int n) {
    int32_t b;
    if (!isfinite(v) || v == 0.f) return v;
    memcpy(&b, &v, 4);
    b += n;
    memcpy(&v, &b, 4);
    return v;
}
static int inside(float x, float y, const float* e) {
    const float s = e[0] + e[1] * x + e[2] * y;
    const float t = e[3] + e[4] * x + e[5] * y;
    return s > -0.0001f && t > -0.0001f && (s + t) < e[6];
}
static void edge_span(float v, float c, int off, float* lo, float* hi) {
    const float ac = fabsf(c);
    float q = floorf(v * ulps(1.0f / ac, off));
    const float r = fmaf(-q, ac, v);
    q = r < 0.f ? q - 1.f : q;
    q = r >= ac ? q + 1.f : q;
    *lo = c > 0.f ? fmaxf(*lo, -q) : *lo;
    *hi = c < 0.f ? fminf(*hi, q) : *hi;
    *hi = c == 0.f && v < 0.f ? -1.f : *hi;
}
static int span_exact(const float* e, float xe, float ye) {
    const float bs = fmaf(fabsf(e[2]), ye, fmaf(fabsf(e[1]), xe, fabsf(e[0])));
    const float bt = fmaf(fabsf(e[5]), ye, fmaf(fabsf(e[4]), xe, fabsf(e[3])));
    return bs + bt <= 8388608.f && e[6] <= 8388608.f;
}
static uint64_t tris, exact, rows_n, pixels, hits, bad, degenerate, degenerate_hits;

static void one(const float px[3], const float py[3], float W, float H) {
    float x[3], y[3], e[7];
    for (int i = 0; i < 3; i++) { x[i] = roundf(px[i]); y[i] = roundf(py[i]); }
    const float min_x = clampf(fminf(fminf(x[0], x[1]), x[2]) - 1, 0, W - 1), max_x = clampf(fmaxf(fmaxf(x[0], x[1]), x[2]), 0, W - 1);
    const float min_y = clampf(fminf(fminf(y[0], y[1]), y[2]) - 1, 0, H - 1), max_y = clampf(fmaxf(fmaxf(y[0], y[1]), y[2]), 0, H - 1);
    const float w = max_x - min_x;
    const float A = 0.5f * (-y[1] * x[2] + y[0] * (-x[1] + x[2]) + x[0] * (y[1] - y[2]) + x[1] * y[2]);
    const float sign = A < 0 ? -1.f : 1.f;
    e[0] = (y[0] * x[2] - x[0] * y[2]) * sign;
    e[1] = (y[2] - y[0]) * sign;
    e[2] = (x[0] - x[2]) * sign;
    e[3] = (x[0] * y[1] - y[0] * x[1]) * sign;
    e[4] = (y[0] - y[1]) * sign;
    e[5] = (x[1] - x[0]) * sign;
    e[6] = 2.0001f * A * sign;
    tris++;
    if (!(w >= 1.f) || !(max_y > min_y)) return;
    if (!span_exact(e, min_x + w, max_y - 1.f)) return;
    exact++;
    const int deg = e[6] == 0.f;
    degenerate += deg;
    const float K = ceilf(e[6]) - 1.f;
    for (float fy = min_y; fy < max_y; fy += 1.f) {
        rows_n++;
        float first = -1.f, last = -2.f;
        int n = 0;
        for (float dx = 0.f; dx < w; dx += 1.f)
            if (inside(min_x + dx, fy, e)) {
                if (!n) first = dx;
                last = dx;
                n++;
            }
        pixels += (uint64_t)w;
        hits += (uint64_t)n;
        if (deg) degenerate_hits += (uint64_t)n;
        const float vs = fmaf(e[2], fy, fmaf(e[1], min_x, e[0]));
        const float vt = fmaf(e[5], fy, fmaf(e[4], min_x, e[3]));
        for (int off = -2; off <= 2; off++) {
            float lo = 0.f, hi = w - 1.f;
            edge_span(vs, e[1], off, &lo, &hi);
            edge_span(vt, e[4], off, &lo, &hi);
            edge_span(K - vs - vt, -(e[1] + e[4]), off, &lo, &hi);
            const int m = hi >= lo ? (int)(hi - lo) + 1 : 0;
            if (m != n || (n && (lo != first || hi != last))) {
                if (bad++ < 10)
                    printf("bad: (%g %g) (%g %g) (%g %g) row %g: %d [%g %g] against %d [%g %g]\n", x[0], y[0], x[1],
                           y[1], x[2], y[2], fy, m, lo, hi, n, first, last);
            }
        }
    }
}

int main(int argc, char** argv) {
    const int per = argc > 1 ? atoi(argv[1]) : 20000;
    rs = argc > 2 ? strtoull(argv[2], 0, 10) : 1;
    const float dims[5][2] = {{64, 48}, {1920, 1080}, {3840, 2160}, {1024, 1024}, {4000, 4000}};
    for (int d = 0; d < 5; d++) {
        const float W = dims[d][0], H = dims[d][1];
        /* size of the triangle around a point anywhere on (and a little off) the screen */
        const float sizes[7] = {0.6f, 1.5f, 4.f, 12.f, 60.f, 300.f, 5000.f};
        for (int k = 0; k < 7; k++) {
            const int n = sizes[k] > 100.f ? per / 200 + 10 : sizes[k] > 50.f ? per / 10 : per;
            for (int i = 0; i < n; i++) {
                const float cx = uni(-0.1f * W, 1.1f * W), cy = uni(-0.1f * H, 1.1f * H);
                float px[3], py[3];
                for (int v = 0; v < 3; v++) { px[v] = cx + uni(-sizes[k], sizes[k]); py[v] = cy + uni(-sizes[k], sizes[k]); }
                if (i % 5 == 0) py[1] = py[0];                       /* a horizontal edge */
                if (i % 7 == 0) px[2] = px[0];                       /* a vertical edge */
                if (i % 11 == 0) { px[2] = px[1]; py[2] = py[1]; }   /* a line */
                one(px, py, W, H);
            }
        }
        /* the corners of the screen and of what still counts as exact */
        const float far[3][2] = {{0, 0}, {W, 0}, {0, H}}, full[3][2] = {{-1, -1}, {2 * W, 0}, {0, 2 * H}};
        float px[3], py[3];
        for (int v = 0; v < 3; v++) { px[v] = far[v][0]; py[v] = far[v][1]; }
        one(px, py, W, H);
        for (int v = 0; v < 3; v++) { px[v] = full[v][0]; py[v] = full[v][1]; }
        one(px, py, W, H);
    }
    printf("triangles %llu, exact %llu, rows %llu, pixels %llu, covered %llu, %llu mismatches\n",
           (unsigned long long)tris, (unsigned long long)exact, (unsigned long long)rows_n, (unsigned long long)pixels,
           (unsigned long long)hits, (unsigned long long)bad);
    printf("degenerate %llu, covering %llu pixels\n", (unsigned long long)degenerate, (unsigned long long)degenerate_hits);
    return bad || degenerate_hits ? 1 : 0;
}
