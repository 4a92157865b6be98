"""The tightened first column and row of a triangle's pixel scan.

tri_setup starts the reference's scan (SR/graphics.cpp:338-349) one column
(row) later when the first one lies further outside the corners than the
rounding of the coverage test reaches.  This runs the same fp32 arithmetic on
the host (gcc, no contraction, no GPU) over random triangles, from slivers of
|u.z| just over 0.01 to thousands of pixels, with corners a few ulps from
pixel columns: no pixel of a dropped column or row may be covered, and small
triangles must in fact lose theirs."""
import shutil
import subprocess

import pytest

pytestmark = pytest.mark.skipif(shutil.which("gcc") is None, reason="needs gcc")

SRC = r"""
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>

static uint64_t st;
static uint64_t nxt(void) {   /* splitmix64 */
    uint64_t z = (st += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
static double u01(void) { return (double)(nxt() >> 11) * 0x1p-53; }
static float step_ulps(float v, int n) {
    for (; n > 0; n--) v = nextafterf(v, INFINITY);
    for (; n < 0; n++) v = nextafterf(v, -INFINITY);
    return v;
}
static float ax, ay, s0x, s0y, s1x, s1y, uz;
static int covered(int px, int py) {
    float s0z = ax - (float)px, s1z = ay - (float)py;
    float p0 = s0y * s1z, p1 = s0z * s1y, p2 = s0z * s1x, p3 = s0x * s1z;
    float ux = p0 - p1, uy = p2 - p3, sum = ux + uy;
    float wx = 1.f - sum / uz, wy = uy / uz, wz = ux / uz;
    return !(wx < 0 || wy < 0 || wz < 0);
}
static float min3(float a, float b, float c) { return fminf(a, fminf(b, c)); }
static float max3(float a, float b, float c) { return fmaxf(a, fmaxf(b, c)); }
static float coord(float centre, double spread) {
    float v = (float)(centre + (u01() * 2 - 1) * spread);
    switch (nxt() % 6) {   /* on a column, or a few ulps beside one */
    case 0: return floorf(v);
    case 1: return step_ulps(floorf(v), (int)(nxt() % 9) - 4);
    default: return v;
    }
}
int main(int argc, char** argv) {
    int scale = atoi(argv[1]);
    long n = atol(argv[2]), bad = 0, dropped = 0, kept = 0;
    st = 1234567u + (uint64_t)scale;
    for (long i = 0; i < n; i++) {
        double spread = ldexp(0.5 + u01(), scale);
        float cx = (float)(spread + u01() * 4000), cy = (float)(spread + u01() * 4000);
        float x[3], y[3];
        for (int k = 0; k < 3; k++) { x[k] = coord(cx, spread); y[k] = coord(cy, spread); }
        if (nxt() % 3 == 0) {   /* a sliver: the third corner next to the line of the others */
            double t = u01() * 3 - 1, off = ldexp(u01() * 2 - 1, -(int)(nxt() % 14));
            x[2] = (float)(x[0] + t * (x[1] - x[0]) - off);
            y[2] = (float)(y[0] + t * (y[1] - y[0]) + off);
        }
        ax = x[0]; ay = y[0];
        s0x = x[2] - x[0]; s0y = x[1] - x[0]; s1x = y[2] - y[0]; s1y = y[1] - y[0];
        float q0 = s0x * s1y, q1 = s0y * s1x;
        uz = q0 - q1;
        if (!(fabsf(uz) > 0.01f)) continue;
        float mnx = fmaxf(0.f, min3(x[0], x[1], x[2])), mny = fmaxf(0.f, min3(y[0], y[1], y[2]));
        float mxx = max3(x[0], x[1], x[2]), mxy = max3(y[0], y[1], y[2]);
        if (mxx < 0 || mxy < 0) continue;
        int x0 = (int)mnx, y0 = (int)mny, x1 = (int)floorf(mxx), y1 = (int)floorf(mxy);
        float M = max3(fmaxf(fabsf(s0x), fabsf(s0y)), fabsf(s1x), fabsf(s1y));
        float mm = M * M, reach = 0x1p-15f * mm * (M + 1.0f), auz = fabsf(uz);
        int dx = (mnx - (float)x0) * auz > reach, dy = (mny - (float)y0) * auz > reach;
        dropped += dx + dy;
        kept += 2 - dx - dy;
        if (dx) for (int p = y0; p <= y1; p++) bad += covered(x0, p);
        if (dy) for (int p = x0; p <= x1; p++) bad += covered(p, y0);
    }
    printf("%ld %ld %ld\n", bad, dropped, kept);
    return 0;
}
"""


@pytest.fixture(scope="module")
def scan(tmp_path_factory):
    d = tmp_path_factory.mktemp("scan")
    (d / "scan.c").write_text(SRC)
    exe = d / "scan"
    subprocess.run(["gcc", "-O2", "-ffp-contract=off", "-o", str(exe), str(d / "scan.c"), "-lm"], check=True)
    return str(exe)


@pytest.mark.parametrize("scale", [-3, -1, 0, 2, 5, 8, 11])
def test_dropped_columns_hold_no_covered_pixel(scan, scale):
    n = 2_000_000 if scale < 5 else 400_000 if scale < 8 else 40_000
    out = subprocess.run([scan, str(scale), str(n)], check=True, capture_output=True, text=True, timeout=300).stdout
    bad, dropped, kept = map(int, out.split())
    assert bad == 0
    # a third of the coordinates lie on or next to a column, the rest anywhere
    assert dropped > kept / 4 if scale <= 5 else dropped > 0
