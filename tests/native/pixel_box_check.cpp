// Checks pixel_box.h by exhaustion: for random triangles (from sub-pixel slivers
// to a few pixels, at frames from 16 to 16384 pixels a side) every sample that
// passes the three edge tests must lie in a pixel of the box, over all pixels
// within 40 of the triangle.  Exit status 0 when none lies outside.
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>

#include "pixel_box.h"

static uint64_t rs = 0x9E3779B97F4A7C15ull;
static double rnd() {
    rs ^= rs << 13;
    rs ^= rs >> 7;
    rs ^= rs << 17;
    return (double)(rs >> 11) / 9007199254740992.0;
}
static double rnd(double a, double b) { return a + (b - a) * rnd(); }

static const float kS8[16] = {0.5625f, 0.3125f, 0.4375f, 0.6875f, 0.8125f, 0.5625f, 0.3125f, 0.1875f,
                              0.1875f, 0.8125f, 0.0625f, 0.4375f, 0.6875f, 0.9375f, 0.9375f, 0.0625f};

int main(int argc, char** argv) {
    const long n = argc > 1 ? atol(argv[1]) : 200000;
    long boxes = 0, small = 0, outside = 0, inside = 0;
    for (long it = 0; it < n; it++) {
        const int W = (int)exp(rnd(log(16.0), log(16384.0))), H = (int)exp(rnd(log(16.0), log(16384.0)));
        // size in pixels, log-uniform down to slivers far below a pixel; thin ones in a random direction
        const double size = exp(rnd(log(1e-4), log(12.0))), thin = exp(rnd(log(1e-5), 0.0));
        const double cx = rnd(-4, W + 4), cy = rnd(-4, H + 4), a = rnd(0, 6.283185307);
        float x[3], y[3];
        for (int k = 0; k < 3; k++) {
            const double s = rnd(-1, 1) * size, t = rnd(-1, 1) * size * thin;
            x[k] = (float)((cx + s * cos(a) - t * sin(a)) * 2 / W - 1);
            y[k] = (float)((cy + s * sin(a) + t * cos(a)) * 2 / H - 1);
        }
        // the edges as the setup computes them
        const float x1 = x[0], x2 = x[1], x3 = x[2], y1 = y[0], y2 = y[1], y3 = y[2];
        const float nx3 = y2 - y1, nx1 = y3 - y2, ny1 = x2 - x3, ny2 = x3 - x1, nx2 = y1 - y3, ny3 = x1 - x2;
        const float c3 = nx3 + ny3, c1 = nx1 + ny1, c2 = nx2 + ny2;
        const float twoW = 2.0f * (float)W, twoH = 2.0f * (float)H, area = (float)(H * W), eps = 1e-8f;
        const float e[3][3] = {
            {twoH * nx3, twoW * ny3, ((fmaf(x2, y1, -c3) - x1 * y2) - eps) * area},
            {twoH * nx1, twoW * ny1, ((fmaf(x3, y2, -c1) - x2 * y3) - eps) * area},
            {twoH * nx2, twoW * ny2, ((fmaf(x1, y3, -c2) - x3 * y1) - eps) * area}};
        for (int msaa = 0; msaa < 2; msaa++) {
            const ifx::PixelBox b = ifx::pixel_box(x, y, e, W, H, msaa != 0);
            const int bx0 = (int)(b.lo & 0xffff), by0 = (int)(b.lo >> 16), bx1 = (int)(b.hi & 0xffff), by1 = (int)(b.hi >> 16);
            if (b.lo == 0u && b.hi == 0xffffffffu) continue;
            boxes++;
            small += bx1 - bx0 <= 7 && by1 - by0 <= 7;
            const int px0 = (int)fmax(0, cx - 40), px1 = (int)fmin(W + 16, cx + 40);
            const int py0 = (int)fmax(0, cy - 40), py1 = (int)fmin(H + 16, cy + 40);
            for (int py = py0; py <= py1; py++)
                for (int px = px0; px <= px1; px++)
                    for (int s = 0; s < (msaa ? 8 : 1); s++) {
                        const float sx = (float)px + (msaa ? kS8[2 * s] : 0.0f), sy = (float)py + (msaa ? kS8[2 * s + 1] : 0.0f);
                        bool in = true;
                        for (int k = 0; k < 3; k++) in = in && fmaf(e[k][1], sy, e[k][0] * sx) < -e[k][2];
                        if (!in) continue;
                        inside++;
                        if (px < bx0 || px > bx1 || py < by0 || py > by1) {
                            if (outside < 8)
                                printf("%dx%d msaa %d: pixel (%d, %d) outside (%d, %d)-(%d, %d)\n", W, H, msaa, px, py,
                                       bx0, by0, bx1, by1);
                            outside++;
                        }
                    }
        }
    }
    printf("%ld triangles, %ld boxes, %ld of up to 8x8 pixels, %ld covered samples, %ld outside\n", n, boxes, small,
           inside, outside);
    return outside ? 1 : 0;
}
