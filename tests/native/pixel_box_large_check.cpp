// Checks pixel_box.h for large triangles: from eight pixels to the whole target, vertices up to
// 64 pixels outside it and at these limits, slivers among them.  Every sample that passes the
// three edge tests must lie in a pixel of the box; looked at are three rings of pixels round
// the box, where the covered set would cross it, and the pixels near each vertex, where a
// thin corner could end between them.  Exit status 0 when none lies outside.
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>

#include "pixel_box.h"

static uint64_t rs = 0xD1B54A32D192ED03ull;
static double rnd() {
    rs ^= rs << 13;
    rs ^= rs >> 7;
    rs ^= rs << 17;
    return (double)(rs >> 11) / 9007199254740992.0;
}
static double rnd(double a, double b) { return a + (b - a) * rnd(); }

static const float kS8[16] = {0.5625f, 0.3125f, 0.4375f, 0.6875f, 0.8125f, 0.5625f, 0.3125f, 0.1875f,
                              0.1875f, 0.8125f, 0.0625f, 0.4375f, 0.6875f, 0.9375f, 0.9375f, 0.0625f};

struct Check {
    const float (*e)[3];
    int W, H, msaa, bx0, by0, bx1, by1;
    long looked = 0, outside = 0;
    // pixels the raster may look at: tiles end up to 15 pixels beyond the target
    void pixel(int px, int py) {
        if (px < 0 || py < 0 || px > W + 16 || py > H + 16) return;
        if (px >= bx0 && px <= bx1 && py >= by0 && py <= by1) return;
        looked++;
        for (int s = 0; s < (msaa ? 8 : 1); s++) {
            const float sx = (float)px + (msaa ? kS8[2 * s] : 0.0f), sy = (float)py + (msaa ? kS8[2 * s + 1] : 0.0f);
            bool in = true;
            for (int k = 0; k < 3; k++) in = in && fmaf(e[k][1], sy, e[k][0] * sx) < -e[k][2];
            if (!in) continue;
            if (outside++ < 4)
                printf("%dx%d msaa %d: pixel (%d, %d) outside (%d, %d)-(%d, %d)\n", W, H, msaa, px, py, bx0, by0, bx1,
                       by1);
        }
    }
};

int main(int argc, char** argv) {
    const long n = argc > 1 ? atol(argv[1]) : 4000;
    long boxes = 0, large = 0, looked = 0, outside = 0;
    for (long it = 0; it < n; it++) {
        const int W = (int)exp(rnd(log(16.0), log(it % 16 ? 2048.0 : 16384.0)));
        const int H = (int)exp(rnd(log(16.0), log(it % 16 ? 2048.0 : 16384.0)));
        const double size = exp(rnd(log(8.0), log(8.0 + W + H))), thin = it % 3 ? 1.0 : exp(rnd(log(1e-5), 0.0));
        const double cx = rnd(-32, W + 32), cy = rnd(-32, H + 32), a = rnd(0, 6.283185307);
        double vx[3], vy[3];
        float x[3], y[3];
        for (int k = 0; k < 3; k++) {
            const double s = rnd(-1, 1) * size, t = rnd(-1, 1) * size * thin;
            // to the limits of where the bound applies, exactly or by a hair inside
            vx[k] = fmin(W + 64.0 - 1e-3, fmax(-64.0 + 1e-3, cx + s * cos(a) - t * sin(a)));
            vy[k] = fmin(H + 64.0 - 1e-3, fmax(-64.0 + 1e-3, cy + s * sin(a) + t * cos(a)));
            if (it % 5 == 0) {  // corners on pixel corners and on their centres
                vx[k] = floor(vx[k]) + (it % 10 ? 0.5 : 0.0);
                vy[k] = floor(vy[k]) + (it % 10 ? 0.5 : 0.0);
            }
            x[k] = (float)(vx[k] * 2 / W - 1);
            y[k] = (float)(vy[k] * 2 / H - 1);
        }
        // the order the setup keeps, by its determinant
        if (x[2] * y[0] + x[1] * y[2] + x[0] * y[1] < x[1] * y[0] + x[0] * y[2] + x[2] * y[1]) {
            const float fx = x[0], fy = y[0];
            x[0] = x[2];
            y[0] = y[2];
            x[2] = fx;
            y[2] = fy;
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
            if (b.lo == 0u && b.hi == 0xffffffffu) continue;
            Check c{e, W, H, msaa, (int)(b.lo & 0xffff), (int)(b.lo >> 16), (int)(b.hi & 0xffff), (int)(b.hi >> 16)};
            boxes++;
            large += c.bx1 - c.bx0 > 63 && c.by1 - c.by0 > 63;
            if (c.bx0 <= c.bx1) {
                for (int r = 1; r <= 3; r++) {
                    for (int px = c.bx0 - r; px <= c.bx1 + r; px++) {
                        c.pixel(px, c.by0 - r);
                        c.pixel(px, c.by1 + r);
                    }
                    for (int py = c.by0 - r; py <= c.by1 + r; py++) {
                        c.pixel(c.bx0 - r, py);
                        c.pixel(c.bx1 + r, py);
                    }
                }
            }
            for (int k = 0; k < 3; k++)
                for (int dy = -12; dy <= 12; dy++)
                    for (int dx = -12; dx <= 12; dx++) c.pixel((int)floor(vx[k]) + dx, (int)floor(vy[k]) + dy);
            looked += c.looked;
            outside += c.outside;
        }
    }
    printf("%ld triangles, %ld boxes, %ld of more than 64x64 pixels, %ld pixels, %ld outside\n", n, boxes, large, looked,
           outside);
    return outside ? 1 : 0;
}
