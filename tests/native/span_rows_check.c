/* Host check of srpSpanRow (include/srp/device/span_rows.h): every pixel
 * that the reference's sequential walk covers lies in a tile the rows list,
 * for random, sliver, tiny-step and non-finite triangles at both tile sides.
 * Prints the misses and the share of box tiles listed; exit code 1 on a miss. */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include "srp/device/abi.h"
#include "srp/device/span_rows.h"

static uint64_t st = 0x9E3779B97F4A7C15ull;
static double u01(void)
{
	uint64_t z = (st += 0x9E3779B97F4A7C15ull);
	z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
	z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
	return (double) ((z ^ (z >> 31)) >> 11) * (1.0 / 9007199254740992.0);
}

static long miss = 0, boxTiles = 0, listed = 0;

static void check(const float* l0, const float* dx, const float* dy, int x0, int y0, int x1, int y1)
{
	for (uint32_t sh = 3; sh <= 4; sh++)
	{
		SrpSpanScan S;
		srpSpanScanInit(&S, l0, dx, dy, x0, y0, x1, y1);
		const uint32_t tx0 = (uint32_t) x0 >> sh, tx1 = (uint32_t) (x1 - 1) >> sh;
		uint32_t total = 0;
		float row[3] = {l0[0], l0[1], l0[2]};
		uint32_t a = 1, b = 0, ty = ~0u;
		for (int y = y0; y < y1; y++)
		{
			if ((uint32_t) y >> sh != ty)
			{
				ty = (uint32_t) y >> sh;
				a = 1; b = 0;
				if (srpSpanRow(&S, ty, sh, &a, &b))
					total += b - a + 1;
				else { a = 1; b = 0; }
				boxTiles += tx1 - tx0 + 1;
				if (a <= b && (a < tx0 || b > tx1))
					miss++;
			}
			float l[3] = {row[0], row[1], row[2]};
			for (int x = x0; x < x1; x++)
			{
				/* the widest edge test: every edge top-left */
				if (l[0] > SRP_EDGE_TL_THRESHOLD && l[1] > SRP_EDGE_TL_THRESHOLD && l[2] > SRP_EDGE_TL_THRESHOLD)
					if ((uint32_t) x >> sh < a || (uint32_t) x >> sh > b)
						miss++;
				for (int e = 0; e < 3; e++) l[e] += dx[e];
			}
			for (int e = 0; e < 3; e++) row[e] += dy[e];
		}
		if (total != srpSpanTiles(&S, sh))
			miss++;
		listed += total;
	}
}

int main(int argc, char** argv)
{
	const int iters = argc > 1 ? atoi(argv[1]) : 300;
	for (int i = 0; i < iters; i++)
	{
		const int W = 64 + (int) (u01() * 1900), H = 64 + (int) (u01() * 1000);
		float sx[3], sy[3];
		const int kind = i % 5;
		for (int k = 0; k < 3; k++)
		{
			sx[k] = (float) (u01() * W * (kind == 1 ? 1.0 : 1.6) - (kind == 1 ? 0.0 : 0.3 * W));
			sy[k] = (float) (u01() * H * (kind == 2 ? 0.02 : 1.4) - 0.2 * H * (kind != 2));
		}
		if (kind == 3)   /* a sliver along a line */
		{
			sx[2] = sx[0] + (sx[1] - sx[0]) * 0.6f + (float) (u01() - 0.5) * 0.02f;
			sy[2] = sy[0] + (sy[1] - sy[0]) * 0.6f + (float) (u01() - 0.5) * 0.02f;
		}
		const float ex[3] = {sx[1] - sx[0], sx[2] - sx[1], sx[0] - sx[2]}, ey[3] = {sy[1] - sy[0], sy[2] - sy[1], sy[0] - sy[2]};
		float area = ex[0] * ey[2] - ey[0] * ex[2];
		float s = area < 0 ? -1.0f : 1.0f;
		area = fabsf(area);
		if (area <= 1e-9f)
			continue;
		float mnx = fminf(sx[0], fminf(sx[1], sx[2])), mxx = fmaxf(sx[0], fmaxf(sx[1], sx[2]));
		float mny = fminf(sy[0], fminf(sy[1], sy[2])), mxy = fmaxf(sy[0], fmaxf(sy[1], sy[2]));
		const int x0 = mnx < 0 ? 0 : (int) mnx, y0 = mny < 0 ? 0 : (int) mny;
		const int x1 = mxx > W ? W : (int) ceilf(mxx), y1 = mxy > H ? H : (int) ceilf(mxy);
		if (x1 <= x0 || y1 <= y0)
			continue;
		float l0[3], dx[3], dy[3];
		for (int e = 0; e < 3; e++)
		{
			const float rx = x0 + 0.5f - sx[(e + 1) % 3], ry = y0 + 0.5f - sy[(e + 1) % 3];
			l0[e] = s * (rx * ey[e] - ry * ex[e]) / area;
			dx[e] = s * ey[e] / area;
			dy[e] = -s * ex[e] / area;
		}
		if (kind == 4)
		{
			/* steps at odds with the triangle: zero, tiny, huge, not finite */
			static const float odd[8] = {0.0f, -0.0f, 1e-40f, -1e-42f, 3e38f, -INFINITY, INFINITY, NAN};
			const int e = (int) (u01() * 3);
			const float v = odd[(int) (u01() * 8)];
			if (u01() < 0.4) dx[e] = v;
			else if (u01() < 0.6) dy[e] = v;
			else l0[e] = v;
		}
		check(l0, dx, dy, x0, y0, x1, y1);
	}
	printf("%ld missed, %.3f of the box tiles listed\n", miss, (double) listed / (double) boxTiles);
	return miss != 0;
}
