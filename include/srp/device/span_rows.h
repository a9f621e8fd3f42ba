/* Tiles of a triangle's bounding box that its fragments can reach, one tile
 * row at a time, for binning triangles without exact masks.
 *
 * The reference covers pixel (x0 + nx, y0 + ny) when its three barycentrics,
 * each the float sum l0 + dy + ... + dy + dx + ... + dx (ny, then nx
 * additions; triangle.c:101-109), pass the edge test, which none below
 * -1.1e-9 does.  In exact arithmetic the sum is l0 + ny*dy + nx*dx, and
 * recursive summation errs by at most gamma(n) * M with n = nx + ny terms,
 * gamma(n) = n*u / (1 - n*u), u = 2^-24, M = |l0| + ny*|dy| + nx*|dx|.  So a
 * pixel can only be covered when for every edge
 *   l0 + ny*dy + nx*dx + slack > 0,   slack >= gamma(n) * M + 1.1e-9,
 * taking n and M at the box's far corner (both grow with nx and ny).  Within
 * a tile row the largest ny*dy lies at its first or last row, and each edge
 * then bounds nx from one side.  The interval found is widened by a pixel on
 * both sides, far more than the rounding of the few float operations here
 * (their share of slack is in its + 8 terms).  A sum or a step that is not
 * finite gives a bound that constrains nothing (fmaxf and fminf drop NaN).
 *
 * Host and device code share this header (tests/native/span_rows_check.c
 * compares it with every pixel's sequential walk); FP contraction must be
 * off, so that every pass finds the same tiles. */
#pragma once

#include <math.h>
#include <stdbool.h>
#include <stdint.h>
#include "srp/detail/qualifiers.h"

typedef struct SrpSpanScan
{
	float c[3], dy[3];   /* l0 + slack; row step */
	float inv[3];        /* 1 / |dx| */
	int low[3];          /* the edge bounds nx from below (else from above) */
	int x0, y0, w, h;    /* box */
} SrpSpanScan;

/* Box [x0, x1) x [y0, y1), not empty. */
SRP_HD static inline void srpSpanScanInit(SrpSpanScan* S, const float* l0, const float* dx, const float* dy, int x0,
                                          int y0, int x1, int y1)
{
	S->x0 = x0;
	S->y0 = y0;
	S->w = x1 - x0;
	S->h = y1 - y0;
	const float nx = (float) (S->w - 1), ny = (float) (S->h - 1);
	const float g = (nx + ny + 8.0f) * (1.0625f * 0x1p-24f);
	for (int e = 0; e < 3; e++)
	{
		const float m = fabsf(l0[e]) + ny * fabsf(dy[e]) + nx * fabsf(dx[e]);
		S->c[e] = l0[e] + (g * m + 4e-9f);
		S->dy[e] = dy[e];
		S->inv[e] = 1.0f / fabsf(dx[e]);
		S->low[e] = !(dx[e] < 0.0f);
	}
}

/* The tile columns [*a, *b] of tile row ty (1 << sh pixels a side, meeting
 * the box) that the triangle can reach; false when there is none. */
SRP_HD static inline bool srpSpanRow(const SrpSpanScan* S, uint32_t ty, uint32_t sh, uint32_t* a, uint32_t* b)
{
	const int r0 = (int) (ty << sh) - S->y0, r1 = r0 + (1 << sh) - 1;
	const float first = (float) (r0 > 0 ? r0 : 0), last = (float) (r1 < S->h ? r1 : S->h - 1);
	float lo = 0.0f, hi = (float) (S->w - 1);
	for (int e = 0; e < 3; e++)
	{
		const float t = (S->c[e] + (S->dy[e] > 0.0f ? last : first) * S->dy[e]) * S->inv[e];
		/* nx > -t, or nx < t */
		const float l = S->low[e] ? -t - 1.0f : 0.0f, h = S->low[e] ? hi : t + 1.0f;
		lo = fmaxf(lo, l);
		hi = fminf(hi, h);
	}
	if (!(lo <= hi))
		return false;
	*a = (uint32_t) (S->x0 + (int) lo) >> sh;
	*b = (uint32_t) (S->x0 + (int) hi) >> sh;
	return true;
}

/* Tiles of the whole box that the triangle can reach. */
SRP_HD static inline uint32_t srpSpanTiles(const SrpSpanScan* S, uint32_t sh)
{
	uint32_t n = 0;
	const uint32_t last = (uint32_t) (S->y0 + S->h - 1) >> sh;
	for (uint32_t ty = (uint32_t) S->y0 >> sh; ty <= last; ty++)
	{
		uint32_t a, b;
		if (srpSpanRow(S, ty, sh, &a, &b))
			n += b - a + 1u;
	}
	return n;
}
