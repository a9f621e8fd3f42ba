/* The reference renderer walks a triangle's barycentrics by repeated float
 * addition (raster/triangle.c:92-107 of kitrofimov/srp): the value at a
 * pixel n steps from the bounding box origin is a + d + d + ... (n
 * additions, each rounded).  srpReplay returns exactly that sum without
 * performing the n additions one by one.
 *
 * Within one binade [2^E, 2^(E+1)) of one sign every float is a multiple of
 * the binade's spacing u, and a + d rounds to the multiple nearest to it.
 * While the exact sums stay inside the binade the sum therefore moves by the
 * same multiple of u at every step - except when d lies exactly halfway
 * between multiples, where round-half-even picks by parity; after one such
 * step the sum has the parity that makes every later step equal.  So: two
 * real additions settle the step, then as many further steps as keep the sum
 * strictly inside the binade are applied at once, and the walk continues
 * from there.  The step and the distance to the binade's end are differences
 * of multiples of u below 2^24 u, so float arithmetic gives them, and the
 * product and sum of the jump, exactly.  The number of iterations is bounded
 * by the binades the walk crosses; short walks are summed directly.
 *
 * The jump's length comes from an approximate quotient, one less than its
 * floor: within 2^-21 of the exact one it never reaches the binade's end,
 * and one step too few only costs the next iteration two additions.  (An
 * integer division there took most of the walk's instructions: 2,000 random
 * triangles at 512x512 went from 2.84 to 2.24 ms a frame without it, the
 * 1080p primitive mix from 20.9 to 19.6.)
 *
 * Host and device code share this header; FP contraction must be off. */
#pragma once

#include <stdint.h>
#include <string.h>
#include "srp/detail/qualifiers.h"

SRP_HD static inline uint32_t srpFloatBits_(float x)
{
	uint32_t b;
	memcpy(&b, &x, 4);
	return b;
}

SRP_HD static inline float srpBitsFloat_(uint32_t b)
{
	float x;
	memcpy(&x, &b, 4);
	return x;
}

/* Walks of at most this many steps are summed directly: the longest of a
 * triangle with exact binning masks.  (8 made those slower, with the same
 * gain elsewhere.) */
#define SRP_REPLAY_DIRECT 24

SRP_HD static inline float srpRecip_(float x)
{
#if defined(__HIP_DEVICE_COMPILE__)
	return __builtin_amdgcn_rcpf(x);
#else
	return 1.0f / x;
#endif
}

/* a + d added n times in sequence (0 <= n <= 65536), bit for bit. */
SRP_HD static inline float srpReplay(float a, float d, int n)
{
	if (n > SRP_REPLAY_DIRECT && d == 0.0f && a - a == 0.0f)
		return a + d;   /* one addition fixes the sign of a zero sum; later ones change nothing */
	while (n > SRP_REPLAY_DIRECT)
	{
		const float b = a + d;
		const float c = b + d;
		const uint32_t ab = srpFloatBits_(a);
		n -= 2;
		a = c;
		/* zero, tiny, subnormal, huge, infinite or NaN sums, or a change of
		 * sign or binade within the two steps: continue from c */
		const uint32_t moved = (ab ^ srpFloatBits_(b)) | (ab ^ srpFloatBits_(c));
		if (((ab >> 23) & 0xFFu) - 24u >= 230u || moved >= 0x800000u)
			continue;
		const float step = c - b;
		if (step == 0.0f)
			return c;   /* c + d rounds back to c: the sum stays */
		/* the end of the binade the walk moves to: away from zero, or towards it */
		const uint32_t away = (srpFloatBits_(step) ^ ab) < 0x80000000u ? 0x800000u : 0u;
		const float end = srpBitsFloat_((ab & 0xFF800000u) + away);
		int k = (int) ((end - c) * srpRecip_(step)) - 1;
		k = k < n ? k : n;
		if (k > 0)
		{
			a = c + (float) k * step;
			n -= k;
		}
	}
	for (int i = 0; i < n; i++)
		a = a + d;
	return a;
}
