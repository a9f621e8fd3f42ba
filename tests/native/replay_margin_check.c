/* Host check of srpReplay's jumps (include/srp/device/replay.h) as the device
 * takes them: by an approximate reciprocal, here the exact one pushed up to
 * four units in the last place either way (the hardware's is within one), or
 * flushed to zero where it is subnormal.  Each walk, of up to 65,536 steps,
 * equals n sequential float additions bit for bit: barycentrics, the x, y and
 * t of lines, and starts a whole number of steps (and a spacing more or less)
 * from the end of a binade, where one step too many would leave it.  Prints
 * the number of mismatches; exit code 1 if any. */
#include <float.h>
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static int push = 0, flush = 0;
static float reciprocal(float x)
{
	float r = 1.0f / x;
	for (int k = 0; k < abs(push); k++)
		r = nextafterf(r, push > 0 ? INFINITY : -INFINITY);
	return flush && fabsf(r) < FLT_MIN ? 0.0f : r;
}

/* the header's device branch, with this reciprocal */
#define __HIP_DEVICE_COMPILE__ 1
#define __builtin_amdgcn_rcpf reciprocal
#include "srp/device/replay.h"

static uint64_t st = 0x13198A2E03707344ull;
static uint64_t rnd(void)
{
	uint64_t z = (st += 0x9E3779B97F4A7C15ull);
	z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
	z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
	return z ^ (z >> 31);
}
static double u01(void) { return (double) (rnd() >> 11) * (1.0 / 9007199254740992.0); }

static long bad = 0, total = 0;
static void check(float a, float d, int n)
{
	float want = a;
	for (int k = 0; k < n; k++)
		want = want + d;
	for (int v = 0; v < 7; v++)
	{
		static const int pushes[7] = {-4, -2, -1, 0, 1, 2, 4};
		push = pushes[v];
		flush = v & 1;
		const float got = srpReplay(a, d, n);
		total++;
		if (memcmp(&want, &got, 4) != 0 && !(isnan(want) && isnan(got)))
		{
			if (bad++ < 10)
				printf("mismatch a=%a d=%a n=%d push=%d: %a, not %a\n", a, d, n, push, got, want);
		}
	}
}

int main(int argc, char** argv)
{
	const long iters = argc > 1 ? atol(argv[1]) : 4000;
	for (long i = 0; i < iters; i++)
	{
		const int steps = 1 + (int) (rnd() % 65535), n = (int) (rnd() % (uint64_t) (steps + 1));
		/* a line's t, and its x or y over a framebuffer of up to 65,535 pixels */
		check(0.0f, (float) (1.0 / (double) steps), n);
		check((float) (u01() * 65535.0), (float) (u01() * 2.0 - 1.0), n);
		const float x0 = (float) (u01() * 65535.0), x1 = (float) (u01() * 65535.0);
		check(x0, (x1 - x0) / (float) steps, n);
		/* a barycentric over a box of that side */
		check((float) (u01() * 3.0 - 1.0), (float) ((u01() - 0.5) * pow(10.0, -5.0 * u01())), (int) (rnd() % 65537));
		/* q steps (and a few spacings) short of the binade's end, on either side of zero */
		const int e = (int) (rnd() % 40) - 20, up = (int) (rnd() & 1);
		const double u = ldexp(1.0, e - 23), sgn = (rnd() & 1) ? 1.0 : -1.0;
		const uint64_t q = 1 + rnd() % 65536, m = 1 + rnd() % (0x7FFFFFu / q);
		const double away = u * ((double) (q * m) + (double) (rnd() % 5) - 2.0);
		const double half = (rnd() % 4 == 0) ? 0.5 : 0.0;
		if (up)
			check((float) (sgn * (ldexp(1.0, e + 1) - away)), (float) (sgn * u * ((double) m + half)), (int) (rnd() % 65537));
		else
			check((float) (sgn * (ldexp(1.0, e) + away)), (float) (-sgn * u * ((double) m + half)), (int) (rnd() % 65537));
		/* steps whose reciprocal is subnormal, from sums far larger and smaller */
		check((float) (sgn * ldexp(1.0 + u01(), 126)), (float) (sgn * -ldexp(1.0 + u01(), 126)), (int) (rnd() % 100));
		check((float) ldexp(1.0 + u01(), -102), (float) (sgn * ldexp(1.0 + u01(), -125)), (int) (rnd() % 65537));
	}
	printf("%ld of %ld walks differ\n", bad, total);
	return bad != 0;
}
