/*
 * lrh_rcp.h's step over every mantissa at the binary exponent given, from the
 * correctly rounded 1/d and the `ulps` floats on either side of it: prints the
 * estimates tried and how many results differ from the correctly rounded 1/d.
 *
 *   rcp_check <exponent> <ulps>
 */
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../../luxcore_amd/csrc/lrh_rcp.h"

int main(int argc, char **argv) {
	if (argc != 3) return 2;
	const int exponent = std::atoi(argv[1]), ulps = std::atoi(argv[2]);
	unsigned long long tried = 0, differ = 0;
	for (uint32_t m = 0; m < (1u << 23); ++m) {
		const float d = std::ldexp(1.0f + (float)m / 8388608.0f, exponent);
		const float want = 1.0f / d;
		for (int k = -ulps; k <= ulps; ++k) {
			uint32_t u;
			std::memcpy(&u, &want, 4);
			u += (uint32_t)k;
			float r;
			std::memcpy(&r, &u, 4);
			++tried;
			if (lrhRefineRcp(d, r) != want) ++differ;
		}
	}
	std::printf("%llu %llu\n", tried, differ);
	return 0;
}
