// Counts, for one slice and one brick, what the brick kernel's row and sample
// bounds (rexlib_amd/csrc/section_bounds.hpp, the kernel's own functions) keep
// and drop, against a walk over every sample of the slice.
#include <algorithm>
#include <cmath>
#include <cstdint>

#define __host__
#define __device__
using std::max;
using std::min;
#include "section_bounds.hpp"

namespace
{

// The first tap of a position (as the kernel's window_taps::first_float).
float first_tap(int taps, float half_width, float c)
{
	if (taps == 1)
	{
		return std::trunc(c + (c < 0.0f ? -0.5f : 0.5f));
	}
	return taps == 2 ? std::floor(c) : std::floor(c - half_width) + 1.0f;
}

} // namespace

// out: samples in the brick, those of them that the bounds drop, rows kept, rows
// that hold a sample, samples kept that the slice does not insert (not written
// in memory). `ulps`: the reciprocals' error.
extern "C" void section_bounds_check(int n, const float *x, const double *y, int last_shell, int taps, float half_width,
	const int *low, const int *extent, int ulps, int64_t *out)
{
	float lower[3], upper[3];
	for (int a = 0; a < 3; ++a)
	{
		rexlib_hip::cell_positions(low[a], extent[a], rexlib_hip::first_tap_offset(taps, half_width), lower[a], upper[a]);
	}
	const auto reciprocal = [ulps](float v)
	{
		float r = 1.0f / v;
		for (int i = 0; i < std::abs(ulps); ++i)
		{
			r = std::nextafter(r, ulps > 0 ? INFINITY : -INFINITY);
		}
		return r;
	};
	const float yf[3] = {static_cast<float>(y[0]), static_cast<float>(y[1]), static_cast<float>(y[2])};
	int range[2][2] = {{0, 0}, {0, 0}};
	float inv_x[3];
	rexlib_hip::bound_slice(n, x, yf, last_shell, lower, upper, reciprocal, range[0], range[1], inv_x);
	for (int copy = 0; copy < 2; ++copy)
	{
		const float sign = copy == 0 ? 1.0f : -1.0f;
		float step[3], y_step[3], inv_step[3];
		for (int a = 0; a < 3; ++a)
		{
			step[a] = sign * x[a];
			y_step[a] = sign * yf[a];
			inv_step[a] = sign * inv_x[a];
		}
		out[2] += std::max(range[copy][1] - range[copy][0], 0);
		for (int ky = -(n / 2); ky <= n / 2; ++ky)
		{
			const bool kept_row = ky >= range[copy][0] && ky < range[copy][1];
			int begin = 0, end = 0;
			if (kept_row)
			{
				rexlib_hip::clip_row(n, ky, copy, last_shell, step, y_step, inv_step, lower, upper, begin, end);
			}
			float base[3];
			for (int a = 0; a < 3; ++a)
			{
				base[a] = static_cast<float>(static_cast<double>(ky) * (copy == 0 ? y[a] : -y[a]));
			}
			bool holds = false;
			for (int kx = copy; kx <= n / 2; ++kx)
			{
				const bool nyquist = n % 2 == 0 && (kx == n / 2 || ky == n / 2 || ky == -(n / 2));
				const int64_t square = static_cast<int64_t>(kx) * kx + static_cast<int64_t>(ky) * ky;
				const bool inserted = !nyquist && square <= static_cast<int64_t>(last_shell) * (last_shell + 1) &&
					last_shell >= 0; // |k| < L + 1/2
				const bool kept = kx >= begin && kx < end;
				if (kept && !inserted)
				{
					++out[4];
				}
				bool inside = inserted;
				for (int a = 0; a < 3 && inside; ++a)
				{
					const float f = first_tap(taps, half_width, rexlib_hip::row_position(base[a], step[a], kx));
					inside = f >= static_cast<float>(low[a]) && f < static_cast<float>(low[a] + extent[a]);
				}
				if (inside)
				{
					++out[0];
					out[1] += kept ? 0 : 1;
					holds = true;
				}
			}
			out[3] += holds ? 1 : 0;
		}
	}
}
