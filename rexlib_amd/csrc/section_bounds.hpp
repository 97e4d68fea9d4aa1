// Which rows and samples of a slice can reach a brick: the bounds by which the
// brick schedule skips the rest. They keep every sample whose first tap lies in
// the brick, and no sample beyond the last shell (the prepared samples past it
// are not written).
#pragma once

#include <cmath>

namespace rexlib_hip
{

// The last stored column that is inserted (an even n's Nyquist column is not).
__host__ __device__ inline int last_column(int n)
{
	return n / 2 - (n % 2 == 0 ? 1 : 0);
}

// Where the first tap's cells of a window begin: a first tap f holds the
// positions [f + offset, f + 1 + offset), of a box window (half-width 1/2)
// -1/2, of a triangle 0, of a Kaiser-Bessel one the half-width - 1.
__host__ __device__ inline float first_tap_offset(int taps, float half_width)
{
	return taps == 1 ? -0.5f : (taps == 2 ? 0.0f : half_width - 1.0f);
}

// The positions whose first tap lies in the cells [low, low + extent) of an axis,
// widened so that rounding never drops a sample (each sample is then tested
// exactly).
__host__ __device__ inline void cell_positions(int low, int extent, float offset, float &lower, float &upper)
{
	lower = static_cast<float>(low) + offset - 0.01f;
	upper = static_cast<float>(low + extent) + offset + 0.01f;
}

// The section of a slice's plane with the box [lower, upper], as real ranges
// of k_x and k_y (of the +k copy; the -k copy's are the negated ones). With
// p = k_x X + k_y Y, eliminating k_x or k_y between the axes a and b gives
//   k_y n = X_a p_b - X_b p_a,  k_x n = Y_b p_a - Y_a p_b,  n = X_a Y_b - X_b Y_a,
// and the three pairs of axes bound each frequency exactly: the section is
// the intersection of three strips, whose projections are the intersections
// of the strips' pairwise ones. The per-axis bound of the reference
// (row_interval.cpp:34-136) takes each axis over the whole k_x range; it kept
// 28 rows per (slice, brick) at 256^3 where 7.4 hold samples, these keep 9.
// The box is widened by 0.01 voxel, the roundings here stay within
// 1e-4 (|X_a| + |X_b|) of the products, which the widening covers.
// `reciprocal` is within an ulp or two.
template <typename Reciprocal>
__host__ __device__ inline void bound_section(const float *x_step, const float *y_step, const float *lower,
	const float *upper, Reciprocal reciprocal, float *kx, float *ky)
{
	const float normal[3] = {x_step[1] * y_step[2] - x_step[2] * y_step[1],
		x_step[2] * y_step[0] - x_step[0] * y_step[2], x_step[0] * y_step[1] - x_step[1] * y_step[0]};
	kx[0] = ky[0] = -3.0e38f;
	kx[1] = ky[1] = 3.0e38f;
#pragma unroll
	for (int c = 0; c < 3; ++c)
	{
		const int a = (c + 1) % 3;
		const int b = (c + 2) % 3;
		if (fabsf(normal[c]) > 1e-30f)
		{
			const float inv = reciprocal(normal[c]);
			const auto narrow = [&](float p, float q, int i, int j, float *range)
			{
				// p [lower_i, upper_i] - q [lower_j, upper_j], over the normal.
				const float p0 = p * lower[i], p1 = p * upper[i];
				const float q0 = q * lower[j], q1 = q * upper[j];
				const float l = (fminf(p0, p1) - fmaxf(q0, q1)) * inv;
				const float u = (fmaxf(p0, p1) - fminf(q0, q1)) * inv;
				range[0] = fmaxf(range[0], fminf(l, u));
				range[1] = fminf(range[1], fmaxf(l, u));
			};
			narrow(x_step[a], x_step[b], b, a, ky);
			narrow(y_step[b], y_step[a], a, b, kx);
		}
	}
}

// The rows [r0, r1) of one sign of a slice whose samples k_x in [first,
// widest] can reach the box [lower, upper], given the section's ranges of
// k_x and k_y (all already of that sign: the -k copy passes the negated box
// and ranges); r0 >= r1 when none. `inv_y` holds 1 / y_step (0 where the step
// is 0). Evaluated per lane, one slice per lane.
__host__ __device__ inline void bound_rows(int n, const float *x_step, const float *y_step,
	const float *inv_y, int last_shell, const float *lower, const float *upper, float kx_low, float kx_high,
	float ky_low, float ky_high, int first, int &r0, int &r1)
{
	r0 = 0;
	r1 = 0;
	// (The highest row of either parity is the last column's frequency.)
	const int widest = min(last_column(n), last_shell);
	const int last_row = widest;
	const float k_low = ceilf(fmaxf(kx_low, static_cast<float>(first)));
	const float k_high = floorf(fminf(kx_high, static_cast<float>(widest)));
	float low = fmaxf(ky_low, -static_cast<float>(last_row));
	float high = fminf(ky_high, static_cast<float>(last_row));
	bool none = last_shell < 0 || k_low > k_high;
#pragma unroll
	for (int a = 0; a < 3; ++a)
	{
		const float at_first = k_low * x_step[a];
		const float at_last = k_high * x_step[a];
		const float lo = lower[a] - fmaxf(at_first, at_last);
		const float hi = upper[a] - fminf(at_first, at_last);
		if (y_step[a] == 0.0f)
		{
			none = none || !(lo <= 0.0f && 0.0f <= hi);
		}
		else
		{
			const float l = lo * inv_y[a];
			const float u = hi * inv_y[a];
			low = fmaxf(low, fminf(l, u));
			high = fminf(high, fmaxf(l, u));
		}
	}
	if (none || low > high)
	{
		return;
	}
	// The box is already widened past the window, so rounding inwards keeps
	// every sample that can reach it.
	r0 = static_cast<int>(ceilf(low));
	r1 = static_cast<int>(floorf(high)) + 1;
}

// The rows of both copies of a slice that can reach the box [lower, upper]:
// [plus[0], plus[1]) of the +k copy, [minus[0], minus[1]) of the -k copy.
// `inv_x` receives the reciprocal steps that clip_row takes (0 where a step is
// 0), shared by both.
template <typename Reciprocal>
__host__ __device__ inline void bound_slice(int n, const float *x_step, const float *y_step, int last_shell,
	const float *lower, const float *upper, Reciprocal reciprocal, int *plus, int *minus, float *inv_x)
{
	// An approximate reciprocal will do: the bounds it feeds are widened by 0.01
	// voxel, far beyond its error.
	float inv_y[3];
#pragma unroll
	for (int a = 0; a < 3; ++a)
	{
		inv_y[a] = y_step[a] == 0.0f ? 0.0f : reciprocal(y_step[a]);
		inv_x[a] = x_step[a] == 0.0f ? 0.0f : reciprocal(x_step[a]);
	}
	float kx[2];
	float ky[2];
	bound_section(x_step, y_step, lower, upper, reciprocal, kx, ky);
	bound_rows(n, x_step, y_step, inv_y, last_shell, lower, upper, kx[0], kx[1], ky[0], ky[1], 0, plus[0], plus[1]);
	const float mirrored_lower[3] = {-upper[0], -upper[1], -upper[2]};
	const float mirrored_upper[3] = {-lower[0], -lower[1], -lower[2]};
	bound_rows(n, x_step, y_step, inv_y, last_shell, mirrored_lower, mirrored_upper, -kx[1], -kx[0], -ky[1], -ky[0], 1,
		minus[0], minus[1]);
}

// Position of sample k_x along one axis from its row's base and step (the
// sign applied): the row base k_y * Y is formed in double and rounded to
// float once per row, then base + k_x * X in float, uncontracted
// (row_insertion_kernel.inl:157-166).
__host__ __device__ inline float row_position(float base, float step, int kx)
{
#pragma clang fp contract(off)
	const float product = static_cast<float>(kx) * step;
	return base + product;
}

// clip_row of one row k_y and sign: the samples k_x in [begin, end) (end <=
// begin when none) within the shell radius whose positions can fall in
// [lower, upper], a box widened by 0.01 voxel beyond every rounding here.
// `inv_step` holds 1 / step per axis (0 where the step is 0); a product with
// it stands for the division.
__host__ __device__ inline void clip_row(int n, int ky, int first, int last_shell, const float *step, const float *y_step,
	const float *inv_step, const float *lower, const float *upper, int &begin, int &end)
{
	const int widest = min(last_column(n), last_shell);
	const float radius = static_cast<float>(last_shell) + 0.5f;
	begin = 0;
	end = 0;
	const float kyf = static_cast<float>(ky);
	const float room = radius * radius - kyf * kyf;
	if (room < 0.0f)
	{
		return;
	}
	const int last = min(widest, static_cast<int>(sqrtf(room)));
	float lo_k = static_cast<float>(first);
	float hi_k = static_cast<float>(last);
	bool none = first > last;
#pragma unroll
	for (int a = 0; a < 3; ++a)
	{
		const float base = kyf * y_step[a];
		if (step[a] == 0.0f)
		{
			none = none || !(lower[a] <= base && base <= upper[a]);
		}
		else
		{
			const float l = (lower[a] - base) * inv_step[a];
			const float u = (upper[a] - base) * inv_step[a];
			lo_k = fmaxf(lo_k, fminf(l, u));
			hi_k = fminf(hi_k, fmaxf(l, u));
		}
	}
	if (!none && lo_k <= hi_k)
	{
		begin = max(static_cast<int>(ceilf(lo_k)), first);
		end = max(begin, min(static_cast<int>(floorf(hi_k)) + 1, last + 1));
	}
}

} // namespace rexlib_hip
