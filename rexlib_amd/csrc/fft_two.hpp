// Transforms of length n = A B in two register steps with one exchange
// through LDS:
//   X[k1 + A k2] = sum_b W_B^(b k2) W_n^(b k1) sum_a x[b + B a] W_A^(a k1).
// Thread (line, j) holds x[j + B a], a < A, transforms them in registers,
// multiplies by W_n^(j k1), and hands them through LDS to thread (line, k1),
// which transforms the B values of its k1. A and B are any of the lengths
// below with prime factors 2, 3, 5, 7, 11 and 13, chosen by the host and
// selected by a switch (uniform over the block), so one kernel serves every
// length of its class; the classes bound the registers a kernel holds.
// The Stockham stages (fft_device.hpp) make an LDS round trip and two
// integer divisions per radix and element: 1,000 images 320^2 took 0.52 ms in
// their row pass and 0.67 ms in their column pass.
#pragma once

#include "fft_device.hpp"

#include <utility>

namespace rexlib_hip
{

namespace two_factor
{

// cos and sin of 2 pi m / r in double, from the Taylor series on [0, pi / 4].
constexpr double series_sin(double x)
{
	double term = x, sum = x;
	for (int k = 1; k < 14; ++k)
	{
		term *= -x * x / ((2 * k) * (2 * k + 1));
		sum += term;
	}
	return sum;
}

constexpr double series_cos(double x)
{
	double term = 1.0, sum = 1.0;
	for (int k = 1; k < 14; ++k)
	{
		term *= -x * x / ((2 * k - 1) * (2 * k));
		sum += term;
	}
	return sum;
}

struct root
{
	float c;
	float s;
};

// exp(2 pi i m / r), exact at the axes, by octants.
constexpr root unit_root(int m, int r)
{
	const double pi = 3.14159265358979323846;
	m %= r;
	// 8 m / r = octant + rest / r.
	const int octant = 8 * m / r;
	const int rest = 8 * m - octant * r;
	const double near = pi / 4 * rest / r;
	const double far = pi / 4 * (r - rest) / r;
	double c = 0.0, s = 0.0;
	switch (octant)
	{
	case 0: c = series_cos(near); s = series_sin(near); break;
	case 1: c = series_sin(far); s = series_cos(far); break;
	case 2: c = -series_sin(near); s = series_cos(near); break;
	case 3: c = -series_cos(far); s = series_sin(far); break;
	case 4: c = -series_cos(near); s = -series_sin(near); break;
	case 5: c = -series_sin(far); s = -series_cos(far); break;
	case 6: c = series_sin(near); s = -series_cos(near); break;
	default: c = series_cos(far); s = -series_sin(far); break;
	}
	return root{static_cast<float>(c), static_cast<float>(s)};
}

template <int R>
struct roots
{
	root w[R];
	constexpr roots() : w()
	{
		for (int m = 0; m < R; ++m)
		{
			w[m] = unit_root(m, R);
		}
	}
};

// The larger factor of R's first split: 4, else its largest prime.
constexpr int split_radix(int r)
{
	for (const int p : {13, 11, 7, 5})
	{
		if (r % p == 0)
		{
			return p;
		}
	}
	return r % 4 == 0 ? 4 : (r % 3 == 0 ? 3 : 2);
}

// In-register DFT of R values, v[k] = sum_n v[n] exp(sign 2 pi i n k / R).
template <int R>
__device__ __forceinline__ void dft_any(float2 *v, float sign)
{
	if constexpr (R == 1)
	{
	}
	else if constexpr (R == 2 || R == 3 || R == 4 || R == 5)
	{
		dft<R>(v, sign);
	}
	else if constexpr (R == 7 || R == 11 || R == 13)
	{
		// A prime: pairs k, R - k share their cosines and sines.
		constexpr roots<R> t{};
		constexpr int half = (R - 1) / 2;
		float2 sum[half], difference[half];
#pragma unroll
		for (int k = 0; k < half; ++k)
		{
			sum[k] = cadd(v[k + 1], v[R - 1 - k]);
			difference[k] = csub(v[k + 1], v[R - 1 - k]);
		}
		const float2 first = v[0];
#pragma unroll
		for (int k = 0; k < half; ++k)
		{
			v[0] = cadd(v[0], sum[k]);
		}
#pragma unroll
		for (int j = 1; j <= half; ++j)
		{
			float2 even = first;
			float2 odd = make_float2(0.0f, 0.0f);
#pragma unroll
			for (int k = 0; k < half; ++k)
			{
				const float c = t.w[j * (k + 1) % R].c;
				const float s = t.w[j * (k + 1) % R].s;
				even = make_float2(even.x + c * sum[k].x, even.y + c * sum[k].y);
				odd = make_float2(odd.x + s * difference[k].x, odd.y + s * difference[k].y);
			}
			const float2 turned = times_i(odd, sign);
			v[j] = cadd(even, turned);
			v[R - j] = csub(even, turned);
		}
	}
	else
	{
		// R = P Q: Q-strided DFTs of P, twiddles, DFTs of Q.
		constexpr int P = split_radix(R);
		constexpr int Q = R / P;
		constexpr roots<R> t{};
		float2 a[R];
#pragma unroll
		for (int n = 0; n < Q; ++n)
		{
			float2 q[P];
#pragma unroll
			for (int m = 0; m < P; ++m)
			{
				q[m] = v[n + Q * m];
			}
			dft_any<P>(q, sign);
#pragma unroll
			for (int k = 0; k < P; ++k)
			{
				a[n + Q * k] = n * k == 0 ? q[k] : cmul(q[k], make_float2(t.w[n * k].c, sign * t.w[n * k].s));
			}
		}
#pragma unroll
		for (int k = 0; k < P; ++k)
		{
			float2 q[Q];
#pragma unroll
			for (int n = 0; n < Q; ++n)
			{
				q[n] = a[n + Q * k];
			}
			dft_any<Q>(q, sign);
#pragma unroll
			for (int m = 0; m < Q; ++m)
			{
				v[k + P * m] = q[m];
			}
		}
	}
}

// The register lengths of a class, by the largest a kernel holds. The larger
// classes leave out what a shorter pair covers.
template <int CLASS, typename F>
__device__ __forceinline__ void with_radix(int radix, F &&f)
{
#define REXLIB_HIP_RADIX(R) \
	case R: \
		f(std::integral_constant<int, R>()); \
		break;
	if constexpr (CLASS <= 16)
	{
		switch (radix)
		{
			REXLIB_HIP_RADIX(4)
			REXLIB_HIP_RADIX(5)
			REXLIB_HIP_RADIX(6)
			REXLIB_HIP_RADIX(7)
			REXLIB_HIP_RADIX(8)
			REXLIB_HIP_RADIX(9)
			REXLIB_HIP_RADIX(10)
			REXLIB_HIP_RADIX(11)
			REXLIB_HIP_RADIX(12)
			REXLIB_HIP_RADIX(13)
			REXLIB_HIP_RADIX(14)
			REXLIB_HIP_RADIX(15)
			REXLIB_HIP_RADIX(16)
		default: break;
		}
	}
	else if constexpr (CLASS <= 22)
	{
		switch (radix)
		{
			REXLIB_HIP_RADIX(8)
			REXLIB_HIP_RADIX(9)
			REXLIB_HIP_RADIX(10)
			REXLIB_HIP_RADIX(11)
			REXLIB_HIP_RADIX(12)
			REXLIB_HIP_RADIX(13)
			REXLIB_HIP_RADIX(14)
			REXLIB_HIP_RADIX(15)
			REXLIB_HIP_RADIX(16)
			REXLIB_HIP_RADIX(18)
			REXLIB_HIP_RADIX(20)
			REXLIB_HIP_RADIX(21)
			REXLIB_HIP_RADIX(22)
		default: break;
		}
	}
	else
	{
		switch (radix)
		{
			REXLIB_HIP_RADIX(10)
			REXLIB_HIP_RADIX(12)
			REXLIB_HIP_RADIX(13)
			REXLIB_HIP_RADIX(14)
			REXLIB_HIP_RADIX(15)
			REXLIB_HIP_RADIX(16)
			REXLIB_HIP_RADIX(18)
			REXLIB_HIP_RADIX(20)
			REXLIB_HIP_RADIX(21)
			REXLIB_HIP_RADIX(22)
			REXLIB_HIP_RADIX(24)
			REXLIB_HIP_RADIX(25)
			REXLIB_HIP_RADIX(26)
			REXLIB_HIP_RADIX(27)
			REXLIB_HIP_RADIX(28)
			REXLIB_HIP_RADIX(30)
			REXLIB_HIP_RADIX(32)
		default: break;
		}
	}
#undef REXLIB_HIP_RADIX
}

// Wavefronts per SIMD a kernel of a class is held to (its register budget:
// 102, 128 and 170; without a bound the switch takes up to 256 registers).
template <int CLASS>
constexpr int waves = CLASS <= 16 ? 5 : (CLASS <= 22 ? 4 : 3);

// How a length runs: n = a b with a <= b, `threads` = b per line, the LDS
// pitches of the exchange (k1 rows of `pitch`, lines `line` apart, both odd).
struct plan
{
	int32_t n;
	int32_t a;
	int32_t b;
	int32_t pitch;
	int32_t line;
	int32_t lines; // per block
	int32_t kind;  // the class: 16, 22 or 32
};

// The plan of a length, or a plan of n = 0 when no pair of register lengths
// gives it (or it is too short to fill a wavefront's lanes).
plan make_plan(int64_t n);

// The transform of one line of the block: `load(i)` gives element i < n,
// `store(k, X)` takes coefficient k. `line` is the line's part of the exchange
// buffer, `tw` holds exp(-2 pi i m / n). Every thread of the block calls it (it
// holds a barrier); with LOAD_LDS or STORE_LDS another barrier lets the loads
// or stores use the exchange buffer itself. Step 1 runs on threads j < b, step
// 2 on j < a.
template <int CLASS, bool LOAD_LDS, bool STORE_LDS, typename Load, typename Store>
__device__ __forceinline__ void transform_line(const plan &p, float2 *line, const float2 *tw, int j, float sign,
	Load &&load, Store &&store)
{
	with_radix<CLASS>(p.a, [&](auto radix)
		{
			constexpr int R = decltype(radix)::value;
			float2 v[R];
			if (j < p.b)
			{
#pragma unroll
				for (int a = 0; a < R; ++a)
				{
					v[a] = load(j + p.b * a);
				}
			}
			if (LOAD_LDS)
			{
				__syncthreads();
			}
			if (j < p.b)
			{
				dft_any<R>(v, sign);
#pragma unroll
				for (int k = 0; k < R; ++k)
				{
					float2 w = tw[j * k];
					w.y *= -sign;
					line[k * p.pitch + j] = k == 0 ? v[k] : cmul(v[k], w);
				}
			}
		});
	__syncthreads();
	with_radix<CLASS>(p.b, [&](auto radix)
		{
			constexpr int R = decltype(radix)::value;
			float2 v[R];
			if (j < p.a)
			{
#pragma unroll
				for (int b = 0; b < R; ++b)
				{
					v[b] = line[j * p.pitch + b];
				}
				dft_any<R>(v, sign);
			}
			if (STORE_LDS)
			{
				__syncthreads();
			}
			if (j < p.a)
			{
#pragma unroll
				for (int k = 0; k < R; ++k)
				{
					store(j + p.a * k, v[k]);
				}
			}
		});
}

// Stages the twiddles of a plan into LDS (n values).
__device__ __forceinline__ void stage_twiddles(const plan &p, float2 *twl, const float2 *tw, int t, int threads)
{
	for (int i = t; i < p.n; i += threads)
	{
		twl[i] = tw[i];
	}
}

// Bytes of LDS of a block: the exchange and the twiddles.
inline std::size_t shared_bytes(const plan &p)
{
	return sizeof(float2) * (static_cast<std::size_t>(p.lines) * p.line + p.n);
}

// Blocks that take `per` of `count` lines each (a whole number per XCD).
inline unsigned blocks_for(int64_t count, int64_t per)
{
	return xcd_grid(static_cast<unsigned>((count + per - 1) / per));
}

// Calls f with the class of a plan as a compile-time constant.
template <typename F>
void with_class(const plan &p, F &&f)
{
	if (p.kind == 16)
	{
		f(std::integral_constant<int, 16>());
	}
	else if (p.kind == 22)
	{
		f(std::integral_constant<int, 22>());
	}
	else
	{
		f(std::integral_constant<int, 32>());
	}
}

} // namespace two_factor

} // namespace rexlib_hip
