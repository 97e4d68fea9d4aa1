// Per-sample arithmetic of the insertion and the wavefront helpers its
// kernels share (the scatter, gather and binned schedules and the sample
// producers).
#pragma once

#include "insertion.hpp"

namespace rexlib_hip
{

constexpr int max_taps = 8;

// ---------------------------------------------------------------------------
// Per-sample arithmetic shared by the schedules
// ---------------------------------------------------------------------------

// Round-half-up |k| of an integer frequency, exactly: the largest s with
// 4 s^2 - 4 s + 1 <= 4 |k|^2 (row_insertion_kernel.inl:180-220). The float
// estimate floor(sqrt(|k|^2) + 1/2) is within one of it for every |k|^2
// below 2^31, so one step each way, by selects, makes it exact.
__device__ inline int shell_of(int kx, int ky)
{
	const int q = kx * kx + ky * ky;
	const int q4 = 4 * q;
	int s = static_cast<int>(sqrtf(static_cast<float>(q)) + 0.5f);
	s += (4 * s * s + 4 * s + 1 <= q4) ? 1 : 0;
	s -= (s > 0 && 4 * s * s - 4 * s + 1 > q4) ? 1 : 0;
	return s;
}

// The window over one axis: the first voxel and the tap weights.
template <int PROFILE>
struct window_taps;

// Box: round halves away from 0 (box_window.inl:16-34).
template <>
struct window_taps<REXLIB_HIP_BOX>
{
	static constexpr int taps = 1;
	__device__ static inline int first(const insertion_params &, float c)
	{
		return static_cast<int>(c + (c < 0.0f ? -0.5f : 0.5f));
	}
	// The same as a float (whole, exact below 2^24).
	__device__ static inline float first_float(const insertion_params &, float c)
	{
		return truncf(c + (c < 0.0f ? -0.5f : 0.5f));
	}
	__device__ static inline int place(const insertion_params &p, float c, float *w)
	{
		w[0] = 1.0f;
		return first(p, c);
	}
};

// Triangle: floor and the fraction (triangle_window.inl:16-38).
template <>
struct window_taps<REXLIB_HIP_TRIANGLE>
{
	static constexpr int taps = 2;
	__device__ static inline int first(const insertion_params &, float c)
	{
		const int t = static_cast<int>(c);
		return t - (c < static_cast<float>(t) ? 1 : 0);
	}
	__device__ static inline float first_float(const insertion_params &, float c)
	{
		return floorf(c);
	}
	__device__ static inline int place(const insertion_params &p, float c, float *w)
	{
		const int below = first(p, c);
		const float f = c - static_cast<float>(below);
		w[0] = 1.0f - f;
		w[1] = f;
		return below;
	}
};

// Kaiser-Bessel: table with linear interpolation (kaiser_bessel_window.inl:65-136).
template <>
struct window_taps<REXLIB_HIP_KAISER_BESSEL>
{
	static constexpr int taps = max_taps;
	__device__ static inline int first(const insertion_params &p, float c)
	{
		const float low = c - p.kb_half_width;
		const int t = static_cast<int>(low);
		return t - (low < static_cast<float>(t) ? 1 : 0) + 1;
	}
	__device__ static inline float first_float(const insertion_params &p, float c)
	{
		return floorf(c - p.kb_half_width) + 1.0f;
	}
	// Weights of the first COUNT taps (at most p.taps are nonzero). Every
	// table entry is loaded before any is used, without a branch, so that the
	// loads of a sample's axes are in flight together.
	template <int COUNT = max_taps>
	__device__ static inline int place(const insertion_params &p, float c, float *w)
	{
		// Both entries of an interpolation by one 8-byte load (4-byte aligned).
		struct __attribute__((packed, aligned(4))) pair
		{
			float below, above;
		};
		const int first = window_taps::first(p, c);
		pair entry[COUNT];
		float fraction[COUNT];
#pragma unroll
		for (int tap = 0; tap < COUNT; ++tap)
		{
			const float d = fabsf(static_cast<float>(first + tap) - c);
			const float position = d * p.kb_scale;
			const int step = static_cast<int>(position);
			const int index = step < p.kb_count ? step : p.kb_count + 1;
			fraction[tap] = position - static_cast<float>(index);
			entry[tap] = *reinterpret_cast<const pair *>(p.kb_table + static_cast<unsigned>(index));
		}
#pragma unroll
		for (int tap = 0; tap < COUNT; ++tap)
		{
			w[tap] = tap < p.taps ? entry[tap].below + fraction[tap] * (entry[tap].above - entry[tap].below) : 0.0f;
		}
		return first;
	}
};

// The sample of stored element (row, column) of slice s: its value v * r *
// (numerator weight) before the sign, its denominator weight, and false when
// it is not inserted.
// sin x for the CTF phase x (radians, |x| up to about 1e5). Cody-Waite
// reduction: x = k pi/2 + r with the product k pi/2 taken in double, so that
// r is exact to float precision; then the Taylor polynomials of sin (through
// r^9) and cos (through r^8) on |r| <= pi/4, whose truncation errors are
// below 2e-9 and 2.5e-8, selected and signed by the quadrant k mod 4.
// (The library sinf takes its multi-word reduction for phases of a few
// hundred radians, several times the cost of the whole sample.)
__host__ __device__ inline float phase_sin(float x)
{
	const float k = rintf(x * 0.636619772367581343f); // 2 / pi
	const float r = static_cast<float>(fma(-static_cast<double>(k), 1.5707963267948966192, static_cast<double>(x)));
	const float r2 = r * r;
	const float s = r + r * r2 * (-1.0f / 6.0f + r2 * (1.0f / 120.0f + r2 * (-1.0f / 5040.0f + r2 * (1.0f / 362880.0f))));
	const float c = 1.0f + r2 * (-0.5f + r2 * (1.0f / 24.0f + r2 * (-1.0f / 720.0f + r2 * (1.0f / 40320.0f))));
	const int q = static_cast<int>(k) & 3;
	const float v = (q & 1) ? c : s;
	return (q & 2) ? -v : v;
}

// chi(k) of a slice (contrast_transfer_function.inl:73-87), with the fused
// products written out: left to the compiler, the kernels that prepare samples
// contract the sum differently, and chi, hundreds of radians, moves by its
// last bit between them.
__device__ inline float ctf_chi(const slice_entry &e, float aberration, float xx, float yy, float xy)
{
	const float norm = xx + yy;
	const float radial = e.ctf_radial * norm;
	const float astigmatic = __builtin_fmaf(e.ctf_axial, xx - yy, radial);
	const float defocus = __builtin_fmaf(e.ctf_diagonal, xy, astigmatic);
	return __builtin_fmaf(-(norm * norm), aberration, defocus) + e.ctf_phase;
}

// The element's value comes from `load`, called only for inserted samples.
template <int VARIANT, typename Load>
__device__ inline bool prepare_value(const insertion_params &p, const slice_entry &e, int64_t s, int row,
	int column, Load load, float2 &value, float &count)
{
	const int n = p.n;
	if ((n % 2 == 0) && (row == n / 2 || column == n / 2))
	{
		return false;
	}
	const int ky = row <= n / 2 ? row : row - n;
	const int kx = column;
	const int shell = shell_of(kx, ky);
	if (shell > e.last_shell)
	{
		return false;
	}
	const float r = p.radial[e.radial_offset + shell * p.radial_s0];
	if (r == 0.0f)
	{
		return false;
	}
	const float2 x = load();
	const float2 *table = p.tables + s * static_cast<int64_t>(p.h + n);
	const float2 shifted = cmul(x, table[column]);
	const float2 v = cmul(shifted, table[p.h + row]);
	float numerator_weight = 1.0f;
	float denominator_weight = 1.0f;
	if (VARIANT == variant_weighted)
	{
		denominator_weight = p.extra[e.extra_offset + row * p.extra_s0 + column * p.extra_s1];
	}
	else if (VARIANT == variant_ctf)
	{
		// contrast_transfer_function.inl:73-87 and ctf_weight.inl:72-103.
		const float fx = static_cast<float>(kx);
		const float fy = static_cast<float>(ky);
		const float xx = fx * fx;
		const float yy = fy * fy;
		const float chi = ctf_chi(e, static_cast<float>(p.ctf_aberration), xx, yy, fx * fy);
		numerator_weight = phase_sin(chi);
		denominator_weight = numerator_weight * numerator_weight;
	}
	const float scale = r * numerator_weight;
	value = make_float2(v.x * scale, v.y * scale);
	count = r * denominator_weight;
	return true;
}

template <int VARIANT>
__device__ inline bool prepare_sample(const insertion_params &p, const slice_entry &e, int64_t s, int row,
	int column, float2 &value, float &count)
{
	return prepare_value<VARIANT>(p, e, s, row, column,
		[&] { return p.slices[e.slice_offset + row * p.slice_s0 + column * p.slice_s1]; }, value, count);
}

// Volume position of sample k_x of row k_y with the sign applied.
__device__ inline void sample_position(const slice_entry &e, int kx, int ky, float sign, float *c)
{
#pragma clang fp contract(off)
	const float fx = static_cast<float>(kx);
	for (int a = 0; a < 3; ++a)
	{
		const float base = static_cast<float>(static_cast<double>(ky) * (static_cast<double>(sign) * e.y_step[a]));
		const float step = sign * e.x_step[a];
		c[a] = base + fx * step;
	}
}

// Volume phase of the stored voxel (x, sy, sz), applied to a contribution.
template <bool ODD>
__device__ inline float2 volume_phase(const insertion_params &p, float2 value, int x, int sy, int sz)
{
	if (ODD)
	{
		return cmul(cmul(cmul(value, p.volume_phase[x]), p.volume_phase[sy]), p.volume_phase[sz]);
	}
	return ((x + sy + sz) & 1) ? make_float2(-value.x, -value.y) : value;
}


// A prepared sample of a slice: v r w (the value with its radial and
// numerator weights) and r w_den, 12 bytes; zero when not inserted.
struct prepared_sample
{
	float re;
	float im;
	float den;
};

// Inclusive prefix sum over the 64 lanes by DPP row shifts (within rows of
// 16) and row broadcasts (across them); lanes without a source add 0.
__device__ __forceinline__ int wave_inclusive_scan(int v)
{
	v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true); // row_shr:1
	v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true); // row_shr:2
	v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true); // row_shr:4
	v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true); // row_shr:8
	v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, true); // row_bcast:15
	v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, true); // row_bcast:31
	return v;
}

// Prefix maximum over the 64 lanes (lane i gets the maximum of lanes 0..i),
// by DPP row shifts within rows of 16 and row broadcasts across them.
// Lanes without a source read 0 (bound_ctrl), which leaves the result
// unchanged wherever lane 0 holds a value of at least 0.
__device__ __forceinline__ int wave_prefix_max(int v)
{
	v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true)); // row_shr:1
	v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true)); // row_shr:2
	v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true)); // row_shr:4
	v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true)); // row_shr:8
	v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, true)); // row_bcast:15
	v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, true)); // row_bcast:31
	return v;
}

// A float held by lane `lane` (uniform), as a scalar.
__device__ inline float lane_value(float v, int lane)
{
	return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// Keeps the compiler from moving LDS accesses across it: the taps of other
// lanes may alias, which it cannot see.
__device__ inline void lds_order()
{
	__asm__ __volatile__("" ::: "memory");
}

// The shell of an element of a slice of extent n <= 720, from |k|^2 as a float
// (exact below 2^24): no |k| is closer than 1 / (8 s) to the boundary s + 1/2,
// 2.4e-4 for the 509 shells of that extent, and the hardware square root with
// the addition stays within 5e-5. Three instructions; shell_of takes 30 with
// its rounded square root and four quarter-rate products.
constexpr int largest_quick_shell = 720;

__device__ inline int quick_shell(float norm)
{
	return static_cast<int>(__builtin_amdgcn_sqrtf(norm) + 0.5f);
}

// The brick schedule reads the elements of a slice with k_x and k_y inside the
// Nyquist frequency and shell <= last_shell; up to this extent the clipped
// rows end exactly at the shell ((2 L + 1)^2 < 2^24 and its square root apart
// from every integer), so the others are not written.
constexpr int largest_exact_clip = 4095;

// prepare_value without branches, for prepare_kernel and the fused column
// passes: every load is in bounds whatever the sample (the radial index is
// clamped to the last shell, the phase tables cover every row and column),
// and the sample is zeroed afterwards where prepare_value rejects it, so the
// loads of several elements can be in flight together. The arithmetic is
// prepare_value's, in the same order. `radial` is the slice's radial weights,
// `y_table` its row phases. `read` says whether the brick schedule reads it.
template <int VARIANT>
__device__ inline prepared_sample prepare_unbranched(const insertion_params &p, const slice_entry &e,
	const float *radial, const float2 *y_table, float2 x_phase, int row, int column, float2 x, bool &read)
{
	const int n = p.n;
	const int ky = row <= n / 2 ? row : row - n;
	const float fx = static_cast<float>(column);
	const float fy = static_cast<float>(ky);
	const float xx = fx * fx;
	const float yy = fy * fy;
	const float norm = xx + yy;
	const int shell = n <= largest_quick_shell ? quick_shell(norm) : shell_of(column, ky);
	const bool nyquist = (n % 2 == 0) && (row == n / 2 || column == n / 2);
	const int clamped = min(shell, max(e.last_shell, 0));
	const float r = p.radial_s0 == 1 ? radial[static_cast<unsigned>(clamped)] : radial[clamped * p.radial_s0];
	const float2 y_phase = y_table[static_cast<unsigned>(row)];
	float numerator_weight = 1.0f;
	float denominator_weight = 1.0f;
	if (VARIANT == variant_weighted)
	{
		denominator_weight = p.extra[e.extra_offset + row * p.extra_s0 + column * p.extra_s1];
	}
	else if (VARIANT == variant_ctf)
	{
		const float chi = ctf_chi(e, static_cast<float>(p.ctf_aberration), xx, yy, fx * fy);
		numerator_weight = phase_sin(chi);
		denominator_weight = numerator_weight * numerator_weight;
	}
	const float2 v = cmul(cmul(x, x_phase), y_phase);
	const float scale = r * numerator_weight;
	const bool within = !nyquist && shell <= e.last_shell;
	read = within || n > largest_exact_clip;
	return within && r != 0.0f ? prepared_sample{v.x * scale, v.y * scale, r * denominator_weight} :
		prepared_sample{0.0f, 0.0f, 0.0f};
}

} // namespace rexlib_hip
