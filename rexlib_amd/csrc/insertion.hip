// Fourier slice insertion on gfx950.
//
// Contract: include/rexlib/em/ops/reconstruction/insert_slices_operation.hpp:31-112
// (and the CTF / weighted variants). The per-sample arithmetic follows the
// reference's CPU row kernel in float32
// (src/backends/cpu/builders/em/reconstruction/row_insertion_kernel.inl:132-361):
//   - the row base k_y * Y is formed in double and rounded, the position is
//     base + k_x * X in float (row_insertion_kernel.inl:157-166);
//   - the shell is round-half-up |k|, exact in integers (row_insertion_kernel.inl:180-220);
//   - v = X(k) * x_phase * y_phase, then times r * (numerator weight), the
//     imaginary part negated for the -k copy (row_insertion_kernel.inl:222-279);
//   - the volume phase is (-1)^(x+y+z) for even N and a product of three table
//     entries for odd N (alternating_sign.inl:10-20, tabulated_phase.inl:12-37).
//
// Two schedules accumulate the same sums:
//   - scatter: one thread per stored slice element, float atomics into the
//     accumulators in HBM (every window, every size);
//   - brick: each workgroup owns a brick of the volume in LDS, gathers the
//     samples of every slice that reach it, and adds the brick to HBM once.
//     This is the GPU form of the reference's tile-owned schedule
//     (slice_insertion_functor.inl:105-156, 271-465).
#include "fft_device.hpp"
#include "fft_two.hpp"
#include "launch.hpp"
#include "sample.hpp"
#include "section_bounds.hpp"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdlib>
#include <tuple>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

namespace rexlib_hip
{

namespace
{

constexpr double pi_d = 3.14159265358979323846;

// ---------------------------------------------------------------------------
// Settle: one block per slice.
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(128) void settle_kernel(insertion_params p)
{
	__shared__ int last_shells[2];
	const int n = p.n;
	const int h = p.h;
	for (int64_t s = blockIdx.x; s < p.slice_count; s += gridDim.x)
	{
		const int64_t kept = s / p.map.reduced_count;
		const int64_t red = s % p.map.reduced_count;
		const auto offset = [&](int slot)
		{
			return kept_offset(p.map, slot, kept) + reduced_offset(p.map, slot, red);
		};
		const float *t = p.transforms + offset(slot_transforms);
		const auto at = [&](int r, int c)
		{
			return static_cast<double>(t[r * p.transform_s0 + c * p.transform_s1]);
		};
		const double scale = static_cast<double>(p.big) / static_cast<double>(n);
		const double centre = static_cast<double>(n / 2);
		const int64_t radial_offset = offset(slot_radial);

		// The last shell with a weight: the threads scan the shells side by side
		// (one thread after another through 129 loads took 20 us of a call).
		const float *radial = p.radial + radial_offset;
		int found = -1;
		for (int shell = threadIdx.x; shell < h; shell += blockDim.x)
		{
			found = radial[shell * p.radial_s0] != 0.0f ? shell : found;
		}
		for (int offset_lanes = 32; offset_lanes > 0; offset_lanes /= 2)
		{
			found = max(found, __shfl_xor(found, offset_lanes, 64));
		}
		__syncthreads(); // the previous slice's value is read
		if ((threadIdx.x & 63) == 0)
		{
			last_shells[threadIdx.x >> 6] = found;
		}
		__syncthreads();

		if (threadIdx.x == 0)
		{
			slice_entry e;
			bool finite = true;
			for (int a = 0; a < 3; ++a)
			{
				const double xs = at(0, a) * scale;
				const double ys = at(1, a) * scale;
				finite = finite && isfinite(xs) && isfinite(ys);
				e.x_step[a] = static_cast<float>(xs);
				e.y_step[a] = ys;
			}
			const int last = max(last_shells[0], last_shells[1]);
			// A non-finite frame bounds no rows (src/backends/cpu/kernels/row_interval.cpp).
			e.last_shell = finite ? last : -1;
			e.ctf_radial = e.ctf_axial = e.ctf_diagonal = e.ctf_phase = 0.0f;
			{
				const float x0 = e.x_step[0], x1 = e.x_step[1], x2 = e.x_step[2];
				const float y0 = static_cast<float>(e.y_step[0]);
				const float y1 = static_cast<float>(e.y_step[1]);
				const float y2 = static_cast<float>(e.y_step[2]);
				slice_plane plane;
				plane.normal[0] = x1 * y2 - x2 * y1;
				plane.normal[1] = x2 * y0 - x0 * y2;
				plane.normal[2] = x0 * y1 - x1 * y0;
				plane.reach = e.last_shell < 0 ? -1.0e30f : (static_cast<float>(e.last_shell) + 0.5f) * 1.001f *
					sqrtf(x0 * x0 + x1 * x1 + x2 * x2 + y0 * y0 + y1 * y1 + y2 * y2) + 1e-3f;
				p.planes[s] = plane;
			}
			e.extra_offset = p.extra != nullptr ? offset(slot_extra) : 0;
			if (p.variant == variant_ctf)
			{
				// contrast_transfer_function.inl:25-70: coefficients in double,
				// rounded to float.
				const float *c = p.extra + e.extra_offset;
				const double du = c[0];
				const double dv = c[p.extra_s0];
				const double angle = c[2 * p.extra_s0];
				const double phase = c[3 * p.extra_s0];
				const double half_difference = 0.5 * (du - dv);
				e.ctf_radial = static_cast<float>(p.ctf_defocus_scale * 0.5 * (du + dv));
				e.ctf_axial = static_cast<float>(p.ctf_defocus_scale * half_difference * cos(2.0 * angle));
				e.ctf_diagonal = static_cast<float>(
					2.0 * p.ctf_defocus_scale * half_difference * sin(2.0 * angle));
				e.ctf_phase = static_cast<float>(phase + p.ctf_phase0);
			}
			e.slice_offset = offset(slot_slices);
			e.radial_offset = radial_offset;
			e.numerator_offset = kept_offset(p.map, slot_numerator_out, kept);
			e.denominator_offset = kept_offset(p.map, slot_denominator_out, kept);
			p.entries[s] = e;
		}

		// Shift phases exp(2 pi i k (c + t) / n) (axis_phase.inl:14-36), in
		// double (angles in units of pi), rounded to float.
		float2 *table = p.tables + s * static_cast<int64_t>(h + n);
		const double x_scale = 2.0 * (centre + at(0, 3)) / static_cast<double>(n);
		const double y_scale = 2.0 * (centre + at(1, 3)) / static_cast<double>(n);
		for (int j = threadIdx.x; j < h + n; j += blockDim.x)
		{
			double angle;
			if (j < h)
			{
				angle = x_scale * static_cast<double>(j);
			}
			else
			{
				const int r = j - h;
				const int f = r <= n / 2 ? r : r - n;
				angle = y_scale * static_cast<double>(f);
			}
			double sn, cs;
			sincospi(angle, &sn, &cs);
			table[j] = make_float2(static_cast<float>(cs), static_cast<float>(sn));
		}
	}
}

// Kaiser-Bessel table: entry i holds the window at i / count of the
// half-width, then two zeros (kaiser_bessel_window.inl:18-50).
__device__ double bessel_i0_series(double x)
{
	const double quarter_square = 0.25 * x * x;
	double sum = 1.0;
	double term = 1.0;
	for (double k = 1.0; k < 500.0; k += 1.0)
	{
		term *= quarter_square / (k * k);
		sum += term;
		if (term <= 2.220446049250313e-16 * sum)
		{
			break;
		}
	}
	return sum;
}

__global__ void kb_table_kernel(float *table, int count, double shape)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= count + 3)
	{
		return;
	}
	if (i > count)
	{
		table[i] = 0.0f;
		return;
	}
	const double ratio = static_cast<double>(i) / static_cast<double>(count);
	table[i] = static_cast<float>(bessel_i0_series(shape * sqrt(1.0 - ratio * ratio)) /
		bessel_i0_series(shape));
}

// exp(-2 pi i f(j) C / N) for the stored index j of an odd N (tabulated_phase.inl:12-22).
__global__ void volume_phase_kernel(float2 *table, int big)
{
	const int j = blockIdx.x * blockDim.x + threadIdx.x;
	if (j >= big)
	{
		return;
	}
	const int half = big / 2;
	const int f = j <= half ? j : j - big;
	const double angle = 2.0 * pi_d * (-static_cast<double>(half)) * static_cast<double>(f) /
		static_cast<double>(big);
	double sn, cs;
	sincos(angle, &sn, &cs);
	table[j] = make_float2(static_cast<float>(cs), static_cast<float>(sn));
}

// Out-of-place insertions start from a copy of the accumulators.
__global__ void copy_accumulators_kernel(insertion_params p, const float2 *num_in, int64_t ni0, int64_t ni1,
	int64_t ni2, const float *den_in, int64_t di0, int64_t di1, int64_t di2)
{
	const int64_t volume = static_cast<int64_t>(p.big) * p.big * p.half;
	const int64_t total = volume * p.map.kept_count;
	for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < total;
		i += static_cast<int64_t>(gridDim.x) * blockDim.x)
	{
		const int64_t kept = i / volume;
		int64_t v = i % volume;
		const int64_t x = v % p.half;
		v /= p.half;
		const int64_t y = v % p.big;
		const int64_t z = v / p.big;
		const float2 a = num_in[kept_offset(p.map, slot_numerator, kept) + z * ni0 + y * ni1 + x * ni2];
		const float b = den_in[kept_offset(p.map, slot_denominator, kept) + z * di0 + y * di1 + x * di2];
		p.numerator[kept_offset(p.map, slot_numerator_out, kept) + z * p.num_s0 + y * p.num_s1 + x * p.num_s2] = a;
		p.denominator[kept_offset(p.map, slot_denominator_out, kept) + z * p.den_s0 + y * p.den_s1 + x * p.den_s2] = b;
	}
}

// ---------------------------------------------------------------------------
// Scatter schedule: a thread per stored slice element, atomics in HBM.
// ---------------------------------------------------------------------------

template <int PROFILE, int VARIANT, bool ODD>
__global__ __launch_bounds__(256) void scatter_kernel(insertion_params p)
{
	// A slice holds n (n/2 + 1) < 2^31 elements: 32-bit indices (a 64-bit
	// division per element would cost more than the sample itself).
	const int elements32 = p.n * p.h;
	const int idx = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
	if (idx >= elements32)
	{
		return;
	}
	const int row = static_cast<int>(static_cast<unsigned>(idx) / static_cast<unsigned>(p.h));
	const int column = idx - row * p.h;
	const int big = p.big;
	const int half_extent = big / 2;
	for (int64_t s = blockIdx.y; s < p.slice_count; s += gridDim.y)
	{
		const slice_entry &e = p.entries[s];
		if (e.last_shell < 0)
		{
			continue;
		}
		float2 value;
		float count;
		if (!prepare_sample<VARIANT>(p, e, s, row, column, value, count))
		{
			continue;
		}
		const int ky = row <= p.n / 2 ? row : row - p.n;
		float2 *num = p.numerator + e.numerator_offset;
		float *den = p.denominator + e.denominator_offset;
		for (int sign_index = 0; sign_index < 2; ++sign_index)
		{
			if (sign_index == 1 && column == 0)
			{
				break;
			}
			const float sign = sign_index == 0 ? 1.0f : -1.0f;
			const float2 signed_value = sign_index == 0 ? value : cconj(value);
			float c[3];
			sample_position(e, column, ky, sign, c);
			float wx[max_taps], wy[max_taps], wz[max_taps];
			const int x0 = window_taps<PROFILE>::place(p, c[0], wx);
			const int y0 = window_taps<PROFILE>::place(p, c[1], wy);
			const int z0 = window_taps<PROFILE>::place(p, c[2], wz);
			const int taps = PROFILE == REXLIB_HIP_KAISER_BESSEL ? p.taps : window_taps<PROFILE>::taps;
			for (int tz = 0; tz < taps; ++tz)
			{
				const int z = z0 + tz;
				if (z < -half_extent || z > half_extent)
				{
					continue;
				}
				const int sz = z < 0 ? z + big : z;
				for (int ty = 0; ty < taps; ++ty)
				{
					const int y = y0 + ty;
					if (y < -half_extent || y > half_extent)
					{
						continue;
					}
					const int sy = y < 0 ? y + big : y;
					const float wzy = wz[tz] * wy[ty];
					for (int tx = 0; tx < taps; ++tx)
					{
						const int x = x0 + tx;
						if (x < 0 || x > half_extent)
						{
							continue;
						}
						const float w = wzy * wx[tx];
						const float2 contribution = volume_phase<ODD>(p,
							make_float2(signed_value.x * w, signed_value.y * w), x, sy, sz);
						float2 *target = num + sz * p.num_s0 + sy * p.num_s1 + x * p.num_s2;
						atomicAdd(&target->x, contribution.x);
						atomicAdd(&target->y, contribution.y);
						atomicAdd(den + sz * p.den_s0 + sy * p.den_s1 + x * p.den_s2, count * w);
					}
				}
			}
		}
	}
}

template <int PROFILE, int VARIANT>
void launch_scatter(const insertion_params &p, hipStream_t stream)
{
	const int64_t elements = static_cast<int64_t>(p.n) * p.h;
	const dim3 block(256);
	const dim3 grid(static_cast<unsigned>((elements + 255) / 256),
		static_cast<unsigned>(std::min<int64_t>(p.slice_count, 65535)));
	if (p.big % 2 == 1)
	{
		scatter_kernel<PROFILE, VARIANT, true><<<grid, block, 0, stream>>>(p);
	}
	else
	{
		scatter_kernel<PROFILE, VARIANT, false><<<grid, block, 0, stream>>>(p);
	}
}

template <int VARIANT>
void dispatch_scatter(const insertion_params &p, hipStream_t stream)
{
	switch (p.profile)
	{
	case REXLIB_HIP_BOX:
		launch_scatter<REXLIB_HIP_BOX, VARIANT>(p, stream);
		break;
	case REXLIB_HIP_TRIANGLE:
		launch_scatter<REXLIB_HIP_TRIANGLE, VARIANT>(p, stream);
		break;
	default:
		launch_scatter<REXLIB_HIP_KAISER_BESSEL, VARIANT>(p, stream);
		break;
	}
}


// ---------------------------------------------------------------------------
// Brick schedule: one wavefront owns a brick of the volume in LDS.
//
// First, a prepare kernel computes every stored element of every slice once:
// v * r * (numerator weight) and r * (denominator weight), or zeros when the
// element is not inserted (row_insertion_kernel.inl:180-279).
//
// Bricks tile the first-tap cells of the volume (signed x in [0, N/2], y and
// z in [-N/2, N/2], each range extended downwards by taps - 1 so that every
// sample reaching the volume has its first tap in some brick). A sample copy
// belongs to the brick holding its first tap, so each copy is added by one
// brick; the brick's LDS holds its cells and the taps - 1 voxels above them.
//
// The wavefront tests 64 slices at a time for planes that pass near the
// brick and queues the few that do; for 64 queued slices at once it bounds
// the rows that can hold their samples (bound_section, bound_rows) and clips
// each row to them (clip_row of src/backends/cpu/kernels/row_interval.cpp,
// restated per brick as the reference restates it per tile,
// slice_insertion_functor.inl:391-440). The rows of the queued slices are
// packed densely over the lanes (64 rows at a time, each with its base
// position, step and first sample in its lane's registers), and their samples
// over the lanes (64 at a time), so a lane carries a sample whatever slice it
// comes from. Bounding the 2.2 hits of each 64 slices on their own spent half
// of the vector instructions, and the queue took a launch of 4,096 slices of
// 256^2 into 256^3 from 1.9 to 1.18 ms. It is bound by LDS now: the index unit is
// busy 84 % of the CU cycles, 48 % of that bank conflicts, the vector units 56 %.
//
// The samples are added by plain LDS read-modify-write, not LDS float
// atomics (which retire at about a third of a lane per clock per CU on
// gfx950, against eight for a read-modify-write). Per round every lane
// holding a sample claims its first-tap cell (a byte per cell: it writes its
// lane, then reads it back); the lanes that read their own lane add their
// taps one after another, the others keep their sample for the next round,
// whose new samples go to the free lanes only. (Smaller Kaiser-Bessel calls make
// the 64 lanes the taps of one sample instead: wide_round, kaiser_bessel_bricks.)
// No two lanes of one tap
// instruction then touch one voxel (a tap is a constant offset from the
// cell). LDS runs a wavefront's accesses in program order and lds_order
// keeps the compiler from moving them; the wavefront is the brick's only
// writer, so there is no barrier anywhere.
//
// The volume phase exp(-2 pi i g C / N) depends on the voxel alone, so the
// brick sums v * w and applies the phase once per voxel when it adds the
// brick to the accumulators (alternating_sign.inl:10-20,
// tabulated_phase.inl:12-37).
//
// Every plane passes through the origin, so bricks near it see every slice
// and bricks far out see few (about 13 / r of them). A task is a brick and a
// share of the slices: heavy bricks are split, and the heaviest tasks start
// first. Voxels that only one task can touch are added to the accumulators
// by plain read-add-write; the others (the taps - 1 layers at each face that
// the neighbouring bricks also reach, every voxel of a split brick, and bricks
// holding the y or z frequency +-N/2 of an even N, two signed frequencies of
// one stored element) add with atomics. Sparse calls take bricks that own
// voxels instead and write each once (bricks_own_voxels).
// ---------------------------------------------------------------------------


// How the rounds of a brick add its samples (see above): each lane its own,
// after claiming its cell, or one sample after another by all 64 lanes, with all
// 4 taps per axis of the layout or fewer.
enum brick_rounds : int
{
	claimed_rounds = 0,
	wide_rounds = 1,
	wide_narrow_rounds = 2
};

// Taps per axis an LDS brick is laid out for: the window's own (box 1,
// triangle 2), at most 4 for Kaiser-Bessel windows on this schedule.
template <int PROFILE>
struct brick_reach
{
	static constexpr int taps = PROFILE == REXLIB_HIP_BOX ? 1 : (PROFILE == REXLIB_HIP_TRIANGLE ? 2 : 4);
};

// LDS pitches of a brick of lx x ly voxels per plane. Up to 2 taps: odd, so
// that lanes stepping along any axis fall in different banks. With 4 taps the
// 64 lanes of an access are the 4 x 4 x 4 taps of one sample: a y pitch of 4
// modulo 8 and a z pitch of 16 modulo 32 put every 32 of them in 32 different
// residues, without a bank conflict.
constexpr int brick_pitch_y(bool wide, int lx)
{
	return wide ? (lx + 3) / 8 * 8 + 4 : (lx % 2 == 0 ? lx + 1 : lx);
}

constexpr int brick_pitch_z(bool wide, int pitch_y, int ly)
{
	return wide ? (pitch_y * ly + 15) / 32 * 32 + 16 : (pitch_y * ly) % 2 == 0 ? pitch_y * ly + 1 : pitch_y * ly;
}

// LDS layout of a brick of first-tap cells EX x EY x EZ with the taps - 1
// voxels above them.
template <int T, bool WIDE, int EX, int EY, int EZ>
struct brick_layout
{
	static constexpr int lx = EX + T - 1;
	static constexpr int ly = EY + T - 1;
	static constexpr int lz = EZ + T - 1;
	static constexpr int pitch_y = brick_pitch_y(WIDE, lx);
	static constexpr int pitch_z = brick_pitch_z(WIDE, pitch_y, ly);
	static_assert(pitch_y >= lx && pitch_z >= pitch_y * ly, "the pitches hold a row and a plane");
	static constexpr int voxels = pitch_z * lz;
	static constexpr int cells = EX * EY * EZ;
};

struct brick_box
{
	int lo[3];  // signed (x, y, z) of the first cell
	int ext[3]; // cells along (x, y, z)
	bool alias_free;
};

// The accumulators the sums are added to, read by bricks that own voxels:
// the caller's inputs (first chunk of an out-of-place call), else the outputs.
struct accumulator_input
{
	const float2 *numerator;
	int64_t num_s0, num_s1, num_s2;
	const float *denominator;
	int64_t den_s0, den_s1, den_s2;
	int num_slot; // whose batch offsets the pointers take
	int den_slot;
	bool in_place;
};

__device__ inline brick_box unpack_brick(int4 b)
{
	brick_box box;
	box.lo[0] = b.x;
	box.lo[1] = b.y;
	box.lo[2] = b.z;
	box.ext[0] = b.w & 0xff;
	box.ext[1] = (b.w >> 8) & 0xff;
	box.ext[2] = (b.w >> 16) & 0xff;
	box.alias_free = ((b.w >> 24) & 1) != 0;
	return box;
}

template <int VARIANT>
__global__ __launch_bounds__(256) void prepare_kernel(insertion_params p, slice_chunk chunk, prepared_sample *prepared)
{
	// A slice holds n (n/2 + 1) < 2^31 elements: 32-bit indices (a 64-bit
	// division per element would cost more than the sample itself).
	const int elements32 = p.n * p.h;
	const int64_t elements = elements32;
	const int idx = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
	if (idx >= elements32)
	{
		return;
	}
	const int row = static_cast<int>(static_cast<unsigned>(idx) / static_cast<unsigned>(p.h));
	const int column = idx - row * p.h;
	const int64_t slices = p.map.kept_count * chunk.count;
	for (int64_t j = blockIdx.y; j < slices; j += gridDim.y)
	{
		const int64_t kept = j / chunk.count;
		const int64_t s = kept * p.map.reduced_count + chunk.begin + j % chunk.count;
		const slice_entry &e = p.entries[s];
		// Branch-free, as in the fused column pass: every element is loaded
		// and the rejected ones zeroed afterwards.
		const float2 *table = p.tables + s * static_cast<int64_t>(p.h + p.n);
		const float2 x = p.slices[e.slice_offset + row * p.slice_s0 + column * p.slice_s1];
		bool read;
		const prepared_sample sample = prepare_unbranched<VARIANT>(p, e, p.radial + e.radial_offset, table + p.h,
			table[column], row, column, x, read);
		if (read)
		{
			prepared[j * elements + idx] = sample;
		}
	}
}

// The rows [begin, end) of row-transformed slices that may hold other values
// than zero (the image rows of a padded slice); the column passes read only
// these.
struct row_range
{
	int begin;
	int end;
};

// The column transforms of 256-point slices fused with the preparation.
// The rows of each slice are transformed already (in p.slices, at the
// slices' own offsets and strides); a block transforms 16 columns k_x of one of
// the chunk's slices by the four-step decomposition and writes the prepared
// samples of those columns directly, so the finished spectra never pass
// through HBM. The Nyquist column k_x = n/2 holds no inserted sample and the
// brick schedule never reads it, so it is skipped: slice j of the chunk takes
// 8 blocks, and everything of the slice is uniform over a block (scalar
// registers; its row phases and radial weights in LDS). It was bound by its
// vector instructions (99 per sample and a 64-bit division chain per line, 66
// % of the SIMD cycles: 0.75 ms for 4,096 slices, 0.60 now). It and the 256-point
// row kernel keep their place beside the two-factor kernels that take 256 too:
// a launch of 4,096 images takes 2.29 ms through them, 2.37 through the others.
template <int VARIANT>
__global__ __launch_bounds__(256) void columns_prepare256_kernel(insertion_params p, slice_chunk chunk,
	row_range held, const float2 *tw, prepared_sample *prepared)
{
	constexpr int n = 256;
	constexpr int h = n / 2 + 1;
	constexpr int groups = n / 2 / fft256_lines; // of 16 columns per slice
	__shared__ float2 exchange[fft256_lines * fft256_line_stride];
	__shared__ float2 twl[n];
	__shared__ float2 row_phase[n];
	__shared__ float radial[h];
	const int t = threadIdx.x;
	const int l = t & (fft256_lines - 1);
	const int j = t / fft256_lines; // n1 in the first half of the transform, k1 in the second
	const unsigned block = xcd_block(blockIdx.x, gridDim.x);
	const int64_t jj = block / groups;
	if (jj >= p.map.kept_count * chunk.count)
	{
		return;
	}
	const int column = static_cast<int>(block % groups) * fft256_lines + l;
	const int64_t kept = p.map.kept_count == 1 ? 0 : jj / chunk.count;
	const int64_t slice = kept * p.map.reduced_count + chunk.begin + (jj - kept * chunk.count);
	const slice_entry &e = p.entries[slice];
	const float2 *table = p.tables + slice * static_cast<int64_t>(h + n);
	// Elements j + 16 k of the column, by pointer steps.
	const float2 *in = p.slices + e.slice_offset + column * p.slice_s1 + j * p.slice_s0;
	const int64_t in_step = 16 * p.slice_s0;
	float2 v[16];
#pragma unroll
	for (int k = 0; k < 16; ++k)
	{
		const int row = j + 16 * k;
		v[k] = row >= held.begin && row < held.end ? in[k * in_step] : make_float2(0.0f, 0.0f);
	}
	twl[t] = tw[t];
	row_phase[t] = table[h + t];
	if (t < h)
	{
		radial[t] = p.radial[e.radial_offset + t * p.radial_s0];
	}
	const float2 x_phase = table[column];
	__syncthreads();
	float2 *x = exchange + l * fft256_line_stride;
	fft256_four_step(v, x, twl, j, -1.0f);
	// The outputs go back to LDS (each thread to slots only it reads), so
	// the preparation loops over them without holding all 16.
	__syncthreads();
#pragma unroll
	for (int k2 = 0; k2 < 16; ++k2)
	{
		x[k2 * 17 + j] = v[k2];
	}
	prepared_sample *out = prepared + jj * static_cast<int64_t>(n * h) + j * h + column;
	// (The radial weights are in LDS at unit stride, the extent is 256.)
	insertion_params q = p;
	q.n = n;
	q.radial_s0 = 1;
#pragma unroll 4
	for (int k2 = 0; k2 < 16; ++k2)
	{
		bool read;
		const prepared_sample sample = prepare_unbranched<VARIANT>(q, e, radial, row_phase, x_phase, j + 16 * k2, column,
			x[k2 * 17 + j], read);
		if (read)
		{
			out[k2 * 16 * h] = sample;
		}
	}
}

// The same fusion for the other lengths the FFT kernels take: a block
// stages `group` columns of the chunk's slices in LDS, transforms them with
// the Stockham stages, and prepares every element from LDS. The lines are (slice j of the chunk,
// column), numbered j columns + column, where columns is n/2 for even n
// (the Nyquist column, never inserted, is skipped) and n/2 + 1 for odd n.
template <int VARIANT>
__global__ __launch_bounds__(256) void columns_prepare_kernel(insertion_params p, slice_chunk chunk, row_range held, fft_plan plan,
	const float2 *tw, int group, prepared_sample *prepared)
{
	extern __shared__ float2 lds[];
	const int n = plan.n;
	const int stride = n + 1;
	float2 *a = lds;
	float2 *b = lds + group * stride;
	float2 *twl = lds + 2 * group * stride;
	int64_t *line_slice = reinterpret_cast<int64_t *>(twl + n);
	int64_t *line_src = line_slice + group;
	int64_t *line_dst = line_src + group;
	int *line_column = reinterpret_cast<int *>(line_dst + group);
	for (int i = threadIdx.x; i < n; i += blockDim.x)
	{
		twl[i] = tw[i];
	}
	const int h = p.h;
	const int columns = n % 2 == 0 ? n / 2 : h;
	const int64_t elements = static_cast<int64_t>(n) * h;
	const int64_t total = p.map.kept_count * chunk.count * columns;
	for (int64_t first = xcd_block(blockIdx.x, gridDim.x) * static_cast<int64_t>(group); first < total;
		first += static_cast<int64_t>(gridDim.x) * group)
	{
		const int lines = static_cast<int>(total - first < group ? total - first : group);
		for (int q = threadIdx.x; q < lines; q += blockDim.x)
		{
			const int64_t line = first + q;
			const int64_t jj = line / columns;
			const int column = static_cast<int>(line - jj * columns);
			const int64_t kept = jj / chunk.count;
			const int64_t slice = kept * p.map.reduced_count + chunk.begin + jj % chunk.count;
			line_slice[q] = slice;
			line_src[q] = p.entries[slice].slice_offset + column * p.slice_s1;
			line_dst[q] = jj * elements + column;
			line_column[q] = column;
		}
		__syncthreads();
		for (int t = threadIdx.x; t < group * n; t += blockDim.x)
		{
			const int e = t / group;
			const int l = t - e * group;
			if (l < lines)
			{
				a[l * stride + e] = e >= held.begin && e < held.end ? p.slices[line_src[l] + e * p.slice_s0] :
					make_float2(0.0f, 0.0f);
			}
		}
		__syncthreads();
		const float2 *z = block_fft(a, b, lines, stride, plan, twl, -1.0f);
		for (int t = threadIdx.x; t < group * n; t += blockDim.x)
		{
			const int e = t / group;
			const int l = t - e * group;
			if (l < lines)
			{
				const int64_t slice = line_slice[l];
				const slice_entry &entry = p.entries[slice];
				const float2 *table = p.tables + slice * static_cast<int64_t>(h + n);
				const int column = line_column[l];
				bool read;
				const prepared_sample sample = prepare_unbranched<VARIANT>(p, entry, p.radial + entry.radial_offset, table + h,
					table[column], e, column, z[l * stride + e], read);
				if (read)
				{
					prepared[line_dst[l] + static_cast<int64_t>(e) * h] = sample;
				}
			}
		}
		__syncthreads();
	}
}

// The same fusion for lengths of two register factors (fft_two.hpp): a block
// of (lines, b) threads transforms `lines` neighbouring columns, and their
// threads prepare the elements from LDS.
template <int VARIANT, int CLASS>
__global__ __launch_bounds__(512, two_factor::waves<CLASS>) void columns_prepare_two_kernel(insertion_params p, slice_chunk chunk,
	row_range held, two_factor::plan plan, const float2 *tw, prepared_sample *prepared)
{
	extern __shared__ float2 lds[];
	const int l = threadIdx.x;
	const int j = threadIdx.y;
	const int n = plan.n;
	float2 *twl = lds + plan.lines * plan.line;
	float2 *x = lds + l * plan.line;
	two_factor::stage_twiddles(plan, twl, tw, j * blockDim.x + l, blockDim.x * blockDim.y);
	__syncthreads();
	const int h = p.h;
	const int columns = n % 2 == 0 ? n / 2 : h;
	const int64_t elements = static_cast<int64_t>(n) * h;
	const int64_t total = p.map.kept_count * chunk.count * columns;
	const int64_t first = xcd_block(blockIdx.x, gridDim.x) * static_cast<int64_t>(plan.lines);
	if (first >= total)
	{
		return;
	}
	const int64_t line = first + l;
	const bool live = line < total;
	const int64_t jj = live ? line / columns : 0;
	const int column = static_cast<int>(live ? line - jj * columns : 0);
	const int64_t kept = jj / chunk.count;
	const int64_t slice = kept * p.map.reduced_count + chunk.begin + jj % chunk.count;
	const slice_entry &e = p.entries[slice];
	const float2 *in = p.slices + e.slice_offset + column * p.slice_s1;
	two_factor::transform_line<CLASS, false, true>(plan, x, twl, j, -1.0f,
		[&](int i) { return live && i >= held.begin && i < held.end ? in[i * p.slice_s0] : make_float2(0.0f, 0.0f); },
		[&](int k, float2 v) { x[k] = v; });
	__syncthreads();
	if (live)
	{
		const float2 *table = p.tables + slice * static_cast<int64_t>(h + n);
		const float2 x_phase = table[column];
		const float *radial = p.radial + e.radial_offset;
		prepared_sample *out = prepared + jj * elements + column;
#pragma unroll 4
		for (int row = j; row < n; row += blockDim.y)
		{
			bool read;
			const prepared_sample sample =
				prepare_unbranched<VARIANT>(p, e, radial, table + h, x_phase, row, column, x[row], read);
			if (read)
			{
				out[row * h] = sample;
			}
		}
	}
}

// Before bricks that own voxels: the inputs that reach the outputs by atomics.
// Blocks up to `split` copy the bricks split into shares (the first `split`
// tasks hold them all), the others the rows of the frequencies +-N/2 of an even
// N along y or z (2 N - 1 of a volume's N^2), which two bricks reach.
template <int T>
__global__ __launch_bounds__(64) void copy_shared_inputs_kernel(insertion_params p, const int4 *tasks, int split,
	accumulator_input input)
{
	const int64_t kept = blockIdx.y;
	const int big = p.big;
	const int he = big / 2;
	const int lane = threadIdx.x;
	const float2 *num = input.numerator + kept_offset(p.map, input.num_slot, kept);
	const float *den = input.denominator + kept_offset(p.map, input.den_slot, kept);
	float2 *num_out = p.numerator + kept_offset(p.map, slot_numerator_out, kept);
	float *den_out = p.denominator + kept_offset(p.map, slot_denominator_out, kept);
	const auto copy = [&](int64_t z, int64_t y, int64_t x)
	{
		num_out[z * p.num_s0 + y * p.num_s1 + x * p.num_s2] =
			num[z * input.num_s0 + y * input.num_s1 + x * input.num_s2];
		den_out[z * p.den_s0 + y * p.den_s1 + x * p.den_s2] =
			den[z * input.den_s0 + y * input.den_s1 + x * input.den_s2];
	};
	if (static_cast<int>(blockIdx.x) >= split)
	{
		const int r = static_cast<int>(blockIdx.x) - split;
		const int z = r < big ? he : (r - big < he ? r - big : r - big + 1);
		const int y = r < big ? r : he;
		for (int x = lane; x < p.half; x += 64)
		{
			copy(z, y, x);
		}
		return;
	}
	const brick_box box = unpack_brick(tasks[2 * blockIdx.x]);
	const int4 share = tasks[2 * blockIdx.x + 1];
	if (share.x != 0 || share.y == 1)
	{
		return;
	}
	const int x = box.lo[0] + T - 1 + lane % 8;
	const int ey = box.ext[1] - (T - 1);
	const int ez = box.ext[2] - (T - 1);
	for (int xs = x; xs <= min(he, box.lo[0] + box.ext[0] - 1); xs += 8)
	{
		for (int r = lane / 8; r < ey * ez; r += 8)
		{
			const int y = box.lo[1] + T - 1 + r % ey;
			const int z = box.lo[2] + T - 1 + r / ey;
			// (+-N/2 of an even N is the rows' above: both write the same input.)
			if (y <= he && z <= he)
			{
				copy(z < 0 ? z + big : z, y < 0 ? y + big : y, xs);
			}
		}
	}
}

// A wavefront owns the brick of one task (a brick and a share of the
// slices): EX x EY x EZ first-tap cells and the voxels their taps reach, in
// LDS.
// Wavefronts per SIMD that the register budget of a kernel is held to: as many
// as the LDS of claimed Kaiser-Bessel bricks allows, four (128 registers) for 8 x
// 6 x 6, which take 137 left alone. 0 leaves the others to the compiler.
template <int PROFILE, int ROUNDS, int EX, int EY, int EZ>
constexpr int brick_waves()
{
	if (PROFILE != REXLIB_HIP_KAISER_BESSEL || ROUNDS != claimed_rounds)
	{
		return 0;
	}
	using L = brick_layout<brick_reach<PROFILE>::taps, false, EX, EY, EZ>;
	const int per_cu = 160 * 1024 / (L::voxels * 12 + L::cells + 2 * 64 * 4);
	return per_cu >= 13 ? 4 : (per_cu + 3) / 4;
}

template <int PROFILE, bool ODD, bool VOXELS, int ROUNDS, int EX, int EY, int EZ>
__global__ __launch_bounds__(64, (brick_waves<PROFILE, ROUNDS, EX, EY, EZ>())) void brick_kernel(insertion_params p,
	slice_chunk chunk, const prepared_sample *prepared,
	const int4 *tasks, int task_count, accumulator_input input)
{
	constexpr int T = brick_reach<PROFILE>::taps;
	constexpr bool WIDE = ROUNDS != claimed_rounds;
	using L = brick_layout<T, WIDE, EX, EY, EZ>;
	// The voxels as two arrays, value and weight. A tap is then a 64-bit and a
	// 32-bit access at even and odd bank pitches; one array of 12-byte voxels
	// took 217 cycles per CU for the 8 taps of 48 lanes, the two arrays 184.
	__shared__ float2 acc_value[L::voxels];
	__shared__ float acc_weight[L::voxels];
	// Claimed rounds, per first-tap cell: the lane that last claimed it.
	__shared__ unsigned char claim[WIDE ? 1 : L::cells];
	// Wide rounds: the axis weights of the samples in the lanes, x, y, z.
	__shared__ float4 axis_weights[WIDE ? 64 * 3 : 1];
	// Per lane: the last row (or slice) starting at or before it.
	__shared__ int marker[64];
	// Slices that hit the brick, waiting for their rows to be bounded.
	__shared__ int queue[64];

	const int lane = threadIdx.x;
	const int big = p.big;
	const int n = p.n;
	const int h = p.h;
	const int64_t elements = static_cast<int64_t>(n) * h;
	const int64_t kept = blockIdx.y;
	const float cell_offset = first_tap_offset(T, p.kb_half_width);
	const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));

	for (int ti = blockIdx.x; ti < task_count; ti += gridDim.x)
	{
		const brick_box box = unpack_brick(tasks[2 * ti]);
		const int4 share = tasks[2 * ti + 1];
		const int64_t share_begin = chunk.count * share.x / share.y;
		const int64_t share_end = chunk.count * (share.x + 1) / share.y;
		float lower[3];
		float upper[3];
		float centre[3];
		float half_extent[3];
		float half_diagonal2 = 0.0f;
		for (int a = 0; a < 3; ++a)
		{
			cell_positions(box.lo[a], box.ext[a], cell_offset, lower[a], upper[a]);
			centre[a] = 0.5f * (lower[a] + upper[a]);
			half_extent[a] = 0.5f * (upper[a] - lower[a]) + 0.01f;
			half_diagonal2 += half_extent[a] * half_extent[a];
		}
		const float half_diagonal = sqrtf(half_diagonal2);
		const float centre_norm = sqrtf(centre[0] * centre[0] + centre[1] * centre[1] + centre[2] * centre[2]);
		const float nearest = centre_norm - half_diagonal - 1e-3f;
		// The middle of the first taps of the brick's EX x EY x EZ cells: a
		// first tap f is the brick's when |f - middle| < E / 2 along each axis.
		// (A brick cut short at the volume's end may take cells beyond its own
		// extents, which no other brick owns: their rows end at `upper`.)
		const float middle[3] = {static_cast<float>(box.lo[0]) + 0.5f * (EX - 1),
			static_cast<float>(box.lo[1]) + 0.5f * (EY - 1), static_cast<float>(box.lo[2]) + 0.5f * (EZ - 1)};

		// The sample this lane holds, not yet added: value, its first-tap cell
		// and voxel, and per axis the fraction past the first tap.
		bool pending = false;
		float held_re = 0.0f, held_im = 0.0f, held_den = 0.0f;
		int held_cell = 0;
		int held_voxel = 0;
		float held_w[3] = {0.0f, 0.0f, 0.0f};

		// One round: every holding lane claims its cell and the winners add
		// their taps; meanwhile (when `fill`) the lanes free after the round
		// load the next samples of the current rows, which they hold from the
		// next round on.
		int next = 0;
		int total = 0;
		int current = 0;
		int row_start = 0;
		int row_count = 0;
		// Lane k describes row k of the current 64 rows (registers, not LDS,
		// so that more wavefronts fit a CU): base position and the first k_x
		// less the row's first sample number (so sample s of the batch has
		// k_x = that + s); step; the prepared element of (row, k_x = 0), bit
		// 31 set for the -k copy.
		float4 row_base = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		float4 row_step = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		uint32_t row_index = 0;
		// Wide rounds: a sample's 64 taps are the 64 lanes. Each lane takes one
		// sample of the rows, puts its 12 axis weights in LDS, and the wavefront
		// then adds the samples one after another, each by one read-add-write
		// of 64 different voxels (no claims, no bank conflicts, every lane
		// busy, but each sample waits for the one before). kaiser_bessel_bricks
		// says when, with both sides' times.
		const int tap_x = lane & 3;
		const int tap_y = (lane >> 2) & 3;
		const int tap_z = lane >> 4;
		// A sample's voxel times `reached` plus `tap_voxel` is the tap's. Windows of
		// fewer than 4 taps send the surplus lanes to the padding of the rows,
		// which is never added to the accumulators (64 rows at least, one a lane):
		// their weights are 0, but a sample that is not finite times 0 is not.
		// (Switching the lanes off for the access took 2,048 slices of 256^2 into
		// 256^3 from 4.4 to 5.3 ms.)
		const bool within = ROUNDS != wide_narrow_rounds || max(max(tap_x, tap_y), tap_z) < p.taps;
		const int reached = within ? 1 : 0;
		static_assert(!WIDE || (L::pitch_y > L::lx && L::ly * L::lz >= 64), "a padding voxel per lane");
		const int tap_voxel = within ? tap_x + L::pitch_y * tap_y + L::pitch_z * tap_z :
			L::lx + L::pitch_y * (lane % L::ly) + L::pitch_z * (lane / L::ly);
		auto wide_round = [&]()
		{
			if constexpr (WIDE)
			{
				const int take = min(64, total - next);
				marker[lane] = lane == 0 ? current : 0;
				lds_order();
				if (row_count > 0 && row_start >= next && row_start < next + 64)
				{
					marker[row_start - next] = lane;
				}
				lds_order();
				const int row = wave_prefix_max(marker[lane]);
				lds_order();
				current = __builtin_amdgcn_readlane(row, take - 1);
				const float4 b = make_float4(__shfl(row_base.x, row, 64), __shfl(row_base.y, row, 64),
					__shfl(row_base.z, row, 64), __shfl(row_base.w, row, 64));
				const float4 st = make_float4(__shfl(row_step.x, row, 64), __shfl(row_step.y, row, 64),
					__shfl(row_step.z, row, 64), 0.0f);
				const uint32_t ix = static_cast<uint32_t>(__shfl(static_cast<int>(row_index), row, 64));
				const int kx = __float_as_int(b.w) + next + lane;
				const bool mine = lane < take;
				prepared_sample q{0.0f, 0.0f, 0.0f};
				if (mine)
				{
					q = prepared[(ix & 0x7fffffffu) + static_cast<uint32_t>(kx)];
				}
				const float c[3] = {row_position(b.x, st.x, kx), row_position(b.y, st.y, kx), row_position(b.z, st.z, kx)};
				float f[3];
#pragma unroll
				for (int a = 0; a < 3; ++a)
				{
					float w[4];
					window_taps<PROFILE>::template place<4>(p, mine ? c[a] : 0.0f, w);
					axis_weights[lane * 3 + a] = make_float4(w[0], w[1], w[2], w[3]);
					f[a] = window_taps<PROFILE>::first_float(p, c[a]) - middle[a];
				}
				const bool own = mine && fabsf(f[0]) < 0.5f * EX && fabsf(f[1]) < 0.5f * EY && fabsf(f[2]) < 0.5f * EZ &&
					!(q.re == 0.0f && q.im == 0.0f && q.den == 0.0f);
				constexpr float first_voxel = 0.5f * ((EX - 1) + L::pitch_y * (EY - 1) + L::pitch_z * (EZ - 1));
				const int voxel = static_cast<int>(fmaf(f[2], L::pitch_z, fmaf(f[1], L::pitch_y, f[0] + first_voxel)));
				const float im = __uint_as_float(__float_as_uint(q.im) ^ (ix & 0x80000000u));
				lds_order();
				const float *weights = reinterpret_cast<const float *>(axis_weights);
				// The weights of the next sample are read before the taps of this
				// one, so a sample waits for LDS once.
				uint64_t left = __ballot(own);
				int s = left != 0 ? __builtin_ctzll(left) : 0;
				float wx = weights[12 * s + tap_x];
				float wy = weights[12 * s + 4 + tap_y];
				float wz = weights[12 * s + 8 + tap_z];
				while (left != 0)
				{
					const int first = __builtin_amdgcn_readlane(voxel, s);
					const int at = (ROUNDS == wide_narrow_rounds ? __mul24(first, reached) : first) + tap_voxel;
					const float wt = wz * wy * wx;
					const float re = lane_value(q.re, s);
					const float imaginary = lane_value(im, s);
					const float den = lane_value(q.den, s);
					left &= left - 1;
					s = left != 0 ? __builtin_ctzll(left) : 0;
					wx = weights[12 * s + tap_x];
					wy = weights[12 * s + 4 + tap_y];
					wz = weights[12 * s + 8 + tap_z];
					float2 v = acc_value[at];
					float d = acc_weight[at];
					v.x += re * wt;
					v.y += imaginary * wt;
					d += den * wt;
					acc_value[at] = v;
					acc_weight[at] = d;
					lds_order();
				}
				next += take;
			}
		};
		auto round = [&](bool fill)
		{
			// Claim: each holding lane writes its lane into the byte of its
			// first-tap cell and reads it back. A plain LDS read after the
			// store (lds_order keeps the compiler from reusing the stored
			// value); a volatile pointer would turn it into a flat load, which
			// is not ordered after the LDS store.
			if (pending)
			{
				claim[held_cell] = static_cast<unsigned char>(lane);
			}
			lds_order();
			const bool win = pending && claim[held_cell] == lane;
			lds_order();

			// The fill starts before the winners' taps: the lanes free after
			// this round (holding nothing, or winning now) take the next
			// samples of the current rows, and the loads of those samples are
			// in flight while the taps run. The samples join the claim of the
			// next round.
			int take = 0;
			int r = 0;
			bool mine = false;
			float4 b = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
			float4 st = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
			uint32_t ix = 0;
			int kx = 0;
			prepared_sample q{0.0f, 0.0f, 0.0f};
			if (fill)
			{
				const bool free = !pending || win;
				const uint64_t free_mask = __ballot(free);
				take = min(static_cast<int>(__popcll(free_mask)), total - next);
				if (take > 0)
				{
					// The row of sample next + lane: rows starting in [next, next + 64)
					// mark their slot, slot 0 starts with the row holding `next`.
					marker[lane] = lane == 0 ? current : 0;
					lds_order();
					if (row_count > 0 && row_start >= next && row_start < next + 64)
					{
						marker[row_start - next] = lane;
					}
					lds_order();
					r = wave_prefix_max(marker[lane]);
					lds_order();
					current = __builtin_amdgcn_readlane(r, take - 1);
					// Free lane k (in lane order) takes sample next + k itself: the
					// row of that sample, then the row's data, by shuffles.
					const int rank = static_cast<int>(__popcll(free_mask & below));
					mine = free && rank < take;
					const int row = __shfl(r, mine ? rank : 0, 64);
					b = make_float4(__shfl(row_base.x, row, 64), __shfl(row_base.y, row, 64),
						__shfl(row_base.z, row, 64), __shfl(row_base.w, row, 64));
					st = make_float4(__shfl(row_step.x, row, 64), __shfl(row_step.y, row, 64),
						__shfl(row_step.z, row, 64), 0.0f);
					ix = static_cast<uint32_t>(__shfl(static_cast<int>(row_index), row, 64));
					kx = __float_as_int(b.w) + next + rank;
					if (mine)
					{
						q = prepared[(ix & 0x7fffffffu) + static_cast<uint32_t>(kx)];
					}
				}
			}

			if (win)
			{
				const int base = held_voxel;
				float wx[T], wy[T], wz[T];
				if constexpr (PROFILE == REXLIB_HIP_TRIANGLE)
				{
					wx[0] = 1.0f - held_w[0];
					wx[1] = held_w[0];
					wy[0] = 1.0f - held_w[1];
					wy[1] = held_w[1];
					wz[0] = 1.0f - held_w[2];
					wz[1] = held_w[2];
				}
				else if constexpr (PROFILE == REXLIB_HIP_BOX)
				{
					wx[0] = 1.0f;
					wy[0] = 1.0f;
					wz[0] = 1.0f;
				}
				else
				{
					window_taps<PROFILE>::template place<T>(p, held_w[0], wx);
					window_taps<PROFILE>::template place<T>(p, held_w[1], wy);
					window_taps<PROFILE>::template place<T>(p, held_w[2], wz);
				}
				// (Of the layout's 4 taps a Kaiser-Bessel window takes its own.)
				const int taps = PROFILE == REXLIB_HIP_KAISER_BESSEL ? p.taps : T;
#pragma unroll
				for (int tz = 0; tz < T; ++tz)
				{
#pragma unroll
					for (int ty = 0; ty < T; ++ty)
					{
						const float wzy = wz[tz] * wy[ty];
#pragma unroll
						for (int tx = 0; tx < T; ++tx)
						{
							if (tx < taps && ty < taps && tz < taps)
							{
								const float wt = wzy * wx[tx];
								const int at = base + tx + L::pitch_y * ty + L::pitch_z * tz;
								float2 v = acc_value[at];
								float d = acc_weight[at];
								v.x += held_re * wt;
								v.y += held_im * wt;
								d += held_den * wt;
								acc_value[at] = v;
								acc_weight[at] = d;
							}
							lds_order();
						}
					}
				}
			}
			lds_order();
			pending = pending && !win;

			if (take > 0)
			{
				const float c[3] = {row_position(b.x, st.x, kx), row_position(b.y, st.y, kx),
					row_position(b.z, st.z, kx)};
				// First taps in float (whole numbers, exact), less the middle.
				float f[3];
				float w[3];
#pragma unroll
				for (int a = 0; a < 3; ++a)
				{
					f[a] = window_taps<PROFILE>::first_float(p, c[a]);
					w[a] = PROFILE == REXLIB_HIP_KAISER_BESSEL ? c[a] : c[a] - f[a];
					f[a] -= middle[a];
				}
				const bool own = fabsf(f[0]) < 0.5f * EX && fabsf(f[1]) < 0.5f * EY && fabsf(f[2]) < 0.5f * EZ;
				if (mine && own)
				{
					pending = true;
					held_re = q.re;
					held_im = __uint_as_float(__float_as_uint(q.im) ^ (ix & 0x80000000u));
					held_den = q.den;
					constexpr float first_cell = 0.5f * ((EX - 1) + EX * (EY - 1) + EX * EY * (EZ - 1));
					constexpr float first_voxel =
						0.5f * ((EX - 1) + L::pitch_y * (EY - 1) + L::pitch_z * (EZ - 1));
					held_cell = static_cast<int>(fmaf(f[2], EX * EY, fmaf(f[1], EX, f[0] + first_cell)));
					held_voxel = static_cast<int>(fmaf(f[2], L::pitch_z, fmaf(f[1], L::pitch_y, f[0] + first_voxel)));
					held_w[0] = w[0];
					held_w[1] = w[1];
					held_w[2] = w[2];
				}
				next += take;
			}
		};

		const slice_plane *planes = p.planes + kept * p.map.reduced_count + chunk.begin;
		const slice_entry *entries = p.entries + kept * p.map.reduced_count + chunk.begin;

		// The rows of the `hits` slices in the queue: one slice per lane.
		const auto insert_hits = [&](int hits)
		{
			const bool near = lane < hits;
			const int js_lane = near ? queue[lane] : 0;
			lds_order();
			float x0 = 0.0f, x1 = 0.0f, x2 = 0.0f, y0 = 0.0f, y1 = 0.0f, y2 = 0.0f;
			int last_shell = -1;
			if (near)
			{
				const slice_entry &e = entries[js_lane];
				last_shell = e.last_shell;
				x0 = e.x_step[0];
				x1 = e.x_step[1];
				x2 = e.x_step[2];
				y0 = static_cast<float>(e.y_step[0]);
				y1 = static_cast<float>(e.y_step[1]);
				y2 = static_cast<float>(e.y_step[2]);
			}
			// The rows of both copies, one slice per lane, and the reciprocal steps
			// of the frame.
			int plus[2] = {0, 0}, minus_range[2] = {0, 0};
			float inv_x[3] = {0.0f, 0.0f, 0.0f};
			if (near)
			{
				const float xs[3] = {x0, x1, x2};
				const float ys[3] = {y0, y1, y2};
				bound_slice(n, xs, ys, last_shell, lower, upper, [](float v) { return __builtin_amdgcn_rcpf(v); }, plus,
					minus_range, inv_x);
			}
			const int plus_rows = near ? max(plus[1] - plus[0], 0) : 0;
			const int minus_rows = near ? max(minus_range[1] - minus_range[0], 0) : 0;
			const int rows = plus_rows + minus_rows;
			const int rows_inclusive = wave_inclusive_scan(rows);
			const int rows_first = rows_inclusive - rows;
			const int total_rows = __builtin_amdgcn_readlane(rows_inclusive, 63);
			for (int rb = 0; rb < total_rows; rb += 64)
			{
				// The slice of row rb + lane: every slice with rows in
				// [rb, rb + 64) marks the slot of its first one (slot 0 for
				// the slice holding row rb); a prefix maximum hands each row
				// its slice's lane.
				marker[lane] = 0;
				lds_order();
				if (rows > 0 && rows_first < rb + 64 && rows_first + rows > rb)
				{
					marker[max(rows_first - rb, 0)] = lane;
				}
				lds_order();
				const int s = wave_prefix_max(marker[lane]);
				lds_order();
				const int r = rb + lane;
				// Every shuffle runs with all lanes active: a lane reads nothing
				// from a source lane that is switched off.
				const int idx = r - __shfl(rows_first, s, 64);
				const int np = __shfl(plus_rows, s, 64);
				const int first_plus = __shfl(plus[0], s, 64);
				const int first_minus = __shfl(minus_range[0], s, 64);
				const bool minus = idx >= np;
				const int ky = minus ? first_minus + (idx - np) : first_plus + idx;
				const float sign = minus ? -1.0f : 1.0f;
				const float frame_x[3] = {__shfl(x0, s, 64), __shfl(x1, s, 64), __shfl(x2, s, 64)};
				const float frame_y[3] = {__shfl(y0, s, 64), __shfl(y1, s, 64), __shfl(y2, s, 64)};
				const float frame_ix[3] = {__shfl(inv_x[0], s, 64), __shfl(inv_x[1], s, 64), __shfl(inv_x[2], s, 64)};
				const int shell = __shfl(last_shell, s, 64);
				const int js = __shfl(js_lane, s, 64);
				float step[3];
				float y_step[3];
				float inv_step[3];
				float base[3];
				int begin = 0;
				int end = 0;
				if (r < total_rows)
				{
					const slice_entry &e = entries[js];
					for (int a = 0; a < 3; ++a)
					{
						step[a] = sign * frame_x[a];
						y_step[a] = sign * frame_y[a];
						inv_step[a] = sign * frame_ix[a];
						base[a] = static_cast<float>(static_cast<double>(ky) *
							(minus ? -e.y_step[a] : e.y_step[a]));
					}
					clip_row(n, ky, minus ? 1 : 0, shell, step, y_step, inv_step, lower, upper, begin, end);
				}
				else
				{
					for (int a = 0; a < 3; ++a)
					{
						step[a] = 0.0f;
						base[a] = 0.0f;
					}
				}
				row_count = end - begin;
				const int count_inclusive = wave_inclusive_scan(row_count);
				row_start = count_inclusive - row_count;
				total = __builtin_amdgcn_readlane(count_inclusive, 63);
				const int stored_row = ky < 0 ? ky + n : ky;
				row_base = make_float4(base[0], base[1], base[2], __int_as_float(begin - row_start));
				row_step = make_float4(step[0], step[1], step[2], 0.0f);
				row_index = r < total_rows ? (static_cast<uint32_t>((kept * chunk.count + js) * elements +
					static_cast<int64_t>(stored_row) * h) | (minus ? 0x80000000u : 0u)) : 0u;
				lds_order();
				next = 0;
				current = 0;
				while (next < total)
				{
					if constexpr (WIDE)
					{
						wide_round();
					}
					else
					{
						round(true);
					}
				}
				lds_order();
			}
		};

		// Slices whose plane passes near the brick: 64 planes are tested at a
		// time (one 16-byte word a lane, the next 64 already in flight), and
		// the few that hit (3.5 % at 256^3) collect in `queue` until 64 wait or
		// the share ends, so that the bounds and rows below run on full lanes.
		int queued = 0;
		// Whether any slice hit the brick (its LDS is cleared for the first).
		bool touched = false;
		slice_plane plane = planes[min(share_begin + lane, chunk.count - 1)];
		for (int64_t window = share_begin;; window += 64)
		{
			const bool last = window >= share_end;
			uint64_t hits = 0;
			bool hit = false;
			if (!last)
			{
				const slice_plane tested = plane;
				plane = planes[min(window + 64 + lane, chunk.count - 1)];
				// The plane meets the box iff |n . c| is at most the box's
				// support sum_a |n_a| h_a along the normal n.
				const float distance = fabsf(tested.normal[0] * centre[0] + tested.normal[1] * centre[1] +
					tested.normal[2] * centre[2]);
				const float support = fabsf(tested.normal[0]) * half_extent[0] + fabsf(tested.normal[1]) * half_extent[1] +
					fabsf(tested.normal[2]) * half_extent[2];
				hit = window + lane < share_end && distance <= support * 1.001f + 1e-3f && nearest <= tested.reach;
				hits = __ballot(hit);
			}
			const int count = static_cast<int>(__popcll(hits));
			if (queued > 0 && (last || queued + count > 64))
			{
				if (!touched)
				{
					for (int v = lane; v < L::voxels; v += 64)
					{
						acc_value[v] = make_float2(0.0f, 0.0f);
						acc_weight[v] = 0.0f;
					}
					touched = true;
				}
				lds_order();
				insert_hits(queued);
				queued = 0;
			}
			if (last)
			{
				break;
			}
			lds_order();
			if (hit)
			{
				queue[queued + static_cast<int>(__popcll(hits & below))] = static_cast<int>(window) + lane;
			}
			queued += count;
		}
		// Samples still held after the last rows.
		if constexpr (!WIDE)
		{
			while (__ballot(pending) != 0)
			{
				round(false);
			}
		}
		lds_order();

		// Add the brick to the accumulators of its kept batch element.
		if (!touched && !(VOXELS && share.x == 0 && !input.in_place))
		{
			continue;
		}
		const int he = big / 2;
		const int64_t num_base = kept_offset(p.map, slot_numerator_out, kept);
		const int64_t den_base = kept_offset(p.map, slot_denominator_out, kept);
		if constexpr (VOXELS)
		{
			// The voxels past the T - 1 lower faces are this brick's alone: out =
			// in + sum, written once. Atomics go to the voxels of a brick split
			// into shares and to +-N/2 of an even N (one stored element that
			// two bricks reach), whose inputs are in the outputs already.
			const bool split = share.y > 1;
			if (split && !touched)
			{
				continue;
			}
			const int64_t num_in = kept_offset(p.map, input.num_slot, kept);
			const int64_t den_in = kept_offset(p.map, input.den_slot, kept);
			const int x_count = min(box.ext[0] - (T - 1), he + 1 - (box.lo[0] + T - 1));
			const int y_count = min(box.ext[1] - (T - 1), he + 1 - (box.lo[1] + T - 1));
			const int z_count = min(box.ext[2] - (T - 1), he + 1 - (box.lo[2] + T - 1));
			// Rows of 7 voxels, 8 lanes each. Every input is loaded before any
			// output is written, so a brick waits for memory once (row by row, the
			// seven round trips were a third of the time of a sparse call).
			constexpr int row = EX - T + 1 <= 8 ? 8 : 16; // lanes along x
			constexpr int steps = ((EY - T + 1) * (EZ - T + 1) + 64 / row - 1) / (64 / row);
			const int lx = lane % row;
			const int x = box.lo[0] + T - 1 + lx;
			float2 in_value[steps];
			float in_weight[steps];
#pragma unroll
			for (int step = 0; step < steps; ++step)
			{
				const int r = lane / row + step * (64 / row);
				const int lz = r / (EY - T + 1);
				const int ly = r - lz * (EY - T + 1);
				const int y = box.lo[1] + T - 1 + ly;
				const int z = box.lo[2] + T - 1 + lz;
				const int sy = y < 0 ? y + big : y;
				const int sz = z < 0 ? z + big : z;
				const int v = (lx + T - 1) + L::pitch_y * (ly + T - 1) + L::pitch_z * (lz + T - 1);
				in_value[step] = make_float2(0.0f, 0.0f);
				in_weight[step] = 0.0f;
				const bool inside = lx < x_count && ly < y_count && lz < z_count && !split;
				// (In place, voxels without a sum keep what they hold.)
				if (inside && (!input.in_place ||
					!(acc_value[v].x == 0.0f && acc_value[v].y == 0.0f && acc_weight[v] == 0.0f)))
				{
					in_value[step] =
						input.numerator[num_in + sz * input.num_s0 + sy * input.num_s1 + x * input.num_s2];
					in_weight[step] =
						input.denominator[den_in + sz * input.den_s0 + sy * input.den_s1 + x * input.den_s2];
				}
			}
#pragma unroll
			for (int step = 0; step < steps; ++step)
			{
				const int r = lane / row + step * (64 / row);
				const int lz = r / (EY - T + 1);
				const int ly = r - lz * (EY - T + 1);
				if (lx < x_count && ly < y_count && lz < z_count)
				{
					const int v = (lx + T - 1) + L::pitch_y * (ly + T - 1) + L::pitch_z * (lz + T - 1);
					const float2 sum = touched ? acc_value[v] : make_float2(0.0f, 0.0f);
					const float weight = touched ? acc_weight[v] : 0.0f;
					const int y = box.lo[1] + T - 1 + ly;
					const int z = box.lo[2] + T - 1 + lz;
					const int sy = y < 0 ? y + big : y;
					const int sz = z < 0 ? z + big : z;
					const float2 value = volume_phase<ODD>(p, sum, x, sy, sz);
					float2 *target = p.numerator + num_base + sz * p.num_s0 + sy * p.num_s1 + x * p.num_s2;
					float *dtarget = p.denominator + den_base + sz * p.den_s0 + sy * p.den_s1 + x * p.den_s2;
					const bool shared = split || (big % 2 == 0 && (sy == he || sz == he));
					const bool none = sum.x == 0.0f && sum.y == 0.0f && weight == 0.0f;
					if (shared)
					{
						if (!none)
						{
							atomicAdd(&target->x, value.x);
							atomicAdd(&target->y, value.y);
							atomicAdd(dtarget, weight);
						}
					}
					else if (!(none && input.in_place))
					{
						*target = make_float2(in_value[step].x + value.x, in_value[step].y + value.y);
						*dtarget = in_weight[step] + weight;
					}
				}
			}
			lds_order();
			continue;
		}
		// Voxels no other task touches (at least taps - 1 past the lower faces,
		// inside the cells, a brick of one task without aliasing) take a plain
		// read-add-write, the others atomics.
		const bool single = share.y == 1 && box.alias_free;
		for (int v = lane; v < L::voxels; v += 64)
		{
			const int lz = v / L::pitch_z;
			const int rest = v - lz * L::pitch_z;
			const int ly = rest / L::pitch_y;
			const int lx = rest - ly * L::pitch_y;
			if (lx >= L::lx || ly >= L::ly)
			{
				continue;
			}
			const float2 sum = acc_value[v];
			const float weight = acc_weight[v];
			if (sum.x == 0.0f && sum.y == 0.0f && weight == 0.0f)
			{
				continue;
			}
			const int x = box.lo[0] + lx;
			const int y = box.lo[1] + ly;
			const int z = box.lo[2] + lz;
			if (x < 0 || x > he || y < -he || y > he || z < -he || z > he)
			{
				continue;
			}
			const int sy = y < 0 ? y + big : y;
			const int sz = z < 0 ? z + big : z;
			const float2 value = volume_phase<ODD>(p, sum, x, sy, sz);
			float2 *target = p.numerator + num_base + sz * p.num_s0 + sy * p.num_s1 + x * p.num_s2;
			float *dtarget = p.denominator + den_base + sz * p.den_s0 + sy * p.den_s1 + x * p.den_s2;
			const bool exclusive = single && lx >= T - 1 && ly >= T - 1 && lz >= T - 1 && lx < box.ext[0] &&
				ly < box.ext[1] && lz < box.ext[2];
			if (exclusive)
			{
				float2 t = *target;
				t.x += value.x;
				t.y += value.y;
				*target = t;
				*dtarget += weight;
			}
			else
			{
				atomicAdd(&target->x, value.x);
				atomicAdd(&target->y, value.y);
				atomicAdd(dtarget, weight);
			}
		}
		lds_order();
	}
}

// Brick shapes (first-tap cells along x, y, z): 16 x 8 x 6,
// 16 x 8 x 8, 16 x 16 x 8, 8 x 8 x 8, 8 x 8 x 6, 8 x 6 x 6 and 8 x 8 x 4, and
// the expected plane hits per task that splits busy bricks. Smaller bricks
// take less LDS (more wavefronts per CU) but hold more halo voxels per cell.
// One entry per volume extent N (0: every extent without an entry of its
// own); a call reads its extent's entry once, so concurrent callers each see
// a whole entry.
struct brick_tuning
{
	int ex;
	int ey;
	int ez;
	int share;
};

// What calls of up to two taps per axis take without an entry: 8 x 8 x 8 bricks
// and 512 plane hits per task (over 64 to 512 voxels and up to 4,096 slices within
// a fifth of the fastest shape), or, with fewer than 3 million samples, larger
// bricks, whose fewer faces count there for more than their tasks: 300 slices of
// 108^2 into 108^3 take 104 us in 16 x 8 x 6 and 117 in 8 x 8 x 8, 1,000 of 32^2
// into 48^3 85 against 92, but 4,000 of 100^2 into 100^3 (16 million) 0.49 ms in
// the one against 0.45, 2,000 of 225^2 into 225^3 0.89 against 0.82. Sparse calls on
// cells (a fixed workspace) are all faces and take the larger bricks too.
// Kaiser-Bessel windows: kaiser_bessel_bricks.
constexpr brick_tuning untuned_bricks{8, 8, 8, 512};
constexpr brick_tuning untuned_small_bricks{16, 8, 6, 256};
constexpr brick_tuning untuned_wide_bricks{8, 6, 6, 512};
constexpr brick_tuning untuned_claimed_bricks{8, 8, 6, 128};
constexpr brick_tuning untuned_sparse_bricks{16, 8, 6, 128};

// Bricks that own voxels: a cell shell of T - 1 is walked twice, so the brick
// has to be a large one of the small ones.
constexpr brick_tuning voxel_tuning{8, 8, 8, 512};

std::mutex tuning_mutex;
std::map<int, brick_tuning> tuning_table;

bool valid_brick_shape(int ex, int ey, int ez)
{
	return (ex == 16 && ey == 8 && (ez == 6 || ez == 8)) || (ex == 16 && ey == 16 && ez == 8) ||
		(ex == 8 && ey == 8 && (ez == 8 || ez == 6 || ez == 4)) || (ex == 8 && ey == 6 && ez == 6);
}

// Table keys: the extent (every window), or the extent plus taps_key times
// the taps per axis of the brick layout (1, 2 or 4) for one window family.
constexpr int taps_key = 1 << 20;

// The entry of an extent for a window of `taps` per axis (0: any window): the
// window's own entry, else the extent's, else the entry for every extent, else
// none (false).
bool find_tuning(int extent, int taps, brick_tuning &t)
{
	std::lock_guard<std::mutex> lock(tuning_mutex);
	auto found = taps > 0 ? tuning_table.find(extent + taps * taps_key) : tuning_table.end();
	if (found == tuning_table.end())
	{
		found = tuning_table.find(extent);
	}
	if (found == tuning_table.end())
	{
		found = tuning_table.find(0);
	}
	if (found == tuning_table.end())
	{
		return false;
	}
	t = found->second;
	return true;
}

// The same, or `fallback` without an entry.
brick_tuning tuning_for(int extent, int taps, const brick_tuning &fallback)
{
	brick_tuning t = fallback;
	find_tuning(extent, taps, t);
	return t;
}

// The bricks of one call.
struct brick_choice
{
	brick_tuning bricks;
	bool voxels; // they own voxels
	bool wide;   // wide rounds
};

template <int PROFILE, int EX, int EY, int EZ>
void launch_brick_shape(const insertion_params &p, slice_chunk chunk, const prepared_sample *prepared, const int4 *tasks,
	int task_count, bool wide, const accumulator_input *input, hipStream_t stream)
{
	const dim3 grid(static_cast<unsigned>(task_count), static_cast<unsigned>(p.map.kept_count));
	const auto launch = [&](auto odd, auto voxels, auto rounds)
	{
		brick_kernel<PROFILE, decltype(odd)::value, decltype(voxels)::value, decltype(rounds)::value, EX, EY, EZ>
			<<<grid, 64, 0, stream>>>(p, chunk, prepared, tasks, task_count,
				input != nullptr ? *input : accumulator_input{});
	};
	if constexpr (PROFILE == REXLIB_HIP_KAISER_BESSEL)
	{
		if (wide)
		{
			const auto launch_wide = [&](auto odd)
			{
				p.taps == 4 ? launch(odd, std::false_type(), std::integral_constant<int, wide_rounds>()) :
					launch(odd, std::false_type(), std::integral_constant<int, wide_narrow_rounds>());
			};
			p.big % 2 == 1 ? launch_wide(std::true_type()) : launch_wide(std::false_type());
			return;
		}
	}
	constexpr std::integral_constant<int, claimed_rounds> claimed{};
	if constexpr (PROFILE != REXLIB_HIP_KAISER_BESSEL && EX == voxel_tuning.ex && EY == voxel_tuning.ey &&
		EZ == voxel_tuning.ez)
	{
		if (input != nullptr)
		{
			p.big % 2 == 1 ? launch(std::true_type(), std::true_type(), claimed) :
				launch(std::false_type(), std::true_type(), claimed);
			return;
		}
	}
	p.big % 2 == 1 ? launch(std::true_type(), std::false_type(), claimed) :
		launch(std::false_type(), std::false_type(), claimed);
}

template <int PROFILE>
void launch_brick(const insertion_params &p, slice_chunk chunk, const prepared_sample *prepared, const int4 *tasks,
	int task_count, const brick_tuning &t, bool wide, const accumulator_input *input, hipStream_t stream)
{
	if (t.ex == 16 && t.ey == 8 && t.ez == 8)
	{
		launch_brick_shape<PROFILE, 16, 8, 8>(p, chunk, prepared, tasks, task_count, wide, input, stream);
	}
	else if (t.ex == 16 && t.ey == 16)
	{
		launch_brick_shape<PROFILE, 16, 16, 8>(p, chunk, prepared, tasks, task_count, wide, input, stream);
	}
	else if (t.ex == 8 && t.ey == 8 && t.ez == 8)
	{
		launch_brick_shape<PROFILE, 8, 8, 8>(p, chunk, prepared, tasks, task_count, wide, input, stream);
	}
	else if (t.ex == 8 && t.ey == 8 && t.ez == 6)
	{
		launch_brick_shape<PROFILE, 8, 8, 6>(p, chunk, prepared, tasks, task_count, wide, input, stream);
	}
	else if (t.ex == 8 && t.ey == 8)
	{
		launch_brick_shape<PROFILE, 8, 8, 4>(p, chunk, prepared, tasks, task_count, wide, input, stream);
	}
	else if (t.ex == 8)
	{
		launch_brick_shape<PROFILE, 8, 6, 6>(p, chunk, prepared, tasks, task_count, wide, input, stream);
	}
	else
	{
		launch_brick_shape<PROFILE, 16, 8, 6>(p, chunk, prepared, tasks, task_count, wide, input, stream);
	}
}

void dispatch_brick(const insertion_params &p, slice_chunk chunk, const prepared_sample *prepared, const int4 *tasks,
	int task_count, const brick_choice &choice, const accumulator_input *input, hipStream_t stream)
{
	switch (p.profile)
	{
	case REXLIB_HIP_BOX:
		launch_brick<REXLIB_HIP_BOX>(p, chunk, prepared, tasks, task_count, choice.bricks, choice.wide, input, stream);
		break;
	case REXLIB_HIP_TRIANGLE:
		launch_brick<REXLIB_HIP_TRIANGLE>(p, chunk, prepared, tasks, task_count, choice.bricks, choice.wide, input, stream);
		break;
	default:
		launch_brick<REXLIB_HIP_KAISER_BESSEL>(p, chunk, prepared, tasks, task_count, choice.bricks, choice.wide, input, stream);
		break;
	}
}

void dispatch_prepare(const insertion_params &p, slice_chunk chunk, prepared_sample *prepared, hipStream_t stream)
{
	const int64_t elements = static_cast<int64_t>(p.n) * p.h;
	const dim3 grid(static_cast<unsigned>((elements + 255) / 256),
		static_cast<unsigned>(std::min<int64_t>(p.map.kept_count * chunk.count, 65535)));
	switch (p.variant)
	{
	case variant_plain:
		prepare_kernel<variant_plain><<<grid, 256, 0, stream>>>(p, chunk, prepared);
		break;
	case variant_weighted:
		prepare_kernel<variant_weighted><<<grid, 256, 0, stream>>>(p, chunk, prepared);
		break;
	default:
		prepare_kernel<variant_ctf><<<grid, 256, 0, stream>>>(p, chunk, prepared);
		break;
	}
}

template <int VARIANT>
void launch_columns_prepare(const insertion_params &p, slice_chunk chunk, row_range held, prepared_sample *prepared,
	hipStream_t stream)
{
	const int n = p.n;
	const int columns = n % 2 == 0 ? n / 2 : p.h;
	const int64_t lines = p.map.kept_count * chunk.count * columns;
	const float2 *tw = twiddles(n);
	const two_factor::plan two = two_factor::make_plan(n);
	if (two.n != 0)
	{
		const unsigned blocks = two_factor::blocks_for(lines, two.lines);
		two_factor::with_class(two, [&](auto kind_class)
			{
				columns_prepare_two_kernel<VARIANT, decltype(kind_class)::value><<<blocks, dim3(two.lines, two.b),
					two_factor::shared_bytes(two), stream>>>(p, chunk, held, two, tw, prepared);
			});
		return;
	}
	const fft_plan plan = make_fft_plan(n);
	const int group = lines_per_group(n);
	const std::size_t shared = sizeof(float2) * (2 * group * (n + 1) + n) + group * (3 * sizeof(int64_t) + sizeof(int));
	const unsigned grid = xcd_grid(static_cast<unsigned>(std::min<int64_t>((lines + group - 1) / group, 1 << 20)));
	columns_prepare_kernel<VARIANT><<<grid, 256, shared, stream>>>(p, chunk, held, plan, tw, group, prepared);
}

void dispatch_columns_prepare(const insertion_params &p, slice_chunk chunk, row_range held, prepared_sample *prepared,
	hipStream_t stream)
{
	if (p.n != 256)
	{
		switch (p.variant)
		{
		case variant_plain:
			launch_columns_prepare<variant_plain>(p, chunk, held, prepared, stream);
			break;
		case variant_weighted:
			launch_columns_prepare<variant_weighted>(p, chunk, held, prepared, stream);
			break;
		default:
			launch_columns_prepare<variant_ctf>(p, chunk, held, prepared, stream);
			break;
		}
		return;
	}
	// 8 blocks of 16 columns per slice.
	const unsigned grid = static_cast<unsigned>(p.map.kept_count * chunk.count * 8);
	const float2 *tw = twiddles(256);
	switch (p.variant)
	{
	case variant_plain:
		columns_prepare256_kernel<variant_plain><<<grid, 256, 0, stream>>>(p, chunk, held, tw, prepared);
		break;
	case variant_weighted:
		columns_prepare256_kernel<variant_weighted><<<grid, 256, 0, stream>>>(p, chunk, held, tw, prepared);
		break;
	default:
		columns_prepare256_kernel<variant_ctf><<<grid, 256, 0, stream>>>(p, chunk, held, tw, prepared);
		break;
	}
}

// The tasks of a brick grid as (packed box, (share, shares)) pairs,
// heaviest first, for slice counts up to `bucket`, on a device that runs
// `slots` brick wavefronts at once.
//
// A plane through the origin meets a brick at distance r with probability
// about min(1, 13 / r), and the samples it leaves there grow as the brick
// nears the origin (the plane's section of the brick widens), about as
// 1 / r down to the brick's half diagonal. The expected load of a brick is
// taken as bucket * 13 / max(r, half diagonal) plane hits, and a brick is
// split into shares of at most `target` of them -- or fewer, so that no task
// carries more than the average load of a slot (the total over `slots`):
// a task longer than that would outlast the rest of the launch.
std::vector<int4> brick_task_items(int big, int64_t bucket, int target, int ex, int ey, int ez, int taps, int slots,
	bool voxels)
{
	const int half = big / 2;
	// First-tap cells: x in [-(taps - 1), N/2]; y, z in [-(N/2) - (taps - 1),
	// N/2] (even N: the ends -N/2 and N/2 are one stored element; odd N: N
	// values from -(N/2)).
	const int reach = taps - 1;
	// Whether the voxels [first, first + count + taps - 1) hold -N/2 or N/2.
	const auto aliased = [&](int first, int count)
	{
		const int end = first + count + reach;
		return (first <= -half && -half < end) || (first <= half && half < end);
	};
	// Bricks that own voxels overlap by the taps - 1 cells whose samples reach
	// the next brick's first voxels.
	const int overlap = voxels ? reach : 0;
	const auto starts = [overlap](int low, int high, int edge)
	{
		std::vector<std::pair<int, int>> out;
		for (int s = low; s + overlap <= high; s += edge - overlap)
		{
			out.emplace_back(s, std::min(edge, high - s + 1));
		}
		return out;
	};
	struct item
	{
		int4 box;
		int4 share;
		double load;
	};
	struct brick
	{
		int4 box;
		double load;
	};
	std::vector<brick> bricks;
	double total = 0.0;
	const double half_diagonal = 0.5 * std::sqrt(static_cast<double>(ex * ex + ey * ey + ez * ez));
	for (const auto &z : starts(-half - reach, half, ez))
	{
		for (const auto &y : starts(-half - reach, half, ey))
		{
			for (const auto &x : starts(-reach, half, ex))
			{
				const bool alias = big % 2 == 0 && (aliased(z.first, z.second) || aliased(y.first, y.second));
				const int w = x.second | (y.second << 8) | (z.second << 16) | ((alias ? 0 : 1) << 24);
				const double cx = x.first + 0.5 * (x.second - 1);
				const double cy = y.first + 0.5 * (y.second - 1);
				const double cz = z.first + 0.5 * (z.second - 1);
				const double r = std::sqrt(cx * cx + cy * cy + cz * cz);
				const double load = static_cast<double>(bucket) * 13.0 / std::max(r, std::max(half_diagonal, 1.0));
				bricks.push_back({make_int4(x.first, y.first, z.first, w), load});
				total += load;
			}
		}
	}
	const double limit = std::min<double>(target, std::max(16.0, total / std::max(slots, 1)));
	std::vector<item> items;
	for (const brick &b : bricks)
	{
		const int shares = static_cast<int>(std::min<double>(64.0, std::max(1.0, std::ceil(b.load / limit))));
		for (int c = 0; c < shares; ++c)
		{
			items.push_back({b.box, make_int4(c, shares, 0, 0), b.load / shares});
		}
	}
	std::stable_sort(items.begin(), items.end(), [](const item &a, const item &b) { return a.load > b.load; });
	std::vector<int4> host;
	for (const auto &i : items)
	{
		host.push_back(i.box);
		host.push_back(i.share);
	}
	return host;
}

// The tasks of a volume of extent N receiving `slices` slices per
// accumulator, cached per device, extent, slice-count bucket, share target
// and brick shape.
struct task_list
{
	std::vector<int4> host;
	int split = 0; // the tasks up to the last one of a split brick
	int4 *device = nullptr;
};

std::mutex task_mutex;
std::map<std::tuple<int, int, int64_t, int, int, int, int, int, bool, bool>, task_list> task_cache;

int64_t slice_bucket(int64_t slices)
{
	int64_t bucket = 1;
	while (bucket < slices)
	{
		bucket *= 2;
	}
	return bucket;
}

// The cached list for a call (made on first use); the caller holds task_mutex.
task_list &brick_task_list(int big, int64_t slices, const brick_choice &choice, int taps)
{
	const brick_tuning &tuning = choice.bricks;
	const bool wide = choice.wide;
	int device = 0;
	REXLIB_HIP_CHECK(hipGetDevice(&device));
	const int64_t bucket = slice_bucket(slices);
	const auto key = std::make_tuple(device, big, bucket, tuning.share, tuning.ex, tuning.ey, tuning.ez, taps, wide,
		choice.voxels);
	auto found = task_cache.find(key);
	if (found == task_cache.end())
	{
		// Brick wavefronts resident at once: as many per CU as its 160 KiB of
		// LDS holds (the brick's voxels, claim bytes or axis weights, 64
		// markers and 64 queued slices, in 512-byte granules).
		int units = 0;
		REXLIB_HIP_CHECK(hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, device));
		const int lx = tuning.ex + taps - 1, ly = tuning.ey + taps - 1, lz = tuning.ez + taps - 1;
		const int pitch_z = brick_pitch_z(wide, brick_pitch_y(wide, lx), ly);
		const int lds = static_cast<int>(align_up(static_cast<std::size_t>(pitch_z * lz * 12 +
			(wide ? 64 * 48 : tuning.ex * tuning.ey * tuning.ez) + 2 * 64 * 4), 512));
		found = task_cache.emplace(key, task_list{}).first;
		found->second.host = brick_task_items(big, bucket, tuning.share, tuning.ex, tuning.ey, tuning.ez, taps,
			units * std::max(1, (160 * 1024) / lds), choice.voxels);
		for (std::size_t i = 0; i < found->second.host.size(); i += 2)
		{
			if (found->second.host[i + 1].y > 1)
			{
				found->second.split = static_cast<int>(i / 2) + 1;
			}
		}
	}
	return found->second;
}

// Workspace bytes the task list of a call takes (with its alignment).
std::size_t brick_task_bytes(int big, int64_t slices, const brick_choice &choice, int taps)
{
	std::lock_guard<std::mutex> lock(task_mutex);
	return align_up(sizeof(int4) * brick_task_list(big, slices, choice, taps).host.size(), 256) + 256;
}

// The device copy of a call's tasks. With a fixed workspace buffer the list
// is copied into it from the host copy the cache keeps (nothing allocated);
// otherwise the device copy is made once and cached.
const int4 *brick_tasks(int big, int64_t slices, const brick_choice &choice, int taps,
	workspace_source &workspace, hipStream_t stream, int &count, int &split)
{
	std::lock_guard<std::mutex> lock(task_mutex);
	task_list &list = brick_task_list(big, slices, choice, taps);
	count = static_cast<int>(list.host.size() / 2);
	split = list.split;
	const std::size_t bytes = sizeof(int4) * list.host.size();
	if (workspace.arena != nullptr)
	{
		int4 *at = static_cast<int4 *>(workspace.take(area_insertion, bytes, stream));
		REXLIB_HIP_CHECK(hipMemcpyAsync(at, list.host.data(), bytes, hipMemcpyHostToDevice, stream));
		return at;
	}
	if (list.device == nullptr)
	{
		REXLIB_HIP_CHECK(hipMalloc(&list.device, bytes));
		REXLIB_HIP_CHECK(hipMemcpy(list.device, list.host.data(), bytes, hipMemcpyHostToDevice));
	}
	return list.device;
}

// Whether the bricks of a call own voxels rather than first-tap cells. A brick
// of cells adds its voxels on the faces that other bricks also reach by
// atomics (they bypass the L2 of an XCD), after a copy of the inputs; a brick
// of voxels writes each of them once, input plus sum, but inserts the samples
// of its T - 1 lower cell layers a second time (512 / 343 of the samples for 8
// x 8 x 8 and two taps). The line is at the density where the one costs what
// the other does, in samples per voxel of the stored half: 256 slices of 256^2
// into 512^3 (0.1 samples per voxel) take 1.15 against 1.75 ms, 512 of 256^2
// into 256^3 (1.6) 0.47 against 0.51 ms, 1,024 (3.1) 0.75 against 0.71 ms. Four
// taps would insert 4 times the samples; a fixed workspace buffer (`fixed`) keeps
// the smaller task list of cells.
bool bricks_own_voxels(int n, int big, int64_t slices, int taps, bool fixed)
{
	const double samples = 0.125 * 3.14159265 * n * n * static_cast<double>(slice_bucket(slices));
	const double voxels = 0.5 * big * big * static_cast<double>(big);
	return taps <= 2 && !fixed && samples < 1.6 * voxels;
}

// Kaiser-Bessel windows of 4 taps add one sample at a time, its taps on the 64
// lanes (wide rounds), while the call has too few samples to keep every
// wavefront's claims busy: 256 slices of 128^2 into 256^3 (1.6 million samples)
// take 0.53 ms against 0.78, 1,024 (6.6 million) 0.81 against 0.92, but 300 of
// 256^2 (7.7 million) 0.82 against 0.71, 1,500 3.3 against 2.7 and 2,048 of 128^2
// into 128^3 (13 million) 1.4 against 1.1. Narrower windows leave those lanes
// idle (3 taps, 300 of 256^2: 1.13 against 0.53 ms); 3 taps take wide rounds only
// in small calls into twice the slices' extent and below 200^3, whose bricks meet
// few samples of a slice: 512 of 64^2 into 128^3 0.18 against 0.24 ms.
//
// A task of claimed rounds takes several times as long per plane hit as one of
// two taps, so an entry's share is cut to 128 (300 of 256^2: 0.71 against 0.99 ms
// with 512).
//
// Sparse calls into large volumes (below 0.25 samples per voxel of the stored
// half, from 200^3 on) spend their time on the atomics of the bricks' faces, of
// which large bricks have fewer: claimed rounds in 16 x 8 x 6 bricks take 0.90 ms
// for 100 slices of 256^2 into 384^3 against 1.20 wide in 8 x 6 x 6, 0.55 against
// 0.75 for 150 of 200^2 into 300^3, 2.4 against 3.2 for 256 of 256^2 into 512^3.
// Below 200^3 the small bricks' tasks win (16 of 128^2 into 128^3 87 against 106
// us), and so do wide rounds for a slice or two (1 of 256^2 into 256^3 63 against
// 72 us).
brick_choice kaiser_bessel_bricks(int n, int big, int64_t slices, int64_t volumes, int window_taps)
{
	const double samples = 0.125 * 3.14159265 * n * n * static_cast<double>(slices);
	const double voxels = 0.5 * big * big * static_cast<double>(big);
	brick_choice c{untuned_wide_bricks, false, false};
	const bool entry = find_tuning(big, 4, c.bricks);
	const bool sparse = !entry && big >= 200 && samples < 0.25 * voxels && samples >= 5e4;
	const double all = samples * static_cast<double>(volumes);
	c.wide = window_taps == 4 ? !sparse && all < 7e6 :
		window_taps == 3 && big >= 2 * n && big < 200 && all < 1e6;
	if (!c.wide)
	{
		if (!entry)
		{
			c.bricks = sparse ? untuned_sparse_bricks : untuned_claimed_bricks;
		}
		c.bricks.share = std::min(c.bricks.share, untuned_claimed_bricks.share);
	}
	return c;
}

// The bricks of a call of `slices` slices into each of `volumes` volumes, for a
// brick layout of `taps` and a window of `window_taps` per axis.
brick_choice choose_bricks(int n, int big, int64_t slices, int64_t volumes, int taps, int window_taps, bool fixed)
{
	if (taps == 4)
	{
		return kaiser_bessel_bricks(n, big, slices, volumes, window_taps);
	}
	const double samples = 0.125 * 3.14159265 * n * n * static_cast<double>(slices);
	const bool small = samples * static_cast<double>(volumes) < 3e6 || bricks_own_voxels(n, big, slices, taps, false);
	brick_choice c{small ? untuned_small_bricks : untuned_bricks, bricks_own_voxels(n, big, slices, taps, fixed), false};
	const bool entry = find_tuning(big, taps, c.bricks);
	if (c.voxels)
	{
		// Their own shape, and an entry's share up to their own: 1,024 slices of
		// 128^2 into 256^3 take 0.31 ms with 512 and 0.38 with 1,024.
		const int share = entry ? c.bricks.share : voxel_tuning.share;
		c.bricks = voxel_tuning;
		c.bricks.share = std::min(share, voxel_tuning.share);
	}
	return c;
}

// Prepared samples take 12 bytes per stored element of a slice; a chunk of slices
// stays within 4 GiB.
constexpr int64_t prepared_limit = int64_t(4) << 30;

int64_t prepared_bytes(int n)
{
	return static_cast<int64_t>(n) * (n / 2 + 1) * static_cast<int64_t>(sizeof(prepared_sample));
}

// Whether an out-of-place call of bricks that own voxels still copies the inputs
// first and inserts in place. The bricks' own copy runs in rows of 7 voxels,
// whose ends share cache lines with other bricks: an empty brick copies at half
// the rate of copy_accumulators_kernel, but a brick with samples saves a pass.
// The line is at 0.04 samples per voxel of the stored half: 16 slices of 256^2
// into 512^3 (0.006) take 0.64 copied against 0.88 ms, 64 (0.025) 0.89 against
// 0.93, 128 (0.05) 1.05 against 0.98; 32 of 128^2 into 256^3 (0.025) 118 against
// 128 us, 128 (0.1) 149 against 144. Where inputs and outputs fit the L2s (8 x 4
// MiB), the copy costs less still: 64 of 64^2 into 128^3 (0.1) 52.5 against 55.7
// us, 64 of 99^2 into 99^3 (0.5) 50.8 against 54.6.
bool copy_first(const insertion_params &p, int64_t slices)
{
	const double samples = 0.125 * 3.14159265 * p.n * p.n * static_cast<double>(slices);
	const double voxels = 0.5 * p.big * p.big * static_cast<double>(p.big);
	const double bytes = 2.0 * (sizeof(float2) + sizeof(float)) * voxels * static_cast<double>(p.map.kept_count);
	return samples < 0.04 * voxels || bytes <= 8.0 * (4 << 20);
}

} // anonymous namespace

void set_insertion_tuning(int extent, int taps, int extent_x, int extent_y, int extent_z, int share)
{
	if (extent < 0 || extent >= taps_key)
	{
		fail(REXLIB_HIP_INVALID_ARGUMENT, "insertion tuning: the extent must be 0 (every extent) or positive, "
			"below 2^20");
	}
	if (taps != 0 && taps != 1 && taps != 2 && taps != 4)
	{
		fail(REXLIB_HIP_INVALID_ARGUMENT, "insertion tuning: taps per axis are 0 (every window), 1 (nearest), "
			"2 (trilinear) or 4 (Kaiser-Bessel)");
	}
	if (!valid_brick_shape(extent_x, extent_y, extent_z))
	{
		fail(REXLIB_HIP_INVALID_ARGUMENT, "insertion tuning: brick extents (x, y, z) are (16, 8, 6), (16, 8, 8), "
			"(16, 16, 8), (8, 8, 8), (8, 8, 6), (8, 8, 4) or (8, 6, 6)");
	}
	if (share < 16 || share > (1 << 20))
	{
		fail(REXLIB_HIP_INVALID_ARGUMENT, "insertion tuning: plane hits per task lie in [16, 2^20]");
	}
	std::lock_guard<std::mutex> lock(tuning_mutex);
	tuning_table[extent + taps * taps_key] = brick_tuning{extent_x, extent_y, extent_z, share};
}

void get_insertion_tuning(int extent, int *extent_x, int *extent_y, int *extent_z, int *share)
{
	const brick_tuning t = tuning_for(extent, 0, untuned_bricks);
	*extent_x = t.ex;
	*extent_y = t.ey;
	*extent_z = t.ez;
	*share = t.share;
}

void insertion_bricks(int n, int extent, int taps, int64_t slices, int *extent_x, int *extent_y, int *extent_z,
	int *share, int *own_voxels)
{
	if (taps < 1 || taps > 4)
	{
		fail(REXLIB_HIP_INVALID_ARGUMENT, "insertion bricks: taps per axis are 1 (nearest), 2 (trilinear), 3 (a "
			"Kaiser-Bessel window of up to 3 taps) or 4 (Kaiser-Bessel)");
	}
	if (n < 1 || extent < 1 || slices < 1)
	{
		fail(REXLIB_HIP_INVALID_ARGUMENT, "insertion bricks: the extents and the number of slices must be positive");
	}
	const int64_t chunk = std::min(slices, std::max<int64_t>(1, prepared_limit / prepared_bytes(n)));
	const brick_choice c = choose_bricks(n, extent, chunk, 1, taps >= 3 ? 4 : taps, taps, false);
	*extent_x = c.bricks.ex;
	*extent_y = c.bricks.ey;
	*extent_z = c.bricks.ez;
	*share = c.bricks.share;
	*own_voxels = c.voxels ? 1 : 0;
}

bool drop_insertion_tuning(int extent, int taps, int *extent_x, int *extent_y, int *extent_z, int *share)
{
	if (taps != 0 && taps != 1 && taps != 2 && taps != 4)
	{
		fail(REXLIB_HIP_INVALID_ARGUMENT, "insertion tuning: taps per axis are 0 (every window), 1 (nearest), "
			"2 (trilinear) or 4 (Kaiser-Bessel)");
	}
	std::lock_guard<std::mutex> lock(tuning_mutex);
	const auto found = tuning_table.find(extent + taps * taps_key);
	if (extent < 0 || extent >= taps_key || found == tuning_table.end())
	{
		return false;
	}
	*extent_x = found->second.ex;
	*extent_y = found->second.ey;
	*extent_z = found->second.ez;
	*share = found->second.share;
	tuning_table.erase(found);
	return true;
}

void clear_insertion_tuning()
{
	std::lock_guard<std::mutex> lock(tuning_mutex);
	tuning_table.clear();
}

// The row transforms of images [first, last) of a pending image insertion;
// `image_rows`: the zero rows of the padding are left out (the column pass
// that follows does not read them).
void launch_rows(const pending_columns &columns, int64_t first, int64_t last, bool image_rows, hipStream_t stream)
{
	const pending_rows &rows = *columns.rows;
	if (last <= first)
	{
		return;
	}
	line_set in = rows.in_rows;
	in.count = (last - first) * rows.m;
	line_set out = rows.out_rows;
	out.count = (last - first) * rows.n;
	const char *images = static_cast<const char *>(rows.images) +
		first * rows.in_rows.s_outer * static_cast<int64_t>(rows.element_bytes);
	const float *scales = rows.scales != nullptr ? rows.scales + first * rows.scale_stride : nullptr;
	launch_rfft_rows(rows.kind, images, in, rows.m, scales, rows.scale_stride,
		columns.spectra + first * rows.out_rows.s_outer, out, padded_rows(rows.m, rows.n, last - first, image_rows), rows.n,
		stream);
}

// Host entry of every insertion: fills the workspace and launches.
void run_insertion(insertion_params p, int schedule, const float2 *num_in, const int64_t *num_in_strides,
	const float *den_in, const int64_t *den_in_strides, bool in_place, double shape, const pending_columns *columns,
	workspace_source &workspace, hipStream_t stream)
{
	const int64_t slices = p.slice_count;
	const int n = p.n;
	const int h = p.h;

	// Workspace: entries, phase tables, the window table, the volume phases.
	static_assert(sizeof(slice_entry) == 96 && sizeof(slice_plane) == 16, "an entry and its plane take 112 bytes");
	const std::size_t entry_bytes = align_up((sizeof(slice_entry) + sizeof(slice_plane)) *
		std::max<int64_t>(slices, 1), 256);
	const std::size_t table_bytes = align_up(sizeof(float2) * (h + n) * std::max<int64_t>(slices, 1), 256);
	const std::size_t kb_bytes = align_up(sizeof(float) * (p.kb_count + 3), 256);
	const std::size_t phase_bytes = align_up(sizeof(float2) * p.big, 256);
	char *base = static_cast<char *>(
		workspace.take(area_insertion, entry_bytes + table_bytes + kb_bytes + phase_bytes, stream));
	p.entries = reinterpret_cast<slice_entry *>(base);
	p.planes = reinterpret_cast<slice_plane *>(p.entries + slices);
	p.tables = reinterpret_cast<float2 *>(base + entry_bytes);
	float *kb = reinterpret_cast<float *>(base + entry_bytes + table_bytes);
	float2 *vphase = reinterpret_cast<float2 *>(base + entry_bytes + table_bytes + kb_bytes);
	p.kb_table = kb;
	p.volume_phase = vphase;

	const auto copy_inputs = [&]()
	{
		const int64_t total = static_cast<int64_t>(p.big) * p.big * p.half * p.map.kept_count;
		if (in_place || total == 0)
		{
			return;
		}
		const unsigned blocks = static_cast<unsigned>(std::min<int64_t>((total + 255) / 256, 1 << 20));
		copy_accumulators_kernel<<<blocks, 256, 0, stream>>>(p, num_in, num_in_strides[0], num_in_strides[1],
			num_in_strides[2], den_in, den_in_strides[0], den_in_strides[1], den_in_strides[2]);
		REXLIB_HIP_CHECK(hipGetLastError());
	};
	if (slices == 0)
	{
		copy_inputs();
		return;
	}

	if (p.profile == REXLIB_HIP_KAISER_BESSEL)
	{
		kb_table_kernel<<<(p.kb_count + 3 + 255) / 256, 256, 0, stream>>>(kb, p.kb_count, shape);
		REXLIB_HIP_CHECK(hipGetLastError());
	}
	if (p.big % 2 == 1)
	{
		volume_phase_kernel<<<(p.big + 255) / 256, 256, 0, stream>>>(vphase, p.big);
		REXLIB_HIP_CHECK(hipGetLastError());
	}
	// The slices of one call go through in chunks whose prepared samples stay
	// within prepared_limit, and with a fixed workspace buffer within what it has
	// left beside the task list. The
	// brick schedule needs the window to span at most 4 voxels; wider
	// Kaiser-Bessel windows take the scatter schedule, and so do calls whose
	// workspace buffer cannot hold one slice's prepared samples.
	const int64_t per_slice = prepared_bytes(p.n) * p.map.kept_count;
	// Taps per axis of the brick layout: 1, 2, or 4 for every Kaiser-Bessel window.
	const int layout_taps = p.profile == REXLIB_HIP_BOX ? 1 : (p.profile == REXLIB_HIP_TRIANGLE ? 2 : 4);
	int64_t chunk_count = 0;
	brick_choice choice{untuned_bricks, false, false};
	if (schedule != schedule_scatter && p.taps <= 4 && p.map.kept_count <= 65535)
	{
		const auto room = [&](std::size_t reserved)
		{
			const std::size_t left = workspace.remaining();
			return left <= reserved + 512 ? int64_t(0) :
				std::min<int64_t>(prepared_limit, static_cast<int64_t>(std::min<std::size_t>(left - reserved - 512,
					std::size_t(1) << 40)));
		};
		chunk_count = std::min<int64_t>(p.map.reduced_count, room(0) / per_slice);
		if (chunk_count >= 1)
		{
			choice = choose_bricks(p.n, p.big, chunk_count, p.map.kept_count, layout_taps, p.taps,
				workspace.arena != nullptr);
		}
		if (chunk_count >= 1 && workspace.arena != nullptr)
		{
			// Tasks made for more slices stay valid for fewer (their shares
			// are fractions of a chunk).
			chunk_count = std::min<int64_t>(chunk_count,
				room(brick_task_bytes(p.big, chunk_count, choice, layout_taps)) / per_slice);
		}
	}
	const bool brick = chunk_count >= 1;
	const bool voxels = brick && choice.voxels;
	// Bricks that own voxels read the inputs themselves, unless most of them
	// would have nothing to add.
	const bool copied = !voxels || copy_first(p, chunk_count);
	if (copied)
	{
		copy_inputs();
	}
	// Pending column transforms run inside the preparation of each chunk on
	// the brick schedule; on the scatter schedule they run here, in place.
	const bool fused_columns = columns != nullptr && brick;
	// Pending row transforms run per chunk (just before the chunk's column
	// pass, so a chunk's spectra are still in the caches) when every chunk is
	// a range of the images (one volume), else here for all images.
	const bool chunk_rows = fused_columns && columns->rows != nullptr && p.map.kept_count == 1;
	if (columns != nullptr && columns->rows != nullptr && !chunk_rows)
	{
		launch_rows(*columns, 0, columns->rows->in_rows.count / columns->rows->m, fused_columns, stream);
	}
	if (columns != nullptr && !fused_columns && columns->lines.count > 0)
	{
		launch_fft_lines(columns->spectra, columns->lines, columns->spectra, columns->lines, p.n, -1.0f, 1.0f,
			stream);
	}
	settle_kernel<<<static_cast<unsigned>(std::min<int64_t>(slices, 1 << 20)), 128, 0, stream>>>(p);
	REXLIB_HIP_CHECK(hipGetLastError());

	if (brick)
	{
		// The rows of the slices that hold image rows; the others are zero.
		const row_range held = columns != nullptr && columns->rows != nullptr ?
			row_range{n / 2 - columns->rows->m / 2, n / 2 - columns->rows->m / 2 + columns->rows->m} : row_range{0, n};
		int count = 0;
		int split = 0; // tasks of split bricks, the first ones
		const int4 *tasks = brick_tasks(p.big, chunk_count, choice, layout_taps, workspace, stream, count, split);
		prepared_sample *prepared = static_cast<prepared_sample *>(workspace.take(area_prepared,
			static_cast<std::size_t>(per_slice * chunk_count), stream));
		for (int64_t begin = 0; begin < p.map.reduced_count; begin += chunk_count)
		{
			const slice_chunk chunk{begin, std::min(chunk_count, p.map.reduced_count - begin)};
			if (chunk_rows)
			{
				launch_rows(*columns, chunk.begin, chunk.begin + chunk.count, true, stream);
			}
			const int prepare_token = timing_begin(REXLIB_HIP_KERNEL_PREPARE, stream);
			if (fused_columns)
			{
				dispatch_columns_prepare(p, chunk, held, prepared, stream);
			}
			else
			{
				dispatch_prepare(p, chunk, prepared, stream);
			}
			REXLIB_HIP_CHECK(hipGetLastError());
			timing_end(prepare_token, stream);
			const int brick_token = timing_begin(REXLIB_HIP_KERNEL_BRICK, stream);
			const bool from_outputs = in_place || copied || begin > 0;
			const accumulator_input input = from_outputs ?
				accumulator_input{p.numerator, p.num_s0, p.num_s1, p.num_s2, p.denominator, p.den_s0, p.den_s1, p.den_s2,
					slot_numerator_out, slot_denominator_out, true} :
				accumulator_input{num_in, num_in_strides[0], num_in_strides[1], num_in_strides[2], den_in,
					den_in_strides[0], den_in_strides[1], den_in_strides[2], slot_numerator, slot_denominator, false};
			const unsigned shared_blocks = static_cast<unsigned>(split + (p.big % 2 == 0 ? 2 * p.big - 1 : 0));
			if (voxels && !input.in_place && shared_blocks > 0)
			{
				const dim3 grid(shared_blocks, static_cast<unsigned>(p.map.kept_count));
				const auto kernel = layout_taps == 1 ? copy_shared_inputs_kernel<1> : copy_shared_inputs_kernel<2>;
				kernel<<<grid, 64, 0, stream>>>(p, tasks, split, input);
				REXLIB_HIP_CHECK(hipGetLastError());
			}
			dispatch_brick(p, chunk, prepared, tasks, count, choice, voxels ? &input : nullptr, stream);
			REXLIB_HIP_CHECK(hipGetLastError());
			timing_end(brick_token, stream);
		}
	}
	else
	{
		const int scatter_token = timing_begin(REXLIB_HIP_KERNEL_SCATTER, stream);
		switch (p.variant)
		{
		case variant_plain:
			dispatch_scatter<variant_plain>(p, stream);
			break;
		case variant_weighted:
			dispatch_scatter<variant_weighted>(p, stream);
			break;
		default:
			dispatch_scatter<variant_ctf>(p, stream);
			break;
		}
		timing_end(scatter_token, stream);
	}
	REXLIB_HIP_CHECK(hipGetLastError());
}

} // namespace rexlib_hip
