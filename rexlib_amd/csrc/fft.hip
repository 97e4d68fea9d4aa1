// Batched FFTs on gfx950.
//
// Lengths of two register factors (every 2-3-5 length from 48 to 1,024 but
// 125, 243, 972 and 1,000, fft_two.hpp) hold a line in the registers of its
// threads and exchange it once through LDS: 4.5 to 5.5 TB/s of the operand
// read and written, from 64 to 512 points, where the LDS stages below reach
// 1.7 to 2.9. The other lengths stage a group of lines in LDS, run the
// radix-4/2/3/5 Stockham stages there (ping-pong between two LDS buffers, one
// butterfly per thread per step), and write the lines back. Real transforms
// pack two real rows of one transform (row_pairs) into one complex line and
// separate the two half spectra afterwards, so a real row costs half a complex
// transform.
//
// Conventions follow pocketfft as rexlib calls it
// (src/backends/cpu/kernels/pocketfft_fourier_transform.cpp:74-163): the
// forward transform is unscaled with exp(-2 pi i), the inverse uses
// exp(+2 pi i) and a scale of 1/n per axis
// (src/ops/fourier/fourier_normalization.cpp:56-71). A complex-to-real
// transform ignores the imaginary parts of the self-conjugate elements.
#include "fft.hpp"
#include "fft_device.hpp"
#include "fft_two.hpp"

#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>

#include <cmath>
#include <cstdint>
#include <map>
#include <mutex>
#include <type_traits>
#include <vector>

namespace rexlib_hip
{

fft_plan make_fft_plan(int64_t n)
{
	fft_plan plan{};
	plan.n = static_cast<int32_t>(n);
	int64_t rest = n;
	const int radices[] = {4, 2, 3, 5};
	// Radix 4 first, then a single 2, then 3 and 5.
	while (rest % 4 == 0)
	{
		plan.radix[plan.stages++] = 4;
		rest /= 4;
	}
	for (const int r : radices)
	{
		while (rest % r == 0)
		{
			if (plan.stages == max_fft_stages)
			{
				fail(REXLIB_HIP_UNSUPPORTED, "fft: length has too many factors");
			}
			plan.radix[plan.stages++] = r;
			rest /= r;
		}
	}
	if (rest != 1)
	{
		fail(REXLIB_HIP_UNSUPPORTED,
			"fft: the gfx950 transforms take lengths whose prime factors are 2, 3, and 5, not " +
				std::to_string(n));
	}
	return plan;
}

const float2 *twiddles(int64_t n)
{
	static std::mutex mutex;
	static std::map<std::pair<int, int64_t>, float2 *> cache;
	int device = 0;
	REXLIB_HIP_CHECK(hipGetDevice(&device));
	std::lock_guard<std::mutex> lock(mutex);
	const auto key = std::make_pair(device, n);
	const auto found = cache.find(key);
	if (found != cache.end())
	{
		return found->second;
	}
	std::vector<float2> host(static_cast<std::size_t>(n));
	for (int64_t m = 0; m < n; ++m)
	{
		const double angle = -2.0 * 3.14159265358979323846 * static_cast<double>(m) / static_cast<double>(n);
		host[m] = make_float2(static_cast<float>(std::cos(angle)), static_cast<float>(std::sin(angle)));
	}
	float2 *device_table = nullptr;
	REXLIB_HIP_CHECK(hipMalloc(&device_table, sizeof(float2) * static_cast<std::size_t>(n)));
	REXLIB_HIP_CHECK(hipMemcpy(device_table, host.data(), sizeof(float2) * static_cast<std::size_t>(n),
		hipMemcpyHostToDevice));
	cache[key] = device_table;
	return device_table;
}

namespace
{

template <int KIND>
__device__ inline float load_real(const void *base, int64_t index);

template <>
__device__ inline float load_real<real_f32>(const void *base, int64_t index)
{
	return static_cast<const float *>(base)[index];
}

template <>
__device__ inline float load_real<real_bf16>(const void *base, int64_t index)
{
	return __bfloat162float(static_cast<const __hip_bfloat16 *>(base)[index]);
}

template <>
__device__ inline float load_real<real_f16>(const void *base, int64_t index)
{
	return __half2float(static_cast<const __half *>(base)[index]);
}

// Four consecutive elements from `index` (a multiple of 4, with the base
// aligned to four elements), as floats.
template <int KIND>
__device__ inline float4 load_real4(const void *base, int64_t index)
{
	if constexpr (KIND == real_f32)
	{
		return *reinterpret_cast<const float4 *>(static_cast<const float *>(base) + index);
	}
	else
	{
		const uint2 bits = *reinterpret_cast<const uint2 *>(static_cast<const unsigned short *>(base) + index);
		const unsigned short e[4] = {static_cast<unsigned short>(bits.x & 0xffff), static_cast<unsigned short>(bits.x >> 16),
			static_cast<unsigned short>(bits.y & 0xffff), static_cast<unsigned short>(bits.y >> 16)};
		float f[4];
#pragma unroll
		for (int i = 0; i < 4; ++i)
		{
			if constexpr (KIND == real_bf16)
			{
				f[i] = __uint_as_float(static_cast<unsigned>(e[i]) << 16);
			}
			else
			{
				f[i] = __half2float(__ushort_as_half(e[i]));
			}
		}
		return make_float4(f[0], f[1], f[2], f[3]);
	}
}

// WIDTH elements of a real row from element c, scaled (zeros when not live):
// one load of all of them (unit stride, base and row aligned to WIDTH
// elements) or, for WIDTH 1, one element at any stride.
template <int KIND, int WIDTH>
__device__ inline void load_reals(const void *base, bool live, int64_t row, int c, int64_t stride, float scale, float *v)
{
#pragma unroll
	for (int q = 0; q < WIDTH; ++q)
	{
		v[q] = 0.0f;
	}
	if (!live)
	{
		return;
	}
	if constexpr (WIDTH == 4)
	{
		const float4 f = load_real4<KIND>(base, row + c);
		v[0] = f.x;
		v[1] = f.y;
		v[2] = f.z;
		v[3] = f.w;
	}
	else if constexpr (WIDTH == 2 && KIND == real_f32)
	{
		const float2 f = *reinterpret_cast<const float2 *>(static_cast<const float *>(base) + row + c);
		v[0] = f.x;
		v[1] = f.y;
	}
	else if constexpr (WIDTH == 2)
	{
		const unsigned bits = *reinterpret_cast<const unsigned *>(static_cast<const unsigned short *>(base) + row + c);
		v[0] = KIND == real_bf16 ? __uint_as_float(bits << 16) :
			__half2float(__ushort_as_half(static_cast<unsigned short>(bits & 0xffff)));
		v[1] = KIND == real_bf16 ? __uint_as_float(bits & 0xffff0000u) :
			__half2float(__ushort_as_half(static_cast<unsigned short>(bits >> 16)));
	}
	else
	{
		v[0] = load_real<KIND>(base, row + c * stride);
	}
#pragma unroll
	for (int q = 0; q < WIDTH; ++q)
	{
		v[q] *= scale;
	}
}

// Rows of real images, two at a time, to half spectra. Images of extent m
// are zero-padded to the transform length n with their origin m/2 moved to
// n/2. Line set `in` lists the image rows, `out` the padded rows; `lines` says
// which of them run, and together. A block takes `pairs` lines at a time.
template <int KIND>
__global__ void rfft_rows_kernel(const void *in, line_set in_rows, int m, const float *scales,
	int64_t scale_stride, float2 *out, line_set out_rows, row_pairs lines, fft_plan plan, const float2 *tw, int pairs,
	float half)
{
	extern __shared__ float2 lds[];
	const int n = plan.n;
	const int h = n / 2 + 1;
	const int stride = n + 1;
	float2 *a = lds;
	float2 *b = lds + pairs * stride;
	float2 *twl = lds + 2 * pairs * stride;
	// Per padded row of the group: its first input element (-1: a zero row
	// of the padding or past the end) and its first output element.
	int64_t *row_in = reinterpret_cast<int64_t *>(twl + n);
	int64_t *row_out = row_in + 2 * pairs;
	float *row_scale = reinterpret_cast<float *>(row_out + 2 * pairs);
	for (int i = threadIdx.x; i < n; i += blockDim.x)
	{
		twl[i] = tw[i];
	}
	const int offset = n / 2 - m / 2;
	const int64_t total = line_count(lines);
	for (int64_t first = blockIdx.x * static_cast<int64_t>(pairs); first < total;
		first += static_cast<int64_t>(gridDim.x) * pairs)
	{
		for (int q = threadIdx.x; q < 2 * pairs; q += blockDim.x)
		{
			const line_row r = row_of(lines, first + q / 2, q & 1);
			row_in[q] = r.in >= 0 ? line_offset(in_rows, r.in) : -1;
			row_out[q] = r.out >= 0 ? line_offset(out_rows, r.out) : -1;
			row_scale[q] = scales != nullptr && r.in >= 0 ? scales[r.transform * scale_stride] : 1.0f;
		}
		__syncthreads();
		for (int t = threadIdx.x; t < pairs * n; t += blockDim.x)
		{
			const int p = t / n;
			const int i = t - p * n;
			const int c = i - offset;
			float value[2] = {0.0f, 0.0f};
			for (int q = 0; q < 2; ++q)
			{
				const int64_t src = row_in[2 * p + q];
				if (src >= 0 && c >= 0 && c < m)
				{
					value[q] = load_real<KIND>(in, src + c * in_rows.s_elem) * row_scale[2 * p + q];
				}
			}
			a[p * stride + i] = make_float2(value[0], value[1]);
		}
		__syncthreads();
		const float2 *z = block_fft(a, b, pairs, stride, plan, twl, -1.0f);
		for (int t = threadIdx.x; t < pairs * h; t += blockDim.x)
		{
			const int p = t / h;
			const int k = t - p * h;
			const float2 zk = z[p * stride + k];
			const float2 zm = cconj(z[p * stride + (n - k) % n]);
			const int64_t dst0 = row_out[2 * p];
			const int64_t dst1 = row_out[2 * p + 1];
			if (dst0 >= 0)
			{
				const float2 sum = cadd(zk, zm);
				out[dst0 + k * out_rows.s_elem] = make_float2(half * sum.x, half * sum.y);
			}
			if (dst1 >= 0)
			{
				// (zk - zm) / (2 i), times the scale
				const float2 diff = csub(zk, zm);
				out[dst1 + k * out_rows.s_elem] = make_float2(half * diff.y, -half * diff.x);
			}
		}
		__syncthreads();
	}
}

// Complex lines from `src` to `dst` (may be the same memory), `group` lines
// per step; consecutive lines of a group are loaded by consecutive threads.
__global__ void fft_lines_kernel(const float2 *src, line_set src_lines, float2 *dst, line_set dst_lines,
	fft_plan plan, const float2 *tw, float sign, float scale, int group)
{
	extern __shared__ float2 lds[];
	const int n = plan.n;
	const int stride = n + 1;
	float2 *a = lds;
	float2 *b = lds + group * stride;
	float2 *twl = lds + 2 * group * stride;
	int64_t *line_src = reinterpret_cast<int64_t *>(twl + n);
	int64_t *line_dst = line_src + group;
	for (int i = threadIdx.x; i < n; i += blockDim.x)
	{
		twl[i] = tw[i];
	}
	const int64_t total = src_lines.count;
	for (int64_t first = blockIdx.x * static_cast<int64_t>(group); first < total;
		first += static_cast<int64_t>(gridDim.x) * group)
	{
		const int lines = static_cast<int>(total - first < group ? total - first : group);
		for (int q = threadIdx.x; q < lines; q += blockDim.x)
		{
			line_src[q] = line_offset(src_lines, first + q);
			line_dst[q] = line_offset(dst_lines, first + q);
		}
		__syncthreads();
		for (int t = threadIdx.x; t < group * n; t += blockDim.x)
		{
			const int e = t / group;
			const int l = t - e * group;
			if (l < lines)
			{
				a[l * stride + e] = src[line_src[l] + e * src_lines.s_elem];
			}
		}
		__syncthreads();
		const float2 *z = block_fft(a, b, lines, stride, plan, twl, sign);
		for (int t = threadIdx.x; t < group * n; t += blockDim.x)
		{
			const int e = t / group;
			const int l = t - e * group;
			if (l < lines)
			{
				const float2 v = z[l * stride + e];
				dst[line_dst[l] + e * dst_lines.s_elem] = make_float2(v.x * scale, v.y * scale);
			}
		}
		__syncthreads();
	}
}

// Real 256-point rows, two to a complex line, by the four-step
// decomposition: a block takes 16 lines (32 rows). Thread (line l, j) loads
// elements j + 16 k of its two rows (16 consecutive elements per line and
// load across the lanes), transforms them with fft256_four_step, and stores
// Z[j + 16 k2] to LDS. The separation of the two half spectra
// (X_a = (Z_k + conj Z_{n-k}) / 2, X_b = (Z_k - conj Z_{n-k}) / 2i) then
// reads pairs from LDS, and writes each output row's 129 values, 16
// consecutive per lane group. Rows of the padding, and columns outside the
// image, are zeros, as in rfft_rows_kernel.
template <int KIND, bool VEC>
__global__ __launch_bounds__(256) void rfft256_rows_kernel(const void *in, line_set in_rows, int m,
	const float *scales, int64_t scale_stride, float2 *out, line_set out_rows, row_pairs lines, const float2 *tw,
	float half)
{
	constexpr int n = 256;
	constexpr int h = n / 2 + 1;
	__shared__ float2 exchange[fft256_lines * fft256_line_stride];
	__shared__ float2 twl[256];
	__shared__ int64_t row_in[2 * fft256_lines];
	__shared__ int64_t row_out[2 * fft256_lines];
	__shared__ float row_scale[2 * fft256_lines];
	const int t = threadIdx.x;
	const int j = t & 15;
	const int l = t >> 4;
	twl[t] = tw[t];
	const int offset = n / 2 - m / 2;
	const int64_t total = line_count(lines);
	for (int64_t first = xcd_block(blockIdx.x, gridDim.x) * static_cast<int64_t>(fft256_lines); first < total;
		first += static_cast<int64_t>(gridDim.x) * fft256_lines)
	{
		if (t < 2 * fft256_lines)
		{
			const line_row r = row_of(lines, first + t / 2, t & 1);
			row_in[t] = r.in >= 0 ? line_offset(in_rows, r.in) : -1;
			row_out[t] = r.out >= 0 ? line_offset(out_rows, r.out) : -1;
			row_scale[t] = scales != nullptr && r.in >= 0 ? scales[r.transform * scale_stride] : 1.0f;
		}
		__syncthreads();
		float2 *x = exchange + l * fft256_line_stride;
		float2 v[16];
		if constexpr (VEC)
		{
			// Rows whose every run of 4 elements is aligned to 4 elements:
			// each thread loads 4 consecutive elements of a row pair at a
			// time (a wave reads whole rows), and the elements reach their
			// threads through the exchange, element i of line l at
			// (i / 16) 17 + i % 16.
#pragma unroll
			for (int step = 0; step < 4; ++step)
			{
				const int q = step * 256 + t;  // float4 index within the block's 16 lines
				const int ll = q >> 6;         // line
				const int i = (q & 63) * 4;    // first element
				const int c = i - offset;
				const int64_t sa = row_in[2 * ll];
				const int64_t sb = row_in[2 * ll + 1];
				float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
				float4 b = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
				if (c >= 0 && c < m)
				{
					if (sa >= 0)
					{
						const float g = row_scale[2 * ll];
						a = load_real4<KIND>(in, sa + c);
						a = make_float4(a.x * g, a.y * g, a.z * g, a.w * g);
					}
					if (sb >= 0)
					{
						const float g = row_scale[2 * ll + 1];
						b = load_real4<KIND>(in, sb + c);
						b = make_float4(b.x * g, b.y * g, b.z * g, b.w * g);
					}
				}
				float2 *xl = exchange + ll * fft256_line_stride + (i >> 4) * 17 + (i & 15);
				xl[0] = make_float2(a.x, b.x);
				xl[1] = make_float2(a.y, b.y);
				xl[2] = make_float2(a.z, b.z);
				xl[3] = make_float2(a.w, b.w);
			}
			__syncthreads();
#pragma unroll
			for (int k = 0; k < 16; ++k)
			{
				v[k] = x[k * 17 + j];
			}
			__syncthreads();
		}
		else
		{
			const int64_t src_a = row_in[2 * l];
			const int64_t src_b = row_in[2 * l + 1];
			const float scale_a = row_scale[2 * l];
			const float scale_b = row_scale[2 * l + 1];
#pragma unroll
			for (int k = 0; k < 16; ++k)
			{
				const int c = j + 16 * k - offset;
				const bool inside = c >= 0 && c < m;
				const float a =
					src_a >= 0 && inside ? load_real<KIND>(in, src_a + c * in_rows.s_elem) * scale_a : 0.0f;
				const float b =
					src_b >= 0 && inside ? load_real<KIND>(in, src_b + c * in_rows.s_elem) * scale_b : 0.0f;
				v[k] = make_float2(a, b);
			}
		}
		fft256_four_step(v, x, twl, j, -1.0f);
		__syncthreads();
#pragma unroll
		for (int k2 = 0; k2 < 16; ++k2)
		{
			x[k2 * 17 + j] = v[k2]; // Z[j + 16 k2]
		}
		__syncthreads();
		const int64_t dst_a = row_out[2 * l];
		const int64_t dst_b = row_out[2 * l + 1];
#pragma unroll
		for (int q = 0; q < 9; ++q)
		{
			const int k = j + 16 * q;
			if (k < h)
			{
				const int km = (n - k) & (n - 1);
				const float2 zk = x[q * 17 + j];
				const float2 zm = cconj(x[(km >> 4) * 17 + (km & 15)]);
				if (dst_a >= 0)
				{
					const float2 sum = cadd(zk, zm);
					out[dst_a + k * out_rows.s_elem] = make_float2(half * sum.x, half * sum.y);
				}
				if (dst_b >= 0)
				{
					// (zk - zm) / (2 i), times the scale
					const float2 diff = csub(zk, zm);
					out[dst_b + k * out_rows.s_elem] = make_float2(half * diff.y, -half * diff.x);
				}
			}
		}
		__syncthreads();
	}
}

// Half-spectrum rows, two at a time, to real rows, scaled.
__global__ void irfft_rows_kernel(const float2 *src, line_set src_rows, float *dst, line_set dst_rows,
	row_pairs lines, fft_plan plan, const float2 *tw, float scale, int pairs)
{
	extern __shared__ float2 lds[];
	const int n = plan.n;
	const int h = n / 2 + 1;
	const int stride = n + 1;
	float2 *a = lds;
	float2 *b = lds + pairs * stride;
	float2 *twl = lds + 2 * pairs * stride;
	int64_t *row_src = reinterpret_cast<int64_t *>(twl + n);
	int64_t *row_dst = row_src + 2 * pairs;
	for (int i = threadIdx.x; i < n; i += blockDim.x)
	{
		twl[i] = tw[i];
	}
	const int64_t total = line_count(lines);
	for (int64_t first = blockIdx.x * static_cast<int64_t>(pairs); first < total;
		first += static_cast<int64_t>(gridDim.x) * pairs)
	{
		for (int q = threadIdx.x; q < 2 * pairs; q += blockDim.x)
		{
			const line_row r = row_of(lines, first + q / 2, q & 1);
			row_src[q] = r.in >= 0 ? line_offset(src_rows, r.in) : -1;
			row_dst[q] = r.out >= 0 ? line_offset(dst_rows, r.out) : -1;
		}
		__syncthreads();
		for (int t = threadIdx.x; t < pairs * n; t += blockDim.x)
		{
			const int p = t / n;
			const int k = t - p * n;
			const bool mirrored = k >= h;
			const int kk = mirrored ? n - k : k;
			const bool self_conjugate = kk == 0 || (n % 2 == 0 && kk == n / 2);
			float2 va = make_float2(0.0f, 0.0f);
			float2 vb = make_float2(0.0f, 0.0f);
			const int64_t src0 = row_src[2 * p];
			const int64_t src1 = row_src[2 * p + 1];
			if (src0 >= 0)
			{
				va = src[src0 + kk * src_rows.s_elem];
			}
			if (src1 >= 0)
			{
				vb = src[src1 + kk * src_rows.s_elem];
			}
			if (self_conjugate)
			{
				va.y = 0.0f;
				vb.y = 0.0f;
			}
			if (mirrored)
			{
				va = cconj(va);
				vb = cconj(vb);
			}
			// Z = A + i B
			a[p * stride + k] = make_float2(va.x - vb.y, va.y + vb.x);
		}
		__syncthreads();
		const float2 *z = block_fft(a, b, pairs, stride, plan, twl, 1.0f);
		for (int t = threadIdx.x; t < pairs * n; t += blockDim.x)
		{
			const int p = t / n;
			const int i = t - p * n;
			const float2 v = z[p * stride + i];
			const int64_t dst0 = row_dst[2 * p];
			const int64_t dst1 = row_dst[2 * p + 1];
			if (dst0 >= 0)
			{
				dst[dst0 + i * dst_rows.s_elem] = v.x * scale;
			}
			if (dst1 >= 0)
			{
				dst[dst1 + i * dst_rows.s_elem] = v.y * scale;
			}
		}
		__syncthreads();
	}
}

// ---------------------------------------------------------------------------
// Lengths of two register factors (fft_two.hpp).
// ---------------------------------------------------------------------------

// Real rows, two to a complex line, to half spectra, as rfft_rows_kernel: a
// block of (b, lines) threads stages its rows in LDS (a line's threads load
// consecutive elements, 4 at a time where VEC), transforms them and separates
// the two half spectra. Bound by HBM: 1,000 images 320^2 take 0.28 ms against
// 0.52 ms through the Stockham stages (0.8 GB: 4.0 against 1.6 TB/s).
template <int KIND, int WIDTH, int CLASS>
__global__ __launch_bounds__(512, two_factor::waves<CLASS>) void rfft_rows_two_kernel(const void *in, line_set in_rows, int m,
	const float *scales, int64_t scale_stride, float2 *out, line_set out_rows, row_pairs lines, two_factor::plan p,
	const float2 *tw, float half)
{
	extern __shared__ float2 lds[];
	const int j = threadIdx.x;
	const int l = threadIdx.y;
	const int threads = blockDim.x;
	const int n = p.n;
	const int h = n / 2 + 1;
	float2 *twl = lds + p.lines * p.line;
	float2 *x = lds + l * p.line;
	two_factor::stage_twiddles(p, twl, tw, l * threads + j, threads * blockDim.y);
	const int offset = n / 2 - m / 2;
	// One group of lines per block: a loop over groups would hoist the
	// twiddles of every register length out of it, into registers.
	const int64_t first = xcd_block(blockIdx.x, gridDim.x) * static_cast<int64_t>(p.lines);
	if (first >= line_count(lines))
	{
		return;
	}
	// The two rows of the line: first input element (-1: a zero row of the
	// padding or none), first output element, scale.
	int64_t src[2], dst[2];
	float scale[2];
#pragma unroll
	for (int q = 0; q < 2; ++q)
	{
		const line_row r = row_of(lines, first + l, q);
		src[q] = r.in >= 0 ? line_offset(in_rows, r.in) : -1;
		dst[q] = r.out >= 0 ? line_offset(out_rows, r.out) : -1;
		scale[q] = scales != nullptr && r.in >= 0 ? scales[r.transform * scale_stride] : 1.0f;
	}
	// Loads of WIDTH elements, two steps of both rows in flight.
#pragma unroll 2
	for (int i = WIDTH * j; i < n; i += WIDTH * threads)
	{
		const int c = i - offset;
		const bool inside = c >= 0 && c < m;
		float a[WIDTH], b[WIDTH];
		load_reals<KIND, WIDTH>(in, inside && src[0] >= 0, src[0], c, in_rows.s_elem, scale[0], a);
		load_reals<KIND, WIDTH>(in, inside && src[1] >= 0, src[1], c, in_rows.s_elem, scale[1], b);
#pragma unroll
		for (int q = 0; q < WIDTH; ++q)
		{
			x[i + q] = make_float2(a[q], b[q]);
		}
	}
	__syncthreads();
	two_factor::transform_line<CLASS, true, true>(p, x, twl, j, -1.0f, [&](int i) { return x[i]; },
		[&](int k, float2 v) { x[k] = v; });
	__syncthreads();
	for (int k = j; k < h; k += threads)
	{
		const float2 zk = x[k];
		const float2 zm = cconj(x[k == 0 ? 0 : n - k]);
		if (dst[0] >= 0)
		{
			const float2 sum = cadd(zk, zm);
			out[dst[0] + k * out_rows.s_elem] = make_float2(half * sum.x, half * sum.y);
		}
		if (dst[1] >= 0)
		{
			// (zk - zm) / (2 i), times the scale
			const float2 diff = csub(zk, zm);
			out[dst[1] + k * out_rows.s_elem] = make_float2(half * diff.y, -half * diff.x);
		}
	}
}

// Half-spectrum rows, two at a time, to real rows, scaled, as
// irfft_rows_kernel: a coefficient is read once and staged with its mirror.
template <int CLASS>
__global__ __launch_bounds__(512, two_factor::waves<CLASS>) void irfft_rows_two_kernel(const float2 *src, line_set src_rows, float *dst,
	line_set dst_rows, row_pairs lines, two_factor::plan p, const float2 *tw, float scale)
{
	extern __shared__ float2 lds[];
	const int j = threadIdx.x;
	const int l = threadIdx.y;
	const int threads = blockDim.x;
	const int n = p.n;
	const int h = n / 2 + 1;
	float2 *twl = lds + p.lines * p.line;
	float2 *x = lds + l * p.line;
	two_factor::stage_twiddles(p, twl, tw, l * threads + j, threads * blockDim.y);
	const int64_t first = xcd_block(blockIdx.x, gridDim.x) * static_cast<int64_t>(p.lines);
	if (first >= line_count(lines))
	{
		return;
	}
	const line_row row0 = row_of(lines, first + l, 0);
	const line_row row1 = row_of(lines, first + l, 1);
	const int64_t src0 = row0.in >= 0 ? line_offset(src_rows, row0.in) : -1;
	const int64_t src1 = row1.in >= 0 ? line_offset(src_rows, row1.in) : -1;
	const int64_t dst0 = row0.out >= 0 ? line_offset(dst_rows, row0.out) : -1;
	const int64_t dst1 = row1.out >= 0 ? line_offset(dst_rows, row1.out) : -1;
	for (int k = j; k < h; k += threads)
	{
		float2 va = src0 >= 0 ? src[src0 + k * src_rows.s_elem] : make_float2(0.0f, 0.0f);
		float2 vb = src1 >= 0 ? src[src1 + k * src_rows.s_elem] : make_float2(0.0f, 0.0f);
		if (k == 0 || 2 * k == n)
		{
			va.y = 0.0f;
			vb.y = 0.0f;
		}
		else
		{
			// conj A + i conj B at n - k.
			x[n - k] = make_float2(va.x + vb.y, vb.x - va.y);
		}
		x[k] = make_float2(va.x - vb.y, va.y + vb.x); // A + i B
	}
	__syncthreads();
	two_factor::transform_line<CLASS, true, false>(p, x, twl, j, 1.0f, [&](int i) { return x[i]; },
		[&](int i, float2 v)
		{
			if (dst0 >= 0)
			{
				dst[dst0 + i * dst_rows.s_elem] = v.x * scale;
			}
			if (dst1 >= 0)
			{
				dst[dst1 + i * dst_rows.s_elem] = v.y * scale;
			}
		});
}

// Complex lines from `src` to `dst` (may be the same memory). ROWS: the
// elements of a line are consecutive and so are the threads of a line, else
// the lines are neighbours in memory and consecutive threads take consecutive
// lines.
template <bool ROWS, int CLASS>
__global__ __launch_bounds__(512, two_factor::waves<CLASS>) void fft_lines_two_kernel(const float2 *src, line_set src_lines, float2 *dst,
	line_set dst_lines, two_factor::plan p, const float2 *tw, float sign, float scale)
{
	extern __shared__ float2 lds[];
	const int j = ROWS ? threadIdx.x : threadIdx.y;
	const int l = ROWS ? threadIdx.y : threadIdx.x;
	float2 *twl = lds + p.lines * p.line;
	float2 *x = lds + l * p.line;
	two_factor::stage_twiddles(p, twl, tw, threadIdx.y * blockDim.x + threadIdx.x, blockDim.x * blockDim.y);
	__syncthreads();
	const int64_t total = src_lines.count;
	const int64_t first = xcd_block(blockIdx.x, gridDim.x) * static_cast<int64_t>(p.lines);
	if (first >= total)
	{
		return;
	}
	const bool live = first + l < total;
	const float2 *in = src + (live ? line_offset(src_lines, first + l) : 0);
	float2 *out = dst + (live ? line_offset(dst_lines, first + l) : 0);
	two_factor::transform_line<CLASS, false, false>(p, x, twl, j, sign,
		[&](int i) { return live ? in[i * src_lines.s_elem] : make_float2(0.0f, 0.0f); },
		[&](int i, float2 v)
		{
			if (live)
			{
				out[i * dst_lines.s_elem] = make_float2(v.x * scale, v.y * scale);
			}
		});
}

unsigned grid_for(int64_t work, int64_t per_block)
{
	const int64_t blocks = (work + per_block - 1) / per_block;
	return static_cast<unsigned>(std::max<int64_t>(1, std::min<int64_t>(blocks, 1 << 16)));
}

} // anonymous namespace

namespace two_factor
{

plan make_plan(int64_t n)
{
	// Register lengths per class (with_radix).
	static const int small[] = {4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16};
	static const int medium[] = {8, 9, 10, 11, 12, 13, 14, 15, 16, 18, 20, 21, 22};
	static const int large[] = {10, 12, 13, 14, 15, 16, 18, 20, 21, 22, 24, 25, 26, 27, 28, 30, 32};
	plan p{};
	if (n < 48 || n > 1024)
	{
		return p;
	}
	const auto search = [&](const int *set, int count, int kind)
	{
		for (int i = 0; i < count && p.n == 0; ++i)
		{
			for (int k = 0; k <= i; ++k)
			{
				if (set[i] * set[k] == n)
				{
					p.n = static_cast<int32_t>(n);
					p.a = set[k];
					p.b = set[i];
					p.kind = kind;
				}
			}
		}
	};
	search(small, 13, 16);
	search(medium, 13, 22);
	search(large, 17, 32);
	if (p.n != 0)
	{
		p.pitch = p.b | 1;
		p.line = (p.a * p.pitch) | 1;
		// 16 lines read whole 128-byte cache lines of strided operands; past 512
		// points (32 KiB of exchange per 8 lines) 8 keep two blocks on a CU.
		p.lines = n <= 512 ? 16 : 8;
	}
	return p;
}

} // namespace two_factor

int lines_per_group(int n)
{
	// About 2048 complex elements (16 KiB) per LDS buffer: small blocks keep
	// more wavefronts per CU (measured faster than 4096 or 8192 at n = 256).
	return std::max(1, std::min(8, 2048 / std::max(n, 1)));
}

// The path's transforms (rfft2, irfft2, irfft3, the image insertion) take
// lengths with prime factors 2, 3 and 5 and refuse others, as make_fft_plan
// says; the general transforms also use the kernels of any two-factor length.
static void check_length(int64_t n, bool any_length)
{
	if (!(any_length && two_factor::make_plan(n).n != 0))
	{
		make_fft_plan(n);
	}
}

void launch_rfft_rows(int kind, const void *in, const line_set &in_rows, int m, const float *scales,
	int64_t scale_stride, float2 *out, const line_set &out_rows, const row_pairs &pairs, int64_t n, hipStream_t stream,
	bool any_length, float scale)
{
	const int64_t lines = line_count(pairs);
	check_length(n, any_length);
	const float2 *tw = twiddles(n);
	if (n == 256)
	{
		const unsigned blocks = xcd_grid(grid_for(lines, fft256_lines));
		// Rows take loads of 4 elements when every run of 4 elements is
		// aligned and contiguous.
		const std::uintptr_t element = kind == real_f32 ? 4 : 2;
		const bool aligned = in_rows.s_elem == 1 && m % 4 == 0 && (n / 2 - m / 2) % 4 == 0 &&
			in_rows.s_outer % 4 == 0 && (in_rows.middle_count == 1 || in_rows.s_middle % 4 == 0) &&
			(in_rows.inner_count == 1 || in_rows.s_inner % 4 == 0) &&
			reinterpret_cast<std::uintptr_t>(in) % (4 * element) == 0;
		auto launch = [&](auto kind_constant, auto vec_constant)
		{
			rfft256_rows_kernel<decltype(kind_constant)::value, decltype(vec_constant)::value>
				<<<blocks, 256, 0, stream>>>(in, in_rows, m, scales, scale_stride, out, out_rows, pairs, tw, 0.5f * scale);
		};
		using vec = std::true_type;
		using scalar = std::false_type;
		switch (kind)
		{
		case real_f32:
			aligned ? launch(std::integral_constant<int, real_f32>(), vec()) :
				launch(std::integral_constant<int, real_f32>(), scalar());
			break;
		case real_bf16:
			aligned ? launch(std::integral_constant<int, real_bf16>(), vec()) :
				launch(std::integral_constant<int, real_bf16>(), scalar());
			break;
		default:
			aligned ? launch(std::integral_constant<int, real_f16>(), vec()) :
				launch(std::integral_constant<int, real_f16>(), scalar());
			break;
		}
		REXLIB_HIP_CHECK(hipGetLastError());
		return;
	}
	const two_factor::plan two = two_factor::make_plan(n);
	if (two.n != 0)
	{
		const unsigned blocks = two_factor::blocks_for(lines, two.lines);
		// Rows take loads of 4 (or 2) elements when every run of them is
		// aligned and contiguous.
		const std::uintptr_t element = kind == real_f32 ? 4 : 2;
		const auto runs_of = [&](int64_t width)
		{
			return n % width == 0 && in_rows.s_elem == 1 && m % width == 0 && (n / 2 - m / 2) % width == 0 &&
				in_rows.s_outer % width == 0 && (in_rows.middle_count == 1 || in_rows.s_middle % width == 0) &&
				(in_rows.inner_count == 1 || in_rows.s_inner % width == 0) &&
				reinterpret_cast<std::uintptr_t>(in) % (width * element) == 0;
		};
		const int width = runs_of(4) ? 4 : (runs_of(2) ? 2 : 1);
		two_factor::with_class(two, [&](auto kind_class)
			{
				constexpr int CLASS = decltype(kind_class)::value;
				const auto launch = [&](auto kind_constant, auto width_constant)
				{
					rfft_rows_two_kernel<decltype(kind_constant)::value, decltype(width_constant)::value, CLASS>
						<<<blocks, dim3(two.b, two.lines), two_factor::shared_bytes(two), stream>>>(in, in_rows, m, scales,
							scale_stride, out, out_rows, pairs, two, tw, 0.5f * scale);
				};
				const auto with_width = [&](auto kind_constant)
				{
					if (width == 4)
					{
						launch(kind_constant, std::integral_constant<int, 4>());
					}
					else if (width == 2)
					{
						launch(kind_constant, std::integral_constant<int, 2>());
					}
					else
					{
						launch(kind_constant, std::integral_constant<int, 1>());
					}
				};
				switch (kind)
				{
				case real_f32: with_width(std::integral_constant<int, real_f32>()); break;
				case real_bf16: with_width(std::integral_constant<int, real_bf16>()); break;
				default: with_width(std::integral_constant<int, real_f16>()); break;
				}
			});
		REXLIB_HIP_CHECK(hipGetLastError());
		return;
	}
	const fft_plan plan = make_fft_plan(n);
	const int group = std::max(1, lines_per_group(static_cast<int>(n)) / 2);
	// Two buffers, the twiddles, then per row two offsets and a scale.
	const std::size_t shared = sizeof(float2) * (2 * group * (n + 1) + n) + 2 * group * (2 * sizeof(int64_t) + 4);
	const unsigned grid = grid_for(lines, group);
	const auto launch = [&](auto kind_constant)
	{
		rfft_rows_kernel<decltype(kind_constant)::value><<<grid, 256, shared, stream>>>(in, in_rows, m, scales,
			scale_stride, out, out_rows, pairs, plan, tw, group, 0.5f * scale);
	};
	switch (kind)
	{
	case real_f32: launch(std::integral_constant<int, real_f32>()); break;
	case real_bf16: launch(std::integral_constant<int, real_bf16>()); break;
	default: launch(std::integral_constant<int, real_f16>()); break;
	}
	REXLIB_HIP_CHECK(hipGetLastError());
}

void launch_fft_lines(const float2 *src, const line_set &src_lines, float2 *dst, const line_set &dst_lines,
	int64_t n, float sign, float scale, hipStream_t stream, bool any_length)
{
	check_length(n, any_length);
	const float2 *tw = twiddles(n);
	const bool rows = src_lines.s_elem == 1 && dst_lines.s_elem == 1;
	const two_factor::plan two = two_factor::make_plan(n);
	if (two.n != 0)
	{
		const unsigned blocks = two_factor::blocks_for(src_lines.count, two.lines);
		two_factor::with_class(two, [&](auto kind_class)
			{
				constexpr int CLASS = decltype(kind_class)::value;
				if (rows)
				{
					fft_lines_two_kernel<true, CLASS><<<blocks, dim3(two.b, two.lines), two_factor::shared_bytes(two),
						stream>>>(src, src_lines, dst, dst_lines, two, tw, sign, scale);
				}
				else
				{
					fft_lines_two_kernel<false, CLASS><<<blocks, dim3(two.lines, two.b), two_factor::shared_bytes(two),
						stream>>>(src, src_lines, dst, dst_lines, two, tw, sign, scale);
				}
			});
		REXLIB_HIP_CHECK(hipGetLastError());
		return;
	}
	const fft_plan plan = make_fft_plan(n);
	const int group = lines_per_group(static_cast<int>(n));
	const std::size_t shared = sizeof(float2) * (2 * group * (n + 1) + n) + 2 * group * sizeof(int64_t);
	const unsigned grid = grid_for(src_lines.count, group);
	fft_lines_kernel<<<grid, 256, shared, stream>>>(src, src_lines, dst, dst_lines, plan, tw, sign, scale, group);
	REXLIB_HIP_CHECK(hipGetLastError());
}

void launch_irfft_rows(const float2 *src, const line_set &src_rows, float *dst, const line_set &dst_rows,
	const row_pairs &pairs, int64_t n, float scale, hipStream_t stream, bool any_length)
{
	check_length(n, any_length);
	const float2 *tw = twiddles(n);
	const two_factor::plan two = two_factor::make_plan(n);
	if (two.n != 0)
	{
		const unsigned blocks = two_factor::blocks_for(line_count(pairs), two.lines);
		two_factor::with_class(two, [&](auto kind_class)
			{
				irfft_rows_two_kernel<decltype(kind_class)::value><<<blocks, dim3(two.b, two.lines),
					two_factor::shared_bytes(two), stream>>>(src, src_rows, dst, dst_rows, pairs, two, tw, scale);
			});
		REXLIB_HIP_CHECK(hipGetLastError());
		return;
	}
	const fft_plan plan = make_fft_plan(n);
	const int group = std::max(1, lines_per_group(static_cast<int>(n)) / 2);
	const std::size_t shared = sizeof(float2) * (2 * group * (n + 1) + n) + 2 * group * 2 * sizeof(int64_t);
	const unsigned grid = grid_for(line_count(pairs), group);
	irfft_rows_kernel<<<grid, 256, shared, stream>>>(src, src_rows, dst, dst_rows, pairs, plan, tw, scale, group);
	REXLIB_HIP_CHECK(hipGetLastError());
}

} // namespace rexlib_hip
