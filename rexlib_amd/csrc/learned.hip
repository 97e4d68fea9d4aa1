// Density compensation of the accumulators: the iterative estimate and a
// small learned predictor of it.
//
// The reference has no density compensation (its reconstruction divides the
// numerator by the denominator, tests/integration/src/em/functional/test_cpu_reconstruction.cpp:457-464).
// Here the compensation is a weight W per voxel of the half spectrum that
// flattens the gridded sampling density:
//   - iterative (the reference estimate and the fallback): starting from
//     W = 1, each pass convolves W * den with K3 = t x t x t, t = (1/6, 2/3,
//     1/6) -- the autocorrelation of the trilinear window at integer lags --
//     and divides: W <- W / max(K3 * (W den), eps);
//   - learned: a multilayer perceptron 10 -> 64 -> 64 -> 64 -> 1 (ReLU)
//     maps per-voxel features to log W. Its weights are float16 and its
//     products run on v_mfma_f32_16x16x16_f16 with float32 accumulation, in
//     the forward pass and in the backward pass that trains it.
//
// Features of a voxel g: |g| / (N/2); log(1 + den(g) * scale); and the 8
// coverage fractions of its radius and direction (below).
//
// The half spectrum is Hermitian: the full-spectrum element (x, y, z) with x
// beyond the stored half is the element (N - x, -y, -z), and a real field
// such as den takes the same value there.
#include "common.hpp"

#include <hip/hip_fp16.h>

#include <cmath>

namespace rexlib_hip
{

namespace
{

// Threads over a (ceil(N half / blockDim), N) grid: (x, y) of plane z.
__device__ inline bool voxel_of_thread(int big, int half, int &x, int &y, int &z)
{
	const int xy = blockIdx.x * blockDim.x + threadIdx.x;
	if (xy >= big * half)
	{
		return false;
	}
	y = xy / half;
	x = xy - y * half;
	z = blockIdx.y;
	return true;
}

// One pass of the iteration, on P = W den: P <- P / max(K3 * P, floor) where
// den > 0, else 0. It starts from P = den (W = 1), and the last pass divides by
// den; the passes between touch P alone. A block takes a tile of `width` x
// height voxels (x, y), an even share of the row, and walks
// `planes` planes along z: a plane goes to LDS with its halo of
// one, is convolved there along x and y, and the three z taps come from
// registers, so a voxel is loaded once per pass and tile (1.4 times with the
// halo). 27 gathers of W and den per voxel took 166 us a pass at 256^3; this
// takes 31 us (68 MB of P read and written), bound by the latency of a plane's
// loads and barrier.
constexpr int compensation_planes = 16; // at most
// Small volumes walk fewer planes per block, until this many blocks run (each
// plane waits for its loads and a barrier): ten passes at 33^3 take 39 us so, 94
// with 16 planes, at 64^3 42 against 95; from 180^3 on 16 fill the chip.
constexpr int compensation_blocks = 512;
constexpr int compensation_width = 40; // at most

template <bool FIRST, bool LAST>
__global__ __launch_bounds__(256) void compensation_pass_kernel(const float *den, const float *p_in, float *out,
	int big, int width, int height, int planes, float floor_value)
{
	// A plane of the tile with its halo, at most two elements per thread.
	__shared__ float product[2][512];
	const int half = big / 2 + 1;
	const int t = threadIdx.x;
	const int ty = t / width;
	const int tx = t - ty * width;
	const int x0 = blockIdx.x * width;
	const int y0 = blockIdx.y * height;
	const int z0 = blockIdx.z * planes;
	const int z1 = min(z0 + planes, big);
	const int x = x0 + tx;
	const int y = y0 + ty;
	const bool live = ty < height && x < half && y < big;
	const int pitch = width + 2;
	const int halo = pitch * (height + 2);
	// This thread's two elements of the tile with the halo. The frequencies
	// past the stored half mirror (x, y, z): the y index is fixed per thread,
	// and the z index flips with it.
	bool held[2];
	bool mirrored[2];
	int64_t offset[2];
#pragma unroll
	for (int k = 0; k < 2; ++k)
	{
		const int q = t + 256 * k;
		const int hy_tile = q / pitch;
		const int hx = x0 + (q - hy_tile * pitch) - 1;
		const int hy = y0 + hy_tile - 1;
		// Tiles that reach past the volume's end need one column and row more.
		held[k] = q < halo && hx <= half && hy <= big;
		const int xw = hx < 0 ? hx + big : hx;
		const int yw = hy < 0 ? hy + big : (hy >= big ? hy - big : hy);
		mirrored[k] = xw >= half;
		const int xs = mirrored[k] ? big - xw : xw;
		const int ys = mirrored[k] && yw != 0 ? big - yw : yw;
		offset[k] = static_cast<int64_t>(ys) * half + xs;
	}
	const int64_t plane_size = static_cast<int64_t>(big) * half;
	float staged[2] = {0.0f, 0.0f};
	const auto load = [&](int z)
	{
		const int zw = z < 0 ? z + big : (z >= big ? z - big : z);
		const int zm = zw == 0 ? 0 : big - zw;
#pragma unroll
		for (int k = 0; k < 2; ++k)
		{
			if (held[k])
			{
				staged[k] = p_in[(mirrored[k] ? zm : zw) * plane_size + offset[k]];
			}
		}
	};
	const float side = 1.0f / 6.0f, middle = 2.0f / 3.0f;
	float below = 0.0f, here = 0.0f, p_here = 0.0f;
	load(z0 - 1);
	for (int z = z0 - 1; z <= z1; ++z)
	{
		float *plane = product[z & 1];
		plane[t] = staged[0];
		plane[t + 256] = staged[1];
		if (z < z1)
		{
			load(z + 1);
		}
		const int64_t i = (z - 1) * plane_size + static_cast<int64_t>(y) * half + x;
		float d = 1.0f;
		if (LAST && z > z0 && live)
		{
			d = den[i];
		}
		__syncthreads();
		float sum = 0.0f;
		float p = 0.0f;
		if (live)
		{
			const float *row = plane + ty * pitch + tx;
#pragma unroll
			for (int dy = 0; dy < 3; ++dy)
			{
				sum += (dy == 1 ? middle : side) * (middle * row[1] + side * (row[0] + row[2]));
				p = dy == 1 ? row[1] : p;
				row += pitch;
			}
		}
		// `sum` is plane z convolved along x and y; plane z - 1 is complete.
		if (z > z0 && live)
		{
			const float c = middle * here + side * (below + sum);
			const float next = (FIRST ? p_here > 0.0f : true) ? p_here / fmaxf(c, floor_value) : 0.0f;
			out[i] = LAST ? (d > 0.0f ? next / d : 0.0f) : next;
		}
		below = here;
		here = sum;
		p_here = p;
	}
}

__global__ void fill_kernel(float *out, int64_t count, float value)
{
	for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < count;
		i += static_cast<int64_t>(gridDim.x) * blockDim.x)
	{
		out[i] = value;
	}
}

// Angular coverage of the slice normals: for radius bin r (of the 8
// spanning |g| in [0, N/2]) and direction u on a 33 x 64 (theta, phi) grid
// (theta = k pi / 32 from pole to pole, phi = k 2 pi / 64: the axes and the
// coordinate planes of the lattice fall on grid directions, so a voxel's
// nearest direction is never a tie between two),
// the fractions of the slices whose plane passes within one voxel of the
// point at that radius and direction, widened by half the grid's spacing
// (|n . u| < 1 / radius + 0.05, so that no plane slips between directions), that fall in
// each of 8 bins of the normal's angle around u, taken modulo pi (n and -n
// are one plane), measured from the local frame e1 = d u / d theta,
// e2 = d u / d phi. All zeros where no plane passes.
constexpr int coverage_radii = 8;
constexpr int coverage_theta = 33;
constexpr int coverage_phi = 64;
constexpr int coverage_bins = 8;
constexpr int coverage_tile = 256;

__device__ inline float3 coverage_direction(int it, int ip, float3 &e1, float3 &e2)
{
	const float theta = static_cast<float>(it) * (3.14159265358979f / (coverage_theta - 1));
	const float phi = static_cast<float>(ip) * (6.28318530717959f / coverage_phi);
	float st, ct, sp, cp;
	sincosf(theta, &st, &ct);
	sincosf(phi, &sp, &cp);
	e1 = make_float3(ct * cp, ct * sp, -st);
	e2 = make_float3(-sp, cp, 0.0f);
	return make_float3(st * cp, st * sp, ct);
}

// One thread per table entry and one slice range per blockIdx.y; the
// workgroup stages the unit normals of 256 slices at a time in LDS. The
// counts of the range are added to `counts` (the table's own memory, as
// uint32, zeroed first) with integer atomics, so the result does not depend
// on the order of the ranges.
__global__ __launch_bounds__(256) void coverage_count_kernel(const float *transforms, int64_t slices, int64_t ts0,
	int64_t ts1, int64_t ts2, int big, int64_t per_block, unsigned *counts)
{
	__shared__ float3 normals[coverage_tile];
	const int entry = blockIdx.x * blockDim.x + threadIdx.x;
	constexpr int entries = coverage_radii * coverage_theta * coverage_phi;
	const bool live = entry < entries;
	const int r = entry / (coverage_theta * coverage_phi);
	const int rest = entry - r * coverage_theta * coverage_phi;
	const int it = rest / coverage_phi;
	const int ip = rest - it * coverage_phi;
	float3 e1, e2;
	const float3 u = coverage_direction(it, ip, e1, e2);
	const float radius = (static_cast<float>(r) + 0.5f) / coverage_radii * (0.5f * static_cast<float>(big));
	const float band = fminf(1.0f, 1.0f / radius + 0.05f);
	unsigned count[coverage_bins];
	for (int b = 0; b < coverage_bins; ++b)
	{
		count[b] = 0;
	}
	const int64_t begin = blockIdx.y * per_block;
	const int64_t end = min<int64_t>(slices, begin + per_block);
	for (int64_t first = begin; first < end; first += coverage_tile)
	{
		const int64_t j = first + threadIdx.x;
		float3 n = make_float3(0.0f, 0.0f, 0.0f);
		if (j < end)
		{
			const float *t = transforms + j * ts0;
			const float x0 = t[0], x1 = t[ts2], x2 = t[2 * ts2];
			const float y0 = t[ts1], y1 = t[ts1 + ts2], y2 = t[ts1 + 2 * ts2];
			n = make_float3(x1 * y2 - x2 * y1, x2 * y0 - x0 * y2, x0 * y1 - x1 * y0);
			const float length = sqrtf(n.x * n.x + n.y * n.y + n.z * n.z);
			const float inv = length > 0.0f ? 1.0f / length : 0.0f;
			n = make_float3(n.x * inv, n.y * inv, n.z * inv);
		}
		__syncthreads();
		normals[threadIdx.x] = n;
		__syncthreads();
		const int tile = static_cast<int>(min<int64_t>(coverage_tile, end - first));
		for (int k = 0; k < tile; ++k)
		{
			const float3 m = normals[k];
			const float along = m.x * u.x + m.y * u.y + m.z * u.z;
			const float a1 = m.x * e1.x + m.y * e1.y + m.z * e1.z;
			const float a2 = m.x * e2.x + m.y * e2.y + m.z * e2.z;
			if (fabsf(along) < band && (a1 != 0.0f || a2 != 0.0f))
			{
				// The angle modulo pi, in [0, pi).
				float angle = atan2f(a2, a1);
				angle = angle < 0.0f ? angle + 3.14159265358979f : angle;
				angle = angle >= 3.14159265358979f ? angle - 3.14159265358979f : angle;
				const int bin = min(coverage_bins - 1, static_cast<int>(angle * (coverage_bins / 3.14159265358979f)));
				for (int b = 0; b < coverage_bins; ++b)
				{
					count[b] += bin == b ? 1u : 0u;
				}
			}
		}
	}
	if (live)
	{
		for (int b = 0; b < coverage_bins; ++b)
		{
			if (count[b] != 0)
			{
				atomicAdd(counts + static_cast<int64_t>(entry) * coverage_bins + b, count[b]);
			}
		}
	}
}

// In place: the uint32 counts of each entry become the fractions of their
// total (zeros when no plane passes).
__global__ __launch_bounds__(256) void coverage_normalize_kernel(float *table)
{
	const int entry = blockIdx.x * blockDim.x + threadIdx.x;
	if (entry >= coverage_radii * coverage_theta * coverage_phi)
	{
		return;
	}
	const unsigned *counts = reinterpret_cast<const unsigned *>(table) + static_cast<int64_t>(entry) * coverage_bins;
	unsigned c[coverage_bins];
	unsigned total = 0;
	for (int b = 0; b < coverage_bins; ++b)
	{
		c[b] = counts[b];
		total += c[b];
	}
	const float scale = total > 0 ? 1.0f / static_cast<float>(total) : 0.0f;
	for (int b = 0; b < coverage_bins; ++b)
	{
		table[static_cast<int64_t>(entry) * coverage_bins + b] = static_cast<float>(c[b]) * scale;
	}
}

// What the features of voxel (x, sy, sz) need: the shell radius |g| / (N/2),
// log(1 + den * density_scale) (the local sample count against the mean of the
// positive weights) and the coverage table's entry nearest to the voxel's
// radius and direction.
struct voxel_features
{
	float radius;
	float density;
	int entry;
};

__device__ inline voxel_features features_of(float den, float density_scale, int x, int sy, int sz, int big)
{
	// Signed frequencies as numpy's fftfreq: index N/2 is -N/2 of an even N, +N/2
	// of an odd one.
	const int y = sy < (big + 1) / 2 ? sy : sy - big;
	const int z = sz < (big + 1) / 2 ? sz : sz - big;
	// log(1 + v) by the hardware logarithm, corrected for the rounding of
	// 1 + v: with u = fl(1 + v), log(u) v / (u - 1) keeps the relative error
	// near one ulp for small v as well (u = 1 gives v itself).
	auto log1 = [](float v)
	{
		const float u = 1.0f + v;
		return u == 1.0f ? v : __logf(u) * (v / (u - 1.0f));
	};
	const float length = sqrtf(static_cast<float>(x * x + y * y + z * z));
	voxel_features f;
	f.radius = length / (0.5f * static_cast<float>(big));
	f.density = log1(fmaxf(den, 0.0f) * density_scale);
	const int r = min(coverage_radii - 1, static_cast<int>(f.radius * coverage_radii));
	const float theta = length > 0.0f ? acosf(fminf(1.0f, fmaxf(-1.0f, static_cast<float>(z) / length))) : 0.0f;
	float phi = atan2f(static_cast<float>(y), static_cast<float>(x));
	phi = phi < 0.0f ? phi + 6.28318530717959f : phi;
	// The nearest grid direction (phi wraps around).
	const int it = min(coverage_theta - 1, static_cast<int>(theta * ((coverage_theta - 1) / 3.14159265358979f) + 0.5f));
	const int ip = static_cast<int>(phi * (coverage_phi / 6.28318530717959f) + 0.5f) % coverage_phi;
	f.entry = (r * coverage_theta + it) * coverage_phi + ip;
	return f;
}

// Features of every voxel, as 16 float16 per voxel (the last 6 zero):
// radius, density and the 8 coverage fractions. The 32 bytes are stored as two
// 16-byte words.
__global__ __launch_bounds__(256) void features_kernel(const float *den, const float *table, float density_scale,
	__half *features, int big)
{
	const int half = big / 2 + 1;
	int x, sy, sz;
	if (!voxel_of_thread(big, half, x, sy, sz))
	{
		return;
	}
	const int64_t i = (static_cast<int64_t>(sz) * big + sy) * half + x;
	const voxel_features v = features_of(den[i], density_scale, x, sy, sz, big);
	float f[16];
	f[0] = v.radius;
	f[1] = v.density;
	const float *entry = table + static_cast<int64_t>(v.entry) * coverage_bins;
	for (int b = 0; b < coverage_bins; ++b)
	{
		f[2 + b] = entry[b];
	}
	for (int k = 10; k < 16; ++k)
	{
		f[k] = 0.0f;
	}
	unsigned packed[8];
	for (int k = 0; k < 8; ++k)
	{
		packed[k] = static_cast<unsigned>(__half_as_ushort(__float2half(f[2 * k]))) |
			(static_cast<unsigned>(__half_as_ushort(__float2half(f[2 * k + 1]))) << 16);
	}
	uint4 *out = reinterpret_cast<uint4 *>(features + i * 16);
	out[0] = make_uint4(packed[0], packed[1], packed[2], packed[3]);
	out[1] = make_uint4(packed[4], packed[5], packed[6], packed[7]);
}

// ---------------------------------------------------------------------------
// The perceptron on MFMA
// ---------------------------------------------------------------------------

// Each wavefront works on its own tile; LDS operations of one wavefront
// retire in order, so only the compiler must be kept from moving LDS
// accesses across these points (no workgroup barrier: the wavefronts of a
// workgroup run different numbers of tiles).
__device__ inline void wave_order()
{
	__asm__ __volatile__("" ::: "memory");
}

typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

constexpr int hidden = 64;
constexpr int inputs = 16; // 10 features, padded

// Parameter layout (float16 copy and float32 master share it), row-major
// W[k][n]: W1 16x64, W2 64x64, W3 64x64, W4 64x16 (column 0 used), then the
// biases b1, b2, b3 (64 each) and b4 (16, element 0 used).
constexpr int off_w1 = 0;
constexpr int off_w2 = off_w1 + inputs * hidden;
constexpr int off_w3 = off_w2 + hidden * hidden;
constexpr int off_w4 = off_w3 + hidden * hidden;
constexpr int off_b1 = off_w4 + hidden * 16;
constexpr int off_b2 = off_b1 + hidden;
constexpr int off_b3 = off_b2 + hidden;
constexpr int off_b4 = off_b3 + hidden;
constexpr int parameter_count = off_b4 + 16;

// D (16x16, float) += A (16x16, fp16) B (16x16, fp16) on one wavefront. Lane
// l holds A[l % 16][4 (l / 16) + j], B[4 (l / 16) + j][l % 16] and
// D[4 (l / 16) + j][l % 16], j = 0..3.
__device__ inline float4_t mfma16(half4_t a, half4_t b, float4_t c)
{
	return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0);
}

// D (16x16, float) += A (16x32, fp16) B (32x16, fp16), gfx950's double-depth
// form: twice the products of mfma16 per instruction. Lane l holds eight
// values of A's row l % 16 and eight of B's column l % 16, the same eight
// depth positions in both; D is laid out as for mfma16.
__device__ inline float4_t mfma32(half8_t a, half8_t b, float4_t c)
{
	return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// Two half4 fragments as one half8.
__device__ inline half8_t join(half4_t lo, half4_t hi)
{
	return half8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

// The perceptron in transposed form: each layer computes Y^T = W^T X^T on a
// tile of 16 samples, the 16 columns of the B operand. The weights are the A
// operands and stay in registers for the whole kernel. An MFMA's output
// fragment (lane l: rows 4 (l / 16) + j, column l % 16) is laid out as a B
// operand, so after ReLU and the float16 rounding the activations never leave
// registers.
// - The first layer (depth 16) takes mfma16: lane l of A holds
//   W^T[m0 + l % 16][4 (l / 16) + j] = W[4 (l / 16) + j][m0 + l % 16].
// - The depth-64 layers take mfma32 over two chunks of 32 hidden units. A
//   sum is the same in any order of its terms, so chunk t gives lane group
//   g = l / 16 the units 32 t + 4 g + j (j < 4) and 32 t + 16 + 4 g + j - 4
//   (j >= 4): its B operand is the two output fragments of m-tiles 2t and
//   2t + 1 side by side, and its A operand holds the weights of the same
//   units.
// The bias is the accumulator a layer starts from, and ReLU runs on pairs of
// rounded values (max and rounding commute), so that the vector work between
// layers is one conversion and one maximum per pair; adding the bias and
// clamping in float32 took three instructions per value and bound the kernel
// (0.31 ms for the voxels of 256^3; with two tiles in flight 0.22 ms, the
// features included).
struct mlp_weights
{
	half4_t w1[4];
	half8_t w2[4][2];
	half8_t w3[4][2];
	half8_t w4[2];
	float b4;
};

// Biases per (layer, m-tile, lane group): the 4 rows a lane's output holds.
typedef float4_t mlp_biases[3][4][4];

// The float16 weights pass through LDS, 16 bytes a lane: straight from memory
// the fragments are 160 scattered 2-byte loads per lane.
__device__ inline void load_mlp(const _Float16 *weights, const float *params_f, mlp_weights &m, mlp_biases &bias)
{
	static_assert(off_b1 % 8 == 0, "whole 16-byte words");
	__shared__ uint4 staged[off_b1 / 8];
	const bool aligned = reinterpret_cast<uintptr_t>(weights) % 16 == 0;
	for (int i = threadIdx.x; i < off_b1 / 8; i += blockDim.x)
	{
		if (aligned)
		{
			staged[i] = reinterpret_cast<const uint4 *>(weights)[i];
		}
		else
		{
			for (int k = 0; k < 8; ++k)
			{
				reinterpret_cast<_Float16 *>(staged)[8 * i + k] = weights[8 * i + k];
			}
		}
	}
	const _Float16 *params_h = reinterpret_cast<const _Float16 *>(staged);
	if (threadIdx.x < 48)
	{
		const int layer = threadIdx.x / 16;
		const int mt = (threadIdx.x / 4) % 4;
		const int g = threadIdx.x % 4;
		const float *b = params_f + off_b1 + layer * hidden + mt * 16 + 4 * g;
		bias[layer][mt][g] = float4_t{b[0], b[1], b[2], b[3]};
	}
	__syncthreads();
	const int lane = threadIdx.x & 63;
	const int g = lane >> 4;
	const int c = lane & 15;
#pragma unroll
	for (int j = 0; j < 4; ++j)
	{
#pragma unroll
		for (int mt = 0; mt < 4; ++mt)
		{
			m.w1[mt][j] = params_h[off_w1 + (4 * g + j) * hidden + mt * 16 + c];
		}
	}
#pragma unroll
	for (int j = 0; j < 8; ++j)
	{
#pragma unroll
		for (int t = 0; t < 2; ++t)
		{
			// Hidden unit of depth position (g, j) in chunk t.
			const int unit = 32 * t + (j < 4 ? 4 * g + j : 16 + 4 * g + j - 4);
#pragma unroll
			for (int mt = 0; mt < 4; ++mt)
			{
				m.w2[mt][t][j] = params_h[off_w2 + unit * hidden + mt * 16 + c];
				m.w3[mt][t][j] = params_h[off_w3 + unit * hidden + mt * 16 + c];
			}
			m.w4[t][j] = params_h[off_w4 + unit * 16 + c];
		}
	}
	m.b4 = params_f[off_b4];
}

// Rounds to float16 and clamps at 0.
__device__ inline half4_t relu_half(float4_t v)
{
	typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
	const half2_t zero = {0, 0};
	const half2_t lo = __builtin_elementwise_max(
		half2_t{static_cast<_Float16>(v[0]), static_cast<_Float16>(v[1])}, zero);
	const half2_t hi = __builtin_elementwise_max(
		half2_t{static_cast<_Float16>(v[2]), static_cast<_Float16>(v[3])}, zero);
	return half4_t{lo[0], lo[1], hi[0], hi[1]};
}

// The perceptron on TILES tiles at once (independent chains of MFMAs, so that
// one tile's fill the gaps of another's): lane (g, c) brings features 4 g ..
// 4 g + 3 of sample c of each; the output of sample c is in lane c (group 0).
template <int TILES>
__device__ __forceinline__ void mlp_tiles(const mlp_weights &m, const mlp_biases &bias, int g, const half4_t *x, float *y)
{
	half4_t h1[TILES][4];
	half4_t h2[TILES][4];
#pragma unroll
	for (int mt = 0; mt < 4; ++mt)
	{
#pragma unroll
		for (int i = 0; i < TILES; ++i)
		{
			h1[i][mt] = relu_half(mfma16(m.w1[mt], x[i], bias[0][mt][g]));
		}
	}
	const auto layer = [&](const half8_t (&w)[4][2], int number, const half4_t (*in)[4], half4_t (*out)[4])
	{
#pragma unroll
		for (int mt = 0; mt < 4; ++mt)
		{
			float4_t acc[TILES];
#pragma unroll
			for (int i = 0; i < TILES; ++i)
			{
				acc[i] = bias[number][mt][g];
			}
#pragma unroll
			for (int t = 0; t < 2; ++t)
			{
#pragma unroll
				for (int i = 0; i < TILES; ++i)
				{
					acc[i] = mfma32(w[mt][t], join(in[i][2 * t], in[i][2 * t + 1]), acc[i]);
				}
			}
#pragma unroll
			for (int i = 0; i < TILES; ++i)
			{
				out[i][mt] = relu_half(acc[i]);
			}
		}
	};
	layer(m.w2, 1, h1, h2);
	layer(m.w3, 2, h2, h1);
#pragma unroll
	for (int i = 0; i < TILES; ++i)
	{
		float4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
		for (int t = 0; t < 2; ++t)
		{
			acc = mfma32(m.w4[t], join(h1[i][2 * t], h1[i][2 * t + 1]), acc);
		}
		// Output row 0 (the one used column of W4) sits in lanes 0..15.
		y[i] = acc[0] + m.b4;
	}
}

// out[i] = MLP(features[i]) for i < count.
__global__ __launch_bounds__(256, 2) void mlp_forward_kernel(const __half *features, const _Float16 *params_h,
	const float *params_f, float *out, int64_t count)
{
	__shared__ mlp_biases bias;
	mlp_weights m;
	load_mlp(params_h, params_f, m, bias);
	const int lane = threadIdx.x & 63;
	const int g = lane >> 4;
	const int c = lane & 15;
	const int64_t pairs = (count + 31) / 32;
	const int64_t waves = static_cast<int64_t>(gridDim.x) * (blockDim.x / 64);
	for (int64_t pair = static_cast<int64_t>(blockIdx.x) * (blockDim.x / 64) + (threadIdx.x >> 6); pair < pairs;
		pair += waves)
	{
		const int64_t row = pair * 32 + c;
		// B fragment of X^T: B[4 g + j][c] = X[row][4 g + j], 8 bytes per lane.
		half4_t x[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
		for (int i = 0; i < 2; ++i)
		{
			if (row + 16 * i < count)
			{
				x[i] = *reinterpret_cast<const half4_t *>(features + (row + 16 * i) * inputs + 4 * g);
			}
		}
		float y[2];
		mlp_tiles<2>(m, bias, g, x, y);
#pragma unroll
		for (int i = 0; i < 2; ++i)
		{
			if (g == 0 && row + 16 * i < count)
			{
				out[row + 16 * i] = y[i];
			}
		}
	}
}

// |g| <= N/2 as learned.inside_nyquist has it, to the last bit: fftfreq scales by
// 1 / (N (1 / N)) in double, which is not 1 for N = 98, 196, 206, 214, ..., and
// there the rounding of the separate products and sums decides the voxels at
// exactly N/2 (a fused one decides some of N = 214 the other way).
__device__ inline bool inside_nyquist(int x, int y, int z, int big, double frequency_scale)
{
#pragma clang fp contract(off)
	const double fy = y * frequency_scale;
	const double fz = z * frequency_scale;
	const double zz = fz * fz;
	const double yy = fy * fy;
	const double xx = static_cast<double>(x) * x;
	return zz + yy + xx <= static_cast<double>(big / 2) * (big / 2);
}

// The predicted weights of a volume in one pass: W = exp(MLP(features)) / den
// where den > 0 within the Nyquist sphere, 1 / den beyond it, 0 elsewhere. A
// lane computes the radius, density and table entry of one of 64 voxels of a
// plane; four tiles of 16 voxels then take theirs by shuffles, the coverage
// fractions from the table, and hand the outputs back. The features (270 MB at
// 256^3), the correction and the masks never reach memory.
__global__ __launch_bounds__(256, 2) void predicted_weights_kernel(const float *den, const float *table,
	float density_scale, const _Float16 *params_h, const float *params_f, float *out, int big,
	double frequency_scale)
{
	__shared__ mlp_biases bias;
	mlp_weights m;
	load_mlp(params_h, params_f, m, bias);
	const int lane = threadIdx.x & 63;
	const int g = lane >> 4;
	const int c = lane & 15;
	const int half = big / 2 + 1;
	const int plane = big * half;
	const int groups = (plane + 63) / 64; // of 64 voxels per plane
	const int waves = gridDim.x * (blockDim.x / 64);
	// (Plane, group) of this wavefront, stepped without a division.
	const int first = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6));
	const int step_planes = waves / groups;
	const int step_groups = waves - step_planes * groups;
	int sz = first / groups;
	int group = first - sz * groups;
	for (; sz < big; sz += step_planes + (group + step_groups >= groups ? 1 : 0),
		group += group + step_groups >= groups ? step_groups - groups : step_groups)
	{
		const int xy = group * 64 + lane;
		const bool live = xy < plane;
		const int sy = live ? xy / half : 0;
		const int x = live ? xy - sy * half : 0;
		const int64_t i = static_cast<int64_t>(sz) * plane + (live ? xy : 0);
		const float d = den[i];
		const voxel_features f = features_of(d, density_scale, x, sy, sz, big);
		const half4_t own = {static_cast<_Float16>(f.radius), static_cast<_Float16>(f.density), 0, 0};
		const int packed = __builtin_bit_cast(int2, own).x;
		// Features 4 g .. 4 g + 3 of tile t's voxel c: (radius, density, bins 0,
		// 1), (bins 2 .. 5), (bins 6, 7, 0, 0), zeros. Every lane loads, so the
		// loads of the four tiles are in flight together. (The table may lie at
		// any multiple of 4 bytes.)
		struct __attribute__((packed, aligned(4))) bin_pair
		{
			float x, y;
		};
		const bin_pair *pairs = reinterpret_cast<const bin_pair *>(table);
		const int low = g == 0 ? 0 : (g == 1 ? 1 : 3);
		bin_pair bins[4][2];
		int head[4];
#pragma unroll
		for (int t = 0; t < 4; ++t)
		{
			const int entry = __shfl(f.entry, 16 * t + c, 64) * (coverage_bins / 2);
			head[t] = __shfl(packed, 16 * t + c, 64);
			bins[t][0] = pairs[entry + low];
			bins[t][1] = pairs[entry + 2];
		}
		half4_t v[4];
#pragma unroll
		for (int t = 0; t < 4; ++t)
		{
			typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
			const int first = __builtin_bit_cast(int,
				half2_t{static_cast<_Float16>(bins[t][0].x), static_cast<_Float16>(bins[t][0].y)});
			const int second = __builtin_bit_cast(int,
				half2_t{static_cast<_Float16>(bins[t][1].x), static_cast<_Float16>(bins[t][1].y)});
			const int a = g == 0 ? head[t] : (g == 3 ? 0 : first);
			const int b = g == 0 ? first : (g == 1 ? second : 0);
			v[t] = __builtin_bit_cast(half4_t, make_int2(a, b));
		}
		float y4[4];
		mlp_tiles<2>(m, bias, g, v, y4);
		mlp_tiles<2>(m, bias, g, v + 2, y4 + 2);
		float correction = 0.0f;
#pragma unroll
		for (int t = 0; t < 4; ++t)
		{
			const float mine = __shfl(y4[t], c, 64);
			correction = g == t ? mine : correction;
		}
		if (live)
		{
			// numpy's fftfreq (of an odd N, index N/2 is +N/2).
			const int y = sy < (big + 1) / 2 ? sy : sy - big;
			const int z = sz < (big + 1) / 2 ? sz : sz - big;
			const bool inside = inside_nyquist(x, y, z, big, frequency_scale);
			out[i] = d > 0.0f ? (inside ? expf(correction) : 1.0f) / d : 0.0f;
		}
	}
}

// Sum and number of the positive weights, one pair per block in double, then
// scale = 1 / mean (1 without any).
constexpr int density_blocks = 1024;

__global__ __launch_bounds__(256) void density_sums_kernel(const float *den, int64_t count, double *partial)
{
	__shared__ double sums[2][4];
	double sum = 0.0, positive = 0.0;
	for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < count; i += gridDim.x * 256ll)
	{
		const float d = den[i];
		sum += d > 0.0f ? static_cast<double>(d) : 0.0;
		positive += d > 0.0f ? 1.0 : 0.0;
	}
	for (int offset = 32; offset > 0; offset /= 2)
	{
		sum += __shfl_down(sum, offset, 64);
		positive += __shfl_down(positive, offset, 64);
	}
	if ((threadIdx.x & 63) == 0)
	{
		sums[0][threadIdx.x >> 6] = sum;
		sums[1][threadIdx.x >> 6] = positive;
	}
	__syncthreads();
	if (threadIdx.x < 2)
	{
		const double *s = sums[threadIdx.x];
		partial[2 * blockIdx.x + threadIdx.x] = s[0] + s[1] + s[2] + s[3];
	}
}

__global__ __launch_bounds__(64) void density_scale_kernel(const double *partial, int blocks, double *scale)
{
	double sum = 0.0, positive = 0.0;
	for (int b = threadIdx.x; b < blocks; b += 64)
	{
		sum += partial[2 * b];
		positive += partial[2 * b + 1];
	}
	for (int offset = 32; offset > 0; offset /= 2)
	{
		sum += __shfl_down(sum, offset, 64);
		positive += __shfl_down(positive, offset, 64);
	}
	if (threadIdx.x == 0)
	{
		scale[0] = positive > 0.0 ? positive / sum : 1.0;
	}
}

// One pass of forward and backward over `count` samples: the mean squared
// error of MLP(features) against `target`, scaled by `loss_scale` for the
// float16 gradients; grads (float32, parameter layout) and loss[0] accumulate.
//
// A wavefront takes tiles of 16 samples in the transposed form of the forward
// pass. The gradient of a layer's output, dY^T, has the layout of its
// activations, so dX^T = W dY^T runs on the same fragments (W's rows as A
// operands). A weight gradient dW = X^T dY contracts over the samples, which
// lie across lanes: both fragments pass through LDS with the samples of a unit
// side by side and come back as 8-byte operands. All sums stay in registers
// over the wavefront's tiles (one wavefront per SIMD holds them with the
// weights); the four wavefronts of a block then hand theirs over through LDS,
// fragment by fragment (plain adds in LDS, one wavefront after another, took 15
// us, LDS atomics 40), and a block adds 9.4 thousand sums to memory. 8,192 rows
// take 25 us; with one atomic per parameter and tile, on operands gathered from
// LDS two bytes at a time, 57.
constexpr int backward_waves = 4;
constexpr int sample_pitch = 20; // halves per unit: 16 samples, padded to 40 bytes

// The 16 x 16 tiles of the weight gradients of layers 1 (4), 2 and 3 (16 each),
// and how many of them the wavefronts exchange at a time.
constexpr int gradient_tiles = 4 + 16 + 16;
constexpr int exchanged_tiles = 12;
// Per wavefront: W4's, the three layers' biases', b4's gradients and the error.
constexpr int small_sums = 4 * hidden + 2;

struct backward_operands
{
	_Float16 weights[off_b1];
	_Float16 left[backward_waves][hidden * sample_pitch];
	_Float16 right[backward_waves][hidden * sample_pitch];
};

union backward_lds
{
	backward_operands operands;
	float4_t tiles[backward_waves][exchanged_tiles][64];
	float small[backward_waves][small_sums];
};

// A fragment (lane (g, c): units unit0 + 4 g + j of sample c) into LDS, a unit's
// samples side by side.
__device__ __forceinline__ void put_samples(_Float16 *lds, int unit0, int g, int c, half4_t v)
{
#pragma unroll
	for (int j = 0; j < 4; ++j)
	{
		lds[(unit0 + 4 * g + j) * sample_pitch + c] = v[j];
	}
}

// Samples 4 g .. 4 g + 3 of unit unit0 + c: an operand of a product over the
// samples.
__device__ __forceinline__ half4_t get_samples(const _Float16 *lds, int unit0, int g, int c)
{
	return *reinterpret_cast<const half4_t *>(lds + (unit0 + c) * sample_pitch + 4 * g);
}

// sums[4 k + n] += sum over the samples of left[16 k ..] right[16 n ..], K tiles
// of left units and 4 of right units.
template <int K>
__device__ __forceinline__ void add_products(const _Float16 *left, const _Float16 *right, int g, int c, float4_t *sums)
{
	half4_t r[4];
#pragma unroll
	for (int n = 0; n < 4; ++n)
	{
		r[n] = get_samples(right, 16 * n, g, c);
	}
#pragma unroll
	for (int k = 0; k < K; ++k)
	{
		const half4_t l = get_samples(left, 16 * k, g, c);
#pragma unroll
		for (int n = 0; n < 4; ++n)
		{
			sums[4 * k + n] = mfma16(l, r[n], sums[4 * k + n]);
		}
	}
}

__global__ __launch_bounds__(64 * backward_waves, 1) void mlp_backward_kernel(const __half *features,
	const float *target, const _Float16 *params_h, const float *params_f, float *grads, float *loss, int64_t count,
	float loss_scale)
{
	__shared__ backward_lds s;
	const int lane = threadIdx.x & 63;
	const int wave = threadIdx.x >> 6;
	const int g = lane >> 4;
	const int c = lane & 15;
	_Float16 *staged = s.operands.weights;
	for (int i = threadIdx.x; i < off_b1; i += 64 * backward_waves)
	{
		staged[i] = params_h[i];
	}
	__syncthreads();
	half4_t w1[4];
	half8_t w2[4][2], w3[4][2], w4[2];   // W^T as A operands (forward)
	half8_t b2[4][2], b3[4][2];          // W as A operands (backward)
	float w4_unit[4][4];                 // W4's column per held unit
	float4_t bias[3][4];
#pragma unroll
	for (int mt = 0; mt < 4; ++mt)
	{
#pragma unroll
		for (int j = 0; j < 4; ++j)
		{
			w1[mt][j] = staged[off_w1 + (4 * g + j) * hidden + mt * 16 + c];
			w4_unit[mt][j] = static_cast<float>(staged[off_w4 + (16 * mt + 4 * g + j) * 16]);
#pragma unroll
			for (int layer = 0; layer < 3; ++layer)
			{
				bias[layer][mt][j] = params_f[off_b1 + layer * hidden + 16 * mt + 4 * g + j];
			}
		}
#pragma unroll
		for (int t = 0; t < 2; ++t)
		{
#pragma unroll
			for (int j = 0; j < 8; ++j)
			{
				const int unit = 32 * t + (j < 4 ? 4 * g + j : 16 + 4 * g + j - 4);
				w2[mt][t][j] = staged[off_w2 + unit * hidden + mt * 16 + c];
				w3[mt][t][j] = staged[off_w3 + unit * hidden + mt * 16 + c];
				b2[mt][t][j] = staged[off_w2 + (mt * 16 + c) * hidden + unit];
				b3[mt][t][j] = staged[off_w3 + (mt * 16 + c) * hidden + unit];
				w4[t][j] = staged[off_w4 + unit * 16 + c];
			}
		}
	}
	const float b4 = params_f[off_b4];
	__syncthreads();

	const float4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
	float4_t tile_sums[gradient_tiles];
	float4_t unit_sums[4][4]; // W4's and the three biases' gradients, per held unit and sample
#pragma unroll
	for (int i = 0; i < gradient_tiles; ++i)
	{
		tile_sums[i] = zero;
	}
#pragma unroll
	for (int i = 0; i < 4; ++i)
	{
		unit_sums[0][i] = unit_sums[1][i] = unit_sums[2][i] = unit_sums[3][i] = zero;
	}
	float gb4 = 0.0f;
	float error = 0.0f;
	_Float16 *left = s.operands.left[wave];
	_Float16 *right = s.operands.right[wave];
	const float inverse = 1.0f / static_cast<float>(count);
	const int64_t tiles = (count + 15) / 16;
	for (int64_t tile = blockIdx.x * static_cast<int64_t>(backward_waves) + wave; tile < tiles;
		tile += static_cast<int64_t>(gridDim.x) * backward_waves)
	{
		const int64_t row = tile * 16 + c;
		half4_t x = {0, 0, 0, 0};
		if (row < count)
		{
			x = *reinterpret_cast<const half4_t *>(features + row * inputs + 4 * g);
		}
		half4_t h1[4], h2[4], h3[4];
#pragma unroll
		for (int mt = 0; mt < 4; ++mt)
		{
			h1[mt] = relu_half(mfma16(w1[mt], x, bias[0][mt]));
		}
#pragma unroll
		for (int mt = 0; mt < 4; ++mt)
		{
			h2[mt] = relu_half(mfma32(w2[mt][1], join(h1[2], h1[3]), mfma32(w2[mt][0], join(h1[0], h1[1]), bias[1][mt])));
		}
#pragma unroll
		for (int mt = 0; mt < 4; ++mt)
		{
			h3[mt] = relu_half(mfma32(w3[mt][1], join(h2[2], h2[3]), mfma32(w3[mt][0], join(h2[0], h2[1]), bias[2][mt])));
		}
		const float4_t y = mfma32(w4[1], join(h3[2], h3[3]), mfma32(w4[0], join(h3[0], h3[1]), zero));
		// dOut = 2 (out - target) / count, scaled; rows beyond count carry 0.
		// The outputs sit in lanes c of group 0.
		float d = 0.0f;
		if (g == 0 && row < count)
		{
			const float difference = y[0] + b4 - target[row];
			error += difference * difference * inverse;
			d = 2.0f * difference * inverse * loss_scale;
			gb4 += d;
		}
		d = __shfl(d, c, 64);

		// Layer 4, and dH3 = dOut W4 where h3 > 0.
		half4_t dh[4];
		const auto masked = [](const half4_t &h, const float4_t &v)
		{
			float4_t m;
#pragma unroll
			for (int j = 0; j < 4; ++j)
			{
				m[j] = static_cast<float>(h[j]) > 0.0f ? v[j] : 0.0f;
			}
			return m;
		};
		const auto rounded = [](const float4_t &v)
		{
			return half4_t{static_cast<_Float16>(v[0]), static_cast<_Float16>(v[1]), static_cast<_Float16>(v[2]),
				static_cast<_Float16>(v[3])};
		};
#pragma unroll
		for (int mt = 0; mt < 4; ++mt)
		{
			float4_t v;
#pragma unroll
			for (int j = 0; j < 4; ++j)
			{
				unit_sums[0][mt][j] += static_cast<float>(h3[mt][j]) * d;
				v[j] = d * w4_unit[mt][j];
			}
			v = masked(h3[mt], v);
			unit_sums[3][mt] += v;
			dh[mt] = rounded(v);
			put_samples(left, 16 * mt, g, c, h2[mt]);
			put_samples(right, 16 * mt, g, c, dh[mt]);
		}
		wave_order();
		add_products<4>(left, right, g, c, tile_sums + 20);
		wave_order();
		// dH2 = W3 dH3 where h2 > 0.
		half4_t next[4];
#pragma unroll
		for (int mt = 0; mt < 4; ++mt)
		{
			const float4_t v = masked(h2[mt], mfma32(b3[mt][1], join(dh[2], dh[3]),
				mfma32(b3[mt][0], join(dh[0], dh[1]), zero)));
			unit_sums[2][mt] += v;
			next[mt] = rounded(v);
			put_samples(left, 16 * mt, g, c, h1[mt]);
			put_samples(right, 16 * mt, g, c, next[mt]);
		}
		wave_order();
		add_products<4>(left, right, g, c, tile_sums + 4);
		wave_order();
		// dH1 = W2 dH2 where h1 > 0.
		put_samples(left, 0, g, c, x);
#pragma unroll
		for (int mt = 0; mt < 4; ++mt)
		{
			const float4_t v = masked(h1[mt], mfma32(b2[mt][1], join(next[2], next[3]),
				mfma32(b2[mt][0], join(next[0], next[1]), zero)));
			unit_sums[1][mt] += v;
			put_samples(right, 16 * mt, g, c, rounded(v));
		}
		wave_order();
		add_products<1>(left, right, g, c, tile_sums);
		wave_order();
	}

	// The samples' sums over the 16 lanes of a group.
	const auto over_samples = [](float v)
	{
#pragma unroll
		for (int offset = 8; offset > 0; offset /= 2)
		{
			v += __shfl_xor(v, offset, 64);
		}
		return v;
	};
	// The tiles, a few at a time: each wavefront writes its own, and adds up and
	// sends on a quarter of them all.
#pragma unroll
	for (int first = 0; first < gradient_tiles; first += exchanged_tiles)
	{
		__syncthreads();
#pragma unroll
		for (int i = 0; i < exchanged_tiles; ++i)
		{
			s.tiles[wave][i][lane] = tile_sums[first + i];
		}
		__syncthreads();
#pragma unroll
		for (int i = 0; i < exchanged_tiles / backward_waves; ++i)
		{
			const int local = i * backward_waves + wave;
			float4_t sum = s.tiles[0][local][lane];
#pragma unroll
			for (int w = 1; w < backward_waves; ++w)
			{
				sum += s.tiles[w][local][lane];
			}
			const int tile = first + local;
			const int k = tile < 4 ? 0 : (tile - 4) % 16 / 4;
			float *target = grads + (tile < 4 ? off_w1 : (tile < 20 ? off_w2 : off_w3)) + (16 * k + 4 * g) * hidden +
				16 * (tile % 4) + c;
#pragma unroll
			for (int j = 0; j < 4; ++j)
			{
				atomicAdd(target + j * hidden, sum[j]);
			}
		}
	}
	__syncthreads();
#pragma unroll
	for (int layer = 0; layer < 4; ++layer)
	{
#pragma unroll
		for (int mt = 0; mt < 4; ++mt)
		{
#pragma unroll
			for (int j = 0; j < 4; ++j)
			{
				const float sum = over_samples(unit_sums[layer][mt][j]);
				if (c == 0)
				{
					s.small[wave][layer * hidden + 16 * mt + 4 * g + j] = sum;
				}
			}
		}
	}
	gb4 = over_samples(gb4);
	error = over_samples(error);
	if (lane == 0)
	{
		s.small[wave][4 * hidden] = gb4;
		s.small[wave][4 * hidden + 1] = error;
	}
	__syncthreads();
	for (int i = threadIdx.x; i < small_sums; i += blockDim.x)
	{
		float sum = 0.0f;
		for (int w = 0; w < backward_waves; ++w)
		{
			sum += s.small[w][i];
		}
		const int unit = i % hidden;
		const int layer = i / hidden;
		float *target = i == 4 * hidden + 1 ? loss : (i == 4 * hidden ? grads + off_b4 :
			grads + (layer == 0 ? off_w4 + unit * 16 : (layer == 1 ? off_b1 : (layer == 2 ? off_b2 : off_b3)) + unit));
		atomicAdd(target, sum);
	}
}

// Adam on the float32 master parameters; refreshes the float16 copy. The
// gradients arrive multiplied by `loss_scale` (except the output layer's,
// which arrive multiplied too) and are cleared for the next step.
__global__ void adam_kernel(float *params, _Float16 *params_h, float *grads, float *m, float *v, int count, float lr,
	float beta1, float beta2, float eps, float correction1, float correction2, float loss_scale)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= count)
	{
		return;
	}
	const float g = grads[i] / loss_scale;
	grads[i] = 0.0f;
	const float mi = beta1 * m[i] + (1.0f - beta1) * g;
	const float vi = beta2 * v[i] + (1.0f - beta2) * g * g;
	m[i] = mi;
	v[i] = vi;
	const float update = lr * (mi / correction1) / (sqrtf(vi / correction2) + eps);
	const float p = params[i] - update;
	params[i] = p;
	params_h[i] = static_cast<_Float16>(p);
}

// The (ceil(N (N/2 + 1) / 256), N) grid of voxel_of_thread.
dim3 volume_grid(int big)
{
	const int64_t plane = static_cast<int64_t>(big) * (big / 2 + 1);
	return dim3(static_cast<unsigned>((plane + 255) / 256), static_cast<unsigned>(big));
}

unsigned blocks_of(int64_t count, int per)
{
	return static_cast<unsigned>(std::max<int64_t>(1, std::min<int64_t>((count + per - 1) / per, 16384)));
}

} // anonymous namespace

int mlp_parameter_count()
{
	return parameter_count;
}

void launch_compensation(const float *den, float *w, float *scratch, int big, int passes, float floor_value,
	hipStream_t stream)
{
	const int64_t count = static_cast<int64_t>(big) * big * (big / 2 + 1);
	// Ping-pong between w and scratch, starting so that the last pass
	// writes w.
	float *a = passes % 2 == 0 ? w : scratch;
	float *b = passes % 2 == 0 ? scratch : w;
	const int half = big / 2 + 1;
	const int columns = (half + compensation_width - 1) / compensation_width;
	const int width = (half + columns - 1) / columns;
	// As many rows as 256 threads and 512 halo elements take.
	const int height = std::min(256 / width, 512 / (width + 2) - 2);
	const int64_t plane_tiles = static_cast<int64_t>(columns) * ((big + height - 1) / height);
	int planes = compensation_planes;
	while (planes > 2 && plane_tiles * ((big + planes - 1) / planes) < compensation_blocks)
	{
		planes /= 2;
	}
	const dim3 tiles(static_cast<unsigned>(columns), static_cast<unsigned>((big + height - 1) / height),
		static_cast<unsigned>((big + planes - 1) / planes));
	for (int p = 0; p < passes; ++p)
	{
		const bool first = p == 0, last = p + 1 == passes;
		const auto kernel = first ? (last ? compensation_pass_kernel<true, true> : compensation_pass_kernel<true, false>) :
			(last ? compensation_pass_kernel<false, true> : compensation_pass_kernel<false, false>);
		kernel<<<tiles, 256, 0, stream>>>(den, first ? den : a, b, big, width, height, planes, floor_value);
		float *t = a;
		a = b;
		b = t;
	}
	if (passes == 0)
	{
		fill_kernel<<<blocks_of(count, 256), 256, 0, stream>>>(w, count, 1.0f);
	}
	REXLIB_HIP_CHECK(hipGetLastError());
}

void launch_coverage(const float *transforms, int64_t slices, int64_t ts0, int64_t ts1, int64_t ts2, int big,
	float *table, hipStream_t stream)
{
	constexpr int entries = coverage_radii * coverage_theta * coverage_phi;
	constexpr int64_t table_size = static_cast<int64_t>(entries) * coverage_bins;
	// Up to 64 slice ranges of whole tiles: 66 x 64 workgroups for large stacks.
	const int64_t tiles = std::max<int64_t>(1, (slices + coverage_tile - 1) / coverage_tile);
	const int64_t per_block = ((tiles + 63) / 64) * coverage_tile;
	const unsigned ranges = static_cast<unsigned>(std::max<int64_t>(1, (slices + per_block - 1) / per_block));
	fill_kernel<<<(table_size + 255) / 256, 256, 0, stream>>>(table, table_size, 0.0f);
	REXLIB_HIP_CHECK(hipGetLastError());
	coverage_count_kernel<<<dim3((entries + 255) / 256, ranges), 256, 0, stream>>>(transforms, slices, ts0, ts1, ts2,
		big, per_block, reinterpret_cast<unsigned *>(table));
	REXLIB_HIP_CHECK(hipGetLastError());
	coverage_normalize_kernel<<<(entries + 255) / 256, 256, 0, stream>>>(table);
	REXLIB_HIP_CHECK(hipGetLastError());
}

void launch_features(const float *den, const float *table, float density_scale, void *features, int big,
	hipStream_t stream)
{
	features_kernel<<<volume_grid(big), 256, 0, stream>>>(den, table, density_scale, static_cast<__half *>(features),
		big);
	REXLIB_HIP_CHECK(hipGetLastError());
}

void launch_density_scale(const float *den, int64_t count, double *scratch, double *scale, hipStream_t stream)
{
	const int blocks = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>((count + 255) / 256, density_blocks)));
	density_sums_kernel<<<blocks, 256, 0, stream>>>(den, count, scratch);
	density_scale_kernel<<<1, 64, 0, stream>>>(scratch, blocks, scale);
	REXLIB_HIP_CHECK(hipGetLastError());
}

int64_t density_scratch()
{
	return 2 * density_blocks;
}

void launch_predicted_weights(const float *den, const float *table, float density_scale, const void *params_h,
	const float *params_f, float *out, int big, hipStream_t stream)
{
	// Two blocks per CU, the registers' limit: each wavefront loads the weights
	// once for dozens of groups.
	const int64_t groups = static_cast<int64_t>((big * (big / 2 + 1) + 63) / 64) * big;
	predicted_weights_kernel<<<blocks_of(std::min<int64_t>(groups, 2048), 4), 256, 0, stream>>>(den, table, density_scale,
		static_cast<const _Float16 *>(params_h), params_f, out, big, 1.0 / (big * (1.0 / big)));
	REXLIB_HIP_CHECK(hipGetLastError());
}

void launch_mlp_forward(const void *features, const void *params_h, const float *params_f, float *out, int64_t count,
	hipStream_t stream)
{
	mlp_forward_kernel<<<static_cast<unsigned>(std::min<int64_t>(blocks_of((count + 31) / 32, 4), 512)), 256, 0, stream>>>(
		static_cast<const __half *>(features), static_cast<const _Float16 *>(params_h), params_f, out, count);
	REXLIB_HIP_CHECK(hipGetLastError());
}

void launch_mlp_backward(const void *features, const float *target, const void *params_h, const float *params_f,
	float *grads, float *loss, int64_t count, float loss_scale, hipStream_t stream)
{
// Two tiles per wavefront at least, one block per CU at most.
	const int64_t tiles = (count + 15) / 16;
	const unsigned blocks = static_cast<unsigned>(std::max<int64_t>(1, std::min<int64_t>((tiles + 2 * backward_waves - 1) /
		(2 * backward_waves), 256)));
	mlp_backward_kernel<<<blocks, 64 * backward_waves, 0, stream>>>(static_cast<const __half *>(features), target,
		static_cast<const _Float16 *>(params_h), params_f, grads, loss, count, loss_scale);
	REXLIB_HIP_CHECK(hipGetLastError());
}

void launch_adam(float *params, void *params_h, float *grads, float *m, float *v, float lr, float beta1, float beta2,
	float eps, int step, float loss_scale, hipStream_t stream)
{
	const float c1 = 1.0f - std::pow(beta1, static_cast<float>(step));
	const float c2 = 1.0f - std::pow(beta2, static_cast<float>(step));
	adam_kernel<<<(parameter_count + 255) / 256, 256, 0, stream>>>(params, static_cast<_Float16 *>(params_h), grads, m,
		v, parameter_count, lr, beta1, beta2, eps, c1, c2, loss_scale);
	REXLIB_HIP_CHECK(hipGetLastError());
}

} // namespace rexlib_hip
