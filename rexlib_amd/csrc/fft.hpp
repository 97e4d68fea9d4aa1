// Batched FFTs of the path: line descriptors and the block transform.
#pragma once

#include "common.hpp"

namespace rexlib_hip
{

constexpr int max_fft_stages = 16;

// A factorisation of the length into radices 4, 2, 3, 5.
struct fft_plan
{
	int32_t n;
	int32_t stages;
	int32_t radix[max_fft_stages];
};

// Lines of a batched transform: the line index l decomposes into
// (outer, middle, inner) = (l / (cm * ci), (l / ci) % cm, l % ci), and its
// first element and element stride are, in elements,
//   outer * s_outer + middle * s_middle + inner * s_inner, s_elem.
struct line_set
{
	int64_t count;
	int64_t middle_count;
	int64_t inner_count;
	int64_t s_outer;
	int64_t s_middle;
	int64_t s_inner;
	int64_t s_elem;
};

__host__ __device__ inline int64_t line_offset(const line_set &l, int64_t line)
{
	const int64_t inner = line % l.inner_count;
	const int64_t rest = line / l.inner_count;
	const int64_t middle = rest % l.middle_count;
	const int64_t outer = rest / l.middle_count;
	return outer * l.s_outer + middle * l.s_middle + inner * l.s_inner;
}

// Which real rows share a complex line: two rows of one transform (an image, or
// the rows along a transformed axis of a general one), never rows of different
// ones. Both halves of a line round relative to the larger of its rows, and a
// NaN or an infinity reaches both, which the transform's other axis does to all of its
// rows anyway; the rows of another transform, and every row where no other axis
// is transformed (`rows` = 1), stay as exact as on a line of their own.
struct row_pairs
{
	int64_t transforms;
	int32_t rows;      // of each transform that run
	int32_t in_rows;   // input rows of each transform
	int32_t in_shift;  // the running row of its first input row
	int32_t out_rows;  // output rows of each transform
	int32_t out_shift; // the output row of the first running row
};

__host__ __device__ inline int64_t line_count(const row_pairs &p)
{
	return p.transforms * ((p.rows + 1) / 2);
}

// Transforms of `rows` rows, in and out, `count` rows in all.
inline row_pairs whole_rows(int64_t rows, int64_t count)
{
	const int32_t r = static_cast<int32_t>(rows);
	return row_pairs{count / rows, r, r, 0, r, 0};
}

// Images of m rows zero-padded to n, their origin m/2 moved to n/2; `image_rows`:
// only the m rows run, the zero rows of the padding are not written.
inline row_pairs padded_rows(int64_t m, int64_t n, int64_t images, bool image_rows)
{
	const int32_t offset = static_cast<int32_t>(n / 2 - m / 2);
	return row_pairs{images, static_cast<int32_t>(image_rows ? m : n), static_cast<int32_t>(m),
		image_rows ? 0 : offset, static_cast<int32_t>(n), image_rows ? offset : 0};
}

// Row `q` (0 or 1) of a line: its transform, and the input and output row among
// all (-1: none).
struct line_row
{
	int64_t transform;
	int64_t in;
	int64_t out;
};

__device__ inline line_row row_of(const row_pairs &p, int64_t line, int q)
{
	const int pairs = (p.rows + 1) / 2;
	const int64_t transform = line / pairs;
	if (p.rows % 2 == 0 && p.in_rows == p.rows && p.out_rows == p.rows)
	{
		// Whole pairs of whole transforms: no division (it costs a row kernel 1 to 2 %
		// where nothing else takes the transform).
		const int64_t all = 2 * line + q;
		return all < p.transforms * p.rows ? line_row{transform, all, all} : line_row{0, -1, -1};
	}
	const int row = 2 * static_cast<int>(line - transform * pairs) + q;
	if (transform >= p.transforms || row >= p.rows)
	{
		return line_row{0, -1, -1};
	}
	const int in = row - p.in_shift;
	return line_row{transform, in >= 0 && in < p.in_rows ? transform * p.in_rows + in : -1,
		transform * p.out_rows + row + p.out_shift};
}

fft_plan make_fft_plan(int64_t n);

// Device twiddles exp(-2 pi i m / n), m < n, computed in double, cached per
// device and length.
const float2 *twiddles(int64_t n);

// Lines per block of the LDS transforms of length n.
int lines_per_group(int n);

// Stage callers: the element type of real lines.
enum real_kind : int
{
	real_f32 = 0,
	real_bf16 = 1,
	real_f16 = 2
};

} // namespace rexlib_hip
