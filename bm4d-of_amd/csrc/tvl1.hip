// TV-L1 optical flow on gfx950: Zach-Pock-Bischof duality scheme as the
// reference implements it (lib/tvl1flow/tvl1flow_lib.c, mask.c,
// bicubic_interpolation.c, zoom.c).
//
// All frame pairs of a sequence are solved together: every kernel takes a
// pair index in blockIdx.y and skips pairs that have converged.  Per-pixel
// arithmetic follows the reference operation by operation (this file is
// compiled with -ffp-contract=off; bicubic and Gaussian sums in double as in
// the reference), so a pixel's update is bit-identical given identical
// inputs.  The per-iteration mean squared update is reduced in double in a
// fixed order; the reference sums it in float in pixel order, so the stopping
// iteration can differ by one where the error lands next to epsilon^2.
#include "ctx.hpp"

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>
#include <algorithm>
#include <array>
#include <mutex>
#include <stdexcept>

namespace bm4dof {

#define TV_MAX_ITERATIONS 300      // tvl1flow_lib.c:24
#define TV_PRESMOOTHING_SIGMA 0.8  // tvl1flow_lib.c:25
#define TV_GRAD_IS_ZERO 1E-10      // tvl1flow_lib.c:26
#define TV_ZOOM_SIGMA_ZERO 0.6     // zoom.c:17
#define TV_THREADS 256

// --------------------------------------------------------------- bicubic

__device__ __forceinline__ int nbc(int x, int n, bool &out) // bicubic_interpolation.c:25-39
{
	if (x < 0) { out = true; return 0; }
	if (x >= n) { out = true; return n - 1; }
	return x;
}

__device__ __forceinline__ double cubic_cell(double v0, double v1, double v2, double v3, double x)
{ // bicubic_interpolation.c:102-112
	return v1 + 0.5 * x * (v2 - v0 +
		x * (2.0 * v0 - 5.0 * v1 + 4.0 * v2 - v3 +
		x * (3.0 * (v1 - v2) + v3 - v0)));
}

// bicubic_interpolation_at (bicubic_interpolation.c:138-234), Neumann case;
// the y-neighbour above uses the x sign, as in the reference.
__device__ float bicubic_at(const float *__restrict__ in, float uu, float vv, int nx, int ny,
                            bool border_out)
{
	const int sx = (uu < 0) ? -1 : 1;
	const int sy = (vv < 0) ? -1 : 1;
	bool out = false;
	const int x = nbc((int)uu, nx, out);
	const int y = nbc((int)vv, ny, out);
	const int mx = nbc((int)uu - sx, nx, out);
	const int my = nbc((int)vv - sx, ny, out);
	const int dx = nbc((int)uu + sx, nx, out);
	const int dy = nbc((int)vv + sy, ny, out);
	const int ddx = nbc((int)uu + 2 * sx, nx, out);
	const int ddy = nbc((int)vv + 2 * sy, ny, out);
	if (out && border_out) return 0.0f;
	const int cols[4] = {mx, x, dx, ddx};
	const double fy = (double)(vv - y);
	double v[4];
#pragma unroll
	for (int c = 0; c < 4; c++) {
		const double a0 = in[cols[c] + nx * my];
		const double a1 = in[cols[c] + nx * y];
		const double a2 = in[cols[c] + nx * dy];
		const double a3 = in[cols[c] + nx * ddy];
		v[c] = cubic_cell(a0, a1, a2, a3, fy);
	}
	return (float)cubic_cell(v[0], v[1], v[2], v[3], (double)(uu - x));
}

// ------------------------------------------------------------ pyramid

// min/max of I0 and I1 per pair (tvl1flow_lib.c:286-320): partials per block.
__global__ void tv_minmax_kernel(const float *__restrict__ I, int size, const int *__restrict__ i0,
                                 const int *__restrict__ i1, float *__restrict__ part)
{
	const int pr = blockIdx.y;
	const float *a = I + (size_t)i0[pr] * size;
	const float *b = I + (size_t)i1[pr] * size;
	float mn0 = INFINITY, mx0 = -INFINITY, mn1 = INFINITY, mx1 = -INFINITY;
	for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < size; i += gridDim.x * blockDim.x) {
		mn0 = fminf(mn0, a[i]); mx0 = fmaxf(mx0, a[i]);
		mn1 = fminf(mn1, b[i]); mx1 = fmaxf(mx1, b[i]);
	}
	__shared__ float s[4][TV_THREADS];
	s[0][threadIdx.x] = mn0; s[1][threadIdx.x] = mx0; s[2][threadIdx.x] = mn1; s[3][threadIdx.x] = mx1;
	__syncthreads();
	for (int st = TV_THREADS / 2; st > 0; st >>= 1) {
		if (threadIdx.x < st) {
			s[0][threadIdx.x] = fminf(s[0][threadIdx.x], s[0][threadIdx.x + st]);
			s[1][threadIdx.x] = fmaxf(s[1][threadIdx.x], s[1][threadIdx.x + st]);
			s[2][threadIdx.x] = fminf(s[2][threadIdx.x], s[2][threadIdx.x + st]);
			s[3][threadIdx.x] = fmaxf(s[3][threadIdx.x], s[3][threadIdx.x + st]);
		}
		__syncthreads();
	}
	if (threadIdx.x < 4) part[((size_t)pr * gridDim.x + blockIdx.x) * 4 + threadIdx.x] = s[threadIdx.x][0];
}

// image_normalization (tvl1flow_lib.c:303-337) into the level-0 buffers.
__global__ void tv_normalize_kernel(const float *__restrict__ I, int size, const int *__restrict__ i0,
                                    const int *__restrict__ i1, const float *__restrict__ part,
                                    int nparts, float *__restrict__ I0n, float *__restrict__ I1n)
{
	const int pr = blockIdx.y;
	float mn0 = INFINITY, mx0 = -INFINITY, mn1 = INFINITY, mx1 = -INFINITY;
	for (int k = 0; k < nparts; k++) {
		const float *q = part + ((size_t)pr * nparts + k) * 4;
		mn0 = fminf(mn0, q[0]); mx0 = fmaxf(mx0, q[1]); mn1 = fminf(mn1, q[2]); mx1 = fmaxf(mx1, q[3]);
	}
	const float max = (mx0 > mx1) ? mx0 : mx1;
	const float min = (mn0 < mn1) ? mn0 : mn1;
	const float den = max - min;
	const float *a = I + (size_t)i0[pr] * size;
	const float *b = I + (size_t)i1[pr] * size;
	float *oa = I0n + (size_t)pr * size, *ob = I1n + (size_t)pr * size;
	for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < size; i += gridDim.x * blockDim.x) {
		if (den > 0) {
			oa[i] = 255.0 * (a[i] - min) / den;
			ob[i] = 255.0 * (b[i] - min) / den;
		} else {
			oa[i] = a[i];
			ob[i] = b[i];
		}
	}
}

// Gaussian smoothing with reflecting boundaries (mask.c:217-333), one pass.
// rows: convolve along x; else along y.  Taps in constant-size array B.
__global__ void tv_gauss_kernel(const float *__restrict__ in, float *__restrict__ out, int nx, int ny,
                                int stride_pair, const double *__restrict__ B, int size, int rows)
{
	const int pr = blockIdx.y;
	const float *I = in + (size_t)pr * stride_pair;
	float *O = out + (size_t)pr * stride_pair;
	const int n = nx * ny;
	for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
		const int i = p / nx, j = p - i * nx;
		// extended coordinate e = (rows ? j : i) + size; R[e] with reflection
		const int len = rows ? nx : ny;
		const int pos = rows ? j : i;
		auto R = [&](int e) -> double {
			int q;
			if (e < size) q = size - e;                  // R[i] = I[size - i]
			else if (e >= len + size) q = len - 1 - (e - len - size); // R[bd+i] = I[len-1-i]
			else q = e - size;
			return rows ? (double)I[i * nx + q] : (double)I[q * nx + j];
		};
		const int e = pos + size;
		double sum = B[0] * R(e);
		for (int t = 1; t < size; t++) sum += B[t] * (R(e - t) + R(e + t));
		O[p] = (float)sum;
	}
}

// zoom_out resampling (zoom.c:66-76) of the pre-smoothed image.
__global__ void tv_zoom_out_kernel(const float *__restrict__ Is, int nx, int ny, int in_stride,
                                   float *__restrict__ out, int nxx, int nyy, int out_stride,
                                   float factor)
{
	const int pr = blockIdx.y;
	const float *I = Is + (size_t)pr * in_stride;
	float *O = out + (size_t)pr * out_stride;
	for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < nxx * nyy; p += gridDim.x * blockDim.x) {
		const int i1 = p / nxx, j1 = p - i1 * nxx;
		const float i2 = (float)i1 / factor;
		const float j2 = (float)j1 / factor;
		O[p] = bicubic_at(I, j2, i2, nx, ny, false);
	}
}

// zoom_in (zoom.c:87-111) followed by the 1/zfactor scaling
// (tvl1flow_lib.c:426-435); `scale` is (float)1.0/zfactor.
__global__ void tv_zoom_in_kernel(const float *__restrict__ in, int nx, int ny, int in_stride,
                                  float *__restrict__ out, int nxx, int nyy, int out_stride,
                                  float scale)
{
	const int pr = blockIdx.y;
	const float *I = in + (size_t)pr * in_stride;
	float *O = out + (size_t)pr * out_stride;
	const float factorx = ((float)nxx / nx);
	const float factory = ((float)nyy / ny);
	for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < nxx * nyy; p += gridDim.x * blockDim.x) {
		const int i1 = p / nxx, j1 = p - i1 * nxx;
		const float i2 = (float)i1 / factory;
		const float j2 = (float)j1 / factorx;
		O[p] = bicubic_at(I, j2, i2, nx, ny, false) * scale;
	}
}

// ------------------------------------------------------------ one scale

// centered_gradient (mask.c:152-209): clamped central differences, 0.5*()
// in double.
__global__ void tv_cgrad_kernel(const float *__restrict__ I1, int nx, int ny, int stride,
                                float *__restrict__ Ix, float *__restrict__ Iy)
{
	const int pr = blockIdx.y;
	const float *in = I1 + (size_t)pr * stride;
	for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < nx * ny; p += gridDim.x * blockDim.x) {
		const int i = p / nx, j = p - i * nx;
		const int jl = j > 0 ? j - 1 : 0, jr = j < nx - 1 ? j + 1 : nx - 1;
		const int iu = i > 0 ? i - 1 : 0, id = i < ny - 1 ? i + 1 : ny - 1;
		Ix[(size_t)pr * stride + p] = 0.5 * (in[i * nx + jr] - in[i * nx + jl]);
		Iy[(size_t)pr * stride + p] = 0.5 * (in[id * nx + j] - in[iu * nx + j]);
	}
}

// Warping of I1, I1x, I1y by u and the constant part of rho
// (tvl1flow_lib.c:142-161).
__global__ void tv_warp_kernel(const float *__restrict__ I0, const float *__restrict__ I1,
                               const float *__restrict__ I1x, const float *__restrict__ I1y,
                               const float *__restrict__ u1a, const float *__restrict__ u2a,
                               const float *__restrict__ u1b, const float *__restrict__ u2b,
                               const int *__restrict__ cur, int nx, int ny, int stride,
                               float *__restrict__ I1wx, float *__restrict__ I1wy, float *__restrict__ grad,
                               float *__restrict__ rho_c)
{
	const int pr = blockIdx.y;
	const size_t off = (size_t)pr * stride;
	const bool flip = cur[pr] != 0;
	const float *__restrict__ u1 = flip ? u1b : u1a;
	const float *__restrict__ u2 = flip ? u2b : u2a;
	for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < nx * ny; p += gridDim.x * blockDim.x) {
		const int i = p / nx, j = p - i * nx;
		const float uu = (float)(j + u1[off + p]);
		const float vv = (float)(i + u2[off + p]);
		const float w = bicubic_at(I1 + off, uu, vv, nx, ny, true);
		const float wx = bicubic_at(I1x + off, uu, vv, nx, ny, true);
		const float wy = bicubic_at(I1y + off, uu, vv, nx, ny, true);
		const float Ix2 = wx * wx;
		const float Iy2 = wy * wy;
		I1wx[off + p] = wx;
		I1wy[off + p] = wy;
		grad[off + p] = (Ix2 + Iy2);
		rho_c[off + p] = (w - wx * u1[off + p] - wy * u2[off + p] - I0[off + p]);
	}
}

// ------------------------------------------------- primal-dual iterations
// K iterations of the TV-L1 primal-dual scheme (tvl1flow_lib.c:165-246) per
// launch, on tiles held in registers: a lane is a column and a thread has R
// rows of it, W waves below one another make the block, so a block covers
// 64 x R W pixels, the tile and K pixels of halo on each side.  After
// iteration j the pixels at least j pixels inside a cut halo edge are exact
// (an iteration reaches one pixel in each direction: the divergence backwards,
// the gradient forwards), so after K iterations the tile itself is, and only
// it is written back.  Per iteration: the TH step, divergence of p and u
// update (phase A), then the forward gradient of the new u and the p update
// (phase B); each pixel's arithmetic is the reference's, operation for
// operation, as in the one-iteration form.  Left and right neighbours come
// from the next lane, those above and below from the thread's own registers;
// only the rows where two waves meet go through LDS.  Pixels outside the
// image hold zeros throughout: what the reference leaves out of the
// divergence at a border is then a zero, and p's components across the last
// row and column stay zero because their gradients are (mask.c:43-144).  The
// squared update of every tile pixel and iteration is summed in double in a
// fixed order into part[pair][j][tile].
//
// The state (u1, u2, p11, p12, p21, p22) is double-buffered: a pair reads
// buffer cur[pair] and writes the other.  ctl[pair] is the number of
// iterations to run this round (0: idle).  The pair's last block of the round
// sums the tiles' partials and applies the stopping test to each iteration of
// the round in order (tv_round_decide); if it fires before the round's last
// iteration, the pair runs that many iterations again from the same source
// buffer (an exact re-run), so the state and the iteration count are those
// of the iteration the test fired on.
//
// Bound, many pairs: vector instructions, some 76 a pixel in phase B (two
// roots in double, four quotients) and 36 in phase A, times 1.29 for the halo
// (1.14 in x, 27 rows of 24 in y), issuing 80 % of the time at four waves a
// SIMD; 38 pairs of 960x540, all active: 550 us a round of four iterations,
// 2.9 TB/s.  With the state in LDS (64 x 32 tiles, 26 LDS accesses a pixel,
// both pipes 75 % busy) both flows of 960x540x20 took 73 ms, with two columns
// a lane or 1024 threads, which leave the loads of a block nothing to run
// beside, 93; five or more rows a thread spill.
// A single pair is latency: 56 x 8 tiles of two rows a thread, 9.3 us a round
// with its test, against 14.2 and 3.7 us for 32 x 16 tiles of three waves and a
// launch for the test.  Flow of one 333x251 pair: 11.2 to 6.7 ms; both flows
// of 960x540x20: 82.5 to 68 ms.
// ---------------------------------------------------------------------------
struct TVPlanes {
	float *u1, *u2, *p11, *p12, *p21, *p22;
};

#define TV_K 4
// mode[pair]: TV_REDO in the re-run, and TV_BLOCK for each block of the round
// that is done.
enum { TV_RUN = 0, TV_REDO = 1, TV_BLOCK = 2 };

// The stopping test of every iteration of a round, in order
// (tvl1flow_lib.c:165, 225), given errs[j] = the mean squared update of
// iteration j: the loop ends when error <= epsilon^2 or the count reaches
// MAX_ITERATIONS.  state[pair] receives the final count.  A round that
// stops before its last iteration is run again from the same source buffer
// with that many iterations (mode TV_REDO), so the state and the count are
// those of the iteration the test fired on.  The next round gets the
// iterations the test needs if the updates go on falling at the last rate,
// at most K: most solves then end with a round and are not run again.
template <int K>
__device__ void tv_round_decide(int pr, int kk, const float (&errs)[K], float eps2, bool redo, int *__restrict__ ctl,
                                int *__restrict__ cur, int *__restrict__ iters, int *__restrict__ mode,
                                int *__restrict__ state, int *__restrict__ n_active)
{
	const int done = iters[pr];
	int stop = -1;
	float last = 0.f, before = 0.f;
#pragma unroll
	for (int j = 0; j < K; j++) {
		if (j >= kk) continue;
		if (stop < 0 && (!(errs[j] > eps2) || done + j + 1 >= TV_MAX_ITERATIONS)) stop = j;
		before = last;
		last = errs[j];
	}
	mode[pr] = TV_RUN;
	if (!redo && stop >= 0 && stop < kk - 1) {
		mode[pr] = TV_REDO;
		ctl[pr] = stop + 1;
		return;
	}
	iters[pr] = done + kk;
	cur[pr] ^= 1;
	if (redo || stop >= 0) {
		state[pr] = done + kk;
		ctl[pr] = 0;
		atomicSub(n_active, 1);
		return;
	}
	int n = K;
	if (kk > 1 && last < before) {
		const float rate = last / before;
		float e = last * rate;
		for (n = 1; n < K && e > eps2; n++) e *= rate;
	}
	ctl[pr] = min(n, TV_MAX_ITERATIONS - (done + kk));
}

// sqrt of a double that is +0 or at least 2^-767, as the compiler's
// correctly rounded sqrt computes it (rsq, then the Newton steps below) with
// its range scaling left out: that scaling applies only below 2^-767, and
// x^2 + y^2 of floats is +0 or at least 2^-298.  Same bits, five
// instructions fewer.  POS: s is positive and finite.
template <bool POS> __device__ __forceinline__ double sqrt_sum_sq(double s)
{
	const double y = __builtin_amdgcn_rsq(s);
	double g = s * y, h = y * 0.5;
	const double r = __builtin_fma(-h, g, 0.5);
	g = __builtin_fma(g, r, g);
	h = __builtin_fma(h, r, h);
	double d = __builtin_fma(-g, g, s);
	g = __builtin_fma(d, h, g);
	d = __builtin_fma(-g, g, s);
	g = __builtin_fma(d, h, g);
	if (POS) return g;
	return __builtin_amdgcn_class(s, 0x260) ? s : g;   // +-0 and +inf give themselves
}

// a / d for several a and one d below 2^126 (whose float reciprocal is then a
// normal number): a times the reciprocal in double (two Newton steps from the
// float one, within 2^-51), rounded to float.  The quotient of two floats is 2^-49 or more away, relatively, from where two
// floats meet, so this is the correctly rounded quotient (of results below
// 2^-126 the last bit can differ).
__device__ __forceinline__ double tv_recip(float d)
{
	const double e = (double)d;
	double y = (double)__builtin_amdgcn_rcpf(d);
	y = __builtin_fma(__builtin_fma(-e, y, 1.0), y, y);
	return __builtin_fma(__builtin_fma(-e, y, 1.0), y, y);
}
__device__ __forceinline__ float tv_quot(float a, double y) { return (float)((double)a * y); }

// Phase A of a pixel: TH, divergence (dp1, dp2), u (tvl1flow_lib.c:170-225).
// yg: the reciprocal of g; flat: g < TV_GRAD_IS_ZERO, where the reference sets
// the quotient 0 (also of a rho that is no number).  Returns the squared update.
__device__ __forceinline__ float tv_pixel_u(float &u1, float &u2, float dp1, float dp2, float wx, float wy, float g,
                                            double yg, bool flat, float rc, float l_t, float theta)
{
	const float rho = rc + (wx * u1 + wy * u2);
	const float lg = l_t * g;
	float fi = flat ? 0.f : tv_quot(-rho, yg);
	fi = rho > lg ? -l_t : fi;
	fi = rho < -lg ? l_t : fi;
	const float v1 = u1 + fi * wx, v2 = u2 + fi * wy;
	const float n1 = v1 + theta * dp1;
	const float n2 = v2 + theta * dp2;
	const float q = (n1 - u1) * (n1 - u1) + (n2 - u2) * (n2 - u2);
	u1 = n1;
	u2 = n2;
	return q;
}

// Phase B: p from the forward gradient of the new u (tvl1flow_lib.c:228-245).
__device__ __forceinline__ void tv_pixel_p(float &p11, float &p12, float &p21, float &p22, float u1x, float u1y,
                                           float u2x, float u2y, float taut)
{
	// x^2 + y^2 in double: the squares are exact, so the fma rounds as the
	// sum does; 2^-400 is lost in a sum that is not zero and gives a zero one
	// a root that rounds to 0
	const double s1 = __builtin_fma((double)u1x, (double)u1x, __builtin_fma((double)u1y, (double)u1y, 0x1p-400));
	const double s2 = __builtin_fma((double)u2x, (double)u2x, __builtin_fma((double)u2y, (double)u2y, 0x1p-400));
	// the reference adds 1.0 in double and stores to float; for a
	// float t >= 0 that is the float sum 1 + t: the double sum is
	// exact for 2^-29 <= t < 2^53, rounds to a value that rounds to 1
	// below, and to t above, as the float sum does
	float ng1 = 1.0f + taut * (float)sqrt_sum_sq<true>(s1);
	float ng2 = 1.0f + taut * (float)sqrt_sum_sq<true>(s2);
	const float b11 = p11 + taut * u1x, b12 = p12 + taut * u1y;
	const float b21 = p21 + taut * u2x, b22 = p22 + taut * u2y;
	const double y1 = tv_recip(ng1), y2 = tv_recip(ng2);
	p11 = tv_quot(b11, y1);
	p12 = tv_quot(b12, y1);
	p21 = tv_quot(b21, y2);
	p22 = tv_quot(b22, y2);
	if (__builtin_expect(!(ng1 + ng2 < 0x1p126f), 0)) {
		asm volatile("");   // (a branch, not both sides)
		ng1 = 1.0f + taut * (float)sqrt_sum_sq<false>((double)u1x * u1x + (double)u1y * u1y);
		ng2 = 1.0f + taut * (float)sqrt_sum_sq<false>((double)u2x * u2x + (double)u2y * u2y);
		p11 = b11 / ng1;
		p12 = b12 / ng1;
		p21 = b21 / ng2;
		p22 = b22 / ng2;
	}
}

// The value of the lane before / after (first / last lane: 0).
__device__ __forceinline__ float tv_lane_before(float v)
{
	return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));   // wave_shr:1
}
__device__ __forceinline__ float tv_lane_after(float v)
{
	return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));   // wave_shl:1
}

template <int R> struct TVRows {
	float u1[R], u2[R], p11[R], p12[R], p21[R], p22[R];
	float wx[R], wy[R], rc[R], g[R];
	double yg[R];
	bool flat[R];
};
// Rows the waves hand to each other: the first row's u, the last row's p12
// and p22.
template <int W> struct TVEdge {
	float u[W][2][64], p[W][2][64];
};

// kk iterations.  x, y0: the thread's column and first row; yt: that row in
// the tile.  XB: the block reaches the first or last column of the image.
template <int R, int W, int K, bool XB>
__device__ __forceinline__ void tv_iterate(TVRows<R> &t, TVEdge<W> &L, int wv, int lane, int x, int y0, int yt, int nx,
                                           int ny, int kk, float l_t, float theta, float taut, double (&err)[K])
{
	constexpr int TX = 64 - 2 * K, TY = R * W - 2 * K;
	const bool own = lane >= K && lane < TX + K && (!XB || x < nx);   // column of the tile
	const bool side = XB && (x == 0 || x == nx - 1), out = XB && (x < 0 || x >= nx), last = XB && x == nx - 1;
	for (int j = 0; j < kk; j++) {
		// with m iterations still to come: u is needed on the tile's rows
		// -m .. TY + m, p on -m .. TY + m - 1
		const int m = kk - 1 - j;
		const int lo = max(-m, yt - y0), hi = min(TY + m, yt - y0 + ny - 1);   // rows of the image among them
		double ej = 0.0;
#pragma unroll
		for (int r = 0; r < R; r++) {
			const int y = yt + r;
			if (y < lo || y > hi) continue;
			const float a11m = tv_lane_before(t.p11[r]), a21m = tv_lane_before(t.p21[r]);
			const float a12u = r ? t.p12[r ? r - 1 : 0] : L.p[wv ? wv - 1 : 0][0][lane];
			const float a22u = r ? t.p22[r ? r - 1 : 0] : L.p[wv ? wv - 1 : 0][1][lane];
			const float h1 = t.p11[r] - a11m, h2 = t.p21[r] - a21m;
			float dp1 = h1 + (t.p12[r] - a12u), dp2 = h2 + (t.p22[r] - a22u);
			if (XB && y0 + r > 0 && y0 + r < ny - 1) {   // in the first and last column the reference sums from the left
				dp1 = side ? (h1 + t.p12[r]) - a12u : dp1;
				dp2 = side ? (h2 + t.p22[r]) - a22u : dp2;
			}
			const float q = tv_pixel_u(t.u1[r], t.u2[r], dp1, dp2, t.wx[r], t.wy[r], t.g[r], t.yg[r], t.flat[r],
			                           t.rc[r], l_t, theta);
			if (y >= 0 && y < TY) ej += (double)(own ? q : 0.f);
		}
#pragma unroll
		for (int q = 0; q < K; q++) if (q == j) err[q] = ej;
		L.u[wv][0][lane] = t.u1[0];
		L.u[wv][1][lane] = t.u2[0];
		__syncthreads();
#pragma unroll
		for (int r = 0; r < R; r++) {
			const int y = yt + r;
			if (y < lo || y > min(hi, TY + m - 1)) continue;
			const float d1 = r + 1 < R ? t.u1[r + 1 < R ? r + 1 : 0] : L.u[wv + 1 < W ? wv + 1 : wv][0][lane];
			const float d2 = r + 1 < R ? t.u2[r + 1 < R ? r + 1 : 0] : L.u[wv + 1 < W ? wv + 1 : wv][1][lane];
			float u1x = tv_lane_after(t.u1[r]) - t.u1[r], u1y = d1 - t.u1[r];
			float u2x = tv_lane_after(t.u2[r]) - t.u2[r], u2y = d2 - t.u2[r];
			if (XB) {
				u1x = out || last ? 0.f : u1x;
				u2x = out || last ? 0.f : u2x;
				u1y = out ? 0.f : u1y;
				u2y = out ? 0.f : u2y;
			}
			if (y0 + r == ny - 1) u1y = u2y = 0.f;
			tv_pixel_p(t.p11[r], t.p12[r], t.p21[r], t.p22[r], u1x, u1y, u2x, u2y, taut);
		}
		L.p[wv][0][lane] = t.p12[R - 1];
		L.p[wv][1][lane] = t.p22[R - 1];
		__syncthreads();
	}
}

template <int R, int W, int K>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(4)))
void tv_iter_kernel(const float *__restrict__ I1wx, const float *__restrict__ I1wy,
                    const float *__restrict__ grad, const float *__restrict__ rho_c, TVPlanes A, TVPlanes B,
                    int nx, int ny, int stride, int tiles_x, float l_t, float theta, float taut,
                    double *__restrict__ part, float eps2, int *__restrict__ ctl, int *__restrict__ cur,
                    int *__restrict__ iters, int *__restrict__ mode, int *__restrict__ state,
                    int *__restrict__ n_active)
{
	constexpr int TX = 64 - 2 * K, TY = R * W - 2 * K;
	__shared__ TVEdge<W> L;
	__shared__ double red[W][K];
	const int pr = blockIdx.y;
	const int kk = ctl[pr];
	if (kk <= 0) return;
	const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const int tile = blockIdx.x, ntiles = gridDim.x;
	const int tx0 = (tile % tiles_x) * TX, ty0 = (tile / tiles_x) * TY;
	const bool flip = cur[pr] != 0;
	const size_t off = (size_t)pr * stride;
	auto planes = [&](bool b) {
		return b ? TVPlanes{B.u1 + off, B.u2 + off, B.p11 + off, B.p12 + off, B.p21 + off, B.p22 + off}
		         : TVPlanes{A.u1 + off, A.u2 + off, A.p11 + off, A.p12 + off, A.p21 + off, A.p22 + off};
	};
	const TVPlanes S = planes(flip), D = planes(!flip);
	const int x = tx0 - K + lane, yt = wv * R - K, y0 = ty0 + yt;
	const bool in = x >= 0 && x < nx;
	TVRows<R> t = {};
	// one byte offset a row for all planes (an image is below 4 GB)
	auto at = [](const float *p, unsigned o) { return *(const float *)((const char *)p + o); };
#pragma unroll
	for (int r = 0; r < R; r++) {
		if (y0 + r < 0 || y0 + r >= ny) continue;
		const unsigned o = 4u * (unsigned)((y0 + r) * nx + x);
		if (!in) continue;
		t.u1[r] = at(S.u1, o);
		t.u2[r] = at(S.u2, o);
		t.p11[r] = at(S.p11, o);
		t.p12[r] = at(S.p12, o);
		t.p21[r] = at(S.p21, o);
		t.p22[r] = at(S.p22, o);
		t.wx[r] = at(I1wx + off, o);
		t.wy[r] = at(I1wy + off, o);
		t.g[r] = at(grad + off, o);
		t.rc[r] = at(rho_c + off, o);
	}
#pragma unroll
	for (int r = 0; r < R; r++) {
		t.flat[r] = t.g[r] < TV_GRAD_IS_ZERO;
		t.yg[r] = tv_recip(t.g[r]);
		if (__any(!(t.g[r] < 0x1p126f))) t.yg[r] = 1.0 / (double)t.g[r];
	}
	L.p[wv][0][lane] = t.p12[R - 1];
	L.p[wv][1][lane] = t.p22[R - 1];
	double err[K];
#pragma unroll
	for (int j = 0; j < K; j++) err[j] = 0.0;
	__syncthreads();
	if (tx0 - K <= 0 || tx0 + TX + K >= nx)   // block-uniform
		tv_iterate<R, W, K, true>(t, L, wv, lane, x, y0, yt, nx, ny, kk, l_t, theta, taut, err);
	else
		tv_iterate<R, W, K, false>(t, L, wv, lane, x, y0, yt, nx, ny, kk, l_t, theta, taut, err);
	// the tile itself to the other buffer
	auto put = [](float *p, unsigned o, float v) { *(float *)((char *)p + o) = v; };
#pragma unroll
	for (int r = 0; r < R; r++) {
		if (yt + r < 0 || yt + r >= TY || y0 + r >= ny) continue;
		if (!in || lane < K || lane >= TX + K) continue;
		const unsigned o = 4u * (unsigned)((y0 + r) * nx + x);
		put(D.u1, o, t.u1[r]);
		put(D.u2, o, t.u2[r]);
		put(D.p11, o, t.p11[r]);
		put(D.p12, o, t.p12[r]);
		put(D.p21, o, t.p21[r]);
		put(D.p22, o, t.p22[r]);
	}
	// squared updates of the tile, per iteration
#pragma unroll
	for (int j = 0; j < K; j++) {
		double v = err[j];
#pragma unroll
		for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
		if (lane == 0) red[wv][j] = v;
	}
	__syncthreads();
	if (wv > 0) return;
	// The pair's last block to get here sums the tiles' partials and decides.
	// The partials go past the caches of this XCD and are out before the block
	// is counted (mode: the count above the bit); every block has read ctl and
	// cur by then.
	double *pp = part + (size_t)pr * K * ntiles;
	if (lane < kk) {
		double v = 0.0;
		for (int w = 0; w < W; w++) v += red[w][lane];
		__hip_atomic_store(pp + (size_t)lane * ntiles + tile, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	}
	asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
	int md = 0;
	if (lane == 0) md = __hip_atomic_fetch_add(mode + pr, TV_BLOCK, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	md = __builtin_amdgcn_readfirstlane(md);
	if (md / TV_BLOCK != ntiles - 1) return;
	// error of iteration j = (sum over the tiles' partials) / pixels: 256
	// strided sums (sum v: tiles v, v + 256, ...) held four to a lane, then a
	// tree over them (sum v += sum v + s for s = 128, 64, ..., 1)
	float errs[K];
#pragma unroll
	for (int j = 0; j < K; j++) {
		errs[j] = 0.f;
		if (j >= kk) continue;
		double v[4];
#pragma unroll
		for (int i = 0; i < 4; i++) {
			double e = 0.0;
			for (int t = lane + 64 * i; t < ntiles; t += 256)
				e += __hip_atomic_load(pp + (size_t)j * ntiles + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
			v[i] = e;
		}
		v[0] = v[0] + v[2];   // s = 128
		v[1] = v[1] + v[3];
		double x = v[0] + v[1];   // s = 64
#pragma unroll
		for (int st = 32; st > 0; st >>= 1) {
			const double o = __shfl_down(x, st, 64);
			if (lane < st) x = x + o;
		}
		errs[j] = (float)x / (float)stride;
	}
	if (lane == 0) tv_round_decide<K>(pr, kk, errs, eps2, md & TV_REDO, ctl, cur, iters, mode, state, n_active);
}

// Per pair: run state of the solve of one warp.
// The state stays in the buffer the last round wrote (cur) from one warp to
// the next; reset_cur at the start of a scale, where it is in the first.
__global__ void tv_round_init_kernel(int P, int K, int *__restrict__ ctl, int *__restrict__ cur,
                                     int *__restrict__ iters, int *__restrict__ mode, int *__restrict__ state,
                                     int *__restrict__ n_active, int reset_cur)
{
	const int pr = blockIdx.x * blockDim.x + threadIdx.x;
	if (pr == 0) *n_active = P;
	if (pr >= P) return;
	ctl[pr] = min(K, TV_MAX_ITERATIONS);
	if (reset_cur) cur[pr] = 0;
	iters[pr] = 0;
	mode[pr] = TV_RUN;
	state[pr] = -1;
}

// End of a scale: pairs whose flow is in the second buffer copy it to the
// first (the pyramid level the zoom and the output read).
__global__ void tv_settle_kernel(TVPlanes A, TVPlanes B, int n, int stride, const int *__restrict__ cur)
{
	const int pr = blockIdx.y;
	if (!cur[pr]) return;
	const size_t off = (size_t)pr * stride;
	for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
		A.u1[off + p] = B.u1[off + p];
		A.u2[off + p] = B.u2[off + p];
	}
}

__global__ void tv_fill_kernel(float *__restrict__ a, size_t n, float v)
{
	for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
		a[i] = v;
}

__global__ void tv_fill_int_kernel(int *__restrict__ a, int n, int v)
{
	for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) a[i] = v;
}

// Writes pair results into the sequence flow layout [F][2][H][W]:
// dst frame `frame` gets (u, v) of pair pr.
__global__ void tv_store_kernel(const float *__restrict__ u1, const float *__restrict__ u2, int size,
                                const int *__restrict__ dst_frame, float *__restrict__ flow)
{
	const int pr = blockIdx.y;
	const int f = dst_frame[pr];
	for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < size; p += gridDim.x * blockDim.x) {
		flow[(size_t)f * 2 * size + p] = u1[(size_t)pr * size + p];
		flow[(size_t)f * 2 * size + size + p] = u2[(size_t)pr * size + p];
	}
}

__global__ void tv_copy_frame_kernel(float *__restrict__ flow, int size, int from, int to)
{
	for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < 2 * size; p += gridDim.x * blockDim.x)
		flow[(size_t)to * 2 * size + p] = flow[(size_t)from * 2 * size + p];
}

} // namespace bm4dof

// ====================================================================== host

using namespace bm4dof;

// Scratch of bm4dof_tvl1_noalloc: one fixed region per GPU, part of the
// loaded code object, held until the process ends.  Host code never uses
// this name as an address: tv_scratch_init records, per device, the address
// hipGetSymbolAddress gives with that device current, and the entry point
// passes that address to the kernels.
static __device__ __align__(256) unsigned char scratch[BM4DOF_TVL1_NOALLOC_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices] = {};
} // namespace

// Called by bm4dof_ctx_create with `device` current.
void bm4dof::tv_scratch_init(int device)
{
	std::lock_guard<std::mutex> lk(g_scratch_mu);
	if (device < 0 || device >= kMaxDevices) throw ArgError("device index above the no-alloc scratch table");
	if (g_scratch_ptr[device]) return;
	void *ptr = nullptr;
	HIPCHK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
	g_scratch_ptr[device] = ptr;
}

namespace {

inline int tv_grid(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>((n + TV_THREADS - 1) / TV_THREADS, 4096)); }
inline int nblk_tv(int64_t n) { return (int)((n + TV_THREADS - 1) / TV_THREADS); }

// Normalised 1-D Gaussian taps (mask.c:227-249), computed on the host with
// the same libm calls as the reference.
int gauss_taps(double sigma, std::vector<double> &B)
{
	const double den = 2 * sigma * sigma;
	const int size = (int)(5 * sigma) + 1;
	B.assign(size, 0.0);
	for (int i = 0; i < size; i++) B[i] = 1 / (sigma * sqrt(2.0 * 3.1415926)) * exp(-i * i / den);
	double norm = 0;
	for (int i = 0; i < size; i++) norm += B[i];
	norm *= 2;
	norm -= B[0];
	for (int i = 0; i < size; i++) B[i] /= norm;
	return size;
}

struct TVPlan {
	int P = 0;                       // number of pairs
	int nscales = 0;
	std::vector<int> nx, ny;         // per scale
	std::vector<size_t> off;         // per-scale offset (floats) in a pyramid of P images
	size_t pyr = 0;                  // floats per pyramid
};

TVPlan tv_plan(int P, int nxx, int nyy, int nscales, float zfactor)
{
	TVPlan pl;
	pl.P = P;
	pl.nscales = nscales;
	pl.nx.resize(nscales);
	pl.ny.resize(nscales);
	pl.off.resize(nscales);
	pl.nx[0] = nxx;
	pl.ny[0] = nyy;
	for (int s = 1; s < nscales; s++) { // zoom_size, zoom.c:24-36
		pl.nx[s] = (int)((float)pl.nx[s - 1] * zfactor + 0.5);
		pl.ny[s] = (int)((float)pl.ny[s - 1] * zfactor + 0.5);
	}
	size_t o = 0;
	for (int s = 0; s < nscales; s++) {
		pl.off[s] = o;
		o += (size_t)P * pl.nx[s] * pl.ny[s];
	}
	pl.pyr = o;
	return pl;
}

// Gaussian smoothing of P images (in -> out, via tmp).
void tv_gauss(bm4dof_ctx *ctx, double *dB, const float *in, float *tmp, float *out, int nx, int ny, int P,
              double sigma)
{
	std::vector<double> B;
	const int size = gauss_taps(sigma, B);
	if (size > nx) throw ArgError("GaussianSmooth: sigma too large");
	if (size >= ny) throw ArgError("GaussianSmooth: sigma too large for the image height");
	if (size > 64) throw ArgError("GaussianSmooth: sigma too large");
	HIPCHK(hipMemcpyAsync(dB, B.data(), size * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
	const int n = nx * ny;
	hipLaunchKernelGGL(tv_gauss_kernel, dim3(tv_grid(n), P), dim3(TV_THREADS), 0, ctx->stream, in, tmp,
	                   nx, ny, n, dB, size, 1);
	hipLaunchKernelGGL(tv_gauss_kernel, dim3(tv_grid(n), P), dim3(TV_THREADS), 0, ctx->stream, tmp, out,
	                   nx, ny, n, dB, size, 0);
	HIPCHK(hipGetLastError());
	// the taps buffer is reused by the next call: keep ordering on the stream
	HIPCHK(hipStreamSynchronize(ctx->stream));
}

// Device memory of one multiscale solve of P pairs: pair indices, the four
// pyramids (I0, I1, u1, u2), 16 working planes at the finest size (12 of
// them the scheme's arrays, the last four with the two Gaussian temporaries
// the second state buffer of the iterations), min/max partials, the
// iterations' per-tile partial sums, the per-pair round control (ctl, cur,
// iters, mode, state, then the active count) and Gaussian taps.
struct TVScratch {
	int *pairs = nullptr;
	float *pyr = nullptr, *work = nullptr, *mm = nullptr;
	double *part = nullptr, *taps = nullptr;
	int *state = nullptr;
};
constexpr int TV_MMB = 64;      // blocks of the min/max reduction per pair
constexpr int TV_WORK = 16;     // working planes at the finest size

// Shapes of the iteration blocks (rows a thread, waves): 56 x 24 pixels, or
// 56 x 8 where those would be fewer than TV_SMALL_BLOCKS blocks over all pairs
// and not fill the CUs.  A pixel's arithmetic does not depend on the tile it
// is in.
struct TVShape { int r, w; int tx() const { return 64 - 2 * TV_K; } int ty() const { return r * w - 2 * TV_K; } };
constexpr TVShape TV_LARGE_TILE = {4, 8}, TV_SMALL_TILE = {2, 8};
#define TV_SMALL_BLOCKS 512
inline int tv_tiles(const TVShape &t, int nx, int ny) { return ((nx + t.tx() - 1) / t.tx()) * ((ny + t.ty() - 1) / t.ty()); }
inline const TVShape &tv_shape(int nx, int ny, int P)
{
	return (int64_t)tv_tiles(TV_LARGE_TILE, nx, ny) * P < TV_SMALL_BLOCKS ? TV_SMALL_TILE : TV_LARGE_TILE;
}
inline int tv_tiles_x(int nx, int ny, int P) { return (nx + tv_shape(nx, ny, P).tx() - 1) / tv_shape(nx, ny, P).tx(); }
inline int tv_tiles_at(int nx, int ny, int P) { return tv_tiles(tv_shape(nx, ny, P), nx, ny); }
// most tiles of any scale: the per-iteration partial sums per pair
inline int tv_part_tiles(const TVPlan &pl)
{
	int m = 0;
	for (int s = 0; s < pl.nscales; s++) m = std::max(m, tv_tiles_at(pl.nx[s], pl.ny[s], pl.P));
	return m;
}

// Partial sums that the account of the fixed scratch counts, which decides the
// pairs that fit it: one per 32 x 16 pixels, or per 64 x 32 where those are 1024
// or more.  (The sums' own number depends on the tiles; bm4dof_tvl1_noalloc
// keeps them elsewhere.)
inline int tv_account_tiles(const TVPlan &pl)
{
	int m = 0;
	for (int s = 0; s < pl.nscales; s++) {
		const int l = ((pl.nx[s] + 63) / 64) * ((pl.ny[s] + 31) / 32);
		m = std::max(m, l >= 1024 ? l : ((pl.nx[s] + 31) / 32) * ((pl.ny[s] + 15) / 16));
	}
	return m;
}

// Byte offsets of the parts of a TVScratch carved from one region, and the
// region's size (the last entry), each part 256-byte aligned.
std::array<size_t, 8> tv_scratch_layout(const TVPlan &pl, size_t size0)
{
	auto al = [](size_t b) { return (b + 255) / 256 * 256; };
	const size_t P = (size_t)pl.P;
	std::array<size_t, 8> o{};
	o[0] = 0;                                                          // pairs
	o[1] = o[0] + al(2 * P * sizeof(int));                             // pyramids
	o[2] = o[1] + al(pl.pyr * 4 * sizeof(float));                      // working planes
	o[3] = o[2] + al(P * size0 * TV_WORK * sizeof(float));             // min/max
	o[4] = o[3] + al(P * TV_MMB * 4 * sizeof(float));                  // iteration partial sums
	o[5] = o[4] + al(P * TV_K * (size_t)tv_account_tiles(pl) * sizeof(double));
	o[6] = o[5] + al((5 * P + 1) * sizeof(int));                       // taps
	o[7] = o[6] + al(64 * sizeof(double));                             // total
	return o;
}

TVScratch tv_scratch_carve(char *base, const std::array<size_t, 8> &o)
{
	TVScratch t;
	t.pairs = (int *)(base + o[0]);
	t.pyr = (float *)(base + o[1]);
	t.work = (float *)(base + o[2]);
	t.mm = (float *)(base + o[3]);
	t.part = (double *)(base + o[4]);
	t.state = (int *)(base + o[5]);
	t.taps = (double *)(base + o[6]);
	return t;
}

TVScratch tv_scratch_ctx(bm4dof_ctx *ctx, const TVPlan &pl, size_t size0)
{
	const size_t P = (size_t)pl.P;
	TVScratch t;
	t.pairs = ctx->tv_pairs.as<int>(2 * P);
	t.pyr = ctx->tv_pyr.as<float>(pl.pyr * 4);
	t.work = ctx->tv_work.as<float>(P * size0 * TV_WORK);
	t.mm = ctx->tv_mm.as<float>(P * TV_MMB * 4);
	t.part = ctx->tv_part.as<double>(P * TV_K * (size_t)tv_part_tiles(pl));
	t.state = ctx->tv_state.as<int>(5 * P + 1);
	t.taps = ctx->tv_taps.as<double>(64);
	return t;
}

void tv_check_params(const bm4dof_tvl1_params &prm)
{
	if (prm.nscales < 1 || prm.warps < 0 || prm.fscale < 0 || !(prm.zfactor > 0 && prm.zfactor < 1))
		throw ArgError("invalid TV-L1 parameters");
}

// Multiscale TV-L1 of P pairs.  frames: device, nfr frames of nxx*nyy;
// pair pr uses frames i0[pr] -> i1[pr].  Result in u1/u2 (P*nxx*nyy each,
// device).  iters (host, may be NULL): P*nscales*warps ints.  Device
// scratch from `fixed` when given (nothing is allocated then), else from the
// context's buffers.
void tv_flow_pairs(bm4dof_ctx *ctx, const bm4dof_tvl1_params &prm, const float *frames, int nxx,
                   int nyy, const std::vector<int> &i0, const std::vector<int> &i1, float *u1out,
                   float *u2out, int *iters, const TVScratch *fixed = nullptr)
{
	const int P = (int)i0.size();
	if (P == 0) return;
	tv_check_params(prm);
	const int nscales = prm.nscales;
	TVPlan pl = tv_plan(P, nxx, nyy, nscales, prm.zfactor);
	ctx->tv_pixel_iters = 0;
	for (int s = 0; s < nscales; s++)
		if (pl.nx[s] < 3 || pl.ny[s] < 3)
			throw ArgError("TV-L1 pyramid level " + std::to_string(s) + " is smaller than 3x3; lower nscales");
	const size_t size0 = (size_t)nxx * nyy;
	hipStream_t st = ctx->stream;

	const TVScratch sc = fixed ? *fixed : tv_scratch_ctx(ctx, pl, size0);
	int *d_pairs = sc.pairs;
	HIPCHK(hipMemcpyAsync(d_pairs, i0.data(), P * sizeof(int), hipMemcpyHostToDevice, st));
	HIPCHK(hipMemcpyAsync(d_pairs + P, i1.data(), P * sizeof(int), hipMemcpyHostToDevice, st));
	// pyramids: I0s, I1s, u1s, u2s
	float *pyr = sc.pyr;
	float *I0s = pyr, *I1s = pyr + pl.pyr, *U1 = pyr + 2 * pl.pyr, *U2 = pyr + 3 * pl.pyr;
	// working arrays at the finest size: tmp, tmp2, I1x, I1y, I1wx, I1wy, grad, rho_c, p11..p22,
	// and four planes that with tmp and tmp2 hold the iterations' second state buffer
	const size_t W = (size_t)P * size0;
	float *work = sc.work;
	float *tmp = work, *tmp2 = work + W, *I1x = work + 2 * W, *I1y = work + 3 * W,
	      *I1wx = work + 4 * W, *I1wy = work + 5 * W, *grad = work + 6 * W, *rho_c = work + 7 * W,
	      *p11 = work + 8 * W, *p12 = work + 9 * W, *p21 = work + 10 * W, *p22 = work + 11 * W;
	const int mmb = TV_MMB;
	float *d_mm = sc.mm;
	double *d_part = sc.part;
	int *d_ctl = sc.state, *d_cur = d_ctl + P, *d_iters = d_cur + P, *d_mode = d_iters + P, *d_state = d_mode + P;
	int *d_nact = d_state + P;

	// normalisation + presmoothing (tvl1flow_lib.c:381-386)
	hipLaunchKernelGGL(tv_minmax_kernel, dim3(mmb, P), dim3(TV_THREADS), 0, st, frames, (int)size0,
	                   d_pairs, d_pairs + P, d_mm);
	hipLaunchKernelGGL(tv_normalize_kernel, dim3(tv_grid(size0), P), dim3(TV_THREADS), 0, st, frames,
	                   (int)size0, d_pairs, d_pairs + P, d_mm, mmb, tmp2, tmp2 + W);
	HIPCHK(hipGetLastError());
	tv_gauss(ctx, sc.taps, tmp2, tmp, I0s + pl.off[0], nxx, nyy, P, TV_PRESMOOTHING_SIGMA);
	tv_gauss(ctx, sc.taps, tmp2 + W, tmp, I1s + pl.off[0], nxx, nyy, P, TV_PRESMOOTHING_SIGMA);
	// pyramid (tvl1flow_lib.c:389-403; zoom_out, zoom.c:43-79)
	const float zsig = TV_ZOOM_SIGMA_ZERO * sqrt(1.0 / (prm.zfactor * prm.zfactor) - 1.0);
	for (int s = 1; s < nscales; s++) {
		const int nx = pl.nx[s - 1], ny = pl.ny[s - 1], n = nx * ny;
		for (int im = 0; im < 2; im++) {
			float *src = (im ? I1s : I0s) + pl.off[s - 1];
			float *dst = (im ? I1s : I0s) + pl.off[s];
			tv_gauss(ctx, sc.taps, src, tmp, tmp2, nx, ny, P, zsig);
			hipLaunchKernelGGL(tv_zoom_out_kernel, dim3(tv_grid(pl.nx[s] * pl.ny[s]), P), dim3(TV_THREADS), 0,
			                   st, tmp2, nx, ny, n, dst, pl.nx[s], pl.ny[s], pl.nx[s] * pl.ny[s], prm.zfactor);
			HIPCHK(hipGetLastError());
		}
	}
	{
		const int s = nscales - 1;
		const size_t n = (size_t)P * pl.nx[s] * pl.ny[s];
		hipLaunchKernelGGL(tv_fill_kernel, dim3(tv_grid(n)), dim3(TV_THREADS), 0, st, U1 + pl.off[s], n, 0.f);
		hipLaunchKernelGGL(tv_fill_kernel, dim3(tv_grid(n)), dim3(TV_THREADS), 0, st, U2 + pl.off[s], n, 0.f);
	}
	if (iters) std::fill(iters, iters + (size_t)P * nscales * prm.warps, -1);
	const float l_t = prm.lambda * prm.theta;
	const float taut = prm.tau / prm.theta;
	const float eps2 = prm.epsilon * prm.epsilon;
	const float scale = (float)1.0 / prm.zfactor;
	std::vector<int> h_state(P);
	// Rounds of TV_K iterations run until the pair's test stops them; the
	// host reads the active count after a batch of rounds: the first batch
	// long enough for the previous warp's iteration count, then two rounds
	// at a time (a round of a finished pair is a launch whose blocks exit).
	// With the pinned words, a poll copies the count and the GPU runs one
	// more round while the host waits for the copy, and a warp's iteration
	// counts are copied at its end and read at the next poll.
	const int max_rounds = TV_MAX_ITERATIONS + 1;
	int guess = 0;   // most iterations of a pair in the last warp read back
	const bool piped = ctx->tv_pin && P <= ctx->tv_pin_pairs;
	int pend_s = -1, pend_w = -1, pend_slot = 0, nwarp = 0;
	size_t pend_n = 0;
	auto take_counts = [&](const int *hs, int s, int w, size_t n) {
		guess = 0;
		for (int pr = 0; pr < P; pr++) {
			ctx->tv_pixel_iters += (uint64_t)std::max(hs[pr], 0) * (uint64_t)n;
			guess = std::max(guess, hs[pr]);
		}
		if (iters)
			for (int pr = 0; pr < P; pr++) iters[((size_t)pr * nscales + s) * prm.warps + w] = hs[pr];
		if (prm.verbose)
			for (int pr = 0; pr < P; pr++)
				fprintf(stderr, "Pair %d scale %d warping %d: iterations %d\n", pr, s, w, hs[pr]);
	};
	// the counts of a warp whose copy a completed poll has passed
	auto take_pending = [&]() {
		if (pend_w < 0) return;
		take_counts(ctx->tv_pin + 1 + (size_t)pend_slot * P, pend_s, pend_w, pend_n);
		pend_w = -1;
	};

	for (int s = nscales - 1; s >= prm.fscale; s--) {
		// Dual_TVL1_optic_flow, tvl1flow_lib.c:93-275
		const int nx = pl.nx[s], ny = pl.ny[s], n = nx * ny;
		float *u1 = U1 + pl.off[s], *u2 = U2 + pl.off[s];
		const float *I0 = I0s + pl.off[s], *I1 = I1s + pl.off[s];
		const int g = tv_grid(n);
		const TVPlanes SA = {u1, u2, p11, p12, p21, p22};
		const TVPlanes SB = {tmp, tmp2, work + 12 * W, work + 13 * W, work + 14 * W, work + 15 * W};
		const TVShape &shape = tv_shape(nx, ny, P);
		const auto kern = shape.r == TV_LARGE_TILE.r ? tv_iter_kernel<TV_LARGE_TILE.r, TV_LARGE_TILE.w, TV_K>
		                                             : tv_iter_kernel<TV_SMALL_TILE.r, TV_SMALL_TILE.w, TV_K>;
		const int tiles_x = tv_tiles_x(nx, ny, P), ntiles = tv_tiles_at(nx, ny, P);
		auto launch_round = [&]() {
			hipLaunchKernelGGL(kern, dim3(ntiles, P), dim3(64 * shape.w), 0, st, I1wx, I1wy, grad, rho_c, SA, SB, nx, ny, n,
			                   tiles_x, l_t, prm.theta, taut, d_part, eps2, d_ctl, d_cur, d_iters, d_mode, d_state, d_nact);
		};
		hipLaunchKernelGGL(tv_cgrad_kernel, dim3(g, P), dim3(TV_THREADS), 0, st, I1, nx, ny, n, I1x, I1y);
		const size_t nP = (size_t)P * n;
		for (float *q : {p11, p12, p21, p22})
			hipLaunchKernelGGL(tv_fill_kernel, dim3(tv_grid(nP)), dim3(TV_THREADS), 0, st, q, nP, 0.f);
		for (int w = 0; w < prm.warps; w++, nwarp++) {
			hipLaunchKernelGGL(tv_round_init_kernel, dim3(nblk_tv(P)), dim3(TV_THREADS), 0, st, P, TV_K, d_ctl,
			                   d_cur, d_iters, d_mode, d_state, d_nact, w == 0 ? 1 : 0);
			hipLaunchKernelGGL(tv_warp_kernel, dim3(g, P), dim3(TV_THREADS), 0, st, I0, I1, I1x, I1y, SA.u1, SA.u2,
			                   SB.u1, SB.u2, d_cur, nx, ny, n, I1wx, I1wy, grad, rho_c);
			HIPCHK(hipGetLastError());
			int batch = guess > 0 ? (guess + TV_K - 1) / TV_K : 3;
			for (int r = 0; r < max_rounds;) {
				const int rb = std::min(batch, max_rounds - r);
				for (int i = 0; i < rb; i++) launch_round();
				r += rb;
				HIPCHK(hipGetLastError());
				int nact = 0;
				if (piped) {
					HIPCHK(hipMemcpyAsync(ctx->tv_pin, d_nact, sizeof(int), hipMemcpyDeviceToHost, st));
					HIPCHK(hipEventRecord(ctx->ev_tvpoll, st));
					if (r < max_rounds) {   // runs while the host waits; a no-op once every pair stopped
						launch_round();
						r++;
					}
					HIPCHK(hipGetLastError());
					HIPCHK(hipEventSynchronize(ctx->ev_tvpoll));
					nact = ctx->tv_pin[0];
					take_pending();
				} else {
					HIPCHK(hipMemcpyAsync(&nact, d_nact, sizeof(int), hipMemcpyDeviceToHost, st));
					HIPCHK(hipStreamSynchronize(st));
				}
				if (nact == 0) break;
				batch = 2;
			}
			if (piped) {
				pend_slot = nwarp & 1;
				HIPCHK(hipMemcpyAsync(ctx->tv_pin + 1 + (size_t)pend_slot * P, d_state, P * sizeof(int),
				                      hipMemcpyDeviceToHost, st));
				pend_s = s;
				pend_w = w;
				pend_n = (size_t)n;
			} else {
				HIPCHK(hipMemcpyAsync(h_state.data(), d_state, P * sizeof(int), hipMemcpyDeviceToHost, st));
				HIPCHK(hipStreamSynchronize(st));
				take_counts(h_state.data(), s, w, (size_t)n);
			}
		}
		// the flow of every pair into the pyramid level
		if (prm.warps > 0)
			hipLaunchKernelGGL(tv_settle_kernel, dim3(g, P), dim3(TV_THREADS), 0, st, SA, SB, n, n, d_cur);
		HIPCHK(hipGetLastError());
		if (!s) break;
		hipLaunchKernelGGL(tv_zoom_in_kernel, dim3(tv_grid(pl.nx[s - 1] * pl.ny[s - 1]), P), dim3(TV_THREADS), 0, st,
		                   u1, nx, ny, n, U1 + pl.off[s - 1], pl.nx[s - 1], pl.ny[s - 1], pl.nx[s - 1] * pl.ny[s - 1], scale);
		hipLaunchKernelGGL(tv_zoom_in_kernel, dim3(tv_grid(pl.nx[s - 1] * pl.ny[s - 1]), P), dim3(TV_THREADS), 0, st,
		                   u2, nx, ny, n, U2 + pl.off[s - 1], pl.nx[s - 1], pl.ny[s - 1], pl.nx[s - 1] * pl.ny[s - 1], scale);
		HIPCHK(hipGetLastError());
	}
	for (int s = prm.fscale - 1; s >= 0; s--) { // tvl1flow_lib.c:438-455
		if (!s) break;
		const int n = pl.nx[s] * pl.ny[s], nn = pl.nx[s - 1] * pl.ny[s - 1];
		hipLaunchKernelGGL(tv_zoom_in_kernel, dim3(tv_grid(nn), P), dim3(TV_THREADS), 0, st, U1 + pl.off[s],
		                   pl.nx[s], pl.ny[s], n, U1 + pl.off[s - 1], pl.nx[s - 1], pl.ny[s - 1], nn, scale);
		hipLaunchKernelGGL(tv_zoom_in_kernel, dim3(tv_grid(nn), P), dim3(TV_THREADS), 0, st, U2 + pl.off[s],
		                   pl.nx[s], pl.ny[s], n, U2 + pl.off[s - 1], pl.nx[s - 1], pl.ny[s - 1], nn, scale);
		HIPCHK(hipGetLastError());
	}
	HIPCHK(hipMemcpyAsync(u1out, U1 + pl.off[0], (size_t)P * size0 * sizeof(float), hipMemcpyDeviceToDevice, st));
	HIPCHK(hipMemcpyAsync(u2out, U2 + pl.off[0], (size_t)P * size0 * sizeof(float), hipMemcpyDeviceToDevice, st));
	HIPCHK(hipStreamSynchronize(st));
	take_pending();
}

bm4dof_ctx *g_tv_ctx = nullptr;

} // namespace

extern "C" {

__attribute__((visibility("default")))
int bm4dof_tvl1(bm4dof_ctx *ctx, const bm4dof_tvl1_params *prm, const float *I0, const float *I1,
                float *u1, float *u2, int nx, int ny, int on_device, int *iters)
{
	if (!ctx || !prm || !I0 || !I1 || !u1 || !u2) { set_error(ctx, "NULL argument"); return BM4DOF_EINVAL; }
	return guarded(ctx, [&] {
		HIPCHK(hipSetDevice(ctx->device));
		if (nx < 3 || ny < 3) throw ArgError("image smaller than 3x3");
		const size_t n = (size_t)nx * ny;
		float *fr = ctx->tv_frames.as<float>(4 * n);
		float *du1 = fr + 2 * n, *du2 = fr + 3 * n;
		const hipMemcpyKind k = on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice;
		HIPCHK(hipMemcpyAsync(fr, I0, n * 4, k, ctx->stream));
		HIPCHK(hipMemcpyAsync(fr + n, I1, n * 4, k, ctx->stream));
		tv_flow_pairs(ctx, *prm, fr, nx, ny, {0}, {1}, du1, du2, iters);
		const hipMemcpyKind kb = on_device ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost;
		HIPCHK(hipMemcpyAsync(u1, du1, n * 4, kb, ctx->stream));
		HIPCHK(hipMemcpyAsync(u2, du2, n * 4, kb, ctx->stream));
		HIPCHK(hipStreamSynchronize(ctx->stream));
	});
}

__attribute__((visibility("default")))
int bm4dof_tvl1_noalloc(bm4dof_ctx *ctx, const bm4dof_tvl1_params *prm, const float *I0, const float *I1,
                        float *u1, float *u2, int nx, int ny, int *iters)
{
	if (!ctx || !prm || !I0 || !I1 || !u1 || !u2) { set_error(ctx, "NULL argument"); return BM4DOF_EINVAL; }
	return guarded(ctx, [&] {
		HIPCHK(hipSetDevice(ctx->device));
		if (nx < 3 || ny < 3) throw ArgError("image smaller than 3x3");
		tv_check_params(*prm);
		void *base = nullptr;
		{
			std::lock_guard<std::mutex> lk(g_scratch_mu);
			if (ctx->device >= 0 && ctx->device < kMaxDevices) base = g_scratch_ptr[ctx->device];
		}
		if (!base) throw ArgError("bm4dof_tvl1_noalloc: no scratch address recorded for this device");
		const size_t n = (size_t)nx * ny;
		const TVPlan pl = tv_plan(1, nx, ny, prm->nscales, prm->zfactor);
		const std::array<size_t, 8> lay = tv_scratch_layout(pl, n);
		const size_t need = lay[7] + (2 * n * sizeof(float) + 255) / 256 * 256;
		if (need > (size_t)BM4DOF_TVL1_NOALLOC_BYTES)
			throw ArgError("bm4dof_tvl1_noalloc: a " + std::to_string(nx) + "x" + std::to_string(ny) +
			               " pair with these parameters needs " + std::to_string(need) +
			               " bytes of scratch; the fixed scratch holds " +
			               std::to_string((size_t)BM4DOF_TVL1_NOALLOC_BYTES));
		char *b = (char *)base;
		TVScratch t = tv_scratch_carve(b, lay);
		float *fr = (float *)(b + lay[7]);
		// the partial sums over the frames, which nothing reads after their
		// normalisation (32 bytes a tile of at least 56 x 8 pixels, or of the
		// pair where it is smaller; 8 bytes a pixel of at least 9)
		t.part = (double *)fr;
		HIPCHK(hipMemcpyAsync(fr, I0, n * 4, hipMemcpyDeviceToDevice, ctx->stream));
		HIPCHK(hipMemcpyAsync(fr + n, I1, n * 4, hipMemcpyDeviceToDevice, ctx->stream));
		tv_flow_pairs(ctx, *prm, fr, nx, ny, {0}, {1}, u1, u2, iters, &t);
	});
}

__attribute__((visibility("default")))
int bm4dof_tvl1_sequence(bm4dof_ctx *ctx, const bm4dof_tvl1_params *prm, const float *frames, int nx,
                         int ny, int F, float *fflow, float *bflow, int on_device)
{
	if (!ctx || !prm || !frames || !fflow || !bflow) { set_error(ctx, "NULL argument"); return BM4DOF_EINVAL; }
	return guarded(ctx, [&] {
		HIPCHK(hipSetDevice(ctx->device));
		if (F < 1 || nx < 3 || ny < 3) throw ArgError("empty sequence or frames smaller than 3x3");
		const size_t n = (size_t)nx * ny;
		float *fr = ctx->tv_frames.as<float>(n * F + (size_t)4 * n * F);
		float *ff = fr + n * F, *bf = ff + 2 * n * F;
		hipStream_t st = ctx->stream;
		HIPCHK(hipMemcpyAsync(fr, frames, n * F * 4, on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, st));
		HIPCHK(hipMemsetAsync(ff, 0, 4 * n * F * 4, st));
		if (F > 1) {
			// scripts/tvl1flow-seq.sh:31-61: bwd(i) = I_i -> I_{i-1}, fwd(i) = I_i -> I_{i+1}
			std::vector<int> i0, i1, dst;
			for (int i = 1; i < F; i++) { i0.push_back(i); i1.push_back(i - 1); dst.push_back(i); }
			for (int i = 0; i < F - 1; i++) { i0.push_back(i); i1.push_back(i + 1); dst.push_back(i); }
			const int P = (int)i0.size();
			DevBuf ub;
			float *u = ub.as<float>((size_t)2 * P * n);
			tv_flow_pairs(ctx, *prm, fr, nx, ny, i0, i1, u, u + (size_t)P * n, nullptr);
			int *d_dst = ctx->tv_pairs.as<int>(P);
			HIPCHK(hipMemcpyAsync(d_dst, dst.data(), P * sizeof(int), hipMemcpyHostToDevice, st));
			const int half = F - 1;
			hipLaunchKernelGGL(tv_store_kernel, dim3(tv_grid(n), half), dim3(TV_THREADS), 0, st, u,
			                   u + (size_t)P * n, (int)n, d_dst, bf);
			hipLaunchKernelGGL(tv_store_kernel, dim3(tv_grid(n), half), dim3(TV_THREADS), 0, st, u + half * n,
			                   u + (size_t)P * n + half * n, (int)n, d_dst + half, ff);
			hipLaunchKernelGGL(tv_copy_frame_kernel, dim3(tv_grid(2 * n)), dim3(TV_THREADS), 0, st, bf, (int)n, 1, 0);
			hipLaunchKernelGGL(tv_copy_frame_kernel, dim3(tv_grid(2 * n)), dim3(TV_THREADS), 0, st, ff, (int)n, F - 2, F - 1);
			HIPCHK(hipGetLastError());
			HIPCHK(hipStreamSynchronize(st));
			ub.release();
		}
		const hipMemcpyKind kb = on_device ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost;
		HIPCHK(hipMemcpyAsync(fflow, ff, 2 * n * F * 4, kb, st));
		HIPCHK(hipMemcpyAsync(bflow, bf, 2 * n * F * 4, kb, st));
		HIPCHK(hipStreamSynchronize(st));
	});
}

__attribute__((visibility("default")))
void Dual_TVL1_optic_flow_multiscale(float *I0, float *I1, float *u1, float *u2, int nxx, int nyy,
                                     float tau, float lambda, float theta, int nscales, int fscale,
                                     float zfactor, int warps, float epsilon, bool verbose)
{
	if (!g_tv_ctx && bm4dof_ctx_create(&g_tv_ctx, 0) != BM4DOF_OK) {
		fprintf(stderr, "Dual_TVL1_optic_flow_multiscale: %s\n", bm4dof_global_error());
		abort();
	}
	bm4dof_tvl1_params prm = {tau, lambda, theta, nscales, fscale, zfactor, warps, epsilon, verbose ? 1 : 0};
	if (bm4dof_tvl1(g_tv_ctx, &prm, I0, I1, u1, u2, nxx, nyy, 0, nullptr) != BM4DOF_OK) {
		fprintf(stderr, "Dual_TVL1_optic_flow_multiscale: %s\n", bm4dof_last_error(g_tv_ctx));
		abort();
	}
}

} // extern "C"
