// Learned gain network: training (forward, backward, Adam) and standalone
// inference.  No counterpart in the reference: the network predicts, from
// the step-1 Haar-domain coefficients of one group row, the step-2 Wiener
// gains y^2 / (y^2 + (beta sigma)^2) (src/core/nldct.cpp:2131) so that one
// pass replaces the two steps.
//
// Parameters: a flat float32 master vector theta (W1 [66][128], b1, W2
// [128][128], b2, W3 [128][64], b3; W[k][j] input-major), Adam moments m, v,
// and two derived copies refreshed after every update:
//   * wq: W1..W3 rounded to bf16 (as float), used by the training forward;
//   * the inference blob: bf16 W1..W3 transposed for the matrix cores, and
//     the float32 biases.
// Training forward rounds the layer inputs to bf16 exactly as the matrix
// cores consume them; backward is straight-through (rounding has slope 1).
// A training step is three launches (mlp_rows_kernel, mlp_wgrad_kernel,
// mlp_update_kernel), its products on the fp32 matrix instructions; inference
// runs on the bf16 ones (mlp_dev.hpp).
#include "common.hpp"
#include "ctx.hpp"
#include "mlp_dev.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

namespace bm4dof {

// offsets in theta
constexpr int OW1 = 0, OB1 = OW1 + MLP_IN * MLP_H, OW2 = OB1 + MLP_H, OB2 = OW2 + MLP_H * MLP_H,
              OW3 = OB2 + MLP_H, OB3 = OW3 + MLP_H * MLP_OUT;
static_assert(OB3 + MLP_OUT == MLP_NPARAMS, "parameter layout");
static_assert(MLP_NPARAMS == BM4DOF_MLP_NPARAMS, "parameter count");
// inference blob (uint16 units), biases after it as float32
constexpr size_t IW1 = 0, IW2 = IW1 + (size_t)MLP_H * MLP_K1, IW3 = IW2 + (size_t)MLP_H * MLP_H,
                 IWEND = IW3 + (size_t)MLP_OUT * MLP_H;
constexpr size_t IB_BYTES = ((IWEND * 2 + 255) / 256) * 256;   // bias area offset (bytes)
constexpr size_t INF_BYTES = IB_BYTES + (size_t)(MLP_H + MLP_H + MLP_OUT) * 4;

MlpInfer mlp_infer_view(const void *blob)
{
	MlpInfer n;
	const uint16_t *w = (const uint16_t *)blob;
	const float *b = (const float *)((const char *)blob + IB_BYTES);
	n.w1t = w + IW1;
	n.w2t = w + IW2;
	n.w3t = w + IW3;
	n.b1 = b;
	n.b2 = b + MLP_H;
	n.b3 = b + 2 * MLP_H;
	return n;
}

__device__ __forceinline__ float bf16r(float f) { return bf16_to_f32(f32_to_bf16(f)); }

// theta -> rounded training copies (wq, same layout as theta's weights) and
// the inference blob.
__global__ void mlp_pack_kernel(const float *__restrict__ theta, float *__restrict__ wq,
                                uint16_t *__restrict__ blob, float *__restrict__ bias)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < MLP_NPARAMS) {
		const bool is_bias = (i >= OB1 && i < OW2) || (i >= OB2 && i < OW3) || i >= OB3;
		wq[i] = is_bias ? theta[i] : bf16r(theta[i]);
	}
	if (i < (int)IWEND) {
		float v = 0.f;
		if (i < (int)IW2) {
			const int j = i / MLP_K1, k = i - j * MLP_K1;
			v = k < MLP_IN ? theta[OW1 + k * MLP_H + j] : 0.f;
		} else if (i < (int)IW3) {
			const int r = i - (int)IW2, j = r / MLP_H, k = r - j * MLP_H;
			v = theta[OW2 + k * MLP_H + j];
		} else {
			const int r = i - (int)IW3, j = r / MLP_H, k = r - j * MLP_H;
			v = theta[OW3 + k * MLP_OUT + j];
		}
		blob[i] = f32_to_bf16(v);
	}
	if (i < MLP_H) bias[i] = theta[OB1 + i];
	if (i < MLP_H) bias[MLP_H + i] = theta[OB2 + i];
	if (i < MLP_OUT) bias[2 * MLP_H + i] = theta[OB3 + i];
}

// ---------------------------------------------------------------------------
// Training step.  Products run on v_mfma_f32_16x16x4_f32 (fp32 in, fp32
// accumulation).  Lane l of a wave, g = l / 16, j = l % 16:
//   A (16 x 4): A[j][g]; B (4 x 16): B[g][j]; D (16 x 16): D[4 g + i][j], i < 4
// Four of them take 16 terms of a sum: instruction v multiplies the terms
// 4 g + v of every lane group, so a lane's four operands are one float4.
//
// Before, a step was 23 launches, and 2.8 of its 3.46 ms (batch 4096) went
// into three column sums of one block each; the products were 16 x 16 tiles
// through LDS (78 us each).  Now the batch's rows are independent up to the
// weight gradients: one launch takes 16 rows through both directions, one
// forms the weight gradients with the rows split over waves, one sums the
// splits and updates.
// ---------------------------------------------------------------------------

typedef float mlp_f32x4 __attribute__((ext_vector_type(4)));

constexpr int TR_R = 16;                        // rows of a block
constexpr int TR_KC = 128;                      // rows of a weight-gradient split, at least
constexpr int TR_SMAX = 64;                     // splits, at most
// per row in the workspace, feature-major [feature][row]: layer inputs
// (rounded), then the gradients at the layers' outputs
constexpr int TX = 0, TH1 = TX + MLP_IN, TH2 = TH1 + MLP_H, TD1 = TH2 + MLP_H, TD2 = TD1 + MLP_H,
              TD3 = TD2 + MLP_H, TEND = TD3 + MLP_OUT;
constexpr int TR_XS = 84, TR_HS = 132, TR_OS = 68;   // LDS row strides (floats)

__device__ __forceinline__ mlp_f32x4 mfma4(const float4 &a, const float4 &b, mlp_f32x4 c)
{
	c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, c, 0, 0, 0);
	c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, c, 0, 0, 0);
	c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, c, 0, 0, 0);
	c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, c, 0, 0, 0);
	return c;
}
__device__ __forceinline__ float4 bf16x4(const uint16_t *p)
{
	const uint2 v = *reinterpret_cast<const uint2 *>(p);
	return make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
	                   __uint_as_float(v.y & 0xffff0000u));
}

// Row of the data set that row r of a batch takes: the whole set in order,
// else one named by a hash of (seed, row).
__device__ __forceinline__ int64_t batch_row(int r, int B, int64_t nrows, uint32_t seed)
{
	if ((int64_t)B == nrows) return r;
	uint64_t s = ((uint64_t)seed << 32) ^ (uint64_t)(r * 2654435761u + 0x9E3779B9u);
	s = s * 6364136223846793005ull + 1442695040888963407ull;
	s ^= s >> 33;
	s *= 0xff51afd7ed558ccdull;
	s ^= s >> 33;
	return (int64_t)(s % (uint64_t)nrows);
}

// Both directions for 16 rows of the batch: the layer inputs and the
// gradients at the layers' outputs into ws (stride Bp, the rows past B zero),
// the block's squared error into sse[block].  Four waves, each a quarter of
// every layer's outputs; activations in LDS, weights from L2 (forward from
// the bf16 copy, whose inputs are contiguous, backward from the rounded
// master, whose outputs are).
// Bound: latency of the five dependent layers.  Batch 4096 (256 blocks): 24
// us, where the products of both directions, rounding, masks and gather were
// 390 us in 17 launches.
__global__ __launch_bounds__(256)
void mlp_rows_kernel(const float *__restrict__ X, const float *__restrict__ T, int64_t nrows, int B, uint32_t seed,
                     MlpInfer net, const float *__restrict__ wq, int Bp, float *__restrict__ ws,
                     double *__restrict__ sse)
{
	__shared__ __align__(16) float xs[TR_R * TR_XS], h1[TR_R * TR_HS], h2[TR_R * TR_HS], d3[TR_R * TR_OS],
	    ts[TR_R * MLP_OUT];
	__shared__ double part[4];
	__shared__ int64_t src[TR_R];   // the rows' places in the data set, -1 past the batch
	const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63, g = l >> 4, j = l & 15;
	const int r0 = blockIdx.x * TR_R;
	if (tid < TR_R) src[tid] = r0 + tid < B ? batch_row(r0 + tid, B, nrows, seed) : -1;
	__syncthreads();
#pragma unroll
	for (int u = 0; u < (TR_R * TR_XS + 255) / 256; u++) {
		const int i = tid + 256 * u, r = i / TR_XS, k = i - r * TR_XS;
		if (i < TR_R * TR_XS) xs[i] = src[r] >= 0 && k < MLP_IN ? bf16r(X[(size_t)src[r] * MLP_IN + k]) : 0.f;
	}
#pragma unroll
	for (int u = 0; u < TR_R * MLP_OUT / 256; u++) {
		const int i = tid + 256 * u, r = i / MLP_OUT, k = i - r * MLP_OUT;
		ts[i] = src[r] >= 0 ? T[(size_t)src[r] * MLP_OUT + k] : 0.f;
	}
	__syncthreads();
	for (int i = tid; i < MLP_IN * TR_R; i += 256) {
		const int k = i / TR_R, r = i - k * TR_R;
		ws[(size_t)(TX + k) * Bp + r0 + r] = xs[r * TR_XS + k];
	}
	// layer 1: outputs 32 wv + 16 t + j
	float z1[2][4], z2[2][4];
#pragma unroll
	for (int t = 0; t < 2; t++) {
		const int n = 32 * wv + 16 * t + j;
		mlp_f32x4 c = {};
		float4 w[5];
#pragma unroll
		for (int q = 0; q < 5; q++)   // inputs 72.. are not stored
			w[q] = q < 4 || g < 2 ? bf16x4(net.w1t + n * MLP_K1 + 16 * q + 4 * g) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
		for (int q = 0; q < 5; q++) c = mfma4(*reinterpret_cast<const float4 *>(xs + j * TR_XS + 16 * q + 4 * g), w[q], c);
		const float bias = wq[OB1 + n];
#pragma unroll
		for (int i = 0; i < 4; i++) {
			z1[t][i] = c[i] + bias;
			h1[(4 * g + i) * TR_HS + n] = r0 + 4 * g + i < B ? bf16r(fmaxf(z1[t][i], 0.f)) : 0.f;
		}
	}
	__syncthreads();
	// layer 2
#pragma unroll
	for (int t = 0; t < 2; t++) {
		const int n = 32 * wv + 16 * t + j;
		mlp_f32x4 c = {};
		float4 w[8];
#pragma unroll
		for (int q = 0; q < 8; q++) w[q] = bf16x4(net.w2t + n * MLP_H + 16 * q + 4 * g);
#pragma unroll
		for (int q = 0; q < 8; q++) c = mfma4(*reinterpret_cast<const float4 *>(h1 + j * TR_HS + 16 * q + 4 * g), w[q], c);
		const float bias = wq[OB2 + n];
		float4 o;
#pragma unroll
		for (int i = 0; i < 4; i++) {
			z2[t][i] = c[i] + bias;
			const float h = r0 + 4 * g + i < B ? bf16r(fmaxf(z2[t][i], 0.f)) : 0.f;
			h2[(4 * g + i) * TR_HS + n] = h;
			(&o.x)[i] = h;
		}
		*reinterpret_cast<float4 *>(ws + (size_t)(TH2 + n) * Bp + r0 + 4 * g) = o;
		float4 p;
#pragma unroll
		for (int i = 0; i < 4; i++) (&p.x)[i] = h1[(4 * g + i) * TR_HS + n];
		*reinterpret_cast<float4 *>(ws + (size_t)(TH1 + n) * Bp + r0 + 4 * g) = p;
	}
	__syncthreads();
	// layer 3, loss and its gradient: outputs 16 wv + j
	double e2 = 0.0;
	{
		const int n = 16 * wv + j;
		mlp_f32x4 c = {};
		float4 w[8];
#pragma unroll
		for (int q = 0; q < 8; q++) w[q] = bf16x4(net.w3t + n * MLP_H + 16 * q + 4 * g);
#pragma unroll
		for (int q = 0; q < 8; q++) c = mfma4(*reinterpret_cast<const float4 *>(h2 + j * TR_HS + 16 * q + 4 * g), w[q], c);
		const float bias = wq[OB3 + n];
		float4 o;
#pragma unroll
		for (int i = 0; i < 4; i++) {
			const float z = c[i] + bias;
			const float gn = 1.f / (1.f + expf(-z));
			const float d = gn - ts[(4 * g + i) * MLP_OUT + n];
			const bool live = r0 + 4 * g + i < B;
			const float dz = live ? 2.f * d / (float)((int64_t)B * MLP_OUT) * gn * (1.f - gn) : 0.f;
			if (live) e2 += (double)d * d;
			d3[(4 * g + i) * TR_OS + n] = dz;
			(&o.x)[i] = dz;
		}
		*reinterpret_cast<float4 *>(ws + (size_t)(TD3 + n) * Bp + r0 + 4 * g) = o;
	}
#pragma unroll
	for (int o = 32; o > 0; o >>= 1) e2 += __shfl_xor(e2, o, 64);
	if (l == 0) part[wv] = e2;
	__syncthreads();   // d3 and part written, h1 and h2 read for the last time
	if (tid == 0) sse[blockIdx.x] = (part[0] + part[1]) + (part[2] + part[3]);
	// gradient at layer 2's outputs (in h2)
#pragma unroll
	for (int t = 0; t < 2; t++) {
		const int n = 32 * wv + 16 * t + j;
		mlp_f32x4 c = {};
		float4 w[4];
#pragma unroll
		for (int q = 0; q < 4; q++) w[q] = *reinterpret_cast<const float4 *>(wq + OW3 + n * MLP_OUT + 16 * q + 4 * g);
#pragma unroll
		for (int q = 0; q < 4; q++) c = mfma4(*reinterpret_cast<const float4 *>(d3 + j * TR_OS + 16 * q + 4 * g), w[q], c);
		float4 o;
#pragma unroll
		for (int i = 0; i < 4; i++) {
			const float d = z2[t][i] > 0.f ? c[i] : 0.f;
			h2[(4 * g + i) * TR_HS + n] = d;
			(&o.x)[i] = d;
		}
		*reinterpret_cast<float4 *>(ws + (size_t)(TD2 + n) * Bp + r0 + 4 * g) = o;
	}
	__syncthreads();
	// gradient at layer 1's outputs
#pragma unroll
	for (int t = 0; t < 2; t++) {
		const int n = 32 * wv + 16 * t + j;
		mlp_f32x4 c = {};
		float4 w[8];
#pragma unroll
		for (int q = 0; q < 8; q++) w[q] = *reinterpret_cast<const float4 *>(wq + OW2 + n * MLP_H + 16 * q + 4 * g);
#pragma unroll
		for (int q = 0; q < 8; q++) c = mfma4(*reinterpret_cast<const float4 *>(h2 + j * TR_HS + 16 * q + 4 * g), w[q], c);
		float4 o;
#pragma unroll
		for (int i = 0; i < 4; i++) (&o.x)[i] = z1[t][i] > 0.f ? c[i] : 0.f;
		*reinterpret_cast<float4 *>(ws + (size_t)(TD1 + n) * Bp + r0 + 4 * g) = o;
	}
}

// Weight and bias gradients of rows [blockIdx.y kc, + kc): one wave per 32 x 32
// tile of a layer's weights (12 of layer 1, 16 of layer 2, 8 of layer 3), its
// sums into part[blockIdx.y][parameter].
// Bound: latency (16 matrix instructions per four loads of a row group); the
// splits give batch 4096 1152 waves.  10 us, where the three products and the
// column sums took 3.0 ms.
__global__ __launch_bounds__(64)
void mlp_wgrad_kernel(const float *__restrict__ ws, int Bp, int kc, float *__restrict__ part)
{
	const int l = threadIdx.x, g = l >> 4, j = l & 15;
	int tile = blockIdx.x, fi, fo, ni, no, ow, ob;   // inputs, outputs, their counts, places in theta
	if (tile < 12) {
		fi = TX, fo = TD1, ni = MLP_IN, no = MLP_H, ow = OW1, ob = OB1;
	} else if (tile < 28) {
		tile -= 12;
		fi = TH1, fo = TD2, ni = MLP_H, no = MLP_H, ow = OW2, ob = OB2;
	} else {
		tile -= 28;
		fi = TH2, fo = TD3, ni = MLP_H, no = MLP_OUT, ow = OW3, ob = OB3;
	}
	const int tn = no / 32, k0 = tile / tn * 32, n0 = tile % tn * 32;
	const int rb = blockIdx.y * kc, re = min(Bp, rb + kc);
	// inputs past the layer's last read it again; their sums are not stored
	const float *a0 = ws + (size_t)(fi + min(k0 + j, ni - 1)) * Bp + 4 * g;
	const float *a1 = ws + (size_t)(fi + min(k0 + 16 + j, ni - 1)) * Bp + 4 * g;
	const float *b0 = ws + (size_t)(fo + n0 + j) * Bp + 4 * g;
	const float *b1 = ws + (size_t)(fo + n0 + 16 + j) * Bp + 4 * g;
	mlp_f32x4 c[2][2] = {};
	float s0 = 0.f, s1 = 0.f;
#pragma unroll 4
	for (int r = rb; r < re; r += 16) {
		const float4 x0 = *reinterpret_cast<const float4 *>(a0 + r), x1 = *reinterpret_cast<const float4 *>(a1 + r);
		const float4 y0 = *reinterpret_cast<const float4 *>(b0 + r), y1 = *reinterpret_cast<const float4 *>(b1 + r);
		c[0][0] = mfma4(x0, y0, c[0][0]);
		c[0][1] = mfma4(x0, y1, c[0][1]);
		c[1][0] = mfma4(x1, y0, c[1][0]);
		c[1][1] = mfma4(x1, y1, c[1][1]);
		s0 += (y0.x + y0.y) + (y0.z + y0.w);
		s1 += (y1.x + y1.y) + (y1.z + y1.w);
	}
	float *out = part + (size_t)blockIdx.y * MLP_NPARAMS;
#pragma unroll
	for (int a = 0; a < 2; a++)
#pragma unroll
		for (int b = 0; b < 2; b++)
#pragma unroll
			for (int i = 0; i < 4; i++) {
				const int k = k0 + 16 * a + 4 * g + i;
				if (k < ni) out[ow + k * no + n0 + 16 * b + j] = c[a][b][i];
			}
	if (k0 == 0) {
		s0 += __shfl_xor(s0, 16, 64);
		s0 += __shfl_xor(s0, 32, 64);
		s1 += __shfl_xor(s1, 16, 64);
		s1 += __shfl_xor(s1, 32, 64);
		if (g == 0) out[ob + n0 + j] = s0;
		if (g == 1) out[ob + n0 + 16 + j] = s1;
	}
}

// Parameter i of the batch: the splits' gradients summed in order; with ADAM
// the update of theta, its moments and the derived copies, else the gradient
// out.  Block 0 also sums the blocks' squared errors.
// Bound: the read of the splits (4.3 MB at batch 4096); 5.6 us.
template <bool ADAM>
__global__ __launch_bounds__(256)
void mlp_update_kernel(const float *__restrict__ part, int ns, const double *__restrict__ sse, int nb,
                       double *__restrict__ sse_out, float *__restrict__ grad, float *__restrict__ theta,
                       float *__restrict__ m, float *__restrict__ v, float lr, float b1, float b2, float eps,
                       float c1, float c2, float *__restrict__ wq, uint16_t *__restrict__ blob,
                       float *__restrict__ bias)
{
	const int i = blockIdx.x * 256 + threadIdx.x;
	if (i < MLP_NPARAMS) {
		float gi = 0.f;
#pragma unroll 8
		for (int s = 0; s < ns; s++) gi += part[(size_t)s * MLP_NPARAMS + i];
		if constexpr (!ADAM) {
			grad[i] = gi;
		} else {
			const float mi = b1 * m[i] + (1.f - b1) * gi;
			const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
			m[i] = mi;
			v[i] = vi;
			const float th = theta[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
			theta[i] = th;
			// as mlp_pack_kernel lays them out
			if (i >= OB3 || (i >= OB2 && i < OW3) || (i >= OB1 && i < OW2)) {
				wq[i] = th;
				bias[i >= OB3 ? 2 * MLP_H + i - OB3 : i >= OB2 ? MLP_H + i - OB2 : i - OB1] = th;
			} else {
				const uint16_t q = f32_to_bf16(th);
				wq[i] = bf16_to_f32(q);
				if (i < OB1) blob[IW1 + (i % MLP_H) * MLP_K1 + i / MLP_H] = q;
				else if (i < OB2) blob[IW2 + ((i - OW2) % MLP_H) * MLP_H + (i - OW2) / MLP_H] = q;
				else blob[IW3 + ((i - OW3) % MLP_OUT) * MLP_H + (i - OW3) / MLP_OUT] = q;
			}
		}
	}
	if (blockIdx.x == 0) {
		__shared__ double red[256];
		double e = 0.0;
		for (int b = threadIdx.x; b < nb; b += 256) e += sse[b];
		red[threadIdx.x] = e;
		__syncthreads();
		for (int o = 128; o > 0; o >>= 1) {
			if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
			__syncthreads();
		}
		if (threadIdx.x == 0) *sse_out = red[0];
	}
}

// Standalone inference of B rows (one wave per 32 rows).
__global__ __launch_bounds__(64)
void mlp_infer_kernel(const float *__restrict__ X, int B, MlpInfer net, float *__restrict__ G)
{
	__shared__ __align__(16) uint16_t xb[32 * MLP_XS];
	__shared__ __align__(16) uint16_t hb[32 * MLP_HS];
	__shared__ float gs[32 * MLP_OUT];
	const int r0 = blockIdx.x * 32;
	for (int i = threadIdx.x; i < 32 * MLP_XS; i += 64) {
		const int r = i / MLP_XS, k = i - r * MLP_XS;
		const float v = (r0 + r < B && k < MLP_IN) ? X[(size_t)(r0 + r) * MLP_IN + k] : 0.f;
		xb[i] = f32_to_bf16(v);
	}
	__syncthreads();
	mlp_rows32(net, xb, hb, gs, MLP_OUT);
	for (int i = threadIdx.x; i < 32 * MLP_OUT; i += 64) {
		const int r = i / MLP_OUT;
		if (r0 + r < B) G[(size_t)r0 * MLP_OUT + i] = gs[i];
	}
}

namespace {

inline int nb(int64_t n, int b) { return (int)((n + b - 1) / b); }

void repack(bm4dof_ctx *ctx)
{
	float *theta = ctx->mlp_theta.as<float>(MLP_NPARAMS);
	float *wq = ctx->mlp_wq.as<float>(MLP_NPARAMS);
	char *blob = ctx->mlp_inf.as<char>(INF_BYTES);
	hipLaunchKernelGGL(mlp_pack_kernel, dim3(nb(std::max<int64_t>(MLP_NPARAMS, IWEND), 256)), dim3(256), 0,
	                   ctx->stream, theta, wq, (uint16_t *)blob, (float *)(blob + IB_BYTES));
	HIPCHK(hipGetLastError());
}

void need_net(bm4dof_ctx *ctx)
{
	if (!ctx->mlp_ready) throw ArgError("no network loaded: call bm4dof_mlp_set first");
}

// Buffers of a batch of B rows: the rows' workspace (Bp: B rounded up to a
// block), the splits' gradients and the blocks' squared errors.
struct TrainBufs {
	int Bp, nblk, kc, ns;
	float *ws, *part;
	double *sse;
};
TrainBufs train_bufs(bm4dof_ctx *ctx, int B, int steps)
{
	TrainBufs q;
	q.nblk = nb(B, TR_R);
	q.Bp = q.nblk * TR_R;
	q.kc = std::max(TR_KC, nb(nb(q.Bp, TR_SMAX), 16) * 16);
	q.ns = nb(q.Bp, q.kc);
	float *p = ctx->mlp_ws.as<float>((size_t)TEND * q.Bp + (size_t)q.ns * MLP_NPARAMS);
	q.ws = p;
	q.part = p + (size_t)TEND * q.Bp;
	q.sse = ctx->mlp_sse.as<double>((size_t)std::max(steps, 1) + q.nblk);
	return q;
}

// Forward and backward of one batch; leaves the splits' gradients in q.part
// and the blocks' squared errors after the steps' losses in q.sse.
void fwd_bwd(bm4dof_ctx *ctx, const TrainBufs &q, const float *x, const float *t, int64_t rows, int B, uint32_t seed,
             double *blk_sse)
{
	const float *wq = ctx->mlp_wq.as<float>(MLP_NPARAMS);
	const MlpInfer net = mlp_infer_view(ctx->mlp_inf.as<char>(INF_BYTES));
	hipLaunchKernelGGL(mlp_rows_kernel, dim3(q.nblk), dim3(256), 0, ctx->stream, x, t, rows, B, seed, net, wq, q.Bp,
	                   q.ws, blk_sse);
	hipLaunchKernelGGL(mlp_wgrad_kernel, dim3(36, q.ns), dim3(64), 0, ctx->stream, q.ws, q.Bp, q.kc, q.part);
	HIPCHK(hipGetLastError());
}

} // namespace

MlpInfer mlp_net(bm4dof_ctx *ctx)
{
	need_net(ctx);
	return mlp_infer_view(ctx->mlp_inf.as<char>(INF_BYTES));
}

} // namespace bm4dof

using namespace bm4dof;

extern "C" {

__attribute__((visibility("default")))
int bm4dof_mlp_set(bm4dof_ctx *ctx, const float *theta)
{
	if (!ctx) return BM4DOF_EINVAL;
	return guarded(ctx, [&] {
		if (!theta) throw ArgError("theta is NULL");
		HIPCHK(hipSetDevice(ctx->device));
		float *d = ctx->mlp_theta.as<float>(MLP_NPARAMS);
		float *m = ctx->mlp_m.as<float>(MLP_NPARAMS);
		float *v = ctx->mlp_v.as<float>(MLP_NPARAMS);
		HIPCHK(hipMemcpyAsync(d, theta, (size_t)MLP_NPARAMS * 4, hipMemcpyHostToDevice, ctx->stream));
		HIPCHK(hipMemsetAsync(m, 0, (size_t)MLP_NPARAMS * 4, ctx->stream));
		HIPCHK(hipMemsetAsync(v, 0, (size_t)MLP_NPARAMS * 4, ctx->stream));
		ctx->mlp_step = 0;
		repack(ctx);
		HIPCHK(hipStreamSynchronize(ctx->stream));
		ctx->mlp_ready = true;
	});
}

__attribute__((visibility("default")))
int bm4dof_mlp_get(const bm4dof_ctx *cctx, float *theta)
{
	bm4dof_ctx *ctx = const_cast<bm4dof_ctx *>(cctx);
	if (!ctx) return BM4DOF_EINVAL;
	return guarded(ctx, [&] {
		need_net(ctx);
		if (!theta) throw ArgError("theta is NULL");
		HIPCHK(hipSetDevice(ctx->device));
		HIPCHK(hipMemcpyAsync(theta, ctx->mlp_theta.as<float>(MLP_NPARAMS), (size_t)MLP_NPARAMS * 4,
		                      hipMemcpyDeviceToHost, ctx->stream));
		HIPCHK(hipStreamSynchronize(ctx->stream));
	});
}

__attribute__((visibility("default")))
int bm4dof_mlp_forward(bm4dof_ctx *ctx, const float *x, int64_t rows, float *gains, int on_device)
{
	if (!ctx) return BM4DOF_EINVAL;
	return guarded(ctx, [&] {
		need_net(ctx);
		if (rows < 0 || (rows > 0 && (!x || !gains))) throw ArgError("bad rows or NULL buffer");
		if (rows == 0) return;
		if (rows > ((int64_t)1 << 31) - 64) throw ArgError("too many rows", BM4DOF_EUNSUPP);
		HIPCHK(hipSetDevice(ctx->device));
		const float *dx = x;
		float *dg = gains;
		if (!on_device) {
			float *bx = ctx->io_noisy.as<float>((size_t)rows * MLP_IN);
			HIPCHK(hipMemcpyAsync(bx, x, (size_t)rows * MLP_IN * 4, hipMemcpyHostToDevice, ctx->stream));
			dx = bx;
			dg = ctx->io_final.as<float>((size_t)rows * MLP_OUT);
		}
		const MlpInfer net = mlp_infer_view(ctx->mlp_inf.as<char>(INF_BYTES));
		hipLaunchKernelGGL(mlp_infer_kernel, dim3(nb(rows, 32)), dim3(64), 0, ctx->stream, dx, (int)rows, net, dg);
		HIPCHK(hipGetLastError());
		if (!on_device)
			HIPCHK(hipMemcpyAsync(gains, dg, (size_t)rows * MLP_OUT * 4, hipMemcpyDeviceToHost, ctx->stream));
		HIPCHK(hipStreamSynchronize(ctx->stream));
	});
}

__attribute__((visibility("default")))
int bm4dof_mlp_grad(bm4dof_ctx *ctx, const float *x, const float *t, int rows, float *loss, float *grad)
{
	if (!ctx) return BM4DOF_EINVAL;
	return guarded(ctx, [&] {
		need_net(ctx);
		if (rows <= 0 || !x || !t) throw ArgError("bad rows or NULL buffer");
		HIPCHK(hipSetDevice(ctx->device));
		float *bx = ctx->mlp_xb.as<float>((size_t)rows * MLP_IN);
		float *bt = ctx->mlp_tb.as<float>((size_t)rows * MLP_OUT);
		const TrainBufs q = train_bufs(ctx, rows, 1);
		HIPCHK(hipMemcpyAsync(bx, x, (size_t)rows * MLP_IN * 4, hipMemcpyHostToDevice, ctx->stream));
		HIPCHK(hipMemcpyAsync(bt, t, (size_t)rows * MLP_OUT * 4, hipMemcpyHostToDevice, ctx->stream));
		double *sse = q.sse;
		fwd_bwd(ctx, q, bx, bt, rows, rows, 0u, sse + 1);
		hipLaunchKernelGGL(mlp_update_kernel<false>, dim3(nb(MLP_NPARAMS, 256)), dim3(256), 0, ctx->stream, q.part, q.ns,
		                   sse + 1, q.nblk, sse, ctx->mlp_grad.as<float>(MLP_NPARAMS), (float *)nullptr,
		                   (float *)nullptr, (float *)nullptr, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, (float *)nullptr,
		                   (uint16_t *)nullptr, (float *)nullptr);
		HIPCHK(hipGetLastError());
		double h_sse = 0.0;
		HIPCHK(hipMemcpyAsync(&h_sse, sse, 8, hipMemcpyDeviceToHost, ctx->stream));
		if (grad)
			HIPCHK(hipMemcpyAsync(grad, ctx->mlp_grad.as<float>(MLP_NPARAMS), (size_t)MLP_NPARAMS * 4,
			                      hipMemcpyDeviceToHost, ctx->stream));
		HIPCHK(hipStreamSynchronize(ctx->stream));
		if (loss) *loss = (float)(h_sse / ((double)rows * MLP_OUT));
	});
}

__attribute__((visibility("default")))
int bm4dof_mlp_train(bm4dof_ctx *ctx, const float *x, const float *t, int64_t rows, int batch, int steps,
                     float lr, unsigned seed, float *losses)
{
	if (!ctx) return BM4DOF_EINVAL;
	return guarded(ctx, [&] {
		need_net(ctx);
		if (rows <= 0 || batch <= 0 || steps < 0 || !x || !t) throw ArgError("bad training arguments");
		if (batch > rows) throw ArgError("batch larger than the data set");
		HIPCHK(hipSetDevice(ctx->device));
		float *theta = ctx->mlp_theta.as<float>(MLP_NPARAMS);
		float *m = ctx->mlp_m.as<float>(MLP_NPARAMS);
		float *v = ctx->mlp_v.as<float>(MLP_NPARAMS);
		float *wq = ctx->mlp_wq.as<float>(MLP_NPARAMS);
		char *blob = ctx->mlp_inf.as<char>(INF_BYTES);
		const TrainBufs q = train_bufs(ctx, batch, steps);
		double *sse = q.sse, *blk = sse + std::max(steps, 1);
		const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
		for (int s = 0; s < steps; s++) {
			fwd_bwd(ctx, q, x, t, rows, batch, seed + (uint32_t)ctx->mlp_step, blk);
			ctx->mlp_step++;
			const float c1 = 1.f - powf(b1, (float)ctx->mlp_step), c2 = 1.f - powf(b2, (float)ctx->mlp_step);
			hipLaunchKernelGGL(mlp_update_kernel<true>, dim3(nb(MLP_NPARAMS, 256)), dim3(256), 0, ctx->stream, q.part,
			                   q.ns, blk, q.nblk, sse + s, (float *)nullptr, theta, m, v, lr, b1, b2, eps, c1, c2, wq,
			                   (uint16_t *)blob, (float *)(blob + IB_BYTES));
			HIPCHK(hipGetLastError());
		}
		if (losses && steps > 0) {
			std::vector<double> h(steps);
			HIPCHK(hipMemcpyAsync(h.data(), sse, (size_t)steps * 8, hipMemcpyDeviceToHost, ctx->stream));
			HIPCHK(hipStreamSynchronize(ctx->stream));
			for (int s = 0; s < steps; s++) losses[s] = (float)(h[s] / ((double)batch * MLP_OUT));
		}
		HIPCHK(hipStreamSynchronize(ctx->stream));
	});
}

} // extern "C"
