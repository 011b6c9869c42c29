// Learned gain network: training (forward, backward, Adam) and standalone
// inference.  No counterpart in the reference: the network predicts, from
// the step-1 Haar-domain coefficients of one group row, the step-2 Wiener
// gains y^2 / (y^2 + (beta sigma)^2) (src/core/nldct.cpp:2131) so that one
// pass replaces the two steps.
//
// Parameters: a flat float32 master vector theta (W1 [66][128], b1, W2
// [128][128], b2, W3 [128][64], b3; W[k][j] input-major), Adam moments m, v,
// and two derived copies refreshed after every update:
//   * wq: W1..W3 rounded to bf16 (as float) as operands of both directions of
//     the training step, and the biases;
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

// Place of term k of a sum in a row of matrix operands: 16 terms go to four
// instructions, of which number v takes terms 4 v + g from lane group g, and a
// lane's four operands lie together (float4 at 4 g).
__host__ __device__ constexpr int term_place(int k) { return (k & ~15) | (k & 3) << 2 | ((k >> 2) & 3); }

// wq (floats): rows of terms in the order above.  Forward: a row per output
// (layer 1: 80 terms, the last 14 zero); backward: W2 and W3, a row per input.
constexpr int TR_K1 = 80;
constexpr int QF1 = 0, QF2 = QF1 + MLP_H * TR_K1, QF3 = QF2 + MLP_H * MLP_H, QB2 = QF3 + MLP_OUT * MLP_H,
              QB3 = QB2 + MLP_H * MLP_H, QBIAS = QB3 + MLP_H * MLP_OUT, QEND = QBIAS + 2 * MLP_H + MLP_OUT;

// The copies of parameter i in wq, given its value rounded as the layers use
// it (biases as they are).
__device__ __forceinline__ void wq_store(float *__restrict__ wq, int i, float v)
{
	if (i < OB1) {
		const int k = i / MLP_H, n = i - k * MLP_H;
		wq[QF1 + n * TR_K1 + term_place(k)] = v;
	} else if (i < OW2) {
		wq[QBIAS + i - OB1] = v;
	} else if (i < OB2) {
		const int k = (i - OW2) / MLP_H, n = i - OW2 - k * MLP_H;
		wq[QF2 + n * MLP_H + term_place(k)] = v;
		wq[QB2 + k * MLP_H + term_place(n)] = v;
	} else if (i < OW3) {
		wq[QBIAS + MLP_H + i - OB2] = v;
	} else if (i < OB3) {
		const int k = (i - OW3) / MLP_OUT, n = i - OW3 - k * MLP_OUT;
		wq[QF3 + n * MLP_H + term_place(k)] = v;
		wq[QB3 + k * MLP_OUT + term_place(n)] = v;
	} else
		wq[QBIAS + 2 * MLP_H + i - OB3] = v;
}
__device__ __forceinline__ bool is_bias(int i) { return (i >= OB1 && i < OW2) || (i >= OB2 && i < OW3) || i >= OB3; }

// theta -> the training copies (wq) and the inference blob.
__global__ void mlp_pack_kernel(const float *__restrict__ theta, float *__restrict__ wq,
                                uint16_t *__restrict__ blob, float *__restrict__ bias)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < MLP_NPARAMS) wq_store(wq, i, is_bias(i) ? theta[i] : bf16r(theta[i]));
	if (i < MLP_H * (TR_K1 - MLP_IN)) {
		const int n = i / (TR_K1 - MLP_IN), k = MLP_IN + i - n * (TR_K1 - MLP_IN);
		wq[QF1 + n * TR_K1 + term_place(k)] = 0.f;
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
// An instruction adds its four terms one after another, each as one fused
// multiply-add, so a chain of them over terms in increasing order
// (term_place) is a sequential sum bit for bit.  Every sum of a step is one:
// over a layer's inputs or outputs, and over the batch's rows for the
// gradients.  The parameters a training ends on depend on that order: a last
// bit of a sum can move a hidden unit across a bfloat16 boundary, and Adam
// turns a difference in a small gradient into one of the size of the rate.
//
// The batch's rows are independent up to the weight gradients: one launch
// takes 16 rows through both directions, one forms the weight gradients, one
// updates.
// ---------------------------------------------------------------------------

typedef float mlp_f32x4 __attribute__((ext_vector_type(4)));

constexpr int TR_R = 16;                        // rows of a block
// per row in the workspace, feature-major [feature][row], the rows of a block
// in the order of term_place: layer inputs (rounded), then the gradients at
// the layers' outputs
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
// every layer's outputs; activations in LDS, weights from L2.  A value goes to
// LDS at its place as a term of the next product; the workspace's rows are read
// from there, so that a lane's four lie together.
// Bound: latency of the five dependent layers, 22 us at batch 4096 (256 blocks).
__global__ __launch_bounds__(256)
void mlp_rows_kernel(const float *__restrict__ X, const float *__restrict__ T, int64_t nrows, int B, uint32_t seed,
                     const float *__restrict__ wq, int Bp, float *__restrict__ ws, double *__restrict__ sse)
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
	for (int u = 0; u < TR_R * TR_K1 / 256; u++) {
		const int i = tid + 256 * u, r = i / TR_K1, k = i - r * TR_K1;
		xs[r * TR_XS + term_place(k)] = src[r] >= 0 && k < MLP_IN ? bf16r(X[(size_t)src[r] * MLP_IN + k]) : 0.f;
	}
#pragma unroll
	for (int u = 0; u < TR_R * MLP_OUT / 256; u++) {
		const int i = tid + 256 * u, r = i / MLP_OUT, k = i - r * MLP_OUT;
		ts[i] = src[r] >= 0 ? T[(size_t)src[r] * MLP_OUT + k] : 0.f;
	}
	__syncthreads();
	for (int i = tid; i < MLP_IN * TR_R; i += 256) {
		const int k = i / TR_R, r = i - k * TR_R;
		ws[(size_t)(TX + k) * Bp + r0 + term_place(r)] = xs[r * TR_XS + term_place(k)];
	}
	// column n of the rows in LDS (stride hs) to feature f: float4 4 g holds rows 4 v + g
	auto keep = [&](const float *h, int hs, int n, int f) {
		const float *p = h + g * hs + term_place(n);
		*reinterpret_cast<float4 *>(ws + (size_t)(f + n) * Bp + r0 + 4 * g) =
		    make_float4(p[0], p[4 * hs], p[8 * hs], p[12 * hs]);
	};
	// the lane's operands of 16 Q terms of a row
	auto row16 = [&](const float *p, auto &w) {
#pragma unroll
		for (int q = 0; q < (int)(sizeof w / sizeof w[0]); q++) w[q] = *reinterpret_cast<const float4 *>(p + 16 * q + 4 * g);
	};
	auto product = [&](const float *h, const auto &w) {
		mlp_f32x4 c = {};
#pragma unroll
		for (int q = 0; q < (int)(sizeof w / sizeof w[0]); q++)
			c = mfma4(*reinterpret_cast<const float4 *>(h + 16 * q + 4 * g), w[q], c);
		return c;
	};
	// layer 1: outputs 32 wv + 16 t + j
	float z1[2][4], z2[2][4];
#pragma unroll
	for (int t = 0; t < 2; t++) {
		const int n = 32 * wv + 16 * t + j;
		float4 w[TR_K1 / 16];
		row16(wq + QF1 + n * TR_K1, w);
		const mlp_f32x4 c = product(xs + j * TR_XS, w);
		const float bias = wq[QBIAS + n];
#pragma unroll
		for (int i = 0; i < 4; i++) {
			z1[t][i] = c[i] + bias;
			h1[(4 * g + i) * TR_HS + term_place(n)] = r0 + 4 * g + i < B ? bf16r(fmaxf(z1[t][i], 0.f)) : 0.f;
		}
	}
	__syncthreads();
	// layer 2
#pragma unroll
	for (int t = 0; t < 2; t++) {
		const int n = 32 * wv + 16 * t + j;
		float4 w[MLP_H / 16];
		row16(wq + QF2 + n * MLP_H, w);
		keep(h1, TR_HS, n, TH1);
		const mlp_f32x4 c = product(h1 + j * TR_HS, w);
		const float bias = wq[QBIAS + MLP_H + n];
#pragma unroll
		for (int i = 0; i < 4; i++) {
			z2[t][i] = c[i] + bias;
			h2[(4 * g + i) * TR_HS + term_place(n)] = r0 + 4 * g + i < B ? bf16r(fmaxf(z2[t][i], 0.f)) : 0.f;
		}
	}
	__syncthreads();
	// layer 3, loss and its gradient: outputs 16 wv + j
	double e2 = 0.0;
	{
		const int n = 16 * wv + j;
		float4 w[MLP_H / 16];
		row16(wq + QF3 + n * MLP_H, w);
#pragma unroll
		for (int t = 0; t < 2; t++) keep(h2, TR_HS, 32 * wv + 16 * t + j, TH2);
		const mlp_f32x4 c = product(h2 + j * TR_HS, w);
		const float bias = wq[QBIAS + 2 * MLP_H + n];
#pragma unroll
		for (int i = 0; i < 4; i++) {
			const float z = c[i] + bias;
			const float gn = 1.f / (1.f + expf(-z));
			const float d = gn - ts[(4 * g + i) * MLP_OUT + n];
			const bool live = r0 + 4 * g + i < B;
			d3[(4 * g + i) * TR_OS + term_place(n)] =
			    live ? 2.f * d / (float)((int64_t)B * MLP_OUT) * gn * (1.f - gn) : 0.f;
			if (live) e2 += (double)d * d;
		}
	}
#pragma unroll
	for (int o = 32; o > 0; o >>= 1) e2 += __shfl_xor(e2, o, 64);
	if (l == 0) part[wv] = e2;
	__syncthreads();   // d3 and part written, h1 and h2 read for the last time
	if (tid == 0) sse[blockIdx.x] = (part[0] + part[1]) + (part[2] + part[3]);
	// gradient at layer 2's outputs (in h2)
	keep(d3, TR_OS, 16 * wv + j, TD3);
#pragma unroll
	for (int t = 0; t < 2; t++) {
		const int n = 32 * wv + 16 * t + j;
		float4 w[MLP_OUT / 16];
		row16(wq + QB3 + n * MLP_OUT, w);
		const mlp_f32x4 c = product(d3 + j * TR_OS, w);
#pragma unroll
		for (int i = 0; i < 4; i++) h2[(4 * g + i) * TR_HS + term_place(n)] = z2[t][i] > 0.f ? c[i] : 0.f;
	}
	__syncthreads();
	// gradient at layer 1's outputs (in h1)
#pragma unroll
	for (int t = 0; t < 2; t++) {
		const int n = 32 * wv + 16 * t + j;
		float4 w[MLP_H / 16];
		row16(wq + QB2 + n * MLP_H, w);
		keep(h2, TR_HS, n, TD2);
		const mlp_f32x4 c = product(h2 + j * TR_HS, w);
#pragma unroll
		for (int i = 0; i < 4; i++) h1[(4 * g + i) * TR_HS + term_place(n)] = z1[t][i] > 0.f ? c[i] : 0.f;
	}
	__syncthreads();
#pragma unroll
	for (int t = 0; t < 2; t++) keep(h1, TR_HS, 32 * wv + 16 * t + j, TD1);
}

// Weight and bias gradients of the batch: one wave per 16 x 16 tile of a
// layer's weights, the bias as the weights of one more input that is 1 in every
// row (5 x 8 tiles of layer 1, 9 x 8 of layer 2, 9 x 4 of layer 3).
// Bound: the chain of Bp / 4 dependent matrix instructions that the order of
// the sums asks for, 25 ns each; the operands of WG_U row blocks are loaded
// ahead of it.  27 us at batch 4096, 125 us at 20000.
constexpr int WG_U = 8;
__global__ __launch_bounds__(64)
void mlp_wgrad_kernel(const float *__restrict__ ws, int Bp, float *__restrict__ grad)
{
	const int l = threadIdx.x, g = l >> 4, j = l & 15;
	int tile = blockIdx.x, fi, fo, ni, no, ow, ob;   // inputs, outputs, their counts, places in theta
	if (tile < 40) {
		fi = TX, fo = TD1, ni = MLP_IN, no = MLP_H, ow = OW1, ob = OB1;
	} else if (tile < 112) {
		tile -= 40;
		fi = TH1, fo = TD2, ni = MLP_H, no = MLP_H, ow = OW2, ob = OB2;
	} else {
		tile -= 112;
		fi = TH2, fo = TD3, ni = MLP_H, no = MLP_OUT, ow = OW3, ob = OB3;
	}
	const int tn = no / 16, k0 = tile / tn * 16, n0 = tile % tn * 16, nblk = Bp / TR_R;
	const bool ones = k0 + j >= ni;   // inputs past the bias' are not stored
	const float *a = ws + (size_t)(fi + min(k0 + j, ni - 1)) * Bp + 4 * g;
	const float *b = ws + (size_t)(fo + n0 + j) * Bp + 4 * g;
	float4 x[WG_U], y[WG_U], xn[WG_U], yn[WG_U];
	auto load = [&](int q0, float4 (&u)[WG_U], float4 (&v)[WG_U]) {
#pragma unroll
		for (int q = 0; q < WG_U; q++) {
			const size_t o = (size_t)min(q0 + q, nblk - 1) * TR_R;
			u[q] = *reinterpret_cast<const float4 *>(a + o);
			v[q] = *reinterpret_cast<const float4 *>(b + o);
		}
	};
	mlp_f32x4 c = {};
	auto add = [&](int q0, const float4 (&u)[WG_U], const float4 (&v)[WG_U]) {
#pragma unroll
		for (int q = 0; q < WG_U; q++)
			if (q0 + q < nblk) c = mfma4(ones ? make_float4(1.f, 1.f, 1.f, 1.f) : u[q], v[q], c);
	};
	load(0, x, y);
	for (int q0 = 0; q0 < nblk; q0 += 2 * WG_U) {
		load(q0 + WG_U, xn, yn);
		add(q0, x, y);
		load(q0 + 2 * WG_U, x, y);
		add(q0 + WG_U, xn, yn);
	}
#pragma unroll
	for (int i = 0; i < 4; i++) {
		const int k = k0 + 4 * g + i;
		if (k <= ni) grad[(k < ni ? ow + k * no : ob) + n0 + j] = c[i];
	}
}

// Sum of the blocks' squared errors, by one block of 256 threads.
__device__ __forceinline__ void mlp_sum_blocks(const double *__restrict__ sse, int nb, double *__restrict__ out)
{
	__shared__ double red[256];
	double e = 0.0;
	for (int b = threadIdx.x; b < nb; b += 256) e += sse[b];
	red[threadIdx.x] = e;
	__syncthreads();
	for (int o = 128; o > 0; o >>= 1) {
		if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
		__syncthreads();
	}
	if (threadIdx.x == 0) *out = red[0];
}

// Adam on the batch's gradient: theta, its moments and the derived copies.
// Block 0 also sums the blocks' squared errors.  Latency, 5 us.
__global__ __launch_bounds__(256)
void mlp_update_kernel(const float *__restrict__ grad, const double *__restrict__ sse, int nb,
                       double *__restrict__ sse_out, float *__restrict__ theta, float *__restrict__ m,
                       float *__restrict__ v, float lr, float b1, float b2, float eps, float c1, float c2,
                       float *__restrict__ wq, uint16_t *__restrict__ blob, float *__restrict__ bias)
{
	const int i = blockIdx.x * 256 + threadIdx.x;
	if (i < MLP_NPARAMS) {
		const float gi = grad[i];
		const float mi = b1 * m[i] + (1.f - b1) * gi;
		const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
		m[i] = mi;
		v[i] = vi;
		const float th = theta[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
		theta[i] = th;
		// as mlp_pack_kernel lays them out
		if (is_bias(i)) {
			wq_store(wq, i, th);
			bias[i >= OB3 ? 2 * MLP_H + i - OB3 : i >= OB2 ? MLP_H + i - OB2 : i - OB1] = th;
		} else {
			const uint16_t q = f32_to_bf16(th);
			wq_store(wq, i, bf16_to_f32(q));
			if (i < OB1) blob[IW1 + (i % MLP_H) * MLP_K1 + i / MLP_H] = q;
			else if (i < OB2) blob[IW2 + ((i - OW2) % MLP_H) * MLP_H + (i - OW2) / MLP_H] = q;
			else blob[IW3 + ((i - OW3) % MLP_OUT) * MLP_H + (i - OW3) / MLP_OUT] = q;
		}
	}
	if (blockIdx.x == 0) mlp_sum_blocks(sse, nb, sse_out);
}

// The batch's squared error alone (bm4dof_mlp_grad).
__global__ __launch_bounds__(256)
void mlp_loss_kernel(const double *__restrict__ sse, int nb, double *__restrict__ sse_out)
{
	mlp_sum_blocks(sse, nb, sse_out);
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
	float *wq = ctx->mlp_wq.as<float>(QEND);
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
// block), the gradient, and the steps' squared errors with the blocks' after
// them.
struct TrainBufs {
	int Bp, nblk;
	float *ws, *grad;
	double *sse;
};
TrainBufs train_bufs(bm4dof_ctx *ctx, int B, int steps)
{
	TrainBufs q;
	q.nblk = nb(B, TR_R);
	q.Bp = q.nblk * TR_R;
	q.ws = ctx->mlp_ws.as<float>((size_t)TEND * q.Bp);
	q.grad = ctx->mlp_grad.as<float>(MLP_NPARAMS);
	q.sse = ctx->mlp_sse.as<double>((size_t)std::max(steps, 1) + q.nblk);
	return q;
}

// Forward and backward of one batch; leaves the gradient in q.grad and the
// blocks' squared errors in blk_sse.
void fwd_bwd(bm4dof_ctx *ctx, const TrainBufs &q, const float *x, const float *t, int64_t rows, int B, uint32_t seed,
             double *blk_sse)
{
	const float *wq = ctx->mlp_wq.as<float>(QEND);
	hipLaunchKernelGGL(mlp_rows_kernel, dim3(q.nblk), dim3(256), 0, ctx->stream, x, t, rows, B, seed, wq, q.Bp, q.ws,
	                   blk_sse);
	hipLaunchKernelGGL(mlp_wgrad_kernel, dim3(148), dim3(64), 0, ctx->stream, q.ws, q.Bp, q.grad);
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
		hipLaunchKernelGGL(mlp_loss_kernel, dim3(1), dim3(256), 0, ctx->stream, sse + 1, q.nblk, sse);
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
		float *wq = ctx->mlp_wq.as<float>(QEND);
		char *blob = ctx->mlp_inf.as<char>(INF_BYTES);
		const TrainBufs q = train_bufs(ctx, batch, steps);
		double *sse = q.sse, *blk = sse + std::max(steps, 1);
		const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
		for (int s = 0; s < steps; s++) {
			fwd_bwd(ctx, q, x, t, rows, batch, seed + (uint32_t)ctx->mlp_step, blk);
			ctx->mlp_step++;
			const float c1 = 1.f - powf(b1, (float)ctx->mlp_step), c2 = 1.f - powf(b2, (float)ctx->mlp_step);
			hipLaunchKernelGGL(mlp_update_kernel, dim3(nb(MLP_NPARAMS, 256)), dim3(256), 0, ctx->stream, q.grad, blk,
			                   q.nblk, sse + s, theta, m, v, lr, b1, b2, eps, c1, c2, wq, (uint16_t *)blob,
			                   (float *)(blob + IB_BYTES));
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
