// Shared host/device definitions of the MI355X BM4D-OF denoiser.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace bm4dof {

// Crop box of one spatial tile, global pixel coordinates; every tile spans
// all frames (the reference tiles only in space, lib_videot.hpp:854-916).
struct TileBox {
	int ox, oy, ex, ey;   // crop [ox,ex) x [oy,ey)
};

// Constants of one step, passed by value to the kernels.
struct StepConst {
	int W, H, F, C;       // video size
	int WH;               // W*H
	int WHC;              // W*H*C (frame stride of a C-channel video)
	int sPx, sPt, P;      // patch: px, pt, px*px*pt
	int sWx;              // spatial search window
	int wtf, wtb;         // temporal search range forward / backward
	int npmax;            // nSimilarPatches (neighbour slots per group)
	float tau2;           // tau*tau*px*px*pt (nldct.cpp:1157)
	float beta_sigma2;    // (beta*sigma)^2      (nldct.cpp:1808-1809)
	float betaM_sigma2;   // (betaMean*sigma)^2  (nldct.cpp:1810-1811)
	float sigma2;         // sigma^2             (nldct.cpp:1813)
	int order_inv;        // orderInvariance
	int use_flow;         // flows present
	int nW, wTmp, hTmp;   // tile grid: columns, interior width / height
	// predictive search (a VBM3D_SEARCH build): window of the frames after
	// the first, matches kept per frame, distance bias dsub^2*255
	int pred_w, pred_np;
	float pred_dsub;
	// channels at the head of an est row that hold samples without the row's
	// weight, which the region fold then applies (0, or C - 1)
	int est_raw;
};

// Pixel block of the ordered aggregation: RX x RY x RT pixels, frame blocks
// counted from tb0.
struct AggRegion { int RX, RY, RT, tb0; };

// Binned ordered aggregation: bins (regions) of 2^lx x 2^ly pixels x 2^lt
// frames; a patch overlaps at most 8 of them.
struct BinShape { int lx, ly, lt; };

// stable radix sort passes (sortscan.hip): threads per block, most pairs per
// thread
#define RS_THREADS 64
#define RS_IPT 256
// most rows per tile of the first bin-sort pass (at most 8 pairs per row)
#define BIN_RT 4096

// Groups that the bounded matching leaves to another matcher: RedoList::N
// lists, a group in the one of its index modulo N, whose counters lie on lines
// of their own.  (One counter for all takes 7 ns a group, 7 ms where a million
// groups are left.)  Without a bound (scale 0) every group is, and nothing is
// listed.
struct RedoList {
	static constexpr int N = 64, LINE = 32;
	uint32_t *p;              // N counters, LINE words apart, then N lists
	const float2 *qp;         // (mid, scale) of the integer samples
	uint32_t *total;          // running total of such groups
	int G;
	__host__ __device__ static size_t words(int G) { return (size_t)N * LINE + (size_t)N * ((G + N - 1) / N); }
	__device__ void add(int g) const
	{
		uint32_t *c = p + (g % N) * LINE;
		const uint32_t i = atomicAdd(c, 1u);
		p[N * LINE + (size_t)(g % N) * ((G + N - 1) / N) + i] = (uint32_t)g;
	}
	// the groups a block of a grid of a multiple of N blocks takes: number
	// i = first(), first() + step(), ... below count() (called once)
	__device__ int first() const { return (int)(blockIdx.x / N); }
	__device__ int step() const { return (int)(gridDim.x / N); }
	__device__ int count() const
	{
		const int l = (int)(blockIdx.x % N);
		const int n = qp->y > 0.f ? (int)p[l * LINE] : (G - l + N - 1) / N;
		if (first() == 0 && threadIdx.x == 0) atomicAdd(total, (uint32_t)n);
		return n;
	}
	__device__ int at(int i) const
	{
		const int l = (int)(blockIdx.x % N);
		return qp->y > 0.f ? (int)p[N * LINE + (size_t)l * ((G + N - 1) / N) + i] : l + N * i;
	}
};

// Decode a 3-index position t*WH + y*W + x.
__host__ __device__ inline void pos_decode(uint32_t pos, int W, int WH, int &x, int &y, int &t)
{
	t = (int)(pos / (uint32_t)WH);
	const uint32_t r = pos - (uint32_t)t * (uint32_t)WH;
	y = (int)(r / (uint32_t)W);
	x = (int)(r - (uint32_t)y * (uint32_t)W);
}

} // namespace bm4dof
