// Node-block (4x4) aggregation AMG preconditioner.
//
// The reference GPU path has no AMG (it preconditions GMRES with node-block
// Jacobi, solvers/cuda/include/Gmres.hpp:47-67); its CPU path uses PETSc
// FIELDSPLIT + GAMG (solvers/cpu/include/TransientFlowRuntime.hpp:176-215) and
// the GPU tet solver a scalar plain-aggregation AMG
// (solvers/cuda/include/AggregationAmg.hpp).  This is a coupled (all four
// fields per node) plain-aggregation hierarchy:
//   * symbolic phase (host, once per mesh, deterministic): strength graph from
//     the first matrix (field-diagonal couplings), greedy aggregation in node
//     order, coarse block pattern, and for every coarse block the ascending
//     list of fine blocks that sum into it;
//   * numeric phase (GPU, every Newton step): A P (the blocks of a row summed
//     per aggregate of their columns) and from it the Galerkin coarse blocks,
//     both as fixed-order segmented sums (no atomics), 4x4 diagonal inverses,
//     and a dense Gauss-Jordan inverse of the coarsest operator;
//   * V-cycle: symmetric multicolour block Gauss-Seidel (greedy node colouring
//     per level, one launch per colour, in place -- rows of one colour are
//     uncoupled), damped block Jacobi with omega = 1.33 / lambda_max(D^-1 A),
//     or a Chebyshev polynomial in D^-1 A on [0.1, 1.1] lambda_max
//     (power-iteration estimate; one fused launch per degree, no colours);
//     restriction = aggregate sums, prolongation = injection; optionally
//     entirely in FP32.  The first smoothing step after the coarse correction
//     needs b - A (x + P xc) = r - (A P) xc with the residual r that was
//     restricted: A P has about a tenth of A's blocks, so that step is not
//     another pass over A.  With two steps before and after, three passes over
//     A instead of four: 1624 -> 1264 us in FP64 and 606 -> 499 us with the FP16
//     smoothing matrices for 16.2 million blocks.
// The prolongator is the 0/1 aggregate map, stored as integers, so it is exact
// in any precision.
#include "tfi_solver.hpp"

#include <algorithm>
#include <cmath>
#include <numeric>

namespace tfi {

namespace {

constexpr double kStrength = 0.25;     // row-relative strength threshold
constexpr int kMaxLevels = 16;
constexpr double kOmegaScale = 1.33;   // block-Jacobi damping = kOmegaScale / lambda_max(D^-1 A)
constexpr int kPre = 2, kPost = 2;      // Jacobi sweeps / Chebyshev degree
constexpr double kChebLow = 0.1, kChebHigh = 1.1;  // Chebyshev interval, in units of lambda_max(D^-1 A)
constexpr int kPowerIterations = 12;
// Workgroups of a power-iteration product, at most: a wave with several rows waits for
// one after the other (16.2 million blocks: 390 us with 4096 workgroups, 368 with
// 16384, 362 with all 37,554; 230 million 5.6, 5.3 and 5.1 ms), and one workgroup
// adds up their sums (6 us).
constexpr int kPowerBlocks = 65536;

template <class T>
__device__ inline T WaveSumT(T v)
{
	for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
	return v;
}

// This lane's share of row `row` of A x for one block-row lane r: the wave
// splits the row's blocks over 16 groups of 4 lanes (lane r of a group takes
// block row r).  In FP32 each lane keeps four blocks in flight (column
// indices, then block rows and x segments as 16-byte vector loads) so that a
// row costs about one memory latency instead of one per block; in FP64 the
// plain loop measured faster (the four 32-byte loads in flight cost
// occupancy).
template <class T>
__device__ inline T RowPartial(const int* __restrict__ ro, const int* __restrict__ cols, const T* __restrict__ vals,
	const T* __restrict__ x, int row, int sub, int r)
{
	typedef T T4 __attribute__((ext_vector_type(4)));
	const int end = ro[row + 1];
	T acc = 0;
	if constexpr (sizeof(T) == 8) {
		for (int k = ro[row] + sub; k < end; k += 16) {
			const T* a = vals + (size_t)k*16 + 4*r;
			const T* xv = x + 4*(size_t)cols[k];
			acc += a[0]*xv[0] + a[1]*xv[1] + a[2]*xv[2] + a[3]*xv[3];
		}
		return acc;
	}
	constexpr int kD = 4;  // blocks in flight per lane (8 measured slower: register pressure)
	for (int k0 = ro[row] + sub; k0 < end; k0 += 16*kD) {
		int c[kD];
#pragma unroll
		for (int u = 0; u < kD; ++u) c[u] = k0 + 16*u < end ? cols[k0 + 16*u] : -1;
		T4 a[kD], xv[kD];
#pragma unroll
		for (int u = 0; u < kD; ++u)
			if (c[u] >= 0) {
				a[u] = *reinterpret_cast<const T4*>(vals + (size_t)(k0 + 16*u)*16 + 4*r);
				xv[u] = *reinterpret_cast<const T4*>(x + 4*(size_t)c[u]);
			}
#pragma unroll
		for (int u = 0; u < kD; ++u)
			if (c[u] >= 0) acc += a[u].x*xv[u].x + a[u].y*xv[u].y + a[u].z*xv[u].z + a[u].w*xv[u].w;
	}
	return acc;
}

// x_out = x_in + omega D^-1 (b - A x_in).
template <class T>
__global__ void __launch_bounds__(256) SmoothKernel(int rows, const int* __restrict__ ro, const int* __restrict__ cols,
	const T* __restrict__ vals, const T* __restrict__ inv, const T* __restrict__ b, const T* __restrict__ xin,
	T* __restrict__ xout, T omega)
{
	const int lane = threadIdx.x & 63;
	const int row = blockIdx.x*4 + (threadIdx.x >> 6);
	if (row >= rows) return;
	const int sub = lane >> 2, r = lane & 3;
	T acc = RowPartial(ro, cols, vals, xin, row, sub, r);
	acc += __shfl_xor(acc, 4, 64);
	acc += __shfl_xor(acc, 8, 64);
	acc += __shfl_xor(acc, 16, 64);
	acc += __shfl_xor(acc, 32, 64);
	// lanes 0..3 hold row residual components after the butterfly
	const T res = b[4*(size_t)row + r] - acc;
	const T r0 = __shfl(res, 0, 64), r1 = __shfl(res, 1, 64), r2 = __shfl(res, 2, 64), r3 = __shfl(res, 3, 64);
	if (sub == 0) {
		const T* d = inv + (size_t)row*16 + 4*r;
		const T corr = d[0]*r0 + d[1]*r1 + d[2]*r2 + d[3]*r3;
		xout[4*(size_t)row + r] = xin[4*(size_t)row + r] + omega*corr;
	}
}

// One Chebyshev step (three-term form): z = D^-1 (b - A x_in), d = cd d + cz z,
// x_out = x_in + d.  d is per row, so it is updated in place.
template <class T>
__global__ void __launch_bounds__(256) ChebyshevKernel(int rows, const int* __restrict__ ro,
	const int* __restrict__ cols, const T* __restrict__ vals, const T* __restrict__ inv, const T* __restrict__ b,
	const T* __restrict__ xin, T* __restrict__ xout, T* __restrict__ d, T cd, T cz)
{
	const int lane = threadIdx.x & 63;
	const int row = blockIdx.x*4 + (threadIdx.x >> 6);
	if (row >= rows) return;
	const int sub = lane >> 2, r = lane & 3;
	T acc = RowPartial(ro, cols, vals, xin, row, sub, r);
	acc += __shfl_xor(acc, 4, 64);
	acc += __shfl_xor(acc, 8, 64);
	acc += __shfl_xor(acc, 16, 64);
	acc += __shfl_xor(acc, 32, 64);
	const T res = b[4*(size_t)row + r] - acc;
	const T r0 = __shfl(res, 0, 64), r1 = __shfl(res, 1, 64), r2 = __shfl(res, 2, 64), r3 = __shfl(res, 3, 64);
	if (sub == 0) {
		const size_t i = 4*(size_t)row + r;
		const T* dv = inv + (size_t)row*16 + 4*r;
		const T z = dv[0]*r0 + dv[1]*r1 + dv[2]*r2 + dv[3]*r3;
		const T dn = cd*d[i] + cz*z;
		d[i] = dn;
		xout[i] = xin[i] + dn;
	}
}

// r = b - A x
template <class T>
__global__ void __launch_bounds__(256) ResidualKernel(int rows, const int* __restrict__ ro, const int* __restrict__ cols,
	const T* __restrict__ vals, const T* __restrict__ b, const T* __restrict__ x, T* __restrict__ r)
{
	const int lane = threadIdx.x & 63;
	const int row = blockIdx.x*4 + (threadIdx.x >> 6);
	if (row >= rows) return;
	const int sub = lane >> 2, rr = lane & 3;
	T acc = 0;
	acc = RowPartial(ro, cols, vals, x, row, sub, rr);
	acc += __shfl_xor(acc, 4, 64);
	acc += __shfl_xor(acc, 8, 64);
	acc += __shfl_xor(acc, 16, 64);
	acc += __shfl_xor(acc, 32, 64);
	if (sub == 0) r[4*(size_t)row + rr] = b[4*(size_t)row + rr] - acc;
}

// Mixed precision, Chebyshev levels: the smoother reads S = D^-1 A, the
// block-Jacobi-scaled matrix, in FP16.  Its diagonal blocks are the identity
// and its other entries of order one, so FP16's 11-bit significand and range
// hold it (a level whose S has an entry above 60000 keeps the FP32 matrix).
// Half the bytes of FP32 blocks per smoothing pass.
// (S x) of one block row, by one wave: a lane takes whole blocks (all four
// rows, 32 bytes of S as two 16-byte loads, the 64 lanes 64 blocks a pass),
// then a butterfly over the 64 lanes; lane l returns row l % 4.
__device__ inline float RowProductHalf(const int* __restrict__ ro, const int* __restrict__ cols,
	const _Float16* __restrict__ s, const float* __restrict__ x, int row, int lane)
{
	typedef float F4 __attribute__((ext_vector_type(4)));
	typedef _Float16 H8 __attribute__((ext_vector_type(8)));
	const int end = ro[row + 1];
	float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f, a3 = 0.0f;
	for (int k = ro[row] + lane; k < end; k += 64) {
		const H8* blk = reinterpret_cast<const H8*>(s + (size_t)k*16);
		const H8 lo = blk[0], hi = blk[1];  // rows 0, 1 | rows 2, 3
		const F4 xv = *reinterpret_cast<const F4*>(x + 4*(size_t)cols[k]);
		a0 += (float)lo[0]*xv.x + (float)lo[1]*xv.y + (float)lo[2]*xv.z + (float)lo[3]*xv.w;
		a1 += (float)lo[4]*xv.x + (float)lo[5]*xv.y + (float)lo[6]*xv.z + (float)lo[7]*xv.w;
		a2 += (float)hi[0]*xv.x + (float)hi[1]*xv.y + (float)hi[2]*xv.z + (float)hi[3]*xv.w;
		a3 += (float)hi[4]*xv.x + (float)hi[5]*xv.y + (float)hi[6]*xv.z + (float)hi[7]*xv.w;
	}
#pragma unroll
	for (int o = 1; o < 64; o <<= 1) {
		a0 += __shfl_xor(a0, o, 64);
		a1 += __shfl_xor(a1, o, 64);
		a2 += __shfl_xor(a2, o, 64);
		a3 += __shfl_xor(a3, o, 64);
	}
	const int r = lane & 3;
	return r == 0 ? a0 : r == 1 ? a1 : r == 2 ? a2 : a3;
}

// S P: the FP16 blocks of S summed in FP32 over the lists of A P (16 lanes per block)
__global__ void ScaledGalerkinKernel(long long blocks, const long long* __restrict__ off, const int* __restrict__ list,
	const _Float16* __restrict__ s, float* __restrict__ out)
{
	const long long t = blockIdx.x*(long long)blockDim.x + threadIdx.x;
	const long long K = t >> 4;
	if (K >= blocks) return;
	const int e = t & 15;
	float v = 0.0f;
	const long long end = off[K + 1];
#pragma unroll 4
	for (long long k = off[K]; k < end; ++k) v += (float)s[(size_t)list[k]*16 + e];
	out[t] = v;
}

// S = D^-1 A in FP16 (D^-1 from the FP64 block inverses) and D in FP32; flag
// set when an entry of S is not finite or above 60000 in magnitude.
__global__ void __launch_bounds__(256) ScaleBlocksKernel(int rows, const int* __restrict__ ro,
	const int* __restrict__ diag, const double* __restrict__ vals, const double* __restrict__ inv,
	_Float16* __restrict__ s16, float* __restrict__ dblock, int* __restrict__ flag)
{
	const int lane = threadIdx.x & 63;
	const int row = blockIdx.x*4 + (threadIdx.x >> 6);
	if (row >= rows) return;
	const int sub = lane >> 2, r = lane & 3;
	const double* iv = inv + (size_t)row*16 + 4*r;
	bool bad = false;
	for (int k = ro[row] + sub; k < ro[row + 1]; k += 16) {
		const double* a = vals + (size_t)k*16;
#pragma unroll
		for (int c = 0; c < 4; ++c) {
			const double v = iv[0]*a[c] + iv[1]*a[4 + c] + iv[2]*a[8 + c] + iv[3]*a[12 + c];
			if (!(fabs(v) <= 60000.0)) bad = true;
			s16[(size_t)k*16 + 4*r + c] = static_cast<_Float16>(v);
		}
	}
	if (sub == 0)
		for (int c = 0; c < 4; ++c)
			dblock[(size_t)row*16 + 4*r + c] = static_cast<float>(vals[(size_t)diag[row]*16 + 4*r + c]);
	if (bad) atomicOr(flag, 1);
}

// The Chebyshev step of ChebyshevKernel on S: z = D^-1 b - S x_in.  The row's own entries are
// asked for ahead of the product (16.2 million blocks, 590 MB: 114 against 117 us,
// of the residual below 107 against 117).
__global__ void __launch_bounds__(256) ChebyshevScaledKernel(int rows, const int* __restrict__ ro,
	const int* __restrict__ cols, const _Float16* __restrict__ s, const float* __restrict__ inv,
	const float* __restrict__ b, const float* __restrict__ xin, float* __restrict__ xout, float* __restrict__ d,
	float cd, float cz)
{
	const int lane = threadIdx.x & 63;
	const int row = blockIdx.x*4 + (threadIdx.x >> 6);
	if (row >= rows) return;
	typedef float F4 __attribute__((ext_vector_type(4)));
	const size_t i = 4*(size_t)row + (lane & 3);
	const F4 iv = *reinterpret_cast<const F4*>(inv + 4*i), bv = *reinterpret_cast<const F4*>(b + 4*(size_t)row);
	const float d0 = d[i], x0 = xin[i];
	const float acc = RowProductHalf(ro, cols, s, xin, row, lane);
	if (lane < 4) {
		const float z = iv.x*bv.x + iv.y*bv.y + iv.z*bv.z + iv.w*bv.w - acc;
		const float dn = cd*d0 + cz*z;
		d[i] = dn;
		xout[i] = x0 + dn;
	}
}

// r = b - A x = D (D^-1 b - S x).
__global__ void __launch_bounds__(256) ResidualScaledKernel(int rows, const int* __restrict__ ro,
	const int* __restrict__ cols, const _Float16* __restrict__ s, const float* __restrict__ inv,
	const float* __restrict__ dblock, const float* __restrict__ b, const float* __restrict__ x,
	float* __restrict__ rout)
{
	const int lane = threadIdx.x & 63;
	const int row = blockIdx.x*4 + (threadIdx.x >> 6);
	if (row >= rows) return;
	typedef float F4 __attribute__((ext_vector_type(4)));
	const size_t i = 4*(size_t)row + (lane & 3);
	const F4 iv = *reinterpret_cast<const F4*>(inv + 4*i), bv = *reinterpret_cast<const F4*>(b + 4*(size_t)row);
	const F4 dv = *reinterpret_cast<const F4*>(dblock + 4*i);
	const float acc = RowProductHalf(ro, cols, s, x, row, lane);
	const float t = iv.x*bv.x + iv.y*bv.y + iv.z*bv.z + iv.w*bv.w - acc;
	const float t0 = __shfl(t, 0, 64), t1 = __shfl(t, 1, 64), t2 = __shfl(t, 2, 64), t3 = __shfl(t, 3, 64);
	if (lane < 4) rout[i] = dv.x*t0 + dv.y*t1 + dv.z*t2 + dv.w*t3;
}

// Power iteration for lambda_max of the Jacobi-preconditioned operator, without
// a host in the loop: y = D^-1 A x / sqrt(*sq) with sq = ||x||^2 from the step
// before, and per workgroup the sum of the squares of its y.  (With the norms
// read back to the host a step of 42,000 rows took 96 us for 54 us of product.)
__global__ void __launch_bounds__(256) DinvAKernel(int rows, const int* __restrict__ ro, const int* __restrict__ cols,
	const double* __restrict__ vals, const double* __restrict__ inv, const double* __restrict__ x,
	const double* __restrict__ sq, double* __restrict__ y, double* __restrict__ partial)
{
	__shared__ double lds[4];
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const int sub = lane >> 2, r = lane & 3;
	const double scale = 1.0/sqrt(*sq);
	double total = 0.0;
	for (int row = blockIdx.x*4 + wave; row < rows; row += 4*gridDim.x) {
		double acc = RowPartial(ro, cols, vals, x, row, sub, r);
		acc += __shfl_xor(acc, 4, 64);
		acc += __shfl_xor(acc, 8, 64);
		acc += __shfl_xor(acc, 16, 64);
		acc += __shfl_xor(acc, 32, 64);
		const double a0 = __shfl(acc, 0, 64), a1 = __shfl(acc, 1, 64), a2 = __shfl(acc, 2, 64), a3 = __shfl(acc, 3, 64);
		if (sub == 0) {
			const double* d = inv + (size_t)row*16 + 4*r;
			const double v = scale*(d[0]*a0 + d[1]*a1 + d[2]*a2 + d[3]*a3);
			y[4*(size_t)row + r] = v;
			total += v*v;
		}
	}
	total = WaveSumT(total);
	if (lane == 0) lds[wave] = total;
	__syncthreads();
	if (threadIdx.x == 0) partial[blockIdx.x] = lds[0] + lds[1] + lds[2] + lds[3];
}

// Deterministic pseudo-random start vector in [-1, 1), and per workgroup the sum of its squares.
__global__ void __launch_bounds__(256) HashVectorKernel(long long n, double* __restrict__ v, double* __restrict__ partial)
{
	__shared__ double lds[4];
	double total = 0.0;
	for (long long i = blockIdx.x*(long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x*blockDim.x) {
		unsigned long long z = (unsigned long long)i*0x9e3779b97f4a7c15ULL + 0x632be59bd9b4e019ULL;
		z = (z ^ (z >> 30))*0xbf58476d1ce4e5b9ULL;
		z = (z ^ (z >> 27))*0x94d049bb133111ebULL;
		z ^= z >> 31;
		const double h = (double)(z >> 11)*(2.0/9007199254740992.0) - 1.0;
		v[i] = h;
		total += h*h;
	}
	total = WaveSumT(total);
	if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = total;
	__syncthreads();
	if (threadIdx.x == 0) partial[blockIdx.x] = lds[0] + lds[1] + lds[2] + lds[3];
}

// *out = sum of partial[0 .. count), one workgroup
constexpr int kSumThreads = 1024;
__global__ void __launch_bounds__(kSumThreads) SumKernel(const double* __restrict__ partial, int count,
	double* __restrict__ out)
{
	__shared__ double lds[kSumThreads/64];
	double total = 0.0;
#pragma unroll 4
	for (int i = threadIdx.x; i < count; i += kSumThreads) total += partial[i];
	total = WaveSumT(total);
	if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = total;
	__syncthreads();
	if (threadIdx.x < 64) {
		total = WaveSumT(threadIdx.x < kSumThreads/64 ? lds[threadIdx.x] : 0.0);
		if (threadIdx.x == 0) *out = total;
	}
}

// One colour of a block Gauss-Seidel sweep, in place: for the rows of this
// colour (no two of them are coupled) x_i += D_i^-1 (b_i - sum_j A_ij x_j).
template <class T>
__global__ void __launch_bounds__(256) GsColorKernel(int count, const int* __restrict__ list, const int* __restrict__ ro,
	const int* __restrict__ cols, const T* __restrict__ vals, const T* __restrict__ inv, const T* __restrict__ b,
	T* __restrict__ x)
{
	const int lane = threadIdx.x & 63;
	const int item = blockIdx.x*4 + (threadIdx.x >> 6);
	if (item >= count) return;
	const int row = list[item];
	const int sub = lane >> 2, r = lane & 3;
	T acc = 0;
	acc = RowPartial(ro, cols, vals, static_cast<const T*>(x), row, sub, r);
	acc += __shfl_xor(acc, 4, 64);
	acc += __shfl_xor(acc, 8, 64);
	acc += __shfl_xor(acc, 16, 64);
	acc += __shfl_xor(acc, 32, 64);
	const T res = b[4*(size_t)row + r] - acc;
	const T r0 = __shfl(res, 0, 64), r1 = __shfl(res, 1, 64), r2 = __shfl(res, 2, 64), r3 = __shfl(res, 3, 64);
	if (sub == 0) {
		const T* d = inv + (size_t)row*16 + 4*r;
		x[4*(size_t)row + r] += d[0]*r0 + d[1]*r1 + d[2]*r2 + d[3]*r3;
	}
}

// bc[I] = sum_{i in aggregate I} r[i]: 16 lanes per aggregate, lane (m, c)
// every fourth member's component c (one lane per component walked the 20 to 30
// members one after the other: 15 us for 150,000 rows, whatever their bytes)
template <class T>
__global__ void __launch_bounds__(256) RestrictKernel(int coarse, const int* __restrict__ aoff,
	const int* __restrict__ amem, const T* __restrict__ r, T* __restrict__ bc)
{
	const int t = blockIdx.x*blockDim.x + threadIdx.x;
	const int I = t >> 4, m = (t >> 2) & 3, c = t & 3;
	T s = 0;
	if (I < coarse)
#pragma unroll 4
		for (int k = aoff[I] + m; k < aoff[I + 1]; k += 4) s += r[4*(size_t)amem[k] + c];
	s += __shfl_xor(s, 4, 64);
	s += __shfl_xor(s, 8, 64);
	if (I < coarse && m == 0) bc[4*(size_t)I + c] = s;
}

// x[i] += xc[agg[i]]
template <class T>
__global__ void ProlongKernel(int fine, const int* __restrict__ agg, const T* __restrict__ xc, T* __restrict__ x)
{
	const int t = blockIdx.x*blockDim.x + threadIdx.x;
	const int i = t >> 2, c = t & 3;
	if (i >= fine) return;
	x[4*(size_t)i + c] += xc[4*(size_t)agg[i] + c];
}

// First smoothing step from x = 0: d = cz D^-1 b, x = d.
template <class T>
__global__ void FirstStepKernel(int rows, const T* __restrict__ inv, const T* __restrict__ b, T* __restrict__ x,
	T* __restrict__ d, T cz)
{
	const int t = blockIdx.x*blockDim.x + threadIdx.x;
	const int row = t >> 2;
	if (row >= rows) return;
	const T* dv = inv + 4*(size_t)t;
	const T* bv = b + 4*(size_t)row;
	const T v = cz*(dv[0]*bv[0] + dv[1]*bv[1] + dv[2]*bv[2] + dv[3]*bv[3]);
	d[t] = v;
	x[t] = v;
}

// Coarse correction and first smoothing step after it: with A P xc from the
// row's blocks of A P, d = cz D^-1 (r - A P xc) and x += xc[agg] + d, in place;
// d takes the place of r.  kScaled: ap holds S P, S = D^-1 A as the level's other
// steps read it, and d = cz (D^-1 r - S P xc).
// A row of A P holds some 14 blocks, one pass of loads: the time is the chain of
// loads of a wave times the waves, so two rows a wave, 32 lanes each, and the row's
// own entries asked for ahead of the product.  150,000 rows, 2.1 million blocks
// (64 bytes each in FP32, 26 us at the read rate): 42 us, with one row a wave and
// its entries after the product 69 us; 42,000 rows 14.6 against 21.8 us.
template <class T, bool kScaled>
__global__ void __launch_bounds__(256) CorrectStepKernel(int rows, const int* __restrict__ ro,
	const int* __restrict__ cols, const T* __restrict__ ap, const T* __restrict__ inv, const int* __restrict__ agg,
	const T* __restrict__ xc, T* __restrict__ x, T* __restrict__ rd, T cz)
{
	typedef T T4 __attribute__((ext_vector_type(4)));
	const int lane = threadIdx.x & 63;
	const int row = blockIdx.x*8 + (threadIdx.x >> 5);
	const int sub = (lane & 31) >> 2, r = lane & 3;
	const bool live = row < rows;
	const int begin = live ? ro[row] : 0, end = live ? ro[row + 1] : 0;
	const size_t i = live ? 4*(size_t)row + r : r;
	const T4 dv = *reinterpret_cast<const T4*>(inv + 4*i);
	const T x0 = x[i], rd0 = rd[i], xa = xc[4*(size_t)agg[i >> 2] + r];
	constexpr int kD = sizeof(T) == 8 ? 2 : 4;  // blocks in flight per lane
	T acc = 0;
	for (int k0 = begin + sub; k0 < end; k0 += 8*kD) {
		T4 a[kD], xv[kD];
#pragma unroll
		for (int u = 0; u < kD; ++u) {
			const int k = min(k0 + 8*u, end - 1);
			a[u] = *reinterpret_cast<const T4*>(ap + (size_t)k*16 + 4*r);
			xv[u] = *reinterpret_cast<const T4*>(xc + 4*(size_t)cols[k]);
		}
#pragma unroll
		for (int u = 0; u < kD; ++u)
			if (k0 + 8*u < end) acc += a[u].x*xv[u].x + a[u].y*xv[u].y + a[u].z*xv[u].z + a[u].w*xv[u].w;
	}
	acc += __shfl_xor(acc, 4, 64);
	acc += __shfl_xor(acc, 8, 64);
	acc += __shfl_xor(acc, 16, 64);
	const T res = kScaled ? rd0 : rd0 - acc;
	const int base = lane & 32;
	const T r0 = __shfl(res, base, 64), r1 = __shfl(res, base + 1, 64), r2 = __shfl(res, base + 2, 64),
		r3 = __shfl(res, base + 3, 64);
	if (live && sub == 0) {
		T z = dv.x*r0 + dv.y*r1 + dv.z*r2 + dv.w*r3;
		if (kScaled) z -= acc;
		const T d = cz*z;
		rd[i] = d;
		x[i] = x0 + (xa + d);
	}
}

// coarse[K] = sum of fine blocks list[off[K]..off[K+1]) (16 lanes per block): A P from A, the coarse
// blocks from A P (from A itself, in one gather, each block's list spans rows far apart: 760 against
// 430 us for 16.2 million blocks)
__global__ void GalerkinKernel(long long cblocks, const long long* __restrict__ off, const int* __restrict__ list,
	const double* __restrict__ fine, double* __restrict__ coarse)
{
	const long long t = blockIdx.x*(long long)blockDim.x + threadIdx.x;
	const long long K = t >> 4;
	const int e = t & 15;
	if (K >= cblocks) return;
	double s = 0.0;
	const long long end = off[K + 1];
#pragma unroll 4
	for (long long k = off[K]; k < end; ++k) s += fine[(size_t)list[k]*16 + e];
	coarse[(size_t)K*16 + e] = s;
}

// The coarsest level as a dense matrix, on a zero-filled n x n buffer (n = 4 rows).
__global__ void DenseKernel(int rows, const int* __restrict__ ro, const int* __restrict__ cols,
	const double* __restrict__ vals, double* __restrict__ dense)
{
	const int i = blockIdx.x;
	const int n = 4*rows;
	for (int k = ro[i]; k < ro[i + 1]; ++k)
		for (int e = threadIdx.x; e < 16; e += blockDim.x)
			dense[(size_t)(4*i + (e >> 2))*n + 4*cols[k] + (e & 3)] = vals[(size_t)k*16 + e];
}

// Dense inverse by in-place Gauss-Jordan elimination with partial pivoting, in
// panels of kPanel columns: no row is moved, column p is exchanged with the row
// r_p it is pivoted on, and at the end inverse[p][r_k] = matrix[r_p][k].
//
// Bound by latency: a pivot needs the column of the pivot before.  A launch
// per pivot plus one for the elimination cost 10.7 us each pivot (676 rows: 7.3
// ms); a panel keeps its columns in the registers of one workgroup, a row per
// thread, where a pivot is one barrier (20.8 us for 16 pivots and the launch),
// and the columns outside the panel take all its pivots as one product of rank
// kPanel over the whole grid (7.3 us): 1.2 ms.  16 columns: 32 registers of a
// thread's 128 at 1024 threads.
constexpr int kPanel = 16;
constexpr int kDenseMax = 1024;   // rows the panel's workgroup holds
constexpr int kUpdateRows = 32;   // rows of a workgroup of PanelUpdateKernel

// Largest value over the wave (0 where a lane has no source), the same in every lane.
__device__ inline unsigned int WaveMax(unsigned int v)
{
	v = max(v, (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false));  // row_shr:1
	v = max(v, (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false));  // row_shr:2
	v = max(v, (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false));  // row_shr:4
	v = max(v, (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false));  // row_shr:8
	v = max(v, (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));  // row_bcast:15
	v = max(v, (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));  // row_bcast:31
	return (unsigned int)__builtin_amdgcn_readlane((int)v, 63);
}

// Pivots columns p0 .. p0 + width - 1.  step[i] is the column row i is pivot
// of, n if none yet; pivot[p] the pivot row of column p; w[t][i] the panel's
// columns afterwards, column by column.  The pivot is the row of the largest
// magnitude to 20 bits of the significand (the upper word of the entry orders
// them), the lowest row on ties.  Every wave offers its best row, scaled as
// pivot row, and after one barrier all threads choose among the at most 16
// offers.  A thread's row is rotated by one column per pivot, so that the loop
// indexes registers by constants and stays small: unrolled over the panel's 16
// pivots the code (35 KB) ran at the rate it was fetched.  The panel is read and
// written by columns (in[row*row_stride + t*column_stride]): neighbouring
// threads, neighbouring addresses.
__global__ void __launch_bounds__(kDenseMax) PanelKernel(int n, int p0, int width, const double* __restrict__ in,
	int row_stride, int column_stride, double* __restrict__ w, int* __restrict__ step, int* __restrict__ pivot,
	int* __restrict__ status)
{
	constexpr int kWaves = kDenseMax/64;
	__shared__ unsigned int key[2][kWaves];
	__shared__ int key_row[2][kWaves];
	__shared__ double offer[2][kWaves][kPanel];
	const int i = threadIdx.x, lane = i & 63, wave = i >> 6;
	if (i < 2*kWaves) key[i/kWaves][i % kWaves] = 0;  // waves the workgroup does not have
	int mine = i < n ? step[i] : 0;
	double a[kPanel];
#pragma unroll
	for (int t = 0; t < kPanel; ++t)
		a[t] = i < n && t < width ? in[(size_t)i*row_stride + (size_t)t*column_stride] : 0.0;
	__syncthreads();
#pragma unroll 1
	for (int c = 0; c < width; ++c) {
		const int buf = c & 1;
		// a row without a pivot: 1 + upper word of |entry| (1 for a NaN, which is never chosen over a number)
		unsigned int k = 0;
		if (mine == n) k = a[0] == a[0] ? 1u + ((unsigned int)__double2hiint(a[0]) & 0x7fffffffu) : 1u;
		const double inv = a[0] != 0.0 ? 1.0/a[0] : 0.0;
		const unsigned int m = WaveMax(k);
		const int first = __ffsll(__ballot(k == m)) - 1;
		if (lane == first) {
			key[buf][wave] = m;
			key_row[buf][wave] = i;
			offer[buf][wave][0] = inv;
#pragma unroll
			for (int t = 1; t < kPanel; ++t) offer[buf][wave][t] = a[t]*inv;
		}
		__syncthreads();
		// lane l of every wave reads offer l; the pivot row goes through scalar registers
		const unsigned int o = key[buf][lane & (kWaves - 1)];
		const int win = __ffsll(__ballot(o == WaveMax(o))) - 1;
		const int chosen = __builtin_amdgcn_readlane(key_row[buf][lane & (kWaves - 1)], win);
		const double part = offer[buf][win][lane & (kPanel - 1)];
		double row[kPanel];
#pragma unroll
		for (int t = 0; t < kPanel; ++t)
			row[t] = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(part), t),
				__builtin_amdgcn_readlane(__double2loint(part), t));
		const double f = a[0];
		if (i == chosen) {
			if (!(fabs(f) > 1e-300) || !isfinite(f)) *status = 1;
			mine = p0 + c;
			pivot[p0 + c] = i;
#pragma unroll
			for (int t = 1; t < kPanel; ++t) a[t - 1] = row[t];
			a[kPanel - 1] = row[0];
		} else {
#pragma unroll
			for (int t = 1; t < kPanel; ++t) a[t - 1] = a[t] - f*row[t];
			a[kPanel - 1] = -f*row[0];
		}
	}
	if (i < n) {
		step[i] = mine;
#pragma unroll
		for (int t = 0; t < kPanel; ++t) w[(size_t)((t + width) % kPanel)*n + i] = a[t];
	}
}

// The panel's pivots applied to the whole matrix, from one buffer to another:
// out[i][j] = (row i is a pivot of the panel ? 0 : in[i][j]) + sum_t w[t][i] in[pivot[p0 + t]][j],
// and the panel's own columns are w.  The columns of the next panel go to next
// as well, column by column.
__global__ void __launch_bounds__(256) PanelUpdateKernel(int n, int p0, int width, const double* __restrict__ in,
	const double* __restrict__ w, const int* __restrict__ step, const int* __restrict__ pivot, double* __restrict__ out,
	double* __restrict__ next)
{
	constexpr int kRows = kUpdateRows/4;  // rows of a wave
	__shared__ double ws[kUpdateRows][kPanel + 1];
	__shared__ int keep[kUpdateRows];
	__shared__ double ps[kPanel][64];  // the pivot rows
	const int j = blockIdx.x*64 + (threadIdx.x & 63), i0 = blockIdx.y*kUpdateRows;
	for (int k = threadIdx.x; k < kUpdateRows*kPanel; k += 256)
		ws[k % kUpdateRows][k/kUpdateRows] = i0 + k % kUpdateRows < n ? w[(size_t)(k/kUpdateRows)*n + i0 + k % kUpdateRows] : 0.0;
	if (threadIdx.x < kUpdateRows) {
		const int s = i0 + threadIdx.x < n ? step[i0 + threadIdx.x] : 0;
		keep[threadIdx.x] = !(s >= p0 && s < p0 + width);
	}
	for (int t = threadIdx.x >> 6; t < kPanel; t += 4)
		ps[t][threadIdx.x & 63] = t < width && j < n ? in[(size_t)pivot[p0 + t]*n + j] : 0.0;
	__syncthreads();
	if (j >= n) return;
	const int r0 = (threadIdx.x >> 6)*kRows;
	const bool panel = j >= p0 && j < p0 + width;
	double acc[kRows];
#pragma unroll
	for (int r = 0; r < kRows; ++r) acc[r] = i0 + r0 + r < n && keep[r0 + r] ? in[(size_t)(i0 + r0 + r)*n + j] : 0.0;
#pragma unroll 4
	for (int t = 0; t < kPanel; ++t) {
		const double p = ps[t][threadIdx.x & 63];
#pragma unroll
		for (int r = 0; r < kRows; ++r) acc[r] += ws[r0 + r][t]*p;
	}
#pragma unroll
	for (int r = 0; r < kRows; ++r)
		if (i0 + r0 + r < n) {
			out[(size_t)(i0 + r0 + r)*n + j] = panel ? ws[r0 + r][j - p0] : acc[r];
			if (j >= p0 + kPanel && j < p0 + 2*kPanel) next[(size_t)(j - p0 - kPanel)*n + i0 + r0 + r] = acc[r];
		}
}

// inverse (n x n, in T) from the eliminated matrix: inverse[p][r_k] = matrix[r_p][k], one row p per workgroup
template <class T>
__global__ void ExtractInverseKernel(int n, const double* __restrict__ matrix, const int* __restrict__ pivot,
	T* __restrict__ inv)
{
	const int p = blockIdx.x;
	const double* row = matrix + (size_t)pivot[p]*n;
	for (int k = threadIdx.x; k < n; k += blockDim.x) inv[(size_t)p*n + pivot[k]] = static_cast<T>(row[k]);
}

// y = Dinv b (dense), one wave per row
template <class T>
__global__ void DenseApplyKernel(int n, const T* __restrict__ inv, const T* __restrict__ b, T* __restrict__ y)
{
	const int row = blockIdx.x*4 + (threadIdx.x >> 6);
	const int lane = threadIdx.x & 63;
	if (row >= n) return;
	T acc = 0;
	for (int j = lane; j < n; j += 64) acc += inv[(size_t)row*n + j]*b[j];
	acc = WaveSumT(acc);
	if (lane == 0) y[row] = acc;
}

__global__ void ToFloatKernel2(long long n, const double* __restrict__ x, float* __restrict__ y)
{
	for (long long i = blockIdx.x*(long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x*blockDim.x)
		y[i] = static_cast<float>(x[i]);
}

__global__ void ToDoubleKernel(long long n, const float* __restrict__ x, double* __restrict__ y)
{
	for (long long i = blockIdx.x*(long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x*blockDim.x)
		y[i] = static_cast<double>(x[i]);
}

__global__ void BlockInverseT32Kernel(long long n, const double* __restrict__ x, float* __restrict__ y)
{
	for (long long i = blockIdx.x*(long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x*blockDim.x)
		y[i] = static_cast<float>(x[i]);
}

int Grid(long long threads, int block = 256)
{
	long long b = (threads + block - 1)/block;
	return static_cast<int>(std::max<long long>(1, std::min<long long>(b, 1LL << 30)));
}

}  // namespace

struct Level {
	int rows = 0;
	long long nnzb = 0;
	// pattern (level 0 borrows the mesh pattern)
	DevBuf<int> ro_own, cols_own, diag_own;
	const int* ro = nullptr;
	const int* cols = nullptr;
	const int* diag = nullptr;
	std::vector<int> h_ro, h_cols, h_diag;
	DevBuf<double> vals;          // own values (levels >= 1)
	const double* vals64 = nullptr;
	DevBuf<double> inv64;
	DevBuf<float> vals32_own, inv32;
	const float* vals32 = nullptr;
	// mixed precision, Chebyshev levels only: S = D^-1 A in FP16 and D in FP32.  scaled: S fits
	// FP16, the level's steps read it and ap32 holds S P; else they read A and ap32 holds A P
	DevBuf<_Float16> s16;
	DevBuf<float> dblock32;
	bool scaled = false;
	// transfer to the next level
	DevBuf<int> agg, aoff, amem;
	// A P: its pattern, the fine blocks of each of its blocks, its values
	DevBuf<int> ap_ro, ap_cols, ap_list;
	DevBuf<long long> ap_off;
	DevBuf<double> ap64;
	DevBuf<float> ap32;
	long long ap_nnzb = 0;
	DevBuf<long long> goff;       // the blocks of A P of each block of the NEXT level
	DevBuf<int> glist;
	// multicolour Gauss-Seidel (gs) or damped block Jacobi; rows grouped by colour
	bool gs = false;
	std::vector<int> color_offsets;
	DevBuf<int> color_rows;
	double lambda_max = 1.0;
	// vectors
	DevBuf<double> x64, y64, b64, r64;
	DevBuf<float> x32, y32, b32, r32;
	BsrView view() const { return {rows, nnzb, ro, cols, diag}; }
};

struct Amg::Impl {
	tfi_mesh* mesh;
	tfi_ctx* ctx;
	int precision;
	AmgOptions opt;
	bool built = false;
	std::vector<std::unique_ptr<Level>> L;
	int nc = 0;  // coarsest dense size (4 * rows)
	DevBuf<double> dense[2], panel, next_panel, dinv64;  // the coarsest matrix under elimination, from one buffer to the other
	DevBuf<float> dinv32;
	DevBuf<int> status, pivot, step;
	DevBuf<int> scale_flags;  // per level: S did not fit FP16
	DevBuf<double> power[2], power_partial, squares;  // power iteration; per level ||D^-1 A x||^2 of its last step

	void Symbolic(const double* fine_values);
	void Numeric(const double* fine_values64, const float* fine_values32);
	void Colour(Level& v);
	template <class T>
	void Cycle(int l, const T* b, T* x);
	void Coarsen(Level& fine, const double* fine_values, Level& coarse);
};

namespace {

// Strength of connection between block rows i and j: the largest coupling of
// one field with itself, scaled by the two field diagonals,
//   s_ij = max_f |A_ij[f][f]| / sqrt(|A_ii[f][f]| |A_jj[f][f]|),
// symmetrised (max of s_ij, s_ji) so that Dirichlet rows (identity velocity
// rows) stay connected through their pressure couplings.  j is strong for i
// when s_ij >= theta * max(rowmax_i, rowmax_j) -- a row-relative threshold.
// Greedy aggregation in node order (deterministic): roots whose strong
// neighbours are all free, then attach, then leftovers.
std::vector<int> Aggregate(int n, const std::vector<int>& ro, const std::vector<int>& cols,
	const std::vector<double>& vals, double theta, int& count)
{
	std::vector<double> dg(4LL*n, 0.0);
	for (int i = 0; i < n; ++i)
		for (int k = ro[i]; k < ro[i + 1]; ++k)
			if (cols[k] == i)
				for (int f = 0; f < 4; ++f) dg[4LL*i + f] = std::abs(vals[(size_t)k*16 + 5*f]);
	const long long nnz = ro[n];
	std::vector<double> s(nnz, 0.0);
	for (int i = 0; i < n; ++i)
		for (int k = ro[i]; k < ro[i + 1]; ++k) {
			const int j = cols[k];
			if (j == i) continue;
			double best = 0.0;
			for (int f = 0; f < 4; ++f) {
				const double d = dg[4LL*i + f]*dg[4LL*j + f];
				if (d > 0.0) best = std::max(best, std::abs(vals[(size_t)k*16 + 5*f])/std::sqrt(d));
			}
			s[k] = best;
		}
	// symmetrise through the (structurally symmetric) pattern
	std::vector<double> sym(s);
	for (int i = 0; i < n; ++i)
		for (int k = ro[i]; k < ro[i + 1]; ++k) {
			const int j = cols[k];
			if (j == i) continue;
			const int* b = cols.data() + ro[j];
			const int* e = cols.data() + ro[j + 1];
			const int* it = std::lower_bound(b, e, i);
			if (it != e && *it == i) sym[k] = std::max(s[k], s[it - cols.data()]);
		}
	std::vector<double> rowmax(n, 0.0);
	for (int i = 0; i < n; ++i)
		for (int k = ro[i]; k < ro[i + 1]; ++k) rowmax[i] = std::max(rowmax[i], sym[k]);
	std::vector<int> sro(n + 1, 0), scols;
	std::vector<double> sval;
	for (int i = 0; i < n; ++i) {
		for (int k = ro[i]; k < ro[i + 1]; ++k) {
			const int j = cols[k];
			if (j == i || sym[k] <= 0.0) continue;
			if (sym[k] >= theta*std::max(rowmax[i], rowmax[j])) {
				scols.push_back(j);
				sval.push_back(sym[k]);
			}
		}
		sro[i + 1] = static_cast<int>(scols.size());
	}
	std::vector<int> agg(n, -1);
	count = 0;
	for (int i = 0; i < n; ++i) {
		if (agg[i] >= 0 || sro[i + 1] == sro[i]) continue;
		bool free = true;
		for (int k = sro[i]; k < sro[i + 1] && free; ++k) free = agg[scols[k]] < 0;
		if (!free) continue;
		agg[i] = count;
		for (int k = sro[i]; k < sro[i + 1]; ++k) agg[scols[k]] = count;
		++count;
	}
	std::vector<int> pass2(n, -1);
	for (int i = 0; i < n; ++i) {
		if (agg[i] >= 0) continue;
		double best = -1.0;
		for (int k = sro[i]; k < sro[i + 1]; ++k)
			if (agg[scols[k]] >= 0 && sval[k] > best) {
				best = sval[k];
				pass2[i] = agg[scols[k]];
			}
	}
	for (int i = 0; i < n; ++i)
		if (agg[i] < 0 && pass2[i] >= 0) agg[i] = pass2[i];
	for (int i = 0; i < n; ++i) {
		if (agg[i] >= 0) continue;
		agg[i] = count;
		for (int k = sro[i]; k < sro[i + 1]; ++k)
			if (agg[scols[k]] < 0) agg[scols[k]] = count;
		++count;
	}
	return agg;
}

}  // namespace

// Greedy node colouring of a Gauss-Seidel level (rows of a colour are uncoupled).
void Amg::Impl::Colour(Level& v)
{
	std::vector<int> col(v.rows, -1), mark;
	int ncol = 0;
	for (int i = 0; i < v.rows; ++i) {
		if ((int)mark.size() < ncol + 1) mark.resize(ncol + 1, -1);
		for (int k = v.h_ro[i]; k < v.h_ro[i + 1]; ++k) {
			const int c = col[v.h_cols[k]];
			if (c >= 0) mark[c] = i;
		}
		int c = 0;
		while (c < ncol && mark[c] == i) ++c;
		if (c == ncol) ++ncol;
		col[i] = c;
	}
	v.color_offsets.assign(ncol + 1, 0);
	for (int i = 0; i < v.rows; ++i) ++v.color_offsets[col[i] + 1];
	for (int c = 0; c < ncol; ++c) v.color_offsets[c + 1] += v.color_offsets[c];
	std::vector<int> rows(v.rows);
	std::vector<int> fill(v.color_offsets.begin(), v.color_offsets.end() - 1);
	for (int i = 0; i < v.rows; ++i) rows[fill[col[i]]++] = i;
	v.color_rows.Allocate(ctx, v.rows);
	v.color_rows.Upload(rows.data(), v.rows);
}

void Amg::Impl::Symbolic(const double* fine_values)
{
	L.clear();
	auto l0 = std::make_unique<Level>();
	l0->rows = mesh->nodes;
	l0->nnzb = mesh->nnzb;
	l0->ro = mesh->row_offsets.data();
	l0->cols = mesh->columns.data();
	l0->diag = mesh->diagonal.data();
	l0->h_ro.resize(mesh->nodes + 1);
	l0->h_cols.resize(mesh->nnzb);
	l0->h_diag.resize(mesh->nodes);
	mesh->row_offsets.Download(l0->h_ro.data(), mesh->nodes + 1);
	mesh->columns.Download(l0->h_cols.data(), mesh->nnzb);
	mesh->diagonal.Download(l0->h_diag.data(), mesh->nodes);
	std::vector<double> hv(mesh->nnzb*16);
	Check(hipMemcpyAsync(hv.data(), fine_values, hv.size()*sizeof(double), hipMemcpyDeviceToHost, ctx->stream),
		"amg download");
	Sync(ctx);
	L.push_back(std::move(l0));
	while ((int)L.size() < kMaxLevels && L.back()->rows > opt.coarse_nodes) {
		Level& f = *L.back();
		int count = 0;
		auto agg = Aggregate(f.rows, f.h_ro, f.h_cols, hv, kStrength, count);
		if (count >= f.rows*0.9 || count < 1) break;  // coarsening stalled
		// aggregate membership lists
		std::vector<int> aoff(count + 1, 0), amem(f.rows);
		for (int i = 0; i < f.rows; ++i) ++aoff[agg[i] + 1];
		for (int c = 0; c < count; ++c) aoff[c + 1] += aoff[c];
		{
			std::vector<int> fill(aoff.begin(), aoff.end() - 1);
			for (int i = 0; i < f.rows; ++i) amem[fill[agg[i]]++] = i;
		}
		// pattern of A P: the aggregates of each row's columns, ascending; the
		// fine blocks of each of its blocks, ascending
		std::vector<int> ap_ro(f.rows + 1, 0), ap_cols, ap_list(f.nnzb), touched, place(count, -1);
		std::vector<long long> ap_off(1, 0);
		ap_cols.reserve(f.nnzb/4);
		ap_off.reserve(f.nnzb/4);
		std::vector<int> fill;
		for (int i = 0; i < f.rows; ++i) {
			const int begin = f.h_ro[i], end = f.h_ro[i + 1];
			touched.clear();
			for (int k = begin; k < end; ++k) {
				const int J = agg[f.h_cols[k]];
				if (place[J] < 0) {
					place[J] = 0;
					touched.push_back(J);
				}
				++place[J];
			}
			std::sort(touched.begin(), touched.end());
			fill.clear();
			for (int J : touched) {
				const int members = place[J];
				place[J] = static_cast<int>(fill.size());
				fill.push_back(static_cast<int>(ap_off.back()));
				ap_cols.push_back(J);
				ap_off.push_back(ap_off.back() + members);
			}
			for (int k = begin; k < end; ++k) ap_list[fill[place[agg[f.h_cols[k]]]]++] = k;
			for (int J : touched) place[J] = -1;
			ap_ro[i + 1] = static_cast<int>(ap_cols.size());
		}
		f.ap_nnzb = ap_ro[f.rows];
		// coarse pattern: the union of the rows of A P of an aggregate's members; the
		// blocks of A P of each coarse block in the order of the members
		auto c = std::make_unique<Level>();
		c->rows = count;
		c->h_ro.assign(count + 1, 0);
		c->h_diag.assign(count, -1);
		std::vector<int> list(f.ap_nnzb);
		std::vector<long long> cnt(1, 0);
		long long written = 0;
		for (int I = 0; I < count; ++I) {
			touched.clear();
			for (int m = aoff[I]; m < aoff[I + 1]; ++m)
				for (int k = ap_ro[amem[m]]; k < ap_ro[amem[m] + 1]; ++k) {
					const int J = ap_cols[k];
					if (place[J] < 0) {
						place[J] = 0;
						touched.push_back(J);
					}
					++place[J];
				}
			std::sort(touched.begin(), touched.end());
			fill.clear();
			for (int J : touched) {
				const int members = place[J];
				place[J] = static_cast<int>(fill.size());
				fill.push_back(static_cast<int>(cnt.back()));
				if (J == I) c->h_diag[I] = static_cast<int>(written);
				c->h_cols.push_back(J);
				cnt.push_back(cnt.back() + members);
				++written;
			}
			for (int m = aoff[I]; m < aoff[I + 1]; ++m)
				for (int k = ap_ro[amem[m]]; k < ap_ro[amem[m] + 1]; ++k) list[fill[place[ap_cols[k]]]++] = k;
			for (int J : touched) place[J] = -1;
			c->h_ro[I + 1] = static_cast<int>(written);
		}
		c->nnzb = written;
		f.agg.Allocate(ctx, f.rows);
		f.agg.Upload(agg.data(), f.rows);
		f.aoff.Allocate(ctx, count + 1);
		f.aoff.Upload(aoff.data(), count + 1);
		f.amem.Allocate(ctx, f.rows);
		f.amem.Upload(amem.data(), f.rows);
		f.ap_ro.Allocate(ctx, f.rows + 1);
		f.ap_ro.Upload(ap_ro.data(), f.rows + 1);
		f.ap_cols.Allocate(ctx, f.ap_nnzb);
		f.ap_cols.Upload(ap_cols.data(), f.ap_nnzb);
		f.ap_off.Allocate(ctx, f.ap_nnzb + 1);
		f.ap_off.Upload(ap_off.data(), f.ap_nnzb + 1);
		f.ap_list.Allocate(ctx, f.nnzb);
		f.ap_list.Upload(ap_list.data(), f.nnzb);
		f.ap64.Allocate(ctx, f.ap_nnzb*16);
		if (precision == TFI_MIXED) f.ap32.Allocate(ctx, f.ap_nnzb*16);
		f.goff.Allocate(ctx, c->nnzb + 1);
		f.goff.Upload(cnt.data(), c->nnzb + 1);
		f.glist.Allocate(ctx, f.ap_nnzb);
		f.glist.Upload(list.data(), f.ap_nnzb);
		c->ro_own.Allocate(ctx, count + 1);
		c->ro_own.Upload(c->h_ro.data(), count + 1);
		c->cols_own.Allocate(ctx, c->nnzb);
		c->cols_own.Upload(c->h_cols.data(), c->nnzb);
		c->diag_own.Allocate(ctx, count);
		c->diag_own.Upload(c->h_diag.data(), count);
		c->ro = c->ro_own.data();
		c->cols = c->cols_own.data();
		c->diag = c->diag_own.data();
		c->vals.Allocate(ctx, c->nnzb*16);
		// coarse values now (the next aggregation needs them)
		Coarsen(f, L.size() == 1 ? fine_values : f.vals.data(), *c);
		hv.assign(c->nnzb*16, 0.0);
		c->vals.Download(hv.data(), hv.size());
		L.push_back(std::move(c));
	}
	// per-level buffers; greedy node colouring of every Gauss-Seidel level
	for (size_t l = 0; l < L.size(); ++l) {
		Level& v = *L[l];
		v.gs = l + 1 < L.size() && opt.smoother == TFI_SMOOTH_GAUSS_SEIDEL && v.rows >= opt.gs_min_rows;
		if (v.gs) Colour(v);
		const long long n = 4LL*v.rows;
		v.inv64.Allocate(ctx, 16LL*v.rows);
		if (precision == TFI_MIXED) {
			v.inv32.Allocate(ctx, 16LL*v.rows);
			v.x32.Allocate(ctx, n);
			v.y32.Allocate(ctx, n);
			v.b32.Allocate(ctx, n);
			v.r32.Allocate(ctx, n);
			if (l > 0) v.vals32_own.Allocate(ctx, v.nnzb*16);
			if (opt.half_smoother && !v.gs && l + 1 < L.size() && opt.smoother == TFI_SMOOTH_CHEBYSHEV) {
				v.s16.Allocate(ctx, v.nnzb*16);
				v.dblock32.Allocate(ctx, 16LL*v.rows);
			}
		} else {
			if (l > 0) {  // the finest level works on the caller's vectors
				v.x64.Allocate(ctx, n);
				v.b64.Allocate(ctx, n);
			}
			v.y64.Allocate(ctx, n);
			v.r64.Allocate(ctx, n);
		}
	}
	nc = 4*L.back()->rows;
	if (nc > kDenseMax) throw Error("AMG coarsest level too large for the dense solve");
	for (auto& d : dense) d.Allocate(ctx, (size_t)nc*nc);
	panel.Allocate(ctx, (size_t)nc*kPanel);
	next_panel.Allocate(ctx, (size_t)nc*kPanel);
	pivot.Allocate(ctx, nc);
	step.Allocate(ctx, nc);
	if (precision == TFI_MIXED) dinv32.Allocate(ctx, (size_t)nc*nc);
	else dinv64.Allocate(ctx, (size_t)nc*nc);
	status.Allocate(ctx, 1);
	scale_flags.Allocate(ctx, L.size());
	power_partial.Allocate(ctx, kPowerBlocks);
	squares.Allocate(ctx, L.size());
	Fill(ctx, squares.data(), 0.0, static_cast<long long>(L.size()));
	built = true;
}

// A P of the fine level, then the coarse values from it
void Amg::Impl::Coarsen(Level& f, const double* fine_values, Level& c)
{
	hipLaunchKernelGGL(GalerkinKernel, dim3(Grid(f.ap_nnzb*16)), dim3(256), 0, ctx->stream, f.ap_nnzb, f.ap_off.data(),
		f.ap_list.data(), fine_values, f.ap64.data());
	TFI_LAUNCH_CHECK("GalerkinKernel A P");
	hipLaunchKernelGGL(GalerkinKernel, dim3(Grid(c.nnzb*16)), dim3(256), 0, ctx->stream, c.nnzb, f.goff.data(),
		f.glist.data(), f.ap64.data(), c.vals.data());
	TFI_LAUNCH_CHECK("GalerkinKernel");
}

void Amg::Impl::Numeric(const double* fine64, const float* fine32)
{
	L[0]->vals64 = fine64;
	L[0]->vals32 = fine32;
	for (size_t l = 0; l + 1 < L.size(); ++l) {
		Level& f = *L[l];
		Level& c = *L[l + 1];
		Coarsen(f, l == 0 ? fine64 : f.vals.data(), c);
		c.vals64 = c.vals.data();
	}
	for (size_t l = 0; l < L.size(); ++l) {
		Level& v = *L[l];
		LaunchBlockInverse64(ctx, v.view(), v.vals64, v.inv64.data(), nullptr);
		if (precision == TFI_MIXED) {
			hipLaunchKernelGGL(BlockInverseT32Kernel, dim3(256), dim3(256), 0, ctx->stream, 16LL*v.rows,
				v.inv64.data(), v.inv32.data());
			TFI_LAUNCH_CHECK("BlockInverseT32Kernel");
			if (l > 0) {
				hipLaunchKernelGGL(ToFloatKernel2, dim3(256), dim3(256), 0, ctx->stream, v.nnzb*16, v.vals64,
					v.vals32_own.data());
				TFI_LAUNCH_CHECK("ToFloatKernel2");
				v.vals32 = v.vals32_own.data();
			}
		}
	}
	// FP16 copies of D^-1 A (and S P) for the Chebyshev levels of the mixed path,
	// FP32 A P for its other levels
	FillInt(ctx, scale_flags.data(), 0, static_cast<long long>(L.size()));
	auto wide_ap = [&](Level& v) {
		hipLaunchKernelGGL(ToFloatKernel2, dim3(Grid(std::min<long long>(v.ap_nnzb*16, 1LL << 22))), dim3(256), 0,
			ctx->stream, v.ap_nnzb*16, v.ap64.data(), v.ap32.data());
		TFI_LAUNCH_CHECK("ToFloatKernel2");
	};
	if (precision == TFI_MIXED)
		for (size_t l = 0; l + 1 < L.size(); ++l) {
			Level& v = *L[l];
			if (v.gs) continue;
			if (!v.s16.size()) {
				wide_ap(v);
				continue;
			}
			hipLaunchKernelGGL(ScaleBlocksKernel, dim3((v.rows + 3)/4), dim3(256), 0, ctx->stream, v.rows, v.ro,
				v.diag, v.vals64, v.inv64.data(), v.s16.data(), v.dblock32.data(), scale_flags.data() + l);
			TFI_LAUNCH_CHECK("ScaleBlocksKernel");
			hipLaunchKernelGGL(ScaledGalerkinKernel, dim3(Grid(v.ap_nnzb*16)), dim3(256), 0, ctx->stream, v.ap_nnzb,
				v.ap_off.data(), v.ap_list.data(), v.s16.data(), v.ap32.data());
			TFI_LAUNCH_CHECK("ScaledGalerkinKernel");
		}
	// lambda_max(D^-1 A) of every Jacobi-smoothed level by power iteration (FP64):
	// squares[l] = ||D^-1 A x||^2 of the last step's normalised x
	for (size_t l = 0; l + 1 < L.size(); ++l) {
		Level& v = *L[l];
		if (v.gs) continue;
		const long long n = 4LL*v.rows;
		if (!power[0].size())  // the first such level is the largest
			for (auto& p : power) p.Allocate(ctx, n);
		double* sq = squares.data() + l;
		const int start = std::min(Grid(n), kPowerBlocks), blocks = std::min((v.rows + 3)/4, kPowerBlocks);
		auto sum = [&](int count) {
			hipLaunchKernelGGL(SumKernel, dim3(1), dim3(kSumThreads), 0, ctx->stream, power_partial.data(), count, sq);
			TFI_LAUNCH_CHECK("SumKernel");
		};
		hipLaunchKernelGGL(HashVectorKernel, dim3(start), dim3(256), 0, ctx->stream, n, power[0].data(),
			power_partial.data());
		TFI_LAUNCH_CHECK("HashVectorKernel");
		sum(start);
		for (int it = 0; it < kPowerIterations; ++it) {
			hipLaunchKernelGGL(DinvAKernel, dim3(blocks), dim3(256), 0, ctx->stream, v.rows, v.ro, v.cols, v.vals64,
				v.inv64.data(), power[it & 1].data(), sq, power[(it + 1) & 1].data(), power_partial.data());
			TFI_LAUNCH_CHECK("DinvAKernel");
			sum(blocks);
		}
	}
	// coarsest dense inverse, built and inverted on the device
	Level& c = *L.back();
	Fill(ctx, dense[0].data(), 0.0, (long long)nc*nc);
	hipLaunchKernelGGL(DenseKernel, dim3(c.rows), dim3(64), 0, ctx->stream, c.rows, c.ro, c.cols, c.vals64,
		dense[0].data());
	TFI_LAUNCH_CHECK("DenseKernel");
	FillInt(ctx, status.data(), 0, 1);
	FillInt(ctx, step.data(), nc, nc);
	const double* matrix = dense[0].data();
	for (int p0 = 0, flip = 1; p0 < nc; p0 += kPanel, flip ^= 1) {
		const int width = std::min(kPanel, nc - p0);
		hipLaunchKernelGGL(PanelKernel, dim3(1), dim3((nc + 63)/64*64), 0, ctx->stream, nc, p0, width,
			p0 ? next_panel.data() : matrix, p0 ? 1 : nc, p0 ? nc : 1, panel.data(), step.data(), pivot.data(),
			status.data());
		hipLaunchKernelGGL(PanelUpdateKernel, dim3((nc + 63)/64, (nc + kUpdateRows - 1)/kUpdateRows), dim3(256), 0,
			ctx->stream, nc, p0, width, matrix, panel.data(), step.data(), pivot.data(), dense[flip].data(),
			next_panel.data());
		matrix = dense[flip].data();
	}
	TFI_LAUNCH_CHECK("PanelUpdateKernel");
	// what the host needs of all this, after one wait
	int st = 0;
	std::vector<int> flags(L.size(), 0);
	std::vector<double> last(L.size(), 0.0);
	status.Download(&st, 1);
	scale_flags.Download(flags.data(), flags.size());
	squares.Download(last.data(), last.size());
	for (size_t l = 0; l + 1 < L.size(); ++l) {
		Level& v = *L[l];
		if (v.gs) continue;
		v.scaled = v.s16.size() > 0 && flags[l] == 0;
		if (v.s16.size() > 0 && !v.scaled) wide_ap(v);  // S did not fit FP16
		const double lambda = std::sqrt(last[l]);
		v.lambda_max = lambda > 0.0 ? lambda : 1.0;
	}
	// with the levels as their matrices are now: only the coarsest inverse stays the old one
	if (st) throw Error("AMG coarsest operator is singular");
	if (precision == TFI_MIXED) {
		hipLaunchKernelGGL(ExtractInverseKernel<float>, dim3(nc), dim3(256), 0, ctx->stream, nc, matrix, pivot.data(),
			dinv32.data());
	} else {
		hipLaunchKernelGGL(ExtractInverseKernel<double>, dim3(nc), dim3(256), 0, ctx->stream, nc, matrix, pivot.data(),
			dinv64.data());
	}
	TFI_LAUNCH_CHECK("ExtractInverseKernel");
}

// x = M^-1 b on level l
template <class T>
void Amg::Impl::Cycle(int l, const T* b, T* x)
{
	Level& v = *L[l];
	constexpr bool f32 = std::is_same<T, float>::value;
	auto pick = [](auto& wide, auto& narrow) -> T* {
		if constexpr (f32) return narrow.data();
		else return wide.data();
	};
	if (l + 1 == (int)L.size()) {
		hipLaunchKernelGGL(DenseApplyKernel<T>, dim3((nc + 3)/4), dim3(256), 0, ctx->stream, nc,
			static_cast<const T*>(pick(dinv64, dinv32)), b, x);
		TFI_LAUNCH_CHECK("DenseApplyKernel");
		return;
	}
	T* y = pick(v.y64, v.y32);
	T* r = pick(v.r64, v.r32);
	const T* vals;
	if constexpr (f32) vals = v.vals32;
	else vals = v.vals64;
	const T* inv = pick(v.inv64, v.inv32);
	const int grid = (v.rows + 3)/4;
	const bool gs = v.gs;
	const bool cheb = !gs && opt.smoother == TFI_SMOOTH_CHEBYSHEV;
	// Smoothing steps before and after the coarse correction.  The first of
	// either needs no pass over A: from x = 0, or from the residual and A P; the
	// others go from x to y and back, and their number before and after is the
	// same, so the result is in x.  Chebyshev steps on [kChebLow, kChebHigh]
	// lambda_max: d lives in the level's r buffer, which the smoothing phases do
	// not otherwise use.
	const int steps = cheb ? opt.chebyshev_degree : kPre;
	static_assert(kPre == kPost, "as many steps after the correction as before");
	const double hi = kChebHigh*v.lambda_max, lo = kChebLow*v.lambda_max;
	const double theta = 0.5*(hi + lo), delta = 0.5*(hi - lo), sigma = theta/delta;
	const T first = static_cast<T>(cheb ? 1.0/theta : kOmegaScale/v.lambda_max);
	T* from = x;
	T* to = y;
	auto more_steps = [&] {
		double rho = 1.0/sigma;
		for (int k = 1; k < steps; ++k) {
			const double rn = 1.0/(2.0*sigma - rho);
			const T cd = static_cast<T>(rn*rho), cz = static_cast<T>(2.0*rn/delta);
			rho = rn;
			bool done = false;
			if constexpr (f32) {
				if (v.scaled) {
					hipLaunchKernelGGL(ChebyshevScaledKernel, dim3(grid), dim3(256), 0, ctx->stream, v.rows, v.ro, v.cols,
						v.s16.data(), inv, b, static_cast<const float*>(from), to, r, cd, cz);
					done = true;
				}
			}
			if (!done && cheb)
				hipLaunchKernelGGL(ChebyshevKernel<T>, dim3(grid), dim3(256), 0, ctx->stream, v.rows, v.ro, v.cols, vals,
					inv, b, static_cast<const T*>(from), to, r, cd, cz);
			else if (!done)
				hipLaunchKernelGGL(SmoothKernel<T>, dim3(grid), dim3(256), 0, ctx->stream, v.rows, v.ro, v.cols, vals, inv,
					b, static_cast<const T*>(from), to, first);
			std::swap(from, to);
		}
		TFI_LAUNCH_CHECK("smoothing step");
	};
	const int ncol = static_cast<int>(v.color_offsets.size()) - 1;
	// after_forward: this backward sweep directly follows a forward one, whose
	// last colour it would repeat with nothing changed in between (a colour's
	// update depends only on the other colours), so that colour is skipped
	auto gs_sweep = [&](bool forward, bool after_forward = false) {
		bool skip = after_forward;
		for (int cc = 0; cc < ncol; ++cc) {
			const int c = forward ? cc : ncol - 1 - cc;
			const int count = v.color_offsets[c + 1] - v.color_offsets[c];
			if (count == 0) continue;
			if (skip) {
				skip = false;
				continue;
			}
			hipLaunchKernelGGL(GsColorKernel<T>, dim3((count + 3)/4), dim3(256), 0, ctx->stream, count,
				v.color_rows.data() + v.color_offsets[c], v.ro, v.cols, vals, inv, b, x);
		}
		TFI_LAUNCH_CHECK("GsColorKernel");
	};
	if (gs) {
		// symmetric multicolour Gauss-Seidel from x = 0
		const long long n = 4LL*v.rows;
		if constexpr (f32) Check(hipMemsetAsync(x, 0, n*sizeof(T), ctx->stream), "memset");
		else Fill(ctx, x, 0.0, n);
		gs_sweep(true);
		if (opt.gs_sweeps > 1) gs_sweep(false, true);
	} else {
		hipLaunchKernelGGL(FirstStepKernel<T>, dim3(Grid(4LL*v.rows)), dim3(256), 0, ctx->stream, v.rows, inv, b, from, r,
			first);
		TFI_LAUNCH_CHECK("FirstStepKernel");
		more_steps();
	}
	bool residual_done = false;
	if constexpr (f32) {
		if (v.scaled) {
			hipLaunchKernelGGL(ResidualScaledKernel, dim3(grid), dim3(256), 0, ctx->stream, v.rows, v.ro, v.cols,
				v.s16.data(), inv, v.dblock32.data(), b, static_cast<const float*>(from), r);
			residual_done = true;
		}
	}
	if (!residual_done)
		hipLaunchKernelGGL(ResidualKernel<T>, dim3(grid), dim3(256), 0, ctx->stream, v.rows, v.ro, v.cols, vals, b,
			static_cast<const T*>(from), r);
	TFI_LAUNCH_CHECK("ResidualKernel");
	Level& c = *L[l + 1];
	T* bc = pick(c.b64, c.b32);
	T* xc = pick(c.x64, c.x32);
	hipLaunchKernelGGL(RestrictKernel<T>, dim3(Grid(16LL*c.rows)), dim3(256), 0, ctx->stream, c.rows, v.aoff.data(),
		v.amem.data(), static_cast<const T*>(r), bc);
	TFI_LAUNCH_CHECK("RestrictKernel");
	Cycle<T>(l + 1, bc, xc);
	if (gs) {
		hipLaunchKernelGGL(ProlongKernel<T>, dim3(Grid(4LL*v.rows)), dim3(256), 0, ctx->stream, v.rows, v.agg.data(),
			static_cast<const T*>(xc), x);
		TFI_LAUNCH_CHECK("ProlongKernel");
		if (opt.gs_sweeps > 1) gs_sweep(true);
		gs_sweep(false, opt.gs_sweeps > 1);
	} else {
		auto correct = [&](auto kernel) {
			hipLaunchKernelGGL(kernel, dim3((v.rows + 7)/8), dim3(256), 0, ctx->stream, v.rows, v.ap_ro.data(), v.ap_cols.data(),
				static_cast<const T*>(pick(v.ap64, v.ap32)), inv, v.agg.data(), static_cast<const T*>(xc), from, r, first);
		};
		if (f32 && v.scaled) correct(CorrectStepKernel<T, f32>);
		else correct(CorrectStepKernel<T, false>);
		TFI_LAUNCH_CHECK("CorrectStepKernel");
		more_steps();
	}
}

Amg::Amg(tfi_mesh* mesh, int precision, const AmgOptions& options) : impl_(std::make_unique<Impl>())
{
	if (options.coarse_nodes < 1 || options.coarse_nodes > 256)
		throw Error("AMG coarsest level must hold between 1 and 256 block rows");
	impl_->mesh = mesh;
	impl_->ctx = mesh->ctx;
	impl_->precision = precision;
	impl_->opt = options;
}

void Amg::Describe(std::vector<int>& rows, std::vector<long long>& nnzb, std::vector<int>& colors) const
{
	rows.clear();
	nnzb.clear();
	colors.clear();
	for (const auto& l : impl_->L) {
		rows.push_back(l->rows);
		nnzb.push_back(l->nnzb);
		colors.push_back(l->gs ? static_cast<int>(l->color_offsets.size()) - 1 : 0);
	}
}

Amg::~Amg() = default;

int Amg::smoother() const { return impl_->opt.smoother; }

void Amg::UseGaussSeidel()
{
	Impl& I = *impl_;
	I.opt.smoother = TFI_SMOOTH_GAUSS_SEIDEL;
	if (!I.built) return;
	for (size_t l = 0; l + 1 < I.L.size(); ++l) {
		Level& v = *I.L[l];
		v.gs = v.rows >= I.opt.gs_min_rows;
		if (v.gs && v.color_offsets.empty()) I.Colour(v);
		// the levels that stay Jacobi-smoothed read A from here on, not S
		v.s16.Release();
		v.dblock32.Release();
		v.scaled = false;
	}
}

int Amg::levels() const { return static_cast<int>(impl_->L.size()); }

void Amg::Setup(const double* values64, const float* values32)
{
	if (!impl_->built) impl_->Symbolic(values64);
	impl_->Numeric(values64, values32);
	singular_ = 0;
}

void Amg::Apply(const double* v, double* z)
{
	Impl& I = *impl_;
	Level& l0 = *I.L[0];
	const long long n = 4LL*l0.rows;
	if (I.precision == TFI_MIXED) {
		hipLaunchKernelGGL(ToFloatKernel2, dim3(Grid(n)), dim3(256), 0, I.ctx->stream, n, v, l0.b32.data());
		TFI_LAUNCH_CHECK("ToFloatKernel2");
		I.Cycle<float>(0, l0.b32.data(), l0.x32.data());
		hipLaunchKernelGGL(ToDoubleKernel, dim3(Grid(n)), dim3(256), 0, I.ctx->stream, n, l0.x32.data(), z);
		TFI_LAUNCH_CHECK("ToDoubleKernel");
	} else {
		if (v < z + n && z < v + n) {  // the cycle writes z while it still reads v
			if (!l0.b64.size()) l0.b64.Allocate(I.ctx, n);
			Copy(I.ctx, v, l0.b64.data(), n);
			v = l0.b64.data();
		}
		I.Cycle<double>(0, v, z);
	}
}

}  // namespace tfi
