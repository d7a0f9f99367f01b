// Flexible GMRES(m), right-preconditioned, with classical Gram-Schmidt applied
// twice (CGS2) through fused multi-vector kernels.
//
// Replaces SolveGmres<4> (solvers/cuda/include/Gmres.hpp:69-213), whose
// modified Gram-Schmidt issues j+1 cuBLAS Ddot/Daxpy pairs per iteration, each
// Ddot a host round trip.  Here one Arnoldi step is: preconditioner, SpMV,
// two passes of {multi-dot over all basis vectors, multi-axpy} (each pass reads
// the basis once from HBM), a fused norm, and one small device->host copy of
// the Hessenberg column for the Givens update on the host.  All reductions
// have a fixed order, so a solve is bitwise reproducible.  The stopping test is
// the true relative residual ||b - A x|| <= rtol ||b|| (PETSc FGMRES with a zero
// guess, TransientFlowRuntime.hpp:176-190), re-checked at every restart.
#include "tfi_internal.hpp"

#include <algorithm>
#include <cmath>

namespace tfi {

namespace {

constexpr int kThreads = 256;
constexpr int kGroup = 8;         // basis vectors of a multi-dot workgroup (one set of wave reductions)
constexpr int kDotPer = 8, kAxpyPer = 4;  // vector entries per thread, at most
constexpr int kLongPer = 4;       // and of a multi-dot over long vectors
constexpr int kDotGroups = 2048;  // workgroups of a pass that keep the chip's memory pipes full
constexpr int kFewBlocks = 32;    // partial sums that the kernel after a multi-dot adds up itself

// Why the split depends on the length: eight entries per thread for any length left
// 158 workgroups for 324,000 entries (25 vectors on average: multi-dot 75 us,
// multi-axpy 57, 0.9 TB/s) and one for 1800 (20 and 16 us).  With the rule below
// 13 and 11 us (4.9 TB/s), and 2.8 and 3.9 us.  The axpy stops at four entries: with
// eight the loads of eight vectors take 96 registers, and half the waves (8.1
// million entries, 50 vectors: 797 us, with four entries 567).
// Entries per thread of a pass over n entries in `lanes` rows of workgroups: as
// many as leave kDotGroups workgroups (8-byte loads in flight against workgroups
// to hide their latency), 1 to `most`.
int EntriesPerThread(long long n, int lanes, int most)
{
	int per = most;
	while (per > 1 && (n + (long long)kThreads*per - 1)/((long long)kThreads*per)*lanes < kDotGroups) per >>= 1;
	return per;
}
int Blocks(long long n, int per)
{
	return static_cast<int>((n + (long long)kThreads*per - 1)/((long long)kThreads*per));
}
// Vectors whose blocks of four entries per thread fill the chip more than twice
// over: a multi-dot workgroup takes all vectors, w in registers (8.1 million entries,
// 9 / 25 / 50 vectors: 107 / 282 / 563 us, in rows of eight vectors 132 / 320 / 607;
// 5 million 66 / 173 / 344 against 78 / 184 / 351, 4.2 million 57 / 154 / 301 against
// 65 / 150 / 280)
bool Long(long long n) { return n >= 5000000; }
// Most row blocks the rules can ask for: below 2*kDotGroups, or with four entries per thread
int MaxBlocks(long long n)
{
	return std::min(Blocks(n, 1), std::max(2*kDotGroups, Blocks(n, std::min(kAxpyPer, kLongPer))));
}
// Vectors too short for a workgroup per CU at one entry per thread: the
// multi-axpy takes 64 entries per workgroup instead
bool Short(const tfi_ctx* ctx, long long n) { return Blocks(n, 1) < ctx->cus; }
int ShortBlocks(long long n) { return static_cast<int>((n + 63)/64); }

__device__ inline double WaveSum(double v)
{
	for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
	return v;
}

// Sums of eight values over the wave: three exchanges halve the values a lane
// carries while they halve its partners (7 shuffles), three more finish (3):
// 10 instead of 48.  Lane l ends with the sum of value (l >> 3).
__device__ inline double WaveSum8(const double (&v)[kGroup])
{
	const int lane = threadIdx.x & 63;
	double a[4], b[2];
	const bool h32 = lane & 32, h16 = lane & 16, h8 = lane & 8;
#pragma unroll
	for (int k = 0; k < 4; ++k) a[k] = (h32 ? v[4 + k] : v[k]) + __shfl_xor(h32 ? v[k] : v[4 + k], 32, 64);
#pragma unroll
	for (int k = 0; k < 2; ++k) b[k] = (h16 ? a[2 + k] : a[k]) + __shfl_xor(h16 ? a[k] : a[2 + k], 16, 64);
	double c = (h8 ? b[1] : b[0]) + __shfl_xor(h8 ? b[0] : b[1], 8, 64);
	c += __shfl_xor(c, 4, 64);
	c += __shfl_xor(c, 2, 64);
	c += __shfl_xor(c, 1, 64);
	return c;
}

// partial[i*gridDim.x + blk] = sum over this block's rows of V_i . w, i < count;
// blockIdx.y: eight of the vectors.
template <int kPer>
__global__ void __launch_bounds__(kThreads) MultiDotKernel(const double* __restrict__ V, long long ld, int count,
	const double* __restrict__ w, long long n, double* __restrict__ partial)
{
	__shared__ double lds[kGroup][4];
	const long long base = (long long)blockIdx.x*kThreads*kPer + threadIdx.x;
	const int g = blockIdx.y*kGroup;
	double wr[kPer];
#pragma unroll
	for (int t = 0; t < kPer; ++t) {
		const long long i = base + (long long)t*kThreads;
		wr[t] = i < n ? w[i] : 0.0;
	}
	double acc[kGroup] = {};
#pragma unroll
	for (int v = 0; v < kGroup; ++v) {
		// past the last vector: its place is read again and not stored
		const double* Vi = V + (long long)min(g + v, count - 1)*ld;
#pragma unroll
		for (int t = 0; t < kPer; ++t) acc[v] += Vi[min(base + (long long)t*kThreads, n - 1)]*wr[t];
	}
	const double s = WaveSum8(acc);
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	if ((lane & 7) == 0) lds[lane >> 3][wave] = s;
	__syncthreads();
	if (threadIdx.x < kGroup && g + (int)threadIdx.x < count) {
		const int v = threadIdx.x;
		partial[(long long)(g + v)*gridDim.x + blockIdx.x] = lds[v][0] + lds[v][1] + lds[v][2] + lds[v][3];
	}
}

// The same for long vectors (Long): a workgroup takes all vectors, eight at a time,
// with its part of w in registers.
__global__ void __launch_bounds__(kThreads) MultiDotLongKernel(const double* __restrict__ V, long long ld, int count,
	const double* __restrict__ w, long long n, double* __restrict__ partial)
{
	constexpr int kPer = kLongPer;
	__shared__ double lds[kGroup][4];
	const long long base = (long long)blockIdx.x*kThreads*kPer + threadIdx.x;
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	double wr[kPer];
#pragma unroll
	for (int t = 0; t < kPer; ++t) {
		const long long i = base + (long long)t*kThreads;
		wr[t] = i < n ? w[i] : 0.0;
	}
	for (int g = 0; g < count; g += kGroup) {
		double acc[kGroup] = {};
#pragma unroll
		for (int v = 0; v < kGroup; ++v) {
			if (g + v >= count) break;
			const double* Vi = V + (long long)(g + v)*ld;
#pragma unroll
			for (int t = 0; t < kPer; ++t) acc[v] += Vi[min(base + (long long)t*kThreads, n - 1)]*wr[t];
		}
		const double s = WaveSum8(acc);
		__syncthreads();  // the sums of the group before have been read
		if ((lane & 7) == 0) lds[lane >> 3][wave] = s;
		__syncthreads();
		if (threadIdx.x < kGroup && g + (int)threadIdx.x < count) {
			const int v = threadIdx.x;
			partial[(long long)(g + v)*gridDim.x + blockIdx.x] = lds[v][0] + lds[v][1] + lds[v][2] + lds[v][3];
		}
	}
}

// out[i] = sum_b partial[i*blocks + b]   (one workgroup per i)
__global__ void ReducePartialsKernel(const double* __restrict__ partial, int blocks, double* __restrict__ out)
{
	__shared__ double lds[4];
	const int i = blockIdx.x;
	double s = 0.0;
	for (int b = threadIdx.x; b < blocks; b += blockDim.x) s += partial[(long long)i*blocks + b];
	s = WaveSum(s);
	if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = s;
	__syncthreads();
	if (threadIdx.x == 0) {
		const double t = lds[0] + lds[1] + lds[2] + lds[3];
		out[i] = t;
	}
}

// w += sign * sum_i coef[i] V_i ; optional per-block partial of ||w||^2.  With
// partial_blocks > 0 coef[i] is the sum of partial[i*partial_blocks ..] (few
// blocks), which workgroup 0 also leaves in coef for the host.
// kSplit = 1: kPer entries per thread; kSplit = 4: 64 entries per workgroup, its
// four waves a quarter of the vectors each (short vectors: the walk over the
// vectors is the time).
template <int kPer, int kSplit>
__global__ void __launch_bounds__(kThreads) MultiAxpyKernel(const double* __restrict__ V, long long ld, int count,
	double* __restrict__ coef, const double* __restrict__ partial, int partial_blocks, double sign,
	double* __restrict__ w, long long n, double* __restrict__ norm_partial)
{
	static_assert(kSplit == 1 || (kSplit == 4 && kPer == 1), "whole vectors, or quarters of one entry per lane");
	__shared__ double c[512];
	__shared__ double lds[4];
	for (int i = threadIdx.x; i < count; i += kThreads) {
		double v;
		if (partial_blocks > 0) {
			v = 0.0;
			for (int b = 0; b < partial_blocks; ++b) v += partial[(long long)i*partial_blocks + b];
			if (blockIdx.x == 0) coef[i] = v;
		} else {
			v = coef[i];
		}
		c[i] = sign*v;
	}
	__syncthreads();
	const int wave = threadIdx.x >> 6;
	const long long base = kSplit == 1 ? (long long)blockIdx.x*kThreads*kPer + threadIdx.x
		: (long long)blockIdx.x*64 + (threadIdx.x & 63);
	// each entry accumulates over the vectors in order; the loads of eight
	// vectors are in flight together
	double acc[kPer];
#pragma unroll
	for (int t = 0; t < kPer; ++t) {
		const long long i = base + (long long)t*kThreads;
		acc[t] = i < n && (kSplit == 1 || wave == 0) ? w[i] : 0.0;
	}
	const int quarter = (count + kSplit - 1)/kSplit;
	const int begin = kSplit == 1 ? 0 : min(count, wave*quarter), end = kSplit == 1 ? count : min(count, begin + quarter);
#pragma unroll 8
	for (int v = begin; v < end; ++v) {
		const double cv = c[v];
		const double* Vv = V + (long long)v*ld;
#pragma unroll
		for (int t = 0; t < kPer; ++t) acc[t] += cv*Vv[min(base + (long long)t*kThreads, n - 1)];
	}
	if constexpr (kSplit > 1) {
		__shared__ double part[kSplit][64];
		part[wave][threadIdx.x & 63] = acc[0];
		__syncthreads();
		if (wave > 0) {
			acc[0] = 0.0;  // no share in the norm
		} else {
			acc[0] = 0.0;
			for (int k = 0; k < kSplit; ++k) acc[0] += part[k][threadIdx.x];
		}
	}
	double sq = 0.0;
#pragma unroll
	for (int t = 0; t < kPer; ++t) {
		const long long i = base + (long long)t*kThreads;
		if (i < n && (kSplit == 1 || wave == 0)) {
			w[i] = acc[t];
			sq += acc[t]*acc[t];
		}
	}
	if (norm_partial) {
		sq = WaveSum(sq);
		if ((threadIdx.x & 63) == 0) lds[wave] = sq;
		__syncthreads();
		if (threadIdx.x == 0) norm_partial[blockIdx.x] = lds[0] + lds[1] + lds[2] + lds[3];
	}
}

// dst = src / norm where norm^2 is *sq, or with partial_blocks > 0 the sum of
// partial[0 .. partial_blocks), which workgroup 0 leaves in *sq.
__global__ void NormalizeKernel(const double* __restrict__ src, double* __restrict__ dst, long long n,
	double* __restrict__ sq, const double* __restrict__ partial, int partial_blocks)
{
	double total = 0.0;
	if (partial_blocks > 0) {
		for (int b = 0; b < partial_blocks; ++b) total += partial[b];
		if (blockIdx.x == 0 && threadIdx.x == 0) *sq = total;
	} else {
		total = *sq;
	}
	const double nrm = sqrt(total);
	const double s = nrm > 1e-300 ? 1.0/nrm : 0.0;
	for (long long i = blockIdx.x*(long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x*blockDim.x)
		dst[i] = src[i]*s;
}

// Launches of the passes: each picks the entries per thread for its length.
// Returns the number of partial sums per vector.
int MultiDot(tfi_ctx* ctx, const double* V, long long n, int count, const double* w, double* partial)
{
	const int groups = (count + kGroup - 1)/kGroup;
	const int per = Long(n) ? kLongPer : EntriesPerThread(n, groups, kDotPer);
	auto launch = [&](auto kernel, int rows) {
		hipLaunchKernelGGL(kernel, dim3(Blocks(n, per), rows), dim3(kThreads), 0, ctx->stream, V, n, count, w, n, partial);
	};
	if (Long(n)) launch(MultiDotLongKernel, 1);
	else if (per == 1) launch(MultiDotKernel<1>, groups);
	else if (per == 2) launch(MultiDotKernel<2>, groups);
	else if (per == 4) launch(MultiDotKernel<4>, groups);
	else launch(MultiDotKernel<8>, groups);
	TFI_LAUNCH_CHECK("MultiDotKernel");
	return Blocks(n, per);
}

// Coefficients from `blocks` partial sums each (0: they are in coef); returns
// the number of norm partials written.
int MultiAxpy(tfi_ctx* ctx, const double* V, long long n, int count, double* coef, const double* partial, int blocks,
	double sign, double* w, double* norm_partial)
{
	if (blocks > kFewBlocks) {
		hipLaunchKernelGGL(ReducePartialsKernel, dim3(count), dim3(256), 0, ctx->stream, partial, blocks, coef);
		TFI_LAUNCH_CHECK("ReducePartialsKernel");
		blocks = 0;
	}
	auto launch = [&](auto kernel, int grid) {
		hipLaunchKernelGGL(kernel, dim3(grid), dim3(kThreads), 0, ctx->stream, V, n, count, coef, partial, blocks, sign,
			w, n, norm_partial);
		TFI_LAUNCH_CHECK("MultiAxpyKernel");
		return grid;
	};
	if (Short(ctx, n)) return launch(MultiAxpyKernel<1, 4>, ShortBlocks(n));
	switch (EntriesPerThread(n, 1, kAxpyPer)) {
	case 1: return launch(MultiAxpyKernel<1, 1>, Blocks(n, 1));
	case 2: return launch(MultiAxpyKernel<2, 1>, Blocks(n, 2));
	default: return launch(MultiAxpyKernel<4, 1>, Blocks(n, 4));
	}
}

}  // namespace

Fgmres::Fgmres(tfi_ctx* ctx, long long n, int restart) : ctx_(ctx), n_(n), m_(restart)
{
	if (restart < 1 || restart > 500) throw Error("FGMRES restart must be in [1, 500]");
	V_.Allocate(ctx, (size_t)(m_ + 1)*n);
	Z_.Allocate(ctx, (size_t)m_*n);
	w_.Allocate(ctx, n);
	r_.Allocate(ctx, n);
	// multi-dot partials of up to m vectors, then the norm partials of a multi-axpy
	partial_.Allocate(ctx, (size_t)(m_ + 1)*MaxBlocks(n) + (Short(ctx, n) ? ShortBlocks(n) : MaxBlocks(n)));
	h_.Allocate(ctx, 2*(m_ + 2) + 8);
	H_.assign((size_t)(m_ + 1)*m_, 0.0);
	cs_.assign(m_, 0.0);
	sn_.assign(m_, 0.0);
	g_.assign(m_ + 1, 0.0);
	y_.assign(m_, 0.0);
}

KrylovResult Fgmres::Solve(const Operator& A, const Precond& M, const double* b, double* x, int maxit, double rtol,
	double absolute_target)
{
	tfi_ctx* ctx = ctx_;
	const long long n = n_;
	const int eblocks = static_cast<int>(std::min<long long>((n + 255)/256, 4096));
	KrylovResult res;
	res.rhs_norm = Norm2(ctx, b, n);
	const double tol = std::max(rtol*res.rhs_norm, absolute_target);
	double* V = V_.data();
	double* Z = Z_.data();
	double* w = w_.data();
	double* h = h_.data();            // h[0..m]: projection coefficients; h[m+1]: squared norm
	double* hsq = h + (m_ + 1);
	double* partial = partial_.data();
	auto true_residual = [&]() {
		A(x, w);
		// r = b - w
		Copy(ctx, b, r_.data(), n);
		Axpy(ctx, -1.0, w, r_.data(), n);
		return Norm2(ctx, r_.data(), n);
	};
	double beta = true_residual();
	res.residual = beta;
	if (res.rhs_norm == 0.0 || beta <= tol) {
		res.converged = true;
		return res;
	}
	double* hcol = ctx->host_pinned;  // pinned staging
	const double beta0 = beta;
	while (res.iterations < maxit) {
		const double beta_cycle = beta;
		Copy(ctx, r_.data(), V, n);
		Scale(ctx, 1.0/beta, V, n);
		std::fill(H_.begin(), H_.end(), 0.0);
		std::fill(g_.begin(), g_.end(), 0.0);
		g_[0] = beta;
		int used = 0;
		bool breakdown = false;
		for (int j = 0; j < m_ && res.iterations < maxit; ++j) {
			double* vj = V + (long long)j*n;
			double* zj = M ? Z + (long long)j*n : vj;
			if (M) M(vj, zj);
			A(zj, w);
			// CGS pass 1: h = V^T w ; w -= V h; pass 2 (re-orthogonalisation) with the norm of w
			double* h2 = h + (m_ + 2);  // second-pass coefficients
			double* npart = partial + (long long)(m_ + 1)*MaxBlocks(n);
			int parts = MultiDot(ctx, V, n, j + 1, w, partial);
			MultiAxpy(ctx, V, n, j + 1, h, partial, parts, -1.0, w, nullptr);
			parts = MultiDot(ctx, V, n, j + 1, w, partial);
			int norms = MultiAxpy(ctx, V, n, j + 1, h2, partial, parts, -1.0, w, npart);
			if (norms > kFewBlocks) {
				hipLaunchKernelGGL(ReducePartialsKernel, dim3(1), dim3(256), 0, ctx->stream, npart, norms, hsq);
				TFI_LAUNCH_CHECK("ReducePartialsKernel");
				norms = 0;
			}
			hipLaunchKernelGGL(NormalizeKernel, dim3(eblocks), dim3(256), 0, ctx->stream, w, V + (long long)(j + 1)*n, n,
				hsq, npart, norms);
			TFI_LAUNCH_CHECK("NormalizeKernel");
			// bring back h (pass 1 + pass 2) and the squared norm
			Check(hipMemcpyAsync(hcol, h, sizeof(double)*(2*(m_ + 2)), hipMemcpyDeviceToHost, ctx->stream), "h download");
			Check(hipStreamSynchronize(ctx->stream), "arnoldi sync");
			for (int i = 0; i <= j; ++i) H_[(size_t)i*m_ + j] = hcol[i] + hcol[m_ + 2 + i];
			const double hn = std::sqrt(hcol[m_ + 1]);
			H_[(size_t)(j + 1)*m_ + j] = hn;
			for (int i = 0; i < j; ++i) {
				const double h0 = H_[(size_t)i*m_ + j], h1 = H_[(size_t)(i + 1)*m_ + j];
				H_[(size_t)i*m_ + j] = cs_[i]*h0 + sn_[i]*h1;
				H_[(size_t)(i + 1)*m_ + j] = -sn_[i]*h0 + cs_[i]*h1;
			}
			const double h0 = H_[(size_t)j*m_ + j], h1 = H_[(size_t)(j + 1)*m_ + j];
			const double mag = std::hypot(h0, h1);
			cs_[j] = mag > 0.0 ? h0/mag : 1.0;
			sn_[j] = mag > 0.0 ? h1/mag : 0.0;
			H_[(size_t)j*m_ + j] = mag;
			H_[(size_t)(j + 1)*m_ + j] = 0.0;
			const double gj = g_[j];
			g_[j] = cs_[j]*gj;
			g_[j + 1] = -sn_[j]*gj;
			++res.iterations;
			used = j + 1;
			res.residual = std::abs(g_[j + 1]);
			if (res.residual <= tol) break;
			if (hn <= 1e-300) {
				breakdown = true;
				break;
			}
		}
		for (int row = used - 1; row >= 0; --row) {
			double v = g_[row];
			for (int c = row + 1; c < used; ++c) v -= H_[(size_t)row*m_ + c]*y_[c];
			const double d = H_[(size_t)row*m_ + row];
			if (std::abs(d) < 1e-300) throw Error("FGMRES Hessenberg matrix is singular");
			y_[row] = v/d;
		}
		Check(hipMemcpyAsync(h, y_.data(), sizeof(double)*used, hipMemcpyHostToDevice, ctx->stream), "y upload");
		MultiAxpy(ctx, M ? Z : V, n, used, h, nullptr, 0, 1.0, x, nullptr);
		beta = true_residual();
		res.residual = beta;
		if (beta <= tol) {
			res.converged = true;
			break;
		}
		if (breakdown) break;
		// a restart cycle that made no progress, or a residual far above the
		// initial one, means the preconditioned operator defeats the method:
		// stop early instead of spending the remaining iterations
		if (!std::isfinite(beta) || beta >= beta_cycle || beta > 10.0*beta0) break;
	}
	return res;
}

}  // namespace tfi
