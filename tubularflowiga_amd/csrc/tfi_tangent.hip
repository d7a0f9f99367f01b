// Tangent of the stabilised (VMS) Navier-Stokes equations on FP64 matrix cores
// (tau-frozen legacy form or exact consistent linearisation), for elements of
// up to kMaxBasis basis functions; the residual beside it comes from
// tfi_residual.hip.
//
// Arithmetic restated from solvers/cuda/include/IgaCudaKernels.cuh:239-409
// (legacy tangent) and the CPU element
// solvers/cpu/include/NavierStokesElement.hpp:121-313 (exact tangent, which
// differentiates tau_M, tau_C and the strong viscous term).
//
// One GEMM per element.  At a Gauss point q the block component (x, y) of a
// (test a, trial b) pair is a bilinear form in the test values phi = (N_a,
// grad N_a) and the trial values psi of b, so
//     T[a][(b, x, y)] = sum over (q, i < 4) of phi_i(a, q) B_i(b, q; x, y),
// with B_i a short combination of psi whose coefficients depend on the point
// and on (x, y) only.  The test factor is the same for all 16 components: the
// 16 columns of one v_mfma_f64_16x16x4f64 are the 16 components of ONE trial
// function (K = 4 points), no column is padding, and an accumulator tile holds
// whole 4x4 blocks: 16 neighbouring lanes hold the 128 contiguous bytes of a
// block, which go to memory without another transposition.  27 functions take
// 28 x 2 x 64 = 3584 MFMAs per element, those of the 28th trial function dropped
// (4224 when each component was a 32 x 32 product of padded functions), 64
// functions 16384 with no padding at all.
// Lane (comp = lane%16, point = lane/16) holds the 12 coefficients of its
// component at its point for a chunk of four points and forms one B value per
// MFMA column with three FMAs, used by the kTi test tiles.  FP64 FMAs and FP64
// MFMAs share the pipeline (measured: 77.7 TFLOP/s of MFMA alone, 68 with two
// FMAs to an MFMA), so the FMAs of B cost 3 x 4.6 of 64 kTi cycles.
//
// A workgroup of four waves holds the test functions of its element and 4 kTb
// of its trial functions (kTi kTb accumulator tiles per wave, at most 128
// registers), two workgroups to a CU, so that one's point work runs beside the
// other's MFMAs.  The fields and the stabilisation at the points come from the
// residual kernel, which has them anyway (21 doubles per point); per slab of
// points the workgroup puts these and the basis records (from the table,
// fetched while the MFMAs of the slab before run) into LDS, and thread (point,
// component) forms its coefficients.
//
// The blocks leave the workgroup in one of two ways, which sum in the same order
// and so to the same bits:
//   * staged: to a buffer of one block per (element, a, b), all elements in one
//     launch; a second launch sums each block's contributions in the order of
//     the elements' colours and writes the Jacobian once;
//   * by colour: added to the Jacobian, one launch per element colour (the
//     elements of a colour share no node).
//
// Measured, residual and tangent together: 109,824 elements of 27 functions
// 41.8 -> 19.7 ms (17.5 in this kernel, 41 TFLOP/s of the 77.7 the MFMAs reach
// alone), 5120 elements of 64 functions 19.5 -> 4.3 ms, 80 elements of 27
// functions 842 -> 61 us, against 8 waves per element with a product of
// padded functions per component (27 functions) and register-tiled FP64
// vector arithmetic (64).  The rest of the time is the point work, whose FP64
// operations wait behind the other workgroup's MFMAs, and the barriers of the
// four slabs.
#include "tfi_internal.hpp"
#include "tfi_point.hpp"

#include <algorithm>

namespace tfi {

namespace {

constexpr int kThreads = 256;
constexpr int kCoefs = 12;                 // per (point, component): test N, then 3 each for test dN/dx_d
constexpr int kCoefStride = 16*kCoefs + 16;  // doubles per point: the points of a chunk on different banks
constexpr int kRec = 6;                    // N, dN/dx, dN/dy, dN/dz, S, w.grad N of a function at a point

typedef double doublex4 __attribute__((ext_vector_type(4)));

struct TangentArgs {
	const int* eoff;
	const int* xoff;         // extraction rows, a column at most once per row
	const uint8_t* xcol;
	const double* xval;
	const double* geometry;
	const double* points;    // point records [item][kTangentRec][kQ]
	const double* table;     // per-element basis records [q][a][kTableRec] at eoff[e]*kQ*kTableRec, or null
	const long long* pair_offsets;
	const int* pair_block;
	const int* elements;     // element ids of this launch, or null: all in order
	int count, tiles;
	double rho, mu, dt;
	double* jac;
	double* staging;         // [pair][16], or null: added to jac
	int max_nen;
	bool atomic;             // jac is in this GPU's own coarse-grained memory
};

__host__ __device__ constexpr int PointStride(int nen) { return kRec*nen | 1; }  // odd: points on different banks

template <int kSlab>
__host__ __device__ constexpr size_t TangentLds(int nen, bool table)
{
	return sizeof(double)*(kSlab*((size_t)PointStride(nen) + kCoefStride + kTangentRec) + (table ? 0 : 64*(size_t)nen));
}

// The lane's component (x, y): 12 coefficients c and the trial values they
// multiply, as offsets into the record of the trial function: test N takes
// c[0..2] with off[0..2]; test dN/dx_d takes c[3+3d] with N, c[4+3d] with off[3]
// and c[5+3d] with off[4+d].  Of the gradient of the trial function a
// component with test direction d needs at most one entry besides off[3].
__device__ inline void TrialOffsets(int x, int y, int off[7])
{
	const bool u = x < 3, v = y < 3;
	off[0] = u ? (v ? 0 : 1) : (v ? 1 + y : 0);
	off[1] = u ? (v ? 4 : 2) : 0;
	off[2] = u ? (v ? 5 : 3) : 0;
	off[3] = u && !v ? 1 + x : 4;
#pragma unroll
	for (int d = 0; d < 3; ++d) off[4 + d] = 1 + (u && v && x != y ? (d == y ? x : d == x ? y : d) : d);
}

// Coefficients of component (x, y) at a point, from its record r in LDS (the
// entries of row x and column y are read by index, not selected).
template <bool kExact>
__device__ inline void PointCoefficients(const double* __restrict__ r, int x, int y, double rho, double mu, double idt,
	double c[kCoefs])
{
	const double m = r[0], tm = r[1], tc = r[2];
	const double* u = r + 3;
	const double* up = r + 6;
	const double* gu = r + 9;
#pragma unroll
	for (int i = 0; i < kCoefs; ++i) c[i] = 0.0;
	if (x < 3 && y < 3) {
		const bool same = x == y;
		const double mr = m*rho, mrt = mr*tm;
		if (kExact) {
			// u' varies with u_y N_b as K[.][y] N_b, K_cf = tau_M^3 strong_c (G u)_f - tau_M du_c/dx_f, and with
			// the strong operator S_b as -tau_M
			const double ux = up[x], gxy = gu[3*x + y], Guy = r[18 + y];
			double K[3], gx[3], w[3];
#pragma unroll
			for (int f = 0; f < 3; ++f) {
				K[f] = -tm*(tm*up[f]*Guy + gu[3*f + y]);
				gx[f] = gu[3*x + f];
				w[f] = u[f] + up[f];
			}
			const double Kx = -tm*(tm*ux*Guy + gu[3*x + y]);
			const double R = gxy + gx[0]*K[0] + gx[1]*K[1] + gx[2]*K[2];
			const double c1 = mr*tc*tm*tm*(gu[0] + gu[4] + gu[8])*Guy;
			c[0] = mr*(R + (same ? idt : 0.0));
			c[1] = -mrt*gxy;
			c[2] = same ? mr : 0.0;
#pragma unroll
			for (int d = 0; d < 3; ++d) {
				c[3 + 3*d] = (d == x ? c1 : 0.0) - mr*(w[d]*Kx + ux*((d == y ? 1.0 : 0.0) + K[d]));
				c[4 + 3*d] = mrt*((d == y ? ux : 0.0) + (same ? w[d] : 0.0));
			}
		} else {
			c[1] = same ? mr : 0.0;
#pragma unroll
			for (int d = 0; d < 3; ++d) c[4 + 3*d] = same ? mrt*u[d] : 0.0;
		}
		const double mm = m*mu, mc = mr*tc;
#pragma unroll
		for (int d = 0; d < 3; ++d)
			c[5 + 3*d] = same ? (d == x ? 2.0*mm + mc : mm) : (d == y ? mm : d == x ? mc : 0.0);
	} else if (x < 3) {
		const double mt = m*tm, ux = kExact ? mt*up[x] : 0.0;
#pragma unroll
		for (int d = 0; d < 3; ++d) {
			if (kExact) c[d] = -mt*gu[3*x + d];
			c[3 + 3*d] = d == x ? -m : 0.0;
			c[4 + 3*d] = mt*(kExact ? u[d] + up[d] : u[d]);
			c[5 + 3*d] = ux;
		}
	} else if (y < 3) {
		const double mt = m*tm, Guy = r[18 + y];
		c[0] = m;
#pragma unroll
		for (int d = 0; d < 3; ++d) {
			if (kExact) c[3 + 3*d] = mt*(tm*up[d]*Guy + gu[3*d + y]);
			c[4 + 3*d] = d == y ? mt : 0.0;
		}
	} else {
		const double mt = m*(tm/rho);
#pragma unroll
		for (int d = 0; d < 3; ++d) c[5 + 3*d] = mt;
	}
}

// kTi: tiles of 16 test functions (nen <= 16 kTi); kTb: trial functions per
// wave; kSlab: points per slab (8 or 16); kTable: basis records from the
// table, else evaluated from the extraction rows.
template <bool kExact, int kTi, int kTb, int kSlab, bool kTable>
__global__ void __launch_bounds__(kThreads, 2) TangentKernel(TangentArgs args)
{
	extern __shared__ double lds[];
	const int tid = threadIdx.x, lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	// workgroups are dealt to the 8 XCDs in turn: the tiles of an element stay on one
	const int local = blockIdx.x >> 3;
	const int item = (local/args.tiles)*8 + (blockIdx.x & 7);
	const int tile = local % args.tiles;
	if (item >= args.count) return;
	const int e = args.elements ? args.elements[item] : item;
	const int b0 = args.eoff[e];
	const int nen = args.eoff[e + 1] - b0;
	if (tile*4*kTb >= nen) return;
	const double idt = args.dt > 0.0 ? 1.0/args.dt : 0.0;
	const double nu = args.mu/args.rho;
	const int qs = PointStride(args.max_nen);
	double* rec = lds;                              // [kSlab][qs]: [a][kRec]
	double* coef = rec + kSlab*qs;                  // [kSlab][kCoefStride]: [coefficient][component]
	double* pt = coef + kSlab*kCoefStride;          // [kSlab][kTangentRec]
	double* C = pt + kSlab*kTangentRec;             // [nen][64] extraction rows without the table
	const double* geo = args.geometry + (size_t)e*kGeomFields*kQ;
	const double* src = args.points + (size_t)item*kTangentRec*kQ;
	const int width = nen*kTableRec;                // table entries of one point
	// a slab's table entries (even count, 16-byte aligned: slabs start at multiples of 8 points)
	// and point records, in flight while the MFMAs of the slab before run
	constexpr int kPre = kTable ? (kSlab*16*kTi*kTableRec/2 + kThreads - 1)/kThreads : 1;
	constexpr int kPrePoint = (kSlab*kTangentRec + kThreads - 1)/kThreads;
	double2 pre[kPre];
	double prep[kPrePoint];
	auto fetch = [&](int q0) {
		if constexpr (kTable) {
			const double2* t = reinterpret_cast<const double2*>(args.table + ((size_t)b0*kQ + (size_t)q0*nen)*kTableRec);
#pragma unroll
			for (int k = 0; k < kPre; ++k) {
				const int i = tid + k*kThreads;
				if (2*i < kSlab*width) pre[k] = t[i];
			}
		}
#pragma unroll
		for (int k = 0; k < kPrePoint; ++k) {
			const int i = tid + k*kThreads;
			if (i < kSlab*kTangentRec) prep[k] = src[(i/kSlab)*kQ + q0 + i%kSlab];
		}
	};
	fetch(0);
	if constexpr (!kTable) {
		for (int i = tid; i < nen*64; i += kThreads) C[i] = 0.0;
		__syncthreads();
		for (int t = tid; t < nen*8; t += kThreads) {
			const int a = t >> 3, end = args.xoff[b0 + a + 1];
			for (int k = args.xoff[b0 + a] + (t & 7); k < end; k += 8) C[64*a + args.xcol[k]] = args.xval[k];
		}
		__syncthreads();
	}
	const int comp = lane & 15, kq = lane >> 4;
	int off[7];
	TrialOffsets(comp >> 2, comp & 3, off);
	const int bw = tile*4*kTb + wave*kTb;           // first trial function of this wave
	doublex4 acc[kTi][kTb];
#pragma unroll
	for (int i = 0; i < kTi; ++i)
#pragma unroll
		for (int j = 0; j < kTb; ++j) acc[i][j] = doublex4{0.0, 0.0, 0.0, 0.0};

	// the MFMAs of four points
	auto multiply = [&](int chunk) {
		const double* point = rec + (4*chunk + kq)*qs;
		const double* pc = coef + (4*chunk + kq)*kCoefStride + comp;
		const double* test[kTi];
#pragma unroll
		for (int ti = 0; ti < kTi; ++ti) test[ti] = point + kRec*min(16*ti + comp, nen - 1);  // rows past nen are not stored
#pragma unroll
		for (int i = 0; i < 4; ++i) {
			const double c0 = pc[16*(3*i)], c1 = pc[16*(3*i + 1)], c2 = pc[16*(3*i + 2)];
			double A[kTi];
#pragma unroll
			for (int ti = 0; ti < kTi; ++ti) A[ti] = test[ti][i];
			const int o0 = i == 0 ? off[0] : 0, o1 = i == 0 ? off[1] : off[3], o2 = i == 0 ? off[2] : off[3 + i];
#pragma unroll
			for (int tb = 0; tb < kTb; ++tb) {
				const double* r = point + kRec*(bw + tb);  // past nen: whatever follows in LDS, not stored
				const double B = c0*r[o0] + c1*r[o1] + c2*r[o2];
#pragma unroll
				for (int ti = 0; ti < kTi; ++ti)
					acc[ti][tb] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[ti], B, acc[ti][tb], 0, 0, 0);
			}
		}
	};

#pragma unroll 1
	for (int q0 = 0; q0 < kQ; q0 += kSlab) {
		// the point work goes first: behind another workgroup's MFMAs it would hold up this one's
		__builtin_amdgcn_s_setprio(2);
		// ---- the slab's basis records (N, grad N, lap N) and point records to LDS
		if constexpr (kTable) {
			// entry 2 t = (point ql, offset r), advanced by 2 kThreads without a division; the
			// addresses are not kept from slab to slab (t is opaque): the registers hold accumulators
			int t = tid;
			asm volatile("" : "+v"(t));
			const int dq = 2*kThreads/width, dr = 2*kThreads - dq*width;
			int ql = 2*t/width, r = 2*t - ql*width;
#pragma unroll
			for (int k = 0; k < kPre; ++k) {
				if (ql >= kSlab) break;
				const int a = r/kTableRec;
				rec[ql*qs + kRec*a + (r - a*kTableRec)] = pre[k].x;
				const int q1 = r + 1 == width ? ql + 1 : ql, r1 = r + 1 == width ? 0 : r + 1, a1 = r1/kTableRec;
				rec[q1*qs + kRec*a1 + (r1 - a1*kTableRec)] = pre[k].y;
				ql += dq;
				r += dr;
				if (r >= width) {
					r -= width;
					++ql;
				}
			}
		} else {
			for (int it = tid; it < nen*kSlab; it += kThreads) {
				const int a = it/kSlab, ql = it - a*kSlab;
				EvalBasis(C + 64*a, geo + q0 + ql, q0 + ql, rec + ql*qs + kRec*a);
			}
		}
#pragma unroll
		for (int k = 0; k < kPrePoint; ++k) {
			const int i = tid + k*kThreads;
			if (i < kSlab*kTangentRec) pt[(i%kSlab)*kTangentRec + i/kSlab] = prep[k];
		}
		__syncthreads();
		// ---- coefficients: thread (point, component)
		if (tid < 16*kSlab) {
			const int ql = tid >> 4, k = tid & 15;
			double c[kCoefs];
			PointCoefficients<kExact>(pt + ql*kTangentRec, k >> 2, k & 3, args.rho, args.mu, idt, c);
#pragma unroll
			for (int i = 0; i < kCoefs; ++i) coef[ql*kCoefStride + 16*i + k] = c[i];
		}
		// ---- S = N/dt + u.grad N - nu lap N (legacy: without the last term) and w.grad N
		for (int it = tid; it < nen*kSlab; it += kThreads) {
			const int a = it/kSlab, ql = it - a*kSlab;
			double* r = rec + ql*qs + kRec*a;
			const double* v = pt + ql*kTangentRec + 3;
			const double g0 = r[1], g1 = r[2], g2 = r[3];
			const double U = v[0]*g0 + v[1]*g1 + v[2]*g2;
			const double S = r[0]*idt + U;
			r[4] = kExact ? S - nu*r[4] : S;
			r[5] = U + v[3]*g0 + v[4]*g1 + v[5]*g2;
		}
		__syncthreads();
		if (q0 + kSlab < kQ) fetch(q0 + kSlab);
		__builtin_amdgcn_s_setprio(0);
		// ---- four points per MFMA
		if (bw < nen)
#pragma unroll 1
			for (int chunk = 0; chunk < kSlab/4; ++chunk) multiply(chunk);
		__syncthreads();
	}

	// ---- blocks out: element i of a lane's accumulator is row 16 ti + 4 i + kq
	const long long pbase = args.pair_offsets[e];
	if (args.staging) {
		double* out = args.staging + 16*pbase + comp;
#pragma unroll
		for (int tb = 0; tb < kTb; ++tb)
#pragma unroll
			for (int ti = 0; ti < kTi; ++ti)
#pragma unroll
				for (int i = 0; i < 4; ++i) {
					const int a = 16*ti + 4*i + kq, b = bw + tb;
					if (a < nen && b < nen) out[16*(a*nen + b)] = acc[ti][tb][i];
				}
		return;
	}
	// Every Jacobian entry receives at most one contribution per launch (the
	// blocks of one colour are disjoint), so the order of the sums is the order of
	// the launches.  In the GPU's own memory an atomic leaves the read-modify-write
	// to the L2, and nothing waits for the old values (1,683,072 elements of 27
	// functions 267 ms, loaded and stored 273; 109,824 elements 19.18 and 19.26).
	// Other memory a kernel can write (pinned, managed, another GPU's) does not
	// carry out FP64 atomics.
	if (args.atomic) {
		int slot[kTb][4*kTi];
#pragma unroll
		for (int tb = 0; tb < kTb; ++tb)
#pragma unroll
			for (int k = 0; k < 4*kTi; ++k)
				slot[tb][k] = args.pair_block[pbase + min(4*k + kq, nen - 1)*nen + min(bw + tb, nen - 1)];
#pragma unroll
		for (int tb = 0; tb < kTb; ++tb)
#pragma unroll
			for (int k = 0; k < 4*kTi; ++k)
				if (4*k + kq < nen && bw + tb < nen)
					__hip_atomic_fetch_add(args.jac + (size_t)slot[tb][k]*16 + comp, acc[k/4][tb][k%4], __ATOMIC_RELAXED,
						__HIP_MEMORY_SCOPE_WORKGROUP);
		return;
	}
#pragma unroll
	for (int tb = 0; tb < kTb; ++tb)
#pragma unroll
		for (int k = 0; k < 4*kTi; ++k)
			if (4*k + kq < nen && bw + tb < nen)
				args.jac[(size_t)args.pair_block[pbase + (4*k + kq)*nen + bw + tb]*16 + comp] += acc[k/4][tb][k%4];
}

// jac[block] = sum of the block's staged contributions, in colour order (16 lanes per block)
__global__ void __launch_bounds__(kThreads) BlockSumKernel(long long blocks, const int* __restrict__ offsets,
	const int* __restrict__ pairs, const double* __restrict__ staging, double* __restrict__ jac)
{
	const long long t = blockIdx.x*(long long)kThreads + threadIdx.x;
	const long long block = t >> 4;
	if (block >= blocks) return;
	const int c = static_cast<int>(t & 15);
	const int begin = offsets[block], end = offsets[block + 1];
	double s = 0.0;
#pragma unroll 4
	for (int k = begin; k < end; ++k) s += staging[16*(size_t)pairs[k] + c];
	jac[16*block + c] = s;
}

__global__ void CountPairsKernel(int pairs, const int* __restrict__ pair_block, int* __restrict__ count)
{
	const int p = blockIdx.x*blockDim.x + threadIdx.x;
	if (p < pairs) atomicAdd(count + pair_block[p], 1);
}

// Appends the pairs of one colour's elements to their blocks' lists; cursor holds each
// block's next place.  The elements of a colour share no node, so no two threads meet.
__global__ void __launch_bounds__(kThreads) FillPairsKernel(const int* __restrict__ elements,
	const long long* __restrict__ pair_offsets, const int* __restrict__ pair_block, int* __restrict__ cursor,
	int* __restrict__ list)
{
	const int e = elements[blockIdx.x];
	const int end = static_cast<int>(pair_offsets[e + 1]);
	for (int p = static_cast<int>(pair_offsets[e]) + threadIdx.x; p < end; p += kThreads)
		list[cursor[pair_block[p]]++] = p;
}

// Staged while the blocks of all elements take at most 4 GiB (46,000 elements of
// 27 functions, 8,192 of 64), else by colour.  A colour is a launch of its own,
// whose last workgroups leave CUs idle, and waits for the one before: 80
// elements of 27 functions 602 us by colour and 61 staged, 5120 of 64
// functions 10.0 and 4.3 ms.  The staged blocks cost one more pass over
// themselves; with 4067 elements per colour (109,824 in all, 10 GB of blocks)
// the two take the same time (19.9 ms by colour, 20.4 staged), so the memory
// decides: beside the 4 GiB, a quarter of what is free at the mesh's first
// tangent assembly.
constexpr long long kStageBytes = 4LL << 30;

// The staging buffer and the pairs of each block, built by the mesh's first tangent assembly
void PrepareStaging(tfi_mesh* m)
{
	if (m->staging.size()) return;
	tfi_ctx* ctx = m->ctx;
	const int pairs = static_cast<int>(m->element_pairs);
	const int grid = (pairs + kThreads - 1)/kThreads;
	DevBuf<int> cursor(ctx, m->nnzb);
	FillInt(ctx, cursor.data(), 0, m->nnzb);
	hipLaunchKernelGGL(CountPairsKernel, dim3(grid), dim3(kThreads), 0, ctx->stream, pairs, m->pair_block.data(),
		cursor.data());
	TFI_LAUNCH_CHECK("CountPairsKernel");
	std::vector<int> offsets(m->nnzb + 1, 0);
	cursor.Download(offsets.data() + 1, m->nnzb);
	for (long long k = 0; k < m->nnzb; ++k) offsets[k + 1] += offsets[k];
	cursor.Upload(offsets.data(), m->nnzb);
	m->block_offsets.Allocate(ctx, m->nnzb + 1);
	m->block_offsets.Upload(offsets.data(), m->nnzb + 1);
	m->block_pairs.Allocate(ctx, pairs);
	for (int c = 0; c < m->colors; ++c) {
		hipLaunchKernelGGL(FillPairsKernel, dim3(m->color_offsets[c + 1] - m->color_offsets[c]), dim3(kThreads), 0,
			ctx->stream, m->color_elements.data() + m->color_offsets[c], m->pair_offsets.data(), m->pair_block.data(),
			cursor.data(), m->block_pairs.data());
		TFI_LAUNCH_CHECK("FillPairsKernel");
	}
	Sync(ctx);
	m->staging.Allocate(ctx, 16*(size_t)pairs);
}

// Memory of this GPU in which FP64 atomics are carried out: plain device allocations.
bool OwnMemory(const tfi_ctx* ctx, const void* p)
{
	hipPointerAttribute_t a{};
	Check(hipPointerGetAttributes(&a, p), "hipPointerGetAttributes");
	return a.type == hipMemoryTypeDevice && !a.isManaged && a.allocationFlags == 0 && a.device == ctx->device;
}

struct Inputs {
	const double* state;
	const double* previous;
	NsParams params;
};

template <bool kExact, int kTi, int kTb, int kSlab, bool kTable>
int LaunchTangent(tfi_mesh* m, TangentArgs a, const Inputs& in, bool staged)
{
	tfi_ctx* ctx = m->ctx;
	const size_t lds = TangentLds<kSlab>(m->max_nen, kTable);
	const void* kernel = reinterpret_cast<const void*>(TangentKernel<kExact, kTi, kTb, kSlab, kTable>);
	if (lds > 65536)
		Check(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)),
			"hipFuncSetAttribute");
	a.tiles = (m->max_nen + 4*kTb - 1)/(4*kTb);
	int launches = 0;
	auto launch = [&](const int* elements, int count) {
		if (count == 0) return;
		ElementResiduals(m, in.state, in.previous, in.params, elements, count, m->point_records.data());
		a.elements = elements;
		a.count = count;
		hipLaunchKernelGGL((TangentKernel<kExact, kTi, kTb, kSlab, kTable>), dim3((count + 7)/8*8*a.tiles),
			dim3(kThreads), lds, ctx->stream, a);
		TFI_LAUNCH_CHECK("TangentKernel");
		++launches;
	};
	if (staged) {
		launch(nullptr, m->elements);
	} else {
		for (int c = 0; c < m->colors; ++c)
			launch(m->color_elements.data() + m->color_offsets[c], m->color_offsets[c + 1] - m->color_offsets[c]);
	}
	return launches;
}

// Trial functions per wave: the most whose accumulators (kTi kTb tiles of 8
// registers) leave room for two waves per SIMD, or fewer (kFew) while the mesh
// is too small to give every CU two workgroups of that size.
template <bool kExact, bool kTable, int kTi, int kTb, int kFew, int kSlab>
int LaunchWidth(tfi_mesh* m, const TangentArgs& a, const Inputs& in, bool staged)
{
	const long long workgroups = (long long)m->elements*((m->max_nen + 4*kTb - 1)/(4*kTb));
	return staged && workgroups < 2LL*m->ctx->cus ? LaunchTangent<kExact, kTi, kFew, kSlab, kTable>(m, a, in, staged)
		: LaunchTangent<kExact, kTi, kTb, kSlab, kTable>(m, a, in, staged);
}

template <bool kExact, bool kTable>
int LaunchClass(tfi_mesh* m, const TangentArgs& a, const Inputs& in, bool staged)
{
	// 28 functions: 7 per wave (27, the quadratic spline element, computes one of 28 in vain);
	// slabs of 16 points while two workgroups' LDS fit a CU, 8 above 32 functions
	const int nen = m->max_nen;
	if (nen <= 28) return LaunchWidth<kExact, kTable, 2, 7, 2, 16>(m, a, in, staged);
	if (nen <= 32) return LaunchWidth<kExact, kTable, 2, 8, 2, 16>(m, a, in, staged);
	if (nen <= 48) return LaunchWidth<kExact, kTable, 3, 5, 1, 8>(m, a, in, staged);
	if (nen <= 64) return LaunchWidth<kExact, kTable, 4, 4, 1, 8>(m, a, in, staged);
	return LaunchWidth<kExact, kTable, 5, 3, 1, 8>(m, a, in, staged);
}

}  // namespace

void AssembleNs(tfi_mesh* m, const double* state, const double* previous, const NsParams& p, double* jacobian,
	double* negative_residual)
{
	const bool exact = p.tangent == TFI_TANGENT_EXACT;
	if (m->max_nen > kMaxBasis) throw Error("element assembly supports at most 80 basis functions per element");
	tfi_ctx* ctx = m->ctx;
	if (!jacobian) {
		StreamTimer timer(ctx, &ctx->timers.residual_ms);
		ElementResiduals(m, state, previous, p, nullptr, m->elements, nullptr);
		SumResiduals(m, negative_residual);
		ctx->timers.residual_calls += 1;
		ctx->timers.residual_flops += AssemblyFlops(m, false, exact);
		return;
	}
	const bool table = m->basis_table.size() > 0;
	if (m->staged < 0) {
		size_t free_bytes = 0, total_bytes = 0;
		Check(hipMemGetInfo(&free_bytes, &total_bytes), "hipMemGetInfo");
		const long long bytes = 128LL*m->element_pairs;
		m->staged = bytes <= kStageBytes && bytes <= static_cast<long long>(free_bytes/4) ? 1 : 0;
	}
	const bool staged = m->staged == 1;
	if (staged) PrepareStaging(m);
	StreamTimer timer(ctx, &ctx->timers.assembly_ms);
	if (!m->point_records.size()) {
		int count = m->elements;
		if (!staged) {
			count = 0;
			for (int c = 0; c < m->colors; ++c) count = std::max(count, m->color_offsets[c + 1] - m->color_offsets[c]);
		}
		m->point_records.Allocate(ctx, (size_t)count*kTangentRec*kQ);
	}
	if (!staged) Fill(ctx, jacobian, 0.0, m->nnzb*16);
	const ExtractionRows rows = m->rows();
	const TangentArgs a{m->eoff.data(), rows.offsets, rows.columns, rows.values, m->geometry.data(),
		m->point_records.data(), table ? m->basis_table.data() : nullptr, m->pair_offsets.data(), m->pair_block.data(),
		nullptr, 0, 0, p.density, p.viscosity, p.dt, jacobian, staged ? m->staging.data() : nullptr, m->max_nen,
		!staged && OwnMemory(ctx, jacobian)};
	const Inputs in{state, previous, p};
	int launches = 0;
	if (exact) launches = table ? LaunchClass<true, true>(m, a, in, staged) : LaunchClass<true, false>(m, a, in, staged);
	else launches = table ? LaunchClass<false, true>(m, a, in, staged) : LaunchClass<false, false>(m, a, in, staged);
	if (staged) {
		hipLaunchKernelGGL(BlockSumKernel, dim3(static_cast<unsigned>((m->nnzb*16 + kThreads - 1)/kThreads)),
			dim3(kThreads), 0, ctx->stream, m->nnzb, m->block_offsets.data(), m->block_pairs.data(), m->staging.data(),
			jacobian);
		TFI_LAUNCH_CHECK("BlockSumKernel");
	}
	SumResiduals(m, negative_residual);
	ctx->timers.assembly_calls += 1;
	ctx->timers.assembly_launches += launches;
	ctx->timers.assembly_flops += AssemblyFlops(m, true, exact);
}

}  // namespace tfi
