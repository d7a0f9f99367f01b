// Residual of the stabilised (VMS) Navier-Stokes equations without the tangent
// (Newton checks, chord steps, warm-start candidates, and the right-hand side
// beside a tangent), for elements of up to kMaxBasis basis functions.
//
// Nothing tabulated per basis function is read: the element's nodal values are
// turned into the 64 Bernstein coefficients of each field by its sparse extraction
// operator, the fields and their derivatives at the 4x4x4 Gauss points follow by
// sum factorisation (one 4-point contraction per direction), and the fluxes return
// to the basis functions the same way, transposed.  Per element of 27 functions
// that reads about 13 KB (extraction 4.3 KB, J^-1, measure and h 6.7 KB, nodal
// values) instead of the 69 KB basis table twice over.  The four waves of the
// workgroup hold one field each (u, v, w with their previous values; p) on the
// way in and one residual component each on the way out.
//
// What bounds it: the chain of an element's dependent loads and stages, with four
// workgroups a CU.  So the first loads are asked for together and the geometry
// before it is used, and the contractions are matrix products of 4 x 4 tables, in
// which a lane reads one value and no table where a sum per lane reads four of
// each (LDS was busy for half of the kernel's time with those sums; now for a
// quarter).  Between the contractions a wave exchanges two of its three lane
// indices through LDS by itself, without a barrier.
//
// The element rows go to a buffer of one row per (element, basis function) and
// a second launch sums each node's rows in element order: a fixed order without
// atomics, two launches whatever the number of element colours.
//
// Measured, kernel and node sums, 109,824 elements of 27 functions: 2714 us for the
// form that read the table (one launch per colour), 1588 us with the contractions
// as sums per lane, 1404 us as matrix products, 1200 us with the early loads; 5120
// elements of 64 functions: 5018 (the tangent kernel run without its tangent), 127,
// 115 and 111 us.  Five workgroups a CU spill registers (1394 us before the early
// loads); the final rows from entries kept since the start, eight lanes a row, take
// the registers of the fourth (1277 us).
#include "tfi_internal.hpp"
#include "tfi_point.hpp"

#include <algorithm>

namespace tfi {

namespace {

constexpr int kThreads = 256;
constexpr int kFields = 22;  // u (3), p, grad u (9), grad p (3), lap u (3), u_prev (3): the order PointRecord takes

struct ResidualArgs {
	const int* eoff;
	const int* conn;
	const int* xoff;      // extraction rows, a column at most once per row
	const uint8_t* xcol;
	const double* xval;
	const double* geometry;
	const double* state;
	const double* previous;
	double rho, mu, dt;
	double* rows;         // [entries][4]
	const int* elements;  // element ids of this launch, or null: all in order
	double* points;       // tangent records [workgroup][kTangentRec][kQ], or null
};

// LDS in doubles: P holds, in turn, the dense extraction rows [nen][64] (columns of
// odd rows with bit 4 turned, see Dense), the waves' scratch [wave][7][kTurn] and
// the fluxes [4][4][64], a wave's own part of them its scratch on the way out; Q
// the Bernstein coefficients [8][kTurn], the fields at the points [kFields][64] and
// the Bernstein residual [64][4].
constexpr int kTurn = 72;
constexpr int kEarly = 4;  // entries of an extraction row that a lane asks for ahead: 32 a row
constexpr int kQDoubles = kFields*64;
static_assert(kQDoubles >= 8*kTurn, "the Bernstein coefficients fit Q");
static_assert(3*kTurn <= 4*64, "the transposed sums fit the wave's own fluxes");
__host__ __device__ constexpr int Rows4(int nen) { return (nen + 3) & ~3; }
__host__ __device__ constexpr int PDoubles(int nen) { return Rows4(nen)*64 > 4*7*kTurn ? Rows4(nen)*64 : 4*7*kTurn; }

// The contractions: v_mfma_f64_4x4x4 takes four products of 4 x 4 matrices, lane
// l the entry A[l%4][l/16], B[l/16][l%4] and D[l/16][l%4] of product (l/4)%4.
// With a table of basis values as A in all four, it sums a 4 x 4 x 4 field over
// the index that lanes hold in their bits 4, 5 and leaves the new index there.
__device__ inline double Contract(double table, double v, double sum = 0.0)
{
	return __builtin_amdgcn_mfma_f64_4x4x4f64(table, v, sum, 0, 0, 0);
}

// A field of the wave with two of its lane indices exchanged, through LDS: bits
// (0, 1) with (4, 5), and bits (2, 3) with (4, 5).  The upper half lies two and
// eight doubles further on: no bank is asked for twice.
__device__ inline void TurnLowStore(double* o, int lane, double v) { o[lane + 2*(lane >> 5)] = v; }
__device__ inline double TurnLowLoad(const double* o, int lane)
{
	return o[(lane >> 4) + (lane & 12) + 16*(lane & 3) + (lane & 2)];
}
__device__ inline void TurnMiddleStore(double* o, int lane, double v) { o[lane + 8*(lane >> 5)] = v; }
__device__ inline double TurnMiddleLoad(const double* o, int lane)
{
	return o[(lane & 3) + 4*(lane >> 4) + 4*(lane & 12) + (lane & 8)];
}

// LDS accesses of one wave take effect in the order of the program: between them
// only the compiler has to be held.
__device__ inline void WaveFence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

// Place of extraction entry (a, q) in P: with a row's 16 columns a wave reads and
// those of the row after it on different banks.
__device__ inline int Dense(int a, int q) { return 64*a + (q ^ ((a & 1) << 4)); }

// four waves per SIMD: 124 registers; without the bound 132, three
__global__ void __launch_bounds__(kThreads, 4) NsResidualKernel(ResidualArgs args, int max_nen)
{
	extern __shared__ double lds[];
	double* P = lds;
	double* Q = P + PDoubles(max_nen);
	double* nodal = Q + kQDoubles;           // [nen, to a multiple of 4][u, u_prev, v, v_prev, w, w_prev, p, 0]
	double* tab = nodal + 8*Rows4(max_nen);  // [B, B', B''][Gauss point][Bernstein index]
	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int e = args.elements ? args.elements[blockIdx.x] : blockIdx.x;
	const int b0 = args.eoff[e];
	const int nen = args.eoff[e + 1] - b0, nen4 = Rows4(nen);
	// first loads of the chains conn -> state and xoff -> entries, then the second
	// ones; a thread holds the first kEarly entries of its eighth of a row
	const int row = min(tid >> 3, nen - 1);
	const int node = args.conn[b0 + min(tid >> 2, nen - 1)];
	const int end = tid < nen*8 ? args.xoff[b0 + row + 1] : 0, begin = args.xoff[b0 + row] + (tid & 7);
	double now = args.state[4*(size_t)node + (tid & 3)], before = args.previous[4*(size_t)node + min(tid & 3, 2)];
	double xv[kEarly];
	int xc[kEarly];
#pragma unroll
	for (int i = 0; i < kEarly; ++i)
		if (begin + 8*i < end) {
			xv[i] = args.xval[begin + 8*i];
			xc[i] = args.xcol[begin + 8*i];
		}
	for (int i = tid; i < nen4*64; i += kThreads) P[i] = 0.0;
	for (int i = tid; i < nen4*4; i += kThreads) {
		const int a = i >> 2, f = i & 3;
		if (i != tid && a < nen) {
			const size_t at = 4*(size_t)args.conn[b0 + a] + f;
			now = args.state[at];
			before = args.previous[f < 3 ? at : at - 1];
		}
		nodal[8*a + 2*f] = a < nen ? now : 0.0;
		nodal[8*a + 2*f + 1] = a < nen && f < 3 ? before : 0.0;
	}
	if (tid < 4) {
		double b[4], d[4], h[4];
		Bern3(kGp[tid], b, d, h);
		for (int i = 0; i < 4; ++i) {
			tab[4*tid + i] = b[i];
			tab[16 + 4*tid + i] = d[i];
			tab[32 + 4*tid + i] = h[i];
		}
	}
	__syncthreads();
#pragma unroll
	for (int i = 0; i < kEarly; ++i)
		if (begin + 8*i < end) P[Dense(row, xc[i])] = xv[i];
	for (int k = begin + 8*kEarly; k < end; k += 8) P[Dense(row, args.xcol[k])] = args.xval[k];
	for (int t = tid + kThreads; t < nen*8; t += kThreads) {
		const int a = t >> 3, last = args.xoff[b0 + a + 1];
		for (int k = args.xoff[b0 + a] + (t & 7); k < last; k += 8) P[Dense(a, args.xcol[k])] = args.xval[k];
	}
	__syncthreads();
	const double* gq = args.geometry + (size_t)e*kGeomFields*kQ + lane;
	double inv[3][3];  // asked for here, used at the points
#pragma unroll
	for (int i = 0; i < 9; ++i) inv[i/3][i%3] = gq[(1 + i)*kQ];
	// Bernstein coefficients of all fields: a wave takes 16 of them, four in each
	// product, and four basis functions an instruction
	{
		const double* row = P + Dense(lane >> 4, 16*wave + (lane & 15));
		const double* n = nodal + 8*(lane >> 4) + (lane & 3);
		double c0 = 0.0, c1 = 0.0;
		for (int a = 0; a < nen4; a += 4) {
			const double x = row[64*a];
			c0 = Contract(x, n[8*a], c0);
			c1 = Contract(x, n[8*a + 4], c1);
		}
		const int q = 16*wave + (lane & 12) + (lane >> 4);
		double* o = Q + (lane & 3)*kTurn + q + 2*(q >> 5);
		o[0] = c0;
		o[4*kTurn] = c1;
	}
	__syncthreads();
	// from here to the points each wave by itself, its field and previous values:
	// lane (y, z, x), then (X, z, y), then (X, Y, z), contracted over the last
	double* scratch = P + wave*7*kTurn;
	const double* coef = Q + 2*wave*kTurn + (lane >> 4) + 4*(lane & 15) + ((lane & 8) >> 2);
	double v = coef[0], old = coef[kTurn];
	__syncthreads();
	{
		const double* t = tab + 4*(lane & 3) + (lane >> 4);
		const double B = t[0], D = t[16], H = t[32];
		TurnLowStore(scratch, lane, Contract(B, v));
		TurnLowStore(scratch + kTurn, lane, Contract(D, v));
		TurnLowStore(scratch + 2*kTurn, lane, Contract(H, v));
		TurnLowStore(scratch + 3*kTurn, lane, Contract(B, old));
		WaveFence();
		const double b = TurnLowLoad(scratch, lane), d = TurnLowLoad(scratch + kTurn, lane),
			h = TurnLowLoad(scratch + 2*kTurn, lane), p = TurnLowLoad(scratch + 3*kTurn, lane);
		WaveFence();
		// [order in xi][order in eta]
		TurnMiddleStore(scratch, lane, Contract(B, b));
		TurnMiddleStore(scratch + kTurn, lane, Contract(D, b));
		TurnMiddleStore(scratch + 2*kTurn, lane, Contract(H, b));
		TurnMiddleStore(scratch + 3*kTurn, lane, Contract(B, d));
		TurnMiddleStore(scratch + 4*kTurn, lane, Contract(D, d));
		TurnMiddleStore(scratch + 5*kTurn, lane, Contract(B, h));
		TurnMiddleStore(scratch + 6*kTurn, lane, Contract(B, p));
		WaveFence();
		const double s00 = TurnMiddleLoad(scratch, lane), s01 = TurnMiddleLoad(scratch + kTurn, lane),
			s02 = TurnMiddleLoad(scratch + 2*kTurn, lane), s10 = TurnMiddleLoad(scratch + 3*kTurn, lane),
			s11 = TurnMiddleLoad(scratch + 4*kTurn, lane), s20 = TurnMiddleLoad(scratch + 5*kTurn, lane);
		old = Contract(B, TurnMiddleLoad(scratch + 6*kTurn, lane));
		v = Contract(B, s00);
		const double g0 = Contract(B, s10), g1 = Contract(B, s01), g2 = Contract(D, s00);
		// the pull-back: lane = Gauss point
		Q[wave*64 + lane] = v;
#pragma unroll
		for (int d2 = 0; d2 < 3; ++d2) Q[(4 + 3*wave + d2)*64 + lane] = g0*inv[0][d2] + g1*inv[1][d2] + g2*inv[2][d2];
		if (wave < 3) {
			const double h00 = Contract(B, s20), h11 = Contract(B, s02), h22 = Contract(H, s00);
			const double h01 = Contract(B, s11), h02 = Contract(D, s10), h12 = Contract(D, s01);
			double m[3][3];
#pragma unroll
			for (int c = 0; c < 3; ++c)
#pragma unroll
				for (int d2 = c; d2 < 3; ++d2) m[c][d2] = inv[c][0]*inv[d2][0] + inv[c][1]*inv[d2][1] + inv[c][2]*inv[d2][2];
			Q[(16 + wave)*64 + lane] = h00*m[0][0] + h11*m[1][1] + h22*m[2][2]
				+ 2.0*(h01*m[0][1] + h02*m[0][2] + h12*m[1][2])
				+ g0*gq[16*kQ] + g1*gq[17*kQ] + g2*gq[18*kQ];
			Q[(19 + wave)*64 + lane] = old;
		}
	}
	__syncthreads();
	// fluxes at the points: the factor of N_a and, pulled back to the parametric
	// directions, that of grad N_a, times the measure
	if (wave == 0) {
		double s[kFields], r[kPointRecord];
#pragma unroll
		for (int i = 0; i < kFields; ++i) s[i] = Q[i*64 + lane];
		PointRecord<kQ>(s, gq, args.rho, args.mu, args.mu/args.rho, args.dt, r);
		if (args.points) {
			double* o = args.points + (size_t)blockIdx.x*kTangentRec*kQ + lane;
#pragma unroll
			for (int i = 0; i < 6; ++i) o[i*kQ] = r[i];
#pragma unroll
			for (int i = 0; i < 3; ++i) {
				o[(6 + i)*kQ] = r[19 + i];
				o[(18 + i)*kQ] = r[34 + i];
			}
#pragma unroll
			for (int i = 0; i < 9; ++i) o[(9 + i)*kQ] = r[25 + i];
		}
		const double m = -r[0];
#pragma unroll
		for (int c = 0; c < 4; ++c) {
			const double f[3] = {c < 3 ? r[9 + 3*c] : -r[19], c < 3 ? r[10 + 3*c] : -r[20],
				c < 3 ? r[11 + 3*c] : -r[21]};
			double* o = P + (4*c)*64 + lane;
			o[0] = m*(c < 3 ? r[6 + c] : r[18]);
#pragma unroll
			for (int k = 0; k < 3; ++k) o[64*(1 + k)] = m*(inv[k][0]*f[0] + inv[k][1]*f[1] + inv[k][2]*f[2]);
		}
	}
	__syncthreads();
	// transposed sums of the wave's residual component: zeta, eta, xi
	{
		double* s = P + 4*wave*64;
		const double* t = tab + 4*(lane >> 4) + (lane & 3);
		const double B = t[0], D = t[16];
		const double f0 = s[lane], f1 = s[64 + lane], f2 = s[128 + lane], f3 = s[192 + lane];
		WaveFence();
		TurnMiddleStore(s, lane, Contract(D, f3, Contract(B, f0)));
		TurnMiddleStore(s + kTurn, lane, Contract(B, f1));
		TurnMiddleStore(s + 2*kTurn, lane, Contract(B, f2));
		WaveFence();
		const double a1 = TurnMiddleLoad(s, lane), a2 = TurnMiddleLoad(s + kTurn, lane),
			a3 = TurnMiddleLoad(s + 2*kTurn, lane);
		WaveFence();
		TurnLowStore(s, lane, Contract(D, a3, Contract(B, a1)));
		TurnLowStore(s + kTurn, lane, Contract(B, a2));
		WaveFence();
		const double b1 = TurnLowLoad(s, lane), b2 = TurnLowLoad(s + kTurn, lane);
		const int q = (lane >> 4) + 4*(lane & 15);  // lane (y, z, x)
		Q[4*q + wave] = Contract(D, b2, Contract(B, b1));
	}
	__syncthreads();
	for (int t = tid; t < nen*4; t += kThreads) {
		const int a = t >> 2, c = t & 3, end = args.xoff[b0 + a + 1];
		double r = 0.0;
#pragma unroll 4
		for (int k = args.xoff[b0 + a]; k < end; ++k) r += args.xval[k]*Q[4*args.xcol[k] + c];
		args.rows[4*((size_t)b0 + a) + c] = r;
	}
}

// negres[node] = sum of the node's element rows, in element order
__global__ void __launch_bounds__(kThreads) NodeSumKernel(int nodes, const int* __restrict__ offsets,
	const int* __restrict__ entries, const double* __restrict__ rows, double* __restrict__ negres)
{
	const long long t = blockIdx.x*(long long)kThreads + threadIdx.x;
	const int node = static_cast<int>(t >> 2), c = static_cast<int>(t & 3);
	if (node >= nodes) return;
	double s = 0.0;
#pragma unroll 4
	for (int k = offsets[node]; k < offsets[node + 1]; ++k) s += rows[4*(size_t)entries[k] + c];
	negres[4*(size_t)node + c] = s;
}

}  // namespace

void ElementResiduals(tfi_mesh* m, const double* state, const double* previous, const NsParams& p, const int* elements,
	int count, double* points)
{
	if (count == 0) return;
	tfi_ctx* ctx = m->ctx;
	if (!m->element_rows.size()) m->element_rows.Allocate(ctx, 4*(size_t)m->basis_entries);
	const ExtractionRows rows = m->rows();
	ResidualArgs a{m->eoff.data(), m->conn.data(), rows.offsets, rows.columns, rows.values, m->geometry.data(),
		state, previous, p.density, p.viscosity, p.dt, m->element_rows.data(), elements, points};
	const int nen = m->max_nen;
	const size_t lds = sizeof(double)*(PDoubles(nen) + kQDoubles + 8*(size_t)Rows4(nen) + 48);
	static_assert(sizeof(double)*(PDoubles(kMaxBasis) + kQDoubles + 8*Rows4(kMaxBasis) + 48) <= 65536,
		"the largest element fits the default dynamic LDS");
	hipLaunchKernelGGL(NsResidualKernel, dim3(count), dim3(kThreads), lds, ctx->stream, a, nen);
	TFI_LAUNCH_CHECK("NsResidualKernel");
}

void SumResiduals(tfi_mesh* m, double* negative_residual)
{
	hipLaunchKernelGGL(NodeSumKernel, dim3(static_cast<unsigned>((4LL*m->nodes + kThreads - 1)/kThreads)),
		dim3(kThreads), 0, m->ctx->stream, m->nodes, m->node_offsets.data(), m->node_entries.data(),
		m->element_rows.data(), negative_residual);
	TFI_LAUNCH_CHECK("NodeSumKernel");
}

}  // namespace tfi
