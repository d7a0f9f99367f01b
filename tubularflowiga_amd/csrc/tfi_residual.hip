// Residual of the stabilised (VMS) Navier-Stokes equations without the tangent
// (Newton checks, chord steps, warm-start candidates, and the right-hand side
// beside a tangent), for elements of up to kMaxBasis basis functions.
//
// What bounds it: the bytes of the element, so nothing tabulated per basis
// function is read.  The element's nodal values are turned into the 64
// Bernstein coefficients of each field by its sparse extraction operator, the
// fields and their derivatives at the 4x4x4 Gauss points follow by sum
// factorisation (one 4-point contraction per direction), and the fluxes return
// to the basis functions the same way, transposed.  Per element of 27 functions
// that reads about 13 KB (extraction 4.3 KB, J^-1, measure and h 6.7 KB, nodal
// values) instead of the 69 KB basis table twice over.  The four waves of the
// workgroup hold one field each (u, v, w with their previous values; p) on the
// way in and one residual component each on the way out; a lane is a Bernstein
// coefficient, a Gauss point or one of the mixed indices in between, so all 64
// lanes work at every stage.
//
// The element rows go to a buffer of one row per (element, basis function) and
// a second launch sums each node's rows in element order: a fixed order without
// atomics, two launches whatever the number of element colours.
//
// Measured, kernel and node sums: 109,824 elements of 27 functions 2714 ->
// 1588 us against the form that read the table (one launch per colour); 5120
// elements of 64 functions 5018 -> 127 us against the tangent kernel run
// without its tangent.
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
	const int* xoff;
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

// LDS in doubles: P holds, in turn, the dense extraction rows [nen][64], the
// xi-eta sums [wave][7][64], the fluxes [4][4][64] and the second transposed
// sums [4][2][64]; Q the Bernstein coefficients [wave][2][64] and the xi sums
// [wave][4][64] behind them, the fields at the points [kFields][64], the first
// transposed sums [4][3][64] and the Bernstein residual [64][4].
constexpr int kQDoubles = (2 + 4)*4*64;
static_assert(kQDoubles >= kFields*64, "the fields at the points fit Q");
__host__ __device__ constexpr int PDoubles(int nen) { return nen*64 > 7*4*64 ? nen*64 : 7*4*64; }

__global__ void __launch_bounds__(kThreads) NsResidualKernel(ResidualArgs args, int max_nen)
{
	extern __shared__ double lds[];
	double* P = lds;
	double* Q = P + PDoubles(max_nen);
	double* nodal = Q + kQDoubles;       // [nen][u, u_prev, v, v_prev, w, w_prev, p, 0]
	double* tab = nodal + 8*max_nen;     // [B, B', B''][Gauss point][Bernstein index]
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const int e = args.elements ? args.elements[blockIdx.x] : blockIdx.x;
	const int b0 = args.eoff[e];
	const int nen = args.eoff[e + 1] - b0;
	for (int i = tid; i < nen*64; i += kThreads) P[i] = 0.0;
	for (int i = tid; i < nen*4; i += kThreads) {
		const int a = i >> 2, f = i & 3;
		const size_t at = 4*(size_t)args.conn[b0 + a] + f;
		nodal[8*a + 2*f] = args.state[at];
		nodal[8*a + 2*f + 1] = f < 3 ? args.previous[at] : 0.0;
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
	for (int t = tid; t < nen*8; t += kThreads) {  // eight lanes per extraction row
		const int a = t >> 3, end = args.xoff[b0 + a + 1];
		for (int k = args.xoff[b0 + a] + (t & 7); k < end; k += 8) P[64*a + args.xcol[k]] = args.xval[k];
	}
	__syncthreads();
	// Bernstein coefficients of the wave's field (and its previous value)
	{
		double v = 0.0, old = 0.0;
		for (int a = 0; a < nen; ++a) {
			const double c = P[64*a + lane];
			const double2 n = *reinterpret_cast<const double2*>(nodal + 8*a + 2*wave);
			v += c*n.x;
			old += c*n.y;
		}
		Q[(2*wave)*64 + lane] = v;
		Q[(2*wave + 1)*64 + lane] = old;
	}
	__syncthreads();
	const int x = lane & 3, y = (lane >> 2) & 3, z = lane >> 4;
	// xi: lane (point x, j = y, k = z)
	{
		const double* u = Q + (2*wave)*64 + (lane & ~3);
		double b = 0.0, d = 0.0, h = 0.0, old = 0.0;
#pragma unroll
		for (int i = 0; i < 4; ++i) {
			b += tab[4*x + i]*u[i];
			d += tab[16 + 4*x + i]*u[i];
			h += tab[32 + 4*x + i]*u[i];
			old += tab[4*x + i]*u[64 + i];
		}
		double* o = Q + 8*64 + (4*wave)*64 + lane;
		o[0] = b;
		o[64] = d;
		o[128] = h;
		o[192] = old;
	}
	__syncthreads();
	// eta: lane (points x, y, k = z)
	{
		const double* s = Q + 8*64 + (4*wave)*64 + x + 16*z;
		double bb = 0.0, bd = 0.0, bh = 0.0, db = 0.0, dd = 0.0, hb = 0.0, old = 0.0;
#pragma unroll
		for (int j = 0; j < 4; ++j) {
			const double B = tab[4*y + j], D = tab[16 + 4*y + j], H = tab[32 + 4*y + j];
			const double b = s[4*j], d = s[64 + 4*j], h = s[128 + 4*j];
			bb += B*b;
			bd += D*b;
			bh += H*b;
			db += B*d;
			dd += D*d;
			hb += B*h;
			old += B*s[192 + 4*j];
		}
		double* o = P + (7*wave)*64 + lane;
		o[0] = bb;
		o[64] = bd;
		o[128] = bh;
		o[192] = db;
		o[256] = dd;
		o[320] = hb;
		o[384] = old;
	}
	__syncthreads();
	// zeta and the pull-back: lane = Gauss point
	const double* gq = args.geometry + (size_t)e*kGeomFields*kQ + lane;
	{
		const double* s = P + (7*wave)*64 + x + 4*y;
		double v = 0.0, g0 = 0.0, g1 = 0.0, g2 = 0.0, old = 0.0;
		double h00 = 0.0, h11 = 0.0, h22 = 0.0, h01 = 0.0, h02 = 0.0, h12 = 0.0;
#pragma unroll
		for (int k = 0; k < 4; ++k) {
			const double B = tab[4*z + k], D = tab[16 + 4*z + k], H = tab[32 + 4*z + k];
			const double bb = s[16*k], bd = s[64 + 16*k], db = s[192 + 16*k];
			v += B*bb;
			g0 += B*db;
			g1 += B*bd;
			g2 += D*bb;
			h00 += B*s[320 + 16*k];
			h11 += B*s[128 + 16*k];
			h22 += H*bb;
			h01 += B*s[256 + 16*k];
			h02 += D*db;
			h12 += D*bd;
			old += B*s[384 + 16*k];
		}
		double inv[3][3];
#pragma unroll
		for (int i = 0; i < 9; ++i) inv[i/3][i%3] = gq[(1 + i)*kQ];
		Q[wave*64 + lane] = v;
#pragma unroll
		for (int d = 0; d < 3; ++d) Q[(4 + 3*wave + d)*64 + lane] = g0*inv[0][d] + g1*inv[1][d] + g2*inv[2][d];
		if (wave < 3) {
			double m[3][3];
#pragma unroll
			for (int c = 0; c < 3; ++c)
#pragma unroll
				for (int d = c; d < 3; ++d) m[c][d] = inv[c][0]*inv[d][0] + inv[c][1]*inv[d][1] + inv[c][2]*inv[d][2];
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
		double inv[3][3];
#pragma unroll
		for (int i = 0; i < 9; ++i) inv[i/3][i%3] = gq[(1 + i)*kQ];
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
		const double* s = P + (4*wave)*64 + x + 4*y;
		double a1 = 0.0, a2 = 0.0, a3 = 0.0;
#pragma unroll
		for (int k = 0; k < 4; ++k) {
			const double B = tab[4*k + z], D = tab[16 + 4*k + z];
			a1 += B*s[16*k] + D*s[192 + 16*k];
			a2 += B*s[64 + 16*k];
			a3 += B*s[128 + 16*k];
		}
		double* o = Q + (3*wave)*64 + lane;
		o[0] = a1;
		o[64] = a2;
		o[128] = a3;
	}
	__syncthreads();
	{
		const double* s = Q + (3*wave)*64 + x + 16*z;
		double b1 = 0.0, b2 = 0.0;
#pragma unroll
		for (int j = 0; j < 4; ++j) {
			const double B = tab[4*j + y], D = tab[16 + 4*j + y];
			b1 += B*s[4*j] + D*s[128 + 4*j];
			b2 += B*s[64 + 4*j];
		}
		double* o = P + (2*wave)*64 + lane;
		o[0] = b1;
		o[64] = b2;
	}
	__syncthreads();
	{
		const double* s = P + (2*wave)*64 + (lane & ~3);
		double r = 0.0;
#pragma unroll
		for (int i = 0; i < 4; ++i) r += tab[4*i + x]*s[i] + tab[16 + 4*i + x]*s[64 + i];
		Q[4*lane + wave] = r;
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
	ResidualArgs a{m->eoff.data(), m->conn.data(), m->xoff.data(), m->xcol.data(), m->xval.data(), m->geometry.data(),
		state, previous, p.density, p.viscosity, p.dt, m->element_rows.data(), elements, points};
	const int nen = m->max_nen;
	const size_t lds = sizeof(double)*(PDoubles(nen) + kQDoubles + 8*(size_t)nen + 48);
	static_assert(sizeof(double)*(PDoubles(kMaxBasis) + kQDoubles + 8*kMaxBasis + 48) <= 65536,
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
