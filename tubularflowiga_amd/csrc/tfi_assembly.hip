// Basis table, Dirichlet rows and boundary-face integrals of the Navier-Stokes
// assembly (the element residual and tangent are in tfi_residual.hip and
// tfi_tangent.hip).  Basis values, gradients and Laplacians are evaluated per
// (basis, point) by sum factorisation of the cubic Bernstein tensor product
// (328 FMA instead of 640 per point, no table reads).
#include "tfi_internal.hpp"
#include "tfi_point.hpp"

#include <algorithm>
#include <cmath>

namespace tfi {

namespace {


__global__ void DirichletMatrixKernel(int nodes, const int* __restrict__ ro, const int* __restrict__ diag,
	const int* __restrict__ vmask, const int* __restrict__ pmask, double* __restrict__ jac)
{
	const int node = blockIdx.x*blockDim.x + threadIdx.x;
	if (node >= nodes) return;
	const bool v = vmask[node] != 0, p = pmask[node] != 0;
	if (!v && !p) return;
	for (int k = ro[node]; k < ro[node + 1]; ++k) {
		double* J = jac + (size_t)k*16;
		for (int f = 0; f < 4; ++f) {
			if (!(f < 3 ? v : p)) continue;
			for (int c = 0; c < 4; ++c) J[4*f + c] = 0.0;
		}
	}
	double* D = jac + (size_t)diag[node]*16;
	for (int f = 0; f < 4; ++f)
		if (f < 3 ? v : p) D[5*f] = 1.0;
}

__global__ void DirichletRhsKernel(int nodes, const int* __restrict__ vmask, const int* __restrict__ pmask,
	const double* __restrict__ vt, const double* __restrict__ pt, const double* __restrict__ state,
	double* __restrict__ rhs)
{
	const int node = blockIdx.x*blockDim.x + threadIdx.x;
	if (node >= nodes) return;
	if (vmask[node])
		for (int c = 0; c < 3; ++c) rhs[4*(size_t)node + c] = vt[3*(size_t)node + c] - state[4*(size_t)node + c];
	if (pmask[node]) rhs[4*(size_t)node + 3] = pt[node] - state[4*(size_t)node + 3];
}

__global__ void DirichletStateKernel(int nodes, const int* __restrict__ vmask, const int* __restrict__ pmask,
	const double* __restrict__ vt, const double* __restrict__ pt, double* __restrict__ state)
{
	const int node = blockIdx.x*blockDim.x + threadIdx.x;
	if (node >= nodes) return;
	if (vmask[node])
		for (int c = 0; c < 3; ++c) state[4*(size_t)node + c] = vt[3*(size_t)node + c];
	if (pmask[node]) state[4*(size_t)node + 3] = pt[node];
}

// Volumetric flow through labelled faces (IntegrateBoundaryFlow,
// solvers/cpu/include/BoundaryFlow.hpp:164-200).  The flow is linear in the
// state, so it is taken from the face's area-weighted basis vectors
// int_face N_a n dA (integrated once, with the same 4x4 Gauss rule, by
// FaceTractionKernel at unit pressure): one 64-lane block per face,
// fixed-order wave sum.
__global__ void FaceFlowVecKernel(int count, const int* __restrict__ felem, const int* __restrict__ eoff,
	const int* __restrict__ conn, const double* __restrict__ vec, const double* __restrict__ state,
	double* __restrict__ flows)
{
	const int f = blockIdx.x;
	if (f >= count) return;
	const int e = felem[f], b0 = eoff[e], nen = eoff[e + 1] - b0;
	double s = 0.0;
	for (int a = threadIdx.x; a < nen; a += 64) {
		const double* v = vec + ((size_t)f*kMaxBasis + a)*3;
		const size_t node = conn[b0 + a];
		s += state[4*node]*v[0] + state[4*node + 1]*v[1] + state[4*node + 2]*v[2];
	}
	for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
	if (threadIdx.x == 0) flows[f] = -s;
}

// Pressure-traction load of one labelled face (IntegrateBoundaryPressureTraction,
// BoundaryFlow.hpp:445-477): local[a][c] = -p sum_pt s w_i w_j / 4 * cof_c(pt) N_a(pt),
// with cof = det J * (row `fixed axis` of J^-1) the face's area vector.  One
// 64-lane block per face; the per-face vectors are summed on the host in face
// order, so the load is deterministic and ordered like the reference's.
__global__ void FaceTractionKernel(int count, const int* __restrict__ felem, const int* __restrict__ fface,
	const double* __restrict__ pressure, const int* __restrict__ eoff, const int* __restrict__ xoff,
	const uint8_t* __restrict__ xcol, const double* __restrict__ xval, const double* __restrict__ bezier,
	double* __restrict__ local)
{
	const int f = blockIdx.x;
	if (f >= count) return;
	__shared__ double bern[16][64];
	__shared__ double wcof[16][3];
	const int e = felem[f], face = fface[f];
	const int fixed_axis[6] = {2, 1, 0, 1, 0, 2};
	const int var0[6] = {0, 0, 1, 0, 1, 0}, var1[6] = {1, 2, 2, 2, 2, 1};
	const double fixed_value[6] = {0.0, 0.0, 1.0, 1.0, 0.0, 1.0};
	const double sign[6] = {-1.0, -1.0, 1.0, 1.0, -1.0, 1.0};
	const double gw[4] = {0.3478548451374539, 0.6521451548625461, 0.6521451548625461, 0.3478548451374539};
	const int lane = threadIdx.x;  // 64 threads
	for (int idx = lane; idx < 16*64; idx += 64) {
		const int pt = idx >> 6, p = idx & 63;
		const int qi = pt >> 2, qj = pt & 3;
		double c[3];
		c[fixed_axis[face]] = fixed_value[face];
		c[var0[face]] = kGp[qi];
		c[var1[face]] = kGp[qj];
		double b[3][4], db[3][4], d2b[3][4];
		for (int d = 0; d < 3; ++d) Bern3(c[d], b[d], db[d], d2b[d]);
		bern[pt][p] = b[0][p & 3]*b[1][(p >> 2) & 3]*b[2][p >> 4];
	}
	if (lane < 16) {
		const int pt = lane, qi = pt >> 2, qj = pt & 3;
		double c[3];
		c[fixed_axis[face]] = fixed_value[face];
		c[var0[face]] = kGp[qi];
		c[var1[face]] = kGp[qj];
		double b[3][4], db[3][4], d2b[3][4];
		for (int d = 0; d < 3; ++d) Bern3(c[d], b[d], db[d], d2b[d]);
		const double* X = bezier + (size_t)e*192;
		double J[3][3] = {};
		for (int k = 0; k < 4; ++k)
			for (int j = 0; j < 4; ++j)
				for (int i = 0; i < 4; ++i) {
					const int p = i + 4*j + 16*k;
					const double g[3] = {db[0][i]*b[1][j]*b[2][k], b[0][i]*db[1][j]*b[2][k], b[0][i]*b[1][j]*db[2][k]};
					for (int x = 0; x < 3; ++x)
						for (int d = 0; d < 3; ++d) J[x][d] += X[3*p + x]*g[d];
				}
		const int a = fixed_axis[face];
		const int a1 = (a + 1)%3, a2 = (a + 2)%3;
		const double w = sign[face]*gw[qi]*gw[qj]*0.25;
		for (int x = 0; x < 3; ++x) {
			const int x1 = (x + 1)%3, x2 = (x + 2)%3;
			wcof[pt][x] = w*(J[x1][a1]*J[x2][a2] - J[x1][a2]*J[x2][a1]);
		}
	}
	__syncthreads();
	const int b0 = eoff[e], nen = eoff[e + 1] - b0;
	const double pf = pressure[f];
	for (int aa = lane; aa < nen; aa += 64) {
		double acc[3] = {0.0, 0.0, 0.0};
		for (int pt = 0; pt < 16; ++pt) {
			double N = 0.0;
			for (int k = xoff[b0 + aa]; k < xoff[b0 + aa + 1]; ++k) N += xval[k]*bern[pt][xcol[k]];
			for (int c = 0; c < 3; ++c) acc[c] += N*wcof[pt][c];
		}
		double* out = local + ((size_t)f*kMaxBasis + aa)*3;
		for (int c = 0; c < 3; ++c) out[c] = -pf*acc[c];
	}
}

// Face mass of one labelled face for the scalar flux / Robin terms
// (AssembleGenericSurfaceKernel, solvers/cuda/include/GenericTransportKernels.cuh:146-215):
// with m = w_i w_j / 4 |t_0 x t_1| at the 4x4 Gauss points of the face,
// mass[f][a][b] = sum_pt N_a N_b m and load[f][a] = sum_pt N_a m.  |t_0 x t_1|
// is the length of the cofactor vector FaceTractionKernel integrates.  One
// 64-lane block per face; `stride` (>= the element's basis count) in both outputs.
__global__ void FaceMassKernel(int count, int stride, const int* __restrict__ felem, const int* __restrict__ fface,
	const int* __restrict__ eoff, const int* __restrict__ xoff, const uint8_t* __restrict__ xcol,
	const double* __restrict__ xval, const double* __restrict__ bezier, double* __restrict__ mass,
	double* __restrict__ load)
{
	const int f = blockIdx.x;
	if (f >= count) return;
	__shared__ double bern[16][64];
	__shared__ double measure[16];
	__shared__ double basis[16][kMaxBasis];
	const int e = felem[f], face = fface[f];
	const int fixed_axis[6] = {2, 1, 0, 1, 0, 2};
	const int var0[6] = {0, 0, 1, 0, 1, 0}, var1[6] = {1, 2, 2, 2, 2, 1};
	const double fixed_value[6] = {0.0, 0.0, 1.0, 1.0, 0.0, 1.0};
	const double gw[4] = {0.3478548451374539, 0.6521451548625461, 0.6521451548625461, 0.3478548451374539};
	const int lane = threadIdx.x;  // 64 threads
	for (int idx = lane; idx < 16*64; idx += 64) {
		const int pt = idx >> 6, p = idx & 63;
		double c[3];
		c[fixed_axis[face]] = fixed_value[face];
		c[var0[face]] = kGp[pt >> 2];
		c[var1[face]] = kGp[pt & 3];
		double b[3][4], db[3][4], d2b[3][4];
		for (int d = 0; d < 3; ++d) Bern3(c[d], b[d], db[d], d2b[d]);
		bern[pt][p] = b[0][p & 3]*b[1][(p >> 2) & 3]*b[2][p >> 4];
	}
	if (lane < 16) {
		const int pt = lane, qi = pt >> 2, qj = pt & 3;
		double c[3];
		c[fixed_axis[face]] = fixed_value[face];
		c[var0[face]] = kGp[qi];
		c[var1[face]] = kGp[qj];
		double b[3][4], db[3][4], d2b[3][4];
		for (int d = 0; d < 3; ++d) Bern3(c[d], b[d], db[d], d2b[d]);
		const double* X = bezier + (size_t)e*192;
		double t0[3] = {}, t1[3] = {};
		for (int k = 0; k < 4; ++k)
			for (int j = 0; j < 4; ++j)
				for (int i = 0; i < 4; ++i) {
					const int p = i + 4*j + 16*k;
					const double g[3] = {db[0][i]*b[1][j]*b[2][k], b[0][i]*db[1][j]*b[2][k], b[0][i]*b[1][j]*db[2][k]};
					for (int x = 0; x < 3; ++x) {
						t0[x] += X[3*p + x]*g[var0[face]];
						t1[x] += X[3*p + x]*g[var1[face]];
					}
				}
		const double n[3] = {t0[1]*t1[2] - t0[2]*t1[1], t0[2]*t1[0] - t0[0]*t1[2], t0[0]*t1[1] - t0[1]*t1[0]};
		measure[pt] = gw[qi]*gw[qj]*0.25*sqrt(n[0]*n[0] + n[1]*n[1] + n[2]*n[2]);
	}
	__syncthreads();
	const int b0 = eoff[e], nen = eoff[e + 1] - b0;
	for (int idx = lane; idx < 16*nen; idx += 64) {
		const int pt = idx/nen, a = idx - pt*nen;
		double N = 0.0;
		for (int k = xoff[b0 + a]; k < xoff[b0 + a + 1]; ++k) N += xval[k]*bern[pt][xcol[k]];
		basis[pt][a] = N;
	}
	__syncthreads();
	double* mf = mass + (size_t)f*stride*stride;
	for (int pair = lane; pair < nen*nen; pair += 64) {
		const int a = pair/nen, b = pair - a*nen;
		double s = 0.0;
		for (int pt = 0; pt < 16; ++pt) s += basis[pt][a]*basis[pt][b]*measure[pt];
		mf[a*stride + b] = s;
	}
	for (int a = lane; a < nen; a += 64) {
		double s = 0.0;
		for (int pt = 0; pt < 16; ++pt) s += basis[pt][a]*measure[pt];
		load[(size_t)f*stride + a] = s;
	}
}

// Basis records of every (point, function) of one element per workgroup, in
// the table layout [q][a][kTableRec] the assembly reads slab by slab.
__global__ void __launch_bounds__(256) BasisTableKernel(const int* __restrict__ eoff, const int* __restrict__ xoff,
	const uint8_t* __restrict__ xcol, const double* __restrict__ xval, const double* __restrict__ geometry,
	double* __restrict__ table)
{
	extern __shared__ double C[];  // [nen][64] extraction rows
	const int e = blockIdx.x;
	const int b0 = eoff[e], nen = eoff[e + 1] - b0;
	for (int i = threadIdx.x; i < nen*64; i += blockDim.x) C[i] = 0.0;
	__syncthreads();
	for (int a = threadIdx.x; a < nen; a += blockDim.x)
		for (int k = xoff[b0 + a]; k < xoff[b0 + a + 1]; ++k) C[64*a + xcol[k]] = xval[k];
	__syncthreads();
	const double* geo = geometry + (size_t)e*kGeomFields*kQ;
	double* dst = table + (size_t)b0*kQ*kTableRec;
	for (int it = threadIdx.x; it < kQ*nen; it += blockDim.x) {
		const int q = it/nen, a = it - q*nen;
		double rec[kTableRec];
		EvalBasis(C + 64*a, geo + q, q, rec);
#pragma unroll
		for (int f = 0; f < kTableRec; ++f) dst[(size_t)it*kTableRec + f] = rec[f];
	}
}

}  // namespace

void SetBasisTable(tfi_mesh* m, int enable)
{
	tfi_ctx* ctx = m->ctx;
	const size_t count = (size_t)m->basis_entries*kQ*kTableRec;
	if (enable < 0) {
		size_t free_bytes = 0, total_bytes = 0;
		Check(hipMemGetInfo(&free_bytes, &total_bytes), "hipMemGetInfo");
		enable = count*sizeof(double) <= free_bytes/2 ? 1 : 0;
	}
	if (!enable) {
		Sync(ctx);
		m->basis_table.Release();
		return;
	}
	if (m->basis_table.size() == count) return;
	m->basis_table.Allocate(ctx, count);
	const ExtractionRows rows = m->rows();
	hipLaunchKernelGGL(BasisTableKernel, dim3(m->elements), dim3(256), sizeof(double)*64*m->max_nen, ctx->stream,
		m->eoff.data(), rows.offsets, rows.columns, rows.values, m->geometry.data(), m->basis_table.data());
	TFI_LAUNCH_CHECK("BasisTableKernel");
	Sync(ctx);
}

// Counted arithmetic of the assembly per element with nen basis functions
// and Q = 64 points: sum-factorised basis and push-forward (656 + 42 flops per
// (a, q), none when the basis table supplies them or no tangent asks for them), field interpolation (44),
// u.grad N and residual row (38), per-point scalars (~300 per q) and the
// tangent (72 flops per (a, b, q) for the legacy tangent; 132 per (a, b, q)
// plus ~100 per (a, q) for the exact one).
double AssemblyFlops(const tfi_mesh* m, bool with_jacobian, bool exact)
{
	const double basis = m->basis_table.size() || !with_jacobian ? 0.0 : 656.0 + 42.0;
	double total = 0.0;
	for (int e = 0; e < m->elements; ++e) {
		const double nen = m->h_eoff[e + 1] - m->h_eoff[e];
		double pair = 0.0;
		if (with_jacobian) pair = exact ? 132.0*nen*nen + 100.0*nen : 72.0*nen*nen;
		total += kQ*(nen*(basis + 44.0 + 38.0) + 300.0 + pair);
	}
	return total;
}

void ApplyDirichlet(tfi_mesh* m, const int* vmask, const int* pmask, const double* vtarget, const double* ptarget,
	const double* state, double* jacobian, double* rhs)
{
	tfi_ctx* ctx = m->ctx;
	const int blocks = (m->nodes + 255)/256;
	if (jacobian) {
		hipLaunchKernelGGL(DirichletMatrixKernel, dim3(blocks), dim3(256), 0, ctx->stream, m->nodes,
			m->row_offsets.data(), m->diagonal.data(), vmask, pmask, jacobian);
		TFI_LAUNCH_CHECK("DirichletMatrixKernel");
	}
	if (rhs) {
		hipLaunchKernelGGL(DirichletRhsKernel, dim3(blocks), dim3(256), 0, ctx->stream, m->nodes, vmask, pmask,
			vtarget, ptarget, state, rhs);
		TFI_LAUNCH_CHECK("DirichletRhsKernel");
	}
}

void SetDirichletState(tfi_mesh* m, const int* vmask, const int* pmask, const double* vtarget,
	const double* ptarget, double* state)
{
	hipLaunchKernelGGL(DirichletStateKernel, dim3((m->nodes + 255)/256), dim3(256), 0, m->ctx->stream, m->nodes, vmask,
		pmask, vtarget, ptarget, state);
	TFI_LAUNCH_CHECK("DirichletStateKernel");
}

void FaceFlowsFromVectors(tfi_mesh* m, int count, const int* element, const double* vec, const double* state,
	double* flows)
{
	if (count <= 0) return;
	hipLaunchKernelGGL(FaceFlowVecKernel, dim3(count), dim3(64), 0, m->ctx->stream, count, element, m->eoff.data(),
		m->conn.data(), vec, state, flows);
	TFI_LAUNCH_CHECK("FaceFlowVecKernel");
}

void FaceMass(tfi_mesh* m, int count, const int* element, const int* face, double* mass, double* load)
{
	if (count <= 0) return;
	if (m->max_nen > kMaxBasis) throw Error("face integrals support at most 80 basis functions");
	hipLaunchKernelGGL(FaceMassKernel, dim3(count), dim3(64), 0, m->ctx->stream, count, m->max_nen, element, face,
		m->eoff.data(), m->xoff.data(), m->xcol.data(), m->xval.data(), m->bezier.data(), mass, load);
	TFI_LAUNCH_CHECK("FaceMassKernel");
}

void FaceTraction(tfi_mesh* m, int count, const int* element, const int* face, const double* pressure,
	double* local)
{
	if (count <= 0) return;
	hipLaunchKernelGGL(FaceTractionKernel, dim3(count), dim3(64), 0, m->ctx->stream, count, element, face, pressure,
		m->eoff.data(), m->xoff.data(), m->xcol.data(), m->xval.data(), m->bezier.data(), local);
	TFI_LAUNCH_CHECK("FaceTractionKernel");
}

}  // namespace tfi
