// Gauss points, cubic Bernstein polynomials and the per-point record of the
// stabilised Navier-Stokes element, shared by the assembly kernels.
#pragma once

#include "tfi_internal.hpp"

namespace tfi {

namespace {

__constant__ double kGp[4] = {0.06943184420297371, 0.33000947820757187, 0.6699905217924281, 0.9305681557970262};

__device__ inline void Bern3(double x, double b[4], double db[4], double d2b[4])
{
	const double y = 1.0 - x;
	b[0] = y*y*y; b[1] = 3.0*y*y*x; b[2] = 3.0*y*x*x; b[3] = x*x*x;
	db[0] = -3.0*y*y; db[1] = 3.0 - 12.0*x + 9.0*x*x; db[2] = 3.0*(2.0 - 3.0*x)*x; db[3] = 3.0*x*x;
	d2b[0] = 6.0*y; d2b[1] = -12.0 + 18.0*x; d2b[2] = 6.0 - 18.0*x; d2b[3] = 6.0*x;
}

constexpr int kTableRec = 5;  // N, dN/dx, dN/dy, dN/dz, lap N

// What the tangent needs of a point, written by the residual kernel as
// [item][kTangentRec][kQ]: measure, tau_M, tau_C, u, u', grad u, G u.
constexpr int kTangentRec = 21;

// Value, physical gradient and Laplacian of the basis function with Bezier
// extraction row c[64] at element point q (Bernstein sum-factorisation in
// xi, eta, zeta; gq = geometry record of the point, field stride kQ).
__device__ inline void EvalBasis(const double* __restrict__ c, const double* __restrict__ gq, int q,
	double out[kTableRec])
{
	double bx[4], dbx[4], d2bx[4], by[4], dby[4], d2by[4], bz[4], dbz[4], d2bz[4];
	Bern3(kGp[q & 3], bx, dbx, d2bx);
	Bern3(kGp[(q >> 2) & 3], by, dby, d2by);
	Bern3(kGp[q >> 4], bz, dbz, d2bz);
	double v = 0, g0 = 0, g1 = 0, g2 = 0, h00 = 0, h11 = 0, h22 = 0, h01 = 0, h02 = 0, h12 = 0;
	for (int k = 0; k < 4; ++k) {
		double s00 = 0, s10 = 0, s01 = 0, s20 = 0, s11 = 0, s02 = 0;
		for (int j = 0; j < 4; ++j) {
			const double* cr = c + 16*k + 4*j;
			const double x0 = cr[0]*bx[0] + cr[1]*bx[1] + cr[2]*bx[2] + cr[3]*bx[3];
			const double x1 = cr[0]*dbx[0] + cr[1]*dbx[1] + cr[2]*dbx[2] + cr[3]*dbx[3];
			const double x2 = cr[0]*d2bx[0] + cr[1]*d2bx[1] + cr[2]*d2bx[2] + cr[3]*d2bx[3];
			s00 += x0*by[j]; s10 += x1*by[j]; s20 += x2*by[j];
			s01 += x0*dby[j]; s11 += x1*dby[j]; s02 += x0*d2by[j];
		}
		v += s00*bz[k]; g0 += s10*bz[k]; g1 += s01*bz[k]; g2 += s00*dbz[k];
		h00 += s20*bz[k]; h11 += s02*bz[k]; h22 += s00*d2bz[k];
		h01 += s11*bz[k]; h02 += s10*dbz[k]; h12 += s01*dbz[k];
	}
	double inv[9];
#pragma unroll
	for (int i = 0; i < 9; ++i) inv[i] = gq[(1 + i)*kQ];
	out[0] = v;
	out[1] = g0*inv[0] + g1*inv[3] + g2*inv[6];
	out[2] = g0*inv[1] + g1*inv[4] + g2*inv[7];
	out[3] = g0*inv[2] + g1*inv[5] + g2*inv[8];
	out[4] = h00*gq[10*kQ] + h11*gq[11*kQ] + h22*gq[12*kQ]
		+ 2.0*(h01*gq[13*kQ] + h02*gq[14*kQ] + h12*gq[15*kQ])
		+ g0*gq[16*kQ] + g1*gq[17*kQ] + g2*gq[18*kQ];
}

// Per-point record from the field sums s (u, p, grad u, grad p, lap u, u_prev
// at the point; 22 values) and the point's geometry record gq (fields 0..9:
// measure and J^-1, field stride kGs): r[0] measure, r[1..2] tau_M, tau_C,
// r[3..5] u, r[6..8] rho (du/dt + w.grad u), r[9..17] stress rows, r[18] div u,
// r[19..21] u', r[22..24] w = u + u', r[25..33] grad u, r[34..36] G u with
// G = J^-T J^-1.
constexpr int kPointRecord = 37;

template <int kGs>
__device__ inline void PointRecord(const double* __restrict__ s, const double* __restrict__ gq, double rho, double mu,
	double nu, double dt, double* __restrict__ r)
{
	double inv[3][3];
	for (int a = 0; a < 3; ++a)
		for (int x = 0; x < 3; ++x) inv[a][x] = gq[(1 + 3*a + x)*kGs];
	const double u[3] = {s[0], s[1], s[2]};
	const double p = s[3];
	double grad[4][3];
	for (int f = 0; f < 4; ++f)
		for (int d = 0; d < 3; ++d) grad[f][d] = s[4 + 3*f + d];
	double dudt[3];
	for (int c = 0; c < 3; ++c) dudt[c] = dt > 0.0 ? (u[c] - s[19 + c])/dt : 0.0;
	double G[3][3] = {}, gv[3] = {};
	for (int i = 0; i < 3; ++i)
		for (int j = 0; j < 3; ++j) {
			for (int k = 0; k < 3; ++k) G[i][j] += inv[k][i]*inv[k][j];
			gv[i] += inv[j][i];
		}
	double GG = 0.0, gg = 0.0, uGu = 0.0;
	for (int i = 0; i < 3; ++i) {
		gg += gv[i]*gv[i];
		for (int j = 0; j < 3; ++j) {
			GG += G[i][j]*G[i][j];
			uGu += u[i]*G[i][j]*u[j];
		}
	}
	const double temporal = dt > 0.0 ? 4.0/(dt*dt) : 0.0;
	const double tau_m = 1.0/sqrt(temporal + uGu + (1.0/12.0)*nu*nu*GG);
	const double tau_c = 1.0/(tau_m*gg);
	double fu[3];
	for (int c = 0; c < 3; ++c) {
		const double conv = u[0]*grad[c][0] + u[1]*grad[c][1] + u[2]*grad[c][2];
		fu[c] = -tau_m*(dudt[c] + conv + grad[3][c]/rho - nu*s[16 + c]);
	}
	const double div = grad[0][0] + grad[1][1] + grad[2][2];
	const double fp = -rho*tau_c*div;
	r[0] = gq[0];
	r[1] = tau_m;
	r[2] = tau_c;
	for (int c = 0; c < 3; ++c) r[3 + c] = u[c];
	const double w[3] = {u[0] + fu[0], u[1] + fu[1], u[2] + fu[2]};
	for (int c = 0; c < 3; ++c) {
		r[6 + c] = rho*(dudt[c] + w[0]*grad[c][0] + w[1]*grad[c][1] + w[2]*grad[c][2]);
		for (int d = 0; d < 3; ++d)
			r[9 + 3*c + d] = mu*(grad[c][d] + grad[d][c]) - rho*fu[c]*w[d] - (c == d ? p + fp : 0.0);
	}
	r[18] = div;
	for (int c = 0; c < 3; ++c) r[19 + c] = fu[c];
	for (int c = 0; c < 3; ++c) r[22 + c] = w[c];
	for (int c = 0; c < 3; ++c)
		for (int d = 0; d < 3; ++d) r[25 + 3*c + d] = grad[c][d];
	for (int i = 0; i < 3; ++i) r[34 + i] = G[i][0]*u[0] + G[i][1]*u[1] + G[i][2]*u[2];
}

}  // namespace

}  // namespace tfi
