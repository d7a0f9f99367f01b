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

// Per-point record from the field sums s (u, p, grad u, grad p, lap u, u_prev
// at the point; 22 values) and the point's geometry record gq (fields 0..9:
// measure and J^-1, field stride kGs): r[0] measure, r[1..2] tau_M, tau_C, r[3..5] u, r[6..8] rho (du/dt +
// w.grad u), r[9..17] stress rows, r[18] div u, r[19..21] u', r[22..24] w =
// u + u', r[25..33] grad u and, with exact_tangent, r[34..54] the
// linearisation of u' (K, R, c1) the consistent tangent needs.
template <int kGs>
__device__ inline void PointRecord(const double* __restrict__ s, const double* __restrict__ gq, double rho, double mu,
	double nu, double dt, bool exact_tangent, double* __restrict__ r)
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
	if (exact_tangent) {
		// d(u')/d(u_f) = N_b K[.][f] - delta tau_M s_b with
		// K_cf = tau_M^3 strong_c (G u)_f - tau_M du_c/dx_f, and
		// R = grad u + grad u K, c1_f = rho tau_C tau_M^2 div (G u)_f.
		double Gu[3];
		for (int i = 0; i < 3; ++i) Gu[i] = G[i][0]*u[0] + G[i][1]*u[1] + G[i][2]*u[2];
		const double tm3 = tau_m*tau_m*tau_m;
		double K[3][3];
		for (int c = 0; c < 3; ++c) {
			const double strong = -fu[c]/tau_m;
			for (int f = 0; f < 3; ++f) K[c][f] = tm3*strong*Gu[f] - tau_m*grad[c][f];
		}
		for (int c = 0; c < 3; ++c)
			for (int f = 0; f < 3; ++f) {
				r[34 + 3*c + f] = K[c][f];
				r[43 + 3*c + f] = grad[c][f] + grad[c][0]*K[0][f] + grad[c][1]*K[1][f] + grad[c][2]*K[2][f];
			}
		for (int f = 0; f < 3; ++f) r[52 + f] = rho*tau_c*tau_m*tau_m*div*Gu[f];
	}
}

}  // namespace

}  // namespace tfi
