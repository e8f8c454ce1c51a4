// Per-cell work of the RK4 adjoint (bm_adjoint.hip), shared by its plain kernels and the row kernels
// that run it between the convolution's x passes (bm_adjrow.hip).
#pragma once

#include "bm_internal.h"
#include "bm_stage.h"

namespace bm {

// layer stacks in the adjoint: per-layer values passed in the kernel arguments (8 layers)
constexpr int kMaxAdjLayers = 8;

struct AdjArgs {
	int nx, ny, nz;
	float ihx2, ihy2, ihz2;
	float A, alpha, grel;
	float K1, K2, ea[3];    // uniaxial anisotropy
	float Hz[3];            // applied field at the step's start time
	float dir[3], sc;       // pulse direction and sinc value at that time (d H / d amp = sc dir)
	float tz;               // ramp: d H / d slope_c = tz e_c (the step's start time), else 0
	int modules;
	const float* Ms;
	int layered;            // layer stack: per-layer A, alpha, K1, no exchange across layers
	int per;                // periodic exchange along x, y, z: bits 0, 1, 2
	float lay_A[kMaxAdjLayers], lay_alpha[kMaxAdjLayers], lay_K1[kMaxAdjLayers];
};

__device__ __forceinline__ CellMat adj_mat(const AdjArgs& a, int k)
{
	if (!a.layered) return CellMat{ a.A, a.alpha, a.K1 };
	CellMat c{ a.lay_A[0], a.lay_alpha[0], a.lay_K1[0] };
#pragma unroll
	for (int l = 1; l < kMaxAdjLayers; l++)
		if (k == l) c = CellMat{ a.lay_A[l], a.lay_alpha[l], a.lay_K1[l] };
	return c;
}

__device__ __forceinline__ F3 lap_at(const float* X, const AdjArgs& a, size_t idx, int i, int j, int k)
{
	const F3 m = ld3(X, idx);
	F3 lx{ 0, 0, 0 }, ly{ 0, 0, 0 }, lz{ 0, 0, 0 };
	const size_t sy = a.nx, sz = (size_t)a.nx * a.ny;
	// periodic axes at the mesh ends: the wrapped neighbour (BorisLib/VEC_VC_Del.h:24-45)
	if (a.nx > 1) {
		if (i > 0 && i < a.nx - 1) lx = ld3(X, idx + 1) + ld3(X, idx - 1) - 2.f * m;
		else if (a.per & 1) lx = (i == 0) ? ld3(X, idx + 1) + ld3(X, idx + (a.nx - 1)) - 2.f * m
		                                  : ld3(X, idx - (a.nx - 1)) + ld3(X, idx - 1) - 2.f * m;
		else if (i == 0) lx = ld3(X, idx + 1) - m;
		else lx = ld3(X, idx - 1) - m;
	}
	if (a.ny > 1) {
		if (j > 0 && j < a.ny - 1) ly = ld3(X, idx + sy) + ld3(X, idx - sy) - 2.f * m;
		else if (a.per & 2) ly = (j == 0) ? ld3(X, idx + sy) + ld3(X, idx + (a.ny - 1) * sy) - 2.f * m
		                                  : ld3(X, idx - (a.ny - 1) * sy) + ld3(X, idx - sy) - 2.f * m;
		else if (j == 0) ly = ld3(X, idx + sy) - m;
		else ly = ld3(X, idx - sy) - m;
	}
	if (a.nz > 1 && !a.layered) {
		if (k > 0 && k < a.nz - 1) lz = ld3(X, idx + sz) + ld3(X, idx - sz) - 2.f * m;
		else if (a.per & 4) lz = (k == 0) ? ld3(X, idx + sz) + ld3(X, idx + (a.nz - 1) * sz) - 2.f * m
		                                  : ld3(X, idx - (a.nz - 1) * sz) + ld3(X, idx - sz) - 2.f * m;
		else if (k == 0) lz = ld3(X, idx + sz) - m;
		else lz = ld3(X, idx - sz) - m;
	}
	return a.ihx2 * lx + a.ihy2 * ly + a.ihz2 * lz;
}

__device__ __forceinline__ float cex(float A, float Ms) { return (2.f * A) / ((float)kMU0 * Ms * Ms); }
__device__ __forceinline__ float pre_llg(const AdjArgs& a, float alpha) { return (float)(-kGAMMA) * a.grel / (1.f + alpha * alpha); }

// field at X: Zeeman + demag (Hd) + exchange + anisotropy; also returns the unscaled Laplacian
__device__ __forceinline__ F3 field_at(const AdjArgs& a, const CellMat& cm, const float* X, F3 Hd, size_t idx,
	int i, int j, int k, float Ms, F3& lap)
{
	F3 H = (a.modules & BM_MOD_ZEEMAN) ? F3{ a.Hz[0], a.Hz[1], a.Hz[2] } : F3{ 0.f, 0.f, 0.f };
	if (a.modules & BM_MOD_DEMAG) H = H + Hd;
	lap = F3{ 0.f, 0.f, 0.f };
	if (a.modules & BM_MOD_EXCHANGE) { lap = lap_at(X, a, idx, i, j, k); H = H + cex(cm.A, Ms) * lap; }
	if (a.modules & BM_MOD_ANIS_UNI) {
		const F3 e{ a.ea[0], a.ea[1], a.ea[2] };
		const float d = dot(ld3(X, idx), e) / Ms;
		H = H + ((2.f / ((float)kMU0 * Ms)) * d * (cm.K1 + 2.f * a.K2 * (1.f - d * d))) * e;
	}
	return H;
}

__device__ __forceinline__ void cell_ijk(const AdjArgs& a, size_t idx, int& i, int& j, int& k)
{
	i = (int)(idx % a.nx); j = (int)((idx / a.nx) % a.ny); k = (int)(idx / ((size_t)a.nx * a.ny));
}

// planar field of a cell (n cells per component; null: none)
__device__ __forceinline__ F3 ld_planar(const float* p, size_t n, size_t idx) { return p ? F3{ p[idx], p[n + idx], p[2 * n + idx] } : F3{ 0.f, 0.f, 0.f }; }

// Forward stage S of the step from Mn in one cell: k = f(X); S < 3: acc (=, +=) w_S k, next = Mn + c_S dt
// k; S == 3: Y = Mn + dt/6 (acc + k), next = Ms Y / |Y|.  The caller stores (put), after all its cells
// are computed, so that their loads do not wait for one another's stores.
struct FwdCell { F3 acc, next, Y; };
template <int S>
__device__ __forceinline__ FwdCell fwd_cell(const AdjArgs& a, const float* X, F3 Hd, const float* Mn, const float* acc, float dt, size_t idx, int i, int j, int k)
{
	const float Ms = a.Ms[idx];
	const CellMat cm = adj_mat(a, k);
	F3 lap;
	const F3 m = ld3(X, idx);
	const F3 H = field_at(a, cm, X, Hd, idx, i, j, k, Ms, lap);
	const F3 mxh = cross(m, H);
	const float iMs = 1.f / Ms;
	const F3 mu{ m.x * iMs, m.y * iMs, m.z * iMs };
	const F3 f = pre_llg(a, cm.alpha) * (mxh + cm.alpha * cross(mu, mxh));
	FwdCell c{ f, f, f };
	if (S == 3) {
		c.Y = ld3(Mn, idx) + (dt / 6) * (ld3(acc, idx) + f);
		c.next = (Ms / norm(c.Y)) * c.Y;
	}
	else {
		if (S > 0) c.acc = ld3(acc, idx) + 2.f * f;
		c.next = ld3(Mn, idx) + (S == 2 ? dt : dt / 2) * f;
	}
	return c;
}
template <int S>
__device__ __forceinline__ void fwd_put(const FwdCell& c, float* acc, float* Xn, float* Yout, float* Mnext, size_t idx)
{
	if (S == 3) { if (Yout) st3(Yout, idx, c.Y); st3(Mnext, idx, c.next); }
	else { st3(acc, idx, c.acc); st3(Xn, idx, c.next); }
}

// Renormalisation adjoint in one cell: lamY = (Ms/|Y|)(lam - y (y.lam)), g += y.lam
__device__ __forceinline__ F3 renorm_cell(const float* Y, float Ms, F3 lam, double& g, size_t idx)
{
	const F3 y = ld3(Y, idx);
	const float nr = norm(y);
	const F3 yh = (1.f / nr) * y;
	const float yl = dot(yh, lam);
	g += (double)yl;
	return (Ms / nr) * (lam - yl * yh);
}

// Stage VJP, part 1, in one cell, from w = (dt/6) wS lamY + cS dt lxn: lx = direct term
// (anisotropy's local field Jacobian included), u (the field adjoint), cu = c u, gM += Ms terms, gz +=
// u . dir sc (amplitude) and u tz (slope).
struct VjpCell { F3 lx, u, cu; };
__device__ __forceinline__ VjpCell vjp_a_cell(const AdjArgs& a, const float* X, F3 Hd, F3 w, double& gM, double gz[4], size_t idx, int i, int j, int k)
{
	const float Ms = a.Ms[idx];
	const CellMat cm = adj_mat(a, k);
	const float pr = pre_llg(a, cm.alpha), al = cm.alpha;
	F3 lap;
	const F3 m = ld3(X, idx);
	const F3 H = field_at(a, cm, X, Hd, idx, i, j, k, Ms, lap);
	const float mh = dot(m, H), mw = dot(m, w), hw = dot(H, w), mm = dot(m, m);
	F3 d = pr * (cross(H, w) + (al / Ms) * (mh * w + mw * H - (2.f * hw) * m));
	const F3 uu = pr * (cross(w, m) + (al / Ms) * (mw * m - mm * w));
	const float ce = cex(cm.A, Ms);
	double g = -(double)pr * (double)al / ((double)Ms * Ms) * (double)dot(cross(m, cross(m, H)), w);
	if (a.modules & BM_MOD_EXCHANGE) g += (double)dot(uu, lap) * (-2.0 * (double)ce / (double)Ms);
	if (a.modules & BM_MOD_ANIS_UNI) {
		// H_an = 2/mu0 s (K1 + 2K2 - 2K2 s^2/Ms^2)/Ms^2 e with s = m.e: its Jacobian is
		// 2/(mu0 Ms^2) (K1 + 2K2 - 6K2 d^2) e e^T (d = s/Ms), its Ms derivative
		// 2/mu0 s e (-2K1 - 4K2 + 8K2 d^2)/Ms^3
		const F3 e{ a.ea[0], a.ea[1], a.ea[2] };
		const float sm = dot(m, e), dd = sm / Ms, ue = dot(uu, e);
		d = d + ((2.f / ((float)kMU0 * Ms * Ms)) * (cm.K1 + 2.f * a.K2 - 6.f * a.K2 * dd * dd) * ue) * e;
		g += 2.0 / kMU0 * (double)sm * (double)ue * (-2.0 * cm.K1 - 4.0 * a.K2 + 8.0 * a.K2 * (double)dd * dd) / ((double)Ms * Ms * Ms);
	}
	gM += g;
	gz[0] += (double)(dot(uu, F3{ a.dir[0], a.dir[1], a.dir[2] }) * a.sc);
	gz[1] += (double)(uu.x * a.tz); gz[2] += (double)(uu.y * a.tz); gz[3] += (double)(uu.z * a.tz);
	return VjpCell{ d, uu, ce * uu };
}

// Stage VJP, part 2, in one cell: lx + N u (Nu) + Lap(c u)
__device__ __forceinline__ F3 vjp_b_cell(const AdjArgs& a, F3 Nu, const float* cu, F3 lx, size_t idx, int i, int j, int k)
{
	F3 v = lx;
	if (a.modules & BM_MOD_DEMAG) v = v + Nu;
	if (a.modules & BM_MOD_EXCHANGE) v = v + lap_at(cu, a, idx, i, j, k);
	return v;
}

// Row kernels (bm_adjrow.hip): the cells' work between the x inverse of one convolution and the x
// forward of the next, in place on the x-side spectra Sx of nz planes of ny rows of nx cells.
struct AdjRow { float2* Sx; int ntl; float scale; };
struct AdjFwd { const float* X; const float* Mn; float* acc; float* Xn; float* Yout; float* Mnext; float* Hd_out; float dt; };
// B: v = vjp_b of the last stage (lx, cu_in), lacc += v.  RN: renormalisation adjoint of lam (B: of lacc +
// v) with Y into lamY and lacc.  A: vjp_a of the next stage at X, Hd into lx, cu_out, gMs, apart (4 per
// work item) and the x forward of its u.  Without A: lacc + v into lam.
struct AdjBwd {
	const float* Y; const float* X; const float* Hd;
	float* lam; float* lamY; float* lacc; float* lx; const float* cu_in; float* cu_out;
	double* gMs; double* apart;
	float wS, cS, dt;
};
int adj_row_fwd(int stage, const AdjArgs& a, const AdjRow& r, const AdjFwd& f, hipStream_t st);
int adj_row_bwd(bool b, bool rn, bool ad, const AdjArgs& a, const AdjRow& r, const AdjBwd& w, hipStream_t st);

} // namespace bm
