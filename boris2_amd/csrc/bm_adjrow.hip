// Row kernels of the RK4 adjoint: what lies between two convolutions' middle passes as one kernel per
// evaluation, in the form of bm_xsplit.h (few rows): x inverse of the field by component, the cells'
// work (bm_adjcell.h), x forward of the next convolution's input.
//
// The separate launches (x inverse, one or two cell kernels, x forward) cost a small mesh four to five
// launches of 4 to 7 us per evaluation; bound: latency.
#include "bm_adjcell.h"
#include "bm_xsplit.h"

namespace {

using namespace bm;

template <int HX, int S>
__global__ void __launch_bounds__((XSplit<HX, xs_groups<HX>()>::BS)) k_adj_fwd(AdjArgs a, AdjRow r, AdjFwd f)
{
	using X = XSplit<HX, xs_groups<HX>()>;
	__shared__ C2<float> tile[3 * X::RP * X::P];
	X x; x.init(tile);
	constexpr int EL = X::E / 2, NP = HX / 2;
	const int w = blockIdx.x, z = w % a.nz, y0 = (w / a.nz) * X::RP;
	const size_t n = (size_t)HX * a.ny * a.nz;
	x.load(r.Sx, z, y0, a.ny, a.nz, r.ntl);
	X::gsync();
	x.template c2r<EL>(r.scale);
	__syncthreads();
	for (int p = threadIdx.x; p < X::RP * NP; p += X::BS) {
		const int rl = p / NP, k = p % NP, y = y0 + rl;
		if (y >= a.ny) continue;
		C2<float>* t = tile + rl * X::P + k;
		C2<float>& tx = t[0]; C2<float>& ty = t[X::RP * X::P]; C2<float>& tz = t[2 * X::RP * X::P];
		const size_t idx = ((size_t)z * a.ny + y) * HX + 2 * k;
		const F3 h0{ tx.x, ty.x, tz.x }, h1{ tx.y, ty.y, tz.y };
		const FwdCell c0 = fwd_cell<S>(a, f.X, h0, f.Mn, f.acc, f.dt, idx, 2 * k, y, z);
		const FwdCell c1 = fwd_cell<S>(a, f.X, h1, f.Mn, f.acc, f.dt, idx + 1, 2 * k + 1, y, z);
		if (f.Hd_out) {
			f.Hd_out[idx] = h0.x; f.Hd_out[n + idx] = h0.y; f.Hd_out[2 * n + idx] = h0.z;
			f.Hd_out[idx + 1] = h1.x; f.Hd_out[n + idx + 1] = h1.y; f.Hd_out[2 * n + idx + 1] = h1.z;
		}
		fwd_put<S>(c0, f.acc, f.Xn, f.Yout, f.Mnext, idx);
		fwd_put<S>(c1, f.acc, f.Xn, f.Yout, f.Mnext, idx + 1);
		const F3 m0 = c0.next, m1 = c1.next;
		tx = mk(m0.x, m1.x); ty = mk(m0.y, m1.y); tz = mk(m0.z, m1.z);
	}
	__syncthreads();
	x.template r2c<EL>();
	X::gsync();
	x.store(r.Sx, z, y0, a.ny, a.nz, r.ntl);
}

template <int HX, bool B, bool RN, bool A>
__global__ void __launch_bounds__((XSplit<HX, xs_groups<HX>()>::BS)) k_adj_bwd(AdjArgs a, AdjRow r, AdjBwd b)
{
	using X = XSplit<HX, xs_groups<HX>()>;
	__shared__ C2<float> tile[3 * X::RP * X::P];
	__shared__ double red[A ? 4 * (X::BS / 64) : 1];
	X x; x.init(tile);
	constexpr int EL = X::E / 2, NP = HX / 2;
	const int w = blockIdx.x, z = w % a.nz, y0 = (w / a.nz) * X::RP;
	const size_t n = (size_t)HX * a.ny * a.nz;
	if constexpr (B) {
		x.load(r.Sx, z, y0, a.ny, a.nz, r.ntl);
		X::gsync();
		x.template c2r<EL>(r.scale);
		__syncthreads();
	}
	double gz[4] = { 0, 0, 0, 0 };
	struct Out { F3 lam, lamY; VjpCell c; double g; };
	auto cell = [&](size_t idx, int i, int y, F3 Nu) {
		Out o{};
		F3 v{ 0.f, 0.f, 0.f };
		if constexpr (B) {
			v = vjp_b_cell(a, Nu, b.cu_in, ld3(b.lx, idx), idx, i, y, z);
			o.lam = ld3(b.lacc, idx) + v;
		}
		else o.lam = ld3(b.lam, idx);
		if constexpr (A) {
			if constexpr (RN) o.lamY = renorm_cell(b.Y, a.Ms[idx], o.lam, o.g, idx);
			else o.lamY = ld3(b.lamY, idx);
			F3 wv = ((b.dt / 6) * b.wS) * o.lamY;
			if constexpr (!RN) wv = wv + (b.cS * b.dt) * v;
			o.c = vjp_a_cell(a, b.X, ld_planar(b.Hd, n, idx), wv, o.g, gz, idx, i, y, z);
			o.g += b.gMs[idx];
		}
		return o;
	};
	auto put = [&](size_t idx, const Out& o) {
		if constexpr (!A) { st3(b.lam, idx, o.lam); return; }
		if constexpr (RN) st3(b.lamY, idx, o.lamY);
		st3(b.lacc, idx, RN ? o.lamY : o.lam);
		st3(b.lx, idx, o.c.lx);
		st3(b.cu_out, idx, o.c.cu);
		b.gMs[idx] = o.g;
	};
	for (int p = threadIdx.x; p < X::RP * NP; p += X::BS) {
		const int rl = p / NP, k = p % NP, y = y0 + rl;
		C2<float>* t = tile + rl * X::P + k;
		C2<float>& tx = t[0]; C2<float>& ty = t[X::RP * X::P]; C2<float>& tz = t[2 * X::RP * X::P];
		if (y >= a.ny) { if constexpr (!B) { tx = ty = tz = mk(0.f, 0.f); } continue; }
		const size_t idx = ((size_t)z * a.ny + y) * HX + 2 * k;
		F3 n0{ 0.f, 0.f, 0.f }, n1 = n0;
		if constexpr (B) { n0 = F3{ tx.x, ty.x, tz.x }; n1 = F3{ tx.y, ty.y, tz.y }; }
		// both cells' loads before either's stores
		const Out o0 = cell(idx, 2 * k, y, n0), o1 = cell(idx + 1, 2 * k + 1, y, n1);
		put(idx, o0); put(idx + 1, o1);
		const F3 u0 = o0.c.u, u1 = o1.c.u;
		if constexpr (A) { tx = mk(u0.x, u1.x); ty = mk(u0.y, u1.y); tz = mk(u0.z, u1.z); }
	}
	if constexpr (A) {
		// deterministic sums of the work item's Zeeman terms
#pragma unroll
		for (int c = 0; c < 4; c++) {
			double s = gz[c];
			for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
			if ((threadIdx.x & 63) == 0) red[c * (X::BS / 64) + (threadIdx.x >> 6)] = s;
		}
		__syncthreads();
		if (threadIdx.x < 4) {
			double s = 0;
			for (int q = 0; q < X::BS / 64; q++) s += red[threadIdx.x * (X::BS / 64) + q];
			b.apart[4 * w + threadIdx.x] += s;
		}
		x.template r2c<EL>();
		X::gsync();
		x.store(r.Sx, z, y0, a.ny, a.nz, r.ntl);
	}
}

} // namespace

int bm::adj_row_fwd(int stage, const AdjArgs& a, const AdjRow& r, const AdjFwd& f, hipStream_t st)
{
	const dim3 g(xs_parts(a.nx, a.ny, a.nz));
	prof_mark_begin(PK_ROW, st);
	switch (a.nx) {
#define C_(V_) case V_: if constexpr (xs_ok<V_>()) { \
		const dim3 b(XSplit<V_, xs_groups<V_>()>::BS); \
		if (stage == 0) hipLaunchKernelGGL((k_adj_fwd<V_, 0>), g, b, 0, st, a, r, f); \
		else if (stage == 1) hipLaunchKernelGGL((k_adj_fwd<V_, 1>), g, b, 0, st, a, r, f); \
		else if (stage == 2) hipLaunchKernelGGL((k_adj_fwd<V_, 2>), g, b, 0, st, a, r, f); \
		else hipLaunchKernelGGL((k_adj_fwd<V_, 3>), g, b, 0, st, a, r, f); \
		prof_mark_end(PK_ROW, st); \
		return BM_OK; } break;
	BM_FOR_ROW_SIZES(C_)
#undef C_
	}
	return fail(BM_ERR_SIZE, "no adjoint row kernel for this row length");
}

int bm::adj_row_bwd(bool vb, bool rn, bool va, const AdjArgs& a, const AdjRow& r, const AdjBwd& w, hipStream_t st)
{
	const dim3 g(xs_parts(a.nx, a.ny, a.nz));
	prof_mark_begin(PK_ROW, st);
	switch (a.nx) {
#define C_(V_) case V_: if constexpr (xs_ok<V_>()) { \
		const dim3 b(XSplit<V_, xs_groups<V_>()>::BS); \
		if (!vb) hipLaunchKernelGGL((k_adj_bwd<V_, false, true, true>), g, b, 0, st, a, r, w); \
		else if (!va) hipLaunchKernelGGL((k_adj_bwd<V_, true, false, false>), g, b, 0, st, a, r, w); \
		else if (rn) hipLaunchKernelGGL((k_adj_bwd<V_, true, true, true>), g, b, 0, st, a, r, w); \
		else hipLaunchKernelGGL((k_adj_bwd<V_, true, false, true>), g, b, 0, st, a, r, w); \
		prof_mark_end(PK_ROW, st); \
		return BM_OK; } break;
	BM_FOR_ROW_SIZES(C_)
#undef C_
	}
	return fail(BM_ERR_SIZE, "no adjoint row kernel for this row length");
}
