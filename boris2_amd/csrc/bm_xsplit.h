// The x passes with one component per wave group, for launches with few rows.
//
// The passes of bm_xpass.h / bm_row.h give a row's three components to one thread group, one
// after another, in tiles of up to 32 rows: right for a mesh that fills the device many times
// over, but a small mesh then runs a handful of workgroups, each a long serial chain.  Here a
// workgroup of 3 W waves holds RP = 64 W / T rows; waves cW .. cW + W - 1 transform component
// c, and every row lies within one wave, so the transform's exchanges need no workgroup
// barrier.  Per-cell work between the transforms takes the three components from LDS, cell
// pairs spread over all waves.  Same plans and arithmetic as the other passes: the same bits.
//
// Bound: latency (one round of loads, one transform chain).
#pragma once

#include "bm_internal.h"
#include "bm_stage.h"
#include "bm_xpass.h"

namespace bm {

// waves per component.  One wave (8 rows of 64 cells, 4 of 128, 2 of 256) measured best for rows
// of part of a wave (RK4 steps: 128x64x1 63.5 us against 68.4 with two and 81.4 with four, 256x256x1
// 73.5 / 78.3 / 90.1); rows of a whole wave need several for usable runs of the spectra (512x512x4
// 464 us with two waves, 413 with four; 1024x1024x1 395 with two, 490 with four).
template <int HX> constexpr int xs_waves() { return plan_T<HX>() <= 32 ? 1 : HX <= 512 ? 4 : 2; }
// a row must lie within one wave
template <int HX> constexpr bool xs_ok() { return plan_T<HX>() <= 64; }

// lengths whose row kernel always takes this form (see xs_few_rows)
template <int HX> constexpr bool xs_row_only() { return xs_ok<HX>() && Plan<HX>::E == 12; }

// wave groups of the kernels with much per-cell work: with 8 values per thread the 32 W E cell pairs of
// a workgroup are a third more than three groups, so rows of 16 lanes or fewer take a fourth wave for
// the per-cell work only (one round instead of two: 128x64 film RK4 step 48.1 -> 46.9 us, ten 128x64
// layers 105 -> 101).
template <int HX> constexpr int xs_groups()
{
	return xs_waves<HX>() == 1 && Plan<HX>::E == 8 && plan_T<HX>() <= 16 ? 4 : 3;
}
// The row kernel at 32 lanes (256 cells per row) has both forms.  Its registers leave three waves per
// SIMD, so a compute unit holds four workgroups of three waves or three of four: the fourth wave
// pays (RK4 steps of 256x256 cells by 1, 3, 6 planes 65.6 -> 63.1, 125.5 -> 121.4, 186.1 -> 180.5 us, of
// 3 layers 123.0 -> 117.4) but where the workgroups are more than three and at most four per compute
// unit, one round without it and two with (256x256 by 7 and 8 planes 205.9 -> 212.9, 208.7 -> 216.0, of
// 8 layers 298 -> 305); from the second round on it pays again (9, 12, 24 planes 303 -> 293, 339 -> 330,
// 607 -> 590).
template <int HX> constexpr bool xs_row_both() { return xs_waves<HX>() == 1 && Plan<HX>::E == 8 && plan_T<HX>() == 32; }
inline bool xs_row_four(int workgroups, int ncu) { return workgroups <= 3 * ncu || workgroups > 4 * ncu; }

template <int HX, int NG = 3> struct XSplit {
	static constexpr int W = xs_waves<HX>(), WT = 64 * W, E = Plan<HX>::E, T = plan_T<HX>();
	static constexpr int BS = NG * WT;
	static constexpr int RP = WT / T, NC = HX + 1, P = xrow_pitch<HX>();
	static constexpr int NL = (RP * NC + WT - 1) / WT;   // spectra values per thread of one component
	int c, q;                // component (3: the fourth wave), thread within its wave group
	C2<float>* mine;         // this component's rows
	C2<float>* row;          // this thread's row
	XThread<HX> th;

	__device__ __forceinline__ void init(C2<float>* tile)
	{
		c = threadIdx.x / WT; q = threadIdx.x % WT;
		th.init_at(q % T);
		mine = tile + c * RP * P;
		row = mine + (q / T) * P;
	}
	// the group's waves wait for each other; a single wave orders its own LDS accesses
	static __device__ __forceinline__ void gsync() { xsync<W == 1>(); }

	__device__ __forceinline__ void load(const float2* Sx, int z, int y0, int ny, int nzs, int ntl) const
	{
		if (c > 2) return;
		const float2* base = Sx + sx_base(c, z, y0, nzs, NC, ntl);
		float2 r[NL];
#pragma unroll
		for (int l = 0; l < NL; l++) {
			const int idx = q + WT * l;
			int kx, yl, off;
			sx_tile_elem<RP, NC>(idx, kx, yl, off);
			r[l] = (idx < RP * NC && y0 + yl < ny) ? base[off] : make_float2(0.f, 0.f);
		}
#pragma unroll
		for (int l = 0; l < NL; l++) {
			const int idx = q + WT * l;
			int kx, yl, off;
			sx_tile_elem<RP, NC>(idx, kx, yl, off);
			if (idx < RP * NC) mine[yl * P + kx] = mk(r[l].x, r[l].y);
		}
	}
	__device__ __forceinline__ void store(float2* Sx, int z, int y0, int ny, int nzs, int ntl) const
	{
		if (c > 2) return;
		float2* base = Sx + sx_base(c, z, y0, nzs, NC, ntl);
#pragma unroll
		for (int l = 0; l < NL; l++) {
			const int idx = q + WT * l;
			int kx, yl, off;
			sx_tile_elem<RP, NC>(idx, kx, yl, off);
			if (idx < RP * NC && y0 + yl < ny) { const C2<float> a = mine[yl * P + kx]; base[off] = make_float2(a.x, a.y); }
		}
	}
	// this thread's row from the spectra in LDS to EL scaled cell pairs in LDS (pair k at k)
	template <int EL> __device__ __forceinline__ void c2r(float scale)
	{
		if (c > 2) return;
		C2<float> v[E];
		c2r_row<HX, true>(th, row, v);
		xsync<true>();                   // the transform's last LDS reads are done
#pragma unroll
		for (int e = 0; e < EL; e++) row[th.t + T * e] = mk(v[e].x * scale, v[e].y * scale);
	}
	// the reverse: EL cell pairs in LDS (zero above) to the row's spectra in LDS
	template <int EL> __device__ __forceinline__ void r2c()
	{
		if (c > 2) return;
		C2<float> v[E];
#pragma unroll
		for (int e = 0; e < E; e++) v[e] = e < EL ? row[th.t + T * e] : mk(0.f, 0.f);
		xsync<true>();
		r2c_row<HX, true>(th, row, v);
	}
};

// P1 (k_fwd_x) in this form: the rows' cells are read once by all waves, two cells per thread,
// into LDS (with ADV the RKDP54 advance on the way), then transformed by component.
template <int HX, bool ADV, bool FULL, bool GEN>
__global__ void __launch_bounds__(XSplit<HX>::BS) k_fwd_xs(FwdArgs a, const FwdArgs* __restrict__ bt)
{
	using X = XSplit<HX>;
	if (bt) a = bt[blockIdx.y];
	__shared__ C2<float> tile[3 * X::RP * X::P];
	X x; x.init(tile);
	constexpr int EL = FULL ? X::E : X::E / 2, NP = FULL ? HX : HX / 2, NXR = FULL ? 2 * HX : HX;
	const int nxr = GEN ? a.nx : NXR, ntiles = (a.ny + X::RP - 1) / X::RP, nwork = a.nz * ntiles;
	for (int w = blockIdx.x; w < nwork; w += gridDim.x) {
		const int z = w % a.nz, y0 = (w / a.nz) * X::RP;
		for (int p = threadIdx.x; p < X::RP * NP; p += X::BS) {
			const int r = p / NP, k = p % NP, y = y0 + r;
			P6 m{ F3{ 0.f, 0.f, 0.f }, F3{ 0.f, 0.f, 0.f } };
			if (y < a.ny) {
				const size_t cell = ((size_t)z * a.ny + y) * (size_t)nxr + 2 * k;
				if constexpr (GEN) {
					if (2 * k < nxr) m.a = ld3(a.M, cell);
					if (2 * k + 1 < nxr) m.b = ld3(a.M, cell + 1);
				}
				else m = ld6(a.M, cell);
				if constexpr (ADV) {
					const P6 e0 = ld6(a.E0, cell);
					st6(a.sM1, cell, m);
					m = m + a.dT5 * e0;
					st6(a.Mout, cell, m);
				}
			}
			C2<float>* t = tile + r * X::P + k;
			t[0] = mk(m.a.x, m.b.x); t[X::RP * X::P] = mk(m.a.y, m.b.y); t[2 * X::RP * X::P] = mk(m.a.z, m.b.z);
		}
		__syncthreads();
		x.template r2c<EL>();
		X::gsync();
		x.store(a.Sx, z + a.zoff, y0, a.ny, a.nzl ? a.nzl : a.nz, a.ntl);
		__syncthreads();
	}
}

// P5 (k_inv_x) in this form; modes as there.  The interleaved outputs go through LDS so that a
// thread moves whole cell pairs.
template <int HX, int MODE> constexpr int xs_inv_groups() { return MODE == 0 ? 3 : xs_groups<HX>(); }
template <int HX, int MODE, bool EN, bool FULL, bool GEN>
__global__ void __launch_bounds__((XSplit<HX, xs_inv_groups<HX, MODE>()>::BS)) k_inv_xs(const float2* __restrict__ Sx, float* __restrict__ out,
	int ny, int nz, int ntl, float scale, const float* __restrict__ M, double* __restrict__ epart,
	int nxr, int zoff, int nzl, const PassBatch* __restrict__ bt)
{
	using X = XSplit<HX, xs_inv_groups<HX, MODE>()>;
	if (bt) { const PassBatch& b = bt[blockIdx.y]; Sx = b.Sx; out = b.out; ny = b.ny; nz = b.nz; ntl = b.ntl; scale = b.scale; }
	__shared__ C2<float> tile[3 * X::RP * X::P];
	__shared__ double ered[EN ? X::BS : 1];
	X x; x.init(tile);
	constexpr int EL = FULL ? X::E : X::E / 2, NP = FULL ? HX : HX / 2;
	const int nx = GEN ? nxr : FULL ? 2 * HX : HX, ntiles = (ny + X::RP - 1) / X::RP, nwork = nz * ntiles;
	const size_t ncell = (size_t)nx * ny * nz;
	for (int w = blockIdx.x; w < nwork; w += gridDim.x) {
		const int z = w % nz, y0 = (w / nz) * X::RP;
		x.load(Sx, zoff + z, y0, ny, nzl ? nzl : nz, ntl);
		X::gsync();
		x.template c2r<EL>(scale);
		__syncthreads();
		double esum = 0.0;
		if constexpr (MODE == 0) {
			// planar: each wave group stores its own component
			for (int p = x.q; x.c < 3 && p < X::RP * NP; p += X::WT) {
				const int r = p / NP, k = p % NP, y = y0 + r;
				if (y >= ny) continue;
				const C2<float> h = x.mine[r * X::P + k];
				float* o = out + (size_t)x.c * ncell + ((size_t)z * ny + y) * nx + 2 * k;
				if constexpr (GEN) {
					if (2 * k < nx) o[0] = h.x;
					if (2 * k + 1 < nx) o[1] = h.y;
				}
				else *reinterpret_cast<float2*>(o) = make_float2(h.x, h.y);
			}
		}
		else {
			for (int p = threadIdx.x; p < X::RP * NP; p += X::BS) {
				const int r = p / NP, k = p % NP, y = y0 + r;
				if (y >= ny) continue;
				const C2<float>* t = tile + r * X::P + k;
				const C2<float> hx = t[0], hy = t[X::RP * X::P], hz = t[2 * X::RP * X::P];
				const P6 h{ F3{ hx.x, hy.x, hz.x }, F3{ hx.y, hy.y, hz.y } };
				const size_t cell = ((size_t)z * ny + y) * nx + 2 * k;
				const bool v0 = !GEN || 2 * k < nx, v1 = !GEN || 2 * k + 1 < nx;
				// single cells: the caller's array need not be aligned beyond 4 bytes
				if (v0) st3(out, cell, MODE == 2 ? ld3(out, cell) + h.a : h.a);
				if (v1) st3(out, cell + 1, MODE == 2 ? ld3(out, cell + 1) + h.b : h.b);
				if constexpr (EN) {
					auto part = [](F3 m, F3 f) { return (double)(m.x * f.x) + (double)(m.y * f.y) + (double)(m.z * f.z); };
					if (v0) esum += part(ld3(M, cell), h.a);
					if (v1) esum += part(ld3(M, cell + 1), h.b);
				}
			}
		}
		if constexpr (EN) {
			// deterministic per-work-item partial of sum M.H
			ered[threadIdx.x] = esum;
			__syncthreads();
			if (threadIdx.x < 64) {
				double s = 0.0;
				for (int b = threadIdx.x; b < X::BS; b += 64) s += ered[b];
				for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
				if (threadIdx.x == 0) epart[w] = s;
			}
		}
		__syncthreads();
	}
}

// The fused row kernel (k_row) in this form; LAY: a layer stack (the planes are the layers), a form of
// its own because the per-layer values cost plain meshes 3 % (RK4 step of a 128x64 film 47.8 -> 49.5 us).
// NG: its wave groups.
template <int HX, int METHOD, int STEP, bool R2C, bool LAY, int NG>
__global__ void __launch_bounds__((XSplit<HX, NG>::BS)) k_rows(StageArgs a, float2* Sx, int ntl, int ntiles, float scale)
{
	using X = XSplit<HX, NG>;
	__shared__ C2<float> tile[3 * X::RP * X::P];
	X x; x.init(tile);
	constexpr int EL = X::E / 2, NP = HX / 2;
	const int ny = a.ny, nz = a.nz, nwork = nz * ntiles;
	float lte_loc = 0.f;
	// XCD-contiguous work as in k_row (gridDim.x a multiple of 8)
	for (int g = 0; g * (int)gridDim.x < nwork; g++) {
		const int w = g * (int)gridDim.x + (int)xcd_chunk(blockIdx.x, gridDim.x);
		if (w >= nwork) continue;     // uniform over the block
		const int z = w % nz, y0 = (w / nz) * X::RP;
		x.load(Sx, z, y0, ny, nz, ntl);
		X::gsync();
		x.template c2r<EL>(scale);
		__syncthreads();
		for (int p = threadIdx.x; p < X::RP * NP; p += X::BS) {
			const int r = p / NP, k = p % NP, y = y0 + r;
			if (y >= ny) continue;
			C2<float>* t = tile + r * X::P + k;
			const C2<float> hx = t[0], hy = t[X::RP * X::P], hz = t[2 * X::RP * X::P];
			const size_t idx = ((size_t)z * ny + y) * HX + 2 * k;
			const P6 mn = stage_pair<METHOD, STEP, LAY>(a, idx, 2 * k, y, z, ld6(a.Min, idx), P6{ F3{ hx.x, hy.x, hz.x }, F3{ hx.y, hy.y, hz.y } }, lte_loc);
			if constexpr (R2C) {
				t[0] = mk(mn.a.x, mn.b.x); t[X::RP * X::P] = mk(mn.a.y, mn.b.y); t[2 * X::RP * X::P] = mk(mn.a.z, mn.b.z);
			}
		}
		__syncthreads();
		if constexpr (R2C) {
			x.template r2c<EL>();
			X::gsync();
			x.store(Sx, z, y0, ny, nz, ntl);
			__syncthreads();
		}
	}
	if (stage_has_lte<METHOD, STEP>()) block_max_to<X::BS>(lte_loc, a);
}

} // namespace bm
