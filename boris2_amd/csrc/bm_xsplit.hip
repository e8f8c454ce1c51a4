// Launchers of the x passes with one component per wave group (bm_xsplit.h).
#include "bm_xsplit.h"

#include <algorithm>

namespace {

using namespace bm;

template <int HX, bool FULL, bool GEN>
void inv_var(int mode, dim3 g, hipStream_t st, const float2* Sx, float* out, int ny, int nz, int ntl, float scale,
	const float* M, double* epart, int nx, int zoff, int nzl)
{
	const PassBatch* nb = nullptr;
	const dim3 b(XSplit<HX, xs_groups<HX>()>::BS);
	if (mode == 0) hipLaunchKernelGGL((k_inv_xs<HX, 0, false, FULL, GEN>), g, dim3(XSplit<HX>::BS), 0, st, Sx, out, ny, nz, ntl, scale, M, epart, nx, zoff, nzl, nb);
	else if (mode == 1 && !epart) hipLaunchKernelGGL((k_inv_xs<HX, 1, false, FULL, GEN>), g, b, 0, st, Sx, out, ny, nz, ntl, scale, M, epart, nx, zoff, nzl, nb);
	else if (mode == 1) hipLaunchKernelGGL((k_inv_xs<HX, 1, true, FULL, GEN>), g, b, 0, st, Sx, out, ny, nz, ntl, scale, M, epart, nx, zoff, nzl, nb);
	else if (!epart) hipLaunchKernelGGL((k_inv_xs<HX, 2, false, FULL, GEN>), g, b, 0, st, Sx, out, ny, nz, ntl, scale, M, epart, nx, zoff, nzl, nb);
	else hipLaunchKernelGGL((k_inv_xs<HX, 2, true, FULL, GEN>), g, b, 0, st, Sx, out, ny, nz, ntl, scale, M, epart, nx, zoff, nzl, nb);
}

} // namespace

// `items`: work items of the plain pass (tiles of XTile rows).  Measured, plain -> split:
//  - stand-alone x passes (field of a mesh) win while the plain pass has fewer than two items
//    per compute unit (one for rows of a whole wave): 64x64x1 20.4 -> 14.7 us, 128x128x4 40.0 ->
//    25.4, 256x256x16 (256 items) 108 -> 101; against it 256x256x32 (512 items) 177 -> 177,
//    512x512x4 (256 items) 104 -> 107, 768x768x4 (384 items) 246 -> 277.
//  - the row kernel likewise (RK4 steps: 128x64x1 188 -> 63 us, 256x256x8 356 -> 265, 256x256x16
//    467 -> 428, 512x512x4 447 -> 414; 256x256x32 752 -> 805, 512x512x7 (448 items) 703 -> 727),
//    and at any size for the radix-3 lengths, whose plain row kernel needs 256 registers, one
//    wave per SIMD (384x384x32 2483 -> 2084, 192x192x128 3482 -> 2909).
bool bm::xs_few_rows(int HX, int ny, int nz, int ncu, bool row)
{
	switch (HX) {
#define C_(V_) case V_: { if (!xs_ok<V_>()) return false; \
		if (row && xs_row_only<V_>()) return true; \
		const long long items = (long long)nz * ((ny + XTile<V_>::v - 1) / XTile<V_>::v); \
		return plan_T<V_>() <= 32 ? items < 2LL * ncu : row ? items <= ncu : items < ncu; }
	BM_FOR_ROW_SIZES(C_)
#undef C_
	}
	return false;
}

int bm::xs_parts(int HX, int ny, int nz)
{
	switch (HX) {
#define C_(V_) case V_: if constexpr (xs_ok<V_>()) return nz * ((ny + XSplit<V_>::RP - 1) / XSplit<V_>::RP); else return 0;
	BM_FOR_ROW_SIZES(C_)
#undef C_
	}
	return 0;
}

int bm::launch_fwd_xs(int HX, bool full, const FwdArgs& a, hipStream_t st)
{
	const FwdArgs* nb = nullptr;
	const dim3 g(xs_parts(HX, a.ny, a.nz));
	switch (HX) {
#define C_(V_) case V_: if constexpr (xs_ok<V_>()) { \
		const dim3 b(XSplit<V_>::BS); \
		if (full) hipLaunchKernelGGL((k_fwd_xs<V_, false, true, false>), g, b, 0, st, a, nb); \
		else if (a.nx != V_) hipLaunchKernelGGL((k_fwd_xs<V_, false, false, true>), g, b, 0, st, a, nb); \
		else if (a.E0) hipLaunchKernelGGL((k_fwd_xs<V_, true, false, false>), g, b, 0, st, a, nb); \
		else hipLaunchKernelGGL((k_fwd_xs<V_, false, false, false>), g, b, 0, st, a, nb); \
		return BM_OK; } break;
	BM_FOR_ROW_SIZES(C_)
#undef C_
	}
	return fail(BM_ERR_SIZE, "no split x pass for this row length");
}

int bm::launch_inv_xs(int HX, bool full, int mode, const float2* Sx, float* out, int ny, int nz, int ntl, float scale, hipStream_t st,
	const float* M, double* epart, int nx, int zoff, int nzl)
{
	const dim3 g(xs_parts(HX, ny, nz));
	switch (HX) {
#define C_(V_) case V_: if constexpr (xs_ok<V_>()) { \
		if (full) inv_var<V_, true, false>(mode, g, st, Sx, out, ny, nz, ntl, scale, M, epart, V_, zoff, nzl); \
		else if (nx != V_) inv_var<V_, false, true>(mode, g, st, Sx, out, ny, nz, ntl, scale, M, epart, nx, zoff, nzl); \
		else inv_var<V_, false, false>(mode, g, st, Sx, out, ny, nz, ntl, scale, M, epart, V_, zoff, nzl); \
		return BM_OK; } break;
	BM_FOR_ROW_SIZES(C_)
#undef C_
	}
	return fail(BM_ERR_SIZE, "no split x pass for this row length");
}

// batched: one mesh per grid row, as many blocks as the largest mesh needs
int bm::batch_fwd_xs(int HX, bool full, const FwdArgs* h_tab, const FwdArgs* d_tab, int nb, hipStream_t st)
{
	int mx = 1;
	for (int b = 0; b < nb; b++) mx = std::max(mx, xs_parts(HX, h_tab[b].ny, h_tab[b].nz));
	const dim3 g(mx, nb);
	FwdArgs a{};
	switch (HX) {
#define C_(V_) case V_: if constexpr (xs_ok<V_>()) { \
		if (full) hipLaunchKernelGGL((k_fwd_xs<V_, false, true, false>), g, dim3(XSplit<V_>::BS), 0, st, a, d_tab); \
		else hipLaunchKernelGGL((k_fwd_xs<V_, false, false, false>), g, dim3(XSplit<V_>::BS), 0, st, a, d_tab); \
		return BM_OK; } break;
	BM_FOR_ROW_SIZES(C_)
#undef C_
	}
	return fail(BM_ERR_SIZE, "no split x pass for this row length");
}

int bm::batch_inv_xs_planar(int HX, bool full, const PassBatch* h_tab, const PassBatch* d_tab, int nb, hipStream_t st)
{
	int mx = 1;
	for (int b = 0; b < nb; b++) mx = std::max(mx, xs_parts(HX, h_tab[b].ny, h_tab[b].nz));
	const dim3 g(mx, nb);
	switch (HX) {
#define C_(V_) case V_: if constexpr (xs_ok<V_>()) { \
		if (full) hipLaunchKernelGGL((k_inv_xs<V_, 0, false, true, false>), g, dim3(XSplit<V_>::BS), 0, st, nullptr, nullptr, 0, 0, 0, 0.f, nullptr, nullptr, V_, 0, 0, d_tab); \
		else hipLaunchKernelGGL((k_inv_xs<V_, 0, false, false, false>), g, dim3(XSplit<V_>::BS), 0, st, nullptr, nullptr, 0, 0, 0, 0.f, nullptr, nullptr, V_, 0, 0, d_tab); \
		return BM_OK; } break;
	BM_FOR_ROW_SIZES(C_)
#undef C_
	}
	return fail(BM_ERR_SIZE, "no split x pass for this row length");
}
