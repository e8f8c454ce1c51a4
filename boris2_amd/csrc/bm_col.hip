// The middle of the convolution as one kernel per group of kx columns: y FFT of a column's lines,
// the product with the demag kernel (2D; layers: the sum over all pairs; 3D: z FFT, product, z
// inverse), y inverse FFT, in place on the x-side spectra Sx.
//
// A workgroup holds the 3 P lines (component, plane) of LPK columns in LDS.  A line is
// transformed by T lanes of one wave, in its own LDS space, so the transforms need no workgroup
// barrier; the lines are spread over the waves, the product over all threads.
//
// Against the separate y, z (or layer product) and y passes it saves two launches, the full
// spectra's four trips through memory and the kernel-wide serial chain of three components per
// thread.  Bound: LDS capacity (3 P lines of N.y values; beyond it the separate passes run), then
// latency (small meshes) or vector issue.
#include "bm_internal.h"
#include "bm_fft.h"
#include "bm_xpass.h"

#include <algorithm>

namespace {

using namespace bm;

// what the product does: one plane with the 2D kernel, layers, or planes along z (N.z)
enum { COL_2D = 1, COL_LAYERS = 2, COL_Z = 3 };
// threads at most (two waves per SIMD, up to 256 registers); layers, whose product items per thread
// (destination, column, ky) are held in registers between reads and writes, take up to 1024 (NZ = 2)
// where 512 cannot hold them: measured 128x128x12 layers 95 us separate, 42.5 with 1024; 256x256x3
// 32.9 with 512, 38.8 with 1024
template <int KIND, int NZ> constexpr int col_threads() { return KIND == COL_LAYERS && NZ == 2 ? 1024 : 512; }
constexpr int kColItems = 4;

struct ColArgs {
	float2* Sx; const float* K; const int* kidx;
	int P, NC, NYH, ntl, nyd, lpk, tr;
	const ColBatch* bt;     // batched: one mesh or stack per grid row
	int ncu;                // compute units (for the launchers)
};

// The columns kx = 0 and kx = N.x / 2 hold real values: in the z form of one mesh from N.z = 16 (PACK),
// whose workgroups fill a compute unit each, the first workgroup takes both as one complex line (first + i second) where a column more
// than a multiple of the compute units would cost a round of its own (RK4 steps: 256x256x8, 257
// columns on 256 units, 235 -> 212 us, 256x128x16 242 -> 228, 512x256x8 389 -> 369).  A real line's transform is X(-ky) = conj X(ky), so the two spectra come apart
// (and together) within the pair (ky, -ky): both are worked on for ky = 0 .. N.y / 2, column 0's
// results at ky and the other's at N.y - ky, both in one value at ky = 0 and N.y / 2.  Not in batches,
// whose meshes share the rounds: a mesh there computes the same bits whatever runs beside it.
__device__ __forceinline__ C2<float> pair_get(const C2<float>* line, int NY, int ky, int col)
{
	const C2<float> a = line[ky], b = line[ky ? NY - ky : 0];
	return col ? mk(0.5f * (a.y + b.y), 0.5f * (b.x - a.x)) : mk(0.5f * (a.x + b.x), 0.5f * (a.y - b.y));
}
__device__ __forceinline__ void pair_put(C2<float>* line, int NY, int ky, int col, C2<float> w)
{
	if (ky == 0 || ky == NY / 2) { if (col) line[ky].y = w.x; else line[ky].x = w.x; }
	else line[col ? NY - ky : ky] = w;
}
// the packed line's value at ky from what pair_put left
__device__ __forceinline__ C2<float> pair_line(const C2<float>* line, int NY, int ky)
{
	const C2<float> v = line[ky];
	if (ky == 0 || ky == NY / 2) return v;
	const C2<float> o = line[NY - ky];
	return ky < NY / 2 ? mk(v.x - o.y, v.y + o.x) : mk(o.x + v.y, v.x - o.y);
}

// the value of the lane whose number differs in bit 0 (or 1), within four lanes
template <int CTRL> __device__ __forceinline__ C2<float> lane_quad(C2<float> v)
{
	return mk(__int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v.x), CTRL, 0xf, 0xf, true)),
		__int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v.y), CTRL, 0xf, 0xf, true)));
}
__device__ __forceinline__ C2<float> lane_xor1(C2<float> v) { return lane_quad<0xB1>(v); }   // lanes 1 0 3 2
__device__ __forceinline__ C2<float> lane_xor2(C2<float> v) { return lane_quad<0x4E>(v); }   // lanes 2 3 0 1

// The z transform of N.z points on M adjacent lanes (up to 8 values each), the plan's stages with
// the exchange between them through lane swaps instead of LDS.
template <int NZ> struct ZLanes {
	static constexpr int M = plan_T<NZ>(), R1 = Plan<NZ>::S > 1 ? Plan<NZ>::R[Plan<NZ>::S - 1] : 1;
	static_assert(M == R1 && M <= 4 && Plan<NZ>::S <= 2, "one radix-8 stage, then one over the lanes");

	template <int DIR> static __device__ __forceinline__ void run(C2<float>* v, int t, const Twiddles<NZ, float>& tw)
	{
		if constexpr (M == 1) Dft<NZ, DIR, float>::run(v);
		else {
			constexpr int B = 8 / M;      // second-stage butterflies per lane: j = t + M b over A_0[j] .. A_(M-1)[j]
			Dft<8, DIR, float>::run(v);
#pragma unroll
			for (int b = 0; b < B; b++) {
				// lane t's values M b .. M b + M - 1 against the other lanes' value M b + t
				C2<float> m[M];
#pragma unroll
				for (int q = 0; q < M; q++) m[q] = v[M * b + q];
#pragma unroll
				for (int q = 0; q < M; q += 2) {
					const C2<float> got = lane_xor1((t & 1) ? m[q] : m[q + 1]);
					if (t & 1) m[q] = got; else m[q + 1] = got;
				}
				if constexpr (M == 4) {
#pragma unroll
					for (int q = 0; q < 2; q++) {
						const C2<float> got = lane_xor2((t & 2) ? m[q] : m[q + 2]);
						if (t & 2) m[q] = got; else m[q + 2] = got;
					}
				}
#pragma unroll
				for (int q = 1; q < M; q++) {
					const C2<float> w = tw.w[plan_twoff<NZ>(1) + b * (M - 1) + q - 1];
					m[q] = DIR < 0 ? cmul(m[q], w) : cmulc(m[q], w);
				}
				Dft<M, DIR, float>::run(m);
#pragma unroll
				for (int q = 0; q < M; q++) v[M * b + q] = m[q];
			}
			// butterfly b's output q is element t + M (b + B q): registers into that order
			C2<float> o[8];
#pragma unroll
			for (int b = 0; b < B; b++)
#pragma unroll
				for (int q = 0; q < M; q++) o[b + B * q] = v[M * b + q];
#pragma unroll
			for (int e = 0; e < 8; e++) v[e] = o[e];
		}
	}
};

inline bool col_packed(int lpk, int NC, int ncu) { return lpk == 1 && NC > ncu && (NC - 1) % ncu == 0; }

template <int NY, int KIND, int NZ, bool FULL, bool PACK>
__global__ void __launch_bounds__((col_threads<KIND, NZ>()), (KIND == COL_LAYERS && NY < 1024 ? 4 : 1)) k_col(ColArgs a)
{
	constexpr int E = Plan<NY>::E, T = plan_T<NY>(), LW = 64 / T, LL = lds_len<NY>(), EL = FULL ? E : E / 2, NZH = NZ / 2 + 1;
	static_assert(T <= 64, "a line must lie within one wave");
	extern __shared__ C2<float> lb[];
	if (a.bt) {
		const ColBatch& b = a.bt[blockIdx.y];
		a.Sx = b.Sx; a.K = b.K; a.kidx = b.kidx; a.P = b.P; a.NC = b.NC; a.NYH = b.NYH; a.ntl = b.ntl; a.nyd = b.nyd;
	}
	const int lane = threadIdx.x & 63, t = lane % T, sub = lane / T, stride = (blockDim.x >> 6) * LW;
	const int P = KIND == COL_2D ? 1 : a.P, lpk = a.lpk, nl = 3 * P * lpk, kx0 = blockIdx.x * lpk;
	const bool both = PACK && blockIdx.x == 0;
	if (kx0 >= a.NC) return;                                   // uniform over the block
	Twiddles<NY, float> tw; tw.init(t);

	// lines li = (c P + z) lpk + column: the next round's values are loaded while this one's are
	// transformed
	C2<float> pre[EL];
	auto fetch = [&](int li) {
		const int cz = li / lpk, kx = kx0 + li % lpk;
		const bool ok = li < nl && kx < a.NC;
#pragma unroll
		for (int e = 0; e < EL; e++) {
			const int y = t + T * e;
			float2 q = make_float2(0.f, 0.f);
			if (ok && y < a.nyd) {
				q = a.Sx[sx_line(cz, kx, y, a.NC, a.ntl)];
				if (both) q.y = a.Sx[sx_line(cz, a.NC - 1, y, a.NC, a.ntl)].x;
			}
			pre[e] = mk(q.x, q.y);
		}
	};
	const int l0 = (threadIdx.x >> 6) * LW;                   // uniform over the wave
	if (l0 < nl) fetch(l0 + sub);
	for (int b = l0; b < nl; b += stride) {
		const int li = b + sub;
		C2<float> v[E];
#pragma unroll
		for (int e = 0; e < E; e++) v[e] = e < EL ? pre[e] : mk(0.f, 0.f);
		if (b + stride < nl) fetch(li + stride);
		C2<float>* line = lb + li * LL;
		fft<NY, -1, float, true>(v, line, 1, t, tw);
		xsync<true>();                                        // the transform's last LDS reads are done
#pragma unroll
		for (int e = 0; e < E; e++) line[t + T * e] = v[e];
	}
	__syncthreads();

	if constexpr (KIND == COL_2D) {
		const size_t kq = (size_t)a.NC * a.NYH;
		for (int i = threadIdx.x; i < lpk * NY; i += blockDim.x) {
			const int il = i / NY, ky = i % NY, kx = min(kx0 + il, a.NC - 1);
			const int kyr = ky <= NY / 2 ? ky : NY - ky;
			const float sy = ky <= NY / 2 ? 1.f : -1.f;
			const size_t ki = (size_t)kx * a.NYH + kyr;
			const float kxx = a.K[ki], kyy = a.K[kq + ki], kzz = a.K[2 * kq + ki], kxy = sy * a.K[3 * kq + ki];
			C2<float>* p = lb + il * LL + ky;
			const C2<float> mx = p[0], my = p[lpk * LL], mz = p[2 * lpk * LL];
			p[0] = lin2(kxx, mx, kxy, my);
			p[lpk * LL] = lin2(kxy, mx, kyy, my);
			p[2 * lpk * LL] = mk(kzz * mz.x, kzz * mz.y);
		}
	}
	else if constexpr (KIND == COL_LAYERS) {
		// item (destination d, column, ky); own layer first, then the others in order (k_ml_mult); four
		// sources' kernel loads in flight (ten 128x64 layers: 32.4 -> 27.0 us with the shared kernels)
		const size_t kq = (size_t)a.NC * a.NYH;
		const int items = P * lpk * NY, cs = P * lpk * LL;        // component stride of the lines
		const float tz = a.tr ? -1.f : 1.f;
		float2 o[kColItems][3];
#pragma unroll
		for (int n = 0; n < kColItems; n++) {
			const int i = threadIdx.x + n * blockDim.x;
			float2 o0 = make_float2(0.f, 0.f), o1 = o0, o2 = o0;
			if (i < items) {
				const int ky = i % NY, dl = i / NY, d = dl / lpk, il = dl % lpk, kx = min(kx0 + il, a.NC - 1);
				const bool up = ky > NY / 2;
				const float sy = up ? -1.f : 1.f;
				const float* Kb = a.K + (size_t)kx * a.NYH + (up ? NY - ky : ky);
				const C2<float>* Fb = lb + il * LL + ky;
#pragma unroll 4
				for (int r = 0; r < P; r++) {
					const int s = r == 0 ? d : (r <= d ? r - 1 : r), p = a.tr ? s * P + d : d * P + s;
					const float* Kp = Kb + (size_t)(a.kidx ? a.kidx[p] : p) * 6 * kq;
					const float kxx = Kp[0], kyy = Kp[kq], kzz = Kp[2 * kq];
					const float kxy = sy * Kp[3 * kq], kxz = tz * Kp[4 * kq], kyz = tz * sy * Kp[5 * kq];
					const C2<float>* F = Fb + s * lpk * LL;
					const C2<float> fx = F[0], fy = F[cs], fz = F[2 * cs];
					o0.x += kxx * fx.x + kxy * fy.x - kxz * fz.y;  o0.y += kxx * fx.y + kxy * fy.y + kxz * fz.x;
					o1.x += kxy * fx.x + kyy * fy.x - kyz * fz.y;  o1.y += kxy * fx.y + kyy * fy.y + kyz * fz.x;
					o2.x += -kxz * fx.y - kyz * fy.y + kzz * fz.x; o2.y += kxz * fx.x + kyz * fy.x + kzz * fz.y;
				}
			}
			o[n][0] = o0; o[n][1] = o1; o[n][2] = o2;
		}
		__syncthreads();                                          // every destination has read its sources
#pragma unroll
		for (int n = 0; n < kColItems; n++) {
			const int i = threadIdx.x + n * blockDim.x;
			if (i < items) {
				C2<float>* p = lb + (i / NY) * LL + i % NY;       // i / NY = d lpk + column, as the lines are
#pragma unroll
				for (int c = 0; c < 3; c++) p[c * cs] = mk(o[n][c].x, o[n][c].y);
			}
		}
	}
	else {
		// a (column, ky) takes M adjacent lanes; lane zt holds planes, and outputs kz, zt + M e
		constexpr int M = ZLanes<NZ>::M, NF = NZ / M, ZD = NZ / 2;
		const size_t kq = (size_t)a.NC * a.NYH * NZH;
		const int zs = lpk * LL, cs = P * zs, zt = threadIdx.x % M;
		Twiddles<NZ, float> tz; tz.init(zt);
		// both: the pair's two items run in adjacent lanes and read before either writes
		for (int i = threadIdx.x; i < (both ? NY + 2 : lpk * NY) * M; i += blockDim.x) {
			const int j = i / M, il = both ? 0 : j / NY, col = both ? j & 1 : 0, ky = both ? j >> 1 : j % NY;
			const int kx = col ? a.NC - 1 : min(kx0 + il, a.NC - 1);
			const int kyr = ky <= NY / 2 ? ky : NY - ky;
			const float sy = ky <= NY / 2 ? 1.f : -1.f;
			const float* kb = a.K + ((size_t)kx * a.NYH + kyr) * NZH;
			C2<float>* p = lb + il * LL;
			C2<float> u[3][NF];
#pragma unroll
			for (int c = 0; c < 3; c++) {
#pragma unroll
				for (int e = 0; e < NF; e++) { const int z = zt + M * e; 
					u[c][e] = M * e < ZD && z < P ? (both ? pair_get(p + c * cs + z * zs, NY, ky, col) : p[c * cs + z * zs + ky]) : mk(0.f, 0.f);
				}
				ZLanes<NZ>::template run<-1>(u[c], zt, tz);
			}
#pragma unroll
			for (int e = 0; e < NF; e++) {
				const int kz = zt + M * e, kzr = kz <= NZ / 2 ? kz : NZ - kz;
				const float sz = kz <= NZ / 2 ? 1.f : -1.f;
				const float kxx = kb[kzr], kyy = kb[kq + kzr], kzz = kb[2 * kq + kzr];
				const float kxy = sy * kb[3 * kq + kzr], kxz = sz * kb[4 * kq + kzr], kyz = sy * sz * kb[5 * kq + kzr];
				const C2<float> mx = u[0][e], my = u[1][e], mz = u[2][e];
				u[0][e] = lin3(kxx, mx, kxy, my, kxz, mz);
				u[1][e] = lin3(kxy, mx, kyy, my, kyz, mz);
				u[2][e] = lin3(kxz, mx, kyz, my, kzz, mz);
			}
#pragma unroll
			for (int c = 0; c < 3; c++) {
				ZLanes<NZ>::template run<1>(u[c], zt, tz);
#pragma unroll
				for (int e = 0; e < NF; e++) {
					const int z = zt + M * e;
					if (M * e < ZD && z < P) {
						if (both) pair_put(p + c * cs + z * zs, NY, ky, col, u[c][e]);
						else p[c * cs + z * zs + ky] = u[c][e];
					}
				}
			}
		}
	}
	__syncthreads();

	for (int b = l0; b < nl; b += stride) {
		const int li = b + sub, cz = li / lpk, kx = kx0 + li % lpk;
		C2<float>* line = lb + li * LL;
		C2<float> v[E];
#pragma unroll
		for (int e = 0; e < E; e++) v[e] = both ? pair_line(line, NY, t + T * e) : line[t + T * e];
		xsync<true>();
		fft<NY, 1, float, true>(v, line, 1, t, tw);
		if (li < nl && kx < a.NC) {
#pragma unroll
			for (int e = 0; e < EL; e++) {
				const int y = t + T * e;
				if (y >= a.nyd) continue;
				a.Sx[sx_line(cz, kx, y, a.NC, a.ntl)] = make_float2(v[e].x, both ? 0.f : v[e].y);
				if (both) a.Sx[sx_line(cz, a.NC - 1, y, a.NC, a.ntl)] = make_float2(v[e].y, 0.f);
			}
		}
	}
}

// Columns per workgroup (a wave's lanes filled where a column's lines are few) and threads.
struct ColShape { int lpk, threads; size_t lds; };
template <int NY, int KIND, int NZ> ColShape col_shape(int P)
{
	constexpr int T = plan_T<NY>(), LW = 64 / T, LL = lds_len<NY>();
	ColShape s;
	s.lpk = std::max(1, 64 / (3 * P * T));
	const int nl = 3 * P * s.lpk, nlp = (nl + LW - 1) / LW * LW;
	// a wave per LW lines; more where the product's items need them
	int waves = nlp / LW;
	if constexpr (KIND == COL_LAYERS) waves = std::max(waves, (P * s.lpk * NY + 64 * kColItems - 1) / (64 * kColItems));
	if constexpr (KIND == COL_Z) waves = std::max(waves, (s.lpk * NY * plan_T<NZ>() + 63) / 64);
	s.threads = std::min(col_threads<KIND, NZ>(), 64 * waves);
	s.lds = (size_t)nlp * LL * sizeof(C2<float>);
	return s;
}

template <int NY, int KIND, int NZ, bool FULL, bool PACK = false>
int launch_col_t(const ColArgs& in, int nb, hipStream_t st)
{
	// the z form of one mesh with one workgroup per compute unit: columns 0 and N.x / 2 as one
	if constexpr (KIND == COL_Z && NZ >= 16 && NY % 3 != 0 && !PACK)
		if (!in.bt && col_packed(col_shape<NY, KIND, NZ>(in.P).lpk, in.NC, in.ncu)) return launch_col_t<NY, KIND, NZ, FULL, true>(in, nb, st);
	const ColShape s = col_shape<NY, KIND, NZ>(in.P);
	ColArgs a = in;
	a.lpk = s.lpk;
	if (s.lds > 65536)
		BM_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_col<NY, KIND, NZ, FULL, PACK>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)s.lds));
	hipLaunchKernelGGL((k_col<NY, KIND, NZ, FULL, PACK>), dim3((a.NC - PACK + s.lpk - 1) / s.lpk, nb), dim3(s.threads), s.lds, st, a);
	return BM_OK;
}

// lengths whose lines lie within one wave
#define BM_FOR_COL_SIZES(M) M(4) M(6) M(8) M(12) M(16) M(24) M(32) M(48) M(64) M(96) M(128) M(192) M(256) M(384) M(512) M(768) M(1024)
constexpr size_t kColLds = 150 * 1024;

// the fewest planes of an open N.z (more than a quarter of it) fit LDS
template <int NY, int NZ> constexpr bool col_z_fits() { return 3 * (NZ / 4 + 1) * lds_len<NY>() * sizeof(C2<float>) <= kColLds; }

// the layers form with 512 (V = 1) or 1024 threads holds P layers; the latter not for N.y = 1024,
// whose 16 values per thread do not fit its 128 registers (512x512x3 99 us separate, 141 so)
template <int NY, int V> bool col_items(int P)
{
	if constexpr (V == 2 && NY >= 1024) return false;
	const ColShape s = col_shape<NY, COL_LAYERS, V>(P);
	return s.lds <= kColLds && (long long)P * s.lpk * NY <= (long long)kColItems * s.threads;
}

} // namespace

// kind: N.z (3D, open z: 4 to 32), 1 (2D) or 0 (layers).  Where the lines fit, against the separate
// passes (field of a mesh, separate -> column): 64x64x1 14.7 -> 12.0 us, 128x128x4 25.3 -> 17.2,
// 128x128x8 31.0 -> 24.5, 512x512x4 104 -> 88, layers 128x128x8 54.1 -> 32.5, 256x256x8 60.0 -> 59.2.
// Not for radix-3 lengths with N.z >= 16 beyond one column per compute unit (256x192x8 52 -> 62,
// 512x192x8 88 -> 95: the longer schedules of 12 values per thread).
bool bm::col_ok(int Ny, int kind, int P, int NC, int ncu)
{
	if (kind > 1 && kind != 4 && kind != 8 && kind != 16 && kind != 32) return false;
	if (kind >= 16 && Ny % 3 == 0 && NC > ncu) return false;
	switch (Ny) {
#define C_(V_) case V_: { if (!kind) return col_items<V_, 1>(P) || col_items<V_, 2>(P); \
		return col_shape<V_, COL_Z, 4>(P).lds <= kColLds; }
	BM_FOR_COL_SIZES(C_)
#undef C_
	}
	return false;
}

namespace {
int launch_any(int Ny, int kind, bool full, const ColArgs& a, int nb, hipStream_t st)
{
	switch (Ny) {
#define C_(V_) case V_: \
		if (kind == 0 && col_items<V_, 1>(a.P)) return full ? launch_col_t<V_, COL_LAYERS, 1, true>(a, nb, st) : launch_col_t<V_, COL_LAYERS, 1, false>(a, nb, st); \
		if constexpr (V_ < 1024) if (kind == 0) return full ? launch_col_t<V_, COL_LAYERS, 2, true>(a, nb, st) : launch_col_t<V_, COL_LAYERS, 2, false>(a, nb, st); \
		if (kind == 1) return full ? launch_col_t<V_, COL_2D, 1, true>(a, nb, st) : launch_col_t<V_, COL_2D, 1, false>(a, nb, st); \
		if constexpr (col_z_fits<V_, 4>()) if (kind == 4) return full ? launch_col_t<V_, COL_Z, 4, true>(a, nb, st) : launch_col_t<V_, COL_Z, 4, false>(a, nb, st); \
		if constexpr (col_z_fits<V_, 8>()) if (kind == 8) return full ? launch_col_t<V_, COL_Z, 8, true>(a, nb, st) : launch_col_t<V_, COL_Z, 8, false>(a, nb, st); \
		if constexpr (col_z_fits<V_, 16>()) if (kind == 16) return full ? launch_col_t<V_, COL_Z, 16, true>(a, nb, st) : launch_col_t<V_, COL_Z, 16, false>(a, nb, st); \
		if constexpr (col_z_fits<V_, 32>()) if (kind == 32) return full ? launch_col_t<V_, COL_Z, 32, true>(a, nb, st) : launch_col_t<V_, COL_Z, 32, false>(a, nb, st); \
		break;
	BM_FOR_COL_SIZES(C_)
#undef C_
	}
	return fail(BM_ERR_SIZE, "no column pass for this length");
}
}

int bm::launch_col(int Ny, int kind, bool full, float2* Sx, const float* K, const int* kidx, int P, int NC, int NYH, int ntl, int nyd, int tr, int ncu,
	hipStream_t st)
{
	return launch_any(Ny, kind, full, ColArgs{ Sx, K, kidx, P, NC, NYH, ntl, nyd, 1, tr, nullptr, ncu }, 1, st);
}

// sized by the largest mesh: LDS and threads by its planes, grid rows by its columns
int bm::batch_col(int Ny, int kind, bool full, const ColBatch* h_tab, const ColBatch* d_tab, int nb, int ncu, hipStream_t st)
{
	ColArgs a{};
	a.lpk = 1; a.bt = d_tab; a.ncu = ncu;
	for (int b = 0; b < nb; b++) { a.P = std::max(a.P, h_tab[b].P); a.NC = std::max(a.NC, h_tab[b].NC); }
	return launch_any(Ny, kind, full, a, nb, st);
}
